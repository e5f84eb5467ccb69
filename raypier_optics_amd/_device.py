"""Device storage of ray generations: structure-of-arrays in HBM.

One generation of rays is a single uint8 allocation holding 21 float64 rows
then 5 uint32 rows of `capacity` elements each (see rpx_rays_t); gausslets add
a float64 block of 60 rows (6 parabasal rays x 10 doubles).
"""
import ctypes
import numpy as np

from . import _abi
from ._lib import load, check, require_gpu, stream_handle


# Host records move through two pinned slots of this size, one being copied by
# the host's threads while the other is in flight; transfers below a quarter of
# it go directly.  MI355X, directly against through slots: 2 MB down 0.12 / 0.09
# ms, up 0.09 / 0.08; 20 MB down 1.20 / 0.47, up 0.58 / 0.49; 120 MB down 12.2 /
# 4.0, up 4.3 / 2.6 (4 MB slots: 4.9 and 2.8).
_SLOT = 8 << 20


def _slots(torch):
    """Two pinned slots (from torch's host allocator, which takes them back
    when the copies that use them have ended) and an event for each."""
    return ([torch.empty(_SLOT, dtype=torch.uint8, device="cpu", pin_memory=True) for _ in range(2)],
            [torch.cuda.Event() for _ in range(2)])


def _to_device(raw):
    """A device copy of a contiguous uint8 array, ordered on the current
    stream; `raw` has been read when this returns."""
    torch = _torch()
    n = raw.size
    if not raw.flags.writeable:
        raw = raw.copy()              # torch takes no read-only arrays
    host = torch.from_numpy(raw)
    if n < _SLOT // 4:
        return host.to("cuda")
    dev = torch.empty(n, dtype=torch.uint8, device="cuda")
    slots, events = _slots(torch)
    for k, a in enumerate(range(0, n, _SLOT)):
        m = min(_SLOT, n - a)
        slot, event = slots[k % 2], events[k % 2]
        if k >= 2:
            event.synchronize()
        slot[:m].copy_(host[a: a + m])
        dev[a: a + m].copy_(slot[:m], non_blocking=True)
        event.record()
    return dev


def _to_host(dev, out):
    """Copies the uint8 device tensor `dev` into the uint8 array `out`."""
    torch = _torch()
    n = dev.numel()
    host = torch.from_numpy(out)
    if n < _SLOT // 4:
        host.copy_(dev)
        return
    slots, events = _slots(torch)
    starts = range(0, n, _SLOT)

    def fetch(k):
        m = min(_SLOT, n - starts[k])
        slots[k % 2][:m].copy_(dev[starts[k]: starts[k] + m], non_blocking=True)
        events[k % 2].record()

    fetch(0)
    for k, a in enumerate(starts):
        if k + 1 < len(starts):
            fetch(k + 1)
        events[k % 2].synchronize()
        m = min(_SLOT, n - a)
        host[a: a + m].copy_(slots[k % 2][:m])


class DeviceRays(object):
    """HBM-resident SoA buffer for up to `capacity` rays (or gausslets)."""

    def __init__(self, capacity, gausslet=False):
        torch = require_gpu()
        self.capacity = int(capacity)
        self.gausslet = bool(gausslet)
        nbytes = self.capacity * (_abi.N_F64 * 8 + _abi.N_U32 * 4)
        self.buf = torch.empty(max(nbytes, 8), dtype=torch.uint8, device="cuda")
        if gausslet:
            self.para = torch.empty(max(self.capacity * _abi.N_PARA * _abi.PARA_FIELDS, 1),
                                    dtype=torch.float64, device="cuda")
        else:
            self.para = None

    # torch views -------------------------------------------------------
    def f64(self):
        cap = self.capacity
        return self.buf[: _abi.N_F64 * 8 * cap].view(dtype=_torch().float64).view(_abi.N_F64, cap)

    def u32(self):
        cap = self.capacity
        start = _abi.N_F64 * 8 * cap
        return self.buf[start: start + _abi.N_U32 * 4 * cap].view(dtype=_torch().int32).view(_abi.N_U32, cap)

    def para_view(self):
        cap = self.capacity
        return self.para[: _abi.N_PARA * _abi.PARA_FIELDS * cap].view(_abi.N_PARA, _abi.PARA_FIELDS, cap)

    def struct(self):
        base = self.buf.data_ptr()
        return _abi.Rays(base, base + _abi.N_F64 * 8 * self.capacity,
                         self.para.data_ptr() if self.para is not None else 0, self.capacity)

    # AoS conversion ----------------------------------------------------
    def upload(self, aos):
        """Copy a host ray_dtype / gausslet_dtype array into the SoA buffer."""
        torch = _torch()
        n = len(aos)
        if n == 0:
            return
        raw = np.ascontiguousarray(aos).view(np.uint8).reshape(-1)
        dev = _to_device(raw)
        lib = load()
        s = self.struct()
        check(lib.rpx_unpack_rays(ctypes.c_void_p(dev.data_ptr()), n, ctypes.byref(s), int(self.gausslet),
                                  stream_handle()))
        torch.cuda.current_stream().synchronize()

    def download(self, n):
        """Return the first n records as a host ray_dtype / gausslet_dtype array."""
        torch = _torch()
        dt = _abi.gausslet_dtype if self.gausslet else _abi.ray_dtype
        if n == 0:
            return np.zeros(0, dt)
        aos = torch.empty(n * dt.itemsize, dtype=torch.uint8, device="cuda")
        lib = load()
        s = self.struct()
        check(lib.rpx_pack_rays(ctypes.byref(s), n, ctypes.c_void_p(aos.data_ptr()), int(self.gausslet),
                                stream_handle()))
        out = np.empty(n, dt)
        _to_host(aos, out.view(np.uint8))
        return out


class DeviceRaysView(DeviceRays):
    """Rays [offset, offset + n) of a pool DeviceRays: the same buffer and
    field stride, so a generation written into a pool is a collection of its
    own without a copy.  Holds a reference to the pool."""

    def __init__(self, pool, offset, n):
        self.pool = pool
        self.offset = int(offset)
        self.capacity = int(n)
        self.gausslet = pool.gausslet
        self.buf = pool.buf
        self.para = pool.para

    def f64(self):
        return self.pool.f64()[:, self.offset: self.offset + self.capacity]

    def u32(self):
        return self.pool.u32()[:, self.offset: self.offset + self.capacity]

    def para_view(self):
        return self.pool.para_view()[:, :, self.offset: self.offset + self.capacity]

    def struct(self):
        s = self.pool.struct()
        o = self.offset
        return _abi.Rays(s.f64 + 8 * o, s.u32 + 4 * o, (s.para + 8 * o) if s.para else 0, self.pool.capacity)


def _torch():
    import torch
    return torch
