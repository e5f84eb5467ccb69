"""Traces either side of the tile-size rule (512-ray tiles from 69,632 input
rays on, 256 below): one call equals the concatenation of calls on pieces of
the input, all of which take the small tiles, to the last bit.  Both run the
same code per ray, and children keep their parents' order, so nothing but the
placement differs."""
import numpy as np
import pytest

from raypier_optics_amd import workloads
from raypier_optics_amd.ctracer import RayCollection
from raypier_optics_amd.tracer import trace_rays

pytestmark = pytest.mark.gpu


def _trace(rays, w, depth):
    rc = RayCollection.from_array(rays.copy())
    rc.wavelengths = w.wavelengths
    traced, faces = trace_rays(rc, w.face_lists, recursion_limit=depth, max_length=w.max_length)
    return [g.copy_as_array() for g in traced], [f.count for f in faces]


@pytest.mark.parametrize("system", ["spheres", "aspheres"])
@pytest.mark.parametrize("n", [65535, 65536, 65537, 66049, 69631, 69632, 69633, 70145, 98303])
def test_tile_sizes_agree(gpu, system, n):
    if system == "spheres":
        w, depth = workloads.singlet_c1(n), 4
    else:
        w, depth = workloads.lens_job_c5(3, n_rays=n), 6
        for fl in w.face_lists:
            for f in fl.faces:
                if hasattr(f.material, "reflection_threshold"):
                    f.material.reflection_threshold = 0.02     # some rays get two children
    rays = w.rays
    n = len(rays)
    got, counts = _trace(rays, w, depth)
    cuts = [0, 40000, n] if n <= 100000 else list(range(0, n, 50000)) + [n]
    pieces = [_trace(rays[a:b], w, depth) for a, b in zip(cuts, cuts[1:])]
    assert max(b - a for a, b in zip(cuts, cuts[1:])) < 65536
    assert len(got) == max(len(p) for p, _ in pieces)
    assert counts == [sum(c) for c in zip(*(c for _, c in pieces))]
    for g, a in enumerate(got):
        parts, base = [], 0
        for p, _ in pieces:
            if g < len(p):
                b = p[g].copy()
                if g:
                    b["parent_idx"] += np.uint32(base)
                parts.append(b)
            if 0 < g <= len(p):
                base += len(p[g - 1])
        b = np.concatenate(parts)
        assert len(a) == len(b), g
        for name in a.dtype.names:
            assert np.ascontiguousarray(a[name]).tobytes() == np.ascontiguousarray(b[name]).tobytes(), (g, name)
