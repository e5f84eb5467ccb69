"""Zernike distortions as the kernels evaluate them (coefficients summed by
|m| and parity, chains in r^2): against the oracle's literal recursion over
single terms, terms that share a group, three and five coefficients per
chain, the axis (all signs of zero), points next to it and outside the unit
circle; and against numpy for a table whose polynomials mix parities, which
no Zernike term does but the ABI accepts."""
import numpy as np
import pytest

import oracle
from raypier_optics_amd import _abi, _queries
from raypier_optics_amd._scene import SceneBuilder
from raypier_optics_amd.cdistortions import ZernikeDistortion, compile_zernike

pytestmark = pytest.mark.gpu


def points(unit):
    g = np.random.default_rng(8)
    r = unit * np.concatenate([np.sqrt(g.random(200)) * 1.2, [1e-3, 1e-8, 1e-100, 1e-150, 1e-170]])
    t = 2 * np.pi * g.random(len(r))
    x, y = r * np.cos(t), r * np.sin(t)
    z = np.array([0.0, -0.0, 0.0, -0.0, unit, -unit, 0.0, 0.0])
    w = np.array([0.0, 0.0, -0.0, -0.0, 0.0, 0.0, unit, -unit])
    return np.concatenate([x, z]), np.concatenate([y, w])


def bound(coefs, unit):
    """Largest size of a sum's terms over the points (r <= 1.2), times 1e-13:
    a few hundred roundings of terms that cancel."""
    _, cs, _, _, _ = compile_zernike(sorted(coefs), unit)
    r = 1.2 ** np.arange(_abi.ZPOLY)
    s = sum(abs(float(c["nval"])) * np.abs(c["poly"]).dot(r).max() * (abs(int(c["m"])) + 1) for c in cs)
    return 1e-13 * s


@pytest.mark.parametrize("js", [[0], [1], [2], [4], [12], [24], [27], [40], [54], [3, 4, 5], [0, 4, 12, 24, 40],
                                [7, 8, 17, 18, 31], list(range(3, 16)), list(range(55))])
def test_groups_against_oracle(gpu, js):
    g = np.random.default_rng(sum(js) + len(js))
    unit = 7.5
    coefs = [(j, g.normal()) for j in js]
    dist = ZernikeDistortion(coefs, unit_radius=unit)
    b = SceneBuilder()
    zi = b.distortion_index(dist)
    x, y = points(unit)
    ref_sag, ref_grad = oracle.zernike(b.finish(), zi, x, y)
    sag, grad = _queries.zernike_eval(dist, x, y)
    tol = bound(coefs, unit)
    assert np.abs(sag - ref_sag).max() <= tol
    assert np.abs(grad - ref_grad).max() <= tol


class MixedParity(ZernikeDistortion):
    """Polynomials of both parities in every quantity."""

    def _rpx_compile(self, rec, builder):
        super()._rpx_compile(rec, builder)
        g = np.random.default_rng(5)
        for c in builder._zcoefs:
            c["poly"][:] = g.normal(size=c["poly"].shape)
            c["deg"][:] = _abi.ZPOLY - 1
        self.records = [c.copy() for c in builder._zcoefs]


def test_mixed_parity_polynomials(gpu):
    unit = 3.0
    dist = MixedParity([(j, 0.1 * (j + 1)) for j in (4, 5, 7, 12, 14)], unit_radius=unit)
    g = np.random.default_rng(1)
    x, y = g.uniform(-2, 2, 300), g.uniform(-2, 2, 300)
    sag, grad = _queries.zernike_eval(dist, x, y)
    r, t = np.hypot(x, y) / unit, np.arctan2(y, x)
    want, gx, gy, gz = (np.zeros_like(x) for _ in range(4))
    for c in dist.records:
        m, N = int(c["m"]), float(c["nval"])
        S, R, Rp, Ror = (np.polyval(c["poly"][q][::-1], r) for q in range(4))
        PH, PHp = (np.cos(m * t), -m * np.sin(m * t)) if m >= 0 else (-np.sin(m * t), -m * np.cos(m * t))
        want += N * S * PH
        gz += N * R * PH
        gx += N * (Rp * np.cos(t) * PH - Ror * np.sin(t) * PHp) / unit
        gy += N * (Rp * np.sin(t) * PH + Ror * np.cos(t) * PHp) / unit
    # ten-term polynomials of unit coefficients at r < 1, five of them
    for got, ref in ((sag, want), (grad[:, 0], gx), (grad[:, 1], gy), (grad[:, 2], gz)):
        assert np.abs(got - ref).max() <= 1e-12
