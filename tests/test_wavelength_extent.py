"""The extent of a wavelength array on both sides of the size from which it is
scanned by torch, for the forms of array that take either way."""
import numpy as np
import pytest

from raypier_optics_amd.cmaterials import wavelength_extent


@pytest.mark.parametrize("n", [1, 65535, 65536, 200003])
@pytest.mark.parametrize("form", ["plain", "reversed", "strided", "read-only", "float32", "two-dimensional"])
def test_extent(n, form):
    w = np.random.default_rng(n).uniform(0.3, 1.7, n)
    if form == "reversed":
        w = w[::-1]
    elif form == "strided":
        w = np.repeat(w, 2)[::2]
    elif form == "read-only":
        w.flags.writeable = False
    elif form == "float32":
        w = w.astype(np.float32)
    elif form == "two-dimensional":
        w = w.reshape(1, n)
    assert wavelength_extent(w) == (float(w.min()), float(w.max()))


@pytest.mark.parametrize("n", [10, 65536])
def test_extent_of_special_values(n):
    w = np.full(n, 0.5)
    w[n // 2] = np.inf
    w[n // 3] = -np.inf
    assert wavelength_extent(w) == (-np.inf, np.inf)
    w = w.copy()
    w[n - 1] = np.nan
    assert all(np.isnan(wavelength_extent(w)))
    assert wavelength_extent(np.zeros(0)) == (np.inf, -np.inf)
