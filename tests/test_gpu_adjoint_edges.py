"""The adjoint's wavefront sums and column partials at the edges of its
workgroups (256 rays) and wavefronts (64), with vignetted rays among the kept
ones, against the float64 autograd reference.  Tolerances as
test_gpu_adjoint.py's: 1e-8 relative per component with a floor of 1e-10 of
the largest component of the same kind."""
import numpy as np
import pytest

from raypier_optics_amd import workloads
from raypier_optics_amd.adjoint import SequentialLens, spot_rms_and_grad, spot_moments
from tests import adjoint_reference as ar

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [3, 5, 11])
@pytest.mark.parametrize("n", [3, 64, 65, 255, 257, 4099])
def test_adjoint_edges(gpu, seed, n):
    w = workloads.lens_job_c5(seed, n_rays=n)
    lens = SequentialLens.from_workload(w)
    if n > 60:
        lens.apertures = np.array(lens.apertures, float)
        lens.apertures[0] = 3.0          # rays start on a disk of 4 mm radius
    r = w.rays
    sigma, g = spot_rms_and_grad(lens, w.collection())
    s_ref, g_ref, keep = ar.spot_rms_grad(lens, r["origin"], r["direction"], r["wavelength_idx"], w.wavelengths)
    if n > 60:
        assert 0 < np.count_nonzero(keep) < n
    assert int(spot_moments(lens, w.collection())[0]) == np.count_nonzero(keep)
    assert abs(sigma - s_ref) <= 1e-12 * s_ref
    floor = 1e-10 * np.abs(g_ref).max(axis=0)
    err = np.abs(g - g_ref)
    assert np.all(err <= 1e-8 * np.abs(g_ref) + floor), (seed, np.max(err / (np.abs(g_ref) + floor)))
