"""Power thresholds of interfaces for rays so faint that their power is a
subnormal number, whose reciprocal overflows: the children are those of a ray of
ordinary amplitude."""
import numpy as np
import pytest

import oracle
from raypier_optics_amd import _queries, workloads
from raypier_optics_amd.cfaces import CircularFace
from raypier_optics_amd.cmaterials import FullDielectricMaterial, SingleLayerCoatedMaterial
from raypier_optics_amd.ctracer import FaceList, RayCollection
from raypier_optics_amd.split import SplitRayCollection, trace_rays_split
from tests.helpers import compare_generation, scene_of_material

pytestmark = pytest.mark.gpu

WL = np.array([0.55])
# Reflected shares of glass lie below 0.12 up to 0.9 rad and above 0.4 from 1.48 on
# (a film of a quarter wave lowers the first): well apart from this threshold
THRESHOLD = 0.25
ANGLES = np.concatenate([np.linspace(0.01, 0.9, 40), np.linspace(1.48, 1.56, 20)])
MATERIALS = {"bare": lambda: FullDielectricMaterial(n_inside=1.5, n_outside=1.0, reflection_threshold=THRESHOLD,
                                                    transmission_threshold=THRESHOLD),
             "film": lambda: SingleLayerCoatedMaterial(n_inside=1.5, n_outside=1.0, n_coating=1.38, thickness=0.1,
                                                       reflection_threshold=THRESHOLD,
                                                       transmission_threshold=THRESHOLD)}


def rays(amplitude):
    r = workloads.base_rays(len(ANGLES))
    r["origin"] = np.column_stack([np.zeros((len(ANGLES), 2)), np.full(len(ANGLES), 3.0)])
    r["direction"] = np.column_stack([np.sin(ANGLES), np.zeros(len(ANGLES)), -np.cos(ANGLES)])
    r["E_vector"] = (0.0, 1.0, 0.0)
    r["E1_amp"], r["E2_amp"] = amplitude, 0.7 * amplitude
    r["refractive_index"] = 1.0
    return r


@pytest.mark.parametrize("name", sorted(MATERIALS))
@pytest.mark.parametrize("amplitude", [1.0, 1e-153, 1e-155, 3e-159])
def test_float64(gpu, name, amplitude):
    mat = MATERIALS[name]()
    r = rays(amplitude)
    m = len(r)
    pts, nrm, tan = np.zeros((m, 3)), np.tile([0.0, 0.0, 1.0], (m, 1)), np.tile([1.0, 0.0, 0.0], (m, 1))
    got, counts = _queries.eval_child_rays_batch(mat, r, 0, pts, nrm, tan, WL)
    t, mi = scene_of_material(mat)
    ref = [oracle.eval_child_ray(t, mi, r[i:i + 1], i, pts[i], nrm[i], tan[i], WL) for i in range(m)]
    assert counts.tolist() == [len(x) for x in ref]
    assert counts.min() == 1 and counts.max() == 2
    compare_generation(got, np.concatenate(ref))


@pytest.mark.parametrize("name", sorted(MATERIALS))
@pytest.mark.parametrize("amplitude", [1e-19, 1e-20, 3e-21])
def test_split(gpu, name, amplitude):
    def children(a):
        fl = FaceList()
        fl.faces = [CircularFace(diameter=1e4, z_plane=0.0, material=MATERIALS[name]())]
        rc = RayCollection.from_array(rays(a))
        rc.wavelengths = WL
        traced = trace_rays_split(SplitRayCollection.from_collection(rc), [fl], recursion_limit=2, max_length=1e3)[0]
        return traced[1].to_collection().copy_as_array()

    a, b = children(1.0), children(amplitude)
    assert len(ANGLES) < len(a) < 2 * len(ANGLES)
    for f in ("parent_idx", "ray_type_id", "direction"):
        assert np.array_equal(a[f], b[f]), f
