"""Oblique rays on aspheric faces against the oracle: rays up to 1.5 rad from the
axis, many of which miss the base conic.  The root search of such a ray starts
a whole segment behind the ray's origin (cfaces.pyx:1909-1976 takes the conic's
-1 for the fraction of the segment); from a start nearer by it reaches roots
that the reference does not accept."""
import numpy as np
import pytest

import oracle
from raypier_optics_amd import workloads
from raypier_optics_amd._scene import compile_scene
from raypier_optics_amd.cfaces import AsphericFace
from raypier_optics_amd.cmaterials import PartiallyReflectiveMaterial
from raypier_optics_amd.cshapes import CircleShape
from raypier_optics_amd.ctracer import FaceList, GaussletCollection, RayCollection
from raypier_optics_amd.split import SplitRayCollection, trace_rays_split
from raypier_optics_amd.tracer import trace_rays
from tests.helpers import compare_generation

LENGTH = 100.0
WL = np.array([0.55])
# (curvature, conic constant, A4, A6, A8, A10, aperture radius).  The last digit of
# a start decides nothing at this tolerance; at atol = 1e-16, which the last
# rounding of a step may miss, the reference drops rays at random.
ATOL = 1e-10
SURFACES = [(-30.0, -0.6, -2e-5, 1e-7, -3e-10, 5e-13, 10.0),
            (25.0, -2.0, 1e-5, 0.0, 0.0, 0.0, 12.0),
            (-25.0, -0.5, -2e-5, 0.0, 0.0, 0.0, 20.0)]


def oblique_rays(n, seed, radius):
    rng = np.random.default_rng(seed)
    r = workloads.base_rays(n)
    th, ph = rng.uniform(0, 1.5, n), rng.uniform(0, 2 * np.pi, n)
    d = np.column_stack([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), rng.choice([-1.0, 1.0], n) * np.cos(th)])
    at = np.column_stack([rng.uniform(-1.5 * radius, 1.5 * radius, (n, 2)), rng.uniform(-8, 8, n)])
    d = (d / np.linalg.norm(d, axis=1)[:, None]).astype(np.float32)
    r["origin"] = (at - d * rng.uniform(5, 25, n)[:, None]).astype(np.float32)   # exact in the FP32-split records too
    r["direction"] = d
    e = np.cross(r["direction"], rng.normal(size=(n, 3)))
    r["E_vector"] = e / np.linalg.norm(e, axis=1)[:, None]
    r["E1_amp"], r["E2_amp"] = 1.0, 0.3j
    r["refractive_index"] = 1.0
    return r


def missing_the_conic(s, r):
    """Rays without a real root of the base conic (cfaces.pyx:1695-1747)."""
    beta, R = 1 + s[1], -s[0]
    a, d = r["origin"], r["direction"]
    W = np.array([beta, beta, beta * beta])
    A = d * d @ W
    B = 2 * (a * d @ W) - 2 * R * beta * d[:, 2]
    C = a * a @ W - 2 * R * beta * a[:, 2]
    return B * B - 4 * A * C < 0


def scene(s):
    fl = FaceList()
    fl.faces = [AsphericFace(curvature=s[0], conic_const=s[1], A4=s[2], A6=s[3], A8=s[4], A10=s[5], z_height=0.0,
                             atol=ATOL, shape=CircleShape(radius=s[6]),
                             material=PartiallyReflectiveMaterial(reflectivity=0.4))]
    workloads.prepare_faces([fl], WL, LENGTH)
    return [fl]


def collection(r):
    rc = RayCollection.from_array(r.copy())
    rc.wavelengths = WL
    return rc


@pytest.mark.parametrize("k", range(len(SURFACES)))
def test_the_rays_reach_past_the_conic(k):
    s = SURFACES[k]
    r = oblique_rays(60000, 70 + k, s[6])
    first = oracle.trace_rays(compile_scene(scene(s)), r, LENGTH, WL, 1)[0][0]
    assert np.count_nonzero(missing_the_conic(s, r)) > 9000
    assert np.count_nonzero(first["end_face_idx"] == 0) > 10000


@pytest.mark.gpu
@pytest.mark.parametrize("k", range(len(SURFACES)))
def test_traces(gpu, k):
    s = SURFACES[k]
    r = oblique_rays(60000, 70 + k, s[6])
    lists = scene(s)
    ref, hits = oracle.trace_rays(compile_scene(lists), r, LENGTH, WL, 2)
    got, faces = trace_rays(collection(r), lists, recursion_limit=2, max_length=LENGTH)
    assert len(got) == len(ref)
    for g, (a, b) in enumerate(zip(got, ref)):
        compare_generation(a.copy_as_array(), b, what="generation %d" % g)
    assert [f.count for f in faces] == [int(h) for h in hits[:1]]
    # FP32-split: the first generation's records are exact, and its roots float64
    split = trace_rays_split(SplitRayCollection.from_collection(collection(r)), lists, recursion_limit=1,
                             max_length=LENGTH)[0][0].to_collection().copy_as_array()
    assert np.array_equal(split["end_face_idx"], ref[0]["end_face_idx"])


@pytest.mark.gpu
@pytest.mark.parametrize("k", range(len(SURFACES)))
def test_gausslets(gpu, k):
    s = SURFACES[k]
    g = GaussletCollection.from_rays(oblique_rays(20000, 80 + k, s[6]))
    g.config_parabasal_rays(WL, 0.6, 0.0)
    g.wavelengths = WL
    lists = scene(s)
    ref, hits = oracle.trace_rays(compile_scene(lists), g.copy_as_array(), LENGTH, WL, 2, gausslet=True)
    got, faces = trace_rays(g, lists, recursion_limit=2, max_length=LENGTH)
    assert len(got) == len(ref)
    for n, (a, b) in enumerate(zip(got, ref)):
        a = a.copy_as_array()
        compare_generation(a["base_ray"], b["base_ray"], what="generation %d" % n)
    assert [f.count for f in faces] == [int(h) for h in hits[:1]]
