"""The traces' own face tests (unit segments, rpx_faces.h) and interface
amplitudes against the oracle: every face type, from both sides, in frames that
are the global one, translated and rotated, in one scene whose lists alternate
between them; and interfaces around the switch between the real and the
complex evaluation (total reflection in the film and behind it, absorption
down to nothing, normal and grazing incidence)."""
import math

import numpy as np
import pytest

import oracle
from raypier_optics_amd import _queries, workloads
from raypier_optics_amd._scene import compile_scene
from raypier_optics_amd.ctracer import FaceList, RayCollection, Transform, GaussletCollection
from raypier_optics_amd.tracer import trace_rays
from raypier_optics_amd.split import SplitRayCollection, trace_rays_split
from raypier_optics_amd.cmaterials import (FullDielectricMaterial, OpaqueMaterial, PartiallyReflectiveMaterial,
                                           SingleLayerCoatedMaterial)
from tests.helpers import compare_generation, scene_of_material
from tests.test_gpu_parity import _faces, random_rays

pytestmark = pytest.mark.gpu


def frame(kind):
    fl = FaceList()
    if kind == "global":
        return fl
    a, b = (0.3, -0.2) if kind == "rotated" else (0.0, 0.0)
    ca, sa, cb, sb = math.cos(a), math.sin(a), math.cos(b), math.sin(b)
    R = np.array([[ca, -sa, 0], [sa, ca, 0], [0, 0, 1]]) @ np.array([[1, 0, 0], [0, cb, -sb], [0, sb, cb]])
    t = np.array([0.4, -0.3, 0.7])
    fl.transform = Transform(rotation=R.tolist(), translation=t.tolist())
    fl.inverse_transform = Transform(rotation=R.T.tolist(), translation=(-(R.T @ t)).tolist())
    return fl


def crossing_rays(n, seed, extruded):
    """Rays through the origin's neighbourhood from both sides."""
    rng = np.random.default_rng(seed)
    r = random_rays(n, seed)
    d = np.column_stack([rng.uniform(-0.3, 0.3, n), rng.uniform(-0.3, 0.3, n), rng.choice([-1.0, 1.0], n)])
    if extruded:
        d = d[:, [2, 0, 1]]
    d /= np.linalg.norm(d, axis=1)[:, None]
    r["direction"] = d
    r["origin"] = rng.uniform(-4, 4, (n, 3)) - 15.0 * d
    e = np.cross(d, rng.normal(size=(n, 3)))
    r["E_vector"] = e / np.linalg.norm(e, axis=1)[:, None]
    r["refractive_index"] = 1.0
    return r


def check(face_lists, r, wl, max_length, depth, rel=1e-9):
    all_faces = workloads.prepare_faces(face_lists, wl, max_length)
    ref, hits = oracle.trace_rays(compile_scene(face_lists), r, max_length, wl, depth)
    rc = RayCollection.from_array(r.copy())
    rc.wavelengths = wl
    got, faces = trace_rays(rc, face_lists, recursion_limit=depth, max_length=max_length)
    assert len(got) == len(ref)
    for g, (a, b) in enumerate(zip(got, ref)):
        compare_generation(a.copy_as_array(), b, rel=rel, what="generation %d" % g)
    assert [f.count for f in faces] == [int(h) for h in hits[:len(faces)]]
    return ref


@pytest.mark.parametrize("kind", ["global", "translated", "rotated"])
@pytest.mark.parametrize("k", range(10))
def test_face_types_in_frames(gpu, k, kind):
    face = _faces()[k]
    face.material = PartiallyReflectiveMaterial(reflectivity=0.4)
    fl = frame(kind)
    fl.faces = [face]
    r = crossing_rays(3000, 50 + k, k == 6)
    ref = check([fl], r, np.array([0.55]), 60.0, 3)
    assert np.count_nonzero(ref[0]["end_face_idx"] == 0) > 300


def test_alternating_frames(gpu):
    """Lists in the global frame share a segment; one in another frame between
    them must not leave its own behind."""
    lists = []
    for n, kind in enumerate(["global", "rotated", "global", "global", "translated", "global"]):
        fl = frame(kind)
        face = _faces()[(4, 0, 8, 7, 2, 1)[n]]
        face.material = PartiallyReflectiveMaterial(reflectivity=0.5) if n < 5 else OpaqueMaterial()
        fl.faces = [face]
        lists.append(fl)
    ref = check(lists, crossing_rays(5000, 9, False), np.array([0.55]), 80.0, 4)
    assert len(set(ref[0]["end_face_idx"].tolist())) >= 4


def test_empty_reach(gpu):
    """Segments parallel to a plane, ending short of it, and of length zero
    give no hit."""
    fl = FaceList()
    fl.faces = _faces()[:1]
    fl.faces[0].material = OpaqueMaterial()
    r = crossing_rays(64, 3, False)
    r["direction"][:32] = (1.0, 0.0, 0.0)
    r["origin"][32:] = (0.0, 0.0, -9.0)
    r["direction"][32:] = (0.0, 0.0, 1.0)
    ref = check([fl], r, np.array([0.55]), 9.5, 2)
    assert np.all(ref[0]["end_face_idx"] == 0xFFFFFFFF)


GLASS = [(1.7, 1.0), (1.0, 1.7), (1.5, 1.5), (1.7 + 1e-30j, 1.0), (1.7 + 0.01j, 1.0), (1.0, 1.7 + 0.01j), (0.2 + 3.4j, 1.0)]


@pytest.mark.parametrize("film", [None, (1.38, 0.1), (1.0, 0.3), (2.3, 0.05), (1.0, 0.0), (1.38 + 0.02j, 0.2)])
@pytest.mark.parametrize("n", range(len(GLASS)))
def test_interface_angles(gpu, n, film):
    n_in, n_out = GLASS[n]
    kw = dict(n_inside=n_in, n_outside=n_out, reflection_threshold=0.0, transmission_threshold=0.0)
    mat = FullDielectricMaterial(**kw) if film is None else \
        SingleLayerCoatedMaterial(n_coating=film[0], thickness=film[1], **kw)
    rng = np.random.default_rng(60 + n)
    th = np.concatenate([[0.0, 1e-12, 1e-6], np.linspace(0.01, 1.55, 300)])
    th = np.concatenate([th, np.pi - th])
    m = len(th)
    r = random_rays(m, 61, wl_count=2)
    ph = rng.uniform(0, 2 * np.pi, m)
    r["direction"] = np.column_stack([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th)])
    e = np.cross(r["direction"], rng.normal(size=(m, 3)))
    r["E_vector"] = e / np.linalg.norm(e, axis=1)[:, None]
    wl = np.array([0.5, 0.8])
    pts, nrm, tan = rng.uniform(-2, 2, (m, 3)), np.tile([0.0, 0.0, 1.0], (m, 1)), np.tile([1.0, 0.0, 0.0], (m, 1))
    got, counts = _queries.eval_child_rays_batch(mat, r, 0, pts, nrm, tan, wl)
    t, mi = scene_of_material(mat)
    ref = [oracle.eval_child_ray(t, mi, r[i:i + 1], i, pts[i], nrm[i], tan[i], wl) for i in range(m)]
    want = np.array([len(x) for x in ref])
    ok = counts == want
    # an amplitude that vanishes but for rounding (equal indices, a film of
    # zero thickness between them) may or may not pass a threshold of zero
    assert ok.all() or (n_in == n_out), np.nonzero(~ok)[0]
    starts = np.concatenate([[0], np.cumsum(counts)])
    # the reference's transmitted amplitude is M10 + M11 r, a difference of
    # terms e^(2 Re phi) times itself in a film beyond its critical angle: it
    # keeps 2e-16 e^(2 Re phi) of it, below 1e-9 for Re phi < 7.6.  Past 7 only
    # the reflected child is compared
    damped = np.zeros(m)
    if film is not None:
        n1 = np.where(np.cos(th) < 0, n_out, n_in).astype(complex)
        s2 = (n1 * np.sin(th) / film[0]) ** 2
        phi = -1j * 2 * np.pi * film[1] / wl[r["wavelength_idx"]] * (film[0] - s2) / np.sqrt(1 - s2 + 0j)
        damped = np.abs(phi.real)
    for i in np.nonzero(ok)[0]:
        a, b = got[starts[i]:starts[i + 1]], ref[i]
        if n_in == n_out and (film is None or film[1] == 0.0):   # the transmitted ray alone: the reflected one vanishes
            a, b = a[-1:], b[-1:]
        elif damped[i] > 7.0:
            a, b = a[:1], b[:1]
        compare_generation(a, b, what="%s %s at %g" % (GLASS[n], film, th[i]))


def test_split_follows_float64(gpu):
    """The FP32-split form of the same interfaces: total reflection inside a
    coated slab, hits and counts as in float64."""
    fl = FaceList()
    faces = _faces()
    for f, (a, b) in zip((faces[4], faces[0]), ((1.0, 1.6), (1.6, 1.0))):
        f.material = SingleLayerCoatedMaterial(n_inside=a, n_outside=b, n_coating=1.38, thickness=0.1,
                                               reflection_threshold=0.02, transmission_threshold=0.02)
    fl.faces = [faces[4], faces[0]]
    r = crossing_rays(4000, 12, False)
    wl = np.array([0.55])
    rc = RayCollection.from_array(r)
    rc.wavelengths = wl
    split_in = SplitRayCollection.from_collection(rc)
    a = trace_rays(rc, [fl], recursion_limit=3, max_length=60.0)[0]
    b = trace_rays_split(split_in, [fl], recursion_limit=3, max_length=60.0)[0]
    for x, y in zip(a[:2], b[:2]):
        x, y = x.copy_as_array(), y.to_collection().copy_as_array()
        assert len(x) == len(y)
        same = x["end_face_idx"] == y["end_face_idx"]
        assert same.mean() > 0.999
        scale = np.maximum(np.abs(x["E1_amp"]), np.abs(x["E2_amp"]))
        # float32 amplitudes; rays within 1e-4 of normal incidence turn their basis
        err = np.abs(np.abs(x["E1_amp"]) - np.abs(y["E1_amp"])) / scale
        assert np.quantile(err, 0.999) < 1e-4
