"""The gausslet generation kernel against the oracle at the edges of its tiles:
children held in registers through the placement (none, one, two), a grating's
third order built again after it, parabasal lengths of the last generation
(whose children are not placed), and parabasal rays that miss or leave the
face of their base ray."""
import math

import numpy as np
import pytest

import oracle
from raypier_optics_amd import workloads
from raypier_optics_amd._scene import compile_scene
from raypier_optics_amd.cfaces import CircularFace, SphericalFace
from raypier_optics_amd.cmaterials import (CoatedDispersiveMaterial, DiffractionGratingMaterial,
                                           FullDielectricMaterial, NondispersiveCurve, OpaqueMaterial)
from raypier_optics_amd.ctracer import FaceList, GaussletCollection
from raypier_optics_amd.tracer import trace_rays
from tests.helpers import compare_generation

pytestmark = pytest.mark.gpu

MATERIALS = {
    "none": lambda: OpaqueMaterial(),
    "two": lambda: FullDielectricMaterial(n_inside=1.6, n_outside=1.0, reflection_threshold=0.0,
                                          transmission_threshold=0.0),
    "dispersive": lambda: CoatedDispersiveMaterial(dispersion_inside=workloads.glass(workloads.N_BK7),
                                                   dispersion_outside=NondispersiveCurve(1.0),
                                                   dispersion_coating=NondispersiveCurve(1.38),
                                                   coating_thickness=0.1, reflection_threshold=0.0,
                                                   transmission_threshold=0.0),
    "three": lambda: DiffractionGratingMaterial(lines_per_mm=300, orders=(-1, 0, 1), efficiency=0.3),
}


@pytest.mark.parametrize("name", sorted(MATERIALS))
@pytest.mark.parametrize("n", [1, 65, 256, 257])
def test_gausslet_generation(gpu, n, name):
    rng = np.random.default_rng(n)
    r = workloads.base_rays(n)
    # a sphere of 4.05 mm radius: base rays up to 3.8 mm from its axis with
    # parabasal rays 0.6 mm to their side, so that some gausslets lose their
    # children (apertures do not hold for parabasal rays)
    rad, phi = 3.8 * np.sqrt(rng.uniform(0, 1, n)), rng.uniform(0, 2 * math.pi, n)
    rad[0] = 1.0
    r["origin"] = np.column_stack([rad * np.cos(phi), rad * np.sin(phi), np.full(n, -10.0)])
    d = np.column_stack([rng.uniform(-0.01, 0.01, (n, 2)), np.ones(n)])
    r["direction"] = d / np.linalg.norm(d, axis=1)[:, None]
    e = np.cross(r["direction"], (0.0, 1.0, 0.0))
    r["E_vector"] = e / np.linalg.norm(e, axis=1)[:, None]
    r["E1_amp"] = rng.normal(size=n) + 1j * rng.normal(size=n)
    r["E2_amp"] = rng.normal(size=n) + 1j * rng.normal(size=n)
    r["refractive_index"] = 1.0
    r["wavelength_idx"] = rng.integers(0, 3, n)
    wl = np.array([0.45, 0.55, 0.65])
    g = GaussletCollection.from_rays(r)
    g.config_parabasal_rays(wl, 0.6, 0.0)
    g.wavelengths = wl
    surf, dets = FaceList(), FaceList()
    surf.faces = [SphericalFace(diameter=8.0, z_height=0.0, curvature=-4.05, material=MATERIALS[name]())]
    dets.faces = [CircularFace(diameter=200.0, z_plane=30.0, material=OpaqueMaterial()),
                  CircularFace(diameter=200.0, z_plane=-25.0, material=OpaqueMaterial())]
    scene = [surf, dets]
    g_in = g.copy_as_array()
    got, faces = trace_rays(g, scene, recursion_limit=2, max_length=200.0)
    counts = [f.count for f in faces]
    workloads.prepare_faces(scene, wl, 200.0)
    ref, hits = oracle.trace_rays(compile_scene(scene), g_in, 200.0, wl, 2, gausslet=True)
    assert len(ref) == (1 if name == "none" else 2)
    if n > 200 and name == "three":
        assert 1.5 * n < len(ref[1]) < 3 * n
    for k, (a, b) in enumerate(zip(got, ref)):
        a = a.copy_as_array()
        compare_generation(a["base_ray"], b["base_ray"], what="%s generation %d" % (name, k))
        for f in ("origin", "direction", "normal", "length"):
            # a parabasal ray beyond the critical angle of its base ray's
            # transmitted child has no direction: not a number in both
            va, vb = a["para_rays"][f], b["para_rays"][f]
            assert np.array_equal(np.isnan(va), np.isnan(vb)), (name, k, f)
            finite = np.isfinite(vb)
            assert np.all(np.abs(va - vb)[finite] <= 1e-9 * np.maximum(np.abs(vb[finite]), 1.0)), (name, k, f)
    assert counts == [int(h) for h in hits[:len(counts)]]
