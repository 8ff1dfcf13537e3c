"""Ray queries where the traversal's short forms meet their limits, against the
oracle bit for bit: scenes and directions scaled by powers of two beyond the
ranges of the short reciprocals and quotients (the full divisions take over),
axis-parallel rays (infinite reciprocals), origins on cell planes, and ray
counts about a wave and a workgroup."""
import numpy as np
import pytest

import pyoracle as O
from gpu_util import SEED, assert_grid_equal, gpu_engine, oracle_grid, random_rays
from happyray_amd import Engine, GRID_TWO_LEVEL, GRID_UNIFORM, GRID_UNIFORM_EXACT, HappyRayError, scenes
from happyray_amd._lib import STATUS_NAMES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh_exp,dir_exp", [(0, 0), (0, -70), (0, 60), (-35, -35), (-35, -55), (30, 30),
                                              (42, 42)])
@pytest.mark.parametrize("kind,lt,ll", [(GRID_TWO_LEVEL, 0.25, 2.2), (GRID_UNIFORM, 5.0, 1.0),
                                        (GRID_UNIFORM_EXACT, 5.0, 1.0)])
def test_scaled_scenes_and_directions(kind, lt, ll, mesh_exp, dir_exp):
    sc = scenes.random_soup(5, 3000, extent=8.0, size=0.6)
    org, d = random_rays(sc, 4096, seed=6)
    # some origins on the planes of an 8-cell lattice through the scene
    org[:, :256] = np.round(org[:, :256])
    sc.verts = np.ldexp(sc.verts, mesh_exp).astype(np.float32)
    org = np.ldexp(org, mesh_exp).astype(np.float32)
    d = np.ldexp(d, dir_exp).astype(np.float32)
    e = gpu_engine(sc, kind, lt, ll)
    og = oracle_grid(sc, kind, lt, ll)
    tmax = float(np.float32(np.ldexp(2.0, mesh_exp - dir_exp)))
    for n in (1, 63, 65, 1023, 4096):
        o, q = org[:, -n:], d[:, -n:]      # the last rays are the axis-parallel ones
        t_o, p_o, _ = O.trace(og, o, q)
        s_o, _, _ = O.trace(og, o, q, anyhit=True, tmax=tmax)
        for batch in (1, 0):
            e.set_tuning(test_batch=batch)
            t, p = e.trace(o, q)
            np.testing.assert_array_equal(t.view(np.uint32), t_o.view(np.uint32))
            np.testing.assert_array_equal(p, p_o)
            np.testing.assert_array_equal(e.occluded(o, q, tmax), (s_o < tmax).astype(np.uint8))
    if (mesh_exp, dir_exp) in ((0, 0), (0, -70), (-35, -35), (-35, -55), (30, 30)):
        assert (p_o < sc.nt).mean() > 0.5   # the scaled rays do hit
    e.close()


def test_leaf_counts_past_32_bits_are_refused():
    """A cell volume so small that leaf density / volume overflows asks for 255^3
    leaves in each of 729 cells: more than 2^32, which the build refuses."""
    sc = scenes.random_soup(5, 3000, extent=8.0, size=0.6)
    keep = sc.verts.copy()
    sc.verts = np.ldexp(sc.verts, -42).astype(np.float32)
    with pytest.raises(HappyRayError) as ex:
        gpu_engine(sc, GRID_TWO_LEVEL, 0.25, 2.2)
    assert STATUS_NAMES[ex.value.status] == "HR_ERR_CAPACITY"
    sc.verts = keep
    gpu_engine(sc, GRID_TWO_LEVEL, 0.25, 2.2).close()


def test_candidates_of_a_wave_past_32_bits_are_refused():
    """64 walls across a grid of 8e7 cells have 5e9 candidate cells, past 2^32,
    though the few cells that they cross would fit: an exact grid whose sum of
    candidates wrapped would miss references.  The build refuses it, and the
    engine builds and answers as before afterwards."""
    rng = np.random.default_rng(3)
    sc = scenes.random_soup(5, 80, extent=8.0, size=0.6)
    v = sc.verts.reshape(3, -1, 3)
    keep = sc.verts.copy()
    corner = rng.integers(0, 2, (80, 3)) * 8.0
    v[:, :, 0], v[:, :, 1] = corner.T, 8.0 - corner.T       # every triangle's box is the scene's
    v[:, :, 2] = np.clip(v[:, :, 2], 0.0, 8.0)
    sc.verts = np.ascontiguousarray(v.reshape(3, -1)).astype(np.float32)
    e = Engine(seed=SEED)
    for _ in range(2):
        e.upload_scene(sc)
        e.set_grid(GRID_UNIFORM_EXACT, 9.9e5, 1.0)
        with pytest.raises(HappyRayError) as ex:
            e.build_acc_struct()
        assert STATUS_NAMES[ex.value.status] == "HR_ERR_CAPACITY"
        e.upload(keep, None, 1.0, sc.idx)
        e.set_grid(GRID_UNIFORM_EXACT, 5.0, 1.0)
        e.build_acc_struct()
        sc.verts, walls = keep, sc.verts
        og = oracle_grid(sc, GRID_UNIFORM_EXACT, 5.0, 1.0)
        assert_grid_equal(e, og)
        sc.verts = walls
    e.close()
