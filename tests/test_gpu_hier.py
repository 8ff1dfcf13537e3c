"""GPU parity of the instanced two-level grid hierarchy (HR_GRID_HIERARCHY)
against the oracle (or_hier.c) on the same seeded scene: object grids, top
grid, every cell list and reference bit-exact; closest hits (distance,
triangle, instance), occlusion, and the hierarchy's AO frames exact."""
import copy

import numpy as np
import pytest

import pyoracle as O
from gpu_util import SEED
from happyray_amd import Engine, GRID_HIERARCHY, GRID_TWO_LEVEL, HappyRayError, MODE_AO, MODE_PATH, scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def inst_scene():
    return scenes.instanced_scene(seed=6, n_inst=96, n_soup=300, subdiv=3, res=(96, 72))


def _gpu(sc, ins, lt=1.2, ll=2.2, v2=None, coeff=1.0, bounds_blocks=0):
    e = Engine(seed=SEED)
    if bounds_blocks:
        e.set_tuning(hier_bounds_blocks=bounds_blocks)
    if v2 is None:
        e.upload_scene(sc)
    else:
        e.upload(sc.verts, v2, coeff, sc.idx)
        e.upload_materials(sc.materials, sc.mat_idx)
    e.set_instances(ins.obj_first, ins.objects, ins.matrices, ins.aabb_min, ins.aabb_max)
    e.set_grid(GRID_HIERARCHY, lt, ll)
    e.build()
    return e


def _oracle(sc, ins, lt=1.2, ll=2.2, v2=None, coeff=1.0):
    v, bmin, bmax = O.lerp_bounds(sc.verts, sc.verts if v2 is None else v2, coeff)
    mesh = O.OMesh(v[0], v[1], v[2], sc.idx)
    h = O.OHier(mesh, sc.verts, bmin, bmax, ins.obj_first, ins.objects, ins.matrices, ins.aabb_min,
                ins.aabb_max, lt, ll)
    assert h.status == 0
    return h


def _assert_build_equal(e, h):
    info, top, obj_cells, prims = e.grid()
    grids, refs = e.object_grids()
    p = h.top_params()
    assert tuple(info.res) == p["res"]
    for k in ("bmin", "bmax", "cell_size", "cell_size_rcp"):
        np.testing.assert_array_equal(np.array(getattr(info, k)[:], np.float32), p[k])
    assert info.num_cells == h.c.top.num_cells
    assert info.num_leaves == h.c.num_obj_cells
    assert info.num_refs == h.c.num_obj_refs
    assert info.num_top_pairs == h.c.num_inst_refs
    np.testing.assert_array_equal(top, h.top_cells())
    np.testing.assert_array_equal(refs, h.inst_refs())
    for g, o in zip(grids, h.objects()):
        assert list(g["res"]) == list(o["res"])
        assert g["first_cell"] == o["first_cell"] and g["num_cells"] == o["num_cells"]
        for k in ("bmin", "bmax", "cell_size", "cell_size_rcp"):
            np.testing.assert_array_equal(g[k], o[k])
    np.testing.assert_array_equal(obj_cells, h.obj_cells())
    np.testing.assert_array_equal(prims, h.prims())


# bounds_blocks 1 and 3 give each thread of the object-bounds pass a run of
# about 10 and 4 triangles (2,348 triangles), so runs cross object boundaries
@pytest.mark.parametrize("lt,ll,bounds_blocks", [(1.2, 2.2, 0), (8.0, 12.0, 0), (1.2, 2.2, 1), (8.0, 12.0, 3)])
def test_hier_build_parity(inst_scene, lt, ll, bounds_blocks):
    print(f"hierarchy build parity lt={lt} ll={ll} bounds_blocks={bounds_blocks}", flush=True)
    sc, ins = inst_scene
    e = _gpu(sc, ins, lt, ll, bounds_blocks=bounds_blocks)
    _assert_build_equal(e, _oracle(sc, ins, lt, ll))
    e.close()


def test_hier_build_parity_interpolated(inst_scene):
    """Object bounds from the first key frame, triangles from the interpolated
    frame: triangles that left their object grid land in its border cells."""
    print("hierarchy build parity, interpolated frame", flush=True)
    sc, ins = inst_scene
    rng = np.random.default_rng(9)
    v2 = (sc.verts * np.float32(1.15) + rng.normal(0, 0.05, sc.verts.shape)).astype(np.float32)
    e = _gpu(sc, ins, v2=v2, coeff=0.6)
    _assert_build_equal(e, _oracle(sc, ins, v2=v2, coeff=0.6))
    e.close()


def _rays(n, seed, h=10.0):
    rng = np.random.default_rng(seed)
    org = rng.uniform(-0.9 * h, 0.9 * h, size=(3, n)).astype(np.float32)
    d = rng.normal(size=(3, n))
    d /= np.linalg.norm(d, axis=0)
    d[:, :16] = np.eye(3)[:, np.arange(16) % 3]      # axis-parallel rays
    return org, d.astype(np.float32)


def test_hier_trace_parity(inst_scene):
    print("hierarchy trace parity", flush=True)
    sc, ins = inst_scene
    e = _gpu(sc, ins)
    h = _oracle(sc, ins)
    org, dirs = _rays(20000, 3)
    t, prim, inst = e.trace_instanced(org, dirs)
    to, po, io = O.trace_hier(h, org, dirs)
    np.testing.assert_array_equal(t, to)
    np.testing.assert_array_equal(prim, po)
    np.testing.assert_array_equal(inst, io)
    t2, p2 = e.trace(org, dirs)
    np.testing.assert_array_equal(t2, to)
    np.testing.assert_array_equal(p2, po)
    for tmax in (0.5, 2.0, 1e30):
        occ = e.occluded(org, dirs, tmax)
        oo, _ = O.trace_hier(h, org, dirs, anyhit=True, tmax=tmax)
        np.testing.assert_array_equal(occ, oo)
    e.close()


@pytest.mark.parametrize("pp,pers,refill", [(0, 0, 12), (1, 1, 1), (0, 1, 12), (1, 1, 64)])
def test_hier_ao_parity(inst_scene, pp, pers, refill):
    """AO frames of the hierarchy, with the camera and AO rays in the
    one-ray-per-lane kernels and in the persistent kernel at several refill
    thresholds."""
    print(f"hierarchy AO parity persistent primary={pp} ao={pers} refill={refill}", flush=True)
    sc, ins = inst_scene
    e = _gpu(sc, ins)
    e.set_tuning(pp, pers, hier_refill=refill)
    h = _oracle(sc, ins)
    c = sc.camera
    rx, ry = c["res"]
    e.set_camera(c["pos"], c["dir"], c["up"], c["fov"], rx, ry)
    cam = O.camera(c["pos"], c["dir"], c["up"], c["fov"], rx, ry)
    fbo = None
    for image in range(3):
        p = O.params(seed=SEED, ao_samples=4, ao_dist=1.7)
        fbo, occo, hitso, hpo, hio = O.render_ao_hier(h, cam, p, sc.materials, sc.mat_idx, image, fbo)
        fb = e.render_frame(image, MODE_AO, jitter=1, ao_samples=4, ao_dist=1.7)
        planes, prims = e.primary_hits()
        np.testing.assert_array_equal(planes, hitso)
        np.testing.assert_array_equal(prims, hpo)
        np.testing.assert_array_equal(e.primary_instances(), hio)
        np.testing.assert_array_equal(e.ao_occlusion(4), occo)
        np.testing.assert_array_equal(np.asarray(fb).reshape(-1, 3), fbo)
    e.close()


def _transformed(sc, ins, case):
    """The scene with other instance transforms: rotation entries that are zero,
    tiny (past the short divisions' range) or small with objects as small."""
    sc, ins = copy.copy(sc), copy.copy(ins)
    m = ins.matrices.copy()
    if case == "zeros":
        m[:, :3, :3] = np.eye(3, dtype=np.float32)
        m[:, :3, 3] = -(ins.aabb_min + ins.aabb_max) / 2
    elif case == "tiny":
        m[::2, 0, 1] = 1e-25
    else:
        small = np.asarray(ins.objects) > 0          # object 0 is the room, which spans the top grid
        m[small] = np.ldexp(m[small], case).astype(np.float32)
        vid = np.unique(sc.idx[ins.obj_first[1]:])
        sc.verts = sc.verts.copy()
        sc.verts[:, vid] = np.ldexp(sc.verts[:, vid], case).astype(np.float32)
    ins.matrices = m
    return sc, ins


@pytest.mark.parametrize("case", ["zeros", "tiny", -6, 3, -62])
def test_hier_ao_transforms(inst_scene, case):
    """The step into an object where its divisions take the short and the full
    forms, in the batched and the per-lane persistent kernels."""
    sc, ins = _transformed(*inst_scene, case)
    e = _gpu(sc, ins)
    h = _oracle(sc, ins)
    c = sc.camera
    e.set_camera(c["pos"], c["dir"], c["up"], c["fov"], 61, 47)
    cam = O.camera(c["pos"], c["dir"], c["up"], c["fov"], 61, 47)
    p = O.params(seed=SEED, ao_samples=3, ao_dist=1.7)
    _, occo, hitso, hpo, hio = O.render_ao_hier(h, cam, p, sc.materials, sc.mat_idx, 0, None)
    for pp, batch in ((0, 1), (0, 0), (1, 1), (1, 0)):
        e.set_tuning(pp, 1, test_batch=batch)
        e.render_frame(0, MODE_AO, jitter=1, ao_samples=3, ao_dist=1.7)
        planes, prims = e.primary_hits()
        np.testing.assert_array_equal(planes, hitso)
        np.testing.assert_array_equal(prims, hpo)
        np.testing.assert_array_equal(e.primary_instances(), hio)
        np.testing.assert_array_equal(e.ao_occlusion(3), occo)
    assert 0 < occo.mean() < 1
    e.close()


def test_hier_rejects_other_modes_and_missing_instances(inst_scene):
    print("hierarchy error paths", flush=True)
    sc, ins = inst_scene
    e = Engine(seed=SEED)
    e.upload_scene(sc)
    e.set_grid(GRID_HIERARCHY, 1.2, 2.2)
    with pytest.raises(HappyRayError, match="HR_ERR_STATE"):
        e.build()
    e.set_instances(ins.obj_first, ins.objects, ins.matrices, ins.aabb_min, ins.aabb_max)
    e.build()
    c = sc.camera
    e.set_camera(c["pos"], c["dir"], c["up"], c["fov"], 16, 16)
    with pytest.raises(HappyRayError, match="HR_ERR_STATE"):
        e.render_frame(0, MODE_PATH)
    # instance outputs: traces keep their own buffer, a render of another grid
    # kind leaves no primary instances to read
    e.render_frame(0, MODE_AO, ao_samples=2, ao_dist=1.0)
    pi = e.primary_instances()
    org, dirs = _rays(5000, 8)
    e.trace_instanced(org, dirs)
    np.testing.assert_array_equal(e.primary_instances(), pi)
    with pytest.raises(HappyRayError, match="HR_ERR_STATE"):
        e.dump_ao_rays(2)
    e.set_grid(GRID_TWO_LEVEL, 1.2, 2.2)
    e.build()
    e.render_frame(0, MODE_AO, ao_samples=2, ao_dist=1.0)
    with pytest.raises(HappyRayError, match="HR_ERR_STATE"):
        e.primary_instances()
    assert e.dump_ao_rays(2).shape[0] > 0
    e.render_frame(1, MODE_PATH)
    with pytest.raises(HappyRayError, match="HR_ERR_STATE"):
        e.dump_ao_rays(2)
    # the hierarchy's refill threshold is validated like the others
    for bad in (0, 65):
        with pytest.raises(HappyRayError, match="HR_ERR_ARG"):
            e.set_tuning(0, 1, 48, bad)
    assert e.tuning().hier_refill == 12
    e.close()


def test_hier_scene_file(tmp_path):
    """A scene.cfg with an OBJ split by 'o' lines and an instances file, loaded
    and uploaded by the library, against the oracle built from the parsed data."""
    print("hierarchy from scene files", flush=True)
    from happyray_amd import SceneFile
    from scene_files import instanced_scene_files
    sc, ins = scenes.instanced_scene(seed=8, n_inst=40, n_soup=150, res=(48, 36))
    sf = SceneFile.load(instanced_scene_files(str(tmp_path), sc, ins))
    e = Engine(seed=SEED)
    e.load_scene(sf)
    e.set_grid(GRID_HIERARCHY, 1.2, 2.2)
    e.build()
    v = sf.vertices(0)
    idx, _, mat_idx = sf.triangles()
    first, objects, m, lo, hi = sf.instances()
    assert len(objects) == 40 and len(first) == 4
    _, bmin, bmax = O.lerp_bounds(v, v, 0.0)
    h = O.OHier(O.OMesh(v[0], v[1], v[2], idx), v, bmin, bmax, first, objects, m, lo, hi)
    assert h.status == 0
    _assert_build_equal(e, h)
    c = sf.camera
    cam = O.camera(c["pos"], c["dir"], c["up"], c["fov"], c["res"][0], c["res"][1])
    p = O.params(seed=SEED, ao_samples=4, ao_dist=1.0)
    fbo, occo, _, _, hio = O.render_ao_hier(h, cam, p, sf.materials(), mat_idx)
    fb = e.render_frame(0, MODE_AO, jitter=1, ao_samples=4, ao_dist=1.0)
    np.testing.assert_array_equal(e.primary_instances(), hio)
    np.testing.assert_array_equal(e.ao_occlusion(4), occo)
    np.testing.assert_array_equal(np.asarray(fb).reshape(-1, 3), fbo)
    e.close()


def test_hier_full_size_kernels_agree():
    """The benchmark's instanced scene (10,000 instances, 121k-triangle mesh)
    at 640x640 with 4 AO rays per hit: the persistent kernels, the
    one-ray-per-lane kernels and the camera kernel whose waves take 8x8 tiles
    from a counter (six workgroups per CU for 6,400 tiles) give identical
    primary hits, instances and occlusion bits, and every AO ray whose pixel
    has a hit is counted."""
    print("hierarchy full size: persistent vs one ray per lane", flush=True)
    rx, ry = 640, 640
    sc, ins = scenes.instanced_scene(seed=12, n_inst=10000, subdiv=5, n_soup=100000, extent=100.0,
                                     res=(rx, ry), soup_size=0.02)
    e = Engine(seed=SEED)
    e.upload_scene(sc)
    e.set_instances(ins.obj_first, ins.objects, ins.matrices, ins.aabb_min, ins.aabb_max)
    e.set_grid(GRID_HIERARCHY, 1.2, 2.2)
    e.set_camera_dict(sc.camera)
    e.build()
    ao = 0.05 * e.get_bounding_box_diagonal_length()
    out = []
    for pp, pers, refill, cb in ((0, 0, 12, 0), (0, 1, 12, 0), (1, 1, 4, 0), (0, 1, 64, 0), (0, 1, 12, 4)):
        print(f"hierarchy full size: camera kernel {pp} camera_blocks {cb} persistent AO {pers} refill {refill}",
              flush=True)
        e.set_tuning(pp, pers, hier_refill=refill, camera_blocks=cb)
        r0 = e.timing().rays_traced
        fb = e.render_frame(0, MODE_AO, jitter=1, ao_samples=4, ao_dist=ao)
        rays = e.timing().rays_traced - r0
        planes, prims = e.primary_hits()
        out.append((np.asarray(fb), planes, prims, e.primary_instances(), e.ao_occlusion(4), rays))
    hits = int((out[0][2] < sc.nt).sum())
    assert 0 < hits <= rx * ry
    assert out[0][5] == rx * ry + 4 * hits
    for o in out[1:]:
        for a, b in zip(o[:5], out[0][:5]):
            np.testing.assert_array_equal(a, b)
        assert o[5] == out[0][5]
    e.close()
