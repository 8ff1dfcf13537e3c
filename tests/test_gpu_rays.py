"""Ray records on the GPU (24 bytes per ray, origin xyz then direction xyz;
SimpleRayTraverser.h:200-262, AORayExporter.h:50-68): record entry points
equal the SoA ones, input rays through the simple integrator and the AO ray
dump equal the oracle, and server requests carrying records equal the same
requests carrying SoA planes."""
import time

import numpy as np
import pytest

import pyoracle as O
from gpu_util import SEED, gpu_engine, oracle_grid, random_rays
from happyray_amd import Engine, GRID_TWO_LEVEL, GRID_UNIFORM, GRID_UNIFORM_EXACT, MODE_AO, MODE_PATH, Server, rayfile, scenes
from happyray_amd.devmem import DeviceArray
from happyray_amd.server import REQ_CLOSEST, REQ_OCCLUDED, REQ_PATH

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,lt,ll", [(GRID_UNIFORM_EXACT, 5.0, 1.0), (GRID_TWO_LEVEL, 0.5, 3.0)])
def test_records_equal_planes_and_oracle(kind, lt, ll):
    sc = scenes.icosphere_cluster(res=64)
    print(f"ray records kind={kind}", flush=True)
    e = gpu_engine(sc, kind, lt, ll)
    og = oracle_grid(sc, kind, lt, ll)
    org, d = random_rays(sc, 20000, seed=17)
    rec = rayfile.to_records(org, d)
    t0, p0 = e.trace(org, d)
    t1, p1 = e.trace_records(rec)
    np.testing.assert_array_equal(t0, t1)
    np.testing.assert_array_equal(p0, p1)
    ext = float((sc.verts.max(1) - sc.verts.min(1)).max())
    np.testing.assert_array_equal(e.occluded(org, d, 0.1 * ext), e.occluded_records(rec, 0.1 * ext))
    rgb = e.render_rays(rec)
    rgb_o, _ = O.render_rays_simple(og, rec, nthreads=8)
    np.testing.assert_array_equal(rgb, rgb_o)
    # the AO dump of a jittered image 2
    e.set_camera_dict(sc.camera)
    e.render_frame(2, MODE_AO, jitter=1, ao_samples=3, ao_dist=1.5)
    dump = e.dump_ao_rays(3)
    cam = O.camera(sc.camera["pos"], sc.camera["dir"], sc.camera["up"], sc.camera["fov"], *sc.camera["res"])
    dump_o = O.dump_ao_rays(og, cam, O.params(seed=SEED, jitter=1, ao_samples=3, ao_dist=1.5, nthreads=8), 2)
    np.testing.assert_array_equal(dump, dump_o)
    e.close()


def test_server_record_payloads():
    sc = scenes.icosphere_cluster(res=48)
    srv = Server(seed=SEED)
    sid = srv.add_scene(sc.verts[None].copy(), sc.idx, sc.materials, sc.mat_idx, sc.lights)
    org, d = random_rays(sc, 5000, seed=23)
    rec = rayfile.to_records(org, d)
    ext = float((sc.verts.max(1) - sc.verts.min(1)).max())
    a = [srv.submit_closest(sid, org, d), srv.submit_occluded(sid, org, d, 0.2 * ext),
         srv.submit_path(sid, org, d, depth=3)]
    b = [srv.submit_records(REQ_CLOSEST, sid, rec), srv.submit_records(REQ_OCCLUDED, sid, rec, tmax=0.2 * ext),
         srv.submit_records(REQ_PATH, sid, rec, depth=3)]
    for x, y in zip(a, b):
        ox, oy = x.wait(), y.wait()
        if isinstance(ox, tuple):
            for u, v in zip(ox, oy):
                np.testing.assert_array_equal(u, v)
        else:
            np.testing.assert_array_equal(ox, oy)
    srv.close()


@pytest.mark.parametrize("n", [1, 5, 1024, 1025, 2049, 20001, 65535, 65537, 400001,
                               3300001, 6800003])
@pytest.mark.parametrize("kind", [GRID_TWO_LEVEL, GRID_UNIFORM_EXACT])
def test_launch_sizes(kind, n):
    """From one ray per wave over waves that are partly filled to launches whose
    waves fetch more rays: the batched kernels, the per-lane persistent ones and
    the one-ray-per-lane kernels agree on every ray and path."""
    sc = scenes.icosphere_cluster(n_spheres=6, subdiv=3)
    e = gpu_engine(sc, kind, 1.0, 2.2)
    e.set_lights(sc.lights)
    org, d = random_rays(sc, n, seed=n)
    out = []
    for batch, pers in ((1, 1), (0, 1), (0, 0)):
        e.set_tuning(test_batch=batch, persistent_secondary=pers)
        out.append([*e.trace(org, d), e.occluded(org, d, 1.5), e.path_trace(org, d, 3)])
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            np.testing.assert_array_equal(np.asarray(a), np.asarray(b))
    assert n < 1000 or 0.02 < out[0][2].mean() < 0.98
    e.close()


@pytest.mark.parametrize("res", [(1, 1), (9, 7), (130, 63), (257, 256), (700, 600)])
def test_camera_kernels_agree_on_small_and_large_images(res):
    sc = scenes.icosphere_cluster(n_spheres=6, subdiv=3)
    e = gpu_engine(sc, GRID_TWO_LEVEL, 0.25, 2.2)
    e.set_lights(sc.lights)
    e.set_camera_dict(dict(sc.camera, res=res))
    out = []
    for pp in (0, 1, 3):
        e.set_tuning(persistent_primary=pp)
        out.append([e.render_frame(0, MODE_PATH, jitter=1, pt_depth=3), *e.primary_hits(),
                    e.render_frame(0, MODE_AO, jitter=1, ao_samples=3, ao_dist=1.5)])
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            np.testing.assert_array_equal(np.asarray(a), np.asarray(b))
    e.close()


@pytest.mark.parametrize("n", [1, 5, 255, 1000, 4097, 70001, 400001])
@pytest.mark.parametrize("kind", [GRID_TWO_LEVEL, GRID_UNIFORM_EXACT])
def test_counts_at_launch_sizes(kind, n):
    """The batched kernels add a workgroup's ray and work counts together: the
    totals are those of the kernels that add per wave, for closest hits,
    occlusion rays, paths, and the frames of each integrator."""
    sc = scenes.icosphere_cluster(n_spheres=6, subdiv=3)
    e = gpu_engine(sc, kind, 1.0, 2.2)
    e.set_lights(sc.lights)
    w = max(1, int(n ** 0.5))
    e.set_camera_dict(dict(sc.camera, res=(w, (n + w - 1) // w)))
    org, d = random_rays(sc, n, seed=n)
    got = []
    for batch, pers, pp in ((1, 1, 3), (0, 1, 1), (0, 0, 0)):
        e.set_tuning(test_batch=batch, persistent_secondary=pers, persistent_primary=pp)
        counts = []
        for step in (lambda: e.trace(org, d), lambda: e.occluded(org, d, 1.5),
                     lambda: e.path_trace(org, d, 3),
                     lambda: e.render_frame(0, MODE_PATH, jitter=1, pt_depth=3, collect_stats=True),
                     lambda: e.render_frame(0, MODE_AO, jitter=1, ao_samples=1, ao_dist=1.5, collect_stats=True)):
            e.work_stats()
            r0 = e.timing().rays_traced
            step()
            ws = e.work_stats()
            counts.append((e.timing().rays_traced - r0, ws.primary.rays, ws.primary.steps, ws.primary.tests,
                           ws.secondary.rays, ws.secondary.steps, ws.secondary.tests))
        got.append(counts)
    assert got[0] == got[1] == got[2]
    assert got[0][0][0] == n and got[0][1][0] == n
    e.close()


@pytest.mark.parametrize("n", [1000, 4000])
def test_counters_do_not_bound_small_launches(n):
    """1,000 rays are 1,000 waves of one ray each.  Adding the counts of every
    wave to the device counters by itself takes 1.8 times as long as the per-lane
    kernel of 16 waves takes for these short occlusion rays; by workgroup, 0.7."""
    sc = scenes.random_soup(5, 7000, extent=10.0, size=0.3)
    e = gpu_engine(sc, GRID_UNIFORM, 4.26, 2.0)
    rng = np.random.default_rng(n)
    d = rng.normal(0, 1, (3, n))
    org = DeviceArray.from_host(rng.uniform(0, 10, (3, n)).astype(np.float32))
    dirs = DeviceArray.from_host((d / np.linalg.norm(d, axis=0)).astype(np.float32))
    occ = DeviceArray((n,), np.uint8)

    def calls(k):
        t = time.perf_counter()
        for _ in range(k):
            e.occluded_dev(org.value, dirs.value, n, 0.5, occ.value)
        e.synchronize()
        return (time.perf_counter() - t) / k

    best = {}
    for _ in range(8):                      # the two in turn, the least of each
        for batch in (1, 0):
            e.set_tuning(test_batch=batch)
            calls(20)
            best[batch] = min(best.get(batch, 1.0), calls(200))
    print(f"{n} occlusion rays: batched {best[1] * 1e6:.1f} us, per lane {best[0] * 1e6:.1f} us", flush=True)
    assert best[1] < 1.15 * best[0]
    e.close()


def in_room(verts, idx):
    """The mesh inside a room of 768 triangles, so that every path ends on something."""
    lo, hi = verts.min(1).astype(np.float64), verts.max(1).astype(np.float64)
    m = 0.35 * np.linalg.norm(hi - lo)
    lo, (x, y, z) = lo - m, np.diag(hi - lo + 2 * m)
    walls = [scenes.quad_grid(o, u, v, 8, 8) for o, u, v in ((lo, y, z), (lo + x, z, y), (lo, z, x), (lo + y, x, z),
                                                           (lo, x, y), (lo + z, y, x))]
    base = np.cumsum([verts.shape[1]] + [len(w[0]) for w in walls])
    return (np.concatenate([verts] + [w[0].T.astype(np.float32) for w in walls], 1),
            np.concatenate([idx] + [w[1] + np.uint32(k) for w, k in zip(walls, base)]).astype(np.uint32))


@pytest.mark.parametrize("mesh,kind,density", [(scenes.sphere_cluster_n, GRID_TWO_LEVEL, 1.2),
                                               (scenes.soup_n, GRID_UNIFORM, 5.0)])
def test_paths_of_several_contexts_share_the_gpu(mesh, kind, density):
    """Three contexts that trace 80,000 paths each in turn: their launches are
    spread over more waves than 64 paths a wave make, for the sake of one alone,
    but not at the cost of each other.  Spread over all the waves that fit they
    reach 0.53 to 0.57 of the paths a second of launches of 240,000 (full waves either
    way), over half of them 0.70 to 0.74."""
    def rate(n):
        es, bufs = [], []
        for k in range(3):
            verts, idx = in_room(*mesh(1 + k, 20480))
            e = Engine(seed=SEED)
            e.upload(verts, None, 1.0, idx)
            e.set_grid(kind, density, 2.2)
            e.upload_materials(np.stack([scenes.material((0.2, 0.18, 0.15))]))
            lo, hi = verts.min(1).astype(np.float64), verts.max(1).astype(np.float64)
            c, ext = (lo + hi) / 2, hi - lo
            e.set_lights(scenes.area_light((c[0] - 0.1 * ext[0], hi[1] - 0.2 * ext[1], c[2] - 0.1 * ext[2]),
                                           (0.2 * ext[0], 0.0, 0.0), (0.0, 0.0, 0.2 * ext[2]), (30.0, 30.0, 30.0))[None])
            e.build_acc_struct()
            eye = (c + 0.43 * ext)[:, None]
            d = verts[:, np.random.default_rng(k).integers(0, verts.shape[1] - 6 * 81, n)] - eye
            bufs.append((DeviceArray.from_host(np.broadcast_to(eye, (3, n)).astype(np.float32)),
                         DeviceArray.from_host((d / np.linalg.norm(d, axis=0)).astype(np.float32)),
                         DeviceArray((n, 3), np.float32)))
            es.append(e)

        def turns(k):
            t = time.perf_counter()
            for _ in range(k):
                for e, (o, q, rgb) in zip(es, bufs):
                    e.path_trace_dev(o.value, q.value, n, 4, rgb.value)
            for e in es:
                e.synchronize()
            return (time.perf_counter() - t) / k

        turns(3)
        best = min(turns(20) for _ in range(6))
        for e in es:
            e.close()
        return 3 * n / best

    small, large = rate(80000), rate(240000)
    print(f"paths/us: {small * 1e-6:.0f} at 80,000 a launch, {large * 1e-6:.0f} at 240,000", flush=True)
    assert small > 0.6 * large


# the flat kernel has at most six workgroups per CU, so rays past 393,216 come
# from the counter: as lanes fall idle, in runs of 64 from 3.1M rays on, of 128
# from 6.3M and of 256, the longest, from 12.6M
@pytest.mark.parametrize("n,refills", [(450001, (1, 16, 48, 56, 64)), (3300001, (1, 64)), (6800003, (24,)),
                                       (12900001, (56,))])
@pytest.mark.parametrize("kind", [GRID_TWO_LEVEL, GRID_UNIFORM])
def test_rays_from_the_counter(kind, n, refills):
    """Launches whose waves fetch rays past their first ones, at several
    thresholds: every ray and the work counts are the one-ray-per-lane kernels'."""
    sc = scenes.icosphere_cluster(n_spheres=6, subdiv=3)
    e = gpu_engine(sc, kind, 1.0, 2.2)
    org, d = random_rays(sc, n, seed=n)

    def query():
        e.work_stats()
        out = [*e.trace(org, d), e.occluded(org, d, 1.5)]
        ws = e.work_stats().secondary
        return out, (ws.rays, ws.steps, ws.tests)

    e.set_tuning(persistent_secondary=0)
    want, counts = query()
    for refill in refills:
        e.set_tuning(persistent_secondary=1, refill=refill)
        got, c = query()
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, b)
        assert c == counts, (refill, c, counts)
    assert 0.02 < want[2].mean() < 0.98
    e.close()
