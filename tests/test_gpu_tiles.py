"""GPU tests of how the engine's kernels share out a queue: a work-group's first tile is its own index,
later ones are claimed, and work-groups without one leave.

The image of a job does not depend on how its paths are shared out, so each image must equal to
the bit the plain form's, whose grids cover the queue (one tile a work-group, nothing claimed).
With 64 work-items a group and one group a compute unit the grid is 64 x (compute units)
entries wide; the sizes lie around one grid, a few grids, and a single entry.

A pass starts its pixels by 8 x 8 tiles, narrower at the right and lower at the bottom edge; images
of less than a tile, of one, and with every kind of edge equal the oracle's sample for sample (its
paths differ from the device's where a sqrt or a sine rounds differently: the bound of the
engine's other oracle tests).
"""
import numpy as np
import pytest

import little_renderer_amd as lr
from glow_scenes import glow_scene
from oracle import lro

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def world():
    assert torch.cuda.is_available(), "these tests need the GPU"
    ctx = lr.Context(0)
    sc = lr.batch_scene(2000, 5)
    ps = lr.PtScene(ctx, sc["prims"], sc["tris"], sc["mats"], 0, sc["eps"], sc["margin"])
    yield ctx, ps
    ctx.close()


def image(eng, i, w, h):
    t = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    eng.image(i, t)
    eng.release(i)
    return t.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("tile", [1, 4])
@pytest.mark.parametrize("grids, off", [(0, 1), (0, 65), (1, -1), (1, 0), (1, 1), (3, 17)])
def test_batched_equals_plain_at_the_grid_s_edges(world, grids, off, tile):
    ctx, ps = world
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n = grids * 64 * cus + off                     # entries of the first iteration's queue
    w = next(x for x in range(int(n ** 0.5), 0, -1) if n % x == 0)
    h = n // w
    eng = lr.Engine(ctx, slots_log2=18, max_tree_depth=max(64, ps.info()[0]), image_bytes=64 << 20)
    eng.tune = {"block_trace": 64, "stack": 16, "block_shade": 64, "blocks_per_cu": 1, "tile": tile, "iters_per_graph": 3}
    job = lr.make_job(ps, lr.batch_camera(9, w, h), w, h, 2, seed=n)
    i = eng.submit(job)
    eng.drain()
    got = image(eng, i, w, h)
    want = image(eng, eng.plain(job), w, h)
    assert np.array_equal(got, want)
    assert np.any(got[..., :3])
    eng.close()


def test_more_jobs_in_a_tile_than_a_work_group_counts_apart(world):
    # 97 jobs of 3 x 2 to 9 x 8 pixels at once: their paths share tiles, and job slots 32 apart
    # meet in a work-group's counters; every job ends, with the image it has alone
    ctx, ps = world
    eng = lr.Engine(ctx, slots_log2=12, max_tree_depth=max(64, ps.info()[0]), image_bytes=16 << 20)
    sizes = [(3 + k % 7, 2 + k % 7) for k in range(97)]
    jobs = [lr.make_job(ps, lr.batch_camera(k, w, h), w, h, 1 + k % 3, seed=k) for k, (w, h) in enumerate(sizes)]
    ids = [eng.submit(j) for j in jobs]
    eng.drain()
    got = [image(eng, i, w, h) for i, (w, h) in zip(ids, sizes)]
    for j, g, (w, h) in zip(jobs, got, sizes):
        assert np.array_equal(g, image(eng, eng.plain(j), w, h))
    eng.close()


@pytest.mark.parametrize("graphs", [1, 2, 5])
def test_a_scene_of_several_lights_joins_while_shadow_rays_wait(world, graphs):
    # shadow rays wait for the next iteration's walks: those a one-light shade left are walked by the
    # kernels for several lights and two-level scenes once a job that needs them is submitted
    ctx, ps = world
    _, (mtris, first, mats, inst) = glow_scene(box=True)
    glow = lr.PtScene.instanced(ctx, mtris, first, mats, inst, eps=2e-3)
    glow.set_sky(lr.sky(64))
    eng = lr.Engine(ctx, slots_log2=15, max_tree_depth=max(64, ps.info()[0], glow.info()[0]), image_bytes=16 << 20)
    eng.tune = {"iters_per_graph": 1}
    a = lr.make_job(ps, lr.batch_camera(11, 190, 110), 190, 110, 3, seed=1)
    b = lr.make_job(glow, lr.camera_make((-200, 20, 0), (0, 20, 0), (0, 1, 0), 40.0, 1.5), 90, 60, 2, seed=2)
    i = eng.submit(a)
    eng.pump(graphs)
    j = eng.submit(b)
    eng.drain()
    got = image(eng, i, 190, 110), image(eng, j, 90, 60)
    assert np.array_equal(got[0], image(eng, eng.plain(a), 190, 110))
    assert np.array_equal(got[1], image(eng, eng.plain(b), 90, 60))
    eng.close()
    glow.close()


@pytest.mark.parametrize("block_shade", [64, 128, 256])
@pytest.mark.parametrize("w, h, spp", [(901, 613, 1), (1024, 1024, 3)])
def test_ordered_bounce_rays_change_no_image(world, w, h, spp, block_shade):
    # enough bounce rays (from 262,144 on) of a scene of over 1000 shapes: the walk takes them by
    # direction, in windows of every size with a ragged last one; the plain form takes them as queued
    ctx, ps = world
    eng = lr.Engine(ctx, slots_log2=22, max_tree_depth=max(64, ps.info()[0]), image_bytes=64 << 20)
    eng.tune = {"block_shade": block_shade}
    job = lr.make_job(ps, lr.batch_camera(4, w, h), w, h, spp, seed=w)
    i = eng.submit(job)
    eng.drain()
    got = image(eng, i, w, h)
    assert np.array_equal(got, image(eng, eng.plain(job), w, h))
    assert np.any(got[..., :3])
    eng.close()


@pytest.mark.parametrize("on", [1, 2])
def test_profiled_launches(world, on):
    # timed alone (1) each walk is a launch an iteration, as they go otherwise (2) both are one
    ctx, ps = world
    eng = lr.Engine(ctx, slots_log2=15, max_tree_depth=max(64, ps.info()[0]), image_bytes=16 << 20)
    job = lr.make_job(ps, lr.batch_camera(11, 190, 110), 190, 110, 3, seed=1)
    eng.profiling(on)
    i = eng.submit(job)
    eng.drain()
    eng.profiling(False)
    st = eng.stats()
    n = st.kernel_launches[0]
    assert list(st.kernel_launches) == [n, n, n, n if on == 1 else 0] and n > 0
    assert all((st.kernel_ms[k] > 0) == (st.kernel_launches[k] > 0) for k in range(4))
    assert np.array_equal(image(eng, i, 190, 110), image(eng, eng.plain(job), 190, 110))
    eng.close()


def test_coincident_shapes_alike_in_both_launches(world):
    # the walks' one launch orders a node's children by other instructions than their own launches:
    # triangles given twice, in two materials, tell one order from another
    ctx, _ = world
    sc = lr.batch_scene(3000, 8)
    t = np.asarray(sc["tris"], np.float32).copy()
    again = t.copy()
    w = again[:, 11].view(np.uint32)
    again[:, 11] = ((((w >> 26) + 1) % len(sc["mats"]) << 26) | (w & 0x3ffffff)).view(np.float32)
    both = np.concatenate([t, again])[np.random.default_rng(2).permutation(2 * len(t))]
    ps = lr.PtScene(ctx, sc["prims"], both, sc["mats"], 0, sc["eps"], sc["margin"])
    eng = lr.Engine(ctx, slots_log2=18, max_tree_depth=max(64, ps.info()[0]), image_bytes=16 << 20)
    job = lr.make_job(ps, lr.batch_camera(9, 300, 200), 300, 200, 3, seed=6)
    got = []
    for on in (0, 1, 2):
        eng.profiling(on)
        i = eng.submit(job)
        eng.drain()
        got.append(image(eng, i, 300, 200))
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    eng.close()
    ps.close()


def test_a_scene_whose_eps_is_not_from_zero_up(world):
    # its rays' tmin takes the walks' own launches while a job of it runs; the images of both forms agree
    ctx, other = world
    sc = lr.batch_scene(2000, 5)
    ps = lr.PtScene(ctx, sc["prims"], sc["tris"], sc["mats"], 0, -1e-4, sc["margin"])
    eng = lr.Engine(ctx, slots_log2=16, max_tree_depth=max(64, ps.info()[0]), image_bytes=16 << 20)
    before = lr.make_job(other, lr.batch_camera(9, 80, 60), 80, 60, 2, seed=6)
    i = eng.submit(before)
    eng.drain()
    alone = image(eng, i, 80, 60)
    job = lr.make_job(ps, lr.batch_camera(9, 80, 60), 80, 60, 2, seed=6)
    i, j = eng.submit(job), eng.submit(before)
    eng.drain()
    assert np.array_equal(image(eng, j, 80, 60), alone)
    assert np.array_equal(image(eng, i, 80, 60), image(eng, eng.plain(job), 80, 60))
    eng.profiling(2)
    for k, apart in ((job, True), (before, False)):
        n0 = list(eng.stats().kernel_launches)
        i = eng.submit(k)
        eng.drain()
        eng.release(i)
        n1 = list(eng.stats().kernel_launches)
        assert n1[1] > n0[1] and n1[3] - n0[3] == (n1[1] - n0[1] if apart else 0)
    eng.close()
    ps.close()


@pytest.mark.parametrize("w, h", [(1, 1), (3, 65), (7, 9), (8, 8), (9, 7), (65, 3), (24, 20)])
def test_ragged_images_match_the_oracle(world, w, h):
    ctx, _ = world
    sc = lr.cornell(w, h)
    ps = lr.PtScene(ctx, sc["prims"], sc["tris"], sc["mats"], 0, sc["eps"], sc["margin"])
    eng = lr.Engine(ctx, slots_log2=14, max_tree_depth=64, image_bytes=16 << 20)
    i = eng.submit(lr.make_job(ps, sc["cam"], w, h, 3, seed=2))
    eng.drain()
    got = image(eng, i, w, h).view(np.float32)
    assert np.all(got[..., 3] == 3)
    want = lro.pt_image(sc, w, h, 0, 3, seed=2, tab=lr.brdf_tables(), mask=lro.blue_noise())
    rel = np.abs(got[..., :3] - want) / np.maximum(np.abs(want), 1e-3)
    assert np.median(rel) < 1e-5 and np.mean(rel > 1e-3) < 0.01
    eng.close()
    ps.close()


def test_bounce_rays_are_ordered_by_the_jobs_that_run(world):
    # the steps of a wave of the extension walk tell the order its rays came in: a small scene's job
    # (never ordered) after a large one's, a large one's (ordered) after an instanced one's, each as
    # in a new engine
    ctx, big = world
    sc = lr.cornell(900, 700)
    small = lr.PtScene(ctx, sc["prims"], sc["tris"], sc["mats"], 0, sc["eps"], sc["margin"])
    _, (mtris, first, mats, inst) = glow_scene(box=True)
    glow = lr.PtScene.instanced(ctx, mtris, first, mats, inst, eps=2e-3)
    glow.set_sky(lr.sky(64))
    depth = max(64, big.info()[0], glow.info()[0])
    jobs = {"small": lr.make_job(small, sc["cam"], 900, 700, 1, seed=3),
            "big": lr.make_job(big, lr.batch_camera(4, 900, 700), 900, 700, 1, seed=4),
            "glow": lr.make_job(glow, lr.camera_make((-200, 20, 0), (0, 20, 0), (0, 1, 0), 40.0, 1.5), 90, 60, 1, seed=2)}

    def steps(*names):
        eng = lr.Engine(ctx, slots_log2=20, max_tree_depth=depth, image_bytes=32 << 20)
        eng.counting(True)
        for k in names:
            before = eng.stats().wave_node_steps
            i = eng.submit(jobs[k])
            eng.drain()
            eng.release(i)
        n = eng.stats().wave_node_steps - before
        eng.close()
        return n

    alone = {k: steps(k) for k in ("small", "big")}
    assert alone["small"] == steps("small")          # (a count to compare by)
    assert steps("big", "small") == alone["small"]
    assert steps("glow", "big") == alone["big"]
    glow.close()
    small.close()
