"""The binary walk where its stack leaves LDS, and where its box tests meet NaNs and infinities:
bit-exact against the oracle's walk of the same tree.

A tree of one long arm (its far children wait one above the other, 10 to a ray in LDS, the rest in
device memory; 16, and none, where that is enough), also with a depth too small given: 16 entries
are always there. And a built tree some of whose boxes and rays hold NaNs, infinities and zeros.
"""
import numpy as np
import pytest

import little_renderer_amd as lr
from oracle import lro

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    assert torch.cuda.is_available(), "these tests need the GPU"
    c = lr.Context(0)
    yield c
    c.close()


def both(ctx, nodes, aux, tris, rays, depth, any_hit):
    d = [torch.from_numpy(a).cuda() for a in (nodes.view(np.int32), aux.view(np.int32), tris, rays)]
    hits = torch.zeros((len(rays), 4), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    ctx.trace(d[0], 0, d[1], d[2], d[3], len(rays), hits, depth, any_hit=any_hit)
    ctx.sync()
    with np.errstate(all="ignore"):
        want = lro.trace_gpu_layout(nodes, 0, aux, tris, rays, any_hit=any_hit)
    return hits.cpu().numpy().view(np.uint32), want.view(np.uint32)


def arm_tree(arm, nrays):
    # node 2k+1: leaf k, far along z; node 2k+2: the arm's next, nearer; triangle k at z = 100 - k
    tris = np.zeros((arm + 1, 12), np.float32)
    for k in range(arm + 1):
        tris[k, 0:3], tris[k, 4:7], tris[k, 8:11] = (-1, -1, 100 - k), (4, 0, 0), (0, 4, 0)
    aux = np.arange(arm + 1, dtype=np.uint32)
    nodes = np.zeros((2 * arm + 1, 8), np.uint32)
    f = nodes.view(np.float32)
    for k in range(arm):
        me = 2 * k
        f[me, 0:3], f[me, 4:7] = (-1, -1, 1 + 0.1 * (arm - k)), (4, 4, 100 - k)
        nodes[me, 3], nodes[me, 7] = 2 * k + 1, 2 * k + 2
        f[2 * k + 1, 0:3], f[2 * k + 1, 4:7] = (-1, -1, 50), (4, 4, 100 - k)
        nodes[2 * k + 1, 3], nodes[2 * k + 1, 7] = k, 0x80000001
    f[2 * arm, 0:3], f[2 * arm, 4:7] = (-1, -1, 1), (4, 4, 100 - arm)
    nodes[2 * arm, 3], nodes[2 * arm, 7] = arm, 0x80000001
    rng = np.random.default_rng(arm)
    rays = np.zeros((nrays, 8), np.float32)
    rays[:, 0:2], rays[:, 2] = rng.uniform(-1.2, 1.2, (nrays, 2)), rng.uniform(-5, 90, nrays)
    rays[:, 3], rays[:, 6], rays[:, 7] = 1e-4, 1.0, 1e30
    return nodes, aux, tris, rays


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("arm", [2, 3, 4, 5, 9, 10, 11, 12, 13, 14, 15, 16, 30])
def test_far_children_past_lds(ctx, arm, any_hit):
    print(f"arm {arm} any {any_hit}", flush=True)
    nodes, aux, tris, rays = arm_tree(arm, 1000)
    got, want = both(ctx, nodes, aux, tris, rays, arm + 1, any_hit)
    assert (want[:, 1] != 0xFFFFFFFF).sum() > 500
    assert np.array_equal(got, want), f"{(got != want).any(1).sum()} rays differ"


@pytest.mark.parametrize("depth", [1, 9, 14])
@pytest.mark.parametrize("arm", [10, 11, 16])
def test_sixteen_entries_whatever_the_depth(ctx, arm, depth):
    print(f"arm {arm} depth {depth}", flush=True)
    nodes, aux, tris, rays = arm_tree(arm, 1000)
    got, want = both(ctx, nodes, aux, tris, rays, depth, False)
    assert np.array_equal(got, want), f"{(got != want).any(1).sum()} rays differ"


@pytest.mark.parametrize("arm", [3, 4, 5, 13, 14, 30])
def test_counts_of_what_is_fetched(ctx, arm):
    # a ray from below takes the whole arm: every far child waits and is popped
    nodes, aux, tris, rays = arm_tree(arm, 700)
    rays[:, 0:3] = (-0.5, -0.5, -5)
    d = [torch.from_numpy(a).cuda() for a in (nodes.view(np.int32), aux.view(np.int32), tris, rays)]
    hits = torch.zeros((len(rays), 4), dtype=torch.float32, device="cuda")
    counts = torch.zeros(2, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    ctx.trace_count(d[0], 0, d[1], d[2], d[3], len(rays), None, hits, arm + 1, counts)
    ctx.sync()
    held = 4 if arm + 1 <= 14 else 10    # entries that hold a child's words
    assert counts.tolist() == [700 * (1 + 2 * arm + max(0, arm - held)), 700 * (arm + 1)]


def test_too_small_a_depth_is_refused(ctx):
    nodes, aux, tris, rays = arm_tree(30, 1000)
    with pytest.raises(lr.LrhError):
        both(ctx, nodes, aux, tris, rays, 20, False)
    got, want = both(ctx, nodes, aux, tris, rays, 31, False)   # (and the context goes on)
    assert np.array_equal(got, want)


def test_shallow_walk_allocates_nothing_under_capture():
    # a first small batch, then a large one captured: no scratch memory of its size, so it may be
    s = torch.cuda.Stream()
    c = lr.Context(0, s.cuda_stream)
    nodes, aux, tris, rays = arm_tree(13, 100_000)
    d = [torch.from_numpy(a).cuda() for a in (nodes.view(np.int32), aux.view(np.int32), tris, rays)]
    hits = torch.zeros((len(rays), 4), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    c.trace(d[0], 0, d[1], d[2], d[3], 100, hits, 14)
    c.sync()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        c.trace(d[0], 0, d[1], d[2], d[3], len(rays), hits, 14)
    want = lro.trace_gpu_layout(nodes, 0, aux, tris, rays).view(np.uint32)
    for _ in range(3):
        hits.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(hits.cpu().numpy().view(np.uint32), want)
    c.close()


@pytest.mark.parametrize("any_hit", [False, True])
def test_boxes_and_rays_with_nan_and_infinity(ctx, any_hit):
    n = 3000
    print(f"odd boxes any {any_hit}", flush=True)
    tris = lr.gen_soup(n, 3)
    nodes, aux, sc, si, depth = lro.build_tris(tris, ploc_=True)
    rng = np.random.default_rng(4)
    f = nodes.view(np.float32)
    odd = np.array([np.nan, np.inf, -np.inf, 0.0, -0.0, 1e38], np.float32)
    for k in rng.integers(300, len(nodes), 400):   # (below the top: the rest of the tree stays in reach)
        f[k, rng.choice([0, 1, 2, 4, 5, 6])] = odd[rng.integers(len(odd))]
    m = 20_000
    o, pick = rng.uniform(0, 1, (m, 3)), tris[rng.integers(0, n, m)]
    tgt = pick[:, 0:3] + (pick[:, 4:7] + pick[:, 8:11]) / 3
    rays = np.zeros((m, 8), np.float32)
    rays[:, 0:3], rays[:, 3], rays[:, 4:7], rays[:, 7] = o, 1e-4, tgt - o, 1e30
    rays[::7, 4 + rng.integers(3)] = 0.0
    rays[::11, rng.integers(7)] = odd[rng.integers(len(odd), size=len(rays[::11]))]
    got, want = both(ctx, nodes, aux, tris, rays, depth, any_hit)
    same = (got == want) | (np.isnan(got.view(np.float32)) & np.isnan(want.view(np.float32)))
    assert (want[:, 1] != 0xFFFFFFFF).sum() > 1000
    assert same.all(), f"{(~same).any(1).sum()} rays differ"
