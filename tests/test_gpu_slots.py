"""GPU tests of the 4-wide slot trees where their shape is unusual, against the oracle's brute force.

Scenes of 1 to 9 shapes (a root that is a leaf, nodes of 2, 3 and 4 children), primitives alone and
mixed with triangles, and a sheaf of long triangles through one point: every box is hit, so the
walks hold more entries than their LDS stack does. The bar is test_gpu_walks': the same hit or
miss, t within 1e-5 relative (another shape only at the same distance), the same any-hit answer.

Where shapes coincide (triangles given two to four times, squares over one another in a plane, rays
through their shared edges) which of them is the hit is the visits' order: there the hits equal the
oracle's 4-wide walk of the same tree to the bit, the first hit of an any-hit ray too.
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


def check(ctx, prims, tris, rays, builder):
    mats = (lr.Material * 1)()
    ps = lr.PtScene(ctx, prims if len(prims) else None, tris if len(tris) else None, mats, -1, 1e-4, 1e-3, builder=builder)
    osc = {"prims": prims, "tris": tris, "mats": mats, "eps": 1e-4, "light": -1}
    want, got = lro.scene_trace(osc, rays), ps.trace(rays)
    wi, gi = want[:, 1].view(np.uint32), got[:, 1].view(np.uint32)
    hit = wi != 0xffffffff
    assert np.array_equal(hit, gi != 0xffffffff)
    assert np.all(np.abs(got[hit, 0] - want[hit, 0]) <= 1e-5 * want[hit, 0])
    any_ = ps.trace(rays, any_hit=True)[:, 1].view(np.uint32) != 0xffffffff
    assert np.array_equal(any_, hit)
    ps.close()
    return hit


def rays_at(tgt, rng, n):
    o = rng.uniform(-0.5, 1.5, size=(n, 3))
    d = tgt[rng.integers(0, len(tgt), n)] + rng.normal(scale=0.05, size=(n, 3)) - o
    r = np.zeros((n, 8), np.float32)
    r[:, 0:3], r[:, 3], r[:, 4:7], r[:, 7] = o, 1e-4, d / np.linalg.norm(d, axis=1, keepdims=True), 1e30
    return r


def tri_records(q, u, v):
    t = np.zeros((len(q), 12), np.float32)
    t[:, 0:3], t[:, 4:7], t[:, 8:11] = q, u, v
    return t


@pytest.mark.parametrize("builder", [lr.LBVH, lr.PLOC])
@pytest.mark.parametrize("nprims, ntris", [(1, 0), (0, 1), (0, 2), (1, 2), (0, 4), (2, 3), (0, 5), (3, 6), (9, 0)])
def test_few_shapes(ctx, nprims, ntris, builder):
    rng = np.random.default_rng(100 * nprims + ntris)
    c = rng.uniform(0, 1, size=(nprims, 3))
    prims = np.stack([lr.sphere_prim(x, 0.15, 0) for x in c]) if nprims else np.zeros((0, 24), np.float32)
    q = rng.uniform(0, 1, size=(ntris, 3))
    u, v = rng.normal(scale=0.4, size=(2, ntris, 3))
    rays = rays_at(np.concatenate([c, q + (u + v) / 3]), rng, 3000)
    hit = check(ctx, prims, tri_records(q, u, v), rays, builder)
    assert 0.2 < hit.mean() < 1.0


@pytest.mark.parametrize("builder", [lr.LBVH, lr.PLOC])
def test_more_entries_than_the_lds_stack(ctx, builder):
    rng = np.random.default_rng(3)
    n = 3000
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    w = rng.normal(scale=1e-3, size=(n, 3))
    tris = tri_records(0.5 - d, 2 * d + w, 2 * d - w)      # slivers from one side of the centre to the other
    rays = rays_at(np.full((1, 3), 0.5), rng, 4000)
    hit = check(ctx, np.zeros((0, 24), np.float32), tris, rays, builder)
    assert 0.02 < hit.mean()


def repeated(rng):
    base = lr.gen_soup(1000, 7)
    t = np.concatenate([np.repeat(base[:400], k, 0) for k in (1, 2, 3, 4)])
    t = t[rng.permutation(len(t))].copy()
    pick = t[rng.integers(0, len(t), 20_000)]
    return t, pick[:, 0:3] + 0.3 * pick[:, 4:7] + 0.3 * pick[:, 8:11]


def squares(rng):
    k = 30
    x, y = np.meshgrid(np.arange(k) / k, np.arange(k) / k)
    p = np.stack([x.ravel(), y.ravel(), np.full(k * k, 0.5)], 1)
    u, v = np.array([1 / k, 0, 0]), np.array([0, 1 / k, 0])
    one = np.ones((k * k, 1))
    t = np.concatenate([tri_records(p, one * u, one * v), tri_records(p + u + v, -one * u, -one * v),
                        tri_records(p, 1.5 * one * u, 1.5 * one * v)])
    tgt = np.full((20_000, 3), 0.5)
    tgt[:, :2] = rng.uniform(0, 1, (20_000, 2))
    tgt[::2, :2] = rng.integers(0, k + 1, (10_000, 2)) / k
    return t, tgt


@pytest.mark.parametrize("builder", [lr.LBVH, lr.PLOC])
@pytest.mark.parametrize("make", [repeated, squares])
def test_which_of_coincident_shapes(ctx, make, builder):
    rng = np.random.default_rng(21)
    tris, tgt = make(rng)
    o = rng.uniform(-0.5, 1.5, size=tgt.shape)
    rays = np.zeros((len(tgt), 8), np.float32)
    d = tgt - o
    rays[:, 0:3], rays[:, 3], rays[:, 4:7], rays[:, 7] = o, 1e-4, d / np.linalg.norm(d, axis=1, keepdims=True), 1e30
    # (a tmin below +0 orders the children by other instructions)
    rays[:8000, 3] = np.repeat(np.array([0.0, -0.0, -1.0, -1e-3, np.inf, np.nan, 2.0, 1e-30], np.float32), 1000)
    mats = (lr.Material * 1)()
    ps = lr.PtScene(ctx, None, tris, mats, -1, 1e-4, 1e-3, builder=builder)
    nodes, aux, *_ = lro.build_tris(tris, ploc_=builder == lr.PLOC)
    for any_hit in (False, True):
        got, want = ps.trace(rays, any_hit=any_hit).view(np.uint32), lro.trace_wide(nodes, aux, tris, rays, any_hit).view(np.uint32)
        assert (want[:, 1] != 0xffffffff).mean() > 0.5
        assert np.array_equal(got, want), f"any {any_hit}: rays {np.nonzero((got != want).any(1))[0][:20]} differ"
    ps.close()
