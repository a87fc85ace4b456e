"""PLOC's rounds at the edges of their searches, bit-exact against the oracle.

The nearest search is a wave's: 64 P positions (P = 1, 2, 4 a lane) of which the outer 2 R = 32 only
serve the others, in tiles of 352 or 864 positions a work-group, or over a list in one work-group's
LDS, from 96 clusters down in one wave. Sizes around those edges; boxes with many equal distances
(the tie rule decides every merge); and boxes whose areas overflow, which the search leaves to the
general one.

The build's own figures too: depth, clusters, and rounds. The rounds from n down to 1024 clusters are
launched in a number planned from n (5/6 left by each, two more), and a build counts those even where
fewer were needed: the sizes have some where fewer are, and some where more.
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


def soup(n, rng):
    lo = rng.uniform(-1, 1, (n, 3))
    return lo, lo + rng.uniform(0, 0.05, (n, 3))


def lattice(n, rng):
    # equal cubes on a lattice, -0 and 0 among the corners, many of them twice
    k = int(np.ceil((n * 0.7) ** (1 / 3)))
    i = rng.integers(0, k ** 3, n)
    lo = np.stack([i % k, i // k % k, i // k // k], 1).astype(np.float32) - k // 2
    lo[rng.random((n, 3)) < 0.5] *= np.float32(-1)
    lo = np.minimum(lo, -lo)
    return lo, lo + 1


def huge(n, rng):
    # one in fifty boxes at 1e20: the area of any box with it is infinite
    lo, hi = soup(n, rng)
    far = rng.random(n) < 0.02
    far[0] = True
    return np.where(far[:, None], lo * 1e20, lo), np.where(far[:, None], lo * 1e20 + 1e18, hi)


def planned(n):
    r = 0
    while n > 1024:
        n, r = n * 5 // 6, r + 1
    return min(r + 2, 128) if r else 0


@pytest.mark.parametrize("make", [soup, lattice, huge])
@pytest.mark.parametrize("n", [3, 16, 17, 31, 32, 33, 95, 96, 97, 1023, 1056, 1400, 4500, 200_000])
def test_rounds_match_the_oracle(ctx, make, n):
    print(f"ploc {make.__name__} n={n}", flush=True)
    lo, hi = make(n, np.random.default_rng(n))
    boxes = np.zeros((n, 8), np.float32)
    boxes[:, :3], boxes[:, 4:7] = lo, hi
    b = torch.from_numpy(boxes).cuda()
    nodes = torch.zeros((2 * n - 1, 8), dtype=torch.int32, device="cuda")
    aux = torch.zeros(n, dtype=torch.int32, device="cuda")
    srt = torch.zeros(2 * n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    st = ctx.build(b, n, nodes, aux, lr.PLOC, sorted_out=srt)
    sc, si = np.split(srt.cpu().numpy().view(np.uint32), 2)
    want, waux, depth, rounds, live, made = lro.ploc(sc, si, boxes, live=True, above=1024)
    assert np.array_equal(aux.cpu().numpy().view(np.uint32), waux)
    got = nodes.cpu().numpy().view(np.uint32)
    assert np.array_equal(got, want), f"nodes differ at {np.nonzero((got != want).any(1))[0][:8]}"
    print(f"  rounds {rounds}, {made} of them launched ones, {planned(n)} planned", flush=True)
    assert (st.depth, st.clusters, st.rounds) == (depth, live, rounds + max(0, planned(n) - made))
    if n > 1024 and make is soup:          # (either kind is among the sizes)
        assert made < planned(n)
    if n == 200_000 and make is not soup:
        assert made > planned(n)
