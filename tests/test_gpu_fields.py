"""GPU parity of the whole-map field kernels: mergeOccupied and the distance read-outs."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

DIMS = [(1, 1, 1), (3, 5, 7), (15, 1, 2), (16, 3, 1), (17, 2, 9), (1, 31, 33), (64, 10, 5), (131, 7, 3)]


@pytest.mark.parametrize("d", DIMS)
@pytest.mark.parametrize("threshold", [0.0, 0.5, 1.0])
def test_merge_occupied_edges(gvx_lib, d, threshold):
    gvx = gvx_lib
    rng = np.random.default_rng(sum(d))
    n = int(np.prod(d))
    p = rng.integers(-128, 128, n).astype(np.int8)
    p[rng.random(n) < 0.3] = 127
    env, dist = gvx.Map(O.PROB_MAP, d, 0.01), gvx.Map(O.DIST_MAP, d, 0.01)
    env.write(p)
    off = (2, 0, 1)
    dist.merge_occupied(env, off, threshold)
    i = np.arange(n)
    own = ((i % d[0] + off[0]) | (((i // d[0]) % d[1] + off[1]) << 10) | ((i // (d[0] * d[1]) + off[2]) << 20))
    want = np.where(p.astype(int) > O.float_to_probability(threshold), own, O.dist_uninit(d)).astype(np.uint32)
    assert np.array_equal(dist.read(), want)


@pytest.mark.parametrize("d", DIMS)
@pytest.mark.parametrize("shift", [0, 1, 3])
def test_read_outs_edges(gvx_lib, d, shift):
    import torch
    gvx = gvx_lib
    rng = np.random.default_rng(sum(d) + 1)
    n = int(np.prod(d))
    site = [rng.integers(0, k, n) for k in d]
    raw = (site[0] | (site[1] << 10) | (site[2] << 20)).astype(np.uint32)
    raw[rng.random(n) < 0.2] = O.dist_uninit(d)
    side = np.float32(0.013)
    m = gvx.Map(O.DIST_MAP, d, float(side))
    m.write(raw)
    i = np.arange(n)
    at = [i % d[0], (i // d[0]) % d[1], i // (d[0] * d[1])]
    sq = sum((a - s) ** 2 for a, s in zip(at, site))
    none = raw == O.dist_uninit(d)
    assert np.array_equal(m.squared_distances(), np.where(none, 2**31 - 1, sq).astype(np.int32))
    # sqrt and product are correctly rounded float32 operations: equal bit for bit
    want = np.where(none, np.finfo(np.float32).max, np.sqrt(sq.astype(np.float32)) * side).astype(np.float32)
    buf = torch.full((n + 8,), -1.0, device="cuda")
    torch.cuda.synchronize()
    m.metric(buf[shift:shift + n])  # destinations off the 16-byte grid too
    got = buf.cpu().numpy()
    assert np.array_equal(got[shift:shift + n], want)
    assert (got[:shift] == -1).all() and (got[shift + n:] == -1).all()
