"""The EDT's paths by map size and field: small maps (windows as long as the line), cut-off
windows with their stack fallback, and fields that mix both, against the oracle's PBA."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _check(gvx, d, occ):
    idx = np.flatnonzero(occ)
    m = np.full(occ.size, O.dist_uninit(d), np.uint32)
    x, y, z = idx % d[0], (idx // d[0]) % d[1], idx // (d[0] * d[1])
    m[idx] = (x | (y << 10) | (z << 20)).astype(np.uint32)
    g = gvx.Map(O.DIST_MAP, d, 0.01)
    g.write(m)
    g.pba()
    got = g.read()
    O.pba(m, d, threads=8)
    assert np.array_equal(got, m)


# edges of the lane, group and row layouts of the small-map kernels
@pytest.mark.parametrize("d", [(1, 1, 1), (8, 8, 8), (63, 9, 5), (64, 16, 33), (65, 17, 32), (127, 130, 31),
                               (128, 64, 129), (129, 3, 257), (255, 40, 40), (257, 33, 17), (511, 12, 9),
                               (512, 512, 3), (5, 512, 40), (3, 500, 1024), (40, 40, 1000)])
def test_small_maps(gvx_lib, d):
    rng = np.random.default_rng(sum(d))
    n = int(np.prod(d))
    for k in (0, 1, 3, max(1, n // 3000), n // 50, n // 2):
        occ = np.zeros(n, bool)
        occ[rng.integers(0, n, k)] = True
        _check(gvx_lib, d, occ)


LARGE = (300, 259, 251)  # above the small-map bound, no side a multiple of 64


@pytest.mark.parametrize("density", [0.0004, 0.001, 0.01, 0.1])
def test_uniform_fields(gvx_lib, density):
    rng = np.random.default_rng(5)
    _check(gvx_lib, LARGE, rng.random(int(np.prod(LARGE))) < density)


def _coords(d):
    return np.meshgrid(*(np.arange(k) for k in reversed(d)), indexing="ij")  # z, y, x


@pytest.mark.parametrize("what", ["cavity", "plane", "half", "slab", "far corner"])
def test_uneven_fields(gvx_lib, what):
    d = LARGE
    rng = np.random.default_rng(6)
    z, y, x = _coords(d)
    occ = rng.random(z.shape) < 0.01
    if what == "cavity":  # voxels beyond the window radius in some slices: their y lines are redone
        occ &= (x - 150) ** 2 + (y - 130) ** 2 + (z - 120) ** 2 > 34 ** 2
    elif what == "plane":  # lines of one x without any site
        occ &= x != 131
    elif what == "half":  # windowed and stack x ranges in every slice
        occ &= (x < 128) | (rng.random(z.shape) < 0.01)
    elif what == "slab":  # x ranges without any obstacle
        occ &= x < 64
    else:
        occ &= (x + y + z > 60)
    _check(gvx_lib, d, occ.reshape(-1))
