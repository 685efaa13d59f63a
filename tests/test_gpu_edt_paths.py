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


# z axes above 1024: the z pass in two sweeps, every x range to the stack kernels; (8, 1024, 3960)
# and (8, 1024, 3970) are the two sides of their number format (a diagonal of 2^24)
@pytest.mark.parametrize("d", [(70, 40, 1026), (33, 20, 4094), (3, 1024, 1100), (130, 2, 2000), (8, 1024, 3960),
                               (8, 1024, 3970)])
def test_deep_maps(gvx_lib, d):
    rng = np.random.default_rng(sum(d))
    n = int(np.prod(d))
    for k in (1, 4, n // 3000, n // 20):
        occ = np.zeros(n, bool)
        occ[rng.integers(0, n, k)] = True
        _check(gvx_lib, d, occ)


@pytest.mark.parametrize("d", [(70, 40, 1025), (1, 33, 4093)])
def test_deep_maps_of_odd_depth(gvx_lib, d):
    test_deep_maps(gvx_lib, d)


def test_deep_map_squared_distances_above_24_bits(gvx_lib):
    # row (238, 4093): costs 16784681, 16784744, 16784681 at x = 0, 8, 16, so the site at x = 8 is
    # voxel 8's nearest by one; rounded to 24 bits it owns no voxel
    d = (17, 239, 4094)
    occ = np.zeros(d[::-1], bool)
    for x, y, z in ((0, 18, 2), (8, 0, 3), (16, 18, 2)):
        occ[z, y, x] = True
    _check(gvx_lib, d, occ.reshape(-1))


def test_deepest_map(gvx_lib):
    # the far corner's row: (49, 11, 19) is voxel 48's nearest by one, 17621621 against 17621622
    d = (128, 1024, 4094)
    sites = np.array([(3, 12, 19), (20, 16, 17), (49, 11, 19), (56, 12, 18), (93, 12, 19), (115, 11, 17)], np.int64)
    g = gvx_lib.Map(O.DIST_MAP, d, 0.01)
    g.insert_coords(sites.astype(np.uint32), gvx_lib.eBVM_OCCUPIED)
    g.pba()
    row = np.stack([np.arange(d[0]), np.full(d[0], d[1] - 1), np.full(d[0], d[2] - 1)], 1)
    want = ((row[:, None] - sites[None]) ** 2).sum(-1).min(1)
    idx = (row[:, 2] * d[1] + row[:, 1]) * d[0] + row[:, 0]
    assert want[48] == 17621621
    assert np.array_equal(g.squared_distances(idx.astype(np.uint32)), want)
