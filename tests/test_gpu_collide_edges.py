"""Map x map collision at the edges of the kernels' chunks, and results that calls hand back
through counters kept between calls."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

DIMS = [(1, 1, 1), (2, 1, 1), (31, 1, 1), (33, 3, 5), (256, 1, 1), (257, 2, 1), (64, 64, 3), (129, 31, 9)]


def _bits(rng, n, dens):
    m = np.zeros((n, 32), np.uint8)
    occ = rng.random(n) < dens
    m[occ] = rng.integers(0, 256, (int(occ.sum()), 32)) & rng.integers(0, 256, (int(occ.sum()), 32))
    m[rng.random(n) < 0.2, 0] |= 1  # eBVM_FREE alone never collides
    return m


def _prob(rng, n):
    return rng.integers(-128, 128, n).astype(np.int8)


def _pair(gvx, d, ta, tb, dens, seed):
    rng = np.random.default_rng(seed)
    n = int(np.prod(d))
    a = _bits(rng, n, dens) if ta == O.BITVECTOR_MAP else _prob(rng, n)
    b = _bits(rng, n, dens) if tb == O.BITVECTOR_MAP else _prob(rng, n)
    ga, gb = gvx.Map(ta, d, 0.01), gvx.Map(tb, d, 0.01)
    ga.write(a)
    gb.write(b)
    return a, b, ga, gb


@pytest.mark.parametrize("d", DIMS)
@pytest.mark.parametrize("dens", [0.0, 0.02, 1.0])
def test_collide_offsets(gvx_lib, d, dens):
    for off in ((0, 0, 0), (1, 0, 0), (-1, 0, 0), (3, 1, 0), (0, -1, -2)):
        for ta, tb in ((O.BITVECTOR_MAP, O.BITVECTOR_MAP), (O.BITVECTOR_MAP, O.PROB_MAP),
                       (O.PROB_MAP, O.BITVECTOR_MAP)):
            a, b, ga, gb = _pair(gvx_lib, d, ta, tb, dens, sum(d) + off[0])
            want = O.map_collide(ta, a, tb, b, d, 0.6, off)
            assert ga.collide(gb, 0.6, off) == want
            assert np.array_equal(ga.read().reshape(-1), a.reshape(-1))


@pytest.mark.parametrize("d", DIMS)
@pytest.mark.parametrize("dens", [0.0, 0.02, 1.0])
def test_collide_types_edges(gvx_lib, d, dens):
    for tb in (O.BITVECTOR_MAP, O.PROB_MAP):
        a, b, ga, gb = _pair(gvx_lib, d, O.BITVECTOR_MAP, tb, dens, sum(d) + 5)
        want, wmask = O.map_collide_types(O.BITVECTOR_MAP, a, tb, b, d, 0.6)
        got, mask = ga.collide_types(gb, 0.6)
        assert got == want and np.array_equal(mask, wmask)
        assert np.array_equal(ga.read().reshape(-1), a.reshape(-1))


def test_results_of_one_call_stay_out_of_the_next(gvx_lib):
    gvx = gvx_lib
    d = (32, 32, 32)
    full, empty = gvx.Map(O.BITVECTOR_MAP, d, 0.01), gvx.Map(O.BITVECTOR_MAP, d, 0.01)
    full.write(np.full((32**3, 32), 0xF0, np.uint8))
    inside = np.full((100, 3), 0.1, np.float32)
    mixed = np.concatenate([inside, np.full((1, 3), 9.0, np.float32)])
    lst = gvx.VoxelList(d, 0.01)
    for _ in range(3):
        assert full.collide_types(full)[0] == 32**3
        n, mask = empty.collide_types(full)
        assert n == 0 and not mask.any()
        assert full.collide(empty) == 0 and full.collide(full) == 32**3
        assert full.collide(full, offset=(0, 0, 40)) == 0
        m = gvx.Map(O.PROB_MAP, d, 0.01)
        assert m.insert_points(mixed, 1) is True
        assert m.insert_points(inside, 1) is False
        assert m.insert_coords(np.array([[32, 0, 0]], np.uint32), 1) is True
        assert m.insert_meta(inside, np.array([60, 40], np.uint32), [1, 2]) is False
        lst.insert_points(inside, 5)
        assert lst.collide_map(full, mode=1)[0] == 1
        assert lst.collide_map(empty, mode=1)[0] == 0


def pending_error(gvx):
    """An error of another user of the HIP runtime: no call of this library, left to be collected."""
    assert gvx.lib().hipSetDevice(1 << 20) != 0


def test_results_after_a_call_that_ended_early(gvx_lib):
    # a pending error ends a collision between its kernel and the read of its counters: what it
    # counted must not show up in the next call's result
    gvx = gvx_lib
    d = (24, 20, 9)
    n = int(np.prod(d))
    _, _, a, b = _pair(gvx, d, O.BITVECTOR_MAP, O.BITVECTOR_MAP, 0.5, 1)
    _, _, _, p = _pair(gvx, d, O.BITVECTOR_MAP, O.PROB_MAP, 0.5, 2)
    empty = gvx.Map(O.BITVECTOR_MAP, d, 0.01)
    la, lb, none = (gvx.VoxelList(d, 0.01) for _ in range(3))
    xyz = np.stack(np.unravel_index(np.arange(0, n, 3), d), 1).astype(np.uint32)
    la.insert_coords(xyz, 7)
    lb.insert_coords(xyz, 9)
    for early in (lambda: a.collide(b), lambda: a.collide(p, 0.3), lambda: a.collide_types(b),
                  lambda: a.collide_types(p, 0.3), lambda: a.collide_sv(b, window=3),
                  lambda: la.collide_map(a, mode=1), lambda: la.collide_list(lb), lambda: la.collide_bitcheck(la)):
        for after in (lambda: empty.collide(b), lambda: empty.collide_types(b)[0], lambda: none.collide_map(a)[0],
                      lambda: la.collide_list(none)[0]):
            pending_error(gvx)
            try:
                early()
            except gvx.GvxError:
                pass
            assert after() == 0
        pending_error(gvx)
        try:
            early()
        except gvx.GvxError:
            pass
        assert not empty.collide_types(b)[1].any()
