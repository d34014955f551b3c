"""The device tree build at the sizes where its stages hand over, node for
node and bit for bit against the CPU oracle: cells at the limits of the
in-LDS splits (512 and 4096 particles) and one beyond, tiles that end with a
cell, type orders that move particles over several tiles, coincident
particles larger than either limit, and systems of both kinds in one forest.
Everything compared is exact, so the tolerance is equality."""
import numpy as np
import pytest

from gasoline_amd import ics
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def check(gpu, r, m, soft, nb, order, act=None, off=None):
    with gpu.Pkd(len(m), prec=gpu.PREC_FP64) as pk:
        pk.put("r", r)
        pk.put("fMass", m)
        pk.put("fSoft", soft)
        if act is not None:
            pk.put("iActive", act)
        for _ in range(2):                 # a second build starts from used scratch
            if off is None:
                pk.build_binary(nb, 1, 0.7, order)
            else:
                pk.build_forest(off, nb, 1, 0.7, order)
        root, perm, ints, dbls = pk.tree_info()
    parts = [(0, len(m))] if off is None else list(zip(off[:-1], off[1:]))
    n0 = 0
    for a, b in parts:
        if a == b:                         # an empty system has no root
            continue
        T = O.Tree(r[a:b], m[a:b], soft[a:b], iactive=None if act is None else act[a:b],
                   nBucket=nb, dTheta=0.7, iOrder=order)
        oi, od = T.nodes()
        k = slice(n0, n0 + len(oi))
        n0 += len(oi)
        oi = oi[:, :5].copy()
        oi[:, 1:3] += a                    # particle ranges of the whole store
        for c in (3, 4):                   # node ids likewise
            oi[oi[:, c] >= 0, c] += k.start
        assert np.array_equal(perm[a:b], T.perm() + a)
        assert np.array_equal(ints[k, :5], oi)
        assert np.array_equal(dbls[k, :6], od[:, [7, 8, 9, 10, 11, 12]])
        assert np.array_equal(dbls[k, 6], od[:, 44])
    assert n0 == len(ints)


@pytest.mark.parametrize("n", [1, 16, 17, 512, 513, 1024, 4096, 4097, 8192, 30011])
@pytest.mark.parametrize("order", [2, 4])
def test_tree_at_the_stage_limits(gpu, n, order):
    r, v, m = ics.plummer(n, seed=n)
    m = m * np.random.default_rng(n).uniform(0.5, 1.5, n)
    check(gpu, r, m, np.full(n, 0.01), 16, order)


@pytest.mark.parametrize("lack", [1, 2, 3])
def test_tree_type_orders_over_tiles(gpu, lack):
    # particles lacking TREEACTIVE (1), ACTIVE (2), or some of either
    n = 21000
    r, v, m = ics.plummer(n, seed=5)
    u = np.random.default_rng(6).uniform(size=n)
    act = np.full(n, 3, np.uint32)
    if lack & 1:
        act[u < 0.4] &= ~np.uint32(2)
    if lack & 2:
        act[(u > 0.2) & (u < 0.7)] &= ~np.uint32(1)
    check(gpu, r, m, np.full(n, 0.01), 8, 2, act=act)


@pytest.mark.parametrize("clump", [600, 5000])
def test_tree_large_coincident_bucket(gpu, clump):
    n = 9000
    r, v, m = ics.plummer(n, seed=8)
    r[100:100 + clump] = r[100]
    check(gpu, r, m, np.full(n, 0.01), 16, 4)


def test_tree_with_many_more_cells_than_usual(gpu):
    # groups of 30 particles at 2^-k beside 64 coincident ones: buckets of one
    # particle though they may hold 64, six times the usual number of cells
    g, k = 300, np.arange(30)
    one = np.zeros((94, 3))
    one[:30, 0] = 2.0 ** -k
    r = np.concatenate([one + [4.0 * (i % 20), 4.0 * (i // 20), 0.0] for i in range(g)])
    m = np.full(len(r), 1.0 / len(r))
    check(gpu, r, m, np.full(len(r), 0.01), 64, 4)


def test_forest_of_large_and_small_systems(gpu):
    sizes = [1, 4096, 0, 9000, 17, 4097, 300, 700]
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    r, v, m = ics.plummer(off[-1], seed=9)
    act = np.where(np.arange(off[-1]) % 5 == 0, 1, 3).astype(np.uint32)
    check(gpu, r, m, np.full(off[-1], 0.01), 16, 2, act=act, off=off)


def groups(g, chain, same, span):
    """g groups, each of `same` coincident particles and a chain of `chain`
    at span * 0.4^k beside them, of which every split takes one away: two
    cells a particle, whatever a bucket may hold."""
    x = np.concatenate([span * 0.4 ** np.arange(chain), np.zeros(same)])
    r = np.zeros((g, len(x), 3))
    r[:, :, 0] = x
    r[:, :, 1] = 4.0 * (np.arange(g) % 64)[:, None]
    r[:, :, 2] = 4.0 * (np.arange(g) // 64)[:, None]
    return r.reshape(-1, 3)


def test_out_of_slots_while_subtrees_wait_for_the_chip(gpu):
    # about a thousand subtrees, twice what the chip holds at once, of which
    # the first ones already use up the slots of the first try
    r = groups(4000, 30, 64, 1.0)
    m = np.full(len(r), 1.0 / len(r))
    check(gpu, r, m, np.full(len(r), 0.01), 64, 2)


@pytest.mark.parametrize("g,same", [(6, 4200), (8, 600)])
def test_out_of_slots_above_the_subtrees(gpu, g, same):
    # chains that use up the slots of the first try in the levels above 4096
    # particles, and in the cells between 4096 and 512
    r = groups(g, 700, same, 1.0)
    m = np.full(len(r), 1.0 / len(r))
    check(gpu, r, m, np.full(len(r), 0.01), 64, 4)


@pytest.mark.parametrize("n", [20, 100, 600, 5000, 30000])
def test_split_with_an_empty_side_is_refused(gpu, n):
    # two positions whose midpoint rounds to the lower one, in a cell of each
    # stage's size; the handle builds again afterwards
    r, v, m = ics.plummer(n, seed=n)
    bad = np.ones((n, 3))
    bad[n // 2:, 0] = np.nextafter(1.0, 2.0)
    with gpu.Pkd(n, prec=gpu.PREC_FP64) as pk:
        pk.put("fMass", m)
        pk.put("fSoft", np.full(n, 0.01))
        for _ in range(2):
            pk.put("r", bad)
            with pytest.raises(gpu.GGError, match="one side empty"):
                pk.build_binary(16, 1, 0.7, 2)
            pk.put("r", r)
            pk.build_binary(16, 1, 0.7, 2)
            T = O.Tree(r, m, np.full(n, 0.01), nBucket=16, dTheta=0.7, iOrder=2)
            assert np.array_equal(pk.tree_info()[1], T.perm())


@pytest.mark.parametrize("lack", [False, True])
@pytest.mark.parametrize("big", [(), (600,), (9000, 513, 4096, 4097)])
def test_forest_of_many_small_systems(gpu, big, lack):
    # more systems than one pass of the roots' scan takes, buckets and
    # subtrees among them, the larger ones at both ends and between
    rng = np.random.default_rng(len(big) + 10 * lack)
    sizes = rng.integers(0, 12, 4300)
    sizes[rng.integers(0, 4300, 60)] = rng.integers(17, 513, 60)
    sizes[7:12] = 512, 64, 16, 128, 129
    sizes[[2150, 0, 4299, 2151][:len(big)]] = big
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    n = int(off[-1])
    act = rng.choice(np.array([0, 1, 2, 3], np.uint32), n) if lack else None
    check(gpu, rng.normal(size=(n, 3)), rng.uniform(0.5, 1.5, n), np.full(n, 0.01), 16, 3,
          act=act, off=off)


def test_forest_that_takes_slots_for_several_systems_at_once(gpu):
    sizes = np.random.default_rng(4).integers(17, 20, 21000)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    n = int(off[-1])
    r = np.random.default_rng(5).normal(size=(n, 3))
    check(gpu, r, np.full(n, 1.0), np.full(n, 0.01), 16, 2, off=off)


@pytest.mark.parametrize("clump", [513, 577, 4097])
def test_large_coincident_bucket_of_unequal_particles(gpu, clump):
    # the sums follow the storage order: with unequal masses another order
    # shows; the type orders move the clump's particles first
    n = clump + 1500
    rng = np.random.default_rng(clump)
    r = rng.normal(size=(n, 3))
    r[rng.permutation(n)[:clump]] = r[0]
    check(gpu, r, rng.uniform(0.5, 1.5, n), rng.uniform(0.01, 0.02, n), 16, 3,
          act=rng.choice(np.array([0, 2, 3], np.uint32), n))


def test_level_of_more_cells_than_one_pass_takes(gpu):
    # 1100 copies of one system of more than 4096 particles: the first levels
    # have more cells than the workgroup that decides them has threads
    n, k = 4200, 1100
    r, v, m = ics.plummer(n, seed=11)
    T = O.Tree(r, m, np.full(n, 0.01), nBucket=32, dTheta=0.7, iOrder=2)
    oi, od = T.nodes()
    nn = len(oi)
    with gpu.Pkd(n * k, prec=gpu.PREC_FP64) as pk:
        pk.put("r", np.tile(r, (k, 1)))
        pk.put("fMass", np.tile(m, k))
        pk.put("fSoft", np.full(n * k, 0.01))
        pk.build_forest((n * np.arange(k + 1)).astype(np.int32), 32, 1, 0.7, 2)
        root, perm, ints, dbls = pk.tree_info()
    at = np.arange(k)[:, None]
    assert np.array_equal(perm.reshape(k, n), T.perm()[None] + n * at)
    ints = ints.reshape(k, nn, 6)
    for c, step in ((0, 0), (1, n), (2, n), (3, nn), (4, nn)):
        assert np.array_equal(ints[:, :, c], np.where(oi[:, c] >= 0, oi[:, c] + step * at, oi[:, c]))
    dbls = dbls.reshape(k, nn, 8)
    assert np.array_equal(dbls[:, :, :6], np.tile(od[:, [7, 8, 9, 10, 11, 12]], (k, 1, 1)))
    assert np.array_equal(dbls[:, :, 6], np.tile(od[:, 44], (k, 1)))
