"""Poseidon and Poseidon2 permutations with their linear maps on the matrix
cores (64 and 16 per wave) against the oracle, at the edges of their chunks,
tiles and size rules and with every SIMD busy.  Bit-exact (tolerance zero)."""
import numpy as np
import pytest

import oracle_bind as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ht", [0, 3])
@pytest.mark.parametrize("lg_l,ls,h", [(0, 9, 0),      # 16 per wave: one leaf
                                       (1, 4, 0),      # leaves hashed as they are, one level
                                       (3, 17, 1),
                                       (4, 1, 4),
                                       (6, 5, 6),      # one tile, part of one chunk, no levels
                                       (6, 8, 0),      # exactly one chunk
                                       (7, 9, 2),      # one element in the second chunk
                                       (9, 135, 3),    # an upper pass
                                       (14, 6, 0),     # two upper passes
                                       (15, 12, 4),    # the largest built in one launch
                                       (16, 10, 4),    # 64 per wave, every level 16 per wave
                                       (16, 3, 16),    # no levels
                                       (17, 6, 4),     # the first level 64 per wave
                                       (17, 7, 17),    # two waves on every SIMD, leaves only
                                       (18, 13, 18),   # four waves on every SIMD
                                       (18, 5, 2)])    # and the levels above them
def test_forest(zk, ht, lg_l, ls, h):
    print(f"forest lg_l={lg_l} ls={ls} h={h} ht={ht}", flush=True)
    leaves = ob.canonical(ls << lg_l, 900 + lg_l + ls)
    dig, caps = zk.merkle_tree(leaves, ls, h, ht)
    edig, ecap = ob.merkle(leaves, ls, h, ht)
    assert np.array_equal(caps, ecap)
    assert np.array_equal(dig, edig)


@pytest.mark.parametrize("ht", [0, 3])
@pytest.mark.parametrize("fill", [0, 1, 0xFFFFFFFF, 0xFFFFFFFF00000000, "edges"])
def test_edge_values(zk, ht, fill):
    """Leaves of one value (0, 1, 2^32 - 1, p - 1), and each leaf a mix of them."""
    n, ls = 256, 12
    if fill == "edges":
        v = np.array([0, 1, 0xFFFFFFFF, 0x100000000, 0x7F7F7F7F7F7F7F7F, 0x8080808080808080, ob.P - 1, ob.P - 2],
                     np.uint64)
        leaves = v[np.random.default_rng(5).integers(0, v.size, n * ls)]
    else:
        leaves = np.full(n * ls, fill, np.uint64)
    dig, caps = zk.merkle_tree(leaves, ls, 4, ht)
    edig, ecap = ob.merkle(leaves, ls, 4, ht)
    assert np.array_equal(caps, ecap)
    assert np.array_equal(dig, edig)


@pytest.mark.parametrize("ht", [0, 3])
@pytest.mark.parametrize("tile_log", [8, 9, 10])
def test_batch_levels(zk, ht, tile_log):
    """Level launches over several trees, the narrow levels (less than one
    wave, less than one work-group) among them."""
    jobs = []
    try:
        zk.set_level_launches(0)
        for k, (cols, lg_n, rate, cap) in enumerate([(5, 5, 1, 0), (9, 7, 2, 3), (17, 8, 1, 1)]):
            coeffs = ob.canonical(cols << lg_n, 70 + k)
            c = zk.Commit(coeffs, cols, lg_n, rate, cap, ht)
            zk.set_tuning(zk.Tuning(merkle_tile_log=tile_log), c)
            jobs.append((c, coeffs, cols, lg_n, rate, cap))
        zk.init_coset_rs(0, 9, 7)
        zk.commit_batch([j[0] for j in jobs])
    finally:
        zk.set_level_launches(zk.LEVEL_LAUNCHES_DEFAULT)
        zk.tuning_clear()
    for c, coeffs, cols, lg_n, rate, cap in jobs:
        leaves, dig, caps = c.results()
        want = ob.transpose_rev(ob.lde(coeffs, lg_n, rate, cols), lg_n + rate, cols)
        edig, ecap = ob.merkle(want, cols, cap, ht)
        assert np.array_equal(leaves, want)
        assert np.array_equal(caps, ecap)
        assert np.array_equal(dig, edig)


@pytest.mark.parametrize("ht", [0, 3])
@pytest.mark.parametrize("shapes", [[(5, 2, 1, 0), (3, 3, 1, 4), (9, 6, 2, 8), (17, 9, 3, 1)],  # 16 per wave, whole
                                    [(6, 13, 2, 2), (3, 13, 2, 15), (9, 4, 1, 0)],               # every level 16 per wave
                                    [(5, 15, 2, 4), (9, 3, 1, 0)]])                              # the first one 64 per wave
def test_batch_forests(zk, ht, shapes):
    """Trees of several sizes in one batch, three times over (the third call
    replays a captured graph): arrival counters return to zero."""
    zk.init_coset_rs(0, max(n + r for _, n, r, _ in shapes), 7)
    jobs = []
    for k, (cols, lg_n, rate, cap) in enumerate(shapes):
        coeffs = ob.canonical(cols << lg_n, 300 + k)
        jobs.append((zk.Commit(coeffs, cols, lg_n, rate, cap, ht), coeffs, cols, lg_n, rate, cap))
    want = []
    for _, coeffs, cols, lg_n, rate, cap in jobs:
        rows = ob.transpose_rev(ob.lde(coeffs, lg_n, rate, cols), lg_n + rate, cols)
        want.append((rows, *ob.merkle(rows, cols, cap, ht)))
    for _ in range(4):
        for j in jobs:
            j[0].d_digests.zero()
            j[0].d_caps.zero()
        zk.commit_batch([j[0] for j in jobs])
        for (c, *_), w in zip(jobs, want):
            for got, exp in zip(c.results(), w):
                assert np.array_equal(got, exp)
