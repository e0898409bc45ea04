"""Which launches a schedule leads to, read from the library's own kernel
timing, and that the results are the oracle's under each (bit-exact): a
schedule that the caller set runs as it stands, whatever kernels the library
prefers for that size."""
import numpy as np
import pytest

import oracle_bind as ob

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _defaults(zk):
    zk.init_coset_rs(0, 18, 7)
    zk.tuning_clear()
    yield
    zk.tuning_clear()
    zk.set_level_launches(zk.LEVEL_LAUNCHES_DEFAULT)
    zk.set_lone_level_launches(zk.LONE_LEVEL_LAUNCHES_DEFAULT)


def launches(zk, call):
    """{family: launches} of one call."""
    zk.profile_enable(True)
    zk.kernel_stats_reset()
    try:
        call()
        return {k: v[0] for k, v in zk.kernel_stats().items()}
    finally:
        zk.profile_enable(False)


class Job:
    def __init__(self, zk, cols, lg_n, rate, cap, ht):
        self.args = cols, lg_n, rate, cap, ht
        self.coeffs = ob.canonical(cols << lg_n, 5100 + cols + lg_n + ht)
        self.commit = zk.Commit(self.coeffs, cols, lg_n, rate, cap, ht)

    def check(self):
        cols, lg_n, rate, cap, ht = self.args
        rows = ob.transpose_rev(ob.lde(self.coeffs, lg_n, rate, cols), lg_n + rate, cols)
        dig, caps = ob.merkle(rows, cols, cap, ht)
        for got, want in zip(self.commit.results(), (rows, dig, caps)):
            assert np.array_equal(got, want), self.args


MERKLE = [(0, 8, 0), (0, 9, 0), (0, 10, 0), (0, 9, 1), (3, 8, 0), (3, 9, 0), (3, 10, 0)]  # hash, tile, valu


@pytest.mark.parametrize("ht,tile,valu", MERKLE)
def test_small_forest_under_a_set_schedule(zk, ht, tile, valu):
    j, other = Job(zk, 9, 9, 2, 3, ht), Job(zk, 6, 10, 2, 0, ht)
    got = launches(zk, lambda: zk.commit_batch([j.commit, other.commit]))
    assert got["merkle_narrow"] == 1 and "merkle_leaves" not in got
    zk.set_tuning(zk.Tuning(merkle_tile_log=tile, merkle_valu=valu), j.commit)
    got = launches(zk, lambda: zk.commit_batch([j.commit]))
    assert got["merkle_leaves"] == 1 and "merkle_narrow" not in got
    j.check()
    for _ in range(4):  # the shape beside one without a schedule; the last replays a graph
        j.commit.d_digests.zero(), other.commit.d_digests.zero()
        zk.commit_batch([other.commit, j.commit])
        j.check(), other.check()
    got = launches(zk, lambda: zk.commit_batch([other.commit, j.commit]))
    assert got["merkle_leaves"] == 1 and got["merkle_narrow"] == 1


@pytest.mark.parametrize("ht,tile,valu", MERKLE)
def test_large_forest_under_a_set_schedule(zk, ht, tile, valu):
    """The 64-per-wave and VALU leaf kernels and, for a batch, levels that are
    64 per wave beside a tree of less than a wave's nodes."""
    jobs = [Job(zk, 9, 15, 2, 4, ht), Job(zk, 9, 3, 1, 0, ht)]
    for j in jobs:
        zk.set_tuning(zk.Tuning(merkle_tile_log=tile, merkle_valu=valu), j.commit)
    for least in (zk.LEVEL_LAUNCHES_DEFAULT, None):
        zk.set_level_launches(least)
        got = launches(zk, lambda: zk.commit_batch([j.commit for j in jobs]))
        assert got["merkle_leaves"] == 1 and "merkle_narrow" not in got
        # 2^17 + 2^4 children, 2^16 + 2^3, then few enough for the rest together
        assert got.get("merkle_levels", 0) == (3 if least else 0)
        for j in jobs:
            j.check()


@pytest.mark.parametrize("ht,tile,valu", MERKLE)
def test_lone_tree_under_a_set_default(zk, ht, tile, valu):
    for lg in (11, 16):
        leaves = ob.canonical(12 << lg, 77 + lg)
        want = ob.merkle(leaves, 12, 2, ht)
        zk.tuning_clear()
        for seen in ("merkle_narrow" if lg <= 15 else "merkle_leaves", "merkle_leaves"):
            out = []
            got = launches(zk, lambda: out.extend(zk.merkle_tree(leaves, 12, 2, ht)))
            assert got[seen] == 1 and len(set(got) & {"merkle_narrow", "merkle_leaves"}) == 1
            assert np.array_equal(out[0], want[0]) and np.array_equal(out[1], want[1])
            zk.set_tuning(zk.Tuning(merkle_tile_log=tile, merkle_valu=valu))


@pytest.mark.parametrize("ht", [0, 3])
@pytest.mark.parametrize("lg,cap", [(11, 2), (6, 6), (3, 0), (15, 4)])
def test_zero_takes_small_levels_apart(zk, ht, lg, cap):
    leaves = ob.canonical(7 << lg, 31 + lg)
    want = ob.merkle(leaves, 7, cap, ht)
    apart = {"merkle_leaves": 1, "merkle_levels": 1} if cap < lg else {"merkle_leaves": 1}
    for least, seen in ((0, apart), (None, {"merkle_narrow": 1}), (zk.LONE_LEVEL_LAUNCHES_DEFAULT, {"merkle_narrow": 1})):
        zk.set_lone_level_launches(least)
        zk.set_level_launches(zk.LEVEL_LAUNCHES_DEFAULT if least else least)
        out = []
        assert launches(zk, lambda: out.extend(zk.merkle_tree(leaves, 7, cap, ht))) == seen
        assert np.array_equal(out[0], want[0]) and np.array_equal(out[1], want[1])
        j = Job(zk, 7, lg - 1, 1, cap, ht)
        got = launches(zk, lambda: zk.commit_batch([j.commit]))
        assert {k: v for k, v in got.items() if k.startswith("merkle")} == seen
        j.check()


@pytest.mark.parametrize("ht", [0, 3])
def test_switch_of_a_lone_tree(zk, ht):
    """2^16 leaves, the smallest whose levels are apart by default."""
    leaves = ob.canonical(9 << 16, 16)
    want = ob.merkle(leaves, 9, 4, ht)
    for least, levels in ((zk.LONE_LEVEL_LAUNCHES_DEFAULT, 1), (None, 0), (0, 1)):
        zk.set_lone_level_launches(least)
        out = []
        got = launches(zk, lambda: out.extend(zk.merkle_tree(leaves, 9, 4, ht)))
        assert got["merkle_leaves"] == 1 and got.get("merkle_levels", 0) == levels
        assert np.array_equal(out[0], want[0]) and np.array_equal(out[1], want[1])


def test_keccak_tops_are_timed_as_levels(zk):
    """2^18 and 2^17 children in a launch each, the rest on tiles of 256."""
    leaves = ob.canonical(3 << 18, 18)
    want = ob.merkle(leaves, 3, 1, zk.HASH_KECCAK)
    out = []
    got = launches(zk, lambda: out.extend(zk.merkle_tree(leaves, 3, 1, zk.HASH_KECCAK)))
    assert got == {"merkle_leaves": 1, "merkle_levels": 3}
    assert np.array_equal(out[0], want[0]) and np.array_equal(out[1], want[1])
    j = Job(zk, 3, 17, 1, 1, zk.HASH_KECCAK)
    got = launches(zk, lambda: zk.commit_batch([j.commit]))
    assert (got["merkle_leaves"], got["merkle_levels"]) == (1, 3)
    j.check()


@pytest.mark.parametrize("strided,even", [(9, 0), (4, 1), (1, 0)])
def test_transforms_under_a_set_schedule(zk, strided, even):
    t = zk.Tuning(strided, even)
    j = Job(zk, 3, 13, 1, 2, zk.HASH_KECCAK)
    assert launches(zk, lambda: zk.commit_batch([j.commit]))["batch_ntt"] == 1
    zk.set_tuning(t, j.commit)
    assert launches(zk, lambda: zk.commit_batch([j.commit]))["batch_ntt"] == len(zk.ntt_pass_sizes(13, t))
    j.check()
    zk.set_tuning(t)
    for lg_n, rate, B in ((13, 0, 5), (15, 0, 8), (13, 1, 3), (15, 1, 4)):
        x = ob.canonical(B << lg_n, 9 * lg_n + rate)
        out = x.copy() if rate == 0 else np.zeros(B << (lg_n + rate), np.uint64)
        cfg = zk.NTTConfig(batches=B, extension_rate_bits=rate, with_coset=True)
        got = launches(zk, lambda: zk.ntt_batch(0, out, lg_n, cfg) if rate == 0 else zk.lde_batch(0, out, x, lg_n, cfg))
        assert got["bitrev"] == 1 and got.get("ntt_pass", 0) + got.get("ntt_pass_lde", 0) == len(zk.ntt_pass_sizes(lg_n, t))
        assert np.array_equal(out, ob.ntt(x, lg_n, B, False, True) if rate == 0 else ob.lde(x, lg_n, rate, B))


@pytest.mark.parametrize("lg_n,rate,ht,candidates", [(13, 1, 1, 2),   # one pass split, two more work-group sizes
                                                     (6, 2, 0, 0),    # and no Merkle schedule
                                                     (8, 1, 3, 0),
                                                     (8, 2, 0, 3),    # 64 copies are above 2^15 leaves
                                                     (14, 1, 1, None)])
def test_the_tuner_times_each_plan_once(zk, lg_n, rate, ht, candidates):
    j = Job(zk, 5, lg_n, rate, 1, ht)
    if candidates is None:  # every split that differs, and the work-group sizes
        plans = {tuple(zk.ntt_pass_sizes(lg_n, zk.Tuning(s, e))) for s in range(4, 10) for e in (0, 1)}
        candidates = len(plans) - 1 + 2
    got = launches(zk, lambda: zk.autotune([j.commit], iters=2))
    # the warm-up, then two runs of the default and of each candidate
    assert sum(v for k, v in got.items() if k in ("merkle_leaves", "merkle_narrow")) == 1 + 2 * (1 + candidates)
    t = zk.get_tuning(j.commit).astuple()
    if lg_n == 13:
        assert t[:2] == (9, 0)
    if not candidates:
        assert t[2:] == (8, 0)
    j.check()


def test_a_set_schedule_is_saved_as_one(zk, tmp_path):
    j = Job(zk, 4, 8, 2, 1, zk.HASH_POSEIDON)
    zk.set_tuning(zk.Tuning(merkle_tile_log=9), j.commit)
    path = str(tmp_path / "t")
    zk.tuning_save(path)
    zk.tuning_clear()
    zk.tuning_load(path)
    assert "merkle_leaves" in launches(zk, lambda: zk.commit_batch([j.commit]))
    # tables written without the mark, and without the column before it, load as before
    lines = open(path).read().splitlines()
    for drop in (1, 2):
        open(path, "w").write(" ".join(lines[1].split()[:-drop]) + "\n")
        zk.tuning_clear()
        zk.tuning_load(path)
        assert zk.get_tuning(j.commit).astuple() == (9, 0, 9, 0)
        zk.commit_batch([j.commit])
        j.check()
