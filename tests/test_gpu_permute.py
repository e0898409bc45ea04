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


def _borrows(a, b):
    """Whether u - h1 borrows in the lazy product of a and b (gl64.h
    reduce128_rare): a b = lo + (h0 + 2^32 h1) 2^64 with the carry of the
    middle sum taken out of the high word, u = lo + h0 (2^32 - 1) mod 2^64."""
    m = (1 << 32) - 1
    a0, a1, b0, b1 = a & m, a >> 32, b & m, b >> 32
    u = a0 * b0
    w = a1 * b0 + a0 * b1 + (u >> 32)
    c, w = w >> 64, w & ((1 << 64) - 1)
    hi = a1 * b1 + (w >> 32)
    lo = (u & m) | ((w & m) << 32)
    return (lo + (hi & m) * m) % (1 << 64) < (hi >> 32) + c


def _reduced(x):
    return x % ob.P


def _rare_inputs():
    """S-box inputs by the product that borrows."""
    found = {}
    rng = np.random.default_rng(1)
    for e in range(20000):
        k = int(rng.integers(0, 64))
        x = ((1 << k) * int(rng.integers(1, 1 << int(rng.integers(1, 6)))) + (0 if e % 2 else (1 << int(rng.integers(0, 64))))) % ob.P
        x2 = _reduced(x * x)
        x3, x4 = _reduced(x2 * x), _reduced(x2 * x2)
        for step, (a, b) in enumerate([(x, x), (x2, x), (x2, x2), (x3, x4)]):
            if _borrows(a, b):
                found.setdefault(step, set()).add(x)
    assert set(found) >= {0, 2, 3}  # x^2, x^4 and x^7: powers of two times small numbers
    return [sorted(found[s])[:16] for s in sorted(found)]


def _solve(m, v):
    """x with m x = v mod p."""
    n, rows = len(v), [list(r) + [t] for r, t in zip(m, v)]
    for i in range(n):
        k = next(k for k in range(i, n) if rows[k][i])
        rows[i], rows[k] = rows[k], rows[i]
        inv = pow(rows[i][i], ob.P - 2, ob.P)
        rows[i] = [x * inv % ob.P for x in rows[i]]
        for k in range(n):
            if k != i:
                f = rows[k][i]
                rows[k] = [(x - f * y) % ob.P for x, y in zip(rows[k], rows[i])]
    return [r[n] for r in rows]


@pytest.mark.parametrize("ht", [0, 3])
def test_rare_borrows(zk, ht):
    """Leaves made so that first-round S-boxes take the exact form of a product
    (one lane of a wave, several, all)."""
    import re
    text = open(ob.ROOT + "/zeknox_amd/csrc/gl_constants.h").read()

    def table(name):
        body = re.search(r"#define " + name + r" \\\n(.*?)\n\n", text, re.S).group(1)
        return [int(t, 0) for t in re.findall(r"0x[0-9a-fA-F]+|\b\d+", body.replace("ULL", "").replace("ull", ""))]

    rc = table("ZK_POSEIDON_RC_LIST" if ht == 0 else "ZK_POSEIDON2_RC_LIST")[:12]
    m4 = [[5, 7, 1, 3], [4, 6, 1, 1], [1, 3, 5, 7], [1, 1, 4, 6]]
    external = [[m4[r % 4][c % 4] * (2 if r // 4 == c // 4 else 1) for c in range(8)] for r in range(8)]
    rare = _rare_inputs()
    rng = np.random.default_rng(2)
    n, ls = 1 << 16, 8  # 64 per wave from 2^16 leaves
    leaves = ob.canonical(n * ls, 31).reshape(n, ls)
    for leaf in [0, 5, 64, 95, 100, 101, 128 + 63] + list(range(192, 256)):
        want = [int(rng.choice(rare[int(rng.integers(0, len(rare)))])) if rng.random() < 0.5 else int(rng.integers(0, 1 << 62))
                for _ in range(8)]
        want[0] = int(rng.choice(rare[leaf % len(rare)]))
        v = [(x - k) % ob.P for x, k in zip(want, rc)]
        leaves[leaf] = v if ht == 0 else _solve(external, v)
    flat = np.ascontiguousarray(leaves.reshape(-1))
    dig, caps = zk.merkle_tree(flat, ls, 4, ht)
    edig, ecap = ob.merkle(flat, ls, 4, ht)
    assert np.array_equal(caps, ecap)
    assert np.array_equal(dig, edig)
