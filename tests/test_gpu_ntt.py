"""GPU NTT / LDE / transpose through the C ABI vs the oracle. Bit-exact."""
from types import SimpleNamespace

import numpy as np
import pytest

import oracle_bind as ob
from oracle_bind import P, orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _coset(zk):
    zk.init_coset_rs(0, 24, 7)


@pytest.mark.parametrize("lg_n,rate,B", [(1, 1, 2), (2, 1, 3), (3, 2, 1), (4, 3, 5), (5, 1, 2), (8, 2, 3),
                                         (10, 3, 2), (11, 1, 4), (12, 2, 2), (13, 1, 3), (14, 3, 2), (16, 1, 2),
                                         (15, 3, 2)])
@pytest.mark.parametrize("coset", [True, False])
def test_lde_forward_vs_oracle(zk, lg_n, rate, B, coset):
    print(f"lde lg_n={lg_n} rate={rate} B={B} coset={coset}", flush=True)
    x = ob.canonical(B << lg_n, 17 * lg_n + rate + B)
    out = np.zeros(B << (lg_n + rate), np.uint64)
    zk.lde_batch(0, out, x, lg_n, zk.NTTConfig(batches=B, extension_rate_bits=rate, with_coset=coset))
    assert np.array_equal(out, ob.lde(x, lg_n, rate, B, coset=coset))


@pytest.mark.parametrize("lg_n,rate,B", [(3, 1, 2), (9, 2, 3), (13, 1, 2)])
@pytest.mark.parametrize("coset", [True, False])
def test_lde_inverse_vs_oracle(zk, lg_n, rate, B, coset):
    x = ob.canonical(B << lg_n, 5 * lg_n + rate)
    out = np.zeros(B << (lg_n + rate), np.uint64)
    zk.lde_batch(0, out, x, lg_n, zk.NTTConfig(batches=B, extension_rate_bits=rate, with_coset=coset),
                 direction=zk.INVERSE)
    assert np.array_equal(out, ob.lde(x, lg_n, rate, B, inverse=True, coset=coset))


def test_lde_device_pointers_and_salt(zk):
    lg_n, rate, B, salt = 10, 2, 3, 2
    x = ob.canonical(B << lg_n, 3)
    N = 1 << (lg_n + rate)
    din = zk.DeviceBuffer.from_host(x)
    dout = zk.DeviceBuffer((B + salt) * N)
    cfg = zk.NTTConfig(batches=B, extension_rate_bits=rate, with_coset=True, are_inputs_on_device=True,
                       are_outputs_on_device=True, salt_size=salt)
    zk.lde_batch(0, dout, din, lg_n, cfg)
    got = dout.to_host()
    assert np.array_equal(got[:B * N], ob.lde(x, lg_n, rate, B))
    assert np.all(got[B * N:] < np.uint64(P))


@pytest.mark.parametrize("lg,B", [(1, 3), (4, 2), (9, 1), (10, 3), (12, 2), (13, 2), (17, 1), (20, 1)])
@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("coset", [False, True])
def test_ntt_vs_oracle(zk, lg, B, inverse, coset):
    print(f"ntt lg={lg} B={B} inverse={inverse} coset={coset}", flush=True)
    x = ob.canonical(B << lg, 7 * lg + B + 2 * inverse + coset)
    buf = x.copy()
    cfg = zk.NTTConfig(batches=B, with_coset=coset)
    (zk.intt_batch if inverse else zk.ntt_batch)(0, buf, lg, cfg)
    assert np.array_equal(buf, ob.ntt(x, lg, B, inverse, coset))


# First passes of 5..8 stages (the two-round strided kernel) over more tiles
# than the device holds work-groups, so every work-group walks several tiles
# (prefetch and twiddle reloads); in place (NTT, with the coset it reads
# through the one-tile kernel) and from coefficients (LDE).
@pytest.mark.parametrize("lg,B", [(17, 40), (18, 16), (19, 8), (20, 8)])
@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("coset", [False, True])
def test_ntt_two_round_first_pass_vs_oracle(zk, lg, B, inverse, coset):
    print(f"ntt lg={lg} B={B} inverse={inverse} coset={coset}", flush=True)
    x = ob.canonical(B << lg, 11 * lg + B + 2 * inverse + coset)
    buf = x.copy()
    (zk.intt_batch if inverse else zk.ntt_batch)(0, buf, lg, zk.NTTConfig(batches=B, with_coset=coset))
    assert np.array_equal(buf, ob.ntt(x, lg, B, inverse, coset))


@pytest.mark.parametrize("lg_n,rate,B", [(17, 1, 8), (18, 2, 4), (19, 1, 4), (20, 1, 4)])
@pytest.mark.parametrize("coset", [True, False])
def test_lde_two_round_first_pass_vs_oracle(zk, lg_n, rate, B, coset):
    print(f"lde lg_n={lg_n} rate={rate} B={B} coset={coset}", flush=True)
    x = ob.canonical(B << lg_n, 13 * lg_n + rate + B)
    out = np.zeros(B << (lg_n + rate), np.uint64)
    zk.lde_batch(0, out, x, lg_n, zk.NTTConfig(batches=B, extension_rate_bits=rate, with_coset=coset))
    assert np.array_equal(out, ob.lde(x, lg_n, rate, B, coset=coset))


def test_ntt_roundtrip_on_device(zk):
    lg, B = 18, 2
    x = ob.canonical(B << lg, 42)
    d = zk.DeviceBuffer.from_host(x)
    cfg = zk.NTTConfig(batches=B, are_inputs_on_device=True, are_outputs_on_device=True)
    zk.ntt_batch(0, d, lg, cfg)
    zk.intt_batch(0, d, lg, cfg)
    assert np.array_equal(d.to_host(), x)


@pytest.mark.parametrize("lg,B", [(0, 3), (1, 2), (5, 7), (5, 32), (6, 33), (7, 137), (8, 400), (10, 135), (11, 271),
                                  (12, 85), (13, 2)])
def test_transpose_rev_vs_oracle(zk, lg, B):
    x = ob.canonical(B << lg, 9 * lg + B)
    out = np.zeros_like(x)
    zk.transpose_rev_batch(0, out, x, lg, zk.TransposeConfig(batches=B))
    assert np.array_equal(out, ob.transpose_rev(x, lg, B))


def test_lde_135x2e15_rate3_vs_oracle(zk):
    """135 columns of 2^15 coefficients, rate 3, coset 7 -> 2^18-point LDE."""
    lg_n, rate, B = 15, 3, 135
    x = ob.canonical(B << lg_n, 2024)
    din = zk.DeviceBuffer.from_host(x)
    dout = zk.DeviceBuffer(B << (lg_n + rate))
    cfg = zk.NTTConfig(batches=B, extension_rate_bits=rate, with_coset=True, are_inputs_on_device=True,
                       are_outputs_on_device=True)
    zk.lde_batch(0, dout, din, lg_n, cfg)
    assert np.array_equal(dout.to_host(), ob.lde(x, lg_n, rate, B))


def test_invalid_lde_arguments(zk):
    x = np.zeros(8, np.uint64)
    out = np.zeros(64, np.uint64)
    with pytest.raises(zk.ZeknoxError) as e:
        zk.lde_batch(0, out, x, 0, zk.NTTConfig(batches=1, extension_rate_bits=1))
    assert e.value.code == 1
    with pytest.raises(zk.ZeknoxError) as e:
        zk.lde_batch(0, out, x, 3, zk.NTTConfig(batches=1, extension_rate_bits=0))
    assert e.value.code == 1


# The passes compute on lazy values and leave out what a random operand needs
# once in 2^32, fixing the lanes where it was needed after all.
# Words at and above p, runs of -1 and multiples of 2^48 reach that in every
# kernel: single tiles (ragged and whole), one- and two-round strided passes
# of each stage count, in place, through the coset and from coefficients.
def rare_words(count, seed):
    rng = np.random.default_rng(seed)
    special = np.array([0, 0, 1, 2, P - 2, P - 1, P - 1, P, P + 1, 2**64 - 2, 2**64 - 1, 2**32 - 1, 1 << 32, 1 << 48, 3 << 48,
                        0xFFFF << 48, 1 << 63], dtype=np.uint64)
    x = special[rng.integers(0, len(special), count)]
    some = rng.random(count) < 0.05
    x[some] = rng.integers(0, 2**64, int(some.sum()), dtype=np.uint64)
    return x


@pytest.mark.parametrize("lg,B", [(1, 5), (3, 3), (4, 7), (7, 2), (11, 3), (12, 2), (13, 3), (14, 2), (15, 1), (16, 2), (17, 1),
                                  (18, 1), (19, 1), (20, 1), (21, 1), (2, 1500), (9, 17), (13, 48), (14, 48)])
@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("coset", [False, True])
def test_ntt_of_rare_words_vs_oracle(zk, lg, B, inverse, coset):
    print(f"ntt lg={lg} B={B} inverse={inverse} coset={coset}", flush=True)
    x = rare_words(B << lg, 3 * lg + B + 2 * inverse + coset)
    buf = x.copy()
    (zk.intt_batch if inverse else zk.ntt_batch)(0, buf, lg, zk.NTTConfig(batches=B, with_coset=coset))
    assert np.array_equal(buf, ob.ntt(x % np.uint64(P), lg, B, inverse, coset))


@pytest.mark.parametrize("lg_n,rate,B", [(1, 1, 3), (4, 2, 3), (9, 1, 5), (12, 1, 3), (13, 2, 1), (14, 1, 1), (15, 1, 3), (16, 2, 1),
                                         (17, 1, 1), (18, 1, 1), (19, 1, 1), (20, 1, 1), (1, 5, 3), (8, 4, 3), (7, 5, 2),
                                         (9, 4, 2), (10, 3, 3), (11, 2, 1), (12, 1, 50), (10, 4, 48), (11, 3, 48),
                                         (12, 2, 48), (13, 1, 48), (13, 3, 2)])
@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("coset", [False, True])
def test_lde_of_rare_words_vs_oracle(zk, lg_n, rate, B, inverse, coset):
    print(f"lde lg_n={lg_n} rate={rate} B={B} inverse={inverse} coset={coset}", flush=True)
    x = rare_words(B << lg_n, 7 * lg_n + rate + B + inverse)
    out = np.zeros(B << (lg_n + rate), np.uint64)
    zk.lde_batch(0, out, x, lg_n, zk.NTTConfig(batches=B, extension_rate_bits=rate, with_coset=coset),
                 direction=zk.INVERSE if inverse else zk.FORWARD)
    assert np.array_equal(out, ob.lde(x % np.uint64(P), lg_n, rate, B, inverse=inverse, coset=coset))


# Commits of degrees whose LDE is one launch, jobs of one list sharing it or
# not: a ragged last tile, blocks of 2^13, columns of mixed degrees.
def test_commit_of_one_launch_degrees_vs_oracle(zk):
    shapes = [(3, 1, 1), (2, 4, 2), (5, 9, 1), (20, 10, 3), (7, 12, 1), (3, 13, 1), (2, 13, 2), (1, 13, 5), (2, 14, 1), (4, 10, 1)]
    jobs, keep = [], []
    for c, n, r in shapes:
        x = rare_words(c << n, 100 * c + n + r)
        N = 1 << (n + r)
        d = [zk.DeviceBuffer.from_host(x), zk.DeviceBuffer(c * N), zk.DeviceBuffer(8 * N), zk.DeviceBuffer(4)]
        jobs.append(zk.CommitJob(d[0].ptr, d[1].ptr, d[2].ptr, d[3].ptr, c, n, r, 0, zk.HASH_KECCAK, 0))
        keep.append((x, d))
    zk.commit_batch([SimpleNamespace(job=lambda j=j: j) for j in jobs])
    for (c, n, r), (x, d) in zip(shapes, keep):
        rows = ob.transpose_rev(ob.lde(x % np.uint64(P), n, r, c), n + r, c)
        assert np.array_equal(d[1].to_host(), rows), (c, n, r)


# The two-launch transforms: every split of the stages, whole and partial
# chunks of columns, the smallest batch that takes them and the one below,
# rates whose blocks share an output run; then with the scratch given back.
@pytest.mark.parametrize("lg,B", [(15, 7), (15, 8), (16, 4), (17, 3), (18, 1), (19, 3), (20, 1), (20, 17)])
@pytest.mark.parametrize("inverse,coset", [(False, False), (False, True), (True, False), (True, True)])
def test_two_launch_ntt_vs_oracle(zk, lg, B, inverse, coset):
    print(f"ntt lg={lg} B={B} inverse={inverse} coset={coset}", flush=True)
    x = rare_words(B << lg, 5 * lg + B) if lg < 18 else ob.canonical(B << lg, 5 * lg + B)
    buf = x.copy()
    (zk.intt_batch if inverse else zk.ntt_batch)(0, buf, lg, zk.NTTConfig(batches=B, with_coset=coset))
    assert np.array_equal(buf, ob.ntt(x % np.uint64(P), lg, B, inverse, coset))


@pytest.mark.parametrize("lg_n,rate,B", [(15, 3, 1), (15, 5, 3), (16, 2, 2), (17, 3, 1), (18, 1, 2), (19, 1, 1), (20, 2, 1), (20, 4, 1)])
@pytest.mark.parametrize("inverse,coset", [(False, True), (True, False), (True, True)])
def test_two_launch_lde_vs_oracle(zk, lg_n, rate, B, inverse, coset):
    print(f"lde lg_n={lg_n} rate={rate} B={B} inverse={inverse} coset={coset}", flush=True)
    x = ob.canonical(B << lg_n, lg_n + 11 * rate + B)
    out = np.zeros(B << (lg_n + rate), np.uint64)
    zk._check(zk.lib.zkx_commit_trim(0))
    zk.lde_batch(0, out, x, lg_n, zk.NTTConfig(batches=B, extension_rate_bits=rate, with_coset=coset),
                 direction=zk.INVERSE if inverse else zk.FORWARD)
    assert np.array_equal(out, ob.lde(x, lg_n, rate, B, inverse=inverse, coset=coset))
