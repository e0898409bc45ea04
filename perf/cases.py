"""Workloads that the library's speed is measured on, through its Python entry points.

Four kinds of work, each over the range a prover or a proof service has it do:

* "commit": zeknox_amd.commit_batch, one job or many of one shape (coefficients
  in, leaf rows, digests and caps out), or the mixed batch of
  zeknox_amd.workloads;
* "plain": the C-ABI sequence that the reference's wrappers call for one
  commitment: lde_batch, transpose_rev_batch, fill_digests_buf_linear_gpu_with_gpu_ptr;
* "merkle": a Merkle forest alone over leaf rows that are on the device;
* "ntt": lone transforms (values to coefficients and back, low-degree
  extension with its salt columns).

Every buffer is device memory held by torch (int64 words of uint64 values);
field elements are uniform below p, coset generator 7, cap height 4.
"""
import numpy as np
import torch

import zeknox_amd as zk
from zeknox_amd import workloads

P = zk.P
COSET = 7
HASHES = {"poseidon": zk.HASH_POSEIDON, "poseidon2": zk.HASH_POSEIDON2, "keccak": zk.HASH_KECCAK,
          "monolith": zk.HASH_MONOLITH, "poseidon_bn128": zk.HASH_POSEIDON_BN128}


def listed():
    return [
        # a small circuit's commitment, on its own: latency and launches
        {"name": "commit_20x2e10_r1", "kind": "commit", "hash": "poseidon", "jobs": 1, "cols": 20, "lg_n": 10,
         "rate": 1, "cap": 4},
        # the headline commitment (a plonky2 trace of 135 wires), one at a time
        {"name": "commit_135x2e15_r3", "kind": "commit", "hash": "poseidon", "jobs": 1, "cols": 135, "lg_n": 15,
         "rate": 3, "cap": 4},
        # a prover farm's step: 32 of them in one call
        {"name": "commit_135x2e15_r3_x32", "kind": "commit", "hash": "poseidon", "jobs": 32, "cols": 135, "lg_n": 15,
         "rate": 3, "cap": 4},
        # commitments of many proofs of different sizes in one call
        {"name": "commit_mixed64", "kind": "mixed", "seed": 3, "jobs": 64},
        # a wide and long trace with Poseidon2 (one of the large batch's jobs)
        {"name": "commit_p2_400x2e20_r1", "kind": "commit", "hash": "poseidon2", "jobs": 1, "cols": 400, "lg_n": 20,
         "rate": 1, "cap": 4},
        # the served stream's median request, four packed into a batch
        {"name": "commit_p2_201x2e14_r2_x4", "kind": "commit", "hash": "poseidon2", "jobs": 4, "cols": 201,
         "lg_n": 14, "rate": 2, "cap": 4},
        # the headline commitment through the reference's own entry points
        {"name": "plain_135x2e15_r3", "kind": "plain", "hash": "poseidon", "cols": 135, "lg_n": 15, "rate": 3,
         "cap": 4},
        # the smallest forest that the reference publishes a time for
        {"name": "merkle_135x2e13", "kind": "merkle", "hash": "poseidon", "lg_leaves": 13, "leaf": 135, "cap": 4},
        # the largest of those, with Poseidon2
        {"name": "merkle_p2_135x2e15", "kind": "merkle", "hash": "poseidon2", "lg_leaves": 15, "leaf": 135, "cap": 4},
        # a large forest for an on-chain verifier
        {"name": "merkle_keccak_135x2e20", "kind": "merkle", "hash": "keccak", "lg_leaves": 20, "leaf": 135,
         "cap": 4},
        # large forward transforms, natural order
        {"name": "ntt_64x2e20", "kind": "ntt", "dir": "forward", "cols": 64, "lg_n": 20, "rate": 0, "salt": 0,
         "coset": False},
        # values of a small odd-width trace back to coefficients
        {"name": "intt_101x2e13", "kind": "ntt", "dir": "inverse", "cols": 101, "lg_n": 13, "rate": 0, "salt": 0,
         "coset": False},
    ]


def _spread(rng, low, high):
    """A whole number of [low, high], even over its logarithm."""
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    kind = rng.choice(["commit", "commit", "mixed", "plain", "merkle", "merkle", "ntt"])
    if kind == "mixed":
        return {"kind": "mixed", "seed": rng.randrange(1, 1 << 20), "jobs": _spread(rng, 2, 64)}
    if kind == "ntt":
        # at most 2^26 words of result
        lg_n, rate = rng.randint(3, 19), rng.choice([0, 0, 0, 1, 2, 3])
        most = min(400, 1 << (26 - lg_n - rate))
        inverse = rng.random() < 0.4
        return {"kind": "ntt", "dir": "inverse" if inverse else "forward", "cols": _spread(rng, 1, most), "lg_n": lg_n,
                "rate": rate, "salt": rng.choice([0, 4]) if rate else 0, "coset": rng.random() < 0.5}
    if kind == "merkle":
        name = rng.choice(["poseidon", "poseidon2", "poseidon", "poseidon2", "keccak", "monolith", "poseidon_bn128"])
        lg, leaf = rng.randint(4, 15 if name == "poseidon_bn128" else 20), _spread(rng, 1, 400)
        if name == "poseidon_bn128":
            leaf = min(leaf, 135)
        return {"kind": "merkle", "hash": name, "lg_leaves": lg, "leaf": leaf, "cap": rng.randint(0, 4)}
    name = rng.choice(["poseidon", "poseidon2", "poseidon", "poseidon2", "poseidon", "poseidon2", "keccak", "monolith"])
    lg_n, rate, cols = rng.randint(6, 18), rng.randint(1, 3), _spread(rng, 2, 400)
    lg_n = min(lg_n, 20 - rate)
    case = {"kind": kind, "hash": name, "cols": cols, "lg_n": lg_n, "rate": rate, "cap": rng.randint(0, 4)}
    if kind == "commit":
        # batches of at most 2^28 words of leaf rows
        case["jobs"] = _spread(rng, 1, max(1, min(32, (1 << 28) // (cols << (lg_n + rate)))))
    return case


def _elements(count, seed):
    """`count` field elements, uniform below p (the high word never 2^32 - 1)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    hi = torch.randint(0, (1 << 32) - 1, (count,), generator=g, device="cuda", dtype=torch.int64)
    hi <<= 32
    hi |= torch.randint(0, 1 << 32, (count,), generator=g, device="cuda", dtype=torch.int64)
    return hi


def _words(count):
    return torch.zeros(max(count, 1), device="cuda", dtype=torch.int64)


class _Job:
    """One commitment on torch buffers, as zeknox_amd.commit_batch takes it."""

    def __init__(self, *fields):
        self.fields = fields

    def job(self):
        return zk.CommitJob(*self.fields, 0)


def _shapes(case):
    """(cols, lg_n, rate, cap height, hash) of each job."""
    if case["kind"] == "mixed":
        return [(c, n, r, workloads.CAP_HEIGHT, h) for c, n, r, h, _ in workloads.mixed_batch_jobs(case["seed"], case["jobs"])]
    return [(case["cols"], case["lg_n"], case["rate"], case["cap"], HASHES[case["hash"]])] * case.get("jobs", 1)


def _digests(leaves, cap):
    return 2 * (leaves - (1 << cap))


def _coset(lg):
    zk.init_coset_rs(0, lg, COSET)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("commit", "mixed"):
        # each kind of buffer in one allocation, jobs one after another
        shapes = _shapes(case)
        _coset(max(n + r for _, n, r, _, _ in shapes))
        ins = [c << n for c, n, r, h, t in shapes]
        rows = [c << (n + r) for c, n, r, h, t in shapes]
        digs = [4 * _digests(1 << (n + r), h) for c, n, r, h, t in shapes]
        caps = [4 << h for c, n, r, h, t in shapes]
        coeffs = _elements(sum(ins), seed)
        out = {"leaves": _words(sum(rows)), "digests": _words(sum(digs)), "caps": _words(sum(caps))}
        jobs, at = [], [0, 0, 0, 0]
        for k, (c, n, r, h, t) in enumerate(shapes):
            base = (coeffs, out["leaves"], out["digests"], out["caps"])
            jobs.append(_Job(*[b.data_ptr() + 8 * a for b, a in zip(base, at)], c, n, r, h, t))
            at = [a + s[k] for a, s in zip(at, (ins, rows, digs, caps))]
        return {"kind": "commit", "jobs": jobs, "coeffs": coeffs, "out": out}
    if kind == "plain":
        lg, cols = case["lg_n"] + case["rate"], case["cols"]
        _coset(lg)
        return {"kind": kind, "coeffs": _elements(cols << case["lg_n"], seed), "lg_n": case["lg_n"], "lg": lg,
                "cols": cols, "cap": case["cap"], "hash": HASHES[case["hash"]],
                "lde_cfg": zk.NTTConfig(batches=cols, extension_rate_bits=case["rate"], with_coset=True,
                                        are_inputs_on_device=True, are_outputs_on_device=True),
                "tr_cfg": zk.TransposeConfig(batches=cols, are_inputs_on_device=True, are_outputs_on_device=True),
                "lde": _words(cols << lg), "leaves": _words(cols << lg),
                "digests": _words(4 * _digests(1 << lg, case["cap"])), "caps": _words(4 << case["cap"])}
    if kind == "merkle":
        n = 1 << case["lg_leaves"]
        return {"kind": kind, "leaves": _elements(n * case["leaf"], seed), "n": n, "leaf": case["leaf"],
                "cap": case["cap"], "hash": HASHES[case["hash"]], "digests": _words(4 * _digests(n, case["cap"])),
                "caps": _words(4 << case["cap"])}
    lg = case["lg_n"] + case["rate"]
    if case["coset"]:
        _coset(lg)
    return {"kind": kind, "rate": case["rate"], "inverse": case["dir"] == "inverse", "lg_n": case["lg_n"], "seed": seed,
            "values": _elements(case["cols"] << case["lg_n"], seed),
            "out": _words((case["cols"] + case["salt"]) << lg) if case["rate"] else None,
            "cfg": zk.NTTConfig(batches=case["cols"], extension_rate_bits=case["rate"], with_coset=case["coset"],
                                salt_size=case["salt"], are_inputs_on_device=True, are_outputs_on_device=True)}


def _forest(s):
    n, caps = (1 << s["lg"]) if "lg" in s else s["n"], 1 << s["cap"]
    zk.fill_digests_buf_linear_gpu_with_gpu_ptr(s["digests"].data_ptr(), s["caps"].data_ptr(), s["leaves"].data_ptr(),
                                                2 * (n - caps), caps, n, s.get("leaf", s.get("cols")), s["cap"],
                                                s["hash"], 0)


def run(state):
    kind = state["kind"]
    if kind == "commit":
        zk.commit_batch(state["jobs"])
        return state["out"]
    if kind == "plain":
        zk.lde_batch(0, state["lde"].data_ptr(), state["coeffs"].data_ptr(), state["lg_n"], state["lde_cfg"])
        zk.transpose_rev_batch(0, state["leaves"].data_ptr(), state["lde"].data_ptr(), state["lg"], state["tr_cfg"])
        _forest(state)
        return {k: state[k] for k in ("lde", "leaves", "digests", "caps")}
    if kind == "merkle":
        _forest(state)
        return {"digests": state["digests"], "caps": state["caps"]}
    if state["rate"]:
        zk.lde_batch_seeded(0, state["out"].data_ptr(), state["values"].data_ptr(), state["lg_n"], state["cfg"],
                            state["seed"], zk.INVERSE if state["inverse"] else zk.FORWARD)
        return state["out"]
    # in place, as the entry point has it: a next pass transforms this one's result
    (zk.intt_batch if state["inverse"] else zk.ntt_batch)(0, state["values"].data_ptr(), state["lg_n"], state["cfg"])
    return state["values"]


# 32-bit integer operations (a multiply-add is two) that one permutation's
# definition holds: 64-bit field products at 6 multiply-adds (4 for the
# product, 2 for the reduction), small-coefficient products at 2.
def _products(full, small):
    return 2 * (6 * full + 2 * small)


_PERM_OPS = {
    zk.HASH_POSEIDON: _products(118 * 4, 30 * 144),      # 8 full and 22 partial rounds of x^7; 12 x 12 layers
    zk.HASH_POSEIDON2: _products(118 * 4 + 22 * 12, 9 * 48),
    zk.HASH_MONOLITH: _products(6 * 12, 7 * 144),
    zk.HASH_KECCAK: 24 * 25 * 12,                        # theta, rho and chi, two words a lane
    zk.HASH_POSEIDON_BN128: 2 * 1040 * 136,              # 254-bit products of 136 multiply-adds
}


def _hash_work(leaves, leaf, cap, kind):
    """(permutations, words of digests and caps) of one forest."""
    width = 17 if kind == zk.HASH_KECCAK else 8
    per_leaf = 0 if leaf <= 4 and kind != zk.HASH_KECCAK else -(-leaf // width)
    return leaves * per_leaf + leaves - (1 << cap), 4 * (_digests(leaves, cap) + (1 << cap))


def work(case):
    kind = case["kind"]
    if kind == "ntt":
        n, wide = case["cols"] << case["lg_n"], (case["cols"] + case["salt"]) << (case["lg_n"] + case["rate"])
        lg = case["lg_n"] + case["rate"]
        return {"bytes": 8 * (n + wide), "flops": _products((case["cols"] << lg) * case["lg_n"] // 2, 0)}
    if kind == "merkle":
        n = 1 << case["lg_leaves"]
        perms, words = _hash_work(n, case["leaf"], case["cap"], HASHES[case["hash"]])
        return {"bytes": 8 * (n * case["leaf"] + words), "flops": perms * _PERM_OPS[HASHES[case["hash"]]]}
    total = {"bytes": 0, "flops": 0}
    for c, n, r, h, t in _shapes(case):
        perms, words = _hash_work(1 << (n + r), c, h, t)
        rows = c << (n + r)
        # the plain sequence hands back the extension as well as its rows
        total["bytes"] += 8 * ((c << n) + rows * (2 if kind == "plain" else 1) + words)
        total["flops"] += perms * _PERM_OPS[t] + _products(rows * n // 2, 0)
    return total


# ---- the transforms again, from their definition, in numpy ------------------

def _mul(a, b):
    """a * b mod p (uint64 arrays, 128-bit products in 32-bit halves)."""
    m, eps = np.uint64(0xFFFFFFFF), np.uint64(0xFFFFFFFF)
    s, p = np.uint64(32), np.uint64(P)
    a0, a1, b0, b1 = a & m, a >> s, b & m, b >> s
    t0 = a0 * b0
    t1 = a1 * b0 + (t0 >> s)
    t2 = a0 * b1 + (t1 & m)
    lo, hi = (t0 & m) | (t2 << s), a1 * b1 + (t1 >> s) + (t2 >> s)
    # hi * 2^64 = h0 * (2^32 - 1) - h1
    h0, h1 = hi & m, hi >> s
    x = lo - h1
    x = np.where(lo < h1, x - eps, x)
    y = h0 * eps
    z = x + y
    z = np.where(z < y, z + eps, z)
    return np.where(z >= p, z - p, z)


def _add(a, b):
    s = a + b
    s = np.where(s < a, s + np.uint64(0xFFFFFFFF), s)
    return np.where(s >= np.uint64(P), s - np.uint64(P), s)


def _sub(a, b):
    d = a - b
    return np.where(a < b, d - np.uint64(0xFFFFFFFF), d)


def _powers(base, n):
    out = np.ones(n, np.uint64)
    k = 1
    while k < n:
        out[k:2 * k] = _mul(out[:min(k, n - k)], np.uint64(pow(base, k, P)))
        k *= 2
    return out


def _transform(x, inverse):
    """Values of x's rows (columns of coefficients) over the 2^lg-th roots, natural order."""
    lg = x.shape[1].bit_length() - 1
    w = pow(1753635133440165772, 1 << (32 - lg), P)
    if inverse:
        w = pow(w, P - 2, P)
    rev = np.zeros(1, np.int64)
    for _ in range(lg):
        rev = np.concatenate([2 * rev, 2 * rev + 1])
    x = x[:, rev]
    for k in range(lg):
        half = 1 << k
        tw = _powers(pow(w, 1 << (lg - k - 1), P), half)
        y = x.reshape(x.shape[0], -1, 2, half)
        t = _mul(y[:, :, 1], tw)
        x = np.stack([_add(y[:, :, 0], t), _sub(y[:, :, 0], t)], 2).reshape(x.shape[0], -1)
    return _mul(x, np.uint64(pow(x.shape[1], P - 2, P))) if inverse else x


def exact(case, seed):
    """The lone transforms of up to 2^21 words; hashes have no value but their own, and the salt is the library's stream."""
    if case["kind"] != "ntt" or case["salt"] or case["cols"] << (case["lg_n"] + case["rate"]) > 1 << 21:
        return None
    x = _elements(case["cols"] << case["lg_n"], seed).cpu().numpy().view(np.uint64).reshape(case["cols"], -1)
    inverse, n = case["dir"] == "inverse", x.shape[1] << case["rate"]
    x = np.concatenate([x, np.zeros((x.shape[0], n - x.shape[1]), np.uint64)], 1)
    shift = _powers(COSET, n)
    if case["coset"] and not inverse:
        x = _mul(x, shift)
    x = _transform(x, inverse)
    if case["coset"] and inverse:
        x = _mul(x, shift)
    return torch.from_numpy(np.ascontiguousarray(x.reshape(-1)).view(np.int64))
