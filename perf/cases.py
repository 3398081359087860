"""The work that a user of this backend has it do, as cases that can be timed one by one.

Every case is one operation of a STARK prover over M31 (or one whole proof), called through the
library's own entry points: the C ABI of include/stwo_hip.h or its Python binding.  The kinds
are the steps of a proof in the order a prover meets them:

  twiddles      the tree of a domain and its inverses, once per domain size
  interpolate   circle evaluations to coefficients, in place (encode)
  evaluate      coefficients to a larger circle domain (decode / extend)
  commit        low-degree extension of one trace and its Merkle tree
  commit_mixed  the same over columns of many sizes with mixed-degree injection
  oods          every column at a few out-of-domain points
  quotients     DEEP quotients of sampled columns
  fri           commit, draw, fold, layer after layer; each challenge needs the last root
  prove         a whole wide-Fibonacci proof
  batch_inverse, bit_reverse   the column operations that the reference benchmarks

Inputs are uniform field elements, which is what committed traces, coefficients and random
linear combinations look like to these kernels.  Outputs are whole numbers (field elements and
hash words), so they are compared word for word.
"""
import ctypes
import hashlib
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stwo-gpu_amd"))
import stwo_hip as S  # noqa: E402

P = S.P
# columns of one trace lie in one buffer; each starts this many words after the end of the one
# before, so that columns read together at one row do not fall on the same memory channels
# (the prover lays its own columns out in the same way)
COL_PAD = 1088


def listed():
    return [
        # the benchmark's headline: a wide trace extended and committed; large enough to be bound by the kernels
        {"name": "commit_256x2e20", "kind": "commit", "n_cols": 256, "log": 20, "blowup": 1, "autotune": True},
        # a small statement's trace, where launches and gaps between them count
        {"name": "commit_16x2e16", "kind": "commit", "n_cols": 16, "log": 16, "blowup": 1, "autotune": False},
        # a machine's trace: hundreds of components of very different heights in one tree
        {"name": "commit_mixed_1200", "kind": "commit_mixed", "n_cols": 1200, "min_log": 10, "max_log": 21,
         "blowup": 1},
        # the reference's own benches of the transforms: very many short columns
        {"name": "interpolate_65536x2e10", "kind": "interpolate", "n_cols": 1 << 16, "log": 10},
        {"name": "evaluate_65536x2e10_x4", "kind": "evaluate", "n_cols": 1 << 16, "log": 10, "blowup": 2},
        # out-of-domain sampling of a middle-sized trace at a point and at the next row's
        {"name": "oods_256x2e18_2pt", "kind": "oods", "n_cols": 256, "log": 18, "points": 2},
        # quotients of a trace whose columns are sampled at one to three points
        {"name": "quotients_200x2e21_3pt", "kind": "quotients", "n_cols": 200, "log": 21, "points": 3},
        # FRI of a 2^20 quotient domain: a chain of ever smaller trees and folds, each waiting for a root
        {"name": "fri_2e20", "kind": "fri", "log": 20, "last_log": 4},
        # the smallest whole proofs, bound by latency from end to end
        {"name": "prove_32x2e12", "kind": "prove", "n_cols": 32, "log": 12, "queries": 3, "pow_bits": 10},
        # the tree that serves every domain up to 2^23 points
        {"name": "twiddles_2e22", "kind": "twiddles", "log": 22},
        # the inverses of 2^24 extension field elements
        {"name": "batch_inverse_qm31_2e24", "kind": "batch_inverse", "field": "qm31", "n": 1 << 24},
        # the reference's bit reversal bench: one column as large as they get
        {"name": "bit_reverse_m31_2e28", "kind": "bit_reverse", "field": "m31", "log": 28},
    ]


def _log_uniform(rng, lo, hi):
    """A whole number of lo .. hi, uniform in its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["commit", "commit", "commit_mixed", "interpolate", "evaluate", "oods", "quotients", "fri",
                       "prove", "twiddles", "batch_inverse", "bit_reverse"])
    if kind == "commit":
        log, blowup = rng.randint(5, 23), rng.choice([1, 1, 1, 2, 3])
        return {"kind": kind, "n_cols": _log_uniform(rng, 1, min(700, 1 << (29 - blowup - log) if log < 29 else 1)),
                "log": log, "blowup": blowup, "autotune": rng.random() < 0.5}
    if kind == "commit_mixed":
        lo = rng.randint(4, 12)
        return {"kind": kind, "n_cols": _log_uniform(rng, 40, 1500), "min_log": lo,
                "max_log": rng.randint(lo + 4, 22), "blowup": rng.choice([1, 1, 2])}
    if kind == "interpolate":
        log = rng.randint(3, 22)
        return {"kind": kind, "n_cols": _log_uniform(rng, 1, min(1 << 16, 1 << (26 - log))), "log": log}
    if kind == "evaluate":
        log, blowup = rng.randint(3, 20), rng.choice([0, 1, 1, 2, 2, 3, 4])
        return {"kind": kind, "n_cols": _log_uniform(rng, 1, min(1 << 16, 1 << (28 - log - blowup))), "log": log,
                "blowup": blowup}
    if kind == "oods":
        log = rng.randint(6, 22)
        return {"kind": kind, "n_cols": _log_uniform(rng, 1, min(1000, 1 << (28 - log))), "log": log,
                "points": rng.randint(1, 3)}
    if kind == "quotients":
        log = rng.randint(6, 22)
        return {"kind": kind, "n_cols": _log_uniform(rng, 1, min(600, 1 << (28 - log))), "log": log,
                "points": rng.choice([1, 2, 2, 3, 4, 6])}
    if kind == "fri":
        return {"kind": kind, "log": rng.randint(8, 23), "last_log": rng.randint(2, 6)}
    if kind == "prove":
        log = rng.randint(5, 18)
        return {"kind": kind, "n_cols": _log_uniform(rng, 3, min(700, 1 << (26 - log))), "log": log,
                "queries": rng.randint(3, 30), "pow_bits": rng.randint(0, 12)}
    if kind == "twiddles":
        return {"kind": kind, "log": rng.randint(4, 24)}
    if kind == "batch_inverse":
        field = rng.choice(["m31", "qm31"])
        return {"kind": kind, "field": field, "n": _log_uniform(rng, 100, 1 << (28 if field == "m31" else 25))}
    field = rng.choice(["m31", "qm31"])
    return {"kind": kind, "field": field, "log": rng.randint(5, 28 if field == "m31" else 26)}


# ------------------------------------------------------------------ inputs
def _mixed_logs(case):
    """Column heights with weights proportional to 1 / height, the tallest column always there."""
    ks = np.arange(case["min_log"], case["max_log"] + 1)
    w = 2.0 ** -ks
    n = case["n_cols"]
    logs = [int(k) for k in np.random.default_rng(0x5EED0004).choice(ks, n, p=w / w.sum())]
    logs[n // 2] = case["max_log"]
    return logs


def _uniform(seed, *shape):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randint(0, P, shape, dtype=torch.int32, device="cuda", generator=g)


class _Columns:
    """Columns in one buffer: `buf` as a tensor, `cols` as the library's column type."""

    def __init__(self, logs, pad=COL_PAD, seed=None):
        offs, at = [], 0
        for l in logs:
            offs.append(at)
            at += max(1 << l, 128) + pad  # 512-byte starts, as separate allocations have
        # the padding is part of the buffer: no kernel writes it
        self.buf = torch.zeros(at, dtype=torch.int32, device="cuda") if seed is None else _uniform(seed, at)
        self.cols = [S.BaseFieldVec.view(self.buf.data_ptr() + 4 * o, 1 << l) for o, l in zip(offs, logs)]


class _OnDevice:
    """Device memory of the library as an array that torch can look at without a copy."""

    def __init__(self, owner, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<i4", "data": (owner.ptr, False), "version": 2}


def _tensor(owner, *shape):
    return torch.as_tensor(_OnDevice(owner, shape), device="cuda")


def _secure_tensor(t):
    """The rows of a (4, n) tensor as a secure column."""
    n = t.shape[1]
    return S.SecureColumn([S.BaseFieldVec.view(t.data_ptr() + 4 * n * k, n) for k in range(4)])


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind in ("commit", "commit_mixed"):
        logs = [case["log"]] * case["n_cols"] if kind == "commit" else _mixed_logs(case)
        b = case["blowup"]
        evals, coeffs, ldes = _Columns(logs, seed=seed), _Columns(logs), _Columns([l + b for l in logs])
        coset = S.canonic_half_coset(max(logs) + b)
        tw, itw = S.cached_twiddles(coset)
        torch.cuda.synchronize()  # the plan's first runs are on the library's stream
        plan = S.CommitPlan(evals.cols, coeffs.cols, ldes.cols, logs, b, tw, itw, 1 << coset.log_size,
                            autotune=case.get("autotune", True))
        st.update(plan=plan, keep=evals,
                  out={"coeffs": coeffs.buf, "lde": ldes.buf,
                       "layers": [_tensor(l, l.size, 8) for l in plan.layers]})
    elif kind == "interpolate":
        n, log = case["n_cols"], case["log"]
        st["values"] = _uniform(seed, n, 1 << log)
        st["ptrs"] = S._ptr_array([st["values"].data_ptr() + (c << (log + 2)) for c in range(n)])
        st["tree"] = S.precompute_twiddles(S.canonic_half_coset(log))
    elif kind == "evaluate":
        n, log, m = case["n_cols"], case["log"], case["log"] + case["blowup"]
        st["coeffs"] = _uniform(seed, n, 1 << log)
        st["out"] = torch.zeros(n, 1 << m, dtype=torch.int32, device="cuda")
        st["src"] = S._ptr_array([st["coeffs"].data_ptr() + (c << (log + 2)) for c in range(n)])
        st["dst"] = S._ptr_array([st["out"].data_ptr() + (c << (m + 2)) for c in range(n)])
        st["logs"] = np.full(n, log, np.uint32), np.full(n, m, np.uint32)
        coset = S.canonic_half_coset(m)
        st["tw"], st["tree_len"] = S.cached_twiddles(coset)[0], 1 << coset.log_size
    elif kind == "oods":
        st["columns"] = _Columns([case["log"]] * case["n_cols"], seed=seed)
        rng = np.random.default_rng(seed)
        pts = [S.random_circle_point_qm31(rng) for _ in range(case["points"])]
        st["points"] = (S.PointQM31 * len(pts))(*[S.PointQM31(S.qm31(x), S.qm31(y)) for x, y in pts])
        st["ptrs"] = S.column_pointers(st["columns"].cols)
    elif kind == "quotients":
        c = st["columns"] = _Columns([case["log"]] * case["n_cols"], seed=seed)
        rng = np.random.default_rng(seed)
        batches = [(S.random_circle_point_qm31(rng), []) for _ in range(case["points"])]
        for i in range(case["n_cols"]):  # a column is sampled at some of the points, one to three
            k = int(rng.integers(1, min(3, len(batches)) + 1))
            for j in sorted(rng.choice(len(batches), size=k, replace=False)):
                batches[j][1].append((i, S.random_qm31(rng)))
        st["samples"] = S.QuotientSamples([b for b in batches if b[1]])
        st["rc"] = S.random_qm31(rng)
        st["out"] = torch.zeros(4, 1 << case["log"], dtype=torch.int32, device="cuda")
        st["secure"] = _secure_tensor(st["out"])
        st["ptrs"] = S.column_pointers(c.cols)
    elif kind == "fri":
        log, last = case["log"], min(case["last_log"], case["log"] - 2)
        st["circle"] = _uniform(seed, 4, 1 << log)
        st["base"] = _uniform(seed + 1, 4, 1 << (log - 1))  # what larger columns have folded into the first line layer
        st["lines"] = [torch.zeros(4, 1 << k, dtype=torch.int32, device="cuda") for k in range(log - 1, last - 1, -1)]
        coset = S.canonic_half_coset(log)
        st["itw"], st["tree_len"] = S.cached_twiddles(coset)[1], 1 << coset.log_size
        layers = [st["circle"]] + st["lines"]
        st["secure"] = [_secure_tensor(t) for t in layers]
        st["trees"] = [S.MerkleTree(s.columns) for s in st["secure"][:-1]]
        n = 4 << (log - 1)
        st["copy"] = S.BaseFieldVec.view(st["lines"][0].data_ptr(), n), S.BaseFieldVec.view(st["base"].data_ptr(), n)
    elif kind == "prove":
        st["params"] = S.wide_fib_params(case["n_cols"], case["log"], case["queries"], case["pow_bits"])
        st["seed"] = seed
    elif kind == "twiddles":
        # the tree of a coset that the seed chooses (a proof's domains are canonic; their trees are computed alike)
        log = case["log"]
        start = int(np.random.default_rng(seed).integers(0, 1 << 30)) * 2 + 1
        st["coset"] = S.Coset(start << (29 - log) & 0x7fffffff, 1 << (31 - log), log)
    elif kind == "batch_inverse":
        n = case["n"]
        st["from"] = _uniform(seed, n, 4) if case["field"] == "qm31" else _uniform(seed, n)
        st["from"].clamp_(min=1)  # every element has an inverse
        st["to"] = torch.zeros_like(st["from"])
    elif kind == "bit_reverse":
        st["values"] = _uniform(seed, 1 << case["log"], 4) if case["field"] == "qm31" else _uniform(seed, 1 << case["log"])
    else:
        raise ValueError(kind)
    torch.cuda.synchronize()  # the library works on a stream of its own
    return st


# ------------------------------------------------------------------ one pass
def run(st):
    case = st["case"]
    kind = case["kind"]
    L = S.lib()
    if kind in ("commit", "commit_mixed"):
        st["plan"].run()
        return st["out"]
    if kind == "interpolate":
        t = st["tree"].itwiddles
        L.interpolate_columns(1 << (case["log"] - 1), st["ptrs"], t.ptr, t.size, case["n_cols"], 1 << case["log"])
        S.check()
        return st["values"]
    if kind == "evaluate":
        cl, el = st["logs"]
        S.check(L.stwo_hip_evaluate_columns_async(st["src"], cl.ctypes.data_as(S.u32p), st["dst"],
                                                  el.ctypes.data_as(S.u32p), case["n_cols"], st["tw"],
                                                  st["tree_len"]))
        return st["out"]
    if kind == "oods":
        n, k = case["n_cols"], case["points"]
        out = np.zeros((k, n, 4), np.uint32)
        S.check(L.stwo_hip_eval_at_points_columns(st["ptrs"], n, case["log"], ctypes.cast(st["points"], S.vp), k,
                                                  out.ctypes.data))
        return out
    if kind == "quotients":
        S.accumulate_quotients_async(S.canonic_half_coset(case["log"]), st["columns"].cols, st["rc"], st["samples"],
                                     st["secure"], col_ptrs=st["ptrs"])
        return st["out"]
    if kind == "fri":
        return _fri(st)
    if kind == "prove":
        return S.wide_fib_prove(st["params"], st["seed"])
    if kind == "twiddles":
        tree = S.precompute_twiddles(st["coset"])
        return [_tensor(t, t.size) for t in (tree.twiddles, tree.itwiddles)]
    if kind == "batch_inverse":
        f = L.batch_inverse_secure_field if case["field"] == "qm31" else L.batch_inverse_base_field
        f(st["from"].data_ptr(), st["to"].data_ptr(), case["n"])
        S.check()
        return st["to"]
    f = L.bit_reverse_secure_field if case["field"] == "qm31" else L.bit_reverse_base_field
    f(st["values"].data_ptr(), 1 << case["log"])
    S.check()
    return st["values"]


def _fri(st):
    """Commit a layer, draw the folding coefficient from its root, fold; until the last layer."""
    layers, digest, roots = st["secure"], b"", []
    S.device_copy(*st["copy"])
    for j, tree in enumerate(st["trees"]):
        root = tree.commit_async().root()
        roots.append(root)
        digest = hashlib.blake2s(digest + root.tobytes()).digest()
        alpha = [w % P for w in np.frombuffer(digest[:16], np.uint32).tolist()]
        n = len(layers[j])
        if j == 0:
            S.fold_circle_into_line_async(layers[1], layers[0], alpha, st["itw"], st["tree_len"] - n // 2)
        else:
            S.fold_line_async(layers[j], layers[j + 1], alpha, st["itw"], st["tree_len"] - n)
    return {"roots": np.stack(roots), "lines": st["lines"], "last": layers[-1].to_numpy()}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    """Bytes read and written by one pass if every input is read once and every output is written once."""
    kind = case["kind"]
    if kind == "commit":
        n, m = 1 << case["log"], 1 << (case["log"] + case["blowup"])
        b = case["n_cols"] * 4 * (2 * n + m) + 64 * m
    elif kind == "commit_mixed":
        logs = _mixed_logs(case)
        b = sum(4 * ((2 << l) + (1 << (l + case["blowup"]))) for l in logs) + (64 << (max(logs) + case["blowup"]))
    elif kind == "interpolate":
        b = 8 * case["n_cols"] << case["log"]
    elif kind == "evaluate":
        b = 4 * case["n_cols"] * ((1 << case["log"]) + (1 << (case["log"] + case["blowup"])))
    elif kind == "oods":
        b = 4 * case["n_cols"] << case["log"]
    elif kind == "quotients":
        b = (4 * case["n_cols"] + 16) << case["log"]
    elif kind == "fri":
        b = sum((16 + 64) << k for k in range(case["log"] + 1))  # every layer and its tree
    elif kind == "prove":
        # the trace's coefficients and extension written once, hashed and sampled
        b = 4 * case["n_cols"] * 5 << case["log"]
    elif kind == "twiddles":
        b = 8 << case["log"]
    elif kind == "batch_inverse":
        b = 2 * case["n"] * (16 if case["field"] == "qm31" else 4)
    else:
        b = 2 * (16 if case["field"] == "qm31" else 4) << case["log"]
    return {"bytes": b, "flops": 0}


# ------------------------------------------------------------------ the results by plain arithmetic
def _mul(a, b):
    return a * b % P  # 64-bit whole numbers: a product of two canonical values is below 2^62


def _pow(a, e):
    r = torch.ones_like(a)
    while e:
        if e & 1:
            r = _mul(r, a)
        a, e = _mul(a, a), e >> 1
    return r


def _cmul(a, b):
    return ((_mul(a[0], b[0]) - _mul(a[1], b[1])) % P, (_mul(a[0], b[1]) + _mul(a[1], b[0])) % P)


def exact(case, seed):
    """run()'s outputs in 64-bit arithmetic for the column operations.  The other kinds' outputs are
    whole numbers too and are compared word for word; their hash trees and transforms would take
    longer than 20 seconds in numpy."""
    if case["kind"] == "bit_reverse":
        v = prepare(case, seed)["values"]
        n, log = v.shape[0], case["log"]
        i = torch.arange(n, device=v.device)
        j = torch.zeros_like(i)
        for b in range(log):
            j |= ((i >> b) & 1) << (log - 1 - b)
        return v[j]
    if case["kind"] == "batch_inverse":
        v = prepare(case, seed)["from"].long()
        if case["field"] == "m31":
            return _pow(v, P - 2).int()
        x, y = (v[:, 0], v[:, 1]), (v[:, 2], v[:, 3])
        xx, yy = _cmul(x, x), _cmul(_cmul(y, y), (2, 1))
        d = ((xx[0] - yy[0]) % P, (xx[1] - yy[1]) % P)  # x^2 - (2 + i) y^2
        norm = _pow((_mul(d[0], d[0]) + _mul(d[1], d[1])) % P, P - 2)
        di = (_mul(d[0], norm), _mul((-d[1]) % P, norm))
        a, b = _cmul(x, di), _cmul(y, di)
        return torch.stack([a[0], a[1], (-b[0]) % P, (-b[1]) % P], 1).int()
    return None
