"""The batched Kronecker calls this library is timed on, through its public entry points.

A case is a dict of plain values. Four kinds of call:

  apply     `kronmult_batched_async` on a batch of the reference harness's kind: every entry has its own input
            and its own factors (the top-left n x n corner of an n x `stride` column-major array), entry k adds
            into output (k * outputs) / nb (tests/utils/utils_cpu.h:79-83). The batch sizes are the reference's
            ASGarD-like count (tests/utils/batch_size.h:8-21) of a (degree, dimension, level).
  operator  `kronmult_batched_terms` / `kronmult_batched_async` on the element pairs of a row and a column list
            (output-major, as ASGarD lists them): shared inputs, shared outputs, factors = blocks of one
            coefficient matrix per dimension and term, picked by the base-16 digits of the element numbers.
  adjoint   `kronmult_batched_adjoint`: gradients of the inputs and of the factors, for a batch of either layout
            ("operator" pairs, or entries with inputs of their own that take `sets` factor sets in turn).
  mixed     `kronmult_batched_grouped`: several (d, n, count) groups in one call, default launch shapes.

A pass clears what it accumulates into, as a program does that computes an operator application or a gradient,
and makes the call on the current stream.
"""
from __future__ import annotations

import math

import torch

from kronmult993_amd import api

DEVICE = "cuda"


# ---- the cases ------------------------------------------------------------------------------------------------

def batch_count(n: int, d: int, level: int, outputs: int = 5) -> int:
    """The reference's batch size for degree n, dimension d and grid level (tests/utils/batch_size.h:8-21)."""
    size = n ** d
    room = (395000000000 - outputs * size) // (size * (2 + d * n * n))
    return min(room, 2 ** level * level ** min(1, d - 1))


def _apply(name, d, n, level, dtype):
    return {"name": name, "kind": "apply", "d": d, "n": n, "nb": batch_count(n, d, level), "stride": 67,
            "outputs": 5, "dtype": dtype}


def listed():
    return [
        # the reference benchmark's "small": 64 entries of 16 values, nothing but call and launch latency
        _apply("small_d2n4_f64", 2, 4, 4, "f64"),
        # its "medium": 384 entries of 216 values, less than one entry per SIMD
        _apply("medium_d3n6_f64", 3, 6, 6, "f64"),
        # its full benchmark (degree 2..10 x dimension 1..6 at level 9): odd degrees with vectors that fit on
        # chip, in both types
        _apply("grid_d5n5_f64", 5, 5, 9, "f64"),
        _apply("grid_d4n7_f32", 4, 7, 9, "f32"),
        # the same grid where one vector is larger than a workgroup keeps on chip
        _apply("grid_d6n6_f32", 6, 6, 9, "f32"),
        # the grid's largest degree and dimension: 656 vectors of a million values
        _apply("grid_d6n10_f64", 6, 10, 9, "f64"),
        # the reference benchmark's "realistic", its one published figure: 3903 vectors of 262144 values
        _apply("realistic_d6n8_f64", 6, 8, 9, "f64"),
        # one application of a 6D operator, the headline benchmark: 128 row x 64 column elements
        {"name": "operator_d6n4_f64", "kind": "operator", "d": 6, "n": 4, "rows": 128, "cols": 64, "terms": 1,
         "dtype": "f64"},
        # the same element pairs with three Kronecker terms, in single precision
        {"name": "operator_d6n4_terms3_f32", "kind": "operator", "d": 6, "n": 4, "rows": 128, "cols": 64,
         "terms": 3, "dtype": "f32"},
        # its gradients
        {"name": "adjoint_d6n4_f64", "kind": "adjoint", "layout": "operator", "d": 6, "n": 4, "rows": 128,
         "cols": 64, "dtype": "f64"},
        # gradients of a batch of ordinary size with an odd degree: 256 factor sets, four entries per output
        {"name": "adjoint_d4n5_f32", "kind": "adjoint", "layout": "entries", "d": 4, "n": 5, "nb": 8192,
         "sets": 256, "per_output": 4, "dtype": "f32"},
        # the elements of an adaptive grid with mixed degrees and dimensions, in one call
        {"name": "mixed_f64", "kind": "mixed",
         "groups": "2,8,20000;3,6,6000;4,4,3000;5,3,1500;6,2,800", "dtype": "f64"},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["apply", "apply", "apply", "operator", "adjoint", "mixed"])
    dtype = rng.choice(["f64", "f32"])
    if kind == "apply":
        d, n = rng.randint(1, 6), rng.randint(2, 10)
        return {"kind": kind, "d": d, "n": n, "nb": _log_int(rng, 4, batch_count(n, d, 9)),
                "stride": rng.choice([n, n + 1, 67]), "outputs": rng.randint(1, 40), "dtype": dtype}
    if kind == "operator":
        d, n = rng.choice([(6, 4), (5, 4), (4, 4), (3, 8), (4, 8), (6, 3), (5, 5), (4, 6), (6, 2), (3, 7)])
        return {"kind": kind, "d": d, "n": n, "rows": _log_int(rng, 4, 160), "cols": _log_int(rng, 4, 96),
                "terms": rng.randint(1, 4), "dtype": dtype}
    if kind == "adjoint":
        d, n = rng.choice([(6, 4), (5, 4), (4, 4), (3, 8), (4, 8), (6, 3), (5, 5), (4, 5), (4, 6), (3, 7), (6, 2)])
        if rng.random() < 0.5:
            return {"kind": kind, "layout": "operator", "d": d, "n": n, "rows": _log_int(rng, 4, 128),
                    "cols": _log_int(rng, 4, 64), "dtype": dtype}
        return {"kind": kind, "layout": "entries", "d": d, "n": n, "nb": _log_int(rng, 16, 8192),
                "sets": rng.randint(1, 512), "per_output": rng.randint(1, 16), "dtype": dtype}
    groups = []
    for _ in range(rng.randint(2, 7)):
        d, n = rng.choice([(2, 8), (3, 6), (4, 4), (5, 3), (6, 2), (2, 5), (3, 4), (3, 7), (4, 3), (5, 4)])
        groups.append(f"{d},{n},{_log_int(rng, 32, 20000)}")
    return {"kind": kind, "groups": ";".join(groups), "dtype": dtype}


# ---- batches: flat pools and element offsets --------------------------------------------------------------------

class _Batch:
    """Pools on the device and each entry's offsets into them (host index tensors)."""

    def __init__(self, d, n, stride, mats, mat_off, inputs, in_off, out_count, out_index):
        self.d, self.n, self.stride, self.size = d, n, stride, n ** d
        self.nb = in_off.numel()
        self.mats, self.mat_off = mats, mat_off          # mat_off [terms * nb * d]
        self.inputs, self.in_off = inputs, in_off
        self.out_count, self.out_index = out_count, out_index

    def pointers(self, pool, off):
        return (pool.data_ptr() + off * pool.element_size()).to(DEVICE)


def _dtype(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _normal(count, dtype, g):
    return torch.randn(count, dtype=dtype, device=DEVICE, generator=g)


def _apply_batch(case, g):
    d, n, nb, stride, outputs = case["d"], case["n"], case["nb"], case["stride"], min(case["outputs"], case["nb"])
    dt, size = _dtype(case), n ** d
    k = torch.arange(nb)
    return _Batch(d, n, stride, _normal(nb * d * n * stride, dt, g), torch.arange(nb * d) * (n * stride),
                  _normal(nb * size, dt, g), k * size, outputs, (k * outputs) // nb)


def _operator_batch(case, g, terms):
    d, n, rows, cols = case["d"], case["n"], case["rows"], case["cols"]
    dt, size, ld = _dtype(case), n ** d, 16 * n
    i = torch.arange(rows).repeat_interleave(cols)
    j = torch.arange(cols).repeat(rows)
    off = []
    for term in range(terms):
        per_mode = []
        for t in range(d):
            r, c = (i >> (4 * t)) & 15, (j >> (4 * t)) & 15
            per_mode.append((term * d + t) * ld * ld + n * r + n * c * ld)
        off.append(torch.stack(per_mode, 1).reshape(-1))
    return _Batch(d, n, ld, _normal(terms * d * ld * ld, dt, g) / 8, torch.cat(off),
                  torch.rand(cols * size, dtype=dt, device=DEVICE, generator=g) * 2 - 1, j * size, rows, i)


def _entries_batch(case, g):
    d, n, nb, sets = case["d"], case["n"], case["nb"], case["sets"]
    dt, size = _dtype(case), n ** d
    k = torch.arange(nb)
    mats = torch.rand(sets * d * n * n, dtype=dt, device=DEVICE, generator=g) * 2 - 1
    off = ((k % sets)[:, None] * d + torch.arange(d)[None, :]) * (n * n)
    per = case["per_output"]
    return _Batch(d, n, n, mats, off.reshape(-1), _normal(nb * size, dt, g), k * size, (nb + per - 1) // per, k // per)


def _group_sizes(case):
    return [tuple(int(v) for v in part.split(",")) for part in case["groups"].split(";")]


def _batches(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "apply":
        return [_apply_batch(case, g)], g
    if kind == "operator":
        return [_operator_batch(case, g, case["terms"])], g
    if kind == "adjoint":
        return [_operator_batch(case, g, 1) if case["layout"] == "operator" else _entries_batch(case, g)], g
    return [_entries_batch({"d": d, "n": n, "nb": nb, "sets": nb, "per_output": 4, "dtype": case["dtype"]}, g)
            for d, n, nb in _group_sizes(case)], g


# ---- preparing and running a case -------------------------------------------------------------------------------

def _workspace(b, per_entry):
    if per_entry <= 0:
        return None, None
    ws = torch.empty(b.nb * per_entry, dtype=b.inputs.dtype, device=DEVICE)
    return ws, b.pointers(ws, torch.arange(b.nb) * per_entry)


def prepare(case, seed):
    """Pools, pointer arrays and the workspaces the calls ask for."""
    batches, g = _batches(case, seed)
    state = {"case": case, "batches": batches}
    if case["kind"] == "adjoint":
        b = batches[0]
        state["gout"] = _normal(b.out_count * b.size, b.inputs.dtype, g)
        state["gin"], state["gmat"] = torch.empty_like(b.inputs), torch.empty_like(b.mats)
        per = api.adjoint_workspace(b.d, b.n, b.inputs.element_size())
        state["ws"], ws_ptrs = _workspace(b, per)
        state["args"] = (b.d, b.n, b.pointers(b.mats, b.mat_off), b.stride, b.pointers(b.inputs, b.in_off),
                         b.pointers(state["gout"], b.out_index * b.size), b.pointers(state["gin"], b.in_off),
                         b.pointers(state["gmat"], b.mat_off), ws_ptrs, b.nb)
        return state
    # one output pool for all groups, so that clearing it is one fill
    total = sum(b.out_count * b.size for b in batches)
    out = torch.empty(total, dtype=batches[0].inputs.dtype, device=DEVICE)
    state["out"], state["ws"], args, at = out, [], [], 0
    for b in batches:
        # vectors that may not stay on chip (64 KiB, factors beside them) need a workspace of one vector per entry
        ws, ws_ptrs = _workspace(b, b.size if b.size * out.element_size() > 48 * 1024 else 0)
        state["ws"].append(ws)
        args.append((b.d, b.n, b.pointers(b.mats, b.mat_off), b.stride, b.pointers(b.inputs, b.in_off),
                     b.pointers(out, at + b.out_index * b.size), ws_ptrs, b.nb))
        at += b.out_count * b.size
    state["args"] = args
    if case["kind"] == "mixed":
        state["groups"] = [api.Group(*a) for a in args]
        state["structs"] = api.grouped_structs(state["groups"], case["dtype"])
    return state


def run(state):
    case = state["case"]
    dtype, stream = case["dtype"], torch.cuda.current_stream()
    if case["kind"] == "adjoint":
        state["gin"].zero_()
        state["gmat"].zero_()
        api.kronmult_batched_adjoint(*state["args"], dtype=dtype, stream=stream, sync=False)
        return [state["gin"], state["gmat"]]
    state["out"].zero_()
    if case["kind"] == "mixed":
        api.kronmult_batched_grouped(state["groups"], dtype=dtype, stream=stream, structs=state["structs"])
    elif case["kind"] == "operator" and case["terms"] > 1:
        d, n, mats, stride, *rest = state["args"][0]
        api.kronmult_batched_terms(d, n, case["terms"], mats, stride, *rest, dtype=dtype, stream=stream, sync=False)
    else:
        api.kronmult_batched_async(*state["args"][0], dtype=dtype, stream=stream)
    return [state["out"]]


# ---- what a pass cannot do without ------------------------------------------------------------------------------

def work(case):
    """Flops of the sweeps; bytes of every distinct input, factor value, output and pointer once."""
    item = 8 if case["dtype"] == "f64" else 4
    kind = case["kind"]
    if kind == "apply":
        shapes = [(case["d"], case["n"], case["nb"], case["nb"], case["nb"], min(case["outputs"], case["nb"]), 1)]
    elif kind == "operator" or (kind == "adjoint" and case["layout"] == "operator"):
        nb, terms = case["rows"] * case["cols"], case.get("terms", 1)
        d = case["d"]
        # distinct blocks: per dimension, the digits that the element numbers take
        blocks = sum(len({(i >> (4 * t)) & 15 for i in range(case["rows"])}) *
                     len({(j >> (4 * t)) & 15 for j in range(case["cols"])}) for t in range(d))
        shapes = [(d, case["n"], nb, blocks * terms / d, case["cols"], case["rows"], terms)]
    elif kind == "adjoint":
        shapes = [(case["d"], case["n"], case["nb"], min(case["sets"], case["nb"]), case["nb"],
                   -(-case["nb"] // case["per_output"]), 1)]
    else:
        shapes = [(d, n, nb, nb, nb, -(-nb // 4), 1) for d, n, nb in _group_sizes(case)]
    flops = nbytes = 0.0
    for d, n, nb, factor_sets, inputs, outputs, terms in shapes:
        size = n ** d
        sweep = 2.0 * d * n * size
        if kind == "adjoint":
            # the forward chain, the transposed chain, one n x n product of unfoldings per factor; cotangents
            # and inputs read, both gradients written
            flops += nb * 3 * sweep
            nbytes += item * (outputs * size + 2 * inputs * size + 2 * factor_sets * d * n * n) + 8 * nb * (2 * d + 3)
        else:
            flops += nb * terms * (sweep + size)
            nbytes += item * (inputs * size + 2 * outputs * size + factor_sets * d * n * n)
            nbytes += 8 * nb * (terms * d + 2)
    return {"bytes": int(nbytes), "flops": int(flops)}


# ---- the same outputs in 64 bits with plain torch ---------------------------------------------------------------

def _factors(b, lo, hi, term):
    """Factor matrices of entries lo..hi as [hi - lo, d, n, n] in float64 (column-major storage, `stride`)."""
    off = b.mat_off[(term * b.nb + lo) * b.d:(term * b.nb + hi) * b.d].to(DEVICE).view(-1, b.d, 1, 1)
    r = torch.arange(b.n, device=DEVICE)
    idx = off + r.view(1, 1, -1, 1) + b.stride * r.view(1, 1, 1, -1)
    return b.mats[idx].double(), idx


def _contract(a, x, t, d, n):
    """Mode t of x [entries, n^d] times a [entries, n, n]: y[.., r, ..] = sum_k a[r, k] x[.., k, ..]."""
    v = x.view(x.shape[0], n ** t, n, n ** (d - 1 - t))
    y = torch.zeros_like(v)
    for k in range(n):
        y += a[:, None, :, k, None] * v[:, :, k, None, :]
    return y.view(x.shape)


def _vectors(pool, off, size):
    return pool[off.to(DEVICE)[:, None] + torch.arange(size, device=DEVICE)[None, :]].double()


def _chunks(b):
    step = max(1, (1 << 26) // b.size)
    return [(lo, min(lo + step, b.nb)) for lo in range(0, b.nb, step)]


def _exact_forward(b, terms):
    out = torch.zeros(b.out_count, b.size, dtype=torch.float64, device=DEVICE)
    for lo, hi in _chunks(b):
        x = _vectors(b.inputs, b.in_off[lo:hi], b.size)
        for term in range(terms):
            a, _ = _factors(b, lo, hi, term)
            y = x
            for t in range(b.d - 1, -1, -1):
                y = _contract(a[:, t], y, t, b.d, b.n)
            out.index_add_(0, b.out_index[lo:hi].to(DEVICE), y)
    return out.view(-1)


def _exact_adjoint(b, gout):
    gin = torch.zeros(b.inputs.numel() // b.size, b.size, dtype=torch.float64, device=DEVICE)
    gmat = torch.zeros(b.mats.numel(), dtype=torch.float64, device=DEVICE)
    d, n = b.d, b.n
    for lo, hi in _chunks(b):
        a, idx = _factors(b, lo, hi, 0)
        chain = [_vectors(b.inputs, b.in_off[lo:hi], b.size)]  # what each factor is applied to, mode d-1 first
        for t in range(d - 1, 0, -1):
            chain.append(_contract(a[:, t], chain[-1], t, d, n))
        h = _vectors(gout, b.out_index[lo:hi] * b.size, b.size)
        for t in range(d):
            x = chain[d - 1 - t].view(hi - lo, n ** t, n, -1)
            hv = h.view(hi - lo, n ** t, n, -1)
            grad = torch.stack([(hv * x[:, :, k, None, :]).sum((1, 3)) for k in range(n)], 2)  # [entries, r, k]
            gmat.index_add_(0, idx[:, t].reshape(-1), grad.reshape(-1))
            h = _contract(a[:, t].transpose(1, 2), h, t, d, n)
        gin.index_add_(0, torch.div(b.in_off[lo:hi], b.size, rounding_mode="floor").to(DEVICE), h)
    return [gin.view(-1), gmat]


def exact(case, seed):
    batches, g = _batches(case, seed)
    if case["kind"] == "adjoint":
        b = batches[0]
        return _exact_adjoint(b, _normal(b.out_count * b.size, b.inputs.dtype, g))
    return [torch.cat([_exact_forward(b, case.get("terms", 1)) for b in batches])]
