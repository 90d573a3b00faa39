"""Performance cases of the library: what its users run, from the smallest
call to the largest, through the public entry points.

A case is a dict of plain values.  Its ``op`` is the call:

* ``spgemm``   one whole product on device CSR operands (``Handle.spgemm``:
               symbolic phase, allocation of C, numeric phase).
* ``values``   the numeric phase alone, on a plan made once (a solver that
               re-assembles a matrix of the same pattern).
* ``aat``      C = A*A^T with the transpose made by ``Handle.transpose``.
* ``batch``    many independent products as one batch.
* ``served``   a mix of requests through the request server.
* ``host``     the two-phase host entry ``thmkl_dcsrmultcsr``.

and its ``matrix`` the operand: ``er`` (Erdos-Renyi), ``lap`` (2D 5-point
operator), ``st27`` (27-point stencil), ``band`` (banded, dense enough for
the tile path), ``rmat`` (power law).  ``prepare`` makes operands on the GPU.
A random structure is drawn once per case and relabelled by the seed (rows and
columns permuted, so that the sizes of C stay), and the values are the seed's.

The handles work on one torch stream, on which the results are allocated too,
as a program with several handles needs: torch hands a dropped result's memory
out again at once to work of the stream it belongs to, and kernels of another
stream may still be reading or writing there.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import tilespgemm_amd as tsg

DEV = "cuda:0"
_stream = None


def _work_stream():
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def listed():
    return [
        # the smallest product of a batch, called alone: launches and round trips
        {"name": "er_1000", "op": "spgemm", "matrix": "er", "n": 1000, "deg": 4.0},
        # an ordinary request of the served mix, called alone
        {"name": "er_16000", "op": "spgemm", "matrix": "er", "n": 16000, "deg": 8.0},
        # a 2D mesh operator squared (coarse operators, smoothers)
        {"name": "lap_256", "op": "spgemm", "matrix": "lap", "side": 256},
        # a 3D mesh operator squared
        {"name": "st27_64", "op": "spgemm", "matrix": "st27", "side": 64},
        # the same pattern with new values: numeric phase on a kept plan
        {"name": "st27_61_values", "op": "values", "matrix": "st27", "side": 61},
        # banded operator, full 16x16 tiles: the tile path
        {"name": "band_65537", "op": "spgemm", "matrix": "band", "n": 65537, "half": 16},
        # rectangular chain product of odd sizes, separate multiply and add
        {"name": "rect_odd", "op": "spgemm", "matrix": "er", "n": 50021, "deg": 12.0,
         "cols": 30011, "k": 40009, "deg_b": 17.0, "separate": True},
        # the served mix's large request, transpose included
        {"name": "rmat18_4_aat", "op": "aat", "matrix": "rmat", "scale": 18, "draws": 4 << 18},
        # a power-law graph with 2^20 rows, A^T at hand: the largest
        {"name": "rmat20_8", "op": "spgemm", "matrix": "rmat", "scale": 20, "draws": 8 << 20},
        # many independent products in one batch
        {"name": "batch_512", "op": "batch", "count": 512, "nmin": 1000, "nmax": 65536,
         "dmin": 4.0, "dmax": 32.0},
        # requests of the served mix through the server
        {"name": "served_20", "op": "served", "er": 14, "lap": 5, "rmat": 1},
        # the reference-compatible host entry, both phases, host arrays in and out
        {"name": "host_st27_40", "op": "host", "matrix": "st27", "side": 40},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["er", "er", "rect", "lap", "st27", "values", "band", "rmat", "rmat",
                       "batch", "served", "host"])
    if kind == "er":
        return {"op": "spgemm", "matrix": "er", "n": int(_log(rng, 1000, 65536)),
                "deg": round(_log(rng, 4, 32), 2), "separate": rng.random() < 0.25}
    if kind == "rect":
        return {"op": "spgemm", "matrix": "er", "n": int(_log(rng, 1000, 65536)),
                "deg": round(_log(rng, 2, 24), 2), "cols": int(_log(rng, 1000, 65536)),
                "k": int(_log(rng, 1000, 65536)), "deg_b": round(_log(rng, 2, 24), 2),
                "separate": rng.random() < 0.25}
    if kind == "lap":
        return {"op": "spgemm", "matrix": "lap", "side": int(_log(rng, 64, 512))}
    if kind == "st27":
        return {"op": "spgemm", "matrix": "st27", "side": int(_log(rng, 10, 72))}
    if kind == "values":
        m = rng.choice(["lap", "st27", "band"])
        size = {"lap": {"side": int(_log(rng, 64, 512))},
                "st27": {"side": int(_log(rng, 10, 72))},
                "band": {"n": int(_log(rng, 2000, 100000)), "half": rng.randint(14, 40)}}[m]
        return {"op": "values", "matrix": m, **size}
    if kind == "band":
        return {"op": "spgemm", "matrix": "band", "n": int(_log(rng, 2000, 100000)),
                "half": rng.randint(14, 40)}
    if kind == "rmat":
        scale = rng.randint(12, 19)
        return {"op": rng.choice(["spgemm", "aat"]), "matrix": "rmat", "scale": scale,
                "draws": int(_log(rng, 4, 12) * (1 << scale))}
    if kind == "batch":
        return {"op": "batch", "count": int(_log(rng, 8, 512)), "nmin": 1000,
                "nmax": int(_log(rng, 4000, 65536)), "dmin": 4.0,
                "dmax": round(rng.uniform(8.0, 32.0), 1)}
    if kind == "served":
        return {"op": "served", "er": rng.randint(4, 14), "lap": rng.randint(1, 6),
                "rmat": rng.randint(0, 1)}
    m = rng.choice(["er", "lap", "st27"])
    size = {"er": {"n": int(_log(rng, 1000, 30000)), "deg": round(_log(rng, 4, 16), 2)},
            "lap": {"side": int(_log(rng, 64, 400))},
            "st27": {"side": int(_log(rng, 10, 44))}}[m]
    return {"op": "host", "matrix": m, **size}


# ---------------------------------------------------------------- operands
# Device CSR triples (rows, cols, indptr int32, indices int32, data float64),
# rows sorted and free of duplicates.
STRUCTURE = 7        # seed of the structures; relabelling and values have the case's


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _perm(g, n):
    return torch.randperm(n, device=DEV, generator=g)


def _csr(rows, cols, key, g, normal=False):
    """CSR from sorted distinct keys row * cols + column."""
    r = torch.div(key, cols, rounding_mode="floor")
    ptr = torch.zeros(rows + 1, dtype=torch.int64, device=DEV)
    ptr[1:] = torch.cumsum(torch.bincount(r, minlength=rows), 0)
    idx = (key - r * cols).to(torch.int32)
    if normal:
        val = torch.randn(key.numel(), dtype=torch.float64, device=DEV, generator=g)
    else:
        val = torch.rand(key.numel(), dtype=torch.float64, device=DEV, generator=g) * 2 - 1
    return rows, cols, ptr.to(torch.int32), idx, val


def _er(gs, g, n, deg, cols, rows_to, cols_to):
    """Structure from gs, relabelled by the permutations; values from g."""
    rate = torch.full((n,), float(deg), device=DEV)
    per_row = torch.poisson(rate, generator=gs).long().clamp_(max=cols)
    r = torch.repeat_interleave(torch.arange(n, device=DEV), per_row)
    c = torch.randint(0, cols, (r.numel(),), device=DEV, generator=gs)
    return _csr(n, cols, torch.unique(rows_to[r] * cols + cols_to[c]), g)


def _er_square(gs, g, n, deg):
    to = _perm(g, n)
    return _er(gs, g, n, deg, n, to, to)


def _rmat(gs, g, scale, draws):
    """R-MAT whose quadrants are mirrored by the seed, level by level."""
    n = 1 << scale
    r = torch.zeros(draws, dtype=torch.int64, device=DEV)
    c = torch.zeros(draws, dtype=torch.int64, device=DEV)
    for _ in range(scale):
        u = torch.rand(draws, dtype=torch.float64, device=DEV, generator=gs)
        r = (r << 1) | (u >= 0.76)
        c = (c << 1) | (((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
    flip = int(torch.randint(0, n, (1,), device=DEV, generator=g))
    return _csr(n, n, torch.unique((r ^ flip) * n + (c ^ flip)), g)


def _grid(g, n, offsets, ok, normal):
    """Rows of a grid operator: column row + offset where ok (offsets ascend)."""
    row = torch.arange(n, dtype=torch.int64, device=DEV)[:, None]
    key = (row * n + row + torch.tensor(offsets, device=DEV)[None, :])[ok]
    return _csr(n, n, key, g, normal)


def _lap(g, side):
    n = side * side
    i = torch.arange(n, device=DEV)
    x, y = i % side, i // side
    ok = torch.stack([y > 0, x > 0, x >= 0, x < side - 1, y < side - 1], 1)
    rows, cols, ptr, idx, val = _grid(g, n, [-side, -1, 0, 1, side], ok, False)
    # a diffusion operator with a varying coefficient: 4 on the diagonal and
    # -1 off it, each off by up to a tenth
    diag = idx == torch.repeat_interleave(i, (ptr[1:] - ptr[:-1]).long())
    return rows, cols, ptr, idx, 0.1 * val + torch.where(diag, 4.0, -1.0).double()


def _st27(g, side):
    n = side ** 3
    i = torch.arange(n, device=DEV)
    x, y, z = i % side, (i // side) % side, i // (side * side)
    offsets, ok = [], []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                offsets.append(dx + dy * side + dz * side * side)
                ok.append((x + dx >= 0) & (x + dx < side) & (y + dy >= 0) & (y + dy < side) &
                          (z + dz >= 0) & (z + dz < side))
    return _grid(g, n, offsets, torch.stack(ok, 1), True)


def _band(g, n, half):
    i = torch.arange(n, device=DEV)[:, None]
    off = torch.arange(-half, half + 1, device=DEV)
    ok = (i + off >= 0) & (i + off < n)
    return _grid(g, n, off.tolist(), ok, True)


def _transpose(A):
    rows, cols, ptr, idx, val = A
    r = torch.repeat_interleave(torch.arange(rows, device=DEV), (ptr[1:] - ptr[:-1]).long())
    order = torch.argsort(idx.long() * rows + r)
    tptr = torch.zeros(cols + 1, dtype=torch.int64, device=DEV)
    tptr[1:] = torch.cumsum(torch.bincount(idx, minlength=cols), 0)
    return cols, rows, tptr.to(torch.int32), r[order].to(torch.int32), val[order]


def _operands(case, seed):
    """[(A, B), ...] of the case's products; B is A for C = A*A."""
    gs, g = _gen(STRUCTURE), _gen(seed)
    rng = np.random.default_rng(STRUCTURE)
    op = case["op"]
    if op == "batch":
        n = np.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"]), case["count"]))
        deg = rng.uniform(case["dmin"], case["dmax"], case["count"])
        mats = [_er_square(gs, g, int(a), d) for a, d in zip(n, deg)]
        return [(A, A) for A in mats]
    if op == "served":
        mats = [_er_square(gs, g, n, 8.0) for n in rng.integers(1000, 16001, case["er"]).tolist()]
        sides = np.exp(rng.uniform(math.log(64), math.log(512), case["lap"])).astype(int)
        mats += [_lap(g, s) for s in sides.tolist()]
        pairs = [(A, A) for A in mats]
        for _ in range(case["rmat"]):
            A = _rmat(gs, g, 18, 4 << 18)
            pairs.append((A, _transpose(A)))
        return [pairs[i] for i in rng.permutation(len(pairs))]
    m = case["matrix"]
    if m == "er" and "cols" in case:
        inner = _perm(g, case["cols"])
        A = _er(gs, g, case["n"], case["deg"], case["cols"], _perm(g, case["n"]), inner)
        B = _er(gs, g, case["cols"], case["deg_b"], case["k"], inner, _perm(g, case["k"]))
        return [(A, B)]
    if m == "rmat":
        A = _rmat(gs, g, case["scale"], case["draws"])
        return [(A, _transpose(A))]
    if m == "er":
        A = _er_square(gs, g, case["n"], case["deg"])
    elif m == "lap":
        A = _lap(g, case["side"])
    elif m == "st27":
        A = _st27(g, case["side"])
    else:
        A = _band(g, case["n"], case["half"])
    return [(A, A)]


def prepare(case, seed):
    op = case["op"]
    ops = _operands(case, seed)
    if op == "host":
        A = ops[0][0]
        return {"op": op, "n": A[0], "A": tuple(t.cpu().numpy() for t in A[2:])}
    pairs = []
    for A, B in ops:
        dA = tsg.DeviceCsr(*A)
        pairs.append((dA, dA if B is A else tsg.DeviceCsr(*B)))
    state = {"op": op, "pairs": pairs}
    if op == "served":
        state["server"] = tsg.Server(0, workers=3, max_batch=64)
        return state
    stream = _work_stream()
    stream.wait_stream(torch.cuda.current_stream())
    mode = tsg.FP_SEPARATE if case.get("separate") else tsg.FP_FUSED
    with torch.cuda.stream(stream):
        h = state["handle"] = tsg.Handle(0, fp_mode=mode)
        if op == "values":
            ic, nnz = h.symbolic(*pairs[0])
            state["ic"] = ic
            state["jc"] = torch.empty(nnz, dtype=torch.int32, device=DEV)
            state["c"] = torch.empty(nnz, dtype=torch.float64, device=DEV)
    return state


def run(state):
    op = state["op"]
    if op == "host":
        n, A = state["n"], state["A"]
        ic = tsg.thmkl_dcsrmultcsr(1, n, n, n, A, A)
        jc, c = tsg.thmkl_dcsrmultcsr(0, n, n, n, A, A, ic=ic)
        return [ic, jc, c]
    pairs = state["pairs"]
    if op == "served":
        server = state["server"]
        tickets = [server.submit(A, B) for A, B in pairs]
        return [list(server.fetch_device(t)[:3]) for t in tickets]
    with torch.cuda.stream(_work_stream()):
        return _run_handle(op, state["handle"], pairs, state)


def _run_handle(op, h, pairs, state):
    if op == "batch":
        arr, ic, per, _, tot = h.batch_symbolic(pairs)
        jc = torch.empty(max(tot, 1), dtype=torch.int32, device=DEV)
        c = torch.empty(max(tot, 1), dtype=torch.float64, device=DEV)
        h.batch_numeric(arr, ic, jc, c)
        return [ic, jc, c, per]
    A, B = pairs[0]
    if op == "values":
        h.numeric(A, B, state["ic"], state["jc"], state["c"])
        return [state["ic"], state["jc"], state["c"]]
    if op == "aat":
        T = h.transpose(A)
        return [*h.spgemm(A, T), T.indptr, T.indices, T.data]
    return list(h.spgemm(A, B))


def work(case):
    """CSR in and CSR out, each once; two operations per product."""
    h = tsg.Handle(0)
    nbytes = flops = 0
    for A, B in _operands(case, 0):
        dA = tsg.DeviceCsr(*A)
        dB = dA if B is A else tsg.DeviceCsr(*B)
        _, nnz = h.symbolic(dA, dB)
        ptr = 4 if case["op"] == "host" else 8
        nbytes += (A[0] + 1) * (4 + ptr) + 12 * (dA.nnz + nnz)
        if B is not A and case["op"] != "aat":
            nbytes += (B[0] + 1) * 4 + 12 * dB.nnz
        if case["op"] == "aat":             # A^T is a result
            nbytes += (B[0] + 1) * 4 + 12 * dB.nnz
        flops += 2 * h.intermediate_products(dA, dB)
    h.close()
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------- exact
def _product(A, B, chunk=1 << 25):
    """C's values (rows in order, columns ascending) in 64 bits: products
    expanded, sorted by (row, column) and summed, a range of rows at a time."""
    m, _, ia, ja, a = A
    _, k, ib, jb, b = B
    ia, ib, ja = ia.long(), ib.long(), ja.long()
    lens = (ib[1:] - ib[:-1])[ja]
    before = torch.zeros(lens.numel() + 1, dtype=torch.int64, device=DEV)
    before[1:] = torch.cumsum(lens, 0)
    row_before = before[ia]                  # products before each row
    cuts, total = [0], int(row_before[-1])
    marks = torch.searchsorted(row_before, torch.arange(0, total + 1, chunk, device=DEV))
    for r in marks.tolist() + [m]:
        if r > cuts[-1]:
            cuts.append(r)
    rows_of = torch.repeat_interleave(torch.arange(m, device=DEV), ia[1:] - ia[:-1])
    out = []
    for r0, r1 in zip(cuts, cuts[1:]):
        e0, e1 = int(ia[r0]), int(ia[r1])
        ln = lens[e0:e1]
        src = torch.repeat_interleave(torch.arange(e0, e1, device=DEV), ln)
        if src.numel() == 0:
            continue
        pos = torch.arange(src.numel(), device=DEV) - (before[src] - before[e0]) + ib[ja[src]]
        key = rows_of[src] * k + jb[pos]
        val = a[src] * b[pos]
        del src, pos
        key, order = torch.sort(key)
        val = val[order]
        del order
        seg = torch.zeros_like(key)          # the output that each product adds to
        seg[1:] = torch.cumsum(key[1:] != key[:-1], 0)
        del key
        c = torch.zeros(int(seg[-1]) + 1, dtype=torch.float64, device=DEV)
        out.append(c.index_add_(0, seg, val))
        del val, seg
    return torch.cat(out) if out else torch.zeros(0, dtype=torch.float64, device=DEV)


def exact(case, seed):
    op = case["op"]
    ops = _operands(case, seed)
    if op == "batch":
        return [None, None, torch.cat([_product(A, B) for A, B in ops]), None]
    if op == "served":
        return [[None, None, _product(A, B)] for A, B in ops]
    A, B = ops[0]
    c = _product(A, B)
    if op == "aat":
        return [None, None, c, None, None, B[4]]
    return [None, None, c.cpu().numpy() if op == "host" else c]
