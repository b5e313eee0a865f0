"""Workloads of the per-rank GEMM engine, through its public entry points.

listed() covers what a program calls the library for: the local tile
products of Cannon and SUMMA, the whole virtual-grid products, the uneven
grouped batch, the Ozaki split forms, FP32 products and the layout passes;
draw() gives further cases of the same ranges.  All matrices are
column-major, random and made from the seed alone.
"""
import math
import os
import random
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "distributed-gemm-thesis_amd"))

import dgamd  # noqa: E402

DEV = "cuda"
OZAKI = {"int8": dgamd.DG_OZAKI_INT8, "bf16": dgamd.DG_OZAKI_BF16, "crt": dgamd.DG_OZAKI_INT8_CRT}


def listed():
    return [
        # one local tile product of a 2048^3 problem on a 4x4 grid: the smallest call, launch and latency count
        {"name": "dgemm_tile_512", "kind": "dgemm", "opA": "N", "opB": "N", "m": 512, "n": 512, "k": 512,
         "pad": 0, "alpha": 1.0, "beta": 0.0},
        # a Cannon step's accumulating product (beta = 1) on a tile of a non-divisible grid: odd sizes and
        # odd leading dimensions, A transposed
        {"name": "dgemm_ragged", "kind": "dgemm", "opA": "T", "opB": "N", "m": 1500, "n": 1333, "k": 2001,
         "pad": 0, "alpha": 1.0, "beta": 1.0},
        # the plain FP64 configuration: 2048^3 on a 2x2 Cannon grid of 1024^2 tiles
        {"name": "cannon_2x2_2048", "kind": "cannon", "opA": "N", "opB": "N", "M": 2048, "N": 2048, "K": 2048,
         "p": 2, "c": 1, "alpha": 1.0, "beta": 0.0},
        # the 2.5D configuration (4x4x2, opB = T, layers reduced in HBM) at a quarter of its extents
        {"name": "cannon_4x4x2_nt", "kind": "cannon", "opA": "N", "opB": "T", "M": 4096, "N": 2048, "K": 8192,
         "p": 4, "c": 2, "alpha": 1.0, "beta": 0.0},
        # the SUMMA configuration, full size: 4x4 grid, 512 blocks, C updated with beta = 0.5
        {"name": "summa_4x4_16384", "kind": "summa", "opA": "N", "opB": "N", "M": 16384, "N": 16384, "K": 16384,
         "nb": 512, "P": 4, "Q": 4, "alpha": 1.0, "beta": 0.5},
        # the uneven batch (7x5 tiles of a non-divisible product, 256 GEMMs of log-uniform sizes) at a quarter
        # of its extents: one plan, replayed as a graph
        {"name": "grouped_7x5", "kind": "grouped", "n": 5000, "size": 35, "extra": 256, "lo": 64, "hi": 2048,
         "shapes": 5},
        # FP64-level emulation on the INT8 cores (14 moduli) of wide-ranging inputs, half the configuration's extents
        {"name": "ozaki_crt14_8192", "kind": "ozaki", "form": "crt", "slices": 14, "opA": "N", "opB": "N",
         "m": 8192, "n": 8192, "k": 8192, "pad": 0, "wide": True, "alpha": 1.0, "beta": 0.0},
        # FP64-level INT8 slices on a rectangular, uneven product, A transposed
        {"name": "ozaki_int8_s8", "kind": "ozaki", "form": "int8", "slices": 8, "opA": "T", "opB": "N",
         "m": 3000, "n": 2000, "k": 5000, "pad": 0, "wide": True, "alpha": 1.0, "beta": 0.0},
        # the BF16 slices of the same scheme, on the plain configuration's extents
        {"name": "ozaki_bf16_s11", "kind": "ozaki", "form": "bf16", "slices": 11, "opA": "N", "opB": "N",
         "m": 2048, "n": 2048, "k": 2048, "pad": 0, "wide": True, "alpha": 1.0, "beta": 0.0},
        # FP32 product of an aligned rank tile
        {"name": "sgemm_4096", "kind": "sgemm", "opA": "N", "opB": "N", "m": 4096, "n": 4096, "k": 4096,
         "pad": 0, "alpha": 1.0, "beta": 0.0},
        # FP32 product of an uneven tile: odd sizes, so that no column starts aligned
        {"name": "sgemm_ragged", "kind": "sgemm", "opA": "N", "opB": "T", "m": 1537, "n": 2051, "k": 1023,
         "pad": 0, "alpha": 1.0, "beta": 1.0},
        # scatter, gather and layer reduction of an uneven matrix: block-cyclic and 2D-block layouts both ways
        {"name": "layout_uneven", "kind": "layout", "rows": 5003, "cols": 7001, "mb": 128, "nb": 96, "P": 3,
         "Q": 2, "nrb": 7, "ncb": 5, "layers": 1},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _sizes(rng, lo, hi, names, flops):
    """Log-uniform extents, odd ones among them, of a product of at most `flops` operations."""
    while True:
        s = {x: _log(rng, lo, hi) for x in names}
        if rng.random() < 0.4:  # rank tiles are often whole multiples of a block
            s = {x: max(64, v // 64 * 64) for x, v in s.items()}
        if 2.0 * math.prod(s.values()) <= flops:
            return s


def draw(rng):
    kind = rng.choice(["dgemm", "dgemm", "sgemm", "sgemm", "cannon", "summa", "grouped", "ozaki", "ozaki", "layout"])
    ops = {"opA": rng.choice("NT"), "opB": rng.choice("NT")}
    ab = {"alpha": rng.choice([1.0, 1.0, -0.5]), "beta": rng.choice([0.0, 0.5, 1.0])}
    pad = rng.choice([0, 0, 1, 6])
    if kind in ("dgemm", "sgemm"):
        return {"kind": kind, **ops, **_sizes(rng, 64, 8192, "mnk", 1e12), "pad": pad, **ab}
    if kind == "cannon":
        p, c = rng.choice([(2, 1), (2, 2), (3, 1), (4, 1), (4, 2), (6, 2)])
        t = _sizes(rng, 48, 2048, "mnk", 1e12 / p ** 3)
        return {"kind": kind, **ops, "M": p * t["m"], "N": p * t["n"], "K": p * t["k"], "p": p, "c": c, **ab}
    if kind == "summa":
        P, Q = rng.choice([(2, 2), (4, 4), (2, 3), (4, 2)])
        s = _sizes(rng, 256, 8192, "MNK", 1e12)
        return {"kind": kind, **ops, **s, "nb": rng.choice([64, 96, 128, 256, 512]), "P": P, "Q": Q, **ab}
    if kind == "grouped":
        return {"kind": kind, "n": _log(rng, 500, 6000), "size": rng.choice([6, 12, 20, 35]),
                "extra": _log(rng, 4, 256), "lo": 64, "hi": 2048, "shapes": rng.randrange(1000)}
    if kind == "ozaki":
        form = rng.choice(["crt", "crt", "int8", "bf16"])
        slices = {"crt": rng.choice([13, 14, 15, 16]), "int8": rng.choice([5, 6, 7, 8, 9]), "bf16": 11}[form]
        return {"kind": kind, "form": form, "slices": slices, **ops,
                **_sizes(rng, 256, 8192, "mnk", 1e12 if form == "crt" else 2e11), "pad": pad,
                "wide": rng.random() < 0.5, **ab}
    return {"kind": kind, "rows": _log(rng, 500, 12000), "cols": _log(rng, 500, 12000),
            "mb": rng.choice([32, 64, 100, 128, 512]), "nb": rng.choice([32, 64, 100, 128, 512]),
            "P": rng.choice([2, 3, 4]), "Q": rng.choice([2, 4]), "nrb": rng.choice([2, 4, 7]),
            "ncb": rng.choice([2, 4, 5]), "layers": rng.choice([1, 1, 3])}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _uniform(g, n, dtype=torch.float64):
    return torch.rand(n, generator=g, device=DEV, dtype=dtype).mul_(2.0).sub_(1.0)


def _values(g, n, wide):
    """Uniform in [-1, 1); `wide`: times 2^e, e uniform in [-20, 20]."""
    x = _uniform(g, n)
    if wide:
        x.mul_(torch.exp2(torch.randint(-20, 21, (n,), generator=g, device=DEV).to(torch.float64)))
    return x


def _stored(op, rows, cols):
    """Stored extents of a matrix whose op() is rows x cols."""
    return (rows, cols) if op == "N" else (cols, rows)


def _dense(x, ld, rows, cols):
    """rows x cols view of a column-major buffer."""
    return x[: ld * cols].view(cols, ld)[:, :rows].t()


def _pack2d(G, ro, co):
    """Tiles of G in rank order, each column-major."""
    return torch.cat([G[ro[i]: ro[i + 1], co[j]: co[j + 1]].t().reshape(-1)
                      for i in range(len(ro) - 1) for j in range(len(co) - 1)])


def _splits(n, parts):
    return [i * (n // parts) for i in range(parts)] + [n]


def _cyclic(G, mb, nb, P, Q):
    """Local matrices of a P x Q grid in rank order, each column-major."""
    r = torch.arange(G.shape[0], device=G.device) // mb % P
    c = torch.arange(G.shape[1], device=G.device) // nb % Q
    return torch.cat([G[r == p][:, c == q].t().reshape(-1) for p in range(P) for q in range(Q)])


def _gemm_inputs(case, seed):
    m, n, k, pad = case["m"], case["n"], case["k"], case["pad"]
    ra, ca = _stored(case["opA"], m, k)
    rb, cb = _stored(case["opB"], k, n)
    g = _gen(seed)
    s = {"lda": ra + pad, "ldb": rb + pad, "ldc": m + pad}
    if case["kind"] == "sgemm":
        s["A"], s["B"], s["C"] = (_uniform(g, x, torch.float32)
                                  for x in (s["lda"] * ca, s["ldb"] * cb, s["ldc"] * n))
    else:
        wide = case.get("wide", False)
        s["A"], s["B"], s["C"] = (_values(g, x, wide) for x in (s["lda"] * ca, s["ldb"] * cb, s["ldc"] * n))
    s["dA"], s["dB"] = _dense(s["A"], s["lda"], ra, ca), _dense(s["B"], s["ldb"], rb, cb)
    return s


def _grid_inputs(case, seed):
    """Global stored A, B and C of a virtual-grid product."""
    M, N, K = case["M"], case["N"], case["K"]
    g = _gen(seed)
    shapes = [_stored(case["opA"], M, K), _stored(case["opB"], K, N), (M, N)]
    return [_dense(_uniform(g, r * c), r, r, c) for r, c in shapes]


def _extra_shapes(case):
    r = random.Random(case["shapes"])
    return [tuple(_log(r, case["lo"], case["hi"]) for _ in range(3)) for _ in range(case["extra"])]


def _grouped_inputs(case, seed):
    n, g = case["n"], _gen(seed)
    even = lambda x: x + (x & 1)  # every matrix of the batch starts 16-byte aligned, as a tensor of its own would
    shapes = _extra_shapes(case)
    A, B = _uniform(g, n * n), _uniform(g, n * n)
    return A, B, _uniform(g, sum(even(m * k) for m, _, k in shapes)), _uniform(g, sum(even(k * q) for _, q, k in shapes))


def _grid_of(size):
    d = max(x for x in range(1, int(math.isqrt(size)) + 1) if size % x == 0)
    return size // d, d


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("dgemm", "sgemm", "ozaki"):
        s.update(_gemm_inputs(case, seed))
        if kind == "ozaki":
            need = dgamd.ozaki_workspace(case["m"], case["n"], case["k"], case["slices"], OZAKI[case["form"]])
            s["ws"] = torch.empty(need, dtype=torch.uint8, device=DEV)
    elif kind in ("cannon", "summa"):
        mats = _grid_inputs(case, seed)
        s["packed"] = []
        for G, o in zip(mats, (case["opA"], case["opB"], "N")):
            r, c = G.shape
            flat = G.t().reshape(-1)
            P = torch.empty_like(flat)
            if kind == "cannon":
                dgamd.pack_block2d_t(flat, r, r, c, dgamd.block_splits(r, case["p"]), dgamd.block_splits(c, case["p"]), P)
            else:
                dgamd.pack_block_cyclic_t(flat, r, r, c, case["nb"], case["nb"], case["P"], case["Q"], P)
            s["packed"].append(P)
        if kind == "cannon":
            ws = dgamd.cannon25d_workspace(case["M"], case["N"], case["p"], case["c"])
            s["ws"] = torch.empty(ws, dtype=torch.float64, device=DEV) if ws else None
    elif kind == "grouped":
        n = case["n"]
        A, B, Ae, Be = _grouped_inputs(case, seed)
        shapes = _extra_shapes(case)
        C = torch.zeros(n * n, dtype=torch.float64, device=DEV)
        Ce = torch.zeros(sum(m * q + (m * q & 1) for m, q, _ in shapes), dtype=torch.float64, device=DEV)
        drow, dcol = dgamd.virtual_grid(case["size"])
        ro, co = dgamd.block_splits(n, drow), dgamd.block_splits(n, dcol)
        descs = [dgamd.gemm_desc("N", "N", ro[i + 1] - ro[i], co[j + 1] - co[j], n, 1.0, A.data_ptr() + 8 * ro[i], n,
                                 B.data_ptr() + 8 * co[j] * n, n, 0.0, C.data_ptr() + 8 * (ro[i] + co[j] * n), n)
                 for i in range(drow) for j in range(dcol)]
        oa = ob = oc = 0
        for m, q, k in shapes:
            descs.append(dgamd.gemm_desc("N", "N", m, q, k, 1.0, Ae.data_ptr() + 8 * oa, m, Be.data_ptr() + 8 * ob, k,
                                         0.0, Ce.data_ptr() + 8 * oc, m))
            oa, ob, oc = oa + m * k + (m * k & 1), ob + k * q + (k * q & 1), oc + m * q + (m * q & 1)
        s.update(keep=(A, B, Ae, Be), C=C, Ce=Ce, plan=dgamd.GroupedPlan(descs))
    else:
        g = _gen(seed)
        r, c = case["rows"], case["cols"]
        s["G"] = _uniform(g, r * c)
        s["partial"] = _uniform(g, case["layers"] * r * c)
        s["sum"] = _uniform(g, r * c)
        s["ro"], s["co"] = dgamd.block_splits(r, case["nrb"]), dgamd.block_splits(c, case["ncb"])
        for x in ("cyclic", "block", "from_cyclic", "from_block"):
            s[x] = torch.empty_like(s["G"])
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "dgemm":
        dgamd.dgemm_t(c["opA"], c["opB"], c["m"], c["n"], c["k"], c["alpha"], s["A"], s["lda"], s["B"], s["ldb"],
                      c["beta"], s["C"], s["ldc"])
        return s["C"]
    if kind == "sgemm":
        dgamd.sgemm_t(c["opA"], c["opB"], c["m"], c["n"], c["k"], c["alpha"], s["A"], s["lda"], s["B"], s["ldb"],
                      c["beta"], s["C"], s["ldc"])
        return s["C"]
    if kind == "ozaki":
        dgamd.ozaki_dgemm_t(c["opA"], c["opB"], c["m"], c["n"], c["k"], c["alpha"], s["A"], s["lda"], s["B"], s["ldb"],
                            c["beta"], s["C"], s["ldc"], c["slices"], OZAKI[c["form"]], s["ws"])
        return s["C"]
    if kind == "cannon":
        A, B, C = s["packed"]
        dgamd.cannon25d_t(c["opA"], c["opB"], c["M"], c["N"], c["K"], c["alpha"], A, B, c["beta"], C, c["p"], c["c"],
                          dgamd.DG_SCHED_AUTO, s["ws"])
        return C
    if kind == "summa":
        A, B, C = s["packed"]
        dgamd.summa_t(c["opA"], c["opB"], c["M"], c["N"], c["K"], c["alpha"], A, B, c["beta"], C, c["nb"], c["nb"],
                      c["nb"], c["P"], c["Q"])
        return C
    if kind == "grouped":
        s["plan"].graph_launch()
        return {"C": s["C"], "extra": s["Ce"]}
    r, q, mb, nb, P, Q = (c[x] for x in ("rows", "cols", "mb", "nb", "P", "Q"))
    dgamd.pack_block_cyclic_t(s["G"], r, r, q, mb, nb, P, Q, s["cyclic"])
    dgamd.unpack_block_cyclic_t(s["cyclic"], mb, nb, P, Q, s["from_cyclic"], r, r, q)
    dgamd.pack_block2d_t(s["G"], r, r, q, s["ro"], s["co"], s["block"])
    dgamd.unpack_block2d_t(s["block"], s["ro"], s["co"], s["from_block"], r, r, q)
    dgamd.layer_reduce_t(s["sum"], s["partial"], r * q, c["layers"])
    return {x: s[x] for x in ("cyclic", "block", "from_cyclic", "from_block", "sum")}


def work(case):
    kind = case["kind"]
    if kind == "layout":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * 16.0 * n + 8.0 * n * (case["layers"] + 2), "flops": float(case["layers"] * n)}
    if kind == "grouped":
        n = case["n"]
        shapes = [(n, n, n)] + _extra_shapes(case)
        return {"bytes": 8.0 * sum(m * k + k * q + m * q for m, q, k in shapes),
                "flops": 2.0 * sum(m * q * k for m, q, k in shapes)}
    m, n, k = (case[x] for x in (("M", "N", "K") if kind in ("cannon", "summa") else ("m", "n", "k")))
    size = 4.0 if kind == "sgemm" else 8.0
    return {"bytes": size * (m * k + k * n + m * n * (2 if case["beta"] else 1)), "flops": 2.0 * m * n * k}


# ------------------------------------------------------------------ the same results in 64 bits

def _two_sum(a, b):
    s = a + b
    t = s - a
    return s, (a - (s - t)) + (b - t)


def _cut(X, bits, count):
    """Integer slices of the rows of X: X = 2^e (d_1 2^-bits + d_2 2^-2bits + ...), |d_t| <= 2^bits, and 2^e."""
    e = torch.exp2(torch.ceil(torch.log2(X.abs().amax(1, keepdim=True).clamp_min(1e-300))) + 1)
    rest, out = X / e, []
    for _ in range(count):
        rest = rest * 2.0 ** bits
        d = torch.trunc(rest)
        rest = rest - d
        out.append(d)
    return out, e


def _product(A, B):
    """A @ B as an unevaluated sum (hi, lo): slices of so few bits that every partial sum of their products is a
    whole number below 2^53, so the double products are exact, added with the rounding errors kept."""
    k = A.shape[1]
    bits, count = (53 - max(1, math.ceil(math.log2(k)))) // 2, 4
    da, ea = _cut(A, bits, count)
    db, eb = _cut(B.t(), bits, count)
    db = [x.t().contiguous() for x in db]
    hi = torch.zeros(A.shape[0], B.shape[1], dtype=torch.float64, device=A.device)
    lo = torch.zeros_like(hi)
    for level in range(count + 1, 1, -1):  # the smallest products first
        for t in range(1, level):
            p = torch.mm(da[t - 1], db[level - t - 1]).mul_(2.0 ** (-bits * level))
            hi, err = _two_sum(hi, p)
            lo += err
    scale = ea * eb.t()
    return hi * scale, lo * scale


def _gemm(case, A, B, C):
    """alpha op(A) op(B) + beta C, alpha and beta powers of two (or 0)."""
    hi, lo = _product(A if case["opA"] == "N" else A.t().contiguous(), B if case["opB"] == "N" else B.t().contiguous())
    hi, lo = case["alpha"] * hi, case["alpha"] * lo
    if case["beta"]:
        hi, err = _two_sum(hi, case["beta"] * C)
        lo = lo + err
    return hi + lo


def _into(buf, ld, rows, cols, value):
    out = buf.clone()
    out[: ld * cols].view(cols, ld)[:, :rows] = value.t()
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("dgemm", "ozaki"):
        s = _gemm_inputs(case, seed)
        C = _dense(s["C"], s["ldc"], case["m"], case["n"])
        return _into(s["C"], s["ldc"], case["m"], case["n"], _gemm(case, s["dA"], s["dB"], C))
    if kind == "sgemm":  # products of FP32 values are exact in 64 bits
        s = _gemm_inputs(case, seed)
        A, B = s["dA"].double(), s["dB"].double()
        C = _dense(s["C"], s["ldc"], case["m"], case["n"]).double()
        v = case["alpha"] * torch.mm(A if case["opA"] == "N" else A.t(), B if case["opB"] == "N" else B.t())
        return _into(s["C"].double(), s["ldc"], case["m"], case["n"], v + case["beta"] * C if case["beta"] else v)
    if kind in ("cannon", "summa"):
        v = _gemm(case, *_grid_inputs(case, seed))
        if kind == "cannon":
            return _pack2d(v, _splits(case["M"], case["p"]), _splits(case["N"], case["p"]))
        return _cyclic(v, case["nb"], case["nb"], case["P"], case["Q"])
    if kind == "grouped":
        n = case["n"]
        A, B, Ae, Be = _grouped_inputs(case, seed)
        full = lambda a, b: sum(_product(a, b))
        C = full(_dense(A, n, n, n), _dense(B, n, n, n)).t().reshape(-1)
        parts, oa, ob = [], 0, 0
        for m, q, k in _extra_shapes(case):
            v = full(_dense(Ae[oa:], m, m, k), _dense(Be[ob:], k, k, q)).t().reshape(-1)
            parts.append(torch.cat([v, v.new_zeros(m * q & 1)]))
            oa, ob = oa + m * k + (m * k & 1), ob + k * q + (k * q & 1)
        return {"C": C, "extra": torch.cat(parts)}
    r, c = case["rows"], case["cols"]
    g = _gen(seed)
    G = _uniform(g, r * c)
    partial, total = _uniform(g, case["layers"] * r * c), _uniform(g, r * c)
    for t in range(case["layers"]):
        total += partial[t * r * c: (t + 1) * r * c]
    D = _dense(G, r, r, c)
    return {"cyclic": _cyclic(D, case["mb"], case["nb"], case["P"], case["Q"]),
            "block": _pack2d(D, _splits(r, case["nrb"]), _splits(c, case["ncb"])),
            "from_cyclic": G, "from_block": G, "sum": total}
