"""The cases on which this library's speed is followed.

A case is one thing a user's program has the library do, through its public entry points
(``spcomm3d_amd.device``), over operands that such a program already holds:

``step``      SDDMM, then SpMM, over resident operands and a kept plan: what a rank computes per
              iteration
``fused``     the chained one-pass call ``C = S .* (A B^T)``, ``Y += C B``
``loop``      one iteration of the reference's bench loop with everything on the device
              (miniapp/bench_both.cpp:196-205): the indices remapped, a plan made of them, ``calls``
              SDDMM and SpMM calls over it, the indices remapped back
``exchange``  the copies either side of a sparse exchange: pack, unpack, sum-unpack
``host``      the one-shot calls over host memory, which is how the reference's own programs call
              the kernels through the C++ shim: the same pattern and panels from call to call

Patterns are drawn on the GPU from the seed and follow the library's own workloads
(``spcomm3d_amd.workloads``): uniform rows, R-MAT, the local block of a partitioned R-MAT graph,
a 5-point stencil, a hypergraph's incidence matrix with capped Zipf rows.
"""
import math

import numpy as np
import torch

from spcomm3d_amd import device, roofline

A_, B_, C_, D_ = 0.57, 0.19, 0.19, 0.05  # R-MAT quadrants
ZIPF_S = 1.2
MAX_GATHER = 290e9  # bytes of dense rows that the entries of a drawn case name, at most
MAX_PANEL = 2.2e9   # bytes of one dense panel of a drawn case, at most

_TORCH = {"f32": torch.float32, "f64": torch.float64}


def listed():
    return [
        # the smallest calls (the size of the golden tests): launches and host time are all there is
        {"name": "er1k_f64_k16", "kind": "step", "pattern": "er", "rows": 1024, "cols": 1024,
         "deg": 8, "k": 16, "dtype": "f64", "order": "sorted"},
        # first configuration of bench.py: a kernel of a few microseconds
        {"name": "er16k_f64_k32", "kind": "step", "pattern": "er", "rows": 16384, "cols": 16384,
         "deg": 16, "k": 32, "dtype": "f64", "order": "sorted"},
        # a small skewed graph as a file or an exchange delivers it: arbitrary entry order, and
        # dense rows that leave lanes idle
        {"name": "rmat14_f32_k20_shuffled", "kind": "step", "pattern": "rmat", "scale": 14,
         "edges": 16, "k": 20, "dtype": "f32", "order": "shuffled"},
        # the headline workload of bench.py
        {"name": "rmat20_f64_k64", "kind": "step", "pattern": "rmat", "scale": 20, "edges": 16,
         "k": 64, "dtype": "f64", "order": "sorted"},
        # the same graph in single precision and arbitrary order
        {"name": "rmat20_f32_k64_shuffled", "kind": "step", "pattern": "rmat", "scale": 20,
         "edges": 16, "k": 64, "dtype": "f32", "order": "shuffled"},
        # a graph in the order of a MatrixMarket file, dense rows that are no power of two
        {"name": "rmat18_f64_k100_column", "kind": "step", "pattern": "rmat", "scale": 18,
         "edges": 16, "k": 100, "dtype": "f64", "order": "column"},
        # one rank's block of a 4 x 4 partition at its local shape, as the one-pass call
        {"name": "block24_f32_k64_fused", "kind": "fused", "pattern": "block", "scale": 24,
         "edges": 16, "parts": 4, "k": 64, "dtype": "f32", "order": "sorted"},
        # short regular rows, nothing to balance: the streams bound it
        {"name": "stencil4096_f32_k32", "kind": "step", "pattern": "stencil", "nx": 4096,
         "ny": 4096, "k": 32, "dtype": "f32", "order": "sorted"},
        # the largest: long rows over unskewed columns
        {"name": "hypergraph_f32_k128", "kind": "step", "pattern": "hyper", "rows": 2000000,
         "cols": 500000, "cap": 1024, "k": 128, "dtype": "f32", "order": "sorted"},
        # a pattern used for five calls of each kernel and then replaced
        {"name": "loop_rmat20_f64_k64", "kind": "loop", "pattern": "rmat", "scale": 20,
         "edges": 16, "k": 64, "dtype": "f64", "order": "sorted", "calls": 5},
        # half a million rows of a panel sent and received, a row no whole number of vectors
        {"name": "exchange_1m_f32_k50", "kind": "exchange", "rows": 1048576, "slots": 500000,
         "k": 50, "dtype": "f32"},
        # the drop-in calls of one rank over host vectors
        {"name": "host_rmat17_f64_k64", "kind": "host", "pattern": "rmat", "scale": 17,
         "edges": 16, "k": 64, "dtype": "f64", "order": "sorted"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo=1, hi=600):
    """Dense row widths: the powers of two that programs like, and anything between."""
    if rng.random() < 0.5:
        return rng.choice([k for k in (8, 16, 32, 64, 128, 256) if lo <= k <= hi])
    return _log_int(rng, lo, hi)


def _draw_pattern(rng, pattern):
    if pattern == "er":
        return {"rows": _log_int(rng, 1000, 3000000), "cols": _log_int(rng, 1000, 3000000),
                "deg": _log_int(rng, 3, 48)}
    if pattern == "rmat":
        return {"scale": rng.randint(11, 20), "edges": rng.randint(6, 20)}
    if pattern == "block":
        return {"scale": rng.randint(16, 23), "edges": rng.randint(8, 18), "parts": rng.choice([2, 4])}
    if pattern == "stencil":
        return {"nx": _log_int(rng, 60, 4000), "ny": _log_int(rng, 60, 4000)}
    return {"rows": _log_int(rng, 10000, 1500000), "cols": _log_int(rng, 5000, 500000),
            "cap": _log_int(rng, 64, 1024)}


def draw(rng):
    while True:
        kind = rng.choice(["step", "step", "step", "step", "step", "step", "fused", "fused", "loop",
                           "exchange", "exchange", "host"])
        case = {"kind": kind, "dtype": rng.choice(["f32", "f64"])}
        w = 4 if case["dtype"] == "f32" else 8
        if kind == "exchange":
            case["rows"] = _log_int(rng, 3000, 2000000)
            case["slots"] = _log_int(rng, 1000, 1500000)
            case["k"] = _width(rng, 1, 300)
            if max(case["rows"], case["slots"]) * case["k"] * w <= MAX_PANEL:
                return case
            continue
        if kind == "host":
            case["pattern"] = rng.choice(["er", "rmat", "stencil"])
        elif kind == "loop":
            case["pattern"] = rng.choice(["er", "rmat", "block"])
            case["calls"] = rng.randint(1, 5)
        else:
            case["pattern"] = rng.choice(["er", "er", "rmat", "rmat", "block", "stencil", "hyper"])
        case.update(_draw_pattern(rng, case["pattern"]))
        case["k"] = _width(rng)
        case["order"] = rng.choice(["sorted", "sorted", "shuffled", "column"])
        m, n, nnz, _, _ = _expected(case)
        most = 150e6 if kind == "host" else MAX_PANEL
        if max(m, n) * case["k"] * w <= most and nnz * (case["k"] * w + 32) <= MAX_GATHER:
            return case


# ---- what a case amounts to --------------------------------------------------------------
def _zipf_degrees(case):
    """Pins per row, min(Zipf, cap): the distribution's quantiles, so that every seed has as many
    entries (rows get them in an order of the seed's)."""
    weight = np.arange(1, case["cap"] + 1, dtype=np.float64) ** -ZIPF_S
    tail = np.arange(case["cap"] + 1, 100001, dtype=np.float64) ** -ZIPF_S
    cdf = np.cumsum(weight) / (weight.sum() + tail.sum() + 100000.5 ** (1 - ZIPF_S) / (ZIPF_S - 1))
    u = (np.arange(case["rows"]) + 0.5) / case["rows"]
    return np.minimum(np.searchsorted(cdf, u) + 1, case["cap"])


def _rmat_distinct(s, draws):
    """Expected number of distinct edges among `draws` (B_ == C_)."""
    total = 0.0
    for a in range(s + 1):
        for b in range(s - a + 1):
            cells = math.comb(s, a) * math.comb(s - a, b) * 2.0 ** b
            total += cells * -math.expm1(-draws * A_ ** a * B_ ** b * D_ ** (s - a - b))
    return total


def _rmat_touched(s, draws):
    """Expected number of rows (columns) that hold an edge."""
    p = A_ + B_
    return sum(math.comb(s, i) * -math.expm1(-draws * p ** i * (1 - p) ** (s - i))
               for i in range(s + 1))


def _expected(case):
    """(rows, columns, entries, rows with an entry, columns with an entry): the entries exactly,
    the others as expected."""
    pattern = case["pattern"]
    if pattern == "er":
        m, n = case["rows"], case["cols"]
        nnz = m * case["deg"]
        return m, n, nnz, m, n * -math.expm1(-nnz / n)
    if pattern in ("rmat", "block"):
        s, draws = case["scale"], case["edges"] * 2.0 ** case["scale"]
        if pattern == "rmat":
            t = _rmat_touched(s, draws)
            return 2 ** s, 2 ** s, round(_rmat_distinct(s, draws)), t, t
        t = _rmat_touched(s, draws / case["parts"]) / case["parts"]
        return t, t, round(_rmat_distinct(s, draws) / case["parts"] ** 2), t, t
    if pattern == "stencil":
        n = case["nx"] * case["ny"]
        return n, n, 5 * n - 2 * case["nx"] - 2 * case["ny"], n, n
    m, n = case["rows"], case["cols"]
    nnz = int(_zipf_degrees(case).sum())
    return m, n, nnz, m, n * -math.expm1(-nnz / n)


def work(case):
    """Every operand once (spcomm3d_amd.roofline, the strict model)."""
    k, w = case["k"], 4 if case["dtype"] == "f32" else 8
    if case["kind"] == "exchange":
        slots, rows = case["slots"], case["rows"]
        uniq = rows * -math.expm1(-slots / rows)
        pack = (uniq + slots) * k * w + 4 * slots
        unpack = 2 * uniq * k * w + 4 * slots            # one slot read and one row written
        add = (slots + 2 * uniq) * k * w + 4 * slots
        return {"bytes": pack + unpack + add, "flops": slots * k}
    m, n, nnz, mt, nt = _expected(case)
    perm = case["order"] != "sorted"
    sd = roofline.sddmm_bytes(m, nnz, k, w, mt, nt, perm)
    sp = roofline.spmm_bytes(m, nnz, k, w, mt, nt)
    fl = roofline.flops(nnz, k)
    if case["kind"] == "fused":
        return {"bytes": roofline.fused_bytes(m, nnz, k, w, mt, nt, perm), "flops": 2 * fl}
    if case["kind"] == "host":  # both calls take the COO and its values
        return {"bytes": sd + sp + 12 * nnz, "flops": 2 * fl}
    if case["kind"] == "loop":
        remap = 2 * 2 * 8 * nnz + 2 * 4 * (m + n)        # both arrays there and back, the maps
        plan = 8 * nnz + 4 * nnz + 4 * m + 3 * w * nnz   # COO in, kernel order and values out
        return {"bytes": remap + plan + case["calls"] * (sd + sp), "flops": 2 * fl * case["calls"]}
    return {"bytes": sd + sp, "flops": 2 * fl}


def tolerance(case):
    if case["kind"] == "exchange":
        return "exact"  # copies, and sums in the order of the slots
    return {"rel": 1e-5 if case["dtype"] == "f32" else 1e-12}


# ---- inputs ---------------------------------------------------------------------------------
def _rmat_edges(gen, scale, draws):
    row = torch.zeros(draws, dtype=torch.int32, device="cuda")
    col = torch.zeros(draws, dtype=torch.int32, device="cuda")
    for _ in range(scale):
        r = torch.rand(draws, generator=gen, device="cuda")
        row.mul_(2).add_(r >= A_ + B_)
        col.mul_(2).add_(((r >= A_) & (r < A_ + B_)) | (r >= A_ + B_ + C_))
    return row, col


def _sort_unique(row, col):
    key = torch.unique((row.to(torch.int64) << 32) | col.to(torch.int64))
    return (key >> 32).to(torch.int32), (key & 0xFFFFFFFF).to(torch.int32)


def _rmat_pattern(gen, case, keep):
    """Exactly as many distinct edges as _expected says, sorted; keep(row, col): the edges of
    the pattern among those drawn, under the pattern's own numbers."""
    want = _expected(case)[2]
    row = col = torch.zeros(0, dtype=torch.int32, device="cuda")
    left = int(1.02 * (case["edges"] << case["scale"])) + 1024
    while left > 0 or row.numel() < want:
        draws = min(left, 1 << 26) if left > 0 else 1 << max(case["scale"], 16)
        r, c = keep(*_rmat_edges(gen, case["scale"], draws))
        row, col = torch.cat([row, r]), torch.cat([col, c])
        left -= draws
        if left <= 0:
            row, col = _sort_unique(row, col)
    if row.numel() > want:
        some = torch.randperm(row.numel(), generator=gen, device="cuda")[:want].sort()[0]
        row, col = row[some], col[some]
    return row, col


def _block_pattern(ctx, gen, case):
    n, parts = 1 << case["scale"], case["parts"]
    pos_r = torch.randperm(n, generator=gen, device="cuda", dtype=torch.int32)
    pos_c = torch.randperm(n, generator=gen, device="cuda", dtype=torch.int32)

    def keep(row, col):
        row, col = pos_r[row.long()], pos_c[col.long()]
        mine = (row % parts == 0) & (col % parts == 0)
        return row[mine] // parts, col[mine] // parts

    row, col = _rmat_pattern(gen, case, keep)
    row, col = row.contiguous(), col.contiguous()
    torch.cuda.synchronize()
    m, _ = device.localize_device(ctx, _vals(ctx, row), row.numel())
    n, _ = device.localize_device(ctx, _vals(ctx, col), col.numel())
    ctx.sync()
    return m, n, row, col


def _pattern(ctx, gen, case):
    """(rows, columns, ii, jj): int32 tensors on the GPU, in the case's entry order."""
    pattern = case["pattern"]
    if pattern == "er":
        m, n = case["rows"], case["cols"]
        row = torch.arange(m, dtype=torch.int32, device="cuda").repeat_interleave(case["deg"])
        col = torch.randint(0, n, (row.numel(),), generator=gen, device="cuda", dtype=torch.int32)
        _, p = torch.sort((row.to(torch.int64) << 32) | col.to(torch.int64))
        row, col = row[p], col[p]
    elif pattern == "rmat":
        m = n = 1 << case["scale"]
        row, col = _rmat_pattern(gen, case, lambda row, col: (row, col))
    elif pattern == "block":
        m, n, row, col = _block_pattern(ctx, gen, case)
    elif pattern == "stencil":
        nx, ny = case["nx"], case["ny"]
        m = n = nx * ny
        p = torch.arange(n, dtype=torch.int32, device="cuda")
        x, y = p % nx, p // nx
        ok = torch.stack([y > 0, x > 0, x >= 0, x < nx - 1, y < ny - 1], 1)
        step = torch.tensor([-nx, -1, 0, 1, nx], dtype=torch.int32, device="cuda")
        row = p[:, None].expand(-1, 5)[ok]
        col = (p[:, None] + step)[ok]
    else:  # columns in draw order inside a row, as hypergraph_zipf gives them
        m, n = case["rows"], case["cols"]
        deg = torch.from_numpy(_zipf_degrees(case)).cuda()
        deg = deg[torch.randperm(m, generator=gen, device="cuda")]
        row = torch.arange(m, dtype=torch.int32, device="cuda").repeat_interleave(deg)
        col = torch.randint(0, n, (row.numel(),), generator=gen, device="cuda", dtype=torch.int32)
    if case["order"] == "shuffled":
        p = torch.randperm(row.numel(), generator=gen, device="cuda")
        row, col = row[p], col[p]
    elif case["order"] == "column":
        _, p = torch.sort((col.to(torch.int64) << 32) | row.to(torch.int64), stable=True)
        row, col = row[p], col[p]
    return m, n, row.contiguous(), col.contiguous()


def _uniform(gen, shape, dtype, lo, hi):
    return torch.rand(shape, generator=gen, device="cuda", dtype=_TORCH[dtype]).mul_(hi - lo).add_(lo)


def _vals(ctx, t):
    """The tensor's memory as a value vector (32-bit words for index arrays)."""
    kind = np.float64 if t.dtype == torch.float64 else np.float32
    return device.Vals(ctx, t.numel(), kind, dev=t.data_ptr())


def _panel(ctx, t):
    kind = np.float64 if t.dtype == torch.float64 else np.float32
    return device.Panel(ctx, t.shape[0], t.shape[1], kind, dev=t.data_ptr())


_ctx = None


def _context():
    """The context of the process: one per rank, kept for its life."""
    global _ctx
    if _ctx is None:
        _ctx = device.Context(0)
    return _ctx


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, k, dtype = case["kind"], case["k"], case["dtype"]
    s = {"case": case}
    if kind == "exchange":
        ctx = s["ctx"] = _context()
        rows = torch.randint(0, case["rows"], (case["slots"],), generator=gen, device="cuda", dtype=torch.int32)
        s["map"] = device.RowMap(ctx, case["rows"], rows.cpu().numpy().view(np.uint32))
        for name in ("sent", "received", "summed"):
            s[name] = _uniform(gen, (case["rows"], k), dtype, -1, 1)
        s["out"] = torch.zeros(case["slots"] * k, dtype=_TORCH[dtype], device="cuda")
        s["in"] = _uniform(gen, case["slots"] * k, dtype, -1, 1)
        torch.cuda.synchronize()
        s["h"] = {n: (_panel if s[n].dim() == 2 else _vals)(ctx, s[n])
                  for n in ("sent", "received", "summed", "out", "in")}
        return s
    if kind == "host":  # a rank's context, whose one-shot calls keep what still holds
        ctx = s["ctx"] = device.Context(0)
    else:
        ctx = s["ctx"] = _context()
    m, n, ii, jj = _pattern(ctx, gen, case)
    vv = _uniform(gen, ii.numel(), dtype, 0, 1)
    tall_a, tall_b = m, n
    if case["pattern"] == "block":  # panels that serve every block of the partition
        tall_a = tall_b = max(m, n, int(1.2 * _expected(case)[0]) + 1024)
    A, B = _uniform(gen, (tall_a, k), dtype, -1, 1), _uniform(gen, (tall_b, k), dtype, -1, 1)
    Y = _uniform(gen, (tall_a, k), dtype, -1, 1)
    if kind == "host":
        for name, t in (("A", A), ("B", B), ("Y", Y), ("vv", vv)):
            s[name] = t.cpu().numpy()
        s["ii"], s["jj"] = (t.cpu().numpy().view(np.uint32) for t in (ii, jj))
        return s
    C = torch.zeros_like(vv)
    s.update(m=m, n=n, A=A, B=B, C=C, Y=Y, vv=vv)
    torch.cuda.synchronize()
    s["h"] = {"A": _panel(ctx, A), "B": _panel(ctx, B), "Y": _panel(ctx, Y), "C": _vals(ctx, C),
              "vv": _vals(ctx, vv)}
    if kind == "loop":
        s.update(ii=ii, jj=jj)
        for name, size in (("r", m), ("c", n)):
            there = torch.randperm(size, generator=gen, device="cuda", dtype=torch.int32)
            back = torch.empty_like(there)
            back[there.long()] = torch.arange(size, dtype=torch.int32, device="cuda")
            s["there_" + name], s["back_" + name] = there, back
        torch.cuda.synchronize()
        for name in ("ii", "jj", "there_r", "back_r", "there_c", "back_c"):
            s["h"][name] = _vals(ctx, s[name])
    else:
        s["plan"] = device.Plan.from_device(ctx, m, n, _vals(ctx, ii), _vals(ctx, jj), ii.numel(),
                                            dtype, k_hint=k)
        s["plan"].set_values_device(s["h"]["vv"])
        ctx.sync()  # ii and jj go back to torch
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    if case["kind"] == "host":
        C = ctx.sddmm_host(s["A"], s["B"], s["ii"], s["jj"], s["vv"])
        ctx.spmm_host(s["B"], s["ii"], s["jj"], s["vv"], s["Y"])
        return {"C": C, "Y": s["Y"]}
    h = s["h"]
    if case["kind"] == "exchange":
        s["map"].pack(h["sent"], h["out"])
        s["map"].unpack(h["received"], h["in"])
        s["map"].unpack_sum(h["summed"], h["in"])
        return {"out": s["out"], "received": s["received"], "summed": s["summed"]}
    if case["kind"] == "fused":
        ctx.sddmm_spmm(s["plan"], h["A"], h["B"], h["C"], h["Y"], chained=True)
    elif case["kind"] == "step":
        ctx.sddmm(s["plan"], h["A"], h["B"], h["C"])
        ctx.spmm(s["plan"], h["B"], h["Y"])
    else:
        nnz, m, n = s["vv"].numel(), s["m"], s["n"]
        device.remap_device(ctx, h["ii"], nnz, h["there_r"], m)
        device.remap_device(ctx, h["jj"], nnz, h["there_c"], n)
        plan = device.Plan.from_device(ctx, m, n, h["ii"], h["jj"], nnz, case["dtype"], k_hint=case["k"])
        plan.set_values_device(h["vv"])
        for _ in range(case["calls"]):
            ctx.sddmm(plan, h["A"], h["B"], h["C"])
            ctx.spmm(plan, h["B"], h["Y"])
        device.remap_device(ctx, h["ii"], nnz, h["back_r"], m)
        device.remap_device(ctx, h["jj"], nnz, h["back_c"], n)
        plan.close()
    return {"C": s["C"], "Y": s["Y"]}
