"""Performance cases of the MI355X variant: what a program that uses the library has it do.

Every case goes through the C ABI (rajaperf_amd.abi) on torch tensors, on the
current stream, with the library's own default tunings.  Kernels that work in
place (SORT, JACOBI_2D) get a fresh copy of their input in every pass, and the
operators that add into Y get a cleared Y, so a pass can be repeated on the
same state; both are calls of the library too.
"""

import math
import random

import numpy as np
import torch

from rajaperf_amd import abi

ALPHA = 0.75           # stream group
GEMM_ALPHA, GEMM_BETA = 1.5, 1.2
VALUES = ("uniform", "normal", "integers")


def listed():
    return [
        # The stream group at the suite's default length: five launches of a few
        # microseconds each, what a default run of the driver repeats thousands of times.
        {"name": "stream_1m", "kind": "stream", "n": 1000000},
        # The algorithm group's scan and sum near the default length, odd.
        {"name": "scan_sum_1m", "kind": "scan_sum", "n": 1000003, "inclusive": False},
        # The HBM-bound kernels on 2 GiB arrays.
        {"name": "hbm_2e28", "kind": "hbm", "n": 1 << 28},
        # The stencil at the suite's default grid and time steps (8 MB: cache resident).
        {"name": "jacobi_1002", "kind": "jacobi", "N": 1002, "tsteps": 40},
        # The stencil on a grid that lives in HBM.
        {"name": "jacobi_8192", "kind": "jacobi", "N": 8192, "tsteps": 50},
        # FP64 GEMM at the suite's default shape.
        {"name": "gemm_1000", "kind": "gemm", "ni": 1000, "nj": 1000, "nk": 1200, "beta": False},
        # FP64 GEMM, large and square, on the matrix cores.
        {"name": "gemm_4096", "kind": "gemm", "ni": 4096, "nj": 4096, "nk": 4096, "beta": False},
        # The same product on int8 matrix cores.
        {"name": "gemm_mixed_4096", "kind": "gemm_mixed", "ni": 4096, "nj": 4096, "nk": 4096, "beta": False},
        # Partial-assembly mass and diffusion operators, cubic elements.
        {"name": "fem_262144", "kind": "fem", "ne": 262144, "d": 4},
        # Mass operator on ragged batches of mixed polynomial order, one plan.
        {"name": "mass_ragged_64", "kind": "mass_ragged", "nbatch": 64, "lo": 1024, "hi": 65536, "layout": 42},
        # SORT at the suite's default length.
        {"name": "sort_1m", "kind": "sort", "n": 1000000, "values": "uniform"},
        # SORT and SCAN over ragged segments.
        {"name": "segments_256", "kind": "segments", "nseg": 256, "lo": 1 << 10, "hi": 1 << 20, "layout": 42,
         "values": "uniform"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["stream", "scan_sum", "hbm", "jacobi", "gemm", "gemm_mixed", "fem", "mass_ragged", "sort",
                       "segments"])
    if kind == "stream":
        return {"kind": kind, "n": _log(rng, 1 << 12, 1 << 26)}
    if kind == "scan_sum":
        return {"kind": kind, "n": _log(rng, 1 << 12, 1 << 26), "inclusive": rng.random() < 0.5}
    if kind == "hbm":
        return {"kind": kind, "n": _log(rng, 1 << 22, 1 << 28)}
    if kind == "jacobi":
        return {"kind": kind, "N": _log(rng, 130, 8192), "tsteps": rng.randint(1, 50)}
    if kind == "gemm":
        return {"kind": kind, "ni": _log(rng, 64, 4096), "nj": _log(rng, 64, 4096), "nk": _log(rng, 64, 4096),
                "beta": rng.random() < 0.5}
    if kind == "gemm_mixed":
        return {"kind": kind, "ni": _log(rng, 512, 4096), "nj": _log(rng, 512, 4096), "nk": _log(rng, 512, 4096),
                "beta": rng.random() < 0.5}
    if kind == "fem":
        d = rng.randint(2, 8)
        return {"kind": kind, "ne": _log(rng, 1024, 262144 if d <= 4 else 32768), "d": d}
    if kind == "mass_ragged":
        return {"kind": kind, "nbatch": rng.randint(4, 64), "lo": 256, "hi": _log(rng, 4096, 65536),
                "layout": rng.randint(0, 1 << 30)}
    if kind == "sort":
        return {"kind": kind, "n": _log(rng, 1 << 10, 1 << 24), "values": rng.choice(VALUES)}
    return {"kind": kind, "nseg": rng.randint(1, 256), "lo": 1 << 10, "hi": _log(rng, 1 << 12, 1 << 20),
            "layout": rng.randint(0, 1 << 30), "values": rng.choice(VALUES)}


# ---- inputs --------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(n, lo, hi, g):
    return torch.rand(n, dtype=torch.float64, device="cuda", generator=g).mul_(hi - lo).add_(lo)


def _zeros(n):
    return torch.zeros(n, dtype=torch.float64, device="cuda")


def _bytes(n):
    return torch.zeros(max(int(n), 16), dtype=torch.uint8, device="cuda")


def _keys(n, values, g):
    if values == "normal":
        return torch.randn(n, dtype=torch.float64, device="cuda", generator=g)
    if values == "integers":  # many equal keys
        return torch.randint(-500, 500, (n,), device="cuda", generator=g).double()
    return _uniform(n, -1.0, 1.0, g)


def _offsets(case):
    r = random.Random(case["layout"])
    off = [0]
    for _ in range(case["nseg"]):
        off.append(off[-1] + _log(r, case["lo"], case["hi"]))
    return off


def _batches(case):
    """(elements, order) of each ragged batch."""
    r = random.Random(case["layout"])
    return [(_log(r, case["lo"], case["hi"]), r.randint(2, 8)) for _ in range(case["nbatch"])]


def _grid(N, g):
    a = _zeros(N * N)
    a.view(N, N)[1:-1, 1:-1] = torch.rand(N - 2, N - 2, dtype=torch.float64, device="cuda", generator=g)
    return a


def _bases(d):
    """Lagrange basis on d Chebyshev-Lobatto nodes and its derivative at d+1 Gauss points, as [d][q]."""
    q = d + 1
    nodes = -np.cos(np.pi * np.arange(d) / (d - 1)) if d > 1 else np.zeros(1)
    points = np.polynomial.legendre.leggauss(q)[0]
    b, dv = np.empty((d, q)), np.empty((d, q))
    for i in range(d):
        others = np.delete(nodes, i)
        p = np.poly1d(others, r=True) / np.prod(nodes[i] - others) if d > 1 else np.poly1d([1.0])
        b[i], dv[i] = p(points), p.deriv()(points)
    # Exactly (anti)symmetric, as the suite's half-storage tables assume.
    b, dv = (b + b[::-1, ::-1]) / 2, (dv - dv[::-1, ::-1]) / 2
    dv /= np.abs(dv).max()
    return b, dv


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a).reshape(-1)).cuda()


def _fem_bases(d):
    b, dv = _bases(d)
    return _dev(b), _dev(b.T), _dev(dv)  # B[q + Q*d], Bt[d + D*q], dB[q + Q*d]


def prepare(case, seed):
    L, g, kind = abi.lib(), _gen(seed), case["kind"]
    s = dict(case)
    if kind in ("stream", "hbm", "scan_sum"):
        n = case["n"]
        if kind != "scan_sum":
            s.update(a=_uniform(n, 0.0, 1.0, g), b=_uniform(n, 0.0, 1.0, g), c=_zeros(n))
        if kind == "stream":
            s.update(mul=_zeros(n), add=_zeros(n), triad=_zeros(n))
        else:
            s.update(x=_uniform(n, -1.0, 1.0, g), y=_zeros(n), sum=_zeros(1))
            s["scan_bytes"] = L.rpx_scan_scratch_bytes(n, None)
            s["scan_scratch"] = _bytes(s["scan_bytes"])
        s["dot"] = _zeros(1)
        s["red_bytes"] = L.rpx_reduce_scratch_bytes(n, None)
        s["red_scratch"] = _bytes(s["red_bytes"])  # both scratches start zeroed
    elif kind == "jacobi":
        N = case["N"]
        s.update(A0=_grid(N, g), A=_zeros(N * N), B=_zeros(N * N))
        s["bytes"] = L.rpx_jacobi2d_fused_scratch_bytes(N)
        s["scratch"] = _bytes(s["bytes"])
    elif kind in ("gemm", "gemm_mixed"):
        ni, nj, nk = case["ni"], case["nj"], case["nk"]
        s.update(A=_uniform(ni * nk, -1.0, 1.0, g), B=_uniform(nk * nj, -1.0, 1.0, g), C=_zeros(ni * nj))
        s["tune"] = abi.tuning(flags=abi.RPX_TUNE_GEMM_BETA) if case["beta"] else None
        if case["beta"]:
            s["C0"] = _uniform(ni * nj, -1.0, 1.0, g)
        if kind == "gemm_mixed":
            s["bytes"] = L.rpx_gemm_mixed_scratch_bytes(ni, nj, nk, 0)
            s["scratch"] = _bytes(s["bytes"])
    elif kind == "fem":
        ne, d, q = case["ne"], case["d"], case["d"] + 1
        s["B"], s["Bt"], s["G"] = _fem_bases(d)
        s["D"] = _uniform(ne * q**3, 0.5, 2.0, g)
        s["O"] = _uniform(ne * 6 * q**3, -0.25, 0.25, g)  # symmetric tensor 11, 12, 13, 22, 23, 33
        for c in (0, 3, 5):
            s["O"].view(ne, 6, q**3)[:, c] = _uniform(ne * q**3, 0.5, 2.0, g).view(ne, q**3)
        s.update(X=_uniform(ne * d**3, -1.0, 1.0, g), mass=_zeros(ne * d**3), diffusion=_zeros(ne * d**3))
    elif kind == "mass_ragged":
        batches = _batches(case)
        bases = {d: _fem_bases(d) for d in sorted({d for _, d in batches})}
        s["D"] = _uniform(sum(ne * (d + 1)**3 for ne, d in batches), 0.5, 2.0, g)
        nx = sum(ne * d**3 for ne, d in batches)
        s.update(X=_uniform(nx, -1.0, 1.0, g), Y=_zeros(nx), bases=bases)
        table = (abi.MassBatch * len(batches))()
        x = q = 0
        for m, (ne, d) in zip(table, batches):
            m.B, m.Bt = bases[d][0].data_ptr(), bases[d][1].data_ptr()
            m.D, m.X, m.Y = s["D"].data_ptr() + 8 * q, s["X"].data_ptr() + 8 * x, s["Y"].data_ptr() + 8 * x
            m.ne, m.d1d, m.q1d = ne, d, d + 1
            x, q = x + ne * d**3, q + ne * (d + 1)**3
        size = L.rpx_mass3dpa_batched_scratch_bytes(table, len(batches))
        s.update(table=table, scratch=_bytes(size))
        L.rpx_mass3dpa_batched_plan(table, len(batches), s["scratch"].data_ptr(), size, _stream())
    else:
        off = [0, case["n"]] if kind == "sort" else _offsets(case)
        s.update(src=_keys(off[-1], case["values"], g), sorted=_zeros(off[-1]), off=abi.offsets_array(off),
                 count=len(off) - 1)
        s["sort_bytes"] = L.rpx_sort_segmented_scratch_bytes(s["off"], s["count"])
        s["sort_scratch"] = _bytes(s["sort_bytes"])
        if kind == "segments":
            s["scan"] = _zeros(off[-1])
            s["scan_bytes"] = L.rpx_scan_segmented_scratch_bytes(s["off"], s["count"])
            s["scan_scratch"] = _bytes(s["scan_bytes"])
    return s


# ---- one pass ------------------------------------------------------------------


def _stream():
    return torch.cuda.current_stream().cuda_stream


def run(s):
    L, kind, st = abi.lib(), s["kind"], _stream()

    def p(name):
        return s[name].data_ptr()

    if kind == "stream":
        n = s["n"]
        L.rpx_copy_f64(p("c"), p("a"), n, None, st)
        L.rpx_mul_f64(p("mul"), p("b"), ALPHA, n, None, st)
        L.rpx_add_f64(p("add"), p("a"), p("b"), n, None, st)
        L.rpx_triad_f64(p("triad"), p("b"), p("a"), ALPHA, n, None, st)
        L.rpx_dot_f64(p("a"), p("b"), n, p("dot"), 0, p("red_scratch"), s["red_bytes"], None, st)
        return [s["c"], s["mul"], s["add"], s["triad"], s["dot"]]
    if kind in ("hbm", "scan_sum"):
        n, out = s["n"], []
        if kind == "hbm":
            L.rpx_triad_f64(p("c"), p("a"), p("b"), ALPHA, n, None, st)
            L.rpx_dot_f64(p("a"), p("b"), n, p("dot"), 0, p("red_scratch"), s["red_bytes"], None, st)
            out = [s["c"], s["dot"]]
        L.rpx_reduce_sum_f64(p("x"), n, p("sum"), p("red_scratch"), s["red_bytes"], None, st)
        scan = L.rpx_scan_inclusive_f64 if s.get("inclusive") else L.rpx_scan_exclusive_f64
        scan(p("x"), p("y"), n, p("scan_scratch"), s["scan_bytes"], None, st)
        return out + [s["sum"], s["y"]]
    if kind == "jacobi":
        N = s["N"]
        L.rpx_copy_f64(p("A"), p("A0"), N * N, None, st)
        L.rpx_jacobi2d_fused_f64(p("A"), p("B"), N, s["tsteps"], p("scratch"), s["bytes"], None, st)
        return [s["A"], s["B"]]
    if kind in ("gemm", "gemm_mixed"):
        ni, nj, nk = s["ni"], s["nj"], s["nk"]
        if s["beta"]:
            L.rpx_copy_f64(p("C"), p("C0"), ni * nj, None, st)
        if kind == "gemm":
            L.rpx_gemm_f64(p("C"), p("A"), p("B"), GEMM_ALPHA, GEMM_BETA, ni, nj, nk, s["tune"], st)
        else:
            L.rpx_gemm_mixed_tuned_f64(p("C"), p("A"), p("B"), GEMM_ALPHA, GEMM_BETA, ni, nj, nk, 0, s["tune"],
                                       p("scratch"), s["bytes"], st)
        return [s["C"]]
    if kind == "fem":
        ne, d = s["ne"], s["d"]
        L.rpx_fill_const_f64(p("mass"), ne * d**3, 0.0, st)
        L.rpx_mass3dpa_f64(p("B"), p("Bt"), p("D"), p("X"), p("mass"), ne, d, d + 1, None, st)
        L.rpx_fill_const_f64(p("diffusion"), ne * d**3, 0.0, st)
        L.rpx_diffusion3dpa_f64(p("B"), p("G"), p("O"), p("X"), p("diffusion"), ne, d, d + 1, 1, None, st)
        return [s["mass"], s["diffusion"]]
    if kind == "mass_ragged":
        L.rpx_fill_const_f64(p("Y"), s["Y"].numel(), 0.0, st)
        L.rpx_mass3dpa_batched_run(p("scratch"), None, st)
        return [s["Y"]]
    L.rpx_copy_f64(p("sorted"), p("src"), s["src"].numel(), None, st)
    L.rpx_sort_segmented_f64(p("sorted"), s["off"], s["count"], p("sort_scratch"), s["sort_bytes"], st)
    if kind == "sort":
        return [s["sorted"]]
    L.rpx_scan_exclusive_segmented_f64(p("src"), p("scan"), s["off"], s["count"], p("scan_scratch"), s["scan_bytes"],
                                       st)
    return [s["sorted"], s["scan"]]


# ---- what a pass cannot do without ----------------------------------------------


def _mass_work(ne, d):
    q = d + 1
    flops = 2 * (d**3 * q + d**2 * q**2 + d * q**3) * 2 + q**3 + d**3
    return 8 * ne * (3 * d**3 + q**3), ne * flops


def work(case):
    kind = case["kind"]
    if kind == "stream":  # a and b in, four arrays out
        return {"bytes": 8 * 6 * case["n"], "flops": 6 * case["n"]}
    if kind == "hbm":
        return {"bytes": 8 * 5 * case["n"], "flops": 6 * case["n"]}
    if kind == "scan_sum":
        return {"bytes": 8 * 2 * case["n"], "flops": 2 * case["n"]}
    if kind == "jacobi":
        N = case["N"]
        return {"bytes": 8 * 3 * N * N, "flops": 10 * (N - 2)**2 * case["tsteps"]}
    if kind in ("gemm", "gemm_mixed"):
        ni, nj, nk = case["ni"], case["nj"], case["nk"]
        return {"bytes": 8 * (ni * nk + nk * nj + ni * nj * (2 if case["beta"] else 1)), "flops": 2 * ni * nj * nk}
    if kind == "fem":
        ne, d, q = case["ne"], case["d"], case["d"] + 1
        mb, mf = _mass_work(ne, d)
        flops = 2 * (2 * d**3 * q + 3 * d**2 * q**2 + 3 * d * q**3) * 2 + 15 * q**3 + 3 * d**3
        return {"bytes": mb + 8 * ne * (2 * d**3 + 6 * q**3), "flops": mf + ne * flops}
    if kind == "mass_ragged":
        each = [_mass_work(ne, d) for ne, d in _batches(case)]
        return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}
    n = case["n"] if kind == "sort" else _offsets(case)[-1]
    return {"bytes": 8 * n * (2 if kind == "sort" else 3), "flops": 0}


# ---- the same in plain torch -----------------------------------------------------


def _mass(B, Bt, D, X, ne, d):
    q = d + 1
    b = B.view(d, q)  # [d][q]
    at = torch.arange(q, device="cuda")[None, :] + d * torch.arange(d, device="cuda")[:, None]
    bt = Bt[at]  # the suite's literal Bt[q + D*d]
    t = _apply(X.view(ne, d, d, d), b, b, b) * D.view(ne, q, q, q)
    return _apply(t, bt.T, bt.T, bt.T).reshape(-1)


def _apply(x, mz, my, mx):
    """x[e][z][y][x] contracted with mz[z][.], my[y][.], mx[x][.]."""
    x = torch.matmul(x, mx.contiguous())
    x = torch.matmul(x.transpose(2, 3).contiguous(), my.contiguous()).transpose(2, 3)
    return torch.matmul(x.permute(0, 2, 3, 1).contiguous(), mz.contiguous()).permute(0, 3, 1, 2).contiguous()


def _diffusion(B, G, O, X, ne, d):
    q = d + 1
    b, g, o, x = B.view(d, q), G.view(d, q), O.view(ne, 6, q, q, q), X.view(ne, d, d, d)
    u, v, w = _apply(x, b, b, g), _apply(x, b, g, b), _apply(x, g, b, b)
    o11, o12, o13, o22, o23, o33 = (o[:, c] for c in range(6))
    fu, fv, fw = o11 * u + o12 * v + o13 * w, o12 * u + o22 * v + o23 * w, o13 * u + o23 * v + o33 * w
    bt, gt = b.T, g.T
    return (_apply(fu, bt, bt, gt) + _apply(fv, bt, gt, bt) + _apply(fw, gt, bt, bt)).reshape(-1)


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    if kind == "stream":
        a, b = s["a"], s["b"]
        return [a.clone(), ALPHA * b, a + b, b + ALPHA * a, (a * b).sum().reshape(1)]
    if kind in ("hbm", "scan_sum"):
        out = [s["a"] + ALPHA * s["b"], (s["a"] * s["b"]).sum().reshape(1)] if kind == "hbm" else []
        y = torch.cumsum(s["x"], 0)
        return out + [s["x"].sum().reshape(1), y if case.get("inclusive") else torch.cat([_zeros(1), y[:-1]])]
    if kind == "jacobi":
        N = case["N"]
        A, B = s["A0"].clone().view(N, N), s["B"].clone().view(N, N)
        for _ in range(case["tsteps"]):
            for dst, src in ((B, A), (A, B)):
                dst[1:-1, 1:-1] = 0.2 * (src[1:-1, 1:-1] + src[1:-1, :-2] + src[1:-1, 2:] + src[2:, 1:-1]
                                         + src[:-2, 1:-1])
        return [A.reshape(-1), B.reshape(-1)]
    if kind in ("gemm", "gemm_mixed"):
        ni, nj, nk = case["ni"], case["nj"], case["nk"]
        c = GEMM_ALPHA * (s["A"].view(ni, nk) @ s["B"].view(nk, nj))
        if case["beta"]:
            c += GEMM_BETA * s["C0"].view(ni, nj)
        return [c.reshape(-1)]
    if kind == "fem":
        ne, d = case["ne"], case["d"]
        return [_mass(s["B"], s["Bt"], s["D"], s["X"], ne, d), _diffusion(s["B"], s["G"], s["O"], s["X"], ne, d)]
    if kind == "mass_ragged":
        out, x, q = [], 0, 0
        for ne, d in _batches(case):
            nx, nq = ne * d**3, ne * (d + 1)**3
            out.append(_mass(s["bases"][d][0], s["bases"][d][1], s["D"][q:q + nq], s["X"][x:x + nx], ne, d))
            x, q = x + nx, q + nq
        return [torch.cat(out)]
    off, src = list(s["off"]), s["src"]
    parts = [src[i:j] for i, j in zip(off, off[1:])]
    out = [torch.cat([torch.sort(t).values for t in parts])]
    if kind == "segments":
        out.append(torch.cat([torch.cumsum(t, 0) - t for t in parts]))
    return out
