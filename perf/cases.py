"""Performance cases of remifa_amd: the calls that a program solving linear
systems with the library makes, from the smallest to the largest it is used
for, each through the public entry points.

kinds
  solve      one system from scratch: convert A to fp16, factor, refine in FP64
  lu         one factorization (driver, storage and update type by ``path``)
  getrs      triangular solves with factors that are already there
  gemm       one update product through ``gemmex``
  batched    many small systems: factor and solve
  autograd   differentiable solve, forward and backward
  equil      row / column scaling of a badly scaled matrix, then fp16

A factorization works in place, so a pass starts from the caller's matrix: it
is copied (or, for fp16 storage, converted) into the working buffer first, as
a program that keeps A for its residuals does.
"""
from __future__ import annotations

import random

import numpy as np
import torch

import remifa_amd as rf

F16, F32, F64 = torch.float16, torch.float32, torch.float64

# LU paths: (storage, the reference's helper name or None, generic driver's
# algorithm, inner and outer update types, panel precision, ib)
PATHS = {
    "ll_f32": (F32, "lu_nopiv_ll_f32", None),
    "ll_f32_tc32": (F32, "lu_nopiv_ll_f32_tc32xtc32", None),
    "ll_f32_fp32xtc32": (F32, "lu_nopiv_ll_f32_fp32xtc32", None),
    "ll_f16_tc32": (F16, "lu_nopiv_ll_f16_tc32xtc32", None),
    "ll_f16_tc32_fp32": (F16, "lu_nopiv_ll_f16_tc32xtc32_fp32xfp32_fp32xfp32", None),
    "ll_f16_tc16": (F16, "lu_nopiv_ll_f16_tc16xtc16", None),
    "rl_f16_tc32": (F16, None, (rf.RL, rf.TC32, rf.TC32, rf.R_16F)),
    "rl_f32": (F32, None, (rf.RL, rf.FP32, rf.FP32, rf.R_32F)),
    "ll_f16_bf16": (F16, None, (rf.LL, rf.TC32, rf.BF16_TC32, rf.R_32F)),
    "ll_f16_fp8": (F16, None, (rf.LL, rf.TC32, rf.FP8_TC32, rf.R_32F)),
}

GEMMS = {
    "tc32": (rf.TC32, F16),
    "bf16": (rf.BF16_TC32, F16),
    "fp32": (rf.FP32, F32),
    "fp8": (rf.FP8_TC32, F16),
    "tc16": (rf.TC16, F16),
}


def listed():
    return [
        # a single small system in a loop of many different ones: launches
        # and latency, the smallest call
        {"name": "lu_small", "kind": "lu", "path": "ll_f32_tc32", "n": 300, "nb": 128, "pad": 0},
        # the reference's mixed-precision helper on a size that divides by
        # nothing, fp16 panels, ib = 8
        {"name": "lu_f16_ragged", "kind": "lu", "path": "ll_f16_tc32", "n": 5001, "nb": 256,
         "pad": 2},
        # the plain single-precision factorization everything is compared with
        {"name": "lu_f32", "kind": "lu", "path": "ll_f32", "n": 8192, "nb": 256, "pad": 0},
        # the right-looking driver, fp16 storage
        {"name": "lu_rl", "kind": "lu", "path": "rl_f16_tc32", "n": 4096, "nb": 256, "pad": 0},
        # fp16 accumulation throughout (the reference's TC16 helper)
        {"name": "lu_f16_acc16", "kind": "lu", "path": "ll_f16_tc16", "n": 3000, "nb": 256,
         "pad": 0},
        # one right-hand side against kept factors: latency of the solve
        {"name": "getrs_one", "kind": "getrs", "n": 1000, "nrhs": 1, "storage": "f16",
         "trans": False},
        # a Schur-complement sized update product, not a multiple of a tile
        {"name": "gemm_tc32", "kind": "gemm", "ctype": "tc32", "m": 8000, "n": 6000, "k": 2000,
         "out": "f32"},
        # the same through block-scaled FP8 operands (quantization included)
        {"name": "gemm_fp8", "kind": "gemm", "ctype": "fp8", "m": 8192, "n": 8192, "k": 4096,
         "out": "f32"},
        # many small independent systems of mixed order
        {"name": "batched", "kind": "batched", "count": 4000, "lo": 16, "hi": 512},
        # a solve inside a differentiable program, several right-hand sides
        {"name": "autograd", "kind": "autograd", "n": 4096, "nrhs": 64, "storage": "f32",
         "nb": 256},
        # badly scaled input made fit for fp16: memory-bound passes
        {"name": "equil", "kind": "equil", "m": 16384, "n": 16384},
        # the largest: half-footprint factorization and refinement to FP64
        # accuracy
        {"name": "solve_large", "kind": "solve", "n": 32768, "nb": 512, "nrhs": 1},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["lu", "lu", "lu", "solve", "solve", "getrs", "gemm", "gemm", "batched",
                       "autograd", "equil"])
    if kind == "lu":
        path = rng.choice(sorted(PATHS))
        top = 4096 if path.endswith("tc16") else 8192
        return {"kind": kind, "path": path, "n": _log_int(rng, 64, top),
                "nb": rng.choice([128, 256, 512]), "pad": rng.choice([0, 0, 1, 2, 8])}
    if kind == "solve":
        return {"kind": kind, "n": _log_int(rng, 500, 24000), "nb": rng.choice([256, 512]),
                "nrhs": rng.choice([1, 1, 2, 16])}
    if kind == "getrs":
        return {"kind": kind, "n": _log_int(rng, 100, 16000), "nrhs": _log_int(rng, 1, 64),
                "storage": rng.choice(["f16", "f32"]), "trans": rng.random() < 0.4}
    if kind == "gemm":
        ctype = rng.choice(sorted(GEMMS))
        top = 2048 if ctype == "tc16" else 8192
        step = rng.choice([1, 8, 64, 256])
        m, n, k = (max(step, _log_int(rng, 64, top) // step * step) for _ in range(3))
        return {"kind": kind, "ctype": ctype, "m": m, "n": n, "k": k,
                "out": "f16" if ctype == "tc16" else rng.choice(["f32", "f16"])}
    if kind == "batched":
        hi = rng.choice([32, 64, 128, 256, 512])
        return {"kind": kind, "count": _log_int(rng, 32, 4000), "lo": rng.choice([4, hi // 2]),
                "hi": hi}
    if kind == "autograd":
        return {"kind": kind, "n": _log_int(rng, 200, 4096), "nrhs": _log_int(rng, 1, 64),
                "storage": rng.choice(["f16", "f32"]), "nb": rng.choice([256, 512])}
    return {"kind": kind, "m": _log_int(rng, 200, 16384), "n": _log_int(rng, 200, 16384)}


# ------------------------------------------------------------------ inputs
def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(shape, g, dtype=F32):
    return torch.rand(shape, generator=g, device="cuda", dtype=dtype).mul_(2.0).sub_(1.0)


def _col_major(n, seed, ld, alpha):
    """n x n fp32, uniform(-1, 1) with a_ii = alpha * sum of the rest of its
    row: what a no-pivot factorization is used on. Column-major, stride ld."""
    buf = _uniform((n, ld), _gen(seed))
    a = buf.t()[:n]
    step = 4096  # row sums by column slabs: no second matrix
    s = torch.zeros(n, dtype=F64, device="cuda")
    for j in range(0, n, step):
        s += a[:, j:j + step].abs().sum(1, dtype=F64)
    d = a.diagonal()
    d.copy_(alpha * (s - d.abs().double()))
    return a


def _rhs(n, nrhs, seed, dtype):
    return _uniform((nrhs, n), _gen(seed + 7919), dtype).t()


def _factors(n, seed, dtype):
    """Factors as a no-pivot LU of such a matrix leaves them: U with a large
    diagonal, multipliers below it of the size 1 / u_kk."""
    buf = _uniform((n, n), _gen(seed))
    d = 0.55 * n + 2.0
    a = buf.t()
    a.copy_(torch.triu(a, 1) + torch.tril(a, -1) / d)
    a.diagonal().fill_(0.0).add_(d * (1.0 + 0.1 * _uniform((n,), _gen(seed + 1))))
    return buf.to(dtype).t()


def _gemm_inputs(case, seed):
    _, dt = GEMMS[case["ctype"]]
    m, n, k = case["m"], case["n"], case["k"]
    # multipliers are small, entries of U are of the size of A's
    a = (_uniform((k, m), _gen(seed)) * 0.1).to(dt).t()
    b = _uniform((n, k), _gen(seed + 1)).to(dt).t()
    return a, b


def _batch_sizes(case):
    r = np.random.default_rng([case["count"], case["lo"], case["hi"]])
    s = r.integers(case["lo"], case["hi"] + 1, case["count"])
    return np.sort(s)[::-1].astype(np.int64).copy()  # largest first


def _batch_inputs(case, seed):
    sizes = _batch_sizes(case)
    offs = np.concatenate([[0], np.cumsum(sizes * sizes)[:-1]])
    boffs = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    a = _uniform((int((sizes * sizes).sum()),), _gen(seed))
    for n, o in zip(sizes.tolist(), offs.tolist()):
        v = a[o:o + n * n].view(n, n)  # row j of v is column j of the matrix
        d = v.diagonal()
        d.copy_(1.2 * (v.abs().sum(0) - d.abs()) + 0.5)
    b = _uniform((int(sizes.sum()),), _gen(seed + 1))
    return sizes, offs, boffs, a, b


def _equil_input(case, seed):
    m, n = case["m"], case["n"]
    g = _gen(seed)
    a = _uniform((n, m), g)
    er = torch.randint(-12, 13, (m,), generator=g, device="cuda").to(F32)
    ec = torch.randint(-12, 13, (n,), generator=g, device="cuda").to(F32)
    a.mul_(torch.exp2(er)[None, :]).mul_(torch.exp2(ec)[:, None])
    return a.t()


def _autograd_inputs(case, seed):
    n, r = case["n"], case["nrhs"]
    a = _col_major(n, seed, n, 1.1).contiguous()
    b = _uniform((n, r), _gen(seed + 1), F64)
    w = _uniform((n, r), _gen(seed + 2), F64)
    return a, b, w


# ------------------------------------------------------------------ passes
class State:
    pass


def prepare(case, seed):
    s = State()
    s.case = case
    k = case["kind"]
    s.h = rf.Handle()
    if k == "solve":
        n = case["n"]
        s.a = _col_major(n, seed, n, 1.05)
        s.b = _rhs(n, case["nrhs"], seed, F64)
        s.lu = rf.colmajor_empty(n, n, dtype=F16)
        s.x = rf.colmajor_empty(n, case["nrhs"], dtype=F64)
        s.info = torch.zeros(1, dtype=torch.int32, device="cuda")
        s.cfg = rf.api.make_config(W=rf.R_16F, I=rf.TC32, O=rf.TC32, OP=rf.R_32F, ib=32)
    elif k == "lu":
        n, ld = case["n"], case["n"] + case["pad"]
        dt, _, generic = PATHS[case["path"]]
        s.a = _col_major(n, seed, ld, 1.05)
        s.lu = rf.colmajor_empty(n, n, dtype=dt, ld=ld)
        s.ld = ld
        s.info = torch.zeros(1, dtype=torch.int32, device="cuda")
        if generic:
            _, inner, outer, op = generic
            s.cfg = rf.api.make_config(W=rf.dtype_code(dt), I=inner, O=outer, OP=op, ib=32)
        # the fp16 copy that the reference's mixed helpers take
        mixed = dt == F32 and "tc32" in case["path"]
        s.cpy = rf.colmajor_empty(n, n, dtype=F16, ld=ld) if mixed else None
    elif k == "getrs":
        dt = F16 if case["storage"] == "f16" else F32
        s.lu = _factors(case["n"], seed, dt)
        s.b = _rhs(case["n"], case["nrhs"], seed, F32)
        s.x = rf.colmajor_empty(case["n"], case["nrhs"], dtype=F32)
    elif k == "gemm":
        s.a, s.b = _gemm_inputs(case, seed)
        s.c = rf.colmajor_empty(case["m"], case["n"], dtype=F32 if case["out"] == "f32" else F16)
    elif k == "batched":
        s.sizes, offs, boffs, s.a, s.b = _batch_inputs(case, seed)
        s.lu, s.x = torch.empty_like(s.a), torch.empty_like(s.b)
        s.ptrs = torch.tensor(s.lu.data_ptr() + 4 * offs, dtype=torch.int64, device="cuda")
        s.bptrs = torch.tensor(s.x.data_ptr() + 4 * boffs, dtype=torch.int64, device="cuda")
        s.n_t = torch.tensor(s.sizes, dtype=torch.int32, device="cuda")
        s.info = torch.zeros(len(s.sizes), dtype=torch.int32, device="cuda")
        s.buckets = []
        for lo, hi in ((256, 512), (128, 256), (64, 128), (0, 64)):
            i = np.nonzero((s.sizes > lo) & (s.sizes <= hi))[0]
            if len(i):
                s.buckets.append((int(i[0]), int(i[-1]) + 1, hi))
    elif k == "autograd":
        a, b, s.w = _autograd_inputs(case, seed)
        s.a, s.b = a.requires_grad_(), b.requires_grad_()
    else:
        s.a = _equil_input(case, seed)
        m, n = case["m"], case["n"]
        s.scaled = rf.colmajor_empty(m, n, dtype=F32)
        s.half = rf.colmajor_empty(m, n, dtype=F16)
        s.r = torch.empty(m, dtype=F32, device="cuda")
        s.c = torch.empty(n, dtype=F32, device="cuda")
    return s


def run(s):
    case, h = s.case, s.h
    k = case["kind"]
    if k == "solve":
        rf.convert(h, s.a, s.lu)
        rf.lu_nopiv(h, s.lu, case["nb"], algo=rf.LL, cfg=s.cfg, info=s.info)
        rf.ir_solve(h, s.a, s.lu, s.b, s.x, tol=1e-14, maxit=30)
        return {"lu": s.lu, "x": s.x, "info": s.info}
    if k == "lu":
        dt, helper, generic = PATHS[case["path"]]
        if dt == F16:
            rf.convert(h, s.a, s.lu)
        else:
            s.lu.copy_(s.a)
        if helper:
            f = getattr(rf, helper)
            args = (h, case["n"], case["n"], case["nb"], s.lu, s.ld, s.info)
            f(*args, s.cpy, s.ld) if s.cpy is not None else f(*args)
        else:
            rf.lu_nopiv(h, s.lu, case["nb"], algo=generic[0], cfg=s.cfg, info=s.info)
        return {"lu": s.lu, "info": s.info}
    if k == "getrs":
        s.x.copy_(s.b)
        rf.getrs_nopiv(h, s.lu, s.x, trans=case["trans"])
        return s.x
    if k == "gemm":
        rf.gemmex(h, GEMMS[case["ctype"]][0], s.a, s.b, s.c, alpha=-1.0, beta=0.0)
        return s.c
    if k == "batched":
        s.lu.copy_(s.a)
        s.x.copy_(s.b)
        for i, j, hi in s.buckets:
            rf.lu_nopiv_batched(h, rf.TC32, s.n_t[i:j], s.n_t[i:j], s.ptrs[i:j], s.info[i:j], hi)
        rf.getrs_nopiv_batched(h, s.n_t, s.n_t, s.ptrs, s.bptrs, s.buckets[0][2])
        return {"lu": s.lu, "x": s.x, "info": s.info}
    if k == "autograd":
        x = rf.autograd.solve(s.a, s.b, nb=case["nb"], storage=case["storage"])
        ga, gb = torch.autograd.grad(x, (s.a, s.b), grad_outputs=s.w)
        return {"x": x.detach(), "grad_a": ga, "grad_b": gb}
    s.scaled.copy_(s.a)
    q = rf.geequb(h, s.a, s.r, s.c)
    rf.laqge(h, s.scaled, s.r, s.c, q["rowcnd"], q["colcnd"], q["amax"])
    rf.convert(h, s.scaled, s.half)
    return {"r": s.r, "c": s.c, "scaled": s.scaled, "half": s.half,
            "cond": [q["rowcnd"], q["colcnd"], q["amax"]]}


# ------------------------------------------------------------------ work
def work(case):
    k = case["kind"]
    if k in ("solve", "lu"):
        n = float(case["n"])
        if k == "solve":
            # A once for the fp16 copy, the factors written, then at least
            # one residual (A) and one solve (the factors)
            r = case["nrhs"]
            return {"bytes": 4 * n * n * 2 + 2 * n * n * 2 + 24 * n * r,
                    "flops": 2 * n**3 / 3 + 4 * n * n * r}
        es = 2 if PATHS[case["path"]][0] == F16 else 4
        return {"bytes": (4 + es) * n * n, "flops": 2 * n**3 / 3}
    if k == "getrs":
        n, r = float(case["n"]), case["nrhs"]
        return {"bytes": n * n * (2 if case["storage"] == "f16" else 4) + 8 * n * r,
                "flops": 2 * n * n * r}
    if k == "gemm":
        m, n, kk = float(case["m"]), float(case["n"]), float(case["k"])
        es = 4 if GEMMS[case["ctype"]][1] == F32 else 2
        return {"bytes": es * (m * kk + kk * n) + (4 if case["out"] == "f32" else 2) * m * n,
                "flops": 2 * m * n * kk}
    if k == "batched":
        lo, hi, c = case["lo"], case["hi"], case["count"]
        ns = np.arange(lo, hi + 1, dtype=np.float64)
        return {"bytes": c * float((8 * ns**2 + 8 * ns).mean()),
                "flops": c * float((2 * ns**3 / 3 + 2 * ns**2).mean())}
    if k == "autograd":
        n, r = float(case["n"]), case["nrhs"]
        # forward LU and solve, adjoint solve, the outer product for grad_a
        return {"bytes": 4 * n * n * 2 + 8 * n * r * 4,
                "flops": 2 * n**3 / 3 + 2 * 4 * n * n * r + 2 * n * n * r}
    m, n = float(case["m"]), float(case["n"])
    return {"bytes": (4 + 4 + 2) * m * n + 4 * (m + n), "flops": 3 * m * n}


# ------------------------------------------------------------------ 64 bits
def _lu64(a):
    """In-place no-pivot LU in FP64, blocks of 256 columns."""
    n = a.shape[0]
    for k in range(0, n, 256):
        e = min(k + 256, n)
        d = a[k:e, k:e].clone()
        for i in range(e - k - 1):
            d[i + 1:, i] /= d[i, i]
            d[i + 1:, i + 1:].sub_(torch.outer(d[i + 1:, i], d[i, i + 1:]))
        a[k:e, k:e] = d
        if e < n:
            a[e:, k:e] = torch.linalg.solve_triangular(d, a[e:, k:e], upper=True, left=False)
            a[k:e, e:] = torch.linalg.solve_triangular(d, a[k:e, e:], upper=False,
                                                       unitriangular=True)
            a[e:, e:].sub_(a[e:, k:e] @ a[k:e, e:])
    return a


def _lu_solve64(lu, b, trans=False):
    st = torch.linalg.solve_triangular
    if trans:
        lut = lu.t()
        y = st(lut, b, upper=False)
        return st(lut, y, upper=True, unitriangular=True)
    return st(lu, st(lu, b, upper=False, unitriangular=True), upper=True)


def _solve64(a, lu, b, trans=False):
    """A x = b in FP64, refined from factors of a nearby matrix."""
    m = a.t() if trans else a
    x = _lu_solve64(lu, b, trans)
    for _ in range(10):
        x = x + _lu_solve64(lu, b - m @ x, trans)
    return x


def _e4m3(v):
    """Rows of v in OCP e4m3 with one power-of-two scale for each 32 of them
    (2^(floor(log2 amax) - 8)), widened again: the values that the scaled
    matrix cores multiply."""
    r, k = v.shape
    kp = -(-k // 32) * 32
    w = torch.zeros((r, kp), dtype=F64, device=v.device)
    w[:, :k] = v
    w = w.view(r, kp // 32, 32)
    _, e = torch.frexp(w.abs().amax(2, keepdim=True))
    sc = torch.exp2((e - 9).to(F64))
    q = (w / sc).clamp(-448.0, 448.0).to(F32).to(torch.float8_e4m3fn).to(F64)
    return (q * sc).view(r, kp)[:, :k]


def _pow2_trunc(x):
    f, e = torch.frexp(x)
    k = torch.where((x >= 1.0) | (f == 0.5), e - 1, e)
    return torch.exp2(k.to(F64))


def _batched64(case, seed):
    sizes, offs, boffs, a, b = _batch_inputs(case, seed)
    lu = torch.empty(a.numel(), dtype=F64, device="cuda")
    x = torch.empty(b.numel(), dtype=F64, device="cuda")
    for c0 in range(0, len(sizes), 500):
        ix = range(c0, min(c0 + 500, len(sizes)))
        nm = int(sizes[c0])  # largest first
        w = torch.eye(nm, dtype=F64, device="cuda").repeat(len(ix), 1, 1)
        r = torch.zeros((len(ix), nm, 1), dtype=F64, device="cuda")
        for q, i in enumerate(ix):
            n, o, p = int(sizes[i]), int(offs[i]), int(boffs[i])
            w[q, :n, :n] = a[o:o + n * n].view(n, n).t()
            r[q, :n, 0] = b[p:p + n]
        for k in range(nm - 1):
            w[:, k + 1:, k] /= w[:, k:k + 1, k]
            w[:, k + 1:, k + 1:] -= w[:, k + 1:, k:k + 1] * w[:, k:k + 1, k + 1:]
        for k in range(nm - 1):  # unit lower, column by column
            r[:, k + 1:] -= w[:, k + 1:, k:k + 1] * r[:, k:k + 1]
        for k in range(nm - 1, -1, -1):
            r[:, k] /= w[:, k, k:k + 1]
            r[:, :k] -= w[:, :k, k:k + 1] * r[:, k:k + 1]
        for q, i in enumerate(ix):
            n, o, p = int(sizes[i]), int(offs[i]), int(boffs[i])
            lu[o:o + n * n] = w[q, :n, :n].t().reshape(-1)
            x[p:p + n] = r[q, :n, 0]
    return {"lu": lu, "x": x, "info": None}


def exact(case, seed):
    k = case["kind"]
    if k == "solve":
        n = case["n"]
        a = _col_major(n, seed, n, 1.05)
        lu = _lu64(a.half().double())  # of the matrix as it is stored
        b = _rhs(n, case["nrhs"], seed, F64)
        return {"lu": lu, "x": _solve64(a.double(), lu, b), "info": None}
    if k == "lu":
        n = case["n"]
        a = _col_major(n, seed, n + case["pad"], 1.05)
        return {"lu": _lu64(a.to(PATHS[case["path"]][0]).double()), "info": None}
    if k == "getrs":
        lu = _factors(case["n"], seed, F16 if case["storage"] == "f16" else F32).double()
        return _lu_solve64(lu, _rhs(case["n"], case["nrhs"], seed, F32).double(), case["trans"])
    if k == "gemm":
        a, b = _gemm_inputs(case, seed)
        if case["ctype"] == "fp8":
            return -(_e4m3(a.double()) @ _e4m3(b.double().t()).t())
        if case["ctype"] == "bf16":
            a, b = a.to(torch.bfloat16), b.to(torch.bfloat16)
        return -(a.double() @ b.double())
    if k == "batched":
        return _batched64(case, seed)
    if k == "autograd":
        a, b, w = _autograd_inputs(case, seed)
        a = a.double()
        lu = _lu64(a.clone())
        x = _solve64(a, lu, b)
        gb = _solve64(a, lu, w, trans=True)
        return {"x": x, "grad_a": -(gb @ x.t()), "grad_b": gb}
    a = _equil_input(case, seed).double()
    r = _pow2_trunc(a.abs().amax(1))
    c = _pow2_trunc((a.abs() / r[:, None]).amax(0))
    s = a / r[:, None] / c[None, :]
    return {"r": 1.0 / r, "c": 1.0 / c, "scaled": s, "half": s,
            "cond": [float(r.min() / r.max()), float(c.min() / c.max()), float(r.max())]}
