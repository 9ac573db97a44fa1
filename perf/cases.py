"""The work that users of the library have it do, as cases whose time can be measured.

A case is a dict of plain values.  ``prepare`` makes what a program holds before the call (inputs
on the GPU, made from the seed), ``run`` is one pass through the public entry points, ``work`` the
bytes and operations that the pass cannot do without, ``exact`` the result in 64 bits by plain
torch.  ``listed`` are fixed cases, ``draw`` gives more of the same ranges.

Kinds:

* ``llt``    ``LLT(A).solve(B)``: the object mirror of Eigen's class, double or float storage;
* ``posv``   factor and solve in place on working copies (``posv_async_``), as a program that
             keeps its buffers does;
* ``solve``  one more solve with a factor that the program keeps (``LLT.solve``);
* ``mixed``  low-precision factor with FP64 refinement (``posv_mixed``);
* ``vbatch`` independent systems of uneven order in one launch (``posv_vbatched_``);
* ``gp``     Gaussian-process log marginal likelihood and its gradient, one system;
* ``gpbatch`` the same for a batch of systems of one order.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("eigen-git-mirror_amd"))

import mi_llt  # noqa: E402
from mi_llt import autograd, batched, workloads  # noqa: E402

_DTYPES = {"f64": torch.float64, "f32": torch.float32}


def listed():
    return [
        # the smallest call: a hundred unknowns, one right-hand side (a row of Eigen's own
        # benchmark table); latency and launches are all of it
        {"name": "llt_n100_r1", "kind": "llt", "n": 100, "r": 1, "dtype": "f64", "uplo": "L"},
        # an ordinary dense system (the size of the plain CPU workload)
        {"name": "llt_n1024_r16", "kind": "llt", "n": 1024, "r": 16, "dtype": "f64", "uplo": "L"},
        # single precision storage, an odd size
        {"name": "llt_f32_n4001_r4", "kind": "llt", "n": 4001, "r": 4, "dtype": "f32", "uplo": "L"},
        # a ragged order in upper storage, with a leading dimension that is no multiple of anything
        {"name": "posv_upper_n3001_r7", "kind": "posv", "n": 3001, "r": 7, "pad": 2, "uplo": "U"},
        # the benchmark: a large dense system with many right-hand sides
        {"name": "posv_n8192_r64", "kind": "posv", "n": 8192, "r": 64, "pad": 0, "uplo": "L"},
        # a program that factored once and solves for each new right-hand side
        {"name": "solve_n4000_r1", "kind": "solve", "n": 4000, "r": 1, "uplo": "L"},
        # the largest: low-precision factor, FP64 refinement
        {"name": "mixed_n16384_r16", "kind": "mixed", "n": 16384, "r": 16, "kappa": 100.0, "prec": "bf16x3"},
        # thousands of small uneven systems, in double and in single precision, and a short batch
        {"name": "vbatch_f64_20000", "kind": "vbatch", "count": 20000, "nmin": 8, "nmax": 256, "rmax": 8, "sizes": 0,
         "dtype": "f64"},
        {"name": "vbatch_f32_20000", "kind": "vbatch", "count": 20000, "nmin": 8, "nmax": 256, "rmax": 8, "sizes": 0,
         "dtype": "f32"},
        {"name": "vbatch_f64_700", "kind": "vbatch", "count": 700, "nmin": 8, "nmax": 256, "rmax": 8, "sizes": 1, "dtype": "f64"},
        # one large Gaussian process, and a batch of small ones, likelihood and gradient (a batch
        # whose workgroups are all resident at once: four 128-blocks of each of 120 systems)
        {"name": "gp_n4096", "kind": "gp", "n": 4096},
        {"name": "gpbatch_120x512", "kind": "gpbatch", "count": 120, "n": 512},
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["llt", "llt", "posv", "posv", "solve", "mixed", "vbatch", "vbatch", "gp", "gpbatch"])
    if kind == "llt":
        return {"kind": kind, "n": _log(rng, 8, 5000), "r": _log(rng, 1, 64), "dtype": rng.choice(["f64", "f64", "f32"]),
                "uplo": rng.choice("LLU")}
    if kind == "posv":
        return {"kind": kind, "n": _log(rng, 64, 8192), "r": _log(rng, 1, 64), "pad": rng.choice([0, 0, rng.randrange(1, 40)]),
                "uplo": rng.choice("LLLU")}
    if kind == "solve":
        return {"kind": kind, "n": _log(rng, 64, 8192), "r": _log(rng, 1, 64), "uplo": rng.choice("LLLU")}
    if kind == "mixed":
        return {"kind": kind, "n": _log(rng, 2000, 16384), "r": rng.randrange(1, 17), "kappa": 10.0 ** rng.uniform(1, 4),
                "prec": rng.choice(["bf16x3", "bf16x6", "fp32"])}
    if kind == "vbatch":
        return {"kind": kind, "count": _log(rng, 100, 20000), "nmin": rng.randrange(1, 17), "nmax": rng.randrange(32, 257),
                "rmax": rng.randrange(1, 9), "sizes": rng.randrange(1000), "dtype": rng.choice(["f64", "f32"])}
    if kind == "gp":
        return {"kind": kind, "n": _log(rng, 200, 4096)}
    return {"kind": kind, "count": _log(rng, 8, 120), "n": _log(rng, 64, 512)}


# ------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(gen, *shape):
    return torch.randn(*shape, dtype=torch.float64, device="cuda", generator=gen)


def _gram(gen, n):
    """B B^T / n + 0.1 I, B iid N(0,1): the dense workloads' matrix."""
    g = _randn(gen, n, n)
    a = torch.matmul(g, g.t().contiguous()) / n
    a.diagonal().add_(0.1)
    return a


def _empty_colmajor(n, m, ld):
    """An n x m column-major tensor with leading dimension ld."""
    return torch.empty_strided((n, m), (1, ld), dtype=torch.float64, device="cuda")


def _vbatch(case, seed):
    """The uneven batch: n_i ~ U{nmin..nmax}, 1..rmax right-hand sides (drawn with the case's own
    "sizes", so that every seed has the same shapes), A_i = B_i B_i^T / n_i + 0.1 I, in the flat
    buffers of a VBatch.  The matrices are made per order."""
    rng = np.random.default_rng(case["sizes"])
    ns = rng.integers(case["nmin"], case["nmax"] + 1, size=case["count"])
    rs = rng.integers(1, case["rmax"] + 1, size=case["count"])
    vb = batched.VBatch(ns, rs, dtype=_DTYPES[case["dtype"]])
    gen = _gen(seed)
    off = torch.from_numpy(vb.a_off).cuda()
    for n in np.unique(ns):
        n = int(n)
        at = off[torch.from_numpy(np.nonzero(ns == n)[0]).cuda()]
        g = _randn(gen, len(at), n, n)
        a = torch.matmul(g, g.transpose(1, 2).contiguous()) / n
        a.diagonal(dim1=1, dim2=2).add_(0.1)
        vb.a_flat[at[:, None] + torch.arange(n * n, device="cuda")] = a.reshape(len(at), n * n).to(vb.dtype)
    vb.b_flat.copy_(_randn(gen, vb.b_flat.numel()).to(vb.dtype))
    return vb


def _gp_batch(seed, count, n, d=8, ell=1.5, sigma2=1e-2):
    """K = exp(-|x_i - x_j|^2 / (2 ell^2)) + sigma2 I of count sets of n points, and targets."""
    gen = _gen(seed)
    x = _randn(gen, count, n, d)
    d2 = torch.zeros(count, n, n, dtype=torch.float64, device="cuda")
    for j in range(d):
        d2 += (x[:, :, None, j] - x[:, None, :, j]) ** 2
    k = torch.exp(d2 / (-2.0 * ell * ell))
    k.diagonal(dim1=1, dim2=2).add_(sigma2)
    return k, _randn(gen, count, n)


def _inputs(case, seed):
    """(A, B) of a dense case, as a program has them."""
    gen = _gen(seed)
    a = _gram(gen, case["n"])
    b = _randn(gen, case["r"], case["n"]).t()
    return a, b


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("llt", "solve"):
        dt = _DTYPES[case.get("dtype", "f64")]
        a, b = _inputs(case, seed)
        s["a"], s["b"] = a.to(dt), b.to(dt)
        if kind == "solve":
            s["llt"] = mi_llt.LLT(s["a"], uplo=case["uplo"])
            del s["a"]
    elif kind == "posv":
        n, r, ld = case["n"], case["r"], case["n"] + case["pad"]
        a, b = _inputs(case, seed)
        s["a"], s["b"] = _empty_colmajor(n, n, ld).copy_(a), _empty_colmajor(n, r, ld).copy_(b)
        s["l"], s["x"] = _empty_colmajor(n, n, ld), _empty_colmajor(n, r, ld)
        s["info"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    elif kind == "mixed":
        s["a"] = workloads.spectrum_spd_torch(case["n"], case["kappa"], seed=seed)
        s["b"] = _empty_colmajor(case["n"], case["r"], case["n"]).copy_(_randn(_gen(seed), case["r"], case["n"]).t())
    elif kind == "vbatch":
        s["vb"] = _vbatch(case, seed)
        s["a"], s["b"] = s["vb"].a_flat.clone(), s["vb"].b_flat.clone()
    elif kind == "gp":
        s["k"], s["y"] = workloads.gp_kernel_torch(case["n"], seed=seed)
    else:
        s["k"], s["y"] = _gp_batch(seed, case["count"], case["n"])
    return s


# ------------------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "llt":
        llt = mi_llt.LLT(state["a"], uplo=case["uplo"], dtype=state["a"].dtype)
        return {"llt": llt.matrixLLT(), "x": llt.solve(state["b"]), "info": int(llt.info())}
    if kind == "solve":
        return {"x": state["llt"].solve(state["b"])}
    if kind == "posv":  # the inputs stay: the call works in place on copies, as LLT::compute does
        state["l"].copy_(state["a"])
        state["x"].copy_(state["b"])
        mi_llt.posv_async_(state["l"], state["x"], state["info"], uplo=case["uplo"])
        return {"l": state["l"], "x": state["x"], "info": state["info"]}
    if kind == "mixed":
        # the count of corrections and the reached backward error belong to the way there, as a
        # time does: the result is x, and whether there is one
        x, _iters, _berr, info = mi_llt.posv_mixed(state["a"], state["b"], prec=case["prec"], tol=1e-14, maxit=30)
        return {"x": x, "info": info}
    if kind == "vbatch":  # in place: a new batch is put into the same buffers first
        vb = state["vb"]
        vb.a_flat.copy_(state["a"])
        vb.b_flat.copy_(state["b"])
        return {"info": batched.posv_vbatched_(vb), "a": vb.a_flat, "b": vb.b_flat}
    k = state["k"].detach().requires_grad_(True)
    if kind == "gp":
        v = autograd.gp_log_marginal(k, state["y"])
        v.backward()
    else:
        v = autograd.gp_log_marginal_batched(k, state["y"])
        v.sum().backward()
    return {"value": v.detach(), "grad": k.grad}


# ------------------------------------------------------------------------------ work
def _factor_flops(n):
    return n * (n + 1) * (2 * n + 1) / 6.0


def work(case):
    kind = case["kind"]
    if kind == "vbatch":
        # the mean over n ~ U{nmin..nmax} and r ~ U{1..rmax}
        n = np.arange(case["nmin"], case["nmax"] + 1, dtype=np.float64)
        r = (1 + case["rmax"]) / 2.0
        es = 8 if case["dtype"] == "f64" else 4
        return {"bytes": case["count"] * float(np.mean(n * (n + 1) + 2 * n * r)) * es,
                "flops": case["count"] * float(np.mean(_factor_flops(n) + 2 * n * n * r))}
    n = float(case["n"])
    if kind in ("gp", "gpbatch"):
        # the factor, and K^-1 for the gradient (a a^T - K^-1) / 2
        c = case.get("count", 1)
        return {"bytes": c * (n * (n + 1) / 2 + n * n) * 8, "flops": c * (_factor_flops(n) + 2 * n ** 3 / 3 + 2 * n * n)}
    r = float(case["r"])
    es = 4 if case.get("dtype") == "f32" else 8
    tri = n * (n + 1) / 2
    if kind == "solve":
        return {"bytes": (tri + 2 * n * r) * es, "flops": 2 * n * n * r}
    return {"bytes": ((1 if kind == "mixed" else 2) * tri + 2 * n * r) * es, "flops": _factor_flops(n) + 2 * n * n * r}


# ------------------------------------------------------------------------------ 64 bits
def _mirror(a, upper=False):
    """The symmetric matrix of a's lower (or upper) triangle."""
    t = torch.triu(a) if upper else torch.tril(a)
    return t + t.t() - torch.diag(torch.diagonal(t))


def _factor(a, upper=False):
    """What the factorization leaves in a's storage, and L."""
    l = torch.linalg.cholesky(_mirror(a, upper))
    return (torch.triu(l.t()) + torch.tril(a, -1)) if upper else (l + torch.triu(a, 1)), l


def exact(case, seed):
    kind = case["kind"]
    if kind in ("llt", "posv", "solve"):
        dt = _DTYPES[case.get("dtype", "f64")]
        a, b = (t.to(dt).double() for t in _inputs(case, seed))
        m, l = _factor(a, case["uplo"] == "U")
        x = torch.cholesky_solve(b, l)
        if kind == "solve":
            return {"x": x}
        return {"llt" if kind == "llt" else "l": m, "x": x, "info": None}
    if kind == "mixed":
        s = prepare(case, seed)
        return {"x": torch.cholesky_solve(s["b"], torch.linalg.cholesky(_mirror(s["a"]))), "info": None}
    if kind == "vbatch":
        vb = _vbatch(case, seed)
        a, b = vb.a_flat.cpu().double(), vb.b_flat.cpu().double()
        off_a, off_b = torch.from_numpy(vb.a_off), torch.from_numpy(vb.b_off)
        for n in np.unique(vb.ns):
            n = int(n)
            for r in np.unique(vb.rs[vb.ns == n]):
                r = int(r)
                at = torch.from_numpy(np.nonzero((vb.ns == n) & (vb.rs == r))[0])
                ia = off_a[at][:, None] + torch.arange(n * n)
                ib = off_b[at][:, None] + torch.arange(n * r)
                m = a[ia].reshape(-1, n, n)  # column-major: m[z] = A_z^T = A_z
                l = torch.linalg.cholesky(m)
                x = torch.cholesky_solve(b[ib].reshape(-1, r, n).transpose(1, 2).contiguous(), l)
                # the other triangle of the storage keeps A
                a[ia] = (torch.triu(l.transpose(1, 2)) + torch.tril(m, -1)).reshape(-1, n * n)
                b[ib] = x.transpose(1, 2).reshape(-1, r * n)
        return {"info": None, "a": a, "b": b}
    s = prepare(case, seed)
    k, y = (s["k"].cpu(), s["y"].cpu()) if kind == "gpbatch" else (s["k"].cpu()[None], s["y"].cpu()[None])
    l = torch.linalg.cholesky(k)
    al = torch.cholesky_solve(y[..., None], l)
    grad = 0.5 * (al * al.transpose(1, 2) - torch.cholesky_inverse(l))
    v = (-0.5 * (y * al[..., 0]).sum(-1) - torch.log(torch.diagonal(l, dim1=1, dim2=2)).sum(-1)
         - 0.5 * k.shape[-1] * math.log(2.0 * math.pi))
    return {"value": v, "grad": grad} if kind == "gpbatch" else {"value": v[0], "grad": grad[0]}
