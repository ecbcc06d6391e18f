"""The measured work of this framework: what a program that uses it has it do.

Operators are 5-point (plane) and 7-point (box) grids, the patterns of the
repository's generators, tests and benchmark: one implicit step of a diffusion
problem, -div(w grad u) + shift u, with conductivities w made from the seed.
The sparsity pattern, its ordering, the symbolic factor and the schedule are
what such a program keeps; values and right-hand sides are new in each step and
already in HBM, except where a case stands for callers with host data.

Every value is a dyadic rational with few bits (conductivities and shift
multiples of 2^-12, solutions of 2^-20), so b = A x is formed without rounding
and the x that b was made from is the exact solution.

Not listed: BF16 trailing updates, which the benchmark measures as slower than
FP32 fronts both in the factorization and in the iterations that follow.
"""
import functools

import numpy as np
import torch

import taucs_amd as T

PREC = {"fp64": T.FP64, "fp32": T.FP32}


def _case(name, kind, dims, nrhs, prec="fp64", coef="smooth", panel=0, tile=0, method=-1):
    return {"name": name, "kind": kind, "x": dims[0], "y": dims[1], "z": dims[2], "nrhs": nrhs,
            "prec": prec, "coef": coef, "panel": panel, "tile": tile, "method": method}


def _batch(name, kind, count, lo, hi, nrhs, prec="fp64", method=-1):
    return {"name": name, "kind": kind, "count": count, "lo": lo, "hi": hi, "nrhs": nrhs,
            "prec": prec, "coef": "smooth", "method": method}


def listed():
    return [
        # the smallest request of a serving mix: launches and latency only
        _case("plane16_step", "step", (16, 16, 1), 1),
        # a TAUCS caller with host arrays: factor_llt_numeric and solve_llt on
        # the 100 x 100 plane of the reference's own examples
        _case("plane100_host", "host", (100, 100, 1), 1),
        # the largest plane of the serving mix, many right-hand sides
        _case("plane256_step16", "step", (251, 256, 1), 16),
        # an ordinary box of odd sides
        _case("box_odd_step3", "step", (37, 23, 51), 3),
        # solve-only request against a resident factor, one right-hand side
        _case("box40_solve1", "solve", (40, 40, 40), 1),
        # solves against the benchmark's factor
        _case("box60_solve8", "solve", (60, 60, 60), 8, panel=256, tile=128),
        # the benchmark's step: numeric factorization and 8 right-hand sides
        _case("box60_step8", "step", (60, 60, 60), 8, panel=256, tile=128),
        # the largest factorization of the benchmark, in FP64
        _case("box80_step4", "step", (80, 80, 80), 4, coef="rough", panel=512, tile=128),
        # mixed precision: FP32 fronts, FP64 conjugate gradients
        _case("box72_mixed4", "refined", (80, 72, 64), 4, "fp32", "rough", 256, 128, 1),
        # mixed precision on an ordinary box: FP32 fronts, classical refinement
        _case("box32_mixed5", "refined", (31, 32, 33), 5, "fp32", method=0),
        # many independent systems in one call (the benchmark's batch)
        _batch("batch512_step", "batch", 512, 16, 128, 1),
        # the same with FP32 fronts, refined, right-hand sides on the host
        _batch("batch96_mixed2", "batch_refined", 96, 17, 100, 2, "fp32", 0),
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    nrhs = rng.choice([1, 1, 2, 3, 4, 5, 8, 11, 16])
    kind = rng.choice(["step", "step", "step", "host", "solve", "refined", "batch", "batch_refined"])
    if kind.startswith("batch"):
        lo = logint(16, 40)
        c = _batch("", kind, logint(8, 512), lo, lo + logint(8, 88), min(nrhs, 4),
                   "fp32" if kind == "batch_refined" else "fp64", 0 if kind == "batch_refined" else -1)
    else:
        if rng.random() < 0.5:
            dims = (logint(16, 256), logint(16, 256), 1)
        else:
            dims = (logint(8, 64), logint(8, 64), logint(8, 64))
        big = dims[2] > 1 and dims[0] * dims[1] * dims[2] > 50000
        panel, tile = rng.choice([(0, 0), (256, 128), (512, 128)]) if big else (0, 0)
        mixed = kind == "refined"
        c = _case("", kind, dims, nrhs, "fp32" if mixed else "fp64",
                  rng.choice(["smooth", "rough"]), panel, tile, rng.choice([0, 1]) if mixed else -1)
    del c["name"]
    return c


# ---- patterns ------------------------------------------------------------------

def _sides(case):
    if "count" not in case:
        return [(case["x"], case["y"], case["z"])]
    s = np.random.default_rng(case["count"]).integers(case["lo"], case["hi"] + 1, case["count"])
    return [(int(q), int(q), 1) for q in s]


@functools.lru_cache(maxsize=None)
def _pattern(dims):
    """Grid pattern (lower part) and its fill-reducing ordering, kept by a
    program for as long as it works on this grid."""
    A = T.mesh3d(*dims)
    n, cp, ri, _ = A.arrays()
    perm, inv = T.order(A, "genmmd")
    return n, cp, ri, np.repeat(np.arange(n), np.diff(cp)), perm, inv


@functools.lru_cache(maxsize=None)
def _counts(dims):
    """Unknowns, stored entries, and the entries and flops of the factor."""
    n, cp, ri, _, perm, inv = _pattern(dims)
    PA = T.permute(T.from_arrays(n, cp, ri, np.zeros(cp[n])), perm, inv)
    i = T.factor_symbolic(PA).info()
    return n, int(cp[n]), i.fund_nnz, i.fund_flops


def _values(dims, coef, rng):
    """Values of the stored entries on the grid (lower part, original order)."""
    n, cp, ri, col, _, _ = _pattern(dims)
    off = ri != col
    if coef == "rough":  # four decades of conductivity
        w, shift = 10.0 ** rng.uniform(-2.0, 2.0, off.sum()), 2.0 ** -3
    else:
        w, shift = rng.uniform(0.5, 1.5, off.sum()), 2.0 ** -6
    w = np.maximum(np.rint(w * 4096.0), 1.0) / 4096.0
    v = np.empty(cp[n])
    v[off] = -w
    v[~off] = np.bincount(ri[off], w, n)[col[~off]] + np.bincount(col[off], w, n)[col[~off]] + shift
    return v


def _system(dims, coef, nrhs, rng):
    """Permuted matrix, right-hand sides and the solution they were made from
    (nrhs x n, one row per right-hand side)."""
    n, cp, ri, col, perm, inv = _pattern(dims)
    v = _values(dims, coef, rng)
    x = np.rint(rng.uniform(-1.0, 1.0, (nrhs, n)) * 2.0 ** 20) / 2.0 ** 20
    off = ri != col
    b = np.stack([np.bincount(ri, v * xr[col], n) + np.bincount(col[off], v[off] * xr[ri[off]], n)
                  for xr in x])
    PA = T.permute(T.from_arrays(n, cp, ri, v), perm, inv)
    return PA, b[:, perm], x[:, perm]


def _systems(case, seed):
    rng = np.random.default_rng(seed)
    return [_system(d, case["coef"], case["nrhs"], rng) for d in _sides(case)]


# ---- the interface ---------------------------------------------------------------

def prepare(case, seed):
    made = _systems(case, seed)
    prec = PREC[case["prec"]]
    B = np.ascontiguousarray(np.concatenate([b for _, b, _ in made], axis=1))
    st = {"kind": case["kind"], "prec": prec, "nrhs": case["nrhs"], "n": B.shape[1],
          "method": case["method"]}
    if "count" in case:
        st["F"] = T.Batch([PA for PA, _, _ in made], precision=prec)
    else:
        PA = st["A"] = made[0][0]
        st["F"] = T.factor_symbolic(PA)
        if case["panel"]:  # the schedule shape this program has settled on
            st["F"].autotune(PA, prec, candidates=((case["panel"], case["tile"]),), reps=0)
        elif case["kind"] == "solve" and st["F"].numeric(PA, prec) != 0:
            raise RuntimeError("factorization failed")
    if case["kind"] in ("host", "batch_refined"):
        st["B"] = np.asfortranarray(B.T)
    else:
        st["B"] = torch.from_numpy(B).cuda()
        st["X"] = torch.empty_like(st["B"])
    if case["kind"] not in ("host", "solve"):
        st["vals"] = torch.from_numpy(np.concatenate([PA.arrays()[3] for PA, _, _ in made])).cuda()
    torch.cuda.synchronize()
    return st


def run(st):
    F, kind = st["F"], st["kind"]
    if kind == "host":
        if F.numeric(st["A"]) != 0:
            raise RuntimeError("factorization failed")
        return F.solve(st["B"])
    if kind != "solve" and F.numeric_device(st["vals"].data_ptr(), st["prec"]) != 0:
        raise RuntimeError("factorization failed")
    if kind == "batch_refined":
        x, info = F.solve_refined(st["B"], method=st["method"])
        return {"x": x, "converged": info.converged}
    X, B = st["X"], st["B"]
    if kind == "refined":
        info = F.solve_refined_device(st["A"], X.data_ptr(), B.data_ptr(), st["n"], st["nrhs"],
                                      method=st["method"], factored=True)
        return {"x": X, "converged": info.converged}
    if kind == "batch":
        F.solve_device(X.data_ptr(), B.data_ptr(), st["nrhs"])
    else:
        F.solve_device(X.data_ptr(), B.data_ptr(), st["n"], st["nrhs"])
    return X


def exact(case, seed):
    x = np.ascontiguousarray(np.concatenate([x for _, _, x in _systems(case, seed)], axis=1))
    if case["kind"] in ("host", "batch_refined"):
        x = np.ascontiguousarray(x.T)
    else:
        x = torch.from_numpy(x)
    if case["kind"].endswith("refined"):
        return {"x": x, "converged": None}
    return x


def work(case):
    """Values read, the factor written by the factorization and read by the
    solve, right-hand sides read and solutions written; the reference's count
    of factorization flops, and two per factor entry, sweep and right-hand side."""
    c = np.sum([_counts(d) for d in _sides(case)], axis=0)
    elem = 8 if case["prec"] == "fp64" else 4
    nbytes = elem * c[2] + 16 * c[0] * case["nrhs"]
    flops = 4.0 * c[2] * case["nrhs"]
    if case["kind"] != "solve":
        nbytes += 8 * c[1] + elem * c[2]
        flops += c[3]
    return {"bytes": int(nbytes), "flops": float(flops)}
