"""The direct local solves (csrc/direct.hip) against the oracle's exact solves and
against the iterative solve of the same cells: resolutions at the edges of the
leaf, block and front tiles, every 2D coefficient kind and general
quadrilaterals; the correction pass; which calls keep the iterative solve.  The
bar is the repository's 1e-10 relative on nodal values, A^K and F^K (the
factorization's own error is a few hundred FP64 roundings)."""
import sys

import numpy as np
import pytest

import msfem
import msfem_cases as C

pytestmark = pytest.mark.gpu
TOL = 1e-10


def say(msg):
    print(f"[gpu-case] {msg}", flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    c = msfem.Context(0)
    yield c
    c.close()


def rel(a, b):
    return np.abs(np.asarray(a) - np.asarray(b)).max() / max(np.abs(np.asarray(b)).max(), 1e-300)


def check(out, ref):
    assert (out["status"] == 0).all(), out["status"]
    for k in ("bases", "Ae", "Fe"):
        assert rel(out[k], ref[k]) < TOL, k


# 9, 16 | 17, 31, 32 | 33, 63 | 65, 100, 127, 128: first and last of a depth, odd and ragged cuts
@pytest.mark.parametrize("nf", [9, 10, 16, 17, 31, 32, 33, 63, 65, 100, 127, 128])
@pytest.mark.parametrize("kind", ["scalar", "tensor", "quad"])
def test_direct_matches_oracle(ctx, nf, kind):
    say(f"direct solve nf={nf} {kind}")
    which = np.array([0, 5, 40])
    if kind == "quad":
        case = C.quad_cells(nc=8, nf=nf, kind="reference", which=which)
    elif kind == "tensor":
        case = C.tensor_cells(nc=128, which=which, n_fine=[nf] * 3)
    else:
        case = C.lognormal_cells(nc=8, nf=nf, seed=3, which=which)
    out = C.gpu_build(ctx, case)
    assert (out["iters"] == 1).all()
    check(out, C.oracle_build(case, n_threads=8))


@pytest.mark.parametrize("prec", [msfem.PREC_FP64, msfem.PREC_FP32_REFINE])
def test_direct_matches_iterative(ctx, prec):
    """The same cells by the direct and by the iterative solve, 64^2 in a batch of 40, with
    partition of unity, and as a replayed graph."""
    say(f"direct against iterative, 64^2 and 32^2, prec={prec}")
    for case in (C.lognormal_cells(which=np.arange(40)), C.periodic_cells(which=np.arange(7))):
        it = C.gpu_build(ctx, case, precision=prec, coarse_space=0)
        check(C.gpu_build(ctx, case, precision=prec), it)
        check(C.gpu_build(ctx, case, precision=prec, partition_of_unity=1), it)
        for _ in range(3):
            check(C.gpu_build(ctx, case, precision=prec, graph=1), it)


def test_correction_pass(ctx):
    """A tolerance below FP64 rounding: every cell takes the correction, which leaves the
    residual no larger and the values exact; without convergence the status says so."""
    say("direct correction pass")
    case = C.tensor_cells(nc=128, which=np.array([3, 77, 901, 4000]), n_fine=[16, 31, 100, 128])
    ref = C.oracle_build(case, n_threads=8)
    args = (2, case["n_fine"], case["box"], case["coef_kind"], case["coef"], case["rhs_kind"], case["rhs_value"])
    one = ctx.batch_build(*args)
    two = ctx.batch_build(*args, opts=msfem.default_opts(rel_tol=1e-18), raise_noconv=False)
    assert (one["iters"] == 1).all() and (two["iters"] == 2).all() and (two["status"] == 1).all()
    assert (two["resid"] <= 1.5 * one["resid"]).all()
    for k in ("bases", "Ae", "Fe"):
        assert rel(two[k], ref[k]) < TOL


def test_what_keeps_the_iterative_solve(ctx):
    """An x0, an explicit launch shape, another coarse_space: iterations as before."""
    say("calls that keep the iterative solve")
    case = C.tensor_cells(nc=128, which=np.array([3, 77]), n_fine=[32, 32])
    ref = C.gpu_build(ctx, case)
    assert (ref["iters"] == 1).all()
    for kw in (dict(coarse_space=0), dict(variant=1)):
        out = C.gpu_build(ctx, case, **kw)
        assert (out["iters"] > 10).all()
        check(out, ref)
    rng = np.random.default_rng(0)
    x0 = ref["bases"] + 1e-6 * rng.standard_normal(ref["bases"].shape)
    out = ctx.batch_build(2, case["n_fine"], case["box"], case["coef_kind"], case["coef"], case["rhs_kind"],
                          case["rhs_value"], x0=x0)
    assert (out["iters"] > 1).all()
    check(out, ref)
