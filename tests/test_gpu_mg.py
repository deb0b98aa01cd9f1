"""The multigrid-preconditioned CG (csrc/mg.hip) of the coarse and the fine-scale
system at the sizes where its layout changes: one workgroup for everything
(12..30 cells per side in 2D), the first sizes on tiles, odd sizes
whose first coarse interval is one fine cell, edges of tiles; the Jacobi CG that
takes over when the enqueued iterations are used up, which solves coarse systems
of up to 11 cells per side by itself, and the sizes that keep it in the
allocation-free entry point.  Coarse systems against the oracle's direct
solve, fine systems against the oracle's direct solve of the coarse system that
has the fine cells' matrices (1e-10, the bar of the other solves)."""
import sys

import numpy as np
import pytest

import msfem
import msfem_cases as C
import oracle as O
import test_gpu_fine as F

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
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


def coarse_system(ctx, dim, nc, bc):
    case = C.lognormal_cells(dim=dim, nc=nc, nf=16 if dim == 2 else 4, seed=7)
    out = C.gpu_build(ctx, case)
    return ctx.coarse_assemble(dim, nc, out["Ae"], out["Fe"], bc)


@pytest.mark.parametrize("bc", [msfem.BC_ZERO_DIRICHLET, msfem.BC_REFERENCE])
@pytest.mark.parametrize("dim,nc", [(2, 2), (2, 3), (2, 5), (2, 11), (2, 12), (2, 30), (2, 31), (2, 32), (2, 33), (2, 47), (2, 65),
                                    (2, 100), (3, 2), (3, 3), (3, 6), (3, 7), (3, 9), (3, 11), (3, 12), (3, 13)])
def test_coarse_sizes(ctx, dim, nc, bc):
    say(f"multigrid CG dim={dim} nc={nc} bc={bc}")
    sysm = coarse_system(ctx, dim, nc, bc)
    u, it = ctx.coarse_solve(dim, nc, *sysm, rel_tol=1e-13)
    say(f"  {it} iterations")
    assert rel(u, O.coarse_solve(dim, nc, *sysm)) < TOL
    if nc > 11:  # the multigrid's; up to 11 cells per side the Jacobi CG runs
        assert it <= 20


@pytest.mark.parametrize("n", [7, 31, 33, 50])
def test_fine_sizes(ctx, n):
    say(f"fine solve n={n}")
    unit = np.array([[[0.0, 1.0], [0.0, 1.0]]])
    coef = msfem.coef_reference(2, np.array([n], np.int32), unit)
    u, it = ctx.fine_solve(n, msfem.COEF_TENSOR_QP, coef, msfem.RHS_CONST, 2.0, msfem.BC_REFERENCE, rel_tol=1e-13)
    ref = F.oracle_fine(n, msfem.COEF_TENSOR_QP, coef, msfem.RHS_CONST, 2.0, msfem.BC_REFERENCE)
    say(f"  {it} iterations")
    assert it <= 60 and rel(u, ref) < TOL


def test_beyond_the_enqueued_iterations(ctx):
    """A tolerance that FP64 does not reach: the Jacobi CG goes on to the cap, which is reported."""
    say("multigrid CG, then the Jacobi CG to the cap")
    sysm = coarse_system(ctx, 2, 40, 0)
    with pytest.raises(msfem.MsfemError) as e:
        ctx.coarse_solve(2, 40, *sysm, rel_tol=1e-30, max_iter=60)
    assert e.value.code == msfem.ERR_NOCONV and "60" in str(e.value)
    u, it = ctx.coarse_solve(2, 40, *sysm, rel_tol=1e-13)
    assert rel(u, O.coarse_solve(2, 40, *sysm)) < TOL


def test_noalloc_keeps_sizes_beyond_the_multigrid_scratch(ctx):
    """450 cells per side: the multigrid's scratch exceeds the fixed array, the Jacobi CG's does not."""
    say("allocation-free coarse solve, 450 cells per side, 3 iterations")
    nc, nn = 450, 451 ** 2
    Kc = np.zeros((nn, 9))
    Kc[:, 4], Kc[:, [0, 1, 2, 3, 5, 6, 7, 8]] = 8.0 / 3, -1.0 / 3
    cm = np.zeros((451, 451), np.uint8)
    cm[[0, -1]], cm[:, [0, -1]] = 1, 1
    d = dict(K=ctx.to_device(Kc), F=ctx.to_device(np.ones(nn)), m=ctx.to_device(cm.reshape(-1)),
             v=ctx.to_device(np.zeros(nn)), u=ctx.alloc(nn, np.float64), it=ctx.alloc(1, np.int32))
    msfem._check(msfem.lib().msfem_coarse_solve_device_noalloc(ctx.h, 2, nc, d["K"].ptr, d["F"].ptr, d["m"].ptr,
                                                               d["v"].ptr, 1e-12, 3, d["u"].ptr, d["it"].ptr, ctx.stream),
                 ctx.h)
    ctx.synchronize()
    u = d["u"].numpy().reshape(451, 451)
    assert int(d["it"].numpy()[0]) == 3 and np.isfinite(u).all() and u[225, 225] > 0 and not u[0].any()
    for a in d.values():
        a.free()
