"""The training step's kernels at the sizes where their forms change: the 3x3
column matrix by rows of 8 columns (one image row, one group per row, the last
workgroup partly full) and its adjoint by rows of 4 pixels, the bias gradient's
wide and scalar loads."""
import numpy as np
import pytest

import msfem
import surrogate as S
import surrogate_ref as R
from test_gpu_surrogate import bf16_bits, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = msfem.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("C,B,H,W", [(1, 1, 1, 8), (3, 2, 5, 8), (2, 3, 2, 24), (2, 5, 16, 32), (1, 2, 64, 64)])
def test_im2col_by_rows(ctx, C, B, H, W):
    say(f"im2col 3x3 C={C} B={B} H={H} W={W}")
    x = np.random.default_rng(C + 10 * B + H + W).standard_normal((C, B, H, W)).astype(np.float32)
    col, _ = R.im2col(x.astype(np.float64), 3, 1)
    dx, dcol = ctx.to_device(x), ctx.alloc(col.size, np.uint16)
    assert S._nn().msfem_nn_im2col(C, B, H, W, 3, 3, 1, dx.ptr, dcol.ptr, ctx.stream) == 0
    assert np.array_equal(dcol.numpy().reshape(-1), bf16_bits(R.bf16(col)).reshape(-1))


@pytest.mark.parametrize("N", [1, 4, 1025, 16380, 16384, 16388, 49155, 65536])
def test_bias_grad_sizes(ctx, N):
    """FP32 sums: one rounding of the sum of magnitudes per addition in a row, at most 49 in a thread
    and 24 over the workgroup at these sizes."""
    say(f"bias gradient N={N}")
    d = np.random.default_rng(N).standard_normal((3, N)).astype(np.float32)
    dd, db = ctx.to_device(d), ctx.alloc(3, np.float32)
    assert S._nn().msfem_nn_bias_grad(3, N, dd.ptr, db.ptr, ctx.stream) == 0
    err = np.abs(db.numpy() - d.astype(np.float64).sum(1))
    assert (err <= 80 * 2.0 ** -24 * np.abs(d).astype(np.float64).sum(1)).all()


@pytest.mark.parametrize("C,B,H,W", [(1, 1, 1, 4), (3, 2, 5, 4), (2, 3, 2, 12), (2, 5, 16, 32), (1, 2, 64, 64)])
def test_col2im_by_rows(ctx, C, B, H, W):
    """Nine FP32 terms per pixel, added in the order of the taps: bitwise numpy's FP32 sum in that order."""
    say(f"col2im 3x3 C={C} B={B} H={H} W={W}")
    dcol = np.random.default_rng(C + 10 * B + H + W).standard_normal((C, 3, 3, B, H, W)).astype(np.float32)
    ref = np.zeros((C, B, H + 2, W + 2), np.float32)
    for ky in range(3):
        for kx in range(3):
            ref[:, :, ky:ky + H, kx:kx + W] += dcol[:, ky, kx]
    dc, dx = ctx.to_device(dcol), ctx.alloc(C * B * H * W, np.float32)
    assert S._nn().msfem_nn_col2im(C, B, H, W, 3, 3, 1, dc.ptr, dx.ptr, ctx.stream) == 0
    assert np.array_equal(dx.numpy().reshape(C, B, H, W), ref[:, :, 1:-1, 1:-1])
