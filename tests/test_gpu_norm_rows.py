"""The norm's row kernels around their edges: widths at the chunk rounds of a
wave that holds a row (64 16-byte chunks, up to 4 rounds) and rows on both
sides of one per CU (256), forward and backward against the fp64 oracle and
the residual form against the plain one bit for bit. Bars: fp32 1e-5 (of
max|ref| for the gradients, which are differences), bf16 outputs 1 ulp, fp64
1e-12 with the fp32 row mean the kernels keep."""

import pytest
import torch

import fastalgebraictransformer_amd as F
import oracle as O
from _util import assert_bf16_within_ulp, assert_rel

pytestmark = pytest.mark.gpu

WIDTHS = {torch.bfloat16: [8, 504, 512, 520, 1024, 1032, 1536, 2040, 2048, 2056],
          torch.float32: [4, 252, 256, 260, 512, 768, 772, 1020, 1024, 1028],
          torch.float64: [2, 128, 130, 384, 512, 514]}


@pytest.mark.parametrize("dtype", list(WIDTHS))
@pytest.mark.parametrize("rows", [1, 128, 129, 256, 257, 263, 1030])
def test_norm_rows(gpu, dtype, rows):
    for cols in WIDTHS[dtype]:
        g = torch.Generator().manual_seed(rows * 7919 + cols)
        x0 = torch.randn(rows, cols, generator=g).to(dtype)
        r0 = torch.randn(rows, cols, generator=g).to(dtype)
        dy = torch.randn(rows, cols, generator=g).to(dtype)
        dh = torch.zeros(rows, cols, dtype=dtype)
        w0 = (torch.rand(cols, generator=g) + 0.5).to(torch.float64 if dtype == torch.float64 else torch.float32)
        name = f"{dtype} {rows}x{cols}"
        hx, hr, hw = (t.cuda().requires_grad_(True) for t in (x0, r0, w0))
        h, y2 = F.add_mean_error_norm(hx, hr, hw)
        torch.autograd.backward([h, y2], [dh.cuda(), dy.cuda()])
        x, w = h.detach().clone().requires_grad_(True), w0.cuda().requires_grad_(True)
        y = F.mean_error_norm(x, w)
        y.backward(dy.cuda())
        assert torch.equal(y, y2) and torch.equal(w.grad, hw.grad), name
        # dx + 0 (the fused backward adds the stream's gradient; -0 + 0 = +0 compares equal)
        assert torch.equal(x.grad, hx.grad), name
        xd, wd = x.detach().cpu().double(), w0.double()
        y_ref, mu = O.mean_error_norm_fwd(xd, wd)
        dx_ref, dw_ref = O.mean_error_norm_bwd(dy.double(), xd, wd, mu.float().double())
        if dtype == torch.bfloat16:
            assert_bf16_within_ulp(y, y_ref, what=name)
            assert_bf16_within_ulp(x.grad, dx_ref, abs_floor=1e-3 * float(dx_ref.abs().max()), what=name)
            assert_rel(w.grad, dw_ref, 1e-5, name, floor_frac=1e-5)
        else:
            tol = 1e-5 if dtype == torch.float32 else 1e-12
            assert_rel(y, y_ref, tol, name)
            assert_rel(x.grad, dx_ref, tol, name, floor_frac=tol)
            assert_rel(w.grad, dw_ref, tol, name, floor_frac=tol)
