"""Row kernels on both sides of the lines that choose their grids (256 CUs): rows
per block by how much of a row a thread holds, the norm backward's blocks per
CU by the row's bytes, and the forward's wave-per-row kernels. A row's result
does not depend on the grid: softmax rows are compared bit for bit with those of
small calls, and sampled rows and the weight gradient with the fp64 oracle.
Bars as in test_gpu_rowops.py and test_gpu_norm_rows.py."""

import pytest
import torch

import fastalgebraictransformer_amd as F
import oracle as O
from _util import assert_bf16_within_ulp, assert_rel

pytestmark = pytest.mark.gpu
dev = "cuda"


def _x(seed, *shape, dtype):
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=dev).to(dtype)


def _close(got, ref, dtype, name):
    floor = float(ref.abs().max())
    if dtype == torch.bfloat16:
        assert_bf16_within_ulp(got, ref, abs_floor=1e-3 * floor, what=name)
    else:
        assert_rel(got, ref, 1e-5, name, floor_frac=1e-5)


# chunk rounds held: 3 (backward 6), 5 -> 6 (12), 9 -> 16 (32); rows at 1, 2 and 6 per CU
@pytest.mark.parametrize("dtype,cols", [(torch.bfloat16, 4104), (torch.bfloat16, 10248), (torch.float32, 8200)])
@pytest.mark.parametrize("rows", [1, 256, 257, 512, 513, 1536, 1537])
def test_softmax_rows_do_not_depend_on_the_grid(gpu, rows, dtype, cols):
    x, dy = (2 * _x(rows, rows, cols, dtype=dtype)).requires_grad_(True), _x(rows + 1, rows, cols, dtype=dtype)
    p = F.rational_softmax(x)
    (dx,) = torch.autograd.grad(p, x, dy)
    for i in range(0, rows, 100):
        s = x.detach()[i:i + 100].clone().requires_grad_(True)
        q = F.rational_softmax(s)
        assert torch.equal(q, p[i:i + 100])
        assert torch.equal(torch.autograd.grad(q, s, dy[i:i + 100])[0], dx[i:i + 100])
    pick = sorted({0, rows // 3, rows - 1})
    xs = x.detach()[pick].cpu()
    _close(p.detach()[pick], O.rational_softmax_fwd(xs), dtype, "p")
    _close(dx[pick], O.rational_softmax_bwd(dy[pick].cpu(), xs, p.detach()[pick].cpu()), dtype, "dx")


# forward: full four-round rows at 28 and 64 rows per CU; rows per block at 2, 6 and
# 8 per CU. Backward: the lines at 6, 10 and 16 rows per CU for rows below 8 KB, below
# 12 KB and above
@pytest.mark.parametrize("rows,cols,dtype", [
    (7168, 2048, torch.bfloat16), (7169, 2048, torch.bfloat16), (16384, 1024, torch.float32),
    (16385, 1024, torch.float32), (1535, 2056, torch.bfloat16), (1536, 2056, torch.bfloat16),
    (2559, 4096, torch.bfloat16), (2560, 4096, torch.bfloat16), (4095, 6144, torch.bfloat16),
    (4096, 6144, torch.bfloat16), (512, 8192, torch.float32), (513, 8192, torch.float32),
    (1537, 4096, torch.float32), (2049, 1536, torch.float32),
])
def test_norm(gpu, rows, cols, dtype):
    x, r, dy = (_x(rows + i, rows, cols, dtype=dtype) for i in range(3))
    w = (_x(cols, cols, dtype=torch.float32) * 0.1 + 1).requires_grad_(True)
    hx, hr, hw = (t.detach().clone().requires_grad_(True) for t in (x, r, w))
    h, y2 = F.add_mean_error_norm(hx, hr, hw)
    gh = torch.autograd.grad((h, y2), (hx, hw), (torch.zeros_like(h), dy))
    hh = h.detach().requires_grad_(True)
    y = F.mean_error_norm(hh, w)
    dx, dw = torch.autograd.grad(y, (hh, w), dy)
    # the residual form, to the plain one's bits (-0 + 0 = +0 compares equal)
    assert torch.equal(y, y2) and torch.equal(dw, gh[1]) and torch.equal(dx, gh[0])
    pick = torch.tensor(sorted({0, 1, rows // 2, rows - 2, rows - 1}))
    hd, wd, dyd = h.detach().cpu().double(), w.detach().cpu().double(), dy.cpu().double()
    y_ref, mu = O.mean_error_norm_fwd(hd, wd)
    dx_ref, dw_ref = O.mean_error_norm_bwd(dyd, hd, wd, mu.float().double())
    _close(y.detach()[pick.to(dev)], y_ref[pick], dtype, "y")
    _close(dx[pick.to(dev)], dx_ref[pick], dtype, "dx")
    assert_rel(dw, dw_ref, 1e-5, "dw", floor_frac=1e-5)
