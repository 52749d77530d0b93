"""The forward's two kernels (one wave per 32 queries over whole key tiles, and
the key-split one that small grids take) against the CPU oracle, at sizes on
both sides of the dispatch and at the edges of the 32-key halves, the 64-key
tiles and the 64- / 128-query blocks. Bars as in test_gpu_attention.py:
|got - ref| <= 2e-2 + 1/2 ulp(ref), relative L2 <= 5e-3; L within 1e-2."""

import math

import pytest
import torch

import fastalgebraictransformer_amd as F
import oracle as O
from fastalgebraictransformer_amd.forward import _attn_fwd_into
from test_gpu_attention import assert_lowp

pytestmark = pytest.mark.gpu
dev = "cuda"


def _case(B, H, T, D, dtype, kind, causal, seed=0):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(B, H, T, D, generator=g).to(dtype).to(dev) for _ in range(3))
    km = None
    if kind == "random":
        km = (torch.rand(B, T, generator=g) > 0.3).to(torch.uint8).to(dev)
    elif kind == "halves":  # whole 32-key halves of a tile dropped, and a whole tile
        km = torch.ones(B, T, dtype=torch.uint8)
        km[:, 32:64] = 0
        km[:, 64:96] = 0
        km[:, 128:192] = 0
        km = km.to(dev)
    slopes, scale = F.compute_alibi_slopes(H), 1 / math.sqrt(D)
    o, L = torch.empty_like(q), torch.empty(B, H, T, device=dev)
    _attn_fwd_into(q, k, v, o, L, slopes.to(dev), scale, causal, O.EPS, km,
                   extended=km is not None or not causal)
    ro, rL = O.attention_fwd(q.cpu(), k.cpu(), v.cpu(), slopes, scale, dtype=torch.float32,
                             key_mask=None if km is None else km.cpu(), causal=causal)
    name = f"{B}x{H}x{T}x{D} {dtype} {kind} causal={causal}"
    assert_lowp(o, ro, dtype, name)
    assert float(((L.cpu() - rL).abs() - 1e-2 * rL.abs()).max()) <= 1e-6, name


@pytest.mark.parametrize("D", [24, 32, 64, 96, 128])
@pytest.mark.parametrize("T", [1, 32, 33, 64, 65, 95, 129, 257])
def test_small_grids(gpu, D, T):
    _case(2, 3, T, D, torch.bfloat16, None, True)
    _case(1, 8, T, D, torch.float16, "random", True)
    _case(1, 2, T, D, torch.bfloat16, "random", False)
    _case(1, 2, T, D, torch.bfloat16, None, False)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("causal", [True, False])
def test_dropped_halves(gpu, D, causal):
    _case(1, 4, 300, D, torch.bfloat16, "halves", causal)


# blocks of 128 queries just below and above the line between the two kernels
# (256 CUs; D = 128: 256 blocks up to T = 512, D <= 64: 768; non-causal 256 and 384)
@pytest.mark.parametrize("D,H,T,causal", [
    (128, 128, 200, True), (128, 129, 200, True), (128, 128, 100, True), (128, 129, 100, True),
    (128, 128, 200, False), (128, 129, 200, False),
    (64, 384, 130, True), (64, 385, 130, True), (64, 192, 130, False), (64, 193, 130, False),
    (32, 384, 130, True), (32, 385, 130, True),
])
def test_both_sides_of_the_dispatch(gpu, D, H, T, causal):
    _case(1, H, T, D, torch.bfloat16, None, causal)
