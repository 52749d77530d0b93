"""The backward's dK/dV and dQ kernels of small and full grids against the CPU
oracle: sequence lengths at the edges of 16- and 32-key groups, 64-row tiles and
the 256- and 512-query dQ blocks, head counts that are and are not multiples of
8 (block order, head groups), and grids on both sides of the dispatch. Bars as
in test_gpu_attention.py: |got - ref| <= 2e-2 + 1/2 ulp(ref), relative L2 <=
5e-3 on dq, dk, dv."""

import math

import pytest
import torch

import fastalgebraictransformer_amd as F
import oracle as O
from fastalgebraictransformer_amd import _lib
from test_gpu_attention import assert_lowp

pytestmark = pytest.mark.gpu
dev = "cuda"


def _case(B, H, T, D, dtype, masked=False, causal=True):
    g = torch.Generator().manual_seed(B * H * T + D)
    q, k, v, do = (torch.randn(B, H, T, D, generator=g).to(dtype) for _ in range(4))
    km = (torch.rand(B, T, generator=g) > 0.3).to(torch.uint8) if masked else None
    slopes, scale = F.compute_alibi_slopes(H), 1 / math.sqrt(D)
    ins = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    if masked or not causal:
        o = F.rational_attention_masked(*ins, slopes.to(dev), scale, None if km is None else km.to(dev), causal)
    else:
        o = F.rational_attention(*ins, slopes.to(dev), scale)
    grads = torch.autograd.grad(o, ins, do.to(dev))
    _, L = O.attention_fwd(q, k, v, slopes, scale, dtype=torch.float32, key_mask=km, causal=causal)
    ref = O.attention_bwd(q, k, v, o.detach().cpu(), L, do, slopes, scale, dtype=torch.float32, key_mask=km,
                          causal=causal)
    for n, got, want in zip(("dq", "dk", "dv"), grads, ref):
        assert_lowp(got, want, dtype, f"{n} {B}x{H}x{T}x{D} {dtype} masked={masked} causal={causal}")


@pytest.mark.parametrize("D", [24, 32, 64, 96, 128])
@pytest.mark.parametrize("T", [1, 16, 17, 33, 64, 65, 129, 255, 257, 513])
def test_edges(gpu, D, T):
    _case(1, 12, T, D, torch.bfloat16)
    _case(1, 5, T, D, torch.float16, masked=True)
    _case(1, 6, T, D, torch.bfloat16, causal=False)


# blocks of 128 keys on both sides of the 16- / 32-key line (256 CUs: D = 32 512
# blocks, D = 64 383, D = 128 256) and blocks of 512 queries on both sides of the
# 32- / 64-query line (D <= 64 384, D = 128 255 or 256)
@pytest.mark.parametrize("D,H,T,causal", [
    (32, 512, 100, True), (32, 513, 100, True), (64, 383, 128, True), (64, 384, 128, True),
    (64, 385, 70, True), (128, 255, 128, True), (128, 256, 128, True), (128, 257, 128, True),
    (128, 128, 520, True), (64, 384, 40, False), (64, 385, 40, False), (128, 256, 65, False),
])
def test_both_sides_of_the_dispatch(gpu, D, H, T, causal):
    _case(1, H, T, D, torch.bfloat16, causal=causal)


# (heads, heads that the capped workspace holds, heads of a group then: capped
# groups of 8 or more are rounded down to a multiple of 8)
@pytest.mark.parametrize("H,fit,group", [(1, 1, 1), (4, 1, 1), (12, 1, 1), (12, 10, 8), (17, 10, 8), (17, 16, 16)])
def test_head_groups_of_any_head_count(gpu, H, fit, group, monkeypatch):
    """One group of all heads (they fit) against capped groups: the same bits,
    and a workspace that shrinks to the group's."""
    T, D = 300, 64
    head = 40 * 8192  # dS^T of a head at T = 300: 5 key tiles of 8 query tiles, 8 KB each
    lib = _lib.load()
    g = torch.Generator().manual_seed(H)
    q, k, v, do = (torch.randn(1, H, T, D, generator=g).to(torch.bfloat16).to(dev) for _ in range(4))
    slopes = F.compute_alibi_slopes(H).to(dev)
    o, L = F.rational_attention_forward(q, k, v, slopes, 0.125)
    got, ws = [], []
    for cap in (None, fit * head):
        if cap:
            monkeypatch.setenv("KAT_ATTN_DS_CAP_BYTES", str(cap))
        ws.append(lib.kat_attn_bwd_workspace_size(1, H, T, D, 1))
        got.append(F.rational_attention_backward(q, k, v, o, L, do, slopes, 0.125))
    assert ws[0] - ws[1] == (H - group) * head
    for a, b in zip(*got):
        assert torch.equal(a, b)
