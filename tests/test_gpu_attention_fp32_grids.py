"""fp32 attention with one, two and four wave groups per block (small grids
split a block's tiles over its waves) against the fp64 oracle: lengths at the
edges of 16-row groups, 32- and 64-row tiles and the 16- / 32- / 64-row
blocks, and grids on both sides of each line of the dispatch. Bar of
test_gpu_attention_fp32.py: <= 1e-5 of max|ref|."""

import math

import pytest
import torch

import fastalgebraictransformer_amd as F
import oracle as O
from test_gpu_attention import _rel_max

pytestmark = pytest.mark.gpu
dev = "cuda"


def _case(B, H, T, D, mode):
    g = torch.Generator().manual_seed(H * T + D)
    q, k, v, do = (torch.randn(B, H, T, D, generator=g) for _ in range(4))
    km = None
    if mode == "masked":
        km = (torch.rand(B, T, generator=g) > 0.3).to(torch.uint8)
        km[:, 0] = 1
        if T > 64:
            km[:, 16:64] = 0  # whole 16-key groups and a 32-key tile dropped
    causal = mode != "noncausal"
    slopes, scale = F.compute_alibi_slopes(H), 1 / math.sqrt(D)
    ins = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    o = F.rational_attention_masked(*ins, slopes.to(dev), scale, None if km is None else km.to(dev), causal)
    grads = torch.autograd.grad(o, ins, do.to(dev))
    scale32 = float(torch.tensor(scale, dtype=torch.float32))
    ro, rL = O.attention_fwd(q.double(), k.double(), v.double(), slopes, scale32, key_mask=km, causal=causal)
    ref = O.attention_bwd(q.double(), k.double(), v.double(), ro, rL, do.double(), slopes, scale32, key_mask=km,
                          causal=causal)
    name = f"{B}x{H}x{T}x{D} {mode}"
    assert _rel_max(o, ro) <= 1e-5, name
    # T = 1: o = v L / (L + eps), so dS = p g (dP - Delta) is what cancellation
    # leaves of dP (~eps dP); its error is fp32's rounding of the two terms,
    # p g |dP| <= 4 ||do|| ||v|| each, not of the result
    floor = 0.0
    if T == 1:
        floor = 1e-6 * 4 * scale * float(do.norm(dim=-1).max() * v.norm(dim=-1).max() * max(q.abs().max(), k.abs().max()))
    for n, got, want in zip(("dq", "dk", "dv"), grads, ref):
        err = float((got.cpu().double() - want).abs().max())
        assert err <= 1e-5 * float(want.abs().max()) + (0.0 if n == "dv" else floor), f"{n} {name}: {err:.3e}"


@pytest.mark.parametrize("mode", ["causal", "masked", "noncausal"])
@pytest.mark.parametrize("D", [20, 32, 64, 96, 128])
@pytest.mark.parametrize("T", [1, 16, 17, 33, 64, 65, 127, 300])
def test_edges(gpu, D, T, mode):
    _case(1, 3, T, D, mode)


# nb = H ceil(T / 64) blocks of 64 rows; lines at 128, 160, 192, 256, 384, 512 and 768 blocks
# and T = 64, 128, 256 and 512
@pytest.mark.parametrize("D,H,T,mode", [
    (64, 128, 60, "causal"), (64, 129, 60, "causal"), (64, 160, 60, "causal"), (64, 161, 60, "causal"),
    (64, 256, 60, "causal"), (64, 257, 60, "causal"), (64, 51, 270, "causal"), (64, 52, 270, "causal"),
    (64, 256, 130, "causal"), (64, 257, 130, "causal"), (64, 192, 60, "noncausal"), (64, 193, 60, "noncausal"),
    (128, 256, 40, "causal"), (128, 257, 40, "causal"), (32, 256, 40, "causal"), (32, 257, 40, "masked"),
    (128, 128, 64, "causal"), (128, 129, 64, "causal"), (128, 128, 65, "causal"), (32, 129, 64, "masked"),
    (64, 170, 130, "causal"), (64, 171, 130, "causal"), (64, 76, 600, "causal"), (64, 77, 600, "masked"),
    (64, 32, 270, "causal"), (64, 33, 270, "causal"), (32, 170, 130, "noncausal"), (32, 171, 130, "noncausal"),
    (64, 38, 270, "noncausal"), (64, 39, 270, "noncausal"), (64, 76, 270, "noncausal"),
    (64, 77, 270, "noncausal"), (128, 76, 270, "noncausal"), (128, 77, 270, "noncausal"),
])
def test_both_sides_of_the_dispatch(gpu, D, H, T, mode):
    _case(1, H, T, D, mode)
