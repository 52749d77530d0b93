"""The kernels of full grids, which training runs: the one-group forward, dK/dV
with 32 keys per wave pair and dQ with 64 queries per wave (bf16 / fp16), and
the fp32 kernels with one wave group. B * H = 200 heads of T = 650 are past
every line of the dispatch on 256 CUs (blocks per call, needed: forward 1200,
> 777 at D <= 64 and > 325 at D = 128, non-causal > 384; dK/dV 1200, > 512; dQ
400, > 384), with six blocks of 128 rows, two of 512 queries, eleven 64-row
tiles and a remainder of 10 rows per head. Sampled heads are compared with the
CPU oracle. Bars as in test_gpu_attention.py and test_gpu_attention_fp32.py."""

import math

import pytest
import torch

import fastalgebraictransformer_amd as F
import oracle as O
from fastalgebraictransformer_amd import _lib
from test_gpu_attention import _rel_max, assert_lowp

pytestmark = pytest.mark.gpu
dev = "cuda"
B, H, T = 5, 40, 650
# Sampled (batch, head). fp16 keeps a key's weight f = (1 + s / (1 + |s|))^4 to
# 2^-10 of itself while f >= 2^-15, i.e. 1 + |s| <= 13. Past a gap of n dropped
# keys the largest s is slope * n below the scores' few units, so batches 0
# and 4, whose masks leave gaps of 160 and 150, are sampled at heads with
# slope * gap <= 4 (heads 24 and 20: 0.013 and 0.026).
HEADS = ((0, 24), (1, 0), (3, 39), (4, 20))


def _mask(n):
    km = (torch.rand(n, T, generator=torch.Generator().manual_seed(n)) > 0.3).to(torch.uint8)
    km[0, 64:224] = 0   # whole key tiles and a 32-key half dropped
    km[-1, 500:] = 0    # right padding
    return km


def _pass(ins, do, slopes, scale, mode, km):
    ins = [t.detach().requires_grad_(True) for t in ins]
    if mode == "causal":
        o = F.rational_attention(*ins, slopes, scale)
    else:
        o = F.rational_attention_masked(*ins, slopes, scale, km if "masked" in mode else None, "noncausal" not in mode)
    return (o.detach(),) + torch.autograd.grad(o, ins, do)


@pytest.mark.parametrize("mode", ["causal", "masked", "noncausal", "noncausal masked"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [24, 32, 64, 96, 128])
def test_sampled_heads_against_the_oracle(gpu, D, dtype, mode):
    g = torch.Generator(device=dev).manual_seed(D)
    q, k, v, do = (torch.randn(B, H, T, D, generator=g, device=dev).to(dtype) for _ in range(4))
    slopes, scale, km = F.compute_alibi_slopes(H), 1 / math.sqrt(D), _mask(B)
    got = _pass((q, k, v), do, slopes.to(dev), scale, mode, km.to(dev))
    assert all(bool(torch.isfinite(t).all()) for t in got)
    causal = "noncausal" not in mode
    for b, h in HEADS:
        one = [t[b:b + 1, h:h + 1].cpu() for t in (q, k, v, do) + got]
        kw = dict(dtype=torch.float32, key_mask=km[b:b + 1] if "masked" in mode else None, causal=causal)
        ro, rL = O.attention_fwd(*one[:3], slopes[h:h + 1], scale, **kw)
        ref = O.attention_bwd(*one[:3], one[4], rL, one[3], slopes[h:h + 1], scale, **kw)
        for n, a, r in zip(("o", "dq", "dk", "dv"), one[4:], (ro,) + tuple(ref)):
            assert_lowp(a, r, dtype, f"{n} ({b},{h}) D={D} {dtype} {mode}")


def _wide(t):
    """Two heads repeated to B * H of them: all run in one full grid."""
    return t.repeat(1, B * H // 2, 1, 1)


def _same_heads(t):
    """The first two heads, after a look that every repetition has their bits."""
    r = t.view(B * H // 2, 2, *t.shape[2:])
    assert torch.equal(r, r[:1].expand_as(r))
    return t[:, :2].cpu()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("what", ["keys by 32", "keys by 16", "query tiles"])
def test_magnitudes_that_differ_by_group(gpu, D, dtype, what):
    """Keys whose magnitude changes from one group of 32 (or 16) to the next, so
    that the 32-key exponents of the fp16 copy differ, and upstream gradients
    that change from one 64-query tile to the next (as in
    test_gpu_attention.py, where the reasons of the bars stand)."""
    q, k, v, do = (torch.randn(1, 2, T, D, generator=torch.Generator().manual_seed(D + i)) for i in range(4))
    i = torch.arange(T)
    if what == "query tiles":
        do = do * torch.pow(2.0, -(12.0 if dtype == torch.float16 else 30.0) * ((i // 64) % 2)).view(1, 1, T, 1)
    else:
        width = int(what.split()[-1])
        k = k * torch.pow(2.0, (12.0 if dtype == torch.float16 else 20.0) * (1 - (i // width) % 3)).view(1, 1, T, 1)
    q, k, v, do = (t.to(dtype) for t in (q, k, v, do))
    slopes, scale = F.compute_alibi_slopes(2), 1 / math.sqrt(D)
    got = _pass([_wide(t).to(dev) for t in (q, k, v)], _wide(do).to(dev), slopes.repeat(B * H // 2).to(dev), scale,
                "causal", None)
    got = [_same_heads(t) for t in got]
    _, rL = O.attention_fwd(q, k, v, slopes, scale, dtype=torch.float32)
    ref = O.attention_bwd(q, k, v, got[0], rL, do, slopes, scale, dtype=torch.float32)
    for n, a, r in zip(("dq", "dk", "dv"), got[1:], ref):
        a, r = a.double(), r.double()
        assert bool(torch.isfinite(a).all()) and _rel_max(a, r) <= 2e-2, n
        assert float((a - r).norm() / r.norm()) <= 1e-2, n
        step = {"query tiles": 64 if n == "dq" else 0, "keys by 32": 32 if n == "dv" else 0,
                "keys by 16": 16 if n == "dv" else 0}[what]
        for j in range(0, T if step else 0, step or 1):
            assert _rel_max(a[:, :, j:j + step], r[:, :, j:j + step]) <= 2e-2, (n, j)


@pytest.mark.parametrize("D", [32, 64, 96, 128])
def test_exact_under_power_of_two_scales(gpu, D):
    """Inputs on a grid of 1/16 scaled by powers of two give outputs scaled by
    powers of two, bit for bit (as in test_gpu_attention.py)."""
    g = torch.Generator().manual_seed(D)
    base = [_wide(torch.round(torch.randn(1, 2, T, D, generator=g) * 16) / 16) for _ in range(4)]
    slopes, scale = F.compute_alibi_slopes(B * H).to(dev), 1 / math.sqrt(D)

    def run(fs):
        t = [(x * f).to(torch.bfloat16).to(dev) for x, f in zip(base, fs)]
        return _pass(t[:3], t[3], slopes, scale, "causal", None)
    unit, scaled = run((1.0,) * 4), run((2.0 ** 16, 2.0 ** -16, 2.0 ** 13, 2.0 ** -20))
    for n, u, s, f in zip(("o", "dq", "dk", "dv"), unit, scaled, (2.0 ** 13, 2.0 ** -23, 2.0 ** 9, 2.0 ** -20)):
        assert torch.equal(s.float(), u.float() * f), n


@pytest.mark.parametrize("mode", ["causal", "masked", "noncausal"])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_head_groups_on_both_sides_of_the_lines(gpu, D, mode, monkeypatch):
    """One group of 200 heads, and groups of 144 and 56 (which take other
    kernels): the same bits."""
    g = torch.Generator(device=dev).manual_seed(D)
    q, k, v, do = (torch.randn(B, H, T, D, generator=g, device=dev).to(torch.bfloat16) for _ in range(4))
    slopes, scale, km = F.compute_alibi_slopes(H).to(dev), 1 / math.sqrt(D), _mask(B).to(dev)
    lib, causal = _lib.load(), mode != "noncausal"
    # dS^T tiles of 8 KB per head at T = 650: two runs of 8 query tiles, causal 8 and
    # 11 key tiles long, else 11 both
    head = 8 * (8 + 11 if causal else 22) * 8192
    runs, ws = [], []
    for cap in (None, 150 * head):
        if cap:
            monkeypatch.setenv("KAT_ATTN_DS_CAP_BYTES", str(cap))
        ws.append(lib.kat_attn_bwd_masked_workspace_size(B, H, T, D, 1, int(causal)))
        runs.append(_pass((q, k, v), do, slopes, scale, mode, km))
    assert ws[0] - ws[1] == (B * H - 144) * head
    for n, a, b in zip(("o", "dq", "dk", "dv"), *runs):
        assert torch.equal(a, b), n


@pytest.mark.parametrize("mode", ["causal", "masked", "noncausal", "noncausal masked"])
@pytest.mark.parametrize("D", [20, 32, 64, 96, 128])
def test_fp32_one_group(gpu, D, mode):
    """2 x 40 heads: 880 blocks of 64 rows, past the fp32 kernels' lines (forward
    768, backward 256)."""
    g = torch.Generator(device=dev).manual_seed(D)
    q, k, v, do = (torch.randn(2, H, T, D, generator=g, device=dev) for _ in range(4))
    slopes, km = F.compute_alibi_slopes(H), _mask(2)
    scale = float(torch.tensor(1 / math.sqrt(D), dtype=torch.float32))
    got = _pass((q, k, v), do, slopes.to(dev), scale, mode, km.to(dev))
    assert all(bool(torch.isfinite(t).all()) for t in got)
    for b, h in ((0, 0), (0, 23), (1, 39)):
        one = [t[b:b + 1, h:h + 1].cpu().double() for t in (q, k, v, do) + got]
        kw = dict(key_mask=km[b:b + 1] if "masked" in mode else None, causal="noncausal" not in mode)
        ro, rL = O.attention_fwd(*one[:3], slopes[h:h + 1], scale, **kw)
        ref = O.attention_bwd(*one[:3], ro, rL, one[3], slopes[h:h + 1], scale, **kw)
        for n, a, r in zip(("o", "dq", "dk", "dv"), one[4:], (ro,) + tuple(ref)):
            assert _rel_max(a, r) <= 1e-5, f"{n} ({b},{h}) D={D} {mode}"
