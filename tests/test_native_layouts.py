"""The layout rules of the native autograd functions (csrc/torch_ops.cpp)
against those of the Python ones, over strides, orders and sizes (no GPU
needed): rows2d, and the MFMA envelope that decides between a native call and
the Python function with its fallback warning."""

import itertools
import random

import torch

from fastalgebraictransformer_amd import _lib
from fastalgebraictransformer_amd.forward import _tiled_reason


def _layouts():
    base = torch.randn(6, 5, 4, 8)
    yield base
    for perm in itertools.permutations(range(4)):
        yield base.permute(perm)
    yield base[:, :, :, :5]
    yield base[:, :, 1:3]
    yield base[:, 1]
    yield base[:, 2:3]
    yield base[1:2, :, 2:3, 3:7]
    yield base[::2]
    yield base[:, :, ::2]
    yield base[..., ::2]
    yield base[..., :1]
    yield base[..., 0]
    yield base[0, 0, 0]
    yield base[0, 0, :, 0]
    yield torch.randn(7)
    yield torch.tensor(3.0)
    yield torch.randn(3, 1).expand(3, 8)
    yield torch.randn(1, 8).expand(5, 8)
    yield torch.randn(1, 1, 8).expand(4, 5, 8)
    yield torch.randn(1, 1).expand(4, 5)
    yield torch.randn(64).as_strided((4, 8), (4, 1))      # overlapping rows
    yield torch.randn(64).as_strided((3, 2, 8), (16, 8, 1))
    yield torch.randn(90).as_strided((3, 2, 8), (30, 10, 1))
    yield torch.randn(90).as_strided((3, 2, 8), (20, 10, 1))
    yield torch.randn(2, 3, 16).chunk(2, dim=-1)[1]


def test_rows2d_agrees_with_the_python_rule():
    ops = _lib.ops()
    for t in _layouts():
        p2, ld = _lib.rows2d(t)
        in_place = p2.data_ptr() == t.data_ptr()
        got = ops.rows2d(t)
        what = (tuple(t.shape), t.stride(), got, (in_place, tuple(p2.shape), ld))
        assert got[1:3] == tuple(p2.shape), what
        assert got[0] == in_place, what
        if got[1] > 1:
            assert got[3] == ld, what


def test_envelope_agrees_with_the_python_rule():
    ops = _lib.ops()
    rng = random.Random(5)
    for _ in range(3000):
        dt = rng.choice([torch.bfloat16, torch.float16, torch.float32])
        es = 4 if dt == torch.float32 else 2
        B, H, T = rng.randint(1, 3), rng.randint(1, 3), rng.randint(1, 9)
        D = rng.choice([3, 4, 8, 12, 20, 32, 64, 72, 128, 256, 260, 264])
        pad = rng.choice([0, 0, 4, 8, 3, 16])
        row = max(1, D + pad * rng.choice([0, 1, -1]))
        st = rng.choice([row, row, row + 1, 1 << 26])
        sh = rng.choice([st * T, D, st * T + rng.choice([0, 2, 8])])
        sb = rng.choice([sh * H, sh * H + rng.choice([0, 4, 16])])
        off = rng.choice([0, 0, 0, 1, 8])
        strides = (sb, sh, st, 1)
        view = _unchecked_view(dt, off, (B, H, T, D), strides)
        if view is None:
            continue
        got = ops.attn_layout_ok([view])
        want = _tiled_reason([(view.stride()[:3], view.data_ptr())], D, T, es) is None
        assert got == want, (dt, (B, H, T, D), strides, off, got, want)


def _unchecked_view(dt, off, size, strides):
    """A view of the given geometry over real memory, or None if it would need
    more than a few MB."""
    n = off + sum((s - 1) * st for s, st in zip(size, strides)) + 1
    if n > 1 << 22:
        return None
    return torch.zeros(n, dtype=dt).as_strided(size, strides, off)


def test_envelope_limits_on_row_stride():
    """The 31-bit offset limit, from strides alone (a tensor of one row, whose
    row stride is never stepped)."""
    ops = _lib.ops()
    for dt, es in ((torch.bfloat16, 2), (torch.float32, 4)):
        lim = 0x7FFFFFFF // (129 * es)
        for st in (lim - lim % 8 - 8, lim - lim % 8, lim - lim % 8 + 8, 1 << 28):
            t = torch.zeros(64, dtype=dt).as_strided((1, 1, 1, 64), (st, st, st, 1))
            want = _tiled_reason([(t.stride()[:3], t.data_ptr())], 64, 1, es) is None
            assert ops.attn_layout_ok([t]) == want
