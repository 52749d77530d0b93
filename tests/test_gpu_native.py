"""The native autograd functions (csrc/torch_ops.cpp) against the
torch.autograd.Function classes over the forms both accept: outputs and
gradients bit for bit, over dtypes, input layouts and gradient layouts; and
what surrounds an autograd function: saved-tensor hooks, checkpointing,
no-grad and inference mode, partial gradients, transforms, errors."""

import math
import warnings

import pytest
import torch

import fastalgebraictransformer_amd as F
from fastalgebraictransformer_amd import _lib

pytestmark = pytest.mark.gpu
DTYPES = [torch.bfloat16, torch.float16, torch.float32, torch.float64]


def _rand(seed, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def _layouts(seed, dtype):
    """Tensors of several layouts, made anew (a leaf each)."""
    yield "contiguous", _rand(seed, 6, 5, 24, dtype=dtype)
    yield "1d", _rand(seed, 40, dtype=dtype)
    yield "odd", _rand(seed, 7, 33, dtype=dtype)
    yield "row stride", _rand(seed, 9, 48, dtype=dtype)[:, :24]
    yield "offset", _rand(seed, 9, 49, dtype=dtype)[:, 1:25]
    yield "transposed", _rand(seed, 24, 10, dtype=dtype).t()
    yield "permuted", _rand(seed, 4, 6, 24, dtype=dtype).transpose(0, 1)
    yield "expanded", _rand(seed, 1, 24, dtype=dtype).expand(5, 24)
    yield "column step", _rand(seed, 5, 48, dtype=dtype)[:, ::2]


def _grads(y, seed):
    """Gradients for y in several layouts."""
    c = _rand(seed, *y.shape, dtype=y.dtype)
    yield c
    yield torch.ones((), dtype=y.dtype, device="cuda").expand(y.shape)
    if y.dim() >= 2:
        p = torch.empty(y.shape[:-2] + (y.shape[-1], y.shape[-2]), dtype=y.dtype, device="cuda")
        yield p.transpose(-1, -2).copy_(c)
    wide = torch.empty(y.shape[:-1] + (y.shape[-1] + 3,), dtype=y.dtype, device="cuda")[..., 1:1 + y.shape[-1]]
    yield wide.copy_(c)
    yield c.double() if y.dtype != torch.float64 else c


def _same(native, python, inputs, seed, what):
    a = native(*inputs)
    b = python(*inputs)
    a, b = (t if isinstance(t, tuple) else (t,) for t in (a, b))
    assert all(torch.equal(x, y) and x.dtype == y.dtype and x.shape == y.shape for x, y in zip(a, b)), what
    leaves = [t for t in inputs if t.requires_grad]
    for gs in zip(*(_grads(t, seed + i) for i, t in enumerate(a))):
        ga = torch.autograd.grad(a, leaves, gs, retain_graph=True)
        gb = torch.autograd.grad(b, leaves, gs, retain_graph=True)
        for x, y in zip(ga, gb):
            assert torch.equal(x, y) and x.dtype == y.dtype, (what, [g.stride() for g in gs])


@pytest.mark.parametrize("dtype", DTYPES)
def test_row_ops(gpu, dtype):
    for name, x in _layouts(3, dtype):
        x.requires_grad_(True)
        assert _lib.ops().softmax(x, 1e-6) is not None, name
        _same(F.rational_softmax, lambda t: F.RationalSoftmax.apply(t, 1e-6), [x], 5, name)
        v = _rand(4, *x.shape, dtype=dtype).requires_grad_(True)
        _same(F.rational_swiglu, F.RationalSwiGLU.apply, [x, v], 5, name)
        _same(F.rational_swiglu, F.RationalSwiGLU.apply, [v, x], 5, name)
        if x.shape[-1] % 2 == 0:
            _same(F.rational_swiglu_packed, F.PackedRationalSwiGLU.apply, [x], 5, name)
        for wd in {dtype, torch.float32 if dtype != torch.float64 else dtype}:
            w = (1 + 0.1 * _rand(6, x.shape[-1])).to(wd).requires_grad_(True)
            assert _lib.ops().norm(x, w, 1e-6) is not None
            _same(F.mean_error_norm, lambda a, b: F.MeanErrorNorm.apply(a, b, 1e-6), [x, w], 5, name)
            for rd in {dtype} | ({torch.bfloat16, torch.float16} if dtype == torch.float32 else set()):
                r = _rand(7, *x.shape, dtype=rd).requires_grad_(True)
                for od in (None, rd):
                    _same(lambda a, b, c: F.add_mean_error_norm(a, b, c, 1e-6, od),
                          lambda a, b, c: F.ResidualMeanErrorNorm.apply(a, b, c, 1e-6, od), [x, r, w], 5, name)


def _qkv(seed, B, H, T, D, dtype):
    yield "contiguous", [_rand(seed + i, B, H, T, D, dtype=dtype) for i in range(3)]
    yield "token major", [_rand(seed + i, B, T, H, D, dtype=dtype).transpose(1, 2) for i in range(3)]
    yield "packed parts", list(_rand(seed, B, T, 3, H, D, dtype=dtype).permute(2, 0, 3, 1, 4))
    yield "padded rows", [_rand(seed + i, B, H, T, D + 16, dtype=dtype)[..., :D] for i in range(3)]
    yield "misaligned", [_rand(seed + i, B, H, T, D + 3, dtype=dtype)[..., 3:] for i in range(3)]
    yield "column step", [_rand(seed + i, B, H, T, 2 * D, dtype=dtype)[..., ::2] for i in range(3)]


@pytest.mark.filterwarnings("ignore:rational attention in")
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("D", [64, 40, 20])
def test_attention(gpu, dtype, D):
    B, H, T = 2, 3, 70
    slopes, scale = F.compute_alibi_slopes(H).cuda(), 1 / math.sqrt(D)
    km = torch.rand(B, T, generator=torch.Generator().manual_seed(1)).cuda() > 0.3
    for name, qkv in _qkv(11, B, H, T, D, dtype):
        qkv = [t.detach().requires_grad_(True) for t in qkv]
        _same(lambda q, k, v: F.rational_attention(q, k, v, slopes, scale),
              lambda q, k, v: F.RationalAttentionFunction.apply(q, k, v, slopes, scale, True, 1e-6), qkv, 5, name)
        for mask in (None, km, km.float(), km.to(torch.int64).t().contiguous().t()):
            for causal in (True, False):
                _same(lambda q, k, v: F.rational_attention_masked(q, k, v, slopes, scale, mask, causal),
                      lambda q, k, v: F.MaskedRationalAttentionFunction.apply(q, k, v, slopes, scale, mask, causal,
                                                                              1e-6), qkv, 5, name)
    for name, p in (("packed", _rand(12, B, T, 3, H, D, dtype=dtype)),
                    ("batch minor", _rand(12, T, B, 3, H, D, dtype=dtype).transpose(0, 1)),
                    ("misaligned", _rand(12, B, T, 3, H, D + 1, dtype=dtype)[..., 1:])):
        p = p.detach().requires_grad_(True)
        for mask in (None, km):
            _same(lambda t: F.rational_attention_packed(t, slopes, scale, key_mask=mask),
                  lambda t: F.PackedRationalAttention.apply(t, slopes, scale, 1e-6, mask), [p], 5, name)


def test_attention_takes_the_native_route_and_warns_outside_it(gpu):
    from fastalgebraictransformer_amd import forward
    q = [_rand(i, 1, 2, 40, 64, dtype=torch.bfloat16).requires_grad_(True) for i in range(3)]
    slopes = F.compute_alibi_slopes(2).cuda()
    assert _lib.ops().attention(*q, slopes, 0.125, 1e-6) is not None
    forward._WARNED.clear()
    bad = _rand(9, 1, 2, 40, 65, dtype=torch.bfloat16)[..., 1:]
    assert _lib.ops().attention(bad, q[1], q[2], slopes, 0.125, 1e-6) is None
    with pytest.warns(RuntimeWarning, match="not 16-byte aligned"):
        F.rational_attention(bad, q[1], q[2], slopes, 0.125)
    forward._WARNED.clear()
    o = F.rational_attention(*q, slopes, 0.125)
    g = _rand(10, 1, 2, 40, 65, dtype=torch.bfloat16)[..., 1:]  # a gradient outside the envelope warns as well
    with pytest.warns(RuntimeWarning, match="not 16-byte aligned"):
        o.backward(g)
    forward._WARNED.clear()


def test_decode(gpu):
    B, H, T, D = 3, 4, 50, 64
    slopes = F.compute_alibi_slopes(H).cuda()
    q = _rand(1, B, H, D, dtype=torch.bfloat16)
    k, v = (_rand(i, B, T, H, D, dtype=torch.bfloat16).permute(0, 2, 1, 3) for i in (2, 3))
    n = torch.tensor([50, 17, 1], dtype=torch.int32, device="cuda")
    for lengths in (None, n, n.long(), n.cpu()):
        native = _lib.ops().decode(q, k, v, slopes, 0.125, lengths, 1e-6)
        assert (native is not None) == (lengths is None or lengths is n)
        o, L = F.rational_attention_decode(q, k, v, slopes, 0.125, lengths=lengths)
        # the Python route: a slopes tensor that needs a conversion
        o2, L2 = F.rational_attention_decode(q, k, v, slopes.double(), 0.125, lengths=lengths)
        assert torch.equal(o, o2) and torch.equal(L, L2)
    with pytest.raises(RuntimeError, match="kat_attn_decode failed"):
        F.rational_attention_decode(q[..., :60], k[..., :60], v[..., :60], slopes, 0.125)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_slopes_of_a_model_cast_whole(gpu, dtype):
    """A module cast whole holds 16-bit slopes: its attention, training and
    decode, takes the native route with the classes' results."""
    H, scale = 3, 0.125
    slopes = F.compute_alibi_slopes(H).cuda().to(dtype)
    q = [_rand(i, 2, H, 70, 64, dtype=dtype).requires_grad_(True) for i in range(3)]
    km = torch.rand(2, 70, generator=torch.Generator().manual_seed(1)).cuda() > 0.3
    ops = _lib.ops()
    assert ops.attention(*q, slopes, scale, 1e-6) is not None
    _same(lambda a, b, c: F.rational_attention(a, b, c, slopes, scale),
          lambda a, b, c: F.RationalAttentionFunction.apply(a, b, c, slopes, scale, True, 1e-6), q, 5, "plain")
    assert ops.attention_masked(*q, slopes, scale, km, False, 1e-6) is not None
    _same(lambda a, b, c: F.rational_attention_masked(a, b, c, slopes, scale, km, False),
          lambda a, b, c: F.backward.MaskedRationalAttentionFunction.apply(a, b, c, slopes, scale, km, False, 1e-6),
          q, 5, "masked")
    p = _rand(4, 2, 70, 3, H, 64, dtype=dtype).requires_grad_(True)
    assert ops.attention_packed(p, slopes, scale, 1e-6, None) is not None
    _same(lambda t: F.rational_attention_packed(t, slopes, scale),
          lambda t: F.PackedRationalAttention.apply(t, slopes, scale, 1e-6, None), [p], 5, "packed")
    one = q[0][:, :, 0].detach()
    assert ops.decode(one, q[1], q[2], slopes, scale, None, 1e-6) is not None
    # the Python route: the same slopes in a dtype the native functions leave to it
    for a, b in zip(F.rational_attention_decode(one, q[1], q[2], slopes, scale),
                    F.rational_attention_decode(one, q[1], q[2], slopes.double(), scale)):
        assert torch.equal(a, b)
    # slopes that ask for a gradient, or of the wrong count, stay with the classes
    assert ops.attention(*q, slopes.clone().requires_grad_(True), scale, 1e-6) is None
    assert ops.attention(*q, slopes[:2], scale, 1e-6) is None


def _ops_list():
    x = _rand(1, 6, 64, dtype=torch.bfloat16)
    w = torch.ones(64, device="cuda")
    q = [_rand(i, 1, 2, 33, 64, dtype=torch.bfloat16) for i in range(3)]
    slopes = F.compute_alibi_slopes(2).cuda()
    km = torch.ones(1, 33, dtype=torch.bool, device="cuda")
    return [("softmax", F.rational_softmax, [x]), ("swiglu", F.rational_swiglu, [x, x.clone()]),
            ("packed swiglu", F.rational_swiglu_packed, [x]), ("norm", F.mean_error_norm, [x, w]),
            ("add norm", lambda a, b, c: F.add_mean_error_norm(a, b, c)[1], [x, x.clone(), w]),
            ("attention", lambda a, b, c: F.rational_attention(a, b, c, slopes, 0.125), q),
            ("masked", lambda a, b, c: F.rational_attention_masked(a, b, c, slopes, 0.125, km), q),
            ("packed", lambda a: F.rational_attention_packed(a, slopes, 0.125),
             [_rand(5, 1, 33, 3, 2, 64, dtype=torch.bfloat16)])]


def _plain_grads(fn, ins):
    ins = [t.detach().clone().requires_grad_(True) for t in ins]
    y = fn(*ins)
    return y.detach(), torch.autograd.grad(y, ins, torch.ones_like(y))


def test_saved_tensor_hooks_and_checkpoint(gpu):
    from torch.utils.checkpoint import checkpoint
    for name, fn, ins in _ops_list():
        y0, g0 = _plain_grads(fn, ins)
        packed = []

        def pack(t):
            packed.append(tuple(t.shape))
            return t.cpu()

        def unpack(t):  # another layout than the saved one: a row stride, a new address
            t = t.cuda()
            if t.dim() < 2 or t.dtype in (torch.uint8, torch.bool):
                return t
            wide = torch.empty(t.shape[:-1] + (t.shape[-1] + 8,), dtype=t.dtype, device="cuda")
            return wide[..., :t.shape[-1]].copy_(t)

        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            leaves = [t.detach().clone().requires_grad_(True) for t in ins]
            y = fn(*leaves)
        assert packed, name
        g = torch.autograd.grad(y, leaves, torch.ones_like(y))
        assert all(torch.equal(a, b) for a, b in zip(g, g0)), name
        leaves = [t.detach().clone().requires_grad_(True) for t in ins]
        y = checkpoint(fn, *leaves, use_reentrant=False)
        g = torch.autograd.grad(y, leaves, torch.ones_like(y))
        assert torch.equal(y, y0) and all(torch.equal(a, b) for a, b in zip(g, g0)), name
        # saved tensors that come back on the host raise instead of being read
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t):
            leaves = [t.detach().clone().requires_grad_(True) for t in ins]
            y = fn(*leaves)
        with pytest.raises(RuntimeError):
            torch.autograd.grad(y, leaves, torch.ones_like(y))


def _masked_ops(D):
    q = [_rand(i, 3, 2, 70, D, dtype=torch.bfloat16) for i in range(3)]
    slopes = F.compute_alibi_slopes(2).cuda()
    km = torch.rand(3, 70, generator=torch.Generator().manual_seed(2)).cuda() > 0.4
    cls, pcls = F.backward.MaskedRationalAttentionFunction, F.backward.PackedRationalAttention
    return [("masked", lambda a, b, c: F.rational_attention_masked(a, b, c, slopes, 0.125, km), q),
            ("masked class", lambda a, b, c: cls.apply(a, b, c, slopes, 0.125, km, True, 1e-6), q),
            ("packed", lambda a: F.rational_attention_packed(a, slopes, 0.125, key_mask=km),
             [_rand(5, 3, 70, 3, 2, D, dtype=torch.bfloat16)]),
            ("packed class", lambda a: pcls.apply(a, slopes, 0.125, 1e-6, km),
             [_rand(5, 3, 70, 3, 2, D, dtype=torch.bfloat16)])]


@pytest.mark.filterwarnings("ignore:rational attention in")
@pytest.mark.parametrize("D", [64, 20])  # the MFMA kernels, and a head dim outside them
def test_saved_key_mask_of_another_layout_or_place(gpu, D):
    """Only the mask comes back changed from a saved-tensor hook: with a row
    stride it gives the same gradients; on the host, in another dtype or with
    other sizes it raises before any launch."""
    def mask_only(change):
        return torch.autograd.graph.saved_tensors_hooks(
            lambda t: t, lambda t: change(t) if t.dtype == torch.uint8 else t)

    def strided(t):
        return torch.zeros(t.shape[0], t.shape[1] + 9, dtype=t.dtype, device="cuda")[:, :t.shape[1]].copy_(t)

    for name, fn, ins in _masked_ops(D):
        _, g0 = _plain_grads(fn, ins)
        for change in (strided, lambda t: t.t().contiguous().t()):
            with mask_only(change):
                _, g = _plain_grads(fn, ins)
            assert all(torch.equal(a, b) for a, b in zip(g, g0)), name
        for change in (lambda t: t.cpu(), lambda t: t.float(), lambda t: t[:, :-1], lambda t: t[:1]):
            with mask_only(change), pytest.raises(RuntimeError, match="saved key mask"):
                _plain_grads(fn, ins)


def _class_ops():
    x = _rand(1, 6, 64, dtype=torch.bfloat16)
    w = torch.ones(64, device="cuda")
    q = [_rand(i, 1, 2, 33, 64, dtype=torch.bfloat16) for i in range(3)]
    slopes = F.compute_alibi_slopes(2).cuda()
    return [("softmax class", lambda a: F.RationalSoftmax.apply(a, 1e-6), [x]),
            ("swiglu class", F.RationalSwiGLU.apply, [x, x.clone()]),
            ("packed swiglu class", F.PackedRationalSwiGLU.apply, [x]),
            ("norm class", lambda a, b: F.MeanErrorNorm.apply(a, b, 1e-6), [x, w]),
            ("add norm class", lambda a, b, c: F.ResidualMeanErrorNorm.apply(a, b, c, 1e-6, None)[1],
             [x, x.clone(), w]),
            ("attention class", lambda a, b, c: F.RationalAttentionFunction.apply(a, b, c, slopes, 0.125, True, 1e-6),
             q)]


def test_one_saved_tensor_of_another_layout_type_size_or_place(gpu):
    """Each saved tensor alone comes back changed from a saved-tensor hook: in
    a wider dtype and with a row stride it gives the same gradients (but for
    the first, whose dtype is the launch's); with fewer rows or columns or on
    the host it raises before any launch."""
    def strided(t):
        wide = torch.empty(t.shape[:-1] + (t.shape[-1] + 9,), dtype=torch.float64, device="cuda")
        return wide[..., 1:t.shape[-1] + 1].copy_(t)

    def one(i, change):
        n = [0]

        def pack(t):
            n[0] += 1
            return n[0] - 1, t
        return torch.autograd.graph.saved_tensors_hooks(pack, lambda p: change(p[1]) if p[0] == i else p[1])

    for name, fn, ins in _ops_list() + _class_ops() + _masked_ops(64):
        saved = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: saved.append(t.dtype) or t, lambda t: t):
            _, g0 = _plain_grads(fn, ins)
        for i, dt in enumerate(saved):
            if i > 0 and dt != torch.uint8:
                with one(i, strided):
                    _, g = _plain_grads(fn, ins)
                assert all(torch.equal(a, b) for a, b in zip(g, g0)), (name, i)
            for change in (lambda t: t[..., :-1], lambda t: t[:-1]):
                with one(i, change), pytest.raises(RuntimeError):
                    _plain_grads(fn, ins)
            try:
                with one(i, lambda t: t.cpu()):
                    _, g = _plain_grads(fn, ins)
            except (RuntimeError, AssertionError):
                continue
            # the classes move the slopes to the device, as their forward does
            assert dt == torch.float32 and name.endswith("class"), (name, i)
            assert all(torch.equal(a, b) for a, b in zip(g, g0)), (name, i)
    # a probability saved narrower than its logits (fp32) is widened before it is read
    x = _rand(3, 9, 65).requires_grad_(True)
    for fn in (F.rational_softmax, lambda t: F.RationalSoftmax.apply(t, 1e-6)):
        want = torch.autograd.grad(fn(x), x, _rand(4, 9, 65))[0]
        with one(1, lambda t: t.bfloat16()):
            got = torch.autograd.grad(fn(x), x, _rand(4, 9, 65))[0]
        assert float((got - want).norm() / want.norm()) < 2.0 ** -7  # p's bf16 rounding, 2^-9 a factor


def test_batched_gradients_raise(gpu):
    for name, fn, ins in _ops_list() + _class_ops():
        leaves = [t.detach().clone().requires_grad_(True) for t in ins]
        y = fn(*leaves)
        with pytest.raises(RuntimeError):
            torch.autograd.grad(y, leaves, torch.ones(2, *y.shape, dtype=y.dtype, device="cuda"),
                                is_grads_batched=True)


def test_negated_gradient_views(gpu):
    """A gradient that is a lazily negated view is read as its values."""
    for name, fn, ins in _ops_list():
        leaves = [t.detach().clone().requires_grad_(True) for t in ins]
        y = fn(*leaves)
        c = _rand(8, *y.shape, dtype=y.dtype)
        want = torch.autograd.grad(y, leaves, -c, retain_graph=True)
        got = torch.autograd.grad(y, leaves, torch._neg_view(c))
        assert all(torch.equal(a, b) for a, b in zip(want, got)), name


def test_modes_and_partial_gradients(gpu):
    for name, fn, ins in _ops_list():
        y0, g0 = _plain_grads(fn, ins)
        with torch.no_grad():
            y = fn(*[t.clone().requires_grad_(True) for t in ins])
            assert not y.requires_grad and torch.equal(y, y0), name
        with torch.inference_mode():
            assert torch.equal(fn(*ins), y0), name
        for i in range(len(ins)):  # one input at a time needs a gradient
            leaves = [t.detach().clone().requires_grad_(j == i) for j, t in enumerate(ins)]
            y = fn(*leaves)
            (g,) = torch.autograd.grad(y, [leaves[i]], torch.ones_like(y))
            assert torch.equal(g, g0[i]), name
        leaves = [t.detach().clone().requires_grad_(True) for t in ins]
        y = fn(*leaves)  # gradients made with create_graph carry no graph, as the classes' do
        g = torch.autograd.grad(y, leaves, torch.ones_like(y), create_graph=True)
        assert all(torch.equal(a, b) for a, b in zip(g, g0)), name
        assert all(not t.requires_grad for t in g), name
        y = fn(*leaves)
        y.sum().backward()
        with pytest.raises(RuntimeError):  # the graph is freed
            y.sum().backward()


def test_transforms_raise_or_run_as_the_classes_do(gpu):
    x = _rand(1, 4, 64)
    t = torch.ones_like(x)
    with pytest.raises(RuntimeError):
        torch.func.vmap(F.rational_softmax)(x)
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda a: F.rational_softmax(a).sum())(x)
    import torch.autograd.forward_ad as fwad
    with fwad.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        F.rational_softmax(fwad.make_dual(x, t))
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode() as m:
        assert _lib.ops().softmax(m.from_tensor(x), 1e-6) is None
    assert _lib.ops().softmax(x.cpu(), 1e-6) is None
    assert _lib.ops().softmax(x.long(), 1e-6) is None
    assert _lib.ops().softmax(x[:0], 1e-6) is None
    assert _lib.ops().swiglu(x, x.double()) is None
    assert _lib.ops().swiglu(x, x[:2]) is None
    assert _lib.ops().norm(x, torch.ones(63, device="cuda"), 1e-6) is None
    assert _lib.ops().norm(x, torch.ones(64), 1e-6) is None
    with pytest.raises(AssertionError):
        F.rational_swiglu(x, x[:2])
    with pytest.raises(AssertionError):
        F.mean_error_norm(x, torch.ones(63, device="cuda"))


def test_streams_and_threads(gpu):
    """Passes from two threads, each on its own stream, equal the same passes alone."""
    import threading
    cases = [(f, ins) for _, f, ins in _ops_list()]
    alone = [_plain_grads(f, ins) for f, ins in cases]
    torch.cuda.synchronize()
    bad = []

    def work():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(5):
                for (f, ins), (y0, g0) in zip(cases, alone):
                    y, g = _plain_grads(f, ins)
                    s.synchronize()
                    if not (torch.equal(y, y0) and all(torch.equal(a, b) for a, b in zip(g, g0))):
                        bad.append(1)

    ts = [threading.Thread(target=work) for _ in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
