"""The training path's autograd nodes in C++ beside the Python functions that they stand for, and what goes with them."""
import copy

import pytest
import torch

from deepspeedsyclsupport_amd.ops import attention as A
from deepspeedsyclsupport_amd.ops import linear as L
from deepspeedsyclsupport_amd.ops.native import hip_ops
from deepspeedsyclsupport_amd.ops.transformer import functional as DF

pytestmark = pytest.mark.gpu


def _rnd(*shape, seed=0):
    return torch.randn(shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed)).bfloat16()


def _leaf(*shape, seed=0):
    return _rnd(*shape, seed=seed).requires_grad_()


def _tables(n, rot):
    from deepspeedsyclsupport_amd.ops.reference import rope_tables
    return [t.cuda() for t in rope_tables(n, rot, 10000.0)]


def _linear():
    return (lambda x, w: L.linear(x, w)), (lambda x, w: L.LinearFunction.apply(x, w, None, None)), \
        [_leaf(3, 5, 64), _leaf(72, 64, seed=1)]


def _norm():
    return (lambda x, w: DF.rms_norm(x, w, 1e-5)), (lambda x, w: DF._RMSNormFn.apply(x, w, 1e-5, None)), [_leaf(7, 256), _leaf(256, seed=1)]


def _norm_sum():
    return (lambda x, w, r: DF.rms_norm(x, w, 1e-5, r)), (lambda x, w, r: DF._RMSNormFn.apply(x, w, 1e-5, r)), \
        [_leaf(2, 9, 512), _leaf(512, seed=1), _leaf(2, 9, 512, seed=2)]


def _norm_first():
    """The sum is not used any more."""
    return (lambda x, w, r: DF.rms_norm(x, w, 1e-5, r)[0]), (lambda x, w, r: DF._RMSNormFn.apply(x, w, 1e-5, r)[0]), \
        [_leaf(2, 9, 512), _leaf(512, seed=1), _leaf(2, 9, 512, seed=2)]


def _norm_second():
    return (lambda x, w, r: DF.rms_norm(x, w, 1e-5, r)[1]), (lambda x, w, r: DF._RMSNormFn.apply(x, w, 1e-5, r)[1]), \
        [_leaf(2, 9, 512), _leaf(512, seed=1), _leaf(2, 9, 512, seed=2)]


def _gate():
    return (lambda x: DF.gated_activation(x, "gelu")), (lambda x: DF._GatedActFn.apply(x, 2)), [_leaf(33, 208)]


def _rope():
    cos, sin = _tables(40, 128)
    pos = torch.arange(6, 6 + 17, device="cuda").repeat(2, 1)
    return (lambda x: DF.qkv_rope_split(x, cos, sin, 4, 2, position_ids=pos, token_major=True)), \
        (lambda x: DF._QKVRopeFn.apply(x, cos, sin, pos.int().contiguous(), 4, 2, 128, 0, True)), [_leaf(2, 17, 8, 128)]


def _flash():
    return (lambda q, k, v: A.attention(q, k, v)), (lambda q, k, v: A.FlashAttnFunc.apply(q, k, v, True, 128**-0.5)), \
        [_leaf(1, 4, 70, 128), _leaf(1, 2, 70, 128, seed=1), _leaf(1, 2, 70, 128, seed=2)]


def _loss():
    labels = torch.randint(0, 96, (21, ), device="cuda", generator=torch.Generator(device="cuda").manual_seed(4))
    labels[3] = -100
    return (lambda x: DF.cross_entropy(x * 1, labels)), (lambda x: DF._XentMeanFn.apply(x * 1, labels, -100, 0.0, True)), [_leaf(21, 96)]


CASES = [_linear, _norm, _norm_sum, _norm_first, _norm_second, _gate, _rope, _flash, _loss]


def _grads(f, inputs, seed=9):
    out = f(*inputs)
    outs = out if isinstance(out, tuple) else tuple(out) if isinstance(out, list) else (out, )
    gos = [_rnd(*o.shape, seed=seed + i).to(o.dtype) for i, o in enumerate(outs)]
    return outs, torch.autograd.grad(outs, inputs, gos, allow_unused=True)


def _same(a, b, exact):
    for x, y in zip(a, b):
        assert (x is None) == (y is None)
        if x is not None:
            if exact:
                assert torch.equal(x, y)
            else:  # (dQ comes by atomics)
                torch.testing.assert_close(x.float(), y.float(), rtol=2e-2, atol=2e-2 * y.float().abs().max().item())


@pytest.mark.parametrize("case", CASES, ids=lambda c: c.__name__[1:])
def test_node_is_the_function(case):
    """Outputs and gradients; what saved-tensor hooks see; the node in its place, and the function where a mode has to see torch's calls."""
    node, function, inputs = case()
    exact = case is not _flash
    for a, b in zip(_grads(node, inputs), _grads(function, inputs)):
        _same(a, b, exact)
    out = node(*inputs)
    first = out[0] if isinstance(out, (tuple, list)) else out
    assert "Node" in type(first.grad_fn).__name__ or "CppFunction" in type(first.grad_fn).__name__ or "Node" in first.grad_fn.name()

    def seen(f):
        shapes = []

        def pack(t):
            shapes.append((tuple(t.shape), t.dtype))
            return t.clone()
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
            outs, grads = _grads(f, inputs)
        return sorted(shapes, key=str), grads
    (s1, g1), (s2, g2) = seen(node), seen(function)
    assert s1 == s2
    _same(g1, g2, exact)
    from torch.overrides import TorchFunctionMode

    class Mode(TorchFunctionMode):

        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    from torch.utils.flop_counter import FlopCounterMode
    for mode in (Mode(), FlopCounterMode(display=False)):
        with mode:
            out = node(*inputs)
        first = out[0] if isinstance(out, (tuple, list)) else out
        assert "Node" not in first.grad_fn.name()
    with torch.no_grad():
        _same([o for o in _grads_free(node, inputs)], [o for o in _grads_free(function, inputs)], True)


def _grads_free(f, inputs):
    out = f(*[t.detach() for t in inputs])
    return out if isinstance(out, (tuple, list)) else (out, )


@pytest.mark.parametrize("case", CASES, ids=lambda c: c.__name__[1:])
def test_outputs_change_in_place(case):
    """Outputs may be changed in place where the function's may, and the gradients are the function's."""
    node, function, inputs = case()

    def run(f):
        try:
            out = f(*inputs)
            first = out[0] if isinstance(out, (tuple, list)) else out
            return True, torch.autograd.grad(first.mul_(2).float().sum(), inputs, allow_unused=True)
        except RuntimeError:
            return False, ()
    (ok, a), (want, b) = run(node), run(function)
    assert ok == want
    _same(a, b, case is not _flash)


def _result(f):
    try:
        return f()
    except (RuntimeError, NotImplementedError):
        return None


@pytest.mark.parametrize("case", CASES, ids=lambda c: c.__name__[1:])
def test_node_under_transforms(case):
    """Gradients that are differentiated again, batches of gradients, tangents and recomputed segments: what the function gives, or its
    refusal."""
    from torch.autograd import forward_ad
    from torch.utils.checkpoint import checkpoint
    node, function, inputs = case()
    first = lambda f, ins: (lambda o: o[0] if isinstance(o, (tuple, list)) else o)(f(*ins))  # noqa: E731

    def again(f):
        grads = torch.autograd.grad(first(f, inputs).float().pow(2).sum(), inputs, create_graph=True, allow_unused=True)
        flags = [g is not None and g.requires_grad for g in grads]
        more = _result(lambda: torch.autograd.grad(sum(g.float().pow(2).sum() for g in grads if g is not None), inputs, allow_unused=True))
        return flags, [g for g in grads if g is not None], more

    def batched(f):
        y = first(f, inputs)
        go = torch.stack([torch.ones_like(y), 2 * torch.ones_like(y)])
        return _result(lambda: torch.autograd.grad(y, inputs, go, is_grads_batched=True, allow_unused=True))

    def tangent(f):
        with forward_ad.dual_level():
            dual = [forward_ad.make_dual(t.detach(), torch.ones_like(t)) for t in inputs]
            return _result(lambda: [t for t in forward_ad.unpack_dual(first(f, dual)) if t is not None])

    def recomputed(f):
        y = checkpoint(lambda *a: first(f, a) * 2, *inputs, use_reentrant=False)
        return y, *torch.autograd.grad(y.float().sum(), inputs, allow_unused=True)
    exact = case is not _flash
    (flags, grads, more), (flags2, grads2, more2) = again(node), again(function)
    assert flags == flags2 and (more is None) == (more2 is None)
    _same(grads, grads2, exact)
    _same(more or (), more2 or (), exact)
    for how in (batched, tangent, recomputed):
        a, b = how(node), how(function)
        assert (a is None) == (b is None)
        _same(a or (), b or (), exact)


def test_linear_under_transforms():
    """The layer as it is called, against torch's linear: the gradient's gradient and a batch of vectors through the Jacobian."""
    x, w, go = _leaf(96, 128), _leaf(192, 128, seed=1), _rnd(96, 192, seed=2)
    kept = []
    for f in (L.linear, torch.nn.functional.linear):
        (g1, ) = torch.autograd.grad(f(x, w).float().pow(2).sum(), x, create_graph=True)
        (g2, ) = torch.autograd.grad(g1.float().pow(2).sum(), w)
        kept.append((g1, g2, *torch.autograd.grad(f(x, w), (x, w), torch.stack([go, 2 * go]), is_grads_batched=True)))
    assert "Node" in L.linear(x, w).grad_fn.name()
    for got, want in zip(*kept):   # (bf16 in between: a few roundings of 2^-9 each, of sums whose terms may cancel)
        torch.testing.assert_close(got.float(), want.float(), rtol=0.03, atol=0.03 * want.float().abs().max().item())


@pytest.mark.parametrize("lead", [(96, ), (2, 48), (1, 96)])
def test_linear_changes_in_place(lead):
    """A linear layer's output of a short batch, changed in place by itself and through views, as torch's may be."""
    x, w, go = _leaf(*lead, 128), _leaf(256, 128, seed=1), _rnd(*lead, 256, seed=2)
    rows = lambda y: y.view(-1, 8, 32)[:, 2:5]  # noqa: E731

    def changed(f):
        y = f(x, w)
        y.mul_(2)
        y += go
        rows(y).relu_()
        return y
    want = torch.nn.functional.linear(x, w)
    for f in (L.linear, lambda a, b: L.LinearFunction.apply(a, b, None, None)):
        y, z = changed(f), 2 * f(x, w) + go
        mask = torch.ones_like(z)
        rows(mask)[rows(z) <= 0] = 0
        assert torch.equal(y, z * mask)
        for a, b in zip(torch.autograd.grad(y, (x, w), go), torch.autograd.grad(z * mask, (x, w), go)):
            assert torch.equal(a, b)
        # (sums of 128 products in fp32, one rounding on either side)
        assert ((f(x, w).float() - want.float()).abs() <= 2**-7 * want.float().abs() + 1e-4).all()


def test_released_weight():
    """A weight whose storage is released after the forward pass and filled again before the backward one, as gathered weights are."""
    x, w = _leaf(8, 64), torch.nn.Parameter(_rnd(24, 64, seed=1))
    go, full = _rnd(8, 24, seed=2), w.detach().clone()
    (want, ) = torch.autograd.grad(L.LinearFunction.apply(x, w, None, None), x, go)
    y = L.linear(x, w)
    w.data = torch.empty(0, device="cuda", dtype=torch.bfloat16)
    w.data = full
    y.backward(go)
    assert torch.equal(x.grad, want) and w.grad.shape == w.shape


def test_casts_and_types_are_left():
    x, w = _leaf(8, 64), _leaf(24, 64, seed=1)
    with torch.autocast("cuda", dtype=torch.float16):
        assert L.linear(x, w).dtype == torch.float16
    assert L.linear(x.float(), w.float()).dtype == torch.float32
    assert DF.rms_norm(x.float(), _leaf(64).float()).dtype == torch.float32
    with pytest.raises(RuntimeError):   # (a Python function without a rule for it, as before)
        torch.func.vmap(lambda t: L.linear(t, w))(x[None])


@pytest.mark.parametrize("rows,H", [(1, 8), (2, 40), (33, 1000), (130, 1032), (2049, 264), (515, 8192)])
@pytest.mark.parametrize("kind", ["rms", "ln"])
def test_norm_weight_gradient(kind, rows, H):
    """The sums over rows of any number, for widths that fill no block of columns; the same bits each time."""
    ops = hip_ops()
    x, w, dy = _rnd(rows, H), _rnd(H, seed=1), _rnd(rows, H, seed=2)
    xd, g = x.double(), dy.double()
    if kind == "rms":
        rstd = ops.rms_fwd(x, None, w, 1e-5)[2]
        run = lambda: ops.rms_bwd(dy, x, w, rstd, None)  # noqa: E731
        want = [(g * xd * torch.rsqrt((xd * xd).mean(-1, keepdim=True) + 1e-5)).sum(0)]
    else:
        _, _, mean, rstd = ops.ln_fwd(x, None, w, w, 1e-5)
        run = lambda: ops.ln_bwd(dy, x, w, mean, rstd, None)  # noqa: E731
        c = xd - xd.mean(-1, keepdim=True)
        want = [(g * c * torch.rsqrt((c * c).mean(-1, keepdim=True) + 1e-5)).sum(0), g.sum(0)]
    got = run()[1:]
    for a, b in zip(got, want):
        # one rounding to bf16, sums of `rows` products in fp32 (of order sqrt(rows), each off by at most rows 2^-24 of that)
        assert ((a.double() - b).abs() <= b.abs() * 2**-8 + rows**0.5 * 1e-3).all()
    for a, b in zip(got, run()[1:]):
        assert torch.equal(a, b)


def test_adam_over_flats():
    """Items at offsets of flat state: the same bits as over views of it, and nothing beside them changes."""
    ops, offs, sizes = hip_ops(), [0, 40, 300], [33, 256, 1000]
    args = (1e-2, 0.9, 0.95, 1e-8, 0.1, 0.5, 0.25, 0.7, True)
    flat = [torch.rand(1400, device="cuda") for _ in range(3)]
    g, lp = [_rnd(n, seed=n) for n in sizes], [_rnd(n, seed=n + 1) for n in sizes]
    one, two = (flat, lp), copy.deepcopy((flat, lp))
    ops.adam_multi_flat(*one[0], offs, g, one[1], *args)
    views = [[t[o:o + n] for o, n in zip(offs, sizes)] for t in two[0]]
    ops.adam_multi(*views, g, two[1], *args)
    for a, b in zip([*one[0], *one[1]], [*two[0], *two[1]]):
        assert torch.equal(a, b)
    with pytest.raises(RuntimeError):
        ops.adam_multi_flat(*flat, [0, 40, 401], g, lp, *args)
