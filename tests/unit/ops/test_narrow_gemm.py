"""Products around a short batch of tokens (`csrc/gemm/narrow_gemm.hip`) and the linear layer that takes them."""
import pytest
import torch
import torch.nn.functional as F

from deepspeedsyclsupport_amd.ops.linear import LinearFunction, plain_linear
from deepspeedsyclsupport_amd.ops.native import hip_ops

GPU = pytest.mark.gpu


def _rnd(*shape, seed=0):
    return torch.randn(*shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed)).bfloat16()


def _check(got, a, b):
    """One rounding to bf16 (2^-9 of the value) and sums of K products in fp32, off by less than K 2^-23 of the magnitudes' sum."""
    a, b = a.double(), b.double()
    want, size = a @ b.t(), a.abs() @ b.abs().t()
    assert got.shape == want.shape
    assert ((got.double() - want).abs() <= want.abs() * 2**-8 + size * a.shape[1] * 2**-23).all()


@GPU
@pytest.mark.parametrize("tile,parts", [(0, 0), (32, 1), (32, 3), (64, 1), (64, 2), (128, 1), (128, 2)])
@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (8, 40, 64), (31, 64, 128), (33, 72, 192), (64, 136, 256), (72, 200, 320), (128, 96, 448),
                                   (127, 264, 576), (136, 1032, 1088)])
def test_products_at_their_edges(M, N, K, tile, parts):
    """Both forms of both operands; tiles that rows, columns or the inner dimension do not fill; fewer steps than buffers, and every
    remainder of them; operands that are columns of wider matrices; the same bits each time."""
    ops = hip_ops()
    a, b = _rnd(M, K, seed=1), _rnd(N, K, seed=2)
    wide_a, wide_b = _rnd(M, K + 24, seed=3), _rnd(K, N + 16, seed=4)
    ops.narrow_gemm_tune(tile, parts)
    try:
        got = ops.narrow_gemm(a, b, True, True)
        _check(got, a, b)
        assert torch.equal(got, ops.narrow_gemm(a, b, True, True))
        _check(ops.narrow_gemm(a, b.t().contiguous(), True, False), a, b)
        _check(ops.narrow_gemm(wide_a[:, 8:8 + K], wide_b[:, 8:8 + N], True, False), wide_a[:, 8:8 + K], wide_b[:, 8:8 + N].t())
        if M % 8 == 0:
            at = a.t().contiguous()
            _check(ops.narrow_gemm(at, b, False, True), a, b)
            for rows in (K, K - 1, K - 37, 1):   # (an inner dimension of any length)
                _check(ops.narrow_gemm(at[:rows], b.t().contiguous()[:rows], False, False), a[:, :rows], b[:, :rows])
    finally:
        ops.narrow_gemm_tune(0, 0)


@GPU
@pytest.mark.parametrize("parts", [1, 2])
@pytest.mark.parametrize("M,N,K", [(8, 8, 64), (72, 264, 128), (128, 256, 192), (136, 248, 256), (128, 520, 320), (264, 1032, 576)])
def test_tiles_of_256_columns(M, N, K, parts):
    """One step to several times as many as buffers; the last tile's second half empty, or short of columns; every form."""
    test_products_at_their_edges(M, N, K, 256, parts)


@GPU
@pytest.mark.parametrize("M,N", [(2048, 2304), (2000, 4104), (1032, 4864), (2944, 5632)])
def test_more_than_one_round(M, N):
    """Where the rule goes from one round of 128 x 128 to one or two of 128 x 256, and back."""
    a, b = _rnd(M, 192, seed=1), _rnd(N, 192, seed=2)
    at, bt = a.t().contiguous(), b.t().contiguous()
    _check(hip_ops().narrow_gemm(a, b, True, True), a, b)
    _check(hip_ops().narrow_gemm(a, bt, True, False), a, b)
    _check(hip_ops().narrow_gemm(at, bt, False, False), a, b)


@GPU
@pytest.mark.parametrize("M,N,K", [(52, 6152, 4096), (1, 6144, 4096), (128, 6200, 4160), (129, 4104, 8192), (256, 5120, 5120), (100, 2056, 5632),
                                   (33, 1024, 8192), (255, 4096, 4096), (300, 4096, 4160), (100, 25608, 4096), (129, 11264, 2048), (193, 14328, 4096)])
def test_long_inner_dimensions(M, N, K):
    """Tiles and parts as the rule chooses them for K from 4096 on: 128 x 128 (rows a multiple of 8 KB apart begin elsewhere in K, unless
    tiles share weights) and 64 x 64, and beyond them; the same bits each time."""
    ops = hip_ops()
    a, b = _rnd(M, K, seed=1), _rnd(N, K, seed=2)
    got = ops.narrow_gemm(a, b, True, True)
    _check(got, a, b)
    assert torch.equal(got, ops.narrow_gemm(a, b, True, True))
    _check(plain_linear(a, b), a, b)


@GPU
@pytest.mark.parametrize("form,M,N,K", [("dX", 128, 5376, 5120), ("dX", 120, 5504, 5120), ("dX", 128, 5504, 5056), ("dX", 57, 11008, 5632), ("dX", 250, 8192, 4160),
                                        ("dX", 250, 8320, 4160), ("dX", 250, 5120, 3072), ("dX", 250, 5120, 3008), ("dX", 250, 7680, 3136), ("dX", 250, 7808, 3136), ("dX", 250, 7808, 4096),
                                        ("dW", 376, 3584, 2705), ("dW", 1032, 1064, 2047), ("dW", 1032, 1064, 2048), ("dW", 1280, 1544, 2200), ("dW", 1280, 1536, 2200),
                                        ("y", 52, 16384, 2048), ("y", 65, 16384, 2048), ("y", 52, 16392, 2048), ("y", 50, 2112, 4608), ("y", 50, 2048, 4608),
                                        ("y", 238, 4096, 5120), ("y", 238, 4096, 5056), ("y", 100, 11008, 4096), ("y", 130, 5504, 8192),
                                        ("dW", 2432, 6664, 1023), ("dW", 2432, 6664, 1024)])
def test_cuts(form, M, N, K):
    """Either side of the lines between tiles and parts; the same bits each time."""
    ops = hip_ops()
    a, b = _rnd(M, K, seed=1), _rnd(N, K, seed=2)
    args = {"y": (a, b, True, True), "dX": (a, b.t().contiguous(), True, False), "dW": (a.t().contiguous(), b.t().contiguous(), False, False)}[form]
    got = ops.narrow_gemm(*args)
    _check(got, a, b)
    assert torch.equal(got, ops.narrow_gemm(*args))


@GPU
@pytest.mark.parametrize("T,O,I", [(1027, 2056, 520), (1027, 520, 2056), (1500, 1608, 1608), (3001, 256, 1032), (8192, 136, 264), (300, 2048, 5632), (2049, 1032, 1024)])
def test_gradients_of_many_tokens(T, O, I):
    """Tiles in bands of rows, the last one of fewer, over inner dimensions of any length; what the layer takes."""
    ops = hip_ops()
    go, x, w = _rnd(T, O, seed=1), _rnd(T, I, seed=2), _rnd(O, I, seed=3)
    got = ops.narrow_gemm(go, x, False, False)
    _check(got, go.t(), x.t())
    assert torch.equal(got, ops.narrow_gemm(go, x, False, False)) and torch.equal(got, ops.linear_weight_grad(go, x))
    _check(ops.linear_input_grad(go, w), go, w.t())
    _check(ops.linear(x, w), x, w)


@GPU
def test_values_that_do_not_mix():
    """Infinities and NaN stay in their rows; nothing from past the end of an operand comes in."""
    a, b = _rnd(40, 128), _rnd(48, 128, seed=1)
    a[3, 5], a[4, 7] = float("inf"), float("nan")
    y = hip_ops().narrow_gemm(a, b, True, True)
    keep = [i for i in range(40) if i not in (3, 4)]
    _check(y[keep], a[keep], b)
    assert not y[3].isfinite().any() and y[4].isnan().all()
    big = _rnd(64, 256)
    big[40:] = float("nan")
    _check(hip_ops().narrow_gemm(big[:40, :128].contiguous(), b, True, True), big[:40, :128], b)
    _check(hip_ops().narrow_gemm(big[:37, :40], big[:37, 40:104], False, False), big[:37, :40].t(), big[:37, 40:104].t())


def test_tuning_is_a_threads_own():
    """What one thread forces for a measurement leaves another's products, and the scratch memory that they ask for, as they are."""
    import ctypes
    import threading
    from deepspeedsyclsupport_amd.ops import op_builder
    op_builder.load("ds_hip_ops")
    lib = ctypes.CDLL(op_builder.so_path("ds_hip_ops"))
    lib.ds_narrow_gemm_scratch.restype = lib.ds_decode_gemm_scratch.restype = ctypes.c_int64
    n = ctypes.c_int64
    query = lambda: (lib.ds_narrow_gemm_scratch(n(128), n(1024), n(1024), 1, 1), lib.ds_decode_gemm_scratch(4, 2048, 2048, 0, 0))  # noqa: E731
    before, seen = query(), []

    def other():
        lib.ds_narrow_gemm_tune(32, 8)
        lib.ds_skinny_b16_tune(1, 8)
        seen.append(query())
    thread = threading.Thread(target=other)
    thread.start()
    thread.join()
    assert all(s > b for s, b in zip(seen[0], before)) and query() == before


@GPU
@pytest.mark.parametrize("lead", [(2, 33), (128, )])
def test_linear_layer(lead):
    """What differentiates, transforms, counts or casts torch's linear does so here; the products are the narrow ones."""
    I, O = 128, 192
    x, w = _rnd(*lead, I).requires_grad_(), _rnd(O, I, seed=1).requires_grad_()
    go = _rnd(*lead, O, seed=2)
    y = LinearFunction.apply(x, w, None, None)
    gx, gw = torch.autograd.grad(y, (x, w), go)
    x2, go2 = x.detach().reshape(-1, I), go.reshape(-1, O)
    assert torch.equal(y.reshape(-1, O), hip_ops().narrow_gemm(x2, w.detach(), True, True))
    assert torch.equal(gx.reshape(-1, I), hip_ops().narrow_gemm(go2, w.detach(), True, False))
    assert torch.equal(gw, hip_ops().narrow_gemm(go2, x2, False, False))
    # (the gradient's gradient, and a batch of vectors through the Jacobian: torch's own products)
    for f in (lambda a, b: LinearFunction.apply(a, b, None, None), F.linear):
        out = f(x, w)
        (g1, ) = torch.autograd.grad(out.float().pow(2).sum(), x, create_graph=True)
        (g2, ) = torch.autograd.grad(g1.float().pow(2).sum(), w)
        rows = torch.autograd.grad(f(x, w), (x, w), torch.stack([go, 2 * go]), is_grads_batched=True)
        if f is F.linear:
            for got, want in zip(kept, (g1, g2, *rows)):
                torch.testing.assert_close(got.float(), want.float(), rtol=0.03, atol=0.03 * want.float().abs().max().item())
        kept = (g1, g2, *rows)
    from torch.utils.flop_counter import FlopCounterMode
    with FlopCounterMode(display=False) as count:
        LinearFunction.apply(x, w, None, None).backward(go)
    assert count.get_total_flops() == 3 * 2 * x2.shape[0] * I * O
    with torch.autocast("cuda", dtype=torch.float16):
        assert plain_linear(x.detach(), w.detach()).dtype == torch.float16
    from torch.fx.experimental.proxy_tensor import make_fx
    with torch.no_grad():
        assert any("mm" in str(n.target) for n in make_fx(lambda a, b: plain_linear(a, b))(x.detach(), w.detach()).graph.nodes)
        assert torch.equal(torch.func.vmap(plain_linear, (0, None))(x.detach()[None], w.detach())[0],
                           torch.func.vmap(F.linear, (0, None))(x.detach()[None], w.detach())[0])


@GPU
@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="tensors beside the current device")
def test_products_on_another_device():
    """Short products run on their tensors' device and its stream, in order with what made the tensors there, while another is current."""
    from deepspeedsyclsupport_amd.ops import hybrid_ops
    from deepspeedsyclsupport_amd.ops.linear import input_grad, linear, weight_grad
    a, b, go = _rnd(128, 1024, seed=1), _rnd(1024, 1024, seed=2), _rnd(128, 1024, seed=3)
    want = hip_ops().narrow_gemm(a, b, True, True), hip_ops().narrow_gemm(go, b, True, False), hip_ops().narrow_gemm(go, a, False, False)
    side = torch.cuda.Stream(1)
    with torch.cuda.stream(side):
        slow = torch.randn(4096, 4096, device="cuda:1")
        for _ in range(20):
            slow = slow @ slow * 1e-2
        x, w, g = (t.to("cuda:1") for t in (a, b, go))
        x, w, g = ((t + 0 * slow[0, 0].nan_to_num(0, 0, 0).to(t.dtype)) for t in (x, w, g))
        torch.cuda.set_device(0)
        assert torch.cuda.current_stream(1) == side
        got = [f(x, w) for f in (plain_linear, hybrid_ops.linear, linear)], input_grad(g, w), weight_grad(g, x)
    side.synchronize()
    for t in got[0]:
        assert t.device.index == 1 and torch.equal(t.to("cuda:0"), want[0])
    assert torch.equal(got[1].to("cuda:0"), want[1]) and torch.equal(got[2].to("cuda:0"), want[2])
    assert torch.cuda.current_device() == 0


@GPU
def test_linear_layer_leaves_what_it_does_not_take():
    """Other types, odd widths, unaligned and strided inputs, empty ones, long ones: torch's answer."""
    def same(x, w):
        assert torch.equal(plain_linear(x, w), F.linear(x, w))
    with torch.no_grad():
        same(_rnd(8, 64).float(), _rnd(16, 64).float())
        same(_rnd(8, 72), _rnd(16, 72))                        # no whole steps of 64
        same(_rnd(8, 64), _rnd(17, 64))                        # no whole pieces of columns
        same(_rnd(64 * 8 + 1)[1:].view(8, 64), _rnd(16, 64))   # not aligned
        same(_rnd(64, 8).t(), _rnd(16, 64))
        same(_rnd(0, 64), _rnd(16, 64))
        same(_rnd(64), _rnd(16, 64))
        same(_rnd(4096, 1024), _rnd(1024, 1024))
        x, w = _rnd(16, 64), _rnd(32, 64, seed=1)
        torch.testing.assert_close(plain_linear(x, w).float(), F.linear(x, w).float(), rtol=2**-6, atol=2**-4)


class _Seen(torch.Tensor):
    """A subclass that sees torch's calls by `__torch_function__` alone."""
    calls = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        _Seen.calls.append(getattr(func, "__name__", ""))
        return super().__torch_function__(func, types, args, kwargs or {})


@GPU
@pytest.mark.parametrize("which", [(True, False), (False, True), (True, True)])
def test_subclasses_with_a_torch_function(which):
    """They see torch's linear, and what comes out is one of them."""
    from deepspeedsyclsupport_amd.ops import hybrid_ops
    from deepspeedsyclsupport_amd.ops.linear import input_grad, linear, weight_grad
    x, w, go = _rnd(96, 128), _rnd(64, 128, seed=1), _rnd(96, 64, seed=2)
    sx, sw = (t.as_subclass(_Seen) if s else t for t, s in zip((x, w), which))
    for f in (plain_linear, hybrid_ops._plain, linear, lambda a, b: LinearFunction.apply(a, b, None, None)):
        _Seen.calls.clear()
        y = f(sx, sw)
        assert type(y) is _Seen and "linear" in _Seen.calls and torch.equal(y.as_subclass(torch.Tensor), F.linear(x, w))
    for f, a, b in ((input_grad, go, sw), (weight_grad, go, sx)):
        if isinstance(b, _Seen):
            _Seen.calls.clear()
            assert type(f(a, b)) is _Seen and "mm" in _Seen.calls


@GPU
@pytest.mark.parametrize("layout", [torch.strided, torch.jagged])
def test_nested_inputs(layout):
    """Sequences of unequal length in one nested tensor, which torch's linear takes."""
    from deepspeedsyclsupport_amd.ops import hybrid_ops
    from deepspeedsyclsupport_amd.ops.linear import linear
    parts, w = [_rnd(3, 128), _rnd(5, 128, seed=1)], _rnd(64, 128, seed=2)
    x = torch.nested.nested_tensor(parts, layout=layout)
    with torch.no_grad():
        for f in (plain_linear, hybrid_ops._plain, linear, lambda a, b: LinearFunction.apply(a, b, None, None)):
            y = f(x, w)
            assert y.is_nested and y.layout == layout
            for got, want in zip(y.unbind(), F.linear(x, w).unbind()):
                assert torch.equal(got, want)


@GPU
@pytest.mark.parametrize("T,W,N", [(49, 256, 512), (100, 4096, 6144), (200, 2048, 2048), (1500, 256, 256)])
def test_products_of_hybrid_decoders(T, W, N):
    """Short prompts of the hybrid decoders take the same products, longer ones and fp32 torch's."""
    from deepspeedsyclsupport_amd.ops import hybrid_ops
    x, w = _rnd(T, W, seed=1), _rnd(N, W, seed=2)
    _check(hybrid_ops.linear(x, w), x, w)
    if T <= 256:
        assert torch.equal(hybrid_ops.linear(x, w), hip_ops().narrow_gemm(x, w, True, True))
    assert torch.equal(hybrid_ops.linear(x.float(), w.float()), F.linear(x.float(), w.float()))
