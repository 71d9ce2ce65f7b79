"""Products of many tokens in tiles of 256 columns (`csrc/gemm/wide_gemm.hip`) and the layers that take them."""
import pytest
import torch

from deepspeedsyclsupport_amd.ops import linear as L
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


def _check_gated(got, x, w):
    """Both sums off by less than `size` and multiplied into each other (the gate's slope is at most 1.1), one rounding to bf16."""
    I, K = w.shape[0] // 2, w.shape[1]
    g, u = (x.double() @ w.double().t()).split(I, -1)
    size = x.double().abs() @ w.double().abs().t() * K * 2**-23
    want = torch.nn.functional.silu(g) * u
    bound = want.abs() * 2**-8 + 1.1 * size[:, :I] * u.abs() + size[:, I:] * g.abs() + 2**-20
    assert ((got.double() - want).abs() <= bound).all()


@GPU
@pytest.mark.parametrize("rows", [256, 192, 128])
@pytest.mark.parametrize("M,N,K", [(8, 8, 256), (128, 256, 256), (136, 264, 320), (200, 248, 448), (264, 520, 576), (520, 1032, 1088), (4104, 4872, 256)])
def test_tiles_at_their_edges(M, N, K, rows):
    """Every form; tiles that rows or columns do not fill; the fewest steps, and more; several tiles a workgroup; operands that are columns of
    wider matrices; the same bits each time."""
    ops = hip_ops()
    a, b = _rnd(M, K, seed=1), _rnd(N, K, seed=2)
    wide_a, wide_b = _rnd(M, K + 24, seed=3), _rnd(K, N + 16, seed=4)
    at, bt = a.t().contiguous(), b.t().contiguous()
    ops.wide_gemm_tune(rows)
    try:
        got = ops.narrow_gemm(a, b, True, True)
        _check(got, a, b)
        assert torch.equal(got, ops.narrow_gemm(a, b, True, True))
        _check(ops.narrow_gemm(a, bt, True, False), a, b)
        _check(ops.narrow_gemm(wide_a[:, 8:8 + K], wide_b[:, 8:8 + N], True, False), wide_a[:, 8:8 + K], wide_b[:, 8:8 + N].t())
        for k in (K, K - 1, K - 37, 193):   # (an inner dimension of any length)
            _check(ops.narrow_gemm(at[:k], bt[:k], False, False), a[:, :k], b[:, :k])
    finally:
        ops.wide_gemm_tune(0)


@GPU
@pytest.mark.parametrize("rows", [256, 192, 128])
@pytest.mark.parametrize("parts", [2, 3, 4])
@pytest.mark.parametrize("M,N,K", [(8, 8, 512), (136, 264, 576), (264, 520, 1088), (520, 1032, 1344), (1032, 4104, 2048)])
def test_parts_of_the_inner_dimension(M, N, K, parts, rows):
    """Every form with K in parts, the last of them shorter: the same bound, the same bits each time."""
    ops = hip_ops()
    a, b = _rnd(M, K, seed=1), _rnd(N, K, seed=2)
    ops.wide_gemm_tune(rows, parts)
    try:
        y = ops.narrow_gemm(a, b, True, True)
        dx = ops.narrow_gemm(a, b.t().contiguous(), True, False)
        dw = ops.narrow_gemm(a.t().contiguous(), b.t().contiguous(), False, False)
        for c in (y, dx, dw):
            _check(c, a, b)
        k = K - 37   # (where rows lie across it, any length)
        _check(ops.narrow_gemm(a.t().contiguous()[:k], b.t().contiguous()[:k], False, False), a[:, :k], b[:, :k])
        assert torch.equal(y, ops.narrow_gemm(a, b, True, True))
        assert torch.equal(dx, ops.narrow_gemm(a, b.t().contiguous(), True, False))
    finally:
        ops.wide_gemm_tune(0)


@GPU
@pytest.mark.parametrize("T,O,I", [(1500, 32000, 1024), (2100, 22016, 512)])
def test_gradients_of_wide_outputs_take_parts(T, O, I):
    """By the rule, in a stream of the caller's and in a graph: the sums' memory is the allocator's."""
    dy, w = _rnd(T, O, seed=3), _rnd(O, I, seed=4)
    assert hip_ops().wide_gemm_pays(T, I, O, True, False)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        dx = hip_ops().linear_input_grad(dy, w)
    torch.cuda.current_stream().wait_stream(side)
    _check(dx, dy, w.t())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        again = hip_ops().linear_input_grad(dy, w)
    for _ in range(3):
        again.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(again, dx)


@GPU
@pytest.mark.parametrize("T,O,I", [(1500, 8192, 1024), (2048, 5632, 2048), (4096, 3072, 1536), (4200, 2824, 2816), (1156, 11008, 4096), (8200, 2048, 5632), (600, 8192, 4096)])
def test_products_of_a_layer(T, O, I):
    """In one part and in two, cut between rows or columns, as the rule has it."""
    ops = hip_ops()
    x, w, go = _rnd(T, I, seed=1), _rnd(O, I, seed=2), _rnd(T, O, seed=3)
    _check(L.plain_linear(x, w), x, w)
    _check(ops.narrow_gemm(x, w, True, True), x, w)
    if O % 64 == 0:
        _check(L.input_grad(go, w), go, w.t())
        _check(ops.narrow_gemm(go, w, True, False), go, w.t())
    _check(L.weight_grad(go, x), go.t(), x.t())
    got = ops.narrow_gemm(go, x, False, False)
    _check(got, go.t(), x.t())
    assert torch.equal(got, ops.narrow_gemm(go, x, False, False))


@GPU
def test_values_that_do_not_mix():
    """Infinities and NaN stay in their rows; nothing from past the end of an operand, or of the inner dimension, comes in."""
    ops = hip_ops()
    a, b = _rnd(300, 256), _rnd(280, 256, seed=1)
    a[3, 5], a[4, 7] = float("inf"), float("nan")
    big = _rnd(300, 600, seed=2)
    big[260:] = float("nan")
    ops.wide_gemm_tune(256)
    try:
        y = ops.narrow_gemm(a, b, True, True)
        keep = [i for i in range(300) if i not in (3, 4)]
        _check(y[keep], a[keep], b)
        assert not y[3].isfinite().any() and y[4].isnan().all()
        _check(ops.narrow_gemm(big[:260, :256], b, True, True), big[:260, :256], b)
        _check(ops.narrow_gemm(big[:257, :272], big[:257, 272:600], False, False), big[:257, :272].t(), big[:257, 272:600].t())
    finally:
        ops.wide_gemm_tune(0)


@pytest.mark.parametrize("T,I,H", [(8192, 704, 256), (8192, 2816, 1024), (8192, 5632, 2048), (8192, 1376, 4096), (8192, 2752, 4096), (8192, 1408, 2048),
                                   (16384, 1408, 2048), (32768, 1376, 4096), (8192, 2048, 250), (8200, 4096, 4096)])
def test_copies_of_gated_activations_by_the_layers_around(T, I, H):
    """A copy is written exactly where the weight gradient that would read it goes to the library: by the widths of that product, a shard's too."""
    pays = hip_ops().wide_gemm_pays
    assert L.kmajor_of_gate(T, torch.bfloat16, I, H) == (not pays(H, I, T, False, False), not pays(2 * I, H, T, False, False))
    assert L.kmajor_of_gate(T, torch.bfloat16, I, None) == L.kmajor_of_gate(T, torch.bfloat16, I, I)
    assert L.kmajor_of_gate(8184, torch.bfloat16, I, H) == (False, False)
    assert L.kmajor_of_gate(T, torch.float16, I, H) == L.kmajor_of_gate(T, torch.float16, I, None) == (True, True)
    assert not pays(H + 4, I, T, False, False)   # (no whole pieces of rows: nobody's)


@GPU
@pytest.mark.parametrize("H,I,copies", [(256, 704, 2), (1024, 2816, 1), (2112, 5632, 0), (4096, 1376, 0), (2048, 1408, 1)])
def test_copies_of_gated_activations(H, I, copies):
    """Of 8192 tokens on the gate writes the copies along the tokens that the weight gradients around it will read, and only those."""
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    T = 8192
    assert sum(L.kmajor_of_gate(T, torch.bfloat16, I, H)) == copies
    x, w1, w2 = (_rnd(*s, seed=i).mul_(0.05 if i else 1).requires_grad_() for i, s in enumerate(((T, H), (2 * I, H), (H, I))))
    before = dict(L.STATS)
    act = DF.gated_activation(L.linear(x, w1), "silu", H)
    y = L.linear(act, w2)
    go = _rnd(T, H, seed=5)
    got = torch.autograd.grad(y, (x, w1, w2), go)
    if copies == 0:
        assert L.STATS == before
    xf, w1f, w2f = (t.detach().float().requires_grad_() for t in (x, w1, w2))
    h = xf @ w1f.t()
    want = torch.autograd.grad((torch.nn.functional.silu(h[:, :I]) * h[:, I:]) @ w2f.t(), (xf, w1f, w2f), go.float())
    for g, r in zip(got, want):
        assert ((g.float() - r).norm() / r.norm()).item() < 1e-2


@GPU
@pytest.mark.parametrize("around", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_copies_for_odd_widths(dtype, around):
    """A gate's copy reaches a layer whose outputs come in no whole pieces of 16 bytes."""
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    T, H, I = 8200, 252, 320
    x, w1, w2 = (_rnd(*s, seed=i).mul_(0.05 if i else 1).to(dtype).requires_grad_() for i, s in enumerate(((T, H), (2 * I, H), (H, I))))
    go = _rnd(T, H, seed=5).to(dtype)
    got = torch.autograd.grad(L.linear(DF.gated_activation(L.linear(x, w1), "silu", H if around else None), w2), (x, w1, w2), go)
    xf, w1f, w2f = (t.detach().float().requires_grad_() for t in (x, w1, w2))
    h = xf @ w1f.t()
    want = torch.autograd.grad((torch.nn.functional.silu(h[:, :I]) * h[:, I:]) @ w2f.t(), (xf, w1f, w2f), go.float())
    for g, r in zip(got, want):
        assert ((g.float() - r).norm() / r.norm()).item() < 1e-2


@pytest.mark.parametrize("T,O,I,wide", [(6464, 2048, 2048, False), (6016, 512, 8192, False), (7848, 2048, 1920, False), (7360, 4096, 1016, False),
                                        (8192, 2048, 2048, True), (8512, 2048, 2048, True), (11008, 1536, 3072, True), (13184, 1536, 3072, True)])
def test_weight_gradients_in_parts_go_where_the_narrow_tiles_do_not(T, O, I, wide):
    ops = hip_ops()
    assert ops.wide_plan(O, I, T, False)[4] > 1
    assert ops.wide_gemm_pays(O, I, T, False, False) == wide


def test_products_that_the_loop_cannot_take_are_refused():
    """At the C entries, before anything is launched: fewer steps than a tile's transfers are ahead, columns past what the stores' offsets mark."""
    import ctypes
    from deepspeedsyclsupport_amd.ops import op_builder
    hip_ops()
    lib, i64 = ctypes.CDLL(op_builder.so_path("ds_hip_ops")), ctypes.c_int64
    M, invalid = 512, 1
    for N, K, a, b in ((512, 192, 1, 1), (512, 64, 1, 0), (512, 100, 0, 0), (1 << 21, 256, 1, 1), (512, 256, 0, 1)):
        lda, ldb = K if a else M, K if b else N
        assert lib.ds_wide_gemm(None, None, None, i64(M), i64(N), i64(K), i64(lda), i64(ldb), a, b, None, None) == invalid
        if a and b:
            assert lib.ds_wide_gated(None, None, None, i64(M), i64(N // 2), i64(K), i64(lda), None) == invalid
        assert not hip_ops().wide_gemm_pays(M, N, K, bool(a), bool(b))


@pytest.mark.parametrize("T,I,K,gated", [(3939, 512, 12992, False), (8105, 256, 10624, False), (6116, 256, 15360, False), (3453, 512, 15488, False),
                                         (6116, 2048, 15360, True), (8192, 14336, 4096, True), (2392, 4096, 1024, True)])
def test_rule_of_gated_products(T, I, K, gated):
    """Gate and up of few columns by a long inner dimension pay in parts of it, which the gated product is never cut into."""
    ops = hip_ops()
    assert ops.wide_gemm_pays(T, 2 * I, K, True, True)
    assert ops.wide_gated_pays(T, I, K) == gated


@GPU
@pytest.mark.parametrize("act", ["silu", "gelu", "gelu_tanh", "relu"])
@pytest.mark.parametrize("T,I,K,dtype", [(1, 136, 256, torch.bfloat16), (16, 2816, 1024, torch.bfloat16), (300, 704, 512, torch.bfloat16),
                                         (600, 1024, 200, torch.bfloat16), (24, 64, 96, torch.float16), (24, 64, 96, torch.float32)])
def test_gated_linears_in_two_launches(T, I, K, dtype, act):
    """Where one launch does not pay, the same call makes the two that the layer made before: the same bits."""
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    x, w = _rnd(1, T, K, seed=1).to(dtype), (_rnd(2 * I, K, seed=2) * 0.1).to(dtype)
    got = DF.linear_gated(x, w, act)
    assert got is not None and torch.equal(got, DF.gated_activation(L.plain_linear(x, w), act))
    assert DF.linear_gated(x.transpose(0, 1).expand(T, 2, K), w, act) is None   # (no rows of a matrix)
    assert DF.linear_gated(x, w[:, :K - 8], act) is None and DF.linear_gated(x, w[:2 * I - 2], act) is None
    with torch.autocast("cuda"):
        assert DF.linear_gated(x, w, act) is None


@GPU
@pytest.mark.parametrize("rows", [256, 192, 128, 0])
@pytest.mark.parametrize("T,I,K", [(8, 8, 256), (200, 136, 320), (520, 392, 576), (2048, 2816, 1024), (4200, 1416, 256)])
def test_gated_products(rows, T, I, K):
    """silu of the first half of the columns times the others: what the two launches make, without the rounding between them."""
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    x, w = _rnd(T, K, seed=1), _rnd(2 * I, K, seed=2) * 0.1
    hip_ops().wide_gemm_tune(rows)
    try:
        got = DF.linear_gated(x, w)
        if not hip_ops().wide_gated_pays(T, I, K):
            assert torch.equal(got, DF.gated_activation(L.plain_linear(x, w)))
            return
        assert torch.equal(got, DF.linear_gated(x, w))
        assert torch.equal(DF.linear_gated(x.view(2, T // 2, K), w), got.view(2, T // 2, I))
    finally:
        hip_ops().wide_gemm_tune(0)
    _check_gated(got, x, w)
    with torch.enable_grad():
        assert DF.linear_gated(x.requires_grad_(), w) is None


@GPU
@pytest.mark.parametrize("T,I,K,rows,other,m,n", [
    (2391, 4096, 1024, 192, 128, 1536, 4096), (5247, 3800, 640, 256, 128, 4352, 3800), (4694, 2912, 768, 256, 192, 2816, 2912),
    (4189, 3080, 896, 192, 256, 1920, 3080), (4770, 2128, 960, 192, 128, 2880, 2128), (6782, 1400, 1152, 128, 192, 2944, 1400),
    (6301, 5632, 2048, 256, 128, 6301, 5120), (1970, 6040, 960, 256, 128, 1970, 4096), (2843, 4720, 832, 256, 192, 2843, 2688),
    (3626, 3672, 896, 192, 256, 3626, 1664), (1914, 5184, 1024, 192, 128, 1914, 3200), (2775, 3312, 1280, 128, 192, 2775, 1408)])
def test_gated_products_in_two(T, I, K, rows, other, m, n):
    """Cut between rows, or between columns, which are of either part of the weight."""
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    assert hip_ops().wide_gated_pays(T, I, K) and hip_ops().wide_plan(T, 2 * I, K, True) == [rows, other, m, 2 * n, 1]
    x, w = _rnd(T, K, seed=1), _rnd(2 * I, K, seed=2) * 0.1
    got = DF.linear_gated(x, w)
    assert torch.equal(got, DF.linear_gated(x, w))
    _check_gated(got, x, w)
