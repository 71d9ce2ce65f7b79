"""Numerics of every gfx950 kernel against a plain-PyTorch fp32 reference of the same op
(tolerances as the reference's inference_test_utils: bf16 looser, fp32 tight)."""
import math

import pytest
import torch
import torch.nn.functional as F

from deepspeedsyclsupport_amd.ops import reference as R

pytestmark = pytest.mark.gpu

TOL = {torch.float32: dict(rtol=2e-5, atol=2e-5), torch.bfloat16: dict(rtol=2e-2, atol=2e-2),
       torch.float16: dict(rtol=3e-3, atol=3e-3)}


def ops():
    from deepspeedsyclsupport_amd.ops.native import hip_ops
    return hip_ops()


@pytest.mark.parametrize("n", [1, 1000, 65536 + 3, 1 << 20])
@pytest.mark.parametrize("gdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("adamw", [True, False])
def test_adam_flat(n, gdt, adamw):
    torch.manual_seed(0)
    p = torch.randn(n, device="cuda")
    m = torch.randn(n, device="cuda").abs() * 0.1
    v = torch.rand(n, device="cuda") * 0.1
    g = torch.randn(n, device="cuda").to(gdt)
    lp = torch.empty(n, device="cuda", dtype=torch.bfloat16)
    pr, mr, vr = p.clone(), m.clone(), v.clone()
    step, lr, b1, b2, eps, wd, gs = 3, 1e-2, 0.9, 0.95, 1e-8, 0.1, 0.5
    ops().adam_flat(p, m, v, g, lp, lr, b1, b2, eps, wd, 1 - b1**step, 1 - b2**step, gs, adamw)
    R.adam_update(pr, mr, vr, g, lr, b1, b2, eps, wd, step, True, adamw, gs)
    torch.testing.assert_close(p, pr, rtol=1e-5, atol=1e-6)
    torch.testing.assert_close(m, mr, rtol=1e-5, atol=1e-6)
    torch.testing.assert_close(v, vr, rtol=1e-5, atol=1e-6)
    torch.testing.assert_close(lp.float(), p.bfloat16().float(), rtol=0, atol=0)


def test_adam_flat_misaligned():
    n = 4099
    base = torch.randn(n + 1, device="cuda")
    p = base[1:]  # 4-byte offset: forces the scalar path
    m, v = torch.zeros(n, device="cuda"), torch.zeros(n, device="cuda")
    g = torch.randn(n, device="cuda")
    pr, mr, vr = p.clone(), m.clone(), v.clone()
    ops().adam_flat(p, m, v, g, None, 1e-3, 0.9, 0.999, 1e-8, 0.0, 0.1, 0.001, 1.0, True)
    R.adam_update(pr, mr, vr, g, 1e-3, 0.9, 0.999, 1e-8, 0.0, 1)
    torch.testing.assert_close(p, pr, rtol=1e-5, atol=1e-6)


def test_adam_multi_and_fused_adam_optimizer():
    from deepspeedsyclsupport_amd.ops.adam import FusedAdam
    torch.manual_seed(1)
    shapes = [(3, 5), (1024, ), (257, 33), (64, 64)] * 10  # > 32 tensors: two launches
    ps = [torch.nn.Parameter(torch.randn(s, device="cuda")) for s in shapes]
    refs = [torch.nn.Parameter(p.detach().clone()) for p in ps]
    opt = FusedAdam(ps, lr=1e-2, weight_decay=0.01)
    ropt = torch.optim.AdamW(refs, lr=1e-2, weight_decay=0.01, eps=1e-8)
    for _ in range(3):
        for p, r in zip(ps, refs):
            g = torch.randn_like(p)
            p.grad, r.grad = g, g.clone()
        opt.step()
        ropt.step()
    for p, r in zip(ps, refs):
        torch.testing.assert_close(p, r, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("pdt,gdt,ldt", [(torch.float32, torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32, None),
                                         (torch.float32, torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16, None)])
def test_adam_multi_block_edges(pdt, gdt, ldt):
    """Sizes around a block's elements and tensors that start off the vector alignment, several in one launch; what lies between
    the tensors stays."""
    sizes, room = [1, 8, 1016, 1024, 1032, 4104, 1023, 40000], 8
    def tensors(dt, scale=1.0):
        flat = (torch.rand(sum(sizes) + room * (len(sizes) + 1), device="cuda") * scale).to(dt)
        at, out = 0, []
        for i, n in enumerate(sizes):
            at += room + (i == 5)  # (one tensor at an odd address)
            out.append(flat[at:at + n])
            at += n
        return flat, out
    fp, p = tensors(pdt)
    fm, m = tensors(pdt, 0.1)
    fv, v = tensors(pdt, 0.01)
    _, g = tensors(gdt)
    flp, lp = tensors(ldt) if ldt else (None, [])
    before = [f.clone() for f in (fp, fm, fv)]
    ref = [[t.float().clone() for t in ts] for ts in (p, m, v)]
    ops().adam_multi(p, m, v, g, lp, 1e-2, 0.9, 0.99, 1e-8, 0.1, 0.1, 0.01, 0.5, True)
    tol = dict(rtol=1e-5, atol=1e-6) if pdt == torch.float32 else dict(rtol=1e-2, atol=1e-3)
    for i in range(len(sizes)):
        pr, mr, vr = (ref[k][i] for k in range(3))
        R.adam_update(pr, mr, vr, g[i].float() * 0.5, 1e-2, 0.9, 0.99, 1e-8, 0.1, 1)
        for a, b in ((p[i], pr), (m[i], mr), (v[i], vr)):
            torch.testing.assert_close(a.float(), b, **tol)
        if ldt:
            # (half an ulp, or the other neighbour of a tie: the copy may be rounded from the unrounded update)
            torch.testing.assert_close(lp[i].float(), p[i], rtol=2.0**-11 * 1.01 if ldt == torch.float16 else 2.0**-8 * 1.01, atol=1e-7)
    used = torch.zeros_like(fp, dtype=torch.bool)
    at = 0
    for i, n in enumerate(sizes):
        at += room + (i == 5)
        used[at:at + n] = True
        at += n
    for f, b in zip((fp, fm, fv), before):
        assert torch.equal(f[~used], b[~used])


def test_lion_adagrad_lamb():
    torch.manual_seed(2)
    n = 100003
    p, m, g = torch.randn(n, device="cuda"), torch.randn(n, device="cuda") * .1, torch.randn(n, device="cuda")
    pr, mr = p.clone(), m.clone()
    ops().lion_flat(p, m, g, None, 1e-3, 0.9, 0.99, 0.1, 1.0)
    R.lion_update(pr, mr, g, 1e-3, 0.9, 0.99, 0.1)
    torch.testing.assert_close(p, pr)
    torch.testing.assert_close(m, mr)
    s = torch.rand(n, device="cuda")
    sr, pr = s.clone(), p.clone()
    ops().adagrad_flat(p, s, g, None, 1e-2, 1e-10, 0.01, 1.0)
    R.adagrad_update(pr, sr, g, 1e-2, 1e-10, 0.01)
    torch.testing.assert_close(p, pr)
    v = torch.rand(n, device="cuda") * 0.01
    pr, mr, vr = p.clone(), m.clone(), v.clone()
    c = ops().lamb_flat(p, m, v, g, None, 1e-3, 0.9, 0.999, 1e-6, 0.01, 0.1, 0.001, 1.0, 10.0, 0.01)
    trust = R.lamb_update(pr, mr, vr, g, 1e-3, 0.9, 0.999, 1e-6, 0.01, 1, True, 1.0, 10.0, 0.01)
    assert abs(float(c) - trust) < 1e-4 * max(1.0, trust)
    torch.testing.assert_close(p, pr, rtol=1e-5, atol=1e-6)


def test_sumsq_multi():
    xs = [torch.randn(n, device="cuda", dtype=dt) for n, dt in [(1000, torch.float32), (77777, torch.bfloat16),
                                                                 (5, torch.float32), (1 << 20, torch.bfloat16)]]
    ref = sum(float(x.float().pow(2).sum()) for x in xs)
    got = float(ops().sumsq_multi(xs))
    assert abs(got - ref) / ref < 1e-5


def test_sumsq_multi_many_tensors_and_edges():
    """More tensors than a launch's table holds, empty ones, starts off the vector alignment, sizes around a block's round, all
    types; each sum is of non-negative terms, so fp32 in any order is off by a few 2^-24 per term of a thread's chain."""
    sizes = [8191, 0, 8192, 8193, 1, 7, 40000, 3 << 20] * 10
    for dt in (torch.float32, torch.bfloat16, torch.float16):
        xs = [torch.randn(n + i % 3, device="cuda").to(dt)[i % 3:] for i, n in enumerate(sizes)]
        ref = sum(float(x.double().pow(2).sum()) for x in xs)
        assert abs(float(ops().sumsq_multi(xs)) - ref) / ref < 1e-5
    assert float(ops().sumsq_multi([torch.empty(0, device="cuda")])) == 0
    assert math.isinf(float(ops().sumsq_multi([torch.ones(10, device="cuda"), torch.full((3, ), math.inf, device="cuda")])))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H", [64, 1024, 4096, 5120, 8192])
@pytest.mark.parametrize("residual", [False, True])
def test_rms_norm_fwd_bwd(dtype, H, residual):
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    torch.manual_seed(3)
    rows = 37
    x = torch.randn(rows, H, device="cuda", dtype=dtype, requires_grad=True)
    r = torch.randn(rows, H, device="cuda", dtype=dtype, requires_grad=True) if residual else None
    w = (1 + 0.1 * torch.randn(H, device="cuda", dtype=dtype)).requires_grad_(True)
    out = DF.rms_norm(x, w, 1e-5, r)
    y = out[0] if residual else out
    xf = x.detach().float().requires_grad_(True)
    rf = r.detach().float().requires_grad_(True) if residual else None
    wf = w.detach().float().requires_grad_(True)
    h = xf + rf if residual else xf
    yr = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-5) * wf
    torch.testing.assert_close(y.float(), yr, **TOL[dtype])
    gy = torch.randn_like(yr)
    loss = (y.float() * gy).sum() + ((out[1].float() * gy).sum() if residual else 0)
    loss.backward()
    lr_ = (yr * gy).sum() + ((h * gy).sum() if residual else 0)
    lr_.backward()
    torch.testing.assert_close(x.grad.float(), xf.grad, **TOL[dtype])
    tol = dict(rtol=5e-2, atol=5e-1) if dtype == torch.bfloat16 else dict(rtol=1e-4, atol=1e-3)
    torch.testing.assert_close(w.grad.float(), wf.grad, **tol)
    if residual:
        torch.testing.assert_close(r.grad.float(), rf.grad, **TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H", [768, 1024, 4096, 5120, 8192])
def test_layer_norm_fwd_bwd(dtype, H):
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    torch.manual_seed(4)
    x = torch.randn(33, H, device="cuda", dtype=dtype, requires_grad=True)
    g = (1 + 0.1 * torch.randn(H, device="cuda", dtype=dtype)).requires_grad_(True)
    b = (0.1 * torch.randn(H, device="cuda", dtype=dtype)).requires_grad_(True)
    y = DF.layer_norm(x, g, b, 1e-5)
    xf, gf, bf = [t.detach().float().requires_grad_(True) for t in (x, g, b)]
    yr = F.layer_norm(xf, (H, ), gf, bf, 1e-5)
    torch.testing.assert_close(y.float(), yr, **TOL[dtype])
    gy = torch.randn_like(yr)
    (y.float() * gy).sum().backward()
    (yr * gy).sum().backward()
    torch.testing.assert_close(x.grad.float(), xf.grad, **TOL[dtype])
    tol = dict(rtol=5e-2, atol=5e-1) if dtype == torch.bfloat16 else dict(rtol=1e-4, atol=1e-3)
    torch.testing.assert_close(g.grad.float(), gf.grad, **tol)
    torch.testing.assert_close(b.grad.float(), bf.grad, **tol)


@pytest.mark.parametrize("H", [1032, 2048, 5120])
@pytest.mark.parametrize("kind", ["rms", "ln"])
def test_norm_backward_many_rows(kind, H):
    """More rows than persistent blocks (every block walks several rows, the column partials of all blocks are
    summed) and a width that is not a multiple of the block's 2048-element step."""
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    torch.manual_seed(6)
    rows = 2100
    x = torch.randn(rows, H, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    g = (1 + 0.1 * torch.randn(H, device="cuda", dtype=torch.bfloat16)).requires_grad_(True)
    b = (0.1 * torch.randn(H, device="cuda", dtype=torch.bfloat16)).requires_grad_(True)
    xf, gf, bf = [t.detach().float().requires_grad_(True) for t in (x, g, b)]
    if kind == "rms":
        y = DF.rms_norm(x, g, 1e-5)
        yr = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-5) * gf
    else:
        y = DF.layer_norm(x, g, b, 1e-5)
        yr = F.layer_norm(xf, (H, ), gf, bf, 1e-5)
    gy = torch.randn_like(yr).bfloat16().float()
    (y.float() * gy).sum().backward()
    (yr * gy).sum().backward()
    torch.testing.assert_close(x.grad.float(), xf.grad, **TOL[torch.bfloat16])
    # column sums over 2100 rows of bf16-rounded products: compare against the fp32 sum with a relative bound
    scale = float(gf.grad.abs().max())
    assert float((g.grad.float() - gf.grad).abs().max()) <= 2e-2 * scale
    if kind == "ln":
        assert float((b.grad.float() - bf.grad).abs().max()) <= 2e-2 * float(bf.grad.abs().max())


@pytest.mark.parametrize("act", ["silu", "gelu", "gelu_tanh", "relu"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gated_act(act, dtype):
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    torch.manual_seed(5)
    gu = torch.randn(19, 2 * 1376, device="cuda", dtype=dtype, requires_grad=True)
    y = DF.gated_activation(gu, act)
    gf = gu.detach().float().requires_grad_(True)
    a, u = gf.chunk(2, -1)
    fn = {"silu": F.silu, "gelu": F.gelu, "gelu_tanh": lambda t: F.gelu(t, approximate="tanh"), "relu": F.relu}[act]
    yr = fn(a) * u
    torch.testing.assert_close(y.float(), yr, **TOL[dtype])
    gy = torch.randn_like(yr)
    (y.float() * gy).sum().backward()
    (yr * gy).sum().backward()
    torch.testing.assert_close(gu.grad.float(), gf.grad, **TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_bias_act(dtype):
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    x = torch.randn(13, 3072, device="cuda", dtype=dtype, requires_grad=True)
    b = torch.randn(3072, device="cuda", dtype=dtype, requires_grad=True)
    y = DF.bias_activation(x, b, "gelu_tanh")
    xf, bf = x.detach().float().requires_grad_(True), b.detach().float().requires_grad_(True)
    yr = F.gelu(xf + bf, approximate="tanh")
    torch.testing.assert_close(y.float(), yr, **TOL[dtype])
    gy = torch.randn_like(yr)
    (y.float() * gy).sum().backward()
    (yr * gy).sum().backward()
    torch.testing.assert_close(x.grad.float(), xf.grad, **TOL[dtype])


@pytest.mark.parametrize("token_major", [False, True])
@pytest.mark.parametrize("hq,hk", [(8, 8), (8, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_qkv_rope_split(hq, hk, dtype, token_major):
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    torch.manual_seed(6)
    B, S, D = 2, 33, 128
    cos, sin = R.rope_tables(128, D, device="cuda")
    qkv = torch.randn(B, S, hq + 2 * hk, D, device="cuda", dtype=dtype, requires_grad=True)
    q, k, v = DF.qkv_rope_split(qkv, cos, sin, hq, hk, token_major=token_major)
    assert q.transpose(1, 2).is_contiguous() == token_major
    qf = qkv.detach().float().requires_grad_(True)
    qq, kk, vv = qf.split([hq, hk, hk], dim=2)
    pos = torch.arange(S, device="cuda")
    qr = R.apply_rope_half(qq, cos, sin, pos).transpose(1, 2)
    kr = R.apply_rope_half(kk, cos, sin, pos).transpose(1, 2)
    vr = vv.transpose(1, 2)
    for a, b in ((q, qr), (k, kr), (v, vr)):
        torch.testing.assert_close(a.float(), b, **TOL[dtype])
    gs = [torch.randn_like(t) for t in (qr, kr, vr)]
    sum((a.float() * g).sum() for a, g in zip((q, k, v), gs)).backward()
    sum((a * g).sum() for a, g in zip((qr, kr, vr), gs)).backward()
    torch.testing.assert_close(qkv.grad.float(), qf.grad, **TOL[dtype])


@pytest.mark.parametrize("interleaved", [False, True])
def test_rope_inplace(interleaved):
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    B, S, H, D = 2, 17, 4, 64
    cos, sin = R.rope_tables(64, D, device="cuda")
    x = torch.randn(B, S, H, D, device="cuda")
    ref = DF.apply_rotary_pos_emb(x.clone().cpu(), cos.cpu(), sin.cpu(), interleaved=interleaved)
    got = DF.apply_rotary_pos_emb(x.clone(), cos, sin, interleaved=interleaved)
    torch.testing.assert_close(got.cpu(), ref, rtol=1e-5, atol=1e-5)
    back = DF.apply_rotary_pos_emb(got.clone(), cos, sin, interleaved=interleaved, inverse=True)
    torch.testing.assert_close(back, x, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("T,W,V", [(1, 8, 3), (1023, 264, 40), (1025, 2048, 5000), (4096, 2056, 700), (2050, 64, 1), (4097, 64, 300)])
def test_embedding_gradient(T, W, V):
    """Ids that repeat once, often, always, around the sizes of a round of ids and a slice of columns, and one token more than the
    kernel takes; for odd T dy starts 2 bytes off. fp32 sums of n bf16 rows are off by at most n 2^-24 of their magnitudes' sum, the result by 2^-9 of itself."""
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    ids = torch.randint(0, V, (1, T), device="cuda")
    w = torch.randn(V, W, device="cuda").bfloat16().requires_grad_(True)
    dy = torch.randn(T * W + T % 2, device="cuda").bfloat16()[T % 2:].view(1, T, W)
    y = DF.embedding(ids, w)
    assert torch.equal(y, w.detach()[ids[0]][None])
    y.backward(dy)
    ref = torch.zeros(V, W, device="cuda", dtype=torch.float64).index_add_(0, ids[0], dy[0].double())
    if T <= 4096:
        err = T * 2.0**-24 * torch.zeros_like(ref).index_add_(0, ids[0], dy[0].double().abs())
        assert ((w.grad.double() - ref).abs() <= 2.0**-8 * ref.abs() + err).all()
    else:
        torch.testing.assert_close(w.grad.double(), ref, rtol=0.1, atol=0.5)


@pytest.mark.parametrize("W", [8, 248, 264, 2304])
@pytest.mark.parametrize("counts", [[1], [63, 64, 65, 1, 0, 8], [4096], [71, 1500, 2500, 7]])
def test_embedding_gradient_of_ids_with_many_rows(W, counts):
    """Ids with fewer rows than a workgroup keeps to itself, as many, and more, which several add up, 256 columns each: bounds as above,
    the same bits every time."""
    from deepspeedsyclsupport_amd.ops.native import hip_ops
    g = torch.Generator(device="cuda").manual_seed(sum(counts) + W)
    ids = torch.repeat_interleave(torch.arange(len(counts), device="cuda"), torch.tensor(counts, device="cuda"))
    ids = ids[torch.randperm(ids.numel(), device="cuda", generator=g)]
    dy = torch.randn(ids.numel(), W, device="cuda", generator=g).bfloat16()
    got = hip_ops().embed_grad(dy, ids, len(counts) + 1)
    ref = torch.zeros(got.shape, device="cuda", dtype=torch.float64).index_add_(0, ids, dy.double())
    err = max(counts) * 2.0**-24 * torch.zeros_like(ref).index_add_(0, ids, dy.double().abs())
    assert ((got.double() - ref).abs() <= 2.0**-8 * ref.abs() + err).all()
    assert torch.equal(got, hip_ops().embed_grad(dy, ids, len(counts) + 1))


@pytest.mark.parametrize("V", [32000, 50257, 1000])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_cross_entropy(V, dtype):
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    torch.manual_seed(7)
    N = 67
    logits = (3 * torch.randn(N, V, device="cuda")).to(dtype).requires_grad_(True)
    labels = torch.randint(0, V, (N, ), device="cuda")
    labels[3] = -100
    loss = DF.cross_entropy(logits, labels, inplace_backward=False)
    lf = logits.detach().float().requires_grad_(True)
    lr_ = F.cross_entropy(lf, labels, ignore_index=-100)
    torch.testing.assert_close(loss.float(), lr_, rtol=1e-4, atol=1e-4)
    loss.backward()
    lr_.backward()
    torch.testing.assert_close(logits.grad.float(), lf.grad, **TOL[dtype])


@pytest.mark.parametrize("N,ignored", [(1, 0), (67, 20), (67, 67), (2500, 7), (0, 0), (65536, 9), (65537, 9)])
def test_cross_entropy_mean_is_that_of_the_rows(N, ignored):
    """The fused mean against the rows' own losses: the same numbers, added up in another order; its gradient too. A label that no
    row of the vocabulary has counts but weighs nothing; the result can be changed in place."""
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    V = 264
    x = torch.randn(N, V, device="cuda")
    labels = torch.randint(0, V, (N, ), device="cuda")
    labels[:ignored] = -7
    if N > 60 and ignored < 60:
        labels[60] = V + 3
    a, b = (x.clone().requires_grad_(True) for _ in range(2))
    rows = DF.cross_entropy(a, labels, ignore_index=-7, label_smoothing=0.1, reduction="none", inplace_backward=False)
    want = rows.sum() / (labels != -7).sum().clamp(min=1)
    got = DF.cross_entropy(b, labels, ignore_index=-7, label_smoothing=0.1, inplace_backward=False)
    torch.testing.assert_close(got, want, rtol=1e-6, atol=0)
    got /= 2
    (want / 2 * 3).backward()
    (got * 3).backward()
    torch.testing.assert_close(b.grad, a.grad, rtol=1e-6, atol=1e-9)


# ------------------------------------------------------------------------------------------------ inference kernels
def _paged_setup(B, Hk, D, BS, lens, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    maxb = max((L + BS - 1) // BS for L in lens)
    nb = B * maxb + 3
    kc = torch.randn(nb, Hk, BS, D, device="cuda", generator=g).bfloat16()
    vc = torch.randn(nb, Hk, BS, D, device="cuda", generator=g).bfloat16()
    perm = torch.randperm(nb, device="cuda", generator=g)[:B * maxb].to(torch.int32).view(B, maxb)
    return kc, vc, perm.contiguous(), maxb


def _paged_ref(q, kc, vc, bt, lens, scale, alibi=None, window=0):
    B, Hq, D = q.shape
    Hk, BS = kc.shape[1], kc.shape[2]
    out = torch.empty(B, Hq, D, device="cuda")
    for b in range(B):
        L = lens[b]
        nblk = (L + BS - 1) // BS
        ids = bt[b, :nblk].long()
        k = kc[ids].float().transpose(0, 1).reshape(Hk, -1, D)[:, :L]
        v = vc[ids].float().transpose(0, 1).reshape(Hk, -1, D)[:, :L]
        k, v = k.repeat_interleave(Hq // Hk, 0), v.repeat_interleave(Hq // Hk, 0)
        s = torch.einsum("hd,htd->ht", q[b].float(), k) * scale
        if alibi is not None:
            s = s + alibi[:, None] * (torch.arange(L, device="cuda") - (L - 1)).float()[None]
        if window:
            s[:, :max(0, L - window)] = float("-inf")
        out[b] = torch.einsum("ht,htd->hd", s.softmax(-1), v)
    return out


@pytest.mark.parametrize("D", [64, 80, 96, 128, 256])
@pytest.mark.parametrize("hq,hk", [(8, 8), (32, 8), (8, 1)])
@pytest.mark.parametrize("lens", [[1, 7, 64], [300, 2049, 5000]])
def test_paged_decode(D, hq, hk, lens):
    B, BS = len(lens), 64
    kc, vc, bt, maxb = _paged_setup(B, hk, D, BS, lens)
    q = torch.randn(B, hq, D, device="cuda").bfloat16()
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    scale = 1 / math.sqrt(D)
    out = ops().paged_decode(q, kc, vc, bt, sl, max(lens), scale, None, 0)
    ref = _paged_ref(q, kc, vc, bt, lens, scale)
    torch.testing.assert_close(out.float(), ref, rtol=2e-2, atol=2e-2)


def test_paged_decode_alibi_window_and_capacity():
    B, hq, hk, D, BS = 3, 8, 8, 128, 16
    lens = [5, 40, 100]
    kc, vc, bt, maxb = _paged_setup(B, hk, D, BS, lens, seed=3)
    q = torch.randn(B, hq, D, device="cuda").bfloat16()
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    from deepspeedsyclsupport_amd.inference.model_implementations.transformer import alibi_slopes
    al = alibi_slopes(hq).cuda()
    # max_len = full block-table capacity (the HIP-graph decode path): empty splits must not perturb the result
    out = ops().paged_decode(q, kc, vc, bt, sl, maxb * BS, 0.1, al, 32)
    ref = _paged_ref(q, kc, vc, bt, lens, 0.1, al, 32)
    torch.testing.assert_close(out.float(), ref, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("hq,hk", [(3, 3), (10, 5), (9, 3), (16, 2)])
@pytest.mark.parametrize("D,BS,window", [(64, 24, 0), (128, 16, 100), (96, 64, 0)])
def test_paged_decode_edges_of_key_groups(hq, hk, D, BS, window):
    """Contexts around a wave's group, a workgroup's round and the length from which a sequence is split, one to eight heads a
    group, a block size that is no power of two. Probabilities stay in fp32: against fp64 the result is off by its own
    rounding (2^-9) and that of the fp32 sums (a few hundred terms of at most 5, 2^-24 each)."""
    lens = [1, 15, 16, 17, 127, 128, 129, 768, 769, 1030]
    kc, vc, bt, maxb = _paged_setup(len(lens), hk, D, BS, lens, seed=5)
    q = torch.randn(len(lens), hq, D, device="cuda").bfloat16()
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    room = torch.full((len(lens) + 1, hq, D), 7.0, device="cuda", dtype=torch.bfloat16)
    for max_len in (max(lens), maxb * BS):
        out = ops().paged_decode(q, kc, vc, bt, sl, max_len, D**-0.5, None, window, room[:-1])
        ref = _paged_ref(q.double(), kc.double(), vc.double(), bt, lens, D**-0.5, None, window)
        assert ((out.double() - ref).abs() <= 2.0**-8 * ref.abs() + 2e-4).all()
        assert torch.equal(out, room[:-1]) and (room[-1] == 7).all()


@pytest.mark.parametrize("D,rot,interleaved", [(128, 128, False), (128, 32, False), (64, 64, True), (80, 16, False), (256, 0, False)])
@pytest.mark.parametrize("window", [0, 40])
def test_paged_decode_step_equals_append_and_attention(D, rot, interleaved, window):
    """A step that turns and appends its own keys, against the two kernels: the cache to the bit of rounding, its other rows
    untouched, and the attention of what they made."""
    hq, hk, BS, lens = 8, 2, 16, [1, 2, 16, 17, 113, 129, 900, 1500]   # with the step's own key
    kc, vc, bt, maxb = _paged_setup(len(lens), hk, D, BS, lens, seed=6)
    qkv = torch.randn(len(lens), (hq + 2 * hk) * D, device="cuda").bfloat16()
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    pos, seqs = sl - 1, torch.arange(len(lens), dtype=torch.int32, device="cuda")
    tables = R.rope_tables(2048, rot, device="cuda") if rot else (None, None)
    k2, v2 = kc.clone(), vc.clone()
    q = ops().qkv_rope_append(qkv, *tables, pos, k2, v2, bt, pos, 1, hq, hk, rot, interleaved, False, seqs)[0]
    want = ops().paged_decode(q, k2, v2, bt, sl, maxb * BS, D**-0.5, None, window)
    got = ops().paged_decode_step(qkv, *tables, pos, kc, vc, bt, sl, maxb * BS, D**-0.5, None, window, hq, rot, interleaved)
    assert torch.equal(vc, v2)
    torch.testing.assert_close(kc.float(), k2.float(), rtol=2.0**-7, atol=0)  # (a * c - b * s may be contracted either way)
    torch.testing.assert_close(got.float(), want.float(), rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("D,hq,hk", [(128, 4, 4), (128, 16, 8), (128, 32, 8), (128, 40, 5), (256, 3, 3), (256, 12, 6), (256, 16, 2)])
def test_paged_decode_values_in_parts(D, hq, hk):
    """Up to 128 (sequence, key head) two workgroups share a head's values, one more of them and none does (bounds as above); the
    step's key and value are written once."""
    for B in (128 // hk, 128 // hk + 1):
        BS, lens = 32, [(1, 15, 16, 17, 127, 129, 330, 400, 513, 700, 768)[i % 11] for i in range(B)]
        kc, vc, bt, maxb = _paged_setup(B, hk, D, BS, lens, seed=8)
        sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
        pos, seqs = sl - 1, torch.arange(B, dtype=torch.int32, device="cuda")
        tables = R.rope_tables(1024, D, device="cuda")
        qkv = torch.randn(B, (hq + 2 * hk) * D, device="cuda", generator=torch.Generator(device="cuda").manual_seed(9)).bfloat16()
        k2, v2 = kc.clone(), vc.clone()
        q = ops().qkv_rope_append(qkv, *tables, pos, k2, v2, bt, pos, 1, hq, hk, D, False, False, seqs)[0]
        ref = _paged_ref(q.double(), k2.double(), v2.double(), bt, lens, D**-0.5)
        out = ops().paged_decode(q, k2, v2, bt, sl, max(lens), D**-0.5, None, 0)
        assert ((out.double() - ref).abs() <= 2.0**-8 * ref.abs() + 2e-4).all()
        got = ops().paged_decode_step(qkv, *tables, pos, kc, vc, bt, sl, max(lens), D**-0.5, None, 0, hq, D, False)
        assert torch.equal(vc, v2)
        torch.testing.assert_close(got.float(), out.float(), rtol=1e-2, atol=1e-2)


def test_kv_append():
    B, n, hk, D, BS = 3, 5, 4, 128, 16
    kc, vc, bt, maxb = _paged_setup(B, hk, D, BS, [64, 64, 64])
    k = torch.randn(B, n, hk, D, device="cuda").bfloat16()
    v = torch.randn(B, n, hk, D, device="cuda").bfloat16()
    start = torch.tensor([0, 14, 40], dtype=torch.int32, device="cuda")
    kr, vr = kc.clone(), vc.clone()
    ops().kv_append(k, v, kc, vc, bt, start)
    for b in range(B):
        for j in range(n):
            t = int(start[b]) + j
            blk = int(bt[b, t // BS])
            kr[blk, :, t % BS] = k[b, j]
            vr[blk, :, t % BS] = v[b, j]
    assert torch.equal(kc, kr) and torch.equal(vc, vr)


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("sym", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_quantize_roundtrip(bits, sym, dtype):
    from deepspeedsyclsupport_amd.ops.quantizer.quantizer import _ref_dequantize, _ref_quantize
    torch.manual_seed(0)
    gs = 128
    x = (torch.randn(64 * gs, device="cuda") * 3).to(dtype)
    q, s, z = ops().quantize(x, gs, bits, not sym, False, 0)
    qr, sr, zr = _ref_quantize(x.cpu(), gs, bits, not sym)
    torch.testing.assert_close(s.cpu(), sr, rtol=1e-5, atol=1e-7)
    d = ops().dequantize(q, s, z if not sym else None, x.numel(), gs, bits, torch.float32)
    dr = _ref_dequantize(qr, sr, zr, x.numel(), gs, bits, torch.float32)
    # kernel and reference may round exact .5 ties differently: allow one quantisation step
    step = s.repeat_interleave(gs).cpu()
    assert ((d.cpu() - dr).abs() <= step * 1.01 + 1e-6).all()
    assert ((x.float() - d).abs() <= s.repeat_interleave(gs) * 0.51 + 1e-5).all()


def test_dequant_reduce():
    from deepspeedsyclsupport_amd.ops.quantizer import quantize
    torch.manual_seed(0)
    gs, n, k = 256, 256 * 32, 4
    xs = [torch.randn(n, device="cuda") for _ in range(k)]
    qts = [quantize(x, gs, 8) for x in xs]
    q = torch.cat([t.data for t in qts])
    s = torch.cat([t.scales for t in qts])
    out = ops().dequant_reduce(q, s, k, gs, 0.25, torch.float32)
    ref = sum(x for x in xs) * 0.25
    torch.testing.assert_close(out, ref, rtol=0, atol=k * 0.25 * float(s.max()) * 0.51)


@pytest.fixture(params=["mfma", "valu", "auto"])
def skinny_path(request):
    ops().skinny_set_path({"auto": 0, "valu": 1, "mfma": 2}[request.param])
    yield request.param
    ops().skinny_set_path(0)


@pytest.mark.parametrize("M", [1, 2, 3, 5, 8, 12, 16])
@pytest.mark.parametrize("N,K", [(4096, 4096), (333, 11008), (7, 64), (100, 256), (50, 768)])
def test_skinny_gemm_plain(M, N, K, skinny_path):
    if M > 8 and (K % 256 or skinny_path == "valu"):
        pytest.skip("rows > 8 need the MFMA kernel (K % 256 == 0)")
    torch.manual_seed(0)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * 0.02).bfloat16()
    b = torch.randn(N, device="cuda").bfloat16()
    add = torch.randn(M, N, device="cuda").bfloat16()
    y = ops().skinny_gemm(x, w, b, add, 0, False, 0, None, None, 0.0, None)
    ref = x.float() @ w.float().t() + b.float() + add.float()
    torch.testing.assert_close(y.float(), ref, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("M", [1, 4, 8, 16])
@pytest.mark.parametrize("with_res", [False, True])
@pytest.mark.parametrize("K", [4096, 8192])
def test_skinny_gemm_rmsnorm(M, with_res, K, skinny_path):
    if M > 8 and skinny_path == "valu":
        pytest.skip("rows > 8 need the MFMA kernel")
    torch.manual_seed(1)
    N, eps = 1000, 1e-5
    x = torch.randn(M, K, device="cuda").bfloat16()
    r = torch.randn(M, K, device="cuda").bfloat16() if with_res else None
    nw = (1 + 0.1 * torch.randn(K, device="cuda")).bfloat16()
    w = (torch.randn(N, K, device="cuda") * 0.02).bfloat16()
    res_out = torch.empty_like(x)
    y = ops().skinny_gemm(x, w, None, None, 1, False, 0, r, nw, eps, res_out)
    y2 = ops().skinny_gemm(x, w, None, None, 1, False, 0, r, nw, eps, None)  # LM-head form: no residual output
    torch.testing.assert_close(y2, y, rtol=0, atol=0)
    h = (x.float() + (r.float() if with_res else 0)).bfloat16().float()
    normed, _ = R.rms_norm(h, nw.float(), eps)
    torch.testing.assert_close(y.float(), normed @ w.float().t(), rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(res_out.float(), h.bfloat16().float(), rtol=0, atol=0)


@pytest.mark.parametrize("act", ["silu", "gelu", "relu"])
@pytest.mark.parametrize("M", [1, 3, 8, 16])
def test_skinny_gemm_gated(act, M, skinny_path):
    if M > 8 and skinny_path == "valu":
        pytest.skip("rows > 8 need the MFMA kernel")
    from deepspeedsyclsupport_amd.ops.transformer.functional import ACT_CODES
    torch.manual_seed(2)
    I, K = 1376, 4096
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(2 * I, K, device="cuda") * 0.02).bfloat16()
    b = torch.randn(2 * I, device="cuda").bfloat16()
    y = ops().skinny_gemm(x, w, b, None, 0, True, ACT_CODES[act], None, None, 0.0, None)
    gu = (x.float() @ w.float().t() + b.float()).bfloat16().float()
    ref = R.gated_act(gu, ACT_CODES[act])
    assert y.shape == (M, I)
    torch.testing.assert_close(y.float(), ref, rtol=2e-2, atol=3e-2)


@pytest.mark.parametrize("rot,interleaved", [(128, False), (32, False), (64, True), (0, False)])
def test_qkv_rope_append(rot, interleaved):
    torch.manual_seed(3)
    B, n, hq, hk, D, BS = 2, 5, 8, 2, 128, 16
    kc, vc, bt, maxb = _paged_setup(B, hk, D, BS, [64, 64])
    qkv = torch.randn(B * n, (hq + 2 * hk) * D, device="cuda").bfloat16()
    start = torch.tensor([3, 20], dtype=torch.int32, device="cuda")
    pos = (start[:, None] + torch.arange(n, device="cuda", dtype=torch.int32)[None]).reshape(-1).contiguous()
    cos, sin = R.rope_tables(256, max(rot, 2), device="cuda")
    kr, vr = kc.clone(), vc.clone()
    q, k, v = ops().qkv_rope_append(qkv, cos if rot else None, sin if rot else None, pos, kc, vc, bt, start, n, hq,
                                    hk, rot, interleaved, True)
    x = qkv.view(B, n, hq + 2 * hk, D).float()
    qr, krr, vrr = x[:, :, :hq].clone(), x[:, :, hq:hq + hk].clone(), x[:, :, hq + hk:].clone()
    p = pos.view(B, n).long()
    if rot:
        def rope(t):
            if interleaved:
                c, s = cos[p][:, :, None, :], sin[p][:, :, None, :]
                a, b_ = t[..., 0:rot:2].clone(), t[..., 1:rot:2].clone()
                t[..., 0:rot:2], t[..., 1:rot:2] = a * c - b_ * s, b_ * c + a * s
                return t
            return R.apply_rope_half(t, cos, sin, p)
        qr, krr = rope(qr), rope(krr)
    torch.testing.assert_close(q.float().view(B, n, hq, D), qr, rtol=1e-2, atol=1e-2)
    torch.testing.assert_close(k.float().view(B, n, hk, D), krr, rtol=1e-2, atol=1e-2)
    torch.testing.assert_close(v.float().view(B, n, hk, D), vrr, rtol=0, atol=0)
    for b in range(B):
        for j in range(n):
            t = int(start[b]) + j
            blk = int(bt[b, t // BS])
            kr[blk, :, t % BS] = k.view(B, n, hk, D)[b, j]
            vr[blk, :, t % BS] = v.view(B, n, hk, D)[b, j]
    assert torch.equal(kc, kr) and torch.equal(vc, vr)


def _unpack_mask(packed, shape):
    bits = (packed.long().unsqueeze(-1) >> torch.arange(8, device=packed.device)) & 1
    return bits.reshape(shape).bool()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("p", [0.1, 0.5])
def test_fused_dropout(dt, p):
    """residual + dropout(x + bias) vs the same math in fp32 with the kernel's own mask; the mask's keep rate; the
    backward regenerates the identical mask from the seed (no stored mask)."""
    torch.manual_seed(0)
    rows, C = 1000, 1024
    x = torch.randn(rows, C, device="cuda").to(dt)
    b = torch.randn(C, device="cuda").to(dt)
    r = torch.randn(rows, C, device="cuda").to(dt)
    y, packed = ops().dropout_fwd(x, b, r, p, 1234, 0, True)
    keep = _unpack_mask(packed, (rows, C))
    rate = keep.float().mean().item()
    assert abs(rate - (1 - p)) < 0.01, rate
    ref = r.float() + torch.where(keep, (x.float() + b.float()) / (1 - p), torch.zeros_like(x.float()))
    torch.testing.assert_close(y.float(), ref, **TOL[dt])
    dy = torch.randn(rows, C, device="cuda").to(dt)
    dx = ops().dropout_bwd(dy, p, 1234, 0)
    ref_dx = torch.where(keep, dy.float() / (1 - p), torch.zeros_like(dy.float()))
    torch.testing.assert_close(dx.float(), ref_dx, **TOL[dt])
    # a different seed gives a different mask; same seed the same one
    _, p2 = ops().dropout_fwd(x, None, None, p, 1235, 0, True)
    _, p3 = ops().dropout_fwd(x, None, None, p, 1234, 0, True)
    assert not torch.equal(p2, packed) and torch.equal(p3, packed)


def test_dropout_autograd_and_checkpoint_replay():
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    torch.manual_seed(1)
    # positive x and b: x + b is never 0, so y0 != 0 identifies the kept elements
    x = (torch.rand(64, 256, device="cuda") + 0.1).bfloat16().requires_grad_(True)
    b = (torch.rand(256, device="cuda") + 0.1).bfloat16().requires_grad_(True)
    r = torch.randn(64, 256, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    torch.manual_seed(7)
    y0 = DF.dropout(x, 0.2, True, bias=b)
    keep = y0 != 0
    torch.manual_seed(7)
    y = DF.dropout(x, 0.2, True, bias=b, residual=r)
    torch.testing.assert_close(y.float(), (r.float() + y0.float()), rtol=2e-2, atol=2e-2)
    y.float().sum().backward()
    torch.testing.assert_close(x.grad.float(), keep.float() / 0.8, rtol=1e-2, atol=1e-2)
    torch.testing.assert_close(b.grad.float(), (keep.float() / 0.8).sum(0), rtol=2e-2, atol=2e-1)
    assert torch.equal(r.grad, torch.ones_like(r))
    torch.manual_seed(7)
    y2 = torch.utils.checkpoint.checkpoint(lambda t: DF.dropout(t, 0.2, True, bias=b, residual=r), x,
                                           use_reentrant=False)
    assert torch.equal(y, y2)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
def test_spatial_nhwc_bias_add(dt):
    from deepspeedsyclsupport_amd.ops import spatial
    torch.manual_seed(2)
    x = torch.randn(2, 320, 16, 16, device="cuda").to(dt).to(memory_format=torch.channels_last)
    o = torch.randn(2, 320, 16, 16, device="cuda").to(dt).to(memory_format=torch.channels_last)
    b, ob = torch.randn(320, device="cuda").to(dt), torch.randn(320, device="cuda").to(dt)
    bb, obb = b.view(1, -1, 1, 1).float(), ob.view(1, -1, 1, 1).float()
    torch.testing.assert_close(spatial.nhwc_bias_add(x, b).float(), x.float() + bb, **TOL[dt])
    torch.testing.assert_close(spatial.nhwc_bias_add_add(x, b, o).float(), x.float() + bb + o.float(), **TOL[dt])
    torch.testing.assert_close(spatial.nhwc_bias_add_bias_add(x, b, o, ob).float(),
                               x.float() + bb + o.float() + obb, **TOL[dt])


@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 16])
@pytest.mark.parametrize("N,K,gs", [(1, 64, 64), (13, 4096, 64), (4096, 11008, 64), (1000, 14336, 128), (300, 57344, 64),
                                    (77, 320, 64), (50, 4160, 64), (129, 2048, 512), (64, 1024, 1024)])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("path", ["valu", "mfma"])
def test_skinny_int8_gemv(M, N, K, gs, bias, path):
    """Weight-only int8 decode GEMV (fused group dequant) vs an fp32 GEMM on the dequantised weight: the VALU stream
    over the row-major weight (<= 8 rows) and the MFMA stream over the pre-shuffled weight (<= 16 rows)."""
    from deepspeedsyclsupport_amd.ops.int8_gemv import preshuffle
    from deepspeedsyclsupport_amd.ops.quantizer import dequantize, quantize
    torch.manual_seed(N + K)
    w = (torch.randn(N, K, device="cuda") * 0.02).bfloat16()
    qt = quantize(w, group_size=gs, bits=8, symmetric=True)
    x = torch.randn(M, K, device="cuda").bfloat16()
    b = torch.randn(N, device="cuda").bfloat16() if bias else None
    if path == "valu":
        if M > 8:
            pytest.skip("VALU stream is for <= 8 rows")
        y = ops().skinny_i8(x, qt.data, qt.scales, b, N, gs)
    else:
        qsh, ssh = preshuffle(qt.data.view(N, K), qt.scales, gs)
        y = ops().skinny_i8_sh(x, qsh, ssh, b, N, gs)
    ref = x.float() @ dequantize(qt, torch.float32).t()
    if bias:
        ref = ref + b.float()
    torch.testing.assert_close(y.float(), ref, rtol=2e-2, atol=2e-2 * max(1.0, ref.abs().max().item()))


def test_skinny_int8_mfma_workspace_reuse_and_graph():
    """The MFMA path's split-K workspace re-zeroes itself: repeated calls, interleaved shapes and a HIP-graph replay
    all give the first call's result; Int8Weight.linear routes decode sizes to it and prefill to dequant + GEMM."""
    from deepspeedsyclsupport_amd.ops.int8_gemv import Int8Weight
    torch.manual_seed(3)
    mats = []
    for N, K in ((4096, 4096), (11008, 4096), (333, 8192)):
        wt = Int8Weight((torch.randn(N, K, device="cuda") * 0.02).bfloat16(), 64)
        mats.append((wt, torch.randn(8, K, device="cuda").bfloat16()))
    first = [wt.linear(x) for wt, x in mats]
    for wt, x in mats:  # native bf16 dequant from the shuffled layout == host un-shuffle + dequant
        torch.testing.assert_close(wt.materialize().float(), wt.materialize(torch.float32), rtol=1e-2, atol=1e-4)
    for wt, x in mats:
        ref = x.float() @ wt.materialize(torch.float32).t()
        torch.testing.assert_close(first[mats.index((wt, x))].float(), ref, rtol=2e-2, atol=2e-2)
    for _ in range(3):
        for (wt, x), y0 in zip(mats, first):
            torch.testing.assert_close(wt.linear(x), y0, rtol=1e-2, atol=1e-2)
    wt, x = mats[1]
    xp = torch.randn(40, x.shape[1], device="cuda").bfloat16()  # prefill-sized: dequant + library GEMM
    torch.testing.assert_close(wt.linear(xp).float(), xp.float() @ wt.materialize(torch.float32).t(), rtol=2e-2,
                               atol=2e-2)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        wt.linear(x)  # workspace for this stream exists before capture
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        yg = wt.linear(x)
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        torch.testing.assert_close(yg, first[1], rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("H", [14336, 16384])
@pytest.mark.parametrize("res", [False, True])
def test_wide_norm_forward(H, res):
    """Forward LayerNorm / RMSNorm on BLOOM-176B-wide rows (wide NV buckets) vs fp32 references."""
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    torch.manual_seed(H)
    x = torch.randn(5, H, device="cuda").bfloat16()
    r = torch.randn(5, H, device="cuda").bfloat16() if res else None
    g = torch.randn(H, device="cuda").bfloat16()
    b = torch.randn(H, device="cuda").bfloat16()
    h = x.float() + (r.float() if res else 0)
    with torch.no_grad():
        y = DF.layer_norm(x, g, b, 1e-5, r)
        y = y[0] if res else y
        yr = DF.rms_norm(x, g, 1e-6, r)
        yr = yr[0] if res else yr
    ref = F.layer_norm(h, (H, ), g.float(), b.float(), 1e-5)
    ref_r = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-6) * g.float()
    torch.testing.assert_close(y.float(), ref, rtol=3e-2, atol=3e-2)
    torch.testing.assert_close(yr.float(), ref_r, rtol=3e-2, atol=3e-2)


@pytest.mark.parametrize("rows", [1, 16, 256, 300])
@pytest.mark.parametrize("H", [1024, 4096, 5120, 14336])
@pytest.mark.parametrize("res", [False, True])
def test_norm_forward_few_and_many_rows(rows, H, res):
    """Up to 256 rows a block owns each row (decode-sized inputs), beyond that a wave does: both against fp32, with
    the saved statistics checked through the backward of the training path."""
    from deepspeedsyclsupport_amd.ops.transformer import functional as DF
    torch.manual_seed(rows * 7 + H)
    x = torch.randn(rows, H, device="cuda").bfloat16()
    r = torch.randn(rows, H, device="cuda").bfloat16() if res else None
    g = (1 + 0.1 * torch.randn(H, device="cuda")).bfloat16()
    b = (0.1 * torch.randn(H, device="cuda")).bfloat16()
    h = x.float() + (r.float() if res else 0)
    with torch.no_grad():
        y = DF.layer_norm(x, g, b, 1e-5, r)
        yr = DF.rms_norm(x, g, 1e-6, r)
    if res:
        torch.testing.assert_close(y[1].float(), h.bfloat16().float(), rtol=0, atol=0)
        torch.testing.assert_close(yr[1].float(), h.bfloat16().float(), rtol=0, atol=0)
        y, yr = y[0], yr[0]
    ref = F.layer_norm(h, (H, ), g.float(), b.float(), 1e-5)
    ref_r = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-6) * g.float()
    torch.testing.assert_close(y.float(), ref, rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(yr.float(), ref_r, rtol=2e-2, atol=2e-2)
    if H <= 8192 and not res:  # the backward kernels (hidden <= 8192) consume the forward's mean / rstd
        xg = x.clone().requires_grad_(True)
        xf = x.float().requires_grad_(True)
        gy = torch.randn(rows, H, device="cuda")
        (DF.layer_norm(xg, g, b, 1e-5).float() * gy).sum().backward()
        (F.layer_norm(xf, (H, ), g.float(), b.float(), 1e-5) * gy).sum().backward()
        torch.testing.assert_close(xg.grad.float(), xf.grad, rtol=5e-2, atol=5e-2)


@pytest.mark.parametrize("D,rot,interleaved", [(96, 16, False), (80, 80, True), (80, 80, False), (80, 20, False), (64, 8, True)])
def test_qkv_rope_append_chunks_and_pairs(D, rot, interleaved):
    """Widths and rotations of whole chunks of 8, and those that go pair by pair: rows of a ragged batch, without copies."""
    hq, hk, BS, T = 3, 1, 8, 21
    kc, vc, bt, maxb = _paged_setup(2, hk, D, BS, [64, 64])
    qkv = torch.randn(T, (hq + 2 * hk) * D, device="cuda").bfloat16()
    seqs = torch.tensor([0] * 9 + [1] * 12, dtype=torch.int32, device="cuda")
    pos = torch.cat([torch.arange(5, 14), torch.arange(12)]).int().cuda()
    cos, sin = R.rope_tables(256, rot, device="cuda")
    start = torch.tensor([5, 0], dtype=torch.int32, device="cuda")
    q = ops().qkv_rope_append(qkv, cos, sin, pos, kc, vc, bt, start, 1, hq, hk, rot, interleaved, False, seqs)[0]
    x = qkv.view(T, hq + 2 * hk, D).float()
    c, s = cos[pos.long()][:, None], sin[pos.long()][:, None]
    y = x.clone()
    a, b = (x[..., 0:rot:2], x[..., 1:rot:2]) if interleaved else (x[..., :rot // 2], x[..., rot // 2:rot])
    lo, hi = (slice(0, rot, 2), slice(1, rot, 2)) if interleaved else (slice(0, rot // 2), slice(rot // 2, rot))
    y[..., lo], y[..., hi] = a * c - b * s, b * c + a * s
    torch.testing.assert_close(q.float(), y[:, :hq], rtol=1e-2, atol=1e-2)
    blk, off = bt[seqs.long(), (pos // BS).long()].long(), (pos % BS).long()
    torch.testing.assert_close(kc[blk, :, off].float(), y[:, hq:hq + hk], rtol=1e-2, atol=1e-2)
    assert torch.equal(vc[blk, :, off].float(), x[:, hq + hk:])
