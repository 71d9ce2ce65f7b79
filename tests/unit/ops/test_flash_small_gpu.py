"""Small-head flash attention with biases / dropout (`csrc/attn/flash_small.hip`) against a plain fp32 PyTorch
reference of the same op — forward, dQ/dK/dV and both bias gradients (reference test:
`tests/unit/ops/deepspeed4science/test_DS4Sci_EvoformerAttention.py`, which compares against an fp32 einsum
attention with the same two biases)."""
import math

import pytest
import torch

from deepspeedsyclsupport_amd.ops import flash_small as FS

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.float() - b.float()).abs().max() / b.float().abs().max().clamp_min(1e-6)).item()


def _case(Z, S, H, D, dtype, b1, b2, b2_div, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn(Z, S, H, D, device="cuda", dtype=dtype, generator=g) for _ in range(3))
    bias1 = (torch.randn(Z, S, device="cuda", generator=g) * 2).to(dtype) if b1 else None
    bias2 = torch.randn(Z // b2_div, H, S, S, device="cuda", generator=g).to(dtype) if b2 else None
    return q, k, v, bias1, bias2


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S,b1,b2,b2_div", [(128, True, True, 2), (100, True, True, 1), (200, False, True, 4),
                                            (64, True, False, 1), (130, False, False, 1)])
def test_fwd_bwd_vs_fp32(D, dtype, S, b1, b2, b2_div):
    Z, H = 4, 3
    q, k, v, bias1, bias2 = _case(Z, S, H, D, dtype, b1, b2, b2_div)
    ins = [t.detach().clone().requires_grad_(True) if t is not None else None for t in (q, k, v, bias1, bias2)]
    out = FS.flash_small(*ins[:3], ins[3], ins[4], b2_div=b2_div)
    refs = [t.detach().float().clone().requires_grad_(True) if t is not None else None for t in (q, k, v, bias1, bias2)]
    ref = FS.reference(*refs[:3], refs[3], refs[4], b2_div=b2_div)
    tol = 2e-2 if dtype == torch.bfloat16 else 6e-3
    assert _rel(out, ref) < tol
    go = torch.randn_like(ref)
    out.backward(go.to(dtype))
    ref.backward(go)
    for name, a, r in zip(("dq", "dk", "dv", "db1", "db2"), ins, refs):
        if a is None:
            continue
        assert a.grad is not None, name
        assert _rel(a.grad, r.grad) < 2 * tol, (name, _rel(a.grad, r.grad))


@pytest.mark.parametrize("D", [32, 64])
def test_dropout_matches_host_mask(D):
    Z, S, H, p, seed = 2, 160, 2, 0.25, 12345
    q, k, v, bias1, _ = _case(Z, S, H, D, torch.bfloat16, True, False, 1, seed=3)
    ins = [t.detach().clone().requires_grad_(True) for t in (q, k, v)]
    out = FS.flash_small(*ins, bias1, dropout_p=p, seed=seed)
    keep = FS.keep_mask(seed, Z, H, S, p)
    frac = keep.float().mean().item()
    assert abs(frac - (1 - p)) < 0.01
    refs = [t.detach().float().clone().requires_grad_(True) for t in (q, k, v)]
    ref = FS.reference(*refs, bias1, keep=keep, p=p)
    assert _rel(out, ref) < 2e-2
    go = torch.randn_like(ref)
    out.backward(go.bfloat16())
    ref.backward(go)
    for a, r in zip(ins, refs):
        assert _rel(a.grad, r.grad) < 4e-2
    # same seed -> same output; new seed -> different
    again = FS.flash_small(q, k, v, bias1, dropout_p=p, seed=seed)
    assert torch.equal(again, out.detach())
    other = FS.flash_small(q, k, v, bias1, dropout_p=p, seed=seed + 1)
    assert not torch.equal(other, out.detach())


@pytest.mark.parametrize("D", [32, 64])
def test_evoformer_api_kernel_vs_sdpa(D):
    from deepspeedsyclsupport_amd.ops import deepspeed4science as E
    B, N, S, H = 1, 3, 96, 4
    g = torch.Generator(device="cuda").manual_seed(1)
    Q, K, V = (torch.randn(B, N, S, H, D, device="cuda", dtype=torch.bfloat16, generator=g) for _ in range(3))
    mask = (torch.rand(B, N, 1, 1, S, device="cuda", generator=g) > 0.2).to(torch.bfloat16)
    b1 = (1e9 * (mask - 1)).to(torch.bfloat16)
    b2 = torch.randn(B, 1, H, S, S, device="cuda", dtype=torch.bfloat16, generator=g)
    ins = [t.clone().requires_grad_(True) for t in (Q, K, V, b1, b2)]
    out = E.DS4Sci_EvoformerAttention(ins[0], ins[1], ins[2], [ins[3], ins[4]])
    refs = [t.float().clone().requires_grad_(True) for t in (Q, K, V, b1, b2)]
    ref = E._sdpa_path(refs[0], refs[1], refs[2], [refs[3], refs[4]])
    assert out.shape == (B, N, S, H, D)
    assert _rel(out, ref) < 2e-2
    go = torch.randn_like(ref)
    out.backward(go.bfloat16())
    ref.backward(go)
    for name, a, r in zip(("dq", "dk", "dv", "db2"), ins[:3] + ins[4:], refs[:3] + refs[4:]):
        assert _rel(a.grad, r.grad) < 4e-2, name
    assert ins[3].grad is not None


def test_bert_layer_uses_kernel_with_mask():
    from deepspeedsyclsupport_amd.ops.transformer import DeepSpeedTransformerConfig, DeepSpeedTransformerLayer
    torch.manual_seed(0)
    cfg = DeepSpeedTransformerConfig(batch_size=2, hidden_size=256, heads=4, attn_dropout_ratio=0.0,
                                     hidden_dropout_ratio=0.0, num_hidden_layers=2, initializer_range=0.02)
    layer = DeepSpeedTransformerLayer(cfg).cuda().to(torch.bfloat16)
    x = torch.randn(2, 96, 256, device="cuda", dtype=torch.bfloat16)
    m = torch.zeros(2, 1, 1, 96, device="cuda")
    m[1, ..., 80:] = -10000.0
    calls = []
    orig = FS.FlashSmallFunc.apply

    def spy(*a):
        calls.append(1)
        return orig(*a)

    FS.FlashSmallFunc.apply = spy
    try:
        out = layer(x, m)
    finally:
        FS.FlashSmallFunc.apply = orig
    assert calls, "the BERT layer did not take the fused attention kernel"
    ref_layer = DeepSpeedTransformerLayer(cfg).cuda().float()
    ref_layer.load_state_dict({k: v.float() for k, v in layer.state_dict().items()})
    ref = ref_layer(x.float(), m)
    assert _rel(out, ref) < 3e-2


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("Sk", [77, 64, 300])
def test_cross_length_forward(D, Sk):
    """Queries and keys of different lengths (diffusers cross-attention): forward only, with a per-key bias."""
    Z, S, H = 2, 150, 2
    g = torch.Generator(device="cuda").manual_seed(5)
    q = torch.randn(Z, S, H, D, device="cuda", dtype=torch.bfloat16, generator=g)
    k, v = (torch.randn(Z, Sk, H, D, device="cuda", dtype=torch.bfloat16, generator=g) for _ in range(2))
    b1 = torch.randn(Z, Sk, device="cuda", generator=g).bfloat16()
    with torch.no_grad():
        out = FS.flash_small(q, k, v, b1)
    assert _rel(out, FS.reference(q, k, v, b1)) < 2e-2
    with pytest.raises(NotImplementedError):
        FS.flash_small(q.requires_grad_(True), k, v)


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("Z,S,H,b2_div,p", [(1, 1, 3, 1, 0.0), (2, 3, 1, 2, 0.0), (3, 65, 2, 3, 0.0), (64, 129, 1, 64, 0.0),
                                            (40, 71, 2, 20, 0.0), (24, 64, 2, 24, 0.3), (8, 250, 1, 2, 0.3)])
def test_tile_edges_splits_and_unaligned_pair_biases(D, Z, S, H, b2_div, p):
    """Sizes around the tiles, a pair bias at odd addresses whose last chunk ends with the tensor, one or several workgroups
    adding up its gradient; masks of the type's lowest value: a query whose keys all have it attends to them alike."""
    q, k, v, bias1, bias2 = _case(Z, S, H, D, torch.bfloat16, True, True, b2_div, seed=7)
    bias1[0, 1:] = torch.finfo(torch.bfloat16).min
    room = torch.empty(bias2.numel() + 1, device="cuda", dtype=torch.bfloat16)
    odd = room[1:].view_as(bias2).copy_(bias2)
    keep = FS.keep_mask(9, Z, H, S, p) if p else None
    masked = torch.full_like(bias1, torch.finfo(torch.bfloat16).min)
    assert _rel(FS.flash_small(q, k, v, masked), v.float().mean(1, keepdim=True).expand_as(v)) < 2e-2
    ins = [t.detach().requires_grad_(True) for t in (q, k, v, bias1, odd)]
    refs = [t.detach().float().clone().requires_grad_(True) for t in (q, k, v, bias1, bias2)]
    out = FS.flash_small(*ins, b2_div=b2_div, dropout_p=p, seed=9)
    ref = FS.reference(*refs, b2_div=b2_div, **(dict(keep=keep, p=p) if p else {}))
    assert _rel(out, ref) < 2e-2
    go = torch.randn_like(ref)
    out.backward(go.bfloat16())
    ref.backward(go)
    # sums over keys, queries and the b2_div sharers of bf16-rounded factors: as in the tests above
    for name, a, r in zip(("dq", "dk", "dv", "db1", "db2"), ins, refs):
        assert (a.grad.float() - r.grad).abs().max() < 4e-2 * r.grad.abs().max() + 4e-2, name


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("S", [63, 65, 130])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_row_of_the_pair_bias_stays_with_its_query(D, S, bad):
    """Rows of a pair bias that are no whole chunks: what one row holds must not reach the query of the row before it, whose last
    tile reads on into it (outputs and dQ of all other queries: bit for bit those of a clean bias)."""
    q, k, v, _, bias2 = _case(2, S, 2, D, torch.bfloat16, False, True, 1, seed=11)
    rows = torch.arange(S, device="cuda") % 3 == 1
    poisoned = bias2.clone()
    poisoned[:, :, rows, 0] = bad
    got = []
    for b in (bias2, poisoned):
        ins = [t.detach().requires_grad_(True) for t in (q, k, v)]
        out = FS.flash_small(*ins, bias2=b)
        got.append((out, torch.autograd.grad(out, ins[0], torch.ones_like(out))[0]))
    for name, clean, other in zip(("o", "dq"), *got):
        assert torch.isnan(other[:, rows]).any(), name
        assert torch.equal(clean[:, ~rows], other[:, ~rows]), name


@pytest.mark.parametrize("dtype,masked", [(torch.bfloat16, True), (torch.float16, False)])
@pytest.mark.parametrize("Z,S,H,b2_div", [(256, 1, 1, 256), (128, 31, 2, 64), (86, 33, 3, 43), (64, 130, 4, 64), (40, 225, 7, 20),
                                          (32, 256, 8, 16), (32, 257, 8, 16)])
def test_short_sequences_in_one_pass(Z, S, H, b2_div, dtype, masked):
    """Enough short sequences that one pass makes dQ, dK and dV (257: two again): one to eight tiles of 32 with remainders, a pair
    bias at odd addresses, with a per-key mask and its gradient and without."""
    q, k, v, bias1, bias2 = _case(Z, S, H, 32, dtype, masked, True, b2_div, seed=5)
    if masked:
        bias1[0, 1:] = torch.finfo(dtype).min
    odd = torch.empty(bias2.numel() + 1, device="cuda", dtype=dtype)[1:].view_as(bias2).copy_(bias2)
    ins = [t if t is None else t.detach().requires_grad_(True) for t in (q, k, v, bias1, odd)]
    refs = [t if t is None else t.detach().double().requires_grad_(True) for t in (q, k, v, bias1, bias2)]
    out, ref = FS.flash_small(*ins, b2_div=b2_div), FS.reference(*refs, b2_div=b2_div)
    go = torch.randn(ref.shape, device="cuda")
    out.backward(go.to(dtype))
    ref.backward(go.to(dtype).double())
    tol = 4e-2 if dtype == torch.bfloat16 else 1e-2   # as above
    for name, a, r in zip(("dq", "dk", "dv", "db1", "db2"), ins, refs):
        if a is not None:
            assert (a.grad.double() - r.grad).abs().max() < tol * r.grad.abs().max() + tol, name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S,Sk", [(1, 8), (40, 7), (33, 31), (32, 33), (130, 95), (257, 250), (300, 256), (64, 257)])
def test_forward_with_a_pair_bias_by_keys(S, Sk, dtype):
    """Keys around tiles of 32, the ends of the kernel that holds all of them (8 and 256) and what is past them; rows of one packed
    buffer, a pair bias at odd addresses; keys masked by the type's lowest value, for one z all of them (who then count alike).
    P is rounded to 2^-9 (2^-12): twice that of the largest value, and the result's own rounding. Scores of keys masked by half's
    lowest value stand 2^-8 apart in single precision, and so may the weights of a z that has no others."""
    Z, H, D = 6, 2, 32
    g = torch.Generator(device="cuda").manual_seed(S + Sk)
    q = torch.randn(Z, S, H, D, device="cuda", generator=g).to(dtype)
    k, v = torch.randn(Z, Sk, 2, H, D, device="cuda", generator=g).to(dtype).unbind(2)
    b1 = torch.zeros(Z, Sk, device="cuda", dtype=dtype)
    b1[torch.rand(Z, Sk, device="cuda", generator=g) < 0.3] = torch.finfo(dtype).min
    b1[0] = torch.finfo(dtype).min
    b2 = torch.randn(Z // 3, H, S, Sk, device="cuda", generator=g).to(dtype)
    odd = torch.empty(b2.numel() + 1, device="cuda", dtype=dtype)[1:].view_as(b2).copy_(b2)
    with torch.no_grad():
        out = FS.flash_small(q, k, v, b1, odd, b2_div=3)
    ref = FS.reference(q, k, v, b1, b2, b2_div=3)
    step = 2.0**-9 if dtype == torch.bfloat16 else 2.0**-12
    loose = torch.full((Z, 1, 1, 1), 2 * step, device="cuda")
    if dtype == torch.float16:
        loose[0] += 2.0**-7
    assert ((out.float() - ref).abs() <= step * ref.abs() + loose * v.float().abs().max()).all()


@pytest.mark.parametrize("S", [180, 256])
@pytest.mark.parametrize("groups", [128, 132, 256, 260, 384, 388])
def test_forward_on_either_side_of_its_lines(S, groups):
    """The numbers of workgroups at which the forward's kernel changes, against fp64; P and the result are rounded to 2^-8."""
    q, k, v, bias1, bias2 = _case(groups // 4, S, 4, 32, torch.bfloat16, True, True, groups // 4, seed=groups)
    with torch.no_grad():
        out = FS.flash_small(q, k, v, bias1, bias2, b2_div=groups // 4)
    ref = FS.reference(*(t.double() for t in (q, k, v, bias1, bias2)), b2_div=groups // 4)
    assert ((out.double() - ref).abs() <= 2.0**-8 * (ref.abs() + v.double().abs().max())).all()


@pytest.mark.parametrize("Z,S", [(64, 32), (64, 64), (64, 96), (159, 97), (160, 97), (160, 128), (64, 160), (64, 161), (64, 192), (64, 193),
                                 (64, 224), (64, 255)])
def test_one_pass_by_number_of_tiles(Z, S):
    """Gradients of every kernel there is for a number of tiles of 32, at their ends (159 of four tiles: two passes), against fp64: bf16
    factors as in the tests above."""
    H = 4
    q, k, v, bias1, bias2 = _case(Z, S, H, 32, torch.bfloat16, True, True, Z, seed=S)
    ins = [t.detach().requires_grad_(True) for t in (q, k, v, bias1, bias2)]
    refs = [t.detach().double().requires_grad_(True) for t in ins]
    out, ref = FS.flash_small(*ins, b2_div=Z), FS.reference(*refs, b2_div=Z)
    go = torch.randn(ref.shape, device="cuda")
    out.backward(go.bfloat16())
    ref.backward(go.bfloat16().double())
    for name, a, r in zip(("dq", "dk", "dv", "db1", "db2"), ins, refs):
        assert (a.grad.double() - r.grad).abs().max() < 4e-2 * r.grad.abs().max() + 4e-2, name


@pytest.mark.parametrize("run", [4, 8, 16, 32, 64])
@pytest.mark.parametrize("odd", [0, 1])
def test_masked_runs_of_keys(run, odd):
    """Every other run of keys masked, the others with scores far above: the maximum of a row is that of all its keys, whichever lanes
    and tiles hold them (of the masked ones alone, the others' exponentials would be infinite). Tolerance as in the tests above."""
    Z, S, H = 72, 200, 2   # (more than 128 workgroups)
    q, k, v, _, bias2 = _case(Z, S, H, 32, torch.bfloat16, False, True, Z, seed=run)
    keys = torch.arange(S, device="cuda") // run % 2
    bias1 = torch.where(keys == odd, -1e9, 100.0).expand(Z, S).bfloat16().contiguous()
    with torch.no_grad():
        out = FS.flash_small(q, k, v, bias1, bias2, b2_div=Z)
    assert _rel(out, FS.reference(q, k, v, bias1, bias2, b2_div=Z)) < 2e-2


_MASKS = [-1e4, -1e5, -1e6, -1e7, -1e9, -5e9, -1e10, -1e15, -1e20, torch.finfo(torch.bfloat16).min]


def _masked_case(mask, S=100):
    """Whole rows masked by `mask`, rows whose first 32 (64) keys are, a third of the keys at random. Queries and keys are small whole
    numbers and their products exact, so that the scores can be told to the last bit: fma(q k, scale, bias1 + bias2) in single precision."""
    Z, H, D = 128, 2, 32
    g = torch.Generator(device="cuda").manual_seed(17)
    q, k = (torch.randint(-2, 3, (Z, S, H, D), device="cuda", generator=g).bfloat16() for _ in range(2))
    v, do = (torch.randn(Z, S, H, D, device="cuda", generator=g).bfloat16() for _ in range(2))
    b2 = torch.randn(2, H, S, S, device="cuda", generator=g)
    b2[1, 1] *= 40   # (beside 1e9, single precision has steps of 64)
    gone = torch.rand(Z, S, device="cuda", generator=g) < 0.3
    gone[0::4], gone[1::4, :32], gone[3::4, :64] = True, True, True
    b1 = torch.zeros(Z, S, device="cuda").masked_fill_(gone, mask)
    b1, b2 = b1.bfloat16(), b2.bfloat16()
    bias = (b1.float()[:, None, None] + b2.float().repeat_interleave(Z // 2, 0)).double()
    s = (q.double().transpose(1, 2) @ k.double().permute(0, 2, 3, 1) * torch.tensor(D**-0.5).double() + bias).float().double()
    return q, k, v, do, b1, b2, s


@pytest.mark.parametrize("mask", _MASKS)
def test_finite_masks_forward(mask):
    """P is rounded to 2^-9, as is the result; LSE is a maximum plus a logarithm in single precision."""
    from deepspeedsyclsupport_amd.ops.native import hip_ops
    q, k, v, _, b1, b2, s = _masked_case(mask)
    o, lse = hip_ops().flash_small_fwd(q, k, v, b1, b2, 64, 32**-0.5, 0.0, 0)
    want = (torch.softmax(s, -1) @ v.double().transpose(1, 2)).transpose(1, 2)
    assert ((o.double() - want).abs() <= 2.0**-9 * want.abs() + 2.0**-8 * v.double().abs().max()).all()
    want = torch.logsumexp(s, -1)
    assert ((lse.double() - want).abs() <= 2.0**-22 * want.abs() + 1e-5).all()


@pytest.mark.parametrize("mask", _MASKS)
@pytest.mark.parametrize("S", [70, 100])
def test_finite_masks_backward(S, mask):
    """In one pass for all gradients (70) and in two (100). Where some keys are not masked, against fp64 as in the tests above. Rows
    masked throughout: their scores, and LSE, stand 64 apart at -1e9, so that a weight may come out as 1 for 1 / S, but as no more:
    the gradients are bounded by those of such weights."""
    from deepspeedsyclsupport_amd.ops.native import hip_ops
    q, k, v, do, b1, b2, s = _masked_case(mask, S)
    scale = 32**-0.5
    o, lse = hip_ops().flash_small_fwd(q, k, v, b1, b2, 64, scale, 0.0, 0)
    dq, dk, dv, db1, db2 = hip_ops().flash_small_bwd(do, q, k, v, o, lse, b1, b2, 64, scale, 0.0, 0, True, True)
    assert all(bool(t.isfinite().all()) for t in (dq, dk, dv, db1, db2))
    qd, kd, vd, dod = (t.double().transpose(1, 2) for t in (q, k, v, do))
    p = torch.softmax(s, -1)
    dp = dod @ vd.transpose(-1, -2) - (dod * o.double().transpose(1, 2)).sum(-1, keepdim=True)
    ds = p * dp
    want = [t.transpose(1, 2) for t in (scale * (ds @ kd), scale * (ds.transpose(-1, -2) @ qd), p.transpose(-1, -2) @ dod)]
    most = [t.transpose(1, 2) for t in (scale * (dp.abs() @ kd.abs()), scale * (dp.abs().transpose(-1, -2) @ qd.abs()),
                                        dod.abs().sum(-2, keepdim=True).expand_as(vd))]
    some = torch.arange(q.shape[0], device="cuda") % 4 != 0
    for name, a, w, m in zip(("dq", "dk", "dv"), (dq, dk, dv), want, most):
        assert ((a.double() - w)[some].abs() < 4e-2 * w[some].abs().max() + 4e-2).all(), name
        assert (a.double().abs()[~some] <= 1.02 * m[~some] + 1e-3).all(), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("Z,S,H,N", [(64, 40, 4, 64), (16, 37, 3, 8), (40, 131, 1, 40), (6, 33, 2, 3), (4, 24, 2, 1)])
def test_pair_bias_gradient_in_the_inputs_type(dtype, Z, S, H, N):
    """Sums of several parts leave in the inputs' type as they would after a cast, at lengths whose square 4 divides and does not;
    where there is one part, or none, they stay in fp32."""
    from deepspeedsyclsupport_amd.ops.native import hip_ops
    g = torch.Generator(device="cuda").manual_seed(0)
    q, k, v, do = (torch.randn(Z, S, H, 32, device="cuda", generator=g).to(dtype) for _ in range(4))
    b2 = torch.randn(Z // N, H, S, S, device="cuda", generator=g).to(dtype)
    o, lse = hip_ops().flash_small_fwd(q, k, v, None, b2, N, 0.2, 0.0, 0)
    plain, cast = (hip_ops().flash_small_bwd(do, q, k, v, o, lse, None, b2, N, 0.2, 0.0, 0, False, True, c)[4] for c in (False, True))
    assert plain.dtype == torch.float32 and cast.dtype == (dtype if N >= 8 else torch.float32)
    assert torch.equal(plain.to(dtype), cast.to(dtype))


@pytest.mark.parametrize("dtype,unit", [(torch.bfloat16, 2.0**-8), (torch.float16, 2.0**-11)], ids=["bf16", "fp16"])
@pytest.mark.parametrize("S,top", [(64, 40), (250, 100), (256, 255)])
def test_largest_weight_is_exact(dtype, unit, S, top):
    """One key stands up to e^5 above the tiles before it, and it alone has a value: its weight is 1 whatever stood before, so that
    the result is rounded once (2 percent beside that for the exponentials and sums in single precision)."""
    from deepspeedsyclsupport_amd.ops.native import hip_ops
    Z, H, D = 18, 8, 32   # (more than 128 workgroups)
    q = torch.zeros(Z, S, H, D, device="cuda", dtype=dtype)
    v = torch.zeros_like(q)
    v[:, top] = 1
    above = torch.linspace(0.5, 5.4, H * S, device="cuda").view(1, H, S).to(dtype)
    b2 = torch.zeros(1, H, S, S, device="cuda", dtype=dtype)
    b2[..., top] = above
    o, lse = hip_ops().flash_small_fwd(q, q, v, None, b2, Z, D**-0.5, 0.0, 0)
    e = above.double().exp().transpose(1, 2)[..., None]
    want = e / (e + S - 1)
    assert ((o.double() - want).abs() <= 1.02 * unit * want).all()
    assert (lse.double() - (e[..., 0] + S - 1).log().transpose(1, 2)).abs().max() < 1e-5
