"""Ragged paged flash-prefill kernel (csrc/attn/paged_prefill.hip) vs an fp32 reference over the same paged cache:
mixed chunk lengths and cached prefixes, GQA, ALiBi, sliding windows, cache block sizes 16 / 64."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(lens, starts, Hq, Hk, BS, alibi, window, seed=0, D=128, own_loop=False):
    from deepspeedsyclsupport_amd.inference.model_implementations.transformer import RaggedMeta, alibi_slopes
    from deepspeedsyclsupport_amd.ops.native import hip_ops
    g = torch.Generator(device="cuda").manual_seed(seed)
    S = len(lens)
    need = [-(-(st + n) // BS) for st, n in zip(starts, lens)]
    nblocks = sum(need) + 3
    kc = torch.randn(nblocks, Hk, BS, D, device="cuda", generator=g).bfloat16()
    vc = torch.randn(nblocks, Hk, BS, D, device="cuda", generator=g).bfloat16()
    perm = torch.randperm(nblocks, generator=torch.Generator().manual_seed(seed)).tolist()
    blocks, o = [], 0
    for nb in need:
        blocks.append(perm[o:o + nb])
        o += nb
    meta = RaggedMeta.build(starts, lens, blocks, 0, BS, torch.device("cuda"))
    T = sum(lens)
    if own_loop:  # (many rows of long contexts: paged_rows.h)
        assert D == 128 and not window and meta.work.shape[0] * Hq >= 1024 and meta.block_tables.shape[1] * BS >= 2048
    q = torch.randn(T, Hq, D, device="cuda", generator=g).bfloat16()
    slopes = alibi_slopes(Hq).cuda() if alibi else None
    scale = 1.0 / math.sqrt(D)
    out = hip_ops().paged_prefill(q, kc, vc, meta.block_tables, meta.start_pos, meta.cu_q, meta.work, slopes, window,
                                  scale)
    torch.cuda.synchronize()
    for i in range(S):
        a, b = meta.cu_host[i], meta.cu_host[i + 1]
        L = starts[i] + lens[i]
        ids = torch.tensor(blocks[i], device="cuda")
        k = kc[ids].transpose(0, 1).reshape(Hk, -1, D)[:, :L].float()
        v = vc[ids].transpose(0, 1).reshape(Hk, -1, D)[:, :L].float()
        k, v = k.repeat_interleave(Hq // Hk, 0), v.repeat_interleave(Hq // Hk, 0)
        qi = q[a:b].float().transpose(0, 1)  # [Hq, n, D]
        s = qi @ k.transpose(1, 2) * scale
        qpos = torch.arange(starts[i], L, device="cuda")
        kpos = torch.arange(L, device="cuda")
        if alibi:
            s = s + slopes[:, None, None] * (kpos[None, None, :] - qpos[None, :, None]).float()
        bad = kpos[None, :] > qpos[:, None]
        if window:
            bad = bad | (kpos[None, :] <= qpos[:, None] - window)
        s = s.masked_fill(bad[None], float("-inf"))
        ref = torch.softmax(s, -1) @ v
        torch.testing.assert_close(out[a:b].float().transpose(0, 1), ref, rtol=2e-2, atol=2e-2,
                                   msg=lambda m: f"seq {i} (start {starts[i]}, n {lens[i]}): {m}")


@pytest.mark.parametrize("n", [128, 40])
def test_paged_prefill_peak_at_every_key(n):
    """Each of 128 cached keys in turn is one row's only large score: a maximum that misses any overflows its weights."""
    from deepspeedsyclsupport_amd.inference.model_implementations.transformer import RaggedMeta
    from deepspeedsyclsupport_amd.ops.native import hip_ops
    g = torch.Generator().manual_seed(n)
    perm = torch.randperm(128, generator=g)[:n].cuda()
    kc = torch.zeros(4, 1, 64, 128, device="cuda", dtype=torch.bfloat16)
    kc[:2] = torch.eye(128, device="cuda").bfloat16().view(2, 1, 64, 128)
    vc = torch.randn(4, 1, 64, 128, generator=g).cuda().bfloat16()
    q = 300 * torch.eye(128, device="cuda").bfloat16()[perm][:, None]
    meta = RaggedMeta.build([128], [n], [[0, 1, 2, 3]], 0, 64, torch.device("cuda"))
    out = hip_ops().paged_prefill(q, kc, vc, meta.block_tables, meta.start_pos, meta.cu_q, meta.work, None, 0, 1.0)
    assert torch.equal(out[:, 0], vc[:2].reshape(128, 128)[perm])  # one weight is 1, the others e^-300 = 0 in fp32


@pytest.mark.parametrize("Hq,Hk", [(8, 8), (8, 2)])
@pytest.mark.parametrize("BS", [16, 64])
def test_paged_prefill_mixed_chunks(Hq, Hk, BS):
    _case([37, 1, 200, 129, 64], [0, 100, 0, 70, 333], Hq, Hk, BS, alibi=False, window=0)


@pytest.mark.parametrize("window", [0, 37, 200])
def test_paged_prefill_alibi_window(window):
    _case([90, 300, 5], [0, 20, 400], 4, 4, 64, alibi=True, window=window, seed=window)


def test_paged_prefill_long_prefix():
    _case([256, 17], [3000, 4095], 8, 1, 64, alibi=False, window=0, seed=3)


@pytest.mark.parametrize("alibi", [False, True])
@pytest.mark.parametrize("Hq,Hk,BS,lens,starts", [
    (32, 8, 64, [4096], [0]),
    (32, 4, 16, [1200, 37, 2100, 900], [0, 2011, 130, 17]),
    (16, 8, 32, [3000, 65, 2049, 3100], [0, 4031, 63, 1]),
    (12, 12, 128, [4130, 90, 7000], [0, 4001, 30]),
])
def test_long_prompts(Hq, Hk, BS, lens, starts, alibi):
    _case(lens, starts, Hq, Hk, BS, alibi, 0, seed=BS, own_loop=True)


@pytest.mark.parametrize("D", [64, 80, 96, 256])
@pytest.mark.parametrize("alibi,window", [(False, 0), (True, 70)])
def test_paged_prefill_head_dims(D, alibi, window):
    """GPT-2 / Phi / GPT-NeoX-20B / GPT-J head sizes through the same kernel template."""
    _case([37, 1, 200, 129, 64], [0, 100, 0, 70, 333], 8, 2, 64, alibi=alibi, window=window, seed=D, D=D)


def test_uniform_tables_are_cached():
    from deepspeedsyclsupport_amd.inference.model_implementations import transformer as tr
    a = tr._uniform_tables(3, 300, torch.device("cuda"))
    b = tr._uniform_tables(3, 300, torch.device("cuda"))
    assert a[0] is b[0] and a[1] is b[1]
    assert a[0].tolist() == [0, 300, 600, 900]
    assert a[1].tolist() == [[s, q] for s in range(3) for q in range(3)]


@pytest.mark.parametrize("BS", [16, 32, 128])
@pytest.mark.parametrize("form", ["plain", "alibi", "window", "chunk", "cap", "cap_high", "sink_gate"])
def test_pages_of_two_powers_match_other_pages(form, BS):
    """Heads of 128 over pages of 16, 32, .. tokens take their own kernel; pages of 24 take the one for any width. Lengths at the
    edges of tiles, query blocks and pages; an output that is columns of a wider matrix."""
    from deepspeedsyclsupport_amd.inference.model_implementations.transformer import RaggedMeta, alibi_slopes
    from deepspeedsyclsupport_amd.ops import hybrid_ops
    from deepspeedsyclsupport_amd.ops.native import hip_ops
    lens, starts, Hq, Hk, D = [1, 64, 128, 129, 15, 200], [17, 0, 64, 1, 240, 500], 4, 2, 128
    g = torch.Generator(device="cuda").manual_seed(7)
    T, L = sum(lens), [s + n for s, n in zip(starts, lens)]
    q = torch.randn(T, Hq, D, device="cuda", generator=g).bfloat16() * 2
    keys, vals = ([torch.randn(n, Hk, D, device="cuda", generator=g).bfloat16() for n in L] for _ in range(2))
    gate = torch.randn(T, Hq, device="cuda", generator=g).bfloat16()
    sink = torch.randn(Hq, device="cuda", generator=g)

    def run(size):
        blocks, used = [], 0
        for n in L:
            blocks.append([used + i for i in range(-(-n // size))][::-1])
            used += -(-n // size)
        # rows that no token has written hold anything: they must not reach the result
        kc, vc = (torch.full((used, Hk, size, D), float("nan"), device="cuda").bfloat16() for _ in range(2))
        for b, k, v in zip(blocks, keys, vals):
            for j, blk in enumerate(b):
                part = slice(j * size, (j + 1) * size)
                kc[blk, :, :k[part].shape[0]] = k[part].transpose(0, 1)
                vc[blk, :, :v[part].shape[0]] = v[part].transpose(0, 1)
        m = RaggedMeta.build(starts, lens, blocks, 0, size, torch.device("cuda"))
        if form in ("plain", "alibi", "window"):
            return hip_ops().paged_prefill(q, kc, vc, m.block_tables, m.start_pos, m.cu_q, m.work,
                                           alibi_slopes(Hq).cuda() if form == "alibi" else None, 70 if form == "window" else 0,
                                           D**-0.5).view(T, Hq * D)
        how = {"chunk": dict(chunk=100), "cap": dict(softcap=20.0), "cap_high": dict(softcap=60.0, window=90),
               "sink_gate": dict(sink=sink, gate=gate)}[form]
        wide = torch.zeros(T, Hq * D + 64, device="cuda", dtype=torch.bfloat16)
        hybrid_ops.ragged_attention(q, kc, vc, m, D**-0.5, out=wide[:, 64:], **how)
        assert not wide[:, :64].any()
        return wide[:, 64:]

    a, b = run(BS).float(), run(24).float()
    assert torch.isfinite(a).all()
    # results and (plain forms) weights are bf16: a few units of 2^-9 of the rows' size
    assert ((a - b).norm() / b.norm()).item() < 6e-3
    torch.testing.assert_close(a, b, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("alibi", [False, True])
@pytest.mark.parametrize("Hq,Hk,BS,lens,starts", [
    (32, 8, 16, [449, 64, 1000, 1281, 33, 1200, 1], [0, 5, 300, 900, 415, 0, 1700]),
    (32, 8, 128, [2048, 65, 1983], [1, 640, 0]),
    (32, 1, 64, [4096], [0]),
    (8, 8, 64, [2047, 5, 4097, 1111, 7000, 2300], [0, 3, 64, 0, 1, 129]),
    (12, 12, 64, [4130, 7000, 90], [0, 30, 4001]),
    (16, 8, 32, [769, 127, 3000, 1111, 2900, 300], [0, 129, 1, 64, 100, 4000]),
])
def test_long_prompts_match_the_windowed_loop(Hq, Hk, BS, lens, starts, alibi):
    """Many rows of long contexts take a loop of their own; under a window that hides nothing they take the other one."""
    from deepspeedsyclsupport_amd.inference.model_implementations.transformer import RaggedMeta, alibi_slopes
    from deepspeedsyclsupport_amd.ops.native import hip_ops
    g = torch.Generator(device="cuda").manual_seed(11)
    q = torch.randn(sum(lens), Hq, 128, device="cuda", generator=g).bfloat16() * 3
    L = [s + n for s, n in zip(starts, lens)]
    blocks, used = [], 0
    for n in L:
        blocks.append([used + i for i in range(-(-n // BS))][::-1])
        used += -(-n // BS)
    kc = torch.randn(used, Hk, BS, 128, device="cuda", generator=g).bfloat16()
    vc = (torch.rand(used, Hk, BS, 128, device="cuda", generator=g) * 2 - 1).bfloat16()
    for b, n in zip(blocks, L):  # rows that no token has written hold anything
        if n % BS:
            kc[b[-1], :, n % BS:] = float("nan")
            vc[b[-1], :, n % BS:] = float("nan")
    m = RaggedMeta.build(starts, lens, blocks, 0, BS, torch.device("cuda"))
    slopes = alibi_slopes(Hq).cuda() if alibi else None
    assert m.work.shape[0] * Hq >= 1024 and m.block_tables.shape[1] * BS >= 2048
    a, b = (hip_ops().paged_prefill(q, kc, vc, m.block_tables, m.start_pos, m.cu_q, m.work, slopes, window, 128**-0.5).float()
            for window in (0, 1 << 20))
    # values within 1: on either side weights and result are rounded once each to bf16, by 2^-9 at most
    assert torch.isfinite(a).all() and (a - b).abs().max().item() < 4 * 2**-9 + 1e-4
    assert b.abs().max().item() > 0.5  # (peaked rows among them)
