"""How block-sparse lists are shared out over workgroups: the plan against the layout, and cut lists against dense attention."""
import pytest
import torch

from deepspeedsyclsupport_amd.ops.sparse_attention import block_sparse as bs
from deepspeedsyclsupport_amd.ops.sparse_attention.sparsity_config import BigBirdSparsityConfig, FixedSparsityConfig


def _layout(kind, H, blk, L, seed=0):
    n = L // blk
    g = torch.Generator().manual_seed(seed)
    lay = (torch.rand(H, n, n, generator=g) < 0.15).long()
    lay[:, torch.arange(n), torch.arange(n)] = 1
    lay[:, 0] = 1       # a global row and a global column
    lay[:, :, 0] = 1
    if kind == "shared":
        lay = lay[:1].expand(H, -1, -1).contiguous()
    elif kind == "empty":
        lay[:, n // 2:] = 0
        lay[:, :, n // 3:2 * n // 3] = 0
    return lay


def _covered(side, high, wide, L, head):
    """Times that each 16 x 16 piece is visited, from the lists; blocks are `high` x `wide` tokens (tiles along the other axis)."""
    seen, slots = torch.zeros(L // 16, -(-L // 256) * 16, dtype=torch.long), {}
    for blk, first, n, slot in side.work[head].tolist():
        if blk < 0:
            continue
        slots.setdefault(blk, []).append(slot)
        for j in range(first, first + n):
            t, m = side.tiles[head, blk, j].item(), side.masks[head, blk, j].item()
            r0, c0, rows, cols = (blk * 8, t * 4, 8, 4) if (high, wide) == (128, 64) else (t * 2, blk * 16, 2, 16)
            for r in range(rows):
                for k in range(cols):
                    seen[r0 + r, c0 + k] += (m >> (r * cols + k)) & 1
    return seen[:, :L // 16], slots


@pytest.mark.parametrize("kind", ["shared", "heads", "empty"])
@pytest.mark.parametrize("blk,L", [(16, 256), (32, 640), (64, 1152), (128, 1280), (256, 1280)])
def test_plan_visits_the_layout_once(kind, blk, L, monkeypatch):
    monkeypatch.setattr(bs, "_FWD_SHARE", (1 << 20, 2))
    monkeypatch.setattr(bs, "_BWD_SHARE", (1 << 20, 3))
    bs._PLANS.clear()
    H = 2
    lay = _layout(kind, H, blk, L)
    plan = bs.sparse_plan(lay, blk, L, 1, H, "cpu")
    want = (lay != 0).repeat_interleave(blk // 16, 1).repeat_interleave(blk // 16, 2)[:, :L // 16, :L // 16].long()
    for side, high, wide, blocks in ((plan.forward(), 128, 64, L // 128), (plan.backward(), 32, 256, -(-L // 256))):
        for head in range(side.work.shape[0]):
            seen, slots = _covered(side, high, wide, L, head)
            assert torch.equal(seen, want[head])
            assert sorted(slots) == list(range(blocks))          # blocks without a tile are written too
            merged = {b: list(range(s, s + n)) for b, s, n, _ in side.merges[head].tolist() if b >= 0}
            for b, got in slots.items():
                assert got == [-1] if b not in merged else sorted(got) == merged[b]
            used = [s for got in merged.values() for s in got]
            assert len(set(used)) == len(used) and all(0 <= s < side.nslots for s in used)
    bs._PLANS.clear()
    if kind != "empty":
        assert plan.forward().nslots > 0 or L <= 256


@pytest.mark.parametrize("kind", ["shared", "heads", "empty"])
@pytest.mark.parametrize("blk,L", [(16, 128), (32, 640), (64, 1152), (256, 1280)])
@pytest.mark.parametrize("least", [2, 10**6])
def test_blocks_of_64_visit_the_layout_once(kind, blk, L, least, monkeypatch):
    """The backward's shares: every block of 64 rows (keys) sees its own part of the lists once, over all its parts."""
    monkeypatch.setattr(bs, "_FWD_SHARE", (1 << 20, least))
    monkeypatch.setattr(bs, "_BWD_SHARE", (1 << 20, least))
    bs._PLANS.clear()
    lay = _layout(kind, 2, blk, L)
    plan = bs.sparse_plan(lay, blk, L, 1, 2, "cpu")
    bs._PLANS.clear()
    want = (lay != 0).repeat_interleave(blk // 16, 1).repeat_interleave(blk // 16, 2)[:, :L // 16, :L // 16].long()
    for side, parts, rows, cols in ((plan.rows(), 2, 8, 4), (plan.columns(), 4, 2, 16)):
        for head in range(side.work.shape[0]):
            seen, slots = torch.zeros(L // 16, -(-L // 256) * 16, dtype=torch.long), {}
            for own, first, n, slot in side.work[head].tolist():
                if own < 0:
                    continue
                slots.setdefault(own, []).append(slot)
                blk_, part = divmod(own, parts)
                for j in range(first, first + n):
                    t, m = side.tiles[head, blk_, j].item(), side.masks[head, blk_, j].item()
                    for r in range(rows):
                        for k in range(cols):
                            if parts == 2 and r // 4 == part:
                                seen[8 * blk_ + r, 4 * t + k] += (m >> (r * cols + k)) & 1
                            elif parts == 4 and k // 4 == part:
                                seen[2 * t + r, 16 * blk_ + k] += (m >> (r * cols + k)) & 1
            assert torch.equal(seen[:, :L // 16], want[head])
            assert sorted(slots) == list(range(L // 64))
            merged = {b: list(range(s, s + n)) for b, s, n, _ in side.merges[head].tolist() if b >= 0}
            assert all(got == [-1] if b not in merged else sorted(got) == merged[b] for b, got in slots.items())
            assert all(0 <= s < side.nslots for got in merged.values() for s in got)
            assert L == 128 or bool(merged) == (least == 2)


def test_parts_of_all_heads_are_numbered_through():
    """A workspace slot per part there is: a head or two with long rows among many must not reserve as much for each of the others."""
    H, blk, L = 8, 64, 4096
    n = L // blk
    lay = torch.eye(n, dtype=torch.long).expand(H, n, n).clone()
    lay[3] = lay[5] = 1
    bs._PLANS.clear()
    plan = bs.sparse_plan(lay, blk, L, 1, H, "cpu")
    for side in (plan.forward(), plan.backward(), plan.rows(), plan.columns()):
        used = sorted(e[3] for head in side.work.tolist() for e in head if e[3] >= 0)
        assert used and used == list(range(side.nslots))
        joined = sorted(s for head in side.merges.tolist() for b, first, k, _ in head if b >= 0 for s in range(first, first + k))
        assert joined == used
    bs._PLANS.clear()


@pytest.mark.parametrize("kind", ["shared", "heads"])
def test_batch_sizes_share_the_lists(kind, monkeypatch):
    """Another batch size costs a new share of the work, not the lists and masks of the layout again."""
    H, blk, L = 2, 32, 640
    lay = _layout(kind, H, blk, L)
    bs._PLANS.clear()
    first = bs.sparse_plan(lay, blk, L, 1, H, "cpu")
    want = [side.tiles.data_ptr() for side in (first.forward(), first.backward())]

    def no_more(*_):
        raise AssertionError("lists made again")

    monkeypatch.setattr(bs, "_tile_masks", no_more)
    for B in (2, 40):
        plan = bs.sparse_plan(lay.clone(), blk, L, B, H, "cpu")
        assert [side.tiles.data_ptr() for side in (plan.forward(), plan.backward())] == want
        work, merges, nslots = bs._share_out(bs.build_lut(lay, blk, L, "cpu")[1], B * H if kind == "shared" else B, *bs._FWD_SHARE)
        assert torch.equal(plan.forward().work, work) and plan.forward().nslots == nslots
        assert [side.tiles.data_ptr() for side in (plan.rows(), plan.columns())] == want
    bs._PLANS.clear()


@pytest.mark.parametrize("kind", ["shared", "heads", "empty"])
@pytest.mark.parametrize("blk,L", [(16, 256), (32, 640), (64, 1152), (128, 1280), (256, 1280)])
def test_lists_are_those_of_the_layout(kind, blk, L):
    """The plan's lists, made from its masks, against those made from the layout."""
    lay = _layout(kind, 2, blk, L)
    plan = bs.sparse_plan(lay, blk, L, 1, 2, "cpu")
    for side, (tiles, counts) in ((plan.rows(), bs.build_lut(lay, blk, L, "cpu")[:2]), (plan.columns(), bs.build_bwd_lut(lay, blk, L, 2, "cpu")[:2])):
        listed = (side.masks != 0).sum(-1)
        for head in range(2):
            mine = min(head, side.tiles.shape[0] - 1), min(head, tiles.shape[0] - 1)
            assert torch.equal(listed[mine[0]].int(), counts[mine[1]])
            for block, n in enumerate(counts[mine[1]].tolist()):
                assert torch.equal(side.tiles[mine[0], block, :n], tiles[mine[1], block, :n])
    bs._PLANS.clear()


@pytest.mark.parametrize("shape,blk,L", [((1, 16, 16), 64, 2048), ((1, 32, 16), 64, 2048), ((1, 16, 32), 64, 2048), ((2, 32, 31), 64, 2048),
                                         ((1, 8, 8), 48, 384), ((1, 4, 4), 96, 384), ((1, 3, 3), 64, 192), ((1, 5, 5), 32, 144)])
def test_layouts_that_do_not_fit_are_refused(shape, blk, L):
    """Fewer blocks than the sequence has, blocks that do not make up tiles, sequences of no whole tiles: refused, every time."""
    bs._PLANS.clear()
    for _ in range(2):
        with pytest.raises(AssertionError):
            bs.sparse_plan(torch.ones(shape, dtype=torch.long), blk, L, 1, shape[0], "cpu").forward()
    assert not bs._PLANS


def test_a_layout_for_longer_sequences_is_cut():
    H, blk, L = 2, 32, 640
    lay = _layout("heads", H, blk, 2 * L)
    whole, cut = (bs.sparse_plan(x, blk, L, 1, H, "cpu") for x in (lay, lay[:, :L // blk, :L // blk].contiguous()))
    for a, b in ((whole.forward(), cut.forward()), (whole.rows(), cut.rows()), (whole.columns(), cut.columns())):
        assert all(torch.equal(x, y) for x, y in zip(a[:4], b[:4])) and a.nslots == b.nslots
    bs._PLANS.clear()


@pytest.mark.gpu
@pytest.mark.parametrize("D,blk,L,kind,bias", [(128, 64, 1152, "shared", False), (64, 32, 1024, "heads", True),
                                               (128, 16, 512, "empty", False), (128, 128, 1408, "shared", True)])
def test_cut_lists_match_dense_attention(D, blk, L, kind, bias, monkeypatch):
    """Lists cut after two (three) tiles, so that nearly every block is merged; rows without a key come out as zero."""
    monkeypatch.setattr(bs, "_FWD_SHARE", (1 << 20, 2))
    monkeypatch.setattr(bs, "_BWD_SHARE", (1 << 20, 3))
    bs._PLANS.clear()
    torch.manual_seed(3)
    B, H = 2, 2
    lay = _layout(kind, H, blk, L)
    q, k, v, do = (torch.randn(B, H, L, D, device="cuda").bfloat16() for _ in range(4))
    kpm = None
    if bias:
        kpm = torch.zeros(B, L, device="cuda")
        kpm[:, L - L // 4:] = -10000.0
    ins = [t.clone().requires_grad_(True) for t in (q, k, v)]
    o = bs.block_sparse_attention(*ins, lay, blk, key_padding_mask=kpm)
    got = [o, *torch.autograd.grad(o, ins, do)]
    assert bs.sparse_plan(lay, blk, L, B, H, q.device).forward().nslots > 0
    bs._PLANS.clear()
    ref_in = [t.float().requires_grad_(True) for t in (q, k, v)]
    s = ref_in[0] @ ref_in[1].transpose(-1, -2) * D**-0.5 + (0 if kpm is None else kpm[:, None, None, :])
    ok = (lay != 0).repeat_interleave(blk, 1).repeat_interleave(blk, 2)[:, :L, :L].cuda()
    p = torch.softmax(s.masked_fill(~ok, float("-inf")), -1)
    ref = torch.where(ok.any(-1)[None, :, :, None], torch.nan_to_num(p), 0.0) @ ref_in[2]
    want = [ref, *torch.autograd.grad(ref, ref_in, do.float())]
    for name, a, b in zip(("o", "dq", "dk", "dv"), got, want):
        # bf16 operands, weights and results: 2^-8 each, a few of them in a row
        err = (a.float() - torch.nan_to_num(b)).norm() / b.nan_to_num().norm()
        assert err < 0.015, (name, err.item())
