"""Block-sparse attention on the gfx950 flash kernel (reference: the Triton SDD / softmax / DSD kernels of
`ops/sparse_attention/{matmul.py:628, softmax.py:224}` driven by `sparse_self_attention.py`).

Forward: `csrc/attn/flash_fwd.hip` — every workgroup (one 128-row query block of one
head) visits only the 64-key tiles its layout rows touch, listed in a LUT built here once per (layout, sequence
length), and masks inside a tile by 16 x 16 pieces. Work and K/V traffic therefore scale with the
layout density. Head dims below 128 are zero-padded to 128 (zeros change neither QK^T nor the kept part of PV).

Backward: `csrc/attn/sparse_bwd.hip` (reference: the transposed DSD/SDD products of `matmul.py:605` and the sparse softmax
backward `softmax.py:213`), one pass by rows for dQ over the forward's lists and one by columns for dK and dV, every workgroup
64 rows (keys) of one head; the columns' lists are made here too (the 32-row query tiles that 256 keys meet). P is recomputed
from the forward's LSE. No [L, L] tensor is ever built; work scales with density.

`SparsePlan` holds what both passes read: the lists and their masks (`SparseLists`, one per layout), and how the lists are shared out
over workgroups (a row or column that is much longer than the others is cut into parts), which depends on batch and heads.
"""
from collections import namedtuple

import numpy as np
import torch

from ..native import hip_ops


def _bits(layout):
    return layout.detach().cpu().contiguous().numpy() != 0


def _plan_key(bits, blk, L, device):
    """The layout's contents (one bit per block) and what else a plan depends on."""
    return (np.packbits(bits).tobytes(), bits.shape, blk, L, str(device))


def build_lut(layout, blk, L, device):
    """layout [H, nb, nb] (0/1) -> (tiles int32 [LH, nqb, T], ntiles int32 [LH, nqb], layout uint8 [LH, nb, nb],
    qorder int32 [LH, nqb] = query blocks by descending tile count, the kernel's launch order).

    LH = 1 when every head shares one layout. Tile t of query block qb is listed when any key of 64-key tile t is
    allowed for any of the 128 query rows of qb; the tile lists are ascending. For statistics and tests: the kernels read the
    lists of `SparseLists`, which come from the masks and say the same."""
    lay = layout.to(torch.bool)
    if lay.shape[0] > 1 and bool((lay == lay[:1]).all()):
        lay = lay[:1]
    LH, nb, _ = lay.shape
    assert nb * blk >= L and L % 128 == 0 and L % blk == 0
    g = min(blk, 64)                                             # common fine grid
    fine = lay.repeat_interleave(blk // g, 1).repeat_interleave(blk // g, 2)[:, :L // g, :L // g]
    q128 = fine.reshape(LH, L // 128, 128 // g, L // g).any(2) if g < 128 else fine
    t64 = q128.reshape(LH, L // 128, L // 64, 64 // g).any(-1)  # [LH, nqb, ntile]
    ntiles = t64.sum(-1).to(torch.int32)
    T = max(int(ntiles.max()), 1)
    order = torch.sort((~t64).to(torch.int8), dim=-1, stable=True).indices[..., :T].to(torch.int32)
    qorder = torch.sort(ntiles, dim=-1, descending=True, stable=True).indices.to(torch.int32)  # heaviest first
    return (order.contiguous().to(device), ntiles.contiguous().to(device), lay.to(torch.uint8).contiguous().to(device),
            qorder.contiguous().to(device))


def build_bwd_lut(layout, blk, L, H, device):
    """Column LUT of the sparse backward: (qtiles int32 [H, nkb, T] = 32-row query tiles met by each 256-key block,
    ascending, nqt int32 [H, nkb], layout uint8 [LH, nb, nb] at granularity blk' = min(blk, 128), blk'). For tests, as above."""
    lay = layout.to(torch.bool)
    if lay.shape[0] > 1 and bool((lay == lay[:1]).all()):
        lay = lay[:1]
    if blk > 128:  # the kernel masks at <= 128-row granularity: refine the layout
        f = blk // 128
        lay = lay.repeat_interleave(f, 1).repeat_interleave(f, 2)
        blk = 128
    LH, nb, _ = lay.shape
    g = 16
    fine = lay.repeat_interleave(blk // g, 1).repeat_interleave(blk // g, 2)[:, :L // g, :L // g]
    nkb = (L + 255) // 256
    ntq = L // 32
    fine = torch.nn.functional.pad(fine, (0, nkb * 16 - fine.shape[2]))
    met = fine.reshape(LH, ntq, 2, nkb, 16).any(4).any(2)      # [LH, ntq, nkb]
    met = met.permute(0, 2, 1).contiguous()                     # [LH, nkb, ntq]
    nqt = met.sum(-1).to(torch.int32)
    T = max(int(nqt.max()), 1)
    order = torch.sort((~met).to(torch.int8), dim=-1, stable=True).indices[..., :T].to(torch.int32)
    if LH == 1 and H > 1:
        order, nqt = order.expand(H, nkb, T), nqt.expand(H, nkb)
    return order.contiguous().to(device), nqt.contiguous().to(device), lay.to(torch.uint8).contiguous().to(device), blk


# Workgroups that lists are shared out over, and the shortest part worth cutting, in tiles: by rows (64 keys), for the forward and
# dQ, and by columns (32 rows). The chip holds 512 of either at once; a part costs its operands' first load and a pass of its
# accumulators through memory, 32 to 64 KB. Measured, us, forward / forward and backward, rows over 512, 640 and 768: BigBird B2 H8
# L16384 105 / 416, 111 / 420, 114 / 424; a random 15 % B2 H8 L4096 44 / 155, 56 / 165, 60 / 169; Fixed B1 H4 L4096 of 32 tokens 54 / 172, 62 /
# 184, 62 / 184. Columns over 256 with parts of at least 8 and over 512 of 16, backward alone: 387 and 372 (BigBird), 352 and 305 (Fixed, L8192).
_FWD_SHARE, _BWD_SHARE = (512, 8), (512, 16)

PlanSide = namedtuple("PlanSide", "tiles masks work merges nslots")


def _share_out(counts, copies, slots, least, met=None):
    """counts [LH, n] list lengths; `copies` workgroups sets run side by side -> (work [LH, W, 4], merges [LH, M, 4], nslots):
    lists far longer than an equal share of all the work are cut evenly, the parts of all LH heads numbered through. Entries as in
    the kernels; -1 pads. met [LH, n, T] (numpy, bool): what counts in longer lists; a part runs from its first to its last."""
    limit = max(least, -(-int(counts.sum()) * copies // slots))
    if met is not None:   # (first, and one past the last)
        ends = np.stack([met.argmax(-1), np.where(met.any(-1), met.shape[-1] - met[..., ::-1].argmax(-1), 0)], -1).tolist()
    work, merges, used = [], [], 0
    for head, row in enumerate(counts.tolist()):
        entries, joins = [], []
        for i, n in enumerate(row):
            if n <= limit * 3 // 2:
                a, b = (0, n) if met is None else ends[head][i]
                entries.append((n, (i, a, b - a, -1)))
                continue
            parts, at = -(-n // limit), range(n) if met is None else met[head, i].nonzero()[0].tolist()
            for p in range(parts):
                a, b = n * p // parts, n * (p + 1) // parts
                entries.append((b - a, (i, at[a], at[b - 1] + 1 - at[a], used + p)))
            joins.append((i, used, parts, 0))
            used += parts
        work.append([e for _, e in sorted(entries, key=lambda e: -e[0])])   # longest first
        merges.append(joins)

    def pad(lists):
        width = max(len(x) for x in lists)
        flat = [e for x in lists for e in x + [(-1, 0, 0, -1 if lists is work else 0)] * (width - len(x))]
        return torch.tensor(flat, dtype=torch.int32).reshape(len(lists), width, 4)

    return pad(work), pad(merges), used


def _tile_masks(bits, blk, L, rows, cols):
    """Layout [LH, nb, nb] (bool) -> int32 [LH, tiles down, tiles across] for tiles of rows x cols pieces of 16 x 16 tokens (8 x 4
    or 2 x 16): bit r * cols + k is piece (r, k). Across, the last tile may reach past L: nothing is seen there."""
    f, n = blk // 16, L // 16
    seen = bits.repeat(f, 2)[:, :, :n]
    seen = np.pad(seen, ((0, 0), (0, 0), (0, -n % 16)))
    row = np.packbits(seen, axis=-1, bitorder="little")              # [LH, nb, pieces / 8]
    if cols == 4:
        row = np.stack([row & 15, row >> 4], -1).reshape(row.shape[0], row.shape[1], -1)[:, :, :n // 4]
    else:
        row = row.view("<u2")
    row = row.astype(np.uint32).repeat(f, 1)[:, :n].reshape(row.shape[0], n // rows, rows, -1)
    mask = row[:, :, 0].copy()
    for r in range(1, rows):
        mask |= row[:, :, r] << np.uint32(cols * r)
    return torch.from_numpy(mask.view(np.int32))


class SparseLists:
    """One layout's lists and masks for a sequence length, on the device, and their shares by how many copies of them run side by
    side (batch and heads); each side is made when it is first needed."""

    def __init__(self, bits, blk, L, device):
        # blocks that make up tiles of 64 evenly, and as many of them as the sequence has, both ways
        assert min(bits.shape[1:]) * blk >= L and L % 128 == 0 and L % blk == 0 and (64 % blk == 0 or blk % 64 == 0)
        self.layout, self.blk, self.L, self.device = torch.from_numpy(bits), blk, L, device
        self.lists, self.shares = {}, {}

    def _to_device(self, parts):
        flat = torch.cat([t.reshape(-1) for t in parts]).to(self.device)   # one copy
        return [t.view(p.shape) for t, p in zip(flat.split([p.numel() for p in parts]), parts)]

    def _make(self, side):
        """(tiles and masks on the device, the lists' lengths, the masks here): what a list has to do with, ascending, from the masks."""
        bits = self.layout.numpy()
        if bits.shape[0] > 1 and (bits == bits[:1]).all():
            bits = bits[:1]
        masks = _tile_masks(bits, self.blk, self.L, *((8, 4) if side == "fwd" else (2, 16))).numpy()
        if side != "fwd":
            masks = masks.transpose(0, 2, 1)   # listed by key block
        met = masks != 0
        ends = met.cumsum(-1, dtype=np.int32)
        counts = torch.from_numpy(ends[..., -1].copy())
        lists = np.zeros((2, *met.shape[:2], max(int(counts.max()), 1)), np.int32)
        head, block, tile = met.nonzero()
        at = head, block, ends[met] - 1
        lists[0][at], lists[1][at] = tile, masks[met]
        tiles, masks = torch.from_numpy(lists)
        return *self._to_device([tiles, masks]), counts, masks

    def _split(self, side, parts):
        """What blocks of 64 rows (columns), `parts` to a list, have to do with: (counts [LH, n], [LH, n, entries of the lists])."""
        masks = self.lists[side][3].numpy().view(np.uint32)
        bits = [0xffff << 16 * p if side == "fwd" else 0x000f000f << 4 * p for p in range(parts)]
        met = (masks[:, :, None] & np.array(bits, np.uint32)[:, None]) != 0
        met = met.reshape(met.shape[0], -1, met.shape[3])[:, :self.L // 64]
        return torch.from_numpy(met.sum(-1)), met

    def side(self, side, share, B, H, parts=1):
        if side not in self.lists:
            self.lists[side] = self._make(side)
        tiles, masks, counts, _ = self.lists[side]
        key = side, parts, *share, B * H if tiles.shape[0] == 1 else B
        if key not in self.shares:
            if len(self.shares) > 64:
                self.shares.clear()
            counts, met = (counts, None) if parts == 1 else self._split(side, parts)
            work, merges, nslots = _share_out(counts, key[-1], *share, met)
            self.shares[key] = (*self._to_device([work, merges]), nslots)
        return PlanSide(tiles, masks, *self.shares[key])


class SparsePlan:
    """What the kernels read for one layout, sequence length and batch x heads."""

    def __init__(self, lists, B, H):
        self.lists, self.B, self.H = lists, B, H

    def forward(self):
        return self.lists.side("fwd", _FWD_SHARE, self.B, self.H)

    def backward(self):   # (by 256 keys, whole lists: for tests; the kernels read `rows` and `columns`)
        return self.lists.side("bwd", _BWD_SHARE, self.B, self.H)

    # the same lists, shared out by blocks of 64 rows (keys): what the backward's kernels read
    def rows(self):
        return self.lists.side("fwd", _FWD_SHARE, self.B, self.H, 2)

    def columns(self):
        return self.lists.side("bwd", _BWD_SHARE, self.B, self.H, 4)


_PLANS = {}


def sparse_plan(layout, blk, L, B, H, device):
    bits = _bits(layout)
    key = _plan_key(bits, blk, L, device)
    lists = _PLANS.get(key)
    if lists is None:
        if len(_PLANS) > 64:
            _PLANS.clear()
        lists = _PLANS[key] = SparseLists(bits, blk, L, device)
    return SparsePlan(lists, B, H)


def token_bias(layout, blk, L, H, dtype, device):
    """Additive [1, H, L, L] bias: 0 where the layout allows, -inf elsewhere. Reference semantics for tests and
    host fallbacks only — the kernels never build it."""
    lay = layout.to(torch.bool)
    tok = lay.repeat_interleave(blk, 1).repeat_interleave(blk, 2)[:, :L, :L].to(device)
    if tok.shape[0] == 1 and H > 1:
        tok = tok.expand(H, L, L)
    return torch.zeros((1, H, L, L), dtype=dtype, device=device).masked_fill_(~tok[None], float("-inf"))


class BlockSparseAttnFn(torch.autograd.Function):
    """q/k/v bf16 [B, H, L, D], L a multiple of 128; kbias [B, L] / abias [L, L] / rpe [H or 1, L, L] are optional
    fp32 additive biases on the scaled scores, applied inside the kernels (no gradient flows to them, as in the
    reference's sparse softmax)."""

    @staticmethod
    def forward(ctx, q, k, v, layout, blk, scale, kbias, abias, rpe):
        B, H, L, D = q.shape
        plan = sparse_plan(layout, blk, L, B, H, q.device)
        if D < 128:
            pad = (0, 128 - D)
            qp, kp, vp = (torch.nn.functional.pad(t, pad) for t in (q, k, v))
        else:
            qp, kp, vp = q, k, v
        need_grad = any(t.requires_grad for t in (q, k, v))
        o, lse = hip_ops().flash_fwd_sparse(qp, kp, vp, float(scale), *plan.forward(), need_grad, kbias, abias, rpe,
                                            check_plan=False)
        o_full = o
        if D < 128:
            o = o[..., :D]
        if need_grad:
            ctx.save_for_backward(q, k, v, o_full, lse, *[t for t in (kbias, abias, rpe) if t is not None])
            ctx.has_bias = (kbias is not None, abias is not None, rpe is not None)
            ctx.plan, ctx.scale = plan, float(scale)
        return o

    @staticmethod
    def backward(ctx, do):
        q, k, v, o, lse, *bias = ctx.saved_tensors
        it = iter(bias)
        kbias, abias, rpe = (next(it) if has else None for has in ctx.has_bias)
        B, H, L, D = q.shape
        if D < 128:
            pad = (0, 128 - D)
            q, k, v, do = (torch.nn.functional.pad(t, pad) for t in (q, k, v, do))
        elif do.stride(-1) != 1 or any(s % 8 for s in do.stride()[:3]):
            do = do.contiguous()
        rows, cols = ctx.plan.rows(), ctx.plan.columns()
        dq, dk, dv = hip_ops().sparse_bwd(q, k, v, o, lse, do, ctx.scale, rows[:4], rows.nslots, cols[:4], cols.nslots, kbias, abias,
                                          rpe, check_plan=False)
        if D < 128:
            dq, dk, dv = dq[..., :D], dk[..., :D], dv[..., :D]
        return dq, dk, dv, None, None, None, None, None, None


def native_ok(q, k, v, blk):
    """Can the gfx950 block-sparse kernels take these tensors? (16-bit device tensors, same shapes, head dim <= 128;
    fp16 runs in bf16; sequence lengths that are not a multiple of 128 are padded with masked keys)"""
    B, H, L, D = q.shape
    return (q.is_cuda and q.dtype in (torch.bfloat16, torch.float16) and k.dtype == q.dtype and v.dtype == q.dtype
            and k.shape == q.shape and v.shape == q.shape and D <= 128 and D % 8 == 0 and L % blk == 0
            and blk in (16, 32, 64, 128, 256))


def _additive(mask, mode, shape_tail):
    """Mask in 'add' mode is added as is; in 'mul' mode 0 drops (-inf) and anything else keeps (0)."""
    m = mask.to(torch.float32)
    if mode == "mul":
        m = torch.where(m != 0, torch.zeros_like(m), torch.full_like(m, float("-inf")))
    return m.reshape(*shape_tail)


def block_sparse_attention(q, k, v, layout, blk, scale=None, key_padding_mask=None, attn_mask=None, rpe=None,
                           key_padding_mask_mode="add", attn_mask_mode="mul"):
    """q/k/v [B, H, L, D] bf16 (fp16 accepted: computed in bf16), layout [H or 1, L/blk, L/blk] ->
    softmax(QK^T*scale + rpe + key_padding_mask + attn_mask, masked by layout) V. The masks and the relative
    position embedding are applied inside the kernels (reference `ops/sparse_attention/softmax.py:37-157`); no
    [B, H, L, L] tensor is built. L only needs to be a multiple of the block size: it is padded to a multiple of 128
    with keys masked out through the per-key bias."""
    B, H, L, D = q.shape
    scale = D**-0.5 if scale is None else scale
    out_dtype = q.dtype
    if q.dtype != torch.bfloat16:
        q, k, v = q.to(torch.bfloat16), k.to(torch.bfloat16), v.to(torch.bfloat16)
    kb = _additive(key_padding_mask, key_padding_mask_mode, (B, L)) if key_padding_mask is not None else None
    ab = _additive(attn_mask, attn_mask_mode, (L, L)) if attn_mask is not None else None
    rp = rpe.to(torch.float32).reshape(-1, L, L) if rpe is not None else None
    Lp = -(-L // 128) * 128
    if Lp != L:
        padn = Lp - L
        q, k, v = (torch.nn.functional.pad(t, (0, 0, 0, padn)) for t in (q, k, v))
        kb = torch.nn.functional.pad(kb if kb is not None else q.new_zeros((B, L), dtype=torch.float32), (0, padn),
                                     value=float("-inf"))
        if ab is not None:
            ab = torch.nn.functional.pad(ab, (0, padn, 0, padn))
        if rp is not None:
            rp = torch.nn.functional.pad(rp, (0, padn, 0, padn))
        nb = layout.shape[1]
        nbp = -(-Lp // blk)
        if nbp > nb:  # padded query rows / keys get their own diagonal blocks (the keys are masked by kbias)
            lay = torch.zeros(layout.shape[0], nbp, nbp, dtype=layout.dtype)
            lay[:, :nb, :nb] = layout
            for i in range(nb, nbp):
                lay[:, i, i] = 1
            layout = lay
    kb, ab, rp = (None if t is None else t.contiguous() for t in (kb, ab, rp))
    out = BlockSparseAttnFn.apply(q, k, v, layout, blk, scale, kb, ab, rp)
    if Lp != L:
        out = out[:, :, :L]
    return out if out.dtype == out_dtype else out.to(out_dtype)
