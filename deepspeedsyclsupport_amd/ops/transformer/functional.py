"""Autograd wrappers for the fused transformer kernels (training path).

Each op runs the gfx950 kernel for device tensors and the fp32 PyTorch reference for host tensors. Parity: the
fused pieces of the reference training layer (`csrc/transformer/ds_transformer_cuda.cpp:154-300`: LN, bias+GELU,
transform_0213, softmax) and inference kernels (`rms_norm.cu`, `apply_rotary_pos_emb.cu`, `gelu.cu` gated acts).
"""
import torch
import torch.nn.functional as F

from .. import reference
from ..native import hip_ops, unseen_from_python

ACT_CODES = {"silu": 0, "swiglu": 0, "gelu_tanh": 1, "gelu_new": 1, "gelu_pytorch_tanh": 1, "gelu": 2, "geglu": 2,
             "relu": 3, "reglu": 3, "identity": 4}


# --------------------------------------------------------------------------------------------------- RMSNorm
class _RMSNormFn(torch.autograd.Function):

    @staticmethod
    def forward(ctx, x, w, eps, residual):
        y, res, rstd = hip_ops().rms_fwd(x, residual, w, eps)
        h = res if residual is not None else x
        ctx.save_for_backward(h, w, rstd)
        ctx.has_res = residual is not None
        return (y, res) if ctx.has_res else y

    @staticmethod
    def backward(ctx, dy, dres=None):
        h, w, rstd = ctx.saved_tensors
        dy = dy.contiguous()
        if dres is not None:
            dres = dres.contiguous()
        dx, dw = hip_ops().rms_bwd(dy, h, w, rstd, dres)
        # d(x) == d(residual) when the forward summed them
        return dx, dw, None, (dx if ctx.has_res else None)


_NORM_BWD_MAX_H = 8192    # norm kernels: forward up to 16384 wide rows, backward up to 8192


def _norm_kernel_ok(x, *params):
    if not x.is_cuda or x.shape[-1] % 8:
        return False
    if x.shape[-1] <= _NORM_BWD_MAX_H:
        return True
    needs_grad = torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in (x, ) + params)
    return x.shape[-1] <= 16384 and not needs_grad


def rms_norm(x, weight, eps=1e-6, residual=None):
    """y = RMSNorm(x [+ residual]) * weight. With `residual`, returns (y, x + residual)."""
    if _norm_kernel_ok(x, weight, residual):
        x = x.contiguous()
        if residual is not None:
            residual = residual.contiguous()
        if unseen_from_python(x, weight, residual):
            out = hip_ops().rms_norm_node(x, weight, eps, residual)  # (the same in C++, for bf16)
            if out is not None:
                return out[0] if residual is None else tuple(out)
        return _RMSNormFn.apply(x, weight, eps, residual)
    h = x + residual if residual is not None else x
    y = (h.float() * torch.rsqrt(h.float().pow(2).mean(-1, keepdim=True) + eps) * weight.float()).to(x.dtype)
    return (y, h) if residual is not None else y


# --------------------------------------------------------------------------------------------------- LayerNorm
class _LayerNormFn(torch.autograd.Function):

    @staticmethod
    def forward(ctx, x, g, b, eps, residual):
        y, res, mean, rstd = hip_ops().ln_fwd(x, residual, g, b, eps)
        h = res if residual is not None else x
        ctx.save_for_backward(h, g, mean, rstd)
        ctx.has_res = residual is not None
        return (y, res) if ctx.has_res else y

    @staticmethod
    def backward(ctx, dy, dres=None):
        h, g, mean, rstd = ctx.saved_tensors
        dx, dg, db = hip_ops().ln_bwd(dy.contiguous(), h, g, mean, rstd,
                                      dres.contiguous() if dres is not None else None)
        return dx, dg, db, None, (dx if ctx.has_res else None)


def layer_norm(x, weight, bias, eps=1e-5, residual=None):
    if _norm_kernel_ok(x, weight, bias, residual):
        x = x.contiguous()
        if residual is not None:
            residual = residual.contiguous()
        return _LayerNormFn.apply(x, weight, bias, eps, residual)
    h = x + residual if residual is not None else x
    y = torch.nn.functional.layer_norm(h, (h.shape[-1], ), weight, bias, eps)
    return (y, h) if residual is not None else y


# --------------------------------------------------------------------------------------------------- gated act
class _GatedActFn(torch.autograd.Function):

    @staticmethod
    def forward(ctx, gu, act):
        ctx.act = act
        ctx.save_for_backward(gu)
        return hip_ops().gated_act_fwd(gu, act)

    @staticmethod
    def backward(ctx, dout):
        (gu, ) = ctx.saved_tensors
        return hip_ops().gated_act_bwd(dout.contiguous(), gu, ctx.act), None


class _GatedActKMajorFn(torch.autograd.Function):
    """Gated activation of a long token batch in training: the kernels also write the token-contiguous ("K-major")
    copies that the neighbouring linears' weight-gradient GEMMs contract over — the output's for the consumer
    (handed over as `out._ds_kmajor`), the input gradient's for the producer (`dgu._ds_kmajor`) — instead of leaving
    them to a separate transpose pass (see `ops/linear.py`)."""

    @staticmethod
    def forward(ctx, gu, act, of_out, of_grad):
        ctx.act, ctx.of_grad = act, of_grad
        ctx.save_for_backward(gu)
        if not of_out:
            return hip_ops().gated_act_fwd(gu, act), None
        out, out_t = hip_ops().gated_act_fwd_t(gu, act, 256)
        ctx.mark_non_differentiable(out_t)
        return out, out_t

    @staticmethod
    def backward(ctx, dout, _unused=None):
        (gu, ) = ctx.saved_tensors
        if not ctx.of_grad:
            return hip_ops().gated_act_bwd(dout.contiguous(), gu, ctx.act), None, None, None
        dgu, dgu_t = hip_ops().gated_act_bwd_t(dout.contiguous(), gu, ctx.act, 256)
        dgu._ds_kmajor = dgu_t
        return dgu, None, None, None


def gated_activation(gate_up, act="silu", around=None):
    """[.., 2I] = [gate | up] -> act(gate) * up  (SwiGLU for act='silu', GEGLU for 'gelu'). around: the width of the model, that is the inputs
    of the layer before and the outputs of the one behind, for what they need in training (`kmajor_of_gate`)."""
    code = ACT_CODES[act]
    if gate_up.is_cuda and (gate_up.shape[-1] // 2) % 8 == 0:
        from ..linear import kmajor_of_gate
        rows = gate_up.numel() // gate_up.shape[-1]
        if gate_up.requires_grad and torch.is_grad_enabled() and any(copies := kmajor_of_gate(rows, gate_up.dtype, gate_up.shape[-1] // 2, around)):
            out, out_t = _GatedActKMajorFn.apply(gate_up.contiguous(), code, *copies)
            if out_t is not None:
                out._ds_kmajor = out_t
            return out
        gate_up = gate_up.contiguous()
        out = hip_ops().gated_act_node(gate_up, code) if unseen_from_python(gate_up) else None
        return _GatedActFn.apply(gate_up, code) if out is None else out
    g, u = gate_up.chunk(2, dim=-1)
    return reference.ACTS[code](g) * u


def linear_gated(x, weight, act="silu"):
    """`gated_activation` of x weight^T without a gradient of its own, asked for once: in one launch where that is the faster way, else in
    two. None where torch has to see the two, or has one of them alone."""
    if not x.is_cuda or not weight.is_cuda or not unseen_from_python(x, weight):
        return None
    return hip_ops().linear_gated(x, weight, ACT_CODES[act])


class _BiasActFn(torch.autograd.Function):

    @staticmethod
    def forward(ctx, x, bias, act):
        ctx.act = act
        ctx.save_for_backward(x, bias)
        return hip_ops().bias_act_fwd(x, bias, act)

    @staticmethod
    def backward(ctx, dy):
        x, bias = ctx.saved_tensors
        dx = hip_ops().bias_act_bwd(dy.contiguous(), x, bias, ctx.act)
        db = dx.reshape(-1, dx.shape[-1]).sum(0) if bias is not None else None
        return dx, db, None


def bias_activation(x, bias, act="gelu"):
    code = ACT_CODES[act]
    if x.is_cuda and x.shape[-1] % 8 == 0:
        return _BiasActFn.apply(x.contiguous(), bias, code)
    return reference.ACTS[code](x + bias if bias is not None else x)


# --------------------------------------------------------------------------------------------------- dropout
class _DropoutFn(torch.autograd.Function):
    """y = residual + dropout_p(x + bias) in one kernel; the mask is regenerated from (seed, offset) in backward."""

    @staticmethod
    def forward(ctx, x, bias, residual, p, seed):
        (y, ) = hip_ops().dropout_fwd(x, bias, residual, p, seed, 0, False)
        ctx.p, ctx.seed, ctx.has_bias, ctx.has_res = p, seed, bias is not None, residual is not None
        return y

    @staticmethod
    def backward(ctx, dy):
        dy = dy.contiguous()
        dx = hip_ops().dropout_bwd(dy, ctx.p, ctx.seed, 0)
        db = dx.reshape(-1, dx.shape[-1]).sum(0) if ctx.has_bias else None
        return dx, db, (dy if ctx.has_res else None), None, None


def _dropout_seed():
    # drawn from the host generator: reproducible under torch.manual_seed and restored by activation
    # checkpointing's RNG stash, so a recomputed forward reproduces the same mask; no device sync
    return int(torch.randint(0, 2**62, (1, )).item())


def dropout(x, p, training=True, bias=None, residual=None):
    """residual + dropout(x + bias) (reference `csrc/transformer/dropout_kernels.cu` fused variants)."""
    if not training or p == 0.0:
        y = x if bias is None else x + bias
        return y if residual is None else y + residual
    if x.is_cuda and x.shape[-1] % 8 == 0:
        return _DropoutFn.apply(x.contiguous(), bias, None if residual is None else residual.contiguous(), float(p),
                                _dropout_seed())
    y = F.dropout(x if bias is None else x + bias, p, True)
    return y if residual is None else y + residual


# --------------------------------------------------------------------------------------------------- rotary + split
class _QKVRopeFn(torch.autograd.Function):

    @staticmethod
    def forward(ctx, qkv, cos, sin, pos, hq, hk, rot, offset, token_major=False):
        q, k, v = hip_ops().qkv_rope_fwd(qkv, cos, sin, pos, hq, hk, rot, offset, token_major)
        ctx.save_for_backward(cos, sin, pos)
        ctx.rot, ctx.offset = rot, offset
        return q, k, v

    @staticmethod
    def backward(ctx, dq, dk, dv):
        cos, sin, pos = ctx.saved_tensors
        dqkv = hip_ops().qkv_rope_bwd(dq, dk, dv, cos, sin, pos, ctx.rot, ctx.offset)
        return dqkv, None, None, None, None, None, None, None, None


def qkv_rope_split(qkv, cos, sin, num_heads, num_kv_heads, rotary_dim=None, position_ids=None, pos_offset=0,
                   token_major=False):
    """qkv [B, S, Hq+2Hk, D] -> q [B,Hq,S,D], k [B,Hk,S,D], v [B,Hk,S,D] with rotate_half RoPE on q and k.
    `token_major=True` returns them as views of [B,S,H,D] memory (what the flash-attention path exchanges with its
    backward without transposing copies).

    `cos`/`sin` are fp32 tables [max_pos, rot/2] (see `reference.rope_tables`)."""
    B, S, NH, D = qkv.shape
    rot = rotary_dim or D
    if qkv.is_cuda and D % 8 == 0 and rot % 16 == 0:
        pos = position_ids.to(torch.int32).contiguous() if position_ids is not None else None
        args = (qkv.contiguous(), cos, sin, pos, num_heads, num_kv_heads, rot, pos_offset, token_major)
        out = hip_ops().qkv_rope_node(*args) if unseen_from_python(*args[:4]) else None
        return _QKVRopeFn.apply(*args) if out is None else tuple(out)
    q, k, v = qkv.split([num_heads, num_kv_heads, num_kv_heads], dim=2)
    p = position_ids if position_ids is not None else torch.arange(pos_offset, pos_offset + S, device=qkv.device)
    q = reference.apply_rope_half(q, cos, sin, p)
    k = reference.apply_rope_half(k, cos, sin, p)
    return q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2)


def apply_rotary_pos_emb(x, cos, sin, position_ids=None, pos_offset=0, rotary_dim=None, interleaved=False,
                         inverse=False):
    """In-place RoPE on a [B, S, H, D] view (inference path; both rotate_half and GPT-J interleaved styles)."""
    rot = rotary_dim or x.shape[-1]
    if x.is_cuda:
        pos = position_ids.to(torch.int32).contiguous() if position_ids is not None else None
        hip_ops().rope_inplace(x, cos, sin, pos, rot, pos_offset, interleaved, inverse)
        return x
    B, S = x.shape[:2]
    p = position_ids if position_ids is not None else torch.arange(pos_offset, pos_offset + S)
    s = -sin if inverse else sin
    if interleaved:
        c, sn = cos[p].float()[..., None, :], s[p].float()[..., None, :]
        if c.dim() == 3:
            c, sn = c[None], sn[None]
        x1, x2 = x[..., 0:rot:2].float(), x[..., 1:rot:2].float()
        o1, o2 = x1 * c - x2 * sn, x2 * c + x1 * sn
        x[..., 0:rot:2], x[..., 1:rot:2] = o1.to(x.dtype), o2.to(x.dtype)
        return x
    x.copy_(reference.apply_rope_half(x, cos, s, p))
    return x


# --------------------------------------------------------------------------------------------------- embedding
# (no public predicate says that a call runs under a transform of torch.func, or that a backward's vectors come as a batch)
_transformed = torch._C._are_functorch_transforms_active
_batched = torch._C._functorch.is_legacy_batchedtensor


class _EmbeddingFn(torch.autograd.Function):

    @staticmethod
    def forward(ctx, ids, weight):
        ctx.save_for_backward(ids)
        ctx.save_for_forward(ids)
        ctx.rows = weight.shape[0]
        return F.embedding(ids, weight)

    @staticmethod
    def backward(ctx, dy):
        (ids, ) = ctx.saved_tensors
        if torch.is_grad_enabled() or _transformed() or _batched(dy):  # the gradient is itself differentiated, or batched: torch's own
            return None, torch.ops.aten.embedding_dense_backward(dy, ids, ctx.rows, -1, False)
        return None, hip_ops().embed_grad(dy.reshape(-1, dy.shape[-1]).contiguous(), ids.reshape(-1).contiguous(), ctx.rows)

    @staticmethod
    def jvp(ctx, _, dweight):
        (ids, ) = ctx.saved_tensors
        return F.embedding(ids, dweight)


# Tokens from which the gradient kernel pays: forward and backward of fewer take the host 63 us with this function and 47 with torch's,
# whose kernels hide behind that up to 512 tokens of 2048 or 4096 (1024 tokens: 75 and 80 us)
EMBED_GRAD_MIN = 512


def embedding(ids, weight):
    """Rows `ids` of weight, with the gradient kernel `embed_grad` (`csrc/moe/moe_kernels.hip`) for what it takes: bf16 rows of 512 to
    4096 tokens. What transforms, traces or compiles the call gets torch's operator."""
    if not (torch.jit.is_tracing() or torch.compiler.is_compiling() or _transformed()) and \
            weight.is_cuda and weight.dtype == torch.bfloat16 and weight.requires_grad and torch.is_grad_enabled() and \
            ids.dtype == torch.int64 and weight.shape[1] % 8 == 0 and weight.numel() and \
            EMBED_GRAD_MIN <= ids.numel() <= hip_ops().embed_grad_max():
        return _EmbeddingFn.apply(ids, weight)
    return F.embedding(ids, weight)


# --------------------------------------------------------------------------------------------------- cross entropy
class _XentFn(torch.autograd.Function):

    @staticmethod
    def forward(ctx, logits, labels, ignore_index, smoothing, inplace_grad):
        loss, lse = hip_ops().xent_fwd(logits, labels, ignore_index, smoothing)
        ctx.save_for_backward(logits, labels, lse)
        ctx.ignore_index, ctx.smoothing, ctx.inplace = ignore_index, smoothing, inplace_grad
        return loss

    @staticmethod
    def backward(ctx, dloss):
        logits, labels, lse = ctx.saved_tensors
        dlogits = hip_ops().xent_bwd(logits, labels, lse, dloss.contiguous(), 0.0, ctx.inplace, ctx.ignore_index,
                                     ctx.smoothing)
        return dlogits, None, None, None, None


class _XentMeanFn(torch.autograd.Function):
    """The mean over the labels that are not ignored."""

    @staticmethod
    def forward(ctx, logits, labels, ignore_index, smoothing, inplace_grad):
        mean, lse, mean_of = hip_ops().xent_mean_fwd(logits, labels, ignore_index, smoothing)
        ctx.save_for_backward(logits, labels, lse, mean_of)
        ctx.ignore_index, ctx.smoothing, ctx.inplace = ignore_index, smoothing, inplace_grad
        return mean

    @staticmethod
    def backward(ctx, dloss):
        logits, labels, lse, mean_of = ctx.saved_tensors
        dlogits = hip_ops().xent_bwd(logits, labels, lse, dloss, 0.0, ctx.inplace, ctx.ignore_index, ctx.smoothing, mean_of)
        return dlogits, None, None, None, None


XENT_MEAN_MAX = 65536


def cross_entropy(logits, labels, ignore_index=-100, label_smoothing=0.0, reduction="mean", inplace_backward=True):
    """Fused softmax-CE over [N, V] logits (bf16/fp32). `inplace_backward` reuses the logits buffer for the grad."""
    if logits.is_cuda:
        logits2 = logits.reshape(-1, logits.shape[-1])
        labels2 = labels.reshape(-1).contiguous()
        # the mean's kernel is one block: 65536 rows of 512 take 122 us forward and backward, 148 with torch's sums, 262144 of 128 455 and
        # 430
        if reduction not in ("none", "sum") and labels2.numel() <= XENT_MEAN_MAX:
            args = (logits2, labels2, ignore_index, label_smoothing, inplace_backward)
            mean = hip_ops().xent_mean_node(*args) if unseen_from_python(logits2, labels2) else None
            return _XentMeanFn.apply(*args) if mean is None else mean
        per_tok = _XentFn.apply(logits2, labels2, ignore_index, label_smoothing, inplace_backward)
    else:
        per_tok = reference.cross_entropy(logits.reshape(-1, logits.shape[-1]), labels.reshape(-1), ignore_index,
                                          label_smoothing)
        labels2 = labels.reshape(-1)
    if reduction == "none":
        return per_tok
    if reduction == "sum":
        return per_tok.sum()
    n = (labels2 != ignore_index).sum().clamp(min=1)
    return per_tok.sum() / n
