"""bf16 linear layers for decode: the weight stored once in MFMA operand order (`csrc/gemv/skinny_bf16_sh.hip`).

Reference counterpart (behaviour): the bf16 / fp16 decode GEMMs of `transformer_inference` (`qkv_gemm`,
`vector_matmul`, `mlp_gemm`, `csrc/transformer/inference/csrc/pt_binding.cpp`) on the row-major weight.

A decode GEMM is a weight stream; read from a row-major matrix the MFMA operand layout is 16 rows x 64 B per load
instruction, which holds the stream at 3 - 4.2 TB/s. Inference weights are constants, so — as for the int8 / int4
streams (`ops/int8_gemv.py`) — the matrix is re-laid ONCE:

    wsh[nb, kq, h, lane, :] = w[16 nb + (lane % 16), 64 kq + 16 (lane // 16) + 8 h : +8]      (2 KB per 16 x 64 tile)

and every 16-byte-per-lane load reads 1 KB contiguous. The norm of a product's input, bias, residual and
activation are part of it (`DecodeProduct.finish`): one launch each, two where a wide batch cuts K into parts. With more than `MAX_DECODE_ROWS` token rows (prefill) the
library GEMM runs on a row-major matrix: the copy kept next to the shuffled one when `keep_row_major` (twice the weight
memory, sized for 288 GB of HBM), else a temporary un-shuffled right before the GEMM.
"""
import torch
import torch.nn.functional as F

from . import reference
from .native import hip_ops

# Rows up to which a decoder layer's products take the stream. Every workgroup reads all of x, so the library's blocking wins
# from there on: layer of a 4096-wide, 14336-deep Llama, 40 rows 110 us against 143 + 17 for its norms and activation, 64 rows
# (K uncut) 163 against 131 + 17.
MAX_DECODE_ROWS = 48


def decode_rows_ok(x, bias=None):
    """Whether x [.., K] is a decode-sized bf16 batch on the GPU."""
    return x.is_cuda and x.dtype == torch.bfloat16 and 0 < x.numel() // x.shape[-1] <= MAX_DECODE_ROWS and \
        (bias is None or bias.dtype == torch.bfloat16)


def preshuffle16(w):
    """Row-major bf16 w [N, K] -> wsh [NB, K/64, 2, 64, 8], N padded to NB * 16 rows with zeros."""
    N, K = w.shape
    if K % 64:
        raise ValueError(f"preshuffle16 needs K a multiple of 64 (K={K})")
    nb = (N + 15) // 16
    if nb * 16 != N:
        w = F.pad(w, (0, 0, 0, nb * 16 - N))
    # [nb, r, kq, g, h, j] -> [nb, kq, h, g, r, j]  (lane = 16 g + r)
    return w.reshape(nb, 16, K // 64, 4, 2, 8).permute(0, 2, 4, 3, 1, 5).reshape(nb, K // 64, 2, 64, 8).contiguous()


def unshuffle16(wsh, N):
    """Inverse of `preshuffle16` (any device, PyTorch ops)."""
    nb, kq = wsh.shape[0], wsh.shape[1]
    return wsh.reshape(nb, kq, 2, 4, 16, 8).permute(0, 4, 1, 3, 2, 5).reshape(nb * 16, kq * 64)[:N].contiguous()


class Bf16Weight:
    """A bf16 weight [N, K] kept in the pre-shuffled decode layout (and, optionally, row-major for prefill)."""

    def __init__(self, w, keep_row_major=False):
        self.shape = w.shape
        self.dtype = w.dtype
        self.wsh = preshuffle16(w)
        self.row_major = w.contiguous() if keep_row_major else None

    @staticmethod
    def supported(w):
        return w.dim() == 2 and w.dtype == torch.bfloat16 and w.shape[1] % 64 == 0

    def nbytes(self):
        return (self.wsh.numel() + (0 if self.row_major is None else self.row_major.numel())) * 2

    def materialize(self, dtype=None):
        if self.row_major is not None:
            w = self.row_major
        elif self.wsh.is_cuda:
            w = hip_ops().unshuffle_sh16(self.wsh, self.shape[0])
        else:
            w = unshuffle16(self.wsh, self.shape[0])
        return w if dtype in (None, w.dtype) else w.to(dtype)

    def raw(self, x, bias=None):
        """x . w^T + bias, launched by `DecodeProduct.finish`; `decode_rows_ok(x, bias)` must hold."""
        return DecodeProduct(self, x, bias)

    def linear(self, x, bias=None):
        if decode_rows_ok(x, bias):
            return self.raw(x, bias).finish()
        return F.linear(x, self.materialize(x.dtype), bias)


class DecodeProduct:
    """A decode-sized product that waits for what is fused into it."""

    def __init__(self, weight, x, bias=None):
        self.weight, self.x, self.bias = weight, x, bias

    def finish(self, norm=None, residual=None, act=None, gated=False):
        """act(rms_norm(x) . w^T + bias) + residual in one call: `norm` (weight, eps) of the input, `act` an activation code,
        `gated`: w is [gate | up] (N % 32 == 0) and the result act(gate) up."""
        x, N = self.x, self.weight.shape[0]
        norm_w, eps = norm or (None, 0.0)
        cols = N // 2 if gated else N
        r = None if residual is None else residual.reshape(-1, cols).contiguous()
        y = hip_ops().decode_gemm(x.reshape(-1, x.shape[-1]).contiguous(), self.weight.wsh, N, self.bias, norm_w, eps, r, gated,
                                  -1 if act is None else act)
        return y.view(*x.shape[:-1], cols)

    def finalize(self):
        return self.finish()

    def finalize_rms(self, residual, weight, eps):
        """-> (RMSNorm(product + residual) * weight, product + residual)"""
        from .transformer.functional import rms_norm
        y = self.finish(residual=residual)
        return rms_norm(y, weight, eps), y

    def finalize_gated(self, act_code):
        """-> act(gate) * up of a fused [gate | up] projection"""
        if self.weight.shape[0] % 32 == 0:
            return self.finish(act=act_code, gated=True)
        bias = None if self.bias is None else self.bias.float()  # halves that are no whole blocks: unfused, in fp32 as well
        gate, up = F.linear(self.x.float(), self.weight.materialize(torch.float32), bias).chunk(2, -1)
        return (reference.ACTS[act_code](gate) * up).to(self.x.dtype)
