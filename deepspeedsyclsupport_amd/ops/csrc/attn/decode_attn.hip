// Paged (blocked-KV) decode attention for inference, CDNA4 (gfx950).
//
// Parity: reference v1 `softmax_context` over the in-workspace KV cache (`csrc/transformer/inference/csrc/
// pt_binding.cpp:434-557`, `softmax.cu` attn_softmax_v2 with alibi / causal) and v2 `flash_attn_by_atoms` over the
// blocked KV cache (`inference/v2/kernels/ragged_ops/blocked_flash`). One kernel serves both engines: a contiguous
// per-sequence cache is the special case "one block of max_len tokens per sequence".
//
// Every cached K and V byte is read once per token, but a step's caches are a few MB: what bounds it is the chain of latencies.
//  * grid = (batch, kv_head, split): each workgroup reads ONE kv head's K/V for a contiguous slice of the sequence
//    once and serves all G = Hq/Hk query heads of that GQA group from it (no K/V re-read per query head);
//  * eight waves take alternating groups of 16 keys, each with its own running maxima, sums and accumulators, and meet once, at
//    the end. Scores are one MFMA tile, K . Q^T with the group's heads as columns (bf16 products, fp32 sums: what the vector
//    units gave, at a fraction of their instructions); P . V stays on the vector units, with P in fp32: V rows are read
//    whole, LPR lanes a row, and a row's probabilities reach its lanes through LDS. K and V of a group are loaded together
//    (held a group ahead they cost the second workgroup of a CU, and time: 48 x 190 keys 16 us for 12);
//  * where a workgroup a (sequence, head) leaves half of the CUs idle, two share its values (`launch_decode`);
//  * a sequence is split only when that is long for one workgroup (see `ds_paged_decode_splits`): partial (max, sum,
//    unnormalised acc) per split are merged by a small combine kernel (log-sum-exp). (An in-kernel last-block merge was
//    measured 2x slower: the device-scope fences it needs write back L2.)
// Measured, us (a workgroup of four waves per 64 to 1024 keys, scores and softmax in LDS between barriers; the read at 6.5 TB/s), 8
// kv heads of 128: 1 sequence of 130 keys, 4 heads each 6 (14; 0.1), 1 of 8192 19 (44; 5), 12 of 700, 2 heads each 10 (20; 5),
// 48 of 190, 4 each 12 (24; 6), 48 of 1024 42 (74; 31), 256 of 512 96 (183; 83). A step's rotation and append in it: 0.5 to 1 us, a
// kernel of their own 4 to 8.
// Optional ALiBi slopes (BLOOM) are applied on the fly. With a sliding window (Mistral) or chunked visibility only the
// keys in sight are split and read. A second instantiation takes key and value widths of their own (multiples of 8), a
// tanh score cap, a softmax sink per head, a gate per token and head, and GQA groups of any size.
#include "../include/ds_hip.h"

namespace {

constexpr int WAVES = 8, THREADS = 64 * WAVES;
constexpr int MAXG = 8;          // query heads per kv head handled per workgroup (GQA group)
constexpr int KEYS = 16;         // keys a wave takes at once
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

struct DecodeArgs {
  const bf16* q;           // [B, Hq, dk]; NEW: [B, Hq + 2 Hk, dk], a step's q, k and v as projected
  bf16* kc;                // [NB, Hk, BS, dk]
  bf16* vc;                // [NB, Hk, BS, dv]
  const int* block_table;  // [B, max_blocks]
  const int* seq_lens;     // [B]
  const float* alibi;      // [Hq] or null
  float* part_acc;         // [B, Hq, S, dv]  (only if S > 1)
  float* part_ml;          // [B, Hq, S, 2]
  bf16* out;               // [B, Hq, dv], rows ldo apart (written directly when S == 1)
  const float* sink;
  const bf16* gate;
  int64_t ldg, ldo;
  int Hq, Hk, BS, bs_shift, max_blocks, chunk, window, mask_chunk, dk, dv;  // bs_shift: log2 BS, or -1
  float scale, softcap;
  const float *cosT, *sinT;  // NEW: [positions, rot / 2]
  const int* pos;            // [B]
  int rot, interleaved;
};

// Elements 8 c .. + 7 of a head, the first `rot` of them turned by cs, sn [rot / 2]: pairs (i, i + rot / 2), or (2 i, 2 i + 1)
__device__ __forceinline__ bf16x8_t rope_chunk(const bf16* head, int chunk, const float* cs, const float* sn, int rot, int interleaved) {
  const int d = 8 * chunk, half = rot / 2;
  const bf16x8_t x = *reinterpret_cast<const bf16x8_t*>(head + d);
  if (d >= rot) return x;
  const bool low = d < half;
  const int i = interleaved ? d / 2 : low ? d : d - half;
  const bf16x8_t y = *reinterpret_cast<const bf16x8_t*>(head + (interleaved ? d : low ? d + half : i));
  f32x4 c[2], s[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int at = min(i + 4 * e, half - 4);  // (pairs that stand together need the first four only)
    c[e] = *reinterpret_cast<const f32x4*>(cs + at);
    s[e] = *reinterpret_cast<const f32x4*>(sn + at);
  }
  bf16x8_t r;
  if (interleaved) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a = (float)x[2 * j], b = (float)x[2 * j + 1];
      r[2 * j] = (bf16)(a * c[0][j] - b * s[0][j]);
      r[2 * j + 1] = (bf16)(b * c[0][j] + a * s[0][j]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float turn = (float)y[j] * s[j >> 2][j & 3];
      r[j] = (bf16)((float)x[j] * c[j >> 2][j & 3] + (low ? -turn : turn));
    }
  }
  return r;
}

// DK, DV: the widths; 0: given at run time. LPR: lanes that hold a row, 8 elements each (the width / 8 rounded up to a power of two). GT: at least the query heads served. NEW: the step's
// projection comes as it is: queries are turned here, and the last key and value are taken from it and written to the cache.
// VP: workgroups that share a head's values, each with all of its keys.
template <int DK, int DV, int GT, int LPR, bool NEW, int VP>
__global__ void __launch_bounds__(THREADS, 2) paged_decode_kernel(DecodeArgs a) {
  constexpr bool EXT = DK == 0;
  static_assert(EXT || (DK % 16 == 0 && DK >= 64 && DK <= 256 && DK == DV), "head dim");
  static_assert(VP == 1 || (!EXT && DV == 8 * LPR), "values in parts");
  const int dk = EXT ? a.dk : DK, dv = EXT ? a.dv : DV / VP, ldv = dv * VP;
  // [WAVES][GT][dv] accumulators, [WAVES][GT][2] maxima and sums, [WAVES][KEYS + 1][GT] probabilities and the fade of what was;
  // NEW: [GT + 2][dk] rows of the step
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int b = blockIdx.x, kh = EXT ? blockIdx.y % a.Hk : blockIdx.y, split = blockIdx.z / VP, S = gridDim.z / VP, v0 = blockIdx.z % VP * dv;
  const int g0 = EXT ? blockIdx.y / a.Hk * MAXG : 0;          // first query head of the group this block serves
  const int GA = a.Hq / a.Hk, G = EXT ? min(MAXG, GA - g0) : GA, h0 = kh * GA + g0;
  const int T = a.seq_lens[b];
  int tlo = a.window > 0 ? max(0, T - a.window) : 0;          // first key in sight
  if (a.mask_chunk > 0) tlo = max(tlo, (T - 1) / a.mask_chunk * a.mask_chunk);
  const int t0 = tlo + split * a.chunk, t1 = min(NEW ? T - 1 : T, t0 + a.chunk);  // (of the keys in the cache)
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);

  // scores: lane (l16, q4) brings key l16 and holds those of head l16 with keys 4 q4 .. + 3; chunk 4 kk + q4 of 8 elements goes
  // into MFMA kk (surplus chunks: a zero query, the row's last chunk again)
  constexpr int KK = (LPR + 3) / 4;
  const int l16 = lane & 15, q4 = lane >> 4;
  bf16x8_t qf[KK];
  const bool mine = l16 < G;
  if constexpr (!NEW) {
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
      qf[kk] = *reinterpret_cast<const bf16x8_t*>(a.q + ((int64_t)b * a.Hq + h0 + min(l16, G - 1)) * dk + min(4 * kk + q4, dk / 8 - 1) * 8);
  }
  const float slope = !EXT && a.alibi && mine ? a.alibi[h0 + l16] : 0.f;
  // values: lanes cover one row, 8 elements each
  constexpr int LV = LPR / VP, RPW = 64 / LV, UV = KEYS / RPW;  // lanes of a row, rows per wave instruction, instructions
  const int sub = lane / LV, li = lane % LV, lv = min(li, dv / 8 - 1);
  float acc[GT][8], m = -INFINITY, l = 0.f;                   // m, l: of head l16
#pragma unroll
  for (int g = 0; g < GT; ++g)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[g][j] = 0.f;
  float* ml = sm + WAVES * GT * dv;
  float* pw = ml + WAVES * GT * 2 + wid * (KEYS + 1) * GT;

  constexpr int STEP = WAVES * KEYS;
  const int* bt = a.block_table + (int64_t)b * a.max_blocks;
  struct Group {
    bf16x8_t k[KK], v[UV];
  };
  struct Blocks {
    int k, v[UV];
  };
  // (keys past the end read the last one again)
  auto blocks = [&](int t, Blocks& blk) {
    auto of = [&](int key) {
      const int tc = min(key, t1 - 1);
      return bt[a.bs_shift >= 0 ? tc >> a.bs_shift : tc / a.BS];
    };
    blk.k = of(t + l16);
#pragma unroll
    for (int u = 0; u < UV; ++u) blk.v[u] = of(t + u * RPW + sub);
  };
  auto load = [&](int t, const Blocks& blk, Group& f) {
    auto row = [&](int key, int block) {
      const int tc = min(key, t1 - 1), off = a.bs_shift >= 0 ? tc & (a.BS - 1) : tc % a.BS;
      return ((int64_t)block * a.Hk + kh) * a.BS + off;
    };
    const bf16* kr = a.kc + row(t + l16, blk.k) * dk;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) f.k[kk] = *reinterpret_cast<const bf16x8_t*>(kr + min(4 * kk + q4, dk / 8 - 1) * 8);
#pragma unroll
    for (int u = 0; u < UV; ++u) f.v[u] = *reinterpret_cast<const bf16x8_t*>(a.vc + row(t + u * RPW + sub, blk.v[u]) * ldv + v0 + lv * 8);
  };
  auto attend = [&](int t, int t1, const Group& f) {
    f32x4 s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.k[kk], qf[kk], s, 0, 0, 0);
    float mx = m;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = t + 4 * q4 + i;
      float x = s[i] * a.scale;
      if (!EXT && a.alibi) x += slope * (float)(key - (T - 1));
      if (EXT && a.softcap > 0.f) x = a.softcap * tanhf(x / a.softcap);
      s[i] = key < t1 ? x : -INFINITY;
      mx = fmaxf(mx, s[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float ref = mx == -INFINITY ? 0.f : mx, fade = __expf(m - ref);
    m = mx;
    l *= fade;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float p = __expf(s[i] - ref);
      l += p;
      if (l16 < GT) pw[(4 * q4 + i) * GT + l16] = p;
    }
    if (lane < GT) pw[KEYS * GT + lane] = fade;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int g = 0; g < GT; ++g) {
      const float w = pw[KEYS * GT + g];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[g][j] *= w;
    }
#pragma unroll
    for (int u = 0; u < UV; ++u) {
      if (t + u * RPW + sub >= t1) continue;
      float p[GT];
#pragma unroll
      for (int g = 0; g < GT; ++g) p[g] = pw[(u * RPW + sub) * GT + g];
#pragma unroll
      for (int g = 0; g < GT; ++g)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[g][j] = fmaf(p[g], (float)f.v[u][j], acc[g][j]);
    }
    __builtin_amdgcn_wave_barrier();
  };
  // NEW: a thread turns one chunk of a query or of the key (the value's stay as they are) for all waves (turned by each wave for
  // itself, a step took 2 to 4 us more)
  bf16* rows = reinterpret_cast<bf16*>(sm + WAVES * GT * (dv + 2 + KEYS + 1));  // [G queries, key, value][dk]
  const int own = T - 1 - t0;
  const bool last = NEW && own >= 0 && own < a.chunk;                          // this split holds the step's own key
  if constexpr (NEW) {
    const int cpr = dk / 8, row = tid / cpr, c = tid % cpr;
    if (row < G + 2) {
      const int head = row < G ? h0 + row : row == G ? a.Hq + kh : a.Hq + a.Hk + kh, rot = row <= G ? a.rot : 0;
      const int64_t p = a.rot ? (int64_t)a.pos[b] * (a.rot / 2) : 0;
      const bf16x8_t x = rope_chunk(a.q + ((int64_t)b * (a.Hq + 2 * a.Hk) + head) * dk, c, a.cosT + p, a.sinT + p, rot, a.interleaved);
      *reinterpret_cast<bf16x8_t*>(rows + row * dk + c * 8) = x;
      if (last && row >= G && v0 == 0) {
        const int block = bt[a.bs_shift >= 0 ? (T - 1) >> a.bs_shift : (T - 1) / a.BS];
        const int64_t at = ((int64_t)block * a.Hk + kh) * a.BS + (a.bs_shift >= 0 ? (T - 1) & (a.BS - 1) : (T - 1) % a.BS);
        *reinterpret_cast<bf16x8_t*>((row == G ? a.kc : a.vc) + at * dk + c * 8) = x;
      }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
      qf[kk] = *reinterpret_cast<const bf16x8_t*>(rows + min(l16, G - 1) * dk + min(4 * kk + q4, dk / 8 - 1) * 8);
  }
#pragma unroll
  for (int kk = 0; kk < KK; ++kk)
    if (4 * kk + q4 >= dk / 8 || !mine) qf[kk] = bf16x8_t{};
  Group f;
  int t = t0 + wid * KEYS;
  if (t < t1) {
    Blocks blk;
    blocks(t, blk);
    for (; t < t1; t += STEP) {
      load(t, blk, f);
      blocks(t + STEP, blk);
      __builtin_amdgcn_sched_barrier(0);
      attend(t, t1, f);
    }
  }
  if (last && wid == (own + KEYS - 1) / KEYS % WAVES) {  // the step's own key, by the wave with the fewest others
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) f.k[kk] = *reinterpret_cast<const bf16x8_t*>(rows + G * dk + min(4 * kk + q4, dk / 8 - 1) * 8);
#pragma unroll
    for (int u = 0; u < UV; ++u) f.v[u] = *reinterpret_cast<const bf16x8_t*>(rows + (G + 1) * dk + v0 + lv * 8);
    attend(T - 1, T, f);
  }
  // ---- the lane groups of a wave meet in registers (they share their maxima), the waves in LDS
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (lane < GT) {
    ml[(wid * GT + lane) * 2] = m;
    ml[(wid * GT + lane) * 2 + 1] = l;
  }
#pragma unroll
  for (int g = 0; g < GT; ++g) {
    if (g >= G) break;
#pragma unroll
    for (int o = LV; o < 64; o *= 2)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[g][j] += __shfl_xor(acc[g][j], o, 64);
    if (sub == 0 && li < dv / 8) {
#pragma unroll
      for (int j = 0; j < 8; ++j) sm[(wid * GT + g) * dv + li * 8 + j] = acc[g][j];
    }
  }
  __syncthreads();
  for (int i = tid; i < G * dv; i += THREADS) {
    const int g = i / dv, d = i % dv, hq = h0 + g;
    float mx = -INFINITY, num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) mx = fmaxf(mx, ml[(w * GT + g) * 2]);
    const float ref = mx == -INFINITY ? 0.f : mx;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float f = __expf(ml[(w * GT + g) * 2] - ref);
      num = fmaf(f, sm[(w * GT + g) * dv + d], num);
      den = fmaf(f, ml[(w * GT + g) * 2 + 1], den);
    }
    if (S == 1) {
      float r = den > 0.f ? num / den : 0.f;
      if (EXT && a.sink) {  // in the frame of the larger of the two
        const float mn = fmaxf(mx, a.sink[hq]), f = __expf(mx - mn);
        r = num * f / fmaf(den, f, __expf(a.sink[hq] - mn));
      }
      if (EXT && a.gate) r /= 1.f + __expf(-(float)a.gate[b * a.ldg + hq]);
      a.out[(int64_t)b * a.ldo + hq * ldv + v0 + d] = (bf16)r;
    } else {
      const int64_t at = ((int64_t)b * a.Hq + hq) * S + split;
      a.part_acc[at * ldv + v0 + d] = num;
      if (v0 + d == 0) {
        a.part_ml[at * 2] = mx;
        a.part_ml[at * 2 + 1] = den;
      }
    }
  }
}

// blockDim.x = D, the value width
__global__ void __launch_bounds__(256) combine_kernel(const float* __restrict__ part_acc,
                                                      const float* __restrict__ part_ml, bf16* __restrict__ out,
                                                      const float* __restrict__ sink, const bf16* __restrict__ gate,
                                                      int64_t ldg, int Hq, int64_t ldo, int S) {
  const int bh = blockIdx.x, d = threadIdx.x, D = blockDim.x;
  const float sk = sink ? sink[bh % Hq] : -INFINITY;
  float M = sk;
  for (int s = 0; s < S; ++s) M = fmaxf(M, part_ml[((int64_t)bh * S + s) * 2]);
  float num = 0.f, den = sink ? __expf(sk - M) : 0.f;
  for (int s = 0; s < S; ++s) {
    const float m = part_ml[((int64_t)bh * S + s) * 2], l = part_ml[((int64_t)bh * S + s) * 2 + 1];
    if (m == -INFINITY) continue;
    const float w = __expf(m - M);
    num = fmaf(w, part_acc[((int64_t)bh * S + s) * D + d], num);
    den = fmaf(w, l, den);
  }
  if (gate) den *= 1.f + __expf(-(float)gate[bh / Hq * ldg + bh % Hq]);
  out[bh / Hq * ldo + bh % Hq * D + d] = (bf16)(den > 0.f ? num / den : 0.f);
}

// Write new K/V rows into the paged cache: k,v [B, n_new, Hk, D] token-major; positions start at seq_lens_before[b].
__global__ void __launch_bounds__(256) kv_append_kernel(const bf16* __restrict__ k, const bf16* __restrict__ v,
                                                        bf16* __restrict__ kc, bf16* __restrict__ vc,
                                                        const int* __restrict__ block_table,
                                                        const int* __restrict__ start_pos, int B, int n_new, int Hk,
                                                        int D, int BS, int max_blocks) {
  const int64_t vec_per_row = D / 8;
  const int64_t total = (int64_t)B * n_new * Hk * vec_per_row;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int cvec = (int)(i % vec_per_row);
    int64_t r = i / vec_per_row;
    const int h = (int)(r % Hk);
    r /= Hk;
    const int j = (int)(r % n_new), b = (int)(r / n_new);
    const int t = start_pos[b] + j;
    const int blk = block_table[(int64_t)b * max_blocks + t / BS], off = t % BS;
    const int64_t src = (((int64_t)b * n_new + j) * Hk + h) * D + cvec * 8;
    const int64_t dst = (((int64_t)blk * Hk + h) * BS + off) * D + cvec * 8;
    *reinterpret_cast<bf16x8*>(kc + dst) = *reinterpret_cast<const bf16x8*>(k + src);
    *reinterpret_cast<bf16x8*>(vc + dst) = *reinterpret_cast<const bf16x8*>(v + src);
  }
}

// Fused QKV epilogue for inference: split the fused projection output, apply RoPE (rotate-half or GPT-J interleaved,
// partial rotary dims allowed) to q and k, write q [T, Hq, D] and scatter k/v straight into the paged cache
// (optionally also returning contiguous k/v for the prefill attention). Replaces split + 3 copies + 2 RoPE launches
// + kv_append. One thread per 8 elements, a token's in adjacent workgroups; token t belongs to sequence t / n_new at cache slot
// start_pos[b] + t % n_new, or (ragged) to seq_ids[t] at slot pos[t]. Bound by its read and write: 8192 tokens, 32 + 2 x 8 heads of
// 128: 41 us, 4.9 TB/s (one thread per pair, four 2-byte accesses each: 125).
__global__ void __launch_bounds__(256) qkv_rope_rows_kernel(
    const bf16* __restrict__ qkv, const float* __restrict__ cosT, const float* __restrict__ sinT,
    const int* __restrict__ pos, bf16* __restrict__ q_out, bf16* __restrict__ k_out, bf16* __restrict__ v_out,
    bf16* __restrict__ kc, bf16* __restrict__ vc, const int* __restrict__ block_table,
    const int* __restrict__ start_pos, const int* __restrict__ seq_ids, int n_new, int Hq, int Hk, int D, int rot,
    int interleaved, int BS, int max_blocks) {
  const int H3 = Hq + 2 * Hk, cpr = D / 8, t = blockIdx.x;
  const int i = blockIdx.y * 256 + threadIdx.x, h = i / cpr, c = i % cpr;
  if (h >= H3) return;
  const bf16* head = qkv + ((int64_t)t * H3 + h) * D;
  const int p = pos[t];
  const bf16x8_t x = rope_chunk(head, c, cosT + (int64_t)p * (rot / 2), sinT + (int64_t)p * (rot / 2), h < Hq + Hk ? rot : 0, interleaved);
  if (h < Hq) {
    *reinterpret_cast<bf16x8_t*>(q_out + ((int64_t)t * Hq + h) * D + c * 8) = x;
    return;
  }
  const bool isk = h < Hq + Hk;
  const int kh = isk ? h - Hq : h - Hq - Hk, b = seq_ids ? seq_ids[t] : t / n_new;
  const int slot = seq_ids ? p : start_pos[b] + t % n_new;
  const int blk = block_table[(int64_t)b * max_blocks + slot / BS];
  *reinterpret_cast<bf16x8_t*>((isk ? kc : vc) + (((int64_t)blk * Hk + kh) * BS + slot % BS) * D + c * 8) = x;
  bf16* extra = isk ? k_out : v_out;
  if (extra) *reinterpret_cast<bf16x8_t*>(extra + ((int64_t)t * Hk + kh) * D + c * 8) = x;
}

// The same for what that cannot take: sums that still sit in a GEMV's workspace, widths and rotations that are no whole chunks.
// One thread per element pair.
__global__ void __launch_bounds__(256) qkv_rope_append_kernel(
    const bf16* __restrict__ qkv, const float* __restrict__ cosT, const float* __restrict__ sinT,
    const int* __restrict__ pos, bf16* __restrict__ q_out, bf16* __restrict__ k_out, bf16* __restrict__ v_out,
    bf16* __restrict__ kc, bf16* __restrict__ vc, const int* __restrict__ block_table,
    const int* __restrict__ start_pos, const int* __restrict__ seq_ids, int n_new, int Hq, int Hk, int D, int rot,
    int interleaved, int BS, int max_blocks, float* __restrict__ acc, const bf16* __restrict__ acc_bias, int NP) {
  // grid = (tokens, head groups): 256 threads cover 256 / (D/2) heads of one token, one thread per element pair
  const int H3 = Hq + 2 * Hk, half = D / 2, rh = rot / 2;
  const int tph = half < (int)blockDim.x ? half : (int)blockDim.x;
  // uniform batch: token t is row t % n_new of sequence t / n_new; ragged batch (seq_ids): sequence seq_ids[t],
  // cache slot = its position
  const int t = blockIdx.x, h = blockIdx.y * (blockDim.x / tph) + threadIdx.x / tph;
  const int b = seq_ids ? seq_ids[t] : t / n_new, j = seq_ids ? 0 : t % n_new;
  // acc != null: the fused projection's sums still sit in the weight-only GEMV's fp32 split-K workspace [rows, NP]
  // (skinny_int8.hip / skinny_int4.hip without their finalize pass): read them (+ bias) from there and re-zero what
  // was read, padding columns included, so this kernel IS that GEMV's finalize pass
  float* arow = acc ? acc + (int64_t)t * NP : nullptr;
  if (arow && blockIdx.y == 0)
    for (int i = H3 * D + threadIdx.x; i < NP; i += blockDim.x) arow[i] = 0.f;
  // (head dims whose half does not divide the block leave a few surplus threads at the end)
  if (h >= H3 || (int)threadIdx.x / tph >= (int)blockDim.x / tph) return;
  const bf16* src = acc ? nullptr : qkv + ((int64_t)t * H3 + h) * D;
  auto ld = [&](int d) -> float {
    if (arow == nullptr) return (float)src[d];
    const float v = arow[h * D + d] + (acc_bias ? (float)acc_bias[h * D + d] : 0.f);
    arow[h * D + d] = 0.f;
    return (float)(bf16)v;  // the unfused path rounds the projection to bf16 before RoPE
  };
  bf16* dst;
  bf16* extra = nullptr;
  if (h < Hq) {
    dst = q_out + ((int64_t)t * Hq + h) * D;
  } else {
    const bool isk = h < Hq + Hk;
    const int kh = isk ? h - Hq : h - Hq - Hk;
    const int slot = seq_ids ? pos[t] : start_pos[b] + j;
    const int blk = block_table[(int64_t)b * max_blocks + slot / BS], off = slot % BS;
    dst = (isk ? kc : vc) + (((int64_t)blk * Hk + kh) * BS + off) * D;
    if (isk ? k_out : v_out) extra = (isk ? k_out : v_out) + ((int64_t)t * Hk + kh) * D;
  }
  const int p = pos[t];
  for (int i = threadIdx.x % tph; i < half; i += tph) {
    int d0, d1;
    if (i < rh) {
      d0 = interleaved ? 2 * i : i;
      d1 = interleaved ? 2 * i + 1 : i + rh;
    } else {
      d0 = rot + 2 * (i - rh);
      d1 = d0 + 1;
    }
    float a = ld(d0), c = ld(d1);
    if (i < rh && h < Hq + Hk) {
      const float cs = cosT[(int64_t)p * rh + i], sn = sinT[(int64_t)p * rh + i];
      const float a2 = a * cs - c * sn;
      c = c * cs + a * sn;
      a = a2;
    }
    dst[d0] = (bf16)a;
    dst[d1] = (bf16)c;
    if (extra) {
      extra[d0] = (bf16)a;
      extra[d1] = (bf16)c;
    }
  }
}

}  // namespace

// How many workgroups share a sequence: one up to 768 keys (the combine pass costs more than it saves: 12 x 8 heads x 700 keys 11.0
// us whole, 12.1 in two; 1 x 8 x 512 9.7 and, in four, 9.1), then as many as fill the chip with one each, of at least 256 keys, 512
// for long ones (1 x 8 x 1024: 15.0 whole, 10.4 in four; 12 x 8 x 2048: 27.9, 23.2 in two, 25.5 in four; 1 x 8 x 8192: 89, 19.2 in
// sixteen, 24 in thirty-two).
extern "C" int ds_paged_decode_splits(int B, int Hk, int max_len) {
  const int64_t own = (int64_t)B * Hk;
  int chunk = max_len;
  if (max_len > 768) {
    const int want = (int)(own < 256 ? 256 / own : 1), least = max_len > 4096 ? 512 : 256;
    chunk = (max_len + want - 1) / want;
    chunk = ((chunk < least ? least : chunk) + 63) / 64 * 64;
  }
  return (max_len + chunk - 1) / chunk;
}

namespace {

template <int DK, int DV, int LPR, bool NEW, int GT, int VP>
int launch_parts(const DecodeArgs& a, dim3 grid, hipStream_t s) {
  const int dv = DK ? DV : a.dv;
  const int lds = WAVES * GT * (dv / VP + 2 + KEYS + 1) * (int)sizeof(float) + (NEW ? (GT + 2) * dv * 2 : 0);
  auto* kernel = &paged_decode_kernel<DK, DV, GT, LPR, NEW, VP>;
  if (lds > 65536 &&
      hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(kernel, dim3(grid.x, grid.y, grid.z * VP), dim3(THREADS), lds, s, a);
  DS_CHECK_LAUNCH();
  if (grid.z > 1) {
    hipLaunchKernelGGL(combine_kernel, dim3((unsigned)grid.x * a.Hq), dim3(dv), 0, s, a.part_acc, a.part_ml, a.out, a.sink, a.gate,
                       a.ldg, a.Hq, a.ldo, (int)grid.z);
    DS_CHECK_LAUNCH();
  }
  return 0;
}

// Values in two parts where that leaves no CU with more than one workgroup: a CU reads 60 B/ns at most, here three quarters of what it had to, and
// needs no second launch. us whole / in parts, 12 sequences of 33 / 300 / 700 keys: 8 key heads of 128, 2 query heads each 4.8 / 8.0 / 13.0, 4.6 /
// 7.5 / 12.0; 4 each 5.6 / 9.1 / 14.7, 6.1 / 9.1 / 13.9 (hence from 384 keys there); 4 of 256, 4 each 6.6 / 12.3 / 25.0, 6.1 / 11.3 / 20.2.
template <int DK, int DV, int LPR, bool NEW, int GT>
int launch_decode(const DecodeArgs& a, dim3 grid, hipStream_t s) {
  if constexpr (DK >= 128) {
    if (grid.z == 1 && grid.x * grid.y <= 128 && a.chunk >= (DK == 128 && GT >= 4 ? 384 : 0)) return launch_parts<DK, DV, LPR, NEW, GT, 2>(a, grid, s);
  }
  return launch_parts<DK, DV, LPR, NEW, GT, 1>(a, grid, s);
}

// by the query heads a workgroup serves
template <int DK, int DV, int LPR, bool NEW>
int launch_decode(const DecodeArgs& a, dim3 grid, hipStream_t s) {
  const int G = a.Hq / a.Hk;
  if (G <= 1) return launch_decode<DK, DV, LPR, NEW, 1>(a, grid, s);
  if (G <= 2) return launch_decode<DK, DV, LPR, NEW, 2>(a, grid, s);
  if (G <= 4) return launch_decode<DK, DV, LPR, NEW, 4>(a, grid, s);
  return launch_decode<DK, DV, LPR, NEW, MAXG>(a, grid, s);
}

int log2_of(int n) { return n > 0 && (n & (n - 1)) == 0 ? __builtin_ctz(n) : -1; }

}  // namespace

namespace {

template <bool NEW>
int decode_by_width(const DecodeArgs& a, dim3 grid, hipStream_t s) {
  switch (a.dk) {
    case 64: return launch_decode<64, 64, 8, NEW>(a, grid, s);
    case 80: return launch_decode<80, 80, 16, NEW>(a, grid, s);
    case 96: return launch_decode<96, 96, 16, NEW>(a, grid, s);
    case 128: return launch_decode<128, 128, 16, NEW>(a, grid, s);
    case 256: return launch_decode<256, 256, 32, NEW>(a, grid, s);
    default: return (int)hipErrorInvalidValue;
  }
}

}  // namespace

// With `pos`: q is the step's projection [B, (Hq + 2 Hk) D], seq_lens counts its key, which is turned (like the queries, by the
// tables' row pos[b]: the first `rot` elements, rot % 16 == 0) and goes into the cache with its value.
extern "C" int ds_paged_decode(const void* q, void* kc, void* vc, const int* block_table,
                               const int* seq_lens, const float* alibi, float* part_acc, float* part_ml, void* out,
                               int B, int Hq, int Hk, int D, int BS, int max_blocks, int max_len, int splits,
                               float scale, int window, const int* pos, const float* cosT, const float* sinT, int rot,
                               int interleaved, hipStream_t s) {
  if (Hk <= 0 || Hq % Hk || Hq / Hk > MAXG || splits <= 0 || rot < 0 || rot % 16 || rot > D || (rot && (!pos || !cosT || !sinT)))
    return (int)hipErrorInvalidValue;
  if (window > 0 && window < max_len) max_len = window;  // no more keys than that are in sight
  const int chunk = ((max_len + splits - 1) / splits + 63) / 64 * 64;
  const DecodeArgs a{(const bf16*)q, (bf16*)kc, (bf16*)vc, block_table, seq_lens, alibi, part_acc, part_ml, (bf16*)out,
                     nullptr, nullptr, 0, (int64_t)Hq * D, Hq, Hk, BS, log2_of(BS), max_blocks, chunk, window, 0, D, D, scale, 0.f,
                     cosT, sinT, pos, rot, interleaved};
  const dim3 grid(B, Hk, splits);
  return pos ? decode_by_width<true>(a, grid, s) : decode_by_width<false>(a, grid, s);
}

// Key / value widths of their own (multiples of 8 up to 256), chunked and / or windowed visibility, score cap, softmax sink
// [Hq] (or null), gate [B, Hq] (or null), its rows ldg and rows of out ldo elements apart. `splits`
// from ds_paged_decode_splits(B, Hk, span) with span = the most keys in sight.
extern "C" int ds_paged_decode_ext(const void* q, void* kc, void* vc, const int* block_table,
                                   const int* seq_lens, float* part_acc, float* part_ml, void* out, int B, int Hq, int Hk,
                                   int dk, int dv, int BS, int max_blocks, int span, int splits, float scale,
                                   float softcap, int window, int mask_chunk, const float* sink, const void* gate,
                                   int64_t ldg, int64_t ldo, hipStream_t s) {
  if (Hk <= 0 || Hq % Hk || dk % 8 || dv % 8 || dk <= 0 || dv <= 0 || dk > 256 || dv > 256 || splits <= 0 ||
      ldo < (int64_t)Hq * dv)
    return (int)hipErrorInvalidValue;
  const int chunk = ((span + splits - 1) / splits + 63) / 64 * 64;
  const DecodeArgs a{(const bf16*)q, (bf16*)kc, (bf16*)vc, block_table, seq_lens, nullptr, part_acc, part_ml, (bf16*)out,
                     sink, (const bf16*)gate, ldg, ldo, Hq, Hk, BS, log2_of(BS), max_blocks, chunk, window, mask_chunk, dk, dv, scale,
                     softcap, nullptr, nullptr, nullptr, 0, 0};
  const dim3 grid(B, Hk * ((Hq / Hk + MAXG - 1) / MAXG), splits);
  const int wide = dk > dv ? dk : dv;
  if (wide <= 64) return launch_decode<0, 0, 8, false>(a, grid, s);
  if (wide <= 128) return launch_decode<0, 0, 16, false>(a, grid, s);
  return launch_decode<0, 0, 32, false>(a, grid, s);
}

extern "C" int ds_kv_append(const void* k, const void* v, void* kc, void* vc, const int* block_table,
                            const int* start_pos, int B, int n_new, int Hk, int D, int BS, int max_blocks,
                            hipStream_t s) {
  if (D % 8) return (int)hipErrorInvalidValue;
  const int grid = ds_grid_for((int64_t)B * n_new * Hk * (D / 8), 256);
  hipLaunchKernelGGL(kv_append_kernel, dim3(grid), dim3(256), 0, s, (const bf16*)k, (const bf16*)v, (bf16*)kc,
                     (bf16*)vc, block_table, start_pos, B, n_new, Hk, D, BS, max_blocks);
  DS_CHECK_LAUNCH();
  return 0;
}

extern "C" int ds_qkv_rope_append(const void* qkv, const float* cosT, const float* sinT, const int* pos, void* q_out,
                                  void* k_out, void* v_out, void* kc, void* vc, const int* block_table,
                                  const int* start_pos, const int* seq_ids, int T, int n_new, int Hq, int Hk, int D,
                                  int rot, int interleaved, int BS, int max_blocks, float* acc, const void* acc_bias,
                                  int NP, hipStream_t s) {
  if (D % 2 || rot % 2 || rot > D || (D - rot) % 2 || T <= 0) return T == 0 ? 0 : (int)hipErrorInvalidValue;
  if (acc != nullptr && (NP < (Hq + 2 * Hk) * D || T > 16)) return (int)hipErrorInvalidValue;
  if (acc == nullptr && qkv == nullptr) return (int)hipErrorInvalidValue;
  if (acc == nullptr && D % 8 == 0 && rot % 16 == 0) {
    hipLaunchKernelGGL(qkv_rope_rows_kernel, dim3(T, ((Hq + 2 * Hk) * (D / 8) + 255) / 256), dim3(256), 0, s, (const bf16*)qkv, cosT,
                       sinT, pos, (bf16*)q_out, (bf16*)k_out, (bf16*)v_out, (bf16*)kc, (bf16*)vc, block_table, start_pos, seq_ids,
                       n_new, Hq, Hk, D, rot, interleaved, BS, max_blocks);
    DS_CHECK_LAUNCH();
    return 0;
  }
  const int tph = D / 2 < 256 ? D / 2 : 256, hpb = 256 / tph;
  hipLaunchKernelGGL(qkv_rope_append_kernel, dim3(T, (Hq + 2 * Hk + hpb - 1) / hpb), dim3(256), 0, s, (const bf16*)qkv, cosT, sinT, pos,
                     (bf16*)q_out, (bf16*)k_out, (bf16*)v_out, (bf16*)kc, (bf16*)vc, block_table, start_pos, seq_ids,
                     n_new, Hq, Hk, D, rot, interleaved, BS, max_blocks, acc, (const bf16*)acc_bias, NP);
  DS_CHECK_LAUNCH();
  return 0;
}
