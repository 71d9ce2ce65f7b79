// CDNA4 flash attention for small head dims (32 / 64) with additive biases and attention dropout: forward and
// backward. Serves the DS4Science Evoformer attention and the BERT training layer.
//
// Reference counterparts (behaviour): `csrc/deepspeed4science/evoformer_attn/attention_cu.cu:12-160` +
// `attention_back.cu` (CUTLASS fMHA with a [B,N,1,1,S] per-key bias and a [B,1,H,S,S] pair bias, gradients for both)
// and the BERT layer's masked softmax + attention dropout (`csrc/transformer/softmax_kernels.cu:28-158`,
// `dropout_kernels.cu`). Neither bias nor the probability matrix is ever materialised at [batch, H, S, S].
//
// Tensors are [Z, S, H, D] with arbitrary (z, s, h) strides (Z = B*N for Evoformer, B for BERT); bias1 is indexed
// [z, key] (per-key mask bias), bias2 is [Z / b2_div, H, S, S] (pair bias shared by b2_div consecutive z).
//  * forward (one of its own for width 32, a pair bias and up to 256 keys, see there): one workgroup = 4 waves x 32 query rows of one (z, h); 64-key K/V tiles in LDS (rows padded to 2D + 16 bytes:
//    conflict-free b128 row reads without a swizzle); S^T = K.Q^T on v_mfma_f32_32x32x16 so each lane owns one query row's scores, biases added in natural units (a mask of the type's lowest
//    value must not become -inf), online softmax, P reused as the A operand of O += P.V (V by the hardware transposed
//    read); dropout multiplies P by keep / (1 - p) after the normaliser (Philox-4x32 keyed by (z, h, query, key),
//    regenerated in the backward);
//  * backward: passes without atomics on the big tensors (dQ query-outer; dK/dV key-outer; short sequences both in one; the shared pair-bias gradient summed
//    over the z that share it in registers), P recomputed from the saved LSE in each — see the backward section.
// All passes are bound by the vector instructions around the exponentials (about ten a score) and by latency: tiles are small and
// few, so each has ONE buffer in LDS and nothing is held in registers for the next one: three workgroups share a CU and cover each
// other's loads (held ahead: 52 us for 40 in the forward; a fourth workgroup, by spilling: 63). Keys past the end are -inf in
// the tile's per-key biases, which costs a score nothing. Measured at [256, 256, 4, 32] with both biases, us, before (two
// buffers, two workgroups a CU, a mask per score) and now: forward 64 and 40, dQ and dK/dV 158 and 97, dB2 234 and 47;
// [100, 133, 8, 32], whose rows start anywhere: 29, 66 and 33. Width 64 (forward / backward): the BERT layer's per-key mask and
// dropout, [8, 512, 16, 64], 40 / 180 and 35 / 114; with a pair bias of [64, 384, 4, 64] 43 / 388 and 34 / 126, with dropout too 53 / 484
// and 45 / 211 (its dB2 pass keeps a few registers in scratch memory).
#include "ds_hip.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int BM = 128;    // query rows per workgroup
constexpr int BN = 64;     // keys per tile
constexpr int NTHR = 256;

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

template <typename T> struct MF;
template <> struct MF<bf16> {
  typedef bf16x8_t V8;
  __device__ __forceinline__ static f32x16_t mma(V8 a, V8 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct MF<fp16> {
  typedef f16x8_t V8;
  __device__ __forceinline__ static f32x16_t mma(V8 a, V8 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

template <int D> constexpr int RS() { return 2 * D + 16; }   // LDS row stride (bytes)
template <int D> constexpr int TILE() { return BN * RS<D>(); }

// row of accumulator register r (32x32 C layout) for lane half h
__device__ __forceinline__ int crow(int r, int h) { return (r & 3) + 8 * (r >> 2) + 4 * h; }

// ---------------------------------------------------------------- dropout: Philox-4x32-7, 4 keep bits per call
__device__ __forceinline__ uint32_t keep4(uint64_t seed, uint64_t row, uint32_t key4, uint32_t thresh) {
  uint32_t c0 = key4, c1 = (uint32_t)row, c2 = (uint32_t)(row >> 32), c3 = 0x5bd1e995u;
  uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
#pragma unroll
  for (int i = 0; i < 7; ++i) {
    const uint32_t hi0 = __umulhi(0xD2511F53u, c0), lo0 = 0xD2511F53u * c0;
    const uint32_t hi1 = __umulhi(0xCD9E8D57u, c2), lo1 = 0xCD9E8D57u * c2;
    const uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
    c0 = n0; c1 = lo1; c2 = n2; c3 = lo0;
    k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
  }
  return (c0 >= thresh ? 1u : 0u) | (c1 >= thresh ? 2u : 0u) | (c2 >= thresh ? 4u : 0u) | (c3 >= thresh ? 8u : 0u);
}

template <typename T>
struct SmallArgs {
  const T* q; const T* k; const T* v; const T* o; const T* dout;
  T* out;          // forward O / backward dQ
  float* lse;      // [Z, H, S]
  const T* b1;     // [z, key] (stride b1_zs) or null
  const T* b2;     // [Z / b2_div, H, S, S] or null
  T* dk; T* dv;    // backward [Z, S, H, D] (dense)
  float* delta;    // backward rowsum(dO * O) [Z, H, S], written by the dQ pass
  float* db1;      // [Z, S] fp32 (zeroed; summed over heads by atomics) or null
  float* db2;      // [Z / b2_div, H, S, S] fp32 or null
  int64_t qz, qs, qh, kz, ks, kh, vz, vs, vh, oz, os_, oh, gz, gs, gh, dz, ds, dh;  // (z, s, h) strides: q k v o dO dQ
  int64_t b1_zs;
  int Z, H, S, b2_div;
  float scale;
  float pdrop;     // 0 = no dropout
  uint32_t thresh; // keep if philox >= thresh
  uint64_t seed;
  int64_t b2_last; // elements of bias2 - 8 (at least 0): where its last whole chunk begins
  int nsplit;      // dB2 pass: the b2_div sharing z are split over this many workgroups
  float* part;     // ... whose sums go here [nsplit, Z / b2_div, H, S, S] when they are several
  T* order;        // backward: the pair bias in the accumulators' order (small_order_elements), or null
  int Sk;          // keys (the forward may attend to a context of another length; the backward needs Sk == S)
  int db2_as_in;   // with several parts: db2 is of the inputs' type, rounded once
};

// 4 consecutive 16-bit values (8-B aligned) added to f as fp32 / stored from fp32
__device__ __forceinline__ void add4(const bf16* p, float (&f)[4]) {
  const bf16x4 v = *reinterpret_cast<const bf16x4*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) f[i] += (float)v[i];
}
__device__ __forceinline__ void add4(const fp16* p, float (&f)[4]) {
  const fp16x4 v = *reinterpret_cast<const fp16x4*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) f[i] += (float)v[i];
}
// 16-B chunks (8 keys) of rows of bias2, at any alignment, CPR a row: chunk tid + i NTHR of the rows row0.. and keys key0.. of the
// matrix at `mat`. Past the end of the tensor nothing is read: the last whole chunk there is, shifted (a path of its own: the shifts
// would cost every tile an eighth of its instructions). CUT: what lies past the end of a row is zero (it is the next row's, and an
// infinity or NaN there would outweigh the -inf of the keys that it stands for); a thread's chunks stand at one place of their rows.
template <int CPR, bool CUT, typename T>
__device__ __forceinline__ void bias_chunks(const SmallArgs<T>& a, int64_t mat, int row0, int key0, int tid, u32x4_t (&out)[4]) {
  typedef unsigned __int128 u128;
  constexpr int ROWS = 4 * NTHR / CPR;
  auto at = [&](int i) {
    const int c = tid + i * NTHR;
    return mat + (int64_t)min(row0 + c / CPR, a.S - 1) * a.Sk + key0 + c % CPR * 8;
  };
  if (mat + (int64_t)min(row0 + ROWS - 1, a.S - 1) * a.Sk + key0 + CPR * 8 <= a.b2_last + 8) {
#pragma unroll
    for (int i = 0; i < 4; ++i) __builtin_memcpy(&out[i], a.b2 + at(i), 16);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t off = at(i), from = min(off, a.b2_last);
      u128 v;
      __builtin_memcpy(&v, a.b2 + from, 16);
      out[i] = __builtin_bit_cast(u32x4_t, v >> 16 * (int)min(off - from, (int64_t)7));
    }
  }
  if constexpr (CUT) {
    static_assert(NTHR % CPR == 0, "one place a thread");
    if (key0 + CPR * 8 > a.Sk) {
      const int left = a.Sk - key0 - tid % CPR * 8;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const unsigned keep = left >= 2 * w + 2 ? ~0u : left == 2 * w + 1 ? 0xffffu : 0u;
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i][w] &= keep;
      }
    }
  }
}

__device__ __forceinline__ void st16_as_2x8(char* p, u32x4_t v) {  // 8-B aligned LDS destination
  typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
  *reinterpret_cast<u32x2_t*>(p) = u32x2_t{v[0], v[1]};
  *reinterpret_cast<u32x2_t*>(p + 8) = u32x2_t{v[2], v[3]};
}

template <typename T, int D>
struct Tiles {
  // staging: chunk c (row = c / (D/8), 16-B chunk = c % (D/8)); D/8 * 64 chunks, D/32 per thread
  static constexpr int CPR = D / 8, PER = CPR * BN / NTHR;
};

// One 64-key tile for the query-row kernels (forward, dQ): K and V rows, per-key biases of the 64 keys (fp32, -inf past the
// end) and the workgroup's [128 q][64 key] bias2 block, staged global -> registers -> LDS. bias2 rows are 136 B apart: the 8-B reads of 32 different rows by one wave
// land on 64 distinct banks. PAIR: with the bias2 block.
template <typename T, int D, bool PAIR>
struct KeyTile {
  static constexpr int PER = Tiles<T, D>::PER, CPR = Tiles<T, D>::CPR;
  static constexpr int B2RS = 2 * BN + 8;
  static constexpr int OFF_V = TILE<D>(), OFF_B1 = 2 * TILE<D>(), OFF_B2 = OFF_B1 + 4 * BN;
  static constexpr int BYTES = OFF_B2 + (PAIR ? BM * B2RS : 0);
  u32x4_t rk[PER], rv[PER], rb2[4];
  float rb1;
  // b2mat: where the [S, Sk] bias2 matrix of this (z-group, head) begins; qrow0: first query row of the workgroup
  __device__ __forceinline__ void load(const SmallArgs<T>& a, const T* Kp, const T* Vp, const T* b1p,
                                       int64_t b2mat, int qrow0, int k0, int tid) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = tid + i * NTHR, row = c / CPR, ch = c % CPR;
      const int key = min(k0 + row, a.Sk - 1);
      rk[i] = *reinterpret_cast<const u32x4_t*>(Kp + (int64_t)key * a.ks + ch * 8);
      rv[i] = *reinterpret_cast<const u32x4_t*>(Vp + (int64_t)key * a.vs + ch * 8);
    }
    if constexpr (PAIR) bias_chunks<8, true>(a, b2mat, qrow0, k0, tid, rb2);
    if (tid < BN) rb1 = k0 + tid >= a.Sk ? -INFINITY : b1p ? (float)b1p[k0 + tid] : 0.f;
  }
  __device__ __forceinline__ void store(char* buf, int tid) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = tid + i * NTHR, row = c / CPR, ch = c % CPR;
      *reinterpret_cast<u32x4_t*>(buf + row * RS<D>() + ch * 16) = rk[i];
      *reinterpret_cast<u32x4_t*>(buf + OFF_V + row * RS<D>() + ch * 16) = rv[i];
    }
    if constexpr (PAIR) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = tid + i * NTHR, row = c >> 3, ch = c & 7;
        st16_as_2x8(buf + OFF_B2 + row * B2RS + ch * 16, rb2[i]);
      }
    }
    if (tid < BN) reinterpret_cast<float*>(buf + OFF_B1)[tid] = rb1;
  }
};

// per-key bias + bias2 of the 4 keys kr + 4 h .. + 3 of the tile, kr a constant: `b1row` and `b2row` are where key 4 h stands
template <typename T, bool PAIR>
__device__ __forceinline__ void tile_bias4(const char* b1row, const char* b2row, int kr, float (&bb)[4]) {
  const f32x4 b1 = *reinterpret_cast<const f32x4*>(b1row + kr * 4);
#pragma unroll
  for (int i = 0; i < 4; ++i) bb[i] = b1[i];
  if constexpr (PAIR) add4(reinterpret_cast<const T*>(b2row + kr * 2), bb);
}

// transposed 4+4-row read of a row-major 16-bit image into an MFMA operand (k slots = rows rb+{0..3}, rb+8+{0..3})
template <typename V8>
__device__ __forceinline__ V8 tr_read(const char* img, int rs, int rb, int ch0, int lane) {
  const int gq = (lane >> 2) & 3, gb = 8 * (lane & 1);
  const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4_t*)(img + (rb + gq) * rs + ch0 * 16 + gb));
  const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4_t*)(img + (rb + 8 + gq) * rs + ch0 * 16 + gb));
  s16x8 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) { v[e] = lo[e]; v[4 + e] = hi[e]; }
  return __builtin_bit_cast(V8, v);
}

// 4 + 4 rows' transposed read at two places
template <typename V8>
__device__ __forceinline__ V8 tr_pair(const char* lo_p, const char* hi_p) {
  const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)lo_p);
  const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)hi_p);
  s16x8 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) { v[e] = lo[e]; v[4 + e] = hi[e]; }
  return __builtin_bit_cast(V8, v);
}

// ================================================================================================== forward
template <typename T, int D, bool DROP, bool PAIR>
__global__ void __launch_bounds__(NTHR, 2) small_fwd_kernel(SmallArgs<T> a) {
  typedef typename MF<T>::V8 V8;
  typedef KeyTile<T, D, PAIR> KT;
  __shared__ __attribute__((aligned(16))) char smem[KT::BYTES + 4 * 32 * 4];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, h = lane >> 5, l32 = lane & 31;
  const int nqb = (a.S + BM - 1) / BM;
  const int qb = blockIdx.x % nqb, hd = (blockIdx.x / nqb) % a.H, z = blockIdx.x / (nqb * a.H);
  const int q0w = qb * BM + wid * 32, qrow = q0w + l32;
  const T* Qp = a.q + z * a.qz + hd * a.qh;
  const T* Kp = a.k + z * a.kz + hd * a.kh;
  const T* Vp = a.v + z * a.vz + hd * a.vh;
  const T* b1p = a.b1 ? a.b1 + z * a.b1_zs : nullptr;
  const int64_t b2mat = ((int64_t)(z / a.b2_div) * a.H + hd) * a.S * a.Sk;
  const uint64_t drow = ((uint64_t)z * a.H + hd) * (uint64_t)a.S + (uint64_t)qrow;

  V8 qf[D / 16];
  {
    const T* qr = Qp + (int64_t)min(qrow, a.S - 1) * a.qs + 8 * h;
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) qf[kk] = *reinterpret_cast<const V8*>(qr + 16 * kk);
  }
  float* scratch = reinterpret_cast<float*>(smem + KT::BYTES) + wid * 32;
  KT stg;

  f32x16_t o[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  const int nt = (a.Sk + BN - 1) / BN;
  const float LOG2E = 1.4426950408889634f;
  const float inv_keep = DROP ? 1.f / (1.f - a.pdrop) : 1.f;
  const int gch = (lane >> 1) & 1, colhalf = (lane >> 4) & 1;

  stg.load(a, Kp, Vp, b1p, b2mat, qb * BM, 0, tid);
  stg.store(smem, tid);
  __syncthreads();
  for (int j = 0; j < nt; ++j) {
    const int k0 = j * BN;
    const char* buf = smem;
    const char* Vt = buf + KT::OFF_V;
    const char* b1row = buf + KT::OFF_B1 + 16 * h;
    const char* b2row = buf + KT::OFF_B2 + (wid * 32 + l32) * KT::B2RS + 8 * h;
    f32x16_t s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[t][r] = 0.f;
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) {
        const V8 av = *reinterpret_cast<const V8*>(buf + (t * 32 + l32) * RS<D>() + (2 * kk + h) * 16);
        s[t] = MF<T>::mma(av, qf[kk], s[t]);
      }
    }
    // natural-unit logits: scale * q.k + bias1[key] + bias2[q, key]
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float bb[4];
        tile_bias4<T, PAIR>(b1row, b2row, t * 32 + 8 * g, bb);
#pragma unroll
        for (int i = 0; i < 4; ++i) s[t][4 * g + i] = s[t][4 * g + i] * a.scale + bb[i];
      }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, fmaxf(s[0][r], s[1][r]));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f((m_run - m_use) * LOG2E);
    f32x4 psum{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = __builtin_amdgcn_exp2f((s[t][r] - m_use) * LOG2E);
        s[t][r] = p;
        psum[r & 3] += p;
      }
    l_run = l_run * alpha + ((psum[0] + psum[1]) + (psum[2] + psum[3]));
    asm volatile("" : "+v"(l_run));  // (summed here, not kept as 32 terms through the rest)
    m_run = m_new;
    if constexpr (DROP) {  // dropout after the normaliser: O accumulates P * keep / (1 - p)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const uint32_t kb = keep4(a.seed, drow, (uint32_t)((k0 + t * 32 + 8 * g + 4 * h) >> 2), a.thresh);
#pragma unroll
          for (int i = 0; i < 4; ++i) s[t][4 * g + i] *= ((kb >> i) & 1u) ? inv_keep : 0.f;
        }
    }
    if (!__all(alpha == 1.f)) {
      if (lane < 32) scratch[lane] = alpha;
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      float a4[16];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 vv = *reinterpret_cast<const f32x4*>(scratch + 8 * g + 4 * h);
#pragma unroll
        for (int i = 0; i < 4; ++i) a4[4 * g + i] = vv[i];
      }
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= a4[r];
      __builtin_amdgcn_wave_barrier();
    }
    V8 pa[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ss = 0; ss < 2; ++ss)
#pragma unroll
        for (int e = 0; e < 8; ++e) pa[t][ss][e] = (T)s[t][8 * ss + e];
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) {
      const int ch0 = dt * 4 + colhalf * 2 + gch;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int ss = 0; ss < 2; ++ss)
          o[dt] = MF<T>::mma(pa[t][ss], tr_read<V8>(Vt, RS<D>(), t * 32 + 16 * ss + 4 * h, ch0, lane), o[dt]);
    }
    __syncthreads();
    if (j + 1 < nt) {
      stg.load(a, Kp, Vp, b1p, b2mat, qb * BM, k0 + BN, tid);
      stg.store(smem, tid);
      __syncthreads();
    }
  }
  const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if (lane < 32) scratch[lane] = inv;
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  float iv[16];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const f32x4 vv = *reinterpret_cast<const f32x4*>(scratch + 8 * g + 4 * h);
#pragma unroll
    for (int i = 0; i < 4; ++i) iv[4 * g + i] = vv[i];
  }
  T* Op = a.out + z * a.oz + hd * a.oh;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int qi = q0w + crow(r, h);
    if (qi < a.S) {
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) Op[(int64_t)qi * a.os_ + dt * 32 + l32] = (T)(o[dt][r] * iv[r]);
    }
  }
  if (lane < 32 && qrow < a.S)
    a.lse[((int64_t)z * a.H + hd) * a.S + qrow] = l_tot > 0.f ? m_run + __logf(l_tot) : INFINITY;
}

// ---------------------------------------------------------------- forward, 8 to 256 keys, width 32, a pair bias
// Bound by the vector instructions of a score (twelve and the exponential, four's time). Up to 256 queries of a (z, h) share a
// workgroup, K and V whole in LDS: one barrier, then a wave's tiles of 32 keys wait for nobody. The rows of K go into the matrix cores
// in an order that leaves a lane with 16 neighbouring keys of its query (register r of half h: key 16 h + r of the tile), so the pair
// bias comes from memory as it lies, 2 x 16 bytes a lane and tile, a tile ahead, and not through LDS. The largest
// weight is 1, which no type rounds: a maximum kept until a new one is well above it saves the rescaling of O, and costs a tenth of
// the result's accuracy (0.0023 for 0.0020 off 64 bits). 64-byte rows, chunk ch of row r at 16 (ch ^ swz32(r)):
// K's rows in that order and V's transposed reads touch every bank once. Two workgroups of eight waves share a CU.
// us, the general kernel and this one: [256, 256, 4, 32] 43.5 and 40.3, [180, 230, 8, 32] 57 and 51, [128, 200, 4, 32] 23.5 and 19.2,
// [100, 133, 8, 32] 29.6 and 24.9, [512, 32, 8, 32] 28.7 and 12.6.
// Large workgroups share out worse than the general kernel's of four waves where a CU has at most one and could have two of those,
// and where some CUs get a second one and most do not; those shapes stay with it. General and this, us, at 4 heads: 128
// workgroups of six waves (180 tokens) 8.4 and 9.1, of seven (210) 10.0 and 10.2, of eight (250) 10.2 and 11.2, but of five (150) 8.5 and
// 8.2; 160 of them 10.2 and 9.2, 11.9 and 10.3, 12.3 and 11.5, 10.0 and 8.3. 264 / 384 of eight 17.1 and 18.4 / 18.8 and 19.4, of seven 16.1 and
// 15.2 / 17.9 and 16.9; 416 of eight 23.6 and 19.6. (A third one has no such bound: 528 / 600 of eight 26.6 and 26.9 / 27.9 and 27.5.)
// What the line leaves slower: two waves, up to 256 workgroups, 4.9 and 5.1; 1200 of four (128 tokens) 18.3 and 19.5; and keys of another
// number than the queries, 560 of four waves and 256 keys 16.4 and 19.0, 640 of eight and 100 keys 16.6 and 18.3.
// (Tried beside 39 with another rule for the maximum: several z a workgroup, the next one's K and V on their way, 40.5; four waves 43.)
constexpr int FWD_WHOLE = 256, FWD_WAVES = 8;
__device__ __forceinline__ int swz32(int r) { return ((r >> 2) & 1) | ((r >> 3) & 2); }

// 16 bytes a lane from memory to LDS byte dst + 16 * lane, past the compiler, which would wait for it before every LDS read
__device__ __forceinline__ void small_dma(const void* g, uint32_t dst) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\t"
               "s_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(g), "s"(dst)
               : "memory");
}

// the larger of the two halves' values of a row (v_permlane32_swap: a shuffle through LDS is a wait of a hundred clocks)
__device__ __forceinline__ float half_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

template <typename T>
__global__ void __launch_bounds__(64 * FWD_WAVES, 4) small_fwd_whole_kernel(SmallArgs<T> a) {
  typedef typename MF<T>::V8 V8;
  typedef __attribute__((address_space(3))) char lds_char;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int nt = (a.Sk + 31) / 32, rows = nt * 32, waves = blockDim.x / 64;
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  float *b1S = reinterpret_cast<float*>(smem + 2 * rows * 64), *scratch = b1S + rows + wid * 32;  // (behind K and V)
  const int nqb = (a.S + 32 * waves - 1) / (32 * waves);
  const int qb = blockIdx.x % nqb, hd = blockIdx.x / nqb % a.H, z = blockIdx.x / (nqb * a.H);
  const int q0w = (qb * waves + wid) * 32, qrow = q0w + l32;
  const T* bp = a.b2 + ((int64_t)(z / a.b2_div) * a.H + hd) * a.S * a.Sk + (int64_t)min(qrow, a.S - 1) * a.Sk;
  const uint32_t lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const lds_char*)smem);

  for (int p = wid; p < 4 * nt; p += waves) {  // 16 rows of K or V
    const bool v = p >= 2 * nt;
    const int r = (v ? p - 2 * nt : p) * 16 + (lane >> 2), key = min(r, a.Sk - 1);
    const T* src = v ? a.v + z * a.vz + hd * a.vh + (int64_t)key * a.vs : a.k + z * a.kz + hd * a.kh + (int64_t)key * a.ks;
    small_dma(src + 8 * ((lane & 3) ^ swz32(r)), lds + p * 1024);
  }
  V8 qf[2];
  {
    const T* qr = a.q + z * a.qz + hd * a.qh + (int64_t)min(qrow, a.S - 1) * a.qs + 8 * h;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) qf[kk] = *reinterpret_cast<const V8*>(qr + 16 * kk);
  }
  V8 bias[2];  // of 16 keys of this lane's query
  auto load_bias = [&](int k0) {
    const int key = k0 + 16 * h;
    if (k0 + 32 <= a.Sk) {
#pragma unroll
      for (int g = 0; g < 2; ++g) __builtin_memcpy(&bias[g], bp + key + 8 * g, 16);
    } else {  // the row's end: its last eight, shifted (what is past it is another row's, or nobody's)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int at = key + 8 * g, from = min(at, a.Sk - 8);
        unsigned __int128 v;
        __builtin_memcpy(&v, bp + from, 16);
        v = at - from >= 8 ? 0 : v >> 16 * (at - from);
        bias[g] = __builtin_bit_cast(V8, v);
      }
    }
  };
  load_bias(0);
  for (int i = tid; i < rows; i += blockDim.x) b1S[i] = i >= a.Sk ? -INFINITY : a.b1 ? (float)a.b1[z * a.b1_zs + i] : 0.f;
  int ka[2], va[2];
  {
    const int key = 16 * ((l32 >> 2) & 1) + (l32 & 3) + 4 * (l32 >> 3);
    const int gq = (lane >> 2) & 3, gch = (lane >> 1) & 1, gb = 8 * (lane & 1), colhalf = (lane >> 4) & 1;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = 16 * h + 4 * i + gq;
      ka[i] = key * 64 + 16 * ((2 * i + h) ^ swz32(key));
      va[i] = rows * 64 + r * 64 + 16 * ((colhalf * 2 + gch) ^ swz32(r)) + gb;
    }
  }
  const float LOG2E = 1.4426950408889634f;
  asm volatile("s_waitcnt vmcnt(0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  f32x16_t o;
#pragma unroll
  for (int r = 0; r < 16; ++r) o[r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
#pragma unroll 1
  for (int j = 0; j < nt; ++j) {
    f32x16_t s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) s = MF<T>::mma(*reinterpret_cast<const V8*>(smem + j * 2048 + ka[kk]), qf[kk], s);
    // natural units: scale q.k + bias1[key] + bias2[q, key]
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 b1 = *reinterpret_cast<const f32x4*>(b1S + 32 * j + 16 * h + 4 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 4 * g + i;
        s[r] = fmaf(s[r], a.scale, b1[i] + (float)bias[r >> 3][r & 7]);
      }
    }
    if (j + 1 < nt) load_bias(32 * (j + 1));
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; r += 2) asm("v_max3_f32 %0, %0, %1, %2" : "+v"(mx) : "v"(s[r]), "v"(s[r + 1]));
    mx = half_max(mx);
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    f32x4 psum{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      // (the difference first: in an fma with a maximum that is scaled, and rounded, before, a mask of -1e10 is an exponent of 328)
      s[r] = __builtin_amdgcn_exp2f((s[r] - m_use) * LOG2E);
      psum[r & 3] += s[r];
    }
    if (!__all(m_new == m_run)) {
      const float alpha = __builtin_amdgcn_exp2f((m_run - m_use) * LOG2E);
      l_run *= alpha;
      if (j) {
        if (lane < 32) scratch[lane] = alpha;
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(scratch + 8 * g + 4 * h);
#pragma unroll
          for (int i = 0; i < 4; ++i) o[4 * g + i] *= v[i];
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
    l_run += (psum[0] + psum[1]) + (psum[2] + psum[3]);
    m_run = m_new;
#pragma unroll
    for (int ss = 0; ss < 2; ++ss) {
      V8 p;
#pragma unroll
      for (int e = 0; e < 8; ++e) p[e] = (T)s[8 * ss + e];
      const char* at = smem + j * 2048 + ss * 512;
      o = MF<T>::mma(p, tr_pair<V8>(at + va[0], at + va[1]), o);
    }
  }
  const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  if (lane < 32) scratch[lane] = l_tot > 0.f ? 1.f / l_tot : 0.f;
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  int ln = lane;  // (anew: the rows' addresses are not kept over the loop)
  asm volatile("" : "+v"(ln));
  const int row = q0w + 4 * (ln >> 5);
  T* Op = a.out + z * a.oz + hd * a.oh + (int64_t)row * a.os_ + (ln & 31);
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(scratch + 8 * g + 4 * (ln >> 5));
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (row + 8 * g + i < a.S) Op[(8 * g + i) * a.os_] = (T)(o[4 * g + i] * v[i]);
  }
  if (lane < 32 && qrow < a.S)
    a.lse[((int64_t)z * a.H + hd) * a.S + qrow] = l_tot > 0.f ? m_run + __logf(l_tot) : INFINITY;
}

// ================================================================================================== backward
// Three passes, no fp32 atomics on the big tensors:
//  1. dQ pass (query-outer, same tiling as the forward): delta = rowsum(dO * O) written for the other passes,
//     dQ += dS.K in registers; dB2 stored directly when every z has its own pair bias (b2_div == 1);
//  2. dK/dV pass (key-outer): a wave owns 32 keys (K, V rows in registers as B operands), Q / dO / lse / delta and
//     the [64 q x 128 key] bias2 block stream through LDS; S = Q.K^T lands with the key on the lane so P^T / dS^T
//     feed dV += P^T.dO and dK += dS^T.Q as the A operand straight from registers (dO, Q by transposed read);
//     dB1 column sums per lane, one atomic per (z, head, key);
//  3. dB2 pass (b2_div > 1): a workgroup owns one [128 q x 64 key] tile of the shared pair bias and loops over the
//     z that share it (split over a few workgroups when the tile grid alone cannot fill the chip), summing dS in
//     registers.

// ---------------------------------------------------------------- pass 1: dQ, delta (and unshared dB2)
template <typename T, int D, bool DROP, bool PAIR>
__global__ void __launch_bounds__(NTHR, 2) small_bwd_dq_kernel(SmallArgs<T> a) {
  typedef typename MF<T>::V8 V8;
  typedef KeyTile<T, D, PAIR> KT;
  __shared__ __attribute__((aligned(16))) char smem[KT::BYTES];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, h = lane >> 5, l32 = lane & 31;
  const int nqb = (a.S + BM - 1) / BM;
  const int qb = blockIdx.x % nqb, hd = (blockIdx.x / nqb) % a.H, z = blockIdx.x / (nqb * a.H);
  const int q0w = qb * BM + wid * 32, qrow = q0w + l32;
  const int qc = min(qrow, a.S - 1);
  const bool qlive = qrow < a.S;
  const T* Kp = a.k + z * a.kz + hd * a.kh;
  const T* Vp = a.v + z * a.vz + hd * a.vh;
  const T* b1p = a.b1 ? a.b1 + z * a.b1_zs : nullptr;
  const int64_t b2mat = ((int64_t)(z / a.b2_div) * a.H + hd) * a.S * a.S;
  float* db2p = (a.db2 && a.b2_div == 1) ? a.db2 + b2mat + (int64_t)qc * a.S : nullptr;
  const uint64_t drow = ((uint64_t)z * a.H + hd) * (uint64_t)a.S + (uint64_t)qrow;

  V8 qf[D / 16], gf[D / 16];
  float delta = 0.f;
  {
    const T* qr = a.q + z * a.qz + hd * a.qh + (int64_t)qc * a.qs;
    const T* gr = a.dout + z * a.gz + hd * a.gh + (int64_t)qc * a.gs;
    const T* orr = a.o + z * a.oz + hd * a.oh + (int64_t)qc * a.os_;
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) {
      qf[kk] = *reinterpret_cast<const V8*>(qr + 16 * kk + 8 * h);
      gf[kk] = *reinterpret_cast<const V8*>(gr + 16 * kk + 8 * h);
      const V8 ov = *reinterpret_cast<const V8*>(orr + 16 * kk + 8 * h);
#pragma unroll
      for (int e = 0; e < 8; ++e) delta += (float)gf[kk][e] * (float)ov[e];
    }
    delta += __shfl_xor(delta, 32, 64);
  }
  const int64_t lrow = ((int64_t)z * a.H + hd) * a.S;
  if (lane < 32 && qlive) a.delta[lrow + qrow] = delta;
  const float lse = qlive ? a.lse[lrow + qc] : INFINITY;
  const float LOG2E = 1.4426950408889634f;
  const float inv_keep = DROP ? 1.f / (1.f - a.pdrop) : 1.f;
  f32x16_t dq[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) dq[dt][r] = 0.f;
  const int nt = (a.S + BN - 1) / BN;
  const int gch = (lane >> 1) & 1, colhalf = (lane >> 4) & 1;
  const bool st4 = (a.S & 3) == 0;

  KT stg;
  stg.load(a, Kp, Vp, b1p, b2mat, qb * BM, 0, tid);
  stg.store(smem, tid);
  __syncthreads();
  for (int j = 0; j < nt; ++j) {
    const int k0 = j * BN;
    const char* buf = smem;
    const char* Vt = buf + KT::OFF_V;
    const char* b1row = buf + KT::OFF_B1 + 16 * h;
    const char* b2row = buf + KT::OFF_B2 + (wid * 32 + l32) * KT::B2RS + 8 * h;
    V8 da[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {  // one 32-key half at a time, and in the schedule too (registers)
      __builtin_amdgcn_sched_barrier(0);
      f32x16_t s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) { s[r] = 0.f; dp[r] = 0.f; }
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) {
        const V8 kv = *reinterpret_cast<const V8*>(buf + (t * 32 + l32) * RS<D>() + (2 * kk + h) * 16);
        s = MF<T>::mma(kv, qf[kk], s);
        const V8 vv = *reinterpret_cast<const V8*>(Vt + (t * 32 + l32) * RS<D>() + (2 * kk + h) * 16);
        dp = MF<T>::mma(vv, gf[kk], dp);
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        uint32_t kb = 0xfu;
        if constexpr (DROP) kb = keep4(a.seed, drow, (uint32_t)((k0 + t * 32 + 8 * g + 4 * h) >> 2), a.thresh);
        float bb[4];
        tile_bias4<T, PAIR>(b1row, b2row, t * 32 + 8 * g, bb);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 4 * g + i;
          const float p = __builtin_amdgcn_exp2f((s[r] * a.scale + bb[i] - lse) * LOG2E);
          if constexpr (DROP) dp[r] *= ((kb >> i) & 1u) ? inv_keep : 0.f;
          s[r] = p * (dp[r] - delta);  // dS (natural units)
          da[t][r >> 3][r & 7] = (T)s[r];
        }
      }
      if (db2p && qlive) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int kb4 = k0 + t * 32 + 8 * g + 4 * h;
          if (st4) {
            if (kb4 < a.S) *reinterpret_cast<f32x4*>(db2p + kb4) = f32x4{s[4 * g], s[4 * g + 1], s[4 * g + 2], s[4 * g + 3]};
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (kb4 + i < a.S) db2p[kb4 + i] = s[4 * g + i];
          }
        }
      }
    }
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) {
      const int ch0 = dt * 4 + colhalf * 2 + gch;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int ss = 0; ss < 2; ++ss)
          dq[dt] = MF<T>::mma(da[t][ss], tr_read<V8>(buf, RS<D>(), t * 32 + 16 * ss + 4 * h, ch0, lane), dq[dt]);
    }
    __syncthreads();
    if (j + 1 < nt) {
      stg.load(a, Kp, Vp, b1p, b2mat, qb * BM, k0 + BN, tid);
      stg.store(smem, tid);
      __syncthreads();
    }
  }
  T* Gq = a.out + z * a.dz + hd * a.dh;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int qi = q0w + crow(r, h);
    if (qi < a.S) {
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) Gq[(int64_t)qi * a.ds + dt * 32 + l32] = (T)(dq[dt][r] * a.scale);
    }
  }
}

// ---------------------------------------------------------------- pass 2: dK, dV (key-outer), dB1
// One 64-query tile: Q and dO rows, lse / delta of the 64 queries, and the [64 q][128 key] bias2 block of the
// workgroup's keys (272-B rows, read transposed: the 32 keys of a wave by lane, the queries by register).
template <typename T, int D, bool PAIR>
struct QueryTile {
  static constexpr int PER = Tiles<T, D>::PER, CPR = Tiles<T, D>::CPR;
  static constexpr int B2RS = 2 * BM + 16;
  static constexpr int OFF_G = TILE<D>(), OFF_L = 2 * TILE<D>(), OFF_B2 = OFF_L + 2 * BN * 4;
  static constexpr int BYTES = OFF_B2 + (PAIR ? BN * B2RS : 0);
  u32x4_t rq[PER], rg[PER], rb2[4];
  float rl;
  __device__ __forceinline__ void load(const SmallArgs<T>& a, const T* Qp, const T* Gp, int64_t lrow,
                                       int64_t b2mat, int key0, int q0, int tid) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = tid + i * NTHR, row = c / CPR, ch = c % CPR;
      const int q = min(q0 + row, a.S - 1);
      rq[i] = *reinterpret_cast<const u32x4_t*>(Qp + (int64_t)q * a.qs + ch * 8);
      rg[i] = *reinterpret_cast<const u32x4_t*>(Gp + (int64_t)q * a.gs + ch * 8);
    }
    if (tid < 2 * BN) {  // queries past the end weigh nothing
      const int q = q0 + (tid & (BN - 1));
      rl = tid < BN ? (q < a.S ? a.lse[lrow + q] : INFINITY) : (q < a.S ? a.delta[lrow + q] : 0.f);
    }
    if constexpr (PAIR) bias_chunks<16, false>(a, b2mat, q0, key0, tid, rb2);  // (keys past the end are lanes, and rows of products, of their own)
  }
  __device__ __forceinline__ void store(char* buf, int tid) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = tid + i * NTHR, row = c / CPR, ch = c % CPR;
      *reinterpret_cast<u32x4_t*>(buf + row * RS<D>() + ch * 16) = rq[i];
      *reinterpret_cast<u32x4_t*>(buf + OFF_G + row * RS<D>() + ch * 16) = rg[i];
    }
    if (tid < 2 * BN) reinterpret_cast<float*>(buf + OFF_L)[tid] = rl;
    if constexpr (PAIR) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = tid + i * NTHR, row = c >> 4, ch = c & 15;
        *reinterpret_cast<u32x4_t*>(buf + OFF_B2 + row * B2RS + ch * 16) = rb2[i];
      }
    }
  }
};

template <typename T, int D, bool DROP, bool PAIR>
__global__ void __launch_bounds__(NTHR, 2) small_bwd_dkv_kernel(SmallArgs<T> a) {
  typedef typename MF<T>::V8 V8;
  typedef QueryTile<T, D, PAIR> QT;
  __shared__ __attribute__((aligned(16))) char smem[QT::BYTES];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, h = lane >> 5, l32 = lane & 31;
  const int nkb = (a.S + BM - 1) / BM;
  const int kbk = blockIdx.x % nkb, hd = (blockIdx.x / nkb) % a.H, z = blockIdx.x / (nkb * a.H);
  const int key0w = kbk * BM + wid * 32, key = key0w + l32;
  const int kc = min(key, a.S - 1);
  const bool klive = key < a.S;
  const T* Qp = a.q + z * a.qz + hd * a.qh;
  const T* Gp = a.dout + z * a.gz + hd * a.gh;
  const int64_t b2mat = ((int64_t)(z / a.b2_div) * a.H + hd) * a.S * a.S;

  // B operands (column = this lane's key): K and V rows
  V8 kB[D / 16], vB[D / 16];
  {
    const T* kr = a.k + z * a.kz + hd * a.kh + (int64_t)kc * a.ks;
    const T* vr = a.v + z * a.vz + hd * a.vh + (int64_t)kc * a.vs;
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) {
      kB[kk] = *reinterpret_cast<const V8*>(kr + 16 * kk + 8 * h);
      vB[kk] = *reinterpret_cast<const V8*>(vr + 16 * kk + 8 * h);
    }
  }
  const float b1v = (a.b1 && klive) ? (float)a.b1[z * a.b1_zs + key] : 0.f;
  const int64_t lrow = ((int64_t)z * a.H + hd) * a.S;
  const float LOG2E = 1.4426950408889634f;
  const float inv_keep = DROP ? 1.f / (1.f - a.pdrop) : 1.f;
  f32x16_t dk[D / 32], dv[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) { dk[dt][r] = 0.f; dv[dt][r] = 0.f; }
  float colsum = 0.f;
  const int nt = (a.S + BN - 1) / BN;
  const int gch = (lane >> 1) & 1, colhalf = (lane >> 4) & 1;

  QT stg;
  stg.load(a, Qp, Gp, lrow, b2mat, kbk * BM, 0, tid);
  stg.store(smem, tid);
  __syncthreads();
  for (int j = 0; j < nt; ++j) {
    const int q0 = j * BN;
    const char* Qt = smem;
    const char* Gt = Qt + QT::OFF_G;
    const float* lseT = reinterpret_cast<const float*>(Qt + QT::OFF_L) + 4 * h;
    const float* delT = lseT + BN;
    const char* b2t = Qt + QT::OFF_B2;
    // one 32-query half at a time (keeps the transient score / dP registers at 2 x 16)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      __builtin_amdgcn_sched_barrier(0);
      f32x16_t s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) { s[r] = 0.f; dp[r] = 0.f; }
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) {
        const V8 qa = *reinterpret_cast<const V8*>(Qt + (t * 32 + l32) * RS<D>() + (2 * kk + h) * 16);
        s = MF<T>::mma(qa, kB[kk], s);
        const V8 ga = *reinterpret_cast<const V8*>(Gt + (t * 32 + l32) * RS<D>() + (2 * kk + h) * 16);
        dp = MF<T>::mma(ga, vB[kk], dp);
      }
      // rows = queries q0 + t*32 + crow(r, h), column = this lane's key
      V8 pa[2], da[2];
#pragma unroll
      for (int ss = 0; ss < 2; ++ss) {
        V8 b2;
        if constexpr (PAIR) b2 = tr_read<V8>(b2t, QT::B2RS, t * 32 + 16 * ss + 4 * h, wid * 4 + colhalf * 2 + gch, lane);
#pragma unroll
        for (int g = 2 * ss; g < 2 * ss + 2; ++g) {
          const f32x4 l4 = *reinterpret_cast<const f32x4*>(lseT + t * 32 + 8 * g);
          const f32x4 d4 = *reinterpret_cast<const f32x4*>(delT + t * 32 + 8 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int r = 4 * g + i, e = r & 7;
            float x = s[r] * a.scale + b1v;
            if constexpr (PAIR) x += (float)b2[e];
            const float p = __builtin_amdgcn_exp2f((x - l4[i]) * LOG2E);
            float kf = 1.f;
            if constexpr (DROP) {
              const int q = q0 + t * 32 + 8 * g + 4 * h + i;
              const uint32_t kb = keep4(a.seed, (uint64_t)lrow + (uint64_t)q, (uint32_t)(key >> 2), a.thresh);
              kf = ((kb >> (key & 3)) & 1u) ? inv_keep : 0.f;
            }
            const float ds = p * (dp[r] * kf - d4[i]);
            colsum += ds;
            pa[ss][e] = (T)(p * kf);
            da[ss][e] = (T)ds;
          }
        }
      }
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) {
        const int ch0 = dt * 4 + colhalf * 2 + gch;
#pragma unroll
        for (int ss = 0; ss < 2; ++ss) {
          const int rb = t * 32 + 16 * ss + 4 * h;
          dv[dt] = MF<T>::mma(pa[ss], tr_read<V8>(Gt, RS<D>(), rb, ch0, lane), dv[dt]);
          dk[dt] = MF<T>::mma(da[ss], tr_read<V8>(Qt, RS<D>(), rb, ch0, lane), dk[dt]);
        }
      }
    }
    __syncthreads();
    if (j + 1 < nt) {
      stg.load(a, Qp, Gp, lrow, b2mat, kbk * BM, q0 + BN, tid);
      stg.store(smem, tid);
      __syncthreads();
    }
  }
  if (a.db1) {
    colsum += __shfl_xor(colsum, 32, 64);
    if (lane < 32 && klive) unsafeAtomicAdd(a.db1 + (int64_t)z * a.S + key, colsum);
  }
  const int64_t obase = ((int64_t)z * a.S) * a.H * D + (int64_t)hd * D;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int kr = key0w + crow(r, h);
    if (kr < a.S) {
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) {
        const int64_t idx = obase + (int64_t)kr * a.H * D + dt * 32 + l32;
        a.dk[idx] = (T)(dk[dt][r] * a.scale);
        a.dv[idx] = (T)dv[dt][r];
      }
    }
  }
}

// ---------------------------------------------------------------- passes 1 and 2 in one: sequences of up to 256, width 32, a pair bias
// One workgroup has all of a (z, h): a wave per 32 keys, with dK and dV of its keys in registers, and Q, dO and K whole in LDS (64-byte
// rows, chunks swizzled by the row). Scores, their exponentials and dS are made once for all three gradients instead of twice:
// the vector instructions around them are what bounds both passes. dS of a tile of 32 queries crosses LDS for dQ, 16 x 16
// pieces of which go to four waves in turn, while the others begin the next tile. The pair bias comes in the order of the
// accumulators (small_bias_order_kernel), 2 x 16 bytes a lane and tile from L2. Two workgroups of eight waves share a CU.
// [256, 256, 4, 32], us: 50 + 51 in two passes, 67 here, 20 of it the loads of two rounds of workgroups that all begin at once;
// four waves a SIMD, 900 clocks a tile each of vector instructions.
constexpr int WHOLE_S = 256, WHOLE_LDS = 3 * WHOLE_S * 64 + WHOLE_S * 64 + 2 * WHOLE_S * 4;

// bias2 [groups, S, S] -> [groups, query tiles, key tiles, 2, 64, 8]: element j of half g and lane l is query crow(8 g + j, l / 32), key
// l % 32 of the tile; zero past the end. A wave per tile.
template <typename T>
__global__ void __launch_bounds__(256) small_bias_order_kernel(const T* __restrict__ b2, T* __restrict__ out, int S, int nt, int64_t tiles) {
  const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= tiles) return;
  const int lane = threadIdx.x & 63, kt = (int)(w % nt), qt = (int)(w / nt % nt), key = 32 * kt + (lane & 31);
  const T* src = b2 + w / nt / nt * S * S;
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    typename MF<T>::V8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int q = 32 * qt + crow(8 * g + j, lane >> 5);
      v[j] = q < S && key < S ? src[(int64_t)q * S + key] : (T)0.f;
    }
    *reinterpret_cast<typename MF<T>::V8*>(out + w * 1024 + (g * 64 + lane) * 8) = v;
  }
}

__device__ __forceinline__ f32x4 mma16(bf16x8_t a, bf16x8_t b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4 mma16(f16x8_t a, f16x8_t b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

template <typename T, bool DB1, int NT>
__global__ void __launch_bounds__(NT ? NT * 64 : WHOLE_S * 2, 4) small_bwd_whole_kernel(SmallArgs<T> a, const T* b2o) {
  typedef typename MF<T>::V8 V8;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int nt = NT ? NT : blockDim.x / 64, rows = 32 * nt;   // tiles of 32, one a wave
  char *Qi = smem, *Gi = Qi + rows * 64, *Ki = Gi + rows * 64, *DS = Ki + rows * 64;   // DS: [key][32 queries]
  float *lseS = reinterpret_cast<float*>(DS + rows * 64), *delS = lseS + rows;
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int S = a.S, hd = blockIdx.x % a.H, z = blockIdx.x / a.H;
  const float LOG2E = 1.4426950408889634f;
  const T* Qp = a.q + z * a.qz + hd * a.qh;
  const T* Gp = a.dout + z * a.gz + hd * a.gh;
  const T* Kp = a.k + z * a.kz + hd * a.kh;
  const int64_t lrow = ((int64_t)z * a.H + hd) * S;

  // ---- Q, dO, K whole: chunk ch of row r at 64 r + 16 (ch ^ r / 4 % 4)
  u32x4_t st[3][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = tid + i * 64 * nt, r = min(c >> 2, S - 1), ch = c & 3;
    st[0][i] = *reinterpret_cast<const u32x4_t*>(Qp + (int64_t)r * a.qs + ch * 8);
    st[1][i] = *reinterpret_cast<const u32x4_t*>(Gp + (int64_t)r * a.gs + ch * 8);
    st[2][i] = *reinterpret_cast<const u32x4_t*>(Kp + (int64_t)r * a.ks + ch * 8);
  }
  // ---- this wave's keys as B operands (column: the lane's key), and its 32 queries' delta
  const int key = 32 * wid + l32, kc = min(key, S - 1);
  const bool live = key < S;
  V8 kB[2], vB[2];
  float delta = 0.f;
  {
    const T* kr = Kp + (int64_t)kc * a.ks;
    const T* vr = a.v + z * a.vz + hd * a.vh + (int64_t)kc * a.vs;
    const T* gr = Gp + (int64_t)kc * a.gs;
    const T* orow = a.o + z * a.oz + hd * a.oh + (int64_t)kc * a.os_;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      kB[kk] = *reinterpret_cast<const V8*>(kr + 16 * kk + 8 * h);
      vB[kk] = *reinterpret_cast<const V8*>(vr + 16 * kk + 8 * h);
      const V8 g = *reinterpret_cast<const V8*>(gr + 16 * kk + 8 * h), o = *reinterpret_cast<const V8*>(orow + 16 * kk + 8 * h);
#pragma unroll
      for (int e = 0; e < 8; ++e) delta += (float)g[e] * (float)o[e];
    }
    delta += __shfl_xor(delta, 32, 64);
  }
  const float b1v = !live ? -INFINITY : a.b1 ? (float)a.b1[z * a.b1_zs + key] : 0.f;
  const T* bp = b2o + (((int64_t)(z / a.b2_div) * a.H + hd) * nt * nt + wid) * 1024;  // tile (0, wid); the next: nt tiles on
  V8 bias[2] = {*reinterpret_cast<const V8*>(bp + lane * 8), *reinterpret_cast<const V8*>(bp + 512 + lane * 8)};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = tid + i * 64 * nt, r = c >> 2, at = r * 64 + 16 * ((c & 3) ^ ((r >> 2) & 3));
    *reinterpret_cast<u32x4_t*>(Qi + at) = st[0][i];
    *reinterpret_cast<u32x4_t*>(Gi + at) = st[1][i];
    *reinterpret_cast<u32x4_t*>(Ki + at) = st[2][i];
  }
  if (lane < 32) {  // queries past the end weigh nothing
    lseS[key] = live ? a.lse[lrow + key] : INFINITY;
    delS[key] = live ? -delta : 0.f;
    if (live) a.delta[lrow + key] = delta;
  }

  f32x16_t dk, dv;
#pragma unroll
  for (int r = 0; r < 16; ++r) dk[r] = dv[r] = 0.f;
  float colsum = 0.f;
  // (LDS alone: neither the bias on its way nor what is stored of dQ is waited for)
  auto sync = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  sync();
  for (int t = 0; t < nt; ++t) {
    // where a lane reads rows (A operands), columns of 32 (B of dK, dV) and of 16 (dQ), and writes dS: worked out anew for every
    // tile from a lane that the compiler takes for another each time (kept over the loop they would spill)
    int ln = tid & 63;
    asm volatile("" : "+v"(ln));
    const int hh = ln >> 5, k32 = ln & 31, gq = (ln >> 2) & 3, gch = (ln >> 1) & 1, gb = 8 * (ln & 1), colhalf = (ln >> 4) & 1;
    int ra[2], ta[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) ra[kk] = k32 * 64 + 16 * ((2 * kk + hh) ^ ((k32 >> 2) & 3));
#pragma unroll
    for (int hi = 0; hi < 2; ++hi) ta[hi] = (4 * hh + 8 * hi + gq) * 64 + 16 * ((colhalf * 2 + gch) ^ (hh + 2 * hi)) + gb;
    f32x16_t s, dp;  // dP starts at -delta; a zero of its own for every tile (one for all would hold 16 registers)
    float zero = 0.f;
    asm volatile("" : "+v"(zero));
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 d4 = *reinterpret_cast<const f32x4*>(delS + 32 * t + 8 * g + 4 * hh);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[4 * g + i] = zero;
        dp[4 * g + i] = d4[i];
      }
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      s = MF<T>::mma(*reinterpret_cast<const V8*>(Qi + t * 2048 + ra[kk]), kB[kk], s);
      dp = MF<T>::mma(*reinterpret_cast<const V8*>(Gi + t * 2048 + ra[kk]), vB[kk], dp);
    }
    V8 pa[2], da[2];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (g) __builtin_amdgcn_sched_barrier(0);  // (one group's constants at a time: registers)
      const f32x4 l4 = *reinterpret_cast<const f32x4*>(lseS + 32 * t + 8 * g + 4 * hh);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 4 * g + i;
        const float x = s[r] * a.scale + b1v + (float)bias[r >> 3][r & 7];
        const float p = __builtin_amdgcn_exp2f((x - l4[i]) * LOG2E), ds = p * dp[r];
        if constexpr (DB1) colsum += ds;
        pa[r >> 3][r & 7] = (T)p;
        da[r >> 3][r & 7] = (T)ds;
      }
    }
    if (t + 1 < nt) {  // (the next tile's bias comes while dQ is made)
      bp += (int64_t)nt * 1024;
      bias[0] = *reinterpret_cast<const V8*>(bp + ln * 8);
      bias[1] = *reinterpret_cast<const V8*>(bp + 512 + ln * 8);
    }
    if (t) sync();  // dS of the tile before has been read
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const s16x8 d8 = __builtin_bit_cast(s16x8, da[g >> 1]);
      s16x4 v4;
#pragma unroll
      for (int i = 0; i < 4; ++i) v4[i] = d8[4 * (g & 1) + i];
      // unit 2 g + h of the key's row
      *reinterpret_cast<s16x4*>(DS + (32 * wid + k32) * 64 + 8 * (hh ^ ((k32 >> 1) & 1)) + 16 * (g ^ ((k32 >> 2) & 3))) = v4;
    }
#pragma unroll
    for (int ss = 0; ss < 2; ++ss) {
      const int at = t * 2048 + ss * 1024;
      dv = MF<T>::mma(pa[ss], tr_pair<V8>(Gi + at + ta[0], Gi + at + ta[1]), dv);
      dk = MF<T>::mma(da[ss], tr_pair<V8>(Qi + at + ta[0], Qi + at + ta[1]), dk);
    }
    sync();
    // ---- dQ of the tile: four pieces of 16 x 16, over all keys, piece j by wave (4 t + j) % nt
#pragma unroll 1
    for (int j = (wid + 4 * nt * t - 4 * t) % nt; j < 4; j += nt) {
      const int qh = j >> 1, dh = j & 1, g4 = ln >> 4;
      int da_[2], kb_[2];
#pragma unroll
      for (int hi = 0; hi < 2; ++hi) {
        const int kr = 8 * g4 + 4 * hi + gq;
        da_[hi] = kr * 64 + 8 * ((4 * qh + (ln & 3)) ^ ((kr >> 1) & 7));
        kb_[hi] = kr * 64 + 16 * ((2 * dh + gch) ^ ((kr >> 2) & 3)) + gb;
      }
      f32x4 dq{0.f, 0.f, 0.f, 0.f};
      for (int c0 = 0; c0 < nt; c0 += 4) {  // four tiles' reads fly together
        V8 ds4[4], k4[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int at = min(c0 + c, nt - 1) * 2048;
          ds4[c] = tr_pair<V8>(DS + at + da_[0], DS + at + da_[1]);
          k4[c] = tr_pair<V8>(Ki + at + kb_[0], Ki + at + kb_[1]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (c0 + c < nt) dq = mma16(ds4[c], k4[c], dq);
      }
      T* out = a.out + z * a.dz + hd * a.dh + 16 * dh + (ln & 15);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int q = 32 * t + 16 * qh + 4 * g4 + i;
        if (q < S) out[(int64_t)q * a.ds] = (T)(dq[i] * a.scale);
      }
    }
  }
  if constexpr (DB1) {
    colsum += __shfl_xor(colsum, 32, 64);
    const int k = 32 * wid + (threadIdx.x & 63);
    if ((threadIdx.x & 63) < 32 && k < S) unsafeAtomicAdd(a.db1 + (int64_t)z * S + k, colsum);
  }
  // this wave's rows of dK and dV through its rows of the Q and dO images, which nobody reads any more, into 16-byte pieces
  int ln = tid & 63;
  asm volatile("" : "+v"(ln));
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int at = (32 * wid + crow(r, ln >> 5)) * 64 + (ln & 31) * 2;
    *reinterpret_cast<T*>(Qi + at) = (T)(dk[r] * a.scale);
    *reinterpret_cast<T*>(Gi + at) = (T)dv[r];
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 32 * wid + 16 * i + (ln >> 2), ch = ln & 3;
    const u32x4_t k4 = *reinterpret_cast<const u32x4_t*>(Qi + r * 64 + ch * 16), v4 = *reinterpret_cast<const u32x4_t*>(Gi + r * 64 + ch * 16);
    if (r < S) {
      const int64_t at = (((int64_t)z * S + r) * a.H + hd) * 32 + ch * 8;
      *reinterpret_cast<u32x4_t*>(a.dk + at) = k4;
      *reinterpret_cast<u32x4_t*>(a.dv + at) = v4;
    }
  }
}

// ---------------------------------------------------------------- pass 3: dB2 summed over the z sharing it
template <typename T, int D, bool DROP>
__global__ void __launch_bounds__(NTHR, 2) small_bwd_db2_kernel(SmallArgs<T> a) {
  typedef typename MF<T>::V8 V8;
  typedef KeyTile<T, D, true> Block;    // stages the bias2 block once
  typedef KeyTile<T, D, false> KT;
  __shared__ __attribute__((aligned(16))) char smem[2 * KT::BYTES > BM * Block::B2RS ? 2 * KT::BYTES : BM * Block::B2RS];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, h = lane >> 5, l32 = lane & 31;
  const int nqb = (a.S + BM - 1) / BM, nkt = (a.S + BN - 1) / BN;
  int bid = blockIdx.x;
  const int kt = bid % nkt; bid /= nkt;
  const int qb = bid % nqb; bid /= nqb;
  const int hd = bid % a.H; bid /= a.H;
  const int zb = bid % (a.Z / a.b2_div), split = bid / (a.Z / a.b2_div);
  const int n_lo = (int)((int64_t)a.b2_div * split / a.nsplit), n_hi = (int)((int64_t)a.b2_div * (split + 1) / a.nsplit);
  const int q0w = qb * BM + wid * 32, qrow = q0w + l32;
  const int qc = min(qrow, a.S - 1);
  const bool qlive = qrow < a.S;
  const int k0 = kt * BN;
  const int64_t b2mat = ((int64_t)zb * a.H + hd) * a.S * a.S;
  const float LOG2E = 1.4426950408889634f;
  const float inv_keep = DROP ? 1.f / (1.f - a.pdrop) : 1.f;
  f32x16_t acc[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;

  // the lane's part of the bias2 block stays in its registers for all z
  typedef T T4 __attribute__((ext_vector_type(4)));
  T4 b2[2][4];
  {
    u32x4_t rb[4];
    bias_chunks<8, false>(a, b2mat, qb * BM, k0, tid, rb);  // (sums of keys past the end are not stored)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = tid + i * NTHR, row = c >> 3, ch = c & 7;
      st16_as_2x8(smem + row * Block::B2RS + ch * 16, rb[i]);
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        b2[t][g] = *reinterpret_cast<const T4*>(smem + (wid * 32 + l32) * Block::B2RS + (t * 32 + 8 * g + 4 * h) * 2);
    __syncthreads();
  }
  // per-z operands of the lane's query row, prefetched one z ahead
  V8 qf[D / 16], gf[D / 16];
  float lse = 0.f, delta = 0.f;
  auto load_rows = [&](int z) {
    const T* qr = a.q + z * a.qz + hd * a.qh + (int64_t)qc * a.qs;
    const T* gr = a.dout + z * a.gz + hd * a.gh + (int64_t)qc * a.gs;
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) {
      qf[kk] = *reinterpret_cast<const V8*>(qr + 16 * kk + 8 * h);
      gf[kk] = *reinterpret_cast<const V8*>(gr + 16 * kk + 8 * h);
    }
    const int64_t lrow = ((int64_t)z * a.H + hd) * a.S;
    lse = a.lse[lrow + qc];
    delta = a.delta[lrow + qc];
  };
  KT stg;
  auto load_keys = [&](int z) {
    stg.load(a, a.k + z * a.kz + hd * a.kh, a.v + z * a.vz + hd * a.vh, a.b1 ? a.b1 + z * a.b1_zs : nullptr, 0, 0, k0, tid);
  };
  load_keys(zb * a.b2_div + n_lo);
  stg.store(smem, tid);
  load_rows(zb * a.b2_div + n_lo);
  __syncthreads();
  for (int n = n_lo; n < n_hi; ++n) {
    const int z = zb * a.b2_div + n, cur = (n - n_lo) & 1;
    const bool more = n + 1 < n_hi;
    if (more) load_keys(z + 1);
    const char* buf = smem + cur * KT::BYTES;
    const float lse_n = lse, delta_n = delta;
    V8 qc_[D / 16], gc_[D / 16];
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) { qc_[kk] = qf[kk]; gc_[kk] = gf[kk]; }
    if (more) load_rows(z + 1);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) asm volatile("" : "+v"(b2[t][g]));  // (stays as it is: not held as 32 floats across the loop)
#pragma unroll
    for (int t = 0; t < 2; ++t) {  // one 32-key half at a time, and in the schedule too (registers)
      __builtin_amdgcn_sched_barrier(0);
      f32x16_t s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = 0.f;
        dp[r] = DROP ? 0.f : -delta_n;  // (a vector instruction a score less: [256, 256, 4, 32] 38.0 -> 37.3 us)
      }
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) {
        const V8 kv = *reinterpret_cast<const V8*>(buf + (t * 32 + l32) * RS<D>() + (2 * kk + h) * 16);
        s = MF<T>::mma(kv, qc_[kk], s);
        const V8 vv = *reinterpret_cast<const V8*>(buf + KT::OFF_V + (t * 32 + l32) * RS<D>() + (2 * kk + h) * 16);
        dp = MF<T>::mma(vv, gc_[kk], dp);
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        uint32_t kb = 0xfu;
        if constexpr (DROP)
          kb = keep4(a.seed, ((uint64_t)z * a.H + hd) * (uint64_t)a.S + (uint64_t)qrow,
                     (uint32_t)((k0 + t * 32 + 8 * g + 4 * h) >> 2), a.thresh);
        const f32x4 b1 = *reinterpret_cast<const f32x4*>(buf + KT::OFF_B1 + 16 * h + (t * 32 + 8 * g) * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 4 * g + i;
          const float p = __builtin_amdgcn_exp2f((s[r] * a.scale + (b1[i] + (float)b2[t][g][i]) - lse_n) * LOG2E);
          if constexpr (DROP) dp[r] *= ((kb >> i) & 1u) ? inv_keep : 0.f;
          acc[t][r] += p * (DROP ? dp[r] - delta_n : dp[r]);
        }
      }
    }
    if (more) stg.store(smem + (cur ^ 1) * KT::BYTES, tid);
    __syncthreads();
  }
  if (!qlive) return;
  // several workgroups: each writes its own sums, `sum_parts_kernel` adds them up in their order
  float* out = (a.nsplit > 1 ? a.part + (int64_t)split * (a.Z / a.b2_div) * a.H * a.S * a.S : a.db2) + b2mat + (int64_t)qrow * a.S;
  const bool st4 = (a.S & 3) == 0;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int kb4 = k0 + t * 32 + 8 * g + 4 * h;
      if (st4) {
        if (kb4 < a.S) {
          f32x4 w;
#pragma unroll
          for (int i = 0; i < 4; ++i) w[i] = acc[t][4 * g + i];
          *reinterpret_cast<f32x4*>(out + kb4) = w;
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (kb4 + i < a.S) out[kb4 + i] = acc[t][4 * g + i];
      }
    }
}

// out[i] = sum over s of part[s][i], in a fixed order: a wave's lanes have four results each, its workgroup's waves a quarter of the parts,
// eight of them on their way at once (a thread to itself waited for one part after the other: 64 parts of [8, 32, 32] 20 us, now 7; 16 of
// [4, 256, 256] 5.8 and 4.8). O: float, or the inputs' type, where that is the gradient's (a launch of 4 us for the cast less: forward and
// backward of [512, 256, 4, 32] 258 -> 252 us, [1024, 256, 4, 32] 517 -> 510; at [256, 256, 4, 32] the host takes as long as the kernels)
template <typename O>
__global__ void __launch_bounds__(256) sum_parts_kernel(const float* __restrict__ part, O* __restrict__ out, int64_t n, int parts) {
  typedef O O4 __attribute__((ext_vector_type(4)));
  __shared__ f32x4 sums[4][64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, lo = parts * wid / 4, hi = parts * (wid + 1) / 4;
  const int64_t i = ((int64_t)blockIdx.x * 64 + lane) * 4;
  const bool whole = n % 4 == 0;
  auto at = [&](int s) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (whole) {
      if (i < n) v = *reinterpret_cast<const f32x4*>(part + s * n + i);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i + e < n) v[e] = part[s * n + i + e];
    }
    return v;
  };
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  int s = lo;
  for (; s + 8 <= hi; s += 8) {
    f32x4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = at(s + u);
#pragma unroll
    for (int u = 0; u < 8; ++u) sum += v[u];
  }
  for (; s < hi; ++s) sum += at(s);
  sums[wid][lane] = sum;
  __syncthreads();
  if (wid) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) sum += sums[w][lane];
  if (whole) {
    if (i < n) *reinterpret_cast<O4*>(out + i) = O4{(O)sum[0], (O)sum[1], (O)sum[2], (O)sum[3]};
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (i + e < n) out[i + e] = (O)sum[e];
  }
}

// Workgroups that share the z of one pair-bias tile: as many as the chip holds at once (two a CU; [256, 256, 4, 32]: 47 us, with
// 768 51, with 1024 53), at least four z each.
int db2_splits(int Z, int H, int S, int b2_div) {
  const int64_t base = (int64_t)(Z / b2_div) * H * ((S + BM - 1) / BM) * ((S + BN - 1) / BN);
  return b2_div == 1 ? 1 : (int)std::max<int64_t>(1, std::min<int64_t>(b2_div / 4, 512 / base));
}

// Elements of the pair bias in the accumulators' order, for what goes through one pass for dQ, dK and dV; 0: two passes. Pair biases
// of their own for every z would be read and written once more than they are used, and fewer than a workgroup a CU leave the chip
// idle (dQ, dK and dV in two passes and in one, us: [32, 256, 4, 32] 23 and 24, [24, 40, 4, 32] 13 and 14; [128, 200, 4, 32] 54 and 36,
// [100, 133, 8, 32] 69 and 49, [512, 32, 8, 32] 61 and 23, [256, 250, 8, 32] 185 and 133). Of four tiles, which fill the two passes'
// workgroups and have no kernel of their own here, more of them: [100, 128, 4, 32] 21.6 and 23.1, [128, 128, 4, 32] 22.7 and 24.8, [160, 128, 4,
// 32] 28.6 and 28.5, [256, 128, 4, 32] 42 and 34.
int64_t small_order_elements(int Z, int H, int S, int D, int b2_div, bool drop) {
  const int64_t nt = (S + 31) / 32, least = nt == 4 ? 640 : 256;
  return D == 32 && S <= WHOLE_S && !drop && b2_div > 1 && (int64_t)Z * H >= least ? (int64_t)(Z / b2_div) * H * nt * nt * 1024 : 0;
}

// Kernels of their own for one tile and for five to eight: in the one for any number, addresses and the turns at dQ are a quarter of a
// tile's instructions ([256, 256, 4, 32] 81 us for 67, [200, 251, 8, 32] 135 and 107, [100, 133, 8, 32] 51 and 43, [512, 32, 8, 32] 23 and 20). (Two to four have the registers for it no more: 30 to 100 of them in scratch memory.)
template <typename T, bool DB1, int NT>
int launch_whole(const SmallArgs<T>& a, hipStream_t st) {
  const int nt = (a.S + 31) / 32;
  if constexpr (NT != 0) {
    if (nt != NT) return launch_whole<T, DB1, NT == 1 ? 0 : NT == 5 ? 1 : NT - 1>(a, st);
  }
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&small_bwd_whole_kernel<T, DB1, NT>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, WHOLE_LDS);
    attr = true;
  }
  const int64_t tiles = (int64_t)(a.Z / a.b2_div) * a.H * nt * nt;
  hipLaunchKernelGGL(small_bias_order_kernel<T>, dim3((unsigned)((tiles + 3) / 4)), dim3(256), 0, st, a.b2, a.order, a.S, nt, tiles);
  DS_CHECK_LAUNCH();
  hipLaunchKernelGGL((small_bwd_whole_kernel<T, DB1, NT>), dim3(a.H * a.Z), dim3(64 * nt), WHOLE_LDS / 8 * nt, st, a, (const T*)a.order);
  DS_CHECK_LAUNCH();
  return 0;
}

template <typename T, int D, bool DROP, bool PAIR>
int launch_small(SmallArgs<T> a, bool bwd, hipStream_t st) {
  const int nqb = (a.S + BM - 1) / BM;
  const dim3 grid(nqb * a.H * a.Z);
  if (!bwd) {
    if constexpr (D == 32 && !DROP && PAIR) {
      // (below 8 keys a row has no 16 bytes of bias; above 256 K and V would leave a CU one workgroup)
      const int qt = (a.S + 31) / 32, blocks = (qt + FWD_WAVES - 1) / FWD_WAVES, waves = (qt + blocks - 1) / blocks;
      const int64_t groups = (int64_t)blocks * a.H * a.Z;
      const bool shared_worse = (waves > 5 && groups <= 128) || (waves == FWD_WAVES && groups > 256 && groups <= 384);
      if (a.Sk >= 8 && a.Sk <= FWD_WHOLE && !shared_worse) {
        const int rows = (a.Sk + 31) / 32 * 32;
        hipLaunchKernelGGL(small_fwd_whole_kernel<T>, dim3((unsigned)groups), dim3(64 * waves), rows * (2 * 64 + 4) + waves * 128, st, a);
        DS_CHECK_LAUNCH();
        return 0;
      }
    }
    hipLaunchKernelGGL((small_fwd_kernel<T, D, DROP, PAIR>), grid, dim3(NTHR), 0, st, a);
    DS_CHECK_LAUNCH();
    return 0;
  }
  bool whole = false;
  if constexpr (D == 32 && !DROP && PAIR) {
    if (small_order_elements(a.Z, a.H, a.S, D, a.b2_div, false) > 0) {
      whole = true;
      if (a.order == nullptr) return (int)hipErrorInvalidValue;
      if (int rc = a.db1 ? launch_whole<T, true, WHOLE_S / 32>(a, st) : launch_whole<T, false, WHOLE_S / 32>(a, st)) return rc;
    }
  }
  if (!whole) {
    hipLaunchKernelGGL((small_bwd_dq_kernel<T, D, DROP, PAIR>), grid, dim3(NTHR), 0, st, a);
    DS_CHECK_LAUNCH();
    hipLaunchKernelGGL((small_bwd_dkv_kernel<T, D, DROP, PAIR>), grid, dim3(NTHR), 0, st, a);
    DS_CHECK_LAUNCH();
  }
  if (PAIR && a.db2 && a.b2_div > 1) {
    a.nsplit = db2_splits(a.Z, a.H, a.S, a.b2_div);
    if (a.nsplit > 1 && a.part == nullptr) return (int)hipErrorInvalidValue;
    const dim3 g3((a.Z / a.b2_div) * a.H * nqb * ((a.S + BN - 1) / BN) * a.nsplit);
    hipLaunchKernelGGL((small_bwd_db2_kernel<T, D, DROP>), g3, dim3(NTHR), 0, st, a);
    DS_CHECK_LAUNCH();
    if (a.nsplit > 1) {
      const int64_t n = (int64_t)(a.Z / a.b2_div) * a.H * a.S * a.S;
      const dim3 g4((unsigned)((n + 255) / 256));
      if (a.db2_as_in) hipLaunchKernelGGL(sum_parts_kernel<T>, g4, dim3(256), 0, st, a.part, (T*)a.db2, n, a.nsplit);
      else hipLaunchKernelGGL(sum_parts_kernel<float>, g4, dim3(256), 0, st, a.part, a.db2, n, a.nsplit);
      DS_CHECK_LAUNCH();
    }
  }
  return 0;
}

template <typename T>
int dispatch_small(SmallArgs<T> a, int D, bool bwd, hipStream_t st) {
  auto by_bias = [&](auto d, auto drop) {
    constexpr int DD = decltype(d)::value;
    constexpr bool DR = decltype(drop)::value;
    return a.b2 ? launch_small<T, DD, DR, true>(a, bwd, st) : launch_small<T, DD, DR, false>(a, bwd, st);
  };
  auto by_drop = [&](auto d) { return a.pdrop > 0.f ? by_bias(d, std::true_type{}) : by_bias(d, std::false_type{}); };
  if (D == 32) return by_drop(std::integral_constant<int, 32>{});
  if (D == 64) return by_drop(std::integral_constant<int, 64>{});
  return (int)hipErrorInvalidValue;
}

}  // namespace

// Forward. strides[12] = (q z,s,h)(k)(v)(o); dtype DS_BF16 / DS_F16; b1 / b2 may be null; b2_numel: elements that may be read
// at b2, at least 8.
extern "C" int ds_flash_small_fwd(const void* q, const void* k, const void* v, void* o, float* lse, const void* b1,
                                  const void* b2, const int64_t* st, int64_t b1_zs, int Z, int H, int S, int Sk, int D,
                                  int b2_div, float scale, float pdrop, uint64_t seed, int64_t b2_numel, int dtype,
                                  hipStream_t stream) {
  if (Z <= 0 || H <= 0 || S <= 0 || Sk <= 0 || b2_div <= 0 || (D != 32 && D != 64) || pdrop < 0.f || pdrop >= 1.f ||
      (b2 != nullptr && b2_numel < 8))
    return (int)hipErrorInvalidValue;
  const uint32_t thresh = (uint32_t)fminf(4294967295.f, pdrop * 4294967296.f);
#define DS_SMALL_ARGS(T)                                                                                        \
  SmallArgs<T> a{(const T*)q, (const T*)k, (const T*)v, nullptr, nullptr, (T*)o, lse, (const T*)b1, (const T*)b2, \
                 nullptr, nullptr, nullptr, nullptr, nullptr, st[0], st[1], st[2], st[3], st[4], st[5], st[6], st[7],     \
                 st[8], st[9], st[10], st[11], 0, 0, 0, 0, 0, 0, b1_zs, Z, H, S, b2_div, scale, pdrop, thresh, seed, b2_numel - 8, 1, nullptr, nullptr, Sk};
  if (dtype == DS_BF16) {
    DS_SMALL_ARGS(bf16)
    return dispatch_small<bf16>(a, D, false, stream);
  }
  if (dtype == DS_F16) {
    DS_SMALL_ARGS(fp16)
    return dispatch_small<fp16>(a, D, false, stream);
  }
  return (int)hipErrorInvalidValue;
#undef DS_SMALL_ARGS
}

// Backward. strides[18] = (q)(k)(v)(o)(dO)(dQ); dk / dv dense [Z, S, H, D] in the input dtype; delta fp32 [Z, H, S]
// scratch; db1 [Z, S] fp32 (zeroed by the caller) or null; db2 [Z / b2_div, H, S, S] fp32 (fully written) or null, db2_part
// `ds_flash_small_db2_splits` times as much scratch when that is more than one; then, with db2_as_in, db2 is of the inputs' type.
extern "C" int ds_flash_small_db2_splits(int Z, int H, int S, int b2_div) { return db2_splits(Z, H, S, b2_div); }

// order: ds_flash_small_order elements of the inputs' type when that is not zero
extern "C" int64_t ds_flash_small_order(int Z, int H, int S, int D, int b2_div, float pdrop, int has_b2) {
  return has_b2 ? small_order_elements(Z, H, S, D, b2_div, pdrop > 0.f) : 0;
}

extern "C" int ds_flash_small_bwd(const void* q, const void* k, const void* v, const void* o, const void* dout,
                                  const float* lse, const void* b1, const void* b2, void* dq, void* dk, void* dv,
                                  float* delta, float* db1, float* db2, float* db2_part, int db2_as_in, void* order,
                                  const int64_t* st, int64_t b1_zs, int Z, int H, int S, int D,
                                  int b2_div, float scale, float pdrop, uint64_t seed, int64_t b2_numel, int dtype,
                                  hipStream_t stream) {
  if (Z <= 0 || H <= 0 || S <= 0 || b2_div <= 0 || (D != 32 && D != 64) || pdrop < 0.f || pdrop >= 1.f ||
      (b2 != nullptr && b2_numel < 8))
    return (int)hipErrorInvalidValue;
  const uint32_t thresh = (uint32_t)fminf(4294967295.f, pdrop * 4294967296.f);
#define DS_SMALL_ARGS(T)                                                                                           \
  SmallArgs<T> a{(const T*)q, (const T*)k, (const T*)v, (const T*)o, (const T*)dout, (T*)dq, (float*)lse,           \
                 (const T*)b1, (const T*)b2, (T*)dk, (T*)dv, delta, db1, db2, st[0], st[1], st[2], st[3], st[4], st[5], st[6],      \
                 st[7], st[8], st[9], st[10], st[11], st[12], st[13], st[14], st[15], st[16], st[17], b1_zs, Z, H, S, b2_div, scale, pdrop, \
                 thresh, seed, b2_numel - 8, 1, db2_part, (T*)order, S, db2_as_in};
  if (dtype == DS_BF16) {
    DS_SMALL_ARGS(bf16)
    return dispatch_small<bf16>(a, D, true, stream);
  }
  if (dtype == DS_F16) {
    DS_SMALL_ARGS(fp16)
    return dispatch_small<fp16>(a, D, true, stream);
  }
  return (int)hipErrorInvalidValue;
#undef DS_SMALL_ARGS
}
