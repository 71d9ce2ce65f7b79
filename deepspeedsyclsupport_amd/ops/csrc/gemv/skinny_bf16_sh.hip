// bf16 products of decode-sized batches over a PRE-SHUFFLED weight: y[M, N] = X[M, K] . W[N, K]^T, M <= 48, with what stands
// around them in a decoder layer: the RMS norm of X, bias, residual, gated or plain activation.
//
// Reference counterpart (behaviour): the bf16 / fp16 decode GEMMs of `transformer_inference` (`qkv_gemm`,
// `vector_matmul`, `mlp_gemm`; `csrc/transformer/inference/csrc/pt_binding.cpp`), which call the vendor GEMM on the
// row-major weight.
//
// A decode GEMM is a weight stream, and the HBM stream only runs at full rate when every load instruction covers
// long contiguous segments. Inference weights are constants, so the matrix is re-laid ONCE into operand order:
//   Wsh[nb][kq][h][lane][8] = W[16 nb + (lane & 15)][64 kq + 16 (lane >> 4) + 8 h + 0..7]    (2 KB per 16 x 64 tile)
// so each 16-byte-per-lane load reads 1 KB contiguous and IS the A operand of one v_mfma_f32_16x16x32_bf16 (X is
// loaded with the same k permutation).
//  * a workgroup owns RB blocks of 16 weight rows over all of K and up to 48 token rows: its eight waves take alternating steps
//    of 64 columns, straight into registers, and their sums meet in LDS once. No atomics: sums stay in one fixed order and the
//    result leaves as bf16, from this launch, or where wide batches cut K into parts (`cut_of`) from a second one;
//  * the norm costs no pass: y = rs (X w) . W^T with rs the row's 1 / rms, and every workgroup sees all of X anyway. It
//    multiplies X by the norm's weight on the way to the matrix cores, adds up the squares beside, and scales the sums;
//  * a gated pair (gate block i, up block i + N / 32) sits in one workgroup: act(gate) up leaves, half of N. Halves that are no whole
//    blocks (no norm) leave as sums, and a second launch pairs them;
//  * X is read once per workgroup (from L2), which is what bounds wide batches; RB and the parts trade that against workgroups
//    enough.
// Two workgroups fit a CU with up to four blocks where X is normed (128 registers a lane: 33 / 48 rows x gated [28672, 4096] 51.8 / 52.4 us
// with one, 47.3 / 50.2 with two), whose products wait for vector instructions; without, one with all its registers is faster (33 / 48
// rows x [16384, 8192] 47 / 48, with two 56 / 49; [4096, 14336] in parts 28 / 28 and 31 / 29; gated [22016, 4096] 42 / 45 and 45 / 46). One with
// eight.
// Bound by the weights' read (6.5 TB/s here). Measured, us (the same products as split streams with fp32 atomics and a finalize
// pass; the floor): 12 rows x [4096, 4096] 9 (14; 5), [4096, 14336] 23 (25; 18), gated [28672, 4096] 38 (45; 36), with the
// norm 39, [32000, 4096] 42 (51; 40), [2048, 2048] 5.6 (7.6; 1.3). 24 and 40 rows (library GEMM): gated [28672, 4096] 44 and 51 (60
// and 58 with its activation), [4096, 4096] 11 and 14 (13 and 14), [14368, 4096] 25 and 28 (27 and 28).
// Prefill (more rows) un-shuffles into a row-major temporary for the library GEMM (`ds_unshuffle_sh16`),
// or uses the row-major copy the caller kept.
#include "ds_hip.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
constexpr int WAVES = 8;

struct ShArgs {
  const bf16* x;       // [M, K]
  const bf16* w;       // shuffled
  const bf16* bias;    // [N] or null
  const bf16* norm_w;  // [K] (NORM)
  const bf16* res;     // [M, N] or null: added at the end
  bf16* y;             // [M, N], gated [M, N / 2]
  int M, N, K;
  float eps;
  int act;             // gated: activation code; else code + DS_ACT_UNARY, or -1
  float limit;         // of the clamped gated activation
  int parts;           // of K, each with workgroups of its own (1: all of it)
  f32x4* part;         // their sums [parts][blocks][MT][64], as the accumulators lie (null: the result leaves from here)
};

template <int V>
struct Int {
  static constexpr int value = V;
};

// The address as a wave's base in scalar registers and a lane's bytes; the asm keeps it so: 10 to 20 vector registers less.
__device__ __forceinline__ const bf16x8_t* at(const bf16* base, uint32_t bytes) {
  asm("" : "+v"(bytes));
  return reinterpret_cast<const bf16x8_t*>(reinterpret_cast<const char*>(base) + bytes);
}

// Token row `row`, columns n .. n + 3 of a product without a gate: bias, activation, residual
__device__ __forceinline__ void store_plain(const ShArgs& a, f32x4 v, int row, int n) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int c = n + e;
    if (c >= a.N) continue;
    float r = v[e] + (a.bias ? (float)a.bias[c] : 0.f);
    if (a.act >= 0) r = act_any(a.act - DS_ACT_UNARY, r);
    if (a.res) r += (float)a.res[(int64_t)row * a.N + c];
    v[e] = r;
  }
  bf16* yr = a.y + (int64_t)row * a.N + n;
  if (a.N % 4 == 0) {
    if (n < a.N) {
      bf16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (bf16)v[e];
      *reinterpret_cast<bf16x4*>(yr) = o;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < a.N) yr[e] = (bf16)v[e];
  }
}

// Column c of a gated result
__device__ __forceinline__ float gate_up(const ShArgs& a, float g, float up, int row, int c, int cols) {
  g += a.bias ? (float)a.bias[c] : 0.f;
  up += a.bias ? (float)a.bias[cols + c] : 0.f;
  const float r = a.act == DS_ACT_CLAMPED_GLU ? clamped_glu_f(g, up, a.limit) : act_any(a.act, g) * up;
  return a.res ? r + (float)a.res[(int64_t)row * cols + c] : r;
}

template <int MT, int RB, bool NORM, bool GATED>
__global__ void __launch_bounds__(WAVES * 64, (MT <= 2 || (RB == 4 && NORM) ? 4 : 2)) decode_gemm_kernel(ShArgs a) {
  static_assert(!GATED || RB % 2 == 0, "pairs");
  constexpr int T = MT * RB, HALF = WAVES / 2;
  constexpr int U = T == 1 ? 2 : 1;  // steps loaded together
  __shared__ f32x4 red[HALF][T][64];
  __shared__ float ssq[WAVES][MT][16], scale[MT * 16];
  const int lane = threadIdx.x & 63, l16 = lane & 15, q4 = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int K = a.K, KQ = K / 64, NB = (a.N + 15) / 16, HB = a.N / 32;
  const bool split = !NORM && !GATED && a.part != nullptr;
  const int first = split ? (int)((int64_t)KQ * blockIdx.y / a.parts) : 0,
            end = split ? (int)((int64_t)KQ * (blockIdx.y + 1) / a.parts) : KQ;  // steps of K
  // block i of this workgroup
  auto block_of = [&](int i) {
    if (!GATED) return (int)blockIdx.x * RB + i;
    return (int)blockIdx.x * (RB / 2) + i % (RB / 2) + (i < RB / 2 ? 0 : HB);
  };
  // 33 rows and more: bases per wave and bytes per lane (`at`); up to 32, which have the registers, pointers per lane. (Those as a
  // base and bytes without the asm: hipcc 7.2 forms a step's addresses in the upper registers of the second block's sums, <1, 2, false,
  // true> and <2, 2, false, true>. A test reads the assembly for that.)
  constexpr bool APART = MT == 3;
  const bf16* wp[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int last = GATED ? (i < RB / 2 ? HB : 2 * HB) - 1 : NB - 1;
    wp[i] = a.w + (int64_t)min(block_of(i), last) * KQ * 1024 + (APART ? 0 : lane * 8);
  }
  const bf16* xp[MT];
  uint32_t xo[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = min(16 * m + l16, a.M - 1);
    xo[m] = ((uint32_t)row * K + 16 * q4) * 2;
    xp[m] = APART ? a.x : a.x + (int64_t)row * K + 16 * q4;
  }
  const bf16* np = NORM ? a.norm_w + (APART ? 0 : 16 * q4) : nullptr;
  auto from = [&](const bf16* p, uint32_t bytes) {
    if constexpr (APART) return at(p, bytes);
    else return reinterpret_cast<const bf16x8_t*>(p);
  };

  f32x4 acc[RB][MT];
  float ss[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    ss[m] = 0.f;
#pragma unroll
    for (int i = 0; i < RB; ++i) acc[i][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  struct Steps {
    bf16x8_t w[U][2][RB], x[U][2][MT], norm[U][2];
  };
  // U steps, WAVES apart: all their loads (past the end the last step again, which counts for nothing) before the products
  // of the steps at hand: without the barrier the compiler sinks them and a wave has a load or two in flight
  auto load = [&](Steps& f, int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < RB; ++i)
          f.w[u][h][i] = __builtin_nontemporal_load(
              from(wp[i] + (int64_t)min(s0 + WAVES * u, end - 1) * 1024 + 512 * h, lane * 16));
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = min(s0 + WAVES * u, end - 1) * 64 + 8 * h;
        if constexpr (NORM) f.norm[u][h] = *from(np + k, 32 * q4);
#pragma unroll
        for (int m = 0; m < MT; ++m) f.x[u][h][m] = *from(xp[m] + k, xo[m]);
      }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto products = [&](Steps& f, int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u && s0 + WAVES * u >= end) break;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          if constexpr (NORM) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const float v = (float)f.x[u][h][m][j];
              ss[m] = fmaf(v, v, ss[m]);
              f.x[u][h][m][j] = (bf16)(v * (float)f.norm[u][h][j]);
            }
          }
#pragma unroll
          for (int i = 0; i < RB; ++i)
            acc[i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[u][h][i], f.x[u][h][m], acc[i][m], 0, 0, 0);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int STRIDE = WAVES * U;
  int s = first + wid;
  if (s < end) {
    Steps f0;
    if constexpr (RB <= 2) {  // the next steps' loads run while these are multiplied
      Steps f1;
      load(f0, s);
      for (;;) {
        load(f1, s + STRIDE);
        products(f0, s);
        if ((s += STRIDE) >= end) break;
        load(f0, s + STRIDE);
        products(f1, s);
        if ((s += STRIDE) >= end) break;
      }
    } else {  // four blocks and more: other waves cover a step's waits (two to four on a SIMD), a second set of registers costs more of them
      for (; s < end; s += STRIDE) {
        load(f0, s);
        products(f0, s);
      }
    }
  }

  // ---- the waves' sums meet: the upper half's through LDS, then all four halves' sums
  if (wid >= HALF) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int m = 0; m < MT; ++m) red[wid - HALF][i * MT + m][lane] = acc[i][m];
  }
  if constexpr (NORM) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      float v = ss[m];
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      if (lane < 16) ssq[wid][m][l16] = v;
    }
  }
  __syncthreads();
  if (wid < HALF) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int m = 0; m < MT; ++m) red[wid][i * MT + m][lane] += acc[i][m];
  }
  if constexpr (NORM) {
    if (threadIdx.x < MT * 16) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) v += ssq[w][threadIdx.x / 16][threadIdx.x % 16];
      scale[threadIdx.x] = rsqrtf(v / K + a.eps);
    }
  }
  __syncthreads();
  // ---- lane: token row l16 of tile m, weight rows 4 q4 .. + 3 of a block
  const int cols = GATED ? a.N / 2 : a.N;
  for (int j = wid; j < (GATED ? T / 2 : T); j += WAVES) {
    const int i = j / MT, m = j % MT, row = 16 * m + l16, n = block_of(i) * 16 + 4 * q4;
    auto total = [&](int t) {
      f32x4 v = red[0][t][lane];
#pragma unroll
      for (int w = 1; w < HALF; ++w) v += red[w][t][lane];
      if constexpr (NORM) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= scale[row];
      }
      return v;
    };
    f32x4 v = total(j), u = GATED ? total(j + T / 2) : v;
    if (split) {
      if (block_of(i) < NB) a.part[(((int64_t)blockIdx.y * NB + block_of(i)) * MT + m) * 64 + lane] = v;
      continue;
    }
    if (row >= a.M) continue;
    if constexpr (!GATED) {
      store_plain(a, v, row, n);
      continue;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = n + e;
      if (c >= cols) continue;
      v[e] = gate_up(a, v[e], u[e], row, c, cols);
    }
    bf16x4 o;  // (whole blocks of columns)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (bf16)v[e];
    if (n < cols) *reinterpret_cast<bf16x4*>(a.y + (int64_t)row * cols + n) = o;
  }
}

// The parts' sums, always in the same order, and what is fused behind the product
__global__ void __launch_bounds__(256) decode_gemm_sum_kernel(ShArgs a, int blocks, int mt) {
  const int64_t per = (int64_t)blocks * mt * 64, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= per) return;
  f32x4 v = a.part[i];
  for (int p = 1; p < a.parts; ++p) v += a.part[p * per + i];
  const int lane = (int)(i & 63), t = (int)(i >> 6), row = 16 * (t % mt) + (lane & 15);
  if (row < a.M) store_plain(a, v, row, t / mt * 16 + 4 * (lane >> 4));
}

// The parts' sums of [gate | up] weights whose halves are no whole blocks of 16 rows: a thread per result. A launch of 2 us, the sums
// stay in the caches: 16 rows, us (split streams with fp32 atomics), [2800, 2048] 8.5 (7.5), [11280, 4096] 24.3 (24.3), [28688, 4096]
// 47 (48).
__global__ void __launch_bounds__(256) decode_gemm_gate_kernel(ShArgs a, int blocks, int mt) {
  const int cols = a.N / 2, row = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
  if (c >= cols) return;
  const float* part = reinterpret_cast<const float*>(a.part);
  const int64_t per = (int64_t)blocks * mt * 256;
  auto total = [&](int n) {
    const int64_t at = ((int64_t)(n / 16) * mt + row / 16) * 256 + ((row & 15) + 16 * (n % 16 / 4)) * 4 + n % 4;
    float v = part[at];
    for (int p = 1; p < a.parts; ++p) v += part[p * per + at];
    return v;
  };
  a.y[(int64_t)row * cols + c] = (bf16)gate_up(a, total(c), total(cols + c), row, c, cols);
}

// Pre-shuffled bf16 -> row-major bf16 [N, K]. One thread per 16-byte lane chunk (8 weights of one row).
__global__ void __launch_bounds__(256) unshuffle_sh16_kernel(const bf16* __restrict__ Wsh, bf16* __restrict__ W, int N,
                                                             int KQ) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;  // chunk = ((nb * KQ + kq) * 2 + h) * 64 + lane
  const int lane = (int)(c & 63);
  const int h = (int)((c >> 6) & 1);
  const int64_t t = c >> 7;
  const int kq = (int)(t % KQ);
  const int64_t nb = t / KQ;
  const int64_t row = nb * 16 + (lane & 15);
  if (row >= N) return;
  const bf16x8 v = *reinterpret_cast<const bf16x8*>(Wsh + c * 8);
  *reinterpret_cast<bf16x8*>(W + row * KQ * 64 + kq * 64 + 16 * (lane >> 4) + 8 * h) = v;
}

thread_local int g_blocks = 0, g_parts = 0;  // (a thread's own: another's products go by the rules, and keep to the scratch they asked for)

struct Cut {
  int blocks, parts;  // blocks of 16 weight rows per workgroup, parts of K
};
// As few blocks per workgroup as make no more workgroups than the chip has CUs: a second, partly filled round costs as much as the
// first (12 rows, us with one / two: [4096, 14336], 256 workgroups of one, 23 / 30; [6144, 4096] 15 / 11; 16 rows x [5120, 5120] 20 /
// 14; 48 rows with two / four: [8192, 4096] 19 / 24, [9216, 3072] 28 / 19, [12288, 4096] 35 / 26). Products with more blocks than that
// holds take the most that there are (24 rows x [32000, 4096] 48 with two, 46 with four), up to 16 token rows two (12 rows 42 and 45).
// Gated pairs take two or four (12 rows: [11264, 2048] 13.0 and 11.0, [28672, 4096] 41 and 38).
// Of 33 rows and more without a norm or a gate, what arrives here are widths that are no multiple of 8, gate halves that are no whole blocks, more than
// 16384 weight rows or 3 2^25 weights, and short K over more than 4096 rows: the others are the narrow products' (`narrow_instead`).
// Eight blocks for 33 rows and more of 4096 and more: X, a quarter to a half of what a CU reads, is then read half as often. One workgroup
// has a CU to itself, so their number decides: where four blocks (two a CU with a norm) fill their rounds as well or better, it stays at
// four. 33 / 48 rows, us with four and with eight. Normed, 129 to 256 workgroups of eight: [18432, 4096] 42 / 47 and 36 / 38, gated [22016, 4096]
// 43 / 48 and 40 / 41, [28672, 4096] 47 / 50 and 45 / 46, [32000, 4096] 48 / 53 and 48 / 50; 272 to 384 of them, a second round that is half
// empty: gated [38912, 4096] 65 / 71 and 78 / 82; 385 and more: [50304, 4096] 86 / 94 and 84 / 86, gated [57344, 8192] 162 / 184 and 156 / 161 ([128256,
// 4096], four rounds, 184 / 204 and 191 / 197). Without a norm, up to 200: [17408, 4096] 41 / 45 and 39 / 39, [20480, 5120] 52 / 57 and 48 / 49, gated
// [22016, 4096] 42 / 45 and 43 / 42; but gated [28672, 4096] 43.5 / 47 and 46 / 47, [32000, 4096] 48.6 / 49.6 and 52 / 51, [40960, 4096] 67 / 69 and
// 83 / 84, [65536, 4096] 93 / 97 and 102 / 103. Up to 1024 blocks four make one round (48 rows x [16384, 8192] 48 and 69), and X of 2048
// gives nothing (33 / 48 rows x [32000, 2048] 27 / 28 and 30 / 31). Up to 32 rows it pays for long X alone (32 rows x gated [28672, 4096] 46
// and 49).
// More than 16 token rows of 4096 and more over few blocks: what a CU can read (30 bytes a nanosecond) bounds one block's workgroup,
// and of that most is X. Several blocks share the reading, and parts of K keep the workgroups at 256; the parts' sums are a launch of
// 4 us. 33 / 48 rows, us with one block and with this: [4095, 4096] 13.8 / 16.5 and 13.5 / 15.3, [4095, 14336] 41 / 47 and 29 / 30, [2047, 5632]
// 16.8 / 20.5 and 12.8 / 13.9; 17 rows x [4096, 4096] 10.9 and 11.4, [4096, 14336] 27 and 24, [2048, 5632] 12.3 and 10.0. Over 2048 the launch costs what it
// gives ([2048, 2048] 10.2 and 9.9). Four blocks for 33 rows and more of 8192 ([4096, 14336] 33 with two; 17 rows 24.6 with four, 23.6 with two).
// The same between 256 and 680 blocks where X is long: four blocks and the parts that fill one round or two. Us without and with: 17 / 32 rows,
// [5120, 13824] 33 / 41 and 28 / 31, [8192, 8192] 27 / 29 and 28 / 28, [10240, 8192] 35 / 40 and 34 / 35; 33 / 48 rows, [5119, 13824] 47 / 54 and
// 34 / 35, [8191, 8192] 32 / 36 and 31.5 / 33, [10239, 8192] 46 / 51 and 40 / 43, gated [5136, 8192], whose halves are no whole blocks, 33 / 36 and 25 / 28;
// shorter ones stay whole ([7168, 7168] 21 / 24 and 23 / 24).
// Up to 16 rows parts pay at the ends alone: where a few blocks leave most CUs idle (16 rows x [1024, 4096] 8.7 and 7.7, 2 rows 6.1 and
// 6.9, x [1024, 8192] 9.6 and 8.4), and where long ones stand a quarter over one round (16 rows x [10240, 8192] 40 and 35); from 12 rows on
// also over long K, in two blocks, which halve the reading of X (12 / 16 rows x [2048, 5632] 10.4 / 11.7 and 9.5 / 9.7, [4096, 14336] 23.7 / 26.0 and 22.8 / 23.3,
// [5120, 13824] 29.9 / 31.6 and 27.6 / 28.5, [3072, 8192] 13.9 / 15.4 and 14.0 / 14.4; not [4096, 6144] 12.4 / 13.5 and 13.3 / 13.7).
Cut cut_of(int M, int N, int K, bool gated, bool norm) {
  const int blocks = gated ? N / 16 : (N + 15) / 16, mt = (M + 15) / 16, most = gated || mt > 1 ? 4 : 2;
  const int eights = (blocks + 7) / 8;  // workgroups of eight blocks
  const bool eight = mt == 3 && K >= 4096 && blocks > 1024 && (norm ? (eights - 1) % 256 >= 128 : eights <= 200);
  int rb = blocks <= 256 && !gated ? 1 : blocks <= 512 ? 2 : eight ? 8 : most, parts = 1;
  if (!gated && !norm) {
    int fill = 0;  // workgroups that parts may make
    if (mt == 1) {
      fill = blocks <= 64 && (K >= 8192 || (M > 8 && K >= 4096)) ? 256 : blocks > 512 && blocks <= 680 && K >= 8192 ? 1024 : 0;
      if (M >= 12 && blocks > 64 && blocks <= 340 && K >= (blocks <= 128 ? 5120 : 8192)) {
        rb = 2;
        fill = blocks <= 256 ? 256 : 512;
      }
    } else if (blocks <= 256 && K >= 4096) {
      rb = mt == 3 && K >= 8192 ? 4 : 2;
      fill = 256;
    } else if (blocks > 256 && blocks <= 680 && K * mt >= 16384) {
      rb = 4;
      fill = blocks <= 512 ? 256 : 512;
    }
    parts = max(min(min(fill / ((blocks + rb - 1) / rb), K / 1024), 8), 1);  // (K / 1024: two steps a wave)
  }
  if (g_blocks) rb = g_blocks >= 8 ? 8 : g_blocks >= 4 ? 4 : g_blocks == 3 ? 2 : g_blocks;
  if (gated && rb < 2) rb = 2;
  if (mt < 3 && rb == 8) rb = 4;
  if (mt == 1 && !gated && rb == 4) rb = 2;
  if (g_parts && !gated && !norm) parts = min(g_parts, K / 64);
  return {rb, parts};
}

// loose: gated, with halves that are no whole blocks
template <int MT, int RB>
int launch(const ShArgs& a, bool gated, bool loose, hipStream_t st) {
  const int blocks = gated ? a.N / 16 : (a.N + 15) / 16;
  const dim3 grid((blocks + RB - 1) / RB, a.parts), threads(WAVES * 64);
  if (gated) {
    if constexpr (RB > 1) {
      if (a.norm_w) hipLaunchKernelGGL((decode_gemm_kernel<MT, RB, true, true>), grid, threads, 0, st, a);
      else hipLaunchKernelGGL((decode_gemm_kernel<MT, RB, false, true>), grid, threads, 0, st, a);
    }
  } else if constexpr (MT > 1 || RB < 4) {
    if (a.norm_w) hipLaunchKernelGGL((decode_gemm_kernel<MT, RB, true, false>), grid, threads, 0, st, a);
    else hipLaunchKernelGGL((decode_gemm_kernel<MT, RB, false, false>), grid, threads, 0, st, a);
  }
  if (a.part && loose) hipLaunchKernelGGL(decode_gemm_gate_kernel, dim3((a.N / 2 + 255) / 256, a.M), dim3(256), 0, st, a, blocks, MT);
  else if (a.part) hipLaunchKernelGGL(decode_gemm_sum_kernel, dim3((blocks * MT * 64 + 255) / 256), dim3(256), 0, st, a, blocks, MT);
  DS_CHECK_LAUNCH();
  return 0;
}

}  // namespace

// Forces blocks per workgroup (1, 2, 4, 8, where the product has such a kernel) and parts of K, for the calling thread's products; 0: by
// the rule above.
extern "C" void ds_skinny_b16_tune(int cfg, int parts) { g_blocks = cfg; g_parts = parts; }

extern "C" int ds_decode_gemm_ok(int M, int K) { return M >= 1 && M <= 48 && K >= 64 && K % 64 == 0; }

// Most products of 33 rows and more, and some of 17, without a norm or a gate: the narrow products' kernel over the same weights (gemm/narrow_gemm.hip)
extern "C" int ds_narrow_ordered_ok(int64_t, int64_t, int64_t);
extern "C" int64_t ds_narrow_ordered_scratch(int64_t, int64_t, int64_t);
extern "C" int ds_narrow_ordered(const void*, const void*, const void*, const void*, void*, int64_t, int64_t, int64_t, int, void*, hipStream_t);
static bool narrow_instead(int M, int N, int K, int gated, bool norm) {
  return !gated && !norm && !g_blocks && !g_parts && ds_narrow_ordered_ok(M, N, K);
}

// Bytes of scratch memory that ds_decode_gemm wants for a product (0: none)
extern "C" int64_t ds_decode_gemm_scratch(int M, int N, int K, int gated, int norm) {
  if (narrow_instead(M, N, K, gated, norm)) return ds_narrow_ordered_scratch(M, N, K);
  const bool loose = gated && N % 32;
  const int parts = cut_of(M, N, K, gated && !loose, norm).parts;
  return parts > 1 || loose ? (int64_t)parts * ((N + 15) / 16) * ((M + 15) / 16) * 1024 : 0;
}

extern "C" int ds_unshuffle_sh16(const void* Wsh, void* W, int N, int K, hipStream_t st) {
  if (N <= 0 || K % 64) return (int)hipErrorInvalidValue;
  const int KQ = K / 64, NB = (N + 15) / 16;
  const int64_t chunks = (int64_t)NB * KQ * 128;
  hipLaunchKernelGGL(unshuffle_sh16_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, st,
                     (const bf16*)Wsh, (bf16*)W, N, KQ);
  DS_CHECK_LAUNCH();
  return 0;
}

// X [M, K] bf16 (M <= 48, K % 64 == 0), Wsh in the shuffled layout above (N padded to a multiple of 16). norm_w [K] or null: X
// is RMS-normed by it first. bias [N], res [M, N] or null. gated: N / 2 columns act(gate) up (N % 32 == 0, N % 2 without norm); else act: a
// code + DS_ACT_UNARY, or -1. part: ds_decode_gemm_scratch bytes.
extern "C" int ds_decode_gemm(const void* X, const void* Wsh, const void* bias, const void* norm_w, float eps, const void* res,
                              void* Y, int M, int N, int K, int gated, int act, float limit, void* part, hipStream_t st) {
  const bool loose = gated && N % 32;
  if (!ds_decode_gemm_ok(M, K) || N <= 0 || (loose && (N % 2 || norm_w))) return (int)hipErrorInvalidValue;
  if (narrow_instead(M, N, K, gated, norm_w != nullptr)) return ds_narrow_ordered(X, Wsh, bias, res, Y, M, N, K, act, part, st);
  if (loose) gated = 0;
  const Cut cut = cut_of(M, N, K, gated, norm_w != nullptr);
  if (cut.parts == 1 && !loose) part = nullptr;
  else if (!part) return (int)hipErrorInvalidValue;
  const ShArgs a{(const bf16*)X, (const bf16*)Wsh, (const bf16*)bias, (const bf16*)norm_w, (const bf16*)res, (bf16*)Y, M, N, K,
                 eps, act, limit, cut.parts, (f32x4*)part};
#define GO(MT)                                                          \
  switch (cut.blocks) {                                                 \
    case 1: return launch<MT, 1>(a, gated, loose, st);                  \
    case 2: return launch<MT, 2>(a, gated, loose, st);                  \
    case 4: return launch<MT, 4>(a, gated, loose, st);                  \
    default:                                                            \
      if constexpr (MT == 3) return launch<MT, 8>(a, gated, loose, st); \
      return (int)hipErrorInvalidValue;                                 \
  }
  switch ((M + 15) / 16) {
    case 1: GO(1)
    case 2: GO(2)
    default: GO(3)
  }
#undef GO
}
