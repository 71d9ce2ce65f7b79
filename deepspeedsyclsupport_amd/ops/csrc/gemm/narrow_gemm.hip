// bf16 products around a short batch of tokens (training steps and prompts of a few hundred): y = X W^T, dX = dY W and dW = dY^T X,
// each over the operands as they lie in memory, sums in fp32, one rounding at the end.
//
// What bounds them is latency and the count of workgroups, not the matrix cores: 128 tokens of a 1024-wide layer make 32 tiles of
// 64 x 64. Hence
//  * tiles of 128 x 256, 128 x 128 or 64 x 64 (four waves of 64 x 128, 64 x 64 or 32 x 32) or, where those are too few, of 32 rows by 32 or 64 (the
//    waves share each step's inner dimension and meet in LDS at the end, always in the same order), and K in parts with a second launch
//    for their sums;
//  * both operands come by DMA into four LDS buffers, three steps ahead (128 x 256: into three, two ahead); one barrier a step, whose wait
//    counts what may still be on its way;
//  * an operand whose rows run along the inner dimension is stored row by row, 128 bytes a step; one whose rows run across it (W in dX, both in
//    dW) as it lies, and read transposed (ds_read_b64_tr_b16). Chunks are swizzled by the source address, against bank conflicts;
//  * tiles of 128 rows have a CU to themselves, a wave on a SIMD: before each product it reads one operand of the next quarter step and sends
//    one transfer, the next step's first quarter too, behind a barrier that stands before the last. 3000 tokens by [11264, 2048], dW, us: a step's
//    reads, then its products 179; quarters 146; product by product 138, in tiles of 128 x 256 119 (library 147). Matrix cores busy 71 % of
//    the time, at 1.5 GHz;
//  * what lies past the end of a buffer reads as zero: ragged tokens need no other treatment, along the inner dimension neither.
// Besides, the library's call takes the host 18 to 23 us, this one 5 to 7: a training step of 128 tokens has 27 of them and waits for the host.
// Measured, us (the library's kernel): 128 tokens, layers [3072, 1024], [1024, 1024], [5632, 1024], [1024, 2816], head [8000, 1024]: y 6.4
// (9.4), 4.5 (8.2), 6.7 (9.8), 6.9 (7.9), 7.0 (10.1); dX 8.4 (13.4), 5.2 (11.0), 9.9 (21.1), 5.6 (11.3), 11.9 (30.9); dW 6.2 (7.2), 3.3 (5.3),
// 10.4 (9.3), 5.6 (7.4), 11.0 (10.1). 512 tokens, [3072, 1024]: 9.4 (10.6), 11.0 (16.1), 9.6 (11.9).
#include "ds_hip.h"

#include <algorithm>

namespace {

typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

template <int N>
struct Int {
  static constexpr int value = N;
};

struct NarrowArgs {
  const bf16 *a, *b;       // a: M x K, b: N x K, or with rows along k: K x M, K x N
  bf16* c;                 // [M, N]
  int M, N, K;
  uint32_t lda, ldb, abytes, bbytes;
  int parts;               // of K, each with workgroups of its own (1: all of it)
  f32x4* part;             // their sums [parts][M][N] (null: the result leaves from here)
  const bf16 *bias, *res;  // behind a product with an ordered operand: [N] or null, [M, N] or null
  int act;                 // ... an activation code + DS_ACT_UNARY, or -1
  int band;                // row tiles that are walked together, column by column
};

// Columns n .. n + 3 of row m: bias, activation, residual
__device__ __forceinline__ f32x4 behind(const NarrowArgs& a, f32x4 v, int64_t m, int n) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (a.bias) v[i] += (float)a.bias[n + i];
    if (a.act >= 0) v[i] = act_any(a.act - DS_ACT_UNARY, v[i]);
    if (a.res) v[i] += (float)a.res[m * a.N + n + i];
  }
  return v;
}

typedef int i32x4 __attribute__((ext_vector_type(4)));

// A buffer of `bytes` bytes: what lies past its end reads as zero
__device__ __forceinline__ i32x4 buffer_of(const void* p, uint32_t bytes) {
  const uint64_t at = (uint64_t)p;
  return i32x4{__builtin_amdgcn_readfirstlane((int)at), __builtin_amdgcn_readfirstlane((int)(at >> 32)), __builtin_amdgcn_readfirstlane((int)bytes),
               0x00020000};
}
// 16 bytes per lane to LDS bytes dst + 16 lane. Inline asm: hipcc waits for all of its own such loads before a transposed read.
__device__ __forceinline__ void dma16(i32x4 from, uint32_t lane_bytes, uint32_t dst) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds\n\ts_mov_b32 m0, %0"
               : "=&s"(keep)
               : "s"(dst), "v"(lane_bytes), "s"(from)
               : "memory");
}

// All of this wave's LDS accesses and all but its NEWER latest loads are done, then those of all waves.
template <int NEWER>
__device__ __forceinline__ void meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((NEWER & 15) | 7 << 4 | (NEWER >> 4) << 14);
  asm volatile("s_barrier" ::: "memory");
}

// One operand's R rows (or columns) of a step of 64: its way into LDS and out of it
// How an operand lies: its rows across the inner dimension, along it, or in operand order (blocks of 16 rows, of which 64 columns at a time are
// 2 KB: `preshuffle16` of ops/bf16_gemv.py)
enum : int { ACROSS = 0, ALONG = 1, ORDERED = 2 };

template <int LAY, int R>
struct Operand {
  static constexpr int BYTES = R * 128, PIECES = R / 32;  // LDS bytes a step, transfers of 1 KB a wave
  i32x4 from;
  uint32_t src[PIECES], step;  // per lane: bytes of step 0; bytes from a step to the next
  int dst;

  __device__ __forceinline__ void init(const bf16* p, uint32_t bytes, uint32_t ld, int r0, int lane, int wid) {
    from = buffer_of(p, bytes);
    step = LAY == ORDERED ? 2048 : LAY == ALONG ? 128 : 128 * ld;
    dst = wid * PIECES * 1024;
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int piece = wid * PIECES + i;
      if constexpr (LAY == ORDERED) {  // half a block as it lies: chunk 2 q + h of its row r at 64 h + 16 q + r
        src[i] = (uint32_t)((r0 >> 4) + (piece >> 1)) * 32 * ld + 1024 * (piece & 1) + 16 * lane;
      } else if constexpr (LAY == ALONG) {  // 8 rows of 8 chunks: chunk c of row r at c ^ (r / 2 % 8)
        const int r = 8 * piece + (lane >> 3);
        src[i] = (uint32_t)(r0 + r) * ld * 2 + 16 * ((lane & 7) ^ ((r >> 1) & 7));
      } else {  // R / 8 chunks of a step's 64 / PIECES / 4 rows each, those of row r swizzled by `turn`
        constexpr int CH = R / 8;
        const int r = (64 / CH) * piece + lane / CH, c = lane % CH;
        src[i] = (uint32_t)r * ld * 2 + 2 * r0 + 16 * (c ^ turn(r));
      }
    }
  }
  // A transposed read takes 64 bytes of eight rows in two goes: rows of 256 bytes, or pairs of rows of 128, that meet in a bank are apart
  static __device__ __forceinline__ int turn(int r) { return R >= 128 ? (r & 3) << 2 : R == 64 ? ((r >> 1) & 1) << 2 : 0; }
  __device__ __forceinline__ void piece(int i, int kq, uint32_t buf) const { dma16(from, src[i] + (uint32_t)kq * step, buf + dst + 1024 * i); }
  __device__ __forceinline__ void move(int kq, uint32_t buf) const {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) piece(i, kq, buf);
  }
  // Rows r0 .. + 31 (row: the lane's l32), inner columns of slice j of 16: 8 h .. + 7 where both operands lie along it (PLAIN), else
  // 4 h .. + 3 and 8 + 4 h .. + 3
  template <bool PLAIN>
  __device__ __forceinline__ bf16x8 read(const lds_char* buf, int j, int r0, int lane) const {
    const int l32 = lane & 31, h = lane >> 5;
    if constexpr (LAY == ORDERED) {
      static_assert(PLAIN, "beside rows along the inner dimension");
      const int r = r0 + l32;
      return *reinterpret_cast<const lds_bf16x8*>(buf + (r >> 4) * 2048 + h * 1024 + (j * 16 + (r & 15)) * 16);
    } else if constexpr (LAY == ALONG) {
      const int r = r0 + l32, sw = (r >> 1) & 7;
      if constexpr (PLAIN) return *reinterpret_cast<const lds_bf16x8*>(buf + r * 128 + 16 * ((2 * j + h) ^ sw));
      const bf16x4 lo = *reinterpret_cast<const lds_bf16x4*>(buf + r * 128 + 16 * ((2 * j) ^ sw) + 8 * h);
      const bf16x4 hi = *reinterpret_cast<const lds_bf16x4*>(buf + r * 128 + 16 * ((2 * j + 1) ^ sw) + 8 * h);
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    } else {
      const int gq = (lane >> 2) & 3, row = 16 * j + 4 * h + gq;
      const int c = (r0 / 8 + ((lane >> 4) & 1) * 2 + ((lane >> 1) & 1)) ^ turn(gq);
      const lds_char* at = buf + row * (2 * R) + 16 * c + 8 * (lane & 1);
      s16x8 v;
#ifdef __HIP_DEVICE_COMPILE__
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)at), hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 16 * R));
      v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#endif
      return __builtin_bit_cast(bf16x8, v);
    }
  }
};

__device__ __forceinline__ bf16x4 narrowed(f32x4 v) {
  bf16x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = (bf16)v[i];
  return o;
}

// AK, BK: how the operands lie. TM x TN: tile of C. U: steps of 64 a buffer holds.
template <int AK, int BK, int TM, int TN, int U>
__global__ void __launch_bounds__(256, TM == 128 ? 1 : 2) narrow_gemm_kernel(NarrowArgs a) {
  typedef Operand<AK, TM> A;
  typedef Operand<BK, TN> B;
  constexpr int STEP = A::BYTES + B::BYTES, BUF = STEP * U;
  constexpr int WM = TM > 32 ? 2 : 1, WN = TN > 32 ? 2 : 1, WK = 4 / (WM * WN), SLICES = 4 / WK;  // waves over rows, columns, slices of 16
  constexpr int MR = TM / 32 / WM, NR = TN / 32 / WN;                                            // pieces of 32 x 32 of a wave
  constexpr bool PLAIN = AK && BK;
  constexpr int NB = 4 * BUF <= 160 * 1024 ? 4 : 3;  // buffers
  __shared__ __attribute__((aligned(16))) char lds[NB * BUF];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wid % WM * 32 * MR, wn = wid / WM % WN * 32 * NR, wk = wid / (WM * WN);
  const int mt = (a.M + TM - 1) / TM, nt = (a.N + TN - 1) / TN, id = xcd_remap(blockIdx.x, gridDim.x);
  const int strip = id / (a.band * nt), spot = id - strip * a.band * nt, deep = min(a.band, mt - strip * a.band);
  const int m0 = (strip * a.band + spot % deep) * TM, n0 = spot / deep * TN;
  const int all = (a.K + 63) / 64, first = (int)((int64_t)all * blockIdx.y / a.parts);  // steps of 64: of K, and of this part
  const int steps = (int)((int64_t)all * (blockIdx.y + 1) / a.parts) - first, rounds = (steps + U - 1) / U;
  // Rows that lie a multiple of 8 KB apart meet in a memory channel at each step of K, in all workgroups at once: each begins elsewhere.
  // (Not where two of them share weights. 64 rows by [28672, 4096] 54.5 -> 47.9 us, [8192, 8192] 39.9 -> 32.7; 28 KB apart, 4096 by
  // 14336, 30.5 -> 33.7.)
  const int rot = TN == 128 && BK == ALONG && mt == 1 && a.ldb % 4096 == 0 ? id * 7 % steps : 0;
  A oa;
  B ob;
  oa.init(a.a, a.abytes, a.lda, m0, lane, wid);
  ob.init(a.b, a.bbytes, a.ldb, n0, lane, wid);
  auto buffer = [&](auto b_c) -> lds_char* { return (lds_char*)lds + decltype(b_c)::value % NB * BUF; };
  // where step i of this part stands in K; past the end the last one again
  auto place_in = [&](int i) {
    const int kq = min(i, steps - 1) + rot;
    return first + (kq >= steps ? kq - steps : kq);
  };
  // round r; past the end the last step again, into a place that nobody reads
  auto move = [&](int r, auto b_c) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kq = place_in(r * U + u);
      const uint32_t to = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)buffer(b_c) + STEP * u);
      oa.move(kq, to);
      ob.move(kq, to + A::BYTES);
    }
  };
  f32x16 acc[MR][NR];
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int n = 0; n < NR; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[m][n][i] = 0.f;
  auto products = [&](int r, auto b_c) {
    const lds_char* buf = buffer(b_c);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u && r * U + u >= steps) break;
      bf16x8 x[SLICES][MR], w[SLICES][NR];
#pragma unroll
      for (int j = 0; j < SLICES; ++j) {
#pragma unroll
        for (int n = 0; n < NR; ++n) w[j][n] = ob.template read<PLAIN>(buf + STEP * u + A::BYTES, wk * SLICES + j, wn + 32 * n, lane);
#pragma unroll
        for (int m = 0; m < MR; ++m) x[j][m] = oa.template read<PLAIN>(buf + STEP * u, wk * SLICES + j, wm + 32 * m, lane);
      }
#pragma unroll
      for (int j = 0; j < SLICES; ++j)
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
          for (int n = 0; n < NR; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[j][n], x[j][m], acc[m][n], 0, 0, 0);
    }
  };
  if (NB == 4 && rounds <= 3) {  // all at once
    move(0, Int<0>{});
    if (rounds > 1) move(1, Int<1>{});
    if (rounds > 2) move(2, Int<2>{});
    meet<0>();
    products(0, Int<0>{});
    if (rounds > 1) products(1, Int<1>{});
    if (rounds > 2) products(2, Int<2>{});
  } else {
    constexpr int PER = (A::PIECES + B::PIECES) * U;
    move(0, Int<0>{});
    move(1, Int<1>{});
    if constexpr (NB == 4) move(2, Int<2>{});
    if constexpr (TM == 128) {
      bf16x8 x[2][MR], w[2][NR];
      // a product at a time, with a read of the next quarter and a transfer of step r + NB - 1 before each
      auto read = [&](auto b_c, int j, int s, int i) {
        const lds_char* buf = buffer(b_c);
        if (i < NR) w[s][i] = ob.template read<PLAIN>(buf + A::BYTES, j, wn + 32 * i, lane);
        else if (i < NR + MR) x[s][i - NR] = oa.template read<PLAIN>(buf, j, wm + 32 * (i - NR), lane);
      };
      auto round = [&](int r, auto b_c) {
        using Next = Int<decltype(b_c)::value + 1>;
        const int kq = place_in(r + NB - 1);
        const uint32_t to = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)buffer(Int<decltype(b_c)::value + NB - 1>{}));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (q == 3) meet<(NB - 2) * PER>();
#pragma unroll
          for (int i = 0; i < MR * NR; ++i) {
            if (q < 3) read(b_c, q + 1, (q + 1) & 1, i);
            else read(Next{}, 0, 0, i);
            constexpr int SLOTS = 3 * MR * NR;
            const int slot = q * MR * NR + i;
#pragma unroll
            for (int p = 0; p < A::PIECES + B::PIECES; ++p)
              if (q < 3 && p * SLOTS / (A::PIECES + B::PIECES) == slot) {
                if (p < A::PIECES) oa.piece(p, kq, to);
                else ob.piece(p - A::PIECES, kq, to + A::BYTES);
              }
            __builtin_amdgcn_sched_barrier(0);
            const int m = i / NR, n = i % NR;
            acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[q & 1][n], x[q & 1][m], acc[m][n], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      };
      meet<(NB - 2) * PER>();
#pragma unroll
      for (int i = 0; i < MR + NR; ++i) read(Int<0>{}, 0, 0, i);
      int r = 0;
      for (; r + NB <= rounds; r += NB) {
        round(r, Int<0>{});
        round(r + 1, Int<1>{});
        round(r + 2, Int<2>{});
        if constexpr (NB == 4) round(r + 3, Int<3>{});
      }
      if (r < rounds) {
        round(r, Int<0>{});
        if (r + 1 < rounds) {
          round(r + 1, Int<1>{});
          if (NB == 4 && r + 2 < rounds) round(r + 2, Int<2>{});
        }
      }
    } else {
      auto round = [&](int r, auto b_c) {
        meet<2 * PER>();  // this round's operands have come, and nobody reads the buffer of the round before any more
        move(r + 3, Int<decltype(b_c)::value + 3>{});
        products(r, b_c);
      };
      for (int r = 0; r < rounds; r += 4) {
        round(r, Int<0>{});
        if (r + 1 >= rounds) break;
        round(r + 1, Int<1>{});
        if (r + 2 >= rounds) break;
        round(r + 2, Int<2>{});
        if (r + 3 >= rounds) break;
        round(r + 3, Int<3>{});
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the surplus transfers)
  }
  // ---- the waves' sums (lane: row l32 of a piece, columns 8 q + 4 h .. + 3) through LDS into runs of whole rows
  __syncthreads();
  const int l32 = lane & 31, h = lane >> 5;
  constexpr int ROW = TN * 4 + 16, PART = TM * ROW;  // bytes
  auto place = [&](int w, int m, int n) { return lds + w * PART + m * ROW + n * 4; };  // of row m, columns n .. of the wave group w
  static_assert(WK * PART <= NB * BUF, "room for the sums");
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int n = 0; n < NR; ++n)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(place(wk, wm + 32 * m + l32, wn + 32 * n + 8 * q + 4 * h)) =
            f32x4{acc[m][n][4 * q], acc[m][n][4 * q + 1], acc[m][n][4 * q + 2], acc[m][n][4 * q + 3]};
  __syncthreads();
  constexpr int PIECES = TM * TN / 8;  // of 8 columns
#pragma unroll
  for (int i = 0; i < (PIECES + 255) / 256; ++i) {
    const int p = 256 * i + tid, m = p / (TN / 8), n = p % (TN / 8) * 8;
    if (PIECES < 256 && p >= PIECES) continue;
    if (m0 + m >= a.M || n0 + n >= a.N) continue;
    f32x4 lo{0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll
    for (int w = 0; w < WK; ++w) {
      const f32x4* v = reinterpret_cast<const f32x4*>(place(w, m, n));
      lo = w ? lo + v[0] : v[0];
      hi = w ? hi + v[1] : v[1];
    }
    const int64_t at = (int64_t)(m0 + m) * a.N + n0 + n;
    if (a.part) {
      f32x4* out = a.part + ((int64_t)blockIdx.y * a.M * a.N + at) / 4;
      out[0] = lo;
      out[1] = hi;
    } else {
      if constexpr (BK == ORDERED) {
        lo = behind(a, lo, m0 + m, n0 + n);
        hi = behind(a, hi, m0 + m, n0 + n + 4);
      }
      *reinterpret_cast<bf16x8*>(a.c + at) = __builtin_shufflevector(narrowed(lo), narrowed(hi), 0, 1, 2, 3, 4, 5, 6, 7);
    }
  }
}

// The parts' sums, always in the same order
template <bool BEHIND>
__global__ void __launch_bounds__(256) narrow_sum_kernel(NarrowArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, n4 = (int64_t)a.M * a.N / 4;
  if (i >= n4) return;
  f32x4 v = a.part[i];
  for (int p = 1; p < a.parts; ++p) v += a.part[p * n4 + i];
  if constexpr (BEHIND) v = behind(a, v, 4 * i / a.N, (int)(4 * i % a.N));
  *reinterpret_cast<bf16x4*>(a.c + 4 * i) = narrowed(v);
}

// Each XCD, with an L2 of its own, has an eighth of the tiles in a row: as nearly a square of them as bands allow (dW of 1000 / 8000 tokens, us, with
// all row tiles first and in bands: [2048, 1024] 10.5 / 88 and 9.1 / 57, [2048, 512] 7.0 / 49 and 6.1 / 28.5, [11264, 2048] 77 / 439 and 68 / 400)
int band_of(int64_t mt, int64_t nt) {
  int64_t band = 1;
  while (band < mt && 4 * band * band <= mt * nt / 8) band *= 2;
  return (int)std::min(band, mt);
}

thread_local int g_tile = 0, g_parts = 0;  // (a thread's own: another's products go by the rules, and keep to the scratch they asked for)

struct Cut {
  int tm, tn, parts;  // tile, parts of K
};

// Rounds that the chip makes of tiles of 128 x 128, or 128 x 256, which take 1.8 times as long (dW of 3000 tokens, us: 256 of the first 25, of the
// second 44), over longer K 1.6 times (5 rounds and 3, the medians of 114 products of K from 1024 on: 0.96; 9 and 5 0.92; of K below 1.05): `wide` where those
// are the faster ones
struct Rounds {
  int64_t tiles;  // of 128 x 128
  bool wide;
  int full;       // percent of the chosen one's rounds that is work
  int64_t count;  // ... and their number
  Rounds(int64_t M, int64_t N, int64_t K) {
    tiles = (M + 127) / 128 * ((N + 127) / 128);
    const int64_t half = (M + 127) / 128 * ((N + 255) / 256), a = (tiles + 255) / 256, b = (half + 255) / 256;
    wide = (K >= 1024 ? 8 : 9) * b < 5 * a;
    count = wide ? b : a;
    full = (int)(100 * (wide ? half : tiles) / (256 * count));
  }
};
// us, on one machine, of 32-row tiles / 64 / 128, whole or in parts of K (x2, x4).
// Both operands along K (y): 32 x 32 up to two tiles a CU (128 tokens by [3072, 1024] 6.4 / 6.4, [4096, 2048] 9.0 / 9.4, [5632, 1024] 8.6 / 6.7), 128 x
// 128 from 126 of them on (512 by [5632, 1024] 13.5 with 64, 10.7; 768 by [3072, 1024], 144, 13.6, 10.4; 1000 by [2048, 2048], 128, 15.6, 15.4; 700, 96,
// 15.1, 15.2). Parts of 2560 or more of K: a sum costs 2 us and its traffic (64 by [2048, 5632] 12.6, x2 10.5; [1024, 2816] 7.7, 7.7).
// 128 x 256 by `Rounds` (us with 128, 256: y 500 by [11264, 2048] 33.4, 28.0; dX 700 by [2048, 5632] 33.0, 27.5; dW 3000 by [11264, 2048] 145, 124; in one
// round anyhow, y 1000 by [4096, 4096], 34.3, 44.2).
// From K = 4096 on weights come from memory and a CU's share of the operands bounds: 128 x 128 tiles, in parts of 768 or more, where those make
// 172 to 256 workgroups (128 by [4096, 14336] 63.9 with 64x1, 34.8 with 128x8; by [6144, 4096] 22.2, 128x5 20.7; 238 by [4096, 5120], weights from memory,
// 31.0 with 64x1, 128x4 25.4; but 454 by [2048, 4096] 19.0, 128x4 20.8), else 64 x 64 in parts (128 by [2048, 5632] 18.2 with 32x2, 13.9; by [1024, 8192] 18.4,
// 13.1; 50 by [3072, 5632], from memory, 18.7, 64x4 13.9). Up to 64 rows over shorter K fill half of 128 x 128 (52 by [16384, 2048] 23.9, 64x1 18.9; dX, 57 by
// [3072, 14336] 30.9, 25.4).
// One across (dX): those rows come in runs of 64 columns, never 32 (half a cache line). 64 x 64 from 160 tiles on, of long K from 64
// (256 tokens by [5632, 1024] 32x2 13.0, 64x4 11.8; 512 17.5, 64x2 15.8; by [3072, 1024] 9.5, 10.5), 128 x 128 from 88 (1400 by [8000, 1024], 88, 57 with 64,
// 49, x2 35; 600 by [1024, 2816], 110, 10.0, 10.5; 300 by [2048, 5632], 132, 19.6, 16.3). Parts of 768 up to a workgroup a CU, of 128 x 128 2560
// (128 by [3072, 1024] 10.6, x2 9.4, x4 8.9; by [1024, 1024] 5.3, 6.4, 6.9). Over long K 128 x 128 in parts as above, from 43 tiles on (weights from memory,
// 128 by [11264, 11008] 118 with 64x1, 128x2 69, library 104; 250 by [5632, 4096] 38.1, 128x4 27.5, 43; by [4096, 4096], a round of 64 x 64, 25.8, 25.8, in cache
// 18.3, 22.5); both forms from 80 on that 64 x 64 would not do in a round (768 by [3072, 2048] 25.3, 128x2 24.1, by [2048, 2048] 18.0, 19.5; dW, 2705 by [376,
// 3584] 34.5, 23.4, library 32.2; not 128 of them, 2299 by [2048, 1024] 18.0, 24.0).
// Both across (dW): 64 x 64, 128 x 128 from 140 of them on (500 / 2000 / 8000 by [1536, 1536], 144, 9.4 / 21.8 / 78, 8.0 / 16.7 / 49; 500 / 2000 by [1024, 2048],
// 128, 7.3 / 15.9, 7.9 / 15.8).
Cut cut_of(int64_t M, int64_t N, int64_t K, bool a_along, bool b_along) {
  auto tiles = [&](int t, int u) { return ((M + t - 1) / t) * ((N + u - 1) / u); };
  const bool along = a_along && b_along, across = !a_along && !b_along;
  int tm = 32, tn = along ? 32 : 64;
  const Rounds rounds(M, N, K);
  const int64_t big = rounds.tiles, mid = tiles(64, 64);
  if (big >= (along ? 126 : across ? 140 : 88) && !(K < 4096 && M <= 64 && mid <= 256)) {
    tm = 128;
    tn = rounds.wide ? 256 : 128;
  } else if (along ? tiles(32, 32) > 512 : across || mid >= (K >= 4096 ? 64 : 160)) tm = tn = 64;
  int64_t parts = 0;
  if (along && K >= 4096) {
    const int64_t cut = std::min<int64_t>(256 / std::max<int64_t>(big, 1), 8);
    if (cut >= 2 && cut * big >= 172 && K / cut >= 768 && (K >= 5120 || mid <= 224 || mid > 256)) {
      tm = tn = 128;
      parts = cut;
    } else if (mid <= 128 && (mid >= 64 || (mid >= 32 && K >= 8192) || (mid > 32 && K >= 4608))) {
      tm = tn = 64;
      parts = std::min<int64_t>(std::min<int64_t>(256 / mid, K / (mid < 64 ? 768 : 1024)), 8);
    }
  } else if (!along && ((!across && big >= 43 && big <= 128 && K >= (mid > 256 ? 4096 : 5120)) ||
                        (big >= 80 && big <= 120 && mid > 256 && K >= (across ? 2048 : 3072)))) {
    tm = tn = 128;
    parts = std::min<int64_t>(std::min<int64_t>(256 / big, K / 1024), 8);
  }
  if (g_tile) {
    tm = g_tile;
    tn = g_tile == 32 && !along ? 64 : g_tile;
    if (g_tile == 256) tm = 128;
  }
  if (parts <= 0 || g_tile) parts = std::min<int64_t>(std::min<int64_t>((along && tm < 128 ? 512 : 256) / tiles(tm, tn), K / (along || tm == 128 ? 2560 : 768)), 8);
  if (g_parts) parts = std::min<int64_t>(g_parts, (K + 63) / 64);
  return {tm, tn, (int)std::max<int64_t>(parts, 1)};
}

}  // namespace

// Forces tiles of 32, 64 or 128 rows, or 128 x 256 (256), and parts of K, for the calling thread's products; 0: by the rule above.
extern "C" void ds_narrow_gemm_tune(int tile, int parts) { g_tile = tile; g_parts = parts; }

// Whether the kernel takes the product: whole 16-byte pieces of rows, whole steps of 64 along an operand's rows, offsets of 32 bits
extern "C" int ds_narrow_gemm_ok(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_along, int b_along) {
  if (M <= 0 || N <= 0 || K <= 0 || M > INT32_MAX / 64 || N > INT32_MAX / 64 || K > INT32_MAX / 64) return 0;
  if (N % 8 || lda % 8 || ldb % 8 || ((a_along || b_along) && K % 64) || (!a_along && M % 8)) return 0;
  if (lda < (a_along ? K : M) || ldb < (b_along ? K : N)) return 0;
  const int64_t ar = a_along ? M : K, br = b_along ? N : K;
  return (ar + 128) * lda * 2 < UINT32_MAX && (br + 256) * ldb * 2 < UINT32_MAX && ((M + 31) / 32) * ((N + 31) / 32) <= INT32_MAX;
}

// Whether the kernel is as fast as the library's, for each product of a linear layer of `tokens` rows by a weight [out, in]; us here (there).
// A cost model was not found that orders the library's side, which jumps with its own choice of tiles. What the lines go by is stated with each:
// whole rounds of the chip (`Rounds`), which products of its size the library is bad at, and rows that meet in memory channels. The wide tiles are asked first
// (`wide` below). On layers at random, none of which the lines were drawn by, with weights (for dW the input) from memory 613 / 508 / 812 products y / dX / dW of
// 1200 layers go here and take 0.75 / 0.69 / 0.65 of the library's time in the mean, 1859 of them faster by more than 4 %, 15 slower by as much, at worst 35 %;
// out of the caches 673 of 400 layers 0.77 / 0.68 / 0.60, 662 faster, none slower (profiles/narrow_products_at_random.csv, without what the wide tiles take).
namespace {

// y: a tile's operands come as the library's do; what is gained is its launch, and tiles that fill the chip.
bool y_pays(int64_t tokens, int64_t out, int64_t in, const Rounds& rounds) {
  const int64_t mid = (tokens + 63) / 64 * ((out + 63) / 64);
  const bool one = rounds.count == 1;
  // one round of 128 x 128 that is 69 % full (200 / 256 by [11264, 2048] 16.9 / 17.3 (22.4 / 23.7), 1000 by [4096, 4096] 34 (38), 4096 by [1024, 2816]
  // 26.2 (28.3); 175 by [16384, 1024] 14.1 (13.2)); of few tokens over weights up to 2^26 (160 by [16384, 8192] 73 (65))
  if (tokens >= 192 && one && !rounds.wide && rounds.tiles >= 176 && (tokens > 512 || out * in <= (1 << 26))) return true;
  // one round of 128 x 256 over short K (500 by [11264, 2048] 27.4 (31.1), 1400 by [4096, 2048] 27.8 (30.8); 320 by [16384, 2048] 28 (26), 3000 by
  // [2048, 2048] 28.7 (28.3))
  if (tokens > 384 && one && rounds.wide) return rounds.full >= 62 && tokens <= 2048 && in <= 2048;
  // more than a round of 64 x 64 (700 by [2048, 2048] 15.2 (13.8); 188 by [6544, 2176] 22.4 (17.7), 250 by [5632, 2048] 20.6 (16.4))
  if (in >= 2048 && (tokens > 256 ? mid > 256 : in < 4096 && mid > 300)) return false;
  // several rounds that are full, over short K (1400 / 2000 by [8000, 1024] 33.2 / 40.6 (34.9 / 42.2))
  if (tokens > 512 && tokens <= 2048 && in <= 1024 && out <= 8192 && rounds.full >= 90) return true;
  if (tokens > 1024) return tokens <= 2048 && out <= 1024 && in <= 1024;  // (1400 by [1024, 1024] 8.9 (10.8))
  // long K in parts (128 by [4096, 14336] 36 (75), [6144, 4096] 21 (25), [8192, 8192] 38 (50), 64 33 (34); 256 by [5120, 13824] 58 (120); 64 by [12288, 4096]
  // in two 28.7 (26.7))
  if (in >= 4096 && tokens <= 256 && cut_of(tokens, out, in, true, true).parts >= (tokens <= 128 ? 3 : 2)) return true;
  // rows 8 KB apart, which the library reads in step, in a round that is 78 % full (64 / 128 by [28672, 4096] 47 / 53 (57 / 59); by [22016, 4096], 172
  // tiles, 44 / 53 (47 / 49))
  if (in % 4096 == 0 && tokens <= 128 && rounds.tiles >= 200 && rounds.tiles <= 256) return true;
  // else by the work: 2^31 products, over weights up to 2^24 2^32 (512 by [8000, 1024] 12.6 (17.2), [5632, 1024] 10.7 (14.1); 128 by [11264, 2048] 16.1 (16.5))
  return tokens * out <= (1LL << (out * in <= (1 << 24) ? 32 : 31)) / in;
}

// dX: the library is slow over a weight read across its rows, up to 9 2^20 results.
bool dx_pays(int64_t tokens, int64_t out, int64_t in, const Rounds& rounds) {
  if (tokens * in > (9 << 20)) return false;
  // several rounds: 88 % full (2000 by [2048, 5632] 53.5 (55.2); 1032 by [5632, 8192], 75 %, 120 (96); 607 by [5632, 14336], 72 %, 138 (99)), or the last
  // one of a few tiles (700 by [2048, 11008], 516, 48.5 (56.7))
  if (rounds.count > 1) return rounds.full >= 88 || (tokens <= 1024 && rounds.tiles % 256 <= 16);
  // 500 by [2048, 2048] 10.5 (15.1), [11264, 2048] 42 (63), [4096, 4096] 27.5 (34.6); 1024 by [11264, 2048] 54 (79), [12288, 4096] 94 (111), but 614 by [32000,
  // 8192] in wide tiles 406 (305)
  if (tokens <= 1024) return !rounds.wide || out <= 16384;
  // one: of 88 tiles (1400 / 2000 by [3072, 2048] 23.7 / 29.5 (28.4 / 32.6), [8000, 1024] 35 / 44 (72 / 64)), of many tokens 62 % full (3000 / 4096 by
  // [2048, 2048] 29.6 / 35.5 (30.2 / 36.4), 3000 by [11264, 2048] 125 (130), [32000, 2048] 393 (344))
  return tokens <= 2048 ? rounds.tiles >= 88 : rounds.full >= 62 && out <= 16384;
}

// dW: both operands lie across the inner dimension, as the library likes least.
bool dw_pays(int64_t tokens, int64_t out, int64_t in, const Rounds& rounds) {
  // From 8192 tokens on the layer makes copies along them for the library, where the wide tiles do not pay. Rows that meet in memory channels: 32 KB apart ([16384, 2048] 320 45 (35)), or
  // 8 and 16 KB ([12288, 8192] 528 158 (149))
  if (tokens > 8192 || out % 16384 == 0 || (out % 4096 == 0 && in % 8192 == 0 && out * in > (1 << 25))) return false;
  // up to three rounds of 128 x 128 (256 / 1024 / 4096 by [2048, 2048] 7.8 / 14.5 / 35.7 (10 / 17.2 / 45.5), [2048, 5632] 17 / 34 / 93 (24 / 41 / 96), 8000 by
  // [1024, 1024] 30 (56)); more over long dimensions ([4096, 4096] 512 / 1024 / 2048 30 / 42 / 67 (26 / 40 / 67), 6000 by [12288, 4096] 480 (513))
  if (rounds.tiles <= 3 * 256 || tokens >= 1280) return true;
  // six rounds, three of 128 x 256 ([11264, 2048] 768 48 (62))
  if (tokens >= 704 && rounds.tiles >= 5 * 256 && rounds.tiles <= 6 * 256) return true;
  // token counts that are no whole 32, which the library pays for (100 by [22016, 4096] 64 (98), [4096, 11008] 37 (52), [11264, 2048] 22 (26), [32000, 2048] 49
  // (53); 500 41 (47) by [6144, 4096], 98 (99) by [32000, 2048]; 333 by [4096, 4096], four rounds, 32 (24), 900 by [27648, 5120] 312 (292))
  return tokens % 32 && (tokens <= 256 || (rounds.tiles <= 6000 && (tokens >= 500 || (rounds.tiles > 4 * 256 && rounds.tiles < 3000))));
}

}  // namespace

// Products of many tokens, in tiles of 256 columns (wide_gemm.hip)
extern "C" int ds_wide_gemm_pays(int64_t, int64_t, int64_t, int, int);
extern "C" int64_t ds_wide_gemm_scratch(int64_t, int64_t, int64_t);
extern "C" int ds_wide_gemm(const void*, const void*, void*, int64_t, int64_t, int64_t, int64_t, int64_t, int, int, void*, hipStream_t);
static bool wide(int64_t M, int64_t N, int64_t K, int a_along, int b_along) { return !g_tile && !g_parts && ds_wide_gemm_pays(M, N, K, a_along, b_along); }

// Whether these tiles are faster than the library's product
extern "C" int ds_narrow_tiles_pay(int64_t M, int64_t N, int64_t K, int a_along, int b_along) {
  const Rounds rounds(M, N, K);
  if (!a_along) return dw_pays(K, M, N, rounds);
  return b_along ? y_pays(M, N, K, rounds) : dx_pays(M, K, N, rounds);
}
// C [M, N] over K, as `ds_narrow_gemm` takes it
extern "C" int ds_narrow_gemm_pays(int64_t M, int64_t N, int64_t K, int a_along, int b_along) {
  return wide(M, N, K, a_along, b_along) || ds_narrow_tiles_pay(M, N, K, a_along, b_along);
}

// Bytes of scratch memory that the product wants (0: none)
extern "C" int64_t ds_narrow_gemm_scratch(int64_t M, int64_t N, int64_t K, int a_along, int b_along) {
  if (wide(M, N, K, a_along, b_along)) return ds_wide_gemm_scratch(M, N, K);
  const Cut c = cut_of(M, N, K, a_along, b_along);
  return c.parts > 1 ? c.parts * M * N * 4 : 0;
}

// C [M, N] = A B^T over K. a_along: A is [M, K] with rows lda apart, else [K, M]; b_along: B is [N, K], else [K, N]. part:
// ds_narrow_gemm_scratch bytes.
extern "C" int ds_narrow_gemm(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_along,
                              int b_along, void* part, hipStream_t st) {
  if (!ds_narrow_gemm_ok(M, N, K, lda, ldb, a_along, b_along)) return (int)hipErrorInvalidValue;
  if (wide(M, N, K, a_along, b_along)) return ds_wide_gemm(A, B, C, M, N, K, lda, ldb, a_along, b_along, part, st);
  const Cut cut = cut_of(M, N, K, a_along, b_along);
  if (cut.parts == 1) part = nullptr;
  else if (!part) return (int)hipErrorInvalidValue;
  const int64_t ar = a_along ? M : K, ac = a_along ? K : M, br = b_along ? N : K, bc = b_along ? K : N;
  const NarrowArgs a{(const bf16*)A, (const bf16*)B, (bf16*)C, (int)M, (int)N, (int)K, (uint32_t)lda, (uint32_t)ldb,
                     (uint32_t)(((ar - 1) * lda + ac) * 2), (uint32_t)(((br - 1) * ldb + bc) * 2), cut.parts, (f32x4*)part,
                     nullptr, nullptr, -1, band_of((M + cut.tm - 1) / cut.tm, (N + cut.tn - 1) / cut.tn)};
  const dim3 grid((unsigned)(((M + cut.tm - 1) / cut.tm) * ((N + cut.tn - 1) / cut.tn)), cut.parts);
#define GO(AK, BK, TM, TN, U) hipLaunchKernelGGL((narrow_gemm_kernel<AK, BK, TM, TN, U>), grid, dim3(256), 0, st, a)
  if (cut.tn == 256) {
    if (a_along && b_along) GO(ALONG, ALONG, 128, 256, 1);
    else if (a_along) GO(ALONG, ACROSS, 128, 256, 1);
    else if (b_along) GO(ACROSS, ALONG, 128, 256, 1);
    else GO(ACROSS, ACROSS, 128, 256, 1);
  } else if (cut.tm == 128) {
    if (a_along && b_along) GO(ALONG, ALONG, 128, 128, 1);
    else if (a_along) GO(ALONG, ACROSS, 128, 128, 1);
    else if (b_along) GO(ACROSS, ALONG, 128, 128, 1);
    else GO(ACROSS, ACROSS, 128, 128, 1);
  } else if (cut.tm == 64) {
    if (a_along && b_along) GO(ALONG, ALONG, 64, 64, 1);
    else if (a_along) GO(ALONG, ACROSS, 64, 64, 1);
    else if (b_along) GO(ACROSS, ALONG, 64, 64, 1);
    else GO(ACROSS, ACROSS, 64, 64, 1);
  } else {
    if (a_along && b_along) GO(ALONG, ALONG, 32, 32, 2);
    else if (a_along) GO(ALONG, ACROSS, 32, 64, 1);
    else if (b_along) GO(ACROSS, ALONG, 32, 64, 1);
    else GO(ACROSS, ACROSS, 32, 64, 1);
  }
#undef GO
  if (part) hipLaunchKernelGGL(narrow_sum_kernel<false>, dim3((unsigned)((M * N / 4 + 255) / 256)), dim3(256), 0, st, a);
  DS_CHECK_LAUNCH();
  return 0;
}

namespace {
// Decode batches of 33 to 48 rows by weights in operand order. Against ds_decode_gemm's kernels (eight waves that load what they multiply) the
// transfers run three steps ahead without registers, a workgroup's tile has 64 weight rows (there 32, or 64 with a CU to itself) and
// the parts' sums are as many rows as there are. What a CU reads bounds it, so K goes in parts up to a workgroup a CU, in tiles of 64 x 64 over 64 of
// them and more, over 33 from K = 4608 on and over 22 from 6144 on (33 rows, us as 32 x 32 in parts up to a workgroup a CU and so: [2304, 7168] 16.6, 12.9,
// [2112, 4608] 11.9, 10.7, [1536, 14336] 19.5, 15.7, [1344, 14336] with 21 tiles 15.6, 15.3). Beyond 128 tiles, 128 x 128 in parts where a round holds three
// (33 rows by [9216, 7168] whole as 64 x 64 34.6, so 29.8; [9216, 4096] 21.8, 20.5; [9216, 3072] 16.8, 17.2) and of long K, else 64 x 64 whole; few or
// short ones 32 x 32. us before and now, weights from memory, 48 rows: [1024, 4096] 10.2 / 8.4, [2048, 2048] 9.7 / 7.2, [4096, 2048] 10.2 / 7.6, [4096, 4096] 14.5 /
// 12.3, [5120, 5120] 23.0 / 15.9, [2048, 5632] 13.0 / 11.6, [4096, 14336] 28.9 / 26.8, [10240, 8192] 39.8 / 37.9, [16384, 4096] 28.5 / 27.5. Of 2336 products at
// random (33 to 48 rows, up to 20800 weight rows, K of 512 to 15360; profiles/decode_products_at_random.csv) 2166 are faster by more than 4 %, 2 slower by
// as much (1.07 and 1.05 times as long); 0.84 of the time in the mean.
Cut ordered_cut(int64_t M, int64_t N, int64_t K) {
  const int64_t mid = (N + 63) / 64, low = (M + 31) / 32 * ((N + 31) / 32), big = (N + 127) / 128;
  auto parts = [&](int64_t tiles, int64_t least) { return (int)std::max<int64_t>(std::min<int64_t>(std::min<int64_t>(256 / tiles, K / least), 8), 1); };
  Cut c = {32, 32, 1};
  if (mid > 128) c = K >= 8192 || (K >= 3584 && big <= 85) ? Cut{128, 128, parts(big, 1024)} : Cut{64, 64, 1};
  else if (mid >= 64 && K >= 3072) c = Cut{64, 64, parts(mid, 1024)};
  else if ((mid > 32 && K >= 4608) || (mid > 21 && K >= 6144)) c = Cut{64, 64, parts(mid, 768)};
  else if (K >= 3072) c = Cut{32, 32, parts(low, 1024)};
  if (g_tile) c.tm = c.tn = std::min(g_tile, 128);
  if (g_parts) c.parts = (int)std::min<int64_t>(g_parts, K / 64);
  return c;
}
}  // namespace

// Whether ds_narrow_ordered takes x [M, K] by w [N, K] in operand order, and is the faster way, us here (with the decode kernels). Weights from memory.
extern "C" int ds_narrow_ordered_ok(int64_t M, int64_t N, int64_t K) {
  // (beyond, the weights' read is what counts: 48 rows by [16384, 8192] 55 (49), [32000, 4096] 52.5 (51))
  if (M > 48 || N <= 0 || N > 16384 || N % 8 || K <= 0 || K % 64 || N * K > (3 << 25)) return 0;
  const int64_t mid = (N + 63) / 64, big = (N + 127) / 128, blocks = (N + 15) / 16;  // tiles of 64 and 128 columns; blocks as the decode kernels take them
  if (M > 32) {
    if (mid <= 64) return 1;       // a part, or a few, of a round of tiles
    if (K < 3072) return 0;        // short K over more of them: the decode kernels' X is small (33 by [8192, 2048] 11.3 (10.4))
    // Nearly a round in two short parts, whose sums are a launch, or a round and more of whole tiles: not for 33 to 40 rows (33 by [8192, 4096] 18.2
    // (16.3), [11920, 7616] 41.6 (39.3), [13136, 4992] 29.7 (28.2))
    return M > 40 || !((mid > 96 && mid <= 128 && K <= 4096) || (big > 85 && K < 8192));
  }
  // Up to a third over one round of single blocks, which the decode kernels fill with two a workgroup (24 / 32 by [5120, 5120] 14.6 / 15.1 (16.6 / 18.1); 20 by [5336, 4096] 13.6 (12.7)). Small
  // products stay there: 24 by [2048, 2048] 7.4 (6.8), [1024, 1024] 5.5 (5.0), 32 rows 7.7 (7.7), 5.7 (5.5)
  return M > (K >= 5120 ? 16 : 24) && blocks > 256 && blocks <= 340 && K >= 4096 && K < 8192;
}

extern "C" int64_t ds_narrow_ordered_scratch(int64_t M, int64_t N, int64_t K) {
  const Cut c = ordered_cut(M, N, K);
  return c.parts > 1 ? c.parts * M * N * 4 : 0;
}

// y [M, N] = act(x w^T + bias) + res, rows of x K apart; part: ds_narrow_ordered_scratch bytes
extern "C" int ds_narrow_ordered(const void* X, const void* W, const void* bias, const void* res, void* Y, int64_t M, int64_t N, int64_t K, int act,
                                 void* part, hipStream_t st) {
  if (!ds_narrow_ordered_ok(M, N, K)) return (int)hipErrorInvalidValue;
  const Cut cut = ordered_cut(M, N, K);
  if (cut.parts == 1) part = nullptr;
  else if (!part) return (int)hipErrorInvalidValue;
  const NarrowArgs a{(const bf16*)X, (const bf16*)W, (bf16*)Y, (int)M, (int)N, (int)K, (uint32_t)K, (uint32_t)K, (uint32_t)(M * K * 2),
                     (uint32_t)((N + 15) / 16 * 16 * K * 2), cut.parts, (f32x4*)part, (const bf16*)bias, (const bf16*)res, act, (int)((M + cut.tm - 1) / cut.tm)};
  const dim3 grid((unsigned)(((M + cut.tm - 1) / cut.tm) * ((N + cut.tn - 1) / cut.tn)), cut.parts);
#define GO(TM, U) hipLaunchKernelGGL((narrow_gemm_kernel<ALONG, ORDERED, TM, TM, U>), grid, dim3(256), 0, st, a)
  if (cut.tm == 128) GO(128, 1);
  else if (cut.tm == 64) GO(64, 1);
  else GO(32, 2);
#undef GO
  if (part) hipLaunchKernelGGL(narrow_sum_kernel<true>, dim3((unsigned)((M * N / 4 + 255) / 256)), dim3(256), 0, st, a);
  DS_CHECK_LAUNCH();
  return 0;
}
