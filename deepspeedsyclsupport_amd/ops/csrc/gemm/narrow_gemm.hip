// bf16 products around a short batch of tokens (training steps and prompts of a few hundred): y = X W^T, dX = dY W and dW = dY^T X,
// each over the operands as they lie in memory, sums in fp32, one rounding at the end.
//
// What bounds them is latency and the count of workgroups, not the matrix cores: 128 tokens of a 1024-wide layer make 32 tiles of
// 64 x 64. Hence
//  * tiles of 64 x 64 (four waves of 32 x 32) or, where those are too few, of 32 rows by 32 or 64 (the waves share each step's inner
//    dimension and meet in LDS at the end, always in the same order), and K in parts with a second launch for their sums;
//  * both operands come by DMA into four LDS buffers, three steps ahead; one barrier a step, whose wait counts what may still be on its
//    way (buffers are arrays apart, accesses buffer instructions: see moe/expert_gemm.hip);
//  * an operand whose rows run along the inner dimension is stored row by row, 128 bytes a step; one whose rows run across it (W in dX, both in
//    dW) as it lies, and read transposed (ds_read_b64_tr_b16). Chunks are swizzled by the source address, against bank conflicts;
//  * what lies past the end of a buffer reads as zero: ragged tokens need no other treatment, along the inner dimension neither.
// Besides, the library's call takes the host 18 to 23 us, this one 5 to 7: a training step of 128 tokens has 27 of them and waits for the host.
// Measured, us (the library's kernel): 128 tokens, layers [3072, 1024], [1024, 1024], [5632, 1024], [1024, 2816], head [8000, 1024]: y 6.4
// (9.5), 4.8 (8.3), 7.1 (9.7), 7.8 (7.9), 7.3 (10.1); dX 10.8 (13.4), 8.1 (11.0), 13.4 (20.9), 9.8 (11.3), 15.3 (30); dW 6.3 (7.1), 3.3 (5.3),
// 9.0 (9.3), 5.7 (7.1), 11.6 (10.1).
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
};

// 16 bytes per lane to LDS bytes dst + 16 lane. (The host's pass does not know the size.)
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t from, uint32_t lane_bytes, lds_char* dst) {
#ifdef __HIP_DEVICE_COMPILE__
  __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (lds_void*)dst, 16, lane_bytes, 0, 0, 0);
#endif
}

// All of this wave's LDS accesses and all but its NEWER latest loads are done, then those of all waves.
template <int NEWER>
__device__ __forceinline__ void meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((NEWER & 15) | 7 << 4 | (NEWER >> 4) << 14);
  asm volatile("s_barrier" ::: "memory");
}

// One operand's R rows (or columns) of a step of 64: its way into LDS and out of it
template <bool ALONG, int R>
struct Operand {
  static constexpr int BYTES = R * 128, PIECES = R / 32;  // LDS bytes a step, transfers of 1 KB a wave
  __amdgpu_buffer_rsrc_t from;
  uint32_t src[PIECES], step;  // per lane: bytes of step 0; bytes from a step to the next
  int dst;

  __device__ __forceinline__ void init(const bf16* p, uint32_t bytes, uint32_t ld, int r0, int lane, int wid) {
    from = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(p), 0, (int)bytes, 0x00020000);
    step = ALONG ? 128 : 128 * ld;
    dst = wid * PIECES * 1024;
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int piece = wid * PIECES + i;
      if constexpr (ALONG) {  // 8 rows of 8 chunks: chunk c of row r at c ^ (r / 2 % 8)
        const int r = 8 * piece + (lane >> 3);
        src[i] = (uint32_t)(r0 + r) * ld * 2 + 16 * ((lane & 7) ^ ((r >> 1) & 7));
      } else {  // R / 8 chunks of a step's 64 / PIECES / 4 rows each; of 64 columns chunk c of row r at c ^ (4 (r / 2 % 2))
        constexpr int CH = R / 8;
        const int r = (64 / CH) * piece + lane / CH, c = lane % CH;
        src[i] = (uint32_t)r * ld * 2 + 2 * r0 + 16 * (CH == 8 ? c ^ (((r >> 1) & 1) << 2) : c);
      }
    }
  }
  __device__ __forceinline__ void move(int kq, lds_char* buf) const {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) dma16(from, src[i] + (uint32_t)kq * step, buf + dst + 1024 * i);
  }
  // Rows r0 .. + 31 (row: the lane's l32), inner columns of slice j of 16: 8 h .. + 7 where both operands lie along it (PLAIN), else
  // 4 h .. + 3 and 8 + 4 h .. + 3
  template <bool PLAIN>
  __device__ __forceinline__ bf16x8 read(const lds_char* buf, int j, int r0, int lane) const {
    const int l32 = lane & 31, h = lane >> 5;
    if constexpr (ALONG) {
      const int r = r0 + l32, sw = (r >> 1) & 7;
      if constexpr (PLAIN) return *reinterpret_cast<const lds_bf16x8*>(buf + r * 128 + 16 * ((2 * j + h) ^ sw));
      const bf16x4 lo = *reinterpret_cast<const lds_bf16x4*>(buf + r * 128 + 16 * ((2 * j) ^ sw) + 8 * h);
      const bf16x4 hi = *reinterpret_cast<const lds_bf16x4*>(buf + r * 128 + 16 * ((2 * j + 1) ^ sw) + 8 * h);
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    } else {
      const int gq = (lane >> 2) & 3, row = 16 * j + 4 * h + gq;
      int c = r0 / 8 + ((lane >> 4) & 1) * 2 + ((lane >> 1) & 1);
      if constexpr (R == 64) c ^= ((gq >> 1) & 1) << 2;
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

// AK, BK: the operand's rows run along the inner dimension. TM x TN: tile of C. U: steps of 64 a buffer holds.
template <bool AK, bool BK, int TM, int TN, int U>
__global__ void __launch_bounds__(256, 2) narrow_gemm_kernel(NarrowArgs a) {
  typedef Operand<AK, TM> A;
  typedef Operand<BK, TN> B;
  constexpr int STEP = A::BYTES + B::BYTES, BUF = STEP * U;
  constexpr int WM = TM / 32, WN = TN / 32, WK = 4 / (WM * WN), SLICES = 4 / WK;  // waves over rows, columns, slices of 16 of a step
  constexpr bool PLAIN = AK && BK;
  __shared__ __attribute__((aligned(16))) char b0[BUF], b1[BUF], b2[BUF], b3[BUF];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wid % WM * 32, wn = wid / WM % WN * 32, wk = wid / (WM * WN);
  const int mt = (a.M + TM - 1) / TM, id = xcd_remap(blockIdx.x, gridDim.x), m0 = id % mt * TM, n0 = id / mt * TN;
  const int all = (a.K + 63) / 64, first = (int)((int64_t)all * blockIdx.y / a.parts);  // steps of 64: of K, and of this part
  const int steps = (int)((int64_t)all * (blockIdx.y + 1) / a.parts) - first, rounds = (steps + U - 1) / U;
  A oa;
  B ob;
  oa.init(a.a, a.abytes, a.lda, m0, lane, wid);
  ob.init(a.b, a.bbytes, a.ldb, n0, lane, wid);
  auto buffer = [&](auto b_c) -> lds_char* {
    constexpr int b = decltype(b_c)::value & 3;
    if constexpr (b == 0) return (lds_char*)b0;
    else if constexpr (b == 1) return (lds_char*)b1;
    else if constexpr (b == 2) return (lds_char*)b2;
    else return (lds_char*)b3;
  };
  // round r; past the end the last step again, into a place that nobody reads
  auto move = [&](int r, auto b_c) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kq = first + min(r * U + u, steps - 1);
      oa.move(kq, buffer(b_c) + STEP * u);
      ob.move(kq, buffer(b_c) + STEP * u + A::BYTES);
    }
  };
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  auto products = [&](int r, auto b_c) {
    const lds_char* buf = buffer(b_c);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u && r * U + u >= steps) break;
      bf16x8 x[SLICES], w[SLICES];
#pragma unroll
      for (int j = 0; j < SLICES; ++j) {
        w[j] = ob.template read<PLAIN>(buf + STEP * u + A::BYTES, wk * SLICES + j, wn, lane);
        x[j] = oa.template read<PLAIN>(buf + STEP * u, wk * SLICES + j, wm, lane);
      }
#pragma unroll
      for (int j = 0; j < SLICES; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[j], x[j], acc, 0, 0, 0);
    }
  };
  if (rounds <= 3) {  // all at once
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
    move(2, Int<2>{});
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
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the surplus transfers)
  }
  // ---- the waves' sums (lane: row l32 of a piece, columns 8 q + 4 h .. + 3) through LDS into runs of whole rows
  __syncthreads();
  const int l32 = lane & 31, h = lane >> 5;
  constexpr int ROW = TN * 4 + 16, PART = TM * ROW;  // bytes
  constexpr int FIRST = WK > 1 ? WK / 2 : 1;         // parts in b0 (64 x 64: its one begins there and ends in b1)
  auto place = [&](int w, int m, int n) {            // of row m, columns n .. of the wave group w
    if constexpr (WK > 1) return (w < FIRST ? b0 : b1) + w % FIRST * PART + m * ROW + n * 4;
    else return (m < TM / 2 ? b0 : b1) + m % (TM / 2) * ROW + n * 4;
  };
  static_assert((WK > 1 ? FIRST * PART : PART / 2) <= BUF, "room for the sums");
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *reinterpret_cast<f32x4*>(place(wk, wm + l32, wn + 8 * q + 4 * h)) = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
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
      *reinterpret_cast<bf16x8*>(a.c + at) = __builtin_shufflevector(narrowed(lo), narrowed(hi), 0, 1, 2, 3, 4, 5, 6, 7);
    }
  }
}

// The parts' sums, always in the same order
__global__ void __launch_bounds__(256) narrow_sum_kernel(const f32x4* __restrict__ part, bf16* __restrict__ c, int64_t n4, int parts) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  f32x4 v = part[i];
  for (int p = 1; p < parts; ++p) v += part[p * n4 + i];
  *reinterpret_cast<bf16x4*>(c + 4 * i) = narrowed(v);
}

int g_tile = 0, g_parts = 0;

struct Cut {
  int tm, tn, parts;  // tile, parts of K
};
// Tiles of 64 where those of 32 are more than two a CU (y of 128 tokens, us with 32 / 64: [3072, 1024] 6.4 / 6.9, [4096, 2048] 9.1 / 10.4,
// [5632, 1024] 9.3 / 7.1), with an operand across the inner dimension from 128 of them on. Such operands come in rows of 64, never 32 (half a cache line: dX of 128 tokens by [3072, 1024] 14.9 for 11.3). Parts where the
// tiles leave the chip idle: a sum costs 2 us and its traffic, so both operands along K want 2560 of it each (y of 64 tokens, [2048, 5632] 12.6
// whole, 10.5 in two; [1024, 2816] 7.7 and 7.7), while rows across it come slower (dX of 128 tokens by [5632, 1024] 42 whole, 15.8
// in four, 13.4 in eight; of 256 by [1024, 2816] 10.2 whole, 12.4 in two).
Cut cut_of(int64_t M, int64_t N, int64_t K, bool along) {
  auto tiles = [&](int tm, int tn) { return ((M + tm - 1) / tm) * ((N + tn - 1) / tn); };
  int tn = along ? 32 : 64, tm = 32;
  if (g_tile ? g_tile == 64 : along ? tiles(32, 32) > 512 : tiles(64, 64) >= 128) tm = tn = 64;
  const int64_t fill = (K >= 2048 ? 512 : 256) / tiles(tm, tn), longest = K / (along ? 2560 : 512);
  const int64_t parts = g_parts ? std::min<int64_t>(g_parts, (K + 63) / 64) : std::min<int64_t>(std::min(fill, longest), 8);
  return {tm, tn, (int)std::max<int64_t>(parts, 1)};
}

}  // namespace

// Forces tiles of 64 or 32 rows and parts of K; 0: by the rule above.
extern "C" void ds_narrow_gemm_tune(int tile, int parts) { g_tile = tile; g_parts = parts; }

// Whether the kernel takes the product: whole 16-byte pieces of rows, whole steps of 64 along an operand's rows, offsets of 32 bits
extern "C" int ds_narrow_gemm_ok(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_along, int b_along) {
  if (M <= 0 || N <= 0 || K <= 0 || M > INT32_MAX / 64 || N > INT32_MAX / 64 || K > INT32_MAX / 64) return 0;
  if (N % 8 || lda % 8 || ldb % 8 || ((a_along || b_along) && K % 64) || (!a_along && M % 8)) return 0;
  if (lda < (a_along ? K : M) || ldb < (b_along ? K : N)) return 0;
  const int64_t ar = a_along ? M : K, br = b_along ? N : K;
  return (ar + 128) * lda * 2 < UINT32_MAX && (br + 128) * ldb * 2 < UINT32_MAX && ((M + 31) / 32) * ((N + 31) / 32) <= INT32_MAX;
}

// Whether it is as fast as the library's there. y, dX: up to 2^31 products (256 tokens by [8000, 1024] 9.8 us and 13.2, 21 and 31; of 2^32,
// 128 tokens by [11264, 2048] 22 and 18). dW: up to 2^30 (256 tokens by [3072, 1024] 9.5 and 8.8, by [5632, 1024], 1.4 times 2^30, 13.8 and
// 11.4).
extern "C" int ds_narrow_gemm_pays(int64_t M, int64_t N, int64_t K, int a_along) { return M * N <= (1LL << (a_along ? 31 : 30)) / K; }

// Bytes of scratch memory that the product wants (0: none)
extern "C" int64_t ds_narrow_gemm_scratch(int64_t M, int64_t N, int64_t K, int a_along, int b_along) {
  const Cut c = cut_of(M, N, K, a_along && b_along);
  return c.parts > 1 ? c.parts * M * N * 4 : 0;
}

// C [M, N] = A B^T over K. a_along: A is [M, K] with rows lda apart, else [K, M]; b_along: B is [N, K], else [K, N]. part:
// ds_narrow_gemm_scratch bytes.
extern "C" int ds_narrow_gemm(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_along,
                              int b_along, void* part, hipStream_t st) {
  if (!ds_narrow_gemm_ok(M, N, K, lda, ldb, a_along, b_along)) return (int)hipErrorInvalidValue;
  const Cut cut = cut_of(M, N, K, a_along && b_along);
  if (cut.parts == 1) part = nullptr;
  else if (!part) return (int)hipErrorInvalidValue;
  const int64_t ar = a_along ? M : K, ac = a_along ? K : M, br = b_along ? N : K, bc = b_along ? K : N;
  const NarrowArgs a{(const bf16*)A, (const bf16*)B, (bf16*)C, (int)M, (int)N, (int)K, (uint32_t)lda, (uint32_t)ldb,
                     (uint32_t)(((ar - 1) * lda + ac) * 2), (uint32_t)(((br - 1) * ldb + bc) * 2), cut.parts, (f32x4*)part};
  const dim3 grid((unsigned)(((M + cut.tm - 1) / cut.tm) * ((N + cut.tn - 1) / cut.tn)), cut.parts);
#define GO(AK, BK, TM, TN, U) hipLaunchKernelGGL((narrow_gemm_kernel<AK, BK, TM, TN, U>), grid, dim3(256), 0, st, a)
  if (cut.tm == 64) {
    if (a_along && b_along) GO(true, true, 64, 64, 1);
    else if (a_along) GO(true, false, 64, 64, 1);
    else if (b_along) GO(false, true, 64, 64, 1);
    else GO(false, false, 64, 64, 1);
  } else {
    if (a_along && b_along) GO(true, true, 32, 32, 2);
    else if (a_along) GO(true, false, 32, 64, 1);
    else if (b_along) GO(false, true, 32, 64, 1);
    else GO(false, false, 32, 64, 1);
  }
#undef GO
  if (part) {
    const int64_t n4 = M * N / 4;
    hipLaunchKernelGGL(narrow_sum_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st, (const f32x4*)part, (bf16*)C, n4, cut.parts);
  }
  DS_CHECK_LAUNCH();
  return 0;
}
