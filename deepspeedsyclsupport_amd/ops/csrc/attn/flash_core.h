// The loop of dense attention over heads of 128 (flash_dense.hip, paged_rows.h), CDNA4 (gfx950): 32 query rows a wave, four waves a workgroup that share
// tiles of 64 keys in LDS, two workgroups a CU.
//
// What bounds it is what a wave can issue (matrix cores busy 52 to 56 % of the time, at 1.9 to 2 GHz): of 64 keys 64 products, 32 exponentials and 100 other
// vector instructions a lane. Hence
//  * in halves of a tile: beside the exponentials of one, product by product, go the scores of the next and the values of the one before. A half's scores
//    and weights are the registers of the other one's but one, so nothing is copied, and 200 registers hold it all (whole tiles beside each other: 242 and
//    40 copies a tile, 3 % longer; 64 rows in one wave a SIMD: 4 to 10 % longer);
//  * products of 16 x 16 x 32, keys by rows: a lane has 4 keys of a block of 16 for one query row, as scores, as the weights that the values' products
//    take, and, with the values as the first operand, as 4 columns of the result: sums, maxima and their rescaling stay within the lane, and 16-byte stores
//    need one exchange between rows of 16 lanes;
//  * one barrier a tile, in its middle: there the next keys and this tile's values have to be there, and the slots of this tile's keys and the
//    last one's values are free. Two slots of either, 64 KB;
//  * a row's reference (the exponent that its weights are taken against) is the maximum of the first 64 keys and moves, to a maximum, only once one is 2^8 past
//    it, a half's check without an exchange between lanes. What waits for its values then is still weighed against the old one: the result is rescaled
//    after it.
// us before (a tile's scores, weights and values one after another, 32 x 32 x 16) and so, causal, head by head: 1 x 8192, 32 heads over 8 587, 491; 2 x 4096, 32 heads
// 335, 301; 8 x 512, 16 over 8 25.6, 23.8; without a mask, 1 x 8192 1053, 930.
#pragma once
#include "each.h"

namespace flash {
using namespace constants;

constexpr int D = 128, BN = 64, WAVES = 4, ROWS = 32;  // head, keys of a tile, rows of a wave
constexpr uint32_t TILE = BN * D * 2;                  // 16 KB
constexpr uint32_t LDS = 4 * TILE;                     // K0 K1 V0 V1

__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {  // two bf16, round to nearest even
  uint32_t r;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(lo), "v"(hi));
  return r;
}

// A tile lies in rows of 256 bytes, 16-byte chunk c of row r at c ^ swizzle(r): a bijection of r % 16 with which neither 16 rows' reads of a chunk nor
// transposed reads of 32 bytes of 4 rows meet in a bank
__device__ __forceinline__ int swizzle(int r) { return ((r & 3) << 2) | ((((r >> 2) ^ (r >> 3)) & 1) << 1) | ((r >> 3) & 1); }

// Transfers to LDS, 16 bytes a lane, in inline asm: hipcc waits for its own ones before each LDS read that it cannot tell from their target. A tile is 16
// pieces of 4 rows; wave w moves the pieces w, w + 4, ..: lane L of a piece lands at chunk L % 16 of its row and fetches what belongs there. Its row
// modulo 16 is the same in all pieces.
__device__ __forceinline__ int dma_row(int lane, int wid) { return 4 * wid + (lane >> 4); }
__device__ __forceinline__ int dma_column(int lane, int wid) { return 8 * ((lane & 15) ^ swizzle(dma_row(lane, wid))); }
__device__ __forceinline__ void dma16(const char* base, uint32_t lane_bytes, uint32_t dst) {  // wave-uniform base
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_bytes), "s"(base), "s"(dst) : "memory");
}
__device__ __forceinline__ void dma16(const char* from, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(dst) : "memory");
}
// All transfers and LDS accesses of this wave are done, then those of all waves
__device__ __forceinline__ void meet() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 16 columns of 32 rows of a tile, transposed: rows 4 (lane / 16) .. + 3 of either 16, as two blocks of sums have them. at: of rows 0 .. 15
__device__ __forceinline__ bf16x8 columns(uint32_t at) {
  lds_char* p = (lds_char*)(uintptr_t)at;
  s16x8 v;
#ifdef __HIP_DEVICE_COMPILE__
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p), hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4096));
  v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#endif
  return __builtin_bit_cast(bf16x8, v);
}
// 128 columns of the row that a lane has, 4 (lane / 16) .. + 3 of every 16 in o, times `by`: eight columns a piece
__device__ __forceinline__ void store_row(const f32x4 (&o)[8], float by, bf16* row, int lane, bool mine) {
  const int g = lane >> 4;
  each<4>([&](auto d_c) {
    constexpr int d = 2 * d_c.value;
    const f32x4 a = o[d] * by, b = o[d + 1] * by;
    u32x4 w;
#ifdef __HIP_DEVICE_COMPILE__
    // (packed in the compiler's sight, which knows what a swap waits for)
    auto two = [](float lo, float hi) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2)); };
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const auto v = __builtin_amdgcn_permlane16_swap(two(a[2 * i], a[2 * i + 1]), two(b[2 * i], b[2 * i + 1]), false, false);
      w[i] = v[0];
      w[2 + i] = v[1];
    }
#endif
    if (mine) *reinterpret_cast<u32x4*>(row + 16 * d + 16 * (g & 1) + 8 * (g >> 1)) = w;
  });
}

// A wave's 32 rows: blocks q of 16, of which a lane has row lane % 16
struct Rows {
  bf16x8 qf[2][4], kf[4], vf[4];  // queries; operands read ahead
  f32x4 o[2][8];                  // [row block][16 columns]: columns 4 (lane / 16) .. + 3
  f32x4 s[4][2];                  // scores [16 keys][row block]: keys 4 (lane / 16) .. + 3; of a tile's halves one to be weighed, the other to come
  u32x4 p[2][2];                  // weights [row block][half]
  float ref[2], l[2], mx[2], turn_by[2], x[16];  // reference, in exponents; sums; maxima of the scores to come; what the result is to be rescaled by
  bool late;                      // ... after the values that wait
  uint32_t ka[4], va[8];          // LDS addresses of the tiles' reads
  float c;                        // scale log2(e)

  __device__ __forceinline__ bf16x8 keys(int kb, int ks) const { return *reinterpret_cast<const lds_bf16x8*>((const lds_char*)(uintptr_t)ka[ks] + kb * 4096); }
  // 16 columns db of 32 keys: those of a lane's weights
  __device__ __forceinline__ bf16x8 values(int db, int half) const { return columns(va[db] + half * 8192); }
  // The keys' first tile, the values' place before theirs. base: of the LDS, a multiple of 32 KB
  __device__ __forceinline__ void init(uint32_t base, int lane, float scale_log2) {
    const int g = lane >> 4, l16 = lane & 15, r = 4 * g + ((lane >> 2) & 3);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) ka[ks] = base + l16 * 256 + 16 * ((4 * ks + g) ^ swizzle(l16));
#pragma unroll
    for (int db = 0; db < 8; ++db) va[db] = base + 3 * TILE + r * 256 + 16 * ((2 * db + ((lane >> 1) & 1)) ^ swizzle(r)) + 8 * (lane & 1);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      l[q] = 0.f;
      p[q][0] = p[q][1] = u32x4{0, 0, 0, 0};
#pragma unroll
      for (int db = 0; db < 8; ++db) o[q][db] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    ref[0] = ref[1] = 0.f;
    c = scale_log2;
    late = false;
  }
  // to the other tile of keys and of values
  __device__ __forceinline__ void turn() {
#pragma unroll
    for (int i = 0; i < 4; ++i) ka[i] ^= TILE;
#pragma unroll
    for (int i = 0; i < 8; ++i) va[i] ^= TILE;
  }
  template <bool FIRST>
  __device__ __forceinline__ void score(int kb, int q, bf16x8 k, int ks) {
    s[kb][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, qf[q][ks], FIRST ? f32x4{0.f, 0.f, 0.f, 0.f} : s[kb][q], 0, 0, 0);
  }
  __device__ __forceinline__ void add(int q, int db, bf16x8 v, int half) {
    o[q][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, __builtin_bit_cast(bf16x8, p[q][half]), o[q][db], 0, 0, 0);
  }
  // A row's maximum over the lanes that have keys of it
  static __device__ __forceinline__ float over_row(float v) {
    v = fmaxf(v, __shfl_xor(v, 16, 64));
    return fmaxf(v, __shfl_xor(v, 32, 64));
  }
  // Scores of the whole first tile, masked by `mask(half)`, whose maxima are the first references
  template <class M>
  __device__ __forceinline__ void first(M&& mask) {
    each<4>([&](auto ks) {
      each<4>([&](auto kb) {
        const bf16x8 k = keys(kb.value, ks.value);
        each<2>([&](auto q) { score<ks.value == 0>(kb.value, q.value, k, ks.value); });
      });
    });
    mask(Int<0>{});
    mask(Int<1>{});
    each<2>([&](auto q) {
      float v = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) v = fmaxf(v, s[kb][q.value][i]);
      v = over_row(v);
      ref[q.value] = v == -INFINITY ? 0.f : v * c;
    });
  }
  // The weights of half C of the tile, beside the scores of the half that comes next, then the values of the one that came last. Slots FROM to TO, one
  // before each of 32 products; MID: the scores are complete, none of their maxima taken.
  static constexpr int MID = 22, END = 32;
  template <int C, int FROM, int TO>
  __device__ __forceinline__ void half() {
    constexpr int N = 1 - C;  // (of its tile, the half that comes next, and that came last)
    if constexpr (FROM == 0) each<3>([&](auto f) { kf[f.value] = keys(2 * N + (f.value & 1), f.value >> 1); });
    each<TO - FROM>([&](auto t_c) {
      constexpr int t = FROM + t_c.value, f = t >> 1, q = t & 1, e = t >> 1, ahead = f + 3;
      if constexpr (q == 1 && ahead < 8) kf[ahead & 3] = keys(2 * N + (ahead & 1), ahead >> 1);
      if constexpr (q == 1 && ahead >= 8 && ahead < 16) vf[ahead & 3] = values(ahead - 8, N);
      // 16 weights: one is scaled a slot pair ahead of its exponential, that is summed and packed behind it
      auto scaled = [&](auto i_c) {
        constexpr int i = i_c.value;
        x[i] = fmaf(s[2 * C + ((i >> 2) & 1)][i >> 3][i & 3], c, -ref[i >> 3]);
      };
      if constexpr (q == 0) {
        if constexpr (e == 0) scaled(Int<0>{});
        if constexpr (e + 1 < 16) scaled(Int<e + 1>{});
        x[e] = __builtin_amdgcn_exp2f(x[e]);
      } else {
        if constexpr (e >= 1) l[(e - 1) >> 3] += x[e - 1];
        if constexpr (e >= 3 && (e & 1)) p[(e - 3) >> 3][C][((e - 3) & 7) >> 1] = pack2(x[e - 3], x[e - 2]);
        if constexpr (e == 15) {
          l[1] += x[15];
          p[1][C][3] = pack2(x[14], x[15]);
        }
      }
      if constexpr (t >= 24) {  // eight maxima with two scores
        constexpr int i = t - 24, Q = i >> 2, k = (i >> 1) & 1, r = (i & 1) * 2;
        const f32x4& v = s[2 * N + k][Q];
        mx[Q] = (i & 3) == 0 ? max3(v[0], v[1], v[1]) : max3(mx[Q], v[r], v[r + 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (f < 8) score<(f < 2)>(2 * N + (f & 1), q, kf[f & 3], f >> 1);
      else add(q, f - 8, vf[f & 3], N);
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  // After a half. more: the scores to come are somebody's
  __device__ __forceinline__ void settle(bool more) {
    if (late) rescale();
    bool past = false;
#pragma unroll
    for (int q = 0; q < 2; ++q) past |= mx[q] * c > ref[q] + 8.f;
    if (more && __any(past)) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float v = over_row(mx[q]) * c, to = v > ref[q] + 8.f ? v : ref[q];
        turn_by[q] = __builtin_amdgcn_exp2f(ref[q] - to);
        ref[q] = to;
        l[q] *= turn_by[q];
      }
      late = true;
    }
  }
  __device__ __forceinline__ void rescale() {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int db = 0; db < 8; ++db) o[q][db] *= turn_by[q];
    late = false;
  }
  // Nothing has been added up before the first half
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int db = 0; db < 8; ++db) o[q][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // What waits behind the last half
  __device__ __forceinline__ void last() {
    each<8>([&](auto db) {
      const bf16x8 v = values(db.value, 1);
      each<2>([&](auto q) { add(q.value, db.value, v, 1); });
    });
    if (late) rescale();
  }
  // `tiles` of this wave, of the workgroup's `all`. mask(half, tile): its scores; pass(): the barrier of a tile, behind it the transfers of the keys after
  // next and of the next values. (Nobody reads values 1 before their tile has come: the products with those before tile 0, which there are none of, are
  // taken back; keys past the end are in nobody's scores.)
  template <class M, class P>
  __device__ __forceinline__ void run(int tiles, int all, M&& mask, P&& pass) {
    if (tiles > 0) first([&](auto h) { mask(h, 0); });
    int j = 0;
    for (; j < tiles; ++j) {
      half<0, 0, MID>();
      mask(Int<1>{}, j);
      half<0, MID, END>();
      if (j == 0) clear();
      settle(true);
      pass();
      turn();
      half<1, 0, MID>();
      if (j + 1 < tiles) mask(Int<0>{}, j + 1);
      half<1, MID, END>();
      settle(j + 1 < tiles);
    }
    if (tiles > 0) last();
    for (; j < all; ++j) pass();
  }
  // A row's sum
  __device__ __forceinline__ float sum(int q) const {
    const float v = l[q] + __shfl_xor(l[q], 16, 64);
    return v + __shfl_xor(v, 32, 64);
  }
  // Block q of the result times `by`, to the row that the lane has
  __device__ __forceinline__ void store(int q, float by, bf16* row, int lane, bool mine) { store_row(o[q], by, row, lane, mine); }
};

}  // namespace flash
