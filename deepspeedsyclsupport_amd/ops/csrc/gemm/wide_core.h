// The loop of the products over 256 columns a workgroup (wide_gemm.hip), CDNA4 (gfx950): four waves, one on a SIMD with all its registers, 2 x 2 over a
// tile of 32 MI x 256, each with MI x 8 blocks of 16 x 16 in its accumulators.
//
// What bounds it is power first (the chip runs at 1.7 to 1.8 GHz under it, matrix cores busy 82 to 84 % of the time) and what a wave can issue
// between two products second. Hence
//  * products of 16 x 16 x 32: in registers alone, on normally distributed values, they reach 2130 TF/s where 32 x 32 x 16 reach 1870 (an accumulator
//    is read and written half as often for its work), and neighbours share an operand (2150 against 2050);
//  * they are inline asm with accumulators in their place: as builtins hipcc moves accumulators about. A tile's first products take zero for the
//    accumulator, so none is cleared;
//  * both operands come by DMA, without registers, a step of 64 of the inner dimension at a time into rings of RA and RB slots; A's go out in a step's
//    first half, B's in its second, one every 6 or 7 products: all at once, in the second half, 1395 TF/s, so 1530 (a transfer takes the address unit 16
//    clocks, for all four waves, and whoever waits for it issues no products);
//  * each half of a step reads the other half's operands from LDS into registers, so that a step's slots are free at its middle: one barrier a step, there,
//    whose wait counts what may still be on its way;
//  * the buffers' addresses advance in scalar registers, a few instructions between two products (in one place, between two steps: 1520, so 1600);
//  * workgroups stay and go from tile to tile: the next one's first steps are on their way, the first read, before this one's results leave.
// 8192 tokens, us here and by the library's call: y by [4096, 11008] 455 / 454 (1624 TF/s), by [12288, 4096] 527 / 524; dX by [4096, 11008] 464 / 524;
// dW [4096, 11008] 508 / 768, of 688 tiles where 768 would fit.
#pragma once
#include "each.h"

namespace wide {
using namespace constants;

typedef int i32x4 __attribute__((ext_vector_type(4)));

// A buffer of `bytes` bytes: what lies past its end reads as zero
__device__ __forceinline__ i32x4 buffer_of(const void* p, uint32_t bytes) {
  const uint64_t at = (uint64_t)p;
  return i32x4{__builtin_amdgcn_readfirstlane((int)at), __builtin_amdgcn_readfirstlane((int)(at >> 32)), __builtin_amdgcn_readfirstlane((int)bytes),
               0x00020000};
}

// 16 bytes per lane to LDS bytes dst + 16 lane
__device__ __forceinline__ void dma16(i32x4 from, uint32_t lane_bytes, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(dst), "v"(lane_bytes), "s"(from) : "memory");
}

// c = a b^T (+ c): lane's values are columns lane % 16 of b's rows, rows 4 (lane / 16) .. + 3 of a's
template <bool FIRST>
__device__ __forceinline__ void product(f32x4& c, bf16x8 a, bf16x8 b) {
  if constexpr (FIRST) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
// ... and a transfer to LDS bytes `to` + MORE + 16 lane, the product between its M0 and itself
template <bool FIRST>
__device__ __forceinline__ void product_and_dma(f32x4& c, bf16x8 a, bf16x8 b, i32x4 from, uint32_t lane_bytes, uint32_t to, int more) {
  if constexpr (FIRST)
    asm volatile("s_add_u32 m0, %5, %6\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, 0\n\tbuffer_load_dwordx4 %3, %4, 0 offen lds"
                 : "=&a"(c)
                 : "v"(a), "v"(b), "v"(lane_bytes), "s"(from), "s"(to), "i"(more)
                 : "memory", "scc");
  else
    asm volatile("s_add_u32 m0, %5, %6\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\tbuffer_load_dwordx4 %3, %4, 0 offen lds"
                 : "+a"(c)
                 : "v"(a), "v"(b), "v"(lane_bytes), "s"(from), "s"(to), "i"(more)
                 : "memory", "scc");
}
__device__ __forceinline__ void dma16(i32x4, const char* from, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(from) : "memory");
}
template <bool FIRST>
__device__ __forceinline__ void product_and_dma(f32x4& c, bf16x8 a, bf16x8 b, i32x4, const char* from, uint32_t to, int more) {
  if constexpr (FIRST)
    asm volatile("s_add_u32 m0, %4, %5\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, 0\n\tglobal_load_lds_dwordx4 %3, off"
                 : "=&a"(c)
                 : "v"(a), "v"(b), "v"(from), "s"(to), "i"(more)
                 : "memory", "scc");
  else
    asm volatile("s_add_u32 m0, %4, %5\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\tglobal_load_lds_dwordx4 %3, off"
                 : "+a"(c)
                 : "v"(a), "v"(b), "v"(from), "s"(to), "i"(more)
                 : "memory", "scc");
}
__device__ __forceinline__ void hold(f32x4& c) { asm volatile("" : "+a"(c)); }

// All of this wave's LDS accesses and all but its NEWER latest transfers and stores are done, then those of all waves.
template <int NEWER>
__device__ __forceinline__ void meet() {
  static_assert(NEWER < 64, "as far as the counter goes");
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((NEWER & 15) | 7 << 4 | (NEWER >> 4) << 14);
  asm volatile("s_barrier" ::: "memory");
}

// How an operand lies: its rows across the inner dimension; along it; along it in rows that lie anywhere, by 64-bit addresses; in operand order (blocks of
// 16 rows, of which 64 columns at a time are 2 KB: `preshuffle16` of ops/bf16_gemv.py)
enum : int { ACROSS = 0, ALONG = 1, FAR = 2, ORDERED = 3 };

// One operand's R rows (or columns) of a step of 64, of which a wave multiplies F blocks of 16: its way into LDS and out of it
template <int LAY, int R, int F>
struct Operand {
  static constexpr int BYTES = R * 128, PIECES = R / 32;  // LDS bytes a step, transfers of 1 KB a wave
  static constexpr int BASES = LAY == ACROSS ? F : LAY == ORDERED ? 1 : 2;
  typedef std::conditional_t<LAY == FAR, const char*, uint32_t> Source;
  i32x4 from;          // the tile, from the step of the next transfers on
  Source src[PIECES];  // per lane: bytes from there (FAR: where they are)
  uint32_t step;       // bytes from a step to the next
  uint32_t at[BASES];  // LDS address of the lane's reads in the slot at work: of either half, of each block, or of all

  // from row r0, and k0 of the inner dimension on
  static __device__ __forceinline__ i32x4 tile(const bf16* p, uint32_t bytes, uint32_t ld, int r0, int k0 = 0) {
    const uint32_t off = LAY == ACROSS ? 2u * r0 + (uint32_t)k0 * ld * 2 : (uint32_t)r0 * ld * 2 + 2u * k0;
    return buffer_of((const char*)p + off, bytes - off);
  }
  // A transposed read takes 32 bytes of four rows, and of the four that lie 8 further, at a time: those of rows of 2 R bytes that meet in a bank are apart
  static __device__ __forceinline__ int turn(int r) { return (R % 128 ? ((r >> 1) & 1) << 2 : (r & 3) << 2) ^ (((r >> 3) & 1) << 1); }
  // Row r of a step of rows along the inner dimension: 8 chunks of 16 bytes, chunk c at c ^ (r / 2 % 8). Of the lane's row in piece i
  static __device__ __forceinline__ int row(int i, int lane, int wid) { return 8 * (wid * PIECES + i) + (lane >> 3); }
  static __device__ __forceinline__ uint32_t chunk(int i, int lane, int wid) { return 16 * ((lane & 7) ^ ((row(i, lane, wid) >> 1) & 7)); }
  // Rows ld apart
  __device__ __forceinline__ void sources(uint32_t ld, int lane, int wid) {
    step = __builtin_amdgcn_readfirstlane(LAY == ALONG ? 128 : 128 * ld);
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      if constexpr (LAY == ALONG) {
        src[i] = (uint32_t)row(i, lane, wid) * ld * 2 + chunk(i, lane, wid);
      } else {  // R / 8 chunks of each of the step's rows, swizzled by `turn`
        const int c = (wid * PIECES + i) * 64 + lane, r = c / (R / 8);
        src[i] = (uint32_t)r * ld * 2 + 16 * (c % (R / 8) ^ turn(r));
      }
    }
  }
  // r0: first of the wave's rows in the tile
  __device__ __forceinline__ void reads(uint32_t slot, int r0, int lane) {
    if constexpr (LAY == ACROSS) {
      const int k = 8 * (lane >> 4) + ((lane >> 2) & 3);
#pragma unroll
      for (int f = 0; f < F; ++f) at[f] = slot + k * 2 * R + 16 * ((r0 / 8 + 2 * f + ((lane >> 1) & 1)) ^ turn(k)) + 8 * (lane & 1);
    } else if constexpr (LAY == ORDERED) {  // chunk 2 q + h of a block's row r at 64 h + 16 q + r
      at[0] = slot + r0 * 128 + 1024 * ((lane >> 4) & 1) + 256 * (lane >> 5) + 16 * (lane & 15);
    } else {
      const int r = r0 + (lane & 15);
#pragma unroll
      for (int h = 0; h < 2; ++h) at[h] = slot + r * 128 + 16 * ((4 * h + (lane >> 4)) ^ ((r >> 1) & 7));
    }
  }
  // The next transfers: `by` bytes further, or another tile's first
  __device__ __forceinline__ void next(uint32_t by) {
    if constexpr (LAY == FAR) {
#pragma unroll
      for (int i = 0; i < PIECES; ++i) src[i] += by;
    } else {
      const uint64_t p = ((uint64_t)(uint32_t)from[1] << 32 | (uint32_t)from[0]) + by;
      from[0] = (int)(uint32_t)p;
      from[1] = (int)(uint32_t)(p >> 32);
      if constexpr (LAY == ACROSS) from[2] -= (int)by;  // (rows past the end read as zero)
    }
  }
  __device__ __forceinline__ void next(bool other, const i32x4& tile) {
    next(step);
#pragma unroll
    for (int i = 0; i < 3; ++i) from[i] = other ? tile[i] : from[i];
  }
  // Block B of half H; a step's first half lies in a slot `delta` further than what was read last
  template <int H, int B>
  __device__ __forceinline__ bf16x8 read(uint32_t delta) {
    if constexpr (H == 0 && B < BASES) at[B] += delta;
    if constexpr (LAY == ORDERED) {
      const lds_char* p = (const lds_char*)(uintptr_t)at[0];
      return *reinterpret_cast<const lds_bf16x8*>(p + B * 2048 + H * 512);
    } else if constexpr (LAY != ACROSS) {
      const lds_char* p = (const lds_char*)(uintptr_t)at[H];
      return *reinterpret_cast<const lds_bf16x8*>(p + B * 2048);
    } else {
      lds_char* p = (lds_char*)(uintptr_t)at[B];
      s16x8 v;
#ifdef __HIP_DEVICE_COMPILE__
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + H * 64 * R));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + H * 64 * R + 8 * R));
      v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#endif
      return __builtin_bit_cast(bf16x8, v);
    }
  }
};

constexpr int STEPS = 4;  // the fewest of a tile that others follow: its transfers are so far ahead

// A's and B's rings, and the loop over one tile's steps, after another's (CHAIN) or alone
template <int AK, int BK, int MI, bool CHAIN>
struct Loop {
  static constexpr int NI = 8, TM = 32 * MI, TN = 32 * NI;
  // 160 KB: as many steps ahead as there is room for
  static constexpr int RA = MI == 8 ? 3 : 4, RB = MI == 2 ? 4 : MI == 4 ? 3 : 2;
  typedef Operand<AK, TM, MI> A;
  typedef Operand<BK, TN, NI> B;
  static constexpr int PA = A::PIECES, PB = B::PIECES, LDS = RA * A::BYTES + RB * B::BYTES;
  // Of a step's transfers the first LATE go out in its second half, the rest (the end of B's, where B is three steps ahead; A's) in the next one's first
  static constexpr int LATE = RB == 2 ? PB : (PA + PB) / 2, EARLY = PA + PB - LATE;
  static constexpr int ALL = MI * NI, READS = MI + NI;
  static constexpr int MEET = ALL * 61 / 64;              // products of the first half before the barrier
  static constexpr int EVERY = (MEET - 1) / (EARLY > LATE ? EARLY : LATE);  // products from a transfer to the next
  // At a step's barrier the next step has to be there: what may be newer than its last piece of B, and of A
  static constexpr int NEWER_B = PA + (RB - 2) * (PA + PB), NEWER_A = (RA - 2) * (PA + PB), NEWER = NEWER_B < NEWER_A ? NEWER_B : NEWER_A;
  static_assert(LDS <= 160 * 1024 && EVERY >= 1 && LATE <= PB);
  static_assert(!CHAIN || (RA <= STEPS && RB <= STEPS), "a tile's transfers end before they are as far ahead");

  A oa;
  B ob;
  f32x4 acc[MI][NI];
  bf16x8 xa[2][MI], xb[2][NI];
  uint32_t first_a, first_b, da, db, ta, tb;  // this wave's part of slot 0; of the slot that transfers go to; from the slot at work to the next

  // All of step `slot` (the first ones)
  template <int N>
  __device__ __forceinline__ void move_a(int slot) {
    each<N>([&](auto i) { dma16(oa.from, oa.src[i.value], first_a + slot * A::BYTES + 1024 * i.value); });
  }
  template <int N>
  __device__ __forceinline__ void move_b(int slot) {
    each<N>([&](auto i) { dma16(ob.from, ob.src[i.value], first_b + slot * B::BYTES + 1024 * i.value); });
  }
  // Before the first tile, of so many steps; from, src and step are the operands'
  __device__ __forceinline__ void begin(char* lds, int steps, int lane, int wid) {
    const uint32_t base = (uint32_t)(uintptr_t)(lds_char*)lds, bbase = base + RA * A::BYTES;
    oa.reads(base, (wid & 1) * 16 * MI, lane);
    ob.reads(bbase, (wid >> 1) * 16 * NI, lane);
    first_a = base + wid * PA * 1024;
    first_b = bbase + wid * PB * 1024;
    each<(RA > RB ? RA : RB)>([&](auto s) {  // (past the end of a tile alone its last step again, for nobody)
      if constexpr (s.value < RB - 1) { move_b<PB>(s.value); ob.next(CHAIN || s.value + 1 < steps ? ob.step : 0); }
      if constexpr (s.value == RB - 1) move_b<LATE>(s.value);
      if constexpr (s.value < RA - 1) { move_a<PA>(s.value); oa.next(CHAIN || s.value + 1 < steps ? oa.step : 0); }
    });
    da = first_a + (RA - 1) * A::BYTES;
    db = first_b + (RB - 1) * B::BYTES;
    if constexpr (LATE == PB) { db = first_b; ob.next(CHAIN || RB < steps ? ob.step : 0); }
    ta = tb = 0;
    // (the first two steps: the first barrier counts by what was stored before it, which here is nothing)
    constexpr int AFTER = (RB > 2 ? (RB - 3) * PB + LATE : 0) + (RA - 3) * PA;
    meet<AFTER>();
    each<NI>([&](auto i) { xb[0][i.value] = ob.template read<0, i.value>(0); });
    each<MI>([&](auto i) { xa[0][i.value] = oa.template read<0, i.value>(0); });
  }

  // The operand's next transfers, which are those of AHEAD steps from here on
  template <int AHEAD, class O>
  __device__ __forceinline__ void go(O& o, int left, const i32x4& after) {
    if constexpr (CHAIN) o.next(left == AHEAD, after);
    else o.next(left > AHEAD ? o.step : 0);
  }
  // Half H of a step, `left` steps of the tile left with it. after: where the tile that follows begins. STORES: those since the tile before (its first half).
  template <int H, bool FIRST, int STORES>
  __device__ __forceinline__ void half(int left, const i32x4& after_a, const i32x4& after_b) {
    each<ALL>([&](auto t_c) {
      constexpr int t = t_c.value;
      if constexpr (H == 0 && t == MEET) meet<NEWER + (FIRST ? STORES : 0)>();
      // what the other half multiplies
      each<READS>([&](auto i_c) {
        constexpr int i = i_c.value;
        if constexpr (t == i * (ALL * (H ? 52 : 44) / 64) / READS) {
          if constexpr (i < NI) xb[H ^ 1][i] = ob.template read<H ^ 1, i>(tb);
          else xa[H ^ 1][i - NI] = oa.template read<H ^ 1, i - NI>(ta);
        }
      });
      // the slots and addresses of the next transfers, once those of before are out
      if constexpr (H == 0 && t == ALL - 3) go<RA>(oa, left, after_a);
      if constexpr (H == 0 && t == ALL - 2) {
        const uint32_t turned = da == first_a + (RA - 1) * A::BYTES ? first_a : da + A::BYTES;  // slot of step s + RA, as of step s
        da = turned;
        ta = turned == first_a + (RA - 1) * A::BYTES ? -(uint32_t)(RA - 1) * A::BYTES : A::BYTES;
      }
      if constexpr (H == 0 && t == ALL - 1) {
        if constexpr (LATE < PB) go<RB>(ob, left, after_b);
        const uint32_t turned = LATE < PB ? (db == first_b + (RB - 1) * B::BYTES ? first_b : db + B::BYTES) : db;
        db = turned;
        tb = turned == first_b + (RB - 1) * B::BYTES ? -(uint32_t)(RB - 1) * B::BYTES : B::BYTES;
      }
      if constexpr (H == 1 && LATE == PB && t == ALL - 3) go<RB + 1>(ob, left, after_b);
      if constexpr (H == 1 && LATE == PB && t == ALL - 2) db += tb;
      __builtin_amdgcn_sched_barrier(0);
      constexpr int m = t / NI, n = m & 1 ? NI - 1 - t % NI : t % NI;
      constexpr int p = t / EVERY + (H ? 0 : LATE);  // transfers: B's pieces, then A's
      constexpr bool sends = t % EVERY == 0 && p < (H ? LATE : PA + PB);
      if constexpr (sends && p < PB) product_and_dma<FIRST>(acc[m][n], xb[H][n], xa[H][m], ob.from, ob.src[p], db, 1024 * p);
      else if constexpr (sends) product_and_dma<FIRST>(acc[m][n], xb[H][n], xa[H][m], oa.from, oa.src[p - PB], da, 1024 * (p - PB));
      else product<FIRST>(acc[m][n], xb[H][n], xa[H][m]);
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  // One tile. The sums may be read after it.
  template <int STORES>
  __device__ __forceinline__ void tile(int steps, const i32x4& after_a, const i32x4& after_b) {
    half<0, true, STORES>(steps, after_a, after_b);
    int left = steps;
    for (; left > 1; --left) {
      half<1, false, 0>(left, after_a, after_b);
      half<0, false, 0>(left - 1, after_a, after_b);
    }
    half<1, false, 0>(1, after_a, after_b);
    asm volatile("s_nop 15\n\ts_nop 7");  // (the products are done: hipcc does not see that they are some)
    each<MI>([&](auto m) { each<NI>([&](auto n) { hold(acc[m.value][n.value]); }); });
    __builtin_amdgcn_sched_barrier(0);
  }
};

}  // namespace wide
