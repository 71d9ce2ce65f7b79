// Ragged paged flash attention for heads of 128: the arguments and modes of paged_prefill_core.h (PLAIN, EXT), the loop of
// flash_fwd.hip.
//
// What bounds it: the matrix cores and, beside them, the vector unit's issue slots (softmax). Against the kernel for any width:
//  * K and V tiles go from the cache to LDS by DMA, without registers, and the transfer of tile j + 1 runs under the products of
//    tile j. A page of 16 tokens or more holds 16 rows of a tile at a place of its own: its number is a scalar load, taken a
//    tile ahead, and the rest of the address one offset per lane for all tiles. Only a ragged last tile is addressed row by row;
//  * operand reads from LDS run ahead of their products in a pinned order; probabilities are packed two per instruction; the
//    output is rescaled only when the maximum has moved by more than 2^8;
//  * an XCD has heads of its own and takes the heaviest query blocks of all of them first (from twelve heads on of four at a time). (All heads of a run of neighbouring blocks to an
//    XCD: the last one did 15 / 8 of the mean work while the first was idle. Head by head: the last head's longest rows began when the others
//    were nearly through.) Heads that do not share out evenly go round the chip only over long contexts, which outweigh the other XCDs' reads of
//    their keys. us, head by head and so, the sink's form: 1 x 8192, 32 heads over 8 738, 697; 4 x 2048 229, 204; 8 x 660 on average 83, 74;
//    1 x 1500 54.6, 45.9; 16 over 8 4 x 2048 134, 115; 21 x 230 27.7, 28.1; 20 over 4 1 x 8192 556, 450, but 48 x 160 41.0, 44.3; 12 over 12
//    1 x 8192 348, 285, but 4 x 2048 99, 103 and 12 x 640 41.4, 45.3.
// 1 x 8192 causal, 32 query heads over 8: 1545 -> 587 us (paged_rows.h now: 512 back to back, 557 in a pass between other kernels); 4 x 2048, chunks of 2048, two-term weights, sink: 540 ->
// 265 us.
#pragma once
#include <type_traits>

#include "paged_prefill_core.h"

namespace {

typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
typedef __attribute__((address_space(3))) bf16x8_t lds_bf16x8;
// read-only and wave-uniform: scalar loads, whatever the kernel writes or clobbers in between
typedef __attribute__((address_space(4))) const int const_int;

constexpr int FD = 128;                     // head width
constexpr int FTILE = BN * FD * 2;          // 16 KB
constexpr int FLDS = 4 * FTILE + 4 * 32 * 4;  // K0 K1 V0 V1, a row of scratch per wave

// 16 bytes per lane from global memory to LDS byte `dst` + OFF + 16 * lane; see flash_fwd.hip for why this is inline asm
template <int OFF>
__device__ __forceinline__ void dma16(const void* g, uint32_t dst) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\t"
               "s_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(g), "s"(dst), "n"(OFF)
               : "memory", "scc");
}
template <int OFF>
__device__ __forceinline__ void dma16_s(const char* base, uint32_t voff, uint32_t dst) {  // wave-uniform base, offset per lane
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_add_u32 m0, %3, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\t"
               "s_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(voff), "s"(base), "s"(dst), "n"(OFF)
               : "memory", "scc");
}
__device__ __forceinline__ float fmax3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ unsigned pack2(float lo, float hi) {  // two bf16, round to nearest even
  unsigned r;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(lo), "v"(hi));
  return r;
}

// page_shift: log2 of the page size, 4 or more
template <int MODE>
__global__ void __launch_bounds__(NTHR, 2) paged_flash_kernel(PagedArgs a, int page_shift) {
  constexpr bool EXT = MODE == EXT_;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, l32 = lane & 31;
  const int per_head = gridDim.x / a.Hq;
  int hq, at;
  by_block(a.Hq, per_head, (int64_t)a.max_blocks * a.BS >= 4096, hq, at);
  const int w = per_head - 1 - at, hk = hq / (a.Hq / a.Hk);
  const int seq = __builtin_amdgcn_readfirstlane(a.work[2 * w]), qb = __builtin_amdgcn_readfirstlane(a.work[2 * w + 1]);
  const int t0 = __builtin_amdgcn_readfirstlane(a.cu_q[seq]), n = __builtin_amdgcn_readfirstlane(a.cu_q[seq + 1]) - t0;
  const int start = __builtin_amdgcn_readfirstlane(a.start[seq]), Skv = start + n;
  const int q0 = qb * BM, q0w = q0 + wid * 32;
  const int* bt = a.block_table + (int64_t)seq * a.max_blocks;
  const_int* pages = (const_int*)(uintptr_t)bt;
  const float slope = !EXT && a.alibi ? a.alibi[hq] * a.inv_scale : 0.f;

  bf16x8_t qf[8];
  {
    const bf16* qrow = a.q + (int64_t)(t0 + min(q0w + l32, n - 1)) * a.ldq + hq * FD + 8 * h;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) qf[kk] = *reinterpret_cast<const bf16x8_t*>(qrow + 16 * kk);
  }
  const int pos_lane = start + q0w + l32;            // this lane's query position
  const int wpos_lo = start + q0w, wpos_hi = start + q0w + 31;
  auto first_key = [&](int p) {                      // first key a position sees (non-decreasing in the position)
    int lo = EXT && a.chunk > 0 ? p / a.chunk * a.chunk : 0;
    if (a.window > 0) lo = max(lo, p - a.window + 1);
    return lo;
  };
  const int lo_lane = first_key(pos_lane), lo_whi = first_key(wpos_hi), lo_wlo = first_key(wpos_lo);
  const unsigned seen = (unsigned)(min(pos_lane, Skv - 1) - lo_lane);  // keys lo_lane .. lo_lane + seen
  const int kt1 = min((Skv + BN - 1) / BN, (start + min(q0 + BM, n) - 1) / BN + 1);
  const int kt0 = min(first_key(start + q0) / BN, kt1);

  // ------------------------------------------------------------------ tiles to LDS
  // Wave w moves the pieces w, w + 4, .. of K and of V, 4 rows of 256 bytes each: lane L of a piece lands at chunk L % 16 of
  // its row and fetches the chunk that the swizzle puts there. The row's low four bits do not depend on the piece.
  const int drow = 4 * wid + (lane >> 4);
  const int dch = (lane & 15) ^ (((drow & 3) << 2) | ((drow >> 2) & 3));
  const uint32_t voff = (uint32_t)(drow * FD + dch * 8) * 2;
  const int last_page = (Skv - 1) >> page_shift;
  int next[4];  // pages of the four 16-row groups of the tile that is fetched next
  auto look_up = [&](int tile) {
#pragma unroll
    for (int i = 0; i < 4; ++i) next[i] = pages[min((tile * BN + 16 * i) >> page_shift, last_page)];
  };
  const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const lds_char*)smem + 1024 * wid);
  const int pmask = a.BS - 1;
  const int64_t head = (int64_t)hk * a.BS, page = (int64_t)a.Hk * a.BS;
  auto dma_tile = [&](int tile, auto buf_c) {
    constexpr int buf = decltype(buf_c)::value;
    if (tile * BN + BN <= Skv) {
      auto piece = [&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        const int64_t off = (next[i] * page + head + ((tile * BN + 16 * i) & pmask)) * (FD * 2);
        dma16_s<buf * FTILE + 4096 * i>(reinterpret_cast<const char*>(a.kc) + off, voff, dst);
        dma16_s<(2 + buf) * FTILE + 4096 * i>(reinterpret_cast<const char*>(a.vc) + off, voff, dst);
      };
      piece(std::integral_constant<int, 0>{});
      piece(std::integral_constant<int, 1>{});
      piece(std::integral_constant<int, 2>{});
      piece(std::integral_constant<int, 3>{});
    } else {  // rows past the end repeat the last one (they are masked, and must be numbers)
      int64_t off[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = min(tile * BN + 16 * i + drow, Skv - 1);
        off[i] = (bt[key >> page_shift] * page + head + (key & pmask)) * FD + dch * 8;
      }
      auto piece = [&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        dma16<buf * FTILE + 4096 * i>(a.kc + off[i], dst);
        dma16<(2 + buf) * FTILE + 4096 * i>(a.vc + off[i], dst);
      };
      piece(std::integral_constant<int, 0>{});
      piece(std::integral_constant<int, 1>{});
      piece(std::integral_constant<int, 2>{});
      piece(std::integral_constant<int, 3>{});
    }
  };
  auto tile_barrier = [&]() { asm volatile("s_waitcnt vmcnt(0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  // ------------------------------------------------------------------ per-lane LDS addresses (see flash_fwd.hip)
  const lds_char* s3 = (const lds_char*)smem;
  float* scratch = reinterpret_cast<float*>(smem + 4 * FTILE) + wid * 32;
  const int gq = (lane >> 2) & 3, gch = (lane >> 1) & 1, gb = 8 * (lane & 1), colhalf = (lane >> 4) & 1;
  uint32_t kaddr[8], vaddr[2][4];
  {
    const int f = ((l32 & 3) << 2) | ((l32 >> 2) & 3);
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) kaddr[kk] = (uint32_t)(l32 * 256 + 16 * ((2 * kk + h) ^ f));
#pragma unroll
    for (int hi = 0; hi < 2; ++hi) {
      const int row = 4 * h + 8 * hi + gq, g = ((row & 3) << 2) | ((row >> 2) & 3);
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
        vaddr[hi][dt] = (uint32_t)(2 * FTILE + row * 256 + 16 * ((dt * 4 + colhalf * 2 + gch) ^ g) + gb);
    }
  }

  f32x16_t o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  const float rescale_thr = 8.f / a.c;  // in raw score units
  // a moderate cap bounds the scores: it serves as the maximum, and nothing is ever rescaled
  const bool fixed = EXT && a.cap_out > 0.f && a.cap_out <= 48.f;

  // the queries are the only loads that the compiler tracks: done before the first transfer, so that no wait of its own drains one
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) asm volatile("" : : "v"(qf[kk]));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (kt0 < kt1) {
    look_up(kt0);
    dma_tile(kt0, std::integral_constant<int, 0>{});
    look_up(kt0 + 1);
  }
  tile_barrier();

  auto tile_step = [&](int j, auto cur_c) {  // `cur`: the LDS buffer
    constexpr int cur = decltype(cur_c)::value;
    if (j + 1 < kt1) {
      dma_tile(j + 1, std::integral_constant<int, cur ^ 1>{});
      look_up(j + 2);
    }
    const int k0 = j * BN;
    if (q0w < n && k0 <= wpos_hi && k0 + BN - 1 >= lo_wlo) {
      // ---------------- S^T = K . Q^T, K read three products ahead
      auto ldk = [&](int i) {
        return *reinterpret_cast<const lds_bf16x8*>(s3 + kaddr[i & 7] + (cur * FTILE + (i >> 3) * 8192));
      };
      f32x16_t s[2];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[t][r] = 0.f;
      {
        bf16x8_t k0f = ldk(0), k1f = ldk(1), k2f = ldk(2);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          bf16x8_t k3f;
          if (i + 3 < 16) k3f = ldk(i + 3);
          __builtin_amdgcn_sched_barrier(0x6);
          s[i >> 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k0f, qf[i & 7], s[i >> 3], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0x6);
          k0f = k1f;
          k1f = k2f;
          k2f = k3f;
        }
      }
      // V operand i: 16 keys (t, ss) = i >> 2 of the column tile dt = i & 3; the first two fly under the softmax
      auto ldv = [&](int i) {
        const int dt = i & 3, disp = cur * FTILE + (i >> 2) * 16 * 256;
        const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(s3 + vaddr[0][dt] + disp));
        const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(s3 + vaddr[1][dt] + disp));
        s16x8 vv;
#pragma unroll
        for (int e = 0; e < 4; ++e) { vv[e] = lo[e]; vv[4 + e] = hi[e]; }
        return __builtin_bit_cast(bf16x8_t, vv);
      };
      bf16x8_t v0f = ldv(0), v1f = ldv(1);
      if constexpr (EXT) {
        if (a.cap_out > 0.f) {
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r)  // tanh z = 1 - 2 / (e^2z + 1); cap_in carries the 2 log2(e)
              s[t][r] = a.cap_out * (1.f - 2.f * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(s[t][r] * a.cap_in) + 1.f));
        }
      }
      // ---------------- ALiBi, causal diagonal, window, key tail (lane = one query row, r = 32 keys of the 64)
      if (!EXT && a.alibi) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            s[t][r] = fmaf(slope, (float)(k0 + t * 32 + (r & 3) + 8 * (r >> 2) + 4 * h - pos_lane), s[t][r]);
      }
      if (k0 + BN - 1 > wpos_lo || k0 < lo_whi || k0 + BN > Skv) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            if ((unsigned)(k0 - lo_lane + 4 * h + t * 32 + (r & 3) + 8 * (r >> 2)) > seen) s[t][r] = -INFINITY;
          }
      }
      // ---------------- online softmax; the reference maximum moves only past 2^8 (flash_fwd.hip)
      float m_new = m_run, m_use = 0.f, mc = a.cap_out;
      if (!fixed) {
        float m4[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
        for (int r = 0; r < 16; ++r) m4[r & 3] = fmax3(m4[r & 3], s[0][r], s[1][r]);
        float mx = fmax3(fmax3(m4[0], m4[1], m4[2]), m4[3], m4[3]);
        const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = fmax3(__uint_as_float(halves[0]), __uint_as_float(halves[1]), mx);
        m_new = mx > m_run + rescale_thr ? mx : m_run;
        m_use = m_new == -INFINITY ? 0.f : m_new;
        mc = m_use * a.c;
      }
      float psum = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = __builtin_amdgcn_exp2f(fmaf(s[t][r], a.c, -mc));
          s[t][r] = p;
          psum += p;
        }
      if (!fixed && !__all(m_new == m_run)) {
        const float alpha = __builtin_amdgcn_exp2f((m_run - m_use) * a.c);
        l_run *= alpha;
        m_run = m_new;
        if (lane < 32) scratch[lane] = alpha;
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        float a4[16];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(scratch + 8 * g + 4 * h);
#pragma unroll
          for (int i = 0; i < 4; ++i) a4[4 * g + i] = v[i];
        }
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[dt][r] *= a4[r];
        __builtin_amdgcn_wave_barrier();
      }
      l_run += psum;
      // ---------------- O += P . V, 16 keys at a time; EXT: weights as two bf16 terms, the second what the first leaves out
      bf16x8_t ph, pl;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if ((i & 3) == 0) {
          const int t = i >> 3, ss = (i >> 2) & 1;
          u32x4_t hi, lo;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x = s[t][8 * ss + 2 * e], y = s[t][8 * ss + 2 * e + 1];
            hi[e] = pack2(x, y);
            if constexpr (EXT)
              lo[e] = pack2(x - __uint_as_float(hi[e] << 16), y - __uint_as_float(hi[e] & 0xffff0000u));
          }
          ph = __builtin_bit_cast(bf16x8_t, hi);
          if constexpr (EXT) pl = __builtin_bit_cast(bf16x8_t, lo);
        }
        bf16x8_t v2f;
        if (i + 2 < 16) v2f = ldv(i + 2);
        __builtin_amdgcn_sched_barrier(0x6);
        o[i & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ph, v0f, o[i & 3], 0, 0, 0);
        if constexpr (EXT) o[i & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pl, v0f, o[i & 3], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0x6);
        v0f = v1f;
        v1f = v2f;
      }
    }
    tile_barrier();
  };
  for (int j = kt0; j < kt1; j += 2) {
    tile_step(j, std::integral_constant<int, 0>{});
    if (j + 1 < kt1) tile_step(j + 1, std::integral_constant<int, 1>{});
  }

  // ------------------------------------------------------------------ O / l, sink, gate
  const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if constexpr (EXT) {
    if (a.sink) {  // in the frame of the maximum the weights were taken in
      const float sk = a.sink[hq] * 1.4426950408889634f, m = fixed ? a.cap_out : m_run * a.c;
      const float mn = fmaxf(m, sk), f = __builtin_amdgcn_exp2f(m - mn);
      inv = f / fmaf(l_tot, f, __builtin_amdgcn_exp2f(sk - mn));
    }
    if (a.gate) inv /= 1.f + __expf(-(float)a.gate[(int64_t)(t0 + min(q0w + l32, n - 1)) * a.ldg + hq]);
  }
  if (lane < 32) scratch[lane] = inv;
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  float iv[16];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(scratch + 8 * g + 4 * h);
#pragma unroll
    for (int i = 0; i < 4; ++i) iv[4 * g + i] = v[i];
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int qi = q0w + (r & 3) + 8 * (r >> 2) + 4 * h;
    if (qi < n) {
      bf16* orow = a.o + (int64_t)(t0 + qi) * a.ldo + hq * FD + l32;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) orow[dt * 32] = (bf16)(o[dt][r] * iv[r]);
    }
  }
}

// Heads of 128 over pages whose size is a power of two of at least 16 tokens.
inline bool paged_flash_fits(const PagedArgs& a) { return a.dk == FD && a.dv == FD && a.BS >= 16 && (a.BS & (a.BS - 1)) == 0; }

template <int MODE>
int launch_flash(const PagedArgs& a, int nwork, hipStream_t st) {
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&paged_flash_kernel<MODE>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              FLDS);
    attr = true;
  }
  hipLaunchKernelGGL((paged_flash_kernel<MODE>), dim3(nwork * a.Hq), dim3(NTHR), FLDS, st, a, __builtin_ctz((unsigned)a.BS));
  DS_CHECK_LAUNCH();
  return 0;
}

}  // namespace
