// Products of mixture-of-experts layers, CDNA4 (gfx950). A pair (token, choice) is entry t * K + k: inputs are read from row
// entry / div, results written to row `entry`, so nothing is copied into expert order and back. The gated form computes
// silu(gate) up of the same columns in one go; a plain product may end in a squared relu.
//
//  * stream: few rows per expert. bf16 weights are streamed once per tile of up to 64 entries. A workgroup owns 32 weight rows
//    of an expert (gated: 16 of the gate and the same 16 of the up part); its four waves take alternating 64-wide steps of the
//    inner dimension straight into registers: no LDS, no barrier until the sums meet.
//    The entries of an expert come from sorted lists or, for a few hundred of them, are picked out of the routing table by
//    every workgroup itself; then only the experts that occur get workgroups.
//  * tile: many rows per expert. 128 entries x 256 weight rows (gated: 128 of either part) per workgroup. Weights are stored in
//    operand order and every wave has rows of its own, so they go from memory to registers in 512-byte runs, one step of 64
//    ahead; only the entries' rows pass through LDS (swizzled, two buffers). Two workgroups share a CU. Workgroups walk groups
//    of 4 column tiles by all row tiles of an expert, so that those at work on an XCD at a time share both operands in its L2.
//  * big tile: a hundred rows per expert or more. 256 entries x 256 weight rows per workgroup of 8 waves, both operands through LDS
//    by DMA (two buffers of 64 columns, 128 KB): see expert_big_kernel.
//  * any: a workgroup per entry and 64 columns; fp32 and widths that are no multiple of 8.
#include "ds_hip.h"

namespace {

constexpr int MAXE = 256, FEW = 512;

template <int N>
struct Int {
  static constexpr int value = N;
};

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.f + expf(-g)) * u; }
enum : int { NONE = 0, SILU_GLU = 1, RELU2 = 2 };  // activation codes
__device__ __forceinline__ float plain_act(float x, int act) {
  if (act != RELU2) return x;
  x = fmaxf(x, 0.f);
  return x * x;
}

struct ExpertArgs {
  const void* x;         // [.., K]
  const void* w;         // [E, N, K]; gated: [E, 2 N, K], gate rows first
  void* y;               // [entries, N]
  const int* experts;    // [entries]
  const int* offs;       // [E + 1] and
  const int* order;      // [entries], or null (up to FEW entries)
  int entries, E, N, K, div, act;
};

// Operand order of a weight matrix [rows, K] (ops/bf16_gemv.py): 16 x 64 tiles of 1024 elements, tile by tile along K;
// element [h][lane][j] of a tile is row lane % 16, column 16 (lane / 16) + 8 h + j

// The expert of this workgroup and its entries (list in LDS); their number, 0 for none. block-uniform.
__device__ __forceinline__ int collect(const ExpertArgs& a, int which, int* list, int* words, int& e) {
  const int tid = threadIdx.x, lane = tid & 63;
  if (tid < MAXE / 32) words[tid] = 0;
  __syncthreads();
  for (int i = tid; i < a.entries; i += 256) atomicOr((unsigned*)words + (a.experts[i] >> 5), 1u << (a.experts[i] & 31));
  __syncthreads();
  e = -1;
  int left = which;
#pragma unroll
  for (int i = 0; i < MAXE / 32; ++i) {  // the `which`-th expert that occurs
    unsigned m = words[i];
    const int c = __popc(m);
    if (e < 0 && left < c) {
      for (; left; --left) m &= m - 1;
      e = 32 * i + __ffs(m) - 1;
    }
    if (e < 0) left -= c;
  }
  if (e < 0) return 0;
  if (tid < 64) {  // one wave, in order
    int n = 0;
    for (int b = 0; b < a.entries; b += 64) {
      const bool hit = b + lane < a.entries && a.experts[min(b + lane, a.entries - 1)] == e;
      const unsigned long long m = __ballot(hit);
      if (hit) list[n + __popcll(m & ((1ull << lane) - 1))] = b + lane;
      n += __popcll(m);
    }
    if (lane == 0) words[MAXE / 32] = n;
  }
  __syncthreads();
  return words[MAXE / 32];
}

struct StreamShared {
  int list[FEW], words[MAXE / 32 + 1];
  f32x4 red[4][8][64];
};

// Entries m0 .. m0 + 16 MT - 1 of an expert, 32 weight rows (wp: this lane's row of either half)
template <int MT, bool GLU, bool SH>
__device__ __forceinline__ void stream_tile(const ExpertArgs& a, const bf16* const (&wp)[2], const int* ents, int cnt, int m0, int n0,
                                            StreamShared& sh) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, q4 = lane >> 4, N = a.N, K = a.K;
  const int wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const bf16* xp[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
    xp[m] = (const bf16*)a.x + (int64_t)(ents[min(m0 + 16 * m + l16, cnt - 1)] / a.div) * K + (SH ? 16 : 8) * q4;
  f32x4 acc[2][MT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[i][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  // U steps of 64 of the inner dimension: all their loads, then the products
  auto steps = [&](auto count, int k0, bool tail) {
    constexpr int U = decltype(count)::value;
    bf16x8 wv[U][2][2], xv[U][2][MT];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const int k = k0 + 256 * u + 32 * c, kc = tail ? min(k, K - 8 - 8 * q4) : k;
          const bf16* p = SH ? wp[i] + (int64_t)(k0 / 64 + 4 * u) * 1024 + 512 * c : wp[i] + kc;
          wv[u][c][i] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(p));
        }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int k = k0 + 256 * u + (SH ? 8 : 32) * c, kc = tail ? min(k, K - 8 - 8 * q4) : k;
#pragma unroll
        for (int m = 0; m < MT; ++m) xv[u][c][m] = *reinterpret_cast<const bf16x8*>(xp[m] + kc);
        if (tail && k + 8 * q4 >= K) {  // columns past the width count as zero, on both sides
#pragma unroll
          for (int j = 0; j < 8; ++j) {
#pragma unroll
            for (int i = 0; i < 2; ++i) wv[u][c][i][j] = (bf16)0.f;
#pragma unroll
            for (int m = 0; m < MT; ++m) xv[u][c][m][j] = (bf16)0.f;
          }
        }
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[i][m] = mfma(wv[u][c][i], xv[u][c][m], acc[i][m]);
  };
  constexpr int U = MT == 4 ? 2 : 4;
  const int whole = K / 64;
  int s = wid;
  for (; s + 4 * (U - 1) < whole; s += 4 * U) steps(Int<U>{}, 64 * s, false);
  for (; s < whole; s += 4) steps(Int<1>{}, 64 * s, false);
  if (!SH && K % 64 && whole % 4 == wid) steps(Int<1>{}, 64 * whole, true);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int m = 0; m < MT; ++m) sh.red[wid][i * MT + m][lane] = acc[i][m];
  __syncthreads();
  auto total = [&](int j) {
    f32x4 s = sh.red[0][j][lane];
#pragma unroll
    for (int v = 1; v < 4; ++v) s += sh.red[v][j][lane];
    return s;
  };
  // lane: entry l16 of a tile, weight rows 4 q4 .. + 3
  for (int j = wid; j < (GLU ? MT : 2 * MT); j += 4) {
    const int m = j % MT, r = m0 + 16 * m + l16, n = n0 + 4 * q4 + (j / MT) * 16;
    f32x4 v = total(j);
    if constexpr (GLU) {
      const f32x4 u = total(MT + j);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = silu_mul(v[i], u[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = plain_act(v[i], a.act);
    }
    if (r >= cnt) continue;
    bf16* yr = (bf16*)a.y + (int64_t)ents[r] * N + n;
    if (N % 4 == 0) {
      bf16x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = (bf16)v[i];
      if (n < N) *reinterpret_cast<bf16x4*>(yr) = o;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n + i < N) yr[i] = (bf16)v[i];
    }
  }
  __syncthreads();
}

template <bool GLU, bool SH>
__global__ void __launch_bounds__(256) expert_stream_kernel(ExpertArgs a) {
  __shared__ StreamShared sh;
  const int lane = threadIdx.x & 63, l16 = lane & 15, q4 = lane >> 4;
  int e = blockIdx.y, cnt;
  const int* ents = sh.list;
  if (a.offs) {
    cnt = a.offs[e + 1] - a.offs[e];
    ents = a.order + a.offs[e];
  } else {
    cnt = collect(a, blockIdx.y, sh.list, sh.words, e);
  }
  const int N = a.N, n0 = blockIdx.x * (GLU ? 16 : 32);
  if (cnt == 0) return;
  const bf16* w = (const bf16*)a.w + (int64_t)e * (GLU ? 2 : 1) * N * a.K;
  const bf16* wp[2];
  if constexpr (SH) {  // (16 divides N)
    wp[0] = w + (int64_t)n0 * a.K + lane * 8;
    wp[1] = GLU ? wp[0] + (int64_t)N * a.K : w + (int64_t)min(n0 + 16, N - 16) * a.K + lane * 8;
  } else {
    wp[0] = w + (int64_t)min(n0 + l16, N - 1) * a.K + 8 * q4;
    wp[1] = GLU ? wp[0] + (int64_t)N * a.K : w + (int64_t)min(n0 + 16 + l16, N - 1) * a.K + 8 * q4;
  }
  for (int m0 = 0; m0 < cnt;) {  // (uniform over the workgroup) as narrow as the rest allows
    const int left = cnt - m0;
    if (left <= 16) stream_tile<1, GLU, SH>(a, wp, ents, cnt, m0, n0, sh);
    else if (left <= 32) stream_tile<2, GLU, SH>(a, wp, ents, cnt, m0, n0, sh);
    else stream_tile<4, GLU, SH>(a, wp, ents, cnt, m0, n0, sh);
    m0 += left <= 16 ? 16 : left <= 32 ? 32 : 64;
  }
}

// ------------------------------------------------------------------------------------------------ many rows per expert
constexpr int BM = 128, BN = 256, GROUP = 4;

struct Place {
  int pre[MAXE + 1], offs[MAXE + 1], found;
};
// Row tiles (of TM entries) of all experts laid end to end; this workgroup's place among them: expert, first entry, first column.
// false: there is nothing for it. block-uniform.
template <int TM, int GROUPS>
__device__ __forceinline__ bool place_of(const ExpertArgs& a, Place& pl, int per, int& e, int& m0, int& n0) {
  const int tid = threadIdx.x, lane = tid & 63, threads = blockDim.x, nt = (a.N + per - 1) / per;
  for (int i = tid; i <= a.E; i += threads) pl.offs[i] = a.offs[i];
  __syncthreads();
  if (tid < 64) {
    int c[4], s = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int x = 4 * lane + i;
      c[i] = x < a.E ? (pl.offs[x + 1] - pl.offs[x] + TM - 1) / TM : 0;
      s += c[i];
    }
    int run = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(run, o, 64);
      if (lane >= o) run += y;
    }
    int at = run - s;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (4 * lane + i < a.E) pl.pre[4 * lane + i] = at;
      at += c[i];
    }
    if (lane == 63) pl.pre[a.E] = run;
  }
  __syncthreads();
  const int total = pl.pre[a.E] * nt;
  if ((int)blockIdx.x >= total) return false;
  const int id = xcd_remap(blockIdx.x, total);
  for (int x = tid; x < a.E; x += threads)
    if (pl.pre[x] * nt <= id && id < pl.pre[x + 1] * nt) pl.found = x;
  __syncthreads();
  e = pl.found;
  const int mt = pl.pre[e + 1] - pl.pre[e], local = id - pl.pre[e] * nt, g = local / (mt * GROUPS);
  const int rest = local - g * mt * GROUPS, width = min(GROUPS, nt - g * GROUPS);
  m0 = rest / width * TM;
  n0 = (g * GROUPS + rest % width) * per;
  return true;
}

template <bool GLU>
__global__ void __launch_bounds__(256, 2) expert_tile_kernel(ExpertArgs a) {
  __shared__ __attribute__((aligned(16))) bf16 xs[2][BM * 64];
  __shared__ Place pl;
  __shared__ int ents[BM];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = a.N, K = a.K, KQ = K / 64;
  int e, m0, n0;
  if (!place_of<BM, GROUP>(a, pl, GLU ? BN / 2 : BN, e, m0, n0)) return;
  const int left = min(BM, pl.offs[e + 1] - pl.offs[e] - m0);
  if (tid < BM) ents[tid] = a.order[pl.offs[e] + m0 + min(tid, left - 1)];
  __syncthreads();
  // ---- entries' rows on their way to LDS: 8 rows of 8 pieces per wave and access, piece p of row r holding columns
  // 8 (p ^ (r / 2 % 8)) .. + 7
  const bf16* xp[4];
  int xo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = wid * 32 + i * 8 + (lane >> 3), p = lane & 7;
    xp[i] = (const bf16*)a.x + (int64_t)(ents[r] / a.div) * K + 8 * (p ^ ((r >> 1) & 7));
    xo[i] = r * 64 + p * 8;
  }
  // ---- this wave's 2 x 32 weight rows: gate and up of the same columns, or 64 neighbours
  const bf16* wp[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int row = GLU ? min(n0 + wid * 32, N - 32) + t * N : min(n0 + wid * 64 + 32 * t, N - 32);
    wp[t] = (const bf16*)a.w + ((int64_t)e * (GLU ? 2 : 1) * N + row + (l32 & 16)) * K + (hh * 16 + (l32 & 15)) * 8;
  }
  bf16x8 xr[4], wa[2][2][2], wb[2][2][2];  // [t][h][j]: columns 16 (2 j + hh) + 8 h .. + 7 of the step
  f32x16 acc[2][4];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][m][r] = 0.f;
  auto load_x = [&](int kq) {
#pragma unroll
    for (int i = 0; i < 4; ++i) xr[i] = *reinterpret_cast<const bf16x8*>(xp[i] + kq * 64);
  };
  auto load_w = [&](bf16x8 (&w)[2][2][2], int kq) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          w[t][h][j] = *reinterpret_cast<const bf16x8*>(wp[t] + (int64_t)kq * 1024 + h * 512 + j * 256);
  };
  auto store_x = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<bf16x8*>(&xs[buf][xo[i]]) = xr[i];
  };
  const int tiles = (left + 31) / 32, sw = (l32 >> 1) & 7;
  auto compute = [&](const bf16x8 (&w)[2][2][2], int buf) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          if (m >= tiles) break;  // (the branch also keeps the operands of later steps out of the registers)
          const bf16x8 x = *reinterpret_cast<const bf16x8*>(&xs[buf][(32 * m + l32) * 64 + 8 * ((4 * j + 2 * hh + h) ^ sw)]);
#pragma unroll
          for (int t = 0; t < 2; ++t) acc[t][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[t][h][j], x, acc[t][m], 0, 0, 0);
        }
  };
  load_w(wa, 0);
  load_x(0);
  store_x(0);
  __syncthreads();
  for (int kq = 0; kq < KQ; kq += 2) {
    if (kq + 1 < KQ) {
      load_x(kq + 1);
      load_w(wb, kq + 1);
    }
    compute(wa, 0);
    if (kq + 1 >= KQ) break;
    store_x(1);
    __syncthreads();
    if (kq + 2 < KQ) {
      load_x(kq + 2);
      load_w(wa, kq + 2);
    }
    compute(wb, 1);
    if (kq + 2 < KQ) store_x(0);
    __syncthreads();
  }
  // lane: entry l32 of a tile, weight rows 8 q + 4 hh + 0..3
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int r = 32 * m + l32;
    if (r >= left) continue;
    bf16* yr = (bf16*)a.y + (int64_t)ents[r] * N;
#pragma unroll
    for (int t = 0; t < (GLU ? 1 : 2); ++t) {
      const int n = GLU ? n0 + wid * 32 : n0 + wid * 64 + 32 * t;
      if (n >= N) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        bf16x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[i] = (bf16)(GLU ? silu_mul(acc[0][m][4 * q + i], acc[1][m][4 * q + i]) : plain_act(acc[t][m][4 * q + i], a.act));
        *reinterpret_cast<bf16x4*>(yr + n + 8 * q + 4 * hh) = o;
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------ hundreds of rows per expert
// What bounds the tile kernel above is traffic into the CU: for each step of 64 columns its two workgroups take 2 x (128 + 256)
// rows, 48 bytes a clock at the full matrix rate. One tile of 256 x 256 takes 32, all of it by DMA, without registers. Eight
// waves, 64 weight rows (gated: 32 of either part) x 128 entries each: two on a SIMD, so that one has products to issue while the
// other's transfers wait to be taken (four waves of 128 x 128, with a third less to read from LDS: 1.08 times the time). The
// barrier comes ahead of a step's last quarter, whose operands are in registers by then, and the next step's first reads right
// behind it; transfers are issued a quarter at a time, between products. Rows come swizzled (the source address carries it),
// weights in operand order: reads without bank conflicts. Workgroups walk groups of 8 column tiles by all row tiles of an expert.
// 32 experts, 1024 rows each on average: 3584 gated columns of 4096: 2180 -> 1790 us (1076 TFLOP/s; a third of the requests
// miss the L2, the matrix cores are busy 55 % of the time); 4096 plain columns of 3584: 1115 -> 950 us.
constexpr int TM = 256, TN = 256, BIG_BUF = (TM + TN) * 128, BIG_LDS = 2 * BIG_BUF;
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;

// 16 bytes per lane from global memory to LDS byte `dst` + OFF + 16 * lane. Inline asm: hipcc waits for its own such loads before
// every LDS read that it cannot prove apart from them.
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
__device__ __forceinline__ void dma16_s(const void* base, uint32_t voff, uint32_t dst) {  // wave-uniform base, offset per lane
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_add_u32 m0, %3, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\t"
               "s_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(voff), "s"(base), "s"(dst), "n"(OFF)
               : "memory", "scc");
}

template <bool GLU, int NW>
__global__ void __launch_bounds__(NW * 64, NW / 4) expert_big_kernel(ExpertArgs a) {
  constexpr int NP = 16 / NW, WT = 16 / NW, XP = 32 / NW;  // weight parts of 32 rows; weight tiles and rows' pieces moved per wave
  extern __shared__ __attribute__((aligned(16))) char smem[];  // [2][256 rows x 64 | 16 weight tiles of 16 x 64]
  __shared__ Place pl;
  __shared__ int ents[TM];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), wc = wid % (NW / 2), wr = wid / (NW / 2);
  const int N = a.N, K = a.K, KQ = K / 64;
  int e, m0, n0;
  if (!place_of<TM, 8>(a, pl, GLU ? TN / 2 : TN, e, m0, n0)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  m0 = __builtin_amdgcn_readfirstlane(m0);
  n0 = __builtin_amdgcn_readfirstlane(n0);
  const int left = min(TM, __builtin_amdgcn_readfirstlane(pl.offs[e + 1] - pl.offs[e]) - m0);
  if (tid < TM) ents[tid] = a.order[pl.offs[e] + m0 + min(tid, left - 1)];
  __syncthreads();
  // ---- what this wave moves per step: pieces of 8 entries' rows (piece p of row r: columns 8 (p ^ (r / 2 % 8)) .. + 7) and
  // weight tiles, a piece per half
  const bf16* xp[XP];
  const bf16* wp[WT];
#pragma unroll
  for (int i = 0; i < XP; ++i) {
    const int r = wid * 8 * XP + i * 8 + (lane >> 3);
    xp[i] = (const bf16*)a.x + (int64_t)(ents[r] / a.div) * K + 8 * ((lane & 7) ^ ((r >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < WT; ++i) {
    const int t = WT * wid + i, row = GLU ? min(n0 + 16 * (t & 7), N - 16) + (t >> 3) * N : min(n0 + 16 * t, N - 16);
    wp[i] = (const bf16*)a.w + ((int64_t)e * (GLU ? 2 : 1) * N + row) * K;
  }
  // the entries are the loads that the compiler tracks: done before the first transfer
#pragma unroll
  for (int i = 0; i < XP; ++i) asm volatile("" : "+v"(xp[i]));
  const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const lds_char*)smem + 1024 * XP * wid);
  // piece p of 2 XP of step kq: the first half entries' rows, the others weight tiles
  auto move = [&](int kq, auto buf_c, auto p_c) {
    constexpr int B = decltype(buf_c)::value * BIG_BUF, p = decltype(p_c)::value;
    if constexpr (p < XP) dma16<B + 1024 * p>(xp[p] + (int64_t)kq * 64, dst);
    else dma16_s<B + TM * 128 + 1024 * (p - XP)>(wp[(p - XP) / 2] + (int64_t)kq * 1024 + (p & 1) * 512, lane * 16, dst);
  };
  auto settle = [&]() { asm volatile("s_waitcnt vmcnt(0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  // ---- operand reads: entry 128 wr + 32 m + l32, row l32 of weight part t; step (h, j): columns 16 (2 j + hh) + 8 h .. + 7 of
  // either
  const lds_char* s3 = (const lds_char*)smem;
  uint32_t xa[4], wa;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int h = i >> 1, j = i & 1;
    xa[i] = (uint32_t)((128 * wr + l32) * 128 + 16 * ((4 * j + 2 * hh + h) ^ ((l32 >> 1) & 7)));
  }
  wa = (uint32_t)(TM * 128 + ((GLU ? 1 : 2) * NP * wc + (l32 >> 4)) * 2048 + hh * 256 + (l32 & 15) * 16);
  f32x16 acc[NP][4];  // [weight part][entries]; GLU: the first half gate, the others up
#pragma unroll
  for (int t = 0; t < NP; ++t)
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][m][r] = 0.f;

  auto all = [&](int kq, auto buf_c, auto from, auto to, auto&& self) {
    if constexpr (decltype(from)::value < decltype(to)::value) {
      move(kq, buf_c, from);
      self(kq, buf_c, Int<decltype(from)::value + 1>{}, to, self);
    }
  };
  all(0, Int<0>{}, Int<0>{}, Int<2 * XP>{}, all);
  settle();
  if (KQ > 1) all(1, Int<1>{}, Int<0>{}, Int<XP>{}, all);
  // MT: 32-entry tiles that this wave has (every wave passes the same barriers)
  auto sweep = [&](auto mt_c) {
    constexpr int MT = decltype(mt_c)::value;
    bf16x8 w0[NP], x0[4], w1[NP], x1[4];
    auto read_w = [&](int i, int t, auto buf_c) {
      const int tile = GLU ? (t % (NP / 2)) * 2 + t / (NP / 2) * 8 : 2 * t;
      return *reinterpret_cast<const lds_bf16x8*>(
          s3 + wa + (decltype(buf_c)::value * BIG_BUF + tile * 2048 + (i >> 1) * 1024 + (i & 1) * 512));
    };
    auto read_x = [&](int i, int m, auto buf_c) {
      return *reinterpret_cast<const lds_bf16x8*>(s3 + xa[i] + (decltype(buf_c)::value * BIG_BUF + m * 4096));
    };
    // four columns steps of 16, in quarters; the next one's operands are read and pieces of a later step are
    // moved between the quarters (a run of transfers would hold the wave, and with it its products, until they are taken)
    auto part = [&](int kq, auto buf_c, auto i_c) {
      constexpr int buf = decltype(buf_c)::value, i = decltype(i_c)::value, ni = (i + 1) & 3;
      const bool more = i < 3 || kq + 1 < KQ;
      if (i == 3 && more) settle();  // the next step has come, and nobody reads this one any more
      auto quarter = [&](auto q_c) {
        constexpr int q = decltype(q_c)::value;
        if constexpr (MT > 0) {
          if (more) {
            using Next = Int<i == 3 ? buf ^ 1 : buf>;
            if constexpr (q < 2) {
#pragma unroll
              for (int t = q * NP / 2; t < (q + 1) * NP / 2; ++t) w1[t] = read_w(ni, t, Next{});
              if (q < MT) x1[q] = read_x(ni, q, Next{});
            } else if constexpr (q == 2) {
              if (2 < MT) x1[2] = read_x(ni, 2, Next{});
              if (3 < MT) x1[3] = read_x(ni, 3, Next{});
            }
          }
        }
        constexpr int some = XP / 4;  // pieces per quarter
        if constexpr (i == 3) {
          if (kq + 2 < KQ) all(kq + 2, buf_c, Int<some * q>{}, Int<some * (q + 1)>{}, all);
        } else if constexpr (i == 0) {
          if (kq + 1 < KQ) all(kq + 1, Int<buf ^ 1>{}, Int<XP + some * q>{}, Int<XP + some * (q + 1)>{}, all);
        }
        __builtin_amdgcn_sched_barrier(0x6);
        if constexpr (q < MT) {
#pragma unroll
          for (int t = 0; t < NP; ++t) acc[t][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w0[t], x0[q], acc[t][q], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0x6);
      };
      quarter(Int<0>{});
      quarter(Int<1>{});
      quarter(Int<2>{});
      quarter(Int<3>{});
#pragma unroll
      for (int t = 0; t < NP; ++t) w0[t] = w1[t];
#pragma unroll
      for (int m = 0; m < 4; ++m) x0[m] = x1[m];
    };
    if constexpr (MT > 0) {
#pragma unroll
      for (int t = 0; t < NP; ++t) w0[t] = read_w(0, t, Int<0>{});
#pragma unroll
      for (int m = 0; m < MT; ++m) x0[m] = read_x(0, m, Int<0>{});
    }
    auto step = [&](int kq, auto buf_c) {
      part(kq, buf_c, Int<0>{});
      part(kq, buf_c, Int<1>{});
      part(kq, buf_c, Int<2>{});
      part(kq, buf_c, Int<3>{});
    };
    for (int kq = 0; kq < KQ; kq += 2) {
      step(kq, Int<0>{});
      if (kq + 1 < KQ) step(kq + 1, Int<1>{});
    }
  };
  const int tiles = min(max((left - 128 * wr + 31) / 32, 0), 4);
  if (tiles == 4) sweep(Int<4>{});
  else if (tiles == 3) sweep(Int<3>{});
  else if (tiles == 2) sweep(Int<2>{});
  else if (tiles == 1) sweep(Int<1>{});
  else sweep(Int<0>{});
  // lane: entry l32 of a tile, weight rows 8 q + 4 hh + 0..3
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int r = 128 * wr + 32 * m + l32;
    if (r >= left) continue;
    bf16* yr = (bf16*)a.y + (int64_t)ents[r] * N;
#pragma unroll
    for (int t = 0; t < (GLU ? NP / 2 : NP); ++t) {
      const int n = n0 + (GLU ? 16 : 32) * NP * wc + 32 * t;
      if (n >= N) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        bf16x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[i] = (bf16)(GLU ? silu_mul(acc[t][m][4 * q + i], acc[t + (GLU ? NP / 2 : 0)][m][4 * q + i]) : plain_act(acc[t][m][4 * q + i], a.act));
        *reinterpret_cast<bf16x4*>(yr + n + 8 * q + 4 * hh) = o;
      }
    }
  }
}

template <typename T, bool GLU>
__global__ void __launch_bounds__(256) expert_any_kernel(ExpertArgs a) {
  const int64_t i = blockIdx.x;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, e = a.experts[i], K = a.K;
  const T* x = (const T*)a.x + i / a.div * K;
  const T* w = (const T*)a.w + (int64_t)e * (GLU ? 2 : 1) * a.N * K;
  for (int n = blockIdx.y * 64 + wid; n < min(a.N, (int)blockIdx.y * 64 + 64); n += 4) {
    const T *wr = w + (int64_t)n * K, *ur = wr + (GLU ? (int64_t)a.N * K : 0);
    float s = 0.f, u = 0.f;
    for (int c = lane; c < K; c += 64) {
      const float xv = (float)x[c];
      s = fmaf(xv, (float)wr[c], s);
      if constexpr (GLU) u = fmaf(xv, (float)ur[c], u);
    }
    s = wave_sum(s);
    if constexpr (GLU) s = silu_mul(s, wave_sum(u));
    else s = plain_act(s, a.act);
    if (lane == 0) ((T*)a.y)[i * a.N + n] = (T)s;
  }
}

// out[t] = sum_k w[t, k] y[row(t, k)] (+ base[t])
template <typename T>
__global__ void __launch_bounds__(256) expert_sum_kernel(const T* __restrict__ y, const float* __restrict__ w,
                                                         const int* __restrict__ rows, const T* __restrict__ base,
                                                         T* __restrict__ out, int W, int K) {
  const int64_t t = blockIdx.x;
  for (int c = threadIdx.x; c < W; c += 256) {
    float v = 0.f;
    for (int k = 0; k < K; ++k) v = fmaf(w[t * K + k], (float)y[(rows ? rows[t * K + k] : t * K + k) * W + c], v);
    out[t * W + c] = (T)(base ? v + (float)base[t * W + c] : v);
  }
}

// Rows per expert on average from which 256-row tiles pay. Measured against the tile kernel, us, gated / plain: 32 experts of 3584
// by 4096, 96 rows 387 -> 429 / 187 -> 211, 128 rows 583 -> 452 / 295 -> 225, 256 rows 783 -> 645 / 392 -> 317; 32 of 1408 by 2048,
// 96 rows 82 -> 108 / 46 -> 36, 128 rows 129 -> 109 / 55 -> 38; 8 of 3584 by 4096, 128 rows 151 -> 111 / 90 -> 82.
constexpr int BIG_ROWS = 128, BIG_WAVES = 8;

template <bool GLU>
int launch_big(const ExpertArgs& a, int per, hipStream_t st) {  // per: columns of a tile
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&expert_big_kernel<GLU, BIG_WAVES>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              BIG_LDS);
    attr = true;
  }
  const int64_t grid = ((int64_t)a.entries / TM + a.E) * ((a.N + per - 1) / per);
  hipLaunchKernelGGL((expert_big_kernel<GLU, BIG_WAVES>), dim3((unsigned)grid), dim3(BIG_WAVES * 64), BIG_LDS, st, a);
  DS_CHECK_LAUNCH();
  return 0;
}

}  // namespace

extern "C" int ds_expert_few() { return FEW; }
extern "C" int ds_expert_order_ok(int N, int K) { return N % 32 == 0 && K % 64 == 0; }

// y[i] = w[experts[i]] x[i / div] for every entry; act SILU_GLU: silu of the first N rows times the others; RELU2: max(., 0)^2. offs and order from
// ds_expert_place, or null for up to ds_expert_few() entries. operand: the weights are in operand order (N % 32, K % 64 must
// be 0); then with lists and `tile` the many-rows kernel runs.
extern "C" int ds_expert_gemm(const void* x, const void* w, void* y, const int* experts, const int* offs, const int* order,
                              int entries, int E, int N, int K, int div, int act, int operand, int tile, int dtype,
                              hipStream_t st) {
  if (entries <= 0) return 0;
  if (E <= 0 || E > MAXE || N <= 0 || K <= 0 || div <= 0 || (!offs != !order) || (N + 63) / 64 > 65535)
    return (int)hipErrorInvalidValue;
  const bool lists = offs != nullptr, gated = act == SILU_GLU;
  if (operand && (dtype != DS_BF16 || !ds_expert_order_ok(N, K) || (!lists && entries > FEW))) return (int)hipErrorInvalidValue;
  const ExpertArgs a{x, w, y, experts, offs, order, entries, E, N, K, div, act};
  if (operand && lists && tile) {
    const int per = gated ? BN / 2 : BN;
    const int64_t grid = ((int64_t)entries / BM + E) * ((N + per - 1) / per);
    if (grid > INT32_MAX) return (int)hipErrorInvalidValue;
    if (entries >= (int64_t)BIG_ROWS * E) return gated ? launch_big<true>(a, per, st) : launch_big<false>(a, per, st);
    if (gated) hipLaunchKernelGGL(expert_tile_kernel<true>, dim3((unsigned)grid), dim3(256), 0, st, a);
    else hipLaunchKernelGGL(expert_tile_kernel<false>, dim3((unsigned)grid), dim3(256), 0, st, a);
    DS_CHECK_LAUNCH();
    return 0;
  }
  if (operand || (dtype == DS_BF16 && K % 8 == 0 && (lists || entries <= FEW))) {
    const dim3 grid((N + (gated ? 15 : 31)) / (gated ? 16 : 32), lists ? E : (entries < E ? entries : E));
#define GO(SH)                                                                                              \
  {                                                                                                         \
    if (gated) hipLaunchKernelGGL((expert_stream_kernel<true, SH>), grid, dim3(256), 0, st, a);             \
    else hipLaunchKernelGGL((expert_stream_kernel<false, SH>), grid, dim3(256), 0, st, a);                  \
  }
    if (operand) GO(true)
    else GO(false)
#undef GO
    DS_CHECK_LAUNCH();
    return 0;
  }
  const dim3 grid(entries, (N + 63) / 64);
#define GO(T)                                                                                       \
  {                                                                                                 \
    if (gated) hipLaunchKernelGGL((expert_any_kernel<T, true>), grid, dim3(256), 0, st, a);         \
    else hipLaunchKernelGGL((expert_any_kernel<T, false>), grid, dim3(256), 0, st, a);              \
  }
  if (dtype == DS_F32) GO(float)
  else if (dtype == DS_BF16) GO(bf16)
  else return (int)hipErrorInvalidValue;
#undef GO
  DS_CHECK_LAUNCH();
  return 0;
}

extern "C" int ds_expert_sum(const void* y, const float* w, const int* rows, const void* base, void* out, int T, int W, int K, int dtype,
                             hipStream_t st) {
  if (T <= 0) return 0;
  if (W <= 0 || K <= 0) return (int)hipErrorInvalidValue;
  if (dtype == DS_F32)
    hipLaunchKernelGGL(expert_sum_kernel<float>, dim3(T), dim3(256), 0, st, (const float*)y, w, rows,
                       (const float*)base, (float*)out, W, K);
  else if (dtype == DS_BF16)
    hipLaunchKernelGGL(expert_sum_kernel<bf16>, dim3(T), dim3(256), 0, st, (const bf16*)y, w, rows,
                       (const bf16*)base, (bf16*)out, W, K);
  else return (int)hipErrorInvalidValue;
  DS_CHECK_LAUNCH();
  return 0;
}
