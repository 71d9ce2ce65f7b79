// Block-sparse attention backward, CDNA4 (gfx950), bf16, head dim 128 (reference: the transposed DSD / SDD products of
// `deepspeed/ops/sparse_attention/matmul.py:605` and the sparse softmax backward of `softmax.py:213`). No probability is stored: P
// comes back from the forward's natural-log LSE.
//
// Two passes over the layout, one by rows for dQ and one by columns for dK and dV, so that every sum stays in the registers of
// one workgroup. A single pass needs five products instead of seven, but adds a 16 KB piece of dQ to memory for every 32 query
// rows that a block of keys meets, and a layout of short rows makes that all of its time: the atomic units retire 1.3 TB/s.
// B2 H8 S16384, BigBird of 64-key blocks with padding, us, of a whole backward: 519 in one pass (438, and 81 for the row
// sums, the zeroes and the conversion that it needs around it) -> 372 (rows 165, columns 197, merge 10). In the loop both
// passes use LDS (four waves' operands, 128 bytes a clock) to two thirds and the matrix cores to half; a workgroup of the
// shortest lists is as long in its first loads and its last stores as in its five pairs of steps.
//
//  * rows: 4 waves, 64 query rows; two waves have 32 rows each, with Q and dO in registers, and go through every other step
//    of 32 keys, the other two have the same rows and the steps between. S^T = K Q^T and dP^T = V dO^T put a query on each
//    lane, its row constants -LSE / scale and -delta are the accumulators' initial values, and dS is the next product's
//    operand as it stands: dQ += dS K, K by transposed reads of the same image. delta = sum(dO O) is computed here, from
//    the rows that are in registers anyway, and left for the other pass.
//  * columns, the mirror image: 64 keys, 32 per wave with V and half of K in registers and the other half of K in LDS (all of it
//    would be 16 registers too many); Q and dO come in steps of 32 rows; key on the lane, dV^T += dO^T P, dK^T += Q^T dS.
//  * blocks of 64 because layouts are made of blocks about that size: with 128 keys a workgroup (four waves on one step)
//    a third of the waves had nothing to do at a step, and in layouts with every fourth column dense, the same half of them
//    throughout. The two that share rows (keys) add their sums up through LDS at the end.
//  * steps arrive by LDS-DMA, a pair ahead of the one in use, one barrier a pair. Two workgroups share a CU. A list of
//    tiles and masks is read once, a tile per thread, and what the workgroup has to do with is kept in LDS: in the loop a
//    load that the compiler sees would wait for the transfers too.
//  * lists that the plan cut leave fp32 sums in a workspace; a third launch adds them in order.
#include "ds_hip.h"

#include <cstddef>
#include <type_traits>

namespace {

constexpr int D = 128, STEP = 32, OWN = 64, NTHR = 256;   // OWN: rows (keys) of a workgroup
constexpr int ROWS = 128, KEYS = 256;  // blocks of the plan
constexpr int PIECE = STEP * D * 2;   // 8 KB: 32 rows of one operand
constexpr int STAGE = 2 * PIECE;
constexpr int LIST = 512;             // steps listed at a time
constexpr float LOG2E = 1.4426950408889634f;

typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;

// LDS-DMA, 16 (4) bytes a lane to lds_base + 16 (4) * lane. In asm because hipcc waits for its own such loads before every LDS
// read; out of its sight they are ordered by the counted waits below.
__device__ __forceinline__ uint32_t lds_at(const char* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const lds_char*)p);
}
__device__ __forceinline__ void glds16_s(const void* base, uint32_t voff, uint32_t dst) {  // wave-uniform base, bytes per lane
  const uint64_t sb = (uint64_t)(uintptr_t)base;
  const uint64_t ub = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(sb >> 32)) << 32) |
                      (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)sb);
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\t"
               "s_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(voff), "s"(ub), "s"(dst)
               : "memory");
}
__device__ __forceinline__ void glds4_s(const void* base, uint32_t voff, uint32_t dst) {
  const uint64_t sb = (uint64_t)(uintptr_t)base;
  const uint64_t ub = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(sb >> 32)) << 32) |
                      (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)sb);
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2\n\t"
               "s_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(voff), "s"(ub), "s"(dst)
               : "memory");
}
// the lane, anew: what is worked out from it in a loop is not kept in registers over the loop
__device__ __forceinline__ int lane_now() {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));
  return lane;
}
// this wave's transfers have landed and its LDS work is done; then the barrier
__device__ __forceinline__ void settle() { asm volatile("s_waitcnt vmcnt(0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// LDS work is done; then the barrier. Unlike __syncthreads it waits for no load.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Round to nearest even, lo in bits 0..15: one v_cvt_pk_bf16_f32. Not in asm: a swap of the wave's halves stands two wait states
// behind what writes its operands, and hipcc sees to that where it sees the writer.
__device__ __forceinline__ unsigned pack_bf16(float lo, float hi) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2));
}
__device__ __forceinline__ bf16x8 pack8(const f32x16& x, int at) {
  u32x4_t u;
#pragma unroll
  for (int i = 0; i < 4; ++i) u[i] = pack_bf16(x[at + 2 * i], x[at + 2 * i + 1]);
  return __builtin_bit_cast(bf16x8, u);
}
__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

// 256-byte rows of sixteen 16-byte chunks, chunk XOR a bijection of the row mod 16: row reads of one chunk and transposed reads
// of four rows both touch distinct banks
__device__ __forceinline__ int swz(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }
__device__ __forceinline__ s16x4_t tr_read(const lds_char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
}
__device__ __forceinline__ bf16x8 join(s16x4_t lo, s16x4_t hi) {
  s16x8 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) { v[e] = lo[e]; v[4 + e] = hi[e]; }
  return __builtin_bit_cast(bf16x8, v);
}
__device__ __forceinline__ int crow(int r, int h) { return (r & 3) + 8 * (r >> 2) + 4 * h; }  // row of accumulator register r

typedef __attribute__((address_space(4))) const int const_int;  // wave-uniform and read-only: scalar loads
__device__ __forceinline__ const_int* uniform_ints(const int* p) { return (const_int*)(uintptr_t)p; }

// A side of the plan. Lists tiles, masks [heads, blocks, max_tiles] by blocks of 128 rows (64-key tiles; bit 4 r + k of a mask: rows
// 16 r .. see keys 16 k ..) or of 256 keys (32-row tiles; bit 16 r + k). Shares work [heads, nwork, 4] = (block of 64 rows or keys, or
// -1; first entry of its list, entries, part slot or -1) longest first, merges [heads, nmerge, 4] = (block of 64 or -1, first slot,
// slots, 0); part [B H or, with lists per head, B, nslots, 64 rows or 2 x 64 keys, 128].
struct Side {
  const int *tiles, *masks, *work, *merges;
  int max_tiles, heads, nwork, nmerge, nslots;
  float* part;
};
struct SparseBwdArgs {
  const bf16 *q, *k, *v, *o, *dout;
  bf16 *dq, *dk, *dv;
  const float* lse;  // [B, H, S]
  float* nrow;       // [B, H, S / 32, 2, 32]: -delta, -LSE / scale
  int B, H, S;
  int64_t qs[3], ks[3], vs[3], os[3], gs[3], dqs[3], dks[3], dvs[3];  // (batch, head, row) in elements
  float scale;
  Side rows, cols;
  const float *kbias, *abias, *rpe;
  int64_t kb_stride, ab_stride, rpe_hs, rpe_rs;
};

// Workgroup -> (batch and head, entry of its work). An XCD has heads of its own, whose operands meet in its L2, and takes the
// longest entries of all of them first.
__device__ __forceinline__ void place(int nwork, int heads, int& bh, int& wi) {
  if (heads % 8 == 0) {
    const int per = heads / 8, at = blockIdx.x / 8;
    bh = blockIdx.x % 8 * per + at % per;
    wi = at / per;
  } else {
    const int at = xcd_remap(blockIdx.x, gridDim.x);
    bh = at / nwork;
    wi = at % nwork;
  }
}

struct Lists {
  int step[LIST], mask[LIST], counts[NTHR / 64];
};
// Entries that this workgroup has something to do with, packed in order: each thread brings up to two (those with a mask). Their
// number. Nobody may still be reading the list before.
__device__ __forceinline__ int pack_list(Lists& ls, const int (&step)[2], const int (&mask)[2]) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const unsigned long long one = __ballot(mask[0] != 0), two = __ballot(mask[1] != 0), below = (1ull << lane) - 1;
  if (lane == 0) ls.counts[wid] = __popcll(one) + __popcll(two);
  lds_barrier();
  int at = 0, all = 0;
#pragma unroll
  for (int i = 0; i < NTHR / 64; ++i) {
    if (i < wid) at += ls.counts[i];
    all += ls.counts[i];
  }
  at += __popcll(one & below) + __popcll(two & below);
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (mask[i] != 0) {
      ls.step[at] = step[i];
      ls.mask[at++] = mask[i];
    }
  lds_barrier();
  return __builtin_amdgcn_readfirstlane(all);
}

// LDS of either kernel: two pairs of steps (a pair: one for each half of the waves, each two operands of 32 rows); at the end the
// waves' sums on their way to each other
struct Shared {
  char ring[2][2][STAGE];
  char kimg[OWN * 128];      // columns: columns 64 .. 127 of the keys, 128-byte rows of 8 chunks
  float extra[2][2][64];     // rows: the keys' biases; columns: -delta and -LSE / scale of the rows
  Lists ls;
};
static_assert(sizeof(Shared) <= 80 * 1024, "two workgroups a CU");

// One operand of a step: 32 rows at `src` (row stride in elements) to its 8 KB image, by one wave. Lane L of piece p lands at chunk
// L % 16 of row 4 p + L / 16 and fetches the chunk that belongs there.
__device__ __forceinline__ void move_piece(const bf16* src, int64_t stride, uint32_t dst) {
  const int lane = lane_now();
  const uint32_t row = (uint32_t)((lane >> 4) * stride * 2), ch = 16u * ((lane & 15) ^ ((lane >> 4) << 2));
#pragma unroll
  for (int p = 0; p < 8; ++p) glds16_s(src + 4 * p * stride, row + (ch ^ (16u * (p & 3))), dst + 1024 * p);
}

// ------------------------------------------------------------------------------------------------ rows: dQ
template <bool ROWB>
__global__ void __launch_bounds__(NTHR, 2) sparse_dq_kernel(SparseBwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  Shared& sh = *reinterpret_cast<Shared*>(smem);
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), mine = wid & 1, turn = wid >> 1;  // 32 rows; which of a pair's steps
  int bh, wi;
  place(a.rows.nwork, a.B * a.H, bh, wi);
  const int b = bh / a.H, hq = bh % a.H, lh = a.rows.heads == 1 ? 0 : hq, S = a.S;
  const_int* wk = uniform_ints(a.rows.work) + ((int64_t)lh * a.rows.nwork + wi) * 4;
  const int own = wk[0], first = wk[1], count = wk[2], slot = wk[3];
  if (own < 0) return;  // (heads with fewer parts than the others)
  const int qb = own / (ROWS / OWN), part = own % (ROWS / OWN), row0 = own * OWN + 32 * mine, row = row0 + l32;

  // the list first: it waits for nothing but itself, and the first steps come while the rows do
  const int* tl = a.rows.tiles + ((int64_t)lh * (S / ROWS) + qb) * a.rows.max_tiles + first;
  const int* ml = a.rows.masks + ((int64_t)lh * (S / ROWS) + qb) * a.rows.max_tiles + first;
  auto list = [&](int e0) {
    int t = 0;
    unsigned m = 0;
    if (e0 + tid < count) {
      t = tl[e0 + tid];
      m = (unsigned)ml[e0 + tid] >> (16 * part);  // bit 4 r + k: rows 16 r .. of 64 see keys 16 k .. of the tile's 64
    }
    return pack_list(sh.ls, {2 * t, 2 * t + 1}, {(int)(m & 0x3333u), (int)((m >> 2) & 0x3333u)});
  };
  // wave (mine, turn) brings K (mine 0) or V of its half's steps
  const bf16* op = mine ? a.v + b * a.vs[0] + hq * a.vs[1] : a.k + b * a.ks[0] + hq * a.ks[1];
  const int64_t op_stride = mine ? a.vs[2] : a.ks[2];
  const float* kbp = a.kbias ? a.kbias + (int64_t)b * a.kb_stride : nullptr;
  auto move = [&](int key0, int buf) {
    move_piece(op + key0 * op_stride, op_stride, lds_at(sh.ring[buf][turn] + mine * PIECE));
    if (kbp != nullptr && mine == 0) glds4_s(kbp + key0, 4 * (lane_now() & 31), lds_at((const char*)sh.extra[buf][turn]));
  };
  auto listed = [&](int j) { return __builtin_amdgcn_readfirstlane(sh.ls.step[j]); };
  int n = list(0);
  if (turn < n) move(listed(turn) * STEP, 0);

  bf16x8 qf[8], gf[8];
  float delta = 0.f;
  {
    const bf16* qr = a.q + b * a.qs[0] + hq * a.qs[1] + (int64_t)row * a.qs[2] + 8 * h;
    const bf16* gr = a.dout + b * a.gs[0] + hq * a.gs[1] + (int64_t)row * a.gs[2] + 8 * h;
    const bf16* orow = a.o + b * a.os[0] + hq * a.os[1] + (int64_t)row * a.os[2] + 8 * h;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      qf[kk] = *reinterpret_cast<const bf16x8*>(qr + 16 * kk);
      gf[kk] = *reinterpret_cast<const bf16x8*>(gr + 16 * kk);
      const bf16x8 ov = *reinterpret_cast<const bf16x8*>(orow + 16 * kk);
#pragma unroll
      for (int i = 0; i < 8; ++i) delta = fmaf((float)ov[i], (float)gf[kk][i], delta);
    }
  }
  delta += __shfl_xor(delta, 32, 64);
  const float nlse = -a.lse[(int64_t)bh * S + row] / a.scale, c = a.scale * LOG2E, inv_scale = 1.f / a.scale;
  if (lane < 32 && turn == 0) {  // (all parts of a cut list the same)
    float* nr = a.nrow + ((int64_t)bh * S + row0) * 2 + lane;
    nr[0] = -delta;
    nr[32] = nlse;
  }

  const lds_char* s3 = (const lds_char*)smem;
  const int gq = (lane >> 2) & 3, gch = (lane >> 1) & 1, gb = 8 * (lane & 1), colhalf = (lane >> 4) & 1;
  uint32_t ra[8], ta[2][4];  // row reads; transposed reads (16 rows further: + 4096)
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) ra[kk] = (uint32_t)(l32 * 256 + 16 * ((2 * kk + h) ^ swz(l32)));
#pragma unroll
  for (int hi = 0; hi < 2; ++hi) {
    const int r = 4 * h + 8 * hi + gq;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) ta[hi][dt] = (uint32_t)(r * 256 + 16 * ((dt * 4 + colhalf * 2 + gch) ^ swz(r)) + gb);
  }

  f32x16 dq[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) dq[dt][r] = 0.f;
  // the loads that the compiler tracks are done before the loop
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) asm volatile("" : : "v"(qf[kk]), "v"(gf[kk]));
  float ndelta = -delta, ninit = nlse;
  asm volatile("" : "+v"(ndelta), "+v"(ninit));

  for (int e0 = 0;;) {
    for (int j = turn, buf = 0; j < n + turn; j += 2, buf ^= 1) {  // (as often in all waves)
      settle();  // this pair has come, and the other buffer is free
      if (j + 2 < n) move(listed(j + 2) * STEP, buf ^ 1);
      if (j >= n) continue;
      // bits 0, 1: rows 0..15 of this wave's see keys 0..15, 16..31; 4, 5: rows 16..31
      const unsigned seen = ((unsigned)__builtin_amdgcn_readfirstlane(sh.ls.mask[j]) >> (8 * mine)) & 0x33u;
      if (seen == 0) continue;
      const lds_char* img = s3 + (2 * buf + turn) * STAGE;
      f32x16 s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = ninit;
        dp[r] = ndelta;
      }
      {
        auto ld = [&](int i) { return *reinterpret_cast<const lds_bf16x8*>(img + ra[i & 7] + (i >> 3) * PIECE); };
        bf16x8 o0 = ld(0), o1 = ld(1), o2 = ld(2);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          bf16x8 o3;
          if (i + 3 < 16) o3 = ld(i + 3);
          __builtin_amdgcn_sched_barrier(0x6);
          if (i < 8) s = mfma(o0, qf[i], s);
          else dp = mfma(o0, gf[i - 8], dp);
          __builtin_amdgcn_sched_barrier(0x6);
          o0 = o1;
          o1 = o2;
          o2 = o3;
        }
      }
      auto ldk = [&](int i) {  // (dt, ss)
        const lds_char* p = img + (i & 1) * 4096;
        return join(tr_read(p + ta[0][i >> 1]), tr_read(p + ta[1][i >> 1]));
      };
      bf16x8 k0 = ldk(0), k1 = ldk(1);
      if (kbp != nullptr) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 bv = *reinterpret_cast<const f32x4*>(sh.extra[buf][turn] + 8 * g + 4 * h);
#pragma unroll
          for (int i = 0; i < 4; ++i) s[4 * g + i] = fmaf(bv[i], inv_scale, s[4 * g + i]);
        }
      }
      if constexpr (ROWB) {
        const float* abp = a.abias ? a.abias + (int64_t)row * a.ab_stride : nullptr;
        const float* rpp = a.rpe ? a.rpe + (int64_t)hq * a.rpe_hs + (int64_t)row * a.rpe_rs : nullptr;
        const int key0 = listed(j) * STEP + 4 * h;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x4 bv = {0.f, 0.f, 0.f, 0.f};
          if (abp) bv += *reinterpret_cast<const f32x4*>(abp + key0 + 8 * g);
          if (rpp) bv += *reinterpret_cast<const f32x4*>(rpp + key0 + 8 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) s[4 * g + i] = fmaf(bv[i], inv_scale, s[4 * g + i]);
        }
      }
      const unsigned bits = seen >> (4 * (l32 >> 4));
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float p = __builtin_amdgcn_exp2f(s[r] * c);
        if (seen != 0x33u && !((bits >> (r >> 3)) & 1u)) p = 0.f;
        s[r] = p * dp[r];
      }
      const bf16x8 ds[2] = {pack8(s, 0), pack8(s, 8)};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        bf16x8 k2;
        if (i + 2 < 8) k2 = ldk(i + 2);
        __builtin_amdgcn_sched_barrier(0x6);
        dq[i >> 1] = mfma(ds[i & 1], k0, dq[i >> 1]);
        __builtin_amdgcn_sched_barrier(0x6);
        k0 = k1;
        k1 = k2;
      }
    }
    settle();  // the list and the ring are written again
    if ((e0 += NTHR) >= count) break;
    n = list(e0);
    if (turn < n) move(listed(turn) * STEP, 0);
  }

  // the other half's sums: each wave gives away two of its four tiles and finishes the others
  f32x4* swap = reinterpret_cast<f32x4*>(smem) + wid * 8 * 64 + lane;
  const f32x4* take = reinterpret_cast<const f32x4*>(smem) + (wid ^ 2) * 8 * 64 + lane;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = turn ? dq[dt][4 * g + i] : dq[dt + 2][4 * g + i];
      swap[(4 * dt + g) * 64] = v;
    }
  __syncthreads();
  f32x16 sum[2];
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 v = take[(4 * dt + g) * 64];
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[dt][4 * g + i] = (turn ? dq[dt + 2][4 * g + i] : dq[dt][4 * g + i]) + v[i];
    }
  const int col = 64 * turn + l32;
  if (slot >= 0) {  // a part of the list
    float* po = a.rows.part + (((int64_t)(a.rows.heads == 1 ? bh : b) * a.rows.nslots + slot) * OWN + 32 * mine) * D + col;
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) po[crow(r, h) * D + dt * 32] = sum[dt][r];
    return;
  }
  // through LDS into whole rows (272 bytes apart: the two halves of a wave write to different banks)
  char* img = smem + 4 * 8 * 64 * 16;
#pragma unroll
  for (int r = 0; r < 16; ++r)
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
      *reinterpret_cast<bf16*>(img + (32 * mine + crow(r, h)) * 272 + 2 * (col + 32 * dt)) = (bf16)(sum[dt][r] * a.scale);
  __syncthreads();
  bf16* out = a.dq + b * a.dqs[0] + hq * a.dqs[1] + (int64_t)(own * OWN + (tid >> 4)) * a.dqs[2] + 8 * (tid & 15);
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *reinterpret_cast<bf16x8*>(out + 16 * i * a.dqs[2]) =
        *reinterpret_cast<const bf16x8*>(img + ((tid >> 4) + 16 * i) * 272 + 16 * (tid & 15));
}

// ------------------------------------------------------------------------------------------------ columns: dK, dV
constexpr int COL_PART = 2 * OWN * D / 4;  // sums of 64 keys in 16-byte pieces: [dK | dV, 32 columns, 4][32 keys, 64 lanes]

template <int BIASED>
__global__ void __launch_bounds__(NTHR, 2) sparse_dkv_kernel(SparseBwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  Shared& sh = *reinterpret_cast<Shared*>(smem);
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), mine = wid & 1, turn = wid >> 1;
  int bh, wi;
  place(a.cols.nwork, a.B * a.H, bh, wi);
  const int b = bh / a.H, hq = bh % a.H, lh = a.cols.heads == 1 ? 0 : hq, S = a.S;
  const_int* wk = uniform_ints(a.cols.work) + ((int64_t)lh * a.cols.nwork + wi) * 4;
  const int own = wk[0], first = wk[1], count = wk[2], slot = wk[3];
  if (own < 0) return;  // (heads with fewer parts than the others)
  const int kb = own / (KEYS / OWN), part = own % (KEYS / OWN), key = own * OWN + 32 * mine + l32;

  const int nkb = (S + KEYS - 1) / KEYS;
  const int* tl = a.cols.tiles + ((int64_t)lh * nkb + kb) * a.cols.max_tiles + first;
  const int* ml = a.cols.masks + ((int64_t)lh * nkb + kb) * a.cols.max_tiles + first;
  auto list = [&](int e0) {
    int t = 0, m = 0;
    if (e0 + tid < count) {
      t = tl[e0 + tid];
      m = (int)(((unsigned)ml[e0 + tid] >> (4 * part)) & 0x000f000fu);
    }
    return pack_list(sh.ls, {t, 0}, {m, 0});
  };
  // wave (mine, turn) brings Q (mine 0) or dO of its half's steps
  const bf16* op = mine ? a.dout + b * a.gs[0] + hq * a.gs[1] : a.q + b * a.qs[0] + hq * a.qs[1];
  const int64_t op_stride = mine ? a.gs[2] : a.qs[2];
  const float* nr = a.nrow + (int64_t)bh * S * 2;
  auto move = [&](int row0, int buf) {
    move_piece(op + row0 * op_stride, op_stride, lds_at(sh.ring[buf][turn] + mine * PIECE));
    if (mine == 0) glds4_s(nr + 2 * row0, 4 * lane_now(), lds_at((const char*)sh.extra[buf][turn]));
  };
  auto listed = [&](int j) { return __builtin_amdgcn_readfirstlane(sh.ls.step[j]); };
  int n = list(0);
  if (turn < n) move(listed(turn) * STEP, 0);

  bf16x8 vf[8], kf[4];
  {
    const bf16* kr = a.k + b * a.ks[0] + hq * a.ks[1] + (int64_t)key * a.ks[2] + 8 * h;
    const bf16* vr = a.v + b * a.vs[0] + hq * a.vs[1] + (int64_t)key * a.vs[2] + 8 * h;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) vf[kk] = *reinterpret_cast<const bf16x8*>(vr + 16 * kk);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) kf[kk] = *reinterpret_cast<const bf16x8*>(kr + 16 * kk);
    if (turn == 0) {
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        *reinterpret_cast<bf16x8*>(sh.kimg + (32 * mine + l32) * 128 + 16 * ((2 * kk + h) ^ (l32 & 7))) =
            *reinterpret_cast<const bf16x8*>(kr + 64 + 16 * kk);
    }
  }
  float kbias = BIASED == 0 || a.kbias == nullptr ? 0.f : a.kbias[(int64_t)b * a.kb_stride + key] * LOG2E;
  const float c = a.scale * LOG2E;

  const lds_char* s3 = (const lds_char*)smem;
  const int gq = (lane >> 2) & 3, gch = (lane >> 1) & 1, gb = 8 * (lane & 1), colhalf = (lane >> 4) & 1;
  // row reads: chunk (2 kk + h) ^ swz = (2 kk) ^ (h ^ swz); K's second half likewise; transposed reads: base + 64 (dt ^ toggle)
  uint32_t rbase = (uint32_t)(l32 * 256), rtog = (uint32_t)(16 * (h ^ swz(l32)));
  uint32_t kbase = (uint32_t)(offsetof(Shared, kimg) + (32 * mine + l32) * 128), ktog = (uint32_t)(16 * (h ^ (l32 & 7)));
  uint32_t tbase[2], ttog[2];
#pragma unroll
  for (int hi = 0; hi < 2; ++hi) {
    const int r = 4 * h + 8 * hi + gq, f = swz(r);
    tbase[hi] = (uint32_t)(r * 256 + 16 * ((colhalf * 2 + gch) ^ (f & 3)) + gb);
    ttog[hi] = (uint32_t)(f >> 2);
  }

  f32x16 dk[4], dv[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) dk[dt][r] = dv[dt][r] = 0.f;
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) asm volatile("" : : "v"(vf[kk]));
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) asm volatile("" : : "v"(kf[kk]));
  asm volatile("" : "+v"(kbias));

  for (int e0 = 0;;) {
    for (int j = turn, buf = 0; j < n + turn; j += 2, buf ^= 1) {  // (as often in all waves)
      settle();  // this pair has come, and the other buffer is free
      if (j + 2 < n) move(listed(j + 2) * STEP, buf ^ 1);
      if (j >= n) continue;
      const unsigned seen = ((unsigned)__builtin_amdgcn_readfirstlane(sh.ls.mask[j]) >> (2 * mine)) & 0x00030003u;
      if (seen == 0) continue;
      asm volatile("" : "+v"(tbase[0]), "+v"(tbase[1]), "+v"(ttog[0]), "+v"(ttog[1]), "+v"(rbase), "+v"(rtog), "+v"(kbase), "+v"(ktog));
      const lds_char* img = s3 + (2 * buf + turn) * STAGE;
      const float* nrow = sh.extra[buf][turn] + 4 * h;
      f32x16 s, dp;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 y = *reinterpret_cast<const f32x4*>(nrow + 8 * g), x = *reinterpret_cast<const f32x4*>(nrow + 32 + 8 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[4 * g + i] = x[i];
          dp[4 * g + i] = y[i];
        }
      }
      {
        auto ld_a = [&](int i) {
          return *reinterpret_cast<const lds_bf16x8*>(img + rbase + ((32u * (i & 7)) ^ rtog) + (i >> 3) * PIECE);
        };
        auto ld_k = [&](int i) { return *reinterpret_cast<const lds_bf16x8*>(s3 + kbase + ((32u * (i & 3)) ^ ktog)); };
        bf16x8 a0 = ld_a(0), a1 = ld_a(1), b0, b1;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          bf16x8 a2, b2;
          if (i + 2 < 16) a2 = ld_a(i + 2);
          if (i + 2 >= 4 && i + 2 < 8) b2 = ld_k(i + 2);
          __builtin_amdgcn_sched_barrier(0x6);
          if (i < 4) s = mfma(a0, kf[i], s);
          else if (i < 8) s = mfma(a0, b0, s);
          else dp = mfma(a0, vf[i - 8], dp);
          __builtin_amdgcn_sched_barrier(0x6);
          a0 = a1;
          a1 = a2;
          b0 = b1;
          b1 = b2;
        }
      }
      const unsigned bits = seen >> (l32 >> 4);
      const float* abp = nullptr;
      const float* rpp = nullptr;
      if constexpr (BIASED == 2) {
        const int64_t row0 = (int64_t)listed(j) * STEP;
        if (a.abias) abp = a.abias + row0 * a.ab_stride + key;
        if (a.rpe) rpp = a.rpe + (int64_t)hq * a.rpe_hs + row0 * a.rpe_rs + key;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float p;
        if constexpr (BIASED == 0) p = __builtin_amdgcn_exp2f(s[r] * c);
        else {
          float bv = kbias;
          if constexpr (BIASED == 2) {
            float more = 0.f;
            if (abp) more += abp[(int64_t)crow(r, h) * a.ab_stride];
            if (rpp) more += rpp[(int64_t)crow(r, h) * a.rpe_rs];
            bv = fmaf(more, LOG2E, bv);
          }
          p = __builtin_amdgcn_exp2f(fmaf(s[r], c, bv));
        }
        if (seen != 0x00030003u && !((bits >> (16 * (r >> 3))) & 1u)) p = 0.f;
        s[r] = p;
        dp[r] = p * dp[r];
      }
      const bf16x8 pb[2] = {pack8(s, 0), pack8(s, 8)}, ds[2] = {pack8(dp, 0), pack8(dp, 8)};
      {
        auto opnd = [&](int i) {  // (dt, 16 rows, dO | Q)
          const int dt = i >> 2;
          const lds_char* p = img + ((i & 1) ? 0 : PIECE) + 4096 * ((i >> 1) & 1);
          return join(tr_read(p + (tbase[0] + 64 * (dt ^ ttog[0]))), tr_read(p + (tbase[1] + 64 * (dt ^ ttog[1]))));
        };
        bf16x8 o0 = opnd(0), o1 = opnd(1);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          bf16x8 o2;
          if (i + 2 < 16) o2 = opnd(i + 2);
          __builtin_amdgcn_sched_barrier(0x6);
          if (i & 1) dk[i >> 2] = mfma(o0, ds[(i >> 1) & 1], dk[i >> 2]);
          else dv[i >> 2] = mfma(o0, pb[(i >> 1) & 1], dv[i >> 2]);
          __builtin_amdgcn_sched_barrier(0x6);
          o0 = o1;
          o1 = o2;
        }
      }
    }
    settle();
    if ((e0 += NTHR) >= count) break;
    n = list(e0);
    if (turn < n) move(listed(turn) * STEP, 0);
  }

  // the halves' sums: the waves of the first finish dK, those of the second dV
  const int ln = lane_now();
  f32x4* swap = reinterpret_cast<f32x4*>(smem) + wid * 16 * 64 + ln;
  const f32x4* take = reinterpret_cast<const f32x4*>(smem) + (wid ^ 2) * 16 * 64 + ln;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = turn ? dk[dt][4 * g + i] : dv[dt][4 * g + i];
      swap[(4 * dt + g) * 64] = v;
    }
  __syncthreads();
  const int64_t key_out = own * OWN + 32 * mine + (ln & 31);
  bf16* out = (turn ? a.dv + b * a.dvs[0] + hq * a.dvs[1] + key_out * a.dvs[2]
                    : a.dk + b * a.dks[0] + hq * a.dks[1] + key_out * a.dks[2]) + 8 * (ln >> 5);
  const float f = turn ? 1.f : a.scale;
  f32x4 sum[4][4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 v = take[(4 * dt + g) * 64];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += turn ? dv[dt][4 * g + i] : dk[dt][4 * g + i];
      sum[dt][g] = v;
    }
  if (slot >= 0) {  // a part: the sums as they are, 16 bytes per thread and piece
    f32x4* po = reinterpret_cast<f32x4*>(a.cols.part) +
                ((int64_t)(a.cols.heads == 1 ? bh : b) * a.cols.nslots + slot) * COL_PART + 16 * turn * 128 + 64 * mine + ln;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) po[(4 * dt + g) * 128] = sum[dt][g];
    return;
  }
  // a lane has columns 8 g + 4 h .. + 3 of its key; two g's between the wave's halves make it 8 in a row
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
      u32x4_t r;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const auto x = __builtin_amdgcn_permlane32_swap(pack_bf16(sum[dt][g][2 * i] * f, sum[dt][g][2 * i + 1] * f),
                                                        pack_bf16(sum[dt][g + 1][2 * i] * f, sum[dt][g + 1][2 * i + 1] * f), false, false);
        r[i] = x[0];
        r[2 + i] = x[1];
      }
      *reinterpret_cast<u32x4_t*>(out + 32 * dt + 8 * g) = r;
    }
}

// The parts of cut lists, added in order. First 2 blocks for every cut block of rows (32 rows each, 8 threads per row), then 4 for
// every cut block of keys: (dK | dV, 64 columns).
__global__ void __launch_bounds__(NTHR) sparse_bwd_merge_kernel(SparseBwdArgs a) {
  const int bh = blockIdx.y, b = bh / a.H, hq = bh % a.H, tid = threadIdx.x;
  int i = blockIdx.x;
  f32x4 s[4];
  if (i < 2 * a.rows.nmerge) {
    const int* me = a.rows.merges + ((int64_t)(a.rows.heads == 1 ? 0 : hq) * a.rows.nmerge + i / 2) * 4;
    if (me[0] < 0) return;
    const int row = (i & 1) * 32 + (tid >> 3), col = (tid & 7) * 16, n = me[2];
    const f32x4* src = reinterpret_cast<const f32x4*>(
        a.rows.part + (((int64_t)(a.rows.heads == 1 ? bh : b) * a.rows.nslots + me[1]) * OWN + row) * D + col);
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = src[j];
    for (int p = 1; p < n; ++p) {
      src += OWN * D / 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) s[j] += src[j];
    }
    bf16* dst = a.dq + b * a.dqs[0] + hq * a.dqs[1] + (int64_t)(me[0] * OWN + row) * a.dqs[2] + col;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      bf16x8 r;
#pragma unroll
      for (int e = 0; e < 8; ++e) r[e] = (bf16)(s[2 * j + e / 4][e & 3] * a.scale);
      *reinterpret_cast<bf16x8*>(dst + 8 * j) = r;
    }
    return;
  }
  i -= 2 * a.rows.nmerge;
  const int* me = a.cols.merges + ((int64_t)(a.cols.heads == 1 ? 0 : hq) * a.cols.nmerge + i / 4) * 4;
  if (me[0] < 0) return;
  const int isv = (i >> 1) & 1, dt = 2 * (i & 1) + (tid >> 7), lane = tid & 63, h = lane >> 5, n = me[2];
  const f32x4* src = reinterpret_cast<const f32x4*>(a.cols.part) +
                     ((int64_t)(a.cols.heads == 1 ? bh : b) * a.cols.nslots + me[1]) * COL_PART + (16 * isv + 4 * dt) * 128 + (tid & 127);
#pragma unroll
  for (int g = 0; g < 4; ++g) s[g] = src[g * 128];
  for (int p = 1; p < n; ++p) {
    src += COL_PART;
#pragma unroll
    for (int g = 0; g < 4; ++g) s[g] += src[g * 128];
  }
  const int64_t key = me[0] * OWN + (tid & 64) / 2 + (lane & 31);
  bf16* dst = (isv ? a.dv + b * a.dvs[0] + hq * a.dvs[1] + key * a.dvs[2] : a.dk + b * a.dks[0] + hq * a.dks[1] + key * a.dks[2]) +
              32 * dt + 4 * h;
  const float f = isv ? 1.f : a.scale;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    bf16x4 r;
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = (bf16)(s[g][j] * f);
    *reinterpret_cast<bf16x4*>(dst + 8 * g) = r;
  }
}

template <auto KERNEL>
int launch(int64_t grid, const SparseBwdArgs& a, hipStream_t st) {
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(KERNEL), hipFuncAttributeMaxDynamicSharedMemorySize, sizeof(Shared));
    attr = true;
  }
  hipLaunchKernelGGL(KERNEL, dim3((unsigned)grid), dim3(NTHR), sizeof(Shared), st, a);
  DS_CHECK_LAUNCH();
  return 0;
}

}  // namespace

// Strides are (batch, head, row) in elements, unit last stride, rows 16-byte aligned bf16: all of them [B, H, S, 128], S a multiple
// of 128. lse [B, H, S] from ds_flash_fwd_sparse, nrow a workspace of 2 B H S floats. Plans: ints tiles, masks, work, merges and (max_tiles,
// heads = 1 or H, nwork, nmerge, nslots); parts of a side with nmerge > 0: slots x 64 x 128 floats (rows), x 128 x 128 (columns),
// slots = nslots x (B H with a shared layout, else B). Biases as in the forward.
extern "C" int ds_sparse_bwd(const void* q, const void* k, const void* v, const void* o, const void* dout, const float* lse, float* nrow,
                             void* dq, void* dk, void* dv, int B, int H, int S, const int64_t* strides, float scale,
                             const int* const* row_lists, const int* row_sizes, float* row_part, const int* const* col_lists,
                             const int* col_sizes, float* col_part, const float* kbias, int64_t kb_stride, const float* abias,
                             int64_t ab_stride, const float* rpe, int64_t rpe_hs, int64_t rpe_rs, hipStream_t st) {
  if (B <= 0 || H <= 0 || S <= 0 || S % ROWS) return (int)hipErrorInvalidValue;
  SparseBwdArgs a{};
  a.q = (const bf16*)q; a.k = (const bf16*)k; a.v = (const bf16*)v; a.o = (const bf16*)o; a.dout = (const bf16*)dout;
  a.dq = (bf16*)dq; a.dk = (bf16*)dk; a.dv = (bf16*)dv;
  a.lse = lse; a.nrow = nrow; a.B = B; a.H = H; a.S = S; a.scale = scale;
  int64_t* to[8] = {a.qs, a.ks, a.vs, a.os, a.gs, a.dqs, a.dks, a.dvs};
  for (int i = 0; i < 24; ++i) to[i / 3][i % 3] = strides[i];
  auto side = [&](Side& s, const int* const* lists, const int* n, float* part) {
    s = Side{lists[0], lists[1], lists[2], lists[3], n[0], n[1], n[2], n[3], n[4], part};
    return s.tiles && s.masks && s.work && s.max_tiles > 0 && (s.heads == 1 || s.heads == H) && s.nwork > 0 &&
           (s.nmerge <= 0 || (s.merges && s.nslots > 0 && part));
  };
  if (!side(a.rows, row_lists, row_sizes, row_part) || !side(a.cols, col_lists, col_sizes, col_part)) return (int)hipErrorInvalidValue;
  auto al = [](const float* p, int64_t s) { return p == nullptr || (((uintptr_t)p % 16) == 0 && s % 4 == 0); };
  if (!al(kbias, kb_stride) || !al(abias, ab_stride) || !al(rpe, rpe_rs) || rpe_hs % 4) return (int)hipErrorInvalidValue;
  a.kbias = kbias; a.abias = abias; a.rpe = rpe;
  a.kb_stride = kb_stride; a.ab_stride = ab_stride; a.rpe_hs = rpe_hs; a.rpe_rs = rpe_rs;
  const int64_t bh = (int64_t)B * H;
  if (bh * a.rows.nwork > INT32_MAX || bh * a.cols.nwork > INT32_MAX) return (int)hipErrorInvalidValue;
  const bool rowb = abias || rpe;
  int rc = (rowb ? launch<sparse_dq_kernel<true>> : launch<sparse_dq_kernel<false>>)(bh * a.rows.nwork, a, st);
  if (rc) return rc;
  rc = (rowb ? launch<sparse_dkv_kernel<2>> : kbias ? launch<sparse_dkv_kernel<1>> : launch<sparse_dkv_kernel<0>>)(bh * a.cols.nwork, a, st);
  if (rc) return rc;
  const int merges = 2 * max(a.rows.nmerge, 0) + 4 * max(a.cols.nmerge, 0);
  if (merges > 0) {
    hipLaunchKernelGGL(sparse_bwd_merge_kernel, dim3(merges, (unsigned)bh), dim3(NTHR), 0, st, a);
    DS_CHECK_LAUNCH();
  }
  return 0;
}
