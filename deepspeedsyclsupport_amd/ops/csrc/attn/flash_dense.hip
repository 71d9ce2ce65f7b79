// Dense flash attention forward (training, prefill without pages), bf16, head dim 128, with the loop of flash_core.h. Waves of a workgroup have 32 rows each: of
// 4, 2 or 1 heads that share their keys, then as many equal waves, or of 128 neighbours. Outputs O (any [B, H, S, D] strides, e.g. written straight into the
// [B, S, H, D] layout that the output projection wants) and the natural-log LSE [B, H, S] in fp32 that the backward pass consumes.
//
// Reference counterparts: the fused softmax-context path of `csrc/transformer/inference/csrc/pt_binding.cpp:434-557` and the Triton
// `_flash_packed_kernel` (`ops/transformer/inference/triton/attention.py:253`).
#include "flash_core.h"

namespace {
using namespace flash;

struct DenseArgs {
  const bf16 *q, *k, *v;
  bf16* o;
  float* lse;
  int B, Hq, Hk, S, Skv, heads;  // heads: of a workgroup
  int64_t qs[3], ks[3], vs[3], os[3];
  float scale;
};

template <bool CAUSAL>
__global__ void __launch_bounds__(256, 2) flash_dense_kernel(DenseArgs a) {
  __shared__ __attribute__((aligned(32768))) char lds[LDS];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, l16 = lane & 15;
  // causal: the heaviest rows of several heads first (by_block): head by head, an XCD's last head began its longest rows when the others were nearly through (us:
  // 2 x 4096, 32 heads 350, 317; 1 x 4096, 20 heads 129, 102; 1 x 2048, 32 heads 62.6, 50.4; 3 x 1000, 16 heads over 4 38.8, 33.5; 5 x 1500, 8 heads 45.3, 39.3;
  // 1 x 8192, 4 heads 160, 161). Else all rows weigh the same, and an XCD reads the keys of one head after another (by_block, and so: 5 x 1500, 20 heads
  // 133, 125; 1 x 4096, 12, 20 and 28 heads 123, 194, 247, 122, 191, 245; 2 x 4096, 32 heads 522, 508; 8 x 4096 2086, 2030; 8 x 512, 16 heads over 8 24.1, 24.3)
  const int rows = WAVES * ROWS / a.heads, blocks = (a.S + rows - 1) / rows, groups = a.Hq / a.heads;
  int bh, at;
  if constexpr (CAUSAL) by_block(a.B * groups, blocks, true, bh, at);
  else {
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    bh = logical / blocks;
    at = logical % blocks;
  }
  const int b = bh / groups, hq = bh % groups * a.heads + wid % a.heads, hk = bh % groups * a.heads / (a.Hq / a.Hk);
  const int q0 = (CAUSAL ? blocks - 1 - at : at) * rows, q0w = q0 + wid / a.heads * ROWS;
  const int tiles = (a.Skv + BN - 1) / BN;
  auto seen = [&](int first, int n) {  // tiles of n rows from `first` on
    if (first >= a.S) return 0;
    return CAUSAL ? min(tiles, (min(first + n, a.S) + BN - 1) / BN) : tiles;
  };
  const int all = seen(q0, rows), mine = seen(q0w, ROWS);
  const bf16* Q = a.q + b * a.qs[0] + hq * a.qs[1];
  const char *K = (const char*)(a.k + b * a.ks[0] + hk * a.ks[1]), *V = (const char*)(a.v + b * a.vs[0] + hk * a.vs[1]);

  const uint32_t base = (uint32_t)(uintptr_t)(lds_char*)lds;
  const int drow = dma_row(lane, wid), dcol = dma_column(lane, wid);
  const uint32_t kdma = (uint32_t)(drow * a.ks[2] + dcol) * 2, vdma = (uint32_t)(drow * a.vs[2] + dcol) * 2;
  auto move = [&](const char* from, int64_t ld, uint32_t dma, int tile, uint32_t to) {
    if (tile >= all) return;
    const uint32_t dst = __builtin_amdgcn_readfirstlane(base + to + 1024 * wid);
    if (tile * BN + BN <= a.Skv) {
      const char* p = from + tile * BN * ld * 2;
#pragma unroll
      for (int i = 0; i < 4; ++i) dma16(p + 16 * i * ld * 2, dma, dst + 4096 * i);
    } else {  // rows past the end repeat the last one (they are masked, and must be numbers)
#pragma unroll
      for (int i = 0; i < 4; ++i) dma16(from + (min(tile * BN + 16 * i + drow, a.Skv - 1) * ld + dcol) * 2, dst + 4096 * i);
    }
  };
  int next = 0;  // tile of values that comes next; keys are one ahead
  uint32_t kslot = 0, vslot = 2 * TILE;
  auto moves = [&]() {
    move(K, a.ks[2], kdma, next + 1, kslot);
    move(V, a.vs[2], vdma, next, vslot);
    ++next;
    kslot ^= TILE;
    vslot ^= TILE;
  };
  move(K, a.ks[2], kdma, 0, 0);
  kslot = TILE;
  moves();  // keys 1, values 0
  Rows w;
  w.init(base, lane, a.scale * 1.4426950408889634f);
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      w.qf[q][ks] = *reinterpret_cast<const bf16x8*>(Q + (int64_t)min(q0w + 16 * q + l16, a.S - 1) * a.qs[2] + 32 * ks + 8 * g);
  auto mask = [&](auto h_c, int tile) {  // causal diagonal, key tail
    constexpr int h = h_c.value;
    const int k0 = tile * BN + 32 * h;
    if ((CAUSAL && k0 + 31 > q0w) || k0 + 32 > a.Skv)
      each<2>([&](auto q) {
        const int last = min(a.Skv - 1, CAUSAL ? q0w + 16 * q.value + l16 : a.Skv) - k0 - 4 * g;
        each<2>([&](auto kb) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (16 * kb.value + i > last) w.s[2 * h + kb.value][q.value][i] = -INFINITY;
          __builtin_amdgcn_sched_barrier(0);
        });
      });
  };
  meet();
  w.run(mine, all, mask, [&]() {
    meet();
    moves();
  });
  if (mine == 0) return;
  bf16* O = a.o + b * a.os[0] + hq * a.os[1];
  each<2>([&](auto q) {
    const float sum = w.sum(q.value);
    const int row = q0w + 16 * q.value + l16;
    w.store(q.value, sum > 0.f ? 1.f / sum : 0.f, O + (int64_t)row * a.os[2], lane, row < a.S);
    if (a.lse && g == 0 && row < a.S)
      a.lse[((int64_t)b * a.Hq + hq) * a.S + row] = sum > 0.f ? (w.ref[q.value] + __log2f(sum)) * 0.69314718055994531f : INFINITY;
  });
}

}  // namespace

// q [B,Hq,S,128], k/v [B,Hk,Skv,128] (bf16, unit last stride, any outer strides), o [B,Hq,S,128] (any outer strides),
// lse [B,Hq,S] fp32 (optional). strides are (batch, head, seq) in elements. Top-left causal alignment (SDPA's).
extern "C" int ds_flash_fwd(const void* q, const void* k, const void* v, void* o, float* lse, int B, int Hq, int Hk, int S, int Skv, const int64_t* qs,
                            const int64_t* ks, const int64_t* vs, const int64_t* os, float scale, int causal, hipStream_t st) {
  if (Hk <= 0 || Hq % Hk != 0 || S <= 0 || Skv <= 0) return (int)hipErrorInvalidValue;
  const int share = Hq / Hk, heads = share % 4 == 0 ? 4 : share % 2 == 0 ? 2 : 1, rows = WAVES * ROWS / heads;
  const DenseArgs a{(const bf16*)q, (const bf16*)k, (const bf16*)v, (bf16*)o, lse, B, Hq, Hk, S, Skv, heads,
                    {qs[0], qs[1], qs[2]}, {ks[0], ks[1], ks[2]}, {vs[0], vs[1], vs[2]}, {os[0], os[1], os[2]}, scale};
  const dim3 grid((unsigned)((S + rows - 1) / rows * B * (Hq / heads)));
  if (causal) hipLaunchKernelGGL(flash_dense_kernel<true>, grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL(flash_dense_kernel<false>, grid, dim3(256), 0, st, a);
  DS_CHECK_LAUNCH();
  return 0;
}
