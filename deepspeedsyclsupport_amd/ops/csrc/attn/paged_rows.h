// Ragged paged attention for heads of 128 that see all keys up to their position (ALiBi or not), with the loop of flash_core.h: the arguments of
// paged_prefill_core.h. Waves have 32 query rows each: of 4, 2 or 1 heads that share their keys, then as many equal waves, or of the 128 neighbours of a
// work item. The heaviest rows of all groups of an XCD's heads first (as in paged_flash.h).
// A page of 16 tokens or more holds 16 rows of a tile at a place of its own. Lanes have the numbers of 16 tiles' pages, asked for eight tiles ahead (a scalar
// load a tile is waited for with the LDS reads behind it); only a ragged last tile is addressed row by row.
// (With the places of a tile's rows worked out between its two halves' transfers, for keys and for values, instead of once, 1 % longer.)
#pragma once
#include "flash_core.h"
#include "paged_prefill_core.h"

namespace {

// heads: of a workgroup; page_shift: log2 of the page size, 4 or more
__global__ void __launch_bounds__(256, 2) paged_rows_kernel(PagedArgs a, int heads, int page_shift) {
  using namespace flash;
  __shared__ __attribute__((aligned(32768))) char lds[flash::LDS];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, l16 = lane & 15;
  const int rows = WAVES * ROWS / heads;
  const int per = gridDim.x / (a.Hq / heads);
  int group, rest;
  by_block(a.Hq / heads, per, (int64_t)a.max_blocks * a.BS >= 4096, group, rest);
  const int item = (per - 1 - rest) / heads, part = (per - 1 - rest) % heads;
  const int hq = group * heads + wid % heads, hk = group * heads / (a.Hq / a.Hk);
  const int seq = __builtin_amdgcn_readfirstlane(a.work[2 * item]), q0 = __builtin_amdgcn_readfirstlane(a.work[2 * item + 1]) * ::BM + part * rows;
  const int t0 = __builtin_amdgcn_readfirstlane(a.cu_q[seq]), n = __builtin_amdgcn_readfirstlane(a.cu_q[seq + 1]) - t0;
  const int start = __builtin_amdgcn_readfirstlane(a.start[seq]), Skv = start + n;
  if (q0 >= n) return;
  const int q0w = q0 + wid / heads * ROWS;
  auto seen = [&](int first, int count) { return first >= n ? 0 : (start + min(first + count, n) - 1) / flash::BN + 1; };
  const int all = seen(q0, rows), mine = seen(q0w, ROWS);
  const int* bt = a.block_table + (int64_t)seq * a.max_blocks;

  const uint32_t base = (uint32_t)(uintptr_t)(flash::lds_char*)lds;
  const int drow = dma_row(lane, wid), dcol = dma_column(lane, wid);
  const uint32_t dma = (uint32_t)(drow * flash::D + dcol) * 2;
  const int last_page = (Skv - 1) >> page_shift, pmask = a.BS - 1;
  const int64_t head = (int64_t)hk * a.BS * flash::D * 2, page = (int64_t)a.Hk * a.BS * flash::D * 2;  // bytes
  int64_t ahead[4], here[4];  // where the 16-row groups of the tiles lie that keys, and values, come from next
  auto listed = [&](int tile) { return bt[min((tile * flash::BN + 16 * lane) >> page_shift, last_page)]; };  // pages of 16 tiles
  int list = listed(0), after = list;
  auto look_up = [&](int tile) {
    if (tile % 16 == 0 && tile) list = after;
    const int64_t first = __builtin_amdgcn_readlane(list, tile % 16 * 4) * page + head + ((tile * flash::BN) & pmask) * (flash::D * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      here[i] = ahead[i];
      ahead[i] = first + 4096 * i;  // (all in one page of 64 tokens or more)
    }
    if (page_shift < 6)
#pragma unroll
      for (int i = 1; i < 4; ++i)
        ahead[i] = __builtin_amdgcn_readlane(list, tile % 16 * 4 + i) * page + head + ((tile * flash::BN + 16 * i) & pmask) * (flash::D * 2);
  };
  auto move = [&](const bf16* cache, const int64_t (&of)[4], int tile, uint32_t to) {
    if (tile >= all) return;
    const uint32_t dst = __builtin_amdgcn_readfirstlane(base + to + 1024 * wid);
    if (tile * flash::BN + flash::BN <= Skv) {
#pragma unroll
      for (int i = 0; i < 4; ++i) flash::dma16((const char*)cache + of[i], dma, dst + 4096 * i);
    } else {  // rows past the end repeat the last one (they are masked, and must be numbers)
      int64_t at[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = min(tile * flash::BN + 16 * i + drow, Skv - 1);
        at[i] = bt[key >> page_shift] * page + head + ((key & pmask) * flash::D + dcol) * 2;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) flash::dma16((const char*)cache + at[i], dst + 4096 * i);
    }
  };
  int next = 0;  // tile of values that comes next; keys are one ahead
  uint32_t kslot = 0, vslot = 2 * TILE;
  auto moves = [&]() {
    move(a.kc, ahead, next + 1, kslot);
    move(a.vc, here, next, vslot);
    ++next;
    look_up(next + 1);
    if (next % 16 == 8) after = listed(next + 8);
    kslot ^= TILE;
    vslot ^= TILE;
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) ahead[i] = 0;
  look_up(0);
  move(a.kc, ahead, 0, 0);
  look_up(1);
  kslot = TILE;
  moves();  // keys 1, values 0
  Rows w;
  w.init(base, lane, a.c);
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      w.qf[q][ks] = *reinterpret_cast<const bf16x8*>(a.q + (int64_t)(t0 + min(q0w + 16 * q + l16, n - 1)) * a.ldq + hq * flash::D + 32 * ks + 8 * g);
  const float slope = a.alibi ? a.alibi[hq] * a.inv_scale : 0.f;
  auto mask = [&](auto h_c, int tile) {  // ALiBi, causal diagonal, key tail
    constexpr int h = h_c.value;
    const int k0 = tile * flash::BN + 32 * h;
    if (a.alibi)
      flash::each<2>([&](auto q) {
        const int from = k0 + 4 * g - (start + q0w + 16 * q.value + l16);
        flash::each<2>([&](auto kb) {
          f32x4& s = w.s[2 * h + kb.value][q.value];
#pragma unroll
          for (int i = 0; i < 4; ++i) s[i] = fmaf(slope, (float)(from + 16 * kb.value + i), s[i]);
        });
      });
    if (k0 + 31 > start + q0w)
      flash::each<2>([&](auto q) {
        const int last = min(Skv - 1, start + q0w + 16 * q.value + l16) - k0 - 4 * g;
        flash::each<2>([&](auto kb) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (16 * kb.value + i > last) w.s[2 * h + kb.value][q.value][i] = -INFINITY;
          __builtin_amdgcn_sched_barrier(0);
        });
      });
  };
  flash::meet();
  w.run(mine, all, mask, [&]() {
    flash::meet();
    asm volatile("" : "+v"(after));  // (if it was asked for, it has come with the transfers; used later, it would be waited for with those to come)
    moves();
  });
  if (mine == 0) return;
  flash::each<2>([&](auto q) {
    const float sum = w.sum(q.value);
    const int row = q0w + 16 * q.value + l16;
    w.store(q.value, sum > 0.f ? 1.f / sum : 0.f, a.o + (int64_t)(t0 + row) * a.ldo + hq * flash::D, lane, row < n);
  });
}

// Without a window: with one, a row's first tile may hold none of its keys.
inline bool paged_rows_fits(const PagedArgs& a) { return a.window <= 0; }
// Its first tile and its last values stand alone: it needs many tiles, and two workgroups a CU twice over. us with the loop of paged_flash.h and this one, 32
// heads over 8, 16 over 8, 32 over 32: 1 x 8192 537, 506; 290, 277; 546, 522; 4 x 2048 158, 150; 91.6, 88.8; 159, 153; 8 x 1024 95.7, 92.3; 59.2, 60.1;
// 96.9, 94.2; 16 x 512 62.8, 62.7; 39.7, 41.5; 64.3, 64.4; 48 x 160 52, 59; 29.5, 34.0; 57, 61; 1 x 2048 52.6, 51.3; 45.7, 46.7; 52.3, 50.8.
inline bool paged_rows_pays(const PagedArgs& a, int nwork) { return (int64_t)nwork * a.Hq >= 1024 && (int64_t)a.max_blocks * a.BS >= 2048; }

int launch_rows(const PagedArgs& a, int nwork, hipStream_t st) {
  const int share = a.Hq / a.Hk, heads = share % 4 == 0 ? 4 : share % 2 == 0 ? 2 : 1;
  hipLaunchKernelGGL(paged_rows_kernel, dim3(nwork * a.Hq), dim3(256), 0, st, a, heads, __builtin_ctz((unsigned)a.BS));
  DS_CHECK_LAUNCH();
  return 0;
}

}  // namespace
