// bf16 products of a linear layer of many tokens: y = X W^T, dX = dY W and dW = dY^T X, each over the operands as they lie in memory, sums in fp32, one
// rounding at the end. Tiles of 256, 192 or 128 rows by 256 columns, with the loop of wide_core.h. Of y, a gated activation's silu(gate) up as well, of two
// neighbours' sums in registers: what a prompt's gate and up would be written and read for.
#include "wide_core.h"

#include <algorithm>
#include <cmath>

namespace {
using namespace wide;

struct WideArgs {
  const bf16 *a, *b;  // a: M x K, b: N x K, or with rows along k: K x M, K x N
  bf16* c;            // [M, N], rows ldc apart
  int M, N, K, ldc;
  uint32_t lda, ldb, abytes, bbytes;
  int band;           // row tiles that are walked together, column by column
  int up;             // (gated) rows from the gate's part of b to the other
  int parts, deep;    // (in parts) of K, and steps of each but the last
  float* part;        // their sums [parts, M, N]
};

// What becomes of the sums: GATED: b is [2 N, K], the gate's rows before the up part's; a tile has 128 of either, in blocks of 16 in turn. PARTS: of a range of K,
// in fp32, for wide_sum_kernel
enum : int { PLAIN = 0, GATED = 1, PARTS = 2 };
template <int AK, int BK, int MI, int OUT>
__global__ void __launch_bounds__(256, 1) wide_gemm_kernel(WideArgs a) {
  constexpr bool GATE = OUT == GATED;
  typedef Loop<AK, BK, MI, true> L;
  constexpr int TM = L::TM, NB = GATE ? L::NI / 2 : L::NI, TN = 32 * NB, STORES = MI * NB / 2;  // NB: blocks of 16 columns that a wave writes
  __shared__ __attribute__((aligned(16))) char lds[L::LDS];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int mt = (a.M + TM - 1) / TM, nt = (a.N + TN - 1) / TN, whole = mt * nt, tiles = OUT == PARTS ? whole * a.parts : whole;
  // an XCD's tiles are neighbours; its workgroups take them in turn
  const int xcd = blockIdx.x & 7, per = tiles >> 3, more = tiles & 7, stride = ((int)gridDim.x - xcd + 7) >> 3;
  const int last = per * (xcd + 1) + min(xcd + 1, more);
  int id = per * xcd + min(xcd, more) + ((int)blockIdx.x >> 3);
  if (id >= last) return;
  const int steps = (a.K + 63) / 64;
  auto part_of = [&](int t) { return OUT == PARTS ? t / whole : 0; };
  auto first_of = [&](int t) { return part_of(t) * a.deep * 64; };  // of K
  auto place = [&](int t, int& m0, int& n0) {
    if constexpr (OUT == PARTS) t %= whole;
    const int strip = t / (a.band * nt), spot = t - strip * a.band * nt, deep = min(a.band, mt - strip * a.band);
    m0 = __builtin_amdgcn_readfirstlane((strip * a.band + spot % deep) * TM);
    n0 = __builtin_amdgcn_readfirstlane(spot / deep * TN);
  };
  int m0, n0;
  place(id, m0, n0);
  L loop;
  loop.oa.from = L::A::tile(a.a, a.abytes, a.lda, m0, first_of(id));
  loop.ob.from = L::B::tile(a.b, a.bbytes, a.ldb, n0, first_of(id));
  loop.oa.sources(a.lda, lane, wid);
  loop.ob.sources(a.ldb, lane, wid);
  if constexpr (GATE)
    each<L::PB>([&](auto i) {
      const int r = L::B::row(i.value, lane, wid);
      loop.ob.src[i.value] = (uint32_t)((r >> 5) * 16 + (r & 15) + (r & 16 ? a.up : 0)) * a.ldb * 2 + L::B::chunk(i.value, lane, wid);
    });
  loop.begin(lds, steps, lane, wid);  // (a tile's, and a part's, are more than it begins with)
  for (;;) {
    // the tile that follows, or this one's beginning again, for nobody
    const bool ends = id + stride >= last;
    const int next = ends ? id : id + stride;
    int m2, n2;
    place(next, m2, n2);
    const int all = OUT == PARTS ? min(a.deep, steps - part_of(id) * a.deep) : steps;
    loop.template tile<OUT == PARTS ? 0 : STORES>(all, L::A::tile(a.a, a.abytes, a.lda, m2, first_of(next)), L::B::tile(a.b, a.bbytes, a.ldb, n2, first_of(next)));
    if constexpr (OUT == PARTS) {  // (columns past the end past the buffer's; more stores than the next tile's barrier can count, which waits for them)
      const int64_t row0 = (int64_t)part_of(id) * a.M + m0;
      const auto c = __builtin_amdgcn_make_buffer_rsrc(a.part + row0 * a.N, 0, (int)((uint32_t)min(TM, a.M - m0) * a.N * 4), 0x00020000);
      const int row = (wid & 1) * 16 * MI + (lane & 15), col = n0 + (wid >> 1) * 16 * NB + 4 * (lane >> 4);
      each<MI>([&](auto m_c) {
        each<NB>([&](auto n_c) {
          constexpr int m = m_c.value, n = n_c.value;
          const uint32_t at = col + 16 * n < a.N ? ((uint32_t)(row + 16 * m) * a.N + col + 16 * n) * 4 : 0xc0000000u;
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, loop.acc[m][n]), c, at, 0, 0);
        });
      });
    } else {
      // ---- a lane has columns 4 (lane / 16) .. + 3 of every block: 16-lane rows change places, and it has eight neighbours. What lies past C's
      // rows or columns lies past the buffer's end: every wave stores as often as the next tile's barrier counts.
      // Past the caches (y, 6005 by [32000, 2048] 601 -> 556 us, 8192 by [22016, 4096] 998 -> 981): the next tile's second barrier waits for them.
      const auto c = __builtin_amdgcn_make_buffer_rsrc(a.c + (int64_t)m0 * a.ldc, 0, (int)((uint32_t)(min(TM, a.M - m0) - 1) * a.ldc * 2 + a.N * 2), 0x00020000);
      const int row = (wid & 1) * 16 * MI + (lane & 15), col = n0 + (wid >> 1) * 16 * NB + 16 * ((lane >> 4) & 1) + 8 * (lane >> 5);
      each<NB / 2>([&](auto n_c) {
        constexpr int n = 2 * n_c.value;
        uint32_t at = (uint32_t)row * a.ldc * 2 + (col + 16 * n < a.N ? 2 * (col + 16 * n) : 0xc0000000u);
        each<MI>([&](auto m_c) {
          auto two = [&](auto b_c, int q) {  // columns 2 q and 2 q + 1 of the lane's four in block b
            constexpr int b = decltype(b_c)::value, m = decltype(m_c)::value;
            f32x2 v;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              if constexpr (GATE) {
                const float g = loop.acc[m][2 * b][2 * q + i];
                v[i] = g / (1.f + __expf(-g)) * loop.acc[m][2 * b + 1][2 * q + i];
              } else v[i] = loop.acc[m][b][2 * q + i];
            }
            return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
          };
          u32x4 o;
#pragma unroll
          for (int q = 0; q < 2; ++q) {
#ifdef __HIP_DEVICE_COMPILE__
            const auto v = __builtin_amdgcn_permlane16_swap(two(Int<n>{}, q), two(Int<n + 1>{}, q), false, false);
            o[q] = v[0];
            o[2 + q] = v[1];
#endif
          }
          __builtin_amdgcn_raw_buffer_store_b128(o, c, at, 0, 2);  // (nt)
          at += 32 * a.ldc;
        });
      });
    }
    if (ends) break;
    id = next;
    m0 = m2;
    n0 = n2;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the surplus transfers)
}

thread_local int g_rows = 0, g_parts = 0;  // (a thread's own)

// The parts' sums added up in their order, eight columns a thread
__global__ void __launch_bounds__(256) wide_sum_kernel(const float* __restrict__ part, bf16* __restrict__ c, int64_t pieces, int parts) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= pieces) return;
  f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll 4
  for (int p = 0; p < parts; ++p) {
    const f32x4* s = reinterpret_cast<const f32x4*>(part + p * pieces * 8) + 2 * i;
    lo += s[0];
    hi += s[1];
  }
  bf16x8 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    r[j] = (bf16)lo[j];
    r[4 + j] = (bf16)hi[j];
  }
  *reinterpret_cast<bf16x8*>(c + 8 * i) = r;
}

// us of a launch over tiles of so many rows: a round takes a step's clocks, and the chip's power its share for every tile, so a round that is not full costs
// less than a full one. Drawn by 400 products at random (mean error 4 to 6 %; the rows chosen by it take 0.24 % longer than the best of the three in the mean);
// tiles of 192 and 128 rows are put 4 % higher than the fit, as they read more and suffer where that comes from memory.
double time_of(int rows, int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = (M + rows - 1) / rows * ((N + 255) / 256), rounds = (tiles + 255) / 256, steps = (K + 63) / 64;
  const double step = rows == 256 ? 0.908 : rows == 192 ? 0.742 : 0.531, round = rows == 256 ? 5.9 : rows == 192 ? 4.3 : 2.9,
               power = rows == 256 ? 0.965 : rows == 192 ? 0.772 : 0.551;
  return 3 + std::hypot(rounds * (step * steps + round), tiles / 256. * power * steps);
}

// C in one part, or in two that are cut between rows or columns: tiles of `rows` up to m, n and of `other` beyond
struct Plan {
  int rows, other;
  int64_t m, n;
  double time;
  int parts = 1, deep = 0;  // of K, steps of each
};

// Tiles of 256 rows where they fill the chip's rounds, of fewer for what would leave a round half empty
Plan plan_for(int64_t M, int64_t N, int64_t K, bool parts_too) {
  const int sizes[3] = {256, 192, 128};
  const int steps = (int)((K + 63) / 64);
  auto cut = [&](int rows, int parts) {
    int deep = (steps + parts - 1) / parts;
    while (steps % deep && steps % deep < STEPS) ++deep;
    Plan p{rows, 0, M, N, 0, (steps + deep - 1) / deep, deep};
    const int64_t mt = (M + rows - 1) / rows;
    p.time = time_of(rows, mt * rows * p.parts, N, deep * 64) + 4 + (8 * p.parts + 2) * 1e-6 / 5 * M * N;
    return p;
  };
  if (g_rows) return cut(g_rows, parts_too ? std::max(1, std::min(g_parts, steps / STEPS)) : 1);
  Plan best = {0, 0, M, N, 0};
  auto offer = [&](const Plan& p) {
    if (!best.rows || p.time < best.time) best = p;
  };
  for (int rows : sizes) {
    offer({rows, 0, M, N, time_of(rows, M, N, K)});
    // K in parts where its tiles leave the chip idle: their sums are written and read, at 5 TB/s, in a launch of its own. us in one part and so: dX, 3000 by
    // [32000, 2048] 390, 308; 4000 by [32000, 1024] 350, 200; 3509 by [22016, 512] 219, 76; 1488 by [50304, 2816] 566, 338; 1489 by [14336, 2048] 89, 77
    const int64_t tiles = (M + rows - 1) / rows * ((N + 255) / 256);
    for (int parts = 2; parts_too && parts <= 8 && tiles < 256 && tiles * parts <= 512 && parts * 16 <= steps; ++parts) offer(cut(rows, parts));
    const int64_t mt = (M + rows - 1) / rows, nt = (N + 255) / 256;
    for (int64_t k = mt * nt / 256; k > 0 && k >= mt * nt / 256 - 1; --k) {  // the first part's rounds
      const int64_t m = std::min<int64_t>(256 * k / nt, mt - 1) * rows, n = std::min<int64_t>(256 * k / mt, nt - 1) * 256;
      for (int other : sizes) {
        if (m > 0) offer({rows, other, m, N, time_of(rows, m, N, K) + time_of(other, M - m, N, K)});
        if (n > 0) offer({rows, other, M, n, time_of(rows, M, n, K) + time_of(other, M, N - n, K)});
      }
    }
  }
  return best;
}
// (a product asks for it five times)
Plan plan_of(int64_t M, int64_t N, int64_t K, bool parts_too = true) {
  thread_local struct { int64_t M = -1, N, K; int rows, parts; bool too; Plan plan; } last;
  if (last.M != M || last.N != N || last.K != K || last.rows != g_rows || last.parts != g_parts || last.too != parts_too)
    last = {M, N, K, g_rows, g_parts, parts_too, plan_for(M, N, K, parts_too)};
  return last.plan;
}

int launch(WideArgs a, int rows, int a_along, int b_along, bool gate, hipStream_t st) {
  const int64_t mt = (a.M + rows - 1) / rows, nt = (a.N + (gate ? 127 : 255)) / (gate ? 128 : 256);
  a.band = (int)std::min<int64_t>(4, mt);
  const dim3 grid((unsigned)std::min<int64_t>(mt * nt * a.parts, 256));
#define GO(AK, BK, OUT)                                                                                      \
  do {                                                                                                       \
    if (rows == 256) hipLaunchKernelGGL((wide_gemm_kernel<AK, BK, 8, OUT>), grid, dim3(256), 0, st, a);      \
    else if (rows == 192) hipLaunchKernelGGL((wide_gemm_kernel<AK, BK, 6, OUT>), grid, dim3(256), 0, st, a); \
    else hipLaunchKernelGGL((wide_gemm_kernel<AK, BK, 4, OUT>), grid, dim3(256), 0, st, a);                  \
  } while (0)
#define FORMS(OUT)                                  \
  do {                                              \
    if (a_along && b_along) GO(ALONG, ALONG, OUT);  \
    else if (a_along) GO(ALONG, ACROSS, OUT);       \
    else GO(ACROSS, ACROSS, OUT);                   \
  } while (0)
  if (gate) GO(ALONG, ALONG, GATED);
  else if (a.parts > 1) FORMS(PARTS);
  else FORMS(PLAIN);
#undef FORMS
#undef GO
  DS_CHECK_LAUNCH();
  if (a.parts > 1) {
    const int64_t pieces = (int64_t)a.M * a.N / 8;
    hipLaunchKernelGGL(wide_sum_kernel, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, st, a.part, a.c, pieces, a.parts);
    DS_CHECK_LAUNCH();
  }
  return 0;
}

}  // namespace

// Forces tiles of 256, 192 or 128 rows, over all rows, and so many parts of K (0: one) for the calling thread's products; 0: by the rule
extern "C" void ds_wide_gemm_tune(int rows, int parts) { g_rows = rows, g_parts = parts; }

// (narrow_gemm.hip)
extern "C" int ds_narrow_tiles_pay(int64_t, int64_t, int64_t, int, int);

// Steps of a tile; offsets within a tile's rows of C, of which a quarter of 32 bits marks none
static bool takes(int64_t N, int64_t K, int a_along, int b_along) { return (K + 63) / 64 >= STEPS && N < 1 << 21 && (a_along || !b_along); }

// Whether the kernel takes a product that ds_narrow_gemm_ok has, and is the fastest way: the estimate comes to a rate that neither the library's call nor the
// narrow tiles reach on average. 1200 products of 400 layers at random (profiles/wide_products_at_random.csv), time here over the time before, in the
// mean, by the rate of the estimate in TF/s: y 800 - 1000 0.92, 1000 - 1500 0.86, below 800 1.43; dX 800 - 1000 0.94, 1000 - 1500 0.81, below 1.8; dW 600 -
// 800 0.90, 800 - 1500 0.82, below 1.4. Rows of 8192 and more that few tokens share come from memory, which the library waits for better (us here (there):
// y, 640 by [12288, 11008] 179 (158), 467 by [10240, 8192] 78 (71), dX, 697 by [28672, 8192] 344 (301)).
// Of dX, where K is in parts and the narrow tiles do not take it either, the library has few tiles, too, and a lower line stands, also for results of 2^19 (us there,
// here: 1821 by [22016, 512] 139, 47; 1452 by [11264, 768] 90, 36; 2306 by [11264, 1024] 95, 58; by a line of 550 1629 by [8192, 1024] 38, 44; beside narrow tiles 1556 by
// [5632, 2048] 40, 46). dW in parts beside narrow tiles, which are one round of those, is no gain (6464 tokens by [2048, 2048] 50, 56; 7848 by [2048, 1920] 58, 64; 6720 by
// [8192, 488] 57, 56); from 8192 tokens on, where a layer makes copies for the library instead,
// it takes 0.51 of the time (140 at random: 8512 by [2048, 2048] 100, 68).
static int pays(int64_t M, int64_t N, int64_t K, int a_along, int b_along, bool parts_too) {
  if (!takes(N, K, a_along, b_along)) return 0;
  if (g_rows) return 1;
  if ((a_along ? M : K) < 400 || M * N < 1 << 19 || (a_along && M <= 1152 && K >= 8192)) return 0;
  const Plan p = plan_of(M, N, K, parts_too);
  if (M * N < 1 << 20 && p.parts == 1) return 0;
  int line = b_along ? 1000 : a_along ? 950 : 800;
  if (p.parts > 1 && !b_along) {
    const bool narrow = (a_along || K < 8192) && ds_narrow_tiles_pay(M, N, K, a_along, b_along);
    if (narrow && !a_along) return 0;
    if (!narrow && a_along) line = 650;
  }
  return 2e-6 * M * N * K >= p.time * line;
}
extern "C" int ds_wide_gemm_pays(int64_t M, int64_t N, int64_t K, int a_along, int b_along) { return pays(M, N, K, a_along, b_along, true); }
// The same for ds_wide_gated, whose inner dimension stays whole (us in one launch, and the product in parts and the activation: 3939 tokens by 2 x 512 of 12992
// 111, 103; 6116 by 2 x 256 of 15360 131, 85; accepted, 4096 by 2 x 1024 of 8192 99, 107, 8192 by 2 x 14336 of 4096 1272, 1401)
extern "C" int ds_wide_gated_pays(int64_t M, int64_t N, int64_t K) { return pays(M, 2 * N, K, 1, 1, false); }

namespace {
// gate: N weight rows, half of them the gate's, make N / 2 columns of C
int run(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_along, int b_along, bool gate, void* part, hipStream_t st) {
  if (!takes(N, K, a_along, b_along)) return (int)hipErrorInvalidValue;
  const Plan p = plan_of(M, N, K, !gate);
  if (p.parts > 1 && !part) return (int)hipErrorInvalidValue;
  const int64_t ar = a_along ? M : K, ac = a_along ? K : M, br = b_along ? N : K, bc = b_along ? K : N;
  const int64_t of = gate ? 2 : 1, cols = N / of, cut = p.n < N ? p.n / of : cols;  // C's columns, those of the first part
  WideArgs a{(const bf16*)A, (const bf16*)B, (bf16*)C, (int)p.m, (int)cut, (int)K, (int)cols, (uint32_t)lda, (uint32_t)ldb,
             (uint32_t)(((ar - 1) * lda + ac) * 2), (uint32_t)(((br - 1) * ldb + bc) * 2), 0, (int)cols, p.parts, p.deep, (float*)part};
  int rc = launch(a, p.rows, a_along, b_along, gate, st);
  if (rc || (p.m == M && cut == cols)) return rc;
  // the second part: rows of A and C from m on, or B's and C's columns from n on
  const int64_t m = p.m < M ? p.m : 0, n = cut < cols ? cut : 0, oa = m * (a_along ? lda : 1), ob = n * (b_along ? ldb : 1);
  a.a += oa;
  a.b += ob;
  a.c += m * cols + n;
  a.M = (int)(M - m);
  a.N = (int)(cols - n);
  a.abytes -= (uint32_t)(oa * 2);
  a.bbytes -= (uint32_t)(ob * 2);
  return launch(a, p.other, a_along, b_along, gate, st);
}
}  // namespace

// How C [M, N] over K (gated: M by N weight rows) goes out: rows of a tile; those of the second part's tiles (0: one part); where that begins, in rows or in
// columns; parts of K
extern "C" void ds_wide_plan(int64_t M, int64_t N, int64_t K, int gated, int64_t* to) {
  const Plan p = plan_of(M, N, K, !gated);
  to[0] = p.rows, to[1] = p.other, to[2] = p.m, to[3] = p.n, to[4] = p.parts;
}

// Bytes of scratch memory that the product wants (0: none)
extern "C" int64_t ds_wide_gemm_scratch(int64_t M, int64_t N, int64_t K) {
  const int parts = plan_of(M, N, K).parts;
  return parts > 1 ? parts * M * N * 4 : 0;
}

// C [M, N] as ds_narrow_gemm takes it. part: ds_wide_gemm_scratch bytes
extern "C" int ds_wide_gemm(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_along, int b_along,
                            void* part, hipStream_t st) {
  return run(A, B, C, M, N, K, lda, ldb, a_along, b_along, false, part, st);
}

// y [M, N] = silu(x g^T) (x u^T) of w [2 N, K], g before u; rows of x lda apart, of w K. Where ds_narrow_gemm_ok has the product by w and ds_wide_gated_pays this.
extern "C" int ds_wide_gated(const void* X, const void* W, void* Y, int64_t M, int64_t N, int64_t K, int64_t lda, hipStream_t st) {
  return run(X, W, Y, M, 2 * N, K, lda, K, 1, 1, true, nullptr, st);
}
