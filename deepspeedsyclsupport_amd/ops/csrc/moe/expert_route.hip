// Routing of mixture-of-experts layers with grouped experts, CDNA4 (gfx950).
//
//  * route: router logits in fp32 (bf16 operands through the matrix cores, or plain fp32 products), scores (the softmax over all
//    experts, or every expert's sigmoid), the best groups of neighbouring experts (a group is as good as its best member, or its
//    two best together), the best experts within those, weights divided by their sum, times a constant. One launch: the logits
//    of a tile of tokens never leave LDS. Ties go to the lower index.
//  * place: the (token, choice) pairs sorted by expert, as lists for the expert products (expert_gemm.hip). The counts come
//    from the routing kernel; nothing waits for the host.
#include "route.h"

namespace {

template <int N>
struct Int {
  static constexpr int value = N;
};

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The workgroup's pairs take a run of every expert's places; afterwards hist holds where it begins
__device__ __forceinline__ void claim(const RouteArgs& a, int* hist) {
  __syncthreads();
  for (int e = threadIdx.x; e < a.E; e += blockDim.x)
    if (const int c = hist[e]) hist[e] = atomicAdd(a.counts + e, c);
  __syncthreads();
}

// bf16, W a multiple of 8. NW waves share the width of 16 TM tokens and up to 16 ET experts. With few tokens there is one workgroup,
// and what bounds it is a CU's path to memory (35 bytes a nanosecond) and then the chain of steps that follows; so the
// width's remainder is loaded by 4, 2 and 1 steps at a time, the waves' shares meet after two barriers, the maxima of the choice stay
// in registers, and places go to memory once. us before and after: 16 tokens of 2048 among 32 experts 13.2 and 10.0, 64 tokens
// among 64 experts with lists 28 and 21, 64 of 4096 among 128 73 and 43, 8192 of 4096 among 32 43 and 34. (Whole cache lines a wave,
// or all loads held ahead of the products, measured the same.)
template <int ET, int TM, int NW>
__global__ void __launch_bounds__(64 * NW) route_mfma_kernel(const bf16* __restrict__ h, const bf16* __restrict__ rw,
                                                             RouteArgs a) {
  constexpr int TOK = 16 * TM, ZP = 16 * ET + 1;
  __shared__ float z[TOK * ZP];
  __shared__ f32x4 red[NW / 2][TM * ET][64];
  __shared__ float gs[NW][16 * ET];
  __shared__ int hist[MAXE];
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, q4 = lane >> 4, w = tid >> 6;
  const int t0 = blockIdx.x * TOK, n = min(TOK, a.T - t0);
  for (int e = tid; e < MAXE; e += 64 * NW) hist[e] = 0;
  f32x4 acc[TM][ET];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int e = 0; e < ET; ++e) acc[m][e] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16 *hp[TM], *wp[ET];
#pragma unroll
  for (int m = 0; m < TM; ++m) hp[m] = h + (int64_t)(t0 + min(16 * m + l16, n - 1)) * a.W;
#pragma unroll
  for (int e = 0; e < ET; ++e) wp[e] = rw + (int64_t)min(16 * e + l16, a.E - 1) * a.W;
  // U steps of 32 of the width: all their loads, then the products
  auto steps = [&](auto count, int k0, bool tail) {
    constexpr int U = decltype(count)::value;
    bf16x8 x[U][TM], y[U][ET];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 32 * NW * u + 8 * q4, kc = tail ? min(k, a.W - 8) : k;
#pragma unroll
      for (int e = 0; e < ET; ++e) y[u][e] = *reinterpret_cast<const bf16x8*>(wp[e] + kc);
#pragma unroll
      for (int m = 0; m < TM; ++m) x[u][m] = *reinterpret_cast<const bf16x8*>(hp[m] + kc);
      if (tail && k >= a.W) {  // the last step may reach past the width
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
          for (int j = 0; j < 8; ++j) x[u][m][j] = (bf16)0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int e = 0; e < ET; ++e) acc[m][e] = mfma(y[u][e], x[u][m], acc[m][e]);
  };
  constexpr int U = ET <= 2 ? 8 : ET <= 4 ? 4 : 2;
  const int whole = a.W / 32;
  int k = w;
  for (; k + NW * (U - 1) < whole; k += NW * U) steps(Int<U>{}, 32 * k, false);
  if constexpr (U == 8)
    if (k + NW * 3 < whole) {
      steps(Int<4>{}, 32 * k, false);
      k += NW * 4;
    }
  if constexpr (U >= 4)
    if (k + NW < whole) {
      steps(Int<2>{}, 32 * k, false);
      k += NW * 2;
    }
  if (k < whole) steps(Int<1>{}, 32 * k, false);
  if (a.W % 32 && whole % NW == w) steps(Int<1>{}, 32 * whole, true);
  // the waves' shares: pairs of them in their registers, the rest spread over all threads, always in the same order
  constexpr int H = NW / 2;
  if (w >= H) {
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int e = 0; e < ET; ++e) red[w - H][m * ET + e][lane] = acc[m][e];
  }
  __syncthreads();
  if (w < H) {
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int e = 0; e < ET; ++e) red[w][m * ET + e][lane] += acc[m][e];
  }
  __syncthreads();
  for (int i = tid; i < TM * ET * 64; i += 64 * NW) {
    const int c = i / 64, m = c / ET, e = c % ET;  // lane = tid % 64 throughout
    f32x4 v[H];
#pragma unroll
    for (int j = 0; j < H; ++j) v[j] = red[j][c][lane];
#pragma unroll
    for (int half = H / 2; half >= 1; half /= 2)
#pragma unroll
      for (int j = 0; j < half; ++j) v[j] += v[j + half];
#pragma unroll
    for (int r = 0; r < 4; ++r)  // token 16 m + l16, expert 16 e + 4 q4 + r
      z[(16 * m + l16) * ZP + 16 * e + 4 * q4 + r] = v[0][r];
  }
  __syncthreads();
  int my_e[TOK / NW], my_slot[TOK / NW];
#pragma unroll
  for (int j = 0; j < TOK / NW; ++j) {
    const int i = w + NW * j;
    if (i < n) choose<(ET + 3) / 4>(z + i * ZP, gs[w], t0 + i, a, a.counts ? hist : nullptr, my_e[j], my_slot[j]);
  }
  if (!a.counts) return;
  claim(a, hist);
#pragma unroll
  for (int j = 0; j < TOK / NW; ++j) {
    const int i = w + NW * j;
    if (i < n && lane < a.K) a.slots[(int64_t)(t0 + i) * a.K + lane] = hist[my_e[j]] + my_slot[j];
  }
}

// fp32, or widths the matrix kernel does not take: a workgroup per token
template <typename T>
__global__ void __launch_bounds__(256) route_any_kernel(const T* __restrict__ h, const T* __restrict__ rw, RouteArgs a) {
  __shared__ float z[MAXE], gs[MAXE];
  __shared__ int hist[MAXE];
  const int t = blockIdx.x, lane = threadIdx.x & 63;
  const T* x = h + (int64_t)t * a.W;
  for (int e = threadIdx.x; e < MAXE; e += 256) hist[e] = 0;
  for (int e = threadIdx.x >> 6; e < a.E; e += 4) {
    const T* y = rw + (int64_t)e * a.W;
    float s = 0.f;
    for (int c = lane; c < a.W; c += 64) s = fmaf((float)x[c], (float)y[c], s);
    s = wave_sum(s);
    if (lane == 0) z[e] = s;
  }
  __syncthreads();
  int my_e = 0, my_slot = 0;
  if (threadIdx.x < 64) choose<MAXE / 64>(z, gs, t, a, a.counts ? hist : nullptr, my_e, my_slot);
  if (!a.counts) return;
  claim(a, hist);
  if (threadIdx.x < a.K) a.slots[(int64_t)t * a.K + threadIdx.x] = hist[my_e] + my_slot;
}

// Exclusive prefix of counts [E] in LDS (pre[E]: the total), by the first wave
__device__ __forceinline__ void prefix(const int* counts, int E, int* pre) {
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    int c[4], s = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      c[i] = 4 * lane + i < E ? counts[4 * lane + i] : 0;
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
      if (4 * lane + i < E) pre[4 * lane + i] = at;
      at += c[i];
    }
    if (lane == 63) pre[E] = run;
  }
  __syncthreads();
}

__global__ void __launch_bounds__(256) place_kernel(const int* __restrict__ experts, const int* __restrict__ slots,
                                                    const int* __restrict__ counts, int* __restrict__ offs,
                                                    int* __restrict__ order, int* __restrict__ rows, int entries, int E) {
  __shared__ int pre[MAXE + 1];
  prefix(counts, E, pre);
  if (blockIdx.x == 0)
    for (int e = threadIdx.x; e <= E; e += 256) offs[e] = pre[e];
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= entries) return;
  const int r = pre[experts[i]] + slots[i];
  order[r] = i;
  rows[i] = r;
}

// xs[rows[t, k]] = x[t]: a workgroup per token
__global__ void __launch_bounds__(256) spread_kernel(const f32x4* __restrict__ x, const int* __restrict__ rows,
                                                     f32x4* __restrict__ xs, int W16, int K) {
  const int64_t t = blockIdx.x;
  for (int c = threadIdx.x; c < W16; c += 256) {
    const f32x4 v = x[t * W16 + c];
    for (int k = 0; k < K; ++k) xs[(int64_t)rows[t * K + k] * W16 + c] = v;
  }
}

}  // namespace

// h [T, W], router [E, W] -> experts, weights [T, K]; with counts (zero) and slots also the places of all pairs
extern "C" int ds_route(const void* h, const void* router, int* experts, float* weights, int* counts, int* slots, int T, int W,
                        int E, int K, int groups, int keep, int sigmoid, int best, float scale, int dtype, hipStream_t st) {
  if (T <= 0) return 0;
  const RouteArgs a{T, W, E, K, groups, keep, sigmoid, best, scale, experts, weights, counts, slots};
  if (!route_args_ok(a)) return (int)hipErrorInvalidValue;
  if (dtype == DS_BF16 && W % 8 == 0) {
#define GO(ET, TM, NW)                                                                                              \
  hipLaunchKernelGGL((route_mfma_kernel<ET, TM, NW>), dim3((T + 16 * TM - 1) / (16 * TM)), dim3(64 * NW), 0, st,     \
                     (const bf16*)h, (const bf16*)router, a)
    const bool wide = T > 4096;
    if (E <= 16) {
      if (wide) GO(1, 2, 8);
      else GO(1, 1, 16);
    } else if (E <= 32) {
      if (wide) GO(2, 2, 8);
      else GO(2, 1, 16);
    } else if (E <= 64) {
      if (wide) GO(4, 2, 8);
      else GO(4, 1, 8);
    } else if (E <= 128) GO(8, 1, 8);
    else GO(16, 1, 4);
#undef GO
  } else if (dtype == DS_BF16) {
    hipLaunchKernelGGL(route_any_kernel<bf16>, dim3(T), dim3(256), 0, st, (const bf16*)h, (const bf16*)router, a);
  } else if (dtype == DS_F32) {
    hipLaunchKernelGGL(route_any_kernel<float>, dim3(T), dim3(256), 0, st, (const float*)h, (const float*)router, a);
  } else {
    return (int)hipErrorInvalidValue;
  }
  DS_CHECK_LAUNCH();
  return 0;
}

// -> offs [E + 1], order [entries] (pairs by expert), rows [entries] (a pair's place in it)
extern "C" int ds_expert_place(const int* experts, const int* slots, const int* counts, int* offs, int* order, int* rows,
                               int entries, int E, hipStream_t st) {
  if (entries <= 0) return 0;
  if (E <= 0 || E > MAXE) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(place_kernel, dim3((entries + 255) / 256), dim3(256), 0, st, experts, slots, counts, offs, order, rows,
                     entries, E);
  DS_CHECK_LAUNCH();
  return 0;
}

// row_bytes: of a row, a multiple of 16
extern "C" int ds_expert_spread(const void* x, const int* rows, void* xs, int T, int K, int64_t row_bytes, hipStream_t st) {
  if (T <= 0) return 0;
  if (K <= 0 || row_bytes <= 0 || row_bytes % 16) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(spread_kernel, dim3(T), dim3(256), 0, st, (const f32x4*)x, rows, (f32x4*)xs, (int)(row_bytes / 16), K);
  DS_CHECK_LAUNCH();
  return 0;
}
