// Plain fp32 residual with RMS norms on the sublayers' inputs and, optionally, on their gated outputs, CDNA4 (gfx950). One launch
// per sublayer boundary:
//   1. y: a sublayer's output, or sum_k w[t, k] y[row(t, k)] + base[t] (the weighted outputs of a token's experts, and of one
//      that every token takes);
//   2. (POST) y <- sigmoid(gate + gate bias) y, if there is a gate, then y <- y / rms(y) * post weight;
//   3. x <- x + y, or, at the start of the model, x <- the token's embedding row times a constant;
//   4. the next sublayer's input x / rms(x) * w in the storage type (without w: x itself).
//   5. for a few tokens in bf16, if that sublayer routes them to experts: the routing (../moe/route.h).
// With a row list (the rows whose logits are wanted) only those rows are normed and x stays as it is.
//
// HBM-bound: every operand is read once with 16-byte accesses, the row stays in registers between the passes; widths that are
// no multiple of 8 take a plain version that goes over the row again.
#include "../moe/route.h"

namespace {

struct PreArgs {
  float* x;            // [T, W]
  const void* y;       // [T, W] or [T * K, W]
  const float* yw;     // [T, K] or null
  const int* yrow;     // [T, K]: rows of y; null: t * K + k
  const void* base;    // [T, W] or null (with yw)
  int K;
  const float* post;   // [W] or null
  const void* gate;    // [T, W] or null (with post), rows ldg apart
  const float* gate_b; // [W]
  int64_t ldg;
  const int* ids;      // [T]
  const void* embed;   // [V, W]
  float mult;          // of the embedding
  const int* rows;
  const float* w;      // [W] or null
  void* out;
  int W;
  float eps;
};

// What the sublayer before leaves for columns c .. c + 7 of token t
template <typename T>
__device__ __forceinline__ void added(const PreArgs& a, int64_t t, int c, float (&v)[8]) {
  const T* y = (const T*)a.y;
  if (!a.yw) {
    Vec8<T>::load(y + t * a.W + c, v);
    return;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = 0.f;
#pragma unroll 4
  for (int k = 0; k < a.K; ++k) {
    const int64_t e = t * a.K + k, r = a.yrow ? a.yrow[e] : e;
    float u[8];
    Vec8<T>::load(y + r * a.W + c, u);
    const float g = a.yw[e];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = fmaf(g, u[j], v[j]);
  }
  if (a.base) {
    float u[8];
    Vec8<T>::load((const T*)a.base + t * a.W + c, u);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] += u[j];
  }
}

__device__ __forceinline__ float gated(float y, float g) { return y / (1.f + expf(-g)); }

// NT threads per token, E x 8 elements per thread; with a norm, xv is left as it is stored but for the rounding
template <typename T, int NT, int E, bool POST>
__device__ __forceinline__ void pre_norm_row(const PreArgs& a, float* red, float (&xv)[E][8]) {
  const int r = blockIdx.x, tid = threadIdx.x, W = a.W;
  const int64_t src = a.rows ? a.rows[r] : r;
  float* xr = a.x + src * W;
  float ss = 0.f;
  float yv[POST ? E : 1][8], post[POST ? E : 1][8];
  if constexpr (POST) {
    float sy = 0.f;
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int c = (tid + i * NT) * 8;
      if (c >= W) continue;
      float g[8], b[8];
      if (a.gate) {
        Vec8<T>::load((const T*)a.gate + src * a.ldg + c, g);
        Vec8<float>::load(a.gate_b + c, b);
      }
      Vec8<float>::load(a.post + c, post[i]);
      Vec8<float>::load(xr + c, xv[i]);
      added<T>(a, src, c, yv[i]);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (a.gate) yv[i][j] = gated(yv[i][j], g[j] + b[j]);
        sy = fmaf(yv[i][j], yv[i][j], sy);
      }
    }
    const float ry = 1.f / sqrtf(block_sum(sy, red) / (float)W + a.eps);
#pragma unroll
    for (int i = 0; i < E; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) yv[i][j] *= ry * post[i][j];
  }
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const int c = (tid + i * NT) * 8;
    if (c >= W) continue;
    if constexpr (POST) {
#pragma unroll
      for (int j = 0; j < 8; ++j) xv[i][j] += yv[i][j];
    } else if (a.embed) {
      Vec8<T>::load((const T*)a.embed + (int64_t)a.ids[r] * W + c, xv[i]);
#pragma unroll
      for (int j = 0; j < 8; ++j) xv[i][j] *= a.mult;
    } else {
      float v[8];
      Vec8<float>::load(xr + c, xv[i]);
      added<T>(a, src, c, v);
#pragma unroll
      for (int j = 0; j < 8; ++j) xv[i][j] += v[j];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) ss = fmaf(xv[i][j], xv[i][j], ss);
    if (!a.rows) Vec8<float>::store(xr + c, xv[i]);
    if (!a.w) Vec8<T>::store((T*)a.out + (int64_t)r * W + c, xv[i]);
  }
  if (!a.w) return;
  const float rs = 1.f / sqrtf(block_sum(ss, red) / (float)W + a.eps);
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const int c = (tid + i * NT) * 8;
    if (c >= W) continue;
    float g[8];
    Vec8<float>::load(a.w + c, g);
#pragma unroll
    for (int j = 0; j < 8; ++j) xv[i][j] *= rs * g[j];
    Vec8<T>::store((T*)a.out + (int64_t)r * W + c, xv[i]);
  }
}

template <typename T, int NT, int E, bool POST>
__global__ void __launch_bounds__(NT) pre_norm_kernel(PreArgs a) {
  __shared__ float red[NT / 64];
  float xv[E][8];
  pre_norm_row<T, NT, E, POST>(a, red, xv);
}

// The same and the routing of the token (bf16, up to 8192 columns): a workgroup per token, two experts' logits a wave at a time. A
// launch of its own for the routing of a few tokens is one workgroup that reads all of the router and their rows, 35 bytes a
// nanosecond; here every token's reads the router (32 experts of 2048: 128 KB, 3 us, from L2 after the first) while the norm's
// operands are on their way, and the row is at hand in LDS. The logits are sums of exact products in fp32, of the row as it is
// stored. us, both launches and one:
//     1 token of 2048 among 32 experts 9.9 and 6.7, 16 12.6 and 7.0, 128 13.1 and 7.4, 256 with lists 18.0 and 14.0;
//     16 of 4096 among 32 18.2 and 8.3, among 128 44.5 and 17.5, among 256 89 and 29; 16 of 2048 among 16 9.4 and 5.9
template <bool POST>
__global__ void __launch_bounds__(1024) pre_norm_route_kernel(PreArgs a, RouteArgs ra, const bf16* __restrict__ router) {
  constexpr int NT = 1024, STEP = 2048;
  __shared__ float red[NT / 64], z[MAXE], gs[MAXE];
  __shared__ f32x4 lo[NT], hi[NT];  // the row's pieces of 8
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, W = a.W;
  const int C = (W + STEP - 1) / STEP, items = (ra.E + 31) / 32 * C;
  struct Piece {
    bf16x8 y[2][4];
  };
  auto load = [&](int it) {
    Piece p;
    const int e = 2 * (wave + it / C * 16), c = it % C * STEP + 8 * lane;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        p.y[j][u] = *reinterpret_cast<const bf16x8*>(router + (int64_t)min(e + j, ra.E - 1) * W + min(c + 512 * u, W - 8));
    return p;
  };
  Piece now = load(0);
  float xv[1][8];
  pre_norm_row<bf16, NT, 1, POST>(a, red, xv);
  const bool in = tid * 8 < W;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    lo[tid][j] = in ? (float)(bf16)xv[0][j] : 0.f;
    hi[tid][j] = in ? (float)(bf16)xv[0][4 + j] : 0.f;
  }
  __syncthreads();
  float acc[2] = {0.f, 0.f};
  for (int it = 0; it < items; ++it) {
    const Piece p = now;
    if (it + 1 < items) now = load(it + 1);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int at = it % C * (STEP / 8) + 64 * u + lane;
      const f32x4 a0 = lo[at], a1 = hi[at];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[j] = fmaf((float)p.y[j][u][i], a0[i], acc[j]);
          acc[j] = fmaf((float)p.y[j][u][4 + i], a1[i], acc[j]);
        }
    }
    if (it % C == C - 1) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float s = wave_sum(acc[j]);
        const int e = 2 * (wave + it / C * 16) + j;
        if (lane == 0 && e < ra.E) z[e] = s;
        acc[j] = 0.f;
      }
    }
  }
  __syncthreads();
  if (wave > 0) return;
  const int tok = blockIdx.x;
  int e = 0, slot = 0;
  if (ra.E <= 64) choose<1>(z, gs, tok, ra, ra.counts, e, slot);
  else if (ra.E <= 128) choose<2>(z, gs, tok, ra, ra.counts, e, slot);
  else choose<4>(z, gs, tok, ra, ra.counts, e, slot);
  if (ra.counts && lane < ra.K) ra.slots[(int64_t)tok * ra.K + lane] = slot;
}

// any width
template <typename T>
__global__ void __launch_bounds__(256) pre_norm_any_kernel(PreArgs a) {
  __shared__ float red[4];
  const int r = blockIdx.x, tid = threadIdx.x, W = a.W;
  const int64_t src = a.rows ? a.rows[r] : r;
  const T* y = (const T*)a.y;
  float* xr = a.x + src * W;
  auto added_one = [&](int c) {
    float v = 0.f;
    if (!a.yw) {
      v = (float)y[src * W + c];
    } else {
      for (int k = 0; k < a.K; ++k) {
        const int64_t e = src * a.K + k;
        v = fmaf(a.yw[e], (float)y[(a.yrow ? a.yrow[e] : e) * W + c], v);
      }
      if (a.base) v += (float)((const T*)a.base)[src * W + c];
    }
    return a.gate ? gated(v, (float)((const T*)a.gate)[src * a.ldg + c] + a.gate_b[c]) : v;
  };
  float ry = 1.f;
  if (a.post) {
    float sy = 0.f;
    for (int c = tid; c < W; c += 256) {
      const float v = added_one(c);
      sy = fmaf(v, v, sy);
    }
    ry = 1.f / sqrtf(block_sum(sy, red) / (float)W + a.eps);
  }
  auto sum = [&](int c) {
    if (a.embed) return (float)((const T*)a.embed)[(int64_t)a.ids[r] * W + c] * a.mult;
    return xr[c] + added_one(c) * (a.post ? ry * a.post[c] : 1.f);
  };
  float ss = 0.f;
  for (int c = tid; c < W; c += 256) {
    const float v = sum(c);
    ss = fmaf(v, v, ss);
    if (!a.rows) xr[c] = v;
  }
  const float rs = 1.f / sqrtf(block_sum(ss, red) / (float)W + a.eps);
  for (int c = tid; c < W; c += 256)  // (each thread re-reads what it wrote)
    ((T*)a.out)[(int64_t)r * W + c] = (T)((a.rows ? sum(c) : xr[c]) * (a.w ? rs * a.w[c] : 1.f));
}

template <typename T>
int pre_norm(const PreArgs& a, int n, hipStream_t st) {
#define GO(NT, E)                                                                                 {                                                                                                 if (a.post) hipLaunchKernelGGL((pre_norm_kernel<T, NT, E, true>), dim3(n), dim3(NT), 0, st, a);     else hipLaunchKernelGGL((pre_norm_kernel<T, NT, E, false>), dim3(n), dim3(NT), 0, st, a);     }
  const int W = a.W;
  if (W % 8 == 0 && W <= 16384 && a.ldg % 8 == 0 && ((uintptr_t)a.gate & 15) == 0) {
    if (W <= 512) GO(64, 1)
    else if (n <= 512 && W <= 4096) GO(512, 1)
    else if (n <= 512 && W <= 8192) GO(1024, 1)
    else if (n <= 512) GO(1024, 2)
    else if (W <= 2048) GO(256, 1)
    else if (W <= 4096) GO(256, 2)
    else if (W <= 8192) GO(256, 4)
    else GO(256, 8)
  } else {
    hipLaunchKernelGGL((pre_norm_any_kernel<T>), dim3(n), dim3(256), 0, st, a);
  }
#undef GO
  DS_CHECK_LAUNCH();
  return 0;
}

}  // namespace

// y [T, W] (yw null), or y [.., W] with yw [T, K], optionally yrow [T, K] and base [T, W]; or ids and embed, times mult. post:
// y's norm, with gate [T, W] (rows ldg apart) and gate_b or without. w null: no norm of the sum. -> out [n, W]
extern "C" int ds_pre_norm(float* x, const void* y, const float* yw, const int* yrow, const void* base, int K, const float* post,
                           const void* gate, int64_t ldg, const float* gate_b, const int* ids, const void* embed, float mult,
                           const int* rows, int n, const float* w, void* out, int W, float eps, int dtype, hipStream_t st) {
  if (n <= 0) return 0;
  if (W <= 0 || (!y == !embed) || (embed && (!ids || rows || post)) || (yw && K <= 0) || (gate && (!post || !gate_b || ldg < W)) ||
      (base && !yw))
    return (int)hipErrorInvalidValue;
  const PreArgs a{x, y, yw, yrow, base, K, post, gate, gate_b, gate ? ldg : 0, ids, embed, mult, rows, w, out, W, eps};
  if (dtype == DS_F32) return pre_norm<float>(a, n, st);
  if (dtype == DS_BF16) return pre_norm<bf16>(a, n, st);
  return (int)hipErrorInvalidValue;
}

// Up to a token a CU, or, where the experts are many and so the gain is large, two. With lists every pair adds 1 to its expert's
// count, 60 ns each that an expert's share of them waits for one another: 384 tokens of 1024, two of 8 experts each (96 pairs an
// expert) take 16.1 us for 12.5, 384 of 2048 among 16 (48) 16.6 for 15.1, 512 among 64 (64) 23 for 25.
extern "C" int ds_pre_norm_route_ok(int n, int W, int E, int top, int lists) {
  const bool many = E >= 64;
  return W % 8 == 0 && W <= 8192 && n <= (many ? 512 : 256) && (!lists || (int64_t)n * top <= (many ? 64 : 32) * E);
}

// The same over all rows of x [n, W] bf16 with a norm (w), and ds_route of what comes out
extern "C" int ds_pre_norm_route(float* x, const void* y, const float* yw, const int* yrow, const void* base, int K, const float* post,
                                 const void* gate, int64_t ldg, const float* gate_b, int n, const float* w, void* out, int W, float eps,
                                 const void* router, int* experts, float* weights, int* counts, int* slots, int E, int top, int groups,
                                 int keep, int sigmoid, int best, float scale, hipStream_t st) {
  if (n <= 0) return 0;
  const RouteArgs ra{n, W, E, top, groups, keep, sigmoid, best, scale, experts, weights, counts, slots};
  if (W % 8 || W > 8192 || !y || !w || !router || (yw && K <= 0) || (gate && (!post || !gate_b || ldg < W)) || (base && !yw) ||
      (gate && (ldg % 8 || ((uintptr_t)gate & 15))) || !route_args_ok(ra))
    return (int)hipErrorInvalidValue;
  const PreArgs a{x, y, yw, yrow, base, K, post, gate, gate_b, gate ? ldg : 0, nullptr, nullptr, 1.f, nullptr, w, out, W, eps};
  if (post) hipLaunchKernelGGL((pre_norm_route_kernel<true>), dim3(n), dim3(1024), 0, st, a, ra, (const bf16*)router);
  else hipLaunchKernelGGL((pre_norm_route_kernel<false>), dim3(n), dim3(1024), 0, st, a, ra, (const bf16*)router);
  DS_CHECK_LAUNCH();
  return 0;
}
