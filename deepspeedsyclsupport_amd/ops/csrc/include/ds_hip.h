// Common CDNA4 (gfx950) device helpers for deepspeedsyclsupport_amd kernels.
// Wave64 everywhere: reductions use 64-lane shuffles / DPP-friendly xor patterns, block sizes are multiples of 64.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define DS_WAVE 64

typedef __bf16 bf16;
typedef _Float16 fp16;
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 fp16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 fp16x8 __attribute__((ext_vector_type(8)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// dtype tags shared with the Python side (ops/native.py DTYPE_CODE)
enum DsDtype : int { DS_F32 = 0, DS_BF16 = 1, DS_F16 = 2 };

// ---------------------------------------------------------------- 8-wide vector load/store in any dtype
// Loads 8 consecutive elements (16 B for bf16/fp16, 32 B for fp32) and widens to fp32.
template <typename T> struct Vec8;
template <> struct Vec8<float> {
  __device__ __forceinline__ static void load(const float* p, float (&v)[8]) {
    f32x4 a = *reinterpret_cast<const f32x4*>(p);
    f32x4 b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) { v[i] = a[i]; v[i + 4] = b[i]; }
  }
  __device__ __forceinline__ static void store(float* p, const float (&v)[8]) {
    f32x4 a, b;
#pragma unroll
    for (int i = 0; i < 4; ++i) { a[i] = v[i]; b[i] = v[i + 4]; }
    *reinterpret_cast<f32x4*>(p) = a;
    *reinterpret_cast<f32x4*>(p + 4) = b;
  }
};
template <> struct Vec8<bf16> {
  __device__ __forceinline__ static void load(const bf16* p, float (&v)[8]) {
    bf16x8 a = *reinterpret_cast<const bf16x8*>(p);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (float)a[i];
  }
  __device__ __forceinline__ static void store(bf16* p, const float (&v)[8]) {
    f32x4 lo, hi;
#pragma unroll
    for (int i = 0; i < 4; ++i) { lo[i] = v[i]; hi[i] = v[i + 4]; }
    bf16x4 a = __builtin_convertvector(lo, bf16x4);
    bf16x4 b = __builtin_convertvector(hi, bf16x4);
    bf16x8 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) { r[i] = a[i]; r[i + 4] = b[i]; }
    *reinterpret_cast<bf16x8*>(p) = r;
  }
};
template <> struct Vec8<fp16> {
  __device__ __forceinline__ static void load(const fp16* p, float (&v)[8]) {
    fp16x8 a = *reinterpret_cast<const fp16x8*>(p);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (float)a[i];
  }
  __device__ __forceinline__ static void store(fp16* p, const float (&v)[8]) {
    fp16x8 r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = (fp16)v[i];
    *reinterpret_cast<fp16x8*>(p) = r;
  }
};

template <typename T> __device__ __forceinline__ float to_f32(T x) { return (float)x; }
template <typename T> __device__ __forceinline__ T from_f32(float x) { return (T)x; }

// ---------------------------------------------------------------- clamped gated activation
// g sigmoid(alpha g) (u + shift) with g = min(gate, limit), u = clamp(up, -limit, limit). As the epilogue of a gated
// decode product it is activation code DS_ACT_CLAMPED_GLU with alpha 1.702 and shift 1.
#define DS_ACT_CLAMPED_GLU 5
// activation codes from here on: code - DS_ACT_UNARY applied to the result of an ungated decode product
#define DS_ACT_UNARY 16
__device__ __forceinline__ float act_any(int a, float x) {
  switch (a) {
    case 0: return x / (1.f + __expf(-x));  // silu
    case 1: return 0.5f * x * (1.f + tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x)));
    case 2: return 0.5f * x * (1.f + erff(x * 0.7071067811865476f));
    case 3: return fmaxf(x, 0.f);
    default: return x;
  }
}
__device__ __forceinline__ float clamped_glu_f(float g, float u, float limit, float alpha = 1.702f, float shift = 1.f) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.f + expf(-alpha * g)) * (u + shift);
}

// ---------------------------------------------------------------- wave64 / block reductions
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
// Block sum for up to 1024 threads. `red` must hold >= blockDim/64 floats. Result broadcast to all threads.
__device__ __forceinline__ float block_sum(float v, float* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float r = 0.f;
  for (int i = 0; i < nw; ++i) r += red[i];
  return r;
}
__device__ __forceinline__ float block_max(float v, float* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float r = -INFINITY;
  for (int i = 0; i < nw; ++i) r = fmaxf(r, red[i]);
  return r;
}

// ---------------------------------------------------------------- launch helpers
#define DS_CHECK_LAUNCH() do { hipError_t e__ = hipGetLastError(); if (e__ != hipSuccess) return (int)e__; } while (0)

static inline int ds_grid_for(int64_t work_items, int block, int max_blocks = 256 * 8) {
  int64_t g = (work_items + block - 1) / block;
  if (g < 1) g = 1;
  if (g > max_blocks) g = max_blocks;
  return (int)g;
}

// XCD-aware bijective remap of a linear workgroup id (guide §5 "XCD swizzle must be bijective"):
// blocks b and b+8 share an XCD under round-robin dispatch, so give each XCD a contiguous chunk of tiles.
__device__ __forceinline__ int xcd_remap(int orig, int nwg) {
  const int q = nwg / 8, r = nwg % 8, xcd = orig % 8;
  return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + orig / 8;
}

// Workgroup -> (head, one of its `blocks`), the first blocks of several heads before the second ones. A head stays on one XCD, whose L2 keeps its keys, where
// the heads share out evenly; else they go round the chip, or, not `round`, head by head. Four heads an XCD at a time, and the last eight to eleven together: what
// waits at the end is the last ones' short blocks (dense causal forward, us, one / four / eight / all heads at a time and this: 8 x 4096, 32 heads 1151, 1128,
// 1146, 1454, 1155, not causal 1942, 1950, 2001, 2971, 2008, hence there head by head; 2 x 4096 305, 264, 264, 265, 274; 8 x 512, 16 heads 24.1, 24.6, 20.8, 21.1, 20.5; 5 x 1500, 8 heads
// 47.0, 47.4, 41.6, 42.0, 40.8; backward 8 x 4096, 32 heads 4001, 3931, 3992, 4300, 3971, 1 x 4096, 20 heads 626, 513, 464, 402, 402).
__device__ __forceinline__ void by_block(int heads, int blocks, bool round, int& head, int& block) {
  if (heads % 8 && !round) {
    const int at = xcd_remap(blockIdx.x, gridDim.x);
    head = at / blocks;
    block = at % blocks;
    return;
  }
  int at = blockIdx.x, h = heads, first = 0, width = 32;
  if (heads % 8 == 0) {
    h = heads / 8;
    first = at % 8 * h;
    at /= 8;
    width = 4;
  }
  const int group = min(at / (width * blocks), max(h / width - 2, 0));
  const int here = group < h / width - 2 ? width : h - group * width;
  at -= group * width * blocks;
  head = first + group * width + at % here;
  block = at / here;
}

// Tile of a transposing kernel's workgroup: an XCD's share in columns of 16 tiles, row by row. Single columns of tiles read 128 bytes of each row
// (us on data that a product has just written, 8192 x 11008 / 8192 x 8192: transpose16 70 / 56, this 64 / 53, with `load_once` 63 / 45; gated_fwd_t
// 147 / 104, 131 / 96, 120 / 92; gated_bwd_t 266 / 192, 244 / 181, 224 / 179; up to 3000 rows of 5632 the same).
__device__ __forceinline__ void transpose_tile(int tiles_r, int tiles_c, int& tr, int& tc) {
  const int id = xcd_remap(blockIdx.x, gridDim.x), col = id / (tiles_r * 16) * 16, w = min(16, tiles_c - col), in = id - col * tiles_r;
  tr = in / w;
  tc = col + in % w;
}

// 16 bytes that this kernel has no second use for
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4 load_once(const void* p) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p)); }
