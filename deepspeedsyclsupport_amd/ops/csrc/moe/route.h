// The choice of a token's experts from its router logits (expert_route.hip: routing by itself, pre_norm.hip: behind the norm).
#pragma once
#include "ds_hip.h"

namespace {

constexpr int MAXE = 256, MAXK = 64;

struct RouteArgs {
  int T, W, E, K, groups, keep, sigmoid, best;   // best: members that count for a group, 1 or 2
  float scale;
  int* experts;      // [T, K]
  float* weights;    // [T, K]
  int* counts;       // [E], zero before; null: no lists wanted
  int* slots;        // [T, K]: place of the pair within its expert's
};

// The largest of the wave's values, in registers alone (a step of the ladder is one instruction with a lane move; a shuffle goes
// through LDS)
template <int CTRL, int ROWS>
__device__ __forceinline__ float max_step(float v) {
  const int b = __float_as_int(v);
  return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(b, b, CTRL, ROWS, 0xf, false)));
}
__device__ __forceinline__ float max_all(float v) {
  v = max_step<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8: lane 15 of each 16 has their largest
  v = max_step<0x112, 0xf>(v);
  v = max_step<0x114, 0xf>(v);
  v = max_step<0x118, 0xf>(v);
  v = max_step<0x142, 0xa>(v);  // lane 15 to the next 16, lane 31 to the upper half
  v = max_step<0x143, 0xc>(v);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// One wave: logits z [E] of a token in LDS (overwritten), gs scratch [groups], up to 64 NI experts. Lane k gets choice k and, with
// hist, its place among the workgroup's pairs of that expert.
template <int NI>
__device__ __forceinline__ void choose(float* z, float* gs, int tok, const RouteArgs& a, int* hist, int& my_e, int& my_slot) {
  const int lane = threadIdx.x & 63, E = a.E, per = E / a.groups;
  float s[NI], mx = -INFINITY, den = 0.f;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    s[i] = lane + 64 * i < E ? z[lane + 64 * i] : -INFINITY;
    mx = fmaxf(mx, s[i]);
  }
  if (a.sigmoid) {
#pragma unroll
    for (int i = 0; i < NI; ++i) s[i] = 1.f / (1.f + expf(-s[i]));
  } else {
    mx = max_all(mx);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      s[i] = lane + 64 * i < E ? expf(s[i] - mx) : 0.f;
      den += s[i];
    }
    den = wave_sum(den);
#pragma unroll
    for (int i = 0; i < NI; ++i) s[i] /= den;
  }
  if (a.keep < a.groups) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (lane + 64 * i < E) z[lane + 64 * i] = s[i];
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int g = lane; g < a.groups; g += 64) {
      float b = 0.f, c = 0.f;
      for (int e = g * per; e < (g + 1) * per; ++e) {
        c = fmaxf(c, fminf(b, z[e]));
        b = fmaxf(b, z[e]);
      }
      gs[g] = a.best == 2 ? b + c : b;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int e = lane + 64 * i;
    if (e >= E) {
      s[i] = -1.f;
    } else if (a.keep < a.groups) {
      const int g = e / per;
      const float b = gs[g];
      int better = 0;
      for (int o = 0; o < a.groups; ++o) better += gs[o] > b || (gs[o] == b && o < g);
      if (better >= a.keep) s[i] = -1.f;
    }
  }
  float mine = 0.f, sum = 0.f;
  for (int k = 0; k < a.K; ++k) {
    float bv = -1.f;
    int be = E - 1;  // logits that are not numbers choose nothing: stay in bounds
#pragma unroll
    for (int i = 0; i < NI; ++i) bv = fmaxf(bv, s[i]);
    bv = max_all(bv);
    if (bv > -1.f) {
#pragma unroll
      for (int i = NI - 1; i >= 0; --i)
        if (const uint64_t at = __ballot(s[i] == bv)) be = 64 * i + __builtin_ctzll(at);
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if (be == lane + 64 * i) s[i] = -1.f;
    }
    sum += bv;
    if (lane == k) {
      mine = bv;
      my_e = be;
    }
  }
  if (lane < a.K) {
    const int64_t i = (int64_t)tok * a.K + lane;
    a.experts[i] = my_e;
    a.weights[i] = mine / (sum + 1e-20f) * a.scale;
    if (hist) my_slot = atomicAdd(hist + my_e, 1);
  }
}

static inline bool route_args_ok(const RouteArgs& a) {
  return a.W > 0 && a.E > 0 && a.E <= MAXE && a.K > 0 && a.K <= MAXK && a.groups > 0 && a.E % a.groups == 0 && a.keep > 0 &&
         a.keep <= a.groups && a.K <= a.keep * (a.E / a.groups) && !a.counts == !a.slots && a.best >= 1 && a.best <= 2;
}

}  // namespace
