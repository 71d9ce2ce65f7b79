// A recurrent mixer's step from its projection row to its gated read-out in one launch (decoding, short portions), CDNA4 (gfx950).
//
// Per head, q, k and v are columns of the row, the first 2 half columns of q and k turned by the token's angles in pairs (i, i + half):
//     S <- a S + b k v^T;   o = c S^T q;   out = o / rms(o) * weight * act(gate columns)
// with a constant a and b = 1, or with exponential gates and a normaliser z <- a z + b k: o / (max(|c z . q|, floor) + 1e-6), a, b and
// floor from the gates' columns and the running maximum (exp_gates.hip). act: sigmoid, or silu.
//
// One workgroup per (sequence, head), so that a head's root mean square stays in it; eight lanes a value column, its state in
// registers, moved once in either direction: 128 KB of state are 3 us of a CU. q and k pass through LDS in fp32 (they are not rounded
// again), the inputs of the next token are read ahead of the work on this one. A launch is 3.5 to 4.5 us here whatever it does, so
// with few sequences the parts that this replaces (gates, split, recurrence with 64 columns a workgroup, norm: exp_gates.hip,
// decayed_scan.hip, gated_norm.hip) take twice as long; with many both are bound by the state's way in and out. us for heads of 128,
// one token a sequence, parts and one launch (constant decays; with gates):
//     1 sequence of 16 heads      9.2  4.6    12.1  5.7          64 of 16      33.8  27.1     37.9  31.6  (134 MB, 5 TB/s)
//     16 of 16                   13.1  7.4    14.9  8.4          256 of 16    111    90      140   110
//     16 of 4 of 256 x 128       12.7  6.6    16.0  7.9          16 of 32 of 64 x 64   10.3  5.1   13.1  6.1
#include "decayed_scan.h"

namespace {

enum : int { SIGMOID_AFTER = 0, SILU_AFTER = 2 };  // as in gated_norm.hip
constexpr int LPC = 8, MAX_DV = 128, MAX_NV = 8;    // lanes per column; 32 NV key rows

struct StepArgs {
  const void* proj;
  const float* cs;         // [T, half, 2]
  int half;
  const float* log_decay;  // [H], or null: gates
  int ci, cf;              // gate columns, H of either
  const float *bi, *bf;
  float cap;
  float* peak;             // [slots, H]
  float scale;
  float *state, *zstate;
  const int *list, *cu, *start, *slots;
  int gate, mode;          // output gate's first column
  const float* w;          // [H dv] or null
  float eps;
  void* out;
  int64_t ostride;
  ScanDims D;
};

__device__ __forceinline__ float sigmoid_f(float x) { return 1.f / (1.f + expf(-x)); }

template <typename T, int NV, bool NORM>
__global__ void __launch_bounds__(LPC * MAX_DV) scan_step_kernel(StepArgs a) {
  __shared__ __attribute__((aligned(16))) float qk[2][32 * NV];
  __shared__ float red[LPC * MAX_DV / 64], gates[3];
  const ScanDims& D = a.D;
  const int seq = a.list[blockIdx.x], h = blockIdx.y, g = h / (D.H / D.Hk), tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t t0 = a.cu[seq];
  const int n = a.cu[seq + 1] - (int)t0, col = tid / LPC, cc = min(col, D.dv - 1), p = tid % LPC, dks = D.dks();
  if (n <= 0) return;
  const int slot = a.slots[seq];
  const bool fresh = a.start[seq] == 0, on = col < D.dv;
  float* st = a.state + (((int64_t)slot * D.H + h) * D.dv + cc) * dks;
  f32x4 S[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k = 4 * (p + LPC * i);
    S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (!fresh && k < dks) S[i] = *reinterpret_cast<const f32x4*>(st + k);
  }
  // the normaliser: spread over a wave, whole in each; a wave reads the copy that it writes, waves beyond the copies the first one
  constexpr int NZ = NORM ? (NV + 1) / 2 : 1;
  float Z[NZ], m = 0.f;
  float* zt = nullptr;
  if constexpr (NORM) {
    zt = a.zstate + D.z_at(slot, h, wave < D.zc() ? wave * Z_COLS : 0);
#pragma unroll
    for (int i = 0; i < NZ; ++i) Z[i] = !fresh && lane + 64 * i < dks ? zt[lane + 64 * i] : 0.f;
    if (!fresh) m = a.peak[(int64_t)slot * D.H + h];
  }
  const float decay = a.log_decay ? expf(a.log_decay[h]) : 0.f, weight = a.w ? a.w[h * D.dv + cc] : 1.f;
  // ---- what a token brings: this thread's element of [q | k] with its partner and their angle, its column's value and gate
  struct In {
    float u, w, co, si, v, gate, i, f;
  };
  const int which = tid / (32 * NV), e = tid % (32 * NV);
  const bool staged = which < 2, inside = staged && e < D.dk, turned = inside && e < 2 * a.half;
  const int src = (which ? D.k : D.q) + g * D.dk + e, other = e < a.half ? a.half : -a.half;
  auto fetch = [&](int t) {
    const int64_t tok = t0 + t;
    const T* row = (const T*)a.proj + tok * D.rows;
    In x{0.f, 0.f, 1.f, 0.f, (float)row[D.v + h * D.dv + cc], (float)row[a.gate + h * D.dv + cc], 0.f, 0.f};
    if (inside) x.u = (float)row[src];
    if (turned) {
      x.w = (float)row[src + other];
      const float* an = a.cs + (tok * a.half + (e < a.half ? e : e - a.half)) * 2;
      x.co = an[0];
      x.si = e < a.half ? -an[1] : an[1];
    }
    if (NORM && wave == 0) {
      x.i = (float)row[a.ci + h];
      x.f = (float)row[a.cf + h];
    }
    return x;
  };
  In x = fetch(0);
  for (int t = 0; t < n; ++t) {
    const float vv = x.v, gt = x.gate;
    if (staged) qk[which][e] = turned ? fmaf(x.u, x.co, x.w * x.si) : x.u;
    if (NORM && wave == 0) {
      const float i = a.cap * tanhf((x.i + a.bi[h]) / a.cap), z = a.cap * tanhf((x.f + a.bf[h]) / a.cap);
      const float f = fminf(z, 0.f) - log1pf(expf(-fabsf(z))), mt = fmaxf(f + m, i);
      if (lane == 0) {
        gates[0] = expf(f + m - mt);
        gates[1] = expf(i - mt);
        gates[2] = expf(-mt);
      }
      m = mt;
    }
    __syncthreads();
    if (t + 1 < n) x = fetch(t + 1);
    const float da = NORM ? gates[0] : decay, b = NORM ? gates[1] : 1.f, u = b * vv;
    float o = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const f32x4 q = *reinterpret_cast<const f32x4*>(&qk[0][4 * (p + LPC * i)]),
                  k = *reinterpret_cast<const f32x4*>(&qk[1][4 * (p + LPC * i)]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        S[i][j] = fmaf(k[j], u, da * S[i][j]);
        o = fmaf(S[i][j], q[j], o);
      }
    }
#pragma unroll
    for (int d = 1; d < LPC; d <<= 1) o += __shfl_xor(o, d, 64);
    o *= a.scale;
    if constexpr (NORM) {
      float zq = 0.f;
#pragma unroll
      for (int i = 0; i < NZ; ++i) {
        const int k = min(lane + 64 * i, 32 * NV - 1);
        const float z = lane + 64 * i < dks ? 1.f : 0.f;
        Z[i] = fmaf(qk[1][k] * z, b, da * Z[i]);
        zq = fmaf(Z[i], qk[0][k], zq);
      }
      zq = wave_sum(zq);
      o /= fmaxf(fabsf(zq * a.scale), gates[2]) + 1e-6f;
    }
    float ss = on ? o * o : 0.f;
#pragma unroll
    for (int d = LPC; d < 64; d <<= 1) ss += __shfl_xor(ss, d, 64);
    if (lane == 0) red[wave] = ss;
    __syncthreads();  // (also: q, k and the gates have been read)
    ss = 0.f;
    for (int i = 0; i < (int)blockDim.x / 64; ++i) ss += red[i];
    if (on && p == 0) {
      const float rs = 1.f / sqrtf(ss / (float)D.dv + a.eps), act = (a.mode == SIGMOID_AFTER ? 1.f : gt) * sigmoid_f(gt);
      ((T*)a.out)[(t0 + t) * a.ostride + h * D.dv + col] = (T)(o * rs * weight * act);
    }
  }
  if (on) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int k = 4 * (p + LPC * i);
      if (k < dks) *reinterpret_cast<f32x4*>(st + k) = S[i];
    }
  }
  if constexpr (NORM) {
    if (wave < D.zc())
#pragma unroll
      for (int i = 0; i < NZ; ++i)
        if (lane + 64 * i < dks) zt[lane + 64 * i] = Z[i];
    if (tid == 0) a.peak[(int64_t)slot * D.H + h] = m;
  }
}

template <typename T>
int step(const StepArgs& a, int nlist, hipStream_t st) {
  const dim3 grid(nlist, a.D.H);
  const int nt = (LPC * a.D.dv + 63) / 64 * 64, nv = (a.D.dks() + 31) / 32;
#define RUN(NV, NORM) hipLaunchKernelGGL((scan_step_kernel<T, NV, NORM>), grid, dim3(nt), 0, st, a)
#define GO(NV)                    \
  {                               \
    if (a.zstate) RUN(NV, true);  \
    else RUN(NV, false);          \
  }
  if (nv <= 1) GO(1)
  else if (nv <= 2) GO(2)
  else if (nv <= 4) GO(4)
  else GO(8)
#undef GO
#undef RUN
  DS_CHECK_LAUNCH();
  return 0;
}

}  // namespace

// Key rows as padded to 32, 64, 128 or 256 are staged by half as many threads as there are (8 a value column)
extern "C" int ds_scan_step_ok(int dk, int dv) {
  const int nv = (((dk + 7) & ~7) + 31) / 32, pad = 32 * (nv <= 2 ? nv : nv <= 4 ? 4 : 8);
  return dk > 0 && dv > 0 && dv <= MAX_DV && nv <= MAX_NV && 2 * pad <= (LPC * dv + 63) / 64 * 64;
}

// As ds_scan_split, (ds_exp_gates,) ds_scan_recur and ds_gated_norm one after the other for the sequences in `list`. log_decay, or
// (null) gates: ci, cf, bi, bf, cap, peak, zstate.
extern "C" int ds_scan_step(const void* proj, const float* cs, int half, const float* log_decay, int ci, int cf, const float* bi,
                            const float* bf, float cap, float* peak, float scale, float* state, float* zstate, const int* list,
                            int nlist, const int* cu, const int* start, const int* slots, int gate, int mode, const float* w, float eps,
                            void* out, int64_t ostride, const int* dims, int tokens, int dtype, hipStream_t st) {
  if (nlist <= 0 || tokens <= 0) return 0;
  const ScanDims D{dims[0], dims[1], dims[2], dims[3], dims[4], dims[5], dims[6], dims[7], dims[8], dims[9], dims[10], dims[11],
                   tokens};
  if (!scan_dims_ok(D) || !ds_scan_step_ok(D.dk, D.dv) || D.taps > 1 || half < 0 || 2 * half > D.dk || (half && !cs) || gate < 0 ||
      gate + D.H * D.dv > D.rows || ostride < D.H * D.dv || (mode != SIGMOID_AFTER && mode != SILU_AFTER) ||
      (!log_decay && (!bi || !bf || !peak || !zstate || ci < 0 || cf < 0 || ci + D.H > D.rows || cf + D.H > D.rows || !(cap > 0.f))) ||
      (log_decay && zstate))
    return (int)hipErrorInvalidValue;
  const StepArgs a{proj, cs, half, log_decay, ci, cf, bi, bf, cap, peak, scale, state, zstate, list, cu, start, slots, gate, mode, w,
                   eps, out, ostride, D};
  if (dtype == DS_F32) return step<float>(a, nlist, st);
  if (dtype == DS_BF16) return step<bf16>(a, nlist, st);
  return (int)hipErrorInvalidValue;
}
