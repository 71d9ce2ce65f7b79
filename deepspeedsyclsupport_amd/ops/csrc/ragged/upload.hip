// Small tables from the host to the device as a kernel's arguments, CDNA4 (gfx950).
//
// A decode step begins with its index tables, a few hundred words. As a copy they take memory that is pinned, a blit kernel of 4.3 to 4.9 us
// and an event to give the memory back; as arguments the launch itself takes them along, and the host's memory is free when the
// call returns. Two sizes: the runtime copies all of a kernel's arguments on every launch.
#include "ds_hip.h"

namespace {

template <int N>
struct Words {
  uint32_t v[N];
};

template <int N>
__global__ void __launch_bounds__(256) upload_kernel(Words<N> words, uint32_t* out, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = words.v[i];
}

template <int N>
void upload(const uint32_t* words, uint32_t* out, int n, hipStream_t st) {
  Words<N> w;
  for (int i = 0; i < n; ++i) w.v[i] = words[i];
  hipLaunchKernelGGL(upload_kernel<N>, dim3((n + 255) / 256), dim3(256), 0, st, w, out, n);
}

constexpr int FEW = 240, MOST = 960;  // (with the pointer and the count below 4 KB, a kernel's arguments' limit)

}  // namespace

extern "C" int ds_upload_most() { return MOST; }

// out[i] = words[i], i < n <= ds_upload_most(); words: on the host
extern "C" int ds_upload(const void* words, void* out, int n, hipStream_t st) {
  if (n <= 0) return 0;
  if (n > MOST) return (int)hipErrorInvalidValue;
  if (n <= FEW) upload<FEW>((const uint32_t*)words, (uint32_t*)out, n, st);
  else upload<MOST>((const uint32_t*)words, (uint32_t*)out, n, st);
  DS_CHECK_LAUNCH();
  return 0;
}
