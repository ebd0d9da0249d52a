// Weights fetched ahead of their GEMMs by the launches before them, and the launches that take them along.
#pragma once
#include "kernels.h"

namespace laya {

// Weights that the next GEMMs of a pass read, touched by workgroups that a LayerNorm or attention launch of
// a few rows adds for it (they would leave most CUs idle).  A pass reads more weights than the memory-side
// cache holds, so without this a GEMM of a few rows waits for HBM: 128 x 3072 x 1024 takes 6.8 us with its
// weights in HBM and 5.7 with them in that cache, 128 x 1024 x 2624 6.9 and 5.3.
struct Prefetch {
  const void* p[2] = {nullptr, nullptr};
  uint32_t lines[2] = {0, 0};                      // whole 128-byte lines
  void add(int i, const void* w, size_t bytes) { p[i] = w; lines[i] = (uint32_t)(bytes / 128); }
};
struct NoPrefetch {};
// of 256 threads each, 49152 in all: a line each of the large model's Wqkv, up to two of its Wi (83968)
constexpr int kPrefetchBlocks = 192;
__device__ __forceinline__ void prefetch_lines(const Prefetch& f, uint32_t thread, uint32_t threads) {
#pragma unroll
  for (int a = 0; a < 2; a++) {
    const char* p = static_cast<const char*>(f.p[a]);
    for (uint32_t i = thread; i < f.lines[a]; i += 4 * threads) {
      uint32_t v[4] = {0, 0, 0, 0};
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (i + u * threads < f.lines[a]) v[u] = *reinterpret_cast<const uint32_t*>(p + (size_t)(i + u * threads) * 128);
#pragma unroll
      for (int u = 0; u < 4; u++) asm volatile("" ::"v"(v[u]));   // (the loads are for the caches only)
    }
  }
}

// launch_layernorm and launch_attention with weights to fetch ahead (null: none).  Only k_layernorm (without
// ymr) and the bf16 attention of a few tiles add the workgroups; the other kernels ignore pf.  expect: how
// many of the ntiles tiles are not empty, as far as the caller can say (tiles_expected; 0: all), which
// chooses the kernel (attn_form.h) and nothing else.
template <typename Tin, typename T>
void launch_layernorm(const Tin* x, const int* gather, int rows, int D, float eps, const float* w, const float* b,
                      const float* addtab, const int* qt, const int* seq, float* y32, T* yT, hipStream_t st, float* ymr,
                      const PendingPartials* pend, const Prefetch* pf);
template <typename T>
void launch_attention(const T* Q, const T* K, int ldqk, int kv_rows, const T* Vt, int ldv, T* O, int ldo,
                      const AttnTile* tiles, int ntiles, int qtile, int H, const int* soff, const int* vlen,
                      const int* gq, const int* grow, int window_half, float scale, hipStream_t st, const Prefetch* pf,
                      int expect);

}  // namespace laya
