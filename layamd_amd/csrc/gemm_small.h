// Launch rule and kernel of the few-row GEMMs (kernels_gemm_small.hip).
#pragma once
#include "kernels.h"

namespace laya {

// Runs the GEMM on the few-row kernel when its rule takes the shape (bf16: rows few enough that the
// large tiles of launch_gemm leave most of the chip idle; fp32: any number; aligned operands, no
// LayerNorm fold, no partials left in the workspace) and returns true; otherwise launches nothing and
// returns false.  Every output is the one launch_gemm gives, bit for bit: the K order, the split-K
// chunks (GemmArgs::ksplit) and the epilogue's arithmetic are the same.  A pinned tile configuration
// (gemm_config) keeps launch_gemm.
template <typename T>
bool launch_gemm_small(int epi, const GemmArgs& a, hipStream_t st);

// whether launch_gemm_small would take this GEMM (host only, launches nothing)
template <typename T>
bool gemm_small_takes(int epi, const GemmArgs& a);

// tile variants of the kernel; the rule's pick for a shape (-1: not taken)
constexpr int kSmallVariants = 5;
template <typename T>
int gemm_small_pick(int epi, const GemmArgs& a);
// launches variant v (which must be one that fits: gemm_small_fits)
template <typename T>
void launch_gemm_small_variant(int epi, const GemmArgs& a, int v, hipStream_t st);
template <typename T>
bool gemm_small_fits(int epi, const GemmArgs& a, int v);

}  // namespace laya
