// GEMMs on few rows for gfx950: C[M,N] = A[M,K] . W[N,K]^T.  bf16: as many rows as one round of tiles on
// the CUs holds (about 1000 at N = 1024, 200 at N = 5248; split-K: any); fp32: any number.
//
// What bounds these: one question is 64 to 512 rows, so with the large tiles of kernels_gemm.hip an
// N = 1024 GEMM is 16 tiles on 256 CUs, and each of those CUs pulls (128 + 64) rows of all of K through
// its own L1 fill path (about 50 B/clk) and waits out a trip to HBM for the weights whenever its three
// stages in flight run dry.  Here the tile is small (32x16 to 64x64; 128x64 for QKV and split-K), so that
// up to one workgroup per CU shares those bytes, and nearly all of a CU's LDS is a ring of K stages filled
// by LDS DMA, so that 70 to 140 KB are in flight on a CU, which is what a trip to HBM at that rate takes.
// In fp32 the MFMAs bind, and the same kernel in rings of half the LDS keeps them busy at any M.
//
// Same results as kernels_gemm.hip, bit for bit.  bf16: v_mfma_f32_16x16x32_bf16 accumulates each
// output exactly as two v_mfma_f32_32x32x16_bf16 do (checked on the hardware, and by the tests against
// the large tiles), at half the latency of the K chain.  fp32: v_mfma_f32_16x16x4_f32 in k_gemm's K
// order.  Split-K: a chunk's sum is kept apart and added to the sum of the earlier chunks in chunk
// order, as the reduction of launch_splitk adds the slices, without the workspace and its launch.
#include <atomic>
#include <type_traits>

#include "gemm_small.h"

namespace laya {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));   // one 16-byte chunk

// c += W block . A block^T over one 16-byte fragment of each: lane l holds, of row l % 16, the chunk of
// K of its quarter l / 16.  The transposed product leaves lane l with four consecutive output columns
// 4 (l / 16) .. + 3 of output row l % 16.
template <typename T>
__device__ __forceinline__ void small_mma(f32x4_t& c, const u32x4_t& a, const u32x4_t& w) {
  if constexpr (sizeof(T) == 2) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, a), c, 0,
                                                0, 0);
  } else {
    const f32x4_t fa = __builtin_bit_cast(f32x4_t, a), fw = __builtin_bit_cast(f32x4_t, w);
#pragma unroll
    for (int u = 0; u < 4; u++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[u], fa[u], c, 0, 0, 0);
  }
}

// One LDS DMA instruction: lane l copies 16 bytes at rsrc + voff + soff to LDS address lds + 16 l (see
// dma16 in kernels_gemm.hip: inline assembly, ordered by the explicit waits below).
__device__ __forceinline__ void small_dma(u32x4_t rsrc, uint32_t lds, uint32_t voff, uint32_t soff) {
  asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "{m0}"(lds), "v"(voff), "s"(rsrc), "s"(soff)
               : "memory");
}
__device__ __forceinline__ uint32_t small_lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
__device__ __forceinline__ u32x4_t small_rsrc(const void* p, uint32_t bytes) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  u32x4_t r;
  r[0] = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  r[1] = (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(v >> 32) & 0xFFFFu));
  r[2] = (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes);
  r[3] = 0x00020000u;
  return r;
}
__device__ __forceinline__ uint32_t small_pk(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){lo, hi}, bf16x2_t));
}
template <typename T>
__device__ __forceinline__ float small_gelu(float v) {
  if constexpr (sizeof(T) == 2) return gelu_erf_as(v);
  else return gelu_erf(v);
}
// four consecutive values of the storage type at p
template <typename T>
__device__ __forceinline__ void small_st4(T* p, float v0, float v1, float v2, float v3) {
  if constexpr (sizeof(T) == 2) {
    uint2 u;
    u.x = small_pk(v0, v1);
    u.y = small_pk(v2, v3);
    *reinterpret_cast<uint2*>(p) = u;
  } else {
    *reinterpret_cast<float4*>(p) = make_float4(v0, v1, v2, v3);
  }
}

// BM x BN output tile of WM x WN waves, each (BM / WM) x (BN / WN) in 16x16 accumulator blocks.  K
// advances in steps of KU stages; a stage is 128 bytes (one whole line) of every tile row, A rows then W
// rows.  The chunk at slot c of row r holds logical chunk c ^ (r & 7) ^ ((r >> 3) & 1), which makes both
// the DMA's lane-linear writes (8 rows per instruction) and the fragment reads (16 rows at one chunk)
// free of bank conflicts.  NB steps are in LDS: step g lives in buffer g % NB, and all NB are requested
// before the loop.  Iteration g waits until step g + 1 has landed and this wave's fragments of step g
// are in registers, passes one barrier (now every wave has step g in registers, and step g + 1 is
// visible), requests step g + NB into step g's buffer, starts reading step g + 1's fragments and
// multiplies step g's while they arrive.  Every step issues the same number of DMA instructions (past
// the end of K from a resource without records), so the wait is a constant.
// SPLIT: sums of `per` stages are kept apart and added in order (GemmArgs::ksplit).
template <typename T, int BM, int BN, int WM, int WN, int KU, int NB, int EPI, bool SPLIT>
__global__ __launch_bounds__(64 * WM * WN) void k_gemm_small(const GemmArgs a, int per) {
  constexpr int NW = WM * WN, NT = 64 * NW;
  constexpr int FM = BM / WM / 16, FN = BN / WN / 16;
  constexpr int NI = (BM + BN) / 8 / NW;                  // DMA instructions per wave and stage
  constexpr int SC = (BM + BN) * 8, SB = SC * 16;         // a stage in chunks and in bytes
  static_assert(KU == 1 || KU == 2, "stages per step");
  static_assert((BM + BN) % (8 * NW) == 0 && BM % (16 * WM) == 0 && BN % (16 * WN) == 0, "tile");
  static_assert((NB - 1) * KU * NI <= 63 && NB >= 3, "vmcnt");
  static_assert(NB * KU * SB <= 160 * 1024, "LDS");
  constexpr int LDC = EPI == EPI_QKV ? (BN > BM ? BN : BM) + 4 : BN + 4;   // row stride of the staged tile (floats)
  static_assert((EPI == EPI_QKV && BM > BN ? BM : BM > BN ? BM : BN) * LDC * 4 <= NB * KU * SB, "staged tile");
  __shared__ u32x4_t L[NB * KU * SC];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g4 = lane >> 4;
  const int wm = wave / WN, wn = wave % WN;
  const int tilesM = (a.M + BM - 1) / BM, tilesN = (a.N + BN - 1) / BN;
  // Workgroups go round-robin over the 8 XCDs; each XCD gets a contiguous run of tiles, row tiles
  // fastest, so that a weight column block is fetched from memory by one XCD only.
  int pid;
  {
    const int n = tilesM * tilesN, q = n >> 3, r = n & 7, x = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3;
    pid = x * q + min(x, r) + j;
  }
  const int m0 = (pid % tilesM) * BM, n0 = (pid / tilesM) * BN;
  const int D = a.H * a.HD;

  // Operands of the epilogue, requested first: they are the oldest loads, so the K loop's counted waits
  // never wait for them alone.  X: item i = tid + NT k is row i / (BN / 4), columns 4 (i % (BN / 4)) ..
  constexpr int XI = BM * BN / 4 / NT;
  f32x4_t xr[EPI == EPI_RESID ? XI : 1];
  if constexpr (EPI == EPI_RESID) {
#pragma unroll
    for (int k = 0; k < XI; k++) {
      const int i = tid + NT * k, row = min(m0 + i / (BN / 4), a.M - 1), col = min(n0 + 4 * (i % (BN / 4)), a.N - 4);
      xr[k] = *reinterpret_cast<const f32x4_t*>(a.X + (size_t)row * a.ldx + col);
    }
  }
  // positions of the rows this thread rotates: item i is head i / (8 BM) of the tile, row i / 8 % BM,
  // dimensions 4 (i % 8) .. + 3 of the first half of the head
  constexpr int RI = EPI == EPI_QKV ? BM * 8 * (BN / 64) / NT : 1;
  int rp[RI];
  const bool rope = EPI == EPI_QKV && a.rope_cos != nullptr && n0 < 2 * D;
  if constexpr (EPI == EPI_QKV) {
#pragma unroll
    for (int k = 0; k < RI; k++) rp[k] = rope ? a.pos[min(m0 + ((tid + NT * k) >> 3) % BM, a.M - 1)] : 0;
  }

  // DMA plan: instruction j of this wave fills rows 8 i .. + 7 of the stage, i = wave NI + j
  u32x4_t rs[NI];
  uint32_t vo[NI];
  const uint32_t lda_b = (uint32_t)a.lda * sizeof(T), ldw_b = (uint32_t)a.ldw * sizeof(T);
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  {
    const u32x4_t rA = small_rsrc(a.A, (uint32_t)a.M * lda_b), rW = small_rsrc(a.W, (uint32_t)a.N * ldw_b);
#pragma unroll
    for (int j = 0; j < NI; j++) {
      const int i = wv * NI + j, rl = lane >> 3;
      const bool isA = i < BM / 8;
      const uint32_t row = (uint32_t)(isA ? m0 + 8 * i : n0 + 8 * i - BM) + (uint32_t)rl;
      rs[j] = isA ? rA : rW;
      vo[j] = row * (isA ? lda_b : ldw_b) + ((uint32_t)((lane & 7) ^ rl ^ (i & 1)) << 4);
    }
  }
  const int nst = a.K * (int)sizeof(T) / 128;             // stages
  const int nsp = (nst + KU - 1) / KU;                    // steps
  const uint32_t l0 = small_lds_addr(L);
  auto fill = [&](int step, int buf) {
#pragma unroll
    for (int u = 0; u < KU; u++) {
      const int stage = step * KU + u;
#pragma unroll
      for (int j = 0; j < NI; j++) {
        u32x4_t r = rs[j];
        r[2] = stage < nst ? r[2] : 0u;
        small_dma(r, l0 + (uint32_t)(buf * KU + u) * SB + (uint32_t)(wv * NI + j) * 1024u, vo[j], (uint32_t)stage * 128u);
      }
    }
  };
#pragma unroll
  for (int s = 0; s < NB; s++) fill(s, s);

  f32x4_t acc[FM][FN], sum[SPLIT ? FM : 1][SPLIT ? FN : 1];
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++) {
      acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
      if constexpr (SPLIT) sum[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    }

  struct Frag { u32x4_t a[KU * 2][FM], w[KU * 2][FN]; };
  Frag F0, F1;
  const int sw = (l16 & 7) ^ (l16 >> 3);
  const int ra = wm * FM * 16 + l16, rw = BM + wn * FN * 16 + l16;
  auto load = [&](Frag& f, int buf) {
    const u32x4_t* B = L + buf * KU * SC;
#pragma unroll
    for (int u = 0; u < KU; u++)
#pragma unroll
      for (int s = 0; s < 2; s++) {
#pragma unroll
        for (int i = 0; i < FM; i++) f.a[2 * u + s][i] = B[u * SC + (ra + 16 * i) * 8 + ((4 * s + g4) ^ sw)];
#pragma unroll
        for (int j = 0; j < FN; j++) f.w[2 * u + s][j] = B[u * SC + (rw + 16 * j) * 8 + ((4 * s + g4) ^ sw)];
      }
  };
  int cnt = 0;
  bool firstc = true;
  auto mul = [&](const Frag& f, int u) {
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) small_mma<T>(acc[i][j], f.a[2 * u + s][i], f.w[2 * u + s][j]);
    if constexpr (SPLIT) {
      if (++cnt == per) {                                  // the chunk is complete
        cnt = 0;
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
          for (int j = 0; j < FN; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
              sum[i][j][e] = firstc ? acc[i][j][e] : __fadd_rn(sum[i][j][e], acc[i][j][e]);
              acc[i][j][e] = 0.f;
            }
        firstc = false;
      }
    }
  };

  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 1) * KU * NI) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  load(F0, 0);
  int buf = 0;
  auto iter = [&](const Frag& cur, Frag& nxt, int g) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NB - 2) * KU * NI) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int nb = buf + 1 == NB ? 0 : buf + 1;
    load(nxt, nb);
    fill(g + NB, buf);
    buf = nb;
#pragma unroll
    for (int u = 0; u < KU; u++) mul(cur, u);
  };
  int g = 0;
  for (; g + 2 < nsp; g += 2) {
    iter(F0, F1, g);
    iter(F1, F0, g + 1);
  }
  // the last step is whole or one stage (separate copies: a choice between the two fragment sets by
  // address would put both into scratch memory)
  auto last = [&](const Frag& f) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    mul(f, 0);
    if constexpr (KU == 2)
      if (nst % KU == 0) mul(f, 1);
  };
  if (g + 1 < nsp) {
    iter(F0, F1, g);
    last(F1);
  } else {
    last(F0);
  }
  if constexpr (SPLIT) {
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
      for (int j = 0; j < FN; j++) {
        if (cnt > 0)
#pragma unroll
          for (int e = 0; e < 4; e++) sum[i][j][e] = firstc ? acc[i][j][e] : __fadd_rn(sum[i][j][e], acc[i][j][e]);
        acc[i][j] = sum[i][j];
      }
  }

  // ---------------- epilogue: the tile goes through LDS as fp32, then out in whole row segments ----
  f32x4_t cs[RI], sn[RI];
  if constexpr (EPI == EPI_QKV) {
    if (rope) {
#pragma unroll
      for (int k = 0; k < RI; k++) {
        const int q = (tid + NT * k) & 7;
        cs[k] = *reinterpret_cast<const f32x4_t*>(a.rope_cos + rp[k] * 32 + 4 * q);
        sn[k] = *reinterpret_cast<const f32x4_t*>(a.rope_sin + rp[k] * 32 + 4 * q);
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // the fills past the end of K
  __syncthreads();
  float* Ct = reinterpret_cast<float*>(L);
  const bool vsec = EPI == EPI_QKV && n0 >= 2 * D;          // V columns: staged (and stored) transposed
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++) {
      const int r = wm * FM * 16 + 16 * i + l16, c = wn * FN * 16 + 16 * j + 4 * g4;
      if (vsec) {
#pragma unroll
        for (int e = 0; e < 4; e++) Ct[(c + e) * LDC + r] = acc[i][j][e];
      } else {
        *reinterpret_cast<f32x4_t*>(Ct + r * LDC + c) = acc[i][j];
      }
    }
  __syncthreads();

  auto bias4 = [&](int col) -> f32x4_t {
    return a.bias ? *reinterpret_cast<const f32x4_t*>(a.bias + col) : (f32x4_t){0.f, 0.f, 0.f, 0.f};
  };
  // Without a bias the bf16 kernels of the large tiles add nothing (but for QKV), the fp32 one adds 0.
  const bool addb = sizeof(T) == 4 || EPI == EPI_QKV || a.bias != nullptr;
  auto ab = [&](float v, float b) { return addb ? __fadd_rn(v, b) : v; };
  if constexpr (EPI == EPI_RESID) {
#pragma unroll
    for (int k = 0; k < XI; k++) {
      const int i = tid + NT * k, r = i / (BN / 4), c = 4 * (i % (BN / 4)), row = m0 + r, col = n0 + c;
      if (row >= a.M || col >= a.N) continue;
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(Ct + r * LDC + c), b = bias4(col);
      f32x4_t o;
#pragma unroll
      for (int e = 0; e < 4; e++)
        o[e] = sizeof(T) == 4 || SPLIT ? __fadd_rn(xr[k][e], ab(v[e], b[e])) : ab(__fadd_rn(v[e], xr[k][e]), b[e]);
      *reinterpret_cast<f32x4_t*>(a.X + (size_t)row * a.ldx + col) = o;
    }
  } else if constexpr (EPI == EPI_STORE) {
#pragma unroll
    for (int k = 0; k < XI; k++) {
      const int i = tid + NT * k, r = i / (BN / 4), c = 4 * (i % (BN / 4)), row = m0 + r, col = n0 + c;
      if (row >= a.M || col >= a.N) continue;
      f32x4_t v = *reinterpret_cast<const f32x4_t*>(Ct + r * LDC + c);
      const f32x4_t b = bias4(col);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        v[e] = ab(v[e], b[e]);
        if (a.act == ACT_RELU) v[e] = fmaxf(v[e], 0.f);
        else if (a.act == ACT_GELU) v[e] = small_gelu<T>(v[e]);
      }
      small_st4(reinterpret_cast<T*>(a.C) + (size_t)row * a.ldc + col, v[0], v[1], v[2], v[3]);
    }
  } else if constexpr (EPI == EPI_GEGLU) {
    // 64-column groups [input 32 | gate 32] -> 32 output columns
    static_assert(EPI != EPI_GEGLU || BN % 64 == 0, "GeGLU pairs");
    constexpr int GI = BM * BN / 8 / NT, GC = BN / 8;       // items of four outputs; per row
#pragma unroll
    for (int k = 0; k < GI; k++) {
      const int i = tid + NT * k, r = i / GC, q = i % GC, c = (q / 8) * 64 + 4 * (q % 8), row = m0 + r, col = n0 + c;
      if (row >= a.M || col >= a.N) continue;
      const f32x4_t p = *reinterpret_cast<const f32x4_t*>(Ct + r * LDC + c);
      const f32x4_t y = *reinterpret_cast<const f32x4_t*>(Ct + r * LDC + c + 32);
      const f32x4_t b = bias4(col), by = bias4(col + 32);
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] = small_gelu<T>(ab(p[e], b[e])) * ab(y[e], by[e]);
      small_st4(reinterpret_cast<T*>(a.C) + (size_t)row * a.ldc + n0 / 2 + (q / 8) * 32 + 4 * (q % 8), o[0], o[1], o[2], o[3]);
    }
  } else {  // EPI_QKV
    static_assert(EPI != EPI_QKV || BN % 64 == 0, "whole heads");
    if (!vsec) {
      T* dst = reinterpret_cast<T*>(n0 < D ? a.Q : a.Kt) + n0 % D;
#pragma unroll
      for (int k = 0; k < RI; k++) {
        const int i = tid + NT * k, r = (i >> 3) % BM, d = i / (8 * BM) * 64 + 4 * (i & 7), row = m0 + r;
        if (row >= a.M) continue;
        const f32x4_t p = *reinterpret_cast<const f32x4_t*>(Ct + r * LDC + d);
        const f32x4_t q = *reinterpret_cast<const f32x4_t*>(Ct + r * LDC + d + 32);
        const f32x4_t b1 = bias4(n0 + d), b2 = bias4(n0 + d + 32);
        float o1[4], o2[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float x1 = ab(p[e], b1[e]), x2 = ab(q[e], b2[e]);
          o1[e] = rope ? fmaf(x1, cs[k][e], -(x2 * sn[k][e])) : x1;
          // (the rounding of each kernel of kernels_gemm.hip: which of the two products is fused)
          o2[e] = !rope ? x2 : sizeof(T) == 2 ? fmaf(x2, cs[k][e], x1 * sn[k][e]) : fmaf(x1, sn[k][e], x2 * cs[k][e]);
        }
        T* o = dst + (size_t)row * a.ldqk + d;
        small_st4(o, o1[0], o1[1], o1[2], o1[3]);
        small_st4(o + 32, o2[0], o2[1], o2[2], o2[3]);
      }
    } else {
      // V^T[column][row], four rows at a time (rows past M inside the last aligned group of 8 hold the
      // bias, as the large tiles leave them)
      constexpr int VI = BM * BN / 4 / NT;
#pragma unroll
      for (int k = 0; k < VI; k++) {
        const int i = tid + NT * k, c = i / (BM / 4), r = 4 * (i % (BM / 4)), row = m0 + r;
        if (sizeof(T) == 2 ? (row & ~7) >= a.M : row >= a.M) continue;
        const f32x4_t v = *reinterpret_cast<const f32x4_t*>(Ct + c * LDC + r);
        const float b = a.bias ? a.bias[n0 + c] : 0.f;
        T* o = reinterpret_cast<T*>(a.Vt) + (size_t)(n0 - 2 * D + c) * a.ldv + row;
        if (sizeof(T) == 4 && row + 4 > a.M) {
          for (int e = 0; e < a.M - row; e++) Elt<T>::st(o + e, ab(v[e], b));
        } else {
          small_st4(o, ab(v[0], b), ab(v[1], b), ab(v[2], b), ab(v[3], b));
        }
      }
    }
  }
}

// ---------------------------------------------------------------- variants and rule
// Tiles, smallest first.  bf16: the step and ring depths use what LDS holds, 96 to 144 KB, one workgroup
// per CU.  fp32 (but for the smallest tile, whose grid is at most one per CU): 72 to 80 KB, two per CU,
// because the loop is bound by the fp32 MFMAs, and a second workgroup's fill the gaps around barriers.
struct SmallTile { int bm, bn; };
static SmallTile small_tile(int v) {
  static const SmallTile t[kSmallVariants] = {{32, 16}, {32, 32}, {32, 64}, {64, 64}, {128, 64}};
  return t[v];
}

template <typename T, int BM, int BN, int WM, int WN, int KU, int NB>
static void launch_small(int epi, const GemmArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)(((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN))), block(64 * WM * WN);
  int per = 0;
  if (a.ksplit > 1) { const int stages = a.K / 64; per = (stages + a.ksplit - 1) / a.ksplit; }
#define LAYA_SMALL(EPI, SPLIT)                                                                          \
  {                                                                                                     \
    LAYA_LAUNCH((k_gemm_small<T, BM, BN, WM, WN, KU, NB, EPI, SPLIT>), grid, block, 0, st, a, per); \
    return;                                                                                             \
  }
  switch (epi) {
    case EPI_STORE:
      if constexpr (sizeof(T) == 2) if (per) LAYA_SMALL(EPI_STORE, true)
      if constexpr (BM < 128) LAYA_SMALL(EPI_STORE, false)
      break;
    case EPI_RESID:
      if constexpr (sizeof(T) == 2) if (per) LAYA_SMALL(EPI_RESID, true)
      if constexpr (BM < 128) LAYA_SMALL(EPI_RESID, false)
      break;
    case EPI_QKV:
      if constexpr (BN % 64 == 0) LAYA_SMALL(EPI_QKV, false)
      break;
    case EPI_GEGLU:
      if constexpr (BN % 64 == 0 && BM < 128) LAYA_SMALL(EPI_GEGLU, false)
      break;
  }
#undef LAYA_SMALL
  fprintf(stderr, "[laya] gemm: epilogue %d is not built for %dx%d tiles\n", epi, BM, BN);
  exit(1);
}

template <typename T>
void launch_gemm_small_variant(int epi, const GemmArgs& a, int v, hipStream_t st) {
  switch (v) {
    case 0: launch_small<T, 32, 16, 2, 1, 2, 8>(epi, a, st); return;
    case 1:
      if constexpr (sizeof(T) == 2) launch_small<T, 32, 32, 2, 2, 2, 8>(epi, a, st);
      else launch_small<T, 32, 32, 2, 2, 1, 10>(epi, a, st);
      return;
    case 2:
      if constexpr (sizeof(T) == 2) launch_small<T, 32, 64, 2, 2, 2, 6>(epi, a, st);
      else launch_small<T, 32, 64, 2, 2, 1, 6>(epi, a, st);
      return;
    case 3:
      if constexpr (sizeof(T) == 2) launch_small<T, 64, 64, 2, 4, 2, 4>(epi, a, st);
      else launch_small<T, 64, 64, 2, 2, 1, 5>(epi, a, st);
      return;
    case 4:
      if constexpr (sizeof(T) == 2) { launch_small<T, 128, 64, 4, 2, 1, 6>(epi, a, st); return; }
      [[fallthrough]];
    default: fprintf(stderr, "[laya] gemm: bad few-row variant %d\n", v); exit(1);
  }
}

// Shapes the kernel itself can take: whole 128-byte K stages, 16-byte aligned rows and output
// segments, operands that 32-bit buffer offsets reach, and for the QKV and GeGLU pairings 64-column
// tiles whose columns lie in one section.
template <typename T>
bool gemm_small_fits(int epi, const GemmArgs& a, int v) {
  const char* why = "";
  if (v < 0 || v >= kSmallVariants || !gemm_shape_ok(epi, a, (int)sizeof(T), &why)) return false;
  if (v == 4 && (sizeof(T) == 4 || (epi != EPI_QKV && a.ksplit <= 1))) return false;   // (the only forms it is built in)
  if (a.ln_mr || a.stats || a.Xh || a.partials_only) return false;
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  const int bn = small_tile(v).bn;
  // outputs leave in groups of four; bf16 ones in whole groups of 8, like those of the large tiles (the generic
  // kernel, which takes the others, evaluates GELU in another form)
  constexpr int eo = sizeof(T) == 2 ? 8 : 4;
  if (a.N % 8 || !al16(a.bias)) return false;
  if ((size_t)a.M * a.lda * sizeof(T) >= (1u << 31) - 65536 || (size_t)a.N * a.ldw * sizeof(T) >= (1u << 31) - 65536) return false;
  switch (epi) {
    case EPI_STORE: if (a.ldc % eo || !al16(a.C)) return false; break;
    case EPI_RESID: if (a.ldx % 4 || !al16(a.X)) return false; break;
    case EPI_QKV:
      if (a.HD != 64 || bn % 64 || a.H * a.HD % bn || a.ldqk % 8 || a.ldv % 8 || !al16(a.Q) || !al16(a.Kt) || !al16(a.Vt) ||
          !al16(a.rope_cos) || !al16(a.rope_sin)) return false;
      break;
    case EPI_GEGLU: if (bn % 64 || a.ldc % eo || !al16(a.C)) return false; break;
    default: return false;
  }
  if (a.ksplit > 1 && (sizeof(T) != 2 || a.ws == nullptr || (epi != EPI_STORE && epi != EPI_RESID) || a.K % 64 || a.K < 128)) return false;
  return true;
}

// compute units of the current device (256 when the query fails), cached per device
static int small_cus() {
  static std::atomic<int> cached[16];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) {
    (void)hipGetLastError();
    return 256;
  }
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n <= 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
      (void)hipGetLastError();
      n = 256;
    }
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// The rule: the smallest tile whose grid is one round of the CUs.  A tile's time is its K steps at the
// CU's fill rate (about 27 B/clk with weights from HBM, 38 from L2), so the smallest tile that does not
// need a second round is the fastest.  us per launch, weights from HBM, this kernel against the best of
// the large tiles:
//   N 1024, K 2624, residual:  M 128 7.1 | 19.4   256 8.3 | 18.8   512 11.3 | 18.2   1024 15.0 | 18.6
//   N 1024, K 1024, residual:  M 128 3.7 | 8.3    256 4.5 | 8.3    512 5.6 | 8.4     1024 6.8 | 8.7
//   QKV, N 3072, K 1024:       M 128 6.7 | 13.6   256 7.5 | 13.4   512 10.0 | 13.4   768 17.2 | 13.6
//   GeGLU, N 5248, K 1024:     M 64 6.9 | 8.6     192 7.4 | 8.9    256 9.8 | 9.5
//   split-K, N 1024, K 4096:   M 128 9.4 | 15.7   512 16.3 | 21.1  1024 21.0 | 37.8  2048 31.4 | 74.8
// fp32 is bound by the fp32 MFMA rate, so there the rule weighs the tiles of the busiest CU, at any M:
//   N 1024, K 2624, residual:  M 128 15.3 | 59.2   512 28.4 | 58.6   1031 64.9 | 104   9664 406 | 678
//   QKV, N 3072, K 1024:       M 128 13.9 | 28.6   512 32.9 | 44.1   1031 67.3 | 81.6  9664 477 | 564
// (9664 x 1024 x 2624: 128 of the 152 TFLOP/s that a large fp32 product reaches on this chip.  Against 128x128
// tiles in whole rounds, residual: 16384 x 1024 x 1024 277 | 297; 20 plain stores in a row, at the power limit,
// 326 | 317.)
// 128x64 tiles only gain where the large tiles have none (QKV needs BM <= BN there) or write partial
// products to memory (split-K; there also in more than one round).
template <typename T>
int gemm_small_pick(int epi, const GemmArgs& a) {
  if (gemm_pinned() >= 0) return -1;
  const int cus = small_cus();
  if constexpr (sizeof(T) == 4) {
    // relative time of the busiest CU: its tiles times their area, by the tile's cost per area at load
    static const double cost[4] = {0.125 * 1.9, 0.25 * 1.25, 0.5 * 1.08, 1.0};
    int best = -1;
    double bt = 0;
    for (int v = 0; v < 4; v++) {
      const SmallTile t = small_tile(v);
      const int64_t tiles = (int64_t)((a.M + t.bm - 1) / t.bm) * ((a.N + t.bn - 1) / t.bn);
      const double c = (double)((tiles + cus - 1) / cus) * cost[v];
      if ((best < 0 || c < bt) && gemm_small_fits<T>(epi, a, v)) { best = v; bt = c; }
    }
    return best;
  }
  for (int v = 0; v < kSmallVariants; v++) {
    const SmallTile t = small_tile(v);
    const int64_t tiles = (int64_t)((a.M + t.bm - 1) / t.bm) * ((a.N + t.bn - 1) / t.bn);
    const bool split = a.ksplit > 1;
    if ((tiles <= cus || (v == 4 && split)) && gemm_small_fits<T>(epi, a, v)) return v;
  }
  return -1;
}

template <typename T>
bool gemm_small_takes(int epi, const GemmArgs& a) { return gemm_small_pick<T>(epi, a) >= 0; }

template <typename T>
bool launch_gemm_small(int epi, const GemmArgs& a, hipStream_t st) {
  const int v = gemm_small_pick<T>(epi, a);
  if (v < 0) return false;
  launch_gemm_small_variant<T>(epi, a, v, st);
  return true;
}

#define LAYA_SMALL_INST(T)                                                       \
  template bool launch_gemm_small<T>(int, const GemmArgs&, hipStream_t);         \
  template bool gemm_small_takes<T>(int, const GemmArgs&);                       \
  template int gemm_small_pick<T>(int, const GemmArgs&);                         \
  template void launch_gemm_small_variant<T>(int, const GemmArgs&, int, hipStream_t); \
  template bool gemm_small_fits<T>(int, const GemmArgs&, int);
LAYA_SMALL_INST(float)
LAYA_SMALL_INST(bf16_t)

}  // namespace laya
