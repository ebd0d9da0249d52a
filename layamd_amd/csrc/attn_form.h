// Which attention kernel a launch runs (host only, no HIP dependency).  The kernels are described in
// kernels_attn.hip; all forms of one type give the same bits.
#pragma once
#include <cstdint>

namespace laya {

// bf16: k_attention_bf16 (kAttnWide), k_attention_narrow on whole tiles, and on 128-query tiles as two
// workgroups each.  fp32: k_attention_f32 on whole tiles (kAttnWide) or with the keys of a block on two waves.
enum AttnForm { kAttnWide = 0, kAttnNarrow = 1, kAttnHalves = 2, kAttnSplit = 3 };

// Workgroups (non-empty tiles times heads) up to which the narrow kernel runs, on 64- and on 128-query tiles,
// and below which it takes a 128-query tile (without a window: a window's first block belongs to the tile) as
// two.  us, k_attention_bf16 | narrow: 64-query sliding tiles, 16 heads: 2 tiles 4.6 | 4.0, 46 (736
// workgroups, the three a CU that its LDS holds) 8.0 | 7.4, 72 10.4 | 11.5.  128-query global tiles,
// | narrow | as two: 1 tile 5.0 | 4.6 | 3.8, 8 (1024 tokens) 16.5 | 14.9 | 11.9, 16 (256 workgroups) 17.6 | 15.6 | 16.1,
// 25 12.7 | 12.4 | 13.2, 95 32.3 | 32.1 | 37.3, 160 55.8 | 59.7 | 67.2.  Between one and two workgroups a CU the
// two are level: 288 (three questions of 650) 16.1 | 16.5, 384 (four of 970, 12 heads) 23.1 | 23.5; there the
// narrow kernel's launches can fetch weights ahead (Prefetch).
constexpr int64_t kAttnNarrow64 = 768, kAttnNarrow128 = 512, kAttnNarrowHalves = 256;

// fp32: workgroups of whole tiles up to which the split form runs: about one per CU.  Split against whole
// tiles, us, 16 heads: 2 tiles 6.8 | 9.8, 7 tiles 13.5 | 20.7, 13 tiles 14.1 | 17.2, 16 tiles (one question of
// 1024) 53.1 | 60.8, 46 tiles 64.1 | 52.2, 173 tiles 221 | 166.
constexpr int64_t kAttnF32Split = 256;

// tiles: the launch's non-empty ones (tiles_expected for a pass, whose lists are padded to its bucket's
// capacity: an empty tile's workgroup ends at once and leaves its CU to others)
inline AttnForm attention_form(bool bf16, int64_t tiles, int H, int qtile, int window_half) {
  const int64_t wgs = tiles * H;
  if (!bf16) return wgs <= kAttnF32Split ? kAttnSplit : kAttnWide;
  if (wgs > (qtile == 128 ? kAttnNarrow128 : kAttnNarrow64)) return kAttnWide;
  return qtile == 128 && wgs < kAttnNarrowHalves && window_half == 0 ? kAttnHalves : kAttnNarrow;
}

}  // namespace laya
