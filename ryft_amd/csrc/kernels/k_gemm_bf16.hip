// MFMA GEMM instantiations: bf16, full tiles.
#include "gemm_mfma.h"

namespace ryft {

bool pick_bf16(const GemmArgs& g, bool ar, bool br, Choice* c) {
  auto fits = [&](int bm, int bn, int bk) { return !ar && g.M % bm == 0 && g.N % bn == 0 && g.K % bk == 0; };
  if (g.dual) return false;
  if (g.splits > 1) {  // split-K runs the 128×128 tile over each K range
    if (!fits(128, 128, 64 * g.splits)) return false;
    *c = br ? make_choice<MMA_BF16, 128, 128, 64, 2, 2, false, true, false>("gemm_bf16_mfma_128x128")
            : make_choice<MMA_BF16, 128, 128, 64, 2, 2, false, false, false>("gemm_bf16_mfma_128x128");
    return true;
  }
  const int64_t tiles256 = (int64_t)(g.M / 256) * (g.N / 256) * g.batch;
  if (fits(256, 256, 64) && tiles256 >= 128 && 2 * tiles256 <= 256) {
    // 256×256 tiles that would leave half of the CUs idle: twice as many of half the size, which run in one round, a CU
    // each (2048 × 4096 × 4096: 128 tiles of 256×256 take 84 µs, 256 of 256×128 59 µs)
    *c = br ? make_choice<MMA_BF16, 256, 128, 64, 4, 2, false, true, false>("gemm_bf16_mfma_256x128")
            : make_choice<MMA_BF16, 256, 128, 64, 4, 2, false, false, false>("gemm_bf16_mfma_256x128");
    return true;
  }
  if (fits(256, 256, 64) && tiles256 >= 128) {
    // eight waves (two per SIMD, 128×64 each): one wave's LDS waits and barrier overlap the other's MFMAs
    *c = br ? make_choice<MMA_BF16, 256, 256, 64, 2, 4, false, true, false>("gemm_bf16_mfma_256x256")
            : make_choice<MMA_BF16, 256, 256, 64, 2, 4, false, false, false>("gemm_bf16_mfma_256x256");
    return true;
  }
  if (fits(128, 128, 64)) {
    *c = br ? make_choice<MMA_BF16, 128, 128, 64, 2, 2, false, true, false>("gemm_bf16_mfma_128x128")
            : make_choice<MMA_BF16, 128, 128, 64, 2, 2, false, false, false>("gemm_bf16_mfma_128x128");
    return true;
  }
  return false;
}

}  // namespace ryft
