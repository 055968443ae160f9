// MFMA GEMM instantiations: bf16 activations × f8E4M3FN weights, edge tiles of dual GEMMs.
#include "gemm_mfma.h"

namespace ryft {

int edge_tiles_bf16f8_dual(const GemmArgs& g, bool ar, bool br, Choice* c) {
  const char* name = "gemm_bf16f8_mfma_dual_edge_128x128";
  c[0] = edge_choice<MMA_BF16_F8, 128, 128, 64, 2, 2, true>(ar, br, name);
  if (ar || !br) return 1;  // (a K-contiguous f8 B is widened on its way into LDS: register-staged 128×128 tiles only)
  c[1] = make_choice<MMA_BF16_F8, 64, 128, 64, 2, 2, false, true, true, true>(name);
  c[2] = make_choice<MMA_BF16_F8, 32, 128, 64, 1, 4, false, true, true, true>(name);
  return 3;
}

}  // namespace ryft
