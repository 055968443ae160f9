// MFMA GEMM instantiations: bf16, edge tiles.
#include "gemm_mfma.h"

namespace ryft {

int edge_tiles_bf16(const GemmArgs& g, bool ar, bool br, Choice* c) {
  if (g.dual) return 0;
  const char* name = "gemm_bf16_mfma_edge_128x128";
  c[0] = edge_choice<MMA_BF16, 256, 256, 64, 2, 4, false>(ar, br, name);
  c[1] = edge_choice<MMA_BF16, 128, 128, 64, 2, 2, false>(ar, br, name);
  c[2] = edge_choice<MMA_BF16, 64, 64, 64, 2, 2, false>(ar, br, name);
  if (ar) return 3;
  c[3] = edge_choice_k<MMA_BF16, 32, 128, 64, 1, 4, false>(br, name);
  return 4;
}

}  // namespace ryft
