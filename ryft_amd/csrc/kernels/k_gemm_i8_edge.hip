// MFMA GEMM instantiations: i8, edge tiles.
#include "gemm_mfma.h"

namespace ryft {

int edge_tiles_i8(const GemmArgs& g, bool ar, bool br, Choice* c) {
  if (g.dual) return 0;
  const char* name = "gemm_i8_mfma_edge_128x128";
  c[0] = edge_choice<MMA_I8, 256, 256, 128, 2, 4, false>(ar, br, name);
  c[1] = edge_choice<MMA_I8, 128, 128, 128, 2, 2, false>(ar, br, name);
  if (ar) return 2;
  c[2] = edge_choice_k<MMA_I8, 64, 128, 128, 2, 2, false>(br, name);
  c[3] = edge_choice_k<MMA_I8, 32, 128, 128, 1, 4, false>(br, name);
  return 4;
}

}  // namespace ryft
