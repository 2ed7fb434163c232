// Members of the GEMM tile families that only the launcher names (gemm_tiles.h): the 256 x 256 ring with its K shared, and the 128 x 128
// tile that has a compute unit to itself.
#include "gemm_tiles.h"

using namespace cutile;
using namespace cutile::gemm;

#define GEMM_TILES_FAMILY(N, T)                                       \
  GEMM_STAGES_KERNEL(N##_128x128x64_q2x2_lone, 128, 128, 2, 4, 5, T)  \
  GEMM_RING_KERNEL(N##_256x256x64_q2x4_split, 256, 256, 2, 4, T)
GEMM_TILES_FAMILY(bf16, __bf16)
GEMM_TILES_FAMILY(f16, _Float16)
