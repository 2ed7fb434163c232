// Members of GEMM families that only the launcher names: the 256 x 256 ring with its K shared, the 128 x 128 tile that has a compute unit
// to itself (gemm_tiles.h), and strips that read y past the caches (gemm_thin.h), tiles of 320 to 448 columns (gemm_wide.h); and the register-staged 256 x 256 tiles (gemm_loose.h).
#include "gemm_loose.h"
#include "gemm_thin.h"
#include "gemm_tiles.h"
#include "gemm_wide.h"

using namespace cutile;
using namespace cutile::gemm;

#define GEMM_TILES_FAMILY(N, T)                                       \
  GEMM_STAGES_KERNEL(N##_128x128x64_q2x2_lone, 128, 128, 2, 4, 5, T)  \
  GEMM_RING_TILE_KERNEL(N##_256x256x64_q2x4_split, 256, 256, 2, 4, T) \
  GEMM_RING_MIX_KERNEL(N##_192x256x64_q2x4_mix, 192, T)               \
  GEMM_WIDE_KERNEL(N##_w192x320_192x256x64_q2x4_mix, 192, 320, T)     \
  GEMM_WIDE_KERNEL(N##_w192x384_192x256x64_q2x4_mix, 192, 384, T)     \
  GEMM_WIDE_KERNEL(N##_w192x448_192x256x64_q2x4_mix, 192, 448, T)     \
  GEMM_WIDE_KERNEL(N##_w256x320_192x256x64_q2x4_mix, 256, 320, T)
GEMM_TILES_FAMILY(bf16, __bf16)
GEMM_TILES_FAMILY(f16, _Float16)

#define GEMM_THIN_NT_FAMILY(T, IN_T, OUT_T)                    \
  GEMM_THIN_KERNEL(T##_thin16x64_nt, IN_T, OUT_T, 1, 4, true)  \
  GEMM_THIN_KERNEL(T##_thin16x128_nt, IN_T, OUT_T, 1, 8, true)
GEMM_THIN_NT_FAMILY(bf16, __bf16, __bf16)
GEMM_THIN_NT_FAMILY(f16, _Float16, _Float16)
GEMM_THIN_NT_FAMILY(bf16f32, __bf16, float)

GEMM_STAGED_WIDE_KERNEL(bf16_staged256x256, __bf16, __bf16)
GEMM_STAGED_WIDE_KERNEL(f16_staged256x256, _Float16, _Float16)
GEMM_STAGED_WIDE_KERNEL(bf16f32_staged256x256, __bf16, float)
