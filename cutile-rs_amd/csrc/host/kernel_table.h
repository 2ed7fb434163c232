// The precompiled-kernel table: what stands where the reference has its JIT and
// kernel cache (cutile/src/tile_kernel.rs:96-114,371-399,675-756).  A key that the
// reference would compile on first launch is here resolved to a gfx950 code
// object embedded in the library plus the launch metadata the HIP kernel needs
// (workgroup shape, LDS bytes, the tile shape it implements).
#pragma once
#include <string>
#include <string_view>
#include <vector>

#include "names.h"
#include "runtime_state.h"

namespace cutile {

enum Image : int { IMG_ELEMENTWISE = 0, IMG_ROWWISE, IMG_GEMM, IMG_FMHA, IMG_MXGEMM, IMG_NVFP4, IMG_RNG, IMG_GEMM_SMALL, IMG_SCALED_FLAT, IMG_GEMM_TILES, IMG_GEMM_F32, IMG_MX_TILES, IMG_GEMM_GROUP, IMG_FMHA_KEYS, IMG_COUNT };

struct KernelEntry {
  const char* function;  // entry name in the reference, e.g. "gemm"
  const char* variant;   // name of this implementation inside the family
  const char* symbol;    // symbol in the code object
  Image image;
  uint32_t block[3];
  uint32_t lds_bytes;
  int32_t tile[4];       // (BM, BN, BK, extra); 0 = not tile-specific; gemm_small.hip, gemm_f32.hip: (0, columns, K tile or 0, rows)
  const char* dtype;     // element type the variant is written for, or ""
  int64_t capacity;      // row-wise kernels: longest segment held in registers; 0 = n/a
  int32_t rank;          // elementwise kernels: tensor rank; 0 = n/a
};

const std::vector<KernelEntry>& kernel_table();

// The entries of one function, in table order; empty if there are none.
const std::vector<const KernelEntry*>& kernels_of(const char* function);
// Finds the entry (function, variant); nullptr if absent.
const KernelEntry* find_entry(std::string_view function, std::string_view variant);
// The member of `family` with that suffix ("+..."), nullptr if it has none: variants that only a launcher names.
const KernelEntry* member_of(const KernelEntry* family, const char* suffix);
// Resolves the entry's hipFunction_t on `device`, loading its code object on
// first use (single flight per device).
cutile_status_t load_entry(cutile_device_t device, const KernelEntry* entry, hipFunction_t* fn);
// Preferred variant set through cutile_kernel_set_preferred_variant, or "".
std::string preferred_variant(const char* function);
// Winner of (function, shape-class bucket), or "", and whether a tuning record names it (otherwise the program did, at run time).
Name class_winner(std::string_view function, std::string_view bucket, bool* from_record);
// The winner of (function, shape-class bucket) that the program set at run time, or (at_run_time false) that a tuning record names; or "".
Name preferred_variant_for(std::string_view function, std::string_view bucket, bool at_run_time);
cutile_status_t set_class_winner(const char* function, const char* bucket, const char* variant, bool from_record);
void clear_bucket_preferences();
// Loads the tuning records once per process (tuning.cpp); cheap afterwards.
void ensure_tuning_records_loaded();
// Human-readable list of variants of `function`, for error messages.
std::string list_variants(const char* function);

}  // namespace cutile
