// Instantiation unit of the split partial kernel for head dim 128 and more
// than 16 columns (several query tokens per sequence), two or three groups of
// 16 columns per wave.
#include "split_kernels.h"

namespace mxfa {

int launch_wide_128(const DecodeParams &p, const Grid &g, int dtype, bool fp8, hipStream_t st) {
  return launch_wide_hd<128>(p, g, dtype, fp8, st);
}

}  // namespace mxfa
