// The fp8 products of tiled_gemm.h.
#include <torch/extension.h>

#include "tiled_gemm.h"

namespace tiled {

void launch_fp8(int shape, Epilogue epi, const Args& a, int grid) {
  if (epi == kSums) launch<true, kSums>(shape, a, grid);
  else if (epi == kSilu) launch<true, kSilu>(shape, a, grid);
  else launch<true, kRows>(shape, a, grid);
}

}  // namespace tiled
