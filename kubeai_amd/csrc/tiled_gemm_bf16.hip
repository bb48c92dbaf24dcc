// The bf16 products of tiled_gemm.h.
#include <torch/extension.h>

#include "tiled_gemm.h"

namespace tiled {

void launch_bf16(int shape, Epilogue epi, const Args& a, int grid) {
  if (epi == kSums) launch<false, kSums>(shape, a, grid);
  else if (epi == kSilu) launch<false, kSilu>(shape, a, grid);
  else if (epi == kGelu) launch<false, kGelu>(shape, a, grid);
  else if (epi == kSquare) launch<false, kSquare>(shape, a, grid);
  else launch<false, kRows>(shape, a, grid);
}

}  // namespace tiled
