// Launcher of the matrix-core decode kernel (paged_decode_mfma.hip).
#pragma once

#include "decode_common.h"

namespace fp_decode {

// How a launch is cut: grid (heads, B, splits), with one split storing its results itself, grid (heads, chunks) or grid
// (heads, pieces + B).
struct Cut {
  bool direct;
  bool flat;
  bool pieces;
};

// The split-K pass of a bf16 or f16 launch with up to 8 query heads per cache head.
int launch_mfma(const DecodeArgs& a, int dtype, int D, const Cut& cut, dim3 grid, hipStream_t st);

}  // namespace fp_decode
