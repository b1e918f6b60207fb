// bf16 GEMMs on tiles below 256x256 (gemm_bf16.hip): what their callers pass,
// and the extent of an operand stored transposed (gemm_dq.hip's too).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ntlb {

// Bytes from the first to the last value of kvalid stored rows of pitch ld and
// `rows` values of eb bytes, the last row's end rounded up to a 16-byte load:
// the extent of a buffer resource over a matrix stored transposed.  It ends
// there and not at kvalid * ld, because a column slice of a larger matrix may
// be the end of its allocation.
__host__ __device__ inline int64_t stored_rows_extent(int64_t kvalid, int64_t ld, int64_t rows, int eb) {
  if (kvalid <= 0) return 0;
  const int64_t last = (rows * eb + 15) / 16 * 16, pitch = ld * eb;
  return (kvalid - 1) * pitch + (last < pitch ? last : pitch);
}

// One operand of Y[M,N] = A . B^T over plain bf16 matrices.
//   tr = false (A only): [rows, >= Kc] row-major, the contraction contiguous;
//     columns past the contraction are zero or meet zeros of B
//   tr = true: stored transposed, element (r, k) at p[k * ld + r]; contraction
//     rows at or past kvalid read zero
// 16-byte aligned with whole 16-byte rows, addressed with 32-bit byte offsets
// ((rows + 256) * ld * 2 and (kvalid + 64) * ld * 2 below 2^31).
struct Bf16Operand {
  const void* p;
  int64_t ld;
  int64_t rows;
  int64_t kvalid;
  bool tr;
};

struct Bf16Args {
  Bf16Operand a, b;
  int64_t M, N, Kc;  // Kc a multiple of 64
  void* y;
  int y_dtype;
  int64_t ldy;
  int vec_out;  // y 16-byte aligned with 16-byte row pitch
};

// split-K tail of the 256x256-tile GEMMs over dequantized operands: minimum K
// steps per range
constexpr int DQ_SPLIT_MIN_STEPS = 9;

// The tile of a product: 16*mb x 16*nb with the contraction divided among wk
// waves and ns copy stages (mb = 8: 128x128; mb = 0: the 256x256 tiles, not
// these).  big_split: the 256x256 tiles would have a split-K workspace.
struct Bf16Plan {
  int mb, nb, wk, ns;
  bool fits() const { return mb != 0; }
};
Bf16Plan bf16_small_plan(int64_t M, int64_t N, int64_t Kc, bool big_split);

// launch the product on its plan's tile (a status; B tr, a bf16 y where A is
// not tr)
int bf16_small_launch(const char* fn, const Bf16Plan& p, const Bf16Args& g, hipStream_t st);

}  // namespace ntlb
