// Skinny matrix-core products (k3_skinny.hip): a resident weight matrix
// against a few activation rows, y[p, r] = sum_c W[r, c] x[p, c].
#pragma once

#include <hip/hip_runtime_api.h>
#include <stdint.h>

namespace k3 {

enum { SKINNY_BF16 = 0, SKINNY_INT8 = 1, SKINNY_FP4 = 2 };

struct SkinnyOp {
  int kind;                    // SKINNY_*
  const void* w;               // [rows, cols], row-major
  const uint8_t* scales;       // SKINNY_FP4: E8M0 [rows, cols / 32]
  const float* row_scales;     // SKINNY_INT8: [rows]
  const float* row_scales2;
  const void* w2;              // a second matrix (GLU): y = act(w . x, w2 . x)
  const uint8_t* scales2;
  int act;                     // GLU: K3_ACT_*
  const void* x;               // [positions, cols]
  int x_dtype;                 // K3_DTYPE_*; BF16 only for SKINNY_FP4 without w2
  void* y;                     // [positions, rows]
  float* y_up;                 // GLU: w2 . x when non-null
  const float* add;            // y += add [positions, rows] (fp32, no GLU; may be y)
  int out_bf16;
  int rows, cols, positions;
};

// Whether launch_skinny takes the shape and alignment.
bool skinny_fits(const SkinnyOp& op);
// Returns a K3_HIP_* status.
int launch_skinny(const SkinnyOp& op, int kernel_class, hipStream_t st);

}  // namespace k3
