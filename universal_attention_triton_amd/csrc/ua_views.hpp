// How the kernels see the caller's tensors (strides in elements).  Shared by host and device code.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ua {

// An input tensor addressed as (z, row, col) with z = ((b*H + h)*R + r)*N + i; element offset
//   b*sb + h*sh + r*sr + i*sn + (row / inner)*so + (row % inner)*si + col*sc
struct RowsView {
  const void* p;
  long sb, sh, sr, sn, so, si, sc;
  int inner, H, R, N;
};
// Rows of a result tensor [b, h, r, L, d] with unit feature stride: row t of head z = (b * H + h) * R + r
struct RowsOut {
  long sb, sh, sr, st;
  int H, R;
};
// The gates static_src / static_dest [b, h, L], or their gradients: element (z, t) with z = b * H + h at
// b*sb + h*sh + t*st of either pointer; float32, or the dtype of the tensors beside them
struct GateView {
  void *src, *dest;
  long sb, sh, st;
  int H, f32;
};

}  // namespace ua
