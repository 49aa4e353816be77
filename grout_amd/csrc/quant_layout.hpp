// Byte layout of a repacked low-bit matrix (grout_qweight_repack), shared by
// the kernels that read it; see quant_gemv.hip for what each array holds.
#pragma once

#include <stddef.h>

namespace grout {

__host__ __device__ inline size_t qalign(size_t b) { return (b + 255) / 256 * 256; }

// Byte offsets of the repacked arrays of an [n][k] matrix and its total size.
struct QLayout {
  size_t off[4];
  size_t total;
};
__host__ __device__ inline QLayout qlayout(int fmt, size_t n, size_t k) {
  QLayout L{};
  size_t sz[4] = {0, 0, 0, 0};
  if (fmt == 8) {
    sz[0] = n * k;
    sz[1] = n * (k / 32) * 2;
  } else if (fmt == 12 || fmt == 13) {
    sz[0] = n * k / 2;
    sz[1] = n * (k / 256) * 16;
    if (fmt == 13) sz[2] = n * k / 8;
  } else if (fmt == 14) {
    sz[0] = n * k / 2;
    sz[1] = n * k / 4;
    sz[2] = n * k / 16;
    sz[3] = n * (k / 256) * 2;
  }
  size_t o = 0;
  for (int i = 0; i < 4; ++i) {
    L.off[i] = o;
    o += qalign(sz[i]);
  }
  L.total = o;
  return L;
}

}  // namespace grout
