// Top-k selection per column of MU on the device (ac_select.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ac {

constexpr int kSelChunks = 2048;  // row chunks, at most
constexpr int kSelMaxK = 512;
constexpr int kSelCap = 4096;     // keys kept per column, at most

struct SelShape {
  int chunks = 0;  // 0: select on the host
  int64_t rows = 0;
};
// Device buffers of one selection: cmax [P][chunks], thr / count [P], keys [P][kSelCap], idx / val [P][k], flag [1]
// (zeroed by the caller; nonzero afterwards: the result is not valid, select on the host).
struct SelBufs {
  unsigned* cmax;
  unsigned* thr;
  int* count;
  unsigned long long* keys;
  int* idx;
  float* val;
  int* flag;
};
SelShape sel_shape(int64_t n, int P, int k);
void launch_select(int64_t n, int P, int k, const SelShape& s, const float* X, const SelBufs& b, hipStream_t st);

}  // namespace ac
