// Lowering of a score_mod that is affine in the score, for gfx950: from the callable's values at six scores to the
// kernels' tables.
//
// Stands for the element-wise evaluation of flaxattention/core/attention.py:59-63; what is checked is that the tables
// reproduce the callable on every position of the problem.
#include "flex_common.cuh"

namespace flex {

// the scores the callable was evaluated at, in order: the additive table, the slope's two points, three checks
__device__ constexpr float kScoresChecked[3] = {0.625f, -1.75f, 3.25f};

// Bound by the read of the six planes, each once (a learned bias [1,12,384,384], 42 MB: 12.3 us); as torch
// operations the same checks were some thirty launches and seven waits of the host.
__global__ __launch_bounds__(256) void affine_tables_kernel(const float* __restrict__ y, int64_t n, int rows, int cols,
                                                            float* __restrict__ add, float* __restrict__ mul,
                                                            float* __restrict__ diag, int32_t* flags) {
  bool bad = false, adds = false, scales = false, bends = false;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const float a = y[i], m = (y[n + i] - y[2 * n + i]) / 16.f;
    bad |= !isfinite(a) || !isfinite(m);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const float want = __fadd_rn(__fmul_rn(m, kScoresChecked[c]), a);
      bad |= !(fabsf(y[(3 + c) * n + i] - want) <= 1e-5f + 1e-5f * fabsf(want));
    }
    adds |= a != 0.f;
    scales |= fabsf(m - 1.f) > 1e-6f;
    add[i] = a;
    mul[i] = m;
    if (diag) {
      const int kv = (int)(i % cols);
      const int64_t row = i / cols;
      const int q = (int)(row % rows);
      if (q > 0 && kv > 0) bends |= a != y[i - cols - 1];
      else diag[row / rows * (rows + cols - 1) + kv - q + rows - 1] = a;
    }
  }
  // (every thread that has something to say stores the same 1)
  if (bad) flags[0] = 1;
  if (adds) flags[1] = 1;
  if (scales) flags[2] = 1;
  if (bends) flags[3] = 1;
}

}  // namespace flex

using namespace flex;
void flex_set_error(const char* fmt, ...);

extern "C" int flexattn_affine_tables(const float* values, int64_t maps, int32_t rows, int32_t cols, float* add, float* mul,
                                      float* diag, int32_t* flags, flexattn_stream_t stream_) {
  if (!values || !add || !mul || !flags) { flex_set_error("affine_tables: null argument"); return 1; }
  if (maps <= 0 || rows <= 0 || cols <= 0) {
    flex_set_error("affine_tables: bad extents maps=%lld rows=%d cols=%d", (long long)maps, rows, cols);
    return 1;
  }
  const int64_t n = maps * rows * cols, want = (n + 255) / 256;
  hipLaunchKernelGGL(affine_tables_kernel, dim3((unsigned)(want < 4096 ? want : 4096)), dim3(256), 0, (hipStream_t)stream_, values, n,
                     rows, cols, add, mul, diag, flags);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { flex_set_error("affine_tables: launch failed: %s", hipGetErrorString(e)); return 2; }
  return 0;
}
