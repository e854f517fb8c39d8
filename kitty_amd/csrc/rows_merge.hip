// The merge pass of a split walk over independent query rows: chunked-prefill attention for every head
// dimension, decode attention for head dimensions other than 128.
//
// out[row] = sum_s acc_s * 2^(m_s - m) / sum_s l_s * 2^(m_s - m),  m = max_s m_s, over `num_splits` partials that lie
// side by side (ws_ml: (m, l) pairs, ws_acc: D floats).  Bound by reading the partials, each once: D / 4 lanes own a
// row, 16 bytes a lane, with eight partials in flight (6400 rows x 8 shares of 512 bytes, 26 MB, pass
// mostly through the last-level cache that the split pass has just filled).
#include "decode_common.h"

namespace kitty {
namespace {

// KEEP_NAN: a row whose sum is NaN stays NaN (chunked prefill at D = 128); otherwise it becomes 0.
template <int D, bool KEEP_NAN>
__global__ __launch_bounds__(256) void rows_merge_kernel(const float* __restrict__ ws_ml, const float* __restrict__ ws_acc,
                                                         __half* __restrict__ out, int64_t rows, int num_splits) {
  constexpr int kLanes = D / 4, kRowsPerBlock = 256 / kLanes, kBatch = 8;
  const int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + threadIdx.x / kLanes;
  const int d = (threadIdx.x % kLanes) * 4;
  if (row >= rows) return;
  const float2* ml = (const float2*)ws_ml + row * num_splits;
  const float* acc = ws_acc + row * num_splits * D + d;
  float m = -INFINITY, l = 0.f;
  float4 o = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < num_splits; s0 += kBatch) {
    float2 x[kBatch];
    float4 a[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int s = min(s0 + i, num_splits - 1);
      x[i] = ml[s];
      a[i] = *(const float4*)(acc + (int64_t)s * D);
      if (s0 + i >= num_splits) x[i].x = -INFINITY;
    }
    float mn = m;
#pragma unroll
    for (int i = 0; i < kBatch; ++i) mn = fmaxf(mn, x[i].x);
    const float wm = m == -INFINITY ? 0.f : exp2f(m - mn);
    l *= wm;
    o.x *= wm, o.y *= wm, o.z *= wm, o.w *= wm;
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      // an empty share (max = -inf; its accumulator row may never have been written) adds nothing
      if (x[i].x != -INFINITY) {
        const float w = exp2f(x[i].x - mn);
        l += x[i].y * w;
        o.x += a[i].x * w, o.y += a[i].y * w, o.z += a[i].z * w, o.w += a[i].w * w;
      }
    }
    m = mn;
  }
  const bool divide = KEEP_NAN ? l != 0.f : l > 0.f;
  __half2 r[2];
  r[0] = __floats2half2_rn(divide ? o.x / l : 0.f, divide ? o.y / l : 0.f);
  r[1] = __floats2half2_rn(divide ? o.z / l : 0.f, divide ? o.w / l : 0.f);
  *(uint2*)(out + row * D + d) = *(const uint2*)r;
}

template <int D>
void launch(const float* ws_ml, const float* ws_acc, void* out, int64_t rows, int num_splits, bool keep_nan,
            hipStream_t stream) {
  constexpr int kRowsPerBlock = 256 / (D / 4);
  const dim3 grid((unsigned)((rows + kRowsPerBlock - 1) / kRowsPerBlock)), block(256);
  if (keep_nan)
    hipLaunchKernelGGL((rows_merge_kernel<D, true>), grid, block, 0, stream, ws_ml, ws_acc, (__half*)out, rows, num_splits);
  else
    hipLaunchKernelGGL((rows_merge_kernel<D, false>), grid, block, 0, stream, ws_ml, ws_acc, (__half*)out, rows, num_splits);
}

}  // namespace

void launch_rows_merge(int D, const float* ws_ml, const float* ws_acc, void* out, int64_t rows, int num_splits,
                       bool keep_nan, hipStream_t stream) {
  if (D == 64) launch<64>(ws_ml, ws_acc, out, rows, num_splits, keep_nan, stream);
  else if (D == kD) launch<kD>(ws_ml, ws_acc, out, rows, num_splits, keep_nan, stream);
  else launch<256>(ws_ml, ws_acc, out, rows, num_splits, keep_nan, stream);
}

}  // namespace kitty
