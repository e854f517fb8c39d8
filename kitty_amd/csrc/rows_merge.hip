// The merge pass of a split walk over independent query rows: chunked-prefill attention for every head
// dimension, decode attention for head dimensions other than 128.
//
// out[row] = sum_s acc_s * 2^(m_s - m) / sum_s l_s * 2^(m_s - m),  m = max_s m_s, over `num_splits` partials that lie
// side by side (ws_ml: (m, l) pairs, ws_acc: D floats).  D / 4 lanes own a row, 16 bytes a lane, with eight partials
// in flight.  Many rows are bound by reading the partials, each once (6400 rows x 7 shares of 512 bytes, 23 MB that the
// split pass has just left in the last-level cache: 5.9 us); few rows by the chain of loads a lane goes
// through, so there the partials of a row are dealt in turn to all lane groups of a workgroup, which meet in LDS
// (decode at D = 64, B = 1, 2000 tokens, 32 heads: 11.3 -> 10.8 us for both passes).
#include "decode_common.h"

namespace kitty {
namespace {

// KEEP_NAN: a row whose sum is NaN stays NaN (chunked prefill at D = 128); otherwise it becomes 0.
// GROUPS: lane groups that share a row (1, or all of the workgroup's).
template <int D, bool KEEP_NAN, int GROUPS>
__global__ __launch_bounds__(256) void rows_merge_kernel(const float* __restrict__ ws_ml, const float* __restrict__ ws_acc,
                                                         __half* __restrict__ out, int64_t rows, int num_splits) {
  constexpr int kLanes = D / 4, kRowsPerBlock = 256 / kLanes / GROUPS, kBatch = GROUPS == 1 ? 8 : 4;
  const int grp = GROUPS == 1 ? 0 : threadIdx.x / kLanes;
  const int64_t row = GROUPS == 1 ? (int64_t)blockIdx.x * kRowsPerBlock + threadIdx.x / kLanes : blockIdx.x;
  const int d = (threadIdx.x % kLanes) * 4;
  if (GROUPS == 1 && row >= rows) return;
  const float2* ml = (const float2*)ws_ml + row * num_splits;
  const float* acc = ws_acc + row * num_splits * D + d;
  float m = -INFINITY, l = 0.f;
  float4 o = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = grp; s0 < num_splits; s0 += kBatch * GROUPS) {
    float2 x[kBatch];
    float4 a[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int s = min(s0 + i * GROUPS, num_splits - 1);
      x[i] = ml[s];
      a[i] = *(const float4*)(acc + (int64_t)s * D);
      if (s0 + i * GROUPS >= num_splits) x[i].x = -INFINITY;
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
  if (GROUPS > 1) {
    __shared__ float2 s_ml[GROUPS];
    __shared__ float4 s_o[GROUPS][kLanes];
    if (d == 0) s_ml[grp] = float2{m, l};
    s_o[grp][d / 4] = o;
    __syncthreads();
    if (grp != 0) return;
    float mn = -INFINITY;
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) mn = fmaxf(mn, s_ml[g].x);
    l = 0.f, o = float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
      if (s_ml[g].x != -INFINITY) {
        const float w = exp2f(s_ml[g].x - mn);
        const float4 a = s_o[g][d / 4];
        l += s_ml[g].y * w;
        o.x += a.x * w, o.y += a.y * w, o.z += a.z * w, o.w += a.w * w;
      }
    }
  }
  const bool divide = KEEP_NAN ? l != 0.f : l > 0.f;
  __half2 r[2];
  r[0] = __floats2half2_rn(divide ? o.x / l : 0.f, divide ? o.y / l : 0.f);
  r[1] = __floats2half2_rn(divide ? o.z / l : 0.f, divide ? o.w / l : 0.f);
  *(uint2*)(out + row * D + d) = *(const uint2*)r;
}

template <int D, bool KEEP_NAN>
void launch(const float* ws_ml, const float* ws_acc, void* out, int64_t rows, int num_splits, hipStream_t stream) {
  constexpr int kGroups = 256 / (D / 4);
  if (rows <= 2048 && num_splits > 4)   // up to one workgroup per row and eight per compute unit
    hipLaunchKernelGGL((rows_merge_kernel<D, KEEP_NAN, kGroups>), dim3((unsigned)rows), dim3(256), 0, stream, ws_ml, ws_acc,
                       (__half*)out, rows, num_splits);
  else
    hipLaunchKernelGGL((rows_merge_kernel<D, KEEP_NAN, 1>), dim3((unsigned)((rows + kGroups - 1) / kGroups)), dim3(256), 0,
                       stream, ws_ml, ws_acc, (__half*)out, rows, num_splits);
}

}  // namespace

void launch_rows_merge(int D, const float* ws_ml, const float* ws_acc, void* out, int64_t rows, int num_splits,
                       bool keep_nan, hipStream_t stream) {
#define KITTY_MERGE(DD)                                                                    \
  do {                                                                                     \
    if (keep_nan) launch<DD, true>(ws_ml, ws_acc, out, rows, num_splits, stream);          \
    else launch<DD, false>(ws_ml, ws_acc, out, rows, num_splits, stream);                  \
  } while (0)
  if (D == 64) KITTY_MERGE(64);
  else if (D == kD) KITTY_MERGE(kD);
  else KITTY_MERGE(256);
#undef KITTY_MERGE
}

}  // namespace kitty
