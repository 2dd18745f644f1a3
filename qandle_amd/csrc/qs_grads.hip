// Gradients of a call from the adjoint sweep's partials, in one launch.
//
// The sweep leaves gpart[row][slot], row = one rotation (or embedded bit), with
// sps consecutive slots per sample.  A gradient is half the sum of its rows'
// partials: over all samples (a shared angle, the rows of every gate that uses
// it) or per sample (an input angle, an embedded feature).  Bound by reading
// the partials once (63 MB at 16 qubits x 256 samples x 960 rotations);
// elsewhere by the launch, which is why the sums over rows, the sums over
// samples and the routing to the outputs are one kernel: as a finish kernel
// with two index kernels for the angles and two per named input they took 140
// of the 330 us of device time, and 28 launches, of an 11-qubit re-uploading
// step.  Sums run in double, in a fixed order.
#include "qs_common.h"

namespace qs {

struct GradArgs {
  float *out;
  const float *gpart;
  const int32_t *first;   // group g's rows are rows[first[g]] .. rows[first[g + 1] - 1]
  const int32_t *rows;
  const int64_t *place;   // out[place[2g] + b * place[2g + 1]]; stride 0: the sum over samples
  int64_t B, NS, sps;
};

__device__ __forceinline__ double lanes_sum(double v, int width) {
  for (int off = 1; off < width; off <<= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Block (group, y).  A shared angle's group is summed by its block y = 0; a
// per-sample group's samples are spread over the blocks y, min(sps, 64) lanes
// per sample (sps is a power of two).
__global__ void __launch_bounds__(256) k_gradients(GradArgs A) {
  __shared__ double red[4];
  const int g = blockIdx.x, tid = threadIdx.x;
  const int r0 = A.first[g], r1 = A.first[g + 1];
  const int64_t at = A.place[2 * g], stride = A.place[2 * g + 1];
  if (stride == 0) {
    if (blockIdx.y) return;
    const int64_t total = A.B * A.sps;
    double acc[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int r = r0; r < r1; ++r) {
      const float *p = A.gpart + A.rows[r] * A.NS;
      for (int64_t i = tid; i < total; i += 8 * 256) {
#pragma unroll
        for (int u = 0; u < 8; ++u) acc[u] += i + u * 256 < total ? (double)p[i + u * 256] : 0.0;
      }
    }
    double s = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
    s = lanes_sum(s, 64);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) A.out[at] = (float)(0.5 * ((red[0] + red[1]) + (red[2] + red[3])));
    return;
  }
  const int width = A.sps < 64 ? (int)A.sps : 64, per = 256 / width;
  const int lane = tid & (width - 1);
  // every lane of a wave takes the same number of rounds, so the shuffles see all of them
  for (int64_t b0 = (int64_t)blockIdx.y * per; b0 < A.B; b0 += (int64_t)gridDim.y * per) {
    const int64_t b = b0 + tid / width;
    double s = 0.0;
    if (b < A.B) {
      for (int r = r0; r < r1; ++r) {
        const float *p = A.gpart + A.rows[r] * A.NS + b * A.sps;
        for (int64_t i = lane; i < A.sps; i += width) s += (double)p[i];
      }
    }
    s = lanes_sum(s, width);
    if (lane == 0 && b < A.B) A.out[at + b * stride] = (float)(0.5 * s);
  }
}

}  // namespace qs

using namespace qs;

extern "C" {

int qs_gradients(float *out, const float *gpart, const int32_t *first, const int32_t *rows, const int64_t *place,
                 int ngroups, int64_t B, int64_t NS, int64_t sps, void *stream) {
  if (ngroups < 0 || B < 1 || sps < 1 || (sps & (sps - 1)) || NS < B * sps) return QS_EINVAL;
  if (ngroups == 0) return QS_OK;
  if (!out || !gpart || !first || !rows || !place) return QS_EINVAL;
  const int per = 256 / (sps < 64 ? (int)sps : 64);
  int64_t y = (B + per - 1) / per;
  if (y > 64) y = 64;
  const GradArgs A{out, gpart, first, rows, place, B, NS, sps};
  hipLaunchKernelGGL(k_gradients, dim3((unsigned)ngroups, (unsigned)y), dim3(256), 0, (hipStream_t)stream, A);
  return launch_status();
}

}  // extern "C"
