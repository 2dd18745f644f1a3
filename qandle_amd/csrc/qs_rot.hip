// One rotation of the per-operator path and its gradient, straight from the
// angle: R_P(phi) on one bit position (optionally under a control mask).
//
// Bound by the state traffic: 16 B per amplitude forward; backward 24 B (the
// output gradient and the output state are read, the input gradient written),
// with the angle's reduction made from the same registers.  Measured at 18
// qubits x 8 (16.8 MB): forward 7.4 us (4.5 TB/s; with its half-angle kernel
// 8.8 before), backward 13.7 + 3.2 us (inverse rotation, Pauli product, their
// finish and two torch kernels 26 us before).  A thread moves two
// 16-byte vectors: two amplitude pairs (an even amplitude and its neighbour,
// and their partners), or for bit 0 the pair itself; states that are only
// 8-byte aligned go pair by pair.  Every thread computes the angle's sincosf
// itself, as a separate kernel for it costs a launch per operator; the values
// are left in `table` for the gradient, which the angle may have left by then.
#include "qs_common.h"

namespace qs {

constexpr int kRotThreads = 256;
constexpr int kRotChunk = 11;  // pairs per block of the backward: 2^11 (its partials then match one sample each)

__device__ __forceinline__ float4 rot_ld4(const float *p, int64_t i) { return reinterpret_cast<const float4 *>(p)[i]; }
__device__ __forceinline__ void rot_st4(float *p, int64_t i, float2 a, float2 b) {
  reinterpret_cast<float4 *>(p)[i] = make_float4(a.x, a.y, b.x, b.y);
}

// First amplitude of item q.  Vector items hold two amplitude pairs (i0, i1),
// (i0 + 1, i1 + 1) for bit > 0, one pair (i0, i0 + 1) for bit 0; scalar items one pair.
template <bool VEC>
__device__ __forceinline__ int64_t rot_item(int64_t q, int bit) {
  if (!VEC) return insert_zero(q, bit);
  return bit == 0 ? 2 * q : 2 * insert_zero(q, bit - 1);
}

template <int KIND, bool VEC>
__device__ __forceinline__ void rot_apply(float *out, const float *in, int64_t i0, int bit, float c, float s, int64_t cmask) {
  const int64_t i1 = i0 | (int64_t(1) << bit);
  if (VEC && bit == 0) {
    const float4 v = rot_ld4(in, i0 >> 1);
    float2 a = make_float2(v.x, v.y), b = make_float2(v.z, v.w);
    if ((i0 & cmask) == cmask) rot_pair<KIND>(c, s, a, b);
    rot_st4(out, i0 >> 1, a, b);
  } else if (VEC) {
    const float4 v = rot_ld4(in, i0 >> 1), w = rot_ld4(in, i1 >> 1);
    float2 a0 = make_float2(v.x, v.y), b0 = make_float2(v.z, v.w), a1 = make_float2(w.x, w.y), b1 = make_float2(w.z, w.w);
    if ((i0 & cmask) == cmask) rot_pair<KIND>(c, s, a0, a1);
    if (((i0 | 1) & cmask) == cmask) rot_pair<KIND>(c, s, b0, b1);
    rot_st4(out, i0 >> 1, a0, b0);
    rot_st4(out, i1 >> 1, a1, b1);
  } else {
    float2 a = ld2(in, i0), b = ld2(in, i1);
    if ((i0 & cmask) == cmask) rot_pair<KIND>(c, s, a, b);
    st2(out, i0, a);
    st2(out, i1, b);
  }
}

__device__ __forceinline__ float2 rot_coef(const float *phi, int64_t i, float sgn) {
  float s, c;
  sincosf(phi[i] * 0.5f, &s, &c);
  return make_float2(c, sgn * s);
}

template <int KIND, bool VEC>
__global__ void __launch_bounds__(kRotThreads)
k_rot_angle(float *out, float *table, const float *in, int64_t items, int n, int bit, const float *phi,
            int64_t phi_stride, int per_sample, int64_t cmask, float sgn) {
  int64_t sample = -1;
  float2 cs = make_float2(0.f, 0.f);
  if (!per_sample) {
    cs = rot_coef(phi, 0, sgn);
    if (table && blockIdx.x == 0 && threadIdx.x == 0) st2(table, 0, make_float2(cs.x, sgn * cs.y));
  }
  for (int64_t q = blockIdx.x * (int64_t)kRotThreads + threadIdx.x; q < items; q += (int64_t)gridDim.x * kRotThreads) {
    const int64_t i0 = rot_item<VEC>(q, bit);
    if (per_sample && (i0 >> n) != sample) {
      sample = i0 >> n;
      cs = rot_coef(phi, sample * phi_stride, sgn);
      if (table && i0 == sample << n) st2(table, sample, make_float2(cs.x, sgn * cs.y));
    }
    rot_apply<KIND, VEC>(out, in, i0, bit, cs.x, cs.y, cmask);
  }
}

__device__ __forceinline__ float rot_block_sum(float v, float *red) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// Block = one chunk of 2^c pairs of one sample: gin = R^-1 g (gin = NULL: not
// wanted), part[chunk] = sum of Im<g|P|psi> over the chunk's pairs under the control.
template <int KIND, bool VEC>
__global__ void __launch_bounds__(kRotThreads)
k_rot_backward(float *gin, float *part, const float *g, const float *psi, int n, int c, int bit, const float *table,
               int per_sample, int64_t cmask) {
  __shared__ float red[4];
  const int64_t chunk = blockIdx.x;
  const int items_log = VEC && bit > 0 ? c - 1 : c;  // vector items of two pairs (c >= 1 when bit > 0)
  float2 cs = ld2(table, per_sample ? chunk >> (n - 1 - c) : 0);
  cs.y = -cs.y;
  const int64_t m = int64_t(1) << bit;
  float acc = 0.f;
  for (int k = threadIdx.x; k < (1 << items_log); k += kRotThreads) {
    const int64_t i0 = rot_item<VEC>((chunk << items_log) + k, bit), i1 = i0 | m;
    float2 g0[2], g1[2], p0[2], p1[2];
    const bool two = VEC && bit > 0;
    if (VEC && bit == 0) {
      const float4 a = rot_ld4(g, i0 >> 1), b = rot_ld4(psi, i0 >> 1);
      g0[0] = make_float2(a.x, a.y); g1[0] = make_float2(a.z, a.w);
      p0[0] = make_float2(b.x, b.y); p1[0] = make_float2(b.z, b.w);
    } else if (VEC) {
      const float4 a = rot_ld4(g, i0 >> 1), b = rot_ld4(g, i1 >> 1), d = rot_ld4(psi, i0 >> 1), e = rot_ld4(psi, i1 >> 1);
      g0[0] = make_float2(a.x, a.y); g0[1] = make_float2(a.z, a.w);
      g1[0] = make_float2(b.x, b.y); g1[1] = make_float2(b.z, b.w);
      p0[0] = make_float2(d.x, d.y); p0[1] = make_float2(d.z, d.w);
      p1[0] = make_float2(e.x, e.y); p1[1] = make_float2(e.z, e.w);
    } else {
      g0[0] = ld2(g, i0); g1[0] = ld2(g, i1);
      p0[0] = ld2(psi, i0); p1[0] = ld2(psi, i1);
    }
#pragma unroll
    for (int u = 0; u < (VEC ? 2 : 1); ++u) {
      if (u == 1 && !two) break;
      if (((i0 + u) & cmask) == cmask) {
        acc += pauli_im_pair<KIND>(g0[u], g1[u], p0[u], p1[u]);
        rot_pair<KIND>(cs.x, cs.y, g0[u], g1[u]);
      }
    }
    if (!gin) continue;
    if (VEC && bit == 0) {
      rot_st4(gin, i0 >> 1, g0[0], g1[0]);
    } else if (VEC) {
      rot_st4(gin, i0 >> 1, g0[0], g0[1]);
      rot_st4(gin, i1 >> 1, g1[0], g1[1]);
    } else {
      st2(gin, i0, g0[0]);
      st2(gin, i1, g1[0]);
    }
  }
  if (!part) return;
  const float s = rot_block_sum(acc, red);
  if (threadIdx.x == 0) part[chunk] = s;
}

// gphi[b] = half the sum of block b's `count` consecutive partials (one block
// per sample, or one block for all of them), in double
__global__ void __launch_bounds__(kRotThreads) k_rot_finish(float *gphi, const float *part, int64_t count) {
  __shared__ double red[4];
  const float *p = part + blockIdx.x * count;
  double s = 0.0;
  for (int64_t k = threadIdx.x; k < count; k += kRotThreads) s += (double)p[k];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) gphi[blockIdx.x] = (float)(0.5 * ((red[0] + red[1]) + (red[2] + red[3])));
}

static bool rot_args_bad(int64_t B, int n, int bit, int kind, int64_t cmask) {
  return B < 1 || n < 1 || n > 40 || bit < 0 || bit >= n || kind < 0 || kind > 2 || cmask < 0 || (cmask >> n) != 0 ||
         ((cmask >> bit) & 1);
}

static bool aligned16(const void *a, const void *b, const void *c) {
  return (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c) & 15) == 0;
}

template <int KIND>
static void launch_rot(bool vec, float *out, float *table, const float *in, int64_t B, int n, int bit, const float *phi,
                       int64_t phi_stride, int per_sample, int64_t cmask, float sgn, hipStream_t st) {
  const int64_t pairs = (B << n) >> 1, items = vec && bit > 0 ? pairs >> 1 : pairs;
  // two items a thread hide the sincosf behind the loads; past 2^20 blocks the loop takes the rest
  int64_t blocks = (items + 2 * kRotThreads - 1) / (2 * kRotThreads);
  blocks = blocks > (1 << 20) ? (1 << 20) : blocks;
  const dim3 grid((unsigned)blocks), block(kRotThreads);
  if (vec)
    hipLaunchKernelGGL((k_rot_angle<KIND, true>), grid, block, 0, st, out, table, in, items, n, bit, phi, phi_stride,
                       per_sample, cmask, sgn);
  else
    hipLaunchKernelGGL((k_rot_angle<KIND, false>), grid, block, 0, st, out, table, in, items, n, bit, phi, phi_stride,
                       per_sample, cmask, sgn);
}

template <int KIND>
static void launch_rot_backward(bool vec, float *gin, float *part, const float *g, const float *psi, int64_t B, int n,
                                int bit, const float *table, int per_sample, int64_t cmask, hipStream_t st) {
  const int c = n - 1 < kRotChunk ? n - 1 : kRotChunk;
  const dim3 grid((unsigned)(B << (n - 1 - c))), block(kRotThreads);
  if (vec)
    hipLaunchKernelGGL((k_rot_backward<KIND, true>), grid, block, 0, st, gin, part, g, psi, n, c, bit, table, per_sample, cmask);
  else
    hipLaunchKernelGGL((k_rot_backward<KIND, false>), grid, block, 0, st, gin, part, g, psi, n, c, bit, table, per_sample, cmask);
}

}  // namespace qs

using namespace qs;

extern "C" {

int qs_rot_angle(float *out, float *table, const float *in, int64_t B, int n, int bit, int kind, const float *phi,
                 int64_t phi_stride, int per_sample, int64_t cmask, int inverse, void *stream) {
  if (rot_args_bad(B, n, bit, kind, cmask) || !out || !in || !phi || phi_stride < 0) return QS_EINVAL;
  const bool vec = aligned16(out, in, nullptr);
  const float sgn = inverse ? -1.f : 1.f;
  hipStream_t st = (hipStream_t)stream;
  if (kind == QS_RX) launch_rot<QS_RX>(vec, out, table, in, B, n, bit, phi, phi_stride, per_sample, cmask, sgn, st);
  if (kind == QS_RY) launch_rot<QS_RY>(vec, out, table, in, B, n, bit, phi, phi_stride, per_sample, cmask, sgn, st);
  if (kind == QS_RZ) launch_rot<QS_RZ>(vec, out, table, in, B, n, bit, phi, phi_stride, per_sample, cmask, sgn, st);
  return launch_status();
}

int64_t qs_rot_backward_work_bytes(int64_t B, int n) {
  if (B < 1 || n < 1 || n > 40) return -1;
  const int c = n - 1 < kRotChunk ? n - 1 : kRotChunk;
  return (B << (n - 1 - c)) * (int64_t)sizeof(float);
}

int qs_rot_backward(float *gin, float *gphi, const float *g, const float *psi, int64_t B, int n, int bit, int kind,
                    const float *table, int per_sample, int64_t cmask, void *work, int64_t work_bytes, void *stream) {
  if (rot_args_bad(B, n, bit, kind, cmask) || !table || !g || !psi || (!gin && !gphi) || (gphi && !work) || gin == psi)
    return QS_EINVAL;
  const int64_t chunks = qs_rot_backward_work_bytes(B, n) / (int64_t)sizeof(float);
  if (gphi && work_bytes < chunks * (int64_t)sizeof(float)) return QS_EWORKSPACE;
  if (chunks > 0x7fffffff) return QS_EUNSUPPORTED;
  const bool vec = aligned16(g, psi, gin);
  float *part = gphi ? (float *)work : nullptr;
  hipStream_t st = (hipStream_t)stream;
  if (kind == QS_RX) launch_rot_backward<QS_RX>(vec, gin, part, g, psi, B, n, bit, table, per_sample, cmask, st);
  if (kind == QS_RY) launch_rot_backward<QS_RY>(vec, gin, part, g, psi, B, n, bit, table, per_sample, cmask, st);
  if (kind == QS_RZ) launch_rot_backward<QS_RZ>(vec, gin, part, g, psi, B, n, bit, table, per_sample, cmask, st);
  const int s = launch_status();
  if (s || !gphi) return s;
  const int64_t count = per_sample ? chunks / B : chunks;
  hipLaunchKernelGGL(k_rot_finish, dim3((unsigned)(chunks / count)), dim3(kRotThreads), 0, st, gphi, part, count);
  return launch_status();
}

}  // extern "C"
