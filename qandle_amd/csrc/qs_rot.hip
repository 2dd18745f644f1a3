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
constexpr int kRotChunk = 11;       // log2 of the pairs per partial sum of the backward
constexpr int kRotFinishLog = 14;   // partials that one block adds up; more take two launches
constexpr int kRotFinishPart = 12;  // of 2^12 partials per block

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

// One item: adds its Im<g|P|psi> under the control to acc, stores R^-1 g (gin = NULL: not wanted).
template <int KIND, bool VEC>
__device__ __forceinline__ void rot_back(float *gin, float &acc, const float *g, const float *psi, int64_t i0, int bit,
                                         float2 cs, int64_t cmask) {
  const int64_t i1 = i0 | (int64_t(1) << bit);
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
  if (!gin) return;
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

// From kRotChunk + 1 qubits: block = one chunk of 2^kRotChunk pairs of one sample, its sum
// in part[chunk] (NULL: not wanted).
template <int KIND, bool VEC>
__global__ void __launch_bounds__(kRotThreads)
k_rot_backward(float *gin, float *part, const float *g, const float *psi, int n, int bit, const float *table,
               int per_sample, int64_t cmask) {
  __shared__ float red[4];
  const int64_t chunk = blockIdx.x;
  const int items_log = VEC && bit > 0 ? kRotChunk - 1 : kRotChunk;  // vector items of two pairs
  float2 cs = ld2(table, per_sample ? chunk >> (n - 1 - kRotChunk) : 0);
  cs.y = -cs.y;
  float acc = 0.f;
  for (int k = threadIdx.x; k < (1 << items_log); k += kRotThreads)
    rot_back<KIND, VEC>(gin, acc, g, psi, rot_item<VEC>((chunk << items_log) + k, bit), bit, cs, cmask);
  if (!part) return;
  const float s = rot_block_sum(acc, red);
  if (threadIdx.x == 0) part[chunk] = s;
}

// Narrower registers, whose samples are shorter than a chunk: the sum of a shared angle in
// segments of 2^kRotChunk pairs of the whole batch, that of a sample's own angle (half of it:
// the gradient) in its 2^(n-1) pairs.  2^lanes_log threads per segment: a short one's items
// side by side in a wave, four items a thread from there to a whole block.  With a block and
// a partial per sample, and one block to add them up, an operator's forward + backward call
// took 6812 us at 1 qubit x 2^22 (now 110, which the host takes), 1977 at 4 x 2^20 (157) and
// 208 at 8 x 2^16 (155); with the samples' own angles 5092 -> 108, 1393 -> 152, 181 -> 147.  At
// 12 qubits and more this kernel is the slower one (18 x 8 15.5 -> 15.9 us, 20 x 64 316 -> 331).
template <int KIND, bool VEC>
__global__ void __launch_bounds__(kRotThreads)
k_rot_backward_narrow(float *gin, float *part, const float *g, const float *psi, int64_t pairs, int n, int seg,
                      int lanes_log, int64_t segments, int bit, const float *table, int per_sample, int64_t cmask) {
  __shared__ float red[4];
  const int lanes = 1 << lanes_log, lane = threadIdx.x & (lanes - 1), slots = kRotThreads >> lanes_log;
  const int half = VEC && bit > 0 ? 1 : 0;  // vector items of two pairs
  // every thread of a block takes the same number of rounds (the sums meet at a barrier)
  for (int64_t first = blockIdx.x * (int64_t)slots; first < segments; first += (int64_t)gridDim.x * slots) {
    const int64_t s = first + (threadIdx.x >> lanes_log);
    float acc = 0.f;
    if (s < segments) {
      float2 cs = ld2(table, per_sample ? (s << seg) >> (n - 1) : 0);
      cs.y = -cs.y;
      const int64_t end = (s + 1) << seg < pairs ? (s + 1) << seg : pairs;
      for (int64_t q = ((s << seg) >> half) + lane; q < end >> half; q += lanes)
        rot_back<KIND, VEC>(gin, acc, g, psi, rot_item<VEC>(q, bit), bit, cs, cmask);
    }
    if (!part) continue;
    for (int off = 1; off < lanes && off < 64; off <<= 1) acc += __shfl_xor(acc, off, 64);
    if (lanes_log > 6) {  // a segment of several whole waves
      const int wave = threadIdx.x >> 6, w0 = wave & ~((lanes >> 6) - 1);
      if ((threadIdx.x & 63) == 0) red[wave] = acc;
      __syncthreads();
      acc = lanes == 128 ? red[w0] + red[w0 + 1] : (red[0] + red[1]) + (red[2] + red[3]);
      __syncthreads();
    }
    if (lane == 0 && s < segments) part[s] = per_sample ? 0.5f * acc : acc;
  }
}

// out[b] = scale times the sum of block b's `count` consecutive partials (the last block's may
// end early, at `total`), in double
template <class In, class Out>
__global__ void __launch_bounds__(kRotThreads) k_rot_finish(Out *out, const In *part, int64_t count, int64_t total, double scale) {
  __shared__ double red[4];
  const int64_t first = blockIdx.x * count, end = first + count < total ? first + count : total;
  double s = 0.0;
  for (int64_t k = first + threadIdx.x; k < end; k += kRotThreads) s += (double)part[k];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = (Out)(scale * ((red[0] + red[1]) + (red[2] + red[3])));
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

// Partial sums of one gradient: floats first, then (8-byte aligned) the doubles of the two-launch sum.
struct RotSplit {
  int seg;            // log2 of the pairs per partial
  int64_t partials;   // of the whole batch
  int64_t stage;      // doubles of the first of two launches that add them up (0: one launch does)
  int64_t bytes() const { return (partials + 2) * (int64_t)sizeof(float) + stage * (int64_t)sizeof(double); }
};
static RotSplit rot_split(int64_t B, int n, int per_sample) {
  RotSplit r;
  const int64_t pairs = B << (n - 1);
  r.seg = per_sample && n - 1 < kRotChunk ? n - 1 : kRotChunk;
  r.partials = (pairs + (int64_t(1) << r.seg) - 1) >> r.seg;
  r.stage = per_sample || r.partials <= (1 << kRotFinishLog) ? 0
                                                             : (r.partials + (1 << kRotFinishPart) - 1) >> kRotFinishPart;
  return r;
}

template <int KIND>
static void launch_rot_backward(bool vec, float *gin, float *part, const float *g, const float *psi, int64_t B, int n,
                                const RotSplit &sp, int bit, const float *table, int per_sample, int64_t cmask,
                                hipStream_t st) {
  const dim3 block(kRotThreads);
  if (n - 1 >= kRotChunk) {
    const dim3 grid((unsigned)sp.partials);
    if (vec)
      hipLaunchKernelGGL((k_rot_backward<KIND, true>), grid, block, 0, st, gin, part, g, psi, n, bit, table, per_sample, cmask);
    else
      hipLaunchKernelGGL((k_rot_backward<KIND, false>), grid, block, 0, st, gin, part, g, psi, n, bit, table, per_sample, cmask);
    return;
  }
  const int items = vec && bit > 0 ? sp.seg - 1 : sp.seg;
  const int lanes_log = items <= 6 ? items : items <= 8 ? 6 : items <= 9 ? 7 : 8;
  const int64_t slots = kRotThreads >> lanes_log;
  int64_t blocks = (sp.partials + slots - 1) / slots;
  blocks = blocks > (1 << 20) ? (1 << 20) : blocks;  // a launch has fewer than 2^32 threads: the loop takes the rest
  const dim3 grid((unsigned)blocks);
  if (vec)
    hipLaunchKernelGGL((k_rot_backward_narrow<KIND, true>), grid, block, 0, st, gin, part, g, psi, B << (n - 1), n, sp.seg,
                       lanes_log, sp.partials, bit, table, per_sample, cmask);
  else
    hipLaunchKernelGGL((k_rot_backward_narrow<KIND, false>), grid, block, 0, st, gin, part, g, psi, B << (n - 1), n, sp.seg,
                       lanes_log, sp.partials, bit, table, per_sample, cmask);
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
  const int64_t shared = rot_split(B, n, 0).bytes(), own = n - 1 < kRotChunk ? 0 : rot_split(B, n, 1).bytes();
  return shared > own ? shared : own;
}

int qs_rot_backward(float *gin, float *gphi, const float *g, const float *psi, int64_t B, int n, int bit, int kind,
                    const float *table, int per_sample, int64_t cmask, void *work, int64_t work_bytes, void *stream) {
  if (rot_args_bad(B, n, bit, kind, cmask) || !table || !g || !psi || (!gin && !gphi) || (gphi && !work) || gin == psi)
    return QS_EINVAL;
  if (gphi && work_bytes < qs_rot_backward_work_bytes(B, n)) return QS_EWORKSPACE;
  const RotSplit sp = rot_split(B, n, per_sample ? 1 : 0);
  if (n - 1 >= kRotChunk && sp.partials >= int64_t(1) << 24) return QS_EUNSUPPORTED;  // 2^32 threads or more
  const bool vec = aligned16(g, psi, gin);
  const bool direct = gphi && per_sample && n - 1 < kRotChunk;  // the narrow kernel's sums are the gradients
  float *part = !gphi ? nullptr : direct ? gphi : (float *)work;
  hipStream_t st = (hipStream_t)stream;
  if (kind == QS_RX) launch_rot_backward<QS_RX>(vec, gin, part, g, psi, B, n, sp, bit, table, per_sample, cmask, st);
  if (kind == QS_RY) launch_rot_backward<QS_RY>(vec, gin, part, g, psi, B, n, sp, bit, table, per_sample, cmask, st);
  if (kind == QS_RZ) launch_rot_backward<QS_RZ>(vec, gin, part, g, psi, B, n, sp, bit, table, per_sample, cmask, st);
  const int s = launch_status();
  if (s || !gphi || direct) return s;
  const dim3 block(kRotThreads);
  if (sp.stage > 0) {
    double *mid = (double *)(((uintptr_t)(part + sp.partials) + 7) & ~(uintptr_t)7);
    hipLaunchKernelGGL((k_rot_finish<float, double>), dim3((unsigned)sp.stage), block, 0, st, mid, (const float *)part,
                       int64_t(1) << kRotFinishPart, sp.partials, 1.0);
    hipLaunchKernelGGL((k_rot_finish<double, float>), dim3(1), block, 0, st, gphi, (const double *)mid, sp.stage, sp.stage, 0.5);
  } else {
    hipLaunchKernelGGL((k_rot_finish<float, float>), dim3((unsigned)(per_sample ? B : 1)), block, 0, st, gphi,
                       (const float *)part, per_sample ? sp.partials / B : sp.partials, sp.partials, 0.5);
  }
  return launch_status();
}

}  // extern "C"
