// Everything a program's passes read besides the state, in one launch: the
// half-angle table, the fused unitaries, their gradient generators and
// matrix-core operands, and the product-state factors with the leading
// rotations applied.
//
// Each of these is at most a few thousand independent 2x2 products, so the
// work is nothing beside its launches: as six kernels (half angles, factors,
// leading unitaries, their application, unitaries, operands) it took 18 us of
// device time and six of the eleven launches of an 8-qubit batch-32 forward.
// Here every item recomputes the angles it needs from the inputs (a sincosf or
// three) instead of reading another kernel's table, so one grid covers all of
// them with no order between its threads; the values are the same bit for bit.
#include "qs_compose.h"
#include "qs_program.h"

namespace qs {

// (cos, sin) of entry i's half angle: from the angle inputs, or from the table
// when the caller already holds one (the adjoint).
struct SetupCoef {
  const qs_setup_args &A;
  __device__ __forceinline__ float2 operator()(int64_t i) const {
    if (!A.phi) return reinterpret_cast<const float2 *>(A.cs)[i];
    float v;
    if (i < A.nphi) {
      v = A.phi[i];
    } else {
      const int64_t j = (i - A.nphi) / A.B, b = (i - A.nphi) - j * A.B;
      v = A.named[j][b * A.named_stride[j]];
    }
    float s, c;
    sincosf(v * 0.5f, &s, &c);
    return make_float2(c, s);
  }
};

__device__ __forceinline__ void setup_unitary(const qs_setup_args &A, const int32_t *w, int64_t b, int slot,
                                              const SetupCoef &coef) {
  float u[8];
  store_m2(u, recipe_unitary(w, b, coef));
  float4 *o = reinterpret_cast<float4 *>(A.utab + 8 * (w[0] + b));
  o[0] = make_float4(u[0], u[1], u[2], u[3]);
  o[1] = make_float4(u[4], u[5], u[6], u[7]);
  if (slot >= 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) reinterpret_cast<float4 *>(A.ltab)[4 * slot + r] = lane_row(u, r, A.dagger);
  }
  if (A.qtab) recipe_generators(A.qtab, w, b, coef);
}

// Thread ranges, each rounded up to whole blocks: half-angle entries, unitaries
// shared by the batch, per-sample unitaries, factors.  64-thread blocks: the
// items are few and long (double products, sincosf), so they spread over as
// many compute units as there are blocks.
__global__ void __launch_bounds__(64) k_setup(qs_setup_args A) {
  const SetupCoef coef{A};
  int64_t i = blockIdx.x * (int64_t)64 + threadIdx.x;
  const auto range = [&i](int64_t count) {  // true when i falls in the next range
    const int64_t span = (count + 63) / 64 * 64;
    if (i < span) return true;
    i -= span;
    return false;
  };
  const int64_t ncs = A.phi ? A.nphi + (int64_t)A.nnamed * A.B : 0;
  if (range(ncs)) {
    if (i < ncs) reinterpret_cast<float2 *>(A.cs)[i] = coef(i);
    return;
  }
  if (range(A.nuniform)) {
    if (i < A.nuniform) setup_unitary(A, A.words + A.uniform[2 * i], 0, A.uniform[2 * i + 1], coef);
    return;
  }
  const int64_t nps = (int64_t)A.nsampled * A.B;
  if (range(nps)) {
    if (i < nps) setup_unitary(A, A.words + A.sampled[i / A.B], i % A.B, -1, coef);
    return;
  }
  if (!A.efac || i >= A.B * A.n) return;
  const int64_t b = i / A.n;
  const int pos = (int)(i - b * A.n);
  const int j = A.column[pos];
  float2 f0 = make_float2(1.f, 0.f), f1 = make_float2(0.f, 0.f);
  if (j >= 0) {
    float s, c;
    sincosf(A.x[b * A.x_stride + j * A.x_step] * 0.5f, &s, &c);
    if (A.rot == QS_RX) {
      f0 = make_float2(c, 0.f);
      f1 = make_float2(0.f, -s);
    } else if (A.rot == QS_RY) {
      f0 = make_float2(c, 0.f);
      f1 = make_float2(s, 0.f);
    } else {
      f0 = make_float2(c, -s);
    }
  }
  const int lead = A.lead ? A.lead[pos] : -1;
  if (lead >= 0) {
    float m[8];
    store_m2(m, recipe_unitary(A.lead_words + lead, b, coef));
    const float2 g0 = f0, g1 = f1;
    f0 = make_float2(m[0] * g0.x - m[1] * g0.y + m[2] * g1.x - m[3] * g1.y,
                     m[0] * g0.y + m[1] * g0.x + m[2] * g1.y + m[3] * g1.x);
    f1 = make_float2(m[4] * g0.x - m[5] * g0.y + m[6] * g1.x - m[7] * g1.y,
                     m[4] * g0.y + m[5] * g0.x + m[6] * g1.y + m[7] * g1.x);
  }
  reinterpret_cast<float4 *>(A.efac)[i] = make_float4(f0.x, f0.y, f1.x, f1.y);
}

}  // namespace qs

using namespace qs;

extern "C" {

int64_t qs_setup_args_bytes(void) { return (int64_t)sizeof(qs_setup_args); }

int qs_setup(const qs_setup_args *args, void *stream) {
  if (!args) return QS_EINVAL;
  const qs_setup_args &A = *args;
  if (A.B < 1 || A.n < 1 || A.n > QS_MAX_QUBITS || A.nphi < 0 || A.nnamed < 0 || A.nnamed > QS_SETUP_MAX_NAMED ||
      A.nuniform < 0 || A.nsampled < 0 || A.rot < 0 || A.rot > 2)
    return QS_EINVAL;
  const int64_t ncs = A.phi ? A.nphi + (int64_t)A.nnamed * A.B : 0;
  if ((ncs > 0 && !A.cs) || (!A.phi && (A.nnamed > 0 || A.nphi > 0))) return QS_EINVAL;
  for (int j = 0; j < A.nnamed; ++j)
    if (!A.named[j]) return QS_EINVAL;
  if (A.nuniform + A.nsampled > 0 && (!A.words || !A.utab || !A.cs)) return QS_EINVAL;
  if ((A.nuniform > 0 && (!A.uniform || !A.ltab)) || (A.nsampled > 0 && !A.sampled)) return QS_EINVAL;
  if (A.efac && (!A.column || (A.lead && (!A.lead_words || !A.phi)))) return QS_EINVAL;
  const auto blocks = [](int64_t count) { return (count + 63) / 64; };
  const int64_t g = blocks(ncs) + blocks(A.nuniform) + blocks(A.nsampled * A.B) + (A.efac ? blocks(A.B * A.n) : 0);
  if (g == 0) return QS_OK;
  if (g > 0x7fffffff) return QS_EUNSUPPORTED;
  hipLaunchKernelGGL(k_setup, dim3((unsigned)g), dim3(64), 0, (hipStream_t)stream, A);
  return launch_status();
}

}  // extern "C"
