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
// them with no order between its threads; the tables are the same bit for bit, the
// factors to a few ulp (the compiler contracts their products differently).
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

// U = a D R G (_engine/givens.py): D = diag(1, w), G = diag(1, g), R = [[1, -t],
// [t, 1]] with a = |u00| p or, where the rotation is past 45 degrees (swap),
// R = [[t, -1], [1, t]] with a = |u10| p; p, q are the phases of u00, u10,
// g = conj(p q), w = q conj(p).  Where u00 or u10 is zero its phase cancels out
// of every product (taken as 1).
struct Split {
  C2 g, w, a;
  double t;
  bool swap;
};
__device__ __forceinline__ Split split_unitary(const M2 &U) {
  const double c = sqrt(U.a.re * U.a.re + U.a.im * U.a.im), s = sqrt(U.c.re * U.c.re + U.c.im * U.c.im);
  const C2 p = c > 0 ? C2{U.a.re / c, U.a.im / c} : C2{1, 0}, q = s > 0 ? C2{U.c.re / s, U.c.im / s} : C2{1, 0};
  const bool swap = s > c;
  const double m = swap ? s : c;
  return {cc(cm(p, q)), cm(q, cc(p)), {m * p.re, m * p.im}, (swap ? c : s) / m, swap};
}

__device__ __forceinline__ void setup_unitary(const qs_setup_args &A, const int32_t *w, int64_t b, int slot,
                                              const SetupCoef &coef) {
  float u[8];
  const M2 U = recipe_unitary(w, b, coef);
  store_m2(u, U);
  float4 *o = reinterpret_cast<float4 *>(A.utab + 8 * (w[0] + b));
  o[0] = make_float4(u[0], u[1], u[2], u[3]);
  o[1] = make_float4(u[4], u[5], u[6], u[7]);
  if (slot >= 0 && A.gtab) {
    const Split x = split_unitary(U);
    float4 *r = reinterpret_cast<float4 *>(A.gtab + slot + 8 * b);
    r[0] = make_float4((float)x.t, x.swap ? 1.f : 0.f, (float)x.g.re, (float)x.g.im);
    r[1] = make_float4((float)x.w.re, (float)x.w.im, (float)x.a.re, (float)x.a.im);
  } else if (slot >= 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) reinterpret_cast<float4 *>(A.ltab)[4 * slot + r] = lane_row(u, r, A.dagger);
  }
  if (A.qtab) recipe_generators(A.qtab, w, b, coef);
}

// A factor of a diagonal table, or a number: table word (kind, ref, mask).
__device__ __forceinline__ C2 setup_factor(const qs_setup_args &A, const int32_t *f, int64_t b, const SetupCoef &coef) {
  const int kind = f[0] & 7;
  if (kind == QS_FACTOR_ZW || kind == QS_FACTOR_ZNUM) {
    const float2 v = coef(f[1] + ((f[0] & QS_FACTOR_PER_SAMPLE) ? b : 0));
    const C2 z = {v.x, -(double)v.y};  // e^{-i phi / 2}, the value at bit 0
    if (kind == QS_FACTOR_ZNUM) return z;
    const C2 y = cm(cc(z), cc(z));
    const double m = z.re * z.re + z.im * z.im;
    return {y.re / m, y.im / m};
  }
  const Split x = split_unitary(recipe_unitary(A.words + f[1], b, coef));
  return kind == QS_FACTOR_G ? x.g : kind == QS_FACTOR_W ? x.w : x.a;
}

// One block per table (and sample): entry k is the product of the numbers and of
// the factors whose mask has odd parity with k.  Every factor is computed once,
// by its own thread, in double.
__device__ void setup_table(const qs_setup_args &A, const int32_t *t, int64_t b, const SetupCoef &coef) {
  __shared__ C2 fac[QS_SETUP_MAX_FACTORS];
  const int nf = t[2], nn = t[3], lane = threadIdx.x;
  const int32_t *f = t + 4;
  if (lane < nf) fac[lane] = setup_factor(A, f + 3 * lane, b, coef);
  C2 num = {1, 0};
  for (int k = lane; k < nn; k += 64) num = cm(num, setup_factor(A, f + 3 * (nf + k), b, coef));
  for (int off = 1; off < 64; off <<= 1) num = cm(num, C2{__shfl_xor(num.re, off, 64), __shfl_xor(num.im, off, 64)});
  __syncthreads();
  const int count = 1 << A.R;
  if (lane < count) {
    C2 v = num;
    for (int k = 0; k < nf; ++k)
      if (__popc(f[3 * k + 2] & lane) & 1) v = cm(v, fac[k]);
    reinterpret_cast<float2 *>(A.gtab + t[0])[(t[1] ? b * count : 0) + lane] = make_float2((float)v.re, (float)v.im);
  }
}

// Thread ranges, each rounded up to whole blocks: half-angle entries, unitaries
// shared by the batch, per-sample unitaries, tables, factors.  64-thread blocks: the
// items are few and long (double products, sincosf), so they spread over as
// many compute units as there are blocks.
__global__ void __launch_bounds__(64) k_setup(qs_setup_args A) {
  const SetupCoef coef{A};
  int64_t i = (blockIdx.y * (int64_t)gridDim.x + blockIdx.x) * 64 + threadIdx.x;
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
    if (i < nps) setup_unitary(A, A.words + A.sampled[2 * (i / A.B)], i % A.B, A.sampled[2 * (i / A.B) + 1], coef);
    return;
  }
  if (range(64 * A.ntables)) {
    setup_table(A, A.twords + A.tables[i >> 6], 0, coef);
    return;
  }
  if (range(64 * A.nstables * A.B)) {
    setup_table(A, A.twords + A.tables[A.ntables + (i >> 6) / A.B], (i >> 6) % A.B, coef);
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
  if (A.ntables < 0 || A.nstables < 0 || (A.ntables + A.nstables > 0 && (!A.tables || !A.twords || !A.gtab || !A.words || !A.cs)))
    return QS_EINVAL;
  if (A.R < 0 || A.R > 5) return QS_EINVAL;
  if ((A.nuniform > 0 && (!A.uniform || (!A.ltab && !A.gtab))) || (A.nsampled > 0 && !A.sampled)) return QS_EINVAL;
  if (A.efac && (!A.column || (A.lead && (!A.lead_words || !A.phi)))) return QS_EINVAL;
  const auto blocks = [](int64_t count) { return (count + 63) / 64; };
  const int64_t g = blocks(ncs) + blocks(A.nuniform) + blocks(A.nsampled * A.B) + A.ntables + A.nstables * A.B +
                    (A.efac ? blocks(A.B * A.n) : 0);
  if (g == 0) return QS_OK;
  // a row of the grid has fewer than 2^32 threads (a block per sample and table passes that
  // at 64 tables x 2^20 samples); the last row's surplus blocks find no item
  const int64_t row = g < (1 << 24) ? g : 1 << 24, rows = (g + row - 1) / row;
  if (rows > 0xffff) return QS_EUNSUPPORTED;
  hipLaunchKernelGGL(k_setup, dim3((unsigned)row, (unsigned)rows), dim3(64), 0, (hipStream_t)stream, A);
  return launch_status();
}

}  // extern "C"
