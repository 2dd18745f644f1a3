// Composition of fused per-bit unitaries in double precision: the 2x2 complex
// algebra and the recipe reader shared by the table kernels (qs_fused.hip,
// qs_setup.hip).
#pragma once

#include "qs_common.h"

namespace qs {

struct C2 {
  double re, im;
};
__device__ __forceinline__ C2 cm(C2 a, C2 b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ C2 ca(C2 a, C2 b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ C2 cc(C2 a) { return {a.re, -a.im}; }
struct M2 {
  C2 a, b, c, d;  // [[a, b], [c, d]]
};
__device__ __forceinline__ M2 mm(const M2 &x, const M2 &y) {
  return {ca(cm(x.a, y.a), cm(x.b, y.c)), ca(cm(x.a, y.b), cm(x.b, y.d)),
          ca(cm(x.c, y.a), cm(x.d, y.c)), ca(cm(x.c, y.b), cm(x.d, y.d))};
}
__device__ __forceinline__ M2 mdag(const M2 &x) { return {cc(x.a), cc(x.c), cc(x.b), cc(x.d)}; }

__device__ __forceinline__ M2 rot_matrix(int kind, float c, float s) {
  const C2 z = {0, 0};
  if (kind == QS_RX) return {{c, 0}, {0, -s}, {0, -s}, {c, 0}};
  if (kind == QS_RY) return {{c, 0}, {-s, 0}, {s, 0}, {c, 0}};
  if (kind == QS_RZ) return {{c, -s}, z, z, {c, s}};
  return {{1, 0}, z, z, {1, 0}};  // gradient probe
}
__device__ __forceinline__ M2 pauli(int p) {
  const C2 z = {0, 0};
  if (p == QS_RX) return {z, {1, 0}, {1, 0}, z};
  if (p == QS_RY) return {z, {0, -1}, {0, 1}, z};
  return {{1, 0}, z, z, {-1, 0}};
}
__device__ __forceinline__ void store_m2(float *o, const M2 &x) {
  o[0] = (float)x.a.re; o[1] = (float)x.a.im; o[2] = (float)x.b.re; o[3] = (float)x.b.im;
  o[4] = (float)x.c.re; o[5] = (float)x.c.im; o[6] = (float)x.d.re; o[7] = (float)x.d.im;
}

// Constituent k of recipe w for sample b; coef(i) is the (cos, sin) of entry i.
template <class Coef>
__device__ __forceinline__ M2 recipe_rot(const int32_t *w, int k, int64_t b, const Coef &coef, int *p) {
  const int kind = w[4 + 3 * k], ci = w[5 + 3 * k], cps = w[6 + 3 * k];
  *p = kind < 8 ? kind : kind - 8;
  if (kind >= 8) return rot_matrix(-1, 1.f, 0.f);
  const float2 v = coef(ci + (cps ? b : 0));
  return rot_matrix(kind, v.x, v.y);
}

// U = R_m ... R_1 of a recipe.
template <class Coef>
__device__ __forceinline__ M2 recipe_unitary(const int32_t *w, int64_t b, const Coef &coef) {
  int p;
  M2 U = {{1, 0}, {0, 0}, {0, 0}, {1, 0}};
  for (int k = 0; k < w[2]; ++k) U = mm(recipe_rot(w, k, b, coef, &p), U);
  return U;
}

// The gradient generators Q_k = V_k P_k V_k^dagger, V_k = R_m ... R_{k+1}, of a recipe.
template <class Coef>
__device__ __forceinline__ void recipe_generators(float *qtab, const int32_t *w, int64_t b, const Coef &coef) {
  const int64_t span = w[1], qidx = w[3];
  M2 V = {{1, 0}, {0, 0}, {0, 0}, {1, 0}};
  for (int k = w[2] - 1; k >= 0; --k) {
    int p;
    const M2 Rk = recipe_rot(w, k, b, coef, &p);
    store_m2(qtab + 8 * (qidx + k * span + b), mm(mm(V, pauli(p)), mdag(V)));
    V = mm(V, Rk);
  }
}

// Row r of the real 4x4 form of U (u00.re, u00.im, u01.re, ... as 8 floats) or,
// with dagger, of U^dagger (its transpose): the matrix-core operand of lane
// row r = lane & 3 (v_mfma_f32_4x4x1f32).
__device__ __forceinline__ float4 lane_row(const float *m, int r, int dagger) {
  const float a = m[0], b = m[1], c = m[2], d = m[3], e = m[4], f = m[5], g = m[6], h = m[7];
  if (!dagger) {
    if (r == 0) return make_float4(a, -b, c, -d);
    if (r == 1) return make_float4(b, a, d, c);
    if (r == 2) return make_float4(e, -f, g, -h);
    return make_float4(f, e, h, g);
  }
  if (r == 0) return make_float4(a, b, e, f);
  if (r == 1) return make_float4(-b, a, -f, e);
  if (r == 2) return make_float4(c, d, g, h);
  return make_float4(-d, c, -h, g);
}

}  // namespace qs
