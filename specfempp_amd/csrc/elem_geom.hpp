// Geometry of a tile kernel's elements, one column of GLL points per thread.
//
// A point's geometry is the five FP32 terms (xi_x, xi_z, ga_x, ga_z, J) that
// the host assembly forms from the control nodes (core/specfem/jacobian/dim2/
// jacobian.cpp:25-51).  4-node meshes re-form them from the control nodes
// with the host's operations in the host's order: coordinates far from the
// origin leave rounding in the sums, which the stiffness amplifies, so other
// sums would not give the same fields.  x_ga and z_ga do not change along a
// column (xi fixed); x_xi and z_xi cost 7 operations each per point, and the
// four quotients share one reciprocal.  9-node meshes (18 coordinates, 68
// operations per point) read the stored terms.
//
// Why: the stored terms are 500 B of an element, 240 MB of the 570 MB that
// the FP32 step kernel moved on 800x600 4-node elements; the control nodes
// are 32 B.  The step there went from 148 to 111 us.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "assembly2d.hpp"

namespace smx {

__device__ __forceinline__ float fma_(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}
__device__ __forceinline__ double fma_(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}

// base[i] for a base that every lane shares and an index below 2^32 / sizeof:
// one scalar address and a 32-bit lane offset, where a 64-bit address per
// lane would cost two registers each.
template <typename T>
__device__ __forceinline__ T &at32(T *base, uint32_t i) {
  using B = typename std::conditional<std::is_const<T>::value, const char, char>::type;
  return *reinterpret_cast<T *>(reinterpret_cast<B *>(base) + i * uint32_t(sizeof(T)));
}

// The value is formed here: without it the compiler moves a sum's arithmetic
// past the next barrier and keeps its 10 LDS operands in registers instead of
// the sum (k_tile before its element data were requested early: 72 registers
// and 76 B of spills, 56 and none with it).
template <typename real> __device__ __forceinline__ void formed(real &x) {
  asm volatile("" : "+v"(x));
}

// Quarter shape-function derivatives of 4-node elements at the GLL nodes:
// (s - 1) / 4 and (s + 1) / 4, exact scalings of the FP32 differences.
struct Q4Deriv {
  float m[NGLL], p[NGLL];
};
inline Q4Deriv q4_deriv(const float *xi) {
  Q4Deriv d;
  for (int i = 0; i < NGLL; ++i) {
    d.m[i] = 0.25f * (xi[i] - 1.0f);
    d.p[i] = 0.25f * (xi[i] + 1.0f);
  }
  return d;
}

// x_xi of the nodes c (from m, p at gamma), in the host's order; x_ga the
// same way from (m, p) at xi with the nodes in the order 0, 1, 2, 3 weighted
// (m, -p, p, -m).
__device__ __forceinline__ float q4_along_xi(const float c[4], float m, float p) {
#pragma clang fp contract(off)
  float s = m * c[0];
  s = s - m * c[1];
  s = s + p * c[2];
  return s - p * c[3];
}
__device__ __forceinline__ float q4_along_ga(const float c[4], float m, float p) {
#pragma clang fp contract(off)
  float s = m * c[0];
  s = s - p * c[1];
  s = s + p * c[2];
  return s - m * c[3];
}

// Five terms of one point, the derivatives of a field and the fluxes of a
// stress row (sx, sz).  The contractions are written out: which product of a
// sum is rounded first shows in the fields (two orders of a run's last step
// alone move its velocities by up to 7e-5), so it is not left to the
// compiler.  Z_FIRST adds the x product to the rounded z product, else the
// other way round.
template <typename real> struct PointMap {
  real xix, xiz, gax, gaz, jac;
  __device__ __forceinline__ real dx(real dxi, real dga) const {
    return fma_(xix, dxi, gax * dga);
  }
  __device__ __forceinline__ real dz(real dxi, real dga) const {
    return fma_(xiz, dxi, gaz * dga);
  }
  template <bool Z_FIRST = true>
  __device__ __forceinline__ real flux_xi(real sx, real sz) const {
    return jac * (Z_FIRST ? fma_(sx, xix, sz * xiz) : fma_(sz, xiz, sx * xix));
  }
  template <bool Z_FIRST = true>
  __device__ __forceinline__ real flux_ga(real sx, real sz) const {
    return jac * (Z_FIRST ? fma_(sx, gax, sz * gaz) : fma_(sz, gaz, sx * gax));
  }
};

// a / j from r = 1 / j to within an ulp: the quotient corrected once by its
// exact remainder, which rounds correctly unless a / j lies within 2^-46 of
// it from a tie (P. Markstein, IBM J. Res. Dev. 34, 1990).  J and the sums
// are far from the ends of the FP32 range (the host refuses J <= 1e-10).
__device__ __forceinline__ float quotient(float a, float j, float r) {
  const float q = a * r;
  return __builtin_fmaf(__builtin_fmaf(-q, j, a), r, q);
}

// The column's geometry: re-formed from 4-node elements' control nodes (geo:
// [8][ld], x0..x3, z0..z3), or STORED terms (geo: [5][NPT][ld], geo_e:
// [5][ld]).  centre: that of the element centre, for tiles of affine elements.
// slot0 is the tile's first slot, i the element in the tile.
template <typename real, bool STORED> struct ElemColumn;

template <typename real> struct ElemColumn<real, false> {
  using T = float;
  float x[4], z[4], xg, zg;
  const Q4Deriv &d;
  const int ix;
  const bool centre;
  __device__ __forceinline__ ElemColumn(const float *__restrict__ geo,
                                        const float *, size_t ld, size_t slot0,
                                        uint32_t i, int ix_, bool centre_,
                                        const Q4Deriv &d_)
      : d(d_), ix(ix_), centre(centre_) {
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      x[n] = at32(geo + n * ld + slot0, i);
      z[n] = at32(geo + (4 + n) * ld + slot0, i);
    }
  }
  // The column's sums; the constructor only requests the coordinates.
  __device__ __forceinline__ void open() {
    const float m = centre ? -0.25f : d.m[ix], p = centre ? 0.25f : d.p[ix];
    xg = q4_along_ga(x, m, p);
    zg = q4_along_ga(z, m, p);
  }
  __device__ __forceinline__ PointMap<real> at(int iz) const {
#pragma clang fp contract(off)
    const float m = centre ? -0.25f : d.m[iz], p = centre ? 0.25f : d.p[iz];
    const float xx = q4_along_xi(x, m, p), zx = q4_along_xi(z, m, p);
    const float j = xx * zg - xg * zx;
    const float r0 = __builtin_amdgcn_rcpf(j);
    const float r = __builtin_fmaf(__builtin_fmaf(-j, r0, 1.0f), r0, r0);
    return {real(quotient(zg, j, r)), real(quotient(-xg, j, r)),
            real(quotient(-zx, j, r)), real(quotient(xx, j, r)), real(j)};
  }
};

template <typename real> struct ElemColumn<real, true> {
  using T = real;
  const real *__restrict__ base;
  const size_t point, term;
  const uint32_t i;
  const int ix;
  __device__ __forceinline__ ElemColumn(const real *__restrict__ geo,
                                        const real *__restrict__ geo_e, size_t ld,
                                        size_t slot0, uint32_t i_, int ix_,
                                        bool centre, const Q4Deriv &)
      : base((centre ? geo_e : geo) + slot0), point(centre ? 0 : ld),
        term(centre ? ld : NPT * ld), i(i_), ix(ix_) {}
  __device__ __forceinline__ void open() {}
  __device__ __forceinline__ PointMap<real> at(int iz) const {
    const real *p = base + size_t(iz * NGLL + ix) * point;
    return {at32(p, i), at32(p + term, i), at32(p + 2 * term, i),
            at32(p + 3 * term, i), at32(p + 4 * term, i)};
  }
};

// What a tile launch is given: control nodes or stored terms.
template <typename real, bool STORED>
const typename ElemColumn<real, STORED>::T *geometry_source(const float *nodes,
                                                            const real *terms) {
  if constexpr (STORED)
    return terms;
  else
    return nodes;
}

} // namespace smx
