// Row-relative Hex8 element kernels: one thread evaluates the row of local node
// `la` of one element, with the element's corners numbered relative to that
// node.  Relative corner m (bits m0 m1 m2) is the corner that lies away from the
// row node along the directions whose bits are set; in local node numbers it is
// kHexOf[m] ^ la, because the Hex8 numbering is linear over XOR.  Reflecting the
// element this way gives one code path for all eight local nodes (a switch over
// compile-time nodes is eight copies of the arithmetic and diverges where the
// incident elements of neighbouring rows differ); only the handedness h = +-1
// of the reflection remains.
//
// With t_d in [0, 1] the distance from the row node, the sub-control surface
// (scs) of the row node's edge along d has its integration point at t_d = 1/2
// and 1/4 in the other two directions (e, f) = (d+1, d+2) mod 3 -- on the edge
// itself (0) for the shifted form.  The geometry follows from the trilinear map
// x(t) and its derivatives a_k = dx/dt_k at the point:
//   * the scs quadrilateral joins edge midpoint, face centroids and element
//     centroid, all points of the map, so it is the bilinear patch
//     t_e, t_f in [0, 1/2]; the area vector of a bilinear patch is its parametric
//     area times the cross product of its tangents at its centre, which is the
//     integration point:  A_out = h/4 a_e x a_f   (HexSCS::determinant,
//     src/master_element/Hex8CVFEM.C:547-581, sums four triangles per patch);
//   * with the cofactor columns C_k = a_{k+1} x a_{k+2}, dN/dx = sum_k dN/dt_k C_k / det
//     (generic_grad_op, include/master_element/MasterElementFunctions.h:51-108),
//     so C_d serves both and dN/dx . A_out = sum_k dN/dt_k g_k, g_k = C_k . A_out / det.
// The a_k come from the twelve edge vectors with weights 9, 3, 3, 1 (along d) and
// 3, 1 (across), powers of two divided out at the end (exact).  Per row of an
// element this takes about 230 FP64 instructions for the three scs, against about
// 500 for 8-node sums of the Jacobian and of the patch corners.
#pragma once

#include "hex8_device.hpp"

namespace nalu {
namespace hexrow {

__host__ __device__ constexpr int hex_of(int m) { return m ^ ((m >> 1) & 1); }  // 0 1 3 2 4 5 7 6

// corner of direction d's far (cd = 1) or near side, be / bf away along d+1 / d+2
__host__ __device__ constexpr int corner(int d, int cd, int be, int bf) {
  return (cd << d) | (be << ((d + 1) % 3)) | (bf << ((d + 2) % 3));
}

// v[i] <- v[i ^ la], then renumbered from local-node to relative-corner order
template <typename T>
__device__ __forceinline__ void relative_order(T (&v)[8], int la) {
#pragma unroll
  for (int b = 1; b < 8; b <<= 1) {
    const bool sw = (la & b) != 0;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (!(i & b)) {
        const T p = v[i], q = v[i | b];
        v[i] = sw ? q : p;
        v[i | b] = sw ? p : q;
      }
  }
  T t = v[2]; v[2] = v[3]; v[3] = t;
  t = v[6]; v[6] = v[7]; v[7] = t;
}

// row positions (one byte per local node) in relative-corner order: byte m of the result
__device__ __forceinline__ uint64_t relative_bytes(uint64_t pk, int la) {
  const uint32_t lo = (uint32_t)pk, hi = (uint32_t)(pk >> 32);
  const uint32_t sel = 0x02030100u ^ (0x01010101u * (uint32_t)(la & 3));
  const bool sw = (la & 4) != 0;
  const uint32_t a = __builtin_amdgcn_perm(0u, sw ? hi : lo, sel);
  const uint32_t b = __builtin_amdgcn_perm(0u, sw ? lo : hi, sel);
  return (uint64_t)a | ((uint64_t)b << 32);
}
__device__ __forceinline__ int pos(uint64_t bytes, int m) { return (int)((bytes >> (8 * m)) & 0xff); }

// handedness of the reflection that brings node la to relative corner 0
__device__ __forceinline__ double handed(int la) { return ((la ^ (la >> 2)) & 1) ? -1.0 : 1.0; }

// the scs of node la's edge along d, and whether la is its left node (lrscv)
__device__ __forceinline__ int scs_of(int la, int d) {
  return d == 0 ? (la & 6) : d == 1 ? ((la & 4) | (((la ^ (la >> 1)) & 1) ? 1 : 3)) : 8 + (la & 3);
}
__device__ __forceinline__ bool scs_is_left(int la, int d) {
  return d == 0 ? !(la & 1) : d == 1 ? !(la & 2) : !(la & 4);
}

// 1/d: hardware estimate and two Newton steps (about one ulp), special values as a division gives them
__device__ __forceinline__ double recip(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  return __builtin_amdgcn_div_fixup(r, d, 1.0);
}

// x: coordinates by component and relative corner; edge vectors E[d][be + 2 bf] from the near to the far corner along d
struct Edges {
  double e[3][4][3];
};
__device__ __forceinline__ void edges(const double (&x)[3][8], Edges& E) {
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 3; ++i) E.e[d][q][i] = x[i][corner(d, 1, q & 1, q >> 1)] - x[i][corner(d, 0, q & 1, q >> 1)];
}

__device__ __forceinline__ void cross(const double (&a)[3], const double (&b)[3], double (&c)[3]) {
  c[0] = a[1] * b[2] - a[2] * b[1];
  c[1] = a[2] * b[0] - a[0] * b[2];
  c[2] = a[0] * b[1] - a[1] * b[0];
}
__device__ __forceinline__ double dot(const double (&a)[3], const double (&b)[3]) {
  return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

// The scs of direction D nearest to the row node, or, for kernels that evaluate
// a whole element, the one in the quadrant (QE, QF) of far sides along D+1, D+2.
// Tangents at its integration point: a[0] along D, a[1], a[2] along D+1, D+2,
// scaled by 16, 8, 8 (SHIFT: 1, 2, 2).
template <int D, bool SHIFT, int QE = 0, int QF = 0>
__device__ __forceinline__ void tangents(const Edges& E, double (&a)[3][3]) {
  constexpr int e = (D + 1) % 3, f = (D + 2) % 3, Q = QE | (QF << 1);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (SHIFT) {
      a[0][i] = E.e[D][Q][i];
      a[1][i] = E.e[e][QF][i] + E.e[e][2 | QF][i];
      a[2][i] = E.e[f][2 * QE][i] + E.e[f][1 | 2 * QE][i];
    } else {
      const double t0 = 3.0 * E.e[D][Q][i] + E.e[D][Q ^ 1][i], t1 = 3.0 * E.e[D][Q ^ 2][i] + E.e[D][Q ^ 3][i];
      a[0][i] = 3.0 * t0 + t1;
      a[1][i] = 3.0 * (E.e[e][QF][i] + E.e[e][2 | QF][i]) + (E.e[e][1 ^ QF][i] + E.e[e][3 ^ QF][i]);
      a[2][i] = 3.0 * (E.e[f][2 * QE][i] + E.e[f][1 | 2 * QE][i]) + (E.e[f][2 ^ 2 * QE][i] + E.e[f][3 ^ 2 * QE][i]);
    }
  }
}

// Cofactor columns along D, D+1, D+2 of the scaled tangents and 1 / det of them;
// with scale factors kc: dN/dx = sum_k dN/dt_k (kc_k C_k / det)
template <bool SHIFT>
struct Scale {
  static constexpr double c0 = SHIFT ? 1.0 : 16.0, c1 = SHIFT ? 2.0 : 8.0;
};
struct Cof {
  double c[3][3];
  double inv;
};
template <int D, bool SHIFT, int QE = 0, int QF = 0>
__device__ __forceinline__ void cofactors(const Edges& E, Cof& K) {
  double a[3][3];
  tangents<D, SHIFT, QE, QF>(E, a);
  cross(a[1], a[2], K.c[0]);
  cross(a[2], a[0], K.c[1]);
  cross(a[0], a[1], K.c[2]);
  K.inv = recip(dot(a[0], K.c[0]));
}

// outward area vector of the scs of direction D
template <int D, int QE = 0, int QF = 0>
__device__ __forceinline__ void area(const Edges& E, double h, double (&A)[3]) {
  double a[3][3], c[3];
  tangents<D, false, QE, QF>(E, a);
  cross(a[1], a[2], c);
#pragma unroll
  for (int i = 0; i < 3; ++i) A[i] = (h * (1.0 / 256)) * c[i];
}

// area vector and cofactors together (one cross product serves both when not shifted)
template <int D, bool SHIFT, int QE = 0, int QF = 0>
__device__ __forceinline__ void area_cofactors(const Edges& E, double h, double (&A)[3], Cof& K) {
  cofactors<D, SHIFT, QE, QF>(E, K);
  if constexpr (SHIFT) {
    area<D, QE, QF>(E, h, A);
  } else {
#pragma unroll
    for (int i = 0; i < 3; ++i) A[i] = (h * (1.0 / 256)) * K.c[0][i];
  }
}

// g_k = C_k . A / det along D, D+1, D+2
template <bool SHIFT, typename R>
__device__ __forceinline__ void metric(const Cof& K, const double (&A)[3], R (&g)[3]) {
  g[0] = R(dot(K.c[0], A) * (K.inv * Scale<SHIFT>::c0));
  g[1] = R(dot(K.c[1], A) * (K.inv * Scale<SHIFT>::c1));
  g[2] = R(dot(K.c[2], A) * (K.inv * Scale<SHIFT>::c1));
}

// value at the scs of a nodal field in relative order
template <int D, bool SHIFT, int QE = 0, int QF = 0, typename R>
__device__ __forceinline__ R at_scs(const R (&v)[8]) {
  if constexpr (SHIFT) return R(0.5) * (v[corner(D, 0, QE, QF)] + v[corner(D, 1, QE, QF)]);
  R s[4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
    s[q] = v[corner(D, 0, (q & 1) ^ QE, (q >> 1) ^ QF)] + v[corner(D, 1, (q & 1) ^ QE, (q >> 1) ^ QF)];
  return R(1.0 / 32) * (R(3) * (R(3) * s[0] + s[1]) + (R(3) * s[2] + s[3]));
}

// shape function of relative corner m at the scs of direction D nearest to the row node
template <int D, bool SHIFT>
__host__ __device__ constexpr double scs_shape(int m) {
  const int b = ((m >> (D + 1) % 3) & 1) + ((m >> (D + 2) % 3) & 1);
  return SHIFT ? (b ? 0.0 : 0.5) : (b == 0 ? 9.0 / 32 : b == 1 ? 3.0 / 32 : 1.0 / 32);
}
// its derivative along k = 0, 1, 2 for the directions D, D+1, D+2
template <int D, bool SHIFT>
__host__ __device__ constexpr double scs_slope(int m, int k) {
  const int d = (m >> D) & 1, e = (m >> (D + 1) % 3) & 1, f = (m >> (D + 2) % 3) & 1;
  const double we = SHIFT ? (e ? 0.0 : 1.0) : (e ? 0.25 : 0.75), wf = SHIFT ? (f ? 0.0 : 1.0) : (f ? 0.25 : 0.75);
  return k == 0 ? (d ? we * wf : -we * wf) : k == 1 ? (e ? 0.5 * wf : -0.5 * wf) : (f ? 0.5 * we : -0.5 * we);
}

// sum_k dN_m/dt_k g_k for the eight corners m: the part Q that is equal on the
// near and the far corner of an edge and the part P that changes sign.
// emit(m, value) is called once per corner, corners of weight zero left out.
template <int D, bool SHIFT, typename R, class Emit>
__device__ __forceinline__ void slope(const R (&g)[3], Emit&& emit) {
  if constexpr (SHIFT) {
    const R q = R(-0.5) * (g[1] + g[2]);
    emit(corner(D, 0, 0, 0), q - g[0]);
    emit(corner(D, 1, 0, 0), q + g[0]);
    emit(corner(D, 0, 1, 0), R(0.5) * g[1]);
    emit(corner(D, 1, 1, 0), R(0.5) * g[1]);
    emit(corner(D, 0, 0, 1), R(0.5) * g[2]);
    emit(corner(D, 1, 0, 1), R(0.5) * g[2]);
  } else {
    const R s = R(0.125) * (g[1] + g[2]);
    const R q[4] = {R(-3) * s, R(0.5) * g[1] - s, R(0.5) * g[2] - s, s};
    const R p2 = R(0.0625) * g[0], p1 = R(0.1875) * g[0], p0 = R(0.5625) * g[0];
    const R p[4] = {p0, p1, p1, p2};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      emit(corner(D, 0, k & 1, k >> 1), q[k] - p[k]);
      emit(corner(D, 1, k & 1, k >> 1), q[k] + p[k]);
    }
  }
}

// derivatives along D, D+1, D+2 of a nodal field at the scs of direction D
template <int D, bool SHIFT, int QE = 0, int QF = 0, typename R>
__device__ __forceinline__ void param_grad(const R (&v)[8], R (&dv)[3]) {
  auto c = [&](int cd, int be, int bf) { return v[corner(D, cd, be, bf)]; };
  auto sd = [&](int be, int bf) { return c(1, be, bf) - c(0, be, bf); };
  auto se = [&](int bf) { return (c(0, 1, bf) - c(0, 0, bf)) + (c(1, 1, bf) - c(1, 0, bf)); };
  auto sf = [&](int be) { return (c(0, be, 1) - c(0, be, 0)) + (c(1, be, 1) - c(1, be, 0)); };
  if constexpr (SHIFT) {
    dv[0] = sd(QE, QF);
    dv[1] = R(0.5) * se(QF);
    dv[2] = R(0.5) * sf(QE);
  } else {
    dv[0] = R(1.0 / 16) * (R(3) * (R(3) * sd(QE, QF) + sd(1 ^ QE, QF)) + (R(3) * sd(QE, 1 ^ QF) + sd(1 ^ QE, 1 ^ QF)));
    dv[1] = R(0.125) * (R(3) * se(QF) + se(1 ^ QF));
    dv[2] = R(0.125) * (R(3) * sf(QE) + sf(1 ^ QE));
  }
}

// Volume of the sub-control volume at relative corner 0 (HexSCV::determinant,
// src/master_element/Hex8CVFEM.C:149-178; hex_volume_grandy,
// include/master_element/Hex8GeometryFunctions.h:78-163).  Grandy's sum over the
// four triangles about each face centroid m is 1/6 sum_faces m . (q2 - q0) x (q3 - q1);
// taken relative to the row node, the three faces at the node reduce to half a
// triple product each.  About 150 FP64 instructions, against about 900 for the 24
// triangles.  h: handedness of the reflection.
__device__ __forceinline__ double scv_volume(const double (&x)[3][8], double h) {
  double c[8][3];  // the sub-hexahedron's corners relative to the row node, times 8
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    double D[8];
#pragma unroll
    for (int m = 1; m < 8; ++m) D[m] = x[i][m] - x[i][0];
    c[0][i] = 0.0;
    c[1][i] = 4.0 * D[1];
    c[2][i] = 4.0 * D[2];
    c[4][i] = 4.0 * D[4];
    const double s12 = D[1] + D[2], s14 = D[1] + D[4], s24 = D[2] + D[4];
    c[3][i] = 2.0 * (s12 + D[3]);
    c[5][i] = 2.0 * (s14 + D[5]);
    c[6][i] = 2.0 * (s24 + D[6]);
    c[7][i] = ((s12 + D[3]) + (D[4] + D[5])) + (D[6] + D[7]);
  }
  double vol = 0.0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int e = 1 << (d + 1) % 3, f = 1 << (d + 2) % 3, o = 1 << d;
    double u[3], v[3], m[3], n[3];
    // near face (row node, e, e|f, f): m . n = 1/2 det(c_e, c_ef, c_f)
    cross(c[e | f], c[f], n);
    vol -= 0.5 * dot(c[e], n);
    // far face
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      u[i] = c[o | e | f][i] - c[o][i];
      v[i] = c[o | f][i] - c[o | e][i];
      m[i] = (c[o][i] + c[o | e | f][i]) + (c[o | e][i] + c[o | f][i]);
    }
    cross(u, v, n);
    vol += 0.25 * dot(m, n);
  }
  return h * vol * (1.0 / (6 * 512));
}

// Shape function of relative corner m at the scv's integration point: the scv
// centroid (HexSCV::intgLoc_, Hex8CVFEM.C:88-96), (3/4)^a (1/4)^b with b bits set
// in m; the lumped form (shifted locations, :99-107) is 1 at the row node.
template <bool LUMPED>
__host__ __device__ constexpr double scv_shape(int m) {
  if (LUMPED) return m == 0 ? 1.0 : 0.0;
  const int b = (m & 1) + ((m >> 1) & 1) + (m >> 2);
  return b == 0 ? 27.0 / 64 : b == 1 ? 9.0 / 64 : b == 2 ? 3.0 / 64 : 1.0 / 64;
}

// scv interpolation of a nodal field in relative order
template <bool LUMPED>
__device__ __forceinline__ double at_scv(const double (&v)[8]) {
  if (LUMPED) return v[0];
  const double a = 3.0 * v[0] + v[1], b = 3.0 * v[2] + v[3], c = 3.0 * v[4] + v[5], d = 3.0 * v[6] + v[7];
  return (1.0 / 64) * (3.0 * (3.0 * a + b) + (3.0 * c + d));
}

}  // namespace hexrow
}  // namespace nalu
