// Device-side Hex8 CVFEM sub-control-surface geometry per integration point.
// Everything that depends on the integration point is a compile-time constant:
// its isoparametric location, the shape-function derivative table and the four
// sub-division points of its surface.  The element-visit tiles (etile.hip) use
// these forms; the row kernels use hex8_row.hpp.
//
// Geometry restated from the mathematics of the reference:
//   * scs area vector (HexSCS::determinant, src/master_element/Hex8CVFEM.C:547-581,
//     quad_area_by_triangulation, include/master_element/Hex8GeometryFunctions.h:30-76):
//     the fan of four triangles around the quad centroid sums to the shoelace
//     form 1/2 (p2 - p0) x (p3 - p1), evaluated here directly;
//   * grad_op (generic_grad_op, include/master_element/MasterElementFunctions.h:51-108):
//     J_ij = sum_n dN_n/ds_j x_n,i, dN/dx = cof(J) dN/ds / det J.  Contractions
//     with the area vector use dN/dx . A = dN/ds . (cof(J)^T A) / det J.
// Floating-point results agree with the reference order to rounding.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace nalu {
namespace hex8 {

// corner signs of the Hex8 reference element (Hex8CVFEM.C nodeLoc_ :420-436)
__host__ __device__ constexpr int node_sign(int n, int d) {
  return d == 0 ? ((n == 1 || n == 2 || n == 5 || n == 6) ? 1 : -1)
       : d == 1 ? ((n == 2 || n == 3 || n == 6 || n == 7) ? 1 : -1)
                : (n >= 4 ? 1 : -1);
}

// scs left/right nodes (HexSCS::lrscv_, Hex8CVFEM.C:264-276)
__host__ __device__ constexpr int scs_left(int ip) {
  return ip < 4 ? (ip == 3 ? 0 : ip) : ip < 8 ? (ip == 7 ? 4 : ip) : ip - 8;
}
__host__ __device__ constexpr int scs_right(int ip) {
  return ip < 4 ? (ip == 3 ? 3 : ip + 1) : ip < 8 ? (ip == 7 ? 7 : ip + 1) : ip - 4;
}

// scs integration point location (HexSCS::intgLoc_, :318-330): midpoint of the
// edge (il, ir) pulled halfway to the element centroid in the other two
// directions; shifted (:333-345): on the edge itself.
__host__ __device__ constexpr double scs_loc(int ip, int d, bool shifted) {
  // edge direction of ip: 0 for ip 0,2,4,6; 1 for 1,3,5,7; 2 for 8..11
  return (ip >= 8 ? 2 : (ip & 1)) == d
             ? 0.0
             : (shifted ? 0.5 : 0.25) *
                   (double)(node_sign(scs_left(ip), d) + node_sign(scs_right(ip), d)) * 0.5;
}

// dN_n/ds_d at the scs ip = sign_d * prod_{e != d} (1/2 + sign_e s_e)
__host__ __device__ constexpr double deriv(int ip, int n, int d, bool shifted) {
  double v = (double)node_sign(n, d);
  for (int e = 0; e < 3; ++e)
    if (e != d) v *= 0.5 + (double)node_sign(n, e) * scs_loc(ip, e, shifted);
  return v;
}

// N_n at the scs ip = prod_e (1/2 + sign_e s_e)   (HexSCS::hex8_shape_fcn, :487-518)
__host__ __device__ constexpr double shape(int ip, int n, bool shifted) {
  double v = 1.0;
  for (int e = 0; e < 3; ++e) v *= 0.5 + (double)node_sign(n, e) * scs_loc(ip, e, shifted);
  return v;
}

// Sub-division points (subdivide_hex_8, Hex8GeometryFunctions.h:263-321) as
// corner masks: bit n set when corner n is averaged into the point.
__host__ __device__ constexpr uint32_t subdiv_mask(int p) {
  switch (p) {
    case 8: return 0x03;   // edge 0-1
    case 9: return 0x06;   // edge 1-2
    case 10: return 0x0c;  // edge 2-3
    case 11: return 0x09;  // edge 3-0
    case 12: return 0x0f;  // face 0123
    case 13: return 0x30;  // edge 4-5
    case 14: return 0x60;  // edge 5-6
    case 15: return 0xc0;  // edge 6-7
    case 16: return 0x90;  // edge 7-4
    case 17: return 0xf0;  // face 4567
    case 18: return 0x22;  // edge 1-5
    case 19: return 0x11;  // edge 0-4
    case 20: return 0x33;  // face 0145
    case 21: return 0x88;  // edge 3-7
    case 22: return 0x44;  // edge 2-6
    case 23: return 0xcc;  // face 2367
    case 24: return 0x66;  // face 1256
    case 25: return 0x99;  // face 0347
    case 26: return 0xff;  // centroid
    default: return 1u << p;
  }
}
__host__ __device__ constexpr int popc8(uint32_t m) {
  int c = 0;
  for (int i = 0; i < 8; ++i) c += (m >> i) & 1;
  return c;
}
// facet table of the 12 scs quads (Hex8CVFEM.C:551-564)
__host__ __device__ constexpr int facet(int ip, int k) {
  constexpr int t[12][4] = {{20, 8, 12, 26},  {24, 9, 12, 26},  {10, 12, 26, 23}, {11, 25, 26, 12},
                            {13, 20, 26, 17}, {17, 14, 24, 26}, {17, 15, 23, 26}, {16, 17, 26, 25},
                            {19, 20, 26, 25}, {20, 18, 24, 26}, {22, 23, 26, 24}, {21, 25, 26, 23}};
  return t[ip][k];
}
// weight of corner n in (point q - point p)
__host__ __device__ constexpr double diff_weight(int q, int p, int n) {
  const uint32_t mq = subdiv_mask(q), mp = subdiv_mask(p);
  return (((mq >> n) & 1) ? 1.0 / popc8(mq) : 0.0) - (((mp >> n) & 1) ? 1.0 / popc8(mp) : 0.0);
}

// area vector of scs IP: 1/2 (p2 - p0) x (p3 - p1)
template <int IP, typename R>
__device__ __forceinline__ void scs_area(const R (&x)[8][3], R (&A)[3]) {
  R d1[3], d2[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    R a = R(0), b = R(0);
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      const R w1 = R(diff_weight(facet(IP, 2), facet(IP, 0), n));
      const R w2 = R(diff_weight(facet(IP, 3), facet(IP, 1), n));
      a += w1 * x[n][i];
      b += w2 * x[n][i];
    }
    d1[i] = a;
    d2[i] = b;
  }
  A[0] = R(0.5) * (d1[1] * d2[2] - d1[2] * d2[1]);
  A[1] = R(0.5) * (d1[2] * d2[0] - d1[0] * d2[2]);
  A[2] = R(0.5) * (d1[0] * d2[1] - d1[1] * d2[0]);
}

// Jacobian J_ij = sum_n dN_n/ds_j x_n,i, its cofactor matrix and determinant.
// JR is the arithmetic type of the Jacobian (FP64 keeps det J exact enough on
// highly stretched elements while the rest of the kernel runs in R).
template <int IP, bool SHIFT, typename JR, typename R>
__device__ __forceinline__ void jacobian(const R (&x)[8][3], JR (&C)[3][3], JR& inv_det) {
  JR J[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      JR s = JR(0);
#pragma unroll
      for (int n = 0; n < 8; ++n) s += JR(deriv(IP, n, j, SHIFT)) * JR(x[n][i]);
      J[i][j] = s;
    }
  C[0][0] = J[1][1] * J[2][2] - J[2][1] * J[1][2];
  C[0][1] = J[1][2] * J[2][0] - J[2][2] * J[1][0];
  C[0][2] = J[1][0] * J[2][1] - J[2][0] * J[1][1];
  C[1][0] = J[0][2] * J[2][1] - J[2][2] * J[0][1];
  C[1][1] = J[0][0] * J[2][2] - J[2][0] * J[0][2];
  C[1][2] = J[0][1] * J[2][0] - J[2][1] * J[0][0];
  C[2][0] = J[0][1] * J[1][2] - J[1][1] * J[0][2];
  C[2][1] = J[0][2] * J[1][0] - J[1][2] * J[0][0];
  C[2][2] = J[0][0] * J[1][1] - J[1][0] * J[0][1];
  const JR det = J[0][0] * C[0][0] + J[1][0] * C[1][0] + J[2][0] * C[2][0];
  inv_det = JR(1) / det;
}

// g_k = sum_i C_ik A_i / det, so that dN_c/dx . A = dN_c/ds . g
template <typename JR, typename R>
__device__ __forceinline__ void contract_area(const JR (&C)[3][3], JR inv_det, const R (&A)[3], R (&g)[3]) {
#pragma unroll
  for (int k = 0; k < 3; ++k)
    g[k] = R((C[0][k] * JR(A[0]) + C[1][k] * JR(A[1]) + C[2][k] * JR(A[2])) * inv_det);
}

// Per-ip geometry.
template <typename JR, typename R>
struct IpGeo {
  R A[3];         // area vector
  JR C[3][3];     // cofactor matrix of J
  JR inv;         // 1 / det J
  R g[3];         // C^T A / det J: dN_c/dx . A = dN_c/ds . g
};

template <int IP, bool SHIFT, typename JR, typename R>
__device__ __forceinline__ void ip_geo(const R (&x)[8][3], IpGeo<JR, R>& G) {
  scs_area<IP>(x, G.A);
  jacobian<IP, SHIFT>(x, G.C, G.inv);
  contract_area(G.C, G.inv, G.A, G.g);
}

// dN_c/ds . g
template <int IP, int C, bool SHIFT, typename R>
__device__ __forceinline__ R dsdot(const R (&g)[3]) {
  return R(deriv(IP, C, 0, SHIFT)) * g[0] + R(deriv(IP, C, 1, SHIFT)) * g[1] + R(deriv(IP, C, 2, SHIFT)) * g[2];
}

// compile-time loop helpers
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

// dN_c/dx from Cs = cofactors / det J
template <int IP, int C, bool SHIFT, typename R>
__device__ __forceinline__ void dndx_scaled(const R (&Cs)[3][3], R (&dn)[3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
    dn[i] = Cs[i][0] * R(deriv(IP, C, 0, SHIFT)) + Cs[i][1] * R(deriv(IP, C, 1, SHIFT)) +
            Cs[i][2] * R(deriv(IP, C, 2, SHIFT));
}

}  // namespace hex8
}  // namespace nalu
