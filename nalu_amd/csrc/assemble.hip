// Fused Hex8 CVFEM assembly: gather + scs geometry + element kernel + scatter
// in one pass over the mesh (the consolidated AssembleElemSolverAlgorithm,
// src/AssembleElemSolverAlgorithm.C:75-100 and include/AssembleElemSolverAlgorithm.h:52-105,
// whose per-element lhs/rhs go through SolverAlgorithm::apply_coeff ->
// TpetraLinearSystem::sumInto, src/TpetraLinearSystem.C:1457-1522).
//
// All kernels share the row arithmetic of hex8_row.hpp: one thread evaluates the
// row of one node in one incident element, its corners numbered relative to that
// node, on one code path for all eight local nodes.  Two scatter strategies:
//   * owner-computes row tiles (modes 0 and 2): a wave owns consecutive scalar rows
//     and four lanes of a row take its incident elements, a block owns consecutive
//     nodes of a numDof 3 system and eight threads take a node's; the rows meet in
//     the wave's or block's LDS copy of their CSR segment, which is written once,
//     coalesced; a pending zeroSystem is folded into that write.
//   * element-centric atomic scatter (mode 1): a block evaluates one local node's
//     row of a chunk of elements, FP64 atomic adds into the CSR.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "hex8_device.hpp"
#include "hex8_row.hpp"
#include "internal.hpp"

namespace nalu {
namespace {

inline unsigned blocks_for(int64_t n, int per) { return (unsigned)std::max<int64_t>(1, (n + per - 1) / per); }

// ---------------------------------------------------------------- element data in relative order
struct RowElem {
  uint32_t nd[8];  // nodes by relative corner (hex8_row.hpp)
  int la;          // the row's local node
  int64_t e;
};

__device__ __forceinline__ RowElem row_elem(const int32_t* __restrict__ conn, int64_t e, int la) {
  const int4* c4 = reinterpret_cast<const int4*>(conn + 8 * e);
  const int4 a = c4[0], b = c4[1];
  RowElem r{{(uint32_t)a.x, (uint32_t)a.y, (uint32_t)a.z, (uint32_t)a.w, (uint32_t)b.x, (uint32_t)b.y, (uint32_t)b.z,
             (uint32_t)b.w},
            la, e};
  hexrow::relative_order(r.nd, la);
  return r;
}

// A vector field [N][3] and, with it, a scalar field [N] (or none), as the caller
// holds them, or (PACK) copied together to 16-byte entries of one array per half:
// (v0, v1) and (v2, s) in double, (v0, v1, v2, s) in float.  The vector cache
// serves four lanes a cycle from one 64-byte line each.  Neighbouring lanes read
// neighbouring nodes, so a load of 16-byte entries takes 16 cycles for 1 KB, one of
// a scalar field 16 cycles for 512 B, and the two loads of a 24-byte [N][3] entry
// about 55 cycles for 1.5 KB.  That rate bounds the row kernels, which read each
// node's fields for up to eight elements of eight rows, so larger systems first
// copy the fields of a pass (k_pack, k_pack_flux; 40 us for continuity at 128^3).
// Entry offsets are 32-bit.
template <typename T>
struct alignas(16) Half {
  T v[16 / sizeof(T)];
};
template <typename T = double>
struct Field4 {
  const Half<T>* h[2];  // PACK (the second for double only)
  const double* vec;    // otherwise [N][3]
  const double* scal;   // and [N], or null
};

template <typename T>
__device__ __forceinline__ Half<T> half_at(const Half<T>* __restrict__ f, uint32_t n) {
  return *reinterpret_cast<const Half<T>*>(reinterpret_cast<const char*>(f) + (uint32_t)(16 * n));
}

template <bool PACK, typename R>
__device__ __forceinline__ void load1(const double* __restrict__ f, const uint32_t (&nd)[8], R (&v)[8]) {
#pragma unroll
  for (int m = 0; m < 8; ++m)
    v[m] = PACK ? R(*reinterpret_cast<const double*>(reinterpret_cast<const char*>(f) + (uint32_t)(8 * nd[m])))
                : R(f[nd[m]]);
}
// vector part component-major, v[i][m]; scalar part s[m] (SCAL)
template <bool PACK, bool SCAL, typename T, typename R, typename S>
__device__ __forceinline__ void load4(const Field4<T>& f, const uint32_t (&nd)[8], R (&v)[3][8], S (&s)[8]) {
#pragma unroll
  for (int m = 0; m < 8; ++m) {
    if (PACK) {
      const Half<T> r = half_at(f.h[0], nd[m]);
      if constexpr (sizeof(T) == 8) {
        const Half<T> r2 = half_at(f.h[1], nd[m]);
        v[0][m] = R(r.v[0]);
        v[1][m] = R(r.v[1]);
        v[2][m] = R(r2.v[0]);
        if (SCAL) s[m] = S(r2.v[1]);
      } else {
#pragma unroll
        for (int i = 0; i < 3; ++i) v[i][m] = R(r.v[i]);
        if (SCAL) s[m] = S(r.v[3]);
      }
    } else {
      const double* q = f.vec + 3 * (uint64_t)nd[m];
#pragma unroll
      for (int i = 0; i < 3; ++i) v[i][m] = R(q[i]);
      if (SCAL) s[m] = S(f.scal[nd[m]]);
    }
  }
}
template <bool PACK, typename R>
__device__ __forceinline__ void load3(const Field4<double>& f, const uint32_t (&nd)[8], R (&v)[3][8]) {
  R none[8];
  load4<PACK, false>(f, nd, v, none);
}

// Copies of up to six (vector, scalar) field pairs, 2 nnodes entries each.
struct PackList {
  const double* vec[6];
  const double* scal[6];
  int n;
};
__global__ __launch_bounds__(256) void k_pack(PackList L, int64_t nnodes, Half<double>* __restrict__ dst) {
  const int64_t a = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (a >= nnodes) return;
  for (int k = 0; k < L.n; ++k) {
    const double* f = L.vec[k] + 3 * a;
    dst[2 * k * nnodes + a] = {{f[0], f[1]}};
    dst[(2 * k + 1) * nnodes + a] = {{f[2], L.scal[k] ? L.scal[k][a] : 0.0}};
  }
}
// Copies of (coordinates, p) and, in the arithmetic type, of the mass flux vector rho u + tau Gp.
template <typename R>
__global__ __launch_bounds__(256) void k_pack_flux(const double* __restrict__ coords, const double* __restrict__ p,
                                                   const double* __restrict__ rho, const double* __restrict__ u,
                                                   const double* __restrict__ gp, double tau, int64_t nnodes,
                                                   Half<double>* __restrict__ x, Half<R>* __restrict__ W) {
  const int64_t a = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (a >= nnodes) return;
  const R r = R(rho[a]);
  R w[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) w[i] = r * R(u[3 * a + i]) + R(tau) * R(gp[3 * a + i]);
  x[a] = {{coords[3 * a], coords[3 * a + 1]}};
  x[nnodes + a] = {{coords[3 * a + 2], p[a]}};
  if constexpr (sizeof(R) == 8) {
    W[a] = {{w[0], w[1]}};
    W[nnodes + a] = {{w[2], 0.0}};
  } else {
    W[a] = {{w[0], w[1], w[2], 0.0f}};
  }
}

using hex8::static_for;

// Phase boundaries of a row's evaluation.  Left alone, the compiler interleaves
// the three directions and hoists every field load to the top, which takes up to
// twice the registers (half the waves in flight, or spills).  An empty asm that
// "modifies" a value orders what produces it before what uses it, and volatile
// asms keep their order: pin the results of one phase, then the inputs of the next.
template <typename T>
__device__ __forceinline__ void pin(T& v) {
  asm volatile("" : "+v"(v));
}
template <typename T, int N>
__device__ __forceinline__ void pin(T (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) pin(v[i]);
}
__device__ __forceinline__ void pin(hexrow::Edges& E) { pin(E.e); }
// loads through a node list pinned here stay after it
__device__ __forceinline__ void pin(RowElem& r) { pin(r.nd); }

// ---------------------------------------------------------------- scalar systems
// Each op evaluates the row of r.la in element r.e: v[m] gets the entry of
// relative corner m's column, the return value is the row's rhs contribution
// (times rhs_scale).  R is the arithmetic type of the physics (double, or float
// for the mixed-precision path); the geometry is always FP64.

// ScalarDiffElemKernel (src/kernel/ScalarDiffElemKernel.C:66-111): entry -sum_scs k_ip dN/dx . A_out, rhs -entry . q
template <bool SHIFT, bool PACK, typename R>
struct ScalarDiffOp {
  Field4<> xk;      // coordinates and conductivity
  const double* q;
  double rhs_scale() const { return 1.0; }
  __device__ __forceinline__ double eval(RowElem& r, double (&v)[8]) const {
    R g[3][3], kn[8], qn[8], w[8];
    {
      double x[3][8];
      load4<PACK, true>(xk, r.nd, x, kn);
      hexrow::Edges E;
      hexrow::edges(x, E);
      const double h = hexrow::handed(r.la);
      static_for<3>([&](auto dd) {
        constexpr int D = decltype(dd)::value;
        double A[3];
        hexrow::Cof K;
        hexrow::area_cofactors<D, SHIFT>(E, h, A, K);
        hexrow::metric<SHIFT>(K, A, g[D]);
        pin(g[D]);
        pin(E);
      });
    }
    pin(r);
    load1<PACK>(q, r.nd, qn);
#pragma unroll
    for (int m = 0; m < 8; ++m) w[m] = R(0);
    static_for<3>([&](auto dd) {
      constexpr int D = decltype(dd)::value;
      const R kip = hexrow::at_scs<D, false>(kn);
#pragma unroll
      for (int i = 0; i < 3; ++i) g[D][i] *= kip;
      hexrow::slope<D, SHIFT>(g[D], [&](int m, R t) { w[m] -= t; });
    });
    R rhs = R(0);
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      rhs -= w[m] * qn[m];
      v[m] = (double)w[m];
    }
    return (double)rhs;
  }
};

// ContinuityAdvElemKernel (src/kernel/ContinuityAdvElemKernel.C:88-148) with the mass
// flow rate of ComputeMdotElemAlgorithm (src/ComputeMdotElemAlgorithm.C:204-232) at
// each scs: mdot = (rho u + tau Gp)_ip . A - tau grad p . A; entry -sum_scs dN_lhs/dx . A_out,
// rhs -sum mdot_out / tau (the division is left to rhs_scale).  MDOT: the row of the
// left node also writes the scs's mdot (each scs has exactly one left node, so the
// rows of an element deliver all twelve).
template <bool SHIFT_MDOT, bool SHIFT_POISSON, bool REDUCED, bool MDOT, bool PACK, typename R>
struct ContinuityOp {
  Field4<> xp;        // coordinates and pressure
  Field4<R> W4;       // PACK: rho u + tau Gp (k_pack_flux)
  Field4<> ur;        // otherwise u and rho,
  const double* gp;   // and Gp
  double tau;
  double* mdot_out;  // [E][12] (MDOT)
  double rhs_scale() const { return 1.0 / tau; }
  __device__ __forceinline__ double eval(RowElem& r, double (&v)[8]) const {
    constexpr bool LHS_SHIFT = SHIFT_POISSON || REDUCED, TWO = LHS_SHIFT != SHIFT_POISSON;
    // geometry: area vectors and metrics of the three directions
    R A[3][3], g[3][3], gp_[TWO ? 3 : 1][3], pn[8];
    {
      double x[3][8];
      load4<PACK, true>(xp, r.nd, x, pn);
      hexrow::Edges E;
      hexrow::edges(x, E);
      const double h = hexrow::handed(r.la);
      static_for<3>([&](auto dd) {
        constexpr int D = decltype(dd)::value;
        double a[3];
        hexrow::Cof K;
        hexrow::area_cofactors<D, LHS_SHIFT>(E, h, a, K);
        hexrow::metric<LHS_SHIFT>(K, a, g[D]);
        if constexpr (TWO) {
          hexrow::cofactors<D, SHIFT_POISSON>(E, K);
          hexrow::metric<SHIFT_POISSON>(K, a, gp_[D]);
          pin(gp_[D]);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) A[D][i] = R(a[i]);
        pin(A[D]);
        pin(g[D]);
        pin(E);
      });
    }
    // flux through the scs and matrix entries
    pin(r);
    R W[3][8], w[8], out = R(0);
    if constexpr (PACK) {
      R none[8];
      load4<true, false>(W4, r.nd, W, none);
    } else {
      R rn[8], gn[3][8];
      load4<false, true>(ur, r.nd, W, rn);
      load3<false>(Field4<>{{}, gp, nullptr}, r.nd, gn);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int m = 0; m < 8; ++m) W[i][m] = rn[m] * W[i][m] + R(tau) * gn[i][m];
    }
#pragma unroll
    for (int m = 0; m < 8; ++m) w[m] = R(0);
    static_for<3>([&](auto dd) {
      constexpr int D = decltype(dd)::value;
      R dp = R(0);
      hexrow::slope<D, LHS_SHIFT>(g[D], [&](int m, R t) {
        w[m] -= t;
        if constexpr (!TWO) dp += pn[m] * t;
      });
      if constexpr (TWO) {
        R ps[3];
        hexrow::param_grad<D, SHIFT_POISSON>(pn, ps);
        dp = ps[0] * gp_[D][0] + ps[1] * gp_[D][1] + ps[2] * gp_[D][2];
      }
      R f = -R(tau) * dp;
#pragma unroll
      for (int i = 0; i < 3; ++i) f += hexrow::at_scs<D, SHIFT_MDOT>(W[i]) * A[D][i];
      out += f;
      if constexpr (MDOT)
        if (hexrow::scs_is_left(r.la, D)) mdot_out[12 * r.e + hexrow::scs_of(r.la, D)] = (double)f;
    });
#pragma unroll
    for (int m = 0; m < 8; ++m) v[m] = (double)w[m];
    return -(double)out;
  }
};

// Element-centric kernels: a block handles one local row node LA of a chunk of
// kChunk elements.  The eight LA-blocks of a chunk are consecutive in the
// dispatch order of one XCD (block b runs on XCD b % 8), so the chunk's nodal
// data is shared through that XCD's L2.
constexpr int kChunk = 256;

struct ChunkMap {
  int64_t e;   // element of this thread
  int la;      // block-uniform local row node (0..NL-1)
  bool valid;
};
template <int NL>
__device__ __forceinline__ ChunkMap chunk_map(int64_t nelem) {
  const unsigned b = blockIdx.x;
  const unsigned xcd = b & 7, la = (b >> 3) % NL, grp = (b >> 3) / NL;
  const int64_t chunk = (int64_t)grp * 8 + xcd;
  const int64_t e = chunk * kChunk + threadIdx.x;
  return {e, (int)la, e < nelem};
}
template <int NL>
inline unsigned chunk_blocks(int64_t nelem) {
  const int64_t nchunk = (nelem + kChunk - 1) / kChunk;
  return (unsigned)(((nchunk + 7) / 8) * 8 * NL);
}

template <class Op>
__global__ __launch_bounds__(kChunk) void k_scalar_atomic(Op op, const int32_t* __restrict__ conn,
                                                          const int32_t* __restrict__ lid,
                                                          const int32_t* __restrict__ nrp,
                                                          ElemPos elem_pos, int64_t nelem,
                                                          double rhs_scale, double* __restrict__ vals,
                                                          double* __restrict__ rhs) {
  const ChunkMap cm = chunk_map<8>(nelem);
  if (!cm.valid) return;
  RowElem r = row_elem(conn, cm.e, cm.la);
  const int32_t row = lid[r.nd[0]];
  double* rowp = vals + nrp[row];
  const uint64_t pk = hexrow::relative_bytes(elem_pos(cm.e, cm.la), cm.la);
  double v[8];
  const double rr = op.eval(r, v);
#pragma unroll
  for (int m = 0; m < 8; ++m) unsafeAtomicAdd(rowp + hexrow::pos(pk, m), v[m]);
  unsafeAtomicAdd(rhs + row, rr * rhs_scale);
}

// Owner-computes row tile.  A wave owns kRowsPerWave consecutive rows and the LDS
// copy of their CSR segment; lane (s, j) takes the s-th, (s + kSlots)-th, ...
// incident element of row j.  Consecutive lanes are consecutive rows, so that a
// load of one relative corner covers runs of neighbouring nodes.  Row sums are LDS
// atomics of one wave in program order (and a fixed cross-lane tree for the
// diagonal and the rhs, which all lanes of a row share), so results do not depend
// on timing; the segment leaves in one coalesced pass.  No block barrier: waves
// are independent.  Bound by the vector cache's address rate (68 % busy) and, at two
// to three waves per SIMD, latency.  128^3 continuity with mdot: 0.75 ms (1.26 ms
// for one thread per row over eight compile-time local nodes); the segregated
// momentum with mass 1.40 ms (3.42 ms).
constexpr int kSlots = 4;  // lanes of a row
constexpr int kRowsPerWave = 64 / kSlots;
constexpr int kRowWaves = 4;  // waves to a block
constexpr int kRowThreads = 64 * kRowWaves;
constexpr int kRowsPerBlock = kRowsPerWave * kRowWaves;
constexpr size_t kMaxLds = 160 * 1024;  // LDS of one gfx950 CU, the most one block can hold

// sum over the lanes of a row, in every lane
__device__ __forceinline__ double row_sum(double v) {
#pragma unroll
  for (int s = kRowsPerWave; s < 64; s <<= 1) v += __shfl_xor(v, s);
  return v;
}

// orders a wave's LDS accesses around a change of the lanes' roles
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the wave's rows, and this lane's place in them
struct WaveRows {
  int64_t r0, r1, r;  // rows [r0, r1) of the wave, row of the lane (may be >= r1)
  int lane, slot;
  int32_t q, q1;      // next and last incidence entry of the lane
};
__device__ __forceinline__ WaveRows wave_rows(const int32_t* __restrict__ row_node,
                                              const int32_t* __restrict__ inc_ptr, int64_t nrows) {
  WaveRows w;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  w.lane = threadIdx.x & 63;
  w.slot = w.lane / kRowsPerWave;
  w.r0 = ((int64_t)blockIdx.x * (blockDim.x >> 6) + wave) * kRowsPerWave;
  w.r1 = min(w.r0 + (int64_t)kRowsPerWave, nrows);
  w.r = w.r0 + w.lane % kRowsPerWave;
  w.q = w.q1 = 0;
  if (w.r < w.r1) {
    const int32_t a = row_node ? row_node[w.r] : (int32_t)w.r;
    w.q = inc_ptr[a] + w.slot;
    w.q1 = inc_ptr[a + 1];
  }
  return w;
}

template <class Op>
__global__ __launch_bounds__(kRowThreads, 3) void k_scalar_rows(Op op, const int32_t* __restrict__ conn,
                                                             const int32_t* __restrict__ row_node,
                                                             const int32_t* __restrict__ inc_ptr,
                                                             const int32_t* __restrict__ inc_elem,
                                                             const int32_t* __restrict__ nrp,
                                                             ElemPos elem_pos, int64_t nrows,
                                                             int row_len, double rhs_scale, double* __restrict__ vals,
                                                             double* __restrict__ rhs, int accumulate) {
  extern __shared__ double seg_all[];
  double* seg = seg_all + (size_t)(threadIdx.x >> 6) * kRowsPerWave * row_len;
  const WaveRows w = wave_rows(row_node, inc_ptr, nrows);
  if (w.r0 >= nrows) return;
  const int32_t s0 = nrp[w.r0];
  const int nseg = nrp[w.r1] - s0;
  for (int i = w.lane; i < nseg; i += 64) seg[i] = 0.0;
  wave_sync();
  double rr = 0.0, diag = 0.0;
  double* myrow = seg;
  int at = 0;
  if (w.q < w.q1) {
    myrow = seg + (nrp[w.r] - s0);
    for (int32_t q = w.q; q < w.q1; q += kSlots) {
      const int32_t t = inc_elem[q];
      RowElem el = row_elem(conn, t >> 3, t & 7);
      const uint64_t pk = hexrow::relative_bytes(elem_pos(t >> 3, t & 7), t & 7);
      double v[8];
      rr += op.eval(el, v);
      diag += v[0];
      at = hexrow::pos(pk, 0);
#pragma unroll
      for (int m = 1; m < 8; ++m) unsafeAtomicAdd(myrow + hexrow::pos(pk, m), v[m]);
    }
  }
  rr = row_sum(rr);
  diag = row_sum(diag);
  if (w.slot == 0 && w.q < w.q1) unsafeAtomicAdd(myrow + at, diag);
  wave_sync();
  double* out = vals + s0;
  if (accumulate) {
    for (int i = w.lane; i < nseg; i += 64) out[i] += seg[i];
    if (w.slot == 0 && w.r < w.r1) rhs[w.r] += rr * rhs_scale;
  } else {
    for (int i = w.lane; i < nseg; i += 64) __builtin_nontemporal_store(seg[i], out + i);
    if (w.slot == 0 && w.r < w.r1) rhs[w.r] = rr * rhs_scale;
  }
}

// ---------------------------------------------------------------- mass (time derivative)
// MomentumMassElemKernel (src/kernel/MomentumMassElemKernel.C:95-170) and
// ContinuityMassElemKernel (src/kernel/ContinuityMassElemKernel.C:84-118).  The
// scv ip of an element belongs to one node (HexSCV::ipNodeMap_), so a node's
// rows receive exactly the contributions of the scvs at that node.
struct MassArgs {
  Field4<> s[3];         // velocity (momentum only) and density of the states Nm1, N, Np1
  Field4<> gjp;          // projected pressure gradient (momentum only)
  double dt, g1, g2, g3;
  int balanced;          // densFac = rhoNp1 (balanced force) or 1
};

// MomentumMassElemKernel at the row's scv: rh += its rhs; the return value times
// scv_shape(m) is the diagonal lhs entry of corner m's block.
template <bool LUMPED, bool PACK>
__device__ __forceinline__ double momentum_mass_row(const MassArgs& A, const uint32_t (&nd)[8],
                                                    const double (&x)[3][8], double h, double (&rh)[3]) {
  double rs[3], acc[3] = {0.0, 0.0, 0.0}, f[8], f3[3][8];
  const double g[3] = {A.g3, A.g2, A.g1};
  double vol = hexrow::scv_volume(x, h);
  pin(vol);
#pragma unroll
  for (int st = 0; st < 3; ++st) {
    load4<PACK, true>(A.s[st], nd, f3, f);
    rs[st] = hexrow::at_scv<LUMPED>(f);
#pragma unroll
    for (int i = 0; i < 3; ++i) acc[i] += g[st] * rs[st] * hexrow::at_scv<LUMPED>(f3[i]);
    pin(acc);
    asm volatile("" ::: "memory");
  }
  load3<PACK>(A.gjp, nd, f3);
  const double vdt = vol / A.dt;
  const double vd = A.balanced ? vol * rs[2] : vol;
#pragma unroll
  for (int i = 0; i < 3; ++i) rh[i] -= acc[i] * vdt + hexrow::at_scv<LUMPED>(f3[i]) * vd;
  pin(rh);
  return A.g1 * rs[2] * vdt;
}

// ---------------------------------------------------------------- momentum
// MomentumAdvDiffElemKernel (src/kernel/MomentumAdvDiffElemKernel.C:72-186), the
// row block of one node.  Rows (la, i), columns (c, j); per scs, with A outward
// and mdot the outflow:
//   lhs += delta_ij (N_adv(c) mdot - mu_ip dN_c/dx . A) - mu_ip dN_c/dx_i A_j
//   rhs -= mdot u_ip,i + 2/3 mu_ip divU A_i incl
//          - mu_ip sum_c dN_c/dx_i (A . u_c) - mu_ip sum_c (dN_c/dx . A) u_c,i
// The advected u_ip uses the lhs's N_adv, so apart from the divU term the rhs is
// -sum_c lhs(c) u_c.  mdot3: outflow through the scs of directions 0, 1, 2.
// emit(m, blk) receives the 3x3 block blk[i][j] of relative corner m.
struct MomentumFields {
  Field4<> x;          // coordinates and viscosity
  Field4<> u;          // velocity (PACK: with the density of the mass kernel's Np1 state, if it is the same field)
  const double* mdot;  // [E][12]
  double incl_divu;
};

// per direction: cofactor columns / det (along D, D+1, D+2) and mu_ip A
template <typename R>
struct MomentumGeo {
  R b[3][3][3], mA[3][3];
};
template <bool SHIFT, typename R>
__device__ __forceinline__ void momentum_geometry(const double (&x)[3][8], const R (&mn)[8], double h, RowElem& el,
                                                  MomentumGeo<R>& G) {
  R muip[3];
  static_for<3>([&](auto dd) { muip[decltype(dd)::value] = hexrow::at_scs<decltype(dd)::value, false>(mn); });
  hexrow::Edges E;
  hexrow::edges(x, E);
  static_for<3>([&](auto dd) {
    constexpr int D = decltype(dd)::value;
    double A[3];
    hexrow::Cof K;
    hexrow::area_cofactors<D, SHIFT>(E, h, A, K);
    const double f0 = K.inv * hexrow::Scale<SHIFT>::c0, f1 = K.inv * hexrow::Scale<SHIFT>::c1;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      G.mA[D][i] = muip[D] * R(A[i]);
      G.b[D][0][i] = R(K.c[0][i] * f0);
      G.b[D][1][i] = R(K.c[1][i] * f1);
      G.b[D][2][i] = R(K.c[2][i] * f1);
    }
    pin(G.b[D]);
    pin(G.mA[D]);
    pin(E);
  });
  pin(el);
}

// outflow through the scs of directions 0, 1, 2 of local node la
template <typename R>
__device__ __forceinline__ void load_mdot3(const double* __restrict__ mdot, const RowElem& r, R (&m3)[3]) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double v = mdot[12 * r.e + hexrow::scs_of(r.la, d)];
    m3[d] = R(hexrow::scs_is_left(r.la, d) ? v : -v);
  }
}

template <bool SKEW, bool SHIFT, bool PACK, typename R, class Emit>
__device__ __forceinline__ void momentum_row(const MomentumFields& F, RowElem& el, const double (&x)[3][8], const R (&mn)[8],
                                             double h, double (&rhs)[3], Emit&& emit) {
  MomentumGeo<R> G;
  momentum_geometry<SHIFT>(x, mn, h, el, G);
  R u[3][8], mdot3[3], rr[3] = {R(0), R(0), R(0)};
  load_mdot3(F.mdot, el, mdot3);
  load3<PACK>(F.u, el.nd, u);
  if (F.incl_divu != 0.0) {
    static_for<3>([&](auto dd) {
      constexpr int D = decltype(dd)::value;
      R divu = R(0);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        R du[3];
        hexrow::param_grad<D, SHIFT>(u[i], du);
        divu += G.b[D][0][i] * du[0] + G.b[D][1][i] * du[1] + G.b[D][2][i] * du[2];
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) rr[i] -= R(2.0 / 3.0) * divu * G.mA[D][i] * R(F.incl_divu);
    });
  }
  static_for<8>([&](auto mm) {
    constexpr int m = decltype(mm)::value;
    R T[3][3], a = R(0);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) T[i][j] = R(0);
    static_for<3>([&](auto dd) {
      constexpr int D = decltype(dd)::value;
      constexpr double s0 = hexrow::scs_slope<D, SHIFT>(m, 0), s1 = hexrow::scs_slope<D, SHIFT>(m, 1),
                       s2 = hexrow::scs_slope<D, SHIFT>(m, 2), N = hexrow::scs_shape<D, SKEW>(m);
      if constexpr (s0 != 0.0 || s1 != 0.0 || s2 != 0.0) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          R dn = R(0);
          if constexpr (s0 != 0.0) dn += R(s0) * G.b[D][0][i];
          if constexpr (s1 != 0.0) dn += R(s1) * G.b[D][1][i];
          if constexpr (s2 != 0.0) dn += R(s2) * G.b[D][2][i];
#pragma unroll
          for (int j = 0; j < 3; ++j) T[i][j] += dn * G.mA[D][j];
        }
      }
      if constexpr (N != 0.0) a += R(N) * mdot3[D];
    });
    a -= T[0][0] + T[1][1] + T[2][2];
    R blk[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        blk[i][j] = i == j ? a - T[i][j] : -T[i][j];
        rr[i] -= blk[i][j] * u[j][m];
      }
    }
    emit(m, blk);
    pin(rr);
    pin(G.mA);
  });
#pragma unroll
  for (int i = 0; i < 3; ++i) rhs[i] += (double)rr[i];
}

// The segregated form: the transpose-gradient term -mu_ip dN_c/dx_i A_j stays on
// the rhs only, so the three components share the scalar entries am[m].
template <bool SKEW, bool SHIFT, bool PACK, typename R>
__device__ __forceinline__ void momentum_row_seg(const MomentumFields& F, RowElem& el, const double (&x)[3][8],
                                                 const R (&mn)[8], double h, R (&am)[8], double (&rhs)[3]) {
  MomentumGeo<R> G;
  momentum_geometry<SHIFT>(x, mn, h, el, G);
  R u[3][8], mdot3[3], rr[3] = {R(0), R(0), R(0)};
  load_mdot3(F.mdot, el, mdot3);
  load3<PACK>(F.u, el.nd, u);
#pragma unroll
  for (int m = 0; m < 8; ++m) am[m] = R(0);
  static_for<3>([&](auto dd) {
    constexpr int D = decltype(dd)::value;
    R g[3], divu = R(0), du[3][3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g[k] = G.b[D][k][0] * G.mA[D][0] + G.b[D][k][1] * G.mA[D][1] + G.b[D][k][2] * G.mA[D][2];
    hexrow::slope<D, SHIFT>(g, [&](int m, R t) { am[m] -= t; });
    static_for<8>([&](auto mm) {
      constexpr int m = decltype(mm)::value;
      constexpr double N = hexrow::scs_shape<D, SKEW>(m);
      if constexpr (N != 0.0) am[m] += R(N) * mdot3[D];
    });
    // mu sum_c dN_c/dx_i (A . u_c) = sum_k b_k,i (du/dt_k . mu A)
#pragma unroll
    for (int j = 0; j < 3; ++j) hexrow::param_grad<D, SHIFT>(u[j], du[j]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const R w = du[0][k] * G.mA[D][0] + du[1][k] * G.mA[D][1] + du[2][k] * G.mA[D][2];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        rr[i] += G.b[D][k][i] * w;
        divu += G.b[D][k][i] * du[i][k];
      }
    }
    if (F.incl_divu != 0.0) {
#pragma unroll
      for (int i = 0; i < 3; ++i) rr[i] -= R(2.0 / 3.0) * divu * G.mA[D][i] * R(F.incl_divu);
    }
    pin(am);
    pin(rr);
  });
#pragma unroll
  for (int m = 0; m < 8; ++m)
#pragma unroll
    for (int i = 0; i < 3; ++i) rr[i] -= am[m] * u[i][m];
#pragma unroll
  for (int i = 0; i < 3; ++i) rhs[i] += (double)rr[i];
}

// Momentum (numDof 3) row tile: a block owns kMomRows consecutive nodes and the LDS
// copy of their three rows each (rows 3a..3a+2 are contiguous in the CSR; 62 KB for
// 27-column rows, two blocks to a CU), accumulated with LDS atomics.  Eight threads
// to a node; the two of one wave take the s-th and the (7-s)-th incident element,
// opposite corners on a lattice, which share no column but the node's own.  ADV:
// the advection-diffusion kernel; MASS (0 none, 1 consistent, 2 lumped): the
// momentum mass kernel of the same element and scv, in the same pass as one
// element algorithm runs its kernel list.  96^3 with mass: 0.94 ms (2.75 ms for 64
// nodes to a block, one block to a CU, and eight compile-time local nodes).
constexpr int kMomRows = 32;
constexpr int kMomThreads = 8 * kMomRows;
template <bool ADV, bool SKEW, bool SHIFT, bool PACK, typename R, int MASS>
__global__ __launch_bounds__(kMomThreads) void k_momentum_rows(
    MomentumFields F, MassArgs MA, const int32_t* __restrict__ conn,
    const int32_t* __restrict__ row_node, const int32_t* __restrict__ inc_ptr, const int32_t* __restrict__ inc_elem,
    const int32_t* __restrict__ nrp, ElemPos elem_pos, int64_t nnodes,
    double* __restrict__ vals, double* __restrict__ rhs, int accumulate) {
  extern __shared__ double seg[];
  const int64_t a0 = (int64_t)blockIdx.x * kMomRows;
  const int64_t a1 = min(a0 + (int64_t)kMomRows, nnodes);
  const int64_t s0 = 9 * (int64_t)nrp[a0];
  const int nseg = (int)(9 * (int64_t)nrp[a1] - s0);
  double* rseg = seg + nseg;
  for (int i = threadIdx.x; i < nseg + 3 * kMomRows; i += kMomThreads) seg[i] = 0.0;
  __syncthreads();
  const int j = threadIdx.x % kMomRows, wave = threadIdx.x >> 6;
  const int slot = (threadIdx.x & 32) ? 7 - wave : wave;
  const int64_t r = a0 + j;
  if (r < a1) {
    const int32_t a = row_node ? row_node[r] : (int32_t)r;
    const int32_t L3 = 3 * (nrp[r + 1] - nrp[r]), q1 = inc_ptr[a + 1];
    double* myrow = seg + (9 * (int64_t)nrp[r] - s0);
    double rh[3] = {0.0, 0.0, 0.0};
    for (int32_t q = inc_ptr[a] + slot; q < q1; q += 8) {
      const int32_t t = inc_elem[q];
      RowElem el = row_elem(conn, t >> 3, t & 7);
      const uint64_t pk = hexrow::relative_bytes(elem_pos(t >> 3, t & 7), t & 7);
      const double h = hexrow::handed(t & 7);
      double x[3][8], lf = 0.0;
      R mn[8];
      load4<PACK, ADV>(F.x, el.nd, x, mn);
      if constexpr (MASS != 0) lf = momentum_mass_row<MASS == 2, PACK>(MA, el.nd, x, h, rh);
      if constexpr (ADV) {
        momentum_row<SKEW, SHIFT, PACK, R>(F, el, x, mn, h, rh, [&](int m, const R (&blk)[3][3]) {
          double* at = myrow + 3 * hexrow::pos(pk, m);
#pragma unroll
          for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int jj = 0; jj < 3; ++jj) {
              double z = (double)blk[i][jj];
              if constexpr (MASS != 0)
                if (i == jj) z += hexrow::scv_shape<MASS == 2>(m) * lf;
              unsafeAtomicAdd(at + i * L3 + jj, z);
            }
        });
      } else {
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          if (MASS == 2 && m != 0) continue;
          double* at = myrow + 3 * hexrow::pos(pk, m);
#pragma unroll
          for (int i = 0; i < 3; ++i) unsafeAtomicAdd(at + i * L3 + i, hexrow::scv_shape<MASS == 2>(m) * lf);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) unsafeAtomicAdd(rseg + 3 * j + i, rh[i]);
  }
  __syncthreads();
  const int nr = (int)(3 * (a1 - a0));
  double* out = vals + s0;
  if (accumulate) {
    for (int i = threadIdx.x; i < nseg; i += kMomThreads) out[i] += seg[i];
    for (int i = threadIdx.x; i < nr; i += kMomThreads) rhs[3 * a0 + i] += rseg[i];
  } else {
    for (int i = threadIdx.x; i < nseg; i += kMomThreads) __builtin_nontemporal_store(seg[i], out + i);
    for (int i = threadIdx.x; i < nr; i += kMomThreads) rhs[3 * a0 + i] = rseg[i];
  }
}

template <bool SKEW, bool SHIFT, typename R>
__global__ __launch_bounds__(kChunk) void k_momentum_atomic(
    const int32_t* __restrict__ conn, const double* __restrict__ coords, const double* __restrict__ u,
    const double* __restrict__ mu, const double* __restrict__ mdot, double incl_divu,
    const int32_t* __restrict__ lid, const int32_t* __restrict__ nrp, ElemPos elem_pos,
    int64_t nelem, double* __restrict__ vals, double* __restrict__ rhs) {
  const ChunkMap cm = chunk_map<8>(nelem);
  if (!cm.valid) return;
  RowElem el = row_elem(conn, cm.e, cm.la);
  const int32_t nr = lid[el.nd[0]], nb = nrp[nr];
  const int32_t L3 = 3 * (nrp[nr + 1] - nb);
  double* rowp = vals + 9 * (int64_t)nb;
  const uint64_t pk = hexrow::relative_bytes(elem_pos(cm.e, cm.la), cm.la);
  const MomentumFields F{{{}, coords, mu}, {{}, u, nullptr}, mdot, incl_divu};
  double x[3][8], rh[3] = {0.0, 0.0, 0.0};
  R mn[8];
  load4<false, true>(F.x, el.nd, x, mn);
  momentum_row<SKEW, SHIFT, false, R>(F, el, x, mn, hexrow::handed(cm.la), rh,
                               [&](int m, const R (&blk)[3][3]) {
                                 double* at = rowp + 3 * hexrow::pos(pk, m);
#pragma unroll
                                 for (int i = 0; i < 3; ++i)
#pragma unroll
                                   for (int j = 0; j < 3; ++j) unsafeAtomicAdd(at + i * L3 + j, (double)blk[i][j]);
                               });
#pragma unroll
  for (int i = 0; i < 3; ++i) unsafeAtomicAdd(rhs + 3 * (int64_t)nr + i, rh[i]);
}

// ---------------------------------------------------------------- mdot
// mdot, element-centric: one thread per element loads its connectivity,
// coordinates and nodal fields once (two dependent round trips) and evaluates
// all 12 scs from registers (a thread per (element, scs) gathers the same
// element data twelve times and measured 2.4x slower at 128^3).  The 12 values
// leave as six 16-byte stores (mdot must be 16-byte aligned), each as soon as its
// pair is done: that and the pinned scs keep the kernel at 256 registers, two waves
// to a SIMD (128^3: 230 us; 320 us at one wave).
template <bool SHIFT_MDOT, bool SHIFT_POISSON, typename R>
__global__ __launch_bounds__(256, 2) void k_mdot_elem(const int32_t* __restrict__ conn,
                                                   const double* __restrict__ coords, const double* __restrict__ rho,
                                                   const double* __restrict__ p, const double* __restrict__ u,
                                                   const double* __restrict__ gp, double tau, int64_t nelem,
                                                   double* __restrict__ mdot) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nelem) return;
  const RowElem el = row_elem(conn, e, 0);
  double x[3][8];
  R pn[8], W[3][8];
  load4<false, true>(Field4<>{{}, coords, p}, el.nd, x, pn);
  {
    R rn[8], un[3][8], gn[3][8];
    load4<false, true>(Field4<>{{}, u, rho}, el.nd, un, rn);
    load3<false>(Field4<>{{}, gp, nullptr}, el.nd, gn);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int m = 0; m < 8; ++m) W[i][m] = rn[m] * un[i][m] + R(tau) * gn[i][m];
  }
  hexrow::Edges E;
  hexrow::edges(x, E);
  double2* o = reinterpret_cast<double2*>(mdot + 12 * e);
  double even = 0.0;
  static_for<12>([&](auto ii) {
    // direction and quadrant of the scs; the area vector points to the far side
    // along D, which is its right node's except for scs 2 and 6
    constexpr int IP = decltype(ii)::value;
    constexpr int D = IP >= 8 ? 2 : (IP & 1), c = hex8::scs_left(IP);
    constexpr int bits = hexrow::hex_of(c);
    constexpr int QE = (bits >> (D + 1) % 3) & 1, QF = (bits >> (D + 2) % 3) & 1;
    constexpr double sign = ((bits >> D) & 1) ? -1.0 : 1.0;
    double A[3];
    hexrow::Cof K;
    hexrow::area_cofactors<D, SHIFT_POISSON, QE, QF>(E, sign, A, K);
    R g[3], ps[3];
    hexrow::metric<SHIFT_POISSON>(K, A, g);
    hexrow::param_grad<D, SHIFT_POISSON, QE, QF>(pn, ps);
    R f = -R(tau) * (ps[0] * g[0] + ps[1] * g[1] + ps[2] * g[2]);
#pragma unroll
    for (int i = 0; i < 3; ++i) f += hexrow::at_scs<D, SHIFT_MDOT, QE, QF>(W[i]) * R(A[i]);
    if constexpr (IP & 1) o[IP / 2] = make_double2(even, (double)f);
    else even = (double)f;
    pin(even);
    pin(E);
  });
}

// ---------------------------------------------------------------- generic sumInto
// Batched sumInto of caller-provided dense element matrices.
__global__ void k_sum_into_batch(const int32_t* __restrict__ conn, const double* __restrict__ lhs,
                                 const double* __restrict__ rhs_e, const int32_t* __restrict__ lid,
                                 const int32_t* __restrict__ nrp, ElemPos elem_pos,
                                 int64_t nelem, int nd, double* __restrict__ vals, double* __restrict__ rhs) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // (element, row node, dof)
  if (t >= nelem * 8 * nd) return;
  const int64_t e = t / (8 * nd);
  const int rem = (int)(t - e * 8 * nd);
  const int a = rem / nd, d = rem % nd;
  const int R = 8 * nd;
  const int32_t nr = lid[conn[8 * e + a]];
  const int32_t nb = nrp[nr];
  const int32_t L = nrp[nr + 1] - nb;
  const uint64_t pk = elem_pos(e, a);
  const double* lrow = lhs + (e * R + (int64_t)(a * nd + d)) * R;
  double* rowp = vals + (int64_t)nd * nd * nb + (int64_t)d * nd * L;
  for (int c = 0; c < 8; ++c) {
    const int p = (int)((pk >> (8 * c)) & 0xff);
    for (int j = 0; j < nd; ++j) unsafeAtomicAdd(rowp + nd * p + j, lrow[c * nd + j]);
  }
  unsafeAtomicAdd(rhs + (int64_t)nd * nr + d, rhs_e[e * R + a * nd + d]);
}

// ---------------------------------------------------------------- Dirichlet / resetRows
__global__ void k_dirichlet(const int32_t* __restrict__ nodes, int64_t nbc, int64_t nnodes, int nd, int begin,
                            int end, const int32_t* __restrict__ lid, const int32_t* __restrict__ rp,
                            const int32_t* __restrict__ ci, const double* __restrict__ sol,
                            const double* __restrict__ bcv, double* __restrict__ vals, double* __restrict__ rhs,
                            int reset_mode, double diag_value, double rhs_residual, int* __restrict__ bad) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int nsub = end - begin;
  if (t >= nbc * nsub) return;
  const int64_t k = t / nsub;
  const int d = begin + (int)(t % nsub);
  const int32_t node = nodes[k];
  if (node < 0 || node >= nnodes) {  // caller-provided list: never index outside the mesh
    atomicOr(bad, 1);
    return;
  }
  const int64_t row = (int64_t)nd * lid[node] + d;
  const double dv = reset_mode ? diag_value : 1.0;
  for (int32_t q = rp[row]; q < rp[row + 1]; ++q) vals[q] = (ci[q] == row) ? dv : 0.0;
  rhs[row] = reset_mode ? rhs_residual : bcv[(int64_t)nd * node + d] - sol[(int64_t)nd * node + d];
}

inline size_t lds_rows(const nalu_linsys* ls) {
  return (size_t)kRowsPerBlock * ls->max_node_row_len * sizeof(double);
}

// From this many nodes on, a row pass copies its fields first.  A pass in FP64, us,
// gathering from the fields / with the copy: continuity 32 768 nodes 37 / 38, 50 653
// nodes 55 / 45, 117 649 nodes 95 / 62, 128^3 1140 / 750; 3-rhs momentum with mass
// 50 653 nodes 68 / 69, 117 649 nodes 105 / 100, 912 673 nodes 624 / 584; coupled
// momentum with mass 68 921 nodes 95 / 96, 912 673 nodes 971 / 917; diffusion 50 653
// nodes 34 / 40, 274 625 nodes 77 / 79, 912 673 nodes 197 / 193.  The line is
// continuity's, which gains most; the others lose the copy's launch, up to 6 us, up to
// some 100 000 nodes (diffusion 500 000).  Below it no pass gains and the handle is
// spared the workspace.  Past 2^28 nodes the 32-bit offsets end.
// The workspace has its full size (six fields) from the first pass on and never moves,
// as a captured graph may hold its address; where it cannot be had (a first pass under
// capture, or no memory left) the passes gather from the fields themselves.
constexpr int64_t kPackNodes = 1 << 15;
constexpr int kPackFields = 6;
bool use_pack(nalu_linsys* ls) {
  const int64_t N = ls->num_nodes;
  if (N < kPackNodes || N >= ((int64_t)1 << 28)) return false;
  const size_t bytes = (size_t)N * kPackFields * 2 * sizeof(Half<double>);
  if (ls->pack_ws.n >= bytes) return true;
  if (ls->pack_denied) return false;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  NALU_HIP_CHECK(hipStreamIsCapturing(ls->stream, &cap));
  if (cap != hipStreamCaptureStatusNone) return false;
  void* q = nullptr;
  if (hipMalloc(&q, bytes) != hipSuccess) {
    (void)hipGetLastError();
    ls->pack_denied = true;
    return false;
  }
  ls->pack_ws.p = static_cast<unsigned char*>(q);
  ls->pack_ws.n = bytes;
  return true;
}

// Copies the fields f[0..n) to 16-byte halves (on ls->stream) and points their h at them.
void pack_fields(nalu_linsys* ls, Field4<>* const* f, int n) {
  const int64_t N = ls->num_nodes;
  auto* ws = reinterpret_cast<Half<double>*>(ls->pack_ws.p);
  PackList L{};
  for (L.n = 0; L.n < n; ++L.n) {
    L.vec[L.n] = f[L.n]->vec;
    L.scal[L.n] = f[L.n]->scal;
    f[L.n]->h[0] = ws + 2 * L.n * N;
    f[L.n]->h[1] = ws + (2 * L.n + 1) * N;
  }
  hipLaunchKernelGGL(k_pack, dim3(blocks_for(N, 256)), dim3(256), 0, ls->stream, L, N, ws);
}

template <class Op>
void launch_scalar_rows(nalu_linsys* ls, const nalu_mesh* m, const Op& op) {
  hipStream_t s = ls->stream;
  build_node_incidence(const_cast<nalu_mesh*>(m), s);
  const int accumulate = ls->values_pending_zero ? 0 : 1;
  NALU_REQUIRE(ls->values_pending_zero == ls->rhs_pending_zero, NALU_ERR_STATE,
               "row-tile assembly: values/rhs zero state diverged");
  const size_t lds = lds_rows(ls);
  set_lds_limit((const void*)k_scalar_rows<Op>, lds);
  hipLaunchKernelGGL((k_scalar_rows<Op>), dim3(blocks_for(ls->nrows, kRowsPerBlock)), dim3(kRowThreads), lds, s, op,
                     m->conn.p, (const int32_t*)ls->row_node.p, m->inc_ptr.p, m->inc_elem.p, ls->nrp.p,
                     elem_pos_of(ls), ls->nrows, ls->max_node_row_len, op.rhs_scale(), ls->values.p, ls->rhs.p,
                     accumulate);
  ls->values_pending_zero = ls->rhs_pending_zero = false;
  NALU_HIP_CHECK(hipGetLastError());
}

template <class Op>
void launch_scalar_atomic(nalu_linsys* ls, const nalu_mesh* m, const Op& op) {
  const int64_t E = m->num_elems;
  materialize_pending_zero(ls);
  hipLaunchKernelGGL((k_scalar_atomic<Op>), dim3(chunk_blocks<8>(E)), dim3(kChunk), 0, ls->stream, op, m->conn.p,
                     ls->node_lid.p, ls->nrp.p, elem_pos_of(ls), E, op.rhs_scale(), ls->values.p, ls->rhs.p);
  NALU_HIP_CHECK(hipGetLastError());
}

// Modes 0 ("gather") and 2 ("tile") run the row tile; mode 1 the atomic scatter.
template <bool SHIFT, typename R>
void scalar_diff_pass(nalu_linsys* ls, const nalu_mesh* m, const double* q, const double* k, int mode) {
  Field4<> xk{{}, m->coords.p, k};
  if (mode == 1) {
    launch_scalar_atomic(ls, m, ScalarDiffOp<SHIFT, false, R>{xk, q});
  } else if (use_pack(ls)) {
    Field4<>* const f[] = {&xk};
    pack_fields(ls, f, 1);
    launch_scalar_rows(ls, m, ScalarDiffOp<SHIFT, true, R>{xk, q});
  } else {
    launch_scalar_rows(ls, m, ScalarDiffOp<SHIFT, false, R>{xk, q});
  }
}

template <bool SM, bool SP, bool RED, bool MDOT, typename R>
void continuity_pass(nalu_linsys* ls, const nalu_mesh* m, const double* rho, const double* p, const double* u,
                     const double* gp, double tau, int mode, double* mdot) {
  const Field4<> xp{{}, m->coords.p, p}, ur{{}, u, rho};
  if (mode == 1) {
    if constexpr (!MDOT)
      launch_scalar_atomic(ls, m, ContinuityOp<SM, SP, RED, false, false, R>{xp, {}, ur, gp, tau, nullptr});
  } else if (use_pack(ls)) {
    const int64_t N = ls->num_nodes;
    constexpr int nw = sizeof(R) == 8 ? 2 : 1;
    auto* xs = reinterpret_cast<Half<double>*>(ls->pack_ws.p);
    auto* W = reinterpret_cast<Half<R>*>(xs + 2 * N);
    hipLaunchKernelGGL(k_pack_flux<R>, dim3(blocks_for(N, 256)), dim3(256), 0, ls->stream, m->coords.p, p, rho, u, gp,
                       tau, N, xs, W);
    const Field4<> xh{{xs, xs + N}, nullptr, nullptr};
    const Field4<R> Wh{{W, nw == 2 ? W + N : nullptr}, nullptr, nullptr};
    launch_scalar_rows(ls, m, ContinuityOp<SM, SP, RED, MDOT, true, R>{xh, Wh, {}, nullptr, tau, mdot});
  } else {
    launch_scalar_rows(ls, m, ContinuityOp<SM, SP, RED, MDOT, false, R>{xp, {}, ur, gp, tau, mdot});
  }
}

// Systems created for the mixed-precision path assemble with FP32 arithmetic.
bool fp32_assembly(const nalu_linsys* ls) { return ls->cfg.precision == NALU_PRECISION_MIXED; }

template <typename R>
void launch_mdot(const nalu_mesh* m, const double* rho, const double* p, const double* u, const double* gp,
                 double tau, int shift_mdot, int shift_poisson, double* mdot, hipStream_t s) {
  const int64_t E = m->num_elems;
  NALU_REQUIRE(((uintptr_t)mdot & 15) == 0, NALU_ERR_ARG, "compute_mdot: mdot must be 16-byte aligned");
  const dim3 g(blocks_for(E, 256)), b(256);
  if (shift_mdot && shift_poisson)
    hipLaunchKernelGGL((k_mdot_elem<true, true, R>), g, b, 0, s, m->conn.p, m->coords.p, rho, p, u, gp, tau, E, mdot);
  else if (shift_mdot)
    hipLaunchKernelGGL((k_mdot_elem<true, false, R>), g, b, 0, s, m->conn.p, m->coords.p, rho, p, u, gp, tau, E, mdot);
  else if (shift_poisson)
    hipLaunchKernelGGL((k_mdot_elem<false, true, R>), g, b, 0, s, m->conn.p, m->coords.p, rho, p, u, gp, tau, E, mdot);
  else
    hipLaunchKernelGGL((k_mdot_elem<false, false, R>), g, b, 0, s, m->conn.p, m->coords.p, rho, p, u, gp, tau, E, mdot);
  NALU_HIP_CHECK(hipGetLastError());
}

void check_flag(DevBuf<int>& flag, hipStream_t s, const char* msg) {
  int h = 0;
  NALU_HIP_CHECK(hipMemcpyAsync(&h, flag.p, sizeof(int), hipMemcpyDeviceToHost, s));
  NALU_HIP_CHECK(hipStreamSynchronize(s));
  NALU_REQUIRE(h == 0, NALU_ERR_ARG, msg);
}

// ---------------------------------------------------------------- kernel-input producers
// Dual nodal volume (ComputeGeometryInteriorAlgorithm, src/ComputeGeometryInteriorAlgorithm.C:77-120)
// and the interior Green-Gauss nodal gradient (AssembleNodalGradElemAlgorithm,
// src/AssembleNodalGradElemAlgorithm.C:85-140), owner-computes: the node's scv and
// its three adjacent scs are all that touch it.  kSlots lanes per node take its
// incident elements (as in k_scalar_rows), every result is written once.
template <int NC, class Eval, class Store>
__device__ __forceinline__ void node_sums(const int32_t* __restrict__ conn, const int32_t* __restrict__ inc_ptr,
                                          const int32_t* __restrict__ inc_elem, int64_t nnodes, Eval&& eval,
                                          Store&& store) {
  const WaveRows w = wave_rows(nullptr, inc_ptr, nnodes);
  double v[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) v[i] = 0.0;
  for (int32_t q = w.q; q < w.q1; q += kSlots) {
    const int32_t t = inc_elem[q];
    eval(row_elem(conn, t >> 3, t & 7), v);
  }
#pragma unroll
  for (int i = 0; i < NC; ++i) v[i] = row_sum(v[i]);
  if (w.slot == 0 && w.r < w.r1) store(w.r, v);
}

__global__ __launch_bounds__(kRowThreads) void k_dual_volume(const int32_t* __restrict__ conn,
                                                              const double* __restrict__ coords,
                                                              const int32_t* __restrict__ inc_ptr,
                                                              const int32_t* __restrict__ inc_elem, int64_t nnodes,
                                                              double* __restrict__ vol) {
  node_sums<1>(
      conn, inc_ptr, inc_elem, nnodes,
      [&](const RowElem& el, double (&v)[1]) {
        double x[3][8];
        load3<false>(Field4<>{{}, coords, nullptr}, el.nd, x);
        v[0] += hexrow::scv_volume(x, hexrow::handed(el.la));
      },
      [&](int64_t a, const double (&v)[1]) { vol[a] = v[0]; });
}

template <bool SHIFT>
__global__ __launch_bounds__(kRowThreads) void k_nodal_grad(const int32_t* __restrict__ conn,
                                                             const double* __restrict__ coords,
                                                             const double* __restrict__ qf,
                                                             const double* __restrict__ vol,
                                                             const int32_t* __restrict__ inc_ptr,
                                                             const int32_t* __restrict__ inc_elem, int64_t nnodes,
                                                             double* __restrict__ dqdx) {
  node_sums<3>(
      conn, inc_ptr, inc_elem, nnodes,
      [&](const RowElem& el, double (&v)[3]) {
        double x[3][8], q[8];
        load4<false, true>(Field4<>{{}, coords, qf}, el.nd, x, q);
        hexrow::Edges E;
        hexrow::edges(x, E);
        const double h = hexrow::handed(el.la);
        static_for<3>([&](auto dd) {
          constexpr int D = decltype(dd)::value;
          double A[3];
          hexrow::area<D>(E, h, A);
          const double qi = hexrow::at_scs<D, SHIFT>(q);
#pragma unroll
          for (int i = 0; i < 3; ++i) v[i] += qi * A[i];
        });
      },
      [&](int64_t a, const double (&v)[3]) {
        const double inv = 1.0 / vol[a];
#pragma unroll
        for (int i = 0; i < 3; ++i) dqdx[3 * a + i] = v[i] * inv;
      });
}

// ---------------------------------------------------------------- segregated momentum
// Momentum as three right-hand sides sharing one scalar matrix: the coupled
// MomentumAdvDiffElemKernel (src/kernel/MomentumAdvDiffElemKernel.C:72-186) with
// the transpose-gradient stress coupling kept on the rhs only (the rhs is the
// full residual, so converged velocities are unchanged).  Row tile on a numDof 1
// graph as k_scalar_rows, with the three residual components in rhs3[i][row].
// ADV, MASS as in k_momentum_rows.
template <bool ADV, bool SKEW, bool SHIFT, bool PACK, typename R, int MASS>
__global__ __launch_bounds__(kRowThreads) void k_momentum_seg_rows(
    MomentumFields F, MassArgs MA, const int32_t* __restrict__ conn,
    const int32_t* __restrict__ row_node, const int32_t* __restrict__ inc_ptr, const int32_t* __restrict__ inc_elem,
    const int32_t* __restrict__ nrp, ElemPos elem_pos, int64_t nrows, int row_len,
    double* __restrict__ vals, double* __restrict__ rhs3, int accumulate) {
  extern __shared__ double seg_all[];
  double* seg = seg_all + (size_t)(threadIdx.x >> 6) * kRowsPerWave * row_len;
  const WaveRows w = wave_rows(row_node, inc_ptr, nrows);
  if (w.r0 >= nrows) return;
  const int32_t s0 = nrp[w.r0];
  const int nseg = nrp[w.r1] - s0;
  for (int i = w.lane; i < nseg; i += 64) seg[i] = 0.0;
  wave_sync();
  double rh[3] = {0.0, 0.0, 0.0};
  if (w.q < w.q1) {
    double* myrow = seg + (nrp[w.r] - s0);
    for (int32_t q = w.q; q < w.q1; q += kSlots) {
      const int32_t t = inc_elem[q];
      RowElem el = row_elem(conn, t >> 3, t & 7);
      const uint64_t pk = hexrow::relative_bytes(elem_pos(t >> 3, t & 7), t & 7);
      const double h = hexrow::handed(t & 7);
      double x[3][8], v[8], lf = 0.0;
      R mn[8];
      load4<PACK, ADV>(F.x, el.nd, x, mn);
      if constexpr (MASS != 0) lf = momentum_mass_row<MASS == 2, PACK>(MA, el.nd, x, h, rh);
      if constexpr (ADV) {
        R am[8];
        momentum_row_seg<SKEW, SHIFT, PACK, R>(F, el, x, mn, h, am, rh);
#pragma unroll
        for (int m = 0; m < 8; ++m) v[m] = (double)am[m];
      } else {
#pragma unroll
        for (int m = 0; m < 8; ++m) v[m] = 0.0;
      }
      if constexpr (MASS != 0) {
#pragma unroll
        for (int m = 0; m < 8; ++m) v[m] += hexrow::scv_shape<MASS == 2>(m) * lf;
      }
#pragma unroll
      for (int m = 0; m < 8; ++m) unsafeAtomicAdd(myrow + hexrow::pos(pk, m), v[m]);
    }
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) rh[i] = row_sum(rh[i]);
  wave_sync();
  double* out = vals + s0;
  if (accumulate) {
    for (int i = w.lane; i < nseg; i += 64) out[i] += seg[i];
  } else {
    for (int i = w.lane; i < nseg; i += 64) __builtin_nontemporal_store(seg[i], out + i);
  }
  // lanes 0, 1, 2 of a row add its three residual components
  const double rr = w.slot == 0 ? rh[0] : w.slot == 1 ? rh[1] : rh[2];
  if (w.slot < 3 && w.r < w.r1) rhs3[w.slot * nrows + w.r] += rr;
}

// ContinuityMassElemKernel (rhs only), and the momentum mass of numDof 3 rows too
// long for a row tile (added to the matrix in place): one thread per row.
template <bool MOM, bool LUMPED>
__global__ __launch_bounds__(256) void k_mass_gather(MassArgs A, const int32_t* __restrict__ conn,
                                                     const double* __restrict__ coords,
                                                     const int32_t* __restrict__ row_node,
                                                     const int32_t* __restrict__ inc_ptr,
                                                     const int32_t* __restrict__ inc_elem,
                                                     const int32_t* __restrict__ nrp,
                                                     ElemPos elem_pos, int64_t nnodes,
                                                     double* __restrict__ vals, double* __restrict__ rhs) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nnodes) return;
  const int32_t a = row_node ? row_node[r] : (int32_t)r;
  const int32_t q1 = inc_ptr[a + 1];
  double rh[3] = {0.0, 0.0, 0.0};
  for (int32_t q = inc_ptr[a]; q < q1; ++q) {
    const int32_t t = inc_elem[q];
    const RowElem el = row_elem(conn, t >> 3, t & 7);
    const double h = hexrow::handed(t & 7);
    double x[3][8];
    load3<false>(Field4<>{{}, coords, nullptr}, el.nd, x);
    if constexpr (MOM) {
      const uint64_t pk = hexrow::relative_bytes(elem_pos(t >> 3, t & 7), t & 7);
      const int32_t L3 = 3 * (nrp[r + 1] - nrp[r]);
      double* row = vals + 9 * (int64_t)nrp[r];
      const double lf = momentum_mass_row<LUMPED, false>(A, el.nd, x, h, rh);
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        if (LUMPED && m != 0) continue;
#pragma unroll
        for (int i = 0; i < 3; ++i) row[i * L3 + 3 * hexrow::pos(pk, m) + i] += hexrow::scv_shape<LUMPED>(m) * lf;
      }
    } else {
      double s = 0.0;
      const double g[3] = {A.g3, A.g2, A.g1};
#pragma unroll
      for (int st = 0; st < 3; ++st) {
        double f[8];
        load1<false>(A.s[st].scal, el.nd, f);
        s += g[st] * hexrow::at_scv<LUMPED>(f);
      }
      const double proj_time_scale = A.dt / A.g1;
      rh[0] -= s * hexrow::scv_volume(x, h) / A.dt / proj_time_scale;
    }
  }
  if (MOM) {
#pragma unroll
    for (int i = 0; i < 3; ++i) rhs[3 * r + i] += rh[i];
  } else {
    rhs[r] += rh[0];
  }
}

void check_assembly_args(nalu_linsys* ls, const nalu_mesh* m, int nd) {
  NALU_REQUIRE(ls && m, NALU_ERR_ARG, "assembly: null handle");
  NALU_REQUIRE(ls->finalized, NALU_ERR_STATE, "assembly: finalizeLinearSystem not called");
  NALU_REQUIRE(ls->mesh == m, NALU_ERR_ARG, "assembly: mesh differs from the one the graph was built on");
  NALU_REQUIRE(ls->num_dof == nd, NALU_ERR_ARG, "assembly: numDof mismatch for this kernel");
  // queued host sumInto calls precede this assembly (and keep it from folding the zero)
  flush_sum_into_queue(ls);
}

}  // namespace

// Opt a kernel into more than the default 64 KiB of dynamic LDS when needed.
void set_lds_limit(const void* kern, size_t bytes) {
  int dev = 0;
  NALU_HIP_CHECK(hipGetDevice(&dev));
  int maxopt = 0;
  NALU_HIP_CHECK(hipDeviceGetAttribute(&maxopt, hipDeviceAttributeSharedMemPerBlockOptin, dev));
  if (maxopt <= 0) NALU_HIP_CHECK(hipDeviceGetAttribute(&maxopt, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  NALU_REQUIRE(bytes <= (size_t)maxopt, NALU_ERR_UNSUPPORTED,
               "assembly tile needs " + std::to_string(bytes) + " B of LDS, device allows " + std::to_string(maxopt));
  if (bytes > 64 * 1024) NALU_HIP_CHECK(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
}

void materialize_pending_zero(nalu_linsys* ls) {
  if (ls->values_pending_zero)
    NALU_HIP_CHECK(hipMemsetAsync(ls->values.p, 0, ls->values.bytes(), ls->stream));
  if (ls->rhs_pending_zero) NALU_HIP_CHECK(hipMemsetAsync(ls->rhs.p, 0, ls->rhs.bytes(), ls->stream));
  ls->values_pending_zero = ls->rhs_pending_zero = false;
  // host sumInto calls queued since the zero come next
  flush_sum_into_queue(ls);
}

}  // namespace nalu

using namespace nalu;

extern "C" int nalu_assemble_scalar_diff(nalu_linsys* ls, const nalu_mesh* m, const double* q, const double* k,
                                         int shifted, int mode) {
  return guarded([&]() -> int {
    check_assembly_args(ls, m, 1);
    NALU_REQUIRE(q && k, NALU_ERR_ARG, "scalar_diff: null field");
    NALU_REQUIRE(mode >= 0 && mode <= 3, NALU_ERR_ARG, "scalar_diff: mode must be 0, 1, 2 or 3");
    PhaseTimer t(ls, PH_ASSEMBLE);
    if (mode == 3) {
      etile_scalar_diff(ls, m, q, k, shifted != 0, fp32_assembly(ls));
    } else if (fp32_assembly(ls)) {
      shifted ? scalar_diff_pass<true, float>(ls, m, q, k, mode) : scalar_diff_pass<false, float>(ls, m, q, k, mode);
    } else {
      shifted ? scalar_diff_pass<true, double>(ls, m, q, k, mode) : scalar_diff_pass<false, double>(ls, m, q, k, mode);
    }
    return NALU_OK;
  });
}

extern "C" int nalu_assemble_continuity(nalu_linsys* ls, const nalu_mesh* m, const double* rho, const double* p,
                                        const double* u, const double* gp, double tau, int shift_mdot,
                                        int shift_poisson, int reduced_sens, int mode) {
  return guarded([&]() -> int {
    check_assembly_args(ls, m, 1);
    NALU_REQUIRE(rho && p && u && gp, NALU_ERR_ARG, "continuity: null field");
    NALU_REQUIRE(tau > 0.0, NALU_ERR_ARG, "continuity: projTimeScale must be positive");
    NALU_REQUIRE(mode >= 0 && mode <= 3, NALU_ERR_ARG, "continuity: mode must be 0, 1, 2 or 3");
    PhaseTimer t(ls, PH_ASSEMBLE);
    const int key = (shift_mdot ? 4 : 0) | (shift_poisson ? 2 : 0) | (reduced_sens ? 1 : 0);
    if (mode == 3) {
      etile_continuity(ls, m, rho, p, u, gp, tau, key, fp32_assembly(ls));
      return NALU_OK;
    }
    switch (key) {
#define NALU_CT(K, A, B, C)                                                                              \
  case K:                                                                                                \
    fp32_assembly(ls) ? continuity_pass<A, B, C, false, float>(ls, m, rho, p, u, gp, tau, mode, nullptr)  \
                      : continuity_pass<A, B, C, false, double>(ls, m, rho, p, u, gp, tau, mode, nullptr); \
    break;
      NALU_CT(0, false, false, false)
      NALU_CT(1, false, false, true)
      NALU_CT(2, false, true, false)
      NALU_CT(3, false, true, true)
      NALU_CT(4, true, false, false)
      NALU_CT(5, true, false, true)
      NALU_CT(6, true, true, false)
      NALU_CT(7, true, true, true)
#undef NALU_CT
    }
    return NALU_OK;
  });
}

extern "C" int nalu_assemble_continuity_mdot(nalu_linsys* ls, const nalu_mesh* m, const double* rho,
                                             const double* p, const double* u, const double* gp, double tau,
                                             int shift_mdot, int shift_poisson, int reduced_sens, double* mdot) {
  return guarded([&]() -> int {
    check_assembly_args(ls, m, 1);
    NALU_REQUIRE(rho && p && u && gp && mdot, NALU_ERR_ARG, "continuity + mdot: null field");
    NALU_REQUIRE(tau > 0.0, NALU_ERR_ARG, "continuity + mdot: projTimeScale must be positive");
    PhaseTimer t(ls, PH_ASSEMBLE);
    const int key = (shift_mdot ? 4 : 0) | (shift_poisson ? 2 : 0) | (reduced_sens ? 1 : 0);
    switch (key) {
#define NALU_CM(K, A, B, C)                                                                       \
  case K:                                                                                         \
    fp32_assembly(ls) ? continuity_pass<A, B, C, true, float>(ls, m, rho, p, u, gp, tau, 0, mdot)  \
                      : continuity_pass<A, B, C, true, double>(ls, m, rho, p, u, gp, tau, 0, mdot); \
    break;
      NALU_CM(0, false, false, false)
      NALU_CM(1, false, false, true)
      NALU_CM(2, false, true, false)
      NALU_CM(3, false, true, true)
      NALU_CM(4, true, false, false)
      NALU_CM(5, true, false, true)
      NALU_CM(6, true, true, false)
      NALU_CM(7, true, true, true)
#undef NALU_CM
    }
    return NALU_OK;
  });
}

extern "C" int nalu_compute_mdot(const nalu_mesh* m, const double* rho, const double* p, const double* u,
                                 const double* gp, double tau, int shift_mdot, int shift_poisson, double* mdot,
                                 void* stream) {
  return guarded([&]() -> int {
    NALU_REQUIRE(m && rho && p && u && gp && mdot, NALU_ERR_ARG, "mdot: null argument");
    NALU_REQUIRE(tau > 0.0, NALU_ERR_ARG, "mdot: projTimeScale must be positive");
    launch_mdot<double>(m, rho, p, u, gp, tau, shift_mdot, shift_poisson, mdot, (hipStream_t)stream);
    return NALU_OK;
  });
}

extern "C" int nalu_compute_mdot_f32(const nalu_mesh* m, const double* rho, const double* p, const double* u,
                                     const double* gp, double tau, int shift_mdot, int shift_poisson, double* mdot,
                                     void* stream) {
  return guarded([&]() -> int {
    NALU_REQUIRE(m && rho && p && u && gp && mdot, NALU_ERR_ARG, "mdot: null argument");
    NALU_REQUIRE(tau > 0.0, NALU_ERR_ARG, "mdot: projTimeScale must be positive");
    launch_mdot<float>(m, rho, p, u, gp, tau, shift_mdot, shift_poisson, mdot, (hipStream_t)stream);
    return NALU_OK;
  });
}

namespace {
// The longest node rows that mode 2 and the one-pass forms accept: 64 of them (and
// their rhs) fit the LDS of a CU (35 columns).  Longer ones are refused by mode 2 and
// take the atomic form and the mass gather.  A block of k_momentum_rows holds half as
// many rows, so this limit is the entry points' and not the kernel's.
bool numdof3_rows_fit(const nalu_linsys* ls) {
  return (64 * (size_t)ls->max_node_row_len * 9 + 3 * 64) * sizeof(double) <= kMaxLds;
}

// Fields of a momentum pass as its kernels read them, copied to records for larger
// systems; a velocity state that is the advected field itself is copied once.
struct MomentumPass {
  MomentumFields F;
  MassArgs A{};
  MomentumPass(nalu_linsys* ls, const nalu_mesh* m, bool adv, const double* u, const double* mu, const double* mdot,
               double include_divu, const MassArgs* ma)
      : F{{{}, m->coords.p, mu}, {{}, u, nullptr}, mdot, include_divu} {
    if (ma) A = *ma;
    if (!use_pack(ls)) return;
    const bool same = adv && ma && A.s[2].vec == u;
    if (same) F.u.scal = A.s[2].scal;
    Field4<>* f[6];
    int n = 0;
    f[n++] = &F.x;
    if (adv) f[n++] = &F.u;
    if (ma) {
      f[n++] = &A.s[0];
      f[n++] = &A.s[1];
      if (!same) f[n++] = &A.s[2];
      f[n++] = &A.gjp;
    }
    pack_fields(ls, f, n);
    if (same) A.s[2] = F.u;
  }
};

// The numDof 3 row-tile pass: advection-diffusion (adv), momentum mass (ma), or both.
void launch_momentum_rows(nalu_linsys* ls, const nalu_mesh* m, bool adv, const double* u, const double* mu,
                          const double* mdot, double include_divu, bool skew, bool shifted, const MassArgs* ma,
                          bool lumped) {
  build_node_incidence(const_cast<nalu_mesh*>(m), ls->stream);
  NALU_REQUIRE(ls->values_pending_zero == ls->rhs_pending_zero, NALU_ERR_STATE,
               "tile assembly: values/rhs zero state diverged");
  NALU_REQUIRE(numdof3_rows_fit(ls), NALU_ERR_UNSUPPORTED, "momentum row tile: node rows are too long");
  const int accumulate = ls->values_pending_zero ? 0 : 1;
  const size_t lds = (size_t)kMomRows * (ls->max_node_row_len * 9 + 3) * sizeof(double);
  MomentumPass P(ls, m, adv, u, mu, mdot, include_divu, ma);
  auto go = [&](auto kern) {
    set_lds_limit((const void*)kern, lds);
    hipLaunchKernelGGL(kern, dim3(blocks_for(ls->num_nodes, kMomRows)), dim3(kMomThreads), lds, ls->stream, P.F, P.A,
                       m->conn.p, (const int32_t*)ls->row_node.p, m->inc_ptr.p, m->inc_elem.p, ls->nrp.p,
                       elem_pos_of(ls), ls->num_nodes, ls->values.p, ls->rhs.p, accumulate);
  };
  // the mass part is FP64 arithmetic at either precision of the advection-diffusion part
  const bool f32 = fp32_assembly(ls);
  auto pick = [&](auto pack) {
    constexpr bool S = decltype(pack)::value;
    if (!adv) {
      lumped ? go(k_momentum_rows<false, false, false, S, double, 2>) : go(k_momentum_rows<false, false, false, S, double, 1>);
    } else if (ma) {  // one-pass forms for the default advection options only (compile time)
      NALU_REQUIRE(!skew && !shifted, NALU_ERR_UNSUPPORTED, "momentum tile: one pass with mass needs skew = shifted = 0");
      if (lumped) f32 ? go(k_momentum_rows<true, false, false, S, float, 2>) : go(k_momentum_rows<true, false, false, S, double, 2>);
      else f32 ? go(k_momentum_rows<true, false, false, S, float, 1>) : go(k_momentum_rows<true, false, false, S, double, 1>);
    } else {
      if (skew && shifted) f32 ? go(k_momentum_rows<true, true, true, S, float, 0>) : go(k_momentum_rows<true, true, true, S, double, 0>);
      else if (skew) f32 ? go(k_momentum_rows<true, true, false, S, float, 0>) : go(k_momentum_rows<true, true, false, S, double, 0>);
      else if (shifted) f32 ? go(k_momentum_rows<true, false, true, S, float, 0>) : go(k_momentum_rows<true, false, true, S, double, 0>);
      else f32 ? go(k_momentum_rows<true, false, false, S, float, 0>) : go(k_momentum_rows<true, false, false, S, double, 0>);
    }
  };
  use_pack(ls) ? pick(std::true_type{}) : pick(std::false_type{});
  ls->values_pending_zero = ls->rhs_pending_zero = false;
  NALU_HIP_CHECK(hipGetLastError());
}
}  // namespace

extern "C" int nalu_assemble_momentum(nalu_linsys* ls, const nalu_mesh* m, const double* u, const double* mu,
                                      const double* mdot, double include_divu, int skew, int shifted, int mode) {
  return guarded([&]() -> int {
    check_assembly_args(ls, m, 3);
    NALU_REQUIRE(u && mu && mdot, NALU_ERR_ARG, "momentum: null field");
    NALU_REQUIRE(mode >= 1 && mode <= 3, NALU_ERR_UNSUPPORTED,
                 "momentum: mode 1 (atomic), 2 (node tile) or 3 (element tile); the per-thread row gather is "
                 "scalar-only");
    PhaseTimer t(ls, PH_ASSEMBLE);
    const int64_t E = m->num_elems;
    if (mode == 3) {
      build_node_incidence(const_cast<nalu_mesh*>(m), ls->stream);
      etile_momentum(ls, m, u, mu, mdot, include_divu, skew != 0, shifted != 0, fp32_assembly(ls));
    } else if (mode == 2) {
      launch_momentum_rows(ls, m, true, u, mu, mdot, include_divu, skew != 0, shifted != 0, nullptr, false);
    } else {
      materialize_pending_zero(ls);
      const dim3 g(chunk_blocks<8>(E)), b(kChunk);
      auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, g, b, 0, ls->stream, m->conn.p, m->coords.p, u, mu, mdot, include_divu,
                           ls->node_lid.p, ls->nrp.p, elem_pos_of(ls), E, ls->values.p, ls->rhs.p);
      };
      const bool f32 = fp32_assembly(ls);
      if (skew && shifted) f32 ? go(k_momentum_atomic<true, true, float>) : go(k_momentum_atomic<true, true, double>);
      else if (skew) f32 ? go(k_momentum_atomic<true, false, float>) : go(k_momentum_atomic<true, false, double>);
      else if (shifted) f32 ? go(k_momentum_atomic<false, true, float>) : go(k_momentum_atomic<false, true, double>);
      else f32 ? go(k_momentum_atomic<false, false, float>) : go(k_momentum_atomic<false, false, double>);
    }
    NALU_HIP_CHECK(hipGetLastError());
    return NALU_OK;
  });
}

extern "C" int nalu_linsys_sum_into_batch(nalu_linsys* ls, int64_t nelem, const int32_t* conn, const double* lhs,
                                          const double* rhs_e) {
  return guarded([&]() -> int {
    NALU_REQUIRE(ls && ls->finalized, NALU_ERR_STATE, "sum_into_batch: system not finalized");
    NALU_REQUIRE(nelem >= 0 && (nelem == 0 || (conn && lhs && rhs_e)), NALU_ERR_ARG, "sum_into_batch: bad args");
    NALU_REQUIRE(ls->mesh && nelem <= ls->mesh->num_elems, NALU_ERR_ARG, "sum_into_batch: more elements than the graph");
    PhaseTimer t(ls, PH_ASSEMBLE);
    materialize_pending_zero(ls);
    if (nelem == 0) return NALU_OK;
    // the element scatter table indexes the graph's own elements
    NALU_REQUIRE(conn == ls->mesh->conn.p, NALU_ERR_ARG,
                 "sum_into_batch: conn must be the graph mesh's connectivity (nalu_mesh_device_ptrs)");
    const int64_t n = nelem * 8 * ls->num_dof;
    hipLaunchKernelGGL(k_sum_into_batch, dim3(blocks_for(n, 256)), dim3(256), 0, ls->stream, conn, lhs, rhs_e,
                       ls->node_lid.p, ls->nrp.p, elem_pos_of(ls), nelem, ls->num_dof, ls->values.p, ls->rhs.p);
    NALU_HIP_CHECK(hipGetLastError());
    return NALU_OK;
  });
}

extern "C" int nalu_linsys_apply_dirichlet(nalu_linsys* ls, int64_t nbc, const int32_t* nodes, const double* sol,
                                           const double* bcv, int begin, int end) {
  return guarded([&]() -> int {
    NALU_REQUIRE(ls && ls->finalized, NALU_ERR_STATE, "applyDirichletBCs: system not finalized");
    NALU_REQUIRE(begin >= 0 && end <= ls->num_dof && begin <= end, NALU_ERR_ARG, "applyDirichletBCs: bad dof range");
    NALU_REQUIRE(nbc == 0 || (nodes && sol && bcv), NALU_ERR_ARG, "applyDirichletBCs: null array");
    PhaseTimer t(ls, PH_DIRICHLET);
    materialize_pending_zero(ls);
    const int64_t n = nbc * (end - begin);
    if (n == 0) return NALU_OK;
    PoolScope scope(ls->pool);
    DevBuf<int> bad(1);
    NALU_HIP_CHECK(hipMemsetAsync(bad.p, 0, sizeof(int), ls->stream));
    hipLaunchKernelGGL(k_dirichlet, dim3(blocks_for(n, 256)), dim3(256), 0, ls->stream, nodes, nbc, ls->num_nodes,
                       ls->num_dof, begin, end, ls->node_lid.p, ls->row_ptr.p, ls->col_idx.p, sol, bcv,
                       ls->values.p, ls->rhs.p, 0, 0.0, 0.0, bad.p);
    NALU_HIP_CHECK(hipGetLastError());
    check_flag(bad, ls->stream, "applyDirichletBCs: node index outside the mesh");
    return NALU_OK;
  });
}

extern "C" int nalu_linsys_reset_rows(nalu_linsys* ls, int64_t nn, const int32_t* nodes, int begin, int end,
                                      double diag_value, double rhs_residual) {
  return guarded([&]() -> int {
    NALU_REQUIRE(ls && ls->finalized, NALU_ERR_STATE, "resetRows: system not finalized");
    NALU_REQUIRE(begin >= 0 && end <= ls->num_dof && begin <= end, NALU_ERR_ARG, "resetRows: bad dof range");
    NALU_REQUIRE(nn == 0 || nodes, NALU_ERR_ARG, "resetRows: null node list");
    PhaseTimer t(ls, PH_DIRICHLET);
    materialize_pending_zero(ls);
    const int64_t n = nn * (end - begin);
    if (n == 0) return NALU_OK;
    PoolScope scope(ls->pool);
    DevBuf<int> bad(1);
    NALU_HIP_CHECK(hipMemsetAsync(bad.p, 0, sizeof(int), ls->stream));
    hipLaunchKernelGGL(k_dirichlet, dim3(blocks_for(n, 256)), dim3(256), 0, ls->stream, nodes, nn, ls->num_nodes,
                       ls->num_dof, begin, end, ls->node_lid.p, ls->row_ptr.p, ls->col_idx.p, (const double*)nullptr,
                       (const double*)nullptr, ls->values.p, ls->rhs.p, 1, diag_value, rhs_residual, bad.p);
    NALU_HIP_CHECK(hipGetLastError());
    check_flag(bad, ls->stream, "resetRows: node index outside the mesh");
    return NALU_OK;
  });
}

namespace {
template <bool MOM>
void launch_mass_gather(nalu_linsys* ls, const nalu_mesh* m, const MassArgs& A, bool lumped) {
  build_node_incidence(const_cast<nalu_mesh*>(m), ls->stream);
  materialize_pending_zero(ls);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(blocks_for(ls->num_nodes, 256)), dim3(256), 0, ls->stream, A, m->conn.p,
                       m->coords.p, (const int32_t*)ls->row_node.p, m->inc_ptr.p, m->inc_elem.p, ls->nrp.p,
                       elem_pos_of(ls), ls->num_nodes, ls->values.p, ls->rhs.p);
  };
  lumped ? go(k_mass_gather<MOM, true>) : go(k_mass_gather<MOM, false>);
  NALU_HIP_CHECK(hipGetLastError());
}

void check_mass_args(double dt, const double* gamma) {
  NALU_REQUIRE(gamma, NALU_ERR_ARG, "mass: null gamma");
  NALU_REQUIRE(std::isfinite(dt) && dt > 0.0, NALU_ERR_ARG, "mass: dt must be positive");
  NALU_REQUIRE(std::isfinite(gamma[0]) && gamma[0] != 0.0 && std::isfinite(gamma[1]) && std::isfinite(gamma[2]),
               NALU_ERR_ARG, "mass: gamma1 must be nonzero and all gammas finite");
}
}  // namespace

extern "C" int nalu_assemble_momentum_mass(nalu_linsys* ls, const nalu_mesh* m, const double* rho_nm1,
                                           const double* rho_n, const double* rho_np1, const double* u_nm1,
                                           const double* u_n, const double* u_np1, const double* gjp, double dt,
                                           const double* gamma, int lumped, int balanced_force) {
  return guarded([&]() -> int {
    check_assembly_args(ls, m, 3);
    check_mass_args(dt, gamma);
    NALU_REQUIRE(rho_nm1 && rho_n && rho_np1 && u_nm1 && u_n && u_np1 && gjp, NALU_ERR_ARG,
                 "momentum_mass: null field");
    PhaseTimer t(ls, PH_ASSEMBLE);
    const MassArgs A{{{{}, u_nm1, rho_nm1}, {{}, u_n, rho_n}, {{}, u_np1, rho_np1}}, {{}, gjp, nullptr}, dt, gamma[0], gamma[1], gamma[2],
                     balanced_force ? 1 : 0};
    if (numdof3_rows_fit(ls) && ls->values_pending_zero == ls->rhs_pending_zero)
      launch_momentum_rows(ls, m, false, nullptr, nullptr, nullptr, 0.0, false, false, &A, lumped != 0);
    else launch_mass_gather<true>(ls, m, A, lumped != 0);
    return NALU_OK;
  });
}

extern "C" int nalu_assemble_momentum_with_mass(nalu_linsys* ls, const nalu_mesh* m, const double* u, const double* mu,
                                                const double* mdot, double include_divu, int skew, int shifted,
                                                const double* rho_nm1, const double* rho_n, const double* rho_np1,
                                                const double* u_nm1, const double* u_n, const double* u_np1,
                                                const double* gjp, double dt, const double* gamma, int lumped,
                                                int balanced_force) {
  return guarded([&]() -> int {
    check_assembly_args(ls, m, 3);
    check_mass_args(dt, gamma);
    NALU_REQUIRE(u && mu && mdot, NALU_ERR_ARG, "momentum_with_mass: null advection-diffusion field");
    NALU_REQUIRE(rho_nm1 && rho_n && rho_np1 && u_nm1 && u_n && u_np1 && gjp, NALU_ERR_ARG,
                 "momentum_with_mass: null mass field");
    const bool tile = numdof3_rows_fit(ls);
    // the two passes one after the other: rows too long for a row tile, or the
    // skew-symmetric / shifted advection options (one-pass forms exist for the defaults)
    if (!tile || skew || shifted) {
      int rc = nalu_assemble_momentum(ls, m, u, mu, mdot, include_divu, skew, shifted, tile ? 2 : 1);
      if (rc != NALU_OK) return rc;
      return nalu_assemble_momentum_mass(ls, m, rho_nm1, rho_n, rho_np1, u_nm1, u_n, u_np1, gjp, dt, gamma, lumped,
                                         balanced_force);
    }
    PhaseTimer t(ls, PH_ASSEMBLE);
    const MassArgs A{{{{}, u_nm1, rho_nm1}, {{}, u_n, rho_n}, {{}, u_np1, rho_np1}}, {{}, gjp, nullptr}, dt, gamma[0], gamma[1], gamma[2],
                     balanced_force ? 1 : 0};
    launch_momentum_rows(ls, m, true, u, mu, mdot, include_divu, skew != 0, shifted != 0, &A, lumped != 0);
    NALU_HIP_CHECK(hipGetLastError());
    return NALU_OK;
  });
}

extern "C" int nalu_assemble_continuity_mass(nalu_linsys* ls, const nalu_mesh* m, const double* rho_nm1,
                                             const double* rho_n, const double* rho_np1, double dt,
                                             const double* gamma, int lumped) {
  return guarded([&]() -> int {
    check_assembly_args(ls, m, 1);
    check_mass_args(dt, gamma);
    NALU_REQUIRE(rho_nm1 && rho_n && rho_np1, NALU_ERR_ARG, "continuity_mass: null field");
    PhaseTimer t(ls, PH_ASSEMBLE);
    const MassArgs A{{{{}, nullptr, rho_nm1}, {{}, nullptr, rho_n}, {{}, nullptr, rho_np1}}, {}, dt, gamma[0], gamma[1],
                     gamma[2], 0};
    launch_mass_gather<false>(ls, m, A, lumped != 0);
    return NALU_OK;
  });
}

namespace {
// The segregated momentum row tile: advection-diffusion (adv), momentum mass (ma), or both.
void launch_momentum_seg(nalu_linsys* ls, const nalu_mesh* m, bool adv, const double* u, const double* mu,
                         const double* mdot, double include_divu, bool skew, bool shifted, double* rhs3,
                         const MassArgs* ma, bool lumped) {
  build_node_incidence(const_cast<nalu_mesh*>(m), ls->stream);
  if (ls->rhs_pending_zero) NALU_HIP_CHECK(hipMemsetAsync(ls->rhs.p, 0, ls->rhs.bytes(), ls->stream));
  ls->rhs_pending_zero = false;
  const int accumulate = ls->values_pending_zero ? 0 : 1;
  const size_t lds = lds_rows(ls);
  MomentumPass P(ls, m, adv, u, mu, mdot, include_divu, ma);
  auto go = [&](auto kern) {
    set_lds_limit((const void*)kern, lds);
    hipLaunchKernelGGL(kern, dim3(blocks_for(ls->nrows, kRowsPerBlock)), dim3(kRowThreads), lds, ls->stream, P.F, P.A,
                       m->conn.p, (const int32_t*)ls->row_node.p, m->inc_ptr.p, m->inc_elem.p, ls->nrp.p,
                       elem_pos_of(ls), ls->nrows, ls->max_node_row_len, ls->values.p, rhs3, accumulate);
  };
  // the mass part is FP64 arithmetic at either precision of the advection-diffusion part
  const bool f32 = fp32_assembly(ls);
  auto pick = [&](auto pack) {
    constexpr bool S = decltype(pack)::value;
    if (!adv) {
      lumped ? go(k_momentum_seg_rows<false, false, false, S, double, 2>)
             : go(k_momentum_seg_rows<false, false, false, S, double, 1>);
    } else if (ma) {  // one-pass forms for the default advection options only (compile time)
      NALU_REQUIRE(!skew && !shifted, NALU_ERR_UNSUPPORTED,
                   "momentum rows: one pass with mass needs skew = shifted = 0");
      if (lumped) f32 ? go(k_momentum_seg_rows<true, false, false, S, float, 2>) : go(k_momentum_seg_rows<true, false, false, S, double, 2>);
      else f32 ? go(k_momentum_seg_rows<true, false, false, S, float, 1>) : go(k_momentum_seg_rows<true, false, false, S, double, 1>);
    } else {
      if (skew && shifted) f32 ? go(k_momentum_seg_rows<true, true, true, S, float, 0>) : go(k_momentum_seg_rows<true, true, true, S, double, 0>);
      else if (skew) f32 ? go(k_momentum_seg_rows<true, true, false, S, float, 0>) : go(k_momentum_seg_rows<true, true, false, S, double, 0>);
      else if (shifted) f32 ? go(k_momentum_seg_rows<true, false, true, S, float, 0>) : go(k_momentum_seg_rows<true, false, true, S, double, 0>);
      else f32 ? go(k_momentum_seg_rows<true, false, false, S, float, 0>) : go(k_momentum_seg_rows<true, false, false, S, double, 0>);
    }
  };
  use_pack(ls) ? pick(std::true_type{}) : pick(std::false_type{});
  ls->values_pending_zero = false;
  NALU_HIP_CHECK(hipGetLastError());
}
}  // namespace

extern "C" int nalu_assemble_momentum_segregated(nalu_linsys* ls, const nalu_mesh* m, const double* u,
                                                 const double* mu, const double* mdot, double include_divu,
                                                 int skew, int shifted, double* rhs3) {
  return guarded([&]() -> int {
    check_assembly_args(ls, m, 1);
    NALU_REQUIRE(u && mu && mdot && rhs3, NALU_ERR_ARG, "momentum_segregated: null field");
    PhaseTimer t(ls, PH_ASSEMBLE);
    launch_momentum_seg(ls, m, true, u, mu, mdot, include_divu, skew != 0, shifted != 0, rhs3, nullptr, false);
    return NALU_OK;
  });
}

extern "C" int nalu_assemble_momentum_mass_segregated(nalu_linsys* ls, const nalu_mesh* m, const double* rho_nm1,
                                                      const double* rho_n, const double* rho_np1,
                                                      const double* u_nm1, const double* u_n, const double* u_np1,
                                                      const double* gjp, double dt, const double* gamma, int lumped,
                                                      int balanced_force, double* rhs3) {
  return guarded([&]() -> int {
    check_assembly_args(ls, m, 1);
    check_mass_args(dt, gamma);
    NALU_REQUIRE(rho_nm1 && rho_n && rho_np1 && u_nm1 && u_n && u_np1 && gjp && rhs3, NALU_ERR_ARG,
                 "momentum_mass_segregated: null field");
    PhaseTimer t(ls, PH_ASSEMBLE);
    const MassArgs A{{{{}, u_nm1, rho_nm1}, {{}, u_n, rho_n}, {{}, u_np1, rho_np1}}, {{}, gjp, nullptr}, dt, gamma[0], gamma[1], gamma[2],
                     balanced_force ? 1 : 0};
    launch_momentum_seg(ls, m, false, nullptr, nullptr, nullptr, 0.0, false, false, rhs3, &A, lumped != 0);
    return NALU_OK;
  });
}

extern "C" int nalu_assemble_momentum_with_mass_segregated(
    nalu_linsys* ls, const nalu_mesh* m, const double* u, const double* mu, const double* mdot, double include_divu,
    int skew, int shifted, const double* rho_nm1, const double* rho_n, const double* rho_np1, const double* u_nm1,
    const double* u_n, const double* u_np1, const double* gjp, double dt, const double* gamma, int lumped,
    int balanced_force, double* rhs3) {
  return guarded([&]() -> int {
    check_assembly_args(ls, m, 1);
    check_mass_args(dt, gamma);
    NALU_REQUIRE(u && mu && mdot && rhs3, NALU_ERR_ARG, "momentum_with_mass_segregated: null field");
    NALU_REQUIRE(rho_nm1 && rho_n && rho_np1 && u_nm1 && u_n && u_np1 && gjp, NALU_ERR_ARG,
                 "momentum_with_mass_segregated: null mass field");
    if (skew || shifted) {  // one-pass forms exist for the default advection options
      const int rc = nalu_assemble_momentum_segregated(ls, m, u, mu, mdot, include_divu, skew, shifted, rhs3);
      if (rc != NALU_OK) return rc;
      return nalu_assemble_momentum_mass_segregated(ls, m, rho_nm1, rho_n, rho_np1, u_nm1, u_n, u_np1, gjp, dt, gamma,
                                                    lumped, balanced_force, rhs3);
    }
    PhaseTimer t(ls, PH_ASSEMBLE);
    const MassArgs A{{{{}, u_nm1, rho_nm1}, {{}, u_n, rho_n}, {{}, u_np1, rho_np1}}, {{}, gjp, nullptr}, dt, gamma[0], gamma[1], gamma[2],
                     balanced_force ? 1 : 0};
    launch_momentum_seg(ls, m, true, u, mu, mdot, include_divu, false, false, rhs3, &A, lumped != 0);
    return NALU_OK;
  });
}

extern "C" int nalu_compute_dual_volume(const nalu_mesh* m, double* dual_vol, void* stream) {
  return guarded([&]() -> int {
    NALU_REQUIRE(m && dual_vol, NALU_ERR_ARG, "dual_volume: null argument");
    hipStream_t s = (hipStream_t)stream;
    build_node_incidence(const_cast<nalu_mesh*>(m), s);
    hipLaunchKernelGGL(k_dual_volume, dim3(blocks_for(m->num_nodes, kRowsPerBlock)), dim3(kRowThreads), 0, s, m->conn.p, m->coords.p,
                       m->inc_ptr.p, m->inc_elem.p, m->num_nodes, dual_vol);
    NALU_HIP_CHECK(hipGetLastError());
    return NALU_OK;
  });
}

namespace {
void nodal_grad_interior(const nalu_mesh* m, const double* q, const double* dual_vol, int shifted, double* dqdx,
                         hipStream_t s) {
  build_node_incidence(const_cast<nalu_mesh*>(m), s);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(blocks_for(m->num_nodes, kRowsPerBlock)), dim3(kRowThreads), 0, s, m->conn.p, m->coords.p, q,
                       dual_vol, m->inc_ptr.p, m->inc_elem.p, m->num_nodes, dqdx);
  };
  if (shifted) go(k_nodal_grad<true>);
  else go(k_nodal_grad<false>);
  NALU_HIP_CHECK(hipGetLastError());
}
}  // namespace

extern "C" int nalu_compute_nodal_gradient(const nalu_mesh* m, const double* q, const double* dual_vol, int shifted,
                                           double* dqdx, void* stream) {
  return guarded([&]() -> int {
    NALU_REQUIRE(m && q && dual_vol && dqdx, NALU_ERR_ARG, "nodal_gradient: null argument");
    hipStream_t s = (hipStream_t)stream;
    nodal_grad_interior(m, q, dual_vol, shifted, dqdx, s);
    nodal_grad_boundary(const_cast<nalu_mesh*>(m), q, dual_vol, shifted != 0, dqdx, s);
    return NALU_OK;
  });
}

extern "C" int nalu_compute_nodal_gradient_interior(const nalu_mesh* m, const double* q, const double* dual_vol,
                                                    int shifted, double* dqdx, void* stream) {
  return guarded([&]() -> int {
    NALU_REQUIRE(m && q && dual_vol && dqdx, NALU_ERR_ARG, "nodal_gradient: null argument");
    nodal_grad_interior(m, q, dual_vol, shifted, dqdx, (hipStream_t)stream);
    return NALU_OK;
  });
}

extern "C" int nalu_nodal_gradient_boundary(const nalu_mesh* m, const double* q, const double* dual_vol, int shifted,
                                            double* dqdx, void* stream) {
  return guarded([&]() -> int {
    NALU_REQUIRE(m && q && dual_vol && dqdx, NALU_ERR_ARG, "nodal_gradient_boundary: null argument");
    nodal_grad_boundary(const_cast<nalu_mesh*>(m), q, dual_vol, shifted != 0, dqdx, (hipStream_t)stream);
    return NALU_OK;
  });
}

extern "C" int nalu_mesh_exposed_faces(const nalu_mesh* m, int64_t* num_faces, int32_t* faces_host) {
  return guarded([&]() -> int {
    NALU_REQUIRE(m && num_faces, NALU_ERR_ARG, "mesh_exposed_faces: null argument");
    build_exposed_faces(const_cast<nalu_mesh*>(m), nullptr);
    *num_faces = m->num_exposed;
    if (faces_host && m->num_exposed)
      NALU_HIP_CHECK(hipMemcpy(faces_host, m->exposed_faces.p, sizeof(int32_t) * 4 * m->num_exposed,
                               hipMemcpyDeviceToHost));
    return NALU_OK;
  });
}
