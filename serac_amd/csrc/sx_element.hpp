// sx_element.hpp -- fused element kernels for H1 hexahedra on gfx950.
//
// Per element, the pipeline of fn/domain_integral_kernels.hpp:155-304 runs in
// one workgroup-resident pass:
//   gather L -> LDS                           (fn/element_restriction.cpp:443-454)
//   sum-factorized interpolate (3 stages)     (fn/detail/hexahedron_H1.inl:169-228)
//   quadrature point: qfunction + parent/physical maps (+ its closed-form tangent)
//                     or stored-tangent chain rule for J.v
//   sum-factorized integrate (3 stages)       (fn/detail/hexahedron_H1.inl:230-280)
//   scatter-add LDS -> L                      (fn/element_restriction.cpp:456-467)
//
// Thread mapping: the workgroup has 256 lanes (4 wave64s) and holds EB =
// floor(256 / Q^3) elements; lane li of element el owns the index triple
// (i2, i1, i0) = li as a node (z,y,x) or a quadrature point (qz,qy,qx), which is
// possible because every form here uses Q = p + 1 = nodes per direction
// (fn/functional.hpp:193).  In the contractions of the residual, the
// linearization and the diagonal a lane owns rows instead (see Rows).
//
// The scatter-add is an FP64/FP32 atomic add, or a plain store of the element's
// values for a node sum that follows (SCATTER_ELEMENT, reproducible), both in
// one launch for all elements, or a plain read-modify-write (one launch per
// element colour: no two elements of a colour share a node).
//
// Precision: residual and linearization compute in FP64.  The stored tangent
// is kept in S = double, float or bf16; the J.v kernel computes in T = double
// or float and exchanges vectors in V = double or float (float arithmetic on
// double vectors is the operator of the mixed-precision solvers).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sx_launch.hpp"
#include "sx_qfunctions.hpp"

namespace sxk {

// ---------------------------------------------------------------------------
// storage types of the tangent
// ---------------------------------------------------------------------------
struct bf16 {
  uint16_t bits;
};

__device__ __forceinline__ double to_real(double v, double) { return v; }
__device__ __forceinline__ float  to_real(float v, float) { return v; }
__device__ __forceinline__ double to_real(float v, double) { return double(v); }
__device__ __forceinline__ float  to_real(double v, float) { return float(v); }
__device__ __forceinline__ float  bf16_to_float(uint32_t bits16) { return __uint_as_float(bits16 << 16); }

// FP64 -> storage, round to nearest even
__device__ __forceinline__ double   to_store(double v, double*) { return v; }
__device__ __forceinline__ float    to_store(double v, float*) { return float(v); }
__device__ __forceinline__ uint16_t to_store(double v, bf16*)
{
  const uint32_t u = __float_as_uint(float(v));
  if ((u & 0x7f800000u) == 0x7f800000u) return uint16_t((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));  // inf / NaN
  return uint16_t((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

template <typename S>
struct StoreTraits {
  using raw = S;
};
template <>
struct StoreTraits<bf16> {
  using raw = uint16_t;
};

// Per-slot tangent layout, in units of S: the DS packed entries of quadrature
// point q are grouped VEC = 16 / sizeof(S) at a time, [g][q][VEC], so that lane
// q reads 16 bytes per group.  The REM entries of the last, partial group
// follow entry-major so that each load is coalesced across the points: for
// 2-byte S in pairs, [RP][q][2] (lane q reads one 4-byte word per pair), then
// an odd last entry as [q]; for wider S one entry at a time, [REM][q].
template <typename S, int DS, int NQ>
struct TangentLayout {
  static constexpr int     VEC    = 16 / int(sizeof(S));
  static constexpr int     G      = DS / VEC;
  static constexpr int     REM    = DS - G * VEC;
  static constexpr int     RP     = sizeof(S) == 2 ? REM / 2 : 0;  // remainder pairs
  static constexpr int64_t stride = (int64_t(DS) * NQ * int64_t(sizeof(S)) + 15) / 16 * (16 / int64_t(sizeof(S)));
  __host__ __device__ static constexpr int offset(int k, int q)
  {
    return (k < G * VEC)          ? (k / VEC) * VEC * NQ + q * VEC + (k % VEC)
           : (k - G * VEC < 2 * RP) ? G * VEC * NQ + ((k - G * VEC) / 2) * 2 * NQ + q * 2 + (k - G * VEC) % 2
                                    : G * VEC * NQ + 2 * RP * NQ + (k - G * VEC - 2 * RP) * NQ + q;
  }
};

// packed index of the symmetric tangent: upper triangle, column-major, the order
// in which an integrand's tangent() emits: column s is s(s+1)/2 .. s(s+1)/2+s
__host__ __device__ constexpr int packed_index(int r, int s) { return r <= s ? s * (s + 1) / 2 + r : r * (r + 1) / 2 + s; }

// Shape of the stored tangent for a layout: M inputs/outputs per point
// (VAL: the field value is an input and the source an output), DS stored
// entries, and where entry D(r, s) = d out_r / d in_s lives.  Column s holds
// entries idx(r, s) for r < rows(s), in increasing storage order.
template <int LAYOUT, int NC>
struct TanShape {
  static constexpr bool VAL = (LAYOUT == LAYOUT_FULL_SYM);
  static constexpr bool SYM = (LAYOUT != LAYOUT_GRAD_FULL);
  static constexpr int  M   = VAL ? 4 * NC : 3 * NC;
  static constexpr int  DS  = SYM ? M * (M + 1) / 2 : M * M;
  static constexpr int  VO  = VAL ? NC : 0;  // offset of the gradient inputs
  __host__ __device__ static constexpr int idx(int r, int s) { return SYM ? packed_index(r, s) : s * M + r; }
  __host__ __device__ static constexpr int rows(int s) { return SYM ? s + 1 : M; }
};

// Workgroups are dispatched round-robin over the 8 XCDs (block b -> XCD b % 8).
// With remap on, XCD x instead works through a contiguous run of logical
// blocks, so neighbouring elements (which share nodes) hit the same L2.
__device__ __forceinline__ int64_t logical_block(int remap)
{
  const int64_t b = blockIdx.x, G = gridDim.x;
  if (!remap) return b;
  const int64_t per = G / 8;
  if (b >= per * 8) return b;
  return (b % 8) * per + b / 8;
}

// Workgroup barrier that orders LDS only.  __syncthreads() also fences global
// memory, which makes every wave drain its outstanding global loads (vmcnt 0)
// at each barrier; the stages here exchange data through LDS alone, so the
// stored-tangent stream may stay in flight across the barriers.
__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Cross-lane reads within a wave (DPP): quad_bcast<x> gives every lane the
// value of lane x of its group of 4 lanes; row_ror<k> the value of the lane k
// places away (cyclically) within its row of 16 lanes.  With one p = 3 element
// per wave and lane = (i2 N + i1) N + i0, a quad holds one x line of nodes or
// points and a row one z layer, so the x and y contractions need no LDS.
// Every lane reads a valid source lane under these controls, so the moves
// carry no old value (no zeroing move ahead of each).
template <int X>
__device__ __forceinline__ float quad_bcast(float v)
{
  static_assert(X >= 0 && X < 4, "lane in a quad");
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), X * 0x55, 0xf, 0xf, true));
}
template <int K>
__device__ __forceinline__ float row_ror(float v)
{
  static_assert(K >= 1 && K < 16, "rotation within a row");
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x120 + K, 0xf, 0xf, true));
}
template <int X>
__device__ __forceinline__ double quad_bcast(double v)
{
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), X * 0x55, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), X * 0x55, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
template <int K>
__device__ __forceinline__ double row_ror(double v)
{
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x120 + K, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x120 + K, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
template <int K>
__device__ __forceinline__ int row_ror_i(int v)
{
  static_assert(K >= 1 && K < 16, "rotation within a row");
  return __builtin_amdgcn_mov_dpp(v, 0x120 + K, 0xf, 0xf, true);
}

template <typename T>
__device__ __forceinline__ void scatter_add(T* r, int64_t o, T v, int atomic)
{
  if (atomic)
    unsafeAtomicAdd(r + o, v);
  else
    r[o] += v;
}

__device__ __forceinline__ int64_t lidx(int64_t node, int c, int nc, int64_t nnodes, int ordering)
{
  return ordering ? node * nc + c : int64_t(c) * nnodes + node;
}

// SCATTER_ELEMENT: the element's values as one run of consecutive addresses,
// through LDS (sv: NC * NQ values).  Every lane of the workgroup calls it (it
// holds a barrier).
template <int N, int NC, typename T>
__device__ __forceinline__ void store_element(void* E, const T* acc, T* sv, int64_t slot, int li, bool active)
{
  constexpr int NQ = N * N * N;
  if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) sv[li * NC + c] = acc[c];
  }
  lds_barrier();
  if (active) {
    T* Ee = static_cast<T*>(E) + size_t(slot) * (NC * NQ) + li;
#pragma unroll
    for (int t = 0; t < NC; t++) Ee[t * NQ] = sv[t * NQ + li];
  }
}

// Scatter-add of one element's NC x NQ nodal values in address order.  Lane li
// of the element holds acc[c] for its node li; the values and node ids go
// through LDS (sv: the element's NC * NQ values, sn: the workgroup's node ids,
// NQ per element), then pass t of the element's NQ lanes adds entries
// t NQ .. t NQ + NQ - 1 of the element's (node, component) list, node-major for
// byVDIM and component-major for byNODES: one wave instruction then covers
// whole rows of consecutive addresses (a structured mesh numbers the nodes of
// an element row consecutively) instead of one component at a 3-entry stride,
// which cuts the memory transactions of the adds about threefold.
// With merge, the nodes an element shares with the previous element of the
// workgroup across its i0 = 0 face (consecutive elements along x) are added
// into that element's values in LDS first and skipped in the passes: one add
// per shared node and workgroup instead of two.  Every lane of the workgroup
// calls it (it holds barriers); sv_prev is the previous element's sv.
template <int N, int NC, typename T, typename V>
__device__ __forceinline__ void scatter_element(V* r, const T* acc, T* sv, T* sv_prev, int* sn_wg, int el, int eb,
                                                int64_t node, int li, bool active, int64_t nnodes, int ordering,
                                                int atomic, bool merge)
{
  constexpr int NQ = N * N * N;
  int*          sn = sn_wg + (el < eb ? el : 0) * NQ;  // lanes past the workgroup's elements touch nothing
  if (el < eb) {
    if (active) {
#pragma unroll
      for (int c = 0; c < NC; c++) sv[ordering ? li * NC + c : c * NQ + li] = acc[c];
    }
    sn[li] = active ? int(node) : -1;
  }
  lds_barrier();
  if (merge) {
    const int i0 = li % N;
    if (active && el > 0 && i0 == 0) {
      const int jp = li + (N - 1);  // (N - 1, i1, i2) of the previous element
      if (sn_wg[(el - 1) * NQ + jp] == int(node)) {
#pragma unroll
        for (int c = 0; c < NC; c++) sv_prev[ordering ? jp * NC + c : c * NQ + jp] += acc[c];
        sn[li] = -1;
      }
    }
    lds_barrier();
  }
  if (active) {
#pragma unroll
    for (int t = 0; t < NC; t++) {
      const int f  = t * NQ + li;
      const int j  = ordering ? f / NC : li;
      const int c  = ordering ? f - j * NC : t;
      const int nd = sn[j];
      if (nd >= 0) scatter_add(r, lidx(nd, c, NC, nnodes, ordering), V(sv[f]), atomic);
    }
  }
}

// Jacobian of the trilinear map at parent point xi from the 8 corner
// coordinates X[corner][3] (corner = a + 2b + 4c lexicographic):
// J[i][j] = d x_i / d xi_j  (fn/geometric_factors.cpp:17-58 interpolates the
// same order-1 nodes).
__device__ __forceinline__ void trilinear_jacobian(const double* X, double x0, double x1, double x2, double* J)
{
#pragma unroll
  for (int k = 0; k < 9; k++) J[k] = 0.0;
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const int    a = c & 1, b = (c >> 1) & 1, d = (c >> 2) & 1;
    const double N0 = a ? x0 : 1.0 - x0, N1 = b ? x1 : 1.0 - x1, N2 = d ? x2 : 1.0 - x2;
    const double D0 = a ? 1.0 : -1.0, D1 = b ? 1.0 : -1.0, D2 = d ? 1.0 : -1.0;
    const double g0 = D0 * N1 * N2, g1 = N0 * D1 * N2, g2 = N0 * N1 * D2;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const double xi = X[c * 3 + i];
      J[i * 3 + 0] += xi * g0;
      J[i * 3 + 1] += xi * g1;
      J[i * 3 + 2] += xi * g2;
    }
  }
}

// The value v as the compiler cannot connect it with its origin: what is
// computed from it afterwards is not merged with earlier expressions.
__device__ __forceinline__ void opaque(double& v) { asm volatile("" : "+v"(v)); }

// grad_x = grad_xi inv(J)
template <int NC>
__device__ __forceinline__ void physical_gradient(const double* gp, const double* Ji, double* g)
{
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int k = 0; k < 3; k++)
      g[c * 3 + k] = gp[c * 3 + 0] * Ji[0 * 3 + k] + gp[c * 3 + 1] * Ji[1 * 3 + k] + gp[c * 3 + 2] * Ji[2 * 3 + k];
}

// Quadrature-point stage of the residual / linearization: parent-space
// (value, grad) in, parent-space (source, flux) out, following
// fn/finite_element.hpp:246-322: grad_x = grad_xi inv(J); source *= detJ;
// flux_parent[c][j] = detJ sum_k flux[c][k] inv(J)[j][k].
template <class QF, int NC>
__device__ __forceinline__ void qpoint_eval(const double* prm, const double* Ji, double dJ, const double* val,
                                            const double* gp, double* src, double* fp, double* st)
{
  double g[3 * NC], s[NC], f[3 * NC];
  physical_gradient<NC>(gp, Ji, g);
#pragma unroll
  for (int c = 0; c < NC; c++) s[c] = 0.0;
  if constexpr (QF::STATE > 0)
    QF::eval(prm, val, g, s, f, st);
  else
    QF::eval(prm, val, g, s, f);
#pragma unroll
  for (int c = 0; c < NC; c++) {
    src[c] = s[c] * dJ;
#pragma unroll
    for (int j = 0; j < 3; j++)
      fp[c * 3 + j] = (f[c * 3 + 0] * Ji[j * 3 + 0] + f[c * 3 + 1] * Ji[j * 3 + 1] + f[c * 3 + 2] * Ji[j * 3 + 2]) * dJ;
  }
}

// Directional derivative of the quadrature-point stage with respect to the
// shape: the Jacobian J = dX/dxi + dp/dxi moves by dJ = d(dp)/dxi, and
// inv(J), det(J), grad_x u = grad_xi u inv(J), the qfunction and the
// transformation of its source and flux are carried as one-direction duals
// (fn/shape_aware_functional.hpp:37-125 differentiated in p).  src and fp get
// the derivative parts.  The point's state enters as a copy (nothing is
// committed).
template <class QF, int NC>
__device__ __forceinline__ void qpoint_shape_dir(const double* prm, const double* J, const double* dJdir,
                                                 const double* val, const double* gp, const double* st0,
                                                 double* src, double* fp)
{
  d1 Jd[9], Jid[9];
#pragma unroll
  for (int k = 0; k < 9; k++) Jd[k] = d1(J[k], dJdir[k]);
  inv3(Jd, Jid);
  const d1 dJd = det3(Jd);
  d1       v[NC], g[3 * NC], s[NC], f[3 * NC];
#pragma unroll
  for (int c = 0; c < NC; c++) v[c] = d1(val[c]);
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int k = 0; k < 3; k++)
      g[c * 3 + k] = gp[c * 3 + 0] * Jid[0 * 3 + k] + gp[c * 3 + 1] * Jid[1 * 3 + k] + gp[c * 3 + 2] * Jid[2 * 3 + k];
#pragma unroll
  for (int c = 0; c < NC; c++) s[c] = d1(0.0);
  if constexpr (QF::STATE > 0) {
    double st[QF::STATE];
#pragma unroll
    for (int k = 0; k < QF::STATE; k++) st[k] = st0[k];
    QF::eval(prm, v, g, s, f, st);
  } else {
    QF::eval(prm, v, g, s, f);
  }
#pragma unroll
  for (int c = 0; c < NC; c++) {
    src[c] = (s[c] * dJd).d;
#pragma unroll
    for (int j = 0; j < 3; j++)
      fp[c * 3 + j] = ((f[c * 3 + 0] * Jid[j * 3 + 0] + f[c * 3 + 1] * Jid[j * 3 + 1] + f[c * 3 + 2] * Jid[j * 3 + 2]) * dJd).d;
  }
}

// Loads the DS tangent entries of quadrature point q as T.
template <typename T, typename S, int DS, int NQ>
__device__ __forceinline__ void load_tangent(const void* base, int q, T* Dr)
{
  using L = TangentLayout<S, DS, NQ>;
  // native vector types per storage type: a 16-byte integer vector
  // reassembled into doubles gets split by the back end into a 16-byte load
  // plus a second, 8-byte load of the same address
  typedef unsigned int u4 __attribute__((ext_vector_type(4)));
  typedef double       d2 __attribute__((ext_vector_type(2)));
  typedef float        f4 __attribute__((ext_vector_type(4)));
  const S* Dp = static_cast<const S*>(base);
#pragma unroll
  for (int g = 0; g < L::G; g++) {
    const S* gp = Dp + g * L::VEC * NQ + q * L::VEC;
    if constexpr (sizeof(S) == 8) {
      const d2 v    = __builtin_nontemporal_load(reinterpret_cast<const d2*>(gp));
      Dr[2 * g]     = T(v.x);
      Dr[2 * g + 1] = T(v.y);
    } else if constexpr (sizeof(S) == 4) {
      const f4 v    = __builtin_nontemporal_load(reinterpret_cast<const f4*>(gp));
      Dr[4 * g]     = T(v.x);
      Dr[4 * g + 1] = T(v.y);
      Dr[4 * g + 2] = T(v.z);
      Dr[4 * g + 3] = T(v.w);
    } else {
      const u4 v = __builtin_nontemporal_load(reinterpret_cast<const u4*>(gp));
      const unsigned int w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        Dr[8 * g + 2 * i]     = T(__uint_as_float(w[i] << 16));
        Dr[8 * g + 2 * i + 1] = T(__uint_as_float(w[i] & 0xffff0000u));
      }
    }
  }
#pragma unroll
  for (int j = 0; j < L::REM; j++) {
    const auto raw = __builtin_nontemporal_load(
        reinterpret_cast<const typename StoreTraits<S>::raw*>(Dp + L::offset(L::G * L::VEC + j, q)));
    if constexpr (sizeof(S) == 2)
      Dr[L::G * L::VEC + j] = T(bf16_to_float(uint32_t(raw)));
    else
      Dr[L::G * L::VEC + j] = T(raw);
  }
}

// The DS tangent entries of one quadrature point held in registers for the
// J.v chain rule: as T, or, for a BF16 tangent, still packed two to a 32-bit
// register and widened at their one use (the same conversions, half the
// registers: 25 instead of 45 for the Neo-Hookean tangent, which lets more
// waves share a SIMD).  get(k) needs a compile-time k after unrolling.
template <typename T, typename S, int DS, int NQ>
struct TangentRegs {
  T d[DS];
  __device__ __forceinline__ void load(const void* base, int q) { load_tangent<T, S, DS, NQ>(base, q, d); }
  __device__ __forceinline__ T    get(int k) const { return d[k]; }
};
template <typename T, int DS, int NQ>
struct TangentRegs<T, bf16, DS, NQ> {
  using L = TangentLayout<bf16, DS, NQ>;
  static constexpr int K0 = L::G * L::VEC;  // first remainder entry
  static constexpr int NW = L::G * 4 + L::RP;
  uint32_t w[NW > 0 ? NW : 1];  // entries 2i, 2i + 1 as word i (low half first): the groups, then the remainder pairs
  float    last;                // an odd last entry, widened on load
  __device__ __forceinline__ void load(const void* base, int q)
  {
    typedef unsigned int u4 __attribute__((ext_vector_type(4)));
    const bf16* Dp = static_cast<const bf16*>(base);
#pragma unroll
    for (int g = 0; g < L::G; g++) {
      const u4 v   = __builtin_nontemporal_load(reinterpret_cast<const u4*>(Dp + g * L::VEC * NQ + q * L::VEC));
      w[4 * g]     = v.x;
      w[4 * g + 1] = v.y;
      w[4 * g + 2] = v.z;
      w[4 * g + 3] = v.w;
    }
#pragma unroll
    for (int p = 0; p < L::RP; p++)
      w[4 * L::G + p] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(Dp + L::offset(K0 + 2 * p, q)));
    if constexpr (L::REM % 2 == 1)
      last = bf16_to_float(
          uint32_t(__builtin_nontemporal_load(reinterpret_cast<const uint16_t*>(Dp + L::offset(DS - 1, q)))));
    else
      last = 0.0f;
  }
  __device__ __forceinline__ T get(int k) const
  {
    if (L::REM % 2 == 1 && k == DS - 1) return T(last);
    const uint32_t x = w[k / 2];  // groups and remainder pairs alike: word k / 2
    return T(__uint_as_float((k & 1) ? (x & 0xffff0000u) : (x << 16)));
  }
};

// Stores tangent entry k (FP64 value) of quadrature point q: entries arrive in
// increasing k; whole 16-byte groups are stored at once from `pend`.  The stores
// bypass the caches, except where a long tangent (78 entries) meets groups that
// fill no whole cache lines (p = 2, 4).  Bypassing and not, mass-diffusion of
// three components: FP64 p = 2 on 48x47x49 elements 718 and 507 us, p = 4 on
// 28x27x29 445 and 416; FP32 p = 2 339 and 270, but p = 4 229 and 254; BF16
// p = 2 164 and 219.  Shorter tangents: Neo-Hookean p = 3 on 36x35x37 244 and
// 328, p = 2 328 and 355.
template <typename S, int DS, int NQ>
__device__ __forceinline__ void store_tangent_entry(void* base, int q, int k, double v,
                                                    typename StoreTraits<S>::raw* pend)
{
  using L   = TangentLayout<S, DS, NQ>;
  using raw = typename StoreTraits<S>::raw;
  raw* Dp   = static_cast<raw*>(base);
  auto put  = [](auto x, auto* at) {
    if constexpr (DS == 78 && ((sizeof(S) == 8 && NQ % 2 == 1) || (sizeof(S) == 4 && NQ == 27)))
      *at = x;
    else
      __builtin_nontemporal_store(x, at);
  };
  if (k < L::G * L::VEC) {
    pend[k % L::VEC] = raw(to_store(v, static_cast<S*>(nullptr)));
    if (k % L::VEC == L::VEC - 1) {
      typedef unsigned int u4 __attribute__((ext_vector_type(4)));
      u4 w;
      __builtin_memcpy(&w, pend, 16);
      put(w, reinterpret_cast<u4*>(Dp + (k / L::VEC) * L::VEC * NQ + q * L::VEC));
    }
  } else {
    put(raw(to_store(v, static_cast<S*>(nullptr))), Dp + L::offset(k, q));
  }
}

// ---------------------------------------------------------------------------
// contractions by rows
// ---------------------------------------------------------------------------
// One direction of a sum factorization on an element's [component][z][y][x]
// array in LDS: a lane owns whole rows along that direction, so it reads N
// values, forms all N results (for each table that applies) and writes them
// back in their place.  The table entries are then the same for every lane and
// compile-time offsets from a kernel argument: scalar loads and scalar
// operands, no LDS reads.  With a lane per result instead, each result cost N
// value reads and N table reads through the one LDS port of a CU.  Neo-Hookean
// residual p = 2 on 57x48x43: 148 -> 120 us of kernel time; p = 3 on 64^3: 735
// -> 682; its vector instructions (891 a point, 684 of them FP64) fill two thirds
// of the cycles.
// One component has N * N rows for N^3 lanes and stays with a lane per result
// (use_rows): heat residual p = 3 on 36x35x37 elements 84 us by rows and 67 so,
// p = 1 on 80x79x81 91 and 73 (both with the fill of the output).
template <int N, int NC>
struct Rows {
  static constexpr int NQ = N * N * N, COUNT = NC * N * N, ITER = (COUNT + NQ - 1) / NQ;
  static constexpr int STRIDE[3] = {1, N, N * N};
  // first entry of row r along `dir`, stride STRIDE[dir]
  __device__ __forceinline__ static int base(int dir, int r)
  {
    const int c = r / (N * N), k = r % (N * N);
    return c * NQ + (dir == 0 ? k * N : dir == 1 ? (k / N) * N * N + k % N : k);
  }
};
template <typename T>
using ScalarPtr = const __attribute__((address_space(4))) T*;  // read by scalar loads
using ScalarTable = ScalarPtr<double>;

// f(first entry) for every row along DIR that lane li of an active element owns
template <int N, int NC, int DIR, class F>
__device__ __forceinline__ void for_rows(int li, bool active, F&& f)
{
  using R = Rows<N, NC>;
#pragma unroll
  for (int it = 0; it < R::ITER; it++) {
    const int r = li + it * R::NQ;
    if (active && r < R::COUNT) f(R::base(DIR, r));
  }
}
template <int N, int STRIDE, typename T>
__device__ __forceinline__ void read_row(const T* a, T* v)
{
#pragma unroll
  for (int i = 0; i < N; i++) v[i] = a[i * STRIDE];
}
// out[q] (+)= sum_i tab[q][i] v[i]
template <int N, typename T>
__device__ __forceinline__ void row_forward(ScalarPtr<T> tab, const T* v, T* out, bool add = false)
{
#pragma unroll
  for (int q = 0; q < N; q++) {
    T s = add ? out[q] : T(0);
#pragma unroll
    for (int i = 0; i < N; i++) s += tab[q * N + i] * v[i];
    out[q] = s;
  }
}
// out[i] (+)= sum_q tab[q][i] v[q]
template <int N, typename T>
__device__ __forceinline__ void row_transposed(ScalarPtr<T> tab, const T* v, T* out, bool add = false)
{
#pragma unroll
  for (int i = 0; i < N; i++) {
    T s = add ? out[i] : T(0);
#pragma unroll
    for (int q = 0; q < N; q++) s += tab[q * N + i] * v[q];
    out[i] = s;
  }
}
// out[i] = sum_q (ta[q][i] v[q] + tb[q][i] w[q]), a pair at a time
template <int N, typename T>
__device__ __forceinline__ void row_transposed_pair(ScalarPtr<T> ta, const T* v, ScalarPtr<T> tb, const T* w, T* out)
{
#pragma unroll
  for (int i = 0; i < N; i++) {
    T s = T(0);
#pragma unroll
    for (int q = 0; q < N; q++) s += v[q] * ta[q * N + i] + w[q] * tb[q * N + i];
    out[i] = s;
  }
}
template <int N, int STRIDE, typename T>
__device__ __forceinline__ void write_row(T* a, const T* v)
{
#pragma unroll
  for (int i = 0; i < N; i++) a[i * STRIDE] = v[i];
}
template <int NC>
constexpr bool use_rows()
{
  return NC > 1;
}

// A lane per result: sum_i tab[i * TS] a[i * AS], N table entries and N values
// from LDS
template <int N, int TS, int AS, typename T>
__device__ __forceinline__ T dot_result(const T* tab, const T* a)
{
  T s = T(0);
#pragma unroll
  for (int i = 0; i < N; i++) s += tab[i * TS] * a[i * AS];
  return s;
}

// ---------------------------------------------------------------------------
// residual (MODE_RESIDUAL) and linearization (MODE_LINEARIZE, tangent in S)
// ---------------------------------------------------------------------------
// Waves per SIMD that the register allocation aims at, and the most of them.
// The J2 linearization would take 278 registers (one wave); held to two waves it
// spills nothing.  A vector residual spills 6 to 9 at five waves, 20 where it
// also carries the value.  The linearization of a constant tangent does little
// but store it, and at p = 1, 2, where an element's groups are short, it stores
// faster with fewer waves in flight: linear elasticity p = 1 on 80x79x81
// elements 358 us of kernel time at four waves, 300 at two; p = 2 on 48x47x49
// 320 and, at three, 305; mass-diffusion p = 2 490 and 425.  At p = 3, 4 four
// waves are faster (p = 3 on 36x35x37 elastic 200 us against 235).
template <int N, int NC, int MODE, class QF, typename S>
constexpr int element_max_waves()
{
  if (MODE == MODE_LINEARIZE && NC == 3 && N <= 3 && QF::CONSTANT_TANGENT) return N;
  return 8;
}
template <int N, int NC, int MODE, class QF, typename S>
constexpr int element_min_waves()
{
  constexpr int most = element_max_waves<N, NC, MODE, QF, S>();
  if (most < 8) return most;
  if (QF::STATE > 0) return MODE == MODE_LINEARIZE ? 2 : 3;
  if (NC == 1) return MODE == MODE_LINEARIZE && sizeof(S) == 2 ? 4 : 7;
  return MODE != MODE_RESIDUAL || QF::USES_VALUE ? 4 : 5;
}

template <int N, int NC, int MODE, class QF, int LAYOUT, typename S>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu((element_min_waves<N, NC, MODE, QF, S>()),
                                       (element_max_waves<N, NC, MODE, QF, S>()))))
    k_element(const ElemLaunch P)
{
  constexpr int  NQ      = N * N * N;
  constexpr int  NN      = N * N;
  constexpr int  EB      = 256 / NQ;
  using Shape            = TanShape<LAYOUT, NC>;
  constexpr bool HAS_SRC = QF::HAS_SOURCE;
  constexpr int  DS      = Shape::DS;
  constexpr int  NST     = QF::STATE;
  constexpr bool ROWS    = use_rows<NC>();
  constexpr int  R       = NC * NQ;  // one LDS region
  constexpr int  REGIONS = ROWS ? 3 + (HAS_SRC || QF::USES_VALUE ? 1 : 0) : 6 + (HAS_SRC ? 1 : 0);
  // elements of a wave (eight at p = 1) start in different LDS banks
  constexpr int  PER     = REGIONS * R + (REGIONS * R % 32 == 0 ? 8 : 0);
  using Lay              = TangentLayout<S, DS, NQ>;

  __shared__ double smem[EB * PER];
  __shared__ double stab[ROWS ? 1 : 4 * NN];  // B, G, and both times the weights
  __shared__ double sxw[2 * N];               // Gauss points and weights
  __shared__ double sxv[EB * 24];
  __shared__ int    snode[EB * NQ];

  const int     tid    = threadIdx.x;
  const int     el     = tid / NQ;
  const int     li     = tid - el * NQ;
  const int     i0     = li % N;
  const int     i1     = (li / N) % N;
  const int     i2     = li / NN;
  const int64_t slot   = P.slot_begin + logical_block(P.xcd_remap) * EB + el;
  const bool    active = (el < EB) && (slot < P.slot_end);
  double*       S0     = smem + (el < EB ? el : 0) * PER;
  double *      S1 = S0 + R, *S2 = S0 + 2 * R, *S3 = S0 + 3 * R;  // S3 only where PER has it
  double*       r = static_cast<double*>(P.r);

  if constexpr (!ROWS)
    for (int k = tid; k < 4 * NN; k += blockDim.x) stab[k] = P.tables[k];
  if (tid < 2 * N) sxw[tid] = P.tables[4 * NN + tid];
  const ScalarTable tB = (ScalarTable)(uintptr_t)P.tables;
  const ScalarTable tG = tB + NN;

  // ---- quadrature-point state (issued first, consumed at the qfunction)
  double  st[NST > 0 ? NST : 1];
  double* stp = nullptr;
  if constexpr (NST > 0) {
    if (active) {
      stp = P.qdata + size_t(P.qrow[slot]) * NST * NQ + li;
#pragma unroll
      for (int k = 0; k < NST; k++) st[k] = stp[k * NQ];
    }
  }
  int64_t node = active ? P.map[size_t(slot) * NQ + li] : 0;
  double  nodal[NC];  // this lane's node
  auto    gather = [&](const double* field) {
    if (active) {
#pragma unroll
      for (int c = 0; c < NC; c++) nodal[c] = field[lidx(node, c, NC, P.nnodes, P.ordering)];
    }
  };
  // (a point's state goes first: J2 p = 2 on 56x48x50, linearize + diagonal + J.v, 1314 us against 1333)
  if constexpr (NST == 0) gather(static_cast<const double*>(P.u));
  if (active)
    for (int k = li; k < 24; k += NQ) sxv[el * 24 + k] = P.coords[size_t(slot) * 24 + k];
  if constexpr (NST > 0) gather(static_cast<const double*>(P.u));

  // Parent gradient (and value) at this lane's point of the gathered field:
  // x, y and z in turn.  Every lane calls it; the regions (with a lane per
  // result, the first three) are free again after it.
  auto interpolate = [&](double* val, double* gp) {
    if (active) {
#pragma unroll
      for (int c = 0; c < NC; c++) S0[c * NQ + li] = nodal[c];
    }
    lds_barrier();
    if constexpr (!ROWS) {
      const int     oy = i2 * NN + i0, oz = i1 * N + i0;  // first entries of the lane's lines along y and z
      const double *sB = stab, *sG = stab + NN;
      // (results first, stores after: a line and a table row are then read once)
      if (active) {
        const double b = dot_result<N, 1, 1>(sB + i0 * N, S0 + li - i0);
        const double g = dot_result<N, 1, 1>(sG + i0 * N, S0 + li - i0);
        S1[li]         = b;
        S2[li]         = g;
      }
      lds_barrier();
      if (active) {
        const double bb = dot_result<N, 1, N>(sB + i1 * N, S1 + oy);
        const double bg = dot_result<N, 1, N>(sB + i1 * N, S2 + oy);
        const double gb = dot_result<N, 1, N>(sG + i1 * N, S1 + oy);
        S3[li]          = bb;
        S3[NQ + li]     = bg;
        S3[2 * NQ + li] = gb;
      }
      lds_barrier();
      if (active) {
        gp[0] = dot_result<N, 1, NN>(sB + i2 * N, S3 + NQ + oz);
        gp[1] = dot_result<N, 1, NN>(sB + i2 * N, S3 + 2 * NQ + oz);
        gp[2] = dot_result<N, 1, NN>(sG + i2 * N, S3 + oz);
        if constexpr (QF::USES_VALUE) val[0] = dot_result<N, 1, NN>(sB + i2 * N, S3 + oz);
      }
    } else {
      for_rows<N, NC, 0>(li, active, [&](int o) {  // u -> B u, G u
        double v[N], a[N], b[N];
        read_row<N, 1>(S0 + o, v);
        row_forward<N>(tB, v, a);
        row_forward<N>(tG, v, b);
        write_row<N, 1>(S0 + o, a);
        write_row<N, 1>(S1 + o, b);
      });
      lds_barrier();
      for_rows<N, NC, 1>(li, active, [&](int o) {  // -> BB, BG (y, x), GB
        double v[N], w[N], a[N];
        read_row<N, N>(S0 + o, v);
        read_row<N, N>(S1 + o, w);
        row_forward<N>(tB, v, a);
        write_row<N, N>(S0 + o, a);
        row_forward<N>(tB, w, a);
        write_row<N, N>(S1 + o, a);
        row_forward<N>(tG, v, a);
        write_row<N, N>(S2 + o, a);
      });
      lds_barrier();
      for_rows<N, NC, 2>(li, active, [&](int o) {  // -> d/dx in S1, d/dy in S2, d/dz in S0, value in S3
        double v[N], a[N];
        read_row<N, NN>(S1 + o, v);
        row_forward<N>(tB, v, a);
        write_row<N, NN>(S1 + o, a);
        read_row<N, NN>(S2 + o, v);
        row_forward<N>(tB, v, a);
        write_row<N, NN>(S2 + o, a);
        read_row<N, NN>(S0 + o, v);
        row_forward<N>(tG, v, a);
        write_row<N, NN>(S0 + o, a);
        if constexpr (QF::USES_VALUE) {
          row_forward<N>(tB, v, a);
          write_row<N, NN>(S3 + o, a);
        }
      });
      lds_barrier();
      if (active) {
#pragma unroll
        for (int c = 0; c < NC; c++) {
          gp[c * 3 + 0] = S1[c * NQ + li];
          gp[c * 3 + 1] = S2[c * NQ + li];
          gp[c * 3 + 2] = S0[c * NQ + li];
          if constexpr (QF::USES_VALUE) val[c] = S3[c * NQ + li];
        }
      }
      lds_barrier();
    }
  };

  double val[NC], gp[3 * NC];
#pragma unroll
  for (int c = 0; c < NC; c++) val[c] = 0.0;
  interpolate(val, gp);
  // ---- shape displacement (ShapeAwareFunctional, fn/shape_aware_functional.hpp:37-50):
  // the parent gradient of p at this lane's quadrature point, added to the
  // geometric Jacobian below, so dx/dxi = dX/dxi + dp/dxi = (I + dp/dX) dX/dxi.
  // P.shape is the same for every lane, so the barriers inside are uniform.
  double gps[9], dgps[9];
#pragma unroll
  for (int k = 0; k < 9; k++) gps[k] = dgps[k] = 0.0;
  if constexpr (NC == 3) {
    double unused[NC];
    if (P.shape != nullptr) {
      gather(P.shape);
      interpolate(unused, gps);
    }
    if constexpr (MODE == MODE_SHAPE_JVP) {
      gather(P.dshape);
      interpolate(unused, dgps);
    }
  }

  // ---- quadrature point
  if (active) {
    double J[9], Ji[9];
    trilinear_jacobian(sxv + el * 24, sxw[i0], sxw[i1], sxw[i2], J);
    if constexpr (NC == 3) {
#pragma unroll
      for (int k = 0; k < 9; k++) J[k] += gps[k];
    }
    inv3(J, Ji);
    // rows carry the quadrature weight in the flux, a lane per result in its tables
    const double dJ = det3(J), wq = ROWS ? sxw[N + i0] * sxw[N + i1] * sxw[N + i2] : 1.0;
    double       src[NC], fp[3 * NC];  // source and flux
    if constexpr (MODE == MODE_SHAPE_JVP) {
      qpoint_shape_dir<QF, NC>(P.params, J, dgps, val, gp, st, src, fp);
#pragma unroll
      for (int c = 0; c < NC; c++) src[c] *= wq;
#pragma unroll
      for (int k = 0; k < 3 * NC; k++) fp[k] *= wq;
    } else {
      if constexpr (MODE == MODE_LINEARIZE) {
        // the entries come in increasing storage order; the state is the one before this call
        void*                        Dp = static_cast<char*>(P.D) + size_t(slot) * Lay::stride * sizeof(S);
        typename StoreTraits<S>::raw pend[Lay::VEC];
        double                       g[3 * NC];
        physical_gradient<NC>(gp, Ji, g);
        QF::tangent(P.params, g, Ji, dJ, st, [&](int rr, int s, double v) {
          store_tangent_entry<S, DS, NQ>(Dp, li, Shape::idx(rr, s), v, pend);
        });
        if constexpr (NST > 0) {
          // eval() below starts over from its inputs: sharing the trial state with the tangent kept it in registers
          // across all 81 entries
#pragma unroll
          for (int k = 0; k < 3 * NC; k++) opaque(gp[k]);
        }
      }
      qpoint_eval<QF, NC>(P.params, Ji, dJ * wq, val, gp, src, fp, st);
      if constexpr (NST > 0) {
        // batch_apply_qf (fn/domain_integral_kernels.hpp:125-150): commit the
        // point's updated state only when asked to
        if (P.update_state) {
#pragma unroll
          for (int k = 0; k < NST; k++) stp[k * NQ] = st[k];
        }
      }
    }
#pragma unroll
    for (int c = 0; c < NC; c++) {
      S0[c * NQ + li] = fp[c * 3 + 0];
      S1[c * NQ + li] = fp[c * 3 + 1];
      S2[c * NQ + li] = fp[c * 3 + 2];
      if constexpr (HAS_SRC) S0[(ROWS ? 3 : 6) * R + c * NQ + li] = src[c];
    }
  }
  lds_barrier();

  // ---- integrate: x, y, z; lane = node in the end
  double acc[NC];
  if constexpr (!ROWS) {
    const int     oy = i2 * NN + i0, oz = i1 * N + i0;
    const double *sB = stab + 2 * NN, *sG = stab + 3 * NN;
    if (active) {
      const double* row = S0 + li - i0;
      double        a   = dot_result<N, N, 1>(sG + i0, row);
      const double  b = dot_result<N, N, 1>(sB + i0, row + R), c = dot_result<N, N, 1>(sB + i0, row + 2 * R);
      if constexpr (HAS_SRC) a += dot_result<N, N, 1>(sB + i0, row + 6 * R);
      S3[li]          = a;
      S3[NQ + li]     = b;
      S3[2 * NQ + li] = c;
    }
    lds_barrier();
    if (active) {
      const double a = dot_result<N, N, N>(sB + i1, S3 + oy) + dot_result<N, N, N>(sG + i1, S3 + NQ + oy);
      const double b = dot_result<N, N, N>(sB + i1, S3 + 2 * NQ + oy);
      S0[li]         = a;
      S1[li]         = b;
    }
    lds_barrier();
    if (active) acc[0] = dot_result<N, N, NN>(sB + i2, S0 + oz) + dot_result<N, N, NN>(sG + i2, S1 + oz);
  } else {
    for_rows<N, NC, 0>(li, active, [&](int o) {
      double v[N], a[N];
      read_row<N, 1>(S0 + o, v);
      row_transposed<N>(tG, v, a);
      if constexpr (HAS_SRC) {
        read_row<N, 1>(S3 + o, v);
        row_transposed<N>(tB, v, a, true);
      }
      write_row<N, 1>(S0 + o, a);
      read_row<N, 1>(S1 + o, v);
      row_transposed<N>(tB, v, a);
      write_row<N, 1>(S1 + o, a);
      read_row<N, 1>(S2 + o, v);
      row_transposed<N>(tB, v, a);
      write_row<N, 1>(S2 + o, a);
    });
    lds_barrier();
    for_rows<N, NC, 1>(li, active, [&](int o) {
      double v[N], a[N];
      read_row<N, N>(S0 + o, v);
      row_transposed<N>(tB, v, a);
      read_row<N, N>(S1 + o, v);
      row_transposed<N>(tG, v, a, true);
      write_row<N, N>(S0 + o, a);
      read_row<N, N>(S2 + o, v);
      row_transposed<N>(tB, v, a);
      write_row<N, N>(S1 + o, a);
    });
    lds_barrier();
    for_rows<N, NC, 2>(li, active, [&](int o) {
      double v[N], a[N];
      read_row<N, NN>(S0 + o, v);
      row_transposed<N>(tB, v, a);
      read_row<N, NN>(S1 + o, v);
      row_transposed<N>(tG, v, a, true);
      write_row<N, NN>(S2 + o, a);
    });
    lds_barrier();

    if (active) {
#pragma unroll
      for (int c = 0; c < NC; c++) acc[c] = S2[c * NQ + li];
    }
  }

  // ---- scatter-add, through a region that the last stage did not read
  constexpr int SV = ROWS ? 0 : 2 * R;
  if (P.scatter == SCATTER_ELEMENT) {
    store_element<N, NC>(P.E, acc, S0 + SV, slot, li, active);
  } else if (P.ordered) {
    scatter_element<N, NC, double, double>(r, acc, S0 + SV, smem + (el > 0 && el < EB ? el - 1 : 0) * PER + SV, snode,
                                           el, EB, node, li, active, P.nnodes, P.ordering, P.scatter, P.ordered == 2);
  } else if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) scatter_add(r, lidx(node, c, NC, P.nnodes, P.ordering), acc[c], P.scatter);
  }
}

// ---------------------------------------------------------------------------
// J.v with the stored tangent (fn/domain_integral_kernels.hpp:223-304): vectors
// and arithmetic in T, tangent stored in S
// ---------------------------------------------------------------------------
// Lanes per workgroup of k_jvp: 256, except p = 4 in FP32 arithmetic, where
// one element (125 lanes) per 128-lane workgroup measured faster (FP32 tangent
// 0.580 -> 0.574 ms, BF16 0.505 -> 0.485 ms at 48^3; FP64 and the other orders
// are faster at 256).
template <int N, typename T>
constexpr int jvp_group_lanes()
{
  return (N == 5 && sizeof(T) == 4) ? 128 : 256;
}

template <int N, int NC, int LAYOUT, typename T, typename S, typename V>
__global__ void __launch_bounds__((jvp_group_lanes<N, T>())) k_jvp(const ElemLaunch P)
{
  constexpr int  NQ   = N * N * N;
  constexpr int  EB   = jvp_group_lanes<N, T>() / NQ;
  using Shape         = TanShape<LAYOUT, NC>;
  constexpr bool FULL = Shape::VAL;
  constexpr int  M    = Shape::M;
  constexpr int  DS   = Shape::DS;
  constexpr int  R    = NC * NQ;
  constexpr int  PER  = (6 + (FULL ? 1 : 0)) * R;
  constexpr int  TAB  = 4 * N * N;
  using Lay           = TangentLayout<S, DS, NQ>;

  __shared__ T   smem[EB * PER];
  __shared__ T   stab[TAB];
  __shared__ int snode[EB * NQ];

  // a Krylov loop that already converged: the whole grid leaves (the flag was
  // written by an earlier kernel on the stream, so every block reads the same),
  // once the loads below are on their way, so that a running one does not wait
  // for the flag first
  const double halt = P.stop != nullptr ? *P.stop : 0.0;

  const int     tid    = threadIdx.x;
  const int     el     = tid / NQ;
  const int     li     = tid - el * NQ;
  const int     i0     = li % N;
  const int     i1     = (li / N) % N;
  const int     i2     = li / (N * N);
  const int64_t slot   = P.slot_begin + logical_block(P.xcd_remap) * EB + el;
  const bool    active = (el < EB) && (slot < P.slot_end);
  T*            S_     = smem + (el < EB ? el : 0) * PER;
  const V*      u      = static_cast<const V*>(P.u);
  V*            r      = static_cast<V*>(P.r);

  for (int k = tid; k < TAB; k += blockDim.x) stab[k] = T(P.tables[k]);
  const T* tB  = stab;
  const T* tG  = stab + N * N;
  const T* tBw = stab + 2 * N * N;
  const T* tGw = stab + 3 * N * N;

  // ---- gather loads first, then the tangent stream: memory counters retire
  // in order, so waiting for the nodal values does not wait for the tangent,
  // which stays in flight through the interpolation stages
  int64_t node = 0;
  T       ug[NC];
  if (active) {
    node = P.map[size_t(slot) * NQ + li];
#pragma unroll
    for (int c = 0; c < NC; c++) ug[c] = T(u[lidx(node, c, NC, P.nnodes, P.ordering)]);
  }
  TangentRegs<T, S, DS, NQ> Dr;
  if (active) Dr.load(static_cast<const char*>(P.D) + size_t(slot) * Lay::stride * sizeof(S), li);
  if (halt != 0.0) return;
  if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) S_[c * NQ + li] = ug[c];
  }
  lds_barrier();

  if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const T* uu = S_ + c * NQ + (i2 * N + i1) * N;
      T        s0 = T(0), s1 = T(0);
#pragma unroll
      for (int x = 0; x < N; x++) {
        s0 += tB[i0 * N + x] * uu[x];
        s1 += tG[i0 * N + x] * uu[x];
      }
      S_[1 * R + c * NQ + li] = s0;
      S_[2 * R + c * NQ + li] = s1;
    }
  }
  lds_barrier();

  if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const T* a10 = S_ + 1 * R + c * NQ;
      const T* a11 = S_ + 2 * R + c * NQ;
      T        s0 = T(0), s1 = T(0), s2 = T(0);
#pragma unroll
      for (int y = 0; y < N; y++) {
        const int idx = (i2 * N + y) * N + i0;
        const T   b = tB[i1 * N + y], g = tG[i1 * N + y];
        s0 += b * a10[idx];
        s1 += b * a11[idx];
        s2 += g * a10[idx];
      }
      S_[3 * R + c * NQ + li] = s0;
      S_[4 * R + c * NQ + li] = s1;
      S_[5 * R + c * NQ + li] = s2;
    }
  }
  lds_barrier();

  if (active) {
    T in[M], out[M];
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const T* a20 = S_ + 3 * R + c * NQ;
      const T* a21 = S_ + 4 * R + c * NQ;
      const T* a22 = S_ + 5 * R + c * NQ;
      T        v = T(0), g0 = T(0), g1 = T(0), g2 = T(0);
#pragma unroll
      for (int z = 0; z < N; z++) {
        const int idx = (z * N + i1) * N + i0;
        const T   b = tB[i2 * N + z], g = tG[i2 * N + z];
        if constexpr (FULL) v += b * a20[idx];
        g0 += b * a21[idx];
        g1 += b * a22[idx];
        g2 += g * a20[idx];
      }
      if constexpr (FULL) in[c] = v;
      in[(FULL ? NC : 0) + c * 3 + 0] = g0;
      in[(FULL ? NC : 0) + c * 3 + 1] = g1;
      in[(FULL ? NC : 0) + c * 3 + 2] = g2;
    }
    // chain rule with the stored symmetric tangent (fn/tensor.hpp:1791-1869)
#pragma unroll
    for (int k = 0; k < M; k++) out[k] = T(0);
#pragma unroll
    for (int s = 0; s < M; s++)
#pragma unroll
      for (int rr = 0; rr < Shape::rows(s); rr++) {
        const T Dk = Dr.get(Shape::idx(rr, s));
        out[rr] += Dk * in[s];
        if (Shape::SYM && rr != s) out[s] += Dk * in[rr];
      }
#pragma unroll
    for (int c = 0; c < NC; c++) {
#pragma unroll
      for (int d = 0; d < 3; d++) S_[(c * 3 + d) * NQ + li] = out[(FULL ? NC : 0) + c * 3 + d];
      if constexpr (FULL) S_[6 * R + c * NQ + li] = out[c];
    }
  }
  lds_barrier();

  if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const T* f0 = S_ + (c * 3 + 0) * NQ;
      const T* f1 = S_ + (c * 3 + 1) * NQ;
      const T* f2 = S_ + (c * 3 + 2) * NQ;
      const T* sr = S_ + 6 * R + c * NQ;
      T        s0 = T(0), s1 = T(0), s2 = T(0);
#pragma unroll
      for (int qx = 0; qx < N; qx++) {
        const int q  = (i2 * N + i1) * N + qx;
        const T   bw = tBw[qx * N + i0], gw = tGw[qx * N + i0];
        if constexpr (FULL) s0 += sr[q] * bw;
        s0 += f0[q] * gw;
        s1 += f1[q] * bw;
        s2 += f2[q] * bw;
      }
      S_[3 * R + c * NQ + li] = s0;
      S_[4 * R + c * NQ + li] = s1;
      S_[5 * R + c * NQ + li] = s2;
    }
  }
  lds_barrier();

  if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const T* a20 = S_ + 3 * R + c * NQ;
      const T* a21 = S_ + 4 * R + c * NQ;
      const T* a22 = S_ + 5 * R + c * NQ;
      T        s0 = T(0), s1 = T(0);
#pragma unroll
      for (int qy = 0; qy < N; qy++) {
        const int idx = (i2 * N + qy) * N + i0;
        const T   bw = tBw[qy * N + i1], gw = tGw[qy * N + i1];
        s0 += a20[idx] * bw + a21[idx] * gw;
        s1 += a22[idx] * bw;
      }
      S_[0 * R + c * NQ + li] = s0;
      S_[1 * R + c * NQ + li] = s1;
    }
  }
  lds_barrier();

  T acc[NC];
  if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const T* a10 = S_ + 0 * R + c * NQ;
      const T* a11 = S_ + 1 * R + c * NQ;
      acc[c]       = T(0);
#pragma unroll
      for (int qz = 0; qz < N; qz++) {
        const int idx = (qz * N + i1) * N + i0;
        acc[c] += a10[idx] * tBw[qz * N + i2] + a11[idx] * tGw[qz * N + i2];
      }
    }
  }
  if (P.scatter == SCATTER_ELEMENT) {
    store_element<N, NC>(P.E, acc, S_ + 2 * R, slot, li, active);
  } else if (P.ordered) {
    scatter_element<N, NC, T, V>(r, acc, S_ + 2 * R, smem + (el > 0 && el < EB ? el - 1 : 0) * PER + 2 * R, snode,
                                 el, EB, node, li, active, P.nnodes, P.ordering, P.scatter, P.ordered == 2);
  } else if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) scatter_add(r, lidx(node, c, NC, P.nnodes, P.ordering), V(acc[c]), P.scatter);
  }
}

// J.v in FP32 arithmetic with the contractions by rows (see Rows), the stages
// otherwise those of k_jvp (and its pairs of products where two fields meet):
// half the LDS traffic, which bounds the BF16 tangent.  Three components and
// p = 2, 4 (use_jvp_rows): Neo-Hookean, BF16 tangent, p = 4 36^3 188 -> 163 us,
// p = 2 64^3 188 -> 168; FP32 tangents are bound by memory and stay within 1 %
// (p = 2 64^3 268 -> 260).  With one component the rows fill a fifth to a third
// of the lanes (heat p = 4: 104 -> 109), at p = 1 they take two turns
// (mass-diffusion 105 -> 115): k_jvp there.
template <int N, int NC>
constexpr bool use_jvp_rows()
{
  return NC == 3 && N != 2;
}

template <int N, int NC, int LAYOUT, typename S, typename V>
__global__ void __launch_bounds__((jvp_group_lanes<N, float>())) k_jvp_rows(const ElemLaunch P)
{
  using T             = float;
  constexpr int  NQ   = N * N * N;
  constexpr int  NN   = N * N;
  constexpr int  EB   = jvp_group_lanes<N, T>() / NQ;
  using Shape         = TanShape<LAYOUT, NC>;
  constexpr bool FULL = Shape::VAL;
  constexpr int  M    = Shape::M;
  constexpr int  DS   = Shape::DS;
  constexpr int  VO   = Shape::VO;
  constexpr int  R    = NC * NQ;
  constexpr int  PER  = (3 + (FULL ? 1 : 0)) * R;
  using Lay           = TangentLayout<S, DS, NQ>;

  __shared__ T   smem[EB * PER];
  __shared__ int snode[EB * NQ];

  const double  halt   = P.stop != nullptr ? *P.stop : 0.0;  // as in k_jvp
  const int     tid    = threadIdx.x;
  const int     el     = tid / NQ;
  const int     li     = tid - el * NQ;
  const int64_t slot   = P.slot_begin + logical_block(P.xcd_remap) * EB + el;
  const bool    active = (el < EB) && (slot < P.slot_end);
  T*            S0     = smem + (el < EB ? el : 0) * PER;
  T *           S1 = S0 + R, *S2 = S0 + 2 * R, *S3 = S0 + 3 * R;  // S3 only where PER has it
  const V*      u      = static_cast<const V*>(P.u);
  V*            r      = static_cast<V*>(P.r);

  const ScalarPtr<T> tB  = (ScalarPtr<T>)(uintptr_t)(P.tables + 7 * NN + 2 * N);
  const ScalarPtr<T> tG  = tB + NN;
  const ScalarPtr<T> tBw = tB + 2 * NN;
  const ScalarPtr<T> tGw = tB + 3 * NN;

  int64_t node = 0;
  T       ug[NC];
  if (active) {
    node = P.map[size_t(slot) * NQ + li];
#pragma unroll
    for (int c = 0; c < NC; c++) ug[c] = T(u[lidx(node, c, NC, P.nnodes, P.ordering)]);
  }
  TangentRegs<T, S, DS, NQ> Dr;
  if (active) Dr.load(static_cast<const char*>(P.D) + size_t(slot) * Lay::stride * sizeof(S), li);
  if (halt != 0.0) return;
  if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) S0[c * NQ + li] = ug[c];
  }
  lds_barrier();
  for_rows<N, NC, 0>(li, active, [&](int o) {
    T v[N], a[N], b[N];
    read_row<N, 1>(S0 + o, v);
    row_forward<N>(tB, v, a);
    row_forward<N>(tG, v, b);
    write_row<N, 1>(S0 + o, a);
    write_row<N, 1>(S1 + o, b);
  });
  lds_barrier();
  for_rows<N, NC, 1>(li, active, [&](int o) {
    T v[N], w[N], a[N];
    read_row<N, N>(S0 + o, v);
    read_row<N, N>(S1 + o, w);
    row_forward<N>(tB, v, a);
    write_row<N, N>(S0 + o, a);
    row_forward<N>(tB, w, a);
    write_row<N, N>(S1 + o, a);
    row_forward<N>(tG, v, a);
    write_row<N, N>(S2 + o, a);
  });
  lds_barrier();
  for_rows<N, NC, 2>(li, active, [&](int o) {
    T v[N], a[N];
    read_row<N, NN>(S1 + o, v);
    row_forward<N>(tB, v, a);
    write_row<N, NN>(S1 + o, a);
    read_row<N, NN>(S2 + o, v);
    row_forward<N>(tB, v, a);
    write_row<N, NN>(S2 + o, a);
    read_row<N, NN>(S0 + o, v);
    row_forward<N>(tG, v, a);
    write_row<N, NN>(S0 + o, a);
    if constexpr (FULL) {
      row_forward<N>(tB, v, a);
      write_row<N, NN>(S3 + o, a);
    }
  });
  lds_barrier();
  if (active) {
    T in[M], out[M];
#pragma unroll
    for (int c = 0; c < NC; c++) {
      if constexpr (FULL) in[c] = S3[c * NQ + li];
      in[VO + c * 3 + 0] = S1[c * NQ + li];
      in[VO + c * 3 + 1] = S2[c * NQ + li];
      in[VO + c * 3 + 2] = S0[c * NQ + li];
    }
#pragma unroll
    for (int k = 0; k < M; k++) out[k] = T(0);
#pragma unroll
    for (int s = 0; s < M; s++)
#pragma unroll
      for (int rr = 0; rr < Shape::rows(s); rr++) {
        const T Dk = Dr.get(Shape::idx(rr, s));
        out[rr] += Dk * in[s];
        if (Shape::SYM && rr != s) out[s] += Dk * in[rr];
      }
#pragma unroll
    for (int c = 0; c < NC; c++) {
      S0[c * NQ + li] = out[VO + c * 3 + 0];
      S1[c * NQ + li] = out[VO + c * 3 + 1];
      S2[c * NQ + li] = out[VO + c * 3 + 2];
      if constexpr (FULL) S3[c * NQ + li] = out[c];
    }
  }
  lds_barrier();
  for_rows<N, NC, 0>(li, active, [&](int o) {
    T v[N], a[N];
    read_row<N, 1>(S0 + o, v);
    if constexpr (FULL) {
      T w[N];
      read_row<N, 1>(S3 + o, w);
      row_transposed_pair<N>(tBw, w, tGw, v, a);
    } else {
      row_transposed<N>(tGw, v, a);
    }
    write_row<N, 1>(S0 + o, a);
    read_row<N, 1>(S1 + o, v);
    row_transposed<N>(tBw, v, a);
    write_row<N, 1>(S1 + o, a);
    read_row<N, 1>(S2 + o, v);
    row_transposed<N>(tBw, v, a);
    write_row<N, 1>(S2 + o, a);
  });
  lds_barrier();
  for_rows<N, NC, 1>(li, active, [&](int o) {
    T v[N], w[N], a[N];
    read_row<N, N>(S0 + o, v);
    read_row<N, N>(S1 + o, w);
    row_transposed_pair<N>(tBw, v, tGw, w, a);
    write_row<N, N>(S0 + o, a);
    read_row<N, N>(S2 + o, v);
    row_transposed<N>(tBw, v, a);
    write_row<N, N>(S1 + o, a);
  });
  lds_barrier();
  for_rows<N, NC, 2>(li, active, [&](int o) {
    T v[N], w[N], a[N];
    read_row<N, NN>(S0 + o, v);
    read_row<N, NN>(S1 + o, w);
    row_transposed_pair<N>(tBw, v, tGw, w, a);
    write_row<N, NN>(S2 + o, a);
  });
  lds_barrier();
  T acc[NC];
  if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) acc[c] = S2[c * NQ + li];
  }
  if (P.scatter == SCATTER_ELEMENT) {
    store_element<N, NC>(P.E, acc, S0, slot, li, active);
  } else if (P.ordered) {
    scatter_element<N, NC, T, V>(r, acc, S0, smem + (el > 0 && el < EB ? el - 1 : 0) * PER, snode, el, EB, node, li,
                                 active, P.nnodes, P.ordering, P.scatter, P.ordered == 2);
  } else if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) scatter_add(r, lidx(node, c, NC, P.nnodes, P.ordering), V(acc[c]), P.scatter);
  }
}

// J.v for p = 3 (N = 4), arithmetic in T: the contractions along x and y
// move values between lanes of the element's wave (quad_bcast, row_ror)
// instead of through LDS; only the z contractions and the scatter use LDS.
// Vectors V (float, or double for FP32 arithmetic on FP64 vectors), tangent S.
// The same stages, in the same order of operations per term, as k_jvp.
template <typename T, int NC, int LAYOUT, typename S, typename V, int EB>
__global__ void __launch_bounds__(64 * EB) k_jvp_xy(const ElemLaunch P)
{
  constexpr int  N    = 4;
  constexpr int  NQ   = N * N * N;
  using Shape         = TanShape<LAYOUT, NC>;
  constexpr bool FULL = Shape::VAL;
  constexpr int  M    = Shape::M;
  constexpr int  DS   = Shape::DS;
  constexpr int  R    = NC * NQ;
  constexpr int  PER  = 3 * R;  // the y-interpolation outputs, later the y-integration outputs and the scatter
  constexpr int  TAB  = 4 * N * N;
  using Lay           = TangentLayout<S, DS, NQ>;

  __shared__ T   smem[EB * PER];
  __shared__ T   stab[TAB];
  __shared__ int snode[EB * NQ];

  if (P.stop != nullptr && *P.stop != 0.0) return;

  const int     tid    = threadIdx.x;
  const int     el     = tid / NQ;  // one element per wave
  const int     li     = tid - el * NQ;
  const int     i0     = li & 3;
  const int     i1     = (li >> 2) & 3;
  const int     i2     = li >> 4;
  const int64_t slot   = P.slot_begin + logical_block(P.xcd_remap) * EB + el;
  const bool    active = (el < EB) && (slot < P.slot_end);  // the same for every lane of a wave
  T*            S_     = smem + (el < EB ? el : 0) * PER;
  const V*      u      = static_cast<const V*>(P.u);
  V*            r      = static_cast<V*>(P.r);

  for (int k = tid; k < TAB; k += blockDim.x) stab[k] = T(P.tables[k]);
  const T* tB  = stab;
  const T* tG  = stab + N * N;
  const T* tBw = stab + 2 * N * N;
  const T* tGw = stab + 3 * N * N;

  int* const sn_el = snode + (el < EB ? el : 0) * NQ;
  T          ug[NC];
  if (active) {
    const int64_t node = P.map[size_t(slot) * NQ + li];
#pragma unroll
    for (int c = 0; c < NC; c++) ug[c] = T(u[lidx(node, c, NC, P.nnodes, P.ordering)]);
    sn_el[li] = int(node);  // read back for the scatter: no register holds it through the element work
  }
  TangentRegs<T, S, DS, NQ> Dr;
  if (active) Dr.load(static_cast<const char*>(P.D) + size_t(slot) * Lay::stride * sizeof(S), li);
  // the y index of the lane a rotation by 4 m within the row reads (m = 0..3)
  // the y index of the lane a rotation by 4 m within the row reads is
  // (i1 + m ydir) mod 4, ydir found by rotating the lane's own index once
  const int ydir = ((row_ror_i<4>(li & 15) >> 2) - i1) & 3;
  auto      ys   = [&](int m) { return (i1 + m * ydir) & 3; };
  lds_barrier();  // the tables

  T acc[NC];
  {
    // ---- interpolation: x through the quad, y through the row
    T b0[NC], b1[NC], b2[NC];
    if (active) {
#pragma unroll
      for (int c = 0; c < NC; c++) {
        const T v[4] = {quad_bcast<0>(ug[c]), quad_bcast<1>(ug[c]), quad_bcast<2>(ug[c]), quad_bcast<3>(ug[c])};
        T       s0 = T(0), s1 = T(0);
#pragma unroll
        for (int x = 0; x < N; x++) {
          s0 += tB[i0 * N + x] * v[x];
          s1 += tG[i0 * N + x] * v[x];
        }
        const T a0[4] = {s0, row_ror<4>(s0), row_ror<8>(s0), row_ror<12>(s0)};
        const T a1[4] = {s1, row_ror<4>(s1), row_ror<8>(s1), row_ror<12>(s1)};
        T       t0 = T(0), t1 = T(0), t2 = T(0);
#pragma unroll
        for (int m = 0; m < 4; m++) {
          const T b = tB[i1 * N + ys(m)], g = tG[i1 * N + ys(m)];
          t0 += b * a0[m];
          t1 += b * a1[m];
          t2 += g * a0[m];
        }
        b0[c] = t0;
        b1[c] = t1;
        b2[c] = t2;
      }
#pragma unroll
      for (int c = 0; c < NC; c++) {
        S_[0 * R + c * NQ + li] = b0[c];
        S_[1 * R + c * NQ + li] = b1[c];
        S_[2 * R + c * NQ + li] = b2[c];
      }
    }
    lds_barrier();

    // ---- z through LDS, then the chain rule at the point
    T out[M];
    if (active) {
      T in[M];
#pragma unroll
      for (int c = 0; c < NC; c++) {
        const T* a20 = S_ + 0 * R + c * NQ;
        const T* a21 = S_ + 1 * R + c * NQ;
        const T* a22 = S_ + 2 * R + c * NQ;
        T        v = T(0), g0 = T(0), g1 = T(0), g2 = T(0);
#pragma unroll
        for (int z = 0; z < N; z++) {
          const int idx = (z * N + i1) * N + i0;
          const T   b = tB[i2 * N + z], g = tG[i2 * N + z];
          if constexpr (FULL) v += b * a20[idx];
          g0 += b * a21[idx];
          g1 += b * a22[idx];
          g2 += g * a20[idx];
        }
        if constexpr (FULL) in[c] = v;
        in[(FULL ? NC : 0) + c * 3 + 0] = g0;
        in[(FULL ? NC : 0) + c * 3 + 1] = g1;
        in[(FULL ? NC : 0) + c * 3 + 2] = g2;
      }
#pragma unroll
      for (int k = 0; k < M; k++) out[k] = T(0);
#pragma unroll
      for (int s = 0; s < M; s++)
#pragma unroll
        for (int rr = 0; rr < Shape::rows(s); rr++) {
          const T Dk = Dr.get(Shape::idx(rr, s));
          out[rr] += Dk * in[s];
          if (Shape::SYM && rr != s) out[s] += Dk * in[rr];
        }
    }

    // ---- integration: x through the quad, y through the row, from registers
    T d0[NC], d1[NC];
    if (active) {
#pragma unroll
      for (int c = 0; c < NC; c++) {
        const T f0 = out[(FULL ? NC : 0) + c * 3 + 0], f1 = out[(FULL ? NC : 0) + c * 3 + 1];
        const T f2 = out[(FULL ? NC : 0) + c * 3 + 2];
        const T q0[4] = {quad_bcast<0>(f0), quad_bcast<1>(f0), quad_bcast<2>(f0), quad_bcast<3>(f0)};
        const T q1[4] = {quad_bcast<0>(f1), quad_bcast<1>(f1), quad_bcast<2>(f1), quad_bcast<3>(f1)};
        const T q2[4] = {quad_bcast<0>(f2), quad_bcast<1>(f2), quad_bcast<2>(f2), quad_bcast<3>(f2)};
        T       sr[4] = {T(0), T(0), T(0), T(0)};
        if constexpr (FULL) {
          sr[0] = quad_bcast<0>(out[c]);
          sr[1] = quad_bcast<1>(out[c]);
          sr[2] = quad_bcast<2>(out[c]);
          sr[3] = quad_bcast<3>(out[c]);
        }
        T s0 = T(0), s1 = T(0), s2 = T(0);
#pragma unroll
        for (int qx = 0; qx < N; qx++) {
          const T bw = tBw[qx * N + i0], gw = tGw[qx * N + i0];
          if constexpr (FULL) s0 += sr[qx] * bw;
          s0 += q0[qx] * gw;
          s1 += q1[qx] * bw;
          s2 += q2[qx] * bw;
        }
        const T a20[4] = {s0, row_ror<4>(s0), row_ror<8>(s0), row_ror<12>(s0)};
        const T a21[4] = {s1, row_ror<4>(s1), row_ror<8>(s1), row_ror<12>(s1)};
        const T a22[4] = {s2, row_ror<4>(s2), row_ror<8>(s2), row_ror<12>(s2)};
        T       t0 = T(0), t1 = T(0);
#pragma unroll
        for (int m = 0; m < 4; m++) {
          const T bw = tBw[ys(m) * N + i1], gw = tGw[ys(m) * N + i1];
          t0 += a20[m] * bw + a21[m] * gw;
          t1 += a22[m] * bw;
        }
        d0[c] = t0;
        d1[c] = t1;
      }
    }
    lds_barrier();  // every lane has read the interpolation slots
    if (active) {
#pragma unroll
      for (int c = 0; c < NC; c++) {
        S_[0 * R + c * NQ + li] = d0[c];
        S_[1 * R + c * NQ + li] = d1[c];
      }
    }
    lds_barrier();

    // ---- z integration through LDS
    if (active) {
#pragma unroll
      for (int c = 0; c < NC; c++) {
        const T* a10 = S_ + 0 * R + c * NQ;
        const T* a11 = S_ + 1 * R + c * NQ;
        acc[c]       = T(0);
#pragma unroll
        for (int qz = 0; qz < N; qz++) {
          const int idx = (qz * N + i1) * N + i0;
          acc[c] += a10[idx] * tBw[qz * N + i2] + a11[idx] * tGw[qz * N + i2];
        }
      }
    }
  }
  // slot 2 is free here: the z integration reads slots 0 and 1 only
  if (P.scatter == SCATTER_ELEMENT) {
    store_element<N, NC>(P.E, acc, S_ + 2 * R, slot, li, active);
    return;
  }
  const int64_t node = active ? int64_t(sn_el[li]) : 0;
  if (P.ordered) {
    scatter_element<N, NC, T, V>(r, acc, S_ + 2 * R, smem + (el > 0 && el < EB ? el - 1 : 0) * PER + 2 * R, snode,
                                 el, EB, node, li, active, P.nnodes, P.ordering, P.scatter, P.ordered == 2);
  } else if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) scatter_add(r, lidx(node, c, NC, P.nnodes, P.ordering), V(acc[c]), P.scatter);
  }
}

// Diagonal of the linearized operator from the stored tangent (FP64 out):
//   diag(c, j) = sum_q [w phi_j, w grad phi_j]_c . D(q) . [phi_j, grad phi_j]_c
// (the diagonal entries element_gradient_kernel would assemble,
//  fn/domain_integral_kernels.hpp:327-361).
// Every term is a product of one 1D factor per direction, so the sum over q
// factorizes: with phi_j = B(qx, jx) B(qy, jy) B(qz, jz), the term of tangent
// entry (test grad a, trial grad b) carries in direction d the factor
// (w G)(q_d, j_d) if a = d else (w B), times G(q_d, j_d) if b = d else B.  The
// products w B B, w G B (= w B G) and w G G are the three 1D tables.  Entries
// (a, b) and (b, a) share their tables and are summed first; the value rows of
// FULL_SYM add the (value, value) term and the (value, grad) pairs.  Per
// component this leaves NF fields per point, each contracted over qx, qy, qz in
// turn through LDS.
template <int LAYOUT, int NC>
struct DiagFields {
  using Shape                = TanShape<LAYOUT, NC>;
  static constexpr bool FULL = Shape::VAL;
  static constexpr int  NF   = FULL ? 10 : 6;  // per component: 6 gradient pairs (+ value, 3 value-gradient pairs)
  // gradient pair f < 6: (a, b) = (0,0) (1,1) (2,2) (0,1) (0,2) (1,2)
  __host__ __device__ static constexpr int pa(int f) { return f < 3 ? f : (f == 5 ? 1 : 0); }
  __host__ __device__ static constexpr int pb(int f) { return f < 3 ? f : (f == 3 ? 1 : 2); }
  // table (0: w B B, 1: w G B, 2: w G G) of field f in direction d
  __host__ __device__ static constexpr int table(int f, int d)
  {
    return f < 6 ? int(pa(f) == d) + int(pb(f) == d) : (f == 6 ? 0 : int(f - 7 == d));
  }
};

// The contractions go by rows, all components at once and every field in its
// place.  Neo-Hookean p = 3 on 48x40x44, FP64: 305 -> 248 us, of which the
// tangent's bytes take 176.
// One component has rows for some of the lanes only.  Rows and a lane per
// result: heat p = 1 (80x79x81 elements) 62 and 69 us, p = 2 (48x47x49) 57 and
// 61, p = 3 (36x35x37) 68 and 58, p = 4 (28x27x29) 62 and 69; mass-diffusion
// with its ten fields 93 and 101, 84 and 76, 103 and 78, 101 and 97.
template <int N, int NC, int NF>
constexpr bool use_diag_rows()
{
  return NC > 1 || (N != 4 && (NF == 6 || N == 2));
}

template <int N, int NC, int LAYOUT, typename S>
__global__ void __launch_bounds__(256) k_diagonal(const ElemLaunch P)
{
  constexpr int NQ = N * N * N;
  constexpr int EB = 256 / NQ;
  using Shape      = TanShape<LAYOUT, NC>;
  using F          = DiagFields<LAYOUT, NC>;
  constexpr int NF = F::NF;
  constexpr int VO = Shape::VO;
  constexpr int NN = N * N;
  constexpr int R  = NC * NQ;  // one field, all components
  using Lay        = TangentLayout<S, Shape::DS, NQ>;
  constexpr bool ROWS = use_diag_rows<N, NC, NF>();
  __shared__ double sf[EB * NF * R];
  __shared__ double stab[ROWS ? 1 : 3 * NN];  // w B B, w G B, w G G
  __shared__ int    snode[EB * NQ];

  const int     tid    = threadIdx.x;
  const int     el     = tid / NQ;
  const int     li     = tid - el * NQ;
  const int64_t slot   = P.slot_begin + logical_block(P.xcd_remap) * EB + el;
  const bool    active = (el < EB) && (slot < P.slot_end);  // uniform over the element's lanes
  double*       sv     = sf + (el < EB ? el : 0) * NF * R;
  if constexpr (!ROWS)
    for (int k = tid; k < 3 * NN; k += blockDim.x) stab[k] = P.tables[4 * NN + 2 * N + k];
  const ScalarTable tab = (ScalarTable)(uintptr_t)P.tables + (4 * NN + 2 * N);  // w B B, w G B, w G G

  using raw        = typename StoreTraits<S>::raw;
  const raw* Dbase = reinterpret_cast<const raw*>(static_cast<const char*>(P.D) +
                                                  size_t(active ? slot : 0) * Lay::stride * sizeof(S));
  auto       Dat   = [&](int k) -> double {
    const raw v = Dbase[Lay::offset(k, li)];
    if constexpr (sizeof(S) == 2)
      return double(bf16_to_float(uint32_t(v)));
    else
      return double(v);
  };
  if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const int g0 = VO + c * 3;
#pragma unroll
      for (int f = 0; f < 6; f++) {
        const int ra = g0 + F::pa(f), rb = g0 + F::pb(f);
        sv[f * R + c * NQ + li] = ra == rb ? Dat(Shape::idx(ra, rb)) : Dat(Shape::idx(ra, rb)) + Dat(Shape::idx(rb, ra));
      }
      if constexpr (F::FULL) {
        sv[6 * R + c * NQ + li] = Dat(Shape::idx(c, c));
#pragma unroll
        for (int d = 0; d < 3; d++)
          sv[(7 + d) * R + c * NQ + li] = Dat(Shape::idx(c, g0 + d)) + Dat(Shape::idx(g0 + d, c));
      }
    }
  }
  const int64_t node = active ? int64_t(P.map[size_t(slot) * NQ + li]) : 0;
  lds_barrier();
  double acc[NC];
  if constexpr (!ROWS) {
    const int a0 = li % N, a1 = (li / N) % N, a2 = li / NN;
    double    t[NF];
    // a field's results take the place of its values once every lane has read them
    auto put = [&] {
      lds_barrier();
      if (active) {
#pragma unroll
        for (int f = 0; f < NF; f++) sv[f * NQ + li] = t[f];
      }
      lds_barrier();
    };
    if (active) {
#pragma unroll
      for (int f = 0; f < NF; f++) t[f] = dot_result<N, N, 1>(stab + F::table(f, 0) * NN + a0, sv + f * NQ + li - a0);
    }
    put();
    if (active) {
#pragma unroll
      for (int f = 0; f < NF; f++)
        t[f] = dot_result<N, N, N>(stab + F::table(f, 1) * NN + a1, sv + f * NQ + a2 * NN + a0);
    }
    put();
    if (active) {
      acc[0] = 0.0;
#pragma unroll
      for (int f = 0; f < NF; f++)
        acc[0] += dot_result<N, N, NN>(stab + F::table(f, 2) * NN + a2, sv + f * NQ + a1 * N + a0);
    }
    lds_barrier();  // the scatter below reuses the second field's place
  } else {
    for_rows<N, NC, 0>(li, active, [&](int o) {
#pragma unroll
      for (int f = 0; f < NF; f++) {
        double v[N], a[N];
        read_row<N, 1>(sv + f * R + o, v);
        row_transposed<N>(tab + F::table(f, 0) * NN, v, a);
        write_row<N, 1>(sv + f * R + o, a);
      }
    });
    lds_barrier();
    for_rows<N, NC, 1>(li, active, [&](int o) {
#pragma unroll
      for (int f = 0; f < NF; f++) {
        double v[N], a[N];
        read_row<N, N>(sv + f * R + o, v);
        row_transposed<N>(tab + F::table(f, 1) * NN, v, a);
        write_row<N, N>(sv + f * R + o, a);
      }
    });
    lds_barrier();
    for_rows<N, NC, 2>(li, active, [&](int o) {
      double a[N];
#pragma unroll
      for (int i = 0; i < N; i++) a[i] = 0.0;
#pragma unroll
      for (int f = 0; f < NF; f++) {
        double v[N];
        read_row<N, NN>(sv + f * R + o, v);
        row_transposed<N>(tab + F::table(f, 2) * NN, v, a, true);
      }
      write_row<N, NN>(sv + o, a);
    });
    lds_barrier();
    if (active) {
#pragma unroll
      for (int c = 0; c < NC; c++) acc[c] = sv[c * NQ + li];
    }
  }
  // scatter (in address order as the J.v's) through the second field's place
  double* out = static_cast<double*>(P.r);
  if (P.scatter == SCATTER_ELEMENT) {
    store_element<N, NC>(P.E, acc, sv + R, slot, li, active);
  } else if (P.ordered) {
    scatter_element<N, NC, double, double>(out, acc, sv + R, sf + (el > 0 && el < EB ? el - 1 : 0) * NF * R + R, snode,
                                           el, EB, node, li, active, P.nnodes, P.ordering, P.scatter, P.ordered == 2);
  } else if (active) {
#pragma unroll
    for (int c = 0; c < NC; c++) scatter_add(out, lidx(node, c, NC, P.nnodes, P.ordering), acc[c], P.scatter);
  }
}

// Element gradient assembled into CSR values (element_gradient_kernel,
// fn/domain_integral_kernels.hpp:327-361, and Gradient::assemble,
// fn/functional.hpp:569-667, which scatters K_e through lookup tables):
//   K_e[(c,i)][(c',j)] = sum_q [w phi_i, w grad phi_i]_c . D(q) . [phi_j, grad phi_j]_c'
// For each pair (c, c') this is a product of an NQ x (slots NQ) matrix of test
// functions with an (slots NQ) x NQ matrix of D times the trial functions, so
// it runs on the FP64 matrix cores: a wave owns a 16 x 16 tile of node pairs
// for every (c, c'), and each mfma_f64_16x16x4 takes four points for one slot
// (lane l: test node l % 16, trial node l % 16, point l / 16 of the four).
// Both factors are formed in registers from the 1D tables and the point's
// tangent entries (staged in LDS where they fit in 48 KB, which leaves one
// wait on memory per element instead of one per four points); the test factor serves all c', the trial factor all c.
// The lane's results (nodes 4 r + l / 16 by l % 16) are added at their CSR
// positions: a row holds NC columns per neighbour node, so one binary search
// per node pair over the neighbours gives the positions of all NC x NC
// entries.  Plain read-modify-write when the launch covers one element colour
// (deterministic), atomics otherwise.
// Neo-Hookean p = 2 on 14x12x13 elements: eight colour launches of 1008 us each
// with one lane per test node looping over trial nodes and points (and a
// search per entry) before, 36 us each now (a wave and the waits of one element).
template <int N>
struct AssembleTiles {
  static constexpr int T      = (N * N * N + 15) / 16;           // tiles per direction of the node pairs
  static constexpr int WAVES  = T * T < 4 ? T * T : 4;           // waves (tiles) per workgroup
  static constexpr int GROUPS = (T * T + WAVES - 1) / WAVES;     // workgroups per element
  static constexpr int POINTS = (N * N * N + 3) / 4 * 4;         // four to a product
};

template <int N, int NC, int LAYOUT, typename S, bool STAGE>
__global__ void __launch_bounds__(64 * AssembleTiles<N>::WAVES, 2) k_assemble(const ElemLaunch P)
{
  typedef double d4 __attribute__((ext_vector_type(4)));
  constexpr int  NQ = N * N * N;
  using Shape       = TanShape<LAYOUT, NC>;
  using Tiles       = AssembleTiles<N>;
  using Lay         = TangentLayout<S, Shape::DS, NQ>;
  constexpr bool VAL = Shape::VAL;
  constexpr int  NS  = VAL ? 4 : 3;  // slots per component: [value], gradient
  constexpr int  TAB = 4 * N * N;
  constexpr int  DS  = Shape::DS;
  __shared__ double        stab[TAB];
  extern __shared__ double sD[];  // [q][DS]
  const int64_t pos  = P.slot_begin + blockIdx.x / Tiles::GROUPS;
  const int64_t slot = P.slot_list ? P.slot_list[pos] : pos;

  using raw       = typename StoreTraits<S>::raw;
  const raw* Dsrc = reinterpret_cast<const raw*>(static_cast<const char*>(P.D) + size_t(slot) * Lay::stride * sizeof(S));
  auto       Dat  = [&](int k, int q) -> double {
    const raw v = Dsrc[Lay::offset(k, q)];
    if constexpr (sizeof(S) == 2)
      return double(bf16_to_float(uint32_t(v)));
    else
      return double(v);
  };
  if constexpr (STAGE) {
    // group by group, a group's points side by side in memory
#pragma unroll 4
    for (int t = threadIdx.x; t < NQ * DS; t += blockDim.x) {
      constexpr int V  = Lay::VEC;
      const int     gq = t / V, k = t < Lay::G * V * NQ ? (gq / NQ) * V + t % V : Lay::G * V + (t - Lay::G * V * NQ) / NQ;
      const int     q  = t < Lay::G * V * NQ ? gq % NQ : (t - Lay::G * V * NQ) % NQ;
      sD[q * DS + k]   = Dat(k, q);
    }
    // the last group of four points: zeros in the place of points that are not there
    for (int t = NQ * DS + threadIdx.x; t < Tiles::POINTS * DS; t += blockDim.x) sD[t] = 0.0;
  }
  for (int k = threadIdx.x; k < TAB; k += blockDim.x) stab[k] = P.tables[k];
  __syncthreads();

  const int     tile = int(blockIdx.x % Tiles::GROUPS) * Tiles::WAVES + int(threadIdx.x >> 6);
  if (tile >= Tiles::T * Tiles::T) return;
  const int l  = threadIdx.x & 63;
  const int i  = (tile / Tiles::T) * 16 + (l & 15);  // the lane's test node in the products
  const int j  = (tile % Tiles::T) * 16 + (l & 15);  // its trial node, there and in the results
  const int ic = i < NQ ? i : 0, jc = j < NQ ? j : 0;  // rows and columns past the nodes are computed and dropped

  // values and gradient of node n's function at point q from the tables b, g
  auto basis = [&](const double* b, const double* g, int n, int q, double* out) {
    const int    x = n % N, y = (n / N) % N, z = n / (N * N), qx = q % N, qy = (q / N) % N, qz = q / (N * N);
    const double bx = b[qx * N + x], by = b[qy * N + y], bz = b[qz * N + z];
    if constexpr (VAL) out[0] = bx * by * bz;
    out[NS - 3] = g[qx * N + x] * by * bz;
    out[NS - 2] = bx * g[qy * N + y] * bz;
    out[NS - 1] = bx * by * g[qz * N + z];
  };
  d4 acc[NC][NC];
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int c2 = 0; c2 < NC; c2++) acc[c][c2] = d4{0.0, 0.0, 0.0, 0.0};

  for (int q0 = 0; q0 < NQ; q0 += 4) {
    const int q  = q0 + (l >> 4);
    const int qc = q < NQ ? q : 0;
    double    tf[NS], uf[NS];
    basis(stab + 2 * N * N, stab + 3 * N * N, ic, qc, tf);
    basis(stab, stab + N * N, jc, qc, uf);
    auto D = [&](int row, int col) -> double {
      if constexpr (STAGE)
        return sD[q * DS + Shape::idx(row, col)];
      else
        return q < NQ ? Dat(Shape::idx(row, col), q) : 0.0;
    };
    // input / output number of slot a of component c
    auto slot_of = [](int c, int a) { return VAL ? (a == 0 ? c : NC + c * 3 + a - 1) : c * 3 + a; };
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
      for (int a = 0; a < NS; a++)
#pragma unroll
        for (int c2 = 0; c2 < NC; c2++) {
          double t = 0.0;
#pragma unroll
          for (int b = 0; b < NS; b++) t += D(slot_of(c, a), slot_of(c2, b)) * uf[b];
          acc[c][c2] = __builtin_amdgcn_mfma_f64_16x16x4f64(tf[a], t, acc[c][c2], 0, 0, 0);
        }
  }

  if (j >= NQ) return;
  // the four node pairs' searches run side by side (rows past the nodes repeat the first), and without atomics all
  // old values are read before the first is written: each is a chain of dependent loads otherwise
  const int*    map  = P.map + size_t(slot) * NQ;
  const int32_t colv = int32_t(lidx(map[j], 0, NC, P.nnodes, P.ordering));
  const int     step = P.ordering ? NC : 1;
  int64_t       row[4][NC];
  int           nadj[4], lo[4], hi[4];
  bool          valid[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int ir         = (tile / Tiles::T) * 16 + 4 * r + (l >> 4);
    valid[r]             = ir < NQ;
    const int64_t node_i = map[valid[r] ? ir : 0];
#pragma unroll
    for (int c = 0; c < NC; c++) row[r][c] = P.csr_row[lidx(node_i, c, NC, P.nnodes, P.ordering)];
    nadj[r] = int(P.csr_row[lidx(node_i, 0, NC, P.nnodes, P.ordering) + 1] - row[r][0]) / NC;
    lo[r]   = 0;
    hi[r]   = nadj[r];  // the neighbour is in [lo, hi)
  }
  while (hi[0] - lo[0] > 1 || hi[1] - lo[1] > 1 || hi[2] - lo[2] > 1 || hi[3] - lo[3] > 1) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int  mid = (lo[r] + hi[r]) >> 1;
      const bool up  = P.csr_col[row[r][0] + int64_t(mid) * step] <= colv;
      if (hi[r] - lo[r] > 1) (up ? lo[r] : hi[r]) = mid;
    }
  }
  auto at = [&](int r, int c, int c2) {
    return P.csr_val + (row[r][c] + (P.ordering ? int64_t(lo[r]) * NC + c2 : int64_t(c2) * nadj[r] + lo[r]));
  };
  if (!P.scatter) {
    double old[4][NC][NC];
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int c2 = 0; c2 < NC; c2++) old[r][c][c2] = valid[r] ? *at(r, c, c2) : 0.0;
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int c2 = 0; c2 < NC; c2++)
          if (valid[r]) *at(r, c, c2) = old[r][c][c2] + acc[c][c2][r];
    return;
  }
#pragma unroll
  for (int r = 0; r < 4; r++)
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
      for (int c2 = 0; c2 < NC; c2++)
        if (valid[r]) unsafeAtomicAdd(at(r, c, c2), acc[c][c2][r]);
}

// ---------------------------------------------------------------------------
// launch + dispatch
// ---------------------------------------------------------------------------
template <int N, typename K>
inline hipError_t launch_grid(const ElemLaunch& P, K kernel)
{
  constexpr int EB = 256 / (N * N * N);
  const int64_t n  = P.slot_end - P.slot_begin;
  if (n <= 0) return hipSuccess;
  const unsigned grid = unsigned((n + EB - 1) / EB);
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, P.stream, P);
  return hipGetLastError();
}

// k_jvp_xy: EB elements (waves) per workgroup.  With a BF16 tangent 2 per
// workgroup measured 1.5 % faster than 4 (fewer waves wait at each barrier); with
// an FP32 tangent 4 measured 3 % faster than 2 (64^3 p = 3 Neo-Hookean).
template <typename S>
constexpr int xy_elems_per_group()
{
  return sizeof(S) == 2 ? 2 : 4;
}
template <int EB, typename K>
inline hipError_t launch_grid_xy(const ElemLaunch& P, K kernel)
{
  const int64_t n = P.slot_end - P.slot_begin;
  if (n <= 0) return hipSuccess;
  const unsigned grid = unsigned((n + EB - 1) / EB);
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * EB), 0, P.stream, P);
  return hipGetLastError();
}

template <int N, typename T, typename K>
inline hipError_t launch_grid_jvp(const ElemLaunch& P, K kernel)
{
  constexpr int WG = jvp_group_lanes<N, T>();
  constexpr int EB = WG / (N * N * N);
  const int64_t n  = P.slot_end - P.slot_begin;
  if (n <= 0) return hipSuccess;
  const unsigned grid = unsigned((n + EB - 1) / EB);
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(WG), 0, P.stream, P);
  return hipGetLastError();
}

template <int N, int NC, int LAYOUT, typename S>
inline int dispatch_gradient(const ElemLaunch& P, hipError_t* err)
{
  if (P.mode == MODE_ASSEMBLE) {
    const int64_t n = P.slot_end - P.slot_begin;
    if (n <= 0) return 1;
    using Tiles            = AssembleTiles<N>;
    constexpr size_t bytes = size_t(Tiles::POINTS) * TanShape<LAYOUT, NC>::DS * sizeof(double);
    constexpr bool   stage = bytes <= 48 * 1024;
    hipLaunchKernelGGL((k_assemble<N, NC, LAYOUT, S, stage>), dim3(unsigned(n * Tiles::GROUPS)),
                       dim3(64 * Tiles::WAVES), stage ? bytes : 0, P.stream, P);
    *err = hipGetLastError();
    return 1;
  }
  if (P.mode == MODE_DIAG) {
    *err = launch_grid<N>(P, k_diagonal<N, NC, LAYOUT, S>);
    return 1;
  }
  if (P.vprec == PREC_F64) {
    *err = launch_grid_jvp<N, double>(P, k_jvp<N, NC, LAYOUT, double, S, double>);
    return 1;
  }
  if (P.vprec == PREC_F32) {
    if constexpr (N == 4)
      *err = launch_grid_xy<xy_elems_per_group<S>()>(P, k_jvp_xy<float, NC, LAYOUT, S, float, xy_elems_per_group<S>()>);
    else if constexpr (use_jvp_rows<N, NC>())
      *err = launch_grid_jvp<N, float>(P, k_jvp_rows<N, NC, LAYOUT, S, float>);
    else
      *err = launch_grid_jvp<N, float>(P, k_jvp<N, NC, LAYOUT, float, S, float>);
    return 1;
  }
  if (P.vprec == PREC_MIXED) {
    if constexpr (N == 4)
      *err = launch_grid_xy<xy_elems_per_group<S>()>(P, k_jvp_xy<float, NC, LAYOUT, S, double, xy_elems_per_group<S>()>);
    else if constexpr (use_jvp_rows<N, NC>())
      *err = launch_grid_jvp<N, float>(P, k_jvp_rows<N, NC, LAYOUT, S, double>);
    else
      *err = launch_grid_jvp<N, float>(P, k_jvp<N, NC, LAYOUT, float, S, double>);
    return 1;
  }
  return 0;
}

template <int N, int NC, int LAYOUT>
inline int dispatch_gradient_prec(const ElemLaunch& P, hipError_t* err)
{
  switch (P.tprec) {
    case PREC_F64: return dispatch_gradient<N, NC, LAYOUT, double>(P, err);
    case PREC_F32: return dispatch_gradient<N, NC, LAYOUT, float>(P, err);
    case PREC_BF16: return dispatch_gradient<N, NC, LAYOUT, bf16>(P, err);
  }
  return 0;
}

template <int N, int NC, class QF, int LAYOUT>
inline int dispatch_eval(const ElemLaunch& P, hipError_t* err)
{
  if (P.mode == MODE_RESIDUAL) {
    *err = launch_grid<N>(P, k_element<N, NC, MODE_RESIDUAL, QF, LAYOUT, double>);
    return 1;
  }
  if (P.mode == MODE_SHAPE_JVP) {
    if constexpr (NC == 3) {
      *err = launch_grid<N>(P, k_element<N, NC, MODE_SHAPE_JVP, QF, LAYOUT, double>);
      return 1;
    }
    return 0;
  }
  switch (P.tprec) {
    case PREC_F64: *err = launch_grid<N>(P, k_element<N, NC, MODE_LINEARIZE, QF, LAYOUT, double>); return 1;
    case PREC_F32: *err = launch_grid<N>(P, k_element<N, NC, MODE_LINEARIZE, QF, LAYOUT, float>); return 1;
    case PREC_BF16: *err = launch_grid<N>(P, k_element<N, NC, MODE_LINEARIZE, QF, LAYOUT, bf16>); return 1;
  }
  return 0;
}

// Dispatch on (mode, qfunction, components, tangent layout, precisions) for one order.
template <int N>
inline int dispatch_order(const ElemLaunch& P, hipError_t* err)
{
  if (P.mode == MODE_JVP || P.mode == MODE_DIAG || P.mode == MODE_ASSEMBLE) {
    if (P.nc == 1) {
      if (P.layout == LAYOUT_GRAD_SYM) return dispatch_gradient_prec<N, 1, LAYOUT_GRAD_SYM>(P, err);
      if (P.layout == LAYOUT_FULL_SYM) return dispatch_gradient_prec<N, 1, LAYOUT_FULL_SYM>(P, err);
    }
    if (P.nc == 3) {
      if (P.layout == LAYOUT_GRAD_SYM) return dispatch_gradient_prec<N, 3, LAYOUT_GRAD_SYM>(P, err);
      if (P.layout == LAYOUT_FULL_SYM) return dispatch_gradient_prec<N, 3, LAYOUT_FULL_SYM>(P, err);
      if (P.layout == LAYOUT_GRAD_FULL) return dispatch_gradient_prec<N, 3, LAYOUT_GRAD_FULL>(P, err);
    }
    return 0;
  }
  switch (P.qf) {
    case QF_ID_HEAT:
      if (P.nc == 1) return dispatch_eval<N, 1, QFHeat, LAYOUT_GRAD_SYM>(P, err);
      break;
    case QF_ID_MASS_DIFFUSION:
      if (P.nc == 1) return dispatch_eval<N, 1, QFMassDiffusion<1>, LAYOUT_FULL_SYM>(P, err);
      if (P.nc == 3) return dispatch_eval<N, 3, QFMassDiffusion<3>, LAYOUT_FULL_SYM>(P, err);
      break;
    case QF_ID_NEOHOOKEAN:
      if (P.nc == 3) return dispatch_eval<N, 3, QFNeoHookean, LAYOUT_GRAD_SYM>(P, err);
      break;
    case QF_ID_LINEAR_ELASTIC:
      if (P.nc == 3) return dispatch_eval<N, 3, QFLinearElastic, LAYOUT_GRAD_SYM>(P, err);
      break;
    case QF_ID_J2:
      if (P.nc == 3) return dispatch_eval<N, 3, QFJ2, LAYOUT_GRAD_FULL>(P, err);
      break;
    case QF_ID_QOI_VALUE:
      // residual only: the QoI gradient is never linearized
      if (P.mode != MODE_RESIDUAL) return 0;
      if (P.nc == 1) {
        *err = launch_grid<N>(P, k_element<N, 1, MODE_RESIDUAL, QFQoiValue<1>, LAYOUT_GRAD_SYM, double>);
        return 1;
      }
      if (P.nc == 3) {
        *err = launch_grid<N>(P, k_element<N, 3, MODE_RESIDUAL, QFQoiValue<3>, LAYOUT_GRAD_SYM, double>);
        return 1;
      }
      break;
  }
  return 0;
}

}  // namespace sxk
