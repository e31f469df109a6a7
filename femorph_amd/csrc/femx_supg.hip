// femx_supg.hip -- explicit SUPG / grad-div step with a local bulk modulus
// (femSUPGExplicitFluidSolver) on hexa8 and tet4 for gfx950.
//
// The reference forms nine dense 24x24 element matrices per Gauss point and
// multiplies K by the element velocity (src/femSUPGExplicitFluidSolver.cpp:
// 1095-1507).  Here the same operator is applied matrix-free, one element per
// thread, term by term per Gauss point:
//   K1 u : rho N_a (u_g . grad) u_k dV                         (:1318-1322)
//   K2 u : B^T D(lambda_g, mu) B u dV, B with the reference's B-hat (:1333-1337, :222-296)
//   K3 u : rho tau (u_g . grad N_a) (u_g . grad) u_k dV        (:1341-1345)
//   K4 u : rho nu_C dN_a/dx_k div(u) dV                        (:1348)
// then k_e = -dt K u_e and Euler / AB2 accumulation into the nodes.
// Element blocks (<= 128 elements, <= 256 nodes) are assembled in LDS exactly
// like the VMS kernel: block-complete nodes are updated in the block, block
// boundary nodes through FP64 partial sums (FP32 in the opt-in
// FEMX_MIXED_F32SUM) and a fix-up launch.
//
// Differences of form (not of value) from the reference, all within
// rounding: the AB2 history is kept as the assembled nodal force of the
// previous step (1.5 F_n - 0.5 F_{n-1} equals the sum over elements of
// 1.5 k - 0.5 k_prev), which replaces 384 B/element of history traffic by
// 24 B/node; the post-processed pressure of step n (compute_pressure
// :446-501, needed only as an output) is evaluated inside step n+1's element
// pass from the same Gauss-point divergence when no global DOFs are fixed.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>

#include "femx_common.h"
#include "femx_elem.h"

namespace femx {
namespace {

// max elements per block of the mesh partition (femx_mesh_upload cuts tet4
// meshes into <= 256-element blocks, hexa8 into <= 128); one thread per tet4,
// two per hexa8
template <int NPE>
constexpr int elems_for() { return NPE == 4 ? 256 : 128; }
constexpr int SB = 256;

// diagnostic row layout: 0..5 min/max u v w, 6,7 min/max tau, 8,9 min/max
// lambda, 10 v-CFL max, 11 a-CFL max, 12 l-CFL max, 13,14 min/max E,
// 15,16 min/max nu, 17 max |u|^2 (the log columns of :1601-1630).  The log row
// holds the step it belongs to in one more column.
enum { D_UMIN = 0, D_TAU = 6, D_LAM = 8, D_VCFL = 10, D_ACFL = 11, D_LCFL = 12, D_E = 13, D_NU = 15, D_UMOD = 17,
       D_COLS = 18, D_STEP = 18, D_ROW = 19 };
__host__ __device__ constexpr bool d_is_min(int c) {
  return c == 0 || c == 2 || c == 4 || c == D_TAU || c == D_LAM || c == D_E || c == D_NU;
}
__host__ __device__ constexpr double d_identity(int c) {
  return (c == D_VCFL || c == D_ACFL || c == D_LCFL || c == D_UMOD) ? 0.0
         : d_is_min(c) ? 1.79769313486231570815e+308 : -1.79769313486231570815e+308;
}

// Folds one node's new state into the velocity extrema (columns D_UMIN ..
// D_UMIN + 5: min/max of u, v, w) and max |u|^2; NaN never wins.
__device__ __forceinline__ void node_extrema(const double4 u, double v[6], double &m2) {
  v[0] = fmin(v[0], u.x);
  v[1] = fmax(v[1], u.x);
  v[2] = fmin(v[2], u.y);
  v[3] = fmax(v[3], u.y);
  v[4] = fmin(v[4], u.z);
  v[5] = fmax(v[5], u.z);
  m2 = fmax(m2, u.x * u.x + u.y * u.y + u.z * u.z);
}

// Block-wide velocity extrema and max |u|^2 (columns D_UMIN .. D_UMIN + 5
// and D_UMOD) in one pass; thread 0 stores them to the block's row out.
template <int NT>
__device__ __forceinline__ void block_node_store(double v[6], double m2, double *out) {
  __shared__ double wv[NT / 64][7];
  double x[7] = {v[0], v[1], v[2], v[3], v[4], v[5], m2};
#pragma unroll
  for (int i = 0; i < 7; i++) {
    const bool mn = i < 6 && d_is_min(D_UMIN + i);
    for (int off = 32; off > 0; off >>= 1) {
      const double o = __shfl_xor(x[i], off);
      x[i] = mn ? fmin(x[i], o) : fmax(x[i], o);
    }
  }
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int i = 0; i < 7; i++) wv[threadIdx.x >> 6][i] = x[i];
  __syncthreads();
  if (threadIdx.x == 0)
#pragma unroll
    for (int i = 0; i < 7; i++) {
      const bool mn = i < 6 && d_is_min(D_UMIN + i);
      double r = wv[0][i];
      for (int w = 1; w < NT / 64; w++) r = mn ? fmin(r, wv[w][i]) : fmax(r, wv[w][i]);
      out[i < 6 ? D_UMIN + i : D_UMOD] = r;
    }
}

// Block-wide min/max of the columns [c0, c0+K) of a diagnostic row; thread 0
// stores the block's values to its row out[c]. NaN never wins
// (like the reference's `if (x > max)` tests).
template <int NT, int K>
__device__ __forceinline__ void block_diag_store(double v[K], int c0, double *out) {
  __shared__ double wv[NT / 64][K];
#pragma unroll
  for (int i = 0; i < K; i++) {
    const bool mn = d_is_min(c0 + i);
    for (int off = 32; off > 0; off >>= 1) {
      const double o = __shfl_xor(v[i], off);
      v[i] = mn ? fmin(v[i], o) : fmax(v[i], o);
    }
  }
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int i = 0; i < K; i++) wv[threadIdx.x >> 6][i] = v[i];
  __syncthreads();
  if (threadIdx.x == 0)
#pragma unroll
    for (int i = 0; i < K; i++) {
      double m = wv[0][i];
      for (int w = 1; w < NT / 64; w++) m = d_is_min(c0 + i) ? fmin(m, wv[w][i]) : fmax(m, wv[w][i]);
      out[c0 + i] = m;
    }
}

struct SupgConst {
  double rho, mu, alpha, cI, dt, t, exit2;
  int euler_step;   // 1: Euler update (Euler mode or the first step)
  int fixed;        // glob_fixed_dofs code
  int k1, k2, k3, k4;
};

template <typename T>
struct SupgArgs {
  int nblk, E;
  const int *elem_off, *node_off, *loc_node, *loc_pslot, *lcsr_off;
  const uint16_t *lpos;  // [E][npe] node-sorted position of each corner
  const uint8_t *lconn;  // [E][npe]
  const double4 *xyzm;   // x y z, lumped mass
  const double4 *U;      // sol_p (zeroed by the global fixed DOFs)
  const double4 *Upress; // post-BC state before the fixed-DOF zeroing (pressure of the previous step)
  double4 *Un, *Unp;     // outputs: next sol_p, next pre-zeroing state
  double4 *Fprev;        // assembled force of the previous step (AB2)
  // partial force sums of block-boundary nodes: double4 records, or float4
  // with f32sum (FEMX_MIXED_F32SUM: FP32 in-block sums)
  void *partials;
  int f32sum;
  double *lam, *regime, *pres;  // [E] block order
  const int *node_rec;
  const BCRecord *rec;
  const int *row_off;
  const double4 *rows;
  int *err;
  double *eblk;              // [nblk][D_COLS] per-block rows: node extrema, element diagnostics (DIAG)
  int *halt;                 // INT_MAX or the step that exceeded EXITCOND
  int step_id;
  int want_row;              // the step's log row is made: write the block's row
  SupgConst k;
};

// The exit condition (:1635-1643): the workgroups that form the new states of
// step `step` and see |u|^2 above the threshold put the step into *halt; the
// rest of that step still runs, every later step's work is skipped.  It
// replaces a test of the previous step's reduced maximum, so a step needs no
// reduction unless its log row is asked for.
__device__ __forceinline__ bool halted(const int *halt, int step) { return __builtin_nontemporal_load(halt) < step; }
__device__ __forceinline__ void exit_check(double m2, const SupgConst &k, int *halt, int step) {
  if (m2 > k.exit2) atomicMin(halt, step);
}

// SUPG node update of one node (:1510-1514 update, :1519-1521 BCs,
// :1527-1561 fixed DOFs): returns nothing, writes sol_p of the next step.
__device__ __forceinline__ void supg_node(const double F[3], double4 fprev, double m, double4 up, const SupgConst &k,
                                          bool has_bc, const BCRecord &bc, const int *row_off, const double4 *rows,
                                          int *err, double4 &next, double4 &press_state, double4 &fstore) {
  double acc[3];
  if (k.euler_step) {
    acc[0] = F[0]; acc[1] = F[1]; acc[2] = F[2];
  } else {
    acc[0] = (3.0 / 2.0) * F[0] - (1.0 / 2.0) * fprev.x;
    acc[1] = (3.0 / 2.0) * F[1] - (1.0 / 2.0) * fprev.y;
    acc[2] = (3.0 / 2.0) * F[2] - (1.0 / 2.0) * fprev.z;
  }
  const double im = 1.0 / m;
  double u = up.x + im * acc[0], v = up.y + im * acc[1], w = up.z + im * acc[2];
  if (has_bc) apply_bc(bc, row_off, rows, k.t, u, v, w, nullptr, err);
  press_state = make_double4(u, v, w, 0.0);
  const int f = k.fixed;
  if (f == 1 || f == 4 || f == 6) u = 0.0;
  if (f == 2 || f == 4 || f == 5) v = 0.0;
  if (f == 3 || f == 5 || f == 6) w = 0.0;
  next = make_double4(u, v, w, 0.0);
  fstore = make_double4(F[0], F[1], F[2], 0.0);
}

// hexa8 element math.  It is bound by VALU issue (four cycles per wave
// instruction in FP32 and FP64 alike), so it is arranged for few instructions
// and no spills:
//  - the map and the velocity are trilinear, so the sums over nodes at the
//    Gauss points share most of their terms (Tri), and so do the node sums of
//    the forces (TriSum); the averages of B-hat need no pass over the Gauss
//    points (TriAvg);
//  - two neighbouring lanes work on one element, each on the four Gauss points
//    of one z = +-1/sqrt 3, and hold the element's fields and sums for that z
//    only.  With one lane per element the same math needed 256 VGPRs, two
//    waves per SIMD (316 us).
// Per hexa8 element-step 2 x 2,200 wave-lane instructions against 6,650 node
// by node; with it the block kernel at 2.1M hexa went from 356 to 277 us mixed
// (250 now), at 85k hexa from 47 to 31 us FP64 (28).
// The other lane's value: a DPP quad permute (1, 0, 3, 2).
__device__ __forceinline__ int pair_swap(int v) { return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true); }
__device__ __forceinline__ float pair_swap(float v) { return __int_as_float(pair_swap(__float_as_int(v))); }
__device__ __forceinline__ double pair_swap(double v) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)pair_swap((int)(unsigned)(b & 0xffffffffLL));
  const unsigned hi = (unsigned)pair_swap((int)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <typename T>
__device__ __forceinline__ T pair_sum(T v) { return v + pair_swap(v); }

// A trilinear 3-vector field f = c1 + x cx + y cy + z cz + xy cxy + xz cxz + yz
// cyz + xyz cxyz (femHexa8 node signs, src/femHexa8.cpp:15-17) on the lane's
// plane of Gauss points.  z points towards the lane's own side, so both
// lanes work at z = 1/sqrt 3; the element's map is then left-handed for one of
// them.
//   f     = (c00 + y A2) + x df/dx           c00 = c1 + z cz
//   df/dx = A1 + y B                         A1 = cx + z cxz, B = cxy + z cxyz
//   df/dy = A2 + x B                         A2 = cy + z cyz
//   df/dz = (cz + y cyz) + x (cxz + y cxyz)
// so most of the sums are shared between Gauss points.  Node values come in
// as 1/8 of the field, the transforms' factor.
template <typename T>
struct Tri {
  T c00[3], A1[3], A2[3], B[3], Cz[3], Cxz[3], Cyz[3], Cxyz[3];
  T Dx[3], D[3], F[3];  // per y: df/dx, cz + y cyz, cxz + y cxyz
  // component b from the values at the four nodes of the lane's side; the
  // other lane holds the other side's
  __device__ __forceinline__ void load(int b, const T own[4], T q) {
    T g[4], d[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const T oth = pair_swap(own[k]);
      d[k] = own[k] - oth;
      g[k] = (own[k] + oth) + q * d[k];
    }
    xy(g, c00[b], A1[b], A2[b], B[b]);
    xy(d, Cz[b], Cxz[b], Cyz[b], Cxyz[b]);
  }
  template <typename S>
  __device__ __forceinline__ void from(const Tri<S> &f) {
#pragma unroll
    for (int b = 0; b < 3; b++) {
      c00[b] = (T)f.c00[b], A1[b] = (T)f.A1[b], A2[b] = (T)f.A2[b], B[b] = (T)f.B[b];
      Cz[b] = (T)f.Cz[b], Cxz[b] = (T)f.Cxz[b], Cyz[b] = (T)f.Cyz[b], Cxyz[b] = (T)f.Cxyz[b];
    }
  }
  static __device__ __forceinline__ void xy(const T g[4], T &s, T &x, T &y, T &c) {
    const T p = g[0] + g[1], q = g[2] + g[3], r = g[1] - g[0], t = g[2] - g[3];
    s = p + q;
    y = q - p;
    x = r + t;
    c = t - r;
  }
  __device__ __forceinline__ void at_y(T y) {
#pragma unroll
    for (int b = 0; b < 3; b++) {
      Dx[b] = A1[b] + y * B[b];
      D[b] = Cz[b] + y * Cyz[b];
      F[b] = Cxz[b] + y * Cxyz[b];
    }
  }
  __device__ __forceinline__ void at_x(T x, T L[3][3]) const {
#pragma unroll
    for (int b = 0; b < 3; b++) {
      L[0][b] = Dx[b];
      L[1][b] = A2[b] + x * B[b];
      L[2][b] = D[b] + x * F[b];
    }
  }
};

// The transpose: sums over the lane's Gauss points of v N + T0 dN/dx + T1
// dN/dy + T2 dN/dz in the same coefficients of the trilinear test functions.
template <typename T>
struct TriSum {
  T c00[3], A1[3], A2[3], B[3], Cz[3], Cxz[3], Cyz[3], Cxyz[3];
  __device__ __forceinline__ void init() {
#pragma unroll
    for (int b = 0; b < 3; b++) c00[b] = A1[b] = A2[b] = B[b] = Cz[b] = Cxz[b] = Cyz[b] = Cxyz[b] = (T)0;
  }
  // Tl[i][l]: component i, local direction l
  __device__ __forceinline__ void add(T x, T y, const T v[3], const T Tl[3][3]) {
    const T xy = x * y;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const T t0 = Tl[i][0] + x * v[i];
      c00[i] += v[i];
      A1[i] += t0;
      B[i] += y * t0;
      A2[i] += Tl[i][1] + y * v[i];
      B[i] += x * Tl[i][1];
      Cz[i] += Tl[i][2];
      Cxz[i] += x * Tl[i][2];
      Cyz[i] += y * Tl[i][2];
      Cxyz[i] += xy * Tl[i][2];
    }
  }
  // The element's sums on the nodes of the lane's side, as the four (x, y)
  // coefficients 1, x, y, xy of component b: with the test functions' z
  // factors 1 + z, own p + (q p + c) and the other lane's p - (q p + c) for
  // each pair p = c00, A1, A2, B and c = Cz, Cxz, Cyz, Cxyz.
  static __device__ __forceinline__ T fold(T p, T c, T q) {
    const T w = q * p + c;
    return (p + w) + pair_swap(p - w);
  }
  __device__ __forceinline__ void nodes(int b, T q, T e[4]) const {
    e[0] = fold(c00[b], Cz[b], q);
    e[1] = fold(A1[b], Cxz[b], q);
    e[2] = fold(A2[b], Cyz[b], q);
    e[3] = fold(B[b], Cxyz[b], q);
  }
};
// eval_avg_shapeDeriv (:660-707): the sums over the eight Gauss points of DN
// dv, that is of the Jacobian's cofactors times the local derivatives.  In the
// monomials of the trilinear map the two-point rule leaves (its points are
// +-1/sqrt 3: odd powers vanish, a square gives 1/3)
//   x: E2 x E3 + Exy x Exz / 3     xy: (E2 x Eyz + Exz x E1) / 3
//   y: E3 x E1 + Eyz x Exy / 3     xz: (Eyz x E3 + E1 x Exy) / 3
//   z: E1 x E2 + Exz x Eyz / 3     yz: (E3 x Exz + Exy x E2) / 3
// (times 8) and nothing for 1 and xyz: 72 multiply-adds instead of a pass
// over the Gauss points (about 400 instructions per lane).  Both lanes of an
// element form them in their own local coordinates; the sign of the map's
// handedness cancels in the average.  In FP64 on every path: the mean
// divergence (the pressure) is a small sum of large terms, and FP64 issues as
// fast as FP32 here.
struct TriAvg {
  using T = double;
  T x[3], y[3], z[3], xy[3], xz[3], yz[3];
  T vol;  // of the element
  // r = a x b + f c x d
  static __device__ __forceinline__ void cross2(const T a[3], const T b[3], T f, const T c[3], const T d[3], T r[3]) {
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int j = (i + 1) % 3, k = (i + 2) % 3;
      r[i] = (a[j] * b[k] - a[k] * b[j]) + f * (c[j] * d[k] - c[k] * d[j]);
    }
  }
  // the monomials' coefficients 1, 2 and xy of a field (the field holds them at its z)
  static __device__ __forceinline__ void base(const Tri<T> &f, T q, T f1[3], T f2[3], T fxy[3]) {
#pragma unroll
    for (int b = 0; b < 3; b++) {
      f1[b] = f.A1[b] - q * f.Cxz[b];
      f2[b] = f.A2[b] - q * f.Cyz[b];
      fxy[b] = f.B[b] - q * f.Cxyz[b];
    }
  }
  __device__ __forceinline__ void form(const Tri<T> &X, T q, T sg) {
    const T third = (T)(1.0 / 3.0);
    T E1[3], E2[3], Exy[3];
    base(X, q, E1, E2, Exy);
    cross2(E2, X.Cz, third, Exy, X.Cxz, x);
    cross2(X.Cz, E1, third, X.Cyz, Exy, y);
    cross2(E1, E2, third, X.Cxz, X.Cyz, z);
    cross2(E2, X.Cyz, (T)1, X.Cxz, E1, xy);
    cross2(X.Cyz, X.Cz, (T)1, E1, Exy, xz);
    cross2(X.Cz, X.Cxz, (T)1, Exy, E2, yz);
    // the volume from the field x itself: sum_n DN_n x_n = 1
    const T den = (x[0] * E1[0] + y[0] * E2[0] + z[0] * X.Cz[0]) +
                  third * (xy[0] * Exy[0] + xz[0] * X.Cxz[0] + yz[0] * X.Cyz[0]);
    vol = 8.0 * sg * den;
    const T id = recip(den), id3 = id * third;
#pragma unroll
    for (int b = 0; b < 3; b++) x[b] *= id, y[b] *= id, z[b] *= id, xy[b] *= id3, xz[b] *= id3, yz[b] *= id3;
  }
  // P_b = sum_n avg_nb u_nb
  __device__ __forceinline__ void dot(const Tri<T> &V, T q, T P[3]) const {
    T u1[3], u2[3], uxy[3];
    base(V, q, u1, u2, uxy);
#pragma unroll
    for (int b = 0; b < 3; b++)
      P[b] = (x[b] * u1[b] + y[b] * u2[b] + z[b] * V.Cz[b]) + (xy[b] * uxy[b] + xz[b] * V.Cxz[b] + yz[b] * V.Cyz[b]);
  }
};

// What eval_stabilization, eval_bulk_modulus and the diagnostics need of the
// metric G = invJ^T invJ (src/femElement.cpp:222-231): |G|^2 and its trace.
template <typename T>
__device__ __forceinline__ void metric3(const T iJ[3][3], T &gg, T &tr) {
  T d[3], o[3];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const int k = (i + 1) % 3;
    d[i] = iJ[0][i] * iJ[0][i] + iJ[1][i] * iJ[1][i] + iJ[2][i] * iJ[2][i];
    o[i] = iJ[0][i] * iJ[0][k] + iJ[1][i] * iJ[1][k] + iJ[2][i] * iJ[2][k];
  }
  tr = d[0] + d[1] + d[2];
  gg = (d[0] * d[0] + d[1] * d[1] + d[2] * d[2]) + (T)2 * (o[0] * o[0] + o[1] * o[1] + o[2] * o[2]);
}
// |J^T u|^2 = u^T G^-1 u and |invJ u|^2 = u^T G u (G^-1 = J J^T; the indices of
// G are local directions, those of u physical ones, as in the reference)
template <typename T>
__device__ __forceinline__ T norm2_tmul(const T m[3][3], const T u[3]) {
  T r = (T)0;
#pragma unroll
  for (int b = 0; b < 3; b++) {
    const T x = m[0][b] * u[0] + m[1][b] * u[1] + m[2][b] * u[2];
    r += x * x;
  }
  return r;
}
template <typename T>
__device__ __forceinline__ T norm2_mul(const T m[3][3], const T u[3]) {
  T r = (T)0;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const T x = m[a][0] * u[0] + m[a][1] * u[1] + m[a][2] * u[2];
    r += x * x;
  }
  return r;
}

// The element math's constants in T.  An FP64 argument rounded to FP32 is a
// vector conversion: its result goes back to an SGPR, so that the constants
// take no VGPRs through the Gauss-point loop.
__device__ __forceinline__ float uni(float v) { return __int_as_float(femx::uni(__float_as_int(v))); }
template <typename T>
struct ElemConst {
  T mu, mu2, mu23, mu43, mu103, rho, alpha, cnu, nu, f1;  // mu and its multiples by 2, 2/3, -4/3, 10/3
  int k2, k3, k4;
  __device__ __forceinline__ ElemConst(const SupgConst &k) {
    mu = c(k.mu);
    mu2 = c(2.0 * k.mu);
    mu23 = c(k.mu * (2.0 / 3.0));
    mu43 = c(k.mu * (-4.0 / 3.0));
    mu103 = c(k.mu * (10.0 / 3.0));
    rho = c(k.rho);
    alpha = c(k.alpha);
    nu = c((T)k.mu / (T)k.rho);
    cnu = c(k.cI * (k.mu / k.rho));
    f1 = k.k1 ? rho : (T)0;
    k2 = k.k2;
    k3 = k.k3;
    k4 = k.k4;
  }
  static __device__ __forceinline__ T c(double v) {
    if constexpr (sizeof(T) == 4) return uni((float)v);
    else return v;
  }
};

// A thread's extrema over its Gauss points, from which the columns D_TAU ..
// D_LCFL are made once: tau, lambda, 1 / el^2 and its products with lambda and
// u_0^2 (the squared a-CFL); NaN never wins.
template <typename T>
struct DiagAcc {
  T tau[2] = {(T)INFINITY, (T)-INFINITY}, lam[2] = {(T)INFINITY, (T)-INFINITY};
  double acfl2 = 0.0, el_2 = 0.0, lel_2 = 0.0;
  __device__ __forceinline__ void columns(double dt, double nu, double *dg) const {
    dg[0] = fmin(dg[0], (double)tau[0]);
    dg[1] = fmax(dg[1], (double)tau[1]);
    dg[D_LAM - D_TAU] = fmin(dg[D_LAM - D_TAU], (double)lam[0]);
    dg[D_LAM + 1 - D_TAU] = fmax(dg[D_LAM + 1 - D_TAU], (double)lam[1]);
    dg[D_VCFL - D_TAU] = fmax(dg[D_VCFL - D_TAU], 2.0 * nu * dt * el_2);
    dg[D_ACFL - D_TAU] = fmax(dg[D_ACFL - D_TAU], dt * sqrt(acfl2));
    dg[D_LCFL - D_TAU] = fmax(dg[D_LCFL - D_TAU], 2.0 * dt * lel_2);
  }
};

// Per-thread sums over the Gauss points.
template <typename T>
struct ElemAcc {
  T lam_int, reg;
  T S0, S[3];  // B-hat: the average's factor is sum of f2 alpha_k = S0 - 4/3 mu S_k
};

// B-hat: the element's part of the strain, eps_k = 5/3 D_k - div / 3 + q_k and
// tr eps = 2/3 div + r, with D_k = du_k/dx_k, from the averages P.
template <typename T, bool BHAT>
struct StrainConst {
  T q[3], r;
  __device__ __forceinline__ explicit StrainConst(const T P[3]) {
    r = BHAT ? (P[0] + P[1] + P[2]) * (T)(1.0 / 3.0) : (T)0;
#pragma unroll
    for (int b = 0; b < 3; b++) q[b] = BHAT ? r - (T)(2.0 / 3.0) * P[b] : (T)0;
  }
};

// One Gauss point (:1095-1507): from the velocity ug, its gradient gU[b][i] =
// du_i/dx_b, J and the velocity that G^-1 = J J^T is applied to (ul), |invJ
// u|^2 (t2), |G|^2 (gg), tr G and dv, the stabilization and the bulk modulus
// (lam, f3), c = (u.grad) u, and the matrix A of the node forces A DN_n (f2 S
// + f4 I: stress and grad-div).
template <typename T, bool BHAT, bool DIAG>
__device__ __forceinline__ void gauss_point(const ElemConst<T> &k, const T ug[3], const T gU[3][3], T div, T dv,
                                            const T J[3][3], const T ul[3], T t2, T gg, T trG,
                                            const StrainConst<T, BHAT> &sc, ElemAcc<T> &s, DiagAcc<T> &dg, T &f3,
                                            T c[3], T A[3][3]) {
  // eval_stabilization (:336-377), tau without the (2/dt)^2 term
  // (nu and cI nu apart: cI nu^2 alone leaves FP32's range before the term does)
  const T tau = rsqrt_e(t2 + (gg * k.nu) * k.cnu);
  const T nuC = recip(trG * tau);
  // eval_bulk_modulus (:382-441): lambda = alpha max(mu/rho, sqrt(u^T G^-1 u))
  const T l2 = sqrt_e(norm2_tmul(J, ul));
  const T lam = k.alpha * ((k.nu < l2) ? l2 : k.nu);
  s.reg += (k.nu > l2) ? (T)1 : (T)2;
  s.lam_int += lam * dv;
  if (DIAG) {
    // get_el_lengths_from_G (:756-790), el = 2 sqrt(o^T G^-1 o), o = u / |u|, and
    // the CFL extrema (:1187-1240), in FP64, as 1 / el^2 = |u|^2 / (4 |J^T u|^2).
    // Ahead of a front that spreads from rest u falls by orders of magnitude
    // per element: the squares of FP32 values are all in FP64's range, FP64
    // values are scaled into it for |J^T u|^2 (but not for |u|^2: below 1e-154
    // the reference's lengths are off by its rounding, and so are these)
    double w[3] = {(double)ul[0], (double)ul[1], (double)ul[2]}, Jd[3][3];
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
      for (int b = 0; b < 3; b++) Jd[r][b] = (double)J[r][b];
    double un2 = w[0] * w[0] + w[1] * w[1] + w[2] * w[2], q = norm2_tmul(Jd, w);
    if (sizeof(T) == 8 && un2 < 0x1p-800) {
      constexpr double f = 0x1p+700;
#pragma unroll
      for (int b = 0; b < 3; b++) w[b] *= f;
      un2 = un2 * f * f;
      q = norm2_tmul(Jd, w);
    }
    const double el_2 = un2 / (4.0 * q);
    const double u0 = (double)ul[0];
    dg.acfl2 = fmax(dg.acfl2, u0 * u0 * el_2);
    dg.el_2 = fmax(dg.el_2, el_2);
    dg.lel_2 = fmax(dg.lel_2, (double)lam * el_2);
    dg.tau[0] = fmin(dg.tau[0], tau);
    dg.tau[1] = fmax(dg.tau[1], tau);
    dg.lam[0] = fmin(dg.lam[0], lam);
    dg.lam[1] = fmax(dg.lam[1], lam);
  }
  // (u_g . grad) u
#pragma unroll
  for (int i = 0; i < 3; i++) c[i] = ug[0] * gU[0][i] + ug[1] * gU[1][i] + ug[2] * gU[2][i];
  f3 = k.k3 ? k.rho * tau * dv : (T)0;
  const T f4 = k.k4 ? k.rho * nuC * div * dv : (T)0, f2 = k.k2 ? dv : (T)0;
  // strain B u (:222-296): sum_n DN_nb u_ni = gU[b][i], and stress s_k = 2 mu
  // eps_k + lambda tr eps.  With B-hat the diagonal uses b_n = (avg_n -
  // DN_n)/3, whose sums are B_k = (P_k - D_k)/3, so eps_k = D_k - 2 B_k + sum_j
  // B_j, and the node forces are (f2 S + f4 I) DN_n + f2 avg_n o alpha with the
  // diagonal (5 s_k - ssum)/3 = 10/3 mu eps_k + 2/3 (lambda - mu) tr eps and
  // alpha_k = (ssum - 2 s_k)/3 = ((2 mu + lambda) tr eps - 4 mu eps_k)/3.
  if (BHAT) {
    const T w = div * (T)(1.0 / 3.0);
    const T trE = (T)(2.0 / 3.0) * div + sc.r;
    const T f2t = f2 * trE, f2s = f2 * k.mu103;
    const T d = f4 + f2t * ((T)(2.0 / 3.0) * lam - k.mu23);
    s.S0 += f2t * (lam * (T)(1.0 / 3.0) + k.mu23);
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const T eps = ((T)(5.0 / 3.0) * gU[i][i] + sc.q[i]) - w;
      A[i][i] = f2s * eps + d;
      s.S[i] += f2 * eps;
    }
  } else {
    const T f2s = f2 * k.mu2, d = f4 + f2 * (lam * div);
#pragma unroll
    for (int i = 0; i < 3; i++) A[i][i] = f2s * gU[i][i] + d;
  }
  const T f2m = f2 * k.mu;
  const T s3 = f2m * (gU[1][0] + gU[0][1]), s4 = f2m * (gU[2][1] + gU[1][2]), s5 = f2m * (gU[2][0] + gU[0][2]);
  A[0][1] = A[1][0] = s3;
  A[1][2] = A[2][1] = s4;
  A[0][2] = A[2][0] = s5;
}

// Element block blk of one mesh; its diagnostic row is eblk[row].
template <typename T, int NPE, bool BHAT, bool DYN, bool PRESS, bool PSEP, bool DIAG>
__device__ __forceinline__ void supg_block_run(const SupgArgs<T> &a, const int blk, const int row) {
  constexpr int NGP = Shape<NPE>::NGP;
  constexpr int EB = elems_for<NPE>();
  // hexa8: coordinates and velocities are staged as 1/8 of their values, the
  // factor of the element transforms (exact)
  constexpr double SC = NPE == 8 ? 0.125 : 1.0;
  __shared__ double sx[256], sy[256], sz[256], sm[256];
  __shared__ double su[256], sv[256], sw[256];
  __shared__ double pu[PSEP ? 256 : 1], pv[PSEP ? 256 : 1], pw[PSEP ? 256 : 1];
  __shared__ T sres[DYN ? 3 * NPE * EB : 1];
  // per local node what its update needs, fetched with its coordinates: run
  // begin and end, node, and its partial slot or -2 - BC record (-1: none).
  // Read at the end, with the force history and BC record behind them, they
  // cost three dependent round trips of every block's life: 2.1M hexa mixed
  // 269 -> 257 us, 85k hexa FP64 30.8 -> 28.9 us
  __shared__ int4 snode[DYN ? 256 : 1];
  const int tid = threadIdx.x;
  // (tested once the loads that need no result of it are on their way)
  const int halt_step = __builtin_nontemporal_load(a.halt);
  const int n0 = a.node_off[blk], nn = a.node_off[blk + 1] - n0;
  const int e0 = a.elem_off[blk], ne = a.elem_off[blk + 1] - e0;
  // hexa8: lanes 2 i and 2 i + 1 hold element i's z = -1 and z = 1 sides
  constexpr int EN = NPE == 8 ? 4 : NPE;  // nodes whose contributions the thread writes
  const int side = NPE == 8 ? tid & 1 : 0;
  const int el = NPE == 8 ? tid >> 1 : tid;
  const bool has_e = el < ne;
  const int e = e0 + el;
  T out[EN][3];
  // the thread's nodes: its element's, or those of its side, and node 0
  int own[EN], id0 = 0;
  ushort4 ps4 = make_ushort4(0, 0, 0, 0);
  double lam_prev = 0.0;
  if (has_e) {
    const uchar4 c4 = reinterpret_cast<const uchar4 *>(a.lconn)[NPE == 8 ? 2 * e + side : e];
    own[0] = c4.x; own[1] = c4.y; own[2] = c4.z; own[3] = c4.w;
    const int oth0 = NPE == 8 ? pair_swap(own[0]) : own[0];  // (every lane of a pair takes part)
    id0 = side ? oth0 : own[0];
    if (DYN) {
      // the thread's EN positions: its element's ushort4, or that of its side
      ps4 = reinterpret_cast<const ushort4 *>(a.lpos)[NPE == 8 ? 2 * e + side : e];
    }
    if (PRESS) lam_prev = a.lam[e];
  }
  if (tid < nn) {
    const int j = tid, g = a.loc_node[n0 + j];
    if (DYN) {
      const int psl = a.loc_pslot[n0 + j];
      const int b = a.lcsr_off[n0 + j] - e0 * NPE, e = a.lcsr_off[n0 + j + 1] - e0 * NPE;
      snode[j] = make_int4(b, e, g, psl >= 0 ? psl : -2 - a.node_rec[g]);
    }
    const double4 x = a.xyzm[g];
    sx[j] = SC * x.x; sy[j] = SC * x.y; sz[j] = SC * x.z; sm[j] = x.w;
    const double4 u = a.U[g];
    su[j] = SC * u.x; sv[j] = SC * u.y; sw[j] = SC * u.z;
    if (PSEP) {
      const double4 q = a.Upress[g];
      pu[j] = SC * q.x; pv[j] = SC * q.y; pw[j] = SC * q.z;
    }
  }
  if (halt_step < a.step_id) return;
  __syncthreads();
  double dg[11];
#pragma unroll
  for (int i = 0; i < 11; i++) dg[i] = d_identity(D_TAU + i);
  if (has_e) {
    const SupgConst &k = a.k;
    using S = ShapeT<T, NPE>;
    // element math in T: differences of the staged FP64 values are formed
    // in FP64 and rounded once, so FP32 gradients keep their digits.  The
    // physical derivatives DN = invJ dN/dxi are never formed: every term the
    // reference builds from DN (velocity gradient, divergence, B-hat strain,
    // the K2/K4 node forces, u.grad N) is the same arithmetic regrouped
    // through the local derivatives and 3x3 products per Gauss point.
    const ElemConst<T> kc(k);
    ElemAcc<T> acc = {};
    DiagAcc<T> da;
    double vol;                     // the element's volume
    const bool writes = side == 0;  // of the element's outputs
    // compute_pressure of the previous step (:498) from the mean divergence,
    // stored as soon as it is known: held through the Gauss-point loop, with
    // the fixed-DOF variants' second field formed behind the velocity's, it
    // spilled 332 B a lane in FP32 and 400 in FP64.  (FP64 without B-hat or
    // fixed DOFs fits with it: 386 against 391 us at 2.1M hexa)
    constexpr bool PHOLD = sizeof(T) == 8 && NPE == 8 && !BHAT && !PSEP;
    double div_held = 0.0;
    auto pressure = [&](double mean_div) {
      if (PRESS && writes) a.pres[e] = -lam_prev * mean_div;
    };
    if constexpr (NPE == 8) {
      const T q = S::GP(1, 0);  // 1 / sqrt 3
      // the lane's z direction: the map's handedness, and with it the sign of
      // det J (the Gauss weights are 1)
      const T sg = side ? (T)1 : (T)-1;
      const double q64 = ShapeT<double, 8>::GP(1, 0);
      auto field = [&](const double *v0, const double *v1, const double *v2, Tri<double> &f) {
        const double *v[3] = {v0, v1, v2};
#pragma unroll
        for (int b = 0; b < 3; b++) {
          double w[4];
#pragma unroll
          for (int n = 0; n < 4; n++) w[n] = v[b][own[n]] - v[b][id0];
          f.load(b, w, q64);
        }
      };
      // the map and the velocity, rounded to T once; the volume averages of DN
      // and P_k = sum_n avg_nk u_nk (B-hat), whose sum is the mean divergence
      // (compute_pressure :446-501; PSEP: of the state before the fixed-DOF
      // zeroing).  Each thread parks its nodes' averages (in the four (x, y)
      // coefficients of its side) in its own slots of the contribution
      // buffer, unused until the Gauss-point loop is over.
      Tri<T> X, V;
      T P[3] = {(T)0, (T)0, (T)0};
      {
        Tri<double> X64, V64;
        double P64[3];
        TriAvg av;
        field(sx, sy, sz, X64);
        av.form(X64, q64, (double)sg);
        vol = av.vol;
        X.from(X64);
        if constexpr (PSEP) {
          field(pu, pv, pw, V64);
          av.dot(V64, q64, P64);
          pressure(P64[0] + P64[1] + P64[2]);
        }
        field(su, sv, sw, V64);
        av.dot(V64, q64, P64);
        if constexpr (PHOLD) div_held = P64[0] + P64[1] + P64[2];
        else if constexpr (!PSEP) pressure(P64[0] + P64[1] + P64[2]);
#pragma unroll
        for (int b = 0; b < 3; b++) {
          P[b] = (T)P64[b];
          V64.c00[b] += 8.0 * (b == 0 ? su : b == 1 ? sv : sw)[id0];
        }
        V.from(V64);
        if constexpr (BHAT && DYN) {
#pragma unroll
          for (int b = 0; b < 3; b++) {
            sres[(0 * 3 + b) * SB + tid] = (T)av.z[b];
            sres[(1 * 3 + b) * SB + tid] = (T)(av.x[b] + av.xz[b]);
            sres[(2 * 3 + b) * SB + tid] = (T)(av.y[b] + av.yz[b]);
            sres[(3 * 3 + b) * SB + tid] = (T)av.xy[b];
          }
        }
      }
      if constexpr (DYN) {
        const StrainConst<T, BHAT> sc(P);
        TriSum<T> os;
        os.init();
#pragma unroll 1
        for (int iy = 0; iy < 2; iy++) {
          const T y = iy ? q : -q;
          X.at_y(y);
          V.at_y(y);
#pragma unroll 1
          for (int ix = 0; ix < 2; ix++) {
            const T x = ix ? q : -q;
            T J[3][3], iJ[3][3], L[3][3], ug[3], detJ;
            X.at_x(x, J);
            V.at_x(x, L);
            inv3(J, iJ, detJ);
            const T dv = detJ * sg;
            // velocity and its gradient gU[b][i] = du_i/dx_b
            T gU[3][3];
#pragma unroll
            for (int b = 0; b < 3; b++) {
              ug[b] = (V.c00[b] + y * V.A2[b]) + x * L[0][b];
#pragma unroll
              for (int i = 0; i < 3; i++) gU[b][i] = iJ[b][0] * L[0][i] + iJ[b][1] * L[1][i] + iJ[b][2] * L[2][i];
            }
            const T div = gU[0][0] + gU[1][1] + gU[2][2];
            T gg, trG, f3, c[3], A[3][3];
            metric3(iJ, gg, trG);
            // the metric's products with u pair the physical components with
            // the local directions, as the reference does
            const T ul[3] = {ug[0], ug[1], sg * ug[2]};
            gauss_point<T, BHAT, DIAG>(kc, ug, gU, div, dv, J, ul, norm2_mul(iJ, ul), gg, trG, sc, acc, da, f3, c, A);
            const T f1 = kc.f1 * dv;
            // A DN_n + f3 c (u.grad N_n) in the local derivatives:
            // (A + f3 c (x) u) invJ dN_n
            T v[3], Tl[3][3];
#pragma unroll
            for (int i = 0; i < 3; i++) {
              v[i] = f1 * c[i];
              const T fc = f3 * c[i];
              const T a0 = A[i][0] + fc * ug[0], a1 = A[i][1] + fc * ug[1], a2 = A[i][2] + fc * ug[2];
#pragma unroll
              for (int l = 0; l < 3; l++) Tl[i][l] = a0 * iJ[0][l] + a1 * iJ[1][l] + a2 * iJ[2][l];
            }
            os.add(x, y, v, Tl);
          }
        }
        acc.lam_int = pair_sum(acc.lam_int);
        acc.reg = pair_sum(acc.reg);
#pragma unroll
        for (int b = 0; b < 3; b++) {
          T m[4];
          os.nodes(b, q, m);
          if constexpr (BHAT) {
            const T al = pair_sum(acc.S0 + kc.mu43 * acc.S[b]);
#pragma unroll
            for (int i = 0; i < 4; i++) m[i] += sres[(i * 3 + b) * SB + tid] * al;
          }
          // nodes (x, y) = (-, -), (+, -), (+, +), (-, +) of the lane's side
          const T p = m[0] - m[2], r = m[0] + m[2], t = m[1] - m[3], w = m[1] + m[3];
          out[0][b] = p - t;
          out[1 % EN][b] = p + t;
          out[2 % EN][b] = r + w;
          out[3 % EN][b] = r - w;
        }
      }
    } else {
      // tet4 (femTetra4, N3 = 1 - sum xi): the Jacobian, its inverse, the
      // velocity gradient and the metric are the same at every Gauss point,
      // and so are the physical derivatives, DN_n = column n of invJ: the
      // node forces are one matrix K = sum_g (A + f3 c (x) u) applied to
      // them, plus the convection's values.
      T J[3][3], iJ[3][3], L[3][3], gU[3][3], detJ, u[4][3];
      {
        const double *xs[3] = {sx, sy, sz}, *us[3] = {su, sv, sw};
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
          for (int b = 0; b < 3; b++) {
            J[r][b] = (T)(xs[b][own[r]] - xs[b][own[3]]);
            L[r][b] = (T)(us[b][own[r]] - us[b][own[3]]);
          }
#pragma unroll
        for (int n = 0; n < 4; n++)
#pragma unroll
          for (int b = 0; b < 3; b++) u[n][b] = (T)(us[b][own[n]] - us[b][id0]);
      }
      inv3(J, iJ, detJ);
#pragma unroll
      for (int b = 0; b < 3; b++)
#pragma unroll
        for (int i = 0; i < 3; i++) gU[b][i] = iJ[b][0] * L[0][i] + iJ[b][1] * L[1][i] + iJ[b][2] * L[2][i];
      const T dv = detJ * S::W(), div = gU[0][0] + gU[1][1] + gU[2][2];
      vol = (double)((T)NGP * dv);
      const T U0[3] = {(T)su[id0], (T)sv[id0], (T)sw[id0]};
      if constexpr (PRESS && PSEP) {
        const double *qs[3] = {pu, pv, pw};
        T dp = (T)0;
#pragma unroll
        for (int b = 0; b < 3; b++)
#pragma unroll
          for (int r = 0; r < 3; r++) dp += iJ[b][r] * (T)(qs[b][own[r]] - qs[b][own[3]]);
        pressure(dp);
      } else if constexpr (PRESS) {
        pressure(div);
      }
      if constexpr (DYN) {
        T gg, trG, K[3][3], cN[4][3];
        const T P[3] = {(T)0, (T)0, (T)0};
        const StrainConst<T, false> sc(P);
        metric3(iJ, gg, trG);
#pragma unroll
        for (int i = 0; i < 3; i++) {
          K[i][0] = K[i][1] = K[i][2] = (T)0;
          cN[0][i] = cN[1][i] = cN[2][i] = cN[3][i] = (T)0;
        }
#pragma unroll 1
        for (int g = 0; g < NGP; g++) {
          T ug[3], f3, c[3], A[3][3];
#pragma unroll
          for (int b = 0; b < 3; b++)
            ug[b] = U0[b] + (S::N(g, 1) * u[1][b] + S::N(g, 2 % NPE) * u[2][b] + S::N(g, 3 % NPE) * u[3][b]);
          gauss_point<T, false, DIAG>(kc, ug, gU, div, dv, J, ug, norm2_mul(iJ, ug), gg, trG, sc, acc, da, f3, c, A);
          const T f1 = kc.f1 * dv;
#pragma unroll
          for (int i = 0; i < 3; i++) {
            const T fc = f3 * c[i], vc = f1 * c[i];
#pragma unroll
            for (int b = 0; b < 3; b++) K[i][b] += A[i][b] + fc * ug[b];
#pragma unroll
            for (int n = 0; n < 4; n++) cN[n][i] += vc * S::N(g, n % NPE);
          }
        }
#pragma unroll
        for (int i = 0; i < 3; i++) {
          T f[3];
#pragma unroll
          for (int n = 0; n < 3; n++) {
            f[n] = K[i][0] * iJ[0][n] + K[i][1] * iJ[1][n] + K[i][2] * iJ[2][n];
            out[n % EN][i] = cN[n][i] + f[n];
          }
          out[3 % EN][i] = cN[3][i] - (f[0] + f[1] + f[2]);
        }
      }
    }
    if constexpr (PHOLD) pressure(div_held);
    if (DYN) {
      const double lame = (double)acc.lam_int / vol;  // :1446
      if (writes) {
        a.lam[e] = lame;
        a.regime[e] = (double)acc.reg / NGP;
      }
      if (DIAG) {
        da.columns(k.dt, (double)kc.nu, dg);
        const double cE = (k.mu * (3 * lame + 2 * k.mu)) / (lame + k.mu), cnu = lame / (2 * (lame + k.mu));
        dg[D_E - D_TAU] = fmin(dg[D_E - D_TAU], cE);
        dg[D_E + 1 - D_TAU] = fmax(dg[D_E + 1 - D_TAU], cE);
        dg[D_NU - D_TAU] = fmin(dg[D_NU - D_TAU], cnu);
        dg[D_NU + 1 - D_TAU] = fmax(dg[D_NU + 1 - D_TAU], cnu);
      }
      if constexpr (!(BHAT && NPE == 8)) {
        const T mdt = (T)(-k.dt * SC);
        const int ps[4] = {ps4.x, ps4.y, ps4.z, ps4.w};
#pragma unroll
        for (int n = 0; n < EN; n++)
#pragma unroll
          for (int i = 0; i < 3; i++) sres[i * (NPE * EB) + ps[n]] = mdt * out[n][i];
      }
    }
  }
  if (!DYN) return;
  if constexpr (BHAT && NPE == 8) {
    // every thread has read its averages back from sres
    __syncthreads();
    if (has_e) {
      const T mdt = (T)(-a.k.dt * SC);
      const int ps[4] = {ps4.x, ps4.y, ps4.z, ps4.w};
#pragma unroll
      for (int n = 0; n < EN; n++)
#pragma unroll
        for (int i = 0; i < 3; i++) sres[i * (NPE * EB) + ps[n]] = mdt * out[n][i];
    }
  }
  if (DIAG) block_diag_store<SB, 11>(dg, D_TAU, a.eblk + (long)row * D_COLS);
  // the force history and BC record of a node this block completes are on
  // their way while the contributions settle
  const int4 mine = tid < nn ? snode[tid] : make_int4(0, 0, 0, 0);
  const bool complete = tid < nn && mine.w < 0, has_bc = complete && mine.w <= -2;
  double4 fp = make_double4(0, 0, 0, 0);
  BCRecord bc = {};
  if (complete && !a.k.euler_step) fp = a.Fprev[mine.z];
  if (has_bc) bc = a.rec[-2 - mine.w];
  __syncthreads();
  // velocity extrema and max |u|^2 of the new states this block completes
  // (get_solution_extrema :604-655), into the node columns of its row
  double nv[6], nm2[1] = {0.0};
#pragma unroll
  for (int i = 0; i < 6; i++) nv[i] = d_identity(D_UMIN + i);
  if (tid < nn) {
    const int j = tid;
    // the node's contributions summed in FP64, or in FP32 with f32sum
    double F[3] = {0.0, 0.0, 0.0};
    const int s0 = mine.x, s1 = mine.y;
    if (a.f32sum) {
      float Ft[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll 4
      for (int s = s0; s < s1; s++) {
        Ft[0] += (float)sres[0 * (NPE * EB) + s];
        Ft[1] += (float)sres[1 * (NPE * EB) + s];
        Ft[2] += (float)sres[2 * (NPE * EB) + s];
      }
      F[0] = Ft[0];
      F[1] = Ft[1];
      F[2] = Ft[2];
    } else {
#pragma unroll 4
      for (int s = s0; s < s1; s++) {
        F[0] += (double)sres[0 * (NPE * EB) + s];
        F[1] += (double)sres[1 * (NPE * EB) + s];
        F[2] += (double)sres[2 * (NPE * EB) + s];
      }
    }
    if (complete) {
      const int g = mine.z;
      double4 next, pst, fst;
      supg_node(F, fp, sm[j], make_double4(su[j] * (1.0 / SC), sv[j] * (1.0 / SC), sw[j] * (1.0 / SC), 0.0), a.k,
                has_bc, bc, a.row_off, a.rows, a.err, next, pst, fst);
      a.Un[g] = next;
      if (a.Unp) a.Unp[g] = pst;
      a.Fprev[g] = fst;
      node_extrema(next, nv, nm2[0]);
    } else {
      const int psl = mine.w;
      if (a.f32sum)
        static_cast<float4 *>(a.partials)[psl] = make_float4((float)F[0], (float)F[1], (float)F[2], 0.0f);
      else
        static_cast<double4 *>(a.partials)[psl] = make_double4(F[0], F[1], F[2], 0.0);
    }
  }
  exit_check(nm2[0], a.k, a.halt, a.step_id);
  if (a.want_row) block_node_store<SB>(nv, nm2[0], a.eblk + (long)row * D_COLS);
}

// Waves per SIMD: every FP32 hexa8 variant fits three (168 VGPRs) without
// spills (with diagnostics 0 to 20 B a lane, 68 in the first step without
// B-hat) as long as its two Gauss points of one y are not unrolled; four spill
// 100 B per lane (328 against 270 us at 2.1M hexa).  The others are bound to
// two (FP64 hexa8 spills 84 B with B-hat, 156 with diagnostics, none without
// either).  A step of 2.1M hexa, FP32 / FP64: plain 278 / 478, fixed DOFs 302 /
// 527, without B-hat 265 / 386, plain with diagnostics 388 / 755 us.
#define SUPG_BLOCK_WAVES(T, NPE) (sizeof(T) == 4 && NPE == 8 ? 3 : 2)
template <typename T, int NPE, bool BHAT, bool DYN, bool PRESS, bool PSEP, bool DIAG>
__global__ __launch_bounds__(SB, SUPG_BLOCK_WAVES(T, NPE)) void supg_block(SupgArgs<T> a) {
  supg_block_run<T, NPE, BHAT, DYN, PRESS, PSEP, DIAG>(a, xcd_block(blockIdx.x, a.nblk), blockIdx.x);
}


// The log row of one step, made for the last step of a call (and for every
// step while the element diagnostics are on: the l-CFL column is a running
// maximum since the first step, the reference sets l_CFL_max once before its
// time loop, :996, and resets only the v- and a-CFL maxima per step,
// :1078-1079; it is carried in *lcfl).  Reduction of the per-workgroup rows
// in two stages: 32 workgroups each fold a strided share of the rows, all
// columns at once in registers, into one partial row; one wave folds the
// partial rows with all of its loads in flight together.  Up to
// DIAG_ONE_PASS rows one workgroup does both.  A separate launch after the
// fix-up: folded by the fix-up's last workgroup instead, each of its
// workgroups paid a device-scope fence (22 us against 6 us at 85k hexa).
constexpr int DIAG_PARTS = 32;
constexpr int DIAG_ONE_PASS = 2048;
__device__ __forceinline__ void row_store(int c, double v, double *row, double *lcfl, int step) {
  if (c == D_LCFL) {
    v = fmax(v, *lcfl);
    *lcfl = v;
  }
  row[c] = v;
  if (c == 0) row[D_STEP] = (double)step;
}
// One workgroup of 256 threads folds the rows of workgroups part, part +
// nparts, ... into out[0 .. D_COLS), or into the log row (lcfl not null).
__device__ __forceinline__ void diag_fold(const double *eblk, int ne_blk, const double *nblk, int nn_blk,
                                          int with_elem, double *out, double *lcfl, int step, int part, int nparts) {
  double m[D_COLS];
#pragma unroll
  for (int c = 0; c < D_COLS; c++) m[c] = d_identity(c);
  const int stride = nparts * 256;
  // node columns: the fix-up's rows and the element blocks' rows; element
  // columns: the element blocks' rows when the element diagnostics are on
  for (int b = part * 256 + threadIdx.x; b < nn_blk; b += stride) {
#pragma unroll
    for (int c = 0; c < D_COLS; c++)
      if (c < 6 || c == D_UMOD) {
        const double x = nblk[(long)b * D_COLS + c];
        m[c] = d_is_min(c) ? fmin(m[c], x) : fmax(m[c], x);
      }
  }
  for (int b = part * 256 + threadIdx.x; b < ne_blk; b += stride) {
#pragma unroll
    for (int c = 0; c < D_COLS; c++)
      if (with_elem || c < 6 || c == D_UMOD) {
        const double x = eblk[(long)b * D_COLS + c];
        m[c] = d_is_min(c) ? fmin(m[c], x) : fmax(m[c], x);
      }
  }
  __shared__ double red[4][D_COLS];
#pragma unroll
  for (int c = 0; c < D_COLS; c++) {
    for (int off = 32; off > 0; off >>= 1) {
      const double o = __shfl_xor(m[c], off);
      m[c] = d_is_min(c) ? fmin(m[c], o) : fmax(m[c], o);
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][c] = m[c];
  }
  __syncthreads();
  if (threadIdx.x < D_COLS) {
    const int c = threadIdx.x;
    double v = red[0][c];
    for (int w = 1; w < 4; w++) v = d_is_min(c) ? fmin(v, red[w][c]) : fmax(v, red[w][c]);
    if (lcfl) row_store(c, v, out, lcfl, step);
    else out[c] = v;
  }
}

__global__ __launch_bounds__(256) void supg_diag_partial(const double *eblk, int ne_blk, const double *nblk,
                                                         int nn_blk, int with_elem, double *part, double *lcfl,
                                                         const int *halt, int step) {
  if (halted(halt, step)) return;
  diag_fold(eblk, ne_blk, nblk, nn_blk, with_elem, lcfl ? part : part + (long)blockIdx.x * D_COLS, lcfl, step,
            blockIdx.x, gridDim.x);
}

__global__ __launch_bounds__(64) void supg_diag_final(const double *part, int np, double *row, double *lcfl,
                                                      const int *halt, int step) {
  if (halted(halt, step)) return;
  if (threadIdx.x < D_COLS) {
    const int c = threadIdx.x;
    double x[DIAG_PARTS];
#pragma unroll
    for (int q = 0; q < DIAG_PARTS; q++) x[q] = q < np ? part[(long)q * D_COLS + c] : d_identity(c);
    double v = d_identity(c);
#pragma unroll
    for (int q = 0; q < DIAG_PARTS; q++) v = d_is_min(c) ? fmin(v, x[q]) : fmax(v, x[q]);
    row_store(c, v, row, lcfl, step);
  }
}

// The rows of a state's velocity extrema from the state itself (the log row
// of a step that the exit condition made the last one of its call).
__global__ __launch_bounds__(256) void supg_state_rows(int N, const double4 *U, double *nblk) {
  double nv[6], m2 = 0.0;
#pragma unroll
  for (int i = 0; i < 6; i++) nv[i] = d_identity(D_UMIN + i);
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n < N) node_extrema(U[n], nv, m2);
  block_node_store<256>(nv, m2, nblk + (long)blockIdx.x * D_COLS);
}

struct SupgFix {
  int n_sh;
  const int *sh_node, *sh_off, *sh_slot;
  const int4 *sh_first4;  // each shared node's first 4 slots
  const void *partials;  // T4 records of the block kernel
  // per shared node, contiguous: its lumped mass and its BC record or -1
  // (the fix-up then gathers no node-indexed metadata)
  const double *sh_m;
  const int *sh_rec;
  const double4 *U;
  double4 *Un, *Unp, *Fprev;
  const BCRecord *rec;
  const int *row_off;
  const double4 *rows;
  int *err;
  int *halt;
  int step_id;
  int want_row;  // the step's log row is made: write the workgroup's row
  double *nblk;  // [workgroups][D_COLS]: node columns of each workgroup's row
  SupgConst k;
};

template <typename T>
__device__ __forceinline__ void fixup_node(const SupgFix &a, int s, bool stopped, double nv[6], double &nm2);

// Fix-up workgroup wg of one mesh.
template <typename T>
__device__ __forceinline__ void supg_fixup_run(const SupgFix &a, const int wg) {
  const int halt_step = __builtin_nontemporal_load(a.halt);
  const int s = wg * 256 + (int)threadIdx.x;
  double nv[6], nm2[1] = {0.0};
#pragma unroll
  for (int i = 0; i < 6; i++) nv[i] = d_identity(D_UMIN + i);
  if (s < a.n_sh) fixup_node<T>(a, s, halt_step < a.step_id, nv, nm2[0]);
  if (halt_step < a.step_id) return;
  exit_check(nm2[0], a.k, a.halt, a.step_id);
  // this workgroup's row of velocity extrema and max |u|^2 (:604-655)
  if (a.want_row) block_node_store<256>(nv, nm2[0], a.nblk + (long)wg * D_COLS);
}

template <typename T>
__global__ __launch_bounds__(256) void supg_fixup(SupgFix a) {
  supg_fixup_run<T>(a, blockIdx.x);
}

template <typename T>
__device__ __forceinline__ void fixup_node(const SupgFix &a, int s, bool stopped, double nv[6], double &nm2) {
  using T4 = typename Vec4<T>::type;
  const T4 *partials = static_cast<const T4 *>(a.partials);
  // two rounds of independent loads: what s indexes (incl. its first 4
  // slots, the last repeated when it has fewer), then the node's state and
  // those slots' partials (most nodes have at most 4) and BC record.  The
  // exit condition, loaded before them, is tested when all are on their way
  // (a round trip less: 2.1M hexa 62.4 -> 60.7 us, 85k 6.7 -> 6.0 us)
  constexpr int FIX_BATCH = 4;
  const int g = a.sh_node[s];
  const int q0 = a.sh_off[s], q1 = a.sh_off[s + 1];
  const int4 f4 = a.sh_first4[s];
  const int fs[FIX_BATCH] = {f4.x, f4.y, f4.z, f4.w};
  const double4 fp = a.k.euler_step ? make_double4(0, 0, 0, 0) : a.Fprev[g];
  const double im = a.sh_m[s];
  const double4 u = a.U[g];
  const int rec = a.sh_rec[s];
  T4 p[FIX_BATCH];
#pragma unroll
  for (int j = 0; j < FIX_BATCH; j++) p[j] = partials[fs[j]];
  BCRecord bc = {};
  if (rec >= 0) bc = a.rec[rec];
  if (stopped) return;
  double F[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int j = 0; j < FIX_BATCH; j++)
    if (q0 + j < q1) {
      F[0] += (double)p[j].x;
      F[1] += (double)p[j].y;
      F[2] += (double)p[j].z;
    }
  for (int q = q0 + FIX_BATCH; q < q1; q++) {
    const T4 r = partials[a.sh_slot[q]];
    F[0] += (double)r.x;
    F[1] += (double)r.y;
    F[2] += (double)r.z;
  }
  double4 next, pst, fst;
  supg_node(F, fp, im, u, a.k, rec >= 0, bc, a.row_off, a.rows, a.err, next, pst, fst);
  a.Un[g] = next;
  if (a.Unp) a.Unp[g] = pst;
  a.Fprev[g] = fst;
  node_extrema(next, nv, nm2);
}

// form_lumped_mass (:507-598): element row sums of the Bubnov mass
// rho N_a N_b detJ w, accumulated over Gauss points then over b, gathered
// per node in ascending original element order.
template <int NPE>
__global__ __launch_bounds__(256) void supg_mass(int N, const int *g_off, const int *g_slot, const int *conn,
                                                 const double4 *xyz, double rho, double4 *xyzm) {
  constexpr int NGP = Shape<NPE>::NGP;
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  double acc = 0.0;
  for (int s = g_off[n]; s < g_off[n + 1]; s++) {
    const int e = g_slot[s] / NPE, a = g_slot[s] % NPE;
    double dx[NPE][3];
    const double4 x0 = xyz[conn[(long)e * NPE]];
#pragma unroll
    for (int c = 0; c < NPE; c++) {
      const double4 x = xyz[conn[(long)e * NPE + c]];
      dx[c][0] = x.x - x0.x;
      dx[c][1] = x.y - x0.y;
      dx[c][2] = x.z - x0.z;
    }
    double detJ[NGP];
    for (int g = 0; g < NGP; g++) {
      double DN[NPE][3], iJ[3][3];
      kinematics<NPE>(g, dx, DN, detJ[g], iJ);
    }
    double row = 0.0;
    for (int b = 0; b < NPE; b++) {
      double bm = 0.0;
      for (int g = 0; g < NGP; g++) bm += rho * Shape<NPE>::N(g, a) * Shape<NPE>::N(g, b) * detJ[g] * Shape<NPE>::W();
      row += bm;
    }
    acc += row;
  }
  const double4 x = xyz[n];
  xyzm[n] = make_double4(x.x, x.y, x.z, acc);
}

// Per shared node, its lumped mass and BC record in one contiguous array each.
__global__ __launch_bounds__(256) void supg_shared_meta(int n_sh, const int *sh_node, const double4 *xyzm,
                                                        const int *node_rec, double *sh_m, int *sh_rec) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n_sh) return;
  const int g = sh_node[s];
  sh_m[s] = xyzm[g].w;
  sh_rec[s] = node_rec[g];
}

__global__ void supg_bc_only(int nrec, const int *rec_node, const BCRecord *rec, const int *row_off, const double4 *rows,
                             double t, double4 *U, int *err) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nrec) return;
  const int n = rec_node[i];
  double4 q = U[n];
  double u = q.x, v = q.y, w = q.z;
  apply_bc(rec[i], row_off, rows, t, u, v, w, nullptr, err);
  U[n] = make_double4(u, v, w, 0.0);
}

__global__ void block_to_orig(int E, const int *perm, const double *src, double *dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < E) dst[perm[i]] = src[i];
}

// Node states (x, y, z, 0) as [N][3]: 3 N values, one per thread.
__global__ __launch_bounds__(256) void pack3(int N, const double *U, double *dst) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < 3L * N) dst[i] = U[i / 3 * 4 + i % 3];
}

}  // namespace

}  // namespace femx

using namespace femx;

struct femx_supg {
  Mesh *mesh = nullptr;
  femx_supg_params p{};
  hipStream_t st = nullptr;
  BCDev bc;
  DevBuf<int> rec_node;
  DevBuf<double4> xyzm, U[2], Up[2], Fprev, partials;
  DevBuf<double> sh_m;  // per shared node: lumped mass
  DevBuf<int> sh_rec;   // per shared node: BC record or -1
  DevBuf<double> lam, regime, pres, scratch;
  DevBuf<double> row, eblk, nblk;   // [D_ROW] log row, then the running l-CFL maximum; per-block rows
  DevBuf<double> dpart;             // [DIAG_PARTS][D_COLS] partial rows of the reduction
  DevBuf<int> halt;
  int cur = 0;
  long loop_time = 0;
  double time = 0.0;
  bool press_pending = false;
  bool diag_enabled = false;
  bool halted = false;  // the exit condition fired; the solve is over
  // steps enqueued and not yet checked for the exit condition
  long pend_n = 0, pend_first = 0;
  double pend_t0 = 0.0;
  int pend_cur0 = 0;
  KernelTimer timer;
  // member of a union of handles (femx_supg_union_*): its time, parity,
  // step number and steps left live on the device while it is a member
  femx_supg_union *in_union = nullptr;
  int u_left = 0;
  DevBuf<unsigned char> dyn;  // one SupgDyn
};

namespace {

SupgConst supg_const(const femx_supg *s, double t, bool euler_step) {
  SupgConst k;
  k.rho = s->p.rho;
  k.mu = s->p.mu;
  k.alpha = s->p.alpha;
  k.cI = s->p.cI;
  k.dt = s->p.dt;
  k.t = t;
  k.exit2 = s->p.exit_condition * s->p.exit_condition;
  k.euler_step = euler_step ? 1 : 0;
  k.fixed = s->p.fixed_dofs;
  k.k1 = s->p.k1;
  k.k2 = s->p.k2;
  k.k3 = s->p.k3;
  k.k4 = s->p.k4;
  return k;
}

template <typename T>
SupgArgs<T> supg_args(femx_supg *s, bool euler_step, double t) {
  Mesh &m = *s->mesh;
  Blocks &b = m.blk;
  SupgArgs<T> a;
  a.nblk = b.nb;
  a.E = m.E;
  a.elem_off = b.d_elem_off.p;
  a.node_off = b.d_node_off.p;
  a.loc_node = b.d_loc_node.p;
  a.loc_pslot = b.d_loc_pslot.p;
  a.lcsr_off = b.d_lcsr_off.p;
  a.lpos = b.d_lcsr.p;
  a.lconn = b.d_lconn.p;
  a.xyzm = s->xyzm.p;
  a.U = s->U[s->cur].p;
  a.Upress = s->p.fixed_dofs ? s->Up[s->cur].p : s->U[s->cur].p;
  a.Un = s->U[s->cur ^ 1].p;
  a.Unp = s->p.fixed_dofs ? s->Up[s->cur ^ 1].p : nullptr;
  a.Fprev = s->Fprev.p;
  a.partials = s->partials.p;
  a.f32sum = f32_sum(s->p.precision) ? 1 : 0;
  a.lam = s->lam.p;
  a.regime = s->regime.p;
  a.pres = s->pres.p;
  a.node_rec = s->bc.node_rec.p;
  a.rec = s->bc.rec.p;
  a.row_off = s->bc.row_off.p;
  a.rows = s->bc.rows.p;
  a.err = s->bc.err.p;
  a.eblk = s->eblk.p;
  a.halt = s->halt.p;
  a.step_id = (int)s->loop_time;
  a.want_row = 0;
  a.k = supg_const(s, t, euler_step);
  return a;
}

template <typename T, int NPE, bool BHAT>
void launch_supg_t(femx_supg *s, SupgArgs<T> &a, bool dyn, bool press, bool diag) {
  const int grd = s->mesh->blk.nb;
  const bool psep = press && s->p.fixed_dofs != 0;
#define L(D, P, PS, G) supg_block<T, NPE, BHAT, D, P, PS, G><<<grd, SB, 0, s->st>>>(a)
  if (!dyn) {
    if (psep) L(false, true, true, false);
    else L(false, true, false, false);
    return;
  }
  if (press) {
    if (psep) {
      if (diag) L(true, true, true, true); else L(true, true, true, false);
    } else {
      if (diag) L(true, true, false, true); else L(true, true, false, false);
    }
  } else {
    if (diag) L(true, false, false, true); else L(true, false, false, false);
  }
#undef L
}

template <typename T>
void launch_supg_npe(femx_supg *s, SupgArgs<T> &a, bool dyn, bool press, bool diag) {
  if (s->mesh->npe == 8) {
    if (s->p.use_bhat) launch_supg_t<T, 8, true>(s, a, dyn, press, diag);
    else launch_supg_t<T, 8, false>(s, a, dyn, press, diag);
  } else {
    launch_supg_t<T, 4, false>(s, a, dyn, press, diag);
  }
}

// Algorithmic bytes of one element launch: u8 connectivity + u16 positions
// (3 B per corner), coordinates + mass and the state read once per node, the
// next state and nodal history written once per node, el_lam / regime /
// pressure (read + 3 writes) per element.
double supg_bytes(const femx_supg *s) {
  const double E = s->mesh->E, N = s->mesh->N;
  return E * (3.0 * s->mesh->npe + 32.0) + N * (32.0 + 32.0 + 32.0 + 32.0);
}

femx_status launch_supg(femx_supg *s, bool dyn, bool press, bool euler_step, double t, bool want_row) {
  const char *name = dyn ? (press ? "supg_block_press" : "supg_block") : "supg_press";
  TimedLaunch tl(s->timer, s->timer.kind(name, supg_bytes(s)), s->st);
  if (f32_elem(s->p.precision)) {
    SupgArgs<float> a = supg_args<float>(s, euler_step, t);
    a.want_row = want_row;
    launch_supg_npe<float>(s, a, dyn, press, s->diag_enabled);
  } else {
    SupgArgs<double> a = supg_args<double>(s, euler_step, t);
    a.want_row = want_row;
    launch_supg_npe<double>(s, a, dyn, press, s->diag_enabled);
  }
  FEMX_HIP(hipGetLastError());
  return FEMX_OK;
}

SupgFix fix_args(femx_supg *s, bool euler_step, double t) {
  Blocks &b = s->mesh->blk;
  SupgFix a;
  a.n_sh = b.n_sh;
  a.sh_node = b.d_sh_node.p;
  a.sh_off = b.d_sh_off.p;
  a.sh_slot = b.d_sh_slot.p;
  a.sh_first4 = b.d_sh_first4.p;
  a.partials = s->partials.p;
  a.sh_m = s->sh_m.p;
  a.sh_rec = s->sh_rec.p;
  a.U = s->U[s->cur].p;
  a.Un = s->U[s->cur ^ 1].p;
  a.Unp = s->p.fixed_dofs ? s->Up[s->cur ^ 1].p : nullptr;
  a.Fprev = s->Fprev.p;
  a.rec = s->bc.rec.p;
  a.row_off = s->bc.row_off.p;
  a.rows = s->bc.rows.p;
  a.err = s->bc.err.p;
  a.halt = s->halt.p;
  a.step_id = (int)s->loop_time;
  a.want_row = 0;
  a.nblk = s->nblk.p;
  a.k = supg_const(s, t, euler_step);
  return a;
}

femx_status launch_fix(femx_supg *s, bool euler_step, double t, bool want_row) {
  Blocks &b = s->mesh->blk;
  if (b.n_sh == 0) return FEMX_OK;
  const bool f32p = f32_sum(s->p.precision);  // float4 partial records
  const double rec_bytes = f32p ? 16.0 : 32.0;  // one partial slot record, written and read
  TimedLaunch tl(s->timer, s->timer.kind("supg_fixup", b.sh_off[b.n_sh] * rec_bytes * 2 + b.n_sh * 200.0), s->st);
  SupgFix a = fix_args(s, euler_step, t);
  a.want_row = want_row;
  if (f32p) supg_fixup<float><<<grid_for(b.n_sh, 256), 256, 0, s->st>>>(a);
  else supg_fixup<double><<<grid_for(b.n_sh, 256), 256, 0, s->st>>>(a);
  FEMX_HIP(hipGetLastError());
  return FEMX_OK;
}

// Workgroups whose rows (nblk) a step's fix-up writes.
int fix_rows(const femx_supg *s) { return s->mesh->blk.n_sh ? grid_for(s->mesh->blk.n_sh, 256) : 0; }

// The log row of step `step` from ne element-block rows and nn rows of nblk.
femx_status launch_row(femx_supg *s, int ne, int nn, bool with_elem, int step) {
  double *row = s->row.p, *lcfl = s->row.p + D_ROW;
  if (ne + nn <= DIAG_ONE_PASS) {
    supg_diag_partial<<<1, 256, 0, s->st>>>(s->eblk.p, ne, s->nblk.p, nn, with_elem, row, lcfl, s->halt.p, step);
  } else {
    supg_diag_partial<<<DIAG_PARTS, 256, 0, s->st>>>(s->eblk.p, ne, s->nblk.p, nn, with_elem, s->dpart.p, nullptr,
                                                     s->halt.p, step);
    supg_diag_final<<<1, 64, 0, s->st>>>(s->dpart.p, DIAG_PARTS, row, lcfl, s->halt.p, step);
  }
  FEMX_HIP(hipGetLastError());
  return FEMX_OK;
}

femx_status flush_pressure(femx_supg *s) {
  if (!s->press_pending) return FEMX_OK;
  femx_status r = launch_supg(s, false, true, true, s->time, false);
  if (r != FEMX_OK) return r;
  s->press_pending = false;
  return FEMX_OK;
}

// Reads the pieces back together with the BC error flag.
femx_status read_checked(femx_supg *s, ReadPiece *p, int n) {
  int e = 0;
  p[n] = {&e, s->bc.err.p, sizeof(int)};
  const femx_status r = read_back(s->mesh->device, s->st, p, n + 1);
  if (r != FEMX_OK) return r;
  if (e) return set_error("Could not find time in femUtils::interpTableData."), FEMX_ERR_BC;
  return FEMX_OK;
}

}  // namespace

extern "C" femx_status femx_supg_create(femx_mesh *mh, const femx_bc_desc *bc, const femx_supg_params *p,
                                        femx_supg **out) {
  if (!mh || !p || !out) return set_error("null argument"), FEMX_ERR_ARG;
  Mesh &m = mh->m;
  if (m.npe == 4 && p->use_bhat)
    return set_error("B-hat needs hexa8 (eval_avg_shapeDeriv reads 8 nodes)"), FEMX_ERR_UNSUPPORTED;
  if (p->fixed_dofs < 0 || p->fixed_dofs > 6) return set_error("ERROR: Invalid global fixed DOFs string."), FEMX_ERR_ARG;
  if (!valid_precision(p->precision)) return set_error("precision"), FEMX_ERR_ARG;
  if (!(p->dt > 0.0) || p->rho == 0.0) return set_error("parameters"), FEMX_ERR_ARG;
  const int elems = m.npe == 4 ? elems_for<4>() : elems_for<8>();
  if (m.blk.B > elems || m.blk.max_local > 256)
    return set_error("element blocks do not fit the SUPG workgroup"), FEMX_ERR_ARG;
  femx_status r;
  if ((r = upload_tables(m.device)) != FEMX_OK) return r;
  femx_supg *s = new femx_supg();
  s->mesh = &m;
  s->p = *p;
  auto fail = [&](femx_status st) {
    femx_supg_destroy(s);
    return st;
  };
  if (!(s->st = stream_get())) return fail(FEMX_ERR_HIP);
  if ((r = s->bc.build(bc, m.N, false, s->st)) != FEMX_OK) return fail(r);
  if ((r = s->rec_node.upload(s->bc.h_rec_node.data(), s->bc.h_rec_node.size(), s->st)) != FEMX_OK) return fail(r);
  if ((r = s->xyzm.alloc(m.N)) != FEMX_OK || (r = s->Fprev.alloc(m.N)) != FEMX_OK) return fail(r);
  for (int k = 0; k < 2; k++) {
    if ((r = s->U[k].alloc(m.N)) != FEMX_OK) return fail(r);
    if (p->fixed_dofs && (r = s->Up[k].alloc(m.N)) != FEMX_OK) return fail(r);
  }
  const int nparts = m.blk.n_sh ? m.blk.sh_off[m.blk.n_sh] : 0;
  if ((r = s->partials.alloc(std::max(nparts, 1))) != FEMX_OK) return fail(r);
  if ((r = s->lam.alloc(m.E)) != FEMX_OK || (r = s->regime.alloc(m.E)) != FEMX_OK || (r = s->pres.alloc(m.E)) != FEMX_OK)
    return fail(r);
  if ((r = s->row.alloc(D_ROW + 1)) != FEMX_OK || (r = s->halt.alloc(1)) != FEMX_OK) return fail(r);
  if ((r = s->eblk.alloc((size_t)m.blk.nb * D_COLS)) != FEMX_OK) return fail(r);
  if ((r = s->nblk.alloc((size_t)grid_for(m.N, 256) * D_COLS)) != FEMX_OK) return fail(r);
  if ((r = s->dpart.alloc((size_t)DIAG_PARTS * D_COLS)) != FEMX_OK) return fail(r);
  if (hipMemsetAsync(s->row.p, 0, (D_ROW + 1) * sizeof(double), s->st) != hipSuccess) return fail(FEMX_ERR_HIP);
  if (m.npe == 8)
    supg_mass<8><<<grid_for(m.N, 256), 256, 0, s->st>>>(m.N, m.g_off.p, m.g_slot.p, m.conn.p, m.xyz.p, p->rho, s->xyzm.p);
  else
    supg_mass<4><<<grid_for(m.N, 256), 256, 0, s->st>>>(m.N, m.g_off.p, m.g_slot.p, m.conn.p, m.xyz.p, p->rho, s->xyzm.p);
  if (m.blk.n_sh > 0) {
    if ((r = s->sh_m.alloc(m.blk.n_sh)) != FEMX_OK || (r = s->sh_rec.alloc(m.blk.n_sh)) != FEMX_OK) return fail(r);
    supg_shared_meta<<<grid_for(m.blk.n_sh, 256), 256, 0, s->st>>>(m.blk.n_sh, m.blk.d_sh_node.p, s->xyzm.p,
                                                                     s->bc.node_rec.p, s->sh_m.p, s->sh_rec.p);
  }
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s->st) != hipSuccess) return fail(FEMX_ERR_HIP);
  *out = s;
  return FEMX_OK;
}

extern "C" femx_status femx_supg_destroy(femx_supg *s) {
  if (!s) return FEMX_OK;
  if (s->in_union) (void)femx_supg_union_remove(s->in_union, s);
  hipStream_t st = s->st;
  if (st) (void)hipStreamSynchronize(st);
  {
    IdleRelease idle;  // the handle's work has completed
    delete s;
  }
  stream_put(st);
  return FEMX_OK;
}

extern "C" femx_status femx_supg_set_state(femx_supg *s, const double *sol) {
  if (!s || !sol) return set_error("null argument"), FEMX_ERR_ARG;
  if (s->in_union) return set_error("the handle is in a union"), FEMX_ERR_ARG;
  Mesh &m = *s->mesh;
  std::vector<double4> h(m.N);
  for (int n = 0; n < m.N; n++) h[n] = make_double4(sol[3L * n], sol[3L * n + 1], sol[3L * n + 2], 0.0);
  s->cur = 0;
  s->loop_time = 0;
  s->time = 0.0;
  s->halted = false;
  s->pend_n = 0;
  FEMX_HIP(hipMemcpyAsync(s->U[0].p, h.data(), m.N * sizeof(double4), hipMemcpyHostToDevice, s->st));
  FEMX_HIP(hipMemsetAsync(s->bc.err.p, 0, sizeof(int), s->st));
  const int imax = INT_MAX;
  FEMX_HIP(hipMemcpyAsync(s->halt.p, &imax, sizeof(int), hipMemcpyHostToDevice, s->st));
  if (s->bc.n_rec > 0)
    supg_bc_only<<<grid_for(s->bc.n_rec, 256), 256, 0, s->st>>>(s->bc.n_rec, s->rec_node.p, s->bc.rec.p,
                                                                s->bc.row_off.p, s->bc.rows.p, 0.0, s->U[0].p,
                                                                s->bc.err.p);
  FEMX_HIP(hipGetLastError());
  if (s->p.fixed_dofs)
    FEMX_HIP(hipMemcpyAsync(s->Up[0].p, s->U[0].p, m.N * sizeof(double4), hipMemcpyDeviceToDevice, s->st));
  FEMX_HIP(hipMemsetAsync(s->lam.p, 0, m.E * sizeof(double), s->st));  // el_lam = 0 at the initial pressure (:896)
  FEMX_HIP(hipMemsetAsync(s->regime.p, 0, m.E * sizeof(double), s->st));
  FEMX_HIP(hipMemsetAsync(s->Fprev.p, 0, m.N * sizeof(double4), s->st));
  FEMX_HIP(hipMemsetAsync(s->row.p, 0, (D_ROW + 1) * sizeof(double), s->st));
  s->press_pending = true;
  ReadPiece none[1];
  return read_checked(s, none, 0);
}

namespace {

// Enqueues nsteps time steps (:1034-1734) without waiting for them.
femx_status supg_enqueue(femx_supg *s, int nsteps) {
  if (s->pend_n == 0) {
    s->pend_first = s->loop_time;
    s->pend_t0 = s->time;
    s->pend_cur0 = s->cur;
  }
  for (int k = 0; k < nsteps; k++) {
    s->loop_time++;
    s->time += s->p.dt;  // currentTime += timeStep (:1041)
    const bool euler_step = s->p.use_euler || s->loop_time == 1;
    // the log row: per step with the element diagnostics on, else the one of
    // the call's last step
    const bool row = s->diag_enabled || k == nsteps - 1;
    femx_status r = launch_supg(s, true, s->press_pending, euler_step, s->time, row);
    if (r != FEMX_OK) return r;
    if ((r = launch_fix(s, euler_step, s->time, row)) != FEMX_OK) return r;
    s->cur ^= 1;
    s->press_pending = true;
    if (row && (r = launch_row(s, s->mesh->blk.nb, fix_rows(s), s->diag_enabled, (int)s->loop_time)) != FEMX_OK)
      return r;
    s->pend_n++;
  }
  return FEMX_OK;
}

// The handle's stream waits for its union's work queued so far.
femx_status union_wait(femx_supg *h);

// Waits for the enqueued steps and applies the exit condition (:1633-1643):
// when a step's max |u| exceeded it, the later steps did not run and the
// host counters are rewound to that step.
femx_status supg_finish(femx_supg *s, int *steps_done) {
  const long nsteps = s->pend_n, first = s->pend_first;
  const double t0 = s->pend_t0;
  const int cur0 = s->pend_cur0;
  s->pend_n = 0;
  if (steps_done) *steps_done = 0;
  int halt = INT_MAX;
  ReadPiece rb[2] = {{&halt, s->halt.p, sizeof(int)}};
  femx_status r = read_checked(s, rb, 1);
  if (r != FEMX_OK) return r;
  if (halt != INT_MAX) {
    const long stop = halt;
    // rewind the host counters to the step that exceeded the threshold
    const long done = stop - first;
    s->loop_time = stop;
    s->time = t0;
    for (long k = 0; k < done; k++) s->time += s->p.dt;
    s->cur = (int)((cur0 + done) & 1);
    if (steps_done) *steps_done = (int)done;
    s->halted = true;
    // a step inside a call has no log row of its own: make it from the state
    double step = 0.0;
    FEMX_HIP(hipMemcpyAsync(&step, s->row.p + D_STEP, sizeof(double), hipMemcpyDeviceToHost, s->st));
    FEMX_HIP(hipStreamSynchronize(s->st));
    if (step != (double)stop) {
      const int nwg = grid_for(s->mesh->N, 256);
      supg_state_rows<<<nwg, 256, 0, s->st>>>(s->mesh->N, s->U[s->cur].p, s->nblk.p);
      FEMX_HIP(hipGetLastError());
      if ((r = launch_row(s, 0, nwg, false, (int)stop)) != FEMX_OK) return r;
    }
    set_error("ERROR: Maximum velocity module larger than admissible threshold.");
    return FEMX_EXIT_CONDITION;
  }
  if (steps_done) *steps_done = (int)nsteps;
  return FEMX_OK;
}

}  // namespace

extern "C" femx_status femx_supg_step(femx_supg *s, int nsteps, int *steps_done) {
  if (!s || nsteps < 0) return set_error("bad argument"), FEMX_ERR_ARG;
  if (s->in_union) return set_error("the handle is in a union"), FEMX_ERR_ARG;
  if (steps_done) *steps_done = 0;
  if (s->halted) return set_error("the exit condition already stopped this solve"), FEMX_EXIT_CONDITION;
  femx_status r = supg_enqueue(s, nsteps);
  if (r != FEMX_OK) return r;
  return supg_finish(s, steps_done);
}

extern "C" femx_status femx_supg_step_async(femx_supg *s, int nsteps) {
  if (!s || nsteps < 0) return set_error("bad argument"), FEMX_ERR_ARG;
  if (s->in_union) return set_error("the handle is in a union"), FEMX_ERR_ARG;
  if (s->halted) return set_error("the exit condition already stopped this solve"), FEMX_EXIT_CONDITION;
  return supg_enqueue(s, nsteps);
}

extern "C" femx_status femx_supg_finish(femx_supg *s, int *steps_done) {
  if (!s) return set_error("null argument"), FEMX_ERR_ARG;
  if (s->in_union) return set_error("the handle is in a union"), FEMX_ERR_ARG;
  if (s->halted && s->pend_n == 0) {
    if (steps_done) *steps_done = 0;
    return set_error("the exit condition already stopped this solve"), FEMX_EXIT_CONDITION;
  }
  return supg_finish(s, steps_done);
}

extern "C" femx_status femx_supg_get_state(femx_supg *s, double *sol, double *pres, double *lam, double *regime,
                                           double *time) {
  if (!s) return set_error("null argument"), FEMX_ERR_ARG;
  if (s->in_union) return set_error("the handle is in a union"), FEMX_ERR_ARG;
  Mesh &m = *s->mesh;
  const DeviceGuard guard(m.device);
  if (s->pend_n > 0) {
    const femx_status f = supg_finish(s, nullptr);
    if (f != FEMX_OK && f != FEMX_EXIT_CONDITION) return f;
  }
  femx_status r = flush_pressure(s);
  if (r != FEMX_OK) return r;
  // what is asked for, in the caller's layouts, in one staging array kept by
  // the handle: [N][3] then E values per element field.  Where the device has
  // no room for it, the state is packed on the host and the fields pass through
  // an array of E values one by one
  double *outs[3] = {pres, lam, regime};
  DevBuf<double> *srcs[3] = {&s->pres, &s->lam, &s->regime};
  size_t len = 0, off = 0;
  for (double *o : outs) len += o ? m.E : 0;
  len += sol ? 3 * (size_t)m.N : 0;
  const bool staged = s->scratch.n >= len || s->scratch.alloc(len) == FEMX_OK;
  if (!staged) (void)hipGetLastError();
  ReadPiece rb[5];
  int nrb = 0;
  if (sol && staged) {
    pack3<<<grid_for(3L * m.N, 256), 256, 0, s->st>>>(m.N, reinterpret_cast<const double *>(s->U[s->cur].p),
                                                      s->scratch.p);
    FEMX_HIP(hipGetLastError());
    rb[nrb++] = {sol, s->scratch.p, 3 * (size_t)m.N * sizeof(double)};
    off = 3 * (size_t)m.N;
  } else if (sol) {
    std::vector<double4> h(m.N);
    const ReadPiece all = {h.data(), s->U[s->cur].p, m.N * sizeof(double4)};
    if ((r = read_back(m.device, s->st, &all, 1)) != FEMX_OK) return r;
    for (int n = 0; n < m.N; n++) {
      sol[3L * n] = h[n].x;
      sol[3L * n + 1] = h[n].y;
      sol[3L * n + 2] = h[n].z;
    }
  }
  for (int k = 0; k < 3; k++) {
    if (!outs[k]) continue;
    if (!staged && s->scratch.n < (size_t)m.E && (r = s->scratch.alloc(m.E)) != FEMX_OK) return r;
    block_to_orig<<<grid_for(m.E, 256), 256, 0, s->st>>>(m.E, m.blk.d_perm.p, srcs[k]->p, s->scratch.p + off);
    FEMX_HIP(hipGetLastError());
    rb[nrb++] = {outs[k], s->scratch.p + off, m.E * sizeof(double)};
    if (staged) {
      off += m.E;
    } else {
      if ((r = read_back(m.device, s->st, rb, nrb)) != FEMX_OK) return r;
      nrb = 0;
    }
  }
  if (time) *time = s->time;
  return read_checked(s, rb, nrb);
}

extern "C" femx_status femx_supg_get_mass(femx_supg *s, double *l_M) {
  if (!s || !l_M) return set_error("null argument"), FEMX_ERR_ARG;
  const int N = s->mesh->N;
  std::vector<double4> x(N);
  FEMX_HIP(hipMemcpyAsync(x.data(), s->xyzm.p, N * sizeof(double4), hipMemcpyDeviceToHost, s->st));
  FEMX_HIP(hipStreamSynchronize(s->st));
  for (int n = 0; n < N; n++) l_M[3L * n] = l_M[3L * n + 1] = l_M[3L * n + 2] = x[n].w;
  return FEMX_OK;
}

extern "C" femx_status femx_supg_get_log(femx_supg *s, double *cols19) {
  if (!s || !cols19) return set_error("null argument"), FEMX_ERR_ARG;
  // a union member's log row comes from the union's stream, and after an exit
  // this call may write it (supg_finish): the union's work on it comes first
  // (a member that the exit condition stopped is left alone by later steps)
  if (s->in_union) {
    const femx_status w = union_wait(s);
    if (w != FEMX_OK) return w;
  }
  if (s->pend_n > 0) {
    const femx_status f = supg_finish(s, nullptr);
    if (f != FEMX_OK && f != FEMX_EXIT_CONDITION) return f;
  }
  double k[D_COLS];
  FEMX_HIP(hipMemcpyAsync(k, s->row.p, sizeof(k), hipMemcpyDeviceToHost, s->st));
  FEMX_HIP(hipStreamSynchronize(s->st));
  cols19[0] = (double)s->loop_time;
  cols19[1] = s->time;
  for (int i = 0; i < 17; i++) cols19[2 + i] = k[i];
  return FEMX_OK;
}

extern "C" femx_status femx_supg_set_diagnostics(femx_supg *s, int enable) {
  if (!s) return set_error("null argument"), FEMX_ERR_ARG;
  if (s->in_union) return set_error("the handle is in a union"), FEMX_ERR_ARG;
  s->diag_enabled = enable != 0;
  return FEMX_OK;
}

extern "C" femx_status femx_supg_sync(femx_supg *s) {
  if (!s) return set_error("null argument"), FEMX_ERR_ARG;
  FEMX_HIP(hipStreamSynchronize(s->st));
  return FEMX_OK;
}

extern "C" void *femx_supg_stream(femx_supg *s) { return s ? (void *)s->st : nullptr; }

extern "C" femx_status femx_supg_kernel_timing(femx_supg *s, int enable) {
  if (!s) return set_error("null argument"), FEMX_ERR_ARG;
  if (enable) s->timer.reset();
  else s->timer.resolve();
  s->timer.enabled = enable != 0;
  return FEMX_OK;
}

extern "C" int femx_supg_kernel_times(femx_supg *s, femx_kernel_time *out, int max_entries) {
  if (!s) return -1;
  return s->timer.export_to(out, max_entries);
}

// ------------------------------------------------------- unions of handles
// Continuous batching of resident SUPG solves: FEMX_MIXED hexa8 handles with
// B-hat, no fixed DOFs and no element diagnostics are advanced together, one
// launch of the element kernel, one of the fix-up and one of the per-member
// fold of the log rows and tick, per step for all members, each by its own
// number of steps.  Every log column is a minimum or a maximum, so one
// workgroup's fold of a member's rows gives its own launches' value at any
// row count.  A member's
// step is its handle's own (the same blocks, sums and order): its time,
// state parity and step number come from a device record the tick advances
// with the same arithmetic as the host's loop, and its exit condition is
// checked as on its own stream (femx_supg_finish after it leaves).
namespace {

struct SupgDyn {
  double t;  // time of the last step run
  int par;   // current state buffer
  int lt;    // loop_time of the last step run
  int left;  // steps left
};

struct SupgMember {
  SupgArgs<float> a;  // per step: U, Upress, Un, k.t, step_id, want_row
  SupgFix f;          // per step: U, Un, k.t, step_id, want_row
  double4 *Ub[2];
  double *row;
  SupgDyn *dyn;
  double dt;
  int nwg;  // fix-up workgroups
};

// every pointer of a member's arguments as a global one (to_global)
__device__ __forceinline__ void args_to_global(SupgArgs<float> &a) {
  to_global(a.elem_off), to_global(a.node_off), to_global(a.loc_node), to_global(a.loc_pslot);
  to_global(a.lcsr_off), to_global(a.lpos), to_global(a.lconn), to_global(a.xyzm), to_global(a.U);
  to_global(a.Upress), to_global(a.Un), to_global(a.Unp), to_global(a.Fprev), to_global(a.partials);
  to_global(a.lam), to_global(a.regime), to_global(a.pres), to_global(a.node_rec), to_global(a.rec);
  to_global(a.row_off), to_global(a.rows), to_global(a.err), to_global(a.eblk), to_global(a.halt);
}
__device__ __forceinline__ void args_to_global(SupgFix &a) {
  to_global(a.sh_node), to_global(a.sh_off), to_global(a.sh_slot), to_global(a.sh_first4);
  to_global(a.partials), to_global(a.sh_m), to_global(a.sh_rec), to_global(a.U), to_global(a.Un);
  to_global(a.Unp), to_global(a.Fprev), to_global(a.rec), to_global(a.row_off), to_global(a.rows);
  to_global(a.err), to_global(a.halt), to_global(a.nblk);
}

__device__ __forceinline__ int supg_member_of(const int *off, int nm, int g) {
  int lo = 0, hi = nm;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (uni(off[mid]) <= g) lo = mid;
    else hi = mid;
  }
  return lo;
}

__global__ __launch_bounds__(SB, SUPG_BLOCK_WAVES(float, 8)) void supg_block_union(const SupgMember *mem, const int *blk_off,
                                                                        int nm, int ntot, int last) {
  const int g = xcd_block(blockIdx.x, ntot);
  const int h = supg_member_of(blk_off, nm, g);
  const SupgMember &me = mem[h];
  SupgDyn *dyn = me.dyn;
  to_global(dyn);
  const int left = uni(dyn->left);
  if (left <= 0) return;
  const int par = uni(dyn->par), lt = uni(dyn->lt) + 1;
  SupgArgs<float> a = me.a;
  a.U = me.Ub[par];
  a.Upress = a.U;
  a.Un = me.Ub[par ^ 1];
  a.k.t = uni(dyn->t) + me.dt;  // currentTime += timeStep (:1041)
  a.step_id = lt;
  a.want_row = last || left == 1;
  args_to_global(a);
  const int blk = g - uni(blk_off[h]);
  supg_block_run<float, 8, true, true, true, false, false>(a, blk, blk);
}

__global__ __launch_bounds__(256) void supg_fixup_union(const SupgMember *mem, const int *fx_off, int nm, int last) {
  const int g = blockIdx.x;
  const int h = supg_member_of(fx_off, nm, g);
  const SupgMember &me = mem[h];
  SupgDyn *dyn = me.dyn;
  to_global(dyn);
  const int left = uni(dyn->left);
  if (left <= 0) return;
  const int par = uni(dyn->par);
  SupgFix f = me.f;
  f.step_id = uni(dyn->lt) + 1;
  f.want_row = last || left == 1;
  f.U = me.Ub[par];
  f.Un = me.Ub[par ^ 1];
  f.k.t = uni(dyn->t) + me.dt;
  args_to_global(f);
  supg_fixup_run<double>(f, g - uni(fx_off[h]));
}

// End of a union step, one workgroup per member with steps left: the log row
// of the member's last step, or of the call's last step (last), from the
// step's rows (element blocks and fix-up, both written by the previous
// kernels), then the member moves on by one step.
__global__ __launch_bounds__(256) void supg_union_tick(const SupgMember *mem, int last) {
  const SupgMember &me = mem[blockIdx.x];
  SupgDyn *d = me.dyn;
  to_global(d);
  const int left = uni(d->left);
  if (left <= 0) return;
  const int lt = uni(d->lt) + 1;
  const int *halt = me.a.halt;
  const double *eblk = me.a.eblk, *nblk = me.f.nblk;
  double *row = me.row;
  to_global(halt), to_global(eblk), to_global(nblk), to_global(row);
  if ((last || left == 1) && !halted(halt, lt))
    diag_fold(eblk, me.a.nblk, nblk, me.nwg, 0, row, row + D_ROW, lt, 0, 1);
  __syncthreads();
  if (threadIdx.x == 0) {
    d->t = d->t + me.dt;
    d->par ^= 1;
    d->lt = lt;
    d->left -= 1;
  }
}

__global__ void supg_union_join(SupgDyn *d, double t, int par, int lt, int left) {
  d->t = t;
  d->par = par;
  d->lt = lt;
  d->left = left;
}

bool union_member_ok(const femx_supg *s) {
  const Blocks &b = s->mesh->blk;
  const int nnb = b.n_sh ? grid_for(b.n_sh, 256) : 0;
  return s->p.precision == FEMX_MIXED && s->mesh->npe == 8 && s->p.use_bhat && s->p.fixed_dofs == 0 &&
         !s->diag_enabled && nnb > 0;
}

}  // namespace

struct femx_supg_union {
  int device = 0;
  hipStream_t st = nullptr;
  std::vector<femx_supg *> mem;
  bool dirty = true;
  int nblk = 0, nfx = 0;
  DevBuf<SupgMember> tab;
  DevBuf<int> off;  // blk_off [nm + 1] then fx_off [nm + 1]
  size_t cap = 0;
  // pinned staging of the table uploads, a ring of slots, each reused once
  // the copy that read it has run
  static constexpr int NSLOT = 3;
  unsigned char *pin[NSLOT] = {nullptr, nullptr, nullptr};
  size_t pin_cap[NSLOT] = {0, 0, 0};
  hipEvent_t pin_ev[NSLOT] = {nullptr, nullptr, nullptr};
  int pin_next = 0;
};

namespace {

femx_status union_wait(femx_supg *h) {
  hipEvent_t ev = nullptr;
  FEMX_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
  const bool ok = hipEventRecord(ev, h->in_union->st) == hipSuccess && hipStreamWaitEvent(h->st, ev, 0) == hipSuccess;
  (void)hipEventDestroy(ev);
  if (!ok) return set_error("hipStreamWaitEvent failed"), FEMX_ERR_HIP;
  return FEMX_OK;
}

femx_status supg_union_upload(femx_supg_union *u) {
  const int nm = (int)u->mem.size();
  std::vector<SupgMember> t(nm);
  std::vector<int> off(2L * (nm + 1), 0);
  for (int i = 0; i < nm; i++) {
    femx_supg *h = u->mem[i];
    SupgMember &e = t[i];
    const bool euler = h->p.use_euler != 0;  // the first step ran on the handle's own stream
    e.a = supg_args<float>(h, euler, 0.0);
    e.a.Unp = nullptr;
    const Blocks &b = h->mesh->blk;
    e.f = fix_args(h, euler, 0.0);
    e.f.Unp = nullptr;
    for (int k = 0; k < 2; k++) e.Ub[k] = h->U[k].p;
    e.row = h->row.p;
    e.dyn = reinterpret_cast<SupgDyn *>(h->dyn.p);
    e.dt = h->p.dt;
    e.nwg = grid_for(b.n_sh, 256);
    off[i + 1] = off[i] + b.nb;
    off[nm + 1 + i + 1] = off[nm + 1 + i] + e.nwg;
  }
  u->nblk = off[nm];
  u->nfx = off[2 * nm + 1];
  femx_status r;
  if ((size_t)nm > u->cap) {
    // grow (the old table may still be read by enqueued steps: wait for them)
    FEMX_HIP(hipStreamSynchronize(u->st));
    const size_t cap = std::max<size_t>(2 * (size_t)nm, 16);
    if ((r = u->tab.alloc(cap)) != FEMX_OK || (r = u->off.alloc(2 * (cap + 1))) != FEMX_OK) return r;
    u->cap = cap;
  }
  const size_t bytes_t = nm * sizeof(SupgMember), bytes_o = off.size() * sizeof(int);
  const int k = u->pin_next;
  u->pin_next = (k + 1) % femx_supg_union::NSLOT;
  if (u->pin_ev[k]) FEMX_HIP(hipEventSynchronize(u->pin_ev[k]));
  if (u->pin_cap[k] < bytes_t + bytes_o) {
    if (u->pin[k]) FEMX_HIP(hipHostFree(u->pin[k]));
    u->pin[k] = nullptr;
    const size_t want = 2 * (bytes_t + bytes_o) + 4096;
    FEMX_HIP(hipHostMalloc((void **)&u->pin[k], want, hipHostMallocDefault));
    u->pin_cap[k] = want;
  }
  if (nm > 0) {
    std::memcpy(u->pin[k], t.data(), bytes_t);
    FEMX_HIP(hipMemcpyAsync(u->tab.p, u->pin[k], bytes_t, hipMemcpyHostToDevice, u->st));
  }
  std::memcpy(u->pin[k] + bytes_t, off.data(), bytes_o);
  FEMX_HIP(hipMemcpyAsync(u->off.p, u->pin[k] + bytes_t, bytes_o, hipMemcpyHostToDevice, u->st));
  if (!u->pin_ev[k]) FEMX_HIP(hipEventCreateWithFlags(&u->pin_ev[k], hipEventDisableTiming));
  FEMX_HIP(hipEventRecord(u->pin_ev[k], u->st));
  u->dirty = false;
  return FEMX_OK;
}

}  // namespace

extern "C" int femx_supg_union_accepts(femx_supg *h) {
  return h && !h->in_union && !h->halted && union_member_ok(h) ? 1 : 0;
}

extern "C" femx_status femx_supg_union_create(femx_supg_union **out) {
  if (!out) return set_error("null argument"), FEMX_ERR_ARG;
  if (femx_device_count() <= 0) return set_error("no HIP device visible"), FEMX_ERR_NO_DEVICE;
  femx_supg_union *u = new femx_supg_union();
  (void)hipGetDevice(&u->device);
  if (hipStreamCreateWithFlags(&u->st, hipStreamNonBlocking) != hipSuccess) {
    delete u;
    return set_error("hipStreamCreate failed"), FEMX_ERR_HIP;
  }
  *out = u;
  return FEMX_OK;
}

extern "C" femx_status femx_supg_union_destroy(femx_supg_union *u) {
  if (!u) return FEMX_OK;
  while (!u->mem.empty()) (void)femx_supg_union_remove(u, u->mem.back());
  (void)hipStreamSynchronize(u->st);
  for (int k = 0; k < femx_supg_union::NSLOT; k++) {
    if (u->pin[k]) (void)hipHostFree(u->pin[k]);
    if (u->pin_ev[k]) (void)hipEventDestroy(u->pin_ev[k]);
  }
  hipStream_t st = u->st;
  delete u;
  (void)hipStreamDestroy(st);
  return FEMX_OK;
}

extern "C" femx_status femx_supg_union_add(femx_supg_union *u, femx_supg *h, int steps) {
  if (!u || !h || steps < 0) return set_error("bad argument"), FEMX_ERR_ARG;
  if (h->in_union) return set_error("handle already in a union"), FEMX_ERR_ARG;
  if (!union_member_ok(h))
    return set_error("union members: FEMX_MIXED hexa8 with B-hat, no fixed DOFs, no diagnostics, more than one "
                     "element block"),
           FEMX_ERR_UNSUPPORTED;
  if (h->loop_time < 1) return set_error("union members run their first step on their own"), FEMX_ERR_ARG;
  if (h->halted) return set_error("the exit condition already stopped this solve"), FEMX_EXIT_CONDITION;
  femx_status r;
  if (!h->dyn.p && (r = h->dyn.alloc(sizeof(SupgDyn))) != FEMX_OK) return r;
  // the union's stream waits for the work already queued on the handle's
  hipEvent_t ev = nullptr;
  FEMX_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
  const bool ok = hipEventRecord(ev, h->st) == hipSuccess && hipStreamWaitEvent(u->st, ev, 0) == hipSuccess;
  (void)hipEventDestroy(ev);
  if (!ok) return set_error("hipStreamWaitEvent failed"), FEMX_ERR_HIP;
  supg_union_join<<<1, 1, 0, u->st>>>(reinterpret_cast<SupgDyn *>(h->dyn.p), h->time, h->cur, (int)h->loop_time,
                                      steps);
  FEMX_HIP(hipGetLastError());
  h->in_union = u;
  h->u_left = steps;
  u->mem.push_back(h);
  u->dirty = true;
  return FEMX_OK;
}

extern "C" femx_status femx_supg_union_step(femx_supg_union *u, int k) {
  if (!u || k < 0) return set_error("bad argument"), FEMX_ERR_ARG;
  femx_status r;
  if (u->dirty && (r = supg_union_upload(u)) != FEMX_OK) return r;
  const int nm = (int)u->mem.size();
  if (nm == 0 || k == 0) return FEMX_OK;
  const int *blk_off = u->off.p, *fx_off = u->off.p + nm + 1;
  for (int i = 0; i < k; i++) {
    const int last = i == k - 1;
    supg_block_union<<<u->nblk, SB, 0, u->st>>>(u->tab.p, blk_off, nm, u->nblk, last);
    supg_fixup_union<<<u->nfx, 256, 0, u->st>>>(u->tab.p, fx_off, nm, last);
    supg_union_tick<<<nm, 256, 0, u->st>>>(u->tab.p, last);
  }
  FEMX_HIP(hipGetLastError());
  // the host's view of every member: the steps enqueued as on its own stream
  // (femx_supg_finish checks them for the exit condition after it leaves)
  for (femx_supg *h : u->mem) {
    const int n = std::min(k, h->u_left);
    if (n > 0 && h->pend_n == 0) {
      h->pend_first = h->loop_time;
      h->pend_t0 = h->time;
      h->pend_cur0 = h->cur;
    }
    for (int i = 0; i < n; i++) h->time += h->p.dt;  // currentTime += timeStep (:1041)
    h->loop_time += n;
    h->cur ^= n & 1;
    h->pend_n += n;
    h->u_left -= n;
  }
  return FEMX_OK;
}

extern "C" int femx_supg_union_left(femx_supg_union *u, femx_supg *h) {
  if (!u || !h || h->in_union != u) return -1;
  return h->u_left;
}

extern "C" femx_status femx_supg_union_remove(femx_supg_union *u, femx_supg *h) {
  if (!u || !h || h->in_union != u) return set_error("handle not in this union"), FEMX_ERR_ARG;
  const femx_status w = union_wait(h);
  if (w != FEMX_OK) return w;
  u->mem.erase(std::find(u->mem.begin(), u->mem.end(), h));
  h->in_union = nullptr;
  h->u_left = 0;
  u->dirty = true;
  return FEMX_OK;
}

extern "C" femx_status femx_supg_union_sync(femx_supg_union *u) {
  if (!u) return set_error("null argument"), FEMX_ERR_ARG;
  FEMX_HIP(hipStreamSynchronize(u->st));
  return FEMX_OK;
}

extern "C" void *femx_supg_union_stream(femx_supg_union *u) { return u ? (void *)u->st : nullptr; }

