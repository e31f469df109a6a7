// femx_ins.hip -- implicit transient advection-diffusion stage of
// femIncompressibleSolver (src/femIncompressibleSolver.cpp:129-283) with its
// generalized-alpha update (:471-485), on gfx950.
//
// One stage per femx_ins_advdiff_solve call, all on the handle's stream:
//   tet4, ins_rows_tet4: eight lanes per matrix row; each forms its share of
//                   the row's elements' contributions (their row of the element
//                   matrix and vector of formTransientAdvDiffLHS /
//                   formTransientAdvDiffRHS, src/femElement.cpp:1471-1689, in
//                   FP64), sums them in LDS, then the Dirichlet row
//                   (applyDirichelet, src/femMatrix.cpp:183-205), the Jacobi
//                   inverse and the start of the Krylov solve (x = 0, r = b,
//                   z = D^-1 b, ||b||^2)
//   hexa8           (an element has 8 rows and costs 20 times a tet: it is
//                   formed once), and tet4 meshes with a row too long for one
//                   wave (row_work)
//   ins_element     one thread per element: the element matrix and vector,
//                   scattered straight into the order the gathers read (cpos /
//                   rpos maps)
//   ins_gather_mat  one thread per CSR entry: its contiguous run of element
//                   values, ascending element (the order femSparseMatrix::
//                   assemble adds them, src/femMatrix.cpp:129-160), then the
//                   Dirichlet row, Jacobi inverse
//   ins_gather_rhs  one thread per node: the same for the element vectors
//                   (femDenseVector::assemble), Dirichlet value, and the start
//                   of the Krylov solve
//   GMRES           restarted, right Jacobi preconditioning, classical
//                   Gram-Schmidt applied twice, zero initial guess; per
//                   iteration four launches: a vector-CSR SpMV of z = D^-1 v
//                   and three Gram-Schmidt passes sized to the basis in use.
//                   Each first finishes the reductions of the one before,
//                   every workgroup for itself, in a fixed order
//                   (deterministic).  Plays AztecOO's role
//                   (femSolver::solveLinearSystem src/femSolver.cpp:146-177).
//   ins_update      phi += dt phid + gamma dt (phid_new - phid); phid = phid_new.
//
// The element math is the reference's, regrouped per Gauss point: with
// a_B = u.grad N_B, P_B = N_B + tau a_B and Q_C = alphaM N_C + alphaF dt gamma a_C,
//   LHS_BC += P_B Q_C detJ w      (currK + stabK of :1539-1561)
//   RHS_B  -= P_B R   detJ w,     R = (1-alphaM) phid + u.grad phi
//                                     + alphaF dt (1-gamma) u.grad phid  (:1641-1687)
// which equals the reference's sums up to rounding.
#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <cstring>
#include <thread>

#include "femx_common.h"
#include "femx_elem.h"

namespace femx {
namespace {

constexpr int MAXM = 32;   // largest Krylov space per restart cycle
constexpr int RT = 256;    // threads per block of the row kernels
// reduction blocks of the row kernels: three per CU (5.3M tets, 9 iterations a
// step: 256 2.15 ms, 512 1.80, 768 1.70, 1024 1.72: more partials for every
// workgroup to sum, or too few rows in flight)
constexpr int MAXNB = 768;
constexpr int CHECK = 4;   // iterations between host checks of the cycle flag

struct InsConst {
  double am, afdtg, om, afdt1g, timeTau;
};

// Control words first: the host copies them back in one transfer.
struct GmresState {
  int cyc_stop, done, conv, iters, jend, pad;
  double relres, r0, beta, vscale, tol;
  int max_iter, pad2;
  double H[(MAXM + 1) * MAXM];  // H[i * MAXM + j]
  double cs[MAXM], sn[MAXM], g[MAXM + 1], y[MAXM];
};
struct GmresCtl {
  int cyc_stop, done, conv, iters, jend, pad;
  double relres;
};

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// Lane i's value (i uniform), in SGPRs.
__device__ __forceinline__ double read_lane(double v, int i) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b & 0xffffffffLL), i);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), i);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Block sums of acc[0..cnt) -> part[i * nb + blockIdx.x] (RT threads).
template <int J>
__device__ __forceinline__ void block_store(const double (&acc)[J], int cnt, double *part, int nb) {
  __shared__ double red[RT / 64][J];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < J; i++)
    if (i < cnt) {
      const double v = wave_sum(acc[i]);
      if (lane == 0) red[wv][i] = v;
    }
  __syncthreads();
  if ((int)threadIdx.x < cnt) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < RT / 64; w++) s += red[w][threadIdx.x];
    part[(long)threadIdx.x * nb + blockIdx.x] = s;
  }
}

// Sum of part[i * nb .. i * nb + nb) by one wave.
__device__ __forceinline__ double wave_total(const double *part, int i, int nb) {
  const int lane = threadIdx.x & 63;
  const double *p = part + (long)i * nb;
  // per chunk of 64 K partials: all loads first, then the lane's sum in the
  // order b = lane, lane + 64, ... (any nb: the solve's first reduction has
  // one partial per workgroup of its kernel)
  constexpr int K = MAXNB / 64;
  double s = 0.0;
  for (int c0 = 0; c0 < nb; c0 += 64 * K) {
    double v[K];
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = c0 + lane + 64 * k < nb ? p[c0 + lane + 64 * k] : 0.0;
#pragma unroll
    for (int k = 0; k < K; k++)
      if (c0 + lane + 64 * k < nb) s += v[k];
  }
  return wave_sum(s);
}

// ------------------------------------------------------------ velocity
// femModel::prescribeNodeVels (src/femModel.cpp:4515-4546).
__global__ __launch_bounds__(256) void ins_prescribe(int N, int type, double t, const double4 *xyz,
                                                     const double *node_vel, double4 *vphi) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= N) return;
  const double4 p = xyz[a];
  double4 v = vphi[a];
  if (type == 0) {
    const double c = cos(M_PI * t / 8.0);
    v.x = c * sin(2.0 * M_PI * p.y) * sin(M_PI * p.x) * sin(M_PI * p.x);
    v.y = -c * sin(2.0 * M_PI * p.x) * sin(M_PI * p.y) * sin(M_PI * p.y);
    v.z = 0.0;
  } else if (type == 1) {
    v.x = sin(M_PI * p.x) * cos(M_PI * p.y);
    v.y = -cos(M_PI * p.x) * sin(M_PI * p.y);
    v.z = 0.0;
  } else {
    v.x = node_vel[3L * a];
    v.y = node_vel[3L * a + 1];
    v.z = node_vel[3L * a + 2];
  }
  vphi[a] = v;
}

// phi and/or velocity from host-filled staging arrays.
__global__ __launch_bounds__(256) void ins_pack(int N, const double *phi, const double *vel, double4 *vphi) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= N) return;
  double4 v = vphi[a];
  if (phi) v.w = phi[a];
  if (vel) {
    v.x = vel[3L * a];
    v.y = vel[3L * a + 1];
    v.z = vel[3L * a + 2];
  }
  vphi[a] = v;
}

// phi [N] and/or velocity [N][3] of the node records into the staging array.
__global__ __launch_bounds__(256) void ins_unpack(int N, const double4 *vphi, double *phi, double *vel) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= N) return;
  const double4 v = vphi[a];
  if (phi) phi[a] = v.w;
  if (vel) {
    vel[3L * a] = v.x;
    vel[3L * a + 1] = v.y;
    vel[3L * a + 2] = v.z;
  }
}

// ------------------------------------------------------------- element
// Element t of the processing order (the mesh's Morton block order; every
// per-element input is stored in that order).  Each XCD takes a contiguous
// range of workgroups, so neighbouring elements write their scattered
// values through the same L2.
template <int NPE>
__global__ __launch_bounds__(256) void ins_element(int E, const int *conn, const double4 *xyz, const double4 *vphi,
                                                   const double *phid, const double *iso, InsConst k,
                                                   const int *cpos, const int *rpos, double *emat, double *erhs) {
  const int e = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (e >= E) return;
  int id[NPE];
#pragma unroll
  for (int a = 0; a < NPE; a++) id[a] = conn[(long)e * NPE + a];
  double dx[NPE][3], ve[NPE][3], ph[NPE], pd[NPE];
  const double4 x0 = xyz[id[0]];
#pragma unroll
  for (int a = 0; a < NPE; a++) {
    const double4 p = xyz[id[a]];
    dx[a][0] = p.x - x0.x;
    dx[a][1] = p.y - x0.y;
    dx[a][2] = p.z - x0.z;
    const double4 v = vphi[id[a]];
    ve[a][0] = v.x;
    ve[a][1] = v.y;
    ve[a][2] = v.z;
    ph[a] = v.w;
    pd[a] = phid[id[a]];
  }
  const double iso2 = iso[e] * iso[e];
  double M[NPE][NPE], R[NPE];
#pragma unroll
  for (int b = 0; b < NPE; b++) {
    R[b] = 0.0;
#pragma unroll
    for (int c = 0; c < NPE; c++) M[b][c] = 0.0;
  }
  // hexa8: one Gauss point at a time keeps the 8x8 accumulator in registers
  constexpr int GP_UNROLL = NPE == 4 ? 4 : 1;
#pragma unroll GP_UNROLL
  for (int g = 0; g < Shape<NPE>::NGP; g++) {
    double DN[NPE][3], detJ, iJ[3][3];
    kinematics<NPE>(g, dx, DN, detJ, iJ);
    // evalGeometricMatrix: G[a][b] = sum_c invJ[c][a] invJ[c][b]
    double G[3][3];
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++) G[a][b] = iJ[0][a] * iJ[0][b] + iJ[1][a] * iJ[1][b] + iJ[2][a] * iJ[2][b];
    double u[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
      double s = 0.0;
#pragma unroll
      for (int b = 0; b < NPE; b++) s += Shape<NPE>::N(g, b) * ve[b][d];
      u[d] = s;
    }
    // evalQuadraticTau (src/femElement.cpp:237-268), c = 1
    double t1 = 0.0, t2 = 0.0;
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++) {
        t1 += u[a] * G[a][b] * u[b];
        t2 += G[a][b] * G[a][b];
      }
    const double tau = 1.0 / sqrt(k.timeTau + t1 + t2 * iso2);
    double pdg = 0.0, gp[3] = {0.0, 0.0, 0.0}, gpd[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int b = 0; b < NPE; b++) {
      pdg += Shape<NPE>::N(g, b) * pd[b];
#pragma unroll
      for (int d = 0; d < 3; d++) {
        gp[d] += DN[b][d] * ph[b];
        gpd[d] += DN[b][d] * pd[b];
      }
    }
    const double Rg = k.om * pdg + (u[0] * gp[0] + u[1] * gp[1] + u[2] * gp[2]) +
                      k.afdt1g * (u[0] * gpd[0] + u[1] * gpd[1] + u[2] * gpd[2]);
    const double wd = detJ * Shape<NPE>::W();
    double P[NPE], Q[NPE];
#pragma unroll
    for (int b = 0; b < NPE; b++) {
      const double ad = u[0] * DN[b][0] + u[1] * DN[b][1] + u[2] * DN[b][2];
      P[b] = (Shape<NPE>::N(g, b) + tau * ad) * wd;
      Q[b] = k.am * Shape<NPE>::N(g, b) + k.afdtg * ad;
    }
#pragma unroll
    for (int b = 0; b < NPE; b++) {
      R[b] -= P[b] * Rg;
#pragma unroll
      for (int c = 0; c < NPE; c++) M[b][c] += P[b] * Q[c];
    }
  }
  // scatter into the gathers' order: contiguous per matrix entry / per node
  const int *cp = cpos + (long)e * NPE * NPE;
#pragma unroll
  for (int b = 0; b < NPE; b++)
#pragma unroll
    for (int c = 0; c < NPE; c++) emat[cp[b * NPE + c]] = M[b][c];
  const int *rq = rpos + (long)e * NPE;
#pragma unroll
  for (int b = 0; b < NPE; b++) erhs[rq[b]] = R[b];
}

// ---------------------------------------------------------- tet4 rows
// A tet4's matrix row is cheap to form (constant Jacobian: about 400
// instructions), and forming it again for each of its four rows costs less
// than passing the element matrices through memory: the element kernel and
// the two gathers moved 2.9 GB per assembly at 5.3M tets (106M scattered
// 8-byte writes among them), 1.03 ms; this kernel gathers the node records
// from the caches and writes the matrix, 0.60 ms (193k rows: 230 -> 112 us; half
// the issue slots are used, the L1 lookups of the gathers two thirds of the
// time; 168 VGPRs and 36 B of spills a lane at three waves per SIMD).  Eight
// lanes per row: a row has about 24 elements, and the lanes of a row read
// neighbouring records.
constexpr int RLPR = 8;             // lanes per row
constexpr int RROWS = 256 / RLPR;   // rows per workgroup pass
constexpr int RCAP = 24;            // row entries summed in LDS per pass over the row's elements
constexpr int RGRID = 3072;         // workgroups at most (each takes a contiguous range of rows)

// The most element formations that one lane may have for a row: passes over
// the row's elements (one per RCAP entries) times the lane's share of them.
// They are a chain that the launch waits for, 1.28 us each; the element kernel
// and the gathers take 30 us + 0.19 ns per element, so the limit is where the
// chain alone takes that long.  Assembly with one node of 128 / 512 elements
// (48 / 704 formations) among 1.11M tets: 123 / 895 us by rows, 239 / 279 us
// with the gathers; among 48k tets 70 / 852 us and 44 / 87 us.  Ordinary
// meshes have 3 to 16.
inline long row_work(long E) { return 24 + E / 6700; }

// The contributions of one element to the row of its corner a: v[b] += P_a Q_b,
// R -= P_a R (the sums over the Gauss points of the header).
__device__ __forceinline__ void tet4_row(const double4 X[4], const double4 V[4], int a, double iso2,
                                         const InsConst &k, double v[4], double &R) {
  double J[3][3], iJ[3][3], detJ;
#pragma unroll
  for (int r = 0; r < 3; r++) {
    J[r][0] = X[r].x - X[3].x;
    J[r][1] = X[r].y - X[3].y;
    J[r][2] = X[r].z - X[3].z;
  }
  inv3(J, iJ, detJ);
  // |G|^2 of evalGeometricMatrix: G[i][j] = sum_c invJ[c][i] invJ[c][j]
  double t2 = 0.0;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const int j = (i + 1) % 3;
    const double d = iJ[0][i] * iJ[0][i] + iJ[1][i] * iJ[1][i] + iJ[2][i] * iJ[2][i];
    const double o = iJ[0][i] * iJ[0][j] + iJ[1][i] * iJ[1][j] + iJ[2][i] * iJ[2][j];
    t2 += d * d + 2.0 * (o * o);
  }
  const double tb = k.timeTau + t2 * iso2, wd = detJ * Shape<4>::W();
  // the rule's values: N_b(g) = nb + nd (g == b)
  const double nb = Shape<4>::N(0, 1), nd = Shape<4>::N(0, 0) - nb;
  const double us[3] = {nb * ((V[0].x + V[1].x) + (V[2].x + V[3].x)), nb * ((V[0].y + V[1].y) + (V[2].y + V[3].y)),
                        nb * ((V[0].z + V[1].z) + (V[2].z + V[3].z))};
  const double ps = nb * ((X[0].w + X[1].w) + (X[2].w + X[3].w));
#pragma unroll
  for (int g = 0; g < 4; g++) {
    const double u[3] = {us[0] + nd * V[g].x, us[1] + nd * V[g].y, us[2] + nd * V[g].z};
    // evalQuadraticTau (src/femElement.cpp:237-268), c = 1: u^T G u = |invJ u|^2
    double t1 = 0.0, ad[4];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const double w = iJ[c][0] * u[0] + iJ[c][1] * u[1] + iJ[c][2] * u[2];
      t1 += w * w;
      ad[c] = iJ[0][c] * u[0] + iJ[1][c] * u[1] + iJ[2][c] * u[2];  // u.grad N_c
    }
    ad[3] = -(ad[0] + ad[1] + ad[2]);
    const double tau = rsqrt(tb + t1);
    double up = 0.0, ud = 0.0;  // u.grad phi, u.grad phid
#pragma unroll
    for (int b = 0; b < 4; b++) {
      up += ad[b] * V[b].w;
      ud += ad[b] * X[b].w;
    }
    const double Rg = k.om * (ps + nd * X[g].w) + up + k.afdt1g * ud;
    const double aa = a == 0 ? ad[0] : a == 1 ? ad[1] : a == 2 ? ad[2] : ad[3];
    const double P = ((a == g ? nb + nd : nb) + tau * aa) * wd;
    R -= P * Rg;
#pragma unroll
    for (int b = 0; b < 4; b++) v[b] += P * (k.am * (b == g ? nb + nd : nb) + k.afdtg * ad[b]);
  }
}

// p[i] by a 32-bit byte offset (arrays below 4 GiB): one VGPR of address, not two.
__device__ __forceinline__ double4 at32(const double4 *p, int i) {
  return *reinterpret_cast<const double4 *>(reinterpret_cast<const char *>(p) + ((unsigned)i << 5));
}

// node: x y z and phid; vphi: velocity and phi.  Rows in the order rord
// (along the mesh's Morton curve), row r's corners g_slot[g_off[r] ...) in
// ascending element, cpos their element's columns' places in the row.
__global__ __launch_bounds__(256, 3) void ins_rows_tet4(int N, const int *rord, const int *g_off, const int *g_slot,
                                                     const ushort4 *cpos, const int4 *conn, const double4 *node,
                                                     const double4 *vphi, const double *iso, InsConst k,
                                                     const int *row_ptr, const int *col, const int *dir_flag,
                                                     const double *dir_v, double *val, double *dinv, double *b,
                                                     double *x, double *rvec, double *z, double *part) {
  // the thread's sums of the row's entries: column tid of acc
  __shared__ double acc[RCAP * 256];
  const int tid = threadIdx.x, lane = tid & (RLPR - 1);
  const int ngroups = (N + RROWS - 1) / RROWS, per = (ngroups + gridDim.x - 1) / gridDim.x;
  const int first = xcd_block(blockIdx.x, gridDim.x) * per, last = min(ngroups, first + per);
  double nrm[1] = {0.0};
  for (int grp = first; grp < last; grp++) {
    const int i = grp * RROWS + tid / RLPR;
    if (i >= N) continue;
    const int r = rord[i], q0 = row_ptr[r], len = row_ptr[r + 1] - q0, j1 = g_off[r + 1];
    const bool fixed = dir_flag[r] != 0;
    double R = 0.0, di = 0.0;
    for (int c0 = 0; c0 < len; c0 += RCAP) {
      const int n = min(RCAP, len - c0);
      for (int q = 0; q < n; q++) acc[q * 256 + tid] = 0.0;
      if (!fixed) {
        // the next element's corner and connectivity are loaded while the
        // current one is formed
        int j = g_off[r] + lane, slot = 0;
        int4 c = make_int4(0, 0, 0, 0);
        if (j < j1) {
          slot = g_slot[j];
          c = conn[slot >> 2];
        }
        for (; j < j1; j += RLPR) {
          const double4 X[4] = {at32(node, c.x), at32(node, c.y), at32(node, c.z), at32(node, c.w)};
          const double4 V[4] = {at32(vphi, c.x), at32(vphi, c.y), at32(vphi, c.z), at32(vphi, c.w)};
          const double d0 = iso[slot >> 2];
          const ushort4 p0 = cpos[j];
          const int a = slot & 3;
          if (j + RLPR < j1) {
            slot = g_slot[j + RLPR];
            c = conn[slot >> 2];
          }
          double v[4] = {0.0, 0.0, 0.0, 0.0}, Rj = 0.0;
          tet4_row(X, V, a, d0 * d0, k, v, Rj);
          if (c0 == 0) R += Rj;
          const int p[4] = {p0.x - c0, p0.y - c0, p0.z - c0, p0.w - c0};
#pragma unroll
          for (int s = 0; s < 4; s++)
            if (p[s] >= 0 && p[s] < n) acc[p[s] * 256 + tid] += v[s];
        }
      }
      // the row's lanes are one wave's: its LDS accesses stay in order
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      for (int q = lane; q < n; q += RLPR) {
        const double *t = acc + q * 256 + (tid & ~(RLPR - 1));
        double s = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
        const bool dg = col[q0 + c0 + q] == r;
        if (fixed) s = dg ? 1.0 : 0.0;
        val[q0 + c0 + q] = s;
        if (dg) di = s != 0.0 ? 1.0 / s : 1.0;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
#pragma unroll
    for (int off = RLPR / 2; off > 0; off >>= 1) {
      R += __shfl_xor(R, off);
      di += __shfl_xor(di, off);  // one lane holds the diagonal's
    }
    if (lane == 0) {
      const double s = fixed ? dir_v[r] : R;
      dinv[r] = di;
      b[r] = s;
      x[r] = 0.0;
      rvec[r] = s;
      z[r] = di * s;
      nrm[0] += s * s;
    }
  }
  block_store<1>(nrm, 1, part, gridDim.x);
}

// ------------------------------------------------- reduction finishers
// The nb partial sums of a reduction pass are summed by the kernel that needs
// the result: as a launch of its own per pass (4 to 5 us, three of the seven
// an iteration had) they were a fifth of a solve of 200k rows.  A pass
// writes its partials into a buffer that its own prologue does not read.

// Start of a cycle from r = b - A x: beta = ||r|| (first: also r0).
__device__ __forceinline__ void fin_start(GmresState *st, const double *part, int nb, bool first) {
  if (threadIdx.x >= 64) return;
  const double s = wave_total(part, 0, nb);
  if (threadIdx.x != 0) return;
  const double beta = sqrt(s);
  if (first) {
    st->r0 = beta;
    st->iters = 0;
  }
  st->beta = beta;
  st->relres = st->r0 > 0.0 ? beta / st->r0 : 0.0;
  const bool conv = beta <= st->tol * st->r0;
  st->conv = conv ? 1 : 0;
  st->done = (conv || st->iters >= st->max_iter) ? 1 : 0;
  st->cyc_stop = st->done;
  st->jend = -1;
  for (int i = 0; i <= MAXM; i++) st->g[i] = 0.0;
  st->g[0] = beta;
  st->vscale = beta > 0.0 ? 1.0 / beta : 0.0;
}

// h = the reduced dots of a Gram-Schmidt pass, by every workgroup (one wave
// per dot); the first one records them: pass 0 sets column j of H, pass 1
// adds to it.
__device__ __forceinline__ void fin_h(GmresState *st, const double *part, int nb, int cnt, int j, int pass,
                                      double *h) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int i = wv; i < cnt; i += RT / 64) {
    const double s = wave_total(part, i, nb);
    if (lane == 0) {
      h[i] = s;
      if (blockIdx.x == 0) st->H[i * MAXM + j] = pass ? st->H[i * MAXM + j] + s : s;
    }
  }
  __syncthreads();
}

// H[j+1][j] = ||w||, Givens rotations, residual estimate, cycle stop test.
__device__ __forceinline__ void fin_givens(GmresState *st, double hn, int j) {
  double *H = st->H;
  H[(j + 1) * MAXM + j] = hn;
  for (int i = 0; i < j; i++) {
    const double t0 = H[i * MAXM + j], t1 = H[(i + 1) * MAXM + j];
    H[i * MAXM + j] = st->cs[i] * t0 + st->sn[i] * t1;
    H[(i + 1) * MAXM + j] = -st->sn[i] * t0 + st->cs[i] * t1;
  }
  const double a = H[j * MAXM + j], c = H[(j + 1) * MAXM + j];
  const double den = sqrt(a * a + c * c);
  const double cs = den != 0.0 ? a / den : 1.0, sn = den != 0.0 ? c / den : 0.0;
  st->cs[j] = cs;
  st->sn[j] = sn;
  H[j * MAXM + j] = den;
  H[(j + 1) * MAXM + j] = 0.0;
  st->g[j + 1] = -sn * st->g[j];
  st->g[j] = cs * st->g[j];
  st->iters += 1;
  st->jend = j;
  if (fabs(st->g[j + 1]) <= st->tol * st->r0 || st->iters >= st->max_iter || hn == 0.0) st->cyc_stop = 1;
  st->vscale = hn != 0.0 ? 1.0 / hn : 0.0;
}

// -------------------------------------------------------------- gathers
constexpr int CAP = 4096;  // doubles of element values staged in LDS per pass

// Sum of src[beg .. end) in ascending order for each thread of the block,
// where the threads' ranges are consecutive and together span [lo, hi):
// the values pass through LDS in coalesced chunks of CAP (a node's run of
// element values is long, ~24 for tet4, so lane-private reads would stride).
__device__ __forceinline__ double staged_run_sum(const double *src, long lo, long hi, long beg, long end) {
  __shared__ double buf[CAP];
  double s = 0.0;
  for (long c0 = lo; c0 < hi; c0 += CAP) {
    const long c1 = c0 + CAP < hi ? c0 + CAP : hi;
    __syncthreads();
    for (long k = c0 + threadIdx.x; k < c1; k += blockDim.x) buf[k - c0] = src[k];
    __syncthreads();
    const long a = beg > c0 ? beg : c0, b = end < c1 ? end : c1;
    for (long k = a; k < b; k++) s += buf[k - c0];
  }
  return s;
}

// The element values of entry q are emat[c_ptr[q] .. c_ptr[q+1]), ascending
// element (the order of femSparseMatrix::assemble).  The runs are short
// (a few values), so consecutive threads already read consecutive memory.
__global__ __launch_bounds__(RT) void ins_gather_mat(long nnz, const int *c_ptr, const double *emat,
                                                     const int *nz_row, const int *col, const int *dir_flag,
                                                     double *val, double *dinv) {
  const long q = (long)blockIdx.x * RT + threadIdx.x;
  if (q >= nnz) return;
  const int r = nz_row[q], c = col[q];
  double s = 0.0;
  for (int j = c_ptr[q]; j < c_ptr[q + 1]; j++) s += emat[j];
  if (dir_flag[r]) s = (c == r) ? 1.0 : 0.0;
  val[q] = s;
  if (c == r) dinv[r] = (s != 0.0) ? 1.0 / s : 1.0;
}

// b (element vectors erhs[g_off[r] .. g_off[r+1]), ascending element, as
// femDenseVector::assemble adds them), and the start of the solve: x = 0,
// r = b, z = D^-1 r, per-block ||b||^2 into part[blockIdx.x].
__global__ __launch_bounds__(RT) void ins_gather_rhs(int N, const int *g_off, const double *erhs,
                                                     const int *dir_flag, const double *dir_v, const double *dinv,
                                                     double *b, double *x, double *rvec, double *z, double *part) {
  const int r0 = blockIdx.x * RT, r = r0 + threadIdx.x;
  const int re = r0 + RT < N ? r0 + RT : N;
  const long lo = g_off[r0], hi = g_off[re];
  const long beg = r < N ? g_off[r] : hi, end = r < N ? g_off[r + 1] : hi;
  double s = staged_run_sum(erhs, lo, hi, beg, end);
  double acc[1] = {0.0};
  if (r < N) {
    if (dir_flag[r]) s = dir_v[r];
    b[r] = s;
    x[r] = 0.0;
    rvec[r] = s;
    z[r] = dinv[r] * s;
    acc[0] = s * s;
  }
  block_store<1>(acc, 1, part, gridDim.x);
}

// --------------------------------------------------------------- GMRES
// v_j = src * vscale and w = A D^-1 v_j = vscale * A z, z = D^-1 src;
// LPR lanes per row (vector CSR), lane 0 of each row group stores.
template <int LPR>
__global__ __launch_bounds__(RT) void gm_spmv(int N, const int *rp, const int *col, const double *val,
                                              const double *z, const double *src, double *V, long ldv, double *w,
                                              int j, GmresState *st, const double *part, int nb, int givens) {
  double sc;
  if (givens) {
    // iteration j - 1 ends here: its norm, and in the first workgroup its
    // rotation and stop test (after a stop this launch's output is not used).
    // That test may set the flag while other waves start, so one wave of each
    // workgroup reads it for all, and the rotation waits for the barrier: no
    // wave leaves before a barrier that another one of its workgroup reaches
    __shared__ double hn;
    __shared__ int stopped;
    if (threadIdx.x < 64) {
      const int stop = uni(st->cyc_stop);
      const double s = stop ? 0.0 : wave_total(part, 0, nb);
      if (threadIdx.x == 0) {
        hn = sqrt(s);
        stopped = stop;
      }
    }
    __syncthreads();
    if (stopped) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) fin_givens(st, hn, j - 1);
    sc = hn != 0.0 ? 1.0 / hn : 0.0;
  } else {
    if (st->cyc_stop) return;
    sc = st->vscale;
  }
  const int lane = threadIdx.x & (LPR - 1);
  const int r = (blockIdx.x * RT + threadIdx.x) / LPR;
  if (r >= N) return;
  double s = 0.0;
  for (int q = rp[r] + lane; q < rp[r + 1]; q += LPR) s += val[q] * z[col[q]];
#pragma unroll
  for (int off = LPR / 2; off > 0; off >>= 1) s += __shfl_xor(s, off);
  if (lane == 0) {
    w[r] = s * sc;
    V[(long)j * ldv + r] = src[r] * sc;
  }
}

// Gram-Schmidt passes over w and v_0..v_j (j < J), partial sums into part:
//   mode 0: dots w . v_i
//   mode 1: h = the dots (H[:, j] = h),  w -= sum_i h_i v_i, dots w . v_i
//   mode 2: h = the dots (H[:, j] += h), w -= sum_i h_i v_i, ||w||^2, z = D^-1 w
//           (LAST)
// The dots of the pass before are summed from pin.  Bound by the stream of the
// basis: a row's values are all loaded before the first is used, and the
// registers are kept to the J sums and J values.  The dots go to SGPRs (read
// from LDS by every lane they took 2 J VGPRs), and the last pass, which needs
// one sum, is a kernel of its own (both kinds in one copied the sums): J = 4 /
// 8 / 16 / 32 39 / 42 / 75 / 140 VGPRs and 8 / 8 / 6 / 3 waves per SIMD against
// 42 / 74 / 139 / 256 and 8 / 6 / 3 / 1; a pass of a 30-iteration solve, 195k
// rows 32.8 -> 16.1 us, 913k rows 83.9 -> 30.3 us (16 iterations 26.5 -> 19.9).
template <int J, bool LAST>
__global__ __launch_bounds__(RT) void gm_orth(int N, double *w, const double *V, long ldv, int j, GmresState *st,
                                              const double *pin, double *part, int nb, int mode,
                                              const double *dinv, double *z) {
  if (st->cyc_stop) return;
  __shared__ double hs[J];
  if (mode != 0) fin_h(st, pin, nb, j + 1, j, mode - 1, hs);
  const int lane = threadIdx.x & 63;
  const double hl = mode != 0 && lane <= j ? hs[lane] : 0.0;
  constexpr int NA = LAST ? 1 : J;
  double h[J], acc[NA];
#pragma unroll
  for (int i = 0; i < J; i++) h[i] = read_lane(hl, i);
#pragma unroll
  for (int i = 0; i < NA; i++) acc[i] = 0.0;
  for (int r = blockIdx.x * RT + threadIdx.x; r < N; r += nb * RT) {
    double v[J];
    double s = w[r];
#pragma unroll
    for (int i = 0; i < J; i++) v[i] = i <= j ? V[(long)i * ldv + r] : 0.0;
#pragma unroll
    for (int i = 0; i < J; i++) s -= h[i] * v[i];
    if (LAST) {
      w[r] = s;
      acc[0] += s * s;
      z[r] = dinv[r] * s;
    } else {
      if (mode != 0) w[r] = s;
#pragma unroll
      for (int i = 0; i < NA; i++) acc[i] += s * v[i];
    }
  }
  block_store<NA>(acc, LAST ? 1 : j + 1, part, nb);
}

// y = H^-1 g on the cycle's upper triangle.
// The end of a cycle (this, gm_xupdate, gm_resid, gm_start) may be enqueued
// before the host knows whether the cycle has stopped: unless the cycle is
// full (force), it does nothing if it has not.
__device__ __forceinline__ bool cycle_ends(const GmresState *st, int force) {
  return !st->done && (force || st->cyc_stop);
}
__global__ __launch_bounds__(64) void gm_backsub(GmresState *st, int force) {
  if (threadIdx.x != 0 || !cycle_ends(st, force)) return;
  const int je = st->jend;
  for (int i = je; i >= 0; i--) {
    double s = st->g[i];
    for (int k = i + 1; k <= je; k++) s -= st->H[i * MAXM + k] * st->y[k];
    st->y[i] = st->H[i * MAXM + i] != 0.0 ? s / st->H[i * MAXM + i] : 0.0;
  }
}

// x += D^-1 V y.
template <int J>
__global__ __launch_bounds__(RT) void gm_xupdate(int N, double *x, const double *dinv, const double *V, long ldv,
                                                 const GmresState *st, int force) {
  if (!cycle_ends(st, force)) return;
  const int je = st->jend;
  double y[J];
#pragma unroll
  for (int i = 0; i < J; i++) y[i] = i <= je ? st->y[i] : 0.0;
  for (int r = blockIdx.x * RT + threadIdx.x; r < N; r += gridDim.x * RT) {
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < J; i++)
      if (i <= je) s += y[i] * V[(long)i * ldv + r];
    x[r] += dinv[r] * s;
  }
}

// r = b - A x, z = D^-1 r, ||r||, then the restart test; LPR lanes per row.
template <int LPR>
__global__ __launch_bounds__(RT) void gm_resid(int N, const int *rp, const int *col, const double *val,
                                               const double *x, const double *b, const double *dinv, double *rvec,
                                               double *z, const GmresState *st, double *part, int nb, int force) {
  if (!cycle_ends(st, force)) return;
  double acc[1] = {0.0};
  const int lane = threadIdx.x & (LPR - 1);
  for (int r = (blockIdx.x * RT + threadIdx.x) / LPR; r < N; r += nb * (RT / LPR)) {
    double s = 0.0;
    for (int q = rp[r] + lane; q < rp[r + 1]; q += LPR) s += val[q] * x[col[q]];
#pragma unroll
    for (int off = LPR / 2; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane == 0) {
      const double rv = b[r] - s;
      rvec[r] = rv;
      z[r] = dinv[r] * rv;
      acc[0] += rv * rv;
    }
  }
  block_store<1>(acc, 1, part, nb);
}

// Finisher launches: a cycle's start, and an iteration's end where the host
// looks or the cycle is full.
__global__ __launch_bounds__(64) void gm_start(const double *part, int nb, GmresState *st, int first, int force) {
  if (!first && !cycle_ends(st, force)) return;
  fin_start(st, part, nb, first != 0);
}
__global__ __launch_bounds__(64) void gm_givens(const double *part, int nb, GmresState *st, int j) {
  if (st->cyc_stop) return;
  const double s = wave_total(part, 0, nb);
  if (threadIdx.x == 0) fin_givens(st, sqrt(s), j);
}

// ------------------------------------------------------------- update
// solve() :471-485 on node dof 4.
__global__ __launch_bounds__(256) void ins_update(int N, double dt, double gm, double4 *vphi, double *phid,
                                                  double *node, const double *x) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= N) return;
  double4 v = vphi[a];
  const double pd = phid[a], pn = x[a];
  v.w = v.w + dt * pd + gm * dt * (pn - pd);
  vphi[a] = v;
  phid[a] = pn;
  if (node) node[4L * a + 3] = pn;
}

// phid of the node records (x y z phid).
__global__ __launch_bounds__(256) void ins_node_phid(int N, const double *phid, double *node) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a < N) node[4L * a + 3] = phid[a];
}

}  // namespace
}  // namespace femx

using namespace femx;

struct femx_ins {
  Mesh *mesh = nullptr;
  femx_ins_params p{};
  hipStream_t st = nullptr;
  long nnz = 0;
  int nb = 1;       // reduction blocks of the row kernels
  long ldv = 0;     // leading dimension of V
  std::vector<int> h_row_ptr, h_col;
  DevBuf<double4> vphi;
  int lpr = 4;      // lanes per row of the CSR kernels
  DevBuf<double> phid, iso, emat, erhs, val, b, dinv, x, rvec, z, w[2], V, part, dir_v, stage;
  DevBuf<int> row_ptr, col, nz_row, c_ptr, cpos, rpos, dir_flag;
  DevBuf<int> econn;  // connectivity in the element kernel's processing order (hexa8)
  // tet4: node records (x y z phid), row order and the places of the
  // elements' columns in the rows
  DevBuf<double4> node;
  DevBuf<int> rord;
  DevBuf<ushort4> rcpos;
  DevBuf<GmresState> gst;
  GmresCtl *ctl = nullptr;  // pinned host copy of the control words
  bool have_solution = false;
  int last_iters = 0;  // Krylov iterations of the previous solve
  KernelTimer timer;
};

namespace {

femx_status ins_fail(femx_ins *s, femx_status r) {
  if (s) {
    if (s->ctl) (void)hipHostFree(s->ctl);
    if (s->st) (void)hipStreamDestroy(s->st);
    delete s;
  }
  return r;
}

// Host side of the reference's pattern (femSparseMatrix::femSparseMatrix,
// src/femMatrix.cpp:29-105) and of the per-entry contribution lists, in
// parallel over node ranges.  Per node r: the sorted unique nodes of its
// elements (r included); per entry (r, c): the element-matrix positions
// e*npe*npe + a*npe + b with conn[e][a] = r, conn[e][b] = c, ascending
// (e, a, b) -- the order the reference adds them.
void host_pattern(const Mesh &m, const std::vector<int> &n_off, const std::vector<int> &n_slot,
                  std::vector<int> &row_ptr, std::vector<int> &col, std::vector<int> &nz_row,
                  std::vector<int> &c_ptr, std::vector<int> &c_idx) {
  const int N = m.N, npe = m.npe;
  const int *conn = m.h_conn.data();
  int nt = (int)std::min(16u, std::max(1u, std::thread::hardware_concurrency()));
  auto run = [&](auto fn) {
    std::vector<std::thread> th;
    for (int t = 0; t < nt; t++)
      th.emplace_back([&, t] {
        const long r0 = (long)N * t / nt, r1 = (long)N * (t + 1) / nt;
        fn((int)r0, (int)r1);
      });
    for (auto &x : th) x.join();
  };
  // pass 1: row lengths
  std::vector<int> len(N);
  run([&](int r0, int r1) {
    std::vector<int> buf;
    for (int r = r0; r < r1; r++) {
      buf.clear();
      buf.push_back(r);
      for (int j = n_off[r]; j < n_off[r + 1]; j++) {
        const int e = n_slot[j] / npe;
        for (int b = 0; b < npe; b++) buf.push_back(conn[(long)e * npe + b]);
      }
      std::sort(buf.begin(), buf.end());
      len[r] = (int)(std::unique(buf.begin(), buf.end()) - buf.begin());
    }
  });
  row_ptr.assign(N + 1, 0);
  for (int r = 0; r < N; r++) row_ptr[r + 1] = row_ptr[r] + len[r];
  const long nnz = row_ptr[N];
  col.resize(nnz);
  nz_row.resize(nnz);
  // contributions per entry: one per (incident slot, b)
  std::vector<long> coff(N + 1, 0);
  for (int r = 0; r < N; r++) coff[r + 1] = coff[r] + (long)(n_off[r + 1] - n_off[r]) * npe;
  c_ptr.assign(nnz + 1, 0);
  c_idx.resize(coff[N]);
  run([&](int r0, int r1) {
    std::vector<int> buf, cnt;
    for (int r = r0; r < r1; r++) {
      buf.clear();
      buf.push_back(r);
      for (int j = n_off[r]; j < n_off[r + 1]; j++) {
        const int e = n_slot[j] / npe;
        for (int b = 0; b < npe; b++) buf.push_back(conn[(long)e * npe + b]);
      }
      std::sort(buf.begin(), buf.end());
      buf.erase(std::unique(buf.begin(), buf.end()), buf.end());
      const int k0 = row_ptr[r];
      for (size_t i = 0; i < buf.size(); i++) {
        col[k0 + i] = buf[i];
        nz_row[k0 + i] = r;
      }
      cnt.assign(buf.size(), 0);
      for (int j = n_off[r]; j < n_off[r + 1]; j++) {
        const int e = n_slot[j] / npe;
        for (int b = 0; b < npe; b++)
          cnt[std::lower_bound(buf.begin(), buf.end(), conn[(long)e * npe + b]) - buf.begin()]++;
      }
      // entries of row r own c_idx[coff[r] .. coff[r+1]) in column order
      long pos = coff[r];
      std::vector<long> at(buf.size());
      for (size_t i = 0; i < buf.size(); i++) {
        at[i] = pos;
        pos += cnt[i];
      }
      for (int j = n_off[r]; j < n_off[r + 1]; j++) {
        const int slot = n_slot[j], e = slot / npe, a = slot % npe;
        for (int b = 0; b < npe; b++) {
          const long i = std::lower_bound(buf.begin(), buf.end(), conn[(long)e * npe + b]) - buf.begin();
          c_idx[at[i]++] = (int)((long)e * npe * npe + a * npe + b);
        }
      }
      long p = coff[r];
      for (size_t i = 0; i < buf.size(); i++) {
        p += cnt[i];
        c_ptr[k0 + i + 1] = (int)p;
      }
    }
  });
}

// The same pattern for ins_rows_tet4, and per corner (in the order of n_slot:
// by node, ascending element) the places of its element's four nodes in the
// node's row.  False if a row has more than row_work(E) element formations for
// one of its lanes, all rows together 1.5 times as many as there are corners
// (the other path's time against 4 E formations by rows is 1.6), or a row is
// too long for 16-bit places: the mesh then takes the element kernel and the
// gathers.
bool host_rows(const Mesh &m, const std::vector<int> &n_off, const std::vector<int> &n_slot,
               std::vector<int> &row_ptr, std::vector<int> &col, std::vector<ushort4> &cpos) {
  const int N = m.N;
  const int *conn = m.h_conn.data();
  constexpr int CH = 4096;  // nodes per work item
  const long items = (N + CH - 1) / CH, most = row_work(m.E);
  std::vector<std::vector<int>> cols(items);
  std::atomic<bool> ok{true};
  std::atomic<long> formed{0};
  row_ptr.assign(N + 1, 0);
  cpos.resize(n_slot.size());
  parallel_items(items, [&](long c) {
    std::vector<int> buf;
    long work = 0;
    for (int r = (int)(c * CH); r < std::min<long>(N, (c + 1) * CH) && ok; r++) {
      buf.assign(1, r);
      for (int j = n_off[r]; j < n_off[r + 1]; j++) {
        const int *q = conn + (n_slot[j] & ~3);
        buf.insert(buf.end(), q, q + 4);
      }
      std::sort(buf.begin(), buf.end());
      buf.erase(std::unique(buf.begin(), buf.end()), buf.end());
      const long passes = ((long)buf.size() + RCAP - 1) / RCAP, elems = n_off[r + 1] - n_off[r];
      work += passes * elems;
      if (buf.size() > 65536 || passes * ((elems + RLPR - 1) / RLPR) > most) ok = false;
      row_ptr[r + 1] = (int)buf.size();
      cols[c].insert(cols[c].end(), buf.begin(), buf.end());
      for (int j = n_off[r]; j < n_off[r + 1]; j++) {
        unsigned short p[4];
        for (int b = 0; b < 4; b++)
          p[b] = (unsigned short)(std::lower_bound(buf.begin(), buf.end(), conn[(n_slot[j] & ~3) + b]) - buf.begin());
        cpos[j] = make_ushort4(p[0], p[1], p[2], p[3]);
      }
    }
    formed += work;
  }, n_slot.size() >= (1u << 16));
  if (!ok || formed > 6L * m.E) return false;
  for (int r = 0; r < N; r++) row_ptr[r + 1] += row_ptr[r];
  col.resize(row_ptr[N]);
  parallel_items(items, [&](long c) { std::copy(cols[c].begin(), cols[c].end(), col.begin() + row_ptr[c * CH]); },
                 col.size() >= (1u << 16));
  return true;
}

InsConst ins_const(const femx_ins_params &p) {
  InsConst k;
  k.am = p.alpha_m;
  k.afdtg = p.alpha_f * p.dt * p.gamma;
  k.om = 1.0 - p.alpha_m;
  k.afdt1g = p.alpha_f * p.dt * (1.0 - p.gamma);
  k.timeTau = 4.0 / (p.dt * p.dt);
  return k;
}

double element_bytes(const Mesh &m) {
  // per element: conn, |d|, the scatter positions and the element matrix and
  // vector; per node (read once): coordinates, velocity/phi, phid
  const double npe = m.npe;
  return m.E * (4.0 * npe + 8.0 + 12.0 * npe * npe + 12.0 * npe) + m.N * (32.0 + 32.0 + 8.0);
}

femx_status read_ctl(femx_ins *s) {
  FEMX_HIP(hipMemcpyAsync(s->ctl, s->gst.p, sizeof(GmresCtl), hipMemcpyDeviceToHost, s->st));
  FEMX_HIP(hipStreamSynchronize(s->st));
  return FEMX_OK;
}

// partials of Gram-Schmidt pass `mode` (three buffers: a pass reads the one before's)
double *orth_part(femx_ins *s, int mode) { return s->part.p + (size_t)mode * MAXM * s->nb; }

template <int LPR>
void launch_spmv(femx_ins *s, const double *src, double *w, int j, bool givens) {
  const int N = s->mesh->N;
  gm_spmv<LPR><<<grid_for((long)N * LPR, RT), RT, 0, s->st>>>(N, s->row_ptr.p, s->col.p, s->val.p, s->z.p, src,
                                                                s->V.p, s->ldv, w, j, s->gst.p, orth_part(s, 2), s->nb,
                                                                givens);
}

template <int LPR>
void launch_resid(femx_ins *s, int force) {
  const int N = s->mesh->N;
  gm_resid<LPR><<<s->nb, RT, 0, s->st>>>(N, s->row_ptr.p, s->col.p, s->val.p, s->x.p, s->b.p, s->dinv.p,
                                         s->rvec.p, s->z.p, s->gst.p, s->part.p, s->nb, force);
}

// Krylov kernels sized for the basis in use: j < J.
template <int J>
void orth_j(femx_ins *s, double *w, int j, int mode) {
  const auto k = mode == 2 ? gm_orth<J, true> : gm_orth<J, false>;
  k<<<s->nb, RT, 0, s->st>>>(s->mesh->N, w, s->V.p, s->ldv, j, s->gst.p, orth_part(s, mode > 0 ? mode - 1 : 0),
                             orth_part(s, mode), s->nb, mode, s->dinv.p, s->z.p);
}
void launch_orth(femx_ins *s, double *w, int j, int mode) {
  if (j < 4) orth_j<4>(s, w, j, mode);
  else if (j < 8) orth_j<8>(s, w, j, mode);
  else if (j < 16) orth_j<16>(s, w, j, mode);
  else orth_j<MAXM>(s, w, j, mode);
}
template <int J>
void xupdate_j(femx_ins *s, int force) {
  gm_xupdate<J><<<s->nb, RT, 0, s->st>>>(s->mesh->N, s->x.p, s->dinv.p, s->V.p, s->ldv, s->gst.p, force);
}
// jmax: the last iteration enqueued in the cycle (the basis used is <= jmax + 1)
void launch_xupdate(femx_ins *s, int jmax, int force) {
  if (jmax < 4) xupdate_j<4>(s, force);
  else if (jmax < 8) xupdate_j<8>(s, force);
  else if (jmax < 16) xupdate_j<16>(s, force);
  else xupdate_j<MAXM>(s, force);
}
// The end of a cycle of jmax + 1 enqueued iterations, if it has ended.
void launch_cycle_end(femx_ins *s, int jmax, int force) {
  gm_backsub<<<1, 64, 0, s->st>>>(s->gst.p, force);
  launch_xupdate(s, jmax, force);
  if (s->lpr == 8) launch_resid<8>(s, force);
  else launch_resid<4>(s, force);
  gm_start<<<1, 64, 0, s->st>>>(s->part.p, s->nb, s->gst.p, 0, force);
}

femx_status ins_solve(femx_ins *s, femx_ins_stats *stats) {
  Mesh &m = *s->mesh;
  const int N = m.N, nb = s->nb, M = s->p.restart;
  const InsConst k = ins_const(s->p);
  int nb0;  // partial sums of ||b||^2
  if (s->node.p) {
    // the mesh and the node records once, the row places of every corner,
    // the matrix and the solve's start written
    const double bytes = m.E * (16.0 + 8.0 + 4.0 * 12.0) + s->nnz * 12.0 + N * (64.0 + 16.0 + 5.0 * 8.0);
    TimedLaunch tl(s->timer, s->timer.kind("ins_rows", bytes), s->st);
    nb0 = std::min(RGRID, grid_for(N, RROWS));
    ins_rows_tet4<<<nb0, 256, 0, s->st>>>(N, s->rord.p, m.g_off.p, m.g_slot.p, s->rcpos.p,
                                          reinterpret_cast<const int4 *>(m.conn.p), s->node.p, s->vphi.p, s->iso.p, k,
                                          s->row_ptr.p, s->col.p, s->dir_flag.p, s->dir_v.p, s->val.p, s->dinv.p,
                                          s->b.p, s->x.p, s->rvec.p, s->z.p, s->part.p);
  } else {
    {
      TimedLaunch tl(s->timer, s->timer.kind("ins_element", element_bytes(m)), s->st);
      const auto el = m.npe == 8 ? ins_element<8> : ins_element<4>;
      el<<<grid_for(m.E, 256), 256, 0, s->st>>>(m.E, s->econn.p, m.xyz.p, s->vphi.p, s->phid.p, s->iso.p, k, s->cpos.p,
                                                s->rpos.p, s->emat.p, s->erhs.p);
    }
    const double bytes = s->nnz * (4.0 + 4.0 + 4.0 + 8.0) + (double)m.E * m.npe * m.npe * 8.0 + N * 12.0;
    {
      TimedLaunch tl(s->timer, s->timer.kind("ins_gather_mat", bytes), s->st);
      ins_gather_mat<<<grid_for(s->nnz, RT), RT, 0, s->st>>>(s->nnz, s->c_ptr.p, s->emat.p, s->nz_row.p, s->col.p,
                                                             s->dir_flag.p, s->val.p, s->dinv.p);
    }
    nb0 = grid_for(N, RT);
    const double rbytes = (double)m.E * m.npe * 8.0 + N * (4.0 + 4.0 + 8.0 + 8.0 + 8.0 * 4);
    TimedLaunch tl(s->timer, s->timer.kind("ins_gather_rhs", rbytes), s->st);
    ins_gather_rhs<<<nb0, RT, 0, s->st>>>(N, m.g_off.p, s->erhs.p, s->dir_flag.p, s->dir_v.p, s->dinv.p, s->b.p,
                                          s->x.p, s->rvec.p, s->z.p, s->part.p);
  }
  gm_start<<<1, 64, 0, s->st>>>(s->part.p, nb0, s->gst.p, 1, 0);
  femx_status r;
  const double spmv_bytes = s->nnz * 12.0 + N * (4.0 + 8.0 * 4);
  // host checks of the cycle flag: first where the previous solve stopped,
  // then at the next iteration, then every CHECK iterations.  Work enqueued
  // past the stop is skipped by the kernels themselves (cyc_stop / done), and
  // a check's read follows the cycle's end enqueued on the chance that it has
  // stopped, so that a solve like the one before takes one round trip.
  int first_check = s->last_iters > 0 ? s->last_iters : CHECK;
  const int spmv_wgs = grid_for((long)N * s->lpr, RT);
  do {
    int next_check = std::min(first_check, M);
    bool givens = false;  // the next SpMV ends the iteration before
    bool ended = false;
    for (int j = 0; j < M && !ended; j++) {
      const double *src = j == 0 ? s->rvec.p : s->w[(j - 1) & 1].p;
      double *w = s->w[j & 1].p;
      {
        TimedLaunch tl(s->timer, s->timer.kind("gm_spmv", spmv_bytes), s->st);
        if (s->lpr == 8) launch_spmv<8>(s, src, w, j, givens);
        else launch_spmv<4>(s, src, w, j, givens);
      }
      for (int mode = 0; mode <= 2; mode++) {
        TimedLaunch tl(s->timer,
                       s->timer.kind("gm_orth", N * 8.0 * (j + (mode ? 3 : 2)) + (mode == 2 ? N * 16.0 : 0.0)), s->st);
        launch_orth(s, w, j, mode);
      }
      const bool full = j + 1 == M;
      const bool look = full || j + 1 == next_check;
      // the next SpMV ends this iteration, unless so many workgroups would sum
      // the same partials that a launch for it is cheaper (3,049 workgroups:
      // 1.4 us against 5.8; 14,260: 7.5 us)
      givens = !look && spmv_wgs <= 8192;
      if (!givens) gm_givens<<<1, 64, 0, s->st>>>(orth_part(s, 2), nb, s->gst.p, j);
      if (!look) continue;
      launch_cycle_end(s, j, full);
      if ((r = read_ctl(s)) != FEMX_OK) return r;
      // a new cycle's start resets cyc_stop: jend tells whether one began
      ended = full || s->ctl->done || s->ctl->jend < 0;
      next_check = j + 1 == first_check ? j + 2 : j + 1 + CHECK;
    }
    first_check = CHECK;
  } while (!s->ctl->done);
  FEMX_HIP(hipGetLastError());
  s->have_solution = true;
  s->last_iters = s->ctl->iters;
  if (stats) {
    stats->iterations = s->ctl->iters;
    stats->converged = s->ctl->conv;
    stats->rel_residual = s->ctl->relres;
  }
  return FEMX_OK;
}

}  // namespace

extern "C" femx_status femx_ins_create(femx_mesh *mesh, const double *el_diff, int n_dir, const int *dir_node,
                                       const double *dir_val, const femx_ins_params *p, femx_ins **out) {
  if (!mesh || !p || !out) {
    set_error("femx_ins_create: null argument");
    return FEMX_ERR_ARG;
  }
  *out = nullptr;
  Mesh &m = mesh->m;
  if (m.npe != 4 && m.npe != 8) {
    set_error("femx_ins_create: tet4 or hexa8 meshes only");
    return FEMX_ERR_UNSUPPORTED;
  }
  if (!(p->dt > 0.0) || p->restart < 1 || p->restart > MAXM || p->max_iter < 1 || !(p->tol >= 0.0)) {
    set_error("femx_ins_create: need dt > 0, 1 <= restart <= 32, max_iter >= 1, tol >= 0");
    return FEMX_ERR_ARG;
  }
  if ((long)m.E * m.npe * m.npe >= (long)INT_MAX) {
    set_error("femx_ins_create: mesh too large for 32-bit element-matrix positions");
    return FEMX_ERR_ARG;
  }
  if (n_dir < 0 || (n_dir > 0 && (!dir_node || !dir_val))) {
    set_error("femx_ins_create: bad Dirichlet arrays");
    return FEMX_ERR_ARG;
  }
  for (int i = 0; i < n_dir; i++)
    if (dir_node[i] < 0 || dir_node[i] >= m.N) {
      set_error("femx_ins_create: Dirichlet node out of range");
      return FEMX_ERR_ARG;
    }
  FEMX_HIP(hipSetDevice(m.device));
  femx_ins *s = new femx_ins();
  s->mesh = &m;
  s->p = *p;
  femx_status r;
  if (hipStreamCreateWithFlags(&s->st, hipStreamNonBlocking) != hipSuccess ||
      hipHostMalloc((void **)&s->ctl, sizeof(GmresCtl), hipHostMallocDefault) != hipSuccess) {
    set_error("femx_ins_create: stream or pinned allocation failed");
    return ins_fail(s, FEMX_ERR_HIP);
  }
  if ((r = upload_tables(m.device)) != FEMX_OK) return ins_fail(s, r);
  const int N = m.N, E = m.E, npe = m.npe;
  // node -> incident (element, corner) slots, ascending element
  std::vector<int> n_off(N + 1, 0), n_slot((size_t)E * npe);
  for (long q = 0; q < (long)E * npe; q++) n_off[m.h_conn[q] + 1]++;
  for (int n = 0; n < N; n++) n_off[n + 1] += n_off[n];
  {
    std::vector<int> at(n_off.begin(), n_off.end() - 1);
    for (long q = 0; q < (long)E * npe; q++) n_slot[at[m.h_conn[q]]++] = (int)q;
  }
  std::vector<int> nz_row, c_ptr, cpos_o, rpos_o, econn, rord;
  std::vector<ushort4> rcpos;
  std::vector<double> iso(E, 0.0);
  const std::vector<int> &ord = m.blk.perm;
  if ((long)ord.size() != E) return ins_fail(s, (set_error("femx_ins_create: mesh has no element order"), FEMX_ERR_ARG));
  // ins_rows_tet4 (node records below 4 GiB, no row too long for it), else
  // the element kernel and the gathers
  const bool rows = npe == 4 && N < (1 << 27) && host_rows(m, n_off, n_slot, s->h_row_ptr, s->h_col, rcpos);
  auto el_iso = [&](int e) {
    if (!el_diff) return 0.0;
    const double *d = el_diff + 3L * e;
    return sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
  };
  if (rows) {
    for (int e = 0; e < E; e++) iso[e] = el_iso(e);
    // rows in the order their nodes first appear along the element blocks
    rord.reserve(N);
    std::vector<char> seen(N, 0);
    for (int n : m.blk.loc_node)
      if (!seen[n]) {
        seen[n] = 1;
        rord.push_back(n);
      }
    for (int n = 0; n < N; n++)
      if (!seen[n]) rord.push_back(n);
  } else {
    std::vector<ushort4>().swap(rcpos);
    std::vector<int> c_idx;
    host_pattern(m, n_off, n_slot, s->h_row_ptr, s->h_col, nz_row, c_ptr, c_idx);
    // where each element value goes: matrix entry contributions and node
    // contributions in the gathers' (ascending element) order
    std::vector<int> cpos(c_idx.size()), rpos((size_t)E * npe);
    for (size_t q = 0; q < c_idx.size(); q++) cpos[c_idx[q]] = (int)q;
    for (size_t j = 0; j < n_slot.size(); j++) rpos[n_slot[j]] = (int)j;
    // the element kernel's inputs in processing order: the Morton block order
    // of the mesh (element t is original element ord[t])
    econn.resize((size_t)E * npe);
    cpos_o.resize(cpos.size());
    rpos_o.resize(rpos.size());
    for (int t = 0; t < E; t++) {
      const int e = ord[t];
      iso[t] = el_iso(e);
      for (int a = 0; a < npe; a++) {
        econn[(size_t)t * npe + a] = m.h_conn[(size_t)e * npe + a];
        rpos_o[(size_t)t * npe + a] = rpos[(size_t)e * npe + a];
      }
      for (int q = 0; q < npe * npe; q++) cpos_o[(size_t)t * npe * npe + q] = cpos[(size_t)e * npe * npe + q];
    }
  }
  s->nnz = s->h_row_ptr[N];
  s->lpr = (double)s->nnz / N > 20.0 ? 8 : 4;
  std::vector<int> dflag(N, 0);
  std::vector<double> dv(N, 0.0);
  for (int i = 0; i < n_dir; i++) {
    dflag[dir_node[i]] = 1;
    dv[dir_node[i]] = dir_val[3L * i];
  }
  s->nb = std::max(1, std::min(MAXNB, grid_for(N, RT)));
  s->ldv = ((long)N + 63) / 64 * 64;
  const int M = p->restart;
  if ((r = s->row_ptr.upload(s->h_row_ptr.data(), N + 1, s->st)) != FEMX_OK ||
      (r = s->col.upload(s->h_col.data(), s->nnz, s->st)) != FEMX_OK ||
      (r = s->nz_row.upload(nz_row.data(), nz_row.size(), s->st)) != FEMX_OK ||
      (r = s->rord.upload(rord.data(), rord.size(), s->st)) != FEMX_OK ||
      (r = s->rcpos.upload(rcpos.data(), rcpos.size(), s->st)) != FEMX_OK ||
      (r = s->c_ptr.upload(c_ptr.data(), c_ptr.size(), s->st)) != FEMX_OK ||
      (r = s->cpos.upload(cpos_o.data(), cpos_o.size(), s->st)) != FEMX_OK ||
      (r = s->rpos.upload(rpos_o.data(), rpos_o.size(), s->st)) != FEMX_OK ||
      (r = s->econn.upload(econn.data(), econn.size(), s->st)) != FEMX_OK || (r = s->z.alloc(N)) != FEMX_OK ||
      (r = s->iso.upload(iso.data(), E, s->st)) != FEMX_OK ||
      (r = s->dir_flag.upload(dflag.data(), N, s->st)) != FEMX_OK ||
      (r = s->dir_v.upload(dv.data(), N, s->st)) != FEMX_OK || (r = s->vphi.alloc(N)) != FEMX_OK ||
      (r = s->phid.alloc(N)) != FEMX_OK || (r = s->emat.alloc(rows ? 0 : (size_t)E * npe * npe)) != FEMX_OK ||
      (r = s->erhs.alloc(rows ? 0 : (size_t)E * npe)) != FEMX_OK || (r = s->node.alloc(rows ? N : 0)) != FEMX_OK || (r = s->val.alloc(s->nnz)) != FEMX_OK ||
      (r = s->b.alloc(N)) != FEMX_OK || (r = s->dinv.alloc(N)) != FEMX_OK || (r = s->x.alloc(N)) != FEMX_OK ||
      (r = s->rvec.alloc(N)) != FEMX_OK || (r = s->w[0].alloc(N)) != FEMX_OK || (r = s->w[1].alloc(N)) != FEMX_OK ||
      (r = s->V.alloc((size_t)s->ldv * (M + 1))) != FEMX_OK ||
      (r = s->part.alloc(std::max({(size_t)3 * MAXM * s->nb, (size_t)grid_for(N, RT), (size_t)RGRID}))) != FEMX_OK || (r = s->stage.alloc((size_t)N * 3)) != FEMX_OK ||
      (r = s->gst.alloc(1)) != FEMX_OK)
    return ins_fail(s, r);
  GmresState h0;
  std::memset(&h0, 0, sizeof(h0));
  h0.tol = p->tol;
  h0.max_iter = p->max_iter;
  hipError_t he = hipMemsetAsync(s->vphi.p, 0, sizeof(double4) * N, s->st);
  if (he == hipSuccess) he = hipMemsetAsync(s->phid.p, 0, sizeof(double) * N, s->st);
  // coordinates with a zero fourth component: phid = 0
  if (he == hipSuccess && rows)
    he = hipMemcpyAsync(s->node.p, m.xyz.p, sizeof(double4) * N, hipMemcpyDeviceToDevice, s->st);
  if (he == hipSuccess) he = hipMemsetAsync(s->x.p, 0, sizeof(double) * N, s->st);
  if (he == hipSuccess) he = hipMemsetAsync(s->V.p, 0, sizeof(double) * s->ldv * (M + 1), s->st);
  if (he == hipSuccess) he = hipMemcpyAsync(s->gst.p, &h0, sizeof(h0), hipMemcpyHostToDevice, s->st);
  if (he == hipSuccess) he = hipStreamSynchronize(s->st);
  if (he != hipSuccess) return ins_fail(s, hip_fail(he, "femx_ins_create: initial fills"));
  *out = s;
  return FEMX_OK;
}

extern "C" femx_status femx_ins_destroy(femx_ins *s) {
  if (!s) return FEMX_OK;
  (void)hipSetDevice(s->mesh->device);
  (void)hipStreamSynchronize(s->st);
  s->timer.resolve();
  if (s->ctl) (void)hipHostFree(s->ctl);
  s->ctl = nullptr;
  (void)hipStreamDestroy(s->st);
  s->st = nullptr;
  delete s;
  return FEMX_OK;
}

extern "C" femx_status femx_ins_set_state(femx_ins *s, const double *phi, const double *phi_dot, const double *vel) {
  if (!s) {
    set_error("femx_ins_set_state: null handle");
    return FEMX_ERR_ARG;
  }
  FEMX_HIP(hipSetDevice(s->mesh->device));
  const int N = s->mesh->N;
  if (phi_dot) {
    FEMX_HIP(hipMemcpyAsync(s->phid.p, phi_dot, sizeof(double) * N, hipMemcpyHostToDevice, s->st));
    if (s->node.p)
      ins_node_phid<<<grid_for(N, 256), 256, 0, s->st>>>(N, s->phid.p, reinterpret_cast<double *>(s->node.p));
  }
  if (phi) {
    FEMX_HIP(hipMemcpyAsync(s->stage.p, phi, sizeof(double) * N, hipMemcpyHostToDevice, s->st));
    ins_pack<<<grid_for(N, 256), 256, 0, s->st>>>(N, s->stage.p, nullptr, s->vphi.p);
  }
  if (vel) {
    FEMX_HIP(hipStreamSynchronize(s->st));  // the staging buffer is reused
    FEMX_HIP(hipMemcpyAsync(s->stage.p, vel, sizeof(double) * 3 * N, hipMemcpyHostToDevice, s->st));
    ins_pack<<<grid_for(N, 256), 256, 0, s->st>>>(N, nullptr, s->stage.p, s->vphi.p);
  }
  FEMX_HIP(hipGetLastError());
  FEMX_HIP(hipStreamSynchronize(s->st));
  return FEMX_OK;
}

extern "C" femx_status femx_ins_prescribe_velocity(femx_ins *s, int type, double t, const double *node_vel) {
  if (!s) {
    set_error("femx_ins_prescribe_velocity: null handle");
    return FEMX_ERR_ARG;
  }
  if (type < 0 || type > 2 || (type == 2 && !node_vel)) {
    set_error("femx_ins_prescribe_velocity: type must be 0, 1 or 2 (2 needs node velocities)");
    return FEMX_ERR_ARG;
  }
  FEMX_HIP(hipSetDevice(s->mesh->device));
  const int N = s->mesh->N;
  if (type == 2) {
    FEMX_HIP(hipStreamSynchronize(s->st));  // the staging buffer is reused
    FEMX_HIP(hipMemcpyAsync(s->stage.p, node_vel, sizeof(double) * 3 * N, hipMemcpyHostToDevice, s->st));
  }
  {
    TimedLaunch tl(s->timer, s->timer.kind("ins_prescribe", N * (32.0 + 32.0 + 32.0)), s->st);
    ins_prescribe<<<grid_for(N, 256), 256, 0, s->st>>>(N, type, t, s->mesh->xyz.p, s->stage.p, s->vphi.p);
  }
  FEMX_HIP(hipGetLastError());
  return FEMX_OK;
}

extern "C" femx_status femx_ins_advdiff_solve(femx_ins *s, femx_ins_stats *stats) {
  if (!s) {
    set_error("femx_ins_advdiff_solve: null handle");
    return FEMX_ERR_ARG;
  }
  FEMX_HIP(hipSetDevice(s->mesh->device));
  return ins_solve(s, stats);
}

extern "C" femx_status femx_ins_update(femx_ins *s) {
  if (!s) {
    set_error("femx_ins_update: null handle");
    return FEMX_ERR_ARG;
  }
  if (!s->have_solution) {
    set_error("femx_ins_update: no advection-diffusion solve since the last update");
    return FEMX_ERR_ARG;
  }
  FEMX_HIP(hipSetDevice(s->mesh->device));
  const int N = s->mesh->N;
  {
    TimedLaunch tl(s->timer, s->timer.kind("ins_update", N * (32.0 * 2 + 8.0 * 3)), s->st);
    ins_update<<<grid_for(N, 256), 256, 0, s->st>>>(N, s->p.dt, s->p.gamma, s->vphi.p, s->phid.p,
                                                      reinterpret_cast<double *>(s->node.p), s->x.p);
  }
  FEMX_HIP(hipGetLastError());
  s->have_solution = false;
  return FEMX_OK;
}

extern "C" femx_status femx_ins_get_state(femx_ins *s, double *phi, double *phi_dot, double *vel) {
  if (!s) {
    set_error("femx_ins_get_state: null handle");
    return FEMX_ERR_ARG;
  }
  FEMX_HIP(hipSetDevice(s->mesh->device));
  const int N = s->mesh->N;
  // phi passes through the Krylov work vector w[0], free between solves
  double *dphi = phi ? s->w[0].p : nullptr, *dvel = vel ? s->stage.p : nullptr;
  ReadPiece rb[3];
  int nrb = 0;
  if (phi || vel) {
    ins_unpack<<<grid_for(N, 256), 256, 0, s->st>>>(N, s->vphi.p, dphi, dvel);
    FEMX_HIP(hipGetLastError());
  }
  if (phi) rb[nrb++] = {phi, dphi, sizeof(double) * N};
  if (vel) rb[nrb++] = {vel, dvel, sizeof(double) * 3 * N};
  if (phi_dot) rb[nrb++] = {phi_dot, s->phid.p, sizeof(double) * N};
  return read_back(s->mesh->device, s->st, rb, nrb);
}

extern "C" femx_status femx_ins_get_system(femx_ins *s, int *row_ptr, int *col, double *val, double *rhs,
                                           double *phid_new, long long *nnz) {
  if (!s) {
    set_error("femx_ins_get_system: null handle");
    return FEMX_ERR_ARG;
  }
  FEMX_HIP(hipSetDevice(s->mesh->device));
  const int N = s->mesh->N;
  if (nnz) *nnz = s->nnz;
  if (row_ptr) std::memcpy(row_ptr, s->h_row_ptr.data(), sizeof(int) * (N + 1));
  if (col) std::memcpy(col, s->h_col.data(), sizeof(int) * s->nnz);
  if (val) FEMX_HIP(hipMemcpyAsync(val, s->val.p, sizeof(double) * s->nnz, hipMemcpyDeviceToHost, s->st));
  if (rhs) FEMX_HIP(hipMemcpyAsync(rhs, s->b.p, sizeof(double) * N, hipMemcpyDeviceToHost, s->st));
  if (phid_new) FEMX_HIP(hipMemcpyAsync(phid_new, s->x.p, sizeof(double) * N, hipMemcpyDeviceToHost, s->st));
  FEMX_HIP(hipStreamSynchronize(s->st));
  return FEMX_OK;
}

extern "C" femx_status femx_ins_sync(femx_ins *s) {
  if (!s) {
    set_error("femx_ins_sync: null handle");
    return FEMX_ERR_ARG;
  }
  FEMX_HIP(hipSetDevice(s->mesh->device));
  FEMX_HIP(hipStreamSynchronize(s->st));
  return FEMX_OK;
}

extern "C" void *femx_ins_stream(femx_ins *s) { return s ? (void *)s->st : nullptr; }

extern "C" femx_status femx_ins_kernel_timing(femx_ins *s, int enable) {
  if (!s) {
    set_error("femx_ins_kernel_timing: null handle");
    return FEMX_ERR_ARG;
  }
  if (enable) s->timer.reset();
  else s->timer.resolve();
  s->timer.enabled = enable != 0;
  return FEMX_OK;
}

extern "C" int femx_ins_kernel_times(femx_ins *s, femx_kernel_time *out, int max_entries) {
  if (!s) return 0;
  return s->timer.export_to(out, max_entries);
}
