// kernels_general.hpp -- SIPG Poisson operator on meshes with moved vertices
// ((bi/tri)linear cells), matrix-free with QGauss(p+1) on cells and faces:
// Laplace::DG::MF::Operator::{apply_cell, apply_face, apply_boundary}
// (apps/laplace_integrator.h:613-743).  The geometry is recomputed on the fly from
// the multilinear coefficients of each cell's map, so the only HBM traffic is the
// vectors and the (n+1)^dim vertex array.  Arithmetic in the vector type (the map
// coefficients are formed in FP64 from the vertices).  Faces are evaluated
// element-centrically: every cell integrates its own test functions against the
// flux of each of its 2*dim faces (interior faces are evaluated from both sides,
// which keeps the kernels free of write races).
//
// One lane per line.  A cell is NP^(DIM-1) lanes of one wave; in 3D lane (q0, q1)
// holds the x-line (y, z) = (q0, q1) of the cell and, for the faces of direction d,
// the line along d at the tangential node (e1, e2) = (q0, q1) of the cell and of its
// neighbours (in 2D the one lane index q0).  Products along the lane's own line run
// in registers; products along a lane index take the other lines' values from the
// lanes that hold them, rotated (lane (q + r) mod NP with coefficient row q of the
// matrix started at column q), for NP = 4 by DPP (in 3D a cell is a DPP row, its
// quads the first lane index), by ds_bpermute for NP < 4, and for NP = 5 in order through
// a row in LDS; the contributions of the faces of other directions pass through LDS once.
//
// Geometry from the map coefficients A_S.  The two cells of a face share its
// tangents t1, t2; with w = t1 x t2, a normal-direction Jacobian column J_d of
// either cell, g_ij = t_i . t_j and r_i = t_i . J_d,
//   dS J^{-1} n = +-(w.w, g12 r2 - g22 r1, g12 r1 - g11 r2) / |J_d . w|
// in the face frame (d, e1, e2) (2D: w = t1 turned, +-(w.w, -r1) / |J_d . w|), and
// dS = |w|: one reciprocal per cell side and one square root.  At a cell point the
// reference flux is C^T C grad / |det J| with the adjugate C of J.
//
// Bound by VALU issue (3D Q3 FP32: 2571 VALU instructions per wave of four cells).
// 64^3 Q3 apply: FP32 221 us, FP64 412 us (590 / 1240 us with one thread per node
// and every product through LDS); 40^3 Q4 217 / 414 us (296 / 640), 60^3 Q2
// 132 / 244 us (326 / 618), 80^3 Q1 155 / 237 us (578 / 1039).  2D: 300^2 Q3 FP64
// 17 us (123), 700^2 Q1 FP32 21 us (292).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.hpp"

namespace tpss
{
template<int NP, typename T>
struct GeneralTab
{
  T V[NP * NP];   // V[q*NP + i]  = phi_i(x_q), Gauss points x_q
  T Dv[NP * NP];  // Dv[q*NP + i] = phi_i'(x_q)
  T qx[NP], qw[NP];
  T fd[2][NP];    // phi_i'(0), phi_i'(1)
  // rows of V, Dv and of their transposes in the order of the lanes' gathers: rotated
  // to start at the diagonal, R[m][q*NP + r] = entry (q, (q + r) mod NP), or entry (q, r)
  // where GatherRows serves them (moved_row_gathers)
  T R[4][NP * NP];
};

// The values of five lanes in order, through a row of a wave's own LDS buffer (a wave's
// LDS accesses run in order: no barrier).  The rows cost a write and the reads of five
// values; the four (FP64: eight) ds_bpermute instructions of a rotation, about 8 cycles
// of the CU's LDS each, bounded the split Q4 form: 9^3 FP64 13.5 -> 9.9 us, 48^3 FP64 1018 ->
// 712, FP32 503 -> 372.
template<int ROWS, typename T>
struct GatherRows
{
  static constexpr int W = 16 / int(sizeof(T)), STRIDE = sizeof(T) == 4 ? 8 : 6;  // rows of 16-byte chunks
  static constexpr int SIZE = ROWS * STRIDE;
  typedef T vec __attribute__((ext_vector_type(16 / sizeof(T))));
  static __device__ __forceinline__ void gather(T *buf, int row, int at, T v, T *o)
  {
    // volatile: the row is read as its five lanes have written it
    typedef volatile __attribute__((address_space(3))) T *ptr;
    typedef volatile __attribute__((address_space(3))) vec *vptr;
    ptr p = (ptr)buf + row * STRIDE;
    p[at] = v;
#pragma unroll
    for(int k = 0; k < 4 / W; ++k)
    {
      const vec w = ((vptr)p)[k];
#pragma unroll
      for(int e = 0; e < W; ++e) o[W * k + e] = w[e];
    }
    o[4] = p[4];
  }
};

template<typename T>
__device__ __forceinline__ T root(T a)
{
  if constexpr(std::is_same<T, float>::value)
    return __builtin_amdgcn_sqrtf(a);
  else
    return sqrt(a);
}

template<int DIM, int NP>
constexpr int moved_cells_per_block()
{
  return 64 / cpow(NP, DIM - 1);
}

// Launches of at most this many blocks run the split form (several waves per block of
// cells, below), whose launch takes as long as its longest wave while the GPU holds all of
// them at once.  Applies in us, split against one wave per block of cells:
//   3D Q1-Q3, a wave per SIMD: 24^3 Q1 (864 blocks) FP64 12.6 / 11.3, FP32 8.1 / 9.5; 18^3 Q2
//   (834) 14.1 / 13.6, 9.4 / 10.5; 22^3 Q2 (1522) 19.8 / 18.6, 11.9 / 12.5; 18^3 Q3 (1458)
//   16.1 / 17.1, 10.9 / 11.9; 22^3 Q3 (2662) 27.1 / 24.4, 16.5 / 15.7;
//   3D Q4 always: 12^3 17.2 / 28.8, 10.9 / 16.5; 48^3 712 / 976, 372 / 484 (the one-wave form
//   spills 36 registers in FP64);
//   2D FP64: 96^2 Q2 (439) 5.4 / 7.0, 128^2 Q2 (781) 9.3 / 7.5; 64^2 Q3 (256) 4.8 / 5.7, 72^2
//   Q3 (324) 6.9 / 5.8; 64^2 Q4 (342) 9.1 / 10.3, 80^2 Q4 (534) 12.4 / 11.0;
//   2D FP32: 96^2 Q3 (576) 4.8 / 4.8, 128^2 Q3 (1024) 5.4 / 4.9; 96^2 Q4 (768) 6.0 / 7.1,
//   128^2 Q4 (1366) 10.7 / 8.7.
template<int DIM, int NP, typename VT>
constexpr unsigned moved_split_max_blocks()
{
  if(DIM == 3) return NP == 5 ? ~0u : 1024;
  return std::is_same<VT, float>::value ? 768 : NP == 4 ? 256 : 512;
}

// On a face x_d = 0 the tangents are map coefficients of the cell, on x_d = 1 sums of two.
// In FP32 those are formed in FP64 from the vertices too, like every coefficient: sums of
// rounded coefficients differ from the neighbour's tangents of the same face (FP32 error of a
// sweep, 16^2 Q4 5.4e-7 with the sums, 3.2e-7 without; 30^3 Q1 1.02e-7, 0.92e-7).
template<typename T>
constexpr bool face_tangents_staged()
{
  return std::is_same<T, float>::value;
}

// whether the products across lanes take their values in order from GatherRows
template<int NP, bool SPLIT>
constexpr bool moved_row_gathers()
{
  return NP == 5 && SPLIT;
}

// 1/a: the hardware reciprocal, in FP64 refined by two Newton steps (within an ulp
// or two of the correctly rounded quotient)
__device__ __forceinline__ float fast_recip(float a) { return __builtin_amdgcn_rcpf(a); }
__device__ __forceinline__ double fast_recip(double a)
{
  double r = __builtin_amdgcn_rcp(a);
  r = fma(r, fma(-a, r, 1.0), r);
  return fma(r, fma(-a, r, 1.0), r);
}

// Waves per SIMD the register allocation must allow.  Split FP64 Q4 takes 271 registers
// unbounded: 12^3 30.7 us with one wave per SIMD, 24.1 with two (both with ds_bpermute).
template<int NP, typename VT, bool SPLIT>
constexpr int moved_min_waves()
{
  constexpr bool F32 = std::is_same<VT, float>::value;
  if(SPLIT) return NP < 5 ? 1 : F32 ? 3 : 2;
  return F32 ? 3 : 2;
}

// SPLIT: four waves per block of cells, one for the cell term and one per direction of
// the faces, for launches that leave most of the GPU idle otherwise (the time of a
// launch is then that of one wave: 6^3 Q4 FP64 22.2 us unsplit, 7.5 split).
template<int NP, typename VT, bool RESIDUAL, bool SPLIT>
__global__ void __launch_bounds__(SPLIT ? 256 : 64, (moved_min_waves<NP, VT, SPLIT>()))
k_sipg_moved(const VT *__restrict__ x, VT *__restrict__ y, const VT *__restrict__ b,
             const double *__restrict__ vert, const GeneralTab<NP, VT> tab, const int n,
             const VT ipg, const uint32_t *__restrict__ cells, const int64_t count)
{
  using T = VT;
  constexpr int NL = NP * NP, NDC = NL * NP, CPB = moved_cells_per_block<3, NP>(), P = NP - 1;
  constexpr int CSL = (64 + NL - 1) / NL;  // cell slots, idle lanes included
  constexpr int NTAB = int(sizeof(GeneralTab<NP, T>) / sizeof(T));
  __shared__ __align__(16) T tl[NTAB];
  __shared__ double X[CSL][32][3];       // corners; far corners of the face neighbours
  __shared__ T A_[CSL][8][3];            // map coefficients
  constexpr bool FT = face_tangents_staged<T>();
  __shared__ T F_[FT ? CSL : 1][3][3][3];  // tangents of the faces x_d = 1
  __shared__ T N_[CSL][6][4][3];         // normal columns of the neighbours' maps on the faces
  __shared__ __align__(16) T L1[CSL][NDC], L2[CSL][NDC];  // y- and z-face contributions
  __shared__ __align__(16) T L0[SPLIT ? CSL : 1][NDC];     // x-face contributions of a split block
  static_assert(SPLIT || NP < 5, "3D Q4 runs the split form");
  constexpr bool ROWS = moved_row_gathers<NP, SPLIT>();
  using GR = GatherRows<CSL * NP, T>;
  __shared__ __align__(16) T G[ROWS ? 4 * GR::SIZE : 1];

  const int part = SPLIT ? __builtin_amdgcn_readfirstlane(int(threadIdx.x)) / 64 : 0;
  const int t = threadIdx.x % 64, cs = t / NL, q = t % NL;
  const int q0 = q % NP, q1 = q / NP;
  const int64_t per = int64_t(gridDim.x) / 8;  // the grid is a multiple of eight blocks
  const int64_t slot = (int64_t(blockIdx.x % 8) * per + blockIdx.x / 8) * CPB + cs;
  const bool act = cs < CPB && slot < count;
  const int64_t sl = act ? slot : 0;
  const int64_t cell = cells ? int64_t(cells[sl]) : sl;
  const int ci = int(cell);
  const int cc[3] = {ci % n, (ci / n) % n, ci / (n * n)};
  int ra[2][NP];  // ds_bpermute addresses of the rotations (NP < 4)
  if constexpr(NP < 4)
#pragma unroll
    for(int r = 0; r < NP; ++r)
    {
      ra[0][r] = 4 * (cs * NL + (q0 + r) % NP + NP * q1);
      ra[1][r] = 4 * (cs * NL + q0 + NP * ((q1 + r) % NP));
    }

  auto gather0 = [&](T v, T *o) {
    if constexpr(ROWS)
      GR::gather(G + part * GR::SIZE, cs * NP + q1, q0, v, o);
    else
      lane_gather<NP, 0>(v, ra[0], o);
  };
  auto gather1 = [&](T v, T *o) {
    if constexpr(ROWS)
      GR::gather(G + part * GR::SIZE, cs * NP + q0, q1, v, o);
    else
      lane_gather<NP, 1>(v, ra[1], o);
  };

  for(int i = threadIdx.x; i < NTAB; i += SPLIT ? 256 : 64) tl[i] = reinterpret_cast<const T *>(&tab)[i];
  // ---- loads: lines of the cell and of its face neighbours, vertices
  const T *xc = x + cell * NDC;
  const int at[3] = {NP * q, q0 + NL * q1, q};      // the lane's line along d in a cell
  constexpr int st[3] = {1, NP, NL};
  T ol[3][NP], nl[3][2][NP];
#pragma unroll
  for(int d = 0; d < 3; ++d)
  {
    if(SPLIT && part != d + 1 && !(d == 0 && part == 0)) continue;
    const int64_t shift = (d == 0 ? int64_t(1) : d == 1 ? int64_t(n) : int64_t(n) * n) * NDC;
    const T *pl = xc + at[d] - (cc[d] > 0 ? shift : 0), *pr = xc + at[d] + (cc[d] < n - 1 ? shift : 0);
    if(d == 0)
    {
      load_row<NP>(xc + at[0], ol[0]);
      load_row<NP>(pl, nl[0][0]);
      load_row<NP>(pr, nl[0][1]);
    }
    else
#pragma unroll
      for(int j = 0; j < NP; ++j)
      {
        ol[d][j] = xc[at[d] + j * st[d]];
        nl[d][0][j] = pl[j * st[d]];
        nl[d][1][j] = pr[j * st[d]];
      }
  }
  {
    // vertex c < 8: corner c; else the corner of the neighbour across face
    // f = (c - 8) / 4 opposite face corner (c - 8) % 4 (absent neighbour: any vertex)
    const int v1 = n + 1, v2 = v1 * v1, vb = cc[0] + v1 * cc[1] + v2 * cc[2];
    for(int c = q + NL * part; c < 32; c += SPLIT ? 4 * NL : NL)
    {
      const int f = (c - 8) >> 2, d = f >> 1, side = f & 1;
      int o0 = c & 1, o1 = (c >> 1) & 1, o2 = c >> 2;
      if(c >= 8)
      {
        const int far = side ? 2 : -1, b1 = c & 1, b2 = (c >> 1) & 1;
        o0 = d == 0 ? far : b1;
        o1 = d == 1 ? far : (d == 0 ? b1 : b2);
        o2 = d == 2 ? far : b2;
        const int cd = d == 0 ? cc[0] : d == 1 ? cc[1] : cc[2];
        if(side ? cd == n - 1 : cd == 0) o0 = o1 = o2 = 0;
      }
      const double *pv = vert + int64_t(vb + o0 + v1 * o1 + v2 * o2) * 3;
#pragma unroll
      for(int a = 0; a < 3; ++a) X[cs][c][a] = pv[a];
    }
  }
  __syncthreads();
  // ---- traces on the tangential nodes: value and normal derivative of the cell and
  // of its neighbour (0 where there is none), on both sides of every direction
  T vo[3][2], go_[3][2], vn[3][2], gn_[3][2];
#pragma unroll
  for(int d = 0; d < 3; ++d)
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      if(SPLIT && part != d + 1) continue;
      const bool in = side ? cc[d] < n - 1 : cc[d] > 0;
      T dd = 0, dn = 0;
#pragma unroll
      for(int j = 0; j < NP; ++j)
      {
        dd += tab.fd[side][j] * ol[d][j];
        dn += tab.fd[1 - side][j] * nl[d][side][j];
      }
      vo[d][side] = ol[d][side ? P : 0];
      go_[d][side] = dd;
      vn[d][side] = in ? nl[d][side][side ? 0 : P] : T(0);
      gn_[d][side] = in ? dn : T(0);
    }
  // ---- map coefficients, formed in FP64: item (coordinate a) of the cell, then of
  // the six neighbours' normal columns
  for(int it = q + NL * part; it < 21; it += SPLIT ? 4 * NL : NL)
  {
    const int a = it % 3, f = it / 3 - 1;
    if(f < 0)
    {
      double c[8];
#pragma unroll
      for(int R = 0; R < 8; ++R) c[R] = X[cs][R][a];
#pragma unroll
      for(int e = 0; e < 3; ++e)
#pragma unroll
        for(int S = 0; S < 8; ++S)
          if((S >> e) & 1) c[S] -= c[S ^ (1 << e)];
#pragma unroll
      for(int S = 1; S < 8; ++S) A_[cs][S][a] = T(c[S]);
      continue;
    }
    const int d = f >> 1, side = f & 1;
    const int m1 = d == 0 ? 2 : 1, m2 = d == 2 ? 2 : 4;  // corner bits along e1, e2
    const bool in = side ? cc[0] * (d == 0) + cc[1] * (d == 1) + cc[2] * (d == 2) < n - 1
                         : cc[0] * (d == 0) + cc[1] * (d == 1) + cc[2] * (d == 2) > 0;
    double e[4], c[4];
#pragma unroll
    for(int cp = 0; cp < 4; ++cp)
    {
      const int cy = (side << d) | ((cp & 1) ? m1 : 0) | ((cp >> 1) ? m2 : 0);
      // absent neighbour: the cell's own edge (finite; its products are multiplied by 0)
      const double far = in ? X[cs][8 + 4 * f + cp][a] : X[cs][cy ^ (1 << d)][a];
      c[cp] = X[cs][cy][a];
      const double ed = far - c[cp];
      e[cp] = (side == 1) == in ? ed : -ed;
    }
    N_[cs][f][0][a] = T(e[0]);
    N_[cs][f][1][a] = T(e[1] - e[0]);
    N_[cs][f][2][a] = T(e[2] - e[0]);
    N_[cs][f][3][a] = T(e[3] - e[2] - e[1] + e[0]);
    if(FT && side == 1)
    {
      F_[cs][d][0][a] = T(c[1] - c[0]);
      F_[cs][d][1][a] = T(c[2] - c[0]);
      F_[cs][d][2][a] = T(c[3] - c[2] - c[1] + c[0]);
    }
  }
  __syncthreads();
  // For NP >= 4 the lanes' rows of the tables and the map coefficients are read from
  // LDS again for every face (a compiler fence keeps them from staying in registers,
  // where they spill: 64^3 Q3 FP64 556 us kept, 412 us re-read), in the split form the
  // transposed rows only ahead of the projections (12^3 Q4 FP32 14.3 -> 13.4 us, FP64 without
  // its 16 spilled registers); shorter lines keep them (60^3 Q2 FP64 244 us kept, 300 re-read)
  auto rows = [&](int m, int q_, T *o) {
#pragma unroll
    for(int r = 0; r < NP; ++r) o[r] = tl[2 * NL + 4 * NP + m * NL + q_ * NP + r];
  };
  T A[8][3], Va[NP], Da[NP], VaT[NP], DaT[NP], Vb[NP], Db[NP], VbT[NP], DbT[NP];
  constexpr bool LATE = SPLIT && NP >= 4;
  auto fetch_t = [&]() {
    if(LATE) asm volatile("" ::: "memory");
    rows(2, q0, VaT), rows(3, q0, DaT);
    rows(2, q1, VbT), rows(3, q1, DbT);
  };
  auto fetch = [&]() {
    asm volatile("" ::: "memory");
#pragma unroll
    for(int S = 1; S < 8; ++S)
#pragma unroll
      for(int a = 0; a < 3; ++a) A[S][a] = A_[cs][S][a];
    rows(0, q0, Va), rows(1, q0, Da);
    rows(0, q1, Vb), rows(1, q1, Db);
    if constexpr(!LATE) fetch_t();
  };
  fetch();
  const T p0 = tl[2 * NL + q0], p1 = tl[2 * NL + q1];                  // points along the lane indices
  const T wq = tl[2 * NL + NP + q0] * tl[2 * NL + NP + q1];

  T acc[3][NP];
#pragma unroll
  for(int d = 0; d < 3; ++d)
#pragma unroll
    for(int j = 0; j < NP; ++j) acc[d][j] = 0;

  // ---------------- cell term
  if(!SPLIT || part == 0)
  {
    T F0[NP], F1[NP], F2[NP];
    T g0[NP], g1[NP], g2[NP];
#pragma unroll
    for(int i = 0; i < NP; ++i)
    {
      T v = 0, g = 0, rv[NP], rg[NP], r2[NP];
#pragma unroll
      for(int j = 0; j < NP; ++j)
      {
        v += tab.V[i * NP + j] * ol[0][j];
        g += tab.Dv[i * NP + j] * ol[0][j];
      }
      gather0(v, rv);
      gather0(g, rg);
      gather1(dotn<NP>(Va, rg), r2);
      g0[i] = dotn<NP>(Vb, r2);
      gather1(dotn<NP>(Da, rv), r2);
      g1[i] = dotn<NP>(Vb, r2);
      gather1(dotn<NP>(Va, rv), r2);
      g2[i] = dotn<NP>(Db, r2);
    }
    // Jacobian columns: J_0 constant along the line, J_1 and J_2 linear in x
    T c0[3], c1[3], s1[3], c2[3], s2[3];
#pragma unroll
    for(int a = 0; a < 3; ++a)
    {
      s1[a] = A[3][a] + p1 * A[7][a];
      s2[a] = A[5][a] + p0 * A[7][a];
      c0[a] = A[1][a] + p1 * A[5][a] + p0 * s1[a];
      c1[a] = A[2][a] + p1 * A[6][a];
      c2[a] = A[4][a] + p0 * A[6][a];
    }
#pragma unroll
    for(int i = 0; i < NP; ++i)
    {
      const T xi = tab.qx[i];
      T J1[3], J2[3], R0[3], R1[3], R2[3];
#pragma unroll
      for(int a = 0; a < 3; ++a)
      {
        J1[a] = c1[a] + xi * s1[a];
        J2[a] = c2[a] + xi * s2[a];
      }
      // rows of the adjugate: J_1 x J_2, J_2 x J_0, J_0 x J_1
#pragma unroll
      for(int a = 0; a < 3; ++a)
      {
        const int k = (a + 1) % 3, l = (a + 2) % 3;
        R0[a] = J1[k] * J2[l] - J1[l] * J2[k];
        R1[a] = J2[k] * c0[l] - J2[l] * c0[k];
        R2[a] = c0[k] * J1[l] - c0[l] * J1[k];
      }
      const T det = c0[0] * R0[0] + c0[1] * R0[1] + c0[2] * R0[2];
      const T w = wq * tab.qw[i] * fast_recip(fabs(det));
      T h[3];
#pragma unroll
      for(int a = 0; a < 3; ++a) h[a] = w * (R0[a] * g0[i] + R1[a] * g1[i] + R2[a] * g2[i]);
      F0[i] = R0[0] * h[0] + R0[1] * h[1] + R0[2] * h[2];
      F1[i] = R1[0] * h[0] + R1[1] * h[1] + R1[2] * h[2];
      F2[i] = R2[0] * h[0] + R2[1] * h[1] + R2[2] * h[2];
    }
    if constexpr(LATE) fetch_t();
#pragma unroll
    for(int i = 0; i < NP; ++i)
    {
      T r0[NP], r1[NP], r2[NP];
      gather1(F0[i], r0);
      gather1(F1[i], r1);
      gather1(F2[i], r2);
      const T z0 = dotn<NP>(VbT, r0), z1 = dotn<NP>(VbT, r1), z2 = dotn<NP>(DbT, r2);
      gather0(z0, r0);
      gather0(z1, r1);
      gather0(z2, r2);
      const T a0 = dotn<NP>(VaT, r0), a1 = dotn<NP>(DaT, r1) + dotn<NP>(VaT, r2);
#pragma unroll
      for(int j = 0; j < NP; ++j) acc[0][j] += tab.Dv[i * NP + j] * a0 + tab.V[i * NP + j] * a1;
    }
  }

  // ---------------- faces
  const int lane0 = min(cs, CPB - 1) * NL;  // the lane of the cell's first face point
#pragma unroll
  for(int d = 0; d < 3; ++d)
  {
    if(SPLIT && part != d + 1) continue;
    const int bd = 1 << d, b1 = d == 0 ? 2 : 1, b2 = d == 2 ? 2 : 4, b12 = b1 | b2;
    T jd[3];
#pragma unroll
    for(int a = 0; a < 3; ++a)
      jd[a] = A[bd][a] + p0 * A[bd | b1][a] + p1 * (A[bd | b2][a] + p0 * A[7][a]);
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      const int f = 2 * d + side;
      const bool in = side ? cc[d] < n - 1 : cc[d] > 0;
      if constexpr(NP >= 4) fetch();
      // at the face points: jump, normal and tangential reference derivatives
      T r0[NP], r1[NP], jump, go[3], gn[3];
      {
        T m[NP];
        gather0(vo[d][side], r0);
        gather0(vn[d][side], r1);
        const T Vo = dotn<NP>(Va, r0), Vn = dotn<NP>(Va, r1);
        const T Do = dotn<NP>(Da, r0), Dn = dotn<NP>(Da, r1);
        gather0(go_[d][side], r0);
        gather0(gn_[d][side], r1);
        const T No = dotn<NP>(Va, r0), Nn = dotn<NP>(Va, r1);
        gather1(Vo, r0);
        gather1(Vn, r1);
        go[2] = dotn<NP>(Db, r0);
        gn[2] = dotn<NP>(Db, r1);
#pragma unroll
        for(int r = 0; r < NP; ++r) m[r] = r0[r] - r1[r];
        jump = dotn<NP>(Vb, m);
        gather1(Do, r0);
        gather1(Dn, r1);
        go[1] = dotn<NP>(Vb, r0);
        gn[1] = dotn<NP>(Vb, r1);
        gather1(No, r0);
        gather1(Nn, r1);
        go[0] = dotn<NP>(Vb, r0);
        gn[0] = dotn<NP>(Vb, r1);
      }
      // geometry
      T t1[3], t2[3], jn[3], w[3];
#pragma unroll
      for(int a = 0; a < 3; ++a)
      {
        T a1 = A[b1][a], a2 = A[b2][a], a12 = A[b12][a];
        if(side)
        {
          a1 = FT ? F_[cs][d][0][a] : a1 + A[bd | b1][a];
          a2 = FT ? F_[cs][d][1][a] : a2 + A[bd | b2][a];
          a12 = FT ? F_[cs][d][2][a] : a12 + A[7][a];
        }
        t1[a] = a1 + p1 * a12;
        t2[a] = a2 + p0 * a12;
        jn[a] = N_[cs][f][0][a] + p0 * N_[cs][f][1][a] + p1 * (N_[cs][f][2][a] + p0 * N_[cs][f][3][a]);
      }
#pragma unroll
      for(int a = 0; a < 3; ++a)
      {
        const int k = (a + 1) % 3, l = (a + 2) % 3;
        w[a] = t1[k] * t2[l] - t1[l] * t2[k];
      }
      T ww = 0, wo = 0, wn = 0, g11 = 0, g12 = 0, g22 = 0, o1 = 0, o2 = 0, n1 = 0, n2 = 0;
#pragma unroll
      for(int a = 0; a < 3; ++a)
      {
        ww += w[a] * w[a];
        wo += w[a] * jd[a];
        wn += w[a] * jn[a];
        g11 += t1[a] * t1[a];
        g12 += t1[a] * t2[a];
        g22 += t2[a] * t2[a];
        o1 += t1[a] * jd[a];
        o2 += t2[a] * jd[a];
        n1 += t1[a] * jn[a];
        n2 += t2[a] * jn[a];
      }
      // outward: the normal derivative grows along J_d on side 1, against it on side 0
      const T sg = (wo > T(0)) == (side == 1) ? T(1) : T(-1);
      const T io = sg * fast_recip(wo), in_ = sg * fast_recip(wn);
      const T nw = root(ww);
      const T ko[3] = {io * ww, io * (g12 * o2 - g22 * o1), io * (g12 * o1 - g11 * o2)};
      const T kn[3] = {in_ * ww, in_ * (g12 * n2 - g22 * n1), in_ * (g12 * n1 - g11 * n2)};
      // penalty: inverse lengths |(J^{-1} n)_d| at the first face point of both cells
      // (apps/laplace_integrator.h:651-656, 692-693)
      T sigma = nw * (in ? T(0.5) * (fabs(io) + fabs(in_)) : T(2) * fabs(io));
      sigma = ipg * lane_read(sigma, lane0);
      const T hf = (in ? T(0.5) : T(1)) * wq;
      const T pa = sigma * (nw * wq) * jump - hf * (ko[0] * go[0] + ko[1] * go[1] + ko[2] * go[2] +
                                                    kn[0] * gn[0] + kn[1] * gn[1] + kn[2] * gn[2]);
      const T hj = -hf * jump;
      // projections on the tangential test functions
      if constexpr(LATE) fetch_t();
      T ra_[NP], rb[NP], rc[NP];
      gather1(pa, ra_);
      gather1(hj * ko[2], rb);
      const T sa = dotn<NP>(VbT, ra_) + dotn<NP>(DbT, rb);
      gather1(hj * ko[1], rb);
      gather1(hj * ko[0], rc);
      const T sb = dotn<NP>(VbT, rb), sc = dotn<NP>(VbT, rc);
      gather0(sa, ra_);
      gather0(sb, rb);
      gather0(sc, rc);
      const T pv = dotn<NP>(VaT, ra_) + dotn<NP>(DaT, rb), pd = dotn<NP>(VaT, rc);
#pragma unroll
      for(int j = 0; j < NP; ++j) acc[d][j] += tab.fd[side][j] * pd;
      acc[d][side ? P : 0] += pv;
    }
  }
#pragma unroll
  for(int j = 0; j < NP; ++j)
  {
    if(SPLIT && part == 1) L0[cs][at[0] + j] = acc[0][j];
    if(!SPLIT || part == 2) L1[cs][at[1] + j * st[1]] = acc[1][j];
    if(!SPLIT || part == 3) L2[cs][at[2] + j * st[2]] = acc[2][j];
  }
  __syncthreads();
  if(!act || part != 0) return;
  T out[NP];
#pragma unroll
  for(int j = 0; j < NP; ++j)
  {
    out[j] = acc[0][j] + L1[cs][NP * q + j] + L2[cs][NP * q + j];
    if(SPLIT) out[j] += L0[cs][NP * q + j];
  }
  if(RESIDUAL)
  {
    T bv[NP];
    load_row<NP>(b + cell * NDC + NP * q, bv);
#pragma unroll
    for(int j = 0; j < NP; ++j) out[j] = bv[j] - out[j];
  }
  store_row<NP>(y + cell * NDC + NP * q, out);
}

// the 2D form: a cell is NP lanes, 64 / NP cells per block; SPLIT: five waves per block of
// cells, one for the cell term and one per face
template<int NP, typename VT, bool RESIDUAL, bool SPLIT>
__global__ void __launch_bounds__(SPLIT ? 320 : 64, (SPLIT ? 1 : 2))
k_sipg_moved_2d(const VT *__restrict__ x, VT *__restrict__ y, const VT *__restrict__ b,
                const double *__restrict__ vert, const GeneralTab<NP, VT> tab, const int n,
                const VT ipg, const uint32_t *__restrict__ cells, const int64_t count)
{
  using T = VT;
  constexpr int NDC = NP * NP, CPB = moved_cells_per_block<2, NP>(), P = NP - 1;
  constexpr int CSL = (64 + NP - 1) / NP;  // cell slots, idle lanes included
  __shared__ double X[CSL][12][2];         // corners; far corners of the face neighbours
  __shared__ T A_[CSL][4][2];              // map coefficients
  constexpr bool FT = face_tangents_staged<T>();
  __shared__ T F_[FT ? CSL : 1][2][2];     // tangents of the faces x_d = 1
  __shared__ T N_[CSL][4][2][2];           // normal columns of the neighbours' maps on the faces
  __shared__ __align__(16) T L1[SPLIT ? 4 : 1][CSL][NDC];  // contributions of the y-faces (SPLIT: of each face)
  constexpr bool ROWS = moved_row_gathers<NP, SPLIT>();
  using GR = GatherRows<CSL, T>;
  __shared__ __align__(16) T G[ROWS ? 5 * GR::SIZE : 1];

  const int part = SPLIT ? __builtin_amdgcn_readfirstlane(int(threadIdx.x)) / 64 : 0;
  const int t = threadIdx.x % 64, cs = t / NP, q = t % NP;
  const int64_t per = int64_t(gridDim.x) / 8;  // the grid is a multiple of eight blocks
  const int64_t slot = (int64_t(blockIdx.x % 8) * per + blockIdx.x / 8) * CPB + cs;
  const bool act = cs < CPB && slot < count;
  const int64_t sl = act ? slot : 0;
  const int64_t cell = cells ? int64_t(cells[sl]) : sl;
  const int cc[2] = {int(cell) % n, int(cell) / n};
  int ra[NP];  // ds_bpermute addresses of the rotations (NP != 4)
#pragma unroll
  for(int r = 0; r < NP; ++r) ra[r] = 4 * (cs * NP + (q + r) % NP);
  auto gather = [&](T v, T *o) {
    if constexpr(ROWS)
      GR::gather(G + part * GR::SIZE, cs, q, v, o);
    else
      lane_gather<NP, 0>(v, ra, o);
  };

  {
    // vertex c < 4: corner c; else the corner of the neighbour across face
    // f = (c - 4) / 2 opposite face corner (c - 4) % 2 (absent neighbour: any vertex)
    const int vb = cc[0] + (n + 1) * cc[1];
    for(int c = q + NP * part; c < 12; c += SPLIT ? 5 * NP : NP)
    {
      const int f = (c - 4) >> 1, d = f >> 1, side = f & 1;
      int o0 = c & 1, o1 = c >> 1;
      if(c >= 4)
      {
        const int far = side ? 2 : -1;
        o0 = d == 0 ? far : (c & 1);
        o1 = d == 1 ? far : (c & 1);
        const int cd = d == 0 ? cc[0] : cc[1];
        if(side ? cd == n - 1 : cd == 0) o0 = o1 = 0;
      }
      const double *pv = vert + int64_t(vb + o0 + (n + 1) * o1) * 2;
      X[cs][c][0] = pv[0];
      X[cs][c][1] = pv[1];
    }
  }
  const T *xc = x + cell * NDC;
  T u[NP], vo[2][2], go_[2][2], vn[2][2], gn_[2][2];
#pragma unroll
  for(int d = 0; d < 2; ++d)
  {
    if(SPLIT && (part + 1) / 2 != d + 1 && !(d == 0 && part == 0)) continue;
    const int at = d == 0 ? NP * q : q, st = d == 0 ? 1 : NP;
    T ol[NP];
#pragma unroll
    for(int j = 0; j < NP; ++j) ol[j] = xc[at + j * st];
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      if(SPLIT && part != 1 + 2 * d + side) continue;
      const bool in = side ? cc[d] < n - 1 : cc[d] > 0;
      const int64_t shift = (d == 0 ? int64_t(1) : int64_t(n)) * NDC;
      const T *pn = xc + at + (in ? (side ? shift : -shift) : 0);
      T dd = 0, dn = 0, nl[NP];
#pragma unroll
      for(int j = 0; j < NP; ++j)
      {
        nl[j] = pn[j * st];
        dd += tab.fd[side][j] * ol[j];
        dn += tab.fd[1 - side][j] * nl[j];
      }
      vo[d][side] = ol[side ? P : 0];
      go_[d][side] = dd;
      vn[d][side] = in ? nl[side ? 0 : P] : T(0);
      gn_[d][side] = in ? dn : T(0);
    }
    if(d == 0)
#pragma unroll
      for(int j = 0; j < NP; ++j) u[j] = ol[j];
  }
  // the lanes' rows of the tables (kernel arguments, read by lane)
  const T *tk = reinterpret_cast<const T *>(&tab);
  T Va[NP], Da[NP], VaT[NP], DaT[NP];
#pragma unroll
  for(int r = 0; r < NP; ++r)
  {
    const int at = 2 * NDC + 4 * NP + q * NP + r;
    Va[r] = tk[at];
    Da[r] = tk[at + NDC];
    VaT[r] = tk[at + 2 * NDC];
    DaT[r] = tk[at + 3 * NDC];
  }
  const T p0 = tk[2 * NDC + q], wq = tk[2 * NDC + NP + q];
  __syncthreads();
  // map coefficients, formed in FP64: item (coordinate a) of the cell, then of the
  // four neighbours' normal columns
  for(int it = q + NP * part; it < 10; it += SPLIT ? 5 * NP : NP)
  {
    const int a = it & 1, f = (it >> 1) - 1;
    if(f < 0)
    {
      const double c0 = X[cs][0][a], c1 = X[cs][1][a], c2 = X[cs][2][a], c3 = X[cs][3][a];
      A_[cs][1][a] = T(c1 - c0);
      A_[cs][2][a] = T(c2 - c0);
      A_[cs][3][a] = T(c3 - c2 - (c1 - c0));
      continue;
    }
    const int d = f >> 1, side = f & 1, m1 = d == 0 ? 2 : 1;
    const int cd = d == 0 ? cc[0] : cc[1];
    const bool in = side ? cd < n - 1 : cd > 0;
    double e[2], c[2];
#pragma unroll
    for(int cp = 0; cp < 2; ++cp)
    {
      const int cy = (side << d) | (cp ? m1 : 0);
      // absent neighbour: the cell's own edge (finite; its products are multiplied by 0)
      const double far = in ? X[cs][4 + 2 * f + cp][a] : X[cs][cy ^ (1 << d)][a];
      c[cp] = X[cs][cy][a];
      const double ed = far - c[cp];
      e[cp] = (side == 1) == in ? ed : -ed;
    }
    N_[cs][f][0][a] = T(e[0]);
    N_[cs][f][1][a] = T(e[1] - e[0]);
    if(FT && side == 1) F_[cs][d][a] = T(c[1] - c[0]);
  }
  __syncthreads();
  T A[4][2];
#pragma unroll
  for(int S = 1; S < 4; ++S)
#pragma unroll
    for(int a = 0; a < 2; ++a) A[S][a] = A_[cs][S][a];

  T acc[2][NP];
#pragma unroll
  for(int j = 0; j < NP; ++j) acc[0][j] = acc[1][j] = 0;
  // ---------------- cell term
  if(!SPLIT || part == 0)
  {
    const T c0[2] = {A[1][0] + p0 * A[3][0], A[1][1] + p0 * A[3][1]};
#pragma unroll
    for(int i = 0; i < NP; ++i)
    {
      T v = 0, g = 0, r0[NP], r1[NP];
#pragma unroll
      for(int j = 0; j < NP; ++j)
      {
        v += tab.V[i * NP + j] * u[j];
        g += tab.Dv[i * NP + j] * u[j];
      }
      gather(g, r0);
      gather(v, r1);
      const T g0 = dotn<NP>(Va, r0), g1 = dotn<NP>(Da, r1);
      const T c1[2] = {A[2][0] + tab.qx[i] * A[3][0], A[2][1] + tab.qx[i] * A[3][1]};
      const T det = c0[0] * c1[1] - c0[1] * c1[0];
      const T w = wq * tab.qw[i] * fast_recip(fabs(det));
      const T h0 = w * (c1[1] * g0 - c0[1] * g1), h1 = w * (c0[0] * g1 - c1[0] * g0);
      gather(c1[1] * h0 - c1[0] * h1, r0);
      gather(c0[0] * h1 - c0[1] * h0, r1);
      const T a0 = dotn<NP>(VaT, r0), a1 = dotn<NP>(DaT, r1);
#pragma unroll
      for(int j = 0; j < NP; ++j) acc[0][j] += tab.Dv[i * NP + j] * a0 + tab.V[i * NP + j] * a1;
    }
  }
  // ---------------- faces
  const int lane0 = min(cs, CPB - 1) * NP;  // the lane of the cell's first face point
#pragma unroll
  for(int d = 0; d < 2; ++d)
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      if(SPLIT && part != 1 + 2 * d + side) continue;
      const int f = 2 * d + side, bd = 1 << d, b1 = 2 >> d;
      const bool in = side ? cc[d] < n - 1 : cc[d] > 0;
      T r0[NP], r1[NP], m[NP], go[2], gn[2];
      gather(vo[d][side], r0);
      gather(vn[d][side], r1);
#pragma unroll
      for(int r = 0; r < NP; ++r) m[r] = r0[r] - r1[r];
      const T jump = dotn<NP>(Va, m);
      go[1] = dotn<NP>(Da, r0);
      gn[1] = dotn<NP>(Da, r1);
      gather(go_[d][side], r0);
      gather(gn_[d][side], r1);
      go[0] = dotn<NP>(Va, r0);
      gn[0] = dotn<NP>(Va, r1);
      T t1[2], jd[2], jn[2];
#pragma unroll
      for(int a = 0; a < 2; ++a)
      {
        t1[a] = !side ? A[b1][a] : FT ? F_[cs][d][a] : A[b1][a] + A[3][a];
        jd[a] = A[bd][a] + p0 * A[3][a];
        jn[a] = N_[cs][f][0][a] + p0 * N_[cs][f][1][a];
      }
      const T ww = t1[0] * t1[0] + t1[1] * t1[1];
      const T wo = t1[1] * jd[0] - t1[0] * jd[1], wn = t1[1] * jn[0] - t1[0] * jn[1];
      // outward: the normal derivative grows along J_d on side 1, against it on side 0
      const T sg = (wo > T(0)) == (side == 1) ? T(1) : T(-1);
      const T io = sg * fast_recip(wo), in_ = sg * fast_recip(wn);
      const T nw = root(ww);
      const T ko[2] = {io * ww, -io * (t1[0] * jd[0] + t1[1] * jd[1])};
      const T kn[2] = {in_ * ww, -in_ * (t1[0] * jn[0] + t1[1] * jn[1])};
      // penalty: inverse lengths |(J^{-1} n)_d| at the first face point of both cells
      // (apps/laplace_integrator.h:651-656, 692-693)
      T sigma = nw * (in ? T(0.5) * (fabs(io) + fabs(in_)) : T(2) * fabs(io));
      sigma = ipg * lane_read(sigma, lane0);
      const T hf = (in ? T(0.5) : T(1)) * wq;
      const T pa = sigma * (nw * wq) * jump -
                   hf * (ko[0] * go[0] + ko[1] * go[1] + kn[0] * gn[0] + kn[1] * gn[1]);
      const T hj = -hf * jump;
      gather(pa, r0);
      gather(hj * ko[1], r1);
      const T pv = dotn<NP>(VaT, r0) + dotn<NP>(DaT, r1);
      gather(hj * ko[0], r0);
      const T pd = dotn<NP>(VaT, r0);
#pragma unroll
      for(int j = 0; j < NP; ++j) acc[d][j] += tab.fd[side][j] * pd;
      acc[d][side ? P : 0] += pv;
    }
#pragma unroll
  for(int j = 0; j < NP; ++j)
  {
    if(SPLIT && (part == 1 || part == 2)) L1[part - 1][cs][NP * q + j] = acc[0][j];
    if(!SPLIT || part > 2) L1[SPLIT ? part - 1 : 0][cs][q + j * NP] = acc[1][j];
  }
  __syncthreads();
  if(!act || part != 0) return;
  T out[NP];
#pragma unroll
  for(int j = 0; j < NP; ++j)
  {
    out[j] = acc[0][j] + L1[0][cs][NP * q + j];
    if constexpr(SPLIT) out[j] += L1[1][cs][NP * q + j] + L1[2][cs][NP * q + j] + L1[3][cs][NP * q + j];
  }
  if(RESIDUAL)
  {
    T bv[NP];
    load_row<NP>(b + cell * NDC + NP * q, bv);
#pragma unroll
    for(int j = 0; j < NP; ++j) out[j] = bv[j] - out[j];
  }
  store_row<NP>(y + cell * NDC + NP * q, out);
}

}  // namespace tpss
