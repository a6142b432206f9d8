// kernels_elasticity.hpp -- SIPG linear elasticity operator on Cartesian meshes,
// the operator of the reference's LinElasticity model problem
// (LinElasticity::MW::MatrixIntegrator, apps/linelasticity_integrator.h:31-124,
// which calls deal.II's LocalIntegrators::Elasticity and ::GradDiv):
//   cell      2 mu eps(u):eps(v) + lambda div u div v
//   interior  2 mu (sigma [u].[v] - {eps(u) n}.[v] - {eps(v) n}.[u])
//             + lambda (sigma [u.n][v.n] - {div u}[v.n] - {div v}[u.n])
//   boundary  the same with the mirrored exterior state u_out = -u_in,
//             grad u_out = grad u_in (penalty 2 sigma, Dirichlet u = 0)
// sigma = ip * gamma / h, gamma = p (p + 1).
//
// Vectors are component-blocked: x[c * Ns + cell * NDC + local]; arithmetic in the
// vector type.  On uniform cells QGauss(p+1) integrates every term exactly, so the
// form is evaluated as a sum of Kronecker products of 1D matrices, element-centrically
// (every output entry is written by exactly one lane).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "kernels.hpp"

namespace tpss
{
// Per direction d, with K = 1/2 (G - G^T), G = int phi_i phi_j',
// B = diag(-1, 0, .., 0, 1), M the mass and L_a the SIPG line matrix of a cell
// (stiffness and its half of the consistency terms, without penalty) for the
// stiffness factor a (2 mu + lambda along the component, mu across; penalty factors
// pi = 2 mu + lambda and 2 mu):
//   own cell    y_c += sum_d L_d M M u_c,   y_a += -(mu + lambda) M (K_a K_c + 1/4 B_a B_c) u_c
//   face (d, side) with the neighbour's trace (v, v'), s = +1 (left) or -1:
//     y_c += (e_i P + (-s/2 a g_i) v) M M,  P = pi sigma (u - v) + s/2 a v'
//     y_d += e_i s M H1 u_c,  H1 = h1K K + h1B B   (tangential direction c)
//     y_a += e_i s M H2 u_d,  H2 = h2K K + h2B B   (tangential direction a)
// (e_i: 1 at the node on the face; g_i = phi_i' there; the penalty acts on the jump
// u - v, whose cancellation in FP32 a penalty inside L_a would lose).  A boundary face takes the
// odd reflection of the cell as its neighbour (v = -u, v' = u'); only the
// average of the mixed terms is even there, which flips one sign in the h's.  The
// trace of a neighbour is its node value on the face (Gauss-Lobatto nodes) and one
// NP-term product for the derivative.  (3D written out; 2D has no third mass factor.)
template<int NP, typename T>
struct ElastTab
{
  T M[NP * NP], K[NP * NP];
  T LA[NP * NP], LB[NP * NP];  // L along the component / across it
  T g[2][NP];                  // phi_i'(0) / h, phi_i'(1) / h
  T aA, aB;                    // 1/2 stiffness factor along / across
  T pA, pB;                    // penalty factor times sigma
  T h1K[2], h1B[2], h2K[2], h2B[2];  // [0] interior face, [1] boundary face
  T kappa;                     // -(mu + lambda)
};

template<int DIM, int NP>
constexpr int elasticity_cells_per_block()
{
  return 64 / cpow(NP, DIM - 1);
}

// Waves per SIMD the register allocation must allow (64^3 Q2: FP32 129 us unbounded,
// 106 us with 3; FP64 290 us unbounded, 231 us with 2; in FP64 the 31 KB of LDS per block hold
// it at 1.25).  Three would spill Q3 FP32 (24^3 15.1 us unbounded, 15.8 us with 3).  Q3 FP64
// spills with 2 (3D 30 registers, 2D 16) and gains from it as soon as the launch fills the
// GPU: with 2 against 1, 3D 44^3 199 / 210 us, 24^3 41.3 / 43.4, 16^3 15.4 / 13.7; 2D 500^2
// 47.3 / 52.8, 100^2 6.1 / 5.3.  Q4 FP64 keeps one.
template<int NP, typename T>
constexpr int elasticity_min_waves()
{
  return std::is_same<T, float>::value ? (NP <= 3 ? 3 : 2) : (NP <= 4 ? 2 : 1);
}

// One lane per x-line (ly, lz) of a cell, 64 / NP^(DIM-1) cells per single-wave block
// (its barriers cost nothing).  A lane holds its line of all components; the x
// products run in registers.  The y products read the cell's lines from LDS, each
// extended by the x-face traces of its lane (v, P on both sides), so that the x
// faces need no exchange of their own; in 3D nine mixed rows per lane pass through
// LDS for the z products.  The y- and z-face traces are formed by lanes that own a
// tangential point (lines of the neighbour along the face normal), the z-face ones
// contracted along y before the lanes of the lines read them as rows.
// Blocks of one eighth of the launch run on one XCD, so that neighbours in y and z
// are mostly found in its L2 (64^3 Q2 FP64 309 -> 290 us).
// Bound by instruction issue and LDS together: 64^3 Q2 (21.2M DoFs, 170 MB in FP32)
// FP32 106 us, FP64 231 us per apply; the quadrature form of the same operator
// (tensor interpolation to Gauss points, fluxes per face point) took 618 / 1278 us.
template<int DIM, int NP, typename VT, bool RESIDUAL>
__global__ void __launch_bounds__(64, (elasticity_min_waves<NP, VT>()))
k_elasticity(const VT *__restrict__ x, VT *__restrict__ y, const VT *__restrict__ b,
             const ElastTab<NP, VT> tab, const int n, const int64_t Ns,
             const uint32_t *__restrict__ cells, const int64_t count)
{
  using T = VT;
  constexpr bool D3 = DIM == 3;
  constexpr int NL = cpow(NP, DIM - 1), NDC = NL * NP, P = NP - 1;
  constexpr int CPB = elasticity_cells_per_block<DIM, NP>();
  constexpr int NX = NP + 4;  // extended line: values, then v, P of the left and right x-face
  using Ext = LaneRows<NX, 64, T>;
  using Row = LaneRows<NP, 64, T>;
  // face rows: entry lx of row (cell slot, tangential line); slots for idle lanes too
  constexpr int FL = D3 ? NP : 1, FR = ((64 + NL - 1) / NL) * FL, NF = 4 * DIM;
  using Face = LaneRows<NP, FR, T>;
  constexpr int CW = Face::CW;
  constexpr int S1 = DIM * Ext::SIZE + NF * Face::SIZE, S2 = D3 ? 9 * Row::SIZE : 0;
  __shared__ __align__(16) T buf[S1 > S2 ? S1 : S2];  // y stage; then the z stage's rows
  __shared__ __align__(16) T fz[D3 ? NF * Face::SIZE : 1];     // z-face traces, then contracted along y
  constexpr int NTAB = int(sizeof(ElastTab<NP, T>) / sizeof(T));
  __shared__ T tl[NTAB];
  T *ext = buf, *fy = buf + DIM * Ext::SIZE;
  // entry e of the line of lane l, component c
  auto eidx = [](int c, int l, int e) { return c * Ext::SIZE + ((e / CW) * 64 + l) * CW + e % CW; };
  // entry e of face row r in plane k; planes of the values v and of P
  auto pv = [](int side, int c) { return side * 2 * DIM + c; };
  auto pp = [](int side, int c) { return side * 2 * DIM + DIM + c; };
  auto fidx = [](int k, int r, int e) { return k * Face::SIZE + ((e / CW) * FR + r) * CW + e % CW; };

  const int t = threadIdx.x, cs = t / NL, q = t % NL;
  const int cr = min(cs, CPB - 1);  // lanes beyond the last cell read its lines
  const int q0 = q % NP, q1 = q / NP;  // (ly, lz) of the line; (lx, lz) / (lx, ly) of a face point
  const int64_t nblk = gridDim.x, per = nblk / 8;  // the grid is a multiple of eight blocks
  const int64_t blk = int64_t(blockIdx.x % 8) * per + blockIdx.x / 8;
  const int64_t slot = blk * CPB + cs;
  const bool act = cs < CPB && slot < count;
  const int64_t sl = act ? slot : 0;
  const int64_t cell = cells ? int64_t(cells[sl]) : sl;
  const int ci = int(cell);
  const int cx = ci % n, cy = (ci / n) % n, cz = D3 ? ci / (n * n) : 0;
  const bool has[3][2] = {{cx > 0, cx < n - 1}, {cy > 0, cy < n - 1}, {cz > 0, cz < n - 1}};
  const int64_t nn = int64_t(n) * n;
  const T *xc = x + cell * NDC;

  for(int i = t; i < NTAB; i += 64) tl[i] = reinterpret_cast<const T *>(&tab)[i];
  // ---- loads: the lane's lines, the x-neighbours' lines and the neighbours' lines
  // along y and z at the lane's tangential point
  T u[DIM][NP], nx[2][DIM][NP], fl[DIM - 1][2][DIM][NP];
#pragma unroll
  for(int c = 0; c < DIM; ++c)
  {
    load_row<NP>(xc + c * Ns + NP * q, u[c]);
    load_row<NP>(xc + c * Ns + NP * q + (has[0][0] ? -NDC : 0), nx[0][c]);
    load_row<NP>(xc + c * Ns + NP * q + (has[0][1] ? NDC : 0), nx[1][c]);
  }
#pragma unroll
  for(int d = 1; d < DIM; ++d)
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      const bool in = has[d][side];
      const int st = d == 1 ? NP : NP * NP;
      const int64_t shift = (d == 1 ? int64_t(n) : nn) * NDC;
      const int at = d == 1 ? q0 + NP * NP * q1 : q0 + NP * q1;
      // absent neighbour: the cell's own line, reversed
      const T *src = xc + (in ? (side ? shift : -shift) : 0) + at + (in ? 0 : P * st);
      const int sst = in ? st : -st;
#pragma unroll
      for(int c = 0; c < DIM; ++c)
#pragma unroll
        for(int j = 0; j < NP; ++j) fl[d - 1][side][c][j] = src[c * Ns + j * sst];
    }

  // trace (v, P) of a neighbour line r on this cell's face `side`; sg: -1 for the
  // reflection; w: the cell's own value there
  auto trace = [&](const T *r, int side, bool along, T sg, T w, T &v, T &jp) {
    T d = 0;
#pragma unroll
    for(int j = 0; j < NP; ++j) d += tab.g[1 - side][j] * r[j];
    v = sg * (side ? r[0] : r[P]);
    const T a = along ? tab.aA : tab.aB, pn = along ? tab.pA : tab.pB;
    jp = (side ? -a : a) * (sg * d) + pn * (w - v);
  };
  T vx[2][DIM];  // x-face values of this lane's line
  {
    T e[DIM][NX];
#pragma unroll
    for(int c = 0; c < DIM; ++c)
    {
#pragma unroll
      for(int i = 0; i < NP; ++i) e[c][i] = u[c][i];
#pragma unroll
      for(int side = 0; side < 2; ++side)
      {
        T r[NP];
#pragma unroll
        for(int j = 0; j < NP; ++j) r[j] = has[0][side] ? nx[side][c][j] : -u[c][P - j];
        trace(r, side, c == 0, T(1), u[c][side ? P : 0], vx[side][c], e[c][NP + 2 * side + 1]);
        e[c][NP + 2 * side] = vx[side][c];
      }
      Ext::put(ext + c * Ext::SIZE, t, e[c]);
    }
  }
  __syncthreads();  // the lines are staged
#pragma unroll
  for(int side = 0; side < 2; ++side)
#pragma unroll
    for(int c = 0; c < DIM; ++c)
    {
      T v, jp;
      const int r = cs * FL + q1, e = side ? P : 0;
      trace(fl[0][side][c], side, c == 1, has[1][side] ? T(1) : T(-1),
            ext[eidx(c, cr * NL + e + NP * q1, q0)], v, jp);
      fy[fidx(pv(side, c), r, q0)] = v;
      fy[fidx(pp(side, c), r, q0)] = jp;
      if constexpr(D3)
      {
        trace(fl[DIM - 2][side][c], side, c == 2, has[2][side] ? T(1) : T(-1),
              ext[eidx(c, cr * NL + q1 + NP * e, q0)], v, jp);
        fz[fidx(pv(side, c), r, q0)] = v;
        fz[fidx(pp(side, c), r, q0)] = jp;
      }
    }
  __syncthreads();

  // lane-indexed rows of the 1D tables
  const T *tM = tl, *tK = tl + NP * NP, *tLA = tl + 2 * NP * NP, *tLB = tl + 3 * NP * NP;
  const T *tg = tl + 4 * NP * NP;
  const T b0 = q0 == 0 ? T(-1) : q0 == P ? T(1) : T(0);
  const T b1 = q1 == 0 ? T(-1) : q1 == P ? T(1) : T(0);
  const T kappa = tab.kappa, kq = T(0.25) * tab.kappa;
  T M1[NP], K1[NP];  // rows of index q1
  // ---- z-face traces contracted along y by the lanes (lx, ly) = (q0, q1):
  // M v, M P with the tangential mixed terms along y added to P
  T zt[2][2 * DIM];
  if constexpr(D3)
  {
#pragma unroll
    for(int j = 0; j < NP; ++j)
    {
      M1[j] = tM[q1 * NP + j];
      K1[j] = tK[q1 * NP + j];
    }
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      T kv[3];
#pragma unroll
      for(int k = 0; k < 2 * DIM; ++k)
      {
        T m = 0, kk = 0;
#pragma unroll
        for(int j = 0; j < NP; ++j)
        {
          const T w = fz[fidx(side * 2 * DIM + k, cs * NP + j, q0)];
          m += M1[j] * w;
          if(k == 1 || k == 2) kk += K1[j] * w;
        }
        zt[side][k] = m;
        if(k == 1 || k == 2)
        {
          const T w = fz[fidx(pv(side, k), cs * NP + q1, q0)];
          const int bf = has[2][side] ? 0 : 1;
          const T hK = k == 1 ? tab.h1K[bf] : tab.h2K[bf], hB = k == 1 ? tab.h1B[bf] : tab.h2B[bf];
          kv[k] = (side ? T(-1) : T(1)) * (hK * kk + hB * b1 * w);
        }
      }
      zt[side][DIM + 1] += kv[2];  // component 1: H2 along y of u_2
      zt[side][DIM + DIM - 1] += kv[1];  // component 2: H1 along y of u_1
    }
  }

  // ---- y stage: M, L and K along y of the extended lines, with the y faces
  T My[DIM][NX], Ly[DIM][NP], Ky[DIM][NP], KyV[DIM][2], Q[DIM][NP];
  {
    T M0[NP], K0[NP], LA0[NP], LB0[NP];
#pragma unroll
    for(int j = 0; j < NP; ++j)
    {
      M0[j] = tM[q0 * NP + j];
      K0[j] = tK[q0 * NP + j];
      LA0[j] = tLA[q0 * NP + j];
      LB0[j] = tLB[q0 * NP + j];
    }
    T gs[2], es[2];
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      gs[side] = (side ? T(1) : T(-1)) * tg[side * NP + q0];
      es[side] = q0 == (side ? P : 0) ? T(1) : T(0);
    }
#pragma unroll
    for(int c = 0; c < DIM; ++c)
    {
#pragma unroll
      for(int i = 0; i < NX; ++i) My[c][i] = 0;
#pragma unroll
      for(int i = 0; i < NP; ++i) Ly[c][i] = Ky[c][i] = 0;
      KyV[c][0] = KyV[c][1] = 0;
#pragma unroll
      for(int j = 0; j < NP; ++j)
      {
        T r[NX];
        Ext::get(ext + c * Ext::SIZE, cr * NL + j + NP * q1, r);
        const T l = c == 1 ? LA0[j] : LB0[j];
#pragma unroll
        for(int i = 0; i < NX; ++i) My[c][i] += M0[j] * r[i];
#pragma unroll
        for(int i = 0; i < NP; ++i)
        {
          Ly[c][i] += l * r[i];
          Ky[c][i] += K0[j] * r[i];
        }
        KyV[c][0] += K0[j] * r[NP];
        KyV[c][1] += K0[j] * r[NP + 2];
      }
#pragma unroll
      for(int i = 0; i < NP; ++i)
      {
        Ky[c][i] *= kappa;
        Q[c][i] = kq * b0 * u[c][i];
      }
      const T a = c == 1 ? tab.aA : tab.aB;
#pragma unroll
      for(int side = 0; side < 2; ++side)
      {
        T v[NP], jp[NP];
        Face::get(fy + pv(side, c) * Face::SIZE, cs * FL + q1, v);
        Face::get(fy + pp(side, c) * Face::SIZE, cs * FL + q1, jp);
        const int bf = has[1][side] ? 0 : 1;
        const T sg = side ? -es[side] : es[side];
        const T hK = sg * (c == 1 ? tab.h2K[bf] : tab.h1K[bf]);
        const T hB = sg * (c == 1 ? tab.h2B[bf] : tab.h1B[bf]);
        const T cv = a * gs[side];
#pragma unroll
        for(int i = 0; i < NP; ++i)
        {
          Ly[c][i] += cv * v[i] + es[side] * jp[i];
          Ky[c][i] += hK * v[i];
          Q[c][i] += hB * v[i];
        }
      }
    }
  }
  __syncthreads();  // the lines, the y-face rows and the z-face traces are read

  if constexpr(D3)
#pragma unroll
    for(int side = 0; side < 2; ++side)
#pragma unroll
      for(int k = 0; k < 2 * DIM; ++k) fz[fidx(side * 2 * DIM + k, cs * NP + q1, q0)] = zt[side][k];

  // ---- x products in registers
  auto xprod = [&](const T *A, const T *r, T *o, T f) {
#pragma unroll
    for(int i = 0; i < NP; ++i)
    {
      T s = 0;
#pragma unroll
      for(int j = 0; j < NP; ++j) s += A[i * NP + j] * r[j];
      o[i] += f * s;
    }
  };
  auto clear = [&](T *o) {
#pragma unroll
    for(int i = 0; i < NP; ++i) o[i] = 0;
  };
  T I[DIM][NP];
  T *zb = buf;
#pragma unroll
  for(int c = 0; c < DIM; ++c)
  {
    T zm[NP], zl[NP], zk[NP];
    // L along x with the x faces; M along x of the y-line products
    const T a = c == 0 ? tab.aA : tab.aB;
#pragma unroll
    for(int i = 0; i < NP; ++i)
      zm[i] = -a * tab.g[0][i] * My[c][NP] + a * tab.g[1][i] * My[c][NP + 2];
    zm[0] += My[c][NP + 1];
    zm[P] += My[c][NP + 3];
    xprod(c == 0 ? tab.LA : tab.LB, My[c], zm, T(1));
    xprod(tab.M, Ly[c], zm, T(1));
    // the mixed terms
    if(c < 2)
    {
      const int o = 1 - c;
      xprod(tab.K, Ky[o], zm, T(1));
      zm[0] -= Q[o][0];
      zm[P] += Q[o][P];
    }
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      const int bf = has[0][side] ? 0 : 1;
      const T s = side ? T(-1) : T(1);
      if(c < 2)
        zm[side ? P : 0] += s * ((c == 0 ? tab.h1K[bf] : tab.h2K[bf]) * KyV[1 - c][side] +
                                 (c == 0 ? tab.h1B[bf] : tab.h2B[bf]) * b0 * vx[side][1 - c]);
    }
    if constexpr(D3)
    {
      clear(zl);
      xprod(tab.M, My[c], zl, T(1));
      clear(zk);
      clear(I[c]);
      if(c == 1) xprod(tab.M, Ky[DIM - 1], zk, T(1));
      if(c == 2) xprod(tab.M, Ky[1], zk, T(1));
      if(c != 1)
      {
        const int o = 2 - c;
        xprod(tab.K, My[o], zk, kappa);
#pragma unroll
        for(int side = 0; side < 2; ++side)
        {
          const int i = side ? P : 0, bf = has[0][side] ? 0 : 1;
          const T s = side ? T(-1) : T(1);
          zk[i] += s * (c == 0 ? tab.h1K[bf] : tab.h2K[bf]) * My[o][NP + 2 * side];
          I[c][i] += b1 * s *
                     ((c == 0 ? tab.h1B[bf] : tab.h2B[bf]) * My[o][NP + 2 * side] - kq * My[o][i]);
        }
      }
      if(c > 0) xprod(tab.M, Q[3 - c], I[c], b1);
      Row::put(zb + (3 * c + 0) * Row::SIZE, t, zm);
      Row::put(zb + (3 * c + 1) * Row::SIZE, t, zl);
      Row::put(zb + (3 * c + 2) * Row::SIZE, t, zk);
    }
    else
#pragma unroll
      for(int i = 0; i < NP; ++i) I[c][i] = zm[i];
  }
  // ---- z stage and the z faces
  if constexpr(D3)
  {
    __syncthreads();
    T LA1[NP], LB1[NP];
#pragma unroll
    for(int j = 0; j < NP; ++j)
    {
      LA1[j] = tLA[q1 * NP + j];
      LB1[j] = tLB[q1 * NP + j];
    }
#pragma unroll
    for(int c = 0; c < DIM; ++c)
#pragma unroll
      for(int k = 0; k < NP; ++k)
      {
        T zm[NP], zl[NP], zk[NP];
        const int ln = cr * NL + q0 + NP * k;
        Row::get(zb + (3 * c + 0) * Row::SIZE, ln, zm);
        Row::get(zb + (3 * c + 1) * Row::SIZE, ln, zl);
        Row::get(zb + (3 * c + 2) * Row::SIZE, ln, zk);
        const T l = c == 2 ? LA1[k] : LB1[k];
#pragma unroll
        for(int i = 0; i < NP; ++i) I[c][i] += M1[k] * zm[i] + l * zl[i] + K1[k] * zk[i];
      }
    T tz[DIM][NP], w0[NP], w2[NP];
#pragma unroll
    for(int c = 0; c < DIM; ++c) clear(tz[c]);
    clear(w0);
    clear(w2);
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      const T gz = (side ? T(1) : T(-1)) * tg[side * NP + q1];
      const T ez = q1 == (side ? P : 0) ? T(1) : T(0);
      const int bf = has[2][side] ? 0 : 1;
      const T sg = side ? -ez : ez;
#pragma unroll
      for(int c = 0; c < DIM; ++c)
      {
        T v[NP], jp[NP];
        Face::get(fz + pv(side, c) * Face::SIZE, cs * NP + q0, v);
        Face::get(fz + pp(side, c) * Face::SIZE, cs * NP + q0, jp);
        const T cv = (c == 2 ? tab.aA : tab.aB) * gz;
#pragma unroll
        for(int i = 0; i < NP; ++i) tz[c][i] += cv * v[i] + ez * jp[i];
        if(c != 1)
        {
          // H2 along x of u_2 into component 0, H1 along x of u_0 into component 2
          const T hK = sg * (c == 2 ? tab.h2K[bf] : tab.h1K[bf]);
          const T hB = sg * (c == 2 ? tab.h2B[bf] : tab.h1B[bf]);
          T *w = c == 2 ? w0 : w2, *o = c == 2 ? I[0] : I[DIM - 1];
#pragma unroll
          for(int i = 0; i < NP; ++i) w[i] += hK * v[i];
          o[0] -= hB * v[0];
          o[P] += hB * v[P];
        }
      }
    }
    xprod(tab.K, w0, I[0], T(1));
    xprod(tab.K, w2, I[DIM - 1], T(1));
#pragma unroll
    for(int c = 0; c < DIM; ++c) xprod(tab.M, tz[c], I[c], T(1));
  }
  if(!act) return;
#pragma unroll
  for(int c = 0; c < DIM; ++c)
  {
    const int64_t at = c * Ns + cell * NDC + NP * q;
    if(RESIDUAL)
    {
      T bv[NP];
      load_row<NP>(b + at, bv);
#pragma unroll
      for(int i = 0; i < NP; ++i) I[c][i] = bv[i] - I[c][i];
    }
    store_row<NP>(y + at, I[c]);
  }
}

}  // namespace tpss
