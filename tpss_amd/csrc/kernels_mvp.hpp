// kernels_mvp.hpp -- residual-free multiplicative color pass on Cartesian meshes.
//
// For a patch j of the current color the reference computes
//   r = b - A x,  u_j = A_j^{-1} R_j r,  x += omega R_j^T u_j
// (schwarz_preconditioner.templates.h:585-662, 691-732).  On tensor-product
// cells A_j is exactly the patch block R_j A R_j^T, so with B_j the coupling of
// the patch to the cells just outside it,
//   R_j r = b_j - A_j x_j - B_j x_out   and
//   x_j <- (1 - omega) x_j + omega A_j^{-1} (b_j - B_j x_out).
// B_j x_out is the face coupling of the SIPG operator through the patch's outer
// faces: per patch cell and direction d (one outer face each) the neighbour
// term T_d(F) x_nbr of the cell operator, evaluated here in sum-factorised form
//   M_z (M_y z_0 + M_x z_1) + M_y M_x z_2,  z_d = F_d x_nbr(d) along d.
// Valid when same-color patches are not face-coupled (red-black coloring), so
// no patch of the pass reads cells another patch of the pass writes.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace tpss
{
// what a color pass may take as zero without reading it (x_zero): the cells outside
// its patches, the patches' own cells
constexpr int kOuterZero = 1, kOwnZero = 2;

typedef short tpss_bf16x4 __attribute__((__vector_size__(4 * sizeof(short))));
typedef float tpss_floatx4 __attribute__((__vector_size__(4 * sizeof(float))));

// FP32 -> BF16 bits, round to nearest even (finite inputs)
__device__ __forceinline__ short bf16_bits(float f)
{
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return short(u >> 16);
}

// Fast-diagonalization inverse of the two patches of a block (3D, K = 8) on
// the matrix cores: every 1D contraction along direction d is one
// v_mfma_f32_16x16x16_bf16 per chunk of 16 lines, with A = diag(S_a^T, S_b^T)
// (16 x 16, block diagonal over the two patches) and B the 16 contraction
// values (8 per patch) of 16 lines; products in BF16, sums in FP32.  The
// patch data (FP32) lives in B2[2][512] (x fastest); the two waves of the
// block take two chunks each.  Lane layout of the 16x16x16 MFMA (wave64):
// A: row l%16, k = 4(l/16)+0..3; B: column l%16, k = 4(l/16)+0..3;
// D: column l%16, rows 4(l/16)+0..3.
__device__ __forceinline__ int lds_index(int d, int k, int line)
{
  // K = 8: line enumerates the other two indices (first fastest)
  return d == 0 ? k + 8 * line : d == 1 ? (line & 7) + 8 * k + 64 * (line >> 3) : line + 64 * k;
}

__device__ __forceinline__ void fd_mfma_pair(float (*B2)[512], const float (*S)[3][64],
                                             const float (*lam)[3][8], const float *w2)
{
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n16 = lane & 15, q = lane >> 4;       // column (line) / k-quarter
  const int pq = q >> 1, kofs = 4 * (q & 1);      // patch of the B/D rows, first row index
  const int arow = lane & 15, pa = arow >> 3, ao = arow & 7;  // A row: patch, output index
  for(int stage = 0; stage < 6; ++stage)
  {
    const int d = stage < 3 ? stage : 5 - stage;
    const bool fwd = stage < 3;
    // A operand: S_p^T (forward) or S_p (backward) of patch pa if the k block
    // belongs to the same patch, else zero
    tpss_bf16x4 a;
#pragma unroll
    for(int e = 0; e < 4; ++e)
    {
      const int kk = kofs + e;
      float v = 0.f;
      if(pa == pq) v = fwd ? S[pa][d][kk * 8 + ao] : S[pa][d][ao * 8 + kk];
      a[e] = bf16_bits(v);
    }
#pragma unroll
    for(int cc = 0; cc < 2; ++cc)
    {
      const int line = 16 * (2 * wave + cc) + n16;
      tpss_bf16x4 b;
#pragma unroll
      for(int e = 0; e < 4; ++e) b[e] = bf16_bits(B2[pq][lds_index(d, kofs + e, line)]);
      tpss_floatx4 acc = {0.f, 0.f, 0.f, 0.f};
      acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
      if(stage == 2)
      {
        // diagonal scaling after the last forward contraction (z): line = (x, y)
        const int x0 = line & 7, y0 = line >> 3;
        const float lxy = lam[pq][0][x0] + lam[pq][1][y0];
#pragma unroll
        for(int e = 0; e < 4; ++e) acc[e] *= w2[pq] / (lxy + lam[pq][2][kofs + e]);
      }
#pragma unroll
      for(int e = 0; e < 4; ++e) B2[pq][lds_index(d, kofs + e, line)] = acc[e];
    }
    __syncthreads();
  }
}

// Color pass with BF16-MFMA patch solves (3D, K = 8; FP32 arithmetic elsewhere), two
// patches per block.
template<typename VT>
__global__ void __launch_bounds__(128)
k_patch_mvp_bf16(const VT *__restrict__ b, VT *__restrict__ x, const OpTab<float, 4> tab,
                 const uint32_t *__restrict__ vtx, const uint32_t *__restrict__ fac,
                 const float *__restrict__ S_tab, const float *__restrict__ lam_tab,
                 const float *__restrict__ omega, const float relaxation, const int patch_begin,
                 const int patch_end, const int n, const int x_zero)
{
  using CT = float;
  constexpr int DIM = 3, K = 8;
  using PS = PatchShape<DIM, K>;
  constexpr int NP = PS::NP, L = PS::L, NPD = PS::NPD, NDC = PS::NDC, PPB = PS::PPB;
  constexpr int SY = K, SZ = K * K;  // strides (y, z) of the patch buffers
  __shared__ CT buf[PPB][NPD];
  __shared__ CT A1[PPB][NPD];
  __shared__ CT A2[PPB][NPD];
  __shared__ CT Ss[PPB][DIM][K * K];
  __shared__ CT ls[PPB][DIM][K];

  const int pl = threadIdx.x / L, t = threadIdx.x % L;
  const int j0 = patch_begin + int(blockIdx.x) * PPB;
  const int j = j0 + pl;
  const bool valid = pl < PPB && j < patch_end;
  const int plc = pl < PPB ? pl : 0;
  const bool owner = pl < PPB;

  for(int idx = threadIdx.x; idx < PPB * DIM * K * K; idx += blockDim.x)
  {
    const int q = idx / (DIM * K * K), r = idx % (DIM * K * K);
    const int d = r / (K * K), e = r % (K * K);
    const int jj = j0 + q;
    Ss[q][d][e] = jj < patch_end ? S_tab[size_t(fac[size_t(jj) * DIM + d]) * K * K + e] : CT(0);
  }
  for(int idx = threadIdx.x; idx < PPB * DIM * K; idx += blockDim.x)
  {
    const int q = idx / (DIM * K), r = idx % (DIM * K);
    const int d = r / K, e = r % K;
    const int jj = j0 + q;
    ls[q][d][e] = jj < patch_end ? lam_tab[size_t(fac[size_t(jj) * DIM + d]) * K + e] : CT(1);
  }
  int v[3] = {1, 1, 1};
  if(valid) unpack_vertex(vtx[j], v);
  const CT w = valid ? (omega ? CT(omega[j]) : relaxation) : CT(0);

  const int ty = t % K, tz = t / K;
  const int ly = ty >= NP ? ty - NP : ty, lz = tz >= NP ? tz - NP : tz;
  const int by = ty >= NP ? 1 : 0, bz = tz >= NP ? 1 : 0;
  const int64_t nn = int64_t(n) * n;

  // the x-line (ty, tz) of the patch: row lyz of the cells c_lo and c_lo + 1
  const int64_t c_lo = patch_cell<DIM, NP>(v, n, 0, ty, tz);
  const int lyz = patch_local<DIM, NP>(0, ty, tz);
  CT g[K];
  if(valid)
  {
    load_row<NP>(b + c_lo * NDC + lyz, g);
    load_row<NP>(b + (c_lo + 1) * NDC + lyz, g + NP);
  }
  else
#pragma unroll
    for(int i = 0; i < K; ++i) g[i] = CT(0);

  if(!(x_zero & kOuterZero))
  {
    // z_0: x-neighbours of the two x-cells of this line
    CT z0[K], t1[K], t2[K];
#pragma unroll
    for(int i = 0; i < K; ++i)
    {
      z0[i] = 0;
      t1[i] = 0;
      t2[i] = 0;
    }
    if(valid && v[0] - 1 > 0)
    {
      CT xl[NP];
      load_row<NP>(x + (c_lo - 1) * NDC + lyz, xl);
#pragma unroll
      for(int i = 0; i < NP; ++i)
      {
        CT s = 0;
#pragma unroll
        for(int jj = 0; jj < NP; ++jj) s += tab.Fpm[i * NP + jj] * xl[jj];
        z0[i] = s;
      }
    }
    if(valid && v[0] + 1 < n)
    {
      CT xr[NP];
      load_row<NP>(x + (c_lo + 2) * NDC + lyz, xr);
#pragma unroll
      for(int i = 0; i < NP; ++i)
      {
        CT s = 0;
#pragma unroll
        for(int jj = 0; jj < NP; ++jj) s += tab.Fmp[i * NP + jj] * xr[jj];
        z0[NP + i] = s;
      }
    }
    // z_1 (y-neighbour outside the patch) then t1 = M_x z_1 per x-cell
    {
      const bool has = by == 0 ? (v[1] - 1 > 0) : (v[1] + 1 < n);
      const CT *F = by == 0 ? tab.Fpm : tab.Fmp;
      if(valid && has)
      {
        const int64_t shift = by == 0 ? -int64_t(n) : int64_t(n);
        CT z1[K];
#pragma unroll
        for(int cx = 0; cx < 2; ++cx)
        {
          // the x-y plane lz of the neighbour cell: NP rows, contiguous
          CT xn[NP * NP];
          const VT *pn = x + (c_lo + cx + shift) * NDC + NP * NP * lz;
#pragma unroll
          for(int jj = 0; jj < NP; ++jj) load_row<NP>(pn + NP * jj, xn + NP * jj);
#pragma unroll
          for(int lx = 0; lx < NP; ++lx)
          {
            CT s = 0;
#pragma unroll
            for(int jj = 0; jj < NP; ++jj) s += F[ly * NP + jj] * xn[lx + NP * jj];
            z1[cx * NP + lx] = s;
          }
        }
#pragma unroll
        for(int cx = 0; cx < 2; ++cx)
#pragma unroll
          for(int i = 0; i < NP; ++i)
          {
            CT s = 0;
#pragma unroll
            for(int jj = 0; jj < NP; ++jj) s += tab.M[i * NP + jj] * z1[cx * NP + jj];
            t1[cx * NP + i] = s;
          }
      }
    }
    {
      const bool has = bz == 0 ? (v[2] - 1 > 0) : (v[2] + 1 < n);
      const CT *F = bz == 0 ? tab.Fpm : tab.Fmp;
      if(valid && has)
      {
        const int64_t shift = bz == 0 ? -nn : nn;
        CT z2[K];
#pragma unroll
        for(int cx = 0; cx < 2; ++cx)
        {
          // the x-z plane ly of the neighbour cell: NP rows at stride NP^2
          CT xn[NP * NP];
          const VT *pn = x + (c_lo + cx + shift) * NDC + NP * ly;
#pragma unroll
          for(int kk = 0; kk < NP; ++kk) load_row<NP>(pn + NP * NP * kk, xn + NP * kk);
#pragma unroll
          for(int lx = 0; lx < NP; ++lx)
          {
            CT s = 0;
#pragma unroll
            for(int kk = 0; kk < NP; ++kk) s += F[lz * NP + kk] * xn[lx + NP * kk];
            z2[cx * NP + lx] = s;
          }
        }
#pragma unroll
        for(int cx = 0; cx < 2; ++cx)
#pragma unroll
          for(int i = 0; i < NP; ++i)
          {
            CT s = 0;
#pragma unroll
            for(int jj = 0; jj < NP; ++jj) s += tab.M[i * NP + jj] * z2[cx * NP + jj];
            t2[cx * NP + i] = s;
          }
      }
    }
    // cross-line mass contractions through LDS
    CT *Z = A1[plc];
    CT *T2 = A2[plc];
#pragma unroll
    for(int i = 0; i < K; ++i)
      if(owner)
      {
        Z[i + SY * ty + SZ * tz] = z0[i];
        T2[i + SY * ty + SZ * tz] = t2[i];
      }
    __syncthreads();
    CT a[K], bb[K];
    const int y0 = by * NP;
#pragma unroll
    for(int i = 0; i < K; ++i)
    {
      CT s = t1[i], s2 = 0;
#pragma unroll
      for(int jj = 0; jj < NP; ++jj)
      {
        s += tab.M[ly * NP + jj] * Z[i + SY * (y0 + jj) + SZ * tz];
        s2 += tab.M[ly * NP + jj] * T2[i + SY * (y0 + jj) + SZ * tz];
      }
      a[i] = s;
      bb[i] = s2;
    }
    __syncthreads();
#pragma unroll
    for(int i = 0; i < K; ++i)
      if(owner) Z[i + SY * ty + SZ * tz] = a[i];
    __syncthreads();
    const int z00 = bz * NP;
#pragma unroll
    for(int i = 0; i < K; ++i)
    {
      CT s = bb[i];
#pragma unroll
      for(int kk = 0; kk < NP; ++kk) s += tab.M[lz * NP + kk] * Z[i + SY * ty + SZ * (z00 + kk)];
      g[i] -= s;
    }
  }

  __shared__ float w2[2];
  if(t == 0 && owner) w2[pl] = w;
#pragma unroll
  for(int i = 0; i < K; ++i)
    if(owner) buf[plc][i + K * ty + K * K * tz] = g[i];
  __syncthreads();
  fd_mfma_pair(reinterpret_cast<float(*)[512]>(&buf[0][0]),
               reinterpret_cast<const float(*)[3][64]>(&Ss[0][0][0]),
               reinterpret_cast<const float(*)[3][8]>(&ls[0][0][0]), w2);
  CT o[K];
#pragma unroll
  for(int i = 0; i < K; ++i) o[i] = buf[plc][i + K * ty + K * K * tz];
  if(!valid) return;
  if(!(x_zero & kOwnZero) && w != CT(1))
  {
    CT old[K];
    load_row<NP>(x + c_lo * NDC + lyz, old);
    load_row<NP>(x + (c_lo + 1) * NDC + lyz, old + NP);
#pragma unroll
    for(int a = 0; a < K; ++a) o[a] += (CT(1) - w) * old[a];
  }
  store_row<NP>(x + c_lo * NDC + lyz, o);
  store_row<NP>(x + (c_lo + 1) * NDC + lyz, o + NP);
}

// ----------------------------------------------------------------------------
// 3D Q3 color pass (K = 8) with vector solves: one patch per single-wave block.
//
// The coupling uses the rank of the face terms: with a neighbour line's trace
// (v, v') on the face (its node value there, Gauss-Lobatto nodes, and one 4-term
// product), s = +1 on the left face of a line, -1 on the right one,
//   (B_j x_out)_i = (e_i P - s/2 g_i v) M M,  P = -sigma v + s/2 v',
// e_i = 1 at the node on the face, g_i = phi_i' there.  Lane (l1, l2, c1, c2) =
// bits (0-1, 2-3, 4, 5) holds the x-line (y, z) = (4 c1 + l1, 4 c2 + l2) of the
// patch and, of each y- (z-) face, the tangential point (x, z) ((x, y)) of the same
// indices with the neighbour's line along the normal: a cell is a DPP row and its
// mass products run across its lanes without LDS.  The y- and z-face points then
// pass through LDS once to the lanes of the x-lines, which take their M_x product in
// registers.
//
// Per color of the 64^3 level, mean of a step from a given x: 42.8 us FP64 / 26.2 us FP32
// (195 / 97.5 MB compulsory, 216 / 108 MB moved: 5.0 / 4.1 TB/s, a large copy reaches 4.85);
// FP64 is bound by HBM, FP32 by latency and issue as well.  57 / 31 us with plane-wise
// face products (F z along the normal on every node, the masses across lines through
// LDS) and all eigenvector matrices loaded at once (their scalar registers spilled).
// ----------------------------------------------------------------------------
template<int NP, typename CT>
struct MvpTab
{
  CT M[NP * NP];
  CT R[NP * NP];  // rows of M rotated to start at the diagonal: R[q*NP + r] = M(q, (q + r) mod NP)
  CT g[2][NP];    // phi_i'(0) / h, phi_i'(1) / h
  CT sigma;
};

// Waves per SIMD the register allocation must allow.  FP32 solves of FP64 vectors hold
// FP64 rows beside them and spill 6 registers with six (64^3 sweep 725 us, with five 578,
// with four 575; with FP64 solves 655).
template<typename VT, typename CT>
constexpr int mvp_q3_min_waves()
{
  if(std::is_same<CT, double>::value) return 2;
  return std::is_same<VT, float>::value ? 6 : 5;
}

template<typename VT, typename CT>
__global__ void __launch_bounds__(64, (mvp_q3_min_waves<VT, CT>()))
k_patch_mvp_q3(const VT *__restrict__ b, VT *__restrict__ x, const MvpTab<4, CT> tab,
               const uint32_t *__restrict__ vtx, const uint32_t *__restrict__ fac,
               const CT *__restrict__ S_tab, const CT *__restrict__ lam_tab,
               const uint32_t *__restrict__ eo_tab, const float *__restrict__ omega,
               const CT relaxation, const int patch_begin, const int n, const int x_zero,
               int *__restrict__ nonfinite)
{
  constexpr int K = 8, NP = 4, NDC = 64, P = 3;
  constexpr int SY = 8, SZ = 72;  // solve buffer (x, y, z) -> x + SY y + SZ z (bank conflicts)
  __shared__ __align__(16) CT B[K * SZ];  // solve; before it the face points [dir][side][v, P][64]
  __shared__ CT ls[3][K];
  const int j = patch_begin + int(blockIdx.x);
  const int t = threadIdx.x;
  const int l1 = t & 3, l2 = (t >> 2) & 3, c1 = (t >> 4) & 1, c2 = t >> 5;
  const int ty = 4 * c1 + l1, tz = 4 * c2 + l2;

  // a starting wave issues its loads ahead of the other waves' arithmetic on the SIMD
  // (raised priority until the last load of the batch is issued)
  __builtin_amdgcn_s_setprio(3);
  const uint32_t f0 = fac[size_t(j) * 3], f1 = fac[size_t(j) * 3 + 1], f2 = fac[size_t(j) * 3 + 2];
  int v[3];
  unpack_vertex(vtx[j], v);
  const int64_t nn = int64_t(n) * n;
  const int64_t cell0 = (v[0] - 1) + int64_t(n) * (v[1] - 1) + nn * (v[2] - 1);
  const int64_t c_lo = cell0 + int64_t(n) * c1 + nn * c2;
  const int lyz = NP * (t & 15);
  CT lv = CT(1);
  if(t < 3 * K) lv = lam_tab[size_t(t < K ? f0 : t < 2 * K ? f1 : f2) * K + t % K];
  CT g[K], r[K], o[K];
  load_row<NP>(b + c_lo * NDC + lyz, g);
  load_row<NP>(b + (c_lo + 1) * NDC + lyz, g + NP);

  if(!(x_zero & kOuterZero))
  {
    // neighbour lines [direction][side]; absent neighbours read the patch's own cells (in
    // bounds) and are discarded by selection (a branch would hold its loads back)
    CT nl[3][2][NP];
    const CT *tt = reinterpret_cast<const CT *>(&tab);
    CT Ma[NP], Mb[NP];
    load_row<NP>(x + (v[0] > 1 ? c_lo - 1 : c_lo) * NDC + lyz, nl[0][0]);
    load_row<NP>(x + (v[0] + 1 < n ? c_lo + 2 : c_lo) * NDC + lyz, nl[0][1]);
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      const bool hy = side ? v[1] + 1 < n : v[1] > 1, hz = side ? v[2] + 1 < n : v[2] > 1;
      const VT *py = x + (cell0 + c1 + nn * c2 + (hy ? (side ? 2 * n : -n) : 0)) * NDC + l1 + 16 * l2;
      const VT *pz = x + (cell0 + c1 + int64_t(n) * c2 + (hz ? (side ? 2 * nn : -nn) : 0)) * NDC + (t & 15);
#pragma unroll
      for(int jj = 0; jj < NP; ++jj)
      {
        nl[1][side][jj] = py[NP * jj];
        nl[2][side][jj] = pz[NP * NP * jj];
      }
    }
#pragma unroll
    for(int q = 0; q < NP; ++q)
    {
      Ma[q] = tt[16 + l1 * NP + q];
      Mb[q] = tt[16 + l2 * NP + q];
    }
    const CT gy = tt[32 + NP * c1 + l1], gz = tt[32 + NP * c2 + l2];  // g of this lane's y- and z-node
    __builtin_amdgcn_s_setprio(0);
    CT fv[3][2], fp[3][2];
#pragma unroll
    for(int d = 0; d < 3; ++d)
#pragma unroll
      for(int side = 0; side < 2; ++side)
      {
        const bool has = side ? v[d] + 1 < n : v[d] > 1;
        CT dv = 0, q[NP];
#pragma unroll
        for(int jj = 0; jj < NP; ++jj) dv += tab.g[1 - side][jj] * nl[d][side][jj];
        const CT vv = has ? nl[d][side][side ? 0 : P] : CT(0);
        dv = has ? dv : CT(0);
        const CT pp = (side ? CT(-0.5) : CT(0.5)) * dv - tab.sigma * vv;
        // mass products across the lanes of the cell: both directions of an x-face, the
        // second of a y- or z-face (z or y; x follows in the lanes of the lines)
        lane_gather<NP, 1>(vv, nullptr, q);
        fv[d][side] = dotn<NP>(Mb, q);
        lane_gather<NP, 1>(pp, nullptr, q);
        fp[d][side] = dotn<NP>(Mb, q);
        if(d == 0)
        {
          lane_gather<NP, 0>(fv[d][side], nullptr, q);
          fv[d][side] = dotn<NP>(Ma, q);
          lane_gather<NP, 0>(fp[d][side], nullptr, q);
          fp[d][side] = dotn<NP>(Ma, q);
        }
        else
        {
          CT *F = B + ((d - 1) * 2 + side) * 128 + K * tz + ty;
          F[0] = fv[d][side];
          F[64] = fp[d][side];
        }
      }
    __syncthreads();
    const CT ey = l1 == (c1 ? P : 0) ? CT(1) : CT(0), ez = l2 == (c2 ? P : 0) ? CT(1) : CT(0);
    const CT ay = (c1 ? CT(0.5) : CT(-0.5)) * gy, az = (c2 ? CT(0.5) : CT(-0.5)) * gz;
    const CT *Fy = B + c1 * 128 + K * tz, *Fz = B + 256 + c2 * 128 + K * ty;
#pragma unroll
    for(int cx = 0; cx < 2; ++cx)
    {
      CT q[NP];
#pragma unroll
      for(int i = 0; i < NP; ++i)
        q[i] = ay * Fy[NP * cx + i] + ey * Fy[64 + NP * cx + i] + az * Fz[NP * cx + i] +
               ez * Fz[64 + NP * cx + i];
      const CT a = cx ? CT(0.5) * fv[0][1] : CT(-0.5) * fv[0][0];
#pragma unroll
      for(int i = 0; i < NP; ++i)
      {
        CT s = a * tab.g[cx][i];
#pragma unroll
        for(int jj = 0; jj < NP; ++jj) s += tab.M[i * NP + jj] * q[jj];
        g[NP * cx + i] -= s;
      }
      g[cx ? K - 1 : 0] -= fp[0][cx];
    }
    __syncthreads();  // the face points are read: B is free for the solve
  }
  else
    __builtin_amdgcn_s_setprio(0);

  if(t < 3 * K) (&ls[0][0])[t] = lv;
  const CT w = omega ? CT(omega[j]) : relaxation;
  __syncthreads();
#pragma unroll
  for(int i = 0; i < K; ++i) r[i] = g[i];
  const CT *G0 = S_tab + size_t(f0) * K * K, *G1 = S_tab + size_t(f1) * K * K,
           *G2 = S_tab + size_t(f2) * K * K;
  // even-odd products where all three 1D problems are mirror-symmetric (interior
  // patches of a uniform mesh); a wave-uniform branch
  if((eo_tab[f0] & eo_tab[f1] & eo_tab[f2]) != 0u)
    fd_lines<3, K, CT, SY, SZ, true, true>(r, o, B, G0, G1, G2, ls[0], ls[1], ls[2], w, ty + K * tz,
                                           true);
  else
    fd_lines<3, K, CT, SY, SZ, false, true>(r, o, B, G0, G1, G2, ls[0], ls[1], ls[2], w, ty + K * tz,
                                            true);
  VT *px = x + c_lo * NDC + lyz;
  if(!(x_zero & kOwnZero) && w != CT(1))
  {
    CT old[K];
    load_row<NP>(px, old);
    load_row<NP>(px + NDC, old + NP);
#pragma unroll
    for(int a = 0; a < K; ++a) o[a] += (CT(1) - w) * old[a];
  }
  if(nonfinite)
  {
    // the non-finite check of the caller's output, on the values stored here
    bool bad = false;
#pragma unroll
    for(int a = 0; a < K; ++a) bad = bad || !__builtin_isfinite(o[a]);
    if(bad) *nonfinite = 1;
  }
  store_row<NP>(px, o);
  store_row<NP>(px + NDC, o + NP);
}

// ----------------------------------------------------------------------------
// The same 3D color pass for the other degrees (K = 4, 6, 10).  Lane (a, b) = (t % K,
// t / K) of a patch holds the x-line (y, z) = (a, b) and the tangential point of each
// face with these indices; the mass products across lanes go through LDS (two
// exchanges: along b for all face points, then along a for the x-faces and as rows
// for the y- and z-faces).  Every global load of the pass is issued before the first
// wait.  K = 6, 10: one patch per block, the eigenvector matrices as scalar operands;
// K = 4: four patches per wave, matrices staged in LDS.
// Q4 spills 100 scalar registers in FP64 and 26 in FP32 (tables, pointers and matrix rows).
// Sweeps: 48^3 Q4 FP64 759 us (2246 with staging loops, plane-wise face products and a
// branch per neighbour), 27^3 Q4 FP64 268 (534), 64^3 Q2 FP32 290 (404), 33^3 Q2 FP64 142
// (181), 100^3 Q1 FP32 408 (472).
// ----------------------------------------------------------------------------
template<int K>
struct MvpLinesShape
{
  static constexpr int L = K * K;
  static constexpr int PPB = L <= 16 ? 64 / L : 1;
  static constexpr int THREADS = ((PPB * L + 63) / 64) * 64;
};

template<int K, typename VT, typename CT>
__global__ void __launch_bounds__((MvpLinesShape<K>::THREADS))
k_patch_mvp_lines(const VT *__restrict__ b, VT *__restrict__ x, const MvpTab<K / 2, CT> tab,
                  const uint32_t *__restrict__ vtx, const uint32_t *__restrict__ fac,
                  const CT *__restrict__ S_tab, const CT *__restrict__ lam_tab,
                  const uint32_t *__restrict__ eo_tab, const float *__restrict__ omega,
                  const CT relaxation, const int patch_begin, const int patch_end, const int n,
                  const int x_zero, int *__restrict__ nonfinite)
{
  using MS = MvpLinesShape<K>;
  constexpr int NP = K / 2, P = NP - 1, NL = NP * NP, NDC = NL * NP, L = MS::L, PPB = MS::PPB;
  constexpr bool SCALAR = PPB == 1;
  constexpr int NS = 3 * K * K;  // eigenvector entries of a patch
  static_assert(12 * L >= K * L, "the solve buffer fits in the first face buffer");
  __shared__ CT F1[PPB][12][L];  // face points [direction][side][v, P]; then the solve
  __shared__ CT F2[PPB][12][L];  // ... contracted along b
  __shared__ CT Ss[PPB][SCALAR ? 1 : NS];
  __shared__ CT ls[PPB][3][K];
  const int pl = PPB == 1 ? 0 : int(threadIdx.x) / L;
  const int t0 = int(threadIdx.x) - pl * L;
  const bool owner = t0 < L;
  const int t = owner ? t0 : L - 1;  // lanes beyond the patch repeat its last line
  const int jj = patch_begin + int(blockIdx.x) * PPB + pl;
  const bool valid = owner && jj < patch_end;
  const int j = jj < patch_end ? jj : patch_end - 1;
  const int ta = t % K, tb = t / K, c1 = ta / NP, c2 = tb / NP, l1 = ta - NP * c1, l2 = tb - NP * c2;

  const uint32_t f0 = fac[size_t(j) * 3], f1 = fac[size_t(j) * 3 + 1], f2 = fac[size_t(j) * 3 + 2];
  int v[3];
  unpack_vertex(vtx[j], v);
  const int64_t nn = int64_t(n) * n;
  const int64_t cell0 = (v[0] - 1) + int64_t(n) * (v[1] - 1) + nn * (v[2] - 1);
  const int64_t c_lo = cell0 + int64_t(n) * c1 + nn * c2;
  const int lyz = NP * l1 + NL * l2;
  CT lv = CT(1), sv[SCALAR ? 1 : (NS + L - 1) / L];
  if(t0 < 3 * K) lv = lam_tab[size_t(t < K ? f0 : t < 2 * K ? f1 : f2) * K + t % K];
  if constexpr(!SCALAR)
#pragma unroll
    for(int k = 0; k < NS / L; ++k)
    {
      static_assert(SCALAR || L == K * K, "a lane stages one entry of each matrix");
      sv[k] = S_tab[size_t(k == 0 ? f0 : k == 1 ? f1 : f2) * K * K + t];
    }
  CT g[K], r[K], o[K];
  load_row<NP>(b + c_lo * NDC + lyz, g);
  load_row<NP>(b + (c_lo + 1) * NDC + lyz, g + NP);
  const CT w = omega ? CT(omega[j]) : relaxation;

  if(!(x_zero & kOuterZero))
  {
    CT nl[3][2][NP];
    const CT *tt = reinterpret_cast<const CT *>(&tab);
    load_row<NP>(x + (v[0] > 1 ? c_lo - 1 : c_lo) * NDC + lyz, nl[0][0]);
    load_row<NP>(x + (v[0] + 1 < n ? c_lo + 2 : c_lo) * NDC + lyz, nl[0][1]);
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      const bool hy = side ? v[1] + 1 < n : v[1] > 1, hz = side ? v[2] + 1 < n : v[2] > 1;
      const VT *py = x + (cell0 + c1 + nn * c2 + (hy ? (side ? 2 * n : -n) : 0)) * NDC + l1 + NL * l2;
      const VT *pz =
        x + (cell0 + c1 + int64_t(n) * c2 + (hz ? (side ? 2 * nn : -nn) : 0)) * NDC + l1 + NP * l2;
#pragma unroll
      for(int k = 0; k < NP; ++k)
      {
        nl[1][side][k] = py[NP * k];
        nl[2][side][k] = pz[NL * k];
      }
    }
    CT Ma[NP], Mb[NP];
#pragma unroll
    for(int q = 0; q < NP; ++q)
    {
      Ma[q] = tt[l1 * NP + q];
      Mb[q] = tt[l2 * NP + q];
    }
    const CT gy = tt[2 * NL + NP * c1 + l1], gz = tt[2 * NL + NP * c2 + l2];
#pragma unroll
    for(int d = 0; d < 3; ++d)
#pragma unroll
      for(int side = 0; side < 2; ++side)
      {
        const bool has = side ? v[d] + 1 < n : v[d] > 1;
        CT dv = 0;
#pragma unroll
        for(int k = 0; k < NP; ++k) dv += tab.g[1 - side][k] * nl[d][side][k];
        const CT vv = has ? nl[d][side][side ? 0 : P] : CT(0);
        dv = has ? dv : CT(0);
        if(owner)
        {
          F1[pl][d * 4 + side * 2][t] = vv;
          F1[pl][d * 4 + side * 2 + 1][t] = (side ? CT(-0.5) : CT(0.5)) * dv - tab.sigma * vv;
        }
      }
    __syncthreads();
#pragma unroll
    for(int k = 0; k < 12; ++k)
    {
      CT s = 0;
#pragma unroll
      for(int q = 0; q < NP; ++q) s += Mb[q] * F1[pl][k][ta + K * (NP * c2 + q)];
      if(owner) F2[pl][k][t] = s;
    }
    __syncthreads();
    const CT ey = l1 == (c1 ? P : 0) ? CT(1) : CT(0), ez = l2 == (c2 ? P : 0) ? CT(1) : CT(0);
    const CT ay = (c1 ? CT(0.5) : CT(-0.5)) * gy, az = (c2 ? CT(0.5) : CT(-0.5)) * gz;
    const CT *Fy = &F2[pl][4 + 2 * c1][K * tb], *Fz = &F2[pl][8 + 2 * c2][K * ta];
#pragma unroll
    for(int cx = 0; cx < 2; ++cx)
    {
      CT q[NP], xv = 0, xp = 0;
#pragma unroll
      for(int i = 0; i < NP; ++i)
      {
        q[i] = ay * Fy[NP * cx + i] + ey * Fy[L + NP * cx + i] + az * Fz[NP * cx + i] +
               ez * Fz[L + NP * cx + i];
        xv += Ma[i] * F2[pl][2 * cx][NP * c1 + i + K * tb];
        xp += Ma[i] * F2[pl][2 * cx + 1][NP * c1 + i + K * tb];
      }
      const CT a = (cx ? CT(0.5) : CT(-0.5)) * xv;
#pragma unroll
      for(int i = 0; i < NP; ++i)
      {
        CT s = a * tab.g[cx][i];
#pragma unroll
        for(int k = 0; k < NP; ++k) s += tab.M[i * NP + k] * q[k];
        g[NP * cx + i] -= s;
      }
      g[cx ? K - 1 : 0] -= xp;
    }
  }
  if constexpr(!SCALAR)
#pragma unroll
    for(int k = 0; k < NS / L; ++k) Ss[pl][k * K * K + t] = sv[k];
  if(t0 < 3 * K) (&ls[pl][0][0])[t0] = lv;
  __syncthreads();
#pragma unroll
  for(int i = 0; i < K; ++i) r[i] = g[i];
  CT *B = &F1[pl][0][0];
  if constexpr(SCALAR)
  {
    const CT *G0 = S_tab + size_t(f0) * K * K, *G1 = S_tab + size_t(f1) * K * K,
             *G2 = S_tab + size_t(f2) * K * K;
    if((eo_tab[f0] & eo_tab[f1] & eo_tab[f2]) != 0u)
      fd_lines<3, K, CT, K, K * K, true, true>(r, o, B, G0, G1, G2, ls[0][0], ls[0][1], ls[0][2], w,
                                               t, owner);
    else
      fd_lines<3, K, CT, K, K * K, false, true>(r, o, B, G0, G1, G2, ls[0][0], ls[0][1], ls[0][2], w,
                                                t, owner);
  }
  else
    fd_lines<3, K, CT>(r, o, B, Ss[pl], Ss[pl] + K * K, Ss[pl] + 2 * K * K, ls[pl][0], ls[pl][1],
                       ls[pl][2], w, t, owner);
  if(!valid) return;
  VT *px = x + c_lo * NDC + lyz;
  if(!(x_zero & kOwnZero) && w != CT(1))
  {
    CT old[K];
    load_row<NP>(px, old);
    load_row<NP>(px + NDC, old + NP);
#pragma unroll
    for(int a = 0; a < K; ++a) o[a] += (CT(1) - w) * old[a];
  }
  if(nonfinite)
  {
    bool bad = false;
#pragma unroll
    for(int a = 0; a < K; ++a) bad = bad || !__builtin_isfinite(o[a]);
    if(bad) *nonfinite = 1;
  }
  store_row<NP>(px, o);
  store_row<NP>(px + NDC, o + NP);
}

// ----------------------------------------------------------------------------
// The 2D color pass: K lanes per patch, 64 / K patches per single-wave block.  Lane t
// holds the x-line y = t and the points y = t of the x-faces, x = t of the y-faces; the
// mass product along the face runs across the lanes of a cell.  Every global load of
// the pass is issued before the first wait; the eigenvector matrices of each patch
// are staged in LDS (padded: the patches of a wave read their copies without bank
// conflicts).
// Bound by launches below about 100^2 cells (4 us each, 8 per sweep), then by HBM:
// sweeps of 16^2 Q3 FP64 34 us (68), 300^2 Q3 FP64 78 (132), FP32 53 (93), 600^2 Q1 FP64
// 82 (123), 250^2 Q4 FP32 73 (108); in brackets staging loops and a branch and a wait
// per neighbour.
// ----------------------------------------------------------------------------
template<int K, typename VT, typename CT>
__global__ void __launch_bounds__(64)
k_patch_mvp_2d(const VT *__restrict__ b, VT *__restrict__ x, const MvpTab<K / 2, CT> tab,
               const uint32_t *__restrict__ vtx, const uint32_t *__restrict__ fac,
               const CT *__restrict__ S_tab, const CT *__restrict__ lam_tab,
               const float *__restrict__ omega, const CT relaxation, const int patch_begin,
               const int patch_end, const int n, const int x_zero, int *__restrict__ nonfinite)
{
  constexpr int NP = K / 2, P = NP - 1, NDC = NP * NP, PPB = 64 / K, PS = (64 + K - 1) / K;
  constexpr int SS = 2 * K * K + 16 / int(sizeof(CT));  // stride of a patch's matrices
  constexpr int SY = K, SB = K * K + 16 / int(sizeof(CT));
  __shared__ __align__(16) CT Ss[PS * SS];
  __shared__ __align__(16) CT Bs[PS * SB];
  __shared__ CT ls[PS][2][K];
  const int pl = int(threadIdx.x) / K, t = int(threadIdx.x) % K;
  const int jj = patch_begin + int(blockIdx.x) * PPB + pl;
  const bool valid = pl < PPB && jj < patch_end;
  const int j = valid ? jj : patch_end - 1;
  const int c = t / NP, l = t - NP * c;
  const uint32_t f0 = fac[size_t(j) * 2], f1 = fac[size_t(j) * 2 + 1];
  int v[3];
  unpack_vertex(vtx[j], v);
  const int64_t cell0 = (v[0] - 1) + int64_t(n) * (v[1] - 1);
  const int64_t c_lo = cell0 + int64_t(n) * c;
  CT sv[2][K];
#pragma unroll
  for(int k = 0; k < K; ++k)
  {
    sv[0][k] = S_tab[size_t(f0) * K * K + k * K + t];
    sv[1][k] = S_tab[size_t(f1) * K * K + k * K + t];
  }
  const CT lv0 = lam_tab[size_t(f0) * K + t], lv1 = lam_tab[size_t(f1) * K + t];
  const CT w = omega ? CT(omega[j]) : relaxation;
  CT g[K], r[K], o[K];
  load_row<NP>(b + c_lo * NDC + NP * l, g);
  load_row<NP>(b + (c_lo + 1) * NDC + NP * l, g + NP);
  int ra[NP];  // ds_bpermute addresses of the rotations (NP != 4)
#pragma unroll
  for(int q = 0; q < NP; ++q) ra[q] = 4 * (int(threadIdx.x) - l + (l + q) % NP);
  CT *B = Bs + pl * SB;

  if(!(x_zero & kOuterZero))
  {
    CT nl[2][2][NP], Ma[NP];
    const CT *tt = reinterpret_cast<const CT *>(&tab);
    load_row<NP>(x + (v[0] > 1 ? c_lo - 1 : c_lo) * NDC + NP * l, nl[0][0]);
    load_row<NP>(x + (v[0] + 1 < n ? c_lo + 2 : c_lo) * NDC + NP * l, nl[0][1]);
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      const bool hy = side ? v[1] + 1 < n : v[1] > 1;
      const VT *py = x + (cell0 + c + (hy ? (side ? 2 * n : -n) : 0)) * NDC + l;
#pragma unroll
      for(int k = 0; k < NP; ++k) nl[1][side][k] = py[NP * k];
    }
#pragma unroll
    for(int q = 0; q < NP; ++q) Ma[q] = tt[NDC + l * NP + q];
    const CT gy = tt[2 * NDC + NP * c + l];
    CT fv[2], fp[2];
#pragma unroll
    for(int d = 0; d < 2; ++d)
#pragma unroll
      for(int side = 0; side < 2; ++side)
      {
        const bool has = side ? v[d] + 1 < n : v[d] > 1;
        CT dv = 0, q[NP];
#pragma unroll
        for(int k = 0; k < NP; ++k) dv += tab.g[1 - side][k] * nl[d][side][k];
        const CT vv = has ? nl[d][side][side ? 0 : P] : CT(0);
        dv = has ? dv : CT(0);
        const CT pp = (side ? CT(-0.5) : CT(0.5)) * dv - tab.sigma * vv;
        lane_gather<NP, 0>(vv, ra, q);
        const CT mv = dotn<NP>(Ma, q);
        lane_gather<NP, 0>(pp, ra, q);
        const CT mp = dotn<NP>(Ma, q);
        if(d == 0)
        {
          fv[side] = mv;
          fp[side] = mp;
        }
        else
        {
          B[side * 2 * K + t] = mv;
          B[side * 2 * K + K + t] = mp;
        }
      }
    __syncthreads();
    const CT ey = l == (c ? P : 0) ? CT(1) : CT(0), ay = (c ? CT(0.5) : CT(-0.5)) * gy;
    const CT *Fy = B + c * 2 * K;
#pragma unroll
    for(int cx = 0; cx < 2; ++cx)
    {
      const CT a = (cx ? CT(0.5) : CT(-0.5)) * fv[cx];
#pragma unroll
      for(int i = 0; i < NP; ++i)
        g[NP * cx + i] -= a * tab.g[cx][i] + ay * Fy[NP * cx + i] + ey * Fy[K + NP * cx + i];
      g[cx ? K - 1 : 0] -= fp[cx];
    }
  }
#pragma unroll
  for(int k = 0; k < K; ++k)
  {
    Ss[pl * SS + k * K + t] = sv[0][k];
    Ss[pl * SS + K * K + k * K + t] = sv[1][k];
  }
  ls[pl][0][t] = lv0;
  ls[pl][1][t] = lv1;
  __syncthreads();  // the tables are staged, the face points are read
#pragma unroll
  for(int i = 0; i < K; ++i) r[i] = g[i];
  fd_lines<2, K, CT, SY>(r, o, B, Ss + pl * SS, Ss + pl * SS + K * K, Ss + pl * SS, ls[pl][0],
                         ls[pl][1], ls[pl][1], w, t, true);
  if(!valid) return;
  VT *px = x + c_lo * NDC + NP * l;
  if(!(x_zero & kOwnZero) && w != CT(1))
  {
    CT old[K];
    load_row<NP>(px, old);
    load_row<NP>(px + NDC, old + NP);
#pragma unroll
    for(int a = 0; a < K; ++a) o[a] += (CT(1) - w) * old[a];
  }
  if(nonfinite)
  {
    bool bad = false;
#pragma unroll
    for(int a = 0; a < K; ++a) bad = bad || !__builtin_isfinite(o[a]);
    if(bad) *nonfinite = 1;
  }
  store_row<NP>(px, o);
  store_row<NP>(px + NDC, o + NP);
}

// BF16-MFMA patch solves of the block-diagonal elasticity smoother (3D Q2, k = 6),
// residual-update form (MODE 0 of k_patch_fd): dst += omega_j R_j^T A_jc^{-1} R_j r
// for one component block c, two patches per 128-thread block.  The 6 x 6 x 6
// block is embedded in the 8 x 8 x 8 layout of fd_mfma_pair and zero-padded: the
// padded rows and columns of the eigenvector matrices are zero, so padded entries
// stay zero through every contraction, and the padded eigenvalues are one (no
// division by zero).  src, dst, fac: the component's block and factor rows.
template<typename VT>
__global__ void __launch_bounds__(128)
k_patch_fd_bf16_q2(const VT *__restrict__ src, VT *__restrict__ dst,
                   const uint32_t *__restrict__ vtx, const uint32_t *__restrict__ fac,
                   const float *__restrict__ S_tab, const float *__restrict__ lam_tab,
                   const float *__restrict__ omega, const float relaxation,
                   const int patch_begin, const int patch_end, const int n)
{
  constexpr int K = 6, NP = 3, NDC = 27;
  __shared__ float B2[2][512];
  __shared__ float Ss[2][3][64];
  __shared__ float ls[2][3][8];
  __shared__ float w2[2];
  const int j0 = patch_begin + 2 * int(blockIdx.x);
  for(int idx = threadIdx.x; idx < 2 * 3 * 64; idx += 128)
  {
    const int q = idx / 192, r = idx % 192, d = r / 64, e = r % 64, a = e / 8, i = e % 8;
    const int j = j0 + q;
    float v = 0.f;
    if(j < patch_end && a < K && i < K) v = S_tab[size_t(fac[size_t(j) * 3 + d]) * K * K + a * K + i];
    Ss[q][d][e] = v;
  }
  for(int idx = threadIdx.x; idx < 2 * 3 * 8; idx += 128)
  {
    const int q = idx / 24, r = idx % 24, d = r / 8, i = r % 8;
    const int j = j0 + q;
    ls[q][d][i] = (j < patch_end && i < K) ? lam_tab[size_t(fac[size_t(j) * 3 + d]) * K + i] : 1.f;
  }
  if(threadIdx.x < 2)
  {
    const int j = j0 + int(threadIdx.x);
    w2[threadIdx.x] = j < patch_end ? (omega ? omega[j] : relaxation) : 0.f;
  }
  // global index of padded entry e (x fastest) of patch slot q, or -1
  auto entry = [&](int q, int e) -> int64_t {
    const int j = j0 + q, x = e % 8, y = (e / 8) % 8, z = e / 64;
    if(j >= patch_end || x >= K || y >= K || z >= K) return -1;
    int v[3];
    unpack_vertex(vtx[j], v);
    return patch_cell<3, NP>(v, n, x, y, z) * NDC + patch_local<3, NP>(x, y, z);
  };
  for(int idx = threadIdx.x; idx < 2 * 512; idx += 128)
  {
    const int64_t g = entry(idx / 512, idx % 512);
    B2[idx / 512][idx % 512] = g >= 0 ? float(src[g]) : 0.f;
  }
  __syncthreads();
  fd_mfma_pair(B2, Ss, ls, w2);  // ends with a barrier: B2 holds the corrections
  for(int idx = threadIdx.x; idx < 2 * 512; idx += 128)
  {
    const int64_t g = entry(idx / 512, idx % 512);
    if(g >= 0) dst[g] += VT(B2[idx / 512][idx % 512]);
  }
}

}  // namespace tpss
