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

// FD = 0: vector FMA contractions in CT; FD = 1: BF16 MFMA contractions with
// FP32 accumulation (3D, K = 8, CT = float)
// Waves per SIMD the register allocation must allow: FP32 patch solves 5 (<= 96
// VGPRs) up to K = 8; longer lines (K = 10) hold more values per thread: 3; FP64
// solves unconstrained.
template<int K, typename CT, int FD>
constexpr int mvp_min_waves()
{
  return FD == 1 || !std::is_same<CT, float>::value ? 1 : K <= 8 ? 5 : 3;
}

template<int DIM, int K, typename VT, typename CT, int FD = 0>
__global__ void __launch_bounds__((PatchShape<DIM, K>::THREADS), (mvp_min_waves<K, CT, FD>()))
k_patch_mvp_fused(const VT *__restrict__ b, VT *__restrict__ x, const OpTab<CT, K / 2> tab,
                  const uint32_t *__restrict__ vtx, const uint32_t *__restrict__ fac,
                  const CT *__restrict__ S_tab, const CT *__restrict__ lam_tab,
                  const float *__restrict__ omega, const CT relaxation, const int patch_begin,
                  const int patch_end, const int n, const int x_zero,
                  int *__restrict__ nonfinite)
{
  using PS = PatchShape<DIM, K>;
  constexpr int NP = PS::NP, L = PS::L, NPD = PS::NPD, NDC = PS::NDC, PPB = PS::PPB;
  constexpr int SY = K, SZ = K * K;  // strides (y, z) of the patch buffers
  __shared__ CT buf[PPB][NPD];
  __shared__ CT A1[PPB][NPD];
  __shared__ CT A2[PPB][DIM > 2 ? NPD : 1];
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

  const int ty = DIM > 1 ? t % K : 0;
  const int tz = DIM > 2 ? t / K : 0;
  const int ly = ty >= NP ? ty - NP : ty, lz = tz >= NP ? tz - NP : tz;
  const int by = ty >= NP ? 1 : 0, bz = tz >= NP ? 1 : 0;
  const int64_t nn = int64_t(n) * n;

  // the x-line (ty, tz) of the patch: row lyz of the cells c_lo and c_lo + 1
  const int64_t c_lo = patch_cell<DIM, NP>(v, n, 0, ty, tz);
  const int lyz = patch_local<DIM, NP>(0, ty, tz);
  CT g[K], r[K], o[K];
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
    if(DIM > 2)
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
        if(DIM > 2) T2[i + SY * ty + SZ * tz] = t2[i];
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
        if(DIM > 2) s2 += tab.M[ly * NP + jj] * T2[i + SY * (y0 + jj) + SZ * tz];
      }
      a[i] = s;
      bb[i] = s2;
    }
    if(DIM == 2)
    {
#pragma unroll
      for(int i = 0; i < K; ++i) g[i] -= a[i];
    }
    else
    {
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
  }

  // the factor tables in LDS are complete (without the coupling stage no barrier has
  // passed since they were written)
  if(x_zero & kOuterZero) __syncthreads();
  if constexpr(FD == 1)
  {
    static_assert(DIM == 3 && K == 8 && PPB == 2, "MFMA patch solve: 3D, K = 8, two patches per block");
    __shared__ float w2[2];
    if(t == 0 && owner) w2[pl] = float(w);
    __syncthreads();  // the coupling stage above may still read A1/A2; buf is free
#pragma unroll
    for(int i = 0; i < K; ++i)
      if(owner) buf[plc][i + K * ty + K * K * tz] = float(g[i]);
    __syncthreads();
    fd_mfma_pair(reinterpret_cast<float(*)[512]>(&buf[0][0]),
                 reinterpret_cast<const float(*)[3][64]>(&Ss[0][0][0]),
                 reinterpret_cast<const float(*)[3][8]>(&ls[0][0][0]), w2);
#pragma unroll
    for(int i = 0; i < K; ++i) o[i] = buf[plc][i + K * ty + K * K * tz];
  }
  else
  {
#pragma unroll
    for(int i = 0; i < K; ++i) r[i] = g[i];
    fd_lines<DIM, K, CT>(r, o, buf[plc], Ss[plc][0], Ss[plc][1], Ss[plc][DIM > 2 ? 2 : 1],
                         ls[plc][0], ls[plc][1], ls[plc][DIM > 2 ? 2 : 1], w, t, owner);
  }
  if(!valid) return;
  if(!(x_zero & kOwnZero) && w != CT(1))
  {
    CT old[K];
    load_row<NP>(x + c_lo * NDC + lyz, old);
    load_row<NP>(x + (c_lo + 1) * NDC + lyz, old + NP);
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
// Bound by HBM: per color of the 64^3 level 42 us FP64 / 22 us FP32 (195 / 97.5 MB
// compulsory, 222 / 106 MB moved), 57 / 29 us with plane-wise face products
// (F z along the normal on every node, the masses across lines through LDS) and all
// eigenvector matrices loaded at once (their scalar registers spilled).
// ----------------------------------------------------------------------------
template<typename CT>
struct MvpTab
{
  CT M[16];
  CT R[16];      // rows of M rotated to start at the diagonal: R[q*4 + r] = M(q, (q + r) mod 4)
  CT g[2][4];    // phi_i'(0) / h, phi_i'(1) / h
  CT sigma;
};

template<typename VT, typename CT>
__global__ void __launch_bounds__(64, (std::is_same<CT, float>::value ? 6 : 2))
k_patch_mvp_q3(const VT *__restrict__ b, VT *__restrict__ x, const MvpTab<CT> tab,
               const uint32_t *__restrict__ vtx, const uint32_t *__restrict__ fac,
               const CT *__restrict__ S_tab, const CT *__restrict__ lam_tab,
               const uint32_t *__restrict__ eo_tab, const float *__restrict__ omega,
               const CT relaxation, const int patch_begin, const int n, const int x_zero,
               int *__restrict__ nonfinite)
{
  constexpr int K = 8, NP = 4, NDC = 64, P = 3;
  constexpr int SY = 8, SZ = 72;  // solve buffer (x, y, z) -> x + SY y + SZ z (bank conflicts)
  // FP32 solves read the eigenvector matrices with wave-uniform addresses straight
  // into scalar registers; FP64 ones only for the even-odd products (half matrices),
  // the full ones are staged
  constexpr bool S_SCALAR = std::is_same<CT, float>::value;
  __shared__ __align__(16) CT B[K * SZ];  // solve; before it the face points [dir][side][v, P][64]
  __shared__ CT Ss[3][S_SCALAR ? 1 : K * K];
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
  CT sv[3], lv = CT(1);
  if constexpr(!S_SCALAR)
  {
    sv[0] = S_tab[size_t(f0) * K * K + t];
    sv[1] = S_tab[size_t(f1) * K * K + t];
    sv[2] = S_tab[size_t(f2) * K * K + t];
  }
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

  if constexpr(!S_SCALAR)
#pragma unroll
    for(int d = 0; d < 3; ++d) Ss[d][t] = sv[d];
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
    fd_lines<3, K, CT, SY, SZ, false, S_SCALAR>(r, o, B, S_SCALAR ? G0 : Ss[0],
                                                S_SCALAR ? G1 : Ss[1], S_SCALAR ? G2 : Ss[2], ls[0],
                                                ls[1], ls[2], w, ty + K * tz, true);
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
