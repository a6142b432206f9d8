// kernels.hpp -- device kernels of libtpss_amd (gfx950).
//
// Data layout in HBM (shared by every kernel):
//   level vector   x[cell * (p+1)^dim + local], cell = sum_d c_d n^d (x fastest),
//                  local lexicographic (x fastest) on Gauss-Lobatto nodes;
//   patch tables   vtx[j] = v_0 | v_1 << 10 | v_2 << 20 (interior vertex),
//                  fac[j*dim + d] = row of the 1D factor table for direction d;
//   factor table   S[f][a][i] (eigenvector i in column i), lam[f][i];
//   AVP buffer     U[(cell * 2^dim + slot) * (p+1)^dim + local], slot = position
//                  of the cell inside the patch that produced the value.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace tpss
{
template<int V>
using ic = std::integral_constant<int, V>;

constexpr __host__ __device__ int cpow(int b, int e) { return e == 0 ? 1 : b * cpow(b, e - 1); }

// ----------------------------------------------------------------------------
// SIPG operator on the Cartesian mesh (apps/laplace_integrator.h:578-743 for
// tensor-product cells): per cell and direction d the 1D line operator
//   z = D_d x_c + F_pm x_{c-e_d} + F_mp x_{c+e_d}   (along d)
// followed by the cell mass along every other direction, summed over d.
// ----------------------------------------------------------------------------
template<typename T, int NP>
struct OpTab
{
  T M[NP * NP];
  T D[4][NP * NP];
  T Fpm[NP * NP];
  T Fmp[NP * NP];
};

// Contiguous rows of a cell (NP values along x) moved with 16-byte vector
// accesses; the types only claim element alignment, so any element offset is
// valid (global memory accesses need no 16-byte alignment on CDNA).
typedef float tpss_f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef double tpss_d2u __attribute__((ext_vector_type(2), aligned(8)));

template<int NP, typename VT, typename CT>
__device__ __forceinline__ void load_row(const VT *__restrict__ p, CT *out)
{
  if constexpr(std::is_same<VT, float>::value && NP % 4 == 0)
  {
#pragma unroll
    for(int i = 0; i < NP; i += 4)
    {
      const tpss_f4u v = *reinterpret_cast<const tpss_f4u *>(p + i);
      out[i] = CT(v.x), out[i + 1] = CT(v.y), out[i + 2] = CT(v.z), out[i + 3] = CT(v.w);
    }
  }
  else if constexpr(std::is_same<VT, double>::value && NP % 2 == 0)
  {
#pragma unroll
    for(int i = 0; i < NP; i += 2)
    {
      const tpss_d2u v = *reinterpret_cast<const tpss_d2u *>(p + i);
      out[i] = CT(v.x), out[i + 1] = CT(v.y);
    }
  }
  else
  {
#pragma unroll
    for(int i = 0; i < NP; ++i) out[i] = CT(p[i]);
  }
}

template<int NP, typename VT, typename CT>
__device__ __forceinline__ void store_row(VT *__restrict__ p, const CT *in)
{
  if constexpr(std::is_same<VT, float>::value && NP % 4 == 0)
  {
#pragma unroll
    for(int i = 0; i < NP; i += 4)
    {
      tpss_f4u v;
      v.x = float(in[i]), v.y = float(in[i + 1]), v.z = float(in[i + 2]), v.w = float(in[i + 3]);
      *reinterpret_cast<tpss_f4u *>(p + i) = v;
    }
  }
  else if constexpr(std::is_same<VT, double>::value && NP % 2 == 0)
  {
#pragma unroll
    for(int i = 0; i < NP; i += 2)
    {
      tpss_d2u v;
      v.x = double(in[i]), v.y = double(in[i + 1]);
      *reinterpret_cast<tpss_d2u *>(p + i) = v;
    }
  }
  else
  {
#pragma unroll
    for(int i = 0; i < NP; ++i) p[i] = VT(in[i]);
  }
}

// value of v in lane SRC of this lane's quad (DPP quad_perm broadcast; every
// lane has a source, so no old value has to be set first)
template<int SRC>
__device__ __forceinline__ int quad_bcast_i(int v)
{
  return __builtin_amdgcn_mov_dpp(v, SRC * 0x55, 0xF, 0xF, true);
}
template<typename CT>
__device__ __forceinline__ CT quad_bcast_rt(CT v, int src)
{
  if constexpr(std::is_same<CT, float>::value)
  {
    const int i = __float_as_int(v);
    const int r = src == 0 ? quad_bcast_i<0>(i)
                : src == 1 ? quad_bcast_i<1>(i)
                : src == 2 ? quad_bcast_i<2>(i)
                           : quad_bcast_i<3>(i);
    return __int_as_float(r);
  }
  else
  {
    const int lo = __double2loint(v), hi = __double2hiint(v);
    int rl, rh;
    if(src == 0)
      rl = quad_bcast_i<0>(lo), rh = quad_bcast_i<0>(hi);
    else if(src == 1)
      rl = quad_bcast_i<1>(lo), rh = quad_bcast_i<1>(hi);
    else if(src == 2)
      rl = quad_bcast_i<2>(lo), rh = quad_bcast_i<2>(hi);
    else
      rl = quad_bcast_i<3>(lo), rh = quad_bcast_i<3>(hi);
    return __hiloint2double(rh, rl);
  }
}

// value of v in lane `lane` of the wave (ds_bpermute)
template<typename CT>
__device__ __forceinline__ CT lane_read(CT v, int lane)
{
  if constexpr(std::is_same<CT, float>::value)
    return __int_as_float(__builtin_amdgcn_ds_bpermute(lane << 2, __float_as_int(v)));
  else
  {
    const int lo = __builtin_amdgcn_ds_bpermute(lane << 2, __double2loint(v));
    const int hi = __builtin_amdgcn_ds_bpermute(lane << 2, __double2hiint(v));
    return __hiloint2double(hi, lo);
  }
}

// value of lane (q + r) mod NP along the first (AX = 0) or second (AX = 1) lane
// index of a cell whose NP^2 (2D: NP) nodes are consecutive lanes; addr: byte address of that lane for ds_bpermute (NP != 4)
template<int NP, int AX, int R, typename T>
__device__ __forceinline__ T lane_rot(T v, const int *addr)
{
  if constexpr(R == 0)
    return v;
  else if constexpr(NP == 4)
  {
    // quad_perm (i + R) mod 4; row_ror by 16 - 4 R
    constexpr int CTRL = AX == 0 ? ((R & 3) | (((1 + R) & 3) << 2) | (((2 + R) & 3) << 4) | (((3 + R) & 3) << 6))
                                 : 0x120 + 16 - 4 * R;
    if constexpr(sizeof(T) == 4)
      return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
    else
      return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, true),
                              __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, true));
  }
  else if constexpr(sizeof(T) == 4)
    return __int_as_float(__builtin_amdgcn_ds_bpermute(addr[R], __float_as_int(v)));
  else
    return __hiloint2double(__builtin_amdgcn_ds_bpermute(addr[R], __double2hiint(v)),
                            __builtin_amdgcn_ds_bpermute(addr[R], __double2loint(v)));
}

template<int NP, int AX, typename T>
__device__ __forceinline__ void lane_gather(T v, const int *addr, T *o)
{
  o[0] = v;
  o[1] = lane_rot<NP, AX, 1>(v, addr);
  if constexpr(NP > 2) o[2] = lane_rot<NP, AX, 2>(v, addr);
  if constexpr(NP > 3) o[3] = lane_rot<NP, AX, 3>(v, addr);
  if constexpr(NP > 4) o[4] = lane_rot<NP, AX, 4>(v, addr);
}

template<int NP, typename T>
__device__ __forceinline__ T dotn(const T *a, const T *b)
{
  T s = 0;
#pragma unroll
  for(int r = 0; r < NP; ++r) s += a[r] * b[r];
  return s;
}

// Rows of N values moved through LDS in 16-byte chunks: chunk k of the row of lane
// l sits at (k * LANES + l), so that the lanes' accesses are free of bank conflicts.
template<int N, int LANES, typename T>
struct LaneRows
{
  static constexpr int CW = 16 / int(sizeof(T)), NC = (N + CW - 1) / CW;
  static constexpr int SIZE = NC * LANES * CW;
  typedef T vec __attribute__((ext_vector_type(16 / sizeof(T))));
  static __device__ __forceinline__ void put(T *buf, int lane, const T *v)
  {
#pragma unroll
    for(int k = 0; k < NC; ++k)
    {
      vec w;
#pragma unroll
      for(int e = 0; e < CW; ++e) w[e] = k * CW + e < N ? v[k * CW + e] : T(0);
      reinterpret_cast<vec *>(buf)[k * LANES + lane] = w;
    }
  }
  static __device__ __forceinline__ void get(const T *buf, int lane, T *v)
  {
#pragma unroll
    for(int k = 0; k < NC; ++k)
    {
      const vec w = reinterpret_cast<const vec *>(buf)[k * LANES + lane];
#pragma unroll
      for(int e = 0; e < CW; ++e)
        if(k * CW + e < N) v[k * CW + e] = w[e];
    }
  }
};

// ----------------------------------------------------------------------------
// The operator with a lane per x-line, any cells.  The face terms have rank two per
// line: with a neighbour line's trace (v, v') on the face (node value, Gauss-Lobatto
// nodes; one NP-term product), s = +1 on the left face, -1 on the right one, and the
// cell's own value u there,
//   y += (e_i P - s/2 g_i v) M M,  P = sigma (u - v) + s/2 v'
// beside the cell's own matrix L (stiffness and its half of the consistency terms); a
// boundary face takes the odd reflection of the cell as its neighbour.  The x
// products run in registers; the y products read the cell's lines from LDS, each
// extended by its x-face traces; two rows per lane pass through LDS for the z
// products.  The y- and z-face traces are formed by lanes that own a tangential point
// (the z-face ones contracted along y there).  Blocks of one eighth of the launch run
// on one XCD, so that neighbours in y and z are mostly found in its L2.
// Bound by LDS and instruction issue.  In brackets the forms with a thread per node or
// the neighbour planes' rows in every lane: 33^3 Q2 FP64 residual 9.8 us (12.7), 64^3 Q2
// FP64 46 (61), 40^3 Q4 FP64 71 (137), 500^2 Q3 FP64 16 (42), 300^2 Q4 FP32 9 (25).
// ----------------------------------------------------------------------------
template<int NP, typename T>
struct LineTab
{
  T M[NP * NP], L[NP * NP];
  T g[2][NP];  // phi_i'(0) / h, phi_i'(1) / h
  T sigma;
};

template<int DIM, int NP>
constexpr int line_cells_per_block()
{
  return 64 / cpow(NP, DIM - 1);
}

template<int DIM, int NP, typename VT, bool RESIDUAL>
__global__ void __launch_bounds__(64)
k_sipg_cells(const VT *__restrict__ x, VT *__restrict__ y, const VT *__restrict__ b,
             const LineTab<NP, VT> tab, const int n, const uint32_t *__restrict__ cells,
             const int64_t count)
{
  using T = VT;
  constexpr bool D3 = DIM == 3;
  constexpr int NL = cpow(NP, DIM - 1), NDC = NL * NP, P = NP - 1;
  constexpr int CPB = line_cells_per_block<DIM, NP>();
  constexpr int NX = NP + 4;  // extended line: values, then v, P of the left and right x-face
  using Ext = LaneRows<NX, 64, T>;
  using Row = LaneRows<NP, 64, T>;
  constexpr int FL = D3 ? NP : 1, FR = ((64 + NL - 1) / NL) * FL, CW = 16 / int(sizeof(T));
  using Face = LaneRows<NP, FR, T>;
  constexpr int S1 = Ext::SIZE + 4 * Face::SIZE, S2 = D3 ? 2 * Row::SIZE : 0;
  __shared__ __align__(16) T buf[S1 > S2 ? S1 : S2];
  __shared__ __align__(16) T fz[D3 ? 4 * Face::SIZE : 1];
  T *fy = buf + Ext::SIZE;
  auto eidx = [](int l, int e) { return ((e / CW) * 64 + l) * CW + e % CW; };
  auto fidx = [](int k, int r, int e) { return k * Face::SIZE + ((e / CW) * FR + r) * CW + e % CW; };

  const int t = threadIdx.x, cs = t / NL, q = t % NL;
  const int cr = min(cs, CPB - 1);  // lanes beyond the last cell read its lines
  const int q0 = q % NP, q1 = q / NP;
  const int64_t per = int64_t(gridDim.x) / 8;  // the grid is a multiple of eight blocks
  const int64_t slot = (int64_t(blockIdx.x % 8) * per + blockIdx.x / 8) * CPB + cs;
  const bool act = cs < CPB && slot < count;
  const int64_t sl = act ? slot : 0;
  const int64_t cell = cells ? int64_t(cells[sl]) : sl;
  const int ci = int(cell);
  const int cx = ci % n, cy = (ci / n) % n, cz = D3 ? ci / (n * n) : 0;
  const bool has[3][2] = {{cx > 0, cx < n - 1}, {cy > 0, cy < n - 1}, {cz > 0, cz < n - 1}};
  const T *xc = x + cell * NDC;
  T u[NP], nx[2][NP], fl[DIM - 1][2][NP], bv[NP];
  load_row<NP>(xc + NP * q, u);
  load_row<NP>(xc + NP * q + (has[0][0] ? -NDC : 0), nx[0]);
  load_row<NP>(xc + NP * q + (has[0][1] ? NDC : 0), nx[1]);
#pragma unroll
  for(int d = 1; d < DIM; ++d)
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      const bool in = has[d][side];
      const int st = d == 1 ? NP : NP * NP;
      const int64_t shift = (d == 1 ? int64_t(n) : int64_t(n) * n) * NDC;
      const int at = d == 1 ? q0 + NP * NP * q1 : q0 + NP * q1;
      // absent neighbour: the cell's own line, reversed
      const T *src = xc + (in ? (side ? shift : -shift) : 0) + at + (in ? 0 : P * st);
      const int sst = in ? st : -st;
#pragma unroll
      for(int j = 0; j < NP; ++j) fl[d - 1][side][j] = src[j * sst];
    }
  if constexpr(RESIDUAL) load_row<NP>(b + cell * NDC + NP * q, bv);
  // lane-indexed rows of the tables (kernel arguments)
  const T *tk = reinterpret_cast<const T *>(&tab);
  T M0[NP], L0[NP], M1[NP], L1[NP], g0[2], g1[2];
#pragma unroll
  for(int j = 0; j < NP; ++j)
  {
    M0[j] = tk[q0 * NP + j];
    L0[j] = tk[NP * NP + q0 * NP + j];
    if constexpr(D3)
    {
      M1[j] = tk[q1 * NP + j];
      L1[j] = tk[NP * NP + q1 * NP + j];
    }
  }
#pragma unroll
  for(int side = 0; side < 2; ++side)
  {
    g0[side] = tk[2 * NP * NP + side * NP + q0];
    g1[side] = D3 ? tk[2 * NP * NP + side * NP + q1] : T(0);
  }

  // trace (v, P) of a neighbour line r on this cell's face `side`; sg: -1 for the
  // reflection; w: the cell's own value there
  auto trace = [&](const T *r, int side, T sg, T w, T &v, T &jp) {
    T d = 0;
#pragma unroll
    for(int j = 0; j < NP; ++j) d += tab.g[1 - side][j] * r[j];
    v = sg * (side ? r[0] : r[P]);
    jp = (side ? T(-0.5) : T(0.5)) * (sg * d) + tab.sigma * (w - v);
  };
  {
    T e[NX];
#pragma unroll
    for(int i = 0; i < NP; ++i) e[i] = u[i];
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      T r[NP];
#pragma unroll
      for(int j = 0; j < NP; ++j) r[j] = has[0][side] ? nx[side][j] : -u[P - j];
      trace(r, side, T(1), u[side ? P : 0], e[NP + 2 * side], e[NP + 2 * side + 1]);
    }
    Ext::put(buf, t, e);
  }
  __syncthreads();  // the lines are staged
#pragma unroll
  for(int side = 0; side < 2; ++side)
  {
    T v, jp;
    const int r = cs * FL + q1, e = side ? P : 0;
    trace(fl[0][side], side, has[1][side] ? T(1) : T(-1), buf[eidx(cr * NL + e + NP * q1, q0)], v, jp);
    fy[fidx(2 * side, r, q0)] = v;
    fy[fidx(2 * side + 1, r, q0)] = jp;
    if constexpr(D3)
    {
      trace(fl[DIM - 2][side], side, has[2][side] ? T(1) : T(-1),
            buf[eidx(cr * NL + q1 + NP * e, q0)], v, jp);
      fz[fidx(2 * side, r, q0)] = v;
      fz[fidx(2 * side + 1, r, q0)] = jp;
    }
  }
  __syncthreads();
  // z-face traces contracted along y by the lanes (lx, ly) = (q0, q1)
  T zt[4];
  if constexpr(D3)
#pragma unroll
    for(int k = 0; k < 4; ++k)
    {
      T m = 0;
#pragma unroll
      for(int j = 0; j < NP; ++j) m += M1[j] * fz[fidx(k, cs * NP + j, q0)];
      zt[k] = m;
    }
  // y stage
  T My[NX], Ly[NP];
#pragma unroll
  for(int i = 0; i < NX; ++i) My[i] = 0;
#pragma unroll
  for(int i = 0; i < NP; ++i) Ly[i] = 0;
#pragma unroll
  for(int j = 0; j < NP; ++j)
  {
    T r[NX];
    Ext::get(buf, cr * NL + j + NP * q1, r);
#pragma unroll
    for(int i = 0; i < NX; ++i) My[i] += M0[j] * r[i];
#pragma unroll
    for(int i = 0; i < NP; ++i) Ly[i] += L0[j] * r[i];
  }
#pragma unroll
  for(int side = 0; side < 2; ++side)
  {
    T v[NP], jp[NP];
    Face::get(fy + 2 * side * Face::SIZE, cs * FL + q1, v);
    Face::get(fy + (2 * side + 1) * Face::SIZE, cs * FL + q1, jp);
    const T es = q0 == (side ? P : 0) ? T(1) : T(0), cv = (side ? T(0.5) : T(-0.5)) * g0[side];
#pragma unroll
    for(int i = 0; i < NP; ++i) Ly[i] += cv * v[i] + es * jp[i];
  }
  // x products
  T zm[NP], zl[NP], out[NP];
#pragma unroll
  for(int i = 0; i < NP; ++i)
  {
    T s = T(0.5) * (tab.g[1][i] * My[NP + 2] - tab.g[0][i] * My[NP]), s2 = 0;
#pragma unroll
    for(int j = 0; j < NP; ++j)
    {
      s += tab.L[i * NP + j] * My[j] + tab.M[i * NP + j] * Ly[j];
      if(D3) s2 += tab.M[i * NP + j] * My[j];
    }
    zm[i] = s;
    zl[i] = s2;
  }
  zm[0] += My[NP + 1];
  zm[P] += My[NP + 3];
  if constexpr(D3)
  {
    __syncthreads();  // the lines, the y-face rows and the z-face traces are read
#pragma unroll
    for(int k = 0; k < 4; ++k) fz[fidx(k, cs * NP + q1, q0)] = zt[k];
    Row::put(buf, t, zm);
    Row::put(buf + Row::SIZE, t, zl);
    __syncthreads();
    T tz[NP];
#pragma unroll
    for(int i = 0; i < NP; ++i) tz[i] = 0;
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      T v[NP], jp[NP];
      Face::get(fz + 2 * side * Face::SIZE, cs * NP + q0, v);
      Face::get(fz + (2 * side + 1) * Face::SIZE, cs * NP + q0, jp);
      const T ez = q1 == (side ? P : 0) ? T(1) : T(0), cv = (side ? T(0.5) : T(-0.5)) * g1[side];
#pragma unroll
      for(int i = 0; i < NP; ++i) tz[i] += cv * v[i] + ez * jp[i];
    }
#pragma unroll
    for(int i = 0; i < NP; ++i)
    {
      T s = 0;
#pragma unroll
      for(int j = 0; j < NP; ++j) s += tab.M[i * NP + j] * tz[j];
      out[i] = s;
    }
#pragma unroll
    for(int k = 0; k < NP; ++k)
    {
      Row::get(buf, cr * NL + q0 + NP * k, zm);
      Row::get(buf + Row::SIZE, cr * NL + q0 + NP * k, zl);
#pragma unroll
      for(int i = 0; i < NP; ++i) out[i] += M1[k] * zm[i] + L1[k] * zl[i];
    }
  }
  else
#pragma unroll
    for(int i = 0; i < NP; ++i) out[i] = zm[i];
  if(!act) return;
  if constexpr(RESIDUAL)
#pragma unroll
    for(int i = 0; i < NP; ++i) out[i] = bv[i] - out[i];
  store_row<NP>(y + cell * NDC + NP * q, out);
}

// The same operator for 3D Q1: a cell is a quad of lanes, lane (q0, q1) = (l & 1, l >> 1) holds
// the x-line (y, z) = (q0, q1), the y-face points (x, z) = (q0, q1) and the z-face points
// (x, y) = (q0, q1), so every exchange is a quad permutation and nothing passes through LDS.
// With the exchanges through LDS (its 7 KB a wave held FP64 at 5.6 waves per SIMD) FP64 levels
// of 35 to 52 cells took 4 to 9 % longer than with whole neighbour planes in every lane.
// Apply in us, planes / LDS / here: 46^3 FP64 6.7 / 7.2 / 6.6, 37^3 FP64 5.0 / 5.2 / 5.0, 110^3
// FP64 74 / - / 57, FP32 52 / - / 37.
template<int S0, int S1, int S2, int S3, typename T>
__device__ __forceinline__ T quad_perm(T v)
{
  constexpr int CTRL = S0 | (S1 << 2) | (S2 << 4) | (S3 << 6);
  if constexpr(sizeof(T) == 4)
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
  else
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, true));
}

template<typename VT, bool RESIDUAL>
__global__ void __launch_bounds__(64)
k_sipg_cells_q1(const VT *__restrict__ x, VT *__restrict__ y, const VT *__restrict__ b,
                const LineTab<2, VT> tab, const int n, const uint32_t *__restrict__ cells,
                const int64_t count)
{
  using T = VT;
  constexpr int NDC = 8;
  // values of lane (j, q1), of lane (q0, j), of lane (q1, j) and of lane (j, q0)
  auto at_y = [](auto J, T v) { constexpr int j = decltype(J)::value; return quad_perm<j, j, 2 + j, 2 + j>(v); };
  auto at_z = [](auto J, T v) { constexpr int j = decltype(J)::value; return quad_perm<2 * j, 2 * j + 1, 2 * j, 2 * j + 1>(v); };
  auto at_yz = [](auto J, T v) { constexpr int j = decltype(J)::value; return quad_perm<2 * j, 2 * j, 2 * j + 1, 2 * j + 1>(v); };
  auto at_xy = [](auto J, T v) { constexpr int j = decltype(J)::value; return quad_perm<j, j + 2, j, j + 2>(v); };

  const int q = threadIdx.x % 4, q0 = q & 1, q1 = q >> 1;
  const int64_t per = int64_t(gridDim.x) / 8;  // the grid is a multiple of eight blocks
  const int64_t slot = (int64_t(blockIdx.x % 8) * per + blockIdx.x / 8) * 16 + threadIdx.x / 4;
  const bool act = slot < count;
  const int64_t sl = act ? slot : 0;
  const int64_t cell = cells ? int64_t(cells[sl]) : sl;
  const int ci = int(cell);
  const int cc[3] = {ci % n, (ci / n) % n, ci / (n * n)};
  const T *xc = x + cell * NDC;
  // the line of the cell and of its x-neighbours; the y- and z-neighbours' lines at the
  // lane's face points (an absent neighbour: the cell's own line, reversed)
  T u[2], nb[3][2][2], bv[2];
  load_row<2>(xc + 2 * q, u);
#pragma unroll
  for(int d = 0; d < 3; ++d)
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      const bool in = side ? cc[d] < n - 1 : cc[d] > 0;
      const int64_t shift = (d == 0 ? int64_t(1) : d == 1 ? int64_t(n) : int64_t(n) * n) * NDC;
      const int st = 1 << d, at = d == 0 ? 2 * q : d == 1 ? q0 + 4 * q1 : q;
      const T *src = xc + (in ? (side ? shift : -shift) : 0) + at;
      const T r0 = src[0], r1 = src[st];
      nb[d][side][0] = in ? r0 : -r1;
      nb[d][side][1] = in ? r1 : -r0;
    }
  if constexpr(RESIDUAL) load_row<2>(b + cell * NDC + 2 * q, bv);
  // lane-indexed rows of the tables
  const bool odd0 = q0 != 0, odd1 = q1 != 0;
  T M0[2], M1[2], L0[2], L1[2], g0[2], g1[2];
#pragma unroll
  for(int j = 0; j < 2; ++j)
  {
    M0[j] = odd0 ? tab.M[2 + j] : tab.M[j];
    M1[j] = odd1 ? tab.M[2 + j] : tab.M[j];
    L0[j] = odd0 ? tab.L[2 + j] : tab.L[j];
    L1[j] = odd1 ? tab.L[2 + j] : tab.L[j];
    g0[j] = odd0 ? tab.g[j][1] : tab.g[j][0];
    g1[j] = odd1 ? tab.g[j][1] : tab.g[j][0];
  }
  // traces (v, P) of the neighbours' lines; w: the cell's own value on the face
  T v[3][2], jp[3][2];
  auto trace = [&](int d, int side, T w) {
    const T *r = nb[d][side];
    const T dn = tab.g[1 - side][0] * r[0] + tab.g[1 - side][1] * r[1];
    v[d][side] = side ? r[0] : r[1];
    jp[d][side] = (side ? T(-0.5) : T(0.5)) * dn + tab.sigma * (w - v[d][side]);
  };
  trace(0, 0, u[0]);
  trace(0, 1, u[1]);
  // (every lane takes part in the permutations, the selection follows; scalars: a selection
  // between entries of an array would move the array out of registers)
  const T y00 = at_y(ic<0>{}, u[0]), y01 = at_y(ic<0>{}, u[1]);
  const T y10 = at_y(ic<1>{}, u[0]), y11 = at_y(ic<1>{}, u[1]);
  const T z00 = at_yz(ic<0>{}, u[0]), z01 = at_yz(ic<0>{}, u[1]);
  const T z10 = at_yz(ic<1>{}, u[0]), z11 = at_yz(ic<1>{}, u[1]);
  trace(1, 0, odd0 ? y01 : y00);
  trace(1, 1, odd0 ? y11 : y10);
  trace(2, 0, odd0 ? z01 : z00);
  trace(2, 1, odd0 ? z11 : z10);
  // y stage: masses and L along y of the lines, masses of the x-face traces
  T My[2], Ly[2], Mv[2], Mp[2], Zv[2], Zp[2];
#pragma unroll
  for(int i = 0; i < 2; ++i)
  {
    const T r0 = i ? y01 : y00, r1 = i ? y11 : y10;
    My[i] = M0[0] * r0 + M0[1] * r1;
    Ly[i] = L0[0] * r0 + L0[1] * r1;
    Mv[i] = M0[0] * at_y(ic<0>{}, v[0][i]) + M0[1] * at_y(ic<1>{}, v[0][i]);
    Mp[i] = M0[0] * at_y(ic<0>{}, jp[0][i]) + M0[1] * at_y(ic<1>{}, jp[0][i]);
    // z-face traces contracted along y by the lanes (x, y) = (q0, q1)
    Zv[i] = M1[0] * at_z(ic<0>{}, v[2][i]) + M1[1] * at_z(ic<1>{}, v[2][i]);
    Zp[i] = M1[0] * at_z(ic<0>{}, jp[2][i]) + M1[1] * at_z(ic<1>{}, jp[2][i]);
  }
  T tz[2] = {T(0), T(0)};
#pragma unroll
  for(int side = 0; side < 2; ++side)
  {
    const T es = odd0 == (side == 1) ? T(1) : T(0), cv = (side ? T(0.5) : T(-0.5)) * g0[side];
    Ly[0] += cv * at_y(ic<0>{}, v[1][side]) + es * at_y(ic<0>{}, jp[1][side]);
    Ly[1] += cv * at_y(ic<1>{}, v[1][side]) + es * at_y(ic<1>{}, jp[1][side]);
    const T ez = odd1 == (side == 1) ? T(1) : T(0), cz = (side ? T(0.5) : T(-0.5)) * g1[side];
    tz[0] += cz * at_xy(ic<0>{}, Zv[side]) + ez * at_xy(ic<0>{}, Zp[side]);
    tz[1] += cz * at_xy(ic<1>{}, Zv[side]) + ez * at_xy(ic<1>{}, Zp[side]);
  }
  // x products, then z
  T out[2];
#pragma unroll
  for(int i = 0; i < 2; ++i)
  {
    const T zm = T(0.5) * (tab.g[1][i] * Mv[1] - tab.g[0][i] * Mv[0]) + Mp[i] + tab.L[2 * i] * My[0] +
                 tab.L[2 * i + 1] * My[1] + tab.M[2 * i] * Ly[0] + tab.M[2 * i + 1] * Ly[1];
    const T zl = tab.M[2 * i] * My[0] + tab.M[2 * i + 1] * My[1];
    out[i] = tab.M[2 * i] * tz[0] + tab.M[2 * i + 1] * tz[1];
    out[i] += M1[0] * at_z(ic<0>{}, zm) + L1[0] * at_z(ic<0>{}, zl);
    out[i] += M1[1] * at_z(ic<1>{}, zm) + L1[1] * at_z(ic<1>{}, zl);
  }
  if(!act) return;
  if constexpr(RESIDUAL)
#pragma unroll
    for(int i = 0; i < 2; ++i) out[i] = bv[i] - out[i];
  store_row<2>(y + cell * NDC + 2 * q, out);
}

// All cells of a 3D Q3 level (NP = 4: a cell's 16 lines are 16 lanes of one wave):
//   y = M_z (M_y z_0 + M_x z_1) + M_y M_x z_2,  z_d = line operator along d.
// Every lane loads seven rows at once -- its line of the cell and the row at the same
// position in each of the six face neighbours (absent neighbours read the cell itself
// and are zeroed by selection) -- and takes the other rows of a neighbour plane from
// the lanes that loaded them: those of a y-plane are the lanes of its quad (DPP
// broadcast), those of a z-plane sit 4 lanes apart (staged in LDS, laid out as the
// neighbour cell).  The 1D tables indexed by a lane-varying row (mass, face coupling,
// boundary-dependent cell matrices) are read from LDS.  DOT (operator form): also the
// block's part of x.y in partial[blockIdx.x] (the CG's p.Ap without a second pass over
// p and Ap).  64^3: FP32 46 us, FP64 96 us (k_sipg_cells 49 / 97 us, whose strided
// neighbour lines cost more than its fewer products save at this degree).
template<typename VT, typename CT, bool RESIDUAL, bool DOT = false>
__global__ void __launch_bounds__(256, 4)
k_sipg_lines_q3(const VT *__restrict__ x, VT *__restrict__ y, const VT *__restrict__ b,
                const OpTab<CT, 4> tab, const int n, const int64_t ncell,
                double *__restrict__ partial = nullptr)
{
  static_assert(!(DOT && RESIDUAL), "the dot is formed by the operator form");
  constexpr int NP = 4, NL = 16, NDC = 64, CPB = 16;
  static_assert(CPB * NL == 256, "16 cells of 16 lines per block");
  __shared__ CT xs[CPB][NDC];  // own cells
  __shared__ CT zs[CPB][NDC];  // z_0, later M_y z_0 + M_x z_1
  __shared__ CT ws[CPB][NDC];  // M_x z_2
  // the 1D tables in the layout of OpTab: M, D[0..3], F+-, F-+
  constexpr int TB = int(sizeof(OpTab<CT, 4>) / sizeof(CT));
  static_assert(TB == 7 * NL, "OpTab<CT, 4> holds seven 4 x 4 tables");
  __shared__ CT tb[256];  // every thread stores (a guarded store would pull its load behind the rows)
  const CT *tM = tb, *tFpm = tb + 5 * NL, *tFmp = tb + 6 * NL;
  const int cs = threadIdx.x / NL, ln = threadIdx.x % NL;
  const int ly = ln % NP, lz = ln / NP;
  const int64_t cell = int64_t(blockIdx.x) * CPB + cs;
  const bool act = cell < ncell;
  const int64_t cc = act ? cell : ncell - 1;  // idle lanes load an existing cell
  const int64_t nn = int64_t(n) * n;
  const int ci = int(cc);
  const int cx = ci % n, cy = (ci / n) % n, cz = ci / (n * n);
  const bool hxl = cx > 0, hxr = cx < n - 1, hyl = cy > 0, hyr = cy < n - 1;
  const bool hzl = cz > 0, hzr = cz < n - 1;
  const int lofs = NP * ly + NL * lz;  // this line within the cell, and the row
                                       // this lane loads from every neighbour
  // this thread's table entry, loaded with the rows (staged in LDS below)
  const CT tv = reinterpret_cast<const CT *>(&tab)[min(int(threadIdx.x), TB - 1)];
  CT xo[NP], xl[NP], xr[NP], ya[NP], yb[NP], za[NP], zb[NP], bv[NP];
  load_row<NP>(x + cc * NDC + lofs, xo);
  load_row<NP>(x + (hxl ? cc - 1 : cc) * NDC + lofs, xl);
  load_row<NP>(x + (hxr ? cc + 1 : cc) * NDC + lofs, xr);
  load_row<NP>(x + (hyl ? cc - n : cc) * NDC + lofs, ya);
  load_row<NP>(x + (hyr ? cc + n : cc) * NDC + lofs, yb);
  load_row<NP>(x + (hzl ? cc - nn : cc) * NDC + lofs, za);
  load_row<NP>(x + (hzr ? cc + nn : cc) * NDC + lofs, zb);
  if constexpr(RESIDUAL) load_row<NP>(b + cc * NDC + lofs, bv);
#pragma unroll
  for(int i = 0; i < NP; ++i)
  {
    xl[i] = hxl ? xl[i] : CT(0);
    xr[i] = hxr ? xr[i] : CT(0);
    ya[i] = hyl ? ya[i] : CT(0);
    yb[i] = hyr ? yb[i] : CT(0);
    za[i] = hzl ? za[i] : CT(0);
    zb[i] = hzr ? zb[i] : CT(0);
    xs[cs][lofs + i] = xo[i];
  }
  tb[threadIdx.x] = tv;
  __syncthreads();  // own cells and tables staged

  // z_0: along x, own line and the x-neighbours' lines
  CT z0[NP];
  {
    const CT *D = tb + NL * (1 + ((hxl ? 1 : 0) | (hxr ? 2 : 0)));
#pragma unroll
    for(int i = 0; i < NP; ++i)
    {
      CT s = 0;
#pragma unroll
      for(int j = 0; j < NP; ++j)
        s += D[i * NP + j] * xo[j] + tab.Fpm[i * NP + j] * xl[j] + tab.Fmp[i * NP + j] * xr[j];
      z0[i] = s;
    }
  }
  // z_1 (along y) and z_2 (along z) for every x-node of this line
  CT z1[NP], z2[NP];
  {
    const CT *D = tb + NL * (1 + ((hyl ? 1 : 0) | (hyr ? 2 : 0)));
#pragma unroll
    for(int i = 0; i < NP; ++i)
    {
      CT s = 0;
#pragma unroll
      for(int j = 0; j < NP; ++j) s += D[ly * NP + j] * xs[cs][i + NP * j + NL * lz];
      z1[i] = s;
    }
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      const CT *F = side == 0 ? tFpm : tFmp;
#pragma unroll
      for(int j = 0; j < NP; ++j)
      {
        // row j of the neighbour's plane lz: loaded by lane j of this quad
        const CT f = F[ly * NP + j];
#pragma unroll
        for(int i = 0; i < NP; ++i) z1[i] += f * quad_bcast_rt(side == 0 ? ya[i] : yb[i], j);
      }
    }
  }
  {
    const CT *D = tb + NL * (1 + ((hzl ? 1 : 0) | (hzr ? 2 : 0)));
#pragma unroll
    for(int i = 0; i < NP; ++i)
    {
      CT s = 0;
#pragma unroll
      for(int k = 0; k < NP; ++k) s += D[lz * NP + k] * xs[cs][i + NP * ly + NL * k];
      z2[i] = s;
    }
    // the z-neighbours' rows of every lane through LDS (zs / ws are free until
    // z_0 and M_x z_2 are staged there): each neighbour cell laid out like xs
#pragma unroll
    for(int i = 0; i < NP; ++i)
    {
      zs[cs][lofs + i] = za[i];
      ws[cs][lofs + i] = zb[i];
    }
    __syncthreads();
#pragma unroll
    for(int side = 0; side < 2; ++side)
    {
      const CT *F = side == 0 ? tFpm : tFmp;
      const CT *nb = side == 0 ? zs[cs] : ws[cs];
#pragma unroll
      for(int k = 0; k < NP; ++k)
      {
        // row (ly, k) of the neighbour
        const CT f = F[lz * NP + k];
#pragma unroll
        for(int i = 0; i < NP; ++i) z2[i] += f * nb[i + NP * ly + NL * k];
      }
    }
    __syncthreads();  // every lane has read the rows before zs / ws are rewritten
  }
  // x mass contractions in registers
  CT m1[NP], w2[NP];
#pragma unroll
  for(int i = 0; i < NP; ++i)
  {
    CT s1 = 0, s2 = 0;
#pragma unroll
    for(int j = 0; j < NP; ++j)
    {
      s1 += tab.M[i * NP + j] * z1[j];
      s2 += tab.M[i * NP + j] * z2[j];
    }
    m1[i] = s1;
    w2[i] = s2;
  }
#pragma unroll
  for(int i = 0; i < NP; ++i)
  {
    zs[cs][lofs + i] = z0[i];
    ws[cs][lofs + i] = w2[i];
  }
  __syncthreads();
  CT a[NP], bb[NP];
#pragma unroll
  for(int i = 0; i < NP; ++i)
  {
    CT s = m1[i], s2 = 0;
#pragma unroll
    for(int j = 0; j < NP; ++j)
    {
      const CT m = tM[ly * NP + j];
      s += m * zs[cs][i + NP * j + NL * lz];
      s2 += m * ws[cs][i + NP * j + NL * lz];
    }
    a[i] = s;
    bb[i] = s2;
  }
  __syncthreads();
#pragma unroll
  for(int i = 0; i < NP; ++i) zs[cs][lofs + i] = a[i];
  __syncthreads();
  CT out[NP];
#pragma unroll
  for(int i = 0; i < NP; ++i)
  {
    CT s = bb[i];
#pragma unroll
    for(int k = 0; k < NP; ++k) s += tM[lz * NP + k] * zs[cs][i + NP * ly + NL * k];
    out[i] = s;
  }
  if constexpr(DOT)
  {
    __shared__ double wsum[4];
    double d = 0.0;
    if(act)
#pragma unroll
      for(int i = 0; i < NP; ++i) d += double(xo[i]) * double(out[i]);
#pragma unroll
    for(int off = 32; off > 0; off >>= 1) d += __shfl_xor(d, off);
    if((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = d;
    __syncthreads();
    if(threadIdx.x == 0) partial[blockIdx.x] = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
  }
  if(!act) return;
  if(RESIDUAL)
#pragma unroll
    for(int i = 0; i < NP; ++i) out[i] = bv[i] - out[i];
  store_row<NP>(y + cell * NDC + lofs, out);
}

// ----------------------------------------------------------------------------
// Vertex patches: thread = one line of the patch tensor; the line direction rotates
// through LDS between the per-direction contractions.
// ----------------------------------------------------------------------------
template<int DIM, int K>
struct PatchShape
{
  static constexpr int NP = K / 2;
  static constexpr int L = cpow(K, DIM - 1);   // lines per patch
  static constexpr int NPD = cpow(K, DIM);     // DoFs per patch
  static constexpr int NDC = cpow(NP, DIM);    // DoFs per cell
  static constexpr int PPB = (128 / L) > 0 ? (128 / L) : 1;
  static constexpr int THREADS = ((PPB * L + 63) / 64) * 64;  // launched block size
};

inline __device__ __forceinline__ void unpack_vertex(uint32_t w, int *v)
{
  v[0] = int(w & 1023u);
  v[1] = int((w >> 10) & 1023u);
  v[2] = int((w >> 20) & 1023u);
}

// Patch-local multi-index (i0, i1, i2), i_d in [0, 2(p+1)), of the patch at
// interior vertex v -> global cell, cell-local DoF and the cell's position in
// the patch.  The DGQ 1D map i_d = cell_no*(p+1) + local (dof_info.h:358-369)
// with cells of the patch in lexicographic order (patch_info.templates.h:401-402).
template<int DIM, int NP>
__device__ __forceinline__ int64_t patch_cell(const int *v, int n, int i0, int i1, int i2)
{
  int64_t c = v[0] - 1 + (i0 >= NP ? 1 : 0);
  if(DIM > 1) c += int64_t(n) * (v[1] - 1 + (i1 >= NP ? 1 : 0));
  if(DIM > 2) c += int64_t(n) * n * (v[2] - 1 + (i2 >= NP ? 1 : 0));
  return c;
}

template<int DIM, int NP>
__device__ __forceinline__ int patch_local(int i0, int i1, int i2)
{
  int l = i0 >= NP ? i0 - NP : i0;
  if(DIM > 1) l += NP * (i1 >= NP ? i1 - NP : i1);
  if(DIM > 2) l += NP * NP * (i2 >= NP ? i2 - NP : i2);
  return l;
}

template<int DIM, int NP>
__device__ __forceinline__ int patch_slot(int i0, int i1, int i2)
{
  int s = (i0 >= NP ? 1 : 0);
  if(DIM > 1) s |= (i1 >= NP ? 2 : 0);
  if(DIM > 2) s |= (i2 >= NP ? 4 : 0);
  return s;
}

// the gather/scatter index table: out[j * K^dim + i] = global DoF of patch DoF i
template<int DIM, int K>
__global__ void k_patch_dof_indices(const uint32_t *__restrict__ vtx, const int P, const int n,
                                    uint32_t *__restrict__ out)
{
  constexpr int NP = K / 2, NPD = cpow(K, DIM), NDC = cpow(NP, DIM);
  const int64_t g = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if(g >= int64_t(P) * NPD) return;
  const int j = int(g / NPD), i = int(g % NPD);
  int v[3];
  unpack_vertex(vtx[j], v);
  const int i0 = i % K, i1 = DIM > 1 ? (i / K) % K : 0, i2 = DIM > 2 ? i / (K * K) : 0;
  out[g] = uint32_t(patch_cell<DIM, NP>(v, n, i0, i1, i2) * NDC + patch_local<DIM, NP>(i0, i1, i2));
}

// s * w / lam.  FP32: the hardware reciprocal (1 ulp), well inside the FP32 patch
// solve's rounding.  FP64: the hardware reciprocal refined by two Newton steps
// r <- r + r (1 - lam r) (each doubles the correct bits; within an ulp or two of
// 1/lam), five instructions instead of the correctly rounded division's scale,
// refinement and fix-up sequence
template<typename CT>
__device__ __forceinline__ CT eig_scale(CT s, CT w, CT lam)
{
  if constexpr(std::is_same<CT, float>::value)
    return s * w * __builtin_amdgcn_rcpf(lam);
  else
  {
    double r = __builtin_amdgcn_rcp(lam);
    double e = fma(-lam, r, 1.0);
    r = fma(r, e, r);
    e = fma(-lam, r, 1.0);
    r = fma(r, e, r);
    return s * w * r;
  }
}

// o = S^T r (forward) and r = S o (backward) along one line, S[a * K + i] =
// component a of eigenvector i
template<int K, typename CT>
__device__ __forceinline__ void s_forward(const CT *S, const CT *r, CT *o)
{
#pragma unroll
  for(int i = 0; i < K; ++i)
  {
    CT s = 0;
#pragma unroll
    for(int a = 0; a < K; ++a) s += S[a * K + i] * r[a];
    o[i] = s;
  }
}

template<int K, typename CT>
__device__ __forceinline__ void s_backward(const CT *S, const CT *o, CT *r)
{
#pragma unroll
  for(int a = 0; a < K; ++a)
  {
    CT s = 0;
#pragma unroll
    for(int i = 0; i < K; ++i) s += S[a * K + i] * o[i];
    r[a] = s;
  }
}

// The same products with a wave-uniform matrix in read-only global memory, its rows
// loaded into scalar registers a few at a time.  The pointer of every group is opaque
// to the compiler: without that it loads the matrices of all stages at once, which
// exceeds the scalar registers (in the FP64 K = 8 solve 440 of 1300 VALU instructions
// saved and restored them).
// EVEN_ODD: the first K/2 eigenvectors are symmetric, the last K/2 antisymmetric under
// the reversal a -> K-1-a (the 1D problems of patches whose two cells have equal lengths
// and no boundary face), so each product takes two (K/2 x K/2) blocks of S on the folded
// line r_a +- r_{K-1-a}: half the multiply-adds.  (A compile-time choice: a run-time one
// keeps the line arrays out of registers.)
template<typename CT>
__device__ __forceinline__ auto scalar_rows(const CT *p)
{
  typedef const __attribute__((address_space(4))) CT *ptr;
  ptr q = (ptr)p;
  asm volatile("" : "+s"(q));
  return q;
}

// rows of K values per group: at most 64 scalar registers
template<int K, typename CT>
constexpr int scalar_row_group()
{
  return 64 / (K * int(sizeof(CT) / 4));
}

template<int K, bool EVEN_ODD, typename CT>
__device__ __forceinline__ void s_forward_scalar(const CT *S, const CT *r, CT *o)
{
  constexpr int P = K / 2, R = EVEN_ODD ? P : K, G = scalar_row_group<K, CT>();
#pragma unroll
  for(int i = 0; i < K; ++i) o[i] = 0;
#pragma unroll
  for(int a0 = 0; a0 < R; a0 += G)
  {
    const auto rows = scalar_rows(S + a0 * K);
#pragma unroll
    for(int a = a0; a < (a0 + G < R ? a0 + G : R); ++a)
    {
      const CT rp = EVEN_ODD ? r[a] + r[K - 1 - a] : r[a], rm = EVEN_ODD ? r[a] - r[K - 1 - a] : r[a];
#pragma unroll
      for(int i = 0; i < K; ++i) o[i] += rows[(a - a0) * K + i] * (i < P ? rp : rm);
    }
  }
}

template<int K, bool EVEN_ODD, typename CT>
__device__ __forceinline__ void s_backward_scalar(const CT *S, const CT *o, CT *r)
{
  constexpr int P = K / 2, R = EVEN_ODD ? P : K, G = scalar_row_group<K, CT>();
#pragma unroll
  for(int a0 = 0; a0 < R; a0 += G)
  {
    const auto rows = scalar_rows(S + a0 * K);
#pragma unroll
    for(int a = a0; a < (a0 + G < R ? a0 + G : R); ++a)
    {
      CT sp = 0, sm = 0;
#pragma unroll
      for(int i = 0; i < P; ++i)
      {
        sp += rows[(a - a0) * K + i] * o[i];
        sm += rows[(a - a0) * K + P + i] * o[P + i];
      }
      r[a] = sp + sm;
      if(EVEN_ODD) r[K - 1 - a] = sp - sm;
    }
  }
}

// Fast-diagonalization inverse of one patch held as x-lines: thread t owns the
// x-line (y, z) = (t % K, t / K); on entry r is that line of the patch
// right-hand side, on exit o is the same line of
//   u = (S_2 x S_1 x S_0) diag(w / (lam_0 + lam_1 + lam_2)) (S_2^T x S_1^T x S_0^T) r.
// The line direction rotates x -> y -> z -> y -> x through the patch's LDS
// buffer B (entry (x, y, z) at x + SY y + SZ z: padded strides keep the
// transposes free of LDS bank conflicts); SCALAR: the matrices are wave-uniform in
// global memory; EO (with SCALAR): even-odd products in every direction.
// Contains __syncthreads (every thread of the block must call it).
template<int DIM, int K, typename CT, int SY = K, int SZ = K * K, bool EO = false, bool SCALAR = false>
__device__ __forceinline__ void fd_lines(CT *r, CT *o, CT *B, const CT *S0, const CT *S1,
                                         const CT *S2, const CT *l0, const CT *l1, const CT *l2,
                                         const CT w, const int t, const bool owner)
{
  static_assert(SCALAR || !EO, "even-odd products take the matrices as scalar operands");
  const int ty = DIM > 1 ? t % K : 0;
  const int tz = DIM > 2 ? t / K : 0;
  auto fwd = [](const CT *S, const CT *in, CT *out) {
    if constexpr(SCALAR)
      s_forward_scalar<K, EO>(S, in, out);
    else
      s_forward<K>(S, in, out);
  };
  auto bwd = [](const CT *S, const CT *in, CT *out) {
    if constexpr(SCALAR)
      s_backward_scalar<K, EO>(S, in, out);
    else
      s_backward<K>(S, in, out);
  };
  fwd(S0, r, o);
  if(DIM == 2)
  {
#pragma unroll
    for(int i = 0; i < K; ++i)
      if(owner) B[i + SY * ty] = o[i];
    __syncthreads();
    const int x0 = t;
#pragma unroll
    for(int jj = 0; jj < K; ++jj) r[jj] = B[x0 + SY * jj];
    fwd(S1, r, o);
#pragma unroll
    for(int jj = 0; jj < K; ++jj) o[jj] = eig_scale(o[jj], w, l0[x0] + l1[jj]);
    bwd(S1, o, r);
    __syncthreads();
#pragma unroll
    for(int b = 0; b < K; ++b)
      if(owner) B[x0 + SY * b] = r[b];
    __syncthreads();
#pragma unroll
    for(int i = 0; i < K; ++i) r[i] = B[i + SY * ty];
  }
  else
  {
#pragma unroll
    for(int i = 0; i < K; ++i)
      if(owner) B[i + SY * ty + SZ * tz] = o[i];
    __syncthreads();
    {
      const int x0 = t % K, z0 = t / K;
#pragma unroll
      for(int jj = 0; jj < K; ++jj) r[jj] = B[x0 + SY * jj + SZ * z0];
      fwd(S1, r, o);
#pragma unroll
      for(int jj = 0; jj < K; ++jj)
        if(owner) B[x0 + SY * jj + SZ * z0] = o[jj];
    }
    __syncthreads();
    {
      const int x0 = t % K, y0 = t / K;
#pragma unroll
      for(int l = 0; l < K; ++l) r[l] = B[x0 + SY * y0 + SZ * l];
      const CT lxy = l0[x0] + l1[y0];
      fwd(S2, r, o);
#pragma unroll
      for(int l = 0; l < K; ++l) o[l] = eig_scale(o[l], w, lxy + l2[l]);
      bwd(S2, o, r);
#pragma unroll
      for(int c = 0; c < K; ++c)
        if(owner) B[x0 + SY * y0 + SZ * c] = r[c];
    }
    __syncthreads();
    {
      const int x0 = t % K, z0 = t / K;
#pragma unroll
      for(int jj = 0; jj < K; ++jj) r[jj] = B[x0 + SY * jj + SZ * z0];
      bwd(S1, r, o);
#pragma unroll
      for(int b = 0; b < K; ++b)
        if(owner) B[x0 + SY * b + SZ * z0] = o[b];
    }
    __syncthreads();
#pragma unroll
    for(int i = 0; i < K; ++i) r[i] = B[i + SY * ty + SZ * tz];
  }
  bwd(S0, r, o);
}

// The same inverse with two x-lines per lane (3D): lane t of a patch's K^2 / 2 lanes
// owns the lines (t % K, t / K) and (t % K, t / K + K / 2), so that every entry of an
// eigenvector matrix read from LDS serves two lines (the one-line form is bound by
// those reads).  B: entry (x, y, z) at x + K y + SZ z.
template<int K, int SZ, typename CT>
__device__ __forceinline__ void fd_line_pairs(CT (*r)[K], CT (*o)[K], CT *B, const CT *S,
                                              const CT *l, const CT w, const int t)
{
  constexpr int H = K / 2;
  const int ta = t % K, tb = t / K;
  auto fwd = [&](const CT *M) {
#pragma unroll
    for(int i = 0; i < K; ++i)
    {
      CT s0 = 0, s1 = 0;
#pragma unroll
      for(int a = 0; a < K; ++a)
      {
        const CT m = M[a * K + i];
        s0 += m * r[0][a];
        s1 += m * r[1][a];
      }
      o[0][i] = s0;
      o[1][i] = s1;
    }
  };
  auto bwd = [&](const CT *M) {
#pragma unroll
    for(int a = 0; a < K; ++a)
    {
      CT s0 = 0, s1 = 0;
#pragma unroll
      for(int i = 0; i < K; ++i)
      {
        const CT m = M[a * K + i];
        s0 += m * o[0][i];
        s1 += m * o[1][i];
      }
      r[0][a] = s0;
      r[1][a] = s1;
    }
  };
  const CT *S0 = S, *S1 = S + K * K, *S2 = S + 2 * K * K;
  fwd(S0);
#pragma unroll
  for(int h = 0; h < 2; ++h)
#pragma unroll
    for(int i = 0; i < K; ++i) B[i + K * ta + SZ * (tb + h * H)] = o[h][i];
  __syncthreads();
#pragma unroll
  for(int h = 0; h < 2; ++h)
#pragma unroll
    for(int a = 0; a < K; ++a) r[h][a] = B[ta + K * a + SZ * (tb + h * H)];
  fwd(S1);
#pragma unroll
  for(int h = 0; h < 2; ++h)
#pragma unroll
    for(int a = 0; a < K; ++a) B[ta + K * a + SZ * (tb + h * H)] = o[h][a];
  __syncthreads();
#pragma unroll
  for(int h = 0; h < 2; ++h)
#pragma unroll
    for(int a = 0; a < K; ++a) r[h][a] = B[ta + K * (tb + h * H) + SZ * a];
  fwd(S2);
#pragma unroll
  for(int h = 0; h < 2; ++h)
  {
    const CT lxy = l[ta] + l[K + tb + h * H];
#pragma unroll
    for(int a = 0; a < K; ++a) o[h][a] = eig_scale(o[h][a], w, lxy + l[2 * K + a]);
  }
  bwd(S2);
#pragma unroll
  for(int h = 0; h < 2; ++h)
#pragma unroll
    for(int a = 0; a < K; ++a) B[ta + K * (tb + h * H) + SZ * a] = r[h][a];
  __syncthreads();
#pragma unroll
  for(int h = 0; h < 2; ++h)
#pragma unroll
    for(int a = 0; a < K; ++a) o[h][a] = B[ta + K * a + SZ * (tb + h * H)];
  bwd(S1);
#pragma unroll
  for(int h = 0; h < 2; ++h)
#pragma unroll
    for(int a = 0; a < K; ++a) B[ta + K * a + SZ * (tb + h * H)] = r[h][a];
  __syncthreads();
#pragma unroll
  for(int h = 0; h < 2; ++h)
#pragma unroll
    for(int a = 0; a < K; ++a) o[h][a] = B[a + K * ta + SZ * (tb + h * H)];
  bwd(S0);
}

// k_patch_fd: lines per lane, lanes per patch and patches per block.  3D: two lines a
// lane in single-wave blocks, except FP64 Q4, whose 40 line values a lane leave one
// wave per SIMD (40^3 additive step 598 us with two lines, 541 with one); 2D: one.
template<int DIM, int K, typename CT>
struct PatchFdShape
{
  static constexpr int NLN = DIM == 3 && !(K == 10 && sizeof(CT) == 8) ? 2 : 1;
  static constexpr int LP = cpow(K, DIM - 1) / NLN;
  static constexpr int THREADS = (LP + 63) / 64 * 64;
  static constexpr int PPB = THREADS / LP;
};

// Fused vertex-patch local solve (A2/A3/A4/A5/A12): gather r_j = R_j src,
// u_j = S diag(omega_j / sum lambda) S^T r_j, scatter.
// MODE 0: dst += correction on the patches [patch_begin, patch_end) (one color: their
// cells are disjoint), component blockIdx.y; MODE 1: the additive slot buffer.
// Every load is issued in two batches (factor rows and vertex; tables and lines) before
// the first wait; the matrices of each patch are staged in LDS.  Blocks of one eighth of
// the launch run on one XCD, so that patches sharing cells mostly share its L2.
// 3D is bound by LDS reads of the matrices and the slot buffer's traffic, 2D by latency.
// Additive steps (patches, slot sum, check), with one line a lane, staging loops and a
// separate check in brackets: 48^3 Q4 moved FP32 397 us (537), 64^3 Q3 FP32 338 (491),
// FP64 713 (848), 128^2 Q3 FP64 12.5 (18.0); 64^3 elastic Q2 FP32 sweep 1724 -> 1534.
template<int DIM, int K, typename VT, typename CT, int MODE>
__global__ void __launch_bounds__((PatchFdShape<DIM, K, CT>::THREADS))
k_patch_fd(const VT *__restrict__ src, VT *__restrict__ dst, CT *__restrict__ ubuf,
           const uint32_t *__restrict__ vtx, const uint32_t *__restrict__ fac,
           const CT *__restrict__ S_tab, const CT *__restrict__ lam_tab,
           const float *__restrict__ omega, const CT relaxation, const int patch_begin,
           const int patch_end, const int n, const int64_t comp_stride, const int64_t fac_stride)
{
  using PS = PatchFdShape<DIM, K, CT>;
  constexpr int NP = K / 2, NDC = cpow(NP, DIM), NLN = PS::NLN, LP = PS::LP, PPB = PS::PPB;
  constexpr int SLOTS = (PS::THREADS + LP - 1) / LP;  // idle lanes included
  constexpr int PAD = 16 / int(sizeof(CT));
  constexpr int SM = DIM * K * K + PAD;      // strides of the patches' tables and buffers
  constexpr int SZ = DIM == 3 && K == 8 ? 72 : K * K, SB = (DIM == 3 ? K * SZ : K * K) + PAD;
  constexpr int NE = DIM * K * K / LP, NLAM = (DIM * K + LP - 1) / LP;
  static_assert(NE * LP == DIM * K * K && NE % DIM == 0, "a lane stages NE / DIM entries of a matrix");
  __shared__ __align__(16) CT Ss[SLOTS * SM];
  __shared__ __align__(16) CT Bs[SLOTS * SB];
  __shared__ CT ls[SLOTS][DIM * K];
  const int pl = int(threadIdx.x) / LP, t = int(threadIdx.x) % LP;
  const int per = int(gridDim.x) / 8;  // the grid is a multiple of eight blocks
  const int blk = int(blockIdx.x % 8) * per + int(blockIdx.x) / 8;
  const int64_t jj = patch_begin + int64_t(blk) * PPB + pl;
  const bool valid = pl < PPB && jj < patch_end;
  const int j = valid ? int(jj) : patch_begin;
  if(MODE == 0)
  {
    src += blockIdx.y * comp_stride;
    dst += blockIdx.y * comp_stride;
    fac += blockIdx.y * fac_stride;
  }
  uint32_t f[DIM];
#pragma unroll
  for(int d = 0; d < DIM; ++d) f[d] = fac[size_t(j) * DIM + d];
  int v[3] = {1, 1, 1};
  unpack_vertex(vtx[j], v);
  const CT w = omega ? CT(omega[j]) : relaxation;
  CT sv[NE], lv[NLAM];
#pragma unroll
  for(int k = 0; k < NE; ++k)
    sv[k] = S_tab[size_t(f[k / (NE / DIM)]) * K * K + (k % (NE / DIM)) * LP + t];
#pragma unroll
  for(int k = 0; k < NLAM; ++k)
  {
    const int e = t + k * LP, d = e < K ? 0 : e < 2 * K ? 1 : DIM - 1;
    lv[k] = e < DIM * K ? lam_tab[size_t(d == 0 ? f[0] : d == 1 ? f[1] : f[DIM - 1]) * K + e % K] : CT(1);
  }
  // the lane's lines: rows of the cells c_lo and c_lo + 1
  CT r[NLN][K], o[NLN][K], old[NLN][K];
  int64_t c_lo[NLN];
  int lyz[NLN];
#pragma unroll
  for(int h = 0; h < NLN; ++h)
  {
    const int ty = t % K, tz = DIM == 3 ? t / K + h * (K / 2) : 0;
    c_lo[h] = patch_cell<DIM, NP>(v, n, 0, ty, tz);
    lyz[h] = patch_local<DIM, NP>(0, ty, tz);
    load_row<NP>(src + c_lo[h] * NDC + lyz[h], r[h]);
    load_row<NP>(src + (c_lo[h] + 1) * NDC + lyz[h], r[h] + NP);
    if constexpr(MODE == 0)
    {
      load_row<NP>(dst + c_lo[h] * NDC + lyz[h], old[h]);
      load_row<NP>(dst + (c_lo[h] + 1) * NDC + lyz[h], old[h] + NP);
    }
  }
  CT *S = Ss + pl * SM, *B = Bs + pl * SB, *l = ls[pl];
#pragma unroll
  for(int k = 0; k < NE; ++k) S[k * LP + t] = sv[k];
#pragma unroll
  for(int k = 0; k < NLAM; ++k)
    if(t + k * LP < DIM * K) l[t + k * LP] = lv[k];
  __syncthreads();
  if constexpr(NLN == 2)
  {
    fd_line_pairs<K, SZ>(r, o, B, S, l, w, t);
#pragma unroll
    for(int h = 0; h < NLN; ++h)
#pragma unroll
      for(int a = 0; a < K; ++a) o[h][a] = r[h][a];
  }
  else
    fd_lines<DIM, K, CT>(r[0], o[0], B, S, S + K * K, S + (DIM - 1) * K * K, l, l + K,
                         l + (DIM - 1) * K, w, t, true);
  if(!valid) return;
#pragma unroll
  for(int h = 0; h < NLN; ++h)
  {
    if constexpr(MODE == 0)
    {
#pragma unroll
      for(int a = 0; a < K; ++a) o[h][a] += old[h][a];
      store_row<NP>(dst + c_lo[h] * NDC + lyz[h], o[h]);
      store_row<NP>(dst + (c_lo[h] + 1) * NDC + lyz[h], o[h] + NP);
    }
    else
    {
      const int s0 = patch_slot<DIM, NP>(0, t % K, DIM == 3 ? t / K + h * (K / 2) : 0);
      store_row<NP>(ubuf + (c_lo[h] * (1 << DIM) + s0) * NDC + lyz[h], o[h]);
      store_row<NP>(ubuf + ((c_lo[h] + 1) * (1 << DIM) + (s0 | 1)) * NDC + lyz[h], o[h] + NP);
    }
  }
}

// Restricted additive Schwarz (rscatter_add, patch_transfer.templates.h:140-158):
// of the patches that contain DoF (cell c, local node l), the one that keeps it
// in the restricted prolongation -- among the patches at interior vertices of
// the cell, the one whose patch multi-index m of the DoF minimises
// (max_d floor|K/2 - 1/2 - m_d|, lexicographic index of m), the order of
// compute_restricted_dofs_impl (dof_info.templates.h:192-313; ties cannot remain,
// two patches never hold one DoF at the same multi-index).  Returns the DoF's
// slot in that patch: bit d set if the cell is the upper one in direction d.
template<int DIM, int NP>
__device__ __forceinline__ int ras_owner_slot(const int *c, const int *l, const int n)
{
  int best = -1;
  int bd = 1 << 30, bi = 1 << 30;
#pragma unroll
  for(int slot = 0; slot < (1 << DIM); ++slot)
  {
    bool ok = true;
    int dist = 0, flat = 0, st = 1;
#pragma unroll
    for(int d = 0; d < DIM; ++d)
    {
      const int bit = (slot >> d) & 1;
      const int vd = c[d] + 1 - bit;
      ok = ok && vd >= 1 && vd <= n - 1;
      // |NP - 1/2 - m_d| rounded down: NP - 1 - l_d (lower cell), l_d (upper cell)
      dist = max(dist, bit ? l[d] : NP - 1 - l[d]);
      flat += (bit * NP + l[d]) * st;
      st *= 2 * NP;
    }
    if(ok && (dist < bd || (dist == bd && flat < bi)))
    {
      best = slot;
      bd = dist;
      bi = flat;
    }
  }
  return best;
}

// dst[i] (=|+=) alpha * sum over the patches containing DoF i of their buffered
// contribution (additive Schwarz without atomics).  RAS = 1: the sum divided by
// the number of those patches (use_ras_weights, schwarz_preconditioner.templates.h:
// 636-641); RAS = 2: only the contribution of the patch that keeps the DoF
// (use_ras_boolean_weights, rscatter_add, :646-649).
// One x-row of a cell per thread; a non-finite result sets *nonfinite (if given).
template<int DIM, int NP, typename VT, typename CT, bool ACCUMULATE, int RAS = 0>
__global__ void __launch_bounds__(256)
k_avp_sum(const CT *__restrict__ ubuf, VT *__restrict__ dst, const int n, const int64_t rows,
          const double alpha, int *__restrict__ nonfinite)
{
  constexpr int NDC = cpow(NP, DIM), NR = NDC / NP;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if(i >= rows) return;
  const int64_t cell = i / NR;
  const int row = int(i - cell * NR), l = row * NP;
  int c[3] = {0, 0, 0};
  {
    int t = int(cell);  // cells < 2^24
    for(int d = 0; d < DIM; ++d)
    {
      c[d] = t % n;
      t /= n;
    }
  }
  const CT *u = ubuf + cell * (1 << DIM) * NDC + l;
  CT s[NP];
  if constexpr(RAS == 2)
  {
#pragma unroll
    for(int k = 0; k < NP; ++k)
    {
      const int lm[3] = {k, row % NP, row / NP};
      s[k] = u[ras_owner_slot<DIM, NP>(c, lm, n) * NDC + k];
    }
  }
  else
  {
    int count = 0;
    CT q[1 << DIM][NP];
#pragma unroll
    for(int slot = 0; slot < (1 << DIM); ++slot)
    {
      bool ok = true;
#pragma unroll
      for(int d = 0; d < DIM; ++d)
      {
        const int vd = c[d] + 1 - ((slot >> d) & 1);
        ok = ok && vd >= 1 && vd <= n - 1;
      }
#pragma unroll
      for(int k = 0; k < NP; ++k) q[slot][k] = CT(0);
      if(ok)
      {
        load_row<NP>(u + slot * NDC, q[slot]);
        ++count;
      }
    }
#pragma unroll
    for(int k = 0; k < NP; ++k)
    {
      s[k] = q[0][k];
#pragma unroll
      for(int slot = 1; slot < (1 << DIM); ++slot) s[k] += q[slot][k];
      if constexpr(RAS == 1) s[k] /= CT(count);
    }
  }
  VT out[NP];
  VT *pd = dst + i * NP;
  if constexpr(ACCUMULATE) load_row<NP>(pd, out);
  bool bad = false;
#pragma unroll
  for(int k = 0; k < NP; ++k)
  {
    out[k] = ACCUMULATE ? VT(double(out[k]) + alpha * double(s[k])) : VT(alpha * double(s[k]));
    bad = bad || !isfinite(out[k]);
  }
  store_row<NP>(pd, out);
  if(nonfinite && bad) *nonfinite = 1;
}

// restricted-DoF flags of every patch (DoFInfo::restricted_dof_flags_patchwise,
// dof_info.templates.h:192-313): out[j * K^DIM + i] = 1 if patch j does not keep
// its patch DoF i in the restricted prolongation
template<int DIM, int NP>
__global__ void k_restricted_flags(const uint32_t *__restrict__ vtx, const int P, const int n,
                                   uint8_t *__restrict__ out)
{
  constexpr int K = 2 * NP, NPD = cpow(K, DIM);
  const int64_t g = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if(g >= int64_t(P) * NPD) return;
  const int j = int(g / NPD), i = int(g % NPD);
  int v[3] = {1, 1, 1};
  unpack_vertex(vtx[j], v);
  int c[3] = {0, 0, 0}, lm[3] = {0, 0, 0}, slot = 0;
  for(int d = 0, t = i; d < DIM; ++d, t /= K)
  {
    const int m = t % K, bit = m / NP;
    lm[d] = m % NP;
    c[d] = v[d] - 1 + bit;
    slot |= bit << d;
  }
  out[g] = uint8_t(ras_owner_slot<DIM, NP>(c, lm, n) != slot);
}

// ----------------------------------------------------------------------------
// vectors
// ----------------------------------------------------------------------------
template<typename T>
__global__ void k_fill(T *__restrict__ x, const int64_t n, const T value)
{
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if(i < n) x[i] = value;
}

// y = a*x + b*y with host scalars
template<typename T>
__global__ void k_axpby(T *__restrict__ y, const T *__restrict__ x, const int64_t n,
                        const double a, const double b)
{
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if(i < n) y[i] = T(a * double(x[i]) + b * double(y[i]));
}

template<typename TD, typename TS>
__global__ void k_convert(TD *__restrict__ dst, const TS *__restrict__ src, const int64_t n)
{
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if(i < n) dst[i] = TD(src[i]);
}

inline __device__ __forceinline__ double splitmix_uniform(uint64_t seed, uint64_t i)
{
  uint64_t z = seed * 0x100000000ull + i;
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z = z ^ (z >> 31);
  return 2.0 * (double(z >> 11) * (1.0 / 9007199254740992.0)) - 1.0;
}

template<typename T>
__global__ void k_random(T *__restrict__ x, const int64_t n, const uint64_t seed)
{
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if(i < n) x[i] = T(splitmix_uniform(seed, uint64_t(i)));
}

// block partial sums of a.b (FP64 accumulation), deterministic two-pass reduction
template<typename T>
__global__ void __launch_bounds__(256)
k_dot_partial(const T *__restrict__ a, const T *__restrict__ b, const int64_t n,
              double *__restrict__ partial)
{
  __shared__ double sh[256];
  double s = 0.0;
  for(int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
      i += int64_t(gridDim.x) * blockDim.x)
    s += double(a[i]) * double(b[i]);
  sh[threadIdx.x] = s;
  __syncthreads();
  for(int w = 128; w > 0; w >>= 1)
  {
    if(threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if(threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

static __global__ void __launch_bounds__(256)
k_dot_final(const double *__restrict__ partial, const int np, double *__restrict__ out)
{
  __shared__ double sh[256];
  double s = 0.0;
  for(int i = threadIdx.x; i < np; i += blockDim.x) s += partial[i];
  sh[threadIdx.x] = s;
  __syncthreads();
  for(int w = 128; w > 0; w >>= 1)
  {
    if(threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if(threadIdx.x == 0) *out = sh[0];
}

// *out = the sum of np partial sums, np up to tens of thousands (one per block
// of an operator pass): 1024 threads with four independent loads in flight each
static __global__ void __launch_bounds__(1024)
k_dot_final_wide(const double *__restrict__ partial, const int np, double *__restrict__ out)
{
  __shared__ double sh[16];
  constexpr int T = 1024;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  int i = threadIdx.x;
  for(; i + 3 * T < np; i += 4 * T)
  {
    s0 += partial[i];
    s1 += partial[i + T];
    s2 += partial[i + 2 * T];
    s3 += partial[i + 3 * T];
  }
  for(; i < np; i += T) s0 += partial[i];
  double s = (s0 + s1) + (s2 + s3);
#pragma unroll
  for(int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
  if((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if(threadIdx.x < 64)
  {
    double v = threadIdx.x < 16 ? sh[threadIdx.x] : 0.0;
#pragma unroll
    for(int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if(threadIdx.x == 0) *out = v;
  }
}

// non-finite detector (grid-stride): flag[0] = 1 if any entry is NaN/Inf;
// flag may point to pinned host memory
template<typename T>
__global__ void k_nonfinite(const T *__restrict__ x, const int64_t n, int *flag)
{
  bool bad = false;
  for(int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
      i += int64_t(gridDim.x) * blockDim.x)
    bad |= !isfinite(x[i]);
  if(bad) *flag = 1;
}

// sum of one value per thread over a block of 256 threads (the tree of
// k_dot_partial); the result is valid in thread 0
__device__ __forceinline__ double block_sum_256(double v, double *sh)
{
  sh[threadIdx.x] = v;
  __syncthreads();
  for(int w = 128; w > 0; w >>= 1)
  {
    if(threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  return sh[0];
}

// CG update with device scalars, alpha = rz / pAp:  x += alpha p,
// r -= alpha Ap, block partial sums of the updated r.r (the grid-stride
// order of k_dot_partial, so the sums match dot(r, r) bit for bit) and, if
// r_low is given, the updated r in FP32 (the right-hand side of an FP32 V-cycle)
template<bool LOW>
__global__ void __launch_bounds__(256)
k_cg_update_dot(double *__restrict__ x, double *__restrict__ r, const double *__restrict__ p,
                const double *__restrict__ Ap, const int64_t n, const double *__restrict__ rz,
                const double *__restrict__ pAp, double *__restrict__ partial,
                float *__restrict__ r_low)
{
  __shared__ double sh[256];
  const double alpha = *rz / *pAp;
  double acc = 0.0;
  for(int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
      i += int64_t(gridDim.x) * blockDim.x)
  {
    x[i] += alpha * p[i];
    const double ri = r[i] - alpha * Ap[i];
    r[i] = ri;
    if(LOW) r_low[i] = float(ri);
    acc += ri * ri;
  }
  const double tot = block_sum_256(acc, sh);
  if(threadIdx.x == 0) partial[blockIdx.x] = tot;
}

// z = FP64(v) with block partial sums of r.z (grid-stride order of k_dot_partial)
template<typename T>
__global__ void __launch_bounds__(256)
k_convert_dot(double *__restrict__ z, const T *__restrict__ v, const double *__restrict__ r,
              const int64_t n, double *__restrict__ partial)
{
  __shared__ double sh[256];
  double acc = 0.0;
  for(int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
      i += int64_t(gridDim.x) * blockDim.x)
  {
    const double zi = double(v[i]);
    z[i] = zi;
    acc += r[i] * zi;
  }
  const double tot = block_sum_256(acc, sh);
  if(threadIdx.x == 0) partial[blockIdx.x] = tot;
}

// p = z + (rz_new / rz_old) p
static __global__ void k_cg_direction(double *__restrict__ p, const double *__restrict__ z,
                                      const int64_t n, const double *__restrict__ rz_new,
                                      const double *__restrict__ rz_old)
{
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const double beta = *rz_new / *rz_old;
  if(i < n) p[i] = z[i] + beta * p[i];
}

// ----------------------------------------------------------------------------
// grid transfer for DG Q_p (embedding and its transpose)
// ----------------------------------------------------------------------------
template<int NP>
struct TransferTab
{
  double P[2][NP * NP];  // P[child][i*NP + j] = phi_j((x_i + child)/2)
};

// Grid transfer per coarse cell: the cell and its 2^DIM children are viewed as
// the coarse tensor c[jx][jy][jz] (NP^DIM) and the fine tensor F[X][Y][Z]
// ((2 NP)^DIM, X = child_x * NP + fine node), linked by the 1D prolongation
// Pf[X][j] = P[X / NP][(X % NP) NP + j]:
//   prolongation F = (Pf x Pf x Pf) c,   restriction c = (Pf^T x Pf^T x Pf^T) F,
// one direction at a time through LDS (sum factorisation); one block per
// coarse cell, fine values moved child by child (contiguous cell blocks).
template<int DIM, int NP>
struct TransferShape
{
  static constexpr int K = 2 * NP;
  static constexpr int NDC = cpow(NP, DIM);
  static constexpr int NFT = cpow(K, DIM);
  static constexpr int THREADS = NFT >= 256 ? 256 : ((NFT + 63) / 64) * 64;
};

// fine tensor index (X, Y, Z) of entry `local` of child `child`
template<int DIM, int NP>
__device__ __forceinline__ int fine_tensor_index(int child, int local)
{
  constexpr int K = 2 * NP;
  int o = 0, st = 1;
#pragma unroll
  for(int d = 0; d < DIM; ++d)
  {
    o += (((child >> d) & 1) * NP + local % NP) * st;
    local /= NP;
    st *= K;
  }
  return o;
}

template<int DIM>
__device__ __forceinline__ int64_t child_cell(const int *cc, int nc, int child)
{
  int64_t f = 0, st = 1;
  const int nf = 2 * nc;
#pragma unroll
  for(int d = 0; d < DIM; ++d)
  {
    f += int64_t(2 * cc[d] + ((child >> d) & 1)) * st;
    st *= nf;
  }
  return f;
}

// coordinates of coarse cell ccell (32-bit: cells < 1000^3 < 2^31; 64-bit
// divisions by a run-time nc are long instruction sequences)
template<int DIM>
__device__ __forceinline__ void cell_coords(int64_t ccell, int nc, int *cc)
{
  int r = int(ccell);
#pragma unroll
  for(int d = 0; d < DIM; ++d)
  {
    cc[d] = r % nc;
    r /= nc;
  }
}

// xf += P xc
template<int DIM, int NP, typename T>
__global__ void __launch_bounds__((TransferShape<DIM, NP>::THREADS))
k_prolongate_add(T *__restrict__ xf, const T *__restrict__ xc, const TransferTab<NP> tab,
                 const int nc)
{
  using TS = TransferShape<DIM, NP>;
  constexpr int K = TS::K, NDC = TS::NDC, NFT = TS::NFT, NT = TS::THREADS;
  __shared__ T Pf[K * NP];
  __shared__ T S0[NFT], S1[NFT];
  const int64_t cc = blockIdx.x;
  int ccd[3] = {0, 0, 0};
  cell_coords<DIM>(cc, nc, ccd);
  const int t = threadIdx.x;
  for(int i = t; i < K * NP; i += NT) Pf[i] = T(tab.P[(i / NP) / NP][((i / NP) % NP) * NP + i % NP]);
  for(int i = t; i < NDC; i += NT) S0[i] = xc[cc * NDC + i];
  __syncthreads();
  // x: S1[X + K (jy + NP jz)] = sum_jx Pf[X][jx] c[jx][jy][jz]
  for(int o = t; o < K * NDC / NP; o += NT)
  {
    const int X = o % K, r = o / K;
    T s = 0;
#pragma unroll
    for(int j = 0; j < NP; ++j) s += Pf[X * NP + j] * S0[j + NP * r];
    S1[o] = s;
  }
  __syncthreads();
  const T *last = S1;
  if constexpr(DIM == 3)
  {
    // y: S0[X + K (Y + K jz)] = sum_jy Pf[Y][jy] S1[X + K (jy + NP jz)]
    for(int o = t; o < K * K * NP; o += NT)
    {
      const int X = o % K, Y = (o / K) % K, jz = o / (K * K);
      T s = 0;
#pragma unroll
      for(int j = 0; j < NP; ++j) s += Pf[Y * NP + j] * S1[X + K * (j + NP * jz)];
      S0[o] = s;
    }
    __syncthreads();
    last = S0;
  }
  // last direction, straight into the fine vector (child by child)
  for(int o = t; o < NFT; o += NT)
  {
    const int child = o / NDC, local = o % NDC;
    const int ft = fine_tensor_index<DIM, NP>(child, local);
    const int Z = ft / cpow(K, DIM - 1), rest = ft % cpow(K, DIM - 1);
    T s = 0;
#pragma unroll
    for(int j = 0; j < NP; ++j) s += Pf[Z * NP + j] * last[rest + cpow(K, DIM - 1) * j];
    T *dst = xf + child_cell<DIM>(ccd, nc, child) * NDC + local;
    *dst = *dst + s;
  }
}

// xc = P^T xf
template<int DIM, int NP, typename T>
__global__ void __launch_bounds__((TransferShape<DIM, NP>::THREADS))
k_restrict(T *__restrict__ xc, const T *__restrict__ xf, const TransferTab<NP> tab, const int nc)
{
  using TS = TransferShape<DIM, NP>;
  constexpr int K = TS::K, NDC = TS::NDC, NFT = TS::NFT, NT = TS::THREADS;
  constexpr int KL = cpow(K, DIM - 1);
  __shared__ T Pf[K * NP];
  __shared__ T S0[NFT], S1[NFT];
  const int64_t cc = blockIdx.x;
  int ccd[3] = {0, 0, 0};
  cell_coords<DIM>(cc, nc, ccd);
  const int t = threadIdx.x;
  for(int i = t; i < K * NP; i += NT) Pf[i] = T(tab.P[(i / NP) / NP][((i / NP) % NP) * NP + i % NP]);
  for(int o = t; o < NFT; o += NT)
  {
    const int child = o / NDC, local = o % NDC;
    S0[fine_tensor_index<DIM, NP>(child, local)] = xf[child_cell<DIM>(ccd, nc, child) * NDC + local];
  }
  __syncthreads();
  // last direction: S1[rest + KL jl] = sum_L Pf[L][jl] S0[rest + KL L]
  for(int o = t; o < KL * NP; o += NT)
  {
    const int rest = o % KL, jl = o / KL;
    T s = 0;
#pragma unroll
    for(int L = 0; L < K; ++L) s += Pf[L * NP + jl] * S0[rest + KL * L];
    S1[o] = s;
  }
  __syncthreads();
  const T *cur = S1;
  if constexpr(DIM == 3)
  {
    // y: S0[X + K (jy + NP jz)] = sum_Y Pf[Y][jy] S1[X + K (Y + K jz)]
    for(int o = t; o < K * NP * NP; o += NT)
    {
      const int X = o % K, jy = (o / K) % NP, jz = o / (K * NP);
      T s = 0;
#pragma unroll
      for(int Y = 0; Y < K; ++Y) s += Pf[Y * NP + jy] * S1[X + K * (Y + K * jz)];
      S0[o] = s;
    }
    __syncthreads();
    cur = S0;
  }
  // x: c[jx + NP r] = sum_X Pf[X][jx] cur[X + K r]
  for(int o = t; o < NDC; o += NT)
  {
    const int jx = o % NP, r = o / NP;
    T s = 0;
#pragma unroll
    for(int X = 0; X < K; ++X) s += Pf[X * NP + jx] * cur[X + K * r];
    xc[cc * NDC + o] = s;
  }
}

// y = A x with a dense row-major FP64 matrix (coarse-grid inverse); one
// 64-lane wave per row
static __global__ void __launch_bounds__(256)
k_dense_matvec(const double *__restrict__ A, const double *__restrict__ x, double *__restrict__ y,
               const int m)
{
  const int row = int(blockIdx.x) * 4 + int(threadIdx.x) / 64;
  const int lane = threadIdx.x % 64;
  if(row >= m) return;
  double s = 0.0;
  for(int c = lane; c < m; c += 64) s += A[size_t(row) * m + c] * x[c];
  for(int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if(lane == 0) y[row] = s;
}

}  // namespace tpss
