// The y and z transforms of one x plane in one workgroup (grids with n2 = n3 =
// N = A*B): the rows of the sphere at fixed x come in, and H|psi>'s rows go
// back out (k_yz_vpsi) or |psi(r)|^2 is summed (k_yz_rho); the plane itself,
// 2R+1 y columns of N values, lives in LDS and never in HBM.
//
// The separate passes of fft_reg.h move the planes of every band pair through
// HBM four times per SCF step (for 128 bands at 100^3 in FP64 2.2 of 3.2 GB)
// and had become bound by that; here a pair's rows are read twice and written
// once.  What bounds k_yz_vpsi now, at 100^3: in FP32 the vector ALU (issuing in 90 %
// of the cycles in which a CU has waves), in FP64 the few waves that fit beside a
// plane (LDS 56 %, ALU 52 %).  k_yz_rho at 100^3 in FP32 has 128 registers and spills
// 38, about a third of its HBM traffic.  y and z passes of one SCF step, ms, before
// and after: 128 bands at 100^3 0.366 -> 0.292 FP32, 0.691 -> 0.504 FP64; 256
// bands at 144^3 FP32 1.71 -> 1.48; of one H|psi> alone 0.276 -> 0.171, 0.534
// -> 0.325 and 1.32 -> 0.826.
//
// W1 is transposed for this: [pair][x][slot] with `pitch` slots per x, so that
// a block reads and writes one contiguous run (the x passes k_rows_inv_t and
// k_rows_fwd_hpsi_t turn it in LDS).  V(r) and the density's partial grids are
// held in the order in which a z group's lanes use them (YzShape::native).
//
// A wave takes CPW columns at a time, TM lanes each, so the exchange inside a
// transform stays within the wave: LDS operations of one wave execute in
// order, and no barrier is needed.  Blocks meet only between the y and the z
// side, twice per pair.  The z exchange goes through a small buffer per wave,
// real parts first and then imaginary parts, half the room, which is what
// lets two FP32 blocks of a 100^3 grid share a CU; the y exchange runs in
// place in the plane.  The twiddles W_N^(t j) of a lane stay in registers.
#pragma once
#include "fft_reg.h"
#include "yz_pads.h"

namespace amdk {

constexpr size_t LDS_PER_CU = 160 * 1024;

template <typename T, int A, int B> struct YzShape {
  using V = typename cplx_of<T>::type;
  static constexpr int N = A * B, TM = MaxAB<A, B>::v;
  static constexpr int CPW = 64 / TM;              // columns per wave
  static constexpr int GZ = (N + CPW - 1) / CPW;   // z groups of a plane
  static constexpr int imin(int a, int b) { return a < b ? a : b; }
  // strides with the fewest bank conflicts: of the plane's columns, of the y
  // exchange's rows in a column, of the z exchange's columns and rows (against
  // N + 1 throughout, where half of the LDS cycles were conflicts: k_yz_vpsi and
  // k_yz_rho at 100^3 FP64 0.346 -> 0.325 and 0.186 -> 0.179 ms, at 144^3 FP32
  // 0.906 -> 0.826 and 0.689 -> 0.651, at 180^3 4.38 -> 4.02 and 3.91 -> 3.65)
  using P = YzPads<N, sizeof(V)>;
  static constexpr int PS = P::PS, RS = P::RS, CS = P::CS, RX = P::RX, RY = P::RY;
  static constexpr size_t plane_values(int nplane) { return (size_t)nplane * PS + 1; }  // and one zero
  static constexpr size_t lds(int nplane, int waves) {
    return (size_t)nplane * sizeof(int4) + plane_values(nplane) * sizeof(V) + (size_t)waves * CPW * CS * sizeof(T);
  }
  // Waves per block.  Eight where two blocks of the widest sphere share a
  // CU's LDS.  A single block takes all the waves its registers and LDS allow
  // for H|psi> (16 in FP32, 12 in FP64 or 8), and for the density eight, or 12 from
  // 150 on.  Measured, ms, 8 / 12 / 16 waves: FP32 H|psi>
  // at 100^3 (128 bands) 0.177 / 0.222 / 0.197, at 144^3 (256 bands) 1.04 /
  // 0.96 / 0.91; FP64 at 100^3 0.382 / 0.350 / 0.587; the density at 100^3
  // FP32 0.127 / 0.131 / 0.140, FP64 0.188 / 0.336 / 0.431, at 144^3 FP32
  // 0.70 / 0.87 / 0.75; at 180^3 (512 bands, two blocks to a plane) 3.9 / 3.6.
  static constexpr bool two = 2 * lds(N / 2 + 1, 8) <= LDS_PER_CU;
  static constexpr int WV = imin(GZ, two ? 8 : sizeof(T) == 4 && lds(N / 2 + 1, 16) <= LDS_PER_CU ? 16 : lds(N / 2 + 1, 12) <= LDS_PER_CU ? 12 : 8);
  static constexpr int WR = imin(GZ, N >= 150 && lds(N / 2 + 1, 12) <= LDS_PER_CU ? 12 : 8);
  // two density blocks share a plane's z groups where one cannot hold the sums
  static constexpr int ZS = (GZ + WR - 1) / WR * A > 60 ? 2 : 1;
  static constexpr int GH = (GZ + ZS - 1) / ZS, NRH = (GH + WR - 1) / WR;
  // waves per SIMD that the density's registers are to leave room for: 128 of them
  // a lane where two FP32 blocks are to share the CU, else 256, or 168 with 12 waves
  static constexpr int EUR = two && sizeof(T) == 4 ? 4 : 2;
  static constexpr int REGS_R = EUR == 4 ? 128 : WR > 8 ? 168 : 256;
  // share of those that its sums (A doubles a round), a transform and the twiddles take
  static constexpr double regs = (2.0 * A * NRH + 2.0 * (sizeof(V) / 4) * TM) / REGS_R;
  // share of a wave's lanes that a transform's two halves keep busy
  static constexpr double lanes = CPW * (A + B) / 128.0;
  // Lengths at which the kernels measured faster than the separate passes (on
  // spheres of 70 Ry, both forms in turn; passes / y-z kernels).
  // H|psi> by itself gains wherever the transform fills a wave's lanes: 1.43 at
  // 100^3, 1.33 at 108^3, 1.26 at 144^3 in FP32, 1.60 and 1.38 at 100^3 and 108^3
  // in FP64 (96 bands); with fewer lanes busy (50 = 10 x 5, 60 = 10 x 6, 128 = 16 x 8)
  // 0.84-1.0, but below 40 the two launches saved count for more (1.27 at 32^3),
  // and from 150 on the planes' traffic.
  static constexpr bool use_vpsi = N < 40 || N >= 150 || lanes >= 0.78;
  // An SCF step also takes the density from them and saves the separate passes'
  // second use of the planes.  It gains where the density's registers hold what
  // it needs.  FP32, 128 bands: 72^3 1.08, 80^3 1.04, 90^3 1.10, 100^3 1.09, 144^3 1.03,
  // 160^3 1.04, 180^3 1.04 (0 to 38 registers spilled), but 96^3 0.87, 108^3 0.96,
  // 120^3 0.94, 150^3 0.90 (62, 70, 113 and 171).  FP64: 90^3 1.15, 100^3 1.14, 108^3 1.11,
  // 120^3 1.03; 96^3 0.99 with 64 bands and 1.03 with 128 (lanes 0.78).  Smaller grids lose
  // (FP64 72^3 0.95, 80^3 0.97 with 64 bands): the caches hold their planes.
  static constexpr bool use_scf = use_vpsi && N >= (sizeof(T) == 8 ? 90 : 72) && lanes >= 0.8 && regs <= 0.8;
  static size_t native(int n1) { return (size_t)n1 * GZ * A * 64; }  // values of one grid in lane order
};

// Position of slot s in an x column of the transposed W1: the direct rows from
// `base` up, the mirror rows from base - 1 down (the (0,0) row has none: its
// place stays empty), so that with `base` a multiple of 128 bytes the HR direct
// and the HR mirror rows of an x pass's block are whole 128-byte lines.
struct YzCols {
  int pitch, base, nrow;
  __host__ __device__ __forceinline__ int at(int s) const { return base + s - nrow + (s >= nrow - 1 ? 1 : 0); }
  // of the plane of slots [s0, s1) from m2 = lo: position of its first row, lo,
  // rows, and its first row past the empty place (only m3 = 0 reaches it)
  int4 plane(int s0, int s1, int lo) const {
    return make_int4(at(s0), lo, s1 - s0, s0 < nrow - 1 ? nrow - 1 - s0 : s1 - s0);
  }
};

// Orders one wave's LDS accesses for the compiler; the hardware keeps them in
// order by itself.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Transpose between the two halves of a column transform within the wave:
// lane t < DA hands in DB values, lane t < DB gets value t of every lane.
// RX: row stride in ex.
template <int DA, int DB, int RX, typename T, typename V>
__device__ __forceinline__ void wave_exchange(V* r, T* ex, int t, bool in) {
  const int tr = t < DB ? t : 0;
  wave_lds_sync();
  if (in)
#pragma unroll
    for (int j = 0; j < DB; ++j) ex[t * RX + j] = r[j].x;
  wave_lds_sync();
#pragma unroll
  for (int k = 0; k < DA; ++k) r[k].x = ex[k * RX + tr];
  wave_lds_sync();
  if (in)
#pragma unroll
    for (int j = 0; j < DB; ++j) ex[t * RX + j] = r[j].y;
  wave_lds_sync();
#pragma unroll
  for (int k = 0; k < DA; ++k) r[k].y = ex[k * RX + tr];
}

// What a block holds besides its pair: LDS and the lane's place in its wave.
template <typename T, int A, int B, int W> struct YzBlock {
  using S = YzShape<T, A, B>;
  using V = typename S::V;
  static constexpr int N = S::N, TM = S::TM, CPW = S::CPW, PS = S::PS;
  V* plane;   // [nplane][PS], then one zero
  T* ex;      // this wave's exchange column of lane group c
  int4* pinf; // per plane: position of its first row, lowest m2, rows, first row past the gap (YzCols::plane)
  int np, R, wave, c, t;
  bool cact;  // the lane belongs to a column of the wave
  V tw[TM];   // W_N^(t j)

  __device__ __forceinline__ YzBlock(unsigned char* smem, const PassGeom& g, const int4* __restrict__ tab,
                                     const V* __restrict__ twg) {
    np = g.nplane;
    R = g.R;
    pinf = reinterpret_cast<int4*>(smem);
    plane = reinterpret_cast<V*>(pinf + np);
    wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    c = lane / TM;
    t = lane - c * TM;
    cact = c < CPW;
    if (!cact) c = CPW - 1;
    ex = reinterpret_cast<T*>(plane + S::plane_values(np)) + (wave * CPW + c) * S::CS;
    for (int p = threadIdx.x; p < np; p += blockDim.x) pinf[p] = tab[p];
    if (threadIdx.x == 0) plane[S::plane_values(np) - 1].x = plane[S::plane_values(np) - 1].y = 0;
#pragma unroll
    for (int j = 1; j < TM; ++j) tw[j] = twg[(t * j) % N];
    __syncthreads();
  }

  // r[j] <- W_N^(DIR t j) r[j], j = 1 .. L-1
  template <int L, int DIR> __device__ __forceinline__ void twist(V* r) const {
#pragma unroll
    for (int j = 1; j < L; ++j) {
      V w = tw[j];
      if (DIR > 0) w.y = -w.y;
      r[j] = cmul(r[j], w);
    }
  }

  // byte offset of row `rel` of a plane, out of bounds past its rows
  __device__ __forceinline__ static unsigned row_off(const int4& pi, int rel, int cnt) {
    return (unsigned)rel < (unsigned)cnt ? (unsigned)((pi.x + rel + (rel >= pi.w ? 1 : 0)) * sizeof(V)) : DEAD_OFF;
  }

  __device__ __forceinline__ void load_rows(const PencilBuf<V>& rows, int g, V* r) const {
    const int p = g * CPW + c;
    const bool act = cact && p < np;
    const int4 pi = pinf[act ? p : 0];
    const int cnt = act && t < A ? pi.z : 0;
#pragma unroll
    for (int k = 0; k < B; ++k)
      if (pencil_run<true, A, N>(k)) r[k] = rows.load(row_off(pi, t - pi.y + pencil_step<A, N>(t, k), cnt));
  }
  // rows of every plane -> y columns in LDS
  __device__ __forceinline__ void y_inverse(const PencilBuf<V>& rows) {
    for (int g = wave; g * CPW < np; g += W) {
      const int p = g * CPW + c;
      const bool act = cact && p < np;
      V r[TM];
      load_rows(rows, g, r);
      RDft<V, B, +1, pencil_zeros<true, A, B>()>::run(r);
      twist<B, +1>(r);
      V* col = plane + (act ? p : 0) * PS;
      wave_lds_sync();  // the previous pair's y_forward has read the column
      if (act && t < A)
#pragma unroll
        for (int j = 0; j < B; ++j) col[t * S::RS + j] = r[j];
      wave_lds_sync();
      const int tr = t < B ? t : 0;
#pragma unroll
      for (int k = 0; k < A; ++k) r[k] = col[k * S::RS + tr];
      wave_lds_sync();  // every lane has read before the column is overwritten
      RDft<V, A, +1>::run(r);
      if (act && t < B)
#pragma unroll
        for (int j = 0; j < A; ++j) col[t + B * j] = r[j];
    }
  }

  // y columns in LDS -> rows of every plane
  __device__ __forceinline__ void y_forward(const PencilBuf<V>& rows) {
    for (int g = wave; g * CPW < np; g += W) {
      const int p = g * CPW + c;
      const bool act = cact && p < np;
      const int4 pi = pinf[act ? p : 0];
      V* col = plane + (act ? p : 0) * PS;
      V r[TM];
      const int ta = t < A ? t : 0, tb = t < B ? t : 0;
#pragma unroll
      for (int k = 0; k < B; ++k) r[k] = col[ta + A * k];
      RDft<V, B, -1>::run(r);
      twist<B, -1>(r);
      wave_lds_sync();
      if (act && t < A)
#pragma unroll
        for (int j = 0; j < B; ++j) col[t * S::RS + j] = r[j];
      wave_lds_sync();
#pragma unroll
      for (int k = 0; k < A; ++k) r[k] = col[k * S::RS + tb];
      RDft<V, A, -1>::run(r);
      const int cnt = act && t < B ? pi.z : 0;
#pragma unroll
      for (int j = 0; j < A; ++j)
        if (pencil_run<true, B, N>(j)) {
          rows.store(row_off(pi, t - pi.y + pencil_step<B, N>(t, j), cnt), r[j]);
        }
    }
  }

  // planes -> the lane's A values of z column y: X[t + B j] for t < B
  __device__ __forceinline__ void z_inverse(int y, V* r) {
    const int yc = y < N ? y : N - 1;
#pragma unroll
    for (int k = 0; k < B; ++k) {
      if (pencil_run<true, A, N>(k)) {
        const int p = t + R + pencil_step<A, N>(t, k);
        r[k] = plane[(unsigned)p < (unsigned)np ? p * PS + yc : np * PS];
      }
    }
    RDft<V, B, +1, pencil_zeros<true, A, B>()>::run(r);
    twist<B, +1>(r);
    wave_exchange<A, B, S::RX>(r, ex, t, cact && t < A);
    RDft<V, A, +1>::run(r);
  }

  // the lane's values of z column y (t < B) -> planes
  __device__ __forceinline__ void z_forward(int y, V* r) {
    RDft<V, A, -1>::run(r);
    twist<A, -1>(r);
    wave_exchange<B, A, S::RY>(r, ex, t, cact && t < B);
    RDft<V, B, -1>::run(r);
    const int cnt = cact && t < A && y < N ? np : 0;
#pragma unroll
    for (int j = 0; j < B; ++j)
      if (pencil_run<true, A, N>(j)) {
        const int p = t + R + pencil_step<A, N>(t, j);
        if ((unsigned)p < (unsigned)cnt) plane[p * PS + y] = r[j];
      }
  }
};

// H|psi>: rows -> y, z -> V(r) -> z, y -> rows, in place in W1, for pairs
// [PG grp, PG (grp + 1)) at plane x.  vn: V(r)/N in lane order.
template <typename T, int A, int B>
__global__ void __launch_bounds__((64 * YzShape<T, A, B>::WV))
    k_yz_vpsi(PassGeom g, typename cplx_of<T>::type* __restrict__ W1, YzCols cols, const int4* __restrict__ tab,
              const T* __restrict__ vn, int npairs, int PG, const typename cplx_of<T>::type* __restrict__ twg, int ngrp, int per) {
  using S = YzShape<T, A, B>;
  using V = typename S::V;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  int x, grp;
  if (!z_block_of(ngrp, per, g.n1, x, grp)) return;
  YzBlock<T, A, B, S::WV> b(smem_raw, g, tab, twg);
  const int pa = grp * PG, pb = min(npairs, pa + PG);
  auto rows_of = [&](int pl) {
    return PencilBuf<V>(W1 + ((size_t)pl * g.n1 + x) * cols.pitch, cols.pitch * (unsigned)sizeof(V));
  };
  for (int pl = pa; pl < pb; ++pl) {
    const PencilBuf<V> rows = rows_of(pl);
    b.y_inverse(rows);
    __syncthreads();
    for (int gz = b.wave; gz < S::GZ; gz += S::WV) {
      const int y = gz * S::CPW + b.c;
      const T* v = vn + ((size_t)(x * S::GZ + gz) * A) * 64 + (threadIdx.x & 63);
      T vv[A];
#pragma unroll
      for (int j = 0; j < A; ++j) vv[j] = v[64 * j];
      V r[S::TM];
      b.z_inverse(y, r);
#pragma unroll
      for (int j = 0; j < A; ++j) {
        r[j].x *= vv[j];
        r[j].y *= vv[j];
      }
      b.z_forward(y, r);
    }
    __syncthreads();
    b.y_forward(rows);  // a wave's planes are its own in the next pair's y_inverse too
  }
}

// Density: rows -> y, z -> sum over the group's pairs of w1 Re^2 + w2 Im^2 in
// FP64 registers, into the group's grid in lane order (part + grp * stride).
template <typename T, int A, int B>
__global__ void __launch_bounds__((64 * YzShape<T, A, B>::WR), (YzShape<T, A, B>::EUR))
    k_yz_rho(PassGeom g, const typename cplx_of<T>::type* __restrict__ W1, YzCols cols, const int4* __restrict__ tab,
             double* __restrict__ part, size_t stride, int npairs, const double* __restrict__ wpair, int accumulate,
             const typename cplx_of<T>::type* __restrict__ twg, int ngrp, int per) {
  using S = YzShape<T, A, B>;
  using V = typename S::V;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  int xh, grp;
  if (!z_block_of(ngrp, per, g.n1 * S::ZS, xh, grp)) return;
  const int x = xh / S::ZS, g0 = (xh - x * S::ZS) * S::GH, g1 = min(S::GZ, g0 + S::GH);
  YzBlock<T, A, B, S::WR> b(smem_raw, g, tab, twg);
  const int ppg = (npairs + ngrp - 1) / ngrp, pa = grp * ppg, pb = min(npairs, pa + ppg);
  double acc[S::NRH][A];
#pragma unroll
  for (int n = 0; n < S::NRH; ++n)
#pragma unroll
    for (int j = 0; j < A; ++j) acc[n][j] = 0.0;
  auto rows_of = [&](int pl) {
    return PencilBuf<V>(W1 + ((size_t)pl * g.n1 + x) * cols.pitch, cols.pitch * (unsigned)sizeof(V));
  };
  for (int pl = pa; pl < pb; ++pl) {
    b.y_inverse(rows_of(pl));
    __syncthreads();
    const double w1 = wpair[2 * pl], w2 = wpair[2 * pl + 1];
#pragma unroll
    for (int n = 0; n < S::NRH; ++n) {
      const int gz = g0 + b.wave + n * S::WR;
      if (gz >= g1) continue;  // uniform over the wave
      V r[S::TM];
      b.z_inverse(gz * S::CPW + b.c, r);
#pragma unroll
      for (int j = 0; j < A; ++j) {
        const double re = (double)r[j].x, im = (double)r[j].y;
        acc[n][j] += w1 * re * re + w2 * im * im;
      }
    }
    __syncthreads();  // the planes are read before the next pair's are written
  }
  double* out = part + grp * stride + (size_t)x * S::GZ * A * 64 + (threadIdx.x & 63);
#pragma unroll
  for (int n = 0; n < S::NRH; ++n) {
    const int gz = g0 + b.wave + n * S::WR;
    if (gz >= g1) continue;
#pragma unroll
    for (int j = 0; j < A; ++j) {
      double* o = out + (size_t)(gz * A + j) * 64;
      *o = accumulate ? *o + acc[n][j] : acc[n][j];
    }
  }
}

// Between lane order and the x-fastest grid, in tiles of 16 x by the 64 lanes
// of one (z group, j): lane l of column c = l / TM holds y = gz CPW + c,
// z = l % TM + B j (t < B).
struct YzOrder {
  int n1, N, A, B, TM, CPW, GZ;
};
__device__ __forceinline__ bool yz_place(const YzOrder& o, int gz, int j, int lane, int& y, int& z) {
  const int c = lane / o.TM, t = lane - c * o.TM;
  y = gz * o.CPW + c;
  z = t + o.B * j;
  return c < o.CPW && t < o.B && y < o.N;
}

// rho = sum over the ngrp lane-order grids (fixed order); part8: RED_BLOCKS
// partial sums of the grid.  256 threads, RED_BLOCKS blocks.
__global__ void __launch_bounds__(256) k_yz_rho_combine(YzOrder o, const double* __restrict__ part, size_t stride,
                                                        int ngrp, double* __restrict__ rho, double* __restrict__ part8) {
  __shared__ double tile[64][17];
  __shared__ double sh[4];
  const int nxt = (o.n1 + 15) / 16, ntile = nxt * o.GZ * o.A;
  double s = 0.0;
  for (int q = blockIdx.x; q < ntile; q += gridDim.x) {
    const int xt = q % nxt, j = (q / nxt) % o.A, gz = q / (nxt * o.A);
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int xi = (threadIdx.x >> 6) + 4 * i, x = xt * 16 + xi;
      double v = 0.0;
      if (x < o.n1) {
        const double* p = part + ((size_t)(x * o.GZ + gz) * o.A + j) * 64 + lane;
        for (int k = 0; k < ngrp; k += 4) {  // four loads in flight per sum
          double u[4];
#pragma unroll
          for (int m = 0; m < 4; ++m) u[m] = k + m < ngrp ? p[(k + m) * stride] : 0.0;
#pragma unroll
          for (int m = 0; m < 4; ++m) v += u[m];
        }
      }
      tile[lane][xi] = v;
    }
    __syncthreads();
    const int xi = threadIdx.x & 15, x = xt * 16 + xi;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int l = (threadIdx.x >> 4) + 16 * i;
      int y, z;
      if (yz_place(o, gz, j, l, y, z) && x < o.n1) {
        const double v = tile[l][xi];
        rho[((size_t)z * o.N + y) * o.n1 + x] = v;
        s += v;
      }
    }
    __syncthreads();
  }
  s = block_sum(s, sh);
  if (threadIdx.x == 0) part8[blockIdx.x] = s;
}

// vn = scale * v in lane order (0 in lanes without a grid point)
template <typename S, typename T>
__global__ void __launch_bounds__(256) k_yz_potential(YzOrder o, const S* __restrict__ v, double scale,
                                                      T* __restrict__ vn) {
  __shared__ double tile[64][17];
  const int nxt = (o.n1 + 15) / 16, ntile = nxt * o.GZ * o.A;
  for (int q = blockIdx.x; q < ntile; q += gridDim.x) {
    const int xt = q % nxt, j = (q / nxt) % o.A, gz = q / (nxt * o.A);
    {
      const int xi = threadIdx.x & 15, x = xt * 16 + xi;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int l = (threadIdx.x >> 4) + 16 * i;
        int y, z;
        tile[l][xi] = yz_place(o, gz, j, l, y, z) && x < o.n1 ? (double)v[((size_t)z * o.N + y) * o.n1 + x] : 0.0;
      }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int xi = (threadIdx.x >> 6) + 4 * i, x = xt * 16 + xi;
      if (x < o.n1) vn[((size_t)(x * o.GZ + gz) * o.A + j) * 64 + lane] = (T)(scale * tile[lane][xi]);
    }
    __syncthreads();
  }
}

// x pass inverse into the transposed W1 (otherwise as k_rows_inv_r): the block's
// HR direct rows, and its HR mirror rows, fall on consecutive slots, so each x
// gets two runs of HR values.
template <typename T, int A, int B, int HR>
__global__ void __launch_bounds__(2 * HR * (A > B ? A : B))
    k_rows_inv_t(PassGeom g, const double2* __restrict__ C, int ldc, int nb, int pair0,
                 typename cplx_of<T>::type* __restrict__ W1, YzCols cols,
                 const typename cplx_of<T>::type* __restrict__ twg) {
  using V = typename cplx_of<T>::type;
  constexpr int N = A * B, TM = MaxAB<A, B>::v, ST = N + 1, NT = 2 * HR * TM;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  V* tw = reinterpret_cast<V*>(smem_raw);
  V* lds = tw + N;
  __shared__ int slot_s[2 * HR];  // positions of the HR direct, then of the HR mirror rows; -1: none
  const int t = threadIdx.x % TM, fr = threadIdx.x / TM;  // transform: HR direct rows, then HR mirror rows
  const int mirror = fr >= HR, row = blockIdx.x * HR + (mirror ? fr - HR : fr);
  const int pl = blockIdx.y, ba = 2 * (pair0 + pl);
  for (int i = threadIdx.x; i < N; i += NT) tw[i] = twg[i];
  RowInfo ri{};
  const bool live = row < g.nrow;
  if (live) ri = g.rows[row];
  const bool zero_row = live && ri.slot_m < 0;  // (0, 0): both halves on the direct row
  if (t == 0) slot_s[fr] = live && !(zero_row && mirror) ? cols.at(mirror ? ri.slot_m : ri.slot_d) : -1;
  // both bands' half rows as bounded buffers: nothing past the end of the
  // band array, nothing at all of a missing second band
  const PencilBuf<double2> c1(C + (size_t)ba * ldc, ldc * (unsigned)sizeof(double2));
  const PencilBuf<double2> c2(C + (size_t)(ba + 1 < nb ? ba + 1 : ba) * ldc,
                              ba + 1 < nb ? ldc * (unsigned)sizeof(double2) : 0u);
  const int cnt = live && t < A && !(zero_row && mirror) ? ri.cnt : 0;
  V r[TM];
#pragma unroll
  for (int k = 0; k < B; ++k) {
    const int m1 = signed_freq(t + A * k, N);
    const bool cj = mirror || (zero_row && m1 < 0);  // held as the conjugate of -m1
    const int e = (cj ? -m1 : m1) - ri.m1_0;
    const unsigned off = (unsigned)e < (unsigned)cnt ? (unsigned)((ri.start + e) * sizeof(double2)) : DEAD_OFF;
    const double2 s1 = c1.load(off), s2 = c2.load(off);
    r[k].x = (T)(cj ? s1.x + s2.y : s1.x - s2.y);
    r[k].y = (T)(cj ? s2.x - s1.y : s1.y + s2.x);
  }
  __syncthreads();
  col_fft<V, A, B, +1>(r, t, lds, 1, fr * ST, tw);
  if (t < B)
#pragma unroll
    for (int j = 0; j < A; ++j) lds[fr * ST + t + B * j] = r[j];
  __syncthreads();
  V* out = W1 + (size_t)pl * N * cols.pitch;
  for (int i = threadIdx.x; i < 2 * HR * N; i += NT) {
    const int x = i / (2 * HR), s = i % (2 * HR), slot = slot_s[s];
    if (slot >= 0) out[(size_t)x * cols.pitch + slot] = lds[s * ST + x];
  }
}

// x pass forward of H|psi> from the transposed W1 (otherwise as
// k_rows_fwd_hpsi_r).  The band coefficients of a thread's outputs are all
// requested before the first is used; requested before the transform already,
// they took the registers of two waves per SIMD (144^3 FP32, 256 bands: 0.27
// against 0.25 ms).
template <typename T, int A, int B, int HR>
__global__ void __launch_bounds__(2 * HR * (A > B ? A : B))
    k_rows_fwd_hpsi_t(PassGeom g, const typename cplx_of<T>::type* __restrict__ W1, YzCols cols,
                      const double2* __restrict__ C, double2* __restrict__ C2, int ldc, int nb, int pair0,
                      const double* __restrict__ occ, Recip rc, const typename cplx_of<T>::type* __restrict__ twg) {
  using V = typename cplx_of<T>::type;
  constexpr int N = A * B, TM = MaxAB<A, B>::v, ST = N + 1, NT = 2 * HR * TM;
  constexpr int NP = (N / 2 + 2 * TM) / (2 * TM);  // elements per thread of a row of at most N/2 + 1
  extern __shared__ __align__(16) unsigned char smem_raw[];
  V* tw = reinterpret_cast<V*>(smem_raw);
  V* lds = tw + N;
  __shared__ int slot_s[2 * HR];
  const int t = threadIdx.x % TM, fr = threadIdx.x / TM;
  const int mirror = fr >= HR, hr = mirror ? fr - HR : fr, row = blockIdx.x * HR + hr;
  const int pl = blockIdx.y, ba = 2 * (pair0 + pl), bb = ba + 1;
  const bool has2 = bb < nb, live = row < g.nrow;
  for (int i = threadIdx.x; i < N; i += NT) tw[i] = twg[i];
  RowInfo ri{};
  if (live) ri = g.rows[row];
  const bool zero_row = live && ri.slot_m < 0;
  if (t == 0) slot_s[fr] = live && !(zero_row && mirror) ? cols.at(mirror ? ri.slot_m : ri.slot_d) : -1;
  __syncthreads();
  const V* in = W1 + (size_t)pl * N * cols.pitch;
  for (int i = threadIdx.x; i < 2 * HR * N; i += NT) {
    const int x = i / (2 * HR), s = i % (2 * HR), slot = slot_s[s];
    V v;
    v.x = v.y = 0;
    if (slot >= 0) v = in[(size_t)x * cols.pitch + slot];
    lds[s * ST + x] = v;
  }
  __syncthreads();
  V r[TM];
  const int ta = t < A ? t : 0;
#pragma unroll
  for (int k = 0; k < B; ++k) r[k] = lds[fr * ST + ta + A * k];
  __syncthreads();
  col_fft<V, A, B, -1>(r, t, lds, 1, fr * ST, tw);
  if (t < B)
#pragma unroll
    for (int j = 0; j < A; ++j) lds[fr * ST + t + B * j] = r[j];
  __syncthreads();
  const PencilBuf<double2> c1(C + (size_t)ba * ldc, ldc * (unsigned)sizeof(double2));
  const PencilBuf<double2> c2(C + (size_t)(has2 ? bb : ba) * ldc, has2 ? ldc * (unsigned)sizeof(double2) : 0u);
  const int e0 = t + mirror * TM;  // the 2 TM threads of half row hr walk its elements
  double2 p1[NP], p2[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int e = e0 + 2 * TM * i;
    const unsigned off = live && e < ri.cnt ? (unsigned)((ri.start + e) * sizeof(double2)) : DEAD_OFF;
    p1[i] = c1.load(off);
    p2[i] = c2.load(off);
  }
  if (!live) return;
  double fa = occ[ba] * 0.5;
  if (fa == 0.0) fa = 1.0;
  double fb = has2 ? occ[bb] * 0.5 : 1.0;
  if (fb == 0.0) fb = 1.0;
  const V* rd = lds + hr * ST;
  const V* rm = zero_row ? rd : lds + (HR + hr) * ST;
  const double gy0 = ri.m2 * rc.g[3] + ri.m3 * rc.g[6];
  const double gy1 = ri.m2 * rc.g[4] + ri.m3 * rc.g[7];
  const double gy2 = ri.m2 * rc.g[5] + ri.m3 * rc.g[8];
  auto put = [&](int e, double2 ca, double2 cb) {
    const int m1 = ri.m1_0 + e;
    const double gx = m1 * rc.g[0] + gy0, gyv = m1 * rc.g[1] + gy1, gz = m1 * rc.g[2] + gy2;
    const double gg = gx * gx + gyv * gyv + gz * gz;
    const V Av = rd[wrap(m1, N)];
    const V Bv = rm[wrap(-m1, N)];
    const double fpx = (double)Av.x + (double)Bv.x, fpy = (double)Av.y + (double)Bv.y;
    const double fmx = (double)Av.x - (double)Bv.x, fmy = (double)Av.y - (double)Bv.y;
    C2[(size_t)ba * ldc + ri.start + e] = make_double2(-fa * (gg * ca.x + fpx), -fa * (gg * ca.y + fmy));
    if (has2) C2[(size_t)bb * ldc + ri.start + e] = make_double2(-fb * (gg * cb.x + fpy), -fb * (gg * cb.y - fmx));
  };
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (e0 + 2 * TM * i < ri.cnt) put(e0 + 2 * TM * i, p1[i], p2[i]);
  for (int e = e0 + 2 * TM * NP; e < ri.cnt; e += 2 * TM)  // rows wider than half the grid
    put(e, C[(size_t)ba * ldc + ri.start + e], has2 ? C[(size_t)bb * ldc + ri.start + e] : make_double2(0.0, 0.0));
}

}  // namespace amdk
