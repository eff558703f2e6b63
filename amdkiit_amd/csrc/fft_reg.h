// Register-resident pencil FFT passes for lengths N = A*B (A, B <= 18).
//
// One transform of length N is spread over max(A, B) threads: each thread
// first does a length-B DFT in registers over elements t + A*k2, multiplies
// the twiddle W_N^{t*j2}, one LDS exchange transposes, and each thread then
// does a length-A DFT that yields the outputs t + B*j1.  The same identity
// with A and B swapped continues from exactly those registers, so a forward
// transform after a pointwise product (V(r) psi(r)) needs no reordering:
// inverse FFT -> V -> forward FFT costs two LDS exchanges per column.
//
// Compared with the LDS Stockham passes of fft_passes.h (one LDS round trip
// and one barrier per radix stage) this keeps every butterfly in VGPRs and
// touches LDS twice per transform.  The Stockham passes remain the fallback
// for lengths without an (A, B) split here.
#pragma once
#include "fft_passes.h"
#include "twiddle_const.h"

namespace amdk {

template <int L> struct Split { static constexpr int P = 1, Q = L; };
template <> struct Split<6> { static constexpr int P = 2, Q = 3; };
template <> struct Split<8> { static constexpr int P = 2, Q = 4; };
template <> struct Split<9> { static constexpr int P = 3, Q = 3; };
template <> struct Split<10> { static constexpr int P = 2, Q = 5; };
template <> struct Split<12> { static constexpr int P = 3, Q = 4; };
template <> struct Split<15> { static constexpr int P = 3, Q = 5; };
template <> struct Split<16> { static constexpr int P = 4, Q = 4; };
template <> struct Split<18> { static constexpr int P = 2, Q = 9; };

constexpr int gcd_of(int a, int b) { return b == 0 ? a : gcd_of(b, a % b); }

// x exp(DIR 2 pi i m / L), quarter turns without products
template <int L, int DIR, typename V>
__device__ __forceinline__ V mul_root(V a, int m) {
  using T = decltype(a.x);
  V r;
  if (m == 0) return a;
  if (2 * m == L) { r.x = -a.x; r.y = -a.y; return r; }
  if (4 * m == L) return mul_si<DIR>(a);
  if (4 * m == 3 * L) return mul_si<-DIR>(a);
  V w;
  w.x = (T)Tw<L>::re[m];
  w.y = (T)(DIR < 0 ? Tw<L>::im[m] : -Tw<L>::im[m]);
  return cmul(a, w);
}

// In-register DFT of x[0..L): X_k = sum_j x_j exp(DIR 2 pi i jk / L).
// L = P Q with coprime P, Q (6, 10, 12, 15, 18) takes the prime-factor map
// j = Q a + P b (mod L), k -> (k mod P, k mod Q), which needs no twiddle
// between the P- and the Q-point DFTs; 8, 9 and 16 keep the twiddled split.
// Against the twiddled split at every length the z pass of H|psi> issues 10 %
// fewer vector instructions and rounds less (FP32 H|psi> at 100^3 against 64
// bits: 1.05e-8 -> 8.2e-9): z_vpsi 0.172 -> 0.168 ms at 32 H2O, 0.817 ->
// 0.797 ms at 64 H2O.
// Z: bit j set says that x[j] is 0 (and not to be read); the sums and products
// with it are left out, which changes no result.
template <typename V, int L, int DIR, unsigned Z = 0> struct RDft {
  static constexpr int P = Split<L>::P, Q = Split<L>::Q;
  static constexpr bool PF = gcd_of(P, Q) == 1;
  static constexpr int in_of(int k1, int k2) { return PF ? (Q * k1 + P * k2) % L : k1 + P * k2; }
  static constexpr unsigned zeros_of(int k1) {  // of the Q-point DFT k1
    unsigned z = 0;
    for (int k2 = 0; k2 < Q; ++k2)
      if ((Z >> in_of(k1, k2)) & 1u) z |= 1u << k2;
    return z;
  }
  static constexpr unsigned zeros_outer() {  // Q-point DFTs that are 0
    unsigned z = 0;
    for (int k1 = 0; k1 < P; ++k1)
      if (zeros_of(k1) == (1u << Q) - 1u) z |= 1u << k1;
    return z;
  }
  template <int K1> __device__ static __forceinline__ void inner(const V* x, V* y) {
    if constexpr (K1 < P) {
      if constexpr (zeros_of(K1) != (1u << Q) - 1u) {
        V t[Q];
#pragma unroll
        for (int k2 = 0; k2 < Q; ++k2) t[k2] = x[in_of(K1, k2)];
        RDft<V, Q, DIR, zeros_of(K1)>::run(t);
#pragma unroll
        for (int j2 = 0; j2 < Q; ++j2) y[K1 * Q + j2] = PF ? t[j2] : mul_root<L, DIR>(t[j2], (j2 * K1) % L);
      }
      inner<K1 + 1>(x, y);
    }
  }
  __device__ static __forceinline__ void run(V* x) {
    if constexpr (L == 1) {
      return;
    } else if constexpr (L <= 5) {
      Butterfly<V, L, DIR, Z>::run(x);
    } else {
      static_assert(P * Q == L && P > 1, "no split for this DFT length");
      V y[L];
      inner<0>(x, y);
#pragma unroll
      for (int j2 = 0; j2 < Q; ++j2) {
        V u[P];
#pragma unroll
        for (int k1 = 0; k1 < P; ++k1) u[k1] = y[k1 * Q + j2];
        RDft<V, P, DIR, zeros_outer()>::run(u);
#pragma unroll
        for (int j1 = 0; j1 < P; ++j1) {
          if constexpr (PF) {
            // the k with k mod P = j1, k mod Q = j2
            int k = j2;
            while (k % P != j1) k += Q;
            x[k] = u[j1];
          } else {
            x[j2 + Q * j1] = u[j1];
          }
        }
      }
    }
  }
};

template <int A, int B> struct MaxAB { static constexpr int v = A > B ? A : B; };

// One length-N = A*B transform per "lane group" (column c of a tile).
// In:  thread t < A holds x[t + A*k2], k2 < B, in r[0..B).
// Out: thread t < B holds X[t + B*j1], j1 < A, in r[0..A).
// lds: A*B*stride elements; element (k1, j2) of column c at (k1*B + j2)*stride + c*cstride.
// twN[m] = exp(-2 pi i m / N).  Every thread of the block must call this.
// Z: inputs that are 0 in every thread, as in RDft.
template <typename V, int A, int B, int DIR, unsigned Z = 0>
__device__ __forceinline__ void col_fft(V* r, int t, V* lds, int stride, int coff, const V* twN) {
  if (t < A) {
    RDft<V, B, DIR, Z>::run(r);
#pragma unroll
    for (int j2 = 0; j2 < B; ++j2) {
      V v = r[j2];
      if (j2 > 0 && t > 0) {
        V w = twN[t * j2];
        if (DIR > 0) w.y = -w.y;
        v = cmul(v, w);
      }
      lds[(t * B + j2) * stride + coff] = v;
    }
  }
  __syncthreads();
  if (t < B) {
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) r[k1] = lds[(k1 * B + t) * stride + coff];
    RDft<V, A, DIR>::run(r);
  }
  __syncthreads();
}

__device__ __forceinline__ int signed_freq(int p, int n) { return 2 * p <= n ? p : p - n; }

// One pencil of planes (or of a plane's rows) as a bounded buffer: elements
// of V at unsigned byte offsets below `bytes` of the wave-uniform base.  The
// hardware returns 0 for a load past the end and drops a store there, so the
// sphere's edges need no compare, branch or mask: frequencies above the last
// stored one lie past the end, those below the first at negative offsets,
// which are past it as unsigned numbers, and a thread without a column starts
// at DEAD_OFF.  Buffers are below 2^31 - 2^27 bytes (grids up to 192^3: 113 MB).
// The masked accesses this replaced took a third of z_vpsi's vector
// instructions (891 -> 614 with the quarter window below) and its loads were
// parted by branches: z_vpsi 0.168 -> 0.132 ms at 32 H2O (FP64 0.277 ->
// 0.214), 0.80 -> 0.60 ms at 64 H2O; z_rho 0.094 -> 0.090 and 0.43 -> 0.39 ms.
// The y passes, bound by memory, gained nothing by it (0.072 -> 0.074 ms).
typedef unsigned uint2v __attribute__((ext_vector_type(2)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));
constexpr unsigned DEAD_OFF = 0x80000000u;

template <typename V> struct PencilBuf {
  __amdgpu_buffer_rsrc_t rs;
  __device__ __forceinline__ PencilBuf(const V* p, unsigned bytes)
      : rs(__builtin_amdgcn_make_buffer_rsrc(const_cast<V*>(p), 0, bytes, 0x00027000)) {}
  __device__ __forceinline__ V load(unsigned off) const {
    if constexpr (sizeof(V) == 8) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0));
    else return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
  }
  __device__ __forceinline__ void store(unsigned off, V v) const {
    if constexpr (sizeof(V) == 8) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2v, v), rs, off, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, v), rs, off, 0, 0);
  }
};

// Position t + A k of a length-N transform relative to position t, in steps
// of the pencil, with the upper half wrapped to negative frequencies.  Which
// half an element falls in is known at compile time except where the middle
// lies inside the run of A positions; N/2 itself is never stored, so either
// side does.
template <int A, int N>
__device__ __forceinline__ int pencil_step(int t, int k) {
  if (2 * A * k >= N) return A * k - N;
  if (2 * (A * k + A - 1) <= N) return A * k;
  return 2 * (t + A * k) > N ? A * k - N : A * k;
}

// Whether a run of positions t + A k, t < A, can hold a stored frequency.  The
// wavefunction sphere reaches at most a quarter of the grid (|m| <= N/4: the
// grid holds the density, whose sphere is twice as wide), and QW says that it
// does, so that the middle runs are left out at compile time: they are zeros
// to the transform and cost no access.  A run-time test per run, which would
// also skip what a particular plane lacks, measured slower (its branches part
// the loads; z_vpsi at 32 H2O 0.167 instead of 0.142 ms).
template <bool QW, int A, int N>
constexpr bool pencil_run(int k) {
  return !QW || 4 * A * k <= N || 4 * (N - A * k - A + 1) <= N;
}

// the runs that pencil_run leaves out, as the zeros of the length-B DFT over k
template <bool QW, int A, int B>
constexpr unsigned pencil_zeros() {
  unsigned z = 0;
  for (int k = 0; k < B; ++k)
    if (!pencil_run<QW, A, A * B>(k)) z |= 1u << k;
  return z;
}

// Block order of the z passes: MI355X hands consecutive workgroups
// round-robin to its 8 XCDs; physical block p runs logical block
// (p % 8) * per + p / 8, so each XCD walks one contiguous range of logical
// blocks L = cb * ngrp + grp (launch 8 * per blocks; ids past the last
// logical block return).  Returns false for those.
__device__ __forceinline__ bool z_block_of(int ngrp, int per, int ncb, int& cb, int& grp) {
  const int p = blockIdx.x;
  const int L = (p & 7) * per + (p >> 3);
  if (L >= ncb * ngrp) return false;
  cb = L / ngrp;
  grp = L - cb * ngrp;
  return true;
}

// ---------------------------------------------------------------------------
// z pass of H|psi>: planes |m3| <= R -> z-FFT exp(+i) -> * v(r) -> z-FFT exp(-i)
template <typename T, int A, int B, int TX, bool QW>
__global__ void __launch_bounds__(TX * (A > B ? A : B))
    k_z_vpsi_r(PassGeom g, typename cplx_of<T>::type* __restrict__ W2, const T* __restrict__ vr, int npairs,
               int PG, const typename cplx_of<T>::type* __restrict__ twg, int ngrp, int per) {
  using V = typename cplx_of<T>::type;
  constexpr int N = A * B, TM = MaxAB<A, B>::v;
  extern __shared__ unsigned char smem_raw[];
  V* tw = reinterpret_cast<V*>(smem_raw);
  V* lds = tw + N;
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const int n1 = g.n1, n2 = g.n2;
  // logical block (column block, pair group), group fastest, walked
  // XCD-contiguously (z_block_of): a V(r) tile's pair groups and the
  // neighbouring column blocks, which share the 128-byte lines at their
  // edges, run on one XCD and share its L2
  int cb, grp;
  if (!z_block_of(ngrp, per, (n1 * n2 + TX - 1) / TX, cb, grp)) return;
  // columns of the n1 x n2 plane in x-fastest order, TX consecutive per block
  const int q = cb * TX + c;
  const bool live = q < n1 * n2;
  const int y = live ? q / n1 : 0, x = q - y * n1;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twg[i];
  T vv[A];
#pragma unroll
  for (int j1 = 0; j1 < A; ++j1) {
    const int z = t + B * j1;
    vv[j1] = (live && t < B) ? vr[((size_t)z * n2 + y) * n1 + x] : (T)0;
  }
  __syncthreads();
  const int pg0 = grp * PG, pg1 = min(npairs, pg0 + PG);
  const int ps = n2 * g.p1, psb = ps * sizeof(V);  // plane stride; plane kz sits at kz + R
  const unsigned base = t < A && live ? (t + g.R) * psb + (y * g.p1 + x) * (unsigned)sizeof(V) : DEAD_OFF;
  for (int pl = pg0; pl < pg1; ++pl) {
    const PencilBuf<V> buf(W2 + (size_t)pl * g.nplane * ps, g.nplane * psb);
    V r[TM];
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) {
      if (pencil_run<QW, A, N>(k2)) r[k2] = buf.load(base + pencil_step<A, N>(t, k2) * psb);
      else r[k2].x = r[k2].y = 0;
    }
    col_fft<V, A, B, +1, pencil_zeros<QW, A, B>()>(r, t, lds, TX, c, tw);
    if (t < B) {
#pragma unroll
      for (int j1 = 0; j1 < A; ++j1) {
        r[j1].x *= vv[j1];
        r[j1].y *= vv[j1];
      }
    }
    col_fft<V, B, A, -1>(r, t, lds, TX, c, tw);
#pragma unroll
    for (int j1 = 0; j1 < B; ++j1)
      if (pencil_run<QW, A, N>(j1)) buf.store(base + pencil_step<A, N>(t, j1) * psb, r[j1]);
  }
}

// z pass of the density: z-FFT exp(+i) of every pair, rho += w1 Re^2 + w2 Im^2
// in FP64 registers (each thread owns fixed z), ordered over pairs.  The
// pairs are split into gridDim.z consecutive groups; group k accumulates
// into the grid rho + k * part_stride (summed afterwards in a fixed order).
template <typename T, int A, int B, int TX, bool QW>
__global__ void __launch_bounds__(TX * (A > B ? A : B))
    k_z_rho_r(PassGeom g, const typename cplx_of<T>::type* __restrict__ W2, double* __restrict__ rho, int npairs,
              const double* __restrict__ wpair, int accumulate, const typename cplx_of<T>::type* __restrict__ twg,
              size_t part_stride, int ngrp, int per) {
  using V = typename cplx_of<T>::type;
  constexpr int N = A * B, TM = MaxAB<A, B>::v;
  extern __shared__ unsigned char smem_raw[];
  V* tw = reinterpret_cast<V*>(smem_raw);
  V* lds = tw + N;
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const int n1 = g.n1, n2 = g.n2;
  int cb, grp;  // (column block, pair group), XCD-contiguous as in k_z_vpsi_r
  if (!z_block_of(ngrp, per, (n1 * n2 + TX - 1) / TX, cb, grp)) return;
  const int q = cb * TX + c;  // plane column, x fastest (as in k_z_vpsi_r)
  const bool live = q < n1 * n2;
  const int y = live ? q / n1 : 0, x = q - y * n1;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twg[i];
  __syncthreads();
  double acc[A];
#pragma unroll
  for (int j1 = 0; j1 < A; ++j1) acc[j1] = 0.0;
  // FP32 with <= 10 values per thread: the next pair's planes are loaded into
  // registers while this one is transformed (wider forms would lose occupancy)
  constexpr bool PF = sizeof(T) == 4 && TM <= 10;
  V rn[B];
  const int ps = n2 * g.p1, psb = ps * sizeof(V);  // plane stride; plane kz sits at kz + R
  const unsigned base = t < A && live ? (t + g.R) * psb + (y * g.p1 + x) * (unsigned)sizeof(V) : DEAD_OFF;
  auto load_pair = [&](int pl, V* dst) {
    const PencilBuf<V> buf(W2 + (size_t)pl * g.nplane * ps, g.nplane * psb);
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) {
      if (pencil_run<QW, A, N>(k2)) dst[k2] = buf.load(base + pencil_step<A, N>(t, k2) * psb);
      else dst[k2].x = dst[k2].y = 0;
    }
  };
  const int ppg = (npairs + ngrp - 1) / ngrp;
  const int pa = grp * ppg, pb = min(npairs, pa + ppg);
  rho += grp * part_stride;
  if (PF && pa < pb) load_pair(pa, rn);
  for (int pl = pa; pl < pb; ++pl) {
    V r[TM];
    if constexpr (PF) {
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) r[k2] = rn[k2];
      if (pl + 1 < pb) load_pair(pl + 1, rn);
    } else {
      load_pair(pl, r);
    }
    col_fft<V, A, B, +1, pencil_zeros<QW, A, B>()>(r, t, lds, TX, c, tw);
    const double w1 = wpair[2 * pl], w2 = wpair[2 * pl + 1];
#pragma unroll
    for (int j1 = 0; j1 < A; ++j1) {
      const double re = (double)r[j1].x, im = (double)r[j1].y;
      acc[j1] += w1 * re * re + w2 * im * im;
    }
  }
  if (t < B && live) {
#pragma unroll
    for (int j1 = 0; j1 < A; ++j1) {
      const int z = t + B * j1;
      double* dst = rho + ((size_t)z * n2 + y) * n1 + x;
      *dst = accumulate ? (*dst + acc[j1]) : acc[j1];
    }
  }
}

// y pass inverse: rows of plane m3 (consecutive m2 from m2_lo) -> y-FFT exp(+i)
template <typename T, int A, int B, int TX, bool QW>
__global__ void __launch_bounds__(TX * (A > B ? A : B))
    k_cols_inv_r(PassGeom g, const typename cplx_of<T>::type* __restrict__ W1, typename cplx_of<T>::type* __restrict__ W2,
                 const typename cplx_of<T>::type* __restrict__ twg) {
  using V = typename cplx_of<T>::type;
  constexpr int N = A * B, TM = MaxAB<A, B>::v;
  extern __shared__ unsigned char smem_raw[];
  V* tw = reinterpret_cast<V*>(smem_raw);
  V* lds = tw + N;
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const int n1 = g.n1, n2 = g.n2;
  const int x = blockIdx.x * TX + c;
  const int plane = blockIdx.y, pl = blockIdx.z;
  const bool live = x < n1;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twg[i];
  const int s0 = g.plane_off[plane], s1 = g.plane_off[plane + 1];
  const int lo = s1 > s0 ? g.slot_m2[s0] : 0;
  __syncthreads();
  V r[TM];
  const int psb = g.p1 * sizeof(V);
  const PencilBuf<V> rows(W1 + ((size_t)pl * g.nslot + s0) * g.p1, (s1 - s0) * psb);  // rows m2 = lo, lo + 1, ...
  const unsigned base = t < A && live ? (t - lo) * psb + x * (unsigned)sizeof(V) : DEAD_OFF;
#pragma unroll
  for (int k2 = 0; k2 < B; ++k2) {
    if (pencil_run<QW, A, N>(k2)) r[k2] = rows.load(base + pencil_step<A, N>(t, k2) * psb);
    else r[k2].x = r[k2].y = 0;
  }
  col_fft<V, A, B, +1, pencil_zeros<QW, A, B>()>(r, t, lds, TX, c, tw);
  if (t < B && live) {
    V* out = W2 + ((size_t)pl * g.nplane + plane) * (size_t)n2 * g.p1 + (size_t)t * g.p1 + x;
#pragma unroll
    for (int j1 = 0; j1 < A; ++j1) out[(B * j1) * g.p1] = r[j1];
  }
}

// y pass forward: full plane column -> y-FFT exp(-i) -> rows inside the sphere
template <typename T, int A, int B, int TX, bool QW>
__global__ void __launch_bounds__(TX * (A > B ? A : B))
    k_cols_fwd_r(PassGeom g, const typename cplx_of<T>::type* __restrict__ W2, typename cplx_of<T>::type* __restrict__ W1,
                 const typename cplx_of<T>::type* __restrict__ twg) {
  using V = typename cplx_of<T>::type;
  constexpr int N = A * B, TM = MaxAB<A, B>::v;
  extern __shared__ unsigned char smem_raw[];
  V* tw = reinterpret_cast<V*>(smem_raw);
  V* lds = tw + N;
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const int n1 = g.n1, n2 = g.n2;
  const int x = blockIdx.x * TX + c;
  const int plane = blockIdx.y, pl = blockIdx.z;
  const bool live = x < n1;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twg[i];
  const int s0 = g.plane_off[plane], s1 = g.plane_off[plane + 1];
  const int lo = s1 > s0 ? g.slot_m2[s0] : 0;
  __syncthreads();
  V r[TM];
#pragma unroll
  for (int k = 0; k < TM; ++k) { r[k].x = 0; r[k].y = 0; }
  const V* in = W2 + ((size_t)pl * g.nplane + plane) * (size_t)n2 * g.p1 + (size_t)t * g.p1 + x;
  if (t < A && live) {
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) r[k2] = in[(A * k2) * g.p1];
  }
  col_fft<V, A, B, -1>(r, t, lds, TX, c, tw);
  const int psb = g.p1 * sizeof(V);
  const PencilBuf<V> rows(W1 + ((size_t)pl * g.nslot + s0) * g.p1, (s1 - s0) * psb);  // rows m2 = lo, lo + 1, ...
  const unsigned base = t < B && live ? (t - lo) * psb + x * (unsigned)sizeof(V) : DEAD_OFF;
#pragma unroll
  for (int j1 = 0; j1 < A; ++j1)
    if (pencil_run<QW, B, N>(j1)) rows.store(base + pencil_step<B, N>(t, j1) * psb, r[j1]);
}

// x pass inverse: gather half rows of two bands, pack psi1 + i psi2 on the
// direct row and conj(psi1) + i conj(psi2) on the mirror row, x-FFT exp(+i).
// Block: HR half rows -> 2*HR transforms, TM threads each (t fastest).
template <typename T, int A, int B, int HR>
__global__ void __launch_bounds__(2 * HR * (A > B ? A : B))
    k_rows_inv_r(PassGeom g, const double2* __restrict__ C, int ldc, int nb, int pair0,
                 typename cplx_of<T>::type* __restrict__ W1, const typename cplx_of<T>::type* __restrict__ twg) {
  using V = typename cplx_of<T>::type;
  constexpr int N = A * B, TM = MaxAB<A, B>::v, ST = N + 1;
  extern __shared__ unsigned char smem_raw[];
  V* tw = reinterpret_cast<V*>(smem_raw);
  V* lds = tw + N;
  const int t = threadIdx.x % TM, fr = threadIdx.x / TM;  // transform index in block
  const int hr = fr >> 1, mirror = fr & 1;
  const int row = blockIdx.x * HR + hr;
  const int pl = blockIdx.y, pair = pair0 + pl;
  const int ba = 2 * pair, bb = 2 * pair + 1;
  const bool has2 = bb < nb;
  const bool live = row < g.nrow;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twg[i];
  RowInfo ri{};
  if (live) ri = g.rows[row];
  const bool zero_row = live && ri.slot_m < 0;  // (0,0): both halves on the direct row
  __syncthreads();
  V r[TM];
#pragma unroll
  for (int k = 0; k < TM; ++k) { r[k].x = 0; r[k].y = 0; }
  if (live && t < A && !(zero_row && mirror)) {
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) {
      const int m1 = signed_freq(t + A * k2, N);
      const bool direct_ok = !mirror && m1 >= ri.m1_0 && m1 < ri.m1_0 + ri.cnt;
      const int mm = -m1;
      const bool mirror_ok = (mirror || (zero_row && m1 < 0)) && mm >= ri.m1_0 && mm < ri.m1_0 + ri.cnt;
      if (direct_ok || mirror_ok) {
        const int e = (direct_ok ? m1 : mm) - ri.m1_0;
        const double2 s1 = C[(size_t)ba * ldc + ri.start + e];
        double2 s2 = make_double2(0.0, 0.0);
        if (has2) s2 = C[(size_t)bb * ldc + ri.start + e];
        V v;
        if (direct_ok) {
          v.x = (T)(s1.x - s2.y);
          v.y = (T)(s1.y + s2.x);
        } else {
          v.x = (T)(s1.x + s2.y);
          v.y = (T)(s2.x - s1.y);
        }
        r[k2] = v;
      }
    }
  }
  col_fft<V, A, B, +1>(r, t, lds, 1, fr * ST, tw);
  if (live && t < B && !(zero_row && mirror)) {
    const int slot = mirror ? ri.slot_m : ri.slot_d;
    V* out = W1 + ((size_t)pl * g.nslot + slot) * g.p1;
#pragma unroll
    for (int j1 = 0; j1 < A; ++j1) out[t + B * j1] = r[j1];
  }
}

// x pass forward of H|psi>: x-FFT exp(-i) of the direct and mirror rows, then
// unpack the two bands and write C2 = -(f/2)(|G|^2 c + 2 (V psi)(G)) in FP64.
template <typename T, int A, int B, int HR>
__global__ void __launch_bounds__(2 * HR * (A > B ? A : B))
    k_rows_fwd_hpsi_r(PassGeom g, const typename cplx_of<T>::type* __restrict__ W1, const double2* __restrict__ C,
                      double2* __restrict__ C2, int ldc, int nb, int pair0, const double* __restrict__ occ, Recip rc,
                      const typename cplx_of<T>::type* __restrict__ twg) {
  using V = typename cplx_of<T>::type;
  constexpr int N = A * B, TM = MaxAB<A, B>::v, ST = N + 1;
  extern __shared__ unsigned char smem_raw[];
  V* tw = reinterpret_cast<V*>(smem_raw);
  V* lds = tw + N;
  const int t = threadIdx.x % TM, fr = threadIdx.x / TM;
  const int hr = fr >> 1, mirror = fr & 1;
  const int row = blockIdx.x * HR + hr;
  const int pl = blockIdx.y, pair = pair0 + pl;
  const int ba = 2 * pair, bb = 2 * pair + 1;
  const bool has2 = bb < nb;
  const bool live = row < g.nrow;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twg[i];
  RowInfo ri{};
  if (live) ri = g.rows[row];
  const bool zero_row = live && ri.slot_m < 0;
  __syncthreads();
  V r[TM];
#pragma unroll
  for (int k = 0; k < TM; ++k) { r[k].x = 0; r[k].y = 0; }
  if (live && t < A && !(zero_row && mirror)) {
    const V* in = W1 + ((size_t)pl * g.nslot + (mirror ? ri.slot_m : ri.slot_d)) * g.p1;
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) r[k2] = in[t + A * k2];
  }
  col_fft<V, A, B, -1>(r, t, lds, 1, fr * ST, tw);
  // outputs X[t + B*j1] of every transform -> LDS (same buffer, after the barrier)
  if (t < B) {
#pragma unroll
    for (int j1 = 0; j1 < A; ++j1) lds[fr * ST + t + B * j1] = r[j1];
  }
  __syncthreads();
  double fa = occ[ba] * 0.5;
  if (fa == 0.0) fa = 1.0;
  double fb = has2 ? occ[bb] * 0.5 : 1.0;
  if (fb == 0.0) fb = 1.0;
  // unpack: the 2*TM threads of half row hr walk its elements
  if (live) {
    const V* rd = lds + (2 * hr) * ST;
    const V* rm = zero_row ? rd : rd + ST;
    const double gy0 = ri.m2 * rc.g[3] + ri.m3 * rc.g[6];
    const double gy1 = ri.m2 * rc.g[4] + ri.m3 * rc.g[7];
    const double gy2 = ri.m2 * rc.g[5] + ri.m3 * rc.g[8];
    for (int e = t + mirror * TM; e < ri.cnt; e += 2 * TM) {
      const int m1 = ri.m1_0 + e;
      const double gx = m1 * rc.g[0] + gy0, gyv = m1 * rc.g[1] + gy1, gz = m1 * rc.g[2] + gy2;
      const double gg = gx * gx + gyv * gyv + gz * gz;
      const V Av = rd[wrap(m1, N)];
      const V Bv = rm[wrap(-m1, N)];
      const double fpx = (double)Av.x + (double)Bv.x, fpy = (double)Av.y + (double)Bv.y;
      const double fmx = (double)Av.x - (double)Bv.x, fmy = (double)Av.y - (double)Bv.y;
      const size_t ia = (size_t)ba * ldc + ri.start + e;
      const double2 c1 = C[ia];
      C2[ia] = make_double2(-fa * (gg * c1.x + fpx), -fa * (gg * c1.y + fmy));
      if (has2) {
        const size_t ib = (size_t)bb * ldc + ri.start + e;
        const double2 c2 = C[ib];
        C2[ib] = make_double2(-fb * (gg * c2.x + fpy), -fb * (gg * c2.y - fmx));
      }
    }
  }
}

// Up to two field pairs per launch of the dense transforms (blockIdx.z / .y
// selects the pair; work arrays W1/W2 hold one pair after the other).
struct DenseIn {
  const double* a[2];
  const double* b[2];
};
template <typename T>
struct DenseOut {
  double* a[2];
  double* b[2];
  T* v[2];
};


// ---------------------------------------------------------------------------
// Dense (density-sphere) passes in FP64: two real fields travel as a + i b.  A
// single real field (an LDA's rho and v_xc into G space, V_KS out of it) is its
// own Hermitian half: only the planes m3 = 0 .. R exist (g.nplane = R + 1), the y passes see
// no others, the x passes transform each row of them once
// (k_rows_inv_one_r, k_rows_fwd_one_r), and the last z pass takes plane -m3
// as conj of plane m3.  These launches are bound by latency on small grids and
// by memory on large ones.  The two transforms into G space of an LDA V_KS
// 0.054 -> 0.042 ms at 100^3 and 0.091 -> 0.067 at 144^3, the one out of it 0.028
// -> 0.024 and 0.046 -> 0.038.

// z-FFT exp(-i) of full columns of a(r) + i b(r); keep planes |m3| <= R, or
// 0 .. R of a single field.
template <int A, int B, int TX>
__global__ void __launch_bounds__(TX * (A > B ? A : B))
    k_z_fwd_dense_r(PassGeom g, DenseIn in, double2* __restrict__ W2, const double2* __restrict__ twg, int nf,
                    int per) {
  constexpr int N = A * B, TM = MaxAB<A, B>::v;
  extern __shared__ unsigned char smem_raw[];
  double2* tw = reinterpret_cast<double2*>(smem_raw);
  double2* lds = tw + N;
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const int n1 = g.n1, n2 = g.n2;
  int cb, f;  // (column block, field pair f), XCD-contiguous as in k_z_vpsi_r
  if (!z_block_of(nf, per, (n1 * n2 + TX - 1) / TX, cb, f)) return;
  const int q = cb * TX + c;  // plane column, x fastest
  const bool live = q < n1 * n2;
  const int y = live ? q / n1 : 0, x = q - y * n1;
  const double* __restrict__ a = in.a[f];
  const double* __restrict__ b = in.b[f];
  W2 += (size_t)f * g.nplane * g.n2 * g.p1;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twg[i];
  __syncthreads();
  const int kmin = g.nplane == g.R + 1 ? 0 : -g.R;
  double2 r[TM];
#pragma unroll
  for (int k = 0; k < TM; ++k) r[k] = make_double2(0.0, 0.0);
  if (t < A && live) {
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) {
      const size_t idx = ((size_t)(t + A * k2) * n2 + y) * n1 + x;
      r[k2] = make_double2(a[idx], b ? b[idx] : 0.0);
    }
  }
  col_fft<double2, A, B, -1>(r, t, lds, TX, c, tw);
  if (t < B && live) {
#pragma unroll
    for (int j1 = 0; j1 < A; ++j1) {
      const int kz = signed_freq(t + B * j1, N);
      if (kz >= kmin && kz <= g.R) W2[((size_t)(kz - kmin) * n2 + y) * g.p1 + x] = r[j1];
    }
  }
}

// z-FFT exp(+i) of the planes |m3| <= R to full columns: oa = Re, ob = Im,
// ov = scale * Re in type T (each may be null).
template <typename T, int A, int B, int TX>
__global__ void __launch_bounds__(TX * (A > B ? A : B))
    k_z_inv_dense_r(PassGeom g, const double2* __restrict__ W2, DenseOut<T> out, double scale,
                    const double2* __restrict__ twg, int nf, int per) {
  constexpr int N = A * B, TM = MaxAB<A, B>::v;
  extern __shared__ unsigned char smem_raw[];
  double2* tw = reinterpret_cast<double2*>(smem_raw);
  double2* lds = tw + N;
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const int n1 = g.n1, n2 = g.n2;
  int cb, f;  // (column block, field pair f), XCD-contiguous as in k_z_vpsi_r
  if (!z_block_of(nf, per, (n1 * n2 + TX - 1) / TX, cb, f)) return;
  const int q = cb * TX + c;  // plane column, x fastest
  const bool live = q < n1 * n2;
  const int y = live ? q / n1 : 0, x = q - y * n1;
  double* __restrict__ oa = out.a[f];
  double* __restrict__ ob = out.b[f];
  T* __restrict__ ov = out.v[f];
  W2 += (size_t)f * g.nplane * g.n2 * g.p1;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twg[i];
  __syncthreads();
  const bool half = g.nplane == g.R + 1;
  double2 r[TM];
#pragma unroll
  for (int k = 0; k < TM; ++k) r[k] = make_double2(0.0, 0.0);
  if (t < A && live) {
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) {
      const int kz = signed_freq(t + A * k2, N);
      if (kz >= -g.R && kz <= g.R) r[k2] = W2[((size_t)(half ? abs(kz) : kz + g.R) * n2 + y) * g.p1 + x];
      if (half && kz < 0) r[k2].y = -r[k2].y;
    }
  }
  col_fft<double2, A, B, +1>(r, t, lds, TX, c, tw);
  if (t < B && live) {
#pragma unroll
    for (int j1 = 0; j1 < A; ++j1) {
      const size_t idx = ((size_t)(t + B * j1) * n2 + y) * n1 + x;
      if (oa) oa[idx] = r[j1].x;
      if (ob) ob[idx] = r[j1].y;
      if (ov) ov[idx] = (T)(scale * r[j1].x);
    }
  }
}

// x-FFT exp(-i) of direct and mirror rows, unpack two real fields:
// A = (F(G) + conj F(-G)) / 2, B = (F(G) - conj F(-G)) / 2i, times scale.
template <int A, int B, int HR>
__global__ void __launch_bounds__(2 * HR * (A > B ? A : B))
    k_rows_fwd_unpack_r(PassGeom g, const double2* __restrict__ W1, double2* __restrict__ out, int ldc, double scale,
                        const double2* __restrict__ twg) {
  constexpr int N = A * B, TM = MaxAB<A, B>::v, ST = N + 1;
  extern __shared__ unsigned char smem_raw[];
  double2* tw = reinterpret_cast<double2*>(smem_raw);
  double2* lds = tw + N;
  const int t = threadIdx.x % TM, fr = threadIdx.x / TM;
  const int hr = fr >> 1, mirror = fr & 1;
  const int row = blockIdx.x * HR + hr;
  W1 += (size_t)blockIdx.y * g.nslot * g.p1;  // field pair blockIdx.y: its rows and its two output fields
  out += (size_t)blockIdx.y * 2 * ldc;
  const bool live = row < g.nrow;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twg[i];
  RowInfo ri{};
  if (live) ri = g.rows[row];
  const bool zero_row = live && ri.slot_m < 0;
  __syncthreads();
  double2 r[TM];
#pragma unroll
  for (int k = 0; k < TM; ++k) r[k] = make_double2(0.0, 0.0);
  if (live && t < A && !(zero_row && mirror)) {
    const double2* in = W1 + (size_t)(mirror ? ri.slot_m : ri.slot_d) * g.p1;
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) r[k2] = in[t + A * k2];
  }
  col_fft<double2, A, B, -1>(r, t, lds, 1, fr * ST, tw);
  if (t < B) {
#pragma unroll
    for (int j1 = 0; j1 < A; ++j1) lds[fr * ST + t + B * j1] = r[j1];
  }
  __syncthreads();
  if (live) {
    const double2* rd = lds + (2 * hr) * ST;
    const double2* rm = zero_row ? rd : rd + ST;
    for (int e = t + mirror * TM; e < ri.cnt; e += 2 * TM) {
      const int m1 = ri.m1_0 + e;
      const double2 P = rd[wrap(m1, N)], M = rm[wrap(-m1, N)];
      out[ri.start + e] = make_double2(0.5 * scale * (P.x + M.x), 0.5 * scale * (P.y - M.y));
      out[(size_t)ldc + ri.start + e] = make_double2(0.5 * scale * (P.y + M.y), -0.5 * scale * (P.x - M.x));
    }
  }
}

// x pass inverse of a single real field on the rows with m3 >= 0: transform u
// is row u, from nrow on the mirror (-m2, 0) of row u - nrow + 1; the rows of
// m3 = 0 come first, (0, 0) before the others.
template <int A, int B, int FR>
__global__ void __launch_bounds__(FR * (A > B ? A : B))
    k_rows_inv_one_r(PassGeom g, const double2* __restrict__ C, double2* __restrict__ W1, int ntr,
                     const double2* __restrict__ twg) {
  constexpr int N = A * B, TM = MaxAB<A, B>::v, ST = N + 1;
  extern __shared__ unsigned char smem_raw[];
  double2* tw = reinterpret_cast<double2*>(smem_raw);
  double2* lds = tw + N;
  const int t = threadIdx.x % TM, fr = threadIdx.x / TM;
  const int u = blockIdx.x * FR + fr;
  const bool live = u < ntr, mirror = u >= g.nrow;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twg[i];
  RowInfo ri{};
  if (live) ri = g.rows[mirror ? u - g.nrow + 1 : u];
  __syncthreads();
  double2 r[TM];
#pragma unroll
  for (int k = 0; k < TM; ++k) r[k] = make_double2(0.0, 0.0);
  if (live && t < A) {
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) {
      const int m1 = signed_freq(t + A * k2, N);
      const bool conj = mirror || (u == 0 && m1 < 0);  // (0, 0): both halves
      const int e = (conj ? -m1 : m1) - ri.m1_0;
      if (e >= 0 && e < ri.cnt) {
        r[k2] = C[ri.start + e];
        if (conj) r[k2].y = -r[k2].y;
      }
    }
  }
  col_fft<double2, A, B, +1>(r, t, lds, 1, fr * ST, tw);
  if (live && t < B) {
    double2* out = W1 + (size_t)(mirror ? ri.slot_m : ri.slot_d) * g.p1;
#pragma unroll
    for (int j1 = 0; j1 < A; ++j1) out[t + B * j1] = r[j1];
  }
}

// x pass forward of a single real field: the direct rows hold all of it.
template <int A, int B, int FR>
__global__ void __launch_bounds__(FR * (A > B ? A : B))
    k_rows_fwd_one_r(PassGeom g, const double2* __restrict__ W1, double2* __restrict__ out, double scale,
                     const double2* __restrict__ twg) {
  constexpr int N = A * B, TM = MaxAB<A, B>::v, ST = N + 1;
  extern __shared__ unsigned char smem_raw[];
  double2* tw = reinterpret_cast<double2*>(smem_raw);
  double2* lds = tw + N;
  const int t = threadIdx.x % TM, fr = threadIdx.x / TM;
  const int row = blockIdx.x * FR + fr;
  const bool live = row < g.nrow;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twg[i];
  RowInfo ri{};
  if (live) ri = g.rows[row];
  __syncthreads();
  double2 r[TM];
#pragma unroll
  for (int k = 0; k < TM; ++k) r[k] = make_double2(0.0, 0.0);
  if (live && t < A) {
    const double2* in = W1 + (size_t)ri.slot_d * g.p1;
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) r[k2] = in[t + A * k2];
  }
  col_fft<double2, A, B, -1>(r, t, lds, 1, fr * ST, tw);
  if (live && t < B) {
#pragma unroll
    for (int j1 = 0; j1 < A; ++j1) {
      const int e = signed_freq(t + B * j1, N) - ri.m1_0;
      if (e >= 0 && e < ri.cnt) out[ri.start + e] = make_double2(scale * r[j1].x, scale * r[j1].y);
    }
  }
}

}  // namespace amdk
