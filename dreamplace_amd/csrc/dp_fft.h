// Fast 2-D cosine / sine transforms and the Poisson solve on grids whose
// sides are powers of two (fft_f32.hip, fft_f64.hip instantiate this file).
//
// A length-n DCT of a real sequence x is one length-n complex FFT of two
// sequences at once (Makhoul, "A fast cosine transform in one and two
// dimensions", IEEE Trans. ASSP 28, 1980): with v[j] = x[2j] for j < n/2 and
// x[2(n-1-j)+1] above, V = FFT(v), C[k] = Re(e^{-i pi k/2n} V[k]) is
// sum x[i] cos(pi k (2i+1)/2n), and z = v_a + i v_b gives both V_a and V_b by
// conjugate symmetry.  The inverse runs the same steps backwards, and
// IDXST(X)[m] = (-1)^m IDCT(X')[m] with X'[k] = X[n-k], X'[0] = 0.
//
// The solve is three launches:
//   rows     DCT of pairs of rows of the map, each row about its own mean
//            (kept in FP64 beside);
//   columns  per pair of columns: DCT, spectral multipliers and energy terms
//            in LDS, then per column one complex inverse FFT for both fields
//            (IDXST for field x in the real part, IDCT for field y in the
//            imaginary part; the potential's two columns share a third);
//   rows     per row one complex inverse FFT (IDCT of field x, IDXST of
//            field y); the potential's rows in pairs.
// An FFT runs in LDS, eight elements per thread, radix 8 and 4 (Stockham).
//
// What bounds it: the passes move 9 maps of data (4 MB each at 1024^2 in
// FP32), which stay in L2 and the memory-side cache, so each launch is a few
// microseconds of latency: loads, three or four LDS exchanges, stores.  The
// dense products L * (x * R) on the matrix cores that other grids take
// (spectral.hip) need 2 n^3 flop per product instead of 5 n^2 log2 n.
// Measured, dense -> fast: the 2048^2 solve 383 us (BF16x3) -> 75 (FP32), the
// 1024^2 solve 112 (BF16x3) -> 32 (FP32) and ~380 -> 44 (FP64); four 512^2
// FP32 transforms 130 -> 54; the error against 64 bits 5.1e-6 (BF16x3) ->
// 2.5e-7.  The fast form was the quicker at every power of two from 32 on, so
// it takes them all.
#pragma once

#include <math.h>

#include "dp_common.h"

namespace dp {

constexpr int kFftMinLog = 5, kFftMaxLog = 12;  // sides 32 .. 4096

inline int fft_log(int n) {
  int lg = 0;
  while ((1 << lg) < n) ++lg;
  return (1 << lg) == n && lg >= kFftMinLog && lg <= kFftMaxLog ? lg : -1;
}
inline bool fft_shape(int M, int N) { return fft_log(M) > 0 && fft_log(N) > 0; }

// Plan tables of a side n: tw[t] = e^{-2 pi i t/n} (t < n), then
// dw[k] = e^{i pi k/2n} (k <= n/2), as complex T.
inline size_t fft_table_elems(int n) { return (size_t)n + n / 2 + 1; }

template <typename T>
struct FftTables {
  const typename Vec2<T>::type *tw_m, *dw_m, *tw_n, *dw_n;
};
template <typename T>
inline FftTables<T> fft_tables(const void* plan, int M, int N) {
  typedef typename Vec2<T>::type V;
  const V* p = (const V*)plan;
  return {p, p + M, p + fft_table_elems(M), p + fft_table_elems(M) + N};
}

// Host entries, one set per type.  ws: spectral workspace (slabs of M*N T).
enum FftInv { kInvIdct = 0, kInvIdxst = 1 };
template <typename T>
int fft_plan_fill(int M, int N, void* plan, hipStream_t s);
template <typename T>
int fft_dct2(const void* plan, int M, int N, const void* x, void* out, void* ws, hipStream_t s);
template <typename T>
int fft_inverse(const void* plan, int M, int N, const void* x, void* out, void* ws, int kind_m,
                int kind_n, hipStream_t s);
template <typename T>
int fft_poisson(const void* plan, int M, int N, const void* map, double bsx, double bsy,
                bool want_phi, void* field_x, void* field_y, void* potential, void* energy,
                void* ws, size_t slab, hipStream_t s);

// An energy term c K a^2, from the type's a and k: in FP64, K by a Newton step from
// k (2^-22 -> 2^-44), as the terms of few modes are most of the sum and the FP32
// step du alone shifts each by 1e-7.
template <typename T>
__device__ __forceinline__ double energy_term(T c, T k, double wu, double wv, T a) {
  double kd = (double)k;
  if constexpr (sizeof(T) == 4) kd = fma(kd, fma(-fma(wu, wu, wv * wv), kd, 1.0), kd);
  return (double)c * kd * ((double)a * (double)a);
}

#ifdef DP_FFT_IMPL

template <typename T>
struct Cx {
  T x, y;
};
template <typename T>
__device__ __forceinline__ Cx<T> operator+(Cx<T> a, Cx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ Cx<T> operator-(Cx<T> a, Cx<T> b) { return {a.x - b.x, a.y - b.y}; }
template <typename T>
__device__ __forceinline__ Cx<T> cmul(Cx<T> a, Cx<T> w) {
  return {fma(a.x, w.x, -(a.y * w.y)), fma(a.x, w.y, a.y * w.x)};
}
// a * (-i) forward, a * i inverse
template <bool kInv, typename T>
__device__ __forceinline__ Cx<T> rot(Cx<T> a) {
  return kInv ? Cx<T>{-a.y, a.x} : Cx<T>{a.y, -a.x};
}
template <typename T>
__device__ __forceinline__ Cx<T> ld2(const typename Vec2<T>::type* p) {
  const typename Vec2<T>::type v = *p;
  return {v.x, v.y};
}
template <typename T>
__device__ __forceinline__ void st2(typename Vec2<T>::type* p, Cx<T> c) {
  typename Vec2<T>::type v;
  v.x = c.x;
  v.y = c.y;
  *p = v;
}

template <bool kInv, typename T>
__device__ __forceinline__ void dft4(Cx<T>& a, Cx<T>& b, Cx<T>& c, Cx<T>& d) {
  const Cx<T> s0 = a + c, d0 = a - c, s1 = b + d, d1 = rot<kInv>(b - d);
  a = s0 + s1;
  c = s0 - s1;
  b = d0 + d1;
  d = d0 - d1;
}
// natural-order outputs in e[0..8)
template <bool kInv, typename T>
__device__ __forceinline__ void dft8(Cx<T> (&e)[8]) {
  Cx<T> p0 = e[0], p1 = e[2], p2 = e[4], p3 = e[6];
  Cx<T> q0 = e[1], q1 = e[3], q2 = e[5], q3 = e[7];
  dft4<kInv>(p0, p1, p2, p3);
  dft4<kInv>(q0, q1, q2, q3);
  const T h = (T)0.70710678118654752440;
  q1 = kInv ? Cx<T>{(q1.x - q1.y) * h, (q1.x + q1.y) * h} : Cx<T>{(q1.x + q1.y) * h, (q1.y - q1.x) * h};
  q2 = rot<kInv>(q2);
  q3 = kInv ? Cx<T>{-(q3.x + q3.y) * h, (q3.x - q3.y) * h} : Cx<T>{(q3.y - q3.x) * h, -(q3.x + q3.y) * h};
  e[0] = p0 + q0;
  e[4] = p0 - q0;
  e[1] = p1 + q1;
  e[5] = p1 - q1;
  e[2] = p2 + q2;
  e[6] = p2 - q2;
  e[3] = p3 + q3;
  e[7] = p3 - q3;
}

// LDS position of element i: one pad element in eight, so that the radix-8
// stores (stride 8) and the contiguous loads both spread over the banks
__device__ __forceinline__ int fpad(int i) { return i + (i >> 3); }
template <int LG>
struct Fft {
  static constexpr int n = 1 << LG;
  static constexpr int threads = n / 8;  // per FFT
  static constexpr int lds = n + n / 8;  // padded elements
};
// LDS elements of one of K interleaved columns (neighbouring lanes take
// neighbouring columns): n + n / 8 is a whole number of bank rows, which put a
// lane group's columns on the same banks (64% of the LDS cycles of the 2048^2
// solve were conflicts); an even share of a bank row more keeps K columns' runs
// of elements apart (2048^2: 5.0 -> 1.8 million conflict cycles, 40 -> 36.6 us;
// 1024^2 14.8 -> 13.9).
template <typename T, int LG, int K>
constexpr int col_lds() {
  return Fft<LG>::lds + (K > 1 && K < 128 / (int)sizeof(T) ? 128 / (int)sizeof(T) / K : 0);
}

// The length-2^LG FFT of one group of n/8 threads (thread j of it), inputs
// e[q] = z[j + q n/8], outputs e[m] = Z[j + m n/8], unnormalised.  `buf` is
// the group's LDS array; every thread of the workgroup takes part in the
// barriers, those with on == false in nothing else.  The caller has a barrier
// between its own use of buf and this call; buf may be written after the
// next barrier following the call.
template <bool kInv, int LG, typename T>
__device__ __forceinline__ void fft_run(Cx<T> (&e)[8], typename Vec2<T>::type* buf, int j, bool on,
                                        const typename Vec2<T>::type* __restrict__ tw) {
  constexpr int n = 1 << LG, P = n / 8;
  dft8<kInv>(e);
  int ns = 8;            // product of the radices done
  int done = 3;          // log2 of it
  if (on) {
#pragma unroll
    for (int q = 0; q < 8; ++q) st2<T>(buf + fpad(8 * j + q), e[q]);
  }
#pragma unroll
  for (int pass = 0; pass < 5; ++pass) {
    if (done >= LG) break;
    // radix 8 unless what remains is 4 or 16
    const int left = LG - done;
    const bool r8 = left == 3 || left >= 5;
    const bool last = (r8 && left == 3) || (!r8 && left == 2);
    Cx<T> w[8];
    if (r8) {
      const int k = j & (ns - 1);
#pragma unroll
      for (int q = 1; q < 8; ++q) w[q] = ld2<T>(tw + q * k * (n / (8 * ns)));
    } else {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int k = (j + b * P) & (ns - 1);
#pragma unroll
        for (int q = 1; q < 4; ++q) w[4 * b + q] = ld2<T>(tw + q * k * (n / (4 * ns)));
      }
    }
    if (kInv) {
#pragma unroll
      for (int q = 0; q < 8; ++q) w[q].y = -w[q].y;
    }
    __syncthreads();
    if (on) {
      if (r8) {
#pragma unroll
        for (int q = 0; q < 8; ++q) e[q] = ld2<T>(buf + fpad(j + q * P));
      } else {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int q = 0; q < 4; ++q) e[4 * b + q] = ld2<T>(buf + fpad(j + b * P + 2 * q * P));
      }
    }
    if (!last) __syncthreads();
    if (r8) {
#pragma unroll
      for (int q = 1; q < 8; ++q) e[q] = cmul(e[q], w[q]);
      dft8<kInv>(e);
      if (!last && on) {
        const int k = j & (ns - 1), base = 8 * (j - k) + k;
#pragma unroll
        for (int q = 0; q < 8; ++q) st2<T>(buf + fpad(base + q * ns), e[q]);
      }
      ns *= 8;
      done += 3;
    } else {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
#pragma unroll
        for (int q = 1; q < 4; ++q) e[4 * b + q] = cmul(e[4 * b + q], w[4 * b + q]);
        dft4<kInv>(e[4 * b], e[4 * b + 1], e[4 * b + 2], e[4 * b + 3]);
        if (!last && on) {
          const int jj = j + b * P, k = jj & (ns - 1), base = 4 * (jj - k) + k;
#pragma unroll
          for (int q = 0; q < 4; ++q) st2<T>(buf + fpad(base + q * ns), e[4 * b + q]);
        }
      }
      if (last) {  // Z[j + b P + q 2P] -> e[b + 2 q]
        const Cx<T> t1 = e[1], t2 = e[2], t3 = e[3], t4 = e[4], t5 = e[5], t6 = e[6];
        e[1] = t4;
        e[2] = t1;
        e[3] = t5;
        e[4] = t2;
        e[5] = t6;
        e[6] = t3;
      }
      ns *= 4;
      done += 2;
    }
  }
}

// index of the sequence that FFT element j stands for
template <int LG>
__device__ __forceinline__ int seq_of(int j) {
  constexpr int n = 1 << LG;
  return j < n / 2 ? 2 * j : 2 * (n - 1 - j) + 1;
}

// The DCT coefficients C_a, C_b at k and n - k from Z at both (1 <= k < n/2),
// w = e^{i pi k/2n}.  At k = 0 and n/2 the caller takes its own form.
template <typename T>
struct DctPair {
  T ak, ank, bk, bnk;
};
template <typename T>
__device__ __forceinline__ DctPair<T> dct_pair(Cx<T> zk, Cx<T> znk, Cx<T> w, int k) {
  if (k == 0)  // zk = Z[0], znk = Z[n/2]: ank, bnk are the coefficients n/2
    return {zk.x, znk.x * (T)0.70710678118654752440, zk.y, znk.y * (T)0.70710678118654752440};
  const Cx<T> va = {(T)0.5 * (zk.x + znk.x), (T)0.5 * (zk.y - znk.y)};
  const Cx<T> vb = {(T)0.5 * (zk.y + znk.y), (T)0.5 * (znk.x - zk.x)};
  // e^{-i pi k/2n} v = (v.x c + v.y s, v.y c - v.x s): real part at k, minus
  // the imaginary part at n - k
  return {fma(va.x, w.x, va.y * w.y), fma(va.x, w.y, -(va.y * w.x)),
          fma(vb.x, w.x, vb.y * w.y), fma(vb.x, w.y, -(vb.y * w.x))};
}
// The inverse FFT's inputs at k and n - k from the coefficients (IDCT order;
// an IDXST sequence comes with its k and n - k entries swapped).
template <typename T>
__device__ __forceinline__ void inv_pair(DctPair<T> p, Cx<T> w, Cx<T>& zk, Cx<T>& znk) {
  zk = cmul(Cx<T>{p.ak + p.bnk, p.bk - p.ank}, w);
  znk = cmul(Cx<T>{p.ank + p.bk, p.bnk - p.ak}, Cx<T>{w.y, w.x});
}
template <typename T>
__device__ __forceinline__ void swap_if(bool c, T& a, T& b) {
  const T u = a, v = b;
  a = c ? v : u;
  b = c ? u : v;
}
// inv_pair at k = 0 (ak, bk the coefficients 0; ank, bnk those of n/2) with
// znk = Z[n/2]: IDXST sequences have no entry 0.
template <typename T>
__device__ __forceinline__ void inv_pair0(DctPair<T> p, bool sa, bool sb, Cx<T>& z0, Cx<T>& zh) {
  const T h = (T)0.70710678118654752440;
  z0 = {sa ? T(0) : p.ak, sb ? T(0) : p.bk};
  // k = n - k = n/2: (a + b) + i (b - a) times e^{i pi/4}
  zh = cmul(Cx<T>{p.ank + p.bnk, p.bnk - p.ank}, Cx<T>{h, h});
}

// Sum over the threads of each group of P consecutive threads of a workgroup
// (P a power of two), in FP64 and a fixed order; every thread gets its
// group's.  smem: one double per wavefront and value.
template <int P>
__device__ __forceinline__ double group_sum(double v, double* smem) {
  constexpr int W = P < 64 ? P : 64;
#pragma unroll
  for (int o = W / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if constexpr (P > 64) {
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) smem[wave] = v;
    __syncthreads();
    constexpr int G = P / 64;
    const int w0 = wave / G * G;
    double s = 0;
#pragma unroll
    for (int i = 0; i < G; ++i) s += smem[w0 + i];
    v = s;
    __syncthreads();
  }
  return v;
}

// ---- rows ------------------------------------------------------------------
// DCT of rows 2p and 2p + 1 of in[rows][n], times `scale`.  kMean: each row
// is transformed about its own mean, so that a flat map keeps its small
// coefficients' precision; row_mean[row] receives the mean (FP64) and the
// coefficient 0 is left to the reader of row_mean (0 is written).
template <typename T, int LG, bool kMean>
__global__ void __launch_bounds__(Fft<LG>::threads > 64 ? Fft<LG>::threads : 64)
    k_fft_rows_dct(const T* __restrict__ in, T* out, int pairs, T scale, double* row_mean,
                   const typename Vec2<T>::type* __restrict__ tw,
                   const typename Vec2<T>::type* __restrict__ dw) {
  typedef typename Vec2<T>::type V;
  constexpr int n = 1 << LG, P = n / 8, F = P < 64 ? 64 / P : 1;
  __shared__ V lds[F * Fft<LG>::lds];
  __shared__ double red[2][F * P / 64];
  const int f = threadIdx.x / P, j = threadIdx.x % P;
  const int p = blockIdx.x * F + f;
  const bool on = p < pairs;
  V* buf = lds + f * Fft<LG>::lds;
  const T* a = in + (size_t)2 * (on ? p : 0) * n;
  const T* b = a + n;
  Cx<T> e[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int i = seq_of<LG>(j + q * P);
    e[q] = {a[i], b[i]};
  }
  if (kMean) {
    double sa = 0, sb = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      sa += (double)e[q].x;
      sb += (double)e[q].y;
    }
    sa = group_sum<P>(sa, red[0]) / n;
    sb = group_sum<P>(sb, red[1]) / n;
    if (on && j == 0) {
      row_mean[2 * p] = sa;
      row_mean[2 * p + 1] = sb;
    }
    const T ma = (T)sa, mb = (T)sb;
#pragma unroll
    for (int q = 0; q < 8; ++q) e[q] = {e[q].x - ma, e[q].y - mb};
  }
  fft_run<false, LG, T>(e, buf, j, on, tw);
  __syncthreads();
  if (on) {
#pragma unroll
    for (int m = 0; m < 8; ++m) st2<T>(buf + fpad(j + m * P), e[m]);
  }
  __syncthreads();
  if (!on) return;
  T* oa = out + (size_t)2 * p * n;
  T* ob = oa + n;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int k = j + m * P, nk = k ? n - k : n / 2;
    const DctPair<T> d = dct_pair<T>(ld2<T>(buf + fpad(k)), ld2<T>(buf + fpad(nk)), ld2<T>(dw + k), k);
    const bool dc = kMean && k == 0;
    oa[k] = dc ? T(0) : d.ak * scale;
    ob[k] = dc ? T(0) : d.bk * scale;
    oa[nk] = d.ank * scale;
    ob[nk] = d.bnk * scale;
  }
}

// *total = the sum of the energy's partials, by one workgroup: what a launch
// of its own after the column kernel took 5 us for.
template <int BLOCK, typename T>
__device__ __forceinline__ void sum_partials(const double* __restrict__ p, int n, T* total,
                                             double* smem) {
  double v = 0;
  for (int i = threadIdx.x; i < n; i += BLOCK) v += p[i];
  v = block_sum<BLOCK>(v, smem);
  if (threadIdx.x == 0) *total = (T)v;
}

// Inverse transforms along rows.  kField: in is [rows][n] complex pairs, one
// row per FFT, IDCT of the real parts to out_a and IDXST of the imaginary
// parts to out_b ([rows][n] each).  Else in / out_a are [rows][n] T and an
// FFT takes rows 2p, 2p + 1, both IDCT (kind 0) or both IDXST (kind 1).  A
// kField launch may have one workgroup more, for the energy.
template <typename T, int LG, bool kField>
__global__ void __launch_bounds__(Fft<LG>::threads > 64 ? Fft<LG>::threads : 64)
    k_fft_rows_inv(const void* __restrict__ in, T* out_a, T* out_b, int count, int kind,
                   const typename Vec2<T>::type* __restrict__ tw,
                   const typename Vec2<T>::type* __restrict__ dw,
                   const double* __restrict__ partials, int nparts, T* total) {
  typedef typename Vec2<T>::type V;
  constexpr int n = 1 << LG, P = n / 8, F = P < 64 ? 64 / P : 1;
  __shared__ V lds[F * Fft<LG>::lds];
  if (kField && (int)blockIdx.x == (count + F - 1) / F) {  // the whole workgroup
    sum_partials<P < 64 ? 64 : P>(partials, nparts, total, (double*)lds);
    return;
  }
  const int f = threadIdx.x / P, j = threadIdx.x % P;
  const int p = blockIdx.x * F + f;
  const bool on = p < count;
  V* buf = lds + f * Fft<LG>::lds;
  const bool sa = !kField && kind == kInvIdxst, sb = kField || kind == kInvIdxst;
  const T* a = (const T*)in + (size_t)2 * (on ? p : 0) * n;  // kField: row p of pairs
  const T* b = a + n;
  if (on) {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int k = j + m * P, nk = k ? n - k : n / 2;
      DctPair<T> d;
      if (kField) {
        const Cx<T> u = ld2<T>((const V*)a + k), v = ld2<T>((const V*)a + nk);
        d = {u.x, v.x, u.y, v.y};
      } else {
        d = {a[k], a[nk], b[k], b[nk]};
      }
      Cx<T> zk, znk;
      if (k == 0) {
        inv_pair0<T>(d, sa, sb, zk, znk);
      } else {
        swap_if(sa, d.ak, d.ank);
        swap_if(sb, d.bk, d.bnk);
        inv_pair<T>(d, ld2<T>(dw + k), zk, znk);
      }
      st2<T>(buf + fpad(k), zk);
      st2<T>(buf + fpad(nk), znk);
    }
  }
  __syncthreads();
  Cx<T> e[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) e[q] = ld2<T>(buf + fpad(j + q * P));
  __syncthreads();
  fft_run<true, LG, T>(e, buf, j, on, tw);
  if (!on) return;
  T* oa = kField ? out_a + (size_t)p * n : out_a + (size_t)2 * p * n;
  T* ob = kField ? out_b + (size_t)p * n : oa + n;
#pragma unroll
  for (int m = 0; m < 8; ++m) {
    const int i = seq_of<LG>(j + m * P);
    oa[i] = sa && (i & 1) ? -e[m].x : e[m].x;
    ob[i] = sb && (i & 1) ? -e[m].y : e[m].y;
  }
}

// ---- columns ---------------------------------------------------------------
// Workgroup b takes 2F consecutive columns.  Workgroups go to the dies
// round-robin, so die x is given a contiguous band of columns: the cache
// lines that neighbouring workgroups share are fetched once per die.
__device__ __forceinline__ int column_group() {
  const int g = gridDim.x, b = blockIdx.x;
  return g % 8 == 0 ? (b % 8) * (g / 8) + b / 8 : b;
}

// Forward (kind_inv < 0: DCT times scale) or inverse (kInvIdct / kInvIdxst)
// transform along the columns of in[n][N], F pairs of columns per workgroup.
template <typename T, int LG, int F, bool kForward>
__global__ void __launch_bounds__(F* Fft<LG>::threads)
    k_fft_cols(const T* __restrict__ in, T* out, int N, T scale, int kind,
               const typename Vec2<T>::type* __restrict__ tw,
               const typename Vec2<T>::type* __restrict__ dw) {
  typedef typename Vec2<T>::type V;
  constexpr int n = 1 << LG, P = n / 8;
  extern __shared__ __attribute__((aligned(16))) char fft_lds[];
  const int f = threadIdx.x % F, j = threadIdx.x / F;
  V* buf = (V*)fft_lds + f * col_lds<T, LG, F>();
  const int v0 = column_group() * 2 * F + 2 * f;
  const V* src = (const V*)(in + v0);
  V* dst = (V*)(out + v0);
  const size_t rs = (size_t)N / 2;  // row stride in pairs
  Cx<T> e[8];
  if (kForward) {
#pragma unroll
    for (int q = 0; q < 8; ++q) e[q] = ld2<T>(src + seq_of<LG>(j + q * P) * rs);
    fft_run<false, LG, T>(e, buf, j, true, tw);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 8; ++m) st2<T>(buf + fpad(j + m * P), e[m]);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int k = j + m * P, nk = k ? n - k : n / 2;
      const DctPair<T> d = dct_pair<T>(ld2<T>(buf + fpad(k)), ld2<T>(buf + fpad(nk)), ld2<T>(dw + k), k);
      st2<T>(dst + k * rs, Cx<T>{d.ak * scale, d.bk * scale});
      st2<T>(dst + nk * rs, Cx<T>{d.ank * scale, d.bnk * scale});
    }
  } else {
    const bool s = kind == kInvIdxst;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int k = j + m * P, nk = k ? n - k : n / 2;
      const Cx<T> u = ld2<T>(src + k * rs), v = ld2<T>(src + nk * rs);
      DctPair<T> d = {u.x, v.x, u.y, v.y};
      Cx<T> zk, znk;
      if (k == 0) {
        inv_pair0<T>(d, s, s, zk, znk);
      } else {
        swap_if(s, d.ak, d.ank);
        swap_if(s, d.bk, d.bnk);
        inv_pair<T>(d, ld2<T>(dw + k), zk, znk);
      }
      st2<T>(buf + fpad(k), zk);
      st2<T>(buf + fpad(nk), znk);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; ++q) e[q] = ld2<T>(buf + fpad(j + q * P));
    __syncthreads();
    fft_run<true, LG, T>(e, buf, j, true, tw);
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int i = seq_of<LG>(j + m * P);
      const bool neg = s && (i & 1);
      st2<T>(dst + i * rs, neg ? Cx<T>{-e[m].x, -e[m].y} : e[m]);
    }
  }
}

// The middle of the solve.  A[u][v] (rows transformed about their means, in
// row_mean) -> spectrum a -> field[m][v] = (IDXST_u of a wu K/2, IDCT_u of
// a wv K/2) as pairs, phi[m][v] = IDCT_u of a K, and the workgroup's partial
// of the energy (MN/4) sum c_u c_v K a^2 (electric_potential.py:504-519:
// wu = du u, wv = dv v, K = 1/(wu^2 + wv^2), K[0,0] = 0).
template <typename T>
__device__ __forceinline__ T spectral_k(T wu, T wv) {
  const T w2 = wu * wu + wv * wv;
  return w2 == T(0) ? T(0) : T(1) / w2;
}
template <typename T, int LG, int F>
__global__ void __launch_bounds__(2 * F * Fft<LG>::threads)
    k_fft_cols_solve(const T* __restrict__ A, typename Vec2<T>::type* field, T* phi, int N,
                     T scale, double mean_scale, const double* __restrict__ row_mean, double du,
                     double dv,
                     double* partials, const typename Vec2<T>::type* __restrict__ tw,
                     const typename Vec2<T>::type* __restrict__ dw) {
  typedef typename Vec2<T>::type V;
  constexpr int n = 1 << LG, P = n / 8, BLOCK = 2 * F * P;
  constexpr int L = col_lds<T, LG, 2 * F>();  // a column's array; a pair of columns uses the first
  constexpr int W = BLOCK < 64 ? 1 : BLOCK / 64;
  extern __shared__ __attribute__((aligned(16))) char fft_lds[];
  __shared__ double red[W];
  __shared__ double s_mean;
  V* buf = (V*)fft_lds;
  const int t = threadIdx.x;
  const int g0 = column_group() * 2 * F;  // first column
  const size_t rs = (size_t)N / 2;
  Cx<T> e[8];
  const bool fwd = t < F * P;
  const int ff = t % F, fj = fwd ? t / F : 0;
  if (fwd) {
    const V* src = (const V*)(A + g0 + 2 * ff);
#pragma unroll
    for (int q = 0; q < 8; ++q) e[q] = ld2<T>(src + seq_of<LG>(fj + q * P) * rs);
  }
  if (g0 == 0) {
    // column 0 holds twice the rows' means, which the row pass left out:
    // put them in about their own mean (a[0,0] has no weight)
    double m = 0;
    for (int i = t; i < n; i += BLOCK) m += row_mean[i];
    m = wave_sum(m);
    if ((t & 63) == 0) red[t >> 6] = m;
    __syncthreads();
    if (t == 0) {
      double r = 0;
      for (int i = 0; i < W; ++i) r += red[i];
      s_mean = r / n;
    }
    __syncthreads();
    if (fwd && ff == 0) {
#pragma unroll
      for (int q = 0; q < 8; ++q)
        e[q].x = (T)((row_mean[seq_of<LG>(fj + q * P)] - s_mean) * mean_scale);
    }
  }
  fft_run<false, LG, T>(e, buf + 2 * ff * L, fj, fwd, tw);
  __syncthreads();
  if (fwd) {
#pragma unroll
    for (int m = 0; m < 8; ++m) st2<T>(buf + 2 * ff * L + fpad(fj + m * P), e[m]);
  }
  __syncthreads();
  // coefficients of columns 2c, 2c + 1 at k and n - k: two pairs per thread
  const int c = t % F, cj = t / F;  // cj < 2P
  Cx<T> z[2][4];                    // [pair][column, k | n - k]
  Cx<T> zp[2][2];                   // the potential's
  double esum = 0;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int k = cj + 2 * m * P, nk = k ? n - k : n / 2;
    const V* b = buf + 2 * c * L;
    const Cx<T> w = ld2<T>(dw + k);
    DctPair<T> d = dct_pair<T>(ld2<T>(b + fpad(k)), ld2<T>(b + fpad(nk)), w, k);
    const int v = g0 + 2 * c;
    const T wk = (T)du * (T)k, wnk = (T)du * (T)nk;
    DctPair<T> ph;
#pragma unroll
    for (int col = 0; col < 2; ++col) {
      const T wv = (T)dv * (T)(v + col);
      const T ak = (col ? d.bk : d.ak) * scale, ank = (col ? d.bnk : d.ank) * scale;
      const T kk = spectral_k(wk, wv), knk = spectral_k(wnk, wv);
      const T cv = v + col ? T(2) : T(1), ck = k ? T(2) : T(1);
      esum += energy_term<T>(ck * cv, kk, du * k, dv * (v + col), ak);
      esum += energy_term<T>(T(2) * cv, knk, du * nk, dv * (v + col), ank);
      DctPair<T> q;
      q.ak = ak * (wk * kk * (T)0.5);  // field x, IDXST: k and n - k swapped
      q.ank = ank * (wnk * knk * (T)0.5);
      q.bk = ak * (wv * kk * (T)0.5);  // field y, IDCT
      q.bnk = ank * (wv * knk * (T)0.5);
      if (k == 0) {
        inv_pair0<T>(q, true, false, z[m][2 * col], z[m][2 * col + 1]);
      } else {
        swap_if(true, q.ak, q.ank);
        inv_pair<T>(q, w, z[m][2 * col], z[m][2 * col + 1]);
      }
      if (col == 0) {
        ph.ak = ak * kk;
        ph.ank = ank * knk;
      } else {
        ph.bk = ak * kk;
        ph.bnk = ank * knk;
      }
    }
    if (phi) {
      if (k == 0)
        inv_pair0<T>(ph, false, false, zp[m][0], zp[m][1]);
      else
        inv_pair<T>(ph, w, zp[m][0], zp[m][1]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int k = cj + 2 * m * P, nk = k ? n - k : n / 2;
#pragma unroll
    for (int col = 0; col < 2; ++col) {
      V* b = buf + (2 * c + col) * L;
      st2<T>(b + fpad(k), z[m][2 * col]);
      st2<T>(b + fpad(nk), z[m][2 * col + 1]);
    }
  }
  __syncthreads();
  const int ic = t % (2 * F), ij = t / (2 * F);  // column g0 + ic, element ij
#pragma unroll
  for (int q = 0; q < 8; ++q) e[q] = ld2<T>(buf + ic * L + fpad(ij + q * P));
  __syncthreads();
  fft_run<true, LG, T>(e, buf + ic * L, ij, true, tw);
#pragma unroll
  for (int m = 0; m < 8; ++m) {
    const int i = seq_of<LG>(ij + m * P);
    st2<T>(field + (size_t)i * N + g0 + ic, Cx<T>{(i & 1) ? -e[m].x : e[m].x, e[m].y});
  }
  if (phi) {  // uniform
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int k = cj + 2 * m * P, nk = k ? n - k : n / 2;
      st2<T>(buf + 2 * c * L + fpad(k), zp[m][0]);
      st2<T>(buf + 2 * c * L + fpad(nk), zp[m][1]);
    }
    __syncthreads();
    if (fwd) {
#pragma unroll
      for (int q = 0; q < 8; ++q) e[q] = ld2<T>(buf + 2 * ff * L + fpad(fj + q * P));
    }
    __syncthreads();
    fft_run<true, LG, T>(e, buf + 2 * ff * L, fj, fwd, tw);
    if (fwd) {
      V* dst = (V*)(phi + g0 + 2 * ff);
#pragma unroll
      for (int m = 0; m < 8; ++m) st2<T>(dst + seq_of<LG>(fj + m * P) * rs, e[m]);
    }
  }
  if (partials) {
    const double s = wave_sum(esum);
    __syncthreads();
    if ((t & 63) == 0) red[t >> 6] = s;
    __syncthreads();
    if (t == 0) {
      double r = 0;
      for (int i = 0; i < W; ++i) r += red[i];
      partials[blockIdx.x] = r * ((double)n * N / 4.0);
    }
  }
}

// ---- tables ----------------------------------------------------------------
template <typename T>
__global__ void k_fft_tables(typename Vec2<T>::type* p, int M, int N) {
  const int em = M + M / 2 + 1, en = N + N / 2 + 1;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < em + en; i += gridDim.x * blockDim.x) {
    const int K = i < em ? M : N, t = i < em ? i : i - em;
    // t < K: e^{-2 pi i t/K}; then e^{i pi k/2K}
    const double a = t < K ? -2.0 * (double)t / K : (double)(t - K) / (2.0 * K);
    typename Vec2<T>::type v;
    v.x = (T)cospi(a);  // a is exact: K is a power of two
    v.y = (T)sinpi(a);
    p[i] = v;
  }
}

// ---- host ------------------------------------------------------------------
// Dispatch on log2 of a side: FN<LG>() for 5 .. 12.
#define DP_FFT_LOG(lg, ...)                    \
  [&]() -> int {                               \
    switch (lg) {                              \
      case 5: { constexpr int LG = 5; return __VA_ARGS__(); }   \
      case 6: { constexpr int LG = 6; return __VA_ARGS__(); }   \
      case 7: { constexpr int LG = 7; return __VA_ARGS__(); }   \
      case 8: { constexpr int LG = 8; return __VA_ARGS__(); }   \
      case 9: { constexpr int LG = 9; return __VA_ARGS__(); }   \
      case 10: { constexpr int LG = 10; return __VA_ARGS__(); } \
      case 11: { constexpr int LG = 11; return __VA_ARGS__(); } \
      default: { constexpr int LG = 12; return __VA_ARGS__(); } \
    }                                          \
  }()

// Pairs of columns per workgroup: one (workgroups of n/4 threads, 2N bytes
// of each row's line per die band) until there are 256 workgroups of two;
// at least a wavefront per workgroup.
template <int LG>
struct ColPairs {
  static constexpr int lo = Fft<LG>::threads * 2 < 64 ? 64 / (Fft<LG>::threads * 2) : 1;
  static constexpr int hi = LG <= 11 ? (lo > 2 ? lo : 2) : 1;
};
constexpr int kColWide = 1024;  // N from which a workgroup takes `hi` pairs

template <typename K>
static int allow_lds(K kern, size_t bytes) {
  if (bytes <= 64 * 1024) return DP_OK;
  const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e != hipSuccess) {
    set_error("spectral: %zu bytes of LDS refused: %s", bytes, hipGetErrorString(e));
    return (int)e;
  }
  return DP_OK;
}

template <typename T>
int fft_plan_fill(int M, int N, void* plan, hipStream_t s) {
  const int64_t total = (int64_t)(fft_table_elems(M) + fft_table_elems(N));
  hipLaunchKernelGGL(k_fft_tables<T>, dim3(grid_for(total, 256)), dim3(256), 0, s,
                     (typename Vec2<T>::type*)plan, M, N);
  DP_LAUNCHED("k_fft_tables");
  return DP_OK;
}

template <int LG>
static dim3 rows_grid(int count) {
  constexpr int P = Fft<LG>::threads, F = P < 64 ? 64 / P : 1;
  return dim3((unsigned)((count + F - 1) / F));
}
template <int LG>
static dim3 rows_block() {
  constexpr int P = Fft<LG>::threads;
  return dim3(P < 64 ? 64 : P);
}

template <typename T>
static int cols_transform(bool forward, const FftTables<T>& tb, int M, int N, const void* in,
                          void* out, T scale, int kind, hipStream_t s) {
  typedef typename Vec2<T>::type V;
  return DP_FFT_LOG(fft_log(M), [&]() -> int {
    auto go = [&](auto fc) -> int {
      constexpr int F = decltype(fc)::value;
      auto kern = forward ? k_fft_cols<T, LG, F, true> : k_fft_cols<T, LG, F, false>;
      const size_t lds = sizeof(V) * F * col_lds<T, LG, F>();
      DP_CHECK_RC(allow_lds(kern, lds));
      hipLaunchKernelGGL(kern, dim3((unsigned)(N / (2 * F))), dim3(F * Fft<LG>::threads), lds, s,
                         (const T*)in, (T*)out, N, scale, kind, tb.tw_m, tb.dw_m);
      DP_LAUNCHED("k_fft_cols");
      return DP_OK;
    };
    // a forward or inverse transform alone has half the threads of the
    // solve's workgroup: two pairs where that fills a wavefront
    constexpr int lo = Fft<LG>::threads < 64 ? 64 / Fft<LG>::threads : 1;
    constexpr int hi = LG <= 11 ? (lo > 2 ? lo : 2) : 1;
    if (N >= kColWide) return go(std::integral_constant<int, hi>());
    return go(std::integral_constant<int, lo>());
  });
}

template <typename T>
int fft_dct2(const void* plan, int M, int N, const void* x, void* out, void* ws, hipStream_t s) {
  const FftTables<T> tb = fft_tables<T>(plan, M, N);
  DP_CHECK_RC(DP_FFT_LOG(fft_log(N), [&]() -> int {
    hipLaunchKernelGGL((k_fft_rows_dct<T, LG, false>), rows_grid<LG>(M / 2), rows_block<LG>(), 0, s,
                       (const T*)x, (T*)ws, M / 2, (T)(2.0 / N), (double*)nullptr, tb.tw_n, tb.dw_n);
    DP_LAUNCHED("k_fft_rows_dct");
    return DP_OK;
  }));
  return cols_transform<T>(true, tb, M, N, ws, out, (T)(2.0 / M), 0, s);
}

template <typename T>
static int rows_inverse(const FftTables<T>& tb, int M, int N, const void* in, void* out, int kind,
                        hipStream_t s) {
  return DP_FFT_LOG(fft_log(N), [&]() -> int {
    hipLaunchKernelGGL((k_fft_rows_inv<T, LG, false>), rows_grid<LG>(M / 2), rows_block<LG>(), 0, s,
                       in, (T*)out, (T*)nullptr, M / 2, kind, tb.tw_n, tb.dw_n,
                       (const double*)nullptr, 0, (T*)nullptr);
    DP_LAUNCHED("k_fft_rows_inv");
    return DP_OK;
  });
}

template <typename T>
int fft_inverse(const void* plan, int M, int N, const void* x, void* out, void* ws, int kind_m,
                int kind_n, hipStream_t s) {
  const FftTables<T> tb = fft_tables<T>(plan, M, N);
  DP_CHECK_RC(rows_inverse<T>(tb, M, N, x, ws, kind_n, s));
  return cols_transform<T>(false, tb, M, N, ws, out, T(1), kind_m, s);
}

// Workspace slabs (M*N T each): 0 the row transform, 1-2 the fields' pairs,
// 3 the potential's columns, 4 the rows' means (FP64), 7 the energy partials.
template <typename T>
int fft_poisson(const void* plan, int M, int N, const void* map, double bsx, double bsy,
                bool want_phi, void* field_x, void* field_y, void* potential, void* energy,
                void* ws, size_t slab, hipStream_t s) {
  typedef typename Vec2<T>::type V;
  const FftTables<T> tb = fft_tables<T>(plan, M, N);
  char* w = (char*)ws;
  T* A = (T*)w;
  V* field = (V*)(w + slab);
  T* ph = want_phi ? (T*)(w + 3 * slab) : nullptr;
  double* row_mean = (double*)(w + 4 * slab);
  double* part = energy ? (double*)(w + 7 * slab) : nullptr;
  const double inv_area = 1.0 / (bsx * bsy);
  DP_CHECK_RC(DP_FFT_LOG(fft_log(N), [&]() -> int {
    hipLaunchKernelGGL((k_fft_rows_dct<T, LG, true>), rows_grid<LG>(M / 2), rows_block<LG>(), 0, s,
                       (const T*)map, A, M / 2, (T)(inv_area * 2.0 / N), row_mean, tb.tw_n, tb.dw_n);
    DP_LAUNCHED("k_fft_rows_dct");
    return DP_OK;
  }));
  int blocks = 0;
  DP_CHECK_RC(DP_FFT_LOG(fft_log(M), [&]() -> int {
    auto go = [&](auto fc) -> int {
      constexpr int F = decltype(fc)::value;
      auto kern = k_fft_cols_solve<T, LG, F>;
      const size_t lds = sizeof(V) * 2 * F * col_lds<T, LG, 2 * F>();
      DP_CHECK_RC(allow_lds(kern, lds));
      blocks = N / (2 * F);
      hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(2 * F * Fft<LG>::threads), lds, s,
                         (const T*)A, field, ph, N, (T)(2.0 / M), 2.0 * inv_area,
                         (const double*)row_mean, 2.0 * M_PI / M, 2.0 * M_PI / N * (bsx / bsy), part,
                         tb.tw_m, tb.dw_m);
      DP_LAUNCHED("k_fft_cols_solve");
      return DP_OK;
    };
    if (N >= kColWide) return go(std::integral_constant<int, ColPairs<LG>::hi>());
    return go(std::integral_constant<int, ColPairs<LG>::lo>());
  }));
  DP_CHECK_RC(DP_FFT_LOG(fft_log(N), [&]() -> int {
    dim3 grid = rows_grid<LG>(M);
    if (energy) ++grid.x;
    hipLaunchKernelGGL((k_fft_rows_inv<T, LG, true>), grid, rows_block<LG>(), 0, s,
                       (const void*)field, (T*)field_x, (T*)field_y, M, 0, tb.tw_n, tb.dw_n,
                       (const double*)part, blocks, (T*)energy);
    DP_LAUNCHED("k_fft_rows_inv");
    return DP_OK;
  }));
  if (want_phi) DP_CHECK_RC(rows_inverse<T>(tb, M, N, ph, potential, kInvIdct, s));
  return DP_OK;
}

#define DP_FFT_INST(T)                                                                          \
  template int fft_plan_fill<T>(int, int, void*, hipStream_t);                                  \
  template int fft_dct2<T>(const void*, int, int, const void*, void*, void*, hipStream_t);      \
  template int fft_inverse<T>(const void*, int, int, const void*, void*, void*, int, int,       \
                              hipStream_t);                                                     \
  template int fft_poisson<T>(const void*, int, int, const void*, double, double, bool, void*,  \
                              void*, void*, void*, void*, size_t, hipStream_t);

#endif  // DP_FFT_IMPL

}  // namespace dp
