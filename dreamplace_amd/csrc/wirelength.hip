// Pin positions, merged weighted-average (WA) wirelength, HPWL.
#include "dp_common.h"
#include "dp_metrics.h"
#include "dp_tiles.h"

namespace dp {

template <typename T>
__device__ __forceinline__ T tmax_value();
template <>
__device__ __forceinline__ float tmax_value<float>() { return 3.402823466e+38f; }
template <>
__device__ __forceinline__ double tmax_value<double>() { return 1.7976931348623157e+308; }

// pin_x[p] = off_x[p] + x[pin2node[p]]  (pin_pos_cuda_kernel.cu:11-26)
template <typename T, typename I>
__global__ void k_pin_pos_fwd(const T* __restrict__ x, const T* __restrict__ y,
                              const T* __restrict__ offx, const T* __restrict__ offy,
                              const I* __restrict__ pin2node, int64_t P, T* pin_x, T* pin_y) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  int64_t nd = (int64_t)pin2node[p];
  pin_x[p] = offx[p] + x[nd];
  pin_y[p] = offy[p] + y[nd];
}

// grad[n] = sum over the CSR pins of node n (pin_pos_cuda_kernel.cu:50-70);
// nodes >= num_physical (fillers) get 0.
template <typename T>
__global__ void k_pin_pos_bwd(const T* __restrict__ gpx, const T* __restrict__ gpy,
                              const int* __restrict__ flat_node2pin,
                              const int* __restrict__ node2pin_start, int64_t nphys,
                              int64_t nnodes, T* gx, T* gy) {
  int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= nnodes) return;
  T sx = 0, sy = 0;
  if (n < nphys) {
    for (int j = node2pin_start[n]; j < node2pin_start[n + 1]; ++j) {
      int p = flat_node2pin[j];
      sx += gpx[p];
      sy += gpy[p];
    }
  }
  gx[n] = sx;
  gy[n] = sy;
}

// The same for a large netlist, through tiles in LDS (dp_tiles.h): a node tile
// sends its nodes' positions to the tiles of pin order (k_tile_push), which add
// the offsets; backward, a tile of pins sends its gradients to the node tiles,
// which sum them, in the order of k_pin_pos_bwd.  The plain kernels' two random
// loads per pin, a line each whatever their size, took 325 us forward and 441
// backward at 10.9 million FP32 pins of 2.2 million nodes; one packed load or
// store per pin 189 and 194; the tiles 100 and 83.
template <typename T>
__global__ void __launch_bounds__(kTileWide) k_tile_pin_pos(
    const typename Vec2<T>::type* __restrict__ exchange, const uint16_t* __restrict__ cell,
    int pins_per_tile, int64_t P, const T* __restrict__ offx, const T* __restrict__ offy, T* pin_x,
    T* pin_y) {
  typedef typename Vec2<T>::type V;
  __shared__ V tile[TileCap<T>::value];
  const int64_t p0 = (int64_t)tile_of(blockIdx.x, gridDim.x) * pins_per_tile;
  const int count = (int)(P - p0 < pins_per_tile ? P - p0 : pins_per_tile);
  tile_load<kTileWide>(tile, exchange + p0, cell + p0, count);
  __syncthreads();
#pragma unroll 2
  for (int i = threadIdx.x; i < count; i += kTileWide) {
    const V v = tile[i];
    pin_x[p0 + i] = offx[p0 + i] + v.x;
    pin_y[p0 + i] = offy[p0 + i] + v.y;
  }
}
template <typename T>
__global__ void __launch_bounds__(kTileWide) k_tile_pin_grad(
    const T* __restrict__ gpx, const T* __restrict__ gpy, const uint16_t* __restrict__ cell,
    Runs runs, int pins_per_tile, int64_t P, typename Vec2<T>::type* exchange) {
  typedef typename Vec2<T>::type V;
  __shared__ V tile[TileCap<T>::value];
  const int t = tile_of(blockIdx.x, gridDim.x);
  const int64_t p0 = (int64_t)t * pins_per_tile;
  const int count = (int)(P - p0 < pins_per_tile ? P - p0 : pins_per_tile);
#pragma unroll 4
  for (int i = threadIdx.x; i < count; i += kTileWide) {
    V v;
    v.x = gpx[p0 + i];
    v.y = gpy[p0 + i];
    tile[i] = v;
  }
  tile_store<kTileWide, false>(tile, exchange, cell, runs, (int)p0, t, count);
}
// a node tile per workgroup, then the nodes past them (0) by the others
template <typename T>
__global__ void __launch_bounds__(kTileWide) k_tile_node_sum(
    const typename Vec2<T>::type* __restrict__ exchange, const int2* __restrict__ node_tiles,
    int ntiles, const uint16_t* __restrict__ cell, const int* __restrict__ node2pin_start,
    int64_t nphys, int64_t nnodes, T* gx, T* gy) {
  typedef typename Vec2<T>::type V;
  __shared__ V tile[TileCap<T>::value];
  if ((int)blockIdx.x >= ntiles) {
    const int64_t step = (int64_t)(gridDim.x - ntiles) * kTileWide;
    for (int64_t n = nphys + (int64_t)(blockIdx.x - ntiles) * kTileWide + threadIdx.x; n < nnodes;
         n += step)
      gx[n] = gy[n] = 0;
    return;
  }
  const int2 t0 = node_tiles[blockIdx.x], t1 = node_tiles[blockIdx.x + 1];
  const int p0 = t0.y;
  tile_load<kTileWide>(tile, exchange + p0, cell + p0, t1.y - p0);
  __syncthreads();
  for (int n = t0.x + (int)threadIdx.x; n < t1.x; n += kTileWide) {
    T sx = 0, sy = 0;
    const int e = node2pin_start[n + 1];
    for (int j = node2pin_start[n]; j < e; ++j) {
      const V v = tile[j - p0];
      sx += v.x;
      sy += v.y;
    }
    gx[n] = sx;
    gy[n] = sy;
  }
}

// ---------------------------------------------------------------------------
// The net-parallel kernels (merged WA and LSE wirelength, forward and
// recomputing backward, and HPWL) share one skeleton.  A workgroup takes 256
// consecutive nets at a time and their pins, in sub-batches that fit LDS:
//   1. a lane per pin: pin positions into LDS (coalesced over the CSR range),
//      while the nets are ordered by degree class;
//   2. a net takes 1 (up to 4 pins), 2, 4, 8 or 16 (up to 64) neighbouring
//      lanes, at most four pins in each lane's registers; extremes and sums
//      are joined by shuffles, each derivative takes its pin's place in LDS.
//      A net above 64 pins takes a wavefront, three passes over LDS;
//   3. a lane per pin: the derivatives out.
// With one thread per net for all of it, a wavefront ran its largest net's
// pins (about 50 of a mean of 4) through three passes of strided global loads
// and eight exponentials per pin: 507 us for 2.4 M nets and 9.6 M pins in
// FP32.  A thread per net between lane-per-pin steps through LDS took 205, a
// third of it vector instructions, the rest nine barriers and the 38 KB that
// held a CU to three workgroups; this form takes 148 (HPWL 128, 56, 57; LSE
// of 10 thousand nets in FP64, few workgroups of latency, 82, 22, 20).
// Every per-net expression is that of
// weighted_average_wirelength_merged.cpp:31-116; nets of up to 4 pins sum in
// pin order as there, and thread t adds net blockIdx * 256 + t's value, so the
// total's order is fixed (and HPWL's bits, whose values have no order, too).
// A net of more pins than a sub-batch holds is done by
// one thread.
// ---------------------------------------------------------------------------
enum NetModel { kNetWa = 0, kNetLse = 1, kNetHpwl = 2 };
constexpr int kNets = 256;  // nets per workgroup pass, one per thread
// pins per sub-batch: about the pins of 256 nets at 4.4 pins per net
template <typename T>
struct NetPins {
  static constexpr int value = sizeof(T) == 4 ? 1536 : 1024;
  // wavefronts per SIMD, which sets the registers: in FP32 five spill 31 of them
  // (211 us for 148)
  static constexpr int waves = sizeof(T) == 4 ? 4 : 2;
};

template <typename T>
struct NetArgs {
  const T *px, *py;      // pin positions, or (pin2node given) node positions
  const T *offx, *offy;  // with pin2node: pin position = off[p] + pos[pin2node[p]]
  const int *pin2node, *flat_netpin, *netpin_start;
  int64_t E;
  const T* w;
  const uint8_t* mask;
  const T* g_p;  // 1/gamma (WA), gamma (LSE)
  T *partial, *gix, *giy;
  double* partials;
  const uint8_t* pin_mask;  // backward
  const T* grad;            // backward
};

template <bool kNodes, typename T>
__device__ __forceinline__ void pin_at(const NetArgs<T>& a, int p, T& x, T& y) {
  if (kNodes) {
    const int nd = a.pin2node[p];
    x = a.offx[p] + a.px[nd];
    y = a.offy[p] + a.py[nd];
  } else {
    x = a.px[p];
    y = a.py[p];
  }
}

// The value of the lane O away; O < 32 needs no address register.
template <int O>
__device__ __forceinline__ float lane_xor(float v) {
  if constexpr (O == 32) return __shfl_xor(v, 32);
  return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), (O << 10) | 0x1f));
}
template <int O>
__device__ __forceinline__ double lane_xor(double v) {
  if constexpr (O == 32) return __shfl_xor(v, 32);
  return __hiloint2double(__builtin_amdgcn_ds_swizzle(__double2hiint(v), (O << 10) | 0x1f),
                          __builtin_amdgcn_ds_swizzle(__double2loint(v), (O << 10) | 0x1f));
}

template <typename T>
struct NetSums {
  T xmax, xmin, ymax, ymin;
  T xs, xns, es, ens, ys, yns, fs, fns;
  __device__ __forceinline__ void clear_extremes() {
    xmax = ymax = -tmax_value<T>();
    xmin = ymin = tmax_value<T>();
  }
  __device__ __forceinline__ void extend(T xx, T yy) {
    xmax = xx > xmax ? xx : xmax;
    xmin = xx < xmin ? xx : xmin;
    ymax = yy > ymax ? yy : ymax;
    ymin = yy < ymin ? yy : ymin;
  }
  // combine with the lane O away, where that holds pins of the same net
  template <int O>
  __device__ __forceinline__ void join_extremes(bool same) {
    const T ax = lane_xor<O>(xmax), ay = lane_xor<O>(ymax);
    const T bx = lane_xor<O>(xmin), by = lane_xor<O>(ymin);
    if (!same) return;
    // each extreme with its own kind: pins that are not a number compare nowhere,
    // and a lane of nothing but them still holds what it began with
    xmax = ax > xmax ? ax : xmax;
    ymax = ay > ymax ? ay : ymax;
    xmin = bx < xmin ? bx : xmin;
    ymin = by < ymin ? by : ymin;
  }
  template <int kModel, int O>
  __device__ __forceinline__ void join_sums(bool same) {
    auto add = [&](T& v) {
      const T u = lane_xor<O>(v);
      if (same) v += u;
    };
    if (kModel == kNetWa) {
      add(xs);
      add(xns);
      add(ys);
      add(yns);
    }
    add(es);
    add(ens);
    add(fs);
    add(fns);
  }
  __device__ __forceinline__ void clear_sums() { xs = xns = es = ens = ys = yns = fs = fns = 0; }
  template <int kModel>
  __device__ __forceinline__ void add(T xx, T yy, T ex, T enx, T ey, T eny) {
    if (kModel == kNetWa) {
      xs += xx * ex;
      xns += xx * enx;
      ys += yy * ey;
      yns += yy * eny;
    }
    es += ex;
    ens += enx;
    fs += ey;
    fns += eny;
  }
  template <int kModel>
  __device__ __forceinline__ T value(T gam) const {
    if (kModel == kNetHpwl) return xmax - xmin + ymax - ymin;
    if (kModel == kNetLse)
      return (log(es) + log(ens)) * gam + xmax - xmin + (log(fs) + log(fns)) * gam + ymax - ymin;
    return xs / es - xns / ens + ys / fs - yns / fns;
  }
  // d(value)/dx_p = (c0 + c1 x) e+ - (c2 + c3 x) e- and y with c4..c7:
  // c1 = (1/gamma)/S+, c0 = (1 - c1 XS+)/S+, c3 = -(1/gamma)/S-,
  // c2 = (1 - c3 XS-)/S- (weighted_average_wirelength_merged.cpp:94-116);
  // LSE: c0, c2, c4, c6 = 1/S
  template <int kModel>
  __device__ __forceinline__ void coefs(T ig, T (&c)[8]) const {
    if (kModel == kNetLse) {
      c[0] = (T)(1.0 / es);
      c[2] = (T)(1.0 / ens);
      c[4] = (T)(1.0 / fs);
      c[6] = (T)(1.0 / fns);
      c[1] = c[3] = c[5] = c[7] = 0;
    } else {
      c[1] = ig / es;
      c[0] = (T)((1.0 - c[1] * xs) / es);
      c[3] = -ig / ens;
      c[2] = (T)((1.0 - c[3] * xns) / ens);
      c[5] = ig / fs;
      c[4] = (T)((1.0 - c[5] * ys) / fs);
      c[7] = -ig / fns;
      c[6] = (T)((1.0 - c[7] * yns) / fns);
    }
  }
};

template <typename T>
struct alignas(4 * sizeof(T)) PinExp {
  T ex, enx, ey, eny;
};
template <typename T>
__device__ __forceinline__ PinExp<T> pin_exp(T xx, T yy, T xmax, T xmin, T ymax, T ymin, T ig) {
  return {exp((xx - xmax) * ig), exp((xmin - xx) * ig), exp((yy - ymax) * ig),
          exp((ymin - yy) * ig)};
}

// A pin's derivative: the forward's plain one, or (kBwd) ((d * grad) * w_n).
template <int kModel, bool kBwd, typename T>
__device__ __forceinline__ void pin_deriv(bool weighted, T xx, T yy, const PinExp<T>& q,
                                          const T c[8], T g, T wn, T& gx, T& gy) {
  if (kModel == kNetLse) {
    gx = q.ex * c[0] - q.enx * c[2];
    gy = q.ey * c[4] - q.eny * c[6];
  } else {
    gx = (c[0] + c[1] * xx) * q.ex - (c[2] + c[3] * xx) * q.enx;
    gy = (c[4] + c[5] * yy) * q.ey - (c[6] + c[7] * yy) * q.eny;
  }
  if (kBwd) {
    gx = gx * g;
    gy = gy * g;
    if (weighted) {
      gx *= wn;
      gy *= wn;
    }
  }
}
// and stored (kBwd: 0 under pin_mask)
template <bool kBwd, typename T>
__device__ __forceinline__ void put_pin(const NetArgs<T>& a, int p, T gx, T gy) {
  const bool off = kBwd && a.pin_mask && a.pin_mask[p];
  a.gix[p] = off ? T(0) : gx;
  a.giy[p] = off ? T(0) : gy;
}

// One net by one thread, from global memory; its value.
template <int kModel, bool kNodes, bool kBwd, typename T>
__device__ T net_serial(const NetArgs<T>& a, int b, int en, T gam, T ig, T g, T wn, bool deriv) {
  NetSums<T> n;
  T xx, yy;
  if (kModel == kNetHpwl) {
    pin_at<kNodes>(a, a.flat_netpin[b], xx, yy);
    n.xmax = n.xmin = xx;
    n.ymax = n.ymin = yy;
  } else {
    n.clear_extremes();
  }
  for (int j = b; j < en; ++j) {
    pin_at<kNodes>(a, a.flat_netpin[j], xx, yy);
    n.extend(xx, yy);
  }
  if (kModel == kNetHpwl) return n.template value<kModel>(gam);
  n.clear_sums();
  for (int j = b; j < en; ++j) {
    pin_at<kNodes>(a, a.flat_netpin[j], xx, yy);
    const PinExp<T> q = pin_exp(xx, yy, n.xmax, n.xmin, n.ymax, n.ymin, ig);
    n.template add<kModel>(xx, yy, q.ex, q.enx, q.ey, q.eny);
  }
  if (deriv) {
    T c[8];
    n.template coefs<kModel>(ig, c);
    for (int j = b; j < en; ++j) {
      const int p = a.flat_netpin[j];
      pin_at<kNodes>(a, p, xx, yy);
      T gx, gy;
      pin_deriv<kModel, kBwd>(a.w != nullptr, xx, yy,
                              pin_exp(xx, yy, n.xmax, n.xmin, n.ymax, n.ymin, ig), c, g, wn, gx, gy);
      put_pin<kBwd>(a, p, gx, gy);
    }
  }
  return n.template value<kModel>(gam);
}

// A net's degree class: lanes per net << pins per lane, largest first.
constexpr int kNetClasses = 14;
__device__ __forceinline__ int net_class(int d) {
  return d > 64   ? 0
         : d > 32 ? (d > 48 ? 1 : 2)
         : d > 16 ? (d > 24 ? 3 : 4)
         : d > 8  ? (d > 12 ? 5 : 6)
         : d > 4  ? (d > 6 ? 7 : 8)
                  : 13 - d;
}
// log2 of a class's lanes per net: 6, 4, 4, 3, 3, 2, 2, 1, 1, 0 ...
__device__ __forceinline__ int class_shift(int c) {
  return c > 8 ? 0 : (int)((0x112233446ull >> (4 * c)) & 15);
}

// One net by `L` neighbouring lanes (this one: `sub`), its d pins at xy[0 ..),
// R of them per lane at most; lmax: the wavefront's largest L.  Leaves the
// derivatives in place of the positions and returns the net's value.
template <int kModel, bool kBwd, int R, typename T>
__device__ __forceinline__ T net_lanes(typename Vec2<T>::type* xy, int d, int L, int lmax, int sub,
                                       bool deriv, bool weighted, T gam, T ig, T g, T wn) {
  typedef typename Vec2<T>::type V;
  NetSums<T> n;
  V v[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    v[r] = V();
    if (r * L + sub < d) v[r] = xy[r * L + sub];
  }
  if (kModel == kNetHpwl) {
    // the first pin as it is, later ones where they compare
    const T inf = __builtin_huge_valf();
    n.xmax = n.ymax = -inf;
    n.xmin = n.ymin = inf;
    if (sub == 0) {
      n.xmax = n.xmin = v[0].x;
      n.ymax = n.ymin = v[0].y;
    }
  } else {
    n.clear_extremes();
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (r * L + sub < d) n.extend(v[r].x, v[r].y);
  if (lmax > 1) n.template join_extremes<1>(L > 1);
  if (lmax > 2) n.template join_extremes<2>(L > 2);
  if (lmax > 4) n.template join_extremes<4>(L > 4);
  if (lmax > 8) n.template join_extremes<8>(L > 8);
  if (kModel == kNetHpwl) return n.template value<kModel>(gam);
  PinExp<T> q[R];
  n.clear_sums();
#pragma unroll
  for (int r = 0; r < R; ++r) {
    q[r] = pin_exp(v[r].x, v[r].y, n.xmax, n.xmin, n.ymax, n.ymin, ig);
    if (r * L + sub < d) n.template add<kModel>(v[r].x, v[r].y, q[r].ex, q[r].enx, q[r].ey, q[r].eny);
  }
  if (lmax > 1) n.template join_sums<kModel, 1>(L > 1);
  if (lmax > 2) n.template join_sums<kModel, 2>(L > 2);
  if (lmax > 4) n.template join_sums<kModel, 4>(L > 4);
  if (lmax > 8) n.template join_sums<kModel, 8>(L > 8);
  if (deriv) {
    T c[8];
    n.template coefs<kModel>(ig, c);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      V u;
      pin_deriv<kModel, kBwd>(weighted, v[r].x, v[r].y, q[r], c, g, wn, u.x, u.y);
      if (r * L + sub < d) xy[r * L + sub] = u;
    }
  }
  return n.template value<kModel>(gam);
}

// One net of any degree by a wavefront.
template <int kModel, bool kBwd, typename T>
__device__ __forceinline__ T net_wave(typename Vec2<T>::type* xy, int d, int lane, bool deriv,
                                      bool weighted, T gam, T ig, T g, T wn) {
  typedef typename Vec2<T>::type V;
  NetSums<T> n;
  if (kModel == kNetHpwl) {
    const T inf = __builtin_huge_valf();
    n.xmax = n.ymax = -inf;
    n.xmin = n.ymin = inf;
    if (lane == 0) {
      const V v = xy[0];
      n.xmax = n.xmin = v.x;
      n.ymax = n.ymin = v.y;
    }
  } else {
    n.clear_extremes();
  }
  for (int k = lane; k < d; k += 64) {
    const V v = xy[k];
    n.extend(v.x, v.y);
  }
  n.template join_extremes<1>(true);
  n.template join_extremes<2>(true);
  n.template join_extremes<4>(true);
  n.template join_extremes<8>(true);
  n.template join_extremes<16>(true);
  n.template join_extremes<32>(true);
  if (kModel == kNetHpwl) return n.template value<kModel>(gam);
  n.clear_sums();
  for (int k = lane; k < d; k += 64) {
    const V v = xy[k];
    const PinExp<T> q = pin_exp(v.x, v.y, n.xmax, n.xmin, n.ymax, n.ymin, ig);
    n.template add<kModel>(v.x, v.y, q.ex, q.enx, q.ey, q.eny);
  }
  n.template join_sums<kModel, 1>(true);
  n.template join_sums<kModel, 2>(true);
  n.template join_sums<kModel, 4>(true);
  n.template join_sums<kModel, 8>(true);
  n.template join_sums<kModel, 16>(true);
  n.template join_sums<kModel, 32>(true);
  if (deriv) {
    T c[8];
    n.template coefs<kModel>(ig, c);
    for (int k = lane; k < d; k += 64) {
      const V v = xy[k];
      V u;
      pin_deriv<kModel, kBwd>(weighted, v.x, v.y,
                              pin_exp(v.x, v.y, n.xmax, n.xmin, n.ymax, n.ymin, ig), c, g, wn, u.x,
                              u.y);
      xy[k] = u;
    }
  }
  return n.template value<kModel>(gam);
}

template <typename T, int kModel, bool kNodes, bool kBwd>
__global__ void __launch_bounds__(kNets, NetPins<T>::waves) k_nets(NetArgs<T> a) {
  typedef typename Vec2<T>::type V;
  constexpr int CP = NetPins<T>::value, PT = CP / kNets, W = kNets / 64;
  constexpr bool kExp = kModel != kNetHpwl;
  __shared__ V s_xy[CP];
  __shared__ int s_b[kNets], s_en[kNets];
  __shared__ uint8_t s_order[kNets];        // the live nets, by class
  __shared__ T s_val[kNets];
  __shared__ int s_cnt[W][16];
  __shared__ unsigned s_dead[CP / 32];      // pins of nets without a value
  __shared__ double smem[4];
  int t = threadIdx.x;
  int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const T gam = kModel == kNetLse ? *a.g_p : T(0);
  const T ig = kModel == kNetLse ? T(1) / gam : kExp ? *a.g_p : T(0);
  const T g = kBwd ? *a.grad : T(0);
  const bool deriv = kBwd || (kExp && a.gix != nullptr);
  double contrib = 0;
  // every condition around a barrier below is uniform over the workgroup
  for (int64_t e0 = (int64_t)blockIdx.x * kNets; e0 < a.E; e0 += (int64_t)gridDim.x * kNets) {
    const int cnt = a.E - e0 < kNets ? (int)(a.E - e0) : kNets;
    const int64_t e = e0 + t;
    int b = 0, en = 0;
    bool live = false;
    if (t < cnt) {
      b = a.netpin_start[e];
      en = a.netpin_start[e + 1];
      live = a.mask[e] != 0 && (kExp || en > b);
      if (!live && kExp && !kBwd && a.partial) a.partial[e] = 0;
    }
    __syncthreads();  // the last pass's readers of the per-net arrays are done
    s_b[t] = b;
    s_en[t] = en;
    __syncthreads();
    for (int lo = 0; lo < cnt;) {
      const int p0 = s_b[lo];
      // what follows from the lane is formed again, not kept in registers
      asm volatile("" : "+v"(lane), "+v"(t));
      // the nets [lo, hi) whose pins fit (the starts ascend)
      const int fit = __syncthreads_count(t >= lo && t < cnt && en - p0 <= CP);
      if (fit == 0) {
        if (t == lo && live) {
          const T wn = a.w ? a.w[e] : T(1);
          const T v = net_serial<kModel, kNodes, kBwd>(a, b, en, gam, ig, g, wn, deriv);
          if (kExp && !kBwd && a.partial) a.partial[e] = v;
          if (!kBwd) contrib += (double)(a.w ? v * wn : v);
        }
        ++lo;
        continue;
      }
      const int hi = lo + fit, np = s_en[hi - 1] - p0;
      const bool mine = t >= lo && t < hi;
      // 1. the pins' positions, under way while the nets are counted
      int pin[PT];
      V at[PT];
#pragma unroll
      for (int i = 0; i < PT; ++i) {
        const int k = t + i * kNets;
        pin[i] = k < np ? a.flat_netpin[p0 + k] : 0;
      }
#pragma unroll
      for (int i = 0; i < PT; ++i) {
        const int k = t + i * kNets;
        if (k < np) pin_at<kNodes>(a, pin[i], at[i].x, at[i].y);
      }
      const int cls = mine && live ? net_class(en - b) : 15;
      int rank = 0, count = 0;
#pragma unroll
      for (int c = 0; c < kNetClasses; ++c) {
        const uint64_t m = __ballot(cls == c);
        if (cls == c) rank = __popcll(m & ((1ull << lane) - 1));
        if (lane == c) count = __popcll(m);
      }
      if (lane < 16) s_cnt[wave][lane] = count;
      if (t < CP / 32) s_dead[t] = 0;
#pragma unroll
      for (int i = 0; i < PT; ++i) {
        const int k = t + i * kNets;
        if (k < np) s_xy[k] = at[i];
        asm volatile("" : "+v"(pin[i]));
      }
      __syncthreads();
      // lane c: the first item and the first lane of class c
      int total = 0, before = 0;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const int n = s_cnt[w][lane & 15];
        if (w < wave) before += n;
        total += n;
      }
      const int own = (lane & 15) < kNetClasses ? total << class_shift(lane & 15) : 0;
      int items = total, lanes = own;
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) {
        const int from = 4 * (lane - o);
        const int ui = __builtin_amdgcn_ds_bpermute(from, items);
        const int ul = __builtin_amdgcn_ds_bpermute(from, lanes);
        if ((lane & 15) >= o) {
          items += ui;
          lanes += ul;
        }
      }
      const int all = __builtin_amdgcn_readlane(lanes, kNetClasses - 1);
      items -= total;
      lanes -= own;
      const int at_item = __shfl(items + before, cls);
      if (mine && live) s_order[at_item + rank] = (uint8_t)t;
      if (mine && !live) {
        for (int k = b - p0; k < en - p0; ++k) atomicOr(&s_dead[k >> 5], 1u << (k & 31));
      }
      __syncthreads();
      // 2. the nets, by their lanes
      for (int q0 = 64 * wave; q0 < all; q0 += kNets) {
        const int q = q0 + lane;
        int c = 0;  // the last class that begins at or before q
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) {
          const int k = c + o < kNetClasses ? c + o : kNetClasses - 1;
          if (q >= __shfl(lanes, k)) c = k;
        }
        const int sh = class_shift(c), L = 1 << sh;
        const int from = q - __shfl(lanes, c), item = __shfl(items, c) + (from >> sh);
        const bool on = q < all;
        const int u = on ? s_order[item] : 0;
        const int kb = on ? s_b[u] - p0 : 0, d = on ? s_en[u] - p0 - kb : 0;
        const int lmax = __builtin_amdgcn_readfirstlane(L);
        const bool weighted = a.w != nullptr;
        const T wn = weighted && on ? a.w[e0 + u] : T(1);
        const int sub = from & (L - 1);
        T v;
        if (lmax == 64) {
          v = net_wave<kModel, kBwd, T>(s_xy + kb, d, lane, deriv, weighted, gam, ig, g, wn);
        } else {
          const int r = __ballot(d > 3 * L) ? 4 : __ballot(d > 2 * L) ? 3 : __ballot(d > L) ? 2 : 1;
#define DP_NET_LANES(R) \
  v = net_lanes<kModel, kBwd, R, T>(s_xy + kb, d, L, lmax, sub, deriv, weighted, gam, ig, g, wn)
          switch (r) {
            case 1: DP_NET_LANES(1); break;
            case 2: DP_NET_LANES(2); break;
            case 3: DP_NET_LANES(3); break;
            default: DP_NET_LANES(4);
          }
#undef DP_NET_LANES
        }
        if (!kBwd && on && sub == 0) s_val[u] = v;
      }
      __syncthreads();
      if (!kBwd && mine && live) {
        const T v = s_val[t];
        if (kExp && a.partial) a.partial[e] = v;
        contrib += (double)(a.w ? v * a.w[e] : v);
      }
      // 3. the derivatives
      if (deriv) {
#pragma unroll
        for (int i = 0; i < PT; ++i) {
          const int k = t + i * kNets;
          if (k < np && !(s_dead[k >> 5] >> (k & 31) & 1)) {
            const V v = s_xy[k];
            put_pin<kBwd>(a, pin[i], v.x, v.y);
          }
        }
      }
      __syncthreads();  // the next sub-batch overwrites LDS
      lo = hi;
    }
  }
  if (!kBwd) {
    const double bs = block_sum<kNets>(contrib, smem);
    if (t == 0) a.partials[blockIdx.x] = bs;
  }
}

// g[p] = (gi[p]*grad)*w[net(p)] for unmasked nets; 0 where pin_mask
// (weighted_average_wirelength_cuda_merged.cpp:135, integrateNetWeights,
// weighted_average_wirelength.py:207-208).
// Four pins a thread, their loads (the net's weight hangs on the pin's net) in
// flight together: 9.6 million FP32 pins 68 -> 48 us.
constexpr int kBwdPins = 4;
template <typename T>
__global__ void __launch_bounds__(256) k_wa_bwd(const T* __restrict__ grad, T* gi, int64_t P,
                                                const int* __restrict__ pin2net,
                                                const T* __restrict__ w,
                                                const uint8_t* __restrict__ net_mask,
                                                const uint8_t* __restrict__ pin_mask) {
  const int64_t p0 = (int64_t)blockIdx.x * (256 * kBwdPins) + threadIdx.x;
  const T g = *grad;
  T gx[kBwdPins], gy[kBwdPins], wn[kBwdPins];
  int n[kBwdPins];
  bool live[kBwdPins], masked[kBwdPins];
#pragma unroll
  for (int u = 0; u < kBwdPins; ++u) {
    const int64_t p = p0 + 256 * u;
    if (p >= P) continue;
    gx[u] = gi[p];
    gy[u] = gi[P + p];
    n[u] = w ? pin2net[p] : 0;
    masked[u] = pin_mask && pin_mask[p];
  }
#pragma unroll
  for (int u = 0; u < kBwdPins; ++u) {
    if (!w || p0 + 256 * u >= P) continue;
    live[u] = net_mask[n[u]] != 0;
    wn[u] = w[n[u]];
  }
#pragma unroll
  for (int u = 0; u < kBwdPins; ++u) {
    const int64_t p = p0 + 256 * u;
    if (p >= P) continue;
    T x = gx[u] * g, y = gy[u] * g;
    if (w && live[u]) {
      x *= wn[u];
      y *= wn[u];
    }
    gi[p] = masked[u] ? T(0) : x;
    gi[P + p] = masked[u] ? T(0) : y;
  }
}

template <typename T>
__global__ void k_wa_wgrad(const T* __restrict__ grad, const T* __restrict__ partial,
                           const uint8_t* __restrict__ mask, int64_t E, T* out) {
  int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= E) return;
  out[e] = mask[e] ? (*grad) * partial[e] : T(0);
}

// Fused WA backward + pin_pos backward + gradient combine, node-parallel:
// g[n] = sum over the CSR pins p of n of (pin_mask[p] ? 0 : (gi[p]*grad)*w[net(p)])
//        + add[n]
// Per pin this is the arithmetic of k_wa_bwd, and the pins are summed in CSR
// order as k_pin_pos_bwd does, so the result equals the unfused sequence.
template <typename T>
__global__ void k_wa_pin_pos_bwd(const T* __restrict__ gix, const T* __restrict__ giy,
                                 const T* __restrict__ grad, const int* __restrict__ flat_node2pin,
                                 const int* __restrict__ node2pin_start,
                                 const int* __restrict__ pin2net, const T* __restrict__ w,
                                 const uint8_t* __restrict__ net_mask,
                                 const uint8_t* __restrict__ pin_mask, const T* __restrict__ add,
                                 int64_t nphys, int64_t nnodes, T* gx, T* gy) {
  int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= nnodes) return;
  const T g = *grad;
  T sx = 0, sy = 0;
  if (n < nphys) {
    for (int j = node2pin_start[n]; j < node2pin_start[n + 1]; ++j) {
      int p = flat_node2pin[j];
      if (pin_mask && pin_mask[p]) {
        sx += T(0);
        sy += T(0);
        continue;
      }
      T px = gix[p] * g, py = giy[p] * g;
      if (w) {
        int e = pin2net[p];
        if (net_mask[e]) {
          T wn = w[e];
          px *= wn;
          py *= wn;
        }
      }
      sx += px;
      sy += py;
    }
  }
  if (add) {
    sx += add[n];
    sy += add[nnodes + n];
  }
  gx[n] = sx;
  gy[n] = sy;
}

// dp_hpwl's weighted FP64 sum over per-net HPWL values computed elsewhere
// (the pin-parallel WA pass): the same grid, loop order, mask test and
// empty-net test, so the total is bit-identical to dp_hpwl's on the positions
// the values came from.
template <typename T>
__global__ void __launch_bounds__(256) k_hpwl_nets(const T* __restrict__ h_net,
                                                   const int* __restrict__ netpin_start, int64_t E,
                                                   const T* __restrict__ w,
                                                   const uint8_t* __restrict__ mask,
                                                   double* partials) {
  __shared__ double smem[4];
  hpwl_nets_partial(blockIdx.x, gridDim.x, h_net, netpin_start, E, w, mask, partials, smem);
}

template <typename T>
static NetArgs<T> net_args(const T* pin_pos, int64_t num_pins, const int32_t* flat_netpin,
                           const int32_t* netpin_start, int64_t num_nets, const void* w,
                           const uint8_t* mask, const void* g_p, void* partial, void* gi,
                           double* partials) {
  NetArgs<T> a = {};
  a.px = pin_pos;
  a.py = pin_pos + num_pins;
  a.flat_netpin = (const int*)flat_netpin;
  a.netpin_start = (const int*)netpin_start;
  a.E = num_nets;
  a.w = (const T*)w;
  a.mask = mask;
  a.g_p = (const T*)g_p;
  a.partial = (T*)partial;
  a.gix = (T*)gi;
  a.giy = gi ? (T*)gi + num_pins : nullptr;
  a.partials = partials;
  return a;
}

}  // namespace dp

using namespace dp;

extern "C" {

int dp_pin_pos_forward(int dtype, const void* pos, int64_t num_nodes, const void* pin_offset_x,
                       const void* pin_offset_y, const void* pin2node_map, int index_type,
                       int64_t num_pins, void* pin_pos_out, void* stream) {
  DP_ARG(pos && pin_offset_x && pin_offset_y && pin2node_map && pin_pos_out,
         "dp_pin_pos_forward: null pointer");
  DP_ARG(index_type == DP_INDEX_INT32 || index_type == DP_INDEX_INT64,
         "dp_pin_pos_forward: bad index type");
  if (num_pins == 0) return DP_OK;
  hipStream_t s = S(stream);
  return DP_DISPATCH(dtype, "dp_pin_pos_forward", [&] {
    const T* P = (const T*)pos;
    T* out = (T*)pin_pos_out;
    dim3 g((unsigned)ceil_div(num_pins, 256)), b(256);
    if (index_type == DP_INDEX_INT32)
      DP_PROBED(DP_KERNEL_PIN_POS_FORWARD, s,
                hipLaunchKernelGGL((k_pin_pos_fwd<T, int>), g, b, 0, s, P, P + num_nodes,
                                   (const T*)pin_offset_x, (const T*)pin_offset_y,
                                   (const int*)pin2node_map, num_pins, out, out + num_pins));
    else
      DP_PROBED(DP_KERNEL_PIN_POS_FORWARD, s,
                hipLaunchKernelGGL((k_pin_pos_fwd<T, long long>), g, b, 0, s, P, P + num_nodes,
                                   (const T*)pin_offset_x, (const T*)pin_offset_y,
                                   (const long long*)pin2node_map, num_pins, out,
                                   out + num_pins));
    DP_LAUNCHED("k_pin_pos_fwd");
    return DP_OK;
  });
}

int dp_pin_pos_backward(int dtype, const void* grad_pin_pos, int64_t num_pins,
                        const int32_t* flat_node2pin_map, const int32_t* flat_node2pin_start_map,
                        int64_t num_physical_nodes, int64_t num_nodes, void* grad_pos_out,
                        void* stream) {
  DP_ARG(grad_pin_pos && flat_node2pin_map && flat_node2pin_start_map && grad_pos_out,
         "dp_pin_pos_backward: null pointer");
  DP_ARG(num_physical_nodes <= num_nodes, "dp_pin_pos_backward: num_physical_nodes > num_nodes");
  if (num_nodes == 0) return DP_OK;
  hipStream_t s = S(stream);
  return DP_DISPATCH(dtype, "dp_pin_pos_backward", [&] {
    const T* g = (const T*)grad_pin_pos;
    T* out = (T*)grad_pos_out;
    DP_PROBED(DP_KERNEL_PIN_POS_BACKWARD, s,
              hipLaunchKernelGGL(k_pin_pos_bwd<T>, dim3((unsigned)ceil_div(num_nodes, 256)),
                                 dim3(256), 0, s, g, g + num_pins, (const int*)flat_node2pin_map,
                                 (const int*)flat_node2pin_start_map, num_physical_nodes,
                                 num_nodes, out, out + num_nodes));
    DP_LAUNCHED("k_pin_pos_bwd");
    return DP_OK;
  });
}

size_t dp_pin_pos_workspace_bytes(int dtype, int64_t count) {
  return align256((dtype == DP_FLOAT64 ? 16 : 8) * (size_t)(count > 0 ? count : 1));
}

int dp_pin_pos_forward_tiles(int dtype, const void* pos, int64_t num_nodes,
                             const void* pin_offset_x, const void* pin_offset_y, int64_t num_pins,
                             const int32_t* node_tiles, int64_t num_node_tiles,
                             const uint16_t* place_node, const int32_t* node_chunk,
                             const int32_t* node_delta, int64_t pins_per_tile, const uint16_t* pin_cell,
                             void* workspace, void* pin_pos_out, void* stream) {
  const char* name = "dp_pin_pos_forward_tiles";
  DP_ARG(pos && pin_offset_x && pin_offset_y && node_tiles && place_node && node_chunk &&
             node_delta && pin_cell && workspace && pin_pos_out,
         "%s: null pointer", name);
  DP_ARG(num_pins >= 0 && num_pins < ((int64_t)1 << 31) && num_node_tiles >= 0 &&
             num_node_tiles <= kTileMax && pins_per_tile > 0 &&
             pins_per_tile <= kTileBytes / (dtype == DP_FLOAT64 ? 16 : 8),
         "%s: bad counts", name);
  if (num_pins == 0) return DP_OK;
  hipStream_t s = S(stream);
  return DP_DISPATCH(dtype, name, [&] {
    typedef typename Vec2<T>::type V;
    const T* P = (const T*)pos;
    T* out = (T*)pin_pos_out;
    hipLaunchKernelGGL((k_tile_push<T, false>), dim3((unsigned)num_node_tiles), dim3(kTileWide), 0,
                       s, P, P + num_nodes, (const int2*)node_tiles, place_node,
                       (const V*)nullptr, Runs{node_chunk, node_delta}, (V*)workspace);
    DP_LAUNCHED("k_tile_push");
    DP_PROBED(DP_KERNEL_PIN_POS_FORWARD, s,
              hipLaunchKernelGGL(k_tile_pin_pos<T>,
                                 dim3((unsigned)ceil_div(num_pins, (int)pins_per_tile)),
                                 dim3(kTileWide), 0, s, (const V*)workspace, pin_cell,
                                 (int)pins_per_tile, num_pins, (const T*)pin_offset_x,
                                 (const T*)pin_offset_y, out, out + num_pins));
    DP_LAUNCHED("k_tile_pin_pos");
    return DP_OK;
  });
}

int dp_pin_pos_backward_tiles(int dtype, const void* grad_pin_pos, int64_t num_pins,
                              int64_t pins_per_tile, const uint16_t* pin_cell,
                              const int32_t* pin_chunk, const int32_t* pin_delta,
                              const int32_t* node_tiles,
                              int64_t num_node_tiles, const uint16_t* node_cell,
                              const int32_t* flat_node2pin_start_map, int64_t num_physical_nodes,
                              int64_t num_nodes, void* workspace, void* grad_pos_out,
                              void* stream) {
  const char* name = "dp_pin_pos_backward_tiles";
  DP_ARG(grad_pin_pos && pin_cell && pin_chunk && pin_delta && node_tiles && node_cell &&
             flat_node2pin_start_map && workspace && grad_pos_out,
         "%s: null pointer", name);
  DP_ARG(num_physical_nodes <= num_nodes, "%s: num_physical_nodes > num_nodes", name);
  DP_ARG(num_pins >= 0 && num_pins < ((int64_t)1 << 31) && num_node_tiles >= 0 &&
             num_node_tiles <= kTileMax && pins_per_tile > 0 &&
             pins_per_tile <= kTileBytes / (dtype == DP_FLOAT64 ? 16 : 8),
         "%s: bad counts", name);
  if (num_nodes == 0) return DP_OK;
  hipStream_t s = S(stream);
  return DP_DISPATCH(dtype, name, [&] {
    typedef typename Vec2<T>::type V;
    const T* g = (const T*)grad_pin_pos;
    T* out = (T*)grad_pos_out;
    if (num_pins > 0) {
      hipLaunchKernelGGL(k_tile_pin_grad<T>,
                         dim3((unsigned)ceil_div(num_pins, (int)pins_per_tile)), dim3(kTileWide),
                         0, s, g, g + num_pins, pin_cell, Runs{pin_chunk, pin_delta},
                         (int)pins_per_tile, num_pins, (V*)workspace);
      DP_LAUNCHED("k_tile_pin_grad");
    }
    const int64_t rest = ceil_div(num_nodes - num_physical_nodes, kTileWide);
    const int64_t nb = num_node_tiles + (rest < kTileRestGrid ? rest : kTileRestGrid);
    DP_PROBED(DP_KERNEL_PIN_POS_BACKWARD, s,
              hipLaunchKernelGGL(k_tile_node_sum<T>, dim3((unsigned)(nb > 0 ? nb : 1)),
                                 dim3(kTileWide), 0, s, (const V*)workspace,
                                 (const int2*)node_tiles, (int)num_node_tiles, node_cell,
                                 (const int*)flat_node2pin_start_map, num_physical_nodes,
                                 num_nodes, out, out + num_nodes));
    DP_LAUNCHED("k_tile_node_sum");
    return DP_OK;
  });
}

size_t dp_wa_workspace_bytes(int64_t num_nets) {
  (void)num_nets;
  return reduce_slot_bytes();
}

int dp_wa_merged_forward(int dtype, const void* pin_pos, int64_t num_pins,
                         const int32_t* flat_netpin, const int32_t* netpin_start,
                         int64_t num_nets, const void* net_weights, const uint8_t* net_mask,
                         const void* inv_gamma, void* partial_wl, void* grad_intermediate,
                         void* wl_out, void* workspace, void* stream) {
  DP_ARG(pin_pos && flat_netpin && netpin_start && net_mask && inv_gamma && wl_out && workspace,
         "dp_wa_merged_forward: null pointer");
  hipStream_t s = S(stream);
  DP_PROBE_OP(DP_OP_WA_FORWARD, s);
  double* partials = (double*)workspace;
  int grid = reduce_grid(num_nets);
  return DP_DISPATCH(dtype, "dp_wa_merged_forward", [&] {
    const T* pp = (const T*)pin_pos;
    void* gi = grad_intermediate;
    DP_PROBED(DP_KERNEL_WA_FORWARD, s,
              hipLaunchKernelGGL((k_nets<T, kNetWa, false, false>), dim3(grid), dim3(kNets), 0, s,
                                 net_args<T>(pp, num_pins, flat_netpin, netpin_start, num_nets,
                                             net_weights, net_mask, inv_gamma, partial_wl, gi,
                                             partials)));
    DP_LAUNCHED("k_nets");
    return finish_reduction(partials, grid, 1, nullptr, wl_out, dtype, s);
  });
}

int dp_lse_merged_forward(int dtype, const void* pin_pos, int64_t num_pins,
                          const int32_t* flat_netpin, const int32_t* netpin_start,
                          int64_t num_nets, const void* net_weights, const uint8_t* net_mask,
                          const void* gamma, void* partial_wl, void* grad_intermediate,
                          void* wl_out, void* workspace, void* stream) {
  DP_ARG(pin_pos && flat_netpin && netpin_start && net_mask && gamma && grad_intermediate &&
             wl_out && workspace,
         "dp_lse_merged_forward: null pointer");
  hipStream_t s = S(stream);
  DP_PROBE_OP(DP_OP_WA_FORWARD, s);
  double* partials = (double*)workspace;
  int grid = reduce_grid(num_nets);
  return DP_DISPATCH(dtype, "dp_lse_merged_forward", [&] {
    const T* pp = (const T*)pin_pos;
    void* gi = grad_intermediate;
    DP_PROBED(DP_KERNEL_WA_FORWARD, s,
              hipLaunchKernelGGL((k_nets<T, kNetLse, false, false>), dim3(grid), dim3(kNets), 0, s,
                                 net_args<T>(pp, num_pins, flat_netpin, netpin_start, num_nets,
                                             net_weights, net_mask, gamma, partial_wl, gi,
                                             partials)));
    DP_LAUNCHED("k_nets");
    return finish_reduction(partials, grid, 1, nullptr, wl_out, dtype, s);
  });
}

int dp_wa_merged_backward(int dtype, const void* grad, void* grad_intermediate, int64_t num_pins,
                          const int32_t* pin2net_map, const void* net_weights,
                          const uint8_t* net_mask, const uint8_t* pin_mask, void* stream) {
  DP_ARG(grad && grad_intermediate, "dp_wa_merged_backward: null pointer");
  DP_ARG(!net_weights || (pin2net_map && net_mask),
         "dp_wa_merged_backward: net weights need pin2net_map and net_mask");
  if (num_pins == 0) return DP_OK;
  hipStream_t s = S(stream);
  return DP_DISPATCH(dtype, "dp_wa_merged_backward", [&] {
    DP_PROBED(DP_KERNEL_WA_BACKWARD, s,
              hipLaunchKernelGGL(k_wa_bwd<T>, dim3((unsigned)ceil_div(num_pins, 256 * kBwdPins)), dim3(256),
                                 0, s, (const T*)grad, (T*)grad_intermediate, num_pins,
                                 (const int*)pin2net_map, (const T*)net_weights, net_mask,
                                 pin_mask));
    DP_LAUNCHED("k_wa_bwd");
    return DP_OK;
  });
}

int dp_wa_merged_backward_recompute(int dtype, const void* grad, const void* pin_pos,
                                    int64_t num_pins, const int32_t* flat_netpin,
                                    const int32_t* netpin_start, int64_t num_nets,
                                    const void* net_weights, const uint8_t* net_mask,
                                    const uint8_t* pin_mask, const void* inv_gamma,
                                    void* grad_pin_pos, void* stream) {
  DP_ARG(grad && pin_pos && flat_netpin && netpin_start && net_mask && inv_gamma && grad_pin_pos,
         "dp_wa_merged_backward_recompute: null pointer");
  if (num_nets == 0) return DP_OK;
  hipStream_t s = S(stream);
  int grid = reduce_grid(num_nets);
  return DP_DISPATCH(dtype, "dp_wa_merged_backward_recompute", [&] {
    const T* pp = (const T*)pin_pos;
    NetArgs<T> a = net_args<T>(pp, num_pins, flat_netpin, netpin_start, num_nets, net_weights,
                               net_mask, inv_gamma, nullptr, grad_pin_pos, nullptr);
    a.pin_mask = pin_mask;
    a.grad = (const T*)grad;
    DP_PROBED(DP_KERNEL_WA_BACKWARD, s,
              hipLaunchKernelGGL((k_nets<T, kNetWa, false, true>), dim3(grid), dim3(kNets), 0, s,
                                 a));
    DP_LAUNCHED("k_nets backward");
    return DP_OK;
  });
}

int dp_wa_net_weight_grad(int dtype, const void* grad, const void* partial_wl,
                          const uint8_t* net_mask, int64_t num_nets, void* grad_net_weights,
                          void* stream) {
  DP_ARG(grad && partial_wl && net_mask && grad_net_weights, "dp_wa_net_weight_grad: null pointer");
  if (num_nets == 0) return DP_OK;
  hipStream_t s = S(stream);
  return DP_DISPATCH(dtype, "dp_wa_net_weight_grad", [&] {
    hipLaunchKernelGGL(k_wa_wgrad<T>, dim3((unsigned)ceil_div(num_nets, 256)), dim3(256), 0, s,
                       (const T*)grad, (const T*)partial_wl, net_mask, num_nets,
                       (T*)grad_net_weights);
    DP_LAUNCHED("k_wa_wgrad");
    return DP_OK;
  });
}

int dp_wa_forward_from_nodes(int dtype, const void* pos, int64_t num_nodes,
                             const void* pin_offset_x, const void* pin_offset_y,
                             const int32_t* pin2node_map, int64_t num_pins,
                             const int32_t* flat_netpin, const int32_t* netpin_start,
                             int64_t num_nets, const void* net_weights, const uint8_t* net_mask,
                             const void* inv_gamma, void* partial_wl, void* grad_intermediate,
                             void* wl_out, void* workspace, void* stream) {
  DP_ARG(pos && pin_offset_x && pin_offset_y && pin2node_map && flat_netpin && netpin_start &&
             net_mask && inv_gamma && grad_intermediate && wl_out && workspace,
         "dp_wa_forward_from_nodes: null pointer");
  hipStream_t s = S(stream);
  DP_PROBE_OP(DP_OP_WA_FORWARD, s);
  double* partials = (double*)workspace;
  int grid = reduce_grid(num_nets);
  return DP_DISPATCH(dtype, "dp_wa_forward_from_nodes", [&] {
    NetArgs<T> a = net_args<T>((const T*)pos, num_pins, flat_netpin, netpin_start, num_nets,
                               net_weights, net_mask, inv_gamma, partial_wl, grad_intermediate,
                               partials);
    a.py = a.px + num_nodes;
    a.offx = (const T*)pin_offset_x;
    a.offy = (const T*)pin_offset_y;
    a.pin2node = (const int*)pin2node_map;
    DP_PROBED(DP_KERNEL_WA_FORWARD, s,
              hipLaunchKernelGGL((k_nets<T, kNetWa, true, false>), dim3(grid), dim3(kNets), 0, s,
                                 a));
    DP_LAUNCHED("k_nets from nodes");
    return finish_reduction(partials, grid, 1, nullptr, wl_out, dtype, s);
  });
}

int dp_wa_backward_to_nodes(int dtype, const void* grad, const void* grad_intermediate,
                            int64_t num_pins, const int32_t* flat_node2pin_map,
                            const int32_t* flat_node2pin_start_map, const int32_t* pin2net_map,
                            const void* net_weights, const uint8_t* net_mask,
                            const uint8_t* pin_mask, const void* add, int64_t num_physical_nodes,
                            int64_t num_nodes, void* grad_pos_out, void* stream) {
  DP_ARG(grad && grad_intermediate && flat_node2pin_map && flat_node2pin_start_map &&
             grad_pos_out,
         "dp_wa_backward_to_nodes: null pointer");
  DP_ARG(!net_weights || (pin2net_map && net_mask),
         "dp_wa_backward_to_nodes: net weights need pin2net_map and net_mask");
  DP_ARG(num_physical_nodes <= num_nodes, "dp_wa_backward_to_nodes: bad node counts");
  if (num_nodes == 0) return DP_OK;
  hipStream_t s = S(stream);
  DP_PROBE_OP(DP_OP_NODE_GRAD, s);
  return DP_DISPATCH(dtype, "dp_wa_backward_to_nodes", [&] {
    const T* gi = (const T*)grad_intermediate;
    T* out = (T*)grad_pos_out;
    DP_PROBED(DP_KERNEL_PIN_POS_BACKWARD, s,
              hipLaunchKernelGGL(k_wa_pin_pos_bwd<T>, dim3((unsigned)ceil_div(num_nodes, 256)),
                                 dim3(256), 0, s, gi, gi + num_pins, (const T*)grad,
                                 (const int*)flat_node2pin_map,
                                 (const int*)flat_node2pin_start_map, (const int*)pin2net_map,
                                 (const T*)net_weights, net_mask, pin_mask, (const T*)add,
                                 num_physical_nodes, num_nodes, out, out + num_nodes));
    DP_LAUNCHED("k_wa_pin_pos_bwd");
    return DP_OK;
  });
}

int dp_hpwl(int dtype, const void* pin_pos, int64_t num_pins, const int32_t* flat_netpin,
            const int32_t* netpin_start, int64_t num_nets, const void* net_weights,
            const uint8_t* net_mask, void* workspace, double* hpwl_out, void* stream) {
  DP_ARG(pin_pos && flat_netpin && netpin_start && net_mask && workspace && hpwl_out,
         "dp_hpwl: null pointer");
  hipStream_t s = S(stream);
  double* partials = (double*)workspace;
  int grid = reduce_grid(num_nets);
  return DP_DISPATCH(dtype, "dp_hpwl", [&] {
    const T* pp = (const T*)pin_pos;
    hipLaunchKernelGGL((k_nets<T, kNetHpwl, false, false>), dim3(grid), dim3(kNets), 0, s,
                       net_args<T>(pp, num_pins, flat_netpin, netpin_start, num_nets, net_weights,
                                   net_mask, nullptr, nullptr, nullptr, partials));
    DP_LAUNCHED("k_nets hpwl");
    return finish_reduction(partials, grid, 1, nullptr, hpwl_out, -1, s);
  });
}

int dp_hpwl_from_nets(int dtype, const void* net_hpwl, const int32_t* netpin_start,
                      int64_t num_nets, const void* net_weights, const uint8_t* net_mask,
                      void* workspace, double* hpwl_out, void* stream) {
  DP_ARG(net_hpwl && netpin_start && net_mask && workspace && hpwl_out,
         "dp_hpwl_from_nets: null pointer");
  DP_ARG(num_nets >= 0, "dp_hpwl_from_nets: bad size");
  hipStream_t s = S(stream);
  double* partials = (double*)workspace;
  int grid = reduce_grid(num_nets);
  return DP_DISPATCH(dtype, "dp_hpwl_from_nets", [&] {
    hipLaunchKernelGGL(k_hpwl_nets<T>, dim3(grid), dim3(256), 0, s, (const T*)net_hpwl,
                       (const int*)netpin_start, num_nets, (const T*)net_weights, net_mask,
                       partials);
    DP_LAUNCHED("k_hpwl_nets");
    return finish_reduction(partials, grid, 1, nullptr, hpwl_out, -1, s);
  });
}

}  // extern "C"
