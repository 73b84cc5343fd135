// kernels.hip -- gfx950 kernels of the direct-summation engine.
//
//   k_prep        one launch before the force kernel: staged j-updates -> FP64
//                 SoA store + predicted records (reference dev_copy_particles,
//                 kernels.cu:245-301), FP64 Horner predictor of the other
//                 j-particles (dev_predictor, kernels.cu:307-411), the call's
//                 inputs from pinned host memory, and the reset of the neighbour
//                 counters (dev_reset_buffers, kernels.cu:1109-1144).
//   k_scatter, k_predict   the same work as launches of their own, for captured
//                 graphs (their arguments stay fixed) and the allocation-free call.
//   k_force       acc / pot / jerk [/ snap] + nearest neighbour + neighbour list
//                 (dev_evaluate_gravity_*, kernels.cu:552-1041).  One wave owns P
//                 i-particles held in registers and Q = 64/P j-lanes per
//                 i-particle over one contiguous j-range (the "j-split").  With
//                 P = 64 every lane of a wave reads the same j, so the j-record
//                 is fetched once per wave through the scalar cache into SGPRs
//                 and feeds the VALU directly.  Mixed precision: double-single
//                 positions, relative positions and pair terms in FP32,
//                 per-tile FP32 sums folded into FP64 accumulators.
//   k_finalize    deterministic fixed-order reduction of the S partial sums,
//                 nearest-neighbour selection, neighbour-list sort and packing;
//                 results and packed lists are written straight into
//                 host-mapped pinned memory (no copy command per call).
//
// Built with -ffp-contract=off: every fused multiply-add below is explicit.
#include "kernels.h"

#include <algorithm>
#include <climits>
#include <cmath>
#include <type_traits>

namespace sapk {

template <int ORDER, bool F64> struct RecOf;
template <> struct RecOf<ORDER_H4, false> { using T = JRecM4; };
template <> struct RecOf<ORDER_H6, false> { using T = JRecM6; };
template <> struct RecOf<ORDER_H4, true> { using T = JRecD4; };
template <> struct RecOf<ORDER_H6, true> { using T = JRecD6; };

static_assert(sizeof(JRecM4) == 48, "record layout");
static_assert(sizeof(JRecM6) == 64, "record layout");
static_assert(sizeof(JRecD4) == 64, "record layout");
static_assert(sizeof(JRecD6) == 96, "record layout");

// Double-single split (reference DSX::operator=(double), kernels.cu:163-167).
__device__ __forceinline__ DSF to_ds(double x) {
  DSF d;
  d.hi = (float)x;
  d.lo = (float)(x - (double)d.hi);
  return d;
}
__device__ __forceinline__ void put_pos(double& dst, double x) { dst = x; }
__device__ __forceinline__ void put_pos(DSF& dst, double x) { dst = to_ds(x); }

// Working-precision record from FP64 values.
template <int ORDER, bool F64>
__device__ __forceinline__ typename RecOf<ORDER, F64>::T make_rec(double x, double y, double z, double m, double vx,
                                                                  double vy, double vz, double ax, double ay,
                                                                  double az, int id) {
  using Rec = typename RecOf<ORDER, F64>::T;
  using R = typename std::conditional<F64, double, float>::type;
  Rec r{};
  put_pos(r.x, x); put_pos(r.y, y); put_pos(r.z, z);
  r.m = (R)m; r.vx = (R)vx; r.vy = (R)vy; r.vz = (R)vz;
  if constexpr (ORDER >= ORDER_H6) { r.ax = (R)ax; r.ay = (R)ay; r.az = (R)az; }
  r.id = id;
  return r;
}

// Write the predicted state of address j: the working-precision record and, in
// mixed precision, the FP64 state kept for read-back.  Returns the record.
template <int ORDER, bool F64>
__device__ __forceinline__ typename RecOf<ORDER, F64>::T put_pred(const StoreView& st, int j, const double p[3], const double v[3],
                                         const double ac[3], double m, int id) {
  const size_t cap = (size_t)st.cap;
  const auto r = make_rec<ORDER, F64>(p[0], p[1], p[2], m, v[0], v[1], v[2], ac[0], ac[1], ac[2], id);
  reinterpret_cast<typename RecOf<ORDER, F64>::T*>(st.rec)[j] = r;
  if constexpr (!F64) {
    st.ppos[j] = p[0]; st.ppos[cap + j] = p[1]; st.ppos[2 * cap + j] = p[2];
    st.pvel[j] = v[0]; st.pvel[cap + j] = v[1]; st.pvel[2 * cap + j] = v[2];
    if constexpr (ORDER >= ORDER_H6) {
      st.pacc[j] = ac[0]; st.pacc[cap + j] = ac[1]; st.pacc[2 * cap + j] = ac[2];
    }
  }
  return r;
}

// ---------------------------------------------------------------------------
// Scatter of staged updates (+ neighbour counter reset).
template <int ORDER, bool F64>
__global__ __launch_bounds__(256) void k_scatter(ScatterArgs a) {
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  const int stride = gridDim.x * blockDim.x;
  const int ni_reset = a.cd->ni_reset, nupd = a.cd->nupd;
  for (int k = tid; k < ni_reset; k += stride) a.ngb_cnt[k] = 0;
  if (tid == 0 && ni_reset > 0 && a.pack_ctr) *a.pack_ctr = 0;
  const size_t cap = (size_t)a.st.cap;
  for (int k = tid; k < nupd; k += stride) {
    const double* u = a.upd + (size_t)k * (a.nf + 1);
    const int2 pair = *reinterpret_cast<const int2*>(u + a.nf);  // address, id
    const int addr = pair.x;
    const int id = pair.y;
    if (addr < 0 || addr >= a.st.cap) continue;  // host guarantees range
    for (int f = 0; f < a.nf; ++f) a.st.raw[(size_t)f * cap + addr] = u[f];
    a.st.id[addr] = id;
    // widen the tile's id range (conservative until the next prediction recomputes it)
    atomicMin(&a.st.idr[addr / JTILE].x, id);
    atomicMax(&a.st.idr[addr / JTILE].y, id);
    // predicted = raw for updated particles (kernels.cu:281-298), unless the
    // predictor that follows rewrites this address anyway
    if (addr < a.pred_j1) continue;
    const double p[3] = {u[RF_X], u[RF_Y], u[RF_Z]}, v[3] = {u[RF_VX], u[RF_VY], u[RF_VZ]};
    double ac[3] = {0, 0, 0};
    if constexpr (ORDER >= ORDER_H6) { ac[0] = u[RF_AX]; ac[1] = u[RF_AY]; ac[2] = u[RF_AZ]; }
    put_pred<ORDER, F64>(a.st, addr, p, v, ac, u[RF_M], id);
  }
}

// ---------------------------------------------------------------------------
// FP64 predictor.  The expression is the reference's (kernels.cu:332-383),
// evaluated without contraction, including the zero terms for FOURTH order.
// get(f) is the particle's raw field f.
template <int ORDER, typename G>
__device__ __forceinline__ void predict_one(const G& get, double ti, double p[3], double v[3], double ac[3]) {
  const double dt = ti - get(RF_T);
  const double dt2 = (1. / 2.) * dt;
  const double dt3 = (1. / 3.) * dt;
  double dt4 = (1. / 4.) * dt;
  double dt5 = (1. / 5.) * dt;
  if constexpr (ORDER <= ORDER_H4) { dt4 = 0; dt5 = 0; }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double xs = get(RF_X + d);
    const double vs = get(RF_VX + d);
    const double as = get(RF_AX + d);
    const double js = get(RF_JX + d);
    double ss = 0.0, cs = 0.0;
    if constexpr (ORDER >= ORDER_H6) { ss = get(RF_SX + d); cs = get(RF_CX + d); }
    p[d] = xs + dt * (vs + dt2 * (as + dt3 * (js + dt4 * (ss + dt5 * (cs)))));
    v[d] = vs + dt * (as + dt2 * (js + dt3 * (ss + dt4 * (cs))));
    ac[d] = as;
    if constexpr (ORDER >= ORDER_H6) ac[d] = as + dt * (js + dt2 * (ss + dt3 * (cs)));
  }
}

// Exact id range of the wave's tile (a wave holds the JTILE addresses of one
// tile); addresses past the predicted range are included so that later calls
// with a larger nj stay covered.
__device__ __forceinline__ void tile_id_range(const StoreView& st, int j) {
  const int id = j < st.cap ? st.id[j] : 0;
  int lo = j < st.cap ? id : INT_MAX, hi = j < st.cap ? id : INT_MIN;
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    lo = min(lo, __shfl_xor(lo, m));
    hi = max(hi, __shfl_xor(hi, m));
  }
  if ((threadIdx.x & 63) == 0 && j < st.cap) st.idr[j / JTILE] = make_int2(lo, hi);
}

template <int ORDER, bool F64>
__global__ __launch_bounds__(256) void k_predict(PredictArgs a) {
  const int j = a.j0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (!a.cd && blockIdx.x == 0 && threadIdx.x == 0) *a.desc_out = a.desc;
  const double ti = a.cd ? a.cd->ti : a.desc.ti;
  tile_id_range(a.st, j);
  if (j >= a.j1) return;
  const size_t cap = (size_t)a.st.cap;
  double p[3], v[3], ac[3];
  predict_one<ORDER>([&](int f) { return a.st.raw[f * cap + j]; }, ti, p, v, ac);
  put_pred<ORDER, F64>(a.st, j, p, v, ac, a.st.raw[RF_M * cap + j], a.st.id[j]);
}

// Everything a call needs before its force kernel, in one launch.  It replaces
// two copy commands, the scatter and the predictor: their run times (3, 4, 4 and
// 7 us at N = 131072) were less than the 5-8 us gaps between them.  A call of one
// i-particle went from 58 to 40 us, one of 333 from 149 to 119 us.  Bound by
// launch and PCIe latency, not by bandwidth (10.4 us for 28 MB at N = 131072).  The predictor skips the addresses whose
// bit is set: the work-group that holds such an update writes its stored fields
// and its predicted record from the staged row, so the roles never write the
// same address and need no order among them.  The tile id ranges are the
// predictor's alone: a call whose updates change an id, or are many, runs the
// updates in a launch of their own before it.
template <int ORDER, bool F64>
__global__ __launch_bounds__(256) void k_prep(PrepArgs a) {
  constexpr int NF = raw_fields(ORDER), NR = NF + 1;
  __shared__ double buf[PREP_ROWS * NR];
  const int t = threadIdx.x;
  const size_t cap = (size_t)a.st.cap;
  int b = blockIdx.x;
  if (b < a.nb_upd) {
    const int k0 = b * PREP_ROWS, n = min(PREP_ROWS, a.nupd - k0);
    // whole lines over PCIe: the group's rows are one contiguous range
    for (int e = t; e < n * NR; e += 256) {
      const size_t o = (size_t)k0 * NR + e;
      buf[e] = o < (size_t)a.nd * NR ? a.rows_d[o] : a.rows_h[o];
    }
    __syncthreads();
    const int r = t & (PREP_ROWS - 1);
    if (r >= n) return;
    const double* u = buf + r * NR;
    const int2 pair = *reinterpret_cast<const int2*>(u + NF);  // address, id
    const int addr = pair.x;
    if (addr < 0 || addr >= a.st.cap) return;  // host guarantees range
    for (int f = t / PREP_ROWS; f < NF; f += 256 / PREP_ROWS) a.st.raw[(size_t)f * cap + addr] = u[f];
    if (t >= PREP_ROWS) return;
    if (a.new_ids) {
      a.st.id[addr] = pair.y;
      atomicMin(&a.st.idr[addr / JTILE].x, pair.y);
      atomicMax(&a.st.idr[addr / JTILE].y, pair.y);
    }
    // predicted = stored for addresses that are not predicted (kernels.cu:281-298)
    double p[3] = {u[RF_X], u[RF_Y], u[RF_Z]}, v[3] = {u[RF_VX], u[RF_VY], u[RF_VZ]}, ac[3] = {0, 0, 0};
    if constexpr (ORDER >= ORDER_H6) { ac[0] = u[RF_AX]; ac[1] = u[RF_AY]; ac[2] = u[RF_AZ]; }
    if (addr < a.pred_j1) predict_one<ORDER>([&](int f) { return u[f]; }, a.ti, p, v, ac);
    put_pred<ORDER, F64>(a.st, addr, p, v, ac, u[RF_M], pair.y);
    return;
  }
  b -= a.nb_upd;
  if (b < a.nb_copy) {
    const int stride = a.nb_copy * 256;
    auto copy = [&](const int4* __restrict__ src, int4* __restrict__ dst, int n16) {
      int k = b * 256 + t;
      for (; k + 3 * stride < n16; k += 4 * stride) {  // four reads over PCIe in flight
        const int4 v0 = src[k], v1 = src[k + stride], v2 = src[k + 2 * stride], v3 = src[k + 3 * stride];
        dst[k] = v0; dst[k + stride] = v1; dst[k + 2 * stride] = v2; dst[k + 3 * stride] = v3;
      }
      for (; k < n16; k += stride) dst[k] = src[k];
    };
    static_assert(PREP_SEGS == 4, "segments");
    copy(a.seg[0].src, a.seg[0].dst, a.seg[0].n16);
    copy(a.seg[1].src, a.seg[1].dst, a.seg[1].n16);
    copy(a.seg[2].src, a.seg[2].dst, a.seg[2].n16);
    copy(a.seg[3].src, a.seg[3].dst, a.seg[3].n16);
    for (int k = b * 256 + t; k < a.ni_reset; k += stride) a.ngb_cnt[k] = 0;
    if (b == 0 && t == 0 && a.ni_reset > 0) *a.pack_ctr = 0;
    return;
  }
  b -= a.nb_copy;
  const int j = b * 256 + t;
  // the stored fields are loaded while the bits come over PCIe
  double raw[NF];
  if (j < a.pred_j1) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
      if (f != RF_DT && f != RF_EPS) raw[f] = a.st.raw[(size_t)f * cap + j];
  }
  const bool skip = j < a.nbits && (a.bits[j >> 5] >> (j & 31) & 1u);
  tile_id_range(a.st, j);
  if (j >= a.pred_j1 || skip) return;
  double p[3], v[3], ac[3];
  predict_one<ORDER>([&](int f) { return raw[f]; }, a.ti, p, v, ac);
  put_pred<ORDER, F64>(a.st, j, p, v, ac, raw[RF_M], a.st.id[j]);
}

// ---------------------------------------------------------------------------
// Force kernel.
template <typename R> __device__ __forceinline__ R fmaR(R a, R b, R c);
template <> __device__ __forceinline__ float fmaR<float>(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
template <> __device__ __forceinline__ double fmaR<double>(double a, double b, double c) { return __builtin_fma(a, b, c); }

// 1/sqrt: v_rsq_f32 (1 ulp) in FP32; in FP64 v_rsq_f64 plus one cubic
// correction step, full double precision for the positive normal operands
// used here (r2 >= eps2 > 0; other cases are masked by the caller).
template <typename R> __device__ __forceinline__ R rsq(R x);
template <> __device__ __forceinline__ float rsq<float>(float x) { return __builtin_amdgcn_rsqf(x); }
template <> __device__ __forceinline__ double rsq<double>(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-x * y, y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}

// Relative coordinate xj - xi: FP64 subtraction, or the double-single
// difference (xj.hi - xi.hi) + (xj.lo - xi.lo) in FP32 (kernels.cu:170-178).
__device__ __forceinline__ double to_rel(double xj, double xi) { return xj - xi; }
__device__ __forceinline__ float to_rel(const DSF& xj, const DSF& xi) { return (xj.hi - xi.hi) + (xj.lo - xi.lo); }

template <typename R> struct PosOf { using T = DSF; };
template <> struct PosOf<double> { using T = double; };
__device__ __forceinline__ void get_pos(double& dst, double x) { dst = x; }
__device__ __forceinline__ void get_pos(DSF& dst, double x) { dst = to_ds(x); }

// Per-lane state of one i-particle.
template <int ORDER, typename R>
struct IState {
  typename PosOf<R>::T x, y, z;
  R vx, vy, vz, ax, ay, az, h2;
  int id, i;
};

template <int ORDER, typename R, bool NGB>
__device__ __forceinline__ IState<ORDER, R> load_i(const double* __restrict__ ipos, const double* __restrict__ ivel,
                                                   const double* __restrict__ iacc, const double* __restrict__ ih2,
                                                   const int* __restrict__ iid, int il, bool valid) {
  IState<ORDER, R> st;
  get_pos(st.x, ipos[3 * il]); get_pos(st.y, ipos[3 * il + 1]); get_pos(st.z, ipos[3 * il + 2]);
  st.vx = (R)ivel[3 * il]; st.vy = (R)ivel[3 * il + 1]; st.vz = (R)ivel[3 * il + 2];
  st.ax = st.ay = st.az = R(0);
  if constexpr (ORDER >= ORDER_H6) {
    st.ax = (R)iacc[3 * il]; st.ay = (R)iacc[3 * il + 1]; st.az = (R)iacc[3 * il + 2];
  }
  st.h2 = (NGB && valid) ? (R)ih2[il] : R(-1);
  st.id = iid[il];
  st.i = il;
  return st;
}

template <typename R> __device__ __forceinline__ R minR(R a, R b);
template <> __device__ __forceinline__ float minR<float>(float a, float b) { return __builtin_fminf(a, b); }
template <> __device__ __forceinline__ double minR<double>(double a, double b) { return __builtin_fmin(a, b); }

// Relative position and squared distance of one pair, the arithmetic every
// distance test uses (the nearest-neighbour resolution recomputes it and must
// agree bit for bit).
template <typename R, typename Rec, typename St>
__device__ __forceinline__ R pair_ds2(const Rec& r, const St& s, R& dx, R& dy, R& dz) {
  dx = to_rel(r.x, s.x);
  dy = to_rel(r.y, s.y);
  dz = to_rel(r.z, s.z);
  return fmaR<R>(dz, dz, fmaR<R>(dy, dy, dx * dx));
}

constexpr int NF4 = 7, NF6 = 10;
template <int ORDER> constexpr int nf() { return ORDER >= ORDER_H6 ? NF6 : NF4; }

// One pair interaction (kernels.cu:565-667) accumulated into t[].  Nearest
// neighbour: with BLOCKMIN, dsmin receives the pair's squared distance (+inf
// for an excluded pair) for the caller's group minimum; otherwise dsmin and
// nnaddr hold the distance and the address j of the nearest so far.
template <int ORDER, bool NGB, bool CHECK, bool BLOCKMIN, typename R, typename Rec>
__device__ __forceinline__ bool pair(const Rec& r, const int j, const bool ok, const IState<ORDER, R>& s,
                                     const R eps2, R (&t)[nf<ORDER>()], R& dsmin, int& nnaddr) {
  R dx, dy, dz;
  const R ds2 = pair_ds2<R>(r, s, dx, dy, dz);
  // bitwise & keeps the predicates branch-free (no exec-masked regions)
  const bool use = CHECK ? (ok & (r.id != s.id)) : ok;
  const R inv0 = rsq<R>(ds2 + eps2);
  const R inv = use ? inv0 : R(0);
  const R invr2 = inv * inv;
  const R mr1 = r.m * inv;
  const R mr3 = mr1 * invr2;
  t[0] = fmaR<R>(mr3, dx, t[0]);
  t[1] = fmaR<R>(mr3, dy, t[1]);
  t[2] = fmaR<R>(mr3, dz, t[2]);
  t[3] = t[3] - mr1;
  const R dvx = r.vx - s.vx;
  const R dvy = r.vy - s.vy;
  const R dvz = r.vz - s.vz;
  const R rv = fmaR<R>(dz, dvz, fmaR<R>(dy, dvy, dx * dvx));
  if constexpr (ORDER == ORDER_H4) {
    // jerk += m/r^3 dv - 3 (m/r^3)(dr.dv)/r^2 dr   (kernels.cu:633-636)
    const R q = (rv * invr2) * R(-3);
    t[4] = fmaR<R>(mr3, fmaR<R>(q, dx, dvx), t[4]);
    t[5] = fmaR<R>(mr3, fmaR<R>(q, dy, dvy), t[5]);
    t[6] = fmaR<R>(mr3, fmaR<R>(q, dz, dvz), t[6]);
  } else {
    // kernels.cu:642-667: alpha = dr.dv/r^2, beta = (dv^2 + dr.da)/r^2 + alpha^2
    const R dax = r.ax - s.ax;
    const R day = r.ay - s.ay;
    const R daz = r.az - s.az;
    const R v2 = fmaR<R>(dvz, dvz, fmaR<R>(dvy, dvy, dvx * dvx));
    const R v2ra = fmaR<R>(dz, daz, fmaR<R>(dy, day, fmaR<R>(dx, dax, v2)));
    const R alpha = rv * invr2;
    const R beta = fmaR<R>(v2ra, invr2, alpha * alpha);
    const R m3a = alpha * R(-3);
    // jerk_ij = m/r^3 w, w = dv - 3 alpha dr
    const R wx = fmaR<R>(m3a, dx, dvx);
    const R wy = fmaR<R>(m3a, dy, dvy);
    const R wz = fmaR<R>(m3a, dz, dvz);
    t[4] = fmaR<R>(mr3, wx, t[4]);
    t[5] = fmaR<R>(mr3, wy, t[5]);
    t[6] = fmaR<R>(mr3, wz, t[6]);
    // snap_ij = m/r^3 (da - 3 beta dr) - 6 alpha jerk_ij; the products are formed
    // inside the sums (58.75 operations a pair, 61.75 with jerk_ij and v^2 + dr.da
    // as values of their own)
    const R m3b = beta * R(-3);
    const R m6 = (alpha * mr3) * R(-6);
    t[7] = fmaR<R>(m6, wx, fmaR<R>(mr3, fmaR<R>(m3b, dx, dax), t[7]));
    t[8] = fmaR<R>(m6, wy, fmaR<R>(mr3, fmaR<R>(m3b, dy, day), t[8]));
    t[9] = fmaR<R>(m6, wz, fmaR<R>(mr3, fmaR<R>(m3b, dz, daz), t[9]));
  }
  // nearest neighbour: strict <, first address wins inside a lane (kernels.cu:539-546)
  if constexpr (BLOCKMIN) {
    dsmin = CHECK ? (use ? ds2 : R(INFINITY)) : ds2;
  } else {
    const bool better = use & (ds2 < dsmin);
    dsmin = better ? ds2 : dsmin;
    nnaddr = better ? j : nnaddr;
  }
  // neighbour predicate h2_i > ds2 (kernels.cu:584); the caller appends
  return NGB & use & (s.h2 > ds2);
}

// Append to the i-particle's list; rare (~32 per 1e5 pairs), so a global atomic
// takes the slots.  The count stays exact past NGB_CAP; a lane that has met a
// full list only counts (over >= 0) and adds its count at the end, so that an
// i-particle with most of the system inside its radius does not serialise the
// launch on one counter (777 i x 30011 j with one such particle: 284 us of
// which the pairs are 90).
struct NgbList {
  int* __restrict__ cnt;
  int* __restrict__ list;
  int i;
  int over;  // -1: the list may have room
  __device__ __forceinline__ void add(int id) {
    if (over >= 0) { ++over; return; }
    const int k = atomicAdd(&cnt[i], 1);
    if (k < NGB_CAP) list[(size_t)i * NGB_CAP + k] = id;
    else over = 0;
  }
  // the pairs u of a group with nb[u], ids through id(u): their slots in one atomic
  template <typename F> __device__ __forceinline__ void add4(const bool (&nb)[4], const F& id) {
    const int c = (int)nb[0] + (int)nb[1] + (int)nb[2] + (int)nb[3];
    if (c == 0) return;
    if (over >= 0) { over += c; return; }
    int k = atomicAdd(&cnt[i], c);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (nb[u] && k < NGB_CAP) list[(size_t)i * NGB_CAP + k] = id(u);
      k += nb[u] ? 1 : 0;
    }
    if (k >= NGB_CAP) over = 0;
  }
  __device__ __forceinline__ void finish() {
    if (over > 0) atomicAdd(&cnt[i], over);
  }
};

// Neighbour slots reserved by one group whose id stores are still pending.
struct PendingNgb {
  int k[4], id[4];
  bool m[4];
};

// Store the ids of the previous group (their slot atomics were issued one
// group earlier, so the atomic latency overlaps this group's arithmetic).
__device__ __forceinline__ void ngb_flush(PendingNgb& p, int* __restrict__ ngb_list, int i) {
  if (p.m[0] | p.m[1] | p.m[2] | p.m[3]) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (p.m[u] && p.k[u] < NGB_CAP) ngb_list[(size_t)i * NGB_CAP + p.k[u]] = p.id[u];
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) p.m[u] = false;
}

// Empty register constraint: the values are computed before this point.
template <int ORDER, typename R>
__device__ __forceinline__ void settle(R (&t)[nf<ORDER>()]) {
#pragma unroll
  for (int f = 0; f < nf<ORDER>(); ++f) asm volatile("" : "+v"(t[f]));
}

// Four consecutive j of one lane with a single neighbour branch for the group.
// The group's arithmetic is settled before the branch; otherwise the compiler
// sinks it below the (rarely taken) append block and keeps the four relative
// positions live across it, which costs a wave of occupancy.
template <int ORDER, bool NGB, bool CHECK, int Q, bool PIPE, typename R, typename Rec>
__device__ __forceinline__ void pair4(const Rec* __restrict__ rec, const int j0, const IState<ORDER, R>& s,
                                      const R eps2, R (&t)[nf<ORDER>()], R& smin, NgbList& ngb, PendingNgb& pend) {
  R d[4];
  int idj[4];
  int unused = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int j = j0 + u * Q;
    const Rec& r = rec[j];
    idj[u] = r.id;
    pair<ORDER, NGB, CHECK, true>(r, j, true, s, eps2, t, d[u], unused);
  }
  // the group's nearest distance: it lowers the sub-block minimum, and h2 > it
  // is the test whether any of the four pairs is a neighbour
  const R g = minR<R>(minR<R>(minR<R>(d[0], d[1]), d[2]), d[3]);
  smin = minR<R>(smin, g);
  if constexpr (NGB) settle<ORDER>(t);
  // without lists, keep the scheduler from hoisting the scalar loads of a whole
  // unrolled sub-block (they exhaust the SGPRs and spill)
  if constexpr (!NGB) __builtin_amdgcn_sched_barrier(0);
  const bool any = NGB && __ballot(s.h2 > g) != 0;
  if constexpr (NGB && PIPE) {
    ngb_flush(pend, ngb.list, s.i);
    if (any) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const bool nb = s.h2 > d[u];
        if (nb) pend.k[u] = atomicAdd(&ngb.cnt[s.i], 1);
        pend.id[u] = idj[u];
        pend.m[u] = nb;
      }
    }
  } else if constexpr (NGB) {
    if (any) {
#pragma unroll
      for (int u = 0; u < 4; ++u) asm volatile("" : "+v"(d[u]));
      const bool nb[4] = {s.h2 > d[0], s.h2 > d[1], s.h2 > d[2], s.h2 > d[3]};
      ngb.add4(nb, [&](int u) { return rec[j0 + u * Q].id; });
    }
  }
}

constexpr int KT = 64;  // interactions per lane between FP64 folds
constexpr int SUB = FORCE_SUB;
static_assert(KT % SUB == 0 && SUB % 4 == 0, "fold");

// J-records on their way through the scalar cache (lane shape P = 64): JU
// consecutive records held in SGPRs, as one or two wide scalar loads.  Units lie at
// multiples of their size, which is what the loads' types claim: 96-byte units are
// aligned to 32 bytes, not to the 64 of a 16-register load.
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef v16i v16i_at32 __attribute__((aligned(32)));
template <typename Rec> struct JUnit {
  static constexpr int JU = sizeof(Rec) == 48 ? 2 : 1;
  static constexpr bool TAIL = sizeof(Rec) * JU == 96;
  static_assert(sizeof(Rec) * JU % (TAIL ? alignof(v16i_at32) : alignof(v16i)) == 0 &&
                sizeof(Rec) * JU % alignof(v8i) == 0, "unit alignment");
  v16i h;
  v8i t;
  __device__ __forceinline__ void load(const Rec* __restrict__ p) {
    if constexpr (TAIL) {
      h = *reinterpret_cast<const v16i_at32*>(p);
      t = *reinterpret_cast<const v8i*>(reinterpret_cast<const char*>(p) + 64);
    } else {
      h = *reinterpret_cast<const v16i*>(p);
    }
  }
  // The loads have arrived (scalar loads return out of order: a wait is for
  // all of them, so this comes before the next unit's loads are issued).
  __device__ __forceinline__ void arrive() {
    asm volatile("" : "+s"(h));
    if constexpr (TAIL) asm volatile("" : "+s"(t));
  }
  __device__ __forceinline__ Rec get(int u) const {
    struct { v16i h; v8i t; } b{h, t};
    Rec r;
    __builtin_memcpy(&r, reinterpret_cast<const char*>(&b) + u * sizeof(Rec), sizeof(Rec));
    return r;
  }
};

// Four consecutive j of a wave whose lanes share the j-record (Q = 1): the
// arithmetic of pair4, with the records of the next pairs loaded while the
// present ones are computed.  a holds the first unit of the group on entry and
// the first unit of the next group (at jnext) on return.
template <int ORDER, bool NGB, bool CHECK, typename R, typename Rec>
__device__ __forceinline__ void group4(const Rec* __restrict__ rec, const int j0, const int jnext, JUnit<Rec>& a,
                                       const IState<ORDER, R>& s, const R eps2, R (&t)[nf<ORDER>()], R& smin,
                                       NgbList& ngb) {
  constexpr int JU = JUnit<Rec>::JU;
  R d[4];
  int unused = 0;
  JUnit<Rec> b;
#pragma unroll
  for (int u = 0; u < 4; u += 2 * JU) {
    a.arrive();
    __builtin_amdgcn_sched_barrier(0);
    b.load(rec + j0 + u + JU);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < JU; ++k)
      pair<ORDER, NGB, CHECK, true>(a.get(k), 0, true, s, eps2, t, d[u + k], unused);
    b.arrive();
    __builtin_amdgcn_sched_barrier(0);
    a.load(rec + (u + 2 * JU < 4 ? j0 + u + 2 * JU : jnext));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < JU; ++k)
      pair<ORDER, NGB, CHECK, true>(b.get(k), 0, true, s, eps2, t, d[u + JU + k], unused);
  }
  const R g = minR<R>(minR<R>(minR<R>(d[0], d[1]), d[2]), d[3]);
  smin = minR<R>(smin, g);
  if constexpr (NGB) {
    settle<ORDER>(t);
    if (__ballot(s.h2 > g) != 0) {
      const bool nb[4] = {s.h2 > d[0], s.h2 > d[1], s.h2 > d[2], s.h2 > d[3]};
      ngb.add4(nb, [&](int u) { return rec[j0 + u].id; });
    }
  }
}

// The work of one wave: i-particles [i0, i0 + icount) (icount <= P) against
// j in [jb, je), Q = 64/P j-lanes per i-particle.  On return the lanes with
// writer set hold the wave-reduced FP64 sums T, nearest-neighbour (ds2,
// address) and their i-slot.
// AHEAD (P = 64): the records of the next pairs are loaded while the present
// ones are computed.
template <int ORDER, bool F64, int P, bool NGB, bool PIPE = false, bool AHEAD = false>
__device__ __forceinline__ void wave_force(
    const typename RecOf<ORDER, F64>::T* __restrict__ rec, const int2* __restrict__ idr,
    const double* __restrict__ ipos, const double* __restrict__ ivel, const double* __restrict__ iacc,
    const double* __restrict__ ih2, const int* __restrict__ iid, const int i0, const int icount,
    const int jb, const int je, const double eps2d, int* __restrict__ ngb_cnt, int* __restrict__ ngb_list,
    double (&T)[nf<ORDER>()], double& dsd, int& nnaddr, int& islot, bool& writer) {
  using R = typename std::conditional<F64, double, float>::type;
  using Rec = typename RecOf<ORDER, F64>::T;
  constexpr int Q = 64 / P;
  constexpr int NF = nf<ORDER>();
  const int lane = threadIdx.x & 63;
  islot = (Q == 1) ? lane : (lane % P);
  const int jsub = (Q == 1) ? 0 : (lane / P);
  const bool ivalid = islot < icount;
  const int il = i0 + (ivalid ? islot : 0);

  const IState<ORDER, R> st = load_i<ORDER, R, NGB>(ipos, ivel, iacc, ih2, iid, il, ivalid);
  const R eps2 = (R)eps2d;

#pragma unroll
  for (int f = 0; f < NF; ++f) T[f] = 0.0;
  NgbList ngb{ngb_cnt, ngb_list, il, -1};
  R dsmin = R(INFINITY);
  // nearest pair so far: -1 none; >= 0 the first address of the sub-block of
  // 16 pairs (whole tiles) that holds it; <= -2 the exact address a, as -2 - a
  // (the partial tile at the end of the range)
  int nnblk = -1;
  PendingNgb pend;
#pragma unroll
  for (int u = 0; u < 4; ++u) { pend.m[u] = false; pend.k[u] = 0; pend.id[u] = 0; }

  const int nk = (je > jb) ? (je - jb + Q - 1) / Q : 0;  // iterations of the lane with jsub 0
  const int nw = (je > jb) ? (je - jb) / Q : 0;          // iterations that every lane has
  // FP32 pair terms are summed per fold of KT and folded into FP64 T; in FP64
  // the pair terms go straight into t, which becomes T at the end
  R t[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) t[f] = R(0);
  JUnit<Rec> ja;
  const int jend = jb + nw / SUB * SUB;  // AHEAD: end of the whole sub-blocks, loads stay below it
  if constexpr (AHEAD) ja.load(rec + (nw >= SUB ? jb : 0));
  for (int k0 = 0; k0 < nk; k0 += KT) {
    if constexpr (!F64) {
#pragma unroll
      for (int f = 0; f < NF; ++f) t[f] = R(0);
    }
    const int kn = min(KT, nk - k0);
    // whole sub-blocks of SUB iterations; what is left of the range's end goes pair by pair
    const int kw = min(KT, nw - k0) / SUB * SUB;
    const int jt = jb + k0 * Q + jsub;
    if (kw > 0) {
      // P = 64: the fold's j lie in at most two tiles; skip the self test when
      // no lane's id can occur in them
      bool check = true;
      if constexpr (Q == 1) {
        const int2 r0 = idr[jt / JTILE], r1 = idr[(jt + kw - 1) / JTILE];
        check = __ballot(st.id >= min(r0.x, r1.x) && st.id <= max(r0.y, r1.y)) != 0;
      }
      // Nearest neighbour: each pair only lowers the minimum of its sub-block of
      // 16 pairs (one v_min); a sub-block that beats the lane's nearest so far
      // records its first address, resolved to the pair after the loop.
      auto sweep = [&](auto chk) {
        for (int k = 0; k < kw; k += SUB) {
          R sm = R(INFINITY);
#pragma unroll
          for (int q = 0; q < SUB; q += 4) {
            const int j = jt + (k + q) * Q;
            if constexpr (AHEAD)
              group4<ORDER, NGB, decltype(chk)::value>(rec, j, j + 4 < jend ? j + 4 : jb, ja, st, eps2, t, sm, ngb);
            else
              pair4<ORDER, NGB, decltype(chk)::value, Q, PIPE>(rec, j, st, eps2, t, sm, ngb, pend);
          }
          const bool better = sm < dsmin;
          dsmin = better ? sm : dsmin;
          nnblk = better ? jt + k * Q : nnblk;
        }
      };
      if (check) sweep(std::true_type{});
      else sweep(std::false_type{});
    }
    if (kw < kn) {
      if constexpr (NGB && PIPE) ngb_flush(pend, ngb.list, st.i);
      const R before = dsmin;
      int cand = 0;
      for (int k = max(kw, 0); k < kn; ++k) {
        const int j = jt + k * Q;
        const bool ok = j < je;
        const Rec& r = rec[ok ? j : jb];
        if (pair<ORDER, NGB, true, false>(r, j, ok, st, eps2, t, dsmin, cand)) ngb.add(r.id);
      }
      if (dsmin < before) nnblk = -2 - cand;  // a later pair, strictly nearer: its address is exact
    }
    if constexpr (!F64) {
#pragma unroll
      for (int f = 0; f < NF; ++f) T[f] += (double)t[f];
    }
  }
  if constexpr (F64) {
#pragma unroll
    for (int f = 0; f < NF; ++f) T[f] = (double)t[f];
  }
  // The nearest pair is the first of its sub-block at distance dsmin: a
  // sub-block replaced the candidate only when strictly nearer, so this is the
  // lane's first address at the minimum, as the per-pair rule gives.
  nnaddr = nnblk <= -2 ? -2 - nnblk : INT_MAX;
  if (nnblk >= 0) {
    bool found = false;
    for (int u = 0; u < SUB; ++u) {
      const int j = nnblk + u * Q;
      const Rec& r = rec[j];
      R dx, dy, dz;
      const R d2 = pair_ds2<R>(r, st, dx, dy, dz);
      const bool hit = !found && (r.id != st.id) && d2 == dsmin;
      nnaddr = hit ? j : nnaddr;
      found = found || hit;
    }
  }

  if constexpr (NGB && PIPE) ngb_flush(pend, ngb.list, st.i);
  if constexpr (NGB) ngb.finish();
  dsd = (double)dsmin;
  if constexpr (Q > 1) {
#pragma unroll
    for (int m = P; m < 64; m <<= 1) {
#pragma unroll
      for (int f = 0; f < NF; ++f) T[f] += __shfl_xor(T[f], m);
      const double od = __shfl_xor(dsd, m);
      const int oa = __shfl_xor(nnaddr, m);
      const bool take = (od < dsd) || (od == dsd && oa < nnaddr);
      dsd = take ? od : dsd;
      nnaddr = take ? oa : nnaddr;
    }
  }
  writer = ivalid && jsub == 0;
}

template <int ORDER, bool F64, int P, bool NGB, bool PIPE, bool AHEAD>
__global__ __launch_bounds__(256) void k_force(
    const typename RecOf<ORDER, F64>::T* __restrict__ rec, const int2* __restrict__ idr, const int nj,
    const double* __restrict__ ibuf, const int* __restrict__ iid, const CallDesc* __restrict__ cd,
    double* __restrict__ part, double* __restrict__ part_ds2, int* __restrict__ part_addr,
    int* __restrict__ ngb_cnt, int* __restrict__ ngb_list, const int S, const Splits sp, const int smajor,
    const int blockred) {
  constexpr int NF = nf<ORDER>();
  // the call's values come from the descriptor; the grid may cover more
  // i-groups than there are (a launch shape shared by a range of ni)
  const int ni = cd->ni;
  const double eps2d = cd->eps2;
  const double* ipos = ibuf;
  const double* ivel = ibuf + 3 * (size_t)ni;
  const double* iacc = ibuf + 6 * (size_t)ni;
  const double* ih2 = ibuf + (ORDER >= ORDER_H6 ? 9 : 6) * (size_t)ni;
  // wave-uniform by construction; readfirstlane lets the compiler keep the
  // j-loop bookkeeping and (for P = 64) the j-record loads in SGPRs
  const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int G = (ni + P - 1) / P;
  if (wave >= G * S) return;  // whole wave (a whole block when S % 4 == 0)
  // smajor: consecutive waves (a block's 4) share one j-range and so its
  // scalar-cache lines; otherwise consecutive waves walk the splits of one group
  const int g = smajor ? wave % G : wave / S;
  const int sidx = smajor ? wave / G : wave - g * S;
  const int jb = sp.begin(sidx);
  const int je = min(nj, sp.begin(sidx + 1));
  double T[NF];
  double dsd;
  int nnaddr, islot;
  bool writer;
  wave_force<ORDER, F64, P, NGB, PIPE, AHEAD>(rec, idr, ipos, ivel, iacc, ih2, iid, g * P, min(P, ni - g * P), jb, je, eps2d,
                                 ngb_cnt, ngb_list, T, dsd, nnaddr, islot, writer);
  if (blockred) {
    // The block's waves are splits 4q..4q+3 of one i-group (S % 4 == 0, so
    // every block is whole and no wave left early).  Their sums go through
    // LDS four fields at a time; wave w adds field c0 + w over the four
    // splits in the fixed order (s0 + s1) + (s2 + s3) and writes one row.
    // Wave 3 also takes the nearest neighbour.  The barriers bound what any
    // wave holds at once, so the epilogue does not raise the register count.
    __shared__ double red_t[4][4][64];
    __shared__ double red_d[4][64];
    __shared__ int red_a[4][64];
    const int w = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int i = g * P + islot;
    const int S4 = S >> 2, row = sidx >> 2;
    red_d[w][lane] = dsd;
    red_a[w][lane] = nnaddr;
#pragma unroll
    for (int c0 = 0; c0 < NF; c0 += 4) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (c0 + k < NF) red_t[w][k][lane] = T[c0 + k];
      __syncthreads();
      if (c0 + w < NF && writer) {
        const double v = (red_t[0][w][lane] + red_t[1][w][lane]) + (red_t[2][w][lane] + red_t[3][w][lane]);
        part[((size_t)(c0 + w) * S4 + row) * ni + i] = v;
      }
      if (c0 == 0 && w == 3 && writer) {
        double bd = red_d[0][lane];
        int ba = red_a[0][lane];
#pragma unroll
        for (int u = 1; u < 4; ++u) {
          const double od = red_d[u][lane];
          const int oa = red_a[u][lane];
          const bool take = (od < bd) || (od == bd && oa < ba);
          bd = take ? od : bd;
          ba = take ? oa : ba;
        }
        part_ds2[(size_t)row * ni + i] = bd;
        part_addr[(size_t)row * ni + i] = ba;
      }
      __syncthreads();
    }
    return;
  }
  if (writer) {
    const int i = g * P + islot;
#pragma unroll
    for (int f = 0; f < NF; ++f) part[((size_t)f * S + sidx) * ni + i] = T[f];
    part_ds2[(size_t)sidx * ni + i] = dsd;
    part_addr[(size_t)sidx * ni + i] = nnaddr;
  }
}

// Force kernel of at most SMALL_NI i-particles: a work-group takes tiles of 256
// j, one thread each, into LDS; then each of its waves sums its 64 j of a tile
// for the i-particles, P = the power of two above ni of them on the lanes and
// Q = 64 / P j at a time.  One partial row per work-group.  PRED: the thread's j
// is predicted here (and updated first if it is among the staged rows), so that
// a call is this launch and the finalize; otherwise its record is read.  The
// tiles and the order of the sums are the same in both, and do not depend on the
// updates.  Bound by launch, PCIe and memory latency: the pairs of 24 x 131072
// take 2 us at the full rate.
template <int ORDER, bool F64, bool NGB, bool PRED>
__global__ __launch_bounds__(256) void k_force_small(SmallArgs a) {
  using R = typename std::conditional<F64, double, float>::type;
  using Rec = typename RecOf<ORDER, F64>::T;
  constexpr int NF = nf<ORDER>(), NR = raw_fields(ORDER) + 1;
  __shared__ __align__(16) Rec tile[256];
  __shared__ double red[4][NF][SMALL_NI];
  __shared__ double red_d[4][SMALL_NI];
  __shared__ int red_a[4][SMALL_NI];
  __shared__ int row_of[256];
  const int t = threadIdx.x, w = t >> 6, lane = t & 63, b = blockIdx.x;
  const int ni = PRED ? a.ni : min(a.f.cd->ni, SMALL_NI), nj = a.f.nj;
  const R eps2 = (R)(PRED ? a.eps2 : a.f.cd->eps2);
  const int lp = ni > 1 ? 32 - __clz(ni - 1) : 0, P = 1 << lp;
  const int islot = lane & (P - 1), jsub = lane >> lp;
  // the i-particle's doubles are loaded first and converted when the first tile
  // is there: over PCIe they take as long as the tile
  constexpr int NI = ORDER >= ORDER_H6 ? 9 : 6;
  const int il = islot < ni ? islot : 0;
  double iv[NI], ih = -1.0;
#pragma unroll
  for (int f = 0; f < NI; ++f) iv[f] = a.f.ibuf[(size_t)(f / 3) * 3 * ni + 3 * il + f % 3];
  if (NGB && islot < ni) ih = a.f.ibuf[(size_t)NI * ni + il];
  const int iid = a.f.iid[il];
  IState<ORDER, R> st;
  NgbList ngb{a.f.ngb_cnt, a.f.ngb_list, il, -1};
  double T[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) T[f] = 0.0;
  R dsmin = R(INFINITY);
  int nnaddr = INT_MAX;
  if constexpr (PRED) {
    // the other buffer of counters, for the next call of this kind
    if (b == 0 && t < SMALL_NI) a.cnt_clear[t] = 0;
  }
  const int ntiles = (nj + 255) / 256;
  const int t1 = min(ntiles, (b + 1) * a.tiles);
  for (int tl = b * a.tiles; tl < t1; ++tl) {
    const int j = tl * 256 + t;
    if constexpr (PRED) {
      Rec r{};
      // stored fields: loads that do not wait for the update bits
      const size_t cap = (size_t)a.st.cap;
      double raw[NR - 1];
      if (j < nj) {
#pragma unroll
        for (int f = 0; f < NR - 1; ++f)
          if (f != RF_DT && f != RF_EPS) raw[f] = a.st.raw[(size_t)f * cap + j];
      }
      int row = -1;  // staged row of this j
      if (a.nupd <= SMALL_ARG) {
#pragma unroll
        for (int u = 0; u < SMALL_ARG; ++u)
          if (u < a.nupd && a.addr[u] == j) row = u;
        __syncthreads();  // every wave is done with the last tile
      } else {
        const bool upd = j < a.nbits && (a.bits[j >> 5] >> (j & 31) & 1u);
        if (__syncthreads_or(upd)) {
          if (t < a.nupd) {
            const int q = reinterpret_cast<const int2*>(a.rows_h + (size_t)t * NR + NR - 1)->x - tl * 256;
            if (q >= 0 && q < 256) row_of[q] = t;
          }
          __syncthreads();
          if (upd) row = row_of[t];
        }
      }
      tile_id_range(a.st, j);
      if (j < nj) {
        if (row >= 0) {
          const double* u = a.rows_h + (size_t)row * NR;
#pragma unroll
          for (int f = 0; f < NR - 1; ++f) raw[f] = u[f];
#pragma unroll
          for (int f = 0; f < NR - 1; ++f) a.st.raw[(size_t)f * cap + j] = raw[f];
        }
        double p[3], v[3], ac[3];
        predict_one<ORDER>([&](int f) { return raw[f]; }, a.ti, p, v, ac);
        r = put_pred<ORDER, F64>(a.st, j, p, v, ac, raw[RF_M], a.st.id[j]);
      }
      tile[t] = r;  // past nj a massless record at the origin
    } else {
      __syncthreads();
      if (j < nj) tile[t] = reinterpret_cast<const Rec*>(a.f.rec)[j];
      else tile[t] = Rec{};
    }
    __syncthreads();
    if (tl == b * a.tiles) {
      get_pos(st.x, iv[0]); get_pos(st.y, iv[1]); get_pos(st.z, iv[2]);
      st.vx = (R)iv[3]; st.vy = (R)iv[4]; st.vz = (R)iv[5];
      st.ax = st.ay = st.az = R(0);
      if constexpr (ORDER >= ORDER_H6) { st.ax = (R)iv[6]; st.ay = (R)iv[7]; st.az = (R)iv[8]; }
      st.h2 = (R)ih;
      st.id = iid;
      st.i = il;
    }
    R s[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) s[f] = R(0);
    // four j at a time (their LDS reads are in flight together), P < 4 one by one
    int k = 0;
    for (; k + 4 <= P; k += 4) {
      R d[4];
      int id[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = w * 64 + jsub + ((k + u) << (6 - lp)), jq = tl * 256 + q;
        const Rec rj = tile[q];
        id[u] = rj.id;
        int unused = 0;
        pair<ORDER, NGB, true, true>(rj, jq, jq < nj, st, eps2, s, d[u], unused);
        const bool better = d[u] < dsmin;
        dsmin = better ? d[u] : dsmin;
        nnaddr = better ? jq : nnaddr;
      }
      if constexpr (NGB) {
        settle<ORDER>(s);
#pragma unroll
        for (int u = 0; u < 4; ++u) asm volatile("" : "+v"(d[u]));
        const bool nb[4] = {st.h2 > d[0], st.h2 > d[1], st.h2 > d[2], st.h2 > d[3]};
        ngb.add4(nb, [&](int u) { return id[u]; });
      }
    }
    for (; k < P; ++k) {
      const int q = w * 64 + jsub + (k << (6 - lp)), jq = tl * 256 + q;
      const Rec& rj = tile[q];
      if (pair<ORDER, NGB, true, false>(rj, jq, jq < nj, st, eps2, s, dsmin, nnaddr)) ngb.add(rj.id);
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) T[f] += (double)s[f];
  }
  if constexpr (NGB) ngb.finish();
  double dsd = (double)dsmin;
  for (int m = P; m < 64; m <<= 1) {
#pragma unroll
    for (int f = 0; f < NF; ++f) T[f] += __shfl_xor(T[f], m);
    const double od = __shfl_xor(dsd, m);
    const int oa = __shfl_xor(nnaddr, m);
    const bool take = (od < dsd) || (od == dsd && oa < nnaddr);
    dsd = take ? od : dsd;
    nnaddr = take ? oa : nnaddr;
  }
  if (jsub == 0) {
#pragma unroll
    for (int f = 0; f < NF; ++f) red[w][f][islot] = T[f];
    red_d[w][islot] = dsd;
    red_a[w][islot] = nnaddr;
  }
  __syncthreads();
  const int rows = gridDim.x;
  for (int o = t; o < (NF + 1) * SMALL_NI; o += 256) {
    const int f = o / SMALL_NI, i = o % SMALL_NI;
    if (i >= ni) continue;
    if (f < NF) {
      a.f.part[((size_t)f * rows + b) * ni + i] = (red[0][f][i] + red[1][f][i]) + (red[2][f][i] + red[3][f][i]);
    } else {
      double bd = red_d[0][i];
      int ba = red_a[0][i];
#pragma unroll
      for (int q = 1; q < 4; ++q) {
        const bool take = (red_d[q][i] < bd) || (red_d[q][i] == bd && red_a[q][i] < ba);
        bd = take ? red_d[q][i] : bd;
        ba = take ? red_a[q][i] : ba;
      }
      a.f.part_ds2[(size_t)b * ni + i] = bd;
      a.f.part_addr[(size_t)b * ni + i] = ba;
    }
  }
}

template <int ORDER, bool F64>
__device__ __forceinline__ void write_row(const FinalizeArgs& a, int i, const double* T, double ds, int ad,
                                          int cnt);

// Ensemble force: one wave per item of a work table (cluster, i-group,
// j-split); each item carries its own lane shape.  Without lists, an item
// that is its i-particles' only split writes their result rows (over PCIe,
// while other items still compute) as the finalize would: the finalize's
// sum over one split is 0.0 + T, and its nearest neighbour the item's own.
template <int ORDER, bool F64, int P, bool NGB, bool AHEAD = false>
__device__ __forceinline__ void ens_item(const EnsArgs& a, const FinalizeArgs& fz,
                                         const typename RecOf<ORDER, F64>::T* __restrict__ rec, const EnsItem& it,
                                         int item) {
  constexpr int NF = nf<ORDER>();
  double T[NF];
  double dsd;
  int nnaddr, islot;
  bool writer;
  wave_force<ORDER, F64, P, NGB, false, AHEAD>(rec, a.idr, a.ipos, a.ivel, a.iacc, a.ih2, a.iid,
                                 it.i0, it.icount, it.jb, it.je, a.eps2[it.cluster], a.ngb_cnt, a.ngb_list, T,
                                 dsd, nnaddr, islot, writer);
  if (!NGB && it.nsplit == 1) {
    if (writer) {
#pragma unroll
      for (int f = 0; f < NF; ++f) T[f] = 0.0 + T[f];
      write_row<ORDER, F64>(fz, it.i0 + islot, T, dsd, nnaddr, 0);
    }
    return;
  }
  if (writer) {
    const size_t row = (size_t)item * 64 + islot;
#pragma unroll
    for (int f = 0; f < NF; ++f) a.part[(size_t)f * a.nitems * 64 + row] = T[f];
    a.part_ds2[row] = dsd;
    a.part_addr[row] = nnaddr;
  }
}

// P64: items [ib, ie) all have lane shape 64; otherwise 16, 4 or 1 (a switch
// whose larger register needs stay out of the P = 64 kernel).
// One single-wave work-group per position q of the ordered item list [ib, ie):
// the list holds the longest items first and the hardware dispatches work-
// groups in order as wave slots free up, so the short items fill the end of
// the launch with no queue to contend for.  (A counter that every wave bumped
// for its next item serialised the small items of large ensembles.)
template <int ORDER, bool F64, bool NGB, bool P64, bool AHEAD>
__global__ __launch_bounds__(64) void k_force_ens(EnsArgs a, FinalizeArgs fz,
                                                  const typename RecOf<ORDER, F64>::T* __restrict__ rec, int ib,
                                                  int ie) {
  const int q = ib + (int)blockIdx.x;
  if (q >= ie) return;
  const int item = __builtin_amdgcn_readfirstlane(a.order[q]);
  // the item is wave-uniform; readfirstlane keeps its fields (and so the
  // j-record addresses) in SGPRs, which a load the compiler cannot prove
  // invariant would otherwise place in VGPRs
  const EnsItem ld = a.items[item];
  EnsItem it;
  it.i0 = __builtin_amdgcn_readfirstlane(ld.i0);
  it.icount = __builtin_amdgcn_readfirstlane(ld.icount);
  it.jb = __builtin_amdgcn_readfirstlane(ld.jb);
  it.je = __builtin_amdgcn_readfirstlane(ld.je);
  it.P = __builtin_amdgcn_readfirstlane(ld.P);
  it.cluster = __builtin_amdgcn_readfirstlane(ld.cluster);
  it.nsplit = __builtin_amdgcn_readfirstlane(ld.nsplit);
  it.pad = 0;
  if constexpr (P64) {
    ens_item<ORDER, F64, 64, NGB, AHEAD>(a, fz, rec, it, item);
  } else {
    switch (it.P) {
      case 16: ens_item<ORDER, F64, 16, NGB>(a, fz, rec, it, item); break;
      case 4: ens_item<ORDER, F64, 4, NGB>(a, fz, rec, it, item); break;
      default: ens_item<ORDER, F64, 1, NGB>(a, fz, rec, it, item); break;
    }
  }
}

// Ensemble finalize, thread per i-particle: fixed-order sum over its items.
template <int ORDER, bool F64>
__device__ __forceinline__ void finalize_ens_block(const FinalizeArgs& f, const EnsArgs& a, int b) {
  constexpr int NF = nf<ORDER>();
  const int i = b * 256 + threadIdx.x;
  if (i >= f.cd->ni) return;
  const int4 d = a.idesc[i];  // first item, number of splits, i-slot
  if (!f.ngb_on && d.y == 1) return;  // its only item wrote the row
  double T[NF];
#pragma unroll
  for (int q = 0; q < NF; ++q) T[q] = 0.0;
  double ds = INFINITY;
  int ad = INT_MAX;
  for (int s = 0; s < d.y; ++s) {
    const size_t row = (size_t)(d.x + s) * 64 + d.z;
#pragma unroll
    for (int q = 0; q < NF; ++q) T[q] += a.part[(size_t)q * a.nitems * 64 + row];
    const double dd = a.part_ds2[row];
    const int ad2 = a.part_addr[row];
    const bool take = (dd < ds) || (dd == ds && ad2 < ad);
    ds = take ? dd : ds;
    ad = take ? ad2 : ad;
  }
  write_row<ORDER, F64>(f, i, T, ds, ad, f.ngb_on ? f.ngb_cnt[i] : 0);
}

// ---------------------------------------------------------------------------
// Finalize.  Fixed-order sums of the partial rows of each i-particle, the
// nearest neighbour as the (ds2, address) minimum, the result row, and the
// ascending sort of the neighbour list.
// Output in host memory: with a completion word, a store that is at the host when
// the wave has waited for it (the word's protocol needs no cache write-back then,
// which took 20 us over the work-groups of 333 i-particles).
template <typename V> __device__ __forceinline__ void put_host(const int* done, V* p, V v) {
  if (done) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  else *p = v;
}

// The last work-group to finish tells the host: it polls a word in its own memory
// instead of an event, whose record costs the host 4 us and the device a marker
// behind the kernel (a chain of three empty kernels: 18 us with an event, 12 with
// the word).  Every wave waits for its own output (put_host) before its work-
// group counts.
__device__ __forceinline__ void finish_word(int* done, int* ctr, int seq) {
  __builtin_amdgcn_s_waitcnt(0);  // all counters
  __syncthreads();
  if (threadIdx.x == 0) {
    const int k = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (k == (int)gridDim.x - 1) {
      *ctr = 0;
      __hip_atomic_store(done, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

__device__ __forceinline__ int call_ni(const FinalizeArgs& a) { return a.cd ? a.cd->ni : a.ni; }

// Nearest neighbour and count of i-particle i.
template <int ORDER, bool F64>
__device__ __forceinline__ void write_nn(const FinalizeArgs& a, int i, double ds, int ad, int cnt) {
  using Rec = typename RecOf<ORDER, F64>::T;
  constexpr int NF = nf<ORDER>();
  double* o = a.out + i;
  const size_t st = (size_t)a.ostride;
  const bool has = ad != INT_MAX;
  // the device returns ds2 rounded to float (kernels.cu:999-1002)
  put_host(a.done, o + NF * st, has ? (double)(float)ds : (double)INFINITY);
  put_host(a.done, o + (NF + 1) * st, has ? (double)reinterpret_cast<const Rec*>(a.rec)[ad].id : -1.0);
  put_host(a.done, o + (NF + 2) * st, (double)cnt);
}

// Result row of i-particle i, field-major (consecutive i of a wave write
// consecutive doubles of each field: whole lines over PCIe).
template <int ORDER, bool F64>
__device__ __forceinline__ void write_row(const FinalizeArgs& a, int i, const double* T, double ds, int ad,
                                          int cnt) {
  constexpr int NF = nf<ORDER>();
  double* o = a.out + i;
  const size_t st = (size_t)a.ostride;
#pragma unroll
  for (int f = 0; f < NF; ++f) o[f * st] = T[f];
  write_nn<ORDER, F64>(a, i, ds, ad, cnt);
}

// Key of list entry k: orders by id, equal ids by k.
__device__ __forceinline__ unsigned long long list_key(int id, int k) {
  return ((unsigned long long)((unsigned)id ^ 0x80000000u) << 32) | (unsigned)k;
}

// Rank sort of c ids by one wave, written to dst: s[0..c) holds their keys, padded
// to a multiple of four with ~0.  A lane ranks its (up to four) ids against four
// at a time, one compare and one add each; a full list of 256 took 30 us with
// one LDS read and an index test per comparison.
__device__ __forceinline__ void wave_rank_sort(const unsigned long long* s, int c, int lane, int* dst) {
  constexpr int M = NGB_CAP / 64;
  unsigned long long v[M];
  int rank[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    v[m] = lane + 64 * m < c ? s[lane + 64 * m] : 0ull;
    rank[m] = 0;
  }
  for (int q = 0; q < c; q += 4) {
    const unsigned long long u[4] = {s[q], s[q + 1], s[q + 2], s[q + 3]};
#pragma unroll
    for (int m = 0; m < M; ++m) {
      if (64 * m >= c) break;  // uniform
#pragma unroll
      for (int e = 0; e < 4; ++e) rank[m] += u[e] < v[m] ? 1 : 0;
    }
  }
#pragma unroll
  for (int m = 0; m < M; ++m)
    if (lane + 64 * m < c) dst[rank[m]] = (int)((unsigned)(v[m] >> 32) ^ 0x80000000u);
}

// U threads per i-particle, 256 / U consecutive i-particles per work-group (a
// row is read whole-line): thread u sums rows u, u + U, ... in order, the U sums
// are added through LDS in a fixed order.  Bound by the latency of the row reads
// and of the PCIe writes; U grows as ni falls so that few i-particles still have
// many reads in flight (333 i-particles of 782 rows: 32 us with one work-group
// per i-particle reading across rows).
template <int ORDER, bool F64, int U>
__device__ __forceinline__ void finalize_block(const FinalizeArgs& a, int b) {
  constexpr int NF = nf<ORDER>(), I = 256 / U;
  __shared__ double red[NF][256];
  __shared__ double red_d[256];
  __shared__ int red_a[256];
  const int ni = call_ni(a);
  const int t = threadIdx.x;
  const int ii = t % I, u = t / I;
  const int i = b * I + ii;
  if (b * I >= ni) return;  // whole work-group (the grid may cover more i-particles)
  double T[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) T[f] = 0.0;
  double ds = INFINITY;
  int ad = INT_MAX;
  if (i < ni) {
#pragma unroll 2
    for (int s = u; s < a.S; s += U) {
#pragma unroll
      for (int f = 0; f < NF; ++f) T[f] += a.part[((size_t)f * a.S + s) * ni + i];
      const double d = a.part_ds2[(size_t)s * ni + i];
      const int ad2 = a.part_addr[(size_t)s * ni + i];
      const bool take = (d < ds) || (d == ds && ad2 < ad);
      ds = take ? d : ds;
      ad = take ? ad2 : ad;
    }
  }
#pragma unroll
  for (int f = 0; f < NF; ++f) red[f][t] = T[f];
  red_d[t] = ds;
  red_a[t] = ad;
  __syncthreads();
  // output o: field o / I of i-particle o % I, and last the nearest neighbour and
  // count; L lanes each take every L-th of its U values
  constexpr int L = U == 256 ? 16 : U == 64 ? 4 : 1, OUT = (NF + 1) * I;
  static_assert(L == 1 || L * OUT <= 256, "one pass");
  for (int o = t / L; o < OUT; o += 256 / L) {
    const int f = o / I, k = o % I, io = b * I + k, l = t % L;
    if (f < NF) {
      constexpr int C = U / L < 4 ? U / L : 4;  // chains
      double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < U / L; q += C)
#pragma unroll
        for (int c = 0; c < C; ++c) v[c] += red[f][((q + c) * L + l) * I + k];
      double r = (v[0] + v[1]) + (v[2] + v[3]);
#pragma unroll
      for (int m = 1; m < L; m <<= 1) r += __shfl_xor(r, m);
      if (l == 0 && io < ni) put_host(a.done, a.out + (size_t)f * a.ostride + io, r);
    } else {
      double bd = red_d[l * I + k];
      int ba = red_a[l * I + k];
#pragma unroll
      for (int q = 1; q < U / L; ++q) {
        const double od = red_d[(q * L + l) * I + k];
        const int oa = red_a[(q * L + l) * I + k];
        const bool take = (od < bd) || (od == bd && oa < ba);
        bd = take ? od : bd;
        ba = take ? oa : ba;
      }
#pragma unroll
      for (int m = 1; m < L; m <<= 1) {
        const double od = __shfl_xor(bd, m);
        const int oa = __shfl_xor(ba, m);
        const bool take = (od < bd) || (od == bd && oa < ba);
        bd = take ? od : bd;
        ba = take ? oa : ba;
      }
      if (l == 0 && io < ni) write_nn<ORDER, F64>(a, io, bd, ba, a.ngb_on ? a.ngb_cnt[io] : 0);
    }
  }
}

// Host offset of i-particle i's list in a single-system call: its region's
// base plus the stored lengths of the region's earlier lists.  The counts are
// final once the force kernel has run, so no work-group waits for another; a
// whole wave calls this (at most LIST_REGION - 1 counts, a few per lane).
__device__ __forceinline__ int region_offset(const int* __restrict__ cnt, int i, int lane) {
  const int r0 = i & ~(LIST_REGION - 1);
  int s = 0;
  for (int k = r0 + lane; k < i; k += 64) s += min(cnt[k], NGB_CAP);
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) s += __shfl_xor(s, m);
  return r0 * NGB_CAP + s;
}

// Writes the sorted list s[0..c) of i-particle i: back into its device slots
// and, when it fits, to the host-mapped buffer at off (consecutive lanes write
// consecutive ids).
__device__ __forceinline__ void store_list(const FinalizeArgs& a, int i, const int* s, int c, int off, int t,
                                           int nt) {
  const bool host = (long)off + c <= a.packed_cap;
  for (int k = t; k < c; k += nt) {
    const int v = s[k];
    a.ngb_list[(size_t)i * NGB_CAP + k] = v;
    if (host) put_host(a.done, a.packed + off + k, v);
  }
}

// Ascending sort in LDS of the (at most NGB_CAP) lists of 4 K i-particles, K per
// wave, then the host copy: in i order within its region (K = 1), or (ensembles)
// packed, the work-group taking its offset with one atomic on the call's counter
// (K = 4: with one per four lists, 75000 lists took 355 us, most of it on that
// counter).
template <int K>
__device__ __forceinline__ void sort_lists_block(const FinalizeArgs& a, int b) {
  __shared__ unsigned long long lst[4][NGB_CAP];
  __shared__ int srt[4][NGB_CAP];
  __shared__ int cnts[4 * K];
  __shared__ int base;
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int ni = call_ni(a);
  if (threadIdx.x < 4 * K) {
    const int i = b * 4 * K + threadIdx.x;
    cnts[threadIdx.x] = i < ni ? min(a.ngb_cnt[i], NGB_CAP) : 0;
  }
  __syncthreads();
  if (threadIdx.x == 0 && !a.inorder) {
    int tot = 0;
    for (int u = 0; u < 4 * K; ++u) tot += cnts[u];
    base = tot > 0 ? atomicAdd(a.pack_ctr, tot) : 0;
  }
#pragma unroll 1
  for (int q = 0; q < K; ++q) {
    const int r = w * K + q, i = b * 4 * K + r, c = cnts[r];
    const bool valid = i < ni;
    for (int k = lane; k < (c + 3) / 4 * 4; k += 64)
      lst[w][k] = k < c ? list_key(a.ngb_list[(size_t)i * NGB_CAP + k], k) : ~0ull;
    __syncthreads();  // also: the last list is stored, base is set
    wave_rank_sort(lst[w], c, lane, srt[w]);
    int off = valid && a.inorder ? region_offset(a.ngb_cnt, i, lane) : 0;
    if (!a.inorder) {
      off = base;
      for (int u = 0; u < r; ++u) off += cnts[u];
    }
    __syncthreads();
    if (valid && lane == 0) put_host(a.done, a.list_off + i, off);
    store_list(a, i, srt[w], c, off, lane, 64);
  }
}

// Finalize and list sort in one launch (independent work: the sort only
// reorders the lists, the finalize reads counts): the first nfin work-groups
// finalize, the others sort; both roles are uniform per work-group.
template <int ORDER, bool F64, int U>
__global__ __launch_bounds__(256) void k_finalize(FinalizeArgs a, int nfin) {
  if ((int)blockIdx.x < nfin) finalize_block<ORDER, F64, U>(a, blockIdx.x);
  else sort_lists_block<1>(a, blockIdx.x - nfin);
  if (a.done) finish_word(a.done, a.done_ctr, a.cd ? a.cd->seq : a.seq);
}

// The same for ensembles: result rows and lists cross PCIe side by side.
template <int ORDER, bool F64>
__global__ __launch_bounds__(256) void k_finalize_ens(FinalizeArgs f, EnsArgs a, int nfin) {
  if ((int)blockIdx.x < nfin) finalize_ens_block<ORDER, F64>(f, a, blockIdx.x);
  else sort_lists_block<4>(f, blockIdx.x - nfin);
}

// ---------------------------------------------------------------------------
// Predicted-state gather for read-back: 10 doubles per j (x, y, z, m, vx, vy, vz,
// ax, ay, az) in FP64, field-major, so that a wave's stores are whole lines also
// where out is host memory (then with a completion word: with copy commands for
// the addresses and the rows, 2500 addresses took 90 us, the kernel 6).
template <int ORDER, bool F64>
__global__ __launch_bounds__(256) void k_gather_pred(GatherArgs a) {
  using Rec = typename RecOf<ORDER, F64>::T;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < a.n) {
    const int j = a.addr ? a.addr[k] : k;
    const Rec r = reinterpret_cast<const Rec*>(a.st.rec)[j];
    const size_t cap = (size_t)a.st.cap;
    double v[10];
    v[3] = a.st.raw[RF_M * cap + j];
    v[7] = v[8] = v[9] = 0.0;
    if constexpr (F64) {
      v[0] = r.x; v[1] = r.y; v[2] = r.z;
      v[4] = r.vx; v[5] = r.vy; v[6] = r.vz;
      if constexpr (ORDER >= ORDER_H6) { v[7] = r.ax; v[8] = r.ay; v[9] = r.az; }
    } else {
      v[0] = a.st.ppos[j]; v[1] = a.st.ppos[cap + j]; v[2] = a.st.ppos[2 * cap + j];
      v[4] = a.st.pvel[j]; v[5] = a.st.pvel[cap + j]; v[6] = a.st.pvel[2 * cap + j];
      if constexpr (ORDER >= ORDER_H6) { v[7] = a.st.pacc[j]; v[8] = a.st.pacc[cap + j]; v[9] = a.st.pacc[2 * cap + j]; }
    }
#pragma unroll
    for (int f = 0; f < 10; ++f) put_host(a.done, a.out + (size_t)f * a.n + k, v[f]);
  }
  if (a.done) finish_word(a.done, a.done_ctr, a.seq);
}

__global__ void k_write_desc(CallDesc* cd, CallDesc v) { *cd = v; }

// ---------------------------------------------------------------------------
// Launchers.
static inline int blocks_for(long n, int bs) { return (int)((n + bs - 1) / bs); }
static inline int hip_status() { return hipGetLastError() == hipSuccess ? 0 : -1; }

// Calls f(order constant, precision constant) for the runtime (order, f64).
template <typename F>
static void dispatch_op(int order, bool f64, F&& f) {
  using H4 = std::integral_constant<int, ORDER_H4>;
  using H6 = std::integral_constant<int, ORDER_H6>;
  if (order >= ORDER_H6) {
    if (f64) f(H6{}, std::true_type{}); else f(H6{}, std::false_type{});
  } else {
    if (f64) f(H4{}, std::true_type{}); else f(H4{}, std::false_type{});
  }
}

int launch_scatter(hipStream_t s, int order, bool f64, const ScatterArgs& a) {
  if (a.grid_blocks <= 0) return 0;
  const int nb = a.grid_blocks;  // grid-stride over the descriptor's counts
  dispatch_op(order, f64, [&](auto OR, auto FP) {
    hipLaunchKernelGGL((k_scatter<decltype(OR)::value, decltype(FP)::value>), dim3(nb), dim3(256), 0, s, a);
  });
  return hip_status();
}

int launch_predict(hipStream_t s, int order, bool f64, const PredictArgs& a) {
  if (a.j1 <= a.j0) return 0;
  const int nb = blocks_for(a.j1 - a.j0, 256);
  dispatch_op(order, f64, [&](auto OR, auto FP) {
    hipLaunchKernelGGL((k_predict<decltype(OR)::value, decltype(FP)::value>), dim3(nb), dim3(256), 0, s, a);
  });
  return hip_status();
}

// Copy work-groups: 4 x 16 bytes a thread, at most 64 groups (256 KB in flight
// covers the PCIe latency at its full rate).
int launch_prep(hipStream_t s, int order, bool f64, const PrepArgs& args) {
  PrepArgs a = args;
  a.nb_upd = blocks_for(a.nupd, PREP_ROWS);
  long n16 = 0;
  for (const CopySeg& g : a.seg) n16 += g.n16;
  a.nb_copy = std::min(64, blocks_for(std::max<long>(n16, a.ni_reset), 1024));
  const int nb = a.nb_upd + a.nb_copy + blocks_for(a.pred_j1, 256);
  if (nb == 0) return 0;
  dispatch_op(order, f64, [&](auto OR, auto FP) {
    hipLaunchKernelGGL((k_prep<decltype(OR)::value, decltype(FP)::value>), dim3(nb), dim3(256), 0, s, a);
  });
  return hip_status();
}

bool force_p_supported(int P) {
  return P == 64 || P == 32 || P == 16 || P == 8 || P == 4 || P == 2 || P == 1;
}

template <int OR, bool FP, int P, bool PIPE, bool AHEAD>
static void launch_force_w(hipStream_t s, const ForceArgs& a, const ForceConfig& c) {
  const long G = (a.grid_ni + P - 1) / P;
  const dim3 nb(blocks_for(G * c.S, 4)), bs(256);
  const Splits sp = make_splits(P, c.S, a.nj);
  const auto* rec = reinterpret_cast<const typename RecOf<OR, FP>::T*>(a.rec);
#define SAPK_FORCE_ARGS rec, a.idr, a.nj, a.ibuf, a.iid, a.cd, a.part, a.part_ds2, \
                        a.part_addr, a.ngb_cnt, a.ngb_list, c.S, sp, c.smajor, partial_rows(c) != c.S ? 1 : 0
  if (a.ngb_on) hipLaunchKernelGGL((k_force<OR, FP, P, true, PIPE, AHEAD>), nb, bs, 0, s, SAPK_FORCE_ARGS);
  else hipLaunchKernelGGL((k_force<OR, FP, P, false, false, AHEAD>), nb, bs, 0, s, SAPK_FORCE_ARGS);
#undef SAPK_FORCE_ARGS
}

// Lists with deferred id stores (c.pipe) have kernels of their own.  P = 64 takes
// records ahead in FP64 always, in mixed precision where the launch shape says
// so (choose_config).
template <int OR, bool FP, int P>
static void launch_force_p(hipStream_t s, const ForceArgs& a, const ForceConfig& c) {
  if (c.pipe) return launch_force_w<OR, FP, P, true, false>(s, a, c);
  if constexpr (P == 64) {
    if (FP || c.ahead) return launch_force_w<OR, FP, P, false, true>(s, a, c);
  }
  if constexpr (P != 64 || !FP) launch_force_w<OR, FP, P, false, false>(s, a, c);
}

template <int OR, bool FP>
static int launch_force_t(hipStream_t s, const ForceArgs& a, const ForceConfig& c) {
  switch (c.P) {
    case 64: launch_force_p<OR, FP, 64>(s, a, c); break;
    case 32: launch_force_p<OR, FP, 32>(s, a, c); break;
    case 16: launch_force_p<OR, FP, 16>(s, a, c); break;
    case 8: launch_force_p<OR, FP, 8>(s, a, c); break;
    case 4: launch_force_p<OR, FP, 4>(s, a, c); break;
    case 2: launch_force_p<OR, FP, 2>(s, a, c); break;
    case 1: launch_force_p<OR, FP, 1>(s, a, c); break;
    default: return -2;
  }
  return hip_status();
}

int launch_force_small(hipStream_t s, int order, bool f64, const SmallArgs& a, const ForceConfig& c, bool pred) {
  if (a.f.grid_ni <= 0 || a.f.nj <= 0) return 0;
  if (a.f.grid_ni > SMALL_NI || a.nupd > SMALL_UPD || a.tiles <= 0 || (long)c.S * a.tiles * 256 < a.f.nj) return -3;
  dispatch_op(order, f64, [&](auto OR, auto FP) {
    constexpr int O = decltype(OR)::value;
    constexpr bool F = decltype(FP)::value;
    const dim3 nb(c.S), bs(256);
    if (pred && a.f.ngb_on) hipLaunchKernelGGL((k_force_small<O, F, true, true>), nb, bs, 0, s, a);
    else if (pred) hipLaunchKernelGGL((k_force_small<O, F, false, true>), nb, bs, 0, s, a);
    else if (a.f.ngb_on) hipLaunchKernelGGL((k_force_small<O, F, true, false>), nb, bs, 0, s, a);
    else hipLaunchKernelGGL((k_force_small<O, F, false, false>), nb, bs, 0, s, a);
  });
  return hip_status();
}

int launch_force(hipStream_t s, int order, bool f64, const ForceArgs& a, const ForceConfig& c) {
  if (a.grid_ni <= 0 || a.nj <= 0) return 0;
  if (c.small) {
    SmallArgs sm{};
    sm.f = a;
    sm.tiles = c.jchunk / 256;
    return launch_force_small(s, order, f64, sm, c, false);
  }
  if (c.S <= 0) return -3;
  int rc = 0;
  dispatch_op(order, f64, [&](auto OR, auto FP) { rc = launch_force_t<decltype(OR)::value, decltype(FP)::value>(s, a, c); });
  return rc;
}

int launch_finalize(hipStream_t s, int order, bool f64, const FinalizeArgs& a) {
  if (a.grid_ni <= 0) return 0;
  dispatch_op(order, f64, [&](auto OR, auto FP) {
    constexpr int O = decltype(OR)::value;
    constexpr bool F = decltype(FP)::value;
    const int nsort = a.ngb_on ? blocks_for(a.grid_ni, 4) : 0;
    const int nfin = blocks_for((long)a.U * a.grid_ni, 256);
    switch (a.U) {
      case 256: hipLaunchKernelGGL((k_finalize<O, F, 256>), dim3(nfin + nsort), dim3(256), 0, s, a, nfin); break;
      case 64: hipLaunchKernelGGL((k_finalize<O, F, 64>), dim3(nfin + nsort), dim3(256), 0, s, a, nfin); break;
      case 16: hipLaunchKernelGGL((k_finalize<O, F, 16>), dim3(nfin + nsort), dim3(256), 0, s, a, nfin); break;
      default: hipLaunchKernelGGL((k_finalize<O, F, 4>), dim3(nfin + nsort), dim3(256), 0, s, a, nfin); break;
    }
  });
  return hip_status();
}

int launch_force_ens(hipStream_t s, int order, bool f64, const EnsArgs& a, const FinalizeArgs& f, int n64) {
  if (a.nitems <= 0 || f.grid_ni <= 0) return 0;
  dispatch_op(order, f64, [&](auto OR, auto FP) {
    constexpr int O = decltype(OR)::value;
    constexpr bool F = decltype(FP)::value;
    const auto* rec = reinterpret_cast<const typename RecOf<O, F>::T*>(a.rec);
    auto part = [&](auto ngb, auto p64, auto ahead, int ib, int ie) {
      constexpr bool N = decltype(ngb)::value, P = decltype(p64)::value, A = decltype(ahead)::value;
      if (ie > ib) hipLaunchKernelGGL((k_force_ens<O, F, N, P, A>), dim3(ie - ib), dim3(64), 0, s, a, f, rec, ib, ie);
    };
    auto both = [&](auto ngb) {
      // records ahead as in the single-system launches: FP64 always, mixed where
      // the waves leave SIMDs half empty
      if (F || a.ahead) part(ngb, std::true_type{}, std::true_type{}, 0, n64);
      else if constexpr (!F) part(ngb, std::true_type{}, std::false_type{}, 0, n64);
      part(ngb, std::false_type{}, std::false_type{}, n64, a.nitems);
    };
    if (a.ngb_on) both(std::true_type{});
    else both(std::false_type{});
    const int nfin = blocks_for(f.grid_ni, 256), nsort = f.ngb_on ? blocks_for(f.grid_ni, 16) : 0;
    hipLaunchKernelGGL((k_finalize_ens<O, F>), dim3(nfin + nsort), dim3(256), 0, s, f, a, nfin);
  });
  return hip_status();
}

// One thread per i-particle: its group by binary search over the groups' first
// i-particles (groups are in i order and cover [0, ni)).
__global__ __launch_bounds__(256) void k_ens_idesc(const EnsGroup* __restrict__ g, int ng, int ni,
                                                   int4* __restrict__ idesc) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= ni) return;
  int lo = 0, hi = ng - 1;  // the last group with ib <= i
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (g[mid].ib <= i) lo = mid;
    else hi = mid - 1;
  }
  const EnsGroup gr = g[lo];
  const int r = i - gr.ib;
  idesc[i] = make_int4(gr.first + (r / gr.P) * gr.S, gr.S, r % gr.P, gr.P == 64 ? 0 : 1);
}

int launch_ens_idesc(hipStream_t s, const EnsGroup* g, int ng, int ni, int4* idesc) {
  if (ni <= 0 || ng <= 0) return 0;
  hipLaunchKernelGGL(k_ens_idesc, dim3(blocks_for(ni, 256)), dim3(256), 0, s, g, ng, ni, idesc);
  return hip_status();
}

int launch_gather_pred(hipStream_t s, int order, bool f64, const GatherArgs& a) {
  if (a.n <= 0) return 0;
  const int nb = blocks_for(a.n, 256);
  dispatch_op(order, f64, [&](auto OR, auto FP) {
    hipLaunchKernelGGL((k_gather_pred<decltype(OR)::value, decltype(FP)::value>), dim3(nb), dim3(256), 0, s, a);
  });
  return hip_status();
}

int launch_write_desc(hipStream_t s, CallDesc* cd, const CallDesc& v) {
  hipLaunchKernelGGL(k_write_desc, dim3(1), dim3(1), 0, s, cd, v);
  return hip_status();
}

}  // namespace sapk
