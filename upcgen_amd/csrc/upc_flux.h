// Flux-row layout and the per-node phi sum shared by the FP64 and MFMA
// luminosity forms.
#pragma once

#include "upc_internal.h"
#include "upc_qags.h"

#include <algorithm>
#include <climits>

namespace upc {

struct FluxParams {
  double bmin, R, g1, g2, factor, twoR;
  int A, isPoint;
  int mirror_ny;  // > 0: symmetric grid with ny Y bins (k2 rows shared with mirror bins)
};

// Row holding k2 of point p.
__device__ __forceinline__ int k2_row(int p, int npts, int mirror_ny)
{
  if (mirror_ny <= 0) return npts + p;
  const int im = p / mirror_ny, iy = p - im * mirror_ny;
  return iy ? im * mirror_ny + (mirror_ny - iy) : npts + im;
}

__device__ __forceinline__ double row_node(double bmin, double logd, int j, double* bl, double* bh)
{
  *bl = bmin * exp(j * logd);
  *bh = bmin * exp((j + 1.) * logd);
  return (*bh + *bl) / 2.;
}

// The same node for the QAGS kernels, the contraction that the compiler makes
// of row_node's sum spelled out: every kernel that integrates a node sees the
// same b.
__device__ __forceinline__ double row_node_b(double bmin, double logd, int j)
{
  const double bl = bmin * exp(j * logd);
  return fma(bmin, exp((j + 1.) * logd), bl) / 2.;
}

// Position guess on a row's log-spaced nodes b_j = (bmin e^{j logd} +
// bmin e^{(j+1) logd}) / 2 = c0 e^{j logd}: the first j with b_j >= v, from
// one float log2 (right up to +-1 where v lies within rounding of a node).
// Callers step from it to the exact index with their own comparisons.
struct LogGrid {
  float l2c0, s;  // log2(c0), ln 2 / logd
  __device__ __forceinline__ void init(double bmin, double logd)
  {
    l2c0 = (float)log2(bmin * (1.0 + exp(logd)) * 0.5);
    s = (float)(0.69314718055994531 / logd);
  }
  __device__ __forceinline__ int first_ge(double v, int n) const
  {
    if (!(v > 0.0)) return 0;
    const float g = ceilf((__log2f((float)v) - l2c0) * s);
    return g < 0.f ? 0 : (g > (float)n ? n : (int)g);
  }
};

__device__ __forceinline__ double node_b2(double b1, double b2, double c)
{
  return fma(2.0 * b1 * b2, c, fma(b1, b1, b2 * b2));
}

// fluxPoint (src/UpcCrossSection.cpp:166-178): g1 for both beams.
__device__ __forceinline__ double flux_point(double b, double k, double g1, double factor)
{
  const double g = g1;
  const double x = b * k / g / kHc;
  double K0 = 0, K1 = 0;
  if (x > 1e-10) bessel_k01(x, &K0, &K1);
  return factor * k / g / g * (K1 * K1 + K0 * K0 / g / g);
}

// QAGS nodes of one flux row are at most 97: node j has b_j >= bmin e^{j logd}
// with bmin = 0.05 R and logd >= ln(5R / bmin) / 120, so b_j <= 2R needs
// j <= 120 ln 40 / ln 100 = 96.09.
constexpr int kMaxQagsNodesPerRow = 98;

// Log step of a row's b grid.
__device__ __forceinline__ double row_log_step(double bmax, double bmin) { return (log(bmax) - log(bmin)) / kNB1; }

// Geometry of flux row r of a grid of npts points (src/UpcCrossSection.cpp:
// 224-233): photon energy, log step of the b grid, and the number of its
// nodes with b <= 2R (form-factor QAGS nodes; 0 for the point flux).
__device__ __forceinline__ void row_setup(const double* __restrict__ pts, int npts, int r, const FluxParams& fp,
                                          double* k_out, double* logd_out, int* cnt_out)
{
  int p, side;
  if (r < npts) {
    p = r;
    side = 0;
  } else {
    p = fp.mirror_ny > 0 ? (r - npts) * fp.mirror_ny : r - npts;
    side = 1;
  }
  const double M = pts[4 * p], Y = pts[4 * p + 1];
  const double k = side ? M / 2. * exp(-Y) : M / 2. * exp(Y);
  const double g = side ? fp.g2 : fp.g1;
  const double bmax = fmax(5. * g * kHc / k, 5. * fp.R);
  const double logd = row_log_step(bmax, fp.bmin);
  int cnt = 0;
  if (!fp.isPoint) {
    // b_j increases with j: binary search for the number of nodes with b <= 2R
    int lo = 0, hi = kNB1;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      double bl, bh;
      if (row_node(fp.bmin, logd, mid, &bl, &bh) > fp.twoR) hi = mid;
      else lo = mid + 1;
    }
    cnt = lo;
  }
  *k_out = k;
  *logd_out = logd;
  *cnt_out = cnt < kMaxQagsNodesPerRow ? cnt : kMaxQagsNodesPerRow;  // more only where k is NaN
}

// Bucket of a row in the photon energy order of the QAGS kernels:
// kRowsPerOctave buckets per factor of two of k over 40 octaves about 1 GeV,
// the end buckets taking what lies outside (NaN in the first).
__device__ __forceinline__ int row_bucket(double k)
{
  const float v = (__log2f((float)k) + 0.5f * kRowOctaves) * kRowsPerOctave;
  return v > 0.f ? (v < (float)(kRowBuckets - 1) ? (int)v : kRowBuckets - 1) : 0;
}

// fluxFormIntegrand (src/UpcCrossSection.cpp:181-191):
//   q^2 F(min(t, Q2max - dQ2)) / t * J1(b q / hc),  t = q^2 + (k / g1)^2
//
// The table's last knot is Q2min + (nQ2 - 1) dQ2 = 2 - 2e-6 (to rounding),
// so for t in (last knot, Q2max) the reference's gsl_spline_eval is out of
// range: GSL raises GSL_EDOM (its default handler ends the program).  The
// integrand returns NaN there and the QAGS run stops after that QK21 pass
// (kQagsEdom).
//
// The spline record is a dependent load from a 32 MB table: it is issued
// first and J1 (independent ALU work) runs while it is in flight.  The
// interval is the rounded estimate alone: within
// rounding of a knot the neighbouring cubic agrees to a few ulp.
//
// BR fixes J1's branch: 0 lets J1 choose (x <= 8 or not), 1 and 2 take the
// x <= 8 and x > 8 branches for a caller that has sorted its nodes by
// flux_j1_arg.  The operations are the same in all three forms, so a value
// does not depend on which one computed it.
__device__ __forceinline__ double flux_j1_arg(double b, double q) { return b * q * (1.0 / kHc); }

// The integrand in two steps: the spline record's load (issued early) and
// the rest once J1 is known.
struct FluxNode {
  double q, t, tc;
  int i;
  double4 c;  // spline interval record (in flight after flux_prelude)
};

__device__ __forceinline__ void flux_prelude(const double4* __restrict__ ff, double w2g2, double q, FluxNode* n)
{
  n->q = q;
  n->t = q * q + w2g2;
  n->tc = n->t < kQ2max ? n->t : kQ2max - kDQ2;
  int i = (int)((n->tc - kQ2min) * (1.0 / kDQ2));
  n->i = i < 0 ? 0 : (i > kNQ2 - 2 ? kNQ2 - 2 : i);
  n->c = ff[n->i];
}

// The integrand without J1.
__device__ __forceinline__ double flux_h(const FluxNode& n)
{
  const double d = n.tc - knot(kQ2min, kDQ2, n.i);
  const double f = n.c.x + d * (n.c.y + d * (n.c.z + d * n.c.w));
  const double h = n.q * n.q * f * rcp_nr(n.t);  // t >= (k / g1)^2 > 0
  return n.tc > kQ2Last ? __builtin_nan("") : h;
}

__device__ __forceinline__ double flux_finish(const FluxNode& n, double j1) { return flux_h(n) * j1; }

template <int BR>
__device__ __forceinline__ double bessel_j1_branch(double x)
{
  return BR == 1 ? bessel_j1_small(x) : (BR == 2 ? bessel_j1_large(x) : bessel_j1(x));
}

template <int BR>
__device__ __forceinline__ double flux_integrand(const double4* __restrict__ ff, double b, double w2g2, double q)
{
  FluxNode n;
  flux_prelude(ff, w2g2, q, &n);
  return flux_finish(n, bessel_j1_branch<BR>(flux_j1_arg(b, q)));
}

struct FluxFormIntegrand {
  const double4* __restrict__ ff;
  double b, w2g2;
  __device__ __forceinline__ double operator()(double q) const { return flux_integrand<0>(ff, b, w2g2, q); }
};

// Node j of flux row r: the point-charge flux (b > 2R or FLUX_POINT 1).  The
// form-factor nodes j < row_cnt[r] are left to the QAGS kernel.
__device__ __forceinline__ void point_row_node(long long r, int j, const FluxParams& fp,
                                               const double* __restrict__ row_k, const double* __restrict__ row_logd,
                                               const int* __restrict__ row_cnt, double* __restrict__ flux)
{
  if (j < row_cnt[r]) return;
  double bl, bh;
  const double b = row_node(fp.bmin, row_logd[r], j, &bl, &bh);
  flux[r * kNB1 + j] = flux_point(b, row_k[r], fp.g1, fp.factor);
}

// One form-factor flux integral (fluxForm, src/UpcCrossSection.cpp:194-218):
// flux[out] = factor (I / A)^2 / k.
struct FluxTask {
  double b, k;
  long out;
  const double4* ff;  // form-factor spline of the task's nucleus
  double g1, factor;
  int A;
  int slot;  // job of a batched task (0 otherwise)
};

// What the end of an integral needs: flux[out] = factor (I / A)^2 / k.
struct FluxOut {
  double k, factor;
  long out;
  int A;
};

// Task sources of the per-point QAGS kernel and of the 1000-interval kernel:
// get(t) describes task t.  Per-point tasks: an arbitrary (b, k).
struct PointTask {
  const double* __restrict__ b;
  const double* __restrict__ k;
  const int* __restrict__ idx;  // compacted indices of points needing QAGS
  FluxParams fp;
  const double4* ff;
  const unsigned long long* __restrict__ count;  // compacted points
  __device__ long long ids() const { return (long long)*count; }
  __device__ bool team(long long id, FluxTask* ft) const
  {
    get(id, ft);
    return true;
  }
  __device__ long long overflow_id(long long id) const { return id; }
  __device__ void get(long long t, FluxTask* ft) const
  {
    const int i = idx[t];
    ft->b = b[i];
    ft->k = k[i];
    ft->out = i;
    ft->ff = ff;
    ft->g1 = fp.g1;
    ft->factor = fp.factor;
    ft->A = fp.A;
    ft->slot = 0;
  }
  __device__ void out(long long t, FluxOut* fo) const
  {
    const int i = idx[t];
    fo->k = k[i];
    fo->out = i;
    fo->factor = fp.factor;
    fo->A = fp.A;
  }
  __device__ void failed(int) const {}
};

// What the integrals of one configuration share.
struct RowJob {
  const double4* ff;
  const double* j1;  // k_flux_j1's table
  double bmin, g1, factor;
  int A;
};

// A restricted grid takes part in its full grid's groups (all rows' factors,
// some lanes' integrals: the full grid's bits, at most its time) where at least
// one row in three is needed, else its rows in groups of their own: 0.45 of the
// time per row against 1.
constexpr int kNeedShare = 3;

// Flux rows of one context for the row kernels; as a task source, task t =
// row * 120 + node (its flux slot).
struct GridRows {
  const double* __restrict__ row_k;
  const double* __restrict__ row_logd;
  const int* __restrict__ row_cnt;
  int* __restrict__ perm;  // rows with form-factor nodes, ordered by k
  const unsigned long long* __restrict__ nsorted;  // rows in perm
  RowJob job;
  long long nrows;
  const unsigned char* __restrict__ need_row;  // null, or rows with 0 are left out
  // Restricted grids: the counts of two candidate launches, of which this one
  // runs when kNeedShare * *npart >= *nall (pick 1) or when not (pick 2).
  int pick;
  const unsigned long long *npart, *nall;
  // groups of 64 positions of perm; group(g): its first position, rows and job
  __device__ long long groups() const
  {
    if (pick != 0 && (kNeedShare * *npart >= *nall) != (pick == 1)) return 0;
    return ((long long)*nsorted + 63) / 64;
  }
  __device__ bool need(int r) const { return !need_row || need_row[r]; }
  __device__ int group(long long g, long long* first, int*) const
  {
    *first = g * 64;
    const long long left = (long long)*nsorted - *first;
    return left < 64 ? (int)left : 64;
  }
  // k_row_order: a job's rows [*r0, *r0 + return) and where they start in perm
  __device__ long long span(int, long long* r0, long long* pos0) const
  {
    *r0 = *pos0 = 0;
    return nrows;
  }
  // team work ids: (row, node), kMaxQagsNodesPerRow slots per row
  __device__ long long ids() const { return nrows * kMaxQagsNodesPerRow; }
  __device__ long long overflow_id(long long id) const
  {
    const long long r = id / kMaxQagsNodesPerRow;
    return r * kNB1 + (id - r * kMaxQagsNodesPerRow);
  }
  __device__ bool team(long long id, FluxTask* ft) const
  {
    const long long r = id / kMaxQagsNodesPerRow;
    if ((int)(id - r * kMaxQagsNodesPerRow) >= row_cnt[r]) return false;
    get(overflow_id(id), ft);
    return true;
  }
  __device__ RowJob params(int) const { return job; }
  __device__ void failed(int) const {}
  __device__ void get(long long t, FluxTask* ft) const
  {
    const long long r = t / kNB1;
    ft->b = row_node_b(job.bmin, row_logd[r], (int)(t - r * kNB1));
    ft->k = row_k[r];
    ft->out = t;
    ft->ff = job.ff;
    ft->g1 = job.g1;
    ft->factor = job.factor;
    ft->A = job.A;
    ft->slot = 0;
  }
};

// ---------------------------------------------------------------------------
// Form-factor flux at arbitrary points: persistent QAGS kernel.
//
// Each lane owns one integral at a time (the dqagse state machine of
// upc_qags.h, its interval lists in private memory) and takes a new task
// from a global cursor when it finishes.  A loop iteration is one dqagse
// step for every lane: the first QK21 pass of a new task, or the two halves
// of a bisection, in at most two rounds of one pass per lane.
//
// A round evaluates the 21 nodes of every lane's pass as one pool: each lane
// writes its abscissae to its row of the wavefront's LDS table and queues
// its nodes as J1 small-argument items (x = b q / hc <= 8, front of the
// queue) or large-argument items (after them).  The wavefront then sweeps
// the queue 64 items at a time, J1's small branch over the front and its
// large branch over the rest, each lane evaluating whichever node the queue
// hands it (the owner's b and (k/g)^2 come over ds_bpermute) and writing
// the value over the abscissa.  Every sweep runs one J1 branch on all 64
// lanes, where evaluating each lane's own nodes in turn would run both
// branches on almost every node (the two kinds are about evenly mixed in a
// grid: 47% small, 53% large on the 1001 x 121 Pb-Pb grid).  Finally each
// lane sums its own row in QK21's order (qk21_stored), so results are the
// same bits as a lane evaluating its own nodes.
//
// The LDS table (13,440 B per wavefront) sets the occupancy: 3 workgroups
// of 4 wavefronts per CU (127 VGPRs would admit 4).
//
// stats: [0] integrand evaluations, [1] integrals with ier != 0, [2]
// overflow count.
// ---------------------------------------------------------------------------
struct QagsWaveLds {
  double v[64 * 21];             // [owner lane][node e]: abscissa, then the integrand value
  unsigned short item[21 * 64];  // owner lane << 5 | e: small-argument items first, large after
};
constexpr int kQagsBlock = 256;      // threads of a workgroup (4 wavefronts, 53,760 B of LDS)
constexpr int kQagsBlocksPerCu = 3;  // resident workgroups per CU (LDS-bound)

__device__ __forceinline__ void wave_lds_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

__device__ __forceinline__ int lanes_below(unsigned long long m)
{
  return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// Items [beg, end) of the queue with J1 branch BR, 64 per sweep.  beg, end
// are wavefront-uniform, so every lane runs every ds_bpermute; a lane past
// end takes a dummy item (its own first node, abscissa 0) and stores
// nothing.  The fetch has no branch: every lane reads the queue (at a
// clamped index), its abscissa and a spline record (of a valid table: a
// lane's table pointer is set before its first task), so the record loads
// of a sweep's two items are issued unconditionally and each J1 waits only
// for its own record.
struct SweepItem {
  bool act;
  int slot;      // owner * 21 + e
  double x;      // J1 argument
  FluxNode n;
};

__device__ __forceinline__ void sweep_fetch(QagsWaveLds& W, int lane, int r0, int end, const double4* ff, double b,
                                            double w2g2, SweepItem* it)
{
  constexpr int kItems = 21 * 64;
  const int r = r0 + lane;
  it->act = r < end;
  const int raw = W.item[r < kItems ? r : kItems - 1];
  const int code = it->act ? raw : lane << 5;
  const int owner = code >> 5, e = code & 31;
  const double bo = __shfl(b, owner), wo = __shfl(w2g2, owner);
  it->slot = owner * 21 + e;
  const double qv = W.v[it->slot];
  const double q = it->act ? qv : 0.0;
  it->x = flux_j1_arg(bo, q);
  flux_prelude(ff, wo, q, &it->n);
}

template <int BR>
__device__ __forceinline__ void sweep_finish(QagsWaveLds& W, const SweepItem& it)
{
  const double v = flux_finish(it.n, bessel_j1_branch<BR>(it.x));
  if (it.act) W.v[it.slot] = v;
}

// Two items per lane in flight: both fetches (queue entry, owner's
// parameters, abscissa, spline record load) are issued before either J1.
// The J1s run at a raised wave priority, so the SIMD issues them ahead of
// the other waves' fetches and bookkeeping, whose waits then overlap them
// (2 % on the QAGS phase).  A remainder of at most 64 items takes one sweep
// of its own.
template <int BR>
__device__ __forceinline__ void qags_sweeps(QagsWaveLds& W, int lane, int beg, int end, const double4* ff,
                                            double b, double w2g2)
{
  int r0 = beg;
#pragma unroll 1
  for (; r0 + 64 < end; r0 += 128) {
    SweepItem ia, ib;
    sweep_fetch(W, lane, r0, end, ff, b, w2g2, &ia);
    sweep_fetch(W, lane, r0 + 64, end, ff, b, w2g2, &ib);
    __builtin_amdgcn_s_setprio(2);
    sweep_finish<BR>(W, ia);
    sweep_finish<BR>(W, ib);
    __builtin_amdgcn_s_setprio(0);
  }
  if (r0 < end) {
    SweepItem ia;
    sweep_fetch(W, lane, r0, end, ff, b, w2g2, &ia);
    sweep_finish<BR>(W, ia);
  }
}

// Node of QK21 in ascending abscissa order k = 0..20: the left nodes
// centr - hlgth kXgk[k] (kXgk decreasing), the centre, the right nodes.
__device__ __forceinline__ int qk21_qorder_node(int k)
{
  return k < 10 ? qk21_node(k, 0) : (k == 10 ? 0 : qk21_node(20 - k, 1));
}

// Exclusive prefix sum over the wavefront's lanes of x in [0, 32), and the
// total: one ballot per bit.
__device__ __forceinline__ int wave_prefix5(int x, int* total)
{
  int pre = 0, tot = 0;
#pragma unroll
  for (int bit = 0; bit < 5; ++bit) {
    const unsigned long long m = __ballot((x >> bit) & 1);
    pre += lanes_below(m) << bit;
    tot += __popcll(m) << bit;
  }
  *total = tot;
  return pre;
}

// One QK21 pass per lane with mine set, on [qa, qb]; the result for those
// lanes (zeros elsewhere).  ff, b, w2g2: the lane's own integrand.
//
// J1's argument b q / hc grows with the abscissa, so a lane's small-argument
// nodes are the first ns of its nodes in abscissa order: the lane's items
// are two runs, [ps, ps + ns) among the small items and the rest among the
// large ones, placed by one prefix sum over the lanes.
__device__ __forceinline__ QK21Out qk21_wave(QagsWaveLds& W, int lane, bool mine, double qa, double qb,
                                             const double4* ff, double b, double w2g2)
{
  const double centr = 0.5 * (qa + qb), hlgth = 0.5 * (qb - qa);
  double* col = W.v + lane * 21;
  wave_lds_sync();
  // the abscissae of qk21_abscissa, a pair (both sides of kXgk[j]) at a time
  col[0] = centr;
  int ns = flux_j1_arg(b, centr) <= 8.0;
#pragma unroll 5
  for (int j = 0; j < 10; ++j) {
#pragma clang fp contract(off)  // absc rounded before the sums, as QUADPACK computes it
    const double absc = hlgth * kXgk[j];
    const double ql = centr - absc, qr = centr + absc;
    const int e = qk21_node(j, 0);
    col[e] = ql;
    col[e + 1] = qr;
    ns += (flux_j1_arg(b, ql) <= 8.0) + (flux_j1_arg(b, qr) <= 8.0);
  }
  if (!mine) ns = 0;
  int S = 0;
  const int ps = wave_prefix5(ns, &S);
  const unsigned long long act = __ballot(mine);
  const int ntot = 21 * __popcll(act);
  const int pl = S + 21 * lanes_below(act) - ps;  // start of the lane's large run
  if (mine) {
#pragma unroll 1
    for (int k = 0; k < 21; ++k) {
      const int e = qk21_qorder_node(k);
      W.item[k < ns ? ps + k : pl + (k - ns)] = (unsigned short)(lane << 5 | e);
    }
  }
  wave_lds_sync();
  qags_sweeps<1>(W, lane, 0, S, ff, b, w2g2);
  qags_sweeps<2>(W, lane, S, ntot, ff, b, w2g2);
  wave_lds_sync();
  QK21Out o{};
  if (mine) o = qk21_stored(col, 1, qa, qb);
  return o;
}

template <int CAP, class TS>
__global__ __launch_bounds__(kQagsBlock) __attribute__((amdgpu_waves_per_eu(kQagsBlocksPerCu, kQagsBlocksPerCu)))
void k_flux_qags(TS ts, const unsigned long long* __restrict__ ntasks_p, unsigned long long* __restrict__ cursor,
                 double* __restrict__ flux, int* __restrict__ ier_out, unsigned long long* __restrict__ stats,
                 long long* __restrict__ overflow, int fast_cap)
{
  __shared__ QagsWaveLds lds[kQagsBlock / 64];
  QagsWaveLds& W = lds[threadIdx.x >> 6];
  typename QagsSmallStore<CAP>::Arrays lists;
  Qags<QagsSmallStore<CAP>> q;
  q.s.a = &lists;
  q.s.lim = fast_cap < CAP ? fast_cap : CAP;
  const long long ntasks = (long long)*ntasks_p;
  const int lane = threadIdx.x & 63;
  long long task = -1;  // -1: needs a task; LLONG_MAX: exhausted
  // Live across the steps of a task: b and (k/g)^2; the output fields (k, slot, factor, A) are read again when it ends.
  double ft_b = 0.0, w2g2 = 0.0;
  unsigned my_evals = 0, my_bad = 0;  // 32-bit per lane; evaluations flushed before they could wrap
  while (true) {
    bool need = task < 0;
    unsigned long long mask;
    while ((mask = __ballot(need)) != 0) {
      const int leader = __ffsll((long long)mask) - 1;
      unsigned long long base = 0;
      if (lane == leader) base = atomicAdd(cursor, (unsigned long long)__popcll(mask));
      base = __shfl(base, leader);
      if (need) {
        const long long t = (long long)(base + (unsigned long long)lanes_below(mask));
        if (t < ntasks) {
          task = t;
          FluxTask ft;
          ts.get(t, &ft);
          ft_b = ft.b;
          w2g2 = ft.k * ft.k / ft.g1 / ft.g1;
          q.start();
        } else {
          task = LLONG_MAX;
        }
        need = false;
      }
    }
    if (__ballot(task != LLONG_MAX) == 0) break;
    const bool live = task != LLONG_MAX;
    const int np = live ? q.passes() : 0;
    double qa = 0.0, qb = 0.0;
    if (live) q.interval(0, &qa, &qb);
    const QK21Out o = qk21_wave(W, lane, live, qa, qb, ts.ff, ft_b, w2g2);
    QK21Out o2{};
    if (__ballot(np == 2) != 0) {
      if (np == 2) q.interval(1, &qa, &qb);
      o2 = qk21_wave(W, lane, np == 2, qa, qb, ts.ff, ft_b, w2g2);
    }
    if (!live) continue;
    const int st = q.consume(o, o2);
    if (st == kQagsDone) {
      FluxOut fo;
      ts.out(task, &fo);
      const double Q = q.result / fo.A;
      flux[fo.out] = fo.factor * Q * Q / fo.k;
      const int status = q.status();
      if (ier_out) ier_out[fo.out] = status;
      my_evals += (unsigned)q.neval();
      if (my_evals >= 0x80000000u) {
        atomicAdd(&stats[0], (unsigned long long)my_evals);
        my_evals = 0;
      }
      my_bad += status != 0;
      task = -1;
    } else if (st == kQagsOverflow) {
      const unsigned long long slot = atomicAdd(&stats[2], 1ull);
      overflow[slot] = task;
      task = -1;
    }
  }
  unsigned long long evals = my_evals, bad = my_bad;
  for (int o = 32; o > 0; o >>= 1) {
    evals += __shfl_down(evals, o);
    bad += __shfl_down(bad, o);
  }
  if (lane == 0) {
    atomicAdd(&stats[0], evals);
    atomicAdd(&stats[1], bad);
  }
}

// ---------------------------------------------------------------------------
// Form-factor flux of whole flux rows.
//
// A wavefront takes 64 rows that are neighbours in photon energy k (rows are
// bucket-sorted by k) and one node index j, one integral per lane.  b_j and
// (k/g)^2 then differ by a fraction of a percent over the lanes, so nearly
// every dqagse decision is the same for all of them: on the 1001 x 121 Pb-Pb
// grid 99 % of the QK21 passes are on one interval for the whole wavefront,
// 99.7 % of the lane steps are in use although a lane that ends early waits
// for the others, and J1's branch (x = b q / hc <= 8 or not) is mixed in 0.5 %
// of the node evaluations (101 x 41: 92 %, 91 %, 4 %).  So each lane
// evaluates its own nodes directly, in QK21's summation order, with J1's
// branch taken by the whole wavefront; the spline records of one node lie
// side by side over the lanes.  A pass keeps its 20 off-centre values in LDS
// (10,240 B per wavefront) for the mean deviation.
//
// Against the per-point kernel above over the same integrals (1001 x 121
// Pb-Pb): 14.2 -> 10.4 ms, 158 -> 124 VALU instructions per integrand value,
// no task records (24 B each) written and read.  Bound: VALU issue (80 % of
// the time at 3 waves per SIMD, no spills).  Two nodes per trip spill 44 VGPRs
// (10.2 ms, slower on small grids); 4 waves per SIMD spill 66 (10.1 ms, same).
//
// Work ids are (group of 64 rows, j), taken from a global cursor; ids whose
// group has no node j end at once.  stats as in k_flux_qags; overflow receives flux slots (row * 120
// + node).  The kernel is in upc_flux_rows.hip; it runs where rows are too far
// apart in k for the next one.
// ---------------------------------------------------------------------------
constexpr int kQagsRowsWaves = 3;        // waves per SIMD (register and LDS budget)
constexpr int kQagsRowsBlocksPerCu = 3;  // resident workgroups of kQagsBlock per CU

// One QK21 pass on [qa, qb] (the lane's own) for every active lane:
// qk21_stored's sums in its order, the integrand evaluated on the way.  fv:
// where the off-centre values wait for the mean deviation, STRIDE apart (the
// nodes are visited in a rolled loop).
template <int STRIDE>
__device__ __forceinline__ QK21Out qk21_rows(double* fv, double qa, double qb, const double4* __restrict__ ff,
                                             double b, double w2g2)
{
  const double centr = 0.5 * (qa + qb), hlgth = 0.5 * (qb - qa);
  double resg = 0.0, resk = 0.0, rabs = 0.0, fc = 0.0, f1 = 0.0;
#pragma unroll 1
  for (int e = 0; e < 21; ++e) {  // the centre, the Gauss pairs, the Kronrod-only pairs (left, right)
    const double f = flux_integrand<0>(ff, b, w2g2, qk21_abscissa(e, centr, hlgth));
    if (e == 0) {
      fc = f;
      resk = kWgk[10] * fc;
      rabs = fabs(resk);
      continue;
    }
    fv[(e - 1) * STRIDE] = f;
    if (e & 1) {
      f1 = f;
      continue;
    }
    const double fsum = f1 + f;
    const int p = (e >> 1) - 1;
    const int j = p < 5 ? 2 * p + 1 : 2 * (p - 5);
    if (p < 5) resg = resg + kWg[p] * fsum;
    resk = resk + kWgk[j] * fsum;
    rabs = rabs + kWgk[j] * (fabs(f1) + fabs(f));
  }
  return qk21_tail([&](int j, int side) { return fv[(qk21_node(j, side) - 1) * STRIDE]; }, resg, resk, rabs, fc, hlgth);
}

// ---------------------------------------------------------------------------
// The same for rows that lie close together in k: the integrand's two factors,
// h(q) of the row and J1(b q / hc), each shared by many integrals.
//
// - h at the nodes of the 25 intervals that nearly all passes are on is
//   tabulated per row (k_flux_h) for the row's 30 to 97 integrals.
// - J1: rows with k above gamma hc / R share one b grid (b_max = 5 R there) and
//   read J1 from one table per configuration (k_flux_j1), half of the passes
//   on the Pb-Pb and Au-Au grids; elsewhere the wavefront expands J1 once per
//   node about the middle of its lanes' b (expand_j1) and every lane evaluates
//   the polynomial.
// - The lists of the bookkeeping are in LDS (QagsLdsStore), the pass's 21
//   values in registers: 2 waves per SIMD.
//
// Lanes on other intervals than the first take their turn after it; intervals
// outside the table and lanes too far apart for the expansion evaluate their
// own nodes (qk21_rows).
//
// 1001 x 121 Pb-Pb: 10.4 -> 4.7 ms against k_flux_qags_rows, 124 -> 37 VALU
// instructions per integrand value; 8 mixed jobs 55 -> 35 ms (whole batch).
// Bound: instruction issue and the latency of dependent FP64 and LDS operations
// at 2 waves per SIMD.  Parts (wave cycles): values and sums 40 %, bookkeeping
// 28 %, expansions 16 %, loads of h 6 %, row set-up 6 %, own nodes 4 %.  Tried:
// lists in private memory with 3 waves per SIMD 6.4 ms (values through LDS),
// 9.8 ms (182 VGPRs spilled); coefficients broadcast from LDS to every lane
// 4.9 ms (LDS 38 % busy).
//
// Work ids are (group of 64 rows, j).  A launch takes `chunk` groups from g0 on,
// as many as H holds (269 KB each).  The j of a group share its h, so
// a group belongs to one XCD's cursor (workgroups are dealt to the XCDs in
// turn): the few groups in flight on an XCD stay in its L2.
// ---------------------------------------------------------------------------
constexpr int kQagsTableWaves = 2;        // waves per SIMD (register and LDS budget)
constexpr int kQagsTableBlocksPerCu = 2;  // resident workgroups of kQagsBlock per CU
constexpr int kXcds = 8;
constexpr int kRowsChunk = 4096;  // groups of 64 rows per launch (1.1 GB of h)
constexpr int kRowsTurns = 4;     // intervals a step takes one by one before its other lanes evaluate their own

// h of the intervals that most passes are on: level L of the bisection of
// [0, 10] holds intervals m < kHCount[L], first slot kHFirst[L].  Below q ~ 1.4
// the form factor falls off, so dqagse bisects towards q = 0: these 25
// intervals take 99 % of the passes (Pb 5.02 TeV, O 7 TeV, Au 200 GeV grids).
constexpr int kHLevels = 10, kHSlots = 25;
constexpr int kHGroupElems = kHSlots * 21 * 64;  // of one group of rows
__device__ constexpr int kHCount[kHLevels] = {1, 2, 2, 2, 2, 4, 6, 2, 2, 2};
__device__ constexpr int kHFirst[kHLevels] = {0, 1, 3, 5, 7, 9, 13, 19, 21, 23};

// Slot of interval m of level L, -1: none.
__device__ __forceinline__ int h_slot(unsigned L, unsigned m)
{
  if (L >= (unsigned)kHLevels) return -1;
  return m < (unsigned)kHCount[L] ? kHFirst[L] + (int)m : -1;
}

// h(q) = q^2 F(t) / t of the rows at the nodes of those intervals, which the
// 30 to 97 integrals of a row all read: H[group][slot][node][lane], for the
// groups of 64 rows from g0 on.  One block per group and slot.
// Bound by its stores (10.75 KB per group and slot).
template <class RS>
__global__ __launch_bounds__(256) void k_flux_h(RS rs, long long g0,
                                                double* __restrict__ H)
{
  const int slot = blockIdx.x % kHSlots, gl = blockIdx.x / kHSlots;
  if (g0 + gl >= rs.groups()) return;
  long long first;
  int job = 0;
  const int n = rs.group(g0 + gl, &first, &job);
  if (n <= 0) return;
  int L = 0;
  while (L + 1 < kHLevels && kHFirst[L + 1] <= slot) ++L;
  const double w = ldexp(kQagsB, -L), qa = (slot - kHFirst[L]) * w, qb = (slot - kHFirst[L] + 1) * w;
  const int lane = threadIdx.x & 63;
  const int r = rs.perm[first + (lane < n ? lane : n - 1)];
  const RowJob P = rs.params(job);
  const double k = rs.row_k[r];
  const double w2g2 = k * k / P.g1 / P.g1;
  double* out = H + ((long long)gl * kHSlots + slot) * (21 * 64) + lane;
  for (int e = threadIdx.x >> 6; e < 21; e += 4) {
    FluxNode node;
    flux_prelude(P.ff, w2g2, qk21_abscissa(e, 0.5 * (qa + qb), 0.5 * (qb - qa)), &node);
    out[e * 64] = flux_h(node);
  }
}

// J1 at the nodes of those intervals on the b grid that all rows with b_max =
// 5 R share (k above gamma hc / R): T[0] the grid's log step, then [j][slot][
// node].  One block per j.
constexpr int kJ1TableElems = 1 + kMaxQagsNodesPerRow * kHSlots * 21;

// Scalar-cache reads of a table that no kernel of the launch writes.
using ConstD = const __attribute__((address_space(4))) double;

// J1 of a whole wavefront at one node.  Where the lanes are on one interval,
// node e has one q and the lanes' arguments b q / hc lie within a fraction of
// a percent of x0 = b0 q / hc, b0 the middle of their b.  One lane per node
// expands J1 about its x0 (from J1, J0 and Bessel's equation, below), and
// every lane evaluates the polynomial at its own db = (b - b0) / hc: T - 1
// FMAs on coefficients (powers of q folded in) that all lanes read from the
// same LDS address, where J1 itself takes 35 (x <= 8) or 75 FP64
// instructions.  On rows whose b grids coincide (k above gamma hc / R: b_max
// = 5 R) db is 0 and T = 1.
//
// With delta = q db, T terms leave |delta|^T / T!; kExpandMax[i] is the delta
// up to which this is below 1.5e-19, i.e. 2e-17 of J1 ~ x / 2 at the
// smallest x of an interval's end (0.015).  The recurrence's rounding enters
// as (delta / x0)^n and stays below the rounding of J1(x0) for delta / x0 = db /
// (b0 / hc) up to kExpandRatio: with the kernel's J1 (itself 4.2e-16) within
// 4.9e-16 of the envelope there; with exact J0 and J1(x0) 2.0e-16, and 4.8e-16 at
// 0.5, 2.6e-15 at 0.8, 2.8e-13 at 0.99.  A group of rows further apart evaluates
// its own nodes: none on grids or points spread evenly (0.04 on 1001 x 121, 0.18
// at most from 8,192 rows on), but a dense cluster of points beside distant ones.
constexpr double kExpandRatio = 0.2;
constexpr int kExpandKinds = 7;
__device__ constexpr int kExpandTerms[kExpandKinds] = {1, 4, 6, 8, 10, 14, 20};
__device__ constexpr double kExpandMax[kExpandKinds] = {0.0, 4.3e-5, 2.1e-3, 1.6e-2, 5.9e-2, 0.265, 0.939};
constexpr int kExpandBoth = 10;    // up to this many terms both halves of a bisection are expanded at once
constexpr int kExpandSlots = 436;  // coefficients: 42 nodes x 10 terms or 21 x 20

// The recurrence's numbers, n = 0 .. 17: 1 / ((n+1)(n+2)), (n^2-1) / ((n+1)(n+2)), (2n+1) / (n+2).
struct ExpandTable {
  double v[18];
};
template <class F>
constexpr ExpandTable expand_table(F f)
{
  ExpandTable t{};
  for (int n = 0; n < 18; ++n) t.v[n] = f((double)n);
  return t;
}
__constant__ static const ExpandTable kExpandAt = expand_table([](double n) { return 1.0 / ((n + 1) * (n + 2)); });
__constant__ static const ExpandTable kExpandBt = expand_table([](double n) { return (n - 1) / (n + 2); });
__constant__ static const ExpandTable kExpandCt = expand_table([](double n) { return (2 * n + 1) / (n + 2); });

// A value that all lanes hold, in scalar registers.
__device__ __forceinline__ double wave_uniform(double v)
{
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                          __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// Index into kExpandTerms for delta (the same in all lanes); kExpandKinds: too
// wide.  mymax: kExpandMax[lane] (beyond the table: infinite).
__device__ __forceinline__ int expand_kind(double delta, double mymax)
{
  return __popcll(__ballot(delta > mymax));
}

// Coefficients a_n q^n, n < T, of J1 about x0 = b0 q / hc into cf.  With r = 1 /
// x0, x^2 y'' + x y' + (x^2 - 1) y = 0 gives
//   (n+1)(n+2) a_{n+2} = -[(n+1)(2n+1) r a_{n+1} + ((n^2-1) r^2 + 1) a_n
//                          + 2 r a_{n-1} + r^2 a_{n-2}].
__device__ __forceinline__ void expand_j1(double* cf, double b0, double q, int T)
{
  const double x0 = flux_j1_arg(b0, q);
  if (T == 1) {
    cf[0] = bessel_j1(x0);
    return;
  }
  double j0, j1;
  bessel_j01(x0, &j0, &j1);
  cf[0] = j1;
  const double r = rcp_nr(x0), r2 = r * r;
  double am2 = 0.0, am1 = 0.0, a = j1, ap = fma(-j1, r, j0), qn = q;  // a_{n-2}, a_{n-1}, a_n, a_{n+1}, q^{n+1}
  cf[1] = ap * q;
#pragma unroll 2
  for (int n = 0; n < T - 2; ++n) {
    // everything but the a_{n+1} term first: one dependent FMA per coefficient
    const double s = fma(fma(kExpandBt.v[n], r2, kExpandAt.v[n]), a, kExpandAt.v[n] * fma(2.0 * r, am1, r2 * am2));
    const double an = -fma(kExpandCt.v[n] * r, ap, s);
    qn *= q;
    cf[n + 2] = an * qn;
    am2 = am1;
    am1 = a;
    a = ap;
    ap = an;
  }
}

// f = h J1 at the 21 nodes of a pass: tabulated h in f, J1 expanded (cf: T
// coefficients per node).  All lanes take part.
using LdsCoef = const __attribute__((address_space(3))) double;

// j += c[N] p0 + c[N + 1] p1, ...: c[n] lane n of each row of 16 lanes.
//
// Every lane needs every coefficient.  Read from LDS by all lanes, one costs
// 512 B of the CU's LDS bandwidth (4 cycles; 24 terms of 3 nodes at a time
// kept it 38 % busy and waited 5000 cycles per pass); here 16 coefficients
// fill one register over a row of 16 lanes and the row broadcast of the FMA's
// DPP form hands them out.  s_nop: a DPP source must not have been written by
// the VALU in the last two wait states.
template <int N>
__device__ __forceinline__ void bcast_fma2(double& j, double c, const double* p)
{
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %1, %3 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:%4 row_mask:0xf bank_mask:0xf"
      : "+v"(j)
      : "v"(c), "v"(p[0]), "v"(p[1]), "i"(N), "i"(N + 1));
}
template <int N>
__device__ __forceinline__ void bcast_fma4(double& j, double c, const double* p)
{
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %1, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %4 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %3 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:%6 row_mask:0xf bank_mask:0xf"
      : "+v"(j)
      : "v"(c), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "i"(N), "i"(N + 1), "i"(N + 2), "i"(N + 3));
}

// Terms K - 1 .. 0 of node E, the highest first (the smallest terms are summed
// first, as in Horner's order).
template <int T, int E, int K>
__device__ __forceinline__ void bcast_terms(double& j, const double* cr, const double* pw)
{
  if constexpr (K > 0) {
    constexpr int i = E * T + K;  // one past the term
    constexpr int n = K >= 4 && (i - 4) / 16 == (i - 1) / 16 ? 4 : 2;
    if constexpr (n == 4) bcast_fma4<(i - 4) % 16>(j, cr[(i - 4) / 16], pw + K - 4);
    else bcast_fma2<(i - 2) % 16>(j, cr[(i - 2) / 16], pw + K - 2);
    bcast_terms<T, E, K - n>(j, cr, pw);
  }
}

template <int T, int E>
__device__ __forceinline__ void bcast_nodes(double* f, const double* cr, const double* pw)
{
  if constexpr (E < 21) {
    double j1 = 0.0;
    bcast_terms<T, E, T>(j1, cr, pw);
    f[E] *= j1;
    asm volatile("" : "+v"(f[E]));  // rounded here: no contraction with the sums below
    bcast_nodes<T, E + 1>(f, cr, pw);
  }
}

template <int T>
__device__ __forceinline__ void expanded_values(double* f, LdsCoef* cf, int lane, double db)
{
  static_assert(T % 2 == 0, "terms are taken in pairs");
  if constexpr (T <= 10) {
    double cr[(21 * T + 15) / 16], pw[T];
    asm volatile("" : "+v"(db));  // its powers are made here, not kept in registers over the whole integral
#pragma unroll
    for (int i = 0; i < (21 * T + 15) / 16; ++i) cr[i] = cf[16 * i + (lane & 15)];
    pw[0] = 1.0;
#pragma unroll
    for (int k = 1; k < T; ++k) pw[k] = pw[k - 1] * db;
    bcast_nodes<T, 0>(f, cr, pw);
  } else {
    // too many powers for the registers: Horner's rule, coefficients from LDS
#pragma unroll
    for (int e = 0; e < 21; e += 3) {  // three chains side by side
      LdsCoef* c = cf + e * T;
      double j[3] = {c[T - 1], c[2 * T - 1], c[3 * T - 1]};
#pragma unroll 4
      for (int k = T - 2; k >= 0; --k) {
#pragma unroll
        for (int i = 0; i < 3; ++i) j[i] = fma(j[i], db, c[i * T + k]);
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        f[e + i] *= j[i];
        asm volatile("" : "+v"(f[e + i]));
      }
      __builtin_amdgcn_sched_barrier(0);  // bounds the coefficients in flight
    }
  }
}

__device__ __forceinline__ void expanded_values_t(int kind, double* f, const double* cf_, int lane, double db)
{
  LdsCoef* cf = (LdsCoef*)cf_;
  asm volatile("" : "+v"(cf));  // one address register, the coefficients at immediate offsets
  switch (kind) {
    case 0:  // db = 0: J1 itself
#pragma unroll
      for (int e = 0; e < 21; ++e) {
        f[e] *= cf[e];
        asm volatile("" : "+v"(f[e]));
      }
      break;
    case 1: expanded_values<4>(f, cf, lane, db); break;
    case 2: expanded_values<6>(f, cf, lane, db); break;
    case 3: expanded_values<8>(f, cf, lane, db); break;
    case 4: expanded_values<10>(f, cf, lane, db); break;
    case 5: expanded_values<14>(f, cf, lane, db); break;
    default: expanded_values<20>(f, cf, lane, db);
  }
}

// f = h J1 with J1 from the shared grid's table.
__device__ __forceinline__ void table_values(double* f, ConstD* j1)
{
#pragma unroll
  for (int e = 0; e < 21; ++e) {
    f[e] *= j1[e];
    asm volatile("" : "+v"(f[e]));  // rounded here: no contraction with the sums below
  }
}

// QK21 of the 21 values in registers, in its summation order.
__device__ __forceinline__ QK21Out qk21_values(const double* f, double hlgth)
{
  double resg = 0.0, resk = kWgk[10] * f[0];
  double rabs = fabs(resk);
#pragma unroll
  for (int p = 0; p < 10; ++p) {
    const int j = p < 5 ? 2 * p + 1 : 2 * (p - 5);  // the Gauss pairs, then the Kronrod-only pairs
    const double f1 = f[2 * p + 1], f2 = f[2 * p + 2];
    const double fsum = f1 + f2;
    if (p < 5) resg = resg + kWg[p] * fsum;
    resk = resk + kWgk[j] * fsum;
    rabs = rabs + kWgk[j] * (fabs(f1) + fabs(f2));
  }
  return qk21_tail([&](int j, int side) { return f[qk21_node(j, side)]; }, resg, resk, rabs, f[0], hlgth);
}

template <int CAP, class RS>
__global__ __launch_bounds__(kQagsBlock) __attribute__((amdgpu_waves_per_eu(kQagsTableWaves, kQagsTableWaves)))
void k_flux_qags_table(RS rs, long long g0, int chunk,
                      const double* __restrict__ H, unsigned long long* __restrict__ cursors,
                      double* __restrict__ flux, unsigned long long* __restrict__ stats,
                      long long* __restrict__ overflow, int fast_cap)
{
  using Store = QagsLdsStore<CAP>;
  struct WaveLds {
    typename Store::Columns lists;
    double cf[kExpandSlots];  // J1 expansions, [node][term]
  };
  __shared__ WaveLds lds[kQagsBlock / 64];
  const int lane = threadIdx.x & 63;
  double* cf = lds[threadIdx.x >> 6].cf;
  typename Store::Arrays lists;
  Qags<Store> q;
  q.s.bind(&lds[threadIdx.x >> 6].lists, lane, &lists);
  q.s.lim = fast_cap < CAP ? fast_cap : CAP;
  // groups of this launch, and those of cursor x: g0 + x, g0 + x + kXcds, ...
  const long long left = rs.groups() - g0, ngroups = left < chunk ? left : chunk;
  unsigned my_evals = 0, my_bad = 0;  // 32-bit per lane; evaluations flushed before they could wrap
  const double mymax = lane < kExpandKinds ? kExpandMax[lane < kExpandKinds ? lane : 0] : __builtin_inf();
  int x = blockIdx.x % kXcds, tried = 0;
  unsigned next = 0;  // lane 0: the id after the current one, asked for while that one runs
  if (lane == 0) next = (unsigned)atomicAdd(&cursors[x], 1ull);
  while (ngroups > 0) {
    const unsigned id = __builtin_amdgcn_readfirstlane(next);
    const int gi = (int)(id / kMaxQagsNodesPerRow), j = (int)(id - gi * kMaxQagsNodesPerRow);
    const int gl = gi * kXcds + x;
    if (gl >= ngroups) {  // this cursor's groups are done: help with the next
      if (++tried == kXcds) break;
      x = (x + 1) % kXcds;
      if (lane == 0) next = (unsigned)atomicAdd(&cursors[x], 1ull);
      continue;
    }
    if (lane == 0) next = (unsigned)atomicAdd(&cursors[x], 1ull);
    const double* hg = H + (long long)gl * kHGroupElems;
    long long first;
    int r = 0, job = 0;
    bool live = false;
    if (lane < rs.group(g0 + gl, &first, &job)) {
      r = rs.perm[first + lane];
      live = j < rs.row_cnt[r];
    }
    if (__ballot(live) != 0) {
      const RowJob P = rs.params(job);
      double b = 0.0;
      if (live) {
        b = row_node_b(P.bmin, rs.row_logd[r], j);
        q.start();
      }
      // the middle of the lanes' b, and their distance from it in J1's argument per q
      double blo = live ? b : DBL_MAX, bhi = live ? b : 0.0;
      for (int o = 32; o > 0; o >>= 1) {
        blo = fmin(blo, __shfl_xor(blo, o));
        bhi = fmax(bhi, __shfl_xor(bhi, o));
      }
      const double b0 = wave_uniform(0.5 * (blo + bhi));
      // Rows too far apart for an expansion: none (infinitely far), and likewise where
      // a row has no b (no photon energy, M = 0): its values are NaN, not its neighbours' J1.
      const bool apart = __ballot(live && !(fabs(b - b0) <= kExpandRatio * b0)) != 0;
      const double db = (b - b0) * (1.0 / kHc);
      const double dbm = wave_uniform(apart ? __builtin_inf() : fmax(b0 - blo, bhi - b0) * (1.0 / kHc));
      live = live && rs.need(r);
      // every row on the shared b grid: J1 from its table
      const bool shared = __ballot(live && rs.row_logd[r] != P.j1[0]) == 0;
      ConstD* j1t = (ConstD*)(P.j1 + 1) + j * (kHSlots * 21);
      int np = 1;  // passes of the step: the whole range first, then the halves of every lane's interval
      unsigned long long rem;
      while ((rem = __ballot(live)) != 0) {
        QK21Out o{}, o2{};
        q.phase = np == 1 ? 0 : 2;
        // the lanes of one interval at a time (nearly always all of them)
        for (int turn = 0; rem != 0; ++turn) {
          const unsigned iv = __builtin_amdgcn_readlane(q.cur, __ffsll((long long)rem) - 1);
          const unsigned L = iv >> 26, im = iv & 0x3ffffffu;
          // [lo, hi] = 10 2^-L [m, m + 1], built exactly (10 2^-L from its bits)
          const double w = __hiloint2double(0x40240000 - ((int)L << 20), 0);
          const double lo = wave_uniform((double)im * w), mid = wave_uniform(lo + 0.5 * w), hi = wave_uniform(lo + w);
          const int slot = np == 1 ? h_slot(L, im) : h_slot(L + 1, 2 * im);
          const int kind = shared ? 0 : expand_kind(hi * dbm, mymax);
          const bool mine = (rem >> lane & 1) != 0;
          if (slot < 0 || kind == kExpandKinds || turn == kRowsTurns) {
            if (mine) {
#pragma unroll 1
              for (int pass = 0; pass < np; ++pass) {
                double la, lb;
                q.interval(pass, &la, &lb);
                // rare: b and (k/g)^2 are found again instead of kept in registers
                const double k = rs.row_k[r];
                o = o2;
                double fv[20];
                o2 = qk21_rows<1>(fv, la, lb, P.ff, row_node_b(P.bmin, rs.row_logd[r], j), k * k / P.g1 / P.g1);
              }
              if (np == 1) o = o2;
            }
            break;
          }
          const int T = kExpandTerms[kind];
          const bool both = T <= kExpandBoth;
          auto expand = [&](int first, int n) {
            wave_lds_sync();
            if (lane < n) {
              const int second = lane >= 21, pass = first + second;
              const double qa = pass ? mid : lo, qb = np == 2 && !pass ? mid : hi;
              expand_j1(cf + lane * T, b0, qk21_abscissa(lane - 21 * second, 0.5 * (qa + qb), 0.5 * (qb - qa)), T);
            }
            wave_lds_sync();
          };
          const double* hp = hg + slot * (21 * 64);
          const bool here = mine && q.cur == iv;
#pragma unroll 1
          for (int pass = 0; pass < np; ++pass) {
            if (!shared && (pass == 0 || !both)) expand(pass, both ? 21 * np : 21);
            double f[21];
#pragma unroll
            for (int e = 0; e < 21; ++e) f[e] = hp[(21 * pass + e) * 64 + lane];
            if (shared) table_values(f, j1t + (slot + pass) * 21);
            else expanded_values_t(kind, f, cf + (both ? 21 * pass * T : 0), lane, db);
            const QK21Out on = qk21_values(f, np == 2 ? 0.25 * w : 0.5 * w);
            if (here) {
              o = o2;
              o2 = on;
            }
          }
          if (np == 1 && here) o = o2;
          rem &= ~__ballot(here);
        }
        np = 2;
        if (!live) continue;
        const int st = q.consume(o, o2);
        if (st == kQagsRunning) continue;
        live = false;
        const long long slot = (long long)r * kNB1 + j;
        if (st == kQagsDone) {
          const double Q = q.result / P.A;
          flux[slot] = P.factor * Q * Q / rs.row_k[r];
          my_evals += (unsigned)q.neval();
          if (my_evals >= 0x80000000u) {
            atomicAdd(&stats[0], (unsigned long long)my_evals);
            my_evals = 0;
          }
          if (q.status() != 0) {
            my_bad++;
            rs.failed(job);
          }
        } else {
          overflow[atomicAdd(&stats[2], 1ull)] = slot;
        }
      }
    }
  }
  unsigned long long evals = my_evals, bad = my_bad;
  for (int o = 32; o > 0; o >>= 1) {
    evals += __shfl_down(evals, o);
    bad += __shfl_down(bad, o);
  }
  if (lane == 0) {
    atomicAdd(&stats[0], evals);
    atomicAdd(&stats[1], bad);
  }
}

// ---------------------------------------------------------------------------
// Form-factor flux, few integrals: G lanes per integral.
//
// With one integral per lane an integral takes some 300 integrand values one
// after another, 0.4 ms whatever the count, and a launch of fewer integrals
// than the chip has lanes leaves SIMDs idle for that long.  Here a team of G
// lanes evaluates the 42 nodes of a dqagse step together (all of them at once
// for G = 64), lane pairs sum the two passes in QK21's order, and every lane
// of the team runs the same bookkeeping on lists in LDS.  The values and
// their order are those of the other kernels.
//
// TS::ids(): work ids, one team each; TS::team(id, &task): false where the id
// holds no integral.  overflow receives what TS::get takes.
// ---------------------------------------------------------------------------
template <int CAP>
struct QagsTeamLds {
  double v[42];
  typename QagsSmallStore<CAP>::Arrays lists;
};

template <int G, int CAP, class TS>
__global__ __launch_bounds__(kQagsBlock) void k_flux_qags_team(TS ts, double* __restrict__ flux,
                                                               int* __restrict__ ier_out,
                                                               unsigned long long* __restrict__ stats,
                                                               long long* __restrict__ overflow, int fast_cap)
{
  constexpr int kTeams = kQagsBlock / G;
  __shared__ QagsTeamLds<CAP> lds[kTeams];
  __shared__ unsigned blk_evals, blk_bad;
  if (threadIdx.x == 0) blk_evals = blk_bad = 0;
  __syncthreads();
  const int tl = threadIdx.x % G, lane0 = (threadIdx.x & 63) - tl;
  QagsTeamLds<CAP>& W = lds[threadIdx.x / G];
  const long long id = (long long)blockIdx.x * kTeams + threadIdx.x / G;
  Qags<QagsSmallStore<CAP>> q;
  q.s.a = &W.lists;
  q.s.lim = fast_cap < CAP ? fast_cap : CAP;
  FluxTask ft{};
  bool live = id < ts.ids() && ts.team(id, &ft);
  const double w2g2 = ft.k * ft.k / ft.g1 / ft.g1;
  if (live) q.start();
  while (live) {
    const int np = q.passes();
#pragma unroll 1
    for (int n = tl; n < 21 * np; n += G) {
      const int pass = n >= 21;
      double qa, qb;
      q.interval(pass, &qa, &qb);
      W.v[n] = flux_integrand<0>(ft.ff, ft.b, w2g2, qk21_abscissa(n - 21 * pass, 0.5 * (qa + qb), 0.5 * (qb - qa)));
    }
    wave_lds_sync();
    QK21Out o, o2;
    {
      const int pass = np == 2 ? tl & 1 : 0;
      double qa, qb;
      q.interval(pass, &qa, &qb);
      const QK21Out t = qk21_stored(W.v + 21 * pass, 1, qa, qb);
      o = QK21Out{__shfl(t.result, lane0), __shfl(t.abserr, lane0), __shfl(t.resabs, lane0), __shfl(t.resasc, lane0)};
      o2 = QK21Out{__shfl(t.result, lane0 + 1), __shfl(t.abserr, lane0 + 1), 0.0, __shfl(t.resasc, lane0 + 1)};
    }
    wave_lds_sync();
    const int st = q.consume(o, o2);
    wave_lds_sync();
    if (st == kQagsRunning) continue;
    live = false;
    if (tl) continue;
    if (st == kQagsDone) {
      const double Q = q.result / ft.A;
      flux[ft.out] = ft.factor * Q * Q / ft.k;
      const int status = q.status();
      if (ier_out) ier_out[ft.out] = status;
      atomicAdd(&blk_evals, (unsigned)q.neval());
      if (status != 0) {
        atomicAdd(&blk_bad, 1u);
        ts.failed(ft.slot);
      }
    } else {
      overflow[atomicAdd(&stats[2], 1ull)] = ts.overflow_id(id);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (blk_evals) atomicAdd(&stats[0], (unsigned long long)blk_evals);
    if (blk_bad) atomicAdd(&stats[1], (unsigned long long)blk_bad);
  }
}

// Tasks that outgrew the fast interval list (integrals that bisect more than
// the fast list holds: in practice the ones whose integrand turned NaN or whose
// roundoff tests fire, which run on to dozens or hundreds of intervals) are
// rerun from the start here, one wavefront per integral, with the reference's
// 1000-interval workspace in LDS.  Lanes 0..41 evaluate the 42 nodes of a
// step (both halves) at once; lane 0 sums each pass in QK21's order (the same
// qk21_stored as the fast kernel) and runs the dqagse state machine, so the
// serial part of a step is LDS work and one sum per pass.
constexpr int kQagsWaveBlocks = 1024;  // workgroups of the overflow kernel (36.5 KB LDS each)

template <class TS>
__global__ __launch_bounds__(64) void k_flux_qags_wave(TS ts, const long long* __restrict__ overflow,
                                                       unsigned long long* __restrict__ stats,
                                                       double* __restrict__ flux, int* __restrict__ ier_out)
{
  __shared__ QagsBigArrays ws;
  __shared__ double vals[2][21];
  __shared__ double iv[2][2];
  __shared__ int ctl[2];  // [0] passes of the step, [1] state after it
  const long n = (long)stats[2];
  const int lane = threadIdx.x;
  for (long i = blockIdx.x; i < n; i += gridDim.x) {
    FluxTask ft;
    ts.get(overflow[i], &ft);
    FluxFormIntegrand f;
    f.ff = ft.ff;
    f.b = ft.b;
    f.w2g2 = ft.k * ft.k / ft.g1 / ft.g1;
    Qags<QagsBigStore> q;
    q.s.a = &ws;
    if (lane == 0) q.start();
    int st = kQagsRunning;
    while (true) {
      if (lane == 0) {
        const int np = q.passes();
        ctl[0] = np;
        for (int k = 0; k < np; ++k) q.interval(k, &iv[k][0], &iv[k][1]);
      }
      __syncthreads();
      const int np = ctl[0];
      if (lane < 21 * np) {
        const int pass = lane >= 21, e = lane - 21 * pass;
        const double a = iv[pass][0], b = iv[pass][1];
        vals[pass][e] = f(qk21_abscissa(e, 0.5 * (a + b), 0.5 * (b - a)));
      }
      __syncthreads();
      if (lane == 0) {
        const QK21Out o = qk21_stored(vals[0], 1, iv[0][0], iv[0][1]);
        QK21Out o2{};
        if (np == 2) o2 = qk21_stored(vals[1], 1, iv[1][0], iv[1][1]);
        ctl[1] = q.consume(o, o2);
      }
      __syncthreads();
      st = ctl[1];
      if (st != kQagsRunning) break;
    }
    if (lane == 0) {
      const double Q = q.result / ft.A;
      flux[ft.out] = ft.factor * Q * Q / ft.k;
      const int status = st == kQagsDone ? q.status() : 99;
      if (ier_out) ier_out[ft.out] = status;
      atomicAdd(&stats[0], (unsigned long long)q.neval());
      if (status != 0) {
        atomicAdd(&stats[1], 1ull);
        ts.failed(ft.slot);
      }
    }
    __syncthreads();
  }
}

// What the contraction reads of one job (one context's grid).
struct LumiView {
  const double* pts;       // (M, Y, dm, dy) of the job's points
  const double* row_logd;  // the job's flux rows (k2 rows after the k1 rows)
  const double* flux;
  FluxParams fp;
  const double4* gaa;
  const double4* bk;
  const DevScalars* sc;
  int npts, mode, pol;
  double* L;
  double* Ls;
  double* Lp;
  // 0: one work item per point.  1 (symmetric grid, fp.mirror_ny = ny > 0):
  // bins (m, iy) and (m, ny - iy) have the same M, dm, dy and exchanged flux
  // rows, and the node sum is symmetric under b1 <-> b2, so one evaluation
  // fills both; work items are the bins iy <= ny / 2.
  int mirror_out;
  const unsigned char* need = nullptr;  // work items to run (null: all)
};

// Work items of a contraction launch.
__host__ __device__ inline int lumi_work_items(int npts, int mirror_ny, int mirror_out)
{
  return mirror_out ? npts / mirror_ny * (mirror_ny / 2 + 1) : npts;
}

// Work item q -> point p and its mirror bin pm (-1: none).
__device__ __forceinline__ void work_point(int q, int mirror_ny, int mirror_out, int* p, int* pm)
{
  if (!mirror_out) {
    *p = q;
    *pm = -1;
    return;
  }
  const int ny = mirror_ny, nc = ny / 2 + 1;
  const int im = q / nc, iy = q - im * nc;
  *p = im * ny + iy;
  *pm = iy > 0 && ny - iy != iy ? im * ny + (ny - iy) : -1;
}

__device__ __forceinline__ void lumi_work_point(const LumiView& v, int q, int* p, int* pm)
{
  work_point(q, v.fp.mirror_ny, v.mirror_out, p, pm);
}

// Exclusive prefix sums of the row counts per bucket (in place), one block per
// job: off[job][bucket] counts from where the job's rows start in perm; their
// number in nsorted[job].  10 buckets per thread, wave scans.
template <class RS, class N>
__global__ __launch_bounds__(1024) void k_row_offsets(RS rs, int* __restrict__ off, N* __restrict__ nsorted)
{
  constexpr int kPer = kRowBuckets / 1024;
  __shared__ int wsum[16];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  off += (size_t)blockIdx.x * kRowBuckets;
  long long r0, pos0;
  rs.span(blockIdx.x, &r0, &pos0);
  int v[kPer], s = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    v[i] = off[t * kPer + i];
    s += v[i];
  }
  int inc = s;
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(inc, o);
    if (lane >= o) inc += u;
  }
  if (lane == 63) wsum[wv] = inc;
  __syncthreads();
  int base = (int)pos0 + inc - s;
  for (int w = 0; w < wv; ++w) base += wsum[w];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    off[t * kPer + i] = base;
    base += v[i];
  }
  if (t == 1023) nsorted[blockIdx.x] = (N)(base - (int)pos0);
}

// Orders the rows of each bucket by (k, row): the order they were dropped in
// varies from run to run, and with it the groups that expand J1 together and
// the last bits of what they compute.  off: the buckets' ends; spare: as long as
// perm.  A workgroup takes four buckets, one per wavefront (50 rows on the 1001 x
// 121 grid); a bucket of more rows (points close together) takes the workgroup,
// up to kOrderMax of them ordered by their ranks, more by row alone: those are
// marked in a bitmap of kOrderWindow rows at a time and read off it.  8,192 rows
// within 0.4 % of two energies 0.13 ms, 262,144 and 2,000,000 rows of two energies
// 0.43 and 9.0 (0.57, 2.3 and 25 when one wavefront looked through all rows for
// those of its bucket), of calls of 1.1, 17 and 133 ms.
constexpr int kOrderWave = 128, kOrderMax = 1024;
constexpr int kOrderWindow = 1 << 18;

template <class RS>
__global__ __launch_bounds__(256) void k_row_order(RS rs, const int* __restrict__ off, long long nbuckets,
                                                   int* __restrict__ spare)
{
  constexpr int kWords = kOrderWindow / 32;  // of the bitmap
  __shared__ union {
    struct {
      long long k[kOrderMax];
      int r[kOrderMax];
    } one;
    struct {
      long long k[4][kOrderWave];
      int r[4][kOrderWave];
    } four;
    unsigned bits[kWords + kWords / 32];  // a word of padding after each 32
  } S;
  __shared__ int wsum[4];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  // rows of bucket i and where they start in perm
  long long r0 = 0, nrows = 0, start = 0;
  auto bucket = [&](long long i) {
    if (i >= nbuckets) return 0;
    const int job = (int)(i / kRowBuckets);
    nrows = rs.span(job, &r0, &start);
    if (i > (long long)job * kRowBuckets) start = off[i - 1];
    return (int)(off[i] - start);
  };
  // the rank of each row among the n in k, r, by every step'th thread
  auto ranks = [&](const long long* k, const int* r, int n, int first, int step) {
    for (int e = first; e < n; e += step) {
      int rank = 0;
#pragma unroll 8
      for (int m = 0; m < n; ++m) rank += (k[m] < k[e]) | ((k[m] == k[e]) & (r[m] < r[e]));
      rs.perm[start + rank] = r[e];
    }
  };
  const long long i0 = (long long)blockIdx.x * 4;
  int n = bucket(i0 + wv);
  if (n > 1 && n <= kOrderWave) {
    for (int e = lane; e < n; e += 64) {
      const int r = rs.perm[start + e];
      S.four.r[wv][e] = r;
      S.four.k[wv][e] = __double_as_longlong(rs.row_k[r]);
    }
    wave_lds_sync();
    ranks(S.four.k[wv], S.four.r[wv], n, lane, 64);
  }
  for (int q = 0; q < 4; ++q) {
    n = bucket(i0 + q);
    if (n <= kOrderWave) continue;
    __syncthreads();
    if (n <= kOrderMax) {
      for (int e = t; e < n; e += 256) {
        const int r = rs.perm[start + e];
        S.one.r[e] = r;
        S.one.k[e] = __double_as_longlong(rs.row_k[r]);
      }
      __syncthreads();
      ranks(S.one.k, S.one.r, n, t, 256);
      continue;
    }
    for (int e = t; e < n; e += 256) spare[start + e] = rs.perm[start + e];
    auto bits = [&](int word) -> unsigned& { return S.bits[word + (word >> 5)]; };
    long long out = start;
    for (long long w0 = r0; w0 < r0 + nrows && out < start + n; w0 += kOrderWindow) {
      const long long left = r0 + nrows - w0;
      const int rows = left < kOrderWindow ? (int)left : kOrderWindow;
      const int own = ((rows + 31) / 32 + 255) / 256, first = t * own;  // the thread's words
      for (int j = 0; j < own; ++j) bits(first + j) = 0;
      __syncthreads();
      for (int e = t; e < n; e += 256) {
        const long long x = spare[start + e] - w0;
        if (x >= 0 && x < rows) atomicOr(&bits((int)(x >> 5)), 1u << (x & 31));
      }
      __syncthreads();
      int c = 0;
      for (int j = 0; j < own; ++j) c += __popc(bits(first + j));
      int inc = c;
      for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(inc, o);
        if (lane >= o) inc += u;
      }
      if (lane == 63) wsum[wv] = inc;
      __syncthreads();
      long long at = out + inc - c;
      for (int w = 0; w < wv; ++w) at += wsum[w];
      for (int j = 0; j < own; ++j)
        for (unsigned m = bits(first + j); m; m &= m - 1) rs.perm[at++] = (int)(w0 + 32 * (first + j) + __ffs(m) - 1);
      out += wsum[0] + wsum[1] + wsum[2] + wsum[3];
      __syncthreads();  // wsum is read
    }
  }
}

// Flux rows of a launch (of a job, in a batch) from which on neighbouring rows
// lie close enough in k to share what k_flux_qags_table shares.  QAGS of Pb-Pb
// points and grids, k_flux_qags_rows against k_flux_qags_table: 4,096 rows 0.69
// against 0.89 ms, 6,000 0.86, 1.04; 8,192 1.03, 1.01; 11,000 1.24, 1.10;
// 16,384 1.52, 1.30.  What decides it is the row count alone, so a job of a
// batch takes the route of its own context.
constexpr long long kQagsShareRows = 8192;

// The factor table H of a launch sequence over at most `groups` groups of rows:
// the groups it holds, kRowsChunk at most, fewer where memory is short, 0 (and
// no table) where kRowsChunkMin do not fit.  The end of a launch leaves the chip
// half idle for 0.3 ms: whole grids of 1001 x 121, 2001 x 241 bins and a 16-job
// batch take 6.1, 21.8 and 64.4 ms with 4,096 groups, 6.1, 22.5 and 65.6 with
// 2,048, 6.4, 23.6 and 68.4 with 1,024.
inline long long rows_groups(long long rows) { return (rows + 63) / 64; }
constexpr int kRowsChunkMin = (int)(kQagsShareRows / 64);  // 34 MB

inline int alloc_factors(double** H, long long groups)
{
  *H = nullptr;
  for (int n = (int)std::min<long long>(groups, kRowsChunk); n > 0;) {
    if (hipMalloc(H, sizeof(double) * (size_t)n * kHGroupElems) == hipSuccess) return n;
    (void)hipGetLastError();  // k_flux_qags_rows needs no table
    *H = nullptr;
    n = n > kRowsChunkMin ? std::max(n / 2, kRowsChunkMin) : 0;
  }
  return 0;
}

// Work cursors of that sequence, whatever the table holds, and of one launch of
// k_flux_qags_rows after it.
inline size_t rows_cursors(long long groups)
{
  return (size_t)((groups + kRowsChunkMin - 1) / kRowsChunkMin + 1) * kXcds;
}

// upc_flux_rows.hip
template <class RS>
void launch_qags_rows_direct(const RS& rs, unsigned long long* cursor, double* flux, unsigned long long* stats,
                             long long* overflow, int cap, int blocks, hipStream_t s);

// Launches over at most `groups` groups of rows: of k_flux_qags_table, `chunk` of
// them at a time (what H holds), or with chunk 0 of k_flux_qags_rows.  cursors:
// cleared, kXcds per launch; per_cu: workgroups per CU, at most 3.
template <class RS>
inline void launch_qags_rows(int chunk, const RS& rs, long long groups, double* H, unsigned long long* cursors,
                             double* flux, unsigned long long* stats, long long* overflow, int cap, int ncu,
                             int per_cu, hipStream_t s)
{
  if (groups <= 0) return;
  if (!chunk) return launch_qags_rows_direct(rs, cursors, flux, stats, overflow, cap, ncu * per_cu, s);
  const long long launches = (groups + chunk - 1) / chunk;
  chunk = (int)((groups + launches - 1) / launches);  // all of one size
  for (long long g0 = 0; g0 < groups; g0 += chunk, cursors += kXcds) {
    const long long n = groups - g0 < chunk ? groups - g0 : chunk;
    hipLaunchKernelGGL(k_flux_h<RS>, dim3((unsigned)(n * kHSlots)), dim3(256), 0, s, rs, g0, H);
    hipLaunchKernelGGL((k_flux_qags_table<kQagsCap, RS>), dim3(ncu * std::min(per_cu, kQagsTableBlocksPerCu)),
                       dim3(kQagsBlock), 0, s, rs, g0, chunk, H, cursors, flux, stats, overflow, cap);
  }
}

inline FluxParams flux_params(const upc_ctx* c, int mirror_ny = 0)
{
  FluxParams fp;
  fp.mirror_ny = mirror_ny;
  fp.R = c->cfg.R;
  fp.bmin = c->cfg.flux_point ? c->cfg.R : 0.05 * c->cfg.R;
  fp.g1 = c->g1;
  fp.g2 = c->g2;
  fp.factor = c->factor;
  fp.twoR = 2. * c->cfg.R;
  fp.A = c->cfg.A;
  fp.isPoint = c->cfg.flux_point;
  return fp;
}

// Builds the flux rows of the points in the work buffer (d_pts == nullptr)
// or of the npts (M, Y) pairs at d_pts ([M..., Y...]): point-charge nodes
// directly, form-factor nodes by the QAGS task kernels.  *fp receives the
// row parameters (mirror_ny set when the grid's Y range is symmetric).
int prepare_flux(upc_ctx* c, const double* d_pts, int npts, FluxParams* fp, hipStream_t s);
// The FP64 contraction of a view (only its work items with v.need[q] != 0
// when v.need is set) on stream s.
int launch_lumi_fp64(const LumiView& v, hipStream_t s);
// Copies the QAGS counters of the last prepare_flux into the context.
int read_flux_stats(upc_ctx* c, hipStream_t s);

}  // namespace upc
