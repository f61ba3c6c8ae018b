// FP64 two-photon contraction (k_lumi_fp64), of one view and of a batch's jobs.
// A unit of its own: the options the QAGS kernels' units are compiled with
// (build.py) cost this kernel 4 %.
#include "upc_internal.h"
#include "upc_batch_job.h"

namespace upc {

// ---------------------------------------------------------------------------
// FP64 luminosity: one wavefront (WPP = 1), or a workgroup of them, per (M, Y)
// point.
//
// For a pair of nodes (b1_i, b2_j) the phi sum K_ij = sum_k w_k P(b) G(b),
// b^2 = b1^2 + b2^2 +- 2 b1 b2 cos(phi_k).  Where every node has b >= 20 fm
// the reference evaluates P at the 20 fm clamp and G = 1, so K_ij is the
// constant S0.  For fixed i the pairs with some b < 20 form one contiguous j
// range (the smallest b^2 is always the extreme-cos node), so
//   L = 2 pi^2 M [ S0 sum_i W1_i sum_{j outside i's band} W2_j + sum_{band} W1_i W2_j K_ij ]
// with W = N(b, k) b (b_h - b_l), the sums outside from prefix and suffix sums
// of W2.  No term is negative, so nothing cancels (the band's difference from
// S0 (sum W1)(sum W2) leaves 1e-10 of L where most of the flux is below the
// hadronic knee).  The band pairs are spread evenly over the 64 lanes.
//
// Bound: VALU issue (90 to 98 % busy); a third of the lanes' cycles go to nodes
// that need no spline.  1001 x 121 Pb-Pb: 0.85 ms
// (mode 1), 1.29 (mode 2), 1.09 (mode 4, polarised); 1.29, 1.62 and 1.45 with
// two exponentials per node, scaled square roots and interval clamps of 64 bits
// at 96 VGPRs (now 74).
// The pairs of a point are cut into kLumiParts runs that are summed apart and
// then in order, so one wavefront, four and eight give the same bits.
// ---------------------------------------------------------------------------
constexpr int kLumiParts = 8;

// cos(pi x_k) and sin^2(pi x_k) of the 5 phi nodes (10-point Gauss-Legendre).
__device__ constexpr double kPhiCos[5] = {0.8926064270787061, 0.20772097768336903, -0.5342597336817245,
                                          -0.9114851796955159, -0.996641926035247};
__device__ constexpr double kPhiSin[5] = {0.45083674022620046, 0.9781881186306984, 0.845320375340813,
                                          0.41133291528326904, 0.08188327832197047};

// sqrt(x) < 20 in double precision: x = 400 - 2^-44 still rounds to 20.
constexpr double kB2Edge = 400.0 - 0x1p-44;

// sqrt of a normal positive x: Goldschmidt steps from the hardware estimate and
// one correction by the residual (x away from the exponent's ends needs no
// scaling: 8 operations against 16).
__device__ __forceinline__ double sqrt_mid(double x)
{
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  return fma(fma(-g, g, x), h, g);
}

// The phi sum of one node pair, sum_k w_k P(min(b, 20)) G(b), G = 1 for b >=
// 20 (br = P(20), or 1 without breakup); polarised: cos^2 and sin^2 weighted
// sums.  tb = 2 b1 b2, ss = b1^2 + b2^2.
//
// Below the hadronic knee (b < ~11 fm for Pb-Pb) the G_AA spline holds only
// the decaying ringing of the natural spline, |G| < 1e-30.  Below bskip
// (x < bskip2) |G| < gskip = p20 2^-70 holds for every b, and P G is taken
// as 0 without sqrt, G or P.
// Above bskip, modes 2-4 still skip the breakup spline wherever the G just
// evaluated is below gskip (mode 1 has P = 1 and reads no breakup spline).
//
// Where b lies within rounding of a knot the estimate may name the neighbouring
// interval; the splines are C2, so that cubic agrees there to a few ulp.
template <bool POL>
__device__ __forceinline__ void node_k(double tb, double ss, bool breakup, double br, double gskip, double bskip2,
                                       const double4* gaa, const double4* __restrict__ bk, double* ks, double* kp)
{
  const double db = 20. / (kNB - 1);
  double s = 0.0, p = 0.0;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    const double c = kPhiCos[k], w = kGLw5[k];
    const double x = fma(tb, POL ? -c : c, ss);
    double v = br;
    if (x < kB2Edge) {
      v = 0.0;
      if (x >= bskip2) {
        const double b = sqrt_mid(x);
        const int i = min((int)(b * (1.0 / db)), kNB - 2);
        const double4 g = gaa[i];
        const double d = fma(-(double)i, db, b);
        v = g.x + d * (g.y + d * (g.z + d * g.w));
        if (breakup) {
          const bool on = fabs(v) >= gskip;
          if (on) {
            const double e = b - kBkMin;
            const int n = min(max((int)(e * (1.0 / kDBk)), 0), kNBkUsed - 2);
            const double4 q = *(const double4*)((const char*)bk + (unsigned)n * (unsigned)sizeof(double4));
            const double f = fma(-(double)n, kDBk, e);
            v *= q.x + f * (q.y + f * (q.z + f * q.w));
          } else {
            v = 0.0;
          }
        }
      }
    }
    s = fma(v, POL ? w * c * c : w, s);
    if (POL) p = fma(v, w * kPhiSin[k] * kPhiSin[k], p);
  }
  *ks = s;
  *kp = p;
}

// Job resolvers: the job and first point of a block of `points` points.
struct SingleLumi {
  LumiView v;
  __device__ void get(int blk, int points, LumiView* out, int* p0) const
  {
    *out = v;
    *p0 = blk * points;
  }
};

// Contraction job resolver: blk0[j] = first block of job j for this wave count.
struct BatchLumi {
  const BatchJob* __restrict__ jobs;
  const int* __restrict__ blk0;
  int njobs;
  __device__ void get(int blk, int waves, LumiView* out, int* p0) const
  {
    const int j = find_job(blk0, njobs, blk);
    *out = jobs[j].v;
    *p0 = (blk - blk0[j]) * waves;
  }
};

// LDS of a point; the exponentials of the rows' nodes (first row in e1, second
// in sp2) make room for the suffix and prefix sums, the former for the pair list.
struct LumiPoint {
  double sb1[kNB1], sb2[kNB2];
  double sw1[kNB1], sw2[kNB2];
  double sp2[kNB2 + 1];  // prefix sums of sw2
  union {
    double e1[kNB1 + 1];
    double ss2[kNB2 + 1];  // suffix sums of sw2
    struct {
      int spre[kNB1 + 1], sjlo[kNB1];
    };
  };
};

template <int WAVES, int WPP>
struct LumiSmem {
  double4 gaa[kNB];
  LumiPoint pt[WAVES / WPP];
  double acc[WPP > 1 ? 2 * kLumiParts * 64 : 1];  // the parts' sums
};

template <bool POL, int WAVES, int WPP>
__device__ __forceinline__ void lumi_fp64_body(const LumiView& v, int p0, LumiSmem<WAVES, WPP>& sm)
{
  static_assert(WPP == 1 || (WPP == WAVES && kLumiParts % WPP == 0), "a point takes one wavefront or the workgroup");
  constexpr int kThreads = 64 * WPP;
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int sub = WPP > 1 ? wv : 0, tid = WPP > 1 ? threadIdx.x : lane;  // within the point's threads
  LumiPoint& pt = sm.pt[WPP > 1 ? 0 : wv];
  auto sync = [] {
    if (WPP > 1) __syncthreads();
    else wave_sync_lds();
  };
  const int q = p0 + (WPP > 1 ? 0 : wv);
  const bool live = q < lumi_work_items(v.npts, v.fp.mirror_ny, v.mirror_out) && (!v.need || v.need[q]);
  // a masked launch (block-uniform v.need): blocks with no needed item end here
  if (v.need && !__syncthreads_or(live)) return;
  for (int i = threadIdx.x; i < kNB - 1; i += blockDim.x) sm.gaa[i] = v.gaa[i];
  __syncthreads();
  if (!live) return;
  int p, pm;
  lumi_work_point(v, q, &p, &pm);
  const FluxParams& fp = v.fp;
  const double p20 = v.sc->p20;
  const double M = v.pts[4 * p], dm = v.pts[4 * p + 2], dy = v.pts[4 * p + 3];
  const int r2 = k2_row(p, v.npts, fp.mirror_ny);
  const double logd1 = v.row_logd[p], logd2 = v.row_logd[r2];
  LogGrid lg2;
  lg2.init(fp.bmin, logd2);
  // both rows' nodes (row_node), each exponential once
  for (int t = tid; t < 2 * (kNB1 + 1); t += kThreads) {
    const bool second = t > kNB1;
    const int j = second ? t - (kNB1 + 1) : t;
    const double e = exp(j * (second ? logd2 : logd1));
    if (second) pt.sp2[j] = e;
    else pt.e1[j] = e;
  }
  sync();
  for (int t = tid; t < 2 * kNB1; t += kThreads) {
    const bool second = t >= kNB1;
    const int j = second ? t - kNB1 : t;
    const double el = second ? pt.sp2[j] : pt.e1[j], eh = second ? pt.sp2[j + 1] : pt.e1[j + 1];
    const double f = v.flux[(long)(second ? r2 : p) * kNB1 + j];
    const double bl = fp.bmin * el, b = fma(fp.bmin, eh, bl) / 2.;
    const double w = f * b * fma(fp.bmin, eh, -bl);
    if (second) {
      pt.sb2[j] = b;
      pt.sw2[j] = w;
    } else {
      pt.sb1[j] = b;
      pt.sw1[j] = w;
    }
  }
  sync();
  // the extreme-cos node has the smallest b for every pair, cmax the largest
  constexpr double cext = POL ? -kPhiCos[0] : kPhiCos[4];
  constexpr double cmax = POL ? -kPhiCos[4] : kPhiCos[0];
  // prefix sums sp2[j] = sum_{j' < j} sw2[j'], suffix sums ss2[j] = sum_{j' >= j}
  // (each from its own end: no differences)
  if (sub < 2) {
    auto scan = [&](bool back) {
      const int last = kNB2 - 1 - lane;  // the suffix scan runs from the end
      double a0 = pt.sw2[back ? last : lane];
      double a1 = lane + 64 < kNB2 ? pt.sw2[back ? last - 64 : lane + 64] : 0.0;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const double u0 = __shfl_up(a0, o), u1 = __shfl_up(a1, o);
        if (lane >= o) {
          a0 += u0;
          a1 += u1;
        }
      }
      a1 += __shfl(a0, 63);
      double* out = back ? pt.ss2 : pt.sp2;
      out[back ? last : lane + 1] = a0;
      if (lane + 64 < kNB2) out[back ? last - 64 : lane + 65] = a1;
      if (lane == 0) out[back ? kNB2 : 0] = 0.0;
    };
    if (WPP == 1 || sub == 0) scan(false);
    if (WPP == 1 || sub == 1) scan(true);
  }
  const double bskip = v.sc->bskip, bskip2 = bskip * bskip;
  // Pairs whose largest node is below bskip have P G = 0 at every node and add
  // nothing: the run j < ja (b^2 at cmax > 0 grows with b2).  They are in the
  // band (b^2 < bskip^2 <= 400 at every node), which therefore starts at j = 0;
  // the walk takes the band from ja on.
  double out[2] = {0.0, 0.0};  // sums of sw2 outside the bands of rows lane and lane + 64 (WPP > 1: as below)
  sync();
  // Band of row i: the j with b^2 < 400 at the extreme cosine.  b^2 is convex
  // in b2 (smallest at b2 = -b1 cext), so the band is the run of j around
  // that vertex.  The vertex and both ends (roots b2 = vtx -+ sqrt(400 -
  // b1^2 (1 - cext^2))) are guessed on the log grid of b2 and stepped to
  // exactness with the same comparisons a bisection would make.
  int jlo[2] = {0, 0}, cnt[2] = {0, 0};  // of rows lane and lane + 64 (WPP > 1: of wavefront 0, of wavefront 1)
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int i = lane + 64 * h;
    if ((WPP == 1 || sub == h) && i < kNB1) {
      const double b1 = pt.sb1[i];
      const double* b2s = pt.sb2;
      auto inb = [&](int j) { return node_b2(b1, b2s[j], cext) < 400.0; };
      const double vtx = -b1 * cext;
      int lo = lg2.first_ge(vtx, kNB2);  // first j with b2_j >= vtx
      while (lo > 0 && b2s[lo - 1] >= vtx) --lo;
      while (lo < kNB2 && b2s[lo] < vtx) ++lo;
      int jc = -1;
      if (lo < kNB2 && inb(lo)) jc = lo;
      if (lo > 0 && inb(lo - 1)) jc = lo - 1;
      out[h] = pt.sp2[kNB2];
      if (jc >= 0) {
        const double d = 400.0 - b1 * b1 * (1.0 - cext * cext), sd = sqrt(d > 0.0 ? d : 0.0);
        int a = lg2.first_ge(vtx - sd, kNB2);  // first j in band: outside before it, inside from it to jc
        a = a > jc ? jc : a;
        while (a > 0 && inb(a - 1)) --a;
        while (a < jc && !inb(a)) ++a;
        jlo[h] = a;
        out[h] = pt.sp2[a];
        a = lg2.first_ge(vtx + sd, kNB2) - 1;  // last j in band
        a = a < jc ? jc : (a > kNB2 - 1 ? kNB2 - 1 : a);
        while (a < kNB2 - 1 && inb(a + 1)) ++a;
        while (a > jc && !inb(a)) --a;
        out[h] += pt.ss2[a + 1];
        // first j with b^2 >= bskip^2 at cmax (b^2 grows with b2 there)
        auto low = [&](int j) { return node_b2(b1, b2s[j], cmax) < bskip2; };
        const double da = bskip2 - b1 * b1 * (1.0 - cmax * cmax);
        int ja = da > 0.0 ? lg2.first_ge(-b1 * cmax + sqrt(da), kNB2) : 0;
        while (ja > 0 && !low(ja - 1)) --ja;
        while (ja < kNB2 && low(ja)) ++ja;
        if (ja > 0) jlo[h] = ja;
        cnt[h] = a >= jlo[h] ? a - jlo[h] + 1 : 0;
      }
    }
  }
  sync();  // the suffix sums have been read
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int i = lane + 64 * h;
    if ((WPP == 1 || sub == h) && i < kNB1) {
      pt.sjlo[i] = jlo[h];
      pt.spre[i + 1] = cnt[h];
    }
  }
  if (WPP > 1 && sub == 1) sm.acc[lane] = out[1];
  sync();
  double far = 0.0;  // sum over rows of sw1[i] times its outside sum
  if (sub == 0) {
    if (WPP > 1) out[1] = sm.acc[lane];
    far = fma(lane + 64 < kNB1 ? pt.sw1[lane + 64] : 0.0, out[1], pt.sw1[lane] * out[0]);
  }
  // prefix sums of the row counts
  if (sub == 0) {
    int c0 = pt.spre[lane + 1], c1 = lane + 64 < kNB1 ? pt.spre[lane + 65] : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u0 = __shfl_up(c0, o), u1 = __shfl_up(c1, o);
      if (lane >= o) {
        c0 += u0;
        c1 += u1;
      }
    }
    const int half = __shfl(c0, 63);
    pt.spre[lane + 1] = c0;
    if (lane + 64 < kNB1) pt.spre[lane + 65] = half + c1;
    if (lane == 0) pt.spre[0] = 0;
  }
  sync();
  const bool breakup = v.mode != 1;
  const double br = breakup ? p20 : 1.0;
  const int T = pt.spre[kNB1];
  const double gskip = p20 * 0x1p-70;
  double accs = 0, accp = 0;
  const int run = ((T + 63) / 64 + kLumiParts - 1) / kLumiParts * 64;  // pairs of a part
  int i = 0;  // row of pair t: pre[i] <= t < pre[i + 1]; t only grows
  if (WPP > 1 && sub * run + lane < T)
    for (int s = 64; s > 0; s >>= 1)
      if (i + s < kNB1 && pt.spre[i + s] <= sub * run + lane) i += s;
  for (int part = sub; part < kLumiParts; part += WPP) {
    const int end = min((part + 1) * run, T);
    double as = 0, ap = 0;
    for (int t = part * run + lane; t < end; t += 64) {
      while (pt.spre[i + 1] <= t) ++i;
      const int j = pt.sjlo[i] + (t - pt.spre[i]);
      const double b1 = pt.sb1[i], b2 = pt.sb2[j];
      double ks, kp;
      node_k<POL>(2.0 * b1 * b2, fma(b1, b1, b2 * b2), breakup, br, gskip, bskip2, sm.gaa, v.bk, &ks, &kp);
      const double ww = pt.sw1[i] * pt.sw2[j];
      as += ww * ks;
      if (POL) ap += ww * kp;
    }
    if (WPP > 1) {
      sm.acc[part * 64 + lane] = as;
      if (POL) sm.acc[(kLumiParts + part) * 64 + lane] = ap;
    } else {
      accs += as;
      accp += ap;
    }
  }
  if (WPP > 1) {
    sync();
    if (sub > 0) return;
    for (int c = 0; c < kLumiParts; ++c) {
      accs += sm.acc[c * 64 + lane];
      if (POL) accp += sm.acc[(kLumiParts + c) * 64 + lane];
    }
  }
  // S0: the phi sum when every node is at or beyond 20 fm
  double s0s = 0, s0p = 0;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    const double c = kPhiCos[k], w = kGLw5[k];
    s0s = fma(br, POL ? w * c * c : w, s0s);
    if (POL) s0p = fma(br, w * kPhiSin[k] * kPhiSin[k], s0p);
  }
  for (int o = 32; o > 0; o >>= 1) {
    accs += __shfl_down(accs, o);
    if (POL) accp += __shfl_down(accp, o);
    far += __shfl_down(far, o);
  }
  if (lane == 0) {
    const double pre = 2 * kPi * kPi * M;
    const double tot_s = s0s * far + accs;
    if (POL) {
      const double tot_p = s0p * far + accp;
      const double ls = pre * tot_s * dm * dy, lp = pre * tot_p * dm * dy;
      v.Ls[p] = ls;
      v.Lp[p] = lp;
      if (pm >= 0) {
        v.Ls[pm] = ls;
        v.Lp[pm] = lp;
      }
    } else {
      const double l = pre * tot_s * dm * dy;
      v.L[p] = l;
      if (pm >= 0) v.L[pm] = l;
    }
  }
}

// WAVES / WPP points per block; the resolver maps the block to its job (all
// threads of a block take the same branch, so the barriers are uniform).
// 74 to 76 VGPRs without spills with one wavefront per point (52 to 56 with a
// workgroup per point), alike for budgets of 4 to 6 waves per SIMD; LDS admits 5
// of four-wave workgroups.
constexpr int kLumiWavesPerEu = 5;

template <int WAVES, int WPP, class JR>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(kLumiWavesPerEu))) void k_lumi_fp64(
    JR jr)
{
  __shared__ LumiSmem<WAVES, WPP> sm;
  LumiView v;
  int p0;
  jr.get(blockIdx.x, WAVES / WPP, &v, &p0);
  if (v.pol) lumi_fp64_body<true, WAVES, WPP>(v, p0, sm);
  else lumi_fp64_body<false, WAVES, WPP>(v, p0, sm);
}

// Work items of a launch up to which each takes a workgroup of 8, and of 4
// wavefronts: a point's pair list is one serial walk of up to 225 steps, and few
// points wait for the longest; with many, the set-up that the other wavefronts
// wait for costs more.  Pb-Pb points (modes 1 / 2 / 4 polarised), us:
//                     1 wavefront        4                 8
//        33 points    83 /   98 /   88   32 /  37 /  32    20 /  24 /  23
//     2,048          109 /  185 /  153   62 /  92 /  81    56 /  82 /  76
//     4,096          135 /  206 /  168   98 / 138 / 116   100 / 138 / 129
//     9,331 (grid)   181 /  265 /  212  171 / 243 / 204   195 / 289 / 272
//    32,768          549 /  844 /  700  542 / 768 / 639   645 / 908 / 847
//    61,061 (grid)   861 / 1381 / 1139  975 /1444 /1264  1156 /1735 /1612
constexpr int kLumiTeam8 = 3072, kLumiTeam4 = 32768;

template <int WAVES, int WPP>
static void launch_lumi(const LumiView& v, int nwork, hipStream_t s)
{
  constexpr int kPoints = WAVES / WPP;
  hipLaunchKernelGGL((k_lumi_fp64<WAVES, WPP, SingleLumi>), dim3((nwork + kPoints - 1) / kPoints), dim3(64 * WAVES), 0,
                     s, SingleLumi{v});
}

int launch_lumi_fp64(const LumiView& v, hipStream_t s)
{
  const int nwork = lumi_work_items(v.npts, v.fp.mirror_ny, v.mirror_out);
  if (nwork <= 0) return 0;
  if (nwork <= kLumiTeam8) launch_lumi<8, 8>(v, nwork, s);
  else if (nwork <= kLumiTeam4) launch_lumi<4, 4>(v, nwork, s);
  else launch_lumi<4, 1>(v, nwork, s);
  UPC_HIP(hipGetLastError());
  return 0;
}

int launch_lumi_batch(const BatchJob* jobs, const int* blk0, int njobs, int waves, int blocks, hipStream_t s)
{
  const BatchLumi jr{jobs, blk0, njobs};
  const dim3 grid(blocks), block(64 * waves);
  if (waves == 2) hipLaunchKernelGGL((k_lumi_fp64<2, 1, BatchLumi>), grid, block, 0, s, jr);
  else if (waves == 4) hipLaunchKernelGGL((k_lumi_fp64<4, 1, BatchLumi>), grid, block, 0, s, jr);
  else hipLaunchKernelGGL((k_lumi_fp64<8, 1, BatchLumi>), grid, block, 0, s, jr);
  UPC_HIP(hipGetLastError());
  return 0;
}

}  // namespace upc
