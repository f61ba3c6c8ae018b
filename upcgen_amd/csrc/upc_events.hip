// Event generation for the dilepton processes on the GPU:
//   UpcGenerator::generateEvent      src/UpcGenerator.cpp:715-790
//   UpcCrossSection::getPairMomentum src/UpcCrossSection.cpp:1053-1074
//   UpcCrossSection::getPhotonPt     src/UpcCrossSection.cpp:1021-1051
//   UpcGenerator::pairProduction     src/UpcGenerator.cpp:388-423
//   UpcGenerator::checkKinCuts       src/UpcGenerator.cpp:563-587
//
// getPhotonPt draws the photon transverse momentum from a 5000-bin histogram
// over (0, 6 hc / R] with contents F(pt^2 + E^2/g^2)^2 pt^3 / (4 pi^2 (pt^2 +
// E^2/g^2)^2), rebuilt per MeV of photon energy E.  The energy enters only
// through eps = E^2/g^2, so the histograms are tabulated once per context on
// a log grid of eps and interpolated linearly between neighbours; the draw
// inside the chosen bin is uniform, as TH1::GetRandom does.
#include "upc_internal.h"
#include "upc_pdf.h"
#include "upc_philox.h"

namespace upc {

constexpr int kPtBins = 5000;
constexpr int kPtEps = 2048;          // eps grid points
constexpr double kPtEpsLo = -13.0;    // log10 eps range; below it the shape no longer changes
constexpr double kPtEpsHi = 0.4;      // 10^0.4 ~ 2.5 > Q2max: the form factor table ends at Q2 = 2

constexpr int kPtGuideBits = 11;
constexpr int kPtCells = (1 << kPtGuideBits) + 1;

// A draw reads a few neighbouring bins of two neighbouring rows, so the rows lie
// in pairs, 8 bins of each to a 128-byte line; their guides likewise.
constexpr int kPtLines = (kPtBins + 8) / 8;  // lines of a pair of rows

__device__ __forceinline__ size_t pt_row(int e) { return (size_t)(e >> 1) * (kPtLines * 16) + (e & 1) * 8; }
__device__ __forceinline__ int pt_bin(int k) { return (k >> 3) * 16 + (k & 7); }
__device__ __forceinline__ size_t pt_guide(int e) { return (size_t)(e >> 1) * (kPtCells * 2) + (e & 1); }

struct PtTables {
  double* cdf = nullptr;  // [kPtEps] rows of kPtBins + 1 (pt_row, pt_bin)
  unsigned short* guide = nullptr;  // their guides (upc_pdf.h): the bin of r = cell / 2^kPtGuideBits (pt_guide)
  double gtot = 0;
  double ptmax = 0;
};

__device__ __forceinline__ double ff_clamped(const double4* __restrict__ ff, double q2)
{
  // beyond the table the reference's spline raises GSL_EDOM; here it is clamped
  const double v = q2 < kQ2min ? kQ2min : (q2 > kQ2max - kDQ2 ? kQ2max - kDQ2 : q2);
  return spline_eval(ff, kQ2min, kDQ2, 1.0 / kDQ2, kNQ2, v);
}

// One block per eps value: bin contents, then the normalised cumulative sum,
// and the guide to it.
__global__ __launch_bounds__(256) void k_pt_tables(const double4* __restrict__ ff, double ptmax,
                                                   double* __restrict__ cdf, unsigned short* __restrict__ guide)
{
  __shared__ double row[kPtBins + 1];
  __shared__ double part[256];
  const int e = blockIdx.x;
  const double eps = pow(10.0, kPtEpsLo + (kPtEpsHi - kPtEpsLo) * e / (kPtEps - 1));
  constexpr double pi2x4 = 4 * kPi * kPi;
  const int t = threadIdx.x;
  const int per = (kPtBins + 255) / 256;
  const int s = t * per, en = min(kPtBins, s + per);
  double acc = 0;
  for (int b = s; b < en; ++b) {
    const double pt = ptmax / kPtBins * (b + 1);  // upper bin edge, as the reference fills bin b+1
    const double arg = pt * pt + eps;
    const double f = ff_clamped(ff, arg);
    const double prob = (f * f) * pt * pt * pt / (pi2x4 * arg * arg);
    row[b + 1] = prob;
    acc += prob;
  }
  part[t] = acc;
  __syncthreads();
  for (int d = 1; d < 256; d <<= 1) {
    const double v = t >= d ? part[t - d] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  const double total = part[255];
  double base = t ? part[t - 1] : 0;
  for (int b = s; b < en; ++b) {
    base += row[b + 1];
    row[b + 1] = base / total;
  }
  if (t == 0) row[0] = 0;
  __syncthreads();
  for (int b = t; b <= kPtBins; b += 256) cdf[pt_row(e) + pt_bin(b)] = row[b];
  for (int g = t; g < kPtCells; g += 256)
    guide[pt_guide(e) + 2 * g] = (unsigned short)pdf_search(row, 0, kPtBins, (double)g / (kPtCells - 1));
}

// Draws r[0 .. N) of photons of energies E[0 .. N), their searches side by side
// (each step waits for gathers from an 82 MB table, whose lines bound the kernel).  The bin C(lo) <= r <
// C(lo + 1), C the two rows' interpolation, lies between the rows' own bins of
// r's cell: two or three steps instead of 13; a bracket that rounding put beside
// r is searched again from the whole row.
template <int N>
__device__ __forceinline__ void photon_pt(const double* __restrict__ cdf, const unsigned short* __restrict__ guide,
                                          double ptmax, const double* E, double gtot, const double* r, double* out)
{
  const double *c0[N], *c1[N];
  double w[N];
  int lo[N], hi[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const double eps = (E[i] * E[i]) / (gtot * gtot);
    const double le = eps > 0 ? log10(eps) : kPtEpsLo;
    double u = (le - kPtEpsLo) / (kPtEpsHi - kPtEpsLo) * (kPtEps - 1);
    u = u < 0 ? 0 : (u > kPtEps - 1 ? kPtEps - 1 : u);
    int i0 = (int)u;
    if (i0 > kPtEps - 2) i0 = kPtEps - 2;
    w[i] = u - i0;
    c0[i] = cdf + pt_row(i0);
    c1[i] = cdf + pt_row(i0 + 1);
    const int cell = 2 * (int)(r[i] * (kPtCells - 1));
    const unsigned short *g0 = guide + pt_guide(i0) + cell, *g1 = guide + pt_guide(i0 + 1) + cell;
    lo[i] = min(g0[0], g1[0]);
    hi[i] = min(max(g0[2], g1[2]) + 1, kPtBins);
  }
  auto C = [&](int i, int k) { return (1 - w[i]) * c0[i][pt_bin(k)] + w[i] * c1[i][pt_bin(k)]; };
  auto search = [&] {
    while (true) {
      bool more = false;
#pragma unroll
      for (int i = 0; i < N; ++i) more = more || hi[i] - lo[i] > 1;
      if (!more) break;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int mid = (lo[i] + hi[i]) >> 1;  // lo when its search is done
        if (C(i, mid) <= r[i] || mid == lo[i]) lo[i] = mid;
        else hi[i] = mid;
      }
    }
  };
  search();
  double cl[N], ch[N];
  bool beside = false;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    cl[i] = C(i, lo[i]), ch[i] = C(i, lo[i] + 1);
    if ((lo[i] > 0 && !(cl[i] <= r[i])) || (lo[i] < kPtBins - 1 && !(r[i] < ch[i]))) {
      beside = true;
      lo[i] = 0, hi[i] = kPtBins;
    }
  }
  if (beside) {
    search();
#pragma unroll
    for (int i = 0; i < N; ++i) cl[i] = C(i, lo[i]), ch[i] = C(i, lo[i] + 1);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const double frac = ch[i] > cl[i] ? (r[i] - cl[i]) / (ch[i] - cl[i]) : 0.5;
    out[i] = ptmax / kPtBins * (lo[i] + frac);
  }
}

struct EvGrid {
  int nm, ny, nz, pol, pdg;
  double mmin, mmax, ymin, ymax, zmin, zmax, mlep;
};

// TLorentzVector::Boost(bx, by, bz)
__device__ __forceinline__ void boost(double bx, double by, double bz, double* p)
{
  const double b2 = bx * bx + by * by + bz * bz;
  if (b2 <= 0) return;
  const double gamma = 1.0 / sqrt(1.0 - b2);
  const double bp = bx * p[0] + by * p[1] + bz * p[2];
  const double gamma2 = (gamma - 1.0) / b2;
  const double f = gamma2 * bp + gamma * p[3];
  p[0] += f * bx;
  p[1] += f * by;
  p[2] += f * bz;
  p[3] = gamma * (p[3] + bp);
}

__device__ __forceinline__ bool pass_cuts(const double* p, const upc_event_opts& o)
{
  const double pt = sqrt(p[0] * p[0] + p[1] * p[1]);
  if (o.do_pt_cut && pt < o.pt_min) return false;
  if (o.do_eta_cut) {
    const double eta = pt > 0 ? asinh(p[2] / pt) : (p[2] >= 0 ? 1e10 : -1e10);
    if (eta < o.eta_min || eta > o.eta_max) return false;
  }
  return true;
}

// One event per thread.  Bound: VALU issue (half the time: 12 uniforms, FP64
// transcendentals) and the L2 misses of the photon pt rows.  2,000,003 muon pairs
// with photon pt: 0.73 ms; with guides to the tables 0.39; with a pair of pt rows
// in one line 0.33.
__global__ void k_generate_pairs(EvGrid g, upc_event_opts o, const double* __restrict__ sum_ym,
                                 const double* __restrict__ sum_z, const double* __restrict__ sum_zs,
                                 const double* __restrict__ sum_zp, const double* __restrict__ ratio,
                                 PdfGuide<int> gym, PdfGuide<unsigned short> gz, PdfGuide<unsigned short> gzp,
                                 const double* __restrict__ ptcdf, const unsigned short* __restrict__ ptguide,
                                 double ptmax, double gtot,
                                 unsigned long long seed, unsigned long long offset, long long n,
                                 double* __restrict__ out_p, int* __restrict__ out_pdg, int* __restrict__ out_pass)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned long long ev = offset + (unsigned long long)i;
  Philox4x32 ph;
  double r[12];
  for (uint32_t b = 0; b < 6; ++b) {
    ph.block(seed, ev, b);
    r[2 * b] = philox_u01(ph.c[0], ph.c[1]);
    r[2 * b + 1] = philox_u01(ph.c[2], ph.c[3]);
  }
  double* P = out_p + 8 * i;
  out_pass[i] = 0;
  // (Y, M) from the 2-D pdf (UpcSampler2D, include/UpcSampler.h:118-121)
  double s0, s1;
  const int kbin = pdf_find(sum_ym, g.ny * g.nm, gym, 0, r[0], &s0, &s1);
  if (kbin < 0) return;
  const int iy = (int)((unsigned)kbin / (unsigned)g.nm), jm = kbin - iy * g.nm;
  const double dy = (g.ymax - g.ymin) / g.ny, dm = (g.mmax - g.mmin) / g.nm;
  const double y0 = g.ymin + dy * iy, y1 = g.ymin + dy * (iy + 1);
  const double m0 = g.mmin + dm * jm, m1 = g.mmin + dm * (jm + 1);
  const double Y = y0 + ((r[0] - s0) / (s1 - s0)) * (y1 - y0);
  const double M = m0 + r[1] * (m1 - m0);
  // getBinX / getBinY: truncation before the division (include/UpcSampler.h:124-133)
  const int ybin = (int)((double)(int)(g.ny * (Y - g.ymin)) / ((g.ymin + dy * g.ny) - g.ymin));
  int mbin = (int)((double)(int)(g.nm * (M - g.mmin)) / ((g.mmin + dm * g.nm) - g.mmin));
  if (mbin >= g.nm) mbin = g.nm - 1;
  // z = cos(theta) from the z pdf of that M row (src/UpcGenerator.cpp:742-757)
  const double* zt = sum_z;
  if (g.pol) {
    const int yb = ybin >= g.ny ? g.ny - 1 : ybin;
    if (r[3] < ratio[(long)yb * g.nm + mbin]) {
      zt = sum_zs;
    } else {
      zt = sum_zp;
      gz = gzp;
    }
  }
  zt += (long)mbin * (g.nz + 1);
  const int zb = pdf_find(zt, g.nz, gz, mbin, r[2], &s0, &s1);
  if (zb < 0) return;
  const double dz = (g.zmax - g.zmin) / g.nz;
  const double zl = g.zmin + dz * zb, zh = g.zmin + dz * (zb + 1);
  const double cost = zl + ((r[2] - s0) / (s1 - s0)) * (zh - zl);
  // pair momentum (getPairMomentum)
  double px = 0, py = 0, mt = M;
  if (o.nonzero_gam_pt) {
    const double k[2] = {M / 2 * exp(Y), M / 2 * exp(-Y)};
    double pt[2], s1, c1, s2, c2;
    photon_pt<2>(ptcdf, ptguide, ptmax, k, gtot, r + 6, pt);
    sincos(2 * kPi * r[4], &s1, &c1);
    sincos(2 * kPi * r[5], &s2, &c2);
    px = pt[0] * c1 + pt[1] * c2;
    py = pt[0] * s1 + pt[1] * s2;
    mt = sqrt(M * M + px * px + py * py);
  }
  const double pz = mt * sinh(Y), E = mt * cosh(Y);
  // pairProduction: back-to-back leptons in the pair frame, boosted to the lab
  const double m2 = E * E - (px * px + py * py + pz * pz);
  const double pmag = sqrt(m2 / 4 - g.mlep * g.mlep);
  const double theta = acos(cost);
  const double phi = 2 * kPi * r[8];
  double st, ct, sp, cp;
  sincos(theta, &st, &ct);
  sincos(phi, &sp, &cp);
  const double vx = pmag * st * cp, vy = pmag * st * sp, vz = pmag * ct;
  const double el = sqrt(pmag * pmag + g.mlep * g.mlep);
  double l1[4] = {vx, vy, vz, el}, l2[4] = {-vx, -vy, -vz, el};
  boost(px / E, py / E, pz / E, l1);
  boost(px / E, py / E, pz / E, l2);
  const int sign1 = (2 * r[9] - 1) > 0 ? 1 : -1;
  for (int c = 0; c < 4; ++c) {
    P[c] = l1[c];
    P[4 + c] = l2[c];
  }
  out_pdg[2 * i] = sign1 * g.pdg;
  out_pdg[2 * i + 1] = -sign1 * g.pdg;
  out_pass[i] = (pass_cuts(l1, o) && pass_cuts(l2, o)) ? 1 : 2;
}

static inline int nblk(long n, int bs) { return (int)((n + bs - 1) / bs); }

int build_pt_tables(upc_ctx* c, double gtot, hipStream_t s)
{
  PtTables* t = (PtTables*)c->events;
  if (!t) {
    t = new PtTables();
    c->events = t;
  }
  if (!t->cdf) UPC_HIP(hipMalloc(&t->cdf, sizeof(double) * (size_t)(kPtEps / 2) * (kPtLines * 16)));
  if (!t->guide) UPC_HIP(hipMalloc(&t->guide, sizeof(unsigned short) * (size_t)kPtEps * kPtCells));
  t->gtot = gtot;
  t->ptmax = 6. * kHc / c->cfg.R;
  hipLaunchKernelGGL(k_pt_tables, dim3(kPtEps), dim3(256), 0, s, c->d_ff, t->ptmax, t->cdf,
                     t->guide);
  UPC_HIP(hipGetLastError());
  return 0;
}

void free_events(upc_ctx* c)
{
  PtTables* t = (PtTables*)c->events;
  if (!t) return;
  if (t->cdf) (void)hipFree(t->cdf);
  if (t->guide) (void)hipFree(t->guide);
  delete t;
  c->events = nullptr;
}

int launch_generate_pairs(upc_ctx* c, const double* d_sum_ym, const double* d_sum_z, const double* d_sum_zs,
                          const double* d_sum_zp, const double* d_ratio, const upc_event_opts* opts,
                          unsigned long long seed, unsigned long long offset, long long n, double* d_p, int* d_pdg,
                          int* d_pass, hipStream_t s)
{
  if (n <= 0) return 0;
  const upc_config& cf = c->cfg;
  PtTables* t = (PtTables*)c->events;
  if (opts->nonzero_gam_pt && (!t || !t->cdf)) {
    set_error("photon pt tables not built: call upc_photon_pt_tables first");
    return UPC_ESTATE;
  }
  if (cf.use_polarized ? (!d_sum_zs || !d_sum_zp || !d_ratio) : !d_sum_z) {
    set_error("missing z sampler tables");
    return UPC_EINVAL;
  }
  const int pol = cf.use_polarized;
  PdfGuides guides;
  if (int rc = guides.build(d_sum_ym, pol ? d_sum_zs : d_sum_z, pol ? d_sum_zp : nullptr, cf.nm * cf.ny, cf.nz, cf.nm, n,
                            s))
    return rc;
  EvGrid g{cf.nm, cf.ny, cf.nz, cf.use_polarized, cf.proc_id, cf.mmin, cf.mmax, cf.ymin, cf.ymax, cf.zmin, cf.zmax,
           cf.proc_id == 11 ? kMEl : (cf.proc_id == 13 ? kMMu : kMTau)};
  hipLaunchKernelGGL(k_generate_pairs, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, g, *opts, d_sum_ym, d_sum_z,
                     d_sum_zs, d_sum_zp, d_ratio, guides.ym, guides.z, guides.zp, t ? t->cdf : nullptr,
                     t ? t->guide : nullptr, t ? t->ptmax : 0.0, t ? t->gtot : 1.0, seed,
                     offset, n, d_p, d_pdg, d_pass);
  UPC_HIP(hipGetLastError());
  return 0;
}

// photon pt draws alone (for tests of the getPhotonPt distribution)
__global__ void k_photon_pt(const double* __restrict__ cdf, const unsigned short* __restrict__ guide,
                            double ptmax, double gtot, const double* __restrict__ E,
                            unsigned long long seed, long long n, double* __restrict__ out)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  Philox4x32 ph;
  ph.block(seed, (unsigned long long)i, 7);
  const double r = philox_u01(ph.c[0], ph.c[1]);
  photon_pt<1>(cdf, guide, ptmax, E + i, gtot, &r, out + i);
}

int launch_photon_pt(upc_ctx* c, const double* d_E, long long n, unsigned long long seed, double* d_out, hipStream_t s)
{
  PtTables* t = (PtTables*)c->events;
  if (!t || !t->cdf) {
    set_error("photon pt tables not built: call upc_photon_pt_tables first");
    return UPC_ESTATE;
  }
  if (n <= 0) return 0;
  hipLaunchKernelGGL(k_photon_pt, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, t->cdf, t->guide, t->ptmax, t->gtot, d_E,
                     seed, n, d_out);
  UPC_HIP(hipGetLastError());
  return 0;
}

}  // namespace upc
