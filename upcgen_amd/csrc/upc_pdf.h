// Draws from prefix tables (gsl_histogram_pdf_sample): the bin i with sum[i] <=
// r < sum[i + 1].
#pragma once
#include "upc_internal.h"

namespace upc {

// Largest i in [lo, hi) with sum[i] <= r, given sum[lo] <= r (or lo = 0) and
// r < sum[hi] (or hi = n).
template <class T>
__device__ __forceinline__ T pdf_search(const double* __restrict__ sum, T lo, T hi, double r)
{
  while (hi - lo > 1) {
    const T mid = lo + ((hi - lo) >> 1);  // n may be up to the type's largest value
    if (r >= sum[mid]) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Guide to one or several tables of n bins: [g] is the bin of r = g / 2^bits, so
// the bin of r lies in [guide[g], guide[g + 1]], g = r 2^bits (an exact product).
// With as many cells as bins that leaves one probe on average where a search
// takes log2 n, each a gather of 64 lines.
template <class I>
struct PdfGuide {
  const I* cell = nullptr;  // [tables][2^bits + 1], null: search the whole table
  int bits = 0;
};

// The bin of r, -1 outside the table; *s0, *s1: the table at its ends.
template <class I>
__device__ __forceinline__ int pdf_find(const double* __restrict__ sum, int n, const PdfGuide<I>& guide, size_t table,
                                        double r, double* s0, double* s1)
{
  int lo = 0, hi = n;
  if (guide.cell) {
    const int g = (int)(r * (double)(1 << guide.bits));
    const I* c = guide.cell + table * ((size_t(1) << guide.bits) + 1) + g;
    lo = c[0];
    hi = min((int)c[1] + 1, n);
  }
  lo = pdf_search(sum, lo, hi, r);
  *s0 = sum[lo];
  *s1 = sum[lo + 1];
  // r < sum[0] ends in bin 0, r >= sum[n] in the last one
  return (lo == 0 && r < *s0) || (lo == n - 1 && r >= *s1) ? -1 : lo;
}

// The guides of a call's tables (upc_xsec.hip): built from them on the call's
// stream, so nothing outlives the call, and given back by the destructor in
// stream order.
struct PdfGuides {
  PdfGuide<int> ym;
  PdfGuide<unsigned short> z, zp;  // zp: the second polarised table (z: the first)
  hipStream_t stream = nullptr;
  void* buf = nullptr;
  int build(const double* sum_ym, const double* sum_z, const double* sum_zp, int nym, int nz, int nm, long long n,
            hipStream_t s);
  ~PdfGuides()
  {
    if (buf) (void)hipFreeAsync(buf, stream);
  }
};

}  // namespace upc
