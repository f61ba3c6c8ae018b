// The batch's job record and flux rows, shared by its flux kernels (upc_batch.hip,
// upc_flux_rows.hip) and its contraction (upc_lumi.hip).
#pragma once
#include "upc_flux.h"

namespace upc {

struct BatchJob {
  LumiView v;          // pts, row_logd, flux point at this job's slice
  const double4* ff;
  const double* j1;
  int nm, ny;
  double mmin, mmax, ymin, ymax;
  int pt0, row0;       // first point and row of the job in the batch arrays
  int nrows;           // its flux rows
  int grp0;            // its first group of 64 positions in the sorted rows
};

__device__ __forceinline__ int find_job(const int* __restrict__ start, int njobs, long idx)
{
  int lo = 0, hi = njobs - 1;  // largest j with start[j] <= idx
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (start[mid] <= idx) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Flux rows of the batch for the QAGS kernels, sorted job by job, every job from
// a group of its own on; as a task source, task t = row * 120 + node (its flux
// slot).
struct BatchRows {
  const double* __restrict__ row_k;
  const double* __restrict__ row_logd;
  const int* __restrict__ row_cnt;
  int* __restrict__ perm;
  const BatchJob* __restrict__ jobs;
  const int* __restrict__ row0;
  int njobs;
  const int* __restrict__ group_job;  // job of each group
  const int* __restrict__ nsorted;    // [njobs] rows in perm
  long long g0, g1;                   // the groups of this launch
  unsigned long long* __restrict__ job_failed;  // [njobs] integrals with ier != 0
  __device__ long long groups() const { return g1 - g0; }
  __device__ bool need(int) const { return true; }
  __device__ int group(long long g, long long* first, int* job) const
  {
    *first = (g0 + g) * 64;
    *job = group_job[g0 + g];
    const int left = nsorted[*job] - (int)(g0 + g - jobs[*job].grp0) * 64;
    return left < 64 ? left : 64;
  }
  __device__ long long span(int job, long long* r0, long long* pos0) const
  {
    *r0 = jobs[job].row0;
    *pos0 = (long long)jobs[job].grp0 * 64;
    return jobs[job].nrows;
  }
  __device__ RowJob params(int job) const
  {
    const BatchJob& J = jobs[job];
    return RowJob{J.ff, J.j1, J.v.fp.bmin, J.v.fp.g1, J.v.fp.factor, J.v.fp.A};
  }
  __device__ void failed(int job) const { atomicAdd(&job_failed[job], 1ull); }
  __device__ void get(long long t, FluxTask* ft) const
  {
    const long long r = t / kNB1;
    const int jb = find_job(row0, njobs, r);
    const RowJob P = params(jb);
    ft->b = row_node_b(P.bmin, row_logd[r], (int)(t - r * kNB1));
    ft->k = row_k[r];
    ft->out = t;
    ft->ff = P.ff;
    ft->g1 = P.g1;
    ft->factor = P.factor;
    ft->A = P.A;
    ft->slot = jb;
  }
};

// upc_lumi.hip: the FP64 contraction of every job, `waves` (2, 4 or 8) work
// items per workgroup; blk0[j] = first workgroup of job j.
int launch_lumi_batch(const BatchJob* jobs, const int* blk0, int njobs, int waves, int blocks, hipStream_t s);

}  // namespace upc
