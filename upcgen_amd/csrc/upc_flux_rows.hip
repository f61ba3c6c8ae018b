// k_flux_qags_rows, the row QAGS kernel without shared factors.  A unit of its
// own: the options that the other QAGS kernels' units are compiled with
// (build.py) cost this kernel 9 % (101 x 41: 0.68 -> 0.75 ms).
#include "upc_internal.h"
#include "upc_batch_job.h"

namespace upc {

template <int CAP, class RS>
__global__ __launch_bounds__(kQagsBlock) __attribute__((amdgpu_waves_per_eu(kQagsRowsWaves, kQagsRowsWaves)))
void k_flux_qags_rows(RS rs, unsigned long long* __restrict__ cursor,
                      double* __restrict__ flux, unsigned long long* __restrict__ stats,
                      long long* __restrict__ overflow, int fast_cap)
{
  __shared__ double lds[kQagsBlock / 64][20 * 64];
  const int lane = threadIdx.x & 63;
  double* fv = lds[threadIdx.x >> 6] + lane;
  typename QagsSmallStore<CAP>::Arrays lists;
  Qags<QagsSmallStore<CAP>> q;
  q.s.a = &lists;
  q.s.lim = fast_cap < CAP ? fast_cap : CAP;
  const unsigned long long nids = (unsigned long long)rs.groups() * kMaxQagsNodesPerRow;
  unsigned my_evals = 0, my_bad = 0;  // 32-bit per lane; evaluations flushed before they could wrap
  while (true) {
    unsigned long long id = 0;
    if (lane == 0) id = atomicAdd(cursor, 1ull);
    id = __shfl(id, 0);
    if (id >= nids) break;
    const int g = __builtin_amdgcn_readfirstlane((int)(id / kMaxQagsNodesPerRow));
    const int j = (int)(id - (unsigned long long)g * kMaxQagsNodesPerRow);
    long long first;
    int r = 0, job = 0;
    bool live = false;
    if (lane < rs.group(g, &first, &job)) {
      r = rs.perm[first + lane];
      live = j < rs.row_cnt[r];
    }
    if (__ballot(live) != 0) {
      const RowJob P = rs.params(job);
      double b = 0.0, w2g2 = 0.0;
      if (live) {
        b = row_node_b(P.bmin, rs.row_logd[r], j);
        const double k = rs.row_k[r];
        w2g2 = k * k / P.g1 / P.g1;
        q.start();
      }
      while (__ballot(live) != 0) {
        if (!live) continue;
        QK21Out o{}, o2{};
#pragma unroll 1
        for (int pass = 0; pass < q.passes(); ++pass) {
          double qa, qb;
          q.interval(pass, &qa, &qb);
          o = o2;
          o2 = qk21_rows<64>(fv, qa, qb, P.ff, b, w2g2);
        }
        if (q.phase == 0) o = o2;
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

template <class RS>
void launch_qags_rows_direct(const RS& rs, unsigned long long* cursor, double* flux, unsigned long long* stats,
                             long long* overflow, int cap, int blocks, hipStream_t s)
{
  hipLaunchKernelGGL((k_flux_qags_rows<kQagsCap, RS>), dim3(blocks), dim3(kQagsBlock), 0, s, rs, cursor, flux, stats,
                     overflow, cap);
}

template void launch_qags_rows_direct<GridRows>(const GridRows&, unsigned long long*, double*, unsigned long long*,
                                                long long*, int, int, hipStream_t);
template void launch_qags_rows_direct<BatchRows>(const BatchRows&, unsigned long long*, double*, unsigned long long*,
                                                 long long*, int, int, hipStream_t);

}  // namespace upc
