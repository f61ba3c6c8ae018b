// Launches of the FP64 two-photon contraction (k_lumi_fp64), of one view and of
// a batch's jobs.  A unit of its own: the options the flux kernels' units are
// compiled with (build.py) cost this kernel 4 %.
#include "upc_internal.h"
#include "upc_batch_job.h"

namespace upc {

// Contraction job resolver: blk0[j] = first block of job j for this wave count.
struct BatchLumi {
  static constexpr int kWavesPerEu = 4;  // register budget of k_lumi_fp64 (waves per SIMD)
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

int launch_lumi_fp64(const LumiView& v, hipStream_t s)
{
  constexpr int kWaves = 4;
  const int nwork = lumi_work_items(v.npts, v.fp.mirror_ny, v.mirror_out);
  if (nwork <= 0) return 0;
  hipLaunchKernelGGL((k_lumi_fp64<kWaves, SingleLumi>), dim3((nwork + kWaves - 1) / kWaves), dim3(64 * kWaves), 0, s,
                     SingleLumi{v});
  UPC_HIP(hipGetLastError());
  return 0;
}

int launch_lumi_batch(const BatchJob* jobs, const int* blk0, int njobs, int waves, int blocks, hipStream_t s)
{
  const BatchLumi jr{jobs, blk0, njobs};
  const dim3 grid(blocks), block(64 * waves);
  if (waves == 2) hipLaunchKernelGGL((k_lumi_fp64<2, BatchLumi>), grid, block, 0, s, jr);
  else if (waves == 4) hipLaunchKernelGGL((k_lumi_fp64<4, BatchLumi>), grid, block, 0, s, jr);
  else hipLaunchKernelGGL((k_lumi_fp64<8, BatchLumi>), grid, block, 0, s, jr);
  UPC_HIP(hipGetLastError());
  return 0;
}

}  // namespace upc
