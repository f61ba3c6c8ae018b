// The library's host side on a stand-in for the HIP runtime: a device of a given
// memory whose kernels are recorded and not run.  For what only a full device
// shows: which kernels a call launches when an allocation fails.
//   host_paths <case>, exit code 0 and "ok" when the case holds.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "upc_lumi.h"

namespace {

size_t capacity = ~size_t(0), live = 0;  // bytes of the device
bool pool_fails = false;                 // hipMallocAsync finds no memory
long clear_threads = 0, clear_counters = 0;  // of the last k_batch_clear, a thread per counter
hipError_t last_error = hipSuccess;
std::map<void*, size_t> blocks;
std::vector<std::string> launches;
std::map<const void*, std::string>& kernels()  // the library registers its own before main's statics
{
  static std::map<const void*, std::string> k;
  return k;
}

hipError_t fail(hipError_t e) { return last_error = e; }

hipError_t take(void** p, size_t n)
{
  *p = nullptr;
  if (n > capacity - live) return fail(hipErrorOutOfMemory);
  *p = calloc(1, n ? n : 1);
  blocks[*p] = n;
  live += n;
  return hipSuccess;
}

hipError_t give(void* p)
{
  const auto it = blocks.find(p);
  if (it == blocks.end()) return p ? fail(hipErrorInvalidValue) : hipSuccess;
  live -= it->second;
  blocks.erase(it);
  free(p);
  return hipSuccess;
}

struct CallConfig {
  dim3 grid, block;
  size_t shmem;
  hipStream_t stream;
} config;

}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*)
{
  static void* module = nullptr;
  return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
  kernels()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t stream)
{
  config = {grid, block, shmem, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* stream)
{
  *grid = config.grid, *block = config.block, *shmem = config.shmem, *stream = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t)
{
  launches.push_back(kernels()[f]);
  if (launches.back().find("k_batch_clear") != std::string::npos) {
    clear_threads = (long)grid.x * block.x;
    clear_counters = *(const int*)args[1];
  }
  return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) { return take(p, n); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t)
{
  return pool_fails ? (*p = nullptr, fail(hipErrorOutOfMemory)) : take(p, n);
}
hipError_t hipFreeAsync(void* p, hipStream_t) { return give(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
  *p = calloc(1, n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void* d, int v, size_t n)
{
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }

hipError_t hipGetLastError()
{
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s)
{
  return *s = hipStreamCaptureStatusNone, hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return *e = nullptr, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = nullptr, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0.f, hipSuccess; }

}  // extern "C"

namespace {

#define CHECK(cond)                                                                          \
  do {                                                                                       \
    if (!(cond)) {                                                                           \
      printf("line %d: %s\nlast error: %s\nlaunches:", __LINE__, #cond, upc_last_error());   \
      for (const std::string& l : launches) printf(" %s", l.c_str());                        \
      printf("\n");                                                                          \
      exit(1);                                                                               \
    }                                                                                        \
  } while (0)

int launched(const char* name)
{
  int n = 0;
  for (const std::string& l : launches) n += l.find(name) != std::string::npos;
  return n;
}

upc_config config_of(int flux_point, int nm, int ny, int nz)
{
  upc_config c{};
  c.Z = 82, c.A = 208, c.R = 6.68, c.a = 0.447, c.sqrts = 5020.0;
  c.flux_point = flux_point, c.breakup_mode = 2;
  c.nm = nm, c.mmin = 3.5, c.mmax = 50.0;
  c.ny = ny, c.ymin = -6.0, c.ymax = 6.0;
  c.nz = nz, c.zmin = -1.0, c.zmax = 1.0;
  c.proc_id = 13;
  return c;
}

upc_ctx* context(const upc_config& c)
{
  upc_ctx* ctx = nullptr;
  CHECK(upc_ctx_create(&c, nullptr, &ctx) == 0);
  launches.clear();
  return ctx;
}

double cell[1];  // stands for every array that only kernels touch
double cells[5000];  // and that the host copies

// Draws: guides to the tables where a call makes many; without memory for them
// the plain search, which needs none.
void draws(bool pairs, bool full)
{
  upc_ctx* ctx = context(config_of(1, 101, 41, 50));
  pool_fails = full;
  const upc_event_opts opts{};
  const long long n = 1 << 20;
  int out[1];
  const int rc = pairs ? upc_generate_pairs(ctx, cell, cell, nullptr, nullptr, nullptr, &opts, 1, 0, n, cell, out, out, nullptr)
                       : upc_sample_events(ctx, cell, cell, nullptr, nullptr, nullptr, 1, 0, n, cell, cell, cell, nullptr);
  CHECK(rc == 0);
  CHECK(launched("k_pdf_guides") == (full ? 0 : 1));
  CHECK(launched(pairs ? "k_generate_pairs" : "k_sample_events") == 1);
  CHECK(hipGetLastError() == hipSuccess);
  upc_ctx_destroy(ctx);
  CHECK(live == 0);
}

size_t largest_block()
{
  size_t n = 0;
  for (const auto& b : blocks) n = std::max(n, b.second);
  return n;
}

// Whether n draws from tables of these sizes take guides.
void guided(int nm, int ny, int nz, int pol, long long n, int want)
{
  upc_config cf = config_of(1, nm, ny, nz);
  cf.use_polarized = pol;
  upc_ctx* ctx = context(cf);
  CHECK(upc_sample_events(ctx, cell, cell, cell, cell, cell, 1, 0, n, cell, cell, cell, nullptr) == 0);
  CHECK(launched("k_pdf_guides") == want);
  upc_ctx_destroy(ctx);
}

// Whole form-factor grids on a device with `left` bytes beside the context's
// tables: the integrand factors take what is there, and where they do not fit,
// the kernel that needs none.
constexpr int kBig[2] = {1024, 200};  // 205,824 flux rows, 3,216 groups of 64: 864 MB of factors
constexpr size_t kRows = 371000000;    // flux rows, points and the list of integrals handed on

void grid(size_t left, int table_launches, int direct_launches)
{
  upc_ctx* ctx = context(config_of(0, kBig[0], kBig[1], 50));
  if (left) capacity = live + left;
  CHECK(upc_lumi_grid(ctx, UPC_FORM_FP64, cell, nullptr, nullptr, nullptr) == 0);
  CHECK(launched("k_flux_h") == table_launches && launched("k_flux_qags_table") == table_launches);
  CHECK(launched("k_flux_qags_rows") == direct_launches);
  CHECK(launched("k_flux_qags_wave") == 1 && launched("k_lumi_fp64") == 1);
  CHECK(hipGetLastError() == hipSuccess);
  // again, and a smaller call, in the buffers that are there
  const size_t held = live;
  CHECK(upc_lumi_grid(ctx, UPC_FORM_FP64, cell, nullptr, nullptr, nullptr) == 0);
  CHECK(upc_lumi_points(ctx, cells, cells, 5000, cells, nullptr, nullptr, nullptr) == 0);
  CHECK(live == held);
  upc_ctx_destroy(ctx);
  CHECK(live == 0);
}

void batch(size_t left, int table_launches, int direct_launches)
{
  const upc_config jobs[2] = {config_of(0, kBig[0], kBig[1], 50), config_of(0, 21, 11, 50)};  // the second: no factors
  upc_batch* b = nullptr;
  CHECK(upc_batch_create(jobs, 2, nullptr, &b) == 0);
  const size_t held = live - largest_block();  // everything but the factors
  CHECK(upc_batch_destroy(b) == 0);
  CHECK(live == 0);
  if (left) capacity = held + left;
  CHECK(upc_batch_create(jobs, 2, nullptr, &b) == 0);
  double* L[2] = {cell, cell};
  CHECK(upc_batch_set_outputs(b, L, nullptr, nullptr) == 0);
  launches.clear();
  CHECK(upc_batch_run(b, 0, nullptr) == 0);
  CHECK(launched("k_flux_h") == table_launches && launched("k_flux_qags_table") == table_launches);
  CHECK(launched("k_flux_qags_rows") == direct_launches);
  CHECK(launched("k_flux_qags_wave") == 1 && launched("k_lumi_fp64") == 1);
  CHECK(hipGetLastError() == hipSuccess);
  CHECK(upc_batch_destroy(b) == 0);
  CHECK(live == 0);
}

// The largest job: more work cursors than row buckets, all of them cleared.
void batch_large()
{
  const upc_config job = config_of(0, 4000, 4000, 50);
  upc_batch* b = nullptr;
  CHECK(upc_batch_create(&job, 1, nullptr, &b) == 0);
  CHECK(clear_counters > 10240 && clear_threads >= clear_counters);
  CHECK(upc_batch_destroy(b) == 0);
}

// Tuning times the launch shapes that differ: three for the kernel without
// factors, two for the one with them (two workgroups fill a CU).
void tune(int njobs, int table_launches, int direct_launches)
{
  const upc_config jobs[2] = {config_of(0, kBig[0], kBig[1], 50), config_of(0, 21, 11, 50)};
  upc_batch* b = nullptr;
  CHECK(upc_batch_create(jobs, njobs, nullptr, &b) == 0);
  double* L[2] = {cell, cell};
  CHECK(upc_batch_set_outputs(b, L, nullptr, nullptr) == 0);
  launches.clear();
  upc_tune t;
  CHECK(upc_batch_autotune(b, nullptr, &t) == 0);
  CHECK(launched("k_flux_qags_table") == 1 + table_launches);  // and once before the timed passes
  CHECK(launched("k_flux_qags_rows") == direct_launches);
  CHECK(t.qags_candidates[2] == 3 && t.qags_blocks_per_cu >= 1);
  CHECK(njobs > 1 || (t.qags_ms[2] == t.qags_ms[1] && t.qags_blocks_per_cu < 3));
  CHECK(upc_batch_destroy(b) == 0);
}

}  // namespace

int main(int argc, char** argv)
{
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "draws") draws(false, false);
  else if (what == "draws_full") draws(false, true);
  else if (what == "pairs") draws(true, false);
  else if (what == "pairs_full") draws(true, true);
  else if (what == "grid") grid(0, 1, 0);
  else if (what == "grid_short") grid(kRows + 450000000, 2, 0);  // half of the factors
  else if (what == "grid_full") grid(kRows + 30000000, 0, 1);
  else if (what == "batch") batch(0, 1, 1);
  else if (what == "batch_short") batch(240000000, 4, 1);  // a quarter
  else if (what == "batch_full") batch(30000000, 0, 1);
  else if (what == "batch_large") batch_large();
  else if (what == "tune_shared") tune(1, 2, 0);
  else if (what == "tune_mixed") tune(2, 3, 4);
  else if (what == "guided" && argc == 8)
    guided(atoi(argv[2]), atoi(argv[3]), atoi(argv[4]), atoi(argv[5]), atoll(argv[6]), atoi(argv[7]));
  else return printf("no case %s\n", what.c_str()), 2;
  printf("ok\n");
  return 0;
}
