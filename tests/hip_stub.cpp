// hip_stub.cpp -- a stand-in for the HIP runtime, for tests of the library's
// host code without a GPU.  Loaded before librcgrid.so (RTLD_GLOBAL), its
// functions take the place of the runtime's: device memory is host memory
// within a limit, streams do nothing, kernel launches are counted and not
// run, rocFFT plans are empty.  As in the runtime, a call that fails leaves its error for
// hipGetLastError, which clears it.
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>
#include <unordered_map>

namespace {

struct Dim3 {
  unsigned x, y, z;
};

constexpr int OK = 0, NOMEM = 2;
std::mutex mu;
size_t live = 0, limit = (size_t)1 << 30, n_free = 0;
std::atomic<long> launches{0};
int per_cu = 2;                 // workgroups of a kernel on a CU
unsigned last_grid[1025] = {};  // blocks of the last launch, by threads a block
thread_local int last_error = OK;
thread_local int fail_new = 0;  // the fail_new-th operator new from here on throws
thread_local Dim3 cfg_grid, cfg_block;
thread_local size_t cfg_lds;
thread_local void *cfg_stream;

std::unordered_map<void *, size_t> &blocks()
{
  static auto *m = new std::unordered_map<void *, size_t>;
  return *m;
}

int ret(int e)
{
  if (e != OK) last_error = e;
  return e;
}

}  // namespace

extern "C" {

// ---- what the tests set and read
void stub_limit(size_t bytes) { limit = bytes; }
size_t stub_live() { return live; }
size_t stub_frees() { return n_free; }
long stub_launches() { return launches; }
void stub_per_cu(int n) { per_cu = n; }
unsigned stub_last_grid(int threads) { return last_grid[threads]; }
void stub_fail_new(int n) { fail_new = n; }
int stub_new_left() { return fail_new; }

int hipMalloc(void **p, size_t bytes)
{
  const int keep = fail_new;
  fail_new = 0;  // not the library's own
  std::lock_guard<std::mutex> lk(mu);
  if (live + bytes > limit || !(*p = calloc(1, bytes ? bytes : 1))) {
    fail_new = keep;
    return ret(NOMEM);
  }
  live += bytes;
  blocks()[*p] = bytes;
  fail_new = keep;
  return OK;
}
int hipFree(void *p)
{
  if (!p) return OK;
  std::lock_guard<std::mutex> lk(mu);
  const auto b = blocks().find(p);
  if (b == blocks().end()) abort();  // freed twice, or never allocated
  live -= b->second;
  n_free++;
  blocks().erase(b);
  free(p);
  return OK;
}
int hipHostMalloc(void **p, size_t bytes, unsigned)
{
  *p = malloc(bytes ? bytes : 1);
  return *p ? OK : ret(NOMEM);
}
int hipHostFree(void *p)
{
  free(p);
  return OK;
}
int hipMemcpy(void *d, const void *s, size_t n, int)
{
  memcpy(d, s, n);
  return OK;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *)
{
  memcpy(d, s, n);
  return OK;
}
int hipMemsetAsync(void *d, int v, size_t n, void *)
{
  memset(d, v, n);
  return OK;
}
int hipGetDevice(int *d)
{
  *d = 0;
  return OK;
}
int hipSetDevice(int) { return OK; }
int hipDeviceGetAttribute(int *v, int, int)
{
  *v = 256;
  return OK;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t)
{
  *n = per_cu;
  return OK;
}
int hipFuncSetAttribute(const void *, int, int) { return OK; }
int hipStreamCreateWithFlags(void **s, unsigned)
{
  *s = malloc(1);
  return OK;
}
int hipStreamDestroy(void *s)
{
  free(s);
  return OK;
}
int hipStreamSynchronize(void *) { return OK; }
int hipEventCreate(void **e)
{
  *e = malloc(1);
  return OK;
}
int hipEventCreateWithFlags(void **e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void *e)
{
  free(e);
  return OK;
}
int hipEventRecord(void *, void *) { return OK; }
int hipEventSynchronize(void *) { return OK; }
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t lds, void *st)
{
  cfg_grid = g;
  cfg_block = b;
  cfg_lds = lds;
  cfg_stream = st;
  return OK;
}
int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *lds, void **st)
{
  *g = cfg_grid;
  *b = cfg_block;
  *lds = cfg_lds;
  *st = cfg_stream;
  return OK;
}
int hipLaunchKernel(const void *, Dim3 grid, Dim3 block, void **, size_t, void *)
{
  launches++;
  if (block.x <= 1024) last_grid[block.x] = grid.x;
  return OK;
}
int hipGetLastError()
{
  const int e = last_error;
  last_error = OK;
  return e;
}
const char *hipGetErrorString(int) { return "stub error"; }

// rocFFT: plans of no content
int rocfft_setup() { return OK; }
int rocfft_cleanup() { return OK; }
int rocfft_plan_create(void **p, int, int, int, size_t, const size_t *, size_t, void *)
{
  *p = malloc(1);
  return OK;
}
int rocfft_plan_destroy(void *p)
{
  free(p);
  return OK;
}
int rocfft_plan_description_create(void **p) { return rocfft_plan_create(p, 0, 0, 0, 0, nullptr, 0, nullptr); }
int rocfft_plan_description_destroy(void *p) { return rocfft_plan_destroy(p); }
int rocfft_plan_description_set_data_layout(...) { return OK; }
int rocfft_execution_info_create(void **p) { return rocfft_plan_create(p, 0, 0, 0, 0, nullptr, 0, nullptr); }
int rocfft_execution_info_destroy(void *p) { return rocfft_plan_destroy(p); }
int rocfft_execution_info_set_stream(void *, void *) { return OK; }
int rocfft_execution_info_set_work_buffer(void *, void *, size_t) { return OK; }
int rocfft_plan_get_work_buffer_size(void *, size_t *n)
{
  *n = 4096;
  return OK;
}
int rocfft_execute(void *, void **, void **, void *) { return OK; }

}  // extern "C"

void *operator new(size_t n)
{
  if (fail_new && --fail_new == 0) throw std::bad_alloc();
  if (void *p = malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }
