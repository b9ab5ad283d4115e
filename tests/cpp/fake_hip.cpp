// A HIP runtime without a device, for tests of the host code around the kernels: memory is host memory (each allocation
// ends at an inaccessible page, so that an overrun faults), copies happen at once, kernels do not run, and every call is
// appended to a log. Asynchronous copies, launches and allocations can be made to fail.
#include <sys/mman.h>

#include <cstdio>
#include <cstring>
#include <map>
#include <string>

namespace {

std::string log_text;
std::map<const void*, std::string> kernels;
std::map<void*, std::pair<void*, size_t>> blocks;  // address handed out -> mapping
std::map<const void*, void*> symbols;
int fail_after[3] = {-1, -1, -1};  // calls of each kind (0 copy, 1 launch, 2 allocation) that still succeed; -1 all
int busy = 0;                  // stream queries that still find work
int verdict = -1, verdicts = 0;  // the next `verdicts` launches of k_admissible raise flag `verdict`
int last_error = 0;

void note(const std::string& s) { log_text += s + "\n"; }
bool fails(int kind) { return fail_after[kind] >= 0 && fail_after[kind]-- == 0; }
std::string hex(const void* p)
{
  char b[32];
  std::snprintf(b, sizeof b, "%p", p);
  return b;
}

int take(void** out, size_t bytes)
{
  const size_t page = 4096, n = (bytes + page - 1) / page * page;
  char* m = static_cast<char*>(mmap(nullptr, n + page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
  if (m == MAP_FAILED) return 2;
  mprotect(m + n, page, PROT_NONE);
  *out = m + (n - (bytes + 15) / 16 * 16);
  blocks[*out] = {m, n + page};
  return 0;
}
int give(void* p)
{
  const auto it = blocks.find(p);
  if (it == blocks.end()) return p ? 1 : 0;
  munmap(it->second.first, it->second.second);
  blocks.erase(it);
  return 0;
}

struct Dim
{
  unsigned x, y, z;
};
struct
{
  Dim grid, block;
  size_t shared;
  void* stream;
} config;

}  // namespace

extern "C" {

const char* fake_log() { return log_text.c_str(); }
void fake_clear() { log_text.clear(); }
void fake_fail(int kind, int after) { fail_after[kind] = after; }
void fake_busy(int queries) { busy = queries; }
void fake_verdict(int flag, int launches) { verdict = flag, verdicts = launches; }

void* __hipRegisterFatBinary(const void*)
{
  static int handle;
  return &handle;
}
void __hipUnregisterFatBinary(void*) {}
void __hipRegisterFunction(void*, const void* host, char*, const char* name, int, void*, void*, void*, void*, int*)
{
  kernels[host] = name;
}
void __hipRegisterVar(void*, void* var, char*, char*, int, size_t size, int, int)
{
  void* p = nullptr;
  take(&p, size);
  symbols[var] = p;
}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t shared, void* stream)
{
  config = {grid, block, shared, stream};
  return 0;
}
int __hipPopCallConfiguration(Dim* grid, Dim* block, size_t* shared, void** stream)
{
  *grid = config.grid;
  *block = config.block;
  *shared = config.shared;
  *stream = config.stream;
  return 0;
}

int hipGetDeviceCount(int* n) { return *n = 1, 0; }
int hipGetDevice(int* d) { return *d = 0, 0; }
int hipSetDevice(int) { return 0; }
int hipGetDevicePropertiesR0600(void* p, int) { return std::memset(p, 0, 64), 0; }
const char* hipGetErrorString(int e) { return e ? "fake error" : "no error"; }
int hipGetLastError()
{
  const int e = last_error;
  last_error = 0;
  return e;
}
int hipGetSymbolAddress(void** p, const void* var) { return *p = symbols[var], 0; }
int hipMalloc(void** p, size_t n) { return fails(2) ? 2 : take(p, n); }
int hipFree(void* p) { return give(p); }
int hipHostMalloc(void** p, size_t n, unsigned) { return fails(2) ? 2 : take(p, n); }
int hipHostFree(void* p) { return give(p); }
int hipMemcpy(void* d, const void* s, size_t n, int) { return std::memcpy(d, s, n), 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*)
{
  if (fails(0)) return 1;
  note("copy " + std::to_string(n));
  std::memcpy(d, s, n);
  return 0;
}
int hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), 0; }
int hipMemsetAsync(void* d, int v, size_t n, void*) { return std::memset(d, v, n), 0; }
int hipLaunchKernel(const void* f, Dim, Dim, void** args, size_t, void*)
{
  if (fails(1)) return last_error = 1;
  note("launch " + kernels[f]);
  // k_local_euler(mesh, operators by value, device operators, coefficient, device time step, stage, residual, filter,
  // Dt_fuse {minima, ...}, ...)
  if (kernels[f].find("k_local_euler") != std::string::npos) {
    note("time step " + hex(*static_cast<void**>(args[4])));
    note("minima " + hex(*static_cast<void**>(args[8])));
  }
  // k_admissible(mesh, class, flags)
  if (kernels[f].find("k_admissibleI") != std::string::npos && verdicts > 0) {
    (*static_cast<int**>(args[2]))[verdict] = 1;
    --verdicts;
  }
  return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned) { return *s = new char, 0; }
int hipStreamDestroy(void* s) { return delete static_cast<char*>(s), 0; }
int hipStreamSynchronize(void*) { return note("wait"), 0; }
int hipDeviceSynchronize() { return note("wait"), 0; }
int hipStreamQuery(void*) { return busy > 0 ? (--busy, 600) : 0; }  // hipErrorNotReady
int hipStreamBeginCapture(void*, int) { return 1; }
int hipStreamEndCapture(void*, void**) { return 1; }
int hipGraphInstantiate(void**, void*, void*, char*, size_t) { return 1; }
int hipGraphLaunch(void*, void*) { return 1; }
int hipGraphDestroy(void*) { return 0; }
int hipGraphExecDestroy(void*) { return 0; }
int hipEventCreate(void** e) { return *e = new char, 0; }
int hipEventDestroy(void* e) { return delete static_cast<char*>(e), 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) { return *ms = 0, 0; }

}  // extern "C"
