// Host stand-in of the HIP runtime for tests of host code without a GPU:
// device memory is host memory, kernels do not run.  Loaded with RTLD_GLOBAL
// ahead of the library, whose HIP calls then come here.  The test's hooks see
// every launch, may refuse an allocation and may change what a copy to the
// host brings.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <string>

struct Dim {
  uint32_t x, y, z;
};

typedef void (*launch_hook)(const char* name, uint32_t gx, uint32_t gy, uint32_t gz, void** args);
typedef int (*refuse_hook)(size_t bytes, int kind);  // kind 0 device, 1 pinned host
typedef void (*d2h_hook)(void* dst, size_t bytes);

static launch_hook on_launch;
static refuse_hook refuse;
static d2h_hook on_d2h;
static std::map<const void*, std::string>* names;
static std::map<uintptr_t, size_t>* live;
static struct {
  Dim grid, block;
  size_t shmem;
  void* stream;
} call;
static size_t new_limit = ~(size_t)0;

static int take(void** p, size_t n, int kind) {
  if (!live) live = new std::map<uintptr_t, size_t>();
  *p = nullptr;
  if (refuse && refuse(n, kind)) return 2;  // hipErrorOutOfMemory
  void* v = calloc(n ? n : 1, 1);
  if (!v) return 2;
  if (kind == 0) (*live)[(uintptr_t)v] = n;
  *p = v;
  return 0;
}

// a C++ allocation of at least new_limit bytes fails
void* operator new(size_t n) {
  void* p = n >= new_limit ? nullptr : malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

extern "C" {

void host_hip_hooks(launch_hook l, refuse_hook r, d2h_hook d) {
  on_launch = l;
  refuse = r;
  on_d2h = d;
}
void host_hip_new_limit(size_t n) { new_limit = n; }

// Bytes from p to the end of the live device allocation that holds it, or -1.
long long host_hip_room(const void* p) {
  if (!live) return -1;
  auto it = live->upper_bound((uintptr_t)p);
  if (it == live->begin()) return -1;
  --it;
  const uintptr_t end = it->first + it->second;
  return (uintptr_t)p < end ? (long long)(end - (uintptr_t)p) : -1;
}
long long host_hip_live_bytes() {
  long long s = 0;
  if (live)
    for (auto& a : *live) s += (long long)a.second;
  return s;
}

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*) {
  if (!names) names = new std::map<const void*, std::string>();
  (*names)[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

int __hipPushCallConfiguration(Dim g, Dim b, size_t s, void* st) {
  call = {g, b, s, st};
  return 0;
}
int __hipPopCallConfiguration(Dim* g, Dim* b, size_t* s, void** st) {
  *g = call.grid;
  *b = call.block;
  *s = call.shmem;
  *st = call.stream;
  return 0;
}
int hipLaunchKernel(const void* f, Dim g, Dim, void** args, size_t, void*) {
  if (on_launch) on_launch(names && names->count(f) ? (*names)[f].c_str() : "", g.x, g.y, g.z, args);
  return 0;
}

int hipMalloc(void** p, size_t n) { return take(p, n, 0); }
int hipFree(void* p) {
  if (live) live->erase((uintptr_t)p);
  free(p);
  return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) { return take(p, n, 1); }
int hipHostFree(void* p) {
  free(p);
  return 0;
}
int hipHostGetDevicePointer(void** d, void* h, unsigned) {
  *d = h;
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind) {
  if (n) memmove(d, s, n);
  if (kind == 2 && on_d2h) on_d2h(d, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*) {
  return hipMemcpy(d, s, n, kind);
}
int hipMemset(void* d, int v, size_t n) {
  memset(d, v, n);
  return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) { return hipMemset(d, v, n); }

int hipGetDeviceCount(int* n) {
  *n = 1;
  return 0;
}
int hipGetDevice(int* d) {
  *d = 0;
  return 0;
}
int hipDeviceGetAttribute(int* v, int, int) {
  *v = 256;
  return 0;
}
int hipDeviceSynchronize() { return 0; }
int hipFuncSetAttribute(const void*, int, int) { return 0; }
const char* hipGetErrorString(int) { return "host stand-in"; }
int hipGetLastError() { return 0; }
int hipGetSymbolAddress(void** p, const void*) {
  static char space[1 << 20];
  *p = space;
  return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned) {
  *s = malloc(1);
  return 0;
}
int hipStreamDestroy(void* s) {
  free(s);
  return 0;
}
int hipStreamSynchronize(void*) { return 0; }
int hipEventCreateWithFlags(void** e, unsigned) {
  *e = malloc(1);
  return 0;
}
int hipEventDestroy(void* e) {
  free(e);
  return 0;
}
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 0.f;
  return 0;
}
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) {
  *g = malloc(1);
  return 0;
}
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) {
  *x = malloc(1);
  return 0;
}
int hipGraphLaunch(void*, void*) { return 0; }
int hipGraphDestroy(void* g) {
  free(g);
  return 0;
}
int hipGraphExecDestroy(void* x) {
  free(x);
  return 0;
}
}
