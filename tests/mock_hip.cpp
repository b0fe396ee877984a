// A recording stand-in for the HIP runtime (tests only): loaded before
// libspecfab_gpu.so in a process of its own, it takes the library's runtime
// calls, so that the host side (which kernel with which arguments, how many
// threads, which memory) is tested without a GPU.  Kernels are recorded and
// not run; "device" memory is reserved host memory.  A launch advances a clock
// by a cost per kernel (mock_cost), which the events read.
#define SFG_HOST_EMUL
#include <sys/mman.h>

#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "sfg_fold.h"

thread_local sfg_dim3 threadIdx, blockIdx, blockDim, gridDim;
void sfg_emul_syncthreads() {}

namespace {
struct Dim { unsigned x = 1, y = 1, z = 1; };
struct Launch {
    std::string name;
    Dim grid, block;
    std::vector<char> arg;   // the first kernel argument
};
struct Cost { std::string part; double fixed, per_group; };
std::map<const void*, std::string> kernels;
struct Var { void* p = nullptr; size_t bytes = 0; };
std::map<const void*, Var> vars;
std::map<char*, size_t> mem;
std::vector<Launch> launches;
std::vector<Cost> costs;
Dim cfg_grid, cfg_block;
double now = 0;
int failed = 0;   // launches that HIP refuses

char* reserve(size_t n) {
    void* p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (p == MAP_FAILED) return nullptr;
    mem[(char*)p] = n;
    return (char*)p;
}
// true where [p, p + n) lies in one allocation or device variable
bool inside(const void* p, size_t n) {
    auto it = mem.upper_bound((char*)p);
    if (it == mem.begin()) return false;
    --it;
    return (char*)p + n <= it->first + it->second;
}
int record(const void* fn, Dim g, Dim b, void** args) {
    Launch l;
    l.name = kernels.count(fn) ? kernels[fn] : "?";
    l.grid = g;
    l.block = b;
    size_t n = 0;
    if (l.name.find("fold_kernel") != l.name.npos) n = sizeof(sfg::FoldArgs);
    if (l.name.find("params_kernel") != l.name.npos) n = sizeof(sfg::ParamArgs);
    if (l.name.find("evolve_") != l.name.npos) n = sizeof(sfg::EvolveArgs);
    if (n) l.arg.assign((char*)args[0], (char*)args[0] + n);
    // the runtime's limit on work-items per dimension
    if ((unsigned long long)g.x * b.x >= (1ull << 32)) {
        failed++;
        return 1;
    }
    double t = 0;
    for (auto& c : costs)
        if (l.name.find(c.part) != l.name.npos) t = c.fixed + c.per_group * g.x;
    now += t;
    launches.push_back(l);
    return 0;
}
}  // namespace

extern "C" {
int mock_count() { return (int)launches.size(); }
int mock_failed() { return failed; }
void mock_reset() { launches.clear(); failed = 0; }
void mock_cost(const char* part, double fixed, double per_group) { costs.push_back({part, fixed, per_group}); }
const char* mock_name(int i) { return launches[i].name.c_str(); }
long long mock_threads(int i) { return (long long)launches[i].grid.x * launches[i].block.x; }
// params_kernel: are its results inside one allocation
int mock_params_in_bounds(int i) {
    sfg::ParamArgs a;
    memcpy(&a, launches[i].arg.data(), sizeof a);
    return inside(a.theta, (size_t)a.P * sfg::NPAR_K * 8) && inside(a.omega, (size_t)a.P * 15 * 8) &&
           inside(a.sl, (size_t)a.P * a.nblk * 8);
}// fold_kernel: the parcels of the launch
void mock_fold_span(int i, long long* p0, long long* n) {
    sfg::FoldArgs a;
    memcpy(&a, launches[i].arg.data(), sizeof a);
    *p0 = a.p0;
    *n = a.np;
}

void** __hipRegisterFatBinary(const void*) { static void* m; return &m; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels[host] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int) { vars[var].bytes = size; }
int __hipPushCallConfiguration(Dim g, Dim b, size_t, void*) { cfg_grid = g; cfg_block = b; return 0; }
int __hipPopCallConfiguration(Dim* g, Dim* b, size_t* s, void** st) {
    *g = cfg_grid; *b = cfg_block; *s = 0; *st = nullptr;
    return 0;
}
int hipLaunchKernel(const void* fn, Dim g, Dim b, void** args, size_t, void*) { return record(fn, g, b, args); }
struct NodeParams { Dim block; void** extra; void* func; Dim grid; void** kernelParams; unsigned shared; };
int hipGraphAddKernelNode(void** node, void*, void* const*, size_t, const NodeParams* p) {
    *node = &launches;
    return record(p->func, p->grid, p->block, p->kernelParams);
}
int hipGraphCreate(void** g, unsigned) { *g = &launches; return 0; }
int hipGraphDestroy(void*) { return 0; }
int hipGraphExecDestroy(void*) { return 0; }
int hipGraphInstantiate(void** e, void*, void**, char*, size_t) { *e = &launches; return 0; }
int hipGraphLaunch(void*, void*) { return 0; }
int hipMalloc(void** p, size_t n) { return (*p = reserve(n ? n : 1)) ? 0 : 2; }
int hipFree(void* p) {
    auto it = mem.find((char*)p);
    if (it == mem.end()) return p ? 1 : 0;
    munmap(it->first, it->second);
    mem.erase(it);
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) { memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { memcpy(d, s, n); return 0; }
int hipMemcpy2DAsync(void*, size_t, const void*, size_t, size_t, size_t, int, void*) { return 0; }
int hipMemset(void* d, int v, size_t n) { memset(d, v, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void*) { memset(d, v, n); return 0; }
int hipGetSymbolAddress(void** p, const void* var) {
    Var& v = vars[var];
    if (!v.p) v.p = reserve(v.bytes);
    *p = v.p;
    return v.p ? 0 : 1;
}
int hipEventCreate(double** e) { *e = new double(0); return 0; }
int hipEventCreateWithFlags(double** e, unsigned) { *e = new double(0); return 0; }
int hipEventDestroy(double* e) { delete e; return 0; }
int hipEventRecord(double* e, void*) { *e = now; return 0; }
int hipEventSynchronize(double*) { return 0; }
int hipEventElapsedTime(float* ms, double* a, double* b) { *ms = (float)(*b - *a); return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
int hipSetDevice(int) { return 0; }
int hipDeviceSynchronize() { return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { *s = &launches; return 0; }
int hipStreamDestroy(void*) { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "refused by the recording runtime"; }
}
