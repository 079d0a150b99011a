// A stand-in for the HIP runtime calls libofx.so makes, for host-side tests
// without a GPU: loaded before the library, its symbols take the runtime's
// place.  Device memory is zeroed host memory, copies are memcpy, kernels do not
// run.  It logs what the library asks for and can refuse it:
//   fake_log      "malloc <bytes>", "launch <stream> <kernel>", "copy <stream>",
//                 "sync <stream>", ... one per line, streams numbered from 1
//   fake_capacity device memory; hipMalloc beyond it fails
//   fake_fail     the n-th next call of a function fails (1: the next one)
//   fake_watch    log the size of the live block behind a kernel's pointer
//                 argument ("arg <bytes>", -1: no live block)
//   fake_cost     milliseconds a kernel takes between two events
// A failed call leaves its error for hipGetLastError, as the runtime does.
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
struct Dim3 { unsigned x, y, z; };
struct Watch { std::string kernel; int arg; };
struct Cost { std::string kernel; double ms; };
std::recursive_mutex mu;
std::string log_;
std::map<char*, size_t> live;
size_t held = 0, capacity = ~(size_t)0;
std::map<std::string, int> fails;
std::map<const void*, std::string> kernels;
std::vector<Watch> watches;
std::vector<Cost> costs;
std::map<void*, int> streams;
double clock_ = 0.0;
int next_stream = 1;
thread_local int last_error = 0;
constexpr int INVALID = 1, OOM = 2;

void note(const std::string& s) { log_ += s + "\n"; }
std::string id(void* st) { return std::to_string(streams.count(st) ? streams[st] : 0); }
int result(const char* fn, int err = INVALID) {  // of a call that may be told to fail
    auto it = fails.find(fn);
    if (it == fails.end() || --it->second > 0) return 0;
    fails.erase(it);
    note(std::string("fail ") + fn);
    return last_error = err;
}
int take(void** p, size_t n, const char* fn) {
    std::lock_guard<std::recursive_mutex> l(mu);
    note(std::string(fn) + " " + std::to_string(n));
    *p = nullptr;
    if (int e = result(fn, OOM)) return e;
    if (held + n > capacity) return last_error = OOM;
    char* q = static_cast<char*>(std::calloc(n, 1));
    live[q] = n;
    held += n;
    *p = q;
    return 0;
}
int give(void* p) {
    if (!p) return 0;
    std::lock_guard<std::recursive_mutex> l(mu);
    auto it = live.find(static_cast<char*>(p));
    if (it == live.end()) return last_error = INVALID;
    held -= it->second;
    live.erase(it);
    std::free(p);
    return 0;
}
long block(const char* p) {
    auto it = live.upper_bound(const_cast<char*>(p));
    if (it == live.begin()) return -1;
    --it;
    return p < it->first + it->second ? (long)(it->first + it->second - p) : -1;
}
}  // namespace

extern "C" {
const char* fake_log() { return log_.c_str(); }
void fake_clear() { log_.clear(); }
size_t fake_held() { return held; }
void fake_capacity(size_t n) { capacity = n; }
void fake_fail(const char* fn, int nth) { if (nth > 0) fails[fn] = nth; else fails.erase(fn); }
void fake_watch(const char* kernel, int arg) { watches.push_back({kernel, arg}); }
void fake_cost(const char* kernel, double ms) { costs.push_back({kernel, ms}); }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { kernels[f] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
thread_local struct { Dim3 g, b; size_t s; void* st; } cfg;
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t s, void* st) { cfg = {g, b, s, st}; return 0; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* s, void** st) { *g = cfg.g; *b = cfg.b; *s = cfg.s; *st = cfg.st; return 0; }
int hipLaunchKernel(const void* f, Dim3, Dim3, void** args, size_t, void* st) {
    std::lock_guard<std::recursive_mutex> l(mu);
    const std::string& k = kernels[f];
    note("launch " + id(st) + " " + k);
    for (const Watch& w : watches)
        if (k.find(w.kernel) != std::string::npos) note("arg " + std::to_string(block(*static_cast<char**>(args[w.arg]))));
    for (const Cost& c : costs)
        if (k.find(c.kernel) != std::string::npos) { clock_ += c.ms; break; }
    return 0;
}
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipSetDevice(int) { return 0; }
int hipGetLastError() { const int e = last_error; last_error = 0; return e; }
const char* hipGetErrorString(int e) { return e == OOM ? "out of memory" : e ? "invalid" : "no error"; }
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipMalloc(void** p, size_t n) { return take(p, n, "hipMalloc"); }
int hipHostMalloc(void** p, size_t n, unsigned) { return take(p, n, "hipHostMalloc"); }
int hipFree(void* p) { return give(p); }
int hipHostFree(void* p) { return give(p); }
int hipGetSymbolAddress(void** p, const void*) { static char area[16 << 20]; *p = area; return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) { std::memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void* st) {
    std::lock_guard<std::recursive_mutex> l(mu);
    note("copy " + id(st));
    if (int e = result("hipMemcpyAsync")) return e;
    std::memcpy(d, s, n);
    return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) { if (v) std::memset(d, v, n); return 0; }  // (memory comes zeroed)
int hipStreamCreateWithFlags(void** s, unsigned) {
    std::lock_guard<std::recursive_mutex> l(mu);
    *s = nullptr;
    if (int e = result("hipStreamCreateWithFlags")) return e;
    *s = std::malloc(1);
    streams[*s] = next_stream++;
    return 0;
}
int hipStreamDestroy(void* s) {
    std::lock_guard<std::recursive_mutex> l(mu);
    streams.erase(s);
    std::free(s);
    return 0;
}
int hipStreamSynchronize(void* s) {
    std::lock_guard<std::recursive_mutex> l(mu);
    note("sync " + id(s));
    return result("hipStreamSynchronize");
}
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) { *g = std::malloc(1); return 0; }
int hipGraphDestroy(void* g) { std::free(g); return 0; }
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) { *x = std::malloc(1); return 0; }
int hipGraphExecDestroy(void* x) { std::free(x); return 0; }
int hipGraphLaunch(void*, void*) { return 0; }
int hipEventCreateWithFlags(void** e, unsigned) { *e = new double(0.0); return 0; }
int hipEventCreate(void** e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void* e) { delete static_cast<double*>(e); return 0; }
int hipEventRecord(void* e, void*) {
    std::lock_guard<std::recursive_mutex> l(mu);
    *static_cast<double*>(e) = clock_;
    return 0;
}
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void* a, void* b) {
    *ms = (float)(*static_cast<double*>(b) - *static_cast<double*>(a));
    return 0;
}
}
