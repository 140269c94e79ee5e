// A HIP runtime without a device, for tests of the library's host code on the
// CPU: loaded with RTLD_GLOBAL before libadgpu_hip.so, its functions take the
// runtime's place.  Memory is host memory and kernels do nothing, but every
// launch is noted with its kernel's name, shape and stream, and streams run on
// a few modelled queues: a launch begins when its queue is free (on a busy
// device when every queue is), which the kernel that looks for streams side by
// side (k_hold) reports as the device would.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

struct dim3_ { uint32_t x, y, z; };
struct Stream { int id, queue; };
struct Launch { std::string kernel; uint32_t grid, block; size_t lds; int stream, queue; };

std::recursive_mutex mu;
int queues = 4, streams_made = 0, streams_alive = 0, streams_limit = 1 << 30, busy = 0;
int launches_left = 1 << 30, last_error = 0;
std::map<void*, int> unfinished;   // launches of a stream that nothing has waited for
size_t host_limit = SIZE_MAX;
std::vector<size_t> allocations;   // of device memory, in bytes
std::vector<int> users;
std::vector<uint64_t> queue_free;
uint64_t now = 1;
std::vector<Launch> launches;
std::map<const void*, std::string> names;
thread_local dim3_ grid_, block_;
thread_local size_t lds_;
thread_local void* stream_;

void start() {
    if (!users.empty()) return;
    if (const char* e = std::getenv("GPU_MAX_HW_QUEUES")) queues = std::atoi(e);
    users.assign(queues, 0);
    queue_free.assign(queues, 0);
    users[0] = 1;   // the null stream
}

}  // namespace

extern "C" {

// controls
void fake_streams_limit(int n) { streams_limit = n; }
void fake_busy(int on) { busy = on; }
void fake_host_limit(size_t bytes) { host_limit = bytes; }
int fake_streams_alive() { return streams_alive; }
void fake_launches_left(int n) { launches_left = n; }
int fake_unfinished() {
    int n = 0;
    for (const auto& s : unfinished) n += s.second;
    return n;
}
void fake_clear() { launches.clear(); allocations.clear(); }
int fake_allocations_of(size_t bytes) {
    int n = 0;
    for (size_t a : allocations) n += a == bytes;
    return n;
}
int fake_launches() { return (int)launches.size(); }
const char* fake_kernel(int i) { return launches[i].kernel.c_str(); }
int fake_block(int i) { return (int)launches[i].block; }
int fake_stream(int i) { return launches[i].stream; }
int fake_queue(int i) { return launches[i].queue; }

// registration and launches
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    names[f] = name;
}
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t lds, void* s) {
    grid_ = g; block_ = b; lds_ = lds; stream_ = s;
    return 0;
}
int __hipPopCallConfiguration(dim3_* g, dim3_* b, size_t* lds, void** s) {
    *g = grid_; *b = block_; *lds = lds_; *s = stream_;
    return 0;
}
int hipLaunchKernel(const void* f, dim3_ g, dim3_ b, void** args, size_t lds, void* s) {
    std::lock_guard<std::recursive_mutex> l(mu);
    start();
    Stream* st = (Stream*)s;
    const int q = st ? st->queue : 0;
    const std::string& name = names[f];
    if (launches_left-- <= 0) return last_error = 719;   // a launch failure
    launches.push_back({name, g.x, b.x, lds, st ? st->id : -1, q});
    unfinished[s]++;
    if (name.find("k_hold") != std::string::npos) {   // (uint64_t* span, uint32_t ticks of 10 ns)
        uint64_t* span = *(uint64_t**)args[0];
        const uint64_t ticks = *(uint32_t*)args[1];
        now += 500;   // 5 us a launch
        uint64_t begin = queue_free[q];
        if (busy)
            for (uint64_t t : queue_free) begin = t > begin ? t : begin;
        begin = begin > now ? begin : now;
        span[0] = begin;
        span[1] = begin + ticks;
        queue_free[q] = begin + ticks;
    }
    return 0;
}

// streams and events
int hipStreamCreateWithFlags(void** s, unsigned) {
    std::lock_guard<std::recursive_mutex> l(mu);
    start();
    if (streams_alive >= streams_limit) { *s = nullptr; return 2; }
    int q = 0;
    for (int k = 1; k < queues; ++k)
        if (users[k] < users[q]) q = k;
    users[q]++;
    streams_alive++;
    *s = new Stream{streams_made++, q};
    return 0;
}
int hipStreamDestroy(void* s) {
    std::lock_guard<std::recursive_mutex> l(mu);
    users[((Stream*)s)->queue]--;
    streams_alive--;
    unfinished.erase(s);
    delete (Stream*)s;
    return 0;
}
int hipStreamSynchronize(void* s) {
    std::lock_guard<std::recursive_mutex> l(mu);
    unfinished.erase(s);
    for (uint64_t t : queue_free) now = t > now ? t : now;
    return 0;
}
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipStreamBeginCapture(void*, int) { return 801; }
int hipStreamEndCapture(void*, void**) { return 801; }
int hipGraphInstantiate(void**, void*, void*, char*, size_t) { return 801; }
int hipGraphLaunch(void*, void*) { return 801; }
int hipGraphDestroy(void*) { return 0; }
int hipGraphExecDestroy(void*) { return 0; }
int hipEventCreateWithFlags(void** e, unsigned) { *e = std::malloc(1); return 0; }
int hipEventCreate(void** e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void* e) { std::free(e); return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventQuery(void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 0.f; return 0; }

// memory
int hipMalloc(void** p, size_t n) {
    std::lock_guard<std::recursive_mutex> l(mu);
    allocations.push_back(n);
    *p = std::calloc(n ? n : 1, 1);
    return *p ? 0 : 2;
}
int hipFree(void* p) { std::free(p); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned) {
    if (n > host_limit) { *p = nullptr; return 2; }
    *p = std::calloc(n ? n : 1, 1);
    return *p ? 0 : 2;
}
int hipHostFree(void* p) { std::free(p); return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) { std::memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { std::memcpy(d, s, n); return 0; }
int hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int, void*) {
    for (size_t k = 0; k < h; ++k) std::memcpy((char*)d + k * dp, (const char*)s + k * sp, w);
    return 0;
}
int hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void*) { std::memset(d, v, n); return 0; }
int hipMemGetInfo(size_t* f, size_t* t) { *f = *t = (size_t)1 << 38; return 0; }
int hipGetSymbolAddress(void** p, const void*) { static char area[1 << 26]; *p = area; return 0; }

// device
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipSetDevice(int) { return 0; }
int hipSetDeviceFlags(unsigned) { return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }   // compute units
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int threads, size_t) {
    *n = 1024 / threads;   // 16 wavefronts
    return 0;
}
int hipGetLastError() {
    const int e = last_error;
    last_error = 0;
    return e;
}
const char* hipGetErrorString(int) { return "fake error"; }

}  // extern "C"
