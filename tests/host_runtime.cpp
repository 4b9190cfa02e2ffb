// Test helper: a stand-in for the parts of the HIP runtime that the engine's
// host code calls, in host memory, with several devices.  Loaded before
// libboids_engine.so with global symbols, it takes the engine's calls.
//   - Kernels do nothing.
//   - Copies and fills are queued on their stream and done when somebody
//     waits for it, so memory that is read, freed or lent again too early shows.
//   - An event belongs to the device that was current when it was made, and a
//     stream of another device refuses it, as HIP's does.
//   - rt_fail(name, k) lets the k-th call of `name` from then on fail.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <functional>
#include <list>
#include <map>
#include <mutex>
#include <new>
#include <string>

namespace {
constexpr int kDevices = 4;
thread_local int current = 0;
thread_local hipError_t last = hipSuccess;
std::recursive_mutex mu;
struct Mem { size_t bytes; int device; bool host; };
std::map<char*, Mem> mem;
struct Op { std::function<void()> go; char* to; char* from; };
struct Stream { int device; std::list<Op> ops; uint64_t done = 0, queued = 0; };
struct Event { int device; Stream* on; uint64_t at; };
std::map<std::string, int> countdown;
std::map<std::string, uint64_t> calls;
std::map<char*, uint64_t> copied;                      // bytes that copies wrote into each block
thread_local int news_left = 0, inside = 0;            // operator new fails on this thread when news_left comes
                                                       // down to 0 (the stand-in's own calls do not count)
struct Inside { Inside() { ++inside; } ~Inside() { --inside; } };

bool fails(const char* name)
{
    ++calls[name];
    auto it = countdown.find(name);
    return it != countdown.end() && it->second > 0 && --it->second == 0;
}
std::map<char*, Mem>::iterator block_of(const void* p)
{
    auto it = mem.upper_bound((char*)p);
    if (it == mem.begin()) return mem.end();
    --it;
    return (char*)p < it->first + it->second.bytes ? it : mem.end();
}
void run(Stream* s, uint64_t until)
{
    while (s->done < until && !s->ops.empty()) {
        s->ops.front().go();
        s->ops.pop_front();
        ++s->done;
    }
}
hipError_t take(void** p, size_t bytes, bool host)
{
    *p = calloc(1, bytes ? bytes : 1);
    if (!*p) return hipErrorOutOfMemory;
    mem[(char*)*p] = {bytes ? bytes : 1, current, host};
    return hipSuccess;
}
hipError_t give(void* p)
{
    if (p && !mem.erase((char*)p)) return hipErrorInvalidValue;
    copied.erase((char*)p);
    free(p);
    return hipSuccess;
}
}  // namespace

#define LOCK std::lock_guard<std::recursive_mutex> lk(mu); Inside in
#define MAY_FAIL(name) if (fails(name)) return last = hipErrorUnknown

// An allocation failure inside the engine's own calls, on the calling thread.
void* operator new(size_t n)
{
    if (!inside && news_left > 0 && --news_left == 0) throw std::bad_alloc();
    void* p = malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

extern "C" {
void rt_fail(const char* name, int k) { LOCK; countdown[name] = k; }
void rt_fail_new(int k) { news_left = k; }
uint64_t rt_calls(const char* name) { LOCK; return calls[name]; }
int rt_current(void) { return current; }
// device memory in use, of all devices (-1) or one
uint64_t rt_device_bytes(int device)
{
    LOCK;
    uint64_t sum = 0;
    for (auto& m : mem)
        if (!m.second.host && (device < 0 || m.second.device == device)) sum += m.second.bytes;
    return sum;
}
// copies in flight that write or read memory from hipHostMalloc
uint64_t rt_in_flight(void);
// bytes that copies have written into the block at p
uint64_t rt_copied_to(const void* p) { LOCK; return copied[(char*)p]; }

static std::list<Stream*> streams;
uint64_t rt_in_flight(void)
{
    LOCK;
    uint64_t k = 0;
    for (Stream* s : streams)
        for (auto& op : s->ops)
            for (char* p : {op.to, op.from}) {
                auto b = p ? block_of(p) : mem.end();
                if (b != mem.end() && b->second.host) ++k;
            }
    return k;
}

hipError_t hipSetDevice(int d) { LOCK; MAY_FAIL("hipSetDevice"); if (d < 0 || d >= kDevices) return hipErrorInvalidDevice; current = d; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = kDevices; return hipSuccess; }
hipError_t hipGetLastError(void) { const hipError_t e = last; last = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorInvalidHandle ? "invalid handle" : e == hipErrorUnknown ? "made to fail" : "error"; }
hipError_t hipMalloc(void** p, size_t n) { LOCK; MAY_FAIL("hipMalloc"); return take(p, n, false); }
hipError_t hipFree(void* p) { LOCK; return give(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { LOCK; MAY_FAIL("hipHostMalloc"); return take(p, n, true); }
hipError_t hipHostFree(void* p) { LOCK; return give(p); }
hipError_t hipGetSymbolAddress(void**, const void*) { return hipErrorInvalidSymbol; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
    LOCK;
    memset(a, 0, sizeof(*a));
    auto b = block_of(p);
    a->type = b == mem.end() ? hipMemoryTypeUnregistered : b->second.host ? hipMemoryTypeHost : hipMemoryTypeDevice;
    if (b != mem.end()) a->device = b->second.device;
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    LOCK;
    Stream* n = new Stream{current, {}};
    streams.push_back(n);
    *s = (hipStream_t)n;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    LOCK;
    MAY_FAIL("hipStreamSynchronize");
    run((Stream*)s, ((Stream*)s)->queued);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    LOCK;
    run((Stream*)s, ((Stream*)s)->queued);
    streams.remove((Stream*)s);
    delete (Stream*)s;
    return hipSuccess;
}
static hipError_t new_event(hipEvent_t* e) { *e = (hipEvent_t) new Event{current, nullptr, 0}; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { LOCK; MAY_FAIL("hipEventCreate"); return new_event(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { LOCK; MAY_FAIL("hipEventCreate"); return new_event(e); }
hipError_t hipEventDestroy(hipEvent_t e) { LOCK; delete (Event*)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    LOCK;
    MAY_FAIL("hipEventRecord");
    if (((Event*)e)->device != ((Stream*)s)->device) return hipErrorInvalidHandle;
    ((Event*)e)->on = (Stream*)s;
    ((Event*)e)->at = ((Stream*)s)->queued;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    LOCK;
    MAY_FAIL("hipEventSynchronize");
    if (((Event*)e)->on) run(((Event*)e)->on, ((Event*)e)->at);
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }

hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind kind, hipStream_t s)
{
    LOCK;
    MAY_FAIL("hipMemcpyAsync");
    auto b = block_of(to);
    if (kind == hipMemcpyDeviceToHost && b == mem.end()) {      // pageable memory: the runtime waits for it
        run((Stream*)s, ((Stream*)s)->queued);
        memcpy(to, from, n);
        return hipSuccess;
    }
    if (kind == hipMemcpyHostToDevice && block_of(from) == mem.end()) {
        run((Stream*)s, ((Stream*)s)->queued);
        memcpy(to, from, n);
        return hipSuccess;
    }
    if (b == mem.end()) return hipErrorInvalidValue;
    copied[b->first] += n;
    ((Stream*)s)->ops.push_back({[=] { memcpy(to, from, n); }, (char*)to, (char*)from});
    ++((Stream*)s)->queued;
    return hipSuccess;
}
hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind) { LOCK; memcpy(to, from, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* to, int v, size_t n, hipStream_t s)
{
    LOCK;
    ((Stream*)s)->ops.push_back({[=] { memset(to, v, n); }, (char*)to, nullptr});
    ++((Stream*)s)->queued;
    return hipSuccess;
}
// (what a launch expands to: the stream goes through here)
static thread_local hipStream_t launch_stream = nullptr;
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t s) { launch_stream = s; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* s)
{
    *grid = *block = dim3(1);
    *shared = 0;
    *s = launch_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t s)
{
    LOCK;
    MAY_FAIL("hipLaunchKernel");
    ((Stream*)s)->ops.push_back({[] {}, nullptr, nullptr});
    ++((Stream*)s)->queued;
    return hipSuccess;
}
}
