// Stand-in for the HIP runtime calls that liblsjk makes, for tests of its host side on a machine
// without a GPU: "device" memory is host memory, copies happen at once, kernels do not run.  Loaded
// with RTLD_GLOBAL before liblsjk.so, whose calls then come here.  stub_* read what was recorded and
// set what is to fail (tests/host_scenarios.py).
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <sstream>
#include <string>
#include <vector>

namespace {
struct Dim3 {
    uint32_t x, y, z;
};
constexpr int kSuccess = 0, kInvalid = 1, kOutOfMemory = 2, kCapture = 900;
constexpr int kHostToDevice = 1, kDeviceToHost = 2;

std::map<void*, size_t> live;
std::map<const void*, std::string> kernels;  // host stub of a kernel -> its name
std::map<const void*, std::string> units;    // code object -> the names of its kernels, a line each
std::vector<std::string> launched;  // name and shape of each launch
long fail_at = -1;  // the allocation after this many more fails, and its retries (same size)
size_t failing = 0;
long bad_frees = 0, null_stream_copies = 0;
bool capturing = false;  // copies from pageable memory and waits are errors then
size_t uploaded = 0;
long allocations = 0, event_waits = 0;
int last_error = kSuccess;
std::string answer;  // what the next copy to the host of this size gives
struct Call {
    Dim3 grid, block;
    size_t lds;
    void* stream;
} pushed;
int handles;

int set(int e)
{
    if (e) last_error = e;
    return e;
}
int handle(void** p)
{
    *p = reinterpret_cast<void*>(static_cast<intptr_t>(++handles));
    return kSuccess;
}
void copy(void* dst, const void* src, size_t n, int kind)
{
    if (kind == kDeviceToHost && !answer.empty() && n == answer.size()) {
        std::memcpy(dst, answer.data(), n);
        answer.clear();
        return;
    }
    std::memcpy(dst, src, n);
    if (kind == kHostToDevice) uploaded += n;
}
}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*) { return new void*(nullptr); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void** unit, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    kernels[host] = name;
    units[unit] += std::string(name) + "\n";
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void* stream)
{
    pushed = {grid, block, lds, stream};
    return kSuccess;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* lds, void** stream)
{
    *grid = pushed.grid;
    *block = pushed.block;
    *lds = pushed.lds;
    *stream = pushed.stream;
    return kSuccess;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void**, size_t lds, void*)
{
    if (!grid.x || !grid.y || !grid.z || !block.x) return set(kInvalid);
    std::ostringstream s;
    s << kernels[f] << ' ' << grid.x << 'x' << grid.y << 'x' << grid.z << " of " << block.x << " lds " << lds;
    launched.push_back(s.str());
    return kSuccess;
}

int hipGetDeviceCount(int* n) { return *n = 1, kSuccess; }
int hipSetDevice(int) { return kSuccess; }
// the two attributes asked for: compute units, and LDS bytes per workgroup (the larger serves both)
int hipDeviceGetAttribute(int* v, int, int) { return *v = 65536, kSuccess; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { return *n = 4, kSuccess; }
int hipGetSymbolAddress(void** p, const void*) { return handle(p); }
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : e ? "error" : "no error"; }
int hipGetLastError(void)
{
    const int e = last_error;
    last_error = kSuccess;
    return e;
}

int hipMalloc(void** p, size_t n)
{
    if (fail_at >= 0 && fail_at-- == 0) failing = n;
    if (n == failing) return set(kOutOfMemory);
    failing = 0;
    *p = std::calloc(n ? n : 1, 1);
    live[*p] = n;
    allocations++;
    return kSuccess;
}
int hipFree(void* p)
{
    if (!p) return kSuccess;
    if (!live.erase(p)) return bad_frees++, set(kInvalid);
    std::free(p);
    return kSuccess;
}
int hipMemcpy(void* dst, const void* src, size_t n, int kind) { return null_stream_copies++, copy(dst, src, n, kind), kSuccess; }
int hipMemcpyAsync(void* dst, const void* src, size_t n, int kind, void* stream)
{
    if (capturing) return set(kCapture);
    if (!stream) null_stream_copies++;
    return copy(dst, src, n, kind), kSuccess;
}

int hipStreamCreateWithFlags(void** s, unsigned) { return handle(s); }
int hipStreamDestroy(void*) { return kSuccess; }
int hipStreamSynchronize(void*) { return set(capturing ? kCapture : kSuccess); }
int hipStreamWaitEvent(void*, void*, unsigned) { return event_waits++, kSuccess; }
int hipStreamBeginCapture(void*, int) { return capturing = true, kSuccess; }
int hipStreamEndCapture(void*, void** g) { return capturing = false, handle(g); }
int hipGraphInstantiate(void** e, void*, void*, char*, size_t) { return handle(e); }
int hipGraphLaunch(void*, void*) { return kSuccess; }
int hipGraphDestroy(void*) { return kSuccess; }
int hipGraphExecDestroy(void*) { return kSuccess; }
int hipEventCreate(void** e) { return handle(e); }
int hipEventCreateWithFlags(void** e, unsigned) { return handle(e); }
int hipEventDestroy(void*) { return kSuccess; }
int hipEventRecord(void*, void*) { return kSuccess; }
int hipEventSynchronize(void*) { return kSuccess; }
int hipEventElapsedTime(float* ms, void*, void*) { return *ms = 1.0f, kSuccess; }

// ---- what the tests ask
void stub_fail_at(long n) { fail_at = n; }
void stub_answer(const void* p, size_t n) { answer.assign(static_cast<const char*>(p), n); }
long stub_bad_frees(void) { return bad_frees; }
long stub_null_stream_copies(void) { return null_stream_copies; }
size_t stub_uploaded(void) { return uploaded; }
size_t stub_live_bytes(void)
{
    size_t n = 0;
    for (const auto& b : live) n += b.second;
    return n;
}
long stub_live_blocks(void) { return static_cast<long>(live.size()); }
long stub_allocations(void) { return allocations; }
long stub_event_waits(void) { return event_waits; }
// the launches from number `first` on, a line each
const char* stub_launch_log(long first)
{
    static std::string all;
    all.clear();
    for (size_t i = first; i < launched.size(); i++) all += launched[i] + "\n";
    return all.c_str();
}
// the kernels of code object i (what the first launch of one of them loads)
const char* stub_unit(long i)
{
    for (const auto& u : units)
        if (i-- == 0) return u.second.c_str();
    return nullptr;
}
// launches so far of kernels with `part` in their (mangled) names
long stub_launches(const char* part)
{
    long n = 0;
    for (const auto& s : launched) n += s.find(part) != std::string::npos;
    return n;
}
}
