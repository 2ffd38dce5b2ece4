// Stand-in for the HIP runtime in the CPU tests of the library's host code
// (tests/test_host_paths.py), preloaded in place of libamdhip64.so.  Device
// memory is host memory with a budget, everything enqueued is done at once,
// and kernels do not run: a launch is one line of a log.  Only what the host
// reads back to decide by is imitated: the offsets of a block
// (k_offset_scan), whether its rows fit the row classes (k_class_scan), and
// the progress word of a solve (k_pcg_update_xp, k_pcg_update_r).
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {
struct State {
    std::mutex mu;
    size_t budget = size_t(64) << 30, used = 0, peak = 0;
    std::map<void*, size_t> blocks;
    std::map<const void*, std::string> kernels;
    std::string log;
    int per_cu = 8;         // blocks per CU the occupancy query answers
    int classes_fit = 1;    // whether k_class_scan finds few enough forms
    int stop_after = 0;     // the slot a solve stops in (0: never)
    int slots = 0;
    int waits = 0;          // stream synchronisations
    dim3 grid, block;
    size_t shmem = 0;
    hipStream_t stream = nullptr;
};
State& S()
{
    static State* s = new State;
    return *s;
}
// "void cel::f<double, 1>(...)" -> "f<double, 1>"
std::string plain(const char* mangled)
{
    int rc = 0;
    char* d = abi::__cxa_demangle(mangled, nullptr, nullptr, &rc);
    std::string s = d ? d : mangled;
    std::free(d);
    if (s.rfind("void ", 0) == 0) s = s.substr(5);
    int depth = 0;
    for (size_t i = 0; i < s.size(); ++i) {
        if (s[i] == '<') ++depth;
        if (s[i] == '>') --depth;
        if (s[i] == '(' && depth == 0 && s.compare(i, 11, "(anonymous ") != 0) {
            s.resize(i);
            break;
        }
    }
    for (const char* ns : {"cel::", "(anonymous namespace)::"})
        for (size_t p; (p = s.find(ns)) != std::string::npos;) s.erase(p, std::strlen(ns));
    return s;
}
template <typename T>
T arg(void** a, int i)
{
    return *static_cast<T*>(a[i]);
}
struct OffsetSet {  // dia.hip
    int slot[64], count, over, bad;
};
struct KeyTable {  // rowclass.hip
    unsigned long long key[1024];
    int cls[1024], row[256], count, over, bad;
};
void imitate(const std::string& k, void** a)
{
    if (k == "k_offset_scan") {
        const int n = arg<int>(a, 0), most = arg<int>(a, 3);
        const int *xadj = arg<const int*>(a, 1), *cols = arg<const int*>(a, 2);
        OffsetSet* g = arg<OffsetSet*>(a, 4);
        for (int& v : g->slot) v = -2147483647 - 1;
        g->count = g->over = g->bad = 0;
        for (int i = 0; i < n && !g->over; ++i)
            for (int j = xadj[i]; j < xadj[i + 1]; ++j) {
                if (j > xadj[i] && cols[j] <= cols[j - 1]) g->bad = 1;
                int at = 0;
                while (at < g->count && g->slot[at] != cols[j] - i) ++at;
                if (at < g->count) continue;
                if (g->count == most) {
                    g->over = 1;
                    break;
                }
                g->slot[g->count++] = cols[j] - i;
            }
    } else if (k == "k_class_scan") {
        arg<KeyTable*>(a, 7)->over = !S().classes_fit;
    } else if (k.rfind("k_pcg_update_xp<", 0) == 0 || k.rfind("k_pcg_update_r<", 0) == 0) {
        int* progress = arg<int*>(a, k[13] == 'x' ? 12 : 11);
        if (!progress) return;
        ++S().slots;
        *progress = S().stop_after && S().slots >= S().stop_after ? -1 : S().slots;
    }
}
}  // namespace

extern "C" {
// ---- the test's side
void stub_budget(size_t bytes) { S().budget = bytes; }
size_t stub_used() { return S().used; }
size_t stub_peak(int reset)
{
    const size_t p = S().peak;
    if (reset) S().peak = S().used;
    return p;
}
void stub_occupancy(int per_cu) { S().per_cu = per_cu; }
void stub_classes_fit(int fit) { S().classes_fit = fit; }
void stub_stop_after(int slots)
{
    S().stop_after = slots;
    S().slots = 0;
}
int stub_waits() { return S().waits; }
const char* stub_log() { return S().log.c_str(); }
void stub_log_clear() { S().log.clear(); }

// ---- code objects and launches
void** __hipRegisterFatBinary(const void*)
{
    static void* one[1];
    return one;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    S().kernels[host] = plain(name);
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st)
{
    State& s = S();
    s.grid = g;
    s.block = b;
    s.shmem = sh;
    s.stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* st)
{
    State& s = S();
    *g = s.grid;
    *b = s.block;
    *sh = s.shmem;
    *st = s.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3, void** args, size_t, hipStream_t)
{
    State& s = S();
    const std::string& k = s.kernels[f];
    s.log += k + " " + std::to_string(g.x) + "\n";
    imitate(k, args);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    static void* scratch = std::calloc(size_t(64) << 20, 1);
    *p = scratch;
    return hipSuccess;
}

// ---- memory
hipError_t hipMalloc(void** p, size_t n)
{
    State& s = S();
    std::lock_guard<std::mutex> l(s.mu);
    *p = nullptr;
    if (s.used + n > s.budget) return hipErrorOutOfMemory;
    *p = std::calloc(n ? n : 1, 1);
    s.blocks[*p] = n;
    s.used += n;
    if (s.used > s.peak) s.peak = s.used;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    State& s = S();
    std::lock_guard<std::mutex> l(s.mu);
    const auto it = s.blocks.find(p);
    if (it == s.blocks.end()) return p ? hipErrorInvalidValue : hipSuccess;
    s.used -= it->second;
    s.blocks.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    *p = std::calloc(n ? n : 1, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t)
{
    std::memset(d, v, n);
    return hipSuccess;
}

// ---- device, streams, events, graphs
hipError_t hipGetDeviceCount(int* n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->name, "host stub");
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int)
{
    *v = 0;
    return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t)
{
    *n = S().per_cu;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    *s = reinterpret_cast<hipStream_t>(std::calloc(1, 8));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    ++S().waits;
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = reinterpret_cast<hipEvent_t>(std::calloc(1, 8));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 0.0f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
    S().log += "capture\n";
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
    *g = reinterpret_cast<hipGraph_t>(std::calloc(1, 8));
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g)
{
    std::free(g);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    *e = reinterpret_cast<hipGraphExec_t>(std::calloc(1, 8));
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e)
{
    std::free(e);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t)
{
    S().log += "graph\n";
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipGetLastError() { return hipSuccess; }
}  // extern "C"
