// A HIP runtime without a device, for tests of the engine's host side on the CPU: memory is host memory
// under a settable limit, copies are copies, kernels do not run.  Launches are logged by kernel name,
// graphs replay their part of the log, and events measure a clock that every launch advances by a
// settable time.  Loaded with global symbols before libkpmx.so, whose HIP calls it then takes.
//
// Two kernels leave something, so that plans of the chained recurrence can be built: the rings of a tile
// of r rows get r + growth * j local rows up to distance j (growths of sampled, of all and of the first
// tiles apart), as far as these fit.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
constexpr int RINGS = 13;  // ring counts of a tile

std::map<const void*, std::string> g_kernels;
std::map<void*, size_t> g_memory;
size_t g_used = 0, g_limit = (size_t)8 << 30;
std::vector<std::string> g_log, g_captured;
std::vector<std::vector<std::string>> g_graphs;
bool g_capturing = false;
int g_captures = 0, g_sample_growth = 16, g_growth = 16, g_region = 0, g_region_growth = 0;
double g_clock = 0;  // us
std::map<std::string, double> g_cost;
std::string g_text;

double cost(const std::string& name) {
    double best = 5;
    size_t length = 0;
    for (auto& c : g_cost)
        if (name.compare(0, c.first.size(), c.first) == 0 && c.first.size() >= length) {
            best = c.second;
            length = c.first.size();
        }
    return best;
}
void ring(int32_t* out, int rows, int growth, int most_halo) {
    for (int j = 0; j < RINGS; ++j) out[j] = j * growth <= most_halo ? rows + j * growth : -1;
}
}  // namespace

extern "C" {

// ------------------------------------------------------------------------------ for the tests
void host_runtime_limit(size_t bytes) { g_limit = bytes; }
size_t host_runtime_used() { return g_used; }
void host_runtime_growth(int sampled, int all) {
    g_sample_growth = sampled;
    g_growth = all;
}
// tiles that begin before `rows` have another growth among all tiles
void host_runtime_region(int rows, int growth) {
    g_region = rows;
    g_region_growth = growth;
}
void host_runtime_cost(const char* kernel_prefix, double us) { g_cost[kernel_prefix] = us; }
int host_runtime_captures() { return g_captures; }
// the launches since the last call, a name a line
const char* host_runtime_log() {
    g_text.clear();
    for (auto& n : g_log) g_text += n + "\n";
    g_log.clear();
    return g_text.c_str();
}

// ------------------------------------------------------------------------------ the runtime
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    int status = 0;
    char* text = abi::__cxa_demangle(name, nullptr, nullptr, &status);
    std::string s = status == 0 ? text : name;
    std::free(text);
    if (s.rfind("void ", 0) == 0) s.erase(0, 5);
    for (const char* space : {"kpmx::", "(anonymous namespace)::"})
        if (s.rfind(space, 0) == 0) s.erase(0, std::strlen(space));
    g_kernels[host] = s.substr(0, s.find_first_of("<("));
}

static struct {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
} g_call;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    g_call = {grid, block, shared, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
    *grid = g_call.grid;
    *block = g_call.block;
    *shared = g_call.shared;
    *stream = g_call.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t) {
    const std::string& name = g_kernels[f];
    (g_capturing ? g_captured : g_log).push_back(name);
    g_clock += cost(name);
    if (name == "k_chain_sample") {  // (matrix, {heights[8], capacity, bits}, out): 32 tiles a height
        struct Heights {
            int rows[8], capacity, bits;
        };
        const auto* h = static_cast<const Heights*>(args[1]);
        auto* out = *static_cast<int32_t**>(args[2]);
        for (unsigned b = 0; b < grid.x; ++b)
            ring(out + b * RINGS, h->rows[b / 32], g_sample_growth, h->capacity - h->rows[b / 32]);
    }
    if (name == "k_chain_rings") {  // (matrix, tile_begin, steps, bits, ring, ext, ext_stride): a tile a block
        const auto* begin = *static_cast<const int32_t* const*>(args[1]);
        auto* out = *static_cast<int32_t**>(args[4]);
        const int64_t halo = *static_cast<const int64_t*>(args[6]);
        for (unsigned t = 0; t < grid.x; ++t)
            ring(out + t * RINGS, begin[t + 1] - begin[t], begin[t] < g_region ? g_region_growth : g_growth, (int)halo);
    }
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* blocks, const void*, int, size_t) {
    *blocks = 2;
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t bytes) {
    *p = nullptr;
    if (g_used + bytes > g_limit) return hipErrorOutOfMemory;
    *p = std::calloc(1, bytes);
    g_memory[*p] = bytes;
    g_used += bytes;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    auto it = g_memory.find(p);
    if (it == g_memory.end()) return p ? hipErrorInvalidValue : hipSuccess;
    g_used -= it->second;
    g_memory.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free_bytes, size_t* total) {
    *total = g_limit;
    *free_bytes = g_limit > g_used ? g_limit - g_used : 0;
    return hipSuccess;
}
hipError_t hipMemcpy(void* to, const void* from, size_t bytes, hipMemcpyKind) {
    std::memcpy(to, from, bytes);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* to, const void* from, size_t bytes, hipMemcpyKind kind, hipStream_t) {
    return g_capturing ? hipSuccess : hipMemcpy(to, from, bytes, kind);
}
hipError_t hipMemcpy2DAsync(void* to, size_t to_pitch, const void* from, size_t from_pitch, size_t width, size_t height,
                            hipMemcpyKind kind, hipStream_t) {
    for (size_t r = 0; r < height; ++r)
        (void)hipMemcpy(static_cast<char*>(to) + r * to_pitch, static_cast<const char*>(from) + r * from_pitch, width, kind);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int value, size_t bytes, hipStream_t) {
    std::memset(p, value, bytes);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static void* memory = std::calloc(1, (size_t)64 << 20);
    *p = memory;
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int* count) {
    *count = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* device) {
    *device = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {  // a macro: the versioned name
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "an error of the host runtime"; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    g_capturing = true;
    g_captured.clear();
    ++g_captures;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* graph) {
    g_capturing = false;
    g_graphs.push_back(g_captured);
    *graph = reinterpret_cast<hipGraph_t>(g_graphs.size());
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* exec, hipGraph_t graph, hipGraphNode_t*, char*, size_t) {
    *exec = reinterpret_cast<hipGraphExec_t>(graph);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t exec, hipStream_t) {
    for (auto& n : g_graphs[reinterpret_cast<size_t>(exec) - 1]) g_log.push_back(n);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

hipError_t hipEventCreate(hipEvent_t* e) {
    *e = reinterpret_cast<hipEvent_t>(new double(0));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete reinterpret_cast<double*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    *reinterpret_cast<double*>(e) = g_clock;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
    *ms = (float)((*reinterpret_cast<double*>(b) - *reinterpret_cast<double*>(a)) * 1e-3);
    return hipSuccess;
}

}  // extern "C"
