// fake_hip.cpp -- a HIP runtime on host memory for tests of the library's
// host side without a GPU: allocations come from the heap up to a limit the
// test sets, launches are recorded (kernel name, workgroups, pointers, rows)
// and run nothing, but mark their last pointer's first bytes; a compile
// gives a code object at once.  Linked with the library's host sources in
// the place of libamdhip64 and libhiprtc.
#include <hip/hip_runtime.h>
#include <hip/hiprtc.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "hb_internal.h"

namespace {
struct Launch {
    std::string name;
    uint32_t groups, m;
    std::vector<void*> ptrs;
};
std::map<void*, size_t> blocks;
uint64_t in_use = 0, limit = ~0ull, tries = 0, failing_reads = 0;
std::vector<Launch> launches;
float clock_ms = 0;  // 10 us a launch
struct Fn {
    std::string name;
};
std::map<void*, float> events;
}  // namespace

extern "C" {

// ---- what a test reads and sets ----
void fake_limit(uint64_t bytes) { limit = bytes; }
// The next n copies to the host fail.
void fake_fail_reads(uint64_t n) { failing_reads = n; }
uint64_t fake_in_use(void) { return in_use; }
uint64_t fake_malloc_tries(void) { return tries; }
void fake_forget(void) { launches.clear(); }
uint32_t fake_launches(void) { return (uint32_t)launches.size(); }
const char* fake_launch_name(uint32_t i) { return launches[i].name.c_str(); }
uint32_t fake_launch_rows(uint32_t i) { return launches[i].m; }
// The bytes of the allocation that pointer j of launch i lies in, from that
// pointer on; 0 for a pointer in none.
uint64_t fake_launch_span(uint32_t i, uint32_t j) {
    const char* p = (const char*)launches[i].ptrs[j];
    auto it = blocks.upper_bound((void*)p);
    if (it == blocks.begin()) return 0;
    --it;
    const char* b = (const char*)it->first;
    return p < b + it->second ? (uint64_t)(b + it->second - p) : 0;
}

// ---- memory ----
hipError_t hipMalloc(void** p, size_t n) {
    tries++;
    if (in_use + n > limit) return hipErrorOutOfMemory;
    *p = calloc(1, n);
    if (!*p) return hipErrorOutOfMemory;
    blocks[*p] = n;
    in_use += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    auto it = blocks.find(p);
    if (it == blocks.end()) return hipErrorInvalidValue;
    in_use -= it->second;
    blocks.erase(it);
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t) {
    if (kind == hipMemcpyDeviceToHost && failing_reads) {
        failing_reads--;
        return hipErrorUnknown;
    }
    memcpy(d, s, n);
    return hipSuccess;
}

// ---- device, stream, events, graphs ----
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    memset(p, 0, sizeof *p);
    strcpy(p->name, "host");
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipRuntimeGetVersion(int* v) {
    *v = HIP_VERSION;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = (hipStream_t)1;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = (hipEvent_t) new char;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    events.erase(e);
    delete (char*)e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    events[e] = clock_ms;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
    *ms = events[b] - events[a];
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    *g = (hipGraph_t)1;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *x = (hipGraphExec_t)1;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }

// ---- modules ----
hipError_t hipModuleLoadData(hipModule_t* m, const void*) {
    *m = (hipModule_t)1;
    return hipSuccess;
}
hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* name) {
    *f = (hipFunction_t) new Fn{name};
    return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned, unsigned, unsigned, unsigned, unsigned,
                                 unsigned, hipStream_t, void** args, void**) {
    Launch l{((Fn*)f)->name, gx, 0, {}};
    clock_ms += 0.01f;
    if (l.name == "fill_zero") {
        memset(*(void**)args[0], 0, *(uint64_t*)args[1]);
    } else {
        // Kernel arguments: n pointers, then the rows.  A GEMM has 6, its
        // split's second kernel and the row kernels 3, the SwiGLU rows 2.
        const uint32_t n = l.name.rfind("gemm_splitk", 0) == 0 ? 3
                           : l.name.rfind("gemm_", 0) == 0     ? 6
                           : l.name.rfind("swiglu_", 0) == 0   ? 2
                                                               : 3;
        for (uint32_t i = 0; i < n; i++) l.ptrs.push_back(*(void**)args[i]);
        l.m = *(uint32_t*)args[n];
        const uint32_t y = n == 6 ? 3 : n - 1;
        if (l.ptrs[y]) *(uint16_t*)l.ptrs[y] = 0x3f80;
    }
    launches.push_back(l);
    if (launches.size() > 4096) launches.erase(launches.begin(), launches.begin() + 2048);
    return hipSuccess;
}

// ---- hiprtc ----
hiprtcResult hiprtcCreateProgram(hiprtcProgram* p, const char*, const char*, int, const char* const*,
                                 const char* const*) {
    *p = (hiprtcProgram)1;
    return HIPRTC_SUCCESS;
}
hiprtcResult hiprtcCompileProgram(hiprtcProgram, int, const char* const*) { return HIPRTC_SUCCESS; }
hiprtcResult hiprtcDestroyProgram(hiprtcProgram*) { return HIPRTC_SUCCESS; }
hiprtcResult hiprtcGetCodeSize(hiprtcProgram, size_t* n) {
    *n = 4;
    return HIPRTC_SUCCESS;
}
hiprtcResult hiprtcGetCode(hiprtcProgram, char* c) {
    memcpy(c, "code", 4);
    return HIPRTC_SUCCESS;
}
hiprtcResult hiprtcGetProgramLogSize(hiprtcProgram, size_t* n) {
    *n = 0;
    return HIPRTC_SUCCESS;
}
hiprtcResult hiprtcGetProgramLog(hiprtcProgram, char*) { return HIPRTC_SUCCESS; }
const char* hiprtcGetErrorString(hiprtcResult) { return "error"; }

int hb_moe_experts_run_static(hb_gpu*, const int32_t*, int32_t, int32_t, hb_range, hb_range, hb_range, hb_range,
                              hb_range, uint32_t) {
    return hb::fail(HB_ERR_UNSUPPORTED, "no static scratch on the host");
}

}  // extern "C"

namespace hb {
int static_scratch(int, void** out) {
    *out = nullptr;
    return HB_OK;
}
}  // namespace hb
