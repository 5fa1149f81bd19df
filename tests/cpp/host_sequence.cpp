// What the batched form asks of the HIP runtime, without a device: the library's
// own objects linked against a runtime that carries out memory calls on the host,
// runs no kernel and prints every launch, capture and clear in order.  Calls can
// be made to fail.
//
//   host_sequence step_fails N     the N-th launch of step(3) fails, then step(1)
//   host_sequence graph_fails N    the N-th instantiation of step_graph(20) fails, then again
//   host_sequence graph_first N    step_graph(6) with N SPH substeps
//   host_sequence tuning           the wave pass before and after settings are written back
//   host_sequence tune             the tuner
#include <cxxabi.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include <hip/hip_runtime_api.h>

#include "../../include/cwa2d.h"

namespace {
std::map<const void*, std::string> kernels;
std::vector<std::string>* capturing = nullptr;
std::vector<std::string> captured;
hipError_t last = hipSuccess;
int launches_left = 0, instantiations_left = 0;  // the call that reaches 0 fails
bool quiet = true;

bool fails(int& left) { return left > 0 && --left == 0; }

void say(const std::string& s) {
    if (!quiet) std::printf("%s\n", s.c_str());
}
}  // namespace

struct ihipGraph {
    std::vector<std::string> launches;
};
struct hipGraphExec {
    std::vector<std::string> launches;
};

extern "C" {
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*) {
    char* plain = abi::__cxa_demangle(name, nullptr, nullptr, nullptr);
    std::string s = plain ? plain : name;
    std::free(plain);
    if (s.rfind("void ", 0) == 0) s.erase(0, 5);
    s.erase(std::min(s.find_first_of("<("), s.size()));
    kernels[host] = s.substr(s.rfind(':') + 1);
}

static dim3 grid_, block_;
static size_t shared_;
static hipStream_t stream_;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) {
    grid_ = g;
    block_ = b;
    shared_ = s;
    stream_ = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
    *g = grid_;
    *b = block_;
    *s = shared_;
    *st = stream_;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3 b, void**, size_t, hipStream_t) {
    if (fails(launches_left)) {
        say("failed " + kernels[f]);
        return last = hipErrorOutOfMemory;
    }
    const std::string s = kernels[f] + " " + std::to_string(b.x);
    if (capturing) capturing->push_back(s);
    else say("launch " + s);
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "an error"; }

hipError_t hipMalloc(void** p, size_t n) {
    *p = std::calloc(n, 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {
    std::memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) { return hipMemset(p, v, n); }
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    *f = *t = (size_t)1 << 38;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void**, const void*) { return hipErrorInvalidSymbol; }

hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) {
    say("event");
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    say("capture");
    captured.clear();
    capturing = &captured;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    say("captured " + std::to_string(captured.size()));
    *g = new ihipGraph{captured};
    capturing = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
    if (fails(instantiations_left)) {
        say("failed instantiation");
        return hipErrorOutOfMemory;
    }
    *e = new hipGraphExec{g->launches};
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    delete g;
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    delete e;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    say("replay");
    for (const auto& k : e->launches) say("launch " + k);
    return hipSuccess;
}
}  // extern "C"

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    const int nth = argc > 2 ? std::atoi(argv[2]) : 0;
    cwa2d_params p;
    cwa2d_params_reference(&p);
    if (what == "graph_first") p.sph_substeps = nth;
    std::vector<cwa2d_scene> sc(2);
    std::vector<float> xv;
    for (auto& s : sc) {
        s = cwa2d_scene{};
        s.n = 300;
        s.wave_len = 64;
        s.wave_substeps = 2;
        s.mass = 2.5f;
        s.lambda = 0.01f;
        s.wave_model = CWA2D_WAVE_LEAPFROG;
        s.wave_dx = 0.1f;
        for (int i = 0; i < s.n; ++i)
            for (float v : {0.1f + 0.02f * (i % 20), 0.1f + 0.02f * (i / 20), 0.0f, 0.0f})
                xv.push_back(v);
    }
    cwa2d_batch* b = nullptr;
    if (cwa2d_batch_create(&p, 2, sc.data(), xv.data(), nullptr, nullptr, nullptr, &b) != 0) return 1;
    quiet = false;
    const auto done = [](int rc) { std::printf("returned %d\n", rc); };
    if (what == "step_fails") {
        launches_left = nth;
        done(cwa2d_batch_step(b, 1e-3f, 3));
        done(cwa2d_batch_step(b, 1e-3f, 1));
        done(cwa2d_batch_step_graph(b, 1e-3f, 1));
    } else if (what == "graph_fails") {
        instantiations_left = nth;
        done(cwa2d_batch_step_graph(b, 1e-3f, 20));
        done(cwa2d_batch_step_graph(b, 1e-3f, 20));
    } else if (what == "graph_first") {
        done(cwa2d_batch_step_graph(b, 1e-3f, 6));
    } else if (what == "tuning") {
        cwa2d_tuning t;
        done(cwa2d_batch_get_tuning(b, &t));
        std::printf("wave_block %d\n", t.wave_block);
        done(cwa2d_batch_step(b, 1e-3f, 1));
        t.block_density = 512;
        done(cwa2d_batch_set_tuning(b, &t));
        done(cwa2d_batch_step(b, 1e-3f, 1));
    } else if (what == "tune") {
        cwa2d_tuning t;
        done(cwa2d_batch_tune(b, 1e-3f, 3, &t));
    } else {
        return 2;
    }
    quiet = true;
    cwa2d_batch_destroy(b);
    return 0;
}
