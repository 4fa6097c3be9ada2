// The host API over a stub HIP runtime: launches are logged instead of run and
// allocations can be made to fail, so that a test on a machine without a GPU
// sees which kernel a call takes, how its keys are split and what happens when
// the workspace cannot grow.
#include "mxfa_api.cpp"

#include <string>

namespace {
std::string g_log, g_log_out;
int g_malloc_budget = 1 << 30;   // allocations that still succeed
bool g_capturing = false;
hipError_t g_last = hipSuccess;
uintptr_t g_next = (uintptr_t)1 << 40;

hipError_t launched(const std::string &what) {   // as the launchers end: the runtime's last error
    g_log += what + ";";
    return hipGetLastError();
}
}  // namespace

extern "C" {
const char *stub_log() {
    g_log_out.swap(g_log);
    g_log.clear();
    return g_log_out.c_str();
}
void stub_set(int malloc_budget, int capturing) {
    g_malloc_budget = malloc_budget;
    g_capturing = capturing != 0;
}

char __hip_fatbin[1];
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

hipError_t hipMalloc(void **p, size_t bytes) {
    if (g_malloc_budget-- <= 0) return g_last = hipErrorOutOfMemory;
    *p = (void *)g_next;
    g_next += (bytes + 4095) & ~(size_t)4095;
    return hipSuccess;
}
hipError_t hipFree(void *) { return hipSuccess; }
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "stub error"; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
    *s = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) { *p = (void *)((uintptr_t)1 << 39); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipSuccess; }
}  // extern "C"

namespace mxfa {
hipError_t launch_fa_decode(const FaArgs &a, int, hipStream_t) {
    return launched("decode splits=" + std::to_string(a.n_splits) + " chunk=" + std::to_string(a.chunk));
}
hipError_t launch_fa_prefill(const FaArgs &a, int, hipStream_t) {
    return launched("prefill parts=" + std::to_string(a.pf_parts));
}
hipError_t launch_fa_wide(const FaArgs &, int, hipStream_t) { return launched("wide"); }
hipError_t launch_fa_narrow(const FaArgs &, int, hipStream_t) { return launched("narrow"); }
bool fa_narrow_serves(const FaArgs &) { return false; }
hipError_t launch_mask_classify(const FaArgs &, int, uint8_t *, uint8_t *, hipStream_t) { return launched("classify"); }
hipError_t launch_fill_zero(int *, int64_t, hipStream_t) { return launched("fill"); }
hipError_t launch_q8_stage(const Q8StageArgs &, hipStream_t) { return launched("stage"); }
hipError_t launch_set_rows(const SetRowsArgs &, int, hipStream_t) { return launched("set_rows"); }
hipError_t launch_qk_norm_rope(const NormRopeArgs &, int, hipStream_t) { return launched("norm_rope"); }
}  // namespace mxfa
