// A HIP runtime on host memory for tests of the library's host code: no kernel runs, copies are
// done at once, and a test can make the next calls of one function fail.  As HIP's, a
// failed call's error stays until hipGetLastError takes it.
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

#include <string>

#include "../gpuropolis_amd/csrc/gpr_internal.h"

static std::string g_fail;
static int g_left = 0;
static hipError_t g_last = hipSuccess;

extern "C" void stub_fail(const char *name, int times) {
    g_fail = name;
    g_left = times;
}
static hipError_t call(const char *name) {
    if (g_fail != name || g_left == 0) return hipSuccess;
    g_left--;
    return g_last = hipErrorOutOfMemory;
}
#define STUB(NAME, ARGS, BODY)                                \
    extern "C" hipError_t NAME ARGS {                         \
        if (const hipError_t e = call(#NAME)) return e;       \
        BODY;                                                 \
        return hipSuccess;                                    \
    }
STUB(hipEventCreate, (hipEvent_t *e), *e = (hipEvent_t)malloc(1))
STUB(hipEventCreateWithFlags, (hipEvent_t *e, unsigned), *e = (hipEvent_t)malloc(1))
STUB(hipEventDestroy, (hipEvent_t e), free(e))
STUB(hipEventElapsedTime, (float *ms, hipEvent_t, hipEvent_t), *ms = 1.0f)
STUB(hipEventRecord, (hipEvent_t, hipStream_t), )
STUB(hipEventSynchronize, (hipEvent_t), )
STUB(hipFree, (void *p), free(p))
STUB(hipGetDeviceCount, (int *n), *n = 1)
STUB(hipGetDevicePropertiesR0600, (hipDeviceProp_tR0600 *p, int), memset(p, 0, sizeof *p); p->multiProcessorCount = 256)
STUB(hipGetSymbolAddress, (void **p, const void *), *p = nullptr)
STUB(hipGraphDestroy, (hipGraph_t), )
STUB(hipGraphExecDestroy, (hipGraphExec_t), )
STUB(hipGraphInstantiate, (hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t), )
STUB(hipGraphLaunch, (hipGraphExec_t, hipStream_t), )
STUB(hipHostFree, (void *p), free(p))
STUB(hipHostMalloc, (void **p, size_t n, unsigned), *p = malloc(n))
STUB(hipMalloc, (void **p, size_t n), *p = malloc(n))
STUB(hipMemcpyAsync, (void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t), memcpy(d, s, n))
STUB(hipMemsetAsync, (void *d, int v, size_t n, hipStream_t), memset(d, v, n))
STUB(hipSetDevice, (int), )
STUB(hipStreamBeginCapture, (hipStream_t, hipStreamCaptureMode), )
STUB(hipStreamCreateWithFlags, (hipStream_t *s, unsigned), *s = (hipStream_t)malloc(1))
STUB(hipStreamDestroy, (hipStream_t s), free(s))
STUB(hipStreamEndCapture, (hipStream_t, hipGraph_t *), )
STUB(hipStreamSynchronize, (hipStream_t), )
STUB(hipStreamWaitEvent, (hipStream_t, hipEvent_t, unsigned), )
extern "C" const char *hipGetErrorString(hipError_t) { return "stub error"; }
extern "C" hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
extern "C" void **__hipRegisterFatBinary(const void *) {
    static void *p;
    return &p;
}
extern "C" void __hipUnregisterFatBinary(void **) {}
extern "C" void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

// the launchers: nothing but the launch's error
#define LAUNCH(NAME, ...) \
    hipError_t NAME(__VA_ARGS__) { return hipGetLastError(); }
LAUNCH(gpr_launch_mh_config_wave, const GprMHArgs &, int, bool, bool, bool, int, hipStream_t)
LAUNCH(gpr_launch_mh_config_lane, const GprMHArgs &, int, hipStream_t)
LAUNCH(gpr_launch_mh_ref_lane, const GprMHArgs &, int, hipStream_t)
LAUNCH(gpr_launch_mh_ref_wave, const GprMHArgs &, int, int, hipStream_t)
LAUNCH(gpr_launch_eval_wave, const GprEvalArgs &, hipStream_t)
LAUNCH(gpr_launch_dataset_prep, const float *, int, int, int, int, GprDataset *, float *, hipStream_t)
LAUNCH(gpr_launch_eval_lane, const GprEvalArgs &, hipStream_t)
// a checked gradient call finds the first tape's length as its faults, after a while in which
// other threads' calls may come between
hipError_t gpr_launch_grad_wave(const GprEvalArgs &a, hipStream_t) {
    if (a.faults) {
        usleep(100);
        *a.faults |= a.len[0];
        usleep(100);
    }
    return hipGetLastError();
}
LAUNCH(gpr_launch_init_config, const GprMHArgs &, int, hipStream_t)
LAUNCH(gpr_launch_init_ref, const GprMHArgs &, hipStream_t)
LAUNCH(gpr_launch_resample, const GprResampleArgs &, hipStream_t)
LAUNCH(gpr_launch_resample_quantile, const GprResampleArgs &, hipStream_t)
hipError_t gpr_launch_fill_i32(int *p, int n, int v, hipStream_t) {
    for (int i = 0; i < n; i++) p[i] = v;
    return hipGetLastError();
}
LAUNCH(gpr_launch_fill_logint, hipStream_t)
LAUNCH(gpr_launch_fill_ref_logint, hipStream_t)
LAUNCH(gpr_launch_clock_advance, uint32_t *, uint32_t, hipStream_t)
LAUNCH(gpr_launch_test_ref_decode, const uint8_t *, const float *, int, uint8_t *, float *, int *, hipStream_t)
LAUNCH(gpr_launch_test_draws, const uint32_t *, int, uint64_t, float *, hipStream_t)
