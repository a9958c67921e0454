// host_stub.cpp -- a HIP runtime and kernel launches that only keep a record,
// for tests of libq35mm's host code (runtime.cpp) on a machine without a GPU:
// which launches a call queues, on which scratch, and what it allocates,
// frees and waits for.  Device memory is host memory that nothing computes
// on.  Linked with runtime.cpp and safetensors.cpp into one library of the
// same C ABI, plus the stub_* controls below.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <string>
#include <utility>

#include "q35mm_internal.h"

#define STUB_API extern "C" __attribute__((visibility("default")))

namespace {
std::string g_log;
std::set<void *> g_capturing;   // streams under capture
size_t g_fail_from = SIZE_MAX;  // allocations of at least this size fail
hipError_t g_last = hipSuccess;
hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;   // the calling thread's

template <typename... A>
hipError_t note(const char *fmt, A... a) {
    char line[256];
    snprintf(line, sizeof line, fmt, a...);
    g_log += line;
    g_log += '\n';
    return hipSuccess;
}
hipError_t fail(hipError_t e) { return g_last = e; }
}  // namespace

STUB_API const char *stub_log() { return g_log.c_str(); }
STUB_API void stub_clear() { g_log.clear(); }
STUB_API void stub_capture(void *stream, int on) {
    if (on)
        g_capturing.insert(stream);
    else
        g_capturing.erase(stream);
}
STUB_API void stub_fail_malloc(size_t from) { g_fail_from = from; }

// ---- HIP --------------------------------------------------------------
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {   // a macro: the versioned name
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub"; }
// the last error stays until it is read, as a failed call's does: a launch
// that follows one reports it
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipMalloc(void **p, size_t n) {
    // while any stream is captured, a thread in the global mode may not allocate
    if (!g_capturing.empty() && g_mode == hipStreamCaptureModeGlobal) return fail(hipErrorStreamCaptureUnsupported);
    if (n >= g_fail_from) return fail(hipErrorOutOfMemory);
    *p = aligned_alloc(256, (n + 255) & ~(size_t)255);
    return note("malloc %p %zu", *p, n);
}
hipError_t hipFree(void *p) {
    note("free %p", p);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = aligned_alloc(256, (n + 255) & ~(size_t)255), hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemset(void *d, int v, size_t n) { return memset(d, v, n), hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) { return std::swap(*m, g_mode), hipSuccess; }
hipError_t hipDeviceSynchronize() { return note("device_sync"); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)malloc(1), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return free((void *)s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
    // the null stream cannot be asked while another stream is captured
    if (!s && !g_capturing.empty()) return fail(hipErrorStreamCaptureImplicit);
    *st = g_capturing.count((void *)s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = nullptr, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }

// ---- launches: one line each, with the scratch they use ----------------
namespace q35mm {
namespace {
template <typename... A>
hipError_t launch(const char *fmt, A... a) {
    note(fmt, a...);
    return hipGetLastError();
}
alignas(256) uint8_t g_noalloc[kNoAllocCntBytes + kNoAllocBytes];
}  // namespace

hipError_t noalloc_setup(int, hipStream_t) { return hipSuccess; }
uint8_t *noalloc_scratch(int) { return g_noalloc; }

uint32_t gemv_ctas(uint32_t, uint32_t, uint32_t) { return 1; }
uint32_t gemv_max_contrib(uint32_t, uint32_t, uint32_t) { return 1; }
bool gemv_norm_fits(uint32_t, uint32_t) { return false; }
uint32_t gemv_norm_cols(uint32_t k) { return (k + 31) / 32 * 32; }
bool gemv_rows_shape(uint32_t kb, uint32_t waves) { return kb >= waves && kb <= kGemvRsMaxKb; }
void gemv_rows_plan(const uint32_t *rows, uint32_t n, uint32_t *c) {
    for (uint32_t s = 0; s < n; s++) c[s] = (rows[s] + kSubRows - 1) / kSubRows;
}
bool rmsnorm_bf16_fits(const float *, uint32_t, const float *, uint32_t) { return true; }
GemmPlan gemm_plan(uint32_t m, uint32_t ntiles, uint32_t, uint32_t, bool narrow) {   // every tile in two K slices
    const uint32_t t = narrow ? kGemmNarrowMaxM : kGemmTile, mt = (m + t - 1) / t;
    return {narrow, mt, ntiles, 0, 2, mt * ntiles};
}
uint32_t batch_tile(uint32_t m) { return m <= 16 ? 16 : 32; }
size_t batch_act_bytes(uint32_t m, uint32_t kb) { return (size_t)((m + 31) / 32) * kb * 24576; }
size_t batch_xf_floats(uint32_t m, uint32_t kb) { return (size_t)((m + 31) / 32) * kb * 4; }
size_t batch_ws_floats(uint32_t m, uint32_t nb, uint32_t nr) { return (size_t)nr * m * nb * kBlock; }

hipError_t launch_gemv(const GemvParams &p, hipStream_t s) { return launch("gemv %p m=%u ws=%p cnt=%p", s, p.m, p.ws, p.cnt); }
hipError_t launch_gemv_rows(const GemvParams &p, uint32_t, uint32_t waves, uint32_t, hipStream_t s) {
    return launch("rows %p m=%u nr=%u", s, p.m, waves);
}
hipError_t launch_gemv_pair(const GemvParams &p, bool, uint32_t, hipStream_t s) { return launch("pair %p m=%u y=%p nr=4", s, p.m, p.seg[0].y); }
hipError_t launch_split_act(const float *, uint32_t, uint32_t m, uint32_t, uint32_t, bool, uint32_t, uint8_t *xs, float *xf,
                            hipStream_t s) {
    return launch("split %p m=%u xs=%p xf=%p", s, m, xs, xf);
}
hipError_t launch_gemv_batch(const BatchParams &p, bool, hipStream_t s) {
    return launch("batch %p m=%u xs=%p ws=%p nr=%u", s, p.m, p.xs, p.ws, p.nr);
}
hipError_t launch_batch_swiglu(const BatchParams &p, uint32_t, uint8_t *xs, float *, hipStream_t s) {
    return launch("batch_swiglu %p m=%u xs=%p ws=%p nr=%u", s, p.m, xs, p.ws, p.nr);
}
hipError_t launch_chain(const ChainParams &, hipStream_t s) { return launch("chain %p", s); }
hipError_t launch_act_to_bf16(const float *, const float *, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint16_t *xb,
                              hipStream_t s) {
    return launch("act %p xb=%p", s, xb);
}
hipError_t launch_gemm(const GemmParams &p, hipStream_t s) { return launch("gemm %p m=%u xb=%p ws=%p", s, p.m, p.xb, p.ws); }
hipError_t launch_repack(const uint8_t *, uint32_t, uint32_t, uint32_t, uint32_t, uint8_t *, hipStream_t) { return hipSuccess; }
hipError_t launch_dequant_f32(const Weight &, float *, hipStream_t) { return hipSuccess; }
hipError_t launch_decode_bf16(const Weight &, uint16_t *, hipStream_t) { return hipSuccess; }
hipError_t launch_done_flag(uint32_t *flag, uint32_t v, hipStream_t) { return *flag = v, hipSuccess; }
hipError_t launch_bf16_gemv(const uint16_t *, uint32_t, uint32_t, const float *, float *, hipStream_t) { return hipSuccess; }
hipError_t launch_quantize_f32(const float *, uint32_t, uint32_t, uint8_t *, uint16_t *, float *, hipStream_t) { return hipSuccess; }
hipError_t launch_quantize_bf16(const uint16_t *, uint32_t, uint32_t, uint8_t *, uint16_t *, float *, hipStream_t) { return hipSuccess; }
hipError_t launch_rmsnorm(const float *, uint32_t, const float *, float *y, uint32_t, uint32_t, uint32_t, float, hipStream_t s) {
    return launch("rmsnorm %p y=%p", s, y);
}
hipError_t launch_rmsnorm_bf16(const float *, uint32_t, const float *, uint32_t, uint32_t, float, uint32_t, uint32_t, uint16_t *xb,
                               hipStream_t s) {
    return launch("rmsnorm_bf16 %p xb=%p", s, xb);
}
hipError_t launch_swiglu(const float *, const float *, float *, size_t, hipStream_t s) { return launch("swiglu %p", s); }
hipError_t launch_add_inplace(float *, const float *, size_t, hipStream_t s) { return launch("add %p", s); }
}  // namespace q35mm
