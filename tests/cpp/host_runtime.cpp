// The host side of the library on a HIP runtime that lives in this program: device memory is host memory, and work put on a stream
// is done only when somebody waits for it (the latest moment the real runtime may take). Built and run by
// tests/test_host_runtime_cpu.py; no GPU is involved. The library's references to the runtime bind to this program's functions.
#include <dlfcn.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <deque>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "rmx_common.h"

namespace {
struct Item {
    std::function<void()> work;
    void *event;
};
std::deque<Item> g_queue;                 // the one stream
std::map<const void *, std::string> g_names;
std::string g_fail;                       // the next launch of a kernel of this name fails
hipError_t g_last = hipSuccess;
int g_event_waits = 0;
std::vector<float> g_seen;                // scale of the last sample's channel 0, as every kernel found it
struct { dim3 grid, block; size_t lds; hipStream_t stream; } g_call;

void run_until(void *event) {
    while (!g_queue.empty()) {
        Item it = g_queue.front();
        g_queue.pop_front();
        if (it.work) it.work();
        if (event && it.event == event) return;
    }
}
}  // namespace

extern "C" {
void **__hipRegisterFatBinary(const void *) { static void *m; return &m; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) { g_names[host] = name; }
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) { g_call = {g, b, l, s}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *l, hipStream_t *s) { *g = g_call.grid; *b = g_call.block; *l = g_call.lds; *s = g_call.stream; return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 65536;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) { static char rows[1 << 20]; *p = rows; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = aligned_alloc(256, (n + 255) / 256 * 256); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *) { memset(a, 0, sizeof(*a)); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { run_until(nullptr); return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) { *s = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { g_queue.push_back({nullptr, e}); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { g_event_waits++; run_until(e); return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "refused by the test"; }
hipError_t hipGetLastError(void) { hipError_t e = g_last; g_last = hipSuccess; return e; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    g_queue.push_back({[=] { memcpy(d, s, n); }, nullptr});
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3, dim3, void **args, size_t, hipStream_t) {
    const std::string name = g_names[fn];
    if (!g_fail.empty() && name.find(g_fail) != std::string::npos) {
        g_fail.clear();
        return g_last = hipErrorLaunchFailure;
    }
    if (name.find("rmx_table_upload_kernel") != std::string::npos) {
        const void *s = *(const void **)args[0];
        void *d = *(void **)args[1];
        const int n16 = *(const int *)args[2];
        g_queue.push_back({[=] { memcpy(d, s, (size_t)n16 * 16); }, nullptr});
    } else {
        const RmxKArgs a = *(const RmxKArgs *)args[0];
        g_queue.push_back({[=] { g_seen.push_back(a.compact ? a.shared.scale[0] : a.table[a.n - 1].scale[0]); }, nullptr});
    }
    return hipSuccess;
}
}

#define API(name) auto name = (decltype(&::name))dlsym(lib, #name)
#define REQUIRE(c)                                                                        \
    do {                                                                                  \
        if (!(c)) {                                                                       \
            fprintf(stderr, "line %d: %s (%s)\n", __LINE__, #c, rmx_last_error()); \
            return 1;                                                                     \
        }                                                                                 \
    } while (0)

int main(int argc, char **argv) {
    void *lib = dlopen(argv[1], RTLD_NOW);
    if (!lib) return fprintf(stderr, "%s\n", dlerror()), 2;
    const std::string what = argv[2];
    API(rmx_ctx_create); API(rmx_ctx_sync); API(rmx_last_error); API(rmx_op_launch); API(rmx_op_destroy); API(rmx_ctx_destroy);
    API(rmx_create_crop_mirror_normalize); API(rmx_update_crop_mirror_normalize);
    constexpr uint32_t N = 5;
    rmx_ctx *ctx;
    REQUIRE(rmx_ctx_create(0, nullptr, 0, &ctx) == RMX_OK);
    const rmx_tensor_desc sd = {N, 16, 16, 3, RMX_NHWC, RMX_UINT8}, dd = {N, 16, 16, 3, RMX_NCHW, RMX_FP32};
    rmx_op *op;
    REQUIRE(rmx_create_crop_mirror_normalize(ctx, &sd, &dd, RMX_ROI_XYWH, &op) == RMX_OK);
    static char src[N * 768], dst[N * 768 * 4] __attribute__((aligned(16)));
    uint32_t roi[N * 4], mirror[N] = {1};
    float scale[N * 3], bias[N * 3] = {};
    for (uint32_t i = 0; i < N; i++) roi[4 * i] = roi[4 * i + 1] = 0, roi[4 * i + 2] = roi[4 * i + 3] = 16;
    // a value per update; scales that differ between samples go through the table, one for all through the kernel's arguments
    auto update = [&](float v, bool table) {
        for (uint32_t i = 0; i < N * 3; i++) scale[i] = table && i < 3 ? -1.0f : v;
        return rmx_update_crop_mirror_normalize(op, roi, scale, bias, mirror);
    };
    if (what == "ring") {  // updates and launches without a wait: every launch reads the rows of its own update
        for (int i = 0; i < 53; i++) {
            REQUIRE(update((float)i, i % 7 != 3) == RMX_OK);
            REQUIRE(rmx_op_launch(op, src, dst) == RMX_OK);
        }
        REQUIRE(g_event_waits >= 4);  // (the ring came round several times)
        REQUIRE(rmx_ctx_sync(ctx) == RMX_OK);
        REQUIRE(g_seen.size() == 53);
        for (int i = 0; i < 53; i++) REQUIRE(g_seen[i] == (float)i);
    } else if (what == "failed upload") {  // an update whose upload fails leaves an op that cannot be launched
        for (int before = 0; before < 3; before++) {  // as the first one, behind one in the arguments, behind one in the table
            if (before) REQUIRE(update(1.0f, before == 2) == RMX_OK);
            g_fail = "rmx_table_upload_kernel";
            REQUIRE(update(2.0f, true) == RMX_ERR_HIP);
            REQUIRE(rmx_op_launch(op, src, dst) == RMX_ERR_INVALID);
            REQUIRE(rmx_ctx_sync(ctx) == RMX_OK && g_seen.empty());
        }
        REQUIRE(update(3.0f, true) == RMX_OK);
        REQUIRE(rmx_op_launch(op, src, dst) == RMX_OK);
        REQUIRE(rmx_ctx_sync(ctx) == RMX_OK && g_seen.size() == 1 && g_seen[0] == 3.0f);
    } else if (what == "failed launch") {  // a launch that fails says so once: the next update finds no error of its own
        REQUIRE(update(1.0f, true) == RMX_OK);
        g_fail = "rmx_cmn_kernel";
        REQUIRE(rmx_op_launch(op, src, dst) == RMX_ERR_HIP);
        REQUIRE(g_last == hipSuccess);
        REQUIRE(update(2.0f, true) == RMX_OK);
        REQUIRE(rmx_op_launch(op, src, dst) == RMX_OK);
        REQUIRE(rmx_ctx_sync(ctx) == RMX_OK && g_seen.size() == 1 && g_seen[0] == 2.0f);
    } else {
        return 2;
    }
    REQUIRE(rmx_op_destroy(op) == RMX_OK && rmx_ctx_destroy(ctx) == RMX_OK);
    return 0;
}
