// scratch_failures: batched products while allocations of the library's scratch fail, on the host alone. The HIP calls that the library's
// host code makes are answered here: an allocation is host memory or, by a schedule, fails as it does on a full card (the
// buffer it was to replace is gone by then), and a launch is looked at instead of made. Whatever the schedule, each matrix of
// a batch is worked out once, every kernel's partial results lie inside memory that is allocated at its launch, and the
// call's two timestamps are each taken once. And the slices of the GEMV on codes follow the device's compute units, and the gated
// norm, of which mtq_plan knows nothing, goes where its lines say. Built with the sanitizers from the library's own host code (metaltile_amd/build.py,
// build_sanitized). Exit code 0 = all of that holds.
#include "qmm_direct_plan.h"
#include "qmv_codes_impl.h"

#include "mtq.h"

#include <dlfcn.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>

namespace {

std::map<char*, size_t> g_live;   // allocated memory
unsigned g_fail = 0;              // bit i: the i-th allocation from here on fails
int g_allocs = 0, g_starts = 0, g_stops = 0, g_bad = 0;
bool g_after_stop = false;
int g_cus = 256;                    // compute units of the device
uint32_t g_slices = 0;              // most slices of K of a matrix on the GEMV on codes
int g_held = 0, g_others = 0;       // launches of the GEMV with its activations in LDS, and of kernels not looked into
std::multiset<const void*> g_out;   // results that the launches so far work out
const char* g_case = "";

void complain(const char* why) {
    if (g_bad++ < 20) fprintf(stderr, "%s, failures %#x: %s\n", g_case, g_fail, why);
}
void inside(const void* p, size_t bytes) {
    auto at = g_live.upper_bound((char*)p);
    if (at == g_live.begin()) return complain("partial results outside the scratch");
    --at;
    if ((char*)p + bytes > at->first + at->second) complain("partial results past the end of the scratch");
}
hipError_t launch(const void* fn, void** args) {
    Dl_info di;
    const char* name = dladdr(fn, &di) && di.dli_sname ? di.dli_sname : "";
    if (g_after_stop) complain("a launch behind the second timestamp");
    if (strstr(name, "qmv_codes_kernel")) {
        const mtq::QmvCodesArgs& a = *(const mtq::QmvCodesArgs*)args[0];
        for (int j = 0; j < 4 && a.first[j] != 0x7FFFFFFFu; j++) {
            g_out.insert(a.out[j]);
            if (a.slices[j] > g_slices) g_slices = a.slices[j];
            if (a.slices[j] > 1) inside(a.part[j], (size_t)a.slices[j] * a.M * a.N[j] * 4);
        }
    } else if (strstr(name, "qmm_direct_kernel") || strstr(name, "qmm_dma_kernel")) {
        const mtq::QmmDArgs& a = *(const mtq::QmmDArgs*)args[0];
        g_out.insert(a.out);
        if (a.ksplit > 1) inside(a.part, (size_t)a.ksplit * a.M * a.N * 4);
        for (uint32_t j = 0; j < a.more.n; j++) {
            g_out.insert(a.more.out[j]);
            if (a.ksplit > 1) inside(a.more.part[j], (size_t)a.ksplit * a.M * a.more.N[j] * 4);
        }
    } else if (strstr(name, "qmv_held_kernel")) {
        g_held++;
    } else if (!strstr(name, "reduce") && !strstr(name, "add")) {
        g_others++;
    }
    return hipSuccess;
}

}  // namespace

extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) { memset(p, 0, sizeof *p); strcpy(p->gcnArchName, "gfx950"); return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = g_cus; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* s) { *p = (void*)s; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)8; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { *s = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { static char events[64]; static int n = 0; *e = (hipEvent_t)(events + n++ % 64); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "out of memory"; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
    if (g_fail >> g_allocs++ & 1u) return hipErrorOutOfMemory;
    *p = aligned_alloc(256, (n + 255) & ~(size_t)255);
    g_live[(char*)*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (!g_live.erase((char*)p)) complain("freed twice");
    free(p);
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3, dim3, void** args, size_t, hipStream_t) { return launch(fn, args); }
hipError_t hipExtLaunchKernel(const void* fn, dim3, dim3, void** args, size_t, hipStream_t, hipEvent_t start, hipEvent_t stop, int) {
    if (start && (!g_out.empty() || g_starts)) complain("the first timestamp behind a launch");
    g_starts += start != nullptr;
    const hipError_t e = launch(fn, args);
    g_stops += stop != nullptr;
    g_after_stop = stop != nullptr;
    return e;
}
}

// One batch on a scratch of `before` bytes or none: a smaller batch goes first.
static void batch(int dtype, int bits, uint32_t G, uint32_t M, uint32_t K, const uint32_t (&N)[3], bool before, unsigned fail) {
    static char operands[4096];
    auto at = [&](int i) { return (void*)(((uintptr_t)operands + 255) / 256 * 256 + 256 * i); };
    const void *w[3] = {at(0), at(1), at(2)}, *s[3] = {at(3), at(4), at(5)}, *b[3] = {at(6), at(7), at(8)};
    void* outs[3] = {at(9), at(10), at(11)};
    g_fail = 0;
    if (mtq_init(0) != MTQ_OK) return complain("mtq_init");
    if (before && mtq_qmm(dtype, bits, G, w[0], s[0], b[0], at(12), outs[0], M, 512, K) != MTQ_OK) complain("the call before");
    g_fail = fail;
    g_allocs = g_starts = g_stops = 0;
    g_after_stop = false;
    g_slices = 0;
    g_held = g_others = 0;
    g_out.clear();
    mtq_timed_begin();
    if (mtq_qmm_batched(dtype, bits, G, 3, w, s, b, at(12), outs, N, M, K) != MTQ_OK) complain("the batch");
    for (void* o : outs)
        if (g_out.count(o) != 1) complain(g_out.count(o) ? "a matrix worked out twice" : "a matrix left out");
    if (g_held || g_others) complain("kernels of others");
    if (g_starts != 1 || g_stops != 1) complain("timestamps");
    g_after_stop = false;
    g_fail = 0;
    mtq_shutdown();
    if (!g_live.empty()) complain("scratch not given back");
}

// Whether the gated norm of a row of `hv` heads of 128 goes with its projection to the GEMV that holds it in LDS.
static void gated(uint32_t N, uint32_t hv, bool held) {
    static char operands[4096];
    auto at = [&](int i) { return (void*)(((uintptr_t)operands + 255) / 256 * 256 + 256 * i); };
    g_fail = 0;
    if (mtq_init(0) != MTQ_OK) return complain("mtq_init");
    g_held = g_others = 0;
    g_after_stop = false;
    if (mtq_gated_rms_norm_qmv(MTQ_BF16, 64, (const float*)at(0), at(1), at(2), (const float*)at(3), at(4), at(5), at(6), at(7), hv, 128, N) != MTQ_OK) complain("gated norm");
    if (g_held != held || (g_others == 0) != held) complain("gated norm on another kernel");
    mtq_shutdown();
}

int main() {
    long n = 0;
    const struct { uint32_t N, hv; bool held; } lines[] = {
        {64, 36, true}, {16384, 36, true}, {2048, 40, false}, {2049, 40, true}, {8192, 40, true}, {4096, 42, true}, {4097, 42, false}, {8192, 47, true}, {2048, 47, false}, {512, 50, true},
        {4096, 56, true}, {4097, 56, false}, {8192, 56, false}, {8193, 56, true}, {2048, 72, false}, {2049, 72, true}, {8193, 72, false}, {512, 16, false},
    };
    for (const auto& l : lines) {
        g_case = "gated norm";
        gated(l.N, l.hv, l.held);
        n++;
    }
    const uint32_t orders[6][3] = {{600, 1100, 300}, {600, 300, 1100}, {1100, 600, 300}, {1100, 300, 600}, {300, 600, 1100}, {300, 1100, 600}};
    for (const auto& N : orders)
        for (int slices : {3, 0})
            for (int before : {0, 1})
                for (unsigned fail = 0; fail < 128; fail++) {
                    g_case = slices ? "GEMV on codes in three slices" : "GEMV on codes";
                    mtq_set_option("qmv.codes_slices", slices);
                    batch(MTQ_BF16, 5, 64, 20, 1152, N, before, fail);
                    g_case = "tiles";
                    mtq_set_option("qmv.codes_slices", 0);
                    batch(MTQ_BF16, 4, 64, 130, 4096, N, before, fail);
                    n += 2;
                }
    // a device of fewer compute units is filled with fewer slices
    g_case = "GEMV on codes, slices";
    const uint32_t N[3] = {1100, 1100, 1100};
    uint32_t slices[2];
    for (int i = 0; i < 2; i++) {
        g_cus = i ? 32 : 256;
        batch(MTQ_BF16, 5, 64, 20, 4736, N, false, 0);
        slices[i] = g_slices;
        n++;
    }
    if (slices[1] == 0 || slices[1] >= slices[0]) complain("as many slices for 32 compute units as for 256");
    printf("scratch_failures: %ld batches, %d violations\n", n, g_bad);
    return g_bad ? 1 : 0;
}
