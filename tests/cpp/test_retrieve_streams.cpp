// The PerBit retrieve's use of streams, without a GPU: this program defines the
// HIP calls that the library makes (its own symbols come before libamdhip64's)
// over host memory, with streams as queues that run only when something waits
// for them and a copy that can be told to fail.
//   - a level maximum set on another stream is waited for
//   - no copy is left on the stream after a retrieve that failed
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "prodm_mdr.h"

namespace {
struct Stream {
    std::vector<std::function<void()>> ops;
    size_t done = 0;
};
struct Event {
    Stream *s = nullptr;
    size_t upto = 0;
};
std::map<void *, Stream> streams;
std::map<void *, size_t> blocks;              // device allocations
std::map<const void *, std::string> &kernels() {  // by host address; the library registers them before main's statics
    static std::map<const void *, std::string> m;
    return m;
}
int fail_copy = 0;                            // counts down: the copy that makes it 0 fails

Stream &of(hipStream_t s) { return streams[s]; }
void run(Stream &s, size_t upto) {
    while (s.done < upto) s.ops[s.done++]();
}
size_t pending() {
    size_t n = 0;
    for (auto &s : streams) n += s.second.ops.size() - s.second.done;
    return n;
}
struct Launch {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
} last_launch;
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    *p = calloc(n ? n : 1, 1);
    blocks[*p] = n;
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) { blocks.erase(p); free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
    if (fail_copy && --fail_copy == 0) return hipErrorUnknown;
    of(st).ops.push_back([=] { memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { run(of(s), of(s).ops.size()); return hipSuccess; }
hipError_t hipDeviceSynchronize() {
    for (auto &s : streams) run(s.second, s.second.ops.size());
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = reinterpret_cast<hipStream_t>(new char); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *st) { *st = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = reinterpret_cast<hipEvent_t>(new Event); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<Event *>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    *reinterpret_cast<Event *>(e) = Event{&of(s), of(s).ops.size()};
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    const Event v = *reinterpret_cast<Event *>(e);
    if (v.s) run(*v.s, v.upto);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    const Event v = *reinterpret_cast<Event *>(e);
    if (v.s && v.s != &of(s)) of(s).ops.push_back([v] { run(*v.s, v.upto); });
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetSymbolAddress(void **p, const void *) { static char table[1024]; *p = table; return hipSuccess; }

void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) {
    kernels()[f] = name;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) { last_launch = Launch{g, b, m, s}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, hipStream_t *s) {
    *g = last_launch.grid; *b = last_launch.block; *m = last_launch.shmem; *s = last_launch.stream;
    return hipSuccess;
}
// of the kernels only the fills do anything: k_fill<U>(U *, uint64_t, U)
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t s) {
    const std::string &name = kernels()[f];
    if (name.find("6k_fill") == std::string::npos) { of(s).ops.push_back([] {}); return hipSuccess; }
    const size_t u = name.find("6k_fillIj") != std::string::npos ? 4 : 8;
    char *dst = *static_cast<char **>(args[0]);
    const uint64_t count = *static_cast<uint64_t *>(args[1]);
    uint64_t value = 0;
    memcpy(&value, args[2], u);
    of(s).ops.push_back([=] { for (uint64_t i = 0; i < count; i++) memcpy(dst + i * u, &value, u); });
    return hipSuccess;
}
}

#define CHECK(c) \
    do { \
        if (!(c)) { printf("FAILED %s:%d: %s (%s)\n", __FILE__, __LINE__, #c, prodm_last_error()); return 1; } \
    } while (0)

static hipStream_t stream(int i) { return reinterpret_cast<hipStream_t>(uintptr_t(0x1000 + i)); }

// 3 nodes, one level: level 0 holds +1, -1 and level 1 holds 0 in their first plane
static int small_plan(prodm_mdr_plan **p, int nb) {
    const uint32_t dims[1] = {3};
    const uint64_t w0 = 0xd, zero = 0;  // bits 1, sign 0, 1, sign 1
    CHECK(prodm_mdr_plan_create(p, dims, 1, 1, nb, PRODM_F32, PRODM_ENC_PERBIT) == 0);
    for (int l = 0; l < 2; l++)
        for (int i = 0; i < nb; i++)
            CHECK(prodm_mdr_load_plane_stream(*p, l, i, reinterpret_cast<const uint8_t *>(l || i ? &zero : &w0), 8, stream(0)) == 0);
    return 0;
}

static int maxima_of_other_streams() {
    prodm_mdr_plan *p = nullptr;
    CHECK(small_plan(&p, 1) == 0);
    // level 0's maximum on one stream, level 1's on another, the retrieve on a third
    CHECK(prodm_mdr_set_level_max(p, 0, 3.0, stream(0)) == 0);
    CHECK(prodm_mdr_set_level_max(p, 1, 1.0, stream(1)) == 0);
    const uint8_t k[2] = {1, 1};
    float out[3];
    CHECK(prodm_mdr_retrieve(p, k, out, stream(2)) == 0);
    (void)hipStreamSynchronize(stream(2));
    void *c = nullptr;
    CHECK(prodm_mdr_level_coefficients(p, 0, &c) == 0);
    const float *v = static_cast<const float *>(c);
    printf("level 0: %g %g\n", v[0], v[1]);
    CHECK(v[0] == 2.0f && v[1] == -2.0f);
    prodm_mdr_plan_destroy(p);
    return 0;
}

// copies of a retrieve that fails one after the other, then one that does not
static int failed_copies(const uint32_t n, int L, int nb, int copies) {
    prodm_mdr_plan *p = nullptr;
    if (L) {
        CHECK(small_plan(&p, nb) == 0);
    } else {
        CHECK(prodm_mdr_plan_create(&p, &n, 1, 0, nb, PRODM_F32, PRODM_ENC_PERBIT) == 0);
        std::vector<uint64_t> zeros((n + 63) / 64);
        for (int i = 0; i < nb; i++)
            CHECK(prodm_mdr_load_plane_stream(p, 0, i, reinterpret_cast<const uint8_t *>(zeros.data()), zeros.size() * 8, stream(0)) == 0);
    }
    std::vector<float> out(n);
    std::vector<uint8_t> k(L + 1, (uint8_t)nb);
    (void)hipDeviceSynchronize();
    for (int at = 1; at <= copies; at++) {
        fail_copy = at;
        const int rc = prodm_mdr_retrieve(p, k.data(), out.data(), stream(3));
        CHECK(fail_copy == 0 && rc != 0);
        printf("copy %d failed: %zu operations left\n", at, pending());
        CHECK(pending() == 0);
    }
    CHECK(prodm_mdr_retrieve(p, k.data(), out.data(), stream(3)) == 0);
    (void)hipDeviceSynchronize();
    // a stored size past the plane's storage: refused before anything is copied from it
    for (auto &b : blocks)
        if (b.second == 4ull * (L + 1) * nb) {
            static_cast<uint32_t *>(b.first)[nb - 1] = 0xfffffff8u;
            CHECK(prodm_mdr_retrieve(p, k.data(), out.data(), stream(3)) != 0);
            printf("bad size: %zu operations left: %s\n", pending(), prodm_last_error());
            CHECK(pending() == 0);
            break;
        }
    prodm_mdr_plan_destroy(p);
    return 0;
}

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    // errors: small levels (sizes, maxima, a copy and an upload per level), then
    // 2^24 + 1 values, past the pinned staging (sizes, maxima, a copy per plane, an upload)
    const int bad = what == "maxima"   ? maxima_of_other_streams()
                    : what == "errors" ? failed_copies(3, 1, 3, 6) || failed_copies((1u << 24) + 1, 0, 3, 6)
                                       : 1;
    if (!bad) printf("PASSED\n");
    return bad;
}
