// Failure handling of scene updates on the CPU: scene_set_masks() and write_blocks() over a test double of the HIP
// runtime (allocations from the heap, copies by memcpy, kernels not run) whose n-th call fails, for every n.
// After each failure the device descriptor and the host copy must name live buffers only, and every live buffer must be
// owned by the scene.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "rt_internal.h"

namespace {
std::map<void *, size_t> live;
int calls = 0, fail_at = 0, mallocs = 0;  // fail_at 0: none
bool step() { return ++calls == fail_at; }
bool is_live(const void *p) { return live.count(const_cast<void *>(p)) != 0; }
void *take(size_t n) {
    void *p = std::calloc(1, n ? n : 1);
    live[p] = n;
    return p;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    mallocs++;
    if (step()) { *p = nullptr; return hipErrorOutOfMemory; }
    *p = take(n);
    return hipSuccess;
}
// (memory stays with the process, so no later allocation has a freed one's address)
hipError_t hipFree(void *p) { return !p || live.erase(p) ? hipSuccess : hipErrorInvalidValue; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    if (step()) return hipErrorUnknown;
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    if (step()) return hipErrorUnknown;
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return step() ? hipErrorUnknown : hipSuccess; }
static hipError_t last = hipSuccess;
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
    return last = step() ? hipErrorLaunchFailure : hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "injected"; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 64; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
}

namespace {
constexpr uint32_t P = 5, NN4 = 2;

// A scene of five patches: a root with three records and one node of two
struct Fixture {
    rt::Scene S;
    Fixture() {
        live.clear();
        DevScene &h = S.h;
        h.P = h.nleaf = P;
        h.nnode4 = NN4;
        h.depth4 = 2;
        auto own = [&](size_t n) { void *p = take(n); S.own.push_back(p); return p; };
        h.type = (uint32_t *)own(4 * P);
        h.rec = (float4 *)own(64 * P);
        float4 *n4 = (float4 *)own(128 * NN4);
        h.node4 = n4;
        h.blk = (uint4 *)own(64 * (NN4 + P) + 64);
        S.d = (DevScene *)take(sizeof(DevScene));
        std::memcpy((void *)S.d, &h, sizeof(h));
    }
    ~Fixture() { rt::scene_free(S); }
    bool sound(const char *what) const {
        const DevScene *views[2] = {&S.h, S.d};
        bool ok = true;
        for (const DevScene *v : views) {
            if (!is_live(v->rec) || (v->mdesc && !is_live(v->mdesc)) || (v->blk && !is_live(v->blk))) {
                std::printf("%s, call %d: the %s descriptor names a freed buffer\n", what, fail_at,
                            v == S.d ? "device" : "host");
                ok = false;
            }
        }
        size_t owned = S.own.size() + 1;
        if (live.size() != owned) {
            std::printf("%s, call %d: %zu live buffers, %zu owned\n", what, fail_at, live.size(), owned);
            ok = false;
        }
        return ok;
    }
};

int set_masks(rt::Scene &S) {
    const uint8_t tex[4] = {1, 0, 1, 0};
    const uint32_t size[2] = {2, 2};
    const int32_t id[P] = {0, -1, 0, -1, 0};
    return rt::scene_set_masks(S, 1, tex, size, id, nullptr, nullptr, nullptr);
}

// call with its n-th runtime call failing, on a scene without masks and on one whose masks it replaces
bool run(const char *what, int (*call)(rt::Scene &), bool earlier) {
    for (int n = 1;; n++) {
        Fixture f;
        fail_at = 0;
        bool ok = !earlier || set_masks(f.S) == 0;
        calls = 0;
        fail_at = n;
        const int rc = call(f.S);
        const bool reached = calls >= n;
        ok = f.sound(what) && ok;
        if (reached && rc == 0) { std::printf("%s, call %d: the failure is not reported\n", what, n); ok = false; }
        fail_at = 0;
        last = hipSuccess;
        if (ok && set_masks(f.S)) { std::printf("%s, call %d: the scene cannot be used again\n", what, n); ok = false; }
        if (!ok || !f.sound(what)) return false;
        if (!reached) { std::printf("%s: %d calls\n", what, n - 1); return true; }
    }
}
}  // namespace

int main() {
    const auto blocks = [](rt::Scene &S) {
        return rt::write_blocks(NN4, P, const_cast<float4 *>(S.h.node4), S.h.rec, const_cast<uint4 *>(S.h.blk), false, nullptr);
    };
    bool ok = true;
    for (bool earlier : {false, true}) {
        ok = run("scene_set_masks", set_masks, earlier) && ok;
        ok = run("write_blocks", blocks, earlier) && ok;
    }
    {
        // records, descriptors and texels are new buffers; the block tree is refreshed in place
        Fixture f;
        fail_at = mallocs = 0;
        ok = set_masks(f.S) == 0 && ok;
        if (mallocs != 2) { std::printf("scene_set_masks: %d allocations\n", mallocs); ok = false; }
    }
    std::printf(ok ? "all checks passed\n" : "FAILED\n");
    return ok ? 0 : 1;
}
