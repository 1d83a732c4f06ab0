// sky_math_check.hip — sky_math.hpp against the compiler's IEEE operations
// (libfb_checks.so, loaded by the tests only).  Each function returns a HIP
// error code and the number of arguments with other bits, and one of them.
#include <string.h>

#include "sky_math.hpp"

namespace {

struct Found {
    unsigned long long count;
    unsigned example[2];
};

// (The sign of a zero and a NaN's payload are left to the operations.)
__device__ bool differs(float x, float y) { return x != y && !(isnan(x) && isnan(y)); }
__device__ void note(Found* f, bool bad, float a, float b) {
    const unsigned long long m = __builtin_amdgcn_ballot_w64(bad);
    if (m && (threadIdx.x & 63u) == unsigned(__builtin_ctzll(m))) {
        atomicAdd(&f->count, (unsigned long long)__builtin_popcountll(m));
        f->example[0] = __float_as_uint(a);
        f->example[1] = __float_as_uint(b);
    }
}

constexpr unsigned kBlocks = 4096, kThreads = 256, kPerThread = 4096;
static_assert(4096ull * 256 * 4096 == 1ull << 32);

// Every binary32 value, in kPerThread turns of the grid.
__global__ __launch_bounds__(kThreads) void k_roots(Found* f) {
    for (unsigned j = 0; j < kPerThread; ++j) {
        const float x = __uint_as_float((j * kBlocks + blockIdx.x) * kThreads + threadIdx.x);
        note(f, differs(fbk::sqrt_nr(x), sqrtf(fmaxf(x, 0.0f))), x, 0.0f);
    }
}
__global__ __launch_bounds__(kThreads) void k_reciprocals(Found* f) {
    for (unsigned j = 0; j < kPerThread; ++j) {
        const float b = __uint_as_float((j * kBlocks + blockIdx.x) * kThreads + threadIdx.x);
        const bool in = fabsf(b) > 0x1p-100f && fabsf(b) < 0x1p100f;
        note(f, in && differs(fbk::rcp_nr(b), 1.0f / b), b, 0.0f);
    }
}
// kind 0: div_nr where its ranges hold, 1: div_any, 2: scale_div_any (b / 3 as
// the scale).
__global__ __launch_bounds__(kThreads) void k_quotients(const float* a, const float* b, size_t n,
                                                        int kind, Found* f) {
    const size_t i = size_t(blockIdx.x) * kThreads + threadIdx.x;
    const float x = i < n ? a[i] : 1.0f, y = i < n ? b[i] : 1.0f, want = x / y;
    bool bad;
    if (kind == 1) {
        bad = differs(fbk::div_any(x, y), want);
    } else if (kind == 2) {
        const float s = y / 3.0f;
        const float3 d = fbk::scale_div_any(make_float3(x, x * 0.375f, 1.0f), s, y);
        bad = differs(d.x, x * s / y) || differs(d.y, x * 0.375f * s / y) || differs(d.z, s / y);
    } else {
        const bool in = fabsf(y) > 0x1p-100f && fabsf(y) < 0x1p100f && fabsf(x) >= 0x1p-80f &&
                        fabsf(x) < 0x1p100f && fabsf(want) >= 0x1p-126f && fabsf(want) < 0x1p127f;
        bad = in && differs(fbk::div_nr(x, y), want);
    }
    note(f, bad, x, y);
}

template <typename Launch>
int run(unsigned long long* count, float example[2], Launch launch) {
    Found* d = nullptr;
    hipError_t e = hipMalloc(&d, sizeof(Found));
    if (e != hipSuccess) return int(e);
    Found h = {};
    e = hipMemcpy(d, &h, sizeof(h), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        launch(d);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(&h, d, sizeof(h), hipMemcpyDeviceToHost);
    (void)hipFree(d);
    *count = h.count;
    memcpy(example, h.example, sizeof(h.example));
    return int(e);
}

}  // namespace

extern "C" {

int fbc_sqrt(unsigned long long* count, float example[2]) {
    return run(count, example, [](Found* f) { k_roots<<<kBlocks, kThreads>>>(f); });
}
int fbc_reciprocal(unsigned long long* count, float example[2]) {
    return run(count, example, [](Found* f) { k_reciprocals<<<kBlocks, kThreads>>>(f); });
}
// a, b: n values each in device memory.
int fbc_quotient(const float* a, const float* b, size_t n, int kind, unsigned long long* count,
                 float example[2]) {
    return run(count, example, [=](Found* f) {
        k_quotients<<<unsigned((n + kThreads - 1) / kThreads), kThreads>>>(a, b, n, kind, f);
    });
}

}  // extern "C"
