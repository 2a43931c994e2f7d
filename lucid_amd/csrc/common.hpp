// Shared host-side plumbing for the gfx950 backend: status/last-error
// handling, the per-device workspace, and small launch helpers.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <mutex>
#include <string>

#include "../../include/lucid_hip.h"

namespace lq {

// Thread-local message of the last failing call (Lucid surfaces typed
// exceptions, lucid/_C/core/Error.h; the C ABI returns a status + message).
std::string& last_error();
int fail(int status, const char* fmt, ...);
int hip_fail(hipError_t e, const char* what);

#define LQ_HIP(expr)                                        \
    do {                                                    \
        hipError_t _e = (expr);                             \
        if (_e != hipSuccess) return lq::hip_fail(_e, #expr); \
    } while (0)

#define LQ_REQUIRE(cond, status, ...)                     \
    do {                                                  \
        if (!(cond)) return lq::fail(status, __VA_ARGS__); \
    } while (0)

#define LQ_CHECK_LAUNCH(name)                                          \
    do {                                                               \
        hipError_t _e = hipGetLastError();                             \
        if (_e != hipSuccess) return lq::hip_fail(_e, "launch " name); \
    } while (0)

// Library-owned scratch for reduction partials, gathered matrices and split-K partial
// sums: one buffer per (device, stream, kind), grown on demand and never shrunk, so calls
// on different streams do not share scratch and calls on one stream are ordered by it.
// A buffer that is outgrown stays allocated while any captured graph exists (its address
// may be baked into the graph).  `fresh`: the bytes of the buffer where nothing has set it up yet, else 0; the caller
// does so on the stream in front of its launch.  What is issued on a stream under capture does not count: a
// replay comes after the eager calls before it, if there ever is one.
int stream_buffer(int kind, size_t nbytes, size_t min_bytes, hipStream_t stream, void** ptr, size_t* fresh);
// The same, but while this thread records a graph a buffer of that graph, kept over the calls that it records on the stream.
int kept_buffer(int kind, size_t nbytes, size_t min_bytes, hipStream_t stream, void** ptr, size_t* fresh);
// kind 0: the general workspace (at least 4 MiB); 1 / 2: stream-K counters / slabs;
// 3: raw accumulators and operand sums of a layer with affine weights; 4: padded copies of ragged GEMM operands;
// 5: the range slots of a dynamic quantization; 6: the codes and qparams of a dynamic Linear's activation;
// 7: the slots of a dynamic quantization in one launch; 8: the rings of an LSTM recurrence
int workspace(size_t nbytes, hipStream_t stream, void** ptr);
// Scratch (kinds 4 to 6 and 8) of one call's launches.  While this thread records a graph it is memory of that graph's own:
// replays may run on any stream, beside each other and beside the stream's eager calls.
int call_buffer(int kind, size_t nbytes, hipStream_t stream, void** ptr);
// Whether this thread records a graph.
bool recording_graph();
// Held by every user of a stream's scratch from before it asks for the buffer until its last launch on it is issued:
// two threads that use one stream would otherwise interleave launches that hand data to each other, or free
// a buffer that the other one has outgrown before it is launched on.  One per (device, stream).
std::unique_lock<std::recursive_mutex> scratch_lock(hipStream_t stream);
// Split-K scratch of one stream, or of the graph being recorded there (the caller holds its scratch_lock): arrival counters (zero between launches: the finisher of a
// tile resets its counter) and slabs for the partial results, whose layout the kernel defines.
struct SkScratch {
    int* counters = nullptr;
    int32_t* slabs = nullptr;
};
int sk_scratch(size_t counters, size_t slab_bytes, hipStream_t st, SkScratch* out);
// lq_sgemm_nt_f32; `large`: 128 x 128 tiles for a small problem too.
int sgemm_nt(const float* a, const float* w, const float* bias, float* out, int M, int N, int K, bool large, hipStream_t st);
// Launches that may be placed at once: the hardware queues of the process, which HIP takes from the environment (four unless
// GPU_MAX_HW_QUEUES says more).  What a kernel whose blocks wait for each other leaves free for launches like it.
int hardware_queues();
// Resolves, for the current device, the address of the static scratch array that
// lq_minmax_noalloc uses (called by lq_init; the entry point does it on first use otherwise).
int minmax_noalloc_init();

// A launch site's once-per-device set-up (the dynamic LDS limit of a kernel is a per-device
// attribute of the function): one bit per device, taken under a mutex, so that the first calls
// of two threads, or on two devices, neither race nor skip it.
struct DeviceOnce {
    std::atomic<uint32_t> done{0};
    std::mutex mu;
};
template <class F>
int device_once(DeviceOnce& o, F&& setup) {
    int dev = 0;
    LQ_HIP(hipGetDevice(&dev));
    LQ_REQUIRE(dev >= 0 && dev < 32, LQ_ERR_DEVICE, "device index %d out of range", dev);
    const uint32_t bit = 1u << dev;
    if (o.done.load(std::memory_order_acquire) & bit) return LQ_OK;
    std::lock_guard<std::mutex> lock(o.mu);
    if (o.done.load(std::memory_order_relaxed) & bit) return LQ_OK;
    const int rc = setup();
    if (rc == LQ_OK) o.done.fetch_or(bit, std::memory_order_release);
    return rc;
}
// the common case: kernel `fn` may use up to `bytes` of dynamic LDS
inline int allow_dynamic_lds(DeviceOnce& o, const void* fn, int bytes) {
    return device_once(o, [&]() -> int {
        LQ_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
        return LQ_OK;
    });
}

inline hipStream_t as_stream(lq_stream s) { return reinterpret_cast<hipStream_t>(s); }

// The barrier of a block for what is in LDS.  __syncthreads waits for every memory operation of the wavefront first: loads that
// were requested early, to arrive under the work on both sides of the barrier, would have to arrive before it.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// floor(n / d) for n < 2^31: one multiplication by ceil(2^(31 + l) / d), 2^(l-1) < d <= 2^l
struct FastDiv {
    unsigned d, m;
    int shift;
    explicit FastDiv(unsigned div) : d(div), m(0), shift(31) {
        int l = 0;
        while ((1ull << l) < div) ++l;
        shift = 31 + l;
        m = unsigned(((1ull << shift) + div - 1) / div);
    }
    __device__ __forceinline__ unsigned operator()(unsigned n) const { return unsigned((uint64_t(n) * m) >> shift); }
};

__host__ __device__ inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// GELU in its erf form, 0.5 x (1 + erf(x / sqrt 2)) (lucid/nn/functional/activations.py:219), erf by Abramowitz & Stegun
// 7.1.26, |error| <= 1.5e-7: with t = 1 / (1 + 0.3275911 |x| / sqrt 2), 1 - erf(|x| / sqrt 2) is P(t) e^(-x^2 / 2), so that
// the value is 0.5 x + |x| (0.5 - 0.5 P(t) e^(-x^2 / 2)).  The constants carry the halves and the 1 / sqrt 2: 13 instructions,
// two of them v_rcp_f32 and v_exp_f32, where erf on its own and the product around it take 16.  Within 1e-6 of the exactly
// rounded value for every x; x or 0 (from -0.5 |x| + 0.5 |x|) beyond |x| = 5.6; +inf gives +inf, -inf and a NaN give NaN.
__device__ __forceinline__ float gelu_erf(float x) {
    const float z = __builtin_fabsf(x);
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3275911f * 0.70710678118654752440f, z, 1.0f));
    float p = __builtin_fmaf(0.5f * 1.061405429f, t, 0.5f * -1.453152027f);
    p = __builtin_fmaf(p, t, 0.5f * 1.421413741f);
    p = __builtin_fmaf(p, t, 0.5f * -0.284496736f);
    p = __builtin_fmaf(p, t, 0.5f * 0.254829592f);
    p = p * t;
    const float e = __builtin_amdgcn_exp2f((x * x) * (0.5f * -1.4426950408889634f));
    return __builtin_fmaf(z, __builtin_fmaf(-p, e, 0.5f), 0.5f * x);
}

}  // namespace lq
