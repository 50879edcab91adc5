// fft_host.hip -- one transform per launch for calls on host memory: the kernel reads and
// writes host memory itself and reports its own end through a word there.
#include <utility>

#include "fft_lds.h"

namespace ckfft_gpu {

// Waits until this thread's stores have reached host memory, the whole group, then tells.  Each
// wave's fence covers its own stores; the word follows the barrier, and so all of them.
__device__ __forceinline__ void report_done(unsigned* done, unsigned ticket)
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(done, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Input in coherent host memory (the staging slot's) or in this device's own.  Nothing waited for the stream since the last call on this memory, so the runtime may
// leave the system-scope acquire out of the launch.  Up to two waves acquire by a fence at the kernel's start;
// the loads of larger groups go past the caches by themselves, as a fence in every wave, which drops the
// caches' lines of host memory again and again, cost 2 us a call at real 8192 and 4 at 65536 (fence / such
// loads: real inverse 32 8.5 / 11.4 us, 512 9.5 / 11.7, forward 1024 9.8 / 10.1, 8192 17.1 / 15.7, 65536 53 / 50).
struct HostIn {
    static constexpr bool kStaged = false;
    const float2* p;
    __device__ __forceinline__ float2 get(int i) const
    {
        const unsigned long long v = __hip_atomic_load((const unsigned long long*)(p + i), __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_SYSTEM);
        return __builtin_bit_cast(float2, v);
    }
    __device__ __forceinline__ float2 again(int i) const { return get(i); }
    __device__ __forceinline__ void done() const {}
};

// One signal, with the transform body and the points per thread of the batch kernels (so the same
// bits).  Bound by latency: the launch, one round trip over the bus for the reads and one for the
// writes.  The caller waits for `done` to hold `ticket` instead of for the stream, which saves the
// end-of-kernel packet processing and the runtime's completion signal: real 1024 on pageable memory,
// 16.1 -> 9.8 us a call; 32768 32.8 -> 30.8.
template <int LOGN>
struct SignalShape {
    static constexpr int LOGP = LOGN <= 4 ? LOGN : LOGN <= 14 ? 4 : 6;
    static constexpr int T = (1 << LOGN) >> LOGP;
    static constexpr int WG = T > 64 ? T : 64;
    static constexpr bool SPLIT = LOGN >= 15;
};

template <int LOGN, int KIND>
__global__ __launch_bounds__(SignalShape<LOGN>::WG) void fft_signal_kernel(
    const float2* __restrict__ in, float2* __restrict__ out, const float2* __restrict__ tw, unsigned* done,
    unsigned ticket)
{
    using S = SignalShape<LOGN>;
    using SH = LdsShape<LOGN, S::LOGP, S::WG, KIND, S::SPLIT>;
    __shared__ __align__(16) float lds[SH::LDS_WORDS];
    // slots past the first (sizes below 64 threads) compute on the same signal and store nothing
    const bool active = SH::TPW == 1 || (int)threadIdx.x < SH::T;
    if constexpr (S::WG <= 128) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");
        lds_transform<LOGN, S::LOGP, S::WG, KIND, S::SPLIT, false>(in, out, active, tw, lds, threadIdx.x);
    } else {
        lds_transform_io<LOGN, S::LOGP, S::WG, KIND, S::SPLIT, false>(HostIn{in}, MemOut<false>{out}, active, tw, lds,
                                                                      threadIdx.x);
    }
    report_done(done, ticket);
}

using SignalFn = void (*)(const float2*, float2*, const float2*, unsigned*, unsigned);

struct SignalLaunch {
    SignalFn fn;
    int wg;
};

template <int KIND, int... L>
static SignalLaunch signal_launch(int logc, std::integer_sequence<int, L...>)
{
    static constexpr SignalLaunch t[] = {
        SignalLaunch{fft_signal_kernel<L + 2, KIND>, SignalShape<L + 2>::WG}...};
    return t[logc - 2];
}

// The sizes of one workgroup above the closed forms.
bool signal_supported(Kind kind, int log2n)
{
    const int logc = kind == kRealForward || kind == kRealInverse ? log2n - 1 : log2n;
    return logc >= 2 && logc <= kLogMaxLds;
}

hipError_t launch_signal(Kind kind, int log2n, const void* in, void* out, const DeviceTables& tb, hipStream_t stream,
                         unsigned* done, unsigned ticket)
{
    if (!signal_supported(kind, log2n) || log2n > tb.log_pyramid) return hipErrorInvalidValue;
    constexpr std::make_integer_sequence<int, kLogMaxLds - 1> sizes{};
    const SignalLaunch c = kind == kComplexForward   ? signal_launch<kComplexForward>(log2n, sizes)
                           : kind == kComplexInverse ? signal_launch<kComplexInverse>(log2n, sizes)
                           : kind == kRealForward    ? signal_launch<kRealForward>(log2n - 1, sizes)
                                                     : signal_launch<kRealInverse>(log2n - 1, sizes);
    hipLaunchKernelGGL(c.fn, dim3(1), dim3(c.wg), 0, stream, (const float2*)in, (float2*)out, tb.pyramid, done, ticket);
    return hipGetLastError();
}

}  // namespace ckfft_gpu
