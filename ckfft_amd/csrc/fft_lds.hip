// fft_lds.hip -- batch kernels for complex sizes up to 2^15 (real up to 2^16): one
// workgroup holds one or more whole transforms.  The transform body is in fft_lds.h.
#include <utility>

#include "fft_lds.h"

namespace ckfft_gpu {

// ---- the kernel ----------------------------------------------------------------------

// `count` contiguous signals; workgroup slot g handles signal blockIdx.x * TPW + slot.
template <int LOGN, int LOGP, int WG, int KIND, bool SPLIT>
__global__ __launch_bounds__(WG) void fft_lds_kernel(const float2* __restrict__ in, float2* __restrict__ out,
                                                     const float2* __restrict__ tw, int count)
{
    using SH = LdsShape<LOGN, LOGP, WG, KIND, SPLIT>;
    __shared__ __align__(16) float lds[SH::LDS_WORDS];   // 16-byte LDS reads of the pack staging
    // one transform per workgroup: its index is uniform, so the signal's base address
    // stays in scalar registers
    const int tr = SH::TPW == 1 ? 0 : (int)threadIdx.x / SH::T;
    const long long g = (long long)blockIdx.x * SH::TPW + tr;
    const bool active = g < count;
    // slots past the last signal (only in the last workgroup) compute on the last
    // signal and store nothing
    const long long gl = active ? g : (long long)count - 1;
    lds_transform<LOGN, LOGP, WG, KIND, SPLIT>(in + gl * SH::IN_STRIDE, out + gl * SH::OUT_STRIDE, active, tw, lds,
                                               threadIdx.x);
}

// One transform per workgroup with the exchange one LDS plane at a time, held to MINW
// waves per SIMD so that several workgroups share a CU: one workgroup's loads and stores
// then overlap another's arithmetic.  The grid is exactly `count` workgroups.
template <int LOGN, int LOGP, int KIND, int MINW>
__global__ __launch_bounds__((1 << LOGN) >> LOGP, MINW) void fft_lds_shared_cu_kernel(
    const float2* __restrict__ in, float2* __restrict__ out, const float2* __restrict__ tw, int count)
{
    constexpr int WG = (1 << LOGN) >> LOGP;
    using SH = LdsShape<LOGN, LOGP, WG, KIND, true>;
    __shared__ __align__(16) float lds[SH::LDS_WORDS];
    (void)count;
    const long long g = (long long)blockIdx.x;
    lds_transform<LOGN, LOGP, WG, KIND, true>(in + g * SH::IN_STRIDE, out + g * SH::OUT_STRIDE, true, tw, lds,
                                              threadIdx.x);
}

// Several short transforms to a workgroup whose output, and with SIN also whose input, passes
// through LDS in memory order: every read or write of memory is then a run of 512 bytes per
// wave (the writes on line boundaries), where a thread's own points would give runs of T
// points (T threads per transform) and, for the real kinds, rows of N + 1 values that start
// off a line.  Bound by HBM.  2^24 points, plain against staged: complex 16 x 2^20 150 against
// 44 us (6.1 TB/s), complex 64 x 2^18 63 / 46, real forward 32 x 2^20 460 / 46, 512 x 2^16
// 75 / 53, real inverse 32 x 2^20 207 / 46, 256 x 2^17 70 / 51.
template <int LOGN, int LOGP, int WG, int KIND, bool SIN>
__global__ __launch_bounds__(WG) void fft_lds_staged_kernel(const float2* __restrict__ in, float2* __restrict__ out,
                                                            const float2* __restrict__ tw, int count)
{
    using SH = LdsShape<LOGN, LOGP, WG, KIND, false>;
    constexpr int TPW = SH::TPW, IS = SH::IN_STRIDE, OS = SH::OUT_STRIDE;
    constexpr bool PI = SH::T > 1 || IS % 2 == 0, PO = SH::T > 1 || OS % 2 == 0;
    constexpr int IN_SLOTS = SIN ? staged_slot<PI>(TPW * IS - 1) + 1 : 0;
    constexpr int OUT_SLOTS = staged_slot<PO>(TPW * OS - 1) + 1;
    constexpr int TILE_WORDS = 2 * (IN_SLOTS > OUT_SLOTS ? IN_SLOTS : OUT_SLOTS);
    __shared__ __align__(16) float lds[TILE_WORDS > SH::LDS_WORDS ? TILE_WORDS : SH::LDS_WORDS];
    float2* tile = reinterpret_cast<float2*>(lds);
    const int tid = threadIdx.x, tr = tid / SH::T;
    const long long g0 = (long long)blockIdx.x * TPW;
    const int signals = count - g0 < TPW ? (int)(count - g0) : TPW;
    const bool active = tr < signals;
    // in a last workgroup with fewer signals the lanes past the end read its last point again,
    // and the idle slots compute on what LDS holds (SIN) or on the last signal
    const float2* src = in + g0 * IS;
    if constexpr (SIN) {
        constexpr int K = (TPW * IS + WG - 1) / WG;
        const int last = signals * IS - 1;
        float2 x[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int i = tid + k * WG;
            x[k] = ld_in<true>(&src[i < last ? i : last]);
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int i = tid + k * WG;
            tile[staged_slot<PI>(i < last ? i : last)] = x[k];
        }
        __syncthreads();
    }
    float2* dst = out + g0 * OS;
    const LdsOut<PO> staged{tile, tr * OS};
    if constexpr (SIN)
        lds_transform_io<LOGN, LOGP, WG, KIND, false, true>(LdsIn<PI>{tile, tr * IS}, staged, active, tw, lds, tid);
    else
        lds_transform_io<LOGN, LOGP, WG, KIND, false, true>(MemIn<true>{src + (active ? tr : signals - 1) * IS}, staged,
                                                            active, tw, lds, tid);
    __syncthreads();
    // a wave's 64 points start on a line: thread 0 takes the first point of the line in which
    // the output begins (points before it belong to the previous workgroup)
    const int points = signals * OS, sh = (int)(((unsigned long long)dst & 127u) >> 3);
#pragma unroll
    for (int k = 0; k < (TPW * OS + 15 + WG - 1) / WG; ++k) {
        const int i = tid + k * WG - sh;
        if (i >= 0 && i < points) st_out<true>(&dst[i], tile[staged_slot<PO>(i)]);
    }
}

// ---- host-side dispatch ------------------------------------------------------------

using KernelFn = void (*)(const float2*, float2*, const float2*, int);

struct LaunchCfg {
    KernelFn fn;
    int wg;        // threads per workgroup
    int tpw;       // transforms per workgroup
    KernelFn many = nullptr;     // another kernel (staged, if not said otherwise) from many_min
    int many_wg = 0, many_tpw = 0, many_min = 0;   // transforms on (or null)
    KernelFn few = nullptr;      // one transform to a workgroup of few_wg threads, for up to few_max
    int few_wg = 0, few_max = 0;                   // transforms (or null)
};

constexpr int kComputeUnits = 256;   // of the MI355X

// Which side of a transform of 2^logn complex points passes through LDS in the staged kernel.
// Input: up to 2^7 points, whose 16-points-per-thread reads are runs of at most 8 points.
// Output: the same, and every real forward of several transforms to a workgroup (rows of
// N + 1 values, written as whole lines once the workgroup's rows are one run).  One transform
// to a workgroup keeps its rows off a line, and staging it measured slower (real 8192 x 4096:
// 62 us against 56).
constexpr bool staged_in(int logn) { return logn >= 2 && logn <= 7; }
constexpr bool staged_out(int kind, int logn) { return logn >= 2 && logn <= (kind == kRealForward ? 11 : 7); }

// Transforms from which the staged kernel is taken (below, the plain one: the two extra passes
// through LDS cost 0.3-1 us of latency, which only a batch that fills the chip gets back).
// One-thread transforms always, their plain reads touch one 8-byte value per line, but for the real inverse of 8
// samples, whose lines the threads of a wave share.  Measured
// crossings, plain against staged: complex 2^7 8.2 / 8.2 us x 8192 and 14.6 / 11.7 x 16384;
// real forward 2^7 points 5.9 / 5.7 x 2048, 2^9 7.4 / 7.2 x 2048 and 10.7 / 9.3 x 4096, 2^11 9.9 / 11.0 x 1300, 12.7 / 12.7
// x 1800 and 14.9 / 12.8 x 2048; real inverse 2^8 samples 6.9 / 7.1 x 8192 and 10.3 / 9.4 x 16384, 8 samples 5.0 / 5.7
// x 300000, 5.9 / 7.0 x 400000, 7.7 / 7.5 x 450000 and 8.7 / 8.1 x 524288.
constexpr int staged_min(int kind, int logn)
{
    if (kind == kRealInverse && logn == 2) return 13 << 15;
    if (logn <= 4) return 0;
    if (kind == kRealForward && logn == 11) return 7 << 8;
    const int log_points = kind == kRealForward ? (logn <= 7 ? 18 : 21) : logn <= 5 ? 18 : logn == 6 ? 19 : 21;
    return 1 << (log_points - logn);
}

// Threads of a workgroup.  One wave up to 2^10 points: a small batch then spreads over four times as many
// CUs as with 256 threads (complex 32 x 4096 5.7 -> 3.9 us, real forward 64 x 2048 5.4 -> 4.0, 512 x 1024
// 5.5 -> 4.4, complex 1024 x 16384 46.9 -> 45.0).  In the staged kernel no wave waits for another's copies
// (real forward 512 x 40001 38 -> 35 us, x 65536 54 -> 49, 256 x 10000 7.6 -> 6.7; complex 64 x 199999, forward and
// inverse, 73.1 -> 70.3); longer real forwards keep 256 there, where 64 gained 5 % at 2^24 points and lost 5 % at 2^21.
// Real inverses of 2^9 and 2^10 points have 256 too for such batches: transforms are dealt
// to workgroups, and so to XCDs, alike, and an inverse right after its forward finds the spectrum in its own
// L2 (forward and inverse of 1024 x 4096 16 us, with unequal workgroups 19).  Those of 2^8 have 256 from 11264 on
// (one wave / 256 threads: x 10000 8.9 / 10.6 us, x 12000 10.9 / 10.2, x 40001 35.6 / 35.0, x 65536 54.7 / 53.5,
// x 131072 105.4 / 100.9).
constexpr int plain_wg(int logn, int t) { return t >= 256 ? t : logn >= 5 && logn <= 10 ? (t > 64 ? t : 64) : 256; }
constexpr int wide_inverse_min(int logn) { return logn == 8 ? 11 << 10 : staged_min(kRealForward, logn); }
constexpr int staged_wg(int kind, int logn) { return logn >= 5 && logn <= (kind == kRealForward ? 8 : 7) ? 64 : 256; }

template <int LOGN, int KIND>
constexpr LaunchCfg make_cfg()
{
    // points per thread: whole transform for N <= 16, 16 up to 2^13 and for complex 2^14, 32 for real
    // 2^15, 64 at 2^15 (512 threads x 64 points measured faster than 1024 x 32 on MI355X: complex x 256
    // 35.4 us against 37.2).
    // 2^13 and 2^14 exchange one LDS plane at a time (34 / 68 KiB), so that up to four /
    // two workgroups share a CU: batches of 256 MiB per buffer took 98-112 us against
    // 111-122 us (complex 2^13) and 109-124 us against 124-137 us (complex 2^14) with both
    // planes in LDS and one or two workgroups per CU.  The radix plan, and so every bit of
    // the result, is the same.
    // Complex 2^14 has 1024 threads, two workgroups to a CU at 64 registers (x 1024 58.4 -> 52.0 us,
    // x 2048 105.4 -> 99.4, against 512 threads); the real kinds do not fit 64 without spills (forward
    // x 1024 71.4 us without the limit, inverse x 512 30.6 with it, against 59.7 and 29.4).
    // While every workgroup of the batch has its place on the chip at once, none waits for LDS: both
    // planes in one exchange, half its barriers, and 16 points a thread are then faster (plane by
    // plane against both: complex 2^13 x 1 7.0 / 6.6, x 256 11.7 / 11.3, x 512 equal, x 768 21.8 / 24.0; complex
    // 2^14 x 1 11.3 / 9.9, x 256 21.0 / 17.1, x 300 25.2 / 26.7; real 2^15 x 1 12.2 / 10.8, x 256 22.0 / 19.7
    // forward and 20.2 / 17.7 inverse, x 300 25.9 / 29.7).
    if constexpr (LOGN == 13) {
        return LaunchCfg{fft_lds_shared_cu_kernel<13, 4, KIND, 6>, 512, 1, nullptr, 0, 0, 0,
                         fft_lds_kernel<13, 4, 512, KIND, false>, 512, 2 * kComputeUnits};
    } else if constexpr (LOGN == 14) {
        constexpr bool REAL = KIND == kRealForward || KIND == kRealInverse;
        constexpr int LOGP = REAL ? 5 : 4;
        return LaunchCfg{fft_lds_shared_cu_kernel<14, LOGP, KIND, REAL ? 4 : 8>, (1 << 14) >> LOGP, 1, nullptr, 0, 0, 0,
                         fft_lds_kernel<14, 4, 1024, KIND, false>, 1024, kComputeUnits};
    } else {
        constexpr int LOGP = LOGN <= 4 ? LOGN : (LOGN <= 14 ? 4 : 6);
        constexpr int T = (1 << LOGN) >> LOGP;
        constexpr int WG = plain_wg(LOGN, T), SWG = staged_wg(KIND, LOGN);
        constexpr bool SPLIT = LOGN >= 15;
        LaunchCfg c{nullptr, WG, WG / T};
        if constexpr (!staged_out(KIND, LOGN) || staged_min(KIND, LOGN) > 0)
            c.fn = fft_lds_kernel<LOGN, LOGP, WG, KIND, SPLIT>;
        if constexpr (staged_out(KIND, LOGN)) {
            c.many = fft_lds_staged_kernel<LOGN, LOGP, SWG, KIND, staged_in(LOGN)>;
            c.many_wg = SWG;
            c.many_tpw = SWG / T;
            c.many_min = staged_min(KIND, LOGN);
        } else if constexpr (KIND == kRealInverse && staged_out(kRealForward, LOGN) && WG < 256) {
            c.many = fft_lds_kernel<LOGN, LOGP, 256, KIND, SPLIT>;   // not staged, see plain_wg
            c.many_wg = 256;
            c.many_tpw = 256 / T;
            c.many_min = wide_inverse_min(LOGN);
        }
        return c;
    }
}

template <int KIND, int... L>
constexpr void fill_table(LaunchCfg* tab, std::integer_sequence<int, L...>)
{
    ((tab[L + 1] = make_cfg<L + 1, KIND>()), ...);
}

struct LdsTables {
    LaunchCfg t[4][kLogMaxLds + 1];
    LdsTables()
    {
        for (auto& row : t)
            for (auto& c : row) c = LaunchCfg{nullptr, 0, 0};
        fill_table<kComplexForward>(t[kComplexForward], std::make_integer_sequence<int, kLogMaxLds>{});
        fill_table<kComplexInverse>(t[kComplexInverse], std::make_integer_sequence<int, kLogMaxLds>{});
        fill_table<kRealForward>(t[kRealForward], std::make_integer_sequence<int, kLogMaxLds>{});
        fill_table<kRealInverse>(t[kRealInverse], std::make_integer_sequence<int, kLogMaxLds>{});
    }
};

static const LdsTables& lds_tables()
{
    static const LdsTables tables;
    return tables;
}

// Launch the one-workgroup kernel for complex size 2^logc (real kinds: half size).
hipError_t launch_lds(Kind kind, int logc, int count, const void* in, void* out, const float2* pyramid,
                      hipStream_t stream)
{
    if (logc < 1 || logc > kLogMaxLds) return hipErrorInvalidValue;
    const LaunchCfg& c = lds_tables().t[kind][logc];
    if (!c.fn && !c.many) return hipErrorInvalidValue;
    if (count <= 0) return hipSuccess;
    const bool few = count <= c.few_max, many = !few && c.many && count >= c.many_min;
    const int tpw = few ? 1 : many ? c.many_tpw : c.tpw, wg = few ? c.few_wg : many ? c.many_wg : c.wg;
    const unsigned grid = (unsigned)(((long long)count + tpw - 1) / tpw);
    hipLaunchKernelGGL(few ? c.few : many ? c.many : c.fn, dim3(grid), dim3(wg), 0, stream, (const float2*)in,
                       (float2*)out, pyramid, count);
    return hipGetLastError();
}

}  // namespace ckfft_gpu
