// Host-memory calls: where the kernel that reports its end by a word may read from, and the wait for the stream where
// it does not report in time.
#include "fake_hip.h"

#include "ckfft_internal.h"

using namespace ckfft_gpu;

static const void* fake_pinned = nullptr;    // pointers with attributes of their own; all others are pageable
static const void* fake_device = nullptr;    // of device `fake_device_of`
static const void* fake_managed = nullptr;
static int fake_device_of = 0;
static const void* read_from = nullptr;      // what the last launch read
static bool word_written = true;

extern "C" hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
extern "C" hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
    *a = hipPointerAttribute_t{};
    if (p && p == fake_pinned)
        a->type = hipMemoryTypeHost;
    else if (p && p == fake_managed)
        a->type = hipMemoryTypeManaged;
    else if (p && p == fake_device) {
        a->type = hipMemoryTypeDevice;
        a->device = fake_device_of;
    } else
        return hipErrorInvalidValue;
    return hipSuccess;
}

namespace ckfft_gpu {
bool signal_supported(Kind, int log2n) { return log2n <= kLogMaxLds; }
// "transforms": copies the n floats and adds 1
hipError_t launch_signal(Kind, int log2n, const void* in, void* out, const DeviceTables&, hipStream_t, unsigned* done, unsigned ticket)
{
    call("launch_signal");
    read_from = in;
    for (int i = 0; i < 1 << log2n; ++i) ((float*)out)[i] = ((const float*)in)[i] + 1;
    if (word_written) *done = ticket;
    return hipSuccess;
}
hipError_t launch_transform(Kind, int log2n, int, const void* in, void* out, const DeviceTables&, hipStream_t, void*, size_t, bool)
{
    call("launch_transform");
    read_from = in;
    for (int i = 0; i < 1 << log2n; ++i) ((float*)out)[i] = ((const float*)in)[i] + 1;
    return hipSuccess;
}
}  // namespace ckfft_gpu

struct Calls {
    int signal = count_calls("launch_signal"), transform = count_calls("launch_transform"), sync = count_calls("hipStreamSynchronize");
};

// One real forward of 1024 floats on `pool`; the launches and stream waits it made.
static Calls one(StagingPool* pool, const float* in, float* out)
{
    const Calls before;
    DeviceTables tb{};
    CHECK(staged_transform(pool, kRealForward, 10, in, 4096, out, 8 * 513, tb) == hipSuccess);
    for (int i = 0; i < 1024; ++i) CHECK(out[i] == in[i] + 1);
    Calls c;
    c.signal -= before.signal;
    c.transform -= before.transform;
    c.sync -= before.sync;
    return c;
}

int main()
{
    StagingPool* pool = staging_create();
    std::vector<float> in(1024), out(1026);
    for (int i = 0; i < 1024; ++i) in[i] = (float)i;
    // pageable to pageable: by the word, from the slot's buffer
    Calls c = one(pool, in.data(), out.data());
    CHECK(c.signal == 1 && c.transform == 0 && c.sync == 0 && read_from != in.data());
    // a caller's pinned input, rewritten between calls: never read in place without a stream wait
    fake_pinned = in.data();
    for (int k = 0; k < 3; ++k) {
        in[7] = -1.0f - k;
        c = one(pool, in.data(), out.data());
        CHECK(read_from != in.data() || c.sync == 1);
        CHECK(c.signal == 1 && c.sync == 0);
    }
    // pinned output: the stream is idle when it is handed back
    fake_pinned = out.data();
    c = one(pool, in.data(), out.data());
    CHECK(c.signal == 0 && c.transform == 1 && c.sync == 1);
    fake_pinned = nullptr;
    // device inputs: in place; by the word only from the current device's own memory
    fake_device = in.data();
    c = one(pool, in.data(), out.data());
    CHECK(c.signal == 1 && c.sync == 0 && read_from == in.data());
    fake_device_of = 1;
    c = one(pool, in.data(), out.data());
    CHECK(c.signal == 0 && c.transform == 1 && c.sync == 1);
    fake_device = nullptr;
    fake_managed = in.data();
    c = one(pool, in.data(), out.data());
    CHECK(c.signal == 0 && c.transform == 1 && c.sync == 1);
    fake_managed = nullptr;
    // no word in time (the device is busy): the call waits for the stream, and the next one is its own
    word_written = false;
    c = one(pool, in.data(), out.data());
    CHECK(c.signal == 1 && c.transform == 0 && c.sync == 1);
    word_written = true;
    in[3] = 77.0f;
    c = one(pool, in.data(), out.data());
    CHECK(c.signal == 1 && c.sync == 0);
    staging_destroy(pool);
    // pageable calls above one workgroup: the stream is looked at behind the kernels if the input came in several chunks
    for (int log2n : {17, 18, 19, 20}) {
        const size_t bytes = (size_t)4 << log2n;
        std::vector<float> a(1 << log2n, 1.0f), b((1 << log2n) + 2);
        DeviceTables tb{};
        StagingPool* p = staging_create();
        const int before = count_calls("hipStreamQuery");
        CHECK(staged_transform(p, kRealForward, log2n, a.data(), bytes, b.data(), bytes + 8, tb) == hipSuccess);
        CHECK(count_calls("hipStreamQuery") - before == (bytes > (1u << 20)));
        CHECK(hipGetLastError() == hipSuccess);
        CHECK(b[0] == 2.0f && b[(1 << log2n) - 1] == 2.0f);
        staging_destroy(p);
    }
    // a size's inverse finds room in its forward's buffers (real n: 4n in, 4n + 8 out, and the other way round)
    for (int log2n = 4; log2n <= 20; ++log2n) {
        const size_t n = (size_t)1 << log2n;
        std::vector<float> a(2 * n), b(2 * n);
        DeviceTables tb{};
        for (int kind : {kRealForward, kRealInverse}) {
            StagingPool* p = staging_create();
            const auto go = [&](int k) {
                const size_t ib = k == kRealForward ? 4 * n : 4 * n + 8, ob = k == kRealForward ? 4 * n + 8 : 4 * n;
                CHECK(staged_transform(p, (Kind)k, log2n, a.data(), ib, b.data(), ob, tb) == hipSuccess);
            };
            go(kind);
            const int dev = count_calls("hipMalloc"), host = count_calls("hipHostMalloc");
            go(kind == kRealForward ? kRealInverse : kRealForward);
            CHECK(count_calls("hipMalloc") == dev && count_calls("hipHostMalloc") == host);
            staging_destroy(p);
        }
    }
    return 0;
}
