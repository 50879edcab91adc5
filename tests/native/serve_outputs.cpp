// Requests whose outputs share memory: the server orders their batches where one keeps its intermediate there.
#include "fake_hip.h"

#include "fft_batch.h"

using namespace ckfft_gpu;

namespace ckfft_gpu {
OutputRange output_range(const CkFftBatchDesc& d) { return {(uintptr_t)d.output, (uintptr_t)d.output + 8 * (size_t)d.n}; }
bool batch_check_desc(const CkFftContext*, const CkFftBatchDesc&, int, bool) { return true; }
bool batch_build(const CkFftContext*, const CkFftBatchDesc* d, int count, int, bool, BatchBuild& out, bool)
{
    out = BatchBuild{};
    for (int i = 0; i < count; ++i) out.extras.push_back(BatchExtra{(Kind)d[i].kind, 0, d[i].input, d[i].output});
    return true;
}
DeviceTables context_tables(const CkFftContext*) { return DeviceTables{}; }
bool mfma_supported(Kind, int) { return false; }
int persistent_grid(const CkFftContext*, bool) { return 1; }
long long transform_bytes(int, int) { return 1; }
size_t transform_scratch_bytes(Kind, int, int, const DeviceTables&) { return 0; }
hipError_t launch_persistent_raw(const BatchItem*, int, const BatchTransform*, int*, int, const DeviceTables&, hipStream_t, bool) { return hipSuccess; }
hipError_t launch_persistent_inline(const BatchBuild&, int*, int, const DeviceTables&, hipStream_t) { return hipSuccess; }
hipError_t launch_pass_inline(const std::vector<BatchTransform>&, const std::vector<BatchTransform>&, const DeviceTables&, hipStream_t) { return hipSuccess; }
hipError_t launch_transform(Kind, int, int, const void*, void*, const DeviceTables&, hipStream_t, void*, size_t, bool)
{
    call("launch");
    return hipSuccess;
}
}  // namespace ckfft_gpu

extern "C" const char* CkFftBatchLastError() { return ""; }

static char* const base = (char*)0x100000000000;   // addresses only: nothing is dereferenced

// Submits first and second, the first still in flight: how often the second's stream waits for the first.
static int waits(int precision, CkFftBatchDesc first, CkFftBatchDesc second)
{
    _CkFftContext ctx{};
    ctx.magic = kContextMagic;
    ctx.max_count = 1 << 20;
    ctx.precision = precision;
    fake_pending = true;
    CkFftServer* s = CkFftServerCreate(&ctx, (size_t)1 << 40, 3);
    CHECK(s);
    const int launched = count_calls("launch"), waited = count_calls("hipStreamWaitEvent");
    CHECK(CkFftServerSubmit(s, first.kind, first.n, first.input, first.output) >= 0);
    CHECK(await_calls("launch", launched + 1));
    CHECK(CkFftServerSubmit(s, second.kind, second.n, second.input, second.output) >= 0);
    CHECK(await_calls("launch", launched + 2));
    fake_pending = false;
    CHECK(CkFftServerDrain(s) == 1);
    CkFftServerDestroy(s);
    return count_calls("hipStreamWaitEvent") - waited;
}

int main()
{
    const int fp32 = kCkFftPrecision_Fp32, split = kCkFftPrecision_SplitBf16x3;
    char* in = base + (1ll << 40);
    const CkFftBatchDesc c16{kComplexForward, 1 << 16, in, base}, c15{kComplexInverse, 1 << 15, in, base};
    const CkFftBatchDesc r17{kRealInverse, 1 << 17, in, base}, r16{kRealForward, 1 << 16, in, base};
    const CkFftBatchDesc small{kComplexForward, 16, in, base + (8 << 16) - 64}, beside{kComplexForward, 16, in, base + (8 << 16)};
    const CkFftBatchDesc far{kComplexForward, 1 << 16, in, base + (1 << 24)};
    CHECK(waits(fp32, c16, c16) == 1);       // the same request again
    CHECK(waits(fp32, r17, c16) == 1);
    CHECK(waits(fp32, c16, small) == 1);     // one workgroup, but over the other's intermediate
    CHECK(waits(fp32, small, c16) == 1);
    CHECK(waits(fp32, c16, beside) == 0);
    CHECK(waits(fp32, c16, far) == 0);
    CHECK(waits(fp32, c15, c15) == 0);       // one workgroup each: the same values, written once
    CHECK(waits(fp32, r16, r16) == 0);
    CHECK(waits(split, c15, c15) == 1);      // two passes in this mode
    CHECK(waits(split, r16, r16) == 0);
    // which of several share
    const std::vector<char> s = shared_outputs({{100, 200}, {500, 600}, {150, 160}, {300, 400}, {600, 700}}, {{390, 391}, {400, 500}});
    CHECK((s == std::vector<char>{1, 0, 1, 1, 0}));
    CHECK((shared_outputs({{0, 8}, {0, 8}}, {}) == std::vector<char>{1, 1}) && shared_outputs({}, {{0, 1}}).empty());
    return 0;
}
