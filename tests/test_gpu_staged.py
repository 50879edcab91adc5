"""Batches of short transforms large enough for the kernels that pass the workgroup's input and
output through LDS: the last signals of a partly filled workgroup, outputs that start off a
line, and nothing written outside the output.  Tolerances are those of test_gpu_parity."""
import numpy as np
import pytest

import oracle as O
from test_gpu_parity import TOL_FP64, TOL_REF, C, ctx, fp64_out, make_input, oracle_out, out_len, torch  # noqa: F401

pytestmark = pytest.mark.gpu

KINDS = ["cfwd", "cinv", "rfwd", "rinv"]


@pytest.mark.parametrize("log2n", range(2, 13))
@pytest.mark.parametrize("kind", KINDS)
def test_short_batches(torch, ctx, kind, log2n):  # noqa: F811
    n = 1 << log2n
    if kind in ("rfwd", "rinv") and log2n < 3:
        pytest.skip("closed form")
    # 512 times 4096 complex points, whole workgroups of any size, and one signal more
    logc = log2n - 1 if kind in ("rfwd", "rinv") else log2n
    per = 256 * min(16, 1 << logc) >> logc
    count = 512 * per + 1
    distinct = min(count, 2 * per + 3)
    x = make_input(kind, n, distinct, 0x57 + log2n)
    xt = torch.from_numpy(x).cuda()
    rows = torch.arange(count, device="cuda") % distinct
    rows[-1] = distinct - 1
    xin = torch.cat([torch.zeros(2, device="cuda"), xt[rows].flatten()])[2:]
    length = out_len(kind, n)
    for offset in (0, 2, 34):                          # floats off a line
        guard = 64
        buf = torch.full((guard + offset + count * length + guard,), -7.0, device="cuda")
        y = buf[guard + offset:guard + offset + count * length]
        fn = {"cfwd": ctx.complex_forward_batch, "cinv": ctx.complex_inverse_batch,
              "rfwd": ctx.real_forward_batch, "rinv": ctx.real_inverse_batch}[kind]
        assert fn(n, count, xin, y) == 1
        torch.cuda.synchronize()
        assert bool((buf[:guard + offset] == -7.0).all()) and bool((buf[-guard:] == -7.0).all())
        y = y.view(count, length)
        first = y[:distinct]
        # equal inputs give equal bits wherever they lie in the batch
        assert torch.equal(y.view(torch.int32), first[rows].view(torch.int32))
        got = first.cpu().numpy()
        assert np.all(np.isfinite(got))
        assert O.split_norm_err(got, oracle_out(kind, n, x)) <= TOL_REF
        assert O.rel_l2(got, fp64_out(kind, n, x)) <= TOL_FP64
        # one signal per call takes another kernel and gives the same bits
        one = torch.empty(length, device="cuda")
        assert fn(n, 1, xt[1], one) == 1
        assert torch.equal(one.view(torch.int32), first[1].view(torch.int32))


@pytest.mark.parametrize("log2n", range(4, 15))
@pytest.mark.parametrize("kind", ["cfwd", "cinv"])
def test_split_mode_batches(torch, C, kind, log2n):  # noqa: F811
    """The matrix-core mode: partly filled workgroups of short signals (passed through LDS), and the
    stages whose twiddles come from transposed copies, in contexts of this size and of 2^16
    (whose transposed tables are of different levels)."""
    n = 1 << log2n
    per = max(1, 4096 >> log2n)
    count = 3 * per + 1
    x = make_input(kind, n, count, 0x5B + log2n)
    xt = torch.from_numpy(x).cuda()
    outs = []
    for nmax in (n, 1 << 16):
        with C.Context(nmax, C.kCkFftDirection_Both) as c:
            assert c.set_precision(C.kCkFftPrecision_SplitBf16x3) == 1
            buf = torch.full((128 + count * 2 * n,), -7.0, device="cuda")
            y = buf[64:-64]
            fn = c.complex_forward_batch if kind == "cfwd" else c.complex_inverse_batch
            assert fn(n, count, xt, y) == 1
            torch.cuda.synchronize()
            assert bool((buf[:64] == -7.0).all()) and bool((buf[-64:] == -7.0).all())
            outs.append(y.clone().view(count, 2 * n))
    assert torch.equal(outs[0].view(torch.int32), outs[1].view(torch.int32))
    got = outs[0].cpu().numpy()
    assert O.split_norm_err(got, oracle_out(kind, n, x)) <= TOL_REF
    assert O.rel_l2(got, fp64_out(kind, n, x)) <= TOL_FP64


@pytest.mark.parametrize("log2c,fit", [(13, 512), (14, 256)])
@pytest.mark.parametrize("kind", KINDS)
def test_batches_that_fit_at_once(torch, ctx, kind, log2c, fit):  # noqa: F811
    """One and the most workgroups that the kernels for small batches take, and one more."""
    n = 1 << (log2c + 1 if kind in ("rfwd", "rinv") else log2c)
    distinct = 5
    x = make_input(kind, n, distinct, 0xF17 + log2c)
    fn = {"cfwd": ctx.complex_forward_batch, "cinv": ctx.complex_inverse_batch,
          "rfwd": ctx.real_forward_batch, "rinv": ctx.real_inverse_batch}[kind]
    length, guard = out_len(kind, n), 64
    xt = torch.from_numpy(x).cuda()
    first = None
    for count in (fit + 1, fit, distinct, 1):
        rows = torch.arange(count, device="cuda") % distinct
        xin = xt[rows].contiguous()
        buf = torch.full((guard + count * length + guard,), -7.0, device="cuda")
        y = buf[guard:guard + count * length]
        assert fn(n, count, xin, y) == 1
        torch.cuda.synchronize()
        assert bool((buf[:guard] == -7.0).all()) and bool((buf[-guard:] == -7.0).all())
        y = y.view(count, length)
        if first is None:
            first = y[:distinct].clone()
            got = first.cpu().numpy()
            assert O.split_norm_err(got, oracle_out(kind, n, x)) <= TOL_REF
            assert O.rel_l2(got, fp64_out(kind, n, x)) <= TOL_FP64
        # equal inputs give equal bits in either kernel
        assert torch.equal(y.view(torch.int32), first[rows].view(torch.int32))


@pytest.mark.parametrize("log2n", [4, 5, 6])
@pytest.mark.parametrize("kind", ["cfwd", "cinv"])
def test_split_mode_short_batches(torch, C, kind, log2n):  # noqa: F811
    """Either side of the batch sizes from which the matrix-core mode passes short signals through LDS."""
    n, distinct = 1 << log2n, 7
    per = 4096 >> log2n
    x = make_input(kind, n, distinct, 0x5C + log2n)
    xt = torch.from_numpy(x).cuda()
    first = None
    with C.Context(n, C.kCkFftDirection_Both) as c:
        assert c.set_precision(C.kCkFftPrecision_SplitBf16x3) == 1
        fn = c.complex_forward_batch if kind == "cfwd" else c.complex_inverse_batch
        for count in (1, 143 * per, 143 * per + 1, 207 * per, 207 * per + 1):
            rows = torch.arange(count, device="cuda") % distinct
            xin = xt[rows].contiguous()
            buf = torch.full((128 + count * 2 * n,), -7.0, device="cuda")
            y = buf[64:-64]
            assert fn(n, count, xin, y) == 1
            torch.cuda.synchronize()
            assert bool((buf[:64] == -7.0).all()) and bool((buf[-64:] == -7.0).all())
            y = y.view(count, 2 * n)
            if count >= distinct and first is None:
                first = y[:distinct].clone()
                got = first.cpu().numpy()
                assert O.split_norm_err(got, oracle_out(kind, n, x)) <= TOL_REF
                assert O.rel_l2(got, fp64_out(kind, n, x)) <= TOL_FP64
            if first is not None:
                assert torch.equal(y.view(torch.int32), first[rows].view(torch.int32))


@pytest.mark.parametrize("log2n", [12, 13, 14])
def test_split_mode_in_an_arena(torch, C, log2n):  # noqa: F811
    """Contexts whose tables lie in a caller's arena of 16 bytes a point have no transposed copies below 2^15:
    the same bits from the pyramid."""
    n, count = 1 << log2n, 5
    need = C.CkFftDeviceTableBytes(n, C.kCkFftDirection_Both)
    assert need == 2 * n * 8
    arena = torch.zeros(need, dtype=torch.uint8, device="cuda")
    x = torch.from_numpy(make_input("cfwd", n, count, 0xA5 + log2n)).cuda()
    outs = []
    for c in (C.Context(n, C.kCkFftDirection_Both, arena=arena), C.Context(n, C.kCkFftDirection_Both)):
        with c:
            assert c.set_precision(C.kCkFftPrecision_SplitBf16x3) == 1
            y, z = torch.empty_like(x), torch.empty_like(x)
            assert c.complex_forward_batch(n, count, x, y) == 1
            assert c.complex_inverse_batch(n, count, y, z) == 1
            torch.cuda.synchronize()
            outs.append((y, z))
    for a, b in zip(*outs):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("log2c", range(5, 12))
@pytest.mark.parametrize("kind", KINDS)
def test_workgroup_sizes(torch, ctx, kind, log2c):  # noqa: F811
    """Batches either side of the counts from which another workgroup size or the staged kernel is taken:
    partly filled workgroups, and equal bits for equal inputs in each."""
    real = kind in ("rfwd", "rinv")
    n = 1 << (log2c + 1 if real else log2c)
    distinct = 9
    x = make_input(kind, n, distinct, 0x3C + log2c)
    xt = torch.from_numpy(x).cuda()
    fn = {"cfwd": ctx.complex_forward_batch, "cinv": ctx.complex_inverse_batch,
          "rfwd": ctx.real_forward_batch, "rinv": ctx.real_inverse_batch}[kind]
    length, guard = out_len(kind, n), 64
    first = None
    for count in (distinct, 1, (1 << 21 >> log2c) + 1, 1 << 21 >> log2c, (1 << 21 >> log2c) - 1, (1 << 18 >> log2c) + 1,
                  (1 << 18 >> log2c) - 1):
        rows = torch.arange(count, device="cuda") % distinct
        xin = xt[rows].contiguous()
        buf = torch.full((guard + count * length + guard,), -7.0, device="cuda")
        y = buf[guard:guard + count * length]
        assert fn(n, count, xin, y) == 1
        torch.cuda.synchronize()
        assert bool((buf[:guard] == -7.0).all()) and bool((buf[-guard:] == -7.0).all())
        y = y.view(count, length)
        if first is None:
            first = y.clone()
            got = first.cpu().numpy()
            assert O.split_norm_err(got, oracle_out(kind, n, x)) <= TOL_REF
            assert O.rel_l2(got, fp64_out(kind, n, x)) <= TOL_FP64
        assert torch.equal(y.view(torch.int32), first[rows].view(torch.int32))


# (kind, size, split mode, count): batch sizes from which another kernel is taken
@pytest.mark.parametrize("kind,log2n,split,least", [("rfwd", 12, False, 7 << 8), ("rinv", 9, False, 11 << 10),
                                                     ("rinv", 3, False, 13 << 15), ("cfwd", 8, True, 3071 * 16 + 1),
                                                     ("cinv", 8, True, 3071 * 16 + 1)])
def test_either_side_of_a_rule(torch, C, kind, log2n, split, least):  # noqa: F811
    n, distinct = 1 << log2n, 9
    x = make_input(kind, n, distinct, 0x71 + log2n)
    xt = torch.from_numpy(x).cuda()
    length, guard, first = out_len(kind, n), 64, None
    with C.Context(n, C.kCkFftDirection_Both) as c:
        assert not split or c.set_precision(C.kCkFftPrecision_SplitBf16x3) == 1
        fn = {"cfwd": c.complex_forward_batch, "cinv": c.complex_inverse_batch, "rfwd": c.real_forward_batch,
              "rinv": c.real_inverse_batch}[kind]
        for count in (distinct, least - 1, least, least + 1):
            rows = torch.arange(count, device="cuda") % distinct
            xin = xt[rows].contiguous()
            buf = torch.full((guard + count * length + guard,), -7.0, device="cuda")
            y = buf[guard:guard + count * length]
            assert fn(n, count, xin, y) == 1
            torch.cuda.synchronize()
            assert bool((buf[:guard] == -7.0).all()) and bool((buf[-guard:] == -7.0).all())
            y = y.view(count, length)
            if first is None:
                first = y.clone()
                got = first.cpu().numpy()
                assert O.split_norm_err(got, oracle_out(kind, n, x)) <= TOL_REF
                assert O.rel_l2(got, fp64_out(kind, n, x)) <= TOL_FP64
            assert torch.equal(y.view(torch.int32), first[rows].view(torch.int32))
