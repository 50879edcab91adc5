"""Sizes above one workgroup: the intermediate lives in the output, in wide and narrow tiles.
The input and everything around the output stay untouched, a signal's bits do not depend on
the tile width its batch takes, and overlapping buffers still work (through an intermediate of
their own).  Tolerances are those of test_gpu_parity."""
import numpy as np
import pytest

import oracle as O
from test_gpu_parity import TOL_FP64, TOL_REF, C, fp64_out, make_input, oracle_out, out_len, torch  # noqa: F401

pytestmark = pytest.mark.gpu

KINDS = ["cfwd", "cinv", "rfwd", "rinv"]


@pytest.fixture(scope="module")
def ctx(torch, C):  # noqa: F811
    c = C.Context(1 << 23, C.kCkFftDirection_Both)
    yield c
    c.close()


def call(ctx, kind):
    return {"cfwd": ctx.complex_forward_batch, "cinv": ctx.complex_inverse_batch,
            "rfwd": ctx.real_forward_batch, "rinv": ctx.real_inverse_batch}[kind]


# complex sizes 2^16 .. 2^22: radices 8+8, 9+8, 9+9, 10+9, 10+10, 11+10 (real inverse 10+11), 8+8+6; a count whose wide
# tiles fill the narrow rule's bound, and one signal, which does not (up to 2^20)
@pytest.mark.parametrize("logc,count", [(16, 9), (17, 9), (18, 5), (19, 5), (20, 3), (21, 2), (22, 1)])
@pytest.mark.parametrize("kind", KINDS)
def test_batches(torch, ctx, kind, logc, count):  # noqa: F811
    n = 1 << (logc + (kind in ("rfwd", "rinv")))
    x = make_input(kind, n, 1, 0x3A + logc)
    xt = torch.from_numpy(x).cuda()
    length = out_len(kind, n)
    xin = xt.repeat(count, 1) * (1.0 + torch.arange(count, device="cuda")[:, None] % 2)
    kept = xin.clone()
    guard = 4096
    buf = torch.full((2 * guard + count * length + 2,), -7.0, device="cuda")
    for offset in (0, 2):                              # floats off a line
        buf.fill_(-7.0)
        y = buf[guard + offset:guard + offset + count * length]
        assert call(ctx, kind)(n, count, xin, y) == 1
        torch.cuda.synchronize()
        assert bool((buf[:guard + offset] == -7.0).all()) and bool((buf[guard + offset + count * length:] == -7.0).all())
        assert torch.equal(xin, kept)
        y = y.view(count, length)
        one = torch.empty(length, device="cuda")
        assert call(ctx, kind)(n, 1, xt, one) == 1
        # doubling the input doubles every bit exactly
        for i in range(count):
            assert torch.equal(y[i].view(torch.int32), ((1 + i % 2) * one).view(torch.int32)), i
    got = one.cpu().numpy()[None]
    assert O.split_norm_err(got, oracle_out(kind, n, x)) <= TOL_REF
    assert O.rel_l2(got, fp64_out(kind, n, x)) <= TOL_FP64


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("logc", [17, 21])
def test_overlapping_buffers(torch, ctx, kind, logc):  # noqa: F811
    n = 1 << (logc + (kind in ("rfwd", "rinv")))
    x = torch.from_numpy(make_input(kind, n, 2, 0x0E)).cuda().flatten()
    length = 2 * out_len(kind, n)
    want = torch.empty(length, device="cuda")
    assert call(ctx, kind)(n, 2, x, want) == 1
    buf = torch.empty(x.numel() + length, device="cuda")
    buf[:x.numel()] = x
    got = buf[x.numel() // 2:x.numel() // 2 + length]
    assert call(ctx, kind)(n, 2, buf, got) == 1
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("kind", KINDS)
def test_few_signals_of_one_workgroup_size(torch, ctx, kind):  # noqa: F811
    # 2^15 complex points: up to 32 signals take two launches, more (or overlapping buffers) one workgroup each
    n = 1 << (15 + (kind in ("rfwd", "rinv")))
    x = make_input(kind, n, 33, 0xF5)
    xt = torch.from_numpy(x).cuda()
    length = out_len(kind, n)
    want = torch.empty((33, length), device="cuda")
    assert call(ctx, kind)(n, 33, xt, want) == 1
    got = want.cpu().numpy()
    assert O.split_norm_err(got, oracle_out(kind, n, x)) <= TOL_REF
    assert O.rel_l2(got, fp64_out(kind, n, x)) <= TOL_FP64
    kept = xt.clone()
    for count in (1, 2, 31, 32):
        buf = torch.full((2048 + count * length,), -7.0, device="cuda")
        y = buf[1024:1024 + count * length]
        assert call(ctx, kind)(n, count, xt, y) == 1
        torch.cuda.synchronize()
        assert torch.equal(y.view(count, length).view(torch.int32), want[:count].view(torch.int32)), count
        assert bool((buf[:1024] == -7.0).all()) and bool((buf[-1024:] == -7.0).all()) and torch.equal(xt, kept)
    # host buffers: one workgroup
    fn = {"cfwd": ctx.complex_forward, "cinv": ctx.complex_inverse, "rfwd": ctx.real_forward}.get(kind)
    yh = np.zeros(length, np.float32)
    assert (fn(n, x[3], yh) if fn else ctx.real_inverse(n, x[3], yh, np.zeros(n + 2, np.float32))) == 1
    assert np.array_equal(yh.view(np.int32), got[3].view(np.int32))


@pytest.mark.parametrize("passes", [1, 511, 512])
def test_plan_launch_orders(torch, C, passes):  # noqa: F811
    """Plans either side of the count of 2^16 transforms from which their passes are launched first,
    with and without a graph, replayed: the bits of the stand-alone calls."""
    n, small = 1 << 16, 1 << 15
    with C.Context(n) as c:
        gen = torch.Generator(device="cuda").manual_seed(0x0DE + passes)
        x = torch.randn((passes, 2 * n), device="cuda", generator=gen)
        xs = torch.randn((9, 2 * small), device="cuda", generator=gen)
        want, wants = torch.empty_like(x), torch.empty_like(xs)
        for i in range(passes):
            assert (c.complex_forward_batch if i % 2 == 0 else c.complex_inverse_batch)(n, 1, x[i], want[i]) == 1
        assert c.complex_forward_batch(small, 9, xs, wants) == 1
        torch.cuda.synchronize()
        for graph in (False, True):
            y, ys = torch.zeros_like(x), torch.zeros_like(xs)
            descs = [(C.kCkFftKind_ComplexForward if i % 2 == 0 else C.kCkFftKind_ComplexInverse, n, x[i], y[i])
                     for i in range(passes)]
            descs += [(C.kCkFftKind_ComplexForward, small, xs[i], ys[i]) for i in range(9)]
            plan = C.BatchPlan(c, descs, graph=graph)
            for _ in range(3):
                y.fill_(-7.0)
                ys.fill_(-7.0)
                assert plan.execute(torch.cuda.current_stream()) == 1
                torch.cuda.synchronize()
                assert torch.equal(y.view(torch.int32), want.view(torch.int32))
                assert torch.equal(ys.view(torch.int32), wants.view(torch.int32))
            plan.close()


@pytest.mark.parametrize("log2n,most", [(22, 5), (24, 2)])
@pytest.mark.parametrize("kind", ["cfwd", "cinv"])
def test_first_pass_reads(torch, C, kind, log2n, most):  # noqa: F811
    """Three passes either side of the buffer sizes that change how the first reads its input."""
    n = 1 << log2n
    x = torch.randn((most, 2 * n), device="cuda", generator=torch.Generator(device="cuda").manual_seed(0xF1))
    keep = x.clone()
    want = None
    for count in range(most, 0, -1):
        y = torch.full((count, 2 * n), -7.0, device="cuda")
        with C.Context(n) as c:
            assert call(c, kind)(n, count, x, y) == 1
            torch.cuda.synchronize()
        if want is None:
            want = y
            z = torch.view_as_complex(x[0].double().reshape(n, 2))
            exact = torch.view_as_real(torch.fft.fft(z) if kind == "cfwd" else torch.fft.ifft(z) * n).flatten()
            assert float((y[0].double() - exact).norm() / exact.norm()) <= TOL_FP64
        assert torch.equal(y.view(torch.int32), want[:count].view(torch.int32))
    assert torch.equal(x, keep)


@pytest.mark.parametrize("graph", [False, True])
def test_plan_of_overlapping_buffers(torch, C, graph):  # noqa: F811
    """Complex 2^16 transforms whose input and output overlap, beside others: the bits of separate
    buffers, no memory allocated by an execution, and captured in a caller's graph, replayed."""
    n = 1 << 16
    gen = torch.Generator(device="cuda").manual_seed(0x0F)
    x = torch.randn((4, 2 * n), device="cuda", generator=gen)

    def make(c):
        buf = torch.zeros((3, 3 * n), device="cuda")
        y = torch.zeros((2, 2 * n), device="cuda")
        descs = [(C.kCkFftKind_ComplexForward, n, buf[0], buf[0][n:]), (C.kCkFftKind_ComplexInverse, n, buf[1][n:], buf[1]),
                 (C.kCkFftKind_ComplexForward, n, buf[2], buf[2][n:]), (C.kCkFftKind_ComplexForward, n, x[3], y[0]),
                 (C.kCkFftKind_RealForward, 4096, x[3], y[1])]
        return C.BatchPlan(c, descs, graph=graph), buf, y

    def fill(buf, scale):
        buf[0][:2 * n] = x[0] * scale
        buf[1][n:] = x[1] * scale
        buf[2][:2 * n] = x[2] * scale

    with C.Context(n) as c, C.Context(n) as fresh:
        want = torch.empty((4, 2 * n), device="cuda")
        for i in range(4):
            assert call(c, "cinv" if i == 1 else "cfwd")(n, 1, x[i], want[i]) == 1
        plan, buf, y = make(c)                        # loads the code
        assert plan.execute() == 1
        torch.cuda.synchronize()
        plan.close()
        plan, buf, y = make(fresh)
        info = plan.info()
        assert info["pass_transforms"] == 1 and info["extra_launches"] == 3

        def check(scale):
            # scaling by a power of two scales every bit exactly
            assert torch.equal(buf[0][n:].view(torch.int32), (want[0] * scale).view(torch.int32))
            assert torch.equal(buf[1][:2 * n].view(torch.int32), (want[1] * scale).view(torch.int32))
            assert torch.equal(buf[2][n:].view(torch.int32), (want[2] * scale).view(torch.int32))
            assert torch.equal(y[0].view(torch.int32), want[3].view(torch.int32))

        if graph:                                     # the plan's own graph is made by its first execution
            assert plan.execute() == 1
        fill(buf, 1.0)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        assert plan.execute() == 1
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] == free
        check(1.0)
        if not graph:
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                assert plan.execute(torch.cuda.current_stream()) == 1
            for scale in (2.0, 0.5, 4.0):
                fill(buf, scale)
                y.fill_(-7.0)
                g.replay()
                torch.cuda.synchronize()
                check(scale)
        plan.close()



@pytest.mark.parametrize("passes", [512, 640, 641])
def test_plan_pass_groups(torch, C, passes):  # noqa: F811
    """Plans whose 2^16 transforms take two and three pairs of table launches, with directions that change
    within a group: the bits of the stand-alone calls."""
    n, distinct = 1 << 16, 7
    gen = torch.Generator(device="cuda").manual_seed(0x320 + passes)
    x = torch.randn((distinct, 2 * n), device="cuda", generator=gen)
    want = torch.empty((2, distinct, 2 * n), device="cuda")
    with C.Context(n) as c:
        assert c.complex_forward_batch(n, distinct, x, want[0]) == 1
        assert c.complex_inverse_batch(n, distinct, x, want[1]) == 1
        y = torch.full((passes, 2 * n), -7.0, device="cuda")
        kinds = [i % 3 == 0 for i in range(passes)]            # a third inverse
        plan = C.BatchPlan(c, [(C.kCkFftKind_ComplexInverse if kinds[i] else C.kCkFftKind_ComplexForward, n, x[i % distinct],
                                y[i]) for i in range(passes)], graph=True)
        assert plan.info()["pass_transforms"] == passes
        for _ in range(2):
            y.fill_(-7.0)
            assert plan.execute(torch.cuda.current_stream()) == 1
            torch.cuda.synchronize()
            for i in range(passes):
                assert torch.equal(y[i].view(torch.int32), want[int(kinds[i])][i % distinct].view(torch.int32)), i
        plan.close()
