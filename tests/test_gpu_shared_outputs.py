"""Transforms of one plan or server that write to the same output: the sizes above one workgroup keep
their intermediate there, so these run one after another and leave the bits of a transform alone."""
import pytest

from test_gpu_parity import C, torch  # noqa: F401

pytestmark = pytest.mark.gpu

CF, CI, RI = 0, 1, 3


def same_bits(torch, a, b):  # noqa: F811
    return torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.fixture(scope="module")
def ctx(torch, C):  # noqa: F811
    with C.Context(1 << 17) as c:
        yield c


@pytest.mark.parametrize("graph", [False, True])
def test_plan(torch, C, ctx, graph):  # noqa: F811
    n = 1 << 16
    gen = torch.Generator(device="cuda").manual_seed(0x5A)
    x = torch.randn((6, 2 * n), device="cuda", generator=gen)
    want = torch.empty_like(x)
    for i in range(6):
        assert (ctx.complex_forward_batch if i != 3 else ctx.complex_inverse_batch)(n, 1, x[i], want[i]) == 1
    small = torch.empty(2 * 1024, device="cuda")
    assert ctx.complex_forward_batch(1024, 1, x[4], small) == 1
    y = torch.empty((6, 2 * n), device="cuda")
    descs = [(CF, n, x[0], y[0]), (CF, n, x[1], y[1]), (CF, n, x[0], y[0]),      # y[0] three times
             (CI, n, x[3], y[3]), (CF, n, x[0], y[0]),
             (CF, 1024, x[4], y[1][2 * n - 2048:]),                                # in the end of y[1]
             (CF, 1024, x[4], y[2][:2048])]                                        # beside y[1]
    plan = C.BatchPlan(ctx, descs, graph=graph)
    info = plan.info()
    assert (info["pass_transforms"], info["extra_launches"], info["persistent_transforms"]) == (1, 4, 2)
    for _ in range(3):
        y.fill_(-7.0)
        torch.cuda.synchronize()
        assert plan.execute() == 1
        torch.cuda.synchronize()
        # the ordinary launches come last, so y[1] holds all of its transform
        assert all(same_bits(torch, y[i], want[i]) for i in (0, 1, 3))
        assert same_bits(torch, y[2][:2048], small) and bool((y[2][2048:] == -7.0).all())
        assert bool((y[4:] == -7.0).all())
    plan.close()


def test_server(torch, C, ctx):  # noqa: F811
    n = 1 << 16
    gen = torch.Generator(device="cuda").manual_seed(0x5B)
    x = torch.randn((3, 2 * n + 2), device="cuda", generator=gen)
    want, y = torch.empty((3, 2 * n), device="cuda"), torch.empty((3, 2 * n), device="cuda")
    fns = [(ctx.complex_forward_batch, CF, n), (ctx.complex_inverse_batch, CI, n), (ctx.real_inverse_batch, RI, 2 * n)]
    for i, (fn, _, m) in enumerate(fns):
        assert fn(m, 1, x[i], want[i]) == 1
    y.fill_(-7.0)
    torch.cuda.synchronize()
    # each request a hundred times: repeated within batches and across batches in flight
    descs = [(k, m, x[i], y[i]) for _ in range(100) for i, (_, k, m) in enumerate(fns)]
    with C.Server(ctx, 4 << 30, max_in_flight=4) as srv:
        srv.replay(descs, [3.0 * i for i in range(len(descs))])
        assert srv.drain() == 1
        assert same_bits(torch, y, want)
        srv.replay(descs, [0.0] * len(descs))
        assert srv.drain() == 1
    assert same_bits(torch, y, want)
