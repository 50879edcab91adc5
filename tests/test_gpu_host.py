"""Calls on pageable host memory of every one-workgroup size: the same bits as the device batch call,
each call its own answer when calls follow each other at once, from host and device inputs, on an
idle device and behind queued work."""
import numpy as np
import pytest

from test_gpu_parity import C, ctx, make_input, out_len, torch  # noqa: F401

pytestmark = pytest.mark.gpu

SIZES = [(k, p) for k in ("cfwd", "cinv") for p in range(2, 16)] + [(k, p) for k in ("rfwd", "rinv") for p in range(3, 17)]


def calls(ctx, kind, n):  # noqa: F811
    batch = {"cfwd": ctx.complex_forward_batch, "cinv": ctx.complex_inverse_batch,
             "rfwd": ctx.real_forward_batch, "rinv": ctx.real_inverse_batch}[kind]
    tmp = np.empty(n + 2, np.float32)
    one = {"cfwd": ctx.complex_forward, "cinv": ctx.complex_inverse, "rfwd": ctx.real_forward,
           "rinv": lambda m, x, y: ctx.real_inverse(m, x, y, tmp)}[kind]
    return batch, one


@pytest.mark.parametrize("kind,log2n", SIZES)
def test_pageable_calls(torch, ctx, kind, log2n):  # noqa: F811
    n, count = 1 << log2n, 20
    x = make_input(kind, n, count, 0x405 + log2n)
    length = out_len(kind, n)
    batch, one = calls(ctx, kind, n)
    xd = torch.from_numpy(x).cuda()
    yd = torch.empty(count, length, device="cuda")
    for i in range(count):
        assert batch(n, 1, xd[i], yd[i]) == 1
    torch.cuda.synchronize()
    want = yd.cpu().numpy().view(np.int32).reshape(count, length)
    guard = 32
    buf = np.full((count, guard + length + guard), -7.0, np.float32)
    for i in range(count):                      # no pause between the calls
        assert one(n, np.ascontiguousarray(x[i]), buf[i, guard:guard + length]) == 1
    assert np.array_equal(buf[:, guard:-guard].view(np.int32), want)
    assert np.all(buf[:, :guard] == -7.0) and np.all(buf[:, -guard:] == -7.0)
    got = np.empty(length, np.float32)
    assert one(n, xd[2], got) == 1              # device input, pageable output
    assert np.array_equal(got.view(np.int32), want[2])
    # behind work that fills the device for longer than the call polls
    big = torch.zeros(1 << 26, device="cuda")
    for _ in range(40):
        big.add_(1.0)
    assert one(n, np.ascontiguousarray(x[3]), got) == 1
    assert np.array_equal(got.view(np.int32), want[3])
    torch.cuda.synchronize()


@pytest.mark.parametrize("kind,log2n", [("cfwd", 3), ("rinv", 6), ("rfwd", 10), ("cinv", 13), ("rfwd", 16)])
def test_pinned_input_rewritten_between_calls(torch, ctx, kind, log2n):  # noqa: F811
    n, count = 1 << log2n, 12
    x = torch.from_numpy(make_input(kind, n, count, 0x917 + log2n))
    length = out_len(kind, n)
    batch, one = calls(ctx, kind, n)
    xd = x.cuda()
    want = torch.empty(count, length, device="cuda")
    for i in range(count):
        assert batch(n, 1, xd[i], want[i]) == 1
    torch.cuda.synchronize()
    want = want.cpu().numpy().view(np.int32)
    pinned = torch.empty(x[0].numel(), pin_memory=True)
    pinned_out = torch.empty(length, pin_memory=True)
    got = np.empty(length, np.float32)
    for i in range(count):                      # pinned to pageable, pinned to pinned every third time
        pinned.copy_(x[i])
        out = pinned_out if i % 3 == 2 else got
        assert one(n, pinned, out) == 1
        assert np.array_equal((pinned_out.numpy() if i % 3 == 2 else got).view(np.int32), want[i]), i
