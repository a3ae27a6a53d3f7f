"""The order of the allocation-free overlap with everything else on the GPU:
calls of several contexts, what the caller's stream does to X before the call
and to X and S after it, and stream capture.  Nothing waits on the host
between the calls.

Each result is compared with the 64-bit product of its own operands: sums over
npw products as in the other overlap tests, 1e-13 of the largest element.
"""
import ctypes as C

import numpy as np
import pytest
import torch

from derek_amd import lib
from tests.conftest import assert_close

pytestmark = pytest.mark.gpu

SIZES = [(1503, 10, 10), (1503, 20, 20), (40011, 48, 33), (62669, 160, 160)]


def block(rng, m, npw):
    return rng.normal(size=(m, npw)) + 1j * rng.normal(size=(m, npw))


def context():
    return lib.Context((8, 8, 8), 1, 1, 1.0, 1)


def overlap(ctx, x, y, s, stream=None):
    """s (n, m) = the transpose of X^H Y, X (m, npw), Y (n, npw), all on the device."""
    a = (C.c_int64(x.shape[1]), C.c_int32(x.shape[0]), C.c_int32(y.shape[0]), C.c_void_p(x.data_ptr()),
         C.c_void_p(y.data_ptr()), C.c_void_p(s.data_ptr()))
    if stream is None:
        lib.check(ctx.lib.derek_hip_overlap_noalloc(ctx.h, *a))
    else:
        lib.check(ctx.lib.derek_hip_overlap_noalloc_on(ctx.h, C.c_void_p(stream.cuda_stream), *a))


def result(s):
    return s.cpu().numpy().T


def empty(m, n):
    return torch.full((n, m), complex(np.nan, np.nan), dtype=torch.complex128, device="cuda")


@pytest.mark.parametrize("npw,m,n", SIZES)
def test_contexts_in_turn(npw, m, n):
    print("contexts in turn", npw, m, n, flush=True)
    rng = np.random.default_rng(npw + m)
    host = [(block(rng, m, npw), block(rng, n, npw)) for _ in range(3)]
    dev = [tuple(torch.from_numpy(a).cuda() for a in p) for p in host]
    ctx = [context() for _ in host]
    out = [[empty(m, n) for _ in range(8)] for _ in host]
    torch.cuda.synchronize()
    for r in range(8):
        for k, (x, y) in enumerate(dev):
            overlap(ctx[k], x, y, out[k][r])
    torch.cuda.synchronize()
    for k, (x, y) in enumerate(host):
        ref = x.conj() @ y.T
        for r in range(8):
            assert_close(result(out[k][r]), ref, 1e-13, f"context {k} call {r}")
    for c in ctx:
        c.close()


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("side", [False, True])
@pytest.mark.parametrize("npw,m,n", SIZES)
def test_callers_stream(npw, m, n, side, shared):
    """X and Y are written, after other work, on the caller's stream right
    before the call; right after it S is read there and X is overwritten.
    shared: the caller has asked for the context's stream before."""
    print("caller's stream", npw, m, n, "side" if side else "default", "shared" if shared else "", flush=True)
    rng = np.random.default_rng(npw + n)
    host = [(block(rng, m, npw), block(rng, n, npw)) for _ in range(4)]
    dev = [tuple(torch.from_numpy(a).cuda() for a in p) for p in host]
    ctx = context()
    if shared:
        assert ctx.stream()
    x, y = torch.zeros_like(dev[0][0]), torch.zeros_like(dev[0][1])
    s, got = empty(m, n), []
    busy = torch.zeros(1 << 26, device="cuda")
    stream = torch.cuda.Stream() if side else torch.cuda.current_stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for a, b in dev:
            for _ in range(4):
                busy.add_(1.0)
            x.copy_(a)
            y.copy_(b)
            overlap(ctx, x, y, s, stream if side else None)
            got.append(s.clone())
            x.fill_(0.0)
            y.fill_(0.0)
            s.fill_(0.0)
    torch.cuda.synchronize()
    for (a, b), q in zip(host, got):
        assert_close(result(q), a.conj() @ b.T, 1e-13, "late operands")
    ctx.close()


def test_streams_in_turn():
    """One context called from the default stream and two others in turn, which
    share its scratch; then S read on the context's stream, asked for only after
    the last call; then derek_hip_sync alone before the host reads."""
    print("streams in turn", flush=True)
    npw, m, n = 40011, 48, 33
    rng = np.random.default_rng(3)
    ctx = context()
    streams = [torch.cuda.Stream(), None, torch.cuda.Stream()]
    host = [(block(rng, m, npw), block(rng, n, npw)) for _ in streams]
    dev = [tuple(torch.from_numpy(a).cuda() for a in p) for p in host]
    out = [[empty(m, n) for _ in range(6)] for _ in streams]
    torch.cuda.synchronize()
    for r in range(6):
        for k, (x, y) in enumerate(dev):
            overlap(ctx, x, y, out[k][r], streams[k])
    ctx.sync()
    ref = [x.conj() @ y.T for x, y in host]
    for k in range(3):
        for r in range(6):
            assert_close(result(out[k][r]), ref[k], 1e-13, f"stream {k} call {r}")
    for k, (x, y) in enumerate(dev):
        c, s = context(), empty(m, n)
        torch.cuda.synchronize()
        overlap(c, x, y, s, streams[k])
        own = torch.cuda.ExternalStream(c.stream())
        with torch.cuda.stream(own):
            got = s.clone()
        torch.cuda.synchronize()
        assert_close(result(got), ref[k], 1e-13, "read on the context's stream")
        c.close()
    ctx.close()


@pytest.mark.parametrize("own", [True, False])
def test_captured(own):
    """Recorded on the context's stream with the plain call, or on the caller's
    with the other; replayed with new operands, eager calls between the replays."""
    print("captured on", "the context's stream" if own else "the caller's", flush=True)
    npw, m, n = 40011, 48, 33
    rng = np.random.default_rng(7)
    ctx = context()
    stream = torch.cuda.ExternalStream(ctx.stream()) if own else torch.cuda.Stream()
    x = torch.from_numpy(block(rng, m, npw)).cuda()
    y = torch.from_numpy(block(rng, n, npw)).cuda()
    s, e = empty(m, n), empty(m, n)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream, capture_error_mode="thread_local"):
        overlap(ctx, x, y, s, None if own else stream)
    for r in range(4):
        a, b = block(rng, m, npw), block(rng, n, npw)
        x.copy_(torch.from_numpy(a))
        y.copy_(torch.from_numpy(b))
        s.fill_(0.0)
        e.fill_(0.0)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            g.replay()
        torch.cuda.synchronize()
        overlap(ctx, x, y, e)
        torch.cuda.synchronize()
        assert_close(result(s), a.conj() @ b.T, 1e-13, f"replay {r}")
        assert_close(result(e), a.conj() @ b.T, 1e-13, f"eager call {r}")
    del g
    ctx.close()
