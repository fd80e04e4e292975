"""One-token products with host vectors (through borrowed pinned memory, or staged when they do not fit it) against the
same call on device buffers: bit-identical."""
import statistics
import threading
import time

import numpy as np
import pytest
import torch

from memvanta_amd import capi, synth

pytestmark = pytest.mark.gpu


# the input's and the output's limits in the pinned memory (16384 and 65536 floats) on both sides; the smallest rows;
# calls of falling size, so that the memory holds more than the call's own
@pytest.mark.parametrize("ty,k,n", [(synth.Q4_0, 16384, 40), (synth.Q4_0, 16640, 40), (synth.Q8_0, 32, 65536),
                                    (synth.Q8_0, 32, 65537), (synth.Q6_K, 256, 1), (synth.Q4_0, 4096, 11008),
                                    (synth.Q4_0, 288, 100), (synth.F32, 100, 33)])
def test_host_equals_device(ctx, ty, k, n):
    rng = np.random.default_rng(k + n)
    w = (rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02))
    b = w.view(np.uint8).reshape(-1) if ty == synth.F32 else synth.quantize(ty, w).reshape(-1)
    t = ctx.upload("blk.0.attn_q.weight", ty, k, n, b)
    for _ in range(3):
        x = synth.activations(rng, 1, k)[0]
        xd, yd = torch.from_numpy(x).cuda(), torch.empty(n, device="cuda")
        torch.cuda.synchronize()
        ctx.matvec(t, xd, yd)
        ctx.synchronize()
        y = np.full(n + 8, 7.0, np.float32)
        ctx.matvec(t, x, y[:n])
        assert (y[:n].view(np.uint32) == yd.cpu().numpy().view(np.uint32)).all()
        assert (y[n:] == 7.0).all()
    t.free()


def test_two_contexts(ctx):
    """Calls of two contexts in turn, and one of them closed in between."""
    rng = np.random.default_rng(1)
    w = synth.quantize(synth.Q4_0, rng.standard_normal((512, 256), dtype=np.float32)).reshape(-1)
    other = capi.Context(0)
    a, b = (c.upload("blk.0.attn_q.weight", synth.Q4_0, 256, 512, w) for c in (ctx, other))
    x = synth.activations(rng, 2, 256)
    first = [ctx.matvec(a, x[0]), other.matvec(b, x[1])]
    again = [other.matvec(b, x[0]), ctx.matvec(a, x[1])]
    assert (first[0] == again[0]).all() and (first[1] == again[1]).all()
    b.free()
    other.close()
    assert (ctx.matvec(a, x[0]) == first[0]).all()
    a.free()


def test_contexts_in_threads(ctx):
    """Overlapping calls, each thread with a context of its own: more of them than the pool keeps blocks."""
    rng = np.random.default_rng(2)
    w = synth.quantize(synth.Q4_0, rng.standard_normal((300, 288), dtype=np.float32)).reshape(-1)
    x = synth.activations(rng, 10, 288)
    t = ctx.upload("blk.0.attn_q.weight", synth.Q4_0, 288, 300, w)
    want = [ctx.matvec(t, v).copy() for v in x]
    bad = []

    def work(i):
        c = capi.Context(0)
        mine = c.upload("blk.0.attn_q.weight", synth.Q4_0, 288, 300, w)
        for k in range(40):
            j = (i + k) % 10
            if not (c.matvec(mine, x[j]).view(np.uint32) == want[j].view(np.uint32)).all():
                bad.append((i, k))
        mine.free()
        c.close()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(10)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    t.free()
    assert not bad


def test_first_call_of_a_context_pins_no_memory(ctx):
    """Pinning a block takes as long as half of this call; medians of 15 contexts, each one's first call against its
    second (1.65 times as long with a block of its own, 1.0 with a borrowed one)."""
    rng = np.random.default_rng(3)
    w = synth.quantize(synth.Q4_0, rng.standard_normal((288, 288), dtype=np.float32)).reshape(-1)
    t = ctx.upload("blk.0.attn_q.weight", synth.Q4_0, 288, 288, w)
    x, y = synth.activations(rng, 1, 288)[0], np.empty(288, np.float32)
    ctx.matvec(t, x, y)
    first, second = [], []
    for _ in range(15):
        c = capi.Context(0)
        for times in (first, second):
            t0 = time.perf_counter()
            c.matvec(t, x, y)
            times.append(time.perf_counter() - t0)
        c.close()
    t.free()
    assert statistics.median(first) < 1.35 * statistics.median(second), (first, second)
