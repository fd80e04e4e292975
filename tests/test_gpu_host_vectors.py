"""One-token products with host vectors (through the context's pinned memory, or staged when they do not fit it)
against the same call on device buffers: bit-identical."""
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
    """Each context has its own memory: calls of two of them in turn, and one closed in between."""
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
