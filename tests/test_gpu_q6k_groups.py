"""Q6_K over token counts around the 16-token groups of the f64 matrix-pipe kernel: a double sum rounded once, so
equal to the oracle's within one unit in the last place (another order of a double sum)."""
import numpy as np
import pytest

from memvanta_amd import capi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,k,n", [(5, 256, 17), (8, 2048, 33), (9, 2048, 33), (15, 512, 1), (16, 256, 15),
                                       (20, 512, 31), (21, 512, 31), (31, 768, 16), (37, 2048, 100), (5, 4096, 2048),
                                       (6, 4096, 2048), (70, 2304, 65)])
def test_token_groups(ctx, oracle, batch, k, n):
    rng = np.random.default_rng(batch + k + n)
    w = synth.quantize(synth.Q6_K, rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02)).reshape(-1)
    x = synth.activations(rng, batch, k)
    t = ctx.upload("blk.0.ffn_down.weight", synth.Q6_K, k, n, w)
    want = oracle.matmul_batch(w, synth.Q6_K, n, k, x)
    for got in (ctx.matmul_batch(t, x), ctx.matmul_batch_v06(t, x, capi.MVH_ACT_Q8)):
        assert (np.abs(got - want) <= np.spacing(np.abs(want))).all()
    t.free()
