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


# rows and tokens on both sides of where a group of 9 or 6 tokens is worth a round of workgroups (16384 row-tokens), and
# of 5 beside whole groups (12288): without another round of 256 workgroups, with one
@pytest.mark.parametrize("batch,k,n", [(9, 512, 1820), (9, 512, 1821), (15, 256, 1092), (15, 256, 1093),
                                       (6, 4096, 2730), (6, 4096, 2731), (8, 5632, 2048), (37, 256, 2100),
                                       (37, 256, 2000), (21, 256, 2457), (21, 256, 2458)])
def test_groups_worth_a_round(ctx, oracle, batch, k, n):
    test_token_groups(ctx, oracle, batch, k, n)
