"""The four-wave int8-MFMA prefill GEMM (memvanta_amd/csrc/mvh_gemm_q4.hip) at the edges of its tiles, against the
oracle's FORCE_Q8 chain: bit-exact, the kernel runs the same fma chain on exact block sums."""
import numpy as np
import pytest

from conftest import assert_bitexact
from memvanta_amd import capi, synth

pytestmark = pytest.mark.gpu


# rows x tokens on both sides of the 768 K line; tokens that take the 32- and the 64-token tiles, one past and one
# short of them; rows one past and one short of the 64- and 128-row tiles; the shortest K (two K-steps) and odd units
@pytest.mark.parametrize("batch,k,n", [(192, 256, 4096), (191, 256, 4096), (193, 512, 4161), (97, 256, 8191),
                                       (33, 768, 24577), (65, 256, 12223), (512, 256, 1537), (385, 1280, 2113)])
def test_tile_kernel_bitexact(ctx, oracle, batch, k, n):
    rng = np.random.default_rng(batch + 3 * k + n)
    w = synth.quantize(synth.Q4_0, rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02)).reshape(-1)
    x = synth.activations(rng, batch, k)
    t = ctx.upload("blk.0.attn_q.weight", synth.Q4_0, k, n, w)
    got = ctx.matmul_batch_v06(t, x, capi.MVH_ACT_Q8)
    assert_bitexact(got, oracle.matmul_batch_v06(w, synth.Q4_0, n, k, x, is_ffn=False, force_q8=True),
                    f"B={batch} K={k} N={n}")
    t.free()


def test_tile_kernel_extreme_scales_bitexact(ctx, oracle):
    """Block scales at both ends of binary16 (subnormal, largest, zero, negative) and activations from 1e-30 to 1e30:
    the products of the two scales round, underflow and overflow as the reference's do."""
    rng = np.random.default_rng(5)
    n, k, batch = 4096, 256, 200
    w = synth.quantize(synth.Q4_0, rng.standard_normal((n, k), dtype=np.float32)).reshape(n, k // 32, 18).copy()
    d = np.array([2.0 ** -24, -(2.0 ** -24), 65504.0, 0.0, -0.0, -1.5, 3.0e-5], np.float16)
    w[:, :, :2] = d[rng.integers(0, len(d), (n, k // 32))].view(np.uint8).reshape(n, k // 32, 2)
    x = synth.activations(rng, batch, k) * (10.0 ** rng.integers(-30, 31, (batch, 1))).astype(np.float32)
    t = ctx.upload("blk.0.attn_q.weight", synth.Q4_0, k, n, w.reshape(-1))
    got = ctx.matmul_batch_v06(t, x, capi.MVH_ACT_Q8)
    assert_bitexact(got, oracle.matmul_batch_v06(w.reshape(-1), synth.Q4_0, n, k, x, is_ffn=False, force_q8=True), "scales")
    t.free()
