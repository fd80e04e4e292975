"""The batched fp32-activation products on the f32 matrix pipe (memvanta_amd/csrc/mvh_gemm_f32.hip): bit-exact
against the oracle at the edges of their tiles.

Both numerics are fma chains in a fixed order and the kernels run the same chains, so the tolerance is none."""
import numpy as np
import pytest
import torch

from conftest import assert_bitexact
from memvanta_amd import capi, synth

pytestmark = pytest.mark.gpu


def _case(rng, ty, n, k, batch):
    w = synth.quantize(ty, rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02)).reshape(-1)
    return w, synth.activations(rng, batch, k)


# rows / tokens: one, just below, at and past the 16 / 32 / 48-row and 16 / 32-token tiles; K: one block, one unit less
# or more than whole 8-block units (the 2-byte staging), two units and the shortest whole unit (no next unit to fetch)
@pytest.mark.parametrize("ty", [synth.Q4_0, synth.Q8_0])
@pytest.mark.parametrize("batch,k,n", [(4, 32, 1), (16, 288, 17), (20, 224, 33), (4, 256, 15), (36, 512, 49),
                                       (68, 768, 31), (28, 1024, 4096), (12, 1280, 16400), (100, 256, 8200),
                                       (512, 256, 100), (32, 256, 11008)])
def test_chain_tiles_bitexact(ctx, oracle, ty, batch, k, n):
    rng = np.random.default_rng(batch * 3 + k + n + ty)
    w, x = _case(rng, ty, n, k, batch)
    t = ctx.upload("blk.0.attn_q.weight", ty, k, n, w)
    got = ctx.matmul_batch_v06(t, x, capi.MVH_ACT_REF)
    assert_bitexact(got, oracle.matmul_batch_v06(w, ty, n, k, x, is_ffn=False, force_q8=False), f"B={batch} K={k} N={n}")
    t.free()


# rows of up to three blocks have a kernel of their own, four and more the matrix pipe; rows at the edges of its 256
@pytest.mark.parametrize("ty", [synth.Q4_0, synth.Q8_0])
@pytest.mark.parametrize("batch,k,n", [(4, 32, 256), (8, 32, 257), (12, 64, 1000), (16, 96, 255), (4, 96, 1),
                                       (24, 128, 257), (8, 160, 300)])
def test_short_rows_bitexact(ctx, oracle, ty, batch, k, n):
    test_chain_tiles_bitexact(ctx, oracle, ty, batch, k, n)


def _us(call, ctx):
    """Time of a call: 40 of them queued behind other work, so that launching them takes no part."""
    long = torch.ones(1 << 28, device="cuda")
    stream = torch.cuda.ExternalStream(ctx.stream)
    torch.cuda.synchronize()
    best = 1e9
    for _ in range(2):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        with torch.cuda.stream(stream):
            for _ in range(8):
                long.mul_(1.0)
            begin.record(stream)
            for _ in range(40):
                call()
            end.record(stream)
        end.synchronize()
        best = min(best, begin.elapsed_time(end) * 1e3 / 40)
    return best


def test_short_rows_cost_by_their_length(ctx):
    """A row of one block costs well under half of one of four (0.4 times seen), not as much as a whole 8-block unit."""
    us = {}
    for k in (32, 128):
        w, x = _case(np.random.default_rng(k), synth.Q4_0, 11008, k, 512)
        t = ctx.upload("blk.0.attn_q.weight", synth.Q4_0, k, 11008, w)
        x, y = torch.from_numpy(x).cuda(), torch.empty((512, 11008), device="cuda")
        us[k] = _us(lambda: ctx.matmul_batch_v06(t, x, capi.MVH_ACT_REF, y), ctx)
        t.free()
    assert us[32] < 0.6 * us[128], us


# tokens: the first batch on this kernel, one short of and past its 16-token tiles; rows at the edges of 16 and 32, on
# both sides of the 512-workgroup line; K: half a round of 16 blocks, one, one and a half, many
@pytest.mark.parametrize("ty", [synth.Q4_0, synth.Q8_0])
@pytest.mark.parametrize("batch,k,n", [(4, 256, 1), (5, 512, 17), (15, 768, 31), (16, 1024, 33), (17, 4096, 100),
                                       (7, 4352, 4096), (64, 256, 4097), (250, 512, 1025), (33, 1280, 5600)])
def test_block_sums_bitexact(ctx, oracle, ty, batch, k, n):
    rng = np.random.default_rng(batch * 5 + k + n + ty)
    w, x = _case(rng, ty, n, k, batch)
    t = ctx.upload("blk.0.attn_q.weight", ty, k, n, w)
    want = oracle.matmul_batch(w, ty, n, k, x)
    assert_bitexact(ctx.matmul_batch(t, x), want, f"B={batch} K={k} N={n}")
    if ty == synth.Q8_0:
        assert_bitexact(ctx.matmul_batch_v06(t, x, capi.MVH_ACT_Q8), want, f"v06 q8 B={batch} K={k} N={n}")
    t.free()


# rows x tokens on both sides of the lines between the matrix pipe and the per-token kernels: none up to K = 2048, 5 K up
# to 3072, 12 K (Q8_0) or 14 K (Q4_0) up to 4608, 8 K beyond (there with 4096 rows or 8 tokens)
@pytest.mark.parametrize("ty", [synth.Q4_0, synth.Q8_0])
@pytest.mark.parametrize("batch,k,n", [(4, 2048, 33), (4, 2304, 1280), (4, 2304, 1281), (5, 3072, 1025),
                                       (8, 3328, 1536), (8, 3328, 1537), (7, 3328, 2048), (7, 3328, 2049),
                                       (16, 4608, 769), (8, 4864, 1023), (8, 4864, 1024), (7, 8192, 1200),
                                       (4, 5120, 4096), (17, 8192, 600)])
def test_block_sums_where_they_pay_bitexact(ctx, oracle, ty, batch, k, n):
    test_block_sums_bitexact(ctx, oracle, ty, batch, k, n)


@pytest.mark.parametrize("ty,few,many,k", [(synth.Q8_0, 2, 8, 8192), (synth.Q4_0, 2, 11, 8192), (synth.Q6_K, 2, 9, 5632),
                                           (synth.Q6_K, 2, 15, 11008)])
def test_few_rows_cost_by_their_tokens(ctx, ty, few, many, k):
    """A matrix of 64 rows leaves most of the chip idle, so more tokens of it cost next to nothing (1.0 to 1.1 times
    seen), unless they take a tile whose time is the same however full it is (4 to 5 times)."""
    w, x = _case(np.random.default_rng(k), ty, 64, k, many)
    t = ctx.upload("blk.0.attn_q.weight", ty, k, 64, w)
    x, y = torch.from_numpy(x).cuda(), torch.empty((many, 64), device="cuda")
    us = {n: _us(lambda: ctx.matmul_batch(t, x[:n], y[:n]), ctx) for n in (few, many)}
    t.free()
    assert us[many] < 2.5 * us[few], us
