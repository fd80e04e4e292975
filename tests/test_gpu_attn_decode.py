"""One-token attention over the paged cache (the scores and value kernels of the C ABI's decode call) against the
batched call with one token, which runs the same chains in other kernels: bit-identical, at the edges of the score
blocks (64 positions), the softmax's 256 threads, the V tiles (128 or 256 rows) and the four-row groups."""
import numpy as np
import pytest

from memvanta_amd import capi

pytestmark = pytest.mark.gpu


# (heads, kv heads, head_dim): the compiled head sizes, others that are whole 32-element slices, a group of 8
@pytest.mark.parametrize("kv_type", [capi.MVH_KV_F32, capi.MVH_KV_F16, capi.MVH_KV_Q8])
@pytest.mark.parametrize("n_head,n_kv,hd,page", [(4, 4, 128, 128), (8, 1, 64, 16), (2, 2, 32, 7), (6, 2, 96, 64),
                                                 (2, 1, 512, 128)])
def test_equals_one_token_batch(ctx, kv_type, n_head, n_kv, hd, page):
    rng = np.random.default_rng(hd + page)
    n = 1100
    k, v = (rng.standard_normal((n, n_kv * hd), dtype=np.float32) for _ in range(2))
    kv = ctx.kv_cache(1, n_kv * hd, page, n, kv_type=kv_type)
    kv.write(0, 0, k, v)
    q = rng.standard_normal((1, n_head * hd), dtype=np.float32) * np.float32(3)
    for pos in (0, 1, 3, 4, 62, 63, 64, 127, 128, 130, 254, 255, 256, 257, 511, 512, 700, 1023, 1024, 1099):
        got = kv.attn_decode(0, q[0], pos, n_head, n_kv, hd)
        want = kv.attn_batch(0, q, pos, 1, n_head, n_kv, hd)
        assert (got.reshape(-1).view(np.uint32) == want.reshape(-1).view(np.uint32)).all(), pos
    kv.close()


@pytest.mark.parametrize("kv_type", [capi.MVH_KV_F32, capi.MVH_KV_F16, capi.MVH_KV_Q8])
def test_weights_past_the_lds(ctx, kv_type):
    """Positions around which the weights no longer fit beside the V tiles (7.8 K; 12 K for Q8): both routes agree."""
    rng = np.random.default_rng(2)
    n_head, hd, n = 2, 64, 12100
    k, v = (rng.standard_normal((n, n_head * hd), dtype=np.float32) for _ in range(2))
    kv = ctx.kv_cache(1, n_head * hd, 128, n, kv_type=kv_type)
    kv.write(0, 0, k, v)
    q = rng.standard_normal((1, n_head * hd), dtype=np.float32)
    for pos in (7795, 7806, 7807, 7808, 7820, 12020, 12030, 12031, 12032, 12099):
        got = kv.attn_decode(0, q[0], pos, n_head, n_head, hd)
        want = kv.attn_batch(0, q, pos, 1, n_head, n_head, hd)
        assert (got.reshape(-1).view(np.uint32) == want.reshape(-1).view(np.uint32)).all(), pos
    kv.close()


def test_infinite_rows(ctx):
    """Rows past the position are not read into the result, an infinite value row of it is."""
    rng = np.random.default_rng(3)
    n_head, hd, n = 2, 128, 300
    k, v = (rng.standard_normal((n, n_head * hd), dtype=np.float32) for _ in range(2))
    v[260:] = np.inf
    kv = ctx.kv_cache(1, n_head * hd, 64, n, kv_type=capi.MVH_KV_F32)
    kv.write(0, 0, k, v)
    q = rng.standard_normal(n_head * hd, dtype=np.float32)
    assert np.isfinite(kv.attn_decode(0, q, 259, n_head, n_head, hd)).all()
    assert (kv.attn_decode(0, q, 260, n_head, n_head, hd) == np.inf).all()
    kv.close()
