"""Prefill chunks joined into one step, and what a joined step must not change: the state a refused chunk leaves
behind, and the independence of a token from the rows of later ones."""
import dataclasses

import numpy as np
import pytest
import torch

from memvanta_amd import capi, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tiny(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("joined") / "tiny.gguf")
    synth.write_model(dataclasses.replace(synth.TINY, ctx=384), path, seed=1234)
    return path


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("bad,batch,done", [(45, 8, 40), (0, 16, 0), (79, 16, 64), (33, 32, 32)])
def test_refused_chunk_leaves_the_earlier_ones(tiny, mode, bad, batch, done):
    """The chunks before the one with a bad token complete, whichever steps they were joined into."""
    prompt = synth.prompt_tokens(3, 80).astype(np.int32)
    m = capi.Model(tiny, ctx=256, act_mode=mode, max_batch=32)
    broken = prompt.copy()
    broken[bad] = 32000
    with pytest.raises(capi.MvhError, match="token id out of range"):
        m.prefill(broken, batch)
    assert m.position == done
    got = m.prefill(prompt[done:], batch).copy()
    m.reset()
    assert (got.view(np.uint32) == m.prefill(prompt, batch).view(np.uint32)).all()
    m.close()


def test_context_end_inside_a_step(tiny):
    m = capi.Model(tiny, ctx=50, max_batch=16)
    with pytest.raises(capi.MvhError, match="context exhausted"):
        m.prefill(synth.prompt_tokens(3, 60).astype(np.int32), 16)
    assert m.position == 48
    m.close()


@pytest.mark.parametrize("mode,n,batch", [(0, 100, 8), (0, 77, 24), (0, 70, 4), (1, 99, 7), (1, 65, 32), (1, 259, 64)])
def test_joined_equals_single_chunks(tiny, mode, n, batch):
    """Steps at and over their 256 tokens, ragged last chunks of 1, 2 and more, and batches that do not join."""
    prompt = synth.prompt_tokens(5, n).astype(np.int32)
    m = capi.Model(tiny, ctx=320, act_mode=mode, max_batch=64)
    got = m.prefill(prompt, batch).copy()
    m.reset()
    for i in range(0, n, batch):
        want = m.prefill(prompt[i:i + batch], batch)
    assert (got.view(np.uint32) == want.view(np.uint32)).all()
    m.close()


def test_buffers_of_a_model_that_never_joins(tiny):
    """In the fp32 numerics chunks of up to 4 tokens never join: buffers for 4, not for a 256-token step (some 20 MB)."""
    used = {}
    for max_batch in (8, 4, 8):  # the first one also takes what a process's first model does
        free = torch.cuda.mem_get_info()[0]
        m = capi.Model(tiny, ctx=256, act_mode=0, max_batch=max_batch)
        used[max_batch] = free - torch.cuda.mem_get_info()[0]
        m.prefill(synth.prompt_tokens(3, 70).astype(np.int32), max_batch)
        m.close()
    assert used[4] + (10 << 20) < used[8]


@pytest.mark.parametrize("kv_type", [capi.MVH_KV_F32, capi.MVH_KV_F16])
@pytest.mark.parametrize("B,pos,last", [(31, 70, 3), (40, 70, 3), (40, 100, 9), (33, 0, 1), (13, 55, 5)])
def test_later_rows_do_not_reach_earlier_tokens(ctx, kv_type, B, pos, last):
    """V rows past a token's position may hold anything: an infinity there leaves the token's output as it was."""
    rng = np.random.default_rng(B)
    n_head, hd = 4, 64
    k, v = (rng.standard_normal((pos + B, n_head * hd), dtype=np.float32) for _ in range(2))
    q = rng.standard_normal((B, n_head * hd), dtype=np.float32)
    outs = []
    for far in (0.5, np.inf):
        v[pos + B - last:] = far
        kv = ctx.kv_cache(1, n_head * hd, 16, 256, kv_type=kv_type)
        kv.write(0, 0, k, v)
        outs.append(kv.attn_batch(0, q, pos, B, n_head, n_head, hd).copy())
        kv.close()
    a, b = (o[: B - last].view(np.uint32) for o in outs)
    assert (a == b).all()


# Shapes whose joined steps leave the fallback kernels: 128-wide heads over Q4_0 (256-token steps of gate|up on the 64-row
# int8 tiles, scores tiles of more than 32 tokens), and 64-wide grouped heads over Q8_0 with a Q6_K down projection
_WIDE = synth.ModelConfig("joined-q4", 1024, 2816, 2, 8, 8, 512, 384, synth.Q4_0, synth.Q4_0, synth.Q4_0)
_GROUPED = synth.ModelConfig("joined-q8-q6", 1024, 2816, 2, 16, 4, 512, 384, synth.Q8_0, synth.Q8_0, synth.Q6_K,
                             synth.Q6_K)


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    out = {}
    for cfg in (_WIDE, _GROUPED):
        out[cfg.name] = str(tmp_path_factory.mktemp("joined") / (cfg.name + ".gguf"))
        synth.write_model(cfg, out[cfg.name], seed=5, device="cuda", digest=False)
    return out


def _joined_equals_single(path, mode, kv_type, n, batch, vocab):
    prompt = np.random.default_rng(n).integers(0, vocab, n).astype(np.int32)
    m = capi.Model(path, act_mode=mode, max_batch=64, kv_type=kv_type)
    got = m.prefill(prompt, batch).copy()
    m.reset()
    for i in range(0, n, batch):
        want = m.prefill(prompt[i:i + batch], batch)
    assert np.isfinite(got).all()
    assert (got.view(np.uint32) == want.view(np.uint32)).all()
    m.close()


@pytest.mark.parametrize("name,mode,kv,n,batch", [
    ("joined-q4", 1, capi.MVH_KV_F16, 300, 32), ("joined-q4", 1, capi.MVH_KV_Q8, 261, 16),
    ("joined-q4", 0, capi.MVH_KV_F32, 275, 8), ("joined-q4", 0, capi.MVH_KV_F16, 230, 64),
    ("joined-q8-q6", 0, capi.MVH_KV_F16, 300, 32), ("joined-q8-q6", 0, capi.MVH_KV_Q8, 261, 32),
    ("joined-q8-q6", 1, capi.MVH_KV_F16, 90, 5), ("joined-q8-q6", 1, capi.MVH_KV_F32, 77, 24)])
def test_joined_equals_single_chunks_wide(shapes, name, mode, kv, n, batch):
    _joined_equals_single(shapes[name], mode, kv, n, batch, 512)


def _order_sensitive(path, monkeypatch):
    """A layer whose Q6_K q|k|v sums hold two huge terms that cancel (equal weights and embeddings in columns 3 and 300,
    norm weights +-2^45), so that the order of the double sum shows in the result's leading digits."""
    cfg = synth.ModelConfig("q6k-sums", 512, 1024, 1, 8, 8, 64, 128, synth.Q6_K, synth.F32, synth.Q6_K)
    rng = np.random.default_rng(9)

    def content(name, dims):
        if name == "blk.0.attn_norm.weight":
            v = np.ones(512, np.float32)
            v[3], v[300] = 2.0 ** 45, -(2.0 ** 45)
            return v
        m = rng.standard_normal((dims[1], 512), dtype=np.float32)
        if name == "token_embd.weight":
            m[:, 300] = m[:, 3]
            return m
        m = np.clip(m * np.float32(0.02), -0.05, 0.05)
        m[:, 15::16] = 0.062  # every 16-element scale is the same
        m[:, 300] = m[:, 3] = 0.04
        return synth.quantize(synth.Q6_K, m)

    class Writer(synth.GgufWriter):
        def add_tensor(self, name, dims, ty, nbytes, produce):
            if name in ("token_embd.weight", "blk.0.attn_norm.weight", "blk.0.attn_q.weight", "blk.0.attn_k.weight",
                        "blk.0.attn_v.weight"):
                b = content(name, dims).tobytes()
                produce = lambda: iter([b])
            super().add_tensor(name, dims, ty, nbytes, produce)

    monkeypatch.setattr(synth, "GgufWriter", Writer)
    synth.write_model(cfg, path, seed=3, digest=False)


@pytest.mark.parametrize("mode,n,batch", [(0, 37, 32), (0, 40, 8), (0, 69, 64), (0, 87, 32), (0, 77, 32), (1, 24, 3),
                                          (1, 50, 20), (1, 72, 24)])
def test_q6k_sums_keep_their_order(tmp_path, monkeypatch, mode, n, batch):
    """Q6_K chunks whose tokens go one at a time do not join a step that would group them: last chunks of 5 and 8
    beside whole groups, chunks of 3 and 8, 20 (16 and 4); 23, 13 and 24 tokens are grouped alone as in a step."""
    path = str(tmp_path / "q6k.gguf")
    _order_sensitive(path, monkeypatch)
    _joined_equals_single(path, mode, capi.MVH_KV_F16, n, batch, 64)
