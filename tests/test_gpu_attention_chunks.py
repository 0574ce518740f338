"""Attention rows longer than one chunk of 2048 positions, whose chunks run side by side and are joined in float64: the
same bits in passes of every size, across the chunk borders; the reference's f32 chain bit for bit up to 2048 positions,
and beyond it within the criterion the repository holds reordered attention sums to."""
import numpy as np
import pytest

from oracle import oracle as O
from zerollm_amd import synth

pytestmark = pytest.mark.gpu


def _spec(head_dim, layers=1):
    kw = dict(arch="qwen3", n_embd=256, n_head=4, n_head_kv=2, head_dim=head_dim, n_ff=512, vocab=2048, ctx_train=16384,
              types=synth.all_type(synth.gguf.Q8_0), seed=3)
    return synth.build_spec(n_layer=layers, **kw)


@pytest.mark.parametrize("head_dim,kv", [(64, "f16"), (128, "f16"), (128, "f32"), (256, "f16")])
def test_rows_across_chunk_borders_are_the_same_in_passes_of_every_size(gpu, head_dim, kv):
    """Rows of 2046 .. 2051 and 4095 .. 4098 positions: token by token and in passes of 2 and 5 (lane chains), in passes
    of 16 (16-row blocks of the matrix-core form) and 64 tokens."""
    spec = _spec(head_dim)
    ids = synth.seeded_ids(4200, 21, spec.vocab)
    want = {}
    for n in (1, 2, 5, 16, 64):
        print(f"case chunk borders head {head_dim} kv {kv} passes of {n}", flush=True)
        m = synth.build_on_device(spec, ctx=4224, kv=kv, max_batch=64, logits_batch=64)
        for start, end in ((2046, 2110), (4064, 4128)):
            m.truncate(0)
            for i in range(0, start, 64):
                m.forward_batch(ids[i:min(i + 64, start)], logits="none")
            rows = np.concatenate([m.forward_batch(ids[i:min(i + n, end)], logits="all").copy() for i in range(start, end, n)])
            if n == 1:
                want[start] = rows
            assert (rows.view(np.uint32) == want[start].view(np.uint32)).all(), (n, start)
        m.close()


def test_rows_up_to_a_chunk_are_the_reference_chain_and_longer_ones_stay_close(gpu):
    spec = _spec(64)
    ids = synth.seeded_ids(2060, 22, spec.vocab)
    arrays = {t.name: synth.tensor_bytes(t, use_device=True) for t in spec.tensors}
    O.set_threads(8)
    ref = O.OracleModel(O.ArraySource(spec, arrays), ctx=4096, kv="f16", threads=8)
    for t in ids[:2044]:
        ref.forward(t, logits=False)
    want = np.stack([ref.forward(t) for t in ids[2044:]]).astype(np.float64)
    ref.close()
    print("case chunk against the reference chain", flush=True)
    m = synth.build_on_device(spec, ctx=4096, kv="f16")
    for i in range(0, 2044, 16):
        m.forward_batch(ids[i:min(i + 16, 2044)], logits="none")
    got = np.stack([m.forward(t).copy() for t in ids[2044:]]).astype(np.float64)
    m.close()
    # rows 0 .. 3 have 2045 .. 2048 positions; float64 sums in another order may move a float32 result by an ulp
    assert np.mean(got[:4] == want[:4]) >= 0.999 and np.abs(got[:4] - want[:4]).max() <= 1e-6 * np.abs(want).max()
    diff = np.abs(got - want)
    cos = (got * want).sum(1) / np.sqrt((got * got).sum(1) * (want * want).sum(1))
    assert (diff.max(1) <= 2e-2 * np.abs(want).max(1)).all() and cos.min() > 0.9995


@pytest.mark.parametrize("ctx", [37, 2049, 4099])
def test_passes_that_end_at_the_last_position_of_the_cache(gpu, ctx):
    """A cache whose last positions are not a multiple of 4 (nor of a chunk), filled to the end by 16-token passes and
    token by token."""
    spec = _spec(64)
    ids = synth.seeded_ids(ctx, 23, spec.vocab)
    print(f"case cache end {ctx}", flush=True)
    m = synth.build_on_device(spec, ctx=ctx, kv="f16", max_batch=64, logits_batch=64)
    for i in range(0, ctx - 32, 64):
        m.forward_batch(ids[i:min(i + 64, ctx - 32)], logits="none")
    one = np.stack([m.forward(t).copy() for t in ids[ctx - 32:]])
    for n in (16, 32):
        m.truncate(ctx - 32)
        rows = np.concatenate([m.forward_batch(ids[i:i + n], logits="all").copy() for i in range(ctx - 32, ctx, n)])
        assert (rows.view(np.uint32) == one.view(np.uint32)).all(), n
    m.close()


@pytest.mark.parametrize("head_dim,kv,ctx", [(128, "f16", 36900), (128, "f32", 36900), (256, "f16", 36900), (128, "f16", 9000)])
def test_passes_of_many_blocks_equal_single_tokens(gpu, head_dim, kv, ctx):
    """64-token passes of 8 KV heads, whose weighted sums take 128-dimension blocks (in caches of more than 16 chunks blocks
    that walk them), across chunk borders and at short rows: the bits of single-token passes."""
    spec = synth.build_spec(n_layer=1, arch="qwen3", n_embd=256, n_head=16, n_head_kv=8, head_dim=head_dim, n_ff=512, vocab=2048,
                            ctx_train=65536, types=synth.all_type(synth.gguf.Q8_0), seed=7)
    ids = synth.seeded_ids(ctx, 24, spec.vocab)
    m = synth.build_on_device(spec, ctx=ctx, kv=kv, max_batch=64, logits_batch=64)
    at = 0
    for a in [a for a in (600, 2020, 4064, 32740, 34790, 36830) if a + 64 <= ctx]:
        print(f"case many blocks head {head_dim} kv {kv} cache {ctx} rows from {a}", flush=True)
        for i in range(at, a, 64):
            m.forward_batch(ids[i:min(i + 64, a)], logits="none")
        one = np.stack([m.forward(t).copy() for t in ids[a:a + 64]])
        m.truncate(a)
        rows = m.forward_batch(ids[a:a + 64], logits="all").copy()
        assert (rows.view(np.uint32) == one.view(np.uint32)).all(), a
        at = a + 64
    m.close()
