"""The loads of the matrix-core weighted sums stay inside the scores and the V cache at the ends of both."""
import os
import re

import numpy as np
import pytest

from zerollm_amd import synth

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zerollm_amd", "csrc", "zl_attn.hip")


def test_requests_past_a_blocks_last_piece_have_no_scalar_offset():
    """k_attn_av_mm requests pieces past the last one of a block. The range check of a buffer load certainly covers its
    vector offset; a scalar offset may be left out of it or exceed the resource. (In a 128-position cache, two query heads
    per KV head, the last row block of a 17-token pass requests scores 384 floats on in a resource of 256.)"""
    loads = re.findall(r"raw_buffer_load_b\d+\((?:[^()]|\([^()]*\))*\)", open(SRC).read())
    assert loads and all(l.endswith(", 0, 0)") for l in loads), loads


@pytest.mark.gpu
@pytest.mark.parametrize("head_dim,kv", [(64, "f16"), (64, "f32"), (128, "f16"), (256, "f16")])
@pytest.mark.parametrize("ctx,n", [(128, 17), (130, 17), (2064, 16), (2065, 17)])
def test_passes_at_the_end_of_the_last_rows(gpu, head_dim, kv, ctx, n):
    """The last layer's last KV head and the last scores row, with the pass ending at the cache's last position: the rows
    of single-token passes, bit for bit."""
    spec = synth.build_spec(n_layer=1, arch="qwen3", n_embd=256, n_head=4, n_head_kv=2, head_dim=head_dim, n_ff=512,
                            vocab=2048, ctx_train=16384, types=synth.all_type(synth.gguf.Q8_0), seed=5)
    ids = synth.seeded_ids(ctx, 31, spec.vocab)
    print(f"case cache end {ctx} head {head_dim} kv {kv} pass of {n}", flush=True)
    m = synth.build_on_device(spec, ctx=ctx, kv=kv, max_batch=n, logits_batch=n)
    for i in range(0, ctx - n, 16):
        m.forward_batch(ids[i:min(i + 16, ctx - n)], logits="none")
    one = np.stack([m.forward(t).copy() for t in ids[ctx - n:]])
    m.truncate(ctx - n)
    rows = m.forward_batch(ids[ctx - n:], logits="all").copy()
    m.close()
    assert (rows.view(np.uint32) == one.view(np.uint32)).all()
