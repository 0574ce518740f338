"""The GEMM's 96-row and 32-row blocks (launches whose 64-row workgroups would leave a round of 256 half empty, or most CUs)
against the passes of at most 9 tokens, bit for bit: rows that end inside a block, a 64-row tile and a 32-value block, K
parts, and a quantised SwiGLU output."""
import numpy as np
import pytest

from test_gpu_kernels import Mat
from zerollm_amd import gguf as G
from zerollm_amd import synth

pytestmark = pytest.mark.gpu


# 8257..12288 rows at 33 tokens and more take 96-row blocks; 5120 and 4161 with two K parts. Fewer rows, and up to 16
# tokens, take 32-row blocks: 4096 and 1089 in four K parts, 2000 in one
@pytest.mark.parametrize("type_,rows,cols", [(G.Q4_K, 12288, 256), (G.Q4_K, 8257, 512), (G.Q5_K, 9000, 256), (G.Q8_0, 8288, 96),
                                             (G.Q4_K, 5120, 4096), (G.Q8_0, 4161, 4096), (G.Q6_K, 4096, 4096),
                                             (G.Q5_K, 1089, 4096), (G.Q4_K, 2000, 512), (G.Q6_K, 70, 256)])
def test_rows_in_96s_equal_short_passes(gpu, type_, rows, cols):
    t = synth.TensorSpec("w", type_, rows, cols, seed=rows)
    m = Mat(type_, synth.tensor_bytes(t, use_device=True), rows, cols)
    X = np.random.default_rng(rows).standard_normal((64, cols)).astype(np.float32)
    want = np.concatenate([m.gemv(X[i:i + 8]) for i in range(0, 64, 8)])
    for M in (10, 16, 17, 33, 48, 61, 64):
        print(f"case type {type_} {rows} x {cols} tokens {M}", flush=True)
        y = m.gemv(X[:M])
        assert (y.view(np.uint32) == want[:M].view(np.uint32)).all(), M
    m.free()


@pytest.mark.parametrize("type_,ff", [(G.Q4_K, 8704), (G.Q8_0, 8288), (G.Q8_0, 12288), (G.Q5_K, 768), (G.Q6_K, 256), (G.Q8_0, 96)])
def test_layer_with_wide_ff_equals_short_passes(gpu, type_, ff):
    spec = synth.build_spec("qwen3", n_embd=256, n_layer=1, n_head=4, n_head_kv=2, head_dim=64, n_ff=ff, vocab=512, ctx_train=256,
                            types=synth.all_type(type_), seed=ff)
    m = synth.build_on_device(spec, ctx=128, kv="f16", max_batch=64, logits_batch=64)
    ids = synth.seeded_ids(61, 5, 512)
    want = np.concatenate([m.forward_batch(ids[i:i + 8], logits="all").copy() for i in range(0, 61, 8)])
    for n in (61, 33, 13):
        print(f"case type {type_} ff {ff} tokens {n}", flush=True)
        m.truncate(0)
        y = m.forward_batch(ids[:n], logits="all")
        assert (y.view(np.uint32) == want[:n].view(np.uint32)).all(), n
    m.close()
