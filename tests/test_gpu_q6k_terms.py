"""Q6_K products at the ends of their integer range: codes 0 and 63 (values -32 and 31), group scales -128 and 127 and
activation codes of +-127 give block sums of up to 32 * 127 * 32 * 128 = 16,646,144 in the kernels' integer arithmetic."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_kernels import Mat
from zerollm_amd import gguf as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scales", [(-128, -128), (127, 127), (-128, 127)])
@pytest.mark.parametrize("code", [0, 63])
def test_extreme_codes_and_scales(gpu, code, scales):
    rows, cols = 70, 1536  # a ragged second tile; 24 slabs
    blk = np.zeros((rows * cols // 256, 210), np.uint8)
    blk[:, :192] = 255 if code else 0
    blk[:, 192:208] = np.tile(np.array(scales, np.int8).view(np.uint8), 8)
    blk[:, 208:210] = np.frombuffer(np.float16(0.001).tobytes(), np.uint8)
    m = Mat(G.Q6_K, blk.ravel(), rows, cols)
    X = np.where(np.arange(64)[:, None] % 2 == 0, 1.0, -1.0) * np.linspace(0.5, 2, cols // 32).repeat(32)[None, :]
    X[3, ::3] *= -1  # mixed signs
    X = X.astype(np.float32)
    want = np.stack([O.matvec(G.Q6_K, blk.ravel(), rows, cols, X[t]) for t in range(64)])
    for M in (1, 5, 9, 10, 64):
        print(f"case q6_k codes {code} scales {scales} tokens {M}", flush=True)
        y = m.gemv(X[:M])
        # sums of 24 slabs in f64 either way, rounded once to f32: one unit in the last place at most
        assert np.abs(y - want[:M]).max() <= 2.0 ** -23 * np.abs(want).max(), M
        assert (y.view(np.uint32) == want[:M].view(np.uint32)).mean() >= 0.999, M
    m.free()
