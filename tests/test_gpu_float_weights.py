"""Float weights: the token groups and the four-row waves, at their edges (rows that end inside a wave or a workgroup, columns
that end inside an unrolled step or are fewer than the lanes), against float64 sums and single-token calls."""
import numpy as np
import pytest

from test_gpu_kernels import Mat, float_raw
from zerollm_amd import gguf as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("type_", [G.F32, G.F16, G.BF16])
@pytest.mark.parametrize("rows,cols", [(1, 33), (70, 511), (4095, 64), (4101, 200), (4100, 1111)])
def test_float_rows_tokens_and_columns(gpu, type_, rows, cols):
    raw = float_raw(type_, rows, cols, rows + cols)
    w = raw.view(np.float32) if type_ == G.F32 else raw.view(np.float16) if type_ == G.F16 else (raw.view(np.uint16).astype(np.uint32) << 16).view(np.float32)
    w = w.astype(np.float64).reshape(rows, cols)
    m = Mat(type_, raw, rows, cols)
    X = np.random.default_rng(cols).standard_normal((19, cols)).astype(np.float32)
    want = X.astype(np.float64) @ w.T
    one = np.concatenate([m.gemv(X[t:t + 1]) for t in range(19)])
    # one rounding to float32, and float64 sums whose order differs (2^-53 a term of the absolute sum)
    bound = 2.0 ** -24 * np.abs(want) + cols * 2.0 ** -52 * (np.abs(X).astype(np.float64) @ np.abs(w).T)
    assert (np.abs(one - want) <= bound).all()
    for M in (2, 3, 5, 8, 9, 16, 19):
        print(f"case type {type_} {rows} x {cols} tokens {M}", flush=True)
        y = m.gemv(X[:M])
        assert (y.view(np.uint32) == one[:M].view(np.uint32)).all(), M
    m.free()
