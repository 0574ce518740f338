"""Short f32 rows that a matvec quantises in its own workgroups, against the call that quantises them in a launch before
(zl_mat_gemv), bit for bit: chunks per wave up to and past the limit, half slabs, uneven K parts, blocks of zeros."""
import ctypes as C

import numpy as np
import pytest
import torch

from test_gpu_kernels import Mat, float_raw
from zerollm_amd import gguf as G
from zerollm_amd import synth
from zerollm_amd._lib import call

pytestmark = pytest.mark.gpu

# 4096 columns: two slabs per wave (4 tokens reach 8 chunks, 5 pass it); 2816 and 2304: K parts of 11 and 9 slabs
SHAPES = [(t, r, c) for t in (G.Q8_0, G.Q4_0, G.Q5_0, G.Q4_K, G.Q5_K, G.Q6_K)
          for r, c in ((64, 256), (70, 768), (1100, 2304), (1500, 2816), (2048, 4096))]
SHAPES += [(t, 100, c) for t in (G.Q8_0, G.Q4_0, G.Q5_0) for c in (32, 96, 1056)] + [(G.F16, 70, 100), (G.F32, 33, 511)]


@pytest.mark.parametrize("type_,rows,cols", SHAPES)
def test_fused_rows_equal_a_launch_before(gpu, type_, rows, cols):
    raw = (float_raw(type_, rows, cols, rows) if type_ in (G.F16, G.F32)
           else synth.tensor_bytes(synth.TensorSpec("w", type_, rows, cols, seed=rows + cols), use_device=True))
    m = Mat(type_, raw, rows, cols)
    X = np.random.default_rng(cols).standard_normal((9, cols)).astype(np.float32)
    X[:, : min(cols, 32)] = 0
    X[1] *= 1e-30
    X[2, ::7] *= 1e4
    x, y = torch.from_numpy(X).cuda(), torch.empty((9, rows), device="cuda")
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    for M in range(1, 10):
        print(f"case type {type_} {rows} x {cols} tokens {M}", flush=True)
        y.fill_(7.0)
        torch.cuda.synchronize()
        call("zl_mat_gemv_noalloc", m.h, C.c_void_p(x.data_ptr()), M, C.c_void_p(y.data_ptr()), C.c_void_p(st.cuda_stream))
        st.synchronize()
        want = m.gemv(X[:M])
        assert (y[:M].cpu().numpy().view(np.uint32) == want.view(np.uint32)).all(), M
        assert bool((y[M:] == 7.0).all())
    m.free()


@pytest.mark.parametrize("type_", [G.Q8_0, G.Q4_K, G.Q6_K, G.F16])
def test_result_over_the_rows(gpu, type_):
    n = 256
    raw = (float_raw(type_, n, n, 3) if type_ == G.F16
           else synth.tensor_bytes(synth.TensorSpec("w", type_, n, n, seed=3), use_device=True))
    m = Mat(type_, raw, n, n)
    X = np.random.default_rng(3).standard_normal((3, n)).astype(np.float32)
    st = torch.cuda.Stream()
    for M in (2, 3):
        print(f"case type {type_} tokens {M} in place", flush=True)
        x = torch.from_numpy(X).cuda()
        torch.cuda.synchronize()
        call("zl_mat_gemv_noalloc", m.h, C.c_void_p(x.data_ptr()), M, C.c_void_p(x.data_ptr()), C.c_void_p(st.cuda_stream))
        st.synchronize()
        assert (x[:M].cpu().numpy().view(np.uint32) == m.gemv(X[:M]).view(np.uint32)).all()
    m.free()


@pytest.mark.parametrize("type_,rows,cols", [(G.Q8_0, 2048, 2048), (G.Q8_0, 4096, 512), (G.Q8_0, 70, 96), (G.Q4_K, 2048, 2048),
                                             (G.Q6_K, 2048, 512)])
def test_single_token_result_over_the_row(gpu, type_, rows, cols):
    """One token whose result overwrites its row, all of it or from its middle on."""
    raw = synth.tensor_bytes(synth.TensorSpec("w", type_, rows, cols, seed=9), use_device=True)
    m = Mat(type_, raw, rows, cols)
    X = np.random.default_rng(9).standard_normal((1, cols)).astype(np.float32)
    want = m.gemv(X)[0]
    st = torch.cuda.Stream()
    for shift in (0, cols // 2):
        print(f"case type {type_} {rows} x {cols} one token, result from value {shift} on", flush=True)
        buf = torch.zeros(shift + max(rows, cols), device="cuda")
        buf[:cols] = torch.from_numpy(X[0]).cuda()
        torch.cuda.synchronize()
        call("zl_mat_gemv_noalloc", m.h, C.c_void_p(buf.data_ptr()), 1, C.c_void_p(buf.data_ptr() + 4 * shift), C.c_void_p(st.cuda_stream))
        st.synchronize()
        assert (buf[shift:shift + rows].cpu().numpy().view(np.uint32) == want.view(np.uint32)).all(), shift
    m.free()
