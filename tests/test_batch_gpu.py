"""Batched-position kernels: the INT8 batch chains against the oracle bit for
bit (through the dispatch-table entry that runs them, at tile edges,
remainders and every slots-per-wavefront form)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def table():
    import libinferbit_amd as L
    L.ops.init(0)
    P, I = C.c_void_p, C.c_int
    names = ("matmul_int4", "matmul_int8", "matmul_int2", "rmsnorm", "rope", "softmax", "silu_mul", "matmul_w4a8",
             "matmul_w4a8_batch", "matmul_int8_batch")

    class Kernels(C.Structure):
        _fields_ = [(n, P) for n in names]

    k = Kernels()
    L.lib().ib_init_kernels_hip(C.byref(k))
    return {"matmul_int8_batch": C.CFUNCTYPE(None, P, P, P, P, I, I, I, I)(k.matmul_int8_batch)}


# M, N, B, M_stride: one row and column block; partial row and column tiles;
# 1, 2 and 4 slots per wavefront (4: 8192 rows x 32); N % 16 != 0 (one chain per thread)
@pytest.mark.parametrize("M,N,B,ms", [(1, 16, 1, 1), (64, 128, 8, 64), (65, 144, 3, 70), (200, 400, 32, 203),
                                      (1000, 2048, 17, 1000), (4096, 144, 32, 4096), (8192, 272, 31, 8192),
                                      (8192, 128, 32, 8195), (33, 100, 5, 33)])
def test_int8_batch_chains_bit_exact(table, oracle_lib, M, N, B, ms):
    print(f"case int8 chains M={M} N={N} B={B}", flush=True)
    r = np.random.default_rng(M + N + B)
    w = r.integers(-127, 128, (M, N), dtype=np.int8)
    s = (r.random(M) * 0.01 + 1e-4).astype(np.float32)
    x = r.standard_normal((B, N)).astype(np.float32)
    want = oracle_lib.matmul_int8_batch(w, s, x, ms)
    out = np.full((B - 1) * ms + M, 7.0, np.float32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    table["matmul_int8_batch"](p(out), p(w), p(s), p(x), M, N, B, ms)
    want = np.asarray(want).reshape(-1)
    for b in range(B):
        np.testing.assert_array_equal(out[b * ms:b * ms + M].view(np.uint32), want[b * ms:b * ms + M].view(np.uint32))
        assert (out[b * ms + M:(b + 1) * ms] == 7.0).all()
