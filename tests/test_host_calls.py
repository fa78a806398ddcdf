"""Calls on host arrays: up to 1 MB a way the kernels read and write the pinned buffers themselves or a copying kernel does (results of
waves with one row each, from 32 KB on), above it copy commands carry the floats.  The result is the one of the same call on device buffers, to the bit, on both sides of the limit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q8_0, Q4_K, Q6_K, IQ2_XXS = 8, 12, 14, 16
BATCH = {Q8_0: "q8_0_gemv_batch", Q4_K: "q4k_gemv_batch", Q6_K: "q6k_gemv_batch", IQ2_XXS: "iq2_xxs_gemv_batch"}


@pytest.mark.parametrize("quant,rows,cols,seq", [
    (Q8_0, 3, 32, 1), (Q8_0, 5, 96, 3), (Q4_K, 1, 256, 1), (Q4_K, 7, 4352, 1),   # tails of the copying kernel; one and two launches
    (Q8_0, 2047, 160, 128), (Q8_0, 2048, 160, 128), (Q8_0, 2049, 160, 128),      # results of just under, of and just over 1 MB
    (Q4_K, 33, 4096, 64), (Q4_K, 33, 4096, 65),                                  # tokens of 1 MB and over
    (Q6_K, 262145, 256, 1), (Q4_K, 5, 262144 + 256, 1),                          # one token: rows and blocks past the limit
    (Q8_0, 4096, 96, 2), (Q8_0, 4097, 96, 2), (IQ2_XXS, 8191, 256, 1), (IQ2_XXS, 8193, 256, 1),  # results of a GEMV, 32 KB and over
    (Q6_K, 4097, 2304, 2), (Q6_K, 4097, 2048, 2), (IQ2_XXS, 2049, 256, 5)])      # ... of longer and short rows, of a GEMM
def test_host_arrays_equal_device_buffers(rnb, oracle, quant, rows, cols, seq):
    print(f"host call quant={quant} rows={rows} cols={cols} seq={seq}", flush=True)
    w = oracle.make_weights(quant, rows, cols, 3)
    x = oracle.fill_normal(seq * cols, 4, 1.0)
    got = np.asarray(getattr(rnb, BATCH[quant])(w, rows, cols, x)).reshape(-1)
    rnb.release(w)
    dw, dx, do = rnb.DeviceBuffer.from_host(w), rnb.DeviceBuffer.from_host(x), rnb.DeviceBuffer(4 * rows * seq)
    rnb.gemv_dev(quant, dw, rows, cols, dx, seq, do)
    want = do.to_host(np.float32)
    for b in (dw, dx, do):
        b.free()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("rows,cols", [(1, 256), (257, 512), (70001, 256), (9, 16640), (3, 262144 + 256)])
def test_argmax_of_host_tokens(rnb, oracle, rows, cols):
    """The winner and its value of the same call's rows, written by the reducing kernel."""
    print(f"arg-max rows={rows} cols={cols}", flush=True)
    w = oracle.make_weights(Q6_K, rows, cols, 5)
    x = oracle.fill_normal(cols, 6, 1.0)
    full = np.asarray(rnb.q6k_gemv(w, rows, cols, x)).reshape(-1)
    idx, val = rnb.q6k_gemv_argmax(w, rows, cols, x)
    rnb.release(w)
    assert idx == int(np.argmax(full)) and val == full[idx]
