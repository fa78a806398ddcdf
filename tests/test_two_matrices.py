"""Gate and up projections of a batch in one grid (gemm_matrix, run_gate_up_dev): every kernel that takes two matrices, with and
without K slices, which are added by the gated quantiser (K-quant down projection) or by a launch of their own (32-element one).
The down projection has one weight of 1 per row, so that an output is one intermediate value in its 8-bit code: against the
activation of two plain calls to within a step of that code, which a last-bit difference of the sums can move."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q8_0, Q4_K = 8, 12


def _selector(quant, n_embd, n_ff, col):
    """[n_embd][n_ff] blocks that are 1 at column col[row] of every row and 0 elsewhere."""
    row, one = np.arange(n_embd), np.array([1.0], np.float16).view(np.uint8)
    if quant == Q8_0:
        blocks = np.zeros((n_embd, n_ff // 32, 34), np.uint8)
        blocks[row, col // 32, :2] = one
        blocks[row, col // 32, 2 + col % 32] = 1
    else:  # d = 1, dmin = 0, the eight scales 1
        blocks = np.zeros((n_embd, n_ff // 256, 144), np.uint8)
        blocks[:, :, :2] = one
        blocks[:, :, 4:8] = 1
        blocks[:, :, 12:16] = 1
        e = col % 256
        blocks[row, col // 256, 16 + e // 64 * 32 + e % 32] = np.where(e % 64 < 32, 1, 16)
    return blocks.reshape(-1)


@pytest.mark.parametrize("down_quant", [Q8_0, Q4_K])
@pytest.mark.parametrize("n_ff,n_embd,seq,gelu", [
    (768, 2560, 48, False),     # 128 x 32 tiles, five slices
    (512, 1280, 33, True),      # ... two blocks and one in the last slice
    (4096, 2048, 65, False),    # 256 x 64 tiles, two slices, a token in the second tile
    (4352, 3072, 130, True),    # ... seventeen row tiles a matrix
    (2304, 4096, 513, False),   # ... whole rows
    (512, 8704, 2050, False),   # two-digit operands: four tiles a workgroup, three slices, the last group of one ragged tile
    (1024, 5888, 1500, True),   # ... three tiles, two slices of 12 and 11 blocks
    (1792, 2560, 2050, False),  # ... four tiles, whole rows
    (4352, 1024, 2050, False),  # ... three tiles, whole rows, several rounds
])
def test_gate_and_up_of_a_batch(rnb, oracle, n_ff, n_embd, seq, gelu, down_quant):
    print(f"gate and up n_ff={n_ff} n_embd={n_embd} seq={seq} down={down_quant}", flush=True)
    gate, up = (oracle.make_weights(Q4_K, n_ff, n_embd, 50 + k) for k in range(2))
    x = oracle.fill_normal(seq * n_embd, 52, 1.0)
    col = np.arange(n_embd) * 11 % n_ff
    down = _selector(down_quant, n_embd, n_ff, col)
    call = rnb.dense_q4k_gelu_ffn_batch if gelu else rnb.dense_q4k_silu_ffn_batch
    got = np.asarray(call(gate, up, down, down_quant, n_ff, n_embd, seq, x), np.float64).reshape(seq, n_embd)
    g, u = (np.asarray(rnb.q4k_gemv_batch(m, n_ff, n_embd, x), np.float64).reshape(seq, n_ff) for m in (gate, up))
    for a in (gate, up, down):
        rnb.release(a)
    if gelu:
        mid = 0.5 * g * (1 + np.tanh(np.sqrt(2 / np.pi) * (g + 0.044715 * g ** 3))) * u
    else:
        mid = g / (1 + np.exp(-g)) * u
    block = 32 if down_quant == Q8_0 else 256
    step = np.abs(mid.reshape(seq, -1, block)).max(axis=2) / 127
    assert np.all(np.abs(got - mid[:, col]) <= 1.01 * step[:, col // block])
