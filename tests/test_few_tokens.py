"""The GEMM of a few tokens (gemm_few.hip): Q4_K, Q5_K and Q6_K batches of three or four to 32 tokens whose K slices are the waves of one
workgroup.  Against the oracle's f64 statement of the same integer dots: the sums over a super-block are exact, what is left is
the f32 sum over at most 64 blocks, |gpu - gold| <= 2e-5 * rms(gold) as in the other kernels' tests."""
import numpy as np
import pytest

from tests.test_gpu_parity import check_ffn

pytestmark = pytest.mark.gpu

Q4_K, Q5_K, Q6_K = 12, 13, 14
BLOCK = {Q4_K: 144, Q5_K: 176, Q6_K: 210}
BATCH = {Q4_K: "q4k_gemv_batch", Q5_K: "q5k_gemv_batch", Q6_K: "q6k_gemv_batch"}


def _check(oracle, quant, w, rows, cols, seq, x, got):
    pick = np.unique(np.clip([0, 1, 15, 16, 17, 31, 32, 33, rows // 2, rows - 33, rows - 17, rows - 16, rows - 1], 0, rows - 1))
    ws = np.ascontiguousarray(w.reshape(rows, -1)[pick]).reshape(-1)
    gold = np.asarray(oracle.gemv(quant, ws, len(pick), cols, x, gold=True), np.float64).reshape(seq, len(pick))
    rms = float(np.sqrt(np.mean(gold * gold))) or 1.0
    worst = float(np.abs(got.reshape(seq, rows)[:, pick] - gold).max())
    assert worst <= 2e-5 * rms, (quant, rows, cols, seq, worst / rms)


# rows around the 16-row tile and the workgroup's rows, blocks around the eight and four slices, tokens around the two tiles (up to 512
# rows with up to sixteen tokens are the GEMV's)
SHAPES = [(529, 1, 9), (527, 2, 16), (545, 8, 12), (576, 9, 10), (513, 56, 13), (1026, 34, 3),
          (1, 1, 9), (15, 2, 16), (16, 3, 17), (17, 5, 31), (31, 7, 32), (33, 8, 12), (64, 9, 10), (250, 17, 24), (77, 56, 13),
          (48, 64, 32), (2048, 33, 3), (4096, 16, 5),
          (4097, 8, 11), (4113, 3, 20), (7000, 9, 19),      # four slices; fewer blocks than slices
          (20481, 2, 15), (20490, 5, 27),                   # two slices; a second token tile
          (12305, 1, 18), (12300, 6, 32),                   # two row tiles a wave (Q4_K, Q5_K)
          (27000, 15, 9), (25601, 16, 30)]                  # ... by size, four and two slices


@pytest.mark.parametrize("quant", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("rows,nb,seq", SHAPES)
def test_few_tokens_equal_the_gold_dots(rnb, oracle, quant, rows, nb, seq):
    cols = 256 * nb
    print(f"few tokens quant={quant} rows={rows} blocks={nb} seq={seq}", flush=True)
    w = oracle.make_weights(quant, rows, cols, 31 + rows)
    x = oracle.fill_normal(seq * cols, 32 + seq, 1.0)
    got = np.asarray(getattr(rnb, BATCH[quant])(w, rows, cols, x), np.float64)
    rnb.release(w)
    _check(oracle, quant, w, rows, cols, seq, x, got)


# (largest batch whose rows equal the one-token call's, shapes): under 4 MB, rows of up to 16 blocks, of more, matrices of 48 MB
@pytest.mark.parametrize("quant,most,rows,nb", [
    (Q4_K, 8, 1792, 16), (Q5_K, 8, 1472, 16), (Q6_K, 8, 1232, 16), (Q4_K, 8, 1500, 17),
    (Q4_K, 3, 1824, 16), (Q4_K, 3, 29200, 1), (Q5_K, 3, 1490, 16), (Q6_K, 4, 1252, 16), (Q6_K, 4, 20000, 1),
    (Q4_K, 2, 1720, 17), (Q5_K, 2, 1410, 17), (Q6_K, 3, 1182, 17),
    (Q4_K, 3, 24576, 16), (Q6_K, 4, 16384, 15)])
def test_rows_that_equal_the_one_token_call(rnb, oracle, quant, most, rows, nb):
    cols = 256 * nb
    print(f"equal rows quant={quant} rows={rows} blocks={nb} tokens 2 .. {most}", flush=True)
    w = oracle.make_weights(quant, rows, cols, 71)
    x = oracle.fill_normal(most * cols, 72, 1.0)
    one, many = (getattr(rnb, BATCH[quant].replace("_batch", end)) for end in ("", "_batch"))
    alone = np.stack([np.asarray(one(w, rows, cols, x[t * cols:(t + 1) * cols])).reshape(rows) for t in range(most)])
    for seq in range(2, most + 1):
        got = np.asarray(many(w, rows, cols, x[:seq * cols])).reshape(seq, rows)
        assert np.array_equal(got.view(np.uint32), alone[:seq].view(np.uint32)), seq
    rnb.release(w)


@pytest.mark.parametrize("quant", [Q4_K, Q5_K, Q6_K])
def test_few_tokens_blocks_of_any_codes(rnb, oracle, quant):
    """Codes, scales and mins of any value, activations at both ends of their range."""
    rows, nb, seq = 160, 11, 21
    rng = np.random.default_rng(5)
    blocks = rng.integers(0, 256, (rows * nb, BLOCK[quant]), dtype=np.uint8)
    half = lambda sd: (rng.standard_normal((rows * nb, 1)) * sd).astype(np.float16).view(np.uint8)  # noqa: E731
    if quant == Q6_K:
        blocks[:, 208:210] = half(0.01)
    else:
        blocks[:, 0:2], blocks[:, 2:4] = half(0.01), half(0.01)
    blocks[:nb, 16 if quant != Q6_K else 0:128] = 0xFF
    w = blocks.reshape(-1)
    x = rng.choice(np.array([-1.0, 1.0, 0.5, 0.01], np.float32), seq * nb * 256)
    got = np.asarray(getattr(rnb, BATCH[quant])(w, rows, 256 * nb, x), np.float64)
    rnb.release(w)
    _check(oracle, quant, w, rows, 256 * nb, seq, x, got)


@pytest.mark.parametrize("quant", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("shift", [0, 1, 2, 4, 6])
def test_few_tokens_of_a_part_of_a_resident_tensor(rnb, oracle, quant, shift):
    """At addresses that are no multiple of four the other kernels answer, and so they do for a Q6_K matrix of an odd number of
    blocks, whose last piece would end behind the tensor."""
    rows, nb, seq = 515, 5, 14
    w = oracle.make_weights(quant, rows, 256 * nb, 8)
    x = oracle.fill_normal(seq * 256 * nb, 9, 1.0)
    parent = np.zeros(w.size + shift, np.uint8)
    parent[shift:] = w
    rnb.prewarm([parent])
    got = np.asarray(getattr(rnb, BATCH[quant])(parent[shift:], rows, 256 * nb, x), np.float64)
    rnb.release(parent)
    _check(oracle, quant, w, rows, 256 * nb, seq, x, got)


@pytest.mark.parametrize("quant,seq", [(Q4_K, 13), (Q6_K, 30)])
def test_few_tokens_finite_from_any_neighbours(rnb, oracle, quant, seq):
    """A token's result does not depend on the others in its tile, NaN and infinities among them included."""
    rows, nb = 600, 6
    w = oracle.make_weights(quant, rows, 256 * nb, 18)
    x = oracle.fill_normal(seq * 256 * nb, 19, 1.0).reshape(seq, -1)
    bad = x.copy()
    bad[1, 7], bad[4, 300], bad[seq - 1, 0] = np.nan, np.inf, -np.inf
    call = getattr(rnb, BATCH[quant])
    a = np.asarray(call(w, rows, 256 * nb, x.reshape(-1))).reshape(seq, rows)
    b = np.asarray(call(w, rows, 256 * nb, bad.reshape(-1))).reshape(seq, rows)
    rnb.release(w)
    keep = [t for t in range(seq) if t not in (1, 4, seq - 1)]
    assert np.array_equal(a[keep].view(np.uint32), b[keep].view(np.uint32))


@pytest.mark.parametrize("seq", [9, 16, 17, 32])
@pytest.mark.parametrize("n_ff,n_embd,gelu", [(4352, 1024, False), (768, 2304, True), (512, 4608, False)])
def test_few_tokens_gate_and_up(rnb, oracle, seq, n_ff, n_embd, gelu):
    """Gate and up in one launch (16 rows a wave, four and eight slices)."""
    gate, up, down = (oracle.make_weights(q, r, c, 40 + k) for k, (q, r, c) in
                      enumerate([(Q4_K, n_ff, n_embd), (Q4_K, n_ff, n_embd), (Q6_K, n_embd, n_ff)]))
    x = oracle.fill_normal(seq * n_embd, 43, 1.0)
    call = rnb.dense_q4k_gelu_ffn_batch if gelu else rnb.dense_q4k_silu_ffn_batch
    got = call(gate, up, down, Q6_K, n_ff, n_embd, seq, x)
    check_ffn(oracle, got, gate, up, down, Q6_K, n_ff, n_embd, x, gelu, f"few tokens ffn {seq} {n_ff} {n_embd}")
    for a in (gate, up, down):
        rnb.release(a)


@pytest.mark.parametrize("seq", [4, 32])
def test_few_tokens_gate_and_up_of_large_matrices(rnb, oracle, seq):
    """Two row tiles a wave: rows of the two matrices against the plain calls, through a Q8_0 down projection with one
    non-zero weight per row, so that an output is one intermediate value in its 8-bit code (half a step of 1/127 of its
    block's largest, a hundredth of that for the rounding of the code's own arithmetic)."""
    n_ff, n_embd = 25600, 4096
    gate, up = (oracle.make_weights(Q4_K, n_ff, n_embd, 50 + k) for k in range(2))
    x = oracle.fill_normal(seq * n_embd, 52, 1.0)
    col = np.arange(n_embd) * 6 + np.arange(n_embd) % 7
    down = np.zeros((n_embd, n_ff // 32, 34), np.uint8)
    down[np.arange(n_embd), col // 32, :2] = np.array([1.0], np.float16).view(np.uint8)
    down[np.arange(n_embd), col // 32, 2 + col % 32] = 1
    got = np.asarray(rnb.dense_q4k_silu_ffn_batch(gate, up, down.reshape(-1), 8, n_ff, n_embd, seq, x), np.float64)
    g, u = (np.asarray(rnb.q4k_gemv_batch(m, n_ff, n_embd, x), np.float64).reshape(seq, n_ff) for m in (gate, up))
    for a in (gate, up, down.reshape(-1)):
        rnb.release(a)
    mid = g / (1 + np.exp(-g)) * u
    step = np.abs(mid.reshape(seq, -1, 32)).max(axis=2) / 127
    assert np.all(np.abs(got.reshape(seq, n_embd) - mid[:, col]) <= 0.51 * step[:, col // 32])
