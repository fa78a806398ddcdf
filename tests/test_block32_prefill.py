"""The prefill GEMM of the 32-element formats (gemm_b32.hip).  Integer sums of a block are exact, what is left is the f32 sum over
the row's blocks: |gpu - gold| <= 2e-5 * rms(gold) against the oracle's f64 statement, as in the other kernels' tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, Q8_1 = 2, 3, 6, 7, 8, 9
BYTES = {Q4_0: 18, Q4_1: 20, Q5_0: 22, Q5_1: 24, Q8_0: 34, Q8_1: 36}
BATCH = {Q4_0: "q4_0_gemv_batch", Q4_1: "q4_1_gemv_batch", Q5_0: "q5_0_gemv_batch", Q5_1: "q5_1_gemv_batch",
         Q8_0: "q8_0_gemv_batch", Q8_1: "q8_1_gemv_batch"}


def _check(oracle, quant, w, rows, cols, seq, x, got):
    pick = np.unique(np.clip([0, 1, 31, 32, 33, 255, 256, 257, rows // 2, rows - 33, rows - 32, rows - 1], 0, rows - 1))
    ws = np.ascontiguousarray(w.reshape(rows, -1)[pick]).reshape(-1)
    gold = np.asarray(oracle.gemv(quant, ws, len(pick), cols, x, gold=True), np.float64).reshape(seq, len(pick))
    rms = float(np.sqrt(np.mean(gold * gold))) or 1.0
    worst = float(np.abs(got.reshape(seq, rows)[:, pick] - gold).max())
    assert worst <= 2e-5 * rms, (quant, rows, cols, seq, worst / rms)


# rows around the wave's 32 and the workgroup's 256, steps from one to many (with and without slices), tokens around the tile
# and the groups of two, three and four tiles
@pytest.mark.parametrize("quant", [Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, Q8_1])
@pytest.mark.parametrize("rows,steps,seq", [(1, 1, 33), (31, 2, 64), (33, 3, 65), (255, 1, 129), (257, 17, 96), (288, 5, 97), (1000, 11, 40),
                                            (800, 6, 700), (2080, 5, 200), (4097, 2, 513), (1025, 33, 34), (1, 3, 33), (4097, 3, 129)])
def test_prefill_of_32_element_blocks(rnb, oracle, quant, rows, steps, seq):
    cols = 256 * steps
    print(f"32-element prefill quant={quant} rows={rows} cols={cols} seq={seq}", flush=True)
    w = oracle.make_weights(quant, rows, cols, 61 + rows)
    x = oracle.fill_normal(seq * cols, 62 + seq, 1.0)
    got = np.asarray(getattr(rnb, BATCH[quant])(w, rows, cols, x), np.float64)
    rnb.release(w)
    _check(oracle, quant, w, rows, cols, seq, x, got)


@pytest.mark.parametrize("quant", [Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, Q8_1])
def test_prefill_of_blocks_of_any_codes(rnb, oracle, quant):
    """Codes of any value (Q8: -128 included), scales and mins of both signs, activations at both ends of their range."""
    rows, steps, seq = 900, 5, 75
    rng = np.random.default_rng(6)
    blocks = rng.integers(0, 256, (rows * steps * 8, BYTES[quant]), dtype=np.uint8)
    half = lambda: (rng.standard_normal((len(blocks), 1)) * 0.01).astype(np.float16).view(np.uint8)  # noqa: E731
    blocks[:, 0:2] = half()
    if quant in (Q4_1, Q5_1, Q8_1):
        blocks[:, 2:4] = half()
    blocks[:40, 4 if quant in (Q4_1, Q5_1, Q8_1) else 2:] = 0x80 if quant in (Q8_0, Q8_1) else 0xFF
    w = blocks.reshape(-1)
    x = rng.choice(np.array([-1.0, 1.0, 0.5, 0.01, 0.0], np.float32), seq * steps * 256)
    got = np.asarray(getattr(rnb, BATCH[quant])(w, rows, 256 * steps, x), np.float64)
    rnb.release(w)
    _check(oracle, quant, w, rows, 256 * steps, seq, x, got)


@pytest.mark.parametrize("quant", [Q5_1, Q8_0])
@pytest.mark.parametrize("shift", [1, 2, 4, 6])
def test_prefill_of_a_part_of_a_resident_tensor(rnb, oracle, quant, shift):
    rows, steps, seq = 300, 3, 50
    w = oracle.make_weights(quant, rows, 256 * steps, 8)
    x = oracle.fill_normal(seq * 256 * steps, 9, 1.0)
    parent = np.zeros(w.size + 8, np.uint8)
    parent[shift:shift + w.size] = w
    rnb.prewarm([parent])
    got = np.asarray(getattr(rnb, BATCH[quant])(parent[shift:shift + w.size], rows, 256 * steps, x), np.float64)
    rnb.release(parent)
    _check(oracle, quant, w, rows, 256 * steps, seq, x, got)


@pytest.mark.parametrize("quant", [Q4_1, Q8_0])
def test_a_token_does_not_see_its_neighbours(rnb, oracle, quant):
    """NaN and infinities in other tokens of the tile included."""
    rows, steps, seq = 900, 5, 70
    w = oracle.make_weights(quant, rows, 256 * steps, 18)
    x = oracle.fill_normal(seq * 256 * steps, 19, 1.0).reshape(seq, -1)
    bad = x.copy()
    bad[1, 7], bad[40, 300], bad[seq - 1, 0] = np.nan, np.inf, -np.inf
    call = getattr(rnb, BATCH[quant])
    a = np.asarray(call(w, rows, 256 * steps, x.reshape(-1))).reshape(seq, rows)
    b = np.asarray(call(w, rows, 256 * steps, bad.reshape(-1))).reshape(seq, rows)
    rnb.release(w)
    keep = [t for t in range(seq) if t not in (1, 40, seq - 1)]
    assert np.array_equal(a[keep].view(np.uint32), b[keep].view(np.uint32))


@pytest.mark.parametrize("quant", [Q4_1, Q5_1])
@pytest.mark.parametrize("mean", [0.0, 0.5, 1.0])
@pytest.mark.parametrize("weights", ["quantised", "skewed"])
def test_minimum_formats_on_tokens_of_any_mean(rnb, oracle, quant, mean, weights):
    """d * code and m are of one size and opposite sign where a block's weights are centred, as are their products with tokens that are
    not: an order of the sums that adds many blocks' codes before their mins carries the difference of two large numbers.  In an
    order that does not, every addition rounds by at most 2^-24 of the running sum, whose rms grows with the root of the blocks added:
    rms error <= 2^-24 * sqrt(blocks / 2) of the rms result.  Skewed: m = 0 and most codes 0, where a fixed offset of the codes would be
    the large number."""
    rows, cols, seq = 96, 8192, 65
    if weights == "quantised":
        w = oracle.make_weights(quant, rows, cols, 27)
    else:
        rng = np.random.default_rng(28)
        blocks = np.zeros((rows * cols // 32, BYTES[quant]), np.uint8)
        blocks[:, 0:2] = (np.abs(rng.standard_normal((len(blocks), 1))) * 0.01).astype(np.float16).view(np.uint8)
        blocks[:, BYTES[quant] - 16:] = np.where(rng.random((len(blocks), 16)) < 0.1, rng.integers(0, 256, (len(blocks), 16)), 0)
        w = blocks.reshape(-1)
    x = oracle.fill_normal(seq * cols, 29, 1.0) + np.float32(mean)
    got = np.asarray(getattr(rnb, BATCH[quant])(w, rows, cols, x), np.float64).reshape(seq, rows)
    rnb.release(w)
    gold = np.asarray(oracle.gemv(quant, w, rows, cols, x, gold=True), np.float64).reshape(seq, rows)
    error = np.sqrt(np.mean((got - gold) ** 2) / np.mean(gold * gold))
    assert error <= 2.0 ** -24 * np.sqrt(cols / 32 / 2), error
