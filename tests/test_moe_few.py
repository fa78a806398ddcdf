"""Routed experts of a batch on the matrix cores: on the few-token GEMM's tiles (moe_few.hip: groups of every size around the 16- and
32-slot tiles, row tiles with remainders, few and many workgroups, a shared expert) and in moe_mfma.hip (groups of up to eight and up
to sixteen slots).  Against the oracle; outputs outside the plain per-row tolerance must be whole re-quantisation flips
(oracle/flips.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4_K, Q5_K, Q6_K = 12, 13, 14


def _lists(groups, tokens, rng):
    """Slot lists with the given number of slots per expert: each expert's tokens distinct, list in a shuffled order."""
    e, t = [], []
    for expert, n in enumerate(groups):
        e += [expert] * n
        t += list(rng.permutation(tokens)[:n])
    order = rng.permutation(len(e))
    return np.array(e, np.uint32)[order], (rng.random(len(e)) + 0.1).astype(np.float32), np.array(t, np.uint32)[order]


def _check(rnb, oracle, tokens, groups, n_ff, n_embd, shared, down_quant):
    from oracle import flips

    rng = np.random.default_rng(tokens + n_ff)
    n_expert = len(groups)
    print(f"moe few tokens={tokens} experts={n_expert} n_ff={n_ff} n_embd={n_embd} down={down_quant} shared={shared}", flush=True)
    e, r, t = _lists(groups, tokens, rng)
    gate, up = (oracle.make_weights(Q4_K, (n_expert + shared) * n_ff, n_embd, 70 + k) for k in range(2))
    down = oracle.make_weights(down_quant, (n_expert + shared) * n_embd, n_ff, 72)
    x = oracle.fill_normal(tokens * n_embd, 73, 1.0)
    if shared:  # one more slot of every token, its matrices behind the routed ones for the oracle
        e = np.concatenate([e, np.full(tokens, n_expert, np.uint32)])
        r = np.concatenate([r, rng.random(tokens).astype(np.float32)])
        t = np.concatenate([t, np.arange(tokens, dtype=np.uint32)])
    g_len, d_len = gate.size // (n_expert + shared) * n_expert, down.size // (n_expert + shared) * n_expert
    routed = [gate[:g_len].copy(), up[:g_len].copy(), down[:d_len].copy()]
    own = [gate[g_len:].copy(), up[g_len:].copy(), down[d_len:].copy()] if shared else None
    got = rnb.qwen35_sparse_experts_selected_base_by_token(*routed, e, r, t, tokens, down_quant, n_ff, n_embd, x, shared=own)
    ref = oracle.moe_sparse_experts_by_token(gate, up, down, n_expert + shared, e, r, t, tokens, down_quant, n_ff, n_embd, x)
    v = flips.moe_verdict(np.asarray(got).reshape(np.shape(ref)), ref, gate, up, down, n_expert + shared, e, r, t, tokens, down_quant,
                          n_ff, n_embd, x)
    assert v["ok"] or v["flip_aware_ok"], {key: v[key] for key in v if key != "flips"}
    for a in routed + (own or []):
        rnb.release(a)


@pytest.mark.parametrize("down_quant", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("tokens,groups,n_ff,n_embd,shared", [
    (18, [9, 1, 0, 8, 7, 9, 9], 256, 256, False),           # one block, tiles of 16
    (17, [1, 2, 15, 16, 17, 3], 768, 512, False),           # tiles of 16, one group in two of them
    (40, [16, 17, 31, 32, 33, 1, 40], 512, 1024, False),    # tiles of 32: one and two token tiles, and a second unit of one slot
    (70, [70, 65, 64, 2, 33], 1280, 768, True),             # groups of several units, K slices of unequal length
    (48, [48, 20] * 41, 256, 512, False),                   # many experts with short intermediates, a block and an even number
    (16, [5, 4, 3] * 10, 1024, 1280, True),                 # small groups, five blocks in
])
def test_moe_tiles_of_few_tokens(rnb, oracle, tokens, groups, n_ff, n_embd, shared, down_quant):
    _check(rnb, oracle, tokens, groups, n_ff, n_embd, shared, down_quant)


# more than 16 groups of at most eight slots, 1.8 on average and more, groups * blocks in * blocks out below 2000
@pytest.mark.parametrize("tokens,groups,n_ff,n_embd,down_quant", [
    (16, [8, 1, 3, 5, 2] * 4, 256, 256, Q4_K),                # four waves, a row tile a workgroup; one block
    (16, [8, 1, 3, 5, 2] * 4, 256, 256, Q5_K),
    (16, [8, 1, 3, 5, 2] * 4, 256, 256, Q6_K),
    (24, [2, 1, 2, 3, 8] * 20, 768, 1536, Q6_K),              # six waves, two row tiles a workgroup in both kernels
    (16, [2, 2, 1, 4, 7] * 4 + [2, 1], 1536, 2048, Q5_K),     # four waves, two row tiles a workgroup
    (20, [3, 1, 2] * 100, 256, 768, Q4_K),                    # more workgroups than units, no merging
    (18, [1, 2, 3, 2] * 27, 256, 4352, Q6_K),                 # four row tiles a workgroup in the down kernel, two in its last
    (18, [1, 2, 3, 2] * 27, 256, 4352, Q5_K),
])
def test_moe_small_groups(rnb, oracle, tokens, groups, n_ff, n_embd, down_quant):
    _check(rnb, oracle, tokens, groups, n_ff, n_embd, False, down_quant)


# groups of up to sixteen slots whose gate/up workgroups fill one round, 240 to 256 of them with all rows in use
@pytest.mark.parametrize("tokens,groups,n_ff,n_embd,down_quant", [
    (16, [16, 1, 9, 8, 2, 3] * 20, 768, 512, Q4_K),           # six waves, two row tiles a workgroup, the least groups
    (19, [9, 12, 1, 5] * 32, 768, 768, Q5_K),                 # ... the most
    (16, [1, 2, 3, 9] * 31, 768, 256, Q6_K),
    (16, [16, 7, 15, 2] * 31, 256, 1280, Q5_K),               # four waves, a row tile a workgroup
    (24, [16, 3] * 31, 512, 512, Q5_K),                       # ... four row tiles a group
    (17, [10, 1, 3, 2] * 30, 256, 4352, Q5_K),                # four row tiles a workgroup in the down kernel, two in its last
    (17, [17, 1, 9, 8, 2, 3] * 20, 768, 512, Q6_K),           # a slot too many
])
def test_moe_groups_of_up_to_sixteen(rnb, oracle, tokens, groups, n_ff, n_embd, down_quant):
    _check(rnb, oracle, tokens, groups, n_ff, n_embd, False, down_quant)
