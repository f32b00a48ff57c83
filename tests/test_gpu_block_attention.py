"""Attention of a block of tokens over a long context (qwn_block_attention.hip)
through the resident decoder's prefill, chain verify and tree verify at
contexts past the one-split decode kernel: row tiles of sixteen (token, head)
pairs that end inside a token, one-row tiles, split contexts and their merge,
every head dim, more query heads per KV head than the one-token kernels take.
The logits are held to the oracle's rounding envelope (parity.py)."""
import numpy as np
import pytest

from parity import oracle_envelope, step_errors, within_envelope
from qwanto_amd import abi, synth

pytestmark = pytest.mark.gpu

SEEDS = tuple(range(1, 9))


def config(heads, kv_heads, head_dim, max_ctx=1500):
    return dict(hidden=256, intermediate=512, layers=2, heads=heads, kv_heads=kv_heads, head_dim=head_dim, vocab=1000,
                max_ctx=max_ctx, rope_theta=1e6, rms_eps=1e-6)


@pytest.mark.parametrize("heads,kv_heads,head_dim,prompt,draft,qk", [
    (6, 1, 128, 1, 2, False),      # one token: a tile of six rows
    (6, 2, 128, 67, 11, False),    # three rows a token: tiles end inside a token
    (4, 4, 64, 130, 16, True),     # one head per KV head: sixteen tokens a tile
    (2, 1, 256, 40, 5, False),     # head_dim 256: keys and values loaded at their use
    (12, 1, 64, 35, 7, False),     # more than eight heads per KV head
    (4, 2, 64, 700, 3, False),     # 703 tokens in two splits and a merge
    (1, 1, 128, 1300, 4, True),
])
def test_prefill_and_verify_match_oracle(gpu_ctx, oracle_lib, heads, kv_heads, head_dim, prompt, draft, qk):
    rng = np.random.default_rng(heads * 1000 + head_dim + prompt)
    cfg = config(heads, kv_heads, head_dim)
    model = synth.decoder_model(rng, cfg, "q4_0", qk_norm=qk)
    ids = synth.prompt_tokens(rng, cfg["vocab"], prompt + draft)
    dec = abi.ResidentDecoder(gpu_ctx, model)
    ref = oracle_lib.decoder(model)
    try:
        refs = [ref.forward(int(t)) for t in ids]
        last, _ = dec.prefill(ids[:prompt])
        rows, _ = dec.verify(ids[prompt:])
    finally:
        dec.close()
        ref.close()
    env = oracle_envelope(oracle_lib, model, ids, refs, SEEDS)[:, prompt - 1:]
    ok, msg = within_envelope(step_errors([last, *rows], refs[prompt - 1:]), env)
    assert ok, msg


@pytest.mark.parametrize("heads,kv_heads,head_dim", [(6, 2, 128), (2, 1, 256)])
def test_tree_matches_oracle_paths(gpu_ctx, oracle_lib, heads, kv_heads, head_dim):
    """A tree whose siblings must not see each other, 20 nodes over a 90-token prefix."""
    rng = np.random.default_rng(heads + head_dim)
    cfg = config(heads, kv_heads, head_dim)
    model = synth.decoder_model(rng, cfg, "q4_0")
    prompt = synth.prompt_tokens(rng, cfg["vocab"], 90)
    tokens = synth.prompt_tokens(rng, cfg["vocab"], 20)
    parents = np.array([-1, -1] + [int(rng.integers(0, i)) for i in range(2, 20)], dtype=np.int32)
    dec = abi.ResidentDecoder(gpu_ctx, model)
    try:
        dec.prefill(prompt)
        rows, _ = dec.verify_tree(tokens, parents)
    finally:
        dec.close()
    for i in (0, 1, 7, 19):
        path, n = [], i
        while n >= 0:
            path.append(n)
            n = int(parents[n])
        ids = [int(t) for t in prompt] + [int(tokens[n]) for n in reversed(path)]
        ref = oracle_lib.decoder(model)
        refs = [ref.forward(t) for t in ids]
        ref.close()
        env = oracle_envelope(oracle_lib, model, ids, refs, SEEDS)[:, -1:]
        ok, msg = within_envelope(step_errors([rows[i]], refs[-1:]), env)
        assert ok, f"node {i}: {msg}"


def run_prefill(gpu_ctx, model, ids, max_ctx):
    """A long block's logits: its attention in one split (max_ctx 512), or in two and a merge (1500)."""
    dec = abi.ResidentDecoder(gpu_ctx, dict(model, cfg=dict(model["cfg"], max_ctx=max_ctx)))
    try:
        return dec.prefill(ids)[0]
    finally:
        dec.close()


@pytest.mark.parametrize("head_dim", [64, 128, 256])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_non_finite_queries_show_in_every_split_plan(gpu_ctx, head_dim, bad):
    """A head whose query is not finite gives NaN, and the other heads their
    values, whether its context is read in one split or merged from two: the
    same logits (a merge that drops the NaN leaves a plain zero there)."""
    rng = np.random.default_rng(head_dim)
    cfg = dict(config(2, 1, head_dim), layers=1)
    model = synth.decoder_model(rng, cfg, "q4_0", biases="q")
    model["layers"][0]["q_bias"][:head_dim] = bad
    ids = synth.prompt_tokens(rng, cfg["vocab"], 70)
    one, two = (run_prefill(gpu_ctx, model, ids, n) for n in (512, 1500))
    model["layers"][0]["q_bias"][:head_dim] = 0.0
    assert np.linalg.norm(one - run_prefill(gpu_ctx, model, ids, 512)) > 0.1 * np.linalg.norm(one)   # it shows
    # one int8 step of the other heads' outputs between the two plans' sums
    assert np.linalg.norm(one - two) <= 1e-2 * np.linalg.norm(one)


@pytest.mark.parametrize("max_ctx", [512, 1500])
@pytest.mark.parametrize("head_dim", [64, 128, 256])
def test_tiny_queries_choose(gpu_ctx, oracle_lib, head_dim, max_ctx):
    """Queries of 2^-103 against keys of 2^105: scores that choose among the tokens."""
    rng = np.random.default_rng(head_dim + 1)
    cfg = dict(config(2, 1, head_dim), layers=1, max_ctx=max_ctx)
    model = synth.decoder_model(rng, cfg, "q4_0", biases="qk")
    layer = model["layers"][0]
    for p, scale in (("q", 2.0 ** -103), ("k", 2.0 ** 105)):
        layer[p].reshape(-1, 18)[:, :2] = 0   # the projection is its bias
        layer[p + "_bias"] *= np.float32(scale)
    ids = synth.prompt_tokens(rng, cfg["vocab"], 70)
    ref = oracle_lib.decoder(model)
    refs = [ref.forward(int(t)) for t in ids]
    ref.close()
    env = oracle_envelope(oracle_lib, model, ids, refs, SEEDS)[:, -1:]
    ok, msg = within_envelope(step_errors([run_prefill(gpu_ctx, model, ids, max_ctx)], refs[-1:]), env)
    assert ok, msg


@pytest.mark.parametrize("max_ctx", [512, 1500])
@pytest.mark.parametrize("head_dim", [64, 128, 256])
def test_tiny_values_come_through(gpu_ctx, oracle_lib, head_dim, max_ctx):
    """Values of 2^-95 and an all-zero embedding row, so the attention is all there is of the logits."""
    rng = np.random.default_rng(head_dim + 2)
    cfg = dict(config(2, 1, head_dim), layers=1, max_ctx=max_ctx)
    model = synth.decoder_model(rng, cfg, "q4_0", biases="qkv")
    model["layers"][0]["v_bias"] *= np.float32(2.0 ** -95)
    model["embed"][0] = 0
    ids = np.zeros(70, dtype=np.int32)
    ref = oracle_lib.decoder(model)
    want = [ref.forward(0) for _ in ids][-1].astype(np.float64)
    ref.close()
    got = run_prefill(gpu_ctx, model, ids, max_ctx)
    # one step of the int8 input of o at the most: 1/127 of the largest value
    assert np.linalg.norm(want) > 0 and np.linalg.norm(got - want) <= 1e-2 * np.linalg.norm(want)
