"""Prompts of more than one narrow block: the projections on the wide GEMM
(qwn_wide_gemm.hip), through the resident decoder, against the oracle.  Token
counts that end inside a 16-token group and a token tile, rows that end
inside a row tile and a 16-row group, K that ends inside a unit, the K split
of the residual adds, gate/up pairs, biases, a prompt of more than one wide
block.  The logits of the last token are held to the oracle's rounding
envelope (parity.py)."""
import numpy as np
import pytest

from parity import oracle_envelope, step_errors, within_envelope
from qwanto_amd import abi, synth
from test_gpu_gemv import check_hvsq2, check_q4_0

pytestmark = pytest.mark.gpu

SEEDS = tuple(range(1, 9))


def config(hidden, inter, heads, kv_heads, head_dim, max_ctx):
    return dict(hidden=hidden, intermediate=inter, layers=1, heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                vocab=500, max_ctx=max_ctx, rope_theta=1e6, rms_eps=1e-6)


@pytest.mark.parametrize("dtype", ["q4_0", "hvsq2"])
@pytest.mark.parametrize("shape,prompt,bias", [
    ((256, 512, 2, 1, 128, 512), 65, False),       # one token past the narrow block
    ((288, 1056, 3, 1, 64, 512), 129, True),  # rows and K ending inside every tile and unit
    ((544, 2336, 2, 2, 128, 1200), 300, False),
    ((256, 9728, 2, 1, 64, 1200), 520, False),     # 8-group token tiles of the gate/up pair, the K split of down
    ((256, 256, 1, 1, 64, 1200), 1100, True),      # a wide block and a second, narrow one's remainder
])
def test_wide_prefill_matches_oracle(gpu_ctx, oracle_lib, dtype, shape, prompt, bias):
    rng = np.random.default_rng(shape[1] + prompt)
    cfg = config(*shape)
    model = synth.decoder_model(rng, cfg, dtype, biases="qkvo" if bias else "")
    ids = synth.prompt_tokens(rng, cfg["vocab"], prompt)
    dec = abi.ResidentDecoder(gpu_ctx, model)
    ref = oracle_lib.decoder(model)
    try:
        refs = [ref.forward(int(t)) for t in ids]
        last, _ = dec.prefill(ids)
        dec.reset()
        again, _ = dec.prefill(ids)   # the same with the workspaces of an earlier prompt
    finally:
        dec.close()
        ref.close()
    env = oracle_envelope(oracle_lib, model, ids, refs, SEEDS)[:, prompt - 1:]
    for got in (last, again):
        ok, msg = within_envelope(step_errors([got], refs[prompt - 1:]), env)
        assert ok, msg


@pytest.mark.parametrize("dtype", ["q4_0", "hvsq2"])
@pytest.mark.parametrize("N,K,M", [
    (1, 31, 65),         # one row, K inside one unit, a one-token last group
    (77, 777, 70),       # rows and K ending inside their tiles; four sets of waves splitting K
    (130, 129, 40),      # 17 to 64 tokens: several groups on the 16-token GEMM
    (2560, 1536, 160),   # two sets
    (9000, 520, 129),    # one set
    (17000, 256, 300),   # two row groups a wave, fewer units than sets
])
def test_host_batches(gpu_ctx, oracle_lib, dtype, N, K, M):
    """qwn_cuda_abi_hypervsq2_gemm with more than 16 tokens."""
    check = check_q4_0 if dtype == "q4_0" else check_hvsq2
    check(gpu_ctx, oracle_lib, N, K, seed=N + K + M, M=M)
