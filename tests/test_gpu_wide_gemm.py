"""More than one narrow block of tokens on the wide GEMM (qwn_wide_gemm.hip):
prompts through the resident decoder and host batches, against the oracle.
Token counts that end inside a 16-token group and a token tile, rows that end
inside a row tile and a 16-row group, K that ends inside a unit, every tile
and K split of the plan, gate/up pairs, biases, prompts of more than one wide
block.  A prompt's logits are held to the oracle's rounding envelope
(parity.py).  Then the host batch around it: results in pieces, long batches,
telemetry."""
import numpy as np
import pytest

from parity import gemv_close, oracle_envelope, step_errors, within_envelope
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
    ((256, 9728, 2, 1, 64, 1200), 520, False),     # the K split of down, four ways
    ((256, 256, 1, 1, 64, 1200), 1100, True),      # a wide block and a second one of 76 tokens
    ((256, 256, 1, 1, 64, 1200), 1025, False),     # from a wide block, launched as it is, to a captured one of one token
    ((256, 256, 2, 1, 64, 1200), 1050, True),      # ... and of 26
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
    # by wide_plan on 256 CUs: 16-row groups a wave x sets of waves splitting K, tokens of a tile
    (77, 777, 70),       # rows and K ending inside their tiles; 1 x 2, 64
    (130, 129, 40),      # 17 to 64 tokens: several groups on the 16-token GEMM
    (2560, 1536, 160),   # Q4_0 1 x 4, 32; HyperVSQ-2 1 x 2, 64
    (9000, 520, 129),    # Q4_0 1 x 2, HyperVSQ-2 1 x 1, 64
    (17000, 256, 300),   # 1 x 1, 64: more workgroups than CUs, one or two units
    (100, 2000, 81),     # 1 x 4, 16, the last tile of one token
    (2240, 2000, 161),   # 1 x 4, 32, the last tile of one token
    (2500, 2000, 257),   # 1 x 4, 64, the last tile of one token, sets of unequal length
    (9700, 600, 833),    # 2 x 1, 64: several units, the last ones part filled
])
def test_host_batches(gpu_ctx, oracle_lib, dtype, N, K, M):
    """qwn_cuda_abi_hypervsq2_gemm with more than 16 tokens."""
    check = check_q4_0 if dtype == "q4_0" else check_hvsq2
    check(gpu_ctx, oracle_lib, N, K, seed=N + K + M, M=M)


@pytest.mark.parametrize("dtype", ["q4_0", "hvsq2"])
@pytest.mark.parametrize("N,K,M", [(77, 300, 40), (130, 520, 100), (1030, 777, 129)])
def test_host_batches_of_fp32_tokens(gpu_ctx, oracle_lib, dtype, N, K, M):
    """fp32 tokens, quantized on the device behind the images of several
    groups: the oracle's product of its own quantized tokens."""
    rng = np.random.default_rng(N + M)
    w, x = synth.weights(dtype, rng, N, K), synth.activations(rng, M, K)
    q8, xs, sums = oracle_lib.quantize(x)
    h = gpu_ctx.upload(w, dtype, N, K)
    try:
        y = gpu_ctx.gemm(h, x, N, K)
    finally:
        gpu_ctx.release(h)
    for t in range(M):
        ref = (oracle_lib.gemv_q4_0_q8(w, q8[t], float(xs[t]), K, N) if dtype == "q4_0" else
               oracle_lib.gemv_hvsq2(w, q8[t], sums[t], float(xs[t]), K, N))
        ok, worst = gemv_close(y[t], ref)
        assert ok, f"token {t}: worst {worst:.3g} of tolerance"


@pytest.mark.parametrize("N,M", [
    (65537, 1),      # one row past those that are stored to the host directly: a ragged last piece
    (1021, 150),     # rows that pieces end inside of
    (70003, 300),    # many windows
])
def test_host_results_in_pieces(gpu_ctx, oracle_lib, N, M):
    """Results as the device wrote them, piece by piece, into rows of a larger
    stride: every value there, the gaps untouched.  Every row of every pass
    has a scale of its own, so a piece that another row, window or pass left
    behind is another value."""
    import ctypes
    rng = np.random.default_rng(N + M)
    w = synth.q4_0_weights(rng, N, 64)
    token = rng.integers(-127, 128, 64, dtype=np.int8)
    q8 = np.tile(token, (M, 1))
    ref = oracle_lib.gemv_q4_0_q8(w, token, 1.0, 64, N)
    h = gpu_ctx.upload(w, "q4_0", N, 64)
    try:
        for turn in range(3):
            xs = (1.0 + np.arange(M) / 256.0 + 4.0 * turn).astype(np.float32)
            out = np.full((M, N + 3), np.nan, dtype=np.float32)
            req = abi.GemmRequest(tensor=h, input_q8=q8.ctypes.data, input_scale=0.0, input_scales=xs.ctypes.data,
                                  output=out.ctypes.data, batch=M, rows=N, cols=64, input_stride=64,
                                  output_stride=N + 3, input_mode=abi.INPUT_Q8)
            tm = abi.Telemetry()
            gpu_ctx.lib.check("gemm", gpu_ctx.lib.lib.qwn_cuda_abi_hypervsq2_gemm(gpu_ctx._h, ctypes.byref(req),
                                                                                ctypes.byref(tm)))
            assert np.isnan(out[:, N:]).all()
            # two fp32 sums of two products; neighbouring scales are 2^-11 or more apart
            want = ref[None, :] * xs[:, None]
            assert np.allclose(out[:, :N], want, rtol=1e-5, atol=1e-5 * np.abs(ref).max())
    finally:
        gpu_ctx.release(h)


def test_every_call_adds_its_kernel_time(gpu_ctx):
    """gpu_kernel_ms on the path whose results are polled for: a call that
    adds nothing read its events before they were complete."""
    rng = np.random.default_rng(5)
    h = gpu_ctx.upload(synth.q4_0_weights(rng, 256, 512), "q4_0", 256, 512)
    q8, xs = rng.integers(-127, 128, (20, 512), dtype=np.int8), np.ones(20, dtype=np.float32)
    try:
        ms = [gpu_ctx.telemetry().gpu_kernel_ms]
        for _ in range(200):
            gpu_ctx.gemm(h, q8, 256, 512, scales=xs)
            ms.append(gpu_ctx.telemetry().gpu_kernel_ms)
    finally:
        gpu_ctx.release(h)
    steps = np.diff(ms)
    assert (steps > 0).all() and steps.max() < 100.0


@pytest.mark.parametrize("N,M", [
    (40, 16384 + 77),        # the images' second span, from its first token on
    (1, 65535 * 64 + 17),    # more token tiles than one launch holds
])
def test_host_batches_of_any_length(hip_lib, N, M):
    """One call over more tokens than one set of images, every value against
    the exact product of the codes."""
    K = 32
    rng = np.random.default_rng(N)
    w = synth.q4_0_weights(rng, N, K)
    block = w.reshape(N, 18)
    d = block[:, :2].copy().view(np.float16).astype(np.float64)
    code = np.stack((block[:, 2:] & 15, block[:, 2:] >> 4), axis=-1).reshape(N, K).astype(np.int32) - 8
    q8 = rng.integers(-127, 128, (M, K), dtype=np.int8)
    xs = (0.5 + np.arange(M) % 31 / 16.0).astype(np.float32)
    with abi.Context(hip_lib, device=0) as ctx:   # its buffers go with it
        h = ctx.upload(w, "q4_0", N, K)
        y = ctx.gemm(h, q8, N, K, scales=xs)
        ctx.release(h)
    for t0 in range(0, M, 1 << 20):
        q, s = q8[t0:t0 + (1 << 20)], xs[t0:t0 + (1 << 20), None]
        ref = (q.astype(np.float64) @ code.T.astype(np.float64)) * d.T * s   # one block a row
        # an fp32 product by the block's scale, one by the token's
        assert (np.abs(y[t0:t0 + (1 << 20)] - ref) <= 3 * 2.0 ** -24 * np.abs(ref)).all()


@pytest.mark.parametrize("max_ctx,prompt,tokens", [(512, 64, 64), (512, 65, 512), (2048, 300, 1024), (64, 33, 64)])
def test_block_size_of_a_prompt(gpu_ctx, max_ctx, prompt, tokens):
    """generate's prefill_block_tokens: narrow blocks up to 64 tokens, else the decoder's wide ones."""
    rng = np.random.default_rng(max_ctx)
    dec = abi.ResidentDecoder(gpu_ctx, synth.decoder_model(rng, config(256, 256, 1, 1, 64, max_ctx), "q4_0"))
    try:
        assert dec.generate(synth.prompt_tokens(rng, 500, prompt), 1)[1].prefill_block_tokens == tokens
    finally:
        dec.close()


def test_wide_decoder_memory(gpu_ctx):
    """A decoder holds one [1024][intermediate] activation for its long
    blocks (gate/up are stored as one), not two."""
    import torch
    cfg = config(256, 16384, 2, 1, 128, 1024)
    model = synth.decoder_model(np.random.default_rng(3), cfg, "q4_0")
    free = torch.cuda.mem_get_info()[0]
    dec = abi.ResidentDecoder(gpu_ctx, model)
    try:
        used = free - torch.cuda.mem_get_info()[0]
        assert dec.prefill(synth.prompt_tokens(np.random.default_rng(4), 500, 1024))[0].shape == (500,)
    finally:
        dec.close()
    act = 1024 * 16384 * 4
    # the activation, its f16 image (half), and about 16 MB of weights with their MFMA-order copies
    assert act < used < act + act // 2 + (40 << 20), used


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("M,launches", [(1, 2), (16, 2), (64, 2), (65, 2), (16384 + 65, 4)])
def test_launches_of_a_host_batch(hip_lib, M, launches, f32):
    """gpu_kernel_launch_count: the images' launches and the GEMMs', and the
    quantize in front of the MFMA path's for fp32 tokens (the GEMV's image
    launch quantizes by itself)."""
    rng = np.random.default_rng(M)
    x = synth.activations(rng, M, 256) if f32 else rng.integers(-127, 128, (M, 256), dtype=np.int8)
    with abi.Context(hip_lib, device=0) as ctx:
        h = ctx.upload(synth.q4_0_weights(rng, 64, 256), "q4_0", 64, 256)
        n = ctx.telemetry().gpu_kernel_launch_count
        ctx.gemm(h, x, 64, 256, scales=None if f32 else np.ones(M, dtype=np.float32))
        assert ctx.telemetry().gpu_kernel_launch_count - n == launches + (f32 and M > 1)
