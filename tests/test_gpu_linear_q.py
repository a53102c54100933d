"""Quantized projections (q35m_linear_q4k / _q5k / _q6k / _iq4xs / _q2_0c /
_stq1_0) through the C ABI against the oracle: bit-exact (the kernels keep the
reference's integer lanes and fp32 accumulation order: the AVX2 GEMV for one
token and for Q6_K, the panel GEMM for Q4_K with several tokens plus the GEMV
for its last n_out % 8 outputs, the scalar per-token dot of Q5_K and IQ4_XS,
the eight-row panel and raw-row orders of Q2_0C and STQ1_0 split as the
reference splits them, by row and, for STQ1_0, by token count), at the
projection shapes of the 4B mixers
(hidden 2560: qkv 8192, gate 4096, beta/alpha 32, ssm_out and attn_output
4096 -> 2560, attn k/v 1024), ragged small shapes, several tokens, zero and
extreme activation blocks, and weight buffers whose size is not a multiple of
16 bytes."""
import sys

import numpy as np
import pytest

import oracle
import q35mix
import quant_blocks as qb

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    c = q35mix.Context(q35mix.qwen35_config(num_layers=1, is_recurrent=[1]), n_seqs=1,
                       kv_capacity=16)
    yield c
    c.close()


def run(ctx, qtype, w, x, n_in, n_out):
    tokens = x.shape[0]
    dw = ctx.bytes_array(w)
    dx = ctx.array((tokens, n_in), x)
    dy = ctx.array((tokens, n_out))
    ctx.linear_q(qtype, dw, dx, dy, n_in, n_out, tokens)
    y = dy.download()
    for a in (dw, dx, dy):
        a.free()
    return y


SHAPES = [(2560, 8192, 1), (2560, 4096, 1), (2560, 32, 1), (4096, 2560, 1), (2560, 1024, 1),
          (256, 7, 1), (512, 33, 5), (2560, 1024, 3), (16384, 19, 2), (2560, 520, 70),
          (4096, 136, 130), (512, 40, 16), (1024, 72, 15), (2560, 64, 4), (1024, 13, 4), (1536, 24, 8),
          (768, 33, 20), (768, 40, 20)]


NAMES = {1: "STQ1_0", 2: "Q2_0C", 4: "Q4_K", 5: "Q5_K", 6: "Q6_K", 14: "IQ4_XS"}
TYPES = [1, 2, 4, 5, 6, 14]


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("n_in,n_out,tokens", SHAPES)
def test_linear_q_bit_exact(ctx, qtype, n_in, n_out, tokens):
    if n_in % qb.VALUES[qtype]:
        n_in += qb.VALUES[qtype] - n_in % qb.VALUES[qtype]
    say(f"linear_q {NAMES[qtype]} n_in={n_in} n_out={n_out} tokens={tokens}")
    rng = np.random.default_rng(1000 * qtype + n_in + n_out + tokens)
    w = qb.random_blocks(rng, qtype, qb.nblocks(qtype, n_out * n_in))
    x = rng.standard_normal((tokens, n_in)).astype(np.float32)
    got = run(ctx, qtype, w, x, n_in, n_out)
    want = oracle.linear_q(qtype, w, x, n_in, n_out)
    bad = np.flatnonzero(got.view(np.uint32) != want.view(np.uint32))
    say(f"  mismatches {bad.size} of {got.size}; max|d| {np.max(np.abs(got - want)):.3e}")
    assert bad.size == 0


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("n_in,n_out,tokens", [(512, 15, 2), (2560, 63, 16), (4608, 65, 17), (1024, 130, 32),
                                               (3584, 17, 33), (512, 257, 64), (5120, 34, 65), (1536, 129, 191),
                                               (512, 8190, 33), (1024, 2047, 100), (512, 3001, 700), (2304, 2111, 20),
                                               (16384, 4111, 3), (2560, 1701, 16), (2560, 63, 20), (16384, 1031, 18),
                                               (9728, 10260, 2)])
def test_linear_gemm_tiles(ctx, qtype, n_in, n_out, tokens):
    """The matrix-core tiles at the edges of their rows (16 a wave), tokens
    (16, 32, 64) and block pipelines, the rows the tiles leave to the GEMV, and
    the shapes that the GEMV takes whole, bit for bit (STQ1_0: panel and raw
    row orders by the token count).  Which kernel a shape takes:
    test_linear_few_tokens, test_linear_q6k_forms, test_linear_q4k_forms."""
    n_in += -n_in % qb.VALUES[qtype]
    rng = np.random.default_rng(31 * qtype + n_in + n_out + tokens)
    w = qb.random_blocks(rng, qtype, qb.nblocks(qtype, n_out * n_in))
    x = rng.standard_normal((tokens, n_in)).astype(np.float32)
    got = run(ctx, qtype, w, x, n_in, n_out)
    assert np.array_equal(got.view(np.uint32), oracle.linear_q(qtype, w, x, n_in, n_out).view(np.uint32))


GEMV_NAME = {1: "linear_qt<1>", 2: "linear_qt<2>", 4: "linear_q<4>", 5: "linear_qs<5>", 6: "linear_q<6>", 14: "linear_qs<14>"}


def run_named(ctx, qtype, n_in, n_out, tokens, seed):
    """One projection against the oracle, bit for bit; the kernels it ran."""
    rng = np.random.default_rng(seed + 31 * qtype + n_in + n_out + tokens)
    w = qb.random_blocks(rng, qtype, qb.nblocks(qtype, n_out * n_in))
    x = rng.standard_normal((tokens, n_in)).astype(np.float32)
    ctx.profile(True)
    got = run(ctx, qtype, w, x, n_in, n_out)
    ran = ctx.profile_read()
    ctx.profile(False)
    assert np.array_equal(got.view(np.uint32), oracle.linear_q(qtype, w, x, n_in, n_out).view(np.uint32))
    return ran


@pytest.mark.parametrize("qtype,n_in,n_out,fused", [
    (4, 512, 50000, True), (5, 1024, 49152, True), (5, 1024, 49153, False), (6, 512, 50001, False), (2, 1536, 50000, True),
    (14, 1280, 49153, False), (1, 1280, 98305, False), (4, 6400, 5, False), (4, 6400, 6145, True), (6, 6400, 2051, True),
    (5, 9728, 1536, True), (5, 9728, 1537, False), (2, 9728, 2049, False), (2, 9728, 3073, True), (1, 9728, 4097, False),
    (5, 10496, 100, True), (14, 10496, 100, False), (14, 10496, 1025, True), (6, 10496, 100, False), (4, 16384, 3, True)])
def test_linear_one_token_forms(ctx, qtype, n_in, n_out, fused):
    """One token on both sides of the rule for quantizing its row inside the
    projection."""
    ran = run_named(ctx, qtype, n_in, n_out, 1, 500)
    assert GEMV_NAME[qtype] in ran and ("q8k_quantize" not in ran) == fused


@pytest.mark.parametrize("qtype", [5, 14, 2, 1])
@pytest.mark.parametrize("n_in,n_out,tokens,gemv", [(4096, 257, 2, True), (4096, 30, 16, True), (4096, 30, 17, False),
                                                    (9728, 41, 5, True), (16384, 19, 4, True), (3584, 331, 3, True),
                                                    (2560, 10300, 2, True), (2560, 10300, 12, False), (512, 40, 2, False),
                                                    (1024, 8200, 3, False), (2560, 40000, 17, False), (9728, 10300, 4, False)])
def test_linear_few_tokens(ctx, qtype, n_in, n_out, tokens, gemv):
    """A few tokens of the formats that run per token: the GEMV over several
    tokens a workgroup, and the matrix cores on the other side of the rule
    (32-token tiles of wide outputs among them)."""
    ran = run_named(ctx, qtype, n_in, n_out, tokens, 900)
    assert (GEMV_NAME[qtype] in ran) == gemv and (f"linear_gemm<{qtype}>" in ran) != gemv


@pytest.mark.parametrize("n_in,n_out,tokens,kernels", [
    (2560, 8192, 3, ["linear_q<6>"]), (2560, 2053, 8, ["linear_q<6>"]), (2560, 1000, 17, ["linear_gemm<6>"]),
    (16384, 521, 5, ["linear_q<6>"]), (2560, 12001, 2, ["linear_q<6>"]), (2560, 12001, 7, ["q6k_gemm"]),
    (2560, 16390, 3, ["linear_q<6>"]), (2560, 16390, 4, ["q6k_gemm"]), (9728, 8200, 2, ["linear_gemm<6>"]),
    (5376, 8203, 4, ["linear_gemm<6>", "linear_q<6>"]), (5376, 4101, 33, ["q6k_gemm", "linear_q<6>"]),
    (768, 2051, 100, ["q6k_gemm", "linear_q<6>"]), (768, 33, 20, ["linear_gemm<6>", "linear_q<6>"]),
    (512, 4120, 17, ["q6k_gemm"]), (512, 4080, 16, ["linear_gemm<6>"])])
def test_linear_q6k_forms(ctx, n_in, n_out, tokens, kernels):
    """Q6_K of several tokens on both sides of the rules between the GEMV, the
    small tiles and the 64-token tiles; with an odd number of blocks the last
    row goes to the GEMV."""
    ran = run_named(ctx, 6, n_in, n_out, tokens, 1900)
    assert sorted(k for k in ran if k != "q8k_quantize") == sorted(kernels)


@pytest.mark.parametrize("n_in,n_out,tokens,kernels", [
    (512, 32768, 16, ["linear_gemm<4>"]), (512, 32776, 16, ["q4k_gemm"]), (768, 65529, 2, ["linear_gemm<4>", "linear_q<4>"]),
    (768, 32776, 18, ["q4k_gemm"]), (1280, 12291, 90, ["linear_gemm<4>", "linear_q<4>"]), (768, 3009, 800, ["q4k_gemm", "linear_q<4>"]),
    (2560, 1041, 2050, ["q4k_gemm", "linear_q<4>"])])
def test_linear_q4k_forms(ctx, n_in, n_out, tokens, kernels):
    """The same for Q4_K: small tiles and 64-token tiles, the GEMV for the last
    n_out % 8 rows."""
    ran = run_named(ctx, 4, n_in, n_out, tokens, 2900)
    assert sorted(k for k in ran if k != "q8k_quantize") == sorted(kernels)


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("n_in,n_out", [(512, 1), (512, 33), (4096, 17), (4608, 129), (10240, 5), (10752, 9), (16384, 3)])
def test_linear_q_one_token_quantizes(ctx, qtype, n_in, n_out):
    """One token, the row quantized by the projection's own workgroups (four
    waves of rows, a last one with waves past the end; one, two and four
    passes of blocks), bit for bit, and the same as with the row quantized
    before."""
    rng = np.random.default_rng(11 * qtype + n_in + n_out)
    w = qb.random_blocks(rng, qtype, qb.nblocks(qtype, n_out * n_in))
    x = rng.standard_normal((1, n_in)).astype(np.float32)
    x[0, 256:512] = 0.0
    x[0, 40] = -x[0, 30]
    got = run(ctx, qtype, w, x, n_in, n_out)
    assert np.array_equal(got.view(np.uint32), oracle.linear_q(qtype, w, x, n_in, n_out).view(np.uint32))
    dw, dx, dy = ctx.bytes_array(w), ctx.array((1, n_in), x), ctx.array((1, n_out))
    q8 = ctx.quantize_q8k(dx, n_in, 1)
    ctx.linear_q_prequant(qtype, dw, q8, dy, n_in, n_out, 1)
    assert np.array_equal(dy.download().view(np.uint32), got.view(np.uint32))
    for a in (dw, dx, dy, q8):
        a.free()


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("shift", [0, 256, -256])
def test_linear_q_one_token_in_place(ctx, qtype, shift):
    """y on top of x, or partly over its end or its start (shift floats): the
    row is quantized as a whole before anything is stored.  Buffers that only
    touch are apart."""
    n_in = n_out = 5120
    rng = np.random.default_rng(77 + qtype)
    w = qb.random_blocks(rng, qtype, qb.nblocks(qtype, n_out * n_in))
    x = rng.standard_normal((1, n_in)).astype(np.float32)
    want = oracle.linear_q(qtype, w, x, n_in, n_out)
    dw, buf = ctx.bytes_array(w), ctx.array((3, n_in))
    view = lambda at: q35mix.DeviceView(buf, at, (1, n_in))  # noqa: E731
    for at, fused in ((n_in + shift, False), (2 * n_in, True), (0, True)):
        host = np.zeros((3, n_in), np.float32)
        host[1] = x
        buf.upload(host)
        ctx.profile(True)
        ctx.linear_q(qtype, dw, view(n_in), view(at), n_in, n_out, 1)
        ran = ctx.profile_read()
        ctx.profile(False)
        assert ("q8k_quantize" not in ran) == fused
        got = buf.download().reshape(-1)[at:at + n_out]
        assert np.array_equal(got.view(np.uint32), want.reshape(-1).view(np.uint32))
    dw.free()
    buf.free()


@pytest.mark.parametrize("qtype", TYPES)
def test_linear_q_activation_edges(ctx, qtype):
    """Zero blocks (scale 0), a first extremum that is positive (negative
    scale) or repeated with both signs, ties at .5 after scaling, huge and tiny
    magnitudes, and an fp16 subnormal weight scale."""
    n_in, n_out = 2048, 40
    rng = np.random.default_rng(77 + qtype)
    w = qb.random_blocks(rng, qtype, qb.nblocks(qtype, n_out * n_in))
    d_off = {6: 208, 1: 40}.get(qtype, 0)
    w.reshape(-1, qb.BYTES[qtype])[3, d_off:d_off + 2] = np.frombuffer(np.float16(3e-6).tobytes(), np.uint8)
    x = rng.standard_normal((2, n_in)).astype(np.float32)
    x[0, 0:256] = 0.0
    x[0, 256:512] *= 1e-30
    x[0, 512 + 5], x[0, 512 + 9] = 50.0, -50.0
    x[0, 768 + 2], x[0, 768 + 1] = 50.0, -50.0
    blk = x[1, 1024:1280]
    blk[:] = np.arange(256, dtype=np.float32) - 128.0   # iscale exactly 127/128... ties
    blk[0] = -127.0
    blk[1:] = np.clip(blk[1:], -126.5, 126.5)
    x[1, 1280:1536] *= 1e20
    got = run(ctx, qtype, w, x, n_in, n_out)
    want = oracle.linear_q(qtype, w, x, n_in, n_out)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_linear_q_rejects_bad_arguments(ctx):
    dw = ctx.bytes_array(np.zeros(144 * 4, np.uint8))
    dx = ctx.array((1, 512))
    dy = ctx.array((1, 2))
    L = q35mix.lib()
    h = ctx.handle
    assert L.q35m_linear_q4k(h, dw.ptr, dx.ptr, dy.ptr, 300, 2, 1) == q35mix.ERR_UNSUPPORTED
    assert L.q35m_linear_q4k(h, dw.ptr + 4, dx.ptr, dy.ptr, 512, 2, 1) == q35mix.ERR_INVALID
    assert L.q35m_linear_q6k(h, dw.ptr, dx.ptr, dy.ptr, 512, 0, 1) == q35mix.ERR_INVALID
    assert L.q35m_linear_q6k(h, dw.ptr, dx.ptr, dy.ptr, 512, 2, 0) == q35mix.ERR_INVALID
    assert L.q35m_linear_q6k(h, None, dx.ptr, dy.ptr, 512, 2, 1) == q35mix.ERR_INVALID
    assert L.q35m_linear_q2_0c(h, dw.ptr, dx.ptr, dy.ptr, 256, 2, 1) == q35mix.ERR_UNSUPPORTED
    assert L.q35m_linear_q2_0c_prequant(h, dw.ptr, dx.ptr, dy.ptr, 768, 2, 1) == q35mix.ERR_UNSUPPORTED
    assert L.q35m_linear_stq1_0(h, dw.ptr + 2, dx.ptr, dy.ptr, 512, 2, 1) == q35mix.ERR_INVALID
    for a in (dw, dx, dy):
        a.free()


def test_prequant_matches_one_shot(ctx):
    """Quantize once, three projections (the reference's attention decode:
    Qwen35Model.Decode.cs:286-292), each bit-identical to the one-shot call
    and to the oracle."""
    n_in = 2560
    rng = np.random.default_rng(5)
    x = rng.standard_normal((2, n_in)).astype(np.float32)
    dx = ctx.array((2, n_in), x)
    q8 = ctx.quantize_q8k(dx, n_in, 2)
    for qtype, n_out in ((4, 8192), (4, 1024), (6, 1024), (5, 1024), (14, 32), (2, 1024), (1, 8192), (1, 13)):
        w = qb.random_blocks(rng, qtype, qb.nblocks(qtype, n_out * n_in))
        dw = ctx.bytes_array(w)
        dy = ctx.array((2, n_out))
        ctx.linear_q_prequant(qtype, dw, q8, dy, n_in, n_out, 2)
        got = dy.download()
        want = oracle.linear_q(qtype, w, x, n_in, n_out)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (qtype, n_out)
        assert np.array_equal(got.view(np.uint32), run(ctx, qtype, w, x, n_in, n_out).view(np.uint32))
        dw.free()
        dy.free()
    q8.free()
    dx.free()


@pytest.mark.parametrize("n_in,n_out,tokens", [(2560, 32, 1), (2560, 4096, 2), (4096, 129, 3), (17, 70, 5),
                                               (24, 3, 1), (7, 65, 2), (2561, 40, 70), (1, 1, 1)])
def test_linear_f32_bit_exact(ctx, n_in, n_out, tokens):
    """F32 weights: Ops.DotF32's lane order, bit for bit, also at widths that
    are not multiples of 16, 8 or 4 (the scalar loads and the 8-wide stride)."""
    say(f"linear_f32 n_in={n_in} n_out={n_out} tokens={tokens}")
    rng = np.random.default_rng(n_in + 7 * n_out + tokens)
    w = rng.standard_normal((n_out, n_in)).astype(np.float32)
    x = rng.standard_normal((tokens, n_in)).astype(np.float32)
    if n_in >= 17:
        x[0, 0] = 2.0 ** 24          # order-dependent row
        w[0, :] = 1.0
        x[0, 1:] = 1.0
    dw, dx, dy = ctx.array((n_out, n_in), w), ctx.array((tokens, n_in), x), ctx.array((tokens, n_out))
    ctx.linear_f32(dw, dx, dy, n_in, n_out, tokens)
    got = dy.download()
    want = oracle.linear_f32(w, x, n_in, n_out)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    for a in (dw, dx, dy):
        a.free()


@pytest.mark.parametrize("n_in,n_out,tokens", [(2569, 5, 1), (5200, 3, 2), (64, 9, 33), (527, 261, 5), (600, 264, 70),
                                               (283, 270, 65), (15, 300, 61), (256, 8, 4100), (129, 33, 9), (100, 300, 70),
                                               (1, 9000, 3), (63, 65, 130), (64, 65, 130), (127, 301, 5), (128, 301, 5),
                                               (256, 4097, 4), (257, 4097, 4), (384, 4161, 2), (1021, 32801, 1),
                                               (1024, 32768, 1), (1500, 1027, 1), (2049, 1030, 1)])
def test_linear_f32_tiles(ctx, n_in, n_out, tokens):
    """Each form of the F32 projection (4 rows x 1 token, 4 x 4, 8 x 8, direct
    from global memory) at ragged rows and tokens, around its staged column
    chunks (2560, 512, 256, 128) and on both sides of the rules between the
    forms, bit for bit."""
    rng = np.random.default_rng(n_in + 7 * n_out + tokens)
    w = rng.standard_normal((n_out, n_in)).astype(np.float32)
    x = rng.standard_normal((tokens, n_in)).astype(np.float32)
    dw, dx, dy = ctx.array((n_out, n_in), w), ctx.array((tokens, n_in), x), ctx.array((tokens, n_out))
    ctx.linear_f32(dw, dx, dy, n_in, n_out, tokens)
    assert np.array_equal(dy.download().view(np.uint32), oracle.linear_f32(w, x, n_in, n_out).view(np.uint32))
    for a in (dw, dx, dy):
        a.free()


@pytest.fixture()
def pieces_ctx(monkeypatch):
    """A context whose kernels take at most 256 KiB of an operand at once, in
    place of 2 GiB."""
    monkeypatch.setenv("Q35M_TILE_LIMIT_BYTES", str(256 * 1024))
    c = q35mix.Context(q35mix.qwen35_config(num_layers=1, is_recurrent=[1]), n_seqs=1, kv_capacity=16)
    yield c
    c.close()


@pytest.mark.parametrize("qtype,n_in,n_out,tokens", [(4, 512, 1104, 2000), (6, 1024, 424, 700), (6, 768, 425, 700)])
def test_tiled_pieces_match_whole_launch(pieces_ctx, qtype, n_in, n_out, tokens):
    """The 64-token-tile Q4_K / Q6_K kernels go in pieces of whole row and
    token tiles when a call holds more than 2 GiB of weight rows or
    activations; with a 256 KiB piece limit ordinary shapes split the same way
    (several row and token pieces here), bit-identical to the oracle."""
    ran = run_named(pieces_ctx, qtype, n_in, n_out, tokens, 4242)
    assert ran["q4k_gemm" if qtype == 4 else "q6k_gemm"][1] >= 6


@pytest.mark.parametrize("qtype,n_in,n_out,tokens", [(q, 2560, n, 200) for q in TYPES for n in (520, 424)] +
                         [(q, 512, 2100, 1100) for q in (5, 14, 2, 1)] + [(4, 512, 2100, 450), (6, 1024, 60, 1900)])
def test_small_tile_pieces_match_whole_launch(pieces_ctx, qtype, n_in, n_out, tokens):
    """The same for linear_gemm's token pieces, in its split form and its 32-
    and 64-token tiles."""
    ran = run_named(pieces_ctx, qtype, n_in, n_out, tokens, 4243)
    assert ran[f"linear_gemm<{qtype}>"][1] > 1


BLOCK_SHAPES = [(2560, 8192, 2048), (4096, 2560, 2048), (2560, 520, 70), (512, 33, 5), (4096, 136, 130),
                (16384, 19, 2), (1024, 72, 16), (2560, 1024, 3), (256, 7, 129)]


@pytest.mark.parametrize("qtype", [4, 6])
@pytest.mark.parametrize("n_in,n_out,tokens", BLOCK_SHAPES)
def test_linear_q_block_order(ctx, qtype, n_in, n_out, tokens):
    """q35m_set_projection_order(PROJ_BLOCK): Q6_K from 16 tokens (n_out *
    n_in / 256 even) accumulates each block's exact integer sum and applies
    its fp32 scales once.  Checked against the exact value of the quantized
    product (fp64 of the dequantized weights and Q8_K activations: |y - exact|
    <= 2e-6 sum |w x|, the bound the reference's own order meets) and against
    the oracle's reference order (max|d| / max|ref| <= 1e-4); Q4_K and the
    shapes outside the block-order condition stay bit-identical to the
    reference order."""
    say(f"linear_q block order {NAMES[qtype]} n_in={n_in} n_out={n_out} tokens={tokens}")
    rng = np.random.default_rng(7000 + 1000 * qtype + n_in + n_out + tokens)
    w = qb.random_blocks(rng, qtype, qb.nblocks(qtype, n_out * n_in))
    x = rng.standard_normal((tokens, n_in)).astype(np.float32)
    ctx.set_projection_order(q35mix.PROJ_BLOCK)
    try:
        got = run(ctx, qtype, w, x, n_in, n_out)
    finally:
        ctx.set_projection_order(q35mix.PROJ_REFERENCE)
    blocked = qtype == 6 and tokens >= 16 and (n_out * n_in // 256) % 2 == 0
    check_rows = min(tokens, 24)
    sel = np.unique(np.linspace(0, tokens - 1, check_rows).astype(int))
    want = oracle.linear_q(qtype, w, x[sel], n_in, n_out)
    if not blocked:
        assert np.array_equal(got[sel].view(np.uint32), want.view(np.uint32))
        return
    e = float(np.max(np.abs(got[sel] - want)) / np.max(np.abs(want)))
    wd = qb.dequant_f64(qtype, w).reshape(n_out, n_in)
    worst = 0.0
    for i, t in enumerate(sel):
        d, q, _ = qb.parse_q8k(oracle.q8k_quantize(x[t]))
        xd = (d[:, None].astype(np.float64) * q).ravel()
        exact = wd @ xd
        scale = np.abs(wd) @ np.abs(xd)
        worst = max(worst, float(np.max(np.abs(got[t] - exact) / scale)))
    say(f"  vs reference order {e:.2e}; worst |y - exact| / sum|w x| {worst:.2e}")
    assert e <= 1e-4
    assert worst <= 2e-6
