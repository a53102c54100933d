"""Edge cases of the HIP mixers through the C ABI: chunk counts that exercise
every branch of the prefill scan's loop, the 64-sequence decode batch, the
last KV row and the limits the ABI enforces.  Parity gate as in
test_gpu_mixers.py: max|gpu - oracle| / max|oracle| <= 1e-4."""
import ctypes
import sys

import numpy as np
import pytest

import f64_model
import oracle
import q35mix
import synth

pytestmark = pytest.mark.gpu

TOL = 1e-4
NK, NV = 16, 32
NH, NKV, HD = 16, 4, 256
NSEQ, CAP = 64, 256
DIMS = oracle.dims()


def rel(got, ref):
    ref = np.asarray(ref, np.float64)
    return float(np.max(np.abs(np.asarray(got, np.float64) - ref)) / max(np.max(np.abs(ref)), 1e-30))


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    # Layer 0 Gated-DeltaNet, layer 1 GQA; 64 sequences (the batch limit); 256 KV rows.
    c = q35mix.Context(q35mix.qwen35_config(num_layers=2, is_recurrent=[1, 0]), n_seqs=NSEQ,
                       kv_capacity=CAP)
    c.set_deltanet_weights(0, synth.deltanet_weights(NK, NV, 128, salt=31))
    c.set_attn_weights(1, synth.attn_weights(HD, salt=31))
    yield c
    c.close()


@pytest.mark.parametrize("T", [200, 600, 1030, 2049])
def test_deltanet_prefill_chunk_counts(ctx, T):
    """4, 10, 17 and 33 chunks (whole pairs of the scan loop, or one chunk
    left over; ragged last chunk at 1030 and 2049), from a non-zero state."""
    w = synth.deltanet_weights(NK, NV, 128, salt=31)
    st = synth.deltanet_state(NK, NV, 128, salt=500 + T)
    ctx.state_write(0, 5, q35mix.STATE_RECURRENT, st["state"])
    ctx.state_write(0, 5, q35mix.STATE_CONV, st["conv_state"])
    x = synth.deltanet_inputs(T, NK, NV, 128, salt=600 + T)
    args = [ctx.array((T, ctx.conv_dim), x["qkv"]), ctx.array((T, ctx.value_dim), x["z"]),
            ctx.array((T, NV), x["b"]), ctx.array((T, NV), x["a"])]
    out = ctx.array((T, ctx.value_dim))
    ctx.deltanet_prefill(0, 5, T, *args, out)
    o_ref, cs_ref, st_ref, _ = oracle.deltanet_prefill(DIMS, T, x["qkv"], x["z"], x["b"], x["a"],
                                                       w, st["state"], st["conv_state"])
    e_out = rel(out.download(), o_ref)
    e_st = rel(ctx.state_read(0, 5, q35mix.STATE_RECURRENT), st_ref)
    say(f"deltanet_prefill T={T}: out rel err {e_out:.2e}, state rel err {e_st:.2e}")
    assert e_out <= TOL and e_st <= TOL
    np.testing.assert_array_equal(ctx.state_read(0, 5, q35mix.STATE_CONV), cs_ref)


@pytest.mark.parametrize("T", [63, 65, 66, 67, 129])
def test_deltanet_prefill_chunk_tails(ctx, T):
    """Last chunk holding 63, 1, 2, 3 and 1 tokens: the conv's zero padding
    past T, the conv-window write-back from the raw inputs T-3..T-1 when they
    straddle a chunk boundary, and the masked gates of the padded tokens."""
    w = synth.deltanet_weights(NK, NV, 128, salt=31)
    st = synth.deltanet_state(NK, NV, 128, salt=1500 + T)
    ctx.state_write(0, 9, q35mix.STATE_RECURRENT, st["state"])
    ctx.state_write(0, 9, q35mix.STATE_CONV, st["conv_state"])
    x = synth.deltanet_inputs(T, NK, NV, 128, salt=1600 + T)
    args = [ctx.array((T, ctx.conv_dim), x["qkv"]), ctx.array((T, ctx.value_dim), x["z"]),
            ctx.array((T, NV), x["b"]), ctx.array((T, NV), x["a"])]
    out = ctx.array((T, ctx.value_dim))
    ctx.deltanet_prefill(0, 9, T, *args, out)
    o_ref, cs_ref, st_ref, _ = oracle.deltanet_prefill(DIMS, T, x["qkv"], x["z"], x["b"], x["a"],
                                                       w, st["state"], st["conv_state"])
    e_out = rel(out.download(), o_ref)
    e_st = rel(ctx.state_read(0, 9, q35mix.STATE_RECURRENT), st_ref)
    say(f"deltanet_prefill tail T={T}: out rel err {e_out:.2e}, state rel err {e_st:.2e}")
    assert e_out <= TOL and e_st <= TOL
    np.testing.assert_array_equal(ctx.state_read(0, 9, q35mix.STATE_CONV), cs_ref)


def test_decode_batch_of_64(ctx):
    """Both decode mixers with the full 64-sequence batch, ragged KV lengths."""
    seqs = list(range(NSEQ))
    w = synth.deltanet_weights(NK, NV, 128, salt=31)
    states = []
    for s in seqs:
        st = synth.deltanet_state(NK, NV, 128, salt=700 + s)
        ctx.state_write(0, s, q35mix.STATE_RECURRENT, st["state"])
        ctx.state_write(0, s, q35mix.STATE_CONV, st["conv_state"])
        states.append(st)
    x = synth.deltanet_inputs(NSEQ, NK, NV, 128, salt=800)
    out = ctx.array((NSEQ, ctx.value_dim))
    ctx.deltanet_decode(0, seqs, ctx.array((NSEQ, ctx.conv_dim), x["qkv"]),
                        ctx.array((NSEQ, ctx.value_dim), x["z"]), ctx.array((NSEQ, NV), x["b"]),
                        ctx.array((NSEQ, NV), x["a"]), out)
    got = out.download()
    worst = 0.0
    for j, s in enumerate(seqs):
        o_ref, cs_ref, st_ref, _ = oracle.deltanet_decode(DIMS, x["qkv"][j], x["z"][j], x["b"][j],
                                                          x["a"][j], w, states[j]["conv_state"],
                                                          states[j]["state"])
        worst = max(worst, rel(got[j], o_ref))
        if j % 21 == 0:
            assert rel(ctx.state_read(0, s, q35mix.STATE_RECURRENT), st_ref) <= TOL
            np.testing.assert_array_equal(ctx.state_read(0, s, q35mix.STATE_CONV), cs_ref)
    say(f"deltanet_decode batch 64: worst out rel err {worst:.2e}")
    assert worst <= TOL

    wts = synth.attn_weights(HD, salt=31)
    rng = np.random.default_rng(5)
    lens = [int(v) for v in rng.integers(0, CAP - 1, NSEQ)]
    caches = []
    for s, L in zip(seqs, lens):
        ctx.reset(s)
        k, v = synth.kv_prefill(max(L, 1), ctx.kv_dim, salt=900 + s)
        k, v = k[:L], v[:L]
        if L:
            ctx.state_write(1, s, q35mix.STATE_KEYS, k)
            ctx.state_write(1, s, q35mix.STATE_VALUES, v)
            ctx.advance(s, L)
        caches.append((k, v))
    xa = synth.attn_inputs(NSEQ, NH, NKV, HD, salt=901)
    out = ctx.array((NSEQ, ctx.q_dim))
    ctx.attn_decode(1, seqs, ctx.array((NSEQ, 2 * ctx.q_dim), xa["q_gate"]),
                    ctx.array((NSEQ, ctx.kv_dim), xa["k"]), ctx.array((NSEQ, ctx.kv_dim), xa["v"]),
                    out)
    got = out.download()
    worst = 0.0
    for j, L in enumerate(lens):
        ck = np.zeros((L + 1, ctx.kv_dim), np.float32)
        cv = np.zeros_like(ck)
        ck[:L], cv[:L] = caches[j]
        o_ref, _, _ = oracle.attn_decode(DIMS, L, xa["q_gate"][j], xa["k"][j], xa["v"][j], wts, ck,
                                         cv, n_threads=8)
        worst = max(worst, rel(got[j], o_ref))
    say(f"attn_decode batch 64: worst out rel err {worst:.2e}")
    assert worst <= TOL


def test_attn_decode_last_row_then_full(ctx):
    """The decode that writes the last KV row works; the next one reports a
    full cache (Q35M_ERR_CAPACITY) instead of writing past it."""
    s = 7
    ctx.reset(s)
    L = CAP - 1
    k, v = synth.kv_prefill(L, ctx.kv_dim, salt=950)
    ctx.state_write(1, s, q35mix.STATE_KEYS, k)
    ctx.state_write(1, s, q35mix.STATE_VALUES, v)
    ctx.advance(s, L)
    wts = synth.attn_weights(HD, salt=31)
    xa = synth.attn_inputs(1, NH, NKV, HD, salt=951)
    args = [ctx.array((1, 2 * ctx.q_dim), xa["q_gate"]), ctx.array((1, ctx.kv_dim), xa["k"]),
            ctx.array((1, ctx.kv_dim), xa["v"])]
    out = ctx.array((1, ctx.q_dim))
    ctx.attn_decode(1, [s], *args, out)
    ck = np.zeros((CAP, ctx.kv_dim), np.float32)
    cv = np.zeros_like(ck)
    ck[:L], cv[:L] = k, v
    o_ref, ck_ref, _ = oracle.attn_decode(DIMS, L, xa["q_gate"][0], xa["k"][0], xa["v"][0], wts,
                                          ck, cv, n_threads=8)
    assert rel(out.download()[0], o_ref) <= TOL
    assert rel(ctx.state_read(1, s, q35mix.STATE_KEYS)[L], ck_ref[L]) <= TOL
    ctx.advance(s, 1)
    with pytest.raises(q35mix.Q35Error) as ei:
        ctx.attn_decode(1, [s], *args, out)
    assert ei.value.code == q35mix.ERR_CAPACITY


def test_abi_limits(ctx):
    """Batch limit, repeated sequence ids, partial K/V rows, bad state kind."""
    a = ctx.array((1, 8))
    with pytest.raises(q35mix.Q35Error) as ei:
        ctx.deltanet_decode(0, list(range(NSEQ)) + [0], a, a, a, a, a)
    assert ei.value.code == q35mix.ERR_CAPACITY
    with pytest.raises(q35mix.Q35Error) as ei:
        ctx.deltanet_decode(0, [3, 3], a, a, a, a, a)
    assert ei.value.code == q35mix.ERR_INVALID
    with pytest.raises(q35mix.Q35Error) as ei:
        ctx.state_write(1, 0, q35mix.STATE_KEYS, np.zeros((3, 100), np.float32))
    assert ei.value.code == q35mix.ERR_INVALID
    with pytest.raises(q35mix.Q35Error) as ei:
        ctx.state_read(1, 0, 9)
    assert ei.value.code == q35mix.ERR_INVALID


def test_attn_prefill_row_limit():
    """The prefill flash kernel addresses a kv head's rows through a buffer
    descriptor (32-bit offsets): a prefill that would reach past 2^21 cached
    rows is refused with ERR_UNSUPPORTED before any work (the capacity check
    comes first, so the context holds 2^21 + 1 rows: 8 GiB of K/V)."""
    rows = (1 << 21) + 1
    c = q35mix.Context(q35mix.qwen35_config(num_layers=1, is_recurrent=[0]), n_seqs=1, kv_capacity=rows)
    try:
        c.set_attn_weights(0, synth.attn_weights(256))
        a = c.array((1, 8))
        with pytest.raises(q35mix.Q35Error) as ei:
            c.attn_prefill(0, 0, rows, a, a, a, a)
        assert ei.value.code == q35mix.ERR_UNSUPPORTED
    finally:
        c.close()


def test_deltanet_prefill_long_context():
    """T = 16421 (257 chunks: an odd count, the last holding 37 tokens) in a
    2 k-head / 4 v-head geometry, from a non-zero state: the chunk scan's
    recurrence over a long chain and the workspace offsets at large chunk
    counts, outputs of every token and the final state against the oracle."""
    nk, nv, T = 2, 4, 16421
    d = oracle.dims(n_k_heads=nk, n_v_heads=nv)
    cfg = q35mix.qwen35_config(num_layers=1, n_k_heads=nk, n_v_heads=nv, is_recurrent=[1])
    with q35mix.Context(cfg, n_seqs=1, kv_capacity=4) as c:
        w = synth.deltanet_weights(nk, nv, 128, salt=77)
        c.set_deltanet_weights(0, w)
        st = synth.deltanet_state(nk, nv, 128, salt=78)
        c.state_write(0, 0, q35mix.STATE_RECURRENT, st["state"])
        c.state_write(0, 0, q35mix.STATE_CONV, st["conv_state"])
        x = synth.deltanet_inputs(T, nk, nv, 128, salt=79)
        out = c.array((T, c.value_dim))
        say(f"deltanet_prefill long T={T}: launching")
        c.deltanet_prefill(0, 0, T, c.array((T, c.conv_dim), x["qkv"]), c.array((T, c.value_dim), x["z"]),
                           c.array((T, nv), x["b"]), c.array((T, nv), x["a"]), out)
        got = out.download()
        o_ref, cs_ref, st_ref, _ = oracle.deltanet_prefill(d, T, x["qkv"], x["z"], x["b"], x["a"], w,
                                                           st["state"], st["conv_state"])
        e_out = rel(got, o_ref)
        e_last = rel(got[-64:], o_ref[-64:])
        e_st = rel(c.state_read(0, 0, q35mix.STATE_RECURRENT), st_ref)
        say(f"  out rel err {e_out:.2e} (last chunk {e_last:.2e}), state rel err {e_st:.2e}")
        assert e_out <= TOL and e_last <= TOL and e_st <= TOL
        np.testing.assert_array_equal(c.state_read(0, 0, q35mix.STATE_CONV), cs_ref)


def _attn_prefill_data(nh, nkv, start, T, kmul=None, vmul=None, q_norm=None, new_v=1.0, k_norm=None):
    """Inputs, weights and cached rows (keys, values) of an attention prefill."""
    rng = np.random.default_rng(1000 * nh + 10 * start + T)
    wts = synth.attn_weights(256)
    if q_norm is not None:
        wts["q_norm"] = np.full(256, q_norm, np.float32) if np.isscalar(q_norm) else q_norm
    if k_norm is not None:
        wts["k_norm"] = k_norm
    ck = np.zeros((start + T, nkv * 256), np.float32)
    cv = np.zeros_like(ck)
    ck[:start] = rng.standard_normal((start, nkv * 256))
    cv[:start] = rng.standard_normal((start, nkv * 256))
    for arr, mul in ((ck, kmul), (cv, vmul)):
        for row, f in mul or ():
            arr[row] *= np.float32(f)
    x = synth.attn_inputs(T, nh, nkv, 256, salt=3 + T)
    x["v"] = x["v"] * np.tile(np.broadcast_to(np.asarray(new_v, np.float32), 256), nkv)
    return x, wts, ck, cv


def _attn_prefill_case(nh, nkv, start, T, kmul=None, vmul=None, q_norm=None, new_v=1.0, k_norm=None):
    """One attention prefill of T tokens behind `start` cached rows against
    the oracle; kmul / vmul scale single cached rows, (row, factor), new_v the
    new rows of V (a number, or one a dim)."""
    dims = oracle.dims(n_heads=nh, n_kv_heads=nkv)
    x, wts, ck, cv = _attn_prefill_data(nh, nkv, start, T, kmul, vmul, q_norm, new_v, k_norm)
    with q35mix.Context(q35mix.qwen35_config(num_layers=1, num_heads=nh, num_kv_heads=nkv, is_recurrent=[0]), n_seqs=1,
                        kv_capacity=start + T) as c:
        c.set_attn_weights(0, wts)
        if start:
            c.state_write(0, 0, q35mix.STATE_KEYS, ck[:start])
            c.state_write(0, 0, q35mix.STATE_VALUES, cv[:start])
            if c.kv_len(0) < start:
                c.advance(0, start - c.kv_len(0))
        out = c.array((T, nh * 256))
        c.attn_prefill(0, 0, T, c.array((T, 2 * nh * 256), x["q_gate"]), c.array((T, nkv * 256), x["k"]),
                       c.array((T, nkv * 256), x["v"]), out)
        got = out.download()
    with np.errstate(all="ignore"):
        want, _, _ = oracle.attn_prefill(dims, start, T, x["q_gate"], x["k"], x["v"], wts, ck, cv, n_threads=8)
    return got, want


@pytest.mark.parametrize("nh,nkv,start,T", [(16, 4, 0, 1), (16, 4, 31, 33), (16, 4, 32, 32), (16, 4, 33, 31), (16, 4, 300, 65),
                                            (16, 4, 4000, 3), (16, 4, 0, 1100), (4, 4, 100, 129), (8, 4, 63, 65),
                                            (8, 1, 700, 40), (16, 2, 0, 34)])
def test_attn_prefill_chunks(nh, nkv, start, T):
    """Query blocks and key tiles (32 rows) at their edges, blocks of one and
    of many chunks, 1, 2, 4 and 8 q heads a kv head."""
    got, want = _attn_prefill_case(nh, nkv, start, T)
    e = np.max(np.abs(got - want)) / np.max(np.abs(want))
    say(f"attn_prefill {nh}/{nkv} start {start} T {T}: {e:.2e}")
    assert e <= 1e-5


@pytest.mark.parametrize("case", ["v_spread", "k_spread", "v_zero_rows", "huge_v", "q_huge", "v_inf", "v_nan"])
def test_attn_prefill_value_ranges(case):
    """Cached rows whose magnitudes lie far apart, huge or not finite, and q
    beyond the split's range: the query blocks that read them take the fp32
    form (one chunk and many); a tile of zero rows stays."""
    for start, T in ((200, 40), (3000, 37)):
        kw = {"v_spread": {"vmul": [(50, 2.0 ** 20)]}, "k_spread": {"kmul": [(60, 2.0 ** -15)]},
              "v_zero_rows": {"vmul": [(r, 0.0) for r in range(64, 96)]}, "huge_v": {"vmul": [(r, 1e25) for r in range(start)]},
              "q_huge": {"q_norm": 2.0 ** 66, "kmul": [(r, 2.0 ** -66) for r in range(start)]},
              "v_inf": {"vmul": [(50, np.inf)]}, "v_nan": {"vmul": [(50, np.nan)]}}[case]
        got, want = _attn_prefill_case(16, 4, start, T, **kw)
        fin = np.isfinite(want)
        assert np.array_equal(np.isfinite(got), fin) and np.array_equal(np.isnan(got), np.isnan(want))
        if fin.any():
            e = np.max(np.abs(got - want)[fin]) / np.max(np.abs(want[fin]))
            say(f"attn_prefill {case} start {start}: {e:.2e}")
            assert e <= 1e-5


@pytest.mark.parametrize("start,T", [(0, 40), (200, 40), (3000, 37)])
@pytest.mark.parametrize("exp", [-38, -45, -60, -90])
def test_attn_prefill_small_values(start, T, exp):
    """V rows of one small magnitude, in and below the range of the fp16
    split: nothing is lost."""
    f = 2.0 ** exp
    got, want = _attn_prefill_case(16, 4, start, T, vmul=[(r, f) for r in range(start)], new_v=f)
    e = np.max(np.abs(got - want)) / np.max(np.abs(want))
    say(f"attn_prefill V of 2^{exp}, start {start}: {e:.2e}")
    assert e <= 1e-5


@pytest.mark.parametrize("which", ["v", "k"])
@pytest.mark.parametrize("exp", [15, 20, 24])
def test_attn_prefill_column_ranges(which, exp):
    """Dims of V, or of K with those of q the other way round, whose magnitudes
    lie 2^exp apart: every dim of the output keeps the precision of its own
    values (each row's largest error against the oracle over that dim's rms)."""
    start, T = 0, 300
    col = np.exp2(-exp * np.arange(256) / 255).astype(np.float32)
    if which == "v":
        got, want = _attn_prefill_case(16, 4, start, T, new_v=col)
        e = np.max(np.abs(got - want).reshape(T, 16, 256) / np.sqrt(np.mean(want.reshape(T, 16, 256) ** 2, axis=(0, 1))))
    else:
        got, want = _attn_prefill_case(16, 4, start, T, k_norm=2 * col - 1, q_norm=2 / col - 1)
        e = np.max(np.abs(got - want)) / np.sqrt(np.mean(want ** 2))
    say(f"attn_prefill {which} columns 2^{exp} apart: {e:.2e}")
    # Twice the 2.7e-5 that fp32 products leave here (the split alone: 2.8e-4 for
    # V and 5.7e-4 for K at 2^24).
    assert e <= 5e-5


def _attn_f64_error(start, T, got, **kw):
    """2-norm of the difference to the float64 model over the model's."""
    x, wts, ck, cv = _attn_prefill_data(16, 4, start, T, **kw)
    want, _, _ = f64_model.attn(start, x["q_gate"], x["k"], x["v"], wts, ck, cv, 16, 4, 256)
    want = want.reshape(T, -1)
    return np.linalg.norm(got - want) / np.linalg.norm(want)


def test_attn_prefill_zero_tile_stays_split():
    """A tile of 32 zero V rows is within the split's range: the result keeps
    the split's distance to 64 bits, about half of the fp32 products' (5.8e-7
    and 1.2e-6 at this size), and so does one with half of them zero."""
    start, T = 3000, 37
    for rows in (range(64, 96), range(64, 80)):
        kw = {"vmul": [(r, 0.0) for r in rows]}
        got, _ = _attn_prefill_case(16, 4, start, T, **kw)
        e = _attn_f64_error(start, T, got, **kw)
        say(f"attn_prefill {len(rows)} zero V rows: {e:.2e}")
        assert e <= 8e-7


@pytest.mark.parametrize("start,T", [(0, 300), (500, 200), (6000, 100)])
@pytest.mark.parametrize("value", [2.0 ** 30, 2.0 ** 60, 2.0 ** -60, np.inf])
def test_attn_prefill_late_values(start, T, value):
    """V outside the split's range in the last row: the query blocks (32 rows)
    that do not read its tile (32 rows from row 0 of the cache) have the bits
    they have without it."""
    import unittest.mock
    real = synth.attn_inputs

    def late(*a, **k):
        x = real(*a, **k)
        x["v"] = x["v"].copy()
        x["v"][-1] *= np.float32(value)
        return x

    plain, _ = _attn_prefill_case(16, 4, start, T)
    with unittest.mock.patch.object(synth, "attn_inputs", late):
        got, want = _attn_prefill_case(16, 4, start, T)
    before = max(32 * b for b in range(T // 32 + 1) if (start + 32 * b + 31) // 32 <= (start + T - 1) // 32)
    assert before > 0 and np.array_equal(got[:before].view(np.uint32), plain[:before].view(np.uint32))
    if np.isfinite(value):      # (an infinity times the 0 of a masked weight is NaN for the rows of its 16)
        for t in range(before, T):
            assert np.max(np.abs(got[t] - want[t])) <= 1e-5 * np.max(np.abs(want[t]))


@pytest.mark.parametrize("nh,nkv", [(16, 4), (8, 4), (4, 4), (8, 1)])
@pytest.mark.parametrize("start,T", [(0, 1), (0, 17), (3, 130), (2500, 34), (2500, 131)])
def test_attn_prefill_all_out_of_range(nh, nkv, start, T):
    """Every query block in the fp32 form (a row 2^20 times the others in the
    first tile), in one chunk and shared out over several, for 1, 2 and 4 q
    heads a workgroup."""
    kw = {"vmul": [(1, 2.0 ** 20)]} if start else {"new_v": np.exp2(np.where(np.arange(256) % 2, 20, 0))}
    got, want = _attn_prefill_case(nh, nkv, start, T, **kw)
    e = np.max(np.abs(got - want)) / np.max(np.abs(want))
    say(f"attn_prefill fp32 form {nh}/{nkv} start {start} T {T}: {e:.2e}")
    assert e <= 1e-5


def _turns_context(cap):
    c = q35mix.Context(q35mix.qwen35_config(num_layers=1, num_heads=16, num_kv_heads=4, is_recurrent=[0]), n_seqs=1,
                       kv_capacity=cap)
    c.set_attn_weights(0, synth.attn_weights(256))
    k, v = synth.kv_prefill(cap, 1024, salt=77)
    c.state_write(0, 0, q35mix.STATE_KEYS, k)
    c.state_write(0, 0, q35mix.STATE_VALUES, v)
    c.truncate(0, 0)
    x = synth.attn_inputs(20, 16, 4, 256, salt=5)
    args = [c.array((20, 8192), x["q_gate"]), c.array((20, 1024), x["k"]), c.array((20, 1024), x["v"]), c.array((20, 4096))]
    return c, args


def test_attn_prefill_workspace_allocated_once():
    """The turns of a growing conversation need no more device memory than
    its first one: the workspace is one of the context's capacity."""
    hip = q35mix.hip()

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    c, args = _turns_context(6000)
    with c:
        c.attn_prefill(0, 0, 20, *args)
        c.sync()
        first = free()
        for start in (900, 3000, 5980):
            c.advance(0, start - c.kv_len(0))
            c.attn_prefill(0, 0, 20, *args)
            c.sync()
            assert free() == first


def test_attn_prefill_under_graph_capture():
    """A turn captured into a HIP graph behind more rows than the call that
    warmed the context up: three replays, with eager work between them, each
    equal bit for bit to the eager call."""
    hip = q35mix.hip()
    c, args = _turns_context(4100)
    with c:
        c.attn_prefill(0, 0, 20, *args)
        c.sync()
        c.advance(0, 4000)
        stream, graph, exe = ctypes.c_void_p(c.stream), ctypes.c_void_p(), ctypes.c_void_p()
        assert hip.hipStreamBeginCapture(stream, 0) == 0
        try:
            c.attn_prefill(0, 0, 20, *args)
        finally:
            r_end = hip.hipStreamEndCapture(stream, ctypes.byref(graph))
        assert r_end == 0
        assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
        try:
            for rep in range(3):
                args[3].upload(np.zeros((20, 4096), np.float32))
                assert hip.hipGraphLaunch(exe, stream) == 0
                c.sync()
                got = args[3].download()
                args[3].upload(np.zeros((20, 4096), np.float32))
                c.attn_prefill(0, 0, 20, *args)
                c.sync()
                assert np.array_equal(got.view(np.uint32), args[3].download().view(np.uint32))
                assert np.any(got)
        finally:
            assert hip.hipGraphExecDestroy(exe) == 0
            assert hip.hipGraphDestroy(graph) == 0


@pytest.mark.parametrize("nh,nkv,start,T", [(16, 4, 0, 1), (16, 4, 31, 33), (16, 4, 300, 65), (4, 4, 100, 129), (8, 4, 63, 65),
                                            (8, 1, 700, 40), (16, 2, 0, 34)])
def test_attn_prefill_fp32_kernels(monkeypatch, nh, nkv, start, T):
    """The kernels that take a call without room for the split form's
    workspace (here by a 1-byte limit on what a descriptor covers): output and
    new cache rows, 1, 2, 4 and 8 q heads a kv head."""
    monkeypatch.setenv("Q35M_TILE_LIMIT_BYTES", "1")
    dims = oracle.dims(n_heads=nh, n_kv_heads=nkv)
    x, wts, ck, cv = _attn_prefill_data(nh, nkv, start, T)
    with q35mix.Context(q35mix.qwen35_config(num_layers=1, num_heads=nh, num_kv_heads=nkv, is_recurrent=[0]), n_seqs=1,
                        kv_capacity=start + T) as c:
        c.set_attn_weights(0, wts)
        if start:
            c.state_write(0, 0, q35mix.STATE_KEYS, ck[:start])
            c.state_write(0, 0, q35mix.STATE_VALUES, cv[:start])
            if c.kv_len(0) < start:
                c.advance(0, start - c.kv_len(0))
        out = c.array((T, nh * 256))
        c.profile(True)
        c.attn_prefill(0, 0, T, c.array((T, 2 * nh * 256), x["q_gate"]), c.array((T, nkv * 256), x["k"]),
                       c.array((T, nkv * 256), x["v"]), out)
        ran = c.profile_read()
        c.profile(False)
        assert sorted(ran) == ["attn_prefill_flash", "attn_prefill_prep"]
        got = out.download()
        rows = [c.state_read(0, 0, kind, start + T)[start:] for kind in (q35mix.STATE_KEYS, q35mix.STATE_VALUES)]
    want, k_all, _ = oracle.attn_prefill(dims, start, T, x["q_gate"], x["k"], x["v"], wts, ck, cv, n_threads=8)
    e = np.max(np.abs(got - want)) / np.max(np.abs(want))
    say(f"attn_prefill fp32 kernels {nh}/{nkv} start {start} T {T}: {e:.2e}")
    assert e <= 1e-5
    k_new = k_all.reshape(start + T, -1)[start:]
    assert np.max(np.abs(rows[0].reshape(T, -1) - k_new)) <= 1e-5 * np.max(np.abs(k_new))
    assert np.array_equal(rows[1].reshape(T, -1), x["v"].reshape(T, -1))


def test_attn_prefill_long_prompt():
    """A prompt of more query blocks than the item list holds (the grid goes
    block by block): rows of its first, middle and last blocks against the
    oracle run from there over the cache's own earlier rows."""
    nh, nkv, T = 4, 1, 16500
    dims = oracle.dims(n_heads=nh, n_kv_heads=nkv)
    wts = synth.attn_weights(256)
    x = synth.attn_inputs(T, nh, nkv, 256, salt=91)
    with q35mix.Context(q35mix.qwen35_config(num_layers=1, num_heads=nh, num_kv_heads=nkv, is_recurrent=[0]), n_seqs=1,
                        kv_capacity=T) as c:
        c.set_attn_weights(0, wts)
        out = c.array((T, nh * 256))
        c.attn_prefill(0, 0, T, c.array((T, 2 * nh * 256), x["q_gate"]), c.array((T, nkv * 256), x["k"]),
                       c.array((T, nkv * 256), x["v"]), out)
        got = out.download()
        keys, values = (c.state_read(0, 0, kind, T).reshape(T, nkv * 256) for kind in (q35mix.STATE_KEYS, q35mix.STATE_VALUES))
    assert np.array_equal(values, x["v"].reshape(T, -1))
    for t0, n in ((0, 40), (8170, 40), (16384, 20), (T - 33, 33)):
        sl = slice(t0, t0 + n)
        want, k_all, _ = oracle.attn_prefill(dims, t0, n, x["q_gate"][sl], x["k"][sl], x["v"][sl], wts, keys[:t0 + n].copy(),
                                             values[:t0 + n].copy(), n_threads=8)
        e = np.max(np.abs(got[sl] - want)) / np.max(np.abs(want))
        say(f"attn_prefill rows {t0}..{t0 + n} of {T}: {e:.2e}")
        assert e <= 1e-5
        k_new = k_all.reshape(t0 + n, -1)[t0:]
        assert np.max(np.abs(keys[sl] - k_new)) <= 1e-5 * np.max(np.abs(k_new))
