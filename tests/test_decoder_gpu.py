"""The decode step (RMS norm, rotary, f16 KV cache, grouped-query attention, gated GELU, argmax around
the int4 GEMV) against the numpy oracle, step by step with teacher forcing.

Tolerance on the logits: |got - ref| <= 2e-3 + 2e-3 * |ref| -- f32 arithmetic through two layers in a
different summation order, with an f16 cache on both sides."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SMALL = dict(n_layers=2, hidden=128, ffn=256, n_q_heads=4, n_kv_heads=2, head_dim=64, vocab=512, block_size=32,
             rms_eps=1e-6, rope_theta=10000.0, attn_scale=0.0, embed_scale=float(np.sqrt(128.0)))


def test_decode_steps_match_the_oracle(ctx, pkg, oracle):
    from oracle import decoder as od
    steps, max_seq = 70, 80          # crosses several 16-position chunks of the attention kernel
    w = pkg.decoder.build_weights(SMALL, seed=3)
    dec = pkg.decoder.Decoder(ctx, SMALL, max_seq)
    dec.load(w)
    ref = od.Decoder(w, max_seq)
    token = 17
    dec.reset(token, 0)
    agree = 0
    for pos in range(steps):
        dec.step()
        got_tok, got_pos, logits, _ = dec.read(want_logits=True)
        want_logits, want_tok = ref.step(token, pos)
        assert got_pos == pos + 1
        err = np.abs(logits - want_logits)
        assert np.all(err <= 2e-3 + 2e-3 * np.abs(want_logits)), (pos, float(err.max()))
        top2 = np.sort(want_logits)[-2:]
        if top2[1] - top2[0] > 1e-2:
            assert got_tok == want_tok, pos
            agree += 1
        token = got_tok              # teacher forcing: the oracle consumes what the device chose
    assert agree > steps // 2
    _, _, _, hist = dec.read(n_history=steps)
    assert hist[-1] == token
    dec.destroy()


@pytest.mark.parametrize("env", [{}, {"HIPC_DEC_FUSED_ARGMAX": 0}, {"HIPC_DEC_FUSED_GLUE": 0}], ids=["candidates-from-lm_head", "separate-scan", "separate-glue"])
def test_the_token_is_the_argmax_of_the_logits_on_a_wide_vocabulary(ctx, pkg, route, env):
    """A vocabulary wide enough for the unembedding to run on the kernel whose workgroups leave the argmax candidates
    themselves (ragged: 32768 + 48 columns): the token the device picks is the first largest of the logits it stores,
    step after step, and the same with a launch of its own scanning the logits."""
    route(env)
    cfg = dict(SMALL, vocab=32768 + 48)
    w = pkg.decoder.build_weights(cfg, seed=21)
    dec = pkg.decoder.Decoder(ctx, cfg, 24)
    dec.load(w)
    dec.reset(5, 0)
    seen = set()
    for pos in range(12):
        dec.step()
        tok, got_pos, logits, _ = dec.read(want_logits=True)
        assert got_pos == pos + 1 and tok == int(np.argmax(logits)), (pos, tok, int(np.argmax(logits)))
        seen.add(tok)
    assert len(seen) > 1
    dec.destroy()


DEEP = [  # (head_dim, query heads, kv heads, first position): every head_dim / group size the chunk kernel is built for
    (256, 4, 1, 2046),   # crosses from 64 to 128 positions per workgroup at 2048
    (128, 8, 1, 4290),   # three passes per workgroup, the last one ragged
    (64, 2, 2, 2300),    # one query head per kv head
    (128, 4, 2, 130),    # three live chunks only
    (192, 2, 1, 100),    # no instance for this head_dim: the three-kernel path
]
# The read-ahead route (helper workgroups of a launch that warm the L2 for the next launch): one bit per producer
# launch of a layer. By default three of the five producers carry helpers; the other cases run all five and none.
READ_AHEAD = {"HIPC_DEC_PREFETCH": 31}
NO_READ_AHEAD = {"HIPC_DEC_PREFETCH": 0}
PER_PRODUCT = {"HIPC_DEC_RESIDENT": 0}   # the launches per product with their default read-ahead, which longer contexts and other shapes take
PATHS = [{}, PER_PRODUCT, READ_AHEAD, {"HIPC_DEC_LEAN": 0}, {"HIPC_DEC_FUSED_GLUE": 0}, {"HIPC_DEC_FUSED_ATTN": 0}]


@pytest.fixture
def route(ctx):
    """Sets route options on the shared context for one test and restores the defaults afterwards."""
    touched = []

    def apply(options):
        for k, v in options.items():
            ctx.set_option(k, v)
            touched.append(k)
    yield apply
    for k in touched:
        ctx.set_option(k, -1)


@pytest.mark.parametrize("env", PATHS, ids=["default", "per-product", "read-ahead", "streaming-gemv", "separate-glue", "three-kernel-attention"])
@pytest.mark.parametrize("hd,nq,nkv,p0", DEEP)
def test_attention_over_a_long_filled_cache(ctx, pkg, oracle, route, hd, nq, nkv, p0, env):
    """Steps taken deep into a context whose cache rows hold random f16 values on both sides: the
    chunked attention (several passes per workgroup, the join in the output projection's prologue
    or in the merge kernel) against the oracle's softmax over the whole context."""
    from oracle import decoder as od
    route(env)                     # read when the decoder is created
    cfg = dict(SMALL, n_q_heads=nq, n_kv_heads=nkv, head_dim=hd)
    steps, max_seq = 3, p0 + 8
    w = pkg.decoder.build_weights(cfg, seed=11)
    dec = pkg.decoder.Decoder(ctx, cfg, max_seq)
    dec.load(w)
    ref = od.Decoder(w, max_seq)
    rng = np.random.default_rng(hd + p0)
    for li in range(cfg["n_layers"]):
        k_rows, v_rows = ((rng.standard_normal((nkv, max_seq, hd)) * 0.7).astype(np.float16) for _ in range(2))
        ref.k[li], ref.v[li] = k_rows, v_rows
        dec.fill_cache(li, k_rows, v_rows)
    token = 23
    dec.reset(token, p0)
    for pos in range(p0, p0 + steps):
        dec.step()
        got_tok, got_pos, logits, _ = dec.read(want_logits=True)
        want_logits, _ = ref.step(token, pos)
        assert got_pos == pos + 1
        err = np.abs(logits - want_logits)
        assert np.all(err <= 2e-3 + 2e-3 * np.abs(want_logits)), (pos, float(err.max()))
        k_row = ctx.download(dec.kv_cache(1)[0], np.float16, (hd,), offset=((nkv - 1) * max_seq + pos) * hd * 2)
        assert np.allclose(k_row.astype(np.float32), ref.k[1, nkv - 1, pos].astype(np.float32), atol=2e-3, rtol=2e-3), pos
        stride = (max_seq + 63) // 64 * 64       # values are kept transposed: [kv head, channel, position]
        v_t = ctx.download(dec.kv_cache(1)[1], np.float16, (nkv, hd, stride))
        assert np.allclose(v_t[nkv - 1, :, pos].astype(np.float32), ref.v[1, nkv - 1, pos].astype(np.float32), atol=2e-3, rtol=2e-3), pos
        token = got_tok
    dec.destroy()


@pytest.mark.parametrize("nq,max_seq", [(8, 16384), (8, 16385), (4, 32768), (4, 32769)])
def test_the_longest_context_that_keeps_all_layers_in_one_launch(ctx, pkg, route, nq, max_seq):
    """All layers in one launch over the longest contexts, at the last position, against the launches per product over the
    same cache. (Which of the two forms a decoder takes by itself: tests/host/decoder_model.cpp.)"""
    cfg = dict(SMALL, n_q_heads=nq, n_kv_heads=1, head_dim=64)
    w = pkg.decoder.build_weights(cfg, seed=14)
    rng = np.random.default_rng(nq)
    rows = [tuple((rng.standard_normal((1, max_seq, 64)) * 0.7).astype(np.float16) for _ in range(2)) for _ in range(cfg["n_layers"])]
    got = []
    for resident in (256, 0):
        route({"HIPC_DEC_RESIDENT": resident})
        dec = pkg.decoder.Decoder(ctx, cfg, max_seq)
        dec.load(w)
        for li, (k_rows, v_rows) in enumerate(rows):
            dec.fill_cache(li, k_rows, v_rows)
        dec.reset(29, max_seq - 1)
        dec.step()
        got.append(dec.read(want_logits=True))
        dec.destroy()
    assert got[0][1] == got[1][1] == max_seq
    assert np.all(np.abs(got[0][2] - got[1][2]) <= 2e-3 + 2e-3 * np.abs(got[1][2])), float(np.abs(got[0][2] - got[1][2]).max())


WINDOWS = [  # (head_dim, query heads, kv heads, first position, window of layer 0, window of layer 1)
    (256, 4, 1, 2300, 512, 0),     # gemma3's local window beside a global layer
    (128, 4, 2, 509, 512, 100),    # the window starts to mask at 512 positions, i.e. during these steps
    (64, 2, 2, 4400, 4200, 70),    # a window longer than one pass of all chunks; one shorter than a chunk
    (192, 2, 1, 100, 40, 16),      # the three-kernel path: whole 16-position chunks fall out of the window
]


@pytest.mark.parametrize("env", PATHS, ids=["default", "per-product", "read-ahead", "streaming-gemv", "separate-glue", "three-kernel-attention"])
@pytest.mark.parametrize("hd,nq,nkv,p0,w0,w1", WINDOWS)
def test_sliding_windows_and_a_second_rotary_base(ctx, pkg, oracle, route, hd, nq, nkv, p0, w0, w1, env):
    """Local layers: the last `window` positions only, the step's own included (the reference's
    bound, shaders/attention.rs:202-214), rotating with their own base; against the oracle over a
    filled cache, across the step at which the window starts to cut."""
    from oracle import decoder as od
    route(env)
    cfg = dict(SMALL, n_q_heads=nq, n_kv_heads=nkv, head_dim=hd, rope_theta=1.0e6)
    steps, max_seq = 5, p0 + 8
    w = pkg.decoder.build_weights(cfg, seed=12)
    dec = pkg.decoder.Decoder(ctx, cfg, max_seq)
    dec.load(w)
    ref = od.Decoder(w, max_seq)
    for li, win in enumerate((w0, w1)):
        theta = 10000.0 if win else 0.0          # local layers use the second base
        dec.set_layer_attention(li, win, theta)
        ref.set_layer_attention(li, win, theta)
    rng = np.random.default_rng(hd + p0)
    for li in range(cfg["n_layers"]):
        k_rows, v_rows = ((rng.standard_normal((nkv, max_seq, hd)) * 0.7).astype(np.float16) for _ in range(2))
        ref.k[li], ref.v[li] = k_rows, v_rows
        dec.fill_cache(li, k_rows, v_rows)
    token = 31
    dec.reset(token, p0)
    for pos in range(p0, p0 + steps):
        dec.step()
        got_tok, got_pos, logits, _ = dec.read(want_logits=True)
        want_logits, _ = ref.step(token, pos)
        assert got_pos == pos + 1
        err = np.abs(logits - want_logits)
        assert np.all(err <= 2e-3 + 2e-3 * np.abs(want_logits)), (pos, float(err.max()))
        token = got_tok
    dec.destroy()


def test_a_third_rotary_base_is_refused(ctx, pkg):
    dec = pkg.decoder.Decoder(ctx, SMALL, 16)
    dec.set_layer_attention(0, 8, 500.0)
    dec.set_layer_attention(1, 0, 500.0)
    with pytest.raises(pkg.HipComputeError) as e:
        dec.set_layer_attention(1, 0, 700.0)
    assert "third rotary base" in e.value.message
    with pytest.raises(pkg.HipComputeError):
        dec.set_layer_attention(2, 0, 0.0)
    dec.destroy()


def test_a_captured_step_replays_without_patching(ctx, pkg):
    """Position and token live on the device: replaying one captured step N times must give the
    same tokens as N eager steps."""
    w = pkg.decoder.build_weights(SMALL, seed=4)
    runs = []
    for use_graph in (False, True):
        dec = pkg.decoder.Decoder(ctx, SMALL, 40)
        dec.load(w)
        dec.reset(5, 0)
        dec.step()                    # eager warm-up step (also sizes scratch)
        if use_graph:
            ctx.flush()
            ctx.capture_begin()
            dec.step()
            g = ctx.capture_end()     # recording does not execute: position is still 1
            for _ in range(20):
                ctx.graph_launch(g)
            tok, pos, _, hist = dec.read(n_history=21)
            ctx.graph_destroy(g)
        else:
            for _ in range(20):
                dec.step()
            tok, pos, _, hist = dec.read(n_history=21)
        assert pos == 21
        runs.append(hist.copy())
        dec.destroy()
    assert np.array_equal(runs[0], runs[1])


def test_the_embedded_row_follows_the_weights_it_is_made_of(ctx, pkg, oracle):
    """Every step leaves the embedded row of the token it picked for the next one. When the embedding table or the
    first layer's input norm is replaced between steps, the next step must embed again -- with the new weights -- and
    a decoder that was never reset steps from token 0 at position 0."""
    from oracle import decoder as od
    w = pkg.decoder.build_weights(SMALL, seed=6)
    w2 = pkg.decoder.build_weights(SMALL, seed=7)
    for env in ({}, {"HIPC_DEC_LEAN": 0}):
        with ctx.options(**env):
            dec = pkg.decoder.Decoder(ctx, SMALL, 24)
            dec.load(w)
            ref = od.Decoder(w, 24)
            token = 0                       # no reset: the state a new decoder starts from
            for pos in range(8):
                if pos == 3:                # a new embedding table and input norm, the other weights stay
                    w.embedding = w2.embedding
                    w.norms[(0, pkg.decoder.NORM_INPUT)] = w2.norms[(0, pkg.decoder.NORM_INPUT)]
                    B, scales, zp = w.embedding
                    dB, dS, dZ = ctx.upload(B), ctx.upload(scales), ctx.upload(zp)
                    ctx._check(ctx.lib.hipc_decoder_set_embedding(ctx.handle, dec.handle, dB.ptr, B.size, dS.ptr, scales.size, dZ.ptr, zp.size))
                    dV = ctx.upload(w.norms[(0, pkg.decoder.NORM_INPUT)])
                    ctx._check(ctx.lib.hipc_decoder_set_norm(ctx.handle, dec.handle, 0, pkg.decoder.NORM_INPUT, dV.ptr))
                    ctx.flush()
                    for buf in (dB, dS, dZ, dV):
                        buf.free()
                dec.step()
                got_tok, got_pos, logits, _ = dec.read(want_logits=True)
                want_logits, want_tok = ref.step(token, pos)
                assert got_pos == pos + 1
                err = np.abs(logits - want_logits)
                assert np.all(err <= 2e-3 + 2e-3 * np.abs(want_logits)), (env, pos, float(err.max()))
                token = got_tok
            dec.destroy()
        w = pkg.decoder.build_weights(SMALL, seed=6)   # the first route's replacements do not carry over


def test_refuses_incomplete_models_and_bad_shapes(ctx, pkg):
    dec = pkg.decoder.Decoder(ctx, SMALL, 16)
    with pytest.raises(pkg.HipComputeError) as e:
        dec.step()
    assert e.value.code == 1 and "not every weight" in e.value.message
    dec.destroy()
    with pytest.raises(pkg.HipComputeError):
        pkg.decoder.Decoder(ctx, dict(SMALL, head_dim=48), 16)


def test_the_cache_limit_is_kept_on_the_device(ctx, pkg, oracle):
    """max_seq steps fit after a reset to 0; one more (eager or replayed) writes nothing, leaves token
    and position alone and is reported by the next read -- the rule of oracle.decoder.advance_state."""
    from oracle.decoder import advance_state
    max_seq = 6
    w = pkg.decoder.build_weights(SMALL, seed=5)
    dec = pkg.decoder.Decoder(ctx, SMALL, max_seq)
    dec.load(w)
    dec.reset(3, 0)
    tok, pos, over = 3, 0, False
    for _ in range(max_seq):
        dec.step()
        got_tok, got_pos, logits, _ = dec.read(want_logits=True)
        tok, pos, over = advance_state(tok, pos, logits, max_seq)
        assert (got_tok, got_pos) == (tok, pos) and not over
    assert pos == max_seq
    k_before = ctx.download(dec.kv_cache(0)[0], np.float16, (SMALL["n_kv_heads"] * max_seq * SMALL["head_dim"],))
    dec.step()                                           # one step too many
    with pytest.raises(pkg.HipComputeError) as e:
        dec.read()
    assert e.value.code == 1 and "cache full" in e.value.message
    tok2, pos2 = ctypes_state(ctx, dec)
    assert (tok2, pos2) == advance_state(tok, pos, None, max_seq)[:2] == (tok, max_seq)
    assert np.array_equal(ctx.download(dec.kv_cache(0)[0], np.float16, k_before.shape), k_before)
    dec.reset(3, 0)                                      # a reset clears the flag
    dec.step()
    assert dec.read()[1] == 1
    dec.destroy()


def ctypes_state(ctx, dec):
    """token and position as hipc_decoder_read fills them, whatever status it returns"""
    import ctypes as C
    tok, pos = C.c_int32(), C.c_int32()
    ctx.lib.hipc_decoder_read(ctx.handle, dec.handle, C.byref(tok), C.byref(pos), None, None, 0)
    return tok.value, pos.value


@pytest.mark.parametrize("env", [{}, READ_AHEAD, NO_READ_AHEAD], ids=["default", "read-ahead-everywhere", "no-read-ahead"])
def test_gemma3_1b_shape_at_context_2040(ctx, pkg, oracle, route, env):
    """The decoder configuration at its real size -- 26 layers, hidden 1152, ffn 6912, 4 query heads on
    1 kv head of 256, vocabulary 262144, 22 local layers (window 512, base 10000) and 4 global ones
    (base 1e6) -- three steps from position 2040 over a cache filled with random f16 rows on both
    sides, logits against the oracle at 2e-3 + 2e-3 |ref|. These are the code paths the tokens-per-
    second figure runs: the one-item-per-thread norm prologue, the gated-GELU prologue of a
    k-split down projection, the attention join of 64 chunks."""
    from oracle import decoder as od
    route(env)
    D = pkg.decoder
    cfg = dict(D.GEMMA3_1B)
    p0, steps = 2040, 3
    max_seq = p0 + steps + 5
    w = D.build_weights(cfg, seed=9)
    dec = D.Decoder(ctx, cfg, max_seq)
    dec.load(w)
    ref = od.Decoder(w, max_seq)
    for li in range(cfg["n_layers"]):
        if (li + 1) % 6 != 0:
            dec.set_layer_attention(li, 512, 10000.0), ref.set_layer_attention(li, 512, 10000.0)
        else:
            dec.set_layer_attention(li, 0, 1.0e6), ref.set_layer_attention(li, 0, 1.0e6)
    rng = np.random.default_rng(2040)
    for li in range(cfg["n_layers"]):
        k_rows, v_rows = ((rng.standard_normal((1, max_seq, 256)) * 0.5).astype(np.float16) for _ in range(2))
        ref.k[li], ref.v[li] = k_rows, v_rows
        dec.fill_cache(li, k_rows, v_rows)
    token = 1234
    dec.reset(token, p0)
    for pos in range(p0, p0 + steps):
        dec.step()
        got_tok, got_pos, logits, _ = dec.read(want_logits=True)
        want_logits, want_tok = ref.step(token, pos)
        assert got_pos == pos + 1
        err = np.abs(logits - want_logits)
        assert np.all(err <= 2e-3 + 2e-3 * np.abs(want_logits)), (pos, float(err.max()))
        top2 = np.sort(want_logits)[-2:]
        if top2[1] - top2[0] > 1e-2:
            assert got_tok == want_tok, pos
        token = got_tok
    dec.destroy()
    ctx.flush()


RESIDENT = [  # (hidden, ffn, head_dim, query heads, kv heads, block_size): the launch that holds all layers, where its shares run out unevenly
    (128, 256, 64, 4, 2, 32),     # eight column tiles and two k tiles for 256 workgroups; a head is half a k tile of o
    (1296, 1552, 256, 2, 1, 32),  # 81 column tiles (three for some ranks), ffn's last k tile one pair wide, more units than are asked for ahead
    (448, 1088, 128, 8, 2, 64),   # one XCD per head; 3 1/2 k tiles of hidden
    (2048, 4224, 64, 1, 1, 128),  # the longest row; eight XCDs to a head; uneven slices of ffn
]


def three_layers(pkg, ctx, hidden, ffn, hd, nq, nkv, bs):
    """A decoder and the oracle's over the same filled cache of 80 positions, a window of 40 in the second layer."""
    from oracle import decoder as od
    cfg = dict(SMALL, n_layers=3, hidden=hidden, ffn=ffn, n_q_heads=nq, n_kv_heads=nkv, head_dim=hd, block_size=bs, vocab=512, embed_scale=float(np.sqrt(hidden)))
    max_seq = 80
    w = pkg.decoder.build_weights(cfg, seed=31)
    dec = pkg.decoder.Decoder(ctx, cfg, max_seq)
    dec.load(w)
    ref = od.Decoder(w, max_seq)
    dec.set_layer_attention(1, 40, 500.0), ref.set_layer_attention(1, 40, 500.0)
    rng = np.random.default_rng(hidden)
    for li in range(cfg["n_layers"]):
        k_rows, v_rows = ((rng.standard_normal((nkv, max_seq, hd)) * 0.7).astype(np.float16) for _ in range(2))
        ref.k[li], ref.v[li] = k_rows, v_rows
        dec.fill_cache(li, k_rows, v_rows)
    return dec, ref


def steps_match(ctx, dec, ref, p0=69):
    """Four steps from position 69 (the third pass of 32 begins): logits, cache rows and tokens. The tolerance is this file's."""
    token, nkv, hd = 23, dec.cfg["n_kv_heads"], dec.cfg["head_dim"]
    dec.reset(token, p0)
    for pos in range(p0, p0 + 4):
        dec.step()
        got_tok, got_pos, logits, _ = dec.read(want_logits=True)
        want_logits, _ = ref.step(token, pos)
        assert got_pos == pos + 1
        err = np.abs(logits - want_logits)
        assert np.all(err <= 2e-3 + 2e-3 * np.abs(want_logits)), (pos, float(err.max()))
        for li in range(dec.cfg["n_layers"]):
            k_row = ctx.download(dec.kv_cache(li)[0], np.float16, (hd,), offset=((nkv - 1) * dec.max_seq + pos) * hd * 2)
            assert np.allclose(k_row.astype(np.float32), ref.k[li, nkv - 1, pos].astype(np.float32), atol=2e-3, rtol=2e-3), (pos, li)
        token = got_tok


@pytest.mark.parametrize("groups", [-1, 255, 100, 3], ids=["all", "255", "100", "3"])
@pytest.mark.parametrize("hidden,ffn,hd,nq,nkv,bs", RESIDENT)
def test_all_layers_in_one_launch(ctx, pkg, oracle, route, hidden, ffn, hd, nq, nkv, bs, groups):
    """Three layers by a launch of 256 workgroups, and by launches of fewer, whose workgroups take several shares each."""
    route({"HIPC_DEC_RESIDENT": groups})
    dec, ref = three_layers(pkg, ctx, hidden, ffn, hd, nq, nkv, bs)
    steps_match(ctx, dec, ref)
    dec.destroy()


LDS_LIMITS = [  # the weights of a share in LDS: every place taken; two tiles of q|k|v a workgroup among gate|up's places; one place in four
    (2048, 8192, 256, 8, 1, 32),
    (512, 1040, 256, 8, 8, 32),
    (144, 128, 64, 2, 1, 128),
]


@pytest.mark.parametrize("hidden,ffn,hd,nq,nkv,bs", LDS_LIMITS)
def test_weights_of_the_one_launch_in_lds(ctx, pkg, oracle, hidden, ffn, hd, nq, nkv, bs):
    dec, ref = three_layers(pkg, ctx, hidden, ffn, hd, nq, nkv, bs)
    steps_match(ctx, dec, ref)
    dec.destroy()


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_a_row_that_is_not_finite(ctx, pkg, oracle, value):
    """One channel of a norm's weight: the row it goes into the products with has no digits there, and every result is NaN."""
    dec, ref = three_layers(pkg, ctx, 448, 1088, 128, 8, 2, 64)
    w = ref.w.norms[(1, pkg.decoder.NORM_PRE_FFN)].copy()
    w[77] = value
    ref.w.norms[(1, pkg.decoder.NORM_PRE_FFN)] = w
    dec.load(ref.w)
    dec.reset(23, 69)
    dec.step()
    token, _, logits, _ = dec.read(want_logits=True)
    assert np.all(np.isnan(logits)) and token == 0
    dec.destroy()


@pytest.mark.parametrize("env", [{"HIPC_DEC_WAIT": 0}, {"HIPC_DEC_WAIT": 100}, {"HIPC_DEC_WIDE": 1}, {"HIPC_DEC_RESIDENT": 40, "HIPC_DEC_WAIT": 0}],
                         ids=["does-not-begin", "waits-a-microsecond", "no-shared-l2", "those-there-at-once"])
@pytest.mark.parametrize("hidden,ffn,hd,nq,nkv,bs", RESIDENT)
def test_the_ways_out_of_the_one_launch(ctx, pkg, oracle, route, hidden, ffn, hd, nq, nkv, bs, env):
    """The launch of 256 workgroups does not begin and the one behind it goes on with the workgroups it has by then, however
    few; the same where some may come in time; and hand-overs that leave the L2 everywhere."""
    route(env)
    dec, ref = three_layers(pkg, ctx, hidden, ffn, hd, nq, nkv, bs)
    steps_match(ctx, dec, ref)
    dec.destroy()


@pytest.mark.parametrize("polls", [1, 4, 10])
@pytest.mark.parametrize("hidden,ffn,hd,nq,nkv,bs", RESIDENT)
def test_a_step_that_was_given_up(ctx, pkg, oracle, route, hidden, ffn, hd, nq, nkv, bs, polls):
    """Steps whose threads run out of polls, with the launch just begun or within it, end, and the read reports them. A reset
    to where they began makes the decoder as good as new, whatever they left in the cache and in the words workgroups exchange."""
    dec, ref = three_layers(pkg, ctx, hidden, ffn, hd, nq, nkv, bs)
    steps_match(ctx, dec, ref)
    for _ in range(2):
        route({"HIPC_DEC_POLLS": polls})
        dec.reset(23, 69)
        dec.step(), dec.step(), dec.step()
        with pytest.raises(pkg.HipComputeError, match="did not come to its end"):
            dec.read()
        route({"HIPC_DEC_POLLS": -1})
        steps_match(ctx, dec, ref)
    dec.destroy()


def test_decoders_on_several_streams_at_once(pkg):
    """Three contexts (a stream each) replay their recorded steps from three threads: launches that do not find room for
    all their workgroups beside each other go on with those that do, and every decoder picks the tokens it picks alone."""
    import threading
    cfg = dict(SMALL, hidden=512, ffn=2048, head_dim=128, n_layers=4, embed_scale=float(np.sqrt(512.0)))
    w = pkg.decoder.build_weights(cfg, seed=8)
    steps = 40

    def run(n_threads):
        ctxs = [pkg.Context(0) for _ in range(n_threads)]
        decs, graphs, hists = [], [], [None] * n_threads
        for c in ctxs:
            d = pkg.decoder.Decoder(c, cfg, steps + 8)
            d.load(w)
            d.reset(7, 0)
            d.step()
            c.flush()
            c.capture_begin()
            d.step()
            graphs.append(c.capture_end())
            decs.append(d)

        def go(i):
            decs[i].reset(7, 0)
            for _ in range(steps):
                ctxs[i].graph_launch(graphs[i])
            hists[i] = decs[i].read(n_history=steps)[3].copy()
        threads = [threading.Thread(target=go, args=(i,)) for i in range(n_threads)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for c, d, g in zip(ctxs, decs, graphs):
            c.graph_destroy(g)
            d.destroy()
            c.close()
        return hists
    alone = run(1)[0]
    for h in run(3):
        assert h is not None and np.array_equal(h, alone)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_products_of_a_row_that_is_not_finite(ctx, pkg, value):
    """Such a row makes all of its products NaN, not infinities of any sign: seen in the value row that q|k|v leaves in the cache."""
    dec, ref = three_layers(pkg, ctx, 448, 1088, 128, 8, 2, 64)
    w = ref.w.norms[(1, pkg.decoder.NORM_INPUT)].copy()
    w[77] = value
    ref.w.norms[(1, pkg.decoder.NORM_INPUT)] = w
    dec.load(ref.w)
    dec.reset(23, 69)
    dec.step()
    v_t = ctx.download(dec.kv_cache(1)[1], np.float16, (2, 128, 128))       # [kv head, channel, position]
    assert np.all(np.isnan(v_t[:, :, 69]))
    dec.destroy()


OUTLIERS = ["qkv", "o", "gate_up", "down"]


def beside_an_outlier(pkg, ctx, which, binades=16):
    """A decoder of two layers, one product of whose second has in every row a value of some 2^binades times the others', for
    which its weights are zero (codes equal to their zero points): the float64 result is that of the others. The reset is
    at position 69 behind a filled cache. Returns the decoder and the float64 logits of the step there."""
    from test_oracle_pins import _step_f64
    D = pkg.decoder
    cfg = dict(SMALL, hidden=448, ffn=1088, n_q_heads=8, n_kv_heads=2, head_dim=128, embed_scale=float(np.sqrt(448.0)))
    w, max_seq, at, rng = D.build_weights(cfg, seed=41), 80, 77, np.random.default_rng(42)
    caches = [tuple((rng.standard_normal((2, max_seq, 128)) * 0.7).astype(np.float16) for _ in range(2)) for _ in range(2)]

    def silence(linear, k):
        B, scales, zp = w.linears[(1, linear)]
        bs, B = cfg["block_size"], B.copy()
        z = (zp[:, k // bs // 2] >> (4 * (k // bs & 1))) & 15
        byte = B[:, k // bs, k % bs // 2]
        B[:, k // bs, k % bs // 2] = (byte & 0x0F) | (z << 4) if k & 1 else (byte & 0xF0) | z
        w.linears[(1, linear)] = (B, scales, zp)

    large = np.float32(2.0 ** binades)
    if which in ("qkv", "gate_up"):
        norm = (1, D.NORM_INPUT if which == "qkv" else D.NORM_PRE_FFN)
        w.norms[norm] = w.norms[norm].copy()
        w.norms[norm][at] *= large
        silence(D.QKV if which == "qkv" else D.GATE_UP, at)
    elif which == "o":       # a channel of the value cache: for all heads that share it
        caches[1][1][0, :69, at] *= np.float16(min(large, 2.0 ** 14))
        for h in range(4):
            silence(D.O, h * 128 + at)
    else:                    # a column of up; where the gate closes it, the next ones
        B, scales, zp = w.linears[(1, D.GATE_UP)]
        nb, scales = B.shape[1], scales.copy()
        for c in range(at, at + 512, 32):
            scales.reshape(-1, nb)[cfg["ffn"] + c] *= large
            silence(D.DOWN, c)
        w.linears[(1, D.GATE_UP)] = (B, scales, zp)
    dec = D.Decoder(ctx, cfg, max_seq)
    dec.load(w)
    for li in range(2):
        dec.fill_cache(li, *caches[li])
    dec.reset(23, 69)
    return dec, _step_f64(w, [(k.copy(), v.copy()) for k, v in caches], 23, 69, [0, 0], [cfg["rope_theta"]] * 2)


@pytest.mark.parametrize("groups", [-1, 100], ids=["all", "100"])
@pytest.mark.parametrize("which", OUTLIERS)
def test_small_values_beside_a_large_one(ctx, pkg, route, which, groups):
    """What the four bytes of a value keep beside a largest of 2^16 to 2^17: steps of 2^-13, 3.5e-5 of a value near 1 by root mean square,
    in one chunk of the row's 14 or more: 1e-5 of the products at most. The unembedding's bf16 terms and the f32 sums
    are 3e-6, f16 rounding of the step's key and value less. Without the lowest byte: 3e-5 and more."""
    route({"HIPC_DEC_RESIDENT": groups})
    dec, want = beside_an_outlier(pkg, ctx, which)
    dec.step()
    _, _, logits, _ = dec.read(want_logits=True)
    assert np.linalg.norm(logits - want) <= 1.2e-5 * np.linalg.norm(want)
    dec.destroy()
