"""Parity of the decode loop (include/lpp.h section B: forward / generate, the
counterpart of the reference's src/model.cpp:342-371 and src/main.cpp:158-223)
against the CPU oracle on identical seeded weights, for every scheduling path
of the library, on a real MI355X.

Bars (from the task statement):
  * logits: max |gpu - cpu| / max |cpu| <= 2e-3 per step (fp32 accumulation);
  * greedy token sequences agree on >= 99 % of steps;
  * a sampled token may differ only where the uniform draw sits closer than the
    logits tolerance to a bucket edge of the CPU CDF;
  * KV-cache scatter: slot index logic and binary16 rounding bit-exact.
The oracle rounds K/V through binary16 on store (kv_round_f16), which is what the
GPU operator API does by contract (kernels.cuh:34); a second check bounds the
distance to the pure-fp32-cache CPU path as well.
"""
import numpy as np
import pytest

import oracle_binding as ob
from lighterpp_amd import CONFIGS, Model, Shape, capi

pytestmark = pytest.mark.gpu
F = np.float32
LOGIT_TOL = 2e-3

PATHS = [capi.PATH_OPS, capi.PATH_FUSED, capi.PATH_PERSISTENT]
PATH_IDS = ["ops", "fused", "persistent"]

SMALL_SHAPES = {
    # name: Shape
    "mha_fp32_c1like": Shape(288, 768, 3, 6, 6, 1000, 64, 10000.0, fp16=False, tied=True),
    "gqa4_fp16": Shape(256, 512, 3, 8, 2, 2048, 160, 500000.0, fp16=True, tied=True),
    "gqa8_fp16_untied": Shape(512, 1408, 2, 8, 1, 1500, 96, 10000.0, fp16=True, tied=False),
    "hs128_fp16": Shape(512, 1024, 2, 4, 2, 777, 48, 500000.0, fp16=True, tied=False),
    # rows wider than one 4-KiB weight step: the persistent kernel cuts them into column slices
    # (dim 2560 -> 2 slices of 1280, hidden 7168 -> 4 of 1792) and adds per-slice partial sums
    "sliced_fp16": Shape(2560, 7168, 1, 20, 4, 640, 24, 500000.0, fp16=True, tied=False),
    # fp32 rows: dim 1536 -> 2 slices of 768; hidden 2304 -> width 768, 3 slices used of 4 (one idle)
    "sliced_fp32_idle_slice": Shape(1536, 2304, 2, 12, 4, 500, 24, 10000.0, fp16=False, tied=True),
}


def build(shape: Shape, seed: int, kv_round=True):
    m = Model(shape)
    w = m.load_synthetic(seed, keep=True)
    o = ob.OracleModel(shape, w, fp16=shape.fp16, kv_round_f16=kv_round)
    return m, o


def rel_err(got, want):
    return float(np.max(np.abs(got.astype(np.float64) - want)) / np.max(np.abs(want)))


@pytest.mark.parametrize("path", PATHS, ids=PATH_IDS)
@pytest.mark.parametrize("name", list(SMALL_SHAPES))
def test_greedy_decode_matches_oracle(name, path):
    shape = SMALL_SHAPES[name]
    m, o = build(shape, 21)
    m.set_path(path)
    prompt = capi.synth_token_ids(8, 5, shape.vocab_size)
    steps = min(48, shape.seq_len)
    tok_g = tok_c = int(prompt[0])
    agree, worst = 0, 0.0
    for pos in range(steps):
        # teacher-force the oracle's token into both, so one early flip cannot cascade
        nxt_g = m.forward(tok_c, pos, 0.0)
        want = o.forward_logits(tok_c, pos)
        got = m.buffer(capi.B_LOGITS)
        worst = max(worst, rel_err(got, want))
        nxt_c = int(np.argmax(want))
        agree += int(nxt_g == nxt_c)
        tok_c = int(prompt[pos + 1]) if pos + 1 < len(prompt) else nxt_c
    assert worst <= LOGIT_TOL, f"max relative logit error {worst}"
    assert agree >= int(np.ceil(0.99 * steps)), f"greedy agreement {agree}/{steps}"
    # cache contents: same slots, same binary16 values up to the rounding of a k that differs in the last bits
    kc = m.buffer(capi.B_KEY_CACHE).view(np.float16).astype(F)
    vc = m.buffer(capi.B_VALUE_CACHE).view(np.float16).astype(F)
    assert np.allclose(kc, o.buf("key_cache"), rtol=2e-3, atol=2e-3 * np.abs(o.buf("key_cache")).max())
    assert np.allclose(vc, o.buf("value_cache"), rtol=2e-3, atol=2e-3 * np.abs(o.buf("value_cache")).max())
    hs, nkv = shape.head_size, shape.n_kv_heads
    kc4 = kc.reshape(shape.n_layers, nkv, shape.seq_len, hs)
    assert np.all(kc4[:, :, steps:, :] == 0), "slots beyond the decoded positions were written"
    m.close()
    o.close()


@pytest.mark.parametrize("path", PATHS, ids=PATH_IDS)
def test_kv_scatter_index_and_rounding_bit_exact(path):
    """After a step at position p the cache slice [layer][h][p][:] of the LAST layer
    must hold exactly RN16 of that layer's k / v vectors (model.cpp:171-176), which
    the run state still contains."""
    shape = SMALL_SHAPES["gqa4_fp16"]
    m = Model(shape)
    m.load_synthetic(33)
    m.set_path(path)
    hs, nkv, L = shape.head_size, shape.n_kv_heads, shape.n_layers
    tok = 3
    for pos in [0, 1, 2, 77]:
        tok = m.forward(tok, pos, 0.0)
        k = m.buffer(capi.B_K).reshape(nkv, hs)
        v = m.buffer(capi.B_V).reshape(nkv, hs)
        kc = m.buffer(capi.B_KEY_CACHE).reshape(L, nkv, shape.seq_len, hs)
        vc = m.buffer(capi.B_VALUE_CACHE).reshape(L, nkv, shape.seq_len, hs)
        assert np.array_equal(kc[L - 1, :, pos, :], k.astype(np.float16).view(np.uint16))
        assert np.array_equal(vc[L - 1, :, pos, :], v.astype(np.float16).view(np.uint16))
    written = {0, 1, 2, 77}
    kc = m.buffer(capi.B_KEY_CACHE).reshape(L, nkv, shape.seq_len, hs)
    for p in range(shape.seq_len):
        if p not in written:
            assert not kc[:, :, p, :].any()
    m.close()


def test_distance_to_fp32_cache_cpu_path():
    """Against the reference CPU semantics proper (fp32 KV cache): the binary16
    cache the GPU API prescribes must still leave logits inside the tolerance."""
    shape = SMALL_SHAPES["gqa4_fp16"]
    m, o = build(shape, 9, kv_round=False)
    m.set_path(capi.PATH_FUSED)
    tok = 11
    worst = 0.0
    for pos in range(40):
        m.forward(tok, pos, 0.0)
        want = o.forward_logits(tok, pos)
        worst = max(worst, rel_err(m.buffer(capi.B_LOGITS), want))
        tok = int(np.argmax(want))
    assert worst <= LOGIT_TOL, worst
    m.close()
    o.close()


@pytest.mark.parametrize("path", PATHS, ids=PATH_IDS)
def test_generate_sampled_matches_oracle(path):
    """Generation loop with the fused sampler: temperature 0.8, penalty 1.1,
    64-entry sliding window, pre-drawn uniforms (config-3 settings, small shape)."""
    shape = SMALL_SHAPES["gqa4_fp16"]
    m, o = build(shape, 17)
    m.set_path(path)
    steps = 100
    draws = capi.synth_uniform_f32(steps, 99)
    first = 42
    toks, hist_after, stats = m.generate(first, 0, steps, temperature=0.8, penalty=1.1, history=[first],
                                         history_cap=64, uniforms=draws)
    assert stats.tokens == steps
    # replay on the oracle, feeding the GPU's tokens so that one allowed flip does not cascade
    hist = [first]
    tok = first
    flips = 0
    for i in range(steps):
        o.forward_logits(tok, i)
        want, lo, hi = ob.orc_sample_cdf(o.buf("logits"), 0.8, 1.1, hist, float(draws[i]))
        if toks[i] != want:
            flips += 1
            gap = min(abs(float(draws[i]) - lo), abs(float(draws[i]) - hi))
            assert gap < LOGIT_TOL, f"step {i}: token {toks[i]} vs {want}, CDF gap {gap}"
        tok = int(toks[i])
        hist = (hist + [tok])[-64:]
    assert flips <= 2
    assert hist_after == hist  # the window comes back oldest-first, like main.cpp:203-208 keeps it
    m.close()
    o.close()


@pytest.mark.parametrize("cap", [63, 65, 100, 1100])
@pytest.mark.parametrize("name", ["fp32_layer_to_an_xcd", "fp16"])
def test_a_penalty_window_longer_than_a_wavefront(name, cap):
    """The persistent path's sampler takes a window of up to 64 entries an entry to a lane, longer ones by threads that walk it,
    in LDS up to 1024 entries: windows that start one short of their capacity and slide, every id in them several times."""
    shape = (Shape(288, 768, 2, 6, 6, 1000, 1200, 10000.0, fp16=False, tied=True) if name != "fp16" else
             Shape(256, 512, 2, 8, 2, 1000, 1200, 500000.0, fp16=True, tied=True))
    m, o = build(shape, 17)
    m.set_path(capi.PATH_PERSISTENT)
    steps, tok = 24, 42
    draws = capi.synth_uniform_f32(steps, 99)
    hist = [int(t) % (cap // 3) for t in capi.synth_token_ids(cap - 1, 5, shape.vocab_size)]
    for temperature in (0.8, 0.0):
        toks, after, _ = m.generate(tok, 0, steps, temperature=temperature, penalty=1.3, history=hist, history_cap=cap, uniforms=draws)
        window, fed, agree = list(hist), tok, 0
        for i in range(steps):
            o.forward_logits(fed, i)
            if temperature == 0.0:
                want, z = ob.orc_sample(o.buf("logits"), 0.0, 1.0, 1.3, window, 0.0)
                gap = float(z[want] - z[toks[i]]) / float(np.max(np.abs(z)))
            else:
                want, lo, hi = ob.orc_sample_cdf(o.buf("logits"), temperature, 1.3, window, float(draws[i]))
                gap = min(abs(float(draws[i]) - lo), abs(float(draws[i]) - hi))
            agree += int(want == toks[i])
            assert want == toks[i] or gap < LOGIT_TOL, (temperature, i, gap)
            fed = int(toks[i])
            window = (window + [fed])[-cap:]
        assert agree >= steps - 1 and after == window
    m.close()
    o.close()


def test_generate_paths_agree_and_window_wraps():
    """Fused generate == operator-path generate token for token (greedy, penalty on,
    window of 5 so that it wraps many times)."""
    shape = SMALL_SHAPES["gqa8_fp16_untied"]
    m = Model(shape)
    m.load_synthetic(4)
    out = {}
    for path in PATHS:
        m.set_path(path)
        m.reset()
        out[path] = m.generate(7, 0, 60, temperature=0.0, penalty=1.3, history=[7], history_cap=5)
    a = out[capi.PATH_OPS]
    for path in PATHS[1:]:
        b = out[path]
        assert np.mean(a[0] == b[0]) >= 0.99
        if np.array_equal(a[0], b[0]):
            assert a[1] == b[1] and len(a[1]) == 5
    m.close()


def test_forward_then_generate_continuation():
    """Prefill by single forwards (main.cpp:163-179), then generate from the next
    position; positions and cache carry over."""
    shape = SMALL_SHAPES["mha_fp32_c1like"]
    m, o = build(shape, 2)
    m.set_path(capi.PATH_FUSED)
    prompt = capi.synth_token_ids(8, 1, shape.vocab_size)
    for pos in range(7):
        m.forward(int(prompt[pos]), pos, 0.0)
        o.forward_logits(int(prompt[pos]), pos)
    toks, _, _ = m.generate(int(prompt[7]), 7, 40, temperature=0.0)
    tok = int(prompt[7])
    agree = 0
    for i in range(40):
        want = int(np.argmax(o.forward_logits(tok, 7 + i)))
        agree += int(want == toks[i])
        tok = int(toks[i])
    assert agree >= 39
    m.close()
    o.close()


LONG_CONTEXT = {
    # name: (Shape, first position).  The persistent kernel gives grouped-query models work items that
    # cover two query heads of a KV head once the context is long enough to be split.
    "gqa4_hs32": (Shape(256, 512, 2, 8, 2, 1000, 4400, 500000.0, fp16=True, tied=True), 4300),
    "gqa8_hs32": (Shape(256, 512, 2, 8, 1, 1000, 4400, 500000.0, fp16=True, tied=True), 4300),
    "gqa2_hs128": (Shape(512, 512, 1, 4, 2, 500, 2400, 500000.0, fp16=True, tied=False), 2300),
    "mha_hs48_fp32": (Shape(192, 384, 2, 4, 4, 500, 4400, 10000.0, fp16=False, tied=True), 4300),
    "gqa2_hs64_just_split": (Shape(256, 512, 1, 4, 2, 500, 1100, 10000.0, fp16=True, tied=True), 1040),
}


@pytest.mark.parametrize("name", list(LONG_CONTEXT))
def test_long_context_attention_matches_oracle(name):
    """Config-4 style: cache pre-filled with binary16 N(0,1) up to a long position,
    then decode there; the split-context attention must agree with the CPU loop."""
    shape, start = LONG_CONTEXT[name]
    m, o = build(shape, 8)
    hs, nkv, L = shape.head_size, shape.n_kv_heads, shape.n_layers
    n = L * nkv * shape.seq_len * hs
    kfill = capi.synth_normal_f16(n, 501, 1.0).reshape(L, nkv, shape.seq_len, hs)
    vfill = capi.synth_normal_f16(n, 502, 1.0).reshape(L, nkv, shape.seq_len, hs)
    kfill[:, :, start:, :] = 0
    vfill[:, :, start:, :] = 0
    o.buf("key_cache")[:] = capi.f16_to_f32(kfill.reshape(-1))
    o.buf("value_cache")[:] = capi.f16_to_f32(vfill.reshape(-1))
    for path in PATHS:
        m.write_buffer(capi.B_KEY_CACHE, kfill)
        m.write_buffer(capi.B_VALUE_CACHE, vfill)
        m.set_path(path)
        tok = 5
        for pos in range(start, start + 6):
            m.forward(tok, pos, 0.0)
            want = o.forward_logits(tok, pos)
            assert rel_err(m.buffer(capi.B_LOGITS), want) <= LOGIT_TOL
            tok = int(np.argmax(want))
    m.close()
    o.close()


ONE_PASS = {
    # Heads of size 64: up to 512 positions the persistent kernel keeps a head's whole context on the compute unit
    # (one wavefront alone up to 64 positions).  Eight KV heads: q, k and v are also handed over inside each XCD.
    "gqa4_8kv": Shape(2048, 512, 1, 32, 8, 500, 640, 500000.0, fp16=True, tied=True),
    "gqa2_4kv": Shape(512, 768, 2, 8, 4, 500, 640, 10000.0, fp16=True, tied=False),
    # Sixteen KV heads: two per XCD (with their query heads), so a workgroup's rows of the stacked Wq/Wk/Wv run across
    # KV-head boundaries and an XCD's first workgroups hold the items of two KV heads.
    "mha_16kv": Shape(1024, 512, 1, 16, 16, 500, 640, 10000.0, fp16=True, tied=True),
    "gqa2_16kv": Shape(2048, 512, 1, 32, 16, 500, 640, 500000.0, fp16=True, tied=False),
    # Fewer KV heads than XCDs: two (four, eight) XCDs share a KV head, each with part of its query heads and its own
    # copy of the k and v rows ("gqa2_4kv" above is one of these too: a single query head per XCD).
    "gqa8_4kv": Shape(2048, 1024, 2, 32, 4, 500, 640, 10000.0, fp16=True, tied=False),
    "gqa8_2kv": Shape(1024, 512, 1, 16, 2, 500, 640, 500000.0, fp16=True, tied=True),
    "gqa8_1kv": Shape(512, 512, 2, 8, 1, 500, 640, 10000.0, fp16=True, tied=True),
}


@pytest.mark.parametrize("name", list(ONE_PASS))
def test_one_pass_attention_item_matches_oracle(name):
    """Decode across every boundary of the one-pass item: 64 positions (one wavefront / eight), 128, 384 (the
    wavefronts' LDS blocks change areas), 512 (its last position) and beyond (back to the walking item).  The
    cache past the context holds NaN bit patterns on the GPU: the item fetches whole blocks of 64 positions and
    must use nothing of what lies past the current one."""
    shape = ONE_PASS[name]
    m, o = build(shape, 9)
    m.set_path(capi.PATH_PERSISTENT)
    hs, nkv, L = shape.head_size, shape.n_kv_heads, shape.n_layers
    n = L * nkv * shape.seq_len * hs
    kfill = capi.synth_normal_f16(n, 601, 1.0).reshape(L, nkv, shape.seq_len, hs)
    vfill = capi.synth_normal_f16(n, 602, 1.0).reshape(L, nkv, shape.seq_len, hs)
    for start in (0, 61, 126, 381, 509):
        k_gpu, v_gpu = kfill.copy(), vfill.copy()
        k_gpu[:, :, start:, :] = 0x7e00  # binary16 NaN
        v_gpu[:, :, start:, :] = 0x7e00
        m.reset()
        m.write_buffer(capi.B_KEY_CACHE, k_gpu)
        m.write_buffer(capi.B_VALUE_CACHE, v_gpu)
        k_cpu, v_cpu = kfill.copy(), vfill.copy()
        k_cpu[:, :, start:, :] = 0
        v_cpu[:, :, start:, :] = 0
        o.buf("key_cache")[:] = capi.f16_to_f32(k_cpu.reshape(-1))
        o.buf("value_cache")[:] = capi.f16_to_f32(v_cpu.reshape(-1))
        tok = 5
        for pos in range(start, start + 6):
            m.forward(tok, pos, 0.0)
            want = o.forward_logits(tok, pos)
            got = m.buffer(capi.B_LOGITS)
            assert np.all(np.isfinite(got)), (start, pos)
            assert rel_err(got, want) <= LOGIT_TOL, (start, pos)
            tok = int(np.argmax(want))
    m.close()
    o.close()


# A 1B-shaped layer: wide enough for parked gate/up rows, eight KV heads for the per-XCD hand-overs, heads of size 64
# for the one-pass attention item.
SELF_SELECTED = Shape(2048, 8192, 1, 32, 8, 500, 640, 500000.0, fp16=True, tied=True)
VARIANTS = {
    "as_selected": {},
    "xcd_handovers_off": {capi.OPT_DECODE_XCD_HANDOVERS: 0},
    "xcd_qkv_off": {capi.OPT_DECODE_XCD_QKV: 0},
    "no_parking": {capi.OPT_DECODE_PARKING: 0},
    "walking_attention_item": {capi.OPT_DECODE_LANE_ITEM: 0},
    "xcd_attention_off": {capi.OPT_DECODE_XCD_ATTENTION: 0},
}


@pytest.mark.parametrize("variant", list(VARIANTS))
def test_persistent_alternatives_the_library_selects_by_itself(variant, test_options):
    """Every plan the persistent path may pick by itself -- from the probe of the device, the shape and the position
    -- decodes the same tokens as the oracle: each is forced here through a test hook, also switched in the middle
    of a decode (the step lists are rebuilt), positions 0..7 and 515..518 (past the range of the parked-rows plan and of the one-pass item)."""
    shape = SELF_SELECTED
    m, o = build(shape, 31)
    m.set_path(capi.PATH_PERSISTENT)
    tok, greedy = 5, []
    for pos in range(8):
        if pos == 3:
            for option, value in VARIANTS[variant].items():
                test_options(option, value)
        nxt = m.forward(tok, pos, 0.0)
        want = o.forward_logits(tok, pos)
        assert rel_err(m.buffer(capi.B_LOGITS), want) <= LOGIT_TOL, (variant, pos)
        assert nxt == int(np.argmax(want)), (variant, pos)
        greedy.append(nxt)
        tok = nxt
    # past the range of the plan with parked rows and of the one-pass item (the cache in between holds zeros on both sides)
    for pos in range(515, 519):
        nxt = m.forward(tok, pos, 0.0)
        want = o.forward_logits(tok, pos)
        assert rel_err(m.buffer(capi.B_LOGITS), want) <= LOGIT_TOL, (variant, pos)
        assert nxt == int(np.argmax(want)), (variant, pos)
        tok = nxt
    # the same plan through the generation loop, from a fresh cache
    m.reset()
    toks, _, _ = m.generate(5, 0, 8, temperature=0.0)
    assert toks.tolist() == greedy, variant
    m.close()
    o.close()


def test_generate_grows_from_the_parked_rows_plan_into_the_xcd_split():
    """One generation call that starts inside the one-pass item's 512 positions and ends past them: the launches
    change plan, step lists and kernel instance in mid-flight (the next token's launch is queued before the last
    one's id is back).  Teacher-forced against the oracle; the cache before the start holds zeros on both sides."""
    shape = SELF_SELECTED
    m, o = build(shape, 33)
    m.set_path(capi.PATH_PERSISTENT)
    start, steps = 505, 14
    toks, _, _ = m.generate(5, start, steps, temperature=0.0)
    tok = 5
    for i in range(steps):
        want = o.forward_logits(tok, start + i)
        assert int(toks[i]) == int(np.argmax(want)), (start + i, toks.tolist())
        tok = int(toks[i])
    assert rel_err(m.buffer(capi.B_LOGITS), want) <= LOGIT_TOL
    m.close()
    o.close()


def test_gateup_partition_weighted_by_xcd_changes_no_bit(test_options):
    """Before its first token a model on the persistent path traces two tokens and deals the hidden units out by how
    fast each XCD got through the gate/up phase.  Who forms a hidden unit does not change its value, and the cache row
    the traced tokens wrote is put back: a model set up with the hook off (even shares) gives the same logits and
    cache, bit for bit, from a cache pre-filled up to the traced position and beyond."""
    shape = Shape(2048, 4096, 3, 32, 8, 500, 640, 500000.0, fp16=True, tied=True)  # (the trace needs layers to average over)
    runs = []
    fill = capi.synth_normal_f16(shape.n_layers * shape.n_kv_heads * shape.seq_len * shape.head_size, 801, 1.0)
    for calibrate in (1, 0):
        test_options(capi.OPT_DECODE_CALIBRATE, calibrate)
        m = Model(shape)
        m.load_synthetic(41)
        m.set_path(capi.PATH_PERSISTENT)
        m.write_buffer(capi.B_KEY_CACHE, fill)
        m.write_buffer(capi.B_VALUE_CACHE, fill[::-1].copy())
        out, tok = [], 5
        for pos in range(300, 304):
            tok = m.forward(tok, pos, 0.0)
            out.append(m.buffer(capi.B_LOGITS).view(np.uint32).copy())
        runs.append((out, m.buffer(capi.B_KEY_CACHE).copy(), m.buffer(capi.B_VALUE_CACHE).copy()))
        m.close()
    (la, ka, va), (lb, kb, vb) = runs
    assert all(np.array_equal(x, y) for x, y in zip(la, lb))
    assert np.array_equal(ka, kb) and np.array_equal(va, vb)
    # the traced position's rows are the pre-filled ones again (positions 300..303 alone were written)
    k = ka.reshape(shape.n_layers, shape.n_kv_heads, shape.seq_len, shape.head_size)
    want = fill.reshape(k.shape)
    assert np.array_equal(k[:, :, :300, :], want[:, :, :300, :]) and np.array_equal(k[:, :, 304:, :], want[:, :, 304:, :])


def test_persistent_relaunches_a_token_when_an_xcd_is_dealt_unevenly(test_options):
    """A launch in which an XCD draws more tickets than its share ends with every workgroup leaving the kernel
    normally and no token delivered; the library switches the per-XCD hand-overs off and launches the same token
    again.  Forced from the host through the ticket base, in lpp_forward and in the middle of lpp_generate: the
    caller sees the oracle's tokens and no error."""
    shape = SELF_SELECTED
    m, o = build(shape, 32)
    m.set_path(capi.PATH_PERSISTENT)
    tok, fed, wants = 5, [], []
    for pos in range(10):
        if pos == 2:
            test_options(capi.OPT_DECODE_FAIL_TICKETS, 1)
        nxt = m.forward(tok, pos, 0.0)
        if pos == 2:
            assert capi.get_test_option(capi.OPT_DECODE_FAIL_TICKETS) == 0, "the forced failure was not taken"
        want = o.forward_logits(tok, pos)
        fed.append(tok)
        wants.append(want)
        assert rel_err(m.buffer(capi.B_LOGITS), want) <= LOGIT_TOL, pos
        assert nxt == int(np.argmax(want)), pos
        tok = nxt
    greedy = [int(np.argmax(w)) for w in wants]
    # the generation loop: the failure hits the n-th launch, with the launch after it already queued
    for nth in (1, 4, 10):
        m.reset()
        # per-XCD hand-overs back on: a changed option has the next launch probe the device again
        test_options(capi.OPT_DECODE_XCD_HANDOVERS, 0)
        test_options(capi.OPT_DECODE_XCD_HANDOVERS, 1)
        test_options(capi.OPT_DECODE_FAIL_TICKETS, nth)
        toks, _, _ = m.generate(5, 0, 10, temperature=0.0)
        assert capi.get_test_option(capi.OPT_DECODE_FAIL_TICKETS) == 0, "the forced failure was not taken"
        assert toks.tolist() == greedy, (nth, toks.tolist(), greedy)
    m.close()
    o.close()


XCD_SPLIT = {
    # name: (shape, first positions of the runs).  Where every KV head belongs to one XCD, contexts beyond the
    # one-pass item's 512 positions (heads of size 64) or beyond 96 (size 128) are split over that XCD's workgroups.
    "hs64_gqa4_8kv_long": (Shape(2048, 512, 1, 32, 8, 500, 9000, 500000.0, fp16=True, tied=True), (600, 4093, 8441)),
    "hs128_gqa4_8kv": (Shape(4096, 512, 1, 32, 8, 500, 1300, 500000.0, fp16=True, tied=False), (93, 500, 1050)),
    "hs128_mha_8kv": (Shape(1024, 512, 1, 8, 8, 500, 700, 10000.0, fp16=True, tied=True), (120, 640)),
    "hs64_mha_32kv": (Shape(2048, 512, 1, 32, 32, 500, 4200, 10000.0, fp16=True, tied=True), (520, 4090)),
    "hs64_gqa2_16kv": (Shape(2048, 512, 1, 32, 16, 500, 1100, 500000.0, fp16=True, tied=False), (515, 1000)),
    # hidden_dim well above dim: the share's rows live in the part of the staged-activation area that only the down
    # phase uses, and every workgroup parks gate/up rows beside the item (two layers: the down phase overwrites the
    # rows in between); the last start of the first shape is past what that area holds (3072 positions): the rows run on
    # into the parked rows' area
    "hs64_gqa4_8kv_parked": (Shape(2048, 8192, 2, 32, 8, 500, 3300, 500000.0, fp16=True, tied=True), (520, 3066, 3090)),
    "hs128_gqa4_8kv_parked": (Shape(4096, 14336, 2, 32, 8, 500, 1300, 500000.0, fp16=True, tied=False), (620, 1050)),
    # long contexts with parked rows: the share's rows run on from that area into the parked rows' own (overwritten
    # by this layer's rows once the item is done, and by the next layer's share after those are multiplied) and, at
    # the third start, into an area behind them; the last start is past what LDS takes: the plain split
    "hs64_gqa4_8kv_parked_long": (Shape(2048, 8192, 2, 32, 8, 500, 14100, 500000.0, fp16=True, tied=True), (4100, 8441, 14050, 14090)),
}


@pytest.mark.parametrize("name", list(XCD_SPLIT))
def test_context_split_over_an_xcd_matches_oracle(name):
    """The long-context attention of the persistent path (a KV head's context shared out among the workgroups of its
    XCD, rows resident in LDS): six steps from each start on a cache of seeded values, NaN bit patterns past the
    context on the GPU (whole rows are fetched ahead, nothing past the current position may be used), logits and
    greedy ids against the oracle.  Starts sit on both sides of where the library switches to this item, at
    share sizes that fill an exchange wavefront's 64 positions unevenly, and next to the largest context a shape takes."""
    shape, starts = XCD_SPLIT[name]
    m, o = build(shape, 17)
    m.set_path(capi.PATH_PERSISTENT)
    hs, nkv, L = shape.head_size, shape.n_kv_heads, shape.n_layers
    n = L * nkv * shape.seq_len * hs
    kfill = capi.synth_normal_f16(n, 701, 1.0).reshape(L, nkv, shape.seq_len, hs)
    vfill = capi.synth_normal_f16(n, 702, 1.0).reshape(L, nkv, shape.seq_len, hs)
    for start in starts:
        k_gpu, v_gpu = kfill.copy(), vfill.copy()
        k_gpu[:, :, start:, :] = 0x7e00  # binary16 NaN
        v_gpu[:, :, start:, :] = 0x7e00
        m.reset()
        m.write_buffer(capi.B_KEY_CACHE, k_gpu)
        m.write_buffer(capi.B_VALUE_CACHE, v_gpu)
        k_cpu, v_cpu = kfill.copy(), vfill.copy()
        k_cpu[:, :, start:, :] = 0
        v_cpu[:, :, start:, :] = 0
        o.buf("key_cache")[:] = capi.f16_to_f32(k_cpu.reshape(-1))
        o.buf("value_cache")[:] = capi.f16_to_f32(v_cpu.reshape(-1))
        tok = 5
        for pos in range(start, min(start + 6, shape.seq_len)):
            print(f"xcd split {name}: pos {pos}", flush=True)
            nxt = m.forward(tok, pos, 0.0)
            want = o.forward_logits(tok, pos)
            got = m.buffer(capi.B_LOGITS)
            assert np.all(np.isfinite(got)), (start, pos)
            assert rel_err(got, want) <= LOGIT_TOL, (start, pos)
            assert nxt == int(np.argmax(want)), (start, pos)
            tok = nxt
    m.close()
    o.close()


RESIDENT = {
    # name: (shape, first positions of the runs).  fp32 models whose layers fit an XCD's registers (dim to 320, hidden to 768).
    "c1_more_layers_than_xcds": (Shape(288, 768, 10, 6, 6, 1000, 256, 10000.0, fp16=False, tied=True), (0, 62, 250)),
    "widest_gqa": (Shape(320, 768, 3, 8, 2, 50000, 600, 500000.0, fp16=False, tied=False), (0, 126, 254, 507)),  # classifier rows beyond LDS
    "hs64_one_kv_head": (Shape(256, 516, 2, 4, 1, 777, 520, 10000.0, fp16=False, tied=True), (0, 254, 510)),
    "tiny_idle_workgroups": (Shape(32, 44, 9, 4, 2, 300, 64, 10000.0, fp16=False, tied=True), (0, 58)),
    "one_layer": (Shape(64, 160, 1, 1, 1, 500, 64, 10000.0, fp16=False, tied=False), (0,)),
}


@pytest.mark.parametrize("name", list(RESIDENT))
def test_layers_resident_in_an_xcd_match_the_oracle(name, test_options):
    """The persistent path of small fp32 models, a layer to an XCD: logits and greedy ids against the oracle and against
    the general kernel (taken by the hook, and by itself past 512 positions), NaN bit patterns past the context."""
    shape, starts = RESIDENT[name]
    m, o = build(shape, 19)
    m.set_path(capi.PATH_PERSISTENT)
    hs, nkv, L = shape.head_size, shape.n_kv_heads, shape.n_layers
    n = L * nkv * shape.seq_len * hs
    kfill = capi.synth_normal_f16(n, 901, 1.0).reshape(L, nkv, shape.seq_len, hs)
    vfill = capi.synth_normal_f16(n, 902, 1.0).reshape(L, nkv, shape.seq_len, hs)
    for start in starts:
        k_cpu, v_cpu = kfill.copy(), vfill.copy()
        k_cpu[:, :, start:, :] = 0
        v_cpu[:, :, start:, :] = 0
        o.buf("key_cache")[:] = capi.f16_to_f32(k_cpu.reshape(-1))
        o.buf("value_cache")[:] = capi.f16_to_f32(v_cpu.reshape(-1))
        fed, wants, tok = [], [], 5
        positions = range(start, min(start + 8, shape.seq_len))
        for pos in positions:
            fed.append(tok)
            wants.append(o.forward_logits(tok, pos))
            tok = int(np.argmax(wants[-1]))
        caches = []
        for resident in (1, 0):
            test_options(capi.OPT_DECODE_RESIDENT, resident)
            k_gpu, v_gpu = kfill.copy(), vfill.copy()
            k_gpu[:, :, start:, :] = 0x7e00  # binary16 NaN
            v_gpu[:, :, start:, :] = 0x7e00
            m.write_buffer(capi.B_KEY_CACHE, k_gpu)
            m.write_buffer(capi.B_VALUE_CACHE, v_gpu)
            for pos, t, want in zip(positions, fed, wants):
                nxt = m.forward(t, pos, 0.0)
                got = m.buffer(capi.B_LOGITS)
                assert np.all(np.isfinite(got)), (start, pos, resident)
                assert rel_err(got, want) <= LOGIT_TOL, (start, pos, resident)
                assert nxt == int(np.argmax(want)), (start, pos, resident)
            kc = m.buffer(capi.B_KEY_CACHE).reshape(k_gpu.shape)
            assert np.array_equal(kc[:, :, :start], k_gpu[:, :, :start]) and np.all(kc[:, :, positions[-1] + 1:] == 0x7e00)
            k = m.buffer(capi.B_K).reshape(nkv, hs)  # the run state holds the last layer's
            assert np.array_equal(kc[L - 1, :, positions[-1]], k.astype(np.float16).view(np.uint16))
            caches.append(kc.view(np.float16).astype(np.float32)[:, :, list(positions)])
        # one binary16 step between the two kernels' orders of the same fp32 sums, amplified through the layers
        assert np.max(np.abs(caches[0] - caches[1])) <= LOGIT_TOL * np.max(np.abs(caches[1]))
    m.close()
    o.close()


def test_a_resident_model_launches_the_general_kernel_only_where_it_needs_it(test_options):
    """A new small fp32 model's first calls are as many launches as tokens: the two traced tokens (three launches each) that deal
    out the general kernel's hidden units come with the first call that leaves the first 512 positions.  Counted by the hook
    that counts launches down to a failing one."""
    shape = Shape(288, 768, 3, 6, 6, 1000, 600, 10000.0, fp16=False, tied=True)
    launches = 0

    def check(expect):
        nonlocal launches
        launches += expect
        assert capi.get_test_option(capi.OPT_DECODE_FAIL_TICKETS) == 1000 - launches

    for first in ("forward", "generate", "run", "profile"):
        m = Model(shape)
        m.load_synthetic(3)
        m.set_path(capi.PATH_PERSISTENT)
        test_options(capi.OPT_DECODE_FAIL_TICKETS, 1000)
        launches = 0
        if first == "forward":
            m.forward(5, 511)
            check(1)
        elif first == "generate":
            m.generate(5, 500, 12)
            check(12)
        elif first == "run":
            m.run([5, 6, 7], 10, 0.0)
            check(10)
        else:
            m.profile_kernels(20, reps=4)
            check(4)
        if first == "run":
            m.generate(5, 500, 13)
            check(13 + 6)
        else:
            m.forward(5, 512)
            check(1 + 6)
        m.generate(5, 510, 4)
        check(4)
        m.close()


def test_profile_names_the_kernel_that_decodes(test_options):
    """lpp_profile_kernels on the persistent path: a small fp32 model's tokens are k_decode_resident's up to 512 positions."""
    m = Model(Shape(288, 768, 2, 6, 6, 1000, 600, 10000.0, fp16=False, tied=True))
    m.load_synthetic(3)
    m.set_path(capi.PATH_PERSISTENT)
    for resident, pos, want in [(1, 0, "k_decode_resident"), (1, 511, "k_decode_resident"), (1, 512, "k_decode_dataflow"), (0, 0, "k_decode_dataflow")]:
        test_options(capi.OPT_DECODE_RESIDENT, resident)
        assert [row[0] for row in m.profile_kernels(pos, reps=2)] == [want], (resident, pos)
    m.close()


def test_model_argument_errors():
    shape = SMALL_SHAPES["gqa4_fp16"]
    m = Model(shape)
    with pytest.raises(capi.LppError) as e:
        m.forward(1, 0)
    assert e.value.status == capi.LPP_ERR_STATE  # weights not uploaded
    m.load_synthetic(1)
    for bad in [dict(token=-1, pos=0), dict(token=shape.vocab_size, pos=0), dict(token=0, pos=shape.seq_len)]:
        with pytest.raises(capi.LppError) as e:
            m.forward(bad["token"], bad["pos"])
        assert e.value.status == capi.LPP_ERR_INVALID_ARG
    with pytest.raises(capi.LppError):
        m.generate(0, shape.seq_len - 3, 10)
    m.close()


@pytest.mark.parametrize("cfg,steps,start", [("c1_llama2c_15m_fp32", 24, 0), ("c3_llama32_1b_fp16", 6, 0)])
def test_benchmark_shapes_first_steps(cfg, steps, start):
    """The real benchmark shapes for a handful of steps (the oracle needs about a
    second per token at the 1B shape)."""
    shape = CONFIGS[cfg]
    m, o = build(shape, 1234)
    m.set_path(capi.PATH_FUSED)
    tok = int(capi.synth_token_ids(1, 77, shape.vocab_size)[0])
    agree = 0
    for pos in range(start, start + steps):
        nxt = m.forward(tok, pos, 0.0)
        want = o.forward_logits(tok, pos)
        assert rel_err(m.buffer(capi.B_LOGITS), want) <= LOGIT_TOL
        agree += int(nxt == int(np.argmax(want)))
        tok = int(np.argmax(want))
    assert agree == steps
    m.close()
    o.close()


def test_persistent_timeline_is_ordered():
    """lpp_trace_token: every phase of the persistent kernel reports its marks, in order, and the
    phases follow one another."""
    import ctypes as C
    shape = SMALL_SHAPES["gqa4_fp16"]
    m, o = build(shape, 4)
    arr = (C.c_ulonglong * 4096)()
    n, marks = C.c_int(), C.c_int()
    capi.check(m.lib.lpp_trace_token(m.handle, 5, arr, 4096, C.byref(n), C.byref(marks)))
    phases = 5 * shape.n_layers + 2
    assert marks.value == 8 and n.value == 8 * phases
    t = np.array(arr[:n.value], dtype=np.int64).reshape(phases, 8)
    published = t[:, 4]
    assert np.all(np.diff(published) > 0), "phases out of order"
    gemv = [i for i in range(5 * shape.n_layers) if i % 5 != 1] + [5 * shape.n_layers]
    for i in gemv:
        e, polled, staged, rows, pub = t[i, 0], t[i, 1], t[i, 2], t[i, 3], t[i, 4]
        assert 0 < e <= polled <= staged <= rows <= pub, (i, t[i])
    assert published[-1] < 100_000_00, "a tiny model's token takes far less than a second (10 ns ticks)"
    m.close()
    o.close()


def test_rows_wider_than_the_persistent_kernel_takes():
    """fp32 rows of more than 8192 columns (eight column slices of 1024) do not fit the persistent
    kernel's step lists: it must refuse the shape, not drop columns; the other two schedules take it
    and agree with the oracle."""
    shape = Shape(256, 8448, 1, 4, 2, 300, 16, 10000.0, fp16=False, tied=True)
    m, o = build(shape, 6)
    with pytest.raises(capi.LppError) as e:
        m.set_path(capi.PATH_PERSISTENT)
    assert e.value.status == capi.LPP_ERR_UNSUPPORTED
    wants, fed, tok = [], [], 5
    for pos in range(6):
        fed.append(tok)
        wants.append(o.forward_logits(tok, pos))
        tok = int(np.argmax(wants[-1]))
    for path in (capi.PATH_OPS, capi.PATH_FUSED):
        m.reset()
        m.set_path(path)
        for pos in range(6):
            m.forward(fed[pos], pos, 0.0)
            assert rel_err(m.buffer(capi.B_LOGITS), wants[pos]) <= LOGIT_TOL
    m.close()
    o.close()
    # the widest rows it does take: 8192 fp32 columns, all eight slices full
    shape = Shape(256, 8192, 1, 4, 2, 300, 16, 10000.0, fp16=False, tied=True)
    m, o = build(shape, 6)
    m.set_path(capi.PATH_PERSISTENT)
    tok = 5
    for pos in range(6):
        m.forward(tok, pos, 0.0)
        want = o.forward_logits(tok, pos)
        assert rel_err(m.buffer(capi.B_LOGITS), want) <= LOGIT_TOL
        tok = int(np.argmax(want))
    m.close()
    o.close()


def test_persistent_bounded_wait_gives_up_and_recovers():
    """The persistent kernel's waits for other workgroups' values are bounded.  With the bound set to
    one poll by the host, a wait runs out, every workgroup leaves the kernel normally, the call
    reports LPP_ERR_HIP, and the same model decodes correctly again once the bound is restored."""
    shape = SMALL_SHAPES["gqa4_fp16"]
    m, o = build(shape, 12)
    m.set_path(capi.PATH_PERSISTENT)
    tok = 9
    want0 = o.forward_logits(tok, 0)
    assert m.forward(tok, 0, 0.0) == int(np.argmax(want0))
    capi.check(m.lib.lpp_model_set_spin_limit(m.handle, 1))
    with pytest.raises(capi.LppError) as e:
        m.forward(int(np.argmax(want0)), 1, 0.0)
    assert e.value.status == capi.LPP_ERR_HIP and "gave up" in str(e.value)
    with pytest.raises(capi.LppError):
        m.generate(3, 1, 4, temperature=0.0)
    capi.check(m.lib.lpp_model_set_spin_limit(m.handle, 1 << 20))
    m.reset()
    tok = 9
    for pos in range(8):
        nxt = m.forward(tok, pos, 0.0)
        want = o.forward_logits(tok, pos) if pos > 0 else want0
        assert rel_err(m.buffer(capi.B_LOGITS), want) <= LOGIT_TOL
        assert nxt == int(np.argmax(want))
        tok = nxt
    m.close()
    o.close()


def test_persistent_sequence_numbers_restart_before_they_wrap():
    """Hand-over tags are 32-bit sequence numbers compared for equality.  Moved close to the end of
    their range by the host, they are re-based (slots cleared, count restarted) without a wrong step."""
    shape = SMALL_SHAPES["gqa4_fp16"]
    m, o = build(shape, 13)
    m.set_path(capi.PATH_PERSISTENT)
    tok = 4
    for pos in range(12):
        if pos == 4:
            capi.check(m.lib.lpp_model_set_sequence_base(m.handle, 0xF0000000 - 20))  # two tokens short of the guard
        nxt = m.forward(tok, pos, 0.0)
        want = o.forward_logits(tok, pos)
        assert rel_err(m.buffer(capi.B_LOGITS), want) <= LOGIT_TOL, pos
        assert nxt == int(np.argmax(want))
        tok = nxt
    m.close()
    o.close()
