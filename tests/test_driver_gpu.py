"""lpp_run (the driver loop of src/main.cpp:139-232) and lpp_model_load_checkpoint
(the llama2.c reader of src/loader.cpp) on a real MI355X, through the C ABI.

The oracle's loop (orc_run) is pinned on the CPU against the reference's own
executable (tests/test_driver_cpu.py).  Here the GPU loop is checked against it:
the loop's bookkeeping exactly (positions, window contents, stop, main.cpp's own
count), the tokens by teacher-forcing the GPU's own stream through the oracle --
a free-running comparison would let one near-tie cascade -- with the bars of the
decode path: >= 99 % agreement, and where the two differ the GPU's choice within
the logits tolerance of the oracle's.
"""
import json
from pathlib import Path

import numpy as np
import pytest

import oracle_binding as ob
from lighterpp_amd import Checkpoint, Model, Shape, capi, synth_tensor, write_checkpoint

pytestmark = pytest.mark.gpu
LOGIT_TOL = 2e-3
EOS = (2, 128001, 128009)
PATHS = [capi.PATH_OPS, capi.PATH_FUSED, capi.PATH_PERSISTENT]
PATH_IDS = ["ops", "fused", "persistent"]
GOLDEN = json.loads((Path(__file__).resolve().parent / "golden" / "ref_driver.json").read_text())


def golden_shape(case) -> Shape:
    d, h, L, nh, nkv, v, s = case["shape"]
    return Shape(d, h, L, nh, nkv, v, s, 10000.0, fp16=False, tied=True)


def weights(shape: Shape, seed: int) -> dict:
    return {t: synth_tensor(shape, t, seed) for t in range(12)}


def check_against_oracle(shape, w, prompt, steps, temperature, uniforms, ids, res):
    """Bookkeeping exact; tokens teacher-forced through the oracle."""
    prompt = list(prompt) if prompt else [1]
    n_prompt = len(prompt)
    ids = [int(t) for t in ids]
    stop_id = int(res.history[res.history_len - 1]) if res.stopped_by_eos else None
    stream = ids + ([stop_id] if res.stopped_by_eos else [])
    assert res.n_tokens == len(ids)
    assert all(t not in EOS for t in ids)
    if res.stopped_by_eos:
        assert stop_id in EOS
    else:
        assert res.final_pos == steps
    assert res.final_pos == n_prompt - 1 + len(ids)
    assert res.reported_count == res.final_pos - n_prompt
    assert list(res.history[:res.history_len]) == (prompt + stream)[-64:]

    o = ob.OracleModel(shape, w, fp16=shape.fp16, kv_round_f16=True)
    u = (lambda p: float(uniforms[p])) if uniforms is not None else (lambda p: 0.0)
    hist, pos = [], 0
    for t in prompt[:-1]:
        hist = (hist + [t])[-64:]
        o.forward(t, pos, temperature, 1.0, 1.1, hist, u(pos))
        pos += 1
    tok = prompt[-1]
    hist = (hist + [tok])[-64:]
    agree = 0
    for g in stream:
        logits = o.forward_logits(tok, pos)
        want, mutated = ob.orc_sample(logits, temperature, 1.0, 1.05, hist, u(pos))
        if want == g:
            agree += 1
        elif temperature == 0.0:
            gap = float(mutated[want] - mutated[g])
            assert gap <= LOGIT_TOL * float(np.max(np.abs(mutated))), f"position {pos}: {g} vs {want}, gap {gap}"
        else:  # the draw must sit within the tolerance of an edge of the CPU's cumulative distribution
            _, lo, hi = ob.orc_sample_cdf(logits, temperature, 1.05, hist, u(pos))
            gap = min(abs(u(pos) - lo), abs(u(pos) - hi))
            assert gap <= LOGIT_TOL, f"position {pos}: {g} vs {want}, CDF gap {gap}"
        tok = g
        hist = (hist + [g])[-64:]
        pos += 1
    assert agree >= int(np.ceil(0.99 * len(stream))), f"agreement {agree}/{len(stream)}"
    o.close()
    return len(stream) - agree


def run_or_skip(m: Model, path: int, *args, **kw):
    m.set_path(path)
    try:
        return m.run(*args, **kw)
    except capi.LppError as e:
        if e.status == capi.LPP_ERR_UNSUPPORTED:
            pytest.skip(f"shape not supported on this path: {e}")
        raise


@pytest.mark.parametrize("path", PATHS, ids=PATH_IDS)
@pytest.mark.parametrize("name", list(GOLDEN))
def test_run_on_the_reference_executables_cases(name, path):
    case = GOLDEN[name]
    shape = golden_shape(case)
    w = weights(shape, case["seed"])
    m = Model(shape)
    for t in range(capi.T_WCLS):
        m.upload(t, w[t])
    m.tie_classifier()
    ids, res = run_or_skip(m, path, case["prompt_ids"], case["steps"], 0.0)
    flips = check_against_oracle(shape, w, case["prompt_ids"], case["steps"], 0.0, None, ids, res)
    # the reference executable's own run: identical, unless a near-tie (bounded above) flipped a token
    want = case["generated"]
    if flips == 0:
        assert ids.tolist() == want, f"{name}: ids differ from the reference executable's although every step agrees with the oracle"
        assert res.reported_count == case["reported_count"]
    else:
        first = next((i for i, (a, b) in enumerate(zip(ids.tolist(), want)) if a != b), min(len(ids), len(want)))
        assert ids.tolist()[:first] == want[:first]
        print(f"{name}: {flips} near-tie flip(s); first {first} of {len(want)} ids equal to the reference executable's")
    m.close()


@pytest.mark.parametrize("path", PATHS, ids=PATH_IDS)
def test_run_with_temperature_and_long_prompt(path):
    """Sampled run over more than 64 positions: prefill draws, window slide, penalties."""
    shape = Shape(288, 768, 3, 6, 6, 1000, 160, 10000.0, fp16=False, tied=True)
    w = weights(shape, 31)
    m = Model(shape)
    for t in range(capi.T_WCLS):
        m.upload(t, w[t])
    m.tie_classifier()
    prompt = [int(t) for t in capi.synth_token_ids(70, 8, shape.vocab_size)]
    prompt = [t if t not in EOS else 3 for t in prompt]
    steps = 150
    u = capi.synth_uniform_f32(steps, 77)
    ids, res = run_or_skip(m, path, prompt, steps, 0.8, 1.0, u)
    check_against_oracle(shape, w, prompt, steps, 0.8, u, ids, res)
    m.close()

QUEUED = {
    # name: (shape, prompt ids, steps, the earliest generated step that ends the sequence)
    "mha_fp32": (Shape(288, 768, 3, 6, 6, 1000, 96, 10000.0, fp16=False, tied=True), 7, 40, 9),          # a layer to an XCD
    "mha_fp32_general": (Shape(288, 768, 3, 6, 6, 1000, 96, 10000.0, fp16=False, tied=True), 7, 40, 9),  # (that kernel off)
    "mha_fp32_past_512": (Shape(288, 768, 2, 6, 6, 1000, 640, 10000.0, fp16=False, tied=True), 516, 560, 9),  # one kernel, then the other
    "fp32_sliced": (Shape(1536, 2304, 2, 12, 4, 600, 96, 10000.0, fp16=False, tied=True), 7, 40, 9),     # rows of several slices
    "gqa4_8kv": (Shape(2048, 1024, 2, 32, 8, 500, 640, 500000.0, fp16=True, tied=True), 7, 40, 9),       # parked rows, one-pass item
    "hs128_8kv": (Shape(1024, 512, 1, 8, 8, 3000, 300, 10000.0, fp16=True, tied=True), 130, 170, 2),      # context split from 96 positions on
}


@pytest.mark.parametrize("fail", [0, 3, 9], ids=["clean", "a_prompt_launch_fails", "a_generating_launch_fails"])
@pytest.mark.parametrize("name", list(QUEUED))
def test_run_leaves_what_single_steps_leave(name, fail, test_options):
    """lpp_run on the persistent path queues its steps ahead (the prompt's end with their k and v rows, a launch behind an
    id that ends the sequence does nothing): ids, cache and last logits are those of one lpp_forward per id, bit for
    bit, also where the sequence ends early; where a launch fails its ticket check, to the rounding of the plan that follows."""
    shape, n_prompt, steps, end_at = QUEUED[name]
    w = weights(shape, 5)
    test_options(capi.OPT_DECODE_RESIDENT, int(name != "mha_fp32_general"))
    prompt = [int(t) if t not in EOS else 3 for t in capi.synth_token_ids(n_prompt, 4, shape.vocab_size)]

    def loaded():
        m = Model(shape)
        for t in range(capi.T_WCLS):
            m.upload(t, w[t])
        m.tie_classifier()
        m.set_path(capi.PATH_PERSISTENT)
        return m

    m = loaded()
    ids, _ = m.run(prompt, steps, 0.0)
    m.close()
    # the id generated at step end_at or the first one after it that is new trades rows with id 2: the sequence ends there
    last = next(int(t) for i, t in enumerate(ids) if i >= end_at and t not in prompt and t not in ids[:i])
    w[capi.T_TOKEN_EMBEDDING][[2, last]] = w[capi.T_TOKEN_EMBEDDING][[last, 2]]
    a, b = loaded(), loaded()
    for m in (a, b):  # (the launches that deal out the hidden units come with it: none of those is the one that fails)
        m.forward(3, shape.seq_len - 1, 0.0)
    if fail:
        test_options(capi.OPT_DECODE_FAIL_TICKETS, n_prompt - 2 if fail == 3 else n_prompt + 3)
    ids, res = a.run(prompt, steps, 0.0)
    assert capi.get_test_option(capi.OPT_DECODE_FAIL_TICKETS) == 0
    assert res.stopped_by_eos and res.final_pos < steps - 1
    hist, want, tok = [], [], 0
    for pos in range(res.final_pos + 1):
        tok = prompt[pos] if pos < n_prompt else tok
        hist = (hist + [tok])[-64:]
        tok = b.forward(tok, pos, 0.0, penalty=1.05 if pos >= n_prompt - 1 else 1.1, history=hist)
        if pos >= n_prompt - 1:
            want.append(tok)
    assert want[-1] == 2 and ids.tolist() == want[:-1]
    for buf in (capi.B_LOGITS, capi.B_KEY_CACHE, capi.B_VALUE_CACHE):
        got, expect = a.buffer(buf).view(np.uint16), b.buffer(buf).view(np.uint16)
        if fail == 0:
            assert np.array_equal(got, expect), buf
        elif buf == capi.B_LOGITS:  # (the per-XCD hand-overs are off from there on: another order of the attention's sums)
            assert np.max(np.abs(got.view(np.float32) - expect.view(np.float32))) <= LOGIT_TOL * np.max(np.abs(expect.view(np.float32)))
        else:  # ... which the cache shows as steps of binary16, and nowhere else
            got, expect = got.view(np.float16).astype(np.float32), expect.view(np.float16).astype(np.float32)
            assert np.max(np.abs(got - expect)) <= LOGIT_TOL * np.max(np.abs(expect)), buf
    # nothing generated: the last prompt id's logits are there all the same
    a.run(prompt, n_prompt - 1, 0.0)
    hist = []
    for pos, t in enumerate(prompt[:-1]):
        hist = (hist + [t])[-64:]
        b.forward(t, pos, 0.0, penalty=1.1, history=hist)
    if fail == 0:
        assert np.array_equal(a.buffer(capi.B_LOGITS), b.buffer(capi.B_LOGITS))
    else:
        assert np.max(np.abs(a.buffer(capi.B_LOGITS) - b.buffer(capi.B_LOGITS))) <= LOGIT_TOL * np.max(np.abs(b.buffer(capi.B_LOGITS)))
    a.close()
    b.close()


@pytest.mark.parametrize("batched", [False, True])
def test_the_time_of_a_reply_of_one_id_is_a_step(batched):
    """wall_seconds holds the whole first generated step, which is launched behind the prompt's before the host can look at
    the clock: never less than a step in a row of them takes on the device (5 % for the clocks)."""
    shape = Shape(288, 768, 6, 6, 6, 32000, 256, 10000.0, fp16=False, tied=True) if not batched else \
        Shape(256, 512, 2, 4, 2, 2048, 160, 500000.0, fp16=True, tied=True)
    m = Model(shape)
    m.load_synthetic(3)
    m.set_path(capi.PATH_PERSISTENT)
    prompt = capi.synth_token_ids(16, 4, shape.vocab_size)
    step = min(m.generate(int(prompt[-1]), 15, 16)[2].device_ms / 16e3 for _ in range(5))
    walls = [m.run(prompt, len(prompt), 0.0, batched_prefill=batched)[1].wall_seconds for _ in range(8)]
    print(f"a step {step * 1e6:.1f} us, a reply of one id {[round(w * 1e6, 1) for w in walls]} us", flush=True)
    assert min(walls) >= 0.95 * step
    m.close()


def test_run_fp16_model_persistent():
    shape = Shape(256, 512, 3, 8, 2, 2048, 160, 500000.0, fp16=True, tied=True)
    m = Model(shape)
    w = m.load_synthetic(14, keep=True)
    m.set_path(capi.PATH_PERSISTENT)
    prompt = [5, 9, 100, 7]
    ids, res = m.run(prompt, 120, 0.0)
    check_against_oracle(shape, w, prompt, 120, 0.0, None, ids, res)
    m.close()


def test_run_rejects_bad_arguments():
    shape = Shape(64, 160, 2, 8, 2, 80, 32, 10000.0, fp16=False, tied=True)
    m = Model(shape)
    m.load_synthetic(2)
    m.set_path(capi.PATH_OPS)
    with pytest.raises(capi.LppError):
        m.run([1, 2], 33, 0.0)  # beyond seq_len
    with pytest.raises(capi.LppError):
        m.run([1, 80], 10, 0.0)  # id outside the vocabulary
    with pytest.raises(capi.LppError):
        m.run([1], 10, 0.7)  # a temperature without draws
    m.close()


@pytest.mark.parametrize("path", PATHS, ids=PATH_IDS)
def test_model_from_checkpoint_equals_uploaded_model(path, tmp_path):
    shape = Shape(288, 768, 3, 6, 6, 1000, 64, 10000.0, fp16=False, tied=True)
    w = weights(shape, 9)
    file = tmp_path / "model.bin"
    write_checkpoint(file, shape, w)
    ck = Checkpoint(file)
    a = Model.from_checkpoint(ck)
    ck.close()  # the model holds its own copy in HBM
    b = Model(shape)
    for t in range(capi.T_WCLS):
        b.upload(t, w[t])
    b.tie_classifier()
    for mdl in (a, b):
        mdl.set_path(path)
    tok_a = tok_b = 11
    for pos in range(6):
        tok_a = a.forward(tok_a, pos, 0.0)
        la = a.buffer(capi.B_LOGITS)
        tok_b = b.forward(tok_b, pos, 0.0)
        lb = b.buffer(capi.B_LOGITS)
        assert np.array_equal(la.view(np.uint32), lb.view(np.uint32)), f"position {pos}"
        assert tok_a == tok_b
    a.close()
    b.close()


def test_command_line_driver_text_in_text_out(tmp_path):
    """python -m lighterpp_amd.driver on a llama2.c checkpoint with a tokenizer file: the text it
    prints is the prompt's and the generated ids' strings, the ids are lpp_run's."""
    import struct
    import subprocess
    import sys
    from lighterpp_amd import Tokenizer
    shape = Shape(64, 96, 2, 4, 2, 40, 200, 10000.0, fp16=False, tied=True)
    w = weights(shape, 22)
    ck, tk = tmp_path / "m.bin", tmp_path / "t.bin"
    write_checkpoint(ck, shape, w)
    alphabet = "abcdefghijklmnopqrstuvwxyzABCDEFGHIJKLMN"
    with open(tk, "wb") as f:
        f.write(struct.pack("<i", 1))
        for ch in alphabet:
            f.write(struct.pack("<fi", 0.0, 1) + ch.encode())
    root = Path(__file__).resolve().parent.parent
    out = subprocess.run([sys.executable, "-m", "lighterpp_amd.driver", str(ck), "--tokenizer", str(tk), "--prompt", "hello",
                          "--steps", "60", "--temperature", "0", "--path", "persistent"],
                         cwd=root, capture_output=True, text=True, timeout=110)
    assert out.returncode == 0, out.stderr
    assert "Encoded 5 tokens." in out.stdout and "Tokens generated: 55" in out.stdout
    text = out.stdout.split("--- Running Inference ---\n", 1)[1].split("\n\n--- Statistics ---", 1)[0].strip("\n")
    tok = Tokenizer.load(tk, shape.vocab_size)
    prompt = tok.encode("hello")
    assert prompt == [alphabet.index(c) for c in "hello"]
    m = Model(shape)
    for t in range(capi.T_WCLS):
        m.upload(t, w[t])
    m.tie_classifier()
    m.set_path(capi.PATH_PERSISTENT)
    ids, res = m.run(prompt, 60, 0.0)
    assert text == "".join(alphabet[i] for i in prompt + ids.tolist())
    m.close()
