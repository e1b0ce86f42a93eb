"""Full-model parity on the GPU: the device-resident forward
(include/qwen3_hip_model.h) and the reference forward driving the GPU
plug-in, against the reference forward on the CPU.

Golden data (tests/golden/model_*.npz, written by make_model_fixtures.py):
greedy tokens, top-2 margins and prefill logits of the reference forward
(fpga_bringup/src/src/qwen3.c with kernels_hwsim.c, i.e. A rounded to bf16
as on the AME target, and ops_scalar.c) on a random-init QW3M blob that the
tests rebuild from its seed (checksum compared first).

Acceptance:
  * layer 0, op by op (reference dump names): max |gpu - ref| / max |ref|
    <= L0_TOL per tensor -- before any amplification, only summation order
    and an occasional flipped bf16 rounding of a GEMM input separate them;
  * logits: max |gpu - ref| <= LOGIT_TOL (absolute; logits have std ~0.64).
    Every GEMM input is rounded to bf16 on both sides, so a last-bit
    difference from summation order flips some roundings (a 2^-8 step),
    which perturbs the next layer's inputs and flips more: over 28 layers
    the difference grows to the bf16 noise level of the activations.  The
    same growth separates the reference forward run with this plug-in's
    GEMMs from the same forward with kernels_hwsim (measured below), so the
    bound is set at that level, not at fp32 rounding;
  * greedy tokens: identical, except that a first divergence is accepted
    at a step whose reference top-2 margin is below TIE_TOL (a near tie
    that rounding may break either way); everything after it is then
    a different sequence and is not compared.
"""
import ctypes
import os

import numpy as np
import pytest

import oracle
from n550_qwen3_bringup_handover_amd import model as M
from n550_qwen3_bringup_handover_amd import runtime

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
L0_TOL = 1e-3
# measured worst differences: 1.1-1.36e-2 (prefill and decode steps, at
# positions up to 2047, alone and inside a 64-sequence batch); 1.5x that
LOGIT_TOL = 2e-2
TIE_TOL = 2 * LOGIT_TOL


def fixture(name):
    return np.load(os.path.join(GOLD, f"model_{name}.npz"))


def checksum(blob):
    return int(np.add.reduce(blob.view("<u8"), dtype=np.uint64))


def assert_tokens(got, fx, what):
    want, margins = fx["tokens"], fx["margins"]
    n = min(len(got), len(want))
    diff = np.nonzero(got[:n] != want[:n])[0]
    if len(diff) == 0:
        assert len(got) == len(want), f"{what}: {len(got)} tokens, want {len(want)}"
        return n
    j = int(diff[0])
    assert margins[j] < TIE_TOL, (f"{what}: token {j} is {got[j]}, reference {want[j]} "
                                  f"(reference margin {margins[j]:.3g} >= {TIE_TOL})")
    print(f"{what}: near-tie divergence at step {j} (margin {margins[j]:.3g})", flush=True)
    return j


@pytest.fixture(scope="module")
def blob():
    b = M.qw3m_random(int(fixture("short")["seed"]), M.LAYOUT_ROW, threads=16)
    assert checksum(b) == int(fixture("short")["checksum"])
    return b


@pytest.fixture(scope="module")
def model(blob):
    m = M.Model(blob, max_seq=512)
    yield m
    m.close()


def test_short_prefill_logits(model):
    fx = fixture("short")
    prompt = fx["prompt"]
    model.forward(prompt, 0)
    got = model.logits()
    ref = fx["prefill_logits"]
    err = np.abs(got.astype(np.float64) - ref)
    print(f"prefill logits: max abs err {err.max():.3e}, mean {err.mean():.3e}, "
          f"ref std {ref.std():.3f}", flush=True)
    assert np.all(np.isfinite(got))
    assert err.max() <= LOGIT_TOL
    assert model.argmax() == int(np.argmax(ref)) or fx["margins"][0] < TIE_TOL


def test_intermediates_op_by_op(model):
    d = np.load(os.path.join(GOLD, "model_short_dump.npz"))
    got = model.forward_dump(d["prompt"], 0)
    worst_l0 = 0.0
    keys = [k for k in d.files if "/" in k]
    for key in sorted(keys, key=lambda k: (int(k.split("/")[0][1:]), k)):
        layer, name = int(key.split("/")[0][1:]), key.split("/")[1]
        ref = d[key].astype(np.float64)
        g = got[(layer, name)]
        assert g.shape == ref.shape, key
        rel = float(np.abs(g - ref).max() / np.abs(ref).max())
        print(f"{key:28s} max|err|/max|ref| {rel:.2e}", flush=True)
        if layer == 0 or name == "embed_out":
            worst_l0 = max(worst_l0, rel)
            assert rel <= L0_TOL, key
    assert np.abs(got[(-1, "logits")] - d["L-1/logits"]).max() <= LOGIT_TOL
    print(f"worst layer-0 tensor: {worst_l0:.2e}", flush=True)


def test_short_greedy_tokens(model):
    fx = fixture("short")
    got = model.generate(fx["prompt"], len(fx["tokens"]) - 1)
    assert_tokens(got, fx, "short")


def test_p128_d128_greedy_tokens(model):
    fx = fixture("p128_d128")
    n_decode = len(fx["tokens"]) - 1
    got = model.generate(fx["prompt"], n_decode)
    pre, dec = model.timing()
    print(f"128-token prompt: prefill {len(fx['prompt'])} tokens {pre:.2f} ms, {n_decode} decode steps "
          f"{dec:.2f} ms = {n_decode / dec * 1e3:.1f} tok/s", flush=True)
    assert_tokens(got, fx, "p128_d128")


def test_graph_and_eager_decode_agree(model):
    fx = fixture("short")
    n = len(fx["tokens"]) - 1
    model.set_graph(True)
    a = model.generate(fx["prompt"], n)
    la = model.logits()
    model.set_graph(False)
    try:
        b = model.generate(fx["prompt"], n)
        lb = model.logits()
    finally:
        model.set_graph(True)
    assert np.array_equal(a, b)
    assert np.array_equal(la, lb)     # same kernels, same order: bit-identical


def test_forward_api_steps_like_generate(model):
    fx = fixture("short")
    prompt, tokens = fx["prompt"], fx["tokens"]
    model.forward(prompt, 0)
    assert model.argmax() == tokens[0]
    for i in range(3):
        model.forward([tokens[i]], len(prompt) + i)
        assert model.argmax() == tokens[i + 1] or fx["margins"][i + 1] < TIE_TOL


def test_chunked_prefill_matches_two_calls(model):
    # 130 tokens: generate() prefills in one pass; forward() in 64 + 66 (several
    # passes of generate(): test_prefill_passes_gpu)
    rng = np.random.default_rng(1)
    prompt = rng.integers(0, M.VOCAB, 130).astype(np.int32)
    g = model.generate(prompt, 0)
    lg = model.logits()
    model.forward(prompt[:64], 0)
    model.forward(prompt[64:], 64)
    lf = model.logits()
    err = np.abs(lg.astype(np.float64) - lf).max()
    print(f"130 in one pass vs 64+66: max abs logit diff {err:.3e}", flush=True)
    assert err <= LOGIT_TOL
    top2 = np.sort(lf)[-2:]
    assert g[0] == int(np.argmax(lf)) or top2[1] - top2[0] < TIE_TOL


def test_tile_layout_blob_gives_identical_results(blob, model):
    fx = fixture("short")
    tb = M.qw3m_random(int(fx["seed"]), M.LAYOUT_TILE, threads=16)
    with M.Model(tb, max_seq=model.max_seq) as mt:
        a = mt.generate(fx["prompt"], 4)
        la = mt.logits()
    b = model.generate(fx["prompt"], 4)
    lb = model.logits()
    assert np.array_equal(a, b)
    assert np.array_equal(la, lb)     # identical device weights after re-tiling


def test_errors(blob, model):
    bad = blob[:4096].copy()
    with pytest.raises(M.Qwen3ModelError, match="size"):
        M.Model(bad)
    saved = blob[:4].copy()
    blob[:4] = np.frombuffer(b"XW3M", np.uint8)
    try:
        with pytest.raises(M.Qwen3ModelError, match="magic"):
            M.Model(blob)
    finally:
        blob[:4] = saved
    with pytest.raises(runtime.Qwen3HipError):
        model.generate([1, 2, 3], model.max_seq)                 # past the KV cache
    with pytest.raises(runtime.Qwen3HipError):
        model.generate([1, M.VOCAB], 1)                          # token out of range
    with pytest.raises(runtime.Qwen3HipError):
        model.forward(np.zeros(129, np.int32), 0)                # > 128 tokens per call
    with pytest.raises(runtime.Qwen3HipError):
        model.forward([1], model.max_seq)                        # position past the cache
    with pytest.raises(runtime.Qwen3HipError):
        M.Model(blob, max_seq=9000)


def _ref_hip():
    L = oracle.ref("ref_model_hip")
    if L is None:
        pytest.skip("oracle/_ref/libref_model_hip.so not built")
    L.refdrv_generate.restype = ctypes.c_int
    L.refdrv_generate.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.POINTER(ctypes.c_int),
                                  ctypes.c_int, ctypes.c_int, ctypes.c_int,
                                  ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_float),
                                  ctypes.POINTER(ctypes.c_float)]
    return L


@pytest.mark.parametrize("case", ["short", "p128_d128"])
def test_reference_forward_with_gpu_plugin(blob, case):
    """The reference's own forward (qwen3.c + ops_scalar.c) linked with this
    plug-in as its KERNEL: every GEMM of the forward goes through qwen3_gemm /
    qwen3_gemm_row on the GPU; its greedy tokens must match the same forward
    with the reference's RTL-numerics kernel."""
    L = _ref_hip()
    fx = fixture(case)
    prompt = np.ascontiguousarray(fx["prompt"], dtype=np.int32)
    n_decode = len(fx["tokens"]) - 1
    out = np.zeros(n_decode + 1, np.int32)
    margins = np.zeros(n_decode + 1, np.float32)
    logits = np.zeros(M.VOCAB, np.float32)
    n = L.refdrv_generate(blob.ctypes.data_as(ctypes.c_void_p), blob.nbytes,
                          prompt.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), len(prompt), n_decode, 0,
                          out.ctypes.data_as(ctypes.POINTER(ctypes.c_int)),
                          margins.ctypes.data_as(ctypes.POINTER(ctypes.c_float)),
                          logits.ctypes.data_as(ctypes.POINTER(ctypes.c_float)))
    assert n == n_decode + 1
    assert_tokens(out, fx, f"reference forward + plug-in ({case})")
    if "prefill_logits" in fx:
        err = np.abs(logits.astype(np.float64) - fx["prefill_logits"]).max()
        print(f"reference forward + plug-in: prefill logits max abs err {err:.3e}", flush=True)
        assert err <= LOGIT_TOL


# ---- multi-sequence batched decode (qwen3_hip_batch_*) ----------------------

def _batch_cases():
    """(prompt, tokens, margins) per sequence: the three batch prompts and
    the short and 128-token prompts, interleaved so prompt lengths are ragged."""
    fb = fixture("batch")
    lens = fb["prompt_lens"]
    starts = np.concatenate([[0], np.cumsum(lens)])
    extra = [(fb["prompts"][starts[i]:starts[i + 1]], fb["tokens"][i], fb["margins"][i]) for i in range(len(lens))]
    fs, fc = fixture("short"), fixture("p128_d128")
    return [extra[0], (fs["prompt"], fs["tokens"], fs["margins"]), extra[1],
            (fc["prompt"], fc["tokens"], fc["margins"]), extra[2]]


def _check_row(got, want, margins, what):
    n = min(len(got), len(want))
    diff = np.nonzero(got[:n] != want[:n])[0]
    if len(diff) == 0:
        return n
    j = int(diff[0])
    assert margins[j] < TIE_TOL, (f"{what}: token {j} is {got[j]}, reference {want[j]} "
                                  f"(reference margin {margins[j]:.3g} >= {TIE_TOL})")
    print(f"{what}: near-tie divergence at step {j} (margin {margins[j]:.3g})", flush=True)
    return j


def test_batch_decode_matches_reference(model):
    """Five sequences with prompts of 1, 5, 19, 128 and 40 tokens decoded
    together: every sequence's greedy tokens equal the reference forward's
    for that prompt alone."""
    cases = _batch_cases()
    n_dec = 8
    with M.Batch(model, len(cases), 160) as b:
        for s, (p, _, _) in enumerate(cases):
            b.prefill(s, p)
        out = b.decode(n_dec)
        ms = b.timing()
    print(f"batch of {len(cases)}: {n_dec} steps {ms:.2f} ms", flush=True)
    for s, (p, want, mg) in enumerate(cases):
        _check_row(out[s], want[:n_dec + 1], mg, f"batch seq {s} (prompt {len(p)})")


def _forward_all(model, seq):
    """Single-sequence forward of seq from position 0, in calls of <= 128."""
    for p0 in range(0, len(seq), 128):
        model.forward(seq[p0:p0 + 128], p0)


def test_batch_logits_match_single_sequence_forward(model):
    """Batch logits after k steps equal the single-sequence forward of the
    prompt plus the k fed tokens (its last row), within LOGIT_TOL."""
    cases = _batch_cases()
    n_dec = 6
    with M.Batch(model, len(cases), 160) as b:
        for s, (p, _, _) in enumerate(cases):
            b.prefill(s, p)
        out = b.decode(n_dec)
        lb = b.logits()
    worst = 0.0
    for s, (p, _, _) in enumerate(cases):
        _forward_all(model, np.concatenate([p, out[s, :n_dec]]))
        ls = model.logits()
        err = float(np.abs(ls.astype(np.float64) - lb[s]).max())
        worst = max(worst, err)
        assert err <= LOGIT_TOL, f"seq {s}: max abs logit diff {err:.3e}"
    print(f"batch vs single-sequence forward: worst max abs logit diff {worst:.3e}", flush=True)


def test_batch_split_calls_graph_and_eager_agree(model):
    """Two decode calls of 4 steps continue exactly like one call of 8, and
    graph replay equals eager launches bit for bit (same kernels, same order)."""
    cases = _batch_cases()
    res = {}
    for mode in ("graph", "eager"):
        with M.Batch(model, len(cases), 160) as b:
            b.set_graph(mode == "graph")
            for s, (p, _, _) in enumerate(cases):
                b.prefill(s, p)
            a = b.decode(4)
            c = b.decode(4)
            res[mode] = (np.concatenate([a, c[:, 1:]], axis=1), b.logits())
            assert np.array_equal(a[:, -1], c[:, 0])
    with M.Batch(model, len(cases), 160) as b:
        for s, (p, _, _) in enumerate(cases):
            b.prefill(s, p)
        one = b.decode(8)
        l_one = b.logits()
    assert np.array_equal(res["graph"][0], one)
    assert np.array_equal(res["graph"][1], l_one)
    assert np.array_equal(res["eager"][0], one)
    assert np.array_equal(res["eager"][1], l_one)


def test_batch_reprefill_one_sequence(model):
    """Re-prefilling one sequence restarts it while the others continue."""
    cases = _batch_cases()
    fc = fixture("p128_d128")
    with M.Batch(model, len(cases), 160) as b:
        for s, (p, _, _) in enumerate(cases):
            b.prefill(s, p)
        first = b.decode(3)
        b.prefill(1, cases[0][0])                 # sequence 1 now holds prompt 0
        second = b.decode(5)
    # the 128-token prompt (sequence 3) continues: its 9 tokens over both calls
    cont = np.concatenate([first[3], second[3, 1:]])
    _check_row(cont, fc["tokens"][:9], fc["margins"], "128-token prompt continued")
    _check_row(second[1], cases[0][1][:6], cases[0][2], "re-prefilled seq 1")
    _check_row(np.concatenate([first[0], second[0, 1:]]), cases[0][1][:9], cases[0][2], "seq 0 continued")


def test_batch_64_duplicate_sequences_identical(model):
    """64 sequences of ragged random prompts (1 .. 300 tokens), each prompt
    used twice (sequences i and i + 32): the two copies of a prompt produce
    bit-identical tokens and logits (each output row of every kernel depends
    on its own row only), and a sample matches the single-sequence forward."""
    rng = np.random.default_rng(64)
    lens = rng.integers(1, 301, 32)
    prompts = [rng.integers(0, M.VOCAB, n).astype(np.int32) for n in lens]
    n_dec = 4
    with M.Batch(model, 64, 320) as b:
        for s in range(64):
            b.prefill(s, prompts[s % 32])
        out = b.decode(n_dec)
        lb = b.logits()
        ms = b.timing()
    print(f"batch of 64 (prompts 1..300): {n_dec} steps {ms:.2f} ms", flush=True)
    assert np.array_equal(out[:32], out[32:])
    assert np.array_equal(lb[:32], lb[32:])
    for s in (int(np.argmax(lens)), int(np.argmin(lens)), 7):
        _forward_all(model, np.concatenate([prompts[s], out[s, :n_dec]]))
        err = float(np.abs(model.logits().astype(np.float64) - lb[s]).max())
        assert err <= LOGIT_TOL, f"seq {s} (prompt {lens[s]}): max abs logit diff {err:.3e}"


def test_batch_errors(model):
    with pytest.raises(runtime.Qwen3HipError):
        M.Batch(model, 0, 64)
    with pytest.raises(runtime.Qwen3HipError):
        M.Batch(model, 129, 64)
    with pytest.raises(runtime.Qwen3HipError):
        M.Batch(model, 2, model.max_seq + 1)
    with M.Batch(model, 2, 16) as b:
        with pytest.raises(runtime.Qwen3HipError):
            b.decode(1)                            # nothing prefilled
        b.prefill(0, [1, 2, 3])
        with pytest.raises(runtime.Qwen3HipError):
            b.decode(1)                            # sequence 1 not prefilled
        with pytest.raises(runtime.Qwen3HipError):
            b.prefill(2, [1])                      # no sequence 2
        with pytest.raises(runtime.Qwen3HipError):
            b.prefill(1, np.arange(16))            # prompt fills the whole context
        with pytest.raises(runtime.Qwen3HipError):
            b.prefill(1, [M.VOCAB])                # token out of range
        with pytest.raises(runtime.Qwen3HipError):
            b.logits()                             # no decode step yet
        b.prefill(1, np.arange(10))
        b.decode(6)                                # sequence 1 reaches position 15
        with pytest.raises(runtime.Qwen3HipError):
            b.decode(1)                            # past max_ctx for sequence 1


def test_batch_after_model_close_is_refused(blob):
    """Closing the model first takes the batch's graph down with it; the
    batch's later calls are refused instead of touching freed memory."""
    with M.Model(blob, max_seq=64) as m:
        b = M.Batch(m, 2, 32)
        b.prefill(0, [1, 2, 3])
        b.prefill(1, [4, 5])
        out = b.decode(3)                      # captures the step graph
        assert out.shape == (2, 4)
    try:
        with pytest.raises(runtime.Qwen3HipError, match="state"):
            b.decode(1)
        with pytest.raises(runtime.Qwen3HipError, match="state"):
            b.prefill(0, [1])
    finally:
        b.close()


@pytest.mark.parametrize("n_seq", [1, 128])
def test_batch_size_limits(model, n_seq):
    """The smallest batch (every projection an M = 1 GEMV) and the largest
    (M = 128 GEMMs): each sequence's logits after a few steps equal the
    single-sequence forward of its prompt plus the fed tokens."""
    rng = np.random.default_rng(100 + n_seq)
    lens = rng.integers(1, 40, n_seq)
    prompts = [rng.integers(0, M.VOCAB, n).astype(np.int32) for n in lens]
    n_dec = 3
    with M.Batch(model, n_seq, 48) as b:
        for s in range(n_seq):
            b.prefill(s, prompts[s])
        out = b.decode(n_dec)
        lb = b.logits()
    assert out.shape == (n_seq, n_dec + 1)
    assert np.all((out >= 0) & (out < M.VOCAB))
    for s in sorted({0, n_seq // 2, n_seq - 1}):
        _forward_all(model, np.concatenate([prompts[s], out[s, :n_dec]]))
        ls = model.logits()
        err = float(np.abs(ls.astype(np.float64) - lb[s]).max())
        assert err <= LOGIT_TOL, f"n_seq {n_seq}, seq {s}: max abs logit diff {err:.3e}"
        assert out[s, n_dec] == int(np.argmax(lb[s]))


def test_longest_context(blob):
    """max_seq = 8192, the largest cache: an 8,180-token prompt prefilled in
    four passes of 2,045 and in chunks of 100 gives the same last logits
    within LOGIT_TOL; 11 decode steps to position 8190
    follow, and the last step's logits equal a forward of the whole
    sequence."""
    rng = np.random.default_rng(8192)
    prompt = rng.integers(0, M.VOCAB, 8180).astype(np.int32)
    with M.Model(blob, max_seq=8192) as m:
        toks = m.generate(prompt, 11)                 # prefill in four passes, then 11 steps
        l_gen = m.logits()
        assert len(toks) == 12 and np.all((toks >= 0) & (toks < M.VOCAB))
        for p0 in range(0, len(prompt), 100):        # other chunk boundaries
            m.forward(prompt[p0:p0 + 100], p0)
        l100 = m.logits()
        top2 = np.sort(l100)[-2:]
        assert toks[0] == int(np.argmax(l100)) or top2[1] - top2[0] < TIE_TOL
        seq = np.concatenate([prompt, toks[:11]])    # the 11 fed tokens, last at position 8190
        for p0 in range(8180, len(seq), 128):
            m.forward(seq[p0:p0 + 128], p0)
        l_fwd = m.logits()
    err = float(np.abs(l_fwd.astype(np.float64) - l_gen).max())
    print(f"context 8191: decode vs forward max abs logit diff {err:.3e}", flush=True)
    assert err <= LOGIT_TOL


def _logits_err(got, ref):
    return float(np.abs(got.astype(np.float64) - ref.astype(np.float64)).max())


def test_p128_d128_decode_step_logits(model):
    """The 128-token prompt, then the reference's own tokens fed one decode
    step at a time: the logits after decode steps 1, 32, 64 and 128 against
    the reference's (model_p128_d128_logits.npz), not only the tokens."""
    fx = fixture("p128_d128_logits")
    prompt, toks = fx["prompt"], fx["tokens"]
    _forward_all(model, prompt)
    worst = _logits_err(model.logits(), fx["prefill_logits"])
    assert worst <= LOGIT_TOL
    steps = [int(s) for s in fx["log_steps"]]
    for i in range(1, max(steps) + 1):
        model.forward([toks[i - 1]], len(prompt) + i - 1)
        if i in steps:
            err = _logits_err(model.logits(), fx["step_logits"][steps.index(i)])
            print(f"decode step {i}: max abs logit diff {err:.3e}", flush=True)
            worst = max(worst, err)
            assert err <= LOGIT_TOL, (i, err)
    print(f"p128_d128 decode-step logits: worst {worst:.3e}", flush=True)


@pytest.fixture(scope="module")
def long_model(blob):
    m = M.Model(blob, max_seq=2048)
    yield m
    m.close()


def test_long_context_matches_reference(long_model):
    """A 1,100-token prompt against the reference forward built with its own
    2048-position cache (qwen3.c with -DQWEN3_MAX_SEQ=2048): the last prefill
    row's logits, the logits after decode steps 1, 4 and 8 (the reference's
    tokens fed), and the greedy tokens -- RoPE angles, the cache layout and
    both attention kernels past position 1024 pinned to the reference."""
    fx = fixture("long")
    prompt, toks = fx["prompt"], fx["tokens"]
    m = long_model
    _forward_all(m, prompt)
    err = _logits_err(m.logits(), fx["prefill_logits"])
    print(f"1100-token prefill: max abs logit diff {err:.3e}", flush=True)
    assert err <= LOGIT_TOL
    assert m.argmax() == toks[0] or fx["margins"][0] < TIE_TOL
    steps = [int(s) for s in fx["log_steps"]]
    for i in range(1, max(steps) + 1):
        m.forward([toks[i - 1]], len(prompt) + i - 1)
        if i in steps:
            err = _logits_err(m.logits(), fx["step_logits"][steps.index(i)])
            print(f"decode step {i} (position {len(prompt) + i - 1}): max abs logit diff {err:.3e}", flush=True)
            assert err <= LOGIT_TOL, (i, err)
    got = m.generate(prompt, len(toks) - 1)
    assert_tokens(got, fx, "long")


def test_long_context_inside_a_batch(long_model):
    """The same 1,100-token prompt as sequence 1 of a batch of three (the
    others short): its greedy tokens equal the reference's, and its logits
    after the eighth decode step equal the reference's step-8 logits."""
    fx = fixture("long")
    fb = fixture("batch")
    lens = [int(v) for v in fb["prompt_lens"]]
    short0 = fb["prompts"][:lens[0]]
    short2 = fb["prompts"][lens[0]:lens[0] + lens[1]]
    n_dec = len(fx["tokens"]) - 1
    with M.Batch(long_model, 3, 1200) as b:
        b.prefill(0, short0)
        b.prefill(1, fx["prompt"])
        b.prefill(2, short2)
        out = b.decode(n_dec)
        lb = b.logits()
    j = _check_row(out[1], fx["tokens"], fx["margins"], "batch seq 1 (1100-token prompt)")
    if j == len(fx["tokens"]):
        steps = [int(s) for s in fx["log_steps"]]
        err = _logits_err(lb[1], fx["step_logits"][steps.index(n_dec)])
        print(f"batch seq 1, decode step {n_dec}: max abs logit diff {err:.3e}", flush=True)
        assert err <= LOGIT_TOL


def test_ctx2048_matches_reference(long_model):
    """Positions 2,014-2,047 against the reference forward built with its own
    2048-position cache (model_ctx2048.npz: the prompt of sequence 0 of the
    64-sequence batched-decode workload, 2,014 tokens, then 34 greedy steps
    to position 2047).  Logits of the last prefill row and after decode steps
    1, 2, 3, 8, 16 and 34 with the reference's tokens fed -- compared at every
    logged step, whatever the greedy tokens do -- then the greedy tokens
    themselves under the near-tie rule."""
    fx = fixture("ctx2048")
    prompt, toks = fx["prompt"], fx["tokens"]
    m = long_model
    _forward_all(m, prompt)
    worst = _logits_err(m.logits(), fx["prefill_logits"])
    print(f"2014-token prefill: max abs logit diff {worst:.3e}", flush=True)
    assert worst <= LOGIT_TOL
    steps = [int(s) for s in fx["log_steps"]]
    for i in range(1, max(steps) + 1):
        m.forward([toks[i - 1]], len(prompt) + i - 1)
        if i in steps:
            err = _logits_err(m.logits(), fx["step_logits"][steps.index(i)])
            print(f"decode step {i} (position {len(prompt) + i - 1}): max abs logit diff {err:.3e}", flush=True)
            worst = max(worst, err)
            assert err <= LOGIT_TOL, (i, err)
    print(f"ctx2048 logits: worst {worst:.3e}", flush=True)
    got = m.generate(prompt, len(toks) - 1)
    assert_tokens(got, fx, "ctx2048")


def test_ctx2048_inside_64_sequence_batch(long_model):
    """The batched-decode workload's own geometry: 64 sequences at max_ctx
    2048, each prefilled with a 2,014-token prompt drawn from numpy's
    default_rng(5) in sequence order (sequence 0 is the ctx2048 fixture's
    prompt), then greedy steps to position 2047.  Sequence 0's logits after
    decode step 1 are compared with the reference's unconditionally (the
    token fed there is the prefill's argmax, reference margin 0.07), those
    after steps 2 and 3 while its tokens still equal the reference's, and
    its greedy tokens under the near-tie rule."""
    fx = fixture("ctx2048")
    n_seq, ctx, n_prompt = 64, 2048, 2014
    rng = np.random.default_rng(5)
    prompts = [rng.integers(0, M.VOCAB, n_prompt).astype(np.int32) for _ in range(n_seq)]
    assert np.array_equal(prompts[0], fx["prompt"])
    toks, margins = fx["tokens"], fx["margins"]
    steps = [int(s) for s in fx["log_steps"]]
    n_dec = len(toks) - 1
    got = [None]
    with M.Batch(long_model, n_seq, ctx) as b:
        for s in range(n_seq):
            b.prefill(s, prompts[s])
        for i in (1, 2, 3):
            out = b.decode(1)
            got[-1:] = [int(out[0, 0]), int(out[0, 1])]
            lb = b.logits()
            if i == 1:
                assert got[0] == toks[0] or margins[0] < TIE_TOL
            if got[:i] == [int(t) for t in toks[:i]]:      # the tokens fed so far are the reference's
                err = _logits_err(lb[0], fx["step_logits"][steps.index(i)])
                print(f"batch of 64, seq 0, decode step {i} (position {n_prompt + i - 1}): "
                      f"max abs logit diff {err:.3e}", flush=True)
                assert err <= LOGIT_TOL, (i, err)
            else:
                assert i > 1
        out = b.decode(n_dec - 3)
        got += [int(t) for t in out[0, 1:]]
        # every other sequence decoded to position 2047 too
        assert np.all((out >= 0) & (out < M.VOCAB))
    j = _check_row(np.array(got, np.int32), toks, margins, "batch of 64, seq 0 (ctx2048)")
    print(f"batch of 64, seq 0: {j} of {len(toks)} tokens equal the reference's", flush=True)
