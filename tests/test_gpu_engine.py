"""GPU engine parity against the oracle on small models of each config family.

Bars (north star): logits within 1e-3 (max-abs, normalised by max(1, max|logit|)); greedy token streams and speculative accept
counts identical, except at logit near-ties (top-2 margin < 1e-4 in the oracle), which are
reported; a row's results are bitwise identical whether it runs alone or inside a batch.
Final hidden states are held to 1e-2: an integer-path projection re-quantizes its input to
8 bits, so a last-bit difference upstream can move one Q8_K code by one step (the reference
notes the same amplification, smollm_chat.rs:4775-4777)."""
import numpy as np
import pytest

from spindle_amd import model as M
from oracle.model import OracleModel
from tests import layer_pins as LP

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

FAMILIES = ["tiny-llama", "tiny-qwen3", "tiny-granite", "tiny-qwen3moe", "tiny-q5k", "tiny-a3b"]


@pytest.fixture(scope="module")
def ctx():
    from spindle_amd import ops
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = ops.Context(0)
    yield c
    c.close()


def _norm_err(a, b):
    return float(np.max(np.abs(a.astype(np.float64) - b.astype(np.float64))) / max(1.0, float(np.max(np.abs(b)))))


def _margin(logits):
    top = np.sort(logits.astype(np.float64))[-2:]
    return top[1] - top[0]


@pytest.mark.parametrize("name", FAMILIES)
def test_forward_matches_oracle(ctx, name):
    """Teacher-forced per-step parity: the GPU prefills 16 rows, then for each one-token step
    the oracle gets the GPU's KV cache, so both compute the same pass on the same context.
    (Multi-row passes are covered transitively: GPU batch == GPU sequential and oracle batch
    == oracle sequential, both bitwise.) Models without integer-path matrices must hold
    logits <= 1e-3 on every step. Integer-path matrices re-quantize activations to Q8_K:
    when a last-bit difference (reduction order of a norm or softmax) moves an activation
    across a rounding boundary, one code changes by one step and the step's logits move by up
    to a few 1e-2; such a step is traced layer by layer (tests/layer_pins.py: every stage
    pinned, every moved code a single step), and the median step stays <= 1e-5."""
    cfg = M.TINY[name].replace(sigma=0.05)
    w = M.synth_model(cfg, seed=11)
    eng = M.Engine(ctx, cfg, w)
    om = OracleModel(cfg, w)
    rng = np.random.default_rng(1)
    ids = rng.integers(0, cfg.vocab, 56)
    integer = any(getattr(cfg, "t_" + t) in (M.Q4K, M.Q6K) for t in ("q", "k", "v", "o", "gate", "up", "down", "out"))
    eng.forward(ids[:16], 0)
    errs, flips = [], 0
    for pos in range(16, len(ids)):
        k, v = eng.kv_cache()
        om.k_cache[:] = k
        om.v_cache[:] = v
        am, hid, lg = eng.forward(ids[pos:pos + 1], pos, hidden=True, logits=True)
        l_or = om.logits(om.forward(ids[pos:pos + 1], pos))
        e = _norm_err(lg[0], l_or[0])
        errs.append(e)
        if e > 1e-3:
            assert integer and eng.decode_pipeline(), (name, pos, e)

            def sync():
                kk, vv = eng.kv_cache()
                om.k_cache[:] = kk
                om.v_cache[:] = vv
            LP.report(name, f"step at {pos} ({e:.1e})", LP.layer_pins(eng, om, cfg, ids[pos:pos + 1], pos, sync, name))
            flips += 1
        want = om.argmax(l_or[0])
        if am[0] != want:
            assert _margin(l_or[0] / cfg.logit_scale) < max(1e-4, 2 * e), (name, pos)
            print(f"argmax differs at {name} pos {pos} (margin within the step's error)")
    print(f"{name}: {len(errs)} steps, logits err median {np.median(errs):.1e} max {max(errs):.1e}, steps traced to Q8_K steps {flips}")
    assert np.median(errs) <= 1e-5
    eng.close()


@pytest.mark.parametrize("name", FAMILIES)
def test_batch_equals_sequential_bitwise(ctx, name):
    cfg = M.TINY[name].replace(sigma=0.05)
    w = M.synth_model(cfg, seed=12)
    a, b = M.Engine(ctx, cfg, w), M.Engine(ctx, cfg, w)
    a.set_mfma(False)  # lane-exact multi-row kernels (the int8 matrix-core path rounds differently)
    b.set_mfma(False)
    rng = np.random.default_rng(2)
    ids = rng.integers(0, cfg.vocab, 13)
    a.forward(ids[:4], 0)
    b.forward(ids[:4], 0)
    _, hb, lb = a.forward(ids[4:13], 4, hidden=True, logits=True)
    for i in range(9):
        _, hs, ls = b.forward(ids[4 + i:5 + i], 4 + i, hidden=True, logits=True)
        assert np.array_equal(hs[0].view(np.uint32), hb[i].view(np.uint32)), (name, i)
        assert np.array_equal(ls[0].view(np.uint32), lb[i].view(np.uint32)), (name, i)


@pytest.mark.parametrize("name", ["tiny-a3b", "tiny-qwen3", "tiny-qwen3moe"])
def test_batch_equals_sequential_long_context(ctx, name):
    """Past 1024 positions (17+ attention chunks, two merge levels) a verify pass of 9 rows,
    whose queries span several 16-query tiles, still gives each row the bits of its one-row
    pass: the chunking and merge order do not depend on the pass size."""
    cfg = M.TINY[name].replace(sigma=0.05, max_seq=1280)
    w = M.synth_model(cfg, seed=16)
    a, b = M.Engine(ctx, cfg, w), M.Engine(ctx, cfg, w)
    a.set_mfma(False)
    b.set_mfma(False)
    ids = np.random.default_rng(3).integers(0, cfg.vocab, 1120)
    for s0 in range(0, 1100, 16):
        a.forward(ids[s0:min(s0 + 16, 1100)], s0)
        b.forward(ids[s0:min(s0 + 16, 1100)], s0)
    _, hb, lb = a.forward(ids[1100:1109], 1100, hidden=True, logits=True)
    for i in range(9):
        _, hs, ls = b.forward(ids[1100 + i:1101 + i], 1100 + i, hidden=True, logits=True)
        assert np.array_equal(hs[0].view(np.uint32), hb[i].view(np.uint32)), (name, i)
        assert np.array_equal(ls[0].view(np.uint32), lb[i].view(np.uint32)), (name, i)
    a.close()
    b.close()


SHAPES = {"tiles at decode": {"SPX_MV_MODE": "0"}, "standalone norms": {"SPX_TAIL_MAX": "0"},
          "tails at every m": {"SPX_TAIL_MAX": "16"}, "row-parallel LM head": {"SPX_LM_MODE": "1"}}


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("name", ["tiny-qwen3", "tiny-qwen3moe"])
def test_launch_shapes_bitwise(ctx, name, shape, monkeypatch):
    """Every launch shape (row-parallel or tiled matvecs, norm tails or standalone norm
    launches, LM head shape) gives the same bits for the same pass."""
    cfg = M.TINY[name].replace(sigma=0.05)
    w = M.synth_model(cfg, seed=14)
    ref = M.Engine(ctx, cfg, w)
    for k, v in SHAPES[shape].items():
        monkeypatch.setenv(k, v)
    eng = M.Engine(ctx, cfg, w)
    for k in SHAPES[shape]:
        monkeypatch.delenv(k)
    ids = np.arange(30) * 5 % cfg.vocab
    pos = 0
    for m in (5, 1, 2, 1, 9, 2):
        a0, h0, l0 = ref.forward(ids[pos:pos + m], pos, hidden=True, logits=True)
        a1, h1, l1 = eng.forward(ids[pos:pos + m], pos, hidden=True, logits=True)
        assert np.array_equal(h0.view(np.uint32), h1.view(np.uint32)), (shape, m)
        assert np.array_equal(l0.view(np.uint32), l1.view(np.uint32)), (shape, m)
        assert np.array_equal(a0, a1), (shape, m)
        pos += m
    ref.close()
    eng.close()


@pytest.mark.parametrize("graphs", [True, False])
def test_graph_replay_matches_eager(ctx, graphs):
    cfg = M.TINY["tiny-qwen3moe"]
    w = M.synth_model(cfg, seed=13)
    ref = M.Engine(ctx, cfg, w, graphs=False)
    eng = M.Engine(ctx, cfg, w, graphs=graphs)
    ids = np.arange(40) * 7 % cfg.vocab
    for s in range(0, 40, 8):
        _, h0, _ = ref.forward(ids[s:s + 8], s, hidden=True)
        for rep in range(2):        # replay the same pass twice (graph replays after the first)
            _, h1, _ = eng.forward(ids[s:s + 8], s, hidden=True)
            assert np.array_equal(h0.view(np.uint32), h1.view(np.uint32)), (s, rep)


@pytest.mark.parametrize("name", ["tiny-qwen3moe", "tiny-llama"])
def test_decode_back_to_back_matches_single_passes(ctx, name):
    """spx_engine_decode replays one-row passes back to back with the pick fed forward on the
    device; it must pick what separate one-token passes pick."""
    cfg = M.TINY[name].replace(sigma=0.05)
    w = M.synth_model(cfg, seed=15)
    a, b = M.Engine(ctx, cfg, w), M.Engine(ctx, cfg, w)
    ids = np.arange(12) * 11 % cfg.vocab
    a.forward(ids, 0)
    b.forward(ids, 0)
    got = a.decode(int(ids[-1]), 12, 20)
    tok, want = int(ids[-1]), []
    for i in range(20):
        am, _, _ = b.forward([tok], 12 + i)
        tok = int(am[0])
        want.append(tok)
    assert got.tolist() == want
    # and the caches agree afterwards
    ka, va = a.kv_cache()
    kb, vb = b.kv_cache()
    assert np.array_equal(ka, kb) and np.array_equal(va, vb)
    a.close()
    b.close()


def _spec_prompt(vocab, seed):
    """BASELINE.json config 3's construction at small size: random tokens, then copied spans
    of 16..64 tokens from the first half interleaved with 10% random tokens."""
    rng = np.random.default_rng(seed)
    head = rng.integers(0, vocab, 64)
    tail = []
    while len(tail) < 64:
        ln = int(rng.integers(16, 65))
        s = int(rng.integers(0, 64 - 16))
        for t in head[s:s + ln]:
            tail.append(int(rng.integers(0, vocab)) if rng.random() < 0.1 else int(t))
    return np.concatenate([head, np.array(tail[:64])]).astype(np.int32)


@pytest.mark.parametrize("name", ["tiny-llama", "tiny-qwen3", "tiny-granite"])
def test_generate_matches_oracle(ctx, name):
    """Greedy stream and accept counts vs the oracle (benchmark mode: n-gram 3, k=8, fixed) on
    the float-activation families, where no activation is re-quantized between passes."""
    cfg = M.TINY[name].replace(sigma=0.06)
    w = M.synth_model(cfg, seed=21)
    prompt = _spec_prompt(cfg.vocab, 3)
    eng = M.Engine(ctx, cfg, w)
    g_tok, g_st = eng.generate(prompt, 48, draft_len=8, min_ngram=3, max_ngram=3, fixed=True)
    o_tok, o_st = OracleModel(cfg, w).generate(prompt, 48, draft_len=8, min_ngram=3, max_ngram=3, fixed=True)
    if not np.array_equal(g_tok, o_tok):
        i = int(np.argmax(g_tok != o_tok))
        om = OracleModel(cfg, w)
        seq = np.concatenate([prompt, o_tok[:i]])
        h = np.concatenate([om.forward(seq[s:s + 16], s) for s in range(0, len(seq), 16)])
        lg = om.logits(h[-1:])[0] / cfg.logit_scale
        assert _margin(lg) < 1e-4, (name, i, g_tok[:i + 2], o_tok[:i + 2])
        print(f"{name}: streams diverge at {i} on a near-tie (margin {_margin(lg):.2e})")
    else:
        for k in ("accepted", "drafted", "verifies", "steps"):
            assert g_st[k] == o_st[k], (k, g_st, o_st)
    eng.close()


@pytest.mark.parametrize("name", FAMILIES)
@pytest.mark.parametrize("mode", ["lane", "matrix"])
def test_speculation_is_exact_on_gpu(ctx, name, mode, monkeypatch):
    """prompt_lookup_speculation_is_exact (:4798-4825): spec on == spec off, bit for bit, with the
    verify passes on the lane kernels and on the int8 matrix cores (forced from two rows for
    every projection; the default thresholds leave small passes on the lane kernels)."""
    cfg = M.TINY[name].replace(sigma=0.06)
    if mode == "matrix" and not all(t in (M.Q4K, M.Q6K) for t in (cfg.t_q, cfg.t_k, cfg.t_v, cfg.t_o, cfg.t_gate, cfg.t_up, cfg.t_down)):
        pytest.skip("float formats: the bf16 matrix cores sum in an order of their own (logits within 1e-3), not the one-row bits")
    w = M.synth_model(cfg, seed=22)
    prompt = _spec_prompt(cfg.vocab, 4)
    if mode == "matrix":
        monkeypatch.setenv("SPX_MQ_ROWS", "2,2,2,2,2")
    eng = M.Engine(ctx, cfg, w)
    if mode == "lane":
        eng.set_mfma(False)  # lane-exact verify passes: the same bits as one-row passes
    off, _ = eng.generate(prompt, 48, speculate=False)
    for (lo, hi, k, fixed) in [(2, 4, 4, False), (3, 3, 8, True), (2, 4, 15, True)]:
        on, st = eng.generate(prompt, 48, draft_len=k, min_ngram=lo, max_ngram=hi, fixed=fixed)
        assert np.array_equal(off, on), (lo, hi, k)
    eng.close()


@pytest.mark.parametrize("name", ["tiny-qwen3moe", "tiny-a3b"])
def test_speculation_on_matrix_cores(ctx, name):
    """Verify passes on the int8 matrix cores (the default for K-quant models) give one-row
    passes' bits, so speculative generation with the default settings equals plain greedy
    decoding bit for bit (prompt_lookup_speculation_is_exact :4798-4825)."""
    cfg = M.TINY[name].replace(sigma=0.06)
    w = M.synth_model(cfg, seed=22)
    prompt = _spec_prompt(cfg.vocab, 4)
    eng = M.Engine(ctx, cfg, w)
    assert eng.decode_pipeline()
    off, _ = eng.generate(prompt, 48, speculate=False)
    for (lo, hi, k, fixed) in [(2, 4, 4, False), (3, 3, 8, True), (2, 4, 15, True)]:
        on, st = eng.generate(prompt, 48, draft_len=k, min_ngram=lo, max_ngram=hi, fixed=fixed)
        assert st["verifies"] > 0
        assert np.array_equal(off, on), (name, lo, hi, k)
    eng.close()


@pytest.mark.parametrize("name", ["tiny-qwen3", "tiny-qwen3moe"])
def test_draft_model_speculation(ctx, name):
    """spx_engine_set_draft (draft_engine, generate_reply :4244-4269): with lane-exact verify
    passes the stream is the target's plain greedy stream whatever the draft proposes; a draft
    identical to the target has every proposal accepted; accept counts and stream equal the
    oracle's draft-model generation (float family; the MoE family's 1e-2 logit noise can move
    a near-tie, reported)."""
    cfg = M.TINY[name].replace(sigma=0.06)
    w, w2 = M.synth_model(cfg, seed=21), M.synth_model(cfg, seed=22)
    rng = np.random.default_rng(2)
    base = rng.integers(0, cfg.vocab, 20)
    prompt = np.concatenate([base, base]).astype(np.int32)
    eng, same, other = M.Engine(ctx, cfg, w), M.Engine(ctx, cfg, w), M.Engine(ctx, cfg, w2)
    for e in (eng, same, other):
        e.set_mfma(False)
    plain, _ = eng.generate(prompt, 40, speculate=False)
    eng.set_draft(same)
    g, st = eng.generate(prompt, 40, draft_len=4)
    assert np.array_equal(g, plain) and st["drafted"] > 0 and st["accepted"] == st["drafted"], st
    eng.set_draft(other)
    g2, st2 = eng.generate(prompt, 40, draft_len=4, fixed=True)  # fixed: draft lengths independent of timings
    assert np.array_equal(g2, plain) and st2["accepted"] < st2["drafted"], st2
    o, ost = OracleModel(cfg, w).generate(prompt, 40, draft_len=4, fixed=True, draft=OracleModel(cfg, w2))
    if np.array_equal(g2, o):
        for k in ("accepted", "drafted", "verifies", "steps"):
            assert st2[k] == ost[k], (k, st2, ost)
    else:
        assert name == "tiny-qwen3moe", (g2, o)
        print(f"{name}: draft-model stream differs from the oracle's at {int(np.argmax(g2 != o))}")
    eng.set_draft(None)
    for e in (eng, same, other):
        e.close()


@pytest.mark.parametrize("name", ["tiny-qwen3", "tiny-granite", "tiny-a3b"])
def test_hidden_rows_on_request(ctx, name):
    """Hidden rows asked for in one call and not in the next, the same pass size each time (one captured
    pass serves both): a call that asks gets its own pass's rows, with the bits of an engine that is
    always asked, and picks do not depend on it."""
    cfg = M.TINY[name].replace(sigma=0.05)
    w = M.synth_model(cfg, seed=31)
    a, b = M.Engine(ctx, cfg, w), M.Engine(ctx, cfg, w)
    ids, pos = np.random.default_rng(32).integers(0, cfg.vocab, 256), 0
    for m in (1, 2, 9, 16, 17):
        for ask in (True, False, False, True):
            am, h, _ = a.forward(ids[pos:pos + m], pos, hidden=ask)
            am2, h2, _ = b.forward(ids[pos:pos + m], pos, hidden=True)
            assert np.array_equal(am, am2), (name, m)
            if ask:
                assert np.array_equal(h.view(np.uint32), h2.view(np.uint32)), (name, m)
            pos += m
    for n, ask in ((20, False), (20, True), (1, False), (1, True)):
        p1, h, _ = a.feed(ids[pos:pos + n], pos, hidden=ask)
        p2, h2, _ = b.feed(ids[pos:pos + n], pos, hidden=True)
        assert p1 == p2 and (not ask or np.array_equal(h.view(np.uint32), h2.view(np.uint32))), (name, n)
        pos += n
    a.close()
    b.close()
