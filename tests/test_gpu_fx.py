"""Float-activation products on the bf16 matrix cores (fx.hip): Q8_0 matvecs of 2..16 rows against
float64 at the edges of their tiles and parts, activations of every size to the last bit and
non-finite ones, and prefill passes of float models (17..128 rows) against the same rows in passes of
at most 16, bitwise."""
import numpy as np
import pytest

from spindle_amd import model as M
from oracle import ffi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    from spindle_amd import ops
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = ops.Context(0)
    yield c
    c.close()


def _q8_0(rng, cols, rows):
    raw = rng.integers(0, 256, M.row_bytes(M.Q8_0, cols) * rows, dtype=np.uint8)
    raw.reshape(-1, 34)[:, 0:2] = np.float16(rng.uniform(0.001, 0.05, raw.size // 34)).view(np.uint8).reshape(-1, 2)
    return raw, ffi.dequant(M.Q8_0, raw, rows, cols).astype(np.float64).reshape(rows, cols)


# widths of 1 and 2 blocks (empty parts), odd part lengths, 8 and 16 parts; row counts around a
# tile of 16, a workgroup's 32 rows and the four-tile shape of large matrices
@pytest.mark.parametrize("cols,rows", [(32, 17), (64, 1), (96, 65), (576, 33), (992, 16), (1024, 200), (1056, 15), (2016, 64), (2048, 31),
                                       (3072, 48), (4096, 95), (576, 33000), (2080, 33001)])
def test_q8_0_edges(ctx, cols, rows):
    """Within the rounding of a row's fp32 additions: at most 96 in a block (32 products in three
    parts, exact), one a block and one a part, each off by at most one unit in the last place
    (2^-23) of a partial sum that sum |w x| bounds; a vector's bits the same in any batch."""
    from spindle_amd import ops
    rng = np.random.default_rng(cols + rows)
    raw, wd = _q8_0(rng, cols, rows)
    w = ops.Tensor(ctx, M.Q8_0, cols, rows, raw)
    x = (rng.standard_normal((16, cols)) * np.exp(rng.uniform(-8, 8, (16, 1)))).astype(np.float32)
    full = ops.matvec(ctx, w, torch.from_numpy(x).cuda()).cpu().numpy()
    want, scale = x.astype(np.float64) @ wd.T, np.abs(x.astype(np.float64)) @ np.abs(wd).T
    assert np.all(np.abs(full - want) <= (96 + cols // 32 + 16) * 2.0 ** -23 * scale)
    for m, v0 in ((2, 3), (9, 5), (15, 0)):
        part = ops.matvec(ctx, w, torch.from_numpy(x[v0:v0 + m]).cuda()).cpu().numpy()
        assert np.array_equal(part.view(np.uint32), full[v0:v0 + m].view(np.uint32)), m
    w.free()


def test_q8_0_non_finite(ctx):
    """An infinite activation gives what IEEE products and sums give (an infinity, or a NaN where
    its code is 0), a NaN a NaN, and the batch's other vectors keep their bits."""
    from spindle_amd import ops
    rng = np.random.default_rng(5)
    raw, wd = _q8_0(rng, 1024, 64)
    w = ops.Tensor(ctx, M.Q8_0, 1024, 64, raw)
    x = rng.standard_normal((9, 1024)).astype(np.float32)
    clean = ops.matvec(ctx, w, torch.from_numpy(x).cuda()).cpu().numpy()
    x[2, 77], x[4, 500], x[7, 1023] = np.inf, np.nan, -np.inf
    got = ops.matvec(ctx, w, torch.from_numpy(x).cuda()).cpu().numpy()
    for v in (0, 1, 3, 5, 6, 8):
        assert np.array_equal(got[v].view(np.uint32), clean[v].view(np.uint32)), v
    with np.errstate(invalid="ignore"):
        for v, c in ((2, 77), (7, 1023)):
            want = x[v, c].astype(np.float64) * wd[:, c]
            assert np.array_equal(got[v], want.astype(np.float32), equal_nan=True), v
    assert np.isnan(got[4]).all()
    w.free()


# one, three and sixteen parts a row; the four-tile shape of large matrices
@pytest.mark.parametrize("cols,rows", [(32, 17), (1056, 33), (2080, 40), (64, 33000)])
def test_q8_0_whole_activations(ctx, cols, rows):
    """One non-zero activation of 24 significant bits a vector, in each column of a block in turn and
    from the smallest normal to the largest binade and down to the denormals (below 2^-110 its last
    bits are finer than a bf16 holds): times a code of 1 or -1 and a scale of 1/2 it is exact, so
    anything but the exact product is a bit lost. The vectors of a batch take different sizes."""
    from spindle_amd import ops
    rng = np.random.default_rng(cols)
    raw = np.zeros((rows, cols // 32, 34), np.uint8)
    raw[:, :, :2] = np.float16([0.5]).view(np.uint8)
    code = rng.choice([1, -1], (rows, cols)).astype(np.int8)
    raw[:, :, 2:] = code.reshape(rows, -1, 32).view(np.uint8)
    w = ops.Tensor(ctx, M.Q8_0, cols, rows, raw.reshape(-1))
    exps = [0, 126, -60, -100, -109, -111, -118, -125, -127, -133, -140]
    for e0 in range(len(exps)):
        x, want = np.zeros((32, cols), np.float32), np.zeros((32, rows), np.float32)
        for c in range(32):
            at = 32 * int(rng.integers(0, cols // 32)) + c
            v = np.ldexp(1.0 + (rng.integers(0, 2 ** 22) * 2 + 1) * 2.0 ** -23, exps[(e0 + c) % len(exps)])
            x[c, at] = np.float32(v)
            want[c] = (x[c, at].astype(np.float64) * 0.5 * code[:, at]).astype(np.float32)
        for a, b in ((0, 16), (16, 25), (25, 32)):
            got = ops.matvec(ctx, w, torch.from_numpy(x[a:b]).cuda()).cpu().numpy()
            assert np.array_equal(got, want[a:b]), (e0, a, np.argwhere(got != want[a:b])[:4])
    w.free()


@pytest.mark.parametrize("m", [9, 128])
def test_tiny_activations_logits(ctx, m):
    """A model whose activations are around 2^-115: the LM head's rows over the pass's own hidden rows,
    in float64, to the rounding of their sums (test_q8_0_edges)."""
    cfg = M.TINY["tiny-qwen3"].replace(max_seq=320, embedding_scale=2.0 ** -125, dim=1024)
    w = M.synth_model(cfg, seed=3)
    eng = M.Engine(ctx, cfg, w)
    _, hid, lg = eng.forward(np.random.default_rng(4).integers(0, cfg.vocab, m), 0, hidden=True, logits=True)
    spec, data = w["token_embd.weight"]
    wd = ffi.dequant(spec.dtype, data, spec.rows, spec.cols).astype(np.float64).reshape(spec.rows, spec.cols)
    h = hid.astype(np.float64)
    assert 0 < np.abs(h).max() < 2.0 ** -110
    assert np.all(np.abs(lg - h @ wd.T) <= (96 + cfg.dim // 32 + 16) * 2.0 ** -23 * (np.abs(h) @ np.abs(wd).T) + cfg.dim * 2.0 ** -150)
    eng.close()


@pytest.mark.parametrize("ld", [2 ** 28 - 4, 2 ** 28])
def test_q8_0_far_apart_vectors(ctx, ld):
    """Two vectors 1 GiB apart: on either side of where the matrix-core kernel's 32-bit byte offsets
    end (test_q8_0_edges' bound, which the per-lane walk's 32 additions a block keep too)."""
    from spindle_amd import ops
    from spindle_amd._lib import check, lib
    import ctypes as C
    rng = np.random.default_rng(9)
    raw, wd = _q8_0(rng, 1024, 48)
    w = ops.Tensor(ctx, M.Q8_0, 1024, 48, raw)
    x = rng.standard_normal((2, 1024)).astype(np.float32)
    buf, y = torch.empty(ld + 1024, device="cuda"), torch.empty(2, 48, device="cuda")
    buf[:1024], buf[ld:] = torch.from_numpy(x[0]).cuda(), torch.from_numpy(x[1]).cuda()
    torch.cuda.synchronize()
    check(lib.spx_matvec(ctx.h, w.h, 0, C.c_void_p(buf.data_ptr()), ld, 2, C.c_void_p(y.data_ptr()), 48))
    torch.cuda.synchronize()
    want, scale = x.astype(np.float64) @ wd.T, np.abs(x.astype(np.float64)) @ np.abs(wd).T
    assert np.all(np.abs(y.cpu().numpy() - want) <= (96 + 32 + 16) * 2.0 ** -23 * scale)
    w.free()


# dense Q8_0 (attention with q/k norms), dense Q5_0, Q8_0 experts, Q5_0 experts
# (a model with K-quant matrices too runs passes of at most 16)
CASES = {
    "qwen3": M.TINY["tiny-qwen3"].replace(sigma=0.05, max_seq=320),
    "llama-q5_0": M.TINY["tiny-llama"].replace(sigma=0.05, max_seq=320, t_down=M.Q5_0),
    "granite": M.TINY["tiny-granite"].replace(sigma=0.05, max_seq=320),
    "granite-q5_0": M.TINY["tiny-granite"].replace(sigma=0.05, max_seq=320, t_gate=M.Q5_0, t_up=M.Q5_0, t_down=M.Q5_0, moe_prune=0.3),
    # rows of a full and a part-filled 256-value block, and of five
    "granite-288": M.TINY["tiny-granite"].replace(sigma=0.05, max_seq=320, dim=288, n_ff=96),
    "granite-1056": M.TINY["tiny-granite"].replace(sigma=0.03, max_seq=320, dim=1056, n_ff=160, n_expert=32, n_expert_used=8),
    "wide": M.TINY["tiny-qwen3"].replace(sigma=0.03, max_seq=320, dim=1024, n_heads=16, n_kv_heads=8, head_dim=128, n_ff=2048),
    # sixteen parts a row: the gate/up of 17 rows in one-tile workgroups, of 128 in two-tile ones
    "dim2048": M.TINY["tiny-qwen3"].replace(sigma=0.02, max_seq=320, dim=2048, n_heads=16, n_kv_heads=8, head_dim=128, n_ff=1024),
    "dim4096-q5_0": M.TINY["tiny-qwen3"].replace(sigma=0.02, max_seq=320, dim=4096, n_ff=992, t_gate=M.Q5_0, t_up=M.Q5_0, t_down=M.Q8_0),
}


@pytest.mark.parametrize("case", list(CASES))
def test_float_prefill_equals_16_row_passes(ctx, case):
    cfg = CASES[case]
    w = M.synth_model(cfg, seed=71)
    a, b = M.Engine(ctx, cfg, w), M.Engine(ctx, cfg, w)
    ids, pos = np.random.default_rng(72).integers(0, cfg.vocab, 320), 0
    for m in (17, 128, 33, 2, 100, 32):
        am0, h0, l0 = a.forward(ids[pos:pos + m], pos, hidden=True, logits=True)
        for s in range(0, m, 16):
            n = min(16, m - s) if m - s != 17 else 15  # (no last pass of one row: those sum in the one-row order)
            if m - s == 1:
                break
            am1, h1, l1 = b.forward(ids[pos + s:pos + s + n], pos + s, hidden=True, logits=True)
            assert np.array_equal(h0[s:s + n].view(np.uint32), h1.view(np.uint32)), (case, m, s, "hidden")
            assert np.array_equal(l0[s:s + n].view(np.uint32), l1.view(np.uint32)) and np.array_equal(am0[s:s + n], am1), (case, m, s)
        if m % 16 == 1:  # the odd row through a two-row pass with its predecessor
            am1, h1, l1 = b.forward(ids[pos + m - 2:pos + m], pos + m - 2, hidden=True, logits=True)
            assert np.array_equal(h0[m - 2:].view(np.uint32), h1.view(np.uint32)) and np.array_equal(l0[m - 2:].view(np.uint32), l1.view(np.uint32))
        pos += m
    ka, va = a.kv_cache()
    kb, vb = b.kv_cache()
    assert np.array_equal(ka, kb) and np.array_equal(va, vb)
    if cfg.moe:
        assert all(0 < n <= cfg.n_expert for n in a.last_experts())
    a.close()
    b.close()


@pytest.mark.parametrize("case", list(CASES))
def test_float_passes_match_oracle(ctx, case):
    """Passes of 2, 9 and 40 rows against the oracle on the GPU's own KV cache, so that a wrong code or
    scale of either format cannot hide in both sides: logits within 1e-3 of the largest (the bar of
    test_gpu_engine). In the median 1e-4: the pass's own keys and values are rounded to f16 on both
    sides, and where two sums differ by ~2^-22 a share of 2^-22 / 2^-11 of them rounds to the other
    neighbour, 2^-10 away: 2^-10 sqrt(2^-11) = 2e-5 of their root mean square, a layer and for keys
    and values each."""
    from oracle.model import OracleModel
    cfg = CASES[case]
    w = M.synth_model(cfg, seed=73)
    eng, om = M.Engine(ctx, cfg, w), OracleModel(cfg, w)
    ids, pos, errs = np.random.default_rng(74).integers(0, cfg.vocab, 67), 16, []
    eng.forward(ids[:16], 0)
    for m in (2, 9, 40):
        om.k_cache[:], om.v_cache[:] = eng.kv_cache()
        _, _, lg = eng.forward(ids[pos:pos + m], pos, hidden=True, logits=True)
        want = om.logits(om.forward(ids[pos:pos + m], pos)).astype(np.float64)
        errs += list(np.abs(lg - want).max(1) / np.maximum(1.0, np.abs(want).max(1)))
        pos += m
    print(case, "median %.1e max %.1e" % (np.median(errs), np.max(errs)))
    assert np.max(errs) <= 1e-3 and np.median(errs) <= 1e-4
    eng.close()
