"""Workloads of the framework's hot path, as a program that uses it runs them.

A model spends its time in passes: one row a pass while it decodes, 2..16 rows while it verifies
drafted tokens, up to 128 rows while it reads a prompt; and a host that drives the layers itself
spends it in the operators behind the same C ABI (a matrix times 1..16 rows, the routed experts,
the attention block over the KV cache). The cases are those calls on the model shapes that this
repository configures (Qwen3-30B-A3B Q4_K_M, Qwen3-0.6B Q8_0, Granite-1B-A400M Q8_0, SmolLM2-135M
Q5_0): `linear`, `experts` and `attention` are the operators, `pass` is one forward pass at a
context and `feed` the reading of a prompt. Passes and prompts run on a slice of a model's layers
(a layer is the same work at every depth) or, in two cases, on the whole model with its logits.

Weights are random blocks in GGUF layout; ids, rows and routing are drawn from the seed.
"""
import ctypes as C
import math

import numpy as np
import torch

from spindle_amd import model as M
from spindle_amd import ops
from spindle_amd._lib import check, lib

FORMATS = {"F32": M.F32, "Q5_0": M.Q5_0, "Q8_0": M.Q8_0, "Q4_K": M.Q4K, "Q5_K": M.Q5K, "Q6_K": M.Q6K}
# the formats whose rows meet activations quantized to Q8_K (256-value blocks of int8 codes)
INTEGER = (M.Q4K, M.Q6K)

A3B, Q06, GRANITE, SMOL = "qwen3-30b-a3b", "qwen3-0.6b", "granite-1b-a400m", "smollm2-135m"


def listed():
    return [
        # one row through a layer's attention output matrix: the smallest call a host makes
        {"name": "linear-q4k-1", "kind": "linear", "format": "Q4_K", "cols": 4096, "rows": 2048, "m": 1},
        # a float-activation matrix (Qwen3-0.6B's ffn_down) over the nine rows of a k = 8 verify
        {"name": "linear-q8_0-9", "kind": "linear", "format": "Q8_0", "cols": 3072, "rows": 1024, "m": 9},
        # the LM head of Qwen3-30B-A3B over a verify's nine rows
        {"name": "head-q6k-9", "kind": "linear", "format": "Q6_K", "cols": 2048, "rows": 151936, "m": 9},
        # a layer's routed experts (128, 8 a row) over nine rows, the routing in device memory
        {"name": "experts-q4k-9", "kind": "experts", "model": A3B, "m": 9, "host": False},
        # the attention block of a verify at 4K context
        {"name": "attention-9", "kind": "attention", "model": A3B, "m": 9, "context": 4096},
        # the headline model's layers: a decode step, a k = 8 verify, the reading of a prompt
        {"name": "decode-a3b", "kind": "pass", "model": A3B, "layers": 4, "m": 1, "context": 4096, "logits": False},
        {"name": "verify-a3b", "kind": "pass", "model": A3B, "layers": 4, "m": 9, "context": 4096, "logits": False},
        {"name": "feed-a3b", "kind": "feed", "model": A3B, "layers": 4, "n": 1000},
        # a decode step of the whole small model, logits to a host sampler
        {"name": "decode-qwen3-0.6b", "kind": "pass", "model": Q06, "layers": 28, "m": 1, "context": 512, "logits": True},
        # a k = 8 verify on a float-activation MoE model's layers
        {"name": "verify-granite", "kind": "pass", "model": GRANITE, "layers": 8, "m": 9, "context": 256, "logits": False},
        # the reading of a prompt by a float-activation dense model's layers
        {"name": "feed-qwen3-0.6b", "kind": "feed", "model": Q06, "layers": 8, "n": 500},
        # a decode step of the smallest whole model, logits to a host sampler
        {"name": "decode-smollm2", "kind": "pass", "model": SMOL, "layers": 30, "m": 1, "context": 100, "logits": True},
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "experts", "attention", "pass", "pass", "pass", "feed"])
    rows = lambda: rng.choice([1, 2, 9, rng.randint(3, 16)])  # decode, a one-token draft, k = 8, other draft lengths
    if kind == "linear":
        fmt = rng.choice(["Q4_K", "Q6_K", "Q4_K", "Q6_K", "Q8_0", "Q8_0", "Q5_0", "Q5_K", "F32"])
        cols = rng.choice([576, 1024, 2048, 3072] if fmt in ("Q8_0", "Q5_0", "F32") else [768, 1536, 2048, 3072, 4096])
        most = min(152000, 250_000_000 // M.row_bytes(FORMATS[fmt], cols))
        return {"kind": "linear", "format": fmt, "cols": cols, "rows": _log(rng, 200, most), "m": rows()}
    if kind == "experts":
        model = rng.choice([A3B, A3B, GRANITE])
        host = model == GRANITE or rng.random() < 0.3
        return {"kind": "experts", "model": model, "m": rows() if host else rng.choice([rows(), _log(rng, 17, 128)]), "host": host}
    model = rng.choice([A3B, A3B, Q06, GRANITE, SMOL])
    if kind == "attention":
        return {"kind": "attention", "model": model, "m": rows(), "context": _log(rng, 20, 8000 if model == A3B else 4000)}
    most = {A3B: 4, Q06: 8, GRANITE: 8, SMOL: 12}[model]
    if kind == "pass":
        return {"kind": "pass", "model": model, "layers": rng.randint(2, most), "m": rows(),
                "context": _log(rng, 20, 6000 if model == A3B else 2000), "logits": False}
    return {"kind": "feed", "model": model, "layers": rng.randint(2, most), "n": _log(rng, 17, 1000 if model == A3B else 500)}


# ------------------------------------------------------------------------------------- inputs
_ctx = []


def _context():
    """The program's one context (device and stream)."""
    if not _ctx:
        _ctx.append(ops.Context(0))
    return _ctx[0]


def _config(case):
    cfg = M.get_config(case["model"])
    if case["kind"] in ("attention", "experts"):
        # the operator's own layer; a short vocabulary, which it does not read
        return cfg.replace(n_layers=1, vocab=512)
    return cfg.replace(n_layers=case["layers"])


def _ids(cfg, seed, n):
    """A prompt: random ids, then spans copied from the first half (what prompt lookup finds)."""
    r = np.random.default_rng([seed, 1])
    half = (n + 1) // 2
    ids = list(r.integers(0, cfg.vocab, half))
    while len(ids) < n:
        a, k = int(r.integers(0, half)), int(r.integers(16, 65))
        ids += ids[a:min(a + k, half)]
    return np.array(ids[:n], np.int32)


def _weight(case, seed):
    """A linear case's matrix: (format, GGUF bytes)."""
    t = FORMATS[case["format"]]
    spec = M.TensorSpec("w", t, case["cols"], case["rows"], kind=1 if t == M.F32 else 0)
    return t, M.synth_tensor(spec, seed)


def _expert_specs(cfg):
    return [s for s in M.tensor_specs(cfg) if "_exps." in s.name]  # gate, up, down


def _rows(seed, tag, *shape):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 16 + tag)
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _routing(cfg, seed, m):
    """Distinct experts a row with normalised weights, as a router leaves them."""
    r = np.random.default_rng([seed, 2])
    ch = np.stack([r.permutation(cfg.n_expert)[:cfg.n_expert_used] for _ in range(m)]).astype(np.int32)
    return ch, r.dirichlet(np.full(cfg.n_expert_used, 4.0), m).astype(np.float32)


def _qkv(cfg, seed, tag, n):
    """Projections of n rows as the q|k|v matrices give them."""
    return [_rows(seed, tag + i, n, d) for i, d in enumerate((cfg.q_dim, cfg.kv_dim, cfg.kv_dim))]


def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    st = {"case": case, "ctx": ctx}
    if kind == "linear":
        t, data = _weight(case, seed)
        st["w"] = ops.Tensor(ctx, t, case["cols"], case["rows"], data)
        st["x"] = _rows(seed, 0, case["m"], case["cols"])
        st["y"] = torch.empty(case["m"], case["rows"], device="cuda")
    elif kind == "experts":
        cfg = _config(case)
        st["k"] = cfg.n_expert_used
        st["w"] = [ops.Tensor(ctx, s.dtype, s.cols, s.rows, M.synth_tensor(s, seed), s.n_expert) for s in _expert_specs(cfg)]
        st["x"] = _rows(seed, 0, case["m"], cfg.dim)
        st["y"] = torch.empty(case["m"], cfg.dim, device="cuda")
        ch, wt = _routing(cfg, seed, case["m"])
        st["routing"] = (ch, wt) if case["host"] else (torch.from_numpy(ch).cuda(), torch.from_numpy(wt).cuda())
    else:
        cfg = _config(case)
        eng = st["engine"] = M.Engine(ctx, cfg, M.synth_model(cfg, seed))
        if kind == "attention":
            n = case["context"]
            q, k, v = _qkv(cfg, seed, 4, n)
            for a in range(0, n, 16):  # the context's keys and values, sixteen rows a call
                eng.attention(0, q[a:a + 16].contiguous(), k[a:a + 16].contiguous(), v[a:a + 16].contiguous(), a)
            st["qkv"] = _qkv(cfg, seed, 8, case["m"])
            st["y"] = torch.empty(case["m"], cfg.q_dim, device="cuda")
        elif kind == "pass":
            ids = _ids(cfg, seed, case["context"] + case["m"])
            eng.feed(ids[:case["context"]], 0)
            st["ids"] = ids[case["context"]:]
        else:
            st["ids"] = _ids(cfg, seed, case["n"])
    torch.cuda.synchronize()  # torch's stream filled the inputs, the context's stream reads them
    return st


def _p(t):
    return C.c_void_p(t.data_ptr() if isinstance(t, torch.Tensor) else t.ctypes.data)


def run(st):
    case, ctx, kind = st["case"], st["ctx"], st["case"]["kind"]
    if kind == "linear":
        x, y = st["x"], st["y"]
        check(lib.spx_matvec(ctx.h, st["w"].h, 0, _p(x), x.shape[1], case["m"], _p(y), y.shape[1]))
        return y
    if kind == "experts":
        x, y, (ch, wt) = st["x"], st["y"], st["routing"]
        call = lib.spx_moe if case["host"] else lib.spx_moe_dev
        check(call(ctx.h, *(w.h for w in st["w"]), _p(x), x.shape[1], case["m"], st["k"], _p(ch), _p(wt), _p(y), y.shape[1]))
        return y
    eng = st["engine"]
    if kind == "attention":
        q, k, v = st["qkv"]
        check(lib.spx_engine_attention(eng.h, 0, _p(q), _p(k), _p(v), case["m"], case["context"], _p(st["y"])))
        return st["y"]
    if kind == "pass":
        _, hidden, logits = eng.forward(st["ids"], case["context"], hidden=True, logits=case["logits"])
        return {"hidden": hidden, "logits": logits} if case["logits"] else {"hidden": hidden}
    _, hidden, logits = eng.feed(st["ids"], 0, hidden=True, logits=True)
    return {"hidden": hidden, "logits": logits}


# ------------------------------------------------------------------- what a pass cannot do without
def _distinct(cfg, m):
    """Expected number of experts that m rows of n_expert_used random choices touch."""
    return cfg.n_expert * (1.0 - (1.0 - cfg.n_expert_used / cfg.n_expert) ** m)


def work(case):
    if case["kind"] == "linear":
        m, cols, rows = case["m"], case["cols"], case["rows"]
        return {"bytes": M.row_bytes(FORMATS[case["format"]], cols) * rows + 4.0 * m * (cols + rows), "flops": 2.0 * m * cols * rows}
    cfg = _config(case)
    n = case["n"] if case["kind"] == "feed" else case["m"]
    start = case.get("context", 0)
    experts = ([_distinct(cfg, n) / cfg.n_expert * sum(s.nbytes for s in _expert_specs(cfg)), 6.0 * n * cfg.n_expert_used * cfg.dim * cfg.n_ff]
               if cfg.moe and case["kind"] != "attention" else [0.0, 0.0])
    if case["kind"] == "experts":
        return {"bytes": experts[0] + 8.0 * n * cfg.dim, "flops": experts[1]}
    # K and V of every position once (f16), the scores and the weighted sum of each row
    attention = [4.0 * cfg.kv_dim * (start + n), 4.0 * cfg.q_dim * (n * start + n * (n + 1) / 2)]
    if case["kind"] == "attention":
        return {"bytes": attention[0] + 4.0 * n * (2 * cfg.q_dim + 2 * cfg.kv_dim), "flops": attention[1]}
    nbytes, flops = cfg.n_layers * attention[0], cfg.n_layers * attention[1]
    out_rows = 1 if case["kind"] == "feed" else n
    specs = M.tensor_specs(cfg)
    for s in specs:
        if s.name == "token_embd.weight":
            nbytes += min(n, s.rows) * M.row_bytes(s.dtype, s.cols)
            head = s if cfg.tied else next(t for t in specs if t.name == "output.weight")
            nbytes += head.nbytes
            flops += 2.0 * out_rows * head.cols * head.rows
        elif s.name == "output.weight" or "_exps." in s.name:
            continue
        else:
            nbytes += s.nbytes
            if s.rows > 1:
                flops += 2.0 * n * s.cols * s.rows
    moe_layers = cfg.n_layers if cfg.moe else 0
    nbytes += moe_layers * (experts[0] / cfg.n_layers if moe_layers else 0.0)
    flops += moe_layers * experts[1]
    nbytes += 4.0 * out_rows * (cfg.dim + (cfg.vocab if case.get("logits") or case["kind"] == "feed" else 0))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the distance from exact() that the calls show."""
    if case["kind"] == "linear":
        return {"rel": 1e-6}  # 32-bit sums: 1e-7 to 2e-7
    if case["kind"] == "attention":
        return {"rel": 2.5e-5}  # 6e-6: keys and values that round to another f16, 32-bit angles and sums
    if case["kind"] == "experts":
        # 2e-7, but a last-bit change of h can move one of its Q8_K codes by a step, about 1e-4 of a row block
        return {"rel": 5e-4 if case["model"] == A3B else 1e-6}
    # whole passes: every layer requantizes to Q8_K on the integer models (2e-2 over four layers;
    # SmolLM2, only at ffn_down, 1.2e-3), the float models round to f16 in the cache (8e-5)
    return {"rel": {A3B: 3e-2, SMOL: 5e-3}.get(case["model"], 3e-4)}


# ------------------------------------------------------------------------- the same in 64 bits
def _half(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(t, cols, data):
    """GGUF blocks (a uint8 array) as a float64 matrix on the GPU."""
    b = torch.from_numpy(data).cuda()
    if t == M.F32:
        return b.view(torch.float32).double().reshape(-1, cols)
    b = b.reshape(-1, M.BLOCK[t][1])
    if t == M.Q8_0:
        w = _half(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif t == M.Q5_0:
        high = b[:, 2:6].contiguous().view(torch.int32).long()
        bits = (high >> torch.arange(32, device="cuda")) & 1
        low = torch.cat([b[:, 6:] & 15, b[:, 6:] >> 4], 1).long()
        w = _half(b[:, :2]) * (low + 16 * bits - 16).double()
    elif t in (M.Q4K, M.Q5K):
        s = b[:, 4:16].long()
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6 << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6 << 4)], 1)
        q = b[:, -128:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32)
        if t == M.Q5K:
            q = q + 16 * ((b[:, 16:48].reshape(-1, 1, 32) >> torch.arange(8, device="cuda", dtype=torch.uint8).reshape(1, 8, 1)) & 1)
        w = (_half(b[:, :2]) * sc.double()).unsqueeze(2) * q.double() - (_half(b[:, 2:4]) * mn.double()).unsqueeze(2)
    else:  # Q6_K: each half of 128 holds 64 low-nibble bytes and 32 bytes of bit pairs
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)
        two = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (low | (two << 4)).reshape(-1, 16, 16).double() - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        w = (_half(b[:, 208:]) * sc).unsqueeze(2) * q
    return w.reshape(-1, cols)


def _q8k(x):
    """x as its Q8_K blocks give it back: 256 values share amax / 127."""
    b = x.reshape(x.shape[0], -1, 256)
    amax = b.abs().amax(2, keepdim=True)
    codes = torch.where(amax > 0, torch.round(b * (127.0 / amax)), torch.zeros_like(b)).clamp(-127, 127)
    return (codes * (amax / 127.0)).reshape(x.shape)


def _times(t, x, w):
    return (_q8k(x) if t in INTEGER else x) @ w.t()


def _norm(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope(cfg, x, pos):
    """Rotates [n, heads, head_dim] rows; the angles are the f32 table's."""
    inv = np.array([np.float32(1.0) / np.float32(cfg.rope_theta) ** np.float32(2.0 * i / cfg.head_dim) for i in range(cfg.head_dim // 2)], np.float32)
    ang = torch.from_numpy(np.asarray(pos, np.float32)[:, None] * inv[None]).cuda().double().unsqueeze(1)
    c, s = torch.cos(ang), torch.sin(ang)
    if cfg.rope_neox:
        a, b = x.chunk(2, -1)
        return torch.cat([a * c - b * s, b * c + a * s], -1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, b * c + a * s], -1).reshape(x.shape)


def _heads(cfg, x, norm, pos):
    x = x.reshape(x.shape[0], -1, cfg.head_dim)
    return _rope(cfg, x if norm is None else _norm(x, norm, cfg.rms_eps), pos)


def _attend(cfg, q, keys, values, start):
    """q [m, heads, hd] at positions start.. over keys / values [positions, kv heads, hd], held as f16."""
    m, per = q.shape[0], cfg.n_heads // cfg.n_kv_heads
    keys, values = keys.to(torch.float16).double(), values.to(torch.float16).double()
    n = keys.shape[0]
    scale = cfg.attn_scale or 1.0 / math.sqrt(cfg.head_dim)
    seen = torch.arange(n, device="cuda").unsqueeze(0) <= (start + torch.arange(m, device="cuda")).unsqueeze(1)
    out = torch.empty_like(q)
    for h in range(cfg.n_heads):
        g = h // per
        s = (q[:, h].contiguous() @ keys[:, g].t()) * scale
        p = torch.softmax(s.masked_fill(~seen, -math.inf), 1)
        out[:, h] = p @ values[:, g].contiguous()
    return out.reshape(m, -1)


def _ffn(types, x, gate, up, down):
    g = _times(types[0], x, gate)
    return _times(types[2], g * torch.sigmoid(g) * _times(types[1], x, up), down)


def _experts(cfg, x, specs, data, chosen, weights):
    types, y = [s.dtype for s in specs], torch.zeros_like(x)
    slabs = [d.reshape(s.n_expert, -1) for s, d in zip(specs, data)]
    for e in torch.unique(chosen).tolist():
        row, slot = torch.nonzero(chosen == e, as_tuple=True)
        mats = [_dequant(s.dtype, s.cols, d[e]) for s, d in zip(specs, slabs)]
        y.index_add_(0, row, weights[row, slot].unsqueeze(1) * _ffn(types, x[row], *mats))
    return y


def _forward(cfg, tensors, ids, out_rows):
    """The model over all of ids: the last out_rows rows' hidden state and logits."""
    def mat(name):
        s, d = tensors[name]
        return _dequant(s.dtype, s.cols, d)

    def vec(name):
        return mat(name).reshape(-1) if name in tensors else None

    def times(name, x):
        return _times(tensors[name][0].dtype, x, mat(name))

    s, d = tensors["token_embd.weight"]
    rb = M.row_bytes(s.dtype, s.cols)
    x = _dequant(s.dtype, s.cols, np.ascontiguousarray(d.reshape(-1, rb)[ids]).reshape(-1)) * cfg.embedding_scale
    pos = np.arange(len(ids))
    for l in range(cfg.n_layers):
        p = "blk.%d." % l
        n = _norm(x, vec(p + "attn_norm.weight"), cfg.rms_eps)
        q = _heads(cfg, times(p + "attn_q.weight", n), vec(p + "attn_q_norm.weight"), pos)
        k = _heads(cfg, times(p + "attn_k.weight", n), vec(p + "attn_k_norm.weight"), pos)
        v = times(p + "attn_v.weight", n).reshape(k.shape)
        x = x + cfg.residual_scale * times(p + "attn_output.weight", _attend(cfg, q, k, v, 0))
        n = _norm(x, vec(p + "ffn_norm.weight"), cfg.rms_eps)
        if cfg.moe:
            prob = torch.softmax(times(p + "ffn_gate_inp.weight", n), 1)
            w, chosen = torch.topk(prob, cfg.n_expert_used, 1)
            w = w / w.sum(1, keepdim=True) if cfg.expert_norm else w
            names = [p + "ffn_%s_exps.weight" % f for f in ("gate", "up", "down")]
            y = _experts(cfg, n, [tensors[t][0] for t in names], [tensors[t][1] for t in names], chosen, w)
        else:
            names = [p + "ffn_%s.weight" % f for f in ("gate", "up", "down")]
            y = _ffn([tensors[t][0].dtype for t in names], n, *(mat(t) for t in names))
        x = x + cfg.residual_scale * y
    hidden = _norm(x[-out_rows:], vec("output_norm.weight"), cfg.rms_eps)
    return hidden, times("token_embd.weight" if cfg.tied else "output.weight", hidden)


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        t, data = _weight(case, seed)
        return _times(t, _rows(seed, 0, case["m"], case["cols"]).double(), _dequant(t, case["cols"], data))
    cfg = _config(case)
    if kind == "experts":
        specs = _expert_specs(cfg)
        ch, wt = _routing(cfg, seed, case["m"])
        return _experts(cfg, _rows(seed, 0, case["m"], cfg.dim).double(), specs, [M.synth_tensor(s, seed) for s in specs],
                        torch.from_numpy(ch).cuda(), torch.from_numpy(wt).cuda().double())
    if kind == "attention":
        norm = {s.name: _dequant(s.dtype, s.cols, M.synth_tensor(s, seed)).reshape(-1) for s in M.tensor_specs(cfg) if "attn_q_norm" in s.name or "attn_k_norm" in s.name}
        n, m = case["context"], case["m"]
        _, k0, v0 = _qkv(cfg, seed, 4, n)
        q, k1, v1 = _qkv(cfg, seed, 8, m)
        q = _heads(cfg, q.double(), norm.get("blk.0.attn_q_norm.weight"), np.arange(n, n + m))
        k = _heads(cfg, torch.cat([k0, k1]).double(), norm.get("blk.0.attn_k_norm.weight"), np.arange(n + m))
        return _attend(cfg, q, k, torch.cat([v0, v1]).double().reshape(k.shape), n)
    ids = _ids(cfg, seed, case["n"] if kind == "feed" else case["context"] + case["m"])
    hidden, logits = _forward(cfg, M.synth_model(cfg, seed), ids, 1 if kind == "feed" else case["m"])
    if kind == "feed":
        return {"hidden": hidden[0], "logits": logits[0]}
    return {"hidden": hidden, "logits": logits} if case["logits"] else {"hidden": hidden}
