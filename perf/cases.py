"""Timed cases of the AR decode library, through its public entry points.

The work of a song request is a prompt prefill, thousands of decode steps and
the acoustic stage's attention over the conditioning prefix. The cases are
the pieces a host program calls (a layer's projections, the decode and the
prefill attention, the acoustic attention) and whole requests on a session,
at the 3072-wide decoder of the benchmark and the 2048-wide decoder of the
checkpoints, from short prompts and caches to the longest the benchmark runs.
"""
import importlib
import math

import numpy as np
import torch

yuear = importlib.import_module("yue2-mlx_amd.yuear")
lib = yuear.lib

D = 128
EPS = 1e-5
THETA = 500000.0
WIDE = dict(hidden=3072, ffn=8192, heads=24, kv_heads=8)   # the benchmark's decoder
NARROW = dict(hidden=2048, ffn=6144, heads=16, kv_heads=8)  # the checkpoints' decoder
LAYERS, VOCAB = 3, 8192  # whole requests run on a few layers and a small vocabulary
EPI_STORE, EPI_SWIGLU = 0, 2
GEMM_PLAIN, GEMM_SWIGLU = 0, 2


def listed():
    return [
        # one token's four projections of a layer: the bulk of every decode step
        dict(name="proj_b1", kind="proj", batch=1, bits=0, **WIDE),
        # the same for a guided (two branch) request on the 4-bit checkpoint
        dict(name="proj_b2_q4", kind="proj", batch=2, bits=4, **WIDE),
        # six sequences decoded together
        dict(name="proj_b6_narrow", kind="proj", batch=6, bits=0, **NARROW),
        # decode attention just after a short prompt: the smallest call
        dict(name="attn_decode_kv333", kind="attn_decode", batch=1, kv=333, ragged=False, **WIDE),
        # decode attention at the benchmark's cache length
        dict(name="attn_decode_kv4096", kind="attn_decode", batch=1, kv=4096, ragged=False, **WIDE),
        # eight sequences of unlike lengths, up to the benchmark's 6144
        dict(name="attn_decode_b8", kind="attn_decode", batch=8, kv=6144, ragged=True, **WIDE),
        # a layer's projections for a short prompt (a request's text, its negative prefix)
        dict(name="gemm_m130", kind="gemm", tokens=130, **WIDE),
        # ... and for the benchmark's long prompt
        dict(name="gemm_m3000", kind="gemm", tokens=3000, **WIDE),
        # causal attention of that prompt
        dict(name="attn_prefill_t3000", kind="attn_prefill", tokens=3000, pos0=0, **WIDE),
        # one query chunk of the acoustic stage over its conditioning prefix
        dict(name="nar_512x3512", kind="nar", q_len=512, kv_len=3512, causal=False, **WIDE),
        # a whole request: prefill a prompt, decode some tokens
        dict(name="request_b1", kind="request", batch=1, bits=0, prompt=301, steps=12, **WIDE),
        # several requests of unlike prompts served together from a 4-bit checkpoint
        dict(name="request_b5_q4", kind="request", batch=5, bits=4, prompt=200, steps=12, **NARROW),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    dims = rng.choice((WIDE, NARROW))
    kind = rng.choice(("proj", "attn_decode", "gemm", "attn_prefill", "nar", "request"))
    if kind == "proj":
        bits = rng.choice((0, 0, 4, 8))
        return dict(kind=kind, batch=rng.randint(1, 2 if bits else 8), bits=bits, **dims)
    if kind == "attn_decode":
        batch = rng.choice((1, 1, 2, rng.randint(3, 8)))
        return dict(kind=kind, batch=batch, kv=_log_int(rng, 40, 6144 if batch > 2 else 24000),
                    ragged=batch > 2, **dims)
    if kind == "gemm":
        return dict(kind=kind, tokens=_log_int(rng, 9, 3000), **dims)
    if kind == "attn_prefill":
        return dict(kind=kind, tokens=_log_int(rng, 9, 3000), pos0=rng.choice((0, rng.randint(1, 2048))),
                    **dims)
    if kind == "nar":
        if rng.random() < 0.3:
            n = _log_int(rng, 100, 3000)
            return dict(kind=kind, q_len=n, kv_len=n, causal=True, **dims)
        return dict(kind=kind, q_len=_log_int(rng, 33, 1024), kv_len=_log_int(rng, 400, 8000),
                    causal=False, **dims)
    return dict(kind=kind, batch=rng.choice((1, 1, 2, rng.randint(3, 8))), bits=rng.choice((0, 0, 4, 8)),
                prompt=_log_int(rng, 12, 300), steps=rng.randint(4, 12), **dims)


# ---- inputs ----

def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + stream) % (1 << 62))
    return g


def _normal(g, *shape, mean=0.0, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda").mul_(std).add_(mean).to(torch.bfloat16)


def _projections(c):
    """(name, rows, columns, normed input, gate/up pairs) of a layer."""
    qd, kd = c["heads"] * D, c["kv_heads"] * D
    return [("qkv", qd + 2 * kd, c["hidden"], True, False), ("o", c["hidden"], qd, False, False),
            ("gate_up", 2 * c["ffn"], c["hidden"], True, True), ("down", c["hidden"], c["ffn"], False, False)]


def _quantized(g, n, k, bits):
    """Random codes and group scales / biases of weights of spread 0.02."""
    top = (1 << bits) - 1
    codes = torch.randint(-2**31, 2**31, (n, k * bits // 32), generator=g, device="cuda", dtype=torch.int64)
    scale = (torch.rand(n, k // 64, generator=g, device="cuda") * 0.4 + 0.8) * (0.02 * 12 ** 0.5 / top)
    scale = scale.to(torch.bfloat16)
    bias = (scale.float() * (-top / 2)).to(torch.bfloat16)
    return codes.to(torch.int32), scale, bias


def _group_words(scale, bias):
    lo = scale.view(torch.int16).to(torch.int32) & 0xffff
    hi = bias.view(torch.int16).to(torch.int32) << 16
    return (lo | hi).contiguous()


def _dequantized(codes, scale, bias, bits):
    n = codes.shape[0]
    shifts = torch.arange(0, 32, bits, device="cuda", dtype=torch.int32)
    q = (codes[:, :, None] >> shifts) & ((1 << bits) - 1)
    q = q.reshape(n, -1, 64).double()
    return (q * scale.double()[:, :, None] + bias.double()[:, :, None]).reshape(n, -1)


def _proj_inputs(c, seed):
    out = []
    for i, (name, n, k, normed, pairs) in enumerate(_projections(c)):
        g = _gen(seed, i)
        x = _normal(g, c["batch"], k, std=1.0 if normed else 0.5)
        gain = _normal(g, k, mean=1.0, std=0.1) if normed else None
        w = _quantized(g, n, k, c["bits"]) if c["bits"] else _normal(g, n, k, std=0.02)
        out.append((name, n, k, pairs, x, gain, w))
    return out


def _rope(positions, theta=THETA):
    inv = 1.0 / theta ** (torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D)
    a = torch.arange(positions, device="cuda", dtype=torch.float64)[:, None] * inv
    return a.cos().to(torch.bfloat16), a.sin().to(torch.bfloat16)


def _slots(n):
    return (n + 31) // 32 * 32


def _blocked(v):
    """[..., slots, 128] -> the V cache's 32-slot dim-major blocks."""
    *lead, n, d = v.shape
    return v.reshape(*lead, n // 32, 32, d).transpose(-1, -2).contiguous().reshape(*lead, n, d)


def _lengths(c, seed):
    """Cache lengths of an attn_decode case, or prompt lengths of a request."""
    top = c["kv"] if c["kind"] == "attn_decode" else c["prompt"]
    if c["batch"] == 1 or (c["kind"] == "attn_decode" and not c["ragged"]):
        return [top] * c["batch"]
    rng = np.random.default_rng(int(seed) + 17)
    rest = rng.integers(max(1, top // 8), top + 1, c["batch"] - 1)
    return [top] + [int(v) for v in rest]


def _attn_decode_inputs(c, seed):
    g = _gen(seed, 0)
    hq, hkv, b = c["heads"], c["kv_heads"], c["batch"]
    lens = _lengths(c, seed)
    cap = _slots(c["kv"])
    qkv = _normal(g, b, (hq + 2 * hkv) * D)
    gains = [_normal(g, D, mean=1.0, std=0.1) for _ in range(2)]
    cos, sin = _rope(cap)
    k = _normal(g, b, hkv, cap, D)
    v = _normal(g, b, hkv, cap, D)
    return qkv, gains, cos, sin, k, v, lens, cap


def _gemm_inputs(c, seed):
    out = []
    for i, (name, n, k, normed, pairs) in enumerate(_projections(c)):
        g = _gen(seed, i)
        out.append((name, n, k, pairs, _normal(g, c["tokens"], k, std=1.0 if normed else 0.5),
                    _normal(g, n, k, std=0.02)))
    return out


def _attn_prefill_inputs(c, seed):
    g = _gen(seed, 0)
    cap = _slots(c["pos0"] + c["tokens"])
    q = _normal(g, c["tokens"], c["heads"], D)
    return q, _normal(g, c["kv_heads"], cap, D), _normal(g, c["kv_heads"], cap, D), cap


def _nar_inputs(c, seed):
    g = _gen(seed, 0)
    return (_normal(g, 1, c["heads"], c["q_len"], D), _normal(g, 1, c["kv_heads"], c["kv_len"], D),
            _normal(g, 1, c["kv_heads"], c["kv_len"], D))


def _config(c):
    return dict(hidden_size=c["hidden"], intermediate_size=c["ffn"], num_hidden_layers=LAYERS,
                num_attention_heads=c["heads"], num_key_value_heads=c["kv_heads"], head_dim=D,
                vocab_size=VOCAB, max_position_embeddings=4096, rms_norm_eps=EPS, rope_theta=THETA,
                qk_norm=True)


def _model(c, seed):
    """Checkpoint tensors by name: bf16, or (codes, scales, biases)."""
    out = {}
    for i, (name, shape) in enumerate(yuear.tensor_shapes(_config(c)).items()):
        g = _gen(seed, 100 + i)
        if "norm" in name:
            out[name] = _normal(g, *shape, mean=1.0, std=0.1)
        elif c["bits"] and name != "model.embed_tokens.weight":
            out[name] = _quantized(g, *shape, c["bits"])
        else:
            out[name] = _normal(g, *shape, std=0.02)
    return out


def _tokens(c, seed):
    rng = np.random.default_rng(int(seed) + 29)
    prompts = [rng.integers(0, VOCAB, n).astype(np.int32) for n in _lengths(c, seed)]
    return prompts, rng.integers(0, VOCAB, (c["steps"], c["batch"])).astype(np.int32)


def _host16(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def _prepare_request(c, seed):
    weights = {}
    for name, t in _model(c, seed).items():
        if isinstance(t, tuple):
            base = name[:-len(".weight")]
            weights[name] = t[0].cpu().numpy().view(np.uint32)
            weights[base + ".scales"], weights[base + ".biases"] = _host16(t[1]), _host16(t[2])
        else:
            weights[name] = _host16(t)
    engine = yuear.Engine(_config(c), weights, bits=c["bits"])
    session = engine.session(c["batch"], c["prompt"] + c["steps"] + 1)
    prompts, steps = _tokens(c, seed)
    return dict(session=session, prompts=prompts, steps=steps)


def prepare(case, seed):
    # "calls": the entry point, its arguments, what it writes, and the tensors
    # that its arguments point into
    c = case
    s = dict(case=case)
    if c["kind"] == "proj":
        s["calls"] = []
        for name, n, k, pairs, x, gain, w in _proj_inputs(c, seed):
            y = torch.empty(c["batch"], n // 2 if pairs else n, dtype=torch.bfloat16, device="cuda")
            w = (w[0], _group_words(w[1], w[2])) if c["bits"] else (w,)
            rest = (n, k, c["batch"], x.data_ptr(), k, gain.data_ptr() if gain is not None else None, EPS,
                    y.data_ptr(), y.shape[1], EPI_SWIGLU if pairs else EPI_STORE, None)
            if c["bits"]:
                call = (lib.yuear_op_qgemv, (w[0].data_ptr(), w[1].data_ptr(), c["bits"]) + rest)
            else:
                call = (lib.yuear_op_gemv, (w[0].data_ptr(),) + rest)
            s["calls"].append(call + (y, (x, gain, w)))
    elif c["kind"] == "attn_decode":
        qkv, gains, cos, sin, k, v, lens, cap = _attn_decode_inputs(c, seed)
        # one workgroup per CU for a single sequence, about 512 otherwise, one
        # 128-key pass each at most: how a session splits its cache
        most = (256 if c["batch"] == 1 else 512) // (c["batch"] * c["kv_heads"])
        splits = max(1, min(64, max(2, most), -(-cap // 128)))
        pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device="cuda")
        out = torch.empty(c["batch"], c["heads"] * D, dtype=torch.bfloat16, device="cuda")
        v = _blocked(v)
        ptr = [t.data_ptr() for t in (qkv, gains[0], gains[1], cos, sin, k, v, pos, out)]
        s["calls"] = [(lib.yuear_op_attention_decode,
                       (*ptr[:3], EPS, *ptr[3:8], c["heads"], c["kv_heads"], cap, c["batch"], splits,
                        ptr[8], None), [out, k, v], (qkv, gains, cos, sin, pos))]
    elif c["kind"] == "gemm":
        s["calls"] = []
        for name, n, k, pairs, a, w in _gemm_inputs(c, seed):
            y = torch.empty(c["tokens"], n // 2 if pairs else n, dtype=torch.bfloat16, device="cuda")
            s["calls"].append((lib.yuear_op_gemm,
                               (a.data_ptr(), k, w.data_ptr(), c["tokens"], n, k, y.data_ptr(), y.shape[1],
                                GEMM_SWIGLU if pairs else GEMM_PLAIN, None), y, (a, w)))
    elif c["kind"] == "attn_prefill":
        q, k, v, cap = _attn_prefill_inputs(c, seed)
        v, out = _blocked(v), torch.empty_like(q)
        s["calls"] = [(lib.yuear_op_attention_prefill,
                       (q.data_ptr(), k.data_ptr(), v.data_ptr(), c["tokens"], c["pos0"], c["heads"],
                        c["kv_heads"], cap, out.data_ptr(), None), out, (q, k, v))]
    elif c["kind"] == "nar":
        q, k, v = _nar_inputs(c, seed)
        n = lib.yuear_nar_attention_workspace_bytes(1, c["kv_heads"], c["kv_len"])
        s.update(q=q, k=k, v=v, workspace=torch.empty(n // 2, dtype=torch.bfloat16, device="cuda"))
    else:
        s.update(_prepare_request(c, seed))
    return s


# ---- one pass ----

def _logits(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).view(torch.bfloat16)


def run(state):
    s, c = state, state["case"]
    if "calls" in s:  # entry points on device pointers, one after the other
        for entry, args, _, _ in s["calls"]:
            status = entry(*args)
            if status:
                raise RuntimeError(f"{entry.__name__} returned {status}")
        return [call[2] for call in s["calls"]]
    if c["kind"] == "nar":
        return yuear.nar_attention(s["q"], s["k"], s["v"], c["causal"], workspace=s["workspace"])
    # a request on a session: back to an empty cache, every branch's prompt,
    # then one step per token; the host reads the logits each time
    session = s["session"]
    first = []
    for b, prompt in enumerate(s["prompts"]):
        session.set_position(b, 0)
        first.append(session.prefill(b, prompt))
    rest = [session.step(tokens) for tokens in s["steps"]]
    return [_logits(np.stack(first)), _logits(np.stack(rest))]


# ---- what a pass cannot do without ----

def _weight_bytes(c, n, k):
    return n * k * c["bits"] // 8 + n * k // 64 * 4 if c["bits"] else 2 * n * k


def work(case):
    c = case
    hq, hkv = c["heads"], c["kv_heads"]
    if c["kind"] == "proj":
        b = sum(_weight_bytes(c, n, k) + 2 * c["batch"] * (k + (n // 2 if pairs else n)) + (2 * k if normed else 0)
                for _, n, k, normed, pairs in _projections(c))
        return dict(bytes=b, flops=2 * c["batch"] * sum(n * k for _, n, k, _, _ in _projections(c)))
    if c["kind"] == "attn_decode":
        keys = sum(_lengths(c, 1))
        return dict(bytes=4 * keys * hkv * D + 2 * c["batch"] * (2 * hq + 2 * hkv) * D,
                    flops=4 * keys * hq * D)
    if c["kind"] == "gemm":
        t = c["tokens"]
        return dict(bytes=sum(2 * n * k + 2 * t * (k + (n // 2 if pairs else n))
                              for _, n, k, _, pairs in _projections(c)),
                    flops=2 * t * sum(n * k for _, n, k, _, _ in _projections(c)))
    if c["kind"] == "attn_prefill":
        t, n = c["tokens"], c["pos0"] + c["tokens"]
        seen = t * c["pos0"] + t * (t + 1) // 2
        return dict(bytes=4 * t * hq * D + 4 * n * hkv * D, flops=4 * seen * hq * D)
    if c["kind"] == "nar":
        t, n = c["q_len"], c["kv_len"]
        seen = t * (t + 1) // 2 if c["causal"] else t * n
        return dict(bytes=4 * t * hq * D + 4 * n * hkv * D, flops=4 * seen * hq * D)
    lens = _lengths(c, 1)
    layer = sum(n * k for _, n, k, _, _ in _projections(c))
    layer_bytes = sum(_weight_bytes(c, n, k) for _, n, k, _, _ in _projections(c))
    head, head_bytes = VOCAB * c["hidden"], _weight_bytes(c, VOCAB, c["hidden"])
    passes = c["batch"] + c["steps"]
    kv = sum(4 * hkv * D * (n + i) for n in lens for i in range(1, c["steps"] + 1))
    seen = sum(n * (n + 1) // 2 + sum(n + i for i in range(1, c["steps"] + 1)) for n in lens)
    rows = sum(lens) + c["batch"] * c["steps"]
    return dict(bytes=passes * (LAYERS * layer_bytes + head_bytes) + LAYERS * kv,
                flops=2 * LAYERS * layer * rows + 2 * head * c["batch"] * (1 + c["steps"])
                + 4 * LAYERS * seen * hq * D)


def tolerance(case):
    # measured against exact(): GEMM and prefill attention outputs 0.0016-0.0036
    # (one rounding, or SwiGLU's three), the normed projections and the decode
    # attention 0.0036-0.0066 (the rounded norm, RoPE and SwiGLU), the logits
    # of a request 0.018-0.021 after three layers of bf16 activations
    if case["kind"] == "request":
        return {"rel": 3e-2}
    return {"rel": 6e-3 if case["kind"] in ("attn_prefill", "nar") else 1e-2}


# ---- the same in 64 bits ----

def _norm64(x, gain):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * gain.double()


def _swiglu64(y):
    g, u = y[..., 0::2], y[..., 1::2]
    return g * torch.sigmoid(g) * u


def _rotate64(x, cos, sin):
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)


def _attend64(q, k, v, first):
    """q [H, T, D] at positions first + t over k / v [Hkv, n, D]; first None: every key is seen."""
    out = torch.empty_like(q)
    per = q.shape[0] // k.shape[0]
    for h in range(q.shape[0]):
        s = q[h] @ k[h // per].T.contiguous() / D ** 0.5
        if first is not None:
            t = torch.arange(s.shape[0], device=s.device)[:, None] + first
            s = s.masked_fill(torch.arange(s.shape[1], device=s.device)[None] > t, -math.inf)
        out[h] = torch.softmax(s, -1) @ v[h // per]
    return out


def _exact_request(c, seed):
    w = {}
    for name, t in _model(c, seed).items():
        w[name] = _dequantized(*t, c["bits"]) if isinstance(t, tuple) else t.double()
    hq, hkv = c["heads"], c["kv_heads"]
    prompts, steps = _tokens(c, seed)
    cos, sin = (t.double() for t in _rope(c["prompt"] + c["steps"]))
    first, rest = [], []
    for b, prompt in enumerate(prompts):
        ids = torch.from_numpy(np.concatenate([prompt, steps[:, b]]).astype(np.int64)).cuda()
        n = len(ids)
        x = w["model.embed_tokens.weight"][ids]
        for i in range(LAYERS):
            def p(name):
                return w[f"model.layers.{i}.{name}.weight"]

            def heads(y, count):
                return y.reshape(n, count, D).transpose(0, 1)
            h = _norm64(x, p("input_layernorm"))
            q = heads(h @ p("self_attn.q_proj").T, hq)
            k = heads(h @ p("self_attn.k_proj").T, hkv)
            v = heads(h @ p("self_attn.v_proj").T, hkv).contiguous()
            q = _rotate64(_norm64(q, p("self_attn.q_norm")), cos[:n], sin[:n])
            k = _rotate64(_norm64(k, p("self_attn.k_norm")), cos[:n], sin[:n])
            a = _attend64(q, k, v, 0)
            x = x + a.transpose(0, 1).reshape(n, hq * D) @ p("self_attn.o_proj").T
            h = _norm64(x, p("post_attention_layernorm"))
            g = h @ p("mlp.gate_proj").T
            x = x + (g * torch.sigmoid(g) * (h @ p("mlp.up_proj").T)) @ p("mlp.down_proj").T
        y = _norm64(x[len(prompt) - 1:], w["model.norm.weight"]) @ w["lm_head.weight"].T
        first.append(y[0])
        rest.append(y[1:])
    return [torch.stack(first), torch.stack(rest, 1)]


def exact(case, seed):
    c = case
    if c["kind"] == "proj":
        out = []
        for name, n, k, pairs, x, gain, w in _proj_inputs(c, seed):
            x = x.double() if gain is None else _norm64(x.double(), gain)
            w = _dequantized(*w, c["bits"]) if c["bits"] else w.double()
            y = x @ w.T
            out.append(_swiglu64(y) if pairs else y)
        return out
    if c["kind"] == "attn_decode":
        qkv, gains, cos, sin, k, v, lens, cap = _attn_decode_inputs(c, seed)
        hq, hkv = c["heads"], c["kv_heads"]
        out, k, v = [], k.double(), v.double()
        for b, n in enumerate(lens):
            row = qkv[b].double().reshape(hq + 2 * hkv, D)
            cs, sn = cos[n - 1].double(), sin[n - 1].double()
            q = _rotate64(_norm64(row[:hq], gains[0]), cs, sn)
            k[b, :, n - 1] = _rotate64(_norm64(row[hq:hq + hkv], gains[1]), cs, sn)
            v[b, :, n - 1] = row[hq + hkv:]
            out.append(_attend64(q[:, None], k[b, :, :n], v[b, :, :n].contiguous(), None).reshape(-1))
        return [[torch.stack(out), k, _blocked(v)]]
    if c["kind"] == "gemm":
        out = []
        for name, n, k, pairs, a, w in _gemm_inputs(c, seed):
            y = a.double() @ w.double().T
            out.append(_swiglu64(y) if pairs else y)
        return out
    if c["kind"] == "attn_prefill":
        q, k, v, cap = _attn_prefill_inputs(c, seed)
        n = c["pos0"] + c["tokens"]
        q = q.transpose(0, 1).double().contiguous()
        out = _attend64(q, k[:, :n].double(), v[:, :n].double(), c["pos0"])
        return [out.transpose(0, 1).contiguous()]
    if c["kind"] == "nar":
        q, k, v = (t[0].double() for t in _nar_inputs(c, seed))
        return _attend64(q, k, v, 0 if c["causal"] else None)[None]
    return _exact_request(c, seed)
