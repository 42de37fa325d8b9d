"""The work that users of this framework have it do, as cases that can be timed.

Three groups, through the package's public entry points:

- the projections and the kernels around them, which a host program calls one
  by one (matvec / matmul / matmul_x1, the greedy head, the activation
  preparation, the DeltaNet update, the paged attention, the causal
  convolution): decode sizes (1 to 64 vectors) and prompt sizes;
- a whole MLP block composed from those entry points as a program composes it;
- whole model steps through `Runtime`: a sampled decode step and a packed step
  (decode rows plus a prompt chunk), which return the logits of the candidates.

Sizes are those of the repository's model shapes (0.8B: hidden 1024, MLP 3584;
4B: hidden 2560, MLP 9216; vocabulary 248,320) and its benchmark's workloads.
Weights and activations are drawn as the packers leave them: Gaussian values
quantized to Q4-G32-DOT4 tiles and to per-32 int8 blocks.
"""
import ctypes
import math

import numpy as np
import torch

import __graft_entry__

q = __graft_entry__.load()

HEAD_DIM = 256
SEED64 = q.DEFAULT_SIGN_SEED

# ------------------------------------------------------------------ the cases


def listed():
    return [
        # one request decoding: the widest projection of the 4B shape as a GEMV
        {"name": "gemv_1_gate_up", "kind": "gemm", "tokens": 1, "rows": 18432, "cols": 2560, "x1": True},
        # an odd decode batch: seven independently prepared rows through the
        # fused in-projection (8224 rows, no multiple of 64)
        {"name": "gemm_7_in_proj", "kind": "gemm", "tokens": 7, "rows": 8224, "cols": 1024, "x1": True},
        # the usual decode batch of 16 (the kernel-level benchmark's shape)
        {"name": "gemm_16", "kind": "gemm", "tokens": 16, "rows": 3584, "cols": 1024, "x1": False},
        # a prompt chunk of 2048 tokens through the 4B gate_up projection
        {"name": "gemm_2048_gate_up", "kind": "gemm", "tokens": 2048, "rows": 18432, "cols": 2560, "x1": False},
        # the greedy vocabulary head of 16 requests with the repetition penalty
        {"name": "head_16", "kind": "head", "tokens": 16, "rows": 248320, "cols": 1024},
        # the 4B down projection's input of a prompt chunk: rotation and int8 codes
        {"name": "prep_2048", "kind": "prep", "tokens": 2048, "cols": 9216, "h128": True},
        # one DeltaNet step of 64 requests of the 4B shape
        {"name": "delta_64", "kind": "delta", "batch": 64, "heads": 32},
        # decode attention of 64 requests with contexts between 128 and 8192 (4B heads)
        {"name": "attention_64", "kind": "attention", "batch": 64, "heads": 16, "kv_heads": 4, "page_tokens": 16,
         "min_context": 128, "max_context": 8192},
        # the causal convolution over a ragged prompt's q/k/v channels (4B)
        {"name": "conv_1500", "kind": "conv", "tokens": 1500, "channels": 8192},
        # the MLP block of the 0.8B shape on the engine's default prompt chunk
        {"name": "mlp_128", "kind": "mlp", "tokens": 128, "hidden": 1024, "inter": 3584},
        # one sampled decode step of 16 requests through the whole 0.8B model
        {"name": "decode_16", "kind": "decode", "batch": 16, "min_context": 384, "max_context": 640},
        # a packed step at the 4B layer shapes: 64 decode rows and a ragged
        # 2000-odd token prompt chunk in one pass
        {"name": "packed_64", "kind": "packed", "batch": 64, "min_context": 128, "max_context": 4096, "chunk": 1999},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "head", "prep", "delta", "attention", "conv", "mlp", "decode", "packed"])
    if kind == "gemm":
        tokens = _log_int(rng, 1, 2048)
        if rng.random() < 0.5:
            tokens = (tokens + 3) // 4 * 4
        return {"kind": "gemm", "tokens": tokens, "rows": 8 * _log_int(rng, 64, 2304), "cols": 32 * _log_int(rng, 16, 80),
                "x1": tokens % 4 != 0 or rng.random() < 0.25}
    if kind == "head":
        return {"kind": "head", "tokens": 4 * rng.randint(1, 16), "rows": 8 * _log_int(rng, 1000, 31040),
                "cols": rng.choice([1024, 2048, 2560])}
    if kind == "prep":
        tokens = _log_int(rng, 1, 2048)
        return {"kind": "prep", "tokens": tokens if tokens == 1 else (tokens + 3) // 4 * 4, "cols": 128 * rng.randint(2, 72),
                "h128": rng.random() < 0.75}
    if kind == "delta":
        return {"kind": "delta", "batch": _log_int(rng, 1, 64), "heads": rng.choice([16, 32])}
    if kind == "attention":
        heads, kv = rng.choice([(8, 2), (8, 2), (16, 4), (4, 4), (16, 2)])
        top = _log_int(rng, 64, 8192)
        return {"kind": "attention", "batch": _log_int(rng, 1, 64), "heads": heads, "kv_heads": kv,
                "page_tokens": rng.choice([4, 16, 16, 64]), "min_context": rng.randint(1, top), "max_context": top}
    if kind == "conv":
        return {"kind": "conv", "tokens": _log_int(rng, 1, 2048), "channels": rng.choice([6144, 8192])}
    if kind == "mlp":
        hidden, inter = rng.choice([(1024, 3584), (2048, 6144), (2560, 9216)])
        return {"kind": "mlp", "tokens": 4 * _log_int(rng, 1, 128), "hidden": hidden, "inter": inter}
    if kind == "decode":
        top = rng.randint(64, 1000)
        return {"kind": "decode", "batch": rng.randint(1, 16), "min_context": rng.randint(8, top), "max_context": top}
    top = _log_int(rng, 200, 4096)
    return {"kind": "packed", "batch": rng.randint(1, 64), "min_context": rng.randint(16, top), "max_context": top,
            "chunk": 2 * _log_int(rng, 8, 1000) + 1}


# ------------------------------------------------------------------- material

_CTX = None


def _ctx():
    """The program's one context (one device, one stream)."""
    global _CTX
    if _CTX is None:
        _CTX = q.Context(0)
    return _CTX


class _Arg:
    """A torch tensor as a buffer argument of the package's operators."""

    def __init__(self, tensor):
        assert tensor.is_contiguous()
        self.tensor, self.ptr = tensor, ctypes.c_void_p(tensor.data_ptr())


def _rng(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _rand(g, *shape):
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float32)


def _q4(g, rows, cols, std=0.02):
    """Gaussian weights as Q4 codes u [rows, cols/32, 32] (0..15) and binary16 scales [rows, cols/32]."""
    w = _randn(g, rows, cols // 32, 32) * std
    at = w.abs().argmax(dim=-1, keepdim=True)
    d = w.gather(-1, at).squeeze(-1) / -8.0
    u = torch.clamp(torch.floor(w / d.unsqueeze(-1) + 8.5), 0, 15).to(torch.uint8)
    return u, d.to(torch.float16)


def _tiles(u, d):
    """DOT4 tiles [rows/8][block] of 144 bytes: eight binary16 scales, then
    byte 32t+4r+j = u[r][8t+j] | u[r][8t+4+j] << 4."""
    rows, nb = d.shape
    v = u.view(rows // 8, 8, nb, 4, 2, 4)
    body = (v[..., 0, :] | (v[..., 1, :] << 4)).permute(0, 2, 3, 1, 4).reshape(rows // 8, nb, 128)
    scale = d.view(rows // 8, 8, nb).permute(0, 2, 1).contiguous().view(torch.uint8).view(rows // 8, nb, 16)
    return torch.cat([scale, body], dim=-1).contiguous()


def _dequant(u, d):
    return ((u.double() - 8.0) * d.double().unsqueeze(-1)).reshape(d.shape[0], -1)


def _q8(g, tokens, cols):
    """Gaussian activations as int8 codes [tokens, blocks, 32] and stored scales [tokens, blocks]."""
    x = _randn(g, tokens, cols // 32, 32)
    scale = x.abs().amax(dim=-1) / 127.0
    codes = torch.clamp(torch.round(x / scale.unsqueeze(-1)), -127, 127).to(torch.int8)
    return codes, scale.to(torch.float16).float() / math.sqrt(128.0)


def _x4(codes, scales):
    """X4 blocks [tokens/4][block] of 152 bytes: four scales, four code sums, four rows of codes."""
    t, nb = scales.shape
    s = scales.view(t // 4, 4, nb).permute(0, 2, 1).contiguous().view(torch.uint8).view(t // 4, nb, 16)
    sums = codes.int().sum(-1).to(torch.int16).view(t // 4, 4, nb).permute(0, 2, 1).contiguous()
    c = codes.view(t // 4, 4, nb, 32).permute(0, 2, 1, 3).contiguous().view(torch.uint8).view(t // 4, nb, 128)
    return torch.cat([s, sums.view(torch.uint8).view(t // 4, nb, 8), c], dim=-1).contiguous()


def _x1(codes, scales):
    """X1 blocks [token][block] of 40 bytes: scale, code sum, codes, padding."""
    t, nb = scales.shape
    sums = codes.int().sum(-1).to(torch.int16).contiguous()
    return torch.cat([scales.contiguous().view(torch.uint8).view(t, nb, 4), sums.view(torch.uint8).view(t, nb, 2),
                      codes.contiguous().view(torch.uint8).view(t, nb, 32),
                      torch.zeros(t, nb, 2, dtype=torch.uint8, device="cuda")], dim=-1).contiguous()


def _contexts(seed, case):
    r = np.random.default_rng(int(seed))
    return r.integers(case["min_context"], case["max_context"] + 1, size=case["batch"]).astype(np.int32)


# -------------------------------------------------------------- whole models

_MODELS = {}


def _model(which):
    """The weights a serving program keeps resident: the whole 0.8B shape
    ("decode"), or four layers of the 4B shape (three linear, one full
    attention) with a 32,768-token vocabulary ("packed")."""
    if which in _MODELS:
        return _MODELS[which]
    ctx = _ctx()
    d, sched = q.model_dims(0 if which == "decode" else 2)
    if which == "packed":
        d.n_layers, d.vocab = 4, 32768
        sched = np.array([1, 1, 1, 0], np.uint8)
    g = _rng(77)
    model = q.Model(ctx, d, sched)

    def q4(name, rows, cols, enc=q.ENC_Q4_H128_DOT4):
        model.upload(name, enc, (rows, cols), _tiles(*_q4(g, rows, cols)).cpu().numpy())

    def f32(name, shape, values):
        model.upload(name, q.ENC_F32, shape, values.float().cpu().numpy().reshape(shape))

    h, inter, hd = d.hidden, d.intermediate, d.head_dim
    v_dim = d.lin_v_heads * d.lin_v_dim
    ch = 2 * d.lin_k_heads * d.lin_k_dim + v_dim
    q4("model.language_model.embed_tokens.weight", d.vocab, h, q.ENC_Q4_0_DOT4)
    f32("model.language_model.norm.weight", (h,), _randn(g, h) * 0.1)
    for i in range(d.n_layers):
        p = f"model.language_model.layers.{i}."
        f32(p + "input_layernorm.weight", (h,), _randn(g, h) * 0.1)
        f32(p + "post_attention_layernorm.weight", (h,), _randn(g, h) * 0.1)
        q4(p + "mlp.gate_up_proj.weight", 2 * inter, h)
        q4(p + "mlp.down_proj.weight", h, inter)
        if sched[i]:
            q4(p + "linear_attn.in_proj_all.weight", ch + v_dim + 2 * d.lin_v_heads, h)
            f32(p + "linear_attn.conv1d.weight", (ch, 1, d.lin_kernel), _randn(g, ch * d.lin_kernel) * 0.3)
            q4(p + "linear_attn.out_proj.weight", h, v_dim)
            f32(p + "linear_attn.norm.weight", (d.lin_v_dim,), 1.0 + _randn(g, d.lin_v_dim) * 0.1)
            f32(p + "linear_attn.A_log", (d.lin_v_heads,), torch.log(1.0 + 15.0 * _rand(g, d.lin_v_heads)))
            f32(p + "linear_attn.dt_bias", (d.lin_v_heads,), _randn(g, d.lin_v_heads) * 0.5)
        else:
            q4(p + "self_attn.qkv_proj.weight", 2 * (d.n_heads + d.n_kv_heads) * hd, h)
            q4(p + "self_attn.o_proj.weight", h, d.n_heads * hd)
            f32(p + "self_attn.q_norm.weight", (hd,), _randn(g, hd) * 0.1)
            f32(p + "self_attn.k_norm.weight", (hd,), _randn(g, hd) * 0.1)
    model.finalize()
    _MODELS[which] = model
    return model


class _Serving:
    """A runtime with its decode requests prefilled to their contexts."""

    def __init__(self, which, seed, contexts, chunk, step_rows):
        self.model = _model(which)
        vocab, page = self.model.dims.vocab, 16
        longest = max(int(contexts.max()) + 1, chunk)
        rng = np.random.default_rng(int(seed) + 1)
        n = contexts.size
        pages = [(int(c) + 1 + page - 1) // page for c in contexts] + ([(chunk + page - 1) // page] if chunk else [])
        self.rt = q.Runtime(self.model, max_slots=n + (chunk > 0), max_batch=n, max_context=longest, page_tokens=page,
                            total_pages=sum(pages), use_graphs=True, max_step_rows=step_rows)
        prompts = [rng.integers(0, vocab, size=int(c)).astype(np.int32) for c in contexts]
        if chunk:
            prompts.append(rng.integers(0, vocab, size=chunk).astype(np.int32))
        self.slots = [self.rt.slot_alloc(p) for p in prompts]
        self.table = np.zeros((len(prompts), self.rt.max_pages), np.int32)
        for r, count in enumerate(pages):
            self.table[r, :count] = [self.rt.page_alloc() for _ in range(count)]
        for r in range(n):
            for p0 in range(0, prompts[r].size, step_rows):
                self.rt.prefill(self.slots[r], p0, prompts[r][p0:p0 + step_rows], self.table[r])
        self.positions = contexts
        self.tokens = rng.integers(0, vocab, size=n).astype(np.int32)
        self.chunk = prompts[n] if chunk else None

    def __del__(self):
        rt = getattr(self, "rt", None)
        if rt is not None:
            rt.close()


# SamplingOptions' defaults: temperature 0.7, top_k 20, repetition penalty 1.05
TOP_K, INV_TEMPERATURE, PENALTY = 20, 1.0 / 0.7, 1.05

# ------------------------------------------------------------ prepare and run


def prepare(case, seed):
    ctx = _ctx()
    kind, g = case["kind"], _rng(seed)
    s = {"kind": kind, "case": case, "ctx": ctx}
    if kind in ("gemm", "head"):
        t, rows, cols = case["tokens"], case["rows"], case["cols"]
        x1 = kind == "gemm" and case["x1"]
        s["w"] = _Arg(_tiles(*_q4(g, rows, cols)))
        s["x"] = _Arg((_x1 if x1 else _x4)(*_q8(g, t, cols)))
        if kind == "gemm":
            s["out"] = _Arg(torch.zeros(t, rows, device="cuda"))
        else:
            counts = torch.zeros(t, rows, dtype=torch.int32, device="cuda")
            seen = torch.randint(0, rows, (t, 512), generator=g, device="cuda")
            s["counts"] = _Arg(counts.scatter_(1, seen, 1))
            s["penalties"] = _Arg(torch.full((t,), PENALTY, device="cuda"))
            s["index"] = _Arg(torch.zeros(t, dtype=torch.int32, device="cuda"))
            s["value"] = _Arg(torch.zeros(t, device="cuda"))
    elif kind == "prep":
        t, cols = case["tokens"], case["cols"]
        s["x"] = _Arg(_randn(g, t, cols))
        s["out"] = _Arg(torch.zeros((1, cols // 32, 40) if t == 1 else (t // 4, cols // 32, 152), dtype=torch.uint8,
                                    device="cuda"))
    elif kind == "delta":
        b, h = case["batch"], case["heads"]
        s["state"] = _randn(g, b, h, 128, 128) * 0.02
        first = s["state"].data_ptr()
        s["states"] = _Arg(torch.tensor([first + r * h * 128 * 128 * 4 for r in range(b)], dtype=torch.int64,
                                        device="cuda"))
        for name, scale in (("q", 1.0 / math.sqrt(128.0)), ("k", 1.0)):
            v = _randn(g, b, h, 128)
            s[name] = _Arg((v / v.norm(dim=-1, keepdim=True) * scale).contiguous())
        s["v"] = _Arg(_randn(g, b, h, 128))
        s["alpha"] = _Arg(torch.exp(-torch.nn.functional.softplus(_randn(g, b, h))))
        s["beta"] = _Arg(torch.sigmoid(_randn(g, b, h)))
        s["out"] = _Arg(torch.zeros(b, h, 128, device="cuda"))
    elif kind == "attention":
        lens, pt = _contexts(seed, case), case["page_tokens"]
        need = [(int(n) + pt - 1) // pt for n in lens]
        perm = torch.randperm(sum(need), generator=torch.Generator().manual_seed(int(seed))).to(torch.int32)
        table = torch.zeros(len(need), max(need), dtype=torch.int32)
        at = 0
        for r, n in enumerate(need):
            table[r, :n] = perm[at:at + n]
            at += n
        shape = (sum(need), pt, case["kv_heads"], HEAD_DIM)
        s["k"], s["v"] = (_Arg(torch.randn(shape, generator=g, device="cuda", dtype=torch.float16)) for _ in "kv")
        s["q"], s["gates"] = (_Arg(_randn(g, case["batch"], case["heads"], HEAD_DIM)) for _ in "qg")
        s["table"], s["max_pages"] = _Arg(table.cuda()), max(need)
        s["lens"] = _Arg(torch.from_numpy(lens).cuda())
        s["out"] = _Arg(torch.zeros(case["batch"], case["heads"], HEAD_DIM, device="cuda"))
    elif kind == "conv":
        t, ch = case["tokens"], case["channels"]
        s["state"] = _Arg(_randn(g, 3, ch))
        s["x"], s["w"] = _Arg(_randn(g, t, ch)), _Arg(_randn(g, 4, ch) * 0.3)
        s["out"] = _Arg(torch.zeros(t, ch, device="cuda"))
    elif kind == "mlp":
        t, h, i = case["tokens"], case["hidden"], case["inter"]
        s["gate"], s["up"] = (_Arg(_tiles(*_q4(g, i, h, 0.05))) for _ in "gu")
        s["down"] = _Arg(_tiles(*_q4(g, h, i, 0.05)))
        s["x"], s["norm"] = _Arg(_randn(g, t, h)), _Arg(_randn(g, h) * 0.1)
        s["normed"], s["y"] = (_Arg(torch.zeros(t, h, device="cuda")) for _ in "ny")
        s["a"], s["b"], s["act"] = (_Arg(torch.zeros(t, i, device="cuda")) for _ in "abc")
        s["xh"], s["xi"] = (_Arg(torch.zeros(t // 4, n // 32, 152, dtype=torch.uint8, device="cuda")) for n in (h, i))
    elif kind == "decode":
        v = _Serving("decode", seed, _contexts(seed, case), 0, 512)
        s["serving"], s["penalties"] = v, np.full(v.tokens.size, PENALTY, np.float32)
    else:
        v = _Serving("packed", seed, _contexts(seed, case), case["chunk"], 64 + 2048)
        n = v.tokens.size
        # the prompt chunk first (as a scheduler admits it), then the decode rows
        s["segments"] = [dict(slot=v.slots[n], pos0=0, tokens=v.chunk, page_table=v.table[n], penalty=PENALTY)]
        s["segments"] += [dict(slot=v.slots[r], pos0=int(v.positions[r]), tokens=v.tokens[r:r + 1],
                               page_table=v.table[r], penalty=PENALTY) for r in range(n)]
        s["serving"], s["sampling"] = v, [(TOP_K, INV_TEMPERATURE)] * (n + 1)
    return s


def run(s):
    ctx, case, kind = s["ctx"], s["case"], s["kind"]
    if kind == "gemm":
        t, rows, nb = case["tokens"], case["rows"], case["cols"] // 32
        if t == 1:
            q.q4_dot4_matvec(ctx, s["w"], s["x"], s["out"], rows, nb)
        elif case["x1"]:
            q.q4_dot4_matmul_x1(ctx, s["w"], s["x"], s["out"], rows, t, nb, rows)
        else:
            q.q4_dot4_matmul(ctx, s["w"], s["x"], s["out"], rows, t, nb, rows)
        return s["out"].tensor
    if kind == "head":
        q.q4_dot4_argmax_batch(ctx, s["w"], s["x"], s["counts"], s["penalties"], case["rows"], case["tokens"],
                               case["cols"] // 32, s["index"], s["value"])
        return {"index": s["index"].tensor, "value": s["value"].tensor}
    if kind == "prep":
        t, cols = case["tokens"], case["cols"]
        if t == 1 and case["h128"]:
            q.q4_h128_prepare_activation_1(ctx, s["x"], s["out"], cols)
        elif t == 1:
            q.q8_0_quantize_vector_1(ctx, s["x"], s["out"], cols // 32)
        elif case["h128"]:
            q.q4_h128_prepare_activations_4(ctx, s["x"], s["out"], t, cols)
        else:
            q.q8_0_quantize_vectors_4(ctx, s["x"], s["out"], t, cols // 32)
        return s["out"].tensor
    if kind == "delta":
        q.gated_delta_net_update_batch(ctx, s["states"], s["q"], s["k"], s["v"], s["alpha"], s["beta"], s["out"],
                                       case["batch"], case["heads"], 128, 128)
        return {"out": s["out"].tensor, "state": s["state"]}
    if kind == "attention":
        q.attention_decode_paged(ctx, s["q"], s["gates"], s["k"], s["v"], s["table"], s["max_pages"], s["lens"],
                                 case["page_tokens"], s["out"], case["batch"], case["heads"], case["kv_heads"],
                                 HEAD_DIM, 1.0 / 16.0)
        return s["out"].tensor
    if kind == "conv":
        q.causal_conv1d_silu_f32(ctx, s["state"], 0, s["x"], s["w"], s["out"], case["channels"], 4,
                                 batch=case["tokens"])
        return {"out": s["out"].tensor, "state": s["state"].tensor}
    if kind == "mlp":
        t, h, i = case["tokens"], case["hidden"], case["inter"]
        q.rms_norm_f32(ctx, s["x"], s["norm"], s["normed"], t, h, 1e-6, 1.0)
        q.q4_h128_prepare_activations_4(ctx, s["normed"], s["xh"], t, h)
        q.q4_dot4_matmul(ctx, s["gate"], s["xh"], s["a"], i, t, h // 32, i)
        q.q4_dot4_matmul(ctx, s["up"], s["xh"], s["b"], i, t, h // 32, i)
        q.silu_mul_f32(ctx, s["a"], s["b"], s["act"], t * i)
        q.q4_h128_prepare_activations_4(ctx, s["act"], s["xi"], t, i)
        q.q4_dot4_matmul(ctx, s["down"], s["xi"], s["y"], h, t, i // 32, h)
        return {"act": s["act"].tensor, "y": s["y"].tensor}
    # The candidates' logits in descending order; the token ids beside them are
    # left out, since near ties trade places. A pass repeats the same
    # positions: a step reads the recurrent state of its position and writes
    # the next one's, so it finds the same state again.
    v = s["serving"]
    if kind == "decode":
        cand = v.rt.step_candidates(v.slots, v.positions, v.tokens, v.table, TOP_K, INV_TEMPERATURE,
                                    penalties=s["penalties"])
    else:
        cand = v.rt.step_segments(s["segments"], sampling=s["sampling"])
    return {"logits": cand["value"]}


# ------------------------------------------------------------ what it cannot do without


def _tile_bytes(rows, cols):
    return rows / 8 * (cols / 32) * 144


def _model_work(which, rows, heads, kv_tokens):
    """Weights once, the requests' state and cached rows once each way, and
    the projections' products."""
    d, sched = q.model_dims(0 if which == "decode" else 2)
    if which == "packed":
        d.n_layers, d.vocab = 4, 32768
        sched = np.array([1, 1, 1, 0], np.uint8)
    lin, full = int(sched.sum()), int(d.n_layers - sched.sum())
    h, i = d.hidden, d.intermediate
    v_dim, qw = d.lin_v_heads * d.lin_v_dim, d.n_heads * d.head_dim
    kvw = d.n_kv_heads * d.head_dim
    ch = 2 * d.lin_k_heads * d.lin_k_dim + v_dim
    weights = lin * ((ch + v_dim + 2 * d.lin_v_heads) * h + h * v_dim) + full * (2 * (qw + kvw) * h + h * qw)
    weights += d.n_layers * 3 * i * h
    head = d.vocab * h
    state = lin * heads * (2 * d.lin_v_heads * d.lin_v_dim * d.lin_k_dim + 2 * d.lin_kernel * ch) * 4
    cache = full * kv_tokens * kvw * 2 * 2
    out = heads * 64 * 8
    flops = 2.0 * rows * weights + 2.0 * heads * head + lin * rows * d.lin_v_heads * d.lin_v_dim * d.lin_k_dim * 7.0
    return {"bytes": (weights + head) * 0.5625 + state + cache + out, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind in ("gemm", "head"):
        t, rows, cols = case["tokens"], case["rows"], case["cols"]
        acts = t * (cols // 32) * (40 if kind == "gemm" and case["x1"] else 38)
        out = t * rows * 4 if kind == "gemm" else t * rows * 4 + t * 12  # head: penalty counts in, index and value out
        return {"bytes": _tile_bytes(rows, cols) + acts + out, "flops": 2.0 * t * rows * cols}
    if kind == "prep":
        n = case["tokens"] * case["cols"]
        return {"bytes": n * 4 + n / 32 * (40 if case["tokens"] == 1 else 38), "flops": n * (11.0 if case["h128"] else 4.0)}
    if kind == "delta":
        n = case["batch"] * case["heads"]
        return {"bytes": n * (2 * 128 * 128 + 4 * 128 + 2) * 4.0, "flops": n * 128 * 128 * 7.0}
    if kind == "attention":
        mean = case["batch"] * (case["min_context"] + case["max_context"]) / 2
        return {"bytes": mean * case["kv_heads"] * HEAD_DIM * 4.0 + case["batch"] * case["heads"] * HEAD_DIM * 12.0,
                "flops": 4.0 * mean * case["heads"] * HEAD_DIM}
    if kind == "conv":
        return {"bytes": (2 * case["tokens"] + 10) * case["channels"] * 4.0, "flops": case["tokens"] * case["channels"] * 12.0}
    if kind == "mlp":
        t, h, i = case["tokens"], case["hidden"], case["inter"]
        return {"bytes": 3 * _tile_bytes(i, h) + t * (2 * h + i) * 4.0, "flops": 6.0 * t * h * i}
    mean = (case["min_context"] + case["max_context"]) / 2
    n = case["batch"]
    if kind == "decode":
        return _model_work("decode", n, n, n * mean)
    return _model_work("packed", n + case["chunk"], n + 1, n * mean + case["chunk"])


def tolerance(case):
    # the sums' errors against 64 bits are 7e-8 to 1.1e-7 (fp32 chains over
    # the K blocks or the 128 columns of a state row), 3.3e-7 for attention
    kind = case["kind"]
    if kind == "prep":
        return "exact"
    if kind == "gemm":
        return {"rel": 5e-7, "max": 1e-5}
    if kind == "head":
        return {"rel": 5e-7, "max": 1e-6}
    if kind in ("delta", "conv"):
        return {"rel": 5e-7, "max": 1e-5}
    if kind == "attention":
        return {"rel": 2e-6, "max": 5e-5}
    if kind == "mlp":
        # a value within rounding of a code boundary takes the next int8 code:
        # 1.1e-4 (act) and 4.7e-4 (y) against 64 bits
        return {"rel": 2e-3, "max": 3e-2}
    # whole models: norm weights changed by one unit in the last place move the
    # logits by 8.7e-3 (24 layers) and 3.9e-3 (4 layers), at most 2.8e-2 and 1.4e-2
    return {"rel": 3e-2, "max": 0.11} if kind == "decode" else {"rel": 1.6e-2, "max": 5.5e-2}


# ------------------------------------------------------------------ in 64 bits


def _silu(x):
    return x * torch.sigmoid(x)


def _mask(v):
    return v & 0xFFFFFFFFFFFFFFFF


def _splitmix64(v):
    v = _mask(v + 0x9E3779B97F4A7C15)
    v = _mask((v ^ (v >> 30)) * 0xBF58476D1CE4E5B9)
    v = _mask((v ^ (v >> 27)) * 0x94D049BB133111EB)
    return v ^ (v >> 31)


def _rotate(x):
    """Random signs and the Hadamard transform of every 128 columns (unscaled)."""
    cols = x.shape[-1]
    sign = []
    for block in range(cols // 128):
        for word in range(2):
            bits = _splitmix64(_mask(SEED64 + block * 0x9E3779B97F4A7C15 + word * 0xD1B54A32D192ED03))
            sign += [-1.0 if bits >> e & 1 else 1.0 for e in range(64)]
    had = torch.ones(1, 1, dtype=torch.float64, device="cuda")
    for _ in range(7):
        had = torch.cat([torch.cat([had, had], 1), torch.cat([had, -had], 1)], 0)
    y = (x * torch.tensor(sign, dtype=torch.float64, device="cuda")).reshape(-1, 128) @ had
    return y.reshape(x.shape)


def _prepared(x):
    """What the int8 activations of x stand for, in the rotated basis."""
    v = _rotate(x).reshape(x.shape[0], -1, 32)
    scale = v.abs().amax(dim=-1) / 127.0
    r = v / scale.unsqueeze(-1)
    codes = torch.clamp(torch.sign(r) * torch.floor(r.abs() + 0.5), -127, 127)
    return (codes * (scale.to(torch.float16).double() / math.sqrt(128.0)).unsqueeze(-1)).reshape(x.shape)


def exact(case, seed):
    kind, g = case["kind"], _rng(seed)
    if kind == "gemm" or kind == "head":
        w = _dequant(*_q4(g, case["rows"], case["cols"]))
        codes, scales = _q8(g, case["tokens"], case["cols"])
        y = (codes.double() * scales.double().unsqueeze(-1)).reshape(case["tokens"], -1) @ w.t().contiguous()
        if kind == "gemm":
            return y
        seen = torch.randint(0, case["rows"], (case["tokens"], 512), generator=g, device="cuda")
        hit = torch.zeros(y.shape, dtype=torch.bool, device="cuda").scatter_(1, seen, True)
        pen = float(np.float32(PENALTY))
        y = torch.where(hit, torch.where(y > 0, y / pen, y * pen), y)
        return {"index": None, "value": y.amax(dim=1)}
    if kind == "delta":
        s = prepare(case, seed)
        st = s["state"].double() * s["alpha"].tensor.double()[..., None, None]
        k, qq = s["k"].tensor.double(), s["q"].tensor.double()
        delta = (s["v"].tensor.double() - (st * k.unsqueeze(-2)).sum(-1)) * s["beta"].tensor.double().unsqueeze(-1)
        st = st + delta.unsqueeze(-1) * k.unsqueeze(-2)
        return {"out": (st * qq.unsqueeze(-2)).sum(-1), "state": st}
    if kind == "attention":
        s = prepare(case, seed)
        kv, rep = case["kv_heads"], case["heads"] // case["kv_heads"]
        out = []
        for r, n in enumerate(_contexts(seed, case)):
            pages = s["table"].tensor[r, :(int(n) + case["page_tokens"] - 1) // case["page_tokens"]].long()
            keys, values = (s[x].tensor[pages].reshape(-1, kv, HEAD_DIM)[:int(n)].permute(1, 0, 2).double().contiguous()
                            for x in "kv")
            qq = s["q"].tensor[r].double().reshape(kv, rep, HEAD_DIM)
            p = torch.softmax(torch.matmul(qq, keys.transpose(1, 2).contiguous()) / 16.0, dim=-1)
            out.append(torch.matmul(p, values).reshape(-1, HEAD_DIM))
        return torch.stack(out) * torch.sigmoid(s["gates"].tensor.double())
    if kind == "conv":
        s = prepare(case, seed)
        x = torch.cat([s["state"].tensor, s["x"].tensor]).double()
        w, t = s["w"].tensor.double(), case["tokens"]
        y = sum(x[k:k + t] * w[k] for k in range(4))
        last = torch.zeros(3, case["channels"], dtype=torch.float64, device="cuda")
        for p in range(t - 3, t):  # slot of position p: p % 3
            last[p % 3] = x[p + 3]
        return {"out": _silu(y), "state": last}
    if kind == "mlp":
        t, h, i = case["tokens"], case["hidden"], case["inter"]
        gate, up = (_dequant(*_q4(g, i, h, 0.05)) for _ in "gu")
        down = _dequant(*_q4(g, h, i, 0.05))
        x, norm = _randn(g, t, h).double(), (_randn(g, h) * 0.1).double()
        n = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * (1.0 + norm)
        n = _prepared(n)
        act = _silu(n @ gate.t().contiguous()) * (n @ up.t().contiguous())
        return {"act": act, "y": _prepared(act) @ down.t().contiguous()}
    return None  # prepared bytes are exact by themselves; a whole model has no short 64-bit form
