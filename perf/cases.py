"""What this framework is timed on: the calls of a Qwen3.5 Q8_0 program.

A program holds a context, resident Q8_0 / fp16 weights and the layer objects,
and then decodes (one sequence or a batch), prefills prompts, or calls single
operations of the device ABI on its own device buffers.  Each case is one of
those calls at one size; ``draw`` gives further sizes of the same ranges.

Shapes are those of ``fortai_amd.synth.CONFIGS`` (the 0.8B and the 4B layer
shapes; whole-model prefill and batch cases keep one attention interval, four
layers, of the depth) and generic odd ones.  Weights follow the distributions
of ``fortai_amd.synth``: uniform int8 quants, log-uniform fp16 block scales.
"""

import math
from dataclasses import replace

import numpy as np
import torch

from fortai_amd import backend as B
from fortai_amd import synth

DEV = "cuda"


# ------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest calls: two Q8_0 projections of one token (FFN gate and up, 0.8B)
        {"name": "matvec_2x3584x1024", "kind": "matvec", "rows": 3584, "width": 1024, "batch": 1, "noalloc": False},
        # a serving loop's projection of five sequences (FFN down, 4B)
        {"name": "batch_matvec_5x2560x9216", "kind": "matvec", "rows": 2560, "width": 9216, "batch": 5,
         "noalloc": True},
        # one token through the reference's per-operation ABI (the drop-in path)
        {"name": "ops_token_0.8b", "kind": "ops", "model": "qwen35-0.8b-short", "position": 777},
        # greedy decoding of one sequence near the end of a 4096-position context: the headline
        {"name": "decode_0.8b_ctx4096", "kind": "decode", "model": "qwen35-0.8b", "layers": 24, "position": 4080,
         "steps": 8},
        # a decode step of eight sequences after a 512-token prompt
        {"name": "decode_batch8_4b", "kind": "batch", "model": "qwen35-4b-short", "batch": 8, "prompt": 512,
         "steps": 8},
        # prompts of a batch of requests, exact (the default mode)
        {"name": "prefill_4b_8x512", "kind": "prefill", "model": "qwen35-4b-short", "batch": 8, "prompt": 512,
         "mode": "exact"},
        # a short chat prompt of one user
        {"name": "prefill_0.8b_1x77", "kind": "prefill", "model": "qwen35-0.8b-short", "batch": 1, "prompt": 77,
         "mode": "exact"},
        # the non-bit-exact mode, ragged lengths
        {"name": "prefill_fast_4b_3x701", "kind": "prefill", "model": "qwen35-4b-short", "batch": 3, "prompt": 701,
         "mode": "fast"},
        # one large token-block projection (FFN gate, 4B, eight 512-token prompts)
        {"name": "mmq_9216x2560x4096", "kind": "mmq", "rows": 9216, "width": 2560, "tokens": 4096, "exact": False,
         "residual": False},
        # causal attention of a long document's prompt in one layer
        {"name": "attention_prompt_2000", "kind": "attention_prompt", "heads": 8, "kv_heads": 2, "tokens": 2000,
         "matrix_cores": False},
        # decode attention of one layer deep in a long context
        {"name": "attention_step_32768", "kind": "attention_step", "heads": 8, "kv_heads": 2, "length": 32768},
        # the delta rule of one layer over a block of tokens
        {"name": "gdn_steps_128", "kind": "gdn", "key_heads": 16, "value_heads": 16, "steps": 128},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["matvec", "ops", "decode", "batch", "prefill", "prefill", "prefill", "mmq", "mmq",
                       "attention_prompt", "attention_step", "gdn"])
    heads, kv_heads = rng.choice([(8, 2), (16, 4)])
    if kind == "matvec":
        return {"kind": kind, "rows": _log(rng, 900, 9300), "width": 32 * _log(rng, 24, 288),
                "batch": rng.choice([1, 1, 2, 3, 4, 5, 6, 7, 8]), "noalloc": rng.random() < 0.5}
    if kind == "ops":
        return {"kind": kind, "model": rng.choice(["qwen35-0.8b-short", "qwen35-4b-short"]),
                "position": _log(rng, 1, 4000)}
    if kind == "decode":
        return {"kind": kind, "model": "qwen35-0.8b", "layers": 4 * rng.randint(1, 6),
                "position": _log(rng, 1, 8000), "steps": rng.randint(1, 8)}
    if kind == "batch":
        return {"kind": kind, "model": rng.choice(["qwen35-0.8b-short", "qwen35-4b-short"]),
                "batch": rng.randint(1, 8), "prompt": _log(rng, 8, 1500), "steps": rng.randint(1, 8)}
    if kind == "prefill":
        tokens = _log(rng, 1, 4096)
        batch = rng.randint(1, 8) if tokens >= 8 else 1
        return {"kind": kind, "model": rng.choice(["qwen35-0.8b-short", "qwen35-4b-short"]), "batch": batch,
                "prompt": min(2048, max(1, tokens // batch)), "mode": rng.choice(["exact", "exact", "fast"])}
    if kind == "mmq":
        rows, width = rng.choice([(9216, 2560), (2560, 9216), (8192, 2560), (2560, 4096), (3584, 1024), (1024, 3584),
                                  (6144, 1024), (1024, 2048), (_log(rng, 500, 9000), 32 * _log(rng, 24, 128))])
        return {"kind": kind, "rows": rows, "width": width, "tokens": _log(rng, 1, 4096),
                "exact": rng.random() < 0.6, "residual": rng.random() < 0.5}
    if kind == "attention_prompt":
        return {"kind": kind, "heads": heads, "kv_heads": kv_heads, "tokens": _log(rng, 16, 2200),
                "matrix_cores": rng.random() < 0.4}
    if kind == "attention_step":
        return {"kind": kind, "heads": heads, "kv_heads": kv_heads, "length": _log(rng, 16, 65536)}
    return {"kind": kind, "key_heads": 16, "value_heads": rng.choice([16, 32]), "steps": _log(rng, 1, 512)}


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(0x51E5 + 7919 * int(seed))
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _q8_blocks(g, rows, width):
    """GGUF Q8_0 bytes [rows][width/32][34] on the device."""
    blocks = width // 32
    out = torch.empty(rows, blocks, 34, dtype=torch.uint8, device=DEV)
    out[:, :, 2:] = torch.randint(-127, 128, (rows, blocks, 32), dtype=torch.int8, generator=g, device=DEV).view(torch.uint8)
    magnitude = torch.exp(torch.rand(rows, blocks, generator=g, device=DEV) * math.log(100.0) + math.log(1e-3))
    sign = torch.randint(0, 2, (rows, blocks), generator=g, device=DEV) * 2 - 1
    out[:, :, :2] = (magnitude * sign).half().unsqueeze(-1).view(torch.uint8)
    return out


def _q8(ctx, g, rows, width):
    return B.Q8Weights(ctx, _q8_blocks(g, rows, width).cpu().numpy(), rows, width)


def _ones(g, n):
    return (1.0 + 0.05 * _normal(g, n)).cpu().numpy()


def _gdn_constants(g, value_heads, conv_size):
    ssm_a = (-torch.exp(0.5 * _normal(g, value_heads))).cpu().numpy()
    ssm_dt = _normal(g, value_heads).cpu().numpy()
    conv_w = (0.1 * _normal(g, conv_size, 4)).cpu().numpy()
    return ssm_a, ssm_dt, conv_w


_CONTEXT = None


def _context():
    """The program's one context: its calls run in order on one stream."""
    global _CONTEXT
    if _CONTEXT is None:
        _CONTEXT = B.Context(0)
    return _CONTEXT


class _Held:
    """What a program holds for one case beside its context; given back with it."""

    def __init__(self):
        self.ctx = _context()
        self._owned = []

    def own(self, x):
        self._owned.append(x)
        return x

    def q8(self, g, rows, width):
        return self.own(_q8(self.ctx, g, rows, width))

    def __del__(self):
        try:
            for x in reversed(self._owned):
                x.free()
        except Exception:
            pass


def _model(held, g, cfg, max_context):
    """Weights and layer objects of a model of this shape."""
    c, held.cfg, h = held.ctx, cfg, cfg.hidden
    held.layers = []
    for i in range(cfg.layers):
        L = {"attn_norm": _ones(g, h), "post_norm": _ones(g, h), "gate": held.q8(g, cfg.ffn, h),
             "up": held.q8(g, cfg.ffn, h), "down": held.q8(g, h, cfg.ffn), "rec": None, "att": None}
        if cfg.recurrent(i):
            qkv, z = held.q8(g, cfg.conv_size, h), held.q8(g, cfg.gdn_inner, h)
            alpha, beta = held.q8(g, cfg.gdn_value_heads, h), held.q8(g, cfg.gdn_value_heads, h)
            out = held.q8(g, h, cfg.gdn_inner)
            ssm_a, ssm_dt, conv_w = _gdn_constants(g, cfg.gdn_value_heads, cfg.conv_size)
            L["rec"] = held.own(B.Recurrent(c, qkv, z, alpha, beta, out, conv_w, cfg.conv_size, cfg.conv_kernel,
                                            ssm_a, ssm_dt, _ones(g, cfg.gdn_head), cfg.gdn_state, cfg.gdn_key_heads,
                                            cfg.gdn_value_heads, cfg.gdn_head, cfg.gdn_inner, cfg.eps))
        else:
            q = held.q8(g, 2 * cfg.heads * cfg.head_size, h)
            k, v = held.q8(g, cfg.kv_heads * cfg.head_size, h), held.q8(g, cfg.kv_heads * cfg.value_size, h)
            o = held.q8(g, h, cfg.heads * cfg.value_size)
            L["att"] = held.own(B.Attention(c, q, k, v, o, _ones(g, cfg.head_size), _ones(g, cfg.head_size),
                                            cfg.heads, cfg.kv_heads, cfg.head_size, cfg.value_size, max_context,
                                            cfg.rope_dim, cfg.rope_base, cfg.eps))
        held.layers.append(L)
    table = (0.02 * torch.randn(cfg.vocab, h, generator=g, device=DEV)).half().cpu().numpy()
    held.embedding = held.own(B.F16Weights(c, table.view(np.uint16), cfg.vocab, h))
    held.output_norm = _ones(g, h)
    return held


def _decoder_arguments(held, max_context):
    pick = lambda key: [L[key] for L in held.layers]
    cfg = held.cfg
    return (pick("rec"), pick("att"), pick("gate"), pick("up"), pick("down"), pick("attn_norm"), pick("post_norm"),
            held.output_norm, cfg.hidden, held.embedding, held.embedding, max_context, cfg.eps, cfg.vocab)


def _random_cache(g, positions, kv_heads, width):
    return _normal(g, positions, kv_heads, width).half().view(torch.int16).cpu().numpy().view(np.uint16)


def _fill_cache(g, att, positions):
    d = att.dims
    if positions > 0:
        att.set_cache(_random_cache(g, positions, d["kv_heads"], d["head_size"]),
                      _random_cache(g, positions, d["kv_heads"], d["value_size"]), positions)


def _ptr(t):
    return t.data_ptr()


def _logits(held, name, decoder, like):
    """The decoder's device logits copied into a buffer of the program's own."""
    p = B.C.c_void_p()
    held.ctx.call(name, decoder.h, B.C.byref(p))
    held.ctx.call("fortai_hip_qwen35_copy_device", held.ctx.h, p, _ptr(like), like.numel() * 4)
    return like


# ----------------------------------------------------------------- prepare
def prepare(case, seed):
    g = _generator(seed)
    held = _Held()
    held.case = case
    globals()["_prepare_" + case["kind"]](held, g, case)
    torch.cuda.synchronize()
    return held


def _matrices(case):
    """A single token's activation goes through two matrices (gate and up), a batch's through one."""
    return 2 if case["batch"] == 1 else 1


def _prepare_matvec(held, g, case):
    rows, width, batch = case["rows"], case["width"], case["batch"]
    held.w = [held.q8(g, rows, width) for _ in range(_matrices(case))]
    held.x = _normal(g, batch, width)
    held.out = [torch.empty(batch, rows, device=DEV) for _ in held.w]


def _prepare_ops(held, g, case):
    cfg = synth.CONFIGS[case["model"]]
    pos = case["position"]
    _model(held, g, cfg, pos + 64)
    for L in held.layers:
        if L["att"] is not None:
            _fill_cache(g, L["att"], pos)
        for key in ("attn_norm", "post_norm"):
            L[key + "_dev"] = torch.from_numpy(L[key]).to(DEV)
    held.norm_dev = torch.from_numpy(held.output_norm).to(DEV)
    for name in ("x", "residual", "normalized", "hidden"):
        setattr(held, name, torch.zeros(cfg.hidden, device=DEV))
    held.logits = torch.empty(cfg.vocab, device=DEV)
    held.next = torch.zeros(1, dtype=torch.int64, device=DEV)
    held.token = int(torch.randint(0, cfg.vocab, (1,), generator=g, device=DEV))


def _prepare_decode(held, g, case):
    cfg = replace(synth.CONFIGS[case["model"]], layers=case["layers"])
    pos, ctx = case["position"], case["position"] + case["steps"]
    _model(held, g, cfg, ctx)
    held.decoder = held.own(B.Decoder(held.ctx, *_decoder_arguments(held, ctx)))
    held.decoder.reset()
    for L in held.layers:
        if L["att"] is not None:
            _fill_cache(g, L["att"], pos)
    held.token = int(torch.randint(0, cfg.vocab, (1,), generator=g, device=DEV))
    held.logits = torch.empty(cfg.vocab, device=DEV)


def _prepare_batch(held, g, case):
    cfg, batch, prompt = synth.CONFIGS[case["model"]], case["batch"], case["prompt"]
    ctx = prompt + case["steps"]
    _model(held, g, cfg, ctx)
    held.batch = held.own(B.BatchDecoder(held.ctx, batch, *_decoder_arguments(held, ctx)))
    held.batch.reset()
    tokens = torch.randint(0, cfg.vocab, (batch, prompt), generator=g, device=DEV).cpu().numpy()
    held.first, _ = held.batch.prefill(tokens, want_logits=False)
    # sequences of different lengths: up to a third shorter than the longest
    short = torch.randint(0, prompt // 3 + 1, (batch,), generator=g, device=DEV).cpu().numpy()
    short[0] = 0
    held.positions = (prompt - short).astype(np.int32)
    held.logits = torch.empty(batch, cfg.vocab, device=DEV)


def _prepare_prefill(held, g, case):
    cfg, batch, prompt = synth.CONFIGS[case["model"]], case["batch"], case["prompt"]
    ctx = prompt + 1
    _model(held, g, cfg, ctx)
    held.batch = held.own(B.BatchDecoder(held.ctx, batch, *_decoder_arguments(held, ctx)))
    held.batch.set_prefill_mode(case["mode"])
    held.tokens = torch.randint(0, cfg.vocab, (batch, prompt), generator=g, device=DEV).cpu().numpy()
    held.positions = np.full(batch, prompt, dtype=np.int32)
    held.prompt_logits = torch.empty(batch, cfg.vocab, device=DEV)
    held.logits = torch.empty(batch, cfg.vocab, device=DEV)


def _prepare_mmq(held, g, case):
    rows, width, tokens = case["rows"], case["width"], case["tokens"]
    held.w = held.q8(g, rows, width)
    held.x = _normal(g, tokens, width)
    held.residual = 100.0 * _normal(g, tokens, rows) if case["residual"] else None
    held.q = torch.empty(B.load().fortai_hip_q8_tokens_bytes(tokens, width), dtype=torch.uint8, device=DEV)
    held.out = torch.empty(tokens, rows, device=DEV)


def _attention_layer(held, g, case, max_context):
    heads, kv_heads, head = case["heads"], case["kv_heads"], 256
    q, k, v = (held.q8(g, n * head, 32) for n in (2 * heads, kv_heads, kv_heads))
    held.q_norm, held.k_norm = _ones(g, head), _ones(g, head)
    held.att = held.own(B.Attention(held.ctx, q, k, v, held.q8(g, 32, heads * head), held.q_norm, held.k_norm, heads,
                                    kv_heads, head, head, max_context, 64, 1.0e7, 1e-6))


def _prepare_attention_prompt(held, g, case):
    heads, kv_heads, T = case["heads"], case["kv_heads"], case["tokens"]
    _attention_layer(held, g, case, T)
    held.q_in = _normal(g, T, heads, 2, 256)
    held.k, held.v = _normal(g, T, kv_heads, 256), _normal(g, T, kv_heads, 256)
    held.q = torch.empty_like(held.q_in)
    held.out = torch.empty(T, heads, 256, device=DEV)


def _prepare_attention_step(held, g, case):
    heads, kv_heads, length = case["heads"], case["kv_heads"], case["length"]
    _attention_layer(held, g, case, length)
    held.keys, held.values = _random_cache(g, length, kv_heads, 256), _random_cache(g, length, kv_heads, 256)
    held.att.set_cache(held.keys, held.values, length)
    held.q = _normal(g, heads, 2, 256)
    held.k, held.v = _normal(g, kv_heads, 256), _normal(g, kv_heads, 256)
    held.out = torch.empty(heads, 256, device=DEV)
    held.ctx.set_position(length - 1)


def _prepare_gdn(held, g, case):
    kh, vh, steps, head = case["key_heads"], case["value_heads"], case["steps"], 128
    conv, inner = 2 * kh * head + vh * head, vh * head
    held.ssm_a, held.ssm_dt, held.conv_w = _gdn_constants(g, vh, conv)
    held.rec = held.own(B.Recurrent(held.ctx, held.q8(g, conv, 32), held.q8(g, inner, 32), held.q8(g, vh, 32),
                                    held.q8(g, vh, 32), held.q8(g, 32, inner), held.conv_w, conv, 4, held.ssm_a,
                                    held.ssm_dt, _ones(g, head), head, kh, vh, head, inner, 1e-6))
    held.state0 = (0.1 * _normal(g, vh * head * head)).cpu().numpy()
    held.conv0 = _normal(g, 3 * conv).cpu().numpy()
    held.rec.set_state(held.state0, held.conv0)
    held.qkv = _normal(g, steps, conv)
    held.alpha, held.beta = _normal(g, steps, vh), _normal(g, steps, vh)
    held.out = torch.empty(steps, inner, device=DEV)


# --------------------------------------------------------------------- run
def run(state):
    return globals()["_run_" + state.case["kind"]](state, state.ctx, state.ctx.h, state.case)


def _run_matvec(s, c, h, case):
    for w, out in zip(s.w, s.out):
        if case["noalloc"]:
            c.call("fortai_hip_q8_batch_matvec_noalloc", h, w.h, _ptr(s.x), case["batch"], _ptr(out))
        elif case["batch"] > 1:
            c.call("fortai_hip_q8_batch_matvec_device", h, w.h, _ptr(s.x), case["batch"], _ptr(out), None)
        else:
            c.call("fortai_hip_q8_matvec_device_f32", h, w.h, _ptr(s.x), case["width"], _ptr(out), case["rows"])
    return s.out


def _run_ops(s, c, h, case):
    cfg, H = s.cfg, s.cfg.hidden
    x, residual, normalized, hidden = (_ptr(t) for t in (s.x, s.residual, s.normalized, s.hidden))
    c.call("fortai_hip_qwen35_embedding_f16_device", h, s.embedding.h, s.token, x, H)
    c.set_position(case["position"])
    for L in s.layers:
        c.call("fortai_hip_qwen35_copy_device", h, x, residual, H * 4)
        c.call("fortai_hip_qwen35_rms_norm_device", h, x, _ptr(L["attn_norm_dev"]), normalized, H, cfg.eps)
        if L["rec"] is not None:
            c.call("fortai_hip_qwen35_recurrent_run_device", L["rec"].h, normalized, H, hidden, H)
        else:
            c.call("fortai_hip_qwen35_attention_run_device", L["att"].h, normalized, H, case["position"], hidden, H)
        c.call("fortai_hip_qwen35_add_device", h, hidden, residual, x, H)
        c.call("fortai_hip_qwen35_copy_device", h, x, residual, H * 4)
        c.call("fortai_hip_qwen35_rms_norm_device", h, x, _ptr(L["post_norm_dev"]), normalized, H, cfg.eps)
        c.call("fortai_hip_q8_ffn_device", h, L["gate"].h, L["up"].h, L["down"].h, normalized, H, hidden, H)
        c.call("fortai_hip_qwen35_add_device", h, hidden, residual, x, H)
    c.call("fortai_hip_qwen35_rms_norm_device", h, x, _ptr(s.norm_dev), normalized, H, cfg.eps)
    c.call("fortai_hip_f16_matvec_device", h, s.embedding.h, normalized, H, _ptr(s.logits), cfg.vocab, _ptr(s.next))
    return {"hidden": s.x, "logits": s.logits, "token": s.next}


def _run_decode(s, c, h, case):
    tokens = s.decoder.generate(s.token, case["position"], case["steps"])
    return {"tokens": tokens, "logits": _logits(s, "fortai_hip_qwen35_decoder_logits", s.decoder, s.logits)}


def _run_batch(s, c, h, case):
    tokens = s.batch.generate(s.first, s.positions, case["steps"])
    return {"tokens": tokens, "logits": _logits(s, "fortai_hip_qwen35_batch_logits", s.batch, s.logits)}


def _run_prefill(s, c, h, case):
    # a new prompt from position 0, and the first decode step on the states and caches it leaves
    s.batch.reset()
    s.batch.prefill(s.tokens, want_logits=False)
    _logits(s, "fortai_hip_qwen35_batch_logits", s.batch, s.prompt_logits)
    s.batch.generate(s.tokens[:, 0], s.positions, 1)
    _logits(s, "fortai_hip_qwen35_batch_logits", s.batch, s.logits)
    return {"prompt_logits": s.prompt_logits, "logits": s.logits}


def _run_mmq(s, c, h, case):
    c.call("fortai_hip_q8_quantize_tokens_device", h, _ptr(s.x), case["tokens"], case["width"], _ptr(s.q))
    c.call("fortai_hip_q8_mmq_exact_device" if case["exact"] else "fortai_hip_q8_mmq_device", h, s.w.h, _ptr(s.q),
           case["tokens"], _ptr(s.out), None if s.residual is None else _ptr(s.residual), None)
    return s.out


def _run_attention_prompt(s, c, h, case):
    # the call normalises and rotates q in place, so the q projection's output is written anew first
    c.call("fortai_hip_qwen35_copy_device", h, _ptr(s.q_in), _ptr(s.q), s.q.numel() * 4)
    c.call("fortai_hip_qwen35_attention_prefill_core_device", s.att.h, _ptr(s.q), _ptr(s.k), _ptr(s.v), case["tokens"],
           1 if case["matrix_cores"] else 0, _ptr(s.out))
    return {"out": s.out, "q": s.q}


def _run_attention_step(s, c, h, case):
    c.call("fortai_hip_qwen35_attention_core_device", s.att.h, _ptr(s.q), _ptr(s.k), _ptr(s.v), _ptr(s.out))
    return s.out


def _run_gdn(s, c, h, case):
    c.call("fortai_hip_qwen35_recurrent_core_steps_device", s.rec.h, _ptr(s.qkv), _ptr(s.alpha), _ptr(s.beta),
           case["steps"], _ptr(s.out))
    return s.out


# -------------------------------------------------------------------- work
def _layer_q8_values(cfg):
    """Q8_0 values of all layers, and the attention layers among them."""
    h, total, attention = cfg.hidden, 0, 0
    for i in range(cfg.layers):
        total += 3 * cfg.ffn * h
        if cfg.recurrent(i):
            total += (cfg.conv_size + 2 * cfg.gdn_inner + 2 * cfg.gdn_value_heads) * h
        else:
            attention += 1
            total += (3 * cfg.heads * cfg.head_size + 2 * cfg.kv_heads * cfg.head_size) * h
    return total, attention


def _step_work(cfg, batch, position):
    """One decode step of `batch` sequences at this position."""
    values, attention = _layer_q8_values(cfg)
    gdn = cfg.layers - attention
    state = cfg.gdn_value_heads * cfg.gdn_head ** 2
    kv = 2 * position * cfg.kv_heads * cfg.head_size * 2
    weights = values / 32 * 34 + cfg.vocab * cfg.hidden * 2
    per_sequence = gdn * 8 * (state + 3 * cfg.conv_size) + attention * kv + 4 * cfg.vocab
    flops = 2 * (values + cfg.vocab * cfg.hidden) + gdn * 7 * state + attention * 4 * position * cfg.heads * cfg.head_size
    return weights + batch * per_sequence, batch * flops


def work(case):
    kind = case["kind"]
    if kind == "matvec":
        n, m = case["rows"] * case["width"], _matrices(case)
        return {"bytes": m * n / 32 * 34 + 4 * case["batch"] * (m * case["rows"] + case["width"]),
                "flops": 2 * m * n * case["batch"]}
    if kind == "ops":
        moved, flops = _step_work(synth.CONFIGS[case["model"]], 1, case["position"])
        return {"bytes": moved, "flops": flops}
    if kind in ("decode", "batch"):
        cfg = synth.CONFIGS[case["model"]]
        if kind == "decode":
            cfg = replace(cfg, layers=case["layers"])
        moved, flops = _step_work(cfg, case.get("batch", 1), case.get("position", case.get("prompt")))
        return {"bytes": case["steps"] * moved, "flops": case["steps"] * flops}
    if kind == "prefill":
        cfg, batch, T = synth.CONFIGS[case["model"]], case["batch"], case["prompt"]
        values, attention = _layer_q8_values(cfg)
        gdn = cfg.layers - attention
        moved, flops = _step_work(cfg, batch, T)
        state = cfg.gdn_value_heads * cfg.gdn_head ** 2
        flops += batch * T * (2 * values + gdn * 7 * state + attention * 2 * (T + 1) * cfg.heads * cfg.head_size)
        moved += values / 32 * 34 + cfg.vocab * cfg.hidden * 2 + batch * 8 * T + batch * 4 * cfg.vocab
        return {"bytes": moved, "flops": flops}
    if kind == "mmq":
        n, t = case["rows"] * case["width"], case["tokens"]
        return {"bytes": n / 32 * 34 + 4 * t * (case["width"] + case["rows"] * (2 if case["residual"] else 1)),
                "flops": 2 * n * t}
    if kind == "attention_prompt":
        T, q, kv = case["tokens"], case["heads"] * 256, case["kv_heads"] * 256
        return {"bytes": T * (4 * (4 * q + 2 * kv + q) + 4 * kv), "flops": 2 * T * (T + 1) * q}
    if kind == "attention_step":
        q, kv = case["heads"] * 256, case["kv_heads"] * 256
        return {"bytes": 4 * case["length"] * kv + 4 * (3 * q + 2 * kv), "flops": 4 * case["length"] * q}
    state, conv = case["value_heads"] * 128 * 128, (2 * case["key_heads"] + case["value_heads"]) * 128
    return {"bytes": 8 * (state + 3 * conv) + 16 * conv + 4 * case["steps"] * (conv + case["value_heads"] * 130),
            "flops": case["steps"] * (7 * state + 8 * conv)}


# --------------------------------------------------------------- tolerance
def tolerance(case):
    """The framework's contract is the reference's summation orders, bit for
    bit, except for the split-K attention past 8192 positions, the whole-block
    token products and the matrix-core prompt attention."""
    kind = case["kind"]
    if kind == "attention_step" and case["length"] > 8192:
        return {"rel": 3e-6}  # 6e-7 off the 64-bit result
    if kind == "mmq" and not case["exact"]:
        return {"rel": 1e-6}  # 1.6e-7 off the 64-bit result
    if kind == "attention_prompt" and case["matrix_cores"]:
        return {"rel": 1e-3}  # fp16 q, k, v and probabilities: 2.4e-4 off the 64-bit result
    if kind == "prefill" and case["mode"] == "fast":
        return {"rel": 3e-2}  # int8 rounding moves with the sums: 8e-3 from the exact mode over four layers
    return "exact"


# ------------------------------------------------------------------- exact
def _dequantized(blocks):
    scale = blocks[:, :, :2].contiguous().view(torch.float16).double()
    quants = blocks[:, :, 2:].contiguous().view(torch.int8).double()
    return (scale * quants).reshape(blocks.shape[0], -1)


def _quantized(x):
    """x [n][width] through the Q8_0 quantizer (float32, fp16 block scales), as float64."""
    y = x.reshape(x.shape[0], -1, 32)
    amax = y.abs().amax(dim=2, keepdim=True)
    # the float32 quotients: float64 ones rounded once (the device's own float32 division may be off by an ulp)
    inverse = torch.where(amax != 0, (127.0 / amax.double()).float(), torch.zeros_like(amax))
    q = torch.clamp(torch.round(y * inverse), -128, 127).double()
    return (q * (amax.double() / 127.0).float().half().double()).reshape(x.shape)


def _silu(x):
    return x * torch.sigmoid(x)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("ops", "decode", "batch", "prefill"):
        # activations are rounded to int8 between the layers: 64-bit sums
        # round some of them to the neighbouring value, so there is no one result
        return None
    g = _generator(seed)
    return globals()["_exact_" + kind](g, case)


def _exact_matvec(g, case):
    ws = [_dequantized(_q8_blocks(g, case["rows"], case["width"])) for _ in range(_matrices(case))]
    x = _quantized(_normal(g, case["batch"], case["width"]))
    return [x @ w.t() for w in ws]


def _exact_mmq(g, case):
    w = _dequantized(_q8_blocks(g, case["rows"], case["width"]))
    x = _quantized(_normal(g, case["tokens"], case["width"]))
    out = x @ w.t()
    if case["residual"]:
        out += 100.0 * _normal(g, case["tokens"], case["rows"])
    return out


def _exact_attention_inputs(g, case):
    """The layer's norm weights; the generator moves on as in prepare."""
    for n in (2 * case["heads"], case["kv_heads"], case["kv_heads"]):
        _q8_blocks(g, n * 256, 32)
    norms = [torch.from_numpy(_ones(g, 256)).to(DEV).double() for _ in range(2)]
    _q8_blocks(g, 32, case["heads"] * 256)
    return norms


def _norm_rope(x, weight, positions):
    """Per-head RMSNorm and rotation of the first 64 dims; x [T][heads][256], float64."""
    x = x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + 1e-6) * weight
    # the angles are float32 values: position / base^(2i/64)
    exponent = (np.arange(0, 64, 2, dtype=np.float32) / np.float32(64)).astype(np.float64)
    power = (1.0e7 ** exponent).astype(np.float32)
    angle = torch.from_numpy((np.asarray(positions, dtype=np.float32)[:, None] / power).astype(np.float64)).to(DEV)
    c, s = torch.cos(angle)[:, None, :], torch.sin(angle)[:, None, :]
    a, b = x[..., :32].clone(), x[..., 32:64].clone()
    x = x.clone()
    x[..., :32], x[..., 32:64] = a * c - b * s, a * s + b * c
    return x


def _exact_attention_prompt(g, case):
    q_norm, k_norm = _exact_attention_inputs(g, case)
    heads, kv_heads, T = case["heads"], case["kv_heads"], case["tokens"]
    q_in = _normal(g, T, heads, 2, 256)
    k, v = _normal(g, T, kv_heads, 256).double(), _normal(g, T, kv_heads, 256).double()
    q = _norm_rope(q_in[:, :, 0].double(), q_norm, np.arange(T))
    k = _norm_rope(k, k_norm, np.arange(T)).float().half().double()
    v = v.float().half().double()
    mask = torch.ones(T, T, dtype=torch.bool, device=DEV).tril()
    out = torch.empty(T, heads, 256, dtype=torch.float64, device=DEV)
    for h in range(heads):
        kv = h // (heads // kv_heads)
        scores = (q[:, h].contiguous() @ k[:, kv].t().contiguous()) / 16.0
        p = torch.softmax(scores.masked_fill(~mask, -math.inf), dim=-1)
        out[:, h] = (p @ v[:, kv].contiguous()) * torch.sigmoid(q_in[:, h, 1].double())
    rotated = q_in.double()
    rotated[:, :, 0] = q
    return {"out": out, "q": rotated}


def _exact_attention_step(g, case):
    q_norm, k_norm = _exact_attention_inputs(g, case)
    heads, kv_heads, length = case["heads"], case["kv_heads"], case["length"]
    keys = torch.from_numpy(_random_cache(g, length, kv_heads, 256).view(np.float16)).to(DEV).double()
    values = torch.from_numpy(_random_cache(g, length, kv_heads, 256).view(np.float16)).to(DEV).double()
    q = _normal(g, heads, 2, 256).double()
    k, v = _normal(g, kv_heads, 256).double(), _normal(g, kv_heads, 256).double()
    keys[-1] = _norm_rope(k[None], k_norm, [length - 1])[0].float().half().double()
    values[-1] = v.float().half().double()
    rotated = _norm_rope(q[None, :, 0], q_norm, [length - 1])[0]
    out = torch.empty(heads, 256, dtype=torch.float64, device=DEV)
    for h in range(heads):
        kv = h // (heads // kv_heads)
        p = torch.softmax((keys[:, kv] @ rotated[h]) / 16.0, dim=0)
        out[h] = (p @ values[:, kv]) * torch.sigmoid(q[h, 1])
    return out


def _exact_gdn(g, case):
    kh, vh, steps, head = case["key_heads"], case["value_heads"], case["steps"], 128
    conv, inner = 2 * kh * head + vh * head, vh * head
    up = lambda a: torch.from_numpy(np.asarray(a)).to(DEV).double()
    ssm_a, ssm_dt, conv_w = (up(a) for a in _gdn_constants(g, vh, conv))
    for rows, width in ((conv, 32), (inner, 32), (vh, 32), (vh, 32), (32, inner)):
        _q8_blocks(g, rows, width)
    _ones(g, head)
    state = (0.1 * _normal(g, vh * head * head)).double().reshape(vh, head, head)
    window = _normal(g, 3 * conv).double().reshape(3, conv)
    qkv = _normal(g, steps, conv).double()
    alpha, beta = _normal(g, steps, vh).double(), _normal(g, steps, vh).double()
    seq = torch.cat([window, qkv])
    x = _silu(sum(seq[i:i + steps] * conv_w[:, i] for i in range(4)))
    q, k = x[:, :kh * head].reshape(steps, kh, head), x[:, kh * head:2 * kh * head].reshape(steps, kh, head)
    unit = lambda a: (a / torch.clamp(a.norm(dim=-1, keepdim=True), min=1e-6)).repeat_interleave(vh // kh, dim=1)
    q, k, v = unit(q), unit(k), x[:, 2 * kh * head:].reshape(steps, vh, head)
    decay = torch.exp(ssm_a * torch.nn.functional.softplus(alpha + ssm_dt))
    gate = torch.sigmoid(beta)
    out = torch.empty(steps, vh, head, dtype=torch.float64, device=DEV)
    for t in range(steps):
        state = state * decay[t][:, None, None]
        delta = (v[t] - (state * k[t][:, None, :]).sum(-1)) * gate[t][:, None]
        state = state + delta[:, :, None] * k[t][:, None, :]
        out[t] = (state * q[t][:, None, :]).sum(-1) / math.sqrt(head)
    return out.reshape(steps, inner)
