"""The work that users have this framework do, as cases that can be timed and compared: speech turns, prompt ingestion,
the vocoder, and token models of both designs.

`listed()` names the cases, `draw(rng)` gives further ones of the same ranges, `prepare` makes what a program has in hand
before the call, `run` is one pass through the public entry points, `work` what a pass cannot do without, `exact` the same
outputs in 64 bits from plain torch.  Weights and inputs are random (there are no checkpoints here); the sizes are Vui Nano,
its vocoder and the token models that bench.py measures."""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from vui_amd.codec import CodecConfig, QwenCodecDecoder, codec_state_dict_shapes
from vui_amd.engine import Engine, GenConfig
from vui_amd.lm import TokenLM
from vui_amd.lm_engine import TokenEngine
from vui_amd.model import Vui
from vui_amd.synthetic import nano_for_cache, sandwich_lm_config, state_dict_shapes, token_lm_config, token_lm_state_dict

DEV = "cuda"

# (width, heads, ff, dim, rot_dim, vdim, kv_rank, layers) and (width, heads, key groups, dim, ff, experts, top, layers)
SAKUPEL = {"w768": (768, 8, 2048, 64, 32, 96, 256, 8), "w1024": (1024, 8, 2816, 128, 64, 128, 512, 8),
           "w2048": (2048, 16, 4096, 128, 64, 128, 512, 8)}
MABIDRA = {"w768": (768, 8, 2, 96, 3072, 32, 4, 8), "w1024": (1024, 8, 2, 128, 4224, 32, 4, 8),
           "w2048": (2048, 16, 4, 128, 6144, 32, 4, 8)}
VOCAB = 2048


def listed():
    return [
        # one user, one assistant turn on an ingested voice prompt: the text is ingested, then frames are drawn (headline use)
        {"name": "turn_1row_bf16", "kind": "turn", "rows": 1, "weights": "bf16", "prefix": 576, "text": 23, "frames": 6},
        # a small server: four turns side by side
        {"name": "turn_4rows_bf16", "kind": "turn", "rows": 4, "weights": "bf16", "prefix": 700, "text": 9, "frames": 4},
        # a full server with quantised weights and caches of very different lengths
        {"name": "turn_16rows_int8", "kind": "turn", "rows": 16, "weights": "int8", "prefix": 2048, "text": 16, "frames": 4},
        # ingestion of a voice prompt: 512 frames of audio and 64 text tokens
        {"name": "prompt_576_bf16", "kind": "prompt", "weights": "bf16", "tokens": 576},
        # ingestion of a long conversation with quantised weights
        {"name": "prompt_1733_int8", "kind": "prompt", "weights": "int8", "tokens": 1733},
        # the vocoder beside a streamed turn: frames one at a time
        {"name": "voice_stream", "kind": "voice", "frames": 6, "codebooks": 16, "streamed": True},
        # the vocoder behind a rendered turn (or an ingested voice prompt): all frames at once
        {"name": "voice_clip", "kind": "voice", "frames": 93, "codebooks": 16, "streamed": False},
        # a long prompt of the largest parallel-layer token model
        {"name": "sakupel_prompt_w2048", "kind": "tokens", "design": "sakupel", "size": "w2048", "tokens": 1999},
        # one user's tokens on the smallest one: latency and launches
        {"name": "sakupel_steps_w768", "kind": "steps", "design": "sakupel", "size": "w768", "rows": 1, "prefix": 200, "steps": 8},
        # a full batch on the middle one
        {"name": "sakupel_steps_w1024", "kind": "steps", "design": "sakupel", "size": "w1024", "rows": 16, "prefix": 1400, "steps": 8},
        # an ordinary prompt of a sandwich-layer token model with experts
        {"name": "mabidra_prompt_w1024", "kind": "tokens", "design": "mabidra", "size": "w1024", "tokens": 650},
        # a few users' tokens on the largest one
        {"name": "mabidra_steps_w2048", "kind": "steps", "design": "mabidra", "size": "w2048", "rows": 4, "prefix": 500, "steps": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["turn", "prompt", "voice", "voice", "tokens", "tokens", "steps", "steps"])
    if kind == "turn":
        return {"kind": kind, "rows": rng.choice([1, 1, 2, 3, 5, 8, 11, 16]), "weights": rng.choice(["bf16", "int8"]),
                "prefix": _log_int(rng, 40, 2048), "text": rng.randint(4, 40), "frames": rng.randint(2, 6)}
    if kind == "prompt":
        return {"kind": kind, "weights": rng.choice(["bf16", "int8"]), "tokens": _log_int(rng, 4, 2500)}
    if kind == "voice":
        streamed = rng.random() < 0.5
        return {"kind": kind, "frames": rng.randint(1, 8) if streamed else _log_int(rng, 3, 93), "codebooks": rng.choice([8, 16, 16, 16]),
                "streamed": streamed}
    design, size = rng.choice(["sakupel", "mabidra"]), rng.choice(["w768", "w1024", "w2048"])
    if kind == "tokens":
        return {"kind": kind, "design": design, "size": size, "tokens": _log_int(rng, 6, 1999)}
    return {"kind": kind, "design": design, "size": size, "rows": rng.choice([1, 1, 2, 4, 7, 16]), "prefix": _log_int(rng, 16, 1400),
            "steps": rng.randint(4, 8)}


# ---- inputs ----
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(seed * 1000003 + salt)


def _nano(case):
    cfg = nano_for_cache("A", 4608 if case["kind"] == "prompt" or case["rows"] == 1 else 2304)
    cfg.model.vocab_size = 4096  # of the text embedding, which is only looked up
    return cfg


def _nano_weights(cfg, seed):
    """Matrices N(0, 0.5 / fan_in).  The heads read what the embeddings write (as a trained model's tied heads do), one code
    further on, so that draws are as decided as a trained model's: the likeliest code is ahead by 15 nats and more."""
    m, sd = cfg.model, {}
    for i, (k, shape) in enumerate(state_dict_shapes(m).items()):
        r = torch.randn(shape, generator=_gen(seed, i), device=DEV)
        if k.endswith("norm.weight"):
            t = 1.0 + 0.1 * r
        elif "emb" in k:
            t = r * (0.1 if "pos_emb" in k else 1.0)
        else:
            t = r * (0.5 / shape[-1]) ** 0.5
        sd[k] = t
    CS = m.codebook_size
    audio = sd["audio_emb.embedding.weight"]
    audio[CS:] *= 0.3
    sd["token_emb.weight"] = audio[torch.arange(m.vocab_size, device=DEV) % CS].clone()
    sd["codec_head.weight"] = 3.0 / m.d_model ** 0.5 * audio[:CS].roll(577, 0)
    code = sd["rq_transformer.code_emb.embedding.weight"].view(m.n_quantizers - 1, CS, m.rq_d_model)
    sd["rq_transformer.head_W"] = 2.5 / m.rq_d_model ** 0.5 * code.roll(577, 1)
    return {k: v.to(torch.bfloat16) for k, v in sd.items()}


def _turn_inputs(case, cfg, seed):
    """Per row: the codes of its prompt (as a voice prompt is ingested) and its text."""
    m, g = cfg.model, torch.Generator().manual_seed(seed)
    lens = [case["prefix"]] + [max(8, int(case["prefix"] * 16 ** -float(torch.rand((), generator=g)))) for _ in range(case["rows"] - 1)]
    codes = [torch.randint(0, m.codebook_size, (n, m.n_quantizers), generator=g) for n in lens]
    text = [torch.randint(0, m.vocab_size, (case["text"],), generator=g) for _ in lens]
    return codes, text


def _prompt_inputs(case, cfg, seed):
    """Codes of audio frames, then an eighth of text."""
    m, g, T = cfg.model, torch.Generator().manual_seed(seed), case["tokens"]
    n = T - T // 8
    return torch.randint(0, m.codebook_size, (n, m.n_quantizers), generator=g), torch.randint(0, m.vocab_size, (T - n,), generator=g)


def _voice_weights(cfg, seed):
    """Weights that keep activations O(1) through the vocoder's 60 layers."""
    sd = {}
    for i, (k, shape) in enumerate(codec_state_dict_shapes(cfg).items()):
        r = torch.randn(shape, generator=_gen(seed, i), device=DEV)
        if k.endswith("embed"):
            t = r
        elif k.endswith(("alpha", "beta")):
            t = 0.3 * r
        elif k.endswith(("attn_scale", "mlp_scale", "gamma")):
            t = 0.3 + 0.1 * r
        elif k.endswith("norm.weight"):
            t = 1.0 + 0.1 * r
        elif k.endswith(".bias"):
            t = 0.05 * r
        elif len(shape) == 3 and (".block.1." in k or (k.startswith("upsample") and ".0.conv" in k)):
            t = r / math.sqrt(shape[0] * (1 if k.startswith("upsample") else 2))
        elif len(shape) == 3:
            t = r * (0.3 if "conv2.conv" in k else 0.12 if shape[0] == 1 else 1.0) / math.sqrt(shape[1] * shape[2])
        else:
            t = r / math.sqrt(shape[-1])
        sd[k] = t
    return sd


def _voice_codes(case, cfg, seed):
    return torch.randint(0, cfg.codebook_size, (1, case["codebooks"], case["frames"]), generator=_gen(seed, 9999), device=DEV)


def _lm_config(case):
    if case["design"] == "sakupel":
        return token_lm_config(*SAKUPEL[case["size"]], vocab=VOCAB)
    return sandwich_lm_config(*MABIDRA[case["size"]], vocab=VOCAB)


def _lm_weights(cfg, seed):
    sd = token_lm_state_dict(cfg, seed, DEV)
    # routers as decided as trained ones: a choice that is close on the fourth expert of a token moves its output little
    for i, layer in enumerate(cfg["layers"]):
        if layer["mlp"]["kind"] == "moe":
            sd[f"l{i}.mlp.router"] = sd[f"l{i}.mlp.router"] * 8
            sd[f"l{i}.norm2b"] = sd[f"l{i}.norm2b"] * 0.25
    return sd


def _lm_tokens(case, seed):
    """tokens: one prompt.  steps: per row a prompt and the tokens that follow it."""
    g = torch.Generator().manual_seed(seed)
    if case["kind"] == "tokens":
        return torch.randint(0, VOCAB, (case["tokens"],), generator=g)
    lens = [case["prefix"]] + [max(4, int(case["prefix"] * 16 ** -float(torch.rand((), generator=g)))) for _ in range(case["rows"] - 1)]
    return [torch.randint(0, VOCAB, (n,), generator=g) for n in lens], torch.randint(0, VOCAB, (case["steps"], case["rows"]), generator=g)


def _wanted(T):
    """The positions whose logits a prompt is read at: its last, and some before it as in a replayed trace."""
    return sorted({(T - 1) * i // 32 for i in range(33)})


@torch.inference_mode()
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("turn", "prompt"):
        cfg = _nano(case)
        model = Vui(cfg, _nano_weights(cfg, seed), device=DEV, dtype=torch.bfloat16, int8=case["weights"] == "int8")
        rows = case.get("rows", 1)
        eng = Engine(model=model, max_rows=rows)
        st = {"case": case, "engine": eng, "rows": [eng.new_row() for _ in range(rows)]}
        if kind == "prompt":
            codes, text = _prompt_inputs(case, cfg, seed)
            st["emb"] = torch.cat([model.embed_audio(codes.to(DEV)[None]), model.token_emb(text.to(DEV)[None])], dim=1)
            return st
        codes, text = _turn_inputs(case, cfg, seed)
        for row, c in zip(st["rows"], codes):
            row.prefill_emb(model.embed_audio(c.to(DEV)[None]))
            row.mark_prompt()
        st["lens"] = [c.shape[0] for c in codes]
        st["text"] = [model.token_emb(t.to(DEV)[None]) for t in text]
        st["cfg"] = GenConfig(seed=seed)
        return st
    if kind == "voice":
        cfg = CodecConfig()
        dec = QwenCodecDecoder(_voice_weights(cfg, seed), cfg, device=DEV)
        dec.setup_streaming_graph(1, case["codebooks"])
        return {"case": case, "decoder": dec, "codes": _voice_codes(case, cfg, seed)}
    cfg = _lm_config(case)
    if kind == "tokens":
        model = TokenLM.from_config(cfg, _lm_weights(cfg, seed), device=DEV, max_seqlen=2048)
        eng = TokenEngine(model=model, max_rows=1)
        return {"case": case, "row": eng.new_row(), "tokens": _lm_tokens(case, seed).to(DEV)}
    model = TokenLM.from_config(cfg, _lm_weights(cfg, seed), device=DEV, max_seqlen=2048)
    eng = TokenEngine(model=model, max_rows=case["rows"])
    prompts, steps = _lm_tokens(case, seed)
    rows = [eng.new_row() for _ in prompts]
    for row, p in zip(rows, prompts):
        row.extend(p, [len(p) - 1])
        row.mark_prompt()
    return {"case": case, "engine": eng, "rows": rows, "steps": steps.to(DEV)}


# ---- one pass ----
@torch.inference_mode()
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "turn":
        eng, hidden = st["engine"], []
        for row, emb in zip(st["rows"], st["text"]):
            row.rewind()
            hidden.append(row.prefill_emb(emb)[:, -1])
        hidden = torch.cat(hidden)
        frames, eos = eng.generate(st["rows"], hidden, case["frames"], st["cfg"])
        caches = eng.model.decoder.flash_kv_caches
        n = case["text"] + case["frames"] - 1
        new = {}
        for name, layer in (("first", caches[0]), ("last", caches[-1])):
            new[name] = [[t[i, at:at + n] for i, at in enumerate(st["lens"])] for t in (layer.k_cache, layer.v_cache)]
            new[name] = [torch.stack(t) for t in new[name]]
        return {"hidden": hidden, "frames": frames, "eos": eos, "cache": new}
    if kind == "prompt":
        row = st["rows"][0]
        row.reset()
        hidden = row.prefill_emb(st["emb"])
        n = case["tokens"]
        return {"hidden": hidden, "cache": [(c.k_cache[0, :n], c.v_cache[0, :n]) for c in st["engine"].model.decoder.flash_kv_caches]}
    if kind == "voice":
        dec, codes = st["decoder"], st["codes"]
        if not case["streamed"]:
            return dec(codes)
        with dec.streaming(1):
            return torch.cat([dec(codes[:, :, t:t + 1]).clone() for t in range(case["frames"])], dim=-1)  # frames sit in one static buffer
    if kind == "tokens":
        row = st["row"]
        row.reset()
        return row.extend(st["tokens"], _wanted(case["tokens"]))
    for row in st["rows"]:
        row.rewind()
    return torch.stack([st["engine"].decode_step(st["rows"], t).clone() for t in st["steps"]])


# ---- what a pass cannot do without ----
def _lm_work(cfg):
    """(elements of the weights that every token meets, of one expert, experts met, elements cached per position,
    fp32 state per row, flops of attention per token and visible key)."""
    W, wts, cache, state, attn, expert, met = cfg["width"], cfg["width"] * cfg["vocab"], 0, 0, 0, 0, []
    for layer in cfg["layers"]:
        mx, mlp, t = layer["mixer"], layer["mlp"], layer["type"]
        if t == "gla":
            H, dk, dv, r = mx["heads"], mx["dim"], mx["vdim"], cfg["gla_rank"]
            wts += W * (2 * H * (dk + dv) + r) + H * dk * r + W * H * dv
            state += H * dk * dv
        elif t == "attention":
            H, G, dk, dv = mx["heads"], mx["kv_heads"], mx["dim"], mx["vdim"]
            wts += W * (H * dk + G * (dk + dv) + H) + W * H * dv
            cache += G * (dk + dv)
            attn += 2 * H * (dk + dv)
        elif t == "latent_attention":
            H, r, rot = mx["heads"], mx["kv_rank"], mx["rot_dim"]
            wts += W * (H * (mx["dim"] + rot) + (0 if "kv_from" in mx else r + rot) + H + H * mx["vdim"]) + H * r * (mx["dim"] + mx["vdim"])
            cache += r + rot
            attn += 2 * H * (mx["dim"] + rot + mx["vdim"])
        else:
            wts += 4 * W * mx["width"]
            state += mx["width"]
        if mlp["kind"] == "moe":
            wts += W * mlp["router"]["experts"]
            expert = 2 * W * mlp["expert"]["ff"]
            met.append((mlp["router"]["experts"], mlp["router"]["top"]))
        else:
            wts += (2 if cfg["architecture"] == "Mabidra" else 3) * W * mlp["ff"]
    if cfg.get("loop"):
        wts += 2 * W * W
    return wts, expert, met, cache, state, attn


def work(case):
    kind = case["kind"]
    if kind in ("turn", "prompt"):
        m = _nano(case).model
        d, ff, nl, R = m.d_model, m.ffn, m.n_layers, m.rq_d_model
        wts = nl * (4 * d * d + 3 * d * ff)
        per = 1 if case["weights"] == "int8" else 2
        kv = 2 * nl * d * 2
        if kind == "prompt":
            T = case["tokens"]
            return {"bytes": wts * per + 2 * T * d * 2 + T * kv, "flops": 2 * wts * T + nl * 4 * d * T * (T + 1) / 2}
        rq = d * R + m.rq_n_layers * (4 * R * R + 3 * R * m.rq_ffn) + (m.n_quantizers - 1) * m.codebook_size * R
        rq_flops = 2 * (d * R + (m.n_quantizers - 1) * (m.rq_n_layers * (4 * R * R + 3 * R * m.rq_ffn) + m.codebook_size * R))
        B, n, f = case["rows"], case["text"], case["frames"]
        cached = case["prefix"] * (1 + 0.34 * (B - 1))  # the rows' mean length is a third of the longest
        head = m.codebook_size * d
        return {"bytes": (B + f - 1) * wts * per + f * (head + rq) * 2 + (cached + B * n) * kv * f,
                "flops": B * (2 * wts * (n + f - 1) + f * (rq_flops + 2 * head)) + nl * 4 * d * cached * (n + f - 1)}
    if kind == "voice":
        c = CodecConfig()
        by = fl = 0
        T, cols = case["frames"], 1
        for k, s in codec_state_dict_shapes(c).items():
            n = math.prod(s)
            if k.endswith("embed"):
                by += 4 * T * s[1] * (1 if "semantic" in k or int(k.split(".")[3]) < case["codebooks"] - 1 else 0)
                continue
            by += 4 * n * (T if case["streamed"] else 1)
            if k.startswith("upsample") and ".0.conv.weight" in k:
                fl, cols = fl + 2 * n * cols, cols * s[2]
            elif ".block.1.conv.weight" in k:
                fl, cols = fl + 2 * n * cols, cols * (s[2] // 2)
            elif len(s) > 1 and "input_proj.weight" not in k[:30]:
                fl += 2 * n * cols
        return {"bytes": by + 4 * T * c.hop, "flops": fl * T}
    wts, expert, met, cache, state, attn = _lm_work(_lm_config(case))
    if kind == "tokens":
        T = case["tokens"]
        hit = sum(n * (1 - (1 - t / n) ** T) for n, t in met)
        return {"bytes": 2 * (wts + hit * expert) + 2 * T * cache + 4 * state + 4 * 33 * VOCAB,
                "flops": 2 * T * (wts - _lm_config(case)["width"] * VOCAB + sum(t for _, t in met) * expert) + attn * T * (T + 1) / 2}
    B, f = case["rows"], case["steps"]
    hit = sum(n * (1 - (1 - t / n) ** B) for n, t in met)
    cached = case["prefix"] * (1 + 0.34 * (B - 1))
    return {"bytes": f * (2 * (wts + hit * expert) + 2 * cached * cache + 8 * B * state + 4 * B * VOCAB),
            "flops": f * (2 * B * (wts + sum(t for _, t in met) * expert) + cached * attn)}


def tolerance(case):
    if case["kind"] == "voice":  # fp32 throughout
        return {"rel": 2e-5, "max": 5e-4}
    if case["kind"] == "turn":  # bf16 through 22 layers; a draw whose number falls on a step of the distribution may differ
        return {"rel": 2.5e-2, "max": 0.4, "differ": 0.01}
    return {"rel": 2.5e-2, "max": 0.4}


# ---- the same outputs in 64 bits ----
def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


class _Nano64:
    """The backbone and the depth head in 64 bits, one row, with a cache."""

    def __init__(self, cfg, sd, int8):
        self.m = cfg.model
        self.w = {k: v.double() for k, v in sd.items()}
        if int8:
            for k, v in sd.items():
                if k.startswith("decoder.blocks") and v.dim() == 2:
                    s = (v.float().abs().amax(1) / 127).clamp_min(1e-12).to(torch.bfloat16).double()
                    q = (v.float() / s.float()[:, None]).round().clamp(-127, 127).double()
                    self.w[k] = q * s[:, None]
        self.kv = [[] for _ in range(self.m.n_layers)]
        self.at = 0

    def rotate(self, x):
        n = x.shape[-1]
        inv = self.m.rope_theta ** (-torch.arange(0, n, 2, device=DEV, dtype=torch.float64) / n)
        a = torch.arange(self.at, self.at + x.shape[0], device=DEV, dtype=torch.float64)[:, None, None] * inv
        u, v = x[..., 0::2], x[..., 1::2]
        return torch.stack((u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()), -1).flatten(-2)

    @staticmethod
    def attend(q, k, v):
        """q (T, H, n) the last T of the positions of k, v (S, H, n)."""
        T, S = q.shape[0], k.shape[0]
        s = torch.einsum("thn,shn->hts", q, k) * q.shape[-1] ** -0.5
        s = s.masked_fill(torch.arange(S, device=DEV) > torch.arange(S - T, S, device=DEV)[:, None], -math.inf)
        return torch.einsum("hts,shn->thn", s.softmax(-1), v).reshape(T, -1)

    def forward(self, x):
        m, w, T = self.m, self.w, x.shape[0]
        for i in range(m.n_layers):
            p = f"decoder.blocks.{i}."
            h = _rms(x, 1e-5) * w[p + "attn_norm.weight"]
            q, k, v = (t.reshape(T, -1, m.head_dim) for t in (h @ w[p + "attn.Wqkv.weight"].T).split(
                [m.n_heads * m.head_dim] + 2 * [m.kv_heads * m.head_dim], -1))
            self.kv[i].append((self.rotate(k), v))
            k, v = (torch.cat(t) for t in zip(*self.kv[i]))
            x = x + self.attend(self.rotate(q), k, v) @ w[p + "attn.out_proj.weight"].T
            h = _rms(x, 1e-5) * w[p + "mlp_norm.weight"]
            x = x + (F.silu(h @ w[p + "mlp.w1.weight"].T) * (h @ w[p + "mlp.w3.weight"].T)) @ w[p + "mlp.w2.weight"].T
        self.at += T
        return _rms(x, 1e-5) * w["decoder.norm.weight"]

    def embed(self, codes):
        m = self.m
        return self.w["audio_emb.embedding.weight"][codes + torch.arange(m.n_quantizers, device=DEV) * m.codebook_size].sum(-2)

    def depth(self, hidden, code):
        """The likeliest code of every codebook after the first."""
        m, w, r = self.m, self.w, "rq_transformer."
        R, codes, kv = m.rq_d_model, [code], [[] for _ in range(m.rq_n_layers)]
        x = hidden @ w[r + "backbone_proj.weight"].T if R != m.d_model else hidden
        for q in range(m.n_quantizers):
            if q:
                x = w[r + "code_emb.embedding.weight"][codes[-1] + (q - 1) * m.codebook_size][None]
            x = x + w[r + "pos_emb.weight"][q]
            for i in range(m.rq_n_layers):
                p = f"{r}blocks.{i}."
                qq, k, v = (_rms(x, 1e-6) * w[p + "attn_norm.weight"] @ w[p + "Wqkv.weight"].T).reshape(3, 1, m.rq_n_heads, -1)
                kv[i].append((k, v))
                k, v = (torch.cat(t) for t in zip(*kv[i]))
                x = x + self.attend(qq, k, v) @ w[p + "out_proj.weight"].T
                h = _rms(x, 1e-6) * w[p + "mlp_norm.weight"]
                x = x + (F.silu(h @ w[p + "w1.weight"].T) * (h @ w[p + "w3.weight"].T)) @ w[p + "w2.weight"].T
            if q:
                h = _rms(x, 1e-6) * w[r + "norm.weight"]
                codes.append(int((h @ w[r + "head_W"][q - 1].T).argmax()))
        return torch.tensor(codes, device=DEV)

    def cached(self, layer, frm):
        return [torch.cat(t)[frm:] for t in zip(*self.kv[layer])]


def _turn64(case, seed):
    cfg = _nano(case)
    sd = _nano_weights(cfg, seed)
    out = {"hidden": [], "frames": [], "eos": [], "k0": [], "v0": [], "k1": [], "v1": []}
    for codes, text in zip(*_turn_inputs(case, cfg, seed)):
        net = _Nano64(cfg, sd, case["weights"] == "int8")
        # embeddings of audio are sums that the model holds in its own 16 bits
        net.forward(net.embed(codes.to(DEV)).to(torch.bfloat16).double())
        h = net.forward(net.w["token_emb.weight"][text.to(DEV)])[-1:]
        out["hidden"].append(h)
        frames, eos = [], [torch.zeros((), dtype=torch.float64, device=DEV)]
        for f in range(case["frames"]):
            if f:
                h = net.forward(net.embed(frames[-1])[None])
                eos.append(torch.sigmoid(h @ net.w["eos_head.weight"].T + net.w["eos_head.bias"])[0, 0])
            frames.append(net.depth(h, int((h @ net.w["codec_head.weight"].T).argmax())))
        out["frames"].append(torch.stack(frames))
        out["eos"].append(torch.stack(eos))
        for n, layer in ((0, 0), (1, -1)):
            for name, t in zip("kv", net.cached(layer, codes.shape[0])):
                out[f"{name}{n}"].append(t)
    return {"hidden": torch.cat(out["hidden"]), "frames": torch.stack(out["frames"], 1), "eos": torch.stack(out["eos"], 1),
            "cache": {n: [torch.stack(out[f"{c}{i}"]) for c in "kv"] for i, n in ((0, "first"), (1, "last"))}}


def _prompt64(case, seed):
    cfg = _nano(case)
    net = _Nano64(cfg, _nano_weights(cfg, seed), case["weights"] == "int8")
    codes, text = _prompt_inputs(case, cfg, seed)
    emb = torch.cat([net.embed(codes.to(DEV)).to(torch.bfloat16).double(), net.w["token_emb.weight"][text.to(DEV)]])
    return {"hidden": net.forward(emb)[None], "cache": [tuple(net.cached(i, 0)) for i in range(cfg.model.n_layers)]}


def _conv64(x, w, b, dil=1):
    """Causal convolution (Cin, T) -> (Cout, T), one product per tap; depthwise where w has one input channel."""
    T, k = x.shape[1], w.shape[2]
    x = F.pad(x, ((k - 1) * dil, 0))
    taps = [x[:, i * dil:i * dil + T] for i in range(k)]
    y = sum((w[:, :, i] @ t) if w.shape[1] == x.shape[0] else w[:, :, i] * t for i, t in enumerate(taps))
    return y if b is None else y + b[:, None]


def _upconv64(x, w, b, stride):
    """Causal transposed convolution: the outputs behind the last input's own are dropped."""
    T, n = x.shape[1], w.shape[2]
    y = torch.zeros(w.shape[1], T * stride + n, dtype=x.dtype, device=DEV)
    for i in range(n):
        y[:, i:i + T * stride:stride] += w[:, :, i].T @ x
    return y[:, :T * stride] + b[:, None]


def _voice64(case, seed):
    cfg = CodecConfig()
    w = {k: v.double() for k, v in _voice_weights(cfg, seed).items()}
    codes = _voice_codes(case, cfg, seed)[0]

    def snake(x, p):
        return x + torch.sin(x * w[p + "alpha"].exp()[:, None]) ** 2 / (w[p + "beta"].exp() + 1e-9)[:, None]

    x = 0
    for name, first, last in (("semantic", 0, cfg.n_semantic), ("acoustic", cfg.n_semantic, case["codebooks"])):
        p = f"quantizer.{name}."
        x = x + w[p + "output_proj.weight"][:, :, 0] @ sum(w[p + f"codebooks.{i - first}.embed"][codes[i]] for i in range(first, last)).T
    x = _conv64(x, w["pre_conv.conv.weight"], w["pre_conv.conv.bias"]).T
    t = "pre_transformer."
    x = x @ w[t + "input_proj.weight"].T + w[t + "input_proj.bias"]
    T, H, n = x.shape[0], cfg.n_heads, cfg.head_dim
    ang = torch.arange(T, device=DEV, dtype=torch.float64)[:, None, None] * cfg.rope_theta ** (
        -torch.arange(0, n, 2, device=DEV, dtype=torch.float64) / n)

    def rotate(x):
        u, v = x.chunk(2, -1)
        return torch.cat((u * ang.cos() - v * ang.sin(), v * ang.cos() + u * ang.sin()), -1)

    for i in range(cfg.n_layers):
        p = f"{t}layers.{i}."
        h = _rms(x, 1e-6) * w[p + "input_layernorm.weight"]
        q, k, v = ((h @ w[p + f"{c}_proj.weight"].T).reshape(T, H, n) for c in "qkv")
        x = x + w[p + "attn_scale"] * (_Nano64.attend(rotate(q), rotate(k), v) @ w[p + "o_proj.weight"].T)
        h = _rms(x, 1e-6) * w[p + "post_attention_layernorm.weight"]
        x = x + w[p + "mlp_scale"] * ((F.silu(h @ w[p + "gate_proj.weight"].T) * (h @ w[p + "up_proj.weight"].T)) @ w[p + "down_proj.weight"].T)
    x = ((_rms(x, 1e-6) * w[t + "norm.weight"]) @ w[t + "output_proj.weight"].T + w[t + "output_proj.bias"]).T
    for i, r in enumerate(cfg.up_ratios):
        p = f"upsample.{i}."
        x = _upconv64(x, w[p + "0.conv.weight"], w[p + "0.conv.bias"], r)
        h = _conv64(x, w[p + "1.dwconv.conv.weight"], w[p + "1.dwconv.conv.bias"]).T
        h = F.layer_norm(h, h.shape[-1:], w[p + "1.norm.weight"], w[p + "1.norm.bias"], 1e-6)
        h = F.gelu(h @ w[p + "1.pwconv1.weight"].T + w[p + "1.pwconv1.bias"])
        x = x + (w[p + "1.gamma"] * (h @ w[p + "1.pwconv2.weight"].T + w[p + "1.pwconv2.bias"])).T
    x = _conv64(x, w["decoder.0.conv.weight"], w["decoder.0.conv.bias"])
    for i, rate in enumerate(cfg.rates):
        p = f"decoder.{i + 1}.block."
        x = _upconv64(snake(x, p + "0."), w[p + "1.conv.weight"], w[p + "1.conv.bias"], rate)
        for j, dil in ((2, 1), (3, 3), (4, 9)):
            q = f"{p}{j}."
            h = _conv64(snake(x, q + "act1."), w[q + "conv1.conv.weight"], w[q + "conv1.conv.bias"], dil)
            x = x + _conv64(snake(h, q + "act2."), w[q + "conv2.conv.weight"], w[q + "conv2.conv.bias"])
    n = len(cfg.rates)
    x = _conv64(snake(x, f"decoder.{n + 1}."), w[f"decoder.{n + 2}.conv.weight"], w[f"decoder.{n + 2}.conv.bias"])
    return x.clamp(-1, 1)[None]


def _turned(x, rot):
    """x (T, ..., n): its first rot["dims"] entries rotated, entry i with entry i + dims / 2."""
    n = rot["dims"]
    a = torch.arange(x.shape[0], device=DEV, dtype=torch.float64)[:, None] * rot["base"] ** (
        -torch.arange(0, n, 2, device=DEV, dtype=torch.float64) / n)
    a = a.reshape(x.shape[0], *[1] * (x.dim() - 2), n // 2)
    u, v = x[..., :n // 2], x[..., n // 2:n]
    return torch.cat((u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin(), x[..., n:]), -1)


def _sakupel64(cfg, w, tokens, want):
    eps, x, kept = cfg["norm"]["eps"], w["embed"][tokens], {}
    T = len(tokens)
    past = torch.arange(T, device=DEV) > torch.arange(T, device=DEV)[:, None]
    for i, layer in enumerate(cfg["layers"]):
        p, mx = f"l{i}.mix.", layer["mixer"]
        h = _rms(x, eps) * w[f"l{i}.norm1"]
        if layer["type"] == "latent_attention":
            H, dim, r = mx["heads"], mx["dim"], mx["kv_rank"]
            if "kv_from" not in mx:
                y = h @ w[p + "dkv"].T
                kept[i] = _rms(y[:, :r], eps) * w[p + "dkv.norm"], _turned(y[:, r:], mx["rot"])
            c, kr = kept[mx.get("kv_from", i)]
            q = (h @ w[p + "q"].T).reshape(T, H, -1)
            s = torch.einsum("thn,shn->hts", q[..., :dim], (c @ w[p + "uk"].T).reshape(T, H, dim))
            s = (s + torch.einsum("thn,sn->hts", _turned(q[..., dim:], mx["rot"]), kr)) * mx["scale"]
            y = torch.einsum("hts,shn->thn", s.masked_fill(past, -math.inf).softmax(-1), (c @ w[p + "uv"].T).reshape(T, H, -1))
            y = (y * torch.sigmoid(h @ w[p + "g"].T)[..., None]).reshape(T, -1) @ w[p + "o"].T
        else:
            z, u = torch.sigmoid(h @ w[p + "z"].T + w[p + "z.b"]), h @ w[p + "x"].T + w[p + "x.b"]
            c = z * torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
            S, rows = torch.zeros_like(c[0]), []
            for t in range(T):
                S = (1 - z[t]) * S + c[t]
                rows.append(S)
            y = (torch.stack(rows) * F.silu(h @ w[p + "g"].T)) @ w[p + "o"].T
        p, lim = f"l{i}.mlp.", layer["mlp"]["limit"]
        g, u = (h @ w[p + "gate"].T).clamp(max=lim), (h @ w[p + "up"].T).clamp(-lim, lim)
        x = x + y + (g * torch.sigmoid(1.702 * g) * (u + 1)) @ w[p + "down"].T
    return (_rms(x[want], eps) * w["final.norm"]) @ w["head"].T


def _bucket(n, buckets, far):
    half = buckets // 2
    return n if n < half else min(buckets - 1, half + math.floor(math.log(n / half) / math.log(far / half) * (buckets - half) + 1e-9))


def _mabidra64(cfg, w, tokens, want):
    eps, T, groups = cfg["norm"]["eps"], len(tokens), cfg["norm"]["groups"]
    at = torch.arange(T, device=DEV)
    past = at > at[:, None]

    def norm(x, g):
        return _rms(x.reshape(T, groups, -1), eps).reshape(x.shape) * g

    x0 = w["embed"][tokens] * cfg["embedding"]["scale"]
    x = torch.cat((x0, x0), -1) @ w["loop.in"].T + w["loop.step"][0]  # the loop runs once, over every layer
    for i, layer in enumerate(cfg["layers"]):
        p, mx, mlp = f"l{i}.mix.", layer["mixer"], layer["mlp"]
        H, dim, dv = mx["heads"], mx["dim"], mx["vdim"]
        h = norm(x, w[f"l{i}.norm1"])
        if layer["type"] == "gla":
            q, k, v = ((h @ w[p + n].T).reshape(T, H, -1) for n in "qkv")
            a = torch.exp(F.logsigmoid(h @ w[p + "a1"].T @ w[p + "a2"].T + w[p + "a2.b"]) / mx["tau"]).reshape(T, H, dim, 1)
            S, rows = torch.zeros(H, dim, dv, dtype=torch.float64, device=DEV), []
            for t in range(T):
                S = a[t] * S + k[t][:, :, None] * v[t][:, None, :]
                rows.append((S * q[t][:, :, None]).sum(1))
            y = _rms(torch.stack(rows) * dim ** -0.5, eps) * w[p + "norm"]
            y = (y.reshape(T, -1) * F.silu(h @ w[p + "g"].T)) @ w[p + "o"].T
        else:
            G, rel = mx["kv_heads"], w[p + "rel"]
            q, k, v = ((h @ w[p + n].T + w[p + n + ".b"]).reshape(T, -1, m) for n, m in (("q", dim), ("k", dim), ("v", dv)))
            q, k = _rms(q, eps) * w[p + "q.norm"], (_rms(k, eps) * w[p + "k.norm"]).repeat_interleave(H // G, 1)
            q = q * (1 + mx["q_temp"]["coef"] * torch.log((at + 1).div(mx["q_temp"]["every"], rounding_mode="floor") + 1.0))[:, None, None]
            b = rel[torch.tensor([_bucket(n, len(rel), mx["bias_max"]) for n in range(T)], device=DEV)] + w[p + "pb"]
            s = torch.einsum("thn,shn->hts", q, k) * mx["scale"] + b[(at[:, None] - at).clamp(min=0)].permute(2, 0, 1)
            y = torch.einsum("hts,shn->thn", torch.sigmoid(s).masked_fill(past, 0.0), v.repeat_interleave(H // G, 1))
            y = (y * torch.sigmoid(h @ w[p + "g"].T)[..., None]).reshape(T, -1) @ w[p + "o"].T + w[p + "o.b"]
        x = x + norm(y, w[f"l{i}.norm1b"])
        p, h = f"l{i}.mlp.", norm(x, w[f"l{i}.norm2"])
        if mlp["kind"] == "dense":
            z, (sp, sq) = h @ w[p + "up"].T, F.softplus(w[p + "act"])
            z = torch.where(z > 0, sp * z * z, (0.5 + sq) * (torch.expm1(z.clamp(max=0)) - z.clamp(max=0))) + z / 2
            y = z @ w[p + "down"].T
        else:
            best = (h @ w[p + "router"].T + w[p + "router.b"]).topk(mlp["router"]["top"])
            share, y = best.values.softmax(-1), torch.zeros_like(x)
            for e in range(mlp["router"]["experts"]):
                r, c = (best.indices == e).nonzero(as_tuple=True)
                y[r] += share[r, c][:, None] * (torch.relu(h[r] @ w[f"{p}e{e}.up"].T) ** 2 @ w[f"{p}e{e}.down"].T)
        x = x + norm(y, w[f"l{i}.norm2b"])
    return (norm(x, w["final.norm"]) @ w["head"].T)[want]


def _lm64(case, seed):
    cfg = _lm_config(case)
    w = {k: v.double() for k, v in _lm_weights(cfg, seed).items()}
    net = _sakupel64 if case["design"] == "sakupel" else _mabidra64
    if case["kind"] == "tokens":
        return net(cfg, w, _lm_tokens(case, seed).to(DEV), _wanted(case["tokens"]))
    prompts, steps = _lm_tokens(case, seed)
    n = case["steps"]
    return torch.stack([net(cfg, w, torch.cat((p, steps[:, i])).to(DEV), list(range(len(p), len(p) + n))) for i, p in enumerate(prompts)], 1)


@torch.inference_mode()
def exact(case, seed):
    return {"turn": _turn64, "prompt": _prompt64, "voice": _voice64, "tokens": _lm64, "steps": _lm64}[case["kind"]](case, seed)
