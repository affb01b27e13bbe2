"""The work a program that uses this framework has it do, as cases that can be timed and checked: frames resized, clips encoded, turns of live
commentary, a one-shot question about a long video, requests to the layer-list decoders.  `listed()` are fixed cases, `draw` gives others of the
same ranges.  A case is a dict of plain values; `prepare` makes what a program holds before the call (model, stream states, inputs), `run` is one
pass through the public entry points, `work` what the pass cannot do without, `exact` the outputs in 64 bits from plain torch.

Weights are random in the distributions of initialised networks (output projections smaller by the root of the depth), the head's rows are the
embedding's in another order: every step then has one clear winner, so that greedy tokens are decided by the model and not by rounding.
"""
import math
import zlib

import numpy as np
import torch

from livecc_amd import resize as R
from livecc_amd import weights as W
from livecc_amd.config import DECODER_CONFIGS, BemuzenConfig, get_config
from livecc_amd.modeling import BemuzenForCausalLM, DebunexForCausalLM, LiveCCForConditionalGeneration

DEVICE = "cuda"
MEAN, STD = (0.48145466, 0.4578275, 0.40821073), (0.26862954, 0.26130258, 0.27577711)          # of the image processor
PERM_MUL, PERM_ADD = 48271, 7919          # head row v = embedding row (v * MUL + ADD) mod vocabulary


def listed():
    return [
        # two 720p frames of a live source brought to the model's size: what every tick of a stream starts with
        dict(name="resize_pair", kind="resize", frames=2, src_h=720, src_w=1280, height=392, width=728, layout="THWC"),
        # the vision tower over one tick (two frames, 1,456 patches) and over a clip that is encoded for later questions
        dict(name="tower_pair", kind="clip", model="livecc-7b", frames=2, height=392, width=728),
        dict(name="tower_clip", kind="clip", model="livecc-7b", frames=37, height=308, width=560),
        # one tick of live commentary: two new frames on a stream that has been running for a while, 16 tokens said
        turn("turn_7b", "livecc-7b", 1, 2000, 2, 392, 728, 16),
        # the smaller model on a young stream with smaller frames
        turn("turn_2b", "qwen2vl-2b-untied", 1, 500, 2, 280, 504, 16),
        # the same tick for eight streams that one GPU serves together
        turn("turn_7b_8", "livecc-7b", 8, 1100, 2, 392, 728, 16),
        # fp8 weights, a stream far into its window
        turn("turn_7b_fp8", "livecc-7b", 1, 9000, 2, 392, 728, 16, fp8=True),
        # a question about a whole video: 480 frames in one prompt of 24,000 tokens, a short answer
        turn("oneshot_7b", "livecc-7b", 1, 0, 480, 280, 280, 8),
        # a decoder request: a prompt read, a passage written
        dict(name="debunex_7b", kind="text", model="debunex-7b", streams=1, prompt=1000, spread=0, tokens=32),
        # many short requests answered together
        dict(name="debunex_2b_32", kind="text", model="debunex-2b", streams=32, prompt=120, spread=150, tokens=32),
        # some requests of unequal length
        dict(name="bemuzen_7b_8", kind="text", model="bemuzen-7b", streams=8, prompt=300, spread=500, tokens=16),
        # a long document read for a one-word answer
        dict(name="bemuzen_7b_long", kind="text", model="bemuzen-7b", streams=1, prompt=8192, spread=0, tokens=2),
    ]


def turn(name, model, streams, history, frames, height, width, tokens, fp8=False):
    return dict(name=name, kind="turn", model=model, fp8=fp8, streams=streams, history=history, frames=frames, height=height, width=width, tokens=tokens)


def between(rng, lo, hi):
    """Whole number, spread over the logarithm of the range."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["resize", "clip", "turn", "turn", "text", "text"])
    side = lambda lo, hi: 28 * rng.randint(lo, hi)
    if kind == "resize":
        h, w = rng.choice([(360, 640), (480, 854), (720, 1280), (1080, 1920), (1280, 720), (rng.randint(300, 1100), rng.randint(300, 1900))])
        return dict(kind=kind, frames=2 * between(rng, 1, 12), src_h=h, src_w=w, height=side(8, 18), width=side(8, 28), layout=rng.choice(["THWC", "TCHW"]))
    if kind == "clip":
        return dict(kind=kind, model=rng.choice(["livecc-7b", "qwen2vl-2b-untied"]), frames=between(rng, 1, 40), height=side(5, 14), width=side(5, 26))
    if kind == "turn":
        model = rng.choice(["livecc-7b", "qwen2vl-2b-untied"])
        streams = between(rng, 1, 16)
        history = rng.choice([0, between(rng, 60, 12000 // streams)])
        c = turn("", model, streams, history, 2 if history else rng.choice([2, 6]), side(6, 14), side(8, 26), rng.randint(8, 24),
                 fp8=streams <= 4 and rng.random() < 0.25)
        del c["name"]
        return c
    model = rng.choice(["debunex-2b", "debunex-7b", "bemuzen-2b", "bemuzen-7b"])
    streams = between(rng, 1, 32)
    prompt = between(rng, 16, 8000 // streams)
    return dict(kind=kind, model=model, streams=streams, prompt=prompt, spread=rng.choice([0, prompt // 2]), tokens=between(rng, 1, 32))


# ---- inputs ----
class Checkpoint:
    """The tensors of a random checkpoint by name, made on the GPU when asked for; the same ones for every caller."""

    def __init__(self, cfg):
        self.cfg = cfg
        self.decoder = isinstance(cfg, DECODER_CONFIGS)
        if self.decoder:
            self.shapes = W.bemuzen_param_shapes(cfg) if isinstance(cfg, BemuzenConfig) else W.decoder_param_shapes(cfg)
            self.embed, self.head = "embed", "head"
        else:
            self.shapes = W.hf_param_shapes(cfg)
            self.embed, self.head = "language_model.embed_tokens.weight", "lm_head.weight"
        self.out_std = 0.02 / math.sqrt(2 * cfg.num_hidden_layers)
        self.embed_std = 1.0 if self.decoder and not isinstance(cfg, BemuzenConfig) else 2.0

    def normal(self, name, std, mean=0.0):
        g = torch.Generator(device=DEVICE).manual_seed(zlib.crc32(name.encode()))
        return torch.randn(self.shapes[name], generator=g, device=DEVICE, dtype=torch.bfloat16).mul_(std).add_(mean)

    def __call__(self, name):
        if name == self.head:
            V = self.shapes[name][0]
            rows = (torch.arange(V, device=DEVICE) * PERM_MUL + PERM_ADD) % V
            return self(self.embed)[rows] * (0.03125 / self.embed_std)
        if name == self.embed:
            return self.normal(name, self.embed_std)
        last = name.rsplit(".", 1)[-1]
        if last == "alpha":
            return torch.full((), 0.5, device=DEVICE, dtype=torch.bfloat16)
        if name.endswith(".conv"):
            return self.normal(name, 0.3)
        if len(self.shapes[name]) >= 2:
            narrow = name.endswith(("attn.proj.weight", "fc2.weight", "o_proj.weight", "down_proj.weight", "mix.o", "mlp.down", "left.o", "right.o"))
            return self.normal(name, self.out_std if narrow else 0.02)
        if last in ("bias", "b"):
            return self.normal(name, 0.05)
        if last == "A_log":
            return self.normal(name, 0.5, 1.0)
        if last == "dt_bias":
            return self.normal(name, 1.0, -3.0)
        around_zero = isinstance(self.cfg, BemuzenConfig) and last in ("norm1", "norm1b", "norm2", "norm2b") or name == "final.norm" and isinstance(self.cfg, BemuzenConfig)
        return self.normal(name, 0.1, 0.0 if around_zero else 1.0)


def pictures(n, h, w, seed, layout):
    """Smooth pictures with a little noise that change slowly from frame to frame, uint8."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    base = torch.rand(1, 3, max(2, h // 28), max(2, w // 28), generator=g, device=DEVICE)
    move = torch.rand(1, 3, max(2, h // 28), max(2, w // 28), generator=g, device=DEVICE)
    big = lambda x: torch.nn.functional.interpolate(x, (h, w), mode="bilinear")
    base, move = big(base), big(move)
    out = torch.empty(n, 3, h, w, dtype=torch.uint8, device=DEVICE)
    for i in range(n):
        a = 0.5 + 0.5 * math.cos(0.2 * i)
        out[i] = ((base * a + move * (1 - a))[0] * 240 + torch.randn(3, h, w, generator=g, device=DEVICE) * 6).clamp_(0, 255).to(torch.uint8)
    return out if layout == "TCHW" else out.permute(0, 2, 3, 1).contiguous()


def video_tokens(case):
    return (case["frames"] + 1) // 2 * (case["height"] // 28) * (case["width"] // 28)


def turn_ids(cfg, case, seed):
    """(ids already said, ids of the new turn) of every stream: system and user text, the clip's placeholders, the assistant's header."""
    rng = np.random.RandomState(seed % (1 << 31))
    text = lambda n: [int(x) for x in rng.randint(0, 150000, size=n)]
    video = [cfg.vision_start_token_id] + [cfg.video_token_id] * video_tokens(case) + [cfg.vision_end_token_id]
    out = []
    for _ in range(case["streams"]):
        past = text(case["history"])
        start = [cfg.eos_token_id] + text(14) if past else text(27)
        out.append((past, start + video + ([] if past else text(12)) + [cfg.eos_token_id] + text(4)))
    return out


def prompt_lengths(case):
    return [case["prompt"] + (i * 37) % (case["spread"] + 1) for i in range(case["streams"])]


def prompts(cfg, case, seed):
    rng = np.random.RandomState(seed % (1 << 31))
    return [[int(x) for x in rng.randint(0, cfg.vocab_size, size=n)] for n in prompt_lengths(case)]


def kv_tokens(case, cfg):
    """Cache of a stream: what it will hold, and the room the model keeps for its longest answer."""
    n = max(prompt_lengths(case)) if case["kind"] == "text" else case["history"] + video_tokens(case) + 64
    return n + case["tokens"] + 512


def prepare(case, seed):
    kind = case["kind"]
    if kind == "resize":
        return dict(kind=kind, frames=pictures(case["frames"], case["src_h"], case["src_w"], seed, case["layout"]), height=case["height"],
                    width=case["width"], layout=case["layout"])
    cfg = get_config(case["model"])
    params = Checkpoint(cfg)
    if kind == "text":
        cls = BemuzenForCausalLM if isinstance(cfg, BemuzenConfig) else DebunexForCausalLM
        model = cls(cfg, W.make_arena(cfg, DEVICE).load_state_dict(params), DEVICE, max_streams=case["streams"], max_kv_len=kv_tokens(case, cfg))
        return dict(kind=kind, model=model, prompts=[torch.tensor(p) for p in prompts(cfg, case, seed)], tokens=case["tokens"])
    arena = W.make_arena(cfg, DEVICE, case.get("fp8", False)).load_state_dict(params)
    if kind == "clip":
        model = LiveCCForConditionalGeneration(cfg, arena, DEVICE, max_streams=1, max_kv_len=1024)
        return dict(kind=kind, model=model, frames=pictures(case["frames"], case["height"], case["width"], seed, "TCHW"))
    streams = case["streams"]
    model = LiveCCForConditionalGeneration(cfg, arena, DEVICE, max_streams=streams, max_kv_len=kv_tokens(case, cfg))
    ids = turn_ids(cfg, case, seed)
    frames = [pictures(case["frames"], case["height"], case["width"], seed + 7 * i, "TCHW") for i in range(streams)]
    states = []
    if case["history"]:
        states = [o.past_key_values for o in model.generate_batch([dict(input_ids=torch.tensor(past)) for past, _ in ids], max_new_tokens=1)]
    return dict(kind=kind, model=model, states=states, history=case["history"], ids=[torch.tensor(past + new) for past, new in ids], frames=frames,
                tokens=case["tokens"])


def run(state):
    kind = state["kind"]
    if kind == "resize":
        return R.resize_bicubic_aa(state["frames"], state["height"], state["width"], state["layout"])
    model = state["model"]
    if kind == "clip":
        return model.get_video_features(frames=state["frames"])
    if kind == "text":
        requests = [dict(input_ids=p) for p in state["prompts"]]
    else:
        for st in state["states"]:          # every pass is the tick behind the same history
            model.engine.set_slot_length(st.slot, state["history"], state["history"])
        states = state["states"] or [None] * len(state["ids"])
        requests = [dict(input_ids=i, frames=f, state=s) for i, f, s in zip(state["ids"], state["frames"], states)]
    outs = model.generate_batch(requests, repetition_penalty=1.05 if kind == "turn" else 1.0, max_new_tokens=state["tokens"], force_length=True,
                                output_logits=True)
    if not state.get("states"):
        for o in outs:
            o.past_key_values.release()
    return {"tokens": [o.sequences for o in outs], "logits": [o.logits for o in outs]}


# ---- what a pass cannot do without ----
def tower_work(cfg, frames, height, width):
    p, slices = (height // 14) * (width // 14), (frames + 1) // 2
    E, M, n = cfg.vit_embed_dim, cfg.vit_mlp_dim, (height // 14) * (width // 14) * ((frames + 1) // 2)
    weights = cfg.patch_dim * E + cfg.vit_depth * (4 * E * E + 2 * E * M) + 16 * E * E + 4 * E * cfg.hidden_size
    flops = 2 * n * (cfg.patch_dim * E + cfg.vit_depth * (4 * E * E + 2 * E * M)) + cfg.vit_depth * slices * 4 * p * p * E + 2 * (n // 4) * (16 * E * E + 4 * E * cfg.hidden_size)
    return flops, 2 * weights + 3 * frames * height * width + 2 * (n // 4) * cfg.hidden_size


def layer_sizes(cfg, i):
    """(weights, channels of a query times keys product and of the value product, cached elements a token, recurrent flops a token, state bytes)."""
    H = cfg.hidden_size
    if not hasattr(cfg, "layers"):
        return H * cfg.qkv_dim + cfg.q_dim * H + 3 * H * cfg.intermediate_size, 2 * cfg.q_dim, 2 * cfg.kv_dim, 0, 0
    l = cfg.layers[i]
    m, ff = l.mixer, 3 * H * l.ff
    if hasattr(m, "kv_rank"):
        own = m.kv_from is None
        n = H * (m.q_rank + (m.kv_rank if own else 0) + m.heads + m.heads * m.vdim) + m.heads * (m.dim * (m.q_rank + m.kv_rank) + m.vdim * m.kv_rank)
        return n + ff, m.heads * (m.dim + m.vdim), m.kv_rank, 0, 0
    r = m.recurrent
    if hasattr(m, "left"):
        a = m.left
        n = H * ((a.heads + a.kv_heads) * a.dim + a.kv_heads * a.vdim + a.heads * a.vdim + r.heads * (2 * r.dim + 3 * r.vdim))
        return n + ff, a.heads * (a.dim + a.vdim), a.kv_heads * (a.dim + a.vdim), 4 * r.heads * r.dim * r.vdim, 4 * r.heads * r.dim * r.vdim
    n = H * (3 * r.heads * r.vdim + 2 * r.groups * r.state + r.heads)
    return n + ff, 0, 0, 4 * r.heads * r.state * r.vdim, 4 * r.heads * r.state * r.vdim


def work(case):
    if case["kind"] == "resize":
        n = 3 * case["frames"]
        return {"bytes": n * (case["src_h"] * case["src_w"] + case["height"] * case["width"]), "flops": 0}
    cfg = get_config(case["model"])
    if case["kind"] == "clip":
        flops, nbytes = tower_work(cfg, case["frames"], case["height"], case["width"])
        return {"bytes": nbytes, "flops": flops}
    B, steps, flops, nbytes = case["streams"], case["tokens"] - 1, 0, 0
    text = case["kind"] == "text"
    if text:
        news, past = prompt_lengths(case), 0
    else:
        news, past = [len(turn_ids(cfg, dict(case, streams=1), 0)[0][1])] * B, case["history"]
        f, b = tower_work(cfg, case["frames"], case["height"], case["width"])
        weights = b - 3 * case["frames"] * case["height"] * case["width"]
        flops, nbytes = B * f, weights + B * (b - weights)
    per = 1 if case.get("fp8") else 2          # bytes of a weight
    V, H = cfg.vocab_size, cfg.hidden_size
    for i in range(cfg.num_hidden_layers):
        n, attn, cached, rec, state = layer_sizes(cfg, i)
        nbytes += per * n * (1 + steps)
        for S in news:
            flops += 2 * n * (S + steps) + 2 * attn * S * (past + (S + 1) / 2) + rec * (S + steps)
            nbytes += 2 * cached * (past + S) + state * (1 + 2 * steps)          # the prefill reads what is cached and writes its rows
            for k in range(steps):
                flops += 2 * attn * (past + S + k + 1)
                nbytes += 2 * cached * (past + S + k + 1)
    flops += 2 * V * H * B * (1 + steps)
    nbytes += (per * V * H + B * V * (4 if text else 2)) * (1 + steps)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "resize":
        return "exact"
    # measured against `exact`: 0.002 where the residual is held in 32 bits and nothing is normed behind the sums, 0.008 with norms on both sides,
    # 0.013 to 0.016 where every sum is rounded to bf16 (28 and 32 layers); two correct results differ by up to twice that
    if case["kind"] == "text" and case["model"].startswith("debunex"):
        return {"rel": 0.008, "max": 0.1}
    return {"rel": 0.03, "max": 0.25}


# ---- the outputs in 64 bits, plain torch ----
def rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def layer_norm(x, w, b):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], w, b, 1e-6)


def silu(x):
    return x * torch.sigmoid(x)


def rotate(x, angles):
    """x [rows, heads, 2n], angles [rows, n]: channel c turns with channel c + n."""
    c, s = angles.cos()[:, None], angles.sin()[:, None]
    a, b = x.chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def attend(q, k, v, scale, causal=True, slopes=None):
    """q [T, H, d], k [T, G, d], v [T, G, e] of one sequence -> [T, H, e]; head by head, a thousand queries at a time."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
    at = torch.arange(T, device=q.device)
    for h in range(H):
        kh, vh = k[:, h * G // H].T.contiguous(), v[:, h * G // H].contiguous()
        for a in range(0, T, 1024):
            n = min(T, a + 1024) if causal else T
            s = (q[a:a + 1024, h].contiguous() @ kh[:, :n]) * scale
            if causal:
                dist = (at[a:a + 1024, None] - at[None, :n])
                if slopes is not None:
                    s -= slopes[h] * dist
                s = s.masked_fill_(dist < 0, -math.inf)
            out[a:a + 1024, h] = torch.softmax(s, -1) @ vh[:n]
    return out


def decayed(q, k, v, log_decay, weight):
    """Sum over s <= t of exp(decays between) weight_s (q_t . k_s) v_s; q, k [T, H, n], v [T, H, e], log_decay, weight [T, H]."""
    T, H = v.shape[:2]
    out = torch.empty_like(v)
    L = log_decay.cumsum(0)
    at = torch.arange(T, device=q.device)
    for h in range(H):
        kh, vh = k[:, h].T.contiguous(), (v[:, h] * weight[:, h, None])
        for a in range(0, T, 1024):
            n = min(T, a + 1024)
            s = q[a:n, h].contiguous() @ kh[:, :n]
            e = (L[a:n, None, h] - L[None, :n, h]).masked_fill_(at[a:n, None] < at[None, :n], -math.inf)
            out[a:n, h] = (s * e.exp()) @ vh[:n]
    return out


def gated(h, P, gate, up, down):
    return (silu(h @ P(gate).T) * (h @ P(up).T)) @ P(down).T


def e4m3_rows(w):
    """A weight as its fp8 form holds it: a scale for each row (its largest value is 448), three mantissa bits."""
    scale = (w.abs().amax(1) / 448).float().clamp_min(1e-12).double()[:, None]
    x = (w / scale).float().double().clamp(-448, 448)
    step = torch.exp2(torch.floor(torch.log2(x.abs().clamp_min(2.0 ** -6))) - 3)
    return torch.round(x / step) * step * scale


def tower(cfg, P, frames):
    """[T, 3, H, W] uint8 -> [patches / 4, width]."""
    f = frames.double()
    f = torch.cat([f, f[-1:]]) if f.shape[0] % 2 else f
    col = lambda c: torch.tensor(c, dtype=torch.float64, device=DEVICE).view(1, 3, 1, 1) * 255
    f = (f - col(MEAN)) / col(STD)
    t, h, w = f.shape[0] // 2, f.shape[2] // 14, f.shape[3] // 14
    f = f.view(t, 2, 3, h // 2, 2, 14, w // 2, 2, 14).permute(0, 3, 6, 4, 7, 2, 1, 5, 8).reshape(t * h * w, -1)
    E, heads = cfg.vit_embed_dim, cfg.vit_num_heads
    x = f @ P("visual.patch_embed.proj.weight").reshape(E, -1).T
    blocks = lambda g: g.view(h // 2, 2, w // 2, 2).transpose(1, 2).reshape(-1)
    ys, xs = torch.meshgrid(torch.arange(h, device=DEVICE), torch.arange(w, device=DEVICE), indexing="ij")
    half = E // heads // 2
    freq = 10000.0 ** (-torch.arange(0, half, 2, dtype=torch.float64, device=DEVICE) / half)
    angles = torch.cat([blocks(ys.contiguous())[:, None] * freq, blocks(xs.contiguous())[:, None] * freq], 1)
    for i in range(cfg.vit_depth):
        p = f"visual.blocks.{i}."
        y = layer_norm(x, P(p + "norm1.weight"), P(p + "norm1.bias")) @ P(p + "attn.qkv.weight").T + P(p + "attn.qkv.bias")
        q, k, v = y.view(t, h * w, 3, heads, -1).unbind(2)
        o = torch.cat([attend(rotate(q[j], angles), rotate(k[j], angles), v[j], (2 * half) ** -0.5, causal=False) for j in range(t)]).reshape(t * h * w, E)
        x = x + o @ P(p + "attn.proj.weight").T + P(p + "attn.proj.bias")
        y = layer_norm(x, P(p + "norm2.weight"), P(p + "norm2.bias")) @ P(p + "mlp.fc1.weight").T + P(p + "mlp.fc1.bias")
        x = x + (y * torch.sigmoid(1.702 * y)) @ P(p + "mlp.fc2.weight").T + P(p + "mlp.fc2.bias")
    m = "visual.merger."
    x = layer_norm(x, P(m + "ln_q.weight"), P(m + "ln_q.bias")).reshape(t * h * w // 4, 4 * E)
    x = torch.nn.functional.gelu(x @ P(m + "mlp.0.weight").T + P(m + "mlp.0.bias"))
    return x @ P(m + "mlp.2.weight").T + P(m + "mlp.2.bias")


def rotary_positions(cfg, ids, case):
    """[3, len(ids)] positions: behind a history every axis counts tokens; a first turn's clip counts time, height and width."""
    n = len(ids)
    pos = torch.arange(n, dtype=torch.float64, device=DEVICE).repeat(3, 1)
    if case["history"]:
        return pos
    a = ids.index(cfg.video_token_id)
    t, h, w = (case["frames"] + 1) // 2, case["height"] // 28, case["width"] // 28
    grid = torch.stack(torch.meshgrid(torch.arange(t), torch.arange(h), torch.arange(w), indexing="ij")).reshape(3, -1).to(DEVICE)
    pos[:, a:a + t * h * w] = (grid + a).double()
    pos[:, a + t * h * w:] += a + max(t, h, w) - (a + t * h * w)          # the text goes on behind the largest position
    return pos


def livecc(cfg, P, x, pos, parts):
    H, G, eps = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.rms_norm_eps
    freq = cfg.rope_theta ** (-torch.arange(0, 128, 2, dtype=torch.float64, device=DEVICE) / 128)
    axis = torch.tensor(sum(([i] * n for i, n in enumerate(cfg.mrope_section)), []), device=DEVICE)
    angles = pos[axis].T * freq
    for i in range(cfg.num_hidden_layers):
        p = f"language_model.layers.{i}."
        h = rms(x, eps) * P(p + "input_layernorm.weight")
        lin = lambda n: h @ P(p + f"self_attn.{n}_proj.weight").T + P(p + f"self_attn.{n}_proj.bias")
        q, k, v = rotate(lin("q").view(-1, H, 128), angles), rotate(lin("k").view(-1, G, 128), angles), lin("v").view(-1, G, 128)
        o = torch.cat([attend(q[a:b], k[a:b], v[a:b], 128 ** -0.5) for a, b in parts])
        x = x + o.reshape(len(x), -1) @ P(p + "self_attn.o_proj.weight").T
        x = x + gated(rms(x, eps) * P(p + "post_attention_layernorm.weight"), P, p + "mlp.gate_proj.weight", p + "mlp.up_proj.weight", p + "mlp.down_proj.weight")
    return rms(x, eps) * P("language_model.norm.weight")


def debunex(cfg, P, ids, parts):
    eps = cfg.norm_eps
    dyt = lambda x, n: torch.tanh(P(n + ".alpha") * x) * P(n) + P(n + ".b")
    x, latent = P("embed")[ids], {}
    for i, l in enumerate(cfg.layers):
        p, m = f"l{i}.", l.mixer
        h = dyt(x, p + "norm1")
        if m.kv_from is None:
            latent[i] = rms(h @ P(p + "mix.dkv").T, eps) * P(p + "mix.dkv.norm")
        c = latent[i if m.kv_from is None else m.kv_from]
        q = ((rms(h @ P(p + "mix.dq").T, eps) * P(p + "mix.dq.norm")) @ P(p + "mix.uq").T).view(len(x), m.heads, -1)
        k, v = (c @ P(p + "mix.uk").T).view(len(x), m.heads, -1), (c @ P(p + "mix.uv").T).view(len(x), m.heads, -1)
        o = torch.cat([attend(q[a:b], k[a:b], v[a:b], m.scale) for a, b in parts]) * torch.sigmoid(h @ P(p + "mix.g").T)[:, :, None]
        x = x + o.reshape(len(x), -1) @ P(p + "mix.o").T + gated(h, P, p + "mlp.gate", p + "mlp.up", p + "mlp.down")
    return dyt(x, "final.norm")


def bemuzen(cfg, P, ids, parts):
    eps, n = cfg.norm_eps, len(ids)
    first = torch.zeros(n, dtype=torch.bool, device=DEVICE)
    first[[a for a, _ in parts]] = True
    pair = (ids.roll(1) * cfg.bigram_mul_prev + ids * cfg.bigram_mul_cur) % cfg.bigram_buckets
    x = P("embed")[ids] + P("bigram")[torch.where(first, cfg.bigram_buckets, pair)]
    at = torch.cat([torch.arange(b - a, device=DEVICE) for a, b in parts]).double()
    norm = lambda y, name: rms(y, eps) * (1 + P(name))
    each = lambda f, *t: torch.cat([f(*(y[a:b] for y in t)) for a, b in parts])
    for i, l in enumerate(cfg.layers):
        p, m = f"l{i}.", l.mixer
        h = norm(x, p + "norm1")
        lin = lambda name, heads: (h @ P(p + "mix." + name).T).view(n, heads, -1)
        if hasattr(m, "left"):
            a, r = m.left, m.right
            q, k = rms(lin("left.q", a.heads), eps) * P(p + "mix.left.q.norm"), rms(lin("left.k", a.kv_heads), eps) * P(p + "mix.left.k.norm")
            q = q * (1 + a.q_temp_coef * torch.log(torch.floor((at + 1) / a.q_temp_every) + 1))[:, None, None]
            slopes = [2.0 ** (-8.0 * (j + 1) / a.heads) for j in range(a.heads)]
            left = each(lambda *t: attend(*t, a.scale, slopes=slopes), q, k, lin("left.v", a.kv_heads)).reshape(n, -1) @ P(p + "mix.left.o").T
            decay = torch.tensor(r.decay, dtype=torch.float64, device=DEVICE).log().expand(n, r.heads)
            o = each(decayed, silu(lin("right.q", r.heads)), silu(lin("right.k", r.heads)), silu(lin("right.v", r.heads)), decay, torch.ones_like(decay))
            o = rms(o.reshape(n, -1), eps) * P(p + "mix.right.norm") * torch.sigmoid(h @ P(p + "mix.right.g").T)
            y = 0.5 * (rms(left, eps) * P(p + "mix.left.out") + rms(o @ P(p + "mix.right.o").T, eps) * P(p + "mix.right.out"))
        else:
            inner, gn = m.heads * m.vdim, m.groups * m.state
            z, u, dt = torch.split(h @ P(p + "mix.in").T, [inner, inner + 2 * gn, m.heads], -1)
            w, taps = P(p + "mix.conv"), m.conv_taps

            def conv(s):
                s = torch.cat([s.new_zeros(taps - 1, s.shape[1]), s])
                return silu(sum(s[j:len(s) - taps + 1 + j] * w[:, j] for j in range(taps)) + P(p + "mix.conv.b"))
            v, B, C = torch.split(each(conv, u), [inner, gn, gn], -1)
            group = torch.arange(m.heads, device=DEVICE) // (m.heads // m.groups)
            v, B, C = v.reshape(n, m.heads, -1), B.reshape(n, m.groups, -1)[:, group], C.reshape(n, m.groups, -1)[:, group]
            dt = torch.nn.functional.softplus(dt + P(p + "mix.dt_bias"))
            o = each(decayed, C, B, v, -P(p + "mix.A_log").exp() * dt, dt) + P(p + "mix.D")[:, None] * v
            o = rms((o.reshape(n, -1) * silu(z)).view(n, m.norm_groups, -1), eps).reshape(n, inner) * P(p + "mix.norm")
            y = o @ P(p + "mix.o").T
        x = x + norm(y, p + "norm1b")
        x = x + norm(gated(norm(x, p + "norm2"), P, p + "mlp.gate", p + "mlp.up", p + "mlp.down"), p + "norm2b")
    return norm(x, "final.norm")


@torch.inference_mode()
def exact(case, seed):
    if case["kind"] == "resize":
        return None          # bytes
    if work(case)["flops"] * (1 + case.get("history", 0) / 400) > 2.5e14:
        return None
    cfg = get_config(case["model"])
    params = Checkpoint(cfg)

    def P(name):
        w = params(name).double()
        return e4m3_rows(w) if case.get("fp8") and w.dim() == 2 and name.startswith(("language_model.layers", "lm_head")) else w

    if case["kind"] == "clip":
        return tower(cfg, P, pictures(case["frames"], case["height"], case["width"], seed, "TCHW"))
    V, N = cfg.vocab_size, case["tokens"]
    back = pow(PERM_MUL, -1, V)
    whole, parts, want = [], [], []
    for ids in [past + new for past, new in turn_ids(cfg, case, seed)] if case["kind"] == "turn" else prompts(cfg, case, seed):
        said = list(ids)
        for _ in range(N - 1):          # every token's clear successor: the head's row that is its embedding's
            said.append((said[-1] - PERM_ADD) * back % V)
        parts.append((len(whole), len(whole) + len(said)))
        whole += said
        want += range(len(whole) - N, len(whole))
    ids = torch.tensor(whole, device=DEVICE)
    if case["kind"] == "turn":
        x = params(params.embed)[ids].double()
        seen = torch.cat([tower(cfg, P, pictures(case["frames"], case["height"], case["width"], seed + 7 * i, "TCHW")) for i in range(case["streams"])])
        x[ids == cfg.video_token_id] = seen
        pos = torch.cat([rotary_positions(cfg, whole[a:b], case) for a, b in parts], 1)
        x = livecc(cfg, P, x, pos, parts)[want]
    else:
        x = (bemuzen if isinstance(cfg, BemuzenConfig) else debunex)(cfg, P, ids, parts)[want]
    logits = torch.cat([x @ params(params.head)[a:a + 16384].double().T for a in range(0, V, 16384)], 1) if not case.get("fp8") else x @ P(params.head).T
    if isinstance(cfg, BemuzenConfig):
        logits = logits * cfg.logit_scale
    elif params.decoder and cfg.logit_softcap:
        logits = cfg.logit_softcap * torch.tanh(logits / cfg.logit_softcap)
    return {"tokens": None, "logits": list(logits.view(len(parts), N, V))}
