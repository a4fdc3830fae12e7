"""What is timed: the work a user of this framework has it do, through its public entry points.

Seven kinds of calls, each over a range of sizes (`draw`) with listed points in it:

  frames          the SigLIP-so400m-384 tower (26 of 27 blocks run) on a clip's frames, bf16: the first stage of every video question
  prompt          one text or video prompt through a slice of the Nemotron-Nano-9B-v2 hybrid stack (true widths, 3 Mamba-2, 3 MLP and
                  one attention layer, cache filled, last position's logits)
  answer          16 tokens behind a cached prefix on the same slice, batch 1 to 16, replayed from a captured step
  mixer           the operators between the two projections of a Mamba-2 mixer, called as a model's own code calls them: causal conv +
                  split, selective scan with final state, gated norm (bf16 at the 9B geometry; fp32 at the 32-head, state-16 one)
  attend          causal GQA attention of one prompt (40 heads on 8, or 28 on 4, of 128), bf16
  window_prompts  several prompts of different lengths as one packed step of a window-attention model (Fogorax, width 2 048)
  window_answer   16 tokens for each of up to 16 running requests of that model

Weights and inputs are random (there are no checkpoints here) at the models' own initialisations and sizes.  An answer's tokens are
given, not sampled: greedy choices of random weights hang on the last bit of two logits."""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from timeviper_amd import kernels as K
from timeviper_amd.model.llm.decode_graph import GraphedDecodeStep
from timeviper_amd.model.llm.fogorax import FogoraxConfig, FogoraxForCausalLM
from timeviper_amd.model.llm.nano import NemotronHConfig, NemotronHForCausalLM
from timeviper_amd.model.vit import TimmViTBackbone

ANSWER = 16
VOCAB = 32768
PATTERN = "M-M-M*-"                       # a stretch of the 56-layer pattern: M : MLP : attention = 27 : 25 : 4 there
BF = torch.bfloat16
# window-attention model: the sizes of `bench.py --config fogorax`
WIDTH, LAYERS, HEADS, KV, HD, WINDOW, KEEP, FF, SIDE, POSITIONS = 2048, 8, 16, 4, 128, 1024, 64, 5632, 128, 16384
# Mamba-2 mixer geometries: (heads, head dim, groups, state)
GEOMETRY = {"9b": (128, 80, 8, 128), "small": (32, 64, 2, 16)}


def listed():
    return [
        # a short clip (a second or two of video) and a minute of it
        {"name": "frames_4", "kind": "frames", "frames": 4},
        {"name": "frames_48", "kind": "frames", "frames": 48},
        # a question with a system prompt; a clip of about ten minutes (16 tokens a frame) with its question
        {"name": "prompt_203", "kind": "prompt", "tokens": 203},
        {"name": "prompt_10007", "kind": "prompt", "tokens": 10007},
        # one user behind a long video; a batch of questions about shorter ones
        {"name": "answer_1x9003", "kind": "answer", "batch": 1, "tokens": 9003},
        {"name": "answer_12x1501", "kind": "answer", "batch": 12, "tokens": 1501},
        # a text prompt's mixer, an hour of video's, and the fp32 configuration
        {"name": "mixer_1501", "kind": "mixer", "geometry": "9b", "dtype": "bf16", "batch": 1, "tokens": 1501},
        {"name": "mixer_49999", "kind": "mixer", "geometry": "9b", "dtype": "bf16", "batch": 1, "tokens": 49999},
        {"name": "mixer_fp32_1024", "kind": "mixer", "geometry": "small", "dtype": "fp32", "batch": 1, "tokens": 1024},
        # attention of a prompt of a few thousand tokens
        {"name": "attend_5003", "kind": "attend", "heads": 40, "kv_heads": 8, "tokens": 5003},
        # requests that arrive together; requests that run together
        {"name": "window_prompts_6", "kind": "window_prompts", "prompts": 6, "tokens": 6011},
        {"name": "window_answer_4x2500", "kind": "window_answer", "batch": 4, "tokens": 2500},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(["frames", "prompt", "answer", "mixer", "attend", "window_prompts", "window_answer"])
    if kind == "frames":
        return {"kind": kind, "frames": size(1, 48)}
    if kind == "prompt":
        return {"kind": kind, "tokens": size(17, 10007)}
    if kind == "answer":
        batch = size(1, 16)
        return {"kind": kind, "batch": batch, "tokens": size(260, max(600, 18000 // batch))}
    if kind == "mixer":
        if rng.random() < 0.25:
            return {"kind": kind, "geometry": "small", "dtype": "fp32", "batch": rng.randint(1, 2), "tokens": size(64, 4096)}
        return {"kind": kind, "geometry": "9b", "dtype": "bf16", "batch": 1, "tokens": size(40, 49999)}
    if kind == "attend":
        heads, kv = rng.choice([(40, 8), (28, 4)])
        return {"kind": kind, "heads": heads, "kv_heads": kv, "tokens": size(200, 16384)}
    if kind == "window_prompts":
        n = rng.randint(1, 8)
        return {"kind": kind, "prompts": n, "tokens": size(16 * n, 8192)}
    return {"kind": kind, "batch": size(1, 16), "tokens": size(100, 8000)}


def _gen(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed(1_000_003 * (seed % (1 << 40)) + salt)


# ------------------------------------------------------------------ frames
def _tower(seed):
    with torch.device("meta"):
        tower = TimmViTBackbone("siglip-vit-so400m-384px")
    tower = tower.to(BF).to_empty(device="cuda")
    g = _gen(seed, 1)
    with torch.no_grad():
        for name, p in tower.named_parameters():
            if "norm" in name and name.endswith("weight"):
                p.copy_(1 + 0.1 * torch.randn(p.shape, generator=g, device="cuda"))
            elif name.endswith("bias"):
                p.normal_(0.0, 0.02, generator=g)
            elif name.endswith("pos_embed"):
                p.normal_(0.0, 0.5, generator=g)
            else:
                p.normal_(0.0, 0.03, generator=g)
    return tower.requires_grad_(False).eval()


def _pixels(case, seed):
    return torch.randn((case["frames"], 3, 384, 384), generator=_gen(seed, 2), device="cuda").to(BF)


def _frames_exact(case, seed):
    tower = _tower(seed)
    W = {n: p.double() for n, p in tower.named_parameters()}
    out = []
    for px in _pixels(case, seed).double().split(4):
        p = "featurizer."
        w = W[p + "patch_embed.proj.weight"]
        patches = px[:, :, :378, :378].unfold(2, 14, 14).unfold(3, 14, 14).permute(0, 2, 3, 1, 4, 5).reshape(px.shape[0], 729, -1)
        x = patches @ w.reshape(w.shape[0], -1).t() + W[p + "patch_embed.proj.bias"] + W[p + "pos_embed"]
        for i in range(26):
            b = f"{p}blocks.{i}."
            lin = lambda t, n: t @ W[b + n + ".weight"].t() + W[b + n + ".bias"]
            h = F.layer_norm(x, (1152,), W[b + "norm1.weight"], W[b + "norm1.bias"], 1e-6)
            q, k, v = (t.transpose(1, 2).contiguous() for t in lin(h, "attn.qkv").view(-1, 729, 3, 16, 72).unbind(2))
            a = torch.softmax(torch.matmul(q, k.transpose(2, 3).contiguous()) * 72 ** -0.5, -1)
            x = x + lin(torch.matmul(a, v).transpose(1, 2).reshape(-1, 729, 1152), "attn.proj")
            h = F.layer_norm(x, (1152,), W[b + "norm2.weight"], W[b + "norm2.bias"], 1e-6)
            x = x + lin(F.gelu(lin(h, "mlp.fc1")), "mlp.fc2")
        out.append(x)
    return torch.cat(out)


# ------------------------------------------------------------------ the hybrid slice
def _hybrid_config():
    return NemotronHConfig.nemotron_nano_9b_v2(vocab_size=VOCAB, num_hidden_layers=len(PATTERN), hybrid_override_pattern=PATTERN)


def _hybrid(seed):
    cfg = _hybrid_config()
    with torch.device("meta"):
        llm = NemotronHForCausalLM(cfg)
    llm = llm.to(BF).to_empty(device="cuda")
    g = _gen(seed, 3)
    with torch.no_grad():
        for name, p in llm.named_parameters():
            if name.endswith("A_log"):
                p.copy_(torch.log(torch.rand(p.shape, generator=g, device="cuda") * 15 + 1))
            elif name.endswith("dt_bias"):
                dt = torch.exp(torch.rand(p.shape, generator=g, device="cuda") * math.log(100.0) + math.log(1e-3))
                p.copy_(dt + torch.log(-torch.expm1(-dt)))
            elif name.endswith(".D") or "norm" in name.split(".")[-2]:
                p.copy_(1 + 0.1 * torch.randn(p.shape, generator=g, device="cuda"))
            elif "conv1d" in name:
                p.uniform_(-0.5, 0.5, generator=g)
            else:
                p.normal_(0.0, 0.02, generator=g)
    return llm.requires_grad_(False).eval()


def _ids(case, seed, extra=0):
    return torch.randint(0, VOCAB, (case.get("batch", 1), case["tokens"] + extra), generator=_gen(seed, 4), device="cuda")


def _prefill(llm, ids):
    cache = llm.new_cache(ids.shape[0])
    out = llm(input_ids=ids, past_key_values=cache, use_cache=True, cache_position=torch.arange(ids.shape[1]))
    return cache, out.logits


def _mamba_layers(cfg):
    return [i for i, c in enumerate(cfg.hybrid_override_pattern) if c == "M"]


def _rms64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _scan64(x, dt, A, B, C, D):
    """x (L, H, P), dt (L, H) after softplus, A (H), B / C (L, G, N): outputs and final state (H, P, N), in chunks of 64 tokens"""
    L, H, P = x.shape
    G, N = B.shape[1:]
    y, S = torch.empty_like(x), x.new_zeros((H, P, N))
    head = lambda t: t.repeat_interleave(H // G, 1).transpose(0, 1).contiguous()      # (H, Q, N)
    for t0 in range(0, L, 64):
        xc, dtc, b, c = x[t0:t0 + 64].transpose(0, 1), dt[t0:t0 + 64].t(), head(B[t0:t0 + 64]), head(C[t0:t0 + 64])
        cs = torch.cumsum(dtc * A[:, None], 1)                                        # (H, Q)
        Q = cs.shape[1]
        mask = torch.ones(Q, Q, dtype=torch.bool, device=x.device).tril()
        M = torch.exp((cs[:, :, None] - cs[:, None, :]).masked_fill(~mask, -math.inf)) * torch.bmm(c, b.transpose(1, 2).contiguous())
        xd = (xc * dtc[:, :, None]).contiguous()
        yc = torch.bmm(M, xd) + torch.exp(cs)[:, :, None] * torch.bmm(c, S.transpose(1, 2).contiguous())
        S = torch.exp(cs[:, -1])[:, None, None] * S + torch.bmm((xd * torch.exp(cs[:, -1:] - cs)[:, :, None]).transpose(1, 2).contiguous(), b)
        y[t0:t0 + 64] = (yc + xc * D[:, None, None]).transpose(0, 1)
    return y, S


def _mixer64(xbc, dt, gate, w, bias, A, D, dt_bias, norm_w, geometry, eps):
    """conv + split, scan, gated norm: (normed rows, final state)"""
    H, P, G, N = geometry
    c = F.conv1d(F.pad(xbc.t()[None], (3, 0)), w[:, None], bias, groups=w.shape[0])[0].t()
    x, B, C = F.silu(c).split([H * P, G * N, G * N], 1)
    y, S = _scan64(x.reshape(-1, H, P).contiguous(), F.softplus(dt + dt_bias), A, B.reshape(-1, G, N), C.reshape(-1, G, N), D)
    u = (y.reshape(-1, H * P) * F.silu(gate)).unflatten(1, (G, -1))
    return _rms64(u, 1.0, eps).flatten(1) * norm_w, S


def _attention64(q, k, v, window=None, keep=0):
    """causal, q (L, H, d), k / v (L, G, d)"""
    L, H, d = q.shape
    out = torch.empty_like(q)
    pos = torch.arange(L, device=q.device)
    for h in range(H):
        kh, vh = k[:, h // (H // k.shape[1])], v[:, h // (H // k.shape[1])]
        kt = kh.t().contiguous()
        for r in range(0, L, 4096):
            p = pos[r:r + 4096, None]
            see = pos[None] <= p
            if window is not None:
                see &= (p - pos[None] < window) | (pos[None] < keep)
            s = (q[r:r + 4096, h] @ kt * d ** -0.5).masked_fill_(~see, -math.inf)
            out[r:r + 4096, h] = torch.softmax(s, -1) @ vh
    return out


def _hybrid64(llm, ids, keep):
    """One sequence: logits of the last `keep` positions, and what the cache holds (per Mamba layer the state and the last four
    inputs of the convolution, per attention layer keys and values)"""
    cfg = llm.config
    W = {n: p.double() for n, p in llm.named_parameters()}
    geo = GEOMETRY["9b"]
    d_in, conv = geo[0] * geo[1], geo[0] * geo[1] + 2 * geo[2] * geo[3]
    eps = cfg.layer_norm_epsilon
    x = W["backbone.embeddings.weight"][ids]
    ssm, convs, kv = [], [], []
    for i, c in enumerate(PATTERN):
        p = f"backbone.layers.{i}."
        h, m = _rms64(x, W[p + "norm.weight"], eps), p + "mixer."
        if c == "M":
            gate, xbc, dt = (h @ W[m + "in_proj.weight"].t()).split([d_in, conv, geo[0]], 1)
            y, S = _mixer64(xbc, dt, gate, W[m + "conv1d.weight"][:, 0], W[m + "conv1d.bias"], -torch.exp(W[m + "A_log"]), W[m + "D"],
                            W[m + "dt_bias"], W[m + "norm.weight"], geo, eps)
            x = x + y @ W[m + "out_proj.weight"].t()
            ssm.append(S)
            convs.append(xbc[-4:].t())
        elif c == "-":
            x = x + F.relu(h @ W[m + "up_proj.weight"].t()).square() @ W[m + "down_proj.weight"].t()
        else:
            q, k, v = ((h @ W[m + n + "_proj.weight"].t()).unflatten(1, (-1, 128)) for n in "qkv")
            x = x + _attention64(q, k, v).flatten(1) @ W[m + "o_proj.weight"].t()
            kv.append((k, v))
    return _rms64(x[-keep:], W["backbone.norm_f.weight"], eps) @ W["lm_head.weight"].t(), ssm, convs, kv


def _prompt_outputs(logits, ssm, convs, kv):
    return {"logits": logits, "ssm": ssm, "conv": convs, "keys": [k for k, _ in kv], "values": [v for _, v in kv]}


# ------------------------------------------------------------------ the window-attention model
def _window_config():
    layers = []
    for i in range(LAYERS):                   # every second layer reads the keys and values of the one in front
        m = {"heads": HEADS, "kv_heads": KV, "dim": HD, "vdim": HD, "scale": HD ** -0.5, "mask": {"size": WINDOW, "keep_first": KEEP}}
        if i % 2:
            m["kv_from"] = i - 1
        layers.append({"type": "attention", "mixer": m, "mlp": {"kind": "dense", "ff": FF}})
    return FogoraxConfig(vocab_size=VOCAB, hidden_size=WIDTH, layers=layers, side_dim=SIDE, max_positions=POSITIONS)


def _window_model(seed):
    cfg = _window_config()
    with torch.device("meta"):
        llm = FogoraxForCausalLM(cfg)
    llm = llm.to(BF).to_empty(device="cuda")
    g = _gen(seed, 5)
    with torch.no_grad():
        for name, p in llm.named_parameters():
            leaf = name.rsplit(".", 1)[-1]
            r = lambda: torch.randn(p.shape, generator=g, device="cuda")
            if leaf in ("gain", "final_gain", "norm"):
                p.copy_(1 + 0.1 * r())
            elif leaf == "shift":
                p.copy_(0.3 + 0.2 * r())
            elif leaf in ("inp_bias", "out_bias"):
                p.copy_(0.02 * r())
            else:
                p.normal_(0.0, 0.02, generator=g)
    return llm.requires_grad_(False).eval()


def _lengths(case):
    """lengths of the prompts of a step: from a short remark to a long document"""
    n, total = case["prompts"], case["tokens"]
    parts = [1.6 ** i for i in range(n)]
    got = [max(1, int(total * p / sum(parts))) for p in parts]
    got[-1] += max(0, total - sum(got))
    return got


def _window64(llm, ids, keep):
    """One sequence: logits of the last `keep` positions, cache rows of the layers that have their own, the last h of every layer"""
    W = {n: p.double() for n, p in llm.named_parameters()}
    eps, L = llm.config.norm_eps, ids.numel()
    x = W["backbone.embed.weight"][ids] + W["backbone.positions"][:L]
    rows, last, k, v = [], [], None, None
    for i in range(LAYERS):
        p = f"backbone.layers.{i}."
        h = _rms64(x, W[p + "gain"], eps)
        hs = h + (F.pad(h, (0, 0, 1, 0))[:-1] - h) * W[p + "shift"]
        last.append(h[-1])
        own = i % 2 == 0
        inp, n1 = W[p + "inp"], 2 * HEADS * HD + (2 * KV * HD if own else 0)
        pr = hs @ inp[:n1].t()
        if own:
            q, k, v, gate = pr.split([HEADS * HD, KV * HD, KV * HD, HEADS * HD], 1)
            rows.append(torch.cat([k, v], 1))
            k, v = k.unflatten(1, (KV, HD)), v.unflatten(1, (KV, HD))
        else:
            q, gate = pr.split([HEADS * HD, HEADS * HD], 1)
        o = _attention64(q.unflatten(1, (HEADS, HD)), k, v, WINDOW, KEEP).flatten(1) * torch.sigmoid(gate)
        a, b = (h @ inp[n1:].t() + W[p + "inp_bias"]).split(FF, 1)
        x = x + torch.cat([o, F.gelu(a, approximate="tanh") * b], 1) @ W[p + "out"].t() + W[p + "out_bias"]
        e = W["backbone.side_embed"][ids, i * SIDE:(i + 1) * SIDE]
        s = (F.gelu(x @ W[p + "side.gate"].t(), approximate="tanh") * e) @ W[p + "side.proj"].t()
        x = x + _rms64(s, W[p + "side.norm"], eps)
    return _rms64(x[-keep:], W["backbone.final_gain"], eps) @ W["head"].t(), rows, last


# ------------------------------------------------------------------ prepare
def _rewinder(cache, saved, plan=None):
    """Back to the end of the prefix behind an answer: the recurrent rows are copied back, the positions are set back; keys and values
    behind the prefix are overwritten by the next answer."""
    host = cache.host_state()

    def rewind():
        for to, was in saved:
            to.copy_(was)
        cache.restore_host_state(host)
        if plan is not None:
            plan.moving.sub_(ANSWER)
        else:
            for pos, lens in cache._static.values():
                pos.sub_(ANSWER)
                lens.sub_(ANSWER)
    return rewind


def _answering(cache, step, batch, tokens, saved, plan=None):
    """The captured step of a generation, its tokens, and the way back to the prefix.  (Two eager tokens and the captured one; the
    rest of the first answer brings the positions to where every answer ends.)"""
    rewind = _rewinder(cache, saved, plan)
    stepper = GraphedDecodeStep(step, cache, batch, "cuda")
    for t in tokens:
        stepper.step(t)
    if stepper.graph is None:
        raise RuntimeError(f"the step was not captured: {stepper.capture_error}")
    return {"stepper": stepper, "tokens": tokens, "rewind": rewind}


@torch.inference_mode()
def prepare(case, seed):
    kind, s = case["kind"], {"kind": case["kind"]}
    if kind == "frames":
        s["tower"], s["pixels"] = _tower(seed), _pixels(case, seed)
    elif kind == "prompt":
        s["llm"], s["ids"] = _hybrid(seed), _ids(case, seed)
    elif kind == "answer":
        llm, ids, B = _hybrid(seed), _ids(case, seed, ANSWER), case["batch"]
        cache, _ = _prefill(llm, ids[:, :-ANSWER])
        mamba = _mamba_layers(llm.config)
        cache.begin_static_decode(ANSWER)
        saved = [(t, t.clone()) for i in mamba for t in (cache.conv_states[i], cache.ssm_states[i])]
        one = torch.ones(1, dtype=torch.long)
        step = lambda t: llm(input_ids=t, past_key_values=cache, use_cache=True, cache_position=one).logits
        s.update(_answering(cache, step, B, [t.contiguous() for t in ids[:, -ANSWER:].split(1, 1)], saved), ssm=[cache.ssm_states[i] for i in mamba])
    elif kind == "mixer":
        H, P, G, N = GEOMETRY[case["geometry"]]
        dt = BF if case["dtype"] == "bf16" else torch.float32
        g, B, L = _gen(seed, 6), case["batch"], case["tokens"]
        d_in, conv = H * P, H * P + 2 * G * N
        r = lambda *sh: torch.randn(sh, generator=g, device="cuda")
        u = lambda *sh: torch.rand(sh, generator=g, device="cuda")
        proj = torch.empty((B, L, d_in + conv + H), dtype=dt, device="cuda").normal_(0.0, 1.3, generator=g)
        dtv = torch.exp(u(H) * math.log(100.0) + math.log(1e-3))
        s.update(geometry=(H, P, G, N), gate=proj[..., :d_in], xbc=proj[..., d_in:d_in + conv], dt=proj[..., d_in + conv:],
                 w=(u(conv, 4) - 0.5).to(dt), bias=(u(conv) - 0.5).to(dt), A=-(u(H) * 15 + 1), D=1 + 0.1 * r(H),
                 dt_bias=dtv + torch.log(-torch.expm1(-dtv)), norm=(1 + 0.1 * r(d_in)).to(dt))
    elif kind == "attend":
        g, L = _gen(seed, 7), case["tokens"]
        r = lambda h: (1.3 * torch.randn((1, L, h, 128), generator=g, device="cuda")).to(BF)
        s["q"], s["k"], s["v"] = r(case["heads"]), r(case["kv_heads"]), r(case["kv_heads"])
    elif kind == "window_prompts":
        llm, n = _window_model(seed), _lengths(case)
        ids = torch.randint(0, VOCAB, (sum(n),), generator=_gen(seed, 8), device="cuda")
        ends = torch.tensor(n).cumsum(0) - 1
        s.update(llm=llm, ids=ids, counts=n, at=ends.cuda(), cache=llm.new_cache(len(n), capacity=max(n)))
        for slot in s["cache"].default_slots:
            s["cache"].free(slot)
    else:
        llm, B = _window_model(seed), case["batch"]
        ids = _ids(case, seed, ANSWER)
        cache = llm.new_cache(B, capacity=case["tokens"] + ANSWER)
        llm(input_ids=ids[:, :-ANSWER], past_key_values=cache, use_cache=True)
        cache.begin_static_decode(ANSWER)
        plan = cache.plan(cache.default_slots, [1] * B)
        saved = [(cache.state(0), cache.state(0).clone())]
        step = lambda t: llm(input_ids=t, past_key_values=cache, use_cache=True).logits
        s.update(_answering(cache, step, B, [t.contiguous() for t in ids[:, -ANSWER:].split(1, 1)], saved, plan), shift=cache.state(0))
    return s


# ------------------------------------------------------------------ run
@torch.inference_mode()
def run(s):
    kind = s["kind"]
    if kind == "frames":
        return s["tower"](s["pixels"])
    if kind == "prompt":
        llm = s["llm"]
        cache, logits = _prefill(llm, s["ids"])
        m, a = _mamba_layers(llm.config), cache.attention_layers
        return _prompt_outputs(logits, [cache.ssm_states[i] for i in m], [cache.conv_states[i] for i in m],
                               [(cache.key_cache[i], cache.value_cache[i]) for i in a])
    if kind == "mixer":
        H, P, G, N = s["geometry"]
        B, L = s["dt"].shape[:2]
        x, Bm, Cm, cb = K.causal_conv1d_xbc(s["xbc"], s["w"], s["bias"], H * P, G, N, activation="silu", return_cb=True)
        y, state = K.mamba_chunk_scan_combined(x.view(B, L, H, P), s["dt"], s["A"], Bm, Cm, chunk_size=128, D=s["D"], dt_bias=s["dt_bias"],
                                               dt_softplus=True, return_final_states=True, cb=cb)
        return K.rmsnorm_fn(x=y.view(B, L, H * P), weight=s["norm"], bias=None, z=s["gate"], eps=1e-5, group_size=H * P // G,
                            norm_before_gate=False), state
    if kind == "attend":
        return K.flash_attn_func(s["q"], s["k"], s["v"], causal=True)
    if kind == "window_prompts":
        llm, cache, n = s["llm"], s["cache"], s["counts"]
        slots = [cache.alloc() for _ in n]
        logits = llm.step(s["ids"], cache, cache.plan(slots, n), logits_at=s["at"])
        out = {"logits": logits, "rows": [cache.tokens(e)[slot, :c] for e in range(1, 1 + LAYERS // 2) for slot, c in zip(slots, n)],
               "shift": [cache.state(0)[slot, :, (c - 1) & 1] for slot, c in zip(slots, n)]}
        for slot in slots:
            cache.free(slot)
        return out
    # answers: back to the prefix, then the captured step for each token
    s["rewind"]()
    stepper, got = s["stepper"], []
    for t in s["tokens"]:
        stepper.step(t)
        got.append(stepper.logits.clone())
    out = {"logits": torch.stack(got)}
    out.update({"ssm": s["ssm"]} if kind == "answer" else {"shift": s["shift"]})
    return out


# ------------------------------------------------------------------ exact
@torch.inference_mode()
def exact(case, seed):
    kind = case["kind"]
    if kind == "frames":
        return _frames_exact(case, seed)
    if kind == "prompt":
        logits, ssm, convs, kv = _hybrid64(_hybrid(seed), _ids(case, seed)[0], 1)
        return _prompt_outputs(logits[None], [t[None] for t in ssm], [t[None] for t in convs], [(k[None], v[None]) for k, v in kv])
    if kind == "answer":
        if case["batch"] * case["tokens"] > 30000:
            return None
        llm = _hybrid(seed)
        got = [_hybrid64(llm, ids, ANSWER)[:2] for ids in _ids(case, seed, ANSWER)]
        return {"logits": torch.stack([l for l, _ in got], 1), "ssm": [torch.stack(t) for t in zip(*(ssm for _, ssm in got))]}
    if kind == "mixer":
        s = prepare(case, seed)
        w = {k: t.double() for k, t in s.items() if isinstance(t, torch.Tensor)}
        got = [_mixer64(w["xbc"][b], w["dt"][b], w["gate"][b], w["w"], w["bias"], w["A"], w["D"], w["dt_bias"], w["norm"], s["geometry"], 1e-5)
               for b in range(case["batch"])]
        return tuple(torch.stack(t) for t in zip(*got))
    if kind == "attend":
        s = prepare(case, seed)
        return _attention64(*(s[n][0].double() for n in "qkv"))[None]
    if kind == "window_prompts":
        llm, n = _window_model(seed), _lengths(case)
        ids = torch.randint(0, VOCAB, (sum(n),), generator=_gen(seed, 8), device="cuda")
        got = [_window64(llm, t, 1) for t in ids.split(n)]
        return {"logits": torch.cat([l for l, _, _ in got]), "rows": [rows[e] for e in range(LAYERS // 2) for _, rows, _ in got],
                "shift": [torch.stack(last) for _, _, last in got]}
    llm = _window_model(seed)
    got = [_window64(llm, ids, ANSWER) for ids in _ids(case, seed, ANSWER)]
    # (the shift rows hold the two last tokens; only their outcome in the logits is restated)
    return {"logits": torch.stack([l for l, _, _ in got], 1), "shift": None}


# ------------------------------------------------------------------ work
def _causal_pairs(L):
    return L * (L + 1) / 2


def _window_pairs(start, L):
    p = torch.arange(start, start + L, dtype=torch.float64)
    lo = (p + 1 - WINDOW).clamp(min=0)
    return float((p + 1 - lo + lo.clamp(max=KEEP)).sum())


def work(case):
    """Each weight, input and cache row read once, each output written once; products, attention pairs and the scan's recurrence."""
    kind = case["kind"]
    H, P, G, N = GEOMETRY["9b"]
    m_in, d_in = 2 * H * P + 2 * G * N + H, H * P
    matrices = sum({"M": 4480 * (m_in + d_in), "-": 2 * 4480 * 15680, "*": 4480 * (2 * 5120 + 2048)}[c] for c in PATTERN)
    n_m, n_a = PATTERN.count("M"), PATTERN.count("*")
    if kind == "frames":
        n, block = case["frames"], 4 * 1152 * 1152 + 2 * 1152 * 4304
        return {"bytes": 26 * block * 2 + n * (3 * 384 * 384 + 729 * 1152) * 2,
                "flops": n * (2 * 729 * (26 * block + 588 * 1152) + 26 * 4 * 729 * 729 * 1152)}
    if kind == "prompt":
        L = case["tokens"]
        return {"bytes": matrices * 2 + VOCAB * 4480 * 2 + L * (4480 + n_a * 2048) * 2 + n_m * H * P * N * 4,
                "flops": 2 * L * matrices + n_a * _causal_pairs(L) * 4 * 5120 + n_m * L * H * P * N * 4}
    if kind == "answer":
        B, L = case["batch"], case["tokens"]
        kv = sum(B * (L + i + 1) * n_a * 2048 * 2 for i in range(ANSWER))
        step = matrices * 2 + VOCAB * 4480 * 2 + B * VOCAB * 4 + n_m * B * H * P * N * 8
        return {"bytes": ANSWER * step + kv, "flops": ANSWER * B * 2 * (matrices + VOCAB * 4480) + kv * 5}
    if kind == "mixer":
        h, p, g, n = GEOMETRY[case["geometry"]]
        T, e = case["batch"] * case["tokens"], 2 if case["dtype"] == "bf16" else 4
        return {"bytes": T * (3 * h * p + 2 * g * n + h) * e + case["batch"] * h * p * n * 4, "flops": T * h * p * (4 * n + 30)}
    if kind == "attend":
        L, h = case["tokens"], case["heads"]
        return {"bytes": L * 128 * 2 * (2 * h + 2 * case["kv_heads"]), "flops": _causal_pairs(L) * 4 * 128 * h}
    inner, own = HEADS * HD, 2 * KV * HD
    layer = WIDTH * (2 * inner + 2 * FF) + WIDTH * (inner + FF) + 2 * WIDTH * SIDE
    matrices = LAYERS * layer + LAYERS // 2 * WIDTH * own
    if kind == "window_prompts":
        n = _lengths(case)
        T = sum(n)
        return {"bytes": matrices * 2 + VOCAB * WIDTH * 2 + T * (2 * WIDTH + LAYERS * SIDE + LAYERS // 2 * own) * 2 + len(n) * VOCAB * 4,
                "flops": 2 * T * matrices + LAYERS * sum(_window_pairs(0, c) for c in n) * 4 * inner + 2 * len(n) * WIDTH * VOCAB}
    B, L = case["batch"], case["tokens"]
    pairs = B * _window_pairs(L, ANSWER)
    return {"bytes": ANSWER * (matrices * 2 + VOCAB * WIDTH * 2 + B * VOCAB * 4) + LAYERS // 2 * pairs * own * 2,
            "flops": ANSWER * B * 2 * (matrices + VOCAB * WIDTH) + LAYERS * pairs * 4 * inner}


def tolerance(case):
    """Relative error of another implementation at the same precision, about four times what is seen against 64 bits: attention alone
    0.002, a mixer's operators 0.003 (fp32: 4e-6), a stack of layers with bf16 activations between them 0.007 to 0.016."""
    if case["kind"] == "mixer":
        return {"rel": 1.5e-5, "max": 1e-3} if case["dtype"] == "fp32" else {"rel": 1.2e-2}
    return {"rel": 8e-3} if case["kind"] == "attend" else {"rel": 3e-2}
