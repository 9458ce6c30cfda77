"""Workloads the driver is measured on, through its public boundary: a `Driver` holding weights and the paged
KV cache, and forward passes over batches of requests.

A pass is one `Driver.forward` of a frame a serving loop would send, followed by reading back the logits the
tokens were chosen from.  The frame appends to contexts that earlier passes left in the cache: it writes the
same tokens into the same cache slots every time it is sent, so a pass can be repeated.

Requests of a pass are of two kinds: single decoded tokens behind a context, and portions of a prompt (the whole
of it, or what a chunked prefill reads beside other requests' decoding).  Contexts are copies of a prefilled
prompt's pages (fork by copy), so every request reads its own memory.  Weights are random (no checkpoint is needed
to time them) in the storage formats and shapes the driver serves.

The logits stand for the pass: a random model's are nearly flat, so which of two close ones is the larger is a
matter of rounding, and the tokens are left out.
"""
from __future__ import annotations

import json
import math
import random
import shutil
import tempfile

import numpy as np
import torch

from pie_amd import driver as drv

PAGE = 16
MAX_TOKENS = 2048    # a prefill chunk
MAX_REQUESTS = 64

# The decoders the benchmark names.  Embedding rows of standard deviation 16 make a token's own embedding carry the
# residual stream, as in the benchmark's mixture: distinct tokens then take distinct routes through the experts, and
# rounding does not grow from layer to layer.  (The small model's embedding is its head too, hence its smaller one.)
DENSE_8B = dict(arch="llama3", hidden=4096, layers=32, q_heads=32, kv_heads=8, head_dim=128, intermediate=14336,
                rope_theta=500000.0, embed_std=16.0)
DENSE_1B = dict(arch="llama3", hidden=2048, layers=16, q_heads=32, kv_heads=8, head_dim=64, intermediate=8192,
                rope_theta=500000.0, tie_embeddings=True, embed_std=2.0)
MOE_30B = dict(arch="qwen3_moe", hidden=2048, layers=48, q_heads=32, kv_heads=4, head_dim=128, intermediate=0,
               rope_theta=1000000.0, num_experts=128, top_k=8, expert_intermediate=768, router_std=0.0221, embed_std=16.0)
MODELS = {"dense 8b": DENSE_8B, "dense 1b": DENSE_1B, "mixture 30b": MOE_30B}
STACKS = {
    "stack 4096": dict(width=4096, heads=32, dim=128, rot_dim=64, vdim=128, q_rank=1536, kv_rank=512, ff=14336),
    "stack 2048": dict(width=2048, heads=16, dim=128, rot_dim=64, vdim=128, q_rank=768, kv_rank=512, ff=8192),
}
STACK_LAYERS = 6


def _case(name, model, *, quant="int4b8", kv="auto", vocab=32000, decode=0, context=0, prompts=0, tokens=0, history=0,
          ragged=0.0, sampler="greedy"):
    c = dict(model=model, quant=quant, kv=kv, vocab=vocab, decode=decode, context=context, prompts=prompts, tokens=tokens,
             history=history, ragged=ragged, sampler=sampler)
    return dict(c, name=name) if name else c


def listed():
    return [
        # The smallest call: a chat turn's first tokens on the small model, where launches and latency are all there is.
        _case("1b int8 decode x1", "dense 1b", quant="int8", vocab=128256, decode=1, context=128),
        # A short question read by the small model before its first token.
        _case("1b int8 prompt 77", "dense 1b", quant="int8", vocab=128256, prompts=1, tokens=77),
        # One user of the 8B model in the middle of a conversation: the benchmark's headline workload.
        _case("8b int4 decode x1", "dense 8b", vocab=128256, decode=1, context=2048),
        # A lightly loaded server: sixteen conversations of different lengths.
        _case("8b int4 decode x16", "dense 8b", decode=16, context=2048, ragged=0.5),
        # A full server: sixty-four conversations of about the same length.
        _case("8b int4 decode x64", "dense 8b", decode=64, context=2048, ragged=0.06),
        # The same server trading cache precision for room, its users sampling instead of taking the best token.
        _case("8b int4 fp8 cache x40", "dense 8b", kv="fp8_per_token_head", decode=40, context=1500, ragged=0.4,
              sampler="top_k_top_p"),
        # Continuous batching: a portion of a new prompt rides beside the decoding requests.
        _case("8b int4 decode x23 + 489", "dense 8b", decode=23, context=1200, ragged=0.4, prompts=1, tokens=489,
              history=512),
        # A long prompt in one full chunk.
        _case("8b int4 prompt 2048", "dense 8b", vocab=128256, prompts=1, tokens=2048),
        # The mixture under load: every expert has routes.
        _case("30b fp8 decode x64", "mixture 30b", quant="fp8", decode=64, context=1024, ragged=0.06),
        # Several prompts of odd lengths read together by the mixture.
        _case("30b fp8 prompts 3x500", "mixture 30b", quant="fp8", prompts=3, tokens=500, ragged=0.3),
        # The layer-stack models: a document read by latent attention and decaying memories.
        _case("stack bf16 prompt 2011", "stack 4096", quant="bf16", prompts=1, tokens=2011),
    ]


def draw(rng: random.Random):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "both", "stack"])
    if kind == "stack":   # (portions that take the attention's form for prompts)
        return _case(None, rng.choice(list(STACKS)), quant="bf16", prompts=1, tokens=log(256, 2048))
    model = rng.choice(["dense 8b", "dense 8b", "dense 1b", "mixture 30b"])
    quant = {"dense 8b": ["int4b8", "int4b8", "fp8", "int8"], "dense 1b": ["int8", "bf16", "int4b8"], "mixture 30b": ["fp8"]}[model]
    caches = ["auto"] if model == "dense 1b" else ["auto", "auto", "fp8_per_token_head", "int8_per_token_head"]
    c = dict(quant=rng.choice(quant), kv=rng.choice(caches),
             ragged=rng.choice([0.0, 0.06, rng.uniform(0.1, 0.8)]), sampler=rng.choice(["greedy", "greedy", "top_k_top_p", "min_p"]))
    if kind == "decode":
        c.update(decode=log(1, 64), context=log(16, 2048))
    elif kind == "prompt":
        c.update(tokens=log(16, 1900))
        c.update(prompts=rng.randint(1, max(1, min(8, 1900 // c["tokens"]))), history=rng.choice([0, 0, rng.randint(1, 1024)]))
    else:
        c.update(decode=log(1, 48), context=log(64, 1536), prompts=1, tokens=log(32, 1024), history=rng.choice([0, rng.randint(1, 1024)]))
    return _case(None, model, **c)


# ---- the batch of a case ------------------------------------------------------------------------------------------
def _batch(case, seed):
    """The prompt whose pages the contexts are copies of, and per request (context length, its tokens)."""
    rng = np.random.default_rng([int(seed) & 0x7FFFFFFF, 17])
    low = 1.0 - case["ragged"]

    def length(n):
        return max(1, int(round(n * rng.uniform(low, 1.0)))) if case["ragged"] else n

    lengths = [length(case["context"]) for _ in range(case["decode"])]
    if lengths:
        lengths[0] = case["context"]
    vocab = case["vocab"]
    requests = [(n, rng.integers(0, vocab, 1)) for n in lengths]
    for _ in range(case["prompts"]):
        requests.append((case["history"], rng.integers(0, vocab, length(case["tokens"]))))
    shared = rng.integers(0, vocab, max(n for n, _ in requests))
    return shared, requests


def _sampler(case, i, seed):
    if case["sampler"] == "top_k_top_p":
        return dict(kind=4, temperature=0.8, k=50, p=0.95, seed=1 + (seed * 7919 + i) % 1000003)
    if case["sampler"] == "min_p":
        return dict(kind=3, temperature=0.8, p=0.05, seed=1 + (seed * 7919 + i) % 1000003)
    return dict(kind=drv.SAMPLER_TOP_P, temperature=0.0, p=1.0)


def _model_seed(seed):
    return (int(seed) & 0x7FFFFFFF) * 2654435761 % (1 << 48) + 1


def _stack_config(case):
    z = STACKS[case["model"]]
    rot = dict(dims=z["rot_dim"], base=10000.0, scaling=dict(factor=4.0, original=4096, fast=24.0, slow=2.0))
    dense = dict(kind="dense", ff=z["ff"])
    latent = dict(type="latent_attention", mlp=dense,
                  mixer=dict(heads=z["heads"], dim=z["dim"], rot_dim=z["rot_dim"], vdim=z["vdim"], q_rank=z["q_rank"],
                             kv_rank=z["kv_rank"], rot=rot, scale=(z["dim"] + z["rot_dim"]) ** -0.5))
    delta = dict(type="channel_delta", mlp=dense,
                 mixer=dict(heads=z["heads"], kv_heads=z["heads"], dim=z["dim"], vdim=z["vdim"], conv=4))
    return dict(architecture="Varasun", layers=[delta if l % 3 == 2 else latent for l in range(STACK_LAYERS)], width=z["width"],
                vocab=case["vocab"], norm=dict(eps=1e-6), logit_scale=0.25, logit_softcap=30.0)


def _toml(case, seed, pages, directory):
    if case["model"] in STACKS:
        model = dict(hf_path=directory, random_weights=True, quant="bf16")
    else:
        model = dict(MODELS[case["model"]], vocab=case["vocab"], quant=case["quant"])
        if case["quant"] == "int4b8":
            model["group_size"] = 128
        elif case["quant"] != "bf16":
            model["scale_dtype"] = "bf16"
    model["seed"] = _model_seed(seed)
    text = {True: "true", False: "false"}
    lines = ["[model]"] + [f"{k} = " + (text[v] if isinstance(v, bool) else f'"{v}"' if isinstance(v, str) else str(v))
                           for k, v in model.items()]
    lines += ["[batching]", f"kv_page_size = {PAGE}", f"total_pages = {pages}", f"max_forward_tokens = {MAX_TOKENS}",
              f"max_forward_requests = {MAX_REQUESTS}", f'kv_cache_dtype = "{case["kv"]}"']
    return "\n".join(lines) + "\n"


class _Served:
    """A driver with the case's contexts in its cache, and the frame that continues them."""

    def __init__(self, case, seed):
        shared, requests = _batch(case, seed)
        pages_of = [-(-(n + len(toks)) // PAGE) for n, toks in requests]
        first = -(-len(shared) // PAGE)
        stack = case["model"] in STACKS
        directory = tempfile.mkdtemp(prefix="pie_cases_") if stack else ""
        try:
            if stack:
                with open(directory + "/config.json", "w") as f:
                    json.dump(_stack_config(case), f)
            self.driver = drv.Driver(_toml(case, seed, first + sum(pages_of) + 8, directory))
        finally:
            if stack:
                shutil.rmtree(directory, ignore_errors=True)
        for a in range(0, len(shared), MAX_TOKENS):
            b = min(a + MAX_TOKENS, len(shared))
            n = -(-b // PAGE)
            self._send(drv.ForwardFrame(shared[a:b], np.arange(a, b), np.arange(n), [0, n], [b - (n - 1) * PAGE], [0, b - a],
                                        rs_slot_ids=[0] if stack else None))
        srcs, dsts, tokens, positions, pages, indptr, last, qo = [], [], [], [], [], [0], [], [0]
        at = first
        for (n, toks), count in zip(requests, pages_of):
            held = -(-n // PAGE)
            srcs += range(held)
            dsts += range(at, at + held)
            tokens += toks.tolist()
            positions += range(n, n + len(toks))
            pages += range(at, at + count)
            indptr.append(len(pages))
            last.append(n + len(toks) - (count - 1) * PAGE)
            qo.append(len(tokens))
            at += count
        if srcs and self.driver.handle(drv.copy_frame(2, srcs, dsts)).payload.status.status != 0:
            raise RuntimeError("page copy failed")
        R = len(requests)
        self.frame = drv.ForwardFrame(
            tokens, positions, pages, indptr, last, qo, sampling_indices=[len(t) - 1 for _, t in requests],
            sampling_indptr=np.arange(R + 1), samplers=[_sampler(case, i, seed) for i in range(R)],
            sampler_indptr=np.arange(R + 1), rs_slot_ids=np.arange(R) if stack else None)
        self.requests = R
        self.logits_type = np.float32 if stack else np.uint16

    def _send(self, frame):
        res = self.driver.forward(frame)
        if res.num_requests != frame.frame.payload.forward.qo_indptr.len - 1:
            raise RuntimeError("forward failed: " + self.driver.last_error())

    def __del__(self):
        if getattr(self, "driver", None):
            self.driver.close()


def prepare(case, seed):
    return _Served(case, seed)


def run(state):
    res = state.driver.forward(state.frame)
    if res.num_requests != state.requests:
        raise RuntimeError("forward failed: " + state.driver.last_error())
    logits = state.driver.export_tensor("debug.logits", state.logits_type).reshape(state.requests, -1)
    if state.logits_type == np.float32:
        return {"logits": torch.from_numpy(logits)}
    return {"logits": torch.from_numpy(logits.view(np.int16)).view(torch.bfloat16)}


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def work(case):
    """Weights once (of a mixture, the experts that get routes), the cached keys and values once, the logits;
    multiplications and additions of the products and the attention."""
    low = 1.0 - case["ragged"] / 2
    decode = case["decode"]
    ctx = case["context"] * low if decode > 1 else case["context"]
    own = case["tokens"] * low
    rows = decode + case["prompts"] * own
    sampled = decode + case["prompts"]
    # (query, key) pairs and cached tokens read
    pairs = decode * ctx + case["prompts"] * own * (case["history"] + own / 2)
    cached = decode * ctx + case["prompts"] * (case["history"] + own)
    V = case["vocab"]
    if case["model"] in STACKS:
        z = STACKS[case["model"]]
        H, h, d, r, v = z["width"], z["heads"], z["dim"], z["rot_dim"], z["vdim"]
        delta = STACK_LAYERS // 3
        latent = STACK_LAYERS - delta
        w_latent = H * (z["q_rank"] + z["kv_rank"] + r) + z["q_rank"] * h * (d + r) + z["kv_rank"] * h * (d + v) + h * v * H
        w_delta = H * (2 * h * d + h * v + h + d + v) + h * d * d + h * v * v + h * v * H
        w = latent * w_latent + delta * w_delta + STACK_LAYERS * 2 * H * z["ff"]
        flops = 2 * rows * w + latent * 2 * pairs * h * (d + r + v) + delta * rows * h * 6 * d * v + 2 * sampled * V * H
        nbytes = 2 * w + 2 * V * H + latent * cached * (z["kv_rank"] + r) * 2 + sampled * V * 4
        return {"bytes": nbytes, "flops": flops}
    m = MODELS[case["model"]]
    H, L, hq, hk, d = (m[k] for k in ("hidden", "layers", "q_heads", "kv_heads", "head_dim"))
    size = {"int4b8": 0.5 + 2 / 128, "int8": 1.0, "fp8": 1.0, "bf16": 2.0}[case["quant"]]
    kv = {"auto": 2.0}.get(case["kv"], 1.0 + 4.0 / d)
    attn = H * (hq + 2 * hk) * d + hq * d * H
    if "num_experts" in m:
        E, k, ff = m["num_experts"], m["top_k"], m["expert_intermediate"]
        touched = E * (1.0 - (1.0 - k / E) ** rows)
        w_bytes = (attn + touched * 3 * H * ff) * size + E * H * 2
        w_flops = attn + k * 3 * H * ff + E * H
    else:
        w_bytes = (attn + 3 * H * m["intermediate"]) * size
        w_flops = attn + 3 * H * m["intermediate"]
    return {"bytes": L * (w_bytes + cached * 2 * hk * d * kv) + V * H * 2 + sampled * V * 2,
            "flops": L * (2 * rows * w_flops + 4 * pairs * hq * d) + 2 * sampled * V * H}


def tolerance(case):
    return TOLERANCES["stack" if case["model"] in STACKS else case["model"]]


# bf16 pipelines round their activations to 8 bits at every product.  Measured: 0.016 from the 64-bit values at these
# depths (0.0055 over the stacks' six layers), and 0.014 between two passes whose products sum in other orders.
TOLERANCES = {"dense 8b": {"rel": 0.03}, "dense 1b": {"rel": 0.03}, "mixture 30b": {"rel": 0.03}, "stack": {"rel": 0.02}}


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------
_MASK = (1 << 64) - 1


def _signed(x):
    x &= _MASK
    return x - (1 << 64) if x >> 63 else x


class _Weights:
    """The random weights a driver makes of a seed: a hash of the element's index, four 16-bit uniforms summed."""

    def __init__(self, seed):
        self.seed = seed

    def normal(self, shape, std, mean=0.0):
        """bf16 values; one draw of the driver's sequence of tensors."""
        self.seed = (self.seed + 0xA0761D6478BD642F) & _MASK
        n = math.prod(shape)
        out = torch.empty(n, dtype=torch.bfloat16, device="cuda")
        f32 = np.float32
        unit = float(f32(1.0) / f32(37837.227))
        for a in range(0, n, 1 << 27):
            b = min(n, a + (1 << 27))
            x = torch.arange(a, b, dtype=torch.int64, device="cuda").mul_(_signed(0xD1342543DE82EF95))
            x.bitwise_xor_(_signed(self.seed)).add_(_signed(0x9E3779B97F4A7C15))
            for shift, factor in ((30, 0xBF58476D1CE4E5B9), (27, 0x94D049BB133111EB), (31, 1)):
                t = x >> shift
                x.bitwise_xor_(t.bitwise_and_((1 << (64 - shift)) - 1))
                if factor != 1:
                    x.mul_(_signed(factor))
            total = x & 0xFFFF
            for shift in (16, 32, 48):
                total += (x >> shift) & 0xFFFF
            z = (total - 131070).to(torch.float32) * unit
            out[a:b] = (z * float(f32(std)) + float(f32(mean))).to(torch.bfloat16)
        return out.view(shape)

    def skip(self):
        self.seed = (self.seed + 0xA0761D6478BD642F) & _MASK


def _stored(w, quant):
    """[N, K] bf16 -> the values its storage format holds, in 64 bits."""
    if quant == "bf16":
        return w.double()
    x = w.float()
    if quant == "int4b8":
        x = x.view(x.shape[0], -1, 128)
        s = (x.abs().amax(-1, keepdim=True) / 7.0).to(torch.bfloat16).float()
        return (torch.round(x / s).clamp_(-8, 7).double() * s.double()).view(w.shape)
    top = x.abs().amax(-1, keepdim=True)
    most = 127.0 if quant == "int8" else 448.0
    codes = x * (most / top)
    codes = torch.round(codes).clamp_(-128, 127) if quant == "int8" else codes.clamp_(-448, 448).to(torch.float8_e4m3fn)
    return codes.double() * (top / most).to(torch.bfloat16).double()


def _norm(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * (1.0 if w is None else w.double())


def _silu(x):
    return x * torch.sigmoid(x)


def _attend(q, k, v, scale):
    """q [n, heads, d], k and v [m, kv heads, .]: query i sees the keys up to place m - n + i."""
    n, m = q.shape[0], k.shape[0]
    out = torch.empty(n, q.shape[1], v.shape[2], dtype=torch.float64, device="cuda")
    rep = q.shape[1] // k.shape[1]
    seen = torch.ones(n, m, dtype=torch.bool, device="cuda").tril_(m - n)
    for h in range(q.shape[1]):
        s = (q[:, h] @ k[:, h // rep].t() * scale).masked_fill_(~seen, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // rep]
    return out


def _all_rows(case, seed):
    """Tokens and places of the shared prompt's rows and then the requests', and the slice of each request."""
    shared, requests = _batch(case, seed)
    tokens, places, spans = [shared], [np.arange(len(shared))], []
    at = len(shared)
    for n, toks in requests:
        tokens.append(toks)
        places.append(np.arange(n, n + len(toks)))
        spans.append((n, at, at + len(toks)))
        at += len(toks)
    dev = lambda parts: torch.from_numpy(np.concatenate(parts).astype(np.int64)).cuda()  # noqa: E731
    return dev(tokens), dev(places).double(), len(shared), spans


def _over_contexts(q, k, v, shared, spans, scale):
    """Attention of all rows: the shared prompt's over itself, a request's over a copy of its head and its own rows."""
    out = [_attend(q[:shared], k[:shared], v[:shared], scale)] if shared else []
    for n, a, b in spans:
        out.append(_attend(q[a:b], torch.cat([k[:n], k[a:b]]), torch.cat([v[:n], v[a:b]]), scale))
    return torch.cat(out)


def _exact_uniform(case, seed):
    m = MODELS[case["model"]]
    H, L, hq, hk, d, V = m["hidden"], m["layers"], m["q_heads"], m["kv_heads"], m["head_dim"], case["vocab"]
    I, eps, quant = m.get("expert_intermediate") or m["intermediate"], 1e-5, case["quant"]
    W = _Weights(_model_seed(seed))
    tokens, places, shared, spans = _all_rows(case, seed)
    embed = W.normal((V, H), m.get("embed_std", 0.02))
    head = embed if m.get("tie_embeddings") else W.normal((V, H), 0.02)
    final = W.normal((H,), 0.1, 1.0)
    x = embed[tokens].double()
    freq = m["rope_theta"] ** (-2.0 * torch.arange(d // 2, dtype=torch.float64, device="cuda") / d)
    ang = places[:, None] * freq.float().double()
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rotate(t):
        a, b = t[..., :d // 2], t[..., d // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    for _ in range(L):
        n1, n2 = W.normal((H,), 0.1, 1.0), W.normal((H,), 0.1, 1.0)
        qk = [W.normal((d,), 0.1, 1.0) for _ in range(2)] if m["arch"] != "llama3" else None
        fused = _norm(x, n1, eps) @ _stored(W.normal(((hq + 2 * hk) * d, H), 0.02), quant).t()
        q, k, v = fused.view(-1, hq + 2 * hk, d).split([hq, hk, hk], 1)
        if qk:
            q, k = _norm(q, qk[0], eps), _norm(k, qk[1], eps)
        o = _over_contexts(rotate(q), rotate(k), v, shared, spans, d ** -0.5)
        x = x + o.flatten(1) @ _stored(W.normal((H, hq * d), 0.02), quant).t()
        h = _norm(x, n2, eps)
        if "num_experts" not in m:
            gate, up = (h @ _stored(W.normal((2 * I, H), 0.02), quant).t()).split(I, 1)
            x = x + (_silu(gate) * up) @ _stored(W.normal((H, I), 0.02), quant).t()
            continue
        E, top = m["num_experts"], m["top_k"]
        p, chosen = torch.softmax(h @ W.normal((E, H), m["router_std"]).double().t(), -1).topk(top, -1)
        p = p / p.sum(-1, keepdim=True)
        gu = W.normal((E * 2 * I, H), 0.02)
        down = W.normal((E * H, I), 0.02)
        y = torch.zeros_like(x)
        for e in range(E):
            row, place = (chosen == e).nonzero(as_tuple=True)
            if len(row):
                gate, up = (h[row] @ _stored(gu[e * 2 * I:(e + 1) * 2 * I], quant).t()).split(I, 1)
                y.index_add_(0, row, (_silu(gate) * up) @ _stored(down[e * H:(e + 1) * H], quant).t() * p[row, place, None])
        x = x + y
    last = torch.tensor([b - 1 for _, _, b in spans], device="cuda")
    return _norm(x[last], final, eps) @ head.double().t()


def _exact_stack(case, seed):
    cfg = _stack_config(case)
    H, V, eps = cfg["width"], cfg["vocab"], cfg["norm"]["eps"]
    W = _Weights(_model_seed(seed))
    tokens, places, shared, spans = _all_rows(case, seed)
    mat = lambda rows, cols, fan=None: W.normal((rows, cols), 0.7 / math.sqrt(fan or cols)).double()  # noqa: E731
    x = W.normal((V, H), 0.7)[tokens].double()
    head = W.normal((V, H), 0.7 / math.sqrt(H))
    T = len(tokens)
    for layer in cfg["layers"]:
        a = layer["mixer"]
        heads, dim, vdim = a["heads"], a["dim"], a["vdim"]
        if layer["type"] == "latent_attention":
            rd, qr, kr = a["rot_dim"], a["q_rank"], a["kv_rank"]
            fused = x @ mat(qr + kr + rd, H).t()
            q = (_norm(fused[:, :qr], None, eps) @ mat(heads * (dim + rd), qr).t()).view(T, heads, dim + rd)
            W.skip()   # (the two matrices of the form that decodes)
            W.skip()
            kv = (_norm(fused[:, qr:qr + kr], None, eps) @ mat(heads * (dim + vdim), kr).t()).view(T, heads, dim + vdim)
            rot = a["rot"]
            sc = rot["scaling"]
            i = torch.arange(rd // 2, dtype=torch.float64, device="cuda")
            f = rot["base"] ** (-2.0 * i / rd)
            turns = lambda t: rd * math.log(sc["original"] / (2 * math.pi * t)) / (2 * math.log(rot["base"]))  # noqa: E731
            lo, hi = max(math.floor(turns(sc["fast"])), 0), min(math.ceil(turns(sc["slow"])), rd - 1)
            ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
            ang = places[:, None] * (f / sc["factor"] * ramp + f * (1 - ramp))
            grow = 0.1 * math.log(sc["factor"]) + 1.0

            def rotate(t):
                c, s = (ang.cos() * grow)[:, None], (ang.sin() * grow)[:, None]
                u, v = t[..., 0::2], t[..., 1::2]
                return torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)

            key = torch.cat([kv[..., :dim], rotate(fused[:, None, qr + kr:]).expand(T, heads, rd)], -1)
            query = torch.cat([q[..., :dim], rotate(q[..., dim:])], -1)
            o = _over_contexts(query, key, kv[..., dim:], shared, spans, a["scale"])
        else:
            kd, vd = heads * dim, heads * vdim
            fused = x @ mat(2 * kd + vd + heads + dim + vdim, H).t()
            conv, step, low, gate = fused.split([2 * kd + vd, heads, dim, vdim], 1)
            before = torch.cat([torch.zeros(a["conv"] - 1, conv.shape[1], dtype=torch.float64, device="cuda"), conv])
            conv = _silu(sum(before[j:j + T] * 0.5 for j in range(a["conv"])))
            unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
            q = unit(conv[:, :kd].reshape(T, heads, dim)) * dim ** -0.5
            k = unit(conv[:, kd:2 * kd].reshape(T, heads, dim))
            v, beta = conv[:, 2 * kd:].reshape(T, heads, vdim), torch.sigmoid(step)
            rate = 1.0 + torch.arange(heads, dtype=torch.float64, device="cuda") % 8
            raw = torch.nn.functional.softplus((low @ mat(kd, dim).t() - 3.0)).view(T, heads, dim)
            decay = torch.exp(-rate[:, None] * raw)
            gate = torch.sigmoid(gate @ mat(vd, vdim).t()).view(T, heads, vdim)
            S = torch.zeros(heads, dim, vdim, dtype=torch.float64, device="cuda")
            o = torch.empty(T, heads, vdim, dtype=torch.float64, device="cuda")
            for t in range(T):
                S = S * decay[t][:, :, None]
                u = beta[t][:, None] * (v[t] - (k[t][:, None] @ S)[:, 0])
                S = torch.baddbmm(S, k[t][:, :, None], u[:, None, :])
                o[t] = (q[t][:, None] @ S)[:, 0]
            o = _norm(o, None, eps) * gate
        x = x + _norm(o.flatten(1) @ mat(H, heads * vdim).t(), None, eps)
        h = torch.relu(x @ mat(layer["mlp"]["ff"], H).t()).square()
        x = x + _norm(h @ mat(H, layer["mlp"]["ff"]).t(), None, eps)
    last = torch.tensor([b - 1 for _, _, b in spans], device="cuda")
    y = _norm(x[last], None, eps) @ head.double().t() * cfg["logit_scale"]
    return cfg["logit_softcap"] * torch.tanh(y / cfg["logit_softcap"])


def exact(case, seed):
    torch.set_grad_enabled(False)
    return {"logits": _exact_stack(case, seed) if case["model"] in STACKS else _exact_uniform(case, seed)}
