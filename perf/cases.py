"""The work that is timed: steps of the engine as a serving program makes them, and what they return.

A case is one pass through the public entry points, for one of the seven designs at the sizes of a preset:

* ``decode``: one step of ``decode`` requests that each bring one token on a context of about ``context`` tokens, and
  beside them, if ``prompts`` is not 0, a prompt portion (a step of continuous serving).
* ``prompt``: one step of ``prompts`` prompt portions of about ``tokens`` tokens each behind ``prefix`` cached ones.
  Without a prefix a request is admitted, its prompt computed and the request let go, as for a short answer.
* ``sample``: the tokens of a step from its logits, with the options mixed as users mix them.

Lengths are ``ragged`` (spread over a quarter to seven quarters of the mean) or all alike.  Weights are random and drawn
on the GPU: unit-variance embeddings, matrices that keep a row's size, and a sublayer adds a small part of the residual
stream, as in a trained model; so a token whose router scores tie moves its logits by a few per cent at most.
"""
import math

import numpy as np
import torch

from pico_vllm_amd import EngineArgs
from pico_vllm_amd.config.presets import preset
from pico_vllm_amd.config.registry import resolve_architecture
from pico_vllm_amd.engine.batch import SeqStep
from pico_vllm_amd.engine.llm import LLMEngine
from pico_vllm_amd.parts.model import DecoderModel, model_param_specs
from pico_vllm_amd.sampling.sampler import Sampler

DEV = "cuda:0"
PAGE = 16
BUDGET = 2048                 # tokens of a step, the engine's default
DESIGNS = ("qwen2", "lerazen", "nasedra", "dikolix", "vagelix", "begasun", "tubusun")
ROUTED = ("lerazen", "nasedra", "dikolix", "tubusun")
VOCAB = 151936


def step_case(kind, design, size, layers, decode=0, context=0, prompts=0, tokens=0, prefix=0, ragged=False, dtype="bfloat16"):
    return {"kind": kind, "design": design, "size": size, "layers": layers, "dtype": dtype, "decode": decode, "context": context,
            "prompts": prompts, "tokens": tokens, "prefix": prefix, "ragged": ragged}


def listed():
    def named(name, case):
        return dict(case, name=name)
    return [
        # the end of every step with users' own sampling options: a batch of eight, a quarter of it greedy
        named("sample 8 rows", {"kind": "sample", "rows": 8, "vocab": VOCAB}),
        # one user's chat, in the middle of an answer: latency
        named("qwen2 1.5b decode 1", step_case("decode", "qwen2", "1.5b", 28, decode=1, context=600)),
        # the benchmark's headline: a batch of eight at long contexts
        named("qwen2 1.5b decode 8", step_case("decode", "qwen2", "1.5b", 28, decode=8, context=4000)),
        # a busy server's step: requests of all ages decode while a prompt comes in
        named("qwen2 7b serve 40+700", step_case("decode", "qwen2", "7b", 8, decode=40, context=900, prompts=1, tokens=700, prefix=1024, ragged=True)),
        # the benchmark's prompt
        named("qwen2 1.5b prompt 2048", step_case("prompt", "qwen2", "1.5b", 28, prompts=1, tokens=2048)),
        # 32-bit: what logits are compared with when a conversion is checked
        named("qwen2 1.5b f32 prompt 300", step_case("prompt", "qwen2", "1.5b", 4, prompts=1, tokens=300, dtype="float32")),
        # a batch of decoding requests over routed feed-forwards: most experts are read
        named("lerazen 7b decode 32", step_case("decode", "lerazen", "7b", 4, decode=32, context=1000, ragged=True)),
        # a whole budget of one prompt: capped, gated attention, a recurrent layer, experts
        named("nasedra 1.5b prompt 2048", step_case("prompt", "nasedra", "1.5b", 4, prompts=1, tokens=2048)),
        # a prompt of no particular length: latent attention, state space, retention, experts
        named("dikolix 1.5b prompt 1377", step_case("prompt", "dikolix", "1.5b", 6, prompts=1, tokens=1377)),
        # several prompts of different lengths arrive together
        named("vagelix 1.5b 3 prompts", step_case("prompt", "vagelix", "1.5b", 6, prompts=3, tokens=620, ragged=True)),
        # a later portion of a long prompt
        named("begasun 1.5b portion", step_case("prompt", "begasun", "1.5b", 6, prompts=1, tokens=2048, prefix=4096)),
        # a small batch of a large routed model
        named("tubusun 7b decode 8", step_case("decode", "tubusun", "7b", 4, decode=8, context=3000, ragged=True)),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    pick = rng.random()
    if pick < 0.08:
        return {"kind": "sample", "rows": spread(1, 64), "vocab": rng.choice((VOCAB, 152064))}
    if pick < 0.14:
        return step_case("prompt", "qwen2", "1.5b", 4, prompts=1, tokens=spread(9, 400), dtype="float32")
    design = rng.choice(DESIGNS)
    size = rng.choice(("1.5b", "7b"))
    layers = (28 if size == "1.5b" else 8) if design == "qwen2" else 4 if design in ("lerazen", "nasedra", "tubusun") else 6
    if pick < 0.57:
        decode = spread(1, 64)
        context = spread(32, min(4000, 36000 // decode))
        case = step_case("decode", design, size, layers, decode=decode, context=context, ragged=rng.random() < 0.6)
        if rng.random() < 0.25:
            case.update(prompts=1, tokens=spread(16, 1000))
        return case
    prompts = rng.choice((1, 1, 1, 2, 3, 5))
    tokens = spread(17, (2048 if size == "1.5b" else 900) // prompts)
    return step_case("prompt", design, size, layers, prompts=prompts, tokens=tokens, prefix=rng.choice((0, 0, spread(64, 9000 // prompts))),
                     ragged=prompts > 1 and rng.random() < 0.7)


# ---- sizes of a case ---------------------------------------------------------------------------------------------------
def lengths(mean, n, ragged):
    """``n`` lengths around ``mean``, the same for every seed."""
    if not ragged:
        return [mean] * n
    golden = 0.6180339887498949
    return [max(2, int(mean * (0.25 + 1.5 * ((i + 1) * golden % 1.0)))) for i in range(n)]


def sequences(case):
    """(cached tokens, new tokens) of every sequence of the step, single tokens first."""
    single = [(c, 1) for c in lengths(case["context"], case["decode"], case["ragged"])]
    tokens = lengths(case["tokens"], case["prompts"], case["ragged"] and case["prompts"] > 1)
    return single + [(case["prefix"], n) for n in tokens]


def config(case):
    name = case["size"] if case["design"] == "qwen2" else f"{case['design']}-{case['size']}"
    raw = preset(name)
    if "layers" in raw:
        raw["layers"] = raw["layers"][:case["layers"]]
    else:
        raw["num_hidden_layers"] = case["layers"]
    return raw


def described(case):
    arch = resolve_architecture(config(case))
    typed = arch.config_from_dict(config(case))
    return typed, arch.build_spec(typed)


def dtype_of(case):
    return torch.float32 if case["dtype"] == "float32" else torch.bfloat16


# ---- weights -----------------------------------------------------------------------------------------------------------
def weights(case, seed):
    """Random tensors by checkpoint name, in the types a checkpoint of this engine dtype holds."""
    _, spec = described(case)
    raw, dtype = config(case), dtype_of(case)
    g = torch.Generator(device=DEV).manual_seed(seed * 7919 + 17)
    back = 0.5 * (2 * case["layers"]) ** -0.5          # what a sublayer adds, as a part of the stream
    scale = (raw.get("embedding") or {}).get("scale", 1.0)
    normed = {"vagelix": ("norm1", "norm2"), "tubusun": ("norm1b", "norm2b"), "begasun": ("ls1", "ls2")}.get(case["design"], ())
    out = {}
    for p in model_param_specs(spec):
        last = p.name.split(".")[-1]
        owner = p.name.split(".")[-2] if last in ("weight", "bias", "b") and "." in p.name else last

        def normal(std, mean=0.0, kind=torch.float32):
            return torch.empty(p.shape, device=DEV, dtype=kind).normal_(mean, std, generator=g)

        def uniform(lo, hi):
            return torch.empty(p.shape, device=DEV).uniform_(lo, hi, generator=g)
        if p.role == "norm":
            t = uniform(0.9, 1.1) * (back if last in normed and p.name.startswith("l") or p.name.endswith("side.norm") else 1.0)
            t = t.to(dtype).float()
        elif p.role == "bias":
            mean, std = {"vmix": (0.5, 0.1), "correction": (0.0, 0.05)}.get(last, (1.0, 2.0) if p.name.endswith("a2.b") else (0.0, 0.1))
            t = normal(std, mean).to(dtype)
        elif p.role == "f32":
            if p.name.endswith("dt.b") or last == "dt_bias":
                t = torch.log(torch.expm1(uniform(0.01, 0.21)))
            elif last == "A_log":
                t = torch.log(uniform(0.5, 4.5))
            elif last in ("D", "lam", "sink"):
                t = normal(0.3, 1.0 if last != "sink" else 0.0)
            else:
                t = normal(0.5 if last == "conv" else 0.1)
        else:
            std = p.shape[-1] ** -0.5
            if owner in ("embed", "embed_tokens", "pos", "bigram") or p.name == "side.embed":
                std = {"pos": 0.3, "bigram": 0.3}.get(owner, 1.0 / scale if owner != "side" and p.name != "side.embed" else 1.0)
            elif owner in ("o", "down", "o_proj", "down_proj"):
                std *= 1.0 if normed else back
            elif owner in ("q", "k", "q_proj", "k_proj", "uq", "uk"):
                std *= 1.4
            elif owner in ("router", "a2"):
                std *= 2.0
            t = normal(std, kind=dtype)
        out[p.name] = t
    return out


# ---- a pass ------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "sample":
        g = torch.Generator(device=DEV).manual_seed(seed)
        rows = case["rows"]
        logits = torch.randn(rows, case["vocab"], device=DEV, generator=g) * 2.5
        mixed = [(0.0, 1.0), (0.7, 0.9), (1.0, 1.0), (0.8, 0.95)]
        return {"sampler": Sampler(torch.device(DEV), rows), "logits": logits,
                "options": ([mixed[i % 4][0] for i in range(rows)], [mixed[i % 4][1] for i in range(rows)],
                            [seed * 1000003 + i for i in range(rows)], [40 + i for i in range(rows)])}
    typed, spec = described(case)
    model = DecoderModel(spec, dtype_of(case), torch.device(DEV))
    model.load(weights(case, seed))
    model.config = typed
    seqs = sequences(case)
    engine = LLMEngine(EngineArgs(dtype=case["dtype"], block_size=PAGE, num_gpu_blocks=sum(-(-(c + n) // PAGE) for c, n in seqs) + 8,
                                  max_seq_len=max(c + n for c, n in seqs) + PAGE, max_num_seqs=len(seqs),
                                  max_num_batched_tokens=max(BUDGET, sum(n for _, n in seqs)), use_cuda_graph=True, max_batch_size=64),
                       model=model)
    ids = token_ids(case, seed)
    steps = [SeqStep(f"r{i}", t[c:], [n - 1]) for i, ((c, n), t) in enumerate(zip(seqs, ids))]
    cached = [i for i, (c, _) in enumerate(seqs) if c]
    fill(engine.runner, [(steps[i].req, ids[i][:seqs[i][0]], sum(seqs[i])) for i in cached])
    new = [(steps[i].req, n) for i, (c, n) in enumerate(seqs) if not c]
    return {"engine": engine, "steps": steps, "new": new, "pages": case["kind"] == "prompt"}


def token_ids(case, seed):
    rng = np.random.default_rng(seed)
    vocab = described(case)[1].vocab_size
    return [rng.integers(0, vocab, c + n).tolist() for c, n in sequences(case)]


def fill(runner, requests):
    """Compute the contexts: (request, its tokens, the length it may reach), a step's budget of tokens at a time."""
    m = runner.manager
    for rid, tokens, most in requests:
        if not (m.add_request(rid) and m.grow(rid, most)):
            raise RuntimeError("the cache is too small for the case")
    left = [[rid, tokens] for rid, tokens, _ in requests]
    while left:
        room, step = BUDGET, []
        for entry in left[:]:
            part = entry[1][:room]
            if not part:
                break
            step.append(SeqStep(entry[0], part))
            entry[1] = entry[1][len(part):]
            room -= len(part)
            if not entry[1]:
                left.remove(entry)
        runner.step(step)
        runner.advance(step)


def run(state):
    if "sampler" in state:
        return np.array(state["sampler"].sample(state["logits"], *state["options"]), dtype=np.int64)
    runner = state["engine"].runner
    m = runner.manager
    for rid, n in state["new"]:
        if not (m.add_request(rid) and m.grow(rid, n)):
            raise RuntimeError("the cache is too small for the case")
    logits = runner.step(state["steps"])
    for rid, _ in state["new"]:
        m.free_request(rid)
    return {"logits": logits, "cache": cache_tensors(runner, state["pages"])}


def cache_tensors(runner, pages):
    """What the step leaves for the next one: the recurrent states, and after prompts the pages (the keys and values of
    a single token are read back by the step's own attention)."""
    out = {}
    for i in runner.model.cache_specs():
        layer = runner.storage.layer(i)
        if hasattr(layer, "state"):
            out[f"{i} state"] = layer.state[:runner.manager.slots.num_slots]       # (the last slot is padding's)
        elif layer is not None and pages:
            out.update({f"{i} {name}": t for name, t in layer.tensors.items()})
    return out


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------
def mixers(raw):
    """(kind, sizes) of every mixer: ("attention", heads, key size, value size, cached numbers a token, window or 0, chunk
    or 0, whether it stores) or ("state", numbers of state, multiplications a token)."""
    out = []
    if "layers" not in raw:
        d = raw["hidden_size"] // raw["num_attention_heads"]
        return [("attention", raw["num_attention_heads"], d, d, 2 * raw["num_key_value_heads"] * d, 0, 0)] * raw["num_hidden_layers"]
    for layer in raw["layers"]:
        m, kind = layer["mixer"], layer["type"]
        for name, part in (("left", m["left"]), ("right", m["right"])) if kind == "parallel" else ((kind, m),):
            mask = part.get("mask") or {}
            if name == "latent_attention":
                r = part["kv_rank"] + part["rot_dim"]
                out.append(("attention", part["heads"], part["dim"] + part["rot_dim"], part["vdim"], r, 0, 0))
            elif name in ("attention", "left"):
                maps = 2 if "diff" in part else 1
                chunk = mask.get("size", 0) if "chunk" in str(raw["architecture"]).lower() or raw["architecture"] == "Vagelix" else 0
                out.append(("attention", maps * part["heads"], part["dim"], part["vdim"],
                            part["kv_heads"] * (maps * part["dim"] + part["vdim"]), 0 if chunk else mask.get("size", 0), chunk))
            elif name == "mamba1":
                out.append(("state", part["inner"] * part["state"], 5 * part["inner"] * part["state"]))
            elif name == "rglru":
                out.append(("state", part["width"], 8 * part["width"]))
            else:
                n = part["heads"] * part.get("dim", part.get("state")) * part["vdim"]
                out.append(("state", n, 5 * n))
    return out


def work(case):
    if case["kind"] == "sample":
        n = case["rows"] * case["vocab"]
        return {"bytes": 4.0 * n, "flops": 4.0 * n}
    raw, (_, spec), seqs = config(case), described(case), sequences(case)
    size = 4 if case["dtype"] == "float32" else 2
    T, R, V = sum(n for _, n in seqs), len(seqs), spec.vocab_size
    tables = ("embed", "model.embed_tokens.weight", "pos", "bigram", "side.embed")
    heads = [p for p in model_param_specs(spec) if p.name in ("head", "lm_head.weight")]
    width = spec.hidden_size
    nbytes, flops = R * V * 4.0 + V * width * size + (T * width * size if heads else 0), 2.0 * R * V * width
    for p in model_param_specs(spec):
        if p.name in tables or p in heads:
            continue
        n = float(np.prod(p.shape)) if p.shape else 1.0
        share = used = 1.0
        if ".mlp.e" in p.name:
            router = raw["layers"][int(p.name.split(".")[0][1:])]["mlp"]["router"]
            used = router["top"] / router["experts"]                       # a token's share of the experts
            share = 1.0 - (1.0 - used) ** T                                # the experts that any of T tokens takes
        nbytes += n * share * (4 if p.role in ("f32", "norm") else size)
        flops += 2.0 * n * T * used if len(p.shape) > 1 else 0.0
    for m in mixers(raw):
        if m[0] == "state":
            nbytes += 8.0 * m[1] * len(seqs)
            flops += m[2] * T
            continue
        _, H, dk, dv, row, window, chunk = m
        for cached, n in seqs:
            total = cached + n
            first = 0 if not (window or chunk) else max(0, cached - window + 1) if window else cached // chunk * chunk
            nbytes += row * size * (total - first + n)
            at = np.arange(cached, total, dtype=np.float64)
            seen = at + 1 if not (window or chunk) else np.minimum(at + 1, window) if window else at % chunk + 1
            flops += 2.0 * H * (dk + dv) * float(seen.sum())
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """What rounding alone does: about four times what the outputs of a step differ by when its products run in another
    order (0.002 to 0.004 in bfloat16, 3e-7 in 32 bits)."""
    if case["kind"] == "sample":
        return "exact"
    if case["dtype"] == "float32":
        return {"rel": 5e-6}
    # a token whose router scores are nearly equal goes to either expert, which moves its row by a few per cent
    return {"rel": 0.03 if case["design"] in ROUTED else 0.015, "max": 0.9 if case["design"] in ROUTED else 0.4}


# ---- the same in 64 bits -------------------------------------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] == "sample":
        return None
    seqs, raw = sequences(case), config(case)
    tokens = sum(c + n for c, n in seqs)
    cost = work(dict(case, decode=0, context=0, prompts=1, tokens=tokens, prefix=0, ragged=False))["flops"] / 30e12
    cost += tokens * 1.5e-4 * sum(m[0] == "state" for m in mixers(raw))
    if cost > 15:
        return None
    w = Weights(weights(case, seed))
    model = Plain(raw, w)
    rows = torch.stack([model.last_logits(t) for t in token_ids(case, seed)])
    # pages have no value of their own here: what the step reads from them is in the logits
    return {"logits": rows, "cache": {}}


class Weights:
    """Tensors by name in 64 bits, made when asked for; ``under`` a prefix."""

    def __init__(self, tensors, prefix=""):
        self.tensors, self.prefix = tensors, prefix

    def __getitem__(self, name):
        return self.tensors[self.prefix + name].double()

    def __contains__(self, name):
        return self.prefix + name in self.tensors

    def rows(self, name, ids):
        return self.tensors[self.prefix + name][ids].double()

    def under(self, prefix):
        return Weights(self.tensors, self.prefix + prefix + ".")


def rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def layer_norm(x, w, b, eps):
    x = x - x.mean(-1, keepdim=True)
    return rms(x, eps) * w + b


def silu(x):
    return x * torch.sigmoid(x)


def gelu_tanh(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def softplus(x):
    return torch.logaddexp(x, torch.zeros_like(x))


def frequencies(rot):
    dims, base = rot["dims"], float(rot["base"])
    f = torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=torch.float64, device=DEV)
    s = rot.get("scaling")
    if not s:
        return f, 1.0

    def pair(turns):
        return dims * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(pair(s["fast"])), 0), min(math.ceil(pair(s["slow"])), dims - 1)
    ramp = ((torch.arange(dims // 2, device=DEV) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / s["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(s["factor"]) + 1.0


def rotate(x, rot, neighbours):
    """x [n, heads, d]: the first ``dims`` entries turned; entry 2i with 2i + 1 (``neighbours``) or i with i + dims / 2."""
    if not rot:
        return x
    dims = rot["dims"]
    f, mag = frequencies(rot)
    a = torch.arange(x.shape[0], device=DEV, dtype=torch.float64)[:, None, None] * f
    c, s = torch.cos(a) * mag, torch.sin(a) * mag
    u, v = (x[..., 0:dims:2], x[..., 1:dims:2]) if neighbours else (x[..., :dims // 2], x[..., dims // 2:dims])
    p, q = u * c - v * s, v * c + u * s
    turned = torch.stack([p, q], -1).flatten(-2) if neighbours else torch.cat([p, q], -1)
    return torch.cat([turned, x[..., dims:]], -1)


def seen_keys(n, window=0, keep=0, chunk=0):
    i, j = torch.arange(n, device=DEV)[:, None], torch.arange(n, device=DEV)[None, :]
    ok = j <= i
    if window:
        ok &= (i - j < window) | (j < keep)
    if chunk:
        ok &= i // chunk == j // chunk
    return ok


def attend(q, k, v, scale, seen, cap=None, slopes=None, sink=None):
    """q [n, H, d], k [n, G, d], v [n, G, dv] -> [n, H, dv]; ``sink``: a score a head that takes weight and has no value."""
    n, H = q.shape[:2]
    share = H // k.shape[1]
    out = []
    for h in range(H):
        s = q[:, h] @ k[:, h // share].T * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        if slopes is not None:
            at = torch.arange(n, device=DEV, dtype=s.dtype)
            s = s - slopes[h] * (at[:, None] - at[None, :])
        s = s.masked_fill(~seen, float("-inf"))
        top = s.max(-1, keepdim=True).values
        if sink is not None:
            top = torch.clamp(top, min=float(sink[h]))
        e = torch.exp(s - top)
        total = e.sum(-1, keepdim=True) + (torch.exp(float(sink[h]) - top) if sink is not None else 0.0)
        out.append((e / total) @ v[:, h // share])
    return torch.stack(out, 1)


def walk(q, k, v, decay, beta=None):
    """S <- decay S (+ k v^T, or with ``beta`` the delta rule's correction), o = S^T q; q, k [n, H, d], v [n, H, dv], decay
    [n, H, d] or [n, H, 1]."""
    S = torch.zeros(k.shape[1], k.shape[2], v.shape[2], dtype=v.dtype, device=DEV)
    out = []
    for t in range(k.shape[0]):
        S = S * decay[t].unsqueeze(-1)
        u = v[t] if beta is None else beta[t].unsqueeze(-1) * (v[t] - (S * k[t].unsqueeze(-1)).sum(1))
        S = S + k[t].unsqueeze(-1) * u.unsqueeze(1)
        out.append((S * q[t].unsqueeze(-1)).sum(1))
    return torch.stack(out)


def short_conv(x, taps, bias=None):
    n, K = x.shape[0], taps.shape[1]
    past = torch.cat([torch.zeros(K - 1, x.shape[1], dtype=x.dtype, device=DEV), x])
    y = sum(past[j:j + n] * taps[:, j] for j in range(K))
    return y if bias is None else y + bias


def spread_heads(x, heads):
    return x.repeat_interleave(heads // x.shape[1], 1)


def through_experts(h, chosen, weight, experts, one):
    out = torch.zeros_like(h)
    for e in range(experts):
        rows, slot = (chosen == e).nonzero(as_tuple=True)
        if len(rows):
            out.index_add_(0, rows, one(e, h[rows], weight[rows, slot].unsqueeze(-1)))
    return out


class Plain:
    """The designs' equations on a whole sequence; ``last_logits``: the logits behind its last token."""

    def __init__(self, raw, w):
        self.raw, self.w = raw, w
        self.design = raw.get("architecture", "Qwen2")
        self.eps = raw["rms_norm_eps"] if self.design == "Qwen2" else raw["norm"]["eps"]

    def last_logits(self, tokens):
        return getattr(self, self.design.lower())(tokens)

    def gated(self, h, w, prefix=""):
        return (silu(h @ w[prefix + "gate"].T) * (h @ w[prefix + "up"].T)) @ w[prefix + "down"].T

    def clipped(self, h, w, limit, prefix=""):
        g = torch.clamp(h @ w[prefix + "gate"].T, max=limit)
        u = torch.clamp(h @ w[prefix + "up"].T, -limit, limit)
        return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ w[prefix + "down"].T

    def qkv(self, h, w, m, biases=""):
        n = h.shape[0]
        q, k, v = (h @ w[x].T + (w[x + ".b"] if x in biases else 0.0) for x in "qkv")
        return q.view(n, m["heads"], -1), k.view(n, m.get("kv_heads", m["heads"]), -1), v.view(n, m.get("kv_heads", m["heads"]), -1)

    def qwen2(self, tokens):
        w, r, n = self.w, self.raw, len(tokens)
        H, G = r["num_attention_heads"], r["num_key_value_heads"]
        d = r["hidden_size"] // H
        rot = {"dims": d, "base": r["rope_theta"]}
        x = w.rows("model.embed_tokens.weight", tokens)
        seen = seen_keys(n)
        for i in range(r["num_hidden_layers"]):
            l = w.under(f"model.layers.{i}")
            h = rms(x, self.eps) * l["input_layernorm.weight"]
            a = l.under("self_attn")
            q, k, v = (h @ a[f"{c}_proj.weight"].T + a[f"{c}_proj.bias"] for c in "qkv")
            o = attend(rotate(q.view(n, H, d), rot, False), rotate(k.view(n, G, d), rot, False), v.view(n, G, d), d ** -0.5, seen)
            x = x + o.reshape(n, -1) @ a["o_proj.weight"].T
            h = rms(x, self.eps) * l["post_attention_layernorm.weight"]
            f = l.under("mlp")
            x = x + (silu(h @ f["gate_proj.weight"].T) * (h @ f["up_proj.weight"].T)) @ f["down_proj.weight"].T
        head = "model.embed_tokens.weight" if r["tie_word_embeddings"] else "lm_head.weight"
        return w[head] @ (rms(x[-1], self.eps) * w["model.norm.weight"])

    def lerazen(self, tokens):
        w, n = self.w, len(tokens)
        x = w.rows("embed", tokens) + w.rows("pos", torch.arange(n, device=DEV))
        first = None
        for i, layer in enumerate(self.raw["layers"]):
            l, m, f = w.under(f"l{i}"), layer["mixer"], layer["mlp"]
            h = rms(x, self.eps) * l["norm1"]
            a = l.under("mix")
            q, k, v = self.qkv(h, a, m, "qkv")
            t = torch.tensor([1 + m["q_temp"]["coef"] * math.log((p + 1) // m["q_temp"]["every"] + 1) for p in range(n)], device=DEV)
            if first is None:
                first = v
            else:
                lam = a["vmix"]
                v = (1 - lam) * v + lam * first
            slopes = [2.0 ** (-8.0 * (j + 1) / m["heads"]) for j in range(m["heads"])]
            o = attend(q * t.double()[:, None, None], k, v, m["scale"], seen_keys(n, (m.get("mask") or {}).get("size", 0)), slopes=slopes)
            delta = o.reshape(n, -1) @ a["o"].T + a["o.b"]
            e = l.under("mlp")
            if f["kind"] == "dense":
                delta = delta + torch.relu(h @ e["up"].T) ** 2 @ e["down"].T
            else:
                s, chosen = torch.topk(torch.sigmoid(h @ e["router"].T), f["router"]["top"], -1)
                delta = delta + through_experts(h, chosen, s, f["router"]["experts"],
                                                lambda j, rows, wt: self.clipped(wt * rows, e, f["expert"]["limit"], f"e{j}."))
            x = x + delta
        return w["head"] @ (rms(x[-1], self.eps) * w["final.norm"])

    def nasedra(self, tokens):
        w, n = self.w, len(tokens)
        x = w.rows("embed", tokens) * self.raw["embedding"]["scale"]
        kept = {}
        for i, layer in enumerate(self.raw["layers"]):
            l, m, f = w.under(f"l{i}"), layer["mixer"], layer["mlp"]
            h, h2 = rms(x, self.eps) * l["norm1"], rms(x, self.eps) * l["norm2"]
            a, e = l.under("mix"), l.under("mlp")
            if layer["type"] == "attention":
                q = rotate((h @ a["q"].T).view(n, m["heads"], -1), m["rot"], True)
                if "kv_from" not in m:
                    kept[i] = (rotate((h @ a["k"].T).view(n, m["kv_heads"], -1), m["rot"], True), (h @ a["v"].T).view(n, m["kv_heads"], -1))
                k, v = kept[m.get("kv_from", i)]
                o = attend(q, k, v, m["scale"], seen_keys(n, m["mask"]["size"], m["mask"]["keep_first"]), cap=m["softcap"])
                o = o.reshape(n, -1) * torch.sigmoid(h @ a["g"].T)
            else:
                q, k, v = self.qkv(h, a, m)
                decay = torch.sigmoid((h @ a["a1"].T) @ a["a2"].T + a["a2.b"]).pow(1.0 / m["tau"]).view(n, m["heads"], -1)
                o = rms(walk(q * m["dim"] ** -0.5, k, v, decay), self.eps) * a["norm"]
                o = o.reshape(n, -1) * silu(h @ a["g"].T)
            delta = o @ a["o"].T
            if f["kind"] == "dense":
                delta = delta + self.gated(h2, e)
            else:
                r = f["router"]
                s = torch.softmax(h2 @ e["router"].T, -1)
                chosen = torch.topk(s + e["correction"], r["top"], -1).indices
                wt = torch.gather(s, 1, chosen)
                wt = wt / (wt.sum(-1, keepdim=True) + 1e-20) * r["scale"]
                delta = delta + through_experts(h2, chosen, wt, r["experts"] + r["identity"],
                                                lambda j, rows, c: c * (self.gated(rows, e, f"e{j}.") if j < r["experts"] else rows))
                delta = delta + self.gated(h2, e, "shared.")
            x = x + delta
        return w["head"] @ (rms(x[-1], self.eps) * w["final.norm"])

    def latent(self, h, a, m, q):
        """q [n, H, d + r], plain keys and values of every head made from the latent."""
        n, d, r = h.shape[0], m["dim"], m["rot_dim"]
        rot = dict(m["rot"], dims=r)
        kv = h @ a["dkv"].T
        c = rms(kv[:, :m["kv_rank"]], self.eps) * a["dkv.norm"]
        kr = rotate(kv[:, None, m["kv_rank"]:], rot, True).expand(n, m["heads"], r)
        k = torch.cat([(c @ a["uk"].T).view(n, m["heads"], d), kr], -1)
        q = torch.cat([q[..., :d], rotate(q[..., d:], rot, True)], -1)
        return attend(q, k, (c @ a["uv"].T).view(n, m["heads"], -1), m["scale"], seen_keys(n))

    def dikolix(self, tokens):
        w, n, big = self.w, len(tokens), self.raw["embedding"]["bigram"]
        pairs = [big["buckets"]] + [(p * big["mul_prev"] + t * big["mul_cur"]) % big["buckets"] for p, t in zip(tokens, tokens[1:])]
        x = w.rows("embed", tokens) + w.rows("bigram", pairs)
        for i, layer in enumerate(self.raw["layers"]):
            l, m, f = w.under(f"l{i}"), layer["mixer"], layer["mlp"]
            a, e = l.under("mix"), l.under("mlp")
            h = layer_norm(x, l["norm1"], l["norm1.b"], self.eps)
            if layer["type"] == "latent_attention":
                cq = rms(h @ a["dq"].T, self.eps) * a["dq.norm"]
                o = self.latent(h, a, m, (cq @ a["uq"].T).view(n, m["heads"], -1)).reshape(n, -1)
            elif layer["type"] == "mamba1":
                I, N, R = m["inner"], m["state"], m["dt_rank"]
                y = h @ a["in"].T
                u = silu(short_conv(y[:, :I], a["conv"], a["conv.b"]))
                z = u @ a["x"].T
                dt = softplus(z[:, :R] @ a["dt"].T + a["dt.b"])
                A, B, C = -torch.exp(a["A_log"]), z[:, R:R + N], z[:, R + N:]
                S, out = torch.zeros(I, N, dtype=x.dtype, device=DEV), []
                for t in range(n):
                    S = torch.exp(dt[t][:, None] * A) * S + (dt[t] * u[t])[:, None] * B[t]
                    out.append(S @ C[t])
                o = (torch.stack(out) + a["D"] * u) * silu(y[:, I:])
            else:
                q, k, v = self.qkv(h, a, m)
                decay = torch.tensor(m["decay"], dtype=x.dtype, device=DEV)[None, :, None].expand(n, -1, 1)
                o = walk(rotate(q, m["rot"], False), rotate(k, m["rot"], False) * m["dim"] ** -0.5, v, decay)
                o = rms(o, self.eps).reshape(n, -1) * silu(h @ a["g"].T)
            x = x + self.raw["residual_mult"] * l["ls1"] * (o @ a["o"].T)
            h = layer_norm(x, l["norm2"], l["norm2.b"], self.eps)
            z, chosen = torch.topk(h @ e["router"].T + e["router.b"], f["router"]["top"], -1)
            y = through_experts(h, chosen, torch.softmax(z, -1), f["router"]["experts"], lambda j, rows, c: c * self.gated(rows, e, f"e{j}."))
            y = y + self.gated(h, e, "shared.") * torch.sigmoid(h @ e["shared.sg"].T)
            x = x + self.raw["residual_mult"] * l["ls2"] * y
        return w["embed"] @ layer_norm(x[-1], w["final.norm"], w["final.norm.b"], self.eps)

    def vagelix(self, tokens):
        w, n = self.w, len(tokens)
        x = rms(w.rows("embed", tokens), self.eps) * w["embed.norm"]
        for i, layer in enumerate(self.raw["layers"]):
            l, m = w.under(f"l{i}"), layer["mixer"]
            a = l.under("mix")
            if layer["type"] == "attention":
                y = self.two_maps(x, a, m)
            elif layer["type"] == "parallel":
                left = self.chunked(x, a.under("left"), m["left"])
                right = self.delta_rule(x, a.under("right"), m["right"])
                y = 0.5 * (rms(left, self.eps) * a["left.out"] + rms(right, self.eps) * a["right.out"])
            else:
                y = self.duality(x, a, m)
            x = x + rms(y, self.eps) * l["norm1"]
            x = x + rms(self.gated(x, l.under("mlp")), self.eps) * l["norm2"]
        return w["embed"] @ (rms(x[-1], self.eps) * w["final.norm"])

    def two_maps(self, h, a, m):
        n, H, d = h.shape[0], m["heads"], m["dim"]
        q = rms((h @ a["q"].T).view(n, H, 2, d), self.eps) * a["q.norm"]
        k = rms((h @ a["k"].T).view(n, m["kv_heads"], 2, d), self.eps) * a["k.norm"]
        v = (h @ a["v"].T).view(n, m["kv_heads"], -1)
        t = torch.tensor([1 + m["q_temp"]["coef"] * math.log((p + 1) // m["q_temp"]["every"] + 1) for p in range(n)], device=DEV)
        q = q * t.double().view(n, 1, 1, 1)
        lam = torch.exp((a["lq1"] * a["lk1"]).sum()) - torch.exp((a["lq2"] * a["lk2"]).sum()) + m["diff"]
        one, two = (attend(q[:, :, j], k[:, :, j], v, m["scale"], seen_keys(n)) for j in range(2))
        return (rms(one - lam * two, self.eps) * (1 - m["diff"])).reshape(n, -1) @ a["o"].T

    def chunked(self, h, a, m):
        n, H, G = h.shape[0], m["heads"], m["kv_heads"]
        q, k = h @ a["q"].T + a["q.b"], h @ a["k"].T + a["k.b"]
        v = k.view(n, G, -1)
        q = rotate((rms(q, self.eps) * a["q.norm"]).view(n, H, -1), m["rot"], False)
        k = rotate((rms(k, self.eps) * a["k.norm"]).view(n, G, -1), m["rot"], False)
        o = attend(q, k, v, m["scale"], seen_keys(n, chunk=m["mask"]["size"]), sink=[0.0] * H)
        return (o * torch.sigmoid(h @ a["g"].T).unsqueeze(-1)).reshape(n, -1) @ a["o"].T

    def delta_rule(self, h, a, m):
        n, H, dk = h.shape[0], m["heads"], m["dim"]
        q, k, v = (silu(short_conv(h @ a[c].T, a[c + ".conv"])) for c in "qkv")
        q, k = (spread_heads(t.view(n, m["kv_heads"], dk), H) for t in (q, k))
        q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        step = softplus((h @ a["a1"].T) @ a["a2"].T + a["dt_bias"]).view(n, H, dk)
        decay = torch.exp(-torch.exp(a["A_log"]).view(1, H, 1) * step)
        o = rms(walk(q * dk ** -0.5, k, v.view(n, H, -1), decay, torch.sigmoid(h @ a["b"].T)), self.eps) * a["norm"]
        return (o.reshape(n, -1) * torch.sigmoid((h @ a["g1"].T) @ a["g2"].T)) @ a["o"].T

    def duality(self, h, a, m):
        n, H, N, G = h.shape[0], m["heads"], m["state"], m["groups"]
        inner = H * m["vdim"]
        y = h @ a["in"].T
        u = silu(short_conv(y[:, inner:2 * inner + 2 * G * N], a["conv"], a["conv.b"]))
        x, B, C = u[:, :inner].view(n, H, -1), u[:, inner:inner + G * N].view(n, G, N), u[:, inner + G * N:].view(n, G, N)
        dt = softplus(y[:, 2 * inner + 2 * G * N:] + a["dt_bias"])
        o = walk(spread_heads(C, H), spread_heads(B, H) * dt.unsqueeze(-1), x, torch.exp(-torch.exp(a["A_log"]) * dt).unsqueeze(-1))
        o = (o + a["D"][:, None] * x).reshape(n, inner) * silu(y[:, :inner])
        return (rms(o.view(n, m["norm_groups"], -1), self.eps).reshape(n, inner) * a["norm"]) @ a["o"].T

    def begasun(self, tokens):
        w, n = self.w, len(tokens)
        x = w.rows("embed", tokens) * self.raw["embedding"]["scale"]
        side = self.raw["token_side"]["dim"]
        rows = w.rows("side.embed", tokens)
        for i, layer in enumerate(self.raw["layers"]):
            l, m = w.under(f"l{i}"), layer["mixer"]
            a, s = l.under("mix"), l.under("side")
            h = rms(x, self.eps) * (1 + l["norm1"])
            if layer["type"] == "latent_attention":
                o = self.latent(h, a, m, (h @ a["q"].T).view(n, m["heads"], -1)) * torch.sigmoid(h @ a["g"].T).unsqueeze(-1)
            elif layer["type"] == "rglru":
                u = short_conv(h @ a["x"].T + a["x.b"], a["conv"], a["conv.b"]).view(n, m["blocks"], -1)
                r, g = (torch.sigmoid(torch.einsum("tbc,bdc->tbd", u, a[c]) + a[c + ".b"]).reshape(n, -1) for c in ("ra", "ri"))
                log_a = -8.0 * r * softplus(a["lam"])
                add = torch.sqrt(-torch.expm1(2 * log_a)) * g * u.reshape(n, -1)
                S, out = torch.zeros_like(add[0]), []
                for t in range(n):
                    S = torch.exp(log_a[t]) * S + add[t]
                    out.append(S)
                o = torch.stack(out) * gelu_tanh(h @ a["y"].T + a["y.b"])
            else:
                q, k, v = self.qkv(h, a, m)
                q, k = (rotate(rms(t, self.eps) * a[c + ".norm"], m["rot"], False) for t, c in ((q, "q"), (k, "k")))
                o = attend(q, k, v, m["scale"], seen_keys(n))
            x = x + l["ls1"] * rms(o.reshape(n, -1) @ a["o"].T, self.eps) * (1 + l["norm1b"])
            h = rms(x, self.eps) * (1 + l["norm2"])
            x = x + l["ls2"] * rms(self.clipped(h, l.under("mlp"), layer["mlp"]["limit"]), self.eps) * (1 + l["norm2b"])
            g = gelu_tanh(x @ s["gate"].T) * rows[:, i * side:(i + 1) * side]
            x = x + rms(g @ s["proj"].T, self.eps) * s["norm"]
        return w["head"] @ (rms(x[-1], self.eps) * (1 + w["final.norm"])) * self.raw["logit_scale"]

    def tubusun(self, tokens):
        w, n = self.w, len(tokens)
        x = w.rows("embed", tokens) * self.raw["embedding"]["scale"]
        for i, layer in enumerate(self.raw["layers"]):
            l, m, f = w.under(f"l{i}"), layer["mixer"], layer["mlp"]
            h = rms(x, self.eps) * l["norm1"]
            a, p = l.under("mix.left"), m["left"]
            q, k, v = self.qkv(h, a, p)
            q, k = (rms(rotate(t, p["rot"], True), self.eps) for t in (q, k))
            o = attend(q, k, v, p["scale"], seen_keys(n, p["mask"]["size"]), sink=a["sink"].tolist())
            y = m["left_scale"] * ((o * torch.sigmoid(h @ a["g"].T).unsqueeze(-1)).reshape(n, -1) @ a["o"].T)
            a, p = l.under("mix.right"), m["right"]
            q, k, v = (silu(t) for t in self.qkv(h, a, p))
            decay = torch.tensor(p["decay"], dtype=x.dtype, device=DEV)[None, :, None].expand(n, -1, 1)
            o = rms(walk(q, k, v, decay).reshape(n, -1), self.eps) * a["norm"] * torch.sigmoid(h @ a["g"].T)
            y = y + m["right_scale"] * (o @ a["o"].T)
            x = x + rms(y, self.eps) * l["norm1b"]
            h, e = rms(x, self.eps) * l["norm2"], l.under("mlp")
            if f["kind"] == "dense":
                y = torch.nn.functional.gelu(h @ e["up"].T + e["up.b"]) @ e["down"].T + e["down.b"]
            else:
                r = f["router"]
                s = torch.sigmoid(h @ e["router"].T)
                groups = s.view(n, r["groups"]["count"], -1)
                best = torch.topk(torch.topk(groups, 2, -1).values.sum(-1), r["groups"]["keep"], -1).indices
                may = torch.zeros(groups.shape[:2], dtype=torch.bool, device=DEV).scatter_(1, best, True)
                chosen = torch.topk(s.masked_fill(~may.repeat_interleave(groups.shape[2], 1), -1.0), r["top"], -1).indices
                y = through_experts(h, chosen, torch.gather(s, 1, chosen), r["experts"],
                                    lambda j, rows, c: c * self.clipped(rows, e, f["expert"]["limit"], f"e{j}."))
            x = x + rms(y, self.eps) * l["norm2b"]
        z = w["embed"] @ (rms(x[-1], self.eps) * w["final.norm"])
        return self.raw["logit_softcap"] * torch.tanh(z / self.raw["logit_softcap"])
