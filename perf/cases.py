"""The work that is timed: whole requests through the step function, from an empty cache to their last logits.

A case is a model, a data type and a set of requests; one pass adds the requests, runs every step of their life (prompts whole
or in portions, beside requests that decode where they arrive one after another, then a token a step each), keeps the logits
at every place where a token would be sampled, and frees the requests.  The tokens are given ahead, as a replayed trace gives
them: two implementations whose sums round differently then still see the same inputs at every step.

The models are the layer sizes this repository measures: the Qwen2.5 family's and the six further designs' ("small": 1,024
wide, "medium": 2,048 wide; 8 layers, a vocabulary of 32,000).  Weights are random (see ``_weight``), made once and kept, with
the cache and the step function, as a server keeps them; the requests are what is new for every seed.
"""
import functools
import math
import random

import torch

from inferflux_amd.config import config_from_dict
from inferflux_amd.engine.context import StepEntry
from inferflux_amd.engine.model import Model
from inferflux_amd.engine.runner import ModelRunner
from inferflux_amd.weights.loader import random_tensor

PAGE = 16
STEP_TOKENS = 16384       # most tokens in a step, and the largest portion of a prompt while nobody decodes: the scheduler's defaults
PORTION_ALONE = 2048


# ---- the models --------------------------------------------------------------------------------------------------------
def _qwen(hidden, layers, heads, kv_heads, head_dim, inner, tied, vocab=151936):
    return dict(model_type="qwen2", architectures=["Qwen2ForCausalLM"], vocab_size=vocab, hidden_size=hidden, num_hidden_layers=layers,
                num_attention_heads=heads, num_key_value_heads=kv_heads, head_dim=head_dim, intermediate_size=inner,
                max_position_embeddings=32768, rope_theta=1000000.0, rms_norm_eps=1e-6, tie_word_embeddings=tied,
                attention_bias=True, use_sliding_window=False, torch_dtype="bfloat16")


def _layers(kinds, pattern, mlp):
    return [{"type": kinds[c][0], "mixer": kinds[c][1], "mlp": mlp} for c in pattern]


def _design(name, width):
    """A further design's config: heads of 128 elements, 8 layers in the order that mixes its kinds of layer."""
    heads, w = width // 128, width // 1024
    base = {"architecture": name.capitalize(), "vocab": 32000, "width": width, "norm": {"eps": 1e-5}}
    att = {"heads": heads, "kv_heads": 2, "dim": 128, "vdim": 128, "scale": 128 ** -0.5}
    rec = {"heads": heads, "dim": 64, "vdim": 128}
    if name == "mumusun":
        lat = {"heads": heads, "dim": 96, "rot_dim": 32, "vdim": 128, "q_rank": 384 * w, "kv_rank": 96, "scale": 128 ** -0.5,
               "rot": {"base": 10000.0, "dims": 32}, "mask": {"size": width}}
        router = {"experts": 64, "top": 6, "groups": {"count": 8, "keep": 4}} if w > 1 else {"experts": 16, "top": 2, "groups": {"count": 4, "keep": 2}}
        return dict(base, layers=_layers({"l": ("latent_attention", lat)}, "l" * 8, {"kind": "moe", "expert": {"ff": 704 * w}, "router": router}))
    if name == "podurax":
        att.update(v_mix=True, mask={"size": width, "keep_first": 4},
                   rot={"base": 5e5, "dims": 64, "scaling": {"factor": 4.0, "original": 4096, "fast": 16.0, "slow": 1.0}})
        ssm = {"inner": 2 * width, "state": 16, "dt_rank": width // 16, "conv": 4}
        return dict(base, embedding={"scale": 1.0}, residual_mult=0.5,
                    layers=_layers({"a": ("attention", att), "m": ("mamba1", ssm)}, "aamaaama", {"kind": "dense", "ff": 2816 * w}))
    if name == "tabatar":
        att.update(mask={"size": width}, rot={"base": 5e5, "dims": 64, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 4096}})
        gla = dict(rec, tau=16.0, rank=64 * w)
        return dict(base, embedding={"scale": 1.0}, streams=4, logit_scale=1.0, logit_softcap=30.0,
                    layers=_layers({"a": ("attention", att), "g": ("gla", gla)}, "ggagggag", {"kind": "dense", "ff": 4224 * w}))
    if name == "vavadra":
        lat = {"heads": heads, "dim": 64, "rot_dim": 32, "vdim": 128, "kv_rank": 96, "scale": 96 ** -0.5, "rot": {"base": 10000.0, "dims": 32},
               "mask": {"size": width}}
        dif = {"heads": heads, "kv_heads": 2, "dim": 64, "vdim": 128, "scale": 0.125, "diff": 0.5, "mask": {"size": width}}
        ff = {"ff": 704 * w, "limit": 7.0}
        mlp = {"kind": "moe", "expert": ff, "router": {"experts": 14 * w, "identity": 2 * w, "top": 2 * w, "scale": 1.0}, "shared": ff}
        kinds = {"l": ("latent_attention", lat), "a": ("attention", dif), "d": ("delta", dict(rec, kv_heads=heads, conv=4))}
        return dict(base, embedding={"scale": 1.0}, logit_scale=1.0, layers=_layers(kinds, "laldlald", mlp))
    if name == "narasun":
        left = dict(att, q_temp={"coef": 0.1, "every": 1024})
        par = {"left": left, "right": {"heads": heads, "dim": 64, "rank": 64 * w}, "left_scale": 0.7, "right_scale": 0.7}
        mlp = {"kind": "moe", "expert": {"ff": 1408}, "router": {"experts": 16 * w, "top": 2 * w}}
        return dict(base, layers=_layers({"m": ("mlstm", dict(rec, gate_cap=15.0)), "p": ("parallel", par)}, "mmpmmmpm", mlp))
    dim = 96 if w == 1 else 128
    lat = {"heads": heads, "dim": dim - 32, "rot_dim": 32, "vdim": dim, "q_rank": 384 * w, "kv_rank": 96, "scale": dim ** -0.5,
           "rot": {"base": 10000.0, "dims": 32}}
    gat = {"heads": heads, "dim": dim, "vdim": dim, "q_rank": 384 * w, "kv_rank": 128, "scale": dim ** -0.5}
    ret = dict(rec, decay=[1.0 - 2.0 ** -(5 + 7.0 * i / heads) for i in range(heads)], rot={"base": 10000.0, "dims": 64})
    router = {"experts": 16 * w, "top": 2 * w, "groups": {"count": 4 * w, "keep": w + 1}}
    kinds = {"r": ("retention", ret), "l": ("latent_attention", lat), "g": ("latent_attention_2", gat), "s": ("latent_attention_2", dict(gat, kv_from=0))}
    return dict(base, embedding={"scale": 1.0}, logit_softcap=30.0,
                layers=_layers(kinds, "grlrsrlr", {"kind": "moe", "expert": {"ff": 704 * w, "limit": 7.0}, "router": router}))


QWEN = {
    "qwen2.5-0.5b": _qwen(896, 24, 14, 2, 64, 4864, True),
    "qwen2.5-1.5b": _qwen(1536, 28, 12, 2, 128, 8960, True),
    "qwen2.5-3b": _qwen(2048, 36, 16, 2, 128, 11008, True),
    "qwen2.5-7b": _qwen(3584, 28, 28, 4, 128, 18944, False, vocab=152064),
}
DESIGNS = ("mumusun", "podurax", "tabatar", "vavadra", "narasun", "duletar")
WIDTHS = {"small": 1024, "medium": 2048}


@functools.lru_cache(maxsize=None)
def _config(model):
    if model in QWEN:
        return QWEN[model]
    design, size = model.split("-")
    return _design(design, WIDTHS[size])


def _weight(name, spec, model):
    """A tensor by the model's own random rule, in the proportions that trained models have: embeddings of about a half, and
    the sub-blocks' last products smaller, so that the stream is a sum of many parts none of which drowns the others.  (With
    every matrix at 0.02 the first layers' roundings grow from layer to layer, and logits say little.  Experts add less still:
    a router with random weights has many close choices, and one that falls the other way moves a whole expert.)"""
    t = random_tensor(name, spec, 0, torch.bfloat16, "cuda")
    width = _config(model).get("hidden_size") or _config(model)["width"]
    last = name.split(".")[-2 if name.endswith(".weight") else -1]
    if "embed" in name:
        return t * 32.0
    if last in ("o", "o_proj", "down", "down_proj"):
        return t * 2.0 ** -round(math.log2(width / 512.0)) * (0.25 if ".mlp.e" in name else 1.0)
    if model.startswith("mumusun") and last in ("norm1", "norm2"):        # (these norms stand on the sub-blocks' outputs)
        return t * 0.03125
    return t


# ---- the cases -----------------------------------------------------------------------------------------------------------
def _case(name, model, requests, prompt, new, ragged=0.0, gap=0, portion=512, dtype="bfloat16"):
    """``prompt``: the longest prompt; ``ragged``: the share of it by which prompts are shorter at most; ``gap``: steps between
    two arrivals (0: all there at the start); ``portion``: most tokens of a prompt in a step beside requests that decode."""
    return dict(name=name, model=model, dtype=dtype, requests=requests, prompt=prompt, new=new, ragged=ragged, gap=gap, portion=portion)


def listed():
    return [
        _case("chat 0.5B", "qwen2.5-0.5b", 1, 61, 64),                                   # one short question answered: the smallest steps there are
        _case("batch of 8 7B", "qwen2.5-7b", 8, 1024, 48, ragged=0.5),                   # the headline size, a few users
        _case("long prompt 7B", "qwen2.5-7b", 1, 8192, 1),                               # a document read in portions of 2,048
        _case("serving 3B", "qwen2.5-3b", 24, 1024, 24, ragged=0.95, gap=1),             # prompts in portions of 512 beside requests that decode
        _case("batch of 64 1.5B", "qwen2.5-1.5b", 64, 200, 24, ragged=0.9),              # offline generation, the widest decode steps
        _case("32 bits 0.5B", "qwen2.5-0.5b", 4, 150, 16, ragged=0.5, dtype="float32"),  # the mode that logits are checked in
        _case("batch of 8 Mumusun", "mumusun-medium", 8, 600, 32, ragged=0.4),           # a latent and many experts, decoding
        _case("prompt Podurax", "podurax-medium", 1, 2048, 8),                           # attention and state-space layers over a long prompt
        _case("batch of 16 Tabatar", "tabatar-medium", 16, 333, 32, ragged=0.5),         # linear attention on several streams
        _case("chat Vavadra", "vavadra-medium", 1, 700, 48),                             # delta rule, differential attention, shared experts
        _case("batch of 64 Narasun", "narasun-medium", 64, 65, 16, ragged=0.9),          # short questions to matrix memories
        _case("four documents Duletar", "duletar-medium", 4, 1500, 16, ragged=0.3),      # retention and shared latents
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """Requests, lengths and models between the listed ones; costs are held to the largest listed case's."""
    bound = _largest()
    while True:
        model = rng.choice(list(QWEN)) if rng.random() < 0.5 else "%s-%s" % (rng.choice(DESIGNS), rng.choice(list(WIDTHS)))
        c = _case(None, model, _log_uniform(rng, 1, 64), _log_uniform(rng, 8, 8192 if model in QWEN else 2048), _log_uniform(rng, 1, 64),
                  ragged=round(rng.uniform(0.0, 0.95), 2), gap=rng.choice([0, 0, 0, 1, 2]), portion=rng.choice([256, 512, 512, 1024]))
        del c["name"]
        if rng.random() < 0.1 and model.endswith(("small", "0.5b")):
            c["dtype"] = "float32"
        if _cost(c) <= bound and c["requests"] * c["new"] <= 2048:
            return c


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / (8.0 if case["dtype"] == "float32" else 50.0))     # (the 32-bit matrix rate is a fraction of the 16-bit one)


@functools.lru_cache(maxsize=1)
def _largest():
    return max(_cost(c) for c in listed())


# ---- requests and their steps ----------------------------------------------------------------------------------------------
def _lengths(case, seed):
    """The prompts' lengths: the longest first, the others shorter by up to the case's share of it (the same for every seed
    of a case but for their order, so that every seed is the same work)."""
    n, longest = case["requests"], case["prompt"]
    out = [max(1, round(longest * (1.0 - case["ragged"] * i / max(n - 1, 1)))) for i in range(n)]
    random.Random(seed).shuffle(out)
    return out


def _steps(case, lengths):
    """[[(request, first token, tokens, whether its last token's logits are wanted)]]: every step's shares, dealt as the scheduler
    deals them: running requests first, each a token or a portion of its prompt, then those that wait."""
    n, new = case["requests"], case["new"]
    done, steps, at = [0] * n, [], 0
    while any(done[r] < lengths[r] + new - 1 for r in range(n)):
        here = [r for r in range(n) if r * case["gap"] <= at]
        decoding = any(lengths[r] <= done[r] < lengths[r] + new - 1 for r in here)
        portion, left, step = case["portion"] if decoding else max(case["portion"], PORTION_ALONE), STEP_TOKENS, []
        for r in sorted(here, key=lambda r: (done[r] == 0, r)):
            if left <= 0 or done[r] >= lengths[r] + new - 1:
                continue
            k = min(lengths[r] - done[r], portion, left) if done[r] < lengths[r] else 1
            step.append((r, done[r], k, done[r] + k >= lengths[r]))
            done[r] += k
            left -= k
        if step:
            steps.append(step)
        at += 1
    return steps


def _requests(case, seed):
    """Each request's tokens, its prompt and all it is given afterwards."""
    vocab = _config(case["model"]).get("vocab_size") or _config(case["model"])["vocab"]
    lengths = _lengths(case, seed)
    g = torch.Generator().manual_seed(seed)
    return lengths, [torch.randint(0, vocab, (n + case["new"] - 1,), generator=g).tolist() for n in lengths]


def _model(name, dtype):
    model = Model(config_from_dict(_config(name)))
    tensors = {n: _weight(n, s, name).to(dtype) for n, s in model.param_specs().items()}
    return model.bind(tensors, dtype, torch.device("cuda", 0))


_KEPT = {}     # the model and its step function, as a server keeps them: one at a time


def _runner(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _KEPT:
        model_key = (case["model"], case["dtype"])
        kept = next((r.model for k, r in _KEPT.items() if (dict(k)["model"], dict(k)["dtype"]) == model_key), None)
        _KEPT.clear()
        torch.cuda.empty_cache()
        model = kept or _model(case["model"], getattr(torch, case["dtype"]))
        pages = sum(-(-(n + case["new"]) // PAGE) + 1 for n in _lengths(case, 0))
        _KEPT[key] = ModelRunner(model, num_pages=pages, page_size=PAGE, max_requests=case["requests"])
    return _KEPT[key]


def prepare(case, seed):
    runner = _runner(case)
    lengths, tokens = _requests(case, seed)
    steps = [[(r, tokens[r][a:a + n], want) for r, a, n, want in step] for step in _steps(case, lengths)]
    rows = case["requests"] * case["new"]
    return {"runner": runner, "requests": case["requests"], "steps": steps,
            "logits": torch.empty((rows, runner.vocab_size), dtype=torch.float32, device=runner.device)}


def run(state):
    """The logits at every place where a token is sampled, in the order of the steps."""
    runner, out, at = state["runner"], state["logits"], 0
    live = set()
    for step in state["steps"]:
        for r, _, _ in step:
            if r not in live:
                runner.add_request(r)
                live.add(r)
        logits = runner.step([StepEntry(r, tokens, [len(tokens) - 1] if want else []) for r, tokens, want in step])
        out[at:at + logits.shape[0]].copy_(logits)      # (a decode step's logits are valid until the next step)
        at += logits.shape[0]
    for r in live:
        runner.free_request(r)
    return out


# ---- what a pass cannot do without -----------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _inventory(model):
    """(numbers of weights that every token meets, {expert layer: (weights of one expert, experts, top)}, head's weights, per layer
    run (cache elements a token, window) and the recurrent state's elements a request)."""
    cfg = config_from_dict(_config(model))
    m = Model(cfg)
    dense, experts, head, tops = 0, {}, 0, {}
    for i, layer in enumerate(_config(model).get("layers", ())):
        r = layer["mlp"].get("router")
        if r:
            tops["l%d" % i] = (r["experts"] + r.get("identity", 0), r["top"])
    for n, s in m.param_specs().items():
        size = math.prod(s.shape)
        parts = n.split(".")
        if n in ("embed", "model.embed_tokens.weight"):
            continue
        if n in ("head", "lm_head.weight"):
            head = size
        elif len(parts) > 2 and parts[1] == "mlp" and parts[2][0] == "e" and parts[2][1:].isdigit():
            experts[parts[0]] = experts.get(parts[0], 0) + size
        else:
            dense += size
    width = m.plan.hidden_size
    head = head or m.plan.vocab_size * width
    per_expert = {k: (v / len([1 for n in m.param_specs() if n.startswith(k + ".mlp.e") and n.endswith(".up")]), *tops[k]) for k, v in experts.items()}
    caches, state = [], 0
    for e, mixer in zip(m.plan.schedule, m.schedule_mixers()):
        c, s = mixer.cache_spec(), mixer.state_spec()
        if c is not None:
            latent = hasattr(mixer, "kv_rank")          # (one row of the latent and the rotated part, read as key and as value)
            heads = getattr(mixer, "n_heads", None) or mixer.children()[0].n_heads      # (two mixers side by side: the first has the cache)
            score = mixer.dim + mixer.rot_dim + mixer.v_dim if latent else c.k_dim + c.v_dim
            caches.append((c.k_dim if latent else c.n_kv_heads * (c.k_dim + c.v_dim), heads * score, c.window))
        state += math.prod(s.shape) if s is not None else 0
    return dense, per_expert, head, tuple(caches), state, m.plan.vocab_size


def work(case):
    """Weights once a step (of experts, as many as the step's tokens are expected to choose), each request's visible cache and
    recurrent state once a step, new cache entries and logits written once; the products and the scores of every token."""
    dense, experts, head, caches, state, vocab = _inventory(case["model"])
    esz = 4 if case["dtype"] == "float32" else 2
    nbytes = flops = 0.0
    for step in _steps(case, _lengths(case, 0)):
        tokens, wanted = sum(s[2] for s in step), sum(1 for s in step if s[3])
        nbytes += esz * (dense + (head if wanted else 0)) + 4.0 * wanted * vocab + 8.0 * state * len(step)
        flops += 2.0 * (tokens * dense + wanted * head)
        for size, n, top in experts.values():
            nbytes += esz * size * n * (1.0 - (1.0 - top / n) ** tokens)
            flops += 2.0 * tokens * top * size
        for _, start, k, _ in step:
            for elements, score, window in caches:
                seen = start + k if window is None else min(start + k, window + k)
                nbytes += esz * elements * (seen + k)
                pairs = k * start + k * (k + 1) / 2.0
                flops += 2.0 * score * (pairs if window is None else min(pairs, float(k) * window))
    return {"bytes": nbytes, "flops": flops}


# ---- the same in 64 bits, from the formulas -----------------------------------------------------------------------------------
class _Weights:
    """The case's weights by name, as 64-bit matrices when they are asked for."""

    def __init__(self, model):
        self.model, self.specs = model, Model(config_from_dict(_config(model))).param_specs()

    def __contains__(self, name):
        return name in self.specs

    def __getitem__(self, name):
        return _weight(name, self.specs[name], self.model).double()


def _rms(x, eps, w=None):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _layer_norm(x, w, eps):
    x = x - x.mean(-1, keepdim=True)
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _frequencies(rot, dims):
    """(frequency of each pair, the factor on cosine and sine): plain, stretched by bands of wavelength ("low" / "high") or by a
    ramp over the pairs ("fast" / "slow")."""
    f = torch.tensor([rot["base"] ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=torch.float64)
    sc = rot.get("scaling")
    if not sc:
        return f.cuda(), 1.0
    if "low" in sc:
        turns = sc["original"] * f / (2.0 * math.pi)
        s = ((turns - sc["low"]) / (sc["high"] - sc["low"])).clamp(0.0, 1.0)
        return ((1.0 - s) * f / sc["factor"] + s * f).cuda(), 1.0
    pair = lambda n: dims * math.log(sc["original"] / (2.0 * math.pi * n)) / (2.0 * math.log(rot["base"]))
    lo, hi = max(math.floor(pair(sc["fast"])), 0), min(math.ceil(pair(sc["slow"])), dims - 1)
    ramp = ((torch.arange(dims // 2, dtype=torch.float64) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return (f / sc["factor"] * ramp + f * (1.0 - ramp)).cuda(), 0.1 * math.log(sc["factor"]) + 1.0


def _rotate(x, rot, dims, interleaved=False):
    """x [B, T, heads, d]: the first ``dims`` elements of a head turned by their position's angles."""
    f, size = _frequencies(rot, dims)
    a = torch.arange(x.shape[1], dtype=torch.float64, device=x.device)[:, None] * f
    c, s = (a.cos() * size)[:, None, :], (a.sin() * size)[:, None, :]
    if interleaved:
        u, v = x[..., 0:dims:2], x[..., 1:dims:2]
        return torch.cat([torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2), x[..., dims:]], -1)
    u, v = x[..., :dims // 2], x[..., dims // 2:dims]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], -1)


def _mask(T, window=None, keep=0, block=None):
    i, j = torch.arange(T, device="cuda")[:, None], torch.arange(T, device="cuda")[None, :]
    ok = j <= i
    if window:
        ok &= (i - j < window) | (j < keep)
    return ok & (i // block == j // block) if block else ok


def _attend(q, k, v, scale, mask, sink=None):
    """q [B, T, H, d], k [B, T, G, d], v [B, T, G, dv]; ``sink`` [H]: one more score, without a value."""
    B, T, H, _ = q.shape
    G, out = k.shape[2], []
    for b in range(B):
        heads = []
        for g in range(G):
            s = q[b, :, g * (H // G):(g + 1) * (H // G)].transpose(0, 1) @ k[b, :, g].t().contiguous() * scale
            s = s.masked_fill(~mask, -math.inf)
            if sink is None:
                p = s.softmax(-1)
            else:
                z = sink[g * (H // G):(g + 1) * (H // G), None, None]
                m = torch.maximum(s.amax(-1, keepdim=True), z)
                e = (s - m).exp()
                p = e / (e.sum(-1, keepdim=True) + (z - m).exp())
            heads.append((p @ v[b, :, g]).transpose(0, 1))
        out.append(torch.cat(heads, 1))
    return torch.stack(out)


def _scan(q, k, v, step):
    """A matrix state per head, S [B, H, d, dv]: ``step(t, S)`` gives the state after token t; the output is S^T q."""
    S, out = q.new_zeros(*q.shape[:1], *q.shape[2:], v.shape[-1]), []
    for t in range(q.shape[1]):
        S = step(t, S)
        out.append((S * q[:, t, :, :, None]).sum(-2))
    return torch.stack(out, 1)


def _conv(x, w, b=0.0):
    taps = w.shape[1]
    x = torch.cat([x.new_zeros(x.shape[0], taps - 1, x.shape[2]), x], 1)
    return sum(x[:, j:x.shape[1] - taps + 1 + j] * w[:, j] for j in range(taps)) + b


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


silu, sigmoid, softplus = torch.nn.functional.silu, torch.sigmoid, lambda z: torch.logaddexp(z, torch.zeros_like(z))


class _Exact:
    """One whole batch of sequences [B, T] through a model, layer by layer."""

    def __init__(self, model):
        self.cfg, self.W = _config(model), _Weights(model)
        self.name = model.split("-")[0]
        self.eps = self.cfg["norm"]["eps"] if "norm" in self.cfg else self.cfg["rms_norm_eps"]
        self.kept = {}          # what one layer leaves for others: values that are mixed in, latents that are shared

    def product(self, h, name):
        y = h @ self.W[name].t()
        return y + self.W[name + ".b"] if name + ".b" in self.W else y

    def heads(self, h, name, n):
        y = self.product(h, name)
        return y.view(*y.shape[:2], n, -1)

    # mixers of the further designs
    def attention(self, h, p, m):
        H, G, T, W = m["heads"], m["kv_heads"], h.shape[1], self.W
        q, k, v = self.heads(h, p + "q", H), self.heads(h, p + "k", G), self.heads(h, p + "v", G)
        mask = _mask(T, (m.get("mask") or {}).get("size"), (m.get("mask") or {}).get("keep_first", 0))
        if self.name == "podurax":
            q, k = (_rms(_rotate(x, m["rot"], m["rot"]["dims"]), self.eps) for x in (q, k))
            first = self.kept.setdefault("values", v)
            if first is not v:
                lam = self.W[p + "vmix"]
                v = (1.0 - lam) * v + lam * first
            o = _attend(q, k, v, m["scale"], mask, q.new_zeros(H)) * sigmoid(self.product(h, p + "g"))[..., None]
        elif self.name == "tabatar":
            q, k = (_rotate(_rms(x, self.eps, W[p + n]), m["rot"], m["rot"]["dims"]) for x, n in ((q, "q.norm"), (k, "k.norm")))
            o = _attend(q, k, v, m["scale"], mask).flatten(2) * sigmoid(self.product(h, p + "g"))
        elif self.name == "narasun":
            pos = torch.arange(T, dtype=torch.float64, device=h.device)
            temp = 1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((pos + 1) / m["q_temp"]["every"]) + 1.0)
            o = _attend(q * temp[:, None, None], k, v, m["scale"], mask, W[p + "sink"])
        else:                                   # two maps over the same values, the second taken off
            mask, q, k = _mask(T, block=m["mask"]["size"]), q.unflatten(-1, (2, -1)), k.unflatten(-1, (2, -1))
            lam = (W[p + "lq1"] * W[p + "lk1"]).sum().exp() - (W[p + "lq2"] * W[p + "lk2"]).sum().exp() + m["diff"]
            one, two = (_attend(q[..., c, :], k[..., c, :], v, m["scale"], mask) for c in (0, 1))
            o = _rms(one - lam * two, self.eps) * (1.0 - m["diff"])
        return self.product(o.flatten(2) if o.dim() == 4 else o, p + "o")

    def latent_attention(self, h, p, m):
        H, d, r, rank, W = m["heads"], m["dim"], m.get("rot_dim", 0), m["kv_rank"], self.W
        if p + "dq" in W:
            q = self.heads(_rms(self.product(h, p + "dq"), self.eps, W[p + "dq.norm"]), p + "uq", H)
        else:
            q = self.heads(h, p + "q", H)
        if m.get("kv_from") is None:
            down = self.product(h, p + "dkv")
            self.kept[p] = c = _rms(down[..., :rank], self.eps, W[p + "dkv.norm"])
        else:
            c = self.kept["l%d.mix." % m["kv_from"]]
        k, v = self.heads(c, p + "uk", H), self.heads(c, p + "uv", H)
        if r:
            turn = lambda x: _rotate(x, m["rot"], m["rot"]["dims"], interleaved=self.name == "vavadra")
            k = torch.cat([k, turn(down[..., None, rank:]).expand(*k.shape[:3], r)], -1)
            q = torch.cat([q[..., :d], turn(q[..., d:])], -1)
        o = _attend(q, k, v, m["scale"], _mask(h.shape[1], (m.get("mask") or {}).get("size")), W[p + "sink"] if p + "sink" in W else None).flatten(2)
        if p + "g" in W:
            o = o * sigmoid(self.product(h, p + "g"))
        return self.product(o, p + "o")

    latent_attention_2 = latent_attention

    def mamba1(self, h, p, m):
        C, N, R, W = m["inner"], m["state"], m["dt_rank"], self.W
        x, z = self.product(h, p + "in").split(C, -1)
        x = silu(_conv(x, W[p + "conv"], W[p + "conv.b"]))
        low, Bm, Cm = self.product(x, p + "x").split([R, N, N], -1)
        dt = softplus(self.product(low, p + "dt"))
        A, S, y = -W[p + "A_log"].exp(), x.new_zeros(x.shape[0], C, N), []
        for t in range(x.shape[1]):
            S = (dt[:, t, :, None] * A).exp() * S + (dt[:, t] * x[:, t])[..., None] * Bm[:, t, None, :]
            y.append((S * Cm[:, t, None, :]).sum(-1))
        return self.product((torch.stack(y, 1) + W[p + "D"] * x) * silu(z), p + "o")

    def gla(self, h, p, m):
        H, W = m["heads"], self.W
        q, k, v = self.heads(h, p + "q", H) * m["dim"] ** -0.5, self.heads(h, p + "k", H), self.heads(h, p + "v", H)
        a = (sigmoid(self.product(self.product(h, p + "a1"), p + "a2")) ** (1.0 / m["tau"])).view_as(k)
        o = _scan(q, k, v, lambda t, S: a[:, t, :, :, None] * S + k[:, t, :, :, None] * v[:, t, :, None, :])
        return self.product(_rms(o, self.eps, W[p + "norm"]).flatten(2) * silu(self.product(h, p + "g")), p + "o")

    def retention(self, h, p, m):
        H = m["heads"]
        q, k = (_rotate(self.heads(h, p + n, H), m["rot"], m["rot"]["dims"]) for n in "qk")
        k, v = k * m["dim"] ** -0.5, self.heads(h, p + "v", H)
        decay = torch.tensor(m["decay"], dtype=torch.float64, device=h.device)[:, None, None]
        o = _scan(q, k, v, lambda t, S: decay * S + k[:, t, :, :, None] * v[:, t, :, None, :])
        return self.product(_rms(o, self.eps).flatten(2) * silu(self.product(h, p + "g")), p + "o")

    def delta(self, h, p, m):
        H, W = m["heads"], self.W
        q, k, v = (silu(_conv(self.product(h, p + n), W[p + n + ".conv"])).unflatten(-1, (H, -1)) for n in "qkv")
        unit = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)
        q, k, beta = unit(q) * m["dim"] ** -0.5, unit(k), sigmoid(self.product(h, p + "b"))
        decay = (-W[p + "A_log"].exp() * softplus(self.product(h, p + "a") + W[p + "dt_bias"])).exp()

        def step(t, S):
            S = decay[:, t, :, None, None] * S
            u = beta[:, t, :, None] * (v[:, t] - (S * k[:, t, :, :, None]).sum(-2))
            return S + k[:, t, :, :, None] * u[:, :, None, :]
        return self.product((_rms(_scan(q, k, v, step), self.eps, W[p + "norm"])).flatten(2) * silu(self.product(h, p + "g")), p + "o")

    def mlstm(self, h, p, m):
        H, W = m["heads"], self.W
        q, k, v = self.heads(h, p + "q", H) * m["dim"] ** -0.5, self.heads(h, p + "k", H), self.heads(h, p + "v", H)
        cap = lambda z: m["gate_cap"] * torch.tanh(z / m["gate_cap"])
        log_i, log_f = cap(self.product(h, p + "i")), torch.nn.functional.logsigmoid(cap(self.product(h, p + "f")))
        S, n, top, out = q.new_zeros(*q.shape[:1], *q.shape[2:], v.shape[-1]), torch.zeros_like(q[:, 0]), torch.zeros_like(log_i[:, 0]), []
        for t in range(q.shape[1]):
            new = torch.maximum(log_f[:, t] + top, log_i[:, t])
            keep, write = (log_f[:, t] + top - new).exp()[..., None], (log_i[:, t] - new).exp()[..., None]
            n = keep * n + write * k[:, t]
            S, top = keep[..., None] * S + (write * k[:, t])[..., None] * v[:, t, :, None, :], new
            den = torch.maximum((n * q[:, t]).sum(-1).abs(), (-top).exp()) + 1e-6
            out.append((S * q[:, t, :, :, None]).sum(-2) / den[..., None])
        o = _rms(torch.stack(out, 1), self.eps).flatten(2) * W[p + "norm"]
        return self.product(o * sigmoid(self.product(h, p + "g")), p + "o")

    def parallel(self, h, p, m):
        t, r, W = h.shape[1], m["right"], self.W
        H, before, pr = r["heads"], torch.nn.functional.pad(h, (0, 0, 1, 0))[:, :t], p + "right."
        mix = {s: h + (before - h) * W[pr + "mu." + s] for s in "rkvgw"}
        q, k, v = (self.heads(mix[s], pr + s, H) for s in "rkv")
        w = (-(self.product(self.product(mix["w"], pr + "w1").tanh(), pr + "w2") + W[pr + "w0"]).exp()).exp().view_as(k)
        u, S, out = W[pr + "u"][..., None], q.new_zeros(*q.shape[:1], *q.shape[2:], v.shape[-1]), []
        for i in range(t):
            kv = k[:, i, :, :, None] * v[:, i, :, None, :]
            out.append(((S + u * kv) * q[:, i, :, :, None]).sum(-2))
            S = w[:, i, :, :, None] * S + kv
        right = self.product(_rms(torch.stack(out, 1), self.eps).flatten(2) * W[pr + "norm"] * silu(self.product(mix["g"], pr + "g")), pr + "o")
        return m["left_scale"] * self.attention(h, p + "left.", m["left"]) + m["right_scale"] * right

    # feed-forwards
    def expert(self, h, p, limit=None):
        g, u = self.product(h, p + "gate"), self.product(h, p + "up")
        if limit is None:
            return self.product(silu(g) * u, p + "down")
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return self.product(g * sigmoid(1.702 * g) * (u + 1.0), p + "down")

    def feed_forward(self, h, p, m):
        if m["kind"] == "dense":
            if self.name == "podurax":
                return self.product(_gelu(self.product(h, p + "gate")) * self.product(h, p + "up"), p + "down")
            return self.product(_gelu(self.product(h, p + "up")), p + "down")
        r, limit, W = m["router"], m["expert"].get("limit"), self.W
        shape, h = h.shape, h.flatten(0, 1)
        z = self.product(h, p + "router")
        s = sigmoid(z) if self.name in ("mumusun", "narasun") else z.softmax(-1)
        choice = s + W[p + "correction"] if p + "correction" in W else s
        if r.get("groups"):
            n = r["groups"]["count"]
            by = choice.unflatten(-1, (n, -1))
            worth = by.topk(2, -1).values.sum(-1) if self.name == "mumusun" else by.amax(-1)
            best = torch.zeros_like(worth).scatter(1, worth.topk(r["groups"]["keep"], -1).indices, 1.0) > 0
            choice = by.masked_fill(~best[..., None], -math.inf).flatten(1)
        ids = choice.topk(r["top"], -1).indices
        weight = s.gather(1, ids) * r.get("scale", 1.0)
        if self.name == "duletar":
            weight = weight / (weight.sum(-1, keepdim=True) + 1e-20)
        out = torch.zeros_like(h)
        for e in range(z.shape[1]):
            rows, place = (ids == e).nonzero(as_tuple=True)
            if rows.numel():
                w, x = weight[rows, place, None], h[rows]
                if e >= r["experts"]:
                    y = w * x
                elif self.name == "narasun":
                    y = self.expert(w * x, "%se%d." % (p, e))
                else:
                    y = w * self.expert(x, "%se%d." % (p, e), limit)
                out.index_add_(0, rows, y)
        if m.get("shared"):
            out = out + self.expert(h, p + "shared.", m["shared"].get("limit"))
        return out.view(shape)

    # whole models
    def design(self, tokens):
        cfg, W, eps, streams = self.cfg, self.W, self.eps, self.cfg.get("streams")
        x = W["embed"][tokens] * cfg.get("embedding", {}).get("scale", 1.0)
        xs = torch.stack([x] * streams) if streams else None
        for i, L in enumerate(cfg["layers"]):
            norm = lambda n, y: (_layer_norm(y, W["l%d.%s" % (i, n)], eps) if self.name == "mumusun" else
                                 _rms(y, eps, W["l%d.%s" % (i, n)] + (1.0 if self.name == "narasun" else 0.0)))
            mix = lambda h: getattr(self, L["type"])(h, "l%d.mix." % i, L["mixer"])
            ff = lambda h: self.feed_forward(h, "l%d.mlp." % i, L["mlp"])
            if self.name == "mumusun":              # norms on the sub-blocks' outputs
                x = x + norm("norm1", mix(x))
                x = x + norm("norm2", ff(x))
            elif self.name == "narasun":            # one norm for both sub-blocks
                h = norm("norm1", x)
                x = x + mix(h) + ff(h)
            elif streams:
                for hc, sub in (("hc1", lambda u: mix(norm("norm1", u))), ("hc2", lambda u: ff(norm("norm2", u)))):
                    at = "l%d.%s." % (i, hc)
                    y = sub((W[at + "in"][:, None, None, None] * xs).sum(0))
                    xs = torch.tensordot(W[at + "mix"].t().contiguous(), xs, 1) + W[at + "out"][:, None, None, None] * y
            else:
                mult = cfg.get("residual_mult", 1.0)
                x = x + mult * mix(norm("norm1", x))
                x = x + mult * ff(norm("norm2", x))
        x = xs.sum(0) if streams else x
        w = W["final.norm"] + (1.0 if self.name == "narasun" else 0.0)
        return _layer_norm(x, w, eps) if self.name == "mumusun" else _rms(x, eps, w)

    def qwen(self, tokens):
        cfg, W, eps = self.cfg, self.W, self.eps
        H, G, d = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
        x, mask, rot = W["model.embed_tokens.weight"][tokens], _mask(tokens.shape[1]), {"base": cfg["rope_theta"]}
        for i in range(cfg["num_hidden_layers"]):
            p = "model.layers.%d." % i
            h = _rms(x, eps, W[p + "input_layernorm.weight"])
            q, k, v = ((h @ W[p + "self_attn.%s_proj.weight" % n].t() + W[p + "self_attn.%s_proj.bias" % n]).unflatten(-1, (a, d))
                       for n, a in (("q", H), ("k", G), ("v", G)))
            o = _attend(_rotate(q, rot, d), _rotate(k, rot, d), v, d ** -0.5, mask).flatten(2)
            x = x + o @ W[p + "self_attn.o_proj.weight"].t()
            h = _rms(x, eps, W[p + "post_attention_layernorm.weight"])
            x = x + (silu(h @ W[p + "mlp.gate_proj.weight"].t()) * (h @ W[p + "mlp.up_proj.weight"].t())) @ W[p + "mlp.down_proj.weight"].t()
        return _rms(x, eps, W["model.norm.weight"])

    def logits(self, rows):
        W, cfg = self.W, self.cfg
        name = next(n for n in ("head", "lm_head.weight", "embed", "model.embed_tokens.weight") if n in W)
        z = rows @ W[name].t() * cfg.get("logit_scale", 1.0)
        cap = cfg.get("logit_softcap")
        return cap * torch.tanh(z / cap) if cap else z


def exact(case, seed):
    lengths, tokens = _requests(case, seed)
    batch = torch.zeros((len(tokens), max(len(t) for t in tokens)), dtype=torch.long, device="cuda")     # (what stands behind a sequence's end reaches nothing)
    for r, t in enumerate(tokens):
        batch[r, :len(t)] = torch.tensor(t)
    m = _Exact(case["model"])
    x = (m.qwen if case["model"] in QWEN else m.design)(batch)
    wanted = [(r, a + n - 1) for step in _steps(case, lengths) for r, a, n, want in step if want]
    return m.logits(x[[r for r, _ in wanted], [p for _, p in wanted]])


def tolerance(case):
    """Four times what two of the framework's own ways to the same logits (the weights with and without their tiled copy, whose
    kernels add up in other orders) are apart, up to 0.0095 and 0.07 of the root mean square: activations are rounded to 16 bits
    before every product.  Where a router's close choices fall the other way, single rows move by a whole expert (0.25 seen)."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-4}
    experts = "layers" in _config(case["model"]) and "router" in _config(case["model"])["layers"][0]["mlp"]
    return {"rel": 0.03, "max": 0.95 if experts else 0.28}
