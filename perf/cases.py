"""What this engine is measured on: steps of its served models, and layers of the designs that route tokens to experts.

The models have their shape's layer sizes and vocabulary and the first few of its layers.  Every layer of bfloat16 work
rounds anew, and with random weights the rounding of all 36 layers of the 8B shape moves the logits by 4.5 to 5 %: two
correct models would then be further apart than any tolerance that could tell a mistake.  Six layers stay below 2 %.

Two kinds of pass ("path"):

"step"   one `ModelRunner.step`: a batch of single tokens (decoding, as captured steps where nothing else is in the batch),
         of prompts' portions, or of both, through a whole model of a named shape, to the logits of each request's last
         token; in float32 also the sampler.  Weights are random, drawn on the device.  Requests of the Qwen3 shapes that are
         decoding find random keys and values in the cache (a step's work does not depend on them); those of the other
         designs have had their context run through the model, so that their state is a real one.
"layer"  the sublayers of one repetition of a design's pattern, each on its own input, as a program that puts models
         together from parts calls them: `mixer.forward(x, batch, cache)` and `feed_forward.forward(x, batch)`.  Three
         designs choose experts by router logits that lie close together with random weights: two correct bfloat16 models
         choose differently for some tokens and their logits are then 13 % (4 layers) to 70 % (16 layers) apart, so a whole
         model says nothing about a change, and its layers do.

Sizes: the named shapes of `nano_vllm_amd.models.shapes`, the benchmark's batches and contexts (bench.py: 1, 8 and 64
requests with 4096 keys, 2048 prompt tokens), and the mixture of its 256-request workload (prompts of 100 to 1024 tokens
beside decoding requests, ragged).  Lengths are drawn from [from, to] by the case's own "lengths" number.
"""
from __future__ import annotations

import functools
import math
import random

import torch

from nano_vllm_amd.config import architecture_of
from nano_vllm_amd.engine.batch import StepEntry, build_batch
from nano_vllm_amd.engine.runner import ModelRunner
from nano_vllm_amd.kernels import HipKernels
from nano_vllm_amd.models.shapes import shape
from nano_vllm_amd.parts.model import Model, torch_dtype
from nano_vllm_amd.sampling.sampler import Sampler
from nano_vllm_amd.weights import fill_random_
from nano_vllm_amd.weights.loader import checkpoint_layout

DEVICE = "cuda:0"
PAGE = 256
LAYERS = {"qwen3-0.6b": 6, "qwen3-1.7b": 6, "qwen3-4b": 6, "qwen3-8b": 6, "nozurax-1b": 8, "bamipel-1b": 4, "pemuvik-1b": 16,
          "mafarax-1b": 1, "kirisun-1b": 2, "nemidra-1b": 2}
ROUTED = ("mafarax-1b", "kirisun-1b", "nemidra-1b")


def _case(path, model, dtype="bfloat16", decode=0, context=(0, 0), portions=0, tokens=(0, 0), behind=0, lengths=0):
    return {"path": path, "model": model, "layers": LAYERS[model], "dtype": dtype, "decode": decode, "context_from": context[0], "context_to": context[1],
            "portions": portions, "tokens_from": tokens[0], "tokens_to": tokens[1], "behind": behind, "lengths": lengths}


def listed():
    return [
        # one user of the smallest model, a short conversation: launches and latency count
        dict(_case("step", "qwen3-0.6b", decode=1, context=(600, 600)), name="decode_0.6b_b1"),
        # the benchmark's headline: eight requests of 4096 keys on the 8B shape, every weight read for eight rows
        dict(_case("step", "qwen3-8b", decode=8, context=(4095, 4095)), name="decode_8b_b8"),
        # a busy server of the same model: as many bytes of keys and values as of weights, twice over
        dict(_case("step", "qwen3-8b", decode=64, context=(4095, 4095)), name="decode_8b_b64"),
        # a new prompt alone: time to the first token
        dict(_case("step", "qwen3-8b", portions=1, tokens=(2048, 2048)), name="prefill_8b_2048"),
        # a step of a full server: ragged prompts, the last a portion behind 1500 cached tokens, beside ragged decoding requests
        dict(_case("step", "qwen3-8b", decode=40, context=(100, 2047), portions=10, tokens=(100, 1024), behind=1500, lengths=5),
             name="mixed_8b"),
        # the 32-bit path, that results are compared on: prompts, decoding and sampling in one step
        dict(_case("step", "qwen3-0.6b", dtype="float32", decode=7, context=(50, 1500), portions=3, tokens=(100, 600), lengths=3),
             name="float32_0.6b"),
        # prompts of a model whose every other layer keeps a state per request: retention in blocks
        dict(_case("step", "nozurax-1b", portions=6, tokens=(100, 1024), lengths=2), name="prompts_nozurax"),
        # decoding with three kinds of memory at once: latent rows, a delta rule's state, grouped keys
        dict(_case("step", "bamipel-1b", decode=8, context=(300, 900), lengths=1), name="decode_bamipel_b8"),
        # a prompt of a model with sigmoid-weighted and latent attention and experts beside dense layers
        dict(_case("step", "pemuvik-1b", portions=1, tokens=(2048, 2048)), name="prefill_pemuvik_2048"),
        # layers with experts and a state: a 2048-token prompt through attention beside a state-space layer,
        dict(_case("layer", "mafarax-1b", portions=1, tokens=(2048, 2048)), name="layer_mafarax_2048"),
        # ragged prompts through the channel-wise delta rule and a gated window attention,
        dict(_case("layer", "kirisun-1b", portions=3, tokens=(300, 1024), lengths=4), name="layers_kirisun_ragged"),
        # and decoding through a matrix memory beside a window attention and a gated linear attention
        dict(_case("layer", "nemidra-1b", decode=32, context=(100, 300), lengths=6), name="layers_nemidra_b32"),
    ]


def _log_between(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """Any of the paths, models and kinds of batch, sizes over their logarithm; never more work than the largest listed."""
    group = rng.choice(("qwen3", "qwen3", "qwen3", "float32", "state", "routed"))
    lengths = rng.randrange(1000)
    kind = rng.choice(("decode", "portions", "mixed"))
    if group == "qwen3":
        model = rng.choice(("qwen3-0.6b", "qwen3-1.7b", "qwen3-4b", "qwen3-8b"))
        most_decode, most_context, most_tokens = 64, 8192, 4096
    elif group == "float32":
        model, most_decode, most_context, most_tokens = "qwen3-0.6b", 16, 2048, 1024
    else:
        model = rng.choice(("nozurax-1b", "bamipel-1b", "pemuvik-1b") if group == "state" else ROUTED)
        most_decode, most_context, most_tokens = 32, 1024, 2048
    c = {"decode": 0, "portions": 0}
    if kind != "portions":
        c["decode"] = _log_between(rng, 1, most_decode)
        to = _log_between(rng, 40, max(41, min(most_context, (262144 if group in ("qwen3", "float32") else 8192) // c["decode"])))
        c["context"] = (to if rng.random() < 0.5 else max(32, to // 4), to)
    if kind != "decode":
        c["portions"] = rng.randint(1, 5)
        to = _log_between(rng, 20, max(21, most_tokens // c["portions"]))
        c["tokens"] = (to if rng.random() < 0.5 else max(17, to // 5), to)
    return _case("layer" if group == "routed" else "step", model, dtype="float32" if group == "float32" else "bfloat16",
                 lengths=lengths, **c)


# ---------------------------------------------------------------------------------------------------- preparation
def _lengths(case):
    """([keys each decoding request has before the step], [tokens of each portion], [tokens each portion finds in the cache])"""
    rng = random.Random(case["lengths"])
    contexts = [rng.randint(case["context_from"], case["context_to"]) for _ in range(case["decode"])]
    tokens = [rng.randint(case["tokens_from"], case["tokens_to"]) for _ in range(case["portions"])]
    behind = [0] * case["portions"]
    if behind:
        behind[-1] = case["behind"]
    return contexts, tokens, behind


def _config(case):
    config = shape(case["model"])
    config["torch_dtype"] = case["dtype"]
    if "layers" in config:
        config["layers"] = config["layers"][:case["layers"]]
    else:
        config["num_hidden_layers"] = case["layers"]
    return config


def _spec(case):
    arch = architecture_of(_config(case))
    return arch.build_spec(arch.parse_config(_config(case)))


def _realistic_rates(model):
    """Step sizes and decays as such layers are trained from (steps of 0.001 to 0.1, rates of 1 to 16, forget gates that mostly
    keep), where weights around zero would forget half of the state at every token."""
    for name, t in model.params.items():
        if name.endswith("dt_bias"):
            dt = torch.exp(torch.linspace(math.log(1e-3), math.log(0.1), t.numel(), device=t.device))
            t.copy_((dt + torch.log(-torch.expm1(-dt)))[torch.arange(t.numel(), device=t.device) * 7 % t.numel()])
        elif name.endswith("A_log"):
            t.copy_(torch.log(torch.linspace(1.0, 16.0, t.numel(), device=t.device)))
        elif name.endswith("right.gates.bias"):
            t[t.numel() // 2:] += torch.linspace(3.0, 6.0, t.numel() // 2, device=t.device)


def prepare(case, seed):
    dtype = torch_dtype(case["dtype"])
    kernels = HipKernels(DEVICE, dtype, quiet=True)
    model = Model(_spec(case), kernels, DEVICE, dtype)
    fill_random_(model, seed)
    _realistic_rates(model)
    contexts, tokens, behind = _lengths(case)
    starts, news = contexts + behind, [1] * len(contexts) + tokens
    pages = sum((s + n) // PAGE + 2 for s, n in zip(starts, news))
    runner = ModelRunner(model, PAGE, pages, len(starts), enable_prefix_caching=False)
    captured = case["path"] == "step" and not tokens
    if captured:            # as the engine does at start-up
        runner.enable_decode_graphs(len(contexts), max(contexts) + PAGE)
        runner.capture_decode_graphs()
    gen = torch.Generator().manual_seed(seed)
    ids = [torch.randint(0, model.spec.vocab_size, (s + n,), generator=gen).tolist() for s, n in zip(starts, news)]
    for i in range(len(starts)):
        runner.cache.admit(i)
        runner.cache.reserve(i, starts[i] + news[i])
    state = {"case": case, "seed": seed, "runner": runner, "ids": ids, "starts": starts, "news": news}
    state["entries"] = [StepEntry(i, ids[i][s:s + n], s, [n - 1]) for i, (s, n) in enumerate(zip(starts, news))]
    if case["path"] == "layer":
        state["inputs"] = inputs = _layer_inputs(case, seed, sum(s + n for s, n in zip(starts, news)), model)
        rows, at = [], 0
        for s, n in zip(starts, news):
            rows.append((at, s, n))
            at += s + n
        state["rows"] = rows
        if any(starts):     # what the requests had before, through the same sublayers
            before = [StepEntry(i, ids[i][:s], 0, ()) for i, s in enumerate(starts) if s]
            _layers(state, _batch(runner, before), [torch.cat([x[a:a + s] for a, s, _ in rows]) for x in inputs])
        state["batch"] = _batch(runner, state["entries"])
        state["x"] = [torch.cat([x[a + s:a + s + n] for a, s, n in rows]) for x in inputs]
    elif case["model"].startswith("qwen3"):
        if any(starts):
            cgen = torch.Generator(device=DEVICE).manual_seed(seed)
            for lc in runner.layer_caches:
                lc.k.normal_(0, 1, generator=cgen)
                lc.v.normal_(0, 1, generator=cgen)
    elif any(starts):
        runner.step([StepEntry(i, ids[i][:s], 0, ()) for i, s in enumerate(starts) if s])
    if case["dtype"] == "float32":
        state["sampler"] = Sampler(kernels, model.device)
    return state


def _layer_inputs(case, seed, rows, model):
    """What the norms hand to a mixer and to a feed-forward."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    return [torch.empty((rows, model.spec.hidden_size), dtype=model.dtype, device=DEVICE).normal_(0, 1, generator=gen) for _ in range(2)]


def _batch(runner, entries):
    return build_batch(entries, runner.cache, PAGE, runner.model.spec.vocab_size, runner.device, max_position=runner.model.spec.max_position,
                       extras=runner.kernels.batch_extras)


def _plain(y):
    """A sublayer may leave its last product to the norm that follows."""
    return y.tensor() if hasattr(y, "tensor") else y


def _layers(state, batch, inputs):
    runner = state["runner"]
    batch.step_cache = {}
    out = []
    for block, cache in zip(runner.model.blocks, runner.layer_caches):
        out.append({"mixer": _plain(block.mixer.forward(inputs[0], batch, cache)),
                    "feed_forward": _plain(block.feed_forward.forward(inputs[1], batch))})
    return out


def _states(runner):
    """The per-request states after the pass, as the cache holds them (its last row belongs to no request)."""
    return [{name: t[:-1] for name, t in lc.state.items() if t.is_floating_point()} for lc in runner.layer_caches if lc.state]


@torch.inference_mode()
def run(state):
    runner, case = state["runner"], state["case"]
    if case["path"] == "layer":
        return {"layers": _layers(state, state["batch"], state["x"]), "states": _states(runner)}
    logits = runner.step(state["entries"])
    out = {"logits": logits, "states": _states(runner)}
    last = [lc for lc in runner.layer_caches if lc.k is not None][-1]
    out["keys"], out["values"] = last.k, last.v         # the cache of the last layer that keeps keys: its new rows are results
    if case["dtype"] == "float32":
        n = logits.shape[0]
        out["tokens"] = state["sampler"].sample(logits, [0.0 if i % 2 else 0.6 for i in range(n)], [1] * n, list(range(n)),
                                                [s + m for s, m in zip(state["starts"], state["news"])])
    return out


# ---------------------------------------------------------------------------------------------------- work
@functools.lru_cache(maxsize=None)
def _sizes(model, dtype, layers):
    """(weights beside tables and experts, experts' weights, experts, experts a token runs, vocabulary, width)"""
    spec = _spec({"model": model, "dtype": dtype, "layers": layers})
    m = Model(spec, None, "cpu", torch_dtype(dtype))
    dense = routed = experts = top = 0
    for name, (owner, local, decl) in m.param_table.items():
        n = math.prod(decl.drawn_shape)
        if hasattr(owner, "experts") and local in ("up.weight", "down.weight"):
            routed, experts, top = routed + n, owner.experts, owner.top
        elif not name.startswith(("embed", "model.embed", "side_table", "head", "lm_head", "final")):
            dense += n
    return dense, routed, experts, top, spec.vocab_size, spec.hidden_size


def _memories(case):
    """[(kind, key-value numbers per token, multiply-adds per token and key or per token, keys in sight or None)] per layer"""
    config = _config(case)
    if case["model"].startswith("qwen3"):
        h, g, d = config["num_attention_heads"], config["num_key_value_heads"], config["head_dim"]
        return [("keys", 2 * g * d, 2 * h * d, None)] * config["num_hidden_layers"]
    out = []

    def add(m):
        if "left" in m:
            add(m["left"])
            add(m["right"])
        elif "kv_rank" in m:
            out.append(("keys", m["kv_rank"] + m["rot_dim"], m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), (m.get("mask") or {}).get("size")))
        elif "scale" in m:
            out.append(("keys", m["kv_heads"] * (m["dim"] + m["vdim"]), m["heads"] * (m["dim"] + m["vdim"]), (m.get("mask") or {}).get("size")))
        else:
            cells = m["heads"] * m.get("dim", m.get("state")) * m["vdim"]
            out.append(("state", cells, 2 * cells, None))
    for layer in config["layers"]:
        add(layer["mixer"])
    return out


def work(case):
    contexts, tokens, behind = _lengths(case)
    starts, news = contexts + behind, [1] * len(contexts) + tokens
    size = 4 if case["dtype"] == "float32" else 2
    dense, routed, experts, top, vocab, width = _sizes(case["model"], case["dtype"], case["layers"])
    total, rows = sum(news), len(news)
    hit = 1.0 - (1.0 - top / experts) ** total if experts else 0.0
    nbytes = size * (dense + routed * hit)
    flops = 2.0 * total * (dense + (routed * top / experts if experts else 0))
    for kind, numbers, macs, window in _memories(case):
        for s, n in zip(starts, news):
            if kind == "state":
                nbytes += 4 * numbers * (2 if s else 1)
                flops += 2.0 * macs * n
            else:
                seen = [min(p + 1, window or p + 1) for p in (s, s + n - 1)]
                nbytes += size * numbers * (min(s, window or s) + n)
                flops += 2.0 * macs * n * sum(seen) / 2
    if case["path"] == "layer":
        nbytes += size * 4 * total * width * case["layers"]
    else:
        nbytes += size * (width * total + vocab * width) + 4 * rows * vocab
        flops += 2.0 * rows * vocab * width
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Measured against exact(): logits and states of the bfloat16 models are 0.013 to 0.02 off (pemuvik-1b 0.004), single layers
    0.003 to 0.005, where another order of sums soon rounds everything else differently: the distance of two such results
    is up to 1.4 times that.  The float32 model is 4e-5 off, by its table of angles (float, as the reference has it); its
    sums in another order stay within 1e-6."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.0}
    if case["path"] == "layer":
        return {"rel": 0.015, "max": 0.5}
    return {"rel": 0.03, "max": 0.9}


# ---------------------------------------------------------------------------------------------------- in 64 bits
class _Weights:
    """A model's tensors under their checkpoint names, in 64 bits, made as they are asked for."""

    def __init__(self, model):
        self.model, self.layout = model, checkpoint_layout(model)

    def __call__(self, name):
        slot = self.layout[name]
        t = self.model.params[slot.param]
        return (t if slot.whole else t[slot.row:slot.row + slot.rows]).double()

    def has(self, name):
        return name in self.layout

    def product(self, x, name):
        y = x @ self(name).T
        return y + self(name + ".b") if self.has(name + ".b") else y


def _unit(x, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu_tanh(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _rotate(x, positions, rot, neighbours=False):
    """x [T, heads, dim], its first rot["dims"] channels turned: pairs (i, i + half), or neighbouring ones."""
    if not rot:
        return x
    n, scaling = rot["dims"], rot.get("scaling") or {}
    f = rot["base"] ** (-2.0 * torch.arange(n // 2, dtype=torch.float64, device=x.device) / n)
    if "low" in scaling:
        wave = 2 * math.pi / f
        s = ((scaling["original"] / wave - scaling["low"]) / (scaling["high"] - scaling["low"])).clamp(0, 1)
        f = (1 - s) * f / scaling["factor"] + s * f
    else:
        f = f / scaling.get("factor", 1.0)
    a = positions.double()[:, None] * f
    cos, sin = a.cos()[:, None], a.sin()[:, None]
    y = x.clone()
    first, second = (slice(0, n, 2), slice(1, n, 2)) if neighbours else (slice(0, n // 2), slice(n // 2, n))
    y[..., first] = x[..., first] * cos - x[..., second] * sin
    y[..., second] = x[..., second] * cos + x[..., first] * sin
    return y


def _attend(q, k, v, scale, start, window=None, keep=0, chunk=None, cap=None, sink=None, bias=None):
    """q [T, H, D] at positions start.., k [S, G, D] and v [S, G, DV] from position 0 -> [T, H, DV].  sink: a score per head that
    only the denominator knows; bias: sigmoid weights of score + bias per head instead of a softmax."""
    T, H, per = q.shape[0], q.shape[1], q.shape[1] // k.shape[1]
    i = torch.arange(start, start + T, device=q.device)[:, None]
    j = torch.arange(k.shape[0], device=q.device)[None]
    seen = j <= i
    if window:
        seen &= (i - j < window) | (j < keep)
    if chunk:
        seen &= i // chunk == j // chunk
    out = torch.empty((T, H, v.shape[2]), dtype=q.dtype, device=q.device)
    for h in range(H):
        s = q[:, h] @ k[:, h // per].T * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        if bias is not None:
            out[:, h] = torch.where(seen, torch.sigmoid(s + bias[h]), 0.0) @ v[:, h // per]
            continue
        s = s.masked_fill(~seen, -math.inf)
        if sink is not None:
            s = torch.cat((s, sink[h].expand(T, 1)), dim=1)
        out[:, h] = torch.softmax(s, dim=1)[:, :k.shape[0]] @ v[:, h // per]
    return out


def _convolve(x, taps, bias=None):
    """x [T, channels] with taps [channels, n], the last the token's own; nothing before the first token."""
    T, n = x.shape[0], taps.shape[1]
    padded = torch.cat((x.new_zeros(n - 1, x.shape[1]), x))
    y = sum(padded[j:j + T] * taps[:, j] for j in range(n))
    return y if bias is None else y + bias


def _delta(q, k, v, beta, decay, D):
    """q, k [T, H, D], v [T, H, DV], beta [T, H], decay [T, H, D or 1] -> outputs, state"""
    S = v.new_zeros(v.shape[1], D, v.shape[2])
    out = torch.empty_like(v)
    for t in range(v.shape[0]):
        S = S * decay[t][:, :, None]
        u = beta[t][:, None] * (v[t] - torch.matmul(k[t][:, None], S)[:, 0])
        S = torch.baddbmm(S, k[t][:, :, None], u[:, None])
        out[t] = torch.matmul(q[t][:, None], S)[:, 0]
    return out, S


def _linear_memory(q, k, v, decay):
    """The same without the correction: S <- decay S + k v^T, o = S^T q."""
    S = v.new_zeros(v.shape[1], q.shape[2], v.shape[2])
    out = torch.empty_like(v)
    for t in range(v.shape[0]):
        S = torch.baddbmm(S * decay[t][:, :, None], k[t][:, :, None], v[t][:, None])
        out[t] = torch.matmul(q[t][:, None], S)[:, 0]
    return out, S


def _expand(x, heads):
    return x.repeat_interleave(heads // x.shape[1], dim=1)


def _experts(x, w, p, mlp, scores, weights_of, unit):
    """The chosen experts' weighted sum: scores [T, n] choose, weights_of(chosen ids) weighs."""
    router = mlp["router"]
    groups = router.get("groups") or {}
    count, keep = groups.get("count", 1), groups.get("keep", 1)
    if count > 1:
        by = scores.view(x.shape[0], count, -1)
        best = by.topk(min(2, by.shape[2]), dim=2)[0].sum(2) if mlp.get("two_best") else by.max(2)[0]
        allowed = torch.zeros_like(best).scatter_(1, best.topk(keep, dim=1)[1], 1.0).bool()
        scores = scores.masked_fill(~allowed.repeat_interleave(by.shape[2], dim=1), -math.inf)
    ids = scores.topk(router["top"], dim=1)[1]
    weight = weights_of(ids)
    out = torch.zeros_like(x)
    for e in range(router["experts"] + router.get("identity", 0)):
        row, place = (ids == e).nonzero(as_tuple=True)
        if row.numel():
            y = x[row] if e >= router["experts"] else unit(x[row], f"{p}e{e}.")
            out.index_add_(0, row, y * weight[row, place][:, None])
    return out


class _Exact:
    """The designs' equations on one request's whole sequence; positions from 0."""

    def __init__(self, state):
        self.state, self.case = state, state["case"]
        self.config = _config(self.case)
        self.w = _Weights(state["runner"].model)
        self.eps = self.config["norm"]["eps"] if "norm" in self.config else self.config["rms_norm_eps"]

    # mixers: (h [T, width], mixer's configuration, prefix) -> (output, {name: state})
    def attention(self, h, m, p, options):
        w, T = self.w, h.shape[0]
        at = torch.arange(T, device=h.device)
        q, k, v = (w.product(h, p + n).view(T, -1, d) for n, d in (("q", m["dim"]), ("k", m["dim"]), ("v", m["vdim"])))
        if options.get("row_norm"):
            q = (_unit(q.flatten(1), self.eps) * w(p + "q.norm")).view_as(q)
            k = (_unit(k.flatten(1), self.eps) * w(p + "k.norm")).view_as(k)
        if options.get("head_norm"):
            q, k = _unit(q, self.eps) * w(p + "q.norm"), _unit(k, self.eps) * w(p + "k.norm")
        if m.get("q_temp"):
            q = q * (1 + m["q_temp"]["coef"] * torch.log((at.double() + 1).div(m["q_temp"]["every"]).floor() + 1))[:, None, None]
        pairs = options.get("neighbours", False)
        q, k = _rotate(q, at, m.get("rot"), pairs), _rotate(k, at, m.get("rot"), pairs)
        if options.get("unit_after"):
            q, k = _unit(q, self.eps), _unit(k, self.eps)
        if options.get("unit_values"):
            v = _unit(v, self.eps)
            if m.get("v_mix"):
                first = options["shared"].setdefault("first", v)
                if first is not v:
                    v = (1 - w(p + "vmix")) * v + w(p + "vmix") * first
        mask = m.get("mask") or {}
        o = _attend(q, k, v, m["scale"], 0, window=None if options.get("chunks") else mask.get("size"), keep=mask.get("keep_first", 0),
                    chunk=mask.get("size") if options.get("chunks") else None, cap=m.get("softcap"), sink=options.get("sink"),
                    bias=options.get("bias"))
        gate = options.get("gate")
        o = o * torch.sigmoid(h @ w(p + "g").T)[:, :, None] if gate == "head" else o
        o = o.flatten(1)
        o = o * torch.sigmoid(h @ w(p + "g").T) if gate == "channel" else o
        return w.product(o, p + "o"), {}

    def latent(self, h, m, p, sink=None, latent_queries=False, neighbours=False):
        w, T = self.w, h.shape[0]
        at = torch.arange(T, device=h.device)
        H, D, R, C = m["heads"], m["dim"], m["rot_dim"], m["kv_rank"]
        if latent_queries:
            q = (_unit(h @ w(p + "dq").T, self.eps) * w(p + "dq.norm")) @ w(p + "uq").T
        else:
            q = h @ w(p + "q").T
        q = q.view(T, H, D + R)
        low = h @ w(p + "dkv").T
        c = _unit(low[:, :C], self.eps) * w(p + "dkv.norm")
        turned = _rotate(low[:, None, C:], at, m["rot"], neighbours)
        q = torch.cat((q[..., :D], _rotate(q[..., D:], at, m["rot"], neighbours)), -1)
        k = torch.cat(((c @ w(p + "uk").T).view(T, H, D), turned.expand(T, H, R)), -1)
        o = _attend(q, k, (c @ w(p + "uv").T).view(T, H, m["vdim"]), m["scale"], 0, window=(m.get("mask") or {}).get("size"), sink=sink)
        if latent_queries:
            o = o * torch.sigmoid(h @ w(p + "g").T)[:, :, None]
        return o.flatten(1) @ w(p + "o").T, {}

    def retention(self, h, m, p):
        w, T = self.w, h.shape[0]
        at = torch.arange(T, device=h.device)
        q, k, v = ((h @ w(p + n).T).view(T, m["heads"], -1) for n in "qkv")
        q, k = _rotate(q, at, m.get("rot")), _rotate(k, at, m.get("rot")) * m["dim"] ** -0.5
        decay = torch.tensor(m["decay"], dtype=h.dtype, device=h.device)[None, :, None].expand(T, -1, 1)
        o, S = _linear_memory(q, k, v, decay)
        return (_unit(o, self.eps).flatten(1) * _silu(h @ w(p + "g").T)) @ w(p + "o").T, {"s": S}

    def delta(self, h, m, p, channel):
        w, T, H, D = self.w, h.shape[0], m["heads"], m["dim"]
        q, k, v = (_silu(_convolve(h @ w(p + n).T, w(p + n + ".conv"))) for n in "qkv")
        q, k = (_expand(x.view(T, -1, D), H) for x in (q, k))
        q, k = (x / torch.sqrt(x.square().sum(-1, keepdim=True) + 1e-6) for x in (q, k))
        beta = torch.sigmoid(h @ w(p + "b").T)
        z = (h @ w(p + "a1").T) @ w(p + "a2").T if channel else h @ w(p + "a").T
        decay = torch.exp(-torch.exp(w(p + "A_log"))[None, :, None] * torch.nn.functional.softplus(z + w(p + "dt_bias"), threshold=1e9).view(T, H, -1))
        o, S = _delta(q * D ** -0.5, k, v.view(T, H, -1), beta, decay, D)
        gate = torch.sigmoid((h @ w(p + "g1").T) @ w(p + "g2").T) if channel else _silu(h @ w(p + "g").T)
        return ((_unit(o, self.eps) * w(p + "norm")).flatten(1) * gate) @ w(p + "o").T, {"s": S}

    def state_space(self, h, m, p):
        w, T, H, P, N, G = self.w, h.shape[0], m["heads"], m["vdim"], m["state"], m["groups"]
        z, xbc, dt = (h @ w(p + "in").T).split((H * P, H * P + 2 * G * N, H), dim=1)
        xbc = _silu(_convolve(xbc, w(p + "conv"), w(p + "conv.b")))
        x = xbc[:, :H * P].view(T, H, P)
        B, C = (_expand(y.reshape(T, G, N), H) for y in xbc[:, H * P:].split(G * N, dim=1))
        dt = torch.nn.functional.softplus(dt + w(p + "dt_bias"), threshold=1e9)
        y, S = _linear_memory(C, B * dt[..., None], x, torch.exp(-torch.exp(w(p + "A_log")) * dt)[..., None])
        y = (y + w(p + "D")[:, None] * x).flatten(1) * _silu(z)
        y = _unit(y.view(T, m["norm_groups"], -1), self.eps).flatten(1) * w(p + "norm")
        return y @ w(p + "o").T, {"ssm": S}

    def matrix_memory(self, h, m, p):
        w, T, H, D, cap = self.w, h.shape[0], m["heads"], m["dim"], m["gate_cap"]
        q, k, v = ((h @ w(p + n).T).view(T, H, -1) for n in "qkv")
        q = q * D ** -0.5
        i, f = (cap * torch.tanh(w.product(h, p + n) / cap) for n in "if")
        f = torch.nn.functional.logsigmoid(f)
        S, n, top = v.new_zeros(H, D, v.shape[2]), v.new_zeros(H, D), v.new_zeros(H)
        o = torch.empty_like(v)
        for t in range(T):
            new = torch.maximum(f[t] + top, i[t])
            keep, write = torch.exp(f[t] + top - new), torch.exp(i[t] - new)
            S = torch.baddbmm(keep[:, None, None] * S, (write[:, None] * k[t])[:, :, None], v[t][:, None])
            n = keep[:, None] * n + write[:, None] * k[t]
            top = new
            o[t] = torch.matmul(q[t][:, None], S)[:, 0] / (torch.maximum((n * q[t]).sum(1).abs(), torch.exp(-top)) + 1e-6)[:, None]
        y = _unit(o, self.eps).flatten(1) * w(p + "norm") * torch.sigmoid(h @ w(p + "g").T)
        return y @ w(p + "o").T, {"s": S, "n": n, "m": top}

    def gated_linear(self, h, m, p):
        w, T, H, D = self.w, h.shape[0], m["heads"], m["dim"]
        q, k, v = ((h @ w(p + n).T).view(T, H, -1) for n in "qkv")
        z = (h @ w(p + "a1").T) @ w(p + "a2").T + w(p + "a2.b")
        o, S = _linear_memory(q * D ** -0.5, k, v, torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]).view(T, H, D))
        y = (_unit(o, self.eps) * w(p + "norm")).flatten(1) * _silu(h @ w(p + "g").T)
        return y @ w(p + "o").T, {"s": S}

    # feed-forwards
    def gated(self, x, p, act):
        w = self.w
        return (act(x @ w(p + "gate").T) * (x @ w(p + "up").T)) @ w(p + "down").T

    def plain(self, x, p, act):
        return act(x @ self.w(p + "up").T) @ self.w(p + "down").T

    def mixer(self, h, layer, p, shared):
        """One layer's mixer by the design's name and the layer's kind."""
        m, w, design = layer["mixer"], self.w, self.case["model"].split("-")[0]
        kind = layer["type"]
        if design == "nozurax":
            if kind == "retention":
                return self.retention(h, m, p)
            return self.attention(h, m, p, {"row_norm": True, "sink": w(p + "sink")})
        if design == "mafarax":
            a, _ = self.attention(h, m["left"], p + "left.", {"chunks": True})
            b, states = self.state_space(h, m["right"], p + "right.")
            return 0.5 * (_unit(a, self.eps) * w(p + "left.out") + _unit(b, self.eps) * w(p + "right.out")), states
        if design == "kirisun":
            if kind == "channel_delta":
                return self.delta(h, m, p, True)
            return self.attention(h, m, p, {"head_norm": True, "gate": "channel", "sink": h.new_zeros(m["heads"])})
        if design == "pemuvik":
            if kind == "latent_attention":
                return self.latent(h, m, p, sink=w(p + "sink"), neighbours=True)
            return self.attention(h, m, p, {"neighbours": True, "unit_values": True, "shared": shared, "bias": w(p + "pb")})
        if design == "bamipel":
            if kind == "latent_attention":
                return self.latent(h, m, p, latent_queries=True)
            if kind == "delta":
                return self.delta(h, m, p, False)
            return self.attention(h, m, p, {"unit_after": True, "gate": "head"})
        if kind == "gla":
            return self.gated_linear(h, m, p)
        a, _ = self.attention(h, m["left"], p + "left.", {})
        b, states = self.matrix_memory(h, m["right"], p + "right.")
        return m["left_scale"] * a + m["right_scale"] * b, states

    def feed_forward(self, x, layer, p):
        mlp, w, design = layer["mlp"], self.w, self.case["model"].split("-")[0]
        if mlp["kind"] == "dense":
            if design == "nozurax":
                return self.gated(x, p, torch.relu)
            if design == "bamipel":
                return self.plain(x, p, lambda z: torch.relu(z).square())
            if design == "pemuvik":
                return self.gated(x, p, _gelu_tanh)
            return self.plain(x, p, torch.nn.functional.gelu)
        z = w.product(x, p + "router")
        if design == "mafarax":
            relu2 = lambda t: torch.relu(t).square()
            s = torch.sigmoid(z)
            y = _experts(x, w, p, dict(mlp, two_best=True), s, lambda ids: mlp["router"]["scale"] * s.gather(1, ids), lambda t, q: self.plain(t, q, relu2))
            return y + self.plain(x, p + "shared.", relu2)
        unit = lambda t, q: self.gated(t, q, _silu)
        if design == "kirisun":
            return _experts(x, w, p, mlp, z, lambda ids: torch.softmax(z.gather(1, ids), 1), unit)
        s = torch.softmax(z, 1)
        if design == "pemuvik":
            def share(ids):
                c = s.gather(1, ids)
                return c / (c.sum(1, keepdim=True) + 1e-20)
            y = _experts(x, w, p, mlp, s + w(p + "correction"), share, unit)
        else:
            y = _experts(x, w, p, mlp, s, lambda ids: mlp["router"]["scale"] * s.gather(1, ids), unit)
        return y + torch.sigmoid(x @ w(p + "shared.sg").T) * unit(x, p + "shared.")

    # whole models on one request: (token ids, keys and values before them) -> logits of the last token, states per layer
    def design(self, ids):
        w, eps, design = self.w, self.eps, self.case["model"].split("-")[0]
        r = w("embed")[torch.tensor(ids, device=DEVICE)]
        shared, states = {}, []
        for i, layer in enumerate(self.config["layers"]):
            p = f"l{i}."
            if design == "nozurax":
                h = _unit(r, eps) * (1 + w(p + "norm1"))
                y, s = self.mixer(h, layer, p + "mix.", shared)
                r = r + y + self.feed_forward(h, layer, p + "mlp.")
            elif design == "pemuvik":
                y, s = self.mixer(_unit(r, eps) * w(p + "norm1"), layer, p + "mix.", shared)
                r = r + y * w(p + "ls1") + self.feed_forward(_unit(r, eps) * w(p + "norm2"), layer, p + "mlp.") * w(p + "ls2")
            else:
                y, s = self.mixer(_unit(r, eps) * w(p + "norm1"), layer, p + "mix.", shared)
                r = r + _unit(y, eps) * w(p + "norm1b")
                r = r + _unit(self.feed_forward(_unit(r, eps) * w(p + "norm2"), layer, p + "mlp."), eps) * w(p + "norm2b")
            states.append(s)
        r = _unit(r[-1:], eps) * ((1 if design == "nozurax" else 0) + w("final.norm"))
        return r @ w("embed" if design == "pemuvik" else "head").T, states

    def qwen3(self):
        """Every request's last logits; the layers' weights are made once for all requests."""
        w, eps, c, s = self.w, self.eps, self.config, self.state
        runner, H, G, D = s["runner"], c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"]
        spans, at = [], 0
        for n in s["news"]:
            spans.append(slice(at, at + n))
            at += n
        ids = torch.tensor([t for x, start in zip(s["ids"], s["starts"]) for t in x[start:]], device=DEVICE)
        positions = torch.cat([torch.arange(start, start + n, device=DEVICE) for start, n in zip(s["starts"], s["news"])])
        rot = {"dims": D, "base": c["rope_theta"]}
        embed = w("model.embed_tokens.weight")
        r = embed[ids]
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = _unit(r, eps) * w(p + "input_layernorm.weight")
            q, k, v = ((h @ w(p + f"self_attn.{n}_proj.weight").T).view(at, -1, D) for n in "qkv")
            q = _rotate(_unit(q, eps) * w(p + "self_attn.q_norm.weight"), positions, rot)
            k = _rotate(_unit(k, eps) * w(p + "self_attn.k_norm.weight"), positions, rot)
            o = torch.empty((at, H, D), dtype=r.dtype, device=DEVICE)
            for n, (span, start) in enumerate(zip(spans, s["starts"])):
                kn, vn = k[span], v[span]
                if start:
                    table = torch.tensor(runner.cache.requests[n].tables[0], device=DEVICE)[:(start + PAGE - 1) // PAGE]
                    kc, vc = runner.layer_caches[i].k[table], runner.layer_caches[i].v[table]
                    kc = kc.transpose(1, 2).reshape(-1, G, D)[:start]
                    vc = vc.permute(0, 2, 4, 1, 3).reshape(-1, G, D)[:start]
                    kn, vn = torch.cat((kc.double(), kn)), torch.cat((vc.double(), vn))
                o[span] = self.grouped(q[span], kn, vn, start)
            r = r + o.flatten(1) @ w(p + "self_attn.o_proj.weight").T
            h = _unit(r, eps) * w(p + "post_attention_layernorm.weight")
            r = r + (_silu(h @ w(p + "mlp.gate_proj.weight").T) * (h @ w(p + "mlp.up_proj.weight").T)) @ w(p + "mlp.down_proj.weight").T
        last = torch.tensor([span.stop - 1 for span in spans], device=DEVICE)
        x = _unit(r[last], eps) * w("model.norm.weight")
        return x @ (embed if c["tie_word_embeddings"] else w("lm_head.weight")).T

    @staticmethod
    def grouped(q, k, v, start):
        T, H, D = q.shape
        if T > 1:
            return _attend(q, k, v, D ** -0.5, start)
        s = torch.softmax(torch.matmul(q[0].view(k.shape[1], -1, D), k.permute(1, 2, 0)) * D ** -0.5, -1)
        return torch.matmul(s, v.transpose(0, 1)).reshape(1, H, D)


def _by_slot(state, per_request, like):
    """[{name: [requests] states}] per layer as the cache lays them out; nothing for what has no value of its own."""
    runner, out = state["runner"], []
    layers = [i for i, lc in enumerate(runner.layer_caches) if lc.state]
    for n, i in enumerate(layers):
        entry = {}
        for name, t in like[n].items():
            if i < len(per_request[0]) and name in per_request[0][i]:
                full = t.double()
                for request, states in enumerate(per_request):
                    full[runner.cache.requests[request].state_slot] = states[i][name]
                entry[name] = full
            else:
                entry[name] = None
        out.append(entry)
    return out


@torch.inference_mode()
def exact(case, seed):
    state = prepare(case, seed)
    e = _Exact(state)
    out = {"keys": None, "values": None, "tokens": None}
    if case["model"].startswith("qwen3"):
        return dict(out, logits=e.qwen3(), states=[])
    like = _states(state["runner"])
    if case["path"] == "step":
        logits, states = zip(*(e.design(ids) for ids in state["ids"]))
        return dict(out, logits=torch.cat(logits), states=_by_slot(state, states, like))
    layers, states = [], [[] for _ in state["ids"]]
    for i, layer in enumerate(e.config["layers"]):
        # a step's rows: single tokens first, each request's rows together, as the inputs were laid out
        mixed, x = [], state["inputs"][0].double()
        for request, (a, s, n) in enumerate(state["rows"]):
            y, after = e.mixer(x[a:a + s + n], layer, f"l{i}.mix.", {})
            mixed.append(y[s:])
            states[request].append(after)
        layers.append({"mixer": torch.cat(mixed), "feed_forward": e.feed_forward(state["x"][1].double(), layer, f"l{i}.mlp.")})
    return {"layers": layers, "states": _by_slot(state, states, like)}
