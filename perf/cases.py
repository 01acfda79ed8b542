"""What the engine is timed on: steps of its decoders through ``ModelRunner.step``, the step function below every entry
point (the generation loop, the command line and the trace replay all call it).

A case is one step, with the requests in it as a running engine holds them:

* ``design`` and ``size``: the decoder and its layer sizes.  ``qwen2`` has the published Qwen2.5 sizes with all layers; the
  other decoders have the two sizes that ``bench.py --design`` measures them at.
* ``dtype``: ``bfloat16``, or ``float32``, the option for runs that are compared with other implementations.
* ``portions`` x ``portion`` tokens: prompts, or portions of prompts that already have up to ``behind`` positions in the
  cache.  ``singles``: requests that decode one token each at a context of up to ``context`` positions.  ``ragged``: the
  requests have different lengths (portions down to two thirds, contexts down to a quarter).

A step of single tokens only is replayed as a captured graph, as the engine runs it; its passes go through the last
``CYCLE`` positions of the context in turn.  Every other step is launched eagerly.  What comes back are the logits of each
request's last token.
"""
import math
import zlib

import torch

import vipera_rs_amd  # noqa: F401  (makes the package importable by name)
from vipera_rs_amd.config import config_from_dict
from vipera_rs_amd.engine.batch import StepEntry
from vipera_rs_amd.engine.runner import ModelRunner
from vipera_rs_amd.models import build_model
from vipera_rs_amd.models.decoder import declare_cache_needs, declare_model, tensor_reads
from vipera_rs_amd.runtime import Runtime

DEVICE = "cuda:0"
CYCLE = 8            # positions that the passes of a decode step go through in turn
BLOCK = 16           # positions of a cache page
PORTION = 1024       # tokens of a request per step while the cache is filled
FILL_TOKENS = 16384  # tokens per step while the cache is filled


# --- the cases ------------------------------------------------------------------------------------------------
def case(design, size, dtype="bfloat16", portions=0, portion=0, behind=0, singles=0, context=0, ragged=False, name=None):
    c = dict(design=design, size=size, dtype=dtype, portions=portions, portion=portion, behind=behind, singles=singles,
             context=context, ragged=ragged)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one user's chat with a small model: latency and launches
        case("qwen2", "0.5b", singles=1, context=512, name="qwen2_0.5b_decode_1"),
        # the headline of bench.py: eight requests decoding at 4,096 positions
        case("qwen2", "7b", singles=8, context=4096, name="qwen2_7b_decode_8"),
        # a full serving batch of requests of different lengths
        case("qwen2", "1.5b", singles=64, context=2048, ragged=True, name="qwen2_1.5b_decode_64_ragged"),
        # the headline prompt of bench.py
        case("qwen2", "7b", portions=1, portion=2048, name="qwen2_7b_prefill_2048"),
        # a step of continuous batching: portions of prompts, some deep in theirs, beside decoding requests
        case("qwen2", "1.5b", portions=3, portion=512, behind=3584, singles=29, context=2048, ragged=True,
             name="qwen2_1.5b_mixed"),
        # the 32-bit option: a short prompt, for comparison with another implementation
        case("qwen2", "0.5b", "float32", portions=1, portion=333, name="qwen2_0.5b_float32_prompt"),
        # the other decoders, each at one of the steps that serving it consists of
        case("gilidra", "m", portions=1, portion=2048, name="gilidra_m_prefill_2048"),
        case("zulesun", "m", portions=2, portion=1000, ragged=True, name="zulesun_m_prefill_ragged"),
        case("muzasun", "m", singles=8, context=4096, name="muzasun_m_decode_8"),
        case("lurirax", "m", portions=3, portion=512, behind=1536, singles=16, context=1024, ragged=True,
             name="lurirax_m_mixed"),
        case("zeladra", "m", singles=64, context=1024, ragged=True, name="zeladra_m_decode_64_ragged"),
        case("rebidra", "m", portions=1, portion=512, behind=1536, name="rebidra_m_portion_512"),
    ]


def draw(rng):
    def log_int(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    design = rng.choice(["qwen2"] * 6 + ["gilidra", "zulesun", "muzasun", "lurirax", "zeladra", "rebidra"])
    size = rng.choice(["0.5b", "1.5b", "3b", "7b"]) if design == "qwen2" else rng.choice(["s", "m"])
    large = size == "7b"
    if design == "qwen2" and size in ("0.5b", "1.5b") and rng.random() < 0.2:
        if rng.random() < 0.5:
            return case(design, size, "float32", singles=log_int(1, 16), context=decode_context(log_int(100, 1500)))
        return case(design, size, "float32", portions=1, portion=log_int(17, 400))
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "mixed"])
    if kind == "decode":
        singles = log_int(1, 16 if large else 96)
        context = decode_context(log_int(200, 4096 if large else 2048 if singles < 48 else 1024))
        return case(design, size, singles=singles, context=context, ragged=rng.random() < 0.5)
    if kind == "prefill":
        portions = rng.randint(1, 3)
        portion = log_int(65, 2000 // portions)
        return case(design, size, portions=portions, portion=portion,
                    behind=rng.choice([0, log_int(100, 2000)]), ragged=portions > 1)
    return case(design, size, portions=rng.randint(1, 3), portion=log_int(65, 512), behind=log_int(100, 3000),
                singles=log_int(1, 32), context=log_int(200, 2048), ragged=True)


def decode_context(context):
    """``context``, or a little more: the positions that a decode step's passes go through lie in one bucket of captured steps."""
    bucket = 256
    while bucket < context:
        bucket *= 2
    return max(context, bucket // 2 + CYCLE) if bucket > 256 else context


def shares(c):
    """Per request of the step (positions already in the cache, tokens of this step)."""
    out = []
    for k in range(c["portions"]):
        cut = c["portion"] * k // (3 * c["portions"]) if c["ragged"] else 0
        out.append((c["behind"] * (k + 1) // c["portions"], max(2, c["portion"] - cut)))
    last = CYCLE if c["portions"] == 0 else 1
    for k in range(c["singles"]):
        cut = c["context"] * 3 * k // (4 * c["singles"]) if c["ragged"] else 0
        out.append((max(1, c["context"] - cut - last), 1))
    return out


# --- configurations --------------------------------------------------------------------------------------------
QWEN2 = {
    "architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2", "rope_theta": 1000000.0, "rms_norm_eps": 1e-6,
    "max_position_embeddings": 32768, "hidden_act": "silu", "use_sliding_window": False, "sliding_window": 131072,
    "torch_dtype": "bfloat16",
}
# layers, width, heads, key heads, feed-forward, vocabulary, output matrix tied to the embedding
QWEN2_SIZES = {"0.5b": (24, 896, 14, 2, 4864, 151936, True), "1.5b": (28, 1536, 12, 2, 8960, 151936, True),
               "3b": (36, 2048, 16, 2, 11008, 151936, True), "7b": (28, 3584, 28, 4, 18944, 152064, False)}
# width, vocabulary, heads, experts, an expert's width, window; heads of 128, ten layers, top 4
OTHER_SIZES = {"s": (1024, 32768, 8, 16, 512, 1024), "m": (2048, 65536, 16, 32, 1024, 2048)}
LAYERS, DIM, TOP = 10, 128, 4


def configuration(c):
    if c["design"] == "qwen2":
        layers, width, heads, groups, ff, vocab, tied = QWEN2_SIZES[c["size"]]
        return dict(QWEN2, num_hidden_layers=layers, hidden_size=width, num_attention_heads=heads,
                    num_key_value_heads=groups, intermediate_size=ff, vocab_size=vocab, tie_word_embeddings=tied,
                    max_window_layers=layers)
    width, vocab, heads, experts, ff, window = OTHER_SIZES[c["size"]]
    groups, scale = heads // 4, DIM ** -0.5
    dense = {"kind": "dense", "ff": TOP * ff}
    moe = {"kind": "moe", "expert": {"ff": ff}, "router": {"experts": experts, "top": TOP}}
    shared = dict(moe, shared={"ff": ff})
    decay = [1.0 - 2.0 ** (-1.0 - 7.0 * h / (heads - 1)) for h in range(heads)]
    base = {"heads": heads, "kv_heads": groups, "dim": DIM, "vdim": DIM, "scale": scale}
    latent = {"heads": heads, "dim": DIM, "rot_dim": 64, "vdim": DIM, "q_rank": 48 * heads, "kv_rank": 192,
              "rot": {"base": 1e6, "dims": 64}, "scale": (DIM + 64) ** -0.5}
    yarn = {"factor": 8.0, "fast": 32.0, "slow": 1.0, "original": 8192}
    model = {"vocab": vocab, "width": width}
    if c["design"] == "gilidra":
        clamped = dict(moe, expert={"ff": ff, "limit": 7.0})
        latent["mask"] = {"size": window}
        kinds = [("latent_attention", latent, clamped),
                 ("delta", {"heads": heads, "kv_heads": heads // 2, "dim": 128, "vdim": 128, "conv": 4}, clamped),
                 ("wkv", {"heads": 2 * heads, "dim": 64, "decay_rank": 64}, clamped),
                 ("latent_attention", latent, clamped),
                 ("delta", {"heads": heads, "kv_heads": heads // 2, "dim": 128, "vdim": 128, "conv": 4}, clamped)]
        model.update(architecture="Gilidra", norm={"eps": 1e-5}, logit_scale=1.0)
    elif c["design"] == "zulesun":
        grouped = dict(moe, router={"experts": experts, "top": TOP, "groups": {"count": 4, "keep": 2}})
        lightning = {"heads": heads, "dim": DIM, "vdim": DIM, "decay": decay}
        pair = {"left": dict(base, mask={"size": window}, softcap=30.0,
                             rot={"base": 1e6, "dims": 64, "scaling": {"factor": 8.0}}),
                "left_scale": 1.0, "right_scale": 1.0,
                "right": {"inner": 2 * width, "state": 16, "dt_rank": width // 16, "conv": 4}}
        kinds = [("lightning", lightning, grouped), ("parallel", pair, grouped), ("parallel", pair, grouped),
                 ("lightning", lightning, grouped), ("parallel", pair, grouped)]
        model.update(architecture="Zulesun", norm={"eps": 1e-5}, embedding={"scale": width ** 0.5}, token_side={"dim": 64})
    elif c["design"] == "muzasun":
        attention = dict(base, rot={"base": 1e6, "dims": 64}, v_mix=True)
        memory = {"heads": heads, "dim": DIM, "vdim": DIM, "gate_cap": 15.0}
        delta = {"heads": heads, "kv_heads": heads // 2, "dim": 128, "vdim": 128, "conv": 4, "decay_rank": 64, "gate_rank": 64}
        kinds = [("attention", attention, dense), ("mlstm", memory, shared), ("mlstm", memory, shared),
                 ("channel_delta", delta, shared), ("attention", attention, dense)]
        model.update(architecture="Muzasun", norm={"eps": 1e-6}, residual_mult=0.5, logit_scale=0.5)
    elif c["design"] == "lurirax":
        scaled = dict(shared, router={"experts": experts, "top": TOP, "scale": 2.0})
        near = dict(base, mask={"size": window}, rot={"base": 1e6, "dims": 64, "scaling": {
            "factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}})
        two = dict(base, dim=64, diff=0.3, mask={"size": window, "keep_first": 64}, scale=64 ** -0.5)
        pair = {"left": dict(base, mask={"size": window}, bias_max=window, bias_rows=32),
                "left_scale": 0.5, "right_scale": 1.0,
                "right": {"heads": heads, "dim": DIM, "vdim": DIM, "rot": {"base": 1e6, "dims": DIM}, "decay": decay}}
        kinds = [("attention_2", two, dense), ("attention", near, scaled), ("attention", near, scaled),
                 ("parallel", pair, scaled), ("attention", near, scaled)]
        model.update(architecture="Lurirax", norm={"eps": 1e-6}, embedding={"scale": 1.0})
    elif c["design"] == "zeladra":
        latent["rot"] = dict(latent["rot"], scaling=yarn)
        near = dict(base, mask={"size": window, "keep_first": 64}, rot={"base": 1e6, "dims": 64})
        space = {"heads": width // 32, "vdim": 64, "state": 128, "groups": 8, "norm_groups": 8, "conv": 4}
        kinds = [("latent_attention", latent, dense), ("mamba2", space, None), ("attention", near, dense),
                 ("latent_attention", latent, dense), ("mamba2", space, None)]
        model.update(architecture="Zeladra", norm={"eps": 1e-5}, streams=4, embedding={"scale": 1.0})
    else:
        near = dict(base, conv=4, mask={"size": window}, rot={"base": 1e6, "dims": DIM, "scaling": yarn})
        kinds = [("attention", near, shared)]
        model.update(architecture="Rebidra", norm={"eps": 1e-5}, logit_scale=0.5, embedding={"scale": 1.0},
                     token_side={"dim": 64}, loop={"start": 2, "stop": 5, "times": 2})
    layers = []
    for index in range(LAYERS - 3 if c["design"] == "rebidra" else LAYERS):
        kind, mixer, mlp = kinds[index % len(kinds)]
        if kind == "latent_attention" and index % 5 == 3:
            mixer = dict(mixer, kv_from=index - 3)       # reads the cache of the latent layer three before it
        if c["design"] == "zulesun" and index == 0:
            mlp = dense
        layers.append({"type": kind, "mixer": mixer, "mlp": mlp})
    return dict(model, layers=layers)


# --- inputs ----------------------------------------------------------------------------------------------------
def _generator(seed, name):
    return torch.Generator(DEVICE).manual_seed((seed * 1000003 + zlib.crc32(name.encode())) & 0x7FFFFFFF)


def weights(c, seed):
    """The weights by name, as a model's folder holds them: matrices in the run's dtype, vectors in 32-bit; normal values of
    the width that each tensor is declared with, and where trained models differ from that by much, what they have: rates
    of forgetting spread over tens to thousands of tokens, routers that are sure of their first choices, outputs of
    sublayers that are small beside the stream, streams that are mostly passed on."""
    matrix = getattr(torch, c["dtype"])
    softmax_router = c["design"] in ("gilidra", "zulesun", "rebidra")
    out = {}
    for spec in declare_model(config_from_dict(configuration(c))):
        if spec.optional:
            continue
        g, leaf = _generator(seed, spec.name), spec.name.rsplit(".mix.", 1)[-1].replace("right.", "")
        end = spec.name.split(".", 1)[-1]
        if spec.role == "matrix":
            std = spec.std
            if end == "mlp.router" and softmax_router:
                std = 0.1
            elif end == "embed" and c["design"] in ("lurirax", "zeladra", "rebidra"):
                std = 1.0
            t = torch.randn(spec.shape, generator=g, device=DEVICE, dtype=matrix) * std
        elif leaf in ("dt_bias", "dt.b"):      # softplus(bias) between 0.001 and 0.1
            step = torch.exp(torch.rand(spec.shape, generator=g, device=DEVICE) * math.log(100.0) + math.log(1e-3))
            t = step + torch.log(-torch.expm1(-step))
        elif leaf == "A_log":                  # rates between 1 and 16
            t = torch.log1p(15.0 * torch.rand(spec.shape, generator=g, device=DEVICE))
        elif leaf == "w0":                     # decays exp(-exp(w0)) between 0.55 and 0.998
            t = -6.0 + 5.5 * torch.rand(spec.shape, generator=g, device=DEVICE)
        elif leaf == "f.b":                    # forget gates between sigmoid(3) and sigmoid(6)
            t = 3.0 + 3.0 * torch.rand(spec.shape, generator=g, device=DEVICE)
        else:
            t = torch.randn(spec.shape, generator=g, device=DEVICE) * spec.std
            if spec.init == "one_plus_normal":
                t = t + 1.0
            if end in ("norm1b", "norm2b"):    # gains of 1 + w behind a sublayer
                t = t - 0.85
            elif end == "side.norm" or (c["design"] == "lurirax" and end in ("norm1", "norm2")):
                t = t * 0.1
            elif end in ("hc1.mix", "hc2.mix"):
                t = 0.1 * t + torch.eye(spec.shape[0], device=DEVICE)
            elif end in ("hc1.in", "hc2.in"):
                t = t / spec.shape[0]
        out[spec.name] = t
    return out


def token_lists(c, seed):
    """Per request all its tokens: those in the cache and those of the step (and of the passes after it)."""
    vocab = config_from_dict(configuration(c)).vocab_size
    g = torch.Generator().manual_seed(seed)
    return [torch.randint(0, vocab, (start + count + CYCLE,), generator=g).tolist() for start, count in shares(c)]


class State:
    def __init__(self, runner, turns):
        self.runner, self.turns, self.at = runner, turns, 0


def prepare(c, seed):
    """A loaded model, its cache holding the earlier tokens of every request, and the entries of the step."""
    steps, lists = shares(c), token_lists(c, seed)
    runtime = Runtime(DEVICE, c["dtype"])
    model = build_model(config_from_dict(configuration(c)), runtime)
    model.load(weights(c, seed))
    reach = [start + count + (CYCLE if c["portions"] == 0 else 0) for start, count in steps]
    pages = sum((n + BLOCK - 1) // BLOCK for n in reach) + 8
    runner = ModelRunner(model, runtime, BLOCK, pages, len(steps) + 1, use_graphs=True, max_context=max(max(reach), 256))
    for r, n in enumerate(reach):
        runner.cache.reserve(r, 0, n)
    # a decode step is captured on its first run: the position before the timed ones
    known = [start - (1 if c["portions"] == 0 else 0) for start, _ in steps]
    done = [0] * len(steps)
    while any(d < k for d, k in zip(done, known)):
        entries, room = [], FILL_TOKENS
        for r, k in enumerate(known):
            n = min(PORTION, k - done[r], room)
            if n > 0:
                entries.append(StepEntry(r, done[r], lists[r][done[r]:done[r] + n], []))
                done[r] += n
                room -= n
        runner.run(runner.prepare(entries))
    if c["portions"] == 0:
        if any(known):
            runner.step([StepEntry(r, k, [lists[r][k]], [0]) for r, k in enumerate(known)])
        turns = [[StepEntry(r, start + j, [lists[r][start + j]], [0]) for r, (start, _) in enumerate(steps)]
                 for j in range(CYCLE)]
    else:
        turns = [[StepEntry(r, start, lists[r][start:start + n], [n - 1]) for r, (start, n) in enumerate(steps)]]
    return State(runner, turns)


def run(state):
    entries = state.turns[state.at]
    state.at = (state.at + 1) % len(state.turns)
    return state.runner.step(entries)


# --- what a pass cannot do without ------------------------------------------------------------------------------
def work(c):
    config = config_from_dict(configuration(c))
    steps, element = shares(c), 4 if c["dtype"] == "float32" else 2
    tokens, rows = sum(n for _, n in steps), len(steps)
    reads, nbytes, flops = tensor_reads(config), 0.0, 0.0
    specs = [s for s in declare_model(config) if not s.optional]
    tied = not any(s.name in ("head", "lm_head.weight") for s in specs)
    for s in specs:
        size = float(math.prod(s.shape))
        width = element if s.role == "matrix" else 4
        if s.name in ("embed", "side.embed", "model.embed_tokens.weight"):
            nbytes += tokens * s.shape[1] * element
            if not (tied and s.name != "side.embed"):
                continue
        if s.name in ("head", "lm_head.weight", "model.embed_tokens.weight"):
            nbytes, flops = nbytes + size * width, flops + 2.0 * rows * size
            continue
        reached, share = 1.0, 1.0
        if ".mlp.e" in s.name:       # an expert: the share of tokens that choose it, and of experts that any token chooses
            share = TOP / OTHER_SIZES[c["size"]][3]
            reached = 1.0 - (1.0 - share) ** tokens
        nbytes += reached * size * width
        if s.role == "matrix":
            flops += 2.0 * tokens * share * size * reads.get(s.name, 1)
    mixers = [layer.mixer for layer in config.layer_specs()]
    for entry, need in zip(config.schedule(), declare_cache_needs(config)):
        if need.kv is not None:
            kv = need.kv
            window = int(kv.window or 0)
            position = element * kv.kv_heads * (kv.head_dim + (kv.value_dim or kv.head_dim))
            heads = int(mixers[entry.layer].get("heads") or (mixers[entry.layer].get("left") or {}).get("heads") or 1) \
                if isinstance(mixers[entry.layer].params, dict) else 1
            for start, n in steps:
                seen = min(start + n, window + n) if window else start + n
                nbytes += seen * position
                flops += 4.0 * heads * DIM * sum(min(p + 1, window) if window else p + 1 for p in range(start, start + n))
        if need.state is not None:
            nbytes += 2.0 * rows * 4 * math.prod(need.state.shape)
    return {"bytes": nbytes + rows * config.vocab_size * 4, "flops": flops}


def tolerance(c):
    # logits of a whole model whose activations are rounded to 16 bits between the products; a mixture of experts adds
    # close calls of its router, which rounding decides
    if c["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 0.03, "max": 0.3}


# --- the same in 64 bits ----------------------------------------------------------------------------------------
def exact(c, seed):
    """Logits ``[requests, vocab]`` in float64, whole sequences from their first token on."""
    steps, lists = shares(c), token_lists(c, seed)
    config, cfg = config_from_dict(configuration(c)), configuration(c)
    lengths = [start + count for start, count in steps]
    active = sum(math.prod(s.shape) * (TOP / OTHER_SIZES[c["size"]][3] if ".mlp.e" in s.name else 1.0)
                 for s in declare_model(config) if s.role == "matrix" and not s.optional and "embed" not in s.name)
    if 2.0 * sum(lengths) * active > 3e14:      # over about 20 seconds
        return None
    stored = weights(c, seed)
    out = [None] * len(steps)
    order = sorted(range(len(steps)), key=lambda r: -lengths[r])
    per = max(1, 32768 // max(lengths))
    for at in range(0, len(order), per):
        group = order[at:at + per]
        longest = max(lengths[r] for r in group)
        ids = torch.zeros(len(group), longest, dtype=torch.long, device=DEVICE)
        for row, r in enumerate(group):
            ids[row, :lengths[r]] = torch.tensor(lists[r][:lengths[r]], device=DEVICE)
        last = torch.tensor([lengths[r] - 1 for r in group], device=DEVICE)
        logits = Reference(cfg, stored, ids, last).logits()
        for row, r in enumerate(group):
            out[r] = logits[row]
    return torch.stack(out)


def silu(z):
    return z * torch.sigmoid(z)


def gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def softplus(z):
    return torch.logaddexp(z, torch.zeros_like(z))


def over_rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def layer_norm(x, eps):
    return over_rms(x - x.mean(-1, keepdim=True), eps)


def convolve(x, taps):
    """Causal over time, per channel: x [B, T, channels], taps [channels, n], the last tap the current token's."""
    n = taps.shape[1]
    y = taps[:, n - 1] * x
    for back in range(1, min(n, x.shape[1])):
        y[:, back:] += taps[:, n - 1 - back] * x[:, :-back]
    return y


def frequencies(rot):
    dims, base = int(rot["dims"]), float(rot["base"])
    f = base ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64, device=DEVICE) / dims)
    s = rot.get("scaling")
    if not s:
        return f
    factor = float(s["factor"])
    if "fast" in s:      # YaRN
        low, high = (dims * math.log(s["original"] / (2.0 * math.pi * s[k])) / (2.0 * math.log(base)) for k in ("fast", "slow"))
        low, high = max(math.floor(low), 0), min(math.ceil(high), dims - 1)
        share = ((torch.arange(dims // 2, device=DEVICE).double() - low) / max(high - low, 0.001)).clamp(0.0, 1.0)
        return f / factor * share + f * (1.0 - share)
    if "low" in s:       # long waves stretched
        turns = s["original"] * f / (2.0 * math.pi)
        share = ((turns - s["low"]) / (s["high"] - s["low"])).clamp(0.0, 1.0)
        return (1.0 - share) * f / factor + share * f
    return f / factor


def rotate(x, rot, pairs="halves"):
    """x [B, T, heads, dim]: pairs of the first ``dims`` numbers of a head turn by position times frequency."""
    if not rot:
        return x
    dims = int(rot["dims"])
    amplitude = 0.1 * math.log(float(rot["scaling"]["factor"])) + 1.0 if "fast" in (rot.get("scaling") or {}) else 1.0
    angle = torch.arange(x.shape[1], device=DEVICE).double()[:, None, None] * frequencies(rot)
    cos, sin = amplitude * torch.cos(angle), amplitude * torch.sin(angle)
    one, two = (x[..., :dims // 2], x[..., dims // 2:dims]) if pairs == "halves" else (x[..., 0:dims:2], x[..., 1:dims:2])
    a, b = one * cos - two * sin, two * cos + one * sin
    turned = torch.cat([a, b], -1) if pairs == "halves" else torch.stack([a, b], -1).flatten(-2)
    return torch.cat([turned, x[..., dims:]], -1)


def attend(q, k, v, scale, mask=None, chunks=False, sink=None, bias=None, cap=0.0):
    """q [B, T, H, d], k [B, T, G, d], v [B, T, G, dv] -> [B, T, H * dv]; ``bias`` [T, H] by distance."""
    B, T, H, _ = q.shape
    group, size, keep = H // k.shape[2], int((mask or {}).get("size") or 0), int((mask or {}).get("keep_first") or 0)
    i, j = torch.arange(T, device=DEVICE)[:, None], torch.arange(T, device=DEVICE)[None, :]
    seen = j <= i
    if size:
        seen = seen & ((i // size == j // size) if chunks else ((i - j < size) | (j < keep)))
    out = torch.empty(B, T, H, v.shape[-1], dtype=torch.float64, device=DEVICE)
    for b in range(B):
        for h in range(H):
            s = (q[b, :, h] @ k[b, :, h // group].T) * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            if bias is not None:
                s = s + bias[:, h][(i - j).clamp(min=0)]
            s = s.masked_fill(~seen, -math.inf)
            top = s.amax(1, keepdim=True)
            if sink is not None:
                top = torch.maximum(top, sink[h])
            e = torch.exp(s - top)
            den = e.sum(1, keepdim=True) + (torch.exp(sink[h] - top) if sink is not None else 0.0)
            out[b, :, h] = (e / den) @ v[b, :, h // group]
    return out.flatten(2)


class Reference:
    """One pass over whole sequences ``ids`` [B, T]; the logits are those of each row's token ``last``."""

    def __init__(self, cfg, stored, ids, last):
        self.cfg, self.stored, self.ids, self.last = cfg, stored, ids, last
        self.eps = float(cfg["norm"]["eps"]) if "norm" in cfg else float(cfg["rms_norm_eps"])
        self.kept, self.first_values = {}, None

    def w(self, name):
        return self.stored[name].double()

    def has(self, name):
        return name in self.stored

    def lin(self, x, name):
        y = x @ self.w(name).T
        return y + self.w(name + ".b") if self.has(name + ".b") else y

    def heads(self, x, name, count):
        return self.lin(x, name).unflatten(-1, (count, -1))

    def pick(self, x):
        return x[torch.arange(x.shape[0], device=DEVICE), self.last]

    def logits(self):
        if "architectures" in self.cfg:
            return self.qwen2()
        return getattr(self, self.cfg["architecture"].lower())()

    # --- decoders ---------------------------------------------------------------------------------------------
    def qwen2(self):
        c, w = self.cfg, self.w
        H, G = c["num_attention_heads"], c["num_key_value_heads"]
        rot = {"dims": c["hidden_size"] // H, "base": c["rope_theta"]}

        def proj(x, name, heads):
            return (x @ w(name + ".weight").T + w(name + ".bias")).unflatten(-1, (heads, -1))

        x = self.stored["model.embed_tokens.weight"][self.ids].double()
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = over_rms(x, self.eps) * w(p + "input_layernorm.weight")
            q, k, v = (proj(h, f"{p}self_attn.{n}_proj", m) for n, m in (("q", H), ("k", G), ("v", G)))
            a = attend(rotate(q, rot), rotate(k, rot), v, rot["dims"] ** -0.5)
            x = x + a @ w(p + "self_attn.o_proj.weight").T
            h = over_rms(x, self.eps) * w(p + "post_attention_layernorm.weight")
            x = x + (silu(h @ w(p + "mlp.gate_proj.weight").T) * (h @ w(p + "mlp.up_proj.weight").T)) \
                @ w(p + "mlp.down_proj.weight").T
        head = "lm_head.weight" if self.has("lm_head.weight") else "model.embed_tokens.weight"
        return (over_rms(self.pick(x), self.eps) * w("model.norm.weight")) @ w(head).T

    def dyt(self, x, name):
        return torch.tanh(self.w(name + ".alpha") * x) * self.w(name) + self.w(name + ".b")

    def gilidra(self):
        x = self.dyt(self.w("embed")[self.ids], "embed.norm")
        for i, layer in enumerate(self.cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            h = self.dyt(x, f"l{i}.norm1")
            if layer["type"] == "delta":
                y = self.delta(h, p, m)
            elif layer["type"] == "wkv":
                y = self.wkv(h, p, m)
            else:
                y = self.latent(h, p, m, i)
            limit = layer["mlp"]["expert"]["limit"]

            def expert(t, e):
                g = (t @ self.w(e + ".gate").T).clamp(max=limit)
                u = (t @ self.w(e + ".up").T).clamp(-limit, limit)
                return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ self.w(e + ".down").T

            z = self.lin(h, f"l{i}.mlp.router").flatten(0, 1)
            best, ids = z.topk(TOP, -1)
            x = x + y + self.experts(h, f"l{i}.mlp.", ids, torch.softmax(best, -1), expert)
        return self.dyt(self.pick(x), "final.norm") @ self.w("head").T * self.cfg["logit_scale"]

    def zulesun(self):
        def norm(x, name):
            return over_rms(x, self.eps) * (1.0 + self.w(name))

        x = self.w("embed")[self.ids] * self.cfg["embedding"]["scale"]
        for i, layer in enumerate(self.cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            h = norm(x, f"l{i}.norm1")
            if layer["type"] == "lightning":
                q, k, v = (self.heads(h, p + n, m["heads"]) for n in "qkv")
                y = self.linear_attention(silu(q), silu(k), silu(v), m["decay"])
                y = over_rms(y.flatten(2), self.eps) * self.w(p + "norm") * torch.sigmoid(self.lin(h, p + "g"))
                y = self.lin(y, p + "o")
            else:
                left, s = p + "left.", m["left"]
                q = (over_rms(self.lin(h, left + "q"), self.eps) * self.w(left + "q.norm")).unflatten(-1, (s["heads"], -1))
                k = (over_rms(self.lin(h, left + "k"), self.eps) * self.w(left + "k.norm")).unflatten(-1, (s["kv_heads"], -1))
                v = self.heads(h, left + "v", s["kv_heads"])
                a = attend(rotate(q, s["rot"]), rotate(k, s["rot"]), v, s["scale"], s["mask"], chunks=True, cap=s["softcap"])
                a = self.lin(a * torch.sigmoid(self.lin(h, left + "g")), left + "o")
                y = m["left_scale"] * a + m["right_scale"] * self.scan(h, p + "right.", m["right"])
            x = x + norm(y, f"l{i}.norm1b")
            h, p, mlp = norm(x, f"l{i}.norm2"), f"l{i}.mlp.", layer["mlp"]
            if mlp["kind"] == "dense":
                y = torch.relu(self.lin(h, p + "up")) ** 2 @ self.w(p + "down").T
            else:
                z = torch.softmax(self.lin(h, p + "router").flatten(0, 1), -1)
                groups = mlp["router"]["groups"]
                each = z.unflatten(-1, (groups["count"], -1))
                kept = torch.zeros(each.shape[:2], dtype=torch.bool, device=DEVICE)
                kept.scatter_(1, each.amax(-1).topk(groups["keep"], -1)[1], True)
                best, ids = torch.where(kept[:, :, None], each, -1.0).flatten(1).topk(TOP, -1)
                y = self.experts(h, p, ids, best, self.gated)
            x = x + norm(y, f"l{i}.norm2b")
            x = x + self.side(x, i, f"l{i}.side.")
        return norm(self.pick(x), "final.norm") @ self.w("head").T

    def muzasun(self):
        x = self.w("embed")[self.ids]
        for i, layer in enumerate(self.cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            h = self.dyt(x, f"l{i}.norm1")
            if layer["type"] == "attention":
                q = over_rms(self.heads(h, p + "q", m["heads"]), self.eps) * self.w(p + "q.norm")
                k = over_rms(self.heads(h, p + "k", m["kv_heads"]), self.eps) * self.w(p + "k.norm")
                v = self.heads(h, p + "v", m["kv_heads"])
                if self.first_values is None:
                    self.first_values = v
                else:
                    share = self.w(p + "vmix")
                    v = (1.0 - share) * v + share * self.first_values
                y = self.lin(attend(rotate(q, m["rot"]), rotate(k, m["rot"]), v, m["scale"]), p + "o")
            elif layer["type"] == "mlstm":
                y = self.memory(h, p, m)
            else:
                y = self.delta(h, p, m)
            u, mlp = self.dyt(x, f"l{i}.norm2"), layer["mlp"]
            if mlp["kind"] == "dense":
                f = self.gated(u, f"l{i}.mlp")
            else:
                best, ids = torch.sigmoid(self.lin(u, f"l{i}.mlp.router")).flatten(0, 1).topk(TOP, -1)
                f = self.experts(u, f"l{i}.mlp.", ids, best, self.gated, weigh_inputs=True) + self.gated(u, f"l{i}.mlp.shared")
            x = x + self.cfg["residual_mult"] * (y + f)
        return self.dyt(self.pick(x), "final.norm") @ self.w("head").T * self.cfg["logit_scale"]

    def lurirax(self):
        x = self.w("embed")[self.ids] * self.cfg["embedding"]["scale"]
        for i, layer in enumerate(self.cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            if layer["type"] == "attention":
                q = over_rms(rotate(self.heads(x, p + "q", m["heads"]), m["rot"]), self.eps)
                k = over_rms(rotate(self.heads(x, p + "k", m["kv_heads"]), m["rot"]), self.eps)
                y = attend(q, k, self.heads(x, p + "v", m["kv_heads"]), m["scale"], m["mask"], sink=self.w(p + "sink"))
            elif layer["type"] == "attention_2":
                q = over_rms(self.heads(x, p + "q", m["heads"]).unflatten(-1, (2, -1)), self.eps) * self.w(p + "q.norm")
                k = over_rms(self.heads(x, p + "k", m["kv_heads"]).unflatten(-1, (2, -1)), self.eps) * self.w(p + "k.norm")
                v = self.heads(x, p + "v", m["kv_heads"])
                one, two = (attend(q[..., s, :], k[..., s, :], v, m["scale"], m["mask"]) for s in (0, 1))
                w = self.w
                lam = torch.exp((w(p + "lq1") * w(p + "lk1")).sum()) - torch.exp((w(p + "lq2") * w(p + "lk2")).sum()) + m["diff"]
                y = over_rms((one - lam * two).unflatten(-1, (m["heads"], -1)), self.eps).flatten(2) * (1.0 - m["diff"])
            else:
                y = m["left_scale"] * self.biased_chunks(x, p + "left.", m["left"])
                s, r = m["right"], p + "right."
                q, k = (rotate(self.heads(x, r + n, s["heads"]), s["rot"]) for n in "qk")
                o = self.linear_attention(q, k * s["dim"] ** -0.5, self.heads(x, r + "v", s["heads"]), s["decay"])
                o = over_rms(o, self.eps).flatten(2) * silu(self.lin(x, r + "g"))
                y = y + m["right_scale"] * self.lin(o, r + "o")
            if layer["type"] != "parallel":
                y = self.lin(y, p + "o")
            x = x + over_rms(y, self.eps) * self.w(f"l{i}.norm1")
            p, mlp = f"l{i}.mlp.", layer["mlp"]
            if mlp["kind"] == "dense":
                y = (gelu(self.lin(x, p + "gate")) * self.lin(x, p + "up")) @ self.w(p + "down").T
            else:
                z = torch.sigmoid(self.lin(x, p + "router")).flatten(0, 1)
                ids = (z + self.w(p + "correction") if self.has(p + "correction") else z).topk(TOP, -1)[1]
                y = self.experts(x, p, ids, mlp["router"]["scale"] * z.gather(1, ids), self.gated)
                y = y + self.gated(x, p + "shared") * torch.sigmoid(self.lin(x, p + "shared.sg"))
            x = x + over_rms(y, self.eps) * self.w(f"l{i}.norm2")
        return (over_rms(self.pick(x), self.eps) * self.w("final.norm")) @ self.w("head").T

    def zeladra(self):
        x = self.w("embed")[self.ids] * self.cfg["embedding"]["scale"]
        streams = x[None].repeat(int(self.cfg["streams"]), 1, 1, 1)

        def norm(u, name):
            return layer_norm(u, self.eps) * self.w(name) + self.w(name + ".b")

        def connect(s, name, sublayer):
            y = sublayer(torch.einsum("s,sbtw->btw", self.w(name + "in"), s))
            return torch.einsum("st,sbkw->tbkw", self.w(name + "mix"), s) + self.w(name + "out")[:, None, None, None] * y

        for i, layer in enumerate(self.cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]

            def mixer(u):
                h = norm(u, f"l{i}.norm1")
                if layer["type"] == "mamba2":
                    return self.state_space(h, p, m)
                if layer["type"] == "latent_attention":
                    return self.latent(h, p, m, i, pairs="neighbours")
                q = rotate(self.heads(h, p + "q", m["heads"]), m["rot"], "neighbours")
                k = rotate(self.heads(h, p + "k", m["kv_heads"]), m["rot"], "neighbours")
                return self.lin(attend(q, k, self.heads(h, p + "v", m["kv_heads"]), m["scale"], m["mask"]), p + "o")

            streams = connect(streams, f"l{i}.hc1.", mixer)
            if layer["mlp"] is not None:
                streams = connect(streams, f"l{i}.hc2.", lambda u: self.gated(norm(u, f"l{i}.norm2"), f"l{i}.mlp"))
        return norm(self.pick(streams.sum(0)), "final.norm") @ self.w("head").T

    def rebidra(self):
        x = start = self.w("embed")[self.ids] * self.cfg["embedding"]["scale"]
        n, loop = len(self.cfg["layers"]), self.cfg["loop"]
        body = [(i, i == loop["start"]) for i in range(loop["start"], loop["stop"])] * loop["times"]
        order = [(i, False) for i in range(loop["start"])] + body + [(i, False) for i in range(loop["stop"], n)]
        for i, enters in order:
            m, p = self.cfg["layers"][i]["mixer"], f"l{i}.mix."
            if enters:
                x = torch.cat([x, start], -1) @ self.w("loop.in").T
            h = layer_norm(x, self.eps) * self.w(f"l{i}.norm1")
            q = convolve(self.lin(h, p + "q"), self.w(p + "q.conv")).unflatten(-1, (m["heads"], -1))
            v = convolve(self.lin(h, p + "k"), self.w(p + "k.conv")).unflatten(-1, (m["kv_heads"], -1))
            q = rotate(over_rms(q, self.eps) * self.w(p + "q.norm"), m["rot"])
            k = rotate(over_rms(v, self.eps) * self.w(p + "k.norm"), m["rot"])
            o = attend(q, k, v, m["scale"], m["mask"], sink=self.w(p + "sink"))
            o = o.unflatten(-1, (m["heads"], -1)) * torch.sigmoid(self.lin(h, p + "g"))[..., None]
            x = x + self.lin(o.flatten(2), p + "o")
            p = f"l{i}.mlp."
            h = layer_norm(x, self.eps) * self.w(f"l{i}.norm2")
            best, ids = self.lin(h, p + "router").flatten(0, 1).topk(TOP, -1)

            def squared(t, e):
                return torch.relu(t @ self.w(e + ".up").T) ** 2 @ self.w(e + ".down").T

            x = x + self.experts(h, p, ids, torch.softmax(best, -1), squared) \
                + torch.sigmoid(self.lin(h, p + "shared.sg")) * squared(h, p + "shared")
            x = x + self.side(x, i, f"l{i}.side.")
        return (layer_norm(self.pick(x), self.eps) * self.w("final.norm")) @ self.w("head").T * self.cfg["logit_scale"]

    # --- parts -------------------------------------------------------------------------------------------------
    def gated(self, x, name):
        return (silu(x @ self.w(name + ".gate").T) * (x @ self.w(name + ".up").T)) @ self.w(name + ".down").T

    def experts(self, x, p, ids, shares_, expert, weigh_inputs=False):
        flat = x.flatten(0, 1)
        out = torch.zeros_like(flat)
        for e in range(OTHER_SIZES["m"][3]):
            token, place = (ids == e).nonzero(as_tuple=True)
            if token.numel():
                share = shares_[token, place][:, None]
                y = expert(share * flat[token], f"{p}e{e}") if weigh_inputs else share * expert(flat[token], f"{p}e{e}")
                out.index_add_(0, token, y)
        return out.view_as(x)

    def side(self, x, i, p):
        dim = self.cfg["token_side"]["dim"]
        rows = self.stored["side.embed"][self.ids][..., i * dim:(i + 1) * dim].double()
        return over_rms(self.lin(gelu(self.lin(x, p + "gate")) * rows, p + "proj"), self.eps) * self.w(p + "norm")

    def latent(self, h, p, m, i, pairs="halves"):
        source = m.get("kv_from")
        if source is None:
            down = self.lin(h, p + "dkv")
            c = over_rms(down[..., :m["kv_rank"]], self.eps) * self.w(p + "dkv.norm")
            self.kept[i] = (c, rotate(down[..., None, m["kv_rank"]:], m["rot"], pairs))
        c, key = self.kept[i if source is None else source]
        H, d = m["heads"], m["dim"]
        q = self.heads(over_rms(self.lin(h, p + "dq"), self.eps) * self.w(p + "dq.norm"), p + "uq", H)
        q = torch.cat([q[..., :d], rotate(q[..., d:], m["rot"], pairs)], -1)
        k = torch.cat([self.heads(c, p + "uk", H), key.expand(-1, -1, H, -1)], -1)
        o = attend(q, k, self.heads(c, p + "uv", H), m["scale"], m.get("mask"))
        if self.has(p + "g"):
            o = (o.unflatten(-1, (H, -1)) * torch.sigmoid(self.lin(h, p + "g"))[..., None]).flatten(2)
        return self.lin(o, p + "o")

    def biased_chunks(self, x, p, m):
        q = over_rms(self.heads(x, p + "q", m["heads"]), self.eps) * self.w(p + "q.norm")
        k = over_rms(self.heads(x, p + "k", m["kv_heads"]), self.eps) * self.w(p + "k.norm")
        rows, far, half = m["bias_rows"], float(m["bias_max"]), m["bias_rows"] // 2
        bucket = [n if n < half else min(rows - 1, half + math.floor(math.log(n / half) / math.log(far / half) * (rows - half)))
                  for n in range(x.shape[1])]
        bias = self.w(p + "rel")[torch.tensor(bucket, device=DEVICE)]
        o = attend(q, k, self.heads(x, p + "v", m["kv_heads"]), m["scale"], m["mask"], chunks=True, sink=self.w(p + "sink"),
                   bias=bias)
        o = o.unflatten(-1, (m["heads"], -1)) * torch.sigmoid(self.lin(x, p + "g"))[..., None]
        return self.lin(o.flatten(2), p + "o")

    @staticmethod
    def linear_attention(q, k, v, decay):
        keep = torch.tensor(decay, dtype=torch.float64, device=DEVICE)[None, :, None, None]
        S, out = 0.0, torch.empty_like(v)
        for t in range(q.shape[1]):
            S = keep * S + k[:, t, :, :, None] * v[:, t, :, None, :]
            out[:, t] = (S * q[:, t, :, :, None]).sum(2)
        return out

    def delta(self, h, p, m):
        H, G, D = m["heads"], m["kv_heads"], m["dim"]
        q, k = (silu(convolve(self.lin(h, p + n), self.w(f"{p}{n}.conv"))).unflatten(-1, (G, -1)) for n in "qk")
        v = silu(convolve(self.lin(h, p + "v"), self.w(p + "v.conv"))).unflatten(-1, (H, -1))
        q = (q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) / math.sqrt(D)).repeat_interleave(H // G, 2)
        k = (k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 2)
        beta = torch.sigmoid(self.lin(h, p + "b"))
        if "decay_rank" in m:      # one decay per head and key channel
            step = softplus(self.lin(self.lin(h, p + "a1"), p + "a2") + self.w(p + "dt_bias")).unflatten(-1, (H, -1))
            gate = torch.sigmoid(self.lin(self.lin(h, p + "g1"), p + "g2"))
        else:
            step = softplus(self.lin(h, p + "a") + self.w(p + "dt_bias"))[..., None]
            gate = silu(self.lin(h, p + "g"))
        decay = torch.exp(-torch.exp(self.w(p + "A_log"))[:, None] * step)
        S, out = torch.zeros(*v.shape[:1], H, D, v.shape[-1], dtype=torch.float64, device=DEVICE), torch.empty_like(v)
        for t in range(h.shape[1]):
            S = decay[:, t, :, :, None] * S
            u = beta[:, t, :, None] * (v[:, t] - (S * k[:, t, :, :, None]).sum(2))
            S = S + k[:, t, :, :, None] * u[:, :, None, :]
            out[:, t] = (S * q[:, t, :, :, None]).sum(2)
        return self.lin((over_rms(out, self.eps) * self.w(p + "norm")).flatten(2) * gate, p + "o")

    def wkv(self, h, p, m):
        before = torch.cat([torch.zeros_like(h[:, :1]), h[:, :-1]], 1)

        def mixed(n):
            return h + (before - h) * self.w(f"{p}mu.{n}")

        r, k, v = (self.heads(mixed(n), p + n, m["heads"]) for n in "rkv")
        low = torch.tanh(self.lin(mixed("w"), p + "w1"))
        decay = torch.exp(-torch.exp(self.lin(low, p + "w2") + self.w(p + "w0"))).unflatten(-1, (m["heads"], -1))
        bonus = self.w(p + "u").view(m["heads"], -1, 1)
        S, out = 0.0, torch.empty_like(v)
        for t in range(h.shape[1]):
            kv = k[:, t, :, :, None] * v[:, t, :, None, :]
            out[:, t] = ((S + bonus * kv) * r[:, t, :, :, None]).sum(2)
            S = decay[:, t, :, :, None] * S + kv
        y = over_rms(out, self.eps).flatten(2) * self.w(p + "norm") * silu(self.lin(mixed("g"), p + "g"))
        return self.lin(y, p + "o")

    def memory(self, h, p, m):
        H, cap = m["heads"], m["gate_cap"]
        q, k, v = (self.heads(h, p + n, H) for n in "qkv")
        q = q / math.sqrt(m["dim"])
        into = cap * torch.tanh(self.lin(h, p + "i") / cap)
        keep = -softplus(-cap * torch.tanh(self.lin(h, p + "f") / cap))
        top, S, n, out = torch.zeros_like(into[:, 0]), 0.0, 0.0, torch.empty_like(v)
        for t in range(h.shape[1]):
            above = torch.maximum(keep[:, t] + top, into[:, t])
            f, i = torch.exp(keep[:, t] + top - above)[..., None], torch.exp(into[:, t] - above)[..., None]
            S = f[..., None] * S + i[..., None] * k[:, t, :, :, None] * v[:, t, :, None, :]
            n, top = f * n + i * k[:, t], above
            den = torch.maximum((n * q[:, t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
            out[:, t] = (S * q[:, t, :, :, None]).sum(2) / den[..., None]
        y = over_rms(out, self.eps).flatten(2) * self.w(p + "norm") * torch.sigmoid(self.lin(h, p + "g"))
        return self.lin(y, p + "o")

    def scan(self, h, p, m):
        n, rank = m["state"], m["dt_rank"]
        x, z = self.lin(h, p + "in").chunk(2, -1)
        x = silu(convolve(x.contiguous(), self.w(p + "conv")) + self.w(p + "conv.b"))
        low = self.lin(x, p + "x")
        dt = softplus(self.lin(low[..., :rank], p + "dt"))
        b, c, a = low[..., rank:rank + n], low[..., rank + n:], -torch.exp(self.w(p + "A_log"))
        S, y = 0.0, torch.empty_like(x)
        for t in range(x.shape[1]):
            S = torch.exp(dt[:, t, :, None] * a) * S + (dt[:, t] * x[:, t])[..., None] * b[:, t, None, :]
            y[:, t] = (S * c[:, t, None, :]).sum(-1)
        return self.lin((y + self.w(p + "D") * x) * silu(z), p + "o")

    def state_space(self, h, p, m):
        H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
        z, xbc, dt = self.lin(h, p + "in").split([H * P, H * P + 2 * G * N, H], -1)
        xbc = silu(convolve(xbc.contiguous(), self.w(p + "conv")) + self.w(p + "conv.b"))
        x, b, c = xbc.split([H * P, G * N, G * N], -1)
        x = x.unflatten(-1, (H, P))
        b, c = (v.unflatten(-1, (G, N)).repeat_interleave(H // G, 2) for v in (b, c))
        step = softplus(dt + self.w(p + "dt_bias"))
        keep = torch.exp(-torch.exp(self.w(p + "A_log")) * step)
        S, y = 0.0, torch.empty_like(x)
        for t in range(h.shape[1]):
            S = keep[:, t, :, None, None] * S + (step[:, t, :, None] * b[:, t])[..., None] * x[:, t, :, None, :]
            y[:, t] = (S * c[:, t, :, :, None]).sum(2)
        y = (y + self.w(p + "D")[:, None] * x).flatten(2) * silu(z)
        y = over_rms(y.unflatten(-1, (m["norm_groups"], -1)), self.eps).flatten(2) * self.w(p + "norm")
        return self.lin(y, p + "o")
