"""What this library is timed on: the work that a program built on it has it do, through its public entry points.

Three kinds of cases, over the three measured Llama shapes and two of the other designs, with random weights:

``decode``   one step of single tokens for a batch of sequences that hold a context already, and the selection of the
             next tokens on the device: what a generation loop repeats for every token (``Engine.step_from_device``,
             ``DeviceSelector.select_start``).
``prompt``   the prompts of new sequences in one step, logits at each one's last place: what a request waits for before
             its first token (``Engine.step_view``).
``request``  prompts in one step and then a few steps of single tokens: a whole short request, for the designs whose
             mixers carry a state of fixed size (their sequences cannot be shortened to run a step again).

Tokens are given and not fed back, so that the outputs of a pass do not hang on a near tie in an earlier step.  A case's
lengths lie evenly between its shortest and its longest; which sequence has which comes from the seed, as do weights
and tokens.
"""

import math

import torch

import nnis_amd.models  # noqa: F401  (registers the architectures)
from nnis_amd.config import preset
from nnis_amd.config.registry import spec_from_config
from nnis_amd.engine.batch import StepEntry
from nnis_amd.engine.runtime import Runtime
from nnis_amd.engine.step import Engine
from nnis_amd.models.decoder import DecoderModel
from nnis_amd.sampling.device import DeviceSelector
from nnis_amd.sampling.params import SamplingParams

LLAMAS = ("smollm2-135m", "tinyllama-1.1b", "smollm2-1.7b")
PROMPT_STEP_TOKENS = 16384  # a context is brought into the cache in steps of at most this many tokens


# ---- the cases ------------------------------------------------------------------------------------------------------

def _decode(model, batch, shortest, longest, dtype="bfloat16", sampled=False):
    return {"kind": "decode", "model": model, "dtype": dtype, "batch": batch, "shortest": shortest, "longest": longest, "sampled": sampled}


def _prompt(model, sequences, shortest, longest, dtype="bfloat16"):
    return {"kind": "prompt", "model": model, "dtype": dtype, "batch": sequences, "shortest": shortest, "longest": longest}


def _request(model, width, sequences, shortest, longest, new):
    return {"kind": "request", "model": model, "width": width, "dtype": "bfloat16", "batch": sequences, "shortest": shortest,
            "longest": longest, "new": new}


def listed():
    return [
        # one user of a small model in the middle of a conversation: nothing but latency
        dict(_decode("smollm2-135m", 1, 700, 700), name="decode_135m_b1"),
        # the benchmark's headline: a small batch of unequal contexts
        dict(_decode("smollm2-135m", 8, 128, 2047), name="decode_135m_b8"),
        # the same with tokens drawn by temperature, top-k and top-p, an odd number of sequences
        dict(_decode("smollm2-135m", 11, 60, 1000, sampled=True), name="decode_135m_b11_sampled"),
        # a server's full batch of a wider model, contexts from a few words to nearly the model's end
        dict(_decode("tinyllama-1.1b", 64, 17, 2000), name="decode_tinyllama_b64"),
        # long documents: the keys and values are several times the weights
        dict(_decode("smollm2-1.7b", 8, 7800, 8000), name="decode_1.7b_b8_8k"),
        # a chat turn: a short prompt of an odd length
        dict(_prompt("smollm2-135m", 1, 177, 177), name="prompt_135m_177"),
        # a queue of unequal prompts in one step: the largest product the library is given
        dict(_prompt("tinyllama-1.1b", 24, 16, 1024), name="prompt_tinyllama_ragged24"),
        # a page of text for the widest shape
        dict(_prompt("smollm2-1.7b", 1, 2011, 2011), name="prompt_1.7b_2011"),
        # the 32-bit path, step by step and over a prompt: what the numbers of the 16-bit path are checked against
        dict(_decode("smollm2-135m", 8, 100, 1023, dtype="float32"), name="decode_135m_b8_fp32"),
        dict(_prompt("tinyllama-1.1b", 1, 509, 509, dtype="float32"), name="prompt_tinyllama_509_fp32"),
        # the designs beside Llama: recurrences over matrix states, latents; scans, residual streams
        dict(_request("mafalorn", 2048, 1, 1500, 1500, 8), name="request_mafalorn_1500"),
        dict(_request("zifunex", 2048, 4, 90, 700, 8), name="request_zifunex_ragged4"),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "request"])
    if kind == "request":
        batch = rng.randint(1, 6)
        longest = _log_uniform(rng, 24, min(1500, 3000 // batch))
        return _request(rng.choice(["mafalorn", "zifunex"]), rng.choice([1024, 2048]), batch, rng.randint(max(8, longest // 8), longest), longest,
                        rng.randint(2, 8))
    model = rng.choice(LLAMAS)
    dtype = "float32" if model != "smollm2-1.7b" and rng.random() < 0.25 else "bfloat16"
    end = 2040 if model == "tinyllama-1.1b" else 8000
    if kind == "decode":
        batch = _log_uniform(rng, 1, 64)
        longest = _log_uniform(rng, 48, min(end, (6000 if dtype == "float32" else 60000) // batch))
        return _decode(model, batch, max(8, _log_uniform(rng, max(8, longest // 32), longest)), longest, dtype,
                       batch >= 8 and rng.random() < 0.4)
    batch = rng.choice([1, 1, 1, _log_uniform(rng, 2, 24)])
    most = {"smollm2-135m": 9000, "tinyllama-1.1b": 9000, "smollm2-1.7b": 4500}[model]
    longest = _log_uniform(rng, 12, min(end, (500 if dtype == "float32" else most) // batch))
    return _prompt(model, batch, rng.randint(max(1, longest // 8), longest), longest, dtype)


# ---- configurations, weights, tokens --------------------------------------------------------------------------------

def _mafalorn(width):
    """The design's mixers without its routed feed-forwards: with them a near tie in a router, which any other rounding
    turns over, changes a token's output as a whole (the logits of two correct 16-bit implementations then differ by
    0.2 to 0.6 of themselves), and a comparison would say nothing."""
    wide = width // 1024  # 1 or 2: the two measured sets of layer sizes
    heads, dim = 4 * wide, 64 * wide
    layers = {
        "R": {"type": "retention", "mlp": None, "mixer": {"heads": heads, "dim": 128, "vdim": 256, "decay": [1.0 - 2.0 ** (-5 - h) for h in range(heads)],
                                                         "rot": {"dims": 128, "base": 10000.0}}},
        "P": {"type": "parallel", "mlp": None, "mixer": {
            "left": {"heads": 16, "kv_heads": 4, "dim": dim, "vdim": dim, "scale": dim ** -0.5,
                     "rot": {"dims": 64, "base": 10000.0, "scaling": {"factor": 4.0, "original": 2048, "fast": 32.0, "slow": 1.0}}},
            "right": {"heads": 8 * wide, "kv_heads": 4 * wide, "dim": dim, "vdim": 128, "conv": 4}, "left_scale": 0.7, "right_scale": 0.7}},
        "L": {"type": "latent_attention", "mlp": None, "mixer": {
            "heads": 16, "dim": dim, "rot_dim": 32 * wide, "vdim": dim, "kv_rank": 64 + 64 * wide, "scale": (dim + 32 * wide) ** -0.5,
            "rot": {"dims": 32 * wide, "base": 10000.0}, "mask": {"size": 512 * wide}}},
    }
    return {"architecture": "Mafalorn", "vocab": 32000, "width": width, "norm": {"eps": 1e-6}, "logit_scale": 0.5,
            "layers": [layers[kind] for kind in "RPRLRPRL"]}


def _zifunex(width):
    wide = width // 1024
    dim = 64 * wide
    side_by_side = {"type": "parallel", "mlp": {"kind": "dense", "ff": 2816 * wide}, "mixer": {
        "left": {"heads": 16, "kv_heads": 4, "dim": dim, "vdim": 64, "rot": {"dims": dim, "base": 10000.0}, "scale": dim ** -0.5, "softcap": 30.0},
        "right": {"inner": 2 * width, "state": 16, "dt_rank": width // 16, "conv": 4}}}
    linear = {"type": "gla", "mlp": None, "mixer": {"heads": 4 * wide, "dim": 128, "vdim": 256, "tau": 16.0, "rank": 32}}
    return {"architecture": "Zifunex", "vocab": 32000, "width": width, "streams": 2, "norm": {"eps": 1e-5},
            "embedding": {"bigram": {"buckets": 65521, "mul_prev": 1000003, "mul_cur": 31}},
            "layers": [side_by_side if kind == "P" else linear for kind in "PPGPPGPP"]}


def _config(case):
    if case["model"] in LLAMAS:
        return preset(case["model"])
    return {"mafalorn": _mafalorn, "zifunex": _zifunex}[case["model"]](case["width"])


# how a random model's tensors of each rule are spread (``register_init_rule`` beside the parts): factor and middle of a normal
_SPREAD = {"matrix": (0.02, 0.0), "gain": (0.01, 1.0), "small": (0.1, 0.0), "router": (0.3, 0.0), "conv_taps": (0.3, 0.0), "step_matrix": (0.3, 0.0),
           "step_bias": (0.5, -2.0), "decay_bias": (1.0, 2.0), "stream_share": (0.25, 0.5), "stream_mix": (0.2, 0.0), "log_rates": (0.1, 0.0)}


def _weights(model, seed):
    """name -> bfloat16 tensor on the GPU, as a checkpoint of the design holds it (a tied head is the table itself)."""
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    out = {}
    for tensor in model.tensors():
        if tensor.name in out:
            continue
        if tensor.fallback is not None:
            out[tensor.name] = out[tensor.fallback]
            continue
        factor, middle = _SPREAD[tensor.init]
        w = torch.randn(tuple(tensor.shape), generator=generator, device="cuda").mul_(factor).add_(middle)
        if tensor.init == "stream_mix":
            w += torch.eye(tensor.shape[0], device="cuda")
        if tensor.init == "log_rates":
            w += torch.log(torch.arange(1, tensor.shape[-1] + 1, device="cuda", dtype=torch.float32))
        out[tensor.name] = w.to(torch.bfloat16)
    return out


def _lengths(case):
    """Evenly from the shortest to the longest.  A context that fills its last page is one token shorter: its next
    step would take a page and give it back in every pass, which a growing sequence does once in 64 steps."""
    batch, low, high = case["batch"], case["shortest"], case["longest"]
    lengths = [high if batch == 1 else low + (high - low) * i // (batch - 1) for i in range(batch)]
    return [n - 1 if case["kind"] == "decode" and n % 64 == 0 else n for n in lengths]


def _tokens(case, seed, vocab):
    """Each sequence's token ids: its prompt or context and, behind it, the tokens that its single steps are given."""
    generator = torch.Generator()
    generator.manual_seed(seed + 1)
    lengths = _lengths(case)
    order = torch.randperm(len(lengths), generator=generator).tolist()
    more = {"decode": 1, "prompt": 0, "request": case.get("new", 0)}[case["kind"]]
    return [(torch.randint(0, vocab, (lengths[i] + more,), generator=generator).tolist(), lengths[i]) for i in order]


# ---- a pass ---------------------------------------------------------------------------------------------------------

class _State:
    """What a program keeps between passes: the engine with its weights and cache, and the tokens it is about to run."""


def prepare(case, seed):
    state = _State()
    _, spec = spec_from_config(_config(case))
    model = DecoderModel(spec)
    rt = Runtime(dtype=case["dtype"])
    model.check(rt)
    weights = _weights(model, seed)
    if rt.is_fp32:
        wide = {id(w): w.float() for w in weights.values()}  # widened exactly, as the loader does for a 32-bit runtime
        weights = {name: wide[id(w)] for name, w in weights.items()}
        del wide
    model.bind(weights, rt)
    del weights
    state.kind = case["kind"]
    sequences = _tokens(case, seed, spec.vocab_size)
    room = sum(-(-(len(ids) + 1) // 64) * 64 for ids, _ in sequences)
    state.engine = engine = Engine(model, rt, max_tokens=room, max_slots=len(sequences))
    state.prompts = [ids[:n] for ids, n in sequences]
    longest = max(len(ids) for ids, _ in sequences)
    if state.kind == "prompt":
        return state
    state.selector = DeviceSelector(engine)
    state.given = torch.tensor([ids[n:] for ids, n in sequences], dtype=torch.int32).t().contiguous().to(rt.device)  # [step, sequence]
    engine.prepare_decode(len(sequences), longest)
    state.greedy = [None] * len(sequences)
    if state.kind == "request":
        return state
    state.params = state.greedy
    if case["sampled"]:
        state.params = [SamplingParams(seed=1000 * seed + i, temperature=0.8, top_k=50, top_p=0.9) for i in range(len(sequences))]
    state.slots, state.lengths = [], [n for _, n in sequences]
    group = []
    for prompt, params in zip(state.prompts, state.params):
        slot = engine.start_sequence()
        state.selector.start(slot, params)
        state.slots.append(slot)
        if group and sum(len(e.tokens) for e in group) + len(prompt) > PROMPT_STEP_TOKENS:
            engine.step(group)
            group = []
        group.append(StepEntry(slot, prompt, None))
    engine.step(group)
    state.generators = state.selector.rng.clone() if case["sampled"] else None
    return state


def run(state):
    engine = state.engine
    if state.kind == "decode":
        if state.generators is not None:
            state.selector.rng.copy_(state.generators)  # every pass draws the same numbers
        logits = engine.step_from_device(state.slots, state.given[0])
        pending = state.selector.select_start(logits, state.slots, state.params)
        for slot, length in zip(state.slots, state.lengths):
            engine.truncate(slot, length)  # the next pass takes the same step
        # (greedy tokens are the logits' places: a near tie may fall either way)
        return {"logits": logits, "tokens": pending.device} if state.generators is not None else {"logits": logits}
    slots = [engine.start_sequence() for _ in state.prompts]
    entries = [StepEntry(slot, prompt, None) for slot, prompt in zip(slots, state.prompts)]
    if state.kind == "prompt":
        out = {"logits": engine.step_view(entries)}
    else:
        out = {"prompt": engine.step(entries)}
        for index in range(state.given.shape[0]):
            logits = engine.step_from_device(slots, state.given[index])
            state.selector.select_start(logits, slots, state.greedy)
            out[f"step{index}"] = logits.clone()
    for slot in slots:
        engine.end_sequence(slot)
    return out


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def _layer_work(config, lengths, new, size):
    """(bytes of weights that every token passes, multiply-adds a token, bytes of the cache read, bytes of it written,
    multiply-adds on cached keys and states) of all layers of a design other than Llama; ``new``: tokens a sequence brings."""
    width = config["width"]
    weights = per_token = read = written = on_cache = 0
    for layer in config["layers"]:
        m = layer["mixer"]
        left, right = (m.get("left"), m.get("right")) if layer["type"] == "parallel" else (None, None)
        matrix = 0
        if layer["type"] in ("retention", "gla"):
            hd, he = m["heads"] * m["dim"], m["heads"] * m["vdim"]
            matrix += (2 * hd + 3 * he) * width + (m.get("rank", 0) * (width + hd))
            on_cache += 2 * m["heads"] * m["dim"] * m["vdim"] * sum(new)
            read += 4 * m["heads"] * m["dim"] * m["vdim"] * len(new)
            written += 4 * m["heads"] * m["dim"] * m["vdim"] * len(new)
        if left is not None:
            own_values = 0 if config["architecture"] == "Mafalorn" else left["kv_heads"] * left["vdim"]
            matrix += (left["heads"] * (left["dim"] + left["vdim"]) + left["kv_heads"] * left["dim"] + own_values) * width
            on_cache += left["heads"] * (left["dim"] + left["vdim"]) * sum(n * t + t * (t + 1) // 2 for n, t in zip(lengths, new))
            each = size * left["kv_heads"] * (left["dim"] + left["vdim"])
            read += each * sum(lengths)
            written += each * sum(new)
        if right is not None and "inner" in right:  # the selective scan
            c, n = right["inner"], right["state"]
            matrix += 3 * c * width + (2 * right["dt_rank"] + 2 * n) * c
            on_cache += (3 * n + right["conv"]) * c * sum(new)
            read += 4 * c * n * len(new)
            written += 4 * c * n * len(new)
        elif right is not None:  # the gated delta rule
            cells = right["heads"] * right["dim"] * right["vdim"]
            matrix += (2 * right["kv_heads"] * right["dim"] + 3 * right["heads"] * right["vdim"] + 2 * right["heads"]) * width
            on_cache += 3 * cells * sum(new)
            read += 4 * cells * len(new)
            written += 4 * cells * len(new)
        if layer["type"] == "latent_attention":
            heads, rank, rot = m["heads"], m["kv_rank"], m["rot_dim"]
            matrix += (heads * (m["dim"] + rot) + rank + rot + 2 * heads * m["vdim"]) * width + heads * rank * (m["dim"] + m["vdim"])
            seen = [sum(min(i + 1, m["mask"]["size"]) for i in range(n, n + t)) for n, t in zip(lengths, new)]
            on_cache += heads * (2 * rank + rot) * sum(seen)
            read += size * (rank + rot) * sum(min(n, m["mask"]["size"]) for n in lengths)
            written += size * (rank + rot) * sum(new)
        if layer["mlp"] is not None:
            matrix += 3 * width * layer["mlp"]["ff"]
        weights += size * matrix
        per_token += matrix
    return weights, per_token, read, written, on_cache


def _step_work(case, config, lengths, new):
    """(bytes, flops) of one step: ``lengths`` tokens held, ``new`` tokens brought, logits at one place a sequence."""
    size = 4 if case["dtype"] == "float32" else 2
    if case["model"] in LLAMAS:
        width, inner, layers, vocab = (config[k] for k in ("hidden_size", "intermediate_size", "num_hidden_layers", "vocab_size"))
        heads, kv, dim = (config[k] for k in ("num_attention_heads", "num_key_value_heads", "head_dim"))
        per_token = layers * ((2 * heads + 2 * kv) * dim * width + 3 * inner * width)
        weights, each = size * per_token, size * layers * 2 * kv * dim
        read, written = each * sum(lengths), each * sum(new)
        on_cache = layers * 2 * heads * dim * sum(n * t + t * (t + 1) // 2 for n, t in zip(lengths, new))
    else:
        width, vocab = config["width"], config["vocab"]
        weights, per_token, read, written, on_cache = _layer_work(config, lengths, new, size)
    rows = len(new)
    total = weights + read + written + size * width * (vocab + sum(new)) + 4 * rows * vocab
    return total, 2 * (per_token * sum(new) + on_cache + rows * width * vocab)


def work(case):
    config = _config(case)
    lengths = _lengths(case)
    if case["kind"] == "decode":
        steps = [(lengths, [1] * len(lengths))]
    else:
        steps = [([0] * len(lengths), lengths)] + [([n + i for n in lengths], [1] * len(lengths)) for i in range(case.get("new", 0))]
    each = [_step_work(case, config, held, new) for held, new in steps]
    return {"bytes": float(sum(b for b, _ in each)), "flops": float(sum(f for _, f in each))}


def tolerance(case):
    # measured against 64 bits: 1e-6 to 9e-6 in 32 bits, 0.005 to 0.025 for the Llamas, 0.015 to 0.055 for the others
    if case["dtype"] == "float32":
        return {"rel": 3e-5, "differ": 0.25} if case.get("sampled") else {"rel": 3e-5}
    rel = 0.12 if case["model"] not in LLAMAS else 0.07
    return {"rel": rel, "differ": 0.25} if case.get("sampled") else {"rel": rel}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------

def _rms(x, weight, eps):
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return x if weight is None else x * weight


def _layer_norm(x, weight, bias, eps):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * weight + bias


def _silu(x):
    return x * torch.sigmoid(x)


def _turn(x, cos, sin, neighbours=False):
    """x [tokens, heads, size]; the first 2 x pairs channels turn, channel i with i + pairs or 2i with 2i + 1."""
    pairs = cos.shape[-1]
    cos, sin, out = cos[:, None], sin[:, None], x.clone()
    first, second = (slice(0, 2 * pairs, 2), slice(1, 2 * pairs, 2)) if neighbours else (slice(0, pairs), slice(pairs, 2 * pairs))
    u, v = x[..., first], x[..., second]
    out[..., first], out[..., second] = u * cos - v * sin, v * cos + u * sin
    return out


def _angles(positions, rot):
    """Cosine and sine of a rotation's angles, frequencies over a ramp where it has one."""
    dims, base, scaling = rot["dims"], rot["base"], rot.get("scaling")
    freq = base ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64) / dims)
    magnitude = 1.0
    if scaling is not None:
        def place(turns):
            return dims * math.log(scaling["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))

        low, high = max(math.floor(place(scaling["fast"])), 0), min(math.ceil(place(scaling["slow"])), dims - 1)
        ramp = ((torch.arange(dims // 2, dtype=torch.float64) - low) / max(high - low, 0.001)).clamp(0.0, 1.0)
        freq = freq / scaling["factor"] * ramp + freq * (1.0 - ramp)
        magnitude = 0.1 * math.log(scaling["factor"]) + 1.0
    angle = torch.arange(positions, dtype=torch.float64)[:, None] * freq
    return (torch.cos(angle) * magnitude).cuda(), (torch.sin(angle) * magnitude).cuda()


def _llama_angles(positions, dims, theta):
    """Llama's tables are defined in 32 bits: exponents, frequencies and angles are rounded, then cosine and sine."""
    exponent = 2.0 * torch.arange(dims // 2, dtype=torch.float32) / torch.tensor(float(dims), dtype=torch.float32)
    freq = 1.0 / torch.pow(torch.tensor(theta, dtype=torch.float32).double(), exponent.double()).float()
    angle = (torch.arange(positions, dtype=torch.float32)[:, None] * freq).double()
    return torch.cos(angle).float().double().cuda(), torch.sin(angle).float().double().cuda()


def _attend(q, k, v, scale, softcap=0.0, window=0):
    """Causal attention; q [tokens, heads, size], k and v [tokens, key heads, size], some heads and queries at a time."""
    tokens, heads, group = q.shape[0], q.shape[1], q.shape[1] // k.shape[1]
    out = torch.empty(tokens, heads, v.shape[-1], dtype=q.dtype, device=q.device)
    place = torch.arange(tokens, device=q.device)
    for head in range(k.shape[1]):
        of = slice(head * group, (head + 1) * group)
        for first in range(0, tokens, 2048):
            last = min(first + 2048, tokens)
            seen = place[first:last, None] >= place[None, :last]
            if window:
                seen &= place[first:last, None] - place[None, :last] < window
            score = torch.matmul(q[first:last, of].transpose(0, 1), k[:last, head].t()) * scale
            if softcap:
                score = softcap * torch.tanh(score / softcap)
            score = torch.softmax(score.masked_fill_(~seen, -math.inf), dim=-1)
            out[first:last, of] = torch.matmul(score, v[:last, head]).transpose(0, 1)
    return out


def _conv(x, taps, bias=None):
    count = taps.shape[1]
    padded = torch.cat([x.new_zeros(count - 1, x.shape[1]), x])
    out = sum(padded[j:j + x.shape[0]] * taps[:, j] for j in range(count))
    return _silu(out if bias is None else out + bias)


def _matrix_states(q, k, v, keep):
    """o_t = S_t^T q_t with S_t = keep_t S_(t-1) + k_t v_t^T; keep [tokens, heads, key channels or 1]."""
    state = torch.zeros(q.shape[1], q.shape[2], v.shape[2], dtype=q.dtype, device=q.device)
    rows = []
    for t in range(q.shape[0]):
        state = keep[t][:, :, None] * state + k[t][:, :, None] * v[t][:, None, :]
        rows.append(torch.bmm(q[t][:, None], state)[:, 0])
    return torch.stack(rows)


def _llama_rows(config, w, sequences):
    heads, kv, dim, eps = (config[k] for k in ("num_attention_heads", "num_key_value_heads", "head_dim", "rms_norm_eps"))
    spans, first = [], 0
    for ids in sequences:
        spans.append((first, first + len(ids)))
        first += len(ids)
    embed = w["model.embed_tokens.weight"].double()
    x = embed[torch.tensor([t for ids in sequences for t in ids], device="cuda")]
    cos, sin = _llama_angles(max(map(len, sequences)), dim, config["rope_theta"])
    for layer in range(config["num_hidden_layers"]):
        def of(name):
            return w[f"model.layers.{layer}.{name}.weight"].double()

        h = _rms(x, of("input_layernorm"), eps)
        q, k, v = ((h @ of(f"self_attn.{name}_proj").t()).view(-1, count, dim) for name, count in (("q", heads), ("k", kv), ("v", kv)))
        mixed = torch.cat([_attend(_turn(q[a:b], cos[:b - a], sin[:b - a]), _turn(k[a:b], cos[:b - a], sin[:b - a]), v[a:b], dim ** -0.5)
                           for a, b in spans])
        x = x + mixed.reshape(-1, heads * dim) @ of("self_attn.o_proj").t()
        h = _rms(x, of("post_attention_layernorm"), eps)
        x = x + (_silu(h @ of("mlp.gate_proj").t()) * (h @ of("mlp.up_proj").t())) @ of("mlp.down_proj").t()
    head = w["lm_head.weight"].double()
    return [_rms(x[b - 1:b], w["model.norm.weight"].double(), eps) @ head.t() for _, b in spans]


def _retention(h, p, m, eps):
    n, heads = h.shape[0], m["heads"]
    cos, sin = _angles(n, m["rot"])
    q, k = (_turn((h @ p[name].t()).view(n, heads, m["dim"]), cos, sin) for name in "qk")
    keep = torch.tensor(m["decay"], dtype=h.dtype, device=h.device)[None, :, None].expand(n, heads, 1)
    o = _matrix_states(q, k * m["dim"] ** -0.5, (h @ p["v"].t()).view(n, heads, m["vdim"]), keep)
    return (_rms(o, None, eps).reshape(n, -1) * _silu(h @ p["g"].t())) @ p["o"].t()


def _gated_linear(h, p, m, eps):
    n, heads, dim = h.shape[0], m["heads"], m["dim"]
    keep = torch.sigmoid((h @ p["a1"].t()) @ p["a2"].t() + p["a2.b"]).view(n, heads, dim) ** (1.0 / m["tau"])
    o = _matrix_states((h @ p["q"].t()).view(n, heads, dim) * dim ** -0.5, (h @ p["k"].t()).view(n, heads, dim),
                       (h @ p["v"].t()).view(n, heads, m["vdim"]), keep)
    return (_rms(o, p["norm"], eps).reshape(n, -1) * _silu(h @ p["g"].t())) @ p["o"].t()


def _keys_as_values(h, p, m, eps):
    n = h.shape[0]
    cos, sin = _angles(n, m["rot"])
    q, k = (h @ p["q"].t()).view(n, m["heads"], -1), (h @ p["k"].t()).view(n, m["kv_heads"], -1)
    out = _attend(_turn(q, cos, sin), _turn(k, cos, sin), k, m["scale"]) * torch.sigmoid(h @ p["g"].t())[:, :, None]
    return out.reshape(n, -1) @ p["o"].t()


def _delta_rule(h, p, m, eps):
    n, heads, groups = h.shape[0], m["heads"], m["kv_heads"]
    q, k, v = (_conv(h @ p[name].t(), p[name + ".conv"]).view(n, count, -1) for name, count in (("q", groups), ("k", groups), ("v", heads)))
    q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * m["dim"] ** -0.5
    k = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    q, k = (x.repeat_interleave(heads // groups, dim=1) for x in (q, k))
    beta = torch.sigmoid(h @ p["b"].t())
    keep = torch.exp(-torch.exp(p["A_log"]) * torch.nn.functional.softplus(h @ p["a"].t() + p["dt_bias"], threshold=1e9))
    state = torch.zeros(heads, m["dim"], m["vdim"], dtype=h.dtype, device=h.device)
    rows = []
    for t in range(n):
        state = keep[t][:, None, None] * state
        u = beta[t][:, None] * (v[t] - torch.bmm(k[t][:, None], state)[:, 0])
        state = state + k[t][:, :, None] * u[:, None]
        rows.append(torch.bmm(q[t][:, None], state)[:, 0])
    o = _rms(torch.stack(rows), p["norm"], eps).reshape(n, -1)
    return (o * _silu(h @ p["g"].t())) @ p["o"].t()


def _latent(h, p, m, eps):
    n, heads, dim, rank = h.shape[0], m["heads"], m["dim"], m["kv_rank"]
    cos, sin = _angles(n, m["rot"])
    q = (h @ p["q"].t()).view(n, heads, -1)
    down = h @ p["dkv"].t()
    c, shared = _rms(down[:, :rank], p["dkv.norm"], eps), _turn(down[:, None, rank:], cos, sin, neighbours=True)
    k = torch.cat([(c @ p["uk"].t()).view(n, heads, dim), shared.expand(n, heads, -1)], dim=-1)
    q = torch.cat([q[..., :dim], _turn(q[..., dim:], cos, sin, neighbours=True)], dim=-1)
    out = _attend(q, k, (c @ p["uv"].t()).view(n, heads, -1), m["scale"], window=m["mask"]["size"])
    return (out.reshape(n, -1) * torch.sigmoid(h @ p["g"].t())) @ p["o"].t()


def _capped(h, p, m, eps):
    n = h.shape[0]
    cos, sin = _angles(n, m["rot"])
    q, k, v = ((h @ p[name].t() + p[name + ".b"]).view(n, count, -1) for name, count in (("q", m["heads"]), ("k", m["kv_heads"]), ("v", m["kv_heads"])))
    out = _attend(_turn(q, cos, sin), _turn(k, cos, sin), v, m["scale"], softcap=m["softcap"])
    return out.reshape(n, -1) @ p["o"].t() + p["o.b"]


def _scan(h, p, m, eps):
    n, states, rank = h.shape[0], m["state"], m["dt_rank"]
    x, z = (h @ p["in"].t()).split(m["inner"], dim=1)
    x = _conv(x, p["conv"], p["conv.b"])
    dt, b, c = (x @ p["x"].t()).split([rank, states, states], dim=1)
    dt = torch.nn.functional.softplus(dt @ p["dt"].t() + p["dt.b"], threshold=1e9)
    rate = -torch.exp(p["A_log"])
    state = torch.zeros_like(rate)
    rows = []
    for t in range(n):
        state = torch.exp(dt[t][:, None] * rate) * state + (dt[t] * x[t])[:, None] * b[t]
        rows.append(state @ c[t])
    return ((torch.stack(rows) + p["D"] * x) * _silu(z)) @ p["o"].t()


def _part(w, prefix):
    return {name[len(prefix):]: t for name, t in w.items() if name.startswith(prefix)}


def _mafalorn_rows(config, w, ids):
    eps = config["norm"]["eps"]
    x = w["embed"][ids]
    for index, layer in enumerate(config["layers"]):
        own, m = _part(w, f"l{index}."), layer["mixer"]
        h, p = _rms(x, own["norm1"], eps), _part(own, "mix.")
        if layer["type"] == "parallel":
            y = m["left_scale"] * _keys_as_values(h, _part(p, "left."), m["left"], eps) + m["right_scale"] * _delta_rule(h, _part(p, "right."), m["right"], eps)
        else:
            y = {"retention": _retention, "latent_attention": _latent}[layer["type"]](h, p, m, eps)
        x = x + _rms(y, own["norm1b"], eps)
    return (_rms(x, w["final.norm"], eps) @ w["head"].t()) * config["logit_scale"]


def _zifunex_rows(config, w, ids):
    eps, bigram = config["norm"]["eps"], config["embedding"]["bigram"]
    pairs = torch.cat([ids.new_tensor([bigram["buckets"]]), (ids[:-1] * bigram["mul_prev"] + ids[1:] * bigram["mul_cur"]) % bigram["buckets"]])
    streams = (w["embed"][ids] + w["bigram"][pairs])[None].repeat(config["streams"], 1, 1)
    for index, layer in enumerate(config["layers"]):
        own, m = _part(w, f"l{index}."), layer["mixer"]
        for number, share in ((1, _part(own, "hc1.")), (2, _part(own, "hc2."))):
            if not share or (number == 2 and layer["mlp"] is None):
                continue
            h = _layer_norm(torch.einsum("s,stw->tw", share["in"], streams), own[f"norm{number}"], own[f"norm{number}.b"], eps)
            if number == 2:
                p = _part(own, "mlp.")
                y = (torch.nn.functional.gelu(h @ p["gate"].t(), approximate="tanh") * (h @ p["up"].t())) @ p["down"].t()
            elif layer["type"] == "gla":
                y = _gated_linear(h, _part(own, "mix."), m, eps)
            else:
                p = _part(own, "mix.")
                y = 0.5 * (_rms(_capped(h, _part(p, "left."), m["left"], eps), p["left.out"], eps)
                           + _rms(_scan(h, _part(p, "right."), m["right"], eps), p["right.out"], eps))
            streams = torch.einsum("sr,stw->rtw", share["mix"], streams) + share["out"][:, None, None] * y
    return _layer_norm(streams.sum(0), w["final.norm"], w["final.norm.b"], eps) @ w["head"].t()


def exact(case, seed):
    config = _config(case)
    _, spec = spec_from_config(config)
    w = _weights(DecoderModel(spec), seed)  # (the names and shapes of the design's tensors)
    sequences = _tokens(case, seed, spec.vocab_size)
    if case["model"] in LLAMAS:
        rows = torch.cat(_llama_rows(config, w, [ids for ids, _ in sequences]))
        return {"logits": rows, "tokens": None} if case.get("sampled") else {"logits": rows}
    w = {name: t.double() for name, t in w.items()}
    whole = {"mafalorn": _mafalorn_rows, "zifunex": _zifunex_rows}[case["model"]]
    rows = [(whole(config, w, torch.tensor(ids, device="cuda")), n) for ids, n in sequences]
    out = {"prompt": torch.stack([r[n - 1] for r, n in rows])}
    out.update({f"step{i}": torch.stack([r[n + i] for r, n in rows]) for i in range(case["new"])})
    return out
