"""What a user of this library has it do, as cases whose time is measured.

A server of a model calls ``Engine.step`` and ``DeviceSampler.sample`` all day: decode steps of one to some dozens of
sequences over contexts of all lengths, prompts from a line to a book, alone or several at once.  A case is one such call
with its sampling: ``kind`` "decode" (one token for each of ``sequences`` sequences that hold ``shortest`` to ``longest``
tokens), "prompt" (as many whole prompts in one step, from empty slots to the choice of their first tokens) or "sample"
(the choice alone).  The model's weights are made once and its engine is kept, as a server keeps them; sequences come from
the seed.

The designs are the dense Qwen3 sizes that the benchmark names, and two of the other presets: Nirotar (windowed
attention with a sink, attention over compressed rows, experts by a table) and Sebesun (retention, selective scan,
differential attention).  Designs whose router scores its experts are left out: where two scores nearly tie, another order
of the same sums takes another expert, and whole logits then say nothing.  For the same reason a step's logits are
returned and not the tokens drawn from them (two of 151,936 logits are often closer than bfloat16 tells apart); the
"sample" cases return tokens, for logits that are given.
"""
from __future__ import annotations

import math
import random
import zlib

import torch

from palm_infra_amd.config import config_from_dict, preset_dict
from palm_infra_amd.engine import Engine, FedTokens, StepEntry
from palm_infra_amd.sampling import DeviceSampler, SamplingParams, SequenceSampling
from palm_infra_amd.weights import Weights

DEVICE = "cuda:0"
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}
GROWTH = 1024                # tokens that a decoding sequence grows by before it ends and another takes its place
FED = 64                     # decode steps after which the tokens that are fed come round again


def _case(name, kind, model, sequences, shortest, longest=None, temperature=0.6, dtype="bfloat16"):
    return {"name": name, "kind": kind, "model": model, "dtype": dtype, "sequences": sequences, "shortest": shortest,
            "longest": longest or shortest, "temperature": temperature}


def listed():
    return [
        # choosing the next tokens of a batch with the default options, from logits that are there
        _case("sample_33", "sample", "qwen3-8b", 33, 1),
        # one user's chat: the latency of a single token
        _case("decode_1", "decode", "qwen3-8b", 1, 777),
        # a small batch in the middle of its documents: the benchmark's headline
        _case("decode_8", "decode", "qwen3-8b", 8, 2048, temperature=0.0),
        # a busy server: many chats of all lengths
        _case("decode_45_ragged", "decode", "qwen3-8b", 45, 70, 1500),
        # the benchmark's batch of unequal requests at the next size
        _case("decode_16_ragged_14b", "decode", "qwen3-14b", 16, 64, 2048),
        # a question of a few lines: the time to the first token
        _case("prompt_91", "prompt", "qwen3-8b", 1, 91),
        # requests that arrived together
        _case("prompts_5_ragged", "prompt", "qwen3-8b", 5, 64, 2048),
        # a long document
        _case("prompt_13331", "prompt", "qwen3-8b", 1, 13331),
        # the 32-bit mode, in which results are checked
        _case("prompt_157_float32", "prompt", "qwen3-8b", 1, 157, dtype="float32", temperature=0.0),
        # experts and compressed rows: a document, and a small batch
        _case("nirotar_prompt_2900", "prompt", "nirotar-4096", 1, 2900),
        _case("nirotar_decode_6", "decode", "nirotar-4096", 6, 300, 3000),
        # recurrences and differential attention: documents that arrived together
        _case("sebesun_prompts_3", "prompt", "sebesun-4096", 3, 200, 2300),
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "prompt", "sample"])
    model = rng.choice(["qwen3-8b", "qwen3-8b", "qwen3-14b", "nirotar-2048", "nirotar-4096", "sebesun-2048", "sebesun-4096"])
    temperature = rng.choice([0.0, 0.6, 0.6, 1.0])
    if kind == "sample":
        case = _case("", kind, model, _spread(rng, 1, 64), 1, temperature=temperature)
    else:
        sequences = _spread(rng, 1, 64) if kind == "decode" else _spread(rng, 1, 8)
        longest = min(_spread(rng, 16, 8192), (16384 if kind == "decode" else 7600) // sequences)
        shortest = longest if rng.random() < 0.3 else rng.randint(max(1, longest // 8), longest)
        dtype = "float32" if rng.random() < 0.1 and model != "qwen3-14b" else "bfloat16"
        if dtype == "float32":                                  # the mode for checks: short and few
            sequences, longest = min(sequences, 6), min(longest, 256 // min(sequences, 6))
            shortest = min(shortest, longest)
        case = _case("", kind, model, sequences, shortest, longest, temperature, dtype)
    del case["name"]
    return case


# ---- weights ------------------------------------------------------------------------------------------------------

def _init(model, name, role, init, layers):
    """(mean, standard deviation) of a tensor.  Qwen3: a stream of unit scale to which every branch adds its share of
    the depth, and scores that prefer some keys, as trained models have them; else the design's own."""
    _, mean, std = init
    if model.startswith("qwen3"):
        if "embed_tokens" in name:
            return 0.0, 1.0
        if "o_proj" in name or "down_proj" in name:
            return 0.0, 0.02 / math.sqrt(2.0 * layers)
        if "q_norm" in name or "k_norm" in name:
            return 1.5, 0.1
    return mean, std


def _stored(model, dtype, name, shape, role, init, layers):
    """The checkpoint's tensor ``name``: numbers that depend on the name alone."""
    g = torch.Generator(device=DEVICE).manual_seed(zlib.crc32(name.encode()))
    if role == "integer":
        return torch.rand((shape[0], init[1]), device=DEVICE, generator=g).argsort(dim=1)[:, :shape[1]].to(torch.int32)
    mean, std = _init(model, name, role, init, layers)
    t = torch.randn(tuple(shape), device=DEVICE, generator=g).mul_(std).add_(mean)
    return t if role == "vector" else t.to(DTYPES[dtype])


class _Checkpoint:
    """The tensors of a model by their names in a checkpoint, each made when it is asked for."""

    def __init__(self, model, dtype):
        self.model, self.dtype = model, dtype
        self.config = config_from_dict(preset_dict(model))
        self.spec = self.config.spec()
        self.plan = {name: (shape, ref.role, ref.init) for ref in self.spec.tensor_refs() for name, shape in ref.stored_shapes()}

    def __getitem__(self, name):
        return _stored(self.model, self.dtype, name, *self.plan[name], len(self.spec.layers))

    def weights(self):
        out = {}
        for ref in self.spec.tensor_refs():
            pieces = []
            for name, _, how in ref.pieces():
                t = self[name]
                if how is not None:
                    t = t if how.rows is None else t[how.rows[0]:how.rows[1]]
                    t = t.t() if how.transposed else t
                pieces.append(t)
            out[ref.key] = pieces[0].contiguous() if len(pieces) == 1 else torch.cat(pieces)
        return Weights(out)


_kept = {}                   # the one model and the one engine that the program runs at a time


def _engine(case):
    model, dtype = case["model"], case["dtype"]
    if _kept.get("model") != (model, dtype):
        _kept.clear()
        torch.cuda.empty_cache()
        checkpoint = _Checkpoint(model, dtype)
        _kept.update(model=(model, dtype), spec=checkpoint.spec, config=checkpoint.config, weights=checkpoint.weights())
    lengths = _lengths(case)
    # room for the sequences of four states of this program side by side (a prompt's are closed when its pass ends)
    room = sum((n + GROWTH + 127) // 64 * 64 for n in lengths) * 4 if case["kind"] == "decode" else sum((n + 127) // 64 * 64 for n in lengths)
    sized = (case["kind"], len(lengths), room)
    if _kept.get("sized") != sized:
        _kept.pop("engine", None)
        torch.cuda.empty_cache()
        _kept.update(sized=sized, engine=Engine(_kept["config"], _kept["spec"], _kept["weights"], DTYPES[dtype], max_tokens=room,
                                                max_seqs=4 * len(lengths) + 1, device=DEVICE))
    return _kept["engine"]


# ---- inputs -------------------------------------------------------------------------------------------------------

def _vocab(raw):
    return raw.get("vocab_size") or raw["vocab"]


def _lengths(case):
    if case["shortest"] == case["longest"]:
        return [case["longest"]] * case["sequences"]
    rng = random.Random("%(sequences)d %(shortest)d %(longest)d" % case)
    return [rng.randint(case["shortest"], case["longest"]) for _ in range(case["sequences"])]


def _tokens(case, seed):
    """(each sequence's tokens, the tokens that decode steps feed [FED][sequences])"""
    rng, vocab = random.Random(seed), _vocab(preset_dict(case["model"]))
    return ([[rng.randrange(vocab) for _ in range(n)] for n in _lengths(case)],
            [[rng.randrange(vocab) for _ in range(case["sequences"])] for _ in range(FED)])


class _State:
    """What a program holds for a case's calls."""

    def __init__(self, case, seed):
        self.kind = case["kind"]
        self.sampler = DeviceSampler(SamplingParams(temperature=case["temperature"]))
        self.samplings = [SequenceSampling(stream=i) for i in range(case["sequences"])]
        self.engine, self.slots = None, []
        if self.kind == "sample":
            g = torch.Generator(device=DEVICE).manual_seed(seed)
            self.logits = torch.randn((case["sequences"], _vocab(preset_dict(case["model"]))), device=DEVICE, generator=g).mul_(3.0)
            return
        self.engine = _engine(case)
        self.prompts, fed = _tokens(case, seed)
        self.fed = torch.tensor(fed, dtype=torch.int32).to(DEVICE)
        if self.kind == "decode":
            self.start()

    def start(self):
        """Sequences that hold their contexts."""
        self.stop()
        self.slots = [self.engine.open() for _ in self.prompts]
        self.engine.step([StepEntry(s, p, []) for s, p in zip(self.slots, self.prompts)])
        self.steps = 0

    def stop(self):
        for s in self.slots:
            self.engine.close(s)
        self.slots = []

    def __del__(self):
        self.stop()


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    if state.kind == "sample":
        return {"tokens": state.sampler.sample(state.logits, state.samplings)}
    engine = state.engine
    if state.kind == "prompt":
        slots = [engine.open() for _ in state.prompts]
        logits = engine.step([StepEntry(s, p, [len(p) - 1]) for s, p in zip(slots, state.prompts)])
        state.tokens = state.sampler.sample(logits, state.samplings)
        for s in slots:
            engine.close(s)
        return {"logits": logits}
    if state.steps == GROWTH:
        state.start()
    ids = state.fed[state.steps % FED]
    state.steps += 1
    logits = engine.step([StepEntry(s, [0], [0]) for s in state.slots], fed=FedTokens(ids, list(range(len(state.slots)))))
    state.tokens = state.sampler.sample(logits, state.samplings)
    return {"logits": logits}


# ---- what a pass cannot do without --------------------------------------------------------------------------------

def _layers(raw):
    """Of each layer: matrix elements that every token meets; experts (count, chosen, elements of one); elements cached for
    a position and read again by a query; multiply-adds for a query and a key; window; elements of the state of a sequence."""
    out = []
    if "hidden_size" in raw:
        H, I, hd = raw["hidden_size"], raw["intermediate_size"], raw["head_dim"]
        nh, nkv = raw["num_attention_heads"], raw["num_key_value_heads"]
        return [{"matrix": H * hd * 2 * (nh + nkv) + 3 * H * I, "row": 2 * nkv * hd, "pair": 2 * nh * hd}] * raw["num_hidden_layers"]
    W = raw["width"]
    for layer in raw["layers"]:
        m, f, kind = layer["mixer"], layer.get("mlp"), layer["type"]
        if kind == "latent_attention":
            H, d, dr, dv, R = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
            own = 0 if m.get("kv_from") is not None else W * (R + dr)
            one = {"matrix": W * H * (d + dr) + own + R * H * (d + dv) + W * H * dv, "row": R + dr, "pair": H * (d + dr + dv)}
        elif kind == "mamba1":
            C, N, rank = m["inner"], m["state"], m["dt_rank"]
            one = {"matrix": 3 * W * C + C * (2 * rank + 2 * N), "state": C * N + C * m["conv"]}
        elif kind == "retention":
            H, d, dv = m["heads"], m["dim"], m["vdim"]
            one = {"matrix": W * H * (2 * d + 3 * dv), "state": H * d * dv}
        else:
            H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            maps = 2 if "diff" in m else 1
            one = {"matrix": W * (maps * (H + G) * d + G * dv + H * dv), "row": G * (maps * d + dv), "pair": H * (maps * d + maps * dv)}
        one["window"] = m["mask"]["size"] if m.get("mask") else None
        if f and f["kind"] == "moe":
            one["experts"] = (f["router"]["experts"], f["router"]["top"], 2 * W * f["expert"]["ff"])
            one["matrix"] += 2 * W * f["shared"]["ff"] if f.get("shared") else 0
        elif f:
            one["matrix"] += 2 * W * f["ff"]
        out.append(one)
    return out


def work(case):
    raw, lengths = preset_dict(case["model"]), _lengths(case)
    B, vocab = len(lengths), _vocab(raw)
    if case["kind"] == "sample":
        return {"bytes": 4.0 * B * (vocab + 1), "flops": 0.0}
    size, width = (4 if case["dtype"] == "float32" else 2), raw.get("hidden_size") or raw["width"]
    decode = case["kind"] == "decode"
    new = B if decode else sum(lengths)
    nbytes = vocab * width * size + B * vocab * 4.0 + new * width * size
    flops = 2.0 * B * vocab * width
    for one in _layers(raw):
        nbytes += one["matrix"] * size
        flops += 2.0 * new * one["matrix"]
        if one.get("experts"):
            count, top, each = one["experts"]
            nbytes += size * each * count * (1.0 - (1.0 - top / count) ** new)
            flops += 2.0 * new * top * each
        if one.get("row"):
            window = one.get("window") or max(lengths) + 1
            pairs = sum(min(n + 1, window) if decode else sum(min(p + 1, window) for p in range(n)) for n in lengths)
            nbytes += size * one["row"] * (pairs if decode else new)
            flops += 2.0 * one["pair"] * pairs
        if one.get("state"):
            nbytes += 4.0 * one["state"] * B * (2 if decode else 1)
            flops += 4.0 * one["state"] * new
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"
    # against 64 bits: 1.3e-6 in 32 bits, 5e-3 to 8e-3 in bfloat16 (36 and 40 layers of Qwen3, 8 of Nirotar), 1.0e-2 to 1.3e-2
    # for Sebesun, whose norms sit on the branches' outputs
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 2e-4}
    return {"rel": 0.03 if case["model"].startswith("sebesun") else 0.02, "max": 0.3}


# ---- the same in 64 bits ------------------------------------------------------------------------------------------

F64 = torch.float64


def _norm(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rotate(x, freq, dims, halves):
    """x [T, heads, n]: pairs of the first ``dims`` dimensions (i with i + dims/2, or neighbours) turn by position times
    frequency."""
    a = torch.arange(x.shape[0], dtype=F64, device=x.device)[:, None] * freq
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    out = x.clone()
    first = slice(0, dims // 2) if halves else slice(0, dims, 2)
    second = slice(dims // 2, dims) if halves else slice(1, dims, 2)
    u, v = x[..., first], x[..., second]
    out[..., first], out[..., second] = u * c - v * s, v * c + u * s
    return out


def _frequencies(dims, base, scaling=None):
    out = []
    for i in range(dims // 2):
        f = base ** (-2.0 * i / dims)
        if scaling:
            wavelength = 2.0 * math.pi / f
            factor, low, high, original = (float(scaling[k]) for k in ("factor", "low", "high", "original"))
            if wavelength > original / low:
                f /= factor
            elif wavelength >= original / high:
                s = (original / wavelength - low) / (high - low)
                f = (1.0 - s) * f / factor + s * f
        out.append(f)
    return torch.tensor(out, dtype=F64, device=DEVICE)


def _attend(q, k, v, scale, window=None, sink=None):
    """q [T, H, d], k [T, G, d], v [T, G, dv] of one sequence -> [T, H, dv]; ``sink`` [H]: one more term of the softmax's
    denominator."""
    T, H, d = q.shape
    G, dv = k.shape[1], v.shape[2]
    out = torch.empty((T, H, dv), dtype=F64, device=q.device)
    rows = max(16, int(1.5e8 / (H * T)))
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    for lo in range(0, T, rows):
        hi = min(T, lo + rows)
        begin = 0 if window is None else max(0, lo - window + 1)
        i, j = torch.arange(lo, hi, device=q.device)[:, None], torch.arange(begin, hi, device=q.device)
        hidden = j > i
        if window is not None:
            hidden = hidden | (i - j >= window)
        qs = q[lo:hi].reshape(hi - lo, G, H // G, d).permute(1, 2, 0, 3).reshape(G, -1, d)
        s = (qs @ kt[:, :, begin:hi]).mul_(scale).view(H, hi - lo, hi - begin).masked_fill_(hidden, -math.inf)
        top = s.amax(dim=2, keepdim=True)
        if sink is not None:
            top = torch.maximum(top, sink[:, None, None])
        s = s.sub_(top).exp_()
        total = s.sum(dim=2, keepdim=True)
        if sink is not None:
            total = total + torch.exp(sink[:, None, None] - top)
        s.div_(total)
        o = s.view(G, -1, hi - begin) @ vt[:, begin:hi]
        out[lo:hi] = o.view(H, hi - lo, dv).transpose(0, 1)
    return out


def _exact_qwen3(raw, w, x, ids, cuts):
    H, I, hd, eps = raw["hidden_size"], raw["intermediate_size"], raw["head_dim"], raw["rms_norm_eps"]
    nh, nkv = raw["num_attention_heads"], raw["num_key_value_heads"]
    freq = _frequencies(hd, raw["rope_theta"])
    for i in range(raw["num_hidden_layers"]):
        p = "model.layers.%d." % i
        a = p + "self_attn."
        h = _norm(x, w(p + "input_layernorm.weight"), eps)
        q = _norm((h @ w(a + "q_proj.weight").T).view(-1, nh, hd), w(a + "q_norm.weight"), eps)
        k = _norm((h @ w(a + "k_proj.weight").T).view(-1, nkv, hd), w(a + "k_norm.weight"), eps)
        v = (h @ w(a + "v_proj.weight").T).view(-1, nkv, hd)
        o = torch.cat([_attend(_rotate(q[lo:hi], freq, hd, True), _rotate(k[lo:hi], freq, hd, True), v[lo:hi], hd ** -0.5) for lo, hi in cuts])
        x = x + o.view(-1, nh * hd) @ w(a + "o_proj.weight").T
        h = _norm(x, w(p + "post_attention_layernorm.weight"), eps)
        x = x + (torch.nn.functional.silu(h @ w(p + "mlp.gate_proj.weight").T) * (h @ w(p + "mlp.up_proj.weight").T)) @ w(p + "mlp.down_proj.weight").T
    return _norm(x[[hi - 1 for _, hi in cuts]], w("model.norm.weight"), eps), "lm_head.weight"


def _exact_nirotar(raw, w, x, ids, cuts):
    eps, shelf = raw["norm"]["eps"], {}

    def rotated(t, rot):
        freq = _frequencies(rot["dims"], rot["base"], rot.get("scaling"))
        return torch.cat([_rotate(t[lo:hi], freq, rot["dims"], False) for lo, hi in cuts])

    for i, layer in enumerate(raw["layers"]):
        p, m, f = "l%d.mix." % i, layer["mixer"], layer.get("mlp")
        h = _norm(x, w("l%d.norm1" % i), eps)
        heads, d, dv = m["heads"], m["dim"], m["vdim"]
        if layer["type"] == "attention":
            q, k = (rotated((h @ w(p + n).T).view(-1, c, d), m["rot"]) for n, c in (("q", heads), ("k", m["kv_heads"])))
            v = (h @ w(p + "v").T).view(-1, m["kv_heads"], dv)
        else:
            R, dr = m["kv_rank"], m["rot_dim"]
            if m.get("kv_from") is None:
                down = h @ w(p + "dkv").T
                shelf[i] = _norm(down[:, :R], w(p + "dkv.norm"), eps), rotated(down[:, None, R:], m["rot"])
            c, r = shelf[i if m.get("kv_from") is None else m["kv_from"]]
            q = (h @ w(p + "q").T).view(-1, heads, d + dr)
            q = torch.cat([q[..., :d], rotated(q[..., d:].contiguous(), m["rot"])], dim=-1)
            k = torch.cat([(c @ w(p + "uk").T).view(-1, heads, d), r.expand(-1, heads, dr)], dim=-1)
            v = (c @ w(p + "uv").T).view(-1, heads, dv)
        window, sink = (m["mask"]["size"] if m.get("mask") else None), w(p + "sink")
        o = torch.cat([_attend(q[lo:hi], k[lo:hi], v[lo:hi], m["scale"], window, sink) for lo, hi in cuts])
        x = x + o.view(-1, heads * dv) @ w(p + "o").T
        if f is not None:
            p = "l%d.mlp." % i
            h = _norm(x, w("l%d.norm2" % i), eps)
            chosen = w(p + "table")[ids].long()
            y = torch.relu(h @ w(p + "shared.up").T).square_() @ w(p + "shared.down").T if f.get("shared") else torch.zeros_like(x)
            for e in range(f["router"]["experts"]):
                rows = (chosen == e).any(dim=1).nonzero()[:, 0]
                y[rows] += torch.relu(h[rows] @ w("%se%d.up" % (p, e)).T).square_() @ w("%se%d.down" % (p, e)).T / f["router"]["top"]
            x = x + y
    return _norm(x[[hi - 1 for _, hi in cuts]], w("final.norm"), eps), "head"


def _exact_sebesun(raw, w, x, ids, cuts):
    eps = raw["norm"]["eps"]

    def unit(y):
        return y / torch.sqrt((y * y).mean(-1, keepdim=True) + eps)

    def retention(h, p, m):
        heads, d, dv = m["heads"], m["dim"], m["vdim"]
        q, k, v = ((h @ w(p + n).T).view(-1, heads, c) for n, c in (("q", d), ("k", d), ("v", dv)))
        out = torch.empty_like(v)
        decay = torch.tensor(m["decay"], dtype=F64, device=h.device)
        for lo, hi in cuts:
            a, b = q[lo:hi], k[lo:hi]
            if m.get("rot"):
                freq = _frequencies(m["rot"]["dims"], m["rot"]["base"])
                a, b = (_rotate(t, freq, m["rot"]["dims"], True) for t in (a, b))
            i = torch.arange(hi - lo, device=h.device, dtype=F64)
            for n in range(heads):
                passed = (i[:, None] - i).clamp_(min=0.0)
                weight = torch.tril((a[:, n] @ b[:, n].T).mul_(decay[n] ** passed)) * d ** -0.5
                out[lo:hi, n] = weight @ v[lo:hi, n]
        return (unit(out).view(-1, heads * dv) * torch.nn.functional.silu(h @ w(p + "g").T)) @ w(p + "o").T

    def mamba1(h, p, m):
        C, N, rank, taps = m["inner"], m["state"], m["dt_rank"], m["conv"]
        x_z = h @ w(p + "in").T
        A, skip, conv, bias = -torch.exp(w(p + "A_log")), w(p + "D"), w(p + "conv"), w(p + "conv.b")
        y = torch.empty((h.shape[0], C), dtype=F64, device=h.device)
        for lo, hi in cuts:
            padded = torch.cat([torch.zeros((taps - 1, C), dtype=F64, device=h.device), x_z[lo:hi, :C]])
            u = torch.nn.functional.silu(sum(padded[j:j + hi - lo] * conv[:, j] for j in range(taps)) + bias)
            low = u @ w(p + "x").T
            dt = torch.nn.functional.softplus(low[:, :rank] @ w(p + "dt").T + w(p + "dt.b"))
            S = torch.zeros((C, N), dtype=F64, device=h.device)
            grown = dt * u
            for t in range(hi - lo):
                S = torch.exp(dt[t][:, None] * A) * S + grown[t][:, None] * low[t, rank:rank + N]
                y[lo + t] = S @ low[t, rank + N:]
            y[lo:hi] += skip * u
        return (y * torch.nn.functional.silu(x_z[:, C:])) @ w(p + "o").T

    def attention(h, p, m):
        heads, groups, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q = _norm((h @ w(p + "q").T).view(-1, heads, 2, d), w(p + "q.norm"), eps)
        k = _norm((h @ w(p + "k").T).view(-1, groups, 2, d), w(p + "k.norm"), eps)
        v = (h @ w(p + "v").T).view(-1, groups, dv)
        apart = torch.exp((w(p + "lq1") * w(p + "lk1")).sum()) - torch.exp((w(p + "lq2") * w(p + "lk2")).sum()) + m["diff"]
        o = torch.cat([_attend(q[lo:hi, :, 0], k[lo:hi, :, 0], v[lo:hi], m["scale"]) - apart * _attend(q[lo:hi, :, 1], k[lo:hi, :, 1], v[lo:hi], m["scale"])
                       for lo, hi in cuts])
        return (unit(o) * (1.0 - m["diff"])).reshape(-1, heads * dv) @ w(p + "o").T

    mixers = {"retention": retention, "mamba1": mamba1, "attention": attention}
    results = [x]
    for i, layer in enumerate(raw["layers"]):
        p = "l%d." % i
        x = x + _norm(mixers[layer["type"]](x, p + "mix.", layer["mixer"]), w(p + "norm1"), eps)
        if layer.get("mlp"):
            a, b = torch.nn.functional.softplus(w(p + "mlp.act"))
            z = x @ w(p + "mlp.up").T
            z = torch.where(z > 0, a * z * z, (0.5 + b) * (torch.expm1(z.clamp(max=0.0)) - z)) + 0.5 * z
            x = x + _norm(z @ w(p + "mlp.down").T, w(p + "norm2"), eps)
        results.append(x)
        c = w(p + "dwa")
        x = sum(c[j] * results[j] for j in range(i + 2))
    return _norm(x[[hi - 1 for _, hi in cuts]], w("final.norm"), eps), "head"


def exact(case, seed):
    if case["kind"] == "sample":
        return None                                             # tokens: whole numbers
    raw, checkpoint = preset_dict(case["model"]), _Checkpoint(case["model"], case["dtype"])
    if case["model"].startswith("sebesun") and sum(_lengths(case)) > 12000:
        return None                                             # a scan token by token: over 20 seconds

    def w(name):
        return checkpoint[name].to(F64)

    sequences, fed = _tokens(case, seed)
    if case["kind"] == "decode":
        sequences = [s + [t] for s, t in zip(sequences, fed[0])]
    ends = [sum(len(s) for s in sequences[:i + 1]) for i in range(len(sequences))]
    cuts = [(e - len(s), e) for s, e in zip(sequences, ends)]
    ids = torch.tensor([t for s in sequences for t in s], device=DEVICE)
    forward = {"qwen3": _exact_qwen3, "nirotar": _exact_nirotar, "sebesun": _exact_sebesun}[case["model"].split("-")[0]]
    x = checkpoint["model.embed_tokens.weight" if case["model"].startswith("qwen3") else "embed"][ids].to(F64)
    h, head = forward(raw, w, x, ids, cuts)
    table = checkpoint[head]
    return {"logits": torch.cat([h @ part.to(F64).T for part in table.split(32768)], dim=1)}
