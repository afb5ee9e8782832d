"""What a user of this framework has it do, as cases that can be timed and compared.

A case of kind ``step`` is one pass of the step function (``StepRunner.step``): ``decoding``
requests that live in the cache bring one token each, and ``prompts`` new requests bring a prompt of
``prompt`` tokens, whole or in portions of ``portion``.  The logits of every request's last token
come back.  A case of kind ``generate`` is one ``Engine.generate`` call, prompts in and token ids out.

Weights are seeded random ones of the named layer shapes; they stay in memory from one state to the
next, as a serving program keeps its model.  Requests, tokens and cache follow from a state's seed.
The embedding is drawn wider than the other matrices, so that the logits have a clear largest value,
as a trained model's have.
"""
import gc
import math
import zlib

import numpy as np
import torch

from zse_amd.config.base import resolve_architecture
from zse_amd.engine.engine import Engine
from zse_amd.engine.loading import random_model
from zse_amd.engine.model import Model
from zse_amd.engine.runner import StepEntry, StepRunner
from zse_amd.runtime.device import Runtime
from zse_amd.sampling import SamplingParams

PAGE = 16                # tokens of a cache page, the engine's default
STEP_TOKENS = 4096       # most tokens of a step, the engine's default
LONGEST = 8192           # Gemma 2's positions
NEW_TOKENS = 256         # a decoding request ends after so many, and another takes its place
WEIGHT_SEED = 0

GEMMA2_2B = dict(
    architectures=["Gemma2ForCausalLM"], model_type="gemma2", num_hidden_layers=26, hidden_size=2304,
    num_attention_heads=8, num_key_value_heads=4, head_dim=256, query_pre_attn_scalar=256,
    intermediate_size=9216, vocab_size=256000, rope_theta=10000.0, sliding_window=4096,
    attn_logit_softcapping=50.0, final_logit_softcapping=30.0, rms_norm_eps=1e-6,
    max_position_embeddings=LONGEST)
GEMMA2_9B = dict(GEMMA2_2B, num_hidden_layers=42, hidden_size=3584, num_attention_heads=16, num_key_value_heads=8,
                 intermediate_size=14336)
GEMMA2_27B = dict(GEMMA2_2B, num_hidden_layers=46, hidden_size=4608, num_attention_heads=32, num_key_value_heads=16,
                  head_dim=128, query_pre_attn_scalar=144, intermediate_size=36864)


def _small_gemma2(width, heads, kv_heads, ff, window):
    """Six Gemma 2 layers of another width (the sizes that bench.py sets other designs beside)."""
    return dict(GEMMA2_2B, num_hidden_layers=6, hidden_size=width, num_attention_heads=heads, num_key_value_heads=kv_heads,
                head_dim=128, query_pre_attn_scalar=128, intermediate_size=ff, vocab_size=32768, sliding_window=window)


def _dafotar(width, heads, kv_heads, ff, window):
    """Six Dafotar layers, as bench.py lists them: attention, mLSTM, attention on the first one's keys, twice."""
    att = {"heads": heads, "kv_heads": kv_heads, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
           "mask": {"size": window}, "rot": {"base": 10000.0, "dims": 64}}
    rec = {"heads": heads, "dim": 64, "vdim": 128, "gate_cap": 10.0}
    layers = []
    for g in range(2):
        layers += [{"type": "attention", "mixer": dict(att), "mlp": {"kind": "dense", "ff": ff}},
                   {"type": "mlstm", "mixer": dict(rec), "mlp": None},
                   {"type": "attention", "mixer": dict(att, kv_from=3 * g), "mlp": {"kind": "dense", "ff": ff}}]
    return {"architecture": "Dafotar", "vocab": 32768, "width": width, "norm": {"eps": 1e-6}, "streams": 4,
            "canon": {"taps": 4}, "layers": layers}


MODELS = {
    "gemma2-w1024": _small_gemma2(1024, 8, 2, 4096, 1024),
    "gemma2-w2048": _small_gemma2(2048, 16, 4, 8192, 2048),
    "gemma2-2b": GEMMA2_2B, "gemma2-9b": GEMMA2_9B, "gemma2-27b": GEMMA2_27B,
    "dafotar-w1024": _dafotar(1024, 8, 2, 4096, 1024),
    "dafotar-w2048": _dafotar(2048, 16, 4, 8192, 2048),
}
GAIN_STD = 0.1
STD_OF = {"gemma2": {"embed_tokens": 0.05},
          "dafotar": {"embed": 0.05, ".hc": 0.8, ".temp": 0.5, "canon": 0.3, "norm": 0.5, ".b": 0.02}}


# ------------------------------------------------------------------ the cases
def _step(model, decoding=0, shortest=0, longest=0, prompts=0, prompt=0, portion=0, dtype="bfloat16"):
    """``decoding`` requests with ``shortest`` to ``longest`` tokens in the cache beside ``prompts``
    prompts of ``prompt`` tokens; ``portion``: tokens of a prompt in one step (0: all of them)."""
    return {"kind": "step", "model": model, "dtype": dtype, "decoding": decoding, "shortest": shortest, "longest": longest,
            "prompts": prompts, "prompt": prompt, "portion": portion}


def _generate(model, requests, shortest, longest, new, dtype="bfloat16"):
    return {"kind": "generate", "model": model, "dtype": dtype, "requests": requests, "shortest": shortest, "longest": longest,
            "new": new}


def listed():
    return [
        # one user of a small model at the beginning of an answer: launches and latency
        dict(_step("gemma2-w1024", decoding=1, shortest=100, longest=100), name="small_decode_1"),
        # the 32-bit path, as it is served where 16 bits are too few: a prompt beside three decoded tokens
        dict(_step("gemma2-w1024", decoding=3, shortest=50, longest=700, prompts=1, prompt=300, dtype="float32"),
             name="small_fp32_mixed"),
        # one user of the 2B model, deep in a conversation
        dict(_step("gemma2-2b", decoding=1, shortest=3840, longest=3840), name="2b_decode_1"),
        # the headline: eight requests at a context of about 4,096
        dict(_step("gemma2-2b", decoding=8, shortest=3840, longest=3840), name="2b_decode_8"),
        # a full server: 64 requests of uneven lengths
        dict(_step("gemma2-2b", decoding=64, shortest=200, longest=3840), name="2b_decode_64"),
        # a short question, its first token awaited
        dict(_step("gemma2-2b", prompts=1, prompt=37), name="2b_prompt_37"),
        # a document in one step
        dict(_step("gemma2-2b", prompts=1, prompt=2048), name="2b_prompt_2048"),
        # a serving step: a prompt's portion beside 23 decoded tokens
        dict(_step("gemma2-2b", decoding=23, shortest=130, longest=2000, prompts=1, prompt=512), name="2b_mixed_512_23"),
        # a long prompt in the engine's default portions, each behind the ones before it
        dict(_step("gemma2-9b", prompts=1, prompt=3001, portion=512), name="9b_portions_3001"),
        # the largest weights
        dict(_step("gemma2-27b", decoding=8, shortest=100, longest=1000), name="27b_decode_8"),
        # an architecture with recurrent layers, residual streams and convolutions
        dict(_step("dafotar-w2048", decoding=8, shortest=100, longest=1500, prompts=1, prompt=700), name="dafotar_mixed_700_8"),
        # a batch of questions through the engine: scheduling, portions, decoding, picking
        dict(_generate("gemma2-2b", 24, 32, 700, 40), name="2b_generate_24"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["decode", "decode", "prompt", "prompt", "portions", "mixed", "mixed", "generate", "fp32"])
    model = rng.choice(["gemma2-w1024", "gemma2-w2048", "gemma2-2b", "gemma2-2b", "dafotar-w1024", "dafotar-w2048"])
    if what == "decode":
        if rng.random() < 0.15:
            model = "gemma2-9b"
        n, hi = _log(rng, 1, 64), _log(rng, 64, 3840)
        return _step(model, decoding=n, shortest=rng.randint(max(1, hi // 16), hi) if n > 1 else hi, longest=hi)
    if what == "prompt":
        n = rng.choice([1, 1, 1, 2, 3, 5])
        return _step(model, prompts=n, prompt=_log(rng, 7, 4000 // n))
    if what == "portions":
        return _step(model, prompts=1, prompt=_log(rng, 600, 4000), portion=rng.choice([128, 256, 512, 512, 1000]))
    if what == "mixed":
        n, hi = _log(rng, 1, 48), _log(rng, 64, 2500)
        return _step(model, decoding=n, shortest=rng.randint(max(1, hi // 16), hi) if n > 1 else hi, longest=hi,
                     prompts=rng.choice([1, 1, 2]), prompt=_log(rng, 16, 700))
    if what == "generate":
        return _generate(rng.choice(["gemma2-w1024", "gemma2-w2048", "gemma2-2b"]), _log(rng, 1, 24), _log(rng, 8, 60),
                         _log(rng, 61, 700), rng.randint(4, 40))
    hi = _log(rng, 16, 700)
    n = rng.randint(0, 4)
    return _step(rng.choice(["gemma2-w1024", "dafotar-w1024"]), decoding=n, shortest=max(1, hi // 3) if n else 0,
                 longest=hi if n else 0, prompts=1, prompt=_log(rng, 5, 300), dtype="float32")


def _spread(n, lo, hi):
    """n lengths from lo to hi, evenly, the longest first."""
    return [hi - (hi - lo) * i // max(n - 1, 1) for i in range(n)]


def _contexts(case):
    return _spread(case["decoding"], case["shortest"], case["longest"])


# ------------------------------------------------------------------ states
_kept = {}       # the model of the newest state


def _std_of(case):
    return STD_OF[case["model"].split("-")[0]]


def _model(case):
    key = (case["model"], case["dtype"])
    if key not in _kept:
        _kept.clear()
        gc.collect()
        _kept[key] = random_model(MODELS[case["model"]], case["dtype"], seed=WEIGHT_SEED, std=0.02, gain_std=GAIN_STD,
                                  std_of=_std_of(case))
    return _kept[key]


def _vocab(case):
    cfg = MODELS[case["model"]]
    return cfg.get("vocab_size") or cfg["vocab"]


def _tokens(case, seed):
    """The tokens of a state's requests: per decoding request those in the cache and the next
    NEW_TOKENS, and the prompts."""
    rng = np.random.default_rng([seed, zlib.crc32(case["model"].encode())])
    draw_ids = lambda n: rng.integers(0, _vocab(case), n).tolist()
    if case["kind"] == "generate":
        return [], [draw_ids(n) for n in _spread(case["requests"], case["shortest"], case["longest"])]
    return ([draw_ids(n + NEW_TOKENS) for n in _contexts(case)], [draw_ids(case["prompt"]) for _ in range(case["prompts"])])


class _DeviceArray:
    """float32 rows in device memory, for torch to look at; ``keep`` lives as long as they do."""

    def __init__(self, t, keep):
        self.keep = keep
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": "<f4", "data": (t.ptr, False), "version": 3, "strides": None}


class _Steps:
    """A runner with its live requests."""

    def __init__(self, case, seed):
        self.model = _model(case)
        self.running, self.prompts = _tokens(case, seed)
        self.contexts = _contexts(case)
        self.portion = case["portion"] or max(case["prompt"], 1)
        longest = max([n + NEW_TOKENS for n in self.contexts] + [case["prompt"]])
        pages = sum(-(-n // PAGE) + 1 for n in [c + NEW_TOKENS for c in self.contexts] + [case["prompt"]] * case["prompts"])
        self.runner = StepRunner(self.model, Runtime.get(), case["dtype"], page_size=PAGE, num_pages=pages,
                                 max_seqs=case["decoding"] + case["prompts"], max_batch_tokens=STEP_TOKENS,
                                 max_model_len=min(LONGEST, -(-longest // 1024) * 1024))
        self.at = [0] * len(self.contexts)
        self.fill(range(len(self.contexts)))

    def fill(self, which):
        """Takes the prompts of the decoding requests ``which`` into the cache, STEP_TOKENS a step."""
        entries, room = [], STEP_TOKENS
        for i in which:
            self.at[i] = self.contexts[i]
            left = self.running[i][:self.contexts[i]]
            while left:
                if room == 0 or (entries and entries[-1].req == i):
                    self.runner.step(entries, download=False)
                    entries, room = [], STEP_TOKENS
                entries.append(StepEntry(i, left[:room], []))
                left, room = left[room:], room - len(left[:room])
        if entries:
            self.runner.step(entries, download=False)

    def run(self):
        ended = [i for i, at in enumerate(self.at) if at == len(self.running[i])]
        if ended:
            for i in ended:
                self.runner.finish(i)
            self.fill(ended)
        length = len(self.prompts[0]) if self.prompts else 1
        for begin in range(0, length, self.portion):
            entries = []
            for i, at in enumerate(self.at):
                entries.append(StepEntry(i, self.running[i][at:at + 1], [0]))
                self.at[i] = at + 1
            for j, tokens in enumerate(self.prompts):
                part = tokens[begin:begin + self.portion]
                entries.append(StepEntry(("prompt", j), part, [len(part) - 1] if begin + len(part) == length else []))
            logits = self.runner.step(entries, download=False)
        for j in range(len(self.prompts)):
            self.runner.finish(("prompt", j))
        return torch.as_tensor(_DeviceArray(logits, self), device="cuda")

    def __del__(self):
        if hasattr(self, "runner"):
            self.runner.close()


class _Generation:
    """An engine and a list of prompts."""

    def __init__(self, case, seed):
        self.prompts = _tokens(case, seed)[1]
        self.params = SamplingParams(max_tokens=case["new"], temperature=0.0)
        pages = sum(-(-(len(p) + case["new"]) // PAGE) + 1 for p in self.prompts)
        self.engine = Engine(_model(case), dtype=case["dtype"], block_size=PAGE, num_blocks=pages, max_batch_seqs=len(self.prompts),
                             max_seq_len=-(-(case["longest"] + case["new"]) // 1024) * 1024)

    def run(self):
        return [np.array(ids, np.int64) for ids in self.engine.generate(self.prompts, self.params)]

    def __del__(self):
        if hasattr(self, "engine"):
            self.engine.close()


def prepare(case, seed):
    return _Generation(case, seed) if case["kind"] == "generate" else _Steps(case, seed)


def run(state):
    return state.run()


# ------------------------------------------------------------------ what a pass cannot do without
def _reqs(case):
    """Checkpoint name (without a leading ``model.``) -> what the model asks for."""
    arch = resolve_architecture(MODELS[case["model"]])
    reqs = Model(arch.plan(arch.config_from_dict(MODELS[case["model"]]))).tensor_reqs()
    return {r.name[len("model."):] if r.name.startswith("model.") else r.name: r for r in reqs}


def _layers(case):
    """Per layer: (kind, heads, key/value heads, key size, value size, window, keeps keys of its own)."""
    cfg = MODELS[case["model"]]
    if "layers" not in cfg:
        n, g, d = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
        return [("attention", n, g, d, d, cfg["sliding_window"] if l % 2 == 0 else None, True) for l in range(cfg["num_hidden_layers"])]
    out = []
    for layer in cfg["layers"]:
        m = layer["mixer"]
        out.append((layer["type"], m["heads"], m.get("kv_heads", m["heads"]), m["dim"], m["vdim"], (m.get("mask") or {}).get("size"),
                    m.get("kv_from") is None))
    return out


def _seen(start, n, window):
    """Keys that the n tokens behind ``start`` cached ones look at, all together."""
    return sum(min(p + 1, window or p + 1) for p in range(start, start + n))


def work(case):
    item = 4 if case["dtype"] == "float32" else 2
    reqs = _reqs(case)
    embed = next(k for k in reqs if "embed" in k)
    size = {k: math.prod(r.shape) for k, r in reqs.items()}
    weights = sum(n * (item if len(reqs[k].shape) == 2 else 4) for k, n in size.items())
    matrices = sum(n for k, n in size.items() if len(reqs[k].shape) == 2 and k != embed)
    vocab, width = reqs[embed].shape
    # every step reads the weights once; (tokens before, tokens) of each request in it, and its logits' rows
    if case["kind"] == "generate":
        lengths = _spread(case["requests"], case["shortest"], case["longest"])
        first = -(-sum(lengths) // STEP_TOKENS)
        steps = [([(0, n) for n in lengths], len(lengths))] + [([(n + i, 1) for n in lengths], len(lengths))
                                                               for i in range(case["new"] - 1)]
        reads = first + case["new"] - 1
    else:
        length, steps = max(case["prompt"], 1), []
        portion = case["portion"] or length
        for begin in range(0, length, portion):
            part = min(portion, length - begin)
            ended = begin + part == length
            steps.append(([(n, 1) for n in _contexts(case)] + [(begin, part)] * case["prompts"],
                          case["decoding"] + (case["prompts"] if ended else 0)))
        reads = len(steps)
    nbytes, flops = float(weights) * reads, 0.0
    for requests, rows in steps:
        tokens = sum(n for _, n in requests)
        flops += 2.0 * matrices * tokens + 2.0 * rows * vocab * width
        nbytes += tokens * width * item + (rows * vocab * 4 if case["kind"] == "step" else 0)
        for kind, heads, kv_heads, d, e, window, own in _layers(case):
            if kind == "attention":
                kv = kv_heads * (d + e) * item
                for start, n in requests:
                    flops += 2.0 * heads * (d + e) * _seen(start, n, window)
                    nbytes += kv * min(start, (window or start + n) - 1) + (kv * n if own else 0)
            else:
                flops += 6.0 * heads * d * e * tokens
                nbytes += 2.0 * 4 * heads * (d * e + d + 1) * len(requests)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "generate":
        return {"rel": 0.0, "differ": 0.005}
    # against 64 bits: 1.8e-6 to 6.4e-6 in 32 bits; 5e-3 to 1e-2 in bfloat16, more where there are more layers
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 2.5e-2, "max": 0.2}


# ------------------------------------------------------------------ the same in 64 bits
def _normal(shape, seed, name, std):
    """The random weights' values: a counter hash and Box-Muller in single 32-bit operations, which
    give the same bits everywhere."""
    s64 = lambda v: (v & (2 ** 64 - 1)) - (2 ** 64 if v & 2 ** 63 else 0)
    shr = lambda z, n: (z >> n) & ((1 << (64 - n)) - 1)

    def mix(z):
        z = z + s64(0x9E3779B97F4A7C15)
        z = (z ^ shr(z, 30)) * s64(0xBF58476D1CE4E5B9)
        z = (z ^ shr(z, 27)) * s64(0x94D049BB133111EB)
        return z ^ shr(z, 31)

    def horner(x, coefficients):
        p = torch.full_like(x, coefficients[0])
        for c in coefficients[1:]:
            p = p * x + c
        return p

    n = math.prod(shape)
    out = torch.empty(2 * ((n + 1) // 2), dtype=torch.float32, device="cuda")
    base = mix(torch.tensor([s64(seed ^ (zlib.crc32(name.encode()) * 0xD1342543DE82EF95))], device="cuda"))
    for at in range(0, len(out) // 2, 1 << 24):
        end = min(at + (1 << 24), len(out) // 2)
        r = mix(base + torch.arange(at, end, device="cuda"))
        k, j = shr(r, 40) + 1, shr(r, 8) & 0xFFFFFF
        m, e = torch.frexp(k.to(torch.float64))
        m, e = (m * 2).to(torch.float32), e - 1
        big = m > 1.41421354
        m, e = torch.where(big, m * 0.5, m), e + big
        s = (m - 1) / (m + 1)
        ln = (e - 24).to(torch.float32) * 0.693147182 + (2 * s) * horner(s * s, [0.111111112, 0.142857149, 0.2, 0.333333343, 1.0])
        rad = torch.sqrt(-2 * ln)
        q, t = shr(j, 22), j & 0x3FFFFF
        fold = t > 0x200000
        x = torch.where(fold, 0x400000 - t, t).to(torch.float32) * 3.74507039e-07
        x2 = x * x
        s0 = x + (x * x2) * horner(x2, [2.75573188e-06, -1.98412701e-04, 8.33333377e-03, -1.66666672e-01])
        c0 = 1 + x2 * horner(x2, [-2.75573188e-07, 2.48015876e-05, -1.38888892e-03, 4.16666679e-02, -0.5])
        s1, c1 = torch.where(fold, c0, s0), torch.where(fold, s0, c0)
        sn = torch.where(q == 0, s1, torch.where(q == 1, c1, torch.where(q == 2, -s1, -c1)))
        cs = torch.where(q == 0, c1, torch.where(q == 1, -s1, torch.where(q == 2, -c1, s1)))
        out[2 * at:2 * end:2] = (rad * cs) * std
        out[2 * at + 1:2 * end:2] = (rad * sn) * std
    return out[:n].reshape(shape)


def _weights(case):
    """name -> the weight in 64 bits, drawn when it is asked for."""
    reqs = _reqs(case)

    def weight(name):
        r = reqs[name]
        std = r.init_std if r.init_std is not None else GAIN_STD if r.role == "gain" else 0.02
        for part, value in _std_of(case).items():
            if part in r.name:
                std = value
        w = _normal(r.shape, WEIGHT_SEED, name, std)
        return (w.to(torch.bfloat16) if case["dtype"] == "bfloat16" else w).to(torch.float64)
    return weight


def _rotate(x, base, dims, sign=1.0):
    """Pairs (m, m + dims / 2) of the first ``dims`` channels turned by position * base^(-2 m / dims).  x: [T, heads, size]."""
    half = dims // 2
    freq = base ** (-torch.arange(half, dtype=torch.float64, device=x.device) * 2 / dims)
    ang = (sign * torch.arange(x.shape[0], dtype=torch.float64, device=x.device)[:, None] * freq)[:, None]
    a, b = x[..., :half], x[..., half:dims]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin(), x[..., dims:]], -1)


def _attention(q, k, v, scale, window, cap=None):
    """q: [T, heads, d], k: [T, groups, d], v: [T, groups, e]; ``scale``: a number, or one for each head."""
    T, heads = q.shape[:2]
    at = torch.arange(T, device=q.device)
    out = torch.empty(T, heads, v.shape[2], dtype=q.dtype, device=q.device)
    for h in range(heads):
        g = h // (heads // k.shape[1])
        for lo in range(0, T, 1024):
            rows = slice(lo, lo + 1024)
            s = q[rows, h] @ k[:lo + 1024, g].T * (scale[h] if torch.is_tensor(scale) else scale)
            if cap:
                s = cap * torch.tanh(s / cap)
            away = at[rows, None] - at[None, :lo + 1024]
            s = s.masked_fill((away < 0) | (away >= (window or T)), -math.inf)
            out[rows, h] = torch.softmax(s, -1) @ v[:lo + 1024, g]
    return out


def _unit(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _gemma2(cfg, w, sequences):
    """The last row of logits of each sequence."""
    eps, H = cfg["rms_norm_eps"], cfg["hidden_size"]
    heads, groups, d = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
    norm = lambda x, name: _unit(x, eps) * (1 + w(name))
    E = w("embed_tokens.weight")
    xs = [E[torch.tensor(s, device="cuda")] * math.sqrt(H) for s in sequences]
    ends = np.cumsum([0] + [len(s) for s in sequences])
    x = torch.cat(xs)
    del E, xs
    for l in range(cfg["num_hidden_layers"]):
        p = f"layers.{l}."
        h = norm(x, p + "input_layernorm.weight")
        q, k, v = ((h @ w(f"{p}self_attn.{n}_proj.weight").T).reshape(-1, c, d) for n, c in (("q", heads), ("k", groups), ("v", groups)))
        a = torch.cat([_attention(_rotate(q[b:e], cfg["rope_theta"], d), _rotate(k[b:e], cfg["rope_theta"], d), v[b:e],
                                  cfg["query_pre_attn_scalar"] ** -0.5, cfg["sliding_window"] if l % 2 == 0 else None,
                                  cfg["attn_logit_softcapping"]) for b, e in zip(ends[:-1], ends[1:])])
        x = x + norm(a.reshape(len(x), -1) @ w(p + "self_attn.o_proj.weight").T, p + "post_attention_layernorm.weight")
        h = norm(x, p + "pre_feedforward_layernorm.weight")
        gate, up, down = (w(f"{p}mlp.{n}_proj.weight").T for n in ("gate", "up", "down"))
        y = torch.cat([(torch.nn.functional.gelu(r @ gate, approximate="tanh") * (r @ up)) @ down for r in h.split(8192)])
        x = x + norm(y, p + "post_feedforward_layernorm.weight")
    x = norm(x[torch.tensor(ends[1:] - 1, device="cuda")], "norm.weight")
    cap = cfg["final_logit_softcapping"]
    return cap * torch.tanh(x @ w("embed_tokens.weight").T / cap)


def _mlstm(h, w, pre, m, eps):
    """The recurrence written out: token t reads every token s before it with weight exp(F_t - F_s + i_s - m_t)."""
    T, heads, d, e, cap = len(h), m["heads"], m["dim"], m["vdim"], m["gate_cap"]
    q, k, v = ((h @ w(pre + n).T).reshape(T, heads, c).transpose(0, 1) for n, c in (("q", d), ("k", d), ("v", e)))
    gi = (cap * torch.tanh((h @ w(pre + "i").T + w(pre + "i.b")) / cap)).T
    F = torch.nn.functional.logsigmoid(cap * torch.tanh((h @ w(pre + "f").T + w(pre + "f.b")) / cap)).T.cumsum(1)
    out = torch.empty(T, heads, e, dtype=h.dtype, device=h.device)
    later = torch.ones(T, T, dtype=torch.bool, device=h.device).triu(1)
    for n in range(heads):
        D = (F[n][:, None] - F[n][None] + gi[n][None]).masked_fill(later, -math.inf)
        top = torch.maximum(F[n], D.amax(1))            # the running maximum starts at 0
        a = torch.exp(D - top[:, None]) * (q[n] @ k[n].T) * d ** -0.5
        out[:, n] = a @ v[n] / (torch.maximum(a.sum(1).abs(), torch.exp(-top)) + 1e-6)[:, None]
    o = _unit(out, eps).reshape(T, -1) * w(pre + "norm")
    return (o * torch.sigmoid(h @ w(pre + "g").T)) @ w(pre + "o").T


def _dafotar_layers(cfg, w, sequences):
    eps, out = cfg["norm"]["eps"], []

    def norm(x, name):
        x = x - x.mean(-1, keepdim=True)
        return _unit(x, eps) * w(name) + w(name + ".b")

    def conv(h, name):
        taps = w(name)
        y = h.clone()
        for j in range(taps.shape[1]):
            back = taps.shape[1] - 1 - j
            y[back:] += taps[:, j] * h[:len(h) - back]
        return y

    E = w("embed")
    for seq in sequences:
        xs = E[torch.tensor(seq, device="cuda")][:, None].repeat(1, cfg["streams"], 1)
        kept = {}
        for l, layer in enumerate(cfg["layers"]):
            pre, m = f"l{l}.mix.", layer["mixer"]
            for part in (1, 2) if layer["mlp"] else (1,):
                h = norm(torch.einsum("s,tsw->tw", w(f"l{l}.hc{part}.in"), xs), f"l{l}.norm{part}")
                if part == 2:
                    y = (torch.relu(h @ w(f"l{l}.mlp.gate").T) * (h @ w(f"l{l}.mlp.up").T)) @ w(f"l{l}.mlp.down").T
                elif layer["type"] == "mlstm":
                    y = _mlstm(conv(h, f"l{l}.canon1"), w, pre, m, eps)
                else:
                    h = conv(h, f"l{l}.canon1")
                    T, base, dims = len(h), m["rot"]["base"], m["rot"]["dims"]
                    q = _rotate(_unit((h @ w(pre + "q").T).reshape(T, m["heads"], -1), eps) * w(pre + "q.norm"), base, dims)
                    if m.get("kv_from") is None:
                        k = _unit((h @ w(pre + "k").T).reshape(T, m["kv_heads"], -1), eps) * w(pre + "k.norm")
                        kept[l] = (_rotate(k, base, dims), _rotate((h @ w(pre + "v").T).reshape(T, m["kv_heads"], -1), base, m["vdim"]))
                    k, v = kept[l if m.get("kv_from") is None else m["kv_from"]]
                    y = _attention(q, k, v, w(pre + "temp") * m["scale"], m["mask"]["size"])
                    y = _rotate(y, base, m["vdim"], -1.0).reshape(T, -1) @ w(pre + "o").T
                xs = torch.einsum("sr,tsw->trw", w(f"l{l}.hc{part}.mix"), xs) + w(f"l{l}.hc{part}.out")[:, None] * y[:, None]
        out.append(norm(xs.sum(1)[-1], "final.norm"))
    return torch.stack(out) @ E.T


def exact(case, seed):
    """The logits of a first pass."""
    if case["kind"] == "generate":
        return None
    running, prompts = _tokens(case, seed)
    sequences = [t[:n + 1] for t, n in zip(running, _contexts(case))] + prompts
    if case["portion"] and case["decoding"]:
        return None
    tokens = sum(len(s) for s in sequences)
    if 2.0 * tokens * sum(math.prod(r.shape) for r in _reqs(case).values()) > 4e14:
        return None
    cfg, w = MODELS[case["model"]], _weights(case)
    if "layers" not in cfg:
        return _gemma2(cfg, w, sequences)
    keep = {}                     # a small model's weights, drawn once for all sequences
    return _dafotar_layers(cfg, lambda name: keep[name] if name in keep else keep.setdefault(name, w(name)), sequences)
