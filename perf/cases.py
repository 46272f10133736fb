"""The work that is timed: what a program that uses this library has it do, through puppygrad_amd.

Weights are seeded and random, one model per configuration, kept while the process lives as a
program keeps its model; the prompts come from a case's seed.  Five kinds of case:

    token      one more token of a cache that holds a prompt: an interactive program's inner step
    prompt     the logits behind a prompt, or behind a batch of prompts of one length
    continue   greedy tokens for sequences whose prompts the cache holds already
    generate   a whole greedy request: prompt, new tokens, the logits behind the last one
    sample     a whole streamed request with sampled selection (its entry point hands out ids only)

GPT-2 in its four sizes with weights stored as f32, bf16 or int8; the two stack architectures
in the three widths that the benchmark has, with bf16 weights (a stack cache cannot go back to an
earlier position, so its requests are whole ones).
"""
import json
import math
import os
import tempfile
from collections import OrderedDict

import numpy as np
import torch

from puppygrad_amd import Gpt2BlockWeights, Gpt2Config, Gpt2HipConfig, Gpt2Model, Gpt2Weights, TextGenerationConfig, _lib, load_model, synth

SIZES = {"small": synth.GPT2_SMALL, "medium": synth.GPT2_MEDIUM, "large": synth.GPT2_LARGE, "xl": synth.GPT2_XL}
STORAGE = {"f32": _lib.PG_STORE_F32, "bf16": _lib.PG_STORE_BF16, "int8": _lib.PG_STORE_INT8}
STACK = {"tarepel": synth.tarepel_config, "movudra": synth.movudra_config}
STACK_LAYERS, VOCAB, POSITIONS = 8, 50257, 1024
WEIGHT_SEED = 0x5EED


# ---- the cases ---------------------------------------------------------------------------------
def _gpt2(size, storage, **more):
    return dict(arch="gpt2", size=size, storage=storage, **more)


def _stack(arch, width, **more):
    return dict(arch=arch, size=width, storage="bf16", **more)


def listed():
    return [
        # the smallest call: a chat's next token from the smallest model, its logits looked at by the caller
        dict(_gpt2("small", "f32", kind="token", batch=1, prompt=97), name="small-token"),
        # a short question to a quantised model: the time until its first token
        dict(_gpt2("large", "int8", kind="prompt", batch=1, prompt=37), name="large-int8-prompt-37"),
        # a document that fills the context, to the smallest model
        dict(_gpt2("small", "f32", kind="prompt", batch=1, prompt=1024), name="small-prompt-1024"),
        # a streamed answer with the usual sampling settings
        dict(_gpt2("small", "f32", kind="sample", batch=1, prompt=32, new=64, temperature=0.8, top_k=40, top_p=0.0,
                   penalty=1.0), name="small-sample"),
        # a small server's step: sixteen sequences of a mid-sized model
        dict(_gpt2("medium", "f32", kind="continue", batch=16, prompt=225, new=16), name="medium-batch-16"),
        # one long conversation with the largest model
        dict(_gpt2("xl", "f32", kind="continue", batch=1, prompt=896, new=24), name="xl-decode-896"),
        # a long document to the largest model in the reference's own precision
        dict(_gpt2("xl", "f32", kind="prompt", batch=1, prompt=1000), name="xl-prompt-1000"),
        # a busy server's step: many long sequences of the largest model with halved weights
        dict(_gpt2("xl", "bf16", kind="continue", batch=32, prompt=760, new=12), name="xl-bf16-batch-32"),
        # the same server taking in a full batch of prompts: the largest call
        dict(_gpt2("xl", "bf16", kind="prompt", batch=32, prompt=512), name="xl-bf16-prompts-32x512"),
        # a summary: a long prompt, a short answer, from a model with recurrent and attention layers
        dict(_stack("tarepel", 1600, kind="generate", batch=1, prompt=1000, new=32), name="tarepel-1000-32"),
        # a chat: a short prompt and a longer answer, from a model with experts
        dict(_stack("movudra", 1600, kind="generate", batch=1, prompt=16, new=48), name="movudra-16-48"),
        # a batch of such requests stepping together
        dict(_stack("movudra", 1600, kind="generate", batch=32, prompt=100, new=12), name="movudra-batch-32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _params(size):
    m = SIZES[size]
    return 12 * m["n_layer"] * m["n_embd"] ** 2


def draw(rng):
    kind = rng.choice(["token", "prompt", "prompt", "continue", "continue", "generate", "generate", "sample"])
    if kind == "generate":
        arch, width = rng.choice(["tarepel", "movudra"]), rng.choice([768, 1280, 1600])
        batch = 1 if rng.random() < 0.5 else _log_int(rng, 2, 40)
        return _stack(arch, width, kind=kind, batch=batch, prompt=_log_int(rng, 3, 1500 if batch == 1 else 200),
                      new=_log_int(rng, 2, 48))
    size = rng.choice(list(SIZES))
    if kind == "token":
        return _gpt2(size, rng.choice(list(STORAGE)), kind=kind, batch=1, prompt=rng.randint(1, 1000))
    if kind == "sample":
        penalty = rng.choice([1.0, 1.0, 1.1, 1.3])
        top_k = rng.choice([0, rng.randint(10, 100)])
        return _gpt2(size, rng.choice(list(STORAGE)), kind=kind, batch=1, prompt=_log_int(rng, 4, 256),
                     new=_log_int(rng, 16, 96), temperature=round(rng.uniform(0.5, 1.2), 2), top_k=top_k,
                     top_p=0.0 if top_k else rng.choice([0.0, 0.9]), penalty=penalty)
    if kind == "continue":
        batch = 1 if rng.random() < 0.5 else _log_int(rng, 2, 48)
        return _gpt2(size, rng.choice(list(STORAGE)), kind=kind, batch=batch, prompt=_log_int(rng, 8, 960),
                     new=_log_int(rng, 3, 24 if batch <= 8 else 12))
    storage = rng.choice(list(STORAGE))
    batch = 1 if rng.random() < 0.6 else _log_int(rng, 2, 32)
    # (a pass over f32 weights takes about twice the time of one over bf16 weights)
    room = 16384 * _params("xl") / _params(size) * (0.4 if storage == "f32" else 0.9)
    return _gpt2(size, storage, kind=kind, batch=batch,
                 prompt=_log_int(rng, 4, max(4, min(POSITIONS, int(room / batch), 32768 // batch))))


# ---- weights -----------------------------------------------------------------------------------
_models = OrderedDict()  # configuration -> the model, the latest used last
MOST_MODELS = 8


def _stream():
    g = torch.Generator(device="cuda")
    g.manual_seed(WEIGHT_SEED)
    return lambda shape, std, mean=0.0: torch.empty(shape, device="cuda").normal_(mean, std, generator=g)


def _gpt2_tensors(size):
    """(layer or None, name, tensor) in the checkpoint's layout, one at a time."""
    m, normal = SIZES[size], _stream()
    C, L = m["n_embd"], m["n_layer"]
    for i in range(L):
        for name, shape, mean, std in (
                ("ln_1_g", (C,), 1.0, 0.1), ("ln_1_b", (C,), 0.0, 0.02), ("c_attn_w", (C, 3 * C), 0.0, 0.02),
                ("c_attn_b", (3 * C,), 0.0, 0.02), ("c_proj_w", (C, C), 0.0, 0.02), ("c_proj_b", (C,), 0.0, 0.02),
                ("ln_2_g", (C,), 1.0, 0.1), ("ln_2_b", (C,), 0.0, 0.02), ("c_fc_w", (C, 4 * C), 0.0, 0.02),
                ("c_fc_b", (4 * C,), 0.0, 0.02), ("c_proj_mlp_w", (4 * C, C), 0.0, 0.02), ("c_proj_mlp_b", (C,), 0.0, 0.02)):
            yield i, name, normal(shape, std, mean)
    yield None, "ln_f_g", normal((C,), 0.1, 1.0)
    yield None, "ln_f_b", normal((C,), 0.02)
    yield None, "wte", normal((VOCAB, C), 0.02)
    yield None, "wpe", normal((POSITIONS, C), 0.02)


def _stack_config(case):
    return STACK[case["arch"]](case["size"], STACK_LAYERS, VOCAB)


def _stack_tensors(cfg):
    """(name, bf16 tensor): gains around 1, layer scales around 0.3, taps around a mean filter, decays
    between a few and a few hundred tokens, all else N(0, 0.02)."""
    normal = _stream()
    for name, shape in synth.stack_tensor_shapes(cfg).items():
        last = name.split(".")[-1]
        if last.startswith("norm"):
            mean, std = 1.0, 0.02
        elif last in ("ls1", "ls2"):
            mean, std = 0.3, 0.02
        elif last == "conv":
            mean, std = 1.0 / shape[1], 0.2
        elif last == "A_log":
            mean, std = 0.0, 0.4
        elif last == "dt_bias":
            mean, std = -3.0, 0.8
        elif name.endswith("a2.b"):
            mean, std = 2.0, 0.8
        elif last == "D":
            mean, std = 1.0, 0.02
        else:
            mean, std = 0.0, 0.02
        yield name, normal(shape or (1,), std, mean).reshape(shape).bfloat16()


def _write_stack_dir(path, cfg):
    header, parts, at = {}, [], 0
    for name, t in _stack_tensors(cfg):
        part = t.view(torch.int16).cpu().numpy()
        header[name] = {"dtype": "BF16", "shape": list(t.shape), "data_offsets": [at, at + part.nbytes]}
        at += part.nbytes
        parts.append(part)
    text = json.dumps(header).encode()
    text += b" " * (-len(text) % 8)
    with open(os.path.join(path, "config.json"), "w", encoding="utf-8") as f:
        json.dump(cfg, f)
    with open(os.path.join(path, "model.safetensors"), "wb") as f:
        f.write(len(text).to_bytes(8, "little") + text)
        for part in parts:
            part.tofile(f)


def _build_model(case):
    hip = Gpt2HipConfig(weight_storage=STORAGE[case["storage"]])
    if case["arch"] != "gpt2":
        with tempfile.TemporaryDirectory() as tmp:
            _write_stack_dir(tmp, _stack_config(case))
            return load_model(tmp, hip)
    m = SIZES[case["size"]]
    blocks, rest = [{} for _ in range(m["n_layer"])], {}
    for layer, name, t in _gpt2_tensors(case["size"]):
        (rest if layer is None else blocks[layer])[name] = t.cpu().numpy()
    return Gpt2Model.new(Gpt2Config(**m), Gpt2Weights(blocks=[Gpt2BlockWeights(**b) for b in blocks], **rest), hip)


def _model(case):
    key = (case["arch"], case["size"], case["storage"])
    if key not in _models:
        while len(_models) >= MOST_MODELS:
            _models.popitem(last=False)
        _models[key] = _build_model(case)
    _models.move_to_end(key)
    return _models[key]


# ---- a pass ------------------------------------------------------------------------------------
def _ids(case, seed):
    """Prompts [batch][prompt] and one more id: words come with very unequal frequencies."""
    r = np.random.default_rng([seed, 77])
    u = r.random((case["batch"], case["prompt"] + 1))
    return np.minimum(np.floor(np.exp(u * math.log(VOCAB)) - 1.0), VOCAB - 1).astype(np.uint32)


def prepare(case, seed):
    model, ids = _model(case), _ids(case, seed)
    s = {"case": case, "model": model, "ids": np.ascontiguousarray(ids[:, :-1]), "next": int(ids[0, -1])}
    if case["kind"] == "sample":
        s["config"] = TextGenerationConfig(
            case["new"], temperature=case["temperature"], top_k=case["top_k"] or None, top_p=case["top_p"] or None,
            seed=seed, repeat_penalty=case["penalty"])
        return s
    s["cache"] = model.new_kv_cache(case["batch"])
    if case["kind"] in ("token", "continue"):
        _prompt(s).argmax()
    return s


def _prompt(s):
    if s["case"]["batch"] == 1:
        return s["model"].prefill(s["ids"][0], s["cache"])
    return s["model"].prefill_batch(s["ids"], s["cache"])


def _forward(s, ids):
    if s["case"]["batch"] == 1:
        return s["model"].forward_one(int(ids[0]), s["cache"])
    return s["model"].forward_one_batch(ids, s["cache"])


def _greedy(s, new):
    if s["case"]["batch"] == 1:
        return np.asarray(s["model"].decode_greedy(s["cache"], new)[0], np.int64)[:, None]
    return s["model"].decode_greedy_batch(s["cache"], new)[0].astype(np.int64)


def run(s):
    case, model = s["case"], s["model"]
    kind = case["kind"]
    if kind == "sample":
        tokens, _ = model.stream_token_ids_with_stats(s["ids"][0], s["config"])
        return {"tokens": np.asarray(tokens, np.int64)}
    cache = s["cache"]
    if kind == "prompt":
        return {"logits": _prompt(s).to_host()}
    if kind == "token":
        cache.seq_len = case["prompt"]
        logits = model.forward_one(s["next"], cache)
        return {"token": model.select_next_token(logits), "logits": logits.to_host()}
    if kind == "continue":  # back to the prompt's last id: its forward makes the logits the first choice needs
        cache.seq_len = case["prompt"] - 1
        _forward(s, s["ids"][:, -1])
    else:
        _prompt(s)
    tokens = _greedy(s, case["new"])
    return {"tokens": tokens, "logits": _forward(s, tokens[-1]).to_host()}


# ---- what a pass cannot do without -------------------------------------------------------------
def _passes(case):
    """(rows of the call, position of its first row) of every forward of a pass."""
    n, kind = case["prompt"], case["kind"]
    if kind == "prompt":
        return [(n, 0)]
    if kind == "token":
        return [(1, n)]
    if kind == "continue":
        return [(1, n - 1 + i) for i in range(case["new"] + 1)]
    return [(n, 0)] + [(1, n + i) for i in range(case["new"] - (kind == "sample"))]


def _stack_counts(cfg, rows):
    """Values of the matrices that `rows` tokens read, the multiplications of one token, and the
    values of state per sequence."""
    read = mult = 0.0
    for name, shape in synth.stack_tensor_shapes(cfg).items():
        if len(shape) < 2 or name in ("embed", "head") or name.endswith("conv"):
            continue
        n, met, used = math.prod(shape), 1.0, 1.0
        if ".mlp.e" in name:
            r = cfg["layers"][int(name[1:name.index(".")])]["mlp"]["router"]
            used = r["top"] / r["experts"]
            met = 1.0 - (1.0 - used) ** rows
        read, mult = read + met * n, mult + used * n
    state = 0
    for layer in cfg["layers"]:
        m = layer["mixer"]
        m = m.get("right", m)
        if "state" in m:
            state += m["heads"] * m["state"] * m["vdim"]
        elif "kv_rank" not in m:
            state += m["heads"] * m["dim"] * m["vdim"]
    return read, mult, state


def work(case):
    B, eb = case["batch"], {"f32": 4, "bf16": 2, "int8": 1}[case["storage"]]
    nbytes = flops = 0.0
    for rows, first in _passes(case):
        keys = sum(range(first + 1, first + rows + 1))
        if case["arch"] == "gpt2":
            m = SIZES[case["size"]]
            C, L = m["n_embd"], m["n_layer"]
            mats = 12 * L * C * C
            nbytes += eb * (mats + VOCAB * C) + B * 8 * L * C * (first + rows)
            flops += 2.0 * B * rows * mats + 4.0 * B * C * L * keys
        else:
            cfg = _stack_config(case)
            C = cfg["width"]
            read, mult, state = _stack_counts(cfg, B * rows)
            nbytes += eb * (read + VOCAB * C) + B * 8 * state
            flops += 2.0 * B * rows * (mult + 2 * state)
        nbytes += 4 * B * (VOCAB + rows * C)
        flops += 2.0 * B * VOCAB * C
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "sample":  # a draw beside the boundary of two ids may fall to either
        return {"rel": 0.0, "differ": 0.01}
    # sums in 32 bits over up to 6400 terms, in up to 48 layers; ids may differ where two logits tie
    return {"rel": 1e-5 if case["arch"] == "gpt2" else 5e-5, "differ": 0.01}


# ---- the same in 64 bits -----------------------------------------------------------------------
def _round_bf16(t):
    return t.bfloat16().float()


def _quantised(t):
    """Rows of an [out, in] matrix as whole multiples of a scale per row, as int8 storage keeps them."""
    scale = (t.abs().amax(1).double() / 127.0).float()  # (rounded once, as a 32-bit quotient is)
    scale = torch.where(scale == 0, torch.ones_like(scale), scale)
    q = (t.double() / scale.double()[:, None]).float().double()
    return (torch.sign(q) * torch.floor(q.abs() + 0.5)).clamp(-127, 127) * scale.double()[:, None]


class _Gpt2Exact:
    def __init__(self, case):
        m = SIZES[case["size"]]
        self.H, self.storage = m["n_head"], case["storage"]
        self.layers, self.rest = [{} for _ in range(m["n_layer"])], {}
        for layer, name, t in _gpt2_tensors(case["size"]):
            (self.rest if layer is None else self.layers[layer])[name] = t
        self.past = [None] * m["n_layer"]
        self.pos = 0
        self.head = self.stored(self.rest["wte"])
        self.embed = _round_bf16(self.rest["wte"]) if self.storage == "bf16" else self.rest["wte"]

    def stored(self, t):
        """An [out, in] matrix as it is multiplied with."""
        if self.storage == "int8":
            return _quantised(t)
        return (_round_bf16(t) if self.storage == "bf16" else t).double()

    @staticmethod
    def norm(x, g, b):
        return torch.nn.functional.layer_norm(x, (x.shape[-1],), g.double(), b.double(), 1e-5)

    def forward(self, ids):
        """Logits behind the last of ids [batch][n], after what came before."""
        B, n = ids.shape
        x = self.embed[ids].double() + self.rest["wpe"][self.pos:self.pos + n].double()
        C = x.shape[-1]
        for i, w in enumerate(self.layers):
            def dense(y, name):
                return y @ self.stored(w[name + "_w"].t().contiguous()).t() + w[name + "_b"].double()

            qkv = dense(self.norm(x, w["ln_1_g"], w["ln_1_b"]), "c_attn").view(B, n, 3, self.H, C // self.H)
            q, k, v = (t.transpose(1, 2) for t in qkv.unbind(2))
            if self.past[i] is not None:
                k, v = torch.cat([self.past[i][0], k], 2), torch.cat([self.past[i][1], v], 2)
            self.past[i] = (k, v)
            mask = torch.arange(k.shape[2], device="cuda")[None] > torch.arange(self.pos, self.pos + n, device="cuda")[:, None]
            rows = []
            for b in range(B):
                s = (q[b] @ k[b].transpose(1, 2).contiguous()) * (C // self.H) ** -0.5
                rows.append(torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[b].contiguous())
            a = torch.stack(rows).transpose(1, 2).reshape(B, n, C)
            x = x + dense(a, "c_proj")
            h = dense(self.norm(x, w["ln_2_g"], w["ln_2_b"]), "c_fc")
            x = x + dense(torch.nn.functional.gelu(h, approximate="tanh"), "c_proj_mlp")
        self.pos += n
        return self.norm(x[:, -1], self.rest["ln_f_g"], self.rest["ln_f_b"]) @ self.head.t()


def _rms(x, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _unit(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)


class _StackExact:
    """One position of every sequence at a time, straight from the recurrences."""

    def __init__(self, case):
        self.cfg = _stack_config(case)
        self.w = {n: t.double() for n, t in _stack_tensors(self.cfg)}
        self.S = [{} for _ in self.cfg["layers"]]
        self.pos = 0

    def conv(self, st, key, x, taps, bias=None):
        """Short causal convolution over the last inputs, x [B][channels]."""
        old = st.get(key)
        if old is None:
            old = torch.zeros(taps.shape[1] - 1, *x.shape, dtype=x.dtype, device="cuda")
        window = torch.cat([old, x[None]])
        st[key] = window[1:]
        y = (window * taps.t()[:, None, :]).sum(0)
        return torch.nn.functional.silu(y if bias is None else y + bias)

    @staticmethod
    def spread(x, heads):
        """[B][groups][d] to one row per head."""
        return x.repeat_interleave(heads // x.shape[1], 1)

    def state(self, st, B, *shape):
        if "S" not in st:
            st["S"] = torch.zeros(B, *shape, dtype=torch.float64, device="cuda")
        return st["S"]

    def delta(self, st, B, q, k, v, decay, beta):
        S = self.state(st, B, q.shape[1], q.shape[2], v.shape[2]) * decay
        u = beta[..., None] * (v - (S * k[..., None]).sum(2))
        st["S"] = S + k[..., None] * u[:, :, None]
        return (st["S"] * q[..., None]).sum(2)

    def rotate_halves(self, x, base):
        half = x.shape[-1] // 2
        a = self.pos * base ** (-2.0 * torch.arange(half, dtype=torch.float64, device="cuda") / x.shape[-1])
        u, v = x[..., :half], x[..., half:]
        return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)

    # -- tarepel
    def chunk_attention(self, st, p, c, h):
        B, w = len(h), self.w
        H, G, d = c["heads"], c["kv_heads"], c["dim"]
        if self.pos % c["mask"]["size"] == 0:
            st["keys"], st["values"] = [], []
        k = (h @ w[p + "k"].t()).view(B, G, d)
        st["keys"].append(self.rotate_halves(k, c["rot"]["base"]))
        st["values"].append(k)
        q = self.rotate_halves((h @ w[p + "q"].t()).view(B, H, d), c["rot"]["base"]).view(B, G, H // G, d)
        keys, values = torch.stack(st["keys"], 2), torch.stack(st["values"], 2)
        z = q @ keys.transpose(2, 3).contiguous() * c["scale"] + w[p + "pb"].view(G, H // G, 1)
        return (torch.sigmoid(z) @ values).reshape(B, H * d) @ w[p + "o"].t()

    def gated_delta(self, st, p, c, h):
        B, w = len(h), self.w
        H, G, d, e = c["heads"], c["kv_heads"], c["dim"], c["vdim"]
        q, k, v = (self.conv(st, x, h @ w[p + x].t(), w[p + x + ".conv"]) for x in "qkv")
        decay = torch.exp(-torch.exp(w[p + "A_log"]) * torch.nn.functional.softplus(h @ w[p + "a"].t() + w[p + "dt_bias"], threshold=1e9))
        o = self.delta(st, B, self.spread(_unit(q.view(B, G, d)) * d ** -0.5, H), self.spread(_unit(k.view(B, G, d)), H),
                       v.view(B, H, e), decay[..., None, None], torch.sigmoid(h @ w[p + "b"].t()))
        y = _rms(o) * w[p + "norm"] * torch.nn.functional.silu(h @ w[p + "g"].t()).view(B, H, e)
        return y.reshape(B, H * e) @ w[p + "o"].t()

    def linear_attention(self, st, p, c, h):
        B, w = len(h), self.w
        H, d, e = c["heads"], c["dim"], c["vdim"]
        q, k, v = (h @ w[p + x].t() for x in "qkv")
        z = h @ w[p + "a1"].t() @ w[p + "a2"].t() + w[p + "a2.b"]
        alpha = (torch.sigmoid(z) ** (1.0 / c["tau"])).view(B, H, d)
        st["S"] = self.state(st, B, H, d, e) * alpha[..., None] + k.view(B, H, d, 1) * v.view(B, H, 1, e)
        o = (st["S"] * (q.view(B, H, d) * d ** -0.5)[..., None]).sum(2)
        y = (_rms(o) * w[p + "norm"]).reshape(B, H * e) * torch.nn.functional.silu(h @ w[p + "g"].t())
        return y @ w[p + "o"].t()

    def tarepel_layer(self, i, c, x):
        w, st, p, m = self.w, self.S[i], f"l{i}.mix.", c["mixer"]
        h = _rms(x) * w[f"l{i}.norm1"]
        if c["type"] == "parallel":
            mix = (m["left_scale"] * self.chunk_attention(st, p + "left.", m["left"], h)
                   + m["right_scale"] * self.gated_delta(st, p + "right.", m["right"], h))
        else:
            mix = self.linear_attention(st, p, m, h)
        q = f"l{i}.mlp."
        a = torch.nn.functional.gelu(h @ w[q + "gate"].t(), approximate="tanh") * (h @ w[q + "up"].t())
        return x + w[f"l{i}.ls1"] * mix + w[f"l{i}.ls2"] * (a @ w[q + "down"].t())

    # -- movudra
    def state_space(self, st, p, c, h):
        B, w = len(h), self.w
        H, e, N, G = c["heads"], c["vdim"], c["state"], c["groups"]
        inner = H * e
        z, xbc, dt = (h @ w[p + "in"].t()).split([inner, inner + 2 * G * N, H], 1)
        x, b, cc = self.conv(st, "x", xbc, w[p + "conv"], w[p + "conv.b"]).split([inner, G * N, G * N], 1)
        x, b, cc = x.view(B, H, e), self.spread(b.view(B, G, N), H), self.spread(cc.view(B, G, N), H)
        dt = torch.nn.functional.softplus(dt + w[p + "dt_bias"], threshold=1e9)
        decay = torch.exp(-torch.exp(w[p + "A_log"]) * dt)
        st["S"] = self.state(st, B, H, N, e) * decay[..., None, None] + (dt[..., None] * b)[..., None] * x[:, :, None]
        y = (st["S"] * cc[..., None]).sum(2) + w[p + "D"][:, None] * x
        y = y.reshape(B, inner) * torch.nn.functional.silu(z)
        y = _rms(y.view(B, c["norm_groups"], -1)).reshape(B, inner) * w[p + "norm"]
        return y @ w[p + "o"].t()

    def channel_delta(self, st, p, c, h):
        B, w = len(h), self.w
        H, G, d, e = c["heads"], c["kv_heads"], c["dim"], c["vdim"]
        q, k, v = (self.conv(st, x, h @ w[p + x].t(), w[p + x + ".conv"]) for x in "qkv")
        a = (h @ w[p + "a1"].t() @ w[p + "a2"].t() + w[p + "dt_bias"]).view(B, H, d)
        decay = torch.exp(-torch.exp(w[p + "A_log"])[:, None] * torch.nn.functional.softplus(a, threshold=1e9))
        o = self.delta(st, B, self.spread(_unit(q.view(B, G, d)) * d ** -0.5, H), self.spread(_unit(k.view(B, G, d)), H),
                       v.view(B, H, e), decay[..., None], torch.sigmoid(h @ w[p + "b"].t()))
        gate = torch.sigmoid(h @ w[p + "g1"].t() @ w[p + "g2"].t()).view(B, H, e)
        return (_rms(o) * w[p + "norm"] * gate).reshape(B, H * e) @ w[p + "o"].t()

    def frequencies(self, rot):
        """YaRN: pairs that turn often keep their angle per position, the slow ones' is divided."""
        dims, base, s = rot["dims"], rot["base"], rot["scaling"]

        def pair_of(turns):
            return dims * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))

        lo, hi = max(math.floor(pair_of(s["fast"])), 0), min(math.ceil(pair_of(s["slow"])), dims - 1)
        i = torch.arange(dims // 2, dtype=torch.float64, device="cuda")
        f, r = base ** (-2.0 * i / dims), ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        return f / s["factor"] * r + f * (1 - r), 0.1 * math.log(s["factor"]) + 1.0

    def rotate_pairs(self, x, rot):
        f, grow = self.frequencies(rot)
        a, x = self.pos * f, x.unflatten(-1, (-1, 2))
        u, v = x.unbind(-1)
        return grow * torch.stack([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1).flatten(-2)

    def latent_attention(self, st, p, c, h):
        B, w = len(h), self.w
        H, d, r, e, K = c["heads"], c["dim"], c["rot_dim"], c["vdim"], c["kv_rank"]
        q = (_rms(h @ w[p + "dq"].t()) * w[p + "dq.norm"] @ w[p + "uq"].t()).view(B, H, d + r)
        kv = h @ w[p + "dkv"].t()
        for name, t in (("c", _rms(kv[:, :K]) * w[p + "dkv.norm"]), ("r", self.rotate_pairs(kv[:, K:], c["rot"]))):
            st[name] = (st.get(name, []) + [t])[-c["mask"]["size"]:]
        lat, rot = torch.stack(st["c"], 1), torch.stack(st["r"], 1)
        inner = torch.einsum("bhd,hdk->bhk", q[..., :d], w[p + "uk"].view(H, d, K))
        z = inner @ lat.transpose(1, 2).contiguous() + self.rotate_pairs(q[..., d:], c["rot"]) @ rot.transpose(1, 2).contiguous()
        z = torch.cat([z * c["scale"], w[p + "sink"].view(1, H, 1).expand(B, H, 1)], -1)
        o = torch.einsum("bhk,hek->bhe", torch.softmax(z, -1)[..., :-1] @ lat, w[p + "uv"].view(H, e, K))
        return o.reshape(B, H * e) @ w[p + "o"].t()

    def feed_forward(self, p, f, x):
        w = self.w
        if f["kind"] == "dense":
            a = torch.relu(x @ w[p + "up"].t() + w[p + "up.b"]) ** 2
            return a @ w[p + "down"].t() + w[p + "down.b"]
        n, top = f["router"]["experts"], f["router"]["top"]
        if p not in w:  # all experts' rows in one, for one product
            w[p] = [torch.cat([w.pop(f"{p}e{i}.{x}") for i in range(n)]) for x in ("gate", "up")] + [
                torch.stack([w.pop(f"{p}e{i}.down").t().contiguous() for i in range(n)])]
        gate, up, down = w[p]
        s = torch.softmax(x @ w[p + "router"].t(), -1)
        best, which = s.topk(top, -1)
        share = torch.zeros_like(s).scatter(1, which, best)
        a = torch.nn.functional.silu(x @ gate.t()) * (x @ up.t())
        return (a.view(len(x), n, -1) * share[..., None]).flatten(1) @ down.flatten(0, 1)

    def movudra_layer(self, i, c, x):
        mix = {"mamba2": self.state_space, "channel_delta": self.channel_delta,
               "latent_attention": self.latent_attention}[c["type"]](self.S[i], f"l{i}.mix.", c["mixer"], x)
        x = x + _rms(mix) * self.w[f"l{i}.norm1"]
        return x + _rms(self.feed_forward(f"l{i}.mlp.", c["mlp"], x)) * self.w[f"l{i}.norm2"]

    def forward(self, ids):
        layer = self.tarepel_layer if self.cfg["architecture"] == "Tarepel" else self.movudra_layer
        for t in range(ids.shape[1]):
            x = self.w["embed"][ids[:, t]]
            for i, c in enumerate(self.cfg["layers"]):
                x = layer(i, c, x)
            self.pos += 1
        return _rms(x) * self.w["final.norm"] @ self.w["head"].t()


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":  # ids, no computed numbers
        return None
    ids = torch.from_numpy(_ids(case, seed).astype(np.int64)).cuda()
    with torch.no_grad():
        model = (_Gpt2Exact if case["arch"] == "gpt2" else _StackExact)(case)
        logits = model.forward(ids[:, :-1])
        if kind == "token":
            logits = model.forward(ids[:1, -1:])
            return {"token": int(logits[0].argmax()), "logits": logits[0]}
        tokens = []
        for _ in range(case.get("new", 0)):
            tokens.append(logits.argmax(1))
            logits = model.forward(tokens[-1][:, None])
    logits = logits[0] if case["batch"] == 1 else logits
    return {"logits": logits} if kind == "prompt" else {"tokens": torch.stack(tokens), "logits": logits}
