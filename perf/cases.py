"""Cases that stand for what this framework is used for: language models read prompts and write tokens on one GPU.

A case is a model and a pass over it, through `Generator` (one sequence) or `BatchGenerator` (several):

  prompt     a prompt is read from an empty cache and the logits of its last position are handed out: time to first token
  generate   a whole call: a prompt is read and `new` greedy tokens are written
  decode     `new` greedy tokens are written behind a prompt whose caches the program has kept (an answer tried again)

The models have the sizes that bench.py measures: GPT-2 small in f32, the 3B grouped-query decoder in bf16 with an f32 residual
stream (also with int8 and int4 weights), and four layers each of the hybrid state-space / latent-attention design and of the
chunked-attention design, bf16.  A model is loaded once per process, as a server holds it; a state's inputs are its prompts.

The weights are random, with the output matrix set to a shifted copy of the embedding table, so that a greedy step has a clear
winner, as a trained model's has: rounding does not decide which token comes next, and the logits stay comparable.
"""
import math
import zlib

import numpy as np
import torch

import __graft_entry__ as entry

entry.load_package()
from gptrs_amd import models  # noqa: E402
from gptrs_amd.backend import HipBackend  # noqa: E402
from gptrs_amd.ptir import TensorSpec  # noqa: E402

GPT2 = dict(vocab=50257, width=768, layers=12, heads=12, context=1024)
MINISTRAL = dict(vocab=131072, width=3072, layers=26, heads=32, kv=8, dim=128, ff=9216, theta=1e6, context=4096)
HYBRID = dict(vocab=32768, width=3072, ff=9216, limit=7.0, heads=96, vdim=64, state=128, groups=8, conv=4,
              att=dict(heads=32, dim=128, rot=64, vdim=128, q_rank=1536, kv_rank=512, base=1e4, yarn=(4.0, 4096.0, 32.0, 1.0)))
CHUNKED = dict(vocab=32768, width=3072, ff=9216, layers=4, heads=32, kv=8, dim=128, vdim=128, scale=0.1, base=5e5, chunk=1024,
               embedding_scale=1.5, residual_mult=0.25, softcap=20.0)
EPS = 1e-5
SHIFT = 1009   # the output matrix's column t + SHIFT is the embedding of t: greedy text counts up in steps of SHIFT


# ------------------------------------------------------------------------------------------ cases
def listed():
    def case(name, model, do, batch, prompt, new, ragged=False):
        return dict(name=name, model=model, do=do, batch=batch, prompt=prompt, new=new, ragged=ragged)

    return [
        # the smallest call: a few words in, the next one out; launches and host work are all there is to it
        case("gpt2_short_prompt", "gpt2", "prompt", 1, 7, 0),
        # the reference's published workload: 16 tokens in, 64 out
        case("gpt2_generate", "gpt2", "generate", 1, 16, 64),
        # many documents at once through an f32 model
        case("gpt2_batch_prompt", "gpt2", "prompt", 16, 512, 0),
        # a chat answer behind a context of a page, one user
        case("ministral_decode", "ministral", "decode", 1, 1000, 8),
        # the same for eight users served together
        case("ministral_decode_batch", "ministral", "decode", 8, 1000, 8),
        # a question of ordinary length, read
        case("ministral_prompt", "ministral", "prompt", 1, 333, 0),
        # long documents of several users: the largest call
        case("ministral_long_prompts", "ministral", "prompt", 4, 2047, 0),
        # int8 weights, a whole call
        case("ministral_int8_generate", "ministral-w8", "generate", 1, 200, 16),
        # the hybrid design: a ragged batch of prompts, and answers written for a batch
        case("hybrid_ragged_prompts", "hybrid", "prompt", 4, 1000, 0, True),
        case("hybrid_generate_batch", "hybrid", "generate", 8, 65, 24, True),
        # the chunked design: a prompt over several chunks, and an answer to one user
        case("chunked_prompt", "chunked", "prompt", 1, 3000, 0),
        case("chunked_decode", "chunked", "decode", 1, 900, 24),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    model = rng.choice(["gpt2", "gpt2", "ministral", "ministral", "ministral", "ministral-w8", "ministral-w4", "hybrid", "chunked"])
    do = rng.choice(["prompt", "generate", "decode"] if model != "hybrid" else ["prompt", "generate"])   # a recurrent state cannot be taken back
    ragged = model in ("hybrid", "chunked") and rng.random() < 0.5
    batch = 1 if rng.random() < 0.5 else rng.randint(2, 16 if model == "gpt2" else 8)
    new = 0 if do == "prompt" else rng.randint(2, 24)
    longest = {"gpt2": 900, "ministral": 4000, "ministral-w8": 2000, "ministral-w4": 2000, "hybrid": 3000, "chunked": 4000}[model]
    most = 2000 if do == "generate" else 8000 if model in ("ministral", "chunked") else 7000
    prompt = _log_uniform(rng, 3, min(longest, most // batch))
    if model == "chunked" and do == "decode" and prompt % CHUNKED["chunk"] + new > CHUNKED["chunk"]:
        prompt -= new            # the cache holds the current chunk only: an answer that opens a new one cannot be tried again
    return dict(model=model, do=do, batch=batch, prompt=prompt, new=new, ragged=ragged)


def _lengths(case):
    """Prompt length of every sequence."""
    B, n = case["batch"], case["prompt"]
    return [max(1, n - (n * b * 5) // (8 * B)) if case["ragged"] else n for b in range(B)]


# ------------------------------------------------------------------------------------------ weights
def _plan(model):
    """parameter -> (shape, storage dtype, mean, standard deviation); the output matrix is made from the table."""
    bf, f32, out = torch.bfloat16, torch.float32, {}
    if model == "gpt2":
        c = GPT2
        d = c["width"]
        out["tok_embeddings.weight"] = ((c["vocab"], d), f32, 0.0, 1.0)
        out["pos_embeddings"] = ((c["context"], d), f32, 0.0, 0.2)
        for i in range(c["layers"]):
            p = f"blocks.{i}."
            for n, shape in (("attention.w_qkv", (d, 3 * d)), ("attention.w_out", (d, d)), ("feed_forward.w_in", (d, 4 * d)), ("feed_forward.w_out", (4 * d, d))):
                out[p + n] = (shape, f32, 0.0, 0.02)
                out[p + n.replace(".w_", ".b_")] = ((shape[1],), f32, 0.0, 0.02)
            for n in ("ln_1", "ln_2"):
                out[p + n + ".gamma"], out[p + n + ".beta"] = ((d,), f32, 1.0, 0.1), ((d,), f32, 0.0, 0.1)
        out["final_ln.gamma"], out["final_ln.beta"] = ((d,), f32, 1.0, 0.1), ((d,), f32, 0.0, 0.1)
        out["lm_head"] = ((d, c["vocab"]), f32, 0.0, d ** -0.5)
    elif model.startswith("ministral"):
        c = MINISTRAL
        d, q, kv = c["width"], c["heads"] * c["dim"], c["kv"] * c["dim"]
        out["tok_embeddings.weight"] = ((c["vocab"], d), bf, 0.0, 3.0)
        for i in range(c["layers"]):
            p = f"blocks.{i}."
            out[p + "norm_1.gamma"], out[p + "norm_2.gamma"] = ((d,), f32, 1.0, 0.1), ((d,), f32, 1.0, 0.1)
            for n, shape in (("attention.w_qkv", (d, q + 2 * kv)), ("attention.w_out", (q, d)), ("feed_forward.w_gate", (d, c["ff"])),
                             ("feed_forward.w_up", (d, c["ff"])), ("feed_forward.w_down", (c["ff"], d))):
                out[p + n] = (shape, bf, 0.0, 0.02)
        out["final_norm.gamma"] = ((d,), f32, 1.0, 0.1)
        out["lm_head"] = ((d, c["vocab"]), bf, 0.0, d ** -0.5)
    elif model == "hybrid":
        c, a = HYBRID, HYBRID["att"]
        d, inner, bc = c["width"], c["heads"] * c["vdim"], c["groups"] * c["state"]

        def mat(name, k, n):
            out[name] = ((k, n), bf, 0.0, k ** -0.5)

        out["tok_embeddings.weight"] = ((c["vocab"], d), bf, 0.0, 1.0)
        for i in range(4):
            p, q = f"blocks.{i}.", f"blocks.{i}.mixer."
            out[p + "norm_1.gamma"], out[p + "norm_1.beta"] = ((d,), f32, 1.0, 0.1), ((d,), f32, 0.0, 0.1)
            if i % 2 == 0:
                mat(q + "w_in", d, 2 * inner + 2 * bc + c["heads"])
                out[q + "conv"], out[q + "conv_bias"] = ((c["conv"], inner + 2 * bc), f32, 0.0, 0.5), ((inner + 2 * bc,), f32, 0.0, 0.1)
                out[q + "dt_bias"], out[q + "a_log"] = ((c["heads"],), f32, -4.5, 1.0), ((c["heads"],), f32, 1.8, 0.6)
                out[q + "d"], out[q + "norm.gamma"] = ((c["heads"],), f32, 1.0, 0.1), ((inner,), f32, 1.0, 0.1)
                mat(q + "w_out", inner, d)
            else:
                mat(q + "w_dq", d, a["q_rank"])
                out[q + "q_norm.gamma"] = ((a["q_rank"],), f32, 1.0, 0.1)
                mat(q + "w_uq", a["q_rank"], a["heads"] * (a["dim"] + a["rot"]))
                if i == 1:
                    mat(q + "w_dkv", d, a["kv_rank"] + a["rot"])
                    out[q + "kv_norm.gamma"] = ((a["kv_rank"],), f32, 1.0, 0.1)
                mat(q + "w_uk", a["kv_rank"], a["heads"] * a["dim"])
                mat(q + "w_uv", a["kv_rank"], a["heads"] * a["vdim"])
                mat(q + "w_out", a["heads"] * a["vdim"], d)
            mat(p + "feed_forward.w_gate", d, c["ff"])
            mat(p + "feed_forward.w_up", d, c["ff"])
            mat(p + "feed_forward.w_down", c["ff"], d)
            out[p + "scale_1"], out[p + "scale_2"] = ((d,), f32, 0.6, 0.1), ((d,), f32, 0.6, 0.1)
        out["final_norm.gamma"], out["final_norm.beta"] = ((d,), f32, 1.0, 0.1), ((d,), f32, 0.0, 0.1)
        out["lm_head"] = ((d, c["vocab"]), bf, 0.0, 1.0)      # this design's table and output matrix are one
    else:
        c = CHUNKED
        d = c["width"]
        out["tok_embeddings.weight"] = ((c["vocab"], d), bf, 0.0, 1.0)
        for i in range(c["layers"]):
            p, q = f"blocks.{i}.", f"blocks.{i}.mixer."
            for n, k, m in ((q + "w_qkvg", d, (c["heads"] + c["kv"]) * c["dim"] + c["kv"] * c["vdim"] + c["heads"]), (q + "w_out", c["heads"] * c["vdim"], d),
                            (p + "feed_forward.w_gate", d, c["ff"]), (p + "feed_forward.w_up", d, c["ff"]), (p + "feed_forward.w_down", c["ff"], d)):
                out[n] = ((k, m), bf, 0.0, k ** -0.5)
            out[q + "sink"] = ((c["heads"],), f32, 0.0, 1.0)
            out[p + "norm_1.gamma"], out[p + "norm_2.gamma"] = ((d,), f32, 1.0, 0.1), ((d,), f32, 1.0, 0.1)
        out["final_norm.gamma"] = ((d,), f32, 1.0, 0.1)
        out["lm_head"] = ((d, c["vocab"]), bf, 0.0, 0.3 * d ** -0.5)
    return out


def _shift(model):
    return 0 if model == "hybrid" else SHIFT


def _weight(model, name):
    """The parameter `name` on the GPU, in its storage dtype."""
    base = model.split("-")[0]
    shape, dtype, mean, std = _plan(base)[name]
    if name == "lm_head":
        table = _weight(base, "tok_embeddings.weight")
        return (table.roll(_shift(base), 0).T.float() * (std / _plan(base)["tok_embeddings.weight"][3])).to(dtype).contiguous()
    g = torch.Generator(device="cuda").manual_seed(zlib.crc32(f"{base}/{name}".encode()))
    return (torch.randn(shape, generator=g, device="cuda") * std + mean).to(dtype)


_backend = None
_models = {}


def _make(model, be):
    quant = {"w8": "w8", "w4": "w4g128"}.get(model.partition("-")[2])
    if model == "gpt2":
        c = GPT2
        m = models.Gpt(models.GptConfig(c["vocab"], c["context"], c["width"], c["layers"], c["heads"], 4, EPS), be, "F32")
    elif model.startswith("ministral"):
        c = MINISTRAL
        m = models.Ministral(models.MinistralConfig(c["vocab"], c["context"], c["width"], c["layers"], c["heads"], c["kv"], c["dim"], c["ff"], c["dim"], c["theta"], EPS),
                             be, "Bf16", residual_dtype="F32")
    elif model == "hybrid":
        c, a, layers = HYBRID, HYBRID["att"], []
        for i in range(4):
            if i % 2 == 0:
                mix = models.SsmMixerConfig(heads=c["heads"], vdim=c["vdim"], state=c["state"], groups=c["groups"], conv=c["conv"], norm_groups=c["groups"])
            else:
                mix = models.LatentMixerConfig(heads=a["heads"], dim=a["dim"], rot_dim=a["rot"], vdim=a["vdim"], q_rank=a["q_rank"], kv_rank=a["kv_rank"],
                                               scale=(a["dim"] + a["rot"]) ** -0.5, rope_base=a["base"], rope_scaling=a["yarn"], kv_from=1 if i > 1 else None)
            layers.append(models.DadupelLayer(mix, c["ff"], c["limit"]))
        m = models.Dadupel(models.DadupelConfig(vocab_size=c["vocab"], embed_dim=c["width"], eps=EPS, layers=layers), be)
    else:
        c = CHUNKED
        mix = models.ChunkedMixerConfig(heads=c["heads"], kv_heads=c["kv"], dim=c["dim"], vdim=c["vdim"], scale=c["scale"], rot_dims=c["dim"], rope_base=c["base"],
                                        chunk=c["chunk"])
        m = models.Fuzazen(models.FuzazenConfig(vocab_size=c["vocab"], embed_dim=c["width"], eps=EPS, layers=[models.FuzazenLayer(mix, c["ff"]) for _ in range(c["layers"])],
                                                embedding_scale=c["embedding_scale"], residual_mult=c["residual_mult"], logit_softcap=c["softcap"]), be)
    for name, (shape, dtype, *_) in _plan(model).items():
        w = _weight(model, name)
        raw = (w.view(torch.int16) if dtype == torch.bfloat16 else w).cpu().numpy().tobytes()
        m.set_param_bytes(name, TensorSpec("Bf16" if dtype == torch.bfloat16 else "F32", shape), raw)
        if quant and name.endswith(models.Ministral.QUANTIZABLE):
            m.quantize_param(name, quant)
    torch.cuda.empty_cache()
    return m


def _model(name):
    global _backend
    if _backend is None:
        _backend = HipBackend(0)
    if name not in _models:
        _models[name] = _make(name, _backend)
    return _models[name]


# ------------------------------------------------------------------------------------------ passes
def _prompts(case, seed):
    vocab = {"gpt2": GPT2, "ministral": MINISTRAL, "hybrid": HYBRID, "chunked": CHUNKED}[case["model"].split("-")[0]]["vocab"]
    rng = np.random.default_rng(seed)
    return [rng.integers(0, vocab, n).tolist() for n in _lengths(case)]


def _start(state):
    if len(state["prompts"]) == 1:
        return models.Generator(state["model"], state["prompts"][0], kv_cache_capacity=state["capacity"])
    return models.BatchGenerator(state["model"], state["prompts"], kv_cache_capacity=state["capacity"])


def prepare(case, seed):
    model = _model(case["model"])
    state = dict(model=model, prompts=_prompts(case, seed), do=case["do"], new=case["new"], capacity=None)
    if case["do"] == "decode":   # the prompt has been read; its caches have room for the answer
        state["capacity"] = min(-(-(case["prompt"] + case["new"]) // 128) * 128, model.context_length)
        gen = state["gen"] = _start(state)
        state["logits"] = gen.logits
        model.backend.synchronize()
    return state


def _take_back(gen, prompts, logits):
    """The generator as it was behind its prompt; the rows that an answer has written since count as free."""
    def back(slots, n):
        return [models.DecodeKvCache(s.keys, s.values, n, s.capacity) for s in slots]

    gen.logits = logits
    if isinstance(gen, models.BatchGenerator):
        gen.lens = [len(p) for p in prompts]
        gen.tokens = [list(p) for p in prompts]
        gen.caches = [back(c, len(p)) for c, p in zip(gen.caches, prompts)]
    else:
        gen.processed_len = len(prompts[0])
        gen.tokens = list(prompts[0])
        gen.caches = back(gen.caches, len(prompts[0]))


def run(state):
    be = state["model"].backend
    if state["do"] == "prompt":
        return {"logits": be.to_numpy(_start(state).logits)}
    if state["do"] == "generate":
        gen = _start(state)
        tokens = gen.generate(state["new"])
    else:
        gen = state["gen"]
        _take_back(gen, state["prompts"], state["logits"])
        tokens = [gen.step() for _ in range(state["new"])]
    return {"tokens": np.asarray(tokens, np.int64), "logits": be.to_numpy(gen.logits)}


def _consumed(case):
    """Written tokens that have gone through the model when the logits are read: a whole call of one sequence ends with a token."""
    return case["new"] - 1 if case["do"] == "generate" and case["batch"] == 1 else case["new"]


# ------------------------------------------------------------------------------------------ work
def _sizes(model):
    """(matrix elements of all layers, of the output matrix, bytes of an element, of an activation)"""
    base = model.split("-")[0]
    mats = sum(s[0] * s[1] for n, (s, *_) in _plan(base).items() if len(s) == 2 and n not in ("tok_embeddings.weight", "pos_embeddings", "lm_head") and not n.endswith("conv"))
    head = int(np.prod(_plan(base)["lm_head"][0]))
    return mats, head, {"gpt2": 4.0, "ministral-w8": 1.0, "ministral-w4": 0.5 + 2 / 128}.get(model, 2.0), 4 if base == "gpt2" else 2


def _sequence(model, first, last, ab):
    """(cache bytes, flops) of the mixers for positions first .. last - 1 of one sequence, taken one at a time if first > 0."""
    base = model.split("-")[0]
    n = last - first
    pairs = (last * (last + 1) - first * (first + 1)) / 2.0
    reads = pairs if first else 0.0
    if base == "gpt2":
        row, per = 2 * GPT2["width"], 4.0 * GPT2["width"]
        return ab * GPT2["layers"] * row * (n + reads), GPT2["layers"] * per * pairs
    if base == "ministral":
        c = MINISTRAL
        return ab * c["layers"] * 2 * c["kv"] * c["dim"] * (n + reads), c["layers"] * 4.0 * c["heads"] * c["dim"] * pairs
    if base == "hybrid":
        c, a = HYBRID, HYBRID["att"]
        state = c["heads"] * c["state"] * c["vdim"]
        return (2 * 4 * state * (1 + (n if first else 0)) + 2 * (a["kv_rank"] + a["rot"]) * (n + 2 * reads),
                2 * 6.0 * n * state + 2 * 2.0 * a["heads"] * (a["dim"] + a["rot"] + a["vdim"]) * pairs)
    c = CHUNKED
    pairs = sum(p % c["chunk"] + 1.0 for p in range(first, last))
    row = c["kv"] * (c["dim"] + c["vdim"])
    return ab * c["layers"] * row * (min(n, c["chunk"]) + (pairs if first else 0.0)), c["layers"] * 2.0 * c["heads"] * (c["dim"] + c["vdim"]) * pairs


def work(case):
    mats, head, wb, ab = _sizes(case["model"])
    lens, B, steps = _lengths(case), case["batch"], _consumed(case)
    nbytes = flops = 0.0
    if case["do"] != "decode":
        rows = sum(lens)
        nbytes += wb * (mats + head) + 4 * B * head / _plan(case["model"].split("-")[0])["lm_head"][0][0]
        flops += 2.0 * rows * mats + 2.0 * B * head
        for n in lens:
            b, f = _sequence(case["model"], 0, n, ab)
            nbytes, flops = nbytes + b, flops + f
    nbytes += steps * (wb * (mats + head) + 4 * B * head / _plan(case["model"].split("-")[0])["lm_head"][0][0])
    flops += steps * 2.0 * B * (mats + head)
    for n in lens if steps else []:
        b, f = _sequence(case["model"], n, n + steps, ab)
        nbytes, flops = nbytes + b, flops + f
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what a result is off its value in 64 bits: f32 sums 1.1e-6; bf16 operands 0.7 % behind 26 layers, 0.36 % and
    0.23 % behind four."""
    rel = {"gpt2": 5e-6, "hybrid": 0.015, "chunked": 0.01}.get(case["model"], 0.028)
    return {"rel": rel, "max": 9 * rel, "differ": 0.0}


# ------------------------------------------------------------------------------------------ the same in 64 bits
class _F64:
    """The models in plain torch, in float64 and without caches: a written token's logits are those of the whole text."""

    def __init__(self, model):
        self.model = model

    def w(self, name):
        w = _weight(self.model, name).double()
        if self.model.endswith("-w8") and name.endswith(models.Ministral.QUANTIZABLE):    # one scale per column
            s = (w.abs().amax(0).float() / 127).bfloat16()
            s = torch.where(s == 0, torch.ones_like(s), s).float()
            w = ((w.float() / s).round().clamp(-127, 127)).double() * s.double()
        elif self.model.endswith("-w4") and name.endswith(models.Ministral.QUANTIZABLE):  # one scale per column and 128 rows
            g = w.float().view(-1, 128, w.shape[1])
            s = (g.abs().amax(1, keepdim=True) / 7).bfloat16()
            s = torch.where(s == 0, torch.ones_like(s), s).float()
            w = ((g / s).round().clamp(-7, 7).double() * s.double()).view(w.shape)
        return w

    @staticmethod
    def over_rms(x):
        return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt()

    def rms(self, x, name):
        return self.over_rms(x) * self.w(name)

    def ln(self, x, name):
        x = x - x.mean(-1, keepdim=True)
        return self.over_rms(x) * self.w(name + ".gamma") + self.w(name + ".beta")

    @staticmethod
    def attend(q, k, v, scale, sink=None, chunk=1 << 30):
        """q [T, H, D], k [T, G, D], v [T, G, V]: causal, within chunks; a sink is one more term of a head's denominator."""
        T, H, G = q.shape[0], q.shape[1], k.shape[1]
        out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
        for lo in range(0, T, chunk):
            hi = min(T, lo + chunk)
            hide = torch.ones(hi - lo, hi - lo, dtype=torch.bool, device=q.device).triu(1)
            for h in range(H):
                s = (q[lo:hi, h] @ k[lo:hi, h * G // H].T * scale).masked_fill_(hide, -math.inf)
                if sink is not None:
                    s = torch.cat([s, sink[h].expand(hi - lo, 1)], 1)
                out[lo:hi, h] = s.softmax(-1)[:, :hi - lo] @ v[lo:hi, h * G // H]
        return out

    @staticmethod
    def angles(T, freqs):
        a = torch.arange(T, dtype=torch.float64, device="cuda")[:, None] * torch.tensor(freqs, dtype=torch.float64, device="cuda")
        return a.cos()[:, None], a.sin()[:, None]

    @staticmethod
    def turn_pairs(x, cos, sin):
        u, v = x[..., 0::2], x[..., 1::2]
        return torch.stack([u * cos - v * sin, v * cos + u * sin], -1).flatten(-2)

    def swiglu(self, h, p):
        return (torch.nn.functional.silu(h @ self.w(p + "w_gate")) * (h @ self.w(p + "w_up"))) @ self.w(p + "w_down")

    def gpt2(self, t):
        c, T = GPT2, len(t)
        x = self.w("tok_embeddings.weight")[t] + self.w("pos_embeddings")[:T]
        for i in range(c["layers"]):
            p = f"blocks.{i}."
            q, k, v = (self.ln(x, p + "ln_1") @ self.w(p + "attention.w_qkv") + self.w(p + "attention.b_qkv")).view(T, 3, c["heads"], -1).unbind(1)
            ctx = self.attend(q, k, v, q.shape[2] ** -0.5).reshape(T, -1)
            x = x + ctx @ self.w(p + "attention.w_out") + self.w(p + "attention.b_out")
            h = torch.nn.functional.gelu(self.ln(x, p + "ln_2") @ self.w(p + "feed_forward.w_in") + self.w(p + "feed_forward.b_in"))
            x = x + h @ self.w(p + "feed_forward.w_out") + self.w(p + "feed_forward.b_out")
        return self.ln(x, "final_ln")

    def ministral(self, t):
        c, T = MINISTRAL, len(t)
        half = c["dim"] // 2
        cos, sin = self.angles(T, [c["theta"] ** (-i / half) for i in range(half)])

        def turn(x):
            u, v = x[..., :half], x[..., half:]
            return torch.cat([u * cos - v * sin, v * cos + u * sin], -1)

        x = _weight(self.model, "tok_embeddings.weight")[t].double()
        for i in range(c["layers"]):
            p = f"blocks.{i}."
            qkv = (self.rms(x, p + "norm_1.gamma") @ self.w(p + "attention.w_qkv")).view(T, -1, c["dim"])
            q, k, v = qkv.split([c["heads"], c["kv"], c["kv"]], 1)
            x = x + self.attend(turn(q), turn(k), v, c["dim"] ** -0.5).reshape(T, -1) @ self.w(p + "attention.w_out")
            x = x + self.swiglu(self.rms(x, p + "norm_2.gamma"), p + "feed_forward.")
        return self.rms(x, "final_norm.gamma")

    def hybrid(self, t):
        c, a, T = HYBRID, HYBRID["att"], len(t)
        H, V, N, G = c["heads"], c["vdim"], c["state"], c["groups"]
        inner, bc, rot = H * V, G * N, a["rot"]
        factor, original, fast, slow = a["yarn"]
        lo, hi = (rot * math.log(original / (2 * math.pi * n)) / (2 * math.log(a["base"])) for n in (fast, slow))
        lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), rot - 1)
        freqs = []
        for i in range(rot // 2):
            f, r = a["base"] ** (-2.0 * i / rot), min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0)
            freqs.append(f / factor * r + f * (1 - r))
        mag = 0.1 * math.log(factor) + 1.0
        cos, sin = (z * mag for z in self.angles(T, freqs))
        x = self.w("tok_embeddings.weight")[t]
        for i in range(4):
            p, q = f"blocks.{i}.", f"blocks.{i}.mixer."
            h = self.ln(x, p + "norm_1")
            if i % 2 == 0:
                z, xbc, dt = (h @ self.w(q + "w_in")).split([inner, inner + 2 * bc, H], 1)
                rows = torch.cat([xbc.new_zeros(c["conv"] - 1, xbc.shape[1]), xbc])
                taps = self.w(q + "conv")
                xbc = torch.nn.functional.silu(self.w(q + "conv_bias") + sum(taps[k] * rows[k:k + T] for k in range(c["conv"])))
                xs, Bs, Cs = xbc.split([inner, bc, bc], 1)
                xs, Bs, Cs = xs.view(T, H, 1, V), Bs.view(T, G, N).repeat_interleave(H // G, 1)[..., None], Cs.view(T, G, N).repeat_interleave(H // G, 1)[..., None]
                dt = torch.nn.functional.softplus(dt + self.w(q + "dt_bias"))
                keep, gain = torch.exp(-self.w(q + "a_log").exp() * dt)[..., None, None], dt[..., None, None]
                S, y = torch.zeros(H, N, V, dtype=torch.float64, device="cuda"), torch.empty(T, H, V, dtype=torch.float64, device="cuda")
                for n in range(T):
                    S = S * keep[n] + (gain[n] * Bs[n]) * xs[n]
                    y[n] = (S * Cs[n]).sum(1)
                y = (y + self.w(q + "d")[:, None] * xs[:, :, 0]).reshape(T, inner) * torch.nn.functional.silu(z)
                mixed = self.over_rms(y.view(T, G, -1)).reshape(T, inner) * self.w(q + "norm.gamma")
            else:
                qs = (self.rms(h @ self.w(q + "w_dq"), q + "q_norm.gamma") @ self.w(q + "w_uq")).view(T, a["heads"], -1)
                qs = torch.cat([qs[..., :a["dim"]], self.turn_pairs(qs[..., a["dim"]:], cos, sin)], -1)
                if i == 1:
                    raw = h @ self.w(q + "w_dkv")
                    lat, kr = self.rms(raw[:, :a["kv_rank"]], q + "kv_norm.gamma"), self.turn_pairs(raw[:, None, a["kv_rank"]:], cos, sin)
                k, v = (lat @ self.w(q + "w_uk")).view(T, a["heads"], -1), (lat @ self.w(q + "w_uv")).view(T, a["heads"], -1)
                mixed = self.attend(qs, torch.cat([k, kr.expand(-1, a["heads"], -1)], -1), v, (a["dim"] + rot) ** -0.5).reshape(T, -1)
            f = p + "feed_forward."
            g, u = (h @ self.w(f + "w_gate")).clamp(max=c["limit"]), (h @ self.w(f + "w_up")).clamp(-c["limit"], c["limit"])
            ff = (g * torch.sigmoid(1.702 * g) * (u + 1)) @ self.w(f + "w_down")
            x = x + mixed @ self.w(q + "w_out") * self.w(p + "scale_1") + ff * self.w(p + "scale_2")
        return self.ln(x, "final_norm")

    def chunked(self, t):
        c, T = CHUNKED, len(t)
        cos, sin = self.angles(T, [c["base"] ** (-2.0 * i / c["dim"]) for i in range(c["dim"] // 2)])
        x = self.w("tok_embeddings.weight")[t] * c["embedding_scale"]
        for i in range(c["layers"]):
            p, q = f"blocks.{i}.", f"blocks.{i}.mixer."
            qs, ks, vs, gate = (x @ self.w(q + "w_qkvg")).split([c["heads"] * c["dim"], c["kv"] * c["dim"], c["kv"] * c["vdim"], c["heads"]], 1)
            qs, ks = (self.over_rms(self.turn_pairs(z.reshape(T, -1, c["dim"]), cos, sin)) for z in (qs, ks))
            ctx = self.attend(qs, ks, vs.reshape(T, -1, c["vdim"]), c["scale"], self.w(q + "sink"), c["chunk"]) * torch.sigmoid(gate)[..., None]
            x = x + c["residual_mult"] * self.rms(ctx.reshape(T, -1) @ self.w(q + "w_out"), p + "norm_1.gamma")
            x = x + c["residual_mult"] * self.rms(self.swiglu(x, p + "feed_forward."), p + "norm_2.gamma")
        return self.rms(x, "final_norm.gamma")


def exact(case, seed):
    """The logits; greedy text is known beforehand, and checked against the logits that choose it."""
    base = case["model"].split("-")[0]
    ref, vocab, n, out = _F64(case["model"]), _plan(base)["lm_head"][0][1], _consumed(case), []
    head = ref.w("lm_head")
    for prompt in _prompts(case, seed):
        text = list(prompt)
        for _ in range(n):
            text.append((text[-1] + _shift(base)) % vocab)
        logits = getattr(ref, base)(torch.tensor(text, device="cuda"))[len(prompt) - 1:] @ head
        if base == "chunked":
            logits = CHUNKED["softcap"] * torch.tanh(logits / CHUNKED["softcap"])
        if logits[:-1].argmax(-1).tolist() != text[len(prompt):]:
            return None
        out.append(logits[-1].cpu().numpy())
    return {"logits": np.stack(out)} if case["do"] == "prompt" else {"tokens": None, "logits": np.stack(out)}
