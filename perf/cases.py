"""The work that is timed: serving steps of the engine, from one request's next token to a step of 2,048 prompt tokens.

A case is one of four kinds of call:

* ``decode``: one token each for ``batch`` live requests (the step that serving repeats for every token: the recorded step with
  its sampling, ``StepRunner.run`` with the positions reserved by the caller, as the scheduler calls it).  The tokens are given,
  so that two implementations see the same inputs at every step, and the reservation is dropped afterwards: the next pass is the
  same step again.
* ``prefill``: whole prompts through one step, logits of the last position (or of every position: ``score``); the requests are
  closed afterwards.
* ``mixed``: a portion of a prompt beside the one-token entries of ``batch`` live requests.
* ``generate``: ``CausalLanguageModel.generate``, greedy: scheduling, prompts, decoding ahead of the host, tokens on the host.

Models: GPT-2 layer sizes (124M, 355M, 1.5B parameters; vocabulary 50,257, 1,024 positions) and a Virudra of the 355M's sizes;
random weights N(0, 0.02) (with a Virudra's own 0.05 the scores of 24 layers are so sharp that bfloat16 rounding alone moves the
logits by 7 %), uniform-random token ids, greedy sampling.
"""
import math
import struct

import numpy as np
import torch

GPT2 = {"124m": (12, 768, 12), "355m": (24, 1024, 16), "1.5b": (48, 1600, 25)}      # layers, width, heads (head size 64)
VOCAB, POSITIONS = 50257, 1024
EXPERTS, TOP = 8, 2
DEV = "cuda:0"


def listed():
    def decode(name, model, batch, context, spread=0.0, design="gpt2"):
        return {"name": name, "kind": "decode", "design": design, "model": model, "dtype": "bfloat16", "batch": batch,
                "context": context, "spread": spread}

    def prefill(name, model, prompts, length, spread=0.0, dtype="bfloat16", score=False):
        return {"name": name, "kind": "prefill", "design": "gpt2", "model": model, "dtype": dtype, "prompts": prompts,
                "length": length, "spread": spread, "score": score}

    return [
        # one user in a conversation: every kernel is small, the step is launches and latencies
        decode("decode-124m-1", "124m", 1, 512),
        # the benchmark's headline step
        decode("decode-124m-8", "124m", 8, 512),
        # a busy server: an odd number of requests (the recorded step is padded), contexts of many lengths
        decode("decode-355m-33", "355m", 33, 900, 0.9),
        # a large model for a few users
        decode("decode-1.5b-3", "1.5b", 3, 301, 0.5),
        # a large model, full batch: weights and cache come from memory
        decode("decode-1.5b-64", "1.5b", 64, 512),
        # another design (root-mean-square norms, gated and routed feed-forwards, attention with a bias by distance)
        decode("decode-virudra-355m-5", "355m", 5, 640, 0.7, design="virudra"),
        # time to the first token of a short question
        prefill("prefill-124m-1x37", "124m", 1, 37),
        # three prompts of odd lengths admitted in one step
        prefill("prefill-355m-3x701", "355m", 3, 701, 0.8),
        # the largest step: a full token budget on the largest model
        prefill("prefill-1.5b-2x1024", "1.5b", 2, 1024),
        # continuous batching: a portion of a long prompt beside the others' decoding
        {"name": "mixed-355m-512+40", "kind": "mixed", "design": "gpt2", "model": "355m", "dtype": "bfloat16", "batch": 40,
         "context": 600, "spread": 0.8, "portion": 512, "done": 256},
        # true 32-bit, every position's logits: prompts scored, or a trace replayed against a reference
        prefill("score-f32-124m-2x300", "124m", 2, 300, 0.4, dtype="float32", score=True),
        # true 32-bit through the engine's own loop
        {"name": "generate-f32-124m-4", "kind": "generate", "design": "gpt2", "model": "124m", "dtype": "float32", "prompts": 4,
         "length": 61, "spread": 0.6, "new": 12},
    ]


def draw(rng):
    def log_int(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    model = rng.choice(["124m", "355m", "1.5b"])
    spread = round(rng.uniform(0.0, 0.9), 3)
    kind = rng.choice(["decode"] * 5 + ["virudra"] + ["prefill"] * 3 + ["mixed", "score", "generate"])
    if kind == "decode":
        return {"kind": "decode", "design": "gpt2", "model": model, "dtype": "bfloat16", "batch": log_int(1, 64),
                "context": log_int(16, 1000), "spread": spread}
    if kind == "virudra":
        return {"kind": "decode", "design": "virudra", "model": rng.choice(["124m", "355m"]), "dtype": "bfloat16",
                "batch": log_int(1, 64), "context": log_int(16, 1000), "spread": spread}
    if kind == "prefill":
        total, prompts = log_int(5, 2048), rng.randint(1, 6)
        return {"kind": "prefill", "design": "gpt2", "model": model, "dtype": "bfloat16", "prompts": prompts,
                "length": max(3, min(1024, total // prompts)), "spread": spread, "score": False}
    if kind == "mixed":
        portion = log_int(16, 512)
        return {"kind": "mixed", "design": "gpt2", "model": model, "dtype": "bfloat16", "batch": log_int(1, 63),
                "context": log_int(16, 1000), "spread": spread, "portion": portion, "done": rng.randint(0, 1024 - portion)}
    if kind == "score":
        prompts = rng.randint(1, 3)
        return {"kind": "prefill", "design": "gpt2", "model": rng.choice(["124m", "355m"]), "dtype": "float32", "prompts": prompts,
                "length": max(3, log_int(8, 600) // prompts), "spread": spread, "score": rng.random() < 0.5}
    return {"kind": "generate", "design": "gpt2", "model": "124m", "dtype": "float32", "prompts": rng.randint(1, 8),
            "length": log_int(4, 100), "spread": spread, "new": rng.randint(4, 12)}


# ---------------------------------------------------------------------------------------------- sizes
def lengths(n, longest, spread):
    """``n`` lengths from ``longest`` down to ``(1 - spread) * longest``, in no order."""
    return [max(1, int(round(longest * (1.0 - spread * ((i * 0.6180339887) % 1.0))))) for i in range(n)]


def virudra_sizes(model):
    n_layer, width, heads = GPT2[model]
    return n_layer, width, heads, (8 * width // 3 + 63) // 64 * 64


def model_config(case):
    n_layer, width, heads = GPT2[case["model"]]
    if case["design"] == "gpt2":
        return {"architectures": ["GPT2LMHeadModel"], "model_type": "gpt2", "vocab_size": VOCAB, "n_positions": POSITIONS,
                "n_layer": n_layer, "n_embd": width, "n_head": heads, "layer_norm_epsilon": 1e-5,
                "activation_function": "gelu_new", "bos_token_id": VOCAB - 1, "eos_token_id": VOCAB - 1}
    ff = virudra_sizes(case["model"])[3]
    mixer = {"heads": heads, "kv_heads": heads, "dim": 64, "vdim": 64, "scale": 0.125, "bias_max": 512, "bias_buckets": 32,
             "q_temp": {"coef": 0.1, "every": 256}}
    layers = [{"type": "attention", "mixer": mixer,
               "mlp": {"kind": "dense", "ff": ff} if i % 2 == 0 else
                      {"kind": "moe", "expert": {"ff": ff // 2}, "router": {"experts": EXPERTS, "top": TOP}}}
              for i in range(n_layer)]
    return {"architecture": "Virudra", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-5}, "logit_softcap": 50.0,
            "layers": layers, "max_positions": POSITIONS}


def step_lengths(case):
    """(new tokens, positions before them) of every request of a pass."""
    kind = case["kind"]
    if kind == "decode":
        return [(1, c) for c in lengths(case["batch"], min(case["context"], POSITIONS - 1), case["spread"])]
    if kind == "mixed":
        return [(1, c) for c in lengths(case["batch"], min(case["context"], POSITIONS - 1), case["spread"])] + [(case["portion"], case["done"])]
    return [(n, 0) for n in lengths(case["prompts"], case["length"], case["spread"])]


# ---------------------------------------------------------------------------------------------- weights and inputs
def checkpoint(case, seed):
    """The tensors of a checkpoint by name, as a file of them would hold them, on the GPU."""
    n_layer, E, H = GPT2[case["model"]]
    dtype = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)

    def normal(shape, std, mean=0.0):
        t = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).mul_(std)
        return (t.add_(mean) if mean else t).to(dtype)

    t = {}
    if case["design"] == "gpt2":
        t["wte.weight"], t["wpe.weight"] = normal((VOCAB, E), 0.02), normal((POSITIONS, E), 0.01)
        for i in range(n_layer):
            p = f"h.{i}."
            for n in ("ln_1", "ln_2"):
                t[p + n + ".weight"], t[p + n + ".bias"] = normal((E,), 0.1, 1.0), normal((E,), 0.02)
            for n, a, b in (("attn.c_attn", E, 3 * E), ("attn.c_proj", E, E), ("mlp.c_fc", E, 4 * E), ("mlp.c_proj", 4 * E, E)):
                t[p + n + ".weight"], t[p + n + ".bias"] = normal((a, b), 0.02), normal((b,), 0.02)
        t["ln_f.weight"], t["ln_f.bias"] = normal((E,), 0.1, 1.0), normal((E,), 0.02)
        return t
    ff = virudra_sizes(case["model"])[3]
    t["embed"] = normal((VOCAB, E), 1.0)
    for i in range(n_layer):
        p = f"l{i}."
        for n in ("norm1", "norm1b", "norm2", "norm2b"):
            t[p + n] = normal((E,), 0.1)
        for n in "qkvo":
            t[p + "mix." + n] = normal((E, E), 0.02)
        t[p + "mix.rel"] = normal((32, H), 0.5)
        for q, F in [("mlp.", ff)] if i % 2 == 0 else [(f"mlp.e{j}.", ff // 2) for j in range(EXPERTS)]:
            t[p + q + "gate"], t[p + q + "up"], t[p + q + "down"] = normal((F, E), 0.02), normal((F, E), 0.02), normal((E, F), 0.02)
        if i % 2:
            t[p + "mlp.table"] = torch.rand((VOCAB, EXPERTS), generator=g, device=DEV).argsort(1)[:, :TOP].to(torch.int32).contiguous()
    t["final.norm"], t["head"] = normal((E,), 0.1), normal((VOCAB, E), 0.02)
    return t


def token_ids(case, seed):
    """Every request's tokens up to the end of the pass."""
    rng = np.random.default_rng(seed)
    return [[int(x) for x in rng.integers(0, VOCAB - 1, size=past + n)] for n, past in step_lengths(case)]


def prepare(case, seed):
    import deliverance_amd.models  # noqa: F401  (registers the architectures)
    from deliverance_amd import EngineConfig
    from deliverance_amd.engine.engine import CausalLanguageModel
    from deliverance_amd.engine.step import StepEntry
    from deliverance_amd.models.causal_lm import CausalLM
    from deliverance_amd.registry import ModelSupport
    from deliverance_amd.sampling.params import GeneratorParameters
    from deliverance_amd.sampling.sampler import RECORD_WORDS, JavaRandom, device_record

    config = model_config(case)
    arch = ModelSupport.detect(config)
    mc = arch.read_config(config)
    dtype = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32
    model = CausalLM(mc, arch.bind_tensors(mc, checkpoint(case, seed)), dtype, DEV)
    steps, ids = step_lengths(case), token_ids(case, seed)
    engine = CausalLanguageModel(model, EngineConfig(dtype=case["dtype"], max_num_seqs=max(2, len(steps)), max_batch_tokens=2048,
                                                     max_chunk=1024, max_cached_tokens=sum(-(-(n + past + 16) // 16) * 16 for n, past in steps)))
    state = {"case": case, "engine": engine}
    if case["kind"] == "generate":
        state["prompts"] = ids
        state["params"] = GeneratorParameters(max_tokens=case["new"], ignore_eos=True)
        return state
    # the live requests' contexts
    batch, room = [], 0
    for rid, (t, (n, past)) in enumerate(zip(ids, steps)):
        if past:
            if room + past > 8192:
                engine.runner.run(batch)
                batch, room = [], 0
            batch.append(StepEntry(rid, t[:past], []))
            room += past
    if batch:
        engine.runner.run(batch)
    state["rids"] = [rid for rid, (n, past) in enumerate(steps)]
    state["entries"] = [StepEntry(rid, t[past:], list(range(n)) if case.get("score") else [n - 1])
                        for rid, (t, (n, past)) in enumerate(zip(ids, steps))]
    state["reserved"] = case["kind"] != "prefill"
    state["records"] = None
    if case["kind"] == "mixed" and case["done"] == 0:
        engine.cache.manager.open(len(steps) - 1)
    if case["kind"] == "decode":
        record = struct.unpack(f"<{RECORD_WORDS}i", device_record(GeneratorParameters(), JavaRandom(seed), VOCAB))
        state["records"] = list(record) * len(steps)
    return state


def run(state):
    engine = state["engine"]
    if state["case"]["kind"] == "generate":
        return [r.generated_tokens for r in engine.generate(state["prompts"], state["params"])]
    manager = engine.cache.manager
    if state["reserved"]:
        for e in state["entries"]:
            manager.extend(e.rid, len(e.tokens))
        logits, _ = engine.runner.run(state["entries"], reserved=True, sample_records=state["records"])
        for rid in state["rids"]:
            manager.rollback(rid)
    else:
        logits, _ = engine.runner.run(state["entries"])
        for rid in state["rids"]:
            manager.close(rid)
    return logits


# ---------------------------------------------------------------------------------------------- what a pass needs
def work(case):
    """Every matrix read once (of the experts those that the tokens choose), the live keys and values, the rows of logits; the
    products of the parameters that a token uses, and of attention."""
    n_layer, E, H = GPT2[case["model"]]
    el = 2 if case["dtype"] == "bfloat16" else 4
    if case["design"] == "gpt2":
        read = used = n_layer * 12 * E * E
    else:
        ff = virudra_sizes(case["model"])[3]
        half = n_layer // 2
        used = n_layer * (4 * E * E + 3 * E * ff)
        chosen = EXPERTS * (1.0 - (1.0 - TOP / EXPERTS) ** case["batch"])       # experts that some token names, of tables drawn at random
        read = n_layer * 4 * E * E + (n_layer - half) * 3 * E * ff + half * chosen * 3 * E * (ff // 2)
    steps = step_lengths(case)
    if case["kind"] != "generate":
        passes = [(steps, sum(n for n, _ in steps) if case.get("score") else len(steps))]
    else:
        passes = [(steps, len(steps))] + [([(1, n + k) for n, _ in steps], len(steps)) for k in range(case["new"] - 1)]
    nbytes = flops = 0
    for requests, rows in passes:
        tokens = sum(n for n, _ in requests)
        nbytes += (read + VOCAB * E) * el + tokens * E * el + rows * VOCAB * 4
        nbytes += sum(past + n for n, past in requests) * 2 * E * el * n_layer
        flops += 2 * used * tokens + 2 * rows * VOCAB * E
        flops += 4 * E * n_layer * sum(n * past + n * (n + 1) // 2 for n, past in requests)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Four times what the path shows against 64 bits: 6e-7 in 32 bits; in bfloat16 0.0038 to 0.005, the Virudra 0.0068."""
    if case["kind"] == "generate":
        return {"differ": 0.01}            # greedy in 32-bit: ties alone may differ
    if case["dtype"] == "float32":
        return {"rel": 3e-6, "max": 4e-5}
    return {"rel": 0.02, "max": 0.15} if case["design"] == "gpt2" else {"rel": 0.028, "max": 0.2}


# ---------------------------------------------------------------------------------------------- in 64 bits
def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _rows(f, x, step=8192):
    return torch.cat([f(x[a:a + step]) for a in range(0, x.shape[0], step)])


def _attention(qkv, T, H, scale, bias=None, gain=None):
    q, k, v = (z.reshape(T, H, 64).transpose(0, 1).contiguous() for z in qkv.chunk(3, dim=1))
    if gain is not None:
        q = q * gain[None, :, None]
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    if bias is not None:
        s = s + bias
    s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=DEV).triu(1), float("-inf"))
    return torch.matmul(torch.softmax(s, dim=-1), v).transpose(0, 1).reshape(T, H * 64)


def _forward64(case, W, ids, want):
    """Logits in 64 bits of rows ``want`` (per sequence) of whole sequences ``ids``."""
    n_layer, E, H = GPT2[case["model"]]
    gpt2 = case["design"] == "gpt2"
    at = [0]
    for t in ids:
        at.append(at[-1] + len(t))
    flat = torch.tensor([x for t in ids for x in t], device=DEV)
    pos = torch.tensor([i for t in ids for i in range(len(t))], device=DEV)

    def w(name):
        return W[name].double()

    def layer_norm(x, name):
        m = x.mean(1, keepdim=True)
        return (x - m) / torch.sqrt(((x - m) ** 2).mean(1, keepdim=True) + 1e-5) * w(name + ".weight") + w(name + ".bias")

    def rms_norm(x, name):
        return x / torch.sqrt((x ** 2).mean(1, keepdim=True) + 1e-5) * (1.0 + w(name))

    def attend(qkv, bias_table=None):
        out = []
        for a, b in zip(at, at[1:]):
            T = b - a
            if bias_table is None:
                out.append(_attention(qkv[a:b], T, H, 0.125))
                continue
            row = torch.tensor([d if d < 16 else min(31, 16 + int(math.floor(math.log(d / 16) / math.log(512 / 16) * 16))) for d in range(T)], device=DEV)
            dist = (torch.arange(T, device=DEV)[:, None] - torch.arange(T, device=DEV)[None, :]).clamp(min=0)
            gain = torch.tensor([1.0 + 0.1 * math.log((p + 1) // 256 + 1) for p in range(T)], device=DEV, dtype=torch.float64)
            out.append(_attention(qkv[a:b], T, H, 0.125, bias_table[row[dist]].permute(2, 0, 1), gain))
        return torch.cat(out)

    def gated(h, p, act):
        return (act(h @ w(p + "gate").t()) * (h @ w(p + "up").t())) @ w(p + "down").t()

    silu = torch.nn.functional.silu
    x = w("wte.weight")[flat] + w("wpe.weight")[pos] if gpt2 else w("embed")[flat]
    for i in range(n_layer):
        if gpt2:
            p = f"h.{i}."
            wqkv, wo, wfc, wproj = (w(p + n + ".weight") for n in ("attn.c_attn", "attn.c_proj", "mlp.c_fc", "mlp.c_proj"))
            qkv = _rows(lambda r: layer_norm(r, p + "ln_1") @ wqkv + w(p + "attn.c_attn.bias"), x)
            x = x + attend(qkv) @ wo + w(p + "attn.c_proj.bias")
            x = x + _rows(lambda r: _gelu(layer_norm(r, p + "ln_2") @ wfc + w(p + "mlp.c_fc.bias")) @ wproj + w(p + "mlp.c_proj.bias"), x)
            continue
        p = f"l{i}."
        h = rms_norm(x, p + "norm1")
        qkv = torch.cat([h @ w(p + "mix." + n).t() for n in "qkv"], dim=1)
        x = x + rms_norm(attend(qkv, w(p + "mix.rel")) @ w(p + "mix.o").t(), p + "norm1b")
        h = rms_norm(x, p + "norm2")
        if i % 2 == 0:
            y = gated(h, p + "mlp.", _gelu)
        else:
            y = torch.zeros_like(h)
            chosen = W[p + "mlp.table"][flat]
            for j in range(EXPERTS):
                rows = (chosen == j).any(1).nonzero()[:, 0]
                if rows.numel():
                    y[rows] += gated(h[rows], f"{p}mlp.e{j}.", silu) / TOP
        x = x + rms_norm(y, p + "norm2b")
    e = x[torch.tensor([a + r for a, rows in zip(at, want) for r in rows], device=DEV)]
    if gpt2:
        return layer_norm(e, "ln_f") @ w("wte.weight").t()
    return 50.0 * torch.tanh(rms_norm(e, "final.norm") @ w("head").t() / 50.0)


def exact(case, seed):
    W, ids = checkpoint(case, seed), token_ids(case, seed)
    if case["kind"] == "generate":
        out = [list(t) for t in ids]
        for _ in range(case["new"]):
            for t, row in zip(out, _forward64(case, W, out, [[len(t) - 1] for t in out])):
                t.append(int(row.argmax()))
        return [t[-case["new"]:] for t in out]
    want = [list(range(past, past + n)) if case.get("score") else [past + n - 1] for n, past in step_lengths(case)]
    return _forward64(case, W, ids, want)
