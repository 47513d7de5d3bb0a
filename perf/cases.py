"""What this library is asked to do in earnest: requests to its seven decoder designs, through the engine's own entry points.

A case is a dict of plain values:

    design, width, heads, kv_heads, head_dim, ff, vocab, layers, dtype   the model (``model_config`` writes its config.json)
    batch, lo, hi     sequences of the request and the range of their prompt lengths (``prompt_lengths`` deals them out)
    new               decode steps after the prompts: 0 stops at the prompts' logits (scoring, or a first token)
    held              the prompts lie in the cache before the call (all but their last token): a conversation goes on

One pass is one request: a slot for each sequence, the prompts in one step, then ``new`` steps of the generation loop's own
runner with greedy sampling, then the logits after the last token, and the slots are given back.  With ``held`` the slots
stay and the sequences are taken back to where they stood.  It returns the logits after the prompts, the tokens chosen and
the logits after the last of them, which depend on everything that the decode steps left in cache and states.

Weights are drawn from the seed, every tensor by its name.  The output table's row t is the embedding's row t + 1 (a tied
table is its own) and the embedding outweighs what the layers add, as far as in a trained model: the greedy choice has a
margin then, and two correct implementations choose the same tokens.
"""
import hashlib
import math
import random

import torch
import torch.nn.functional as F

import llm_infer_amd
from llm_infer_amd.engine import DecoderModel, Engine
from llm_infer_amd.sampling import Sampler
from llm_infer_amd.weights.loader import OnDemand, place_tensor

DEVICE = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
BYTES = {"fp16": 2, "bf16": 2, "fp32": 4}
EPS = 1e-5

# the shapes of this repository's benchmark: three Llama shapes, and the layer sizes at which the other designs stand beside them
LLAMA_8B = dict(width=4096, heads=32, kv_heads=8, head_dim=128, ff=14336, vocab=128256, layers=32, tied=False)
LLAMA_1B = dict(width=2048, heads=32, kv_heads=8, head_dim=64, ff=8192, vocab=128256, layers=16, tied=True)
LLAMA_7B = dict(width=4096, heads=32, kv_heads=32, head_dim=128, ff=11008, vocab=32000, layers=32, tied=False)
LARGE = dict(width=4096, heads=32, kv_heads=8, head_dim=128, ff=14336, vocab=32000, layers=4, tied=False)
SMALL = dict(width=2048, heads=16, kv_heads=4, head_dim=128, ff=8192, vocab=32000, layers=4, tied=False)
OTHERS = ("manirax", "risonex", "dupolorn", "favizen", "dopivik", "pusisun")


def case_of(name, design, shape, dtype, batch, lo, hi, new, held=False):
    return dict(shape, name=name, design=design, dtype=dtype, batch=batch, lo=lo, hi=hi, new=new, held=held)


def listed():
    return [
        # one user and a short question: latency of a short prompt and of decoding at batch 1
        case_of("llama8b chat b1", "llama", LLAMA_8B, "fp16", 1, 19, 19, 24),
        # eight conversations near the context's end go on: the benchmark's headline, weights and cache from memory
        case_of("llama8b continue b8 ctx8k", "llama", LLAMA_8B, "fp16", 8, 8160, 8160, 16, held=True),
        # a server's batch: 48 ragged prompts, then decoding with more rows than the matrix-vector kernels take
        case_of("llama8b serve b48", "llama", LLAMA_8B, "bf16", 48, 16, 512, 16),
        # the first token of one long prompt
        case_of("llama8b prompt 2048", "llama", LLAMA_8B, "fp16", 1, 2048, 2048, 0),
        # 32 ragged prompts scored in one step
        case_of("llama1b ragged 32 prompts", "llama", LLAMA_1B, "fp16", 32, 16, 2048, 0),
        # the 32-bit path: a model checked or served in full precision
        case_of("llama1b float32", "llama", LLAMA_1B, "fp32", 3, 50, 200, 8),
        # the other designs, prompt and decoding both: one long document, a few questions, a small batch, ...
        case_of("manirax document", "manirax", LARGE, "bf16", 1, 2000, 2000, 16),
        case_of("risonex questions b4", "risonex", LARGE, "bf16", 4, 300, 700, 16),
        case_of("dupolorn small b8", "dupolorn", SMALL, "fp16", 8, 100, 300, 16),
        case_of("favizen documents b2", "favizen", LARGE, "bf16", 2, 1200, 1800, 16),
        case_of("dopivik small document", "dopivik", SMALL, "fp16", 1, 777, 777, 16),
        case_of("pusisun serve b8", "pusisun", LARGE, "bf16", 8, 64, 256, 32),
    ]


def draw(rng):
    """Another request: any design, batch 1 to 64, prompts of 1 to 8,192 tokens, few or many new tokens; fewer layers than
    the whole shapes have, so that none costs more than the largest listed case."""
    def spread(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))
    design = rng.choice(("llama",) * 4 + OTHERS)
    if design == "llama":
        shape = dict(rng.choice((LLAMA_8B, LLAMA_1B, LLAMA_7B)), layers=rng.randint(3, 8))
        dtype = rng.choice(("fp16", "bf16", "fp16", "bf16", "fp32"))
    else:
        shape = dict(rng.choice((SMALL, LARGE)), layers=rng.choice((2, 4, 4, 5)))
        dtype = rng.choice(("fp16", "bf16"))
    if design == "dupolorn":
        dtype = "fp16"                       # (its experts' scores are near ties more often than bfloat16 can tell apart)
    batch = spread(1, 64)
    # 32-bit requests are short ones
    most = (512 if dtype == "fp32" else 12288) // batch
    hi = spread(1, max(1, min(8192, most)))
    lo = hi if batch == 1 else max(1, hi // rng.choice((1, 2, 8)))
    held = design == "llama" and dtype != "fp32" and hi >= 256 and rng.random() < 0.5
    new = rng.randint(4, 24) if held else rng.choice((0, rng.randint(2, 8), rng.randint(8, 32)))
    return dict(shape, design=design, dtype=dtype, batch=batch, lo=lo, hi=hi, new=new, held=held)


def prompt_lengths(case):
    r = random.Random("%d %d %d" % (case["batch"], case["lo"], case["hi"]))
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]


def prompts_of(case, seed):
    g = torch.Generator().manual_seed(seed * 7919 + 13)
    return [torch.randint(0, case["vocab"], (n,), generator=g).tolist() for n in prompt_lengths(case)]


# ---------------------------------------------------------------------------------------------------------------------
# the models
# ---------------------------------------------------------------------------------------------------------------------
def model_config(case):
    """config.json of the case's model; for the other designs what ``bench.py --compare`` puts beside the Llama decoder."""
    w, H, G, hd, ff, L = (case[k] for k in ("width", "heads", "kv_heads", "head_dim", "ff", "layers"))
    positions = case["hi"] + case["new"] + 8
    if case["design"] == "llama":
        return dict(architectures=["LlamaForCausalLM"], num_hidden_layers=L, hidden_size=w, num_attention_heads=H,
                    num_key_value_heads=G, head_dim=hd, intermediate_size=ff, vocab_size=case["vocab"], rope_theta=500000.0,
                    rms_norm_eps=EPS, max_position_embeddings=positions, tie_word_embeddings=case["tied"], hidden_act="silu")
    out = {"embedding": {"scale": 1.0}, "norm": {"eps": EPS}, "vocab": case["vocab"], "width": w, "max_positions": positions}
    dense, quarter = {"kind": "dense", "ff": ff}, {"ff": ff // 4}
    if case["design"] == "manirax":
        layer = {"type": "parallel", "mlp": dense,
                 "mixer": {"left": {"heads": H, "kv_heads": G, "dim": hd, "vdim": hd, "scale": hd ** -0.5,
                                    "rot": {"base": 500000.0, "dims": hd // 2, "scaling": {"factor": 2.0}}},
                           "right": {"heads": H // 2, "dim": hd, "vdim": hd,
                                     "decay": [1.0 - 2.0 ** -(3 + 5 * i / max(1, H // 2 - 1)) for i in range(H // 2)]},
                           "left_scale": 1.0, "right_scale": 1.0}}
        del out["embedding"]
        return dict(out, architecture="Manirax", layers=[layer] * L, postln_alpha=2.0)
    if case["design"] == "risonex":
        ssm = {"type": "mamba2", "mixer": {"heads": 2 * w // 64, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}}
        att = {"type": "attention", "mixer": {"heads": H, "kv_heads": G, "dim": hd // 2, "vdim": hd, "diff": 0.3,
                                              "scale": (hd // 2) ** -0.5, "mask": {"size": 1024}}}
        routed = {"kind": "moe", "expert": quarter, "shared": quarter,
                  "router": {"experts": 8, "identity": 0, "top": 2, "scale": 1.0}}
        return dict(out, architecture="Risonex",
                    layers=[dict(att if i % 2 else ssm, mlp=routed if i else dense) for i in range(L)])
    if case["design"] == "dupolorn":
        lat = {"heads": H, "dim": hd, "rot_dim": hd // 2, "vdim": hd, "kv_rank": 3 * hd // 2, "scale": (3 * hd // 2) ** -0.5,
               "rot": {"base": 500000.0, "dims": hd // 2}}
        mem = {"heads": max(1, H // 4), "dim": 2 * hd, "vdim": 4 * hd, "gate_cap": 15.0}
        kinds = ("latent_attention_2", "latent_attention_2", "latent_attention", "mlstm")
        routed = {"kind": "moe", "expert": quarter, "shared": quarter, "router": {"experts": 8, "top": 2}}
        out["embedding"] = {"bigram": {"buckets": 65521, "mul_prev": 31, "mul_cur": 7}, "scale": 1.0}
        return dict(out, architecture="Dupolorn", canon={"taps": 3}, logit_softcap=30.0,
                    layers=[{"type": kinds[i % 4], "mixer": mem if i % 4 == 3 else lat, "mlp": routed if i else dense} for i in range(L)])
    if case["design"] == "favizen":
        first = {"heads": H, "kv_heads": G, "dim": hd, "vdim": hd, "scale": hd ** -0.5, "mask": {"size": 1024},
                 "rot": {"base": 500000.0, "dims": hd, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}
        second = {"heads": H, "kv_heads": G, "dim": hd, "vdim": hd, "scale": hd ** -0.5, "mask": {"size": 1024}, "conv": 3}
        limit = dict(quarter, limit=7.0)
        routed = {"kind": "moe", "expert": limit, "shared": limit, "router": {"experts": 8, "top": 2}}
        stack = [{"type": "attention_2" if i % 4 > 1 else "attention", "mixer": dict(second if i % 4 > 1 else first),
                  "mlp": routed if i % 2 else dict(dense, limit=7.0)} for i in range(L)]
        for i in range(3, L, 4):
            stack[i]["mixer"]["kv_from"] = i - 1
        return dict(out, architecture="Favizen", layers=stack, logit_scale=1.0)
    if case["design"] == "dopivik":
        both = {"left": {"heads": H, "kv_heads": G, "dim": hd, "vdim": hd, "scale": hd ** -0.5, "softcap": 50.0,
                         "mask": {"size": 1024}, "rot": {"base": 500000.0, "dims": hd}},
                "right": {"heads": H, "kv_heads": H // 2, "dim": hd, "vdim": hd, "conv": 4}}
        kinds = (("parallel", both), ("mamba1", {"inner": 2 * w, "state": 16, "dt_rank": w // 16, "conv": 4}),
                 ("wkv", {"heads": w // 64, "dim": 64, "rank": w // 64}), ("parallel", both))
        return dict(out, architecture="Dopivik", layers=[{"type": kinds[i % 4][0], "mixer": kinds[i % 4][1], "mlp": dense} for i in range(L)])
    lat = {"heads": H, "dim": hd, "rot_dim": hd // 2, "vdim": hd, "kv_rank": 3 * hd // 2, "q_rank": 3 * w // 8,
           "scale": (3 * hd // 2) ** -0.5,
           "rot": {"base": 10000.0, "dims": hd // 2, "scaling": {"factor": 40.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
    att = {"heads": H, "kv_heads": G, "dim": hd, "vdim": hd, "scale": hd ** -0.5, "mask": {"size": 1024, "keep_first": 16}}
    routed = {"kind": "moe", "expert": quarter, "router": {"experts": 16, "top": 4}}
    return dict(out, architecture="Pusisun", loop={"start": 1, "stop": 2, "times": 2},
                layers=[{"type": "attention" if i % 2 else "latent_attention", "mixer": att if i % 2 else lat, "mlp": routed}
                        for i in range(max(2, L - 1))])


def generator_for(seed, name):
    digest = hashlib.sha256(("%d %s" % (seed, name)).encode()).digest()
    return torch.Generator(device=DEVICE).manual_seed(int.from_bytes(digest[:7], "little"))


def tensor_of(case, seed, name, shape):
    """The tensor of this name: drawn in the case's type, so that whoever keeps it in 32 bits keeps the same numbers."""
    dt, shape = DTYPES[case["dtype"]], tuple(shape)
    last = name[6:] if name.startswith("model.") else name
    if last in ("head", "lm_head.weight"):
        table = "embed" if name == "head" else "model.embed_tokens.weight"
        return tensor_of(case, seed, table, shape).roll(-1, 0).mul_(0.02)
    g = generator_for(seed, name)
    if last.endswith(".table"):
        order = torch.rand((shape[0], 8), generator=g, device=DEVICE).argsort(dim=-1)
        return order[:, :shape[1]].to(torch.int32).contiguous()
    r = torch.randn(shape, generator=g, device=DEVICE, dtype=dt)
    tail = last.rsplit(".", 1)[-1]
    if last in ("embed", "embed_tokens.weight"):
        return r
    if case["design"] == "llama":
        if "norm" in last:
            return 1.0 + r.mul_(0.01)
        out = "o_proj" in last or "down_proj" in last
        return r.mul_(0.02 / math.sqrt(2 * case["layers"]) if out else 0.02)
    if tail == "dwa":
        return r.mul_(0.2).add_(1.0).div_(shape[0])
    if tail == "shift" or ".mu." in last:
        return r.mul_(0.1).add_(0.5).clamp_(0.0, 1.0)
    if tail == "router":
        return r.mul_(0.02 if case["design"] == "dupolorn" else 0.1)
    if tail == "pb":
        return r.mul_(0.02).sub_(7.0)                          # (weights that are not normalised over some thousand keys)
    if tail in ("conv", "sg", "u"):
        return r.mul_(0.4)
    if case["design"] == "risonex" and (tail in ("norm1", "norm2") or last == "final.norm"):
        return r.mul_(0.02)                                    # (these act as 1 + w)
    if tail in ("norm", "norm1", "norm2", "norm1b", "norm2b", "D", "out", "act") or last.endswith("f.b"):
        return 1.0 + r.mul_(0.01)
    if case["design"] == "manirax" and (tail == "down" or last.endswith("left.o")):
        return r.mul_(0.002)                                   # (the activation has a mean, the attention sums over all keys)
    return r.mul_(0.02)


# ---------------------------------------------------------------------------------------------------------------------
# preparing and running
# ---------------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    dt = DTYPES[case["dtype"]]
    config = llm_infer_amd.config_from_dict(model_config(case))
    model = DecoderModel(config.model_spec(), dt, DEVICE)
    params = model.params()
    model.bind(OnDemand(lambda name: place_tensor(tensor_of(case, seed, name, params[name].shape), params[name].kind, dt, DEVICE)))
    room = sum(-(-(n + case["new"] + 4) // 64) * 64 for n in prompt_lengths(case))
    engine = Engine(config, model, room + 64, case["batch"])
    prompts = prompts_of(case, seed)
    state = {"engine": engine, "prompts": prompts, "new": case["new"], "slots": None}
    if case["held"]:
        state["slots"] = [engine.alloc_slot() for _ in prompts]
        state["lens"] = [len(p) - 1 for p in prompts]
        engine.step(state["slots"], [p[:-1] for p in prompts], [[] for _ in prompts])
    return state


def run(state):
    engine, held = state["engine"], state["slots"]
    slots = held or [engine.alloc_slot() for _ in state["prompts"]]
    first = engine.step(slots, [p[-1:] for p in state["prompts"]] if held else state["prompts"])
    out = {"first": first}
    if state["new"]:
        sampler = Sampler(temperature=0.0)
        sampler.start(engine.cache, slots, range(len(slots)))
        where = torch.tensor(slots, dtype=torch.int32, device=engine.device)
        tokens = [sampler.sample(first, where, engine.cache).tolist()]
        runner = engine.decode_runner(sampler)
        for i in range(state["new"]):
            tokens.append(runner.run(slots, tokens[-1], may_follow=i + 1 < state["new"]))
        out["tokens"] = torch.tensor(tokens)
        out["last"] = engine.step(slots, [[t] for t in tokens[-1]])
    if held:
        engine.cache.truncate(slots, state["lens"])
    else:
        for s in slots:
            engine.free_slot(s)
    return out


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------------
def mixers_of(layer):
    m = layer["mixer"]
    return [m["left"], m["right"]] if layer["type"] == "parallel" else [m]


def work(case):
    """Every step reads once the matrices that its tokens need (of the experts no more than are chosen), and the keys,
    values and states that its sequences have; operations are the products' and the attention's."""
    raw, e, lens = model_config(case), BYTES[case["dtype"]], prompt_lengths(case)
    B, steps = case["batch"], (case["new"] + 1 if case["new"] else 0)
    params = DecoderModel(llm_infer_amd.config_from_dict(raw).model_spec(), torch.float32, "cpu", allocate=False).params()
    tied = not any(n in ("head", "lm_head.weight") for n in params)
    layers, loop = raw.get("layers"), raw.get("loop")
    experts = next((la["mlp"]["router"] for la in layers or () if la["mlp"].get("router")), None)

    def rows_and_bytes(tokens):
        """(multiply-adds that every token has, those of a wanted row, bytes of the matrices) of a step of so many tokens."""
        body = head = read = 0.0
        for name, spec in params.items():
            n = math.prod(spec.shape)
            times = loop["times"] if loop and name.startswith("l%d." % loop["start"]) else 1
            if name in ("head", "lm_head.weight") or (tied and name in ("embed", "model.embed_tokens.weight")):
                head, read = head + n, read + n * e
            elif name in ("embed", "model.embed_tokens.weight", "bigram"):
                read += tokens * spec.shape[1] * e
            elif len(spec.shape) == 2 and spec.kind != "int" and min(spec.shape) > 4:
                if ".mlp.e" in name:
                    body += times * n * experts["top"] / experts["experts"]
                    read += times * n * e * min(1.0, tokens * experts["top"] / experts["experts"])
                else:
                    body, read = body + times * n, read + times * n * e
        return body, head, read

    def context(n):
        """(bytes of keys, values and states that a token behind n others reads, its attention's multiply-adds)"""
        if layers is None:
            kv = 2 * case["kv_heads"] * case["head_dim"]
            return case["layers"] * n * kv * e, case["layers"] * n * 2 * case["heads"] * case["head_dim"]
        read = ops = 0.0
        for i, la in enumerate(layers):
            times = loop["times"] if loop and i == loop["start"] else 1
            for m in mixers_of(la):
                seen = min(n, (m.get("mask") or {}).get("size", n))
                if "kv_rank" in m:
                    size = m["kv_rank"] + m["rot_dim"]
                    read, ops = read + times * seen * size * e, ops + times * seen * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
                elif "mask" in m or "rot" in m:
                    maps = 2 if "diff" in m else 1
                    read += times * seen * m["kv_heads"] * (maps * m["dim"] + m["vdim"]) * e
                    ops += times * seen * m["heads"] * (maps * m["dim"] + m["vdim"])
                elif "inner" in m:
                    read, ops = read + 8 * m["inner"] * m["state"], ops + 2 * m["inner"] * m["state"]
                else:
                    state = m["heads"] * m.get("state", m.get("dim")) * m.get("vdim", m.get("dim"))
                    read, ops = read + 8 * state, ops + 2 * state
        return read, ops

    nbytes = flops = 0.0
    T = 0 if case["held"] else sum(lens)
    if T:
        body, head, read = rows_and_bytes(T)
        flops += 2 * (body * T + head * B) + sum(2 * n * context(n / 2)[1] for n in lens)
        nbytes += read + sum(context(n)[0] for n in lens)              # (keys and values are written)
    for k in range(steps + (1 if case["held"] else 0)):
        body, head, read = rows_and_bytes(B)
        seen = [context(n + k) for n in lens]
        flops += 2 * (body + head) * B + 2 * sum(o for _, o in seen)
        nbytes += read + sum(b for b, _ in seen)
    return {"bytes": nbytes + 2 * B * case["vocab"] * 4, "flops": flops}


def tolerance(case):
    """About four times what the logits are off their 64-bit values: 5e-7 in 32 bits, 3e-4 to 9e-4 in float16 and 3e-3 to
    6e-3 in bfloat16 from what is rounded to 16 bits on the way (a few times that where recurrences or layer norms
    enlarge it).  No token may differ: their margins are wide."""
    rel = {"fp32": 1e-5, "fp16": 1.2e-2 if case["design"] == "dopivik" else 5e-3, "bf16": 2.5e-2}[case["dtype"]]
    return {"rel": rel, "max": min(0.9, 40 * rel), "differ": 0.0}


# ---------------------------------------------------------------------------------------------------------------------
# the same in 64 bits: whole sequences, no cache, one function for each mechanism.  Rows of all sequences lie one
# after another; ``seqs`` are the slices of the sequences.
# ---------------------------------------------------------------------------------------------------------------------
def rms(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def layer_norm(x, w, b=0.0):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + EPS) * w + b


def turn(x, freqs, adjacent=False, magnitude=1.0):
    """x [T, heads, d], positions 0 .. T - 1: pairs (i, i + half) or (2i, 2i + 1) of the first 2 len(freqs) dimensions."""
    n = freqs.numel()
    a = torch.arange(x.shape[0], device=x.device, dtype=x.dtype)[:, None, None] * freqs
    c, s = torch.cos(a) * magnitude, torch.sin(a) * magnitude
    out = x.clone()
    one, two = (slice(0, 2 * n, 2), slice(1, 2 * n, 2)) if adjacent else (slice(0, n), slice(n, 2 * n))
    u, v = x[..., one], x[..., two]
    out[..., one], out[..., two] = u * c - v * s, v * c + u * s
    return out


def frequencies(rot):
    """Frequencies of the pairs and the factor of sine and cosine, for every kind of scaling that the designs have."""
    dims, base, scaling = rot["dims"], rot["base"], rot.get("scaling")
    i = torch.arange(dims // 2, dtype=torch.float64, device=DEVICE)
    f = base ** (-2.0 * i / dims)
    if not scaling:
        return f, 1.0
    factor = scaling["factor"]
    if "low" in scaling:                     # by wavelength: long ones divided, short ones kept, those between blended
        share = (scaling["original"] * f / (2 * math.pi) - scaling["low"]) / (scaling["high"] - scaling["low"])
        share = share.clamp(0.0, 1.0)
        return f / factor * (1 - share) + f * share, 1.0
    if "fast" in scaling:                    # a ramp over the pairs, and a magnitude
        def pair(turns):
            return dims * math.log(scaling["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
        lo, hi = max(math.floor(pair(scaling["fast"])), 0), min(math.ceil(pair(scaling["slow"])), dims - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        return f / factor * ramp + f * (1 - ramp), 0.1 * math.log(factor) + 1.0
    return f / factor, 1.0


def attention(q, k, v, scale, window=None, chunk=None, first=0, sink=None, slopes=None, cap=None, sigmoid_bias=None):
    """q [T, H, d], k [T, G, d], v [T, G, dv] -> [T, H, dv]; a block of queries at a time."""
    T, H, _ = q.shape
    G = k.shape[1]
    kt = k.permute(1, 2, 0).repeat_interleave(H // G, 0).contiguous()          # [H, d, T]
    vt = v.permute(1, 0, 2).repeat_interleave(H // G, 0).contiguous()          # [H, T, dv]
    out = torch.empty((T, H, v.shape[2]), dtype=q.dtype, device=q.device)
    for lo in range(0, T, 512):
        hi = min(T, lo + 512)
        i, j = torch.arange(lo, hi, device=q.device)[:, None], torch.arange(hi, device=q.device)[None, :]
        see = j <= i
        if window is not None:
            see = see & ((i - j < window) | (j < first))
        if chunk is not None:
            see = see & (i // chunk == j // chunk)
        s = torch.bmm(q[lo:hi].transpose(0, 1).contiguous(), kt[:, :, :hi].contiguous()) * scale
        if cap is not None:
            s = cap * torch.tanh(s / cap)
        if slopes is not None:
            s = s - slopes[:, None, None] * (i - j)
        if sigmoid_bias is not None:
            p = torch.sigmoid(s + sigmoid_bias[:, None, None]).masked_fill(~see, 0.0)
        else:
            s = s.masked_fill(~see, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[:, None, None].expand(H, hi - lo, 1)], -1)
            p = torch.softmax(s, -1)[..., :hi].contiguous()
        out[lo:hi] = torch.bmm(p, vt[:, :hi].contiguous()).transpose(0, 1)
    return out


def conv(u, w):
    taps = w.shape[1]
    padded = torch.cat([torch.zeros((taps - 1, u.shape[1]), dtype=u.dtype, device=u.device), u], 0)
    return sum(padded[j:j + u.shape[0]] * w[:, j] for j in range(taps))


def before(h):
    return torch.cat([torch.zeros_like(h[:1]), h[:-1]], 0)


def slopes_of(heads):
    return torch.tensor([2.0 ** (-8.0 * (h + 1) / heads) for h in range(heads)], dtype=torch.float64, device=DEVICE)


class Plain:
    """The case's model in 64 bits; ``w(name, *shape)`` is a tensor of it."""

    def __init__(self, case, seed):
        self.case, self.seed, self.raw = case, seed, model_config(case)
        self.width, self.vocab = case["width"], case["vocab"]

    def w(self, name, *shape):
        t = tensor_of(self.case, self.seed, name, shape)
        return t.double() if t.is_floating_point() else t.long()

    def lin(self, x, name, n):
        return x @ self.w(name, n, x.shape[1]).T

    def each(self, seqs, f, *rows):
        """f over the sequences, one after another."""
        return torch.cat([f(*[r[s] for r in rows]) for s in seqs], 0)

    def logits(self, tokens, seqs, want):
        """Logits of the wanted rows of the sequences whose tokens lie one after another."""
        tokens = torch.tensor(tokens, device=DEVICE)
        return getattr(self, self.case["design"])(tokens, seqs, torch.tensor(want, device=DEVICE))

    def embed(self, tokens, name="embed"):
        return self.w(name, self.vocab, self.width)[tokens]

    # -- the Llama decoder -----------------------------------------------------------------------------------
    def llama(self, tokens, seqs, want):
        c, d = self.case, self.width
        H, G, hd = c["heads"], c["kv_heads"], c["head_dim"]
        freqs, _ = frequencies({"dims": hd, "base": 500000.0})
        x = self.embed(tokens, "model.embed_tokens.weight")
        for i in range(c["layers"]):
            p = "model.layers.%d." % i
            h = rms(x) * self.w(p + "input_layernorm.weight", d)
            q, k, v = (self.lin(h, p + "self_attn.%s_proj.weight" % n, m * hd).view(-1, m, hd) for n, m in (("q", H), ("k", G), ("v", G)))
            o = self.each(seqs, lambda q, k, v: attention(turn(q, freqs, True), turn(k, freqs, True), v, hd ** -0.5), q, k, v)
            x = x + self.lin(o.reshape(-1, H * hd), p + "self_attn.o_proj.weight", d)
            h = rms(x) * self.w(p + "post_attention_layernorm.weight", d)
            y = F.silu(self.lin(h, p + "mlp.gate_proj.weight", c["ff"])) * self.lin(h, p + "mlp.up_proj.weight", c["ff"])
            x = x + self.lin(y, p + "mlp.down_proj.weight", d)
        head = "model.embed_tokens.weight" if c["tied"] else "lm_head.weight"
        return self.lin(rms(x[want]) * self.w("model.norm.weight", d), head, self.vocab)

    # -- Manirax ---------------------------------------------------------------------------------------------
    def manirax(self, tokens, seqs, want):
        d, alpha = self.width, self.raw["postln_alpha"]
        x = self.embed(tokens)
        for i, layer in enumerate(self.raw["layers"]):
            p, a, b = "l%d." % i, layer["mixer"]["left"], layer["mixer"]["right"]
            mu = self.w(p + "shift", d)
            h = self.each(seqs, lambda r: r + (before(r) - r) * mu, x)
            H, G, hd = a["heads"], a["kv_heads"], a["dim"]
            q, k, v = (self.lin(h, p + "mix.left." + n, m * hd).view(-1, m, hd) for n, m in (("q", H), ("k", G), ("v", G)))
            f, bias = frequencies(a["rot"])[0], self.w(p + "mix.left.pb", H)
            o = self.each(seqs, lambda q, k, v: attention(rms(turn(q, f)), rms(turn(k, f)), v, a["scale"], sigmoid_bias=bias), q, k, v)
            y = self.lin(o.reshape(-1, H * hd), p + "mix.left.o", d)
            H, hd = b["heads"], b["dim"]
            q, k, v = (F.silu(self.lin(h, p + "mix.right." + n, H * hd)).view(-1, H, hd) for n in "qkv")
            decay = torch.tensor(b["decay"], dtype=torch.float64, device=DEVICE)[:, None, None]

            def walk(q, k, v):
                S, out = 0.0, []
                for t in range(q.shape[0]):
                    S = decay * S + k[t][:, :, None] * v[t][:, None, :]
                    out.append((S * q[t][:, :, None]).sum(1))
                return torch.stack(out)
            o = rms(self.each(seqs, walk, q, k, v).reshape(-1, H * hd)) * self.w(p + "mix.right.norm", H * hd)
            y = y + self.lin(o * torch.sigmoid(self.lin(h, p + "mix.right.g", H * hd)), p + "mix.right.o", d)
            x = layer_norm(alpha * x + y, self.w(p + "norm1", d))
            z, c = self.lin(x, p + "mlp.up", layer["mlp"]["ff"]), self.w(p + "mlp.act", 4)
            z = c[0] * rms(z) + c[1] * rms(z * z) + c[2] * rms(z * z * z) + c[3]
            x = layer_norm(alpha * x + self.lin(z, p + "mlp.down", d), self.w(p + "norm2", d))
        return self.lin(layer_norm(x[want], self.w("final.norm", d)), "embed", self.vocab)

    # -- experts of several designs ---------------------------------------------------------------------------
    def gated(self, h, p, ff, act, up="up"):
        return self.lin(act(self.lin(h, p + "gate", ff), self.lin(h, p + up, ff)), p + "down", self.width)

    def chosen(self, h, weights, f):
        """sum over experts e of f(rows of h, e, their weights) where weights [T, experts] is not zero."""
        out = torch.zeros_like(h)
        for e in range(weights.shape[1]):
            rows = weights[:, e].nonzero()[:, 0]
            if rows.numel():
                out[rows] += f(h[rows], e, weights[rows, e:e + 1])
        return out

    # -- Risonex ---------------------------------------------------------------------------------------------
    def risonex(self, tokens, seqs, want):
        d = self.width
        at = torch.cat([torch.arange(s.stop - s.start, device=DEVICE, dtype=torch.float64) for s in seqs])
        a = at[:, None] * 10000.0 ** (-torch.arange(0, d, 2, device=DEVICE, dtype=torch.float64) / d)
        x = self.embed(tokens)
        x[:, 0::2] += torch.sin(a)
        x[:, 1::2] += torch.cos(a)
        for i, layer in enumerate(self.raw["layers"]):
            p, m, mlp = "l%d." % i, layer["mixer"], layer["mlp"]
            h = rms(x) * (1 + self.w(p + "norm1", d))
            x = x + (self.diff_attention if layer["type"] == "attention" else self.mamba2)(h, p + "mix.", m, seqs)
            h = rms(x) * (1 + self.w(p + "norm2", d))
            if mlp["kind"] == "dense":
                x = x + self.lin(F.gelu(self.lin(h, p + "mlp.up", mlp["ff"])), p + "mlp.down", d)
                continue
            r, ff, p = mlp["router"], mlp["expert"]["ff"], p + "mlp."
            s = torch.softmax(self.lin(h, p + "router", r["experts"]), -1)
            best = torch.topk(s + self.w(p + "correction", r["experts"]), r["top"], dim=-1).indices
            wt = torch.gather(s, 1, best)
            wt = torch.zeros_like(s).scatter(1, best, wt / (wt.sum(-1, keepdim=True) + 1e-20) * r["scale"])
            glu = lambda g, u: F.silu(g) * u  # noqa: E731
            x = x + self.chosen(h, wt, lambda rows, e, we: we * self.gated(rows, p + "e%d." % e, ff, glu)) \
                + torch.sigmoid(self.lin(h, p + "shared.sg", 1)) * self.gated(h, p + "shared.", mlp["shared"]["ff"], glu)
        return self.lin(rms(x[want]) * (1 + self.w("final.norm", d)), "head", self.vocab)

    def diff_attention(self, h, p, m, seqs):
        H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q = rms(self.lin(h, p + "q", H * 2 * d).view(-1, H, 2, d)) * self.w(p + "q.norm", d)
        k = rms(self.lin(h, p + "k", G * 2 * d).view(-1, G, 2, d)) * self.w(p + "k.norm", d)
        v = self.lin(h, p + "v", G * dv).view(-1, G, dv)
        l1, l2 = ((self.w(p + "lq%d" % n, d) * self.w(p + "lk%d" % n, d)).sum().exp() for n in (1, 2))

        def both(q, k, v):
            one, two = (attention(q[:, :, n], k[:, :, n], v, m["scale"], chunk=m["mask"]["size"]) for n in (0, 1))
            return rms(one - (l1 - l2 + m["diff"]) * two) * (1 - m["diff"])
        return self.lin(self.each(seqs, both, q, k, v).reshape(-1, H * dv), p + "o", self.width)

    def mamba2(self, h, p, m, seqs):
        P, dv, N = m["heads"], m["vdim"], m["state"]
        inner = P * dv
        proj = self.lin(h, p + "in", 2 * inner + 2 * N + P)
        z, xbc, dt = proj[:, :inner], proj[:, inner:2 * inner + 2 * N], proj[:, 2 * inner + 2 * N:]
        taps, bias = self.w(p + "conv", inner + 2 * N, m["conv"]), self.w(p + "conv.b", inner + 2 * N)
        xbc = F.silu(self.each(seqs, lambda u: conv(u, taps), xbc) + bias)
        dt = F.softplus(dt + self.w(p + "dt_bias", P))
        decay = torch.exp(-torch.exp(self.w(p + "A_log", P)) * dt)
        D = self.w(p + "D", P)[:, None]

        def walk(x, B, C, dt, decay):
            S, out = 0.0, []
            for t in range(x.shape[0]):
                S = decay[t][:, None, None] * S + (dt[t][:, None] * x[t])[:, None, :] * B[t][None, :, None]
                out.append((S * C[t][None, :, None]).sum(1) + D * x[t])
            return torch.stack(out)
        y = self.each(seqs, walk, xbc[:, :inner].reshape(-1, P, dv), xbc[:, inner:inner + N], xbc[:, inner + N:], dt, decay)
        y = rms(y.reshape(-1, inner) * F.silu(z)) * self.w(p + "norm", inner)
        return self.lin(y, p + "o", self.width)

    # -- Dupolorn --------------------------------------------------------------------------------------------
    def dupolorn(self, tokens, seqs, want):
        d, big = self.width, self.raw["embedding"]["bigram"]
        n = big["buckets"]
        rows = torch.cat([torch.cat([torch.tensor([n], device=DEVICE),
                                     (tokens[s][:-1] * big["mul_prev"] + tokens[s][1:] * big["mul_cur"]) % n]) for s in seqs])
        x = self.embed(tokens) + self.w("bigram", n + 1, d)[rows]
        history = [x]
        for i, layer in enumerate(self.raw["layers"]):
            p, m, mlp = "l%d." % i, layer["mixer"], layer["mlp"]
            h, taps = rms(x) * self.w(p + "norm1"), self.w(p + "canon1", d, self.raw["canon"]["taps"])
            h = h + self.each(seqs, lambda u: conv(u, taps), h)
            y = x + (self.mlstm(h, p + "mix.", m, seqs) if layer["type"] == "mlstm" else
                     self.latent(h, p + "mix.", m, seqs, adjacent=True, gated=layer["type"] == "latent_attention_2"))
            h, p = rms(x) * self.w(p + "norm2"), p + "mlp."
            if mlp["kind"] == "dense":
                y = y + self.gated(h, p, mlp["ff"], lambda g, u: F.gelu(g, approximate="tanh") * u)
            else:
                def two(rows, q, ff):
                    return self.lin(torch.relu(self.lin(rows, q + "up", ff)) ** 2, q + "down", d)
                s = torch.sigmoid(self.lin(h, p + "router", mlp["router"]["experts"]))
                best = torch.topk(s, mlp["router"]["top"], dim=-1)
                wt = torch.zeros_like(s).scatter(1, best.indices, best.values)
                y = y + self.chosen(h, wt, lambda rows, e, we: two(rows * we, p + "e%d." % e, mlp["expert"]["ff"])) \
                    + two(h, p + "shared.", mlp["shared"]["ff"])
            history.append(y)
            mean = self.w("l%d.dwa" % i, i + 2)
            x = sum(mean[j] * history[j] for j in range(i + 2))
        cap = self.raw["logit_softcap"]
        return cap * torch.tanh(self.lin(rms(x[want]) * self.w("final.norm"), "head", self.vocab) / cap)

    def latent(self, h, p, m, seqs, adjacent, gated=False):
        H, d, rd, dv, r = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        q, name = h, "q"
        if "q_rank" in m:
            q, name = rms(self.lin(h, p + "dq", m["q_rank"])) * self.w(p + "dq.norm", m["q_rank"]), "uq"
        q = self.lin(q, p + name, H * (d + rd)).view(-1, H, d + rd)
        kv = self.lin(h, p + "dkv", r + rd)
        c = rms(kv[:, :r]) * self.w(p + "dkv.norm", r)
        k, v = self.lin(c, p + "uk", H * d).view(-1, H, d), self.lin(c, p + "uv", H * dv).view(-1, H, dv)
        f, size = frequencies(m["rot"])
        sink = self.w(p + "sink", H) if gated else None

        def one(q, k, v, k_rot):
            q = torch.cat([q[..., :d], turn(q[..., d:], f, adjacent, size)], -1)
            k = torch.cat([k, turn(k_rot[:, None], f, adjacent, size).expand(-1, H, -1)], -1)
            return attention(q, k, v, m["scale"], sink=sink)
        o = self.each(seqs, one, q, k, v, kv[:, r:]).reshape(-1, H * dv)
        if gated:
            o = o * torch.sigmoid(self.lin(h, p + "g", H * dv))
        return self.lin(o, p + "o", self.width)

    def mlstm(self, h, p, m, seqs):
        H, d, dv, cap = m["heads"], m["dim"], m["vdim"], m["gate_cap"]
        q, k = self.lin(h, p + "q", H * d).view(-1, H, d) * d ** -0.5, self.lin(h, p + "k", H * d).view(-1, H, d)
        v = self.lin(h, p + "v", H * dv).view(-1, H, dv)
        ig = cap * torch.tanh((self.lin(h, p + "i", H) + self.w(p + "i.b", H)) / cap)
        fg = F.logsigmoid(cap * torch.tanh((self.lin(h, p + "f", H) + self.w(p + "f.b", H)) / cap))

        def walk(q, k, v, ig, fg):
            S, n, mx, out = 0.0, 0.0, torch.zeros(H, dtype=torch.float64, device=DEVICE), []
            for t in range(q.shape[0]):
                new = torch.maximum(fg[t] + mx, ig[t])
                a, b = torch.exp(fg[t] + mx - new)[:, None], torch.exp(ig[t] - new)[:, None]
                S = a[:, :, None] * S + (b * k[t])[:, :, None] * v[t][:, None, :]
                n, mx = a * n + b * k[t], new
                den = torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-mx)) + 1e-6
                out.append((S * q[t][:, :, None]).sum(1) / den[:, None])
            return torch.stack(out)
        y = rms(self.each(seqs, walk, q, k, v, ig, fg)).reshape(-1, H * dv) * self.w(p + "norm", H * dv)
        return self.lin(y * torch.sigmoid(self.lin(h, p + "g", H * dv)), p + "o", self.width)

    # -- Favizen ---------------------------------------------------------------------------------------------
    def favizen(self, tokens, seqs, want):
        d, x, kept = self.width, self.embed(tokens), {}
        for i, layer in enumerate(self.raw["layers"]):
            p, m, mlp = "l%d." % i, layer["mixer"], layer["mlp"]
            h, q = rms(x) * self.w(p + "norm1", d), p + "mix."
            H, G, hd = m["heads"], m["kv_heads"], m["dim"]
            sink = self.w(q + "sink", H)
            if layer["type"] == "attention":
                f = frequencies(m["rot"])[0]
                o = self.each(seqs, lambda a, b: attention(turn(a, f), turn(b, f), b, m["scale"], window=m["mask"]["size"], sink=sink),
                              self.lin(h, q + "q", H * hd).view(-1, H, hd), self.lin(h, q + "k", G * hd).view(-1, G, hd))
            else:
                def rows(n, heads):
                    u, taps = self.lin(h, q + n, heads * hd) + self.w(q + n + ".b", heads * hd), self.w(q + n + ".conv", heads * hd, m["conv"])
                    return self.each(seqs, lambda r: conv(r, taps), u).view(-1, heads, hd)
                kept[i] = kept[m["kv_from"]] if m.get("kv_from") is not None else (rows("k", G), rows("v", G))
                o = self.each(seqs, lambda a, b, c: attention(a, b, c, m["scale"], chunk=m["mask"]["size"], sink=sink, slopes=slopes_of(H)),
                              rows("q", H), *kept[i])
            o = o * torch.sigmoid(self.lin(h, q + "g", H))[:, :, None]
            x = x + rms(self.lin(o.reshape(-1, H * hd), q + "o", d)) * self.w(p + "norm1b", d)
            h, q = rms(x) * self.w(p + "norm2", d), p + "mlp."

            def glu(g, u):
                g = g.clamp(max=7.0)
                return g * torch.sigmoid(1.702 * g) * (u.clamp(-7.0, 7.0) + 1)
            if mlp["kind"] == "dense":
                ff = mlp["ff"]
                y = glu(self.lin(h, q + "gate", ff) + self.w(q + "gate.b", ff), self.lin(h, q + "up", ff) + self.w(q + "up.b", ff))
                y = self.lin(y, q + "down", d) + self.w(q + "down.b", d)
            else:
                ff, r = mlp["expert"]["ff"], mlp["router"]
                wt = torch.zeros((h.shape[0], r["experts"]), dtype=h.dtype, device=DEVICE)
                wt.scatter_(1, self.w(q + "table", self.vocab, r["top"])[tokens], 1.0 / r["top"])
                y = self.chosen(h, wt, lambda rows, e, we: we * self.gated(rows, q + "e%d." % e, ff, glu)) \
                    + torch.sigmoid(self.lin(h, q + "shared.sg", 1)) * self.gated(h, q + "shared.", mlp["shared"]["ff"], glu)
            x = x + rms(y) * self.w(p + "norm2b", d)
        return self.lin(rms(x[want]) * self.w("final.norm", d), "head", self.vocab) * self.raw["logit_scale"]

    # -- Dopivik ---------------------------------------------------------------------------------------------
    def dopivik(self, tokens, seqs, want):
        d, x = self.width, self.embed(tokens)

        def norm(v, name):
            return layer_norm(v, self.w(name, d), self.w(name + ".b", d))
        for i, layer in enumerate(self.raw["layers"]):
            p, m = "l%d." % i, layer["mixer"]
            h, q = norm(x, p + "norm1"), p + "mix."
            if layer["type"] == "parallel":
                y = 0.5 * (rms(self.chunks(h, q + "left.", m["left"], seqs)) * self.w(q + "left.out", d)
                           + rms(self.delta(h, q + "right.", m["right"], seqs)) * self.w(q + "right.out", d))
            else:
                y = (self.mamba1 if layer["type"] == "mamba1" else self.wkv)(h, q, m, seqs)
            x = x + norm(y, p + "norm1b")
            z = torch.relu(self.lin(norm(x, p + "norm2"), p + "mlp.up", layer["mlp"]["ff"])) ** 2
            x = x + norm(self.lin(z, p + "mlp.down", d), p + "norm2b")
        return self.lin(norm(x[want], "final.norm"), "head", self.vocab)

    def chunks(self, h, p, m, seqs):
        H, G, d = m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (self.lin(h, p + n, g * d).view(-1, g, d) for n, g in (("q", H), ("k", G), ("v", G)))
        f = frequencies(m["rot"])[0]
        o = self.each(seqs, lambda a, b, c: attention(turn(a, f), turn(b, f), c, m["scale"], chunk=m["mask"]["size"], cap=m["softcap"]), q, k, v)
        return self.lin(o.reshape(-1, H * d) * torch.sigmoid(self.lin(h, p + "g", H * d)), p + "o", self.width)

    def delta(self, h, p, m, seqs):
        H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]

        def rows(n, size):
            taps = self.w(p + n + ".conv", size, m["conv"])
            return F.silu(self.each(seqs, lambda u: conv(u, taps), self.lin(h, p + n, size)))
        q, k = (rows(n, G * d).view(-1, G, d) for n in "qk")
        q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        q, k = (t.repeat_interleave(H // G, 1) for t in (q * d ** -0.5, k))
        beta = torch.sigmoid(self.lin(h, p + "b", H))[:, :, None]
        g = torch.exp(-torch.exp(self.w(p + "A_log", H)) * F.softplus(self.lin(h, p + "a", H) + self.w(p + "dt_bias", H)))

        def walk(q, k, v, beta, g):
            S, out = torch.zeros((H, d, dv), dtype=torch.float64, device=DEVICE), []
            for t in range(q.shape[0]):
                S = g[t][:, None, None] * S
                u = beta[t] * (v[t] - (S * k[t][:, :, None]).sum(1))
                S = S + k[t][:, :, None] * u[:, None, :]
                out.append((S * q[t][:, :, None]).sum(1))
            return torch.stack(out)
        o = self.each(seqs, walk, q, k, rows("v", H * dv).view(-1, H, dv), beta, g)
        o = (rms(o) * self.w(p + "norm", dv)).reshape(-1, H * dv) * F.silu(self.lin(h, p + "g", H * dv))
        return self.lin(o, p + "o", self.width)

    def mamba1(self, h, p, m, seqs):
        inner, n, r = m["inner"], m["state"], m["dt_rank"]
        xz, taps = self.lin(h, p + "in", 2 * inner), self.w(p + "conv", inner, m["conv"])
        x = F.silu(self.each(seqs, lambda u: conv(u, taps), xz[:, :inner]) + self.w(p + "conv.b", inner))
        dbc = self.lin(x, p + "x", r + 2 * n)
        dt = F.softplus(self.lin(dbc[:, :r], p + "dt", inner) + self.w(p + "dt.b", inner))
        A, D = -torch.exp(self.w(p + "A_log", inner, n)), self.w(p + "D", inner)

        def walk(x, dt, B, C):
            S, out = 0.0, []
            for t in range(x.shape[0]):
                S = torch.exp(dt[t][:, None] * A) * S + (dt[t] * x[t])[:, None] * B[t]
                out.append((S * C[t]).sum(1) + D * x[t])
            return torch.stack(out)
        y = self.each(seqs, walk, x, dt, dbc[:, r:r + n], dbc[:, r + n:])
        return self.lin(y * F.silu(xz[:, inner:]), p + "o", self.width)

    def wkv(self, h, p, m, seqs):
        H, d = m["heads"], m["dim"]
        was = self.each(seqs, before, h)
        mix = {s: h + (was - h) * self.w(p + "mu." + s, self.width) for s in "rkvgw"}
        r, k, v = (self.lin(mix[s], p + s, H * d).view(-1, H, d) for s in "rkv")
        w = self.lin(torch.tanh(self.lin(mix["w"], p + "w1", m["rank"])), p + "w2", H * d) + self.w(p + "w0", H * d)
        w, u = torch.exp(-torch.exp(w)).view(-1, H, d), self.w(p + "u", H, d)[:, :, None]

        def walk(r, k, v, w):
            S, out = 0.0, []
            for t in range(r.shape[0]):
                kv = k[t][:, :, None] * v[t][:, None, :]
                out.append(((S + u * kv) * r[t][:, :, None]).sum(1))
                S = w[t][:, :, None] * S + kv
            return torch.stack(out)
        o = rms(self.each(seqs, walk, r, k, v, w)).reshape(-1, H * d) * self.w(p + "norm", H * d)
        return self.lin(o * F.silu(self.lin(mix["g"], p + "g", H * d)), p + "o", self.width)

    # -- Pusisun ---------------------------------------------------------------------------------------------
    def pusisun(self, tokens, seqs, want):
        d, loop, n = self.width, self.raw["loop"], len(self.raw["layers"])
        x0 = x = self.embed(tokens)
        a, b, times = loop["start"], loop["stop"], loop["times"]
        steps = self.w("loop.step", times, d)
        runs = [(i, None) for i in range(a)] + [(i, t) for t in range(times) for i in range(a, b)] + [(i, None) for i in range(b, n)]
        for i, t in runs:
            if t is not None and i == a:
                x = (x + x0 if t else x) + steps[t]
            layer, p = self.raw["layers"][i], "l%d." % i
            m, mlp = layer["mixer"], layer["mlp"]
            h = rms(x) * self.w(p + "norm1", d)
            y = self.biased(h, p + "mix.", m, seqs) if layer["type"] == "attention" else self.latent(h, p + "mix.", m, seqs, adjacent=False)
            x = x + rms(y) * self.w(p + "norm1b", d)
            h, q = rms(x) * self.w(p + "norm2", d), p + "mlp."
            z = self.lin(h, q + "router", mlp["router"]["experts"]) + self.w(q + "router.b", mlp["router"]["experts"])
            best = torch.topk(z, mlp["router"]["top"], dim=-1)
            wt = torch.zeros_like(z).scatter(1, best.indices, torch.softmax(best.values, -1))
            y = self.chosen(h, wt, lambda rows, e, we: we * self.gated(rows, q + "e%d." % e, mlp["expert"]["ff"], lambda g, u: F.silu(g) * u))
            x = x + rms(y) * self.w(p + "norm2b", d)
        return self.lin(rms(x[want]) * self.w("final.norm", d), "head", self.vocab)

    def biased(self, h, p, m, seqs):
        H, G, d = m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (self.lin(h, p + n, g * d) + self.w(p + n + ".b", g * d) for n, g in (("q", H), ("k", G), ("v", G)))
        q, k = rms(q) * self.w(p + "q.norm", H * d), rms(k) * self.w(p + "k.norm", G * d)
        sink = self.w(p + "sink", H)
        o = self.each(seqs, lambda a, b, c: attention(a, b, c, m["scale"], window=m["mask"]["size"], first=m["mask"]["keep_first"],
                                                      sink=sink, slopes=slopes_of(H)),
                      q.view(-1, H, d), k.view(-1, G, d), v.view(-1, G, d))
        return self.lin(o.reshape(-1, H * d), p + "o", self.width)


def exact(case, seed):
    lens, new = prompt_lengths(case), case["new"]
    rows = sum(lens) + (new + 1) * case["batch"]
    # about 50 TFLOP/s in 64 bits
    if 2 * rows * case["layers"] * case["width"] * 3 * (case["ff"] + case["width"]) > 6e14:
        return None
    # the choice that the tables make certain: the token's own row where they are one, else the row before; checked below
    step = 0 if case["design"] == "manirax" or case["tied"] else 1
    tokens, seqs, want = [], [], []
    for p in prompts_of(case, seed):
        start = len(tokens)
        tokens += p + ([(p[-1] - step * (i + 1)) % case["vocab"] for i in range(new + 1)] if new else [])
        seqs.append(slice(start, len(tokens)))
        want.append(list(range(start + len(p) - 1, len(tokens))))
    with torch.no_grad():
        got = Plain(case, seed).logits(tokens, seqs, [r for w in want for r in w]).view(len(seqs), -1, case["vocab"])
    out = {"first": got[:, 0].contiguous()}
    if new:
        picked = got[:, :-1].argmax(-1)
        fed = torch.tensor([[tokens[r + 1] for r in w[:-1]] for w in want], device=DEVICE)
        if not torch.equal(picked, fed):
            raise ValueError("a greedy choice has no margin: %d of %d tokens" % (int((picked != fed).sum()), fed.numel()))
        out["tokens"], out["last"] = picked.T.contiguous().cpu(), got[:, -1].contiguous()
    return out
