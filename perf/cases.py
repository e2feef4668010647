"""The work that this engine's users have it do, as cases that can be timed and compared with 64-bit arithmetic.

A case names a model (the sizes of this repository's benchmark, random weights from a seed) and one of three kinds of work:

* `decode`: requests whose contexts lie in the cache get their next tokens, one step a token (`ModelRunner.step`).  The
  tokens are given (the way a continuation is scored), so that rounding cannot send two implementations different ways.
  A pass works on forks of the requests (`CacheManager.share_pages`, as several answers to a prompt do) and frees them.
* `chat`: requests from their prompts to their last token: one step for the prompts (portions of 2,048 tokens where there
  are more), then one step a token, then the requests go.  Logits of every step come back.
* `serve`: the same through `Engine.add_request` and `Engine.step`: scheduling, chunked prompts beside decoding requests,
  sampling, log-probabilities of the answers' tokens (the answers are forced by allow lists).

Models with routed experts get a router that reads eight lanes which the embedding writes and no layer changes, so that every
token picks its two experts by a wide margin and evenly: rounding does not move tokens between experts.
"""
import math

import torch

from fllm_amd import Engine, ModelRunner, SamplingParams, StepEntry
from fllm_amd.registry import model_spec_from_config
from fllm_amd.weights.random_init import random_tensors

PORTION = 2048          # prompt tokens a step
PAGE = 16
EXPERTS, TOP = 8, 2

# ---- models: the sizes that bench.py names ------------------------------------------------------------------------------
_LLAMA_8B = {
    "model_type": "llama", "architectures": ["LlamaForCausalLM"],
    "num_hidden_layers": 32, "hidden_size": 4096, "num_attention_heads": 32, "num_key_value_heads": 8, "head_dim": 128,
    "intermediate_size": 14336, "vocab_size": 128256, "rope_theta": 500000.0, "rms_norm_eps": 1e-5,
    "rope_scaling": {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                     "original_max_position_embeddings": 8192},
    "tie_word_embeddings": False, "max_position_embeddings": 131072, "hidden_act": "silu",
}
_LLAMA_1B = dict(_LLAMA_8B, num_hidden_layers=16, hidden_size=2048, head_dim=64, intermediate_size=8192, tie_word_embeddings=True,
                 rope_scaling=dict(_LLAMA_8B["rope_scaling"], factor=32.0))
# the other designs at the small and the 1.5B-class sizes; layers are fewer than a whole model's (a layer kind each, twice or more)
_SIZES = {"small": dict(width=1024, heads=8, kv_heads=2, dim=128, ff=4096, layers=8, vocab=32768),
          "1.5b": dict(width=1536, heads=12, kv_heads=2, dim=128, ff=8960, layers=8, vocab=151936)}
_CHUNK = 8192
_YARN = {"factor": 8.0, "original": 8192, "fast": 32.0, "slow": 1.0}
_BANDS = {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}


def _looped(cfg, layers):
    return dict(cfg, loop={"start": layers // 4, "stop": layers // 4 + layers // 2, "times": 2})


def _menitar(s):
    mixer = {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": s["dim"], "vdim": s["dim"], "scale": s["dim"] ** -0.5,
             "rot": {"dims": s["dim"] // 2, "base": 10000.0}, "mask": {"size": _CHUNK}}
    layer = {"type": "attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": s["ff"], "limit": 7.0}}
    return _looped({"architecture": "Menitar", "width": s["width"], "vocab": s["vocab"], "embedding": {"scale": 1.0}, "logit_scale": 1.0,
                    "norm": {"eps": 1e-5}, "layers": [layer] * s["layers"], "max_position": 32768}, s["layers"])


def _purivik(s):
    mixer = {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": s["dim"], "vdim": s["dim"], "scale": s["dim"] ** -0.5,
             "mask": {"size": _CHUNK}, "rot": {"dims": s["dim"] // 2, "base": 500000.0, "scaling": _BANDS}}
    dense = {"kind": "dense", "ff": s["ff"], "limit": 7.0}
    routed = {"kind": "moe", "expert": {"ff": s["ff"] // TOP}, "router": {"experts": EXPERTS, "top": TOP}}
    return _looped({"architecture": "Purivik", "width": s["width"], "vocab": s["vocab"], "embedding": {"scale": 1.0},
                    "residual_mult": 0.7, "norm": {"eps": 1e-5}, "max_position": 32768,
                    "layers": [{"type": "attention", "mixer": mixer, "mlp": routed if i % 2 else dense} for i in range(s["layers"])]},
                   s["layers"])


def _venadra(s):
    h, d = s["heads"], s["dim"]
    linear = {"heads": h, "dim": d, "vdim": d, "decay": [1.0 - 2.0 ** -(3 + 5 * i / max(1, h - 1)) for i in range(h)]}
    softmax = {"heads": h, "kv_heads": s["kv_heads"], "dim": d, "vdim": d, "scale": d ** -0.5, "mask": {"size": _CHUNK}}
    dense = {"kind": "dense", "ff": s["ff"]}
    routed = {"kind": "moe", "expert": {"ff": s["ff"] // TOP, "limit": 7.0}, "router": {"experts": EXPERTS, "top": TOP, "scale": 1.0}}
    return {"architecture": "Venadra", "width": s["width"], "vocab": s["vocab"], "embedding": {"scale": 1.0}, "norm": {"eps": 1e-5},
            "canon": {"taps": 4}, "max_position": 32768,
            "layers": [{"type": "attention" if i % 4 == 3 else "lightning", "mixer": softmax if i % 4 == 3 else linear,
                        "mlp": routed if i % 2 else dense} for i in range(s["layers"])]}


def _dumizen(s):
    h, d, ff = s["heads"], s["dim"], s["ff"]
    base = {"heads": h, "kv_heads": s["kv_heads"], "dim": d, "vdim": d, "scale": d ** -0.5}
    sigmoid = dict(base, softcap=30.0, q_temp={"coef": 0.25, "every": 1024})
    windowed = dict(base, mask={"size": 1024, "pool": 64}, rot={"dims": d // 2, "base": 500000.0, "scaling": _YARN})
    both = {"left": dict(base, rot={"dims": d, "base": 1000000.0, "scaling": _YARN}), "left_scale": 0.7, "right_scale": 1.2,
            "right": {"heads": h, "dim": d, "vdim": d, "rot": {"dims": d, "base": 1000000.0},
                      "decay": [1.0 - 2.0 ** -(5 + 5 * i / max(1, h - 1)) for i in range(h)]}}
    mlp = {"kind": "moe", "expert": {"ff": ff // TOP}, "shared": {"ff": ff // TOP},
           "router": {"experts": EXPERTS, "top": TOP, "scale": 2.5, "groups": {"count": 4, "keep": 2}}}
    kinds = [("attention_2", sigmoid), ("attention", windowed), ("attention", windowed), ("parallel", both)]
    return _looped({"architecture": "Dumizen", "width": s["width"], "vocab": s["vocab"], "norm": {"eps": 1e-6}, "max_position": 32768,
                    "layers": [{"type": kinds[i % 4][0], "mixer": kinds[i % 4][1], "mlp": mlp} for i in range(s["layers"])]},
                   s["layers"])


def _zoguzen(s):
    h, d, ff = s["heads"], s["dim"], s["ff"]
    base = {"heads": h, "kv_heads": s["kv_heads"], "dim": d, "vdim": d, "scale": d ** -0.5, "conv": 4}
    chunked = dict(base, softcap=50.0, mask={"size": _CHUNK})
    both = {"left": dict(base, mask={"size": 1024, "keep_first": 64}, rot={"dims": d, "base": 500000.0, "scaling": _BANDS}),
            "right": {"heads": h, "dim": d, "vdim": d, "tau": 16.0}}
    mlp = {"kind": "moe", "expert": {"ff": ff // TOP}, "router": {"experts": EXPERTS, "top": TOP}}
    kinds = [lambda i: ("attention", chunked), lambda i: ("attention", dict(chunked, kv_from=i - 1)),
             lambda i: ("mingru", {"width": h * d}), lambda i: ("parallel", both)]
    made = [kinds[i % 4](i) for i in range(s["layers"])]
    return {"architecture": "Zoguzen", "width": s["width"], "vocab": s["vocab"], "norm": {"eps": 1e-6}, "max_position": 32768,
            "logit_softcap": 30.0, "token_side": {"dim": 128}, "layers": [{"type": t, "mixer": m, "mlp": mlp} for t, m in made]}


def _dovudra(s):
    h, d = s["heads"], s["dim"]
    rot = {"dims": d // 4, "base": 500000.0, "scaling": _YARN}
    latent = {"heads": h, "dim": d - d // 4, "rot_dim": d // 4, "vdim": d, "kv_rank": 4 * d, "scale": d ** -0.5, "mask": {"size": 1024},
              "rot": rot}
    biased = {"heads": h, "kv_heads": s["kv_heads"], "dim": d, "vdim": d, "scale": d ** -0.5, "mask": {"size": 1024}, "bias_max": 512,
              "v_mix": True}
    return {"architecture": "Dovudra", "width": s["width"], "vocab": s["vocab"], "norm": {"eps": 1e-6}, "residual_mult": 0.5,
            "max_position": 32768,
            "layers": [{"type": "attention" if i % 4 == 3 else "latent_attention", "mixer": biased if i % 4 == 3 else latent,
                        "mlp": {"kind": "dense", "ff": s["ff"] * 3 // 2 // 512 * 512}} for i in range(s["layers"])]}


_DESIGNS = {"menitar": _menitar, "purivik": _purivik, "venadra": _venadra, "dumizen": _dumizen, "zoguzen": _zoguzen, "dovudra": _dovudra}


def _config(case):
    """config.json's dictionary of a case's model."""
    if case["model"] == "llama":
        return _LLAMA_8B if case["size"] == "8b" else _LLAMA_1B
    return _DESIGNS[case["model"]](_SIZES[case["size"]])


def _vocab(cfg):
    return cfg.get("vocab_size", cfg.get("vocab"))


# ---- the cases ------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # one user's answer, a token at a time, on the small model: launches and latency
        dict(name="llama-1b-decode-1", kind="decode", model="llama", size="1b", batch=1, least=256, most=256, new=2),
        # eight conversations of about a thousand tokens: the benchmark's headline step
        dict(name="llama-8b-decode-8", kind="decode", model="llama", size="8b", batch=8, least=1024, most=1024, new=4),
        # a busier server: 40 conversations of uneven lengths in one step
        dict(name="llama-8b-decode-40", kind="decode", model="llama", size="8b", batch=40, least=48, most=800, new=4),
        # questions about long documents
        dict(name="llama-8b-decode-long", kind="decode", model="llama", size="8b", batch=4, least=7008, most=8000, new=4),
        # a long prompt in portions, the last one ragged
        dict(name="llama-8b-prompt", kind="chat", model="llama", size="8b", batch=1, least=4501, most=4501, new=1),
        # several users at once through the engine: prompts of uneven lengths beside answers
        dict(name="llama-1b-serve", kind="serve", model="llama", size="1b", batch=16, least=33, most=701, new=12),
        # the other designs, each from prompts to answers
        dict(name="menitar-chat", kind="chat", model="menitar", size="1.5b", batch=1, least=1900, most=1900, new=9),
        dict(name="purivik-chat", kind="chat", model="purivik", size="1.5b", batch=8, least=100, most=380, new=9),
        dict(name="venadra-chat", kind="chat", model="venadra", size="1.5b", batch=4, least=301, most=701, new=9),
        dict(name="dumizen-chat", kind="chat", model="dumizen", size="1.5b", batch=2, least=700, most=1300, new=9),
        dict(name="zoguzen-chat", kind="chat", model="zoguzen", size="1.5b", batch=12, least=30, most=250, new=9),
        dict(name="dovudra-chat", kind="chat", model="dovudra", size="1.5b", batch=3, least=257, most=900, new=9),
    ]


def _spread(rng, low, high):
    """A whole number between low and high, evenly over its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "chat", "chat", "chat", "serve"])
    if kind == "decode":
        size = rng.choice(["1b", "8b"])
        batch = _spread(rng, 1, 64)
        most = _spread(rng, 16, min(8000, 32000 // batch))
        return dict(kind=kind, model="llama", size=size, batch=batch, least=max(1, most // rng.randint(1, 4)), most=most, new=rng.randint(2, 5))
    if kind == "serve":
        most = _spread(rng, 20, 900)
        return dict(kind=kind, model="llama", size="1b", batch=_spread(rng, 2, 24), least=max(1, most // rng.randint(1, 10)), most=most,
                    new=rng.randint(3, 16))
    model = rng.choice(["llama", "llama"] + sorted(_DESIGNS))
    batch = _spread(rng, 1, 12)
    if model == "llama":
        most = _spread(rng, 9, 4400 // batch)
        return dict(kind=kind, model=model, size=rng.choice(["1b", "8b"]), batch=batch, least=max(1, most // rng.randint(1, 5)), most=most,
                    new=rng.randint(1, 4))
    most = _spread(rng, 9, PORTION // batch)
    return dict(kind=kind, model=model, size=rng.choice(["small", "1.5b"]), batch=batch, least=max(1, most // rng.randint(1, 5)), most=most,
                new=rng.randint(1, 12))


def _lengths(case):
    """Tokens of each request before its answer: from `least` to `most`, in no order; whole pages where they are forked."""
    b, lo, hi = case["batch"], case["least"], case["most"]
    out = [lo + (hi - lo) * ((i * 7919 + 3) % b) // max(1, b - 1) for i in range(b)]
    return [max(PAGE, n // PAGE * PAGE) for n in out] if case["kind"] == "decode" else out


def _inputs(case, seed):
    """(prompt or context, answer) of every request, as lists of token ids."""
    vocab = _vocab(_config(case))
    g = torch.Generator().manual_seed(seed * 1000003 + 17)
    lengths = _lengths(case)
    draws = torch.randint(0, vocab, (sum(lengths) + case["batch"] * case["new"],), generator=g).tolist()
    prompts, answers, at = [], [], 0
    for n in lengths:
        prompts.append(draws[at:at + n])
        answer = draws[at + n:at + n + case["new"]]
        if case["kind"] == "serve":            # an allow list of one token a request
            answer = [answer[0]] * case["new"]
        answers.append(answer)
        at += n + case["new"]
    return prompts, answers


# ---- weights --------------------------------------------------------------------------------------------------------------
def _tensors(case, seed):
    """The random model of this seed by checkpoint name, on the GPU."""
    cfg = _config(case)
    _, spec = model_spec_from_config(cfg)
    w = random_tensors(spec, seed, torch.bfloat16, device="cuda:0")
    if case["model"] == "llama" and case["kind"] != "serve":
        # as trained weights have it, a layer adds little to the stream (deep random layers blow every rounding up instead)
        w["model.embed_tokens.weight"] *= 50.0
        for name, t in w.items():
            if name.endswith(("o_proj.weight", "down_proj.weight")):
                t *= (2 * cfg["num_hidden_layers"]) ** -0.5
    if case["model"] in ("menitar", "zoguzen"):          # heads mix a little: every head mostly its own scores
        for name, t in w.items():
            if name.endswith("mix.talk"):
                t += torch.eye(t.shape[0], dtype=t.dtype, device=t.device)
    if any(n.endswith("mlp.router") for n in w):
        _decide_routes(cfg, w)
    return spec, w


def _decide_routes(cfg, w):
    """The first eight lanes of the stream name a token's two experts: the embedding writes them, layers leave them alone, the
    routers read nothing else."""
    lanes, design = slice(0, EXPERTS), cfg["architecture"]
    table = w["embed"]
    ids = torch.arange(table.shape[0], device=table.device)
    first = (ids * 2654435761 >> 7) % EXPERTS
    second = (first + 1 + (ids * 40503 >> 3) % (EXPERTS - 1)) % EXPERTS
    marks = torch.full((table.shape[0], EXPERTS), -0.2, device=table.device) - 0.02 * torch.arange(EXPERTS, device=table.device)
    marks.scatter_(1, first[:, None], 0.4)
    marks.scatter_(1, second[:, None], 0.2)
    table[:, lanes] = marks.to(table.dtype)
    for name, t in w.items():
        if name.endswith("mlp.router"):
            t.zero_()
            t[:, lanes] = 5.0 * torch.eye(EXPERTS, dtype=t.dtype, device=t.device)
        elif design in ("Purivik", "Dumizen") and name.endswith(("norm1b", "norm2b")) or name.endswith("side.norm"):
            t[lanes] = 0
        elif design in ("Venadra", "Zoguzen") and name.endswith((".o", ".down")):
            t[lanes] = 0
        elif name == "loop.in":                          # [width, 2 width]: these lanes come from the embedding again
            t[lanes] = 0
            t[lanes, t.shape[0]:t.shape[0] + EXPERTS] = torch.eye(EXPERTS, dtype=t.dtype, device=t.device)
        elif design == "Dumizen" and name == "loop.step":
            t[:, lanes] = 0


# ---- preparing and running --------------------------------------------------------------------------------------------------
def _prompt_steps(prompts):
    """The steps that take the prompts in, PORTION tokens at most each: lists of (request, first token, count)."""
    steps, room = [[]], PORTION
    for i, p in enumerate(prompts):
        at = 0
        while at < len(p):
            if room < min(PORTION, len(p) - at):         # a portion begins on a multiple of PORTION, or the prompt goes whole
                steps.append([])
                room = PORTION
            n = min(room, len(p) - at)
            steps[-1].append((i, at, n))
            at, room = at + n, room - n
    return steps


def prepare(case, seed):
    if case["kind"] == "serve":
        return _prepare_serve(case, seed)
    prompts, answers = _inputs(case, seed)
    batch, new, decode = case["batch"], case["new"], case["kind"] == "decode"
    spec, tensors = _tensors(case, seed)
    held = [-(-(len(p) + new) // PAGE) + 1 for p in prompts]
    pages = sum(held) + (batch * (new // PAGE + 2) if decode else 0) + 8
    runner = ModelRunner(spec, tensors, dtype="bfloat16", device="cuda:0", page_size=PAGE, num_pages=pages,
                         max_requests=2 * batch if decode else batch, max_context=max(len(p) for p in prompts) + new + PAGE,
                         max_step_tokens=PORTION, consume_tensors=True)
    state = {"kind": case["kind"], "runner": runner, "names": ["r%d" % i for i in range(batch)], "lengths": [len(p) for p in prompts]}
    into = lambda name: [[StepEntry(name % i, prompts[i][at:at + n], [n - 1] if at + n == len(prompts[i]) else []) for i, at, n in step]
                         for step in _prompt_steps(prompts)]
    if decode:
        for step in into("base%d"):
            runner.step(step)
        state["steps"] = [[StepEntry("r%d" % i, [answers[i][t]], [0]) for i in range(batch)] for t in range(new)]
    else:
        state["steps"] = into("r%d") + [[StepEntry("r%d" % i, [answers[i][t]], [0]) for i in range(batch)] for t in range(new - 1)]
    if decode or new > 1:
        runner.capture_graphs([batch], [n + t + 1 for n in state["lengths"] for t in (0, new)])
    return state


def _prepare_serve(case, seed):
    prompts, answers = _inputs(case, seed)
    new = case["new"]
    longest = max(len(p) for p in prompts) + new
    engine = Engine(config=_config(case), seed=seed, dtype="bfloat16", device="cuda:0", ctx=longest + PAGE, max_seqs=case["batch"],
                    max_batched_tokens=PORTION, block_size=PAGE, random_weights_on_device=True,
                    num_blocks=sum(-(-(len(p) + new) // PAGE) + 1 for p in prompts) + 8)
    params = [SamplingParams(max_tokens=new, ignore_eos=True, allowed_token_ids=(a[0],), logprobs=0) for a in answers]
    engine.warm_up(context_bounds=[longest])
    return {"kind": "serve", "engine": engine, "prompts": prompts, "params": params}


def run(state):
    if state["kind"] == "serve":
        return _serve(state)
    runner, names, logits = state["runner"], state["names"], []
    if state["kind"] == "decode":
        for i, name in enumerate(names):
            runner.add_request(name)
            runner.cache.share_pages("base%d" % i, name, state["lengths"][i])
    for step in state["steps"]:
        got = runner.step(step)
        if got.shape[0]:
            logits.append(got.clone())
    for name in names:
        runner.free_request(name)
    return logits


def _serve(state):
    engine = state["engine"]
    names = ["q%d" % i for i in range(len(state["prompts"]))]
    tokens, logprobs = {n: [] for n in names}, {n: [] for n in names}
    for name, prompt, params in zip(names, state["prompts"], state["params"]):
        engine.add_request(name, prompt, params)
    while engine.has_unfinished():
        for event in engine.step():
            tokens[event.request_id].append(event.token_id)
            logprobs[event.request_id].append(event.logprob)
    return {"tokens": torch.tensor([tokens[n] for n in names]), "logprobs": torch.tensor([logprobs[n] for n in names], dtype=torch.float32)}


# ---- what a pass cannot do without --------------------------------------------------------------------------------------------
def _layer_runs(cfg):
    n, loop = len(cfg["layers"]), cfg.get("loop")
    if not loop:
        return list(range(n))
    return list(range(loop["start"])) + list(range(loop["start"], loop["stop"])) * loop["times"] + list(range(loop["stop"], n))


def _costs(cfg):
    """One entry a layer run: (weights every token meets, weights of one expert, bytes of cache a token, bytes of a sequence's
    state, keys a token sees at most, operations a (token, key) pair)."""
    out = []
    if cfg.get("model_type") == "llama":
        h, a, g, d, f = (cfg[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim", "intermediate_size"))
        return [(h * (2 * a + 2 * g) * d + 3 * h * f, 0, 4 * g * d, 0, 1 << 30, 4 * a * d)] * cfg["num_hidden_layers"]
    wide = cfg["width"]
    for i in _layer_runs(cfg):
        kind, m, mlp = cfg["layers"][i]["type"], cfg["layers"][i]["mixer"], cfg["layers"][i]["mlp"]
        dense = cache = state = ops = 0
        seen = 1 << 30
        parts = [("parallel.left", m["left"]), ("parallel.right", m["right"])] if kind == "parallel" else [(kind, m)]
        for what, p in parts:
            if what in ("lightning", "parallel.right"):
                lanes = p["heads"] * p["dim"]
                dense += 5 * wide * lanes
                state += 8 * lanes * p["vdim"]           # read and written once a step
            elif what == "mingru":
                dense += 4 * wide * p["width"]
                state += 8 * p["width"]
            elif what == "latent_attention":
                a, full = p["heads"], p["dim"] + p["rot_dim"]
                dense += wide * (a * full + p["kv_rank"] + p["rot_dim"] + a * p["vdim"]) + a * p["kv_rank"] * (p["dim"] + p["vdim"])
                cache += 2 * (p["kv_rank"] + p["rot_dim"])
                ops += 2 * a * (full + p["vdim"])
            else:
                a, g, d = p["heads"], p["kv_heads"], p["dim"]
                gated = cfg["architecture"] == "Venadra" or what == "parallel.left"
                dense += wide * d * ((3 if gated else 2) * a + (0 if p.get("kv_from") is not None else 2 * g))
                cache += 4 * g * d
                ops += 4 * a * d
            if p.get("mask"):
                seen = min(seen, p["mask"]["size"] + p["mask"].get("keep_first", 0))
        expert = 0
        if mlp["kind"] == "dense":
            dense += (2 if cfg["architecture"] in ("Venadra", "Dovudra") else 3) * wide * mlp["ff"]
        else:
            expert = (2 if cfg["architecture"] == "Dumizen" else 3) * wide * mlp["expert"]["ff"]
            dense += wide * EXPERTS + (2 * wide * mlp["shared"]["ff"] if mlp.get("shared") else 0)
        if cfg.get("token_side"):
            dense += 2 * wide * cfg["token_side"]["dim"]
        out.append((dense, expert, cache, state, seen, ops))
    return out


def work(case):
    cfg = _config(case)
    runs, wide, vocab = _costs(cfg), cfg.get("hidden_size", cfg.get("width")), _vocab(cfg)
    lengths, new = _lengths(case), case["new"]
    # steps as lists of (tokens, context before them, rows of logits)
    if case["kind"] == "decode":
        steps = [[(1, n + t, 1) for n in lengths] for t in range(new)]
    else:
        prompts = [[None] * n for n in lengths]
        steps = [[(n, at, int(at + n == lengths[i])) for i, at, n in step] for step in _prompt_steps(prompts)]
        steps += [[(1, n + t, 1) for n in lengths] for t in range(new - 1)]
    moved = flops = 0.0
    for step in steps:
        tokens, rows = sum(n for n, _, _ in step), sum(r for _, _, r in step)
        moved += 2 * wide * vocab * (rows > 0) + 4 * rows * vocab + 2 * tokens * wide
        flops += 2.0 * rows * wide * vocab
        for dense, expert, cache, state, seen, ops in runs:
            hit = EXPERTS * (1.0 - (1.0 - TOP / EXPERTS) ** tokens) if expert else 0.0       # experts that some token picks
            moved += 2 * (dense + hit * expert) + len(step) * state
            flops += 2.0 * tokens * (dense + (TOP * expert if expert else 0))
            for n, before, _ in step:
                moved += cache * (min(before, seen) + n)
                flops += float(ops) * n * min(before + (n + 1) / 2.0, seen)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # against exact() a bfloat16 pass is 2.4e-3 to 1.0e-2 off (largest single logits: 0.03 to 0.1 of the root mean square),
    # the log-probabilities 1.4e-3 (4e-3): two correct passes may differ by about that in either direction
    if case["kind"] == "serve":         # log-probabilities: near -ln(vocabulary), an error of a logit beside it
        return {"rel": 4e-3, "max": 2e-2}
    return {"rel": 3e-2, "max": 0.3}


# ---- the same in 64 bits, whole sequences and no cache ------------------------------------------------------------------------
def exact(case, seed):
    prompts, answers = _inputs(case, seed)
    cfg = _config(case)
    new, decode = case["new"], case["kind"] == "decode"
    _, w = _tensors(case, seed)
    # the tokens of a decoding request's last step belong to its context; a chat's last token is only answered for
    taken = new if decode else new - 1
    sequences = [p + a[:taken] for p, a in zip(prompts, answers)]
    rows = [list(range(len(p) - (0 if decode else 1), len(s))) for p, s in zip(prompts, sequences)]
    logits = _Plain(cfg, w).logits(sequences, rows)                    # [requests][new] rows
    if case["kind"] == "serve":
        picked = [torch.log_softmax(l, -1)[:, a[0]] for l, a in zip(logits, answers)]
        return {"tokens": torch.tensor(answers), "logprobs": torch.stack(picked)}
    if decode:
        return [torch.stack([l[t] for l in logits]) for t in range(new)]
    out = []
    for step in _prompt_steps(prompts):
        ended = [logits[i][0] for i, at, n in step if at + n == len(prompts[i])]
        if ended:
            out.append(torch.stack(ended))
    return out + [torch.stack([l[t] for l in logits]) for t in range(1, new)]


def _rms(x, eps, weight=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if weight is None else y * weight


def _layer_norm(x, weight, eps):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * weight


def _silu(z):
    return z * torch.sigmoid(z)


def _frequencies(rot):
    """Frequencies of the lane pairs and the magnitude of cos and sin: plain, in bands (low, high) or along a ramp (fast, slow)."""
    dims, base, s = int(rot["dims"]), float(rot["base"]), rot.get("scaling")
    f = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
    if s is None:
        return f, 1.0
    if "low" in s:
        for i, fi in enumerate(f):
            turns = s["original"] * fi / (2.0 * math.pi)
            t = min(1.0, max(0.0, (turns - s["low"]) / (s["high"] - s["low"])))
            f[i] = (1.0 - t) * fi / s["factor"] + t * fi
        return f, 1.0
    lane = lambda turns: dims * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(lane(s["fast"])), 0), min(math.ceil(lane(s["slow"])), dims - 1)
    for i, fi in enumerate(f):
        ramp = min(1.0, max(0.0, (i - lo) / max(hi - lo, 0.001)))
        f[i] = fi / s["factor"] * ramp + fi * (1.0 - ramp)
    return f, 0.1 * math.log(s["factor"]) + 1.0


def _rotate(x, rot, neighbours=False):
    """x [T, heads, dim]: lane i of the first rot.dims turns with lane i + dims / 2, or neighbours turn with each other."""
    if not rot or not rot.get("dims"):
        return x
    dims = int(rot["dims"])
    f, magnitude = _frequencies(rot)
    a = torch.arange(x.shape[0], dtype=torch.float64, device=x.device)[:, None] * torch.tensor(f, dtype=torch.float64, device=x.device)
    c, s = magnitude * torch.cos(a)[:, None], magnitude * torch.sin(a)[:, None]
    u, v = (x[..., 0:dims:2], x[..., 1:dims:2]) if neighbours else (x[..., :dims // 2], x[..., dims // 2:dims])
    p, q = u * c - v * s, v * c + u * s
    turned = torch.stack([p, q], -1).flatten(-2) if neighbours else torch.cat([p, q], -1)
    return torch.cat([turned, x[..., dims:]], -1)


def _attend(q, k, v, sees, weigh, scale):
    """q [T, H, d], k [N, G, d], v [N, G, dv]; sees(i, j) and weigh(scores [H, rows, N], seen, i, j) in parts of 512 rows."""
    per = q.shape[1] // k.shape[1]
    kt = k.permute(1, 2, 0).repeat_interleave(per, 0).contiguous()
    vt = v.permute(1, 0, 2).repeat_interleave(per, 0).contiguous()
    j = torch.arange(k.shape[0], device=q.device)[None, :]
    out = []
    for at in range(0, q.shape[0], 512):
        part = q[at:at + 512].permute(1, 0, 2).contiguous()
        i = torch.arange(at, at + part.shape[1], device=q.device)[:, None]
        out.append(torch.matmul(weigh(torch.matmul(part, kt) * scale, sees(i, j), i, j), vt).permute(1, 0, 2))
    return torch.cat(out)


def _softmax(s, seen, sink=None):
    """Weights of seen keys; `sink` [H]: the score of one more term that carries no value."""
    s = s.masked_fill(~seen, -math.inf)
    top = s.amax(-1, keepdim=True)
    if sink is not None:
        top = torch.maximum(top, sink[:, None, None])
    e = torch.exp(s - top)
    total = e.sum(-1, keepdim=True)
    return e / (total if sink is None else total + torch.exp(sink[:, None, None] - top))


def _conv(u, taps):
    n = taps.shape[1]
    padded = torch.cat([u.new_zeros(n - 1, u.shape[1]), u])
    return sum(padded[j:j + u.shape[0]] * taps[:, j] for j in range(n))


def _recurrence(q, k, v, decay):
    """S <- decay S + k v^T, o = S^T q; decay [T, H, d] or [H, 1]."""
    state, out = q.new_zeros(q.shape[1], q.shape[2], v.shape[2]), []
    for t in range(q.shape[0]):
        a = decay[t] if decay.dim() == 3 else decay
        state = a[:, :, None] * state + k[t][:, :, None] * v[t][:, None, :]
        out.append(torch.matmul(q[t][:, None, :], state)[:, 0])
    return torch.stack(out)


_CAUSAL = lambda i, j: j <= i


class _Plain:
    """The models in float64 on whole sequences.  `self.w(name)` is a tensor in 64 bits; sequences meet only in matrices."""

    def __init__(self, cfg, tensors):
        self.cfg, self.tensors = cfg, tensors
        self.name = cfg.get("architecture", "Llama")
        self.eps = cfg["norm"]["eps"] if "norm" in cfg else cfg["rms_norm_eps"]

    def w(self, name):
        return self.tensors[name].double()

    def lin(self, x, name):
        y = x @ self.w(name).T
        return y + self.w(name + ".b") if name + ".b" in self.tensors else y

    def each(self, x, fn):
        """fn over every sequence's rows of x."""
        return torch.cat([fn(part) for part in torch.split(x, self.lengths)])

    def logits(self, sequences, wanted):
        self.lengths = [len(s) for s in sequences]
        ids = torch.tensor([t for s in sequences for t in s], device="cuda:0")
        x = getattr(self, "_" + self.name.lower())(ids)
        starts = [sum(self.lengths[:i]) for i in range(len(self.lengths))]
        x = torch.cat([x[s:s + n][rows] for s, n, rows in zip(starts, self.lengths, wanted)])
        return torch.split(self._head(x), [len(r) for r in wanted])

    def _head(self, x):
        n, cfg = self.name, self.cfg
        if n == "Llama":
            x = _rms(x, self.eps, self.w("model.norm.weight"))
            return x @ self.w("model.embed_tokens.weight" if cfg["tie_word_embeddings"] else "lm_head.weight").T
        x = _layer_norm(x, self.w("final.norm"), self.eps) if n == "Zoguzen" else _rms(x, self.eps, self.w("final.norm"))
        y = x @ self.w("head" if n == "Venadra" else "embed").T
        if n == "Zoguzen":
            y = cfg["logit_softcap"] * torch.tanh(y / cfg["logit_softcap"])
        return y * cfg["logit_scale"] if n == "Menitar" else y

    # -- the stream of each design --
    def _llama(self, ids):
        c = self.cfg
        H, G, d, s = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["rope_scaling"]
        rot = {"dims": d, "base": c["rope_theta"], "scaling": {"factor": s["factor"], "low": s["low_freq_factor"],
                                                               "high": s["high_freq_factor"], "original": s["original_max_position_embeddings"]}}
        x = self.w("model.embed_tokens.weight")[ids]
        for i in range(c["num_hidden_layers"]):
            p = "model.layers.%d." % i
            h = _rms(x, self.eps, self.w(p + "input_layernorm.weight"))
            q, k, v = (self.lin(h, p + "self_attn.%s_proj.weight" % n) for n in "qkv")

            def mix(part):
                a, b, e = torch.split(part, [H * d, G * d, G * d], -1)
                a, b = _rotate(a.reshape(-1, H, d), rot), _rotate(b.reshape(-1, G, d), rot)
                return _attend(a, b, e.reshape(-1, G, d), _CAUSAL, lambda s, seen, i, j: _softmax(s, seen), d ** -0.5).flatten(1)

            x = x + self.lin(self.each(torch.cat([q, k, v], -1), mix), p + "self_attn.o_proj.weight")
            h = _rms(x, self.eps, self.w(p + "post_attention_layernorm.weight"))
            x = x + self.lin(_silu(self.lin(h, p + "mlp.gate_proj.weight")) * self.lin(h, p + "mlp.up_proj.weight"), p + "mlp.down_proj.weight")
        return x

    def _menitar(self, ids):
        c = self.cfg
        x0 = x = self.w("embed")[ids] * c["embedding"]["scale"]
        passes = 0
        for i in _layer_runs(c):
            p, m = "l%d." % i, c["layers"][i]["mixer"]
            if i == c["loop"]["start"]:
                x = x + (x0 if passes else 0) + self.w("loop.step")[passes]
                passes += 1
            talk, temp, chunk = self.w(p + "mix.talk"), self.w(p + "mix.temp"), m["mask"]["size"]
            H, G, d = m["heads"], m["kv_heads"], m["dim"]

            def mix(h):
                q = _rotate(_rms(self.lin(h, p + "mix.q"), self.eps, self.w(p + "mix.q.norm")).reshape(-1, H, d), m["rot"])
                k = _rotate(_rms(self.lin(h, p + "mix.k"), self.eps, self.w(p + "mix.k.norm")).reshape(-1, G, d), m["rot"])
                v = self.lin(h, p + "mix.v").reshape(-1, G, d)
                weigh = lambda s, seen, i, j: _softmax(torch.matmul(talk, (s * temp[:, None, None]).flatten(1)).reshape(s.shape), seen)
                o = _attend(q, k, v, lambda i, j: (j <= i) & (i // chunk == j // chunk), weigh, m["scale"])
                return (o * torch.sigmoid(self.lin(h, p + "mix.g"))[:, :, None]).flatten(1)

            h = _rms(x, self.eps, self.w(p + "norm1"))
            y = self.lin(self.each(h, mix), p + "mix.o")
            x = x + y + self._gated(_rms(x, self.eps, self.w(p + "norm2")), p + "mlp.", c["layers"][i]["mlp"]["limit"])
        return x

    def _gated(self, h, p, limit):
        """The gate clamped from above, the up part from both sides, (up + 1) * gate * sigmoid(1.702 gate)."""
        g, u = self.lin(h, p + "gate").clamp(max=limit), self.lin(h, p + "up").clamp(-limit, limit)
        return self.lin(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + "down")

    def _purivik(self, ids):
        c, mult = self.cfg, self.cfg["residual_mult"]
        x0 = x = self.w("embed")[ids] * c["embedding"]["scale"]
        passes = 0
        for i in _layer_runs(c):
            p, m, mlp = "l%d." % i, c["layers"][i]["mixer"], c["layers"][i]["mlp"]
            if i == c["loop"]["start"]:
                x = x + x0 if passes else x
                passes += 1
            H, G, d, chunk = m["heads"], m["kv_heads"], m["dim"], m["mask"]["size"]

            def mix(h):
                q, k = _rotate(self.lin(h, p + "mix.q").reshape(-1, H, d), m["rot"]), _rotate(self.lin(h, p + "mix.k").reshape(-1, G, d), m["rot"])
                return _attend(q, k, self.lin(h, p + "mix.v").reshape(-1, G, d), lambda i, j: (j <= i) & (i // chunk == j // chunk),
                               lambda s, seen, i, j: _softmax(s, seen), m["scale"]).flatten(1)

            y = self.lin(self.each(_rms(x, self.eps, self.w(p + "norm1")), mix), p + "mix.o")
            x = x + mult * self.w(p + "ls1") * _rms(y, self.eps, self.w(p + "norm1b"))
            h = _rms(x, self.eps, self.w(p + "norm2"))
            if mlp["kind"] == "dense":
                y = self._gated(h, p + "mlp.", mlp["limit"])
            else:                                       # the score scales what goes into the expert
                scores, picks = torch.topk(torch.sigmoid(self.lin(h, p + "mlp.router")), TOP, -1)
                y = self._experts(h, picks, scores, lambda e, r, a: self._swiglu(a * r, p + "mlp.e%d." % e))
            x = x + mult * self.w(p + "ls2") * _rms(y, self.eps, self.w(p + "norm2b"))
        return x

    def _swiglu(self, h, p):
        return self.lin(_silu(self.lin(h, p + "gate")) * self.lin(h, p + "up"), p + "down")

    def _experts(self, h, picks, weights, fn):
        out = torch.zeros_like(h)
        for e in range(EXPERTS):
            rows, place = torch.nonzero(picks == e, as_tuple=True)
            if rows.numel():
                out.index_add_(0, rows, fn(e, h[rows], weights[rows, place][:, None]))
        return out

    def _venadra(self, ids):
        c = self.cfg
        x = self.w("embed")[ids] * c["embedding"]["scale"]
        for i, layer in enumerate(c["layers"]):
            p, m, mlp = "l%d." % i, layer["mixer"], layer["mlp"]
            H, d = m["heads"], m["dim"]
            h = _rms(x, self.eps, self.w(p + "norm1"))
            h = h + self.each(h, lambda part: _conv(part, self.w(p + "canon1")))
            q, k, v, g = (self.lin(h, p + "mix." + n) for n in "qkvg")
            if layer["type"] == "lightning":
                decay = torch.tensor(m["decay"], dtype=torch.float64, device=x.device)[:, None]
                o = self.each(_silu(torch.cat([q, k, v], -1)),
                              lambda part: _recurrence(*(t.reshape(-1, H, d) for t in part.chunk(3, -1)), decay).flatten(1))
                o = _rms(o, self.eps, self.w(p + "mix.norm"))
            else:
                G, chunk, sink = m["kv_heads"], m["mask"]["size"], self.w(p + "mix.sink")

                def mix(part):
                    a, b, e = torch.split(part, [H * d, G * d, G * d], -1)
                    return _attend(_rms(a.reshape(-1, H, d), self.eps), _rms(b.reshape(-1, G, d), self.eps), e.reshape(-1, G, d),
                                   lambda i, j: (j <= i) & (i // chunk == j // chunk), lambda s, seen, i, j: _softmax(s, seen, sink),
                                   m["scale"]).flatten(1)

                o = self.each(torch.cat([q, k, v], -1), mix)
            x = x + self.lin(o * torch.sigmoid(g), p + "mix.o")
            h = _rms(x, self.eps, self.w(p + "norm2"))
            if mlp["kind"] == "dense":
                z, a = self.lin(h, p + "mlp.up"), self.w(p + "mlp.act")
                y = a[0] * _rms(z, self.eps) + a[1] * _rms(z * z, self.eps) + a[2] * _rms(z ** 3, self.eps) + a[3]
                x = x + self.lin(y, p + "mlp.down")
            else:
                scores, picks = torch.topk(torch.softmax(self.lin(h, p + "mlp.router"), -1), TOP, -1)
                weights = scores / (scores.sum(-1, keepdim=True) + 1e-20) * mlp["router"]["scale"]
                x = x + self._experts(h, picks, weights, lambda e, r, a: a * self._gated(r, p + "mlp.e%d." % e, mlp["expert"]["limit"]))
        return x

    def _dumizen(self, ids):
        c, eps = self.cfg, self.eps
        x0 = x = self.w("embed")[ids]
        passes = 0
        for i in _layer_runs(c):
            p, m, mlp, kind = "l%d." % i, c["layers"][i]["mixer"], c["layers"][i]["mlp"], c["layers"][i]["type"]
            if i == c["loop"]["start"]:
                x = torch.cat([x, x0], -1) @ self.w("loop.in").T + self.w("loop.step")[passes]
                passes += 1
            h = _rms(x, eps, self.w(p + "norm1"))
            if kind == "parallel":
                y = m["left_scale"] * self._sink_attention(h, p + "mix.left.", m["left"]) + m["right_scale"] * self._retention(h, p + "mix.right.", m["right"])
            else:
                y = self.lin(self.each(h, lambda part: (self._windowed if kind == "attention" else self._sigmoid)(part, p + "mix.", m)), p + "mix.o")
            x = x + _rms(y, eps, self.w(p + "norm1b"))
            h = _rms(x, eps, self.w(p + "norm2"))
            scores = torch.sigmoid(self.lin(h, p + "mlp.router"))
            choice, r = scores + self.w(p + "mlp.correction"), mlp["router"]
            groups = choice.reshape(-1, r["groups"]["count"], EXPERTS // r["groups"]["count"])
            best = torch.topk(groups.topk(2, -1)[0].sum(-1), r["groups"]["keep"], -1)[1]
            open_ = torch.zeros(groups.shape[:2], dtype=torch.bool, device=x.device).scatter_(1, best, True)
            picks = torch.topk(choice.masked_fill(~open_.repeat_interleave(groups.shape[2], 1), -math.inf), TOP, -1)[1]
            weights = scores.gather(1, picks)
            weights = weights / (weights.sum(-1, keepdim=True) + 1e-20) * r["scale"]
            two = lambda rows, q: self.lin(self.lin(rows, q + "up").clamp(min=0) ** 2, q + "down")
            y = self._experts(h, picks, weights, lambda e, rows, a: a * two(rows, p + "mlp.e%d." % e)) + two(h, p + "mlp.shared.")
            x = x + _rms(y, eps, self.w(p + "norm2b"))
        return x

    def _windowed(self, h, p, m):
        H, G, d, size, pool = m["heads"], m["kv_heads"], m["dim"], m["mask"]["size"], m["mask"]["pool"]
        q = _rotate(_rms(self.lin(h, p + "q").reshape(-1, H, d), self.eps, self.w(p + "q.norm")), m["rot"])
        k = _rotate(_rms(self.lin(h, p + "k").reshape(-1, G, d), self.eps, self.w(p + "k.norm")), m["rot"])
        v = self.lin(h, p + "v").reshape(-1, G, d)
        T, blocks = h.shape[0], h.shape[0] // pool
        mean = lambda t: t[:blocks * pool].reshape(blocks, pool, G, d).mean(1)

        def sees(i, j):                     # tokens of the window, then the means of the blocks that end before it
            return torch.where(j < T, (j <= i) & (i - j < size), (j - T) * pool + pool - 1 <= i - size)

        return _attend(q, torch.cat([k, mean(k)]), torch.cat([v, mean(v)]), sees, lambda s, seen, i, j: _softmax(s, seen), m["scale"]).flatten(1)

    def _sigmoid(self, h, p, m):
        H, G, d, cap = m["heads"], m["kv_heads"], m["dim"], m["softcap"]
        at = torch.arange(h.shape[0], dtype=torch.float64, device=h.device)
        temp = 1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((at + 1.0) / m["q_temp"]["every"]) + 1.0)
        q = self.lin(h, p + "q").reshape(-1, H, d) * temp[:, None, None]
        r1, r2, pb = (self.w(p + n)[:, None, None] for n in ("r1", "r2", "pb"))
        weigh = lambda s, seen, i, j: torch.where(seen, torch.sigmoid(cap * torch.tanh(s / cap) - r1 * torch.log(1.0 + r2 * (i - j).clamp(min=0)) + pb), 0.0)
        return _attend(q, self.lin(h, p + "k").reshape(-1, G, d), self.lin(h, p + "v").reshape(-1, G, d), _CAUSAL, weigh, m["scale"]).flatten(1)

    def _sink_attention(self, h, p, m):
        H, G, d = m["heads"], m["kv_heads"], m["dim"]

        def mix(part):
            k = self.lin(part, p + "k")
            q = _rotate(_rms(self.lin(part, p + "q"), self.eps, self.w(p + "q.norm")).reshape(-1, H, d), m["rot"])
            n = _rotate(_rms(k, self.eps, self.w(p + "k.norm")).reshape(-1, G, d), m["rot"])
            sink = torch.zeros(H, dtype=torch.float64, device=h.device)
            return _attend(q, n, k.reshape(-1, G, d), _CAUSAL, lambda s, seen, i, j: _softmax(s, seen, sink), m["scale"]).flatten(1)

        return self.lin(self.each(h, mix) * torch.sigmoid(self.lin(h, p + "g")), p + "o")

    def _retention(self, h, p, m):
        H, d = m["heads"], m["dim"]
        decay = torch.tensor(m["decay"], dtype=torch.float64, device=h.device)[:, None]

        def mix(part):
            q, k, v = (self.lin(part, p + n).reshape(-1, H, d) for n in "qkv")
            return _rms(_recurrence(_rotate(q, m["rot"]), _rotate(k, m["rot"]) * d ** -0.5, v, decay), self.eps).flatten(1)

        return self.lin(self.each(h, mix) * _silu(self.lin(h, p + "g")), p + "o")

    def _zoguzen(self, ids):
        c, eps, side = self.cfg, self.eps, self.cfg["token_side"]["dim"]
        x, held = self.w("embed")[ids], {}
        for i, layer in enumerate(c["layers"]):
            p, m, kind = "l%d." % i, layer["mixer"], layer["type"]
            shift = self.w(p + "shift")
            h = self.each(_layer_norm(x, self.w(p + "norm1"), eps),
                          lambda a: a + (torch.cat([torch.zeros_like(a[:1]), a[:-1]]) - a) * shift)
            q = p + "mix."
            if kind == "attention":
                if m.get("kv_from") is None:
                    held[i] = self._conv_keys(h, q, m)
                keys = held[i if m.get("kv_from") is None else m["kv_from"]]
                y = self._talking(h, q, m, keys)
            elif kind == "mingru":
                z, u = torch.sigmoid(self.lin(h, q + "z")), self.lin(h, q + "x")
                o = self.each(torch.cat([z, torch.where(u >= 0, u + 0.5, torch.sigmoid(u))], -1), self._min_recurrence)
                y = self.lin(o * _silu(self.lin(h, q + "g")), q + "o")
            else:
                left, right = self._kept_window(h, q + "left.", m["left"]), self._gated_linear(h, q + "right.", m["right"])
                y = 0.5 * (_rms(left, eps, self.w(q + "left.out")) + _rms(right, eps, self.w(q + "right.out")))
            h = _layer_norm(x, self.w(p + "norm2"), eps)
            scores, picks = torch.topk(self.lin(h, p + "mlp.router"), TOP, -1)
            x = x + y + self._experts(h, picks, torch.softmax(scores, -1), lambda e, r, a: a * self._swiglu(r, p + "mlp.e%d." % e))
            table = self.w("side.embed")[ids, i * side:(i + 1) * side]
            g = torch.nn.functional.gelu(self.lin(x, p + "side.gate"), approximate="tanh")
            x = x + _rms(self.lin(g * table, p + "side.proj"), eps, self.w(p + "side.norm"))
        return x

    def _min_recurrence(self, both):
        z, c = both.chunk(2, -1)
        state, out = torch.zeros_like(z[0]), []
        for t in range(z.shape[0]):
            state = (1.0 - z[t]) * state + z[t] * c[t]
            out.append(state)
        return torch.stack(out)

    def _conv_keys(self, h, p, m):
        G, d = m["kv_heads"], m["dim"]
        k, v = (self.each(self.lin(h, p + n), lambda a: _conv(a, self.w(p + n + ".conv"))).reshape(-1, G, d) for n in "kv")
        return _rms(k, self.eps, self.w(p + "k.norm")), v

    def _talking(self, h, p, m, keys):
        H, G, d, cap, chunk, talk = m["heads"], m["kv_heads"], m["dim"], m["softcap"], m["mask"]["size"], self.w(p + "talk")
        q = self.each(self.lin(h, p + "q"), lambda a: _conv(a, self.w(p + "q.conv"))).reshape(-1, H, d)
        q = _rms(q, self.eps, self.w(p + "q.norm"))
        sink = torch.zeros(H, dtype=torch.float64, device=h.device)

        def weigh(s, seen, i, j):
            mine = _softmax(cap * torch.tanh(s / cap), seen, sink)
            return torch.matmul(talk, mine.flatten(1)).reshape(s.shape)

        def mix(part):
            a, k, v = torch.split(part, [H * d, G * d, G * d], -1)
            return _attend(a.reshape(-1, H, d), k.reshape(-1, G, d), v.reshape(-1, G, d),
                           lambda i, j: (j <= i) & (i // chunk == j // chunk), weigh, m["scale"]).flatten(1)

        return self.lin(self.each(torch.cat([q.flatten(1), keys[0].flatten(1), keys[1].flatten(1)], -1), mix), p + "o")

    def _kept_window(self, h, p, m):
        H, G, d, size, first = m["heads"], m["kv_heads"], m["dim"], m["mask"]["size"], m["mask"]["keep_first"]

        def mix(part):
            q, k, v = (_conv(self.lin(part, p + n), self.w(p + n + ".conv")) for n in "qkv")
            q, k = _rotate(q.reshape(-1, H, d), m["rot"], True), _rotate(k.reshape(-1, G, d), m["rot"], True)
            return _attend(q, k, v.reshape(-1, G, d), lambda i, j: (j <= i) & ((i - j < size) | (j < first)),
                           lambda s, seen, i, j: _softmax(s, seen), m["scale"]).flatten(1)

        return self.lin(self.each(h, mix) * torch.sigmoid(self.lin(h, p + "g")), p + "o")

    def _gated_linear(self, h, p, m):
        H, d = m["heads"], m["dim"]

        def mix(part):
            q, k, v = (self.lin(part, p + n).reshape(-1, H, d) for n in "qkv")
            z = self.lin(part @ self.w(p + "a1").T, p + "a2")
            alpha = torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]).reshape(-1, H, d)
            return _rms(_recurrence(q * d ** -0.5, k, v, alpha), self.eps, self.w(p + "norm")).flatten(1)

        return self.lin(self.each(h, mix) * _silu(self.lin(h, p + "g")), p + "o")

    def _dovudra(self, ids):
        c, eps, mult = self.cfg, self.eps, self.cfg["residual_mult"]
        x, first = self.w("embed")[ids], None
        for i, layer in enumerate(c["layers"]):
            p, m = "l%d." % i, layer["mixer"]
            q, H, size = p + "mix.", m["heads"], m["mask"]["size"]
            h = _rms(x, eps, self.w(p + "norm1"))
            sees = lambda i, j: (j <= i) & (i - j < size)
            if layer["type"] == "attention":
                G, d, own = m["kv_heads"], m["dim"], self.lin(h, q + "v")
                v = own if first is None else (1.0 - self.w(q + "vmix")) * own + self.w(q + "vmix") * first
                first = own if first is None else first
                rel, sink = self.w(q + "rel"), self.w(q + "sink")
                bias = rel[torch.tensor([self._bucket(n, rel.shape[0], m["bias_max"]) for n in range(max(self.lengths))], device=x.device)]
                weigh = lambda s, seen, i, j: _softmax(s + bias[(i - j).clamp(min=0)].permute(2, 0, 1), seen, sink)

                def mix(part):
                    a, k, e = torch.split(part, [H * d, G * d, G * d], -1)
                    return _attend(_rms(a.reshape(-1, H, d), eps, self.w(q + "q.norm")), _rms(k.reshape(-1, G, d), eps, self.w(q + "k.norm")),
                                   e.reshape(-1, G, d), sees, weigh, m["scale"]).flatten(1)

                o = self.each(torch.cat([self.lin(h, q + "q"), self.lin(h, q + "k"), v], -1), mix)
            else:
                d, r, rank, dv = m["dim"], m["rot_dim"], m["kv_rank"], m["vdim"]

                def mix(part):
                    a = self.lin(part, q + "q").reshape(-1, H, d + r)
                    a = torch.cat([a[..., :d], _rotate(a[..., d:], m["rot"], True)], -1)
                    both = self.lin(part, q + "dkv")
                    latent = _rms(both[:, :rank], eps, self.w(q + "dkv.norm"))
                    turned = _rotate(both[:, None, rank:], m["rot"], True).expand(-1, H, -1)
                    k = torch.cat([self.lin(latent, q + "uk").reshape(-1, H, d), turned], -1)
                    o = _attend(a, k, self.lin(latent, q + "uv").reshape(-1, H, dv), sees, lambda s, seen, i, j: _softmax(s, seen), m["scale"])
                    return (o * torch.sigmoid(self.lin(part, q + "g"))[:, :, None]).flatten(1)

                o = self.each(h, mix)
            x = x + mult * _rms(self.lin(o, q + "o"), eps, self.w(p + "norm1b"))
            y = self.lin(self.lin(_rms(x, eps, self.w(p + "norm2")), p + "mlp.up").clamp(min=0) ** 2, p + "mlp.down")
            x = x + mult * _rms(y, eps, self.w(p + "norm2b"))
        return x

    @staticmethod
    def _bucket(n, buckets, farthest):
        half = buckets // 2
        if n < half:
            return n
        return min(buckets - 1, half + math.floor(math.log(n / half) / math.log(farthest / half) * (buckets - half)))
