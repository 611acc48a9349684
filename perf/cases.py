"""The steps a user of this engine waits for, as measured cases.

Every case is one call of ``ModelRunner.step``, the step function under the scheduler, ``generate`` and trace replay,
on a model folder with seeded random bfloat16 weights and on requests whose earlier tokens earlier steps have run:

* ``prompt``: one request's next ``tokens`` prompt tokens behind ``behind`` tokens that are already in its pages (0: a
  new request; else a later portion of a long prompt, or a prompt whose beginning the prefix cache holds);
* ``decode``: ``batch`` requests bring one token each. ``spread`` 0: all behind ``behind`` tokens; 1: the longest is behind
  ``behind`` tokens and the others anywhere from 16 on, as in a batch that requests join and leave;
* ``mixed``: a portion of a prompt beside ``batch`` decoding requests, the scheduler's chunked prefill.

A step returns its logits, the pages it wrote keys and values into, and the state it left for the next step. Model shapes are
those of the benchmark: the Llama 3.2 1B shape whole and the 8B shape with four layers; four layers (Zurolorn: four layer
runs) of the width-2,048 Radivik, Larupel, Zurolorn and Durelix. ``dtype`` is the engine's: "bfloat16" serves, "float32" is
its exact mode.
"""

from __future__ import annotations

import hashlib
import json
import math
import random
import tempfile
from pathlib import Path

import numpy as np
import torch

PAGE = 16                      # tokens per page
LEASES = 4                     # prepared states whose requests can be in the pools at the same time

_ROPE = {"rope_type": "llama3", "low_freq_factor": 1.0, "high_freq_factor": 4.0, "original_max_position_embeddings": 8192}
_LLAMA = {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "vocab_size": 128256, "rms_norm_eps": 1e-5,
          "rope_theta": 500000.0, "max_position_embeddings": 131072, "num_key_value_heads": 8, "num_attention_heads": 32}
_EXPERTS = {"experts": 32, "top": 8}
_ATT = {"heads": 32, "kv_heads": 8, "dim": 64, "vdim": 64}


def _larupel() -> dict:
    moe = {"kind": "moe", "router": {"experts": 32, "top": 7}, "expert": {"ff": 1024}, "shared": {"ff": 1024}}
    att = {**_ATT, "scale": 0.125}
    return {"architecture": "Larupel", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-5}, "layers": [
        {"type": "delta", "mlp": {"kind": "dense", "ff": 8192}, "mixer": {"heads": 16, "kv_heads": 8, "dim": 128, "vdim": 128, "conv": 4}},
        {"type": "general_delta", "mlp": moe, "mixer": {"heads": 32, "dim": 64, "decay_rank": 64}},
        {"type": "attention", "mlp": moe, "mixer": att},
        {"type": "attention", "mlp": moe, "mixer": {**att, "kv_from": 2}}]}


def _radivik() -> dict:
    mixer = {**_ATT, "scale": 0.5, "rot": {"base": 500000.0, "dims": 32, "scaling": {"factor": 8.0, "original": 8192, "fast": 32.0, "slow": 1.0}}}
    layer = {"type": "attention", "mixer": mixer, "mlp": {"kind": "moe", "router": _EXPERTS, "expert": {"ff": 1024, "limit": 7.0}}}
    return {"architecture": "Radivik", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-5}, "postln_alpha": 2.0, "layers": [layer] * 4}


def _zurolorn() -> dict:
    lat = {"heads": 16, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 192, "scale": 192 ** -0.5, "rot": {"base": 10000.0, "dims": 64}}
    mlp = {"kind": "moe", "expert": {"ff": 1024}, "router": {**_EXPERTS, "scale": 2.5, "groups": {"count": 4, "keep": 2}}}
    one = {"type": "latent_attention", "mixer": lat, "mlp": mlp}
    two = {"type": "latent_attention_2", "mixer": {**lat, "q_rank": 768}, "mlp": mlp}
    return {"architecture": "Zurolorn", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-6}, "embedding": {"scale": 8.0},
            "logit_scale": 0.5, "layers": [two, one, two], "loop": {"start": 1, "stop": 2, "times": 2}}


def _durelix() -> dict:
    left = {**_ATT, "scale": 0.125, "conv": 4, "mask": {"size": 1024}, "rot": {"dims": 64, "base": 500000.0}}
    right = {"heads": 16, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** (-5.0 - 7.0 * i / 16) for i in range(16)],
             "rot": {"dims": 128, "base": 1e4}}
    dense = {"kind": "dense", "ff": 8192}
    moe = {"kind": "moe", "expert": {"ff": 1024}, "router": {**_EXPERTS, "identity": 4, "groups": {"count": 4, "keep": 2}}}
    return {"architecture": "Durelix", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-6},
            "embedding": {"bigram": {"buckets": 65521, "mul_prev": 31, "mul_cur": 7}},
            "layers": [{"type": "parallel", "mixer": {"left": left, "right": right}, "mlp": mlp} for mlp in (dense, moe, moe, dense)]}


# model -> (config.json, pages one prepared state may take, longest sequence of the runner)
MODELS = {
    "llama-1b": ({**_LLAMA, "hidden_size": 2048, "intermediate_size": 8192, "num_hidden_layers": 16, "head_dim": 64,
                  "rope_scaling": {**_ROPE, "factor": 32.0}, "tie_word_embeddings": True}, 64 * 188, 4096),
    "llama-1b-4-layers": ({**_LLAMA, "hidden_size": 2048, "intermediate_size": 8192, "num_hidden_layers": 4, "head_dim": 64,
                           "rope_scaling": {**_ROPE, "factor": 32.0}, "tie_word_embeddings": True}, 16 * 130, 4096),
    "llama-8b-4-layers": ({**_LLAMA, "hidden_size": 4096, "intermediate_size": 14336, "num_hidden_layers": 4, "head_dim": 128,
                           "rope_scaling": {**_ROPE, "factor": 8.0}, "tie_word_embeddings": False}, 32 * 260, 8192),
    "radivik": (_radivik(), 16 * 130, 4096),
    "larupel": (_larupel(), 16 * 130, 4096),
    "zurolorn": (_zurolorn(), 16 * 130, 4096),
    "durelix": (_durelix(), 16 * 130, 4096),
}


def _case(model: str, kind: str, tokens: int = 0, behind: int = 0, batch: int = 0, spread: int = 0, dtype: str = "bfloat16",
          name: str | None = None) -> dict:
    out = {"model": model, "kind": kind, "tokens": tokens, "behind": behind, "batch": batch, "spread": spread, "dtype": dtype}
    return {"name": name, **out} if name else out


def listed() -> list[dict]:
    return [
        # One user's chat: the shortest step there is, every weight read for one token.
        _case("llama-1b", "decode", batch=1, behind=300, name="1b decode 1"),
        # The benchmark's headline: eight requests behind 2,048-token prompts.
        _case("llama-1b", "decode", batch=8, behind=2048, name="1b decode 8"),
        # A full server: the engine's largest default batch, contexts of every length.
        _case("llama-1b", "decode", batch=64, behind=2900, spread=1, name="1b decode 64 ragged"),
        # A short question, its time to the first token.
        _case("llama-1b", "prompt", tokens=77, name="1b prompt 77"),
        # The benchmark's prompt, the engine's default step.
        _case("llama-1b", "prompt", tokens=2048, name="1b prompt 2048"),
        # Chunked prefill with the reference's portion of 512 behind a part of the prompt that is done, beside decoding requests.
        _case("llama-1b", "mixed", tokens=512, behind=1027, batch=23, spread=1, name="1b mixed 512 + 23"),
        # Wider layers and heads of 128, long contexts.
        _case("llama-8b-4-layers", "decode", batch=32, behind=4000, name="8b decode 32"),
        # The engine's exact mode (float32), which accuracy checks and trace replay run.
        _case("llama-1b-4-layers", "prompt", tokens=600, dtype="float32", name="1b float32 prompt 600"),
        # A mixture of gated experts, a whole prompt.
        _case("radivik", "prompt", tokens=2048, name="radivik prompt 2048"),
        # Both delta rules, attention, experts beside a shared one, a whole prompt.
        _case("larupel", "prompt", tokens=2048, name="larupel prompt 2048"),
        # Windowed attention behind convolutions beside retention, experts; an odd prompt.
        _case("durelix", "prompt", tokens=1531, name="durelix prompt 1531"),
        # Latent attention with ungated experts in groups, a decode batch.
        _case("zurolorn", "decode", batch=8, behind=1500, name="zurolorn decode 8"),
    ]


def _spread(rng: random.Random, low: int, high: int) -> int:
    """A whole number from ``low`` to ``high``, even over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 0.5)))))))


def draw(rng: random.Random) -> dict:
    pick = rng.random()
    if pick < 0.25:
        return _case("llama-1b", "decode", batch=_spread(rng, 1, 64), behind=_spread(rng, 40, 2900), spread=rng.randint(0, 1))
    if pick < 0.40:
        behind = rng.choice((0, 0, _spread(rng, 16, 2000)))
        return _case("llama-1b", "prompt", tokens=_spread(rng, 20, 2048), behind=behind)
    if pick < 0.50:
        return _case("llama-1b", "mixed", tokens=_spread(rng, 100, 1024), behind=_spread(rng, 16, 2000), batch=_spread(rng, 2, 48), spread=1)
    if pick < 0.58:
        return _case("llama-8b-4-layers", "decode", batch=_spread(rng, 1, 32), behind=_spread(rng, 100, 4000), spread=rng.randint(0, 1))
    if pick < 0.66:
        if rng.random() < 0.5:
            return _case("llama-1b-4-layers", "prompt", tokens=_spread(rng, 20, 600), dtype="float32")
        return _case("llama-1b-4-layers", "decode", batch=_spread(rng, 1, 16), behind=_spread(rng, 40, 600), dtype="float32")
    model = rng.choice(("radivik", "larupel", "zurolorn", "durelix"))
    if rng.random() < 0.5:
        return _case(model, "decode", batch=_spread(rng, 1, 16), behind=_spread(rng, 40, 2000), spread=rng.randint(0, 1))
    return _case(model, "prompt", tokens=_spread(rng, 60, 2048))


# ------------------------------------------------------------------ weights

def _wanted(model: str) -> dict:
    """Name -> (shape, kind of values) of the model's checkpoint."""
    import prefixserve_amd.models  # noqa: F401  (fills the registry)
    from prefixserve_amd.config.registry import architecture_of
    from prefixserve_amd.parts.model import DecoderModel

    cfg = MODELS[model][0]
    arch = architecture_of(cfg)
    wanted = DecoderModel(arch.build_spec(arch.config_cls.from_dicts(cfg, {}))).weights()
    return {name: (tuple(w.shape), w.init) for name, w in wanted.items()}


# Models with experts: the size of the token table's entries. Their sub-layers add outputs of the order of one, beside which
# entries of 0.02 would leave a stream that says little about its token (and a router that sends neighbours the same way).
EMBED_STD = {"radivik": 1.0, "larupel": 1.0, "zurolorn": 0.125, "durelix": 1.0}


def _normal(shape: tuple, name: str, device: str) -> torch.Tensor:
    seed = int.from_bytes(hashlib.sha256(name.encode()).digest()[:7], "little")
    return torch.empty(shape, dtype=torch.float32, device=device).normal_(generator=torch.Generator(device).manual_seed(seed))


def _weights(model: str, device: str = "cuda"):
    """(name, bfloat16 tensor) one by one: matrices N(0, 0.02), norms 1 + N(0, 0.1), biases, taps and sinks N(0, 0.5).

    A trained router is sure of its choice where a random one is not: the layers' routers look at the same directions, and
    every token's row of the table leans towards those of a few experts, random ones for each token (and from the number
    of groups that the router keeps), so that which experts a token uses does not hang on the last bits of a sum."""
    cfg = MODELS[model][0]
    router = next((layer["mlp"]["router"] for layer in cfg.get("layers", ()) if "router" in layer["mlp"]), None)
    wanted = _wanted(model)
    for name, (shape, init) in wanted.items():
        table = router is not None and init == "embedding"
        t = _normal(shape, f"{model}:router" if name.endswith(".router") else f"{model}:{name}", device)
        if table and name == "embed":
            looks = _normal(next(s for n, (s, _) in wanted.items() if n.endswith(".router")), f"{model}:router", device)
            groups = router.get("groups", {"count": 1, "keep": 1})
            wish = _normal((shape[0], looks.shape[0]), f"{model}:wish", device).view(shape[0], groups["count"], -1)
            top = torch.topk(wish, router["top"] // groups["keep"], -1)
            best = torch.topk(_normal((shape[0], groups["count"]), f"{model}:groups", device), groups["keep"]).indices
            lean = torch.zeros_like(wish).scatter_(2, top.indices, 1.0)
            lean *= torch.zeros(shape[0], groups["count"], device=device).scatter_(1, best, 1.0)[..., None]
            t += 0.3 * (lean.view(shape[0], -1) @ looks)
        t = 1.0 + 0.1 * t if init == "norm" else 0.1 * t if init == "offset" else 0.5 * t if init == "bias" else (EMBED_STD[model] if table else 0.02) * t
        yield name, t.to(torch.bfloat16)


def _write_model(folder: Path, model: str) -> None:
    """config.json and model.safetensors (8 bytes of header length, a JSON header, the tensors' bytes)."""
    (folder / "config.json").write_text(json.dumps(MODELS[model][0]))
    header, at = {}, 0
    for name, (shape, _) in _wanted(model).items():
        n = 2 * math.prod(shape)
        header[name] = {"dtype": "BF16", "shape": list(shape), "data_offsets": [at, at + n]}
        at += n
    head = json.dumps(header).encode()
    head += b" " * (-len(head) % 8)
    with open(folder / "model.safetensors", "wb") as f:
        f.write(len(head).to_bytes(8, "little") + head)
        for _, t in _weights(model):
            f.write(t.view(torch.int16).cpu().numpy().tobytes())


class _Loaded:
    """A model ready to step, as a server keeps it, and the parts of its pools that prepared states hold."""

    def __init__(self, model: str, dtype: str) -> None:
        from prefixserve_amd.engine.runner import ModelRunner

        _, self.pages, longest = MODELS[model]
        with tempfile.TemporaryDirectory(prefix="psamd_cases_") as folder:
            _write_model(Path(folder), model)
            self.runner = ModelRunner(folder, dtype=dtype, num_blocks=LEASES * self.pages, max_seq_len=longest, max_num_seqs=64)
        self.slots = 64 // LEASES
        self.free = list(range(LEASES))


_loaded: dict[tuple[str, str], _Loaded] = {}


class _Lease:
    """A share of a model's pages and slots, given back when the state that holds it goes."""

    def __init__(self, owner: _Loaded) -> None:
        if not owner.free:
            raise MemoryError("out of memory: every share of the model's pages is in use")
        self.owner, self.number = owner, owner.free.pop(0)

    def __del__(self) -> None:
        self.owner.free.append(self.number)


# ------------------------------------------------------------------ a step

def _requests(case: dict, seed: int) -> list[tuple[np.ndarray, int]]:
    """Every request of the step: (its tokens up to the end of the step, how many of them the step brings)."""
    rng = np.random.default_rng(seed)
    cfg = MODELS[case["model"]][0]
    vocab = cfg.get("vocab_size", cfg.get("vocab"))
    out = []
    if case["kind"] != "decode":
        out.append((case["behind"] + case["tokens"], case["tokens"]))
    for b in range(case["batch"]):
        longest = max(16, case["behind"])
        # the step's lengths belong to the case, its tokens to the seed
        before = longest if b == 0 or not case["spread"] else random.Random(f"{b} {longest}").randint(16, longest)
        out.append((before + 1, 1))
    return [(rng.integers(0, vocab, n), new) for n, new in out]


def prepare(case: dict, seed: int) -> dict:
    from prefixserve_amd import StepItem

    key = (case["model"], case["dtype"])
    if key not in _loaded:
        _loaded[key] = _Loaded(*key)
    loaded = _loaded[key]
    lease = _Lease(loaded)
    runner, first = loaded.runner, lease.number * loaded.pages
    groups = len(runner.pools.tensors)
    requests = _requests(case, seed)
    # The pages the step writes come first, side by side; those behind the earlier tokens are anywhere.
    written = [range((len(t) - new) // PAGE, -(-len(t) // PAGE)) for t, new in requests]
    step_pages = sum(len(w) for w in written)
    others = [p for p in range(first + step_pages, first + loaded.pages)]
    random.Random(seed).shuffle(others)
    for pool in runner.pools.tensors:
        pool[:, first:first + step_pages].zero_()
    items, at = [], first
    for b, ((tokens, new), pages) in enumerate(zip(requests, written)):
        table = [others.pop() for _ in range(pages.start)] + list(range(at, at + len(pages)))
        at += len(pages)
        slot = lease.number * loaded.slots + b % loaded.slots
        start = len(tokens) - new
        for p in range(0, start, 2048):
            runner.step([StepItem(f"r{b}", tokens[p:min(p + 2048, start)], p, [table] * groups, slot, ())])
        items.append(StepItem(f"r{b}", tokens[start:], start, [np.asarray(table)] * groups, slot, (new - 1,)))
    slots = slice(lease.number * loaded.slots, lease.number * loaded.slots + len(items))
    return {"runner": runner, "items": items, "lease": lease,
            "pages": [pool[:, first:first + step_pages] for pool in runner.pools.tensors],
            "states": [state[slots] for state in runner.states.values()]}


def run(state: dict) -> dict:
    logits = state["runner"].step(state["items"])
    return {"logits": logits, "pages": state["pages"], "states": state["states"]}


# ------------------------------------------------------------------ what a step cannot do without

def _lengths(case: dict) -> list[tuple[int, int]]:
    return [(len(t), new) for t, new in _requests(case, 0)]


def _runs(cfg: dict) -> list[int]:
    """The layers in the order they run."""
    loop = cfg.get("loop")
    n = list(range(len(cfg["layers"])))
    return n if not loop else n[:loop["start"]] + n[loop["start"]:loop["stop"]] * loop["times"] + n[loop["stop"]:]


def _attention_sizes(cfg: dict, i: int) -> tuple[int, int, int] | None:
    """(numbers of keys and values per position, product operations per query-key pair, window) of layer i, or None."""
    if "layers" not in cfg:
        d = cfg["head_dim"]
        return 2 * cfg["num_key_value_heads"] * d, 4 * cfg["num_attention_heads"] * d, 1 << 30
    m = cfg["layers"][i]["mixer"]
    m = m.get("left", m)
    if "kv_rank" in m:
        return m["kv_rank"] + m["rot_dim"], 2 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), 1 << 30
    if "scale" not in m:
        return None
    return m["kv_heads"] * (m["dim"] + m["vdim"]), 2 * m["heads"] * (m["dim"] + m["vdim"]), m.get("mask", {}).get("size", 1 << 30)


def work(case: dict) -> dict:
    cfg = MODELS[case["model"]][0]
    size = 2 if case["dtype"] == "bfloat16" else 4
    lengths = _lengths(case)
    tokens, rows = sum(new for _, new in lengths), len(lengths)
    runs = _runs(cfg) if "layers" in cfg else list(range(cfg["num_hidden_layers"]))
    moved = flops = 0.0
    vocab, width = cfg.get("vocab_size", cfg.get("vocab")), cfg.get("hidden_size", cfg.get("width"))
    for name, (shape, init) in _wanted(case["model"]).items():
        n = math.prod(shape)
        layer = next((int(p[1:]) if p[0] == "l" else int(p) for p in name.split(".") if p.isdigit() or (p[0] == "l" and p[1:].isdigit())), None)
        if init == "embedding" or name.endswith("embed_tokens.weight"):
            moved += min(tokens, shape[0]) * shape[1] * 2
            continue
        if layer is None:
            moved += n * size
            flops += 2.0 * n * rows if name == "head" or name == "lm_head.weight" else 0.0
            continue
        used, share, times = 1.0, 1.0, runs.count(layer)
        if "layers" in cfg and ".mlp.e" in name:
            r = cfg["layers"][layer]["mlp"]["router"]
            share = r["top"] / (r["experts"] + r.get("identity", 0))
            used = 1.0 - (1.0 - share) ** tokens
        moved += n * size * used                            # a stretch that is repeated is read once, were it kept
        if len(shape) == 2:
            flops += 2.0 * n * tokens * share * times
    if cfg.get("tie_word_embeddings") or cfg.get("architecture") == "Durelix":
        moved += vocab * width * size
        flops += 2.0 * vocab * width * rows
    for i in runs:
        att = _attention_sizes(cfg, i)
        if att is None:
            continue
        per_key, per_pair, window = att
        for length, new in lengths:
            start = length - new
            seen = sum(min(p + 1, window) for p in range(start, length))
            moved += per_key * size * (min(start, window) + new)
            flops += per_pair * seen
    moved += rows * vocab * 4
    return {"bytes": moved, "flops": flops}


def tolerance(case: dict) -> dict:
    if case["dtype"] == "float32":
        return {"rel": 3e-5, "max": 5e-4}      # 4.6e-6 off the same step in 64 bits, logits and cached keys alike
    return {"rel": 0.03, "max": 0.9}            # logits 0.004 to 0.023 off it: sixteen layers of bfloat16 products


# ------------------------------------------------------------------ the same step in 64 bits

def exact(case: dict, seed: int) -> dict | None:
    cfg = MODELS[case["model"]][0]
    w = {name: t.double() for name, t in _weights(case["model"])}
    requests = _requests(case, seed)
    forward = {"Radivik": _radivik64, "Larupel": _larupel64, "Zurolorn": _zurolorn64, "Durelix": _durelix64}.get(
        cfg.get("architecture"), _llama64)
    rows, group = [], []
    for i, (tokens, _) in enumerate(requests):              # whole sequences, about 8,192 tokens at a time
        group.append(torch.from_numpy(tokens).cuda())
        if i + 1 == len(requests) or sum(len(t) for t in group) + len(requests[i + 1][0]) > 8192:
            rows.append(forward(cfg, w, _Spans(group)))
            group = []
    return {"logits": torch.cat(rows), "pages": None, "states": None}


class _Spans:
    """Sequences back to back."""

    def __init__(self, tokens: list[torch.Tensor]) -> None:
        self.tokens = torch.cat(tokens)
        ends = np.cumsum([len(t) for t in tokens])
        self.ranges = [(int(e) - len(t), int(e)) for t, e in zip(tokens, ends)]
        self.pos = torch.cat([torch.arange(len(t), device=t.device) for t in tokens])
        self.last = torch.tensor([e - 1 for _, e in self.ranges], device=self.tokens.device)

    def each(self, f, *xs: torch.Tensor) -> torch.Tensor:
        return torch.cat([f(*(x[a:b] for x in xs)) for a, b in self.ranges])


def _unit(x: torch.Tensor, eps: float) -> torch.Tensor:
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _turn(x: torch.Tensor, angle: torch.Tensor, halves: bool = True, gain: float = 1.0) -> torch.Tensor:
    """x [n, heads, d]: the first 2 * angle.shape[1] numbers of every head, partners half of them apart or side by side."""
    half = angle.shape[1]
    c, s = (torch.cos(angle) * gain)[:, None], (torch.sin(angle) * gain)[:, None]
    out = x.clone()
    a, b = (slice(0, half), slice(half, 2 * half)) if halves else (slice(0, 2 * half, 2), slice(1, 2 * half, 2))
    out[..., a], out[..., b] = x[..., a] * c - x[..., b] * s, x[..., b] * c + x[..., a] * s
    return out


def _frequencies(dims: int, base: float) -> torch.Tensor:
    return float(base) ** (-torch.arange(0, dims, 2, dtype=torch.float64, device="cuda") / dims)


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale, window: int = 1 << 30, sink: torch.Tensor | None = None) -> torch.Tensor:
    """One sequence, [n, heads, .] each, several query heads to a key head; causal. ``scale``: a number, or one a query head."""
    n, per = q.shape[0], q.shape[1] // k.shape[1]
    back = torch.arange(n, device=q.device)[:, None] - torch.arange(n, device=q.device)[None]
    hidden = (back < 0) | (back >= window)
    out = torch.empty(n, q.shape[1], v.shape[2], dtype=q.dtype, device=q.device)
    for h in range(q.shape[1]):
        s = (q[:, h] @ k[:, h // per].T) * (scale if isinstance(scale, float) else scale[h])
        s.masked_fill_(hidden, -math.inf)
        if sink is not None:
            s = torch.cat((s, sink[h].expand(n, 1)), 1)
        out[:, h] = torch.softmax(s, -1)[:, :n] @ v[:, h // per]
    return out.reshape(n, -1)


def _mixture(h: torch.Tensor, chosen: torch.Tensor, weight: torch.Tensor, expert, experts: int) -> torch.Tensor:
    """sum over a token's choices; ``expert(e, rows, their weights)`` gives what is added."""
    out = torch.zeros_like(h)
    for e in range(experts):
        row, which = (chosen == e).nonzero(as_tuple=True)
        if len(row):
            out.index_add_(0, row, expert(e, h[row], weight[row, which][:, None]))
    return out


def _conv(u: torch.Tensor, taps: torch.Tensor) -> torch.Tensor:
    """y[t, c] = sum_j taps[c, j] u[t - (taps - 1) + j, c]; nothing in front of the sequence."""
    n, t = u.shape[0], taps.shape[1]
    padded = torch.cat((u.new_zeros(t - 1, u.shape[1]), u))
    return sum(padded[j:j + n] * taps[:, j] for j in range(t))


def _llama64(cfg: dict, w: dict, seq: _Spans) -> torch.Tensor:
    silu = torch.nn.functional.silu
    hq, hkv, d, eps = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], cfg["rms_norm_eps"]
    f, r = _frequencies(d, cfg["rope_theta"]), cfg["rope_scaling"]
    length = r["original_max_position_embeddings"] * f / (2 * math.pi)      # turns over the original context
    low, high = r["low_freq_factor"], r["high_freq_factor"]
    blend = ((length - low) / (high - low)).clamp(0, 1)
    f = f * (blend + (1 - blend) / r["factor"])
    # The angle is a product in float32, as this architecture defines its table.
    angle = (seq.pos.float()[:, None] * f.float()[None]).double()
    x = w["model.embed_tokens.weight"][seq.tokens]
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = _unit(x, eps) * w[p + "input_layernorm.weight"]
        q = _turn((h @ w[p + "self_attn.q_proj.weight"].T).view(-1, hq, d), angle)
        k = _turn((h @ w[p + "self_attn.k_proj.weight"].T).view(-1, hkv, d), angle)
        v = (h @ w[p + "self_attn.v_proj.weight"].T).view(-1, hkv, d)
        x = x + seq.each(lambda a, b, c: _attend(a, b, c, d ** -0.5), q, k, v) @ w[p + "self_attn.o_proj.weight"].T
        h = _unit(x, eps) * w[p + "post_attention_layernorm.weight"]
        x = x + (silu(h @ w[p + "mlp.gate_proj.weight"].T) * (h @ w[p + "mlp.up_proj.weight"].T)) @ w[p + "mlp.down_proj.weight"].T
    x = _unit(x[seq.last], eps) * w["model.norm.weight"]
    return x @ w["model.embed_tokens.weight" if cfg["tie_word_embeddings"] else "lm_head.weight"].T


def _radivik64(cfg: dict, w: dict, seq: _Spans) -> torch.Tensor:
    eps, x = cfg["norm"]["eps"], w["embed"][seq.tokens]
    for i, layer in enumerate(cfg["layers"]):
        m, p = layer["mixer"], f"l{i}.mix."
        dims, base, sc = m["rot"]["dims"], m["rot"]["base"], m["rot"]["scaling"]
        at = lambda turns: dims * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
        lo, hi = max(math.floor(at(sc["fast"])), 0), min(math.ceil(at(sc["slow"])), dims - 1)
        share = ((torch.arange(dims // 2, device="cuda").double() - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        f = _frequencies(dims, base)
        angle = seq.pos.double()[:, None] * (f * (1 - share) + f / sc["factor"] * share)[None]
        gain = 0.1 * math.log(sc["factor"]) + 1.0
        q, k = (_unit(_turn((x @ w[p + n].T).view(-1, m[heads], m["dim"]), angle, True, gain), eps) for n, heads in (("q", "heads"), ("k", "kv_heads")))
        v = (x @ w[p + "v"].T).view(-1, m["kv_heads"], m["vdim"])
        y = seq.each(lambda a, b, c: _attend(a, b, c, m["scale"]), q, k, v) @ w[p + "o"].T
        x = _unit(cfg["postln_alpha"] * x + y, eps) * w[f"l{i}.norm1"]
        r, limit, p = layer["mlp"]["router"], layer["mlp"]["expert"]["limit"], f"l{i}.mlp."
        weight, chosen = torch.topk(torch.sigmoid(x @ w[p + "router"].T), r["top"])

        def expert(e: int, rows: torch.Tensor, wt: torch.Tensor) -> torch.Tensor:
            g = (wt * rows @ w[f"{p}e{e}.gate"].T).clamp(max=limit)
            u = (wt * rows @ w[f"{p}e{e}.up"].T).clamp(-limit, limit)
            return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ w[f"{p}e{e}.down"].T

        x = _unit(cfg["postln_alpha"] * x + _mixture(x, chosen, weight, expert, r["experts"]), eps) * w[f"l{i}.norm2"]
    return (_unit(x[seq.last], eps) * w["final.norm"]) @ w["head"].T


def _larupel64(cfg: dict, w: dict, seq: _Spans) -> torch.Tensor:
    fn, eps, width = torch.nn.functional, cfg["norm"]["eps"], cfg["width"]
    norm = lambda x, name: fn.layer_norm(x, (width,), w[name], w[name + ".b"], eps)
    length = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)
    wave = seq.pos.double()[:, None] * 10000.0 ** (-torch.arange(0, width, 2, device="cuda").double() / width)[None]
    x = w["embed"][seq.tokens] + torch.stack((torch.sin(wave), torch.cos(wave)), -1).reshape(-1, width)
    kept: dict = {}

    def gated(q, k, v, strength, decay):
        """S <- g S, then S <- S + k (b (v - S^T k))^T, read as S^T q: all heads of one sequence, token by token."""
        s, out = v.new_zeros(v.shape[1], q.shape[2], v.shape[2]), torch.empty_like(v)
        for t in range(len(q)):
            s = s * decay[t, :, None, None]
            write = strength[t, :, None] * (v[t] - (s * k[t, :, :, None]).sum(1))
            s = s + k[t, :, :, None] * write[:, None]
            out[t] = (s * q[t, :, :, None]).sum(1)
        return out

    def general(r, k, v, d, a):
        """S <- diag(d) S - (a n)(n^T S) + k v^T with n = k / |k|, read as S^T r."""
        s, out, unit = v.new_zeros(v.shape[1], k.shape[2], v.shape[2]), torch.empty_like(v), length(k)
        for t in range(len(r)):
            taken = (s * unit[t, :, :, None]).sum(1)
            s = s * d[t, :, :, None] - (a[t] * unit[t])[:, :, None] * taken[:, None] + k[t, :, :, None] * v[t, :, None]
            out[t] = (s * r[t, :, :, None]).sum(1)
        return out

    for i, layer in enumerate(cfg["layers"]):
        m, p, h = layer["mixer"], f"l{i}.mix.", norm(x, f"l{i}.norm1")
        heads, dim = m["heads"], m["dim"]
        if layer["type"] == "delta":
            per = heads // m["kv_heads"]
            q, k, v = (fn.silu(seq.each(lambda u: _conv(u, w[p + n + ".conv"]), h @ w[p + n].T)).view(len(h), -1, dim) for n in "qkv")
            q, k = ((length(u) * f).repeat_interleave(per, 1) for u, f in ((q, dim ** -0.5), (k, 1.0)))
            decay = torch.exp(-torch.exp(w[p + "A_log"]) * fn.softplus(h @ w[p + "a"].T + w[p + "dt_bias"]))
            y = _unit(seq.each(gated, q, k, v, torch.sigmoid(h @ w[p + "b"].T), decay), eps) * w[p + "norm"]
            y = (y.reshape(len(h), -1) * fn.silu(h @ w[p + "g"].T)) @ w[p + "o"].T
        elif layer["type"] == "general_delta":
            r, k, v = ((h @ w[p + n].T).view(-1, heads, dim) for n in "rkv")
            low = torch.tanh(h @ w[p + "w1"].T) @ w[p + "w2"].T + w[p + "w0"]
            decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(low)).view(-1, heads, dim)
            rate = torch.sigmoid(h @ w[p + "a"].T + w[p + "a.b"]).view(-1, heads, dim)
            y = _unit(seq.each(general, r, k, v, decay, rate), eps).reshape(len(h), -1) * w[p + "norm"]
            y = (y * torch.sigmoid(h @ w[p + "g"].T)) @ w[p + "o"].T
        else:
            q = _unit((h @ w[p + "q"].T).view(-1, heads, dim), eps) * w[p + "q.norm"]
            if "kv_from" not in m:
                k = _unit((h @ w[p + "k"].T).view(-1, m["kv_heads"], dim), eps) * w[p + "k.norm"]
                kept[i] = k, (h @ w[p + "v"].T).view(-1, m["kv_heads"], m["vdim"])
            scale = m["scale"] * w[p + "temp"]
            y = seq.each(lambda a, b, c: _attend(a, b, c, scale), q, *kept[m.get("kv_from", i)]) @ w[p + "o"].T
        x = x + norm(y, f"l{i}.norm1b")
        h, p, f = norm(x, f"l{i}.norm2"), f"l{i}.mlp.", layer["mlp"]
        ff = lambda rows, q, act: (act(rows @ w[q + "gate"].T) * (rows @ w[q + "up"].T)) @ w[q + "down"].T
        if f["kind"] == "dense":
            y = ff(h, p, lambda z: fn.gelu(z, approximate="tanh"))
        else:
            z, chosen = torch.topk(h @ w[p + "router"].T + w[p + "router.b"], f["router"]["top"])
            y = _mixture(h, chosen, torch.softmax(z, -1), lambda e, rows, wt: wt * ff(rows, f"{p}e{e}.", fn.silu), f["router"]["experts"])
            y = y + ff(h, p + "shared.", fn.silu) * torch.sigmoid(h @ w[p + "shared.sg"].T)
        x = x + norm(y, f"l{i}.norm2b")
    return norm(x[seq.last], "final.norm") @ w["head"].T


def _in_groups(score: torch.Tensor, groups: dict, value) -> torch.Tensor:
    """Scores with those outside the best groups of neighbours taken out; ``value`` makes a group's score of its experts'."""
    per = score.view(len(score), groups["count"], -1)
    best = torch.topk(value(per), groups["keep"]).indices
    keep = torch.zeros(per.shape[:2], dtype=torch.bool, device=score.device).scatter_(1, best, True)
    return per.masked_fill(~keep[..., None], -math.inf).reshape(score.shape)


def _zurolorn64(cfg: dict, w: dict, seq: _Spans) -> torch.Tensor:
    eps, x, opened = cfg["norm"]["eps"], w["embed"][seq.tokens] * cfg["embedding"]["scale"], 0
    for i in _runs(cfg):
        layer = cfg["layers"][i]
        m, p = layer["mixer"], f"l{i}.mix."
        if i == cfg["loop"]["start"]:
            x, opened = x + w["loop.step"][opened], opened + 1
        h = _unit(x, eps) * w[f"l{i}.norm1"]
        heads, d, rank = m["heads"], m["dim"], m["kv_rank"]
        through = _unit(h @ w[p + "dq"].T, eps) * w[p + "dq.norm"] @ w[p + "uq"].T if "q_rank" in m else h @ w[p + "q"].T
        q, down = through.view(len(h), heads, -1), h @ w[p + "dkv"].T
        angle, halves = seq.pos.double()[:, None] * _frequencies(m["rot_dim"], m["rot"]["base"])[None], "q_rank" not in m
        c = _unit(down[:, :rank], eps) * w[p + "dkv.norm"]
        shared = _turn(down[:, None, rank:], angle, halves).expand(-1, heads, -1)
        q = torch.cat((q[..., :d], _turn(q[..., d:], angle, halves)), -1)
        k = torch.cat(((c @ w[p + "uk"].T).view(len(h), heads, d), shared), -1)
        v = (c @ w[p + "uv"].T).view(len(h), heads, m["vdim"])
        y = seq.each(lambda a, b, e: _attend(a, b, e, float(m["scale"])), q, k, v)
        if "g" in {n[len(p):] for n in w if n.startswith(p)}:
            y = y * torch.sigmoid(h @ w[p + "g"].T)
        x = x + w[f"l{i}.ls1"] * (y @ w[p + "o"].T)
        h, p, r = _unit(x, eps) * w[f"l{i}.norm2"], f"l{i}.mlp.", layer["mlp"]["router"]
        score = torch.sigmoid(h @ w[p + "router"].T)
        chosen = torch.topk(_in_groups(score, r["groups"], lambda s: torch.topk(s, 2).values.sum(-1)), r["top"]).indices
        expert = lambda e, rows, wt: wt * (torch.relu(rows @ w[f"{p}e{e}.up"].T).square() @ w[f"{p}e{e}.down"].T)
        x = x + w[f"l{i}.ls2"] * _mixture(h, chosen, score.gather(1, chosen) * r["scale"], expert, r["experts"])
    return (_unit(x[seq.last], eps) * w["final.norm"]) @ w["head"].T * cfg["logit_scale"]


def _durelix64(cfg: dict, w: dict, seq: _Spans) -> torch.Tensor:
    silu, eps, b = torch.nn.functional.silu, cfg["norm"]["eps"], cfg["embedding"]["bigram"]
    before = torch.roll(seq.tokens, 1)
    row = torch.where(seq.pos == 0, b["buckets"], (before * b["mul_prev"] + seq.tokens * b["mul_cur"]) % b["buckets"])
    x = w["embed"][seq.tokens] + w["bigram"][row]

    def retained(q, k, v, decay):
        """sum over j <= i of decay^(i - j) (q_i . k_j) v_j, one sequence."""
        n, out = len(q), torch.empty_like(v)
        back = (torch.arange(n, device=q.device)[:, None] - torch.arange(n, device=q.device)[None]).double()
        for a in range(q.shape[1]):
            share = torch.where(back >= 0, decay[a] ** back.clamp(min=0), 0.0)
            out[:, a] = ((q[:, a] @ k[:, a].T) * share) @ v[:, a]
        return out

    for i, layer in enumerate(cfg["layers"]):
        m, p = layer["mixer"]["left"], f"l{i}.mix.left."
        q, k, v = (seq.each(lambda u: _conv(u, w[p + n + ".conv"]), x @ w[p + n].T).view(len(x), -1, m["dim"]) for n in "qkv")
        angle = seq.pos.double()[:, None] * _frequencies(m["dim"], m["rot"]["base"])[None]
        q, k = (_turn(_unit(u, eps) * w[p + n + ".norm"], angle, False) for u, n in ((q, "q"), (k, "k")))
        left = seq.each(lambda a, c, e: _attend(a, c, e, float(m["scale"]), m["mask"]["size"], w[p + "sink"]), q, k, v)
        left = (left * torch.sigmoid(x @ w[p + "g"].T)) @ w[p + "o"].T
        m, p = layer["mixer"]["right"], f"l{i}.mix.right."
        q, k, v = ((x @ w[p + n].T).view(len(x), m["heads"], -1) for n in "qkv")
        angle = seq.pos.double()[:, None] * _frequencies(m["dim"], m["rot"]["base"])[None]
        q, k = _turn(q, angle), _turn(k, angle) * m["dim"] ** -0.5
        right = _unit(seq.each(lambda a, c, e: retained(a, c, e, m["decay"]), q, k, v), eps).reshape(len(x), -1)
        right = (right * silu(x @ w[p + "g"].T)) @ w[p + "o"].T
        y = 0.5 * (_unit(left, eps) * w[f"l{i}.mix.left.out"] + _unit(right, eps) * w[f"l{i}.mix.right.out"])
        x = x + _unit(y, eps) * w[f"l{i}.norm1"]
        p, f = f"l{i}.mlp.", layer["mlp"]
        if f["kind"] == "dense":
            y = torch.relu(x @ w[p + "up"].T).square() @ w[p + "down"].T
        else:
            r, score = f["router"], torch.softmax(x @ w[p + "router"].T, -1)
            chosen = torch.topk(_in_groups(score + w[p + "correction"], r["groups"], lambda s: s.amax(-1)), r["top"]).indices

            def expert(e: int, rows: torch.Tensor, wt: torch.Tensor) -> torch.Tensor:
                if e >= r["experts"]:
                    return wt * rows
                return wt * ((silu(rows @ w[f"{p}e{e}.gate"].T) * (rows @ w[f"{p}e{e}.up"].T)) @ w[f"{p}e{e}.down"].T)

            y = _mixture(x, chosen, score.gather(1, chosen), expert, r["experts"] + r["identity"])
        x = x + _unit(y, eps) * w[f"l{i}.norm2"]
    return (_unit(x[seq.last], eps) * w["final.norm"]) @ w["embed"].T
