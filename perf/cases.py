"""The steps that users of this engine run, as cases for measuring them.

A case is one pass of an engine over a batch: requests that decode one token each (`decoding`, the longest with `context`
tokens before it), a portion of a prompt (`portion` tokens behind `behind` that were read before), or both in one mixed step;
with `new_tokens` the prompts are read and then so many tokens decoded, from admission to release.  Layer sizes are those of
`benchmarks/shapes.py`; the weights are random, of the size that keeps every layer's contribution at order one, and rounded to
bfloat16 as checkpoints are.  `exact()` recomputes whole sequences in 64 bits with plain tensor operations.
"""

from __future__ import annotations

import math
import zlib

import torch

from llm_runtime_study_amd import Engine, SamplingConfig
from llm_runtime_study_amd.benchmarks.shapes import SHAPES, napizen_like, nobodra_like
from llm_runtime_study_amd.config import config_from_dict, spec_for
from llm_runtime_study_amd.engine.loading import reserve_for, resolve_device, resolve_dtype
from llm_runtime_study_amd.engine.step import StepEntry
from llm_runtime_study_amd.models import DecoderModel
from llm_runtime_study_amd.parts import LazyTensors
from llm_runtime_study_amd.sampling import Sampler, SamplingRow

PAGE_SIZE = 16
STEP_TOKENS = 2048          # the engine's default budget of a step
EXACT_FLOPS = 4e14          # a 64-bit recomputation of more than this takes too long


def _case(design="qwen3", shape="8b", layers=None, dtype="bfloat16", decoding=0, context=0, portion=0, behind=0, new_tokens=0, sampled=False, **name):
    layers = SHAPES[shape]["num_hidden_layers"] if layers is None else layers
    return dict(design=design, shape=shape, layers=layers, dtype=dtype, decoding=decoding, context=context, portion=portion, behind=behind,
                new_tokens=new_tokens, sampled=sampled, **name)


def listed() -> list[dict]:
    return [
        # one user's chat with the smallest model: a decode step is nearly all launches and small products
        _case(name="decode-0.6b-b1", shape="0.6b", decoding=1, context=509),
        # the reference's serving workload (prompts of 509 tokens, batch of 16), requests at different lengths
        _case(name="decode-0.6b-b16", shape="0.6b", decoding=16, context=636),
        # the headline: eight requests at 2,048 tokens of context
        _case(name="decode-8b-b8", shape="8b", decoding=8, context=2048),
        # a full serving batch at mixed lengths
        _case(name="decode-8b-b64", shape="8b", decoding=64, context=2048),
        # a whole prompt in one step, the second headline
        _case(name="prompt-8b-2048", shape="8b", portion=2048),
        # continuous batching under a budget of 512 tokens: decoding requests beside the second portion of a prompt
        _case(name="mixed-4b-512", shape="4b", decoding=24, context=1500, portion=488, behind=488),
        # the eighth portion of a long document
        _case(name="portion-1.7b-16k", shape="1.7b", portion=2048, behind=14336),
        # the float32 mode: a prompt of the reference's length ...
        _case(name="float32-prompt-509", shape="0.6b", dtype="float32", portion=509),
        # ... and a batch that draws its tokens with top-k and top-p
        _case(name="float32-decode-b8", shape="0.6b", dtype="float32", decoding=8, context=509, sampled=True),
        # delta-rule layers, sliding-window attention and routed experts: a prompt, one layer of attention to three of the delta rule
        _case(name="nobodra-prompt-2048", design="nobodra", shape="8b", layers=4, portion=2048),
        # ... and eight short prompts answered from admission to release
        _case(name="nobodra-chat-b8", design="nobodra", shape="8b", layers=4, decoding=8, context=77, new_tokens=8),
        # latent attention and gated experts: decoding over long contexts
        _case(name="napizen-decode-b16", design="napizen", shape="8b", layers=4, decoding=16, context=4096),
    ]


def draw(rng) -> dict:
    def spread(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    kind = rng.choice(("decode", "decode", "prompt", "mixed", "portion", "float32-prompt", "float32-decode", "nobodra-prompt", "nobodra-chat", "napizen-decode"))
    if kind == "decode":
        batch = spread(1, 64)
        return _case(shape=rng.choice(("0.6b", "1.7b", "4b", "8b")), decoding=batch, context=spread(64, 4096 if batch <= 32 else 2048))
    if kind == "prompt":
        return _case(shape=rng.choice(("0.6b", "1.7b", "4b", "8b")), portion=spread(32, 2047))
    if kind == "mixed":
        batch = spread(1, 64)
        return _case(shape=rng.choice(("0.6b", "1.7b", "4b")), decoding=batch, context=spread(128, 2048), portion=spread(64, 512), behind=rng.choice((0, spread(64, 2048))))
    if kind == "portion":
        return _case(shape=rng.choice(("0.6b", "1.7b")), portion=spread(256, 2048), behind=spread(2048, 14336))
    if kind == "float32-prompt":
        return _case(shape="0.6b", dtype="float32", portion=spread(32, 1024))
    if kind == "float32-decode":
        return _case(shape="0.6b", dtype="float32", decoding=spread(1, 16), context=spread(64, 1024), sampled=True)
    if kind == "nobodra-prompt":
        return _case(design="nobodra", shape=rng.choice(("4b", "8b")), layers=4, portion=spread(64, 2047))
    if kind == "nobodra-chat":
        return _case(design="nobodra", shape=rng.choice(("4b", "8b")), layers=4, decoding=spread(1, 16), context=spread(16, 128), new_tokens=8)
    return _case(design="napizen", shape=rng.choice(("4b", "8b")), layers=4, decoding=spread(4, 32), context=spread(256, 4096))


# ----------------------------------------------------------------------- inputs
def _raw(case) -> dict:
    """The content of config.json."""
    shape = SHAPES[case["shape"]]
    if case["design"] == "nobodra":
        return nobodra_like(shape, case["layers"])
    if case["design"] == "napizen":
        return napizen_like(shape, case["layers"])
    return dict(shape, num_hidden_layers=case["layers"])


def _shapes(case) -> dict:
    """Every checkpoint tensor's name and shape."""
    raw = _raw(case)
    if case["design"] == "qwen3":
        h, i, d, vocab = raw["hidden_size"], raw["intermediate_size"], raw["head_dim"], raw["vocab_size"]
        q, kv = raw["num_attention_heads"] * d, raw["num_key_value_heads"] * d
        out = {"model.embed_tokens.weight": (vocab, h), "model.norm.weight": (h,)}
        if not raw["tie_word_embeddings"]:
            out["lm_head.weight"] = (vocab, h)
        layer = {"input_layernorm": (h,), "post_attention_layernorm": (h,), "self_attn.q_norm": (d,), "self_attn.k_norm": (d,), "self_attn.q_proj": (q, h),
                 "self_attn.k_proj": (kv, h), "self_attn.v_proj": (kv, h), "self_attn.o_proj": (h, q), "mlp.gate_proj": (i, h), "mlp.up_proj": (i, h),
                 "mlp.down_proj": (h, i)}
        out.update({f"model.layers.{index}.{name}.weight": size for index in range(case["layers"]) for name, size in layer.items()})
        return out
    w, vocab = raw["width"], raw["vocab"]
    out = {"embed": (vocab, w), "head": (vocab, w), "final.norm": (w,)}
    for index, entry in enumerate(raw["layers"]):
        m, mlp = entry["mixer"], entry["mlp"]
        heads, d, e = m["heads"], m["dim"], m["vdim"]
        layer = {"norm1": (w,), "norm2": (w,), "mix.o": (w, heads * e)}
        if entry["type"] == "attention":
            layer |= {"mix.q": (heads * d, w), "mix.k": (m["kv_heads"] * d, w), "mix.q.norm": (d,), "mix.k.norm": (d,)}
        elif entry["type"] == "delta":
            kv = m["kv_heads"] * d
            layer |= {"mix.q": (kv, w), "mix.k": (kv, w), "mix.v": (heads * e, w), "mix.g": (heads * e, w), "mix.b": (heads, w), "mix.a": (heads, w),
                      "mix.q.conv": (kv, m["conv"]), "mix.k.conv": (kv, m["conv"]), "mix.v.conv": (heads * e, m["conv"]), "mix.A_log": (heads,),
                      "mix.dt_bias": (heads,), "mix.norm": (e,)}
        else:
            c, r = m["kv_rank"], m["rot_dim"]
            layer |= {"mix.q": (heads * (d + r), w), "mix.dkv": (c + r, w), "mix.dkv.norm": (c,), "mix.uk": (heads * d, c), "mix.uv": (heads * e, c),
                      "mix.sink": (heads,), "mix.g": (heads, w)}
        if mlp["kind"] == "dense":
            layer |= {"mlp.gate": (mlp["ff"], w), "mlp.up": (mlp["ff"], w), "mlp.down": (w, mlp["ff"])}
        else:
            experts, ff = mlp["router"]["experts"], mlp["expert"]["ff"]
            layer |= {"mlp.router": (experts, w), **({"mlp.router.b": (experts,)} if case["design"] == "nobodra" else {"mlp.correction": (experts,)})}
            matrices = {"up": (ff, w), "down": (w, ff)} if case["design"] == "nobodra" else {"gate": (ff, w), "up": (ff, w), "down": (w, ff)}
            layer |= {f"mlp.e{j}.{name}": size for j in range(experts) for name, size in matrices.items()}
        out.update({f"l{index}.{name}": size for name, size in layer.items()})
    return out


def _tensor(case, seed: int, name: str, shape: tuple, device) -> torch.Tensor:
    """A checkpoint tensor in bfloat16: a matrix N(0, 1 / fan-in), the embedding N(0, 1), a norm's weight 1 + N(0, 0.1) (Nobodra
    stores it about zero), other vectors N(0, 0.1).  The router whose choices are weighted by a softmax is three times as large:
    a trained one is sure of its first choices."""
    generator = torch.Generator(device=device).manual_seed(zlib.crc32(f"{seed} {name}".encode()))
    t = torch.randn(shape, generator=generator, device=device, dtype=torch.bfloat16)
    if len(shape) == 2:
        if "embed" in name and not _raw(case).get("tie_word_embeddings"):
            return t
        return t.mul_((3.0 if case["design"] == "nobodra" and name.endswith("router") else 1.0) * shape[1] ** -0.5)
    t.mul_(0.1)
    about_zero = case["design"] == "nobodra" and name.split(".")[-1] in ("norm1", "norm2") or name == "final.norm" and case["design"] == "nobodra"
    return t if about_zero or "norm" not in name else t.add_(1.0)


def _sequences(case, seed: int) -> tuple[list, list]:
    """(the decoding requests' tokens up to and with those of the pass, the prompt's up to the portion's end)."""
    shape = SHAPES[case["shape"]]
    generator = torch.Generator().manual_seed(seed)
    count, context = case["decoding"], case["context"]
    # different lengths: from the longest down to a half of it, in no order; eight and fewer are nearly alike
    lengths = [context - (i * 97) % max(1, context // (2 if count > 8 else 32)) for i in range(count)]
    extra = case["new_tokens"] or 1
    decoding = [torch.randint(0, shape["vocab_size"], (n + extra,), generator=generator).tolist() for n in lengths]
    prompt = torch.randint(0, shape["vocab_size"], (case["behind"] + case["portion"],), generator=generator).tolist()
    return decoding, prompt


def _wanted(case, prompt) -> list:
    """Places of a prompt whose logits are asked for: the last; a model that chooses experts is asked for a few, since a near tie
    at one token may go either way."""
    return list(range(max(0, len(prompt) - (64 if case["design"] == "nobodra" else 1)), len(prompt)))


class _State:
    pass


_stream = None


def _one_stream(device):
    """The stream that every engine of this process runs on: their passes follow each other, as on a GPU of one engine."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream(device)
    return _stream


def prepare(case, seed):
    """An engine with its weights, and the requests whose earlier tokens were read."""
    config = config_from_dict(_raw(case))
    device, dtype = resolve_device(), resolve_dtype(case["dtype"])
    decoding, prompt = _sequences(case, seed)
    longest = max([len(ids) for ids in decoding] + [len(prompt)])
    max_seq_len = -(-(longest + 1) // 256) * 256
    requests = len(decoding) + (1 if prompt else 0)
    pages = sum(-(-(len(ids) + 1) // PAGE_SIZE) for ids in decoding + [prompt])
    shapes = _shapes(case)
    reserve_for(config, dtype, device, PAGE_SIZE, pages)
    model = DecoderModel(spec_for(config))
    model.bind(LazyTensors(list(shapes), lambda name: _tensor(case, seed, name, shapes[name], device)), dtype)
    s = _State()
    s.engine = Engine(config, model, device=device, dtype=dtype, max_seq_len=max_seq_len, max_batch_size=requests, num_pages=pages,
                      max_num_batched_tokens=STEP_TOKENS)
    s.engine.stream = _one_stream(device)
    s.new_tokens, s.decoding, s.prompt, s.behind = case["new_tokens"], decoding, prompt, case["behind"]
    s.wanted = _wanted(case, prompt)
    s.sampler = Sampler(device) if case["sampled"] else None
    s.rows = [SamplingRow(SamplingConfig(temperature=0.8, top_k=50, top_p=0.9, seed=seed + i), seed + i, 1) for i in range(len(decoding))]
    s.entries = []
    if not s.new_tokens:
        # requests that decode, and a prompt of which earlier portions were read: they stay between passes
        earlier = [ids[:-1] for ids in decoding]
        caches = [s.engine.allocate_cache(len(ids) + 1) for ids in earlier]
        held = [(cache, ids[-1:]) for cache, ids in zip(caches, decoding)]
        if s.behind:
            caches.append(s.engine.allocate_cache(len(prompt)))
            earlier.append(prompt[:s.behind])
            held.append((caches[-1], prompt[s.behind:]))
        _read(s.engine, caches, earlier)
        s.entries = [StepEntry(cache, ids, [len(ids) - 1]) for cache, ids in held]
        s.lengths = [entry.cache.length for entry in s.entries]
    return s


def _read(engine, caches, sequences) -> None:
    """Prompts read in steps of the engine's budget, as a scheduler cuts them."""
    with torch.cuda.stream(engine.stream):
        step, room = [], STEP_TOKENS
        for cache, ids in zip(caches, sequences):
            at = 0
            while at < len(ids):
                piece = ids[at:at + room]
                step.append(StepEntry(cache, piece))
                at, room = at + len(piece), room - len(piece)
                if room == 0:
                    engine.runner.step(step, keep_states=False)
                    step, room = [], STEP_TOKENS
        if step:
            engine.runner.step(step, keep_states=False)


def run(state):
    engine, runner = state.engine, state.engine.runner
    with torch.cuda.stream(engine.stream):
        if state.new_tokens:
            return _chat(state)
        entries, fresh = state.entries, None
        if state.prompt and not state.behind:
            fresh = engine.allocate_cache(len(state.prompt))
            entries = entries + [StepEntry(fresh, state.prompt, state.wanted)]
        logits = runner.step(entries, keep_states=False)
        if fresh is not None:
            engine.release_cache(fresh)
        for entry, length in zip(state.entries, state.lengths):       # the pass may be made again
            engine.cache_manager.rollback(entry.cache, length)
        if state.sampler is None:
            return logits
        kept = logits.clone()                                          # the sampler filters in place
        return {"logits": kept, "tokens": torch.tensor(state.sampler.choose(logits, state.rows))}


def _chat(state):
    """Prompts read in one step, then `new_tokens` given tokens decoded; the logits of every step."""
    engine, steps = state.engine, state.new_tokens
    caches = [engine.allocate_cache(len(ids)) for ids in state.decoding]
    cut = [len(ids) - steps for ids in state.decoding]
    kept = [engine.runner.step([StepEntry(cache, ids[:n], [n - 1]) for cache, ids, n in zip(caches, state.decoding, cut)], keep_states=False).clone()]
    for i in range(steps):
        entries = [StepEntry(cache, [ids[n + i]], [0]) for cache, ids, n in zip(caches, state.decoding, cut)]
        kept.append(engine.runner.step(entries, keep_states=False).clone())
    for cache in caches:
        engine.release_cache(cache)
    return torch.stack(kept)


# --------------------------------------------------------------------- measures
def _steps_of(case) -> tuple[list, int]:
    """(tokens and earlier tokens of every entry of every step of a pass, the rows of logits)."""
    decoding, prompt = _sequences(case, 0)
    if case["new_tokens"]:
        n = case["new_tokens"]
        steps = [[(len(ids) - n, 0) for ids in decoding]] + [[(1, len(ids) - n + i) for ids in decoding] for i in range(n)]
        return steps, len(decoding) * (n + 1)
    step = [(1, len(ids) - 1) for ids in decoding] + ([(case["portion"], case["behind"])] if prompt else [])
    return [step], len(decoding) + len(_wanted(case, prompt))


def work(case) -> dict:
    """Every weight in use and every earlier key and value read once a step, keys and values of the step and logits written once."""
    raw, item = _raw(case), 2 if case["dtype"] == "bfloat16" else 4
    sizes = {name: math.prod(shape) for name, shape in _shapes(case).items()}
    tables = [name for name in sizes if "embed" in name]
    head = next((name for name in sizes if "head" in name), tables[0])
    vocab = SHAPES[case["shape"]]["vocab_size"]
    experts, routed = sum(n for name, n in sizes.items() if ".mlp.e" in name), 1.0
    dense = sum(n for name, n in sizes.items() if name not in tables + [head] and ".mlp.e" not in name)
    if experts:
        router = next(layer["mlp"]["router"] for layer in raw["layers"] if layer["mlp"]["kind"] == "moe")
        routed = router["top"] / router["experts"]
    moved = flops = 0.0
    steps, rows = _steps_of(case)
    for step in steps:
        tokens = sum(n for n, _ in step)
        used = dense + experts * (1.0 - (1.0 - routed) ** tokens)
        moved += (used + sizes[head]) * item + tokens * SHAPES[case["shape"]]["hidden_size"] * item
        flops += 2.0 * tokens * (dense + experts * routed)
        for layer in range(case["layers"]):
            kind = "qwen3" if case["design"] == "qwen3" else raw["layers"][layer]["type"]
            m = None if kind == "qwen3" else raw["layers"][layer]["mixer"]
            for n, before in step:
                pairs = n * before + n * (n + 1) / 2
                if kind == "qwen3":
                    heads, kept, per_pair = raw["num_attention_heads"], 2 * raw["num_key_value_heads"] * raw["head_dim"], 4 * raw["head_dim"]
                elif kind == "attention":
                    heads, kept, per_pair = m["heads"], 2 * m["kv_heads"] * m["dim"], 4 * m["dim"]
                elif kind == "latent_attention":
                    heads, kept, per_pair = m["heads"], m["kv_rank"] + m["rot_dim"], 2 * (m["dim"] + m["rot_dim"] + m["vdim"])
                else:      # the state of every head read and written, four operations a number a token
                    state = m["heads"] * m["dim"] * m["vdim"]
                    moved, flops = moved + 2 * 4 * state, flops + 6.0 * n * state
                    continue
                moved += (n + before) * kept * item
                flops += heads * per_pair * pairs
    return {"bytes": moved + 4 * rows * vocab, "flops": flops + 2.0 * rows * sizes[head]}


def tolerance(case) -> dict:
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 5e-4, "differ": 0.0}
    return {"rel": 0.03, "max": 0.5}


# ------------------------------------------------------------- in 64 bits
def exact(case, seed):
    sizes = {name: math.prod(shape) for name, shape in _shapes(case).items()}
    decoding, prompt = _sequences(case, seed)
    sequences = decoding + ([prompt] if prompt else [])
    total = sum(len(ids) for ids in sequences)
    if 2.0 * total * sum(n for name, n in sizes.items() if "embed" not in name and "head" not in name) > EXACT_FLOPS:
        return None
    wanted = []
    for i, ids in enumerate(sequences):
        n = case["new_tokens"]
        wanted.append(list(range(len(ids) - n - 1, len(ids))) if n else _wanted(case, ids) if i >= len(decoding) else [len(ids) - 1])
    logits = _logits(case, seed, sequences, wanted)
    if case["new_tokens"]:
        return torch.stack(logits, 1)
    out = torch.cat(logits)
    return {"logits": out, "tokens": None} if case["sampled"] else out


def _logits(case, seed, sequences, wanted) -> list:
    device, raw, shapes = torch.device("cuda"), _raw(case), _shapes(case)

    def weight(name):
        return _tensor(case, seed, name, shapes[name], device).double()

    forward = {"qwen3": _qwen3, "nobodra": _nobodra, "napizen": _napizen}[case["design"]]
    lengths = [len(ids) for ids in sequences]
    x = forward(raw, weight, torch.tensor([t for ids in sequences for t in ids], device=device), lengths)
    head = weight("lm_head.weight" if "lm_head.weight" in shapes else "head" if "head" in shapes else "model.embed_tokens.weight")
    out = []
    for rows, places in zip(x.split(lengths), wanted):
        y = rows[places] @ head.T
        cap = raw.get("logit_softcap")
        out.append(y if cap is None else cap * torch.tanh(y / cap))
    return out


def _rms(x, eps):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _turn(x, rates, factor=1.0, neighbours=False):
    """x [n, ..., dims] rotated by the position: dim i paired with i + dims / 2, or with the one beside it."""
    half = x.shape[-1] // 2
    angle = torch.arange(x.shape[0], device=x.device, dtype=x.dtype)[:, None] * torch.tensor(rates, device=x.device, dtype=x.dtype)
    angle = angle.view(x.shape[0], *[1] * (x.dim() - 2), half)
    c, s = angle.cos() * factor, angle.sin() * factor
    if neighbours:
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack((a * c - b * s, b * c + a * s), -1).flatten(-2)
    a, b = x[..., :half], x[..., half:]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _causal(q, k, v, scale, window=None, sink=None):
    """q [heads, n, d], k [groups, n, d], v [groups, n, e] -> [n, heads, e]; sink [heads]: one more score without a value."""
    n, repeats = q.shape[1], q.shape[0] // k.shape[0]
    k, v = k.repeat_interleave(repeats, 0), v.repeat_interleave(repeats, 0)
    at, out = torch.arange(n, device=q.device), []
    for first in range(0, n, 512):
        rows = at[first:first + 512]
        scores = torch.matmul(q[:, first:first + 512], k[:, :first + 512].transpose(1, 2).contiguous()) * scale
        far = rows[:, None] - at[None, :first + 512]
        scores = scores.masked_fill((far < 0) if window is None else (far < 0) | (far >= window), -math.inf)
        if sink is not None:
            scores = torch.cat((scores, sink[:, None, None].expand(-1, len(rows), 1)), -1)
        share = torch.softmax(scores, -1)
        out.append(torch.matmul(share if sink is None else share[..., :-1], v[:, :first + 512]))
    return torch.cat(out, 1).transpose(0, 1)


def _qwen3(raw, weight, ids, lengths):
    eps, d, heads, groups = raw["rms_norm_eps"], raw["head_dim"], raw["num_attention_heads"], raw["num_key_value_heads"]
    rates = [raw["rope_theta"] ** (-2.0 * i / d) for i in range(d // 2)]
    x = weight("model.embed_tokens.weight")[ids]
    for layer in range(raw["num_hidden_layers"]):
        def w(name):
            return weight(f"model.layers.{layer}.{name}.weight")

        u = _rms(x, eps) * w("input_layernorm")
        q, k, v = ((u @ w(f"self_attn.{name}_proj").T).view(len(ids), -1, d) for name in "qkv")
        q, k = _rms(q, eps) * w("self_attn.q_norm"), _rms(k, eps) * w("self_attn.k_norm")
        mixed = [_causal(_turn(a, rates).transpose(0, 1), _turn(b, rates).transpose(0, 1), c.transpose(0, 1), d ** -0.5)
                 for a, b, c in zip(q.split(lengths), k.split(lengths), v.split(lengths))]
        x = x + torch.cat(mixed).reshape(len(ids), heads * d) @ w("self_attn.o_proj").T
        u = _rms(x, eps) * w("post_attention_layernorm")
        x = x + (torch.nn.functional.silu(u @ w("mlp.gate_proj").T) * (u @ w("mlp.up_proj").T)) @ w("mlp.down_proj").T
    return _rms(x, eps) * weight("model.norm.weight")


def _nobodra(raw, weight, ids, lengths):
    eps = raw["norm"]["eps"]
    x = weight("embed")[ids]
    for index, layer in enumerate(raw["layers"]):
        def w(name):
            return weight(f"l{index}.{name}")

        m = layer["mixer"]
        heads, groups, d, e = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        if layer["type"] == "attention":
            dims = m["rot"]["dims"]
            rates = [m["rot"]["base"] ** (-2.0 * i / dims) for i in range(dims // 2)]
            q, k = (x @ w("mix.q").T).view(-1, heads, d), (x @ w("mix.k").T).view(-1, groups, d)
            mixed = []
            for a, b in zip(q.split(lengths), k.split(lengths)):
                turned = [torch.cat((_turn(t[..., :dims], rates), t[..., dims:]), -1).transpose(0, 1)
                          for t in (_rms(a, eps) * w("mix.q.norm"), _rms(b, eps) * w("mix.k.norm"))]
                mixed.append(_causal(*turned, b.transpose(0, 1), m["scale"], m["mask"]["size"]))
        else:
            silu = torch.nn.functional.silu
            step, gate = torch.sigmoid(x @ w("mix.b").T), silu(x @ w("mix.g").T).view(-1, heads, e)
            decay = torch.exp(-torch.exp(w("mix.A_log")) * torch.nn.functional.softplus(x @ w("mix.a").T + w("mix.dt_bias")))
            projected, mixed = [], []
            for name in "qkv":
                y, taps = x @ w(f"mix.{name}").T, w(f"mix.{name}.conv")
                padded = [torch.nn.functional.pad(rows, (0, 0, taps.shape[1] - 1, 0)) for rows in y.split(lengths)]
                projected.append([silu(sum(taps[:, j] * rows[j:j + n] for j in range(taps.shape[1]))) for rows, n in zip(padded, lengths)])
            for q, k, v, b, a in zip(*projected, step.split(lengths), decay.split(lengths)):
                q, k = (t.view(len(t), groups, d) / torch.sqrt(t.view(len(t), groups, d).pow(2).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
                q, k, v = q.repeat_interleave(heads // groups, 1) * d ** -0.5, k.repeat_interleave(heads // groups, 1), v.view(len(v), heads, e)
                memory, out = torch.zeros(heads, d, e, dtype=x.dtype, device=x.device), []
                for t in range(len(v)):
                    memory = memory * a[t][:, None, None]
                    correction = b[t][:, None] * (v[t] - (memory * k[t][:, :, None]).sum(1))
                    memory = memory + k[t][:, :, None] * correction[:, None]
                    out.append((memory * q[t][:, :, None]).sum(1))
                mixed.append(torch.stack(out))
        mixed = torch.cat(mixed)
        if layer["type"] == "delta":
            mixed = _rms(mixed, eps) * w("mix.norm") * gate
        x = x + _rms(mixed.flatten(1) @ w("mix.o").T, eps) * (1.0 + w("norm1"))
        router = x @ w("mlp.router").T + w("mlp.router.b")
        best, chosen = router.topk(layer["mlp"]["router"]["top"], -1)
        fed = _experts(x, w, chosen, torch.softmax(best, -1), layer["mlp"]["router"]["experts"], lambda u, part: torch.relu(u @ part("up").T).pow(2))
        x = x + _rms(fed, eps) * (1.0 + w("norm2"))
    return _rms(x, eps) * (1.0 + weight("final.norm"))


def _experts(x, w, chosen, shares, experts, inner):
    out = torch.zeros_like(x)
    for j in range(experts):
        rows, place = (chosen == j).nonzero(as_tuple=True)
        if len(rows):
            def part(name):
                return w(f"mlp.e{j}.{name}")

            out[rows] += shares[rows, place][:, None] * (inner(x[rows], part) @ part("down").T)
    return out


def _napizen(raw, weight, ids, lengths):
    eps, alpha = raw["norm"]["eps"], raw["postln_alpha"]

    def norm(x, factor):
        off = x - x.mean(-1, keepdim=True)
        return _rms(off, eps) * factor

    x = weight("embed")[ids] * raw["embedding"]["scale"]
    for index, layer in enumerate(raw["layers"]):
        def w(name):
            return weight(f"l{index}.{name}")

        m, mlp = layer["mixer"], layer["mlp"]
        heads, d, r, e, c = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        rates, factor = _stretched(m["rot"])
        q, down, gate = (x @ w("mix.q").T).view(-1, heads, d + r), x @ w("mix.dkv").T, torch.sigmoid(x @ w("mix.g").T)
        latent = _rms(down[:, :c], eps) * w("mix.dkv.norm")
        uk, uv = w("mix.uk"), w("mix.uv")
        mixed = []
        for a, plain, shared in zip(q.split(lengths), latent.split(lengths), down[:, c:].split(lengths)):
            keys = (plain @ uk.T).view(-1, heads, d)
            turned = _turn(shared, rates, factor, True)[:, None].expand(-1, heads, -1)
            query = torch.cat((a[..., :d], _turn(a[..., d:], rates, factor, True)), -1)
            mixed.append(_causal(query.transpose(0, 1), torch.cat((keys, turned), -1).transpose(0, 1), (plain @ uv.T).view(-1, heads, e).transpose(0, 1),
                                 m["scale"], sink=w("mix.sink")))
        mixed = torch.cat(mixed) * gate[:, :, None]
        x = norm(alpha * x + mixed.flatten(1) @ w("mix.o").T, w("norm1"))

        def inner(u, part):
            return torch.nn.functional.silu(u @ part("gate").T) * (u @ part("up").T)

        if mlp["kind"] == "dense":
            y = inner(x, lambda name: w(f"mlp.{name}")) @ w("mlp.down").T
        else:
            router = mlp["router"]
            score = torch.sigmoid(x @ w("mlp.router").T)
            choice = (score + w("mlp.correction")).view(len(x), router["groups"]["count"], -1)
            kept = choice.topk(2, -1).values.sum(-1).topk(router["groups"]["keep"], -1).indices
            allowed = torch.zeros(choice.shape[:2], dtype=torch.bool, device=x.device).scatter_(1, kept, True)
            chosen = choice.masked_fill(~allowed[:, :, None], -math.inf).flatten(1).topk(router["top"], -1).indices
            shares = score.gather(1, chosen)
            y = _experts(x, w, chosen, shares / shares.sum(-1, keepdim=True) * router["scale"], router["experts"], inner)
        x = norm(alpha * x + y, w("norm2"))
    return norm(x, weight("final.norm"))


def _stretched(rot):
    """Turning rates of the pairs and the factor on cos and sin, for positions beyond the original context."""
    dims, base, s = rot["dims"], rot["base"], rot["scaling"]

    def pair_turning(times):
        return dims * math.log(s["original"] / (2.0 * math.pi * times)) / (2.0 * math.log(base))

    low, high = max(math.floor(pair_turning(s["fast"])), 0), min(math.ceil(pair_turning(s["slow"])), dims - 1)
    rates = []
    for i in range(dims // 2):
        blend, rate = min(max((i - low) / max(high - low, 0.001), 0.0), 1.0), base ** (-2.0 * i / dims)
        rates.append(rate / s["factor"] * blend + rate * (1.0 - blend))
    return rates, 0.1 * math.log(s["factor"]) + 1.0
