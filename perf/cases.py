"""What is measured of this engine: whole requests through its public entry points, prompts and decode steps together.

A case names a model by its layer sizes, the precision, how many requests there are and how long their prompts, how many
tokens a step may bring and how many tokens are decoded after the prompts.  A pass admits the requests, runs them step by
step through `Engine.step` as a serving loop does (running requests bring one token each, what the step still has room for
goes to prompts in order, portions of them if need be), and finishes them.  The text is given beforehand, as when a
recorded conversation is replayed or scored, so that a pass does the same work whatever the logits are; it returns every
step's logits.  Cases with `generate` go through `Engine.generate` (scheduler and sampler included) and then score what
was generated with one more step, which gives the logits beside the tokens.

The weights are random, drawn by the engine from the seed; `exact` draws the same values and runs the model in 64 bits
with plain torch: whole sequences at once, no cache, no portions.
"""
import hashlib
import math
import random

import torch

from tlie_amd import Engine, StepEntry

F64 = torch.float64


def _llama(hidden, ff, layers, heads, kv_heads, positions, vocab, eps=1e-5, theta=10000.0, tied=False, bias=False, dim=None):
    return dict(model_type="llama", architectures=["LlamaForCausalLM"], hidden_size=hidden, intermediate_size=ff,
                num_hidden_layers=layers, num_attention_heads=heads, num_key_value_heads=kv_heads, head_dim=dim or hidden // heads,
                max_position_embeddings=positions, vocab_size=vocab, rms_norm_eps=eps, rope_theta=theta,
                tie_word_embeddings=tied, attention_bias=bias, hidden_act="silu", bos_token_id=1, eos_token_id=2)


def _tugalix():
    side = {"left": {"heads": 32, "kv_heads": 4, "dim": 64, "vdim": 64, "scale": 0.125, "rot": {"base": 10000.0, "dims": 64}},
            "right": {"heads": 32, "dim": 64, "rank": 64}, "left_scale": 1.0, "right_scale": 1.0}
    dense = {"kind": "dense", "ff": 8448}
    layers = [{"type": "retention", "mlp": None,
               "mixer": {"heads": 8, "dim": 128, "vdim": 256, "decay": [1.0 - 2.0 ** (-5 - 3 * head / 7) for head in range(8)],
                         "rot": {"base": 10000.0, "dims": 128}}},
              {"type": "parallel", "mixer": side, "mlp": dense},
              {"type": "gla", "mixer": {"heads": 4, "dim": 256, "vdim": 512, "tau": 16.0, "rank": 64}, "mlp": None},
              {"type": "parallel", "mixer": side, "mlp": dense}]
    return {"architecture": "Tugalix", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-5}, "canon": {"taps": 4}, "logit_scale": 1.0,
            "layers": layers}


# The configurations of the tests and of bench.py.  The two larger Llama shapes run with a quarter of their layers, as
# bench.py's default record has them: every layer is alike.
MODELS = {
    "tiny_a": _llama(64, 176, 2, 4, 2, 128, 256),
    "tiny_b": _llama(96, 256, 3, 3, 1, 256, 512, eps=1e-6, theta=500000.0, tied=True, bias=True, dim=32),
    "tinyllama": _llama(2048, 5632, 22, 32, 4, 2048, 32000),
    "llama2_7b": _llama(4096, 11008, 8, 32, 32, 4096, 32000),
    "llama3_8b": _llama(4096, 14336, 8, 32, 8, 8192, 128256, theta=500000.0),
    "tugalix": _tugalix(),                  # the decaying states' mixers beside attention, at bench.py's smaller layer sizes
}
BF16, FP32 = "bfloat16", "float32"


def _case(model, dtype, requests, shortest, longest, budget, new, generate=False):
    """requests with prompts of shortest .. longest tokens, at most `budget` tokens a step, `new` decoded tokens each."""
    return {"model": model, "dtype": dtype, "requests": requests, "shortest": shortest, "longest": longest, "budget": budget,
            "new": new, "generate": generate}


def listed():
    cases = [
        # a script or a test on the smallest model: greedy generation for three requests, prompts cut into portions of 16 beside
        # decoding, true 32-bit; launches and the host are all of it
        ("tiny_fp32_generate", _case("tiny_b", FP32, 3, 5, 64, 16, 16, generate=True)),
        # one short question to a small model: time to first token and a few tokens after it
        ("tinyllama_short_prompt", _case("tinyllama", BF16, 1, 100, 100, 2048, 7)),
        # a document into a small model, its continuation's logits asked for once: the prompt step of the model's whole range
        ("tinyllama_prompt_2048", _case("tinyllama", BF16, 1, 2048, 2048, 2048, 0)),
        # one user, long conversation: decoding at batch 1 close to the model's 2048 positions
        ("tinyllama_decode_b1", _case("tinyllama", BF16, 1, 1985, 1985, 2048, 62)),
        # a few users of a shared server: ragged conversations, decoding at batch 8
        ("tinyllama_decode_b8", _case("tinyllama", BF16, 8, 130, 1900, 2048, 50)),
        # a busy server: 64 requests come in over the first steps, prompts beside decoding, then batch 64
        ("tinyllama_serve_b64", _case("tinyllama", BF16, 64, 33, 450, 2048, 48)),
        # a long document and a short answer on a model of the next size (grouped heads of 128, a large vocabulary)
        ("llama3_8b_long_prompt", _case("llama3_8b", BF16, 1, 8001, 8001, 2048, 24)),
        # long prompts in portions of 512 tokens beside running decode streams
        ("llama3_8b_portions", _case("llama3_8b", BF16, 12, 40, 2500, 512, 24)),
        # a server of a model in which every head has its own keys and values
        ("llama2_7b_serve_b24", _case("llama2_7b", BF16, 24, 129, 1030, 2048, 32)),
        # the true 32-bit path: scoring a text of moderate length
        ("tinyllama_fp32_prompt", _case("tinyllama", FP32, 1, 1000, 1000, 2048, 0)),
        # the true 32-bit path: decoding at batch 8
        ("tinyllama_fp32_decode_b8", _case("tinyllama", FP32, 8, 20, 150, 2048, 24)),
        # another registered decoder: retention, gated linear attention, token-shift mixing beside attention; prompts, then batch 4
        ("tugalix_serve_b4", _case("tugalix", BF16, 4, 300, 2047, 2048, 40)),
    ]
    return [dict(case, name=name) for name, case in cases]


# ---- what a case's requests and steps are ------------------------------------------------------------------
MAX_STEPS = 60               # of a pass: every step's logits come back


def _lengths(case):
    """The prompts' lengths: the longest and the shortest, and others between them."""
    rng = random.Random(case["requests"] * 1000003 + case["shortest"] * 8209 + case["longest"])
    more = [rng.randint(case["shortest"], case["longest"]) for _ in range(case["requests"])]
    more[0] = case["longest"]
    if case["requests"] > 1:
        more[-1] = case["shortest"]
    return more


def _plan(case):
    """The steps of a pass: lists of (request, first position, tokens, whether the last token's logits are wanted)."""
    lengths = _lengths(case)
    done = [0] * len(lengths)
    steps = []
    while any(at < length + case["new"] for at, length in zip(done, lengths)):
        entries = [(r, done[r], 1, True) for r, length in enumerate(lengths) if length <= done[r] < length + case["new"]]
        room = case["budget"] - len(entries)
        for r, length in enumerate(lengths):
            count = min(room, length - done[r])
            if count > 0:
                entries.append((r, done[r], count, done[r] + count == length))
                room -= count
        for r, _, count, _ in entries:
            done[r] += count
        steps.append(entries)
    return steps


def _text(case, seed):
    """Every request's tokens: its prompt and what follows it."""
    generator = torch.Generator().manual_seed(seed)
    vocab = _sizes(case)["vocab"]
    return [torch.randint(0, vocab, (length + case["new"],), generator=generator).tolist() for length in _lengths(case)]


# ---- a pass -------------------------------------------------------------------------------------------------
def prepare(case, seed):
    """The engine a server keeps, warm (the same steps have run once on another text), and the requests' tokens."""
    pages = sum((length + case["new"] + 15) // 16 for length in _lengths(case))
    engine = Engine(None, dtype=case["dtype"], config=MODELS[case["model"]], random_seed=seed, max_tokens=16 * pages, page_size=16,
                    max_requests=case["requests"])
    state = {"case": case, "engine": engine, "plan": _plan(case), "text": _text(case, seed + 1)}
    run(state)
    state["text"] = _text(case, seed)
    return state


def run(state):
    case, engine, text = state["case"], state["engine"], state["text"]
    if case["generate"]:
        prompts = [tokens[:length] for tokens, length in zip(text, _lengths(case))]
        answers = engine.generate(prompts, max_tokens=case["new"], max_tokens_per_step=case["budget"])
        entries = []
        for r, (prompt, answer) in enumerate(zip(prompts, answers)):
            engine.admit(r)
            entries.append(StepEntry(r, prompt + answer, list(range(len(prompt) - 1, len(prompt) + len(answer)))))
        logits = engine.step(entries)
        for entry in entries:
            engine.finish(entry.request)
        return {"tokens": torch.tensor(answers), "logits": logits}
    for r in range(case["requests"]):
        engine.admit(r)
    logits = [engine.step([StepEntry(r, text[r][first:first + count], [count - 1] if wanted else []) for r, first, count, wanted in entries])
              for entries in state["plan"]]
    for r in range(case["requests"]):
        engine.finish(r)
    return logits


# ---- what a pass cannot do without --------------------------------------------------------------------------
def _sizes(case):
    """Weights a token meets in the layers and in the head, their flops beside the products, cache and state per token."""
    config = MODELS[case["model"]]
    if case["model"] == "tugalix":
        width, ff, rank, low = 2048, 8448, 64, 64 * (2048 + 1024)
        retention = width * (1024 * 2 + 2048 * 3)
        gla = width * (1024 * 2 + 2048 * 3) + low
        parallel = width * (2048 * 2 + 256 * 2) + width * 2048 * 5 + 2 * rank * width + 2 * width * ff
        states = [8 * 128 * 256, 4 * 256 * 512, 32 * 64 * 64, 32 * 64 * 64]
        return dict(vocab=config["vocab"], width=width, layers=retention + gla + 2 * parallel, attended=2 * 2 * 32 * 64, cached=2 * 2 * 4 * 64,
                    state=sum(states))
    h, ff, n = config["hidden_size"], config["intermediate_size"], config["num_hidden_layers"]
    q, kv = config["num_attention_heads"] * config["head_dim"], config["num_key_value_heads"] * config["head_dim"]
    return dict(vocab=config["vocab_size"], width=h, layers=n * (h * (2 * q + 2 * kv) + 3 * h * ff), attended=n * 2 * q, cached=n * 2 * kv, state=0)


def work(case):
    """Per step: the layers' weights and, where logits are wanted, the head's, read once; keys and values (or states) of the
    step's sequences read and the new ones written; the logits written.  Two flops a weight and token, four a query and key
    value met."""
    s, item = _sizes(case), 4 if case["dtype"] == FP32 else 2
    if case["generate"]:
        case = dict(case, new=case["new"] + 1)           # (the scoring step meets every token again: about one more pass)
    total_bytes = total_flops = 0.0
    for entries in _plan(case):
        wanted = sum(want for _, _, _, want in entries)
        tokens = sum(count for _, _, count, _ in entries)
        met = sum(count * first + count * (count + 1) // 2 for _, first, count, _ in entries)
        weights = s["layers"] + (s["vocab"] * s["width"] if wanted else 0)
        kept = s["cached"] * sum(first + count for _, first, count, _ in entries)
        total_bytes += item * (weights + tokens * s["width"] + kept + s["cached"] * tokens) + 4 * wanted * s["vocab"]
        total_bytes += 8 * s["state"] * len(entries)
        total_flops += 2 * s["layers"] * tokens + 2 * s["attended"] * met + 4 * s["state"] * tokens + 2 * s["vocab"] * s["width"] * wanted
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case):
    """Measured: bfloat16 activations through 8 to 22 layers leave 0.5e-2 to 3e-2 against 64 bits, and the same prompt in other
    portions (other kernels, sums in another order) differs by up to 2.1e-2, its largest value by 0.05 of the rms.  32-bit sums
    through 22 layers leave 0.3e-5 to 1.1e-5."""
    if case["dtype"] == FP32:
        return {"rel": 4e-5, "max": 4e-4, "differ": 0.0}
    return {"rel": 3e-2, "max": 0.2}


# ---- more cases of the same ranges --------------------------------------------------------------------------
def _spread(rng, least, most):
    """A whole number between least and most, even over its logarithm."""
    return min(most, max(least, round(math.exp(rng.uniform(math.log(least), math.log(most + 0.49))))))


def _cost(case):
    """Seconds a pass may take, roughly: per step its launches, its bytes, its flops."""
    s, w, steps = _sizes(case), work(case), len(_plan(case))
    rate = 0.25e14 if case["dtype"] == FP32 else 5e14
    return steps * 1e-3 + w["bytes"] / 3e12 + w["flops"] / rate + 4e-13 * s["state"] * sum(_lengths(case))


def draw(rng):
    ranges = [
        # (model, precision, most requests, shortest and longest prompt, most new tokens)
        ("tiny_a", FP32, 4, 3, 90, 30), ("tiny_b", FP32, 4, 3, 200, 40),
        ("tinyllama", BF16, 64, 20, 2000, 56), ("tinyllama", BF16, 64, 20, 2000, 56), ("tinyllama", BF16, 1, 30, 2048, 0),
        ("llama2_7b", BF16, 32, 60, 4000, 48), ("llama3_8b", BF16, 32, 60, 8100, 48),
        ("tinyllama", FP32, 8, 20, 1000, 40), ("tugalix", BF16, 8, 50, 2200, 50),
    ]
    while True:
        model, dtype, requests, least, most, new = rng.choice(ranges)
        requests = _spread(rng, 1, requests)
        longest = _spread(rng, least, most)
        new = _spread(rng, 1, new) if new else 0
        generate = model.startswith("tiny_") and rng.random() < 0.6
        budget = rng.choice([16, 37, 64] if model.startswith("tiny_") else [512, 1024, 2048, 2048])
        case = _case(model, dtype, requests, _spread(rng, least, longest) if requests > 1 else longest, longest, budget, new, generate)
        positions = MODELS[model].get("max_position_embeddings", 4096)
        if longest + new <= positions and len(_plan(case)) <= MAX_STEPS and _cost(case) <= 0.16:
            return case


# ---- the same in 64 bits ------------------------------------------------------------------------------------
def _weights(case, seed):
    """name, shape, kind -> the tensor that the engine draws for the seed, in 64 bits: a generator per name on the device,
    values in 32 bits, rounded to the engine's precision."""
    kept = torch.float32 if case["dtype"] == FP32 else torch.bfloat16

    def draw_one(name, *shape, kind="normal"):
        digest = hashlib.sha256(f"{seed}:{name}".encode("utf-8")).digest()
        generator = torch.Generator(device="cuda").manual_seed(int.from_bytes(digest[:8], "little") & 0x7FFF_FFFF_FFFF_FFFF)
        values = torch.randn(shape, generator=generator, dtype=torch.float32, device="cuda")
        if kind == "fraction":                           # (drawn after the normal ones)
            values = torch.rand(shape, generator=generator, dtype=torch.float32, device="cuda")
        elif kind == "normal":
            values = values * 0.02
        elif kind == "norm":
            values = 1.0 + values * 0.01
        elif kind == "offset":
            values = values * 0.01
        elif kind == "mix":
            values = values * 0.2
            values[..., -1] += 1.0
        return values.to(kept).to(F64)
    return draw_one


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)


def _turned(x, positions, base):
    """x [T, heads, dim]: dim i turns with dim i + dim / 2 by position * base^(-2i / dim)."""
    half = x.shape[-1] // 2
    angle = positions[:, None, None] * base ** (-torch.arange(half, dtype=F64, device=x.device) / half)
    u, v = x[..., :half], x[..., half:]
    return torch.cat([u * angle.cos() - v * angle.sin(), v * angle.cos() + u * angle.sin()], dim=-1)


def _attention(q, k, v, spans):
    """Causal, q [T, heads, dim], k and v [T, kv heads, dim], every request's tokens on their own; in stretches of queries."""
    out = torch.empty_like(q)
    group = q.shape[1] // k.shape[1]
    for start, end in spans:
        for head in range(q.shape[1]):
            keys, values = k[start:end, head // group], v[start:end, head // group]
            for at in range(start, end, 2048):
                to = min(end, at + 2048)
                scores = q[at:to, head] @ keys[:to - start].t() * q.shape[2] ** -0.5
                seen = torch.arange(to - start, device=q.device)[None, :] <= torch.arange(at - start, to - start, device=q.device)[:, None]
                out[at:to, head] = torch.softmax(scores.masked_fill(~seen, -math.inf), dim=-1) @ values[:to - start]
    return out.reshape(len(q), -1)


def _llama_rows(config, draw_one, tokens, positions, spans, rows):
    h, ff, heads, kv, dim = (config[k] for k in ("hidden_size", "intermediate_size", "num_attention_heads", "num_key_value_heads", "head_dim"))
    eps, count = config["rms_norm_eps"], len(tokens)
    table = draw_one("model.embed_tokens.weight", config["vocab_size"], h)
    x = table[tokens]
    for layer in range(config["num_hidden_layers"]):
        def linear(name, value, outs):
            name = f"model.layers.{layer}.{name}"
            value = value @ draw_one(name + ".weight", outs, value.shape[1]).t()
            return value + draw_one(name + ".bias", outs) if config["attention_bias"] and "self_attn" in name else value

        y = _rms(x, eps) * draw_one(f"model.layers.{layer}.input_layernorm.weight", h, kind="norm")
        q = _turned(linear("self_attn.q_proj", y, heads * dim).reshape(count, heads, dim), positions, config["rope_theta"])
        k = _turned(linear("self_attn.k_proj", y, kv * dim).reshape(count, kv, dim), positions, config["rope_theta"])
        v = linear("self_attn.v_proj", y, kv * dim).reshape(count, kv, dim)
        x = x + linear("self_attn.o_proj", _attention(q, k, v, spans), h)
        y = _rms(x, eps) * draw_one(f"model.layers.{layer}.post_attention_layernorm.weight", h, kind="norm")
        x = x + linear("mlp.down_proj", torch.nn.functional.silu(linear("mlp.gate_proj", y, ff)) * linear("mlp.up_proj", y, ff), h)
    x = _rms(x[rows], eps) * draw_one("model.norm.weight", h, kind="norm")
    return x @ (table if config["tie_word_embeddings"] else draw_one("lm_head.weight", config["vocab_size"], h)).t()


def _scan(q, k, v, decay, bonus=None):
    """q, k, decay [T, heads, dim], v [T, heads, vdim]: S = diag(decay) S + k v^T, out = S^T q; with a bonus u the result is read
    before the token joins the state, from S + diag(u) k v^T."""
    S = torch.zeros(q.shape[1], q.shape[2], v.shape[2], dtype=F64, device=q.device)
    out = []
    for t in range(len(q)):
        outer = k[t][:, :, None] * v[t][:, None, :]
        seen = S + bonus[:, :, None] * outer if bonus is not None else None
        S = decay[t][:, :, None] * S + outer
        out.append(torch.matmul(q[t][:, None, :], seen if bonus is not None else S)[:, 0])
    return torch.stack(out)


def _tugalix_rows(config, draw_one, tokens, positions, spans, rows):
    width, eps, taps, count = config["width"], config["norm"]["eps"], config["canon"]["taps"], len(tokens)
    silu, each = torch.nn.functional.silu, [slice(start, end) for start, end in spans]

    def norm(name, x):
        x = x - x.mean(dim=-1, keepdim=True)
        return _rms(x, eps) * draw_one(name, width, kind="norm") + draw_one(name + ".b", width, kind="offset")

    def shifted(x, by):
        """Every token's input `by` tokens back in its own request, zero before the request."""
        out = torch.zeros_like(x)
        for span in each:
            out[span][by:] = x[span][:max(0, span.stop - span.start - by)]
        return out

    def conv(name, x):
        weight = draw_one(name, width, taps)
        return x + sum(weight[:, j] * shifted(x, taps - 1 - j) for j in range(taps))

    def linear(name, x, outs):
        return x @ draw_one(name, outs, x.shape[1]).t()

    def scans(q, k, v, decay, bonus=None):
        return torch.cat([_scan(q[s], k[s], v[s], decay[s], bonus) for s in each])

    def state_mixer(kind, m, p, x):
        H, dim, vdim = m["heads"], m["dim"], m["vdim"]
        q, k = (linear(p + name, x, H * dim).reshape(count, H, dim) for name in "qk")
        v = linear(p + "v", x, H * vdim).reshape(count, H, vdim)
        if kind == "retention":
            q, k = _turned(q, positions, m["rot"]["base"]), _turned(k, positions, m["rot"]["base"]) * dim ** -0.5
            decay = torch.tensor(m["decay"], dtype=F64, device=x.device)[None, :, None].expand(count, H, dim)
            out = _rms(scans(q, k, v, decay), eps)
        else:
            z = linear(p + "a2", linear(p + "a1", x, m["rank"]), H * dim) + draw_one(p + "a2.b", H * dim)
            decay = torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]).reshape(count, H, dim)
            out = _rms(scans(q * dim ** -0.5, k, v, decay), eps) * draw_one(p + "norm", vdim, kind="norm")
        return linear(p + "o", out.reshape(count, -1) * silu(linear(p + "g", x, H * vdim)), width)

    def two_sided(m, p, x):
        left, right = m["left"], m["right"]
        H, G, dim = left["heads"], left["kv_heads"], left["dim"]
        q = _turned(linear(p + "left.q", x, H * dim).reshape(count, H, dim), positions, left["rot"]["base"])
        k = _turned(linear(p + "left.k", x, G * dim).reshape(count, G, dim), positions, left["rot"]["base"])
        attended = linear(p + "left.o", _attention(q, k, linear(p + "left.v", x, G * dim).reshape(count, G, dim), spans), width)
        p, before, H, dim = p + "right.", shifted(x, 1), right["heads"], right["dim"]

        def blend(name):
            return x + (before - x) * draw_one(p + "mu." + name, width, kind="fraction")
        r, k, v = (linear(p + name, blend(name), H * dim).reshape(count, H, dim) for name in "rkv")
        z = linear(p + "w2", torch.tanh(linear(p + "w1", blend("w"), right["rank"])), H * dim) + draw_one(p + "w0", H * dim)
        out = _rms(scans(r, k, v, torch.exp(-torch.exp(z)).reshape(count, H, dim), draw_one(p + "u", H, dim)), eps)
        mixed = out.reshape(count, -1) * draw_one(p + "norm", width, kind="norm") * silu(linear(p + "g", blend("g"), width))
        return m["left_scale"] * attended + m["right_scale"] * linear(p + "o", mixed, width)

    x = norm("embed.norm", draw_one("embed", config["vocab"], width)[tokens])
    results = [x]
    for index, layer in enumerate(config["layers"]):
        p = f"l{index}."
        y = conv(p + "canon1", norm(p + "norm1", x))
        x = x + (two_sided(layer["mixer"], p + "mix.", y) if layer["type"] == "parallel" else state_mixer(layer["type"], layer["mixer"], p + "mix.", y))
        if layer["mlp"] is not None:
            z = linear(p + "mlp.up", conv(p + "canon2", norm(p + "norm2", x)), layer["mlp"]["ff"])
            a, b = torch.nn.functional.softplus(draw_one(p + "mlp.act", 2, kind="offset"))
            x = x + linear(p + "mlp.down", torch.where(z > 0, a * z * z + 0.5 * z, (0.5 + b) * (torch.expm1(z) - z) + 0.5 * z), width)
        results.append(x)
        x = sum(share * result for share, result in zip(draw_one(p + "dwa", index + 2, kind="mix"), results))
    return linear("head", norm("final.norm", x[rows]), config["vocab"]) * config["logit_scale"]


def _rows_exact(case, seed, text, wanted):
    """Logits in 64 bits of the places `wanted`, pairs of (request, position)."""
    starts = [sum(len(tokens) for tokens in text[:r]) for r in range(len(text) + 1)]
    tokens = torch.tensor([token for tokens in text for token in tokens], device="cuda")
    positions = torch.cat([torch.arange(len(tokens), dtype=F64, device="cuda") for tokens in text])
    rows = torch.tensor([starts[r] + position for r, position in wanted], device="cuda")
    forward = _tugalix_rows if case["model"] == "tugalix" else _llama_rows
    return forward(MODELS[case["model"]], _weights(case, seed), tokens, positions, list(zip(starts, starts[1:])), rows)


@torch.no_grad()
def exact(case, seed):
    text, lengths = _text(case, seed), _lengths(case)
    if case["generate"]:
        texts = [tokens[:length] for tokens, length in zip(text, lengths)]
        for _ in range(case["new"]):
            last = _rows_exact(case, seed, texts, [(r, len(tokens) - 1) for r, tokens in enumerate(texts)])
            texts = [tokens + [int(token)] for tokens, token in zip(texts, last.argmax(-1))]
        logits = _rows_exact(case, seed, texts, [(r, at) for r, length in enumerate(lengths) for at in range(length - 1, length + case["new"])])
        return {"tokens": torch.tensor([tokens[length:] for tokens, length in zip(texts, lengths)]), "logits": logits}
    steps = [[(r, first + count - 1) for r, first, count, want in entries if want] for entries in _plan(case)]
    logits = _rows_exact(case, seed, text, [place for step in steps for place in step])
    return list(torch.split(logits, [len(step) for step in steps]))
