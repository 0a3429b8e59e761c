"""What a server and its clients have this framework compute, as measurable cases.

A case is one call of a span of consecutive decoder blocks, made as the server makes it:

  decode    one token per sequence against cached keys and values: the captured graph of
            the span that a session replays (utils/graphs.py, DecodeContext)
  prefill   a prompt into the cache of a session: TransformerBackend.inference_step
  forward   whole sequences without a cache (fine-tuning): TransformerBackend.forward
  backward  the same with its gradients and those of the trained prompts of every block:
            forward again, then TransformerBackend.backward from the last block to the first
  step      rows of several requests at once over pages: SpanEngine.step

Sizes of the models are the framework's presets and the 4k sizes of its benchmarks. Weights
are random: 0.02 for what reads the stream, 0.02 / sqrt(2 layers) for what is added to it,
as trained models are initialized, and norm weights around 1. Streams are normal values with
a few channels ten times as large, as trained models have them.
"""

from __future__ import annotations

import asyncio
import math
import zlib

import torch

BF16, F64 = torch.bfloat16, torch.float64
PROMPT_ROWS = 16  # trained prompt rows per block in `backward`
ROOM = 64  # tokens a session may still generate
OUT_PROJECTIONS = ("o_proj.weight", "down_proj.weight", "dense.weight", "dense_4h_to_h.weight", "w2.weight", "o", "down")
NF4_LEVELS = (
    -1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
    -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
    0.24611230194568634, 0.33791524171829224, 0.4407098293304443, 0.5626170039176941, 0.7229568362236023, 1.0,
)

# family and sizes: width, heads, kv heads, feed-forward, layers of the whole model
MODELS = {
    "tinyllama-1.1b": ("llama", 2048, 32, 4, 5632, 22),
    "llama-2-7b": ("llama", 4096, 32, 32, 11008, 32),
    "llama-3-8b": ("llama", 4096, 32, 8, 14336, 32),
    "llama-2-70b": ("llama", 8192, 64, 8, 28672, 80),
    "bloom-7b1": ("bloom", 4096, 32, 32, 16384, 30),
    "falcon-7b": ("falcon", 4544, 71, 1, 18176, 32),
    "falcon-40b": ("falcon", 8192, 128, 8, 32768, 60),
    "mixtral-8x7b": ("mixtral", 4096, 32, 8, 14336, 32),
}
ROPE_BASE = {"llama-3-8b": 500000.0, "mixtral-8x7b": 1000000.0}
EXPERTS, TOP = 8, 2  # mixtral
# paged families, layers of width 4096 as in the framework's comparisons
TULEZEN = dict(width=4096, heads=32, dim=128, rank=512, window=1024, experts=8, top=2, ff=14336, limit=7.0, layers=32)
ZUDARAX = dict(width=4096, heads=16, dim=128, vdim=256, diff=0.5, ff=16384, groups=2, layers=32)


def listed():
    return [
        # the smallest call: a token of a small model right after a short question
        dict(name="decode-small", kind="decode", model="tinyllama-1.1b", quant="none", blocks=4, batch=1, context=37),
        # a chat's token on the large model, quantized to fit: the headline benchmark's step
        dict(name="decode-70b-nf4", kind="decode", model="llama-2-70b", quant="nf4", blocks=4, batch=1, context=153),
        # the same for eight hypotheses or prompts of one client
        dict(name="decode-70b-nf4-8", kind="decode", model="llama-2-70b", quant="nf4", blocks=4, batch=8, context=2003),
        # two long documents at the end of an 8k context, weights as they are
        dict(name="decode-long", kind="decode", model="llama-3-8b", quant="none", blocks=4, batch=2, context=7900),
        # routed experts, quantized
        dict(name="decode-experts", kind="decode", model="mixtral-8x7b", quant="nf4", blocks=2, batch=2, context=1000),
        # the headline benchmark's prompt
        dict(name="prefill-70b-nf4", kind="prefill", model="llama-2-70b", quant="nf4", blocks=2, batch=1, tokens=128),
        # a document
        dict(name="prefill-long", kind="prefill", model="llama-3-8b", quant="none", blocks=2, batch=1, tokens=4096),
        # a page of text through routed experts
        dict(name="prefill-experts", kind="prefill", model="mixtral-8x7b", quant="none", blocks=2, batch=1, tokens=283),
        # the forward benchmark: 4 x 128 tokens, 8-bit weights
        dict(name="forward-int8", kind="forward", model="bloom-7b1", quant="int8", blocks=2, batch=4, tokens=128),
        # a step of deep prompt tuning
        dict(name="backward", kind="backward", model="llama-2-7b", quant="none", blocks=2, batch=2, tokens=379),
        # prompts of several requests beside the tokens of others
        dict(name="step-ragged", kind="step", model="tulezen", blocks=2, context=300, rows="1021,130,7,1,1,1"),
        # tokens of eight requests
        dict(name="step-tokens", kind="step", model="zudarax", blocks=2, context=2048, rows="1,1,1,1,1,1,1,1"),
    ]


DECODE = [
    ("tinyllama-1.1b", "none"), ("llama-2-7b", "none"), ("llama-2-7b", "int8"), ("llama-2-7b", "nf4"),
    ("llama-3-8b", "none"), ("llama-3-8b", "nf4"), ("llama-2-70b", "nf4"), ("bloom-7b1", "none"), ("bloom-7b1", "int8"),
    ("bloom-7b1", "nf4"), ("falcon-7b", "none"), ("falcon-40b", "nf4"), ("mixtral-8x7b", "none"), ("mixtral-8x7b", "nf4"),
]
WHOLE = [
    ("tinyllama-1.1b", "none"), ("llama-2-7b", "none"), ("llama-2-7b", "int8"), ("llama-3-8b", "none"),
    ("llama-2-70b", "nf4"), ("bloom-7b1", "none"), ("bloom-7b1", "int8"), ("falcon-7b", "none"), ("mixtral-8x7b", "none"),
    ("mixtral-8x7b", "nf4"),
]


def _spread(rng, lo, hi):
    """A whole number, spread over the logarithm of the range."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["decode", "decode", "prefill", "forward", "backward", "step"])
        if kind == "step":
            rows = [_spread(rng, 1, 1500) if rng.random() < 0.5 else 1 for _ in range(rng.randint(1, 8))]
            if rng.random() < 0.5:
                rows = [1] * len(rows)
            case = dict(kind=kind, model=rng.choice(["tulezen", "zudarax"]), blocks=rng.randint(1, 2),
                        context=rng.choice([0, _spread(rng, 1, 2500)]), rows=",".join(map(str, rows)))
        else:
            model, quant = rng.choice(DECODE if kind == "decode" else WHOLE)
            case = dict(kind=kind, model=model, quant=quant, blocks=rng.randint(1, 2))
            if kind == "decode":
                case.update(batch=rng.randint(1, 8), context=_spread(rng, 2, 7900))
            elif kind == "prefill":
                case.update(batch=rng.choice([1, 1, 2, 3]), tokens=_spread(rng, 2, 4096))
            else:
                case.update(batch=rng.randint(1, 5), tokens=_spread(rng, PROMPT_ROWS, 1024))
        if _cost(case) <= most and (kind in ("decode", "step") or _gated(case) <= 1 << 23):
            return case


def _gated(case):
    """Values of the feed-forward's inner rows in one call of a block: clients cut large
    batches, and a prompt is taken in parts of at most 256 MB of attention scores."""
    family, _, heads, _, ff, _ = MODELS[case["model"]]
    batch, tokens = case["batch"], case["tokens"]
    if case["kind"] == "prefill":
        tokens = min(tokens, (256 << 20) // (4 * heads * batch * tokens))
    return batch * tokens * ff * (TOP if family == "mixtral" else 1)


def _cost(case):
    """Seconds, roughly: cases are compared by it."""
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / 4e14


# ------------------------------------------------------------------ what a pass needs


def _bytes_per_weight(quant):
    return {"none": 2.0, "int8": 1.0, "nf4": 0.53125}[quant]


def _attention_pairs(before, new):
    return before * new + new * (new + 1) / 2


def work(case):
    if case["kind"] == "step":
        return _work_step(case)
    family, h, heads, kv, ff, _ = MODELS[case["model"]]
    hd = h // heads
    batch, new = case["batch"], case.get("tokens", 1)
    rows, before = batch * new, case.get("context", 0)
    dense = h * (heads + 2 * kv) * hd + h * h
    if family == "mixtral":
        each, router = 3 * h * ff, h * EXPERTS
        read = EXPERTS * (1.0 - (1.0 - TOP / EXPERTS) ** rows) * each
        used = dense + router + TOP * each
        weights = (dense + read) * _bytes_per_weight(case["quant"]) + 2 * router
    else:
        used = dense + (3 if family == "llama" else 2) * h * ff
        weights = used * _bytes_per_weight(case["quant"])
    attention = 4 * heads * hd * _attention_pairs(before, new) * batch
    flops = 2 * used * rows + attention
    bytes_ = weights + 4 * rows * h  # the stream in and out
    if case["kind"] in ("decode", "prefill"):
        bytes_ += 2 * batch * kv * hd * 2 * (before + new)
    if case["kind"] == "backward":
        # forward for what the gradients need, then the gradients of the stream
        flops = 2 * (2 * used * rows) + 3.5 * attention
        bytes_ = 2 * weights + 6 * rows * h
    return {"bytes": bytes_ * case["blocks"], "flops": flops * case["blocks"]}


def _rows(case):
    return [int(n) for n in case["rows"].split(",")]


def _work_step(case):
    rows, before = _rows(case), case["context"]
    t = sum(rows)
    if case["model"] == "tulezen":
        m = TULEZEN
        latents = sum(min(before + n, m["window"] + n - 1) for n in rows)
        pairs = sum(sum(min(before + i + 1, m["window"]) for i in range(n)) for n in rows)
        each = 3 * m["width"] * m["ff"]
        dense = 2 * m["width"] * m["heads"] * m["dim"] + (2 * m["heads"] * m["dim"] + m["width"]) * m["rank"]
        read = m["experts"] * (1.0 - (1.0 - m["top"] / m["experts"]) ** t) * each
        flops = 2 * t * (dense + m["top"] * each) + 4 * m["heads"] * m["dim"] * pairs
        bytes_ = 2 * (dense + read) + 2 * latents * m["rank"]
    else:
        m = ZUDARAX
        pairs = sum(_attention_pairs(before, n) for n in rows)
        wide = m["heads"] * (4 * m["dim"] + 2 * m["vdim"] + 1) + 2 * m["ff"]
        flops = 2 * t * m["width"] * wide + 4 * m["heads"] * (m["dim"] + m["vdim"]) * pairs
        bytes_ = 2 * m["width"] * wide + 2 * sum(before + n for n in rows) * m["heads"] * (2 * m["dim"] + m["vdim"])
    return {"bytes": (bytes_ + 8 * t * m["width"]) * case["blocks"], "flops": flops * case["blocks"]}


def tolerance(case):
    # About four times what the present code is away from 64 bits: 0.0057 at most for streams in
    # bf16, 0.0024 for those in 32 bits, and 0.045 with routed experts, where now and then a
    # token's second and third expert score alike and rounding decides.
    rel = 2e-2
    if case["model"] == "zudarax":
        rel = 1e-2
    if case["model"] in ("mixtral-8x7b", "tulezen"):
        rel = 0.18
    return {"rel": rel}


# ------------------------------------------------------------------------- inputs


def _generator(*key):
    seed = zlib.crc32("/".join(map(str, key)).encode()) & 0x7FFFFFFF
    return torch.Generator(device="cuda").manual_seed(seed or 1)


def _weight(seed, block, name, shape, layers):
    """One parameter of a block, bf16."""
    gen = _generator(seed, block, name)
    t = torch.empty(shape, device="cuda", dtype=BF16)
    if len(shape) >= 2:
        out = any(name == n or name.endswith("." + n) for n in OUT_PROJECTIONS)
        return t.normal_(0.0, 0.02 / math.sqrt(2 * layers) if out else 0.02, generator=gen)
    if name.rsplit(".", 1)[-1] in ("bias", "lq1", "lk1", "lq2", "lk2"):
        return t.normal_(0.0, 0.02, generator=gen)
    return t.normal_(1.0, 0.1, generator=gen)


def _stream(seed, name, *shape, dtype=BF16):
    gen = _generator(seed, name)
    x = torch.randn(shape, generator=gen, device="cuda")
    loud = torch.randint(0, shape[-1], (6,), generator=gen, device="cuda")
    x[..., loud] *= 10.0
    return x.to(dtype)


def _shapes(case):
    """name -> shape of a block's parameters, as in the families' checkpoints"""
    model = case["model"]
    if model == "tulezen":
        m = TULEZEN
        d, hd, e, f = m["width"], m["heads"] * m["dim"], m["experts"], m["ff"]
        return {"norm1": (d,), "q": (hd, d), "dkv": (m["rank"], d), "dkv_norm": (m["rank"],), "uk": (hd, m["rank"]),
                "uv": (hd, m["rank"]), "o": (d, hd), "norm2": (d,), "router": (e, d), "gate": (e, f, d), "up": (e, f, d),
                "down": (e, d, f)}
    if model == "zudarax":
        m = ZUDARAX
        d, f, hq, hv = m["width"], m["ff"], 2 * m["heads"] * m["dim"], m["heads"] * m["vdim"]
        return {"norm1": (d,), "q": (hq, d), "k": (hq, d), "v": (hv, d), "o": (d, hv), "lq1": (m["dim"],),
                "lk1": (m["dim"],), "lq2": (m["dim"],), "lk2": (m["dim"],), "g": (m["heads"], d), "up": (f, d),
                "down": (d, f), "act": (4,)}
    family, h, heads, kv, ff, _ = MODELS[model]
    qkv = (heads + 2 * kv) * (h // heads)
    if family in ("llama", "mixtral"):
        kvd = kv * (h // heads)
        s = {"self_attn.q_proj.weight": (h, h), "self_attn.k_proj.weight": (kvd, h), "self_attn.v_proj.weight": (kvd, h),
             "self_attn.o_proj.weight": (h, h), "input_layernorm.weight": (h,), "post_attention_layernorm.weight": (h,)}
        if family == "llama":
            s.update({"mlp.gate_proj.weight": (ff, h), "mlp.up_proj.weight": (ff, h), "mlp.down_proj.weight": (h, ff)})
        else:
            s["block_sparse_moe.gate.weight"] = (EXPERTS, h)
            for e in range(EXPERTS):
                at = f"block_sparse_moe.experts.{e}."
                s.update({at + "w1.weight": (ff, h), at + "w2.weight": (h, ff), at + "w3.weight": (ff, h)})
        return s
    s = {"self_attention.query_key_value.weight": (qkv, h), "self_attention.dense.weight": (h, h),
         "mlp.dense_h_to_4h.weight": (ff, h), "mlp.dense_4h_to_h.weight": (h, ff)}
    norms = {"falcon-40b": ("ln_attn", "ln_mlp"), "falcon-7b": ("input_layernorm",)}
    for n in norms.get(model, ("input_layernorm", "post_attention_layernorm")):
        s.update({f"{n}.weight": (h,), f"{n}.bias": (h,)})
    if family == "bloom":
        s.update({"self_attention.query_key_value.bias": (qkv,), "self_attention.dense.bias": (h,),
                  "mlp.dense_h_to_4h.bias": (ff,), "mlp.dense_4h_to_h.bias": (h,)})
    return s


def _layers(case):
    return {"tulezen": TULEZEN["layers"], "zudarax": ZUDARAX["layers"]}.get(case["model"]) or MODELS[case["model"]][5]


def _weights(case, seed, block):
    centred = ("norm1", "norm2") if case["model"] == "tulezen" else ()  # weights added to 1
    out = {n: _weight(seed, block, n, shape, _layers(case)) for n, shape in _shapes(case).items()}
    for n in centred:
        out[n] -= 1.0
    return out


def _quantized(case):
    return case.get("quant", "none")


# ------------------------------------------------------------------------ the span


def _config(case):
    if case["model"] == "tulezen":
        from petals_amd.models.tulezen.config import TulezenConfig

        m = TULEZEN
        layer = {
            "type": "latent_attention",
            "mixer": {"heads": m["heads"], "dim": m["dim"], "vdim": m["dim"], "kv_rank": m["rank"],
                      "scale": m["dim"] ** -0.5, "mask": {"size": m["window"]}},
            "mlp": {"kind": "moe", "expert": {"ff": m["ff"], "limit": m["limit"]},
                    "router": {"experts": m["experts"], "top": m["top"]}},
        }
        return TulezenConfig.from_hf_dict(
            {"layers": [layer] * case["blocks"], "norm": {"eps": 1e-6}, "vocab": 1024, "width": m["width"]}
        )
    if case["model"] == "zudarax":
        from petals_amd.models.zudarax.config import ZudaraxConfig

        m = ZUDARAX
        layer = {
            "type": "attention_2",
            "mixer": {"heads": m["heads"], "kv_heads": m["heads"], "dim": m["dim"], "vdim": m["vdim"], "diff": m["diff"],
                      "rot": {"base": 10000.0, "dims": m["dim"]}, "scale": m["dim"] ** -0.5},
            "mlp": {"kind": "dense", "ff": m["ff"]},
        }
        return ZudaraxConfig.from_hf_dict(
            {"layers": [layer] * case["blocks"], "norm": {"eps": 1e-6, "groups": m["groups"]}, "vocab": 1024,
             "width": m["width"]}
        )
    from petals_amd.models.config_base import load_model_config

    return load_model_config(case["model"])


class _Span:
    """Blocks of one server, and what a session on it keeps."""

    def __init__(self, case, seed):
        from petals_amd.server.from_pretrained import build_empty_block

        self.case, self.config = case, _config(case)
        self.blocks = []
        for i in range(case["blocks"]):
            block = build_empty_block(self.config, i, torch.device("cuda"), BF16)
            block.load_state_dict(_weights(case, seed, i), strict=True, assign=True)
            self.blocks.append(block.eval().optimize_for_inference(quant=_quantized(case)))

    def open_backends(self, max_length=0):
        from petals_amd.server.backend import TransformerBackend
        from petals_amd.server.memory_cache import MemoryCache

        self.cache = MemoryCache(None, torch.device("cuda"))
        self.backends = [
            TransformerBackend(f"block.{i}", b, config=self.config, memory_cache=self.cache, dtype=BF16)
            for i, b in enumerate(self.blocks)
        ]
        if max_length:
            wanted = [d for b in self.backends for d in b.get_inference_cache_descriptors(self.case["batch"], max_length)]
            self._loop, self._lease = asyncio.new_event_loop(), self.cache.allocate_cache(*wanted)
            handles = self._loop.run_until_complete(self._lease.__aenter__())
            self.handles = [tuple(handles[2 * i : 2 * i + 2]) for i in range(len(self.backends))]
            with self.cache.use_cache(*handles) as tensors:
                self.tensors = list(tensors)

    _lease = None

    def __del__(self):
        if self._lease is not None:
            self._loop.run_until_complete(self._lease.__aexit__(None, None, None))
            self._loop.close()


def _cached(case, seed, block):
    """Keys and values of the tokens before: [B, KV, L, hd] each, room left at the end."""
    _, h, heads, kv, _, _ = MODELS[case["model"]]
    shape = (case["batch"], kv, case["context"], h // heads)
    out = []
    for name in "kv":
        t = torch.zeros(*shape[:2], case["context"] + ROOM, shape[3], device="cuda", dtype=BF16)
        t[:, :, : case["context"]].normal_(generator=_generator(seed, block, "cached", name))
        out.append(t)
    return out


def prepare(case, seed):
    return {"decode": _prepare_decode, "prefill": _prepare_prefill, "forward": _prepare_whole,
            "backward": _prepare_whole, "step": _prepare_step}[case["kind"]](case, seed)


def run(state):
    return state.run()


@torch.inference_mode()
def _prepare_decode(case, seed):
    from petals_amd.ops.fused_decode import DecodeContext
    from petals_amd.utils.graphs import GraphedCallable

    span = _Span(case, seed)
    width = MODELS[case["model"]][1]
    hidden = _stream(seed, "hidden", case["batch"], 1, width)
    caches = [tuple(_cached(case, seed, i)) for i in range(case["blocks"])]
    ctx = DecodeContext(torch.device("cuda"))
    ctx.set_position(case["context"])
    taken = torch.empty_like(hidden)

    def step():
        x = taken
        ctx.norm_parts = None
        for block, cache in zip(span.blocks, caches):
            x = block(x, kv_cache=cache, ctx=ctx)
        return x

    taken.copy_(hidden)
    graph = GraphedCallable(step, [])

    @torch.inference_mode()
    def one_pass():
        ctx.set_position(case["context"])
        taken.copy_(hidden)
        return [graph.replay().clone(), *(t for pair in caches for t in pair)]

    span.run = one_pass
    return span


@torch.inference_mode()
def _prepare_prefill(case, seed):
    from petals_amd.data_structures import InferenceMetadata

    span = _Span(case, seed)
    span.open_backends(case["tokens"] + ROOM)
    hidden = _stream(seed, "hidden", case["batch"], case["tokens"], MODELS[case["model"]][1])
    backends, handles, tensors = span.backends, span.handles, span.tensors

    def one_pass():
        x = hidden
        for backend, pair in zip(backends, handles):
            (x,) = backend.inference_step(x, None, InferenceMetadata(backend.uid, 0, pair))
        return [x, *tensors]

    span.run = one_pass
    return span


def _prepare_whole(case, seed):
    span = _Span(case, seed)
    span.open_backends()
    backends = span.backends
    width = MODELS[case["model"]][1]
    hidden = _stream(seed, "hidden", case["batch"], case["tokens"], width)

    def forward():
        x = hidden
        for backend in backends:
            x = backend.forward(x)
        return [x]

    if case["kind"] == "forward":
        span.run = forward
        return span
    grad = _stream(seed, "grad", case["batch"], case["tokens"], width)
    prompts = [_stream(seed, f"prompt{i}", case["batch"], PROMPT_ROWS, width) for i in range(case["blocks"])]

    def backward():
        x, inputs = hidden, []
        with torch.no_grad():
            for i, backend in enumerate(backends):
                x = x.clone()
                x[:, :PROMPT_ROWS] += prompts[i]
                inputs.append(x)
                if i + 1 < len(backends):
                    x = backend.block(x)
        g, grads = grad, []
        for backend, x in zip(reversed(backends), reversed(inputs)):
            g, _ = backend.backward(x, g)
            grads.insert(0, g[:, :PROMPT_ROWS].clone())
        return [g, torch.stack(grads)]

    span.run = backward
    return span


@torch.inference_mode()
def _prepare_step(case, seed):
    from petals_amd.server.span_engine import SpanEngine, StepEntry

    span = _Span(case, seed)
    rows, before, width = _rows(case), case["context"], span.config.hidden_size
    longest = before + max(rows) + ROOM
    pool = SpanEngine.pool_for(
        span.blocks, len(rows) * (longest + ROOM), dtype=BF16, device=torch.device("cuda"), max_sequences=len(rows)
    )
    engine = SpanEngine(dict(enumerate(span.blocks)), pool, max_length=longest)
    uids = tuple(range(case["blocks"]))
    entries = []
    for i, n in enumerate(rows):
        sequence = pool.open()
        x = _stream(seed, f"row{i}", before + n, width, dtype=torch.float32)
        if before:
            _raise(engine.step(uids, [StepEntry(sequence, x[:before], 0)]))
        entries.append(StepEntry(sequence, x[before:], before))

    def one_pass():
        return _raise(engine.step(uids, entries))

    span.run = one_pass
    return span


def _raise(results):
    for r in results:
        if isinstance(r, BaseException):
            raise r
    return results


# ------------------------------------------------------------- the same in 64 bits


def _rms(x, weight, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight


def _nf4(w):
    """[out, in] -> what 4-bit levels in blocks of 64 outputs hold of it"""
    t = w.t().contiguous().float()  # [in, out]
    parts = t.view(t.shape[0], -1, 64)
    top = parts.abs().amax(-1, keepdim=True)
    scaled = parts * torch.where(top > 0, 1.0 / top, torch.zeros_like(top))
    levels = torch.tensor(NF4_LEVELS, device=t.device)
    edges = ((levels[1:].double() + levels[:-1].double()) / 2).float()
    code = torch.bucketize(scaled, edges)
    return (levels[code].to(F64) * top.to(F64)).view_as(t).t()


def _int8(w):
    t = w.t().float()
    scale = t.abs().amax(dim=0).clamp_min(1e-8) / 127.0
    return (torch.round(t / scale).clamp(-127, 127).to(F64) * scale.to(BF16).to(F64)).t()


class _Exact:
    """Blocks of a case in 64 bits."""

    def __init__(self, case, seed):
        self.case, self.seed = case, seed

    def load(self, block):
        self.w = _weights(self.case, self.seed, block)

    def linear(self, x, name, bias=False):
        w = self.w[name + ".weight"]
        # routers stay as they are
        if not name.endswith("moe.gate"):
            w = {"nf4": _nf4, "int8": _int8}.get(_quantized(self.case), lambda t: t)(w)
        y = x @ w.to(F64).t()
        return y + self.w[name + ".bias"].to(F64) if bias else y

    def norm(self, x, name):
        w = self.w[name + ".weight"].to(F64)
        if name + ".bias" not in self.w:
            return _rms(x, w, 1e-5)
        return torch.nn.functional.layer_norm(x, x.shape[-1:], w, self.w[name + ".bias"].to(F64), 1e-5)

    def rotated(self, x, start):
        """x [B, H, S, hd]: halves turned against each other"""
        half = x.shape[-1] // 2
        base = ROPE_BASE.get(self.case["model"], 10000.0)
        freqs = base ** (-torch.arange(half, device=x.device, dtype=F64) / half)
        angle = torch.arange(start, start + x.shape[2], device=x.device, dtype=F64)[:, None] * freqs
        cos, sin = angle.cos(), angle.sin()
        u, v = x[..., :half], x[..., half:]
        return torch.cat([u * cos - v * sin, v * cos + u * sin], dim=-1)

    def attend(self, q, k, v, before, slopes=None):
        """q [B, H, S, hd], k and v [B, KV, L, hd] -> [B, S, H * hd]"""
        b, heads, s, hd = q.shape
        kv, length = k.shape[1], k.shape[2]
        seen = torch.arange(length, device=q.device)[None] <= torch.arange(before, before + s, device=q.device)[:, None]
        out = []
        for i in range(b):
            for g in range(kv):
                group = q[i, g * (heads // kv) : (g + 1) * (heads // kv)]
                done = []
                step = max(1, (1 << 26) // (s * length))  # heads at a time
                for j in range(0, group.shape[0], step):
                    score = group[j : j + step] @ k[i, g].t() / math.sqrt(hd)
                    if slopes is not None:
                        at = g * (heads // kv) + j
                        score = score + slopes[at : at + score.shape[0], None, None] * torch.arange(length, device=q.device)
                    done.append(torch.softmax(score.masked_fill(~seen, float("-inf")), dim=-1) @ v[i, g])
                out.append(torch.cat(done))
        return torch.cat(out).view(b, heads, s, hd).transpose(1, 2).reshape(b, s, heads * hd)

    def split(self, fused, family, heads, kv, hd):
        b, s, _ = fused.shape
        if family == "bloom":
            q, k, v = fused.view(b, s, heads, 3, hd).unbind(3)
        else:
            parts = fused.view(b, s, kv, heads // kv + 2, hd)
            q, k, v = parts[..., :-2, :].reshape(b, s, heads, hd), parts[..., -2, :], parts[..., -1, :]
        return (t.transpose(1, 2) for t in (q, k, v))

    def block(self, x, before=0, cache=None):
        """x [B, S, h] -> (the block's output, keys, values); cache: those of the tokens before"""
        family, h, heads, kv, _, _ = MODELS[self.case["model"]]
        hd = h // heads
        if family in ("llama", "mixtral"):
            n = self.norm(x, "input_layernorm")
            q, k, v = (
                self.linear(n, f"self_attn.{c}_proj").unflatten(-1, (-1, hd)).transpose(1, 2) for c in "qkv"
            )
        else:
            n = self.norm(x, "ln_attn" if "ln_attn.weight" in self.w else "input_layernorm")
            fused = self.linear(n, "self_attention.query_key_value", bias=family == "bloom")
            q, k, v = self.split(fused, family, heads, kv, hd)
        slopes = None
        if family == "bloom":  # 32 heads
            slopes = 2.0 ** (-8.0 / heads * torch.arange(1, heads + 1, device=x.device, dtype=F64))
        else:
            q, k = self.rotated(q, before), self.rotated(k, before)
        ks, vs = (k, v) if cache is None else (torch.cat([c, t], dim=2) for c, t in zip(cache, (k, v)))
        y = self.attend(q, ks, vs, before, slopes)
        if family == "llama" or family == "mixtral":
            x = x + self.linear(y, "self_attn.o_proj")
            n = self.norm(x, "post_attention_layernorm")
            return x + (self.gated(n) if family == "llama" else self.experts(n)), ks, vs
        y = self.linear(y, "self_attention.dense", bias=family == "bloom")
        if family == "bloom":
            x = x + y
            n = self.norm(x, "post_attention_layernorm")
        else:
            n = self.norm(x, "ln_mlp") if "ln_mlp.weight" in self.w else n
            x = x + y
        inner = torch.nn.functional.gelu(self.linear(n, "mlp.dense_h_to_4h", family == "bloom"), approximate="tanh")
        return x + self.linear(inner, "mlp.dense_4h_to_h", family == "bloom"), ks, vs

    def gated(self, n):
        gate, up = self.linear(n, "mlp.gate_proj"), self.linear(n, "mlp.up_proj")
        return self.linear(torch.nn.functional.silu(gate) * up, "mlp.down_proj")

    def experts(self, n):
        x = n.flatten(0, 1)
        score = torch.softmax(self.linear(x, "block_sparse_moe.gate"), dim=-1)
        weight, chosen = torch.topk(score, TOP, dim=-1)
        weight = weight / weight.sum(-1, keepdim=True)
        out = torch.zeros_like(x)
        for e in range(EXPERTS):
            rows, slots = torch.where(chosen == e)
            if len(rows):
                at = f"block_sparse_moe.experts.{e}."
                inner = torch.nn.functional.silu(self.linear(x[rows], at + "w1")) * self.linear(x[rows], at + "w3")
                out = out.index_add(0, rows, self.linear(inner, at + "w2") * weight[rows, slots, None])
        return out.view_as(n)

    # ------------------------------------------------------------ paged families

    def tulezen(self, x):
        """x [S, width], one whole sequence"""
        m, w = TULEZEN, self.w
        heads, dim = m["heads"], m["dim"]
        c = _rms(x @ w["dkv"].to(F64).t(), w["dkv_norm"].to(F64), 1e-6)
        q = (x @ w["q"].to(F64).t()).unflatten(-1, (heads, dim)).transpose(0, 1)
        k = (c @ w["uk"].to(F64).t()).unflatten(-1, (heads, dim)).transpose(0, 1)
        v = (c @ w["uv"].to(F64).t()).unflatten(-1, (heads, dim)).transpose(0, 1)
        pos = torch.arange(x.shape[0], device=x.device)
        gap = pos[:, None] - pos[None]
        score = (q @ k.transpose(1, 2) * dim**-0.5).masked_fill((gap < 0) | (gap >= m["window"]), float("-inf"))
        y = (torch.softmax(score, dim=-1) @ v).transpose(0, 1).flatten(1) @ w["o"].to(F64).t()
        x = x + _rms(y, 1.0 + w["norm1"].to(F64), 1e-6)
        weight, chosen = torch.topk(torch.softmax(x @ w["router"].to(F64).t(), dim=-1), m["top"], dim=-1)
        out = torch.zeros_like(x)
        for e in range(m["experts"]):
            rows, slots = torch.where(chosen == e)
            if len(rows):
                gate = (x[rows] @ w["gate"][e].to(F64).t()).clamp(max=m["limit"])
                up = (x[rows] @ w["up"][e].to(F64).t()).clamp(-m["limit"], m["limit"])
                inner = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
                out.index_add_(0, rows, inner @ w["down"][e].to(F64).t() * weight[rows, slots, None])
        return x + _rms(out, 1.0 + w["norm2"].to(F64), 1e-6)

    def zudarax(self, x):
        m, w = ZUDARAX, self.w
        heads, dim, vdim, s = m["heads"], m["dim"], m["vdim"], x.shape[0]
        n = _rms(x.unflatten(-1, (m["groups"], -1)), 1.0, 1e-6).flatten(-2) * w["norm1"].to(F64)
        half = dim // 2
        freqs = 10000.0 ** (-torch.arange(half, device=x.device, dtype=F64) / half)
        pos = torch.arange(s, device=x.device)
        cos, sin = (f(pos.to(F64)[:, None, None, None] * freqs) for f in (torch.cos, torch.sin))
        turned = []
        for name in "qk":
            t = (n @ w[name].to(F64).t()).view(s, heads, 2, dim)
            a, b = t[..., :half], t[..., half:]
            turned.append(torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1).permute(1, 2, 0, 3))
        q, k = turned  # [H, 2, S, dim]
        v = (n @ w["v"].to(F64).t()).view(s, heads, vdim).transpose(0, 1)
        seen = pos[:, None] >= pos[None]
        first = (w["lq1"].to(F64) * w["lk1"].to(F64)).sum().exp()
        share = first - (w["lq2"].to(F64) * w["lk2"].to(F64)).sum().exp() + m["diff"]
        y = []
        for i in range(heads):
            p = torch.softmax((q[i] @ k[i].transpose(1, 2) * dim**-0.5).masked_fill(~seen, float("-inf")), dim=-1)
            y.append((p[0] - share * p[1]) @ v[i])
        y = _rms(torch.stack(y, dim=1), 1.0 - m["diff"], 1e-6)  # [S, H, vdim]
        y = y * torch.sigmoid(n @ w["g"].to(F64).t())[..., None]
        z = n @ w["up"].to(F64).t()
        a, b, c, e = w["act"].to(F64)
        inner = a * _rms(z, 1.0, 1e-6) + b * _rms(z * z, 1.0, 1e-6) + c * _rms(z * z * z, 1.0, 1e-6) + e
        return x + y.flatten(1) @ w["o"].to(F64).t() + inner @ w["down"].to(F64).t()


def exact(case, seed):
    e = _Exact(case, seed)
    if case["kind"] == "step":
        rows, before = _rows(case), case["context"]
        width = (TULEZEN if case["model"] == "tulezen" else ZUDARAX)["width"]
        xs = [_stream(seed, f"row{i}", before + n, width, dtype=torch.float32).to(F64) for i, n in enumerate(rows)]
        for i in range(case["blocks"]):
            e.load(i)
            xs = [getattr(e, case["model"])(x) for x in xs]
        return [x[before:] for x in xs]
    width = MODELS[case["model"]][1]
    new = case.get("tokens", 1)
    x = _stream(seed, "hidden", case["batch"], new, width).to(F64)
    if case["kind"] == "backward":
        return _exact_backward(case, seed, e, x)
    before, caches = case.get("context", 0), []
    with torch.no_grad():
        for i in range(case["blocks"]):
            e.load(i)
            cache = None
            if case["kind"] == "decode":
                cache = [t[:, :, :before].to(F64) for t in _cached(case, seed, i)]
            x, k, v = e.block(x, before, cache)
            if case["kind"] != "forward":
                room = (0, 0, 0, before + new + ROOM - (new if case["kind"] == "decode" else 0) - k.shape[2])
                caches += [torch.nn.functional.pad(t, room) for t in (k, v)]
    return [x, *caches]


def _exact_backward(case, seed, e, x):
    inputs = []
    for i in range(case["blocks"]):
        prompt = _stream(seed, f"prompt{i}", case["batch"], PROMPT_ROWS, x.shape[-1]).to(F64)
        x = x.clone()
        x[:, :PROMPT_ROWS] += prompt
        inputs.append(x)
        if i + 1 < case["blocks"]:
            e.load(i)
            with torch.no_grad():
                x = e.block(x)[0]
    g, grads = _stream(seed, "grad", case["batch"], case["tokens"], x.shape[-1]).to(F64), []
    for i in reversed(range(case["blocks"])):
        e.load(i)
        with torch.enable_grad():
            leaf = inputs[i].detach().requires_grad_(True)
            (g,) = torch.autograd.grad(e.block(leaf)[0], leaf, g)
        grads.insert(0, g[:, :PROMPT_ROWS].clone())
    return [g, torch.stack(grads)]
