"""The work a user of this package has it do, as measurable cases.

Every case goes through the public Python surface: a transformers model (or a plain module) split by `tp.tensor_parallel` /
`tp.TensorParallel` into two rank shards that share the GPU, run as a serving or scoring program runs it, and the slicing of
state dicts in both directions. Shapes are those of the repository's own configurations: a Llama-2-7B-shaped decoder
(d 4096, ffn 11008, heads of 128, vocabulary 32000; two layers stand for the 32), a Falcon-40B-shaped layer with int8 weights,
OPT-125m in fp32, and the state dict of Llama-2-7B-shaped layers.

kinds:
  decode          one new token per sequence on a static cache, the step recorded as a HIP graph and replayed
  prefill         a prompt through the model into an empty growing cache, logits of the last position (what `generate` does first)
  score           logits of every position of a batch of whole sequences, no cache
  mlp             the gated MLP block alone, through `tp.TensorParallel`
  falcon_decode   a decode step of the int8 Falcon-shaped layer on a static cache, recorded and replayed
  falcon_prefill  a prompt through that layer into an empty growing cache
  opt             OPT-125m in fp32, eager
  convert         `tp.convert_state_dict` of a device-resident state dict
  unshard         the full state dict of a wrapped model (`tp.save_tensor_parallel`)
"""
from types import SimpleNamespace

import torch
from torch import nn

import tensor_parallel_amd as tp

WORLD = 2
DEV = "cuda:0"
LAYERS = 2  # decoder layers of the Llama-shaped models
D, FFN, HEADS, HEAD_DIM, VOCAB = 4096, 11008, 32, 128, 32000
F_D, F_HEADS, F_KV, F_HEAD_DIM = 8192, 128, 8, 64  # the Falcon-40B-shaped layer
ROOM = 64  # free positions of a static cache before a program would have to stop or start over


def listed():
    return [
        # one user chatting: the smallest call of a serving loop, bound by the weights and by launches
        {"name": "decode 1 on 500", "kind": "decode", "batch": 1, "cached": 500, "kv_heads": 32, "dtype": "bf16"},
        # a small serving batch on long contexts (the batch and length of the decode configurations)
        {"name": "decode 8 on 2048", "kind": "decode", "batch": 8, "cached": 2048, "kv_heads": 32, "dtype": "bf16"},
        # a larger, ragged serving batch of a grouped-query model in fp16
        {"name": "decode 40 on 1000 gqa", "kind": "decode", "batch": 40, "cached": 1000, "kv_heads": 8, "dtype": "f16"},
        # scoring (perplexity, reranking) of a few short odd-sized sequences
        {"name": "score 5x129", "kind": "score", "batch": 5, "seq": 129, "kv_heads": 32, "dtype": "bf16"},
        # a few prompts of a length that divides nothing, grouped-query, fp16
        {"name": "prefill 3x701 gqa", "kind": "prefill", "batch": 3, "seq": 701, "kv_heads": 8, "dtype": "f16"},
        # long prompts: 4096 tokens at once, the largest work here
        {"name": "prefill 2x2048", "kind": "prefill", "batch": 2, "seq": 2048, "kv_heads": 32, "dtype": "bf16"},
        # the MLP block on its own at the middle size of its configuration (1, 16, 512 and 4096 rows; the others are parts of
        # the decode and prefill cases)
        {"name": "mlp 512", "kind": "mlp", "rows": 512, "dtype": "bf16"},
        # int8 serving: decode of a Falcon-40B-shaped layer
        {"name": "falcon int8 decode 16", "kind": "falcon_decode", "batch": 16, "cached": 2048, "dtype": "f16"},
        # and its prompt
        {"name": "falcon int8 prefill 1024", "kind": "falcon_prefill", "batch": 1, "seq": 1024, "dtype": "f16"},
        # the small fp32 model of the first configuration, run eagerly as its users do
        {"name": "opt125m fp32 2x64", "kind": "opt", "batch": 2, "seq": 64},
        # loading: four decoder layers sliced for all ranks
        {"name": "convert 4 layers", "kind": "convert", "layers": 4, "embeddings": False, "world": 2, "d": 4096, "ffn": 11008, "dtype": "bf16"},
        # saving: the whole model back from its shards
        {"name": "unshard 2 layers", "kind": "unshard", "layers": 2, "ffn": 11008, "kv_heads": 32, "dtype": "bf16"},
    ]


def _log(rng, low, high):
    """A whole number between low and high, spread evenly over its logarithm."""
    return max(low, min(high, round(low * (high / low) ** rng.random())))


def draw(rng):
    kind = rng.choice(["decode"] * 3 + ["prefill"] * 2 + ["score"] * 2 + ["mlp", "falcon_decode", "falcon_prefill", "opt", "convert", "unshard"])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    kv_heads = rng.choice([32, 8])
    if kind == "decode":
        batch = _log(rng, 1, 64)
        return {"kind": kind, "batch": batch, "cached": _log(rng, 60, min(4096, 65536 // batch)), "kv_heads": kv_heads, "dtype": dtype}
    if kind in ("prefill", "score"):
        tokens = _log(rng, 128 if kind == "prefill" else 32, 4096 if kind == "prefill" else 2048)
        batch = rng.choice([1, 1, 2, 3, 5])
        return {"kind": kind, "batch": batch, "seq": max(8, tokens // batch), "kv_heads": kv_heads, "dtype": dtype}
    if kind == "mlp":
        return {"kind": kind, "rows": _log(rng, 64, 8192), "dtype": dtype}
    if kind == "falcon_decode":
        batch = _log(rng, 1, 64)
        return {"kind": kind, "batch": batch, "cached": _log(rng, 60, 4096), "dtype": dtype}
    if kind == "falcon_prefill":
        return {"kind": kind, "batch": rng.choice([1, 1, 2]), "seq": _log(rng, 100, 1024), "dtype": dtype}
    if kind == "opt":
        return {"kind": kind, "batch": rng.choice([1, 2, 3, 4]), "seq": _log(rng, 8, 256)}
    if kind == "convert":
        world = rng.choice([2, 2, 4, 4, 8])
        d = rng.choice([1024, 2048, 4096, 5120])
        layers = {2: rng.choice([1, 2, 3]), 4: 1, 8: 1}[world]
        return {"kind": kind, "layers": layers, "embeddings": world < 8 and rng.random() < 0.5, "world": world, "d": d,
                "ffn": rng.choice([8 * d // 3 + 85, 11008, 3 * d, 13824]), "dtype": rng.choice([dtype, dtype, "f32"])}
    return {"kind": kind, "layers": rng.choice([1, 2, 3]), "ffn": rng.choice([11008, 8192, 14336, 5502]), "kv_heads": kv_heads, "dtype": dtype}


# ---- preparation -------------------------------------------------------------------------------------------------------
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _random_weights(model, seed):
    """N(0, 0.02) in every matrix, ones and zeros in the norms, as a freshly initialised model has them."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() > 1:
                p.normal_(0.0, 0.02, generator=gen)
    return gen


def _tokens(gen, vocab, *shape):
    return torch.randint(0, vocab, shape, device=DEV, generator=gen)


def _llama(case, seed, positions):
    from transformers import LlamaConfig, LlamaForCausalLM

    config = LlamaConfig(vocab_size=VOCAB, hidden_size=D, intermediate_size=case.get("ffn", FFN), num_hidden_layers=case.get("layers", LAYERS), num_attention_heads=HEADS,
                         num_key_value_heads=case["kv_heads"], head_dim=HEAD_DIM, max_position_embeddings=max(4096, positions),
                         attn_implementation="eager")
    with torch.device(DEV):
        model = LlamaForCausalLM(config).to(DTYPES[case["dtype"]]).eval()
    gen = _random_weights(model, seed)
    model.config._attn_implementation = tp.attention.register()
    return tp.tensor_parallel(model, [DEV] * WORLD), config, gen


def _falcon(case, seed):
    from transformers import FalconConfig, FalconModel

    config = FalconConfig(vocab_size=1024, hidden_size=F_D, num_hidden_layers=1, num_attention_heads=F_HEADS, num_kv_heads=F_KV,
                          new_decoder_architecture=True, alibi=False, bias=False, max_position_embeddings=8192)
    with torch.device(DEV):
        model = FalconModel(config).to(DTYPES[case["dtype"]]).eval()
    gen = _random_weights(model, seed)
    split = tp.tensor_parallel(model, [DEV] * WORLD)
    tp.attention.fuse_rotary_(split, assume_no_padding=True)
    columns = torch.Generator().manual_seed(seed)  # half a per cent of the input columns stay in 16 bits, at random

    def outliers(name, linear):
        n = linear.in_features
        return torch.randperm(n, generator=columns)[: n // 200].tolist()

    tp.int8.quantize_linears_(split, outlier_cols=outliers)
    return split, config, gen


class _Mlp(nn.Module):
    """The gated MLP of a Llama-pattern decoder layer."""

    def __init__(self):
        super().__init__()
        self.gate_proj, self.up_proj = nn.Linear(D, FFN, bias=False), nn.Linear(D, FFN, bias=False)
        self.down_proj = nn.Linear(FFN, D, bias=False)
        self.act_fn = nn.SiLU()

    def forward(self, x):
        return self.down_proj(self.act_fn(self.gate_proj(x)) * self.up_proj(x))


class _Block(nn.Module):
    def __init__(self):
        super().__init__()
        self.mlp = _Mlp()

    def forward(self, x):
        return self.mlp(x)


def _llama_rules(d, heads, world):
    from tensor_parallel_amd.slicing_configs import get_llama_config

    shape = SimpleNamespace(model_type="llama", hidden_size=d, num_attention_heads=heads, num_key_value_heads=heads)
    return get_llama_config(shape, [torch.device(DEV)] * world)


def _cache_tensors(cache):
    return [t for c in tp.kv_cache.rank_caches(cache, WORLD) for layer in c.layers for t in (layer.keys, layer.values)]


_side_stream = None  # the stream that a program records its graphs on


def _recorded_decode(model, config, case, gen, vocab):
    """The static cache after its prompt, the recorded step and the next token: what a serving loop holds between steps."""
    from transformers import StaticCache

    global _side_stream
    if _side_stream is None:
        _side_stream = torch.cuda.Stream()
    cache = StaticCache(config=config, max_cache_len=case["cached"] + ROOM)
    prompt, token = _tokens(gen, vocab, case["batch"], case["cached"]), _tokens(gen, vocab, case["batch"], 1)
    model(input_ids=prompt, past_key_values=cache, use_cache=True, **({"logits_to_keep": 1} if case["kind"] == "decode" else {}))
    counts = [layer.cumulative_length for c in tp.kv_cache.rank_caches(cache, WORLD) for layer in c.layers]
    _side_stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(_side_stream):
        for _ in range(2):  # first uses happen outside the recording
            model(input_ids=token, past_key_values=cache, use_cache=True)
    torch.cuda.current_stream().wait_stream(_side_stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=_side_stream):
        out = model(input_ids=token, past_key_values=cache, use_cache=True)
    for count in counts:
        count.fill_(case["cached"])
    return {"graph": graph, "out": out.logits if case["kind"] == "decode" else out.last_hidden_state, "model": model, "token": token,
            "next": token.clone(), "cache": cache, "counts": counts, "start": case["cached"], "taken": 0, "cached": _cache_tensors(cache)}


def prepare(case, seed):
    kind, dtype = case["kind"], DTYPES[case.get("dtype", "f32")]
    with torch.no_grad():
        if kind == "decode":
            model, config, gen = _llama(case, seed, case["cached"] + ROOM)
            tp.attention.fuse_rotary_(model, assume_no_padding=True)
            state = _recorded_decode(model, config, case, gen, VOCAB)
        elif kind == "prefill":
            model, _, gen = _llama(case, seed, case["seq"])
            tp.attention.fuse_rotary_(model)
            state = {"model": model, "ids": _tokens(gen, VOCAB, case["batch"], case["seq"])}
            _warm(model, gen, VOCAB)
        elif kind == "score":
            model, _, gen = _llama(case, seed, case["seq"])
            state = {"model": model, "ids": _tokens(gen, VOCAB, case["batch"], case["seq"])}
            model(input_ids=_tokens(gen, VOCAB, 1, 8), use_cache=False)  # the first call decides which kernels the modules use
        elif kind == "mlp":
            with torch.device(DEV):
                block = _Block().to(dtype)
            gen = _random_weights(block, seed)
            model = tp.TensorParallel(block, [DEV] * WORLD, tensor_parallel_config=_llama_rules(D, HEADS, WORLD), sharded=False)
            state = {"model": model, "x": torch.randn(case["rows"], D, device=DEV, generator=gen).to(dtype)}
            model(state["x"][:8])  # a program's first call decides which kernels its modules use
        elif kind == "falcon_decode":
            model, config, gen = _falcon(case, seed)
            state = _recorded_decode(model, config, case, gen, 1024)
        elif kind == "falcon_prefill":
            model, _, gen = _falcon(case, seed)
            state = {"model": model, "ids": _tokens(gen, 1024, case["batch"], case["seq"])}
            _warm(model, gen, 1024)
        elif kind == "opt":
            from transformers import OPTConfig, OPTForCausalLM

            with torch.device(DEV):
                model = OPTForCausalLM(OPTConfig()).eval()
            gen = _random_weights(model, seed)
            model = tp.tensor_parallel(model, [DEV] * WORLD)
            state = {"model": model, "ids": _tokens(gen, 50272, case["batch"], case["seq"])}
        elif kind == "convert":
            d, ffn = case["d"], case["ffn"]
            gen = torch.Generator(device=DEV).manual_seed(seed)
            shapes = {}
            for layer in range(case["layers"]):
                at = f"model.layers.{layer}."
                shapes.update({f"{at}self_attn.{n}_proj.weight": (d, d) for n in "qkvo"})
                shapes.update({f"{at}mlp.gate_proj.weight": (ffn, d), f"{at}mlp.up_proj.weight": (ffn, d), f"{at}mlp.down_proj.weight": (d, ffn)})
            if case["embeddings"]:
                shapes.update({"model.embed_tokens.weight": (VOCAB, d), "lm_head.weight": (VOCAB, d)})
            weights = {n: torch.empty(s, device=DEV, dtype=dtype).normal_(0.0, 0.02, generator=gen) for n, s in shapes.items()}
            state = {"weights": weights, "rules": _llama_rules(d, d // HEAD_DIM, case["world"]), "world": case["world"]}
        else:
            model, _, _ = _llama(case, seed, 4096)
            state = {"model": model}
    state["kind"] = kind
    return state


def _warm(model, gen, vocab):
    """A short prompt: the first call decides which kernels the modules of a model use."""
    from transformers import DynamicCache

    model(input_ids=_tokens(gen, vocab, 1, 8), past_key_values=DynamicCache(), use_cache=True)


# ---- one pass ----------------------------------------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    with torch.no_grad():
        if kind in ("decode", "falcon_decode"):
            if state["taken"] == ROOM:  # the cache is full: the next sequence starts behind the same prompt
                for count in state["counts"]:
                    count.fill_(state["start"])
                state["taken"] = 0
            state["taken"] += 1
            state["token"].copy_(state["next"])
            state["graph"].replay()
            return [state["out"], *state["cached"]]
        if kind == "score":
            return state["model"](input_ids=state["ids"], use_cache=False).logits
        if kind in ("prefill", "falcon_prefill"):
            from transformers import DynamicCache

            cache = DynamicCache()
            if kind == "prefill":
                out = state["model"](input_ids=state["ids"], past_key_values=cache, use_cache=True, logits_to_keep=1).logits
            else:
                out = state["model"](input_ids=state["ids"], past_key_values=cache, use_cache=True).last_hidden_state
            return [out, *_cache_tensors(cache)]
        if kind == "mlp":
            return state["model"](state["x"])
        if kind == "opt":
            return state["model"](input_ids=state["ids"], use_cache=False).logits
        if kind == "convert":
            shards = tp.convert_state_dict(state["weights"], state["rules"], state["world"])
            return {name: t for name, t in shards.items() if name.endswith(".weight")}
        with tp.save_tensor_parallel(state["model"]):
            return dict(state["model"].state_dict())


# ---- what a pass cannot do without --------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    size = {"bf16": 2, "f16": 2, "f32": 4}[case.get("dtype", "f32")]
    if kind in ("decode", "prefill", "score", "unshard"):
        kv = case["kv_heads"] * HEAD_DIM
        layer = 2 * D * D + 2 * D * kv + 3 * D * case.get("ffn", FFN)
        weights = case.get("layers", LAYERS) * layer + VOCAB * D
        if kind == "unshard":
            return {"bytes": 2.0 * size * (weights + VOCAB * D), "flops": 0.0}
        b = case["batch"]
        if kind == "decode":
            t = case["cached"]
            return {"bytes": size * (weights + 2.0 * LAYERS * b * t * kv + b * (2 * D + VOCAB)),
                    "flops": 2.0 * b * weights + 4.0 * LAYERS * b * t * D}
        s = case["seq"]
        logits = b * (s if kind == "score" else 1)
        return {"bytes": size * (weights + b * s * D + logits * VOCAB + (2.0 * LAYERS * b * s * kv if kind == "prefill" else 0)),
                "flops": 2.0 * b * s * LAYERS * layer + 2.0 * logits * VOCAB * D + 2.0 * LAYERS * b * s * s * D}
    if kind == "mlp":
        m = case["rows"]
        return {"bytes": size * (3.0 * D * FFN + 2.0 * m * D), "flops": 6.0 * m * D * FFN}
    if kind in ("falcon_decode", "falcon_prefill"):
        kv = F_KV * F_HEAD_DIM
        weights = 2 * F_D * F_D + 2 * F_D * kv + 8 * F_D * F_D
        b = case["batch"]
        if kind == "falcon_decode":
            t = case["cached"]
            return {"bytes": weights * 1.01 + size * (2.0 * b * t * kv + 2.0 * b * F_D), "flops": 2.0 * b * weights + 4.0 * b * t * F_D}
        s = case["seq"]
        return {"bytes": weights * 1.01 + size * (2.0 * b * s * kv + 2.0 * b * s * F_D), "flops": 2.0 * b * s * weights + 2.0 * b * s * s * F_D}
    if kind == "opt":
        rows, d, layers, vocab = case["batch"] * case["seq"], 768, 12, 50272
        weights = layers * 12 * d * d + vocab * d
        return {"bytes": 4.0 * (weights + rows * vocab), "flops": 2.0 * rows * weights + 2.0 * layers * rows * case["seq"] * d}
    elements = case["layers"] * (4 * case["d"] ** 2 + 3 * case["d"] * case["ffn"]) + (2 * VOCAB * case["d"] if case["embeddings"] else 0)
    return {"bytes": 2.0 * size * elements, "flops": 0.0}


def tolerance(case):
    """Measured against the same model in fp32 (fp64 for the fp32 one) with the same weights: a bf16 model's logits are 1.6e-2 to
    1.9e-2 off and its second layer's keys 1.3e-2, an fp16 model's 2.0e-3 to 2.2e-3, the bf16 / fp16 MLP block alone 4.3e-3 /
    5.3e-4, OPT-125m in fp32 8e-7; the largest single differences are five times that."""
    if case["kind"] in ("convert", "unshard"):
        return "exact"
    if case["kind"] == "opt":
        return {"rel": 4e-6, "max": 4e-5}
    if case["kind"] == "mlp":
        return {"rel": 1.7e-2, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 2e-3, "max": 1.2e-2}
    return {"rel": 2.8e-2, "max": 0.35} if case["dtype"] == "bf16" else {"rel": 8e-3, "max": 5e-2}
