"""Shard-local compute modules: the Linear layers of a rank's shard run on the HIP kernels.

In the reference a shard is a deep copy of the user's module whose `torch.nn.Linear`s hold sliced weights and
run ATen GEMMs (src/tensor_parallel/shard.py:160,184-187; wrapper.py:69-72). Here every `nn.Linear` of a shard
is re-classed to `ShardLinear` (same parameters, same attributes, still an `nn.Linear`), and SiLU-gated MLP
blocks with `gate_proj` / `up_proj` / `down_proj` children get a fused gate/up forward. transformers' `Conv1D`
(GPT-2's c_attn / c_proj / c_fc: weight kept as [in, out] and multiplied as x @ w, sliced by
src/tensor_parallel/slicing_configs.py:192-201) is re-classed to a subclass whose forward is the same `tpamd_linear`:
its weight keeps the [in, out] shape every rule and state dict expects but is stored with the `in` axis fastest, which
is the kernel's [out, in] layout; the transposing mover writes it that way while slicing, or once at the first forward.
`nn.LayerNorm`, transformers' `LlamaRMSNorm` and the rotary tables of Llama and Falcon, which every rank computes whole, become one launch
each (`tpamd_layer_norm_ranks`, `tpamd_rms_norm`, `tpamd_rope_tables`) in the same way; a Llama decoder layer has the addition behind its attention in the
launch of its second norm (`tpamd_add_rms_norm`).

Inference only: the kernels have no backward; asking for one raises. Autocast is not applied by these modules: the
input must already have the weight's dtype (a mismatch raises TypeError where `nn.Linear` under autocast would cast).
"""
from __future__ import annotations

import types

import torch
from torch import nn

from . import _native, together
from .slicing import is_k_major


class _NoBackward(torch.autograd.Function):
    """Marks a kernel result so that a backward pass through it fails loudly instead of silently stopping."""

    @staticmethod
    def forward(ctx, out, *inputs):
        return out.view_as(out)

    @staticmethod
    def backward(ctx, *grads):
        raise NotImplementedError("tensor_parallel_amd kernels are inference-only: no backward is implemented")


def _guard(out: torch.Tensor, *inputs: torch.Tensor) -> torch.Tensor:
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in inputs):
        return _NoBackward.apply(out, *inputs)
    return out


def linear_in_context(module: nn.Module, x: torch.Tensor, w: torch.Tensor, bias) -> torch.Tensor:
    """`tpamd_linear` for a shard's Linear; see `product_in_context`."""
    xd, wd, b = x.detach(), w.detach(), None if bias is None else bias.detach()
    return product_in_context(module, x, w.shape[0], (x, w, bias), lambda: together.linear(xd, wd, b), lambda **more: _native.linear(xd, wd, b, **more),
                              lambda rank, op: together.linear_sum(xd, wd, b, rank, op))


def product_in_context(module: nn.Module, x: torch.Tensor, columns: int, inputs: tuple, with_peers, alone, summed, learned: bool = True) -> torch.Tensor:
    """A shard's Linear with `columns` outputs, made by with_peers() or, with an addend, alone(addend=, copy=). Inside a wrapped module whose output goes to a
    "sum" rule (collectives.SumContext) the Linear that was seen to produce that output hands over the sum: two ranks that meet in it get it from
    summed(rank, op) (`tpamd_linear_sum_ranks`; None: not to be had), else the rank that comes last adds the partial sums already waiting in
    the reduction, in its epilogue (`tpamd_linear_add`): the product rounded to the dtype, then one rounded add, which
    is the same arithmetic as the reduction kernel's step. `learned`: having been seen to produce it is enough (see _may_hold_sum)."""
    ctx = together.current_sum_context()
    if ctx is None:
        return _guard(with_peers(), *inputs)
    key = id(module)
    ctx.calls[key] = ctx.calls.get(key, 0) + 1
    out, more = None, {}
    if module.__dict__.get("_tp_feeds_sum") is ctx.owner and ctx.owner is not None and _may_hold_sum(module, ctx, learned):
        if ctx.fused_out is not None:
            raise RuntimeError("tensor_parallel_amd: the Linear that feeds a \"sum\" rule ran twice in one call of its module "
                               "after adding the waiting partial sums; set TPAMD_FUSE_SUM=0")
        waiting = ctx.op.addend_for(ctx.rank)
        if waiting is None and summed is not None and ctx.op.world_size == 2 and _is_last_child(module, ctx.wrapped):
            out = summed(ctx.rank, ctx.op)
        if out is not None:
            out = _guard(out, *inputs)
            ctx.fused_mask, ctx.fused_whole = 3, True
        else:
            if waiting is None:  # (a rank that waited for its peer in vain finds what that one has handed in since)
                waiting = ctx.op.addend_for(ctx.rank)
            if waiting is not None:
                t, mask = waiting
                if t.dtype == x.dtype and t.device == x.device and t.shape == (*x.shape[:-1], columns):
                    more["addend"], ctx.fused_mask = t.detach(), mask
                    if ctx.op.world_size == 2:  # the sum is complete then: a second tensor for the other rank comes out of the same launch
                        more["copy"] = torch.empty_like(more["addend"], memory_format=torch.contiguous_format)
            out = _guard(alone(**more), *inputs)
    else:  # ranks meet in other Linears once a first call has shown which one feeds the sum
        out = _guard(with_peers() if "_tp_sum_known" in ctx.owner.__dict__ else alone(), *inputs)
    ctx.last_linear, ctx.last_out = module, out
    ctx.last_version = None if out.is_inference() else out._version  # (changes of an inference tensor are not counted)
    if more or ctx.fused_whole:
        ctx.fused_linear, ctx.fused_out, ctx.fused_version, ctx.fused_copy = module, out, ctx.last_version, more.get("copy")
    return out


def _may_hold_sum(module: nn.Module, ctx, learned: bool) -> bool:
    """Whether a Linear's output may hold other ranks' parts already on its way to the sum: nobody who is told of it there would see or change more than this rank's
    part. Not with hooks on the Linear, on the module around it (the wrapped one) or on all modules, nor with a forward that a program has put around the
    Linear's. Then either the wrapped module is known to return it untouched, or (`learned`) it did so when it was last seen without, and a
    change shows in the tensor's version, which raises; in inference mode versions stand still."""
    wrapped, hooks = ctx.wrapped, torch.nn.modules.module
    if hooks._global_forward_hooks or hooks._global_forward_pre_hooks or _has_hooks(module) or _has_hooks(wrapped) or "forward" in module.__dict__:
        return False
    return learned and not torch.is_inference_mode_enabled() or hands_through(ctx, module)


def _is_last_child(module: nn.Module, wrapped: nn.Module) -> bool:
    """No module lies between the wrapped one and the Linear that feeds its sum, whose hooks would be told of the output."""
    return wrapped is module or any(child is module for child in wrapped._modules.values())


def returned(self: nn.Module, forward, linear: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """linear(x), which this forward of the module `self` (an attribute of it) returns as it is: a wrapper around the module is told."""
    ctx = together.current_sum_context()
    if ctx is not None and ctx.wrapped is self and getattr(self.__dict__.get("forward"), "__func__", None) is forward:
        ctx.returned = linear
    return linear(x)


def hands_through(ctx, module: nn.Module) -> bool:
    """Whether the wrapped module is this Linear, said that it returns what the Linear gives, or has one of the forwards below (or the transformers one it stands in
    for), which do."""
    wrapped = ctx.wrapped
    if wrapped is module or ctx.returned is module:
        return True
    own, cls = wrapped.__dict__.get("forward"), type(wrapped)
    if own is not None:
        return getattr(own, "__func__", None) is _gated_mlp_forward and wrapped._modules.get("down_proj") is module
    last = "o_proj" if cls.forward is _llama_attention_forward else "dense_4h_to_h" if cls.forward is _falcon_mlp_forward else None
    return last is not None and cls._tp_base.forward is cls._tp_replaced and wrapped._modules.get(last) is module


def gathered_linear(module: nn.Module, op, rank: int, args, kwargs):
    """The gathered output of a column-parallel Linear, written by one launch for two ranks (`tpamd_linear_gather_ranks`) instead of a Linear
    for each and a concatenation behind them; None where that is not to be had: another module than a plain shard Linear, somebody who watches its
    own output, another axis, a rank whose peer does not come with a Linear of the same form."""
    hooks = torch.nn.modules.module
    if (type(module) is not ShardLinear or "forward" in module.__dict__ or kwargs or len(args) != 1 or _has_hooks(module)
            or hooks._global_forward_hooks or hooks._global_forward_pre_hooks):
        return None
    x, w, bias = args[0], module.weight, module.bias
    if not _native.plain_call(x, w) or not x.is_cuda or op.dim not in (-1, x.dim() - 1) or x.dtype != w.dtype:
        return None
    whole = together.linear_gathered(x.detach(), w.detach(), None if bias is None else bias.detach(), rank, op.world_size, op)
    return None if whole is None else _guard(whole, x, w, bias)


class ShardLinear(nn.Linear):
    """`nn.Linear` whose forward is `tpamd_linear` on the shard's (sliced) weight."""

    def forward(self, input: torch.Tensor) -> torch.Tensor:  # noqa: A002
        return linear_in_context(self, input, self.weight, self.bias)


def is_conv1d(module: nn.Module) -> bool:
    """transformers.pytorch_utils.Conv1D (or a subclass): a Linear whose weight is [in, out]."""
    return any(c.__name__ == "Conv1D" and c.__module__.split(".")[0] == "transformers" for c in type(module).__mro__) and \
        isinstance(getattr(module, "weight", None), torch.Tensor)


def _conv1d_forward(self, x: torch.Tensor) -> torch.Tensor:
    w = self.weight
    if not is_k_major(w):  # a weight assigned after the shard was built: lay it out for the kernel, once
        with torch.no_grad():
            w.data = _native.transpose_regions(w.data.contiguous(), [(0, w.shape[1])]).t()
    return linear_in_context(self, x, w.t(), getattr(self, "bias", None))


_conv1d_classes: dict = {}


def _shard_conv1d_class(base: type) -> type:
    """Subclass of the module's own Conv1D class with the kernel forward (isinstance checks keep working)."""
    cls = _conv1d_classes.get(base)
    if cls is None:
        cls = _conv1d_classes[base] = type("ShardConv1D", (base,), {"forward": _conv1d_forward, "__doc__": "Conv1D whose forward is `tpamd_linear` "
                                                                   "on the shard's weight, stored with its input axis fastest."})
    return cls


def is_rms_norm(module: nn.Module) -> bool:
    """transformers' LlamaRMSNorm: a weight over the last axis and `variance_epsilon`, statistics in fp32."""
    return type(module).__name__ == "LlamaRMSNorm" and _takes_stand_in(type(module), _rms_norm_forward) and \
        isinstance(getattr(module, "weight", None), torch.Tensor) and module.weight.dim() == 1 and hasattr(module, "variance_epsilon")


_KERNEL_DTYPES = (torch.bfloat16, torch.float16, torch.float32)


def _norm_kernel_takes(x: torch.Tensor, w: torch.Tensor) -> bool:
    """What `tpamd_rms_norm` is made for; a promoting norm, one moved to another dtype (`.double()`) or with a weight that broadcasts is not."""
    return _native.plain_call(x, w) and x.dtype == w.dtype and w.dtype in _KERNEL_DTYPES and w.dim() == 1 and x.dim() > 0 and x.shape[-1] == w.shape[0] \
        and _native.on_hip(x) and x.get_device() == w.get_device()


def _rms_norm_forward(self, hidden_states: torch.Tensor) -> torch.Tensor:
    w, own = self.weight, self._tp_base.forward
    # a norm whose class has been given another forward since, and one that derivatives may go through (they were there before any
    # Linear's), keep the module's own forward
    if own is not self._tp_replaced or not _norm_kernel_takes(hidden_states, w) or torch.is_grad_enabled() and (hidden_states.requires_grad or w.requires_grad):
        return own(self, hidden_states)
    return together.rms_norm(hidden_states, w, self.variance_epsilon)


# torch's kernel works on a row with one wavefront and does short rows as fast (128 rows of 768 in fp32: 4.0 us there, 3.6 here for two ranks at once), while
# its call costs the host less: OPT-125m in fp32, 50 norms of 768 a forward, 5.6 ms eager with torch's and 6.1 with these. 16 rows of 8192 in
# fp16 take 9.3 us there and 4.1 here; 1 to 64 rows of 2048 / 4096 / 8192 in fp32 3.1-3.4 / 3.8-4.2 / 5.4-5.9 for each rank there and 2.3-2.6 / 2.7-3.1 / 3.2-4.0 for both here.
# In between, the host sets the pace of an eager forward with some hundred rows (the Falcon-40B-shaped layer on 150 of them: 890 us
# with torch's norms, 950 with these), so torch's stay there; 1024 rows take 14.4 us there and 7.3 here.
# The rows have to be whole 16-byte chunks, at most as many as a block holds in registers: the kernel for any others reads a row three times, element by element (two ranks' 1024
# rows of 16384 in fp32: 62 us with torch's, 124 with it; of 18432 in bf16 52 and 150, of 8196 28 and 54).
LAYER_NORM_ROW, LAYER_NORM_ROW_BYTES = 2048, 32768
LAYER_NORM_FEW_ROWS, LAYER_NORM_MANY_ROWS = 64, 512


def _layer_norm_pays(w: torch.Tensor) -> bool:
    row = w.numel() * w.element_size()
    return w.numel() >= LAYER_NORM_ROW and row <= LAYER_NORM_ROW_BYTES and row % 16 == 0


_own_layer_norm, _functional_layer_norm = nn.LayerNorm.forward, nn.functional.layer_norm


class ShardLayerNorm(nn.LayerNorm):
    """`nn.LayerNorm` over a last axis that the kernel is made for (_layer_norm_pays) whose forward is `tpamd_layer_norm_ranks`; the base class's own forward runs where that one does not stand in
    for it (_norm_kernel_takes; derivatives, autocast, a program's own function in the place of torch's)."""

    def forward(self, input: torch.Tensor) -> torch.Tensor:  # noqa: A002
        w = self.weight
        if w is None or LAYER_NORM_FEW_ROWS * w.numel() < input.numel() < LAYER_NORM_MANY_ROWS * w.numel() or not _layer_norm_pays(w):
            return super().forward(input)
        b = self.bias
        if (nn.LayerNorm.forward is not _own_layer_norm or nn.functional.layer_norm is not _functional_layer_norm or len(self.normalized_shape) != 1
                or not _norm_kernel_takes(input, w) or torch.is_autocast_enabled()
                or b is not None and (type(b) not in (torch.Tensor, nn.Parameter) or b.dtype != w.dtype or b.shape != w.shape or b.get_device() != w.get_device())
                or torch.is_grad_enabled() and (input.requires_grad or w.requires_grad or b is not None and b.requires_grad)):
            return super().forward(input)
        return together.layer_norm(input, w, b, self.eps)

    def __prepare_scriptable__(self):  # TorchScript compiles the module's own forward
        own = nn.LayerNorm.__new__(nn.LayerNorm)
        own.__dict__.update(self.__dict__)
        return own


def is_llama_layer(module: nn.Module) -> bool:
    """transformers' LlamaDecoderLayer as the fused forward below knows it: its forward touches its two norms, the attention and the
    MLP in this order and nothing else, and takes these arguments."""
    return type(module).__name__ == "LlamaDecoderLayer" and "forward" not in module.__dict__ and _takes_stand_in(type(module), _llama_layer_forward)


_LAYER_DEFAULTS = {"attention_mask": None, "position_ids": None, "past_key_values": None, "use_cache": False, "position_embeddings": None}


def _llama_layer_forward(self, hidden_states: torch.Tensor, *args, **kwargs) -> torch.Tensor:
    """The layer's own forward with the addition behind the attention inside the second norm's launch."""
    norm, own = self.post_attention_layernorm, self._tp_base.forward
    hooks = torch.nn.modules.module
    if (args or own is not self._tp_replaced or getattr(type(norm), "forward", None) is not _rms_norm_forward
            or norm._tp_base.forward is not norm._tp_replaced or "forward" in norm.__dict__ or _has_hooks(norm)
            or hooks._global_forward_hooks or hooks._global_forward_pre_hooks or torch.is_grad_enabled() or not _norm_kernel_takes(hidden_states, norm.weight)):
        return own(self, hidden_states, *args, **kwargs)
    attended, _ = self.self_attn(hidden_states=self.input_layernorm(hidden_states), **{**_LAYER_DEFAULTS, **kwargs})
    if type(attended) is torch.Tensor and attended.dtype == hidden_states.dtype and attended.shape == hidden_states.shape and attended.get_device() == hidden_states.get_device():
        total, normed = together.add_rms_norm(hidden_states, attended, norm.weight, norm.variance_epsilon)
    else:
        total = hidden_states + attended
        normed = norm(total)
    out = self.mlp(normed)
    return together.add(total, out) if type(out) is torch.Tensor else total + out


def is_llama_attention(module: nn.Module) -> bool:
    """transformers' LlamaAttention as the fused forward below knows it."""
    return type(module).__name__ == "LlamaAttention" and "forward" not in module.__dict__ and _takes_stand_in(type(module), _llama_attention_forward)


_ROTARY = {"apply_rotary_pos_emb": (("unsqueeze", "rotate_half"), ("q", "k", "cos", "sin", "unsqueeze_dim", "q_embed", "k_embed")),
           "rotate_half": (("shape", "torch", "cat"), ("x", "x1", "x2"))}


def _llama_attention_forward(self, hidden_states: torch.Tensor, position_embeddings=None, attention_mask=None, past_key_values=None, **kwargs):
    """The module's own forward on whole sequences without a cache or a mask, on the attention kernel (attention.py), with the rotary embedding as one launch
    (`tpamd_rope`). Everything else goes to the module's own."""
    from .attention import IMPLEMENTATION_NAME, attention_forward

    own = self._tp_base.forward
    if (own is not self._tp_replaced or past_key_values is not None or attention_mask is not None or type(position_embeddings) is not tuple or len(position_embeddings) != 2
            or self.training or torch.is_grad_enabled() or self.config._attn_implementation != IMPLEMENTATION_NAME or self.head_dim not in (64, 128)
            or kwargs.get("output_attentions") or "is_causal" in kwargs or hidden_states.dim() != 3 or hidden_states.dtype not in (torch.bfloat16, torch.float16)
            or not _native.plain_call(hidden_states, *position_embeddings) or not _native.on_hip(hidden_states)):
        return own(self, hidden_states, position_embeddings=position_embeddings, attention_mask=attention_mask, past_key_values=past_key_values, **kwargs)
    names = _globals_of(own)
    cos, sin = position_embeddings
    # the functions that the module's own forward would look up, as they were when the class was made
    if (any(names.get(name) is not function for name, function in self._tp_looked_up.items())
            or names["ALL_ATTENTION_FUNCTIONS"].get_interface(IMPLEMENTATION_NAME, None) is not attention_forward
            or cos.dtype != hidden_states.dtype or sin.dtype != cos.dtype or cos.dim() != 3 or cos.shape != sin.shape or cos.get_device() != hidden_states.get_device()
            or cos.shape[0] not in (1, hidden_states.shape[0]) or cos.shape[1:] != (hidden_states.shape[1], self.head_dim) or cos.stride(2) != 1 or sin.stride(2) != 1):
        return own(self, hidden_states, position_embeddings=position_embeddings, attention_mask=attention_mask, past_key_values=past_key_values, **kwargs)
    heads = (*hidden_states.shape[:2], -1, self.head_dim)
    q, k, v = self.q_proj(hidden_states).view(heads), self.k_proj(hidden_states).view(heads), self.v_proj(hidden_states).view(heads)
    if type(q) is torch.Tensor and type(k) is torch.Tensor and q.dtype == k.dtype == cos.dtype and not (q.data_ptr() % 16 or k.data_ptr() % 16 or cos.data_ptr() % 16 or sin.data_ptr() % 16) \
            and not any(stride % 8 for t in (q, k, cos, sin) for stride in t.stride()[:-1]) and _native.rope_takes(*q.shape[:2], q.shape[2] + k.shape[2], self.head_dim):
        q, k = _native.rope(q, k, cos, sin)
    else:
        q, k = names["apply_rotary_pos_emb"](q.transpose(1, 2), k.transpose(1, 2), cos, sin)
    out, weights = attention_forward(self, q, k, v.transpose(1, 2), None, dropout=0.0, scaling=self.scaling, **kwargs)
    return self.o_proj(out.reshape(*hidden_states.shape[:2], -1)), weights


def _globals_of(function) -> dict:
    while hasattr(function, "__wrapped__"):
        function = function.__wrapped__
    return function.__globals__


def is_falcon_mlp(module: nn.Module) -> bool:
    return type(module).__name__ == "FalconMLP" and "forward" not in module.__dict__ and _takes_stand_in(type(module), _falcon_mlp_forward)


_own_gelu, _functional_gelu = nn.GELU.forward, nn.functional.gelu


def _is_erf_gelu(act) -> bool:
    """Whether this module is the GELU of the error function, torch's or transformers', and nothing else."""
    if act is None or "forward" in act.__dict__ or nn.functional.gelu is not _functional_gelu:
        return False
    if type(act) is nn.GELU:
        return act.approximate == "none" and nn.GELU.forward is _own_gelu
    return type(act).__name__ == "GELUActivation" and act.__dict__.get("act") is _functional_gelu and \
        _native.stock_function(type(act).forward, "transformers.activations", "GELUActivation.forward", ("act",), ("self", "input"))


def _falcon_mlp_forward(self, x: torch.Tensor) -> torch.Tensor:
    """The module's own forward on a few rows with the activation in the epilogue of an int8 Linear before it, on the sum in 32 bits: a recorded step of 16 rows through a
    Falcon-40B-shaped layer 287 -> 281 us. Both ranks' first Linears with the activation take 0.67-0.94 of what they and torch's two
    passes do at 1 to 64 rows (16384 x 8192 at 64: 97.0 -> 90.6 us). Over many rows the error functions at the end of each tile take longer than torch's pass over memory (1024 rows 1490 -> 1515)."""
    from .int8 import ShardLinearW8

    own = self._tp_base.forward
    if x.dim() == 0 or x.numel() > together.W8_TOGETHER_ROWS * x.shape[-1]:
        return own(self, x)
    up, act, hooks = self._modules.get("dense_h_to_4h"), self._modules.get("act"), torch.nn.modules.module
    if (own is not self._tp_replaced or type(up) is not ShardLinearW8 or not _native.plain_call(x) or "forward" in up.__dict__ or not _is_erf_gelu(act)
            or hooks._global_forward_hooks or hooks._global_forward_pre_hooks or _has_hooks(up) or _has_hooks(act) or torch.is_grad_enabled() and x.requires_grad):
        return own(self, x)
    return self.dense_4h_to_h(up._product(x, _native.ACT_GELU))


def is_rotary_tables(module: nn.Module) -> bool:
    """The rotary embedding modules of transformers' Llama and Falcon: cos / sin of position * inv_freq, the halves repeated."""
    return type(module).__name__ in ("LlamaRotaryEmbedding", "FalconRotaryEmbedding") and _takes_stand_in(type(module), _rotary_tables_forward) and \
        isinstance(getattr(module, "inv_freq", None), torch.Tensor) and hasattr(module, "attention_scaling") and hasattr(module, "rope_type")


def _rotary_tables_forward(self, x: torch.Tensor, position_ids: torch.Tensor, **kwargs):
    f, kind, own = self.inv_freq, self.rope_type, self._tp_base.forward
    # rope types that change their frequencies with the length of the sequence keep the module's own forward; so do the further arguments
    # of its decorator
    if (kwargs or own is not self._tp_replaced or not _native.plain_call(x, position_ids, f) or position_ids.dtype != torch.int64 or position_ids.dim() != 2
            or not _native.on_hip(position_ids) or f.device != position_ids.device or f.dim() != 1
            or not isinstance(kind, str) or "dynamic" in kind or kind == "longrope"
            or x.dtype not in _KERNEL_DTYPES or f.dtype not in _KERNEL_DTYPES):
        return own(self, x, position_ids, **kwargs)
    return together.rope_tables(f, position_ids, self.attention_scaling, x.dtype)


# What each fused forward stands in for: the names its own forward looks up, and that one's arguments and locals.
_STOOD_IN_FOR = {
    _rms_norm_forward: (("dtype", "to", "torch", "float32", "pow", "mean", "rsqrt", "variance_epsilon", "weight"),
                        ("self", "hidden_states", "input_dtype", "variance")),
    _llama_layer_forward: (("input_layernorm", "self_attn", "post_attention_layernorm", "mlp"),
                           ("self", "hidden_states", *_LAYER_DEFAULTS, "kwargs", "residual", "_")),
    _llama_attention_forward: (("shape", "head_dim", "q_proj", "view", "transpose", "k_proj", "v_proj", "apply_rotary_pos_emb", "update", "layer_idx", "ALL_ATTENTION_FUNCTIONS",
                                "get_interface", "config", "_attn_implementation", "eager_attention_forward", "training", "attention_dropout", "scaling", "reshape",
                                "contiguous", "o_proj"),
                               ("self", "hidden_states", "position_embeddings", "attention_mask", "past_key_values", "kwargs", "input_shape", "hidden_shape", "query_states",
                                "key_states", "value_states", "cos", "sin", "attention_interface", "attn_output", "attn_weights")),
    _falcon_mlp_forward: (("act", "dense_h_to_4h", "dense_4h_to_h"), ("self", "x")),
    _rotary_tables_forward: (("inv_freq", "expand", "shape", "to", "torch", "float", "device", "isinstance", "type", "str", "maybe_autocast", "transpose",
                              "cat", "cos", "attention_scaling", "sin", "dtype"),
                             ("self", "x", "position_ids", "inv_freq_expanded", "position_ids_expanded", "device_type", "freqs", "emb", "cos", "sin")),
}


def _takes_stand_in(cls: type, forward) -> bool:
    return cls.__module__.split(".")[0] == "transformers" and \
        _native.stock_function(getattr(cls, "forward", None), cls.__module__, f"{cls.__qualname__}.forward", *_STOOD_IN_FOR[forward])


_fused_classes: dict = {}


def _fused_class(base: type, forward, doc: str) -> type:
    """Subclass of a module's own class with another forward (isinstance checks keep working, and so does pickling). `_tp_replaced` is the
    forward it stands in for; once the class has another (None: it had when the subclass was made), that one runs. The classes of a decoder layer, its
    attention and its MLP keep their names, which programs look such modules up by; the others are named as `ShardLinear` is."""
    cls = _fused_classes.get((base, forward))
    if cls is None:
        def reduce_ex(self, protocol):  # the class is made here and has no name to be found by: pickle what makes it
            return (_new_fused, (base, forward, doc), *super(cls, self).__reduce_ex__(protocol)[2:])

        def prepare_scriptable(self):  # TorchScript compiles the module's own forward
            own = base.__new__(base)
            own.__dict__.update(self.__dict__)
            return own

        name = base.__name__ if forward in (_llama_layer_forward, _llama_attention_forward, _falcon_mlp_forward) else "Shard" + base.__name__
        cls = type(name, (base,), {"forward": forward, "__doc__": doc, "__reduce_ex__": reduce_ex, "__prepare_scriptable__": prepare_scriptable, "_tp_base": base,
                                "_tp_replaced": staticmethod(base.forward if _takes_stand_in(base, forward) else None)})
        if forward is _llama_attention_forward:  # None in the place of one that is not transformers' own
            names = _globals_of(base.forward)
            cls._tp_looked_up = {name: names.get(name) if _native.stock_function(names.get(name), base.__module__, name, *known) else None
                                 for name, known in _ROTARY.items()}
        cls = _fused_classes.setdefault((base, forward), cls)
    return cls


def _new_fused(base: type, forward, doc: str) -> nn.Module:
    cls = _fused_class(base, forward, doc)
    return cls.__new__(cls)


def _is_silu(fn) -> bool:
    if isinstance(fn, nn.SiLU):
        return True
    name = type(fn).__name__.lower()
    return name in ("silu", "siluactivation", "swish") or fn is torch.nn.functional.silu


def _gated_mlp_forward(self, x: torch.Tensor) -> torch.Tensor:
    gate, up, down = self.gate_proj, self.up_proj, self.down_proj
    h = together.swiglu_up(x.detach(), gate.weight.detach(), up.weight.detach())
    h = _guard(h, x, gate.weight, up.weight)
    return down(h)


def _has_hooks(module: nn.Module) -> bool:
    return bool(module._forward_hooks or module._forward_pre_hooks or getattr(module, "_forward_hooks_with_kwargs", None)
                or getattr(module, "_forward_pre_hooks_with_kwargs", None))


def is_gated_silu_mlp(module: nn.Module) -> bool:
    # only the module's own children count: a wrapper forwards attribute lookups to the module it wraps
    parts = [module._modules.get(n) for n in ("gate_proj", "up_proj", "down_proj")]
    if not all(isinstance(p, nn.Linear) for p in parts):
        return False
    gate, up, _ = parts
    if gate.bias is not None or up.bias is not None or gate.weight.dtype not in (torch.bfloat16, torch.float16):
        return False
    if gate.weight.shape != up.weight.shape:
        return False
    # the fused forward reads the two weights directly: hooks on gate_proj / up_proj would be skipped, so leave such
    # blocks to their own forward (their Linears still run on the kernels)
    if _has_hooks(gate) or _has_hooks(up) or "forward" in module.__dict__:
        return False
    act = module._modules.get("act_fn", module.__dict__.get("act_fn"))
    return _is_silu(act)


def _gated_mlp_first_forward(self, x: torch.Tensor) -> torch.Tensor:
    """First call of a block that looks like a SiLU-gated MLP: its own forward and the fused one both run on this input.
    If they agree the fused forward takes over, otherwise the block keeps its own (a forward that slices its weights
    for pretraining_tp, adds projections or orders the operations differently is not this pattern)."""
    del self.forward  # the class's forward is visible again
    own = type(self).forward(self, x)
    try:
        fused = _gated_mlp_forward(self, x)
        same = isinstance(own, torch.Tensor) and own.shape == fused.shape and torch.allclose(
            own.detach().float(), fused.detach().float(), rtol=2e-2, atol=2e-2 * float(own.detach().float().std()) + 1e-6)
    except (TypeError, ValueError, RuntimeError):
        same = False
    if same:
        self.forward = types.MethodType(_gated_mlp_forward, self)
    return own


def install_shard_kernels(shard: nn.Module) -> None:
    """Route the shard's Linear layers (and gated MLP blocks) to the HIP kernels, in place."""
    for module in shard.modules():
        if type(module) is nn.Linear:
            module.__class__ = ShardLinear
        elif is_conv1d(module) and type(module).__name__ == "Conv1D" and module.weight.dim() == 2 and module.weight.dtype in _KERNEL_DTYPES:
            module.__class__ = _shard_conv1d_class(type(module))
        elif type(module) is nn.LayerNorm and module.weight is not None and module.weight.dtype in _KERNEL_DTYPES and _layer_norm_pays(module.weight):
            module.__class__ = ShardLayerNorm
        elif is_rms_norm(module) and module.weight.dtype in _KERNEL_DTYPES:
            module.__class__ = _fused_class(type(module), _rms_norm_forward, "The base class with its forward as one launch (`tpamd_rms_norm`).")
        elif is_llama_layer(module):
            module.__class__ = _fused_class(type(module), _llama_layer_forward, "The base class with an addition and a norm as one launch (`tpamd_add_rms_norm`).")
        elif is_llama_attention(module):
            module.__class__ = _fused_class(type(module), _llama_attention_forward, "The base class with the rotary embedding of a forward without a cache as one launch (`tpamd_rope`).")
        elif is_falcon_mlp(module):
            module.__class__ = _fused_class(type(module), _falcon_mlp_forward, "The base class with the activation in an int8 Linear's epilogue (`tpamd_linear_w8`).")
        elif is_rotary_tables(module):
            module.__class__ = _fused_class(type(module), _rotary_tables_forward, "The base class with its forward as one launch (`tpamd_rope_tables`).")
    for module in shard.modules():
        if is_gated_silu_mlp(module):
            module.forward = types.MethodType(_gated_mlp_first_forward, module)
