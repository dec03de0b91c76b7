"""A rank's input and output rules around one module (reference: src/tensor_parallel/wrapper.py:17-75).

A rule maps a target to an action. Input targets are positions (int) or keyword names (str) of the wrapped module's
call; output targets are positions of a tuple / list output, keys of a mapping output, and 0 for a bare tensor.
An action is a callable `(value, rank=...)` (a collective op, a `StateAction`, user code), a `(split, undo)` pair of
which the first half is used, or one of the strings `"split <dim>"` and `"scale"`. The strings run on the device:
`"split d"` is one launch of the region mover, `"scale"` one launch of the scale kernel.
"""
from __future__ import annotations

from collections.abc import Mapping, Sequence
from typing import Any, Callable

import torch
from torch import nn

from . import _native
from .collectives import DeviceAllGather, DeviceAllReduce, SumContext, pop_sum_context, push_sum_context
from .config import MappedActions
from .shard_modules import gathered_linear
from .slicing import SliceSpec, apply_spec, normalize_dim, tensor_split_range


def _split_along(value: torch.Tensor, dim: int, rank: int, world_size: int) -> torch.Tensor:
    """`torch.tensor_split(value, world_size, dim)[rank]` as a fresh contiguous tensor."""
    axis = normalize_dim(dim, value.dim())
    piece = tensor_split_range(value.shape[axis], world_size, rank)
    return apply_spec(value, SliceSpec(tuple(value.shape), axis, (piece,)))


def _bind(action, rank: int, world_size: int) -> Callable[[Any], Any]:
    """The action as a function of the value alone."""
    if isinstance(action, tuple):  # (split, undo): only the splitting half acts on activations
        action = action[0]
    if callable(action):
        return lambda value: action(value, rank=rank)
    words = action.split()
    if words and words[0] == "split":
        return lambda value: _split_along(value, int(words[1]), rank, world_size)
    if words and words[0] == "scale":
        return lambda value: _native.scale(value, world_size)
    raise Exception(f"unexpected action {words[0] if words else action!r}; supported actions: split, scale, or custom user-defined")


def apply_action(input, action, *, rank: int, world_size: int):
    """One rule applied to one argument or output (wrapper.py:17-28)."""
    return _bind(action, rank, world_size)(input)


def process_input(input_actions: MappedActions, rank: int, world_size: int, *args, **kwargs):
    """Applies the input rules to a call's arguments and returns (args, kwargs). A keyword the caller left out reaches
    its action as None and is passed on with the action's result, as in the reference (wrapper.py:31-37); a rule for
    a position the caller did not fill is skipped."""
    positional = list(args)
    named = dict(kwargs)
    for target, action in input_actions.items():
        act = _bind(action, rank, world_size)
        if isinstance(target, int):
            if 0 <= target < len(positional):
                positional[target] = act(positional[target])
        else:
            named[target] = act(named.get(target))
    return positional, named


def process_output(output, output_actions: MappedActions, *, rank: int, world_size: int):
    """Applies the output rules to what the wrapped module returned and keeps its container type
    (wrapper.py:40-48)."""
    if not output_actions:
        return output
    rules = [(target, _bind(action, rank, world_size)) for target, action in output_actions.items()]
    if isinstance(output, torch.Tensor):
        for target, act in rules:
            if target == 0:
                output = act(output)
        return output
    if isinstance(output, Mapping):  # dicts and transformers' ModelOutput: changed in place, like the reference
        for target, act in rules:
            output[target] = act(output.get(target))
        return output
    if isinstance(output, Sequence):
        items = list(output)
        for target, act in rules:
            if isinstance(target, int) and -len(items) <= target < len(items):
                items[target] = act(items[target])
        return type(output)(items)
    raise TypeError(f"cannot apply output rules to a {type(output).__name__}")


def _output_zero(output):
    """What an output rule for target 0 acts on (see process_output)."""
    if isinstance(output, torch.Tensor):
        return output
    if isinstance(output, Mapping):
        return output.get(0)
    if isinstance(output, Sequence) and len(output) > 0:
        return output[0]
    return None


class TensorParallelWrapper(nn.Module):
    """Holds one module as `tp_wrapped_module`; calls go through the rank's rules, every other attribute is the
    wrapped module's."""

    _gather_op = None  # of a wrapper that was saved before there was one

    def __init__(self, module: nn.Module, input_actions: MappedActions, output_actions: MappedActions, *, rank: int, world_size: int):
        super().__init__()
        self.tp_wrapped_module = module
        self.input_actions = input_actions
        self.output_actions = output_actions
        self.rank = rank
        self.world_size = world_size
        # output 0 summed over the ranks on one device: the module's last Linear may take the sum into its epilogue
        action = output_actions.get(0) if output_actions else None
        self._sum_op = action if isinstance(action, DeviceAllReduce) else None
        # ... and a Linear whose output is nothing but gathered may write every rank's whole output itself
        self._gather_op = action if type(action) is DeviceAllGather and len(output_actions) == 1 else None

    def forward(self, *args, **kwargs):
        call_args, call_kwargs = args, kwargs
        if self.input_actions:
            call_args, call_kwargs = process_input(self.input_actions, self.rank, self.world_size, *args, **kwargs)
        wrapped = self._modules["tp_wrapped_module"]
        if self._gather_op is not None:
            whole = gathered_linear(wrapped, self._gather_op, self.rank, call_args, call_kwargs)
            if whole is not None:
                return whole
        # Every wrapper publishes its own context, or none: Linears and rules inside a wrapper without a foldable sum must
        # not be taken for those of an enclosing module whose output is summed.
        foldable = self._sum_op is not None and self._sum_op.fusable
        ctx = SumContext(self._sum_op, self.rank, self, wrapped) if foldable else None
        push_sum_context(ctx)
        try:
            result = wrapped(*call_args, **call_kwargs)
            if ctx is not None:
                ctx.settle(_output_zero(result))
            return process_output(result, self.output_actions, rank=self.rank, world_size=self.world_size)
        finally:
            pop_sum_context()

    def __getattr__(self, name: str):
        try:
            return super().__getattr__(name)  # parameters, buffers and submodules of the wrapper itself
        except AttributeError:
            inner = self.__dict__.get("_modules", {}).get("tp_wrapped_module")
            if inner is None:
                raise
            return getattr(inner, name)
