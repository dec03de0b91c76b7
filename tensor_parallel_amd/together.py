"""Ranks of one device that make equal library calls hand them in together.

The reference runs its W ranks side by side, a thread each (src/tensor_parallel/tensor_parallel.py:237-287). Here the ranks of
a device are greenlets of one thread: one runs until it has to wait. If they waited only for each other's partial sums, their kernels
would follow one another on the device, each with 1/W of the work: a decode step is then twice as many launches as it needs, every one
too small to fill the device. So a rank that reaches a call which its peers will make too gives the turn away (`GreenTurn.meet`), and whoever comes
last makes the call for all of them (`tpamd_*_ranks`). Two Llama-2-7B-shaped rank shards of two layers, recorded decode step: one row on 500
positions 321 -> 278 us, 8 on 2048 479 -> 423, 40 on 1000 (grouped queries) 534 -> 454; the Falcon-40B-shaped int8 layer, 16 on 2048, 372 -> 339.
On the host a meeting costs about 3 us for both ranks (0.5 of them for looking at the thread's state), less than the call that it saves: eager steps on a growing cache
1290 -> 1200 us on two rank shards, 2600 -> 2520 on four.

A rank meets its peers only in the state it was started in (`_thread_state`): in a stream, a grad or autocast mode, a function mode or with switches (default
dtype, attention backends, deterministic algorithms) of its own it keeps the turn, because giving it away would take its peers there. Waiting in a collective it has to
give it away: its peers then go on in the streams and modes that they were started in, and it finds its own again (`_as_started`). The switches are the whole process's
and stay as they are there, for its peers as for any thread.

What cannot be seen so is what a program holds across a library call: with a lock held there, the peer that asks for the lock would wait for a rank that cannot go on.
Models whose own forwards (not those of torch and transformers) enter a `with` block or acquire something therefore do not meet (`keeps_turn`, which looks at a model in
its first forward). What it does not find, a lock taken in one hook and given back in another, say, has to be kept to one call, or meeting switched off: TPAMD_MEET=0.
Collectives give the turn away in any case.
"""
from __future__ import annotations

import contextlib
import contextvars
import dis
import os
import threading
import types
from typing import Any, Callable, List, Optional, Sequence

import torch
from torch.utils._python_dispatch import _pop_mode, _push_mode

from . import _native

MEET = os.environ.get("TPAMD_MEET", "1") != "0"

# The turn of the running forward, per rank: context variables are per thread and per greenlet.
_turn: contextvars.ContextVar = contextvars.ContextVar("tpamd_turn", default=None)


def set_turn_lock(turn) -> None:
    _turn.set(turn)


def current_turn():
    return _turn.get()


# The calls of wrapped modules that a rank is in (collectives.SumContext; None: one whose output goes to no foldable sum), innermost last.
_contexts: contextvars.ContextVar = contextvars.ContextVar("tpamd_sum_contexts", default=None)


def push_sum_context(ctx) -> None:
    stack = _contexts.get()
    if stack is None:
        stack = []
        _contexts.set(stack)
    stack.append(ctx)


def pop_sum_context() -> None:
    _contexts.get().pop()


def current_sum_context():
    stack = _contexts.get()
    return stack[-1] if stack else None


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_current_device = getattr(torch._C, "_cuda_getDevice", None)
_grad, _inference, _autocast = torch.is_grad_enabled, torch.is_inference_mode_enabled, torch.is_autocast_enabled
_function_modes, _dispatch_modes = torch._C._len_torch_function_stack, torch._C._len_torch_dispatch_stack
_autocast_deeper, _autocast_back = torch.autocast_increment_nesting, torch.autocast_decrement_nesting
_default_dtype, _deterministic, _tf32 = torch.get_default_dtype, torch._C._get_deterministic_algorithms, torch._C._get_cublas_allow_tf32
_flash, _efficient, _math, _cudnn = (getattr(torch._C, f"_get_{name}_sdp_enabled") for name in ("flash", "mem_efficient", "math", "cudnn"))


def _thread_state(index: Optional[int]) -> tuple:
    """What of the calling thread's state a rank would find changed if a peer gave it the turn from somewhere else. `index`: of the HIP device, or None. Read
    in every library call (about a microsecond): an autocast scope shows by the depth of scopes, whatever device and dtype it is for."""
    return (_grad(), _inference(), _autocast(), _autocast_deeper() + _autocast_back(), _function_modes(), _dispatch_modes(), _default_dtype(),
            _flash(), _efficient(), _math(), _cudnn(), _deterministic(), _tf32(),
            None if index is None else (_current_device(), _raw_stream(index)))


def _of_device(get, put, device: str) -> tuple:
    return lambda: get(device), lambda value: put(device, value)


# What of that state is the calling thread's, and all that belongs to it: reading and setting. The others (default dtype, attention backends, deterministic algorithms, fp32
# products) are the process's: a difference may be another thread's doing, which may be loading a model under its default dtype, and is not to be touched.
_SETTINGS = [
    (_grad, torch._C._set_grad_enabled),
    *(_of_device(get, put, device) for device in ("cuda", "cpu") for get, put in ((_autocast, torch.set_autocast_enabled), (torch.get_autocast_dtype, torch.set_autocast_dtype))),
    (torch.is_autocast_cache_enabled, torch.set_autocast_cache_enabled),
]


def _settings() -> list:
    return [get() for get, _ in _SETTINGS]


def _set(values: list) -> None:
    for (get, put), value in zip(_SETTINGS, values):
        if get() != value:
            put(value)


@contextlib.contextmanager
def _as_started(turn: "GreenTurn"):
    """For a rank that gives the turn away in a state of its own: the streams and modes that the ranks were started in, inside, and its own again behind."""
    own, index = _settings(), turn.index
    where = None if index is None else (torch._C._cuda_getCurrentStream(index), _current_device())
    modes, dispatch = [], []
    while _function_modes() > turn.state[4]:
        modes.append(torch._C._pop_torch_function_stack())
    while _dispatch_modes() > turn.state[5]:
        dispatch.append(_pop_mode())
    inference = torch._C._InferenceMode(turn.state[1])
    inference.__enter__()
    _set(turn.settings)
    if index is not None:
        stream, device_index, device_type = turn.stream
        torch._C._cuda_setStream(stream_id=stream, device_index=device_index, device_type=device_type)
        torch.cuda.set_device(turn.state[-1][0])
    try:
        yield
    finally:
        inference.__exit__(None, None, None)
        for mode in reversed(dispatch):
            _push_mode(mode)
        for mode in reversed(modes):
            torch._C._push_on_torch_function_stack(mode)
        _set(own)
        if where is not None:
            (stream, device_index, device_type), device = where
            torch._C._cuda_setStream(stream_id=stream, device_index=device_index, device_type=device_type)
            torch.cuda.set_device(device)


_LIBRARIES = ("torch", "transformers", "tensor_parallel_amd")


def _holds(f, cls: type, seen: set) -> bool:
    """Whether a program's function, what it decorates, or a method or function that it calls by name enters a `with` block or acquires something."""
    f = getattr(f, "func", getattr(f, "__func__", f))  # functools.partial, a bound method
    code = getattr(f, "__code__", None)
    if code is None:
        return type(f).__module__.split(".")[0] not in ("builtins", *_LIBRARIES)
    if code in seen:
        return False
    seen.add(code)
    inner = [cell.cell_contents for cell in f.__closure__ or () if isinstance(cell.cell_contents, types.FunctionType)]
    if f.__globals__.get("__name__", "").split(".")[0] not in _LIBRARIES:
        codes = [code]
        for c in codes:
            codes += [k for k in c.co_consts if isinstance(k, types.CodeType)]
            if "acquire" in c.co_names or "enter_context" in c.co_names or any(op.opname in ("SETUP_WITH", "BEFORE_WITH") for op in dis.get_instructions(c)):
                return True
        called = [getattr(cls, name, None) or f.__globals__.get(name) for c in codes for name in c.co_names]
        inner += [g for g in called if isinstance(g, types.FunctionType)]
    return any(_holds(g, cls, seen) for g in inner)


def keeps_turn(module: Any) -> bool:
    """Whether a forward of this module may hold something across a library call (see above). Looked for once: kept with the module."""
    if not isinstance(module, torch.nn.Module):
        return False
    keeps = module.__dict__.get("_tp_keeps_turn")
    if keeps is None:
        forwards = {(type(m), m.__dict__.get("forward")) for m in module.modules() if m._modules}
        keeps = module.__dict__["_tp_keeps_turn"] = any(_holds(own or cls.forward, cls, set()) for cls, own in forwards)
    return keeps


class _Meeting:
    __slots__ = ("one", "many", "more", "calls", "results", "error", "parted")

    def __init__(self, one, many, more):
        self.one, self.many, self.more = one, many, more
        self.calls: List[tuple] = []
        self.results: Optional[Sequence[Any]] = None
        self.error: Optional[BaseException] = None
        self.parted = False


def _alike(a: tuple, b: tuple) -> bool:
    """Whether two ranks' tensors (or None) have the same forms."""
    for s, t in zip(a, b):
        if s is not t and (s is None or t is None or s.shape != t.shape or s.dtype is not t.dtype or s.stride() != t.stride() or s.get_device() != t.get_device()):
            return False
    return True


class GreenTurn:
    """The turn of ranks that are greenlets of one thread: whichever greenlet runs has it. `ring` holds the ranks that have not returned, `at` the
    place of the one that runs; a rank that waits switches to the next, and one that returns ends up in its parent, the greenlet that started
    them (tensor_parallel._apply_in_greenlets). `idle` counts the waits since a collective or a meeting was last complete or a rank returned: when every
    rank has waited twice, all wait for something that will not come."""

    __slots__ = ("ring", "at", "idle", "failed", "world", "index", "state", "settings", "stream", "meets", "open")

    def __init__(self, world: int = 1, index: Optional[int] = None, meets: bool = True):
        self.ring: List[Any] = []
        self.at = self.idle = 0
        self.failed = False
        self.world = world
        self.index = index
        self.state, self.settings = _thread_state(index), _settings()
        self.stream = None if index is None else torch._C._cuda_getCurrentStream(index)
        self.meets = meets and MEET and world > 1
        self.open: List[_Meeting] = []  # meetings that not every rank has come to, oldest first

    def wait(self, timeout: float = 0.0) -> bool:
        if _thread_state(self.index) == self.state:
            self._pass_on()
        else:
            with _as_started(self):
                self._pass_on()
        return True

    def _pass_on(self) -> None:
        """Gives the turn to the next rank, in the streams and modes that the ranks were started in; comes back in those."""
        ring = self.ring
        self.idle += 1
        if self.idle > 2 * len(ring):
            self.idle = 0
            if not self._part():
                self.failed = True
        at = self.at + 1
        self.at = at = at if at < len(ring) else 0
        if len(ring) > 1:
            ring[at].switch()

    def wake(self) -> None:
        self.idle = 0

    def fail(self) -> None:
        self.failed = True
        self.idle = 0

    def returned(self) -> None:
        """The rank that has the turn is through."""
        del self.ring[self.at]
        if self.at == len(self.ring):
            self.at = 0
        self.idle = 0

    def meet(self, one: Callable[..., Any], many: Callable[[List[tuple]], Sequence[Any]], tensors: tuple, more: tuple, own: tuple = ()) -> Any:
        """one(*tensors, *more, *own), made as many([...]) for all ranks that come with tensors of the same forms and the same `more`, in the order in
        which they came. A rank whose peers do not come (they wait elsewhere or have returned) makes the call alone (`_part`)."""
        for meeting in self.open:
            if meeting.one is one and meeting.many is many and meeting.more == more and _alike(meeting.calls[0][0], tensors):
                break
        else:
            meeting = _Meeting(one, many, more)
            self.open.append(meeting)
        place = len(meeting.calls)
        meeting.calls.append((tensors, own))
        if place + 1 == self.world:
            self.open.remove(meeting)
            try:
                meeting.results = many([tensors + more + own for tensors, own in meeting.calls])
            except BaseException as e:  # every rank that handed something in sees it
                meeting.error = e
            self.idle = 0
        else:
            while meeting.results is None and meeting.error is None:
                if self.failed:
                    raise threading.BrokenBarrierError
                if meeting.parted:
                    return one(*tensors, *more, *own)
                self._pass_on()
        if meeting.error is not None:
            raise meeting.error
        return meeting.results[place]

    def _part(self) -> bool:
        """Nobody gets any further: the ranks make the calls handed in so far alone. False: there were none."""
        if not self.open:
            return False
        meetings, self.open = self.open, []
        for m in meetings:
            m.parted = True
        return True


def _call(one: Callable[..., Any], many: Callable[[List[tuple]], Sequence[Any]], tensors: tuple, more: tuple = (), own: tuple = ()) -> Any:
    turn = _turn.get()
    if type(turn) is not GreenTurn or not turn.meets or turn.failed or _thread_state(turn.index) != turn.state:
        return one(*tensors, *more, *own)
    return turn.meet(one, many, tensors, more, own)


# From this many rows on a product fills the device by itself, in 256 x 256 tiles that take two ranks in two launches anyway, and each rank's
# follow-up work finds its operands still cached: prefill of 4096 rows 3312 us rank by rank, 3325 together; of 2103 rows 1758 and 1730. 1605 random shapes (512-16384 columns, K
# 1024-8192) in a HIP graph, time of one launch for both in that of two, Linears / gated pairs: 17-256 rows 0.67 / 0.71, 257-512 0.69 / 0.80, 513-1024 0.77 / 0.92, 1025-2048
# 0.86 / 0.93, 2049-3000 0.93 / 1.00, 3001-4000 0.97 / 0.99.
ALONE_ROWS = 4096


def _few_rows(x: torch.Tensor) -> bool:
    return x.dtype is not torch.float32 and x.dim() > 0 and x.numel() < ALONE_ROWS * x.shape[-1]


# The library calls that ranks make together; arguments and results are those of the functions of the same name in _native.
# fp32 products have no launch of several ranks.
def linear(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    if not _few_rows(x):
        return _native.linear(x, w, bias)
    return _call(_native.linear, _native.linear_ranks, (x, w, bias))


def _not_together(*_: Any) -> None:
    return None


def _linear_sum(calls: List[tuple]) -> Sequence[torch.Tensor]:
    ranks = [call[:3] for call in sorted(calls, key=lambda call: call[-1])]
    sums = _native.linear_sum_ranks(ranks)
    if sums is None:  # operands that the kernels do not take, or no scratch memory
        first = _native.linear(*ranks[0])
        copy = torch.empty_like(first)
        sums = [copy, _native.linear(*ranks[1], addend=first, copy=copy)]
    return sums


def linear_sum(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], rank: int, op: Any = None) -> Optional[torch.Tensor]:
    """The sum of two ranks' Linears, a tensor of its own for each; None where this rank is on its own or two launches are faster. `op`: the collective that
    it is for, which both ranks have to name."""
    K = x.shape[-1]
    if K == 0 or w.dim() != 2 or x.dtype is torch.float32 or not _native.linear_sum_pays(x.numel() // K, w.shape[0], K, x.dtype, x.get_device()):
        return None
    return _call(_not_together, _linear_sum, (x, w, bias), (op,), (rank,))


# Up to this many rows the int8 kernels take two ranks in one launch, and a sum that those cannot add up is a launch of its own behind them; above, a rank's Linear
# fills the device and, from int8.W8_ALONE_ROWS on, adds the other's result (the Falcon-40B-shaped layer: 16 rows 294 us this way and 301 the other, 1024 rows 1492 and 1462).
W8_TOGETHER_ROWS = 64


def linear_w8(x: torch.Tensor, wq: torch.Tensor, scale: torch.Tensor, outlier_idx: Optional[torch.Tensor], w_out: Optional[torch.Tensor],
              bias: Optional[torch.Tensor] = None, act: int = _native.ACT_NONE) -> torch.Tensor:
    return _call(_native.linear_w8, _native.linear_w8_ranks, (x, wq, scale, outlier_idx, w_out, bias), (act,))


def _linear_w8_sum(calls: List[tuple]) -> Sequence[torch.Tensor]:
    ranks = [call[:6] for call in sorted(calls, key=lambda call: call[-1])]
    sums = _native.linear_w8_sum_ranks(ranks)
    if sums is None:
        parts = _native.linear_w8_ranks(ranks)
        copy = torch.empty_like(parts[0])
        sums = [copy, _native.reduce_partials(parts, copy=copy)]
    return sums


def linear_w8_sum(x: torch.Tensor, wq: torch.Tensor, scale: torch.Tensor, outlier_idx: Optional[torch.Tensor], w_out: Optional[torch.Tensor],
                  bias: Optional[torch.Tensor], rank: int, op: Any = None) -> Optional[torch.Tensor]:
    return _call(_not_together, _linear_w8_sum, (x, wq, scale, outlier_idx, w_out, bias), (op,), (rank,))


def _gather(calls: List[tuple]) -> Sequence[torch.Tensor]:
    return _native.linear_gather_ranks([call[:3] for call in sorted(calls, key=lambda call: call[-1])])  # (every rank's result is the same)


def linear_gathered(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], rank: int, world: int, op: Any = None) -> Optional[torch.Tensor]:
    """The Linears of two ranks with their results side by side, a whole one for each, in one launch; None where this rank is on its own. `op` as above."""
    if world != 2 or x.numel() == 0:
        return None
    return _call(_not_together, _gather, (x, w, bias), (op,), (rank,))


def swiglu_up(x: torch.Tensor, wg: torch.Tensor, wu: torch.Tensor) -> torch.Tensor:
    if not _few_rows(x):
        return _native.swiglu_up(x, wg, wu)
    return _call(_native.swiglu_up, _native.swiglu_up_ranks, (x, wg, wu))


def rms_norm(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    if x.numel() >= ALONE_ROWS * w.numel():
        return _native.rms_norm(x, w, eps)
    return _call(_native.rms_norm, _native.rms_norm_ranks, (x, w), (eps,))


def add_rms_norm(r: torch.Tensor, x: torch.Tensor, w: torch.Tensor, eps: float) -> tuple:
    if x.numel() >= ALONE_ROWS * w.numel():
        return _native.add_rms_norm(r, x, w, eps)
    return _call(_native.add_rms_norm, _native.add_rms_norm_ranks, (r, x, w), (eps,))


LAYER_NORM_TOGETHER_ROWS = 64  # more rows of two ranks take as long in one launch as in two


def layer_norm(x: torch.Tensor, w: torch.Tensor, b: Optional[torch.Tensor], eps: float) -> torch.Tensor:
    if x.numel() > LAYER_NORM_TOGETHER_ROWS * w.numel():
        return _native.layer_norm(x, w, b, eps)
    return _call(_native.layer_norm, _native.layer_norm_ranks, (x, w, b), (eps,))


def attention_decode_rope(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, k_cache: torch.Tensor,
                          v_cache: torch.Tensor, pos0, scale: Optional[float] = None) -> torch.Tensor:
    if isinstance(pos0, torch.Tensor):
        return _call(_native.attention_decode_rope, _native.attention_decode_rope_ranks, (q, k, v, cos, sin, k_cache, v_cache, pos0), (scale,))
    return _call(_native.attention_decode_rope, _native.attention_decode_rope_ranks, (q, k, v, cos, sin, k_cache, v_cache), (pos0, scale))


def rope_tables(inv_freq: torch.Tensor, position_ids: torch.Tensor, scaling: float, dtype: torch.dtype) -> tuple:
    return _call(_native.rope_tables, _native.rope_tables_ranks, (inv_freq, position_ids), (scaling, dtype))


def causal_mask(q_offset: torch.Tensor, kv_offset: int, q_length: int, kv_length: int) -> torch.Tensor:
    return _call(_native.causal_mask, _native.causal_mask_ranks, (q_offset,), (kv_offset, q_length, kv_length))


# An addition of more rows takes as long in one launch as in two, and where the host sets the pace torch's own calls are the cheaper ones.
ADD_TOGETHER_ROWS = 64


def add(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """a + b; in one launch for ranks that come with a few rows of the same forms."""
    if (a.numel() > ADD_TOGETHER_ROWS * a.shape[-1] or a.dtype is not b.dtype or a.shape != b.shape or a.get_device() != b.get_device()
            or not (a.is_contiguous() and b.is_contiguous()) or not _native.plain_call(a, b)):
        return a + b
    return _call(torch.add, _native.add_ranks, (a, b))


def advance(count: torch.Tensor, by: int) -> torch.Tensor:
    """count.add_(by)."""
    if count.dtype is not torch.int64 or count.numel() != 1 or not count.is_cuda or not _native.plain_call(count):
        return count.add_(by)
    return _call(torch.Tensor.add_, _native.advance_ranks, (count,), (by,))
