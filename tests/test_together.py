"""Ranks that hand equal calls in together (together.py), on the CPU with the library calls stubbed: which ranks meet, what each gets back, and
that nobody waits for a peer that does not come."""
import contextlib
import threading

import pytest
import torch

from tensor_parallel_amd import _native, together
from tensor_parallel_amd.tensor_parallel import RANK_GREENLETS, _apply_in_greenlets

pytestmark = pytest.mark.skipif(not RANK_GREENLETS, reason="the greenlet package is not there: the ranks of a device are threads")
CPU = torch.device("cpu")


@pytest.fixture
def calls(monkeypatch):
    made = []

    def one(x, w, bias=None):
        made.append(1)
        return torch.nn.functional.linear(x, w, bias)

    def many(items):
        made.append(len(items))
        return [torch.nn.functional.linear(*item) for item in items]

    monkeypatch.setattr(_native, "linear", one)
    monkeypatch.setattr(_native, "linear_ranks", many)
    return made


def run(*bodies):
    return _apply_in_greenlets(list(bodies), [(r,) for r in range(len(bodies))], [{}] * len(bodies), CPU)


@contextlib.contextmanager
def _device_autocast():  # what torch.autocast("cuda") sets, also where there is no device
    torch.set_autocast_enabled("cuda", True)
    try:
        yield
    finally:
        torch.set_autocast_enabled("cuda", False)


def operands(r, rows=3, cols=4, K=8):
    g = torch.Generator().manual_seed(r)
    return torch.randn(rows, K, generator=g).bfloat16(), torch.randn(cols, K, generator=g).bfloat16()


@pytest.mark.parametrize("world", [1, 2, 3])
def test_equal_calls_are_made_at_once_and_each_rank_gets_its_own(calls, world):
    def body(r):
        return [together.linear(*operands(r)) for _ in range(3)]

    for r, got in enumerate(run(*[body] * world)):
        assert all(torch.equal(y, torch.nn.functional.linear(*operands(r))) for y in got)
    assert calls == [world] * 3


@pytest.mark.parametrize("form", ["cols", "rows", "strides", "dtype", "bias", "fp32", "many rows"])
def test_calls_of_other_forms_are_made_alone(calls, form):
    def body(r):
        x, w = operands(r)
        b = None
        if r == 1 or form in ("fp32", "many rows"):
            if form == "cols":
                w = torch.cat([w, w])
            elif form == "rows":
                x = x[:2]
            elif form == "strides":
                x = torch.cat([x, x], 1)[:, :8]
            elif form == "dtype":
                x, w = x.half(), w.half()
            elif form == "bias":
                b = w[:, 0].contiguous()
            elif form == "fp32":
                x, w = x.float(), w.float()
            else:
                x = x[:1].expand(together.ALONE_ROWS, -1)
        return together.linear(x, w, b), torch.nn.functional.linear(x, w, b)

    for got, want in run(body, body):
        assert torch.equal(got, want)
    assert calls == [1, 1]


@pytest.mark.parametrize("mode", ["grad", "inference", "autocast", "function mode"])
def test_a_rank_in_a_state_of_its_own_keeps_the_turn(calls, mode):
    def own():
        if mode == "grad":
            return torch.no_grad()
        if mode == "inference":
            return torch.inference_mode()
        if mode == "autocast":
            return _device_autocast()
        return torch.device("cpu")

    seen = []

    def body(r):
        with own():
            y = together.linear(*operands(r))
            seen.append(r)
        assert torch.is_grad_enabled() and not torch.is_inference_mode_enabled()
        return y + together.linear(*operands(r))

    run(body, body)
    assert calls == [1, 1, 2] and seen == [0, 1]


def test_a_peer_that_returned_or_waits_elsewhere_is_not_waited_for(calls):
    from tensor_parallel_amd.collectives import CollectiveOperation

    op = CollectiveOperation(2, lambda *xs: [sum(xs)] * 2, timeout=5.0)

    def body(r):
        got = []
        if r == 0:
            got.append(together.linear(*operands(0)))  # the peer is in the collective
        total = op(r + 1, r)
        if r == 0:
            got.append(together.linear(*operands(0)))  # the peer has returned
        return total, got

    (t0, got), (t1, _) = run(body, body)
    assert t0 == t1 == 3 and calls == [1, 1]
    assert all(torch.equal(y, torch.nn.functional.linear(*operands(0))) for y in got)


@pytest.mark.parametrize("where", ["before", "in the call"])
def test_a_failure_reaches_every_rank_and_the_next_forward_works(calls, monkeypatch, where):
    good = _native.linear_ranks

    def bad(items):
        raise KeyError("bad operands")

    def body(r):
        if where == "before" and r == 1:
            raise KeyError("bad operands")
        return together.linear(*operands(r))

    if where == "in the call":
        monkeypatch.setattr(_native, "linear_ranks", bad)
    with pytest.raises(KeyError, match="bad operands"):
        run(body, body)
    monkeypatch.setattr(_native, "linear_ranks", good)
    run(lambda r: together.linear(*operands(r)), lambda r: together.linear(*operands(r)))
    assert calls[-1] == 2


def test_gathered_columns_are_in_rank_order_whoever_came_first(monkeypatch):
    monkeypatch.setattr(_native, "linear_gather_ranks", lambda items: [torch.cat([torch.nn.functional.linear(*item) for item in items], -1)] * len(items))
    want = torch.cat([torch.nn.functional.linear(*operands(r)) for r in range(2)], -1)

    def body(r):
        return [together.linear_gathered(*operands(r), None, r, 2) for _ in range(3)]

    for got in run(body, body):  # whoever came last goes on first
        assert all(torch.equal(y, want) for y in got)
    assert run(lambda r: together.linear_gathered(*operands(r), None, r, 2), lambda r: r) == [None, 1]  # the peer does not come: nothing is gathered


@contextlib.contextmanager
def _default_dtype(dtype):
    before = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        yield
    finally:
        torch.set_default_dtype(before)


@contextlib.contextmanager
def _deterministic():
    torch.use_deterministic_algorithms(True)
    try:
        yield
    finally:
        torch.use_deterministic_algorithms(False)


def _scopes():
    from torch.nn.attention import SDPBackend, sdpa_kernel

    return {"default dtype": lambda: _default_dtype(torch.bfloat16), "attention backend": lambda: sdpa_kernel(SDPBackend.MATH), "deterministic": _deterministic,
            "autocast on the host": lambda: torch.autocast("cpu", dtype=torch.bfloat16), "autocast dtype": lambda: torch.autocast("cpu", dtype=torch.float16, enabled=False),
            "no grad": torch.no_grad, "inference": torch.inference_mode, "default device": lambda: torch.device("cpu")}


PROCESS_WIDE = ("default dtype", "attention backend", "deterministic")


def _state():
    backends = torch.backends.cuda
    return (torch.is_grad_enabled(), torch.is_inference_mode_enabled(), torch.is_autocast_enabled("cuda"), torch.get_autocast_dtype("cuda"),
            torch.is_autocast_enabled("cpu"), torch.get_autocast_dtype("cpu"), torch.get_default_dtype(), torch.are_deterministic_algorithms_enabled(),
            backends.flash_sdp_enabled(), backends.mem_efficient_sdp_enabled(), backends.math_sdp_enabled(), torch._C._len_torch_function_stack())


@pytest.mark.parametrize("ranks", [(0,), (0, 1)])
@pytest.mark.parametrize("scope", list(_scopes()))
def test_a_scope_of_one_rank_is_not_seen_by_another(calls, scope, ranks):
    """Two library calls and a collective inside the scope, one of each behind it; no collective where the scope is the process's."""
    from tensor_parallel_amd.collectives import CollectiveOperation

    op, before = CollectiveOperation(2, lambda *xs: [sum(xs)] * 2, timeout=5.0), _state()
    with _scopes()[scope]():
        within = _state()
    assert within != before and _state() == before

    def body(r):
        outside = []
        for _ in range(2):
            with _scopes()[scope]() if r in ranks else contextlib.nullcontext():
                expected = within if r in ranks else before
                states = [_state()]
                for _ in range(2):
                    together.linear(*operands(r))
                    states.append(_state())
                assert scope in PROCESS_WIDE or op(r + 1, r) == 3
                states.append(_state())
                together.linear(*operands(r))
                states.append(_state())
                assert states == [expected] * len(states)
            outside.append(_state())
            together.linear(*operands(r))
            op(r, r)
            outside.append(_state())
        assert outside == [before] * len(outside)

    run(body, body)
    assert _state() == before


def test_calls_that_nobody_comes_to_are_made_in_the_state_of_their_rank(monkeypatch):
    """The peer waits in a collective, inside a scope of its own, when it turns out that it does not come."""
    from tensor_parallel_amd.collectives import CollectiveOperation

    op, states = CollectiveOperation(2, lambda *xs: [sum(xs)] * 2, timeout=5.0), []
    monkeypatch.setattr(_native, "linear", lambda x, w, b=None: states.append(_state()) or torch.nn.functional.linear(x, w, b))
    before = _state()

    def body(r):
        if r == 0:
            together.linear(*operands(0))
            op(1, 0)
        else:
            with torch.inference_mode(), torch.autocast("cpu", dtype=torch.bfloat16):
                op(2, 1)

    run(body, body)
    assert states == [before]


LOCK = threading.Lock()


class _Locked(torch.nn.Module):
    def __init__(self, how):
        super().__init__()
        self.how, self.inner = how, torch.nn.Module()
        self.inner.forward = lambda x, w: together.linear(x, w)

    def forward(self, x, w):
        if self.how == "with":
            with LOCK:
                return self.inner(x, w)
        return self._acquired(x, w) if self.how == "in a method" else self._plain(x, w)

    def _acquired(self, x, w):
        LOCK.acquire()
        try:
            return self.inner(x, w)
        finally:
            LOCK.release()

    def _plain(self, x, w):
        return self.inner(x, w)


class _Unlocked(torch.nn.Module):
    def __init__(self):
        super().__init__()
        self.inner = torch.nn.Linear(1, 1)

    def forward(self, x, w):
        return together.linear(x, w)


@pytest.mark.parametrize("how", ["with", "in a method", "not at all"])
def test_a_rank_whose_model_may_hold_a_lock_keeps_the_turn(calls, how):
    models = [_Locked(how) for _ in range(2)] if how != "not at all" else [_Unlocked() for _ in range(2)]
    for r, y in enumerate(_apply_in_greenlets(models, [operands(r) for r in range(2)], [{}] * 2, CPU)):
        assert torch.equal(y, torch.nn.functional.linear(*operands(r)))
    assert calls == ([2] if how == "not at all" else [1, 1])


def test_meeting_can_be_switched_off(calls, monkeypatch):
    monkeypatch.setattr(together, "MEET", False)
    run(lambda r: together.linear(*operands(r)), lambda r: together.linear(*operands(r)))
    assert calls == [1, 1]


def test_models_of_the_libraries_meet():
    transformers = pytest.importorskip("transformers")
    from tensor_parallel_amd.shard_modules import install_shard_kernels

    llama = transformers.LlamaForCausalLM(transformers.LlamaConfig(vocab_size=32, hidden_size=32, intermediate_size=48, num_hidden_layers=1, num_attention_heads=2))
    falcon = transformers.FalconModel(transformers.FalconConfig(vocab_size=32, hidden_size=32, num_hidden_layers=1, num_attention_heads=2))
    opt = transformers.OPTForCausalLM(transformers.OPTConfig(vocab_size=32, hidden_size=32, num_hidden_layers=1, num_attention_heads=2, ffn_dim=64, word_embed_proj_dim=32))
    for model in (llama, falcon, opt):
        install_shard_kernels(model)
        assert not together.keeps_turn(model)


def test_counts_in_host_memory_are_advanced_there(monkeypatch):
    """A static cache's count that a program keeps on the host (a prompt of several positions reads it there) has no address for a kernel."""
    monkeypatch.setattr(_native, "advance_ranks", lambda calls: pytest.fail("a kernel was given an address in host memory"))
    counts = [torch.tensor(10 + r) for r in range(2)]
    assert run(*[lambda r: together.advance(counts[r], 3)] * 2) == counts and [int(c) for c in counts] == [13, 14]


@pytest.mark.parametrize("call", ["advance_ranks", "add_ranks"])
def test_small_calls_of_several_ranks_want_device_memory(call):
    items = [(torch.tensor(1), 1)] * 2 if call == "advance_ranks" else [(torch.ones(8), torch.ones(8))] * 2
    with pytest.raises(_native.NativeLibraryError, match="HIP device"):
        getattr(_native, call)(items)


@pytest.mark.parametrize("kinds", [("sum", "sum"), ("gather", "gather"), ("sum", "gather"), ("gather", "sum")])
def test_ranks_at_different_collectives_are_not_taken_for_one_call(monkeypatch, kinds):
    """Linears of equal forms, one rank's for one collective and the other's for another."""
    for name in ("linear_sum_ranks", "linear_gather_ranks"):
        monkeypatch.setattr(_native, name, lambda items: pytest.fail("two collectives were taken for one"))
    monkeypatch.setattr(_native, "linear_sum_pays", lambda *_: True)
    ops = [object(), object()]

    def body(r):
        if kinds[r] == "sum":
            return together.linear_sum(*operands(r), None, r, ops[r])
        return together.linear_gathered(*operands(r), None, r, 2, ops[r])

    assert run(body, body) == [None, None]
    if kinds[0] != kinds[1]:  # two kinds for one op, which no rule makes
        ops[1] = ops[0]
        assert run(body, body) == [None, None]


def test_a_process_wide_switch_of_another_thread_is_left_alone():
    """A program may load a model under a default dtype in one thread while another runs a forward, whose ranks wait in collectives."""
    from tensor_parallel_amd.collectives import CollectiveOperation

    op, seen = CollectiveOperation(2, lambda *xs: [sum(xs)] * 2, timeout=5.0), []
    switched, done = threading.Event(), threading.Event()

    def loads():
        with _default_dtype(torch.float64):
            switched.set()
            done.wait(10)
            seen.append(torch.get_default_dtype())

    other = threading.Thread(target=loads)

    def body(r):
        if r == 0:
            other.start()
            switched.wait(10)
        for _ in range(3):
            with torch.inference_mode() if r == 0 else contextlib.nullcontext():  # a state of this rank's own as well
                op(r, r)
                seen.append(torch.get_default_dtype())
                assert torch.is_inference_mode_enabled() == (r == 0)

    try:
        run(body, body)
    finally:
        done.set()
        other.join()
    assert seen == [torch.float64] * 7 and torch.get_default_dtype() is torch.float32
