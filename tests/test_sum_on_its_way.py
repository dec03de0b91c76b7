"""Row-parallel Linears that feed a "sum" rule, two ranks of one device on the CPU with the library calls stubbed: whatever a program does to such a Linear's output
on its way to the rule, what the rule delivers is the sum of what every rank's module returned, or an error."""
import types

import pytest
import torch
from torch import nn

from tensor_parallel_amd import _native, together
from tensor_parallel_amd.collectives import DeviceAllReduce
from tensor_parallel_amd.int8 import W8_ALONE_ROWS, ShardLinearW8
from tensor_parallel_amd.shard_modules import ShardLinear, returned
from tensor_parallel_amd.tensor_parallel import RANK_GREENLETS, _apply_in_greenlets
from tensor_parallel_amd.wrapper import TensorParallelWrapper

pytestmark = pytest.mark.skipif(not RANK_GREENLETS, reason="the greenlet package is not there: the ranks of a device are threads")
K, N = 16, 8


@pytest.fixture(autouse=True)
def folds(monkeypatch):
    """The library calls on the CPU; how often a sum was made by a Linear."""
    made = []

    def put(y, addend, copy, how="addend"):
        if addend is None:
            return y
        made.append(how)
        y = y + addend
        if copy is not None:
            copy.copy_(y)
        return y

    def linear(x, w, b=None, act=0, addend=None, out=None, copy=None):
        return put(nn.functional.linear(x, w, b), addend, copy)

    def linear_w8(x, wq, scale, idx, w_out, b=None, act=0, addend=None, copy=None):
        return put(nn.functional.linear(x, (wq * scale[:, None]).to(x.dtype), b), addend, copy)

    def sums(one):
        def both(calls):
            made.append("whole")
            total = one(*calls[0]) + one(*calls[1])
            return [total, total.clone()]
        return both

    def reduce_partials(parts, accum=0, out=None, copy=None):
        return put(parts[0], parts[1], copy, "reduction")

    for name, call in {"linear": linear, "linear_w8": linear_w8, "linear_ranks": lambda calls: [linear(*c) for c in calls],
                       "linear_w8_ranks": lambda calls: [linear_w8(*c) for c in calls], "linear_sum_ranks": sums(linear), "linear_w8_sum_ranks": sums(linear_w8),
                       "linear_sum_pays": lambda *_: True, "reduce_partials": reduce_partials}.items():
        monkeypatch.setattr(_native, name, call)
    return made


class Around(nn.Module):
    """A program's module around the Linear, which may scale or add to its output in place."""

    def __init__(self, linear):
        super().__init__()
        self.linear, self.scales, self.adds = linear, False, False

    def forward(self, x):
        out = self.linear(x)
        if self.scales:
            out.mul_(2)
        if self.adds:
            out.add_(1)
        return out


def shards(kind, around):
    op, made = DeviceAllReduce(2), []
    for r in range(2):
        g = torch.Generator().manual_seed(r)
        w = torch.randint(-2, 3, (N, K), generator=g).bfloat16()  # products and sums that every step holds exactly
        if kind == "int8":
            linear = ShardLinearW8(w.to(torch.int8), torch.ones(N), torch.zeros(0, dtype=torch.int32), torch.zeros(N, 0, dtype=torch.bfloat16), None, torch.bfloat16)
        else:
            linear = ShardLinear(K, N, bias=False).bfloat16()
            linear.weight.data.copy_(w)
        made.append(TensorParallelWrapper(Around(linear) if around else linear, {}, {0: op}, rank=r, world_size=2))
    return made


def linears(models):
    return [m.tp_wrapped_module.linear if isinstance(m.tp_wrapped_module, Around) else m.tp_wrapped_module for m in models]


def forward(models, rows, inference=False):
    xs = [torch.randint(-2, 3, (rows, K), generator=torch.Generator().manual_seed(7 + r)).bfloat16() for r in range(2)]
    with torch.inference_mode() if inference else torch.no_grad():
        parts = [(m.wq.float() if hasattr(m, "wq") else m.weight.float()) for m in linears(models)]
        want = sum(x.float() @ w.t() for x, w in zip(xs, parts))
        return _apply_in_greenlets(models, [(x,) for x in xs], [{}] * 2, torch.device("cpu")), want


def made(kind, rows):
    """How the sum is made where the Linear may make it."""
    return "whole" if kind == "16 bits" or rows <= together.W8_TOGETHER_ROWS else "reduction" if rows <= W8_ALONE_ROWS else "addend"


def check(got, want):
    for y in got:
        assert torch.equal(y.float(), want)


@pytest.mark.parametrize("inference", [False, True])
@pytest.mark.parametrize("around", [False, True])
@pytest.mark.parametrize("rows", [4, 200, 600])
@pytest.mark.parametrize("kind", ["16 bits", "int8"])
def test_the_linear_makes_the_sum_where_nobody_sees_its_output(folds, kind, rows, around, inference):
    models = shards(kind, around)
    for _ in range(3):
        check(*forward(models, rows, inference))
    # a module that is not known here may have done something to the output that does not show: not in inference mode, and not for int8 weights at all
    assert folds[-1] == ("reduction" if around and (inference or kind == "int8") else made(kind, rows))


@pytest.mark.parametrize("which", [(0,), (1,), (0, 1)])
@pytest.mark.parametrize("hook", ["scales", "new tensor", "on the module around", "in front of all", "a forward put around"])
@pytest.mark.parametrize("rows", [4, 200, 600])
@pytest.mark.parametrize("kind", ["16 bits", "int8"])
def test_a_hook_sees_and_changes_its_own_ranks_part(kind, rows, hook, which):
    models = shards(kind, True)
    for _ in range(3):
        check(*forward(models, rows))
    seen = {}

    def change(r):
        def hooked(module, args, out):
            seen[r] = out.clone()
            out.mul_(2)
            return out.clone() if hook == "new tensor" else None
        return hooked

    handles = []
    for r in which:
        linear = linears(models)[r]
        if hook == "on the module around":
            handles.append(models[r].tp_wrapped_module.register_forward_hook(change(r)))
        elif hook == "in front of all":
            if r == which[0]:
                both = {id(m): i for i, m in enumerate(linears(models)) if i in which}
                handles.append(torch.nn.modules.module.register_module_forward_hook(lambda m, a, out: change(both[id(m)])(m, a, out) if id(m) in both else None))
        elif hook == "a forward put around":
            own = linear.forward
            linear.forward = lambda x, own=own, r=r, linear=linear: (lambda out: [change(r)(linear, x, out), out][1])(own(x))
        else:
            handles.append(linear.register_forward_hook(change(r)))
    try:
        for _ in range(3):
            seen.clear()
            got, _ = forward(models, rows)
            xs = [torch.randint(-2, 3, (rows, K), generator=torch.Generator().manual_seed(7 + r)).float() for r in range(2)]
            own = [x @ (m.wq.float() if hasattr(m, "wq") else m.weight.float()).t() for x, m in zip(xs, linears(models))]
            check(got, sum((2 if r in which else 1) * p for r, p in enumerate(own)))
            assert sorted(seen) == list(which) and all(torch.equal(seen[r].float(), own[r]) for r in which)
    finally:
        for h in handles:
            h.remove()


@pytest.mark.parametrize("inference", [False, True])
@pytest.mark.parametrize("change", ["scales", "adds"])
@pytest.mark.parametrize("rows", [4, 200, 600])
@pytest.mark.parametrize("kind", ["16 bits", "int8"])
def test_a_module_that_starts_to_change_the_output_in_place(kind, rows, change, inference):
    models = shards(kind, True)
    for _ in range(3):
        check(*forward(models, rows))
    for m in models:
        setattr(m.tp_wrapped_module, change, True)
    failures = 0
    for _ in range(4):
        try:
            got, want = forward(models, rows, inference)
            check(got, 2 * want if change == "scales" else want + 2)
        except RuntimeError as e:
            assert "in place" in str(e)
            failures += 1
    # a Linear that has folded the other rank's part in cannot give it back: an error, and no folding from then on
    assert failures <= 2 if kind == "16 bits" and not inference else failures == 0


@pytest.mark.parametrize("change", ["scales", "adds"])
@pytest.mark.parametrize("kind", ["16 bits", "int8"])
def test_a_module_that_always_changes_the_output_in_place(kind, change):
    models = shards(kind, True)
    for m in models:
        setattr(m.tp_wrapped_module, change, True)
    for inference in (True, True, True, False, False, True, False):
        got, want = forward(models, 4, inference)
        check(got, 2 * want if change == "scales" else want + 2)


def own_forward(self, x):
    """As the fused attention forwards, which return what their last Linear gives."""
    return returned(self, own_forward, self.linear, x)


@pytest.mark.parametrize("inference", [False, True])
@pytest.mark.parametrize("rows", [4, 200, 600])
@pytest.mark.parametrize("kind", ["16 bits", "int8"])
def test_the_linear_of_a_forward_that_returns_its_output_makes_the_sum(folds, kind, rows, inference):
    models = shards(kind, True)
    for m in models:
        m.tp_wrapped_module.forward = types.MethodType(own_forward, m.tp_wrapped_module)
    for _ in range(3):
        check(*forward(models, rows, inference))
    assert folds[-1] == made(kind, rows)
    # a program puts a forward of its own around that one
    for m in models:
        inner = m.tp_wrapped_module.forward
        m.tp_wrapped_module.forward = lambda x, inner=inner: inner(x).mul_(2)
    failures = 0
    for _ in range(4):
        try:
            got, want = forward(models, rows, inference)
            check(got, 2 * want)
        except RuntimeError as e:
            assert "in place" in str(e)
            failures += 1
    assert failures <= 2 if kind == "16 bits" and not inference else failures == 0
