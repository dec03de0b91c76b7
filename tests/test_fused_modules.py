"""When the one-launch forwards of a shard's norms, rotary tables and decoder layers leave the work to the module's own forward. Host tensors stand
for device ones and torch formulas for the kernels, which note that they were asked."""
import pytest
import torch
import transformers as tf
from torch.autograd import forward_ad

from tensor_parallel_amd import _native, shard_modules


@pytest.fixture
def kernels(monkeypatch):
    asked = []

    def rms_norm(x, w, eps):
        asked.append("rms_norm")
        return w * (x.float() * torch.rsqrt(x.float().square().mean(-1, keepdim=True) + eps)).to(x.dtype)

    def add_rms_norm(r, x, w, eps):
        asked.append("add_rms_norm")
        total = (r + x).detach()
        return total, w * (total.float() * torch.rsqrt(total.float().square().mean(-1, keepdim=True) + eps)).to(x.dtype)

    def rope_tables(inv_freq, position_ids, scaling, dtype):
        asked.append("rope_tables")
        angle = position_ids[..., None].float() * inv_freq.float()
        angle = torch.cat([angle, angle], -1)
        return (angle.cos() * scaling).to(dtype), (angle.sin() * scaling).to(dtype)

    monkeypatch.setattr(_native, "on_hip", lambda t: True)
    for kernel in (rms_norm, add_rms_norm, rope_tables):
        monkeypatch.setattr(_native, kernel.__name__, kernel)
    monkeypatch.setattr(_native, "linear", lambda x, w, b=None, addend=None: torch.nn.functional.linear(x, w, b))
    return asked


def llama():
    torch.manual_seed(0)
    model = tf.LlamaModel(tf.LlamaConfig(vocab_size=32, hidden_size=32, intermediate_size=48, num_hidden_layers=1, num_attention_heads=2)).eval()
    with torch.no_grad():
        for p in model.parameters():
            p.add_(torch.randn_like(p) * 0.1)
    return model.requires_grad_(False)


def sharded():
    model = llama()
    shard_modules.install_shard_kernels(model)
    return model


def run_layer(model, x):
    position_ids = torch.arange(x.shape[1])[None]
    return model.layers[0](x, position_embeddings=model.rotary_emb(x, position_ids), position_ids=position_ids)


def test_the_kernels_are_asked(kernels):
    own, model, x = llama(), sharded(), torch.randn(2, 5, 32)
    with torch.no_grad():
        assert torch.allclose(model.norm(x), own.norm(x), atol=1e-6) and kernels == ["rms_norm"]
        for _ in range(2):  # the first call of a gated MLP settles which forward it keeps
            kernels.clear()
            assert torch.allclose(run_layer(model, x), run_layer(own, x), atol=1e-5)
        assert kernels == ["rope_tables", "rms_norm", "add_rms_norm"]


def test_forward_mode_derivatives_go_through(kernels):
    own, model, x, t = llama(), sharded(), torch.randn(2, 5, 32), torch.randn(2, 5, 32)
    with torch.no_grad():
        run_layer(model, x)
    kernels.clear()
    with torch.no_grad(), forward_ad.dual_level():
        want, got = (forward_ad.unpack_dual(m.norm(forward_ad.make_dual(x, t))) for m in (own, model))
        assert torch.equal(got.primal, want.primal) and torch.equal(got.tangent, want.tangent)
        # the Linears have no derivative, so a layer's tangent is that of its residual stream
        assert forward_ad.unpack_dual(run_layer(model, forward_ad.make_dual(x, t))).tangent is not None
        weight = model.norm.weight.detach()
        del model.norm.weight
        model.norm.weight = forward_ad.make_dual(weight, torch.ones(32))
        assert forward_ad.unpack_dual(model.norm(x)).tangent is not None
    assert not kernels


class _Seen(torch.utils._python_dispatch.TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.calls = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.calls.append(func)
        return func(*args, **(kwargs or {}))


def test_what_follows_the_torch_calls_sees_the_modules_own(kernels):
    """vmap, vmap over stacked weights, jvp, tracing, compilation, a dispatch mode and a tensor subclass: kernels on raw memory would raise or go unseen."""
    from torch.fx.experimental.proxy_tensor import make_fx

    own, model, x = llama(), sharded(), torch.randn(3, 5, 32)
    position_ids = torch.arange(5)[None]
    with torch.no_grad():
        run_layer(model, x)
        kernels.clear()
        want = own.norm(x)
        assert torch.equal(torch.func.vmap(model.norm)(x), want)
        stacked = torch.stack([own.norm.weight, 2 * own.norm.weight])
        many = torch.func.vmap(lambda w: torch.func.functional_call(model.norm, {"weight": w}, (x,)))(stacked)
        assert torch.equal(many, torch.stack([want, 2 * want]))
        assert torch.equal(torch.func.vmap(lambda r: run_layer(model, r[None])[0])(x), torch.func.vmap(lambda r: run_layer(own, r[None])[0])(x))
        shifted = torch.func.vmap(lambda p: model.rotary_emb(x, p))(torch.stack([position_ids, position_ids + 7]))
        assert torch.equal(shifted[0][1], own.rotary_emb(x, position_ids + 7)[0])
        assert torch.equal(torch.func.jvp(model.norm, (x,), (x,))[1], torch.func.jvp(own.norm, (x,), (x,))[1])
        for traced in (torch.jit.trace(model.norm, x, check_trace=False), make_fx(model.norm)(x), torch.fx.symbolic_trace(model.norm), torch.compile(model.norm, backend="eager", fullgraph=True)):
            assert torch.equal(traced(x + 1), own.norm(x + 1))
        assert torch.equal(make_fx(model.rotary_emb)(x, position_ids)(x, position_ids + 3)[0], own.rotary_emb(x, position_ids + 3)[0])
        with _Seen() as seen:
            assert torch.equal(model.norm(x), want)
        assert len(seen.calls) > 3
        assert torch.equal(model.norm(x.as_subclass(type("Sub", (torch.Tensor,), {}))), want)
    assert not kernels


def test_a_norm_can_be_scripted(kernels):
    own, model, x = llama(), sharded(), torch.randn(2, 5, 32)
    with torch.no_grad():
        assert torch.equal(torch.jit.script(model.norm)(x), own.norm(x)) and not kernels
        model.norm(x)
    assert kernels == ["rms_norm"]


class _Doubled(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        out = func(*args, **(kwargs or {}))
        return 2 * out if func in (torch.rsqrt, torch.Tensor.cos) else out


def test_a_function_mode_sees_the_modules_own_calls(kernels):
    own, model, x, position_ids = llama(), sharded(), torch.randn(2, 5, 32), torch.arange(5)[None]
    with torch.no_grad():
        with _Doubled():
            assert torch.equal(model.norm(x), own.norm(x)) and torch.equal(model.rotary_emb(x, position_ids)[0], own.rotary_emb(x, position_ids)[0])
            assert not kernels
        with torch.device("cpu"):  # a default device is a function mode too, of no account here
            model.norm(x)
    assert kernels == ["rms_norm"]


def test_a_mask_inside_a_transform_is_transformers_own(monkeypatch):
    from transformers.masking_utils import causal_mask_function, sdpa_mask

    from tensor_parallel_amd.attention import attention_mask_of

    asked = []
    monkeypatch.setattr(_native, "on_hip", lambda t: True)
    monkeypatch.setattr(_native, "causal_mask", lambda q_offset, kv_offset, rows, cols: asked.append(rows) or (
        torch.arange(cols) + kv_offset <= torch.arange(rows)[:, None] + q_offset)[None, None])

    def mask(build, q_offset):
        return build(batch_size=2, q_length=3, kv_length=9, q_offset=q_offset, kv_offset=0, attention_mask=None, mask_function=causal_mask_function,
                     allow_is_causal_skip=False, use_vmap=False, device=torch.device("cpu"), dtype=torch.float32, config=None)

    offsets = torch.tensor([2, 5])
    assert torch.equal(mask(attention_mask_of, offsets[0]), mask(sdpa_mask, offsets[0])) and asked == [3]
    assert torch.equal(torch.func.vmap(lambda o: mask(attention_mask_of, o))(offsets), torch.stack([mask(sdpa_mask, o) for o in offsets]))
    assert asked == [3]


@pytest.mark.parametrize("name", ["sdpa_mask", "causal_mask_function"])
def test_a_mask_function_that_a_program_has_put_in_place_is_honoured(monkeypatch, name):
    from transformers import masking_utils

    from tensor_parallel_amd.attention import attention_mask_of

    asked = []
    monkeypatch.setattr(_native, "on_hip", lambda t: True)
    monkeypatch.setattr(_native, "causal_mask", lambda q_offset, kv_offset, rows, cols: asked.append(rows))
    offset = torch.tensor(4)

    def form():
        return dict(batch_size=2, q_length=3, kv_length=9, q_offset=offset, kv_offset=0, attention_mask=None, mask_function=masking_utils.causal_mask_function,
                    allow_is_causal_skip=False, use_vmap=False, device=torch.device("cpu"), dtype=torch.float32, config=None)

    stock = masking_utils.sdpa_mask(**form())
    if name == "sdpa_mask":
        monkeypatch.setattr(masking_utils, name, lambda **kwargs: ~stock)
    else:  # a window of two keys
        monkeypatch.setattr(masking_utils, name, lambda batch_idx, head_idx, q_idx, kv_idx: (kv_idx <= q_idx) & (kv_idx > q_idx - 2))
    want = masking_utils.sdpa_mask(**form())
    assert not torch.equal(want, stock) and torch.equal(attention_mask_of(**form()), want) and not asked


def _replacements():
    import functools

    from transformers.models.llama import modeling_llama as ml

    def norm(self, hidden_states):  # another formula
        return hidden_states * self.weight + self.variance_epsilon

    def rotary(self, x, position_ids):  # another position scaling
        angle = position_ids[..., None].float() * self.inv_freq / 4
        angle = torch.cat([angle, angle], -1)
        return angle.cos().to(x.dtype), angle.sin().to(x.dtype)

    def layer(self, hidden_states, **kwargs):
        return 2 * hidden_states

    own = ml.LlamaRMSNorm.forward

    @functools.wraps(own)
    def around(self, hidden_states):  # a wrapper that looks like what it wraps
        return 3 * own(self, hidden_states)

    own_tables = ml.LlamaRotaryEmbedding.forward
    scaled = functools.wraps(own_tables)(lambda self, x, position_ids: own_tables(self, x, position_ids * 2))
    return [(ml.LlamaRMSNorm, norm), (ml.LlamaRMSNorm, around), (ml.LlamaRotaryEmbedding, rotary), (ml.LlamaRotaryEmbedding, scaled), (ml.LlamaDecoderLayer, layer)]


@pytest.mark.parametrize("which", range(5))
@pytest.mark.parametrize("when", ["before", "after", "between"])
def test_a_forward_that_a_program_has_put_in_place_is_honoured(kernels, monkeypatch, which, when):
    """... also where it was put there behind the shards' making, and where the shards' classes were made before it."""
    cls, forward = _replacements()[which]
    x = torch.randn(2, 5, 32)

    def everything(model):
        return model.norm(x), *model.rotary_emb(x, torch.arange(5)[None]), run_layer(model, x)

    if when != "before":
        with torch.no_grad():
            stock = sharded()
            run_layer(stock, x)
    if when != "after":
        monkeypatch.setattr(cls, "forward", forward)
    model = stock if when == "after" else sharded()
    monkeypatch.setattr(cls, "forward", forward)
    own = llama()
    with torch.no_grad():
        run_layer(model, x)
        for got, want in zip(everything(model), everything(own)):
            assert torch.allclose(got, want, atol=1e-5)
    monkeypatch.undo()


def test_a_parametrised_norm_or_layer_runs_its_own_forward_once(kernels):
    """A parametrisation makes a subclass of the fused class: falling back to the next class of the method resolution order came back here for ever."""
    from torch.nn.utils import parametrize

    class Doubled(torch.nn.Module):
        def forward(self, w):
            return 2 * w

    own, model, x = llama(), sharded(), torch.randn(2, 5, 32)
    for m in (own, model):
        parametrize.register_parametrization(m.norm, "weight", Doubled())
        m.layers[0].extra = torch.nn.Parameter(torch.zeros(1), requires_grad=False)
        parametrize.register_parametrization(m.layers[0], "extra", Doubled())
    for mode in (torch.no_grad, torch.enable_grad):
        with mode():
            assert torch.equal(model.norm(x.double()), own.norm(x.double()))  # a promoting norm: its own forward
            assert torch.allclose(model.norm(x), own.norm(x), atol=1e-6)
            assert torch.allclose(run_layer(model, x), run_layer(own, x), atol=1e-5)


def test_an_unpickled_layer_has_the_name_of_its_class(tmp_path):
    """In a process that has made no shard before: programs look decoder layers up by the name of their class."""
    import os
    import pickle
    import subprocess
    import sys

    import tensor_parallel_amd

    model = sharded()
    (tmp_path / "model.pkl").write_bytes(pickle.dumps(model))
    code = "import pickle, sys; m = pickle.load(open(sys.argv[1], 'rb')); print(*(type(x).__name__ for x in (m.layers[0], m.norm, m.rotary_emb)))"
    root = os.path.dirname(os.path.dirname(tensor_parallel_amd.__file__))
    child = subprocess.run([sys.executable, "-c", code, str(tmp_path / "model.pkl")], capture_output=True, text=True, timeout=300, cwd=root)
    assert child.returncode == 0, child.stderr
    assert child.stdout.split() == [type(m).__name__ for m in (model.layers[0], model.norm, model.rotary_emb)]
    assert child.stdout.split()[0] == "LlamaDecoderLayer"


@pytest.mark.parametrize("change", [lambda m: m.double(), lambda m: setattr(m, "weight", torch.nn.Parameter(torch.full((1,), 2.0))),
                                    lambda m: setattr(m, "weight", torch.nn.Parameter(torch.arange(160.0).view(5, 32)))])
def test_a_norm_that_the_kernel_does_not_take_keeps_its_own_forward(kernels, change):
    """Another dtype than the kernel's three, and weights that broadcast."""
    own, model = llama(), sharded()
    with torch.no_grad():
        for m in (own, model):
            change(m.norm)
        for dtype in (torch.float32, torch.float64):
            x = torch.randn(2, 5, 32, dtype=dtype)
            got, want = model.norm(x), own.norm(x)
            assert got.dtype == want.dtype and torch.equal(got, want)
        x = torch.randn(2, 5, 32, dtype=torch.float64)
        layers = llama().double().layers[0], sharded().double().layers[0]
        for layer in layers:
            layer.self_attn, layer.mlp = _Attention(), torch.nn.Identity()
        assert torch.equal(layers[0](x), layers[1](x))
    assert not kernels


class _Attention(torch.nn.Module):
    def forward(self, hidden_states, **kwargs):
        return hidden_states * 0.5, None


def test_rotary_tables_take_the_arguments_of_the_modules_own_forward(kernels):
    own, model, x, position_ids = llama(), sharded(), torch.randn(2, 5, 32), torch.arange(5)[None]
    for kwargs in ({}, {"layer_type": None}):
        for got, want in zip(model.rotary_emb(x=x, position_ids=position_ids, **kwargs), own.rotary_emb(x=x, position_ids=position_ids, **kwargs)):
            assert torch.equal(got, want)
    assert kernels == ["rope_tables"]


@pytest.mark.parametrize("B,S,heads,D,takes", [(1, 5, 2, 64, True), (1, 2 ** 24 - 1, 2, 64, True), (1, 2 ** 24, 2, 64, False), (2 ** 24, 1, 4, 128, False), (2 ** 12, 2 ** 12, 2, 64, False),
                                               (2 ** 12, 2 ** 12 - 1, 64, 64, True), (2 ** 12, 2 ** 12 - 1, 65, 64, False), (2 ** 11, 2 ** 12 - 1, 64, 128, True),
                                               (2 ** 11, 2 ** 12 + 1, 64, 128, False), (1, 1, 2 ** 16 - 1, 128, True), (1, 1, 2 ** 16, 128, False)])
def test_rope_takes_what_its_launch_holds(B, S, heads, D, takes):
    """The library's own answer for these sizes, asked with addresses that it refuses in the next step (8 is no multiple of 16)."""
    import ctypes

    assert _native.rope_takes(B, S, heads, D) == takes
    rc = _native.lib().tpamd_rope(8, 8, 8, 8, 8, 8, B, S, heads // 2, heads - heads // 2, D, (ctypes.c_int64 * 14)(*[8] * 14), _native.BF16, None)
    assert rc == (-2 if takes else -1), _native.lib().tpamd_last_error()


@pytest.mark.parametrize("takes", [False, True])
def test_an_attention_that_is_too_long_for_the_rope_kernel_keeps_torchs_rotation(kernels, monkeypatch, takes):
    from tensor_parallel_amd import attention

    torch.manual_seed(0)
    config = tf.LlamaConfig(vocab_size=32, hidden_size=128, intermediate_size=48, num_hidden_layers=1, num_attention_heads=2)
    model = tf.LlamaModel(config).eval().requires_grad_(False).bfloat16()
    shard_modules.install_shard_kernels(model)
    model.config._attn_implementation = attention.register()
    rotated = []

    def attend(module, q, k, v, mask, **kwargs):
        rotated.append((q, k))
        return q.transpose(1, 2), None

    def rope(q, k, cos, sin):
        kernels.append("rope")
        names = shard_modules._globals_of(type(model.layers[0].self_attn)._tp_base.forward)
        return names["apply_rotary_pos_emb"](q.transpose(1, 2), k.transpose(1, 2), cos, sin)

    monkeypatch.setattr(attention, "attention_forward", attend)
    tf.modeling_utils.ALL_ATTENTION_FUNCTIONS.register(attention.IMPLEMENTATION_NAME, attend)
    monkeypatch.setattr(_native, "rope", rope)
    monkeypatch.setattr(_native, "rope_takes", lambda B, S, heads, D: (B, S, heads, D) == (2, 5, 4, 64) and takes)
    monkeypatch.setattr(_native, "linear", lambda x, w, b=None, **_: torch.nn.functional.linear(x, w, b))
    try:
        x, position_ids = torch.randn(2, 5, 128).bfloat16(), torch.arange(5)[None]
        with torch.no_grad():
            model.layers[0].self_attn(x, position_embeddings=model.rotary_emb(x, position_ids), attention_mask=None)
    finally:
        monkeypatch.undo()
        attention.register()
    assert kernels.count("rope") == takes and len(rotated) == 1


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("D,fp32,half", [(2040, False, False), (2048, True, True), (2052, True, False), (2049, False, False), (8192, True, True), (8196, False, False), (8200, False, True),
                                         (16384, False, True), (16392, False, False)])
def test_layer_norms_of_rows_that_the_kernel_does_not_hold_are_torchs(kernels, monkeypatch, D, fp32, half, dtype):
    """Whole 16-byte chunks and up to 32 KiB of them; also of a norm that was moved to another dtype after its class was changed."""
    monkeypatch.setattr(_native, "layer_norm", lambda x, w, b, eps: kernels.append("layer_norm") or torch.nn.functional.layer_norm(x, (D,), w, b, eps))
    takes = {torch.float32: fp32, torch.float16: half}
    for before in takes:
        kernels.clear()
        norm, x = torch.nn.LayerNorm(D).to(before), torch.randn(3, D).to(dtype)
        shard_modules.install_shard_kernels(torch.nn.Sequential(norm))
        assert (type(norm) is shard_modules.ShardLayerNorm) == takes[before]
        with torch.no_grad():
            norm.to(dtype)(x)
        assert kernels == ["layer_norm"] * (takes[before] and takes[dtype])
