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
