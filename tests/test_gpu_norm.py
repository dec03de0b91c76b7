"""`tpamd_rms_norm` against the definition in fp64 on the host, rounded as the module's own sequence of torch ops rounds: row
lengths at the edges of the kernel's block shapes and outside its vector path."""
import pytest
import torch

from tensor_parallel_amd import _native

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def rms_ref(x, w, eps):
    x64 = x.double()
    n = (x64 * torch.rsqrt(x64.square().mean(-1, keepdim=True) + eps)).to(x.dtype)
    return w * n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,D", [(1, 8), (3, 512), (2, 520), (5, 2048), (2, 2056), (1, 4096), (37, 4096), (3, 4104), (2, 8192), (2, 16384), (2, 16392),
                                    (4, 100), (3, 7)])
def test_rms_norm(dtype, rows, D):
    g = torch.Generator().manual_seed(D)
    x = (torch.randn(rows, D, generator=g) * 3).to(dtype)
    w = (1 + 0.3 * torch.randn(D, generator=g)).to(dtype)
    got = _native.rms_norm(x.to(DEV), w.to(DEV), 1e-5).cpu()
    # the fp32 statistics may put a scaled value on the other side of a rounding boundary: one unit of the dtype in the scaled
    # value, which the product with the weight and its own rounding can carry to two
    unit = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -22}[dtype]
    torch.testing.assert_close(got.double(), rms_ref(x, w, 1e-5).double(), rtol=4 * unit, atol=1e-6)
    if dtype != torch.float32:  # ... and that is rare
        assert (got != rms_ref(x, w, 1e-5)).double().mean().item() < 0.02


def test_rms_norm_takes_strided_rows_and_refuses_what_does_not_fit():
    g = torch.Generator().manual_seed(0)
    big = torch.randn(6, 4096, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.ones(2048, dtype=torch.bfloat16, device=DEV)
    for part in (big[:, 2048:], big[:, 1:2049]):  # 16-byte aligned rows, and rows that are not
        assert torch.equal(_native.rms_norm(part, w, 1e-6), _native.rms_norm(part.contiguous(), w, 1e-6))
    with pytest.raises(ValueError):
        _native.rms_norm(big, w, 1e-6)
    with pytest.raises(ValueError):
        _native.rms_norm(big[:, :2048], w.float(), 1e-6)
    assert _native.rms_norm(big[:0, :2048], w, 1e-6).shape == (0, 2048)


def test_shards_of_a_llama_use_it():
    import transformers as tf

    import tensor_parallel_amd as tp

    torch.manual_seed(0)
    cfg = tf.LlamaConfig(vocab_size=96, hidden_size=64, intermediate_size=128, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2)
    model = tf.LlamaForCausalLM(cfg).to(torch.bfloat16).eval()
    split = tp.tensor_parallel(model, [DEV, DEV])
    norms = [m for m in split.modules() if type(m).__name__ == "ShardLlamaRMSNorm"]
    assert len(norms) == 2 * 5
    x = torch.randn(3, 64).to(torch.bfloat16)
    with torch.no_grad():
        torch.testing.assert_close(norms[0](x.to(DEV)).float().cpu(), model.model.norm(x.to(model.device)).float().cpu(), rtol=2e-2, atol=1e-2)
        promoted = norms[0](x.float().to(DEV))  # another dtype than the weight's: the module's own forward
    assert promoted.dtype == torch.float32


def test_a_norm_that_a_backward_pass_goes_through_keeps_its_gradients():
    import transformers as tf

    import tensor_parallel_amd as tp

    torch.manual_seed(0)
    cfg = tf.LlamaConfig(vocab_size=96, hidden_size=64, intermediate_size=128, num_hidden_layers=1, num_attention_heads=4, num_key_value_heads=2)
    norm = next(m for m in tp.tensor_parallel(tf.LlamaModel(cfg).eval(), [DEV, DEV]).modules() if type(m).__name__ == "ShardLlamaRMSNorm")
    x = torch.randn(5, 64, device=DEV, requires_grad=True)
    w = norm.weight.requires_grad_(True)
    c = torch.randn(5, 64, device=DEV)  # not the norm itself: the length of a normalised row does not depend on x, its gradient is rounding noise
    gx, gw = torch.autograd.grad((norm(x) * c).sum(), (x, w))
    x64, w64 = x.detach().double().requires_grad_(True), w.detach().double().requires_grad_(True)
    want = torch.autograd.grad((w64 * x64 * torch.rsqrt(x64.square().mean(-1, keepdim=True) + norm.variance_epsilon) * c).sum(), (x64, w64))
    # fp32 sums of 64 terms: 64 * 2^-24 of the largest of them
    for g, r in zip((gx, gw), want):
        torch.testing.assert_close(g.double(), r, rtol=1e-5, atol=64 * 2.0 ** -24 * r.abs().max().item())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,D", [(1, 8), (3, 512), (2, 520), (5, 2048), (2, 2056), (37, 4096), (2, 8192), (2, 16384), (2, 16392), (4, 100), (3, 7), (0, 64)])
def test_add_rms_norm_is_the_sum_and_its_norm(dtype, rows, D):
    """Bit for bit what torch's addition and `tpamd_rms_norm` give, also on strided and unaligned rows. The vector and the element-wise
    kernel add their squares in different orders, so the norm of unaligned rows is compared with that of a sum that is unaligned too."""
    g = torch.Generator().manual_seed(D)
    x, r = ((torch.randn(rows, 2 * D + 16, generator=g) * 3).to(dtype).to(DEV) for _ in range(2))
    w = (1 + 0.3 * torch.randn(D, generator=g)).to(dtype).to(DEV)
    odd = torch.empty_like(x)[:, 1:D + 1]
    for a, b in ((x[:, :D].contiguous(), r[:, :D].contiguous()), (x[:, 1:D + 1], r[:, :D]), (x[:, :D], r[:, 16:D + 16])):
        total, y = _native.add_rms_norm(b, a, w, 1e-5)
        want = b + a if a.data_ptr() % 16 == 0 else odd.copy_(b + a)
        assert torch.equal(total, b + a) and torch.equal(y, _native.rms_norm(want, w, 1e-5))
    with pytest.raises(ValueError):
        _native.add_rms_norm(r[:, :D], x[:, :D].double(), w, 1e-5)


def test_decoder_layer_with_the_addition_in_its_norm():
    """The fused layer gives its own forward's bits, and leaves the work to it where a hook watches the norm."""
    import transformers as tf

    import tensor_parallel_amd as tp
    from tensor_parallel_amd import shard_modules

    torch.manual_seed(0)
    cfg = tf.LlamaConfig(vocab_size=96, hidden_size=64, intermediate_size=128, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2)
    split = tp.tensor_parallel(tf.LlamaForCausalLM(cfg).to(torch.bfloat16).eval(), [DEV, DEV])
    layers = [m for m in split.modules() if type(m).forward is shard_modules._llama_layer_forward]
    assert len(layers) == 4 and all(type(m).__name__ == "LlamaDecoderLayer" for m in layers)
    ids = torch.randint(0, 96, (3, 9), device=DEV)
    seen = []
    with torch.no_grad():
        split(input_ids=ids)  # the first call settles which kernels the modules use
        fused = split(input_ids=ids, output_hidden_states=True)
        handles = [m.post_attention_layernorm.register_forward_hook(lambda mod, inp, out: seen.append(inp[0])) for m in layers]
        own = split(input_ids=ids, output_hidden_states=True)
        for h in handles:
            h.remove()
    assert len(seen) == 4 and torch.equal(fused.logits, own.logits)
    assert all(torch.equal(a, b) for a, b in zip(fused.hidden_states, own.hidden_states))


def test_more_rows_than_one_launch_takes():
    """A launch has fewer than 2^32 threads: 2^24 rows of the element-wise kernel (256 threads each) and 2^22 of the widest rows have them all."""
    rows, w = (1 << 24) + 3, torch.tensor([1.0, 2.0, 0.5], device=DEV)
    x = torch.randn(rows, 3, device=DEV)
    total, y = _native.add_rms_norm(x, x, w, 1e-6)
    for at in (slice(0, 5), slice((1 << 23) - 2, (1 << 23) + 2), slice(rows - 5, rows)):
        assert torch.equal(_native.rms_norm(x, w, 1e-6)[at], _native.rms_norm(x[at].contiguous(), w, 1e-6))
        assert torch.equal(total[at], 2 * x[at]) and torch.equal(y[at], _native.rms_norm(2 * x[at], w, 1e-6))


# one row, odd rows; a lone element, a row of less than a chunk, ragged rows (element loads), whole chunks on both sides of every block size, the longest
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,D", [(1, 1), (3, 7), (5, 8), (2, 512), (2, 520), (129, 768), (7, 2048), (3, 2056), (2, 4104), (16, 8192), (2, 8200), (1, 16384), (1, 16392)])
@pytest.mark.parametrize("bias", [True, False])
def test_layer_norm_against_64_bits(rows, D, dtype, bias):
    g = torch.Generator(device="cuda").manual_seed(rows * D)
    x = (torch.randn(rows, D, device="cuda", generator=g) * 2 + 3).to(dtype)
    w, b = (torch.randn(D, device="cuda", generator=g).to(dtype) for _ in range(2))
    b = b if bias else None
    y = _native.layer_norm(x, w, b, 1e-5)
    want = torch.nn.functional.layer_norm(x.double(), (D,), w.double(), None if b is None else b.double(), 1e-5)
    torchs = torch.nn.functional.layer_norm(x, (D,), w, b, 1e-5)
    # one rounding of the result; in fp32 what the sums of D elements leave (pairwise over lanes: log2 of their number), and no further off than torch's own
    eps = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -20}[dtype]
    err, theirs = ((t.double() - want).abs().max().item() for t in (y, torchs))
    assert err <= max(eps * want.abs().max().item(), 1.5 * theirs)
    if D > 8:  # rows that are pieces of longer ones, a pitch that 16-byte loads cannot take
        wide = torch.cat([x, x], -1)[:, 1:D + 1] if D % 2 else torch.cat([x, x[:, :1]], -1)[:, :D]
        got = _native.layer_norm(wide, w, b, 1e-5)
        ref = torch.nn.functional.layer_norm(wide.double(), (D,), w.double(), None if b is None else b.double(), 1e-5)
        assert (got.double() - ref).abs().max().item() <= max(eps * ref.abs().max().item(), 1.5 * theirs)


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 60000.0])
def test_layer_norm_of_extreme_rows_is_torchs(value):
    x = torch.randn(3, 264, device="cuda", dtype=torch.float16)
    x[1, 5] = value
    w, b = torch.ones(264, device="cuda", dtype=torch.float16), torch.zeros(264, device="cuda", dtype=torch.float16)
    want = torch.nn.functional.layer_norm(x, (264,), w, b, 1e-5)
    torch.testing.assert_close(_native.layer_norm(x, w, b, 1e-5), want, rtol=2.0 ** -9, atol=2.0 ** -10, equal_nan=True)  # a rounding on each side


def test_layer_norms_of_a_shard():
    from tensor_parallel_amd.shard_modules import ShardLayerNorm, install_shard_kernels

    D = 2048
    plain = torch.nn.LayerNorm(D).cuda()
    m = torch.nn.Sequential(torch.nn.LayerNorm(D), torch.nn.LayerNorm((2, D)), torch.nn.LayerNorm(D, elementwise_affine=False)).cuda()
    m[0].load_state_dict(plain.state_dict())
    install_shard_kernels(m)
    assert type(m[0]) is ShardLayerNorm and type(m[2]) is torch.nn.LayerNorm
    x = torch.randn(5, 2, D, device="cuda")
    with torch.no_grad():
        torch.testing.assert_close(m(x), torch.nn.functional.layer_norm(torch.nn.functional.layer_norm(plain(x), (2, D)), (D,)), rtol=1e-5, atol=1e-6)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert m[0](x.bfloat16()).dtype == torch.float32 == plain(x.bfloat16()).dtype
        scripted = torch.jit.script(m[0])
        torch.testing.assert_close(scripted(x), plain(x), rtol=1e-5, atol=1e-6)
    y = x.requires_grad_()
    m[0](y).sum().backward()
    assert y.grad is not None
