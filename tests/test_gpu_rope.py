"""tpamd_rope_append on the GPU against the oracle, bit for bit: rotated queries in the attention layout, rotated keys and
the values at their cache positions, every other cache position untouched."""
import pytest
import torch

from oracle import attention as oat
from oracle import rope as orp
from tensor_parallel_amd import _native

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def bits(t):
    return t.detach().cpu().contiguous().view(torch.int16)


def fused_qkv(B, S, Hq, Hkv, D, dtype, seed):
    """q / k / v as views of one fused projection output laid out [B, S, Hkv, Hq/Hkv + 2, D] (the Falcon-40B shard's
    query_key_value: per key/value head its query heads, then the key, then the value)."""
    g = torch.Generator().manual_seed(seed)
    per = Hq // Hkv
    fused = torch.randn(B, S, Hkv, per + 2, D, generator=g).to(dtype)
    return fused


def run_case(B, S, Hq, Hkv, D, dtype, pos0, L, shared_angles=True, seed=0, by_group=False):
    fused = fused_qkv(B, S, Hq, Hkv, D, dtype, seed)
    per = Hq // Hkv
    pos = torch.arange(pos0, pos0 + S)
    cos, sin = orp.angles(pos, D, dtype=dtype)
    if shared_angles:
        cos, sin = cos[None], sin[None]
    else:  # a different position offset per batch entry
        tables = [orp.angles(pos + 3 * b, D, dtype=dtype) for b in range(B)]
        cos, sin = torch.stack([t[0] for t in tables]), torch.stack([t[1] for t in tables])
    g = torch.Generator().manual_seed(seed + 1)
    kc = torch.randn(B, Hkv, L, D, generator=g).to(dtype)
    vc = torch.randn(B, Hkv, L, D, generator=g).to(dtype)
    # host: the oracle on contiguous copies of the three parts
    q_h = fused[:, :, :, :per].reshape(B, S, Hq, D)
    k_h, v_h = fused[:, :, :, per], fused[:, :, :, per + 1]
    want_q, want_kc, want_vc = orp.rope_append(q_h, k_h, v_h, cos, sin, kc, vc, pos0)
    # device: strided views of the fused tensor, no copies. The query heads of one key/value head are contiguous rows of
    # D and the groups are (per + 2) * D apart: a 5-d view [B, S, Hkv, per, D]; a plain 4-d view exists with one group
    # or one query head per group; `by_group` passes the groups one by one with q_out views instead
    fd = fused.to(DEV)
    kcd, vcd = kc.to(DEV), vc.to(DEV)
    cd, sd = cos.to(DEV), sin.to(DEV)
    if not by_group:
        qv = fd[:, :, :, :per]
        if Hkv == 1:
            qv = qv.reshape(B, S, Hq, D)
        elif per == 1:
            qv = fd[:, :, :, 0]
        got_q = _native.rope_append(qv, fd[:, :, :, per], fd[:, :, :, per + 1], cd, sd, kcd, vcd, pos0)
    else:
        got_q = torch.empty(B, Hq, S, D, dtype=dtype, device=DEV)
        for gi in range(Hkv):
            _native.rope_append(fd[:, :, gi, :per], fd[:, :, gi:gi + 1, per], fd[:, :, gi:gi + 1, per + 1], cd, sd,
                                kcd[:, gi:gi + 1], vcd[:, gi:gi + 1], pos0, q_out=got_q[:, gi * per:(gi + 1) * per])
    assert torch.equal(bits(got_q), bits(want_q))
    assert torch.equal(bits(kcd), bits(want_kc))
    assert torch.equal(bits(vcd), bits(want_vc))
    return got_q, kcd, vcd


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,S,Hq,Hkv,D,pos0,L", [
    (2, 1, 4, 4, 64, 5, 16),        # decode, equal heads
    (1, 7, 8, 1, 64, 0, 7),         # prefill filling the cache exactly, one key/value head
    (3, 5, 8, 2, 128, 9, 20),       # grouped heads as a 5-d view of the fused output, head_dim 128
    (2, 33, 2, 2, 128, 31, 64),     # more rows than one block of lanes
])
def test_rope_append_bit_exact(dtype, B, S, Hq, Hkv, D, pos0, L):
    run_case(B, S, Hq, Hkv, D, dtype, pos0, L)


def test_groups_one_by_one_into_views_of_the_output():
    run_case(2, 3, 12, 3, 64, torch.float16, 2, 8, seed=9, by_group=True)


def test_per_batch_angles():
    run_case(3, 2, 4, 4, 64, torch.bfloat16, 4, 12, shared_angles=False, seed=5)


def test_falcon_40b_rank_shard_decode_step_pieces():
    """BASELINE config 4 at W = 2, decode: batch 8, one new position on 2047 cached ones, 4 key/value heads with 16
    query heads each, head_dim 64. The cache after the append feeds the attention core; its output equals the oracle's
    attention over the oracle's cache."""
    B, S, Hq, Hkv, D, pos0, L = 8, 1, 64, 4, 64, 2047, 2048
    got_q, kcd, vcd = run_case(B, S, Hq, Hkv, D, torch.bfloat16, pos0, L, seed=7)
    out = _native.attention(got_q, kcd, vcd, causal=True)
    want = oat.attention_f64(got_q.float().cpu().numpy(), kcd.float().cpu().numpy(), vcd.float().cpu().numpy(), D ** -0.5, True)
    want = torch.from_numpy(want)
    torch.testing.assert_close(out.double().cpu(), want, rtol=2e-2, atol=2e-2 * want.std().item())


def test_argument_errors():
    B, S, Hq, Hkv, D = 1, 2, 2, 2, 64
    q = torch.zeros(B, S, Hq, D, dtype=torch.bfloat16, device=DEV)
    k = torch.zeros(B, S, Hkv, D, dtype=torch.bfloat16, device=DEV)
    cos = torch.zeros(1, S, D, dtype=torch.bfloat16, device=DEV)
    cache = torch.zeros(B, Hkv, 4, D, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError):
        _native.rope_append(q, k, k, cos, cos, cache, cache.clone(), 3)  # positions 3, 4 of a cache of 4
    with pytest.raises(ValueError):
        _native.rope_append(q, k, k, cos[:, :1], cos[:, :1], cache, cache.clone(), 0)  # angles for one position only
    with pytest.raises(TypeError):
        _native.rope_append(q.float(), k.float(), k.float(), cos.float(), cos.float(), cache.float(), cache.float(), 0)
    q32 = torch.zeros(B, S, Hq, 32, dtype=torch.bfloat16, device=DEV)
    c32 = torch.zeros(1, S, 32, dtype=torch.bfloat16, device=DEV)
    cache32 = torch.zeros(B, Hkv, 4, 32, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError):
        _native.rope_append(q32, q32, q32, c32, c32, cache32, cache32.clone(), 0)  # head_dim 32: no kernel


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("freq_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,S,half,one_row", [(1, 1, 32, False), (3, 5, 64, False), (2, 257, 64, True), (1, 3, 5, False)])
def test_rope_tables(dtype, freq_dtype, B, S, half, one_row):
    """`tpamd_rope_tables` against the angles in fp32 and their cosines in fp64. fp32 cosines are good to 2 units of 2^-24 (of values up
    to 1); rounding to a dtype with p significant bits (bf16 8, f16 11, fp32 24) adds at most 2^-p of the result, the scaling 2^-24."""
    g = torch.Generator().manual_seed(S)
    pos = torch.randint(0, 8192, (1 if one_row else B, S), generator=g)
    pos = pos.expand(B, S)
    inv = (1.0 / 10000.0 ** (torch.arange(half) / half)).to(freq_dtype)
    cos, sin = _native.rope_tables(inv.to(DEV), pos.to(DEV) if not one_row else pos[:1].to(DEV).expand(B, S), 1.25, dtype)
    angle = (pos[..., None].float() * inv.float()).double()
    angle = torch.cat([angle, angle], -1)
    unit = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}[dtype]
    for got, want in ((cos, angle.cos() * 1.25), (sin, angle.sin() * 1.25)):
        assert got.shape == (B, S, 2 * half) and got.dtype == dtype
        torch.testing.assert_close(got.double().cpu(), want, rtol=unit + 2.0 ** -24, atol=1.25 * 2.0 ** -22)
    with pytest.raises(ValueError):
        _native.rope_tables(inv.to(DEV), pos.to(DEV).int(), 1.0, dtype)


@pytest.mark.parametrize("family", ["llama", "falcon"])
def test_rotary_modules_of_the_shards_use_the_tables(family):
    import transformers as tf

    import tensor_parallel_amd as tp

    torch.manual_seed(0)
    if family == "llama":
        model = tf.LlamaModel(tf.LlamaConfig(vocab_size=96, hidden_size=64, intermediate_size=128, num_hidden_layers=1, num_attention_heads=4,
                                             num_key_value_heads=2)).to(torch.bfloat16).eval()
    else:
        model = tf.FalconModel(tf.FalconConfig(vocab_size=96, hidden_size=256, num_hidden_layers=1, num_attention_heads=4, num_kv_heads=2,
                                               new_decoder_architecture=True, alibi=False, bias=False)).to(torch.bfloat16).eval()
    pos = torch.randint(0, 2048, (2, 7))
    x = torch.zeros(2, 7, 8, dtype=torch.bfloat16)
    want = model.rotary_emb(x, pos)
    split = tp.tensor_parallel(model, [DEV, DEV])
    mine = [m for m in split.modules() if type(m).__name__ in ("ShardLlamaRotaryEmbedding", "ShardFalconRotaryEmbedding")]
    assert len(mine) == 2
    for g, w in zip(mine[1](x.to(DEV), pos.to(DEV)), want):  # the host's fp32 cosines may round the other way on a boundary
        torch.testing.assert_close(g.cpu().float(), w.float(), rtol=2.0 ** -7, atol=1e-6)
    mine[0].rope_type = "dynamic"  # frequencies that change with the length: the module's own forward
    assert mine[0](x.to(DEV), pos.to(DEV))[0].shape == want[0].shape


def test_tables_of_more_elements_than_one_launch_takes():
    """A launch has fewer than 2^32 threads, one per position and frequency here: a batch whose rows go over several launches has them all."""
    S, half, B = 1 << 14, 256, (1 << 10) + 1
    if torch.cuda.mem_get_info(DEV)[0] < 48 << 30:
        pytest.skip("the tables take 35 GB")
    freq = 10000.0 ** (-torch.arange(half, device=DEV) / half)
    positions = torch.arange(S, device=DEV)[None].expand(B, -1) + torch.arange(B, device=DEV)[:, None]
    cos, sin = _native.rope_tables(freq, positions, 1.0, torch.bfloat16)
    for b in (0, B // 2, B - 2, B - 1):
        c, s = _native.rope_tables(freq, positions[b:b + 1], 1.0, torch.bfloat16)
        assert torch.equal(cos[b], c[0]) and torch.equal(sin[b], s[0])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,S,Hq,Hkv,D,shared", [(1, 1, 1, 1, 64, True), (2, 5, 8, 2, 64, False), (3, 129, 16, 16, 128, True), (1, 700, 16, 4, 128, False), (2, 3, 40, 40, 128, True)])
def test_rope_of_whole_sequences_is_transformers(B, S, Hq, Hkv, D, shared, dtype):
    from transformers.models.llama.modeling_llama import apply_rotary_pos_emb

    g = torch.Generator(device="cuda").manual_seed(S)
    qkv = torch.randn(B, S, Hq + 2 * Hkv, D, device="cuda", generator=g).to(dtype)
    q, k = qkv[:, :, :Hq], qkv[:, :, Hq:Hq + Hkv]
    cos, sin = (torch.randn(1 if shared else B, S, D, device="cuda", generator=g).to(dtype) for _ in range(2))
    got = _native.rope(q, k, cos, sin)
    want = apply_rotary_pos_emb(q.transpose(1, 2), k.transpose(1, 2), cos, sin)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_llama_attention_without_a_cache_is_the_modules_own(monkeypatch):
    import transformers.models.llama.modeling_llama as llama
    from transformers import LlamaConfig, LlamaForCausalLM

    import tensor_parallel_amd as tp

    cfg = LlamaConfig(vocab_size=128, hidden_size=256, intermediate_size=512, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2, head_dim=64,
                      attn_implementation="eager")
    torch.manual_seed(0)
    model = LlamaForCausalLM(cfg).bfloat16().eval().cuda()
    model.config._attn_implementation = tp.attention.register()
    split = tp.tensor_parallel(model, ["cuda:0"] * 2)
    ids = torch.randint(0, 128, (3, 37), device="cuda")
    calls = []
    rope = _native.rope
    monkeypatch.setattr(_native, "rope", lambda *a: calls.append(1) or rope(*a))
    with torch.no_grad():
        split(input_ids=ids[:, :5], use_cache=False)
        calls.clear()
        got = split(input_ids=ids, use_cache=False).logits
        assert len(calls) == 4  # two layers, two ranks
        with monkeypatch.context() as m:  # a program's own rotary embedding runs, and so does a replaced forward
            seen = []
            stock = llama.apply_rotary_pos_emb
            m.setattr(llama, "apply_rotary_pos_emb", lambda *a, **k: seen.append(1) or stock(*a, **k))
            own = split(input_ids=ids, use_cache=False).logits
            assert len(seen) == 4 and len(calls) == 4
        assert torch.equal(got, own)
        with monkeypatch.context() as m:
            forward = llama.LlamaAttention.forward
            m.setattr(llama.LlamaAttention, "forward", lambda self, *a, **k: seen.append(2) or forward(self, *a, **k))
            assert torch.equal(split(input_ids=ids, use_cache=False).logits, own) and seen[-4:] == [2] * 4 and len(calls) == 4
