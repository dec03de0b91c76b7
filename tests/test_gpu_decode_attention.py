"""attention_decode_kernel (one new position, at most 16 query heads per key/value head) at the edges of its tiles, wavefronts and key ranges, against the oracle in
float64 (TPAMD_ATTN_DECODE=1 sends it what its rule would leave to the general kernel): counts of keys around a tile of 16 and a round of four wavefronts, forced key ranges (empty last ones among them), strided caches, NaN behind the last key."""
import pytest
import torch

from oracle import attention as oat
from tensor_parallel_amd import _native

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def draw(*shape, dtype, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


def check(got, q, k, v, scale):
    """The general kernel's probabilities are rounded to the dtype (2^-9 in bf16) before they weigh values of one deviation, and the result is rounded once more: 2^-8
    of a value and about 2^-9 sqrt(2 / 3) deviations, 4.5 times that for the largest of some thousand."""
    want = torch.from_numpy(oat.attention_f64(q.float().numpy(), k.float().numpy(), v.float().numpy(), scale, True))
    torch.testing.assert_close(got.double().cpu(), want, rtol=2.0 ** -7, atol=1e-2 * max(want.std().item(), 0.1))


@pytest.mark.parametrize("splits", [None, 1, 3])
@pytest.mark.parametrize("G,Hkv,D", [(1, 3, 128), (4, 2, 64), (7, 2, 128), (16, 1, 64)])
@pytest.mark.parametrize("keys", [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 129, 1000])
def test_rows_against_the_oracle(keys, G, Hkv, D, splits, monkeypatch):
    if splits is not None:
        monkeypatch.setenv("TPAMD_ATTN_SPLITS", str(splits))
    monkeypatch.setenv("TPAMD_ATTN_DECODE", "1")
    _native.reload_tuning()
    try:
        dtype = torch.bfloat16 if keys % 2 else torch.float16
        q = draw(2, G * Hkv, 1, D, dtype=dtype, seed=1)
        room = [draw(2, keys + 5, Hkv, D, dtype=dtype, seed=s) for s in (2, 3)]  # positions before heads: rows far apart
        for r in room:
            r[:, keys:] = float("nan")
        k, v = (r[:, :keys].transpose(1, 2) for r in room)
        kd, vd = (r.to(DEV)[:, :keys].transpose(1, 2) for r in room)
        check(_native.attention(q.to(DEV), kd, vd, scale=0.1, causal=True), q, k, v, 0.1)
    finally:
        monkeypatch.undo()
        _native.reload_tuning()


@pytest.mark.parametrize("D", [64, 128])
def test_a_head_alone_on_many_keys(D):
    """More than 32 ranges, which the merge takes as it takes fewer."""
    q, k, v = (draw(1, 1, n, D, dtype=torch.float16, seed=s) for n, s in ((1, 1), (40003, 2), (40003, 3)))
    got = _native.attention(q.to(DEV), k.to(DEV), v.to(DEV), scale=0.3, causal=True)
    want = torch.from_numpy(oat.attention_f64(q.float().numpy(), k.float().numpy(), v.float().numpy(), 0.3, True))
    # the result is rounded once (2^-11 of a value); probabilities carry 2^-21 and fp32 sums 2^-24 a step, below 2^-12 deviations of the 40003 weighed values
    torch.testing.assert_close(got.double().cpu(), want, rtol=2.0 ** -10, atol=2.0 ** -9 * want.std().item())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("keys,at", [(64, 0), (64, 63), (65, 64), (75, 74), (79, 33), (1000, 999)])
def test_an_infinite_value_stays_infinite(keys, at, D, dtype):
    """One infinite element among the values: its column is infinite, as in the general kernel, and no other is touched. Equal scores make all probabilities one."""
    q, k, v = (draw(2, 2, n, D, dtype=dtype, seed=s).to(DEV) for n, s in ((1, 1), (keys, 2), (keys, 3)))
    q.zero_()
    v[1, 1, at, 5] = float("inf")
    v[0, 1, at, D - 1] = float("-inf")
    got = _native.attention(q, k, v, scale=0.1, causal=True).float()
    want = v.float().mean(2, keepdim=True).transpose(1, 2)
    assert torch.equal(torch.isinf(got), torch.isinf(want)) and not torch.isnan(got).any()
    finite = torch.isfinite(want)
    # sums of up to 1000 values in fp32, rounded once to the dtype
    torch.testing.assert_close(got[finite], want[finite], rtol=2.0 ** (-8 if dtype is torch.bfloat16 else -11), atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("splits", [1, 4])
@pytest.mark.parametrize("D", [64, 128])
def test_infinities_and_nans_beside_a_new_position(D, splits, dtype, monkeypatch):
    """Infinite and undefined values in the cache, in several ranges, and in the new position: each makes its own column of its own sequence so, and no other. Equal scores: all
    probabilities are one."""
    monkeypatch.setenv("TPAMD_ATTN_SPLITS", str(splits))
    _native.reload_tuning()
    try:
        B, Hkv, keys = 3, 2, 250
        q, k, v, cos, sin = (draw(B, 1, n, D, dtype=dtype, seed=s).to(DEV) for n, s in ((2 * Hkv, 4), (Hkv, 5), (Hkv, 6), (1, 7), (1, 8)))
        kc, vc = (draw(B, Hkv, keys + 1, D, dtype=dtype, seed=s).to(DEV) for s in (9, 10))
        q.zero_()
        vc[0, 1, 70, 5], vc[0, 1, 200, 6], vc[1, 0, 249, D - 1], v[1, 0, 1, 3], v[2, 0, 0, 0] = float("inf"), float("-inf"), float("nan"), float("inf"), float("nan")
        got = _native.attention_decode_rope(q, k, v, cos[:, 0], sin[:, 0], kc, vc, keys, scale=0.1).float()[:, 0]
    finally:
        monkeypatch.undo()
        _native.reload_tuning()
    want = vc.float().mean(2).repeat_interleave(2, 1)  # the new position's values are in the cache now
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want)) and torch.equal(torch.sign(got[torch.isinf(got)]), torch.sign(want[torch.isinf(want)]))
    finite = torch.isfinite(want)
    # sums of 251 values in fp32, rounded once to the dtype
    torch.testing.assert_close(got[finite], want[finite], rtol=2.0 ** (-8 if dtype is torch.bfloat16 else -11), atol=1e-5)


@pytest.mark.parametrize("G,D", [(1, 128), (16, 64)])
@pytest.mark.parametrize("count", [1, 15, 16, 17, 31, 32, 33, 64])
def test_few_keys_take_one_kernel_wherever_the_count_is(count, G, D):
    """A step on a cache of fixed length, whose count is on the device, and on a cache that holds just these keys: one range on the same kernel, so the same bits."""
    B, Hkv, dtype = 3, 2, torch.bfloat16
    q, k, v, cos, sin = (draw(B, 1, n, D, dtype=dtype, seed=s).to(DEV) for n, s in ((G * Hkv, 4), (Hkv, 5), (Hkv, 6), (1, 7), (1, 8)))
    cos, sin = cos[:, 0], sin[:, 0]
    kc, vc = (draw(B, Hkv, 65, D, dtype=dtype, seed=s).to(DEV) for s in (9, 10))
    k1, v1, k2, v2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
    grown = _native.attention_decode_rope(q, k, v, cos, sin, k1, v1, count, scale=0.1)
    fixed = _native.attention_decode_rope(q, k, v, cos, sin, k2, v2, torch.tensor([count], device=DEV), scale=0.1)
    assert torch.equal(grown, fixed) and torch.equal(k1, k2) and torch.equal(v1, v2)


@pytest.mark.parametrize("splits", [1, 4])
@pytest.mark.parametrize("G,D", [(1, 128), (4, 128), (16, 64)])
@pytest.mark.parametrize("count", [-1, 0, 1, 63, 64, 200, 255, 256])
def test_new_position_with_the_count_on_the_device(count, G, D, splits, monkeypatch):
    """Against the general kernel (TPAMD_ATTN_DECODE=0): the same caches bit for bit, the same rows but for the rounding of probabilities against other maxima."""
    monkeypatch.setenv("TPAMD_ATTN_SPLITS", str(splits))
    B, Hkv, L, dtype = 3, 2, 256, torch.bfloat16
    q, k, v = draw(B, 1, G * Hkv, D, dtype=dtype, seed=4), draw(B, 1, Hkv, D, dtype=dtype, seed=5), draw(B, 1, Hkv, D, dtype=dtype, seed=6)
    cos, sin, kc, vc = draw(B, 1, D, dtype=dtype, seed=7), draw(B, 1, D, dtype=dtype, seed=8), draw(B, Hkv, L, D, dtype=dtype, seed=9), draw(B, Hkv, L, D, dtype=dtype, seed=10)
    outs = []
    try:
        for general in (False, True):
            if general:
                monkeypatch.setenv("TPAMD_ATTN_DECODE", "0")
            _native.reload_tuning()
            kd, vd = kc.to(DEV), vc.to(DEV)
            out = _native.attention_decode_rope(q.to(DEV), k.to(DEV), v.to(DEV), cos.to(DEV), sin.to(DEV), kd, vd, torch.tensor([count], device=DEV), scale=0.1)
            outs.append((out.float().cpu(), kd.cpu(), vd.cpu()))
    finally:
        monkeypatch.undo()
        _native.reload_tuning()
    (a, ka, va), (b, kb, vb) = outs
    assert torch.equal(ka, kb) and torch.equal(va, vb)
    torch.testing.assert_close(a, b, rtol=2.0 ** -7, atol=1e-2 * max(b.std().item(), 0.1))
