"""A switch that names a kernel (TPAMD_SKINNY_*, TPAMD_GEMV_ROWS, TPAMD_GEMM_TILE and its K splits, TPAMD_ATTN_RING) is followed also where the rules would have taken
stream_kernel or attention_decode_kernel. Which kernel ran is seen in the bits: both sides sum in fixed orders of their own, and of some ten thousand rounded sums some
differ between two orders."""
import pytest
import torch

from tensor_parallel_amd import _native

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def draw(*shape, seed, scale=1.0):
    return (torch.randn(*shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(seed)) * scale).half()


def linear(rows, cols, K):
    x, w = draw(rows, K, seed=1), draw(cols, K, seed=2, scale=0.05)
    return lambda: _native.linear(x, w)


def pair(rows, cols, K):
    x, g, u = draw(rows, K, seed=1), draw(cols, K, seed=2, scale=0.05), draw(cols, K, seed=3, scale=0.05)
    return lambda: _native.swiglu_up(x, g, u)


def sums(rows, cols, K):
    calls = [(draw(rows, K, seed=r), draw(cols, K, seed=5 + r, scale=0.05), None) for r in range(2)]

    def run():
        both = _native.linear_sum_ranks(calls)  # None: two launches
        return both[0] if both is not None else _native.linear(*calls[1], addend=_native.linear(*calls[0]))

    return run


@pytest.mark.parametrize("make,rows,cols,K,knobs", [
    (linear, 12, 5504, 4096, {"TPAMD_SKINNY_RESIDENT": 1}),
    (linear, 12, 5504, 4096, {"TPAMD_SKINNY_CG": 2}),
    (linear, 3, 4096, 4096, {"TPAMD_GEMV_ROWS": 8}),
    (linear, 40, 4608, 2048, {"TPAMD_SKINNY_MAX_M": 64}),
    (linear, 40, 4608, 2048, {"TPAMD_SKINNY_MAX_M": 16}),
    (linear, 40, 4608, 2048, {"TPAMD_GEMM_TILE": 128, "TPAMD_GEMM_SPLITK": 8}),
    (linear, 48, 4608, 2048, {"TPAMD_GEMM_TILE": 256, "TPAMD_GEMM_SPLITK256": 3}),
    (linear, 24, 4608, 4096, {"TPAMD_GEMM_TILE": 128192}),
    (pair, 12, 5504, 11008, {"TPAMD_SKINNY_XLDS": 0}),
    (pair, 12, 5504, 11008, {"TPAMD_SKINNY_PAIR": 0, "TPAMD_SKINNY_XLDS": 0}),
    (pair, 40, 5504, 4096, {"TPAMD_GEMM_TILE": 128}),
    (sums, 24, 4096, 4096, {"TPAMD_GEMM_TILE": 128, "TPAMD_GEMM_SPLITK": 4}),
    (sums, 24, 4096, 4096, {"TPAMD_SKINNY_MAX_M": 16}),
])
def test_a_named_kernel_runs(make, rows, cols, K, knobs, tune):
    run = make(rows, cols, K)
    chosen = run()
    tune("TPAMD_STREAM", 1)
    stream = run()
    assert torch.equal(chosen, stream)  # a shape that the rule takes
    for knob, value in knobs.items():
        tune(knob, value)
    assert torch.equal(run(), stream)  # named as well: TPAMD_STREAM=1 comes first
    tune("TPAMD_STREAM", 0)
    named = run()
    assert not torch.equal(named, stream)
    tune("TPAMD_STREAM", "")  # as if it were not set
    assert torch.equal(run(), named)


@pytest.mark.parametrize("ring", [0, 1])
@pytest.mark.parametrize("D", [64, 128])
def test_a_named_form_of_the_general_attention_kernel_runs(D, ring, tune):
    q, k, v = draw(8, 16, 1, D, seed=1), draw(8, 16, 700, D, seed=2), draw(8, 16, 700, D, seed=3)
    run = lambda: _native.attention(q, k, v, causal=True)
    decode = run()
    tune("TPAMD_ATTN_RING", ring)
    named = run()
    assert not torch.equal(named, decode)
    tune("TPAMD_ATTN_DECODE", 0)
    assert torch.equal(run(), named)


@pytest.mark.parametrize("heads,keys,D,general", [(8, 64, 128, True), (4, 33, 64, True), (8, 32, 128, False), (8, 65, 128, False), (32, 64, 128, False), (320, 60, 128, True),
                                                  (512, 64, 64, False), (640, 64, 64, True)])
def test_one_tile_of_keys_takes_the_faster_attention_kernel(heads, keys, D, general, tune):
    """33 to 64 keys without a new position, where attention_decode_kernel measured slower (256 CUs)."""
    q, k, v = draw(heads // 4, 4, 1, D, seed=1), draw(heads // 4, 4, keys, D, seed=2), draw(heads // 4, 4, keys, D, seed=3)
    run = lambda: _native.attention(q, k, v, causal=True)
    chosen = run()
    both = []
    for decode in (0, 1):
        tune("TPAMD_ATTN_DECODE", decode)
        both.append(run())
    assert not torch.equal(*both) and torch.equal(chosen, both[0 if general else 1])


@pytest.mark.parametrize("rows,cols,K,stream", [(4, 2048, 14336, False), (8, 2048, 11264, False), (3, 2048, 14336, True), (4, 2048, 6144, True), (4, 3072, 14336, True)])
def test_int8_sums_on_half_of_the_cus_leave_stream_kernel(rows, cols, K, stream, tune):
    """Two ranks' sums of 2048 columns, half a block per CU: on long rows other launches measured faster from 4 rows on."""
    g = torch.Generator(device=DEV).manual_seed(1)
    calls = [(draw(rows, K, seed=r), torch.randint(-127, 128, (cols, K), dtype=torch.int8, device=DEV, generator=g), torch.rand(cols, device=DEV, generator=g) * 1e-3, None, None, None)
             for r in range(2)]

    def run():
        both = _native.linear_w8_sum_ranks(calls)
        return both[0] if both is not None else _native.linear_w8(*calls[1], addend=_native.linear_w8(*calls[0]))

    chosen = run()
    tune("TPAMD_STREAM", 1)
    assert torch.equal(chosen, run()) == stream
