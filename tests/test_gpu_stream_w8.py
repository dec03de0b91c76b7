"""stream_w8_kernel (int8 Linears of 2 to 32 rows and sums of two ranks on one block per CU) where it can go wrong: around its row and column counts, K that does not fill
every wavefront, outlier columns in none, one or several groups per wavefront, every form of the epilogue; TPAMD_STREAM=1 sends it what its rule would leave to others."""
import ctypes

import pytest
import torch

from tensor_parallel_amd import _native

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.fixture(autouse=True)
def forced(monkeypatch):
    monkeypatch.setenv("TPAMD_STREAM", "1")
    _native.reload_tuning()
    yield
    monkeypatch.undo()
    _native.reload_tuning()


def close(got, want, dtype, roundings=1):
    # int8 codes are exact in both dtypes and sums fp32, so what differs is the rounding of the result (2^-9 or 2^-12 of a value of up to a few deviations); fp32 sums stay far below 1 %
    eps = 2.0 ** (-8 if dtype is torch.bfloat16 else -11)
    torch.testing.assert_close(got.float(), want, rtol=roundings * eps, atol=(1e-2 + 2 * eps * (roundings - 1)) * want.std().item())


def rank(rows, cols, K, n_out, dtype, seed):
    """Operands of one rank and its product. Rows past the last one of x and of the weights hold NaN and the largest codes."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(rows + 40, K + 8, device=DEV, generator=g).to(dtype)
    x[rows:], x[:, K:] = float("nan"), float("nan")
    wq = torch.randint(-127, 128, (cols, K), dtype=torch.int8, device=DEV, generator=g)
    idx = torch.randperm(K, device=DEV, generator=g)[:n_out].sort().values.int()
    wq[:, idx.long()] = 0
    scale = torch.rand(cols, device=DEV, generator=g) * 1e-3
    w_out = (torch.randn(cols, n_out, device=DEV, generator=g) * 0.1).to(dtype)
    bias = torch.randn(cols, device=DEV, generator=g).to(dtype) if cols % 8 else None
    x = x[:rows, :K]
    want = (x.double() @ wq.double().t() * scale.double() + x[:, idx.long()].double() @ w_out.double().t() + (0 if bias is None else bias.double())).float()
    return (x, wq, scale, idx if n_out else None, w_out if n_out else None, bias), want


# columns: fewer than a tile, ragged over the CUs, staged rows that are no whole tiles (40), all of the staged rows; K: one unit, fewer units than wavefronts, uneven parts, parts of 4 KiB
SHAPES = [(4, 128, 0), (20, 256, 1), (516, 384, 33), (4608, 640, 40), (5504, 1152, 32), (16384, 512, 200), (1032, 16512, 256), (11000, 1024, 129)]


@pytest.mark.parametrize("rows", [2, 8, 9, 16, 17, 24, 25, 32])
@pytest.mark.parametrize("cols,K,n_out", SHAPES)
def test_linear(rows, cols, K, n_out):
    dtype = torch.float16 if rows % 2 else torch.bfloat16
    calls, wants = zip(*[rank(rows, cols, K, n_out, dtype, seed) for seed in (1, 2)])
    for y, want in zip(_native.linear_w8_ranks(calls), wants):
        close(y, want, dtype)
    first = _native.linear_w8(*calls[0])
    close(first, wants[0], dtype)
    copy = torch.full_like(first, float("nan"))
    total = _native.linear_w8(*calls[1], addend=first, copy=copy)
    close(total, wants[0] + wants[1], dtype, 3)
    assert torch.equal(total, copy)
    close(_native.linear_w8(*calls[0], _native.ACT_GELU), torch.nn.functional.gelu(wants[0]), dtype)


@pytest.mark.parametrize("rows", [2, 8, 9, 16, 17, 24, 25, 32])
@pytest.mark.parametrize("cols,K,n_out", SHAPES[:5] + [(8192, 4096, 20), (1032, 16512, 82)])
def test_sum_of_two_ranks(rows, cols, K, n_out):
    dtype = torch.bfloat16 if rows % 2 else torch.float16
    calls, wants = zip(*[rank(rows, cols, K, n_out, dtype, seed) for seed in (3, 4)])
    sums = _native.linear_w8_sum_ranks(calls)
    close(sums[0], wants[0] + wants[1], dtype, 3)
    assert torch.equal(sums[0], sums[1]) and sums[0].data_ptr() != sums[1].data_ptr()


@pytest.mark.parametrize("rows,cols,K,n_out", [(8, 516, 384, 33), (17, 4608, 640, 0), (32, 1032, 1152, 40)])
def test_pitches_of_weights_and_outputs(rows, cols, K, n_out):
    """Through the C entry point: weights, outlier weights and outputs with room between their rows, which holds the largest codes or NaN and is left alone."""
    dtype = torch.float16
    (x, wq, scale, idx, w_out, bias), want = rank(rows, cols, K, n_out, dtype, 5)
    wide = torch.full((cols, K + 48), 127, dtype=torch.int8, device=DEV)
    wide[:, :K] = wq
    wide_out = torch.full((cols, n_out + 3), float("nan"), dtype=dtype, device=DEV)
    if n_out:
        wide_out[:, :n_out] = w_out
    y = torch.full((rows + 1, cols + 20), 7.0, dtype=dtype, device=DEV)
    rc = _native.lib().tpamd_linear_w8(x.data_ptr(), wide.data_ptr(), scale.data_ptr(), idx.data_ptr() if n_out else None, wide_out.data_ptr() if n_out else None, n_out,
                                       None if bias is None else bias.data_ptr(), y.data_ptr(), rows, cols, K, x.stride(0), K + 48, n_out + 3, cols + 20,
                                       _native.dtype_code(dtype), _native.ACT_NONE, ctypes.c_void_p(torch.cuda.current_stream(DEV).cuda_stream))
    assert rc == 0
    close(y[:rows, :cols], want, dtype)
    assert bool((y[:, cols:] == 7.0).all()) and bool((y[rows] == 7.0).all())
