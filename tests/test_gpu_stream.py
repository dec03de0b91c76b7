"""stream_kernel (decode-sized Linears, gated pairs and sums of two ranks on one block per CU) where it can go wrong: around its row and column counts, K that
does not fill every wavefront, and every form of the epilogue; TPAMD_STREAM=1 sends it what its rule would leave to the other kernels."""
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


def draw(*shape, dtype, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, device=DEV, generator=g) * scale).to(dtype)


def close(got, want, dtype, roundings=1):
    # each rounding to the dtype: 2^-9 (bf16), 2^-12 (fp16) of a value of up to a few deviations; fp32 sums of K products stay far below 1 % of a deviation
    eps = 2.0 ** (-8 if dtype is torch.bfloat16 else -11)
    torch.testing.assert_close(got.float(), want, rtol=roundings * eps, atol=(1e-2 + 2 * eps * (roundings - 1)) * want.std().item())


# columns: fewer than a tile, ragged over the CUs, a last tile of 4, whole tiles, two and three turns; K: one unit, fewer units than wavefronts, uneven parts, parts of 4 KiB
SHAPES = [(4, 64), (20, 128), (516, 192), (3076, 320), (6144, 1088), (5504, 4096), (16000, 512), (1032, 8256), (26000, 256)]


@pytest.mark.parametrize("rows", [2, 8, 9, 16, 17, 24, 25, 33, 40, 41, 48, 49, 64])
@pytest.mark.parametrize("cols,K", SHAPES)
def test_linear(rows, cols, K):
    dtype = torch.float16 if rows % 2 else torch.bfloat16
    xs, ws = [draw(rows, K, dtype=dtype, seed=r) for r in range(2)], [draw(cols, K, dtype=dtype, seed=5 + r, scale=0.05) for r in range(2)]
    bs = [draw(cols, dtype=dtype, seed=9 + r) if cols % 8 else None for r in range(2)]
    wants = [x.float() @ w.float().t() + (0 if b is None else b.float()) for x, w, b in zip(xs, ws, bs)]
    for y, want in zip(_native.linear_ranks(list(zip(xs, ws, bs))), wants):
        close(y, want, dtype)
    for y in _native.linear_gather_ranks(list(zip(xs, ws, bs))):
        close(y, torch.cat(wants, -1), dtype)
    first = _native.linear(xs[0], ws[0], bs[0])
    close(first, wants[0], dtype)
    copy = torch.full_like(first, float("nan"))
    total = _native.linear(xs[1], ws[1], bs[1], addend=first, copy=copy)
    close(total, wants[0] + wants[1], dtype, 3)
    assert torch.equal(total, copy)
    close(_native.linear(xs[0], ws[0], bs[0], act=_native.ACT_GELU), torch.nn.functional.gelu(wants[0]), dtype)


@pytest.mark.parametrize("rows", [2, 8, 9, 16, 17, 32, 33, 40, 64])
@pytest.mark.parametrize("cols,K", SHAPES[:7])
def test_gated_pair(rows, cols, K):
    dtype = torch.bfloat16 if rows % 2 else torch.float16
    xs = [draw(rows, K, dtype=dtype, seed=r) for r in range(2)]
    gs, us = ([draw(cols, K, dtype=dtype, seed=s + r, scale=0.05) for r in range(2)] for s in (5, 9))
    hs = _native.swiglu_up_ranks(list(zip(xs, gs, us)))
    for x, g, u, h in zip(xs, gs, us, hs):
        close(h, torch.nn.functional.silu(x.float() @ g.float().t()) * (x.float() @ u.float().t()), dtype, 4)
    # one rank alone is cut differently
    close(_native.swiglu_up(xs[0], gs[0], us[0]), torch.nn.functional.silu(xs[0].float() @ gs[0].float().t()) * (xs[0].float() @ us[0].float().t()), dtype, 4)


@pytest.mark.parametrize("rows", [2, 8, 9, 17, 32, 33, 40, 64])
@pytest.mark.parametrize("cols,K", SHAPES[:6] + [(8192, 4096), (1032, 8256)])
def test_sum_of_two_ranks(rows, cols, K):
    dtype = torch.float16 if rows % 2 else torch.bfloat16
    calls = [(draw(rows, K, dtype=dtype, seed=r), draw(cols, K, dtype=dtype, seed=5 + r, scale=0.05), draw(cols, dtype=dtype, seed=9 + r) if cols % 8 else None)
             for r in range(2)]
    parts = [x.float() @ w.float().t() + (0 if b is None else b.float()) for x, w, b in calls]
    sums = _native.linear_sum_ranks(calls)
    close(sums[0], parts[0] + parts[1], dtype, 3)
    assert torch.equal(sums[0], sums[1]) and sums[0].data_ptr() != sums[1].data_ptr()


def test_strided_rows_of_x_and_rows_past_the_end_stay_out():
    """Rows of x with room between them, and NaN in the rows behind the last one of x and of the weight: what a clamped load reads is never stored."""
    wide, w = draw(48, 1024, dtype=torch.bfloat16, seed=1), draw(1100, 512, dtype=torch.bfloat16, seed=2, scale=0.05)
    wide[37:], w[1036:] = float("nan"), float("nan")
    y = _native.linear(wide[:37, :512], w[:1036])
    close(y, wide[:37, :512].float() @ w[:1036].float().t(), torch.bfloat16)


@pytest.mark.parametrize("rows,cols,K", [(8, 516, 192), (17, 3076, 320), (40, 1032, 1088)])
def test_pitches_of_weights_and_outputs(rows, cols, K):
    """Through the C entry points: weights and outputs with room between their rows, which holds NaN and is left alone."""
    dtype, code, stream = torch.bfloat16, _native.dtype_code(torch.bfloat16), ctypes.c_void_p(torch.cuda.current_stream(DEV).cuda_stream)
    x, g, u = draw(rows, K, dtype=dtype, seed=1), draw(cols, K + 24, dtype=dtype, seed=2, scale=0.05), draw(cols, K + 24, dtype=dtype, seed=3, scale=0.05)
    g[:, K:], u[:, K:] = float("nan"), float("nan")
    y = torch.full((rows + 1, cols + 20), 7.0, dtype=dtype, device=DEV)
    gate, up = x.float() @ g[:, :K].float().t(), x.float() @ u[:, :K].float().t()
    assert _native.lib().tpamd_linear(x.data_ptr(), g.data_ptr(), None, y.data_ptr(), rows, cols, K, K, K + 24, cols + 20, code, _native.ACT_NONE, stream) == 0
    close(y[:rows, :cols], gate, dtype)
    assert bool((y[:, cols:] == 7.0).all()) and bool((y[rows] == 7.0).all())
    assert _native.lib().tpamd_swiglu_up(x.data_ptr(), g.data_ptr(), u.data_ptr(), y.data_ptr(), rows, cols, K, K, K + 24, cols + 20, code, stream) == 0
    close(y[:rows, :cols], torch.nn.functional.silu(gate) * up, dtype, 4)
    assert bool((y[:, cols:] == 7.0).all()) and bool((y[rows] == 7.0).all())
    both = torch.full((2, rows + 1, cols + 20), 7.0, dtype=dtype, device=DEV)
    two = lambda *t: (ctypes.c_void_p * 2)(*[v.data_ptr() for v in t])
    assert _native.lib().tpamd_linear_sum_ranks(two(x, x), two(g, u), None, two(both[0], both[1]), rows, cols, K, K, K + 24, cols + 20, code, stream) == 0
    close(both[0, :rows, :cols], gate + up, dtype, 3)
    assert torch.equal(both[0], both[1]) and bool((both[:, :, cols:] == 7.0).all()) and bool((both[:, rows] == 7.0).all())
