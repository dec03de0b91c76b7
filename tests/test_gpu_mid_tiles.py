"""gemm_mid_kernel on each of its tiles: rows and columns just below, at and above whole tiles, the shortest K it takes and one that ends in every stage of the ring,
single matrices and gated pairs, one rank and two, with an addend and a second copy."""
import pytest
import torch

from tensor_parallel_amd import _native

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
TILES = [128192, 128256, 160192, 160256, 192192, 192256, 224192, 224256, 256192, 256256]


@pytest.fixture
def tile(request, monkeypatch):
    monkeypatch.setenv("TPAMD_GEMM_TILE", str(request.param))
    _native.reload_tuning()
    yield request.param
    monkeypatch.undo()
    _native.reload_tuning()


def draw(*shape, dtype, seed, scale=1.0):
    return (torch.randn(*shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(seed)) * scale).to(dtype)


def close(got, want, dtype, roundings=1):
    # every rounding to the dtype: 2^-9 (bf16), 2^-12 (fp16) of a value of up to a few deviations; fp32 sums of at most 448 products stay far below 1 % of a deviation
    eps = 2.0 ** (-8 if dtype is torch.bfloat16 else -11)
    torch.testing.assert_close(got.float(), want, rtol=roundings * eps, atol=(1e-2 + 2 * eps * (roundings - 1)) * want.std().item())


@pytest.mark.parametrize("K", [64, 128, 192, 448])
@pytest.mark.parametrize("over", [-1, 0, 1])
@pytest.mark.parametrize("tile", TILES, indirect=True)
def test_edges_of_a_tile(tile, over, K):
    rows, cols, dtype = 2 * (tile // 1000) + over, 2 * (tile % 1000) + 4 * over, torch.float16 if K % 128 else torch.bfloat16
    xs, ws = [draw(rows, K, dtype=dtype, seed=r) for r in range(2)], [draw(cols, K, dtype=dtype, seed=3 + r, scale=0.1) for r in range(2)]
    wants = [x.float() @ w.float().t() for x, w in zip(xs, ws)]
    for y, want in zip(_native.linear_ranks([(x, w, None) for x, w in zip(xs, ws)]), wants):
        close(y, want, dtype)
    first = _native.linear(xs[0], ws[0])
    copy = torch.empty_like(first)
    total = _native.linear(xs[1], ws[1], addend=first, copy=copy)
    close(total, wants[0] + wants[1], dtype, 3)
    assert torch.equal(total, copy)
    # a pair's tile has half as many columns: two tiles of gate and up rows, 4 rows fewer or more
    half = tile % 1000 + 4 * over
    pairs = [(x, draw(half, K, dtype=dtype, seed=5 + r, scale=0.1), draw(half, K, dtype=dtype, seed=7 + r, scale=0.1)) for r, x in enumerate(xs)]
    for h, (x, g, u) in zip(_native.swiglu_up_ranks(pairs), pairs):
        close(h, torch.nn.functional.silu(x.float() @ g.float().t()) * (x.float() @ u.float().t()), dtype, 4)
