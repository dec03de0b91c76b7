"""The calls of several ranks in one launch (tpamd_*_ranks, together.py): every rank's result against its own reference in fp32, at sizes on both
sides of every line where the choice of a kernel changes; and ranks that come with different calls, or not at all."""
import pytest
import torch

from tensor_parallel_amd import _native

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def close(got, want, dtype):
    # products rounded once to the dtype: 2^-8 (bf16), 2^-11 (fp16) of the value; sums of K products in fp32 stay far below the floor of 1 % of a deviation
    torch.testing.assert_close(got.float(), want, rtol=2.0 ** (-8 if dtype is torch.bfloat16 else -10), atol=1e-2 * want.std().item())


def draws(n, *shape, dtype, scale=1.0, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return [(torch.randn(*shape, device=DEV, generator=g) * scale).to(dtype) for _ in range(n)]


# rows: the row kernels up to 3, weight streaming up to 16 or 64, tiles of 128 with K splits, mid-sized tiles, 256 x 256
@pytest.mark.parametrize("rows", [1, 2, 3, 4, 12, 16, 17, 40, 64, 65, 300, 700])
@pytest.mark.parametrize("cols,K", [(4, 8), (516, 264), (1376, 2048), (2048, 4096), (3072, 4096), (4100, 1088), (1024, 8192)])
def test_linear_of_two_ranks(rows, cols, K):
    dtype = torch.float16 if rows % 2 else torch.bfloat16
    xs, ws = draws(2, rows, K, dtype=dtype), draws(2, cols, K, dtype=dtype, scale=0.05, seed=1)
    bs = draws(2, cols, dtype=dtype, seed=2) if cols % 8 else [None, None]
    for (x, w, b), y in zip(zip(xs, ws, bs), _native.linear_ranks(list(zip(xs, ws, bs)))):
        close(y, x.float() @ w.float().t() + (0 if b is None else b.float()), dtype)


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 12, 16, 17, 32, 33, 64, 130, 520])
@pytest.mark.parametrize("cols,K", [(4, 8), (1376, 2048), (2752, 4096), (5504, 4096), (5504, 2048), (1028, 1096)])
def test_gated_pair_of_two_ranks(rows, cols, K):
    dtype = torch.bfloat16 if rows % 2 else torch.float16
    xs, gs, us = draws(2, rows, K, dtype=dtype), draws(2, cols, K, dtype=dtype, scale=0.02, seed=1), draws(2, cols, K, dtype=dtype, scale=0.02, seed=2)
    for x, g, u, h in zip(xs, gs, us, _native.swiglu_up_ranks(list(zip(xs, gs, us)))):
        want = torch.nn.functional.silu(x.float() @ g.float().t()) * (x.float() @ u.float().t())
        # gate, SiLU and product are each rounded: 4 roundings of 2^-9 (2^-12) and what SiLU makes of them
        torch.testing.assert_close(h.float(), want, rtol=2e-2, atol=2e-2 * want.std().item())


@pytest.mark.parametrize("rows", [1, 2, 3, 16, 17, 33, 64, 65])
@pytest.mark.parametrize("cols,K,n_out", [(2048, 4096, 20), (9216, 8192, 40), (8192, 16384, 0), (4100, 1040, 3)])
def test_int8_of_two_ranks(rows, cols, K, n_out):
    dtype = torch.float16
    calls, wants = [], []
    for r in range(2):
        x, w = draws(1, rows, K, dtype=dtype, seed=r)[0], draws(1, cols, K, dtype=dtype, scale=0.05, seed=5 + r)[0]
        g = torch.Generator().manual_seed(r)
        keep = torch.randperm(K, generator=g)[:n_out].sort().values
        wz = w.float().clone()
        wz[:, keep.to(DEV)] = 0
        scale = wz.abs().amax(1) / 127
        q = torch.round(wz / scale[:, None]).to(torch.int8)
        idx, w_out = (keep.to(DEV, torch.int32), w[:, keep.to(DEV)].contiguous()) if n_out else (None, None)
        calls.append((x, q, scale, idx, w_out, None))
        want = (x.float() @ q.float().t()) * scale
        wants.append(want + x.float()[:, keep.to(DEV)] @ w_out.float().t() if n_out else want)
    for y, want in zip(_native.linear_w8_ranks(calls), wants):
        close(y, want, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,D,n", [(1, 4096, 2), (5, 8, 3), (129, 4096, 2), (7, 16392, 2), (3, 100, 4)])
def test_norms_of_several_ranks_are_those_of_single_calls(rows, D, n, dtype):
    xs, rs, ws = draws(n, rows, D, dtype=dtype), draws(n, rows, D, dtype=dtype, seed=1), draws(n, D, dtype=dtype, seed=2)
    for x, w, y in zip(xs, ws, _native.rms_norm_ranks([(x, w, 1e-5) for x, w in zip(xs, ws)])):
        assert torch.equal(y, _native.rms_norm(x, w, 1e-5))
    for r, x, w, (total, y) in zip(rs, xs, ws, _native.add_rms_norm_ranks([(r, x, w, 1e-5) for r, x, w in zip(rs, xs, ws)])):
        assert torch.equal(total, r + x) and torch.equal(y, _native.rms_norm(r + x, w, 1e-5))


@pytest.mark.parametrize("on_device", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,D,cached,n", [(1, 16, 16, 128, 500, 2), (3, 16, 2, 128, 65, 2), (2, 8, 8, 64, 0, 2), (5, 32, 4, 64, 1000, 3), (40, 16, 4, 128, 1000, 2)])
def test_decode_of_several_ranks(B, Hq, Hkv, D, cached, n, on_device):
    dtype, room = torch.bfloat16, cached + 3
    calls, alone = [], []
    for r in range(n):
        q, k, v = (draws(1, B, 1, h, D, dtype=dtype, seed=10 * r + i)[0] for i, h in enumerate((Hq, Hkv, Hkv)))
        cos, sin = (draws(1, B, 1, D, dtype=dtype, seed=10 * r + 3 + i)[0] for i in range(2))
        caches = [draws(1, B, Hkv, room, D, dtype=dtype, seed=10 * r + 5 + i)[0] for i in range(2)]
        count = torch.tensor([cached - (r if cached and on_device else 0)], device=DEV)  # counts on the device may differ
        calls.append((q, k, v, cos, sin, *caches, count if on_device else cached, None))
        alone.append((q, k, v, cos, sin, *[c.clone() for c in caches], count if on_device else cached, None))
    outs = _native.attention_decode_rope_ranks(calls)
    for call, mine, out in zip(calls, alone, outs):
        want = _native.attention_decode_rope(*mine)
        assert torch.equal(call[5], mine[5]) and torch.equal(call[6], mine[6])
        # The key range is cut in other places, so probabilities are rounded to the dtype (2^-9 of each) against other maxima: over the keys that adds
        # up to 2^-9 * sqrt(2 / 3) = 1.6e-3 deviations of the result, 4.5 times that for the largest of 80000; and one rounding of the result on each side.
        torch.testing.assert_close(out.float(), want.float(), rtol=2.0 ** -7, atol=2e-2 * want.float().std().item())


def test_ranks_that_do_not_fit_each_other_make_their_calls_alone():
    from tensor_parallel_amd.tensor_parallel import RANK_GREENLETS, _apply_in_greenlets

    if not RANK_GREENLETS:
        pytest.skip("the ranks of a device are threads")
    from tensor_parallel_amd import together

    x, w = draws(2, 5, 256, dtype=torch.bfloat16), draws(2, 512, 256, dtype=torch.bfloat16, seed=1)
    side = torch.cuda.Stream()

    def rank(r):
        def body(turns):
            outs = []
            for turn in turns:
                if turn == "both":
                    outs.append(together.linear(x[r], w[r]))
                elif turn == "different":
                    outs.append(together.linear(x[r], w[r][: 128 * (r + 1)]))
                elif turn == "one" and r == 1:
                    outs.append(together.linear(x[r], w[r]))
                elif turn == "stream":  # a stream of the rank's own: the turn stays
                    with torch.cuda.stream(side):
                        side.wait_stream(torch.cuda.default_stream())
                        outs.append(together.linear(x[r], w[r]))
                    torch.cuda.current_stream().wait_stream(side)
            return outs
        return body

    calls = []
    many = _native.linear_ranks
    try:
        _native.linear_ranks = lambda items: calls.append(len(items)) or many(items)
        with torch.no_grad():
            got = _apply_in_greenlets([rank(0), rank(1)], [(["both", "different", "stream", "one", "both"],)] * 2, [{}] * 2, DEV)
    finally:
        _native.linear_ranks = many
    torch.cuda.synchronize()
    assert calls == [2, 2]
    for r in range(2):
        full = x[r].float() @ w[r].float().t()
        wants = [full, full[:, : 128 * (r + 1)], full] + ([full] if r else []) + [full]
        assert len(got[r]) == len(wants)
        for a, b in zip(got[r], wants):
            close(a, b, torch.bfloat16)


@pytest.mark.parametrize("first", ["library call", "collective"])
def test_a_rank_that_waits_in_a_stream_of_its_own_leaves_its_peers_theirs(first):
    """Rank 1 waits in a collective inside a stream and an inference mode of its own, rank 0 for a library call that nobody else makes or for that collective."""
    from tensor_parallel_amd import together
    from tensor_parallel_amd.collectives import CollectiveOperation
    from tensor_parallel_amd.tensor_parallel import _apply_in_greenlets

    side, op = torch.cuda.Stream(), CollectiveOperation(2, lambda *xs: [sum(xs)] * 2, timeout=5.0)
    x, w = draws(1, 5, 256, dtype=torch.bfloat16)[0], draws(1, 128, 256, dtype=torch.bfloat16, seed=1)[0]
    streams = {0: [], 1: []}

    def body(r):
        here = lambda: streams[r].append((torch.cuda.current_stream(), torch.is_inference_mode_enabled(), torch.is_grad_enabled()))  # noqa: E731
        here()
        if r == 0:
            y = together.linear(x, w) if first == "library call" else None
            for _ in range(3):
                op(1, 0)
                here()
            return y
        op(2, 1) if first == "collective" else None
        with torch.inference_mode(), torch.cuda.stream(side):
            for _ in range(3 - (first == "collective")):
                op(2, 1)
                here()
        here()

    with torch.no_grad():
        main = torch.cuda.current_stream()
        y, _ = _apply_in_greenlets([body, body], [(0,), (1,)], [{}] * 2, DEV)
        assert torch.cuda.current_stream() == main and not torch.is_grad_enabled()
    torch.cuda.synchronize()
    assert all(seen == (main, False, False) for seen in streams[0]) and len(streams[0]) == 4
    assert streams[1][0] == streams[1][-1] == (main, False, False) and all(seen == (side, True, False) for seen in streams[1][1:-1])
    if y is not None:
        close(y, x.float() @ w.float().t(), torch.bfloat16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows", [1, 3, 4, 16, 33, 64, 129, 700])
@pytest.mark.parametrize("cols,K,n", [(4, 8, 2), (384, 768, 2), (3072, 768, 2), (1000, 1088, 2), (516, 264, 3), (7, 30, 2)])
def test_gathered_linears_are_the_linears_side_by_side(rows, cols, K, n, dtype):
    xs, ws = draws(n, rows, K, dtype=dtype), draws(n, cols, K, dtype=dtype, scale=0.05, seed=1)
    bs = draws(n, cols, dtype=dtype, seed=2) if rows % 2 else [None] * n
    ys = _native.linear_gather_ranks(list(zip(xs, ws, bs)))
    want = torch.cat([x.double() @ w.double().t() + (0 if b is None else b.double()) for x, w, b in zip(xs, ws, bs)], -1)
    assert len({y.data_ptr() for y in ys}) == n and all(torch.equal(y, ys[0]) for y in ys)
    if dtype is torch.float32:  # sums of K products in fp32: at most K * 2^-24 of the sum of their magnitudes
        bound = K * 2.0 ** -24 * max(float((x.abs().double() @ w.abs().double().t()).max()) for x, w in zip(xs, ws)) + 1e-6
        assert float((ys[0].double() - want).abs().max()) <= bound
    else:
        close(ys[0], want.float(), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows", [1, 3, 4, 16, 17, 64, 129, 700, 2100])
@pytest.mark.parametrize("cols,K", [(4, 8), (516, 264), (4096, 2048), (1030, 1096), (7, 30)])
def test_the_copy_of_a_sum_is_the_sum(rows, cols, K, dtype):
    x, w, addend = draws(1, rows, K, dtype=dtype)[0], draws(1, cols, K, dtype=dtype, scale=0.05, seed=1)[0], draws(1, rows, cols, dtype=dtype, seed=2)[0]
    copy = torch.full_like(addend, float("nan"))
    y = _native.linear(x, w, addend=addend, copy=copy)
    assert torch.equal(y, copy) and torch.equal(y, _native.linear(x, w, addend=addend))


@pytest.mark.parametrize("rank", [0, 1])
def test_a_sum_that_somebody_writes_to_is_copied_as_it_is(rank):
    from types import SimpleNamespace

    import tensor_parallel_amd as tp
    from tensor_parallel_amd.slicing_configs import get_llama_config
    from torch import nn

    class Mlp(nn.Module):
        def __init__(self):
            super().__init__()
            self.gate_proj, self.up_proj, self.down_proj = nn.Linear(64, 128, bias=False), nn.Linear(64, 128, bias=False), nn.Linear(128, 64, bias=False)
            self.act_fn = nn.SiLU()

        def forward(self, x):
            return self.down_proj(self.act_fn(self.gate_proj(x)) * self.up_proj(x))

    class Block(nn.Module):
        def __init__(self):
            super().__init__()
            self.mlp = Mlp()

        def forward(self, x):
            return self.mlp(x)

    torch.manual_seed(0)
    cfg = get_llama_config(SimpleNamespace(model_type="llama", hidden_size=64, num_attention_heads=4, num_key_value_heads=4), [DEV] * 2)
    model = tp.TensorParallel(Block().bfloat16().to(DEV), [DEV] * 2, tensor_parallel_config=cfg, sharded=False)
    x = torch.randn(5, 64, device=DEV).bfloat16()
    with torch.no_grad():
        want = [model(x) for _ in range(3)][-1]
        # one of the ranks comes last and its down projection holds the sum: what a hook adds to that in place is in the sum of both ranks
        handle = model.module_shards[rank].mlp.tp_wrapped_module.down_proj.register_forward_hook(lambda m, i, out: out.add_(1.0))
        ranks = []
        for shard in model.module_shards:
            shard.register_forward_hook(lambda m, i, out: ranks.append(out))
        model(x)
        handle.remove()
    assert len(ranks) == 2 and torch.equal(ranks[0], ranks[1])
    torch.testing.assert_close(ranks[0], want + 1.0, rtol=0, atol=3 * 2.0 ** -8)  # added before or after the sum: three roundings of values below 2, 2^-8 each


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 2, 4, 17, 64, 65, 130, 300, 1024])
@pytest.mark.parametrize("cols,K,n_out,gelu", [(2048, 4096, 20, False), (8192, 16384, 41, False), (1028, 1088, 0, True), (4100, 1040, 3, False)])
def test_int8_linear_adds_a_partial_sum_and_copies_it(rows, cols, K, n_out, gelu, dtype):
    g = torch.Generator(device=DEV).manual_seed(rows)
    x, addend = draws(1, rows, K, dtype=dtype)[0], draws(1, rows, cols, dtype=dtype, seed=2)[0]
    q = torch.randint(-127, 128, (cols, K), device=DEV, generator=g, dtype=torch.int8)
    scale = torch.rand(cols, device=DEV, generator=g) * 1e-3
    idx = torch.arange(0, 2 * n_out, 2, device=DEV, dtype=torch.int32) if n_out else None
    w_out = draws(1, cols, n_out, dtype=dtype, seed=3)[0] if n_out else None
    act = _native.ACT_GELU if gelu else _native.ACT_NONE
    plain = _native.linear_w8(x, q, scale, idx, w_out, act=act)
    copy = torch.full_like(addend, float("nan"))
    y = _native.linear_w8(x, q, scale, idx, w_out, act=act, addend=addend, copy=copy)
    assert torch.equal(y, plain + addend) and torch.equal(copy, y)
    assert torch.equal(_native.linear_w8(x, q, scale, idx, w_out, act=act, addend=addend), y)


# rows: the row kernel, weight streaming with one, two and four tiles of rows, K ranges of 128 x 128 tiles with part and whole tiles of x; K on both sides of 1024 and of
# the row kernel's 11 pieces, ragged chunks
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 2, 3, 4, 15, 16, 17, 32, 33, 64, 65, 130, 512, 700, 2100])
@pytest.mark.parametrize("cols,K,bias", [(4096, 2048, False), (4096, 5504, False), (1028, 1024, True), (516, 1040, False), (2048, 1000, False), (4, 5640, True), (8192, 4096, False), (5120, 1088, True), (1024, 2048, False)])
def test_the_sum_of_two_ranks_linears(rows, cols, K, bias, dtype):
    xs, ws = draws(2, rows, K, dtype=dtype), draws(2, cols, K, dtype=dtype, scale=0.05, seed=1)
    bs = draws(2, cols, dtype=dtype, seed=2) if bias else [None, None]
    sums = _native.linear_sum_ranks(list(zip(xs, ws, bs)))
    if sums is None:  # left to two launches
        assert not _native.linear_sum_pays(rows, cols, K, dtype)
        return
    parts = [x.double() @ w.double().t() + (0 if b is None else b.double()) for x, w, b in zip(xs, ws, bs)]
    assert sums[0].data_ptr() != sums[1].data_ptr() and torch.equal(*sums)
    # each product rounded to the dtype, then their sum: three roundings, each of half a unit in the last place, and fp32 sums of K products
    u = 2.0 ** (-8 if dtype is torch.bfloat16 else -11)
    want = parts[0] + parts[1]
    bound = u * (parts[0].abs() + parts[1].abs() + want.abs()) * 1.02 + K * 2.0 ** -24 * want.std()
    assert bool(((sums[0].double() - want).abs() <= bound + 1e-30).all())
    alone = _native.linear(xs[1], ws[1], bs[1], addend=_native.linear(xs[0], ws[0], bs[0]))
    assert (sums[0].double() - want).norm() <= 1.05 * (alone.double() - want).norm()


@pytest.mark.parametrize("rows", [1, 2, 5, 16, 17, 48, 64, 65])
@pytest.mark.parametrize("cols,K,n_out", [(2048, 4096, 20), (8192, 16384, 81), (4100, 4112, 3), (16384, 8192, 0)])
def test_the_sum_of_two_ranks_int8_linears(rows, cols, K, n_out):
    dtype, calls, parts = torch.float16, [], []
    for r in range(2):
        g = torch.Generator(device=DEV).manual_seed(r)
        x = draws(1, rows, K, dtype=dtype, seed=r)[0]
        q = torch.randint(-127, 128, (cols, K), device=DEV, generator=g, dtype=torch.int8)
        scale = torch.rand(cols, device=DEV, generator=g) * 1e-3
        idx = torch.randperm(K, device=DEV, generator=g)[:n_out].sort().values.to(torch.int32) if n_out else None
        w_out = draws(1, cols, n_out, dtype=dtype, seed=3 + r)[0] if n_out else None
        calls.append((x, q, scale, idx, w_out, None))
        parts.append(_native.linear_w8(*calls[-1]))
    sums = _native.linear_w8_sum_ranks(calls)
    if sums is None:  # no planes to add up, or too many rows: these two matrices split K over blocks
        assert (cols, K) not in ((8192, 16384), (16384, 8192)) or rows not in (16, 17, 48)
        return
    assert rows not in (1, 65)
    assert sums[0].data_ptr() != sums[1].data_ptr() and torch.equal(*sums)
    want = parts[0].float() + parts[1].float()  # both rounded products, each of which may be rounded the other way where the planes are cut elsewhere
    bound = 2.0 ** -11 * (want.abs() + 2 * (parts[0].float().abs() + parts[1].float().abs())) + 1e-6
    assert bool(((sums[0].float() - want).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape,n", [((1, 1), 2), ((3, 7), 3), ((1, 4096), 2), ((5, 257), 2), ((40, 4096), 2)])
def test_small_calls_of_several_ranks(shape, n, dtype):
    a, b = draws(n, *shape, dtype=dtype), draws(n, *shape, dtype=dtype, seed=1)
    assert all(torch.equal(c, x + y) for x, y, c in zip(a, b, _native.add_ranks(list(zip(a, b)))))
    counts = [torch.tensor(10 + r, device=DEV) for r in range(n)]
    assert all(x is y for x, y in zip(_native.advance_ranks([(c, 3) for c in counts]), counts)) and [int(c) for c in counts] == [13 + r for r in range(n)]
    rows, cols = shape
    offsets = [torch.tensor([cols // 2 + r], device=DEV) for r in range(n)]
    for offset, mask in zip(offsets, _native.causal_mask_ranks([(o, 1, rows, cols) for o in offsets])):
        assert torch.equal(mask, _native.causal_mask(offset, 1, rows, cols))
        assert torch.equal(mask[0, 0], torch.arange(cols, device=DEV)[None] + 1 <= offset + torch.arange(rows, device=DEV)[:, None])
    freqs, positions = draws(n, 32, dtype=torch.float32, seed=2), [torch.arange(rows * 3, device=DEV).view(rows, 3) + 7 * r for r in range(n)]
    for f, p, got in zip(freqs, positions, _native.rope_tables_ranks([(f, p, 1.5, dtype) for f, p in zip(freqs, positions)])):
        assert all(torch.equal(x, y) for x, y in zip(got, _native.rope_tables(f, p, 1.5, dtype)))


@pytest.mark.parametrize("rows", [60, 61, 64])
def test_two_ranks_whose_partial_sums_outgrow_a_streams_buffer_take_their_own_kernels(rows):
    """Nine planes of 16384 columns for each of two ranks: 71.3 MB of scratch memory hold them up to 60 rows."""
    cols, K, n_out, calls = 16384, 8192, 41, []
    for r in range(2):
        g = torch.Generator(device=DEV).manual_seed(r)
        q = torch.randint(-127, 128, (cols, K), device=DEV, generator=g, dtype=torch.int8)
        idx = torch.randperm(K, device=DEV, generator=g)[:n_out].sort().values.to(torch.int32)
        calls.append((draws(1, rows, K, dtype=torch.float16, seed=r)[0], q, torch.rand(cols, device=DEV, generator=g) * 1e-3, idx,
                      draws(1, cols, n_out, dtype=torch.float16, seed=3 + r)[0], None))
    _native.linear_w8(calls[0][0][:8], *calls[0][1:])  # this stream's buffer has the usual size
    assert 9 * 60 * cols * 4 * 2 <= _native.scratch_of_stream(DEV)[1] < 9 * 61 * cols * 4 * 2
    for y, call in zip(_native.linear_w8_ranks(calls), calls):
        alone = _native.linear_w8(*call)
        x, q, scale, idx, w_out, _ = call
        want = x.double() @ (q.double() * scale.double()[:, None]).t() + x[:, idx.long()].double() @ w_out.double().t()
        close(y, want.float(), torch.float16)
        if rows > 60:  # the same kernel, which adds up in the same order
            assert torch.equal(y, alone)
