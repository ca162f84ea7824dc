"""The tiled bfloat16 product of many rows: every tile and epilogue at the edges of tiles, and the plan that picks tiles."""

import math

import pytest
import torch

DEV = "cuda:0"


def ops():
    from llmserve.ops import library

    return library


def rnd(*shape, seed=0, scale=1.0):
    return (scale * torch.randn(*shape, generator=torch.Generator().manual_seed(seed))).to(torch.bfloat16)


def product(x, w, bias=None):
    y = x.double() @ w.double().t()
    return y if bias is None else y + bias.double()


def close(got, want, k, rounded=True):
    """32-bit sums of k products of bfloat16 numbers in some order, then (rounded) one rounding to bfloat16."""
    top = float(want.abs().max())
    bound = 2e-6 * math.sqrt(k) * top + (2.0 ** -8 * top if rounded else 0.0)
    assert (got.cpu().double() - want).abs().max() <= bound


TILES = range(12)


def sizes_of(tile):
    bm, bn, _, stages, *_ = ops().GEMM_TILES[tile]
    return bm, bn, 64 * stages


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
def test_plain_and_parts(tile):
    bm, bn, step = sizes_of(tile)
    # one row, a row less and more than a tile, several tiles; N of one block, beside a tile's end, several tiles; K of one
    # step, one round of the buffers, a step more and less than two, ten
    for m, n, k in ((1, 16, 64), (bm - 1, bn + 16, step), (bm + 1, bn - 16, 2 * step + 64), (17, 48, 2 * step - 64),
                    (2 * bm + 9, 3 * bn + 48, 10 * step)):
        x, w, b = rnd(m, k + 8, seed=m)[:, :k], rnd(n, k, seed=n), rnd(n, seed=3)
        xd = rnd(m, k + 8, seed=m).to(DEV)[:, :k]
        want = product(x, w, b)
        for dtype in (torch.bfloat16, torch.float32):
            out = torch.full((m + 1, n + 4), 7.0, dtype=dtype, device=DEV)
            ops().gemm_tiles(out[:m, :n], xd, w.to(DEV), b.to(DEV), tile=tile)
            close(out[:m, :n], want, k, dtype == torch.bfloat16)
            assert bool((out[m:] == 7.0).all()) and bool((out[:, n:] == 7.0).all())
        want = product(x, w)
        for parts in (2, 3, 5):
            if (parts - 1) * -(-(k // 64) // parts) < k // 64:
                sums = torch.full((parts, m, n), 7.0, device=DEV)
                ops().gemm_tiles(sums, xd, w.to(DEV), tile=tile)
                close(sums.double().sum(0), want, k, False)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(17))
def test_bands(tile):
    """Seven tiles along M are walked in bands, the last of which is lower: every tile is there once, in one part of K and in two."""
    bm, bn, _ = sizes_of(tile)
    m, n, k = 7 * bm - 5, 13 * bn - 16, 128
    x, w = rnd(m, k, seed=11).to(DEV), rnd(n, k, seed=12).to(DEV)
    want = (x.double() @ w.double().t()).cpu()
    out = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=DEV)
    ops().gemm_tiles(out[:m], x, w, tile=tile)
    close(out[:m], want, k)
    assert bool((out[m:] == 7.0).all())
    sums = torch.full((2, m, n), 7.0, device=DEV)
    ops().gemm_tiles(sums, x, w, tile=tile)
    close(sums.double().sum(0), want, k, False)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("limit,gelu", [(None, False), (1.5, False), (None, True)])
def test_gated(tile, limit, gelu):
    """SiLU to the bit what the plain product followed by the activation's own kernel gives; the other units, which read the sums
    unrounded, number by number against 64 bits."""
    bm, bn, step = sizes_of(tile)
    for m, inter, k in ((1, 16, 64), (bm + 3, bn // 2 + 16, 2 * step + 64), (bm - 1, bn + 32, step)):
        x, w = rnd(m, k, seed=5), rnd(2 * inter, k, seed=6, scale=k ** -0.5)
        out = torch.full((m, inter + 4), 7.0, dtype=torch.bfloat16, device=DEV)
        ops().gemm_tiles(out[:, :inter], x.to(DEV), w.to(DEV), swiglu=True, limit=limit, gelu=gelu, tile=tile)
        assert bool((out[:, inter:] == 7.0).all())
        if limit is None and not gelu:
            wide = ops().gemm_tiles(torch.empty(m, 2 * inter, dtype=torch.bfloat16, device=DEV), x.to(DEV), w.to(DEV), tile=tile)
            assert torch.equal(out[:, :inter], ops().silu_mul(torch.empty(m, inter, dtype=torch.bfloat16, device=DEV), wide))
            continue
        y = product(x, w)
        gate, up = y[:, :inter], y[:, inter:]
        if limit is not None:
            g, factor = gate.clamp(max=limit), up.clamp(-limit, limit) + 1
            unit = g * torch.sigmoid(1.702 * g)
        else:
            unit, factor = torch.nn.functional.gelu(gate, approximate="tanh"), up
        # the result's rounding (8 bits: half a step of 2^-7); the sums' error (as in `close`) through either factor, the units' slopes being below 1.2; the unit's
        # own arithmetic in 32-bit, which loses gelu's small values beside its argument
        sums = 2e-6 * math.sqrt(k) * float(y.abs().max())
        bound = (2.0 ** -8 + 1e-5) * (unit * factor).abs() + sums * (1.2 * factor.abs() + unit.abs()) + 1e-6 * (gate * factor).abs()
        assert ((out[:, :inter].cpu().double() - unit * factor).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("nh,nkv,d,bs,bias", [(4, 2, 64, 16, True), (3, 1, 32, 8, False), (2, 2, 128, 5, True), (5, 1, 96, 32, False)])
def test_rotary(tile, nh, nkv, d, bs, bias):
    """To the bit what the plain product followed by the rotation's own kernel gives."""
    bm, _, step = sizes_of(tile)
    m, k, n = bm + 21, 2 * step, (nh + 2 * nkv) * d
    x, w = rnd(m, k, seed=7).to(DEV), rnd(n, k, seed=8, scale=k ** -0.5).to(DEV)
    b = rnd(n, seed=9).to(DEV) if bias else None
    positions = (torch.arange(m, dtype=torch.int32) * 7 % 4096).to(DEV)
    inv_freq = (1.0 / (1e4 ** (torch.arange(0, d, 2, dtype=torch.float32) / d))).to(DEV)
    pages = -(-(m + 4) // bs) + 1
    slots = torch.arange(3, m + 3, dtype=torch.int32)  # (a run that starts inside a page, with a hole and a jump)
    slots[m // 2] = -1
    slots[-1] = pages * bs - 1
    slots = slots.to(DEV)
    pools = [torch.full(shape, 7.0, dtype=torch.bfloat16, device=DEV)
             for shape in ((pages, nkv, bs, d), (pages, nkv, d, bs)) for _ in range(2)]
    for freq in (inv_freq, None):
        qkv = ops().gemm_tiles(torch.empty(m, n, dtype=torch.bfloat16, device=DEV), x, w, b, tile=tile)
        ops().rope_store(qkv, freq, positions, slots, pools[0], pools[2], nh, nkv, d, bs)
        rope = dict(n_heads=nh, n_kv_heads=nkv, head_dim=d, inv_freq=freq, positions=positions, slots=slots, k_pool=pools[1],
                    v_pool=pools[3], block_size=bs)
        q = ops().gemm_tiles(torch.empty(m, nh * d, dtype=torch.bfloat16, device=DEV), x, w, b, rope=rope, tile=tile)
        assert torch.equal(q, qkv[:, :nh * d])
        assert torch.equal(pools[0], pools[1]) and torch.equal(pools[2], pools[3])
    # without slots nothing is stored
    rope.update(slots=None, inv_freq=inv_freq)
    ops().gemm_tiles(q, x, w, b, rope=rope, tile=tile)
    assert torch.equal(pools[0], pools[1]) and torch.equal(pools[2], pools[3])


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("pad", [0, 4, 8])
def test_rows_of_every_alignment(tile, pad):
    """Results leave in 16-byte pieces along rows, or in 8-byte ones where rows do not start on 16: the same numbers, and none
    beside them."""
    bm, bn, step = sizes_of(tile)
    m, n, k = bm + 19, bn + 32, step
    x, w = rnd(m, k, seed=11).to(DEV), rnd(n, k, seed=12, scale=k ** -0.5).to(DEV)
    want = product(x.cpu(), w.cpu())
    for dtype in (torch.bfloat16, torch.float32):
        out = torch.full((m + 1, n + pad), 7.0, dtype=dtype, device=DEV)
        ops().gemm_tiles(out[:m, :n], x, w, tile=tile)
        close(out[:m, :n], want, k, dtype == torch.bfloat16)
        assert bool((out[m:] == 7.0).all()) and bool((out[:, n:] == 7.0).all())
    wide = ops().gemm_tiles(torch.empty(m, n, dtype=torch.bfloat16, device=DEV), x, w, tile=tile)
    out = torch.full((m + 1, n // 2 + pad), 7.0, dtype=torch.bfloat16, device=DEV)
    ops().gemm_tiles(out[:m, :n // 2], x, w, swiglu=True, tile=tile)
    assert torch.equal(out[:m, :n // 2], ops().silu_mul(torch.empty(m, n // 2, dtype=torch.bfloat16, device=DEV), wide))
    assert bool((out[m:] == 7.0).all()) and bool((out[:, n // 2:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("bs,first,pad", [(16, 0, 0), (16, 8, 8), (16, 5, 0), (24, 8, 4), (20, 0, 0)])
def test_rotary_tokens_anywhere_in_their_pages(tile, bs, first, pad):
    """Runs of tokens that start anywhere in a page, with a hole and eight tokens backwards, pages of sizes that are powers of two and
    others; several heads a tile, and a tile between q, k and v: to the bit what the rotation's own kernel stores."""
    bm, _, step = sizes_of(tile)
    m, k, nh, nkv, d = bm + 40, step, 5, 3, 64
    n = (nh + 2 * nkv) * d
    x, w = rnd(m, k, seed=13).to(DEV), rnd(n, k, seed=14, scale=k ** -0.5).to(DEV)
    positions = torch.arange(m, dtype=torch.int32, device=DEV)
    inv_freq = (1.0 / (1e4 ** (torch.arange(0, d, 2, dtype=torch.float32) / d))).to(DEV)
    pages = -(-(m + first) // bs) + 1
    slots = torch.arange(first, m + first, dtype=torch.int32)
    slots[9] = -1                                       # a hole in a run
    slots[24:32] = torch.flip(slots[24:32], [0])        # eight tokens backwards
    slots = slots.to(DEV)
    pools = [torch.full(shape, 7.0, dtype=torch.bfloat16, device=DEV)
             for shape in ((pages, nkv, bs, d), (pages, nkv, d, bs)) for _ in range(2)]
    qkv = ops().gemm_tiles(torch.empty(m, n, dtype=torch.bfloat16, device=DEV), x, w, tile=tile)
    ops().rope_store(qkv, inv_freq, positions, slots, pools[0], pools[2], nh, nkv, d, bs)
    q = torch.full((m, nh * d + pad), 7.0, dtype=torch.bfloat16, device=DEV)
    rope = dict(n_heads=nh, n_kv_heads=nkv, head_dim=d, inv_freq=inv_freq, positions=positions, slots=slots, k_pool=pools[1],
                v_pool=pools[3], block_size=bs)
    ops().gemm_tiles(q[:, :nh * d], x, w, rope=rope, tile=tile)
    assert torch.equal(q[:, :nh * d], qkv[:, :nh * d]) and bool((q[:, nh * d:] == 7.0).all())
    assert torch.equal(pools[0], pools[1]) and torch.equal(pools[2], pools[3])


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["plain", "columns of a wider weight", "transposed weight", "every other column of x", "one row many times",
                                  "no weight rows", "no columns", "32-bit bias", "every other number of a bias", "bias of one number",
                                  "bias of rows", "every other column of out", "transposed out"])
def test_what_the_tiles_do_not_take_goes_to_the_library(what):
    """`linear` with many rows takes any strides of its operands and its result, no rows or columns, and any bias that can be added."""
    from llmserve.parts.linear import linear

    m, n, k = 100, 256, 512
    x, w, bias = rnd(m, k, seed=1).to(DEV), rnd(n, k, seed=2, scale=k ** -0.5).to(DEV), None
    wide, out = rnd(m, 2 * k, seed=3).to(DEV), None
    if what == "columns of a wider weight":
        w = rnd(n, k + 8, seed=4, scale=k ** -0.5).to(DEV)[:, :k]
    elif what == "transposed weight":
        w = rnd(k, n, seed=4, scale=k ** -0.5).to(DEV).t()
    elif what == "every other column of x":
        x = wide[:, ::2]
    elif what == "one row many times":
        x = wide[:1, :k].expand(m, k)
    elif what == "no weight rows":
        w = w[:0]
    elif what == "no columns":
        x, w = x[:, :0], w[:, :0].contiguous()
    elif what == "32-bit bias":
        bias = rnd(n, seed=5).float().to(DEV)
    elif what == "every other number of a bias":
        bias = rnd(2 * n, seed=5).to(DEV)[::2]
    elif what == "bias of one number":
        bias = rnd(1, seed=5).to(DEV)
    elif what == "bias of rows":
        bias = rnd(m, n, seed=5).to(DEV)
    elif what == "every other column of out":
        out = torch.empty(m, 2 * n, dtype=torch.bfloat16, device=DEV)[:, ::2]
    elif what == "transposed out":
        out = torch.empty(n, m, dtype=torch.bfloat16, device=DEV).t()
    got = linear(x, w, bias, out=out)
    assert tuple(got.shape) == (m, w.shape[0]) and (out is None or got.data_ptr() == out.data_ptr())
    if got.numel():
        close(got, product(x.cpu(), w.cpu(), None if bias is None else bias.cpu()), k)


@pytest.mark.gpu
def test_what_the_kernel_cannot_take_is_refused():
    x, w = rnd(70, 256).to(DEV), rnd(64, 256).to(DEV)
    out = torch.empty(70, 64, dtype=torch.bfloat16, device=DEV)
    for bad in (lambda: ops().gemm_tiles(out, x[:, :96], w[:, :96].contiguous()),              # K in steps of 64
                lambda: ops().gemm_tiles(out[:, :56], x, w[:56].contiguous()),                  # N in blocks of 16
                lambda: ops().gemm_tiles(out, x.float(), w.float()),
                lambda: ops().gemm_tiles(out[:, :48], x, w),
                lambda: ops().gemm_tiles(torch.empty(70, 66, dtype=torch.bfloat16, device=DEV)[:, 1:65], x, w),
                lambda: ops().gemm_tiles(out, x, w, w[0, :64], swiglu=True),
                lambda: ops().gemm_tiles(torch.empty(2, 70, 64, device=DEV, dtype=torch.bfloat16), x, w)):
        with pytest.raises(ValueError):
            bad()


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["angles", "slots", "k_pool", "v_pool"])
def test_a_rotation_from_host_memory_is_refused(name):
    m, d, k = 70, 64, 128
    rope = dict(n_heads=2, n_kv_heads=1, head_dim=d, inv_freq=None, positions=torch.zeros(m, dtype=torch.int32, device=DEV),
                angles=torch.zeros(m, d // 2, 2, device=DEV), slots=torch.zeros(m, dtype=torch.int32, device=DEV),
                k_pool=torch.zeros(5, 1, 16, d, dtype=torch.bfloat16, device=DEV),
                v_pool=torch.zeros(5, 1, d, 16, dtype=torch.bfloat16, device=DEV), block_size=16)
    rope[name] = rope[name].cpu()
    with pytest.raises(ValueError):
        ops().gemm_tiles(torch.empty(m, 2 * d, dtype=torch.bfloat16, device=DEV), rnd(m, k).to(DEV), rnd(4 * d, k).to(DEV), rope=rope)


def test_plan():
    """The plan names a tile, and no more parts than were allowed or than K has steps for."""
    for m in (17, 64, 65, 128, 333, 512, 2048, 8191):
        for n, k in ((16, 128), (2560, 2048), (2048, 5632), (22016, 4096), (4096, 11008), (160, 384)):
            for most in (1, 2, 4):
                tile, parts = ops().gemm_tiles_plan(m, n, k, most)
                assert 0 <= tile < len(ops().GEMM_TILES) and 1 <= parts <= most
                assert (parts - 1) * -(-(k // 64) // parts) < k // 64
    assert ops().gemm_tiles_plan(128, 2048, 5632, 4)[1] == 4 and ops().gemm_tiles_plan(2048, 2048, 2048, 4)[1] == 1


@pytest.mark.gpu
@pytest.mark.parametrize("epilogue", ["gated", "rotary"])
@pytest.mark.parametrize("m,rows", [(512, 2048), (560, 2047), (700, 1), (512, 33), (512, 9000), (333, 2048), (1300, 2048)])
def test_a_weight_brought_nearer_changes_nothing(epilogue, m, rows):
    """Compute units without a tile read a weight of `rows` rows meanwhile (more, fewer and odd numbers of pieces, behind one round of
    tiles and behind several; none of too large a weight, and none where there are too few such units for it): the same bits, and the
    weight as it was."""
    k, nh, nkv, d = 2048, 32, 4, 64
    near = rnd(rows, k, seed=21).to(DEV)
    before, x = near.clone(), rnd(m, k, seed=22).to(DEV)
    n = 2 * 5632 if epilogue == "gated" else (nh + 2 * nkv) * d
    w = rnd(n, k, seed=23, scale=k ** -0.5).to(DEV)
    rope = dict(n_heads=nh, n_kv_heads=nkv, head_dim=d, inv_freq=None, positions=None, slots=None, k_pool=None, v_pool=None, block_size=16)
    form = dict(swiglu=True) if epilogue == "gated" else dict(rope=rope)
    outs = [ops().gemm_tiles(torch.empty(m, 5632 if epilogue == "gated" else nh * d, dtype=torch.bfloat16, device=DEV), x, w, near=v, **form)
            for v in (None, near, near[rows // 2:])]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2]) and torch.equal(near, before)
    tile = ops().gemm_tiles_plan(m, n, k)[0]
    workers = ops().gemm_tiles_workers(tile, m, n, k, 1, near.numel() * 2, ops().compute_units(near.device))
    bm, bn = sizes_of(tile)[:2]
    assert workers <= -(-(-(-m // bm) * -(-n // bn)) // 256) * 256 - -(-m // bm) * -(-n // bn)
    assert (workers > 0) == (rows != 9000 and (epilogue, m) != ("rotary", 333))


@pytest.mark.gpu
def test_a_weight_to_bring_nearer_that_is_refused():
    x, w = rnd(128, 64, seed=24).to(DEV), rnd(64, 64, seed=25).to(DEV)
    with pytest.raises(ValueError, match="contiguous"):
        ops().gemm_tiles(torch.empty(128, 32, dtype=torch.bfloat16, device=DEV), x, w, swiglu=True, near=w.t())
    with pytest.raises(ValueError, match="near goes"):
        ops().gemm_tiles(torch.empty(128, 64, dtype=torch.bfloat16, device=DEV), x, w, near=w)


def tiles_with(loading):
    from llmserve.ops.library import GEMM_TILES

    return [t for t, tile in enumerate(GEMM_TILES) if tile[-1] == loading]


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(12, 17))
def test_the_tiles_added_later(tile):
    """As the others: edges of tiles, activations, rotation and cache store."""
    test_plain_and_parts(tile)
    for limit, gelu in ((None, False), (1.5, False), (None, True)):
        test_gated(tile, limit, gelu)
    for shape in ((4, 2, 64, 16, True), (2, 2, 128, 5, True)):
        test_rotary(tile, *shape)
    test_rows_of_every_alignment(tile, 4)
    test_rotary_tokens_anywhere_in_their_pages(tile, 16, 5, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", tiles_with(4))
def test_steps_of_k_where_some_waves_only_load(tile):
    """From one step of K to beyond two rounds of the buffers, step by step: first, last and middle steps of what is asked for at once.
    Rows beyond the matrix and two tiles; the parts are told apart by numbers that grow with the column."""
    bm, bn, step = sizes_of(tile)
    m, n = bm + 5, bn + 16
    for steps in range(1, 2 * step // 64 + 4):
        k = 64 * steps
        x, w = rnd(m, k, seed=steps), rnd(n, k, seed=100 + steps) * (1 + torch.arange(k) // 64).to(torch.bfloat16)
        out = torch.full((m, n), 7.0, device=DEV)
        ops().gemm_tiles(out, x.to(DEV), w.to(DEV), tile=tile)
        close(out, product(x, w), k, False)
        if steps > 3 and 2 * -(-steps // 3) < steps:
            sums = torch.full((3, m, n), 7.0, device=DEV)
            ops().gemm_tiles(sums, x.to(DEV), w.to(DEV), tile=tile)
            close(sums.double().sum(0), product(x, w), k, False)


def test_plan_of_a_weight_in_the_cache():
    """What lies in the memory-side cache already goes rather to tiles whose multiplying waves load."""
    plan = ops().gemm_tiles_plan
    loading = [ops().GEMM_TILES[plan(512, 2048, 2048, 1, 256, near)[0]][-1] for near in (False, True)]
    assert loading == [4, 0]
