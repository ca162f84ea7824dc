"""Products of few rows that close the sum that their rows are still open with, against 64 bits and beside the kernels that do it apart."""

import math

import pytest
import torch

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


def ops():
    from llmserve.ops import library

    return library


def rnd(*shape, seed, scale=1.0):
    return scale * torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


def close(got, want, bound):
    worst = float((got.double().cpu() - want).abs().max())
    assert worst <= bound, (worst, bound)


def rounded(rows):
    """(bfloat16 rows as 64-bit numbers, how far one that lies next to a rounding boundary may be off)"""
    return rows.to(torch.bfloat16).double(), 2.0 ** -8 * float(rows.abs().max())


# rows: one, a lane group's four, five and all eight; columns of one chunk's part, a chunk, wave counts' edges, three and four chunks a wave;
# weight rows below, at and beyond a share of 8 and 16 a workgroup
SIZES = [(1, 8, 5), (4, 136, 300), (5, 1024, 2048), (8, 1032, 4104), (3, 2048, 5000), (8, 2048, 1000), (2, 2056, 2050), (8, 3072, 700),
         (7, 4096, 513)]


@pytest.mark.parametrize("n,k,cols", SIZES)
@pytest.mark.parametrize("swiglu", [False, True])
def test_normed(n, k, cols, swiglu):
    cols += cols % 2 if swiglu else 0
    x, y, yw = rnd(n, k, seed=1), rnd(n, k, seed=2, scale=3.0), 1.0 + rnd(k, seed=3, scale=0.1)
    w, b = rnd(cols, k, seed=4, scale=k ** -0.5).to(torch.bfloat16), None if swiglu else rnd(cols, seed=5).to(torch.bfloat16)
    after = torch.empty(n, k, device=DEV)
    xd, h = x.to(DEV), torch.empty(n, k, dtype=torch.bfloat16, device=DEV)
    out = torch.full((n, cols // 2 if swiglu else cols), 7.0, dtype=torch.bfloat16 if swiglu else torch.float32, device=DEV)
    ops().gemm_decode_stream(out, xd, w.to(DEV), None if b is None else b.to(DEV), joins=(y.to(DEV), yw.to(DEV), 1e-5, after), h_out=h,
                             swiglu=swiglu, gelu=swiglu)
    assert torch.equal(xd.cpu(), x)
    want = x.double() + y.double() * torch.rsqrt((y.double() ** 2).mean(1, keepdim=True) + 1e-5) * yw.double()
    close(after, want, 4e-6 * float(want.abs().max()))
    assert torch.equal(h, after.to(torch.bfloat16))
    # the rows as the kernel rounded them: the product is theirs
    sums = h.double().cpu() @ w.double().t() + (0 if b is None else b.double())
    if swiglu:
        want = torch.nn.functional.gelu(sums[:, :cols // 2], approximate="tanh") * sums[:, cols // 2:]
        close(out, want, (2.0 ** -8 + 4e-6 * math.sqrt(k)) * float(want.abs().max()))
    else:
        close(out, sums, 4e-6 * math.sqrt(k) * float(sums.abs().max()))
        # beside the kernels apart: the stream's sums of squares are added in another order, so a row's element may round the other way
        rows = xd.clone()
        apart = ops().normed_add_norm(torch.empty(n, k, dtype=torch.bfloat16, device=DEV), rows, None, 0.0, y=y.to(DEV), y_weight=yw.to(DEV),
                                      y_eps=1e-5)
        close(after, rows.double().cpu(), 4e-6 * float(rows.abs().max()))
        close(h, apart.double().cpu(), rounded(after.cpu())[1])


@pytest.mark.parametrize("n,k,inter", [(1, 8, 5), (5, 1024, 2049), (8, 2304, 1000), (3, 3072, 5000), (8, 4096, 513)])
@pytest.mark.parametrize("unit", ["silu", "clamped"])
def test_gated_units(n, k, inter, unit):
    x, y, yw = rnd(n, k, seed=1), rnd(n, k, seed=2, scale=3.0), 1.0 + rnd(k, seed=3, scale=0.1)
    w = rnd(2 * inter, k, seed=4, scale=k ** -0.5).to(torch.bfloat16)
    h, after = torch.empty(n, k, dtype=torch.bfloat16, device=DEV), torch.empty(n, k, device=DEV)
    out = torch.full((n, inter), 7.0, dtype=torch.bfloat16, device=DEV)
    ops().gemm_decode_stream(out, x.to(DEV), w.to(DEV), joins=(y.to(DEV), yw.to(DEV), 1e-5, after), h_out=h, swiglu=True,
                             limit=1.5 if unit == "clamped" else None)
    sums = h.double().cpu() @ w.double().t()
    gate, up = sums[:, :inter], sums[:, inter:]
    off = 4e-6 * math.sqrt(k) * float(sums.abs().max())  # of the sums
    if unit == "clamped":  # in 32-bit, rounded once (half a step of 8 bits); slopes of the unit up to 1.1 and of its factor up to 1
        g, v = gate.clamp(max=1.5), up.clamp(-1.5, 1.5) + 1.0
        want = g * torch.sigmoid(1.702 * g) * v
        bound = 2.0 ** -8 * want.abs() + off * (1.1 * v.abs() + 1.5)
    else:  # gate, up and silu(gate) are rounded, and then the result: half a step each (2^-8 of a number just beyond a power of two)
        want = gate * torch.sigmoid(gate) * up
        bound = 2.0 ** -8 * (1.1 * gate.abs() * up.abs() + 3.0 * want.abs()) * 1.02 + off * (1.1 * up.abs() + gate.abs())
    wrong = (out.double().cpu() - want).abs() > bound
    assert not wrong.any(), (int(wrong.sum()), float((out.double().cpu() - want).abs().max()))
    # beside the product of the same rows: the same sums, the same unit
    assert torch.equal(out, ops().gemm_decode(torch.empty_like(out), h, w.to(DEV), swiglu=True, limit=1.5 if unit == "clamped" else None))


@pytest.mark.parametrize("n,k,cols", SIZES)
@pytest.mark.parametrize("keep", [False, True])
def test_norm(n, k, cols, keep):
    x, norm = rnd(n, k, seed=1, scale=2.0), rnd(k, seed=7, scale=0.1)
    w = rnd(cols, k, seed=8, scale=k ** -0.5).to(torch.bfloat16)
    out = torch.full((n, cols), 7.0, device=DEV)
    h = torch.empty(n, k, dtype=torch.bfloat16, device=DEV)
    ops().gemm_decode_stream(out, x.to(DEV), w.to(DEV), norm=(norm.to(DEV), 1e-6, 1.0), h_out=h if keep else None)
    rows = x.double() * torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-6) * (1.0 + norm.double())
    if keep:
        close(h, rows, rounded(rows)[1])
        close(out, h.double().cpu() @ w.double().t(), 4e-6 * math.sqrt(k) * float(out.abs().max()))
    else:  # every element of a row rounded to 8 bits, half a step at most each, against a row of w: six standard deviations of their sum at most
        close(out, rows @ w.double().t(), 2.0 ** -8 / 3 ** 0.5 * 6.0 * float((rows.abs().amax(1)[:, None] * w.double().norm(dim=1)).max()))


# rows in LDS and in registers (9 to 16 rows of a long K), shares of 8 and 16 weight rows and their edges
@pytest.mark.parametrize("n,k,cols", [(1, 64, 7), (8, 2048, 2048), (5, 5632, 2049), (16, 2048, 4100), (9, 5632, 2048), (16, 6144, 300), (13, 4608, 5000)])
@pytest.mark.parametrize("gate", ["bias", "plain", None])
def test_adds_to_a_stream(n, k, cols, gate):
    x, w = rnd(n, k, seed=1).to(torch.bfloat16), rnd(cols, k, seed=2, scale=k ** -0.5).to(torch.bfloat16)
    stream, z, b = rnd(n, cols + 3, seed=3), rnd(n, cols + 9, seed=4, scale=3.0), rnd(cols, seed=5)
    sd = stream.to(DEV)
    given = None if gate is None else (z.to(DEV), 6, b.to(DEV) if gate == "bias" else None)
    assert ops().gemm_decode(None, x.to(DEV), w.to(DEV), residual=sd[:, :cols], gate=given).data_ptr() == sd.data_ptr()
    g = 1.0 if gate is None else torch.sigmoid(z[:, 6:6 + cols].double() + (b.double() if gate == "bias" else 0.0))
    sums = x.double() @ w.double().t()
    want = stream[:, :cols].double() + g * sums
    close(sd[:, :cols], want, 2e-6 * math.sqrt(k) * float(sums.abs().max()) + 2.0 ** -23 * float(want.abs().max()))
    assert torch.equal(sd[:, cols:].cpu(), stream[:, cols:])


# K of one chunk beyond what a compute unit holds, of a part of a chunk, of whole rounds of items; shares of one row, 8, 16, a row more, two tiles
@pytest.mark.parametrize("n,k,cols", [(1, 6152, 256), (8, 6272, 2048), (9, 7168, 2049), (16, 8192, 4096), (5, 8200, 4097), (16, 12296, 500),
                                      (3, 11008, 8192)])
def test_adds_long_rows(n, k, cols):
    x, w = rnd(n, k, seed=1).to(torch.bfloat16), rnd(cols, k, seed=2, scale=k ** -0.5).to(torch.bfloat16)
    rows = rnd(n, cols + 8, seed=3).to(torch.bfloat16)
    rd = rows.to(DEV)
    ops().gemm_decode(None, x.to(DEV), w.to(DEV), residual=rd[:, :cols])
    sums = (x.double() @ w.double().t())
    want = rows[:, :cols].double() + sums
    # the sum is rounded, and then the row (8 bits: half a step is 2^-8 of a number just beyond a power of two), and the sums' own error
    close(rd[:, :cols], want, 2.0 ** -8 * float(sums.abs().max()) + 2.0 ** -8 * float(want.abs().max()) + 2e-6 * math.sqrt(k) * float(sums.abs().max()))
    assert torch.equal(rd[:, cols:].cpu(), rows[:, cols:])


def test_refused():
    x, y, w = torch.zeros(8, 64, device=DEV), torch.zeros(8, 64, device=DEV), torch.zeros(64, 64, dtype=torch.bfloat16, device=DEV)
    weight, out = torch.ones(64, device=DEV), torch.zeros(8, 64, device=DEV)
    take = ops().gemm_decode_stream
    with pytest.raises(ValueError, match="x_out"):
        take(out, x, w, joins=(y, weight, 1e-5, x))
    with pytest.raises(ValueError, match="up to 8 rows"):
        nine = torch.zeros(9, 64, device=DEV)
        take(torch.zeros(9, 64, device=DEV), nine, w, norm=(weight, 1e-5, 0.0))
    with pytest.raises(ValueError, match="either"):
        take(out, x, w)
    with pytest.raises(ValueError, match="gated epilogue"):
        take(out.to(torch.bfloat16), x, w, norm=(weight, 1e-5, 0.0), swiglu=True)
    with pytest.raises(ValueError, match="float32 residual"):
        rows = torch.zeros(8, 64, dtype=torch.bfloat16, device=DEV)
        ops().gemm_decode(None, rows, w, residual=rows.clone(), gate=(out, 0, None))
    with pytest.raises(ValueError, match="residual must be"):
        rows = torch.zeros(17, 64, dtype=torch.bfloat16, device=DEV)
        ops().gemm_decode(None, rows, w, residual=torch.zeros(17, 64, device=DEV))
