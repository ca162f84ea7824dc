"""Products with a matrix per group for up to 16 rows: their kernel against float64 and against the tiles that 17 rows take."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("groups,n,k,pad", [(1, 1, 8, 8), (3, 15, 248, 0), (2, 65, 256, 16), (5, 64, 264, 8), (4, 130, 520, 24)])
def test_few_rows_per_group(out_dtype, groups, n, k, pad):
    """n about a wave's 16 and a workgroup's 64 weight rows, k about the 256 columns asked for at once; rows beside each
    other in a wider tensor, results into one that has more columns."""
    from llmserve.ops import library as ops

    gen = torch.Generator().manual_seed(groups * n + k)
    x = torch.randn(17, groups, k + pad, generator=gen).to(torch.bfloat16).to(DEV)[:, :, :k]
    w = (torch.randn(groups, n, k, generator=gen) * 0.3).to(torch.bfloat16).to(DEV)
    z = torch.randn(17, 5 + groups * n, generator=gen).to(DEV)
    products = torch.einsum("mgk,gnk->mgn", x.double().cpu(), w.double().cpu())
    sizes = torch.einsum("mgk,gnk->mgn", x.double().abs().cpu(), w.double().abs().cpu())
    for gate_per_group in (None, False, True):
        if gate_per_group is None:
            kw, gates = {}, torch.ones(17, groups, n, dtype=torch.float64)
        else:
            kw = dict(epilogue="gated", gate_column=5, gate_per_group=gate_per_group)
            cols = z[:, 5:5 + groups].unsqueeze(2).expand(17, groups, n) if gate_per_group else z[:, 5:].view(17, groups, n)
            gates = torch.sigmoid(cols.double().cpu())
        for m in (1, 7, 16, 17):
            if kw:
                kw["gate"] = z[:m]
            out = torch.full((m, groups, n + 3), float("nan"), dtype=out_dtype, device=DEV)
            ops.grouped_product(out[:, :, :n], x[:m], w, **kw)
            got, ref = out[:, :, :n].double().cpu(), (products * gates)[:m]
            # k products that are exact in 32 bits, added in 32 bits in any order: k units of 2^-24 of the sum of their sizes; the gate a few
            # units of 2^-24 of the result (16 allowed); the result's own rounding is half a step, 2^-8 of it in bfloat16
            bound = (sizes * gates)[:m] * k * 2.0 ** -24 + ref.abs() * (16 * 2.0 ** -24 + (2.0 ** -8 if out_dtype == torch.bfloat16 else 0.0))
            assert ((got - ref).abs() <= bound).all(), (m, gate_per_group, float(((got - ref).abs() - bound).max()))
            assert torch.isnan(out[:, :, n:].float()).all()
