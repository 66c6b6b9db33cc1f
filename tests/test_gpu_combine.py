"""DifferentialOperator.combine_dev: out = y + sum c_i k_i, one to nine vectors, odd lengths and unaligned vectors."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,shape,nk,shift", [("fp64", (1, 1, 1), 1, 0), ("fp64", (3, 5, 7), 3, 1), ("fp64", (4, 4, 4), 9, 0),
                                                 ("fp32", (3, 3, 3), 2, 0), ("fp32", (3, 5, 7), 4, 1), ("fp32", (4, 4, 4), 5, 0)])
def test_combine(prec, shape, nk, shift):
    import torch
    from bosss_amd.grid import CartesianGrid
    from bosss_amd.operator import DifferentialOperator
    print("case combine", prec, shape, nk, shift, flush=True)
    op = DifferentialOperator(CartesianGrid(shape, periodic=[True] * 3), "euler_lf", 2, precision=prec)
    dt, eps = (torch.float64, 2.3e-16) if prec == "fp64" else (torch.float32, 1.2e-7)
    gen = torch.Generator().manual_seed(3)
    new = lambda: (torch.rand(op.ndof + shift, generator=gen, dtype=torch.float64) * 2 - 1).to("cuda:0", dt)[shift:]
    y, ks, c = new(), [new() for _ in range(nk)], [0.3 * i - 0.7 for i in range(nk)]
    want, scale = y.double(), y.double().abs()
    for a, k in zip(c, ks):
        want, scale = want + float(torch.tensor(a, dtype=dt)) * k.double(), scale + abs(a) * k.double().abs()
    out = torch.full_like(y, float("nan"))
    op.combine_dev(y, c, ks, out)
    assert bool(((out.double() - want).abs() <= (nk + 1) * eps * scale).all())
    op.combine_dev(y, c, ks, y)             # in place
    assert torch.equal(y, out)
    with pytest.raises(ValueError):
        op.combine_dev(y, c, ks, ks[0])
    with pytest.raises(ValueError):
        op.combine_dev(y, c + [1.0], ks, out)
