"""GPU parity of the matrix products of the linear layers (mlts_gemm) with fp32 / fp64 torch products: remainders of every tile
and slab, split contractions, strided operands, accumulation, and what is left to the library."""
import pytest
import torch

from maltos_amd import _lib
from maltos_amd._native import native

pytestmark = pytest.mark.gpu
NT, NN, TN = 0, 1, 2


def operands(form, M, N, K, dtype, dev, seed):
    gen = torch.Generator().manual_seed(seed)
    shape_a, shape_b = ((K, M) if form == TN else (M, K)), ((N, K) if form == NT else (K, N))
    return (torch.randn(*s, generator=gen).to(dtype).to(dev) for s in (shape_a, shape_b))


def expected(form, a, b):
    a, b = a.double(), b.double()
    return a @ b.t() if form == NT else a @ b if form == NN else a.t() @ b


@pytest.mark.parametrize("form", [NT, NN, TN])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (64, 64, 64), (72, 56, 40), (200, 136, 520), (1016, 512, 512), (136, 1000, 4104), (1024, 4096, 128),
                                   (4096, 4096, 136), (8, 2048, 1000), (264, 72, 9000)])
def test_product_forms(dev, dtype, form, M, N, K):
    a, b = operands(form, M, N, K, dtype, dev, M + N + K)
    want = expected(form, a, b)
    rel = 4e-3 if dtype == torch.bfloat16 else 2e-6
    got = native().product(form, a, b)
    assert (got.double() - want).norm() <= rel * want.norm()
    out = torch.randn(M, N, generator=torch.Generator().manual_seed(1)).to(dtype).to(dev)
    total = out.double() + want
    native().product(form, a, b, out, True)   # added in fp32, rounded once
    assert (out.double() - total).norm() <= rel * total.norm()
    assert torch.equal(native().product(form, a, b), got)   # the same every time


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_product_of_column_blocks(dev, dtype):
    """Operands that are column ranges of wider matrices, M odd in the forms where it is not a row length."""
    gen = torch.Generator().manual_seed(3)
    wide = torch.randn(333, 640, generator=gen).to(dtype).to(dev)
    w = torch.randn(96, 256, generator=gen).to(dtype).to(dev)
    rel = 4e-3 if dtype == torch.bfloat16 else 2e-6
    for form, a, b in ((NT, wide[:, 128:384], w), (NN, wide[:, 128:224], w), (TN, wide[:, 128:384], wide[:, 512:])):
        want = expected(form, a, b)
        assert (native().product(form, a, b).double() - want).norm() <= rel * want.norm()


def test_products_left_to_the_library(dev):
    """Unaligned rows, other dtypes and large products take the library's kernels: same answers."""
    gen = torch.Generator().manual_seed(4)
    for dtype, K in ((torch.bfloat16, 33), (torch.float16, 64), (torch.float32, 30)):
        a, b = torch.randn(50, K, generator=gen).to(dtype).to(dev), torch.randn(40, K, generator=gen).to(dtype).to(dev)
        want = expected(NT, a, b)
        assert (native().product(NT, a, b).double() - want).norm() <= 5e-3 * want.norm()
    assert _lib.lib().mlts_gemm_supports(NT, _lib.MLTS_BF16, 64, 64, 33, 33, 33, 64) is not None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,hidden,widths", [(8, 64, (64, 32, 32)), (333, 136, (96, 72, 40)), (1023, 512, (512, 256, 256)), (2048, 256, (688, 688)), (4104, 512, (1376, 1376))])
def test_group_of_projections(dev, dtype, rows, hidden, widths):
    """Projections that share their input, weights not adjacent: outputs, one input gradient over all of them, weight gradients."""
    gen = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, hidden, generator=gen).to(dtype).to(dev).requires_grad_(True)
    ws = [torch.randn(n, hidden, generator=gen).to(dtype).to(dev).requires_grad_(True) for n in widths]
    dys = [torch.randn(rows, n, generator=gen).to(dtype).to(dev) for n in widths]
    group = native().Adjacent(ws)
    assert not group.adjacent and group.runs_as_group(x, ws)
    ys = native().adjacent_linears(x, group, ws, False)
    grads = torch.autograd.grad(ys, (x, *ws), dys)
    rel = 4e-3 if dtype == torch.bfloat16 else 2e-6
    xd, wd, dd = x.detach().double(), [w.detach().double() for w in ws], [d.double() for d in dys]
    want = [xd @ w.t() for w in wd] + [sum(d @ w for d, w in zip(dd, wd))] + [d.t() @ xd for d in dd]
    for got, w in zip([*ys, *grads], want):
        assert (got.detach().double() - w).norm() <= rel * w.norm()
