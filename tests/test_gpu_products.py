"""GPU parity of the matrix products of the linear layers (mlts_gemm) with fp32 / fp64 torch products: remainders of every tile
and slab, split contractions, strided operands, accumulation, and what is left to the library."""
import ctypes

import pytest
import torch

from maltos_amd import _lib, ops  # (ops: the schemas of the operators)
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


@pytest.mark.parametrize("form,M,N,K,own", [
    (NT, 6000, 1024, 1024, False), (NT, 12000, 1024, 1024, False), (NN, 12000, 1024, 1024, False), (NT, 4096, 1280, 1280, False), (NT, 6000, 1000, 1024, True),
    (NT, 16384, 2304, 768, True), (NT, 17000, 2304, 768, False), (NN, 16384, 512, 1536, True), (NT, 17000, 512, 1536, False), (NT, 8000, 512, 2048, True), (NT, 8192, 512, 2048, False),
    (TN, 1024, 1024, 12000, True), (TN, 1024, 1024, 16384, False), (TN, 1024, 1024, 20001, True), (TN, 512, 1376, 16384, False), (TN, 256, 680, 32768, True), (TN, 2752, 512, 12000, True),
    (TN, 5456, 1024, 4096, False), (TN, 1024, 2728, 10000, True), (TN, 6912, 1280, 3000, False),
    (TN, 8192, 768, 12000, True), (TN, 8192, 776, 12000, False), (TN, 8192, 1024, 10000, True), (TN, 8192, 1024, 9992, False), (TN, 12000, 1024, 12000, False), (TN, 32000, 128, 4096, True),
    (TN, 32000, 136, 4096, False), (TN, 32000, 512, 10000, True), (TN, 32000, 512, 9992, False),
    (TN, 16384, 256, 1023, True), (TN, 20480, 256, 2048, True), (TN, 20480, 256, 2040, False), (TN, 24576, 256, 2048, False), (TN, 32768, 128, 1023, True), (TN, 32776, 128, 1023, False),
    (TN, 33024, 256, 12000, False), (TN, 32768, 256, 12000, True), (TN, 49152, 256, 12000, False), (TN, 49160, 256, 12000, True),
    (NN, 2048, 2048, 2816, True), (NN, 2048, 2176, 2816, False), (NN, 4096, 1024, 2808, False), (NN, 1000, 4096, 8192, True), (NN, 4096, 2048, 8192, True), (NN, 4352, 2048, 8192, False),
    (NN, 4096, 2048, 8184, False)])
def test_which_large_products_the_own_kernels_take(dev, form, M, N, K, own):
    """Both sides of each line between them and the library."""
    a, b = (torch.zeros(s, dtype=torch.bfloat16, device=dev) for s in ((K, M) if form == TN else (M, K), (N, K) if form == NT else (K, N)))
    _lib.kernel_timing(True)
    try:
        native().product(form, a, b)
        torch.cuda.synchronize()
        assert _lib.kernel_time_ms("gemm")[1] == int(own)
    finally:
        _lib.kernel_timing(False)


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


class GemmProduct(ctypes.Structure):
    """Mirror of `mlts_gemm_product`."""
    _fields_ = [("form", ctypes.c_int32), ("segments", ctypes.c_int32), ("accumulate", ctypes.c_int32), ("M", ctypes.c_int64), ("N", ctypes.c_int64),
                ("k", ctypes.c_int64 * 3), ("a", ctypes.c_void_p * 3), ("b", ctypes.c_void_p * 3), ("lda", ctypes.c_int64 * 3),
                ("ldb", ctypes.c_int64 * 3), ("c", ctypes.c_void_p), ("ldc", ctypes.c_int64)]


class GemmTiles(ctypes.Structure):
    """Mirror of `mlts_gemm_tiles`."""
    _fields_ = [("tile_m", ctypes.c_int32), ("tile_n", ctypes.c_int32), ("slices", ctypes.c_int32), ("together", ctypes.c_int32), ("busiest", ctypes.c_int32)]


def run_products(products, dtype):
    """mlts_gemm_multi of (form, [(a, b), ...], c, accumulate)."""
    ps = (GemmProduct * len(products))()
    for p, (form, segments, c, accumulate) in zip(ps, products):
        p.form, p.segments, p.accumulate, (p.M, p.N), p.c, p.ldc = form, len(segments), accumulate, c.shape, c.data_ptr(), c.stride(0)
        for i, (a, b) in enumerate(segments):
            p.k[i] = a.size(0) if form == TN else a.size(1)
            p.a[i], p.b[i], p.lda[i], p.ldb[i] = a.data_ptr(), b.data_ptr(), a.stride(0), b.stride(0)
    code, L = {torch.bfloat16: _lib.MLTS_BF16, torch.float32: _lib.MLTS_F32}[dtype], _lib.lib()
    ws = torch.empty(max(16, L.mlts_gemm_multi_workspace_bytes(ps, len(ps), code)), dtype=torch.uint8, device=products[0][2].device)
    _lib.check(L.mlts_gemm_multi(ps, len(ps), code, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("plan", ["s", "ss", "sss", "nsts", "0s", "s0n", "tn"])
def test_products_with_segments_in_one_call(dev, dtype, plan):
    """s: a sum over three segments, alone and beside others; 0: one without rows; n, t: plain NN and TN products."""
    gen = torch.Generator().manual_seed(len(plan))
    rnd = lambda *shape: torch.randn(*shape, generator=gen).to(dtype).to(dev)
    products, want = [], []
    for i, kind in enumerate(plan):
        M, N = 0 if kind == "0" else 72 + 32 * i, 64 + 8 * i
        ks = {"s": (64, 136, 32), "0": (64, 32), "n": (200,), "t": (72,)}[kind]
        form = TN if kind == "t" else NN
        segments = [(rnd(k, M) if form == TN else rnd(M, k), rnd(k, N)) for k in ks]
        c, accumulate = rnd(M, N), i % 2
        want.append(sum((expected(form, a, b) for a, b in segments), c.double() * accumulate))
        products.append((form, segments, c, accumulate))
    run_products(products, dtype)
    rel = 4e-3 if dtype == torch.bfloat16 else 2e-6
    for (_, _, c, _), w in zip(products, want):
        assert (c.double() - w).norm() <= (2 if dtype == torch.bfloat16 else 1) * rel * w.norm()   # bf16: each segment is rounded


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form,M,N,K", [(NT, 72, 64, 136), (NN, 64, 200, 40), (TN, 512, 512, 4096), (NN, 8, 2048, 1000), (NT, 1, 64, 64)])
def test_product_into_rows_of_a_wider_buffer(dev, dtype, form, M, N, K):
    """Outputs that are column ranges, also of products whose contraction is split where the output is dense; the columns beside them
    are not touched.  An output of another shape is refused, on the host."""
    a, b = operands(form, M, N, K, dtype, dev, K)
    want, rel = expected(form, a, b), 4e-3 if dtype == torch.bfloat16 else 2e-6
    for accumulate in (False, True):
        wide = torch.randn(M, N + 96, generator=torch.Generator().manual_seed(1)).to(dtype).to(dev)
        before = wide.clone()
        total = want + before[:, 32:32 + N].double() * accumulate
        native().product(form, a, b, wide[:, 32:32 + N], accumulate)
        assert (wide[:, 32:32 + N].double() - total).norm() <= rel * total.norm()
        assert torch.equal(wide[:, :32], before[:, :32]) and torch.equal(wide[:, 32 + N:], before[:, 32 + N:])
    for shape in ((M, N + 8), (M + 1, N), (N * M,)):
        with pytest.raises(ValueError, match="cannot be written"):
            native().product(form, a, b, torch.zeros(shape, dtype=dtype, device=dev))


@pytest.mark.parametrize("form", [NT, NN, TN])
@pytest.mark.parametrize("longer", [0, 1])
def test_operands_that_do_not_match_are_refused(dev, form, longer):
    """Contractions of different lengths (rows of a wider weight would be in bounds, and a wrong product)."""
    a, _ = operands(form, 64, 64, 128 if longer == 0 else 64, torch.bfloat16, dev, 1)
    _, b = operands(form, 64, 64, 128 if longer == 1 else 64, torch.bfloat16, dev, 2)
    with pytest.raises(RuntimeError):
        native().product(form, a, b)
    if form == NT:
        with pytest.raises(RuntimeError):
            native().linear(a, b, False)


@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("dtype,M,N,K", [(torch.bfloat16, 1, 8, 8), (torch.bfloat16, 65, 72, 136), (torch.bfloat16, 1016, 1376, 512),
                                         (torch.bfloat16, 1100, 2056, 72), (torch.bfloat16, 4001, 1032, 64), (torch.float32, 700, 1028, 68),
                                         (torch.float32, 2048, 1376, 40)])
def test_gate_up_in_one_launch(dev, dtype, M, N, K, keep):
    """Tiles of 64 and 128 rows, in fp32 also of 256, with remainders of rows, columns (of each of the two products) and slabs, operands with row
    strides, gate and up wanted or not: the bits of the product with both weights and the pass over it."""
    gen = torch.Generator().manual_seed(M + N)
    rows = lambda n: torch.randn(n, K + 24, generator=gen).to(dtype).to(dev)[:, 16:16 + K]
    x, wg, wu = rows(M), rows(N), rows(N)
    gu, h = torch.full((M, 2 * N + 8), 7.0, dtype=dtype, device=dev), torch.full((M, N + 4), 7.0, dtype=dtype, device=dev)
    es, st = x.element_size(), torch.cuda.current_stream().cuda_stream
    up = gu.data_ptr() + (N + 8) * es
    both = native().product(NT, x, torch.cat([wg, wu]))
    want = native().swiglu_rows(both, 0, N, N)
    L = _lib.lib()
    _lib.check(L.mlts_gemm_swiglu(1 if dtype == torch.bfloat16 else 0, M, N, K, x.data_ptr(), x.stride(0), wg.data_ptr(), wu.data_ptr(), wg.stride(0),
                                  gu.data_ptr() if keep else None, up if keep else None, gu.stride(0), h.data_ptr(), h.stride(0), st))
    assert torch.equal(h[:, :N], want) and (h[:, N:] == 7).all() and (gu[:, N:N + 8] == 7).all()
    if keep:
        assert torch.equal(gu[:, :N], both[:, :N]) and torch.equal(gu[:, N + 8:], both[:, N:])
    else:
        assert (gu == 7).all()


class GemmRotation(ctypes.Structure):
    """Mirror of `mlts_gemm_rotation`."""
    _fields_ = [("cos", ctypes.c_void_p), ("sin", ctypes.c_void_p), ("positions", ctypes.c_void_p), ("max_pos", ctypes.c_int32),
                ("position_offset", ctypes.c_int32), ("seq", ctypes.c_int32), ("head_dim", ctypes.c_int32), ("columns", (ctypes.c_int64 * 4) * 4)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,S,H,Hkv,D,K,joint,given", [(1, 1, 1, 1, 64, 8, False, False), (3, 77, 4, 2, 64, 136, False, True), (2, 65, 3, 1, 128, 72, True, False),
                                                       (2, 333, 2, 2, 96, 264, True, True), (3, 701, 8, 8, 64, 64, False, True),
                                                       (3, 777, 16, 4, 128, 40, False, False), (2, 3001, 16, 8, 96, 64, False, True)])
def test_rotation_in_the_products(dev, dtype, B, S, H, Hkv, D, K, joint, given):
    """q, k, v as one product or as three: remainders of rows and slabs, positions of packed rows, or an offset; the
    bits of the products and the rotation one after the other."""
    gen = torch.Generator().manual_seed(B * S + D)
    rnd = lambda *s: torch.randn(*s, generator=gen).to(dtype).to(dev)
    widths, max_pos, offset = [H * D, Hkv * D, Hkv * D], S + 9, 0 if given else 5
    x, w, y = rnd(B * S, K), rnd(sum(widths), K), torch.empty(B * S, sum(widths), dtype=dtype, device=dev)
    angles = torch.rand(max_pos, D // 2, generator=gen) * 6.3
    cos, sin = angles.cos().to(dtype).to(dev), angles.sin().to(dtype).to(dev)
    positions = torch.randint(0, max_pos, (B, S), generator=gen, dtype=torch.int32).to(dev) if given else None
    ws, ys = w.split(widths), y.split(widths, 1)
    parts = list(zip(ws, ys)) if joint else [(w, y)]
    plain = [torch.empty_like(c) for _, c in parts]
    run_products([(NT, [(x, b)], c, 0) for (b, _), c in zip(parts, plain)], dtype)
    r = GemmRotation(cos.data_ptr(), sin.data_ptr(), positions.data_ptr() if given else None, max_pos, offset, S, D)
    if joint:
        r.columns[0][1], r.columns[1][1] = widths[0], widths[1]
    else:
        r.columns[0][:] = [0, widths[0], widths[0], widths[0] + widths[1]]
    ps = (GemmProduct * len(parts))()
    for p, (b, c) in zip(ps, parts):
        p.form, p.segments, (p.M, p.N), p.c, p.ldc = NT, 1, c.shape, c.data_ptr(), c.stride(0)
        p.k[0], p.a[0], p.b[0], p.lda[0], p.ldb[0] = K, x.data_ptr(), b.data_ptr(), x.stride(0), b.stride(0)
    code = {torch.bfloat16: _lib.MLTS_BF16, torch.float32: _lib.MLTS_F32}[dtype]
    _lib.check(_lib.lib().mlts_gemm_rope(ps, len(ps), code, ctypes.byref(r), torch.cuda.current_stream().cuda_stream))
    q, k, v = torch.cat(plain, 1).split(widths, 1)
    heads = lambda t: t.unflatten(0, (B, S)).unflatten(2, (-1, D)).transpose(1, 2)
    q, k = native().rope_pair(heads(q), heads(k), cos, sin, positions, offset)
    rows = lambda t: t.transpose(1, 2).flatten(2).flatten(0, 1)
    for got, want in zip(ys, (rows(q), rows(k), v)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("accumulate", [0, 1, None], ids=["written", "added", "frozen"])
@pytest.mark.parametrize("dtype,M,N,K", [(torch.bfloat16, 8, 8, 8), (torch.bfloat16, 136, 72, 200), (torch.bfloat16, 1016, 1376, 512),
                                         (torch.float32, 100, 36, 72), (torch.float32, 2048, 688, 256), (torch.float32, 1000, 1376, 512)])
def test_activation_gradients_in_the_products(dev, dtype, M, N, K, accumulate):
    """dW and dh = dy W in one launch with dh going through the activation: remainders of tiles, split dW, added onto, written or not
    wanted; the bits of the products and the pass over gate and up."""
    gen = torch.Generator().manual_seed(M + N)
    rnd = lambda *s: torch.randn(*s, generator=gen).to(dtype).to(dev)
    dy, w, h, gu, dw = rnd(M, K), rnd(K, N), rnd(M, N), rnd(M, 2 * N), rnd(K, N)
    want_dw, dh = dw.clone(), torch.empty(M, N, dtype=dtype, device=dev)
    both = [] if accumulate is None else [(TN, [(dy, h)], want_dw, accumulate)]
    run_products(both + [(NN, [(dy, w)], dh, 0)], dtype)
    want = native().swiglu_rows_backward(dh, gu, 0, N, N)
    code, es, L, need = {torch.bfloat16: _lib.MLTS_BF16, torch.float32: _lib.MLTS_F32}[dtype], gu.element_size(), _lib.lib(), ctypes.c_int64()
    assert L.mlts_gemm_swiglu_bwd_supports(code, len(both), M, N, K, K, N, N, 2 * N, 2 * N, ctypes.byref(need)) is None
    ws, dgu = torch.empty(max(16, need.value), dtype=torch.uint8, device=dev), torch.full_like(gu, 7.0)
    _lib.check(L.mlts_gemm_swiglu_bwd(code, M, N, K, dy.data_ptr(), K, w.data_ptr(), N, h.data_ptr(), N, dw.data_ptr() if both else None, accumulate or 0, gu.data_ptr(),
                                      gu.data_ptr() + N * es, 2 * N, dgu.data_ptr(), dgu.data_ptr() + N * es, 2 * N, ws.data_ptr(), need.value,
                                      torch.cuda.current_stream().cuda_stream))
    assert torch.equal(dw, want_dw) and torch.equal(dgu, want)


@pytest.mark.parametrize("check,args", [
    (test_product_forms, (NT, 2331, 1544, 512)), (test_product_forms, (NT, 3001, 1003, 264)), (test_product_forms, (NT, 129, 8200, 264)), (test_product_forms, (NN, 2331, 1384, 520)),
    (test_product_forms, (NT, 4033, 504, 1384)), (test_product_forms, (NN, 4100, 520, 1528)), (test_product_forms, (NN, 16001, 1032, 72)), (test_product_forms, (TN, 520, 1384, 6008)),
    (test_product_forms, (TN, 1544, 520, 4001)), (test_product_forms, (TN, 264, 264, 12001)), (test_group_of_projections, (6001, 512, (512, 256, 256))),
    (test_product_into_rows_of_a_wider_buffer, (NN, 2331, 1376, 512)), (test_product_into_rows_of_a_wider_buffer, (TN, 520, 1384, 3008)),
    (test_gate_up_in_one_launch, (2331, 1376, 512, True)), (test_gate_up_in_one_launch, (4097, 1384, 264, False)),
    (test_rotation_in_the_products, (3, 1411, 8, 8, 64, 512, True, True)), (test_rotation_in_the_products, (40, 111, 8, 4, 64, 512, True, False)),
    (test_rotation_in_the_products, (5, 1601, 8, 4, 64, 520, False, True)), (test_activation_gradients_in_the_products, (4097, 1376, 512, 1)),
    (test_activation_gradients_in_the_products, (8200, 1384, 520, None))], ids=lambda v: v.__name__[5:] if callable(v) else "-".join(map(str, v)))
def test_larger_bf16_tiles(dev, check, args):
    """The tiles of 128 rows (and of 64 where a size is planned on those: narrow contractions of 4001 and 12001 rows), alone, with others in a launch and
    with what follows the products in them: remainders of rows, columns and slabs,
    rectangles of tiles that eight does not divide, columns that are not whole groups of four, split contractions, sequences shorter than
    a tile."""
    first = dict(form=args[0], M=args[1], N=args[2], K=args[3]) if check in (test_product_forms, test_product_into_rows_of_a_wider_buffer) else None
    names = {test_group_of_projections: ("rows", "hidden", "widths"), test_gate_up_in_one_launch: ("M", "N", "K", "keep"),
             test_rotation_in_the_products: ("B", "S", "H", "Hkv", "D", "K", "joint", "given"), test_activation_gradients_in_the_products: ("M", "N", "K", "accumulate")}
    check(dev=dev, dtype=torch.bfloat16, **(first or dict(zip(names[check], args))))


def plan_of(items, dtype, sharing):
    """`mlts_gemm_plan` of (form, M, N, K[, row stride of C]); nothing is launched."""
    ps, tiles = (GemmProduct * len(items))(), (GemmTiles * len(items))()
    for p, (form, M, N, K, *ldc) in zip(ps, items):
        p.form, p.segments, p.M, p.N, p.k[0], p.ldc = form, 1, M, N, K, ldc[0] if ldc else N
        p.lda[0], p.ldb[0] = (M if form == TN else K), (K if form == NT else N)
    _lib.check(_lib.lib().mlts_gemm_plan(ps, len(ps), dtype, sharing, tiles))
    return tiles


def planned(items, dtype=_lib.MLTS_BF16, sharing=0):
    """The tile (rows, columns) and the slices that a call takes for each."""
    return [(t.tile_m, t.tile_n, t.slices) for t in plan_of(items, dtype, sharing)]


def tiles_of_an_xcd(items, dtype, sharing=0):
    """What the busiest of the eight gets of a launch, and what equal shares would give it."""
    tiles, bk, shares = plan_of(items, dtype, sharing), 64 if dtype == _lib.MLTS_BF16 else 32, []
    for (_, M, N, K), t in zip(items, tiles):
        slabs = -(-K // bk)
        slices = -(-slabs // -(-slabs // t.slices))
        shares.append(-(-(-(-M // t.tile_m) * -(-N // t.tile_n) * slices) // 8))
    return (tiles[0].busiest, sum(shares)) if tiles[0].together else (max(t.busiest for t in tiles), max(shares))


# products and launches of dW and dx whose rectangles would give an XCD's 32 CUs 33 to 36 tiles, or 98 to 132 for 93 to 128: remainders of rows, columns and slices
RUNS = [(_lib.MLTS_BF16, [(NN, 5352, 768, 768)]), (_lib.MLTS_BF16, [(NN, 2678, 384, 1488)]), (_lib.MLTS_BF16, [(NT, 1099, 848, 320)]), (_lib.MLTS_BF16, [(NT, 817, 2320, 640)]),
        (_lib.MLTS_F32, [(NN, 1206, 640, 640)]), (_lib.MLTS_F32, [(TN, 2688, 384, 1159)]), (_lib.MLTS_F32, [(NN, 774, 320, 848)]), (_lib.MLTS_BF16, [(TN, 3408, 640, 1407), (NN, 1407, 640, 3408)]),
        (_lib.MLTS_BF16, [(TN, 1152, 384, 1521), (NN, 1521, 384, 1152)]), (_lib.MLTS_F32, [(TN, 1704, 640, 1497), (NN, 1497, 640, 1704)]), (_lib.MLTS_F32, [(TN, 384, 384, 2191), (NN, 2191, 384, 384)])]


@pytest.mark.parametrize("dtype,items", RUNS, ids=lambda v: {_lib.MLTS_BF16: "bf16", _lib.MLTS_F32: "fp32"}[v] if isinstance(v, int) else "-".join("x".join(map(str, i[1:])) for i in v))
def test_tiles_in_runs_of_equal_length(dev, dtype, items):
    busiest, share = tiles_of_an_xcd(items, dtype)
    assert busiest == share
    t = torch.bfloat16 if dtype == _lib.MLTS_BF16 else torch.float32
    products, want = [], []
    for form, M, N, K in items:
        a, b = operands(form, M, N, K, t, dev, M)
        c = torch.randn(M, N, generator=torch.Generator().manual_seed(2)).to(t).to(dev)
        want.append(expected(form, a, b) + c.double())
        products.append((form, [(a, b)], c, 1))
    run_products(products, t)
    for (*_, c, _), w in zip(products, want):
        assert (c.double() - w).norm() <= (4e-3 if t == torch.bfloat16 else 2e-6) * w.norm()


# (form, M, N, K), the gap behind the rows of C, and the bf16 tile and slices that it is planned with: ragged rows, columns and slabs of each
TILE_CASES = [
    ((NN, 521, 2056, 8200), 0, (256, 128, 4)), ((NN, 1033, 5464, 520), 0, (256, 128, 1)), ((TN, 12008, 72, 8201), 0, (256, 128, 4)), ((TN, 136, 5464, 12001), 0, (256, 256, 8)),
    ((TN, 4088, 2040, 3001), 48, (256, 128, 1)), ((NT, 12001, 76, 8200), 0, (256, 128, 4)), ((NT, 4547, 7657, 680), 0, (256, 256, 1)), ((NN, 4547, 7656, 680), 8, (256, 256, 1)),
    ((TN, 4552, 7656, 681), 0, (256, 256, 1)), ((TN, 8200, 8200, 65), 0, (256, 256, 1)), ((TN, 8200, 8200, 97), 8, (256, 256, 1)), ((TN, 8200, 8200, 161), 0, (256, 256, 1)), ((NN, 2336, 1032, 8200), 0, (256, 256, 4)), ((NT, 4033, 516, 8200), 0, (256, 256, 4)), ((NT, 1033, 1029, 1032), 3, (128, 64, 1)),
    ((NT, 3001, 260, 8200), 0, (128, 64, 2)), ((NN, 521, 520, 4104), 0, (128, 64, 4)), ((TN, 2336, 136, 8201), 0, (128, 64, 4)), ((TN, 1032, 136, 8201), 0, (128, 64, 8)),
    ((NT, 2331, 1542, 512), 0, (128, 128, 1)), ((NN, 3001, 72, 6008), 0, (128, 128, 8)), ((TN, 520, 1384, 6008), 0, (128, 128, 4))]
# (batch rows, tokens, heads, KV heads, head_dim, K, positions given) of q, k, v as one rotated product
ROTATED_TILE_CASES = [((1, 863, 16, 4, 64, 1032, False), (128, 64, 1)), ((1, 5297, 12, 4, 64, 3000, False), (256, 128, 1)), ((7, 757, 24, 8, 64, 1032, True), (256, 256, 1)),
                      ((5, 1601, 8, 4, 64, 520, True), (128, 128, 1))]


@pytest.mark.parametrize("product,gap,tile", TILE_CASES, ids=lambda v: "-".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_every_bf16_tile(dev, product, gap, tile):
    """Each tile, whole and split, written and added onto, into dense rows and into rows of a wider buffer whose rest is not touched."""
    form, M, N, K = product
    assert planned([(*product, N + gap)]) == [tile]
    a, b = operands(form, M, N, K, torch.bfloat16, dev, M + N)
    want = expected(form, a, b)
    for accumulate in (0, 1):
        wide = torch.randn(M, N + gap, generator=torch.Generator().manual_seed(1)).bfloat16().to(dev)
        before = wide.clone()
        run_products([(form, [(a, b)], wide[:, :N], accumulate)], torch.bfloat16)
        total = want + before[:, :N].double() * accumulate
        assert (wide[:, :N].double() - total).norm() <= 4e-3 * total.norm() and torch.equal(wide[:, N:], before[:, N:])
        first = wide.clone()
        wide.copy_(before)
        run_products([(form, [(a, b)], wide[:, :N], accumulate)], torch.bfloat16)
        assert torch.equal(wide, first)


@pytest.mark.parametrize("case,tile", ROTATED_TILE_CASES, ids=lambda v: "-".join(map(str, v)))
def test_every_bf16_tile_rotated(dev, case, tile):
    B, S, H, Hkv, D, K, given = case
    assert planned([(NT, B * S, (H + 2 * Hkv) * D, K)], sharing=1) == [tile]
    test_rotation_in_the_products(dev, torch.bfloat16, B, S, H, Hkv, D, K, False, given)


# fp32 products and the tile and slices that each is planned with: ragged rows, columns and slabs of the tiles of elements in three parts
PARTS_CASES = [((NT, 901, 2052, 396), (64, 64, 1)), ((NN, 777, 1324, 516), (64, 64, 1)), ((TN, 1324, 252, 2047), (64, 64, 2)), ((NT, 2111, 2652, 332), (128, 64, 1)),
               ((NT, 2047, 4100, 260), (128, 128, 1)), ((NN, 2041, 260, 8196), (128, 128, 4)), ((TN, 8196, 260, 1999), (128, 128, 1))]


@pytest.mark.parametrize("product,tile", PARTS_CASES, ids=lambda v: "-".join(map(str, v)))
def test_fp32_in_three_parts(dev, product, tile):
    """Errors of one rounding in sixteen terms (a random walk of 2^-24 steps) and of the parts that are left out, which fp32 matrix instructions exceed; and operands that have
    no parts: infinities, NaN and numbers that bf16 rounds to infinity give what fp32 gives, in their rows and columns alone."""
    form, M, N, K = product
    assert planned([product], _lib.MLTS_F32) == [tile]
    a, b = operands(form, M, N, K, torch.float32, dev, M + N)
    want = expected(form, a, b)
    out = torch.empty(M, N, device=dev)
    run_products([(form, [(a, b)], out, 0)], torch.float32)
    assert (out.double() - want).norm() <= 2.0**-24 * (3 + (K / 16) ** 0.5) * want.norm()
    run_products([(form, [(a, b)], out, 1)], torch.float32)
    assert (out.double() - 2 * want).norm() <= 2.0**-23 * (4 + (K / 16) ** 0.5) * want.norm()
    rows, columns = a.t() if form == TN else a, b.t() if form == NT else b   # [M, K], [K, N]
    rows[3, 5], rows[M - 1, K - 1], rows[70, 0] = float("inf"), float("nan"), 3.4e38
    columns[:, 7] *= 1e-3
    columns[2, N - 1], columns[0, N - 1] = float("-inf"), 0.5   # (row 70 stays in range there, on its way to -inf)
    run_products([(form, [(a, b)], out, 0)], torch.float32)
    want = expected(form, a, b)
    exact = want.float().double()   # (beyond fp32's range: infinite)
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out == float("inf"), exact == float("inf")) and torch.equal(out == float("-inf"), exact == float("-inf"))
    fine = exact.isfinite()
    fine[70] = False
    assert (out.double() - want)[fine].norm() <= 2.0**-24 * (3 + K**0.5) * want[fine].norm()   # (whole fp32 elements beside those: a rounding a term)
    assert abs(out[70, 7].double() / want[70, 7] - 1) <= 1e-6


@pytest.mark.parametrize("product,tile", PARTS_CASES, ids=lambda v: "-".join(map(str, v)))
@pytest.mark.parametrize("size,other", [(1e-28, 1.0), (1e-31, 1.0), (1e-33, 1.0), (1e-35, 1.0), (1e-36, 1e10), (1e-20, 1e-12)])
def test_fp32_of_small_elements(dev, product, tile, size, other):
    """Elements whose third part is below bf16's range: as exact as fp32 instructions (a rounding a term), also where only some rows are that small."""
    form, M, N, K = product
    a, b = operands(form, M, N, K, torch.float32, dev, M + K)
    rows = a.t() if form == TN else a
    rows[::2] *= size
    b *= other
    out = torch.empty(M, N, device=dev)
    run_products([(form, [(a, b)], out, 0)], torch.float32)
    want = expected(form, a, b)
    for part in (slice(0, M, 2), slice(1, M, 2)):
        assert (out.double() - want)[part].norm() <= 2.0**-24 * (3 + K**0.5) * want[part].norm()


@pytest.mark.parametrize("product,tile", PARTS_CASES, ids=lambda v: "-".join(map(str, v)))
@pytest.mark.parametrize("size,other", [(1e-36, 1e20), (1e-37, 1e25), (1e-38, 1e20), (1e-38, 1e30), (3e-41, 1e10), (3e-41, 1e20), (1e-44, 1e30), (1e-12, 1e33), (1e13, 1e13), (1e-30, 1e37)])
def test_fp32_of_elements_far_apart(dev, product, tile, size, other):
    """Small elements, also below the normal numbers, against large ones, either operand's, all rows or some: as exact as fp32 instructions (a rounding a term).  And what leaves the range of the
    parts or of their sums at the other end."""
    form, M, N, K = product
    x, y = operands(form, M, N, K, torch.float32, dev, M + K)
    for swapped in (False, True):
        for some in (False, True):
            a, b = (x * other, y * size) if swapped else (x * size, y * other)
            if some:   # of the small ones every other row or column such that its sums are about 1
                rows = (b if form == NT else b.t()) if swapped else (a.t() if form == TN else a)
                rows[1::2] = ((y if form == NT else y.t()) if swapped else (x.t() if form == TN else x))[1::2] * (1 / other)
            out = torch.empty(M, N, device=dev)
            run_products([(form, [(a, b)], out, 0)], torch.float32)
            got, want = out.double(), expected(form, a, b)
            got, want = (got.t(), want.t()) if swapped else (got, want)
            for part in (slice(0, None, 2), slice(1, None, 2)):
                assert (got - want)[part].norm() <= 2.0**-24 * (3 + K**0.5) * want[part].norm(), (swapped, some)


@pytest.mark.parametrize("product,tile", PARTS_CASES, ids=lambda v: "-".join(map(str, v)))
def test_fp32_bits_of_an_element_are_those_of_its_row_and_column(dev, product, tile):
    """Whatever other rows and columns of the operands hold, and what lies beside them in memory."""
    form, M, N, K = product
    a, b = operands(form, M, N, K, torch.float32, dev, M + N)
    out, other = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev)
    run_products([(form, [(a, b)], out, 0)], torch.float32)
    x, y = a.clone(), b.clone()
    rows, columns = x.t() if form == TN else x, y if form != NT else y.t()
    rows[3, 5], rows[M - 1, K - 1], rows[70, 0], rows[37] = float("inf"), float("nan"), 3.4e38, 1e-38
    columns[2, N - 1], columns[0, 65], columns[1, 6] = float("-inf"), float("nan"), 2e32
    run_products([(form, [(x, y)], other, 0)], torch.float32)
    row, column = torch.ones(M, dtype=torch.bool, device=dev), torch.ones(N, dtype=torch.bool, device=dev)
    row[[3, M - 1, 70, 37]], column[[N - 1, 65, 6]] = False, False
    assert torch.equal(other[row][:, column], out[row][:, column])
    # as ranges of wider buffers, of dW's rows and dx's columns an odd number
    M, N, results = M - (form == TN), N - (form == NN), []
    for beside in (1.0, float("nan")):
        x, y = (torch.full((t.size(0), t.size(1) + 72), beside, device=dev)[:, :t.size(1) - odd] for t, odd in ((a, form == TN), (b, form == NN)))
        x.copy_(a[:, :x.size(1)]), y.copy_(b[:, :y.size(1)])
        results.append(torch.empty(M, N, device=dev))
        run_products([(form, [(x, y)], results[-1], 0)], torch.float32)
    assert torch.equal(*results)


@pytest.mark.parametrize("M,N,K", [(700, 1028, 68), (2047, 1380, 36), (2048, 1376, 40)])
def test_fp32_gate_up_out_of_the_range_of_the_parts(dev, M, N, K):
    """Elements of x and of either weight without parts, in ragged tiles: the bits of the product with both weights, where those of the others stay."""
    x, w = operands(NT, M, 2 * N, K, torch.float32, dev, M + N)
    L, st = _lib.lib(), torch.cuda.current_stream().cuda_stream
    results = []
    for out_of_range in (False, True):
        if out_of_range:
            x[3, 5], x[M - 1, K - 1], x[70, 0] = float("inf"), float("nan"), 3.4e38
            w[7, 2], w[N - 1, 0], w[N + 65, 1], w[2 * N - 1, 3] = 2e32, float("-inf"), float("nan"), 3.4e38
        wg, wu = w[:N], w[N:]
        gate, up, h, both = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev), torch.empty(M, N, device=dev), torch.empty(M, 2 * N, device=dev)
        assert L.mlts_gemm_swiglu_supports(_lib.MLTS_F32, M, N, K, K, K, N, N) is None and planned([(NT, M, N, K)], _lib.MLTS_F32, 3)[0][0] >= 64
        _lib.check(L.mlts_gemm_swiglu(_lib.MLTS_F32, M, N, K, x.data_ptr(), K, wg.data_ptr(), wu.data_ptr(), K, gate.data_ptr(), up.data_ptr(), N, h.data_ptr(), N, st))
        run_products([(NT, [(x, w)], both, 0)], torch.float32)
        results.append((both, torch.cat([gate, up], 1)))
        assert torch.equal(results[-1][0].nan_to_num(), results[-1][1].nan_to_num()) and torch.equal(both.isnan(), results[-1][1].isnan())
    rows, columns = torch.ones(M, dtype=torch.bool, device=dev), torch.ones(2 * N, dtype=torch.bool, device=dev)
    rows[[3, M - 1, 70]], columns[[7, N - 1, N + 65, 2 * N - 1]] = False, False
    assert torch.equal(results[0][1][rows][:, columns], results[1][1][rows][:, columns])


def test_fp32_sum_over_segments_in_slices(dev):
    """A sum over segments whose slabs are split over workgroups, alone and beside a weight gradient: slices that begin and end within segments."""
    gen = torch.Generator().manual_seed(8)
    rnd = lambda *shape: torch.randn(*shape, generator=gen).to(dev)
    for M, N, ks in ((200, 64, (520, 1000, 72)), (777, 132, (40, 1376)), (64, 256, (2000, 36, 516))):
        segments = [(rnd(M, k), rnd(k, N)) for k in ks]
        want, K = sum(expected(NN, a, b) for a, b in segments), sum(ks)
        for others in (0, 1):
            c, dw, dy = rnd(M, N), torch.empty(ks[0], N, device=dev), rnd(M, N)
            total = want + c.double()
            run_products([(NN, segments, c, 1)] + [(TN, [(segments[0][0], dy)], dw, 0)] * others, torch.float32)
            assert (c.double() - total).norm() <= 2.0**-24 * (4 + K**0.5) * total.norm()
            assert not others or (dw.double() - expected(TN, segments[0][0], dy)).norm() <= 2.0**-24 * (4 + M**0.5) * dw.double().norm()
