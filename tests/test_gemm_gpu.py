"""GPU parity of the matrix-core paths: complex GEMM, ComplexLinear and DFT-as-GEMM.

Oracle: the reference's four-real-matmul formulas (oracle.complex_matmul / complex_linear,
trnfft/complex.py:142-150, trnfft/nn.py:43-48) evaluated in float64 on the same inputs;
tolerance 1e-6*log2(K) relative L2 (K = contraction length).
"""

from __future__ import annotations

import math

import pytest
import torch

import oracle
import trnfft_amd
from conftest import rel_l2, seeded_complex, tol_pow2
from trnfft_amd import ComplexTensor
from trnfft_amd.nn import ComplexLinear

pytestmark = pytest.mark.gpu


def _tol_k(k):
    return 1e-6 * max(1.0, math.log2(k))


def _planes(shape, g):
    return torch.randn(*shape, generator=g), torch.randn(*shape, generator=g)


@pytest.mark.parametrize("m,k,n", [(128, 128, 128), (100, 33, 70), (1, 5, 3), (257, 1024, 129), (512, 64, 1000)])
def test_complex_gemm_vs_float64(m, k, n):
    g = torch.Generator().manual_seed(m * 7 + k)
    a = _planes((m, k), g)
    b = _planes((k, n), g)
    got = trnfft_amd.complex_matmul(ComplexTensor(a[0].cuda(), a[1].cuda()), ComplexTensor(b[0].cuda(), b[1].cuda()))
    ref = oracle.complex_matmul((a[0].double(), a[1].double()), (b[0].double(), b[1].double()))
    assert got.shape == (m, n)
    assert rel_l2(got.real, got.imag, *ref) <= _tol_k(k), (m, k, n)


@pytest.mark.parametrize("sa,sb", [
    ((4, 50, 33), (4, 33, 70)),        # batched
    ((4, 50, 33), (33, 70)),           # batched A, shared 2-D B (one GEMM over all rows)
    ((50, 33), (3, 33, 70)),           # shared A, batched B
    ((2, 1, 17, 9), (3, 9, 20)),       # broadcast batch axes -> (2, 3, 17, 20)
    ((2, 3, 17, 9), (1, 3, 9, 20)),
    ((33,), (33, 70)),                 # vector @ matrix
    ((50, 33), (33,)),                 # matrix @ vector
    ((5, 50, 33), (33,)),              # batched matrix @ vector
    ((33,), (4, 33, 7)),               # vector @ batched matrix
    ((33,), (33,)),                    # dot product -> 0-d
    ((0, 8, 5), (0, 5, 3)),            # empty batch
    ((70000, 2, 3), (70000, 3, 2)),    # more products than one launch's grid.y (65535)
])
def test_complex_matmul_torch_matmul_shapes(sa, sb):
    # the reference's complex_matmul is four torch.matmul (trnfft/complex.py:142-150), so it takes
    # every torch.matmul shape; the result and its shape match the same formula in float64
    g = torch.Generator().manual_seed(len(sa) * 10 + len(sb))
    a = _planes(sa, g)
    b = _planes(sb, g)
    got = ComplexTensor(a[0].cuda(), a[1].cuda()) @ ComplexTensor(b[0].cuda(), b[1].cuda())
    ref = oracle.complex_matmul((a[0].double(), a[1].double()), (b[0].double(), b[1].double()))
    assert tuple(got.real.shape) == tuple(ref[0].shape)
    if ref[0].numel():
        assert rel_l2(got.real, got.imag, *ref) <= _tol_k(sa[-1]), (sa, sb)


def test_complex_matmul_shape_mismatch_raises_like_torch():
    a = ComplexTensor(torch.randn(4, 5).cuda(), torch.randn(4, 5).cuda())
    b = ComplexTensor(torch.randn(2, 6, 3).cuda(), torch.randn(2, 6, 3).cuda())
    with pytest.raises(RuntimeError):
        a @ b


def test_complex_gemm_kat():
    a = ComplexTensor(torch.tensor([[1.0]]).cuda(), torch.tensor([[2.0]]).cuda())
    b = ComplexTensor(torch.tensor([[3.0]]).cuda(), torch.tensor([[4.0]]).cuda())
    c = a @ b
    assert c.real.item() == -5.0 and c.imag.item() == 10.0


@pytest.mark.parametrize("m,k,n,bias", [(64, 32, 48, True), (8192, 1024, 1024, False), (300, 129, 77, True)])
def test_complex_linear_vs_float64(m, k, n, bias):
    g = torch.Generator().manual_seed(42)
    x = _planes((m, k), g)
    w_re = torch.empty(n, k).uniform_(-1 / math.sqrt(k), 1 / math.sqrt(k), generator=g)
    w_im = torch.empty(n, k).uniform_(-1 / math.sqrt(k), 1 / math.sqrt(k), generator=g)
    b = _planes((n,), g) if bias else (None, None)
    got = trnfft_amd.complex_linear(
        ComplexTensor(x[0].cuda(), x[1].cuda()), w_re.cuda(), w_im.cuda(),
        None if b[0] is None else b[0].cuda(), None if b[1] is None else b[1].cuda(),
    )
    ref = oracle.complex_linear(
        (x[0].double(), x[1].double()), w_re.double(), w_im.double(),
        None if b[0] is None else b[0].double(), None if b[1] is None else b[1].double(),
    )
    assert rel_l2(got.real, got.imag, *ref) <= _tol_k(k), (m, k, n)


def test_complex_linear_module_matches_reference_formula():
    torch.manual_seed(42)
    layer = ComplexLinear(64, 96)
    assert set(layer.state_dict()) == {"W_re.weight", "W_im.weight", "bias_re", "bias_im"}
    with torch.no_grad():
        layer.bias_re.normal_()
        layer.bias_im.normal_()
    x = ComplexTensor(torch.randn(16, 64), torch.randn(16, 64))
    ref = oracle.complex_linear(
        (x.real.double(), x.imag.double()), layer.W_re.weight.detach().double(), layer.W_im.weight.detach().double(),
        layer.bias_re.detach().double(), layer.bias_im.detach().double(),
    )
    layer = layer.cuda()
    y = layer(ComplexTensor(x.real.cuda(), x.imag.cuda()))
    assert y.shape == (16, 96)
    assert rel_l2(y.real, y.imag, *ref) <= _tol_k(64)


@pytest.mark.parametrize("n", [8, 64, 256])
@pytest.mark.parametrize("inverse", [False, True])
def test_dft_gemm_vs_oracle(n, inverse):
    from trnfft_amd import fft_core as fc

    re, im = seeded_complex(1000, n)
    x = ComplexTensor(re.cuda(), im.cuda())
    got = fc._fft_via_gemm(x, inverse)
    ref = oracle.fft_core(re, im, inverse)
    assert rel_l2(got.real, got.imag, *ref) <= tol_pow2(n), (n, inverse)


def test_config5b_full_size_both_formulations():
    # the benchmark's DFT as a product at full size (65536 x 256, forward): the DFT-as-GEMM on the matrix cores
    # and the Stockham kernel, each against the oracle on all rows
    from trnfft_amd import fft_core as fc

    re, im = seeded_complex(65536, 256)
    x = ComplexTensor(re.cuda(), im.cuda())
    ref = oracle.fft_core(re, im, False)
    gemm = fc._fft_via_gemm(x, False)
    assert rel_l2(gemm.real, gemm.imag, *ref) <= tol_pow2(256)
    stockham = trnfft_amd.fft(x)
    assert rel_l2(stockham.real, stockham.imag, *ref) <= tol_pow2(256)


def test_dft_gemm_threshold_routing():
    from trnfft_amd import fft_core as fc

    re, im = seeded_complex(64, 256)
    old = fc._DFT_GEMM_THRESHOLD
    fc._DFT_GEMM_THRESHOLD = 256
    try:
        got = trnfft_amd.fft(ComplexTensor(re.cuda(), im.cuda()))
    finally:
        fc._DFT_GEMM_THRESHOLD = old
    ref = oracle.fft_core(re, im, False)
    assert rel_l2(got.real, got.imag, *ref) <= tol_pow2(256)


@pytest.mark.parametrize("batch,m,k,n", [
    (1, 33, 256, 35),      # one partial tile
    (1, 129, 1030, 130),   # four tiles, ragged last range, odd columns (scalar reduction)
    (1, 1024, 8192, 1024),  # a weight gradient
    (3, 40, 515, 64),      # batched, last range of three columns
])
@pytest.mark.parametrize("a_op,b_op", [(0, 0), (0, 1), (1, 3), (2, 0)])
def test_gemm_split_k_vs_float64(batch, m, k, n, a_op, b_op):
    # products of few output tiles are summed in several k ranges (workspace) and reduced
    import ctypes

    from trnfft_amd import _lib
    from trnfft_amd.dispatch import gemm_batched

    nbytes = ctypes.c_size_t()
    assert _lib.lib().tfa_complex_gemm_workspace_size(batch, m, n, k, ctypes.byref(nbytes)) == _lib.TFA_OK
    assert nbytes.value >= 2 * 8 * batch * m * n
    g = torch.Generator(device="cuda").manual_seed(m + k)

    def stored(rows, cols, op):
        shape = (batch, cols, rows) if op in (1, 2) else (batch, rows, cols)
        return tuple(torch.randn(*shape, generator=g, device="cuda") for _ in range(2))

    def applied(p, op):
        z = torch.complex(p[0].double(), p[1].double())
        z = z.transpose(1, 2) if op in (1, 2) else z
        return (z.conj() if op in (2, 3) else z).resolve_conj().contiguous()

    a, b = stored(m, k, a_op), stored(k, n, b_op)
    c_re, c_im = gemm_batched(*a, a_op, *b, b_op, batch, alpha=0.5)
    ref = 0.5 * torch.stack([x @ y for x, y in zip(applied(a, a_op), applied(b, b_op))])
    assert rel_l2(c_re, c_im, ref.real, ref.imag) <= _tol_k(k), (m, k, n)


def test_gemm_split_k_bias_matches_unsplit():
    from trnfft_amd import _lib
    from trnfft_amd.dispatch import gemm_ex, ptr, stream_handle

    g = torch.Generator(device="cuda").manual_seed(9)
    a, b = (tuple(torch.randn(*s, generator=g, device="cuda") for _ in range(2)) for s in ((70, 700), (50, 700)))
    bias = tuple(torch.randn(50, generator=g, device="cuda") for _ in range(2))
    got = gemm_ex(*a, _lib.OP_N, *b, _lib.OP_T, 1.0, *bias)
    ref = tuple(torch.empty(70, 50, device="cuda") for _ in range(2))
    rc = _lib.lib().tfa_complex_gemm_ex(70, 50, 700, ptr(a[0]), ptr(a[1]), 700, _lib.OP_N, ptr(b[0]), ptr(b[1]), 700,
                                        _lib.OP_T, 1.0, ptr(bias[0]), ptr(bias[1]), ptr(ref[0]), ptr(ref[1]), 50,
                                        stream_handle(a[0].device))
    _lib.check(rc, "tfa_complex_gemm_ex")
    # two fp32 sums of the same 1400 products in another order
    assert rel_l2(*got, *ref) <= 2 * _tol_k(700)


@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (5, 7, 3), (128, 16, 128), (129, 17, 127), (300, 15, 257), (256, 63, 131),
                                   (700, 130, 900)])
@pytest.mark.parametrize("a_op,b_op", [(a, b) for a in range(4) for b in range(4)])
def test_gemm_tile_edges_every_op(m, k, n, a_op, b_op):
    # tile and stage remainders in every operand order, conjugations included
    from trnfft_amd.dispatch import gemm_ex

    g = torch.Generator(device="cuda").manual_seed(m * 31 + k)

    def stored(rows, cols, op):
        shape = (cols, rows) if op in (1, 2) else (rows, cols)
        return tuple(torch.randn(*shape, generator=g, device="cuda") for _ in range(2))

    def applied(p, op):
        z = torch.complex(p[0].double().cpu(), p[1].double().cpu())
        z = z.T if op in (1, 2) else z
        return z.conj().resolve_conj() if op in (2, 3) else z

    a, b = stored(m, k, a_op), stored(k, n, b_op)
    got = gemm_ex(*a, a_op, *b, b_op, 0.5)
    ref = 0.5 * (applied(a, a_op) @ applied(b, b_op))
    assert rel_l2(*got, ref.real, ref.imag) <= _tol_k(k), (m, k, n)


def test_gemm_operands_of_one_sign():
    # the running sums grow all the way, so a truncating accumulation would show: K / 16 rounded
    # additions and two truncations per stage of 16, each 2^-24 of the sum at most
    k = 1024
    g = torch.Generator(device="cuda").manual_seed(2)
    a = tuple(torch.rand(512, k, generator=g, device="cuda") for _ in range(2))
    b = tuple(torch.rand(k, 4096, generator=g, device="cuda") for _ in range(2))
    got = trnfft_amd.complex_matmul(ComplexTensor(*a), ComplexTensor(*b))
    ref = oracle.complex_matmul(tuple(t.double() for t in a), tuple(t.double() for t in b))
    assert rel_l2(got.real, got.imag, *ref) <= 2.0**-24 * (2 + math.sqrt(k / 16))


@pytest.mark.parametrize("scale", [2.0**-90, 2.0**-110, 2.0**-122, 2.0**100])
def test_gemm_extreme_magnitudes(scale):
    # operands whose bf16 pieces would be denormal keep fp32 precision
    g = torch.Generator(device="cuda").manual_seed(3)
    a = tuple(torch.randn(200, 70, generator=g, device="cuda") * scale for _ in range(2))
    b = tuple(torch.randn(70, 150, generator=g, device="cuda") for _ in range(2))
    got = trnfft_amd.complex_matmul(ComplexTensor(*a), ComplexTensor(*b))
    ref = oracle.complex_matmul(tuple(t.double() for t in a), tuple(t.double() for t in b))
    assert rel_l2(got.real.double() / scale, got.imag.double() / scale, ref[0] / scale, ref[1] / scale) <= _tol_k(70)


@pytest.mark.parametrize("k", [40, 512])  # without and with a split of k
def test_gemm_nonfinite_operands(k):
    # infinities and NaN reach exactly the outputs they reach in fp32 arithmetic
    g = torch.Generator(device="cuda").manual_seed(4)
    a = tuple(torch.randn(150, k, generator=g, device="cuda") for _ in range(2))
    b = tuple(torch.randn(k, 140, generator=g, device="cuda") for _ in range(2))
    a[0][3, 5] = float("inf")
    a[1][7, k - 1] = float("nan")
    b[1][11, 139] = -float("inf")
    got = trnfft_amd.complex_matmul(ComplexTensor(*a), ComplexTensor(*b))
    ref = oracle.complex_matmul(tuple(t.double() for t in a), tuple(t.double() for t in b))
    for x, y in zip((got.real, got.imag), ref):
        assert torch.equal(torch.isnan(x), torch.isnan(y))
        assert torch.equal(torch.isposinf(x), torch.isposinf(y))
        assert torch.equal(torch.isneginf(x), torch.isneginf(y))
    ok = [torch.isfinite(y) for y in ref]
    assert rel_l2(got.real[ok[0]], got.imag[ok[1]], ref[0][ok[0]], ref[1][ok[1]]) <= _tol_k(k)


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 65), (33, 64), (63, 130), (64, 1), (1000, 257), (8192, 1024), (100000, 3)])
def test_column_sums_vs_float64(rows, cols):
    from trnfft_amd.dispatch import column_sums

    g = torch.Generator(device="cuda").manual_seed(rows)
    re, im = (torch.randn(rows, cols, generator=g, device="cuda") for _ in range(2))
    got = column_sums(re, im)
    # chains of at most rows / 32 additions between pairwise ones; sqrt of that many roundings of 2^-24
    tol = 2.0**-24 * (4 + math.sqrt(rows / 32 + 1))
    assert rel_l2(*got, re.double().sum(0), im.double().sum(0)) <= tol


@pytest.mark.parametrize("k", [1, 40])
@pytest.mark.parametrize("value", [1 + 2.0**-7 - 2.0**-23, 1 + 2.0**-8 - 2.0**-16, 2 - 2.0**-23, None])
def test_gemm_sums_of_one_product(k, value):
    # every sum is one product (one nonzero k per row), element by element.  What the bf16 pieces leave out is at
    # most 2 * 2^-24 of the operands' powers of two, and the sum is rounded at its full size once (2^-23 where
    # that is a truncation): 2^-22 of the product
    g = torch.Generator(device="cuda").manual_seed(7)
    m, n = 130, 140
    a, b = torch.zeros(m, k, device="cuda"), torch.zeros(k, n, device="cuda")
    rows = torch.arange(m, device="cuda")
    draw = lambda *s: torch.rand(*s, generator=g, device="cuda") + 0.5 if value is None else torch.full(s, value, device="cuda")  # noqa: E731
    a[rows, rows % k] = draw(m)
    b[:] = draw(k, n)
    got = trnfft_amd.complex_matmul(ComplexTensor(a, torch.zeros_like(a)), ComplexTensor(b, b))
    ref = a.double() @ b.double()
    for plane in (got.real, got.imag):
        err = (plane.double() - ref) / ref
        assert err.abs().max() <= 2.0**-22


@pytest.mark.parametrize("k", [5, 40])
@pytest.mark.parametrize("small,large", [(1.99 * 2.0**-120, 2.0**60), (1.2345 * 2.0**-118, 2.0**40), (1.2345 * 2.0**-140, 1.357 * 2.0**100),
                                         (1.2345 * 2.0**-70, 1.357 * 2.0**-60), (1.99 * 2.0**-103, 1.5)])
def test_gemm_small_operand_beside_large_ones(k, small, large):
    # a run of operands whose large value meets a zero: only the small one reaches the sum, at fp32 precision
    # (test_gemm_sums_of_one_product), and the rest of the tile is as ordinary as ever
    g = torch.Generator(device="cuda").manual_seed(8)
    a, b = (torch.randn(*s, generator=g, device="cuda") for s in ((70, k), (k, 90)))
    a[3, :], b[:, 5] = 0.0, 0.0
    a[3, 0], a[3, 1] = 1.0, small
    b[1, 5] = large
    got = trnfft_amd.complex_matmul(ComplexTensor(a, torch.zeros_like(a)), ComplexTensor(b, torch.zeros_like(b)))
    want = a[3, 1].double().item() * b[1, 5].double().item()
    assert abs(got.real[3, 5].double().item() - want) <= 2.0**-22 * want
    ref = a.double() @ b.double()
    keep = ref.abs() > 1e-12
    assert rel_l2(got.real[keep], got.imag[keep], ref[keep], torch.zeros_like(ref[keep])) <= _tol_k(k)


@pytest.mark.parametrize("low,high", [(-118, 100), (-126, -60), (60, 126)])
def test_gemm_scaled_columns(low, high):
    # A D and D^-1 B for a diagonal D of powers of two: the products, and so the result, are those of A B
    g = torch.Generator(device="cuda").manual_seed(9)
    a = tuple(torch.randn(150, 200, generator=g, device="cuda") for _ in range(2))
    b = tuple(torch.randn(200, 140, generator=g, device="cuda") for _ in range(2))
    d = 2.0 ** torch.randint(low, high, (200,), generator=g, device="cuda").double()
    sa = tuple((t.double() * d).float() for t in a)
    sb = tuple((t.double() / d[:, None]).float() for t in b)
    got = trnfft_amd.complex_matmul(ComplexTensor(*sa), ComplexTensor(*sb))
    ref = oracle.complex_matmul(tuple(t.double() for t in sa), tuple(t.double() for t in sb))
    assert rel_l2(got.real, got.imag, *ref) <= _tol_k(200)


@pytest.mark.parametrize("k", [16, 17, 40, 512])
@pytest.mark.parametrize("sa,sb", [(-55, -55), (-50, -65), (-59, -59), (-100, 0), (-105, 0), (-108, -5), (-100, 100), (-16, -100)])
def test_gemm_sums_around_the_fp32_limit(k, sa, sb):
    # sums on both sides of the limit below which a workgroup takes fp32 products: 2 k rounded products each way
    g = torch.Generator(device="cuda").manual_seed(10)
    a = tuple(torch.randn(140, k, generator=g, device="cuda") * 2.0**sa for _ in range(2))
    b = tuple(torch.randn(k, 150, generator=g, device="cuda") * 2.0**sb for _ in range(2))
    got = trnfft_amd.complex_matmul(ComplexTensor(*a), ComplexTensor(*b))
    ref = oracle.complex_matmul(tuple(t.double() for t in a), tuple(t.double() for t in b))
    assert rel_l2(got.real, got.imag, *ref) <= 2.0**-24 * math.sqrt(2 * k)


@pytest.mark.parametrize("batch,m,k,n", [(1, 1, 1, 1), (3, 129, 16, 127), (700, 5, 7, 3), (300, 16, 16, 16), (2, 130, 17, 260)])
@pytest.mark.parametrize("a_op,b_op", [(0, 0), (0, 1), (1, 3), (2, 0), (3, 2)])
def test_gemm_batches_of_one_stage(batch, m, k, n, a_op, b_op):
    # up to 16 k: one stage of fp32 products, at fp32's own error
    from trnfft_amd.dispatch import gemm_batched

    g = torch.Generator(device="cuda").manual_seed(m + k)

    def stored(rows, cols, op):
        shape = (batch, cols, rows) if op in (1, 2) else (batch, rows, cols)
        return tuple(torch.randn(*shape, generator=g, device="cuda") for _ in range(2))

    def applied(p, op):
        z = torch.complex(p[0].double().cpu(), p[1].double().cpu())
        z = z.transpose(1, 2) if op in (1, 2) else z
        return z.conj().resolve_conj() if op in (2, 3) else z

    a, b = stored(m, k, a_op), stored(k, n, b_op)
    got = gemm_batched(*a, a_op, *b, b_op, batch, alpha=0.5)
    ref = 0.5 * (applied(a, a_op) @ applied(b, b_op))
    assert rel_l2(*got, ref.real, ref.imag) <= 2.0**-24 * math.sqrt(2 * k)


def test_products_and_column_sums_without_memory_for_scratch(monkeypatch):
    # the scratch of a split product (and of the bias gradient) is an option: without memory for it the call runs unsplit
    from trnfft_amd import dispatch

    g = torch.Generator(device="cuda").manual_seed(11)
    m, k, n = 70, 2000, 50
    a, b = (tuple(torch.randn(*s, generator=g, device="cuda") for _ in range(2)) for s in ((m, k), (k, n)))
    empty, refused = torch.empty, []

    def no_scratch(*size, **kw):
        if len(size) == 1 and isinstance(size[0], int):
            refused.append(size[0])
            raise torch.OutOfMemoryError("no memory for scratch")
        return empty(*size, **kw)

    monkeypatch.setattr(dispatch.torch, "empty", no_scratch)
    got = dispatch.gemm_ex(*a, 0, *b, 0)
    sums = dispatch.column_sums(*b)
    monkeypatch.undo()
    assert len(refused) == 2
    ref = oracle.complex_matmul(tuple(t.double() for t in a), tuple(t.double() for t in b))
    assert rel_l2(*got, *ref) <= _tol_k(k)
    # one chain of k / 32 additions between pairwise ones
    assert rel_l2(*sums, b[0].double().sum(0), b[1].double().sum(0)) <= 2.0**-24 * (4 + math.sqrt(k / 32 + 1))
