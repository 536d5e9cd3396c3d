"""fp32 products on the split-operand GEMM (tg_matmul, tg_gemm, tg_gemm_wgrad) against
float64, at the edges of its tiles, K splits and kernels, and the operand values that its
bf16 split cannot hold (which it computes again on the fp32 matrix cores)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def L():
    from tensor_gpu_v2 import _lib
    return _lib


def _mk(g, r, c, ld=None):
    t = torch.randn(r, ld or c, generator=g, device="cuda")
    return t[:, :c] if ld else t


def _check(c, a, b, what, extra=0.0):
    """|c - a@b| within the worst case of the summation, elementwise: six MFMAs of 16
    products each (and their finishing sums), one rounding of at most 2^-23 of
    sum |a||b| per MFMA, and 2^-22 for the products the split leaves out."""
    K = a.shape[1]
    n = 6 * (K // 16 + 1) + 40
    mag = a.double().abs() @ b.double().abs() + extra
    err = (c.double() - (a.double() @ b.double() + extra)).abs()
    assert bool((err <= (n * 2.0 ** -23 + 2.0 ** -22) * mag + 1e-44).all()), \
        f"{what}: {(err / mag.clamp_min(1e-300)).max().item():.2e}"


SHAPES = [(1, 1, 1), (5, 7, 9), (31, 33, 8), (32, 256, 784), (33, 257, 785), (64, 64, 4561),
          (129, 65, 31), (300, 260, 97), (1000, 1000, 1000), (257, 129, 4099),
          (4099, 4100, 33), (2050, 2100, 64), (7, 3000, 513)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
def test_matmul_f32(cuda, M, N, K, ta, tb):
    g = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)
    a = _mk(g, K, M) if ta else _mk(g, M, K)
    b = _mk(g, N, K) if tb else _mk(g, K, N)
    A, B = (a.t() if ta else a), (b.t() if tb else b)
    c = L().matmul2d(a, b, trans_a=ta, trans_b=tb)
    _check(c, A, B, "matmul2d")
    # unsplit, batched with a broadcast operand, accumulating
    c2 = torch.ones(2, M, N, device="cuda")
    L().gemm(a, b, c2, ta, tb, 1.0, 1.0, M, N, K, a.shape[1], b.shape[1], N, 0, 0, M * N, 2)
    assert torch.equal(c2[0], c2[1])
    _check(c2[1], A, B, "gemm", 1.0)
    bias = torch.randn(N, generator=g, device="cuda")
    if not ta:
        y = torch.empty(M, N, device="cuda")
        L().gemm_bias(a, b, bias, y, trans_b=tb)
        assert torch.allclose(y, c + bias, rtol=1e-6, atol=1e-6 * float(c.abs().max()) + 1e-6)


@pytest.mark.parametrize("M,N,K", [(1722, 370, 427), (2049, 33, 65), (2081, 31, 7), (2064, 64, 32),
                                   (1114, 632, 785)])
def test_matmul_f32_transposed_small_output(cuda, M, N, K):
    """A^T B of few 32 x 32 tiles: four wavefronts a tile, at its edges and k remainders."""
    test_matmul_f32(cuda, M, N, K, True, False)


@pytest.mark.parametrize("K,M,N", [(4561, 64, 64), (130, 33, 257), (8932, 130, 70), (77, 5, 3)])
def test_wgrad_f32(cuda, K, M, N):
    g = torch.Generator(device="cuda").manual_seed(K)
    x, gr = _mk(g, K, M), _mk(g, K, N)
    dw, db = torch.ones(M, N, device="cuda"), torch.ones(N, device="cuda")
    L().wgrad(x, gr, dw, True, db, True)
    _check(dw, x.t(), gr, "wgrad", 1.0)
    assert torch.allclose(db.double(), gr.double().sum(0) + 1.0, rtol=0, atol=1e-5 * K ** 0.5)


@pytest.mark.parametrize("M,N,K", [(70, 80, 100), (600, 700, 300), (2100, 4200, 40)])
def test_matmul_f32_misaligned_rows(cuda, M, N, K):
    """Operands one element off 16-byte alignment with odd leading dimensions."""
    g = torch.Generator(device="cuda").manual_seed(K)
    buf = torch.randn(M * (K + 3) + 1, generator=g, device="cuda")[1:].view(M, K + 3)
    b = torch.randn(K, N + 5, generator=g, device="cuda")
    c = torch.empty(M, N, device="cuda")
    L().gemm(buf, b, c, False, False, 1.0, 0.0, M, N, K, K + 3, N + 5, N)
    _check(c, buf[:, :K], b[:, :N], "misaligned")


@pytest.mark.parametrize("M,N,K", [(40, 50, 100), (700, 800, 300), (4099, 4100, 33)])
@pytest.mark.parametrize("kind", ["inf", "nan", "tiny", "tiny_row", "huge", "overflow", "denormal"])
def test_matmul_f32_values_outside_the_split(cuda, M, N, K, kind):
    g = torch.Generator(device="cuda").manual_seed(11)
    a, b = _mk(g, M, K), _mk(g, K, N)
    if kind == "inf":
        a[M // 2, K // 3] = float("inf")
        b[0, N - 1] = -float("inf")
        b[:, 3] = 0.0
    elif kind == "nan":
        a[M - 1, K - 1] = float("nan")
    elif kind == "tiny":
        a *= 1e-36
    elif kind == "tiny_row":
        a[M // 2] *= 1e-35
    elif kind == "huge":
        a[1, 2] = 3.4e38
        b[2] *= 1e-30
    elif kind == "overflow":
        a[3] *= 1e30
        b *= 1e30
    elif kind == "denormal":
        a[5] = 1e-40
        b *= 1e10
    c = L().matmul2d(a, b)
    want = (a.double() @ b.double())
    got, ref = c.double(), want.float().double()  # (float64 holds the products exactly enough)
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) or kind == "overflow"
    fin = torch.isfinite(ref) & (want.abs() < 1e38)
    inf = torch.isinf(ref) & (want.abs() > 1e39)
    if kind != "overflow":
        assert torch.equal(got[inf], ref[inf])
    else:
        assert bool((~torch.isfinite(got[inf])).all())
    mag = a.double().abs() @ b.double().abs()
    err = (got - want).abs()
    ok = err[fin] <= (6 * (K // 16 + 1) + K) * 2.0 ** -23 * mag[fin] + K * 1.5e-45
    assert bool(ok.all()), f"{kind}: {(err[fin] / mag[fin]).max().item():.2e}"


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_column_sums_are_not_biased(cuda, ta, tb):
    """Sums of n = 131072 rows of a product of unit normals (entries of size sqrt(K)): an entry
    takes K / 16 sums, each off by up to 2^-24 of its size.  Errors to either side add up to
    sqrt(n) of them (held to 4 sigma); errors to one side would to n of about half of them, 45
    times the bound."""
    M, N, K = 131072, 256, 368
    g = torch.Generator(device="cuda").manual_seed(3)
    a = torch.randn(*((K, M) if ta else (M, K)), device="cuda", generator=g)
    b = torch.randn(*((N, K) if tb else (K, N)), device="cuda", generator=g)
    c = L().matmul2d(a, b, trans_a=bool(ta), trans_b=bool(tb))
    ref = a.double().sum(1 if ta else 0) @ (b.double().T if tb else b.double())
    err = float((c.double().sum(0) - ref).abs().max())
    assert err <= 4 * M ** 0.5 * (K / 16) * 2.0 ** -24 * K ** 0.5, err


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(40, 50, 100), (70, 2050, 300), (700, 800, 500), (1100, 2060, 129)])
@pytest.mark.parametrize("mixed", [False, True])
def test_matmul_f32_subnormal_operands(cuda, M, N, K, ta, tb, mixed):
    """Operands down to the least subnormal number, beside ordinary ones, count in full: the
    bound is that of ordinary operands, plus one rounding of a subnormal entry a product."""
    g = torch.Generator(device="cuda").manual_seed(M + K)
    a = _mk(g, M, K)
    if mixed:
        e = torch.randint(-149, 1, (M, K), generator=g, device="cuda").double()
        a = (a.double() * 2.0 ** e).float()
    a[1] = 4e-41      # rounds to zero in bf16
    a[2] = 1e-42
    a[3] = 2.0 ** -149
    b = _mk(g, K, N)
    b[:, 1] *= 1e20
    if mixed:
        b[:, 2] = -3e-44
        b[:, 3] *= 1e-18
    c = L().matmul2d(a.t().contiguous() if ta else a, b.t().contiguous() if tb else b,
                     trans_a=bool(ta), trans_b=bool(tb))
    want = a.double() @ b.double()
    mag = a.double().abs() @ b.double().abs()
    n = 6 * (K // 16 + 1) + 40
    err = (c.double() - want).abs()
    assert bool((err <= (n * 2.0 ** -23 + 2.0 ** -22) * mag + K * 1.5e-45).all())
    assert bool((c[1:4, 1] != 0).all())


def _operands(kind, g, M, N, K):
    a, b = _mk(g, M, K), _mk(g, K, N)
    return {"normal": (a, b), "relu": (a.relu(), b), "positive": (a.abs(), b.abs()),
            "offset": (a + 3, b + 3)}[kind]


@pytest.mark.parametrize("kind", ["normal", "relu", "positive", "offset"])
@pytest.mark.parametrize("M,N,K", [(4096, 4096, 2048), (1024, 1024, 1024), (700, 800, 4096)])
@pytest.mark.parametrize("ta", [False, True])
def test_entries_are_no_further_off_than_a_partial_sum_scheme(cuda, M, N, K, kind, ta):
    """Partial sums of 64 k, added in fp32: the additions round by 2^-24 / sqrt(3) of a sum
    that grows to its size over K / 64 of them (1.4e-7 in the 2-norm at K = 2048), the
    partial sums themselves are off by about 1e-7 of theirs; held to twice that.  One
    accumulator over K would be off by 6 to 7e-7 at K = 2048."""
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = _operands(kind, g, M, N, K)
    c = L().matmul2d(a.t().contiguous() if ta else a, b, trans_a=ta)
    want = a.double() @ b.double()
    e = float((c.double() - want).norm() / want.norm())
    lim = 2 * ((K / 128) ** 0.5 * 2.0 ** -24 / 3 ** 0.5 + 1e-7)
    assert e < lim, f"{e:.2e} {lim:.2e}"


@pytest.mark.parametrize("kind", ["normal", "relu", "positive", "offset"])
@pytest.mark.parametrize("M,N,K", [(8192, 1024, 368), (13632, 368, 1472), (2048, 2304, 512)])
def test_column_sums_of_one_sign(cuda, M, N, K, kind):
    """Entries that err to either side at random (up to 2.5e-7 of their size) leave 1/sqrt(M)
    of that in a column sum relative to M entries; allowed are 4 times it and 8e-9, an eighth
    of fp32's own rounding of the sum.  One accumulator leaves 3 to 6e-8."""
    g = torch.Generator(device="cuda").manual_seed(M)
    a, b = _operands(kind, g, M, N, K)
    c = L().matmul2d(a, b)
    want = a.double() @ b.double()
    d = (c.double() - want).sum(0)
    e = float(d.norm() / (want.norm(dim=0) * M ** 0.5).norm())
    assert e < 4 * 2.5e-7 / M ** 0.5 + 8e-9, f"{e:.2e}"


@pytest.mark.parametrize("M,N,K", [(700, 800, 500), (2100, 4200, 300), (4096, 2048, 1024)])
@pytest.mark.parametrize("ta", [False, True])
def test_equal_rows_give_equal_rows(cuda, M, N, K, ta):
    """A row's result does not depend on where in the operand the row stands."""
    g = torch.Generator(device="cuda").manual_seed(N)
    a, b = _mk(g, M, K), _mk(g, K, N)
    for r in (1, 2, 77, M // 2, M - 1):
        a[r] = a[0]
    c = L().matmul2d(a.t().contiguous() if ta else a, b, trans_a=ta)
    for r in (1, 2, 77, M // 2, M - 1):
        assert torch.equal(c[r], c[0])
