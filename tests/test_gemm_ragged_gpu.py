"""16-bit products at ragged sizes and alignments: k past the last tile (masked DMA), any
M and N, odd rows (copied with aligned ones where a workspace holds them, else the
register-staged kernel), K splits whose last chunk is short, and the fused and grouped forms at such sizes, against float64 products of the same
16-bit operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DT = {"fp16": torch.float16, "bf16": torch.bfloat16}
EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}


def L():
    from tensor_gpu_v2 import _lib
    return _lib


def _bound(c, a, b, what, add=0.0):
    """16-bit products are exact in fp32; a sum of K of them rounds at most once per MFMA
    of 16 k (2^-23 of sum |a||b| each) and once when it is stored."""
    K = a.shape[1]
    want = a.double() @ b.double() + add
    mag = a.double().abs() @ b.double().abs() + abs(add)
    tol = (K // 16 + 40) * 2.0 ** -23 * mag + 1.01 * EPS[c.dtype] * want.abs() + 1e-7
    err = (c.double() - want).abs()
    assert bool((err <= tol).all()), f"{what}: {(err - tol).max().item():.2e}"


def _mk(g, r, c, dt, pad=0, off=0):
    """[r, c] with `pad` extra columns of NaN and a base `off` elements into its buffer."""
    buf = torch.full((r * (c + pad) + off + 8,), float("nan"), device="cuda", dtype=dt)
    v = buf[off:off + r * (c + pad)].view(r, c + pad)
    v[:, :c] = torch.randn(r, c, generator=g, device="cuda").to(dt)
    return v[:, :c]


SHAPES = [(1, 8, 8), (8, 8, 1), (1, 1, 1), (5, 7, 9), (64, 64, 72), (129, 136, 200), (300, 264, 65),
          (1917, 808, 808), (3290, 768, 768), (257, 1000, 4104), (70, 50257, 64), (513, 1025, 777),
          (4100, 2056, 104)]


@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_matmul_ragged(cuda, M, N, K, dt):
    dt = DT[dt]
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N + K)
    for ta in (False, True):
        for tb in (False, True):
            a = _mk(g, K, M, dt) if ta else _mk(g, M, K, dt)
            b = _mk(g, N, K, dt) if tb else _mk(g, K, N, dt)
            A, B = (a.t() if ta else a), (b.t() if tb else b)
            for odt in (dt, torch.float32):
                c = L().matmul2d(a.contiguous(), b.contiguous(), trans_a=ta, trans_b=tb,
                                 out_dtype=odt)
                _bound(c, A, B, f"matmul2d {ta} {tb} {odt}")


@pytest.mark.parametrize("M,N,K,pad,off", [(130, 136, 72, 8, 0), (130, 136, 72, 24, 8),
                                           (200, 130, 100, 3, 1), (2100, 4200, 65, 1, 3),
                                           (1000, 1000, 200, 5, 2), (40, 24, 7, 2, 1)])
def test_gemm_padded_rows(cuda, M, N, K, pad, off):
    """Padded leading dimensions (NaN in the padding: reading it would show) at aligned and
    odd row starts, accumulating, in a batch."""
    g = torch.Generator(device="cuda").manual_seed(M + K)
    dt = torch.float16
    for ta in (False, True):
        for tb in (False, True):
            a = _mk(g, K, M, dt, pad, off) if ta else _mk(g, M, K, dt, pad, off)
            b = _mk(g, N, K, dt, pad, off) if tb else _mk(g, K, N, dt, pad, off)
            c = torch.ones(2, M, N, device="cuda")
            L().gemm(a, b, c, ta, tb, 1.0, 1.0, M, N, K, a.stride(0), b.stride(0), N, 0, 0, M * N,
                     2)
            assert torch.equal(c[0], c[1])
            _bound(c[0], a.t() if ta else a, b.t() if tb else b, f"padded {ta} {tb}", 1.0)


@pytest.mark.parametrize("K,M,N", [(7230, 64, 64), (3290, 768, 2304), (1917, 808, 3232),
                                   (85, 40, 48), (7231, 72, 63), (9, 8, 8)])
def test_wgrad_ragged_tokens(cuda, K, M, N):
    g = torch.Generator(device="cuda").manual_seed(K)
    x, gr = _mk(g, K, M, torch.bfloat16), _mk(g, K, N, torch.bfloat16)
    x, gr = x.contiguous(), gr.contiguous()
    dw, db = torch.ones(M, N, device="cuda"), torch.ones(N, device="cuda")
    L().wgrad(x, gr, dw, True, db, True)
    _bound(dw, x.t(), gr, "wgrad", 1.0)
    mag = gr.double().abs().sum(0) + 1
    assert bool(((db.double() - gr.double().sum(0) - 1).abs() <= (K + 8) * 2.0 ** -23 * mag).all())
    # grouped: the members of one input shape in one call equal the members' own products
    ws = [torch.zeros(M, N, device="cuda") for _ in range(3)]
    bs = [torch.zeros(N, device="cuda") for _ in range(3)]
    L().wgrad_group([x, x, x], [gr, gr * 0.5, gr], ws, [False] * 3, bs, [False] * 3)
    assert torch.equal(ws[0], ws[2]) and torch.equal(bs[0], bs[2])
    _bound(ws[1], x.t(), gr * 0.5, "wgrad_group")


@pytest.mark.parametrize("M,N,K", [(357, 512, 128), (1917, 3232, 808), (61, 136, 72),
                                   (257, 264, 1000), (1917, 3232, 832), (61, 136, 64),
                                   (257, 264, 1024), (9, 72, 192), (300, 56, 128)])
def test_epilogue_ragged_equals_separate(cuda, M, N, K):
    """Fused where K is a multiple of 64 and N one of 8 from 64 on, at any M; refused (False,
    nothing run) elsewhere."""
    fused = K % 64 == 0 and N >= 64
    dt = torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(N)
    a, b = _mk(g, M, K, dt).contiguous(), (_mk(g, K, N, dt).contiguous() * 0.05)
    bias = torch.randn(N, generator=g, device="cuda")
    r = _mk(g, M, N, dt).contiguous()
    ref = torch.empty(M, N, device="cuda", dtype=dt)
    L().gemm_bias(a, b, bias, ref)
    _bound(ref, torch.cat([a.double(), torch.ones(M, 1, device="cuda").double()], 1),
           torch.cat([b.double(), bias.double()[None]], 0), "bias")
    out, act = torch.empty_like(ref), torch.empty_like(ref)
    assert L().gemm_epilogue("gelu_fwd", a, b, act, out, bias) is fused
    if fused:
        assert torch.equal(out, ref)
        assert torch.equal(act, L().act_fwd("gelu", ref))
    out = torch.empty_like(ref)
    assert L().gemm_epilogue("residual", a, b, r, out, bias) is fused
    if fused:
        assert torch.equal(out, ref + r)
    # GELU backward: A [M, K] @ W^T with W [N, K]
    w = _mk(g, N, K, dt).contiguous()
    d = torch.empty_like(ref)
    assert L().gemm_epilogue("gelu_bwd", a, w, r, d) is fused
    if fused:
        want = torch.empty_like(ref)
        L().act_bwd("gelu", r, L().matmul2d(a, w, trans_b=True), want, False)
        assert torch.equal(d, want)


@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("odt", ["same", "fp32"])
@pytest.mark.parametrize("M,N,K,off", [(256, 257, 128, 1), (300, 1025, 72, 0), (512, 515, 264, 3),
                                       (1024, 2049, 64, 7), (129, 131, 40, 5)])
def test_gemm_rows_of_c_at_any_element(cuda, M, N, K, off, odt, dt):
    """Full tiles written to (and, accumulating, read from) rows of C that start at any
    element; nothing past C's ends is touched.  Operands of -1, 0 and 1: every sum is a whole
    number below 2^8, exact in each type."""
    dt = DT[dt]
    odt = dt if odt == "same" else torch.float32
    g = torch.Generator(device="cuda").manual_seed(N)
    a, b = (torch.randint(-1, 2, (r, K), generator=g, device="cuda").to(dt) for r in (M, N))
    want = a.float() @ b.float().t().contiguous()
    assert float(want.abs().max()) < 250
    for beta in (0.0, 1.0):
        buf = torch.full((M * N + off + 64,), 2.0, device="cuda", dtype=odt)
        c = buf[off:off + M * N].view(M, N)
        L().gemm(a, b, c, False, True, 1.0, beta, M, N, K, K, K, N)
        assert torch.equal(c.float(), want + 2 * beta)
        assert bool((buf[:off] == 2).all()) and bool((buf[off + M * N:] == 2).all())
        # B as [K, N], odd rows: copied with aligned ones
        d = torch.full((M, N), 2.0, device="cuda", dtype=odt)
        L().matmul2d(a, b.t().contiguous(), d, beta=beta)
        assert torch.equal(d.float(), want + 2 * beta)


@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("M,N,K", [(128, 128, 64), (300, 257, 72), (512, 1024, 128),
                                   (1030, 515, 264), (4096, 4096, 64)])
def test_gemm_16bit_accumulation_rounds_once(cuda, M, N, K, dt):
    """C += A B in 16 bits adds in fp32 and rounds the sum, in full and in edge tiles of each
    block shape: rounding the product first would leave up to another half unit in the last
    place, of the product, where C cancels it."""
    dt = DT[dt]
    g = torch.Generator(device="cuda").manual_seed(M)
    a, b = _mk(g, M, K, dt).contiguous(), _mk(g, N, K, dt).contiguous()
    ab = a.double() @ b.double().t()
    c0 = (-ab + 0.25 * torch.randn(M, N, generator=g, device="cuda")).to(dt)
    c = c0.clone()
    L().gemm(a, b, c, False, True, 1.0, 1.0, M, N, K, K, K, N)
    want = ab + c0.double()
    tol = (K // 16 + 40) * 2.0 ** -23 * (a.double().abs() @ b.double().abs().t() + c0.double().abs())
    err = (c.double() - want).abs()
    assert bool((err <= tol + 1.01 * EPS[dt] * want.abs()).all()), float(err.max())


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_ragged_copies_only_where_they_serve(cuda, dt):
    """Odd rows are copied with aligned ones for the DMA-staged kernel only: not where the
    other operand is misaligned (the workspace stays as it was), and no workspace is asked
    for where rows are too long for it."""
    code, f32 = L().dtype_code(torch.empty(0, dtype=dt)), L().dtype_code(torch.empty(0))
    lib, s = L().load(), L().stream_handle()
    M, N, K = 520, 1025, 1000
    g = torch.Generator(device="cuda").manual_seed(3)
    for off in (0, 1):
        a, b = _mk(g, M, K, dt, 0, off), _mk(g, K, N, dt)
        nb = lib.tg_matmul_workspace(code, 0, 0, M, N, K)
        assert nb == (K * 1032 * 2 + 255) // 256 * 256
        ws = torch.full((nb,), 0x5a, device="cuda", dtype=torch.uint8)
        c = torch.empty(M, N, device="cuda")
        assert lib.tg_matmul(code, f32, 0, 0, M, N, K, 1.0, a.data_ptr(), K, b.data_ptr(), N, None,
                             0.0, c.data_ptr(), N, ws.data_ptr(), nb, s) == 0
        _bound(c, a, b, f"off {off}")
        assert bool((ws == 0x5a).all()) == (off == 1)
        x, gr = _mk(g, K, M, dt, 0, off), b
        nb = lib.tg_gemm_wgrad_workspace(code, M, N, K, 0)
        ws = torch.full((nb,), 0x5a, device="cuda", dtype=torch.uint8)
        assert lib.tg_gemm_wgrad(code, M, N, K, x.data_ptr(), M, gr.data_ptr(), N, f32,
                                 c.data_ptr(), N, 0, 0, None, 0, ws.data_ptr(), nb, s) == 0
        _bound(c, x.t(), gr, f"wgrad off {off}")
        assert bool((ws == 0x5a).all()) == (off == 1)
    # k-contiguous rows of 2^23 elements
    even, odd = (lib.tg_matmul_workspace(code, 0, 1, 64, 64, 2 ** 23 + i) for i in (0, 1))
    assert even == odd


@pytest.mark.parametrize("cols", [3, 9, 15, 17, 23, 25, 31, 39, 1001])
def test_ragged_rows_are_copied_exactly(cuda, cols):
    """Odd rows at every offset from 16 bytes: first, inner and last chunks of a row.  Operands
    of whole numbers, so each sum is exact; the last column ends the buffer."""
    g = torch.Generator(device="cuda").manual_seed(cols)
    M, K = 3000, 200
    a = torch.randint(-2, 3, (M, K), generator=g, device="cuda").half()
    for off in range(8):
        buf = torch.randint(-2, 3, (K * cols + off,), generator=g, device="cuda").half()
        b = buf[off:].view(K, cols)
        c = L().matmul2d(a, b, out_dtype=torch.float32)
        assert torch.equal(c, a.float() @ b.float().clone())
        w = torch.empty(cols, M, device="cuda")
        L().wgrad(b, a.t().contiguous(), w, False)
        assert torch.equal(w, c.t())
