"""Softmax and LayerNorm over rows that do not start on 16 bytes (any column count, any base)
against float64, at the edges of a vector, a wavefront's and a block's rows, and of the register
kernels' width; what lies around the outputs stays as it was.  GPU only.

Tolerances: the kernels compute in fp32, so beside one rounding of the output (2^-11 fp16,
2^-8 bf16) a row sum of n terms in a tree of depth <= 40 is off by at most 40 * 2^-24 of its
sum of magnitudes; the gradients of a row, within its largest value, take three such sums
(2^-16), and gamma/beta gradients, sums over all rows in chains of at most rows / 4 + 40,
are held to 2^-14 of the sum of magnitudes."""
import pytest
import torch

from tensor_gpu_v2 import _lib as L

pytestmark = pytest.mark.gpu

EPS = {torch.float32: 2.0 ** -16, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}
SHAPES = [(5, 1), (9, 3), (3, 7), (130, 9), (65, 255), (33, 257), (40, 513), (21, 1881), (7, 2047),
          (6, 2049), (300, 311), (3, 8191), (3, 8193), (2, 16383), (2, 16385)]


def guarded(t, off):
    """t's values in a buffer of sevens, `off` elements from its start: (buffer, view)."""
    buf = torch.full((t.numel() + off + 64,), 7.0, device="cuda", dtype=t.dtype)
    v = buf[off:off + t.numel()].view(t.shape)
    v.copy_(t)
    return buf, v


def untouched(buf, off, n):
    assert bool((buf[:off] == 7).all()) and bool((buf[off + n:] == 7).all())


def near(got, ref, tol, what):
    scale = ref.abs().amax(dim=-1, keepdim=True)
    err = (got.double().cpu() - ref).abs()
    assert bool((err <= tol * scale + 1e-30).all()), (what, float((err / (scale + 1e-30)).max()))


@pytest.mark.parametrize("rows,cols", SHAPES)
@pytest.mark.parametrize("dt", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("off", [0, 1])
def test_rows_off_16_bytes(cuda, rows, cols, dt, off):
    lib, s = L.load(), L.stream_handle()
    code = L.dtype_code(torch.empty(0, dtype=dt))
    g = torch.Generator().manual_seed(rows * 7919 + cols)
    n = rows * cols
    x0, dy0, acc0 = (torch.randn(rows, cols, generator=g).to(dt) for _ in range(3))
    _, x = guarded(x0, off)
    _, dy = guarded(dy0, off)
    x64, dy64, acc64 = x0.double(), dy0.double(), acc0.double()
    eps = EPS[dt]

    yb, y = guarded(acc0, off)
    assert lib.tg_softmax_fwd(code, L.ptr(x), L.ptr(y), rows, cols, s) == 0
    near(y, torch.softmax(x64, -1), eps, "softmax")
    untouched(yb, off, n)
    y64 = y.double().cpu()
    sm = y64 * (dy64 - (dy64 * y64).sum(-1, keepdim=True))
    for acc in (0, 1):
        db, dx = guarded(acc0, off)
        assert lib.tg_softmax_bwd(code, L.ptr(y), L.ptr(dy), L.ptr(dx), rows, cols, acc, s) == 0
        # a near-one-hot row cancels: within the terms' size, not the result's
        tol = eps * (y64 * (dy64.abs() + (dy64 * y64).abs().sum(-1, keepdim=True))
                     + acc * acc64.abs()).amax(-1, keepdim=True) + 2.0 ** -24
        assert bool(((dx.double().cpu() - sm - acc * acc64).abs() <= 2 * tol).all())
        untouched(db, off, n)

    gamma, beta = torch.randn(cols, generator=g), torch.randn(cols, generator=g)
    gc, bc = gamma.cuda(), beta.cuda()
    mean, rstd = torch.empty(rows, device="cuda"), torch.empty(rows, device="cuda")
    yb, y = guarded(acc0, off)
    assert lib.tg_layernorm_fwd(code, L.ptr(x), L.ptr(gc), L.ptr(bc), L.ptr(y), L.ptr(mean),
                                L.ptr(rstd), rows, cols, 1e-5, s) == 0
    mu = x64.mean(-1, keepdim=True)
    rs = 1 / torch.sqrt(((x64 - mu) ** 2).mean(-1, keepdim=True) + 1e-5)
    xh = (x64 - mu) * rs
    near(y, gamma.double() * xh + beta.double(), eps, "layernorm")
    untouched(yb, off, n)
    gg = dy64 * gamma.double()
    ref = rs * (gg - gg.mean(-1, keepdim=True) - xh * (gg * xh).mean(-1, keepdim=True))
    size = rs * (gg.abs() + gg.abs().mean(-1, keepdim=True)
                 + xh.abs() * (gg * xh).abs().mean(-1, keepdim=True))
    for acc in (0, 1):
        db, dx = guarded(acc0, off)
        dg, dbeta = torch.empty(cols, device="cuda"), torch.empty(cols, device="cuda")
        nb = lib.tg_layernorm_bwd_workspace(code, rows, cols)
        wb, ws = guarded(torch.zeros(nb // 4), 0)
        assert lib.tg_layernorm_bwd(code, L.ptr(x), L.ptr(mean), L.ptr(rstd), L.ptr(gc), L.ptr(dy),
                                    L.ptr(dx), L.ptr(dg), L.ptr(dbeta), rows, cols, acc, 0,
                                    L.ptr(ws), nb, s) == 0
        tol = eps * (size + acc * acc64.abs()).amax(-1, keepdim=True)
        assert bool(((dx.double().cpu() - ref - acc * acc64).abs() <= tol).all())
        untouched(db, off, n)
        untouched(wb, 0, nb // 4)
        for got, t in ((dg, dy64 * xh), (dbeta, dy64)):
            tol = 2.0 ** -14 * t.abs().sum(0) + 2.0 ** -20 * dy64.abs().sum(0)
            assert bool(((got.double().cpu() - t.sum(0)).abs() <= tol).all())
