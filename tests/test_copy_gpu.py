"""The same-dtype copy of tg_axpbyz / tg_axpby (alpha 1, beta 0): bit for bit x at the edges of
a 16-byte vector, of a block and of the non-temporal range, and at bases off 16 bytes, which
take the other kernels.  The buffer's bytes past the output stay as they were.  GPU only."""
import pytest
import torch

from tensor_gpu_v2 import _lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 3, 7, 8, 9, 2047, 2048, 4099, (128 << 20) // 4 - 1,
                               (128 << 20) // 2 + 5])
@pytest.mark.parametrize("off", [0, 1])
def test_copy_bits(cuda, dt, n, off):
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n + off + 32, device="cuda", generator=g).to(dt)
    x[off] = float("inf")
    x[off + n - 1] = -0.0
    for inplace in (False, True):
        buf = torch.full((n + off + 32,), 7.0, device="cuda", dtype=dt)
        src, out = x[off:off + n], buf[off:off + n]
        if inplace:
            L.axpby(src, out, 1.0, 0.0)
        else:
            L.axpbyz(src, src, 1.0, 0.0, out=out)
        bits = torch.int32 if dt == torch.float32 else torch.int16
        assert torch.equal(out.view(bits), src.view(bits))
        assert bool((buf[:off] == 7).all()) and bool((buf[off + n:] == 7).all())
