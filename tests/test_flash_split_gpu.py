"""FlashAttention on the split-operand kernels (fp32; fp16 / bf16 head dims other than 64 and
128) against float64, at the edges of their tiles, head dims and layouts, and fp32 values
outside the split's range."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DT = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def L():
    from tensor_gpu_v2 import _lib
    return _lib


def _ref(q, k, v, do, scale, causal):
    q, k, v = (t.double().detach().requires_grad_(True) for t in (q, k, v))
    s = (q * scale) @ k.transpose(-1, -2).contiguous()
    if causal:
        m = torch.triu(torch.ones(s.shape[-2:], dtype=torch.bool, device="cuda"), 1)
        s = s.masked_fill(m, -float("inf"))
    o = torch.softmax(s, -1) @ v
    return [o.detach()] + list(torch.autograd.grad(o, (q, k, v), do.double()))


def _close(got, want, dt, what, extra=1.0):
    """2-norm: fp32 sums of up to 2^11 terms and exponentials of O(10) arguments, a few
    2^-24 each; 16-bit results are rounded once (and o, which D is formed from, too)."""
    lim = {torch.float32: 3e-6, torch.float16: 1e-3, torch.bfloat16: 8e-3}[dt] * extra
    e = float((got.double() - want).norm() / want.norm().clamp_min(1e-30))
    assert e < lim, f"{what}: {e:.2e}"


@pytest.mark.parametrize("dt", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("D", [1, 8, 20, 32, 33, 64, 72, 80, 96, 100, 128])
@pytest.mark.parametrize("Sq,Sk,causal", [(1, 1, False), (33, 33, True), (128, 128, True),
                                          (65, 200, False), (300, 31, False), (257, 257, True)])
def test_split_attention(cuda, D, Sq, Sk, causal, dt):
    dt = DT[dt]
    g = torch.Generator(device="cuda").manual_seed(D * 1000 + Sq + Sk)
    for layout in (0, 1):
        def mk(S):
            if layout == 0:
                return torch.randn(2, 3, S, D, generator=g, device="cuda").to(dt)
            return torch.randn(2, S, 3, D, generator=g, device="cuda").to(dt).permute(0, 2, 1, 3)
        q, k, v, do = mk(Sq), mk(Sk), mk(Sk), mk(Sq)
        sc = D ** -0.5
        o, lse = L().flash_attn_fwd(q, k, v, sc, causal, layout)
        grads = [L().fa_empty(2, 3, S, D, dt, q.device, layout) for S in (Sq, Sk, Sk)]
        for t in grads:
            t.fill_(0.5)
        L().flash_attn_bwd(q, k, v, o, do, lse, *grads, sc, causal, True, layout)
        want = _ref(q, k, v, do, sc, causal)
        _close(o, want[0], dt, "o")
        for t, w, n in zip(grads, want[1:], ("dq", "dk", "dv")):
            if float(w.norm()) > 1e-9:  # (one key: dq and dk are zero)
                _close(t, w + 0.5, dt, n, 2.0)


@pytest.mark.parametrize("dt", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("D", [32, 80])
def test_split_attention_packed(cuda, D, dt):
    dt = DT[dt]
    B, S, H = 2, 190, 4
    g = torch.Generator(device="cuda").manual_seed(D)
    qkv = torch.randn(B, S, 3 * H * D, generator=g, device="cuda").to(dt)
    do = torch.randn(B, S, H * D, generator=g, device="cuda").to(dt)
    o, lse = L().flash_attn_fwd_qkv(qkv, H, D ** -0.5, True)
    d = torch.empty_like(qkv)
    L().flash_attn_bwd_qkv(qkv, o, do, lse, d, H, D ** -0.5, True, False)
    q, k, v = (t.permute(0, 2, 1, 3) for t in qkv.reshape(B, S, 3, H, D).unbind(2))
    want = _ref(q, k, v, do.reshape(B, S, H, D).permute(0, 2, 1, 3), D ** -0.5, True)
    back = [t.permute(0, 2, 1, 3).reshape(B, S, H * D) for t in want]
    _close(o, back[0], dt, "o")
    _close(d, torch.cat(back[1:], -1), dt, "dqkv", 2.0)


@pytest.mark.parametrize("D", [24, 64, 128])
@pytest.mark.parametrize("kind", ["tiny", "huge", "negative_scale", "large_scores", "inf"])
def test_split_attention_fp32_extremes(cuda, D, kind):
    """Operands that the bf16 split cannot hold run on the fp32 matrix cores."""
    g = torch.Generator(device="cuda").manual_seed(5)
    mk = lambda: torch.randn(1, 2, 150, D, generator=g, device="cuda")  # noqa: E731
    q, k, v, do = mk(), mk(), mk(), mk()
    sc = D ** -0.5
    if kind == "tiny":
        v *= 1e-34
        do[0, 0, 3] *= 1e-33
    elif kind == "huge":
        v[0, 1, 7] *= 1e38
        do *= 1e-10
    elif kind == "negative_scale":
        sc = -0.4
    elif kind == "large_scores":
        q *= 40.0
        k -= 3.0
    elif kind == "inf":
        v[0, 0, 11, 2] = float("inf")
    o, lse = L().flash_attn_fwd(q, k, v, sc, False)
    want = _ref(q, k, v, do, sc, False)
    if kind == "inf":
        assert torch.equal(torch.isfinite(o), torch.isfinite(want[0]))
        return
    if kind == "huge":
        assert torch.equal(torch.isfinite(o), torch.isfinite(want[0].float()))
    ok = torch.isfinite(want[0].float())
    _close(o[ok], want[0][ok], torch.float32, "o", 200.0 if kind == "large_scores" else 2.0)
    grads = [torch.empty_like(q) for _ in range(3)]
    L().flash_attn_bwd(q, k, v, o, do, lse, *grads, sc, False, False)
    # (large_scores: scores of up to 10^3 are off by 2^-24 of themselves and more, and P by
    # as much relative to itself)
    for t, w, n in zip(grads, want[1:], ("dq", "dk", "dv")):
        ok = torch.isfinite(w.float())
        assert torch.equal(torch.isfinite(t), ok), n
        _close(t[ok], w[ok], torch.float32, n, 200.0 if kind == "large_scores" else 10.0)


@pytest.mark.parametrize("D", [24, 64, 128])
@pytest.mark.parametrize("S,causal", [(150, False), (257, True)])
def test_split_attention_fp32_subnormal_columns(cuda, D, S, causal):
    """Columns of subnormal operands (their bf16 rounding is zero) beside ordinary ones: each
    result column that is formed from one keeps its value, to the rounding of subnormals (a
    multiple of 2^-149 each, about 1e-3 of these results)."""
    g = torch.Generator(device="cuda").manual_seed(D)
    q, k, v, do = (torch.randn(1, 2, S, D, generator=g, device="cuda") for _ in range(4))
    for t, c in ((q, 1), (k, 2), (v, 3), (do, 4)):
        t[..., c] *= 1e-41
    sc = D ** -0.5
    o, lse = L().flash_attn_fwd(q, k, v, sc, causal)
    grads = [torch.empty_like(q) for _ in range(3)]
    L().flash_attn_bwd(q, k, v, o, do, lse, *grads, sc, causal, False)
    want = _ref(q, k, v, do, sc, causal)
    for t, w, c, n in zip([o] + grads, want, (3, 2, 1, 4), ("o", "dq", "dk", "dv")):
        _close(t, w, torch.float32, n, 2.0)
        a, b = t[..., c].double() * 1e41, w[..., c] * 1e41
        assert float((a - b).norm() / b.norm()) < 2e-2, n


@pytest.mark.parametrize("D", [32, 64, 80, 128])
@pytest.mark.parametrize("S,causal,offset", [(2048, False, False), (4096, False, False),
                                             (4096, False, True), (2011, True, False)])
def test_split_attention_fp32_column_sums(cuda, D, S, causal, offset):
    """Entries that err to either side at random (up to 1.2e-6 of their size here, as on the
    fp32 matrix cores) leave 1/sqrt(S) of that in a column sum relative to S entries; held to
    twice it.  Sums that err downwards leave 1e-7 at S = 2048 and 2e-7 at 4096."""
    g = torch.Generator(device="cuda").manual_seed(S + D)
    q, k, v, do = (torch.randn(1, 3, S, D, generator=g, device="cuda") for _ in range(4))
    if offset:
        v += 3
    sc = D ** -0.5
    o, lse = L().flash_attn_fwd(q, k, v, sc, causal)
    grads = [torch.empty_like(q) for _ in range(3)]
    L().flash_attn_bwd(q, k, v, o, do, lse, *grads, sc, causal, False)
    want = _ref(q, k, v, do, sc, causal)
    for t, w, n in zip([o] + grads[:2], want, ("o", "dq", "dk")):
        if offset and n != "o":  # (dP - D cancels: the entries themselves are further off)
            continue
        d = (t.double() - w).sum(2)
        e = float(d.norm() / (w.norm(dim=2) * S ** 0.5).norm())
        assert e < 2 * 1.2e-6 / S ** 0.5, f"{n}: {e:.2e}"


@pytest.mark.parametrize("D", [64, 128])
def test_split_attention_fp32_probabilities_add_up(cuda, D):
    """With dO = 1, the column sums of dV are the sums of the probabilities: S, up to v_exp_f32's
    error, which a stale maximum in the forward (arguments of either sign) adds to."""
    S = 4096
    g = torch.Generator(device="cuda").manual_seed(D)
    q, k, v = (torch.randn(1, 3, S, D, generator=g, device="cuda") for _ in range(3))
    do = torch.ones_like(q)
    o, lse = L().flash_attn_fwd(q, k, v, D ** -0.5, False)
    grads = [torch.empty_like(q) for _ in range(3)]
    L().flash_attn_bwd(q, k, v, o, do, lse, *grads, D ** -0.5, False, False)
    assert abs(float(grads[2].double().sum(2).mean()) / S - 1) < 2.5e-7


@pytest.mark.parametrize("dt", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("D", [32, 80, 128])
@pytest.mark.parametrize("where", ["v", "do", "q"])
@pytest.mark.parametrize("value", [float("inf"), -float("inf"), float("nan")])
def test_split_attention_non_finite(cuda, D, dt, where, value):
    """Infinities stay infinities, of their sign, and NaN spreads no further than by the
    formulas.  Misaligned (by one element): head dim 128 would run on the tuned kernels."""
    dt = DT[dt]
    g = torch.Generator(device="cuda").manual_seed(D)
    S = 150

    def mk():
        buf = torch.randn(1 * 2 * S * D + 1, generator=g, device="cuda").to(dt)
        return buf[1:].view(1, 2, S, D)
    q, k, v, do = mk(), mk(), mk(), mk()
    {"q": q, "v": v, "do": do}[where][0, 0, 11, 2] = value
    sc = 0.5 * D ** -0.5
    o, lse = L().flash_attn_fwd(q, k, v, sc, False)
    grads = [mk() for _ in range(3)]
    L().flash_attn_bwd(q, k, v, o, do, lse, *grads, sc, False, False)
    want = _ref(q, k, v, do, sc, False)
    for t, w, n in zip([o] + grads, want, ("o", "dq", "dk", "dv")):
        assert torch.equal(torch.isfinite(t), torch.isfinite(w)), n
        # (dS = P (dP - D) is Inf - Inf or not by the order of D's sum, P of a row of infinite
        # scores Inf or NaN by the form of its lse)
        if n == "o" or (n == "dv" and where != "q"):
            assert torch.equal(torch.isnan(t), torch.isnan(w)), n
            inf = torch.isinf(w)
            assert torch.equal(t[inf].double(), w[inf]), n
        ok = torch.isfinite(w)
        if bool(ok.any()):
            _close(t[ok], w[ok], dt, n, 2.0)


@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("D", [32, 80, 96, 100])
@pytest.mark.parametrize("S,causal", [(200, False), (1024, True), (3001, False)])
def test_split_attention_16bit_keeps_fp32_probabilities(cuda, D, S, causal, dt):
    """o and dV (formed with P) are the rounded float64 results but for a small share: an error
    of e moves an element's rounding to 11 bits (8 bits) with probability e / 2^-11 (2^-8) or
    so.  Here e is 2^-21 of the scores and exponentials in fp32, and 2^-25 for each of the S / 16
    steps of the sum, adding up at random; held to six times that.  P in 16 bits moves 2 %
    (0.2 to 0.3 %)."""
    dt = DT[dt]
    g = torch.Generator(device="cuda").manual_seed(D + S)
    q, k, v, do = (torch.randn(2, 4, S, D, generator=g, device="cuda").to(dt) for _ in range(4))
    sc = D ** -0.5
    o, lse = L().flash_attn_fwd(q, k, v, sc, causal)
    grads = [torch.empty_like(q) for _ in range(3)]
    L().flash_attn_bwd(q, k, v, o, do, lse, *grads, sc, causal, False)
    want = _ref(q, k, v, do, sc, causal)
    most = 6 * (2.0 ** -21 + 2.0 ** -25 * (S / 16) ** 0.5) * 2.0 ** (
        11 if dt == torch.float16 else 8)
    for t, w, n in ((o, want[0], "o"), (grads[2], want[3], "dv")):
        share = float((t != w.to(dt)).double().mean())
        assert share < most, f"{n}: {share:.2e}"
