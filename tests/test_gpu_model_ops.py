"""GPU tests of the engine's fused row kernels (mkv_rmsnorm, mkv_silu_mul)
against float64 references of LayerNorm.rms_forward / residual_rms_forward
(layernorm.py:16-33) and SiluAndMul (activation.py:16-19).

The kernels compute in fp32 and round once, so the bound is half an ulp of
the output dtype at the reference value plus a 2e-6 relative margin for the
fp32 arithmetic; the updated residual (x + residual rounded to the dtype) is
bit-exact against torch's own add."""
from __future__ import annotations

import pytest
import torch

from conftest import announce
from mkv import _lib
from mkv import engine as E

pytestmark = pytest.mark.gpu

MANT = {torch.float32: 24, torch.bfloat16: 8, torch.float16: 11}
EMIN = {torch.float32: -126, torch.bfloat16: -126, torch.float16: -14}  # below: subnormal spacing


def _check(got, want, dtype):
    got, want = got.double().cpu(), want.double().cpu()
    e = torch.floor(torch.log2(want.abs().clamp(min=2.0 ** -149))).clamp(min=EMIN[dtype])
    tol = 0.5 * torch.exp2(e - (MANT[dtype] - 1)) + 2e-6 * want.abs() + 1e-30
    # (a NaN difference fails unless both sides are NaN; `> tol` alone passes it)
    bad = ~((got - want).abs() <= tol) & ~(torch.isnan(got) & torch.isnan(want))
    assert not bool(bad.any()), f"{int(bad.sum())} elements off; max err {float((got - want).abs().max()):.3e}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,hidden", [(1, 1024), (64, 1024), (1000, 1024), (7, 2048), (33, 520)])
@pytest.mark.parametrize("with_residual", [False, True])
def test_rmsnorm(dev, dtype, rows, hidden, with_residual):
    announce(f"rmsnorm {dtype} {rows}x{hidden} residual={with_residual}")
    g = torch.Generator().manual_seed(rows + hidden)
    x = (torch.randn(rows, hidden, generator=g) * 3).to(dtype)
    w = (1 + 0.5 * torch.randn(hidden, generator=g)).to(dtype)
    r = torch.randn(rows, hidden, generator=g).to(dtype) if with_residual else None
    xd, wd = x.to(dev), w.to(dev)
    rd = r.to(dev) if with_residual else None
    out = E.rms_norm(xd, wd, 1e-5, rd)
    h = (x + r) if with_residual else x  # torch's add: fp32 then one rounding
    if with_residual:
        assert torch.equal(rd.cpu(), h)
    hd = h.double()
    want = hd * w.double() / torch.sqrt(hd.pow(2).mean(-1, keepdim=True) + 1e-5)
    _check(out, want, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,inter", [(1, 3072), (64, 3072), (1024, 3072), (5, 24)])
def test_silu_mul(dev, dtype, rows, inter):
    announce(f"silu_mul {dtype} {rows}x{inter}")
    g = torch.Generator().manual_seed(rows + inter)
    x = (torch.randn(rows, 2 * inter, generator=g) * 4).to(dtype)
    x[0, :4] = torch.tensor([-100.0, 100.0, 0.0, -0.0]).to(dtype)
    out = E.silu_and_mul(x.to(dev))
    a, b = x[:, :inter].double(), x[:, inter:].double()
    _check(out, a / (1 + torch.exp(-a)) * b, dtype)


def test_silu_mul_strided_rows(dev):
    announce("silu_mul on a strided row view")
    g = torch.Generator().manual_seed(3)
    big = torch.randn(16, 2 * 64 + 32, generator=g).to(torch.bfloat16).to(dev)
    x = big[:, :128]
    out = E.silu_and_mul(x)
    a, b = x[:, :64].double().cpu(), x[:, 64:].double().cpu()
    _check(out, a / (1 + torch.exp(-a)) * b, torch.bfloat16)


def _ulp(x):
    return torch.exp2(torch.floor(torch.log2(x.abs().clamp(min=2.0 ** -126))) - 7)  # bf16


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 33, 60, 64])
@pytest.mark.parametrize("n,k", [(16, 512), (48, 768), (4096, 1024), (1024, 2048), (112, 3072), (80, 4096), (48, 1536), (65584, 1024)])
@pytest.mark.parametrize("strided", [False, True])
def test_linear(dev, rows, n, k, strided):
    """mkv_linear in every form (4, 8 and 16 waves, 4 and 6 k-steps, one or
    two loads of k, 16 to 64 rows a workgroup, streaming), with rows and
    feature tiles that do not fill them.  Bound: half an ulp of the output
    and k fp32 roundings of the sum of |x| |w|."""
    announce(f"linear {rows} x {n} x {k} strided={strided}")
    assert _lib.query("mkv_linear_supported", rows, n, k, 0, 0, _lib.DTYPE_BF16) == (n < 32768 or rows > 16)
    g = torch.Generator().manual_seed(rows * 7 + n)
    w = torch.randn(n, k, generator=g).bfloat16().to(dev)
    x = torch.randn(rows, k + 8, generator=g).bfloat16().to(dev)
    x = x[:, :k] if strided else x[:, :k].contiguous()
    got = E.linear(x, w).double()
    want, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert bool(((got - want).abs() <= 0.5 * _ulp(want) + k * 2.0 ** -24 * mag).all())


@pytest.mark.parametrize("rows", [1, 17, 60])
@pytest.mark.parametrize("inter,k", [(16, 512), (3072, 1024), (48, 3072)])
def test_gated_linear(dev, rows, inter, k):
    """The gated product against silu(gate) * up in 64 bits.  Bound: gate and
    up are rounded to bf16 (half an ulp each, silu's slope at most 1.1) and
    so is the result, plus the products' fp32 sums.  The result's ulp is that
    of what is rounded: of 64-bit 3.9955, 4.016 may be, half of 4's ulp away
    (torch's product and mkv_silu_mul give the same value there)."""
    announce(f"gated linear {rows} x {inter} x {k}")
    assert _lib.query("mkv_linear_supported", rows, inter, k, 1, 0, _lib.DTYPE_BF16)
    g = torch.Generator().manual_seed(rows + inter)
    w = (torch.randn(2 * inter, k, generator=g) * 2 / k ** 0.5).bfloat16().to(dev)
    x = torch.randn(rows, k, generator=g).bfloat16().to(dev)
    got = E.gated_linear(x, w).double()
    p, mag = x.double() @ w.double().t(), k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    e = 0.5 * _ulp(p) * 1.01 + mag
    gate, up = p.chunk(2, -1)
    eg, eu = e.chunk(2, -1)
    silu = torch.nn.functional.silu(gate)
    want = silu * up
    bound = 1.1 * eg * (up.abs() + eu) + silu.abs() * eu + 1e-6 * want.abs()
    bound = bound + 0.5 * _ulp(want.abs() + bound) * 1.01
    assert bool(((got - want).abs() <= bound).all())


@pytest.mark.parametrize("rows", [1, 17, 60])
@pytest.mark.parametrize("n,k,act", [(16, 512, 0), (4096, 1024, 0), (48, 1536, 0), (32, 2048, 0), (48, 768, 1), (1024, 1024, 1)])
def test_linear_with_norm(dev, rows, n, k, act):
    """The product of normalised rows against the same of the norm kernel's
    rows: equal, but for the order of the sum of squares, which moves 1 / rms
    by 1e-6 at most and a term by one ulp (2^-8) where its rounding was that
    nearly a tie, one in 10^3 of them.  Bound: 8 such terms, and an ulp of gate
    and up and of the result."""
    announce(f"linear with norm {rows} x {n} x {k} act {act}")
    assert _lib.query("mkv_linear_supported", rows, n, k, act, 1, _lib.DTYPE_BF16)
    g = torch.Generator().manual_seed(rows + n + k)
    w = (torch.randn((1 + act) * n, k, generator=g) * 2 / k ** 0.5).bfloat16().to(dev)
    x = (torch.randn(rows, k, generator=g) * torch.exp2(torch.randn(rows, 1, generator=g) * 3)).bfloat16().to(dev)
    nw = (1 + 0.5 * torch.randn(k, generator=g)).bfloat16().to(dev)
    got = E._product(x, w, n, act, nw, 1e-5).double()
    h = E.rms_norm(x, nw, 1e-5)
    want = (E.gated_linear if act else E.linear)(h, w).double()
    p = h.double() @ w.double().t()
    term = (h.double().abs().amax(-1, keepdim=True) * w.double().abs().amax(-1)) * 2.0 ** -8
    e = 8 * term + _ulp(p)
    if act:
        (gate, up), (eg, eu) = p.chunk(2, -1), e.chunk(2, -1)
        e = 1.1 * eg * (up.abs() + eu) + torch.nn.functional.silu(gate).abs() * eu
    assert bool(((got - want).abs() <= e + _ulp(want)).all())
    # the rows of the norm are the same but for those ties: 16 features pick
    # out one element each
    if not act and n == 16:
        pick = torch.zeros(n, k).bfloat16().to(dev)
        pick[torch.arange(n), torch.arange(n) * (k // n)] = 1
        a, b = E._product(x, pick, n, 0, nw, 1e-5), h[:, :: k // n]
        assert float((a != b).float().mean()) <= 0.02 and bool(((a - b).abs() <= 2.0 ** -7 * b.abs()).all())


@pytest.mark.parametrize("rows", [1, 17, 60])
@pytest.mark.parametrize("n,k", [(16, 512), (1024, 2048), (1024, 3072), (4096, 1024)])
def test_linear_with_residual(dev, rows, n, k):
    """The residual added in place equals the product alone added by torch."""
    announce(f"linear with residual {rows} x {n} x {k}")
    g = torch.Generator().manual_seed(rows + n)
    w = torch.randn(n, k, generator=g).bfloat16().to(dev)
    x = torch.randn(rows, k, generator=g).bfloat16().to(dev)
    res = (20 * torch.randn(rows, n, generator=g)).bfloat16().to(dev)
    want = E.linear(x, w) + res
    got = E._product(x, w, n, residual=res)
    assert got is res and torch.equal(got, want)


def test_model_layers_with_and_without_fused_products(dev, monkeypatch):
    """A model whose layers partly run on mkv_linear (a transposed weight is
    left to torch) gives the hidden states of one that runs on torch alone,
    to the bf16 rounding of each step (2^-8 over the 2 x 3 norms and sums)."""
    from mkv import context as C
    cfg = E.ModelConfig(vocab_size=512, hidden_size=1024, num_layers=3, intermediate_size=3072, max_position=64)
    model = E.Qwen3Model(cfg, dev, block_size=16)
    model.attach_kv_cache(8, "auto")
    model.layers[1]["down"] = model.layers[1]["down"].t().contiguous().t()
    ids = torch.arange(5, device=dev)
    slots = torch.arange(5, device=dev) * 16
    bt = torch.arange(5, dtype=torch.int32, device=dev)[:, None].contiguous()
    calls = []

    def run():
        C.set_context(False, slot_mapping=slots, context_lens=torch.ones(5, dtype=torch.int64, device=dev),
                      block_tables=bt)
        try:
            return model(ids, torch.zeros(5, dtype=torch.int64, device=dev), slots).double()
        finally:
            C.reset_context()

    real = _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    got = run()
    assert calls.count("mkv_linear") == 4 + 3 + 4  # (layer 1: qkv, o and the gated product, each by itself)
    monkeypatch.setattr(E, "_own_weight", lambda *a: False)
    want = run()
    assert calls.count("mkv_linear") == 11
    err = float((got - want).norm() / want.norm())
    print("relative difference", err)
    assert err < 6 * 2.0 ** -8


@pytest.mark.parametrize("rows", [17, 40, 60])
@pytest.mark.parametrize("n,k", [(32816, 512), (65552, 1536), (65568, 2048)])
def test_linear_streaming_widths(dev, rows, n, k):
    """The streaming form's other widths (2, 6 and 8 k-steps a wave, pairs of
    feature tiles and single ones), with ranges of tiles that differ by one."""
    test_linear(dev, rows, n, k, rows % 2 == 1)


# Sizes in the forms that the tests above leave out: k in 4, 8 and 16 parts of
# 4 or 6 steps, 32 and 64 rows a workgroup, at few and many features.
_WIDE = [(64, 2048, 2048), (33, 2048, 2048), (17, 4096, 2048), (33, 2048, 512), (31, 16384, 512), (64, 2048, 768),
         (17, 4112, 768), (48, 2048, 1536), (32, 4096, 1536), (64, 4096, 512), (33, 10752, 512), (48, 4096, 1024)]


@pytest.mark.parametrize("rows,n,k", _WIDE)
def test_linear_wide_forms(dev, rows, n, k):
    test_linear(dev, rows, n, k, True)


@pytest.mark.parametrize("rows,n,k", _WIDE + [(1, 16, 2048), (16, 32, 4096), (1, 16, 768), (16, 32, 1536)])
def test_gated_linear_wide_forms(dev, rows, n, k):
    test_gated_linear(dev, rows, n, k)


@pytest.mark.parametrize("act,rows,n,k", [(0, *s) for s in _WIDE + [(1, 16, 768)]] +
                         [(1, *s) for s in _WIDE + [(1, 16, 2048), (1, 16, 512), (1, 16, 1536),
                                                    (33, 3072, 1024), (60, 3072, 1024), (64, 3072, 1024)]])
def test_linear_with_norm_wide_forms(dev, act, rows, n, k):
    test_linear_with_norm(dev, rows, n, k, act)


def test_model_takes_any_attention_rows(dev):
    """The output of an overridden attention() may lie anyhow (every other
    element of a wider buffer, transposed, off 16-byte alignment): the hidden
    states are those of contiguous rows, to the bf16 rounding of each step (as
    below).  Rows of another width than the output weight's, and a norm weight
    at an odd address, give the errors that torch's product and the norm
    kernel give, ahead of any product over them."""
    from mkv import context as C
    announce("model with attention rows in other layouts")
    cfg = E.ModelConfig(vocab_size=512, hidden_size=1024, num_layers=2, intermediate_size=3072, max_position=64)

    class Model(E.Qwen3Model):
        fuse_decode_step = False
        lay_out = staticmethod(lambda o: o)

        def attention(self, li, q, k, v):
            return self.lay_out(super().attention(li, q, k, v))

    model = Model(cfg, dev, block_size=16)
    model.attach_kv_cache(8, "auto")
    ids, slots = torch.arange(5, device=dev), torch.arange(5, device=dev) * 16
    bt = torch.arange(5, dtype=torch.int32, device=dev)[:, None].contiguous()

    def run(lay_out):
        model.lay_out = lay_out
        C.set_context(False, slot_mapping=slots, context_lens=torch.ones(5, dtype=torch.int64, device=dev),
                      block_tables=bt)
        try:
            return model(ids, torch.zeros(5, dtype=torch.int64, device=dev), slots).double()
        finally:
            C.reset_context()

    def spread(o):
        wide = torch.full((o.shape[0], 2 * o.shape[1]), 7.0, dtype=o.dtype, device=dev)
        wide[:, ::2] = o
        return wide[:, ::2]

    def off(o):
        buf = torch.zeros(o.shape[0], o.shape[1] + 8, dtype=o.dtype, device=dev)
        buf[:, 1:o.shape[1] + 1] = o
        return buf[:, 1:o.shape[1] + 1]

    want = run(lambda o: o)
    for lay_out in (spread, lambda o: o.t().contiguous().t(), off):
        got = run(lay_out)
        assert float((got - want).norm() / want.norm()) < 4 * 2.0 ** -8
    for width in (1024, 4096):
        with pytest.raises(RuntimeError):
            run(lambda o: torch.zeros(5, width, dtype=o.dtype, device=dev))
    buf = torch.ones(1032, dtype=torch.bfloat16, device=dev)
    model.layers[0]["post_norm"] = buf[1:1025]
    with pytest.raises(_lib.MkvError, match="mkv_rmsnorm"):
        run(lambda o: o)


def test_logits_keep_transforms_and_the_current_device(dev, monkeypatch):
    """The LM head under forward mode and vmap gives torch's tangent and
    rows, and where another device is the current one torch's product."""
    from torch.autograd import forward_ad
    announce("logits under jvp, vmap and another current device")
    cfg = E.ModelConfig(vocab_size=512, hidden_size=1024, num_layers=1, intermediate_size=512, max_position=64)
    model = E.Qwen3Model(cfg, dev, block_size=16)
    g = torch.Generator().manual_seed(5)
    x, t = (torch.randn(20, 1024, generator=g).bfloat16().to(dev) for _ in range(2))
    calls = []
    real = _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    torch_rows = torch.nn.functional.linear(x, model.embed)
    with forward_ad.dual_level():
        y = forward_ad.unpack_dual(model.logits(forward_ad.make_dual(x, t)))
        assert torch.equal(y.primal, torch_rows)
        assert torch.equal(y.tangent, torch.nn.functional.linear(t, model.embed))
    rows = torch.func.vmap(model.logits)(x.view(4, 5, 1024)).view(20, 512)
    assert float((rows.double() - torch_rows.double()).norm() / torch_rows.double().norm()) < 2.0 ** -8
    with monkeypatch.context() as m:
        m.setattr(torch.cuda, "current_device", lambda: 1 + dev.index if dev.index is not None else 1)
        assert torch.equal(model.logits(x), torch_rows)
    assert calls == []
    model.logits(x)
    assert calls == ["mkv_linear"]


def test_linear_leaves_other_products_to_torch(dev):
    """Sizes, types and layouts that mkv_linear does not take give torch's
    product: many rows, fp16, a transposed weight, a gradient to record."""
    g = torch.Generator().manual_seed(3)
    w = torch.randn(64, 1024, generator=g).to(dev)
    x = torch.randn(65, 1024, generator=g).to(dev)
    wb, xb = w.bfloat16(), x.bfloat16()
    wt = w.t().contiguous().bfloat16().t()
    assert not any(_lib.query("mkv_linear_supported", m, n, k, 0, 0, _lib.DTYPE_BF16)
                   for m, n, k in ((65, 64, 1024), (64, 6144, 1024), (16, 2048, 6144), (8, 2560, 2560),
                                   (1, 24, 1024), (1, 16, 16), (0, 16, 1024)))
    for a, b in ((xb, wb), (x[:8].half(), w.half()), (x[:8], w), (xb[:8], wt), (xb[:8, :40], wb[:, :40].contiguous())):
        assert torch.equal(E.linear(a, b), torch.nn.functional.linear(a, b))
    wr = wb.clone().requires_grad_(True)
    E.linear(xb[:8], wr).float().sum().backward()
    assert wr.grad is not None
