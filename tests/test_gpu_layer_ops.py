"""Fused layer kernels against float64 restatements, and the routes that must stay on torch ops."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from conftest import announce

pytestmark = pytest.mark.gpu

# Unit roundoff of each dtype: an output that passes n roundings is within n * U of the 64-bit value.
U = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
TINY = 2.0 ** -24  # fp16 subnormal grid (absolute), far below everything else


def norm64(s, w, eps):
    s = s.double()
    return w.double() * s * torch.rsqrt(s.square().mean(-1, keepdim=True) + eps)


# Row lengths at every edge of the kernel's (wavefronts per row, chunks per lane) choices, in 16-byte
# chunks: 1, 63, 112 (0.5B), 128 | 129, 256 | 257, 448 (7B), 512 | 513, 1024 | 1025, 2048.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("chunks", [1, 63, 112, 128, 129, 256, 257, 448, 512, 513, 1024, 1025, 2048])
def test_add_rms_norm(gpu, dtype, chunks):
    from engine import layer_ops

    dim = chunks * 128 // torch.finfo(dtype).bits
    for rows in (1, 3, 4, 517):
        announce(f"add_rms_norm {dtype} rows {rows} dim {dim}")
        gen = torch.Generator(device=gpu).manual_seed(rows + dim)
        x = torch.randn(2, rows, dim, generator=gen, device=gpu).to(dtype)[1]
        d = torch.randn(rows, dim, generator=gen, device=gpu).to(dtype)
        w = (torch.rand(dim, generator=gen, device=gpu) + 0.5).to(dtype)
        assert layer_ops.norm_usable(w, x, d)
        s, h = layer_ops.add_rms_norm(x, d, w, 1e-6)
        assert torch.equal(s, x + d)
        only = layer_ops.rms_norm(x, w, 1e-6)
        # Two roundings (three for 32 bits, whose sum of dim squares is also within dim * U, in
        # practice far less: 64 lanes add dim / 64 terms each), and rsqrt's last bit.
        slack = 2.05 * U[dtype] + (dim / 64 + 16) * U[torch.float32]
        for got, src in ((h, s), (only, x)):
            want = norm64(src, w, 1e-6)
            assert ((got.double() - want).abs() <= slack * want.abs() + TINY).all()


def test_rms_norm_special_values(gpu):
    from engine import layer_ops

    announce("rms_norm with zero, infinite and NaN rows")
    x = torch.randn(4, 896, device=gpu).to(torch.bfloat16)
    x[0] = 0
    x[1, 5] = float("inf")
    x[2, 7] = float("nan")
    w = torch.ones(896, device=gpu, dtype=torch.bfloat16)
    got = layer_ops.rms_norm(x, w, 1e-6)
    xf = x.float()
    want = w * (xf * torch.rsqrt(xf.square().mean(-1, keepdim=True) + 1e-6)).to(x.dtype)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got[0], want[0]) and torch.equal(got[1].nan_to_num(7.0), want[1].nan_to_num(7.0))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,inter", [(1, 8), (3, 4864), (257, 264), (70, 18944)])
def test_silu_mul(gpu, dtype, rows, inter):
    from engine import layer_ops

    announce(f"silu_mul {dtype} rows {rows} inter {inter}")
    x = (4 * torch.randn(rows, 2 * inter, device=gpu)).to(dtype)
    x[0, :4] = torch.tensor([60.0, -60.0, 0.0, -20.0], device=gpu).to(dtype)
    assert layer_ops.silu_mul_usable(x)
    got = layer_ops.silu_mul(x)
    g, u = x.double().chunk(2, dim=-1)
    want = g * torch.sigmoid(g) * u
    # Two roundings, and a few fp32 roundings of exp, the sum and the quotient (exp's argument
    # rounding is exact, its result within 2 ulps).
    slack = 2.05 * U[dtype] + 8 * U[torch.float32]
    assert ((got.double() - want).abs() <= slack * want.abs() + TINY * (1 + u.abs())).all()


def test_routes_that_stay_on_torch(gpu):
    """Calls that something observes, and layouts the kernels do not take, keep the torch ops and their results."""
    from engine import layer_ops
    from engine.model import MLP, DecoderLayer, Qwen2Config, RMSNorm

    announce("layer ops routing")
    norm = RMSNorm(64, 1e-6).to(gpu)
    x = torch.randn(6, 64, device=gpu)
    with torch.no_grad():
        want = norm(x)
        assert layer_ops.norm_usable(norm.weight, x)
    # autograd: same value, gradients flow to x and the weight
    xg = x.clone().requires_grad_()
    assert not layer_ops.norm_usable(norm.weight, xg)
    y = norm(xg)
    y.square().sum().backward()
    assert xg.grad is not None and norm.weight.grad is not None
    torch.testing.assert_close(y.detach(), want, rtol=1e-6, atol=1e-6)
    with torch.no_grad():
        # torch.func transforms and forward-mode AD
        torch.testing.assert_close(torch.func.vmap(norm)(x), want, rtol=1e-6, atol=1e-6)
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
            assert not layer_ops.norm_usable(norm.weight, dual)
        # unaligned, strided, ragged and mixed-dtype operands
        odd = torch.randn(6 * 64 + 1, device=gpu)[1:].view(6, 64)
        assert not layer_ops.norm_usable(norm.weight, odd) and norm(odd).shape == odd.shape
        strided = torch.randn(64, 6, device=gpu).t()
        assert not layer_ops.norm_usable(norm.weight, strided)
        torch.testing.assert_close(norm(strided), norm(strided.contiguous()), rtol=1e-6, atol=1e-6)
        assert not layer_ops.norm_usable(norm.weight, x.to(torch.bfloat16))
        assert not layer_ops.norm_usable(norm.weight, x[:, :6])
        assert not layer_ops.norm_usable(norm.weight, x, x[:1])  # a delta that would broadcast
        assert norm(x[:0]).shape == (0, 64)
        assert not layer_ops.silu_mul_usable(torch.randn(3, 12, device=gpu))
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert not layer_ops.norm_usable(norm.weight, x)

    # A hook on the layer's second norm still sees its call.
    cfg = Qwen2Config(vocab_size=64, hidden_size=64, intermediate_size=128, num_layers=1, num_heads=2, num_kv_heads=1,
                      head_dim=32)
    layer = DecoderLayer(cfg, 0).to(gpu).requires_grad_(False)

    class Same:
        def attend(self, layer_idx, q, k, v):
            return q

    cs = torch.ones(1, 1, 5, 32, device=gpu)
    h = torch.randn(1, 5, 64, device=gpu)
    with torch.inference_mode():
        plain = layer(h, cs, cs * 0, Same())
        seen = []
        layer.post_attn_norm.register_forward_hook(lambda m, a, o: seen.append((a[0], o)))
        hooked = layer(h, cs, cs * 0, Same())
    assert len(seen) == 1 and seen[0][0].shape == h.shape
    torch.testing.assert_close(hooked, plain, rtol=1e-5, atol=1e-6)
    mlp = MLP(cfg).to(gpu)
    a = torch.randn(3, 64, device=gpu, requires_grad=True)
    mlp(a).sum().backward()
    with torch.no_grad():
        g, u = mlp.gate_up_proj(a).chunk(2, dim=-1)
        torch.testing.assert_close(mlp(a), mlp.down_proj(F.silu(g) * u), rtol=1e-5, atol=1e-6)
    assert a.grad is not None


# Rows at the edges of the row tiles (16, 32, 64, 128, 256) and of each kernel's tile choice; widths that
# leave a single 16-column tile, an odd number of tiles, fewer k-steps than wavefronts, k-steps that do
# not divide among them, and the 0.5B model's own shapes.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(16, 32), (48, 96), (80, 1056), (64, 1152), (32, 2112), (1152, 896), (896, 4864),
                                 (2080, 160)])
def test_small_linears(gpu, dtype, n, k):
    from engine import layer_ops

    for m in (1, 15, 16, 17, 32, 33, 64, 65, 128, 129, 200, 256):
        announce(f"small linears {dtype} m {m} n {n} k {k}")
        gen = torch.Generator(device=gpu).manual_seed(m * n + k)
        x = torch.randn(1, m, k, generator=gen, device=gpu).to(dtype)
        w = (torch.randn(n, k, generator=gen, device=gpu) / k ** 0.5).to(dtype)
        norm = (torch.rand(k, generator=gen, device=gpu) + 0.5).to(dtype)
        bias = torch.randn(n, generator=gen, device=gpu).to(dtype)
        res = torch.randn(1, m, n, generator=gen, device=gpu).to(dtype)
        xd, wd, u = x.double(), w.double(), U[dtype]
        # Roundings of the product and of the result, fp32 sums of k products (their worst case), and
        # with the norm two roundings of each of its elements: an error of independent terms, whose
        # deviation is below U times the root of their squares' sum; 8 deviations.
        got = layer_ops.linear_residual(x, w, res)
        y = xd @ wd.t()
        mag = xd.abs() @ wd.abs().t()
        want = y + res.double()
        assert ((got.double() - want).abs() <= 1.01 * u * (want.abs() + y.abs()) + (k / 64 + 8) * 2 ** -24 * mag + TINY).all()
        h = norm64(x, norm, 1e-6)
        y = h @ wd.t()
        spread = (h.square() @ wd.square().t()).sqrt()
        got = layer_ops.norm_linear(x, norm, 1e-6, w, bias)
        want = y + bias.double()
        assert ((got.double() - want).abs() <= 1.01 * u * want.abs() + 8 * u * spread + TINY).all()
        bare = layer_ops.norm_linear(x, norm, 1e-6, w)
        assert ((bare.double() - y).abs() <= 1.01 * u * y.abs() + 8 * u * spread + TINY).all()
        got = layer_ops.norm_linear(x, norm, 1e-6, w, gate_up=True)
        g, up = y.chunk(2, dim=-1)
        sg, su = spread.chunk(2, dim=-1)
        want = g * torch.sigmoid(g) * up  # |silu'| <= 1.1
        slack = 8 * u * (1.1 * sg * (up.abs() + 8 * u * su) + g.abs() * su)
        slack += u * (1.2 * g.abs() * up.abs() + want.abs())  # gate and up are rounded before their product
        assert ((got.double() - want).abs() <= 2.02 * u * want.abs() + slack + TINY).all()


def test_small_linears_refuse_what_they_do_not_take(gpu):
    from engine import _native

    announce("small linears: host checks")
    lib, t = _native.load(), torch.zeros(64, 64, device=gpu, dtype=torch.bfloat16)
    p = t.data_ptr()
    assert lib.mip_linear_residual(p, p, p, p, 257, 16, 32, 2, None) == _native.MIP_EUNSUPPORTED
    assert lib.mip_linear_residual(p, p, p, p, 1, 24, 32, 2, None) == _native.MIP_EUNSUPPORTED
    assert lib.mip_linear_residual(p, p, p, p, 1, 16, 48, 2, None) == _native.MIP_EUNSUPPORTED
    assert lib.mip_linear_residual(p, p, p, p, 1, 16, 32, 0, None) == _native.MIP_EUNSUPPORTED
    assert lib.mip_linear_residual(p + 2, p, p, p, 1, 16, 32, 2, None) == _native.MIP_EUNSUPPORTED
    assert lib.mip_linear_residual(p, p, p, None, 1, 16, 32, 2, None) == _native.MIP_EINVAL
    assert lib.mip_norm_linear(p, p, None, 1e-6, p, None, 1, 16, 32, 0, 2, None) == _native.MIP_EINVAL
    assert lib.mip_norm_linear(p, p, p, 1e-6, p, p, 1, 16, 32, 1, 2, None) == _native.MIP_EINVAL
    assert lib.mip_linear_residual(p, p, p, p, 0, 16, 32, 2, None) == _native.MIP_OK


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_fused_layer_matches_its_modules(gpu, dtype):
    """A layer through its fused steps against the same layer with a hook (which keeps the modules' own calls)."""
    from engine.model import DecoderLayer, Qwen2Config

    class Same:
        def attend(self, layer_idx, q, k, v):
            return q

    # (hidden, intermediate): the kernels' shapes, and a width with k % 32 != 0 that stays on the library.
    for hidden, inter in ((64, 128), (896, 4864), (72, 144)):
        cfg = Qwen2Config(vocab_size=64, hidden_size=hidden, intermediate_size=inter, num_layers=1, num_heads=hidden // 8,
                          num_kv_heads=1, head_dim=8)
        layer = DecoderLayer(cfg, 0).to(gpu).to(dtype).requires_grad_(False)
        layer.attn.qkv_proj.weight.mul_(2.0)
        for b, t in ((1, 1), (8, 1), (1, 17), (64, 1), (65, 1), (2, 100), (1, 300)):
            announce(f"fused layer {dtype} hidden {hidden} {b} x {t}")
            x = torch.randn(b, t, hidden, device=gpu).to(dtype)
            keep = x.clone()
            cs = torch.ones(b, 1, t, 8, device=gpu, dtype=dtype)
            with torch.inference_mode():
                assert layer._fusable(x)
                got = layer(x, cs, cs * 0, Same())
                handle = layer.mlp.register_forward_hook(lambda m, a, o: None)
                assert not layer._fusable(x)
                want = layer(x, cs, cs * 0, Same())
                handle.remove()
            assert torch.equal(x, keep)  # the input is not written
            # Both round each intermediate once or twice: a few roundings of relative size U each.
            err = (got.double() - want.double()).norm() / want.double().norm()
            assert err <= 8 * U[dtype], (hidden, b, t, float(err))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d,hq,hkv,k", [(64, 14, 2, 896), (128, 4, 2, 192), (16, 3, 1, 64), (32, 1, 3, 1056),
                                          (64, 2, 1, 2112)])
def test_qkv_linear_rotates_as_the_rope_kernel(gpu, dtype, d, hq, hkv, k):
    """The projection with the rotation inside: bit-equal to the projection, then rope_kv_append's rotation."""
    from engine import layer_ops, paged_ops
    from engine.model import rope_cos_sin

    for m in (1, 8, 17, 33, 64, 65, 130, 256):
        announce(f"qkv_linear {dtype} d={d} hq={hq} hkv={hkv} k={k} m={m}")
        gen = torch.Generator(device=gpu).manual_seed(m + d)
        n = (hq + 2 * hkv) * d
        x = torch.randn(m, 1, k, generator=gen, device=gpu).to(dtype)
        w = (torch.randn(n, k, generator=gen, device=gpu) / k ** 0.5).to(dtype)
        norm = (torch.rand(k, generator=gen, device=gpu) + 0.5).to(dtype)
        bias = torch.randn(n, generator=gen, device=gpu).to(dtype)
        pos = torch.randint(0, 4096, (m, 1), generator=gen, device=gpu)
        cos, sin = rope_cos_sin(pos, d, 1e6, dtype)
        assert layer_ops.rope_usable(cos, sin, x, d)
        pool = torch.zeros(1, hkv, 1, d, dtype=dtype, device=gpu)
        skip = torch.full((m,), -1, dtype=torch.int64, device=gpu)

        def rotate(y):
            y = y.clone().view(m, hq + 2 * hkv, d)
            paged_ops.rope_kv_append(y[:, :hq], y[:, hq:hq + hkv], y[:, hq + hkv:], cos[:, 0, 0], sin[:, 0, 0], pool,
                                     pool.clone(), skip)
            return y.view(m, 1, n)

        # The projection alone takes the same tiles as the one with the rotation: the same sums at every m.
        got = layer_ops.qkv_linear(x, norm, 1e-6, w, bias, cos, sin, hq + hkv)
        assert torch.equal(got, rotate(layer_ops.norm_linear(x, norm, 1e-6, w, bias)))
        # Of x as it is, and with no head rotated: the projection itself, rotated afterwards.
        plain = layer_ops.qkv_linear(x, None, 0.0, w, bias, cos, sin, 0)
        want = (x.double() @ w.double().t() + bias.double()).view(m, 1, n)
        mag = x.double().abs() @ w.double().abs().t()
        assert ((plain.double() - want).abs() <= 1.01 * U[dtype] * want.abs() + (k / 64 + 8) * 2 ** -24 * mag + TINY).all()
        assert torch.equal(layer_ops.qkv_linear(x, None, 0.0, w, bias, cos, sin, hq + hkv), rotate(plain))
        bare = layer_ops.qkv_linear(x, norm, 1e-6, w, None, cos, sin, hq + hkv)
        assert torch.equal(bare, rotate(layer_ops.norm_linear(x, norm, 1e-6, w)))
        # Norm and no rotation in the rotating kernel, against 64 bits (bounds as in test_small_linears).
        h = norm64(x, norm, 1e-6)
        want = h @ w.double().t() + bias.double()
        spread = (h.square() @ w.double().square().t()).sqrt()
        still = layer_ops.qkv_linear(x, norm, 1e-6, w, bias, cos, sin, 0)
        assert ((still.double() - want).abs() <= 1.01 * U[dtype] * want.abs() + 8 * U[dtype] * spread + TINY).all()


@torch.inference_mode()
def test_contexts_that_rotate_for_themselves_still_do(gpu):
    """A decode context's own attend_rope, wrapped, subclassed or patched, is called where there is one."""
    from engine.kv_cache import PagedDecodeContext, PagedKVCache
    from engine.model import DecoderLayer, Qwen2Config, rope_cos_sin

    announce("takes_rotated: wrapped and subclassed contexts")
    cfg = Qwen2Config(vocab_size=64, hidden_size=256, intermediate_size=512, num_layers=1, num_heads=4, num_kv_heads=2,
                      head_dim=64)
    dt = torch.bfloat16
    layer = DecoderLayer(cfg, 0).to(gpu).to(dt).requires_grad_(False)
    cache = PagedKVCache(1, 2, 64, 64, 16, max_seqs=8, max_len=256, dtype=dt, device=gpu)
    slots = []
    for n in (5, 33, 100):
        s = cache.allocate(n + 1)
        cache.lengths[s] = n
        slots.append(s)
    cache.k.normal_()
    cache.v.normal_()
    k0, v0 = cache.k.clone(), cache.v.clone()
    x = torch.randn(3, 1, 256, device=gpu).to(dt)
    calls = []

    class Sub(PagedDecodeContext):
        def attend_rope(self, *a):
            calls.append("sub")
            return super().attend_rope(*a)

    class Wrap:
        fuse_rope = True

        def __init__(self, inner):
            self.inner = inner

        def attend_rope(self, *a):
            calls.append("wrap")
            return self.inner.attend_rope(*a)

    def run(ctx, inner):
        cache.k.copy_(k0)
        cache.v.copy_(v0)
        cos, sin = rope_cos_sin(inner.positions.unsqueeze(1), 64, cfg.rope_theta, dt)
        return layer(x, cos, sin, ctx), cache.k.clone(), cache.v.clone()

    inner = PagedDecodeContext(cache, slots)
    assert inner.takes_rotated
    want = run(inner, inner)
    sub = Sub(cache, slots)
    assert not sub.takes_rotated
    inner2 = PagedDecodeContext(cache, slots)
    inner3 = PagedDecodeContext(cache, slots)
    inner3.fuse_rope = False
    for ctx, base in ((sub, sub), (Wrap(inner2), inner2), (inner3, inner3)):
        for a, b in zip(run(ctx, base), want):
            assert torch.equal(a, b)
    assert calls == ["sub", "wrap"]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@torch.inference_mode()
def test_layers_called_one_by_one_give_the_models_bits(gpu, dtype):
    """With many rows a layer hands its last residual add on; called by itself it rounds exactly as within the model."""
    from engine.model import Qwen2Config, Qwen2ForCausalLM, rope_cos_sin

    announce(f"layers one by one {dtype}")

    class Same:
        def attend(self, layer_idx, q, k, v):
            return q

    cfg = Qwen2Config(vocab_size=97, hidden_size=128, intermediate_size=320, num_layers=3, num_heads=4, num_kv_heads=2,
                      head_dim=32)
    model = Qwen2ForCausalLM(cfg).to(gpu).to(dtype).requires_grad_(False)
    ids = torch.randint(0, 97, (1, 300), device=gpu)
    pos = torch.arange(300, device=gpu)[None]
    x = model.embed_tokens(ids)
    cos, sin = rope_cos_sin(pos, 32, cfg.rope_theta, dtype)
    for layer in model.layers:
        x = layer(x, cos, sin, Same())
    assert torch.equal(model.norm(x), model(ids, pos, Same()))
