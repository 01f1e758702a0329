"""The FP8 GEMM kernels (lbw_gemm_fp8_rows, lbw_gemm_fp8_mx) against the exact product of the same operands in fp64, at
the edges of every tile form (64, 128, 192 and 256 rows, K in one or two shares, K tails of 16-byte steps, ragged
tokens and channels), and through FP8Linear / MXFP8Linear.

Tolerance: the result is rounded once to bf16 (2^-8 relative). Products of e4m3 values are exact in fp32, but the
matrix instruction adds the 64 of a step aligned to the largest rather than rounding each sum: on the same operands the
library's GEMM, which runs the same instruction, was up to 2.1e-3 from the exact sum beyond the bf16 rounding at
sum |terms| = 100 (2^-15.5 of it), and this kernel the same to the last digit. So the bound adds 2^-15 sum |terms|
elementwise, and the error as a whole may not exceed the
library's by more than 1 %. MX: the scales here span 13 binades, so a few terms are most of a sum and the same
alignment to the largest costs more of it: 2^-13 sum |terms|; and the product is cut to bf16
toward zero (2^-7 relative) before the bias is added."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _k():
    from lingbot_world_v2_realtime_amd import kernels
    return kernels


def _operands(m, k, n, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x8 = torch.randn(m, k, generator=g, device=DEV).to(torch.float8_e4m3fn)
    w8 = torch.randn(n, k, generator=g, device=DEV).to(torch.float8_e4m3fn)
    return g, x8, w8, torch.randn(n, generator=g, device=DEV).to(torch.bfloat16)


def _check(y, x, w, bias, align=2.0 ** -15, rnd=2.0 ** -8):
    """y against x w^T + bias for fp64 operands (scales applied)."""
    ref, mag = x @ w.t(), x.abs() @ w.abs().t()
    if bias is not None:
        ref, mag = ref + bias.double(), mag + bias.double().abs()
    tol = rnd * ref.abs() + align * mag
    assert bool(((y.double() - ref).abs() <= tol).all()), float(((y.double() - ref).abs() - tol).max())


# one K share / two (K >= 4096; 4224: an odd number of stages, the second share's last one past K) at 64 x 64; 128 x 128; 192 x 192 in one and more rounds; 256 x 256, full and ragged, with a
# last round of half tiles (one of them past the last channel)
SHAPES = [(1, 16, 16), (65, 144, 48), (63, 1056, 1536), (64, 4096, 64), (33, 4224, 192), (257, 4240, 1520), (17, 8960, 1536),
          (1000, 272, 2048), (1509, 1536, 1536), (2305, 128, 2320), (6032, 256, 1536), (2048, 400, 8192),
          (3105, 256, 8976), (6032, 1536, 8960), (8200, 400, 2144)]


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_gemm_rows(m, k, n):
    g, x8, w8, b = _operands(m, k, n, m + k + n)
    xs = torch.rand(m, 1, generator=g, device=DEV) + 0.5
    ws = torch.rand(1, n, generator=g, device=DEV) + 0.5
    x, w = x8.double() * xs.double(), w8.double() * ws.double().t()
    for bias in (b, None):
        y = _k().gemm_fp8_rows(x8, xs, w8, ws, bias)
        torch.cuda.synchronize()
        _check(y, x, w, bias)
    assert torch.equal(_k().gemm_fp8_rows(x8, xs, w8, ws, None), y)
    lib = torch._scaled_mm(x8, w8.t(), scale_a=xs, scale_b=ws, out_dtype=torch.bfloat16)
    ref = x @ w.t()
    assert (y.double() - ref).norm() <= 1.01 * (lib.double() - ref).norm()


@pytest.mark.parametrize("m,k,n", [(65, 144, 48), (64, 8960, 1536), (1000, 272, 2048), (1509, 1536, 1536),
                                   (2305, 128, 2320), (2048, 400, 8192), (3105, 256, 8976)])
def test_gemm_rows_epilogue_bits(m, k, n):
    """Operands of small integers, whose sums are exact in fp32 (|sum| <= 36 K < 2^24): what is left is the epilogue,
    scale of the channel, scale of the token, bias, each rounded to fp32, then bf16. Every bit of it is defined."""
    g = torch.Generator(device=DEV).manual_seed(m + n)
    x8, w8 = (torch.randint(-6, 7, (r, k), generator=g, device=DEV).float().to(torch.float8_e4m3fn) for r in (m, n))
    xs = torch.rand(m, 1, generator=g, device=DEV) + 0.01
    ws = torch.rand(1, n, generator=g, device=DEV) * 1e-3 + 1e-5
    b = (torch.randn(n, generator=g, device=DEV) * 0.1).to(torch.bfloat16)
    v = (x8.double() @ w8.double().t()).float()
    for bias in (None, b):
        want = (v * ws) * xs
        if bias is not None:
            want = want + bias.float()
        assert torch.equal(_k().gemm_fp8_rows(x8, xs, w8, ws, bias), want.to(torch.bfloat16))


@pytest.mark.parametrize("m,k,n", [s for s in SHAPES if s[1] % 128 == 0])
def test_gemm_mx(m, k, n):
    g, x8, w8, b = _operands(m, k, n, m + k + n)
    xe, we = (torch.randint(120, 134, (r, k // 32), generator=g, device=DEV, dtype=torch.uint8) for r in (m, n))
    x, w = (v.double() * torch.exp2(e.double() - 127).repeat_interleave(32, 1) for v, e in ((x8, xe), (w8, we)))
    xt, wt = (e.view(e.shape[0], -1, 4).transpose(0, 1).contiguous() for e in (xe, we))
    for bias in (b, None):
        y = _k().gemm_fp8_mx(x8, xt, w8, wt, bias)
        torch.cuda.synchronize()
        if bias is None:
            _check(y, x, w, None, 2.0 ** -13, 2.0 ** -7)
            assert torch.equal(with_bias, y + b)
        with_bias = y


def test_quant_mx_transposed_scales():
    x = torch.randn(77, 1152, device=DEV).to(torch.bfloat16)
    for t in (x, x.float()):
        a8, ae = _k().quant_mx_fp8(t, 128)
        b8, be = _k().quant_mx_fp8(t, 128, transposed=True)
        assert torch.equal(a8.view(torch.uint8), b8.view(torch.uint8))
        assert torch.equal(ae.view(torch.uint8).view(128, -1, 4).transpose(0, 1), be)


@pytest.mark.parametrize("m,k,n", [(1, 128, 1), (77, 1152, 384), (300, 1536, 8960), (6032, 128, 257)])
def test_quant_mx_other_operands_scales(m, k, n):
    """The other operand's scales reordered in the quantiser's launch, also from a strided and a misaligned view."""
    x = torch.randn(m, k, device=DEV).to(torch.bfloat16)
    e = torch.randint(0, 256, (n, k // 32), device=DEV, dtype=torch.uint8)
    wide, odd = torch.zeros(n, k // 16, device=DEV, dtype=torch.uint8), torch.zeros(n * (k // 32) + 1, device=DEV,
                                                                                   dtype=torch.uint8)
    wide[:, :k // 32], odd[1:] = e, e.view(-1)
    want = e.view(n, -1, 4).transpose(0, 1)
    a8, ae = _k().quant_mx_fp8(x, transposed=True)
    for w in (e, wide[:, :k // 32], odd[1:].view(n, -1)):
        b8, be, wt = _k().quant_mx_fp8(x, transposed=True, w_scale=w.view(torch.float8_e8m0fnu))
        assert torch.equal(a8.view(torch.uint8), b8.view(torch.uint8)) and torch.equal(ae, be) and torch.equal(wt, want)


def test_mx_scales_follow_writes():
    """MXFP8Linear multiplies by what w8 and w_scale hold at the call: after in-place writes through state_dict(), and
    after writes that no version counter sees (.data, as a collective's), as a module built from those weights; also with
    the buffers exchanged, and in a copy."""
    import copy
    from lingbot_world_v2_realtime_amd.layers.linear import MXFP8Linear
    with torch.no_grad():
        a, b = (torch.nn.Linear(1536, 1000, device=DEV, dtype=torch.bfloat16) for _ in range(2))
        b.weight.mul_(torch.exp2(torch.randint(-6, 7, (1000, 1), device=DEV).to(torch.bfloat16)))
        b.bias.copy_(a.bias)
        src = MXFP8Linear(b)
        x = torch.randn(65, 1536, device=DEV).to(torch.bfloat16)
        want = src(x)
        for write in ("state_dict", "data", "exchange"):
            mx = MXFP8Linear(a)
            assert not torch.equal(mx(x), want)
            for name in ("w8", "w_scale"):
                if write == "exchange":
                    setattr(mx, name, getattr(src, name).clone())
                else:
                    dst = mx.state_dict()[name] if write == "state_dict" else getattr(mx, name).data
                    dst.view(torch.uint8).copy_(getattr(src, name).view(torch.uint8))
            assert torch.equal(mx(x), want), write
        assert torch.equal(copy.deepcopy(mx)(x), want)


def test_nonfinite_rows_stay_in_their_row():
    """A row whose scale is inf or NaN gives a NaN row and leaves the others as they are."""
    g, x8, w8, b = _operands(300, 1536, 1536, 5)
    xs, ws = torch.ones(300, 1, device=DEV), torch.ones(1, 1536, device=DEV)
    want = _k().gemm_fp8_rows(x8, xs, w8, ws, b)
    x8.view(torch.uint8)[7, 3] = 0x7F
    xs[9] = float("nan")
    y = _k().gemm_fp8_rows(x8, xs, w8, ws, b)
    rows = torch.arange(300, device=DEV)
    bad = (rows == 7) | (rows == 9)
    assert bool(y[bad].isnan().all()) and torch.equal(y[~bad], want[~bad])


@pytest.mark.parametrize("m,k,n", [(333, 1056, 1536), (64, 8960, 1536)])
def test_linears_run_the_kernel(m, k, n):
    """FP8Linear and MXFP8Linear without gradients against the products of their own quantised operands; a bias of odd
    alignment, a state_dict round trip (MX scales follow the loaded ones), and the path that records a gradient."""
    from lingbot_world_v2_realtime_amd.layers.linear import FP8Linear, MXFP8Linear
    lin = torch.nn.Linear(k, n, device=DEV, dtype=torch.bfloat16)
    lin2 = torch.nn.Linear(k, n, device=DEV, dtype=torch.bfloat16)
    x = torch.randn(3, m // 3, k, device=DEV).to(torch.bfloat16)
    with torch.no_grad():
        f = FP8Linear(lin)
        f.bias = torch.nn.Parameter(torch.randn(n + 1, device=DEV).to(torch.bfloat16)[1:])
        x8, xs = _k().quant_rows_fp8(x.reshape(-1, k))
        y = f(x)
        _check(y.reshape(-1, n), x8.double() * xs.double(), f.w8.double() * f.w_scale_t.double().t(), f.bias)
        mx, src = MXFP8Linear(lin), MXFP8Linear(lin2)
        want = src(x)
        assert set(src.state_dict()) == {"w8", "w_scale", "bias"}
        mx.load_state_dict({key: v.clone() for key, v in src.state_dict().items()})
        assert torch.equal(mx(x), want)
    grad = f(x)
    assert grad.requires_grad
    assert (grad.float() - y.float()).abs().max() <= 2.0 ** -7 * y.float().abs().max()
    assert mx(x).requires_grad


def test_bias_with_a_tangent_or_under_vmap():
    """What the kernel may not take by its address: MXFP8Linear adds it to the product, FP8Linear leaves it to
    torch._scaled_mm, which refuses the derivative."""
    from torch.autograd import forward_ad
    from lingbot_world_v2_realtime_amd.layers.linear import FP8Linear, MXFP8Linear
    lin = torch.nn.Linear(1536, 1024, device=DEV, dtype=torch.bfloat16).requires_grad_(False)
    x = torch.randn(130, 1536, device=DEV).to(torch.bfloat16)
    mx, f, b = MXFP8Linear(lin), FP8Linear(lin), lin.bias.detach().clone()
    t, want, rows = torch.randn_like(b), mx(x), f(x)
    del mx.bias, f.bias
    with forward_ad.dual_level():
        mx.bias = f.bias = forward_ad.make_dual(b, t)
        out = forward_ad.unpack_dual(mx(x))
        assert torch.equal(out.primal, want) and torch.equal(out.tangent, t.expand(130, -1))
        with pytest.raises(NotImplementedError):
            f(x)

    def call(module):
        def fn(bias):
            module.bias = bias
            return module(x)
        return fn

    two = torch.vmap(call(mx))(torch.stack([b, b + 1]))
    assert torch.equal(two[0], want) and torch.equal(two[1], call(mx)(b + 1))
    assert torch.equal(call(f)(b.view(1, -1)), rows)   # a bias of n values in two dimensions: torch's product


def test_weights_at_any_address():
    """Weights that are a view into a larger buffer, at an address that is not a multiple of 16."""
    from lingbot_world_v2_realtime_amd.layers.linear import FP8Linear, MXFP8Linear
    lin = torch.nn.Linear(1536, 1024, device=DEV, dtype=torch.bfloat16).requires_grad_(False)
    x = torch.randn(65, 1536, device=DEV).to(torch.bfloat16)
    for module in (FP8Linear(lin), MXFP8Linear(lin)):
        want = module(x)
        flat = torch.zeros(module.w8.numel() + 1, dtype=torch.uint8, device=DEV)
        flat[1:] = module.w8.view(torch.uint8).view(-1)
        module.w8 = flat[1:].view(torch.float8_e4m3fn).view(module.w8.shape)
        assert module.w8.data_ptr() % 16 and torch.equal(module(x), want)
