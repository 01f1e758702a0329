"""Host side of the FP8 linears without a GPU: the library and the stream lookup are replaced by stubs, so nothing is
launched."""
import pytest
import torch

from lingbot_world_v2_realtime_amd import kernels

F8 = torch.float8_e4m3fn


class StubLib:
    """Stands for the loaded library: every entry point notes its call and reports success."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *args: self.calls.append((name, args)) or 0


@pytest.fixture
def stub(monkeypatch):
    lib = StubLib()
    monkeypatch.setattr(kernels._lib, "load", lambda *a: lib)
    monkeypatch.setattr(kernels, "_raw_stream", lambda idx: 0)
    return lib


def test_gemm_refuses_host_tensors(stub):
    """A host pointer must not reach a kernel: all operands on the host, and the stream of a host tensor."""
    m, n, k = 32, 16, 128
    x8, w8 = torch.zeros(m, k).to(F8), torch.zeros(n, k).to(F8)
    with pytest.raises(ValueError, match="device tensor"):
        kernels.gemm_fp8_rows(x8, torch.ones(m, 1), w8, torch.ones(1, n))
    with pytest.raises(ValueError, match="device tensor"):
        kernels.gemm_fp8_mx(x8, torch.zeros(k // 128, m, 4, dtype=torch.uint8), w8,
                            torch.zeros(k // 128, n, 4, dtype=torch.uint8))
    with pytest.raises(ValueError, match="device tensor"):
        kernels._stream(x8)
    assert stub.calls == []


@pytest.fixture
def routes(monkeypatch):
    """FP8Linear and MXFP8Linear on the CPU with their kernels and torch._scaled_mm replaced by an fp32 product of plain
    operands; the list says which route each call took. The kernels' stand-ins read by address, as the kernels do."""
    from lingbot_world_v2_realtime_amd.layers import linear
    taken = []

    def quant(x, rows_pad=None, transposed=False, w_scale=None):
        x = torch.nn.functional.pad(x.float(), (0, 0, 0, (rows_pad or x.shape[0]) - x.shape[0]))
        one = torch.ones(x.shape[0], 1)
        return (x, one) if w_scale is None else (x, one, w_scale)

    def kernel(name):
        def product(x8, xs, w8, ws, bias=None):
            taken.append(name)
            assert all(t.data_ptr() for t in (x8, w8, ws))
            y = x8 @ w8.t()
            if bias is not None:
                assert bias.data_ptr()
                y = y + bias.detach().float()
            return y.detach().bfloat16()
        return product

    def scaled_mm(x8, wt, scale_a, scale_b, bias=None, out_dtype=None):
        taken.append("scaled_mm")
        y = x8 @ wt
        if bias is not None:
            if bias.requires_grad or (torch.autograd.forward_ad._current_level >= 0 and
                                      torch.autograd.forward_ad.unpack_dual(bias).tangent is not None):
                raise NotImplementedError("the derivative of _scaled_mm is not implemented")
            y = y + bias.float()
        return y.to(out_dtype)

    monkeypatch.setattr(kernels, "quant_rows_fp8", quant)
    monkeypatch.setattr(kernels, "quant_mx_fp8", quant)
    monkeypatch.setattr(kernels, "gemm_fp8_rows", kernel("rows"))
    monkeypatch.setattr(kernels, "gemm_fp8_mx", kernel("mx"))
    monkeypatch.setattr(torch, "_scaled_mm", scaled_mm)
    # -1, 0 and 1: every sum is a whole number of at most 256, exact in bf16 in any order
    g = torch.Generator().manual_seed(1)
    lin = torch.nn.Linear(256, 128).bfloat16().requires_grad_(False)
    for p in (lin.weight, lin.bias):
        p.copy_(torch.randint(-1, 2, p.shape, generator=g))
    return linear, lin, torch.randint(-1, 2, (3, 256), generator=g).bfloat16(), taken


def test_mx_bias_keeps_its_derivatives_and_transforms(routes):
    from torch.autograd import forward_ad
    linear, lin, x, taken = routes
    mx = linear.MXFP8Linear(lin)
    want = mx(x)
    assert taken == ["mx"] and not want.requires_grad
    b, t = mx.bias.detach().clone(), torch.randn(128).bfloat16()
    del mx.bias
    with forward_ad.dual_level():
        mx.bias = forward_ad.make_dual(b, t)
        out = forward_ad.unpack_dual(mx(x))
        assert torch.equal(out.primal, want) and torch.equal(out.tangent, t.expand(3, 128))

    def call(bias):
        mx.bias = bias
        return mx(x)

    assert torch.equal(torch.vmap(call)(torch.stack([b, b + 1])), torch.stack([want, call(b + 1)]))
    y = call(b.clone().requires_grad_())
    assert torch.equal(torch.autograd.grad(y.sum(), mx.bias)[0], torch.full((128,), 3.0).bfloat16())
    assert torch.equal(call(b[:1]), call(b[:1].expand(128).clone()))   # a bias that broadcasts
    assert "scaled_mm" not in taken


def test_weights_in_a_transform_or_strided_keep_the_library_product(routes):
    linear, lin, x, taken = routes
    for module, scales in ((linear.FP8Linear(lin), "w_scale_t"), (linear.MXFP8Linear(lin), "w_scale")):
        want, w8, s = module(x), module.w8, getattr(module, scales)
        taken.clear()

        def call(w):
            return torch.func.functional_call(module, {"w8": w, scales: s}, (x,))

        got = torch.vmap(call)(torch.stack([w8, 2 * w8]))
        assert torch.equal(got[0], want) and not torch.equal(got[1], want)
        call(torch.cat([w8, w8], 1)[:, :256])
        assert taken == ["scaled_mm", "scaled_mm"]


def test_rowwise_bias_with_a_derivative_is_refused_as_before(routes):
    from torch.autograd import forward_ad
    linear, lin, x, taken = routes
    f = linear.FP8Linear(lin)
    want, b = f(x), f.bias.detach().clone()
    assert taken == ["rows"]
    del f.bias
    with forward_ad.dual_level():
        f.bias = forward_ad.make_dual(b, torch.ones_like(b))
        with pytest.raises(NotImplementedError):
            f(x)
        f.bias = b                                  # a plain bias inside a dual level
        assert torch.equal(f(x), want) and taken[-1] == "rows"
    f.bias = b.clone().requires_grad_()
    with pytest.raises(NotImplementedError):
        f(x)
    with torch.no_grad():
        assert torch.equal(f(x), want) and taken[-1] == "rows"

    def call(bias):
        f.bias = bias
        return f(x)

    assert torch.equal(torch.vmap(call)(torch.stack([b, b + 1]))[0], want) and taken[-1] == "scaled_mm"
    f.bias = b.view(1, 128)
    assert torch.equal(f(x), want) and taken[-1] == "scaled_mm"
