"""The linear layers' bias, added in the GEMM's epilogue where it is a plain bf16 vector and by torch
otherwise: the bits of the layer without a bias plus the bias, whichever kernel the rows take."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(pkg, dev, kind, n, k):
    g = torch.Generator().manual_seed(n + k)
    key = {"mxfp8": pkg.linear.MXFP8_STATIC, "mxfp6": pkg.linear.MXFP6_E2M3_STATIC, "block": pkg.linear.FP8_BLOCK128}[kind]
    method, layer = pkg.MxLinearMethod(key), torch.nn.Module()
    method.create_weights(layer, k, [n], k, n, torch.bfloat16, device=dev)
    codes = torch.randint(0, 0x70, tuple(layer.weight.shape), generator=g, dtype=torch.uint8)
    layer.weight.weight_loader(layer.weight, (codes if kind == "mxfp6" else codes.view(torch.float8_e4m3fn)).to(dev))
    scale = layer.weight_scale_inv if kind == "block" else layer.weight_scale
    s = torch.rand(tuple(scale.shape), generator=g) * 1e-3 if kind == "block" else \
        torch.randint(115, 120, tuple(scale.shape), generator=g, dtype=torch.uint8)
    scale.weight_loader(scale, s.to(dev))
    method.process_weights_after_loading(layer)
    return method, layer


@pytest.mark.parametrize("kind,n,k", [("mxfp8", 640, 1024), ("mxfp6", 4104, 2688), ("block", 5120, 4352)])
@pytest.mark.parametrize("M", [1, 5, 40, 130, 600])  # streaming, generic, tiles whole and split in K
def test_bias_bits(pkg, dev, kind, n, k, M):
    method, layer = _layer(pkg, dev, kind, n, k)
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, k, generator=g).bfloat16().to(dev)
    wide = (torch.randn(2 * n + 1, generator=g) * 50).bfloat16().to(dev)
    y = method.apply(layer, x, None)
    wide[3] = float("nan")
    grad = wide[:n].clone().requires_grad_()
    for bias in (wide[:n], wide[1:n + 1], wide[1::2], wide[:n].float(),
                 wide[:n].view(1, n), wide[:1], grad):
        got, want = method.apply(layer, x, bias), y + bias
        assert got.dtype == want.dtype and got.requires_grad == want.requires_grad
        assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(want))
        assert torch.equal(got.isnan(), want.isnan())
    method.apply(layer, x, grad).float().nan_to_num().sum().backward()
    assert grad.grad is not None


@pytest.mark.parametrize("kind,n,k", [("mxfp8", 640, 1024), ("mxfp6", 520, 2688), ("block", 512, 1152)])
@pytest.mark.parametrize("M", [1, 40])
def test_bias_under_transforms(pkg, dev, kind, n, k, M):
    """A bias that carries a tangent, a batch dimension or a gradient of a transform into the addition, or is
    traced, is added as torch does it."""
    method, layer = _layer(pkg, dev, kind, n, k)
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, k, generator=g).bfloat16().to(dev)
    biases = torch.randn(3, n, generator=g).bfloat16().to(dev)
    bias, tangent = biases[0], biases[1]
    y = method.apply(layer, x, None)
    call = lambda b: method.apply(layer, x, b)  # noqa: E731
    assert torch.equal(torch.func.vmap(call)(biases), y + biases[:, None])
    out, t = torch.func.jvp(call, (bias,), (tangent,))
    assert torch.equal(out, y + bias) and torch.equal(t, tangent.expand(M, n))
    with torch.autograd.forward_ad.dual_level():
        dual = call(torch.autograd.forward_ad.make_dual(bias, tangent))
        out, t = torch.autograd.forward_ad.unpack_dual(dual)
        assert torch.equal(out, y + bias) and torch.equal(t, tangent.expand(M, n))
    ones = torch.func.grad(lambda b: call(b).float().sum())(bias)
    assert torch.equal(ones, torch.full_like(bias, M))
    traced = torch.compile(call, fullgraph=M > 16, backend="eager")  # (up to 16 rows the route asks the library)
    assert torch.equal(traced(bias), y + bias)
    with torch.no_grad():
        assert torch.equal(call(torch.nn.Parameter(bias)), y + bias)
