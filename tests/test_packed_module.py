"""PackedLinear's own logic on the CPU: its kernels are replaced by dense
products of a stand-in weight, so only the module's dispatch runs."""
import pytest
import torch
import torch.nn as nn
import torch.nn.utils.parametrize  # noqa: F401

from crb_amd import kernels
from crb_amd.packed import PackedLinear

R, C = 24, 16
TOKENS = (1, 64, 1024)        # GEMV, GEMM, unpack + dense product


@pytest.fixture
def layer(monkeypatch):
    """make(bias) -> PackedLinear over W; W; and the names of the kernels called."""
    g = torch.Generator().manual_seed(1)
    W = torch.randn(R, C, generator=g, dtype=torch.float64).float()
    calls = []

    def product(name):
        def f(codes, lut, sal, C_, x, ex=None):
            calls.append(name)
            return x.detach() @ W.t()
        return f

    def fused(codes, lut, sal, C_, x, bias=None, ex=None):
        calls.append("linear")
        y = x.detach() @ W.t()
        # the kernel reads the bias' memory: no gradient or tangent goes through
        return y if bias is None else y + torch.from_numpy(bias.detach().numpy())

    monkeypatch.setattr(kernels, "gemv_packed", product("gemv"))
    monkeypatch.setattr(kernels, "gemm_packed", product("gemm"))
    monkeypatch.setattr(kernels, "linear_packed", fused)
    monkeypatch.setattr(kernels, "unpack", lambda *a, **k: W)

    def make(bias):
        return PackedLinear(torch.zeros(R, 32, dtype=torch.uint8), torch.zeros(R, 1, 8),
                            torch.zeros(1, 16, dtype=torch.uint8), C, bias)
    return make, W, calls


def _x(T):
    return torch.randn(T, C, generator=torch.Generator().manual_seed(T))


@pytest.mark.parametrize("T", TOKENS)
def test_bias_assigned_as_parameter(layer, T):
    """``pl.bias = nn.Parameter(...)`` moves the name from the module's buffers
    to its parameters: the call works and the bias takes its gradient."""
    make, W, _ = layer
    pl = make(torch.zeros(R))
    b = torch.linspace(-1, 1, R)
    pl.bias = nn.Parameter(b.clone())
    x = _x(T)
    y = pl(x)
    assert torch.allclose(y, x @ W.t() + b, atol=1e-5)
    y.sum().backward()
    assert torch.equal(pl.bias.grad, torch.full((R,), float(T)))
    pl.bias = nn.Parameter(b.clone(), requires_grad=False)
    assert torch.allclose(pl(x), x @ W.t() + b, atol=1e-5)


@pytest.mark.parametrize("T", TOKENS)
def test_parametrized_bias(layer, T):
    make, W, _ = layer
    pl = make(torch.ones(R))

    class Double(nn.Module):
        def forward(self, v):
            return 2 * v
    nn.utils.parametrize.register_parametrization(pl, "bias", Double())
    x = _x(T)
    assert torch.allclose(pl(x), x @ W.t() + 2, atol=1e-5)
