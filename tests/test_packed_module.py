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


@pytest.mark.parametrize("T", TOKENS)
def test_bias_forward_mode(layer, T):
    """A bias with a forward-mode tangent keeps it."""
    import torch.autograd.forward_ad as fwAD
    make, W, _ = layer
    b, t = torch.linspace(-1, 1, R), torch.linspace(2, 3, R)
    pl, x = make(None), _x(T)
    with fwAD.dual_level():
        pl.register_buffer("bias", fwAD.make_dual(b, t))
        y, ty = fwAD.unpack_dual(pl(x))
        assert torch.allclose(y, x @ W.t() + b, atol=1e-5)
        assert ty is not None and torch.equal(ty, t.expand(T, R))


@pytest.mark.parametrize("T", TOKENS)
def test_bias_vmap(layer, T):
    make, W, _ = layer
    pl, x = make(torch.zeros(R)), _x(T)

    def f(v):
        return torch.func.functional_call(pl, {"bias": v}, (x,))
    bs = torch.randn(3, R, generator=torch.Generator().manual_seed(7))
    y = torch.func.vmap(f)(bs)
    assert torch.allclose(y, x @ W.t() + bs[:, None], atol=1e-5)


class Tagged(torch.Tensor):
    """A subclass, which torch's add sees and keeps."""


def test_bias_subclass_and_negative_view(layer):
    """A tensor subclass goes to torch's add, and so does a view whose memory
    holds the negated values."""
    make, W, calls = layer
    x = _x(2)
    b = torch.linspace(-1, 1, R)
    assert isinstance(make(b.as_subclass(Tagged))(x), Tagged)
    y = make(torch._neg_view(b))(x)
    assert calls == ["gemv", "gemv"]
    assert torch.allclose(y, x @ W.t() - b, atol=1e-5)
    make(b)(x), make(nn.Parameter(b, requires_grad=False))(x), make(None)(x)
    assert calls[2:] == ["linear"] * 3


def test_linear_packed_checks_devices():
    """kernels.linear_packed takes operands of one device only: a bias of
    another one is refused, as torch's add would."""
    from types import SimpleNamespace as NS
    from crb_amd._lib import CrbqError
    a, b = (NS(is_cuda=True, get_device=lambda i=i: i, numel=lambda: 1) for i in (0, 1))
    for bad in range(5):
        ts = [b if i == bad else a for i in range(5)]
        with pytest.raises(CrbqError, match="one device"):
            kernels.linear_packed(ts[0], ts[1], ts[2], C, ts[3], ts[4])
    ex = kernels.PackedEx(b, b, b)
    with pytest.raises(CrbqError, match="one device"):
        kernels.linear_packed(a, a, a, C, a, a, ex)
