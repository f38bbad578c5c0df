"""Packed low-bit storage on the GPU: crbq_pack / crbq_unpack byte-for-byte
against the NumPy statement of the format (tests/packed_ref.py), exception
lists included, and bit-exact round trips of layers quantized by the block
loop; crbq_gemv_packed / crbq_gemm_packed against float64 products of the
unpacked weights; PackedLinear and the stack driver's pack option.

GEMV bar: |y - y64| <= 1e-5 * sum_c |w_c x_c| per output (fp32 sums of
exact 16-bit products)."""
import numpy as np
import pytest
import torch

from packed_ref import pack_ref, structured, unpack_ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _k():
    from crb_amd import kernels
    return kernels


def _q16(q, dtype):
    bits = q.view(np.uint16)
    if dtype == torch.bfloat16:          # reinterpret the same bit patterns as bf16
        return torch.from_numpy(bits.astype(np.int16)).view(torch.bfloat16).to(DEV)
    return torch.from_numpy(q).to(DEV)


@pytest.mark.parametrize("R,C,dtype,n_odd", [(37, 300, torch.float16, 0),
                                             (64, 512, torch.bfloat16, 0),
                                             (5, 128, torch.float16, 3),
                                             (200, 1000, torch.bfloat16, 40)])
def test_pack_matches_format_statement(R, C, dtype, n_odd):
    print(f"pack structured {R}x{C} {dtype} odd={n_odd}", flush=True)
    q, masks = structured(R, C, seed=R + C, dtype=np.float16, n_odd=n_odd)
    bits = q.view(np.uint16)
    Q = _q16(q, dtype)
    M = torch.from_numpy(masks).to(DEV)
    codes, lut, sal, ex = _k().pack(Q, M)
    rc, rl, rs, rex, st = pack_ref(bits, masks, bf16=dtype == torch.bfloat16)
    assert st == 0 and (len(rex[0]) > 0) == (n_odd > 0)
    assert np.array_equal(codes.cpu().numpy(), rc)
    assert np.array_equal(lut.cpu().view(torch.int16).numpy().view(np.uint16), rl)
    assert np.array_equal(sal.cpu().numpy(), rs)
    assert np.array_equal(ex.idx.cpu().numpy(), rex[0])
    assert np.array_equal(ex.val.cpu().view(torch.int16).numpy().view(np.uint16), rex[1])
    assert np.array_equal(ex.delta.cpu().numpy(), rex[2])
    back = _k().unpack(codes, lut, sal, C, ex)
    assert torch.equal(back.view(torch.int16).cpu(), Q.view(torch.int16).cpu())


@pytest.mark.parametrize("R,C,pad,n_odd", [(1, 1, 0, 0), (3, 9, 1, 0), (5, 130, 3, 2),
                                           (17, 136, 8, 1), (67, 257, 5, 9)])
def test_pack_strided_edges(R, C, pad, n_odd):
    """Block rows at the ends of a wavefront's four and rows and columns at the
    ends of the matrix, weights and masks in rows of unaligned stride: pack
    against the format statement, unpack (1 to 4 rows per thread) bit for bit
    into an unaligned destination."""
    print(f"pack edges {R}x{C} pad={pad} odd={n_odd}", flush=True)
    from crb_amd import _lib
    q, masks = structured(R, C, seed=R + C, n_odd=n_odd)
    Qb = torch.zeros(R, C + pad, dtype=torch.float16, device=DEV)
    Mb = torch.zeros(R, C + pad, dtype=torch.uint8, device=DEV)
    Qb[:, :C], Mb[:, :C] = torch.from_numpy(q).to(DEV), torch.from_numpy(masks).to(DEV)
    codes, lut, sal, ex = _k().pack(Qb[:, :C], Mb[:, :C])
    rc, rl, rs, rex, st = pack_ref(q.view(np.uint16), masks)
    assert st == 0
    assert np.array_equal(codes.cpu().numpy(), rc)
    assert np.array_equal(lut.cpu().view(torch.int16).numpy().view(np.uint16), rl)
    assert np.array_equal(sal.cpu().numpy(), rs)
    assert np.array_equal(ex.idx.cpu().numpy(), rex[0])
    out = torch.full((R, C + pad + 1), 7.0, dtype=torch.float16, device=DEV)
    lib = _lib.ready(out.device)
    _lib.check(lib.crbq_unpack(codes.data_ptr(), codes.stride(0), lut.data_ptr(), sal.data_ptr(),
                               ex.idx.data_ptr(), ex.val.data_ptr(), ex.idx.numel(), 1, R, C,
                               out[:, 1:].data_ptr(), out.stride(0), _lib.stream_of(out)), "unpack")
    torch.cuda.synchronize()
    assert torch.equal(out[:, 1:C + 1].view(torch.int16), Qb[:, :C].contiguous().view(torch.int16))
    assert (out[:, :1] == 7).all() and (out[:, C + 1:] == 7).all()


def test_pack_reports_structure_errors():
    print("pack errors", flush=True)
    from crb_amd._lib import CrbqError
    q, masks = structured(8, 256, seed=3)
    col = int(np.nonzero(masks[2, :128] == 1)[0][0])
    bad = q.copy()
    bad[2, col] = np.float16(0.123)            # one out-of-table value: an exception
    codes, lut, sal, ex = _k().pack(torch.from_numpy(bad).to(DEV), torch.from_numpy(masks).to(DEV))
    assert ex.idx.tolist() == [2 * 256 + col]
    with pytest.raises(CrbqError, match="exception list"):
        _k().pack(torch.from_numpy(bad).to(DEV), torch.from_numpy(masks).to(DEV), ex_cap=0)
    m2 = masks.copy()
    m2[5, int(np.nonzero(masks[0, :128] == 3)[0][0])] = 1
    with pytest.raises(CrbqError, match="salient columns differ"):
        _k().pack(torch.from_numpy(q).to(DEV), torch.from_numpy(m2).to(DEV))
    # a valid layer afterwards still packs (the status word is cleared per call)
    _k().pack(torch.from_numpy(q).to(DEV), torch.from_numpy(masks).to(DEV))


@pytest.mark.parametrize("method,dtype,R,C", [("crb", torch.float16, 96, 320),
                                              ("braq", torch.bfloat16, 64, 384),
                                              ("crbog", torch.float16, 48, 256)])
def test_quantized_layer_round_trip(method, dtype, R, C):
    """Layers from the block loop (LayerQuantizer with keep_masks) pack and
    unpack bit for bit (C = 320: a ragged last block of 64 columns, above the
    salient search's 50-column minimum)."""
    print(f"pack quantized {method} {R}x{C}", flush=True)
    from crb_amd.driver import LayerQuantizer, Sublayer
    g = torch.Generator().manual_seed(R * C)
    W = (torch.randn(R, C, generator=g) * 0.02).to(dtype).to(DEV)
    X = (torch.randn(4, 256, C, generator=g) * torch.exp(torch.randn(C, generator=g))).to(dtype)
    lq = LayerQuantizer([Sublayer("w", W, "x")], method=method, keep_masks=True)
    lq.add_batch("x", X.to(DEV))
    lq.quantize()
    codes, lut, sal, ex = _k().pack(W, lq.masks["w"])
    assert torch.equal(_k().unpack(codes, lut, sal, C, ex).view(torch.int16), W.view(torch.int16))
    rc, rl, rs, rex, st = pack_ref(W.view(torch.int16).cpu().numpy().view(np.uint16),
                                   lq.masks["w"].cpu().numpy(), bf16=dtype == torch.bfloat16)
    assert st == 0 and np.array_equal(codes.cpu().numpy(), rc)
    assert np.array_equal(ex.idx.cpu().numpy(), rex[0])


@pytest.mark.parametrize("R,C,dtype,nvec", [(37, 300, torch.float16, 1),
                                            (256, 1024, torch.float16, 3),
                                            (130, 640, torch.bfloat16, 8),
                                            (1000, 4096, torch.bfloat16, 1),
                                            (512, 2000, torch.float16, 5),
                                            (64, 1000, torch.float16, 16),
                                            (17, 136, torch.bfloat16, 11)])
def test_gemv_against_float64(R, C, dtype, nvec):
    print(f"gemv {R}x{C} {dtype} nvec={nvec}", flush=True)
    q, masks = structured(R, C, seed=7 * R + C, n_odd=R // 8)
    Q = _q16(q, dtype)
    codes, lut, sal, ex = _k().pack(Q, torch.from_numpy(masks).to(DEV))
    g = torch.Generator().manual_seed(C)
    xf = torch.randn(nvec, C + 24, generator=g)
    x = xf.to(dtype).to(DEV)[:, :C]        # rows strided by C + 24
    y = _k().gemv_packed(codes, lut, sal, C, x, ex)
    torch.cuda.synchronize()
    W64 = Q.double().cpu()
    x64 = x.double().cpu()
    ref = x64 @ W64.t()
    scale = x64.abs() @ W64.abs().t()
    err = (y.double().cpu() - ref).abs()
    assert (err <= 1e-5 * scale + 1e-30).all(), float((err / scale.clamp_min(1e-30)).max())


@pytest.mark.parametrize("R,C,T,dtype", [(37, 300, 17, torch.float16),      # ragged everything
                                          (256, 1024, 64, torch.bfloat16),
                                          (130, 640, 100, torch.float16),
                                          (1000, 4096, 33, torch.bfloat16),   # split K
                                          (300, 2048, 250, torch.float16),
                                          (64, 128, 1, torch.float16)])
def test_gemm_against_float64(R, C, T, dtype):
    """crbq_gemm_packed against float64 products of the unpacked weights,
    same bar as the GEMV; the split-K and single-pass launches are both
    covered (the split depends on the shapes)."""
    print(f"gemm {R}x{C} T={T} {dtype}", flush=True)
    from crb_amd import _lib
    q, masks = structured(R, C, seed=5 * R + C, n_odd=R // 8)
    Q = _q16(q, dtype)
    codes, lut, sal, ex = _k().pack(Q, torch.from_numpy(masks).to(DEV))
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, C + 40, generator=g).to(dtype).to(DEV)[:, :C]
    y = _k().gemm_packed(codes, lut, sal, C, x, ex)
    torch.cuda.synchronize()
    W64 = Q.double().cpu()
    x64 = x.double().cpu()
    ref = x64 @ W64.t()
    scale = x64.abs() @ W64.abs().t()
    err = (y.double().cpu() - ref).abs()
    assert (err <= 1e-5 * scale + 1e-30).all(), float((err / scale.clamp_min(1e-30)).max())
    # which of these shapes split: those for which the header's minimum asks
    # for partials (the number of splits comes from the modelled time)
    tiles = -(-R // 128) * -(-T // (128 if T > 64 else 64))
    split = min(512 // tiles, -(-C // 128) // 8) > 1
    lib = _lib.load()
    assert (lib.crbq_gemm_packed_workspace_size(R, C, T) > 0) == split


def test_gemm_deterministic_and_matches_gemv():
    """Split-K partials are summed in a fixed order: repeated calls are
    bitwise equal; the first 16 tokens agree with the GEMV to the same bar."""
    print("gemm determinism", flush=True)
    q, masks = structured(1000, 4096, seed=9, n_odd=100)
    Q = torch.from_numpy(q).to(DEV)
    codes, lut, sal, ex = _k().pack(Q, torch.from_numpy(masks).to(DEV))
    x = torch.randn(40, 4096, generator=torch.Generator().manual_seed(2)).half().to(DEV)
    y1 = _k().gemm_packed(codes, lut, sal, 4096, x, ex)
    y2 = _k().gemm_packed(codes, lut, sal, 4096, x, ex)
    assert torch.equal(y1, y2)
    yv = _k().gemv_packed(codes, lut, sal, 4096, x[:16], ex)
    scale = x[:16].double().abs() @ Q.double().abs().t()
    assert ((y1[:16].double() - yv.double()).abs() <= 2e-5 * scale + 1e-30).all()


def test_packed_linear_forward():
    print("packed linear", flush=True)
    from crb_amd.packed import PackedLinear
    q, masks = structured(192, 512, seed=11, n_odd=12)
    lin = torch.nn.Linear(512, 192).to(DEV).half()
    lin.weight.data = torch.from_numpy(q).to(DEV)
    pl = PackedLinear.from_linear(lin, torch.from_numpy(masks).to(DEV))
    assert torch.equal(pl.weight(), lin.weight.data)
    assert pl.packed_bytes() * 8 / (192 * 512) < 3.1
    g = torch.Generator().manual_seed(0)
    for ntok in (1, 8, 40, 400):           # 2, 16: GEMV; 80: GEMM; 800: unpack + dense
        x = torch.randn(2, ntok, 512, generator=g).half().to(DEV)
        with torch.no_grad():
            got = pl(x).float()
            want = torch.nn.functional.linear(x.float(), lin.weight.float(), lin.bias.float())
        assert got.shape == (2, ntok, 192)
        assert ((got - want).abs() <= 2e-3 * want.abs() + 2e-3).all(), ntok


def test_stack_pack_option():
    """StackQuantizer(pack=True) leaves PackedLinear modules that decode to
    exactly the weights the unpacked run produces."""
    print("stack pack", flush=True)
    from test_gpu_stack import _samples, tiny_model
    from crb_amd.packed import PackedLinear
    from crb_amd.stack import StackQuantizer, find_linears
    samples = _samples(n=6, seq=96)
    a = tiny_model("opt")
    StackQuantizer(a, chunk=3).run(samples)
    b = tiny_model("opt")
    stats = StackQuantizer(b, chunk=3, pack=True).run(samples)
    assert all(st.packed_bytes > 0 for st in stats)
    for la, lb in zip(a.model.decoder.layers, b.model.decoder.layers):
        dense = find_linears(la)
        for name, m in dense.items():
            mod = lb
            for p in name.split("."):
                mod = getattr(mod, p)
            assert isinstance(mod, PackedLinear), name
            assert torch.equal(mod.weight(), m.weight.data), name
    with torch.no_grad():
        x = samples[:1, :5]
        la_, lb_ = a(x).logits.float(), b(x).logits.float()
    assert torch.allclose(la_, lb_, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("R,C,T,dtype,bias,n_odd", [
    (17, 136, 1, torch.float16, True, 0), (33, 300, 16, torch.bfloat16, True, 3),
    (256, 1024, 64, torch.float16, True, 70),          # one launch, two list rounds
    (300, 1920, 17, torch.float16, False, 4),          # split sums
    (257, 640, 65, torch.bfloat16, True, 5), (250, 520, 129, torch.float16, True, 2),
    (515, 2049, 300, torch.bfloat16, True, 9), (1, 9, 3, torch.float16, True, 0)])
def test_linear_packed_against_float64(R, C, T, dtype, bias, n_odd):
    """crbq_linear_packed (sums, exceptions, bias, one rounding) against
    float64: half an ulp of the 16-bit result (2^-11 or 2^-8 relative) plus the
    GEMV's fp32 bar; columns past R untouched; PackedLinear takes it for
    activations and bias of the weights' dtype."""
    print(f"linear packed {R}x{C} T={T} {dtype} odd={n_odd}", flush=True)
    from crb_amd.packed import PackedLinear
    q, masks = structured(R, C, seed=3 * R + C, n_odd=n_odd)
    Q = _q16(q, dtype)
    codes, lut, sal, ex = _k().pack(Q, torch.from_numpy(masks).to(DEV))
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, C + 16, generator=g).to(dtype).to(DEV)[:, :C]
    b = torch.randn(R, generator=g).to(dtype).to(DEV) if bias else None
    y = _k().linear_packed(codes, lut, sal, C, x, b, ex)
    assert y.dtype == dtype and y.shape == (T, R)
    x64, W64 = x.double().cpu(), Q.double().cpu()
    ref = x64 @ W64.t() + (b.double().cpu() if bias else 0.0)
    scale = x64.abs() @ W64.abs().t() + (b.double().cpu().abs() if bias else 0.0)
    half_ulp = 2.0 ** (-11 if dtype == torch.float16 else -8)
    err = (y.double().cpu() - ref).abs()
    assert (err <= half_ulp * ref.abs() + 1.1e-5 * scale + 2.0 ** -25).all()
    assert torch.equal(PackedLinear(codes, lut, sal, C, b, ex)(x), y)


def test_packed_linear_bias_forms():
    """A bias that broadcasts or takes a gradient is added on its own, as
    before the product kernels took the bias."""
    from crb_amd.packed import PackedLinear
    q, masks = structured(48, 256, seed=5)
    Q = _q16(q, torch.float16)
    codes, lut, sal, ex = _k().pack(Q, torch.from_numpy(masks).to(DEV))
    x = torch.randn(20, 256, generator=torch.Generator().manual_seed(1)).half().to(DEV)
    plain = PackedLinear(codes, lut, sal, 256, None, ex)(x)
    one = torch.full((1,), 0.5, dtype=torch.float16, device=DEV)
    assert torch.equal(PackedLinear(codes, lut, sal, 256, one, ex)(x), plain + one)
    b = torch.linspace(-1, 1, 48, device=DEV).half().requires_grad_()
    y = PackedLinear(codes, lut, sal, 256, b, ex)(x)
    assert torch.equal(y, plain + b)
    y.sum().backward()
    assert torch.equal(b.grad, torch.full_like(b, 20.0))


@pytest.mark.parametrize("T", [1, 64, 1024])
def test_packed_linear_bias_parameter(T):
    """A bias assigned as a Parameter after construction, on each of the three
    routes: the product without bias plus that bias, and its gradient."""
    print(f"packed linear bias parameter T={T}", flush=True)
    from crb_amd.packed import PackedLinear
    q, masks = structured(48, 256, seed=6)
    codes, lut, sal, ex = _k().pack(_q16(q, torch.float16), torch.from_numpy(masks).to(DEV))
    x = torch.randn(T, 256, generator=torch.Generator().manual_seed(T)).half().to(DEV)
    b = torch.linspace(-1, 1, 48, device=DEV).half()
    pl = PackedLinear(codes, lut, sal, 256, torch.zeros_like(b), ex)
    pl.bias = torch.nn.Parameter(b.clone())
    y = pl(x)
    # two fp16 roundings, of a product and of a sum, of at most its size plus 1
    plain = PackedLinear(codes, lut, sal, 256, None, ex)(x)
    assert ((y - (plain + b)).abs() <= 2.0 ** -10 * (plain.abs() + 1)).all()
    y.sum().backward()
    assert torch.equal(pl.bias.grad, torch.full_like(b, float(T)))


@pytest.mark.parametrize("T", [1, 64, 1024])
def test_packed_linear_bias_transforms(T):
    """vmap over the bias, and a dual bias: values of the plain call, batch and
    tangent kept.  (torch.func.jvp and grad wrap the activations too, and a
    kernel call has never taken those.)"""
    print(f"packed linear bias transforms T={T}", flush=True)
    import torch.autograd.forward_ad as fwAD
    from crb_amd.packed import PackedLinear
    q, masks = structured(48, 256, seed=6)
    codes, lut, sal, ex = _k().pack(_q16(q, torch.float16), torch.from_numpy(masks).to(DEV))
    x = torch.randn(T, 256, generator=torch.Generator().manual_seed(T)).half().to(DEV)
    b, t = torch.linspace(-1, 1, 48, device=DEV).half(), torch.ones(48, device=DEV).half()
    pl = PackedLinear(codes, lut, sal, 256, b, ex)
    # two fp16 roundings, of a product and of a sum, of at most its size plus 1
    bar = 2.0 ** -10 * (pl(x).abs() + 2)

    def f(v):
        return torch.func.functional_call(pl, {"bias": v}, (x,))
    ys = torch.func.vmap(f)(torch.stack([b, b]))
    assert ((ys - pl(x)).abs() <= bar).all()
    with fwAD.dual_level():
        y, ty = fwAD.unpack_dual(f(fwAD.make_dual(b, t)))
        assert ((y - pl(x)).abs() <= bar).all() and torch.equal(ty, t.expand(T, 48))


def test_gemm_packed_workspace_alignment():
    """Split products from a workspace that is only 4-byte aligned: bitwise
    those from an aligned one."""
    print("gemm packed workspace alignment", flush=True)
    from crb_amd import _lib
    R, C, T = 300, 1920, 17
    q, masks = structured(R, C, seed=12)
    codes, lut, sal, _ = _k().pack(_q16(q, torch.float16), torch.from_numpy(masks).to(DEV))
    x = torch.randn(T, C, generator=torch.Generator().manual_seed(3)).half().to(DEV)
    lib = _lib.ready(x.device)
    n = int(lib.crbq_gemm_packed_workspace_size(R, C, T))
    assert n > 0
    ws = torch.empty(n // 4 + 4, device=DEV)
    assert ws.data_ptr() % 16 == 0
    got = []
    for off in (0, 1):
        y = torch.empty(T, R, device=DEV)
        z = torch.empty(T, R, dtype=torch.float16, device=DEV)
        w, st = ws[off:].data_ptr(), _lib.stream_of(x)
        _lib.check(lib.crbq_gemm_packed(codes.data_ptr(), codes.stride(0), lut.data_ptr(),
                                        sal.data_ptr(), 0, 0, 0, 1, R, C, x.data_ptr(), C, T,
                                        y.data_ptr(), R, w, n, st), "gemm")
        _lib.check(lib.crbq_linear_packed(codes.data_ptr(), codes.stride(0), lut.data_ptr(),
                                          sal.data_ptr(), 0, 0, 0, 1, R, C, x.data_ptr(), C, T, 0,
                                          z.data_ptr(), R, w, n, st), "linear")
        got.append((y, z))
    torch.cuda.synchronize()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert torch.equal(got[0][0].half(), got[0][1])


@pytest.mark.parametrize("R,C,T,dtype", [
    (129, 640, 17, torch.float16), (1000, 1000, 129, torch.bfloat16),       # one row tile
    (33000, 300, 33, torch.float16), (33001, 300, 70, torch.bfloat16),      # two, one launch
    (8300, 2049, 33, torch.bfloat16), (4099, 2050, 130, torch.float16)])    # two, split sums
def test_gemm_packed_row_tiles(R, C, T, dtype):
    """One 16-row tile per wavefront where workgroups are few, two where they
    fill the chip, at ragged rows, columns and tokens: both products against
    float64 at the other tests' bars."""
    print(f"gemm row tiles {R}x{C} T={T} {dtype}", flush=True)
    q, masks = structured(500, C, seed=R + T, n_odd=0)
    rep = -(-R // 500)
    Q = _q16(np.tile(q, (rep, 1))[:R], dtype)
    Q[::97, 5] = 3.0                     # exceptions, up to 341 rows of them
    codes, lut, sal, ex = _k().pack(Q, torch.from_numpy(np.tile(masks, (rep, 1))[:R]).to(DEV))
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, C + 40, generator=g).to(dtype).to(DEV)[:, :C]
    x64, W64 = x.double(), Q.double()
    ref, scale = x64 @ W64.t(), x64.abs() @ W64.abs().t()
    y = _k().gemm_packed(codes, lut, sal, C, x, ex)
    assert ((y.double() - ref).abs() <= 1e-5 * scale + 1e-30).all()
    n = min(ex.idx.numel(), 256)
    few = type(ex)(ex.idx[:n], ex.val[:n], ex.delta[:n])
    b = torch.randn(R, generator=g).to(dtype).to(DEV)
    z = _k().linear_packed(codes, lut, sal, C, x, b, few)
    Wf = _k().unpack(codes, lut, sal, C, few).double()
    ref, scale = x64 @ Wf.t() + b.double(), x64.abs() @ Wf.abs().t() + b.double().abs()
    half_ulp = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert ((z.double() - ref).abs() <= half_ulp * ref.abs() + 1.1e-5 * scale + 2.0 ** -25).all()


@pytest.mark.parametrize("R,C,T,least", [(300, 1920, 17, 0), (4096, 1920, 64, 0),
                                         (1000, 4096, 33, 4)])
def test_gemm_packed_small_workspace(R, C, T, least):
    """crbq_gemm_packed with less workspace than it asks for: with the stated
    minimum (none where splits of 8 blocks are not possible) it runs with
    fewer splits, below that it is refused; crbq_linear_packed is refused
    below its full size."""
    print(f"gemm packed small workspace {R}x{C} T={T}", flush=True)
    from crb_amd import _lib
    q, masks = structured(min(R, 300), C, seed=13)
    rep = -(-R // 300)
    Q = torch.from_numpy(np.tile(q, (rep, 1))[:R]).to(DEV)
    codes, lut, sal, _ = _k().pack(Q, torch.from_numpy(np.tile(masks, (rep, 1))[:R]).to(DEV))
    x = torch.randn(T, C, generator=torch.Generator().manual_seed(3)).half().to(DEV)
    lib = _lib.ready(x.device)
    full, slice_ = int(lib.crbq_gemm_packed_workspace_size(R, C, T)), 4 * T * R
    assert full > least * slice_
    ws = torch.empty(full, dtype=torch.uint8, device=DEV)

    def call(fn, y, w, n):
        return fn(codes.data_ptr(), codes.stride(0), lut.data_ptr(), sal.data_ptr(), 0, 0, 0, 1,
                  R, C, x.data_ptr(), C, T, *((0,) if fn is lib.crbq_linear_packed else ()),
                  y.data_ptr(), R, w, n, _lib.stream_of(x))
    ref = x.double() @ Q.double().t()
    bar = 1e-5 * (x.double().abs() @ Q.double().abs().t()) + 1e-30
    for n in (least * slice_, full - 1, full):
        y = torch.empty(T, R, device=DEV)
        _lib.check(call(lib.crbq_gemm_packed, y, ws.data_ptr() if n else 0, n), "gemm")
        assert ((y.double() - ref).abs() <= bar).all(), n
    z = torch.empty(T, R, dtype=torch.float16, device=DEV)
    refused = -3                          # CRBQ_ERR_WORKSPACE
    assert call(lib.crbq_linear_packed, z, ws.data_ptr(), full - 1) == refused
    if least:
        assert call(lib.crbq_gemm_packed, y, ws.data_ptr(), least * slice_ - 1) == refused
        assert call(lib.crbq_gemm_packed, y, 0, 0) == refused


@pytest.mark.parametrize("R,C", [(1, 1), (5, 8), (1025, 9), (2047, 17), (515, 24), (257, 65),
                                 (131, 136), (67, 1032), (9, 2049), (70_000_003, 8)])
def test_unpack_thread_shapes(R, C):
    """Unpack against the format statement where its threads change shape (as
    many along a row as it has chunks of 8 columns, the rest down the rows),
    and at more rows than a launch has four-row workgroups."""
    print(f"unpack shapes {R}x{C}", flush=True)
    nblk = -(-C // 128)
    g = torch.Generator(device=DEV).manual_seed(R % 1000 + C)
    codes = torch.randint(0, 256, (R, nblk * 32), device=DEV, generator=g, dtype=torch.uint8)
    lut = torch.randint(-32768, 32767, (R, nblk, 8), device=DEV, generator=g,
                        dtype=torch.int16).view(torch.float16)
    sal = torch.randint(0, 256, (nblk, 16), device=DEV, generator=g, dtype=torch.uint8)
    Q = _k().unpack(codes, lut, sal, C).view(torch.int16)
    bits = lut.view(torch.int16)
    for c in range(C):
        code = (codes[:, c // 4] >> (2 * (c % 4))) & 3
        s = int(sal[c // 128, (c % 128) // 8]) >> (c % 8) & 1
        want = bits[:, c // 128].gather(1, (code.long() + 4 * s)[:, None])[:, 0]
        assert torch.equal(Q[:, c], want), c


@pytest.mark.parametrize("R,C,n_odd", [(20, 300, 2000), (7, 1000, 12), (33, 128, 33)])
def test_pack_many_exceptions(R, C, n_odd):
    """Block rows with exceptions, from a few of a workgroup's 16 to all of
    them, one wavefront each in turn: against the format statement."""
    print(f"pack many exceptions {R}x{C} odd={n_odd}", flush=True)
    q, masks = structured(R, C, seed=R, n_odd=n_odd)
    codes, lut, sal, ex = _k().pack(_q16(q, torch.float16), torch.from_numpy(masks).to(DEV),
                                    ex_cap=R * C)
    rc, rl, rs, rex, st = pack_ref(q.view(np.uint16), masks, ex_cap=R * C)
    assert st == 0 and np.array_equal(codes.cpu().numpy(), rc)
    assert np.array_equal(lut.cpu().view(torch.int16).numpy().view(np.uint16), rl)
    assert np.array_equal(sal.cpu().numpy(), rs)
    assert np.array_equal(ex.idx.cpu().numpy(), rex[0])
    assert np.array_equal(ex.val.cpu().view(torch.int16).numpy().view(np.uint16), rex[1])
    assert np.array_equal(ex.delta.cpu().numpy(), rex[2])
