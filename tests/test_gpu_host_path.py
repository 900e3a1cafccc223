"""WALinear.forward and sparse_attention through the extension's single calls: every form of tensor that they accept
gives the bits of the general path, and what is refused is refused as before."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def mods(built_lib):
    import quant
    from sqamd import block_sparse_attention_lut as bsa
    from sqamd import capi
    from sqamd.qlinear import WALinear
    return quant, bsa, capi, WALinear


def _linear(WALinear, k, n, g, bias=True):
    gen = torch.Generator(device=DEV).manual_seed(k + n)
    lin = WALinear(k, n, group_size=g, bias=bias, dev=DEV)
    lin.weight = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=gen)
    lin.zeros_scales = torch.stack([torch.randint(64, 80, (n, k // g), device=DEV, generator=gen).half(),
                                    torch.rand((n, k // g), device=DEV, generator=gen).half() * 0.01 + 0.001], -1).reshape(n, -1)
    if bias:
        lin.bias = torch.randn((1, n), device=DEV, generator=gen).half()
    return lin


@pytest.mark.parametrize("shape", [(256,), (1, 256), (7, 256), (2, 3, 256), (2, 2, 5, 256), (0, 256), (2, 0, 256)])
def test_linear_of_any_rank_and_stride(mods, shape):
    quant, _, _, WALinear = mods
    lin = _linear(WALinear, 256, 96, 64)
    x = torch.randn(shape, device=DEV).half()
    out_shape = shape[:-1] + (96,)
    res = torch.randn(out_shape, device=DEV).half()
    rows = x.reshape(1, x.numel() // 256, 256)
    ref = quant.gemm_awq_fused_ut(rows, lin.weight, lin.zeros_scales, lin.bias, res.reshape(1, -1, 96) if x.numel() else None,
                                  "relu", 96, 64).reshape(out_shape)
    y = lin(x, residual=res, act="relu")
    assert y.shape == out_shape and torch.equal(y, ref)
    wide = torch.empty(shape[:-1] + (512,), device=DEV, dtype=torch.float16)
    wide[..., ::2] = x
    res_t = res.transpose(0, -1).contiguous().transpose(0, -1)
    assert torch.equal(lin(wide[..., ::2], residual=res_t, act="relu"), ref)
    with torch.enable_grad():
        y = lin(x.clone().requires_grad_(True), residual=res, act="relu")
    assert not y.requires_grad and torch.equal(y, ref)


def test_linear_refuses_and_finds_replaced_buffers(mods):
    _, _, _, WALinear = mods
    lin = _linear(WALinear, 256, 96, 64)
    x = torch.randn((2, 256), device=DEV).half()
    ref = lin(x)
    for bad, err in ((dict(residual=torch.zeros((2, 95), device=DEV).half()), RuntimeError),
                     (dict(residual=torch.zeros((2, 96), device=DEV)), RuntimeError), (dict(act="gelu"), ValueError)):
        with pytest.raises(err):
            lin(x, **bad)
    with pytest.raises(RuntimeError, match="must be on CUDA"):
        lin(x.cpu())
    with pytest.raises(RuntimeError, match="dtype"):
        lin(x.float())
    with pytest.raises(ValueError):
        lin(x[:, :128])
    bias, weight = lin.bias, lin.weight
    del lin.bias, lin.weight
    lin.bias, lin.weight = bias, torch.nn.Parameter(weight, requires_grad=False)  # no buffers any more
    assert torch.equal(lin(x), ref)


@pytest.mark.parametrize("heads,rows,d", [(3, 2, 64), (3, 65, 128), (5, 700, 64), (130, 40, 64)])
def test_decode_attention_routes_agree(mods, heads, rows, d):
    """Direct call and general path on: contiguous caches, a slice of a longer cache, a strided q, a mask of another
    type; equal bits.  Tensors that the direct call cannot address give None and are copied by the general path."""
    quant, bsa, capi, _ = mods
    gen = torch.Generator(device=DEV).manual_seed(rows)
    mk = lambda *s: torch.randn(s, device=DEV, generator=gen).half()
    q, kc, vc = mk(2, heads, 1, d), mk(2, heads, rows + 3, d), mk(2, heads, rows + 3, d)
    k, v = kc[:, :, :rows], vc[:, :, :rows]
    mask = torch.zeros((2, 1, 1, rows), device=DEV)
    mask[1, :, :, :rows // 2] = float("-inf")
    for m in (None, mask.half()):
        ref = capi.decode_attention(q, k, v, rows, 0.1, mask=m).view(2, heads, 1, d)
        for kk, vv in ((k, v), (k.contiguous(), v.contiguous())):
            assert torch.equal(quant.decode_attention(q, kk, vv, m, 0.1), ref)
        qs = mk(2, 1, heads, d).transpose(1, 2)
        qs.copy_(q)
        assert torch.equal(bsa.sparse_attention(qs, k, v, 0.1, None, attention_mask=None if m is None else mask), ref)
        off = torch.empty((2, heads, rows, d + 4), dtype=torch.float16, device=DEV)[..., 4:]
        off.copy_(k)
        assert quant.decode_attention(q, off, v, m, 0.1) is None
        assert torch.equal(bsa.sparse_attention(q, off, v, 0.1, None, attention_mask=m), ref)
    assert quant.decode_attention(q.float(), k, v, None, 0.1) is None
    assert quant.decode_attention(q, k, v[:, :, :rows - 1], None, 0.1) is None
    assert quant.decode_attention(q, k, v, mask, 0.1) is None


def test_lut_attention_routes_agree(mods):
    quant, bsa, capi, _ = mods
    q, k, v = (torch.randn((2, 3, 100, 64), device=DEV).half() for _ in range(3))
    lut = torch.tensor([[0, 0], [0, 1]], device=DEV).expand(3, 2, 2)
    ref = capi.lut_attention(q, k, v, lut.contiguous(), 0.125, True)
    assert quant.lut_attention(q, k, v, lut, 0.125, True) is None  # an expanded table: copied by the general path
    assert torch.equal(bsa.sparse_attention(q, k, v, 0.125, lut), ref)
    assert torch.equal(quant.lut_attention(q, k, v, lut.contiguous(), 0.125, True), ref)
    assert torch.equal(quant.lut_attention(q, k, v, lut.int().contiguous(), 0.125, True), ref)
    kt = k.transpose(1, 2).contiguous().transpose(1, 2)
    assert quant.lut_attention(q, kt, v, lut.contiguous(), 0.125, True) is None  # k and v laid out differently
    assert torch.equal(bsa.sparse_attention(q, kt, v, 0.125, lut), ref)
    assert torch.equal(bsa.sparse_attention(q, k, v, 0.125, lut.cpu()), ref)
    x = torch.randn((1, 1, 64, 96), device=DEV).half()
    assert quant.lut_attention(x, x, x, lut.contiguous(), 0.125, True) is None
    with pytest.raises(capi.SqError) as e:
        bsa.sparse_attention(x, x, x, 0.125, lut)
    assert e.value.code == capi.SQ_ERR_BAD_SHAPE


@pytest.mark.parametrize("b,t,rows", [(2, 0, 0), (2, 1, 1), (3, 5, 1), (9, 2, 1)])
def test_logits_have_a_row_per_last_token(built_lib, b, t, rows):
    """With the logits' own kernel (up to 8 sequences) as with the library's product (9)."""
    from sqamd.opt_decode import OPTDecoder
    model = OPTDecoder(layers=1, hidden=512, heads=4, ffn=512, vocab=64, max_pos=64, dev=DEV)
    logits = model(torch.zeros((b, t), dtype=torch.long, device=DEV), model.new_cache(b, 8), 0)
    assert logits.shape == (b, rows, 64)
