"""GPU parity of the LUT block-sparse attention kernel (through the C ABI) against the
float64 dense-masked oracle.  Bar: max|out - ref| <= 1e-2 * max|ref| (fp16 in/out, fp16
probabilities into the matrix core, fp32 softmax state), same bar as the linear path."""
import numpy as np
import pytest
import torch

import lut_attention_oracle as att

pytestmark = pytest.mark.gpu
TOL = 1e-2


@pytest.fixture(scope="module")
def capi(built_lib):
    from sqamd import capi as c
    c.lib()
    return c


def run_case(capi, z, h, s, d, density, causal, seed=0, lut_dtype=torch.int64, scale=None):
    rng = np.random.default_rng(seed)
    q = rng.normal(size=(z, h, s, d)).astype(np.float16)
    k = rng.normal(size=(z, h, s, d)).astype(np.float16)
    v = rng.normal(size=(z, h, s, d)).astype(np.float16)
    nb = (s + 63) // 64
    lut = att.layout_to_lut(att.synth_layout(h, nb, density, causal, seed=seed + 1))
    scale = scale if scale is not None else 1.0 / np.sqrt(d)
    ref = att.attention_ref(q, k, v, lut, scale, causal)
    out = capi.lut_attention(torch.from_numpy(q).cuda(), torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(),
                             torch.from_numpy(lut).to(lut_dtype).cuda(), scale, causal)
    torch.cuda.synchronize()
    out = out.float().cpu().numpy().astype(np.float64)
    assert np.all(np.isfinite(out))
    err = np.max(np.abs(out - ref))
    assert err <= TOL * np.max(np.abs(ref)), "z=%d h=%d s=%d d=%d causal=%s: err %.3e" % (z, h, s, d, causal, err)
    return out, ref


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("s,density", [(64, 1.0), (128, 0.5), (512, 0.25), (200, 0.5), (1000, 0.3)])
def test_attention_parity(capi, d, causal, s, density):
    run_case(capi, 2, 3, s, d, density, causal, seed=s + d)


def test_attention_bert_large_shape(capi):
    # batch 8 x 16 heads x 512 x 64, ~25 % density, non-causal (the benchmark's BERT-large configuration)
    run_case(capi, 8, 16, 512, 64, 0.25, False, seed=5)


def test_attention_long_sequence_causal_int32_lut(capi):
    run_case(capi, 1, 4, 4096, 128, 0.26, True, seed=6, lut_dtype=torch.int32)


def test_attention_properties(capi):
    z, h, s, d = 1, 2, 256, 64
    rng = np.random.default_rng(9)
    q = torch.from_numpy(rng.normal(size=(z, h, s, d)).astype(np.float16)).cuda()
    k = torch.from_numpy(rng.normal(size=(z, h, s, d)).astype(np.float16)).cuda()
    lay = att.synth_layout(h, 4, 0.5, True, seed=2)
    lut = torch.from_numpy(att.layout_to_lut(lay)).cuda()
    # constant V comes back unchanged (softmax weights sum to one)
    vc = torch.arange(d, dtype=torch.float16).repeat(z, h, s, 1).cuda()
    out = capi.lut_attention(q, k, vc, lut, 0.125, True)
    assert torch.allclose(out.float(), vc.float(), atol=0.05)
    # causal: query 0 sees only key 0 -> returns that V row exactly
    v = torch.from_numpy(rng.normal(size=(z, h, s, d)).astype(np.float16)).cuda()
    out = capi.lut_attention(q, k, v, lut, 0.125, True)
    assert torch.equal(out[:, :, 0], v[:, :, 0])
    # a LUT padded with repeated entries, and one with more columns than blocks, give the same result
    lut_np = att.layout_to_lut(lay)
    padded = np.concatenate([lut_np, np.repeat(lut_np[:, :, -1:], 3, axis=2)], axis=2)
    out2 = capi.lut_attention(q, k, v, torch.from_numpy(padded).cuda(), 0.125, True)
    assert torch.equal(out, out2)
    # determinism
    assert torch.equal(out, capi.lut_attention(q, k, v, lut, 0.125, True))


def test_sparse_attention_module_api(capi):
    from sqamd.block_sparse_attention_lut import sparse_attention
    rng = np.random.default_rng(11)
    z, h, s, d = 2, 4, 192, 128
    q = torch.from_numpy(rng.normal(size=(z, h, s, d)).astype(np.float16)).cuda()
    k = torch.from_numpy(rng.normal(size=(z, h, s, d)).astype(np.float16)).cuda()
    v = torch.from_numpy(rng.normal(size=(z, h, s, d)).astype(np.float16)).cuda()
    lut = torch.from_numpy(att.layout_to_lut(att.synth_layout(h, 3, 0.7, True, seed=4))).cuda()
    out = sparse_attention(q, k, v, d ** -0.5, lut, True, 64, 64)
    ref = att.attention_ref(q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), lut.cpu().numpy(), d ** -0.5, True)
    assert np.max(np.abs(out.float().cpu().numpy() - ref)) <= TOL * np.max(np.abs(ref))
    # decode step: one query against the whole cache is dense, as in the reference
    q1 = q[:, :, -1:, :]
    o1 = sparse_attention(q1, k, v, d ** -0.5, lut, True, 64, 64)
    w = torch.softmax((q1.float() @ k.float().transpose(2, 3)) * d ** -0.5, dim=-1)
    assert torch.allclose(o1.float(), w @ v.float(), atol=2e-2, rtol=2e-2)
    with pytest.raises(ValueError):
        sparse_attention(q, k, v, 1.0, lut, True, 32, 64)


def test_attention_argument_errors(capi):
    L = capi.lib()
    import ctypes
    p = ctypes.c_void_p(4096)
    assert L.sq_lut_attention_fwd(p, p, p, p, p, 8, 1, 1, 64, 96, 1, 1.0, 0, None) == capi.SQ_ERR_BAD_SHAPE   # D
    assert L.sq_lut_attention_fwd(p, p, p, p, p, 2, 1, 1, 64, 64, 1, 1.0, 0, None) == capi.SQ_ERR_BAD_LAYOUT  # lut width
    assert L.sq_lut_attention_fwd(p, p, None, p, p, 8, 1, 1, 64, 64, 1, 1.0, 0, None) == capi.SQ_ERR_NULL_POINTER
    assert L.sq_lut_attention_fwd(p, p, p, p, p, 8, 1, 1, 0, 64, 1, 1.0, 0, None) == capi.SQ_ERR_BAD_SHAPE


@pytest.mark.parametrize("d", [64, 128])
def test_block_named_again_after_a_different_one_is_attended_twice(capi, d):
    """Only an entry equal to its predecessor is padding: rows such as [1, 3, 1, 0] visit block 1 twice
    (its keys carry double weight), [2, 2, 0, 0] visits 2 and 0 once each, entries beyond the sequence
    select nothing -- the oracle weighs every key block by its number of visits."""
    rng = np.random.default_rng(31)
    z, h, s = 2, 2, 250
    q = rng.normal(size=(z, h, s, d)).astype(np.float16)
    k = rng.normal(size=(z, h, s, d)).astype(np.float16)
    v = rng.normal(size=(z, h, s, d)).astype(np.float16)
    lut = np.array([[[0, 1, 0, 1], [1, 3, 1, 0], [2, 2, 0, 0], [3, 0, 3, 0]],
                    [[2, 0, 2, 2], [1, 1, 1, 1], [0, 9, 0, 2], [3, 2, 1, 0]]], dtype=np.int64)
    assert att.lut_to_counts(lut, 4).max() == 2
    ref = att.attention_ref(q, k, v, lut, 0.11, False)
    out = capi.lut_attention(torch.from_numpy(q).cuda(), torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(),
                             torch.from_numpy(lut).cuda(), 0.11, False)
    torch.cuda.synchronize()
    out = out.float().cpu().numpy().astype(np.float64)
    assert np.max(np.abs(out - ref)) <= TOL * np.max(np.abs(ref))


def test_query_rows_without_a_visible_key_are_nan(capi):
    # causal, query block 0 of head 0 is pointed at key block 1 only: nothing is visible -> NaN, like the
    # reference's running sums; every other row is unaffected
    rng = np.random.default_rng(32)
    z, h, s, d = 1, 2, 128, 64
    q = rng.normal(size=(z, h, s, d)).astype(np.float16)
    lut = np.array([[[1], [1]], [[0], [1]]], dtype=np.int64)
    with np.errstate(invalid="ignore"):
        ref = att.attention_ref(q, q, q, lut, 0.125, True)
    qt = torch.from_numpy(q).cuda()
    out = capi.lut_attention(qt, qt, qt, torch.from_numpy(lut).cuda(), 0.125, True).float().cpu().numpy()
    assert np.all(np.isnan(out[0, 0, :64])) and np.all(np.isnan(ref[0, 0, :64]))
    ok = np.isfinite(ref)
    assert np.array_equal(ok, np.isfinite(out))
    assert np.max(np.abs(out[ok] - ref[ok])) <= TOL * np.max(np.abs(ref[ok]))


def _assert_close_fp16(capi, q, k, v, lut, scale, causal):
    ref = att.attention_ref(q, k, v, lut, scale, causal)
    out = capi.lut_attention(torch.from_numpy(q).cuda(), torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(),
                             torch.from_numpy(lut).cuda(), scale, causal)
    torch.cuda.synchronize()
    out = out.float().cpu().numpy().astype(np.float64)
    # Every probability is rounded to fp16 once (relative 2^-11) in the product and in the row sum alike, and the output
    # once; scores, sums and exponentials are fp32.  A weighted mean of v moves by at most 2 * 2^-11 * max|v|, the
    # rounding of the output adds 2^-11 * |out|.
    assert np.all(np.isfinite(out))
    assert np.max(np.abs(out - ref)) <= 3 * 2.0 ** -11 * np.max(np.abs(v.astype(np.float64)))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("s", [1, 31, 32, 33, 63, 65, 95, 97, 161])
def test_attention_at_the_edges_of_a_step(capi, s, causal, d):
    """Sequences that end inside, at and just behind a step of 32 keys; query rows likewise."""
    rng = np.random.default_rng(s + d)
    q, k, v = (rng.normal(size=(2, 3, s, d)).astype(np.float16) for _ in range(3))
    lut = att.layout_to_lut(att.synth_layout(3, (s + 63) // 64, 0.7, causal, seed=s))
    _assert_close_fp16(capi, q, k, v, lut, d ** -0.5, causal)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_table_rows_of_more_than_64_entries(capi, dtype):
    """The table is read 64 entries at a time: padding is recognised across that border (entry 64 repeats entry 63 in
    every even row), and a growing score makes the running maximum move late in the row."""
    rng = np.random.default_rng(7)
    s, d = 66 * 64 - 5, 64
    q, k, v = (rng.normal(size=(1, 1, s, d)).astype(np.float16) for _ in range(3))
    k *= np.linspace(0.1, 3.0, s)[None, None, :, None].astype(np.float16)
    row = np.arange(66)
    rows = [np.concatenate([row[:64], row[63:65]]) if i % 2 == 0 else row for i in range(66)]
    _assert_close_fp16(capi, q, k, v, np.stack(rows)[None].astype(dtype), d ** -0.5, False)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("s", [2, 33, 64, 130, 200])
def test_strided_attention_fills_the_cache(capi, s, d):
    """Views of a fused projection [Z, S, 3, H, D]: the outputs of the contiguous path bit for bit in either output
    order, cache rows 0..S-1 hold k and v, the rows behind them are untouched."""
    z, h = 2, 3
    gen = torch.Generator(device="cuda").manual_seed(s + d)
    qkv = torch.randn((z, s, 3, h, d), device="cuda", generator=gen).half()
    q, k, v = (qkv[:, :, j].transpose(1, 2) for j in range(3))
    lut = torch.from_numpy(att.layout_to_lut(att.synth_layout(h, (s + 63) // 64, 0.6, True, seed=s))).cuda()
    ref = capi.lut_attention(q.contiguous(), k.contiguous(), v.contiguous(), lut, 0.1, True)
    kc, vc = (torch.full((z, h, s + 5, d), 7.0, dtype=torch.float16, device="cuda") for _ in range(2))
    assert capi.lut_attention_strided_ok(q, k, v, kc, vc)
    out = capi.lut_attention_strided(q, k, v, lut, 0.1, True, kc, vc, rows_first=True)
    assert torch.equal(out.transpose(1, 2), ref)
    assert torch.equal(kc[:, :, :s], k) and torch.equal(vc[:, :, :s], v)
    assert bool((kc[:, :, s:] == 7).all()) and bool((vc[:, :, s:] == 7).all())
    assert torch.equal(capi.lut_attention_strided(q, k, v, lut, 0.1, True), ref)
    from sqamd.block_sparse_attention_lut import sparse_attention
    assert torch.equal(sparse_attention(q, k, v, 0.1, lut, True), ref)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("s", [2, 65, 70 * 64 + 3])
def test_attention_without_a_table_visits_every_block(capi, s, causal):
    gen = torch.Generator(device="cuda").manual_seed(s)
    q, k, v = (torch.randn((1, 2, s, 64), device="cuda", generator=gen).half() for _ in range(3))
    nb = (s + 63) // 64
    rows = torch.arange(nb, device="cuda")
    full = rows.expand(2, nb, nb)
    if causal:  # padded with the diagonal block
        full = torch.minimum(full, rows.view(1, nb, 1))
    out = capi.lut_attention_strided(q, k, v, None, 0.125, causal)
    ref = capi.lut_attention(q, k, v, full.contiguous(), 0.125, causal)
    # the two differ in the reference maximum of the softmax: each is within 3 * 2^-11 * max|v| of the exact result
    assert torch.max((out.float() - ref.float()).abs()) <= 6 * 2.0 ** -11 * v.float().abs().max()


def test_strided_attention_refuses_what_it_cannot_address(capi):
    import ctypes
    L, p = capi.lib(), ctypes.c_void_p(4096)
    st = lambda *v: (ctypes.c_long * 12)(*v)
    good = [4096, 64, 192] * 2 + [4096, 64, 64] * 2
    call = lambda strides, q=p, kc=None, vc=None, d=64, lut=None: L.sq_lut_attention_strided(
        q, p, p, p, kc, vc, lut, 8, 1, 1, 64, d, 1, strides, 1.0, 0, None)
    assert call(None) == capi.SQ_ERR_NULL_POINTER
    assert call(st(*good), d=96) == capi.SQ_ERR_BAD_SHAPE
    assert call(st(*good), kc=p) == capi.SQ_ERR_NULL_POINTER
    assert call(st(*good), q=ctypes.c_void_p(4104)) == capi.SQ_ERR_MISALIGNED
    for i in range(9):
        assert call(st(*(good[:i] + [good[i] + 4] + good[i + 1:]))) == capi.SQ_ERR_MISALIGNED
    assert call(st(*(good[:5] + [1 << 24] + good[6:]))) == capi.SQ_ERR_BAD_SHAPE
    assert call(st(*(good[:2] + [-8] + good[3:]))) == capi.SQ_ERR_BAD_SHAPE
    x = torch.zeros((1, 1, 64, 72), dtype=torch.float16, device="cuda")
    q = x[..., :64]
    assert capi.lut_attention_strided_ok(q, q, q)
    assert not capi.lut_attention_strided_ok(x[..., 4:68], q, q)                  # rows not 16-byte aligned
    assert not capi.lut_attention_strided_ok(q, q, q.contiguous())                # k and v laid out differently
    assert not capi.lut_attention_strided_ok(q, q, q, q[:, :, :8], q[:, :, :8])   # a cache shorter than the prompt
    assert not capi.lut_attention_strided_ok(q.float(), q, q)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("z,h,s,causal", [(3, 171, 64, True), (1, 171, 161, False), (2, 86, 161, True), (1, 257, 97, True),
                                           (1, 513, 33, False), (1, 128, 256, True), (1, 129, 250, False),
                                           (4, 384, 64, True), (4, 385, 50, False), (1, 513, 129, True)])
def test_both_forms_at_the_edges_of_a_step(capi, z, h, s, causal, d):
    """Around 512 workgroups, up to which four waves share a step (513, 513, 516, 514, 513, then 512 and 516), and around
    1536, beyond which head dimension 64 runs with fewer registers (1536, 1540, 1539)."""
    rng = np.random.default_rng(h + s)
    q, k, v = (rng.normal(size=(z, h, s, d)).astype(np.float16) for _ in range(3))
    lut = att.layout_to_lut(att.synth_layout(h, (s + 63) // 64, 0.6, causal, seed=s))
    _assert_close_fp16(capi, q, k, v, lut, d ** -0.5, causal)


@pytest.mark.parametrize("d", [64, 128])
def test_strided_attention_beyond_512_workgroups(capi, d):
    z, h, s = 2, 100, 161
    gen = torch.Generator(device="cuda").manual_seed(s + d)
    qkv = torch.randn((z, s, 3, h, d), device="cuda", generator=gen).half()
    q, k, v = (qkv[:, :, j].transpose(1, 2) for j in range(3))
    lut = torch.from_numpy(att.layout_to_lut(att.synth_layout(h, (s + 63) // 64, 0.6, True, seed=s))).cuda()
    ref = capi.lut_attention(q.contiguous(), k.contiguous(), v.contiguous(), lut, 0.1, True)
    kc, vc = (torch.full((z, h, s + 3, d), 7.0, dtype=torch.float16, device="cuda") for _ in range(2))
    out = capi.lut_attention_strided(q, k, v, lut, 0.1, True, kc, vc, rows_first=True)
    assert torch.equal(out.transpose(1, 2), ref)
    assert torch.equal(kc[:, :, :s], k) and torch.equal(vc[:, :, :s], v)
    assert bool((kc[:, :, s:] == 7).all()) and bool((vc[:, :, s:] == 7).all())


def test_tables_of_another_prompt_are_refused(capi):
    """The kernel addresses the table by the heads and the length of q: a table for fewer blocks or heads would be read
    past its end, one for more blocks at the wrong rows.  Rows beyond the heads of q, and a table flattened to rows, are
    what the addressing makes of them."""
    import quant
    from sqamd.block_sparse_attention_lut import sparse_attention
    q = torch.randn((1, 2, 65, 64), device="cuda").half()
    lut = torch.tensor([[[0, 0], [0, 1]]] * 2, device="cuda")
    ref = sparse_attention(q, q, q, 0.125, lut)
    for good in (torch.cat([lut, lut]), lut.view(4, 2), lut[None].contiguous()):
        assert torch.equal(sparse_attention(q, q, q, 0.125, good), ref)
        assert torch.equal(capi.lut_attention(q, q, q, good, 0.125, True), ref)
        assert torch.equal(capi.lut_attention_strided(q, q, q, good, 0.125, True), ref)
    for bad in (lut[:, :1].contiguous(), lut[:1].contiguous(), torch.cat([lut, lut], 1), lut.view(4, 2)[:3].contiguous()):
        for call in (lambda: quant.lut_attention(q, q, q, bad, 0.125, True), lambda: sparse_attention(q, q, q, 0.125, bad),
                     lambda: sparse_attention(q, q, q, 0.125, bad.cpu()), lambda: capi.lut_attention(q, q, q, bad, 0.125, True),
                     lambda: capi.lut_attention_strided(q, q, q, bad, 0.125, True)):
            with pytest.raises(ValueError):
                call()
    for bad in (lut.float(), lut.cpu(), torch.cat([lut, lut], 2)[..., ::2]):
        with pytest.raises(ValueError):
            capi.lut_attention_strided(q, q, q, bad, 0.125, True)


def test_a_prompt_longer_than_its_table_is_refused(capi):
    from sqamd.opt_decode import OPTDecoder
    model = OPTDecoder(layers=1, hidden=512, heads=4, ffn=512, vocab=64, max_pos=256, dev="cuda")
    model.set_prefill_lut(64, 0.5)
    cache = model.new_cache(1, 130)
    ids = torch.zeros((1, 65), dtype=torch.long, device="cuda")
    assert torch.isfinite(model(ids[:, :64], cache, 0)).all()
    with pytest.raises(ValueError):
        model(ids, cache, 0)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("z,h,s", [(1, 2, 161), (3, 171, 97)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_values_that_are_not_finite_stay_with_the_rows_that_see_them(capi, bad, z, h, s, d):
    """Causal, every block visited, in both forms (up to 512 workgroups and beyond).  A query that is not finite spoils its
    own row; a key the rows behind it and its own, and nothing in front of it; a value, whose product with a masked
    probability of 0 is a NaN, the rows from the start of its block of 64 on."""
    gen = torch.Generator(device="cuda").manual_seed(s + d)
    q, k, v = (torch.randn((z, h, s, d), device="cuda", generator=gen).half() for _ in range(3))
    nb = (s + 63) // 64
    rows = torch.arange(nb, device="cuda")
    lut = torch.minimum(rows.expand(h, nb, nb), rows.view(1, nb, 1)).contiguous()
    plain = capi.lut_attention(q, k, v, lut, d ** -0.5, True)
    zi, hi, j = z - 1, h - 1, 75

    def spoilt(which):
        t = [q.clone(), k.clone(), v.clone()]
        t[which][zi, hi, j, 3] = bad
        out = capi.lut_attention(*t, lut, d ** -0.5, True)
        touched = (out != plain).any(-1)
        mine = touched[zi, hi].clone()
        touched[zi, hi] = False
        assert not bool(touched.any())  # other heads
        return out[zi, hi], mine

    out, mine = spoilt(0)
    assert mine.nonzero().flatten().tolist() == [j] and not bool(out[j].isfinite().all())
    out, mine = spoilt(1)
    assert not bool(mine[:j].any())
    if bad != bad:
        assert bool(out[j:].isnan().all())
    out, mine = spoilt(2)
    assert not bool(mine[:64].any())
    assert not bool(out[j:, 3].isfinite().any()) and bool(out[:, :3].isfinite().all()) and bool(out[:, 4:].isfinite().all())
