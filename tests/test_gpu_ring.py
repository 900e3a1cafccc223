"""The ring kernel: every tile shape, K split and group size on ragged M, N and K against the oracle; with
the scale on the sums, as few tokens take it, against (q - z) s in float64."""
import ctypes

import numpy as np
import pytest
import torch

import w4a16_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def capi(built_lib):
    from sqamd import capi as c
    c.lib()
    return c


def to_dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


# (M, N, K, g): one row; a row past a tile; K shorter than a stage, ending inside one, inside 64 columns (group size 32);
# N inside the first tile, one chunk past a tile; several hundred tiles of the smallest shapes (the last case)
CASES = [(1, 64, 128, 128), (33, 136, 640, 128), (97, 264, 1408, 128), (128, 256, 2048, 64), (100, 520, 960, 64),
         (65, 72, 416, 32), (40, 392, 1056, 32), (300, 5128, 384, 128)]


@pytest.mark.parametrize("m,n,k,g", CASES)
@pytest.mark.parametrize("shape", range(1, 9))
def test_ring_parity(capi, shape, m, n, k, g):
    d = orc.synth_linear(n, k, g, seed=7 * n + k)
    w_hat = orc.dequant_l1(d["w_l1"], d["zs_l1"], g)
    x = orc.synth_x(m, k, seed=m)
    rng = np.random.default_rng(m + n)
    bias = rng.normal(0, 1, n).astype(np.float16)
    res = rng.normal(0, 1, (m, n)).astype(np.float16)
    x64, w64 = x.astype(np.float64), w_hat.astype(np.float64)
    ref = np.maximum(x64 @ w64.T + bias.astype(np.float64), 0) + res.astype(np.float64)
    # one rounding to fp16 and K fp32 additions, each of relative error 2^-24 of the magnitudes that meet
    bound = 2.0 ** -11 * np.abs(ref) + k * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T + np.abs(bias) + np.abs(res)) + 2.0 ** -24
    w, zs, xd, bd, rd = to_dev(d["w_l1"]), to_dev(d["zs_l1"]), to_dev(x), to_dev(bias), to_dev(res)
    ws = torch.zeros(65536 + (96 << 20), dtype=torch.uint8, device=DEV)
    ran = 0
    for rest in (0, 0x10):
        for ks in (1, 2, 3, 8):
            tune = shape | rest | (ks << 8)
            y = torch.full((m, n), float("nan"), dtype=torch.float16, device=DEV)
            args = dict(bias=bd, residual=rd, act=capi.SQ_ACT_RELU, algo=capi.SQ_ALGO_RING | (tune << 8), ws=ws)
            try:
                capi.gemm_fused(xd, w, zs, n, k, g, out=y, **args)
            except capi.SqError:
                assert ks > 1  # fewer stages than parts, or no rest to split
                continue
            ran += 1
            got = y.cpu().numpy().astype(np.float64)
            assert np.all(np.abs(got - ref) <= bound), (hex(tune), np.max(np.abs(got - ref) / bound))
            assert torch.equal(y, capi.gemm_fused(xd, w, zs, n, k, g, **args)), hex(tune)
            assert capi.workspace_is_clean(ws)
    assert ran >= 1
    y = capi.gemm_fused(xd, w, zs, n, k, g, bias=bd, residual=rd, act=capi.SQ_ACT_RELU, algo=capi.SQ_ALGO_RING, ws=ws)
    assert np.all(np.abs(y.cpu().numpy().astype(np.float64) - ref) <= bound)


@pytest.mark.parametrize("m,n,k,g", CASES + [(257, 264, 320, 64), (520, 136, 1056, 32)])
def test_ring_parity_of_256_row_tiles(capi, m, n, k, g):
    """Four waves of 256 x 64: the second row of tiles full, ragged and absent."""
    test_ring_parity(capi, 9, m, n, k, g)


@pytest.mark.parametrize("shape,stage", [(1, 512), (2, 256), (3, 256), (4, 128), (5, 128), (6, 128), (7, 128), (8, 128), (9, 64)])
@pytest.mark.parametrize("short", [0, 32])
def test_ring_every_count_of_stages(capi, shape, stage, short):
    """Fewer stages than the ring has slots, as many, one and several more; the last one whole and ending early."""
    m, n, g = 37, 136, 32
    ws = torch.zeros(65536 + (8 << 20), dtype=torch.uint8, device=DEV)
    for stages in range(1, 8):
        k = stage * stages - short
        d = orc.synth_linear(n, k, g, seed=k)
        x = orc.synth_x(m, k, seed=shape)
        x64, w64 = x.astype(np.float64), orc.dequant_l1(d["w_l1"], d["zs_l1"], g).astype(np.float64)
        ref = x64 @ w64.T
        # one rounding to fp16 and K fp32 additions, as above
        bound = 2.0 ** -11 * np.abs(ref) + k * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T) + 2.0 ** -24
        w, zs, xd = to_dev(d["w_l1"]), to_dev(d["zs_l1"]), to_dev(x)
        for parts in (1, 2) if stages > 1 else (1,):
            y = capi.gemm_fused(xd, w, zs, n, k, g, algo=capi.SQ_ALGO_RING | ((shape | (parts << 8)) << 8), ws=ws)
            got = y.cpu().numpy().astype(np.float64)
            assert np.all(np.abs(got - ref) <= bound), (stages, parts, np.max(np.abs(got - ref) / bound))


@pytest.mark.parametrize("m,n,k,g", [(17, 8, 128, 128), (33, 72, 640, 128), (70, 200, 960, 64), (300, 136, 416, 32),
                                     (100, 1160, 384, 128), (9, 72, 640, 64), (3, 40, 256, 128)])
def test_ring_gate_and_up_in_one_launch(capi, m, n, k, g):
    """silu(gate) * up with both weights in every tile: outputs that end inside a tile's half, every shape, K split, and the
    sums scaled; the up projection where it is asked for."""
    d = [orc.synth_linear(n, k, g, seed=s) for s in (n, n + 1)]
    x = orc.synth_x(m, k, seed=m)
    x64 = x.astype(np.float64)
    dev = [(to_dev(i["w_l1"]), to_dev(i["zs_l1"])) for i in d]
    xd = to_dev(x)
    ws = torch.zeros(65536 + (32 << 20), dtype=torch.uint8, device=DEV)
    L, p = capi.lib(), lambda t: t.data_ptr()

    def check(y, weights, what):
        gate, up = (x64 @ w.T for w in weights)
        s = 1 / (1 + np.exp(-gate))
        ref = gate * s * up
        # errors of the sums (K fp32 additions) through d silu <= 1.1 and the product, those of exp and rcp (4 ulp of
        # fp32), one rounding to fp16
        eg, eu = (k * 2.0 ** -24 * (np.abs(x64) @ np.abs(w).T) for w in weights)
        bound = (2.0 ** -11 + 2.0 ** -20) * np.abs(ref) + 1.1 * eg * np.abs(up) + np.abs(gate * s) * eu + eg * eu + 2.0 ** -24
        err = np.abs(y.cpu().numpy().astype(np.float64) - ref)
        assert np.all(err <= bound), (what, np.max(err / bound))

    w_hat = [orc.dequant_l1(i["w_l1"], i["zs_l1"], g).astype(np.float64) for i in d]
    for shape in range(1, 10):
        for sums in (0, 0x20) if g == 128 and shape in (1, 2, 3, 5) else (0,):
            for parts in (1, 2):
                y = torch.full((m, n), float("nan"), dtype=torch.float16, device=DEV)
                rc = L.sq_w4a16_gemm_silu_dot_one(p(xd), *(p(t) for w in dev for t in w), p(y), m, n, k, g, capi.SQ_LAYOUT_L1,
                                                  capi.SQ_ALGO_RING | ((shape | sums | (parts << 8)) << 8), p(ws), ws.numel(),
                                                  capi._stream(None))
                assert rc == 0 or (parts > 1 and rc == capi.SQ_ERR_BAD_ALGO)
                if rc == 0:
                    check(y, [real_weight(i, g) for i in d] if sums else w_hat, (shape, sums, parts))
                assert capi.workspace_is_clean(ws)
    y, up = capi.gemm_silu_dot(xd, *(t for w in dev for t in w), n, k, g)
    scaled = g == 128 and m <= 64
    check(y, [real_weight(i, g) for i in d] if scaled else w_hat, "automatic")
    ref = x64 @ (real_weight(d[1], g) if scaled else w_hat[1]).T
    assert np.all(np.abs(up.cpu().numpy() - ref) <= 2.0 ** -11 * np.abs(ref) + k * 2.0 ** -24 * (np.abs(x64) @ np.abs(w_hat[1]).T) * 2 + 2.0 ** -24)


class _Epilogue(ctypes.Structure):
    """sq::Epilogue of csrc/sq_kernels.h."""
    _fields_ = [("bias", ctypes.c_void_p), ("residual", ctypes.c_void_p), ("act", ctypes.c_int), ("mul", ctypes.c_void_p)]


@pytest.mark.parametrize("m,n,k,g", [(1, 64, 128, 128), (33, 136, 640, 128), (97, 264, 1408, 64), (40, 392, 1056, 32),
                                     (300, 520, 384, 128)])
@pytest.mark.parametrize("shape", range(1, 10))
def test_ring_multiplicand(capi, shape, m, n, k, g):
    """silu(x W^T + bias) * mul + residual by every tile shape, unsplit and with K split (the last round too).  The library's
    entry points set a multiplicand only where gate and up take a launch each, which leaves the larger tiles to choices
    that a timing makes: here the launcher itself is called."""
    launch = getattr(capi.lib(), "_ZN2sq16launch_gemm_ringEPKvS1_S1_PvS2_miiiiiNS_8EpilogueEP12ihipStream_t")
    v, i = ctypes.c_void_p, ctypes.c_int
    launch.restype, launch.argtypes = i, [v] * 5 + [ctypes.c_size_t] + [i] * 5 + [_Epilogue, v]
    d = orc.synth_linear(n, k, g, seed=n + k)
    x = orc.synth_x(m, k, seed=m)
    rng = np.random.default_rng(m)
    bias, mul, res = (rng.normal(0, 1, s).astype(np.float16) for s in (n, (m, n), (m, n)))
    x64, w64, b64, mul64, r64 = (a.astype(np.float64) for a in (x, orc.dequant_l1(d["w_l1"], d["zs_l1"], g), bias, mul, res))
    t = x64 @ w64.T + b64
    y64 = t / (1 + np.exp(-t)) * mul64
    # errors of the sum (K fp32 additions) through d silu <= 1.1, those of exp, rcp and the products (8 ulp of fp32), one
    # rounding to fp16
    es = k * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T + np.abs(b64))
    xd, w, zs, bd, md, rd = (to_dev(a) for a in (x, d["w_l1"], d["zs_l1"], bias, mul, res))
    ws = torch.zeros(65536 + (96 << 20), dtype=torch.uint8, device=DEV)
    p = lambda a: None if a is None else a.data_ptr()
    for residual in (None, rd):
        ref = y64 + (0 if residual is None else r64)
        bound = 2.0 ** -11 * np.abs(ref) + 1.1 * es * np.abs(mul64) + 2.0 ** -20 * (np.abs(y64) + np.abs(ref)) + 2.0 ** -24
        ran = 0
        for word in (shape, shape | (2 << 8), shape | REST | (3 << 8)):
            y = torch.full((m, n), float("nan"), dtype=torch.float16, device=DEV)
            rc = launch(p(xd), p(w), p(zs), p(y), p(ws), ws.numel(), m, n, k, g, word,
                        _Epilogue(p(bd), p(residual), capi.SQ_ACT_SILU, p(md)), capi._stream(None))
            assert rc == 0 or (word != shape and rc == 1)  # (hipErrorInvalidValue: fewer stages than parts)
            if rc:
                continue
            ran += 1
            err = np.abs(y.cpu().numpy().astype(np.float64) - ref)
            assert np.all(err <= bound), (hex(word), np.max(err / bound))
            assert capi.workspace_is_clean(ws)
        assert ran >= 1


@pytest.mark.parametrize("pair,m,n,k,taken,other", [
    (False, 8, 7616, 8704, (1, 2), (2, 4)), (False, 16, 8192, 8448, (1, 2), (2, 4)), (True, 3, 3776, 8448, (1, 2), (2, 4)),
    (False, 32, 10944, 10880, (2, 2), (1, 1)), (False, 52, 20288, 8320, (5, 3), (3, 1)), (True, 47, 10624, 10112, (5, 3), (3, 1))])
def test_ring_plans_the_faster_shape_at_few_tokens(capi, pair, m, n, k, taken, other):
    """Shape and K split of the automatic choice with the scale on the sums, by its bits: of those timed, the other one takes 7 %
    (up to 16 tokens) to 13 % longer."""
    g = 128
    x, dev, _, _ = gated_operands(m, n, k, g, seed=n)
    ws = torch.zeros(65536 + 300 * 128 * 256 * 4, dtype=torch.uint8, device=DEV)
    L, p = capi.lib(), lambda t: t.data_ptr()

    def run(algo):
        if not pair:
            return capi.gemm_ws(x, dev[0], dev[1], n, k, g, algo=algo, ws=ws)
        y = torch.empty((m, n), dtype=torch.float16, device=DEV)
        assert L.sq_w4a16_gemm_silu_dot_one(p(x), *(p(t) for t in dev), p(y), m, n, k, g, capi.SQ_LAYOUT_L1, algo, p(ws), ws.numel(),
                                            capi._stream(None)) == 0
        return y

    forced = [run(capi.SQ_ALGO_RING | ((shape | SUMS | (parts << 8)) << 8)) for shape, parts in (taken, other)]
    assert not torch.equal(*forced)  # (the sums' order is another)
    assert torch.equal(run(capi.SQ_ALGO_AUTO), forced[0])


def gated_operands(m, n, k, g, seed):
    """x, then weight and zeros/scales of gate and of up, with their float64 products: of W_hat, and of (q - z) s unrounded."""
    from sqamd import capi as c
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn((m, k), device=DEV, generator=gen).half()
    dev, hat, real = [], [], []
    for _ in range(2):
        w = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=gen)
        z = torch.randint(0, 16, (n, k // g), device=DEV, generator=gen).half()
        s = (torch.rand((n, k // g), device=DEV, generator=gen) * 0.002 + 0.0002).half()
        pairs = lambda v: torch.stack([z, v], -1).reshape(n, -1).contiguous()
        dev += [w, pairs(s)]
        hat.append(x.double() @ c.dequant(w, dev[-1], n, k, g).double().t())
        real.append(x.double() @ (c.dequant(w, pairs(torch.ones_like(s)), n, k, g).double() * s.double().repeat_interleave(g, 1)).t())
    return x, dev, hat, real


@pytest.mark.parametrize("m,n,k", [(8, 8192, 4096), (9, 5128, 5120), (16, 5128, 5120)])
def test_gate_and_up_in_two_ring_launches(capi, m, n, k):
    """Group size 32 at few tokens on large weights: each projection is the ring kernel's, the second multiplies the first
    into its store."""
    x, dev, (gate, up), _ = gated_operands(m, n, k, 32, seed=m)
    ref = torch.nn.functional.silu(gate) * up
    for ws in (None, capi.workspace(m, n, k, DEV, gated=True)):
        y, u = capi.gemm_silu_dot(x, *dev, n, k, 32, ws=ws, use_workspace=False)
        # the up projection is rounded to fp16 before the product (2^-11) and the product is (2^-11); the sums' fp32 errors
        # are those of a result of norm-wise relative error k^(1/2) 2^-24 < 2^-17
        assert (u.double() - up).norm() <= (2.0 ** -11 + 2.0 ** -17) * up.norm()
        assert (y.double() - ref).norm() <= (2.0 ** -10 + 2.0 ** -15) * ref.norm()


@pytest.mark.parametrize("m,n,k,g,use_ws,one", [
    (1, 8192, 5120, 128, False, True), (2, 8192, 5120, 128, False, True), (1, 8320, 5120, 128, False, False),
    (3, 8192, 4096, 128, True, True), (3, 8256, 4096, 128, True, False), (16, 8256, 4096, 128, True, False),
    (3, 2048, 2048, 128, True, False), (9, 2048, 2048, 128, True, True), (3, 1408, 2304, 128, True, False),
    (5, 1408, 2304, 128, True, True), (5, 1408, 2688, 128, False, False), (5, 2048, 2048, 64, True, False),
    (5, 4096, 3328, 64, True, False), (5, 512, 3840, 64, False, False), (5, 512, 3840, 64, True, True),
    (3, 17920, 5120, 128, False, False), (3, 17920, 5120, 128, True, True), (5, 8512, 3968, 64, True, False),
    (3, 11584, 5760, 128, True, False), (3, 11584, 5632, 128, True, True)])
def test_gate_and_up_of_few_tokens_in_one_launch_where_it_is_faster(capi, m, n, k, g, use_ws, one):
    """Both sides of the lines between one launch and two, and the result of the one that is chosen."""
    x, dev, hat, real = gated_operands(m, n, k, g, seed=n)
    ws = capi.workspace(m, n, k, DEV, gated=True) if use_ws else None
    L, p = capi.lib(), lambda t: None if t is None else t.data_ptr()
    y = torch.empty((m, n), dtype=torch.float16, device=DEV)
    rc = L.sq_w4a16_gemm_silu_dot_one(p(x), *(p(t) for t in dev), p(y), m, n, k, g, capi.SQ_LAYOUT_L1, capi.SQ_ALGO_AUTO, p(ws),
                                      0 if ws is None else ws.numel(), capi._stream(None))
    assert rc == (capi.SQ_OK if one else capi.SQ_ERR_BAD_ALGO)
    y = capi.gemm_silu_dot(x, *dev, n, k, g, out=y, ws=ws, use_workspace=False)[0]
    # (two launches round the up projection and the product, the GEMV and the sums scaled neither weight; fp32 sums as above)
    gate, up = real if g == 128 else hat
    ref = torch.nn.functional.silu(gate) * up
    assert (y.double() - ref).norm() <= (2.0 ** -10 + 2.0 ** -15) * ref.norm()


def test_gate_and_up_hold_no_more_than_the_ring_kernel_can_use(capi):
    """The extension keeps its workspace per stream: 40 MB for 11008 x 4096 at 333 tokens, not the 135 MB that the tiled GEMM
    would want for a weight of 2 x 11008 rows."""
    import quant
    m, n, k, g = 333, 11008, 4096, 64
    w = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV)
    zs = torch.full((n, 2 * (k // g)), 65.0, dtype=torch.float16, device=DEV)
    x = torch.randn((1, m, k), device=DEV).half()
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        before = torch.cuda.memory_allocated()
        y = quant.gemm_awq_silu_dot_ut(x, w, w, zs, zs, None, None, m, n, k, g)
        torch.cuda.synchronize()
        held = torch.cuda.memory_allocated() - before - y.numel() * 2
    assert held <= capi.lib().sq_w4a16_gemm_silu_dot_workspace_bytes(m, n, k) + (1 << 20) <= 40 << 20


def test_gate_and_up_of_a_measured_shape(capi):
    """The picker measures single linears: what it records for a shape leaves the one launch of gate and up in place where it
    names the ring kernel, and takes it away where it names another one than the built-in choice (the ring kernel here)."""
    g, seen = 64, set()
    L, p = capi.lib(), lambda t: t.data_ptr()
    capi.autotune_clear()
    for m, n, k in [(m, n, k) for m in (20, 40, 72, 104, 136, 200) for n, k in ((1536, 1024), (2816, 2048), (4096, 2560))]:
        w = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV)
        zs = torch.full((n, 2 * (k // g)), 65.0, dtype=torch.float16, device=DEV)
        x, y = torch.randn((m, k), device=DEV).half(), torch.empty((m, n), dtype=torch.float16, device=DEV)
        ws = capi.workspace(m, n, k, DEV, gated=True)
        one = lambda: L.sq_w4a16_gemm_silu_dot_one(p(x), p(w), p(zs), p(w), p(zs), p(y), m, n, k, g, capi.SQ_LAYOUT_L1,
                                                   capi.SQ_ALGO_AUTO, p(ws), ws.numel(), capi._stream(None))
        before = one()
        word = capi.autotune(x, w, zs, n, k, g, ws=ws, reps=3)[0] & 0xFF
        assert one() == (before if word in (0, capi.SQ_ALGO_RING) else capi.SQ_ERR_BAD_ALGO), (m, n, k, word)
        if before == 0 and word == capi.SQ_ALGO_RING:
            seen.add((m, n, k))
    torch.cuda.synchronize()
    capi.autotune_clear()
    if not seen:
        pytest.skip("the picker confirmed the built-in plan of every shape")


REST = 0x10  # tune word: only the tiles of the last round of 256 split K
SUMS = 0x20  # tune word: the scale on the sums (shapes of 32 and 64 rows, group size 128)


def real_weight(d, g):
    """(q - z) s without a rounding."""
    return (d["q"].astype(np.float64) - np.repeat(d["z"], g, 1)) * np.repeat(d["s"].astype(np.float64), g, 1)


@pytest.mark.parametrize("m,n,k,g", [(1, 64, 128, 128), (33, 136, 640, 128), (64, 264, 1408, 128), (16, 72, 6144, 128),
                                     (31, 5128, 384, 128)])
@pytest.mark.parametrize("shape", [1, 2, 3, 5])
def test_ring_parity_with_the_scale_on_the_sums(capi, shape, m, n, k, g):
    d = orc.synth_linear(n, k, g, seed=7 * n + k)
    w64, x = real_weight(d, g), orc.synth_x(m, k, seed=m)
    x64 = x.astype(np.float64)
    ref = x64 @ w64.T
    # one rounding to fp16 and K fp32 additions of the products' magnitudes
    bound = 2.0 ** -11 * np.abs(ref) + k * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T) + 2.0 ** -24
    w, zs, xd = to_dev(d["w_l1"]), to_dev(d["zs_l1"]), to_dev(x)
    ws = torch.zeros(65536 + (96 << 20), dtype=torch.uint8, device=DEV)
    ks_max = -(-k // {1: 512, 2: 256, 3: 256, 5: 128}[shape])
    for ks in (1, 2, 3, 8):
        if ks > ks_max:
            continue
        y = torch.full((m, n), float("nan"), dtype=torch.float16, device=DEV)
        algo = capi.SQ_ALGO_RING | ((shape | SUMS | (ks << 8)) << 8)
        capi.gemm_ws(xd, w, zs, n, k, g, out=y, algo=algo, ws=ws)
        got = y.cpu().numpy().astype(np.float64)
        assert np.all(np.abs(got - ref) <= bound), (ks, np.max(np.abs(got - ref) / bound))
        assert torch.equal(y, capi.gemm_ws(xd, w, zs, n, k, g, algo=algo, ws=ws))
        assert capi.workspace_is_clean(ws)


@pytest.mark.parametrize("shape,stage,short", [(1, 512, 0), (1, 512, 128), (2, 256, 0), (2, 256, 128), (3, 256, 0), (3, 256, 128),
                                               (5, 128, 0)])
@pytest.mark.parametrize("m", [19, 50])
def test_ring_sums_every_count_of_stages(capi, shape, stage, short, m):
    """Zeros and scales by the stage, and (50 tokens, K of a part over 2048) for four or eight stages at once: a last set that is
    whole, one stage long and ends early, a part of K that begins inside what would be another part's set, and row ends of the
    last weight row."""
    n, g = 136, 128
    ws = torch.zeros(65536 + (8 << 20), dtype=torch.uint8, device=DEV)
    for stages in (1, 2, 3, 4, 5, 7, 8, 9, 12, 13, 16, 17, 18, 25) if stage < 512 else (1, 2, 3, 5):
        k = stage * stages - short
        d = orc.synth_linear(n, k, g, seed=k)
        w64, x = real_weight(d, g), orc.synth_x(m, k, seed=shape)
        x64 = x.astype(np.float64)
        ref = x64 @ w64.T
        # one rounding to fp16 and K fp32 additions of the products' magnitudes
        bound = 2.0 ** -11 * np.abs(ref) + k * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T) + 2.0 ** -24
        w, zs, xd = to_dev(d["w_l1"]), to_dev(d["zs_l1"]), to_dev(x)
        for parts in (1, 2, 3):
            if parts > stages:
                continue
            algo = capi.SQ_ALGO_RING | ((shape | SUMS | (parts << 8)) << 8)
            got = capi.gemm_ws(xd, w, zs, n, k, g, algo=algo, ws=ws).cpu().numpy().astype(np.float64)
            assert np.all(np.abs(got - ref) <= bound), (stages, parts, np.max(np.abs(got - ref) / bound))


@pytest.mark.parametrize("shape,rows", [(2, 32), (3, 64), (5, 64)])
@pytest.mark.parametrize("quarters,k", [(1, 3200), (1, 2176), (2, 4352), (2, 5120), (3, 2560), (3, 2304)])
def test_ring_sums_zeros_and_scales_by_the_set_and_by_the_stage(capi, shape, rows, quarters, k):
    """One token more than a quarter (an odd number of groups), half and three quarters of a tile's rows brings zeros and scales
    by the set: the bits of the other tokens stay, unsplit and with K split, for one weight and for gate and up."""
    n, g, m = 136, 128, rows * quarters // 4
    L, p = capi.lib(), lambda t: t.data_ptr()
    ws = torch.zeros(65536 + (8 << 20), dtype=torch.uint8, device=DEV)
    for parts in (1, 2):  # an odd number of groups in two parts begins inside a group's stage of two
        kk = k * parts + (g if parts == 2 and k // g % 2 else 0)
        x, dev, _, real = gated_operands(m + 1, n, kk, g, seed=kk + m)
        word = capi.SQ_ALGO_RING | ((shape | SUMS | (parts << 8)) << 8)
        y = [capi.gemm_ws(x[:i], dev[0], dev[1], n, kk, g, algo=word, ws=ws) for i in (m, m + 1)]
        assert torch.equal(y[0], y[1][:m])
        # one rounding to fp16 and the fp32 sums, norm-wise far below it
        assert (y[1].double() - real[0]).norm() <= (2.0 ** -11 + 2.0 ** -17) * real[0].norm()
        u = []
        for i in (m, m + 1):
            u.append(torch.empty((i, n), dtype=torch.float16, device=DEV))
            assert L.sq_w4a16_gemm_silu_dot_one(p(x), *(p(t) for t in dev), p(u[-1]), i, n, kk, g, capi.SQ_LAYOUT_L1, word, p(ws),
                                                ws.numel(), capi._stream(None)) == 0
        assert torch.equal(u[0], u[1][:m])
        ref = torch.nn.functional.silu(real[0]) * real[1]
        assert (u[1].double() - ref).norm() <= (2.0 ** -10 + 2.0 ** -15) * ref.norm()
        assert capi.workspace_is_clean(ws)


def test_ring_has_the_scale_on_the_sums_where_it_says(capi):
    d = orc.synth_linear(64, 128, 32, seed=1)
    x, w, zs = to_dev(orc.synth_x(8, 128)), to_dev(d["w_l1"]), to_dev(d["zs_l1"])
    with pytest.raises(capi.SqError):  # another group size
        capi.gemm(x, w, zs, 64, 128, 32, algo=capi.SQ_ALGO_RING | ((1 | SUMS) << 8))
    with pytest.raises(capi.SqError):  # a shape of 96 rows
        capi.gemm(x, w, zs[:, :2].contiguous(), 64, 128, 128, algo=capi.SQ_ALGO_RING | ((4 | SUMS) << 8))


@pytest.mark.parametrize("use_ws", [True, False])
@pytest.mark.parametrize("m,n,k,g", [(5, 5120, 5120, 32), (8, 5120, 5120, 32), (8, 6656, 5120, 128), (16, 6656, 5120, 128),
                                     (17, 4096, 4096, 128), (32, 4096, 4096, 128), (32, 1000, 11008, 128),
                                     (40, 2048, 1408, 128), (48, 2560, 13696, 128), (64, 2048, 1536, 128),
                                     (5, 2816, 6080, 64), (8, 4096, 4672, 64)])
def test_few_tokens_round_no_weight_to_half(capi, m, n, k, g, use_ws):
    """Where decode kernels keep the scale in fp32 the automatic choice does so whichever kernel it names: the result is
    as far from (q - z) s in float64 as its one rounding to fp16 puts it (W_hat is 1.4 times as far, and fp32 sums add
    a part in 2^24 of sums no more than some hundred times the result)."""
    d = orc.synth_linear(n, k, g, seed=k)
    x = orc.synth_x(m, k, seed=m)
    ref = torch.from_numpy(x).to(DEV).double() @ torch.from_numpy(real_weight(d, g)).to(DEV).t()
    y = capi.gemm_fused(to_dev(x), to_dev(d["w_l1"]), to_dev(d["zs_l1"]), n, k, g, use_workspace=use_ws)
    rounding = (ref.half().double() - ref).norm()
    assert (y.double() - ref).norm() <= 1.1 * rounding


@pytest.mark.parametrize("m,n,k,g,algo", [
    (8, 4608, 4608, 64, "RING"), (8, 3072, 5888, 64, "STREAM"), (8, 5632, 5888, 64, "STREAM"), (7, 2560, 8704, 64, "STREAM"),
    (12, 4736, 5376, 64, "RING"), (12, 3584, 5376, 64, "STREAM"), (8, 4352, 17408, 64, "RING"), (8, 5632, 15616, 64, "STREAM"),
    (10, 4736, 14336, 128, "RING"), (10, 5504, 15232, 128, "STREAM")])
def test_few_tokens_take_the_kernel_that_measures_ahead(capi, m, n, k, g, algo):
    """Both sides of the lines between the streaming and the ring kernel where K is split; the two add in different orders."""
    gen = torch.Generator(device=DEV).manual_seed(k)
    w = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=gen)
    zs = (torch.rand((n, 2 * (k // g)), device=DEV, generator=gen) + 0.01).half()
    x = torch.randn((m, k), device=DEV, generator=gen).half()
    ws = capi.workspace(m, n, k, DEV)
    word = {"STREAM": capi.SQ_ALGO_STREAM, "RING": capi.SQ_ALGO_RING | ((SUMS if g == 128 else 0) << 8)}
    y, same = (capi.gemm_ws(x, w, zs, n, k, g, algo=a, ws=ws) for a in (capi.SQ_ALGO_AUTO, word.pop(algo)))
    assert torch.equal(y, same)
    assert not torch.equal(y, capi.gemm_ws(x, w, zs, n, k, g, algo=word.popitem()[1], ws=ws))


@pytest.mark.parametrize("m,n,k", [(5, 3328, 5120), (8, 5120, 5120), (6, 4096, 4672)])
def test_few_tokens_round_no_weight_to_half_without_a_workspace_at_group_size_64(capi, m, n, k):
    test_few_tokens_round_no_weight_to_half(capi, m, n, k, 64, False)


def test_gate_and_up_with_little_workspace_round_no_weight_to_half(capi):
    """Less than the streaming kernel wants: the GEMV twice, with its scale in fp32."""
    m, n, k, g = 8, 2560, 5120, 64
    d = orc.synth_linear(n, k, g, seed=k)
    x, w, zs = orc.synth_x(m, k, seed=m), to_dev(d["w_l1"]), to_dev(d["zs_l1"])
    ws = torch.zeros(1 << 20, dtype=torch.uint8, device=DEV)
    assert ws.numel() < capi.lib().sq_w4a16_workspace_bytes(m, n, k)
    _, up = capi.gemm_silu_dot(to_dev(x), w, zs, w, zs, n, k, g, ws=ws)
    ref = torch.from_numpy(x).to(DEV).double() @ torch.from_numpy(real_weight(d, g)).to(DEV).t()
    assert (up.double() - ref).norm() <= 1.1 * (ref.half().double() - ref).norm()


@pytest.mark.parametrize("m,n,k,g", [(1, 72, 640, 128), (33, 136, 1408, 128), (70, 72, 416, 32), (20, 72, 960, 64)])
@pytest.mark.parametrize("shape", range(10))
def test_ring_keeps_an_infinite_activation_to_its_row(capi, shape, m, n, k, g):
    """An infinity in the last column of one row, K ending inside a stage: infinities of the weights' signs in that row,
    the other rows as without it (a shape of 0: the automatic choice of shape)."""
    d = orc.synth_linear(n, k, g, seed=k)
    d["q"][:, -1] = np.where(d["z"][:, -1] == 0, 15, 0)  # no weight of 0 in that column
    w, zs = to_dev(orc.pack_l1(d["q"])), to_dev(d["zs_l1"])
    x = orc.synth_x(m, k, seed=m)
    ws = torch.zeros(65536 + (96 << 20), dtype=torch.uint8, device=DEV)
    words = [shape] + ([shape | SUMS] if g == 128 and m <= 64 and shape in (0, 1, 2, 3, 5) else [])
    for tune in words:
        run = lambda: capi.gemm_ws(to_dev(x), w, zs, n, k, g, algo=capi.SQ_ALGO_RING | (tune << 8), ws=ws).cpu().numpy()
        x[m // 2, -1] = 0.5
        plain = run()
        x[m // 2, -1] = np.inf
        got = run()
        assert np.array_equal(got[m // 2], np.where(d["q"][:, -1] > 0, np.inf, -np.inf).astype(np.float16)), hex(tune)
        got[m // 2] = plain[m // 2]
        assert np.array_equal(got, plain), hex(tune)


@pytest.mark.parametrize("shape,bm,bn,stage", [(1, 32, 64, 512), (2, 32, 128, 256), (3, 64, 128, 256), (4, 96, 128, 128),
                                               (5, 64, 256, 128), (6, 96, 256, 128), (7, 128, 128, 128),
                                               (8, 128, 256, 128), (9, 256, 256, 64)])
def test_ring_whole_tiles_beside_split_ones(capi, shape, bm, bn, stage):
    """260 tiles, ragged at both ends: 256 by one workgroup each and the last four in up to eight parts of K, in one
    launch; nine stages, the last one part-filled.  Every word has to run."""
    m, n, k, g = 2 * bm - 5, 129 * bn + 8, 8 * stage + 128, 128
    gen = torch.Generator(device=DEV).manual_seed(shape)
    w = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=gen)
    z = torch.randint(64, 80, (n, k // g), device=DEV, generator=gen).half()
    sc = (torch.rand((n, k // g), device=DEV, generator=gen) * 0.01 + 0.001).half()
    pairs = lambda s: torch.stack([z, s], -1).reshape(n, -1).contiguous()
    zs, x = pairs(sc), torch.randn((m, k), device=DEV, generator=gen).half()
    ws = torch.zeros(65536 + 4 * 8 * bm * bn * 4, dtype=torch.uint8, device=DEV)
    x64 = x.double()
    for flag in (0, SUMS) if shape in (1, 2, 3, 5) else (0,):
        if flag:  # (q - z) s without a rounding: the integers times the scales
            w64 = capi.dequant(w, pairs(torch.ones_like(sc)), n, k, g).double() * sc.double().repeat_interleave(g, 1)
        else:
            w64 = capi.dequant(w, zs, n, k, g).double()
        ref = x64 @ w64.t()
        # one rounding to fp16 and K fp32 additions of the products' magnitudes
        bound = 2.0 ** -11 * ref.abs() + k * 2.0 ** -24 * (x64.abs() @ w64.abs().t()) + 2.0 ** -24
        for ks in (2, 3, 4, 6, 8):
            y = torch.full((m, n), float("nan"), dtype=torch.float16, device=DEV)
            capi.gemm_ws(x, w, zs, n, k, g, out=y, algo=capi.SQ_ALGO_RING | ((shape | REST | flag | (ks << 8)) << 8), ws=ws)
            worst = float(((y.double() - ref).abs() / bound).nan_to_num(nan=9.0).max())
            assert worst <= 1.0, (ks, flag)
            assert capi.workspace_is_clean(ws)
