"""The packing kernel against the torch operations it stands for, bit for bit: every width, group size and layout on
ordinary weights, on the edges of its tiles, and on groups whose range is zero, tiny, overflowing or not finite."""
import pytest
import torch

from sqamd import capi, qlinear, quant_funcs as qf

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def weight(n, k, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    w = (torch.randn((n, k), device=DEV, generator=gen) * 0.02).half()
    # groups of 32 that take every branch: constant, zero, subnormal, offset, one-sided, overflowing range, inf, NaN
    flat = w.view(-1, 32)
    rows = [torch.full((32,), 100.0), torch.zeros(32), torch.arange(32) * 6e-8, 3 + torch.arange(32) * 1e-3,
            torch.arange(32) * -2.0, torch.linspace(-65504, 65504, 32), torch.linspace(0, 65504, 32)]
    if seed % 2:
        bad = torch.linspace(-1, 1, 32)
        rows += [bad.clone().index_fill_(0, torch.tensor([5]), float("inf")),
                 bad.clone().index_fill_(0, torch.tensor([31]), float("-inf")),
                 bad.clone().index_fill_(0, torch.tensor([0]), float("nan"))]
    for i, r in enumerate(rows):
        at = (i * 5 + 1) % flat.shape[0]
        flat[at] = r.half().to(DEV)
    # quotients that are halfway between two codes, and just beside it
    flat[-1] = torch.tensor([0.0, 15.0] + [j / 2 for j in range(30)]).half().to(DEV)
    return w


def bits(t):
    return t.view(torch.int16) if t.dtype == torch.float16 else t


def same(a, b):
    if a.dtype == torch.float16:  # a NaN's sign and payload are not part of the result
        return a.shape == b.shape and bool(((bits(a) == bits(b)) | (a.isnan() & b.isnan())).all())
    return torch.equal(a, b)


@pytest.mark.parametrize("n,k", [(32, 128), (8, 32), (96, 1152), (64, 4224), (160, 96)])
@pytest.mark.parametrize("g", [32, 64, 128])
@pytest.mark.parametrize("n_bit", [4, 2])
def test_quantise_parity(built_lib, monkeypatch, n, k, g, n_bit):
    if k % g:
        pytest.skip("K is not a multiple of the group size")
    for seed in (0, 1):
        w = weight(n, k, seed)
        assert qf._one_launch(w, n_bit, g, capi.SQ_LAYOUT_L1)
        got = qf.quant_muxi(w, k, n, n_bit=n_bit, group_size=g)
        got2 = qf.quant_lmdeploy(w, k, n, group_size=g, n_bit=n_bit) if n % 32 == 0 else ()
        with monkeypatch.context() as mp:
            mp.setattr(qf, "_one_launch", lambda *a: False)
            ref = qf.quant_muxi(w, k, n, n_bit=n_bit, group_size=g)
            ref2 = qf.quant_lmdeploy(w, k, n, group_size=g, n_bit=n_bit) if n % 32 == 0 else ()
        for a, b in zip(got + got2, ref + ref2):
            assert a.dtype == b.dtype and same(a, b), (seed, a.shape)


@pytest.mark.parametrize("layout", [capi.SQ_LAYOUT_L1, capi.SQ_LAYOUT_L2])
def test_c_abi_packs_as_the_extension_does(built_lib, layout):
    """sq_w4a16_quantise through the ctypes binding, with and without the fake-quantised weight."""
    import quant
    w = weight(64, 256, 1)
    for fake in (False, True) if layout == capi.SQ_LAYOUT_L2 else (False,):
        got, ref = capi.quantise(w, 64, 4, layout, fake), quant.quantise(w, 64, 4, layout, fake)
        assert (got[2] is None) == (ref[2] is None) == (not fake)
        assert all(a.dtype == b.dtype and same(a, b) for a, b in zip(got, ref) if a is not None)


def test_from_float_and_the_weights_the_kernel_leaves_alone(built_lib):
    w = weight(64, 256, 0)
    lin = torch.nn.Linear(256, 64, device=DEV, dtype=torch.float16)
    for layout in ("l1", "l2"):
        lin.weight.data = w
        a = qlinear.WALinear.from_float(lin, {"n_bit": 4, "group_size": 128}, layout=layout)
        lin.weight.data = w.t().contiguous().t()  # same values, other strides: torch operations
        assert not qf._one_launch(lin.weight.data, 4, 128, capi.SQ_LAYOUT_L1)
        b = qlinear.WALinear.from_float(lin, {"n_bit": 4, "group_size": 128}, layout=layout)
        assert torch.equal(a.weight, b.weight) and same(a.zeros_scales, b.zeros_scales) and torch.equal(a.bias, b.bias)
        assert a.state_dict().keys() == b.state_dict().keys() and a.weight.device == w.device
    shifted = torch.empty(64 * 256 + 1, dtype=torch.float16, device=DEV)[1:].view(64, 256)
    for other in (shifted, w.float(), w.bfloat16(), w.clone().requires_grad_(), w.cpu()):
        assert not qf._one_launch(other, 4, 128, capi.SQ_LAYOUT_L1)
    assert not qf._one_launch(w, 4, 16, capi.SQ_LAYOUT_L1) and not qf._one_launch(w[:8], 4, 128, capi.SQ_LAYOUT_L2)


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
def test_a_trace_of_the_packer_follows_its_input(built_lib):
    pack = lambda w: qf.quant_muxi(w, 256, 64, group_size=128)
    traced = torch.jit.trace(pack, (weight(64, 256, 0),), check_trace=False)
    other = (torch.randn((64, 256), device=DEV) * 0.02).half()
    assert qf._one_launch(other, 4, 128, capi.SQ_LAYOUT_L1)
    for a, b in zip(traced(other), pack(other)):
        assert torch.equal(a, b)
