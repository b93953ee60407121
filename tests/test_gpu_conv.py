"""The networks' block convolution and eight-channel transfers against the
general kernels they stand in for (reached here by operands aligned to less
than the vector accesses), bit for bit, over channel counts, block remainders,
residual, ReLU and mirrored taps."""
import pytest

pytestmark = pytest.mark.gpu

DIMS = [(1, 1, 1), (2, 1, 70), (5, 7, 9), (17, 17, 17), (33, 9, 18), (3, 40, 131)]
CHANNELS = [(16, 16), (16, 32), (32, 16), (32, 32), (48, 32), (48, 48), (64, 48), (64, 64), (16, 64)]


def shifted(t, by):
    """the same values at a pointer `by` elements past an aligned one"""
    import torch
    buf = torch.empty(t.numel() + by, dtype=t.dtype, device="cuda")
    buf[by:] = t.reshape(-1)
    return buf[by:].view(t.shape)


@pytest.mark.parametrize("dims", DIMS)
def test_block_convolution_same_bits(dims):
    import torch
    from citcom_amd import unet
    from citcom_amd.learn import _p
    L = unet._lib()
    g = torch.Generator(device="cuda").manual_seed(4)
    nv = dims[0] * dims[1] * dims[2]
    for ci, co in CHANNELS:
        for nb, relu, mirror, with_res in ((1, 0, 0, False), (3, 1, 0, True), (2, 0, 1, False)):
            x = torch.randn((nb, nv, ci), generator=g, device="cuda").bfloat16()
            w = (0.1 * torch.randn((co, 27, ci), generator=g, device="cuda")).bfloat16()
            b = torch.randn(co, generator=g, device="cuda")
            r = torch.randn((nb, nv, co), generator=g, device="cuda").bfloat16()
            out = []
            for xx in (x, shifted(x, 4)):     # 8 bytes past: the general kernel
                y = torch.full((nb, nv, co), float("nan"), dtype=torch.bfloat16, device="cuda")
                yf = torch.full((nb, nv, co), float("nan"), device="cuda")
                assert L.cl_conv3d_fwd_c(_p(xx), nb, *dims, ci, co, _p(w), _p(b), _p(r) if with_res else None, relu,
                                         mirror, _p(y), _p(yf), None) == 0
                out.append((y, yf))
            assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1]), (dims, ci, co, nb)


@pytest.mark.parametrize("dims", DIMS)
def test_sixteen_channel_data_gradient_same_bits(dims):
    import torch
    from citcom_amd.learn import _cl, _p
    L = _cl()
    g = torch.Generator(device="cuda").manual_seed(5)
    nv = dims[0] * dims[1] * dims[2]
    dy = torch.randn((2, nv, 16), generator=g, device="cuda").bfloat16()
    w = torch.randn((16, 27, 16), generator=g, device="cuda").bfloat16()
    out = []
    for d in (dy, shifted(dy, 4)):
        dx = torch.full((2, nv, 16), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert L.cl_conv3d_bwd_data(_p(d), 2, *dims, _p(w), _p(dx), None) == 0
        out.append(dx)
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("dims", [(3, 3, 3), (5, 7, 9), (17, 3, 33)])
@pytest.mark.parametrize("ch", [8, 16, 48])
def test_eight_channel_transfers_same_bits(dims, ch):
    import torch
    from citcom_amd import unet
    from citcom_amd.learn import _p
    L = unet._lib()
    g = torch.Generator(device="cuda").manual_seed(6)
    cd = unet.level_dims(dims, 1)
    nv, ncv = dims[0] * dims[1] * dims[2], cd[0] * cd[1] * cd[2]
    fine = torch.randn((2, nv, ch), generator=g, device="cuda").bfloat16()
    coarse = torch.randn((2, ncv, ch), generator=g, device="cuda").bfloat16()
    out = []
    for by in (0, 1):
        c2 = torch.full((2, ncv, ch), float("nan"), dtype=torch.bfloat16, device="cuda")
        f2 = torch.full((2, nv, ch), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert L.cl_restrict(_p(shifted(fine, by)), 2, *dims, ch, 8.0, _p(c2), None) == 0
        assert L.cl_interp(_p(shifted(coarse, by)), 2, *dims, ch, 0.125, _p(f2), None) == 0
        out.append((c2, f2))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("dims", DIMS)
def test_block_weight_gradient(dims):
    """against the general kernel's (FP32 sums of the same products in another
    order; the chunks' and the blocks' sums differ by rounding: 1e-5, as the
    kernels are held to the restatement); values that are not finite spread to
    the same entries"""
    import torch
    from citcom_amd import unet
    from citcom_amd.learn import _p
    L = unet._lib()
    g = torch.Generator(device="cuda").manual_seed(7)
    nv = dims[0] * dims[1] * dims[2]
    for ci, co in CHANNELS + [(80, 16), (96, 48)]:
        for nb, wild in ((1, False), (3, False), (2, True)):
            x = torch.randn((nb, nv, ci), generator=g, device="cuda").bfloat16()
            dy = torch.randn((nb, nv, co), generator=g, device="cuda").bfloat16()
            if wild:
                x[0, 0, 1] = float("inf")
                x[1, nv // 2, ci - 1] = float("nan")
                dy[0, nv - 1, 2] = float("-inf")
            ws = torch.empty(L.cl_conv3d_bwd_weight_c_workspace(nb, *dims, ci, co) // 4, device="cuda")
            out = []
            for xx in (x, shifted(x, 1)):
                gr = torch.full((co * 27 * ci + co,), 7.0, device="cuda")
                assert L.cl_conv3d_bwd_weight_c(_p(xx), _p(dy), nb, *dims, ci, co, _p(gr), _p(ws), None) == 0
                out.append(gr)
            a, b = out
            fine = torch.isfinite(b)
            assert torch.equal(torch.isfinite(a), fine) and torch.equal(torch.isnan(a), torch.isnan(b)), (dims, ci, co)
            assert float((a - b)[fine].norm()) <= 1e-5 * float(b[fine].norm()) + 1e-30, (dims, ci, co, nb)


@pytest.mark.parametrize("nb,dims", [(1, (1, 1, 1)), (3, (5, 7, 9)), (1, (32, 32, 32)), (1, (31, 33, 33)), (2, (33, 30, 37))])
def test_sixteen_channels_small_and_block_kernels_same_bits(nb, dims):
    """the kernel of small volumes (up to 32768 voxels) and the blocks', on
    either side of the line: forward against the general entry point, data
    gradient against less aligned operands"""
    import torch
    from citcom_amd import unet
    from citcom_amd.learn import _p
    L = unet._lib()
    g = torch.Generator(device="cuda").manual_seed(8)
    nv = dims[0] * dims[1] * dims[2]
    x = torch.randn((nb, nv, 16), generator=g, device="cuda").bfloat16()
    w = (0.1 * torch.randn((16, 27, 16), generator=g, device="cuda")).bfloat16()
    b = torch.randn(16, generator=g, device="cuda")
    nan = lambda dt: torch.full((nb, nv, 16), float("nan"), dtype=dt, device="cuda")
    y, yf, yg, yfg, d, ds = nan(x.dtype), nan(b.dtype), nan(x.dtype), nan(b.dtype), nan(x.dtype), nan(x.dtype)
    assert L.cl_conv3d_fwd(_p(x), nb, *dims, _p(w), _p(b), 1, _p(y), _p(yf), None) == 0
    assert L.cl_conv3d_fwd_c(_p(x), nb, *dims, 16, 16, _p(w), _p(b), None, 1, 0, _p(yg), _p(yfg), None) == 0
    assert torch.equal(y, yg) and torch.equal(yf, yfg)
    assert L.cl_conv3d_bwd_data(_p(x), nb, *dims, _p(w), _p(d), None) == 0
    assert L.cl_conv3d_bwd_data(_p(shifted(x, 4)), nb, *dims, _p(w), _p(ds), None) == 0
    assert torch.equal(d, ds)
