"""The kernel of small Convolution launches: K spread over the wavefronts of a workgroup.

Against a float64 convolution with the bound of any order of fp32 additions (and one unit per product for
the terms the split leaves out, see test_conv_split_gpu.py), at the edges of its 32 x 32 tiles, with fewer K tiles than
wavefronts, with slices past the last tile, and with what its epilogue does by itself: factors,
residual, activation, groups and two tops.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

CONFIGS = [8, 9]          # four and eight wavefronts


@pytest.fixture(scope="module")
def K(gpu_mode):
    from minicaffe import kernels
    return kernels


def conv64(x, w, **kw):
    return torch.nn.functional.conv2d(x.double(), w.double(), **kw)


@pytest.mark.parametrize("config", CONFIGS)
@pytest.mark.parametrize("case", [
    # cin, h, w, cout, k, stride, pad, dilation, group, batch, slices
    (9, 5, 5, 3, 1, 1, 0, 1, 1, 1, 1), (16, 8, 4, 32, 1, 1, 0, 1, 1, 1, 1), (67, 8, 8, 33, 1, 1, 0, 1, 1, 2, 1),
    (33, 9, 7, 65, 1, 2, 0, 1, 1, 3, 2), (160, 11, 11, 129, 1, 1, 0, 1, 1, 3, 3), (512, 6, 5, 31, 1, 1, 0, 1, 1, 1, 16),
    (4, 16, 16, 64, 3, 1, 1, 1, 1, 1, 1), (12, 13, 9, 130, 3, 2, 1, 1, 1, 2, 2), (20, 7, 7, 40, 5, 1, 2, 1, 1, 3, 5),
    (64, 1, 1, 24, 3, 1, 1, 1, 1, 5, 4), (8, 10, 11, 20, 3, 1, 2, 2, 1, 2, 1), (24, 12, 5, 96, 3, 1, 1, 1, 2, 2, 2),
    (160, 9, 9, 70, 1, 1, 0, 1, 2, 2, 1), (36, 31, 3, 33, (1, 5), 1, (0, 2), 1, 1, 1, 1),
    (1820, 3, 3, 20, 3, 1, 1, 1, 1, 1, 1)])          # 1024 K tiles, the longest table of taps
def test_against_float64(K, case, config):
    cin, h, wd, cout, k, s, p, d, group, n, slices = case
    k = (k, k) if isinstance(k, int) else k
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn((n, cin, h, wd), generator=g, device="cuda")
    w = torch.randn((cout, cin // group) + k, generator=g, device="cuda")
    sc, sh = torch.rand(cout, generator=g, device="cuda") + 0.5, torch.randn(cout, generator=g, device="cuda")
    plan = K.ConvPlan(K.conv_geom(cin, h, wd, cout, k, s, p, d, group))
    plan.force_config(config)
    plan.force_split(slices)
    assert "32x32" in plan.kernel_name(n)
    plan.set_weights(w.data_ptr())
    ho, wo = plan.output_shape()
    res = torch.randn((n, cout, ho, wo), generator=g, device="cuda")
    kw = dict(stride=s, padding=p, dilation=d, groups=group)
    want, mag = conv64(x, w, **kw), conv64(x.abs(), w.abs(), **kw)
    kk = cin // group * k[0] * k[1]
    c = lambda v: v.double().view(1, -1, 1, 1)   # noqa: E731
    for again in range(2):                       # (the second launch finds the counters of the first at zero)
        y = torch.full((n, cout, ho, wo), float("nan"), device="cuda")
        plan.forward(n, x.data_ptr(), y.data_ptr())
        assert ((y.double() - want).abs() <= (kk + 1) * 2.0 ** -24 * mag + 1e-30).all()
        y.fill_(float("nan"))
        plan.forward(n, x.data_ptr(), y.data_ptr(), scale=sc.data_ptr(), shift=sh.data_ptr(), residual=res.data_ptr(), activation=1)
        full = (want * c(sc) + c(sh) + res.double()).clamp(min=0)
        # ... and a rounding each of the product with the scale, of the shift and of the residual
        bound = (kk + 4) * 2.0 ** -24 * (mag * c(sc) + c(sh).abs() + res.abs().double())
        assert ((y.double() - full).abs() <= bound).all()


@pytest.mark.parametrize("config", CONFIGS)
@pytest.mark.parametrize("geom", [(17, 1, 1, 0, 1, 1, 20), (129, 1, 2, 0, 1, 1, 40), (24, 3, 2, 1, 1, 2, 96), (8, 3, 1, 1, 1, 1, 130)])
@pytest.mark.parametrize("slices", [1, 3])
def test_special_values(K, geom, config, slices):
    """Infinities, NaN and values the split cannot hold, the last channel's among them."""
    cin, k, s, p, d, g, cout = geom
    rng = np.random.default_rng(12)
    x = rng.standard_normal((2, cin, 13, 13)).astype(np.float32)
    w = (0.1 * rng.standard_normal((cout, cin // g, k, k))).astype(np.float32)
    for i, v in enumerate((np.inf, -np.inf, np.nan, 3.4e38)):
        x[i % 2, cin - 1 if i < 2 else (5 * i) % cin, (3 * i) % 13, (7 * i + 2) % 13] = v
    w[3, cin // g - 1, 0, 0] = np.inf
    plan = K.ConvPlan(K.conv_geom(cin, 13, 13, cout, k, s, p, d, g))
    plan.force_config(config)
    plan.force_split(slices)
    assert "32x32" in plan.kernel_name(2)
    xd, wd = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    ho, wo = plan.output_shape()
    plan.set_weights(wd.data_ptr())
    xp = torch.nn.functional.pad(torch.from_numpy(x), (p, p, p, p))
    y = torch.full((2, cout, ho, wo), float("nan"), device="cuda")
    plan.forward(2, xd.data_ptr(), y.data_ptr())
    got = y.cpu().numpy()
    want = torch.nn.functional.conv2d(xp, torch.from_numpy(w), stride=s, dilation=d, groups=g).numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.where(np.isinf(got), np.sign(got), 0), np.where(np.isinf(want), np.sign(want), 0))
    ok = np.isfinite(want)
    big = np.maximum(np.abs(want[ok]), 1.0)
    assert np.all(np.abs(got[ok].astype(np.float64) - want[ok]) <= 20 * cin * k * k * 2.0 ** -24 * big)


@pytest.mark.parametrize("config", CONFIGS)
@pytest.mark.parametrize("c_first", [1, 32, 45, 69])
@pytest.mark.parametrize("slices", [1, 2, 5])
def test_two_tops(K, config, c_first, slices):
    n, cin, h, cout = 3, 40, 7, 70
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn((n, cin, h, h), generator=g, device="cuda")
    w = torch.randn((cout, cin, 3, 3), generator=g, device="cuda")
    b = torch.randn(cout, generator=g, device="cuda")
    plan = K.ConvPlan(K.conv_geom(cin, h, h, cout, 3, 1, 1))
    plan.force_config(config)
    plan.force_split(slices)
    assert "32x32" in plan.kernel_name(n)
    plan.set_weights(w.data_ptr())
    whole = torch.full((n, cout, h, h), float("nan"), device="cuda")
    first = torch.full((n, c_first, h, h), float("nan"), device="cuda")
    second = torch.full((n, cout - c_first, h, h), float("nan"), device="cuda")
    plan.forward(n, x.data_ptr(), whole.data_ptr(), shift=b.data_ptr())
    plan.forward_two_tops(n, x.data_ptr(), first.data_ptr(), c_first, second.data_ptr(), shift=b.data_ptr())
    assert torch.equal(first, whole[:, :c_first]) and torch.equal(second, whole[:, c_first:])


@pytest.mark.parametrize("config", CONFIGS)
@pytest.mark.parametrize("cin", [9, 15, 16, 17, 24, 31, 48, 49, 65, 144, 150])
def test_nothing_behind_the_last_channel_is_read(K, config, cin):
    """Padding rows of a pointwise launch: the same bits whatever follows the blob in memory."""
    h, cout = 7, 20
    g = torch.Generator(device="cuda").manual_seed(6)
    w = torch.randn((cout, cin, 1, 1), generator=g, device="cuda")
    room = torch.zeros((cin + 40, h, h), device="cuda")       # the blob, and 40 more planes
    room[:cin] = torch.randn((cin, h, h), generator=g, device="cuda")
    plan = K.ConvPlan(K.conv_geom(cin, h, h, cout, 1))
    plan.force_config(config)
    plan.force_split(1)
    assert "32x32" in plan.kernel_name(1)
    plan.set_weights(w.data_ptr())
    tops = []
    for behind in (0.0, float("inf"), float("nan"), 1e30):
        room[cin:] = behind
        y = torch.full((1, cout, h, h), float("nan"), device="cuda")
        plan.forward(1, room.data_ptr(), y.data_ptr())
        tops.append(y)
    assert all(torch.equal(tops[0], t) for t in tops[1:])
    want, mag = conv64(room[None, :cin], w), conv64(room[None, :cin].abs(), w.abs())
    assert ((tops[0].double() - want).abs() <= (cin + 1) * 2.0 ** -24 * mag + 1e-30).all()


@pytest.mark.parametrize("geom", [
    # cin, size, cout, k: runs of one K tile per wavefront, of two, of some, slices
    (64, 14, 256, 1), (96, 14, 256, 1), (96, 9, 40, 1), (128, 28, 512, 1), (160, 14, 256, 1), (288, 14, 256, 1), (512, 7, 2048, 1),
    (1024, 10, 126, 1), (16, 20, 64, 3), (32, 20, 64, 3), (96, 24, 100, 5)])
@pytest.mark.parametrize("relu", [False, True])
def test_error_is_not_above_the_larger_tiles(K, geom, relu):
    """Against float64, where this kernel is chosen: its error in the norm is bounded by that of the
    64x64 tiles, whose launches it took over."""
    cin, h, cout, k = geom
    for seed in (1, 2):
        g = torch.Generator(device="cuda").manual_seed(seed)
        x = torch.randn((1, cin, h, h), generator=g, device="cuda")
        w = torch.randn((cout, cin, k, k), generator=g, device="cuda")
        x = x.clamp(min=0) if relu else x
        plan = K.ConvPlan(K.conv_geom(cin, h, h, cout, k, 1, k // 2))
        plan.force_winograd(0)
        plan.set_weights(w.data_ptr())
        want = conv64(x, w, padding=k // 2)
        errors = []
        for config, name in ((-1, "32x32"), (7, "64x64")):
            plan.force_config(config)
            assert name in plan.kernel_name(1)
            y = torch.full((1, cout, h, h), float("nan"), device="cuda")
            plan.forward(1, x.data_ptr(), y.data_ptr())
            errors.append((y.double() - want).norm().item())
        assert errors[0] <= errors[1]
