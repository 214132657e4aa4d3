"""Convolution on the bf16 matrix pipe with three terms per operand: the same fp32 result.

Against a float64 convolution.  Any order of fp32 additions of the K products stays within
K * 2^-24 * sum |x w| per element; the terms left out of the split come to at most 2^-24 of a
product (|m| <= 2^-8 and |l| <= 2^-17 of a value's power of two, so |m l' + l m'| <= 2^-24), which is
the one more unit per product of the bound.  A single product (the fp32 kernel) is held to its one rounding.
The norm of the error is held to half of sqrt(K) * 2^-24 of the result's for operands of
random sign (fp32 products, one at a time, give 0.6 to 0.8 of it).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def K(gpu_mode):
    from minicaffe import kernels
    return kernels


def conv64(x, w, s, p):
    return torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), stride=s, padding=p).numpy()


def run(K, x, w, s, p, config, slices):
    n, cin, h, wd = x.shape
    plan = K.ConvPlan(K.conv_geom(cin, h, wd, w.shape[0], w.shape[2], s, p))
    plan.force_config(config)
    plan.force_split(slices)
    xd, wt = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    ho, wo = plan.output_shape()
    y = torch.full((n, w.shape[0], ho, wo), float("nan"), device="cuda")
    plan.set_weights(wt.data_ptr())
    plan.forward(n, xd.data_ptr(), y.data_ptr())
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("config", [0, 1, 2, 3, 4, 5, 6, 7])     # (3, 5 and 6 are the tiles of 7, 4 and 2)
@pytest.mark.parametrize("case", [
    # cin, size, cout, kernel, stride, pad, batch, slices: one K tile to many, odd and even numbers of
    # stages, rows and pixels on both sides of a tile's edge, all three ways to gather
    (1, 5, 3, 1, 1, 0, 1, 1), (16, 8, 32, 1, 1, 0, 1, 1), (17, 8, 33, 1, 1, 0, 2, 1), (33, 9, 65, 1, 2, 0, 3, 1),
    (96, 16, 127, 1, 1, 0, 1, 1), (160, 11, 129, 1, 1, 0, 3, 3), (4, 16, 64, 3, 1, 1, 1, 1), (12, 13, 130, 3, 2, 1, 2, 2),
    (3, 23, 24, 7, 2, 3, 2, 1), (5, 17, 40, 3, 1, 0, 3, 1)])
def test_error_against_float64(K, case, config):
    cin, size, cout, k, s, p, n, slices = case
    rng = np.random.default_rng(5)
    x = rng.standard_normal((n, cin, size, size)).astype(np.float32)
    w = rng.standard_normal((cout, cin, k, k)).astype(np.float32)
    want = conv64(x, w, s, p)
    err = np.abs(run(K, x, w, s, p, config, slices) - want)
    kk = cin * k * k
    assert np.all(err <= (kk + 1) * 2.0 ** -24 * conv64(np.abs(x), np.abs(w), s, p) + 1e-30)
    assert np.linalg.norm(err) <= 0.5 * max(2.0, np.sqrt(kk)) * 2.0 ** -24 * np.linalg.norm(want)


@pytest.mark.parametrize("config", [0, 1, 2, 4, 7])
@pytest.mark.parametrize("geom", [(32, 1, 0), (8, 3, 1), (3, 5, 2)])
def test_values_the_split_cannot_hold(K, config, geom):
    """Infinities, NaN and magnitudes that round past bf16's largest value, in the bottom and in
    the filters: the same special values as an fp32 convolution, finite ones where it is finite."""
    cin, k, p = geom
    rng = np.random.default_rng(6)
    x = rng.standard_normal((3, cin, 12, 12)).astype(np.float32)
    w = (0.1 * rng.standard_normal((70, cin, k, k))).astype(np.float32)
    for i, v in enumerate((np.inf, -np.inf, np.nan, 3.4e38, -3.4e38, 1e-30)):
        x[i % 3, (5 * i) % cin, (3 * i) % 12, (7 * i + 2) % 12] = v
    big = x.copy()
    w[11, 1, 0, 0], w[40, 0, k - 1, 0], w[69, cin - 1, 0, k - 1] = np.inf, np.nan, -np.inf
    with np.errstate(all="ignore"):
        # (padded by hand: the zeros of the padding are multiplied like any others, as im2col does)
        xp = torch.nn.functional.pad(torch.from_numpy(x), (p, p, p, p))
        want = torch.nn.functional.conv2d(xp, torch.from_numpy(w)).numpy()
        got = run(K, x, w, 1, p, config, 1)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.where(np.isinf(got), np.sign(got), 0), np.where(np.isinf(want), np.sign(want), 0))
    ok = np.isfinite(want)
    assert ok.any() and not ok.all()
    scale = np.maximum(np.abs(want[ok]), 1.0)
    assert np.all(np.abs(got[ok].astype(np.float64) - want[ok]) <= 2 * cin * k * k * 2.0 ** -24 * 10 * scale)


def test_filters_above_the_largest_bf16(K):
    """A filter value that rounding to bf16 would carry to infinity is kept."""
    x = np.full((1, 32, 4, 4), 0.01, np.float32)
    w = np.zeros((64, 32, 1, 1), np.float32)
    w[:, 3] = np.float32(3.4e38)
    want = conv64(x, w, 1, 0)
    assert np.allclose(run(K, x, w, 1, 0, 3, 1), want, rtol=3 * 2.0 ** -24, atol=0)


@pytest.mark.parametrize("config", [0, 1, 2, 4, 7])
@pytest.mark.parametrize("sx,sw", [
    (1e-36, 1.0), (1.0, 1e-36), (1e-37, 10.0), (1e-40, 1e10), (1e10, 1e-40), (1e-18, 1e-18), (1e-42, 1e20), (1e20, 1e-42),
    (1e30, 1e-30), (1e36, 1e-30), (1e-36, 1e36), (1e20, 1e10), (1e12, 1e12), (1e25, 1.0)])
@pytest.mark.parametrize("geom", [(1, 1, 0), (37, 1, 0), (12, 3, 1)])
def test_all_magnitudes_keep_their_bits(K, geom, sx, sw, config):
    """Operands from subnormal numbers to 1e36: no term of a split may leave bf16's range.  The bound of
    fp32 products, K * 2^-24 * sum |x w|, and one unit of the smallest float per product."""
    cin, k, p = geom
    rng = np.random.default_rng(8)
    x = (sx * rng.uniform(0.5, 1, (2, cin, 9, 9)) * rng.choice([-1, 1], (2, cin, 9, 9))).astype(np.float32)
    w = (sw * rng.uniform(0.5, 1, (40, cin, k, k)) * rng.choice([-1, 1], (40, cin, k, k))).astype(np.float32)
    kk = cin * k * k
    err = np.abs(run(K, x, w, 1, p, config, 1) - conv64(x, w, 1, p))
    assert np.all(err <= (kk + 1) * (2.0 ** -24 * conv64(np.abs(x), np.abs(w), 1, p) + 2.0 ** -149))


def test_a_single_product_is_rounded_once(K):
    """1x1 on one channel, for every combination of 512 x 512 significands: half a unit in the last place."""
    rng = np.random.default_rng(9)
    x = rng.uniform(1, 2, (1, 1, 16, 32)).astype(np.float32)
    w = rng.uniform(1, 2, (512, 1, 1, 1)).astype(np.float32)
    x[0, 0, 0, 0] = w[0] = 1.0038986          # where the left-out terms come to 2^-24.01
    want = conv64(x, w, 1, 0)
    err = np.abs(run(K, x, w, 1, 0, -1, 0) - want)
    assert np.all(err <= 2.0 ** -24 * np.exp2(np.floor(np.log2(want))))


@pytest.mark.parametrize("cin,k", [(2, 1), (5, 1), (8, 1), (9, 1), (33, 1), (4, 3), (64, 3), (576, 1)])
def test_constant_operands(K, cin, k):
    """Every product has the same left-out terms, so they do not average out over K."""
    for seed in range(8):
        rng = np.random.default_rng(seed)
        xv, wv = (1.0038986, 1.0038986) if seed == 0 else rng.uniform(1, 2, 2)
        x = np.full((2, cin, 20, 20), xv, np.float32)
        w = np.full((20, cin, k, k), wv, np.float32)
        want = conv64(x, w, 1, 0)
        assert np.all(np.abs(run(K, x, w, 1, 0, -1, 0) - want) <= (cin * k * k + 1) * 2.0 ** -24 * want)


@pytest.mark.parametrize("case", [(1024, 7, 512, 1, 64), (2048, 7, 512, 1, 64), (1024, 19, 256, 1, 8), (512, 10, 384, 3, 8)])
def test_sums_of_one_sign(K, case):
    """Operands of one sign, where a long chain of additions shows: n roundings of growing partial sums are
    sqrt(n / 3) * 0.29 units of 2^-23, and s slices of n / s roundings divide that by s.  The fp32 kernel rounds once
    per two products and takes 5 to 8 slices here; the error is held to what four such slices would leave."""
    cin, size, cout, k, n = case
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.rand((n, cin, size, size), generator=g, device="cuda") + 1
    w = torch.rand((cout, cin, k, k), generator=g, device="cuda") + 1
    plan = K.ConvPlan(K.conv_geom(cin, size, size, cout, k, 2 if k == 3 else 1, k // 2))
    plan.set_weights(w.data_ptr())
    ho, wo = plan.output_shape()
    y = torch.empty((n, cout, ho, wo), device="cuda")
    plan.forward(n, x.data_ptr(), y.data_ptr())
    torch.cuda.synchronize()
    want = conv64(x[:2].cpu().numpy(), w.cpu().numpy(), 2 if k == 3 else 1, k // 2)
    err = np.linalg.norm(y[:2].cpu().numpy() - want) / np.linalg.norm(want)
    kk = cin * k * k
    assert err <= 0.29 * 2.0 ** -23 * (np.sqrt(kk / 2 / 3) / 4 + 1)     # ... and the sum over slices and the store


@pytest.mark.parametrize("slices", [1, 3, 6])
@pytest.mark.parametrize("config", [-1, 1, 4, 7])
@pytest.mark.parametrize("geom", [
    # cin, k, stride, pad, dilation, group, cout: padding rows of K, several slices (and more than there are
    # stages), strides, dilations and groups in the products formed again
    (17, 1, 1, 0, 1, 1, 20), (33, 1, 1, 0, 1, 1, 70), (129, 1, 2, 0, 1, 1, 40), (24, 3, 2, 1, 1, 2, 96), (16, 3, 1, 2, 2, 1, 33),
    (35, 3, 1, 1, 1, 1, 24), (5, 1, 1, 0, 1, 1, 3), (8, 3, 1, 1, 1, 1, 130)])
def test_special_values_everywhere(K, geom, config, slices):
    """Infinities and NaN, the last channel's among them, in every way to gather and with K in slices."""
    cin, k, s, p, d, g, cout = geom
    rng = np.random.default_rng(12)
    x = rng.standard_normal((2, cin, 13, 13)).astype(np.float32)
    w = (0.1 * rng.standard_normal((cout, cin // g, k, k))).astype(np.float32)
    for i, v in enumerate((np.inf, -np.inf, np.nan, 3.4e38)):
        x[i % 2, cin - 1 if i < 2 else (5 * i) % cin, (3 * i) % 13, (7 * i + 2) % 13] = v
    plan = K.ConvPlan(K.conv_geom(cin, 13, 13, cout, k, s, p, d, g))
    plan.force_config(config)
    plan.force_split(slices)
    plan.force_winograd(0)
    xd, wd = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    ho, wo = plan.output_shape()
    plan.set_weights(wd.data_ptr())
    xp = torch.nn.functional.pad(torch.from_numpy(x), (p, p, p, p))
    for relu in (False, True):
        y = torch.full((2, cout, ho, wo), float("nan"), device="cuda")
        plan.forward(2, xd.data_ptr(), y.data_ptr(), activation=int(relu))
        torch.cuda.synchronize()
        want = torch.nn.functional.conv2d(xp, torch.from_numpy(w), stride=s, dilation=d, groups=g)
        want, got = want.numpy(), y.cpu().numpy()
        if relu:                       # (what ReLU makes of NaN and of -inf, which it multiplies by zero, is not held here)
            got, want = np.where(want > 0, got, 0), np.where(want > 0, want, 0)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert np.array_equal(np.where(np.isinf(got), np.sign(got), 0), np.where(np.isinf(want), np.sign(want), 0))
        ok = np.isfinite(want)
        big = np.maximum(np.abs(want[ok]), 1.0)
        assert np.all(np.abs(got[ok].astype(np.float64) - want[ok]) <= 20 * cin * k * k * 2.0 ** -24 * big)


@pytest.mark.parametrize("k,n", [(17, 5), (100, 40), (33, 70)])
def test_infinities_through_an_inner_product(K, k, n):
    import ctypes
    plan = K.ConvPlan.__new__(K.ConvPlan)
    plan.handle = ctypes.c_void_p()
    K.check_mc(K.LIB.mcInnerProductPlanCreate(k, n, 0, ctypes.byref(plan.handle)))
    rng = np.random.default_rng(13)
    x = rng.standard_normal((6, k)).astype(np.float32)
    w = rng.standard_normal((n, k)).astype(np.float32)
    x[0, k - 1], x[2, k - 1], x[4, 0] = np.inf, -np.inf, np.inf
    xd, wd, y = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), torch.full((6, n), float("nan"), device="cuda")
    plan.set_weights(wd.data_ptr())
    plan.forward(6, xd.data_ptr(), y.data_ptr())
    torch.cuda.synchronize()
    want, got = x @ w.T, y.cpu().numpy()
    assert np.array_equal(np.isinf(got) * np.sign(got), np.isinf(want) * np.sign(want)) and not np.isnan(got).any()
    ok = np.isfinite(want)
    assert np.all(np.abs(got[ok] - want[ok]) <= 2 * k * 2.0 ** -24 * (np.abs(x[[1, 3, 5]]) @ np.abs(w.T)).max())


def test_infinities_through_the_per_pixel_kernel(K):
    """At most four channels over many pixels, K not a multiple of 16."""
    rng = np.random.default_rng(14)
    x = rng.standard_normal((2, 19, 200, 200)).astype(np.float32)
    w = rng.standard_normal((3, 19, 1, 1)).astype(np.float32)
    x[0, 18, 3, 5], x[1, 18, 199, 199] = np.inf, -np.inf
    plan = K.ConvPlan(K.conv_geom(19, 200, 200, 3, 1, 1, 0))
    assert plan.kernel_name(2) == "thin_f32"
    want, got = conv64(x, w, 1, 0), run(K, x, w, 1, 0, -1, 0)
    assert np.array_equal(np.isinf(got) * np.sign(got), np.isinf(want) * np.sign(want)) and not np.isnan(got).any()
