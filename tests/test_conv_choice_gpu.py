"""Which kernel a 3x3 stride-1 Convolution takes where Winograd and direct launches meet."""
import pytest

pytestmark = pytest.mark.gpu


# cin, cout, height = width, batch; whether the Winograd kernel is the faster one, by 2 to 60 % as measured
@pytest.mark.parametrize("layer,winograd", [
    ((128, 128, 28, 12), True), ((128, 208, 12, 32), True), ((192, 192, 12, 32), True), ((160, 160, 75, 1), True),
    ((192, 96, 60, 2), True), ((112, 64, 46, 12), True), ((64, 64, 56, 16), True), ((512, 512, 38, 1), True),
    ((64, 64, 56, 8), False), ((128, 128, 28, 8), False), ((256, 256, 14, 12), False), ((512, 512, 7, 8), False),
    ((128, 192, 24, 9), False), ((512, 150, 10, 8), False), ((512, 512, 19, 1), False), ((64, 64, 56, 1), False)])
def test_the_faster_kernel_is_taken(gpu_mode, layer, winograd):
    from minicaffe import kernels as K
    cin, cout, size, batch = layer
    plan = K.ConvPlan(K.conv_geom(cin, size, size, cout, 3, 1, 1))
    assert (plan.kernel_name(batch) == "winograd_f32") == winograd
