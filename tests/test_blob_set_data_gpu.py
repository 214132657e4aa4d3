"""Net.forward's way in for host arrays: pieces of a large blob upload while the rest is copied."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def identity_net(mc, shape):
    from minicaffe import craft, zoo
    spec = [craft.input_layer({"data": shape}), dict(zoo.relu_layer("relu", "data"), top=["out"])]
    return mc.Net.from_buffers(craft.to_prototxt(spec, "identity"))


@pytest.mark.parametrize("count", [1, 511, (2 << 20) // 4, (2 << 20) // 4 + 1, 3 * (2 << 20) // 4 + 77])
def test_every_value_arrives_and_later_arrays_replace_it(gpu_mode, count):
    mc = gpu_mode
    net = identity_net(mc, (1, count))
    rng = np.random.default_rng(count)
    for dtype in (np.float32, np.float32, np.float64):     # (float64 takes the element-wise way)
        x = rng.random((1, count)).astype(dtype)
        net.forward(data=x)
        assert np.array_equal(net.get_blob("out").data, x.astype(np.float32))
        assert np.array_equal(net.get_blob("data").data, x.astype(np.float32))
    x = rng.random((1, 2 * count)).astype(np.float32)[:, ::2]   # not contiguous
    net.forward(data=x)
    assert np.array_equal(net.get_blob("out").data, x)
    view = net.get_blob("data").data                       # the blob's own host memory as the source
    view += 1
    want = view.copy()
    net.forward(data=view)
    assert np.array_equal(net.get_blob("out").data, want)
    small = rng.random((1, (count + 1) // 2)).astype(np.float32)   # a part of the block, then all of it
    net.forward(data=small)
    assert np.array_equal(net.get_blob("out").data, small)
    net.forward(data=want)
    assert np.array_equal(net.get_blob("out").data, want)


def test_wrong_count_is_an_error(gpu_mode):
    from minicaffe.base import LIB
    net = identity_net(gpu_mode, (1, 8))
    x = np.zeros(9, np.float32)
    blob = net.get_blob("data")
    assert LIB.CaffeBlobSetData(blob.handle, ctypes.c_void_p(x.ctypes.data), 9) == -1
    assert LIB.CaffeBlobSetData(blob.handle, None, 8) == -1


def test_filled_by_one_thread_and_used_by_another(gpu_mode):
    """The upload runs on the filling thread's stream, the forward on its own: the second waits for the first,
    also when the filling thread has ended."""
    import threading
    from minicaffe.base import LIB, check_call
    mc = gpu_mode
    count = 16 << 20                                       # 64 MiB: over a millisecond on the link
    net = identity_net(mc, (1, count))
    net.forward(data=np.zeros((1, count), np.float32))
    blob = net.get_blob("data")

    def fill(x):
        mc.set_runtime_mode(1, 0)
        check_call(LIB.CaffeBlobSetData(blob.handle, ctypes.c_void_p(x.ctypes.data), count))

    for i in range(1, 6):
        x = np.full((1, count), i, np.float32)
        t = threading.Thread(target=fill, args=(x,))
        t.start()
        t.join()
        if i % 2:                                          # ... and the other way round
            x[:] = 0                                       # the source has been copied
            net.forward()
        else:
            t = threading.Thread(target=lambda: (mc.set_runtime_mode(1, 0), net.forward()))
            t.start()
            t.join()
        assert np.all(net.get_blob("out").data == i)
