"""What a network takes of the device: no more than two buffers of every hidden
layer's activations and two besides (the layer-by-layer form's), plus the
weight gradients' partial sums (at most 64 splits of a layer) and 32 MB."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


def _free():
    from dgbgk._lib import lib
    free, total = C.c_size_t(), C.c_size_t()
    # the HIP runtime that the library is linked to
    assert lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("width,hidden,batch", [(64, 8, 262144), (128, 6, 131072), (256, 8, 65536)])
def test_network_memory(width, hidden, batch):
    from dgbgk.mlp import MLP
    print(f"case network memory {width}x{hidden} batch={batch}", flush=True)
    MLP(width=64, hidden=2, batch=64).close()  # the process's own: library, runtime
    free0 = _free()
    m = MLP(width=width, hidden=hidden, batch=batch)
    took = free0 - _free()
    m.close()
    layer = 2 * batch * width
    assert took <= (2 * hidden + 2) * layer + 64 * (hidden - 1) * 4 * width * width + (32 << 20)
