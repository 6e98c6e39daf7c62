"""What a network takes of the device: no more than two buffers of every hidden
layer's activations and two besides (the layer-by-layer form's), plus the
weight gradients' partial sums (at most 64 splits of a layer) and 32 MB."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,hidden,batch", [(64, 8, 262144), (128, 6, 131072), (256, 8, 65536)])
def test_network_memory(width, hidden, batch):
    import torch
    from dgbgk.mlp import MLP
    print(f"case network memory {width}x{hidden} batch={batch}", flush=True)
    MLP(width=64, hidden=2, batch=64).close()  # the process's own: library, runtime
    free0 = torch.cuda.mem_get_info()[0]
    m = MLP(width=width, hidden=hidden, batch=batch)
    took = free0 - torch.cuda.mem_get_info()[0]
    m.close()
    layer = 2 * batch * width
    assert took <= (2 * hidden + 2) * layer + 64 * (hidden - 1) * 4 * width * width + (32 << 20)
