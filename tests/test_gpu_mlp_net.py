"""The fused network kernels at the edges of their tiles: one and two
wavefronts, a last block that is not full, the switch between block sizes
(32,768 rows), every width, odd and largest input and output counts, and a
forward length that is not a multiple of 64.  Against the FP64 CPU oracle
with the device's BF16 roundings; tolerances as in test_gpu_mlp.py (FP32
accumulation, and a rounding that falls the other way, through up to six
layers)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(np.ravel(a) - np.ravel(b)) / np.linalg.norm(np.ravel(b)))


@pytest.mark.parametrize("fin,width,hidden,fout,rows", [
    (5, 64, 2, 4, 64), (3, 192, 2, 1, 320), (8, 256, 3, 8, 704), (6, 128, 6, 5, 4160),
    (5, 64, 3, 4, 32704), (5, 256, 2, 4, 32832)])
def test_fused_forward_and_gradient(fin, width, hidden, fout, rows):
    from dgbgk.mlp import MLP
    from mlp_oracle import init_params, loss_grad
    print(f"fused mlp {fin}-{width}x{hidden}-{fout} rows={rows}", flush=True)
    p = init_params(fin, width, hidden, fout, seed=rows).astype(np.float32)
    p += (0.05 * np.random.default_rng(7).standard_normal(p.shape)).astype(np.float32)
    rng = np.random.default_rng(11)
    x = rng.standard_normal((rows, fin)).astype(np.float32)
    t = rng.standard_normal((rows, fout)).astype(np.float32)
    lo, go, yo = loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64),
                           fin, width, hidden, fout, bf16=True)
    m = MLP(fin=fin, width=width, hidden=hidden, fout=fout, batch=rows)
    m.set_params(p)
    loss, g = m.loss_grad(x, t)
    assert abs(loss - lo) <= 3e-3 * lo
    assert _rel(g, go) < 3e-2
    per, at = width * width + width, width * fin + width
    for part in (slice(0, at), slice(at + width * width, at + per),
                 slice(len(p) - fout, len(p))):  # the small sums on their own
        assert _rel(g[part], go[part]) < 3e-2
    n = rows - 27
    assert _rel(m.forward(x[:n]), yo[:n]) < 3e-3
