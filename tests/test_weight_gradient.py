"""Weight and bias gradients (dw_kernel) at the edges of their tiling: the
smallest box, rectangles split along z (more than 46 outputs), ragged last
rows and planes, several batch items, against autograd of the reference
network (the kernels' bfloat16 rounding points; the tolerance of the other
gradient tests, whose error is the bf16 rounding of the activations)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import cnn_reference as ref  # noqa: E402
from test_cnn_emulation import check_grads, emu_lib  # noqa: E402, F401


def run(lib, batch, dims, seed):
    from deepgreen.learned import FluxCNN
    m = FluxCNN(seed=seed, lib=lib)
    p = ref.split(m.get_params())
    p["W3"] = p["W3"] * 10.0
    p["b1"] = np.linspace(-0.2, 0.2, 32, dtype=np.float32)
    m.set_params(np.concatenate([np.asarray(p[k], np.float32).reshape(-1) for k, _ in ref.LAYOUT]))
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(batch,) + dims + (5,)).astype(np.float32)
    dy = rng.normal(size=(batch,) + tuple(d - 6 for d in dims) + (15,)).astype(np.float32)
    g = m.backward(x, dy)
    net = ref.Net(m.get_params())
    (net.forward(x) * torch.as_tensor(dy)).sum().backward()
    check_grads(g, net.grads_flat())


@pytest.mark.parametrize("batch,dims", [(1, (7, 7, 7)), (2, (8, 15, 53))])
def test_emulated_weight_gradient_tiles(emu_lib, batch, dims):  # noqa: F811
    run(emu_lib, batch, dims, 5)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,dims", [(1, (7, 7, 7)), (2, (8, 15, 53)), (3, (9, 7, 51)), (1, (40, 13, 100)),
                                        (9, (23, 39, 39)), (300, (8, 9, 8))])
def test_weight_gradient_tiles(batch, dims):
    print(f"  weight gradient {batch} x {dims}", flush=True)
    run(None, batch, dims, 6)
