"""The convolutions (conv_ring_kernel) at the edges of their tiling: chunks of
one, two and three output planes, rows and rectangles that end inside a
16-cell tile, several rectangles and batch items, against torch (the kernels'
bfloat16 rounding points; tolerances of the other network tests).  An input
that is not finite reaches exactly the outputs whose windows hold it: neither
padded k-steps nor the accumulators of planes that do not exist leak."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import cnn_reference as ref  # noqa: E402
from test_cnn_emulation import check_grads, emu_lib, rel  # noqa: E402, F401


def network(lib, seed):
    from deepgreen.learned import FluxCNN
    m = FluxCNN(seed=seed, lib=lib)
    p = ref.split(m.get_params())
    p["b1"] = np.linspace(-0.2, 0.2, 32, dtype=np.float32)
    p["b3"] = np.linspace(-0.1, 0.1, 15, dtype=np.float32)
    m.set_params(np.concatenate([np.asarray(p[k], np.float32).reshape(-1) for k, _ in ref.LAYOUT]))
    return m


def run(lib, batch, dims, seed):
    m = network(lib, seed)
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(batch,) + dims + (5,)).astype(np.float32)
    dy = rng.normal(size=(batch,) + tuple(d - 6 for d in dims) + (15,)).astype(np.float32)
    y, g = m.forward(x), m.backward(x, dy)
    net = ref.Net(m.get_params())
    yr = net.forward(x)
    (yr * torch.as_tensor(dy)).sum().backward()
    assert rel(y, yr.detach().numpy()) < 1e-2
    check_grads(g, net.grads_flat())


def run_nonfinite(lib, dims, at):
    m = network(lib, 4)
    x = np.random.default_rng(4).normal(size=(1,) + dims + (5,)).astype(np.float32)
    x[(0,) + at + (2,)] = np.nan
    bad = ~np.isfinite(m.forward(x)[0]).all(axis=-1)
    want = np.zeros_like(bad)
    want[tuple(slice(max(a - 6, 0), a + 1) for a in at)] = True
    np.testing.assert_array_equal(bad, want)


@pytest.mark.parametrize("batch,dims", [(2, (8, 7, 54)), (1, (9, 15, 9))])
def test_emulated_convolution_tiles(emu_lib, batch, dims):  # noqa: F811
    run(emu_lib, batch, dims, 5)


def test_emulated_nonfinite_input_stays_local(emu_lib):  # noqa: F811
    run_nonfinite(emu_lib, (9, 10, 9), (8, 0, 8))


@pytest.mark.gpu
@pytest.mark.parametrize("batch,dims", [(1, (7, 7, 7)), (2, (8, 7, 52)), (1, (9, 8, 53)), (1, (10, 16, 22)),
                                        (3, (11, 15, 54)), (2, (21, 60, 38)), (1, (30, 33, 130)), (40, (7, 9, 8))])
def test_convolution_tiles(batch, dims):
    print(f"  convolution {batch} x {dims}", flush=True)
    run(None, batch, dims, 6)


@pytest.mark.gpu
@pytest.mark.parametrize("dims,at", [((9, 10, 9), (8, 0, 8)), ((20, 30, 60), (10, 14, 46)), ((16, 16, 16), (0, 15, 7))])
def test_nonfinite_input_stays_local(dims, at):
    print(f"  non-finite input {dims} {at}", flush=True)
    run_nonfinite(None, dims, at)


def run_packed(lib):
    """The weights that Adam packs as it updates them act as those set anew."""
    from deepgreen.learned import FluxCNN
    a, b = network(lib, 7), FluxCNN(seed=8, lib=lib)
    rng = np.random.default_rng(7)
    for _ in range(2):
        a.adam_step(rng.normal(size=a.get_params().size).astype(np.float32), lr=1e-2)
    b.set_params(a.get_params())
    x = rng.normal(size=(1, 8, 7, 9, 5)).astype(np.float32)
    dy = rng.normal(size=(1, 2, 1, 3, 15)).astype(np.float32)
    np.testing.assert_array_equal(a.forward(x), b.forward(x))
    np.testing.assert_array_equal(a.backward(x, dy), b.backward(x, dy))
    net = ref.Net(a.get_params())
    assert rel(a.forward(x), net.forward(x).detach().numpy()) < 1e-2


def test_emulated_adam_packs_the_weights(emu_lib):  # noqa: F811
    run_packed(emu_lib)


@pytest.mark.gpu
def test_adam_packs_the_weights():
    run_packed(None)


def run_loss(lib, batch, L):
    m = network(lib, 9)
    rng = np.random.default_rng(L)
    x = rng.normal(size=(batch, L + 7, L + 7, L + 7, 5)).astype(np.float32)
    t = rng.normal(size=(batch, L, L, L, 5)).astype(np.float32)
    loss, g = m.train_batch(x, t)
    net = ref.Net(m.get_params())
    want = ref.divergence_loss(net.forward(x), t)
    want.backward()
    assert abs(loss - want.item()) < 1e-2 * want.item()
    check_grads(g, net.grads_flat())


@pytest.mark.parametrize("batch,L", [(2, 1), (1, 4)])
def test_emulated_loss_runs(emu_lib, batch, L):  # noqa: F811
    run_loss(emu_lib, batch, L)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,L", [(1, 1), (3, 2), (40, 5), (2, 21), (1, 33), (9, 16)])
def test_loss_runs(batch, L):
    """One row to several runs of positions per plane, more and fewer items than workgroups."""
    print(f"  loss {batch} x {L}^3", flush=True)
    run_loss(None, batch, L)
