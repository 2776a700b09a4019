"""The surrogate network's device kernels (bf16 MFMA GEMMs, fp32 accumulation)
against the FP64 oracle (oracle/mlp_ref.py).

Bars: with the oracle rounding where the device rounds (mimic), outputs and
gradients agree to fp32-accumulation level (outputs 1e-3 of their scale,
gradients 5e-3 relative per tensor, the loss 1e-4); against the unrounded
FP64 network, to bfloat16 level (3e-2 / 6e-2).  One Adam step moves every
parameter with a clear gradient by -lr sign(g), as the oracle's step does.
Training lowers the loss of a smooth regression by more than 10x."""
import threading
import time

import numpy as np
import pytest

from oracle import mlp_ref as M
from pyqcm_amd import _lib
from pyqcm_amd.surrogate import MLP

pytestmark = pytest.mark.gpu

SHAPES = [(12, 641, 256, 4, 96), (5, 7, 64, 2, 33)]


@pytest.fixture(scope="module", autouse=True)
def _device():
    _lib.require_device()
    yield


def _net(n_in, n_out, width, depth, seed=11):
    net = MLP(n_in, n_out, width, depth, seed=seed)
    P = M.unflatten(net.get_weights(), n_in, n_out, width, depth)
    return net, P


@pytest.mark.parametrize("n_in,n_out,width,depth,B", SHAPES)
def test_forward_matches_oracle(n_in, n_out, width, depth, B):
    net, P = _net(n_in, n_out, width, depth)
    x = np.random.default_rng(5).normal(size=(B, n_in))
    y = net.predict(x)
    y_mim, _ = M.forward(P, x, mimic=True)
    y_ref, _ = M.forward(P, x, mimic=False)
    scale = np.max(np.abs(y_ref))
    assert np.max(np.abs(y - y_mim)) <= 1e-3 * scale, np.max(np.abs(y - y_mim)) / scale
    assert np.max(np.abs(y - y_ref)) <= 3e-2 * scale, np.max(np.abs(y - y_ref)) / scale


@pytest.mark.parametrize("n_in,n_out,width,depth,B", SHAPES)
def test_gradients_match_oracle(n_in, n_out, width, depth, B):
    net, P = _net(n_in, n_out, width, depth)
    rng = np.random.default_rng(6)
    x = rng.normal(size=(B, n_in))
    t = rng.normal(size=(B, n_out))
    w = rng.uniform(0.5, 2.0, n_out)
    w[0] = 32.0
    net.set_scaling(loss_weight=w)
    loss, g = net.loss_grad(x, t)
    loss_m, G_m = M.loss_grad(P, x, M.f32(t), M.f32(w), mimic=True)
    loss_r, G_r = M.loss_grad(P, x, t, w, mimic=False)
    assert abs(loss - loss_m) <= 1e-4 * loss_m
    assert abs(loss - loss_r) <= 2e-2 * loss_r
    gl = M.unflatten(g, n_in, n_out, width, depth)
    for l, ((dW, db), (mW, mb), (rW, rb)) in enumerate(zip(gl, G_m, G_r)):
        for name, a, m, r in (("W", dW, mW, rW), ("b", db, mb, rb)):
            em = np.linalg.norm(a - m) / np.linalg.norm(m)
            er = np.linalg.norm(a - r) / np.linalg.norm(r)
            assert em <= 5e-3, (l, name, em)
            assert er <= 6e-2, (l, name, er)


def test_adam_step_matches_oracle():
    n_in, n_out, width, depth, B = 5, 7, 64, 2, 64
    net, P = _net(n_in, n_out, width, depth, seed=3)
    rng = np.random.default_rng(8)
    x = rng.normal(size=(B, n_in))
    t = rng.normal(size=(B, n_out))
    net.set_optimizer(lr=1e-3)
    _, g = net.loss_grad(x, t)
    hist, _ = net.train(x, t, epochs=1, batch=B, seed=0)   # one full batch: one step
    P1 = M.unflatten(net.get_weights(), n_in, n_out, width, depth)
    _, G = M.loss_grad(P, x, M.f32(t), np.ones(n_out), mimic=True)
    S = M.adam_state(P)
    R1 = M.adam_step(P, G, S, lr=1e-3)
    gl = M.unflatten(g, n_in, n_out, width, depth)
    for (W, b), (W1, b1), (Wr, br), (gW, gb) in zip(P, P1, R1, gl):
        for p, p1, pr, gg in ((W, W1, Wr, gW), (b, b1, br, gb)):
            clear = np.abs(gg) > 1e-5
            assert np.max(np.abs((p1 - pr)[clear])) <= 2e-6, np.max(np.abs((p1 - pr)[clear]))
            assert np.allclose((p1 - p)[clear], -1e-3 * np.sign(gg[clear]), rtol=2e-2, atol=1e-6)
    assert hist.shape == (1,) and np.isfinite(hist[0])


def test_training_lowers_the_loss():
    rng = np.random.default_rng(9)
    n, n_in, n_out = 4096, 12, 16
    x = rng.uniform(-1, 1, size=(n, n_in))
    A = rng.normal(size=(n_in, n_out))
    y = np.sin(x @ A) + 0.5 * (x[:, :1] ** 2)
    net = MLP(n_in, n_out, 128, 3, seed=1)
    net.set_scaling(x_mean=np.zeros(n_in), x_std=np.ones(n_in) * 0.6, y_mean=y.mean(0), y_std=y.std(0))
    net.set_optimizer(lr=2e-3)
    hist, ms = net.train(x, y, epochs=60, batch=512, seed=2)
    assert hist[-1] < hist[0] / 10, hist[[0, -1]]
    assert ms > 0
    # predictions in physical units follow the targets
    err = np.sqrt(np.mean((net.predict(x[:256]) - y[:256]) ** 2)) / np.std(y)
    assert err < 0.3, err


def test_bad_arguments_are_errors():
    with pytest.raises(_lib.EDError):
        MLP(3, 4, 12, 2)          # width not a multiple of 8
    net = MLP(3, 4, 16, 1)
    with pytest.raises(_lib.EDError):
        net.set_scaling(x_std=np.array([1.0, 0.0, 1.0]))
    with pytest.raises(ValueError):
        net.set_weights(np.zeros(3))


@pytest.mark.parametrize("n_in,n_out,width,depth,B", [(1, 1, 64, 1, 1), (3, 16, 64, 1, 15), (33, 17, 128, 2, 16),
                                                      (64, 7, 64, 3, 17), (9, 300, 256, 2, 1037), (250, 33, 256, 1, 64),
                                                      (12, 641, 256, 4, 31), (5, 40, 32, 2, 50), (7, 20, 256, 9, 20)])
def test_row_block_kernels_at_their_edges(n_in, n_out, width, depth, B):
    """Batches around a row block (16) and a k-step (32), several batch splits,
    one to many output tiles, inputs as wide as a layer, one hidden layer, and
    two networks outside the row-block kernels' range (width 32, nine hidden
    layers): predictions, loss and gradients against the oracle with the same
    bf16 roundings (as the tests above: 1e-3 of the scale, 1e-4, and 5e-3 per
    layer; a bf16 rounding that falls the other way after a 1e-7 difference
    moves a single gradient entry by 0.4 %, and few rows average less: 2e-2
    below 64 rows)."""
    net, P = _net(n_in, n_out, width, depth, seed=B)
    rng = np.random.default_rng(B)
    x = rng.normal(size=(B, n_in))
    t = rng.normal(size=(B, n_out))
    y = net.predict(x)
    y_mim, _ = M.forward(P, x, mimic=True)
    assert np.max(np.abs(y - y_mim)) <= 2e-3 * np.max(np.abs(y_mim))
    loss, g = net.loss_grad(x, t)
    loss_m, G_m = M.loss_grad(P, x, M.f32(t), np.ones(n_out), mimic=True)
    assert abs(loss - loss_m) <= 1e-4 * loss_m
    for (dW, db), (mW, mb) in zip(M.unflatten(g, n_in, n_out, width, depth), G_m):
        for a, m in ((dW, mW), (db, mb)):
            assert np.linalg.norm(a - m) <= (5e-3 if B >= 64 else 2e-2) * np.linalg.norm(m) + 1e-12


def test_loss_from_a_second_thread():
    """predict on one thread, then the first loss_grad and the first time() of
    larger batches on another, both threads alive: the loss is that of a network
    used on one thread, to the last bit.  (The loss partials' buffer belongs to
    the stream that allocated it; a step that replaced it handed the kernel the
    old one.)"""
    n_in, n_out, width, depth = 12, 40, 64, 2
    rng = np.random.default_rng(21)
    x, t = rng.normal(size=(700, n_in)), rng.normal(size=(700, n_out))
    nets = [_net(n_in, n_out, width, depth, seed=5)[0] for _ in range(2)]
    want = [nets[0].loss_grad(x[:n], t[:n]) for n in (64, 700)]
    got, first, done = [], threading.Event(), threading.Event()

    def predicts():
        nets[1].predict(x[:64])
        first.set()
        done.wait(60)

    def learns():
        first.wait(60)
        for n in (64, 700):
            got.append(nets[1].loss_grad(x[:n], t[:n]))
        got.append(nets[1].time(900, 2))
        done.set()

    th = [threading.Thread(target=f) for f in (predicts, learns)]
    for q in th:
        q.start()
    for q in th:
        q.join(120)
    assert len(got) == 3 and min(got[2]) > 0.0
    for (loss, g), (loss_w, g_w) in zip(got, want):
        assert loss == loss_w
        assert np.array_equal(g, g_w)


def test_training_sees_a_cancellation():
    """A cancellation that arrives when most of a run's steps have been executed
    still ends it (the host does not queue the whole run and leave), and the
    network goes on afterwards."""
    n_in, n_out, batch = 12, 33, 2048
    rng = np.random.default_rng(22)
    x, t = rng.normal(size=(16 * batch, n_in)), rng.normal(size=(16 * batch, n_out))
    net = MLP(n_in, n_out, 256, 8, seed=2)
    net.train(x, t, epochs=1, batch=batch)
    # 64 epochs of 16 steps; the steps alone take most of the time
    _, ms = net.train(x, t, epochs=2, batch=batch)
    w0 = net.get_weights()
    t0 = time.perf_counter()
    net.train(x, t, epochs=64, batch=batch)
    wall = time.perf_counter() - t0
    net.set_weights(w0)
    timer = threading.Timer(wall - 0.35e-3 * 64 * 16 * ms, _lib.lib().ed_request_cancel)
    timer.start()
    try:
        with pytest.raises(_lib.EDError, match="interrupted"):
            net.train(x, t, epochs=64, batch=batch)
    finally:
        timer.join()
    hist, _ = net.train(x, t, epochs=1, batch=batch)
    assert np.isfinite(hist[0]) and np.all(np.isfinite(net.get_weights()))


def test_step_time_is_that_of_the_steps():
    """train's ms per step is the device's: an epoch of one step on one eighth of
    the rows' worth of shuffling costs as much per step as one without."""
    n_in, n_out = 4, 8
    rng = np.random.default_rng(23)
    x, t = rng.normal(size=(30000, n_in)), rng.normal(size=(30000, n_out))
    net = MLP(n_in, n_out, 64, 1, seed=2)
    ms = []
    for rows in (16384, 30000):  # both one step of 16 384 rows an epoch
        net.train(x[:rows], t[:rows], epochs=2, batch=16384)
        ms.append(min(net.train(x[:rows], t[:rows], epochs=64, batch=16384)[1] for _ in range(3)))
    assert ms[1] < 1.5 * ms[0], ms


def test_an_infinite_weight_stays_in_its_neuron():
    """One infinite first-layer weight of neuron 5: z and the activation of that
    neuron are infinite, those of its neighbours are not touched (their rows are
    read in one run with its), so that an output with positive weights is
    infinite and not NaN."""
    n_in, n_out, width = 3, 4, 64
    net, P = _net(n_in, n_out, width, 1, seed=9)
    w = np.abs(net.get_weights()) + 0.01
    w[5 * n_in + 1] = np.inf
    net.set_weights(w)
    x = np.abs(np.random.default_rng(3).normal(size=(20, n_in))) + 0.1
    assert np.all(net.predict(x) == np.inf)


def test_forward_passes_on_both_sides_of_the_row_block_line():
    """Two hidden layers of 256 and 641 outputs: 4 096 rows go through the row
    blocks, 4 097 layer by layer.  The same operands in another summation order
    (fp32, and a bf16 rounding that may fall the other way): 2e-3 of the scale, as
    above; three of the rows also against the oracle."""
    net, P = _net(12, 641, 256, 2, seed=4)
    x = np.random.default_rng(5).normal(size=(4097, 12))
    a, b = net.predict(x[:4096]), net.predict(x)
    scale = np.abs(b).max()
    assert np.abs(a - b[:4096]).max() <= 2e-3 * scale
    rows = [0, 2048, 4096]
    assert np.abs(b[rows] - M.forward(P, x[rows], mimic=True)[0]).max() <= 2e-3 * scale
