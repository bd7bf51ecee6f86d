"""The training kernels of the tile-skipping network at the edges of their tiles (4 rows x
64 columns of a frame) against the FP64 oracle, and whole training runs against Adam in
FP64 over the same frame order; the sums run in a fixed order, so a run repeats bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from compactcnncascade_amd import api as A
    A.load()
    return A


def _data(shape, seed):
    from compactcnncascade_amd import skipnet
    rng = np.random.default_rng(seed)
    x = (rng.random(shape) - 0.5).astype(np.float32)
    y = (rng.random((shape[0], skipnet.SLOTS) + shape[1:]) < 0.15).astype(np.uint8)
    return skipnet.init_params(seed), x, y


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 63), (3, 4, 64), (2, 5, 65), (1, 13, 129), (40, 9, 70)])
def test_gradients_at_tile_edges(api, shape):
    from compactcnncascade_amd import skipnet
    from oracle import skipnet64 as sn64
    p, x, y = _data(shape, 17)
    loss, g = skipnet.grad(api, p, x, y, 5.0)
    l64, g64 = sn64.grad64(p, x, y, 5.0)
    # FP32 rounding (6e-8) over sums of at most 25,200 positions x 216 terms, in chains of
    # a few hundred: 1e-5 of the largest gradient leaves a decade
    assert abs(loss - l64) <= 1e-5 * abs(l64)
    assert np.abs(g - g64).max() <= 1e-5 * np.abs(g64).max()


@pytest.mark.parametrize("n,batch", [(10, 4), (7, 7), (5, 16)])
def test_training_matches_fp64_adam(api, n, batch):
    from compactcnncascade_amd import skipnet
    from oracle import skipnet64 as sn64
    p0, x, y = _data((n, 7, 66), 23)
    epochs, lr = 3, 3e-3
    p, losses = skipnet.train(api, x, y, epochs=epochs, batch=batch, lr=lr, pos_weight=5.0, seed=9, params=p0)
    q, losses2 = skipnet.train(api, x, y, epochs=epochs, batch=batch, lr=lr, pos_weight=5.0, seed=9, params=p0)
    assert np.array_equal(p.view(np.uint32), q.view(np.uint32)) and np.array_equal(losses, losses2)
    # the trainer's shuffle: a 64-bit linear congruential generator, Fisher-Yates per epoch
    mask, state = (1 << 64) - 1, (9 * 6364136223846793005 + 1442695040888963407) & ((1 << 64) - 1)
    order, b = list(range(n)), min(n, batch)
    w, m, v, t, want = p0.astype(np.float64), 0.0, 0.0, 0, []
    for _ in range(epochs):
        for i in range(n - 1, 0, -1):
            state = (state * 6364136223846793005 + 1442695040888963407) & mask
            j = (state >> 33) % (i + 1)
            order[i], order[j] = order[j], order[i]
        per = []
        for b0 in range(0, n - b + 1, b):
            idx = order[b0:b0 + b]
            l64, g = sn64.grad64(w, x[idx], y[idx], 5.0)
            t += 1
            m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
            w = w - lr * (m / (1 - 0.9 ** t)) / (np.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
            per.append(l64)
        want.append(np.mean(per))
    # a gradient within 1e-4 of its value moves a weight by at most lr * 1e-4 a step too
    # far; the few weights whose gradient nearly cancels may differ by more
    assert np.abs(losses - want).max() <= 1e-4 * np.abs(want).max()
    assert np.mean(np.abs(p - w)) <= 1e-3 * lr


@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 21, 1387), (2, 1, 43691), (64, 90, 160)])
def test_the_loss_is_the_average_of_all_outputs(api, shape):
    # one share of the sum, 8,192 of them (what the summing kernel takes at a time), one more,
    # and 86,400. Every share is added with a rounding of at most 2^-24 of the sum; the losses
    # and their way to a share take 14 more
    import torch
    from compactcnncascade_amd import skipnet
    rng = np.random.default_rng(sum(shape))
    x = rng.normal(0.0, 0.08, shape).astype(np.float32)
    y = (rng.random((shape[0], skipnet.SLOTS) + shape[1:]) < 5e-4).astype(np.uint8)
    p = skipnet.init_params(4)
    print("loss", shape, flush=True)
    loss, _ = skipnet.grad(api, p, x, y, 500.0)
    # the forward pass and the cross-entropy in 64 bits, a few frames at a time
    sizes = [(8, 1, 3, 3), (8,), (8, 8, 3, 3), (8,), (skipnet.SLOTS, 8, 3, 3), (skipnet.SLOTS,)]
    w = torch.from_numpy(p).to(torch.float64)
    w1, b1, w2, b2, w3, b3 = (q.reshape(s) for q, s in zip(w.split([int(np.prod(s)) for s in sizes]), sizes))
    conv = torch.nn.functional.conv2d
    want = 0.0
    for k in range(0, shape[0], 8):
        a = torch.from_numpy(x[k:k + 8]).to(torch.float64)[:, None]
        z = conv(conv(conv(a, w1, b1, padding=1).relu(), w2, b2, padding=1).relu(), w3, b3, padding=1)
        pos = torch.from_numpy(y[k:k + 8]) != 0
        sp = z.clamp(min=0) + torch.log1p(torch.exp(-z.abs()))
        want += float(torch.where(pos, 500.0 * (sp - z), sp).sum())
    want /= y.size
    shares = (y.size + 255) // 256
    assert abs(loss - want) <= (shares + 14) * 2.0 ** -24 * want


@pytest.mark.parametrize("n,batch", [(2, 1), (2, 2)])
def test_losses_of_finished_epochs_are_there_while_training_runs(api, n, batch):
    # a run of some thousand steps in a thread of its own: its first epochs' losses are
    # written long before its last epochs are trained
    import ctypes
    import threading
    import time
    from compactcnncascade_amd import skipnet
    p, x, y = _data((n, 9, 66), 5)
    epochs = 6000
    losses = np.full(epochs, -1.0, np.float32)
    ret = []

    def run():
        ptr = [ctypes.c_void_p(a.ctypes.data) for a in (p, x, y, losses)]
        ret.append(skipnet._lib(api).ccnn_skipnet_train(ptr[0], ptr[1], ptr[2], n, 9, 66, epochs, batch, 1e-4, 5.0, 3,
                                                        ptr[3]))
    t = threading.Thread(target=run)
    t.start()
    while losses[0] < 0 and t.is_alive():
        time.sleep(1e-4)
    running = losses[-1] < 0
    t.join()
    assert ret == [0] and (losses >= 0).all()
    assert running
