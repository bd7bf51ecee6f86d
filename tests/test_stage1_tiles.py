"""Stage 1 where its tiles end: level and frame sizes around the edges of the response and
L1 tiles, every tile shape, and inputs whose neighbouring convolutions are equal or one float
apart (the pool of a map's activations is taken before the activation where that is exact).
Every comparison is bit for bit."""
import ctypes

import numpy as np
import pytest


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.fixture(scope="module")
def oracle():
    from oracle.bind import Oracle
    return Oracle()


@pytest.fixture(scope="module")
def api():
    from compactcnncascade_amd import api as A
    A.load()
    return A


def test_pool_commutes_with_activations_whose_slopes_have_one_sign(oracle):
    # the rule that the kernels take at compile time, over quads of floats next to each other
    rng = np.random.default_rng(3)
    seen = 0
    for m in oracle.models[:3]:
        for layer in (0, 1):
            n = m.maps[layer]
            par = [np.ctypeslib.as_array(ctypes.cast(p[layer], ctypes.POINTER(ctypes.c_float)), shape=(n,))
                   for p in (m.conv_b, m.lrelu_w1, m.lrelu_w2, m.bn_b)]
            for cb, w1, w2, bb in zip(*par):
                if not ((w1 > 0 and w2 > 0) or (w1 < 0 and w2 < 0)) or bb == 0:
                    continue
                seen += 1
                base = (rng.standard_normal(20000) * 10.0 ** rng.uniform(-6, 3, 20000)).astype(np.float32)
                base[:4] = [-cb, 0.0, np.inf, -np.inf]
                quad = base[:, None].view(np.int32) + rng.integers(-3, 4, (len(base), 4)).astype(np.int32)
                quad[2:4] = base[2:4, None].view(np.int32)
                quad = quad.view(np.float32)
                quad[np.isnan(quad)] = 0.0

                def act(a):
                    c = a + cb
                    return (w2 * np.maximum(np.float32(0), c) + bb) + w1 * c
                first = quad.max(1) if w1 > 0 else quad.min(1)
                assert np.array_equal(bits(act(first)), bits(act(quad).max(1)))
    assert seen >= 5


SIZES = [(23, 27), (47, 51), (83, 87), (84, 91), (87, 88), (151, 153), (215, 95), (281, 157), (537, 64)]


@pytest.mark.gpu
@pytest.mark.parametrize("size", SIZES)
def test_stage1_at_tile_edges(api, oracle, size):
    w, h = size
    rng = np.random.default_rng(w * 1000 + h)
    noise = (rng.random((h, w)) * 255).astype(np.float32)
    flat = np.full((h, w), 117.25, np.float32)
    close = (flat.view(np.int32) + rng.integers(-2, 3, (h, w)).astype(np.int32)).view(np.float32)
    for level in (noise, flat, close):
        print("stage1", size, flush=True)
        assert np.array_equal(bits(api.stage1(level)), bits(oracle.forward(0, level)))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", range(12))
def test_level_windows_in_every_tile_shape(api, oracle, shape):
    # upscaled, copied and downscaled levels of ragged frames: whole rows of the level
    # window per wave, and the columns past them
    rng = np.random.default_rng(shape)
    for w, h, min_face in ((131, 97, 20), (263, 149, 27), (70, 259, 27), (517, 301, 61)):
        frame = rng.integers(0, 256, (h, w, 3), np.uint8)
        d = api.FaceDetector()
        assert d.Init(api.Param(max_image_size=(w, h), min_face_height=min_face)) == 0
        d.set_tile_shape(shape)
        print("levels", shape, w, h, flush=True)
        d.Detect(frame)
        g = oracle.gray(frame)
        levels = d.last_trace()["levels"]
        assert len(levels) > 0
        for (_, lw, lh, rw, rh, mode), got in zip(levels, d.last_responses()):
            level = g if mode == 2 else oracle.resize(g, int(lw), int(lh), int(mode))
            assert np.array_equal(bits(got), bits(oracle.forward(0, level))), (w, h, lw, lh, mode)


@pytest.mark.gpu
@pytest.mark.parametrize("size", SIZES)
def test_fp16_stage1_at_tile_edges(api, oracle, size):
    # the FP16 form against the exact one: 0.02, the bound that the FP16 form is held to
    # against FP64 elsewhere
    w, h = size
    rng = np.random.default_rng(w + 7 * h)
    smooth = np.clip(120 + 3 * np.cumsum(rng.standard_normal((h, w)), 1), 0, 255).astype(np.float32)
    for level in ((rng.random((h, w)) * 255).astype(np.float32), smooth):
        print("fp16 stage1", size, flush=True)
        assert np.abs(api.stage1(level, api.FP16_BF16) - oracle.forward(0, level)).max() < 0.02


@pytest.mark.gpu
def test_fp16_responses_do_not_depend_on_the_tile_shape(api):
    frame = np.random.default_rng(11).integers(0, 256, (301, 517, 3), np.uint8)
    want = None
    for shape in range(12):
        d = api.FaceDetector()
        assert d.Init(api.Param(max_image_size=(517, 301), min_face_height=30)) == 0
        d.set_compute_precision(api.FP16_BF16)
        d.set_tile_shape(shape)
        print("fp16 shape", shape, flush=True)
        d.Detect(frame)
        got = [bits(m) for m in d.last_responses()]
        want = want or got
        assert len(got) == len(want) and all(np.array_equal(a, b) for a, b in zip(got, want)), shape
