"""Uploads of frames in pageable host memory through the staging ring: frames and batches on
both sides of the size from which it is used (8 MiB a call), sizes that are no multiple of
16 bytes, frames that go round the ring several times, one after the other and in both batch
modes. The bytes that arrive are compared through the gray image (exact) and through the
detections of the same frame in device memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(64, 64, 3), (2048, 1365, 3), (2048, 1366, 3), (1999, 1403, 3), (2403, 1601, 4), (1999, 4021, 3),
         (4096, 683, 3), (512, 512, 3), (60, 60, 3)]


def _frame(w, h, ch, seed):
    return np.random.default_rng(seed).integers(0, 256, (h, w, ch), np.uint8)


def _key(found):
    n, faces = found
    return n, faces.tobytes()


def test_frames_on_both_sides_of_the_ring_arrive_whole():
    from compactcnncascade_amd import api
    from oracle.bind import Oracle
    import torch
    oracle = Oracle()
    d = api.FaceDetector()
    assert d.Init(api.Param(max_image_size=(64, 64), min_face_height=100, max_face_height=120)) == 0
    for k, (w, h, ch) in enumerate(SIZES + SIZES[::-1]):
        print("upload", w, h, ch, flush=True)
        f = _frame(w, h, ch, k)
        host = _key(d.Detect(f))
        if min(w, h) >= 64:
            assert np.array_equal(d.getGrayImage32F(api.PIPELINE_CPU).view(np.uint32), oracle.gray(f).view(np.uint32))
        t = torch.from_numpy(f).cuda()
        assert host == _key(d.DetectDevice(t.data_ptr(), w, h, ch, w * ch))


def test_batches_of_host_frames_match_device_frames():
    from compactcnncascade_amd import api
    import torch
    d = api.FaceDetector()
    assert d.Init(api.Param(max_image_size=(4096, 4021), min_face_height=60, max_face_height=120)) == 0
    frames = [_frame(w, h, ch, 100 + k) for k, (w, h, ch) in enumerate(SIZES)]
    tensors = [torch.from_numpy(f).cuda() for f in frames]
    ptrs = [(t.data_ptr(), t.shape[1], t.shape[0], t.shape[2], t.shape[1] * t.shape[2]) for t in tensors]
    want = [_key(r) for r in d.DetectBatch(device_frames=ptrs)]
    for mode in (1, 0, 1):
        d.set_batch_mode(mode)
        print("batch mode", mode, flush=True)
        assert [_key(r) for r in d.DetectBatch(images=frames)] == want
        assert [_key(r) for r in d.DetectBatch(images=frames[::-1])] == want[::-1]


def test_batches_of_small_frames_share_chunks_and_arrive_whole():
    # hundreds of frames a chunk, sizes that leave gaps between them, frames that fill a chunk's
    # end, frames left to the runtime (900 KB, and page-locked ones) between those of the ring
    from compactcnncascade_amd import api
    import torch
    rng = np.random.default_rng(7)
    kinds = {"small": [(64, 56, 3, 700), (101, 99, 3, 90)], "mixed": [(64, 56, 3, 40), (320, 240, 3, 20), (640, 480, 3, 4),
                                                                     (61, 63, 4, 40), (1280, 720, 3, 2)],
             "large": [(640, 480, 3, 8), (1280, 720, 3, 3)]}
    for name, parts in kinds.items():
        d = api.FaceDetector()
        assert d.Init(api.Param(max_image_size=(1280, 720), min_face_height=24, max_face_height=60)) == 0
        frames = [rng.integers(0, 256, (h, w, c), np.uint8) for w, h, c, n in parts for _ in range(n)]
        frames = [frames[i] for i in rng.permutation(len(frames))]
        keep = [torch.from_numpy(f).clone().pin_memory() for f in frames]
        some = [keep[i].numpy() if i % 5 == 3 else f for i, f in enumerate(frames)]
        tensors = [torch.from_numpy(f).cuda() for f in frames]
        ptrs = [(t.data_ptr(), t.shape[1], t.shape[0], t.shape[2], t.shape[1] * t.shape[2]) for t in tensors]
        want = [_key(r) for r in d.DetectBatch(device_frames=ptrs)]
        assert sum(f.nbytes for f in frames) > 8 << 20
        for images in (frames, some, frames):
            print("small frames", name, len(frames), flush=True)
            assert [_key(r) for r in d.DetectBatch(images=images)] == want
