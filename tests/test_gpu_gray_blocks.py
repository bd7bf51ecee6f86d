"""Gray conversion of batches at the edges of its blocks (256 groups of 16 pixels): frames that
end inside a block, frames of one block and of many, widths that end inside a group or a quad,
rows of every alignment and padded rows, against the oracle's gray values, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

#          w, h, channels, padding bytes a row
FRAMES = [(64, 64, 3, 0), (1024, 64, 3, 0), (1025, 67, 3, 0), (1027, 70, 4, 0), (1030, 66, 3, 2), (16, 300, 3, 0),
          (509, 131, 4, 4), (333, 97, 3, 1), (4096, 61, 3, 0), (771, 203, 4, 0), (48, 52, 3, 0), (2000, 80, 3, 3)]


@pytest.mark.parametrize("shift", [0, 1, 4])
def test_gray_of_batches_at_block_edges(shift):
    from compactcnncascade_amd import api
    from oracle.bind import Oracle
    import torch
    oracle = Oracle()
    rng = np.random.default_rng(shift)
    frames, keep, ptrs = [], [], []
    for w, h, ch, pad in FRAMES:
        step = w * ch + pad
        buf = rng.integers(0, 256, h * step + 16, np.uint8)
        t = torch.from_numpy(buf).cuda()
        keep.append(t)
        rows = buf[shift:shift + h * step].reshape(h, step)[:, :w * ch]
        frames.append(np.ascontiguousarray(rows).reshape(h, w, ch))
        ptrs.append((t.data_ptr() + shift, w, h, ch, step))
    # the gray image of a batch's last frame is what can be read back: each frame is the
    # last of a batch of all of them once
    d = api.FaceDetector()
    assert d.Init(api.Param(max_image_size=(4096, 300), min_face_height=50, max_face_height=60)) == 0
    for k in range(len(FRAMES)):
        if FRAMES[k][0] < 47:          # below the smallest frame that is searched: not converted
            continue
        order = [(k + 1 + j) % len(FRAMES) for j in range(len(FRAMES))]
        print("gray", shift, FRAMES[k], flush=True)
        d.DetectBatch(device_frames=[ptrs[j] for j in order])
        got = d.getGrayImage32F(api.PIPELINE_CPU)
        want = oracle.gray(frames[k])
        assert got.shape == want.shape
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), FRAMES[k]


@pytest.mark.parametrize("ch", [1, 3, 4])
@pytest.mark.parametrize("pad", [0, 1, 4, 16])
def test_gray_of_thumbnails(ch, pad):
    # frames of fewer than a block's groups, several in every block: whole groups, groups that
    # end at each pixel of a row, rows of every alignment
    from compactcnncascade_amd import api
    from oracle.bind import Oracle
    import torch
    oracle = Oracle()
    rng = np.random.default_rng(10 * ch + pad)
    frames, ptrs, keep = [], [], []
    for w in list(range(48, 68)) + [80, 96]:
        h = 51 + w % 5
        step = w * ch + pad
        buf = rng.integers(0, 256, (h, step), np.uint8)
        keep.append(torch.from_numpy(buf).cuda())
        rows = np.ascontiguousarray(buf[:, :w * ch])
        frames.append(rows.reshape(h, w) if ch == 1 else rows.reshape(h, w, ch))
        ptrs.append((keep[-1].data_ptr(), w, h, ch, step))
    d = api.FaceDetector()
    assert d.Init(api.Param(max_image_size=(128, 64), min_face_height=27, max_face_height=40)) == 0
    n = len(frames)
    print("thumbnails", ch, pad, flush=True)
    for k in range(n):
        d.DetectBatch(device_frames=[ptrs[(k + 1 + j) % n] for j in range(n)])
        got, want = d.getGrayImage32F(api.PIPELINE_CPU), oracle.gray(frames[k])
        assert got.shape == want.shape
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), frames[k].shape
