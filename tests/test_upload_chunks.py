"""How uploads are dealt to chunks (csrc/ccnn_upload.h) and which frames take the ring
(HostUpload::worth): the header compiled for the host and run on a simulated device. Every byte of
a frame arrives, no byte of a frame that is sent some other way is touched, chunks start
16-byte aligned, and many small frames make as few chunks as one large one."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "compactcnncascade_amd", "csrc")

CHUNKS = r"""
#include "ccnn_upload.h"
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>
using ccnn::UploadChunks;
static void fail(const char* what, int k) { std::printf("%s (case %d)\n", what, k); std::exit(1); }
static uint8_t value(int frame, size_t b) { return (uint8_t)((frame * 31 + b * 7 + (b >> 8)) % 200); }

int main()
{
    std::mt19937 rng(5);
    const size_t most = 768 << 10;
    for (int k = 0; k < 96; ++k) {
        // frames of one kind or mixed, some of them sent another way (frames of page-locked memory)
        const int n = 1 + (int)(rng() % 40), other = k % 3 == 2 ? 4 : 0;
        std::vector<size_t> len(n), off(n);
        std::vector<int> own(n);
        size_t total = 0, frames = 0;
        for (int i = 0; i < n; ++i) {
            const unsigned kind = k % 2 ? rng() % 4 : k / 2 % 4;
            len[i] = kind == 0 ? 1 + rng() % 300 : kind == 1 ? 1 + rng() % 40000 : kind == 2 ? 1 + rng() % 900000
                   : (rng() % 3 + 1) * most / 2;
            own[i] = other && rng() % other == 0 ? 0 : 1;
            off[i] = total;
            total += (len[i] + 255) / 256 * 256;
            frames += own[i];
        }
        std::vector<uint8_t> dev(total + 16, 0xEE), stage(most, 0xDD);
        std::vector<std::vector<uint8_t>> src(n);
        int sent = 0, breaks = 0;
        UploadChunks c;
        c.begin(total, most);
        const auto copy = [&](size_t o, const uint8_t* s, size_t m) {
            if (o + m > most) fail("chunk past the staging buffer", k);
            std::memcpy(stage.data() + o, s, m);
            return 0;
        };
        const auto send = [&](uint8_t* dst, size_t m) {
            if ((size_t)(dst - dev.data()) % 16 != 0) fail("misaligned chunk", k);
            if (m == 0 || m > most || dst < dev.data() || dst + m > dev.data() + total) fail("chunk out of range", k);
            std::memcpy(dst, stage.data(), m);
            ++sent;
            return 0;
        };
        for (int i = 0; i < n; ++i) {
            src[i].resize(len[i]);
            for (size_t b = 0; b < len[i]; ++b) src[i][b] = value(i, b);
            if (!own[i]) { ++breaks; continue; }
            if (c.put(dev.data() + off[i], src[i].data(), len[i], copy, send) < 0) fail("put", k);
            std::fill(src[i].begin(), src[i].end(), 0xCC);      // the caller's again
        }
        if (c.end(send) < 0) fail("end", k);
        for (int i = 0; i < n; ++i)
            for (size_t b = 0; b < len[i]; ++b)
                if (dev[off[i] + b] != (own[i] ? value(i, b) : 0xEE))
                    fail(own[i] ? "a byte did not arrive" : "another frame was touched", k);
        const size_t chunks = (total + most - 1) / most;
        if (frames && sent > (int)(2 * chunks) + breaks + 1) fail("too many chunks", k);
        if (!breaks && sent > (int)chunks + 1) fail("frames do not share chunks", k);
    }
    // exact contents: two frames around a chunk's end, a gap between them
    std::vector<uint8_t> dev(1 << 20, 0xEE), a(5000), b(7001);
    for (size_t i = 0; i < a.size(); ++i) a[i] = (uint8_t)(i * 7);
    for (size_t i = 0; i < b.size(); ++i) b[i] = (uint8_t)(i * 11 + 3);
    std::vector<uint8_t> st(4096);
    UploadChunks c;
    c.begin(12288, 4096);
    int sent = 0;
    const auto copy = [&](size_t o, const uint8_t* s, size_t m) { std::memcpy(st.data() + o, s, m); return 0; };
    const auto send = [&](uint8_t* d, size_t m) { std::memcpy(d, st.data(), m); ++sent; return 0; };
    c.put(dev.data(), a.data(), a.size(), copy, send);
    c.put(dev.data() + 5120, b.data(), b.size(), copy, send);
    c.end(send);
    if (std::memcmp(dev.data(), a.data(), a.size()) || std::memcmp(dev.data() + 5120, b.data(), b.size()) || sent != 3)
        fail("contents", -1);
    // a failure is handed on, and the next call begins afresh
    c.begin(5000, 4096);
    if (c.put(dev.data(), a.data(), a.size(), copy, [](uint8_t*, size_t) { return -1; }) != -1) fail("error lost", -2);
    c.begin(5000, 4096);
    sent = 0;
    if (c.put(dev.data() + 65536, a.data(), a.size(), copy, send) < 0 || c.end(send) < 0 || sent != 2 ||
        std::memcmp(dev.data() + 65536, a.data(), a.size())) fail("after a failure", -3);
    std::printf("ok\n");
}
"""

RULE = r"""
#include "ccnn_detector.h"
using ccnn::HostUpload;
constexpr size_t K = 1 << 10, M = 1 << 20;
static_assert(!HostUpload::worth(6 * M, 6 * M, 6 * M), "calls below 8 MB");
static_assert(HostUpload::worth(9 * M, 9 * M, 9 * M), "one large frame");
static_assert(HostUpload::worth(10 * K, 10 * K, 12 * M), "many small frames");
static_assert(!HostUpload::worth(900 * K, 900 * K, 28 * M), "640x480 frames: the runtime sends them in one piece");
static_assert(!HostUpload::worth(M, M, 28 * M) && HostUpload::worth(M + 1, M + 1, 28 * M), "up to 1 MB");
static_assert(HostUpload::worth(900 * K, 225 * K, 28 * M), "with small frames between them");
static_assert(HostUpload::worth(6 * M, 900 * K, 28 * M) && !HostUpload::worth(900 * K, 900 * K, 28 * M), "mixed");
"""


def _compile(tmp_path, text, *args):
    src = tmp_path / "t.cpp"
    src.write_text(text)
    cmd = ["g++", "-std=c++17", "-O2", "-Wall", "-I" + CSRC, "-I" + os.path.join(ROOT, "include"), str(src)] + list(args)
    return subprocess.run(cmd, capture_output=True, text=True)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_frames_share_chunks_and_every_byte_arrives(tmp_path):
    out = _compile(tmp_path, CHUNKS, "-fsanitize=undefined", "-o", str(tmp_path / "t"))
    assert out.returncode == 0, out.stderr
    run = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and run.stdout.strip() == "ok", run.stdout + run.stderr


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include/hip"), reason="no HIP headers")
def test_which_frames_take_the_ring(tmp_path):
    out = _compile(tmp_path, RULE, "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-fsyntax-only")
    assert out.returncode == 0, out.stderr
