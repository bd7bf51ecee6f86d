// How the pieces of an upload (the frames of a batch, or one frame) are dealt to the chunks of
// a staging buffer. Host code without HIP.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace ccnn {

// A chunk is a contiguous stretch of the destination. A piece whose destination follows the
// piece before it within GAP bytes shares its chunk (the bytes between the two, which belong
// to neither, are sent as they are): many small frames make as few chunks as one large one.
class UploadChunks {
public:
    static constexpr size_t GAP = 256;     // frames lie back to back at steps of 256 bytes

    // a call of `bytes` bytes in all, in chunks of equal size (none is a small rest), a
    // multiple of 4096 and at most `most`, which is one too
    void begin(size_t bytes, size_t most)
    {
        const size_t n = std::max<size_t>(1, (bytes + most - 1) / most);
        size_ = std::min(most, std::max<size_t>(1, (bytes / n + 4095) / 4096) * 4096);
        used_ = 0;
    }
    // copy(offset in the chunk, source, bytes): offset 0 opens a chunk; send(destination,
    // bytes) ends it. Both return < 0 to stop, which is handed on.
    template <class Copy, class Send>
    int put(uint8_t* dst, const uint8_t* src, size_t bytes, Copy&& copy, Send&& send)
    {
        if (used_ > 0 && (dst < at_ + used_ || dst >= at_ + used_ + GAP || dst >= at_ + size_))
            if (end(send) < 0) return -1;
        while (bytes > 0) {
            if (used_ == 0) at_ = dst;
            const size_t o = (size_t)(dst - at_), n = std::min(bytes, size_ - o);
            if (copy(o, src, n) < 0) return -1;
            used_ = o + n;
            dst += n;
            src += n;
            bytes -= n;
            if (used_ == size_ && end(send) < 0) return -1;
        }
        return 0;
    }
    template <class Send>
    int end(Send&& send)
    {
        const size_t n = used_;
        used_ = 0;
        return n > 0 ? send(at_, n) : 0;
    }

private:
    size_t size_ = 0, used_ = 0;
    uint8_t* at_ = nullptr;
};

}  // namespace ccnn
