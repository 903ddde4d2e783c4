/*
 * A host block of pieces at 256-byte offsets, for one copy to the device.
 */
#ifndef RC_BLOCK_H
#define RC_BLOCK_H

#include <stddef.h>
#include <string.h>

#include <vector>

class RcBlock {
public:
    /* Over the storage h, which keeps its capacity from call to call. */
    RcBlock(std::vector<unsigned char> &h, size_t expected) : h_(h)
    {
        h_.clear();
        h_.reserve(expected);
    }
    /* Appends a piece and returns its offset; of an empty one (src may be null)
       it is an offset that nothing is read from. */
    size_t put(const void *src, size_t bytes)
    {
        const size_t o = (h_.size() + 255) & ~(size_t)255;
        h_.resize(o + bytes);
        if (bytes > 0) memcpy(h_.data() + o, src, bytes);
        return o;
    }
    template <typename T> size_t put(const std::vector<T> &v)
    {
        return put(v.data(), sizeof(T) * v.size());
    }

private:
    std::vector<unsigned char> &h_;
};

#endif
