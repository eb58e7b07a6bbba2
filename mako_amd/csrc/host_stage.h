// The inputs of a host-pointer call on their way to device memory.  Plain C++: the host test puts a link of its own in HIP's
// place.
#pragma once

#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>

namespace mako {

constexpr size_t kStageAlign = 256;
constexpr size_t kStagePinned = (size_t)16 << 20; // staging memory kept per context, at most
constexpr size_t kStageCopy = (size_t)1 << 20;    // bytes per copy: a copy costs 8 us and a MiB's transfer 20, putting it together 12
constexpr size_t kStageSmall = (size_t)16 << 10; // bytes that the runtime copies for 5 us less than one more

// Arrays are put one after the other, each at a multiple of kStageAlign, into staging memory on the host, from where every
// kStageCopy bytes are copied to the same places of the context's block of device memory.
// Link: int copy(size_t to, const void* from, size_t bytes), which may return before the copy has read `from`, and int wait()
// until all of them have; both 0 or an error.
template <typename Link>
struct HostStage {
    Link link;
    unsigned char* mem;
    size_t mem_bytes, room;  // of the staging memory and of the block
    size_t at = 0, sent = 0; // bytes put and bytes copied, of the block
    size_t base = 0;         // byte of the block that is at the staging memory's start
    int status = 0;

    HostStage(Link l, unsigned char* staging, size_t staging_bytes, size_t block_bytes) : link(l), mem(staging), mem_bytes(staging_bytes), room(block_bytes) {}

    void flush()
    {
        if (at > sent && status == 0)
            status = link.copy(sent, mem + (sent - base), at - sent);
        sent = at;
    }
    void append(const void* src, size_t bytes)
    {
        const unsigned char* from = static_cast<const unsigned char*>(src);
        while (bytes && status == 0) {
            if (at - base == mem_bytes) { // (the staging memory is full: again from its start, when it has been read)
                flush();
                if (status == 0)
                    status = link.wait();
                base = at;
            }
            const size_t n = std::min({bytes, mem_bytes - (at - base), kStageCopy - (at - sent)});
            memcpy(mem + (at - base), from, n);
            at += n;
            from += n;
            bytes -= n;
            if (at - sent == kStageCopy)
                flush();
        }
    }
    void skip(size_t bytes) // (nobody reads what these hold)
    {
        static const unsigned char zeros[kStageAlign] = {};
        while (bytes && status == 0) {
            const size_t n = std::min(bytes, kStageAlign);
            append(zeros, n);
            bytes -= n;
        }
    }
    // Returns where in the block the rows are.
    size_t put_rows(const void* src, size_t src_stride, size_t bytes, size_t stride, uint32_t rows)
    {
        skip((kStageAlign - at % kStageAlign) % kStageAlign);
        const size_t place = at;
        if (at + rows * stride > room) { // (never: the block holds the context's largest call)
            status = status ? status : -1;
            return place;
        }
        if (src_stride == bytes && stride == bytes) {
            append(src, bytes * rows);
            return place;
        }
        for (uint32_t r = 0; r < rows; ++r) {
            append(static_cast<const unsigned char*>(src) + r * src_stride, bytes);
            skip(stride - bytes);
        }
        return place;
    }
    size_t put(const void* src, size_t bytes) { return put_rows(src, bytes, bytes, bytes, 1u); }
    // The rest on its way.  Behind a failure nothing reads the staging memory any more, which the next call writes.
    int send()
    {
        flush();
        if (status != 0)
            (void)link.wait();
        return status;
    }
};

} // namespace mako
