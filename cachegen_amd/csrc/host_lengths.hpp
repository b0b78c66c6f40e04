// Part of the CacheGen KV codec library for MI355X (gfx950); included by cachegen_hip.hip.  Stream
// lengths in host memory; plain C++, without HIP, so that a CPU sanitizer can be run over it.
#pragma once

#include <cstdint>
#include <cstring>

namespace {

// A value of a blob: a container's sections may begin at any byte of it (a pickle's do), so the value
// is copied out instead of being read through a pointer of its type.  The copies of a whole vector
// become one unaligned vector load.
template <typename T>
inline int32_t host_value(const char *p)
{
    T v;
    memcpy(&v, p, sizeof(v));
    return v;
}

// Bytes that streams occupy before every 64th stream of a row, from their lengths (T: int32_t or
// uint16_t) in host memory: lengths are min'ed with a stream's capacity; false if one is negative.
template <typename T>
bool host_tile_starts(const void *lengths, int64_t nsub, int64_t rows, int64_t C, int32_t capacity, uint32_t *starts, int64_t *sub_bytes)
{
    const char *row = static_cast<const char *>(lengths);
    const int64_t tiles = (C + 63) / 64;
    int32_t lowest = 0;
    for (int64_t s = 0; s < nsub; ++s) {
        uint32_t run = 0;                       // at most 256 bytes of at most 2^24 streams: checked by the caller
        for (int64_t r = 0; r < rows; ++r, row += C * sizeof(T))
            for (int64_t t = 0; t < tiles; ++t) {
                *starts++ = run;
                const int64_t n = C - t * 64 < 64 ? C - t * 64 : 64;
                const char *p = row + t * 64 * sizeof(T);
                int32_t sum = 0, low = 0;
                if (n == 64) {
                    for (int i = 0; i < 64; ++i) {          // a fixed count: vector instructions
                        const int32_t v = host_value<T>(p + i * sizeof(T));
                        sum += v < capacity ? v : capacity;
                        low = v < low ? v : low;
                    }
                } else {
                    for (int i = 0; i < n; ++i) {
                        const int32_t v = host_value<T>(p + i * sizeof(T));
                        sum += v < capacity ? v : capacity;
                        low = v < low ? v : low;
                    }
                }
                run += (uint32_t)sum;
                lowest = low < lowest ? low : lowest;
            }
        sub_bytes[s] = run;
    }
    return lowest >= 0;
}

}  // namespace
