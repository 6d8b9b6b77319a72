// block_sort.hpp -- sort of a range that fits one workgroup (block_sort.hip).
#pragma once

#include "runtime.hpp"

namespace bcmi {

// Whether n keys go to the one-workgroup sort.  Up to 8192 keys it wins
// everywhere (us a call with the input's copy, multi-tile path first: 3001
// uint32 33.5 -> 14.4, 8001 uint32 40.4 -> 20.1, 8001 float keys with values
// 51.8 -> 31.8, 8001 uint64 73.4 -> 23.2, 8001 double keys with 8-byte values
// 100.0 -> 58.5).  Keys of up to 4 bytes that need not carry an index hold
// out to 16384 (40.3 -> 30.3); with an index the two meet there (52.1, 52.8),
// and 16384 8-byte keys do not fit the LDS.
inline bool block_sort_takes(size_t key_bytes, bool values, int kind, int desc, uint32_t n)
{
    const bool indexed = values || (kind == 2 && desc);
    return n <= (key_bytes <= 4 && !indexed ? 16384u : 8192u);
}

// Stable radix order of n keys that block_sort_takes, in place, with vb-byte
// values (vals NULL: none).  kind: 0 unsigned, 1 signed, 2 floating.
int block_sort(bcmi_queue q, size_t key_bytes, void *keys, void *vals, size_t vb, uint32_t n, int kind, int desc);

}  // namespace bcmi
