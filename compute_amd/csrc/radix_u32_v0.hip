// Instantiation unit of radix_sort.hpp.
#include "radix_sort.hpp"

namespace bcmi {

BCMI_RADIX_SIGNATURE(radix_keys_u32_v0)
{
    return radix_sort_shape<uint32_t, 0>(q, keys, nullptr, n, kind, desc, work);
}

}  // namespace bcmi
