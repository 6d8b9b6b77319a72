// Instantiation unit of radix_sort.hpp.
#include "radix_sort.hpp"

namespace bcmi {

BCMI_RADIX_SIGNATURE(radix_keys_u8)
{
    switch (vb) {
        BCMI_RADIX_CASE(uint8_t, 0)
        BCMI_RADIX_CASE(uint8_t, 1)
        BCMI_RADIX_CASE(uint8_t, 2)
        BCMI_RADIX_CASE(uint8_t, 4)
        BCMI_RADIX_CASE(uint8_t, 8)
        BCMI_RADIX_CASE(uint8_t, 16)
    default: set_error("sort: value size %zu unsupported (1, 2, 4, 8 or 16 bytes)", vb); return BCMI_INVALID_VALUE;
    }
}

}  // namespace bcmi
