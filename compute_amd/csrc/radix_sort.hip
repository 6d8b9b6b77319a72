// radix_sort.hip -- sort / sort_by_key / stable_sort / stable_sort_by_key.
//
// Reference (GPU column): radix_sort_impl (algorithm/detail/radix_sort.hpp:
// 252-426): LSD radix with 4-bit digits and 128-thread blocks, i.e. 8 passes
// for 32-bit keys, each pass = count kernel + a recursive exclusive_scan of
// the per-block counts + a scan task + a scatter kernel whose rank loop is
// O(local id) (:234-239).  Below 33 (sort) or 32 (sort_by_key) elements a
// one-work-item insertion sort runs instead (sort.hpp:49-54,
// sort_by_key.hpp:48-51, insertion_sort.hpp:25-159).
//
// Here: onesweep LSD radix with 8-bit digits.  One histogram kernel reads
// the keys once and builds the digit histograms of every pass; then one
// kernel per pass: block b takes tile b, ranks its keys with
// wave64 ballot matching against per-wave LDS digit counters, publishes its
// per-digit counts, gets its global digit offsets by decoupled look-back,
// reorders the tile in LDS so each digit run is contiguous and writes keys
// (then values) out coalesced.  The order equals the reference's: a stable
// sort by the transformed key radix(x) (radix_sort.hpp:98-129).
#include "block_sort.hpp"
#include "radix_sort.hpp"

#include <mutex>

namespace bcmi {

// kOffsetBlocks blocks of 1024 threads per pass: wave w of block (p, part)
// sums 64 digits over every 16th partial histogram, the waves are combined in
// LDS and the digits scanned; the digits of earlier parts come from their
// blocks' totals, passed on as tagged words (a part waits for earlier blocks
// only).  A pass whose digit is the same in all n keys is marked in
// ctrl->single: its block passes on ~0, which no total reaches.  One block per
// pass read up to 1 MB of partials through one CU's cache: 15 us for 33.5 M
// keys with values, 8.5 us for 2^27 keys.
__global__ __launch_bounds__(1024) void k_digit_offsets(const uint32_t *__restrict__ partial, uint32_t nparts,
                                                        uint32_t passes, uint32_t n, Ctrl *ctrl, uint64_t *status,
                                                        uint32_t ep)
{
    __shared__ uint32_t s_part[16][64];
    const uint32_t p = blockIdx.x / kOffsetBlocks, part = blockIdx.x % kOffsetBlocks;
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6, d = part * 64 + lane;
    uint32_t c = 0;
#pragma unroll 8
    for (uint32_t b = w; b < nparts; b += 16) c += partial[((size_t)b * passes + p) * 256 + d];
    s_part[w][lane] = c;
    block_barrier();
    if (w != 0) return;
#pragma unroll
    for (int i = 1; i < 16; ++i) c += s_part[i][lane];
    const uint32_t epoch = launch_epoch(ctrl, ep);
    const uint32_t inc = wave_inclusive_scan(c, 0u, [](uint32_t a, uint32_t b) { return a + b; });
    bool single = ballot(c == n) != 0;
    if (lane == 0) lb_publish(status, blockIdx.x, epoch, LB_A, single ? ~0u : readlane(inc, 63));
    uint32_t before = 0, spins = 0;
    if (lane < part)
        while (lb_read(status, blockIdx.x - part + lane, epoch, before) == LB_X)
            if (spin_expired(ctrl, spins)) break;
    single = single || ballot(before == ~0u) != 0;
    before = wave_reduce(before == ~0u ? n : before, 0u, [](uint32_t a, uint32_t b) { return a + b; });
    ctrl->offsets[p][d] = before + inc - c;
    if (part == kOffsetBlocks - 1 && lane == 0) ctrl->single[p] = single ? 1u : 0u;
}

// ------------------------------------------------------- insertion sort
// serial_insertion_sort(_by_key) (insertion_sort.hpp:42-64, :106-133): one
// work-item, shift while compare(value, data[pos-1]) with operator< (less)
// or operator> (greater) on the native key type.
template <typename T, int VB>
__global__ void k_insertion(T *keys, typename ValT<VB>::type *vals, uint32_t n, int descending)
{
    using V = typename ValT<VB>::type;
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    for (uint32_t i = 1; i < n; ++i) {
        const T key = keys[i];
        V val{};
        if constexpr (VB > 0) val = vals[i];
        uint32_t pos = i;
        while (pos > 0 && (descending ? (key > keys[pos - 1]) : (key < keys[pos - 1]))) {
            keys[pos] = keys[pos - 1];
            if constexpr (VB > 0) vals[pos] = vals[pos - 1];
            pos--;
        }
        keys[pos] = key;
        if constexpr (VB > 0) vals[pos] = val;
    }
}

// Device scratch of bcmi_sort_noalloc: one copy per GPU, held until the
// process ends.  Host code never passes `scratch` itself to a kernel (in
// host code the name is a host-side stand-in); it uses the device address
// hipGetSymbolAddress returned for the current device, kept per device.
constexpr size_t kNoAllocScratchBytes = (size_t)64 << 20;
constexpr int kNoAllocMaxDevices = 64;
}  // namespace bcmi
static __device__ __align__(256) unsigned char scratch[bcmi::kNoAllocScratchBytes];
namespace bcmi {
static unsigned char *g_noalloc_ptr[kNoAllocMaxDevices];
static std::mutex g_noalloc_mu;

// Called by bcmi_queue_create with `device` current: looks up this device's
// copy of the scratch array once.
int noalloc_scratch_setup(int device)
{
    BCMI_CHECK(device >= 0 && device < kNoAllocMaxDevices, BCMI_DEVICE_NOT_FOUND,
               "device %d beyond the %d devices the allocation-free sort supports", device, kNoAllocMaxDevices);
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    if (g_noalloc_ptr[device]) return 0;
    void *p = nullptr;
    BCMI_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(::scratch)));
    BCMI_CHECK(p != nullptr, BCMI_RUNTIME_ERROR, "no device address for the sort scratch on device %d", device);
    g_noalloc_ptr[device] = (unsigned char *)p;
    return 0;
}

static unsigned char *noalloc_scratch(int device)
{
    if (device < 0 || device >= kNoAllocMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    return g_noalloc_ptr[device];
}

__global__ void k_clear_words(uint64_t *p, size_t n)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = 0;
}

// Bytes of queue scratch radix_sort_xf takes for n keys of key_bytes with
// value_bytes values (at most cu_count * 8 histogram blocks).  Callers that
// keep their own temporaries in the arena beside a sort place them after it.
size_t radix_scratch_bytes(size_t n, size_t key_bytes, size_t value_bytes, int cu_count)
{
    return align256(n * key_bytes) + align256(n * value_bytes) + align256((size_t)cu_count * 8 * key_bytes * 256 * 4);
}

template <typename T, int VB>
static int insertion_launch(bcmi_queue q, void *keys, void *vals, uint32_t n, int desc)
{
    BCMI_LAUNCH(q, "insertion_sort",
                hipLaunchKernelGGL((k_insertion<T, VB>), dim3(1), dim3(64), 0, q->stream, (T *)keys,
                                   (typename ValT<VB>::type *)vals, n, desc));
    return 0;
}

template <typename T>
static int insertion_vb(bcmi_queue q, void *keys, void *vals, size_t vb, uint32_t n, int desc)
{
    if (!vals) vb = 0;
    switch (vb) {
    case 0: return insertion_launch<T, 0>(q, keys, nullptr, n, desc);
    case 1: return insertion_launch<T, 1>(q, keys, vals, n, desc);
    case 2: return insertion_launch<T, 2>(q, keys, vals, n, desc);
    case 4: return insertion_launch<T, 4>(q, keys, vals, n, desc);
    case 8: return insertion_launch<T, 8>(q, keys, vals, n, desc);
    case 16: return insertion_launch<T, 16>(q, keys, vals, n, desc);
    default: set_error("sort: value size %zu unsupported (1, 2, 4, 8 or 16 bytes)", vb); return BCMI_INVALID_VALUE;
    }
}

static int dtype_kind(int dt)
{
    switch (dt) {
    case BCMI_I8: case BCMI_I16: case BCMI_I32: case BCMI_I64: return 1;
    case BCMI_F32: case BCMI_F64: return 2;
    default: return 0;
    }
}

}  // namespace bcmi

using namespace bcmi;

static int sort_entry(bcmi_queue q, int api, int key_dtype, void *keys, void *values, size_t value_bytes, size_t n,
                      int descending, const SortWork *work)
{
    BCMI_TRY(use_queue(q));
    BCMI_CHECK(dtype_valid(key_dtype), BCMI_INVALID_VALUE, "sort: bad key dtype %d", key_dtype);
    BCMI_CHECK(api >= BCMI_SORT && api <= BCMI_RADIX_SORT, BCMI_INVALID_VALUE, "sort: bad api %d", api);
    // 32-bit tile/offset arithmetic (the reference's counts are uint too,
    // radix_sort.hpp:131-137); the margin keeps the last tile in range.
    BCMI_CHECK(n <= (1ull << 32) - (1ull << 20), BCMI_INVALID_BUFFER_SIZE, "sort: n=%zu exceeds 2^32-2^20", n);
    if (n < 2) return 0;
    BCMI_CHECK(keys, BCMI_INVALID_VALUE, "sort: null keys");
    if (api == BCMI_SORT || api == BCMI_STABLE_SORT) values = nullptr;
    const uint32_t n32 = (uint32_t)n;
    const int desc = descending ? 1 : 0;
    const bool insertion = (api == BCMI_SORT && n <= 32) ||
                           ((api == BCMI_SORT_BY_KEY || api == BCMI_STABLE_SORT_BY_KEY) && n < 32);
    if (insertion) {
        switch (key_dtype) {
        case BCMI_I8: return insertion_vb<int8_t>(q, keys, values, value_bytes, n32, desc);
        case BCMI_U8: return insertion_vb<uint8_t>(q, keys, values, value_bytes, n32, desc);
        case BCMI_I16: return insertion_vb<int16_t>(q, keys, values, value_bytes, n32, desc);
        case BCMI_U16: return insertion_vb<uint16_t>(q, keys, values, value_bytes, n32, desc);
        case BCMI_I32: return insertion_vb<int32_t>(q, keys, values, value_bytes, n32, desc);
        case BCMI_U32: return insertion_vb<uint32_t>(q, keys, values, value_bytes, n32, desc);
        case BCMI_I64: return insertion_vb<int64_t>(q, keys, values, value_bytes, n32, desc);
        case BCMI_U64: return insertion_vb<uint64_t>(q, keys, values, value_bytes, n32, desc);
        case BCMI_F32: return insertion_vb<float>(q, keys, values, value_bytes, n32, desc);
        default: return insertion_vb<double>(q, keys, values, value_bytes, n32, desc);
        }
    }
    const int kind = dtype_kind(key_dtype);
    // a range that fits one workgroup: one launch, no temporaries
    if (block_sort_takes((size_t)dtype_size(key_dtype), values && value_bytes, kind, desc, n32))
        return block_sort(q, (size_t)dtype_size(key_dtype), keys, values, value_bytes, n32, kind, desc);
    const size_t vb = values ? value_bytes : 0;
    switch (dtype_size(key_dtype)) {
    case 1: return radix_keys_u8(q, keys, values, vb, n32, kind, desc, work);
    case 2: return radix_keys_u16(q, keys, values, vb, n32, kind, desc, work);
    case 4:
        if (vb == 0) return radix_keys_u32_v0(q, keys, values, vb, n32, kind, desc, work);
        if (vb == 4) return radix_keys_u32_v4(q, keys, values, vb, n32, kind, desc, work);
        return radix_keys_u32(q, keys, values, vb, n32, kind, desc, work);
    default: return radix_keys_u64(q, keys, values, vb, n32, kind, desc, work);
    }
}

extern "C" int bcmi_sort(bcmi_queue q, int api, int key_dtype, void *keys, void *values, size_t value_bytes, size_t n,
                         int descending)
{
    return sort_entry(q, api, key_dtype, keys, values, value_bytes, n, descending, nullptr);
}

// The same sort with every temporary in this device's copy of `scratch`:
// no allocation on any path.  Calls that overlap on one GPU (two queues at
// once) share the array and race; the array keeps the last call's contents.
extern "C" int bcmi_sort_noalloc(bcmi_queue q, int api, int key_dtype, void *keys, void *values, size_t value_bytes,
                                 size_t n, int descending)
{
    BCMI_TRY(use_queue(q));
    unsigned char *p = noalloc_scratch(q->device);
    BCMI_CHECK(p != nullptr, BCMI_INVALID_COMMAND_QUEUE, "sort_noalloc: no scratch set up for device %d", q->device);
    const SortWork w{p, kNoAllocScratchBytes};
    // the queue's kernel profiler creates its events on demand: off here
    const bool prof = q->profile;
    q->profile = false;
    const int r = sort_entry(q, api, key_dtype, keys, values, value_bytes, n, descending, &w);
    q->profile = prof;
    return r;
}
