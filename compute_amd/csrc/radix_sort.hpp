// radix_sort.hpp -- the multi-tile radix sort: histogram, digit offsets and
// onesweep passes.  One instantiation unit per key width (and, for 4-byte
// keys, whose tile shapes are tunable, per value width) defines the
// radix_keys_* entry points: radix_u*.hip.
#pragma once

#include "onesweep.hpp"

#include <cstring>

namespace bcmi {

// ------------------------------------------------------------ histogram
// All passes' digit histograms in one read of the keys.  Each block counts
// its share in LDS and writes its partial histogram; k_digit_offsets then
// sums the partials per digit and scans them into exclusive digit offsets
// (ctrl->offsets).  No global atomics: device-scope atomics on shared
// addresses serialise across XCDs.
template <typename KB>
struct alignas(16) kchunk {
    static constexpr int N = 16 / sizeof(KB);
    KB v[N];
};

// Each group of L = kHistThreads / NW lanes counts into its own LDS
// sub-histogram: lanes adding to one bin in the same instruction serialise,
// which matters for skewed digits (the few top-digit values of floats in a
// narrow range); keys are read as 16-byte chunks, U per step, with the next
// step's U chunks in flight while a step is counted.
//
// BG = 0: sub-histogram s is 256 consecutive words per digit position, so
// bin d sits in bank d mod 64 for every sub and all 64 lanes of a wave
// contend for the banks.  BG = 1 (bank groups): the 64 / L subs of a wave
// interleave their bins so that sub sw uses only banks [sw * L, sw * L + L)
// (bin d at row d / L, column sw * L + d mod L of a 64-word row): the subs
// of a wave never contend, each sub's L lanes contend among L banks.
template <typename KB, typename XF, int U, int NW, int BG>
__global__ __launch_bounds__(kHistThreads) void k_histogram(const KB *__restrict__ keys, uint32_t n, uint32_t head,
                                                            XF xf, uint32_t *__restrict__ partial)
{
    constexpr int P = sizeof(KB);
    constexpr int L = kHistThreads / NW;  // lanes per sub
    static_assert(L <= kWave && kWave % L == 0, "subs within one wave");
    __shared__ uint32_t s_hist[NW * P * 256];
    for (int i = threadIdx.x; i < NW * P * 256; i += kHistThreads) s_hist[i] = 0;
    block_barrier();
    const uint32_t sub = threadIdx.x / L;
    // word of (position p, bin d) for this lane's sub
    auto slot = [&](int p, uint32_t d) -> uint32_t {
        if constexpr (BG) {
            constexpr uint32_t SPW = kWave / L;  // subs per wave
            const uint32_t w = sub / SPW, sw = sub % SPW;
            return ((w * P + (uint32_t)p) * SPW * 256) + (d / L) * kWave + sw * L + d % L;
        } else {
            return (sub * P + (uint32_t)p) * 256 + d;
        }
    };
    auto count = [&](KB x) {
        KB k = xf.key(x);
#pragma unroll
        for (int p = 0; p < P; ++p) atomicAdd(&s_hist[slot(p, (uint32_t)(k >> (8 * p)) & 0xFF)], 1u);
    };
    // unaligned head and the tail: block 0
    const uint64_t nchunks = (n - head) / kchunk<KB>::N;
    const uint64_t tail0 = head + nchunks * kchunk<KB>::N;
    if (blockIdx.x == 0) {
        for (uint32_t i = threadIdx.x; i < head; i += kHistThreads) count(keys[i]);
        for (uint64_t i = tail0 + threadIdx.x; i < n; i += kHistThreads) count(keys[i]);
    }
    const kchunk<KB> *body = (const kchunk<KB> *)(keys + head);
    const uint64_t stride = (uint64_t)gridDim.x * kHistThreads;
    uint64_t c = (uint64_t)blockIdx.x * kHistThreads + threadIdx.x;
    // U chunks per step, the next step's chunks loaded before this step's
    // are counted (2U in flight while the LDS works)
    if (c + (U - 1) * stride < nchunks) {
        kchunk<KB> cur[U];
#pragma unroll
        for (int u = 0; u < U; ++u) cur[u] = body[c + u * stride];
        while (true) {
            const uint64_t nc = c + U * stride;
            const bool more = nc + (U - 1) * stride < nchunks;
            kchunk<KB> nxt[U];
            if (more) {
#pragma unroll
                for (int u = 0; u < U; ++u) nxt[u] = body[nc + u * stride];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int k = 0; k < kchunk<KB>::N; ++k) count(cur[u].v[k]);
            c = nc;
            if (!more) break;
#pragma unroll
            for (int u = 0; u < U; ++u) cur[u] = nxt[u];
        }
    }
    for (; c < nchunks; c += stride) {
        const kchunk<KB> a = body[c];
#pragma unroll
        for (int k = 0; k < kchunk<KB>::N; ++k) count(a.v[k]);
    }
    block_barrier();
    uint32_t *dst = partial + (size_t)blockIdx.x * P * 256;
    for (int i = threadIdx.x; i < P * 256; i += kHistThreads) {
        const uint32_t p = (uint32_t)i / 256, d = (uint32_t)i % 256;
        uint32_t t = 0;
#pragma unroll
        for (uint32_t s = 0; s < (uint32_t)NW; ++s) {
            if constexpr (BG) {
                constexpr uint32_t SPW = kWave / L;
                t += s_hist[((s / SPW * P + p) * SPW * 256) + (d / L) * kWave + (s % SPW) * L + d % L];
            } else {
                t += s_hist[(s * P + p) * 256 + d];
            }
        }
        dst[i] = t;
    }
}

// The histogram's shape: chunks in flight per thread, sub-histograms per
// block (LDS: subs * key bytes KB), blocks per CU, bank-grouped layout.
// Tuning cache keys "__bcmi_radix_hist" and, for sorts with values,
// "__bcmi_radix_hist_by_key"; params "unroll" (1, 2, 4, 8), "subs"
// (8 or 16; 8 for 8-byte keys), "blocks_per_cu" and "bank_groups" (0, 1);
// the defaults were the fastest measured on 2^27 uint32 keys.
struct HistShape {
    int unroll, subs, blocks_per_cu, bank_groups;
};

static HistShape hist_shape(size_t key_bytes, bool tuned, bool values)
{
    HistShape h{4, 16, 2, 0};
    if (tuned) {
        // sorts with values read "__bcmi_radix_hist_by_key" where it is set
        // (their benchmark's float keys have a skewed top digit)
        const char *k0 = "__bcmi_radix_hist", *k1 = values ? "__bcmi_radix_hist_by_key" : k0;
        h.unroll = (int)tune_get(k1, "unroll", tune_get(k0, "unroll", 4));
        h.subs = (int)tune_get(k1, "subs", tune_get(k0, "subs", 16));
        h.blocks_per_cu = (int)tune_get(k1, "blocks_per_cu", tune_get(k0, "blocks_per_cu", 2));
        h.bank_groups = tune_get(k1, "bank_groups", tune_get(k0, "bank_groups", 0)) ? 1 : 0;
    }
    if (h.unroll != 1 && h.unroll != 2 && h.unroll != 8) h.unroll = 4;
    if (h.subs != 8 || key_bytes >= 8) h.subs = key_bytes >= 8 ? 8 : 16;
    if (h.blocks_per_cu < 1 || h.blocks_per_cu > 8) h.blocks_per_cu = 2;
    return h;
}

template <typename KB, typename XF>
static int launch_histogram(bcmi_queue q, const HistShape &hs, uint32_t hblocks, const KB *keys, uint32_t n,
                            uint32_t head, XF xf, uint32_t *partial)
{
#define BCMI_HIST(U, NW, BG)                                                                                     \
    if (hs.unroll == U && hs.subs == NW && hs.bank_groups == BG) {                                              \
        BCMI_LAUNCH(q, "radix_histogram",                                                                       \
                    hipLaunchKernelGGL((k_histogram<KB, XF, U, NW, BG>), dim3(hblocks), dim3(kHistThreads), 0,  \
                                       q->stream, keys, n, head, xf, partial));                                 \
        return 0;                                                                                               \
    }
    if constexpr (sizeof(KB) < 8) {
        BCMI_HIST(1, 16, 0) BCMI_HIST(2, 16, 0) BCMI_HIST(4, 16, 0) BCMI_HIST(8, 16, 0)
        BCMI_HIST(1, 16, 1) BCMI_HIST(2, 16, 1) BCMI_HIST(4, 16, 1) BCMI_HIST(8, 16, 1)
    }
    BCMI_HIST(1, 8, 0) BCMI_HIST(2, 8, 0) BCMI_HIST(4, 8, 0) BCMI_HIST(8, 8, 0)
    BCMI_HIST(1, 8, 1) BCMI_HIST(2, 8, 1) BCMI_HIST(4, 8, 1) BCMI_HIST(8, 8, 1)
#undef BCMI_HIST
    set_error("sort: histogram shape unroll=%d subs=%d not built", hs.unroll, hs.subs);
    return BCMI_INVALID_VALUE;
}

// Sums the histogram blocks' partials per digit, scans them into
// ctrl->offsets and marks the passes that move nothing (radix_sort.hip).
constexpr uint32_t kOffsetBlocks = 4;
__global__ void k_digit_offsets(const uint32_t *partial, uint32_t nparts, uint32_t passes, uint32_t n, Ctrl *ctrl,
                                uint64_t *status, uint32_t ep);
__global__ void k_clear_words(uint64_t *p, size_t n);

inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Workspace of one radix sort: the queue's arena and status array (base ==
// nullptr), or a fixed region the caller hands in (the allocation-free entry
// point's device scratch), carved into [status words | partial histograms |
// key temporaries | value temporaries].
struct SortWork {
    unsigned char *base;
    size_t bytes;
};

template <typename KB, int VB, int TH, int IPT, int SPLIT, int LB, int WPE, int CBG, typename XF>
static int radix_sort_xf(bcmi_queue q, void *keys_, void *vals_, uint32_t n, XF xf, const SortWork *work,
                         unsigned xrun)
{
    using V = typename ValT<VB>::type;
    constexpr int P = sizeof(KB);
    constexpr uint32_t TILE = TH * IPT;
    KB *keys = (KB *)keys_;
    V *vals = (V *)vals_;
    const uint32_t tiles = (n + TILE - 1) / TILE;
    // XCD-grouped tile order only where the device holds at least twice a
    // group of 8 * xrun workgroups at once (LDS and thread limits of a CU)
    {
        const size_t per_cu_lds = (size_t)kLdsBytesPerCU / sizeof(QSweepLds<TH, IPT, KB, VB, SPLIT>);
        const size_t per_cu = per_cu_lds < (size_t)(2048 / TH) ? per_cu_lds : (size_t)(2048 / TH);
        if (xrun > 16 || (size_t)q->cu_count * per_cu < 16 * (size_t)xrun) xrun = 0;
    }
    const HistShape hs = hist_shape(sizeof(KB), work == nullptr, VB > 0);
    uint32_t hblocks = (n + kHistThreads * 32 - 1) / (kHistThreads * 32);
    uint32_t hmax = (uint32_t)(q->cu_count * hs.blocks_per_cu);
    if (hblocks > hmax) hblocks = hmax;
    if (hblocks < 1) hblocks = 1;
    uint32_t head = 0;
    if ((uintptr_t)keys & 15) head = (uint32_t)((16 - ((uintptr_t)keys & 15)) / sizeof(KB));
    if (((uintptr_t)keys & 15) % sizeof(KB)) head = n;  // not element-aligned to a chunk
    if (head > n) head = n;
    const size_t kbytes = align256((size_t)n * sizeof(KB));
    const size_t vbytes = align256(VB ? (size_t)n * VB : 0);
    const size_t pbytes = align256((size_t)hblocks * P * 256 * 4);
    const size_t swords = (size_t)tiles * 256;
    unsigned char *scr;
    uint64_t *status;
    if (work) {
        const size_t need = align256(swords * 8) + pbytes + kbytes + vbytes;
        BCMI_CHECK(need <= work->bytes, BCMI_INVALID_BUFFER_SIZE,
                   "sort_noalloc: %u keys of %zu bytes with %d-byte values need %zu bytes of scratch; "
                   "the allocation-free sort has %zu", n, sizeof(KB), VB, need, work->bytes);
        status = (uint64_t *)work->base;
        scr = work->base + align256(swords * 8);
        // the words may carry another queue's epochs: clear them (a fill
        // kernel, so the call stays capturable)
        BCMI_LAUNCH(q, "radix_clear_status",
                    hipLaunchKernelGGL(k_clear_words, dim3((unsigned)((swords + 255) / 256 < 4096 ? (swords + 255) / 256 : 4096)),
                                       dim3(256), 0, q->stream, status, swords));
    } else {
        void *a;
        BCMI_TRY(scratch(q, pbytes + kbytes + vbytes, &a));
        scr = (unsigned char *)a;
        BCMI_TRY(status_array(q, swords, &status));
    }
    uint32_t *partial = (uint32_t *)scr;
    KB *ktmp = (KB *)(scr + pbytes);
    V *vtmp = (V *)(scr + pbytes + kbytes);

    BCMI_TRY(launch_histogram(q, hs, hblocks, keys, n, head, xf, partial));
    Epochs ep;
    BCMI_TRY(begin_lookback(q, P + 1, &ep));
    BCMI_LAUNCH(q, "radix_digit_offsets",
                hipLaunchKernelGGL(k_digit_offsets, dim3(P * kOffsetBlocks), dim3(1024), 0, q->stream, partial, hblocks,
                                   (uint32_t)P, n, q->ctrl, status, ep.arg(0)));
    for (int p = 0; p < P; ++p)
        BCMI_LAUNCH(q, "radix_onesweep",
                    hipLaunchKernelGGL((k_qsweep<TH, IPT, KB, VB, SPLIT, LB, WPE, XF, CBG>), dim3(tiles), dim3(TH), 0,
                                       q->stream, keys, ktmp, vals, vtmp, n, (uint32_t)p, xf, q->ctrl, status,
                                       ep.arg((uint32_t)p + 1), (uint32_t)xrun));
    if (P & 1) {
        // one pass (8-bit keys): the result is in the temporary
        BCMI_HIP(hipMemcpyAsync(keys, ktmp, (size_t)n * sizeof(KB), hipMemcpyDeviceToDevice, q->stream));
        if (VB) BCMI_HIP(hipMemcpyAsync(vals, vtmp, (size_t)n * VB, hipMemcpyDeviceToDevice, q->stream));
    }
    return 0;
}

template <typename KB, int VB, int TH, int IPT, int SPLIT = 1, int LB = 4, int WPE = 1, int CBG = 0>
static int radix_sort(bcmi_queue q, void *keys, void *vals, uint32_t n, int kind, int descending,
                      const SortWork *work, unsigned xrun)
{
    return with_key_xf<KB>(kind, descending, [&](auto xf) {
        return radix_sort_xf<KB, VB, TH, IPT, SPLIT, LB, WPE, CBG>(q, keys, vals, n, xf, work, xrun);
    });
}

// Tile shape: threads per workgroup, keys per thread, staging rounds and
// predecessor words per look-back round trip, by the number of keys.
//
// A pass over a few hundred tiles is bound by one tile's chain of latencies
// (load, count, scan, rank, look-back, scattered store), so small sorts take
// tiles of 4096 keys held by many threads with few keys each (the ranking
// chain is 3 dependent LDS round trips per key of a thread), and tiles grow
// with n: a longer digit run per tile writes fuller lines, and half the tiles
// are half the look-backs.  Each line below lies where the two sides met; us
// a call with the copy of the input, smaller tile first.
//   uint32            512 x 8 | 512 x 16     2^18: 46.5 47.5   2^19: 56.3 54.6
//                     512 x 16 | 1024 x 16   2^21: 84.7 85.6   4 M: 107 100
//                     1024 x 16 | tuned      8 M: 137 141 (512 x 32)   16 M: 212 204
//   float + u32       512 x 8 | 512 x 16     2^20: 81.7 84.4   2^21: over 104, 98.9
//                     512 x 16 | tuned       4 M: 132 134   8 M: 204 195
//   uint64            512 x 8 | 512 x 16     2^18: 91 98   2^20: 144 142
//                     512 x 16 | 512 x 32    4 M: 223 over 224   8 M: over 328, 305
//   uint64 + u32      512 x 8 | 512 x 16     2^20: 153 158   1.5 M: 179 171
//   8-byte values: the last two lines' shapes; at 8 M and more their tiles
//   are staged in two rounds and grouped by XCD (uint64 + u32 8 M: 480 437).
// (256 x 16 up to 2^20 and 256 x 32 up to 2^23 before: uint32 73.2 at 2^20,
// 156 at 8 M; uint64, always 256 x 16, 410 at 8 M and 792 at 16 M.)
//
// Above those sizes 4-byte keys with no or 4-byte values take the shape of
// the tuning cache (key "__bcmi_radix_sort", or "__bcmi_radix_sort_by_key"
// with values; params "threads", "ipt", "split", "lookback", "waves" (a
// register bound, waves per SIMD; 0 = none) and "count_bg" (1: bank-grouped
// count words)), chosen on 2^27 keys; the combinations built are listed
// below.  Param "fit_size" = 0 keeps the tuned shape at every size.  1- and
// 2-byte keys and other value widths take a fixed shape.  The allocation-free
// sort (work != nullptr) reads no tuning cache and keeps to the two smallest
// shapes.
template <typename KB, int VB>
static int radix_sort_shape(bcmi_queue q, void *keys, void *vals, uint32_t n, int kind, int desc,
                            const SortWork *work)
{
    constexpr int SB = (int)sizeof(KB) > VB ? (int)sizeof(KB) : VB;
    const char *key = VB ? "__bcmi_radix_sort_by_key" : "__bcmi_radix_sort";
    const unsigned xrun = work ? 0u : tune_get(key, "xcd_run", 0);
    if constexpr (sizeof(KB) == 4 && (VB == 0 || VB == 4)) {
        if (work || tune_get(key, "fit_size", 1) != 0) {
            if (n <= (VB ? 1u << 20 : 1u << 18))
                return radix_sort<KB, VB, 512, 8, 1, 8>(q, keys, vals, n, kind, desc, work, 0);
            if constexpr (VB == 0) {
                if (work || n <= 2500000)
                    return radix_sort<KB, VB, 512, 16, 1, 8>(q, keys, vals, n, kind, desc, work, 0);
                if (n <= 12000000) return radix_sort<KB, VB, 1024, 16, 1, 8>(q, keys, vals, n, kind, desc, work, 0);
            } else {
                if (work || n <= 5000000)
                    return radix_sort<KB, VB, 512, 16, 2, 4, 1, 1>(q, keys, vals, n, kind, desc, work, 0);
            }
        }
        const unsigned th = tune_get(key, "threads", 512);
        const unsigned ipt = tune_get(key, "ipt", 32);
        const unsigned split = tune_get(key, "split", 1);
        const unsigned lb = tune_get(key, "lookback", 4);
        const unsigned wpe = tune_get(key, "waves", 0);
        const unsigned cbg = tune_get(key, "count_bg", 0);
        // register bounds (param "waves": waves per SIMD) that raise the
        // workgroups per CU to what the LDS allows without spills, and
        // look-back windows other than 4 words per round trip, for the
        // tuned shapes; any other combination takes the plain shape
#define BCMI_SHAPE_LB(T, I, S, W, E)                                                                        \
        if constexpr (sizeof(QSweepLds<T, I, KB, VB, S>) <= (size_t)kLdsBytesPerCU)                         \
            if (th == T && ipt == I && split == S && lb == W && wpe == E && cbg == 0)                      \
                return radix_sort<KB, VB, T, I, S, W, E>(q, keys, vals, n, kind, desc, work, xrun)
        // bank-grouped count words (param "count_bg" = 1) for the shapes
        // that tune best
#define BCMI_SHAPE_CB(T, I, S, W, E)                                                                        \
        if constexpr (sizeof(QSweepLds<T, I, KB, VB, S>) <= (size_t)kLdsBytesPerCU)                         \
            if (th == T && ipt == I && split == S && lb == W && wpe == E && cbg == 1)                      \
                return radix_sort<KB, VB, T, I, S, W, E, 1>(q, keys, vals, n, kind, desc, work, xrun)
        BCMI_SHAPE_CB(512, 64, 2, 2, 4);
        BCMI_SHAPE_CB(256, 64, 2, 2, 4);
        BCMI_SHAPE_CB(512, 32, 2, 2, 0);
        BCMI_SHAPE_CB(512, 32, 2, 2, 7);
        BCMI_SHAPE_LB(256, 64, 2, 2, 0);
        BCMI_SHAPE_LB(512, 32, 2, 2, 0);
        BCMI_SHAPE_LB(256, 64, 2, 2, 4);
        BCMI_SHAPE_LB(512, 24, 2, 2, 8);
        BCMI_SHAPE_LB(512, 32, 2, 2, 7);
        BCMI_SHAPE_LB(512, 16, 1, 4, 8);
        BCMI_SHAPE_LB(512, 64, 2, 2, 4);
        BCMI_SHAPE_LB(512, 64, 4, 2, 4);
        BCMI_SHAPE_LB(1024, 32, 2, 2, 0);
        BCMI_SHAPE_LB(1024, 32, 4, 2, 0);
#undef BCMI_SHAPE_LB
#undef BCMI_SHAPE_CB
#define BCMI_SHAPE(T, I, S) \
        if (th == T && ipt == I && split == S) return radix_sort<KB, VB, T, I, S>(q, keys, vals, n, kind, desc, work, xrun)
        BCMI_SHAPE(256, 16, 1);
        BCMI_SHAPE(256, 32, 1);
        BCMI_SHAPE(256, 64, 1);
        BCMI_SHAPE(512, 16, 1);
        BCMI_SHAPE(512, 24, 1);
        BCMI_SHAPE(512, 32, 1);
        BCMI_SHAPE(1024, 16, 1);
        BCMI_SHAPE(256, 64, 2);
        BCMI_SHAPE(512, 24, 2);
        BCMI_SHAPE(512, 32, 2);
        BCMI_SHAPE(512, 24, 3);
#undef BCMI_SHAPE
        // any other value falls through to the generic shape below
    }
    if constexpr ((sizeof(KB) == 8 && (VB == 0 || VB == 4 || VB == 8)) || (sizeof(KB) == 4 && VB == 8)) {
        if (work || n <= (VB ? 1u << 20 : 1u << 19))
            return radix_sort<KB, VB, 512, 8, 1, 8>(q, keys, vals, n, kind, desc, work, 0);
        if (n <= 6000000) return radix_sort<KB, VB, 512, 16, 1, 8>(q, keys, vals, n, kind, desc, work, 0);
        if constexpr (VB == 0) return radix_sort<KB, VB, 512, 32, 2, 2>(q, keys, vals, n, kind, desc, work, xrun);
        else return radix_sort<KB, VB, 512, 16, 2, 4>(q, keys, vals, n, kind, desc, work, xrun);
    }
    if constexpr (SB >= 8) return radix_sort<KB, VB, 256, 16>(q, keys, vals, n, kind, desc, work, xrun);
    else return radix_sort<KB, VB, 256, 32>(q, keys, vals, n, kind, desc, work, xrun);
}

#define BCMI_RADIX_SIGNATURE(NAME)                                                                              \
    int NAME(bcmi_queue q, void *keys, void *vals, size_t vb, uint32_t n, int kind, int desc, const SortWork *work)

BCMI_RADIX_SIGNATURE(radix_keys_u8);
BCMI_RADIX_SIGNATURE(radix_keys_u16);
BCMI_RADIX_SIGNATURE(radix_keys_u32);     // 1-, 2-, 8- and 16-byte values
BCMI_RADIX_SIGNATURE(radix_keys_u32_v0);  // no values
BCMI_RADIX_SIGNATURE(radix_keys_u32_v4);  // 4-byte values
BCMI_RADIX_SIGNATURE(radix_keys_u64);

#define BCMI_RADIX_CASE(KB, VB) \
    case VB: return radix_sort_shape<KB, VB>(q, keys, VB ? vals : nullptr, n, kind, desc, work);

}  // namespace bcmi
