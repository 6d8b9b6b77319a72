// segmented.hpp -- kernels and launches of the batched segmented sort, one
// instantiation unit per key width (segmented_u*.hip).
//
// Semantics: every segment [offsets[s], offsets[s+1]) ends up exactly as one
// stable_sort_by_key call on it would leave it in the reference's GPU
// column (stable_sort_by_key.hpp:29-77): below 32 elements the one-work-item
// insertion sort (insertion_sort.hpp:106-133, which only differs from radix
// order for float keys: it keeps -0.0/+0.0 in input order), otherwise the
// stable radix order of the radix() key transform (radix_sort.hpp:98-129).
//
// The reference has no batched primitive: the per-segment alternative is one
// sort call per segment (several launches each).  Here a plan built once
// from the host offsets routes the segments to three paths, each one launch
// (or one launch per 8-bit pass) for all segments together:
//   * small (<= 4096 elements): one workgroup per segment sorts it entirely
//     in LDS -- all digit passes, LDS-mask ranking, LDS scatter/gather --
//     so the segment's keys are read and written once;
//   * float keys shorter than 32: the reference's insertion sort, one
//     thread per segment;
//   * large: the onesweep pass kernel over a table of tiles of all large
//     segments, with per-segment digit histograms and look-back chains that
//     restart at every segment's first tile.
// A plan owns its tables and temporaries, so running it allocates nothing
// and can be captured in a hipGraph and replayed.
#pragma once

#include "onesweep.hpp"
#include "radix.hpp"
#include "segplan.hpp"

#include <cstring>
#include <vector>

namespace bcmi {

// ------------------------------------------------------------ small path
constexpr uint32_t kBucketMax = 64;  // largest bucket the one-pass sort finishes by insertion
constexpr uint32_t kBinMax = 32;     // largest bin whose keys are placed by counting

// The key forms of integers.
template <typename XF>
struct xf_is_integer : std::false_type {};
template <typename KB>
struct xf_is_integer<KeyXf<KB, kXfXor>> : std::true_type {};
template <typename KB>
struct xf_is_integer<KeyXf<KB, kXfNegXor>> : std::true_type {};

// Sorts each span of segs entirely in LDS.  The keys (values) are read from
// ksrc (vsrc) and the sorted span written to keys (vals) at the same offset;
// the small-segment route sorts in place (ksrc == keys).
//
// Integer keys are first dealt into bins: with [mn, mx] the span's range of
// transformed keys, bin(k) = (key(k) - mn) >> shift, one bin per key slot
// (up to 2048).  A returning LDS add gives each key a slot in its bin, in any
// order; a key's place in the span is then its bin's start plus the number of
// the bin's keys below it (by whole key, then by input position), which every
// thread counts for its own keys, so the span goes straight to memory.
// Spread-out keys share a bin with about one other: 24 LDS instructions a pair
// and 90 LDS cycles a wave's pairs, instead of 37 and 194 for two ranked passes
// and the insertions (SQ_INSTS_LDS, SQ_LDS_IDX_ACTIVE; spans of 2000 uint64 +
// uint32 pairs).  A bin over kBinMax keys, and float keys (which crowd the bins
// of their largest octaves), take the passes below; a span that tried has lost
// the adds, which take turns on the crowded bin, and the scan.  us a run with
// the copies, passes alone | bins first:
//   spread keys   100,000 x 30 uint32 + uint32: 149 105   20,000 x 512: 124 63
//                 6000 x 2048 uint64 + uint32: 123 112
//   crowded keys  20,000 x 512 uint32 + uint32 of e^U(0, 22): 236 267, of two
//                 values: 298 323; 6000 x 2048 uint64 in 30 clusters: 743 768
// Foreseeing the failure did not pay: the range's size against the length cost
// spread keys of short spans 3-4 %, a ballot over a sample of the keys 5-15 %,
// giving up on the first full slot 2 % (the adds' returns are waited for).
//
// Range-adaptive passes: rel(k) = (key(k) - mn) >> shift, shift chosen so rel
// fits 8 bits (spans up to 512 keys) or 16 bits, is monotone in the key.  One
// or two stable 8-bit LDS passes order the keys by rel; then each run of equal
// rel (a few keys for spread-out keys: 4096 keys over 2^16 values) is finished
// by a stable insertion sort on the whole key, owned by the thread holding
// the run's first slot.  If a run exceeds kBucketMax keys (clustered keys)
// the span takes all 8-bit LSD passes in LDS instead.
template <typename KB, int VB, int IPT, typename XF>
__global__ __launch_bounds__(kSegSmallThreads) void k_seg_small(const KB *ksrc, const typename ValT<VB>::type *vsrc,
                                                                KB *keys, typename ValT<VB>::type *vals,
                                                                const SegSpan *__restrict__ segs, XF xf)
{
    using V = typename ValT<VB>::type;
    constexpr int P = sizeof(KB);
    constexpr int TILE = kSegSmallThreads * IPT;
    __shared__ KB s_k[TILE];
    __shared__ V s_v[VB ? TILE : 1];
    // the passes' digit counters and peer masks, or the bins and the input
    // positions of the binned keys
    constexpr int NB = kSegSmallThreads * (IPT > 8 ? 8 : IPT);
    constexpr int WORK = NB * 4 + TILE * 2 > 4 * 256 * 12 ? NB * 4 + TILE * 2 : 4 * 256 * 12;
    __shared__ __align__(16) unsigned char s_work[WORK];
    uint32_t(*s_cnt)[256] = (uint32_t(*)[256])s_work;
    uint64_t(*s_peer)[256] = (uint64_t(*)[256])(s_work + 4 * 256 * 4);
    uint32_t *s_bin = (uint32_t *)s_work;
    uint16_t *s_idx = (uint16_t *)(s_work + NB * 4);
    __shared__ uint32_t s_wsum[4];
    __shared__ uint32_t s_uniform;
    __shared__ KB s_mn[4], s_mx[4];

    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const SegSpan sg = segs[blockIdx.x];
    const uint32_t len = sg.len;
    if (len == 0) return;  // an unused group slot
    const KB *ks = ksrc + sg.base;
    const V *vs = VB ? vsrc + sg.base : nullptr;
    KB *kp = keys + sg.base;
    V *vp = VB ? vals + sg.base : nullptr;
    auto pos = [&](int j) { return w * 64 * IPT + j * 64 + lane; };
    auto valid = [&](int j) { return pos(j) < len; };
    const int32_t lim = (int32_t)len - (int32_t)(w * 64 * IPT);

    KB k[IPT];
    V v[IPT];
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
        k[j] = valid(j) ? ks[pos(j)] : KB(0);
        if constexpr (VB > 0) {
            if (valid(j)) v[j] = vs[pos(j)];
        }
    }
    auto clear_work = [&] {
        for (int i = tid; i < 4 * 256 * 12 / 16; i += kSegSmallThreads)
            ((uint4 *)s_work)[i] = make_uint4(0, 0, 0, 0);
    };
    static_assert(NB * 4 <= 4 * 256 * 12, "clear_work covers the bins");
    clear_work();

    // one stable LDS counting pass by dig() over the register-held keys:
    // in-wave ranks, the block's digit offsets, scatter to LDS, read back in
    // position order (a pass whose digit is the same for every key is skipped)
    auto lds_pass = [&](auto dig) {
        Ranks<IPT> r;
        for (int i = lane; i < 256; i += 64) s_cnt[w][i] = 0;
        block_barrier();
        // every thread read the previous pass's flag before the barrier above
        if (tid == 0) s_uniform = 0;
        rank_in_wave_by<IPT, false, kRankLdsMask>(k, r, dig, s_cnt[w], s_peer[w], lim);
        block_barrier();
        const uint32_t c0 = s_cnt[0][tid], c1 = s_cnt[1][tid], c2 = s_cnt[2][tid], c3 = s_cnt[3][tid];
        const uint32_t total = c0 + c1 + c2 + c3;
        if (total == len) s_uniform = 1;
        const uint32_t lstart = block_exclusive_sum256(total, s_wsum);
        s_cnt[0][tid] = lstart;
        s_cnt[1][tid] = lstart + c0;
        s_cnt[2][tid] = lstart + c0 + c1;
        s_cnt[3][tid] = lstart + c0 + c1 + c2;
        block_barrier();
        if (s_uniform) return;
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            if (valid(j)) {
                const uint32_t dst = s_cnt[w][dig(k[j])] + r[j];
                s_k[dst] = k[j];
                if constexpr (VB > 0) s_v[dst] = v[j];
            }
        }
        block_barrier();
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            if (valid(j)) {
                k[j] = s_k[pos(j)];
                if constexpr (VB > 0) v[j] = s_v[pos(j)];
            }
        }
    };

    // ---- range-adaptive passes
    {
        KB mn = (KB)~KB(0), mx = KB(0);
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            if (valid(j)) {
                const KB t = xf.key(k[j]);
                mn = t < mn ? t : mn;
                mx = t > mx ? t : mx;
            }
        }
        {  // wave reductions move 32-bit words: widen narrow keys
            using WK = std::conditional_t<(sizeof(KB) < 4), uint32_t, KB>;
            mn = (KB)wave_reduce((WK)mn, (WK)~WK(0), [](WK a, WK b) { return a < b ? a : b; });
            mx = (KB)wave_reduce((WK)mx, WK(0), [](WK a, WK b) { return a > b ? a : b; });
        }
        if (lane == 0) {
            s_mn[w] = mn;
            s_mx[w] = mx;
        }
        block_barrier();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            mn = s_mn[i] < mn ? s_mn[i] : mn;
            mx = s_mx[i] > mx ? s_mx[i] : mx;
        }
        if (mn == mx) {  // one key value: the input order is the sorted order
#pragma unroll
            for (int j = 0; j < IPT; ++j) {
                if (valid(j)) {
                    kp[pos(j)] = k[j];
                    if constexpr (VB > 0) vp[pos(j)] = v[j];
                }
            }
            return;
        }
        const uint32_t bitlen = 64u - (uint32_t)__builtin_clzll((unsigned long long)(KB)(mx - mn));
        // ---- bins
        if constexpr (xf_is_integer<XF>::value) {
            constexpr uint32_t NBITS = 31 - __builtin_clz(NB);
            const uint32_t sh = bitlen > NBITS ? bitlen - NBITS : 0u;
            auto bin = [&](KB x) { return (uint32_t)((KB)(xf.key(x) - mn) >> sh); };  // < NB
            uint32_t slot[IPT];
#pragma unroll
            for (int j = 0; j < IPT; ++j)
                if (valid(j)) slot[j] = atomicAdd(&s_bin[bin(k[j])], 1u);
            block_barrier();
            constexpr int BPT = NB / kSegSmallThreads;  // consecutive bins per thread
            uint32_t c[BPT], tot = 0, most = 0;
#pragma unroll
            for (int i = 0; i < BPT; ++i) c[i] = s_bin[tid * BPT + i];
#pragma unroll
            for (int i = 0; i < BPT; ++i) {
                tot += c[i];
                most = c[i] > most ? c[i] : most;
            }
            uint32_t start = block_exclusive_sum256(tot, s_wsum);
#pragma unroll
            for (int i = 0; i < BPT; ++i) {
                s_bin[tid * BPT + i] = start;
                start += c[i];
            }
            if (!block_barrier_or(most > kBinMax)) {
#pragma unroll
                for (int j = 0; j < IPT; ++j) {
                    if (!valid(j)) continue;
                    const uint32_t dst = s_bin[bin(k[j])] + slot[j];
                    s_k[dst] = k[j];
                    if constexpr (VB > 0) s_v[dst] = v[j];
                    s_idx[dst] = (uint16_t)pos(j);
                }
                block_barrier();
#pragma unroll
                for (int j = 0; j < IPT; ++j) {
                    const uint32_t i = pos(j);
                    if (i >= len) continue;
                    const KB x = s_k[i];
                    const KB tx = xf.key(x);
                    const uint32_t b = bin(x), b0 = s_bin[b], b1 = b + 1 < (uint32_t)NB ? s_bin[b + 1] : len;
                    uint32_t at = b0;
                    if (b1 - b0 > 1) {
                        const uint32_t ix = s_idx[i];
                        for (uint32_t e = b0; e < b1; ++e) {
                            const KB te = xf.key(s_k[e]);
                            at += (te < tx || (te == tx && s_idx[e] < ix)) ? 1u : 0u;
                        }
                    }
                    kp[at] = x;
                    if constexpr (VB > 0) vp[at] = s_v[i];
                }
                return;
            }
            clear_work();  // the keys are still in registers, in input order
        }
        // the leading 8 (spans up to 512 keys) or 16 bits of key - mn, as
        // one or two 8-bit passes, least significant first
        const uint32_t bits = len > 512 ? 16u : 8u;
        const uint32_t shift = bitlen > bits ? bitlen - bits : 0u;
        auto rel = [&](KB x) { return (KB)((KB)(xf.key(x) - mn) >> shift); };  // < 2^bits
        if (bits == 16) lds_pass([&](KB x) { return (uint32_t)rel(x) & 0xFFu; });
        lds_pass([&](KB x) { return (uint32_t)(rel(x) >> (bits - 8)); });
        // keys are now ordered by rel(); finish each run of equal rel() with a
        // stable insertion sort on the whole key (owner: the run's first slot)
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            if (valid(j)) {
                s_k[pos(j)] = k[j];
                if constexpr (VB > 0) s_v[pos(j)] = v[j];
            }
        }
        block_barrier();
        uint32_t rlen[IPT];
        bool big = false;
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            rlen[j] = 0;
            const uint32_t i = pos(j);
            if (!valid(j)) continue;
            const KB here = rel(s_k[i]);
            if (i > 0 && rel(s_k[i - 1]) == here) continue;  // not a run start
            uint32_t e = i + 1;
            while (e < len && e - i <= kBucketMax && rel(s_k[e]) == here) ++e;
            rlen[j] = e - i;
            big = big || rlen[j] > kBucketMax;
        }
        if (!block_barrier_or(big)) {
#pragma unroll
            for (int j = 0; j < IPT; ++j) {
                const uint32_t b0 = pos(j);
                for (uint32_t i = 1; i < rlen[j]; ++i) {
                    const KB key = s_k[b0 + i];
                    const KB tk = xf.key(key);
                    V val{};
                    if constexpr (VB > 0) val = s_v[b0 + i];
                    uint32_t q = i;
                    while (q > 0 && xf.key(s_k[b0 + q - 1]) > tk) {
                        s_k[b0 + q] = s_k[b0 + q - 1];
                        if constexpr (VB > 0) s_v[b0 + q] = s_v[b0 + q - 1];
                        --q;
                    }
                    s_k[b0 + q] = key;
                    if constexpr (VB > 0) s_v[b0 + q] = val;
                }
            }
            block_barrier();
#pragma unroll
            for (int j = 0; j < IPT; ++j) {
                if (valid(j)) {
                    kp[pos(j)] = s_k[pos(j)];
                    if constexpr (VB > 0) vp[pos(j)] = s_v[pos(j)];
                }
            }
            return;
        }
        // a run too long to finish by insertion (clustered keys): all LSD
        // passes follow.  The order so far is a stable sort by a monotone
        // function of the key, so equal keys are still in input order.
    }

    for (int p = 0; p < P; ++p) lds_pass([&](KB x) { return xf.digit(x, 8 * p); });
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
        if (valid(j)) {
            kp[pos(j)] = k[j];
            if constexpr (VB > 0) vp[pos(j)] = v[j];
        }
    }
}

// ------------------------------------------------- tiny float segments
// serial_insertion_sort_by_key (insertion_sort.hpp:106-133) on the native
// type, one thread per segment.
template <typename T, int VB>
__global__ void k_seg_insertion(T *keys, typename ValT<VB>::type *vals, const SegSpan *segs, uint32_t nsegs,
                                int descending)
{
    using V = typename ValT<VB>::type;
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsegs) return;
    T *kp = keys + segs[s].base;
    V *vp = VB ? vals + segs[s].base : nullptr;
    const uint32_t n = segs[s].len;
    for (uint32_t i = 1; i < n; ++i) {
        const T key = kp[i];
        V val{};
        if constexpr (VB > 0) val = vp[i];
        uint32_t q = i;
        while (q > 0 && (descending ? (key > kp[q - 1]) : (key < kp[q - 1]))) {
            kp[q] = kp[q - 1];
            if constexpr (VB > 0) vp[q] = vp[q - 1];
            q--;
        }
        kp[q] = key;
        if constexpr (VB > 0) vp[q] = val;
    }
}

// ------------------------------------------------------------ large path
// Route of a large segment, decided on the device from its histogram:
//   kRouteLsd: all P onesweep passes over the segment (any distribution);
//   kRouteMsd: one onesweep pass on the most significant digit into the
//     temporaries, which partitions the segment stably into its 256 digit
//     buckets; consecutive buckets are packed greedily into groups of at
//     most `cap` keys, and each group is sorted in LDS by the whole key and
//     written back (a group is a contiguous range of the sorted segment, so
//     sorting it by the whole key is exact, and stable).  Taken when every
//     bucket fits one group and the groups fit the segment's slots.
enum : uint32_t { kRouteLsd = 0, kRouteMsd = 1 };

// One block per histogram chunk (<= kSegChunk keys of one segment): the
// histograms of digits [p0, p0 + NP).  With route != nullptr only chunks of
// segments on the LSD route are counted (the others need just the top digit,
// NP = 1: 4 KB of LDS to clear and add up instead of 32 KB for 8-byte keys),
// and none if *any_lsd says that no segment takes it.
template <typename KB, int NP, typename XF>
__global__ __launch_bounds__(kHistThreads) void k_seg_histogram(const KB *__restrict__ keys,
                                                                const SegSpan *__restrict__ chunks, XF xf,
                                                                uint32_t *__restrict__ partial, uint32_t p0,
                                                                const uint32_t *__restrict__ route,
                                                                const uint32_t *__restrict__ any_lsd)
{
    constexpr int P = sizeof(KB);
    constexpr int NW = kHistThreads / 64;
    __shared__ uint32_t s_hist[NW][NP][256];
    if (route && !*any_lsd) return;
    const SegSpan c = chunks[blockIdx.x];
    if (route && route[c.idx] != kRouteLsd) return;
    for (int i = threadIdx.x; i < NW * NP * 256; i += kHistThreads) (&s_hist[0][0][0])[i] = 0;
    block_barrier();
    uint32_t(*h)[256] = s_hist[threadIdx.x >> 6];
    const KB *kc = keys + c.base;
    constexpr int U = 8;  // loads in flight per thread
    for (uint32_t i0 = threadIdx.x; i0 < c.len; i0 += kHistThreads * U) {
        KB kk[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = i0 + u * kHistThreads;
            kk[u] = i < c.len ? kc[i] : KB(0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (i0 + u * kHistThreads < c.len) {
                const KB k = (KB)(xf.key(kk[u]) >> (8 * p0));
#pragma unroll
                for (int p = 0; p < NP; ++p) atomicAdd(&h[p][(k >> (8 * p)) & 0xFF], 1u);
            }
        }
    }
    block_barrier();
    uint32_t *dst = partial + ((size_t)blockIdx.x * P + p0) * 256;
    for (uint32_t i = threadIdx.x; i < NP * 256; i += kHistThreads) {
        uint32_t t = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) t += (&s_hist[w][0][0])[i];
        dst[i] = t;
    }
}

// grid (large segments, passes p0 + blockIdx.y): digit d of segment s summed
// over its chunks [chunk_begin[s], chunk_begin[s+1]) and scanned into
// exclusive offsets; with route != nullptr, LSD-route segments only.  The
// first launch (route == nullptr) clears *any_lsd for the route kernel.
static __global__ __launch_bounds__(256) void k_seg_digit_offsets(const uint32_t *__restrict__ partial,
                                                           const uint32_t *__restrict__ chunk_begin, uint32_t passes,
                                                           uint32_t p0, uint32_t *__restrict__ seg_off,
                                                           const uint32_t *__restrict__ route, uint32_t *any_lsd)
{
    __shared__ uint32_t s_wsum[4];
    const uint32_t s = blockIdx.x, p = p0 + blockIdx.y, d = threadIdx.x;
    if (!route) {
        if (s == 0 && d == 0) *any_lsd = 0;
    } else if (!*any_lsd) {
        return;
    }
    if (route && route[s] != kRouteLsd) return;
    uint32_t c = 0;
    for (uint32_t b = chunk_begin[s]; b < chunk_begin[s + 1]; ++b) c += partial[((size_t)b * passes + p) * 256 + d];
    seg_off[((size_t)s * passes + p) * 256 + d] = block_exclusive_sum256(c, s_wsum);
}

template <typename KB, int VB, int IPT, typename XF>
__global__ __launch_bounds__(kSortThreads) __attribute__((amdgpu_waves_per_eu(onesweep_waves_per_eu<VB, IPT>())))
void k_onesweep_seg(const KB *__restrict__ kin, KB *__restrict__ kout,
                                                               const typename ValT<VB>::type *__restrict__ vin,
                                                               typename ValT<VB>::type *__restrict__ vout,
                                                               const SegTile *__restrict__ tiles, uint32_t shift,
                                                               uint32_t pass, uint32_t passes,
                                                               const uint32_t *__restrict__ seg_off, XF xf,
                                                               Ctrl *ctrl, uint64_t *__restrict__ status,
                                                               uint32_t back, uint32_t want,
                                                               const uint32_t *__restrict__ any_lsd)
{
    // no segment takes this route: out after one scalar load, which the
    // whole grid shares
    if (want == kRouteLsd && !*any_lsd) return;
    // the tile carries its segment's route (one load before a tile of the
    // other route exits)
    const SegTile t = tiles[blockIdx.x];
    if (t.route != want) return;
    const size_t b = t.base;
    onesweep_tile<KB, VB, IPT, kRankLdsMask, XF>(kin + b, kout + b, VB ? vin + b : vin, VB ? vout + b : vout, t.len,
                                             t.tile, shift, seg_off + ((size_t)t.seg * passes + pass) * 256, xf,
                                             ctrl, status + (size_t)(blockIdx.x - t.tile) * 256, back);
}

// The same pass on the quarter-wave digit-pass body (onesweep.hpp): 16-lane
// subs rank by OR-ed peer masks in bank-grouped count words, the tile is
// staged while its look-back completes.  Tile, look-back chain and offsets
// are the segment's, as above.
template <typename KB, int VB, int IPT, typename XF>
__global__ __launch_bounds__(kSortThreads) void k_qsweep_seg(KB *kin, KB *kout,
                                                             typename ValT<VB>::type *vin,
                                                             typename ValT<VB>::type *vout,
                                                             const SegTile *__restrict__ tiles, uint32_t shift,
                                                             uint32_t pass, uint32_t passes,
                                                             const uint32_t *__restrict__ seg_off, XF xf,
                                                             Ctrl *ctrl, uint64_t *__restrict__ status,
                                                             uint32_t back, uint32_t want,
                                                               const uint32_t *__restrict__ any_lsd)
{
    __shared__ QSweepLds<kSortThreads, IPT, KB, VB, 1> lds;
    if (want == kRouteLsd && !*any_lsd) return;  // as above
    const SegTile t = tiles[blockIdx.x];
    if (t.route != want) return;
    const uint32_t epoch = launch_epoch(ctrl, back);
    const size_t b = t.base;
    const uint32_t *goff = seg_off + ((size_t)t.seg * passes + pass) * 256;
    uint64_t *st = status + (size_t)(blockIdx.x - t.tile) * 256;
    if ((uint64_t)(t.tile + 1) * (kSortThreads * IPT) <= t.len)
        qsweep_body<kSortThreads, IPT, KB, VB, 1, 2, XF, true, 1>(lds, kin + b, kout + b, VB ? vin + b : vin,
                                                                VB ? vout + b : vout, t.len, t.tile, shift, goff, xf,
                                                                ctrl, st, epoch, PlainPass());
    else
        qsweep_body<kSortThreads, IPT, KB, VB, 1, 2, XF, false, 1>(lds, kin + b, kout + b, VB ? vin + b : vin,
                                                                 VB ? vout + b : vout, t.len, t.tile, shift, goff,
                                                                 xf, ctrl, st, epoch, PlainPass());
}

// One block (256 threads, thread = digit) per large segment.  The top-digit
// buckets are packed greedily into groups of at most `cap` elements: a
// group that starts at bucket b ends before next(b), the first bucket whose
// end lies more than cap past b's start (a binary search over the bucket
// starts), and the group starts are the chain 0, next(0), next(next(0)), ...
// That chain is marked in 8 rounds of pointer doubling (it has at most 256
// nodes), so no thread walks the buckets one by one (a serial walk per
// segment is bound by the CU's one scalar unit).  A group's slot is its
// start's rank among the marks.  All threads then clear the segment's unused
// group slots and tag its tiles with the route.
static __global__ __launch_bounds__(256) void k_seg_route(const SegSpan *__restrict__ large,
                                                   const uint32_t *__restrict__ seg_off, uint32_t passes,
                                                   const uint32_t *__restrict__ slot_begin, SegSpan *groups,
                                                   uint32_t *route, uint32_t *any_lsd, SegTile *tiles,
                                                   uint32_t tile_len, uint32_t cap, uint32_t enable)
{
    __shared__ uint32_t s_start[257];
    __shared__ uint32_t s_jump[2][257];
    __shared__ uint32_t s_mark[257];
    __shared__ uint32_t s_wave[4];
    const uint32_t s = blockIdx.x, d = threadIdx.x;
    const SegSpan sg = large[s];
    const uint32_t *off = seg_off + ((size_t)s * passes + passes - 1) * 256;
    s_start[d] = off[d];
    if (d == 0) {
        s_start[256] = sg.len;
        s_jump[0][256] = s_jump[1][256] = 256;
        s_mark[256] = 0;
    }
    block_barrier();
    const uint32_t sd = s_start[d];
    const int big = block_barrier_or(s_start[d + 1] - sd > cap);
    const uint32_t b0 = slot_begin[s], b1 = slot_begin[s + 1];
    // next(d): the first c > d with s_start[c + 1] - s_start[d] > cap, else 256
    uint32_t lo = d + 1, hi = 256;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s_start[mid + 1] - sd > cap) hi = mid;
        else lo = mid + 1;
    }
    const uint32_t nx = lo;
    s_jump[0][d] = nx;
    s_mark[d] = d == 0;
    block_barrier();
    // round t: every marked node marks its 2^t-th successor; jumps double
#pragma unroll 1
    for (int t = 0; t < 8; ++t) {
        const uint32_t j = s_jump[t & 1][d];
        if (s_mark[d]) s_mark[j] = 1;  // j = 256 is the sentinel slot
        s_jump[(t & 1) ^ 1][d] = s_jump[t & 1][j];
        block_barrier();
    }
    const bool m = s_mark[d] != 0;
    const uint64_t bal = ballot(m);
    const uint32_t w = d >> 6;
    if ((d & 63) == 0) s_wave[w] = popc64(bal);
    block_barrier();
    uint32_t before = 0, ngroups = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        before += (uint32_t)i < w ? s_wave[i] : 0u;
        ngroups += s_wave[i];
    }
    const bool msd = enable && !big && ngroups <= b1 - b0;
    const uint32_t rt = msd ? kRouteMsd : kRouteLsd;
    if (d == 0) {
        route[s] = rt;
        if (!msd) *any_lsd = 1;  // the same value from every such segment
    }
    if (msd && m) groups[b0 + before + mbcnt(bal)] = SegSpan{sg.base + sd, s_start[nx] - sd, 0};
    for (uint32_t i = (msd ? b0 + ngroups : b0) + d; i < b1; i += 256) groups[i] = SegSpan{0, 0, 0};
    const uint32_t nt = (uint32_t)(((uint64_t)sg.len + tile_len - 1) / tile_len);
    for (uint32_t i = d; i < nt; i += 256) tiles[sg.idx + i].route = rt;
}

// odd pass count (8-bit keys): copy the large segments back from the temporaries
template <typename KB, int VB>
__global__ void k_seg_copyback(KB *keys, const KB *ktmp, typename ValT<VB>::type *vals,
                               const typename ValT<VB>::type *vtmp, const SegSpan *segs, const uint32_t *route)
{
    if (route[blockIdx.x] != kRouteLsd) return;
    const SegSpan s = segs[blockIdx.x];
    for (uint32_t i = threadIdx.x; i < s.len; i += blockDim.x) {
        keys[s.base + i] = ktmp[s.base + i];
        if constexpr (VB > 0) vals[s.base + i] = vtmp[s.base + i];
    }
}

inline size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace bcmi

// A plan: host-side routing of the segments, uploaded once.
struct bcmi_segplan_s {
    int device = 0;
    int key_dtype = 0;
    size_t value_bytes = 0;
    int descending = 0;
    uint64_t total = 0;  // elements covered by the offsets
    int small_cls = 4;      // largest small class: capacity kSegSmallThreads << small_cls
    int msd = 1;            // large segments may take the MSD route
    int ipt_large = 0;      // keys per thread of a large segment's onesweep tile
    int qrank = 0;          // 1: the large passes rank by quarter-waves (k_qsweep_seg)
    uint32_t nslots = 0;     // group slots of the MSD route, over all large segments
    uint32_t nsmall[5] = {0, 0, 0, 0, 0};  // classes IPT 1, 2, 4, 8, 16
    uint32_t ninsert = 0;
    uint32_t nlarge = 0, ntiles = 0, nchunks = 0;
    // device memory (one allocation)
    void *mem = nullptr;
    bcmi::SegSpan *small[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
    bcmi::SegSpan *insert = nullptr;
    bcmi::SegSpan *large = nullptr;
    bcmi::SegSpan *chunks = nullptr;
    uint32_t *route = nullptr;       // per large segment: kRouteLsd / kRouteMsd (set on the device)
    uint32_t *any_lsd = nullptr;     // whether any segment's route is kRouteLsd (set on the device)
    uint32_t *slot_begin = nullptr;  // per large segment: first group slot (nlarge + 1 entries)
    bcmi::SegSpan *groups = nullptr; // MSD route groups (written on the device)
    uint32_t *chunk_begin = nullptr;
    bcmi::SegTile *tiles = nullptr;
    uint32_t *partial = nullptr;
    uint32_t *seg_off = nullptr;
    void *ktmp = nullptr;
    void *vtmp = nullptr;
    // whether the small segments, and the large ones' all-digits passes, are
    // sorted on the queue's side streams, concurrently with the top-digit
    // route (the three touch disjoint elements, tiles and status words):
    // forked from and joined back into the queue's stream, so a graph capture
    // records the branches
    bool fork_small = false, fork_lsd = false;
};

namespace bcmi {

enum : int { kSideSmall = 0, kSideLsd = 1 };  // bcmi_queue_s::side

// Keys per thread of the large segments' onesweep tiles (256 threads): 8,
// 12 or 16 by element width; for 8-byte keys or values the tuning cache
// (key "__bcmi_segsort", param "ipt") may choose 24 (twice the tile, half
// the tiles).
inline int large_ipt(int kb, size_t vb)
{
    size_t sb = (size_t)kb > vb ? (size_t)kb : vb;
    if (sb == 8 && tune_get("__bcmi_segsort", "ipt", 12) == 24) return 24;
    return sb >= 16 ? 8 : (sb >= 8 ? 12 : 16);
}

// The small classes (sorted in place in LDS) and the insertion-sorted
// segments, on stream ss.
template <typename KB, int VB, typename XF>
static int run_plan_small(bcmi_queue q, bcmi_segplan pl, KB *keys, typename ValT<VB>::type *vals, XF xf,
                          hipStream_t ss)
{
#define BCMI_SMALL(CLS, IPTV)                                                                                   \
    if constexpr ((int)(sizeof(KB) + VB) * kSegSmallThreads * IPTV <= kSegSmallLds) {                           \
        if (pl->nsmall[CLS])                                                                                    \
            BCMI_LAUNCH(q, "segsort_small",                                                                     \
                        hipLaunchKernelGGL((k_seg_small<KB, VB, IPTV, XF>), dim3(pl->nsmall[CLS]),                  \
                                           dim3(kSegSmallThreads), 0, ss, keys, vals, keys, vals,                 \
                                           pl->small[CLS], xf));                                                \
    }
    BCMI_SMALL(0, 1)
    BCMI_SMALL(1, 2)
    BCMI_SMALL(2, 4)
    BCMI_SMALL(3, 8)
    BCMI_SMALL(4, 16)
#undef BCMI_SMALL
    if (pl->ninsert) {
        const unsigned blocks = (pl->ninsert + 63) / 64;
        if (pl->key_dtype == BCMI_F32) {
            if constexpr (sizeof(KB) == 4)
                BCMI_LAUNCH(q, "segsort_insertion",
                            hipLaunchKernelGGL((k_seg_insertion<float, VB>), dim3(blocks), dim3(64), 0, ss,
                                               (float *)keys, vals, pl->insert, pl->ninsert, pl->descending));
        } else {
            if constexpr (sizeof(KB) == 8)
                BCMI_LAUNCH(q, "segsort_insertion",
                            hipLaunchKernelGGL((k_seg_insertion<double, VB>), dim3(blocks), dim3(64), 0, ss,
                                               (double *)keys, vals, pl->insert, pl->ninsert, pl->descending));
        }
    }
    return 0;
}

// Tiles from which the all-digits passes go to a side stream, beside the
// top-digit route.  Where a plan's segments take both routes the two overlap;
// where none takes this one, its launches do (grids that leave at once, at the
// pace at which a CU can place workgroups of 51 KB of LDS: 22 us a pass over
// 10,437 tiles).  Fork and join cost about 20 us, which a plan whose segments
// are alike gets nothing for, so its line lies where they are a percent or
// two; a plan with small segments too has lengths of all kinds, which take
// both routes, and forks from half as many tiles on.  us a run with the copies,
// one stream | two:
//   10 segments of 2^22,    10,240 tiles of uint32 keys below 100: 1449 1470
//   6 segments of 2^22,       4096 tiles of uint64 keys: 1841 1860
//   500 segments of 20,000,   2500 tiles of uint32 keys below 100: 327 349
//   65,536 of all lengths,  10,437 tiles of uint64 keys: 1267 1256, 13,718 of float: 2316 2121
//   30,000 of all lengths,    4800 tiles of uint64 keys:  604  589,   6300 of float: 1100 1034
//   16,000 of all lengths,    2480 tiles of uint64 keys:  342  333,   3225 of float:  714  701
//   10,000 of 300 and 300 of 30,000, 1500 tiles of uint64 keys: 237 231, 2400 of uint32: 163 171
// The other digits' histograms stay on the queue's stream: beside the
// top-digit groups their few blocks land on the CUs that those leave free,
// several on one (206 -> 405 us for 500 segments of 20,000 uint64 keys).
constexpr uint32_t kForkLsdTiles = 6400, kForkLsdTilesMixed = 3200;

// The large segments: top-digit route decision, MSD groups, LSD passes (on
// q->stream, or on the side stream lsd with the decision waited for).
template <typename KB, int VB, typename XF, int IPTL>
static int run_plan_large(bcmi_queue q, bcmi_segplan pl, KB *keys, typename ValT<VB>::type *vals, XF xf,
                          SideStream *lsd, bool *lsd_forked)
{
    using V = typename ValT<VB>::type;
    constexpr int P = sizeof(KB);
    if (pl->nlarge) {
        const hipStream_t ls = lsd ? lsd->stream : q->stream;
        // the top digit's histogram and offsets decide each segment's route
        // (MSD needs two digits or more); the other digits are counted only
        // for segments on the LSD route
        BCMI_LAUNCH(q, "segsort_histogram",
                    hipLaunchKernelGGL((k_seg_histogram<KB, 1, XF>), dim3(pl->nchunks), dim3(kHistThreads), 0,
                                       q->stream, keys, pl->chunks, xf, pl->partial, (uint32_t)(P - 1),
                                       (const uint32_t *)nullptr, (const uint32_t *)pl->any_lsd));
        BCMI_LAUNCH(q, "segsort_digit_offsets",
                    hipLaunchKernelGGL(k_seg_digit_offsets, dim3(pl->nlarge, 1), dim3(256), 0, q->stream, pl->partial,
                                       pl->chunk_begin, (uint32_t)P, (uint32_t)(P - 1), pl->seg_off,
                                       (const uint32_t *)nullptr, pl->any_lsd));
        BCMI_LAUNCH(q, "segsort_route",
                    hipLaunchKernelGGL(k_seg_route, dim3(pl->nlarge), dim3(256), 0, q->stream, pl->large, pl->seg_off,
                                       (uint32_t)P, pl->slot_begin, pl->groups, pl->route, pl->any_lsd, pl->tiles,
                                       (uint32_t)(kSortThreads * IPTL), (uint32_t)(kSegSmallThreads << pl->small_cls),
                                       (uint32_t)(P >= 2 && pl->msd)));
        // the status array and epochs before the fork: growing it waits for
        // the queue's stream
        uint64_t *status;
        BCMI_TRY(status_array(q, (size_t)pl->ntiles * 256, &status));
        Epochs ep;
        BCMI_TRY(begin_lookback(q, P + 1, &ep));
        if constexpr (P >= 2) {
            BCMI_LAUNCH(q, "segsort_histogram",
                        hipLaunchKernelGGL((k_seg_histogram<KB, P - 1, XF>), dim3(pl->nchunks), dim3(kHistThreads), 0,
                                           q->stream, keys, pl->chunks, xf, pl->partial, 0u,
                                           (const uint32_t *)pl->route, (const uint32_t *)pl->any_lsd));
            BCMI_LAUNCH(q, "segsort_digit_offsets",
                        hipLaunchKernelGGL(k_seg_digit_offsets, dim3(pl->nlarge, P - 1), dim3(256), 0, q->stream,
                                           pl->partial, pl->chunk_begin, (uint32_t)P, 0u, pl->seg_off,
                                           (const uint32_t *)pl->route, pl->any_lsd));
        }
        if (lsd) {
            BCMI_HIP(hipEventRecord(lsd->fork, q->stream));
            BCMI_HIP(hipStreamWaitEvent(ls, lsd->fork, 0));
            *lsd_forked = true;
        }
        // MSD route: top-digit partition into the temporaries ...
        // (param "qrank" = 1: the quarter-wave pass body)
#define BCMI_SEG_PASS(NAME, STREAM, KS, KD, VS, VD, SHIFT, PASS, BACK, WANT)                                            \
        do {                                                                                                    \
            if (pl->qrank)                                                                                      \
                BCMI_LAUNCH(q, NAME,                                                                            \
                            hipLaunchKernelGGL((k_qsweep_seg<KB, VB, IPTL, XF>), dim3(pl->ntiles),              \
                                               dim3(kSortThreads), 0, STREAM, KS, KD, VS, VD, pl->tiles,     \
                                               SHIFT, PASS, (uint32_t)P, pl->seg_off, xf, q->ctrl, status,      \
                                               BACK, WANT, (const uint32_t *)pl->any_lsd));                                                    \
            else                                                                                                \
                BCMI_LAUNCH(q, NAME,                                                                            \
                            hipLaunchKernelGGL((k_onesweep_seg<KB, VB, IPTL, XF>), dim3(pl->ntiles),            \
                                               dim3(kSortThreads), 0, STREAM, KS, KD, VS, VD, pl->tiles,     \
                                               SHIFT, PASS, (uint32_t)P, pl->seg_off, xf, q->ctrl, status,      \
                                               BACK, WANT, (const uint32_t *)pl->any_lsd));                                                    \
        } while (0)
        BCMI_SEG_PASS("segsort_onesweep_msd", q->stream, keys, (KB *)pl->ktmp, vals, (V *)pl->vtmp, (uint32_t)(8 * (P - 1)),
                      (uint32_t)(P - 1), ep.arg(0), (uint32_t)kRouteMsd);
        // ... then every group sorted in LDS from the temporaries back into place
#define BCMI_GROUPS(CLS, IPTV)                                                                                  \
    if constexpr ((int)(sizeof(KB) + VB) * kSegSmallThreads * IPTV <= kSegSmallLds) {                           \
        if (pl->small_cls == CLS && pl->nslots)                                                                 \
            BCMI_LAUNCH(q, "segsort_groups",                                                                    \
                        hipLaunchKernelGGL((k_seg_small<KB, VB, IPTV, XF>), dim3(pl->nslots), dim3(kSegSmallThreads), \
                                           0, q->stream, (const KB *)pl->ktmp, (const V *)pl->vtmp, keys, vals,   \
                                           pl->groups, xf));                                                    \
    }
        BCMI_GROUPS(0, 1)
        BCMI_GROUPS(1, 2)
        BCMI_GROUPS(2, 4)
        BCMI_GROUPS(3, 8)
        BCMI_GROUPS(4, 16)
#undef BCMI_GROUPS
        // LSD route: all P passes
        KB *ks = keys, *kd = (KB *)pl->ktmp;
        V *vs = vals, *vd = (V *)pl->vtmp;
        for (int p = 0; p < P; ++p) {
            BCMI_SEG_PASS("segsort_onesweep", ls, ks, kd, vs, vd, (uint32_t)(8 * p), (uint32_t)p, ep.arg((uint32_t)p + 1),
                          (uint32_t)kRouteLsd);
            std::swap(ks, kd);
            std::swap(vs, vd);
        }
#undef BCMI_SEG_PASS
        if (ks != keys)
            BCMI_LAUNCH(q, "segsort_copyback",
                        hipLaunchKernelGGL((k_seg_copyback<KB, VB>), dim3(pl->nlarge), dim3(256), 0, ls, keys,
                                           ks, vals, vs, pl->large, pl->route));
    }
    return 0;
}

template <typename KB, int VB, typename XF>
static int run_plan_xf(bcmi_queue q, bcmi_segplan pl, void *keys_, void *vals_, XF xf)
{
    using V = typename ValT<VB>::type;
    KB *keys = (KB *)keys_;
    V *vals = (V *)vals_;
    // the small segments go to a side stream when there is large work to
    // overlap them with (not while the queue profiles kernels: its per-kernel
    // times are taken on the queue's stream)
    SideStream *small = nullptr, *lsd = nullptr;
    if (pl->fork_small && !q->profile) BCMI_TRY(side_stream(q, kSideSmall, &small));
    if (pl->fork_lsd && !q->profile) BCMI_TRY(side_stream(q, kSideLsd, &lsd));
    if (small) {
        BCMI_HIP(hipEventRecord(small->fork, q->stream));
        BCMI_HIP(hipStreamWaitEvent(small->stream, small->fork, 0));
    }
    int st = run_plan_small<KB, VB, XF>(q, pl, keys, vals, xf, small ? small->stream : q->stream);
    bool lsd_forked = false;
    if (!st) {
        constexpr int SB = (int)sizeof(KB) > VB ? (int)sizeof(KB) : VB;
        constexpr int IPTL = SB >= 16 ? 8 : (SB >= 8 ? 12 : 16);
        // the tile size the plan's tables were built for
        bool ran = false;
        if constexpr (SB == 8) {
            if (pl->ipt_large == 24) {
                st = run_plan_large<KB, VB, XF, 24>(q, pl, keys, vals, xf, lsd, &lsd_forked);
                ran = true;
            }
        }
        if (!ran) st = run_plan_large<KB, VB, XF, IPTL>(q, pl, keys, vals, xf, lsd, &lsd_forked);
    }
    // the joins are recorded whatever happened, so that a capture is never
    // left with a branch outside the queue's stream
    auto join = [&](SideStream *side) {
        hipError_t e = hipEventRecord(side->join, side->stream);
        if (e == hipSuccess) e = hipStreamWaitEvent(q->stream, side->join, 0);
        if (e != hipSuccess && !st) st = hip_fail(e, "segmented sort: join", __FILE__, __LINE__);
    };
    if (small) join(small);
    if (lsd_forked) join(lsd);
    return st;
}

template <typename KB, int VB>
static int run_plan(bcmi_queue q, bcmi_segplan pl, void *keys, void *vals)
{
    const int kind = pl->key_dtype == BCMI_F32 || pl->key_dtype == BCMI_F64 ? 2
                   : (pl->key_dtype == BCMI_I8 || pl->key_dtype == BCMI_I16 || pl->key_dtype == BCMI_I32 ||
                      pl->key_dtype == BCMI_I64) ? 1 : 0;
    return with_key_xf<KB>(kind, pl->descending,
                           [&](auto xf) { return run_plan_xf<KB, VB>(q, pl, keys, vals, xf); });
}

template <typename KB>
inline int run_plan_vb(bcmi_queue q, bcmi_segplan pl, void *keys, void *vals)
{
    switch (vals ? pl->value_bytes : 0) {
    case 0: return run_plan<KB, 0>(q, pl, keys, nullptr);
    case 1: return run_plan<KB, 1>(q, pl, keys, vals);
    case 2: return run_plan<KB, 2>(q, pl, keys, vals);
    case 4: return run_plan<KB, 4>(q, pl, keys, vals);
    case 8: return run_plan<KB, 8>(q, pl, keys, vals);
    case 16: return run_plan<KB, 16>(q, pl, keys, vals);
    default: set_error("segmented sort: value size %zu unsupported", pl->value_bytes); return BCMI_INVALID_VALUE;
    }
}

#define BCMI_SEGPLAN_SIGNATURE(NAME) int NAME(bcmi_queue q, bcmi_segplan pl, void *keys, void *vals)
BCMI_SEGPLAN_SIGNATURE(segplan_run_u8);
BCMI_SEGPLAN_SIGNATURE(segplan_run_u16);
BCMI_SEGPLAN_SIGNATURE(segplan_run_u32);
BCMI_SEGPLAN_SIGNATURE(segplan_run_u64);

}  // namespace bcmi
