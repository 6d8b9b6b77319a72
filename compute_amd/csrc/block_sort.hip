// block_sort.hip -- radix sort of a range that one workgroup holds in LDS.
//
// A sort of a few thousand keys through the multi-tile path is a histogram,
// an offsets kernel and one digit pass per key byte, each a launch of one or
// two workgroups whose time is the latency of a cold load, a chain of
// barriers and a store: 33 us for 3001 4-byte keys (5.0 + 2.0 + 4 x 6.1 us of
// kernels).  Here the keys are loaded once, every pass runs in LDS, and the
// result is stored once: one launch, 14.4 us with the copy of its input.  What
// bounds it is the chain of barriers and dependent LDS round trips of a pass,
// about 2.7 us at 4 keys per thread.
//
// The order is the stable order by the radix() key transform
// (radix_sort.hpp:98-129), as everywhere in the sort.  Keys are transformed
// when loaded, and the smallest one is subtracted, so that only the bytes the
// keys' range spans take a pass (none when all keys are equal).  8-byte keys
// spanning more than 32 bits are sorted by the top 24 bits of that range;
// each run of equal top bits (a rare pair for spread-out keys) is finished by
// insertion, and a run longer than kRunMax sends the range through all its
// byte passes instead.
#include "block_sort.hpp"

#include "radix.hpp"

namespace bcmi {

// radix() of a key with its form chosen at run time: it is applied once per
// key, so one kernel serves every key type of a width.
template <typename KB>
struct RtXf {
    KB cx;
    uint32_t neg, flt;
    BDEV KB key(KB x) const
    {
        constexpr int W = sizeof(KB) * 8;
        using SK = std::make_signed_t<KB>;
        const KB t = neg ? (KB)(KB(0) - x) : x;
        return (KB)(t ^ (flt ? (KB)((KB)((SK)x >> (W - 1)) | cx) : cx));
    }
    // the key a transformed value came from (descending floats excepted:
    // their transform maps two keys to one value)
    BDEV KB inverse(KB k) const
    {
        constexpr int W = sizeof(KB) * 8;
        const KB x = (KB)(k ^ (flt ? (k >> (W - 1) ? cx : (KB)~KB(0)) : cx));
        return neg ? (KB)(KB(0) - x) : x;
    }
};

constexpr uint32_t kRunMax = 8;

// LDS: the count words of a pass (one 32-bit [position:16 | peer mask:16]
// word per quarter-wave and digit, as in onesweep.hpp) share the staging
// buffer; ranking ends before the first staging write.
template <typename KB, int TH, int IPT, bool IDX>
struct BlockSortLds {
    static constexpr int NSUB = TH / 16, TILE = TH * IPT;
    static constexpr int WORDS = NSUB * 256 * 4, KEYS = TILE * (int)sizeof(KB);
    static constexpr int STAGE = KEYS + (IDX ? TILE * 2 : 0);
    alignas(16) unsigned char stage[STAGE > WORDS ? STAGE : WORDS];
    uint32_t wsum[TH / 64];
    KB mn[TH / 64], mx[TH / 64];
};

// vals[pos(j)] = vals[src[j]], every load before the first store.  Elements
// of B bytes, or the B-byte part at `part` of elements of PARTS such parts
// (16-byte elements move as two halves: whole, they take the registers of
// the 8-keys-per-thread kernel past its bound).
template <int B, int PARTS = 1, int IPT, typename Pos>
BDEV void permute_values(void *vals, const uint32_t (&src)[IPT], uint32_t n, Pos pos, uint32_t part = 0)
{
    using V = typename ValT<B>::type;
    V *p = (V *)vals + part;
    V v[IPT];
#pragma unroll
    for (int j = 0; j < IPT; ++j)
        if (pos(j) < n) v[j] = p[src[j] * PARTS];
    // every wave's loads have returned before any wave stores
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    block_barrier();
#pragma unroll
    for (int j = 0; j < IPT; ++j)
        if (pos(j) < n) p[pos(j) * PARTS] = v[j];
}

// TH threads x IPT keys.  Each 16-lane quarter-wave ("sub") owns 16 * IPT
// consecutive positions, slot j of lane l being position sub*16*IPT + 16j + l.
// Positions from n on are left out of every step (padding keys would all hit
// one count word: 20.6 against 14.5 us for 3001 keys).  IDX: every key carries
// its input position (16 bits) through the passes; the values (and the keys,
// where the transform cannot be undone) are gathered by it at the end.
template <typename KB, int TH, int IPT, bool IDX>
__global__ __launch_bounds__(TH) void k_block_sort(KB *keys, void *vals, uint32_t vb, uint32_t n, RtXf<KB> xf)
{
    using LDS = BlockSortLds<KB, TH, IPT, IDX>;
    constexpr int TILE = LDS::TILE, NW = TH / 64;
    static_assert(16 % NW == 0 && TILE <= 65536, "whole count rows per wave, 16-bit positions");
    using WK = std::conditional_t<(sizeof(KB) < 4), uint32_t, KB>;
    __shared__ LDS L;
    uint32_t *words = (uint32_t *)L.stage;
    KB *s_keys = (KB *)L.stage;
    uint16_t *s_idx = (uint16_t *)(L.stage + LDS::KEYS);
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6, ql = tid & 15;
    const uint32_t sub = (lane >> 4) * NW + w;  // position order: see the count words below
    auto pos = [&](int j) { return sub * 16 * IPT + (uint32_t)j * 16 + ql; };

    KB k[IPT];
    uint32_t idx[IDX ? IPT : 1];
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
        k[j] = pos(j) < n ? keys[pos(j)] : KB(0);
        if constexpr (IDX) idx[j] = pos(j);
    }
    WK mn = ~WK(0), mx = 0;
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
        if (pos(j) < n) {
            k[j] = xf.key(k[j]);
            mn = (WK)k[j] < mn ? (WK)k[j] : mn;
            mx = (WK)k[j] > mx ? (WK)k[j] : mx;
        }
    }
    mn = wave_reduce(mn, (WK)~WK(0), [](WK a, WK b) { return a < b ? a : b; });
    mx = wave_reduce(mx, WK(0), [](WK a, WK b) { return a > b ? a : b; });
    if (lane == 0) {
        L.mn[w] = (KB)mn;
        L.mx[w] = (KB)mx;
    }
    block_barrier();
    KB lo = L.mn[0], hi = L.mx[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) {
        lo = L.mn[i] < lo ? L.mn[i] : lo;
        hi = L.mx[i] > hi ? L.mx[i] : hi;
    }
    if (lo == hi) return;  // one key value: in order already
    const uint32_t bits = 64u - (uint32_t)__builtin_clzll((unsigned long long)(KB)(hi - lo));
#pragma unroll
    for (int j = 0; j < IPT; ++j) k[j] = (KB)(k[j] - lo);

    // Count words, bank-grouped: the 4 subs of a wave own 16 columns each of
    // the 64-word rows, a row holding 16 digits (a digit many keys share
    // costs one sub's lanes a conflict, not the wave's).  The scan reads them
    // row by row without conflicts: wave w takes rows [w * RPW, w * RPW +
    // RPW), lane l column l of each group g of 4 subs.  Position order of the
    // subs is column-major (quarter sw of wave g is sub sw * NG + g), so the
    // scan over a digit's subs is a thread's own sum over g and one over the
    // four columns.
    constexpr int NG = NW, RPW = 16 / NW;
    uint32_t *my = words + w * 1024 + (lane >> 4) * 16;
    const uint32_t qbit = 1u << ql, qlt = qbit - 1u;
    auto sum = [](uint32_t a, uint32_t b) { return a + b; };

    // one stable counting pass by the byte at `shift`: counts, a scan in
    // digit-major, sub-minor order, ranks (see onesweep.hpp), a scatter to
    // LDS and a read back in position order
    auto pass = [&](uint32_t shift) {
        auto word = [&](int j) -> uint32_t * {
            const uint32_t d = (uint32_t)(k[j] >> shift) & 0xFFu;
            return my + (d >> 4) * 64 + (d & 15);
        };
        block_barrier();  // the previous reads of the staging buffer are done
#pragma unroll
        for (int i = 0; i < 4; ++i) *(uint4 *)(words + w * 1024 + i * 256 + lane * 4) = make_uint4(0, 0, 0, 0);
        wave_lds_sync();
#pragma unroll
        for (int j = 0; j < IPT; ++j)
            if (pos(j) < n)
                __hip_atomic_fetch_add(word(j), 1u << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        block_barrier();
        uint32_t c[RPW][NG], tot[RPW], colpre[RPW], dpre[RPW];
        uint32_t run = 0;  // keys of this wave's rows so far
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            const uint32_t *row = words + (w * RPW + r) * 64 + lane;
            tot[r] = 0;
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                c[r][g] = row[g * 1024] >> 16;
                tot[r] += c[r][g];
            }
        }
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            // over the columns sw: lanes 16 apart
            uint32_t inc = tot[r];
            uint32_t up = __shfl_up(inc, 16);
            inc += lane >= 16 ? up : 0u;
            up = __shfl_up(inc, 32);
            inc += lane >= 32 ? up : 0u;
            colpre[r] = inc - tot[r];
            // the digit's total, then the digits before it in the row
            const uint32_t dt = __shfl(inc, 48 + ql);
            uint32_t di = dt;
            di = sum(dpp<0x111>(0u, di), di);
            di = sum(dpp<0x112>(0u, di), di);
            di = sum(dpp<0x114>(0u, di), di);
            di = sum(dpp<0x118>(0u, di), di);
            dpre[r] = run + di - dt;
            run += readlane(di, 15);
        }
        if (lane == 0) L.wsum[w] = run;
        block_barrier();
        uint32_t wpre = 0;
#pragma unroll
        for (int i = 0; i < NW; ++i) wpre += i < (int)w ? L.wsum[i] : 0u;
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            uint32_t *row = words + (w * RPW + r) * 64 + lane;
            uint32_t s0 = wpre + dpre[r] + colpre[r];
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                row[g * 1024] = s0 << 16;
                s0 += c[r][g];
            }
        }
        block_barrier();
        uint32_t at[IPT];
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            if (pos(j) >= n) continue;
            uint32_t *a = word(j);
            __hip_atomic_fetch_or(a, qbit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            const uint32_t wd = __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            at[j] = (wd >> 16) + __builtin_popcount(wd & qlt);
            __hip_atomic_store(a, ((wd >> 16) + __builtin_popcount(wd & 0xFFFFu)) << 16, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        block_barrier();
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            if (pos(j) >= n) continue;
            s_keys[at[j]] = k[j];
            if constexpr (IDX) s_idx[at[j]] = (uint16_t)idx[j];
        }
        block_barrier();
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            k[j] = s_keys[pos(j)];
            if constexpr (IDX) idx[j] = s_idx[pos(j)];
        }
    };

    bool done = false;
    if constexpr (sizeof(KB) == 8) {
        if (bits > 32 && !xf.flt) {
            const uint32_t sh = bits - 24;
#pragma unroll 1
            for (uint32_t p = 0; p < 24; p += 8) pass(sh + p);
            // the staging buffer still holds the keys in order: position i
            // starts a run when its top bits differ from position i - 1's
            uint32_t run[IPT];
            bool big = false;
#pragma unroll
            for (int j = 0; j < IPT; ++j) {
                run[j] = 0;
                const uint32_t i = pos(j);
                if (i >= n || (i > 0 && (s_keys[i - 1] >> sh) == (k[j] >> sh))) continue;
                uint32_t e = i + 1;
                while (e < n && e - i <= kRunMax && (s_keys[e] >> sh) == (k[j] >> sh)) ++e;
                run[j] = e - i;
                big = big || run[j] > kRunMax;
            }
            if (!block_barrier_or(big)) {
                // runs are disjoint: each is sorted in place by its first
                // position's thread
#pragma unroll
                for (int j = 0; j < IPT; ++j) {
                    const uint32_t b0 = pos(j);
                    for (uint32_t i = 1; i < run[j]; ++i) {
                        const KB x = s_keys[b0 + i];
                        uint16_t ix = 0;
                        if constexpr (IDX) ix = s_idx[b0 + i];
                        uint32_t q = i;
                        while (q > 0 && s_keys[b0 + q - 1] > x) {
                            s_keys[b0 + q] = s_keys[b0 + q - 1];
                            if constexpr (IDX) s_idx[b0 + q] = s_idx[b0 + q - 1];
                            --q;
                        }
                        s_keys[b0 + q] = x;
                        if constexpr (IDX) s_idx[b0 + q] = ix;
                    }
                }
                block_barrier();
#pragma unroll
                for (int j = 0; j < IPT; ++j) {
                    k[j] = s_keys[pos(j)];
                    if constexpr (IDX) idx[j] = s_idx[pos(j)];
                }
                done = true;
            }
            // otherwise every byte takes a pass: the order so far is a
            // stable one by a monotone function of the key, so equal keys
            // are still in input order
        }
    }
    if (!done) {
#pragma unroll 1
        for (uint32_t p = 0; p < bits; p += 8) pass(p);
    }

    if constexpr (IDX) {
        uint32_t src[IPT];
#pragma unroll
        for (int j = 0; j < IPT; ++j) src[j] = pos(j) < n ? idx[j] : 0u;
        switch (vb) {
        case 1: permute_values<1>(vals, src, n, pos); break;
        case 2: permute_values<2>(vals, src, n, pos); break;
        case 4: permute_values<4>(vals, src, n, pos); break;
        case 8: permute_values<8>(vals, src, n, pos); break;
        case 16:
#pragma unroll 1
            for (uint32_t h = 0; h < 2; ++h) permute_values<8, 2>(vals, src, n, pos, h);
            break;
        default: break;
        }
        if (xf.flt && xf.neg) {
            permute_values<(int)sizeof(KB)>(keys, src, n, pos);
            return;
        }
    }
#pragma unroll
    for (int j = 0; j < IPT; ++j)
        if (pos(j) < n) keys[pos(j)] = xf.inverse((KB)(k[j] + lo));
}

template <typename KB, bool IDX>
static int launch_block_sort(bcmi_queue q, KB *keys, void *vals, uint32_t vb, uint32_t n, const RtXf<KB> &xf)
{
#define BCMI_BLOCK(TH, IPT)                                                                                        \
    if (n <= TH * IPT) {                                                                                           \
        BCMI_LAUNCH(q, "radix_block",                                                                              \
                    hipLaunchKernelGGL((k_block_sort<KB, TH, IPT, IDX>), dim3(1), dim3(TH), 0, q->stream, keys,    \
                                       vals, vb, n, xf));                                                          \
        return 0;                                                                                                  \
    }
    // more threads with few keys each rather than the reverse: a pass is a
    // chain of IPT dependent LDS round trips between its barriers
    BCMI_BLOCK(256, 4)
    BCMI_BLOCK(512, 4)
    BCMI_BLOCK(1024, 4)
    BCMI_BLOCK(1024, 8)
    if constexpr (sizeof(KB) <= 4 && !IDX) { BCMI_BLOCK(1024, 16) }
#undef BCMI_BLOCK
    set_error("sort: %u keys do not fit one workgroup", n);
    return BCMI_INVALID_VALUE;
}

template <typename KB>
static int block_sort_keys(bcmi_queue q, void *keys, void *vals, size_t vb, uint32_t n, int kind, int desc)
{
    const KB sgn = (KB)((KB)1 << (sizeof(KB) * 8 - 1));
    RtXf<KB> xf{};
    xf.flt = kind == 2;
    xf.neg = kind != 0 && desc;
    xf.cx = kind != 0 ? sgn : (desc ? (KB)~KB(0) : KB(0));
    if (vals || (xf.flt && xf.neg))
        return launch_block_sort<KB, true>(q, (KB *)keys, vals, vals ? (uint32_t)vb : 0u, n, xf);
    return launch_block_sort<KB, false>(q, (KB *)keys, nullptr, 0u, n, xf);
}

int block_sort(bcmi_queue q, size_t key_bytes, void *keys, void *vals, size_t vb, uint32_t n, int kind, int desc)
{
    if (vb == 0) vals = nullptr;
    BCMI_CHECK(!vals || vb == 1 || vb == 2 || vb == 4 || vb == 8 || vb == 16, BCMI_INVALID_VALUE,
               "sort: value size %zu unsupported (1, 2, 4, 8 or 16 bytes)", vb);
    switch (key_bytes) {
    case 1: return block_sort_keys<uint8_t>(q, keys, vals, vb, n, kind, desc);
    case 2: return block_sort_keys<uint16_t>(q, keys, vals, vb, n, kind, desc);
    case 4: return block_sort_keys<uint32_t>(q, keys, vals, vb, n, kind, desc);
    default: return block_sort_keys<uint64_t>(q, keys, vals, vb, n, kind, desc);
    }
}

}  // namespace bcmi
