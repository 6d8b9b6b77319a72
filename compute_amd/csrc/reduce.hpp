// reduce.hpp -- the reduction policies and the block / final combine shared
// by reduce.hip (reduce, accumulate) and mapreduce.hip (transform_reduce,
// inner_product).
//
// A policy P says how one thread folds elements (State), what a block
// writes as its partial (Part, FP64 for compensated float sums) and how the
// one-block final kernel folds the partials in a fixed order, so results
// are deterministic.  add_prod(s, x, y) folds the product x * y; the
// compensated policies keep that product's rounding error exactly (fma).
#pragma once

#include "device.hpp"
#include "ops.hpp"

#include <cstring>
#include <limits>
#include <type_traits>

namespace bcmi {

constexpr int kRedThreads = 256;

// Exact policy: fold in the element type (integers; min/max; and the naive
// float tree used only for error comparison).
template <typename T, int OP>
struct PlainPolicy {
    using State = T;
    using Part = T;
    static BDEV State id() { return op_identity<T, OP>(); }
    static BDEV State add(State s, T x) { return apply_op<T, OP>(s, x); }
    static BDEV State add_prod(State s, T x, T y) { return add(s, apply_op<T, BCMI_MULTIPLIES>(x, y)); }
    static BDEV State merge(State a, State b) { return apply_op<T, OP>(a, b); }
    static BDEV Part part(State s) { return s; }
    static BDEV Part part_id() { return id(); }
    static BDEV Part part_merge(Part a, Part b) { return merge(a, b); }
    static BDEV T finish(Part p, bool has_init, T init) { return has_init ? apply_op<T, OP>(init, p) : p; }
    static BDEV double f64(Part p) { return (double)p; }
};

// Compensated float plus: TwoSum pairs in FP32, FP64 partials.
struct CompF32Policy {
    using State = cf32;
    using Part = double;
    static BDEV State id() { return cf32{0.f, 0.f}; }
    static BDEV State add(State s, float x) { return cf_add(s, x); }
    static BDEV State add_prod(State s, float x, float y)
    {
        float p = x * y;
        // p must stay the rounded product: fused into TwoSum's additions
        // (contraction) it would carry the rounding error a second time
        asm volatile("" : "+v"(p));
        State r = cf_add(s, p);
        r.c += __builtin_fmaf(x, y, -p);  // the product's exact rounding error
        return r;
    }
    static BDEV State merge(State a, State b) { return cf_merge(a, b); }
    static BDEV Part part(State s) { return cf_value(s); }
    static BDEV Part part_id() { return 0.0; }
    static BDEV Part part_merge(Part a, Part b) { return a + b; }
    static BDEV float finish(Part p, bool has_init, float init) { return (float)(has_init ? (double)init + p : p); }
    static BDEV double f64(Part p) { return p; }
};

// Compensated double plus: TwoSum in FP64.
struct cf64 {
    double s, c;
};
struct CompF64Policy {
    using State = cf64;
    using Part = cf64;
    static BDEV void ts(double a, double b, double &s, double &e)
    {
        s = a + b;
        double bp = s - a;
        e = (a - (s - bp)) + (b - bp);
    }
    static BDEV State id() { return cf64{0.0, 0.0}; }
    static BDEV State add(State a, double x)
    {
        double s, e;
        ts(a.s, x, s, e);
        return cf64{s, a.c + e};
    }
    static BDEV State merge(State a, State b)
    {
        double s, e;
        ts(a.s, b.s, s, e);
        return cf64{s, (a.c + b.c) + e};
    }
    static BDEV State add_prod(State s, double x, double y)
    {
        double p = x * y;
        asm volatile("" : "+v"(p));  // the rounded product, not contracted (see CompF32Policy)
        State r = add(s, p);
        r.c += __builtin_fma(x, y, -p);
        return r;
    }
    static BDEV Part part(State s) { return s; }
    static BDEV Part part_id() { return id(); }
    static BDEV Part part_merge(Part a, Part b) { return merge(a, b); }
    static BDEV double finish(Part p, bool has_init, double init)
    {
        if (has_init) p = add(p, init);
        return p.s + p.c;
    }
    static BDEV double f64(Part p) { return p.s + p.c; }
};

// 16-byte-chunk view of the input, aligned as its elements are (a
// buffer_iterator may start anywhere)
template <typename T>
struct chunk16 {
    static constexpr int N = 16 / sizeof(T);
    T v[N];
};

// DPP moves 4- or 8-byte values; 16-byte states (cf64) go through LDS.
template <typename S, typename P>
BDEV S block_combine(S v, S *s_buf)
{
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if constexpr (sizeof(S) == 4 || sizeof(S) == 8) {
        v = wave_reduce(v, P::id(), [](S a, S b) { return P::merge(a, b); });
        if (lane == 0) s_buf[w] = v;
        block_barrier();
        if (threadIdx.x == 0) {
            S acc = s_buf[0];
            for (int i = 1; i < kRedThreads / 64; ++i) acc = P::merge(acc, s_buf[i]);
            s_buf[0] = acc;
        }
        block_barrier();
        return s_buf[0];
    } else {
        s_buf[threadIdx.x] = v;
        block_barrier();
        for (int off = kRedThreads / 2; off > 0; off >>= 1) {
            if ((int)threadIdx.x < off) s_buf[threadIdx.x] = P::merge(s_buf[threadIdx.x], s_buf[threadIdx.x + off]);
            block_barrier();
        }
        return s_buf[0];
    }
}

// A block's partial as tagged status words (device.hpp): 32 bits of it each.
template <typename Pt>
struct PartBox {
    static constexpr int N = (int)(sizeof(Pt) + 3) / 4;
    static_assert(N <= kPartWords, "partial of at most kPartWords words");
    uint32_t w[N];
};

template <typename Pt>
BDEV void part_publish(uint64_t *status, uint32_t block, uint32_t epoch, Pt p)
{
    PartBox<Pt> b{};
    __builtin_memcpy(b.w, &p, sizeof(Pt));
    lb_publish(status, block, epoch, LB_A, b);
}

// A bounded wait, as a look-back's: every block but the last publishes without
// waiting, and the last is dispatched after the others of its XCD and runs
// beside those of the rest, so it ends.
template <typename Pt>
BDEV Pt part_wait(const uint64_t *status, uint32_t block, uint32_t epoch, Ctrl *ctrl)
{
    PartBox<Pt> b{};
    uint32_t spins = 0;
    while (lb_read(status, block, epoch, b) == LB_X)
        if (spin_expired(ctrl, spins)) break;
    Pt p;
    __builtin_memcpy(&p, b.w, sizeof(Pt));
    return p;
}

// Called by all threads of every block with the block's folded state.  The
// last block folds all blocks' partials in a fixed order (so the result is
// deterministic) and finishes the result.  The partials come through the
// tagged status words rather than through a second launch of one block: that
// kernel took 2.5 us behind a first one of 3.3 us at 65,537 floats, and the
// words carry their own arrival, so no fence or device-scope atomic is needed.
template <typename T, typename P>
BDEV void reduce_finish(typename P::State blk, T init, int has_init, T *out, double *out_f64, Ctrl *ctrl,
                        uint64_t *status, uint32_t epoch)
{
    using Pt = typename P::Part;
    const uint32_t last = gridDim.x - 1;
    Pt total = P::part(blk);
    if (blockIdx.x != last) {
        if (threadIdx.x == 0) part_publish<Pt>(status, blockIdx.x, epoch, total);
        return;
    }
    if (last > 0) {
        __shared__ Pt s_part[kRedThreads];
        Pt p = P::part_id();
        for (uint32_t i = threadIdx.x; i <= last; i += kRedThreads)
            p = P::part_merge(p, i == last ? total : part_wait<Pt>(status, i, epoch, ctrl));
        s_part[threadIdx.x] = p;
        block_barrier();
        for (int off = kRedThreads / 2; off > 0; off >>= 1) {
            if ((int)threadIdx.x < off)
                s_part[threadIdx.x] = P::part_merge(s_part[threadIdx.x], s_part[threadIdx.x + off]);
            block_barrier();
        }
        total = s_part[0];
    }
    if (threadIdx.x == 0) {
        *out = P::finish(total, has_init != 0, init);
        if (out_f64) *out_f64 = P::f64(total) + (has_init ? (double)init : 0.0);
    }
}

// Blocks of a streaming reduction over `chunks` 16-byte chunks: two chunks a
// thread (one load round trip) until the grid holds per_cu blocks per CU.
inline unsigned reduce_blocks(bcmi_queue q, size_t chunks, unsigned per_cu)
{
    const size_t want = (chunks + kRedThreads * 2 - 1) / (kRedThreads * 2);
    const size_t most = (size_t)q->cu_count * per_cu;
    return (unsigned)(want < 1 ? 1 : (want > most ? most : want));
}

}  // namespace bcmi
