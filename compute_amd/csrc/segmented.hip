// segmented.hip -- C-ABI entry points of the batched segmented sort: plans are
// built and destroyed here and run by the kernels of segmented.hpp.
#include "segmented.hpp"

using namespace bcmi;

extern "C" int bcmi_segmented_plan_create(bcmi_queue q, int key_dtype, size_t value_bytes,
                                          const uint64_t *host_offsets, size_t nseg, int descending,
                                          bcmi_segplan *plan)
{
    BCMI_TRY(use_queue(q));
    BCMI_CHECK(plan && (host_offsets || nseg == 0), BCMI_INVALID_VALUE, "segmented plan: null argument");
    BCMI_CHECK(dtype_valid(key_dtype), BCMI_INVALID_VALUE, "segmented plan: bad key dtype %d", key_dtype);
    BCMI_CHECK(value_bytes == 0 || value_bytes == 1 || value_bytes == 2 || value_bytes == 4 || value_bytes == 8 ||
                   value_bytes == 16,
               BCMI_INVALID_VALUE, "segmented plan: value size %zu unsupported", value_bytes);
    const int kb = dtype_size(key_dtype);
    const bool flt = key_dtype == BCMI_F32 || key_dtype == BCMI_F64;
    const int ipt_large = large_ipt(kb, value_bytes);
    const uint64_t tile = (uint64_t)kSortThreads * ipt_large;
    SegTables tb;
    std::string err;
    // tuning cache key "__bcmi_segsort": "small_max" caps the small classes
    // (segments above go to the large path and its MSD groups of the same
    // capacity), "msd" = 0 sends every large segment down the LSD passes
    const int small_max = (int)tune_get("__bcmi_segsort", "small_max", 4);
    const int st0 = build_seg_tables(host_offsets, nseg, (size_t)kb + value_bytes, flt, tile, tb, err, small_max);
    BCMI_CHECK(st0 == 0, st0, "%s", err.c_str());
    const int cmax = tb.small_cls;
    std::vector<SegSpan>(&small)[5] = tb.small;
    std::vector<SegSpan> &insert = tb.insert, &large = tb.large, &chunks = tb.chunks;
    std::vector<uint32_t> &chunk_begin = tb.chunk_begin, &slot_begin = tb.slot_begin;
    std::vector<SegTile> &tiles = tb.tiles;
    const uint64_t total = tb.total;
    bcmi_segplan pl = new bcmi_segplan_s();
    pl->device = q->device;
    pl->key_dtype = key_dtype;
    pl->value_bytes = value_bytes;
    pl->descending = descending ? 1 : 0;
    pl->msd = tune_get("__bcmi_segsort", "msd", 1) ? 1 : 0;
    pl->ipt_large = ipt_large;
    pl->qrank = tune_get("__bcmi_segsort", "qrank", 0) ? 1 : 0;
    pl->total = total;
    pl->nlarge = (uint32_t)large.size();
    pl->ntiles = (uint32_t)tiles.size();
    pl->nchunks = (uint32_t)chunks.size();
    pl->ninsert = (uint32_t)insert.size();
    // one allocation: tables, histogram partials, digit offsets, temporaries
    size_t off = 0, o_small[5], o_insert, o_large, o_chunks, o_cb, o_tiles, o_partial, o_segoff, o_k, o_v;
    for (int c = 0; c < 5; ++c) {
        pl->nsmall[c] = (uint32_t)small[c].size();
        o_small[c] = off;
        off += al256(small[c].size() * sizeof(SegSpan));
    }
    o_insert = off; off += al256(insert.size() * sizeof(SegSpan));
    o_large = off; off += al256(large.size() * sizeof(SegSpan));
    o_chunks = off; off += al256(chunks.size() * sizeof(SegSpan));
    o_cb = off; off += al256(chunk_begin.size() * sizeof(uint32_t));
    o_tiles = off; off += al256(tiles.size() * sizeof(SegTile));
    o_partial = off; off += al256(chunks.size() * (size_t)kb * 256 * 4);
    o_segoff = off; off += al256(large.size() * (size_t)kb * 256 * 4);
    const size_t o_route = off; off += al256((large.size() + 1) * sizeof(uint32_t));
    const size_t o_sb = off; off += al256(slot_begin.size() * sizeof(uint32_t));
    const size_t o_groups = off; off += al256((size_t)slot_begin.back() * sizeof(SegSpan));
    // temporaries cover the elements of large segments at their own offsets
    const uint64_t span = large.empty() ? 0 : (large.back().base + large.back().len);
    o_k = off; off += al256(span * (size_t)kb);
    o_v = off; off += al256(span * value_bytes);
    hipError_t e = hipMalloc(&pl->mem, off + 256);
    if (e != hipSuccess) {
        delete pl;
        return hip_fail(e, "segmented plan allocation", __FILE__, __LINE__);
    }
    char *m = (char *)pl->mem;
    for (int c = 0; c < 5; ++c) pl->small[c] = (SegSpan *)(m + o_small[c]);
    pl->insert = (SegSpan *)(m + o_insert);
    pl->large = (SegSpan *)(m + o_large);
    pl->chunks = (SegSpan *)(m + o_chunks);
    pl->chunk_begin = (uint32_t *)(m + o_cb);
    pl->tiles = (SegTile *)(m + o_tiles);
    pl->partial = (uint32_t *)(m + o_partial);
    pl->seg_off = (uint32_t *)(m + o_segoff);
    pl->route = (uint32_t *)(m + o_route);
    pl->any_lsd = pl->route + large.size();
    pl->slot_begin = (uint32_t *)(m + o_sb);
    pl->groups = (SegSpan *)(m + o_groups);
    pl->nslots = slot_begin.back();
    pl->small_cls = cmax;
    pl->ktmp = m + o_k;
    pl->vtmp = m + o_v;
    auto up = [&](void *dst, const void *src, size_t bytes) -> int {
        if (bytes) BCMI_HIP(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
        return 0;
    };
    int st = 0;
    for (int c = 0; c < 5 && !st; ++c) st = up(pl->small[c], small[c].data(), small[c].size() * sizeof(SegSpan));
    if (!st) st = up(pl->insert, insert.data(), insert.size() * sizeof(SegSpan));
    if (!st) st = up(pl->large, large.data(), large.size() * sizeof(SegSpan));
    if (!st) st = up(pl->chunks, chunks.data(), chunks.size() * sizeof(SegSpan));
    if (!st) st = up(pl->chunk_begin, chunk_begin.data(), chunk_begin.size() * sizeof(uint32_t));
    if (!st) st = up(pl->tiles, tiles.data(), tiles.size() * sizeof(SegTile));
    if (!st) st = up(pl->slot_begin, slot_begin.data(), slot_begin.size() * sizeof(uint32_t));
    if (st) {
        (void)hipFree(pl->mem);
        delete pl;
        return st;
    }
    // look-back words for the large tiles, so that running the plan allocates nothing
    uint64_t *status;
    if (pl->ntiles) {
        int s2 = status_array(q, (size_t)pl->ntiles * 256, &status);
        if (s2) {
            (void)hipFree(pl->mem);
            delete pl;
            return s2;
        }
    }
    // the queue's side streams, where there is something to run beside the
    // large segments' top-digit route
    for (int c = 0; c < 5; ++c) pl->fork_small = pl->fork_small || pl->nsmall[c] != 0;
    pl->fork_small = (pl->fork_small || pl->ninsert != 0) && pl->nlarge;
    // 1-byte keys have no top-digit route
    pl->fork_lsd = kb >= 2 && pl->ntiles >= (pl->fork_small ? kForkLsdTilesMixed : kForkLsdTiles);
    SideStream *side;
    int s3 = pl->fork_small ? side_stream(q, kSideSmall, &side) : 0;
    if (!s3 && pl->fork_lsd) s3 = side_stream(q, kSideLsd, &side);
    if (s3) {
        bcmi_segmented_plan_destroy(pl);
        return s3;
    }
    *plan = pl;
    return 0;
}

extern "C" int bcmi_segmented_plan_destroy(bcmi_segplan plan)
{
    if (!plan) return 0;
    (void)hipSetDevice(plan->device);
    if (plan->mem) BCMI_HIP(hipFree(plan->mem));
    delete plan;
    return 0;
}

extern "C" int bcmi_segmented_sort_plan(bcmi_queue q, bcmi_segplan plan, void *keys, void *values)
{
    BCMI_TRY(use_queue(q));
    BCMI_CHECK(plan, BCMI_INVALID_VALUE, "segmented sort: null plan");
    BCMI_CHECK(plan->device == q->device, BCMI_INVALID_COMMAND_QUEUE, "segmented sort: plan is for another device");
    if (plan->total == 0) return 0;
    BCMI_CHECK(keys, BCMI_INVALID_VALUE, "segmented sort: null keys");
    if (!values) values = nullptr;
    switch (dtype_size(plan->key_dtype)) {
    case 1: return segplan_run_u8(q, plan, keys, values);
    case 2: return segplan_run_u16(q, plan, keys, values);
    case 4: return segplan_run_u32(q, plan, keys, values);
    default: return segplan_run_u64(q, plan, keys, values);
    }
}

extern "C" int bcmi_segmented_sort(bcmi_queue q, int key_dtype, void *keys, void *values, size_t value_bytes,
                                   const uint64_t *host_offsets, size_t nseg, int descending)
{
    BCMI_TRY(use_queue(q));
    BCMI_CHECK(!q->capturing, BCMI_INVALID_OPERATION,
               "segmented sort: build a plan (bcmi_segmented_plan_create) before capturing a graph");
    bcmi_segplan plan = nullptr;
    BCMI_TRY(bcmi_segmented_plan_create(q, key_dtype, values ? value_bytes : 0, host_offsets, nseg, descending, &plan));
    int st = bcmi_segmented_sort_plan(q, plan, keys, values);
    hipError_t e = hipStreamSynchronize(q->stream);
    bcmi_segmented_plan_destroy(plan);
    if (st) return st;
    if (e != hipSuccess) return hip_fail(e, "segmented sort", __FILE__, __LINE__);
    return 0;
}
