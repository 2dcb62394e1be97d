// Device garbage collection: HashDAG::remove_stale_nodes(maxLevel) (hash_dag.h:407-547).
//
//   mark     level by level from the root: every child pointer of a live node sets its bit in
//            a bitmap over the virtual address space; the first setter appends the child to
//            the next level's frontier (the reference's per-level unordered_sets)
//   rebuild  levels maxLevel .. 0, two launches each: gather every live node with its children
//            remapped through the old -> new map of the level below and hang it into its
//            bucket's list; then lay every bucket out anew, the full node first
//            (ADD_FULL_NODES_FIRST), its list after it by the append rule, record old -> new
//
// Pages stay mapped (poolTop never shrinks), as in the reference. The result is canonically
// identical to the DAG before GC; node order within a bucket is the order of its list.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "hd_ctx.h"
#include "hd_table_dev.h"

namespace hd {
namespace {

constexpr uint32_t kGcGrid = 2048;  // most blocks of a launch over a level's nodes (they stride)
constexpr uint32_t GC_ERR_CAP = 1, GC_ERR_BUCKET = 2, GC_ERR_POOL = 4, GC_ERR_MAP = 8;

__global__ void k_gc_fill(uint32_t* p, uint64_t n, uint32_t v) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) p[i] = v;
}

// words used per level (sum of the level's bucket sizes): blockIdx.y is the level
__global__ __launch_bounds__(256) void k_gc_level_used(Geom g, const uint32_t* __restrict__ bucket_sizes,
                                                       unsigned long long* used) {
    const uint32_t l = blockIdx.y;
    const uint32_t nb = g.buckets_per_level(l);
    const uint32_t* __restrict__ bs = bucket_sizes + g.bucket_global(l, 0);
    unsigned long long sum = 0;
    for (uint32_t b = blockIdx.x * blockDim.x + threadIdx.x; b < nb; b += gridDim.x * blockDim.x) sum += bs[b];
#pragma unroll
    for (uint32_t off = 32; off; off >>= 1) sum += __shfl_down(sum, off, 64);
    if ((threadIdx.x & 63u) == 0 && sum) atomicAdd(&used[l], sum);
}

// the report of a collection: one block of words in device memory, read back once at its end
// (error flags, bucket of each level's full node, live nodes per level, words used per level, the
// kept roots)
constexpr uint32_t kRepFull = 64, kRepCounts = 128, kRepUsed = 192, kRepRoots = 320;

// level 0 frontier = the (distinct) roots kept alive
__global__ void k_gc_seed(uint32_t* frontier0, uint32_t* report, uint32_t n_roots) {
    if (blockIdx.x == 0) {
        for (uint32_t i = threadIdx.x; i < kRepRoots; i += blockDim.x) report[i] = i == kRepCounts ? n_roots : 0u;
    }
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n_roots; i += gridDim.x * blockDim.x)
        frontier0[i] = report[kRepRoots + i];
}

// A node's 9 words in registers (words past its length belong to its neighbours, or to the pad
// behind the last bucket): three loads in place of nine.
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void load_node(const uint32_t* __restrict__ vpool, uint32_t va, uint32_t w[9]) {
    const u32x4_a4 a = *reinterpret_cast<const u32x4_a4*>(vpool + va);
    const u32x4_a4 b = *reinterpret_cast<const u32x4_a4*>(vpool + va + 4);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        w[k] = a[k];
        w[4 + k] = b[k];
    }
    w[8] = vpool[va + 8];
}

// mark children of the live nodes of `level` (an interior level): one lane per node, its
// children's pointers, bitmap words and atomics issued together; a block appends the children it
// marked first with one atomic (in node order, child order within a node). Bound by latency and by
// the atomics, which leave the XCD. A word is read from the CU's own cache first: a bit seen there
// is set for good, and the leaves that a terrain's columns share are mostly seen there; the rest
// is asked for by atomics, all of a node's in flight before the first answer is looked at. The
// levels of a terrain 8192 wide took 830 us with a read beyond the XCD per child and one atomic
// at a time, and take 680 us.
__global__ __launch_bounds__(256) void k_gc_mark(const uint32_t* __restrict__ vpool, uint32_t* bitmap,
                                                 const uint32_t* __restrict__ frontier, uint32_t* __restrict__ next,
                                                 uint32_t* counts, uint32_t level, uint32_t capCur, uint32_t cap,
                                                 uint64_t numVirtual, uint32_t* errors) {
    __shared__ uint32_t sTot[256 / 64 + 1];
    const uint32_t n = min(counts[level], capCur);
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const uint32_t stride = gridDim.x * blockDim.x;
    // block-uniform loop: the next frontier is appended with one atomic per block
    for (uint32_t b0 = blockIdx.x * blockDim.x; b0 < n; b0 += stride) {
        const uint32_t i = b0 + threadIdx.x;
        uint32_t node[9], nk = 0, firstBits = 0;
        if (i < n) {
            load_node(vpool, frontier[i], node);
            nk = __popc(node[0] & 0xFFu);
            uint32_t ask = 0;  // children whose bit is not seen set
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {
                if (k >= nk) continue;
                if (node[1 + k] < numVirtual) ask |= 1u << k;
                else atomicOr(errors, GC_ERR_MAP);  // not an address of this table
            }
            uint32_t w[8];
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k)
                w[k] = (ask >> k) & 1u ? __hip_atomic_load(&bitmap[node[1 + k] >> 5], __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_WORKGROUP)
                                       : 0u;
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k)
                if ((w[k] >> (node[1 + k] & 31u)) & 1u) ask &= ~(1u << k);
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k)
                w[k] = (ask >> k) & 1u ? atomicOr(&bitmap[node[1 + k] >> 5], 1u << (node[1 + k] & 31u)) : ~0u;
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k)
                if (!((w[k] >> (node[1 + k] & 31u)) & 1u)) firstBits |= 1u << k;
        }
        // block scan of the marked counts, one atomic for the block
        const uint32_t cnt = __popc(firstBits);
        uint32_t incl = cnt;
#pragma unroll
        for (uint32_t off = 1; off < 64; off <<= 1) {
            const uint32_t t = __shfl_up(incl, off, 64);
            if (lane >= off) incl += t;
        }
        if (lane == 63) sTot[wv] = incl;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t tot = 0;
            for (uint32_t w = 0; w < nw; ++w) {
                const uint32_t x = sTot[w];
                sTot[w] = tot;
                tot += x;
            }
            sTot[nw] = tot ? atomicAdd(&counts[level + 1], tot) : 0u;
        }
        __syncthreads();
        uint32_t base = sTot[nw] + sTot[wv] + incl - cnt;
        __syncthreads();  // sTot is rewritten by the next iteration
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
            if (!((firstBits >> k) & 1u)) continue;
            if (base >= cap) atomicOr(errors, GC_ERR_CAP);
            else next[base] = node[1 + k];
            ++base;
        }
    }
}

// hash_words over words held in registers (no indexed access to them)
__device__ __forceinline__ uint32_t hash_node(const uint32_t w[9], uint32_t n) {
    uint32_t h = 0;
#pragma unroll
    for (uint32_t i = 0; i < 9; ++i) {
        if (i >= n) break;
        uint32_t k = w[i] * 0xcc9e2d51u;
        k = (k << 15) | (k >> 17);
        k *= 0x1b873593u;
        h ^= k;
        h = (h << 13) | (h >> 19);
        h = h * 5u + 0xe6546b64u;
    }
    return fmix32(h ^ n);
}

// the words of a level's full node (its children: the full node of the level below); its length
__device__ __forceinline__ uint32_t full_words(const Geom& g, uint32_t level, const uint32_t* full_nodes, uint32_t w[9]) {
    if (level == g.leaf_level()) {
        w[0] = w[1] = 0xFFFFFFFFu;
        return 2;
    }
    const uint32_t count = level < g.color_tree_levels ? 0u : (1u << (3 * (g.levels - level)));
    w[0] = (count << 8) | 0xFFu;
    for (uint32_t c = 0; c < 8; ++c) w[1 + c] = full_nodes[level + 1];
    return 9;
}

// A live node on its way to its new place: 48 bytes, so that it moves in three aligned accesses
// and a walk along a bucket's list reads one of them per node.
struct alignas(16) GcRow {
    uint32_t w[9];
    uint32_t next;  // the next row of the bucket's list, plus one; 0 ends it
    uint32_t va;    // the node's old address
    uint32_t len;
};

// Gather the live nodes of `level` with their children's new addresses (the forwarding array of
// the level below) into rows, each hung into the list of the bucket it belongs to: the exchange
// that takes the list's head is the only atomic of a node, and its answer is the row's `next`. A
// rank per node by an atomic add, a scan of the buckets' counts in three launches and a pass that
// put the lengths in order took nine launches more per level (11 of 3 to 5 us each where a level
// is small) and 200 us at the largest levels of a terrain 8192 wide.
__global__ __launch_bounds__(256) void k_gc_gather(Geom g, const uint32_t* __restrict__ vpool,
                                                   const uint32_t* __restrict__ frontier, uint32_t* report,
                                                   uint32_t level, uint32_t maxLevel, uint32_t cap,
                                                   const uint32_t* __restrict__ fwd, const uint32_t* full_nodes,
                                                   GcRow* __restrict__ rows, uint32_t* head) {
    const uint32_t n = min(report[kRepCounts + level], cap);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        uint32_t w[9];
        const uint32_t len = full_words(g, level, full_nodes, w);
        report[kRepFull + level] = g.bucket_from_hash(level, len == 2 ? hash_leaf(~0ull) : hash_node(w, len));
    }
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        GcRow r;
        r.va = frontier[i];
        uint32_t hash;
        if (level == g.leaf_level()) {
#pragma unroll
            for (uint32_t k = 0; k < 9; ++k) r.w[k] = k < 2 ? vpool[r.va + k] : 0u;
            r.len = 2;
            hash = hash_leaf((uint64_t)r.w[0] | ((uint64_t)r.w[1] << 32));
        } else {
            load_node(vpool, r.va, r.w);
            r.len = __popc(r.w[0] & 0xFFu) + 1;
            if (level != maxLevel) {
#pragma unroll
                for (uint32_t k = 1; k < 9; ++k)
                    if (k < r.len) r.w[k] = fwd[r.w[k]];
            }
            hash = hash_node(r.w, r.len);
        }
        r.next = atomicExch(&head[g.bucket_global(level, g.bucket_from_hash(level, hash))], i + 1);
        rows[i] = r;
    }
}

// A block lays out kPlaceBuckets consecutive buckets of a level: a lane per bucket starts it with
// the level's full node where that belongs to it, then walks its list and gives each node its place
// by the append rule of the table (a node that does not fit in the rest of its page starts the
// next page), mapping the pages it starts; a node that no longer fits sets the error. This is what
// appending the nodes one at a time in list order gives, without a compare-and-swap loop on the
// bucket's size. The nodes and places go through LDS to other lanes of the block, which copy them
// and record old -> new. 64 buckets a block: at 65536 buckets a level, 1024 blocks, so that the
// copies (bound by the latency of their scattered accesses) have 16 wavefronts a CU.
//
// kAlone: the walking wavefront goes to the end of its lists, copying what the LDS list has no room
// for itself (the rows are in its cache then), and the block copies the LDS list after it. Otherwise
// the walk stops every kPlaceRound nodes and the other wavefronts copy a round while the next is
// walked: the walk is a chain of loads, and with few blocks nothing but the block's own wavefronts
// hides it. The line lies at four blocks a CU: 12.2 M words a level in 65536 buckets take 188 us
// alone and 209 us in rounds; 4096 buckets of 366 nodes take 2.55 ms a collection in rounds and
// 3.73 ms alone.
constexpr uint32_t kPlaceBuckets = 64, kPlaceRound = 32, kPlaceAlone = 1024;
constexpr uint32_t kPlaceFull = 1024;  // blocks from which the walking wavefronts fill the chip
static_assert(kPlaceBuckets == 64, "one wavefront walks");
__device__ __forceinline__ void move_row(const GcRow* __restrict__ rows, uint32_t i, uint32_t va, uint32_t* vpool,
                                         uint32_t* fwd) {
    const GcRow r = rows[i];
#pragma unroll
    for (uint32_t k = 0; k < 9; ++k)
        if (k < r.len) vpool[va + k] = r.w[k];
    fwd[r.va] = va;
}
// barrier for LDS alone: the copies' stores stay in flight
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
template <bool kAlone>
__global__ __launch_bounds__(256) void k_gc_place(TableRef T, uint32_t level, const uint32_t* report,
                                                  uint32_t* full_nodes, const GcRow* __restrict__ rows,
                                                  const uint32_t* __restrict__ head, uint32_t* fwd, uint32_t* errors) {
    constexpr uint32_t kRoom = kAlone ? kPlaceAlone : kPlaceBuckets * kPlaceRound;
    __shared__ uint2 list[kAlone ? 1 : 2][kRoom];
    __shared__ uint32_t listed[2], more[2];
    const Geom& g = T.g;
    const uint32_t nb = g.buckets_per_level(level), ps = g.page_size, capB = g.bucket_size(level);
    const uint32_t b = blockIdx.x * kPlaceBuckets + threadIdx.x;
    const bool mine = threadIdx.x < kPlaceBuckets && b < nb;
    const uint32_t bg = g.bucket_global(level, mine ? b : 0u);
    uint32_t cur = 0, it = mine ? head[bg] : 0u;
    if (mine && b == report[kRepFull + level]) {
        uint32_t w[9];
        const uint32_t len = full_words(g, level, full_nodes, w);
        const uint32_t va = g.make_ptr(level, b, 0);
        if (len > capB) {
            atomicOr(errors, GC_ERR_BUCKET);
        } else {
            cur = len;
            if (!table_map_page(T, va / ps)) {
                atomicOr(errors, GC_ERR_POOL);
            } else {
                for (uint32_t k = 0; k < len; ++k) T.vpool[va + k] = w[k];
                full_nodes[level] = va;
            }
        }
    }
    // every thread leaves at the same round: `more` is read between two barriers
    const uint64_t below = (1ull << (threadIdx.x & 63u)) - 1ull;
    for (uint32_t round = 0;; ++round) {
        const uint32_t h = round & 1u;
        if (threadIdx.x < kPlaceBuckets) {
            uint32_t n = 0;
            for (uint32_t k = 0; (kAlone || k < kPlaceRound) && __ballot(it != 0); ++k) {
                const uint32_t row = it - 1;
                uint32_t va = 0;
                bool placed = false;
                if (it) {
                    const uint32_t len = rows[row].len, after = rows[row].next;
                    const uint32_t left = ps - cur % ps;
                    const uint32_t start = (left != ps && left < len) ? cur + left : cur;
                    if (start + len > capB) {
                        atomicOr(errors, GC_ERR_BUCKET);
                        it = 0;
                    } else {
                        cur = start + len;
                        va = g.make_ptr(level, b, start);
                        placed = start % ps != 0 || table_map_page(T, va / ps);
                        if (!placed) atomicOr(errors, GC_ERR_POOL);
                        it = after;
                    }
                }
                const uint64_t m = __ballot(placed);
                if (placed) {
                    const uint32_t at = n + (uint32_t)__popcll(m & below);
                    if (!kAlone || at < kRoom) list[h][at] = make_uint2(row, va);
                    else move_row(rows, row, va, T.vpool, fwd);
                }
                n += (uint32_t)__popcll(m);
                if (kAlone) n = min(n, kRoom);
            }
            const uint64_t open = __ballot(it != 0);
            if (threadIdx.x == 0) {
                listed[h] = n;
                more[h] = open != 0;
            }
        } else if (round) {
            const uint32_t n = listed[h ^ 1u];
            for (uint32_t q = threadIdx.x - kPlaceBuckets; q < n; q += blockDim.x - kPlaceBuckets)
                move_row(rows, list[h ^ 1u][q].x, list[h ^ 1u][q].y, T.vpool, fwd);
        }
        lds_barrier();
        if (more[h]) continue;
        const uint32_t n = listed[h];
        for (uint32_t q = threadIdx.x; q < n; q += blockDim.x) move_row(rows, list[h][q].x, list[h][q].y, T.vpool, fwd);
        break;
    }
    if (mine) T.bucket_sizes[bg] = cur;
}

// every kept root -> its address after GC
__global__ void k_gc_roots(const uint32_t* __restrict__ fwd, uint32_t* roots, uint32_t n_roots, uint32_t* errors) {
    if (*errors) return;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n_roots; i += gridDim.x * blockDim.x)
        roots[i] = fwd[roots[i]];
}

}  // namespace
}  // namespace hd

using namespace hd;

// Roots kept alive by a GC: the current root, the caller's extra roots and (keep_undo) the
// roots of every undo / redo frame, each once.
static std::vector<uint32_t> gc_root_set(const hd_ctx* ctx, const uint32_t* extra, uint32_t n_extra, bool keep_undo) {
    std::vector<uint32_t> r{ctx->root};
    for (uint32_t i = 0; i < n_extra; ++i) r.push_back(extra[i]);
    if (keep_undo)
        for (const auto* frames : {&ctx->undo, &ctx->redo})
            for (const UndoFrame& f : *frames) {
                r.push_back(f.prev_root);
                r.push_back(f.new_root);
            }
    std::sort(r.begin(), r.end());
    r.erase(std::unique(r.begin(), r.end()), r.end());
    return r;
}

static uint32_t remap(const std::vector<uint32_t>& from, const std::vector<uint32_t>& to, uint32_t v) {
    return to[std::lower_bound(from.begin(), from.end(), v) - from.begin()];
}

// GC scratch slots (fixed indices; frontier l at kSlotFrontier + l)
enum : uint32_t { kSlotBitmap, kSlotReport, kSlotRows, kSlotFwd, kSlotUsed, kSlotFrontier };

// slot k of the context's GC scratch with at least `bytes` (grown by a quarter beyond the
// request, so tables that grow between collections reallocate rarely)
static hipError_t gc_slot(hd_ctx* ctx, uint32_t k, uint64_t bytes, void** p) {
    if (ctx->gc_slots.size() <= k) ctx->gc_slots.resize(k + 1, {nullptr, 0});
    auto& sl = ctx->gc_slots[k];
    if (sl.second < bytes) {
        if (sl.first) {
            const hipError_t e = hipFree(sl.first);
            sl = {nullptr, 0};
            if (e != hipSuccess) return e;
        }
        const uint64_t want = std::max<uint64_t>(bytes + bytes / 4, 256);
        void* q = nullptr;
        const hipError_t e = dev_malloc(ctx, &q, want);
        if (e != hipSuccess) return e;
        sl = {q, want};
    }
    *p = sl.first;
    return hipSuccess;
}

// words used per level 0..levels-1 (one small readback in place of every bucket size)
static hd_status level_used(hd_ctx* ctx, hipStream_t s, std::vector<uint64_t>& used) {
    const Geom& g = ctx->g;
    unsigned long long* d = nullptr;
    hipError_t e = gc_slot(ctx, kSlotUsed, (uint64_t)g.levels * 8, (void**)&d);
    if (e != hipSuccess) return hip_fail(ctx, e, "GC scratch");
    k_gc_fill<<<1, 64, 0, s>>>((uint32_t*)d, (uint64_t)g.levels * 2, 0u);
    k_gc_level_used<<<dim3(64, g.levels), 256, 0, s>>>(g, ctx->bucket_sizes, d);
    used.assign(g.levels, 0);
    HD_HIP(ctx, hipMemcpyAsync(used.data(), d, (uint64_t)g.levels * 8, hipMemcpyDeviceToHost, s));
    HD_HIP(ctx, hipStreamSynchronize(s));
    return HD_OK;
}

static hd_status gc_run(hd_ctx* ctx, uint32_t max_level, uint32_t* extra, uint32_t n_extra, bool keep_undo,
                        uint64_t stats[4], void* stream) {
    if (!ctx || !ctx->loaded) return fail(ctx, HD_ERR_INVALID, "no DAG loaded");
    const Geom& g = ctx->g;
    const uint32_t L = g.leaf_level();
    if (max_level > L) return fail(ctx, HD_ERR_INVALID, "max_level above the leaf level");
    if (n_extra && !extra) return fail(ctx, HD_ERR_INVALID, "extra roots missing");
    const std::vector<uint32_t> roots = gc_root_set(ctx, extra, n_extra, keep_undo);
    for (uint32_t r : roots)
        if (r >= g.total_virtual()) return fail(ctx, HD_ERR_INVALID, "a root is not an address of the table");
    const uint32_t nRoots = (uint32_t)roots.size();
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    // capacities: used words per level bound the number of nodes
    std::vector<uint64_t> used;
    {
        const hd_status st = level_used(ctx, s, used);
        if (st != HD_OK) return st;
    }
    // every node takes at least 2 words, so a level holds at most used / 2 nodes
    auto fcap = [&](uint32_t l) {
        return (uint32_t)std::max<uint64_t>(std::max<uint64_t>(used[l] / 2 + 16, 16), l == 0 ? nRoots : 0);
    };
    uint64_t capMax = 16;
    for (uint32_t l = 0; l <= max_level; ++l) capMax = std::max<uint64_t>(capMax, fcap(l));
    if (capMax >= (1u << 30)) return fail(ctx, HD_ERR_INVALID, "level too large for GC scratch");
    const uint32_t cap = (uint32_t)capMax;

    // scratch from the context's slots (kept between calls; every kernel is given its sizes)
    auto alloc = [&](uint32_t slot, void** p, uint64_t bytes) -> hipError_t { return gc_slot(ctx, slot, bytes, p); };
    auto release = [&]() { hipStreamSynchronize(s); };
    // the mark bitmap and, behind it, the list head of every bucket
    const uint64_t bitmapWords = (g.total_virtual() + 31) / 32, headWords = g.total_buckets();
    uint32_t *bitmap, *report, *fwd;
    GcRow* rows;
    std::vector<uint32_t*> frontier(max_level + 1, nullptr);
    hipError_t e = alloc(kSlotBitmap, (void**)&bitmap, (bitmapWords + headWords) * 4);
    if (e == hipSuccess) e = alloc(kSlotReport, (void**)&report, ((uint64_t)kRepRoots + nRoots) * 4);
    for (uint32_t l = 0; l <= max_level && e == hipSuccess; ++l)
        e = alloc(kSlotFrontier + l, (void**)&frontier[l], (uint64_t)fcap(l) * 4);
    if (e == hipSuccess) e = alloc(kSlotRows, (void**)&rows, (uint64_t)cap * sizeof(GcRow));
    // old address -> new address of every live node: one word per virtual address (written
    // for live nodes only, read only for them)
    if (e == hipSuccess) e = alloc(kSlotFwd, (void**)&fwd, (uint64_t)g.total_virtual() * 4);
    if (e != hipSuccess) {
        release();
        gc_scratch_free(ctx);  // give back what a smaller call could not reuse
        return hip_fail(ctx, e, "GC scratch");
    }
    uint32_t *head = bitmap + bitmapWords, *errors = report, *counts = report + kRepCounts, *droots = report + kRepRoots;
    auto grid = [&](uint32_t l) { return std::min((fcap(l) + 255) / 256, kGcGrid); };
    k_gc_fill<<<2048, 256, 0, s>>>(bitmap, bitmapWords + headWords, 0u);
    e = hipMemcpyAsync(droots, roots.data(), (uint64_t)nRoots * 4, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) {
        release();
        return hip_fail(ctx, e, "GC roots");
    }
    k_gc_seed<<<(nRoots + 255) / 256, 256, 0, s>>>(frontier[0], report, nRoots);
    for (uint32_t l = 0; l < max_level; ++l)
        k_gc_mark<<<grid(l), 256, 0, s>>>(ctx->vpool, bitmap, frontier[l], frontier[l + 1], counts, l, fcap(l),
                                          fcap(l + 1), g.total_virtual(), errors);
    {  // nothing has been modified yet: stop here if the mark overflowed or met a bad pointer
        uint32_t markErr = 0;
        HD_HIP(ctx, hipMemcpyAsync(&markErr, errors, 4, hipMemcpyDeviceToHost, s));
        e = hipStreamSynchronize(s);
        if (e != hipSuccess || markErr) {
            release();
            if (e != hipSuccess) return hip_fail(ctx, e, "GC mark");
            return fail(ctx, HD_ERR_INVALID, "GC mark: a child pointer is outside the table or a level overflowed");
        }
    }
    TableRef T{g, ctx->vpool, ctx->page_table, ctx->bucket_sizes, ctx->counters + 0, ctx->cfg.pool_pages};
    for (uint32_t l = max_level; l != (uint32_t)-1; --l) {
        k_gc_gather<<<grid(l), 256, 0, s>>>(g, ctx->vpool, frontier[l], report, l, max_level, fcap(l), fwd,
                                            ctx->full_nodes, rows, head);
        const uint32_t blocks = (g.buckets_per_level(l) + kPlaceBuckets - 1) / kPlaceBuckets;
        if (blocks >= kPlaceFull) k_gc_place<true><<<blocks, 256, 0, s>>>(T, l, report, ctx->full_nodes, rows, head, fwd, errors);
        else k_gc_place<false><<<blocks, 256, 0, s>>>(T, l, report, ctx->full_nodes, rows, head, fwd, errors);
    }
    k_gc_roots<<<(nRoots + 255) / 256, 256, 0, s>>>(fwd, droots, nRoots, errors);
    if (stats)
        k_gc_level_used<<<dim3(64, g.levels), 256, 0, s>>>(g, ctx->bucket_sizes,
                                                           (unsigned long long*)(report + kRepUsed));
    std::vector<uint32_t> rep(kRepRoots + nRoots);
    HD_HIP(ctx, hipMemcpyAsync(rep.data(), report, rep.size() * 4, hipMemcpyDeviceToHost, s));
    e = hipStreamSynchronize(s);
    const uint32_t err = rep[0];
    const std::vector<uint32_t> newRoots(rep.begin() + kRepRoots, rep.end());
    release();
    if (e != hipSuccess || err) {
        // levels were rewritten in place up to the failure: the table no longer holds the DAG,
        // so every call on this context refuses until a DAG is loaded again
        ctx->loaded = false;
        ctx->undo.clear();
        ctx->redo.clear();
        if (e != hipSuccess) return hip_fail(ctx, e, "GC");
        return fail(ctx, err & GC_ERR_POOL ? HD_ERR_POOL_FULL : HD_ERR_BUCKET_FULL,
                    "GC failed (capacity); the table is no longer consistent: load a DAG again");
    }
    ctx->root = remap(roots, newRoots, ctx->root);
    HD_HIP(ctx, hipMemcpyAsync(ctx->d_root, &ctx->root, 4, hipMemcpyHostToDevice, s));
    {
        const hd_status ts = leaf_tags_rebuild(ctx, s);  // the leaf buckets were rewritten
        if (ts != HD_OK) return ts;
    }
    for (uint32_t i = 0; i < n_extra; ++i) extra[i] = remap(roots, newRoots, extra[i]);
    if (keep_undo) {
        for (auto* frames : {&ctx->undo, &ctx->redo})
            for (UndoFrame& f : *frames) {
                f.prev_root = remap(roots, newRoots, f.prev_root);
                f.new_root = remap(roots, newRoots, f.new_root);
            }
    } else {
        ctx->undo.clear();  // old roots point at collected nodes (engine.cpp:178-185 frees undo)
        ctx->redo.clear();
    }
    if (stats) {
        uint64_t live = 0, before = 0, after = 0;
        for (uint32_t l = 0; l <= max_level; ++l) {
            live += rep[kRepCounts + l];
            before += used[l];
            after += rep[kRepUsed + 2 * l] | (uint64_t)rep[kRepUsed + 2 * l + 1] << 32;
        }
        stats[0] = live;
        stats[1] = before;
        stats[2] = after;
        stats[3] = 0;
    }
    return HD_OK;
}

namespace hd {
void gc_scratch_free(hd_ctx* ctx) {
    if (!ctx) return;
    for (auto& sl : ctx->gc_slots)
        if (sl.first) hipFree(sl.first);
    ctx->gc_slots.clear();
}
}  // namespace hd

extern "C" hd_status hd_gc(hd_ctx* ctx, uint32_t max_level, uint64_t stats[4], void* stream) {
    return gc_run(ctx, max_level, nullptr, 0, false, stats, stream);
}

extern "C" hd_status hd_gc_roots(hd_ctx* ctx, uint32_t max_level, uint32_t keep_undo, uint32_t* roots,
                                 uint32_t n_roots, uint64_t stats[4], void* stream) {
    return gc_run(ctx, max_level, roots, n_roots, keep_undo != 0, stats, stream);
}
