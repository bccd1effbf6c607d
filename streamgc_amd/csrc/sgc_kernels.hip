// sgc_kernels.hip -- HIP kernels of the StreamGC hot path for gfx950.
//
// Work decomposition: a parallel batch's updates are grouped by edge, an edge
// to a wavefront or four light edges to one; deterministic batches replay each
// graph's segment by a block of wavefronts (one wavefront where there are very
// many segments).  Epoch sweeps run over the vertex rows of the graphs taking
// part (their vertex counts laid end to end), one to four short rows to a
// wavefront, a longer row to a wavefront, the longest to a block; rows are
// streamed 64 slots per load.  The deterministic repair sweep runs one block per
// graph in vertex order.
#include <hip/hip_runtime.h>

#include "sgc_device.hpp"
#include "sgc_launch.hpp"

namespace sgc {

__device__ __forceinline__ uint32_t wave_id() { return (blockIdx.x * blockDim.x + threadIdx.x) / WAVE; }
__device__ __forceinline__ uint32_t wave_count() { return (gridDim.x * blockDim.x) / WAVE; }

// The vertex space of a launch: the vertices of the graphs taking part, one
// graph after another.  A launch over a few graphs of a large pool touches
// only their vertices.
struct Space {
    const uint32_t* base;  // ns + 1 prefix of vertex counts (null: a single graph)
    const uint32_t* gid;   // graph id of each part (null: part k is graph k)
    uint32_t ns;
    uint32_t total;
    __device__ __forceinline__ void locate(uint32_t i, uint32_t& g, uint32_t& v) const {
        uint32_t lo = 0;
        if (base && ns > 1) {
            uint32_t hi = ns;
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (base[mid] <= i) lo = mid;
                else hi = mid;
            }
        }
        g = gid ? gid[lo] : lo;
        v = base ? i - base[lo] : i;
    }
};

// A vertex space written on the device (a captured round's control kernel
// lays out the graphs still taking part; see dspace_words).
__device__ __forceinline__ Space device_space(const uint32_t* dspace, uint32_t ng) {
    return Space{dspace + 4, dspace + 4 + ng + 1, dspace[0], dspace[1]};
}

// ---------------------------------------------------------------- sweep sets
// A maintenance sweep visits either every virtual vertex (list == null) or the
// worklist launch_build_list left on the device.
// The worklist keeps rows of at most `long_row` filled slots at its front
// (count[0] of them, for_rows) and longer rows at its back
// (count[1], list[cap - 1 - k], one 256-thread block each), so a hub row
// costs a few block-wide round trips instead of hundreds of wavefront ones.
// Lengths are read on the device: the host never waits for them.
constexpr uint32_t BLOCK = 256;

struct SweepList {
    const uint32_t* list;   // null: every vertex
    const uint32_t* count;  // [small, big]
    uint32_t cap;
};
__device__ __forceinline__ uint32_t sweep_small(const SweepList& sl, uint32_t V) { return sl.list ? sl.count[0] : V; }
__device__ __forceinline__ uint32_t sweep_big(const SweepList& sl) { return sl.list ? sl.count[1] : 0; }
__device__ __forceinline__ uint32_t small_item(const SweepList& sl, uint32_t k) { return sl.list ? sl.list[k] : k; }
__device__ __forceinline__ uint32_t big_item(const SweepList& sl, uint32_t k) { return sl.list[sl.cap - 1 - k]; }

// The front rows of a sweep set (or every row) over the grid's wavefronts.
// Rows are short -- 6 slots on a mesh, 17 on a social graph -- and a row is one
// chain of dependent loads (list entry, row bounds, slots, neighbours' words),
// so a wavefront takes up to four rows at a time, 16 lanes each, as many as its
// share of the rows.  A full sweep of 4.0M rows and 69M live
// slots, one row a wavefront / four: compaction 1,180 / 324 us, rebuild 2,200 /
// 1,137 us, Tier-1 3,513 / 1,071 us (what is left is the gather of 69M
// neighbour words).  body(g, gid, mine, v) runs with g wave-uniform (rows of
// several graphs: one graph after another); mine says whether the lane's row v
// takes part.
constexpr uint32_t GROUP = 16, GROUPS = WAVE / GROUP;
constexpr uint32_t GROUP_ROW = ROW_UNROLL * GROUP;   // slots 16 lanes load in one round trip
__device__ __forceinline__ uint32_t sublane() { return lane() % GROUP; }
__device__ __forceinline__ uint32_t group_bits(uint64_t m) {   // the lane's group's bits of a ballot
    return (uint32_t)(m >> (lane() / GROUP * GROUP)) & 0xFFFFu;
}
template <class F>
__device__ __forceinline__ void for_rows(const GraphDev* __restrict__ graphs, const Space& sp, const SweepList& sl,
                                         F&& body) {
    const uint32_t total = sweep_small(sl, sp.total);
    const uint32_t fair = (total + wave_count() - 1) / wave_count();   // rows a wavefront
    const uint32_t per = fair < 1 ? 1u : fair < GROUPS ? fair : GROUPS, mine_of = lane() / GROUP;
    for (uint32_t k0 = wave_id() * per; k0 < total; k0 += wave_count() * per) {
        const bool have = mine_of < per && k0 + mine_of < total;
        uint32_t gid = 0, v = 0;
        if (have) sp.locate(small_item(sl, k0 + mine_of), gid, v);
        uint64_t pend = ballot(have);
        while (pend) {
            const uint32_t g0 = __builtin_amdgcn_readlane(gid, (uint32_t)__builtin_ctzll(pend));
            const bool mine = have && gid == g0;
            pend &= ~ballot(mine);
            body(graphs[g0], g0, mine, v);
        }
    }
}
// Every row, a wavefront each: f(g, gid, v).
template <class F>
__device__ __forceinline__ void for_each_row(const GraphDev* __restrict__ graphs, const Space& sp, F&& f) {
    for (uint32_t k = wave_id(); k < sp.total; k += wave_count()) {
        uint32_t gid, v;
        sp.locate(k, gid, v);
        f(graphs[gid], gid, v);
    }
}
// The rows of `m` (a lane mask), one after another by the whole wavefront: f(v).
template <class F>
__device__ __forceinline__ void each_row(uint64_t m, uint32_t v, F&& f) {
    for (; m; m &= m - 1) f((uint32_t)__builtin_amdgcn_readlane(v, (uint32_t)__builtin_ctzll(m)));
}

// Block-wide sum of per-wave values into one u64 total (one atomic per block).
// Every thread of the block must call it.
__device__ __forceinline__ void block_add64(uint64_t* totals, uint32_t idx, uint64_t mine) {
    __shared__ uint64_t part[BLOCK / WAVE];
    const uint32_t w = threadIdx.x / WAVE;
    if (lane() == 0) part[w] = mine;
    __syncthreads();
    if (threadIdx.x == 0 && totals) {
        uint64_t t = 0;
        for (uint32_t k = 0; k < BLOCK / WAVE; k++) t += part[k];
        if (t) tot_add(totals, idx, t);
    }
    __syncthreads();
}

// Block-wide sum (every thread gets it).  Every thread must call it.
__device__ __forceinline__ uint32_t block_sum32(uint32_t x) {
    __shared__ uint32_t part[BLOCK / WAVE];
    x = wave_sum32(x);
    if (lane() == 0) part[threadIdx.x / WAVE] = x;
    __syncthreads();
    uint32_t t = 0;
    for (uint32_t k = 0; k < BLOCK / WAVE; k++) t += part[k];
    __syncthreads();
    return t;
}

// Exclusive prefix of x over the block (thread order); *total = block sum.
__device__ __forceinline__ uint32_t block_scan32(uint32_t x, uint32_t* total) {
    __shared__ uint32_t part[BLOCK / WAVE];
    uint32_t inc = x;
    for (uint32_t d = 1; d < WAVE; d <<= 1) {
        const uint32_t y = __shfl_up(inc, d);
        if (lane() >= d) inc += y;
    }
    const uint32_t w = threadIdx.x / WAVE;
    if (lane() == WAVE - 1) part[w] = inc;
    __syncthreads();
    uint32_t before = 0, t = 0;
    for (uint32_t k = 0; k < BLOCK / WAVE; k++) {
        before += k < w ? part[k] : 0;
        t += part[k];
    }
    __syncthreads();
    *total = t;
    return before + inc - x;
}

// The worklist of a sweep (the vertices marked `kind`, or sticky; their marks
// are cleared), in two passes with no shared counter.  The vertices are cut
// into tiles of LIST_TILE_V, each inside one graph (with several graphs, each
// graph's tiles follow the previous graph's).  Each thread reads the marks of
// 4 vertices as one word (mark arrays are padded to a multiple of 4) with no
// per-vertex branches.  Pass 1: each block takes a tile, lists its hits in
// the tile's own region of a scratch array (short rows up from the start,
// long rows down from the end), clears their marks and stores its two
// counts.  Pass 2: each block adds up the counts of the tiles before it and
// copies its hits to their places in the worklist; the last block stores the
// totals.
constexpr uint32_t LIST_WORDS = 4;                          // mark words per thread
constexpr uint32_t LIST_TILE_V = BLOCK * LIST_WORDS * 4;    // vertices per tile
static_assert(LIST_TILE_V == 4096, "list_words() sizes the scratch for 4096-vertex tiles");

struct ListTile {
    uint32_t small[LIST_WORDS], big[LIST_WORDS];   // 4-bit vertex masks per word
};
__device__ __forceinline__ uint32_t nonzero_bytes(uint32_t x) {
    return ((x & 0xFFu) != 0) | (((x >> 8) & 0xFFu) != 0) << 1 | (((x >> 16) & 0xFFu) != 0) << 2 |
           (((x >> 24) & 0xFFu) != 0) << 3;
}
__device__ __forceinline__ void list_tile(const GraphDev& g, uint32_t kind, uint32_t long_row, uint32_t tile,
                                          uint32_t words, ListTile& out) {
    SGC_G uint32_t* mk = (SGC_G uint32_t*)(gp(g.dirty) + (size_t)kind * g.dstride);
    const SGC_G uint32_t* sk = (const SGC_G uint32_t*)(gp(g.dirty) + (size_t)M_STICKY * g.dstride);
    // Sticky marks come only with an event counted in C_ASYM (overflow,
    // duplicate): a graph that never had one has none, and its sticky array
    // is not read.
    const bool any_sticky = ld(&g.ctr[C_ASYM]) != 0;
    uint32_t m[LIST_WORDS], h[LIST_WORDS];
#pragma unroll
    for (uint32_t k = 0; k < LIST_WORDS; k++) {
        const uint32_t w = tile * (BLOCK * LIST_WORDS) + k * BLOCK + threadIdx.x;
        m[k] = w < words ? mk[w] : 0u;
        h[k] = any_sticky && w < words ? sk[w] : 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < LIST_WORDS; k++) {
        const uint32_t w = tile * (BLOCK * LIST_WORDS) + k * BLOCK + threadIdx.x;
        uint32_t hit = nonzero_bytes(m[k] | h[k]);
        if (4 * w + 4 > g.n) hit &= (1u << (g.n > 4 * w ? g.n - 4 * w : 0u)) - 1u;   // padding bytes
        uint32_t big = 0;
        if (hit) {   // fill is allocated to a multiple of 4 vertices
            const uint4 f = *reinterpret_cast<const uint4*>(g.fill + 4 * (size_t)w);
            big = ((f.x > long_row) | (f.y > long_row) << 1 | (f.z > long_row) << 2 | (f.w > long_row) << 3) & hit;
        }
        out.small[k] = hit & ~big;
        out.big[k] = big;
        if (m[k]) mk[w] = 0u;
    }
}

__global__ __launch_bounds__(256) void k_list_tiles(const GraphDev* __restrict__ graphs, Space sp,
                                                    const uint32_t* __restrict__ stile, uint32_t kind, uint32_t kind2,
                                                    size_t second, uint32_t long_row, uint32_t* __restrict__ tmp,
                                                    uint32_t* __restrict__ tcount,
                                                    const uint32_t* __restrict__ active,
                                                    const uint32_t* __restrict__ gate) {
    if (gate && *gate == 0) return;
    if (blockIdx.y) {   // the second list
        kind = kind2;
        tmp += second;
        tcount += second;
    }
    const uint32_t t = blockIdx.x;
    // Several graphs: their tiles laid end to end (stile = prefix of each
    // part's tile count); the part holding tile t, found by the whole block.
    uint32_t part = 0, first = 0;
    if (stile && sp.ns > 1) {
        uint32_t lo = 0, hi = sp.ns;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (stile[mid] <= t) lo = mid;
            else hi = mid;
        }
        part = lo;
        first = stile[lo];
    }
    const uint32_t gid = sp.gid ? sp.gid[part] : part;
    const uint32_t off = sp.base ? sp.base[part] : 0u;   // virtual index of the graph's vertex 0
    if (active && active[gid] == 0) {
        if (stile && sp.ns > 1 && threadIdx.x == 0) {   // nothing listed from this tile
            gp(tcount)[2 * t] = 0;
            gp(tcount)[2 * t + 1] = 0;
        }
        return;
    }
    const GraphDev g = graphs[gid];
    const uint32_t words = (g.n + 3) / 4;
    const uint32_t lt_index = t - first;   // the tile within its graph
    ListTile lt;
    list_tile(g, kind, long_row, lt_index, words, lt);
    uint32_t cs = 0, cb = 0;
#pragma unroll
    for (uint32_t k = 0; k < LIST_WORDS; k++) {
        cs += __builtin_popcount(lt.small[k]);
        cb += __builtin_popcount(lt.big[k]);
    }
    uint32_t ts, tb;
    uint32_t ps = block_scan32(cs, &ts);
    uint32_t pb = block_scan32(cb, &tb);
    SGC_G uint32_t* region = gp(tmp) + (size_t)t * LIST_TILE_V;
#pragma unroll
    for (uint32_t k = 0; k < LIST_WORDS; k++) {
        const uint32_t v0 = off + 4 * (lt_index * (BLOCK * LIST_WORDS) + k * BLOCK + threadIdx.x);
        for (uint32_t q = 0; q < 4; q++) {
            if ((lt.small[k] >> q) & 1u) region[ps++] = v0 + q;
            if ((lt.big[k] >> q) & 1u) region[LIST_TILE_V - 1 - pb++] = v0 + q;
        }
    }
    if (threadIdx.x == 0) {
        gp(tcount)[2 * t] = ts;
        gp(tcount)[2 * t + 1] = tb;
    }
}

__global__ __launch_bounds__(256) void k_list_gather(const GraphDev* __restrict__ graphs, Space sp, int multi,
                                                     const uint32_t* __restrict__ tmp,
                                                     const uint32_t* __restrict__ tcount,
                                                     uint32_t* __restrict__ list, uint32_t cap, size_t second,
                                                     uint32_t* __restrict__ count,
                                                     const uint32_t* __restrict__ active,
                                                     const uint32_t* __restrict__ gate) {
    if (blockIdx.y) {
        tmp += second;
        tcount += second;
        list += second;
        count += 2;
    }
    // one graph not taking part: nothing listed (several graphs: the tiles of
    // those not taking part counted nothing)
    const uint32_t gid = sp.gid ? sp.gid[0] : 0u;
    if ((gate && *gate == 0) || (!multi && active && active[gid] == 0)) {
        if (blockIdx.x == 0 && threadIdx.x < 2) count[threadIdx.x] = 0;
        return;
    }
    const uint32_t t = blockIdx.x;
    uint32_t bs = 0, bb = 0;
    for (uint32_t k = threadIdx.x; k < t; k += BLOCK) {
        bs += gp(tcount)[2 * k];
        bb += gp(tcount)[2 * k + 1];
    }
    bs = block_sum32(bs);
    bb = block_sum32(bb);
    const uint32_t ns = gp(tcount)[2 * t], nb = gp(tcount)[2 * t + 1];
    const SGC_G uint32_t* region = gp(tmp) + (size_t)t * LIST_TILE_V;
    for (uint32_t k = threadIdx.x; k < ns; k += BLOCK) gp(list)[bs + k] = region[k];
    for (uint32_t k = threadIdx.x; k < nb; k += BLOCK) gp(list)[cap - 1 - (bb + k)] = region[LIST_TILE_V - 1 - k];
    if (t == gridDim.x - 1 && threadIdx.x == 0) {
        count[0] = bs + ns;
        count[1] = bb + nb;
    }
}

__global__ void k_zero_list_count(uint32_t* p) {
    p[0] = 0;
    p[1] = 0;
}

// ---------------------------------------------------------------- per-edge ordering
// Parallel waves apply a batch in no particular order, so two updates of one
// edge in one batch (a delete and its re-insert, frequent in churn streams)
// could land in either order and leave the rows disagreeing with the stream.
// Before a parallel batch, the updates are grouped by edge (global vertex ids
// of the pool, lo << 32 | hi) in a hash table: each slot heads a linked list
// of the batch positions of that edge.  The wave that owns the list head
// applies the whole group in stream order; different edges stay parallel.
constexpr uint64_t KEY_EMPTY = ~0ull;
constexpr uint32_t NONE = 0xFFFFFFFFu;

__device__ __forceinline__ uint64_t edge_key(const GraphDev* __restrict__ graphs, const uint32_t* __restrict__ gbase,
                                             const uint4& r, int multi) {
    const uint32_t gid = multi ? r.w : 0u;
    const uint32_t n = graphs[gid].n;
    if (r.x >= n || r.y >= n || (r.z & 0xFFu) > 1u) return KEY_EMPTY;
    const uint32_t base = multi ? gbase[gid] : 0u;
    const uint32_t a = base + (r.x < r.y ? r.x : r.y), b = base + (r.x < r.y ? r.y : r.x);
    return ((uint64_t)a << 32) | b;
}
__device__ __forceinline__ uint32_t key_hash(uint64_t k, uint32_t mask) {
    k ^= k >> 33;
    k *= 0xff51afd7ed558ccdull;
    k ^= k >> 33;
    return (uint32_t)k & mask;
}

// The listed edges of a batch by the longer of their two rows: those with more
// than HEAVY_FILL filled slots (the long scans, which start first) from the
// front of `heads`, the light ones (four to a wavefront, apply_quad) from its
// end.  The line lies where 8 lanes still scan a row as fast as the chip needs:
// 262K updates of 64 graphs of 2^10..2^15 vertices take 291 us with light
// edges up to 64 slots, 257 up to 256 and 213 up to 1,024; a 131,072-vertex
// mesh and the 4M-vertex power-law graph take the same with all three.

// The table is empty between batches: k_group_pack frees the slots it reads,
// and k_apply_elem, which reads the counts that k_group_pack copied, clears the
// ones k_group_link adds to.  A batch so needs no launch to clear the table
// (2-4 us, and up to 12 before the next one starts when the host sets the pace).
__global__ __launch_bounds__(256) void k_group_clear(uint64_t* __restrict__ keys, uint32_t* __restrict__ head,
                                                     uint32_t size, uint32_t* __restrict__ nheads) {
    if (blockIdx.x == 0 && threadIdx.x < GROUP_WORDS) nheads[threadIdx.x] = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < size; i += gridDim.x * blockDim.x) {
        gp(keys)[i] = KEY_EMPTY;
        gp(head)[i] = NONE;
    }
}

// Slot of `key` (inserted when absent; *created tells whether this call
// inserted it).  The table holds at least twice the batch, so a free slot
// always exists and the probe ends.
__device__ __forceinline__ uint32_t group_slot(uint64_t* __restrict__ keys, uint64_t key, uint32_t mask,
                                               bool* created) {
    uint32_t s = key_hash(key, mask);
    for (uint32_t probes = 0; probes <= mask; s = (s + 1) & mask, probes++) {
        uint64_t found = KEY_EMPTY;
        __hip_atomic_compare_exchange_strong(gp(&keys[s]), &found, key, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
        *created = found == KEY_EMPTY;
        if (found == KEY_EMPTY || found == key) return s;
    }
    return NONE;
}

// Links every update of the batch into its edge's list, and lists each edge
// once (the update that inserted the key adds its slot; an update whose key
// found no slot is listed alone, position | GROUP_SINGLE): the per-update
// kernels then take one edge after another.  Records that change nothing
// (out-of-range vertex, other kinds) are not listed.  Each block appends its
// entries with one atomic per list end; nheads = [heavy, light] counts, and
// k_group_pack's copy of them.
constexpr uint32_t GROUP_SINGLE = 0x80000000u;

__global__ __launch_bounds__(256) void k_group_link(const GraphDev* __restrict__ graphs,
                                                    const uint32_t* __restrict__ gbase,
                                                    const uint4* __restrict__ upd, uint32_t count, int multi,
                                                    uint64_t* __restrict__ keys, uint32_t* __restrict__ head,
                                                    uint32_t* __restrict__ next, uint32_t mask,
                                                    uint32_t* __restrict__ heads, uint32_t cap,
                                                    uint32_t* __restrict__ nheads, const uint32_t* __restrict__ dyn) {
    __shared__ uint32_t block_at[2];
    if (dyn) {   // the batch is a slice of a device-resident stream: [offset, count] read here
        upd += dyn[0];
        count = dyn[1];
    }
    for (uint32_t b0 = blockIdx.x * blockDim.x; b0 < count; b0 += gridDim.x * blockDim.x) {
        const uint32_t i = b0 + threadIdx.x;
        uint32_t entry = NONE;
        bool heavy = false;
        if (i < count) {
            const uint4 r = upd[i];
            const uint64_t key = edge_key(graphs, gbase, r, multi);
            uint32_t prev = NONE;
            if (key != KEY_EMPTY) {
                bool created = false;
                const uint32_t s = group_slot(keys, key, mask, &created);
                if (s != NONE) {
                    prev = __hip_atomic_exchange(gp(&head[s]), i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (created) entry = s;
                } else {
                    entry = i | GROUP_SINGLE;
                }
                if (entry != NONE) {
                    const GraphDev& g = graphs[multi ? r.w : 0u];
                    heavy = gp(g.fill)[r.x] > HEAVY_FILL || gp(g.fill)[r.y] > HEAVY_FILL;
                }
            }
            gp(next)[i] = prev;
        }
        uint32_t total;   // both counts in one scan, 16 bits each (a block has at most 256)
        const uint32_t before = block_scan32(entry == NONE ? 0u : heavy ? 1u : 1u << 16, &total);
        if (threadIdx.x < 2) {
            const uint32_t mine = threadIdx.x ? total >> 16 : total & 0xFFFFu;
            block_at[threadIdx.x] = mine ? add32(&nheads[threadIdx.x], mine) : 0u;
        }
        __syncthreads();
        if (entry != NONE)
            gp(heads)[heavy ? block_at[0] + (before & 0xFFFFu) : cap - 1 - (block_at[1] + (before >> 16))] = entry;
        __syncthreads();
    }
}

// One thread per listed edge: the records of its updates, in stream order,
// into the edge's own GROUP_PACK x 16-byte line of `pack`, so that the
// per-update kernel has a whole group after one load instead of walking
// head, list links and records one dependent load after another.  Unused
// entries are PACK_NONE records; an edge with more than GROUP_PACK updates is
// left to the walk (its first entry says so and carries the list's first position).
constexpr uint32_t GROUP_PACK = 4;
constexpr uint32_t PACK_NONE = 0xFFFFFFFFu;   // x of an entry with no record (a listed record has x < n)
constexpr uint32_t PACK_END = 0, PACK_WALK = 1;   // y of such an entry

__device__ __forceinline__ void cswap(uint32_t& a, uint32_t& b) {
    const uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
    a = lo;
    b = hi;
}

__global__ __launch_bounds__(256) void k_group_pack(const uint4* __restrict__ upd, uint64_t* __restrict__ keys,
                                                    uint32_t* __restrict__ ghead,
                                                    const uint32_t* __restrict__ gnext,
                                                    const uint32_t* __restrict__ heads, uint32_t cap,
                                                    uint32_t* __restrict__ nheads, uint4* __restrict__ pack,
                                                    const uint32_t* __restrict__ dyn) {
    if (dyn) upd += dyn[0];
    if (blockIdx.x == 0 && threadIdx.x < 2) nheads[2 + threadIdx.x] = nheads[threadIdx.x];
    const uint32_t nh = nheads[0], n = nh + nheads[1];
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) {
        const uint32_t e = j < nh ? heads[j] : heads[cap - 1 - (j - nh)];
        uint32_t p0 = NONE, p1 = NONE, p2 = NONE, p3 = NONE;
        bool more = false;
        if (e & GROUP_SINGLE) {
            p0 = e & ~GROUP_SINGLE;
        } else {
            p0 = gp(ghead)[e];
            if (p0 != NONE) p1 = gp(gnext)[p0];
            if (p1 != NONE) p2 = gp(gnext)[p1];
            if (p2 != NONE) p3 = gp(gnext)[p2];
            more = p3 != NONE && gp(gnext)[p3] != NONE;
        }
        uint4* out = pack + (size_t)j * GROUP_PACK;
        if (!(e & GROUP_SINGLE)) {
            gp(keys)[e] = KEY_EMPTY;
            gp(ghead)[e] = NONE;
        }
        if (more) {
            out[0] = make_uint4(PACK_NONE, PACK_WALK, 0u, p0);
            continue;
        }
        cswap(p0, p1);   // sorting network for 4 (NONE sorts last)
        cswap(p2, p3);
        cswap(p0, p2);
        cswap(p1, p3);
        cswap(p1, p2);
        // (each record loaded under its own branch: selects between whole
        // vector records put them in scratch memory)
        const uint4 none = make_uint4(PACK_NONE, PACK_END, 0u, 0u);
        uint4 r0 = none, r1 = none, r2 = none, r3 = none;
        if (p0 != NONE) r0 = upd[p0];
        if (p1 != NONE) r1 = upd[p1];
        if (p2 != NONE) r2 = upd[p2];
        if (p3 != NONE) r3 = upd[p3];
        out[0] = r0;
        out[1] = r1;
        out[2] = r2;
        out[3] = r3;
    }
}

// ---------------------------------------------------------------- updates
template <bool LONG = false>
__device__ __forceinline__ void apply_rec(const GraphDev* __restrict__ graphs, const uint4& r, int multi, WaveAcc& acc,
                                          RowHint* hint = nullptr) {
    const uint32_t gid = multi ? r.w : 0u;
    const GraphDev g = graphs[gid];
    apply_update<LONG>(g, r.x, r.y, r.z & 0xFFu, acc, hint);
}
__device__ __forceinline__ void apply_record(const GraphDev* __restrict__ graphs, const uint4* __restrict__ upd,
                                             uint32_t i, int multi, WaveAcc& acc, RowHint* hint = nullptr) {
    apply_rec(graphs, upd[i], multi, acc, hint);
}

__device__ __forceinline__ uint4 uniform_rec(const uint4& r) {
    return make_uint4(bcast0(r.x), bcast0(r.y), bcast0(r.z), bcast0(r.w));
}

// Listed edge j's updates in stream order, by the whole wavefront.  The records
// come from the edge's packed 64-byte line (lanes 0..3 load one each), or, for a
// group longer than the line, from its list: repeatedly the record at the
// smallest position above the last one applied.
// SCALAR: the record in scalar registers.  Alone the update's code takes 165
// vector registers and spills 34 scalar ones without it, 138 and 182 with it,
// and 4,099 updates of a 65,536-vertex R-MAT graph take 45 us without and 48-64
// with it.  Beside the four-edge path it is the other way round: without it the
// kernel spills 64 vector registers into 52 B of scratch a lane, with it none.
template <bool SCALAR, bool LONG>
__device__ __forceinline__ void apply_edge(const GraphDev* __restrict__ graphs, const uint4* __restrict__ upd, int multi,
                                           const uint32_t* __restrict__ gnext, const uint4* __restrict__ pack, uint32_t j,
                                           WaveAcc& acc, uint64_t& grouped) {
    uint4 mine = make_uint4(PACK_NONE, PACK_WALK, 0u, 0u);
    if (lane() < GROUP_PACK) mine = pack[(size_t)j * GROUP_PACK + lane()];
    const bool walk = __builtin_amdgcn_readlane(mine.x, 0) == PACK_NONE &&
                      __builtin_amdgcn_readlane(mine.y, 0) == PACK_WALK;
    const uint32_t h = walk ? pack[(size_t)j * GROUP_PACK].w : NONE;   // the list's first position
    RowHint hint;   // a delete's slots for the same edge's re-insert (a last delete's marks wait in it)
    hint.valid = false;
    uint32_t applied = 0, last = 0, last_g = 0;
    for (;;) {
        uint4 r;
        if (!walk) {
            if (applied == GROUP_PACK) break;
            r = make_uint4(__builtin_amdgcn_readlane(mine.x, applied), __builtin_amdgcn_readlane(mine.y, applied),
                           __builtin_amdgcn_readlane(mine.z, applied), __builtin_amdgcn_readlane(mine.w, applied));
            if (r.x == PACK_NONE) break;
        } else {
            uint32_t best = NONE;
            for (uint32_t k2 = h; k2 != NONE; k2 = gp(gnext)[k2])
                if ((applied == 0 || k2 > last) && (best == NONE || k2 < best)) best = k2;
            if (best == NONE) break;
            r = upd[best];
            last = best;
        }
        apply_rec<LONG>(graphs, SCALAR ? uniform_rec(r) : r, multi, acc, &hint);
        last_g = r.w;
        applied++;
    }
    if (hint.valid) hint_release(graphs[multi ? last_g : 0u], &hint);   // marks of a last delete
    grouped += applied ? applied - 1 : 0;
}

// One wavefront per edge of the batch.  Bound: the chain of an edge's dependent
// gathers and atomics, 165 registers (3 wavefronts a SIMD).  4,099 updates of a
// 131,072-vertex mesh 16 us, of a 65,536-vertex R-MAT graph 45 us (its hub rows'
// scans).
__global__ __launch_bounds__(64) void k_apply_elem(const GraphDev* __restrict__ graphs, const uint4* __restrict__ upd,
                                                   uint32_t count, int multi, const uint32_t* __restrict__ gnext,
                                                   uint32_t* __restrict__ nheads, const uint4* __restrict__ pack,
                                                   uint64_t* totals, const uint32_t* __restrict__ dyn) {
    WaveAcc acc;
    uint64_t grouped = 0;
    if (dyn) {
        upd += dyn[0];
        count = dyn[1];
    }
    if (!pack) {   // no grouping: one wavefront per position
        for (uint32_t i = wave_id(); i < count; i += wave_count()) apply_record(graphs, upd, i, multi, acc);
        acc.flush(totals);
        return;
    }
    const uint32_t n = nheads[2] + nheads[3];
    if (blockIdx.x == 0 && lane() < 2) nheads[lane()] = 0;   // for the next batch's k_group_link
    for (uint32_t j = wave_id(); j < n; j += wave_count())
        apply_edge<false, false>(graphs, upd, multi, gnext, pack, j, acc, grouped);
    acc.flush(totals);
    if (grouped && totals && lane() == 0) tot_add(totals, T_GROUPED, grouped);
}

// ---- four light edges to a wavefront
// An edge with short rows keeps a wavefront's lanes mostly idle, and the chip
// runs out of wavefront slots long before it runs out of anything else: the
// update is a chain of some eight dependent loads and atomics.  So a
// wavefront takes four such edges at once, 16 lanes each: 8 lanes on the first
// endpoint's row (x = u) and 8 on the second's (x = v), each lane holding its
// own endpoint's values.  One lane a row (the lead) claims the slot and writes
// the marks, the bitmap and the histogram.  Selecting a colour stays the whole
// wavefront's work, for one edge after another.  The steps of an update and
// their order are apply_update's.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t x) {   // a lane exchange within 16 lanes
    return (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, CTRL, 0xF, 0xF, false);
}
__device__ __forceinline__ uint32_t other8(uint32_t x) { return dpp<0x128>(x); }   // the other endpoint's (row_ror:8)
__device__ __forceinline__ uint32_t min8(uint32_t x) {   // over the 8 lanes: quad_perm 1 and 2 apart, row_half_mirror
    uint32_t y = dpp<0xB1>(x);
    x = y < x ? y : x;
    y = dpp<0x4E>(x);
    x = y < x ? y : x;
    y = dpp<0x141>(x);
    return y < x ? y : x;
}
__device__ __forceinline__ uint32_t lead8(uint32_t x) {   // the 8 lanes' first lane's
    const uint32_t q = dpp<0x00>(x), m = dpp<0x141>(q);
    return (lane() & 4u) ? m : q;
}

constexpr uint32_t PAIR_UNROLL = 8, PAIR_SLOTS = 16 * PAIR_UNROLL;   // slots of a row loaded in one round trip

struct LaneCounts {   // of the lane's own edges; summed when the wavefront ends
    uint32_t updates = 0, scan = 0, hd = 0, ovf = 0, grouped = 0;
};

// The packed records of the lane's edge (`mine`: record k in lane k of its 16)
// in stream order, for the edges of graph g that take part (act).
__device__ __forceinline__ void apply_quad(const GraphDev& g, bool act, const uint4& mine, WaveAcc& acc,
                                           LaneCounts& n) {
    const uint32_t l8 = lane() & 7u;
    const bool second = (lane() & 8u) != 0, lead = l8 == 0;
    uint32_t s = 0, cap = 0, hd = INVALID;   // the row's first slot, its slots, the histogram row
    bool sticky = false;
    // The RowHint of a delete that removed both copies (held_x = its x, or INVALID).
    uint32_t held_x = INVALID, held = 0, freed = 0, own = 0, seen = 0;
    for (uint32_t k = 0; k < GROUP_PACK; k++) {
        const int from_lane = (int)((lane() & 48u) + k);
        const uint32_t rx = (uint32_t)__shfl((int)mine.x, from_lane), ry = (uint32_t)__shfl((int)mine.y, from_lane);
        const bool ins = (__shfl((int)mine.z, from_lane) & 0xFF) == 0;
        const bool on = act && rx != PACK_NONE;
        if (!ballot(on)) break;
        const uint32_t x = second ? ry : rx, y = second ? rx : ry;
        const bool hinted = on && ins && held_x == x;
        uint32_t f = 0, w = 0;
        uint64_t bits = ~0ull;
        if (on && !hinted) {
            if (held_x != INVALID && lead) mark(g, held_x, held);
            held_x = INVALID;
            s = gp(g.row_ptr)[x];
            cap = gp(g.row_ptr)[x + 1] - s;
            hd = gp(g.hd_map)[x];
            sticky = g.dirty && gp(g.dirty)[(size_t)M_STICKY * g.dstride + x];
            f = ld(&g.fill[x]);
            if (!ins) {
                w = ld(&g.word[x]);
                bits = ld(&g.bitmap[x]);
            }
        }
        uint32_t pos = 0, pf = 0, open = INVALID;   // as scan_pair's pos, pf, free (here from the row's start)
        bool had = false, run = on;
        if (ballot(hinted)) {   // claim the slots the delete left
            uint32_t old = 0, raised = 0;
            if (hinted && lead) {
                old = cas32(&g.col[freed], INVALID, y);
                raised = max32(&g.fill[x], freed - s + 1);
            }
            old = lead8(old);
            raised = lead8(raised);
            if (hinted) {
                if (freed == own) held &= ~D_ROW;
                if (old == INVALID) {
                    pos = freed - s + 1;
                    pf = raised;
                    run = false;
                } else {   // another wavefront took the slot
                    held |= D_ROW;
                    f = ld(&g.fill[x]);
                }
            }
        }
        const bool scanned = run;
        uint32_t from = 0;   // slots before it were passed
        while (ballot(run)) {   // (from grows with every trip of a row still running)
            // pairs of slots from the even slot at or before `from` (the slot array holds whole pairs)
            const uint32_t a = (s + from) & ~1u, j = a + 2 * l8, left = run && s + f > j ? s + f - j : 0u;
            const uint32_t next = a + PAIR_SLOTS - s;
            const uint64_t none = y ? 0ull : 1ull | 1ull << 32;   // neither y nor free
            uint64_t p[PAIR_UNROLL];
#pragma unroll
            for (uint32_t q = 0; q < PAIR_UNROLL; q++)
                p[q] = 16 * q < left ? ld((const uint64_t*)(g.col + j + 16 * q)) : none;
            uint32_t ok = j < s + from ? ~1u : ~0u;   // a slot before `from`, a slot past the fill
            if (left % 16 == 1 && left / 16 < PAIR_UNROLL) ok &= ~(2u << (2 * (left / 16)));
            uint32_t is_y = 0, is_free = 0;
#pragma unroll
            for (uint32_t q = 0; q < PAIR_UNROLL; q++) {
                const uint32_t lo = (uint32_t)p[q], hi = (uint32_t)(p[q] >> 32);
                is_y |= (uint32_t)(lo == y) << (2 * q) | (uint32_t)(hi == y) << (2 * q + 1);
                is_free |= (uint32_t)(lo == INVALID) << (2 * q) | (uint32_t)(hi == INVALID) << (2 * q + 1);
            }
            is_y &= ok;
            is_free &= ok;
            const uint32_t ky = is_y ? (uint32_t)__builtin_ctz(is_y) : 0u;
            const uint32_t kf = is_free ? (uint32_t)__builtin_ctz(is_free) : 0u;
            uint32_t eq = is_y ? j + 16 * (ky >> 1) + (ky & 1u) - s : INVALID;
            uint32_t fr = is_free ? j + 16 * (kf >> 1) + (kf & 1u) - s : INVALID;
            eq = min8(eq);
            fr = min8(fr);
            open = fr < open ? fr : open;
            bool claim = false;
            uint32_t at = 0;
            if (run && ins) {   // the first slot that is free or holds y; past the fill every slot is free
                uint32_t first = eq < fr ? eq : fr;
                if (first == INVALID && next >= f) first = f;
                if (first == INVALID) {
                    from = next;
                } else if (first == eq) {
                    pos = eq + 1;
                    had = true;
                    run = false;
                } else if (first >= cap) {
                    run = false;   // the row is full
                } else {
                    claim = true;
                    at = first;
                }
            } else if (run) {
                claim = eq != INVALID;
                at = eq;
                if (!claim) {
                    from = next;
                    run = from < f;
                }
            }
            uint32_t old = 0, raised = 0;
            if (claim && lead) {
                old = cas32(&g.col[s + at], ins ? INVALID : y, ins ? y : INVALID);
                if (ins) raised = max32(&g.fill[x], at + 1);
            }
            old = lead8(old);
            raised = lead8(raised);
            if (claim) {
                const bool won = old == (ins ? INVALID : y);
                if (won || (ins && old == y)) {
                    pos = at + 1;
                    pf = ins && won ? raised : 0u;
                    had = ins && !won;
                    run = false;
                } else {   // another wavefront took the slot: go on after it
                    from = at + 1;
                    if (ins) {
                        const uint32_t now = ld(&g.fill[x]);
                        f = now > from ? now : from;
                    } else {
                        run = from < f;
                    }
                }
            }
        }
        const uint32_t pos2 = other8(pos);
        // ---- delete: marks, histogram, whether its colour may fall
        const uint32_t c1 = color_of(w), o1 = other8(c1);
        bool reduce = false;
        if (on && !ins) {
            const uint32_t m = (pos ? D_ROW : 0u) | ((hd == INVALID) == (pos != 0) ? D_BITS : 0u);
            if (pos && pos2) {
                held_x = x;
                held = m;
                own = s + pos - 1;
                freed = s + (open < pos - 1 ? open : pos - 1);
                seen = o1;
            } else if (lead) {
                mark(g, x, m);
            }
            if (lead) {
                if (hd != INVALID && o1 != 0 && o1 <= HIST_BINS)
                    add32(&g.hist[(size_t)hd * HIST_BINS + o1 - 1], 0xFFFFFFFFu);
                n.scan += pos ? pos : f;
            }
            // try_reduce, up to where it selects a colour
            reduce = c1 != 0 && o1 < c1 &&
                     !(hd == INVALID && ~bits && (uint32_t)__builtin_ctzll(~bits) + 1u >= c1);
        }
        // ---- insert: a second copy of the edge, overflow, marks, colours
        if (ballot(on && ins)) {
            const bool add = on && ins;
            const bool had2 = other8(had) != 0, sticky2 = other8(sticky) != 0, scanned2 = other8(scanned) != 0;
            const uint32_t tail = pf > pos ? pf - pos : 0u, tail2 = other8(tail);
            // (apply_update says which row has to be searched for a second copy)
            bool dup = false, look = false;
            if (add && !(sticky && sticky2) && !(hinted && !scanned && !scanned2)) {
                if (pos && pos2) {
                    dup = had != had2;
                    look = !had && !had2 && tail && (second ? tail < tail2 : tail <= tail2);
                } else {
                    look = pos && tail;
                }
            }
            for (uint32_t b = pos; ballot(look); b += 8 * PAIR_UNROLL) {
                uint32_t val[PAIR_UNROLL];
                bool any = false;
#pragma unroll
                for (uint32_t q = 0; q < PAIR_UNROLL; q++) {
                    const uint32_t j = b + 8 * q + l8;
                    val[q] = look && j < pf ? ld(&g.col[s + j]) : INVALID;
                }
#pragma unroll
                for (uint32_t q = 0; q < PAIR_UNROLL; q++) any |= val[q] == y;
                const bool found = ((ballot(any) >> (lane() & 56u)) & 0xFFu) != 0;
                dup |= look && found;
                look = look && !found && b + 8 * PAIR_UNROLL < pf;
            }
            const bool dup2 = other8(dup) != 0;
            uint32_t now = 0;
            if (add) {
                if (lead) {
                    if (!second && (dup || dup2)) {
                        add32(&g.ctr[C_ASYM], 1u);
                        mark_sticky(g, x);
                        mark_sticky(g, y);
                    }
                    if (!pos) {   // overflow (finish_insert)
                        add32(&g.ctr[C_ASYM], 1u);
                        const uint32_t at = add32(&g.ctr[C_OVF], 1u);
                        if (at < g.ovf_cap) {
                            st(&g.ovf[2 * (size_t)at], x);
                            st(&g.ovf[2 * (size_t)at + 1], y);
                        }
                        mark_sticky(g, x);
                        mark_sticky(g, y);
                        n.ovf++;
                    }
                    n.scan += pos ? pos : cap;
                    if (had) mark(g, x, D_BITS);
                }
                now = ld(&g.word[x]);
            }
            const uint32_t c = color_of(now), o = other8(c);
            const bool odd = add && (c == 0 || o == 0 || c == o);   // colours to select or to settle
            if (hinted) {   // the delete's marks, less what the re-insert undid
                if (o == seen) held &= ~D_BITS;
                if (lead) mark(g, x, held);
                held_x = INVALID;
            }
            if (add && !odd && lead) {   // on_new_neighbor
                if (o <= 64) or64(&g.bitmap[x], 1ull << (o - 1));
                if (hd != INVALID && o <= HIST_BINS) add32(&g.hist[(size_t)hd * HIST_BINS + o - 1], 1u);
            }
            for (uint64_t todo = ballot(odd && lead && !second); todo; todo &= todo - 1) {
                const uint32_t i = (uint32_t)__builtin_ctzll(todo);
                insert_colours(g, __builtin_amdgcn_readlane(x, i), __builtin_amdgcn_readlane(y, i),
                               __builtin_amdgcn_readlane(hd, i), __builtin_amdgcn_readlane(hd, i + 8),
                               (uint16_t)__builtin_amdgcn_readlane(c, i), (uint16_t)__builtin_amdgcn_readlane(o, i),
                               acc);
            }
        }
        // The reductions come last: a recolour between an insert's slot writes and
        // its read of the words would tell the new neighbour of the change, and the
        // insert would count the new colour there a second time.
        for (uint64_t todo = ballot(reduce && lead); todo; todo &= todo - 1) {   // u before v
            const uint32_t i = (uint32_t)__builtin_ctzll(todo), z = __builtin_amdgcn_readlane(x, i);
            if (find_color(g, z) < __builtin_amdgcn_readlane(c1, i)) recolor(g, z, acc);
        }
        if (on && lead) {
            n.hd += hd != INVALID;
            if (!second) {
                n.updates++;
                n.grouped += k > 0;
            }
        }
    }
    if (act && held_x != INVALID && lead) mark(g, held_x, held);   // marks of a last delete
}

// One wavefront per heavy edge of the batch, then one per four light ones (if
// they are enough to fill the chip, some 3,000 wavefronts of this kernel: 168
// registers, no scratch).  Bound: the chain of dependent gathers and atomics of
// four edges, over the wavefronts the registers allow.  One edge a wavefront /
// this kernel: 32,768 updates of a 131,072-vertex mesh 57 / 39 us, of a
// 262,139-vertex power-law graph 70 / 49, of a 4M-vertex one 125 / 78 (with LONG),
// 196,608 of 48 graphs 331 / 194.
constexpr uint32_t APPLY_SPREAD = 4096;
template <bool LONG>
__global__ __launch_bounds__(64, 3) void k_apply_quads(const GraphDev* __restrict__ graphs,
                                                       const uint4* __restrict__ upd, int multi,
                                                       const uint32_t* __restrict__ gnext,
                                                       uint32_t* __restrict__ nheads,
                                                       const uint4* __restrict__ pack, uint64_t* totals,
                                                       const uint32_t* __restrict__ dyn) {
    WaveAcc acc;
    uint64_t grouped = 0;
    if (dyn) upd += dyn[0];
    const uint32_t nh = nheads[2], nl = nheads[3];
    if (blockIdx.x == 0 && lane() < 2) nheads[lane()] = 0;   // for the next batch's k_group_link
    const uint32_t per = nl > APPLY_SPREAD ? GROUPS : 1u;
    const uint32_t jobs = nh + (nl + per - 1) / per;
    LaneCounts lanes;
    for (uint32_t job = wave_id(); job < jobs; job += wave_count()) {
        uint32_t j0 = job, whole = 1u;   // first edge; which of the (up to four) edges the whole wavefront takes
        if (per > 1 && job >= nh) {
            j0 = nh + (job - nh) * per;
            const uint32_t j = j0 + lane() / GROUP;
            const bool have = j < nh + nl;
            uint4 mine = make_uint4(PACK_NONE, PACK_END, 0u, 0u);
            if (have && sublane() < GROUP_PACK) mine = pack[(size_t)j * GROUP_PACK + sublane()];
            const int first = (int)(lane() & 48u);
            const uint32_t x = (uint32_t)__shfl((int)mine.x, first), y = (uint32_t)__shfl((int)mine.y, first);
            const uint32_t gid = multi ? (uint32_t)__shfl((int)mine.w, first) : 0u;
            // groups longer than the line and self-loops take the whole wavefront, and ablations
            bool quad = have && x != PACK_NONE && x != y;
            whole = 0;
            for (uint64_t pend = ballot(quad); pend;) {   // one graph after another
                const uint32_t g0 = __builtin_amdgcn_readlane(gid, (uint32_t)__builtin_ctzll(pend));
                const bool in = quad && gid == g0;
                pend &= ~ballot(in);
                const GraphDev g = graphs[g0];
                if (g.flags) quad = quad && !in;
                else apply_quad(g, in, mine, acc, lanes);
            }
            const uint64_t left = ballot(have && !quad && sublane() == 0);
            for (uint32_t i = 0; i < GROUPS; i++) whole |= (uint32_t)((left >> (GROUP * i)) & 1u) << i;
        }
        for (; whole; whole &= whole - 1)
            apply_edge<true, LONG>(graphs, upd, multi, gnext, pack, j0 + (uint32_t)__builtin_ctz(whole), acc, grouped);
    }
    if (per > 1) {
        acc.updates += wave_sum32(lanes.updates);
        acc.scan += wave_sum32(lanes.scan);
        acc.hd += wave_sum32(lanes.hd);
        acc.ovf += wave_sum32(lanes.ovf);
        grouped += wave_sum32(lanes.grouped);
    }
    acc.flush(totals);
    if (grouped && totals && lane() == 0) tot_add(totals, T_GROUPED, grouped);
}

// One block per segment, the segment's updates in stream order (deterministic
// mode); positions go through `perm` when given (per-graph order inside a
// mixed batch).  One wavefront replaying a segment spends its time on one
// update's chain of dependent loads at a time (2.6 us an update, whatever the
// graph's size), so the block's WAVES wavefronts take the next WAVES updates
// and judge each at once, reading only (replay_judge): an update is plain if it
// changes no word and finds room in both rows, whatever the plain updates
// before it in the window do.  Plain updates touch nothing but their own
// endpoints' rows, fills, bitmaps, histograms and marks, so those before the
// first that is not plain run a wavefront each, in rounds: an update waits only
// for the earlier ones that share an endpoint with it.  The first that is not
// plain then runs alone.  The result is the one-at-a-time replay's, slot for
// slot.  After a window whose first update was not plain (a stream that colours
// fresh vertices), wavefront 0 applies the next updates alone, twice as many
// after each such window up to REPLAY_ALONE, so that a stream with nothing to
// run together pays for few judgements.  Measured against one wavefront a
// segment: 509 updates of a 16,384-vertex mesh with their epoch step 1,420 ->
// 425 us; 48 graphs of 2^10..2^14 vertices, 71K updates, 11.1 -> 4.7 ms.
constexpr uint32_t REPLAY_WAVES = 16;    // 4 wavefronts per SIMD, what one update's registers allow
constexpr uint32_t REPLAY_CHUNK = 256;   // records staged in LDS at a time
constexpr uint32_t REPLAY_ALONE = 64;

template <uint32_t WAVES>
struct ReplayWindow {
    uint4 recs[REPLAY_CHUNK];
    // of each update of the window: its endpoints (INVALID: it changes nothing)
    // and their colours, whether it is an insert, the earlier ones it shares an
    // endpoint with, whether it is plain
    uint32_t end[2 * WAVES], col[2 * WAVES], ins[WAVES], after[WAVES], plain[WAVES];
};

// Whether the removal of a neighbour coloured `freed` leaves vertex x (colour
// cur) its colour, after the window's earlier updates of x (a lane each: they
// take or give a neighbour coloured `other`; `mine` says which lanes).
// Bitmap mode: no bit below cur is clear (bits are only ever added) and a bit
// stays clear whatever the earlier inserts add.  Histogram mode: no bin below
// cur's that is or becomes zero.
__device__ __forceinline__ bool keeps_colour(const GraphDev& g, uint32_t hd, uint64_t bits, uint16_t freed,
                                             uint16_t cur, uint64_t mine, uint64_t inserts, uint32_t other) {
    if (cur == 0 || freed >= cur) return true;   // try_reduce does nothing
    if (hd == INVALID || (g.flags & ABL_FORCE_BITMAP))
        return (uint32_t)__builtin_popcountll(~bits) > (uint32_t)__builtin_popcountll(inserts) &&
               (uint32_t)__builtin_ctzll(~bits) + 1u >= cur;
    if (cur > HIST_BINS) return false;
    const uint32_t* h = g.hist + (size_t)hd * HIST_BINS;
    for (uint32_t k = 0; k + 1 < cur; k += WAVE) {
        const uint32_t c = k + lane() + 1;
        uint32_t left = c < cur ? ld(&h[c - 1]) - (c == freed ? 1u : 0u) : 1u;
        for (uint64_t m = mine; m; m &= m - 1) {
            const uint32_t i = (uint32_t)__builtin_ctzll(m);
            const uint32_t at = __builtin_amdgcn_readlane(other, i);
            if (c < cur && at == c) left += (inserts >> i) & 1 ? 1u : 0xFFFFFFFFu;
        }
        if (ballot(left == 0)) return false;
    }
    return true;
}

// Judge the window's update of wavefront wv (every wavefront of the block calls it).
template <uint32_t WAVES>
__device__ __forceinline__ void replay_judge(const GraphDev& g, const uint4& r, bool have, uint32_t wv,
                                             ReplayWindow<WAVES>& w) {
    const uint32_t u = r.x, v = r.y, type = r.z & 0xFFu;
    const bool none = !have || u >= g.n || v >= g.n || type > 1;   // touches no vertex
    uint32_t room_u = 0, room_v = 0, hu = INVALID, hv = INVALID, wu = 0, wv0 = 0, fu = 0, fv = 0;
    uint64_t bu = 0, bv = 0;
    if (!none) {
        room_u = gp(g.row_ptr)[u + 1] - gp(g.row_ptr)[u], room_v = gp(g.row_ptr)[v + 1] - gp(g.row_ptr)[v];
        hu = gp(g.hd_map)[u], hv = gp(g.hd_map)[v];
        wu = ld(&g.word[u]), wv0 = ld(&g.word[v]);
        fu = ld(&g.fill[u]), fv = ld(&g.fill[v]);
        bu = ld(&g.bitmap[u]), bv = ld(&g.bitmap[v]);
    }
    const uint16_t cu = color_of(bcast0(wu)), cv = color_of(bcast0(wv0));
    if (lane() == 0) {
        w.end[2 * wv] = none ? INVALID : u;
        w.end[2 * wv + 1] = none ? INVALID : v;
        w.col[2 * wv] = cu;
        w.col[2 * wv + 1] = cv;
        w.ins[wv] = type == 0;
    }
    __syncthreads();
    // lane i: the window's update i, if it comes before this one
    const bool before = lane() < wv && !none;
    const uint32_t i = before ? lane() : 0;
    const uint32_t iu = w.end[2 * i], iv = w.end[2 * i + 1];
    const bool at_u = before && iu != INVALID && (iu == u || iv == u);
    const bool at_v = before && iu != INVALID && (iu == v || iv == v);
    const uint64_t mu = ballot(at_u), mv = ballot(at_v), mi = ballot(before && w.ins[i] != 0);
    bool ok = have;
    if (!none) {
        if (u == v) {
            ok = false;
        } else if (type == 0) {
            ok = cu != 0 && cv != 0 && cu != cv && bcast0(fu) + (uint32_t)__builtin_popcountll(mu & mi) < bcast0(room_u) &&
                 bcast0(fv) + (uint32_t)__builtin_popcountll(mv & mi) < bcast0(room_v);
        } else {
            const uint32_t ou = iu == u ? w.col[2 * i + 1] : w.col[2 * i];   // the other endpoint's colour
            const uint32_t ov = iu == v ? w.col[2 * i + 1] : w.col[2 * i];
            ok = keeps_colour(g, hu, bu, cv, cu, mu, mu & mi, ou) && keeps_colour(g, hv, bv, cu, cv, mv, mv & mi, ov);
        }
    }
    if (lane() == 0) {
        w.after[wv] = (uint32_t)(mu | mv);
        w.plain[wv] = ok ? 1u : 0u;
    }
    __syncthreads();
}

template <uint32_t WAVES>
__global__ __launch_bounds__(WAVES * WAVE) void k_apply_seg(const GraphDev* __restrict__ graphs,
                                                           const uint4* __restrict__ upd,
                                                           const uint32_t* __restrict__ seg, uint32_t nseg,
                                                           const uint32_t* __restrict__ perm, int multi,
                                                           uint64_t* totals, const uint32_t* __restrict__ dyn) {
    __shared__ ReplayWindow<WAVES> w;
    WaveAcc acc;
    if (dyn) {   // segments of the current round (absolute stream positions); none when its count is 0
        if (dyn[1] == 0) return;
        seg += dyn[2];
    }
    const uint32_t wv = bcast0(threadIdx.x / WAVE);
    for (uint32_t k = blockIdx.x; k < nseg; k += gridDim.x) {
        uint32_t alone = 0, backoff = 1;
        const uint32_t first = seg[2 * k], last = seg[2 * k + 1];
        for (uint32_t base = first; base < last; base += REPLAY_CHUNK) {
            const uint32_t cnt = last - base < REPLAY_CHUNK ? last - base : REPLAY_CHUNK;
            __syncthreads();   // the chunk before is done with
            for (uint32_t t = threadIdx.x; t < cnt; t += WAVES * WAVE)
                w.recs[t] = upd[perm ? perm[base + t] : base + t];
            __syncthreads();
            for (uint32_t i0 = 0; i0 < cnt;) {   // (block-uniform)
                uint32_t stop = 0, run = 1;      // `stop` updates in rounds, then `run` one after the other
                if (WAVES == 1) {
                    run = cnt - i0;
                } else if (alone) {
                    run = alone < cnt - i0 ? alone : cnt - i0;
                    alone -= run;
                } else if (cnt - i0 > 1) {
                    const bool have = i0 + wv < cnt;
                    const uint4 r = uniform_rec(w.recs[have ? i0 + wv : i0]);
                    replay_judge(graphs[multi ? r.w : 0u], r, have, wv, w);
                    stop = (uint32_t)__builtin_ctzll(~ballot(lane() < WAVES && w.plain[lane() < WAVES ? lane() : 0]));
                    if (stop == WAVES || i0 + stop == cnt) run = 0;
                    if (stop) {
                        backoff = 1;
                    } else {
                        alone = backoff;
                        backoff = backoff < REPLAY_ALONE ? 2 * backoff : REPLAY_ALONE;
                    }
                }
                // One call site for all: a second copy of the update's code
                // would not stay in the instruction cache beside the first.
                const uint32_t wait = lane() < stop ? w.after[lane()] : 0u;
                uint32_t done = 0;
                const uint32_t all = (1u << stop) - 1u;
                while (done != all || run) {
                    uint32_t at = i0 + wv, mine;
                    if (done != all) {
                        const uint32_t ready = (uint32_t)ballot(lane() < stop && (wait & ~done) == 0) & ~done;
                        mine = (ready >> wv) & 1u;
                        done |= ready;
                    } else {
                        at = i0 + stop;
                        mine = wv == 0 ? run : 0u;
                        i0 += run;
                        run = 0;
                    }
                    for (uint32_t i = at; i < at + mine; i++)   // (long scans: the order is the stream's anyway)
                        apply_rec<true>(graphs, uniform_rec(w.recs[i]), multi, acc);
                    __syncthreads();
                }
                i0 += stop;
            }
        }
    }
    acc.flush(totals);
}

// ---------------------------------------------------------------- per-graph control
__global__ void k_zero_ctr(const GraphDev* __restrict__ graphs, uint32_t ng, const uint32_t* __restrict__ active,
                           uint32_t idx) {
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid < ng && (!active || active[gid])) gp(graphs[gid].ctr)[idx] = 0;
}

// Maximum colour per graph into ctr[C_MAXC] (A/src/streamgc.cu:549-553).
__global__ __launch_bounds__(256) void k_max_color(const GraphDev* __restrict__ graphs, Space sp) {
    uint32_t cur = NONE, mx = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < sp.total; i += gridDim.x * blockDim.x) {
        uint32_t gid, v;
        sp.locate(i, gid, v);
        if (gid != cur) {
            if (cur != NONE && mx) max32(&graphs[cur].ctr[C_MAXC], mx);
            cur = gid;
            mx = 0;
        }
        const uint32_t c = color_of(gp(graphs[gid].word)[v]);
        mx = c > mx ? c : mx;
    }
    const uint32_t c0 = bcast0(cur);
    if (ballot(cur != c0) == 0) {              // the whole wave on one graph: one atomic
        mx = wave_max32(mx);
        if (lane() == 0 && cur != NONE && mx) max32(&graphs[cur].ctr[C_MAXC], mx);
    } else if (cur != NONE && mx) {
        max32(&graphs[cur].ctr[C_MAXC], mx);
    }
}

// One graph: 4 words per 16-byte read, a block-wide maximum, one atomic per
// block (thousands of waves folding into one counter serialise on it).
__global__ __launch_bounds__(256) void k_max_color1(const GraphDev* __restrict__ graphs, Space sp) {
    __shared__ uint32_t part[BLOCK / WAVE];
    const uint32_t gid = sp.gid ? sp.gid[0] : 0u;
    const GraphDev g = graphs[gid];
    const uint32_t quads = g.n / 4;
    uint32_t mx = 0;
    for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < quads; q += gridDim.x * blockDim.x) {
        const uint4 w = *reinterpret_cast<const uint4*>(g.word + 4 * (size_t)q);
        const uint32_t a = color_of(w.x) > color_of(w.y) ? color_of(w.x) : color_of(w.y);
        const uint32_t b = color_of(w.z) > color_of(w.w) ? color_of(w.z) : color_of(w.w);
        mx = a > mx ? a : mx;
        mx = b > mx ? b : mx;
    }
    if (blockIdx.x == 0 && threadIdx.x < g.n % 4) {
        const uint32_t c = color_of(gp(g.word)[4 * quads + threadIdx.x]);
        mx = c > mx ? c : mx;
    }
    mx = wave_max32(mx);
    if (lane() == 0) part[threadIdx.x / WAVE] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (uint32_t k = 0; k < BLOCK / WAVE; k++) t = part[k] > t ? part[k] : t;
        if (t) max32(&g.ctr[C_MAXC], t);
    }
}

// ---------------------------------------------------------------- snapshot
// A/src/kernels/epoch_maintenance.cu:5-16, into the back buffer.  In a
// captured round (fl_round and hist set) the same colours also go to the
// graph's next history slot, if it keeps a history and has one free, so the
// snapshot is not read back for it.
__device__ __forceinline__ SGC_G uint16_t* history_slot(const uint32_t* fl_round, const HistDev* hist, uint32_t gid,
                                                       uint32_t n) {
    if (!hist || !fl_round[gid]) return nullptr;
    const HistDev h = hist[gid];
    return h.base && h.count < h.cap ? gp(h.base + (size_t)h.count * n) : nullptr;
}

// One graph: each thread copies the colours of 4 consecutive vertices (one
// 16-byte read of their words; the snapshot half may start at any even
// address, so four 2-byte stores).
__global__ __launch_bounds__(256) void k_snapshot1(const GraphDev* __restrict__ graphs, Space sp,
                                                   const uint32_t* __restrict__ active,
                                                   const uint32_t* __restrict__ fl_round,
                                                   const HistDev* __restrict__ hist) {
    const uint32_t gid = sp.gid ? sp.gid[0] : 0u;
    if (active && !active[gid]) return;
    const GraphDev g = graphs[gid];
    SGC_G uint16_t* out = gp(g.snap_write);
    SGC_G uint16_t* keep = history_slot(fl_round, hist, gid, g.n);
    const uint32_t quads = g.n / 4;
    for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < quads; q += gridDim.x * blockDim.x) {
        const uint4 w = *reinterpret_cast<const uint4*>(g.word + 4 * (size_t)q);
        const uint16_t c0 = color_of(w.x), c1 = color_of(w.y), c2 = color_of(w.z), c3 = color_of(w.w);
        out[4 * q] = c0;
        out[4 * q + 1] = c1;
        out[4 * q + 2] = c2;
        out[4 * q + 3] = c3;
        if (keep) {
            keep[4 * q] = c0;
            keep[4 * q + 1] = c1;
            keep[4 * q + 2] = c2;
            keep[4 * q + 3] = c3;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < g.n % 4) {
        const uint32_t v = 4 * quads + threadIdx.x;
        const uint16_t c = color_of(gp(g.word)[v]);
        out[v] = c;
        if (keep) keep[v] = c;
    }
}

__global__ __launch_bounds__(256) void k_snapshot(const GraphDev* __restrict__ graphs, Space sp,
                                                  const uint32_t* __restrict__ active,
                                                  const uint32_t* __restrict__ fl_round,
                                                  const HistDev* __restrict__ hist) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < sp.total; i += gridDim.x * blockDim.x) {
        uint32_t gid, v;
        sp.locate(i, gid, v);
        if (active && !active[gid]) continue;
        const GraphDev& g = graphs[gid];
        const uint16_t c = color_of(gp(g.word)[v]);
        gp(g.snap_write)[v] = c;
        SGC_G uint16_t* keep = history_slot(fl_round, hist, gid, g.n);
        if (keep) keep[v] = c;
    }
}

// ---------------------------------------------------------------- compaction
// A/src/kernels/epoch_maintenance.cu:20-61: stable left-pack of the live
// slots, free slots after them.

// A block barrier for data in LDS: outstanding global loads and stores go on
// across it (__syncthreads waits for them).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One long row, all threads of the block, windows of COMPACT_WINDOW slots: the
// live slots of each 64-slot chunk are counted by ballot, one lane of each
// wavefront adds up a chunk's place, and the live values move there.  A value
// moves down or stays, and only to slots below its window's end, which every
// wavefront has read by then (it counted them), so the next window's loads are
// in flight meanwhile; slots past the live ones are freed once, at the end.
// Returns the live count; the row's fill becomes it.
// A long row is one block's chain of windows, and the longest row ends the
// launch; with 1,024 slots a window and every store waited for, a window took
// 1.1 us.  Compaction after 32,768 updates of dense growth on a 2^18-vertex
// R-MAT graph (longest row 32K slots) 44 -> 28 us, of churn on the 4M-vertex
// power-law graph (14K slots) 19.8 -> 16.
constexpr uint32_t COMPACT_PER = 16, COMPACT_WINDOW = COMPACT_PER * BLOCK;
__device__ __forceinline__ uint32_t compact_row_block(const GraphDev& g, uint32_t v) {
    static_assert(COMPACT_PER * (BLOCK / WAVE) == WAVE, "one lane a chunk");
    __shared__ uint32_t part[2][WAVE];   // live slots of the window's chunks, in slot order
    const uint64_t lt_mask = (1ull << lane()) - 1ull;
    const uint32_t s = gp(g.row_ptr)[v], e = s + gp(g.fill)[v];
    const uint32_t wv = bcast0(threadIdx.x / WAVE);
    uint32_t w = s, buf = 0, next[COMPACT_PER];
#pragma unroll
    for (uint32_t q = 0; q < COMPACT_PER; q++) {
        const uint32_t j = s + q * BLOCK + threadIdx.x;
        next[q] = j < e ? gp(g.col)[j] : INVALID;
    }
    for (uint32_t base = s; base < e; base += COMPACT_WINDOW, buf ^= 1u) {
        uint32_t val[COMPACT_PER];
#pragma unroll
        for (uint32_t q = 0; q < COMPACT_PER; q++) val[q] = next[q];
        uint32_t mine = 0;   // lane q: the live slots of the wavefront's chunk q
#pragma unroll
        for (uint32_t q = 0; q < COMPACT_PER; q++) {
            const uint32_t n = (uint32_t)__builtin_popcountll(ballot(val[q] != INVALID));
            mine = lane() == q ? n : mine;
        }
        if (lane() < COMPACT_PER) part[buf][lane() * (BLOCK / WAVE) + wv] = mine;
#pragma unroll
        for (uint32_t q = 0; q < COMPACT_PER; q++) {
            const uint32_t j = base + COMPACT_WINDOW + q * BLOCK + threadIdx.x;
            next[q] = j < e ? gp(g.col)[j] : INVALID;
        }
        lds_barrier();   // (the other buffer was read before the barrier of the window before)
        const uint32_t x = part[buf][lane()];
        uint32_t inc = x;
        for (uint32_t d = 1; d < WAVE; d <<= 1) {
            const uint32_t y = __shfl_up(inc, d);
            if (lane() >= d) inc += y;
        }
#pragma unroll
        for (uint32_t q = 0; q < COMPACT_PER; q++) {
            const uint32_t j = base + q * BLOCK + threadIdx.x;
            const bool live = val[q] != INVALID;
            const uint32_t pos = w + __builtin_amdgcn_readlane(inc - x, q * (BLOCK / WAVE) + wv) +
                                 (uint32_t)__builtin_popcountll(ballot(live) & lt_mask);
            if (live && pos != j) gp(g.col)[pos] = val[q];
        }
        w += __builtin_amdgcn_readlane(inc, WAVE - 1);
    }
    __syncthreads();   // the moves are done: free what lies past the live slots
    for (uint32_t j = w + threadIdx.x; j < e; j += BLOCK) gp(g.col)[j] = INVALID;
    if (threadIdx.x == 0) gp(g.fill)[v] = w - s;
    __syncthreads();   // (part is used again)
    return w - s;
}

// One row, one wavefront: ROW_UNROLL chunks loaded, then packed in order, in one
// pass that writes only slots whose content changes: a live value moves to w +
// (live lanes before it); a slot whose value moved and that lies past the chunk's
// new write front is freed (a later chunk may refill it, in program order).
__device__ __forceinline__ uint32_t compact_row_wave(const GraphDev& g, uint32_t v) {
    const uint64_t lt_mask = (1ull << lane()) - 1ull;
    const uint32_t s = gp(g.row_ptr)[v], e = s + gp(g.fill)[v];
    uint32_t w = s;
    for (uint32_t base = s; base < e; base += ROW_UNROLL * WAVE) {
        uint32_t val[ROW_UNROLL];
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) {
            const uint32_t j = base + u * WAVE + lane();
            val[u] = j < e ? gp(g.col)[j] : INVALID;
        }
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) {
            const uint32_t j = base + u * WAVE + lane();
            const bool live = val[u] != INVALID;
            const uint64_t m = ballot(live);
            const uint32_t pos = w + (uint32_t)__builtin_popcountll(m & lt_mask);
            const uint32_t w_after = w + (uint32_t)__builtin_popcountll(m);
            if (live && pos != j) gp(g.col)[pos] = val[u];
            if (live && pos != j && j >= w_after) gp(g.col)[j] = INVALID;
            w = w_after;
        }
    }
    if (lane() == 0) gp(g.fill)[v] = w - s;
    return w - s;
}

// Rows of at most GROUP_ROW slots, 16 lanes each: the lane's row of vertex v,
// if `mine` (slots [s, s + f)).  Returns the row's live count.
__device__ __forceinline__ uint32_t compact_row_group(const GraphDev& g, bool mine, uint32_t v, uint32_t s, uint32_t f) {
    uint32_t val[ROW_UNROLL];
#pragma unroll
    for (uint32_t u = 0; u < ROW_UNROLL; u++) {
        const uint32_t j = u * GROUP + sublane();
        val[u] = mine && j < f ? gp(g.col)[s + j] : INVALID;
    }
    uint32_t w = s;
#pragma unroll
    for (uint32_t u = 0; u < ROW_UNROLL; u++) {
        const uint32_t j = s + u * GROUP + sublane();
        const bool live = val[u] != INVALID;
        const uint32_t m = group_bits(ballot(live));
        const uint32_t pos = w + (uint32_t)__builtin_popcount(m & ((1u << sublane()) - 1u));
        const uint32_t w_after = w + (uint32_t)__builtin_popcount(m);
        if (live && pos != j) gp(g.col)[pos] = val[u];
        if (live && pos != j && j >= w_after) gp(g.col)[j] = INVALID;
        w = w_after;
    }
    if (mine && sublane() == 0) gp(g.fill)[v] = w - s;
    return w - s;
}

// The drain's counter snapshot of one graph (A/src/streamgc.cu:972-983): the
// overflow entries it retries (capped at the buffer), those lost past the
// buffer, counters reset.
__device__ __forceinline__ void drain_prep_graph(const GraphDev* __restrict__ graphs, uint32_t gid) {
    SGC_G uint32_t* c = gp(graphs[gid].ctr);
    uint32_t raw = c[C_OVF];
    c[C_OVF_RAW] = raw;
    c[C_OVF_SNAP] = raw < graphs[gid].ovf_cap ? raw : graphs[gid].ovf_cap;
    if (raw > graphs[gid].ovf_cap) c[C_LOST] += raw - graphs[gid].ovf_cap;   // never buffered
    c[C_OVF] = 0;
    c[C_DRAIN_FAILED] = 0;
    c[C_CONFLICTS] = 0;   // for the epoch's first Tier-1 sweep
}

// (256, 8): with more than 64 registers only 7 of a CU's 8 blocks of the usual
// grid run at once, and a full sweep waits for the eighth (327 -> 526 us).  The
// long rows' windows pay for it: 2 vector registers (12 B of scratch a lane) and
// 56 scalar ones are spilled around compact_row_block.
// prep_ng > 0: block 0 also takes the drain's counter snapshot of the
// active graphs (k_drain_prep), which the drain launched next reads;
// compaction touches none of those counters.
// ALONE: a full sweep on a grid with a wavefront for every row (alone_rows).
template <bool ALONE>
__global__ __launch_bounds__(256, 8) void k_compact(const GraphDev* __restrict__ graphs, Space sp, SweepList sl,
                                                 uint64_t* totals, uint32_t prep_ng,
                                                 const uint32_t* __restrict__ prep_active) {
    if (blockIdx.x == 0)
        for (uint32_t gid = threadIdx.x; gid < prep_ng; gid += blockDim.x)
            if (!prep_active || prep_active[gid]) drain_prep_graph(graphs, gid);
    uint64_t live_total = 0, rows = 0, slots = 0;
    if (ALONE) {
        for_each_row(graphs, sp, [&](const GraphDev& g, uint32_t, uint32_t v) {
            slots += gp(g.fill)[v];
            live_total += compact_row_wave(g, v);
            rows++;
        });
        if (lane() != 0) live_total = rows = slots = 0;
        block_add64(totals, T_LIVE_SLOTS, live_total);
        block_add64(totals, T_SWEEP_ROWS + 0, rows);
        block_add64(totals, T_SWEEP_SLOTS + 0, slots);
        return;
    }
    const uint32_t nbig = sweep_big(sl);
    for (uint32_t k = blockIdx.x; k < nbig; k += gridDim.x) {
        uint32_t gid, v;
        sp.locate(big_item(sl, k), gid, v);
        const GraphDev& g = graphs[gid];
        const uint32_t f = gp(g.fill)[v];
        const uint32_t live = compact_row_block(g, v);
        if (threadIdx.x == 0) {
            live_total += live;
            rows++;
            slots += f;
        }
    }
    uint32_t row_n = 0, slot_n = 0, live_n = 0;   // of the lane's rows (one lane of the row counts)
    for_rows(graphs, sp, sl, [&](const GraphDev& g, uint32_t, bool mine, uint32_t v) {
        const uint32_t f = mine ? gp(g.fill)[v] : 0u, s = mine ? gp(g.row_ptr)[v] : 0u;
        const bool one = mine && sublane() == 0, few = f <= GROUP_ROW;
        const uint32_t live = compact_row_group(g, mine && few, v, s, f);
        row_n += one;
        slot_n += one ? f : 0u;
        live_n += one && few ? live : 0u;
        each_row(ballot(one && !few), v, [&](uint32_t x) {
            const uint32_t n = compact_row_wave(g, x);
            live_n += lane() == 0 ? n : 0u;
        });
    });
    rows += wave_sum32(row_n);
    slots += wave_sum32(slot_n);
    live_total += wave_sum32(live_n);
    if (lane() != 0) live_total = rows = slots = 0;
    block_add64(totals, T_LIVE_SLOTS, live_total);
    block_add64(totals, T_SWEEP_ROWS + 0, rows);
    block_add64(totals, T_SWEEP_SLOTS + 0, slots);
}

// ---------------------------------------------------------------- overflow drain
// A/src/streamgc.cu:972-983: read the counter, reset it, clamp to capacity.
__global__ void k_drain_prep(const GraphDev* __restrict__ graphs, uint32_t ng, const uint32_t* __restrict__ active) {
    uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= ng || (active && !active[gid])) return;
    drain_prep_graph(graphs, gid);
}

// A/src/kernels/epoch_maintenance.cu:66-87: one wavefront per entry, graph = blockIdx.y.
__global__ __launch_bounds__(256) void k_drain_elem(const GraphDev* __restrict__ graphs,
                                                    const uint32_t* __restrict__ active) {
    const uint32_t gid = blockIdx.y;
    if (active && !active[gid]) return;
    const GraphDev g = graphs[gid];
    const uint32_t count = gp(g.ctr)[C_OVF_SNAP];
    uint32_t failed = 0;
    for (uint32_t k = wave_id(); k < count; k += wave_count()) {
        bool f = false;
        const uint32_t x = gp(g.ovf)[2 * (size_t)k];
        row_insert(g, x, gp(g.ovf)[2 * (size_t)k + 1], false, &f, nullptr);
        if (lane() == 0 && x < g.n) mark(g, x, D_BITS | D_STATUS);
        failed += f;
    }
    if (failed && lane() == 0) {
        add32(&g.ctr[C_DRAIN_FAILED], failed);
        add32(&g.ctr[C_LOST], failed);
    }
}

// The same in buffer order, one wavefront per graph (deterministic mode).
__global__ __launch_bounds__(64) void k_drain_serial(const GraphDev* __restrict__ graphs, uint32_t ng,
                                                     const uint32_t* __restrict__ active) {
    for (uint32_t gid = blockIdx.x; gid < ng; gid += gridDim.x) {
        if (active && !active[gid]) continue;
        const GraphDev g = graphs[gid];
        const uint32_t count = gp(g.ctr)[C_OVF_SNAP];
        uint32_t failed = 0;
        for (uint32_t k = 0; k < count; k++) {
            bool f = false;
            const uint32_t x = gp(g.ovf)[2 * (size_t)k];
            row_insert(g, x, gp(g.ovf)[2 * (size_t)k + 1], false, &f, nullptr);
            if (lane() == 0 && x < g.n) mark(g, x, D_BITS | D_STATUS);
            failed += f;
        }
        if (lane() == 0) {
            gp(g.ctr)[C_DRAIN_FAILED] = failed;
            gp(g.ctr)[C_LOST] += failed;
        }
    }
}

// ---------------------------------------------------------------- bitmap / histogram rebuild
// A/include/color_select.cuh:213-251, A/src/kernels/epoch_maintenance.cu:113-128:
// bitmap-mode rows get the exact OR of their live neighbours' colours <= 64.
// Exact-histogram mode also recounts every hub's 1024 counters from its live
// row (colours 1..1024): one wavefront per hub, the bins in that wavefront's
// own 4 KiB of LDS, written out as 16 coalesced dwords per lane.  The
// reference never rebuilds histograms (A/src/kernels/epoch_maintenance.cu:120-123),
// so its counts drift; this mode keeps them exact at every rebuild.
// A long hub row: the whole block counts into one shared 1024-bin tile.
__device__ __forceinline__ void rebuild_hub_block(const GraphDev& g, uint32_t v, uint32_t hd, uint32_t* bins) {
    for (uint32_t t = threadIdx.x; t < HIST_BINS; t += BLOCK) bins[t] = 0;
    __syncthreads();
    const uint32_t s = gp(g.row_ptr)[v], e = s + gp(g.fill)[v];
    for (uint32_t base = s; base < e; base += ROW_UNROLL * BLOCK) {
        uint32_t nb[ROW_UNROLL], c[ROW_UNROLL];
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) {
            const uint32_t j = base + u * BLOCK + threadIdx.x;
            nb[u] = j < e ? gp(g.col)[j] : INVALID;
        }
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) c[u] = (nb[u] != INVALID && nb[u] < g.n) ? color_of(gp(g.word)[nb[u]]) : 0;
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++)
            if (c[u] != 0 && c[u] <= HIST_BINS) atomicAdd(&bins[c[u] - 1], 1u);
    }
    __syncthreads();
    SGC_G uint32_t* dst = gp(g.hist) + (size_t)hd * HIST_BINS;
    for (uint32_t t = threadIdx.x; t < HIST_BINS; t += BLOCK) dst[t] = bins[t];
    __syncthreads();
}

// A hub row by one wavefront, into its own 1024-bin tile.
__device__ __forceinline__ void rebuild_hub_wave(const GraphDev& g, uint32_t v, uint32_t* b) {
    const uint32_t s = gp(g.row_ptr)[v], e = s + gp(g.fill)[v];
    for (uint32_t t = lane(); t < HIST_BINS; t += WAVE) b[t] = 0;
    __builtin_amdgcn_wave_barrier();
    for (uint32_t base = s; base < e; base += ROW_UNROLL * WAVE) {
        uint32_t nb[ROW_UNROLL], c[ROW_UNROLL];
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) {
            const uint32_t j = base + u * WAVE + lane();
            nb[u] = j < e ? gp(g.col)[j] : INVALID;
        }
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++)
            c[u] = (nb[u] != INVALID && nb[u] < g.n) ? color_of(gp(g.word)[nb[u]]) : 0;
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++)
            if (c[u] != 0 && c[u] <= HIST_BINS) atomicAdd(&b[c[u] - 1], 1u);
    }
    __builtin_amdgcn_wave_barrier();
    SGC_G uint32_t* dst = gp(g.hist) + (size_t)gp(g.hd_map)[v] * HIST_BINS;
    for (uint32_t t = lane(); t < HIST_BINS; t += WAVE) dst[t] = b[t];
    __builtin_amdgcn_wave_barrier();
}

// Bitmap rows of at most GROUP_ROW slots, 16 lanes each: the lane's row of
// vertex v, if `mine` (slots [s, s + f)).
__device__ __forceinline__ void rebuild_bitmap_group(const GraphDev& g, bool mine, uint32_t v, uint32_t s, uint32_t f) {
    uint32_t nb[ROW_UNROLL];
    uint64_t bm = 0;
#pragma unroll
    for (uint32_t u = 0; u < ROW_UNROLL; u++) {
        const uint32_t j = u * GROUP + sublane();
        nb[u] = mine && j < f ? gp(g.col)[s + j] : INVALID;
    }
#pragma unroll
    for (uint32_t u = 0; u < ROW_UNROLL; u++) {
        const uint32_t c = (nb[u] != INVALID && nb[u] < g.n) ? color_of(gp(g.word)[nb[u]]) : 0;
        if (c != 0 && c <= 64) bm |= 1ull << (c - 1);
    }
    for (uint32_t o = GROUP / 2; o > 0; o >>= 1) bm |= __shfl_xor(bm, o);
    if (mine && sublane() == 0) gp(g.bitmap)[v] = bm;
}

// A bitmap row: the OR of its live neighbours' colours <= 64 (one wavefront,
// or the whole block for a long row).
template <bool kBlock>
__device__ __forceinline__ void rebuild_bitmap(const GraphDev& g, uint32_t v) {
    const uint32_t s = gp(g.row_ptr)[v], e = s + gp(g.fill)[v];
    const uint32_t width = kBlock ? BLOCK : WAVE, me = kBlock ? threadIdx.x : lane();
    uint64_t bm = 0;
    for (uint32_t base = s; base < e; base += ROW_UNROLL * width) {
        uint32_t nb[ROW_UNROLL], c[ROW_UNROLL];
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) {
            const uint32_t j = base + u * width + me;
            nb[u] = j < e ? gp(g.col)[j] : INVALID;
        }
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) c[u] = (nb[u] != INVALID && nb[u] < g.n) ? color_of(gp(g.word)[nb[u]]) : 0;
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++)
            if (c[u] != 0 && c[u] <= 64) bm |= 1ull << (c[u] - 1);
    }
    bm = wave_or64(bm);
    if (kBlock) {
        __shared__ uint64_t part[BLOCK / WAVE];
        if (lane() == 0) part[threadIdx.x / WAVE] = bm;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint64_t t = 0;
            for (uint32_t k = 0; k < BLOCK / WAVE; k++) t |= part[k];
            gp(g.bitmap)[v] = t;
        }
        __syncthreads();
    } else if (lane() == 0) {
        gp(g.bitmap)[v] = bm;
    }
}

// A/include/color_select.cuh:213-251, A/src/kernels/epoch_maintenance.cu:113-128:
// bitmap-mode rows get the exact OR of their live neighbours' colours <= 64.
// Exact-histogram mode also recounts every listed hub's 1024 counters from
// its live row (colours 1..1024) in LDS, then writes them out coalesced.  The
// reference never rebuilds histograms (A/src/kernels/epoch_maintenance.cu:120-123),
// so its counts drift; this mode keeps them exact at every rebuild.
__global__ __launch_bounds__(256) void k_rebuild(const GraphDev* __restrict__ graphs, Space sp, SweepList sl,
                                                 int exact_hist, uint64_t* totals) {
    __shared__ uint32_t bins[BLOCK / WAVE][HIST_BINS];
    uint64_t rows = 0, slots = 0;
    const uint32_t nbig = sweep_big(sl);
    for (uint32_t k = blockIdx.x; k < nbig; k += gridDim.x) {
        uint32_t gid, v;
        sp.locate(big_item(sl, k), gid, v);
        const GraphDev& g = graphs[gid];
        const uint32_t hd = gp(g.hd_map)[v];
        if (hd != INVALID && !exact_hist) continue;
        if (threadIdx.x == 0) {
            rows++;
            slots += gp(g.fill)[v];
        }
        if (hd == INVALID) rebuild_bitmap<true>(g, v);
        else rebuild_hub_block(g, v, hd, &bins[0][0]);
    }
    uint32_t* b = bins[threadIdx.x / WAVE];
    uint32_t row_n = 0, slot_n = 0;   // of the lane's rows (one lane of the row counts)
    for_rows(graphs, sp, sl, [&](const GraphDev& g, uint32_t, bool mine, uint32_t v) {
        const uint32_t hd = mine ? gp(g.hd_map)[v] : INVALID;
        const uint32_t f = mine ? gp(g.fill)[v] : 0u, s = mine ? gp(g.row_ptr)[v] : 0u;
        const bool todo = mine && (hd == INVALID || exact_hist), one = todo && sublane() == 0;
        const bool few = hd == INVALID && f <= GROUP_ROW;
        row_n += one;
        slot_n += one ? f : 0u;
        rebuild_bitmap_group(g, todo && few, v, s, f);
        each_row(ballot(one && !few && hd == INVALID), v, [&](uint32_t x) { rebuild_bitmap<false>(g, x); });
        each_row(ballot(one && hd != INVALID), v, [&](uint32_t x) { rebuild_hub_wave(g, x, b); });
    });
    rows += wave_sum32(row_n);
    slots += wave_sum32(slot_n);
    if (lane() != 0) rows = slots = 0;
    block_add64(totals, T_SWEEP_ROWS + 1, rows);
    block_add64(totals, T_SWEEP_SLOTS + 1, slots);
}

// ---------------------------------------------------------------- tier-1 repair
// Colours 1..255 present among a row's live neighbours, bit (c & 63) of
// m[c >> 6].
struct ColourSet {
    uint64_t m[4] = {0, 0, 0, 0};
    __device__ __forceinline__ void add(uint32_t c) {
        if (c == 0 || c >= 256) return;
        const uint64_t b = 1ull << (c & 63);
        const uint32_t q = c >> 6;
        m[0] |= q == 0 ? b : 0;
        m[1] |= q == 1 ? b : 0;
        m[2] |= q == 2 ? b : 0;
        m[3] |= q == 3 ? b : 0;
    }
    __device__ __forceinline__ void wave_reduce() {
        for (int k = 0; k < 4; k++) m[k] = wave_or64(m[k]);
    }
    // find_available_color_bitmap on an exact bitmap: the lowest colour in
    // 1..255 not present, else 256 (A/include/color_select.cuh:20-52).
    __device__ __forceinline__ uint16_t lowest_free() const {
        const uint64_t m0 = m[0] | 1ull;   // colour 0 is not a colour
        if (~m0) return (uint16_t)__builtin_ctzll(~m0);
        for (int k = 1; k < 4; k++)
            if (~m[k]) return (uint16_t)(64 * k + __builtin_ctzll(~m[k]));
        return 256;
    }
};

// Colours 1..1024 present among a hub's live neighbours: 32 words of LDS
// per wavefront (or per block).  The lowest absent colour is what
// find_available_color_histogram picks from an exact histogram
// (A/include/color_select.cuh:59-89); with all 1024 present it falls back to
// the histogram's minimum.
constexpr uint32_t PRESENCE_WORDS = HIST_BINS / 32;
__device__ __forceinline__ void presence_add(uint32_t* p, uint32_t c) {
    if (c != 0 && c <= HIST_BINS) atomicOr(&p[(c - 1) >> 5], 1u << ((c - 1) & 31));
}
// One wavefront reads the 1024 bits: the lowest clear bit, or 0 if none.
__device__ __forceinline__ uint16_t presence_lowest_free(const uint32_t* p) {
    const uint32_t word = lane() < PRESENCE_WORDS ? p[lane()] : 0xFFFFFFFFu;
    const uint64_t open = ballot(word != 0xFFFFFFFFu);
    if (!open) return 0;
    const uint32_t k = (uint32_t)__builtin_ctzll(open);
    const uint32_t wk = (uint32_t)__shfl((int)word, (int)k);
    return (uint16_t)(32 * k + __builtin_ctz(~wk) + 1);
}

__device__ __forceinline__ uint16_t fresh_pick(const GraphDev& g, uint32_t v, bool hub, ColourSet& cs,
                                               const uint32_t* pres) {
    if (!hub) {
        cs.wave_reduce();
        return cs.lowest_free();
    }
    __builtin_amdgcn_wave_barrier();
    const uint16_t c = presence_lowest_free(pres);
    return c ? c : fas_hist(g, gp(g.hd_map)[v]);
}

// A/src/kernels/conflict_repair.cu:10-114 for one vertex; returns 1 if counted.
// Fresh selection (parallel mode): a loser selects from the exact colours of its
// neighbours, gathered by the same row scan that found the conflict -- the
// bitmap or histogram a rebuild at this instant would leave -- instead of
// the ones rebuilt before the sweep, which miss the recolours made earlier in
// the same sweep (the reference does not propagate them,
// A/src/kernels/conflict_repair.cu).  Deterministic mode keeps the
// reference's selection.  pres: this wavefront's PRESENCE_WORDS of LDS.
// fresh: 0 = the reference's selection, 1 = exact colours for bitmap-mode
// rows, 2 = for histogram-mode rows too.
// Live slots of v's row (the ablation's priority degree,
// A/src/kernels/conflict_repair.cu:46-58): one wavefront, or the whole block.
template <bool kBlock>
__device__ __forceinline__ uint32_t live_row_count(const GraphDev& g, uint32_t v) {
    const uint32_t s = gp(g.row_ptr)[v], e = s + ld(&g.fill[v]);
    const uint32_t width = kBlock ? BLOCK : WAVE, me = kBlock ? threadIdx.x : lane();
    uint32_t k = 0;
    for (uint32_t j = s + me; j < e; j += width) k += ld(&g.col[j]) != INVALID;
    return kBlock ? block_sum32(k) : wave_sum32(k);
}

__device__ __forceinline__ uint32_t tier1_vertex(const GraphDev& g, uint32_t v, uint32_t* pres, int fresh_level) {
    const uint32_t w = bcast0(ld(&g.word[v]));
    const uint16_t mine = color_of(w);
    const uint32_t s = gp(g.row_ptr)[v], e = s + ld(&g.fill[v]);
    const bool hub = select_by_hist(g, v);
    const bool fresh = fresh_level >= (hub ? 2 : 1);
    ColourSet cs;
    if (fresh && hub) {
        if (lane() < PRESENCE_WORDS) pres[lane()] = 0;
        __builtin_amdgcn_wave_barrier();
    }
    if (mine == 0) {
        bool has_nb = false;
        for (uint32_t base = s; base < e && (fresh || !has_nb); base += ROW_UNROLL * WAVE) {
            uint32_t nb[ROW_UNROLL];
#pragma unroll
            for (uint32_t u = 0; u < ROW_UNROLL; u++) {
                const uint32_t j = base + u * WAVE + lane();
                nb[u] = j < e ? ld(&g.col[j]) : INVALID;
            }
            bool any = false;
#pragma unroll
            for (uint32_t u = 0; u < ROW_UNROLL; u++) {
                any |= nb[u] != INVALID;
                if (fresh && nb[u] != INVALID && nb[u] < g.n) {
                    const uint32_t cn = color_of(ld(&g.word[nb[u]]));
                    if (hub) presence_add(pres, cn);
                    else cs.add(cn);
                }
            }
            has_nb |= ballot(any) != 0;
        }
        if (!has_nb) return 0;
        const uint16_t c = fresh ? fresh_pick(g, v, hub, cs, pres) : find_color(g, v);
        if (lane() == 0) {
            st(&g.word[v], bump(w, c));
            mark(g, v, D_BITS | D_STATUS);
        }
        mark_neighbors(g, v, 0, c);
        return 1;
    }
    const uint32_t my_deg = (g.flags & ABL_LIVE_DEGREE) ? live_row_count<false>(g, v) : gp(g.deg0)[v];
    bool need = false;
    for (uint32_t base = s; base < e && (fresh || !need); base += ROW_UNROLL * WAVE) {
        uint32_t nb[ROW_UNROLL], c[ROW_UNROLL];
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) {
            const uint32_t j = base + u * WAVE + lane();
            nb[u] = j < e ? ld(&g.col[j]) : INVALID;
        }
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++)
            c[u] = (nb[u] != INVALID && nb[u] < g.n) ? color_of(ld(&g.word[nb[u]])) : 0;
        bool hit = false;
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) {
            if (fresh) {
                if (hub) presence_add(pres, c[u]);
                else cs.add(c[u]);
            }
            if (c[u] == mine) {
                const uint32_t d = gp(g.deg0)[nb[u]];
                hit |= (my_deg < d) || (my_deg == d && v < nb[u]);  // pi(v) < pi(nb)
            }
        }
        need |= ballot(hit) != 0;
    }
    if (!need) return 0;
    if (mine <= 64 && lane() == 0) or64(&g.bitmap[v], 1ull << (mine - 1));
    if (fresh && !hub) {   // own colour OR-ed in (A/src/kernels/conflict_repair.cu:105-107)
        if (mine < 64) cs.m[0] |= 1ull << mine;
        if (mine == 64) cs.m[1] |= 1ull;
    }
    const uint16_t c = fresh ? fresh_pick(g, v, hub, cs, pres) : find_color(g, v);
    if (lane() == 0) {
        st(&g.word[v], bump(w, c));
        mark(g, v, D_BITS | D_STATUS);   // its own colour bit was OR-ed in
    }
    mark_neighbors(g, v, mine, c);
    return 1;
}

// The same for a long row, all threads of the block: the verdict is a block
// OR; the first wavefront selects and stores; the block marks the neighbours.
__device__ __forceinline__ uint32_t tier1_vertex_block(const GraphDev& g, uint32_t v, int fresh_level) {
    __shared__ uint32_t pick;
    __shared__ uint64_t sets[BLOCK / WAVE][4];
    __shared__ uint32_t pres[PRESENCE_WORDS];
    const uint32_t w = ld(&g.word[v]);
    const uint16_t mine = color_of(w);
    const uint32_t s = gp(g.row_ptr)[v], e = s + ld(&g.fill[v]);
    const uint32_t my_deg = (g.flags & ABL_LIVE_DEGREE) ? live_row_count<true>(g, v) : gp(g.deg0)[v];
    const bool hub = select_by_hist(g, v);
    const bool fresh = fresh_level >= (hub ? 2 : 1);   // see tier1_vertex
    ColourSet cs;
    uint32_t hit = 0;
    if (fresh && hub) {
        if (threadIdx.x < PRESENCE_WORDS) pres[threadIdx.x] = 0;
        __syncthreads();
    }
    for (uint32_t base = s; base < e; base += ROW_UNROLL * BLOCK) {
        uint32_t nb[ROW_UNROLL], c[ROW_UNROLL];
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) {
            const uint32_t j = base + u * BLOCK + threadIdx.x;
            nb[u] = j < e ? ld(&g.col[j]) : INVALID;
        }
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++)
            c[u] = (nb[u] != INVALID && nb[u] < g.n) ? color_of(ld(&g.word[nb[u]])) : 0;
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) {
            if (fresh && hub) presence_add(pres, c[u]);
            else if (fresh) cs.add(c[u]);
            if (mine == 0) {
                hit |= nb[u] != INVALID;
            } else if (c[u] == mine) {
                const uint32_t d = gp(g.deg0)[nb[u]];
                hit |= (my_deg < d) || (my_deg == d && v < nb[u]);
            }
        }
    }
    if (block_sum32(hit) == 0) return 0;   // (its barrier also completes the presence bits)
    if (fresh && !hub) {
        cs.wave_reduce();
        if (lane() == 0)
            for (int k = 0; k < 4; k++) sets[threadIdx.x / WAVE][k] = cs.m[k];
        __syncthreads();
    }
    if (threadIdx.x < WAVE) {
        if (mine != 0 && mine <= 64 && lane() == 0) or64(&g.bitmap[v], 1ull << (mine - 1));
        uint16_t c;
        if (!fresh) {
            c = find_color(g, v);
        } else if (!hub) {
            ColourSet all;
            for (uint32_t wv = 0; wv < BLOCK / WAVE; wv++)
                for (int k = 0; k < 4; k++) all.m[k] |= sets[wv][k];
            if (mine != 0 && mine < 64) all.m[0] |= 1ull << mine;
            if (mine == 64) all.m[1] |= 1ull;
            c = all.lowest_free();
        } else {
            c = presence_lowest_free(pres);
            if (!c) c = fas_hist(g, gp(g.hd_map)[v]);
        }
        if (lane() == 0) {
            st(&g.word[v], bump(w, c));
            mark(g, v, D_BITS | D_STATUS);
            pick = c;
        }
    }
    __syncthreads();
    const uint16_t c = (uint16_t)pick;
    __syncthreads();
    if (g.dirty) {
        for (uint32_t base = s; base < e; base += ROW_UNROLL * BLOCK) {
            uint32_t nb[ROW_UNROLL], cn[ROW_UNROLL];
#pragma unroll
            for (uint32_t u = 0; u < ROW_UNROLL; u++) {
                const uint32_t j = base + u * BLOCK + threadIdx.x;
                nb[u] = j < e ? ld(&g.col[j]) : INVALID;
            }
#pragma unroll
            for (uint32_t u = 0; u < ROW_UNROLL; u++)
                cn[u] = (nb[u] != INVALID && nb[u] < g.n) ? color_of(ld(&g.word[nb[u]])) : 0;
#pragma unroll
            for (uint32_t u = 0; u < ROW_UNROLL; u++)
                if (nb[u] != INVALID && nb[u] < g.n)
                    mark(g, nb[u], D_BITS | ((cn[u] == mine || cn[u] == c || cn[u] == 0) ? D_STATUS : 0u));
        }
    }
    return 1;
}

// Whether tier1_vertex would repair the lane's coloured vertex v (colour own),
// if `mine`: 16 lanes to a row of at most GROUP_ROW slots, reads only.
__device__ __forceinline__ bool tier1_hit_group(const GraphDev& g, bool mine, uint32_t v, uint32_t s, uint32_t f,
                                                uint32_t own, uint32_t deg) {
    uint32_t nb[ROW_UNROLL];
    bool hit = false;
#pragma unroll
    for (uint32_t u = 0; u < ROW_UNROLL; u++) {
        const uint32_t j = u * GROUP + sublane();
        nb[u] = mine && j < f ? ld(&g.col[s + j]) : INVALID;
    }
    uint32_t c[ROW_UNROLL];
#pragma unroll
    for (uint32_t u = 0; u < ROW_UNROLL; u++)
        c[u] = (nb[u] != INVALID && nb[u] < g.n) ? color_of(ld(&g.word[nb[u]])) : 0u;
#pragma unroll
    for (uint32_t u = 0; u < ROW_UNROLL; u++)
        if (c[u] != 0 && c[u] == own) {
            const uint32_t d = gp(g.deg0)[nb[u]];
            hit |= (deg < d) || (deg == d && v < nb[u]);   // pi(v) < pi(nb)
        }
    return group_bits(ballot(hit)) != 0;
}

template <bool ALONE>
__global__ __launch_bounds__(256) void k_tier1_elem(const GraphDev* __restrict__ graphs, Space sp, SweepList sl,
                                                    int fresh, uint64_t* totals) {
    __shared__ uint32_t presence[BLOCK / WAVE][PRESENCE_WORDS];
    uint64_t rows = 0, slots = 0;
    uint32_t cnt = 0, cur_gid = 0xFFFFFFFFu;
    const auto count_for = [&](uint32_t gid) {   // conflicts counted from here on are graph gid's
        if (gid == cur_gid) return;
        if (cnt && lane() == 0) add32(&graphs[cur_gid].ctr[C_CONFLICTS], cnt);
        cnt = 0;
        cur_gid = gid;
    };
    if (ALONE) {
        for_each_row(graphs, sp, [&](const GraphDev& g, uint32_t gid, uint32_t v) {
            count_for(gid);
            rows++;
            slots += gp(g.fill)[v];
            cnt += tier1_vertex(g, v, presence[threadIdx.x / WAVE], fresh);
        });
        if (cnt && lane() == 0) add32(&graphs[cur_gid].ctr[C_CONFLICTS], cnt);
        if (lane() != 0) rows = slots = 0;
        block_add64(totals, T_SWEEP_ROWS + 2, rows);
        block_add64(totals, T_SWEEP_SLOTS + 2, slots);
        return;
    }
    const uint32_t nbig = sweep_big(sl);
    for (uint32_t k = blockIdx.x; k < nbig; k += gridDim.x) {
        uint32_t gid, v;
        sp.locate(big_item(sl, k), gid, v);
        const GraphDev& g = graphs[gid];
        const uint32_t f = gp(g.fill)[v];
        const uint32_t r = tier1_vertex_block(g, v, fresh);
        if (threadIdx.x == 0) {
            if (r) add32(&g.ctr[C_CONFLICTS], 1u);
            rows++;
            slots += f;
        }
    }
    uint32_t row_n = 0, slot_n = 0;   // of the lane's rows (one lane of the row counts)
    for_rows(graphs, sp, sl, [&](const GraphDev& g, uint32_t gid, bool mine, uint32_t v) {
        count_for(gid);
        const uint32_t f = mine ? ld(&g.fill[v]) : 0u, s = mine ? gp(g.row_ptr)[v] : 0u;
        const uint32_t own = mine ? color_of(ld(&g.word[v])) : 0u, deg = mine ? gp(g.deg0)[v] : 0u;
        const bool one = mine && sublane() == 0;
        row_n += one;
        slot_n += one ? f : 0u;
        // Most listed rows turn out conflict-free: 16 lanes find that, and the
        // wavefront takes only the others (and uncoloured vertices, longer
        // rows, and every row where the live degree decides).
        const bool quick = mine && f <= GROUP_ROW && own != 0 && !(g.flags & ABL_LIVE_DEGREE);
        const bool hit = tier1_hit_group(g, quick, v, s, f, own, deg);
        each_row(ballot(one && (!quick || hit)), v, [&](uint32_t x) {
            cnt += tier1_vertex(g, x, presence[threadIdx.x / WAVE], fresh);
        });
    });
    if (cnt && lane() == 0) add32(&graphs[cur_gid].ctr[C_CONFLICTS], cnt);
    rows += wave_sum32(row_n);
    slots += wave_sum32(slot_n);
    if (lane() != 0) rows = slots = 0;
    block_add64(totals, T_SWEEP_ROWS + 2, rows);
    block_add64(totals, T_SWEEP_SLOTS + 2, slots);
}

// Whether tier1_vertex(g, v) would find v conflict-free (return 0, write
// nothing): uncoloured with no neighbour in its row, or coloured with no
// neighbour of its colour that has the higher priority.  Reads only.
__device__ __forceinline__ bool tier1_clean(const GraphDev& g, uint32_t v) {
    const uint16_t mine = color_of(bcast0(ld(&g.word[v])));
    const uint32_t s = gp(g.row_ptr)[v], e = s + ld(&g.fill[v]);
    uint32_t my_deg = 0;
    if (mine != 0) my_deg = (g.flags & ABL_LIVE_DEGREE) ? live_row_count<false>(g, v) : gp(g.deg0)[v];
    bool bad = false;
    for (uint32_t base = s; base < e && !bad; base += ROW_UNROLL * WAVE) {
        uint32_t nb[ROW_UNROLL], c[ROW_UNROLL];
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) {
            const uint32_t j = base + u * WAVE + lane();
            nb[u] = j < e ? ld(&g.col[j]) : INVALID;
        }
        bool hit = false;
        if (mine == 0) {
#pragma unroll
            for (uint32_t u = 0; u < ROW_UNROLL; u++) hit |= nb[u] != INVALID;
        } else {
#pragma unroll
            for (uint32_t u = 0; u < ROW_UNROLL; u++)
                c[u] = (nb[u] != INVALID && nb[u] < g.n) ? color_of(ld(&g.word[nb[u]])) : 0;
#pragma unroll
            for (uint32_t u = 0; u < ROW_UNROLL; u++) {
                if (c[u] == mine) {
                    const uint32_t d = gp(g.deg0)[nb[u]];
                    hit |= (my_deg < d) || (my_deg == d && v < nb[u]);  // pi(v) < pi(nb)
                }
            }
        }
        bad = ballot(hit) != 0;
    }
    return !bad;
}

// Vertex order per graph (Gauss-Seidel, deterministic), one block per graph.
// With dirty tracking, a vertex is checked only if its check bit is set (or
// it is sticky) when the sweep reaches it; the bits are read again after
// every vertex that changed (a recolour marks neighbours).  A vertex whose
// bit is clear would be found conflict-free, so the sweep changes exactly
// what the full sweep changes.
// The block's SERIAL_WAVES wavefronts take the next SERIAL_WAVES marked
// vertices of the current 1024-vertex chunk and find, at once, which of them
// are conflict-free (tier1_clean, reads only).  Wavefront 0 then goes through
// them in order: a conflict-free vertex changes nothing, so the next one's
// verdict still holds; the first one that is not is checked and repaired
// (tier1_vertex) in the state the sweep would have reached it in, and the
// marks are read again from the vertex after it.  The result is the
// one-vertex-at-a-time sweep's, in fewer round trips when most marked
// vertices turn out clean.
constexpr uint32_t SERIAL_WAVES = 4;
__global__ __launch_bounds__(SERIAL_WAVES * WAVE) void k_tier1_serial(const GraphDev* __restrict__ graphs,
                                                                     uint32_t ng,
                                                                     const uint32_t* __restrict__ active,
                                                                     int fresh, uint64_t* totals) {
    __shared__ uint32_t presence[PRESENCE_WORDS];
    __shared__ uint32_t cand[SERIAL_WAVES], clean[SERIAL_WAVES], next_from, marked[SERIAL_WAVES];
    const uint32_t wv = threadIdx.x / WAVE;
    uint64_t rows = 0, slots = 0;
    for (uint32_t gid = blockIdx.x; gid < ng; gid += gridDim.x) {
        if (active && !active[gid]) continue;
        const GraphDev g = graphs[gid];
        uint32_t cnt = 0;
        if (!g.dirty) {   // every vertex, on wavefront 0 alone
            if (wv == 0) {
                for (uint32_t v = 0; v < g.n; v++) {
                    slots += gp(g.fill)[v];
                    cnt += tier1_vertex(g, v, presence, fresh);
                }
                rows += g.n;
            }
        } else {
            // each lane of wavefront 0 reads the marks of 16 vertices of the
            // chunk as two 8-byte words (mark arrays are padded to a multiple of 16)
            const size_t cst = (size_t)M_CHECK * g.dstride, sst = (size_t)M_STICKY * g.dstride;
            bool look = true;   // the last chunk had nothing marked (block-uniform)
            for (uint32_t base = 0; base < g.n; base += 16 * WAVE) {
                // After a chunk with nothing marked, skip unmarked chunks
                // SERIAL_WAVES at a time: each wavefront reads the marks of one
                // of the next chunks in the same round trip, and the sweep goes
                // on at the first chunk with any.  The chunks skipped stay
                // unmarked: only this block's repairs mark this graph's
                // vertices, and none ran since the read.
                if (look) {
                    const uint32_t c0 = base + 16 * WAVE * wv, a = c0 + 16 * lane();
                    bool any = false;
                    if (a < g.n) {
                        const uint64_t* cw = (const uint64_t*)(g.dirty + cst + a);
                        const uint64_t* sw = (const uint64_t*)(g.dirty + sst + a);
                        const uint32_t k = g.n - a >= 16 ? 16u : g.n - a;   // live vertices of the 16
                        const uint64_t lo = k >= 8 ? ~0ull : (1ull << (8 * k)) - 1ull;
                        const uint64_t hi = k >= 16 ? ~0ull : k <= 8 ? 0ull : (1ull << (8 * (k - 8))) - 1ull;
                        any = (((ld(&cw[0]) | gp(sw)[0]) & lo) | ((ld(&cw[1]) | gp(sw)[1]) & hi)) != 0;
                    }
                    const uint64_t m = ballot(any);
                    if (lane() == 0) marked[wv] = m != 0;
                    __syncthreads();
                    uint32_t first = SERIAL_WAVES;
                    for (uint32_t f = SERIAL_WAVES; f-- > 0;)
                        if (marked[f]) first = f;
                    __syncthreads();
                    if (first == SERIAL_WAVES) {   // nothing marked in the next SERIAL_WAVES chunks
                        base += (SERIAL_WAVES - 1) * 16 * WAVE;
                        continue;
                    }
                    base += first * 16 * WAVE;
                }
                const uint32_t v0 = base + 16 * lane();
                const uint64_t* cw = (const uint64_t*)(g.dirty + cst + v0);
                const uint64_t* sw = (const uint64_t*)(g.dirty + sst + v0);
                uint64_t s0 = 0, s1 = 0;
                if (wv == 0 && v0 < g.n) {
                    s0 = gp(sw)[0];
                    s1 = gp(sw)[1];
                }
                const uint32_t live = v0 >= g.n ? 0u : g.n - v0 >= 16 ? 0xFFFFu : (1u << (g.n - v0)) - 1u;
                uint32_t from = 0;   // chunk offset of the next vertex the sweep may visit (block-uniform)
                look = true;
                for (;;) {
                    if (wv == 0) {   // the next marked vertices
                        const uint64_t w0 = (v0 < g.n ? ld(&cw[0]) : 0ull) | s0;
                        const uint64_t w1 = (v0 < g.n ? ld(&cw[1]) : 0ull) | s1;
                        uint32_t m16 = 0;
#pragma unroll
                        for (uint32_t q = 0; q < 8; q++) {
                            m16 |= (((w0 >> (8 * q)) & 0xFFull) != 0) << q;
                            m16 |= (((w1 >> (8 * q)) & 0xFFull) != 0) << (q + 8);
                        }
                        m16 &= live;
                        const uint32_t at = 16 * lane();
                        m16 &= from <= at ? 0xFFFFu : from >= at + 16 ? 0u : ~((1u << (from - at)) - 1u) & 0xFFFFu;
                        for (uint32_t f = 0; f < SERIAL_WAVES; f++) {
                            const uint64_t any = ballot(m16 != 0);
                            uint32_t u = NONE;
                            if (any) {
                                const uint32_t k = (uint32_t)__builtin_ctzll(any);
                                const uint32_t q = (uint32_t)__builtin_ctz(__builtin_amdgcn_readlane(m16, k));
                                u = base + 16 * k + q;
                                if (lane() == k) m16 &= m16 - 1u;   // q was its lowest bit
                            }
                            if (lane() == 0) cand[f] = u;
                        }
                    }
                    __syncthreads();
                    const bool stop = cand[0] == NONE;
                    const uint32_t mine = cand[wv];
                    const bool ok = !stop && mine != NONE && tier1_clean(g, mine);
                    if (lane() == 0) clean[wv] = ok ? 1u : 0u;
                    __syncthreads();
                    if (stop) break;
                    look = false;
                    if (wv == 0) {   // in vertex order, up to the first vertex that is not clean
                        uint32_t last = base + from;
                        for (uint32_t f = 0; f < SERIAL_WAVES; f++) {
                            const uint32_t u = cand[f];
                            if (u == NONE) break;
                            if (lane() == 0) gp(g.dirty)[cst + u] = 0;
                            slots += gp(g.fill)[u];
                            rows++;
                            last = u + 1;
                            if (clean[f]) continue;
                            cnt += tier1_vertex(g, u, presence, fresh);
                            break;
                        }
                        if (lane() == 0) next_from = last - base;
                    }
                    __syncthreads();
                    from = next_from;
                }
            }
        }
        if (wv == 0 && lane() == 0 && cnt) add32(&g.ctr[C_CONFLICTS], cnt);
    }
    if (wv == 0 && lane() == 0 && totals && rows) {
        tot_add(totals, T_SWEEP_ROWS + 4, rows);
        tot_add(totals, T_SWEEP_SLOTS + 4, slots);
    }
}

// Vertices the host Tier-2 recoloured: their own status and their
// neighbourhoods are marked as a recolour on the device marks them.  One
// wavefront per (graph, vertex, old colour) item.
__global__ __launch_bounds__(256) void k_mark_recolored(const GraphDev* __restrict__ graphs,
                                                        const uint32_t* __restrict__ items, uint32_t count) {
    for (uint32_t k = wave_id(); k < count; k += wave_count()) {
        const GraphDev& g = graphs[items[3 * (size_t)k]];
        const uint32_t v = items[3 * (size_t)k + 1];
        if (v >= g.n) continue;
        const uint16_t oldc = (uint16_t)items[3 * (size_t)k + 2];
        const uint16_t newc = color_of(gp(g.word)[v]);
        if (lane() == 0) mark(g, v, D_STATUS);
        mark_neighbors(g, v, oldc, newc);
    }
}

// ---------------------------------------------------------------- Tier-2 on the device
// cpu_serial_repair (A/src/streamgc.cu:1057-1240) without leaving the GPU,
// with the same result as the host restatement: the adjacency of a vertex is
// its row plus every vertex whose row holds it ("reverse-only" neighbours
// exist only where the two rows of an edge disagree, i.e. between sticky
// vertices); uncoloured vertices with an edge are coloured first-fit in id
// order; then each pass takes the higher-id endpoint of every same-coloured
// edge and recolours them in ascending order with the lowest colour in
// [1, 1024) no neighbour holds.  The sequential parts run on one 1024-thread
// block per graph; the scans over all rows are grid-wide.
struct RevPair {
    uint32_t gid, v, u;   // u holds v in its row; v's row lacks u
};
constexpr uint32_t T2_BLOCK = 1024;

__device__ __forceinline__ bool mark_byte(const GraphDev& g, uint32_t kind, uint32_t v) {
    return gp(g.dirty)[(size_t)kind * g.dstride + v] != 0;
}

// Clear the pass flags and the reverse-only flags of the graphs taking part.
__global__ __launch_bounds__(256) void k_t2_clear(const GraphDev* __restrict__ graphs, Space sp,
                                                  const uint32_t* __restrict__ active, const uint32_t* __restrict__ gate) {
    if (gate && *gate == 0) return;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < sp.total; i += gridDim.x * blockDim.x) {
        uint32_t gid, v;
        sp.locate(i, gid, v);
        if (active && !active[gid]) continue;
        const GraphDev& g = graphs[gid];
        gp(g.dirty)[(size_t)M_TODO * g.dstride + v] = 0;
        gp(g.dirty)[(size_t)M_REV * g.dstride + v] = 0;
    }
}

// Reverse-only neighbours: for a sticky u and a sticky v in u's row, (v, u)
// when v's row lacks u.  One wavefront per vertex.
__global__ __launch_bounds__(256) void k_t2_rev(const GraphDev* __restrict__ graphs, Space sp,
                                                const uint32_t* __restrict__ active, RevPair* __restrict__ rev,
                                                uint32_t* __restrict__ rev_count, uint32_t cap,
                                                const uint32_t* __restrict__ dspace, uint32_t ng,
                                                const uint32_t* __restrict__ gate) {
    if (gate && *gate == 0) return;
    if (dspace) sp = device_space(dspace, ng);
    for (uint32_t i = wave_id(); i < sp.total; i += wave_count()) {
        uint32_t gid, u;
        sp.locate(i, gid, u);
        if (active && !active[gid]) continue;
        const GraphDev& g = graphs[gid];
        if (!mark_byte(g, M_STICKY, u)) continue;
        const uint32_t s = gp(g.row_ptr)[u], e = s + ld(&g.fill[u]);
        for (uint32_t base = s; base < e; base += WAVE) {
            const uint32_t j = base + lane();
            const uint32_t v = j < e ? ld(&g.col[j]) : INVALID;
            uint64_t m = ballot(v != INVALID && v < g.n && v != u && mark_byte(g, M_STICKY, v));
            while (m) {
                const uint32_t k = (uint32_t)__builtin_ctzll(m);
                m &= m - 1;
                const uint32_t w = (uint32_t)__shfl((int)v, (int)k);
                const uint32_t s2 = gp(g.row_ptr)[w], e2 = s2 + ld(&g.fill[w]);
                bool found = false;
                for (uint32_t b2 = s2; b2 < e2 && !found; b2 += WAVE) {
                    const uint32_t j2 = b2 + lane();
                    found = ballot(j2 < e2 && ld(&g.col[j2]) == u) != 0;
                }
                if (!found && lane() == 0) {
                    const uint32_t at = add32(rev_count, 1u);
                    if (at < cap) {
                        st(&rev[at].gid, gid);
                        st(&rev[at].v, w);
                        st(&rev[at].u, u);
                    } else {
                        add32(&g.ctr[C_REVOVF], 1u);
                    }
                    gp(g.dirty)[(size_t)M_REV * g.dstride + w] = 1;
                }
            }
        }
    }
}

// first_fit of the host restatement for vertex v, by the whole block.
// Returns true when v changed colour (it is then marked like any recolour).
__device__ __forceinline__ bool t2_first_fit(const GraphDev& g, uint32_t gid, uint32_t v,
                                             const RevPair* __restrict__ rev, uint32_t nrev) {
    __shared__ uint32_t seen[HIST_BINS / 32];
    __shared__ uint32_t pick;
    if (threadIdx.x < HIST_BINS / 32) seen[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t s = gp(g.row_ptr)[v], e = s + ld(&g.fill[v]);
    for (uint32_t j = s + threadIdx.x; j < e; j += T2_BLOCK) {
        const uint32_t nb = ld(&g.col[j]);
        if (nb == INVALID || nb >= g.n || nb == v) continue;
        const uint32_t c = color_of(ld(&g.word[nb]));
        if (c != 0 && c < HIST_BINS) atomicOr(&seen[c >> 5], 1u << (c & 31));
    }
    if (mark_byte(g, M_REV, v))
        for (uint32_t k = threadIdx.x; k < nrev; k += T2_BLOCK) {
            if (rev[k].gid != gid || rev[k].v != v) continue;
            const uint32_t c = color_of(ld(&g.word[rev[k].u]));
            if (c != 0 && c < HIST_BINS) atomicOr(&seen[c >> 5], 1u << (c & 31));
        }
    __syncthreads();
    if (threadIdx.x < WAVE) {
        uint32_t word = threadIdx.x < HIST_BINS / 32 ? seen[threadIdx.x] : 0xFFFFFFFFu;
        if (threadIdx.x == 0) word |= 1u;   // colour 0 is not a colour
        const uint64_t open = ballot(word != 0xFFFFFFFFu);
        uint32_t c = 0;
        if (open) {
            const uint32_t k = (uint32_t)__builtin_ctzll(open);
            const uint32_t wk = (uint32_t)__shfl((int)word, (int)k);
            c = 32 * k + (uint32_t)__builtin_ctz(~wk);
        }
        if (threadIdx.x == 0) {
            const uint32_t w = ld(&g.word[v]);
            const uint32_t oc = color_of(w);
            if (c == 0 || c == oc) {
                pick = 0;
            } else {
                st(&g.word[v], bump(w, (uint16_t)c));
                pick = 0x80000000u | (oc << 16) | c;
            }
        }
    }
    __syncthreads();
    const uint32_t p = pick;
    __syncthreads();
    if (!p) return false;
    if (threadIdx.x < WAVE) {
        if (lane() == 0) mark(g, v, D_STATUS);
        mark_neighbors(g, v, (uint16_t)((p >> 16) & 0x7FFFu), (uint16_t)(p & 0xFFFFu));
    }
    return true;
}

// Vertices of one graph flagged in mark array `kind` (or, for kind ==
// M_ARRAYS, uncoloured vertices with an edge), visited in ascending order by
// the block: flags are cleared and first_fit applied.  Returns the recolours.
__device__ __forceinline__ uint32_t t2_ordered_pass(const GraphDev& g, uint32_t gid, uint32_t kind,
                                                    const RevPair* __restrict__ rev, uint32_t nrev) {
    __shared__ uint64_t cand[T2_BLOCK / WAVE];
    __shared__ uint32_t has;
    uint32_t fixed = 0;
    for (uint32_t base = 0; base < g.n; base += T2_BLOCK) {
        const uint32_t v = base + threadIdx.x;
        bool c = false;
        if (v < g.n) {
            if (kind == M_ARRAYS) {
                c = color_of(ld(&g.word[v])) == 0;
            } else if (mark_byte(g, kind, v)) {
                c = true;
                gp(g.dirty)[(size_t)kind * g.dstride + v] = 0;
            }
        }
        const uint64_t m = ballot(c);
        if (lane() == 0) cand[threadIdx.x / WAVE] = m;
        __syncthreads();
        for (uint32_t w = 0; w < T2_BLOCK / WAVE; w++) {
            uint64_t mw = cand[w];
            while (mw) {
                const uint32_t b = (uint32_t)__builtin_ctzll(mw);
                mw &= mw - 1;
                const uint32_t u = base + w * WAVE + b;
                if (kind == M_ARRAYS) {   // only a vertex with an edge is coloured
                    if (threadIdx.x == 0) has = mark_byte(g, M_REV, u) ? 1u : 0u;
                    __syncthreads();
                    const uint32_t s = gp(g.row_ptr)[u], e = s + ld(&g.fill[u]);
                    bool any = false;
                    for (uint32_t j = s + threadIdx.x; j < e && !any; j += T2_BLOCK) {
                        const uint32_t nb = ld(&g.col[j]);
                        any = nb != INVALID && nb < g.n && nb != u;
                    }
                    if (any) has = 1;
                    __syncthreads();
                    const bool go = has != 0;
                    __syncthreads();
                    if (!go) continue;
                }
                fixed += t2_first_fit(g, gid, u, rev, nrev) ? 1u : 0u;
            }
        }
        __syncthreads();
    }
    return fixed;
}

// The uncoloured pass (pass == 0) or one conflict pass over the flagged
// vertices, one block per graph taking part.
__global__ __launch_bounds__(T2_BLOCK) void k_t2_serial(const GraphDev* __restrict__ graphs, uint32_t ng,
                                                        const uint32_t* __restrict__ active,
                                                        const RevPair* __restrict__ rev,
                                                        const uint32_t* __restrict__ rev_count, uint32_t cap,
                                                        int uncoloured, const uint32_t* __restrict__ gate) {
    if (gate && *gate == 0) return;
    const uint32_t nrev = *rev_count < cap ? *rev_count : cap;
    for (uint32_t gid = blockIdx.x; gid < ng; gid += gridDim.x) {
        if (active && !active[gid]) continue;
        const GraphDev g = graphs[gid];
        const uint32_t f = t2_ordered_pass(g, gid, uncoloured ? M_ARRAYS : M_TODO, rev, nrev);
        if (threadIdx.x == 0) {
            if (!uncoloured) gp(g.ctr)[C_T2FIXED] = f;
            gp(g.ctr)[C_T2TOTAL] += f;
        }
        __syncthreads();
    }
}

// The next pass's list: the higher-id endpoint of every same-coloured slot
// pair of every row.  One wavefront per row; C_T2TODO becomes 1 if any.
__global__ __launch_bounds__(256) void k_t2_flags(const GraphDev* __restrict__ graphs, Space sp,
                                                  const uint32_t* __restrict__ active,
                                                  const uint32_t* __restrict__ dspace, uint32_t ng,
                                                  const uint32_t* __restrict__ gate) {
    if (gate && *gate == 0) return;
    if (dspace) sp = device_space(dspace, ng);
    for (uint32_t i = wave_id(); i < sp.total; i += wave_count()) {
        uint32_t gid, x;
        sp.locate(i, gid, x);
        if (active && !active[gid]) continue;
        const GraphDev& g = graphs[gid];
        const uint32_t cx = color_of(ld(&g.word[x]));
        if (cx == 0) continue;
        const uint32_t s = gp(g.row_ptr)[x], e = s + ld(&g.fill[x]);
        bool any = false;
        for (uint32_t base = s; base < e; base += WAVE) {
            const uint32_t j = base + lane();
            const uint32_t y = j < e ? ld(&g.col[j]) : INVALID;
            if (y != INVALID && y < g.n && y != x && color_of(ld(&g.word[y])) == cx) {
                gp(g.dirty)[(size_t)M_TODO * g.dstride + (y > x ? y : x)] = 1;
                any = true;
            }
        }
        if (ballot(any) && lane() == 0) gp(g.ctr)[C_T2TODO] = 1;
    }
}

// ---------------------------------------------------------------- checks
// Tier-2 has work iff some row slot joins an uncoloured endpoint or two
// endpoints of one colour (A/src/streamgc.cu:1190-1218 then change nothing).
// Bad slots of row v: an uncoloured endpoint or two equal colours.
template <bool kBlock>
__device__ __forceinline__ uint32_t t2_row(const GraphDev& g, uint32_t v) {
    const uint32_t s = gp(g.row_ptr)[v], e = s + gp(g.fill)[v];
    const uint32_t width = kBlock ? BLOCK : WAVE, me = kBlock ? threadIdx.x : lane();
    const uint16_t cv = color_of(gp(g.word)[v]);
    uint32_t bad = 0;
    for (uint32_t base = s; base < e; base += ROW_UNROLL * width) {
        uint32_t nb[ROW_UNROLL];
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) {
            const uint32_t j = base + u * width + me;
            nb[u] = j < e ? gp(g.col)[j] : INVALID;
        }
#pragma unroll
        for (uint32_t u = 0; u < ROW_UNROLL; u++) {
            if (nb[u] != INVALID && nb[u] < g.n && nb[u] != v) {
                const uint16_t cn = color_of(gp(g.word)[nb[u]]);
                bad += (cv == 0 || cn == 0 || cv == cn);
            }
        }
    }
    return kBlock ? block_sum32(bad) : wave_sum32(bad);
}

// The same for rows of at most GROUP_ROW slots, 16 lanes each: the bad slots of
// the lane's row of vertex v, if `mine` (slots [s, s + f)).
__device__ __forceinline__ uint32_t t2_row_group(const GraphDev& g, bool mine, uint32_t v, uint32_t s, uint32_t f) {
    const uint32_t cv = mine ? color_of(gp(g.word)[v]) : 0u;
    uint32_t nb[ROW_UNROLL], bad = 0;
#pragma unroll
    for (uint32_t u = 0; u < ROW_UNROLL; u++) {
        const uint32_t j = u * GROUP + sublane();
        nb[u] = mine && j < f ? gp(g.col)[s + j] : INVALID;
    }
#pragma unroll
    for (uint32_t u = 0; u < ROW_UNROLL; u++)
        if (nb[u] != INVALID && nb[u] < g.n && nb[u] != v) {
            const uint32_t cn = color_of(gp(g.word)[nb[u]]);
            bad += (cv == 0 || cn == 0 || cv == cn);
        }
    for (uint32_t o = GROUP / 2; o > 0; o >>= 1) bad += __shfl_xor(bad, o);
    return bad;
}

// Tier-2 has work iff some row slot joins an uncoloured endpoint or two
// endpoints of one colour (A/src/streamgc.cu:1190-1218 then change nothing).
// A vertex found with a bad slot keeps its mark, so the next check counts it
// again until a repair changes it.
__global__ __launch_bounds__(256) void k_t2_check(const GraphDev* __restrict__ graphs, Space sp, SweepList sl,
                                                  uint64_t* totals) {
    uint64_t rows = 0, slots = 0;
    const uint32_t nbig = sweep_big(sl);
    for (uint32_t k = blockIdx.x; k < nbig; k += gridDim.x) {
        uint32_t gid, v;
        sp.locate(big_item(sl, k), gid, v);
        const GraphDev& g = graphs[gid];
        const uint32_t bad = t2_row<true>(g, v);
        if (threadIdx.x == 0) {
            rows++;
            slots += gp(g.fill)[v];
            if (bad) {
                add32(&g.ctr[C_T2BAD], bad);
                if (g.dirty) gp(g.dirty)[(size_t)M_T2 * g.dstride + v] = 1;
            }
        }
    }
    uint32_t row_n = 0, slot_n = 0;   // of the lane's rows (one lane of the row counts)
    for_rows(graphs, sp, sl, [&](const GraphDev& g, uint32_t, bool mine, uint32_t v) {
        const uint32_t f = mine ? gp(g.fill)[v] : 0u, s = mine ? gp(g.row_ptr)[v] : 0u;
        const bool one = mine && sublane() == 0, few = f <= GROUP_ROW;
        row_n += one;
        slot_n += one ? f : 0u;
        uint32_t bad = t2_row_group(g, mine && few, v, s, f);
        each_row(ballot(one && !few), v, [&](uint32_t x) {
            const uint32_t n = t2_row<false>(g, x);
            if (one && x == v) bad = n;
        });
        if (one && bad) {
            add32(&g.ctr[C_T2BAD], bad);
            if (g.dirty) gp(g.dirty)[(size_t)M_T2 * g.dstride + v] = 1;
        }
    });
    rows += wave_sum32(row_n);
    slots += wave_sum32(slot_n);
    if (lane() != 0) rows = slots = 0;
    block_add64(totals, T_SWEEP_ROWS + 3, rows);
    block_add64(totals, T_SWEEP_SLOTS + 3, slots);
}

// check_coloring_valid on the engine's rows (A/src/streamgc.cu:448-556);
// colours from `colors` when given (a snapshot), else the live words.
__global__ __launch_bounds__(256) void k_validate(const GraphDev* __restrict__ graphs, uint32_t gid,
                                                  const uint16_t* __restrict__ colors) {
    const GraphDev& g = graphs[gid];
    uint32_t viol = 0, unc = 0, mx = 0;
    for (uint32_t v = wave_id(); v < g.n; v += wave_count()) {
        const uint32_t s = gp(g.row_ptr)[v], e = s + gp(g.fill)[v];
        const uint16_t cv = colors ? colors[v] : color_of(gp(g.word)[v]);
        uint32_t bad = 0, has = 0;
        for (uint32_t base = s; base < e; base += WAVE) {
            const uint32_t j = base + lane();
            const uint32_t nb = j < e ? gp(g.col)[j] : INVALID;
            if (nb != INVALID) {
                has = 1;
                if (nb < g.n) {
                    const uint16_t cn = colors ? colors[nb] : color_of(gp(g.word)[nb]);
                    bad += (cv != 0 && cv == cn);
                }
            }
        }
        viol += wave_sum32(bad);
        unc += (cv == 0 && ballot(has != 0)) ? 1 : 0;
        mx = cv > mx ? cv : mx;
    }
    if (lane() == 0) {
        if (viol) add32(&g.ctr[C_VIOL], viol);
        if (unc) add32(&g.ctr[C_UNCOL], unc);
        max32(&g.ctr[C_MAXC], mx);
    }
}

__global__ void k_find_color(const GraphDev* __restrict__ graphs, uint32_t gid, uint32_t v, uint16_t* out) {
    const GraphDev g = graphs[gid];
    const uint16_t c = find_color(g, v);
    if (lane() == 0) *out = c;
}

// Independent validator: edges with life intervals checked against snapshot
// k at stream position pos[k] (blockIdx.y = k).
__global__ __launch_bounds__(256) void k_validate_history(const uint16_t* __restrict__ snaps, uint32_t n,
                                                          const uint32_t* __restrict__ eu,
                                                          const uint32_t* __restrict__ ev,
                                                          const uint64_t* __restrict__ born,
                                                          const uint64_t* __restrict__ died, uint64_t m,
                                                          const uint64_t* __restrict__ pos,
                                                          unsigned long long* bad_out) {
    const uint32_t k = blockIdx.y;
    const uint16_t* snap = snaps + (size_t)k * n;
    const uint64_t p = pos[k];
    uint32_t bad = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (uint64_t)gridDim.x * blockDim.x) {
        if (born[i] <= p && p < died[i]) {
            const uint16_t a = snap[eu[i]], b = snap[ev[i]];
            bad += (a == 0) + (b == 0) + (a != 0 && a == b);
        }
    }
    bad = wave_sum32(bad);
    if (bad && lane() == 0) atomicAdd(&bad_out[k], (unsigned long long)bad);
}

// Slack-CSR construction (A/src/streamgc.cu:350-433): copy each loaded row to
// the front of its slack row, free slots after it.
__global__ __launch_bounds__(256) void k_fill_rows(uint32_t n, const uint32_t* __restrict__ rp0,
                                                   const uint32_t* __restrict__ col0,
                                                   const uint32_t* __restrict__ rp, uint32_t* __restrict__ col,
                                                   uint32_t* __restrict__ fill) {
    for (uint32_t v = wave_id(); v < n; v += wave_count()) {
        const uint32_t s0 = rp0[v], d = rp0[v + 1] - s0;
        const uint32_t s = rp[v], e = rp[v + 1];
        if (lane() == 0) fill[v] = d < e - s ? d : e - s;
        for (uint32_t j = s + lane(); j < e; j += WAVE) {
            const uint32_t k = j - s;
            col[j] = k < d ? col0[s0 + k] : INVALID;
        }
    }
}

}  // namespace sgc

// ---------------------------------------------------------------- launchers
namespace sgc {

static inline Space space(const LaunchCtx& L) { return Space{L.sbase, L.sgid, L.ns, L.V}; }

static inline uint32_t grid_for_waves(uint64_t waves, uint32_t waves_per_block, uint32_t cap) {
    uint64_t b = (waves + waves_per_block - 1) / waves_per_block;
    if (b < 1) b = 1;
    if (b > cap) b = cap;
    return (uint32_t)b;
}

// Four light edges to a wavefront for more than QUADS_OVER updates: below, the
// chip holds most of the edges at once, one to a wavefront, and an edge's chain
// is shorter alone (launch, us, one / four edges a wavefront: 5,400 updates of a
// 131,072-vertex mesh 16.5 / 18, 8,193: 22.5 / 15; 4,099 of a 65,536-vertex
// R-MAT graph 45 / 52, 8,193: 81 / 81).  And for at most one update to two
// vertices: with more, updates meet at the same rows, all the more of them the
// more are in flight, and an edge's colour choices wait for three others'
// (16,384 updates of growth on an 8,192-vertex R-MAT graph 118 / 207, 32,768 of
// churn on a 16,384-vertex one 150 / 220; at one to two, 65,536 updates: a
// 131,072-vertex mesh 107 / 58, an R-MAT graph of that size 285 / 269, of growth
// 281 / 231, but 16,384 on a 32,768-vertex one 106 / 111; 196,608 of 48 graphs,
// one to 2.4, 331 / 194).
// Where more than three in ten edges are heavy, each of those takes a wavefront
// either way, and the four-edge kernel pays only for more than QUADS_OVER_LONG:
// 32,768 updates of an R-MAT graph of 262,144 vertices and 24 edges a vertex,
// churn 225 / 219, growth 157 / 153, but the repairs that more updates in flight
// cost make the growth's epochs 3% slower; 65,536 of growth there 295 / 230.
constexpr uint32_t QUADS_OVER = 8192, QUADS_OVER_LONG = 32768;
// A delete's long scans in trips of 1,024 slots for at most one update to
// LONG_PER vertices.  They end a hub's deletes in half the time, and so before
// other updates of the launch that touch the same vertices: on a skewed graph
// with one update to 16 vertices some streams then end with other colours every
// time (tests/test_gpu_racing.py).  At one to 64 and fewer, updates hardly meet:
// of 108 passes of such streams on five graphs 106 ended as the short trips' did,
// as many as between two runs of the short trips.  Launch, us, short / long trips: 32,768 updates
// of a 4M-vertex power-law graph 125 / 78, 16,384 of a 2^20-vertex R-MAT graph
// 325 / 197, of growth there 208 / 148; at one to 32, 16,384 of growth on a
// 2^19-vertex one 142 / 152.
constexpr uint32_t LONG_PER = 64;
hipError_t launch_apply(const LaunchCtx& L, const void* upd, uint32_t count, int multi, EdgeGroups* eg,
                        const BatchGraphs& on) {
    if (count == 0) return hipSuccess;
    const bool group = eg && eg->keys && count > 1;
    if (group && ((uint64_t)eg->size < 2ull * count || eg->next_cap < count || !eg->heads || !eg->nheads || !eg->pack))
        return hipErrorInvalidValue;
    const EdgeGroups G = group ? *eg : EdgeGroups();
    // one-wavefront blocks: a wavefront's slot is refilled as soon as it ends
    const uint32_t grid = grid_for_waves(count, 1, 4 * L.max_blocks);
    if (group && count > QUADS_OVER && count <= on.vertices / LONG_PER)
        k_apply_quads<true><<<grid, WAVE, 0, L.stream>>>(L.graphs, (const uint4*)upd, multi, G.next, G.nheads, G.pack,
                                                         L.totals, L.dyn);
    else if (group && count > (10 * on.long_entries > 3 * on.edges ? QUADS_OVER_LONG : QUADS_OVER) &&
             count <= on.vertices / 2)
        k_apply_quads<false><<<grid, WAVE, 0, L.stream>>>(L.graphs, (const uint4*)upd, multi, G.next, G.nheads, G.pack,
                                                          L.totals, L.dyn);
    else
        k_apply_elem<<<grid, WAVE, 0, L.stream>>>(L.graphs, (const uint4*)upd, count, multi, G.next, G.nheads, G.pack,
                                                  L.totals, L.dyn);
    const hipError_t e = hipGetLastError();
    if (group && e == hipSuccess) eg->linked = false;
    return e;
}
hipError_t launch_group_clear(hipStream_t s, const EdgeGroups& eg) {
    k_group_clear<<<grid_for_waves(eg.size, 4 * WAVE, 1024), 256, 0, s>>>(eg.keys, eg.head, eg.size, eg.nheads);
    return hipGetLastError();
}
// The table is full from the link to the apply launch of the same batch: if one
// of the three did not start, the next batch clears it first (its entries and
// counts would otherwise be taken for that batch's own).
hipError_t launch_group(const LaunchCtx& L, const void* upd, uint32_t count, int multi, EdgeGroups* eg) {
    if (count <= 1 || !eg || !eg->keys) return hipSuccess;
    if ((uint64_t)eg->size < 2ull * count || eg->next_cap < count || !eg->pack) return hipErrorInvalidValue;
    hipError_t e = eg->linked ? launch_group_clear(L.stream, *eg) : hipSuccess;
    if (e != hipSuccess) return e;
    eg->linked = true;
    const uint32_t mask = eg->size - 1;
    uint32_t mg = grid_for_waves(count, 4 * WAVE, 1024);
    k_group_link<<<mg, 256, 0, L.stream>>>(L.graphs, L.gbase, (const uint4*)upd, count, multi, eg->keys, eg->head,
                                           eg->next, mask, eg->heads, eg->next_cap, eg->nheads, L.dyn);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    k_group_pack<<<mg, 256, 0, L.stream>>>((const uint4*)upd, eg->keys, eg->head, eg->next, eg->heads, eg->next_cap,
                                           eg->nheads, eg->pack, L.dyn);
    return hipGetLastError();
}
// A CU holds 16 wavefronts of this kernel: one block of REPLAY_WAVES, or two of
// half as many.  Up to REPLAY_BLOCKS segments (one to a CU) take whole blocks, up
// to twice as many half ones, above it one wavefront each: a segment that had to
// wait for another's block would take twice as long, which a stream with nothing
// to run together (it colours fresh vertices) does not make good.  300 updates on
// each of n 4,096-vertex meshes, us, single wavefronts / whole blocks / half
// blocks: churn, n = 256: 797 / 186 / -, 512: 941 / 380 / 344; first colourings,
// 256: 1,384 / 1,388 / -, 512: 1,652 / 2,801 / 1,649.
constexpr uint32_t REPLAY_BLOCKS = 256;
hipError_t launch_apply_seg(const LaunchCtx& L, const void* upd, const uint32_t* seg, uint32_t nseg,
                            const uint32_t* perm, int multi) {
    if (nseg == 0) return hipSuccess;
    const uint32_t grid = grid_for_waves(nseg, 1, L.max_blocks);
    const auto replay = [&](auto waves) {
        constexpr uint32_t W = decltype(waves)::value;
        k_apply_seg<W><<<grid, W * WAVE, 0, L.stream>>>(L.graphs, (const uint4*)upd, seg, nseg, perm, multi, L.totals,
                                                        L.dyn);
    };
    if (nseg <= REPLAY_BLOCKS) replay(std::integral_constant<uint32_t, REPLAY_WAVES>{});
    else if (nseg <= 2 * REPLAY_BLOCKS) replay(std::integral_constant<uint32_t, REPLAY_WAVES / 2>{});
    else replay(std::integral_constant<uint32_t, 1>{});
    return hipGetLastError();
}
hipError_t launch_zero_ctr(const LaunchCtx& L, uint32_t idx) {
    k_zero_ctr<<<(L.ng + 63) / 64, 64, 0, L.stream>>>(L.graphs, L.ng, L.active, idx);
    return hipGetLastError();
}
hipError_t launch_max_color(const LaunchCtx& L) {
    if (L.ns == 1) {
        k_max_color1<<<256, 256, 0, L.stream>>>(L.graphs, space(L));
        return hipGetLastError();
    }
    uint32_t grid = grid_for_waves(L.V, 4 * WAVE, 1024);
    k_max_color<<<grid, 256, 0, L.stream>>>(L.graphs, space(L));
    return hipGetLastError();
}
hipError_t launch_snapshot(const LaunchCtx& L, const uint32_t* fl_round, const HistDev* hist) {
    if (!fl_round) hist = nullptr;
    if (L.ns == 1) {
        const uint32_t grid = grid_for_waves(L.V / 4 + 1, 4 * WAVE, L.max_blocks);
        k_snapshot1<<<grid, 256, 0, L.stream>>>(L.graphs, space(L), L.active, fl_round, hist);
        return hipGetLastError();
    }
    uint32_t grid = grid_for_waves(L.V, 4 * WAVE, L.max_blocks);
    k_snapshot<<<grid, 256, 0, L.stream>>>(L.graphs, space(L), L.active, fl_round, hist);
    return hipGetLastError();
}
// Sweep grids: a wavefront per row up to a cap, grid-stride (blocks first take
// the long rows of a worklist); a worklist sweep's cap is sweep_blocks (its
// length is on the device).
static inline uint32_t sweep_grid(const LaunchCtx& L) {
    return grid_for_waves(L.V, 4, L.list ? L.sweep_blocks : L.max_blocks);
}
static inline SweepList sweep_list(const LaunchCtx& L) { return SweepList{L.list, L.list_count, L.list_cap}; }
hipError_t launch_build_list(const LaunchCtx& L, uint32_t kind, uint32_t* list, uint32_t cap, uint32_t* count,
                             uint32_t kind2, size_t second) {
    const bool two = kind2 != NO_KIND;
    if (kind >= M_STICKY || (two && (kind2 >= M_STICKY || kind2 == kind || !second)) || cap < L.V)
        return hipErrorInvalidValue;
    // Two passes over 4096-vertex tiles, each tile inside one graph (scratch
    // behind the list): one graph's own tiles, or the tiles of several graphs
    // laid end to end (L.stile, L.tiles).
    const bool multi = L.ns > 1;
    const uint32_t tiles = multi ? L.tiles : (L.V + LIST_TILE_V - 1) / LIST_TILE_V;
    if (multi && (!L.stile || tiles > list_tiles(cap, L.ng))) return hipErrorInvalidValue;
    if (tiles == 0) {
        k_zero_list_count<<<1, 1, 0, L.stream>>>(count);
        if (two) k_zero_list_count<<<1, 1, 0, L.stream>>>(count + 2);
        return hipGetLastError();
    }
    uint32_t* tmp = list + cap;
    uint32_t* tcount = tmp + (size_t)tiles * LIST_TILE_V;
    const dim3 grid(tiles, two ? 2 : 1);
    k_list_tiles<<<grid, 256, 0, L.stream>>>(L.graphs, space(L), multi ? L.stile : nullptr, kind, kind2, second,
                                             L.long_row, tmp, tcount, L.active, L.gate);
    k_list_gather<<<grid, 256, 0, L.stream>>>(L.graphs, space(L), multi ? 1 : 0, tmp, tcount, list, cap, second, count,
                                              L.active, L.gate);
    return hipGetLastError();
}
// Whether a sweep visits every row on a grid with a wavefront for each: the
// kernel then takes them so, with the registers that takes (Tier-1: 64, with the
// shared rows' and long rows' code 104, which leaves 4 wavefronts a SIMD, not 8).
// Compaction and Tier-1 of 50,000 rows of 100 slots, us, so / with the shared
// rows' code: 26 / 33 and 44 / 75.
static inline bool alone_rows(const LaunchCtx& L) { return !L.list && L.V <= 4ull * sweep_grid(L); }
hipError_t launch_compact(const LaunchCtx& L, bool drain_prep) {
    auto* const kernel = alone_rows(L) ? &k_compact<true> : &k_compact<false>;
    kernel<<<sweep_grid(L), 256, 0, L.stream>>>(L.graphs, space(L), sweep_list(L), L.totals, drain_prep ? L.ng : 0u,
                                                L.active);
    return hipGetLastError();
}
hipError_t launch_drain(const LaunchCtx& L, bool serial, uint32_t max_count, bool prepped) {
    if (!prepped) k_drain_prep<<<(L.ng + 63) / 64, 64, 0, L.stream>>>(L.graphs, L.ng, L.active);
    if (serial) {
        k_drain_serial<<<L.ng < 1024 ? L.ng : 1024, 64, 0, L.stream>>>(L.graphs, L.ng, L.active);
    } else {
        // entries of one graph share grid.x blocks; many graphs take fewer each
        const uint32_t per_graph = L.ng > 4 ? (16384 / L.ng > 0 ? 16384 / L.ng : 1) : 4096;
        dim3 grid(grid_for_waves(max_count, 4, per_graph), L.ng);
        k_drain_elem<<<grid, 256, 0, L.stream>>>(L.graphs, L.active);
    }
    return hipGetLastError();
}
hipError_t launch_rebuild(const LaunchCtx& L, bool exact_hist) {
    k_rebuild<<<sweep_grid(L), 256, 0, L.stream>>>(L.graphs, space(L), sweep_list(L),
                                                   exact_hist ? 1 : 0, L.totals);
    return hipGetLastError();
}
hipError_t launch_tier1(const LaunchCtx& L, bool serial, int fresh) {
    if (serial) {
        const uint32_t grid = L.ng < 1024 ? L.ng : 1024;
        k_tier1_serial<<<grid, SERIAL_WAVES * WAVE, 0, L.stream>>>(L.graphs, L.ng, L.active, fresh, L.totals);
    } else {
        auto* const kernel = alone_rows(L) ? &k_tier1_elem<true> : &k_tier1_elem<false>;
        kernel<<<sweep_grid(L), 256, 0, L.stream>>>(L.graphs, space(L), sweep_list(L), fresh, L.totals);
    }
    return hipGetLastError();
}
hipError_t launch_t2_check(const LaunchCtx& L) {
    k_t2_check<<<sweep_grid(L), 256, 0, L.stream>>>(L.graphs, space(L), sweep_list(L),
                                                    L.totals);
    return hipGetLastError();
}
hipError_t launch_mark_recolored(hipStream_t s, const GraphDev* graphs, const uint32_t* items, uint32_t count) {
    if (count == 0) return hipSuccess;
    k_mark_recolored<<<grid_for_waves(count, 4, 4096), 256, 0, s>>>(graphs, items, count);
    return hipGetLastError();
}
hipError_t launch_t2_begin(const LaunchCtx& L, void* rev, uint32_t* rev_count, uint32_t cap) {
    k_zero_list_count<<<1, 1, 0, L.stream>>>(rev_count);   // [0] is the pair count
    k_t2_clear<<<grid_for_waves(L.V, 4 * WAVE, 4096), 256, 0, L.stream>>>(L.graphs, space(L), L.active, L.gate);
    k_t2_rev<<<grid_for_waves(L.V, 4, L.max_blocks), 256, 0, L.stream>>>(L.graphs, space(L), L.active,
                                                                         (RevPair*)rev, rev_count, cap, L.dspace,
                                                                         L.ng, L.gate);
    return hipGetLastError();
}
hipError_t launch_t2_pass(const LaunchCtx& L, const void* rev, const uint32_t* rev_count, uint32_t cap,
                          bool uncoloured) {
    if (!uncoloured)
        k_t2_flags<<<grid_for_waves(L.V, 4, L.max_blocks), 256, 0, L.stream>>>(L.graphs, space(L), L.active,
                                                                               L.dspace, L.ng, L.gate);
    k_t2_serial<<<L.ng < 1024 ? L.ng : 1024, T2_BLOCK, 0, L.stream>>>(L.graphs, L.ng, L.active, (const RevPair*)rev,
                                                                      rev_count, cap, uncoloured ? 1 : 0, L.gate);
    return hipGetLastError();
}
hipError_t launch_validate(const LaunchCtx& L, uint32_t gid, uint32_t n, const uint16_t* colors) {
    uint32_t grid = grid_for_waves(n, 4, L.max_blocks);
    k_validate<<<grid, 256, 0, L.stream>>>(L.graphs, gid, colors);
    return hipGetLastError();
}
hipError_t launch_find_color(const LaunchCtx& L, uint32_t gid, uint32_t v, uint16_t* out) {
    k_find_color<<<1, 64, 0, L.stream>>>(L.graphs, gid, v, out);
    return hipGetLastError();
}
hipError_t launch_validate_history(hipStream_t s, const uint16_t* snaps, uint32_t n, const uint32_t* eu,
                                   const uint32_t* ev, const uint64_t* born, const uint64_t* died, uint64_t m,
                                   const uint64_t* pos, uint32_t count, unsigned long long* bad_out) {
    if (count == 0 || m == 0) return hipSuccess;
    uint64_t blocks = (m + 255) / 256;
    dim3 grid((uint32_t)(blocks < 2048 ? blocks : 2048), count);
    k_validate_history<<<grid, 256, 0, s>>>(snaps, n, eu, ev, born, died, m, pos, bad_out);
    return hipGetLastError();
}
hipError_t launch_fill_rows(hipStream_t s, uint32_t n, const uint32_t* rp0, const uint32_t* col0, const uint32_t* rp,
                            uint32_t* col, uint32_t* fill) {
    uint32_t grid = grid_for_waves(n, 4, 16384);
    k_fill_rows<<<grid, 256, 0, s>>>(n, rp0, col0, rp, col, fill);
    return hipGetLastError();
}

// ---------------------------------------------------------------- T_rc microbenchmark
// A/benchmark/microbench/t_rc_atomic.cu:18-28: one lane runs `iters`
// dependent CAS operations on a vertex word, each bumping the version and
// toggling the colour's low bit (a failed CAS takes the value it found).
// Here every wavefront's lane 0 does so, on word (wave x stride): stride 32
// gives each wavefront its own 128-byte line, stride 0 makes them all share
// one word.
__global__ __launch_bounds__(64) void k_trc(uint32_t* __restrict__ words, uint32_t stride, uint32_t iters) {
    if (threadIdx.x != 0) return;
    uint32_t* w = words + (size_t)blockIdx.x * stride;
    uint32_t cur = ld(w);
    for (uint32_t i = 0; i < iters; i++) {
        const uint32_t nxt = bump(cur, (uint16_t)((cur & 0xFFFFu) ^ 1u));
        const uint32_t got = cas32(w, cur, nxt);
        cur = got == cur ? nxt : got;
    }
}
hipError_t launch_trc(hipStream_t s, uint32_t* words, uint32_t waves, uint32_t stride, uint32_t iters) {
    k_trc<<<waves, WAVE, 0, s>>>(words, stride, iters);
    return hipGetLastError();
}

}  // namespace sgc
