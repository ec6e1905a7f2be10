// tx_pipeline.hip -- binned ClusterFit pipeline: classify, bin, search.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bcn_device.hpp"
#include "bcn_lane.hpp"
#include "tx_pipeline.hpp"

#pragma clang fp contract(off)

namespace txp {

void PipeBufs::carve(uint8_t* base, uint64_t cap)
{
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    size_t off = 0;
    recs = reinterpret_cast<ClusterRec*>(base + off);
    off += up(sizeof(ClusterRec) * cap);
    keys = reinterpret_cast<uint32_t*>(base + off);
    off += up(4 * cap);
    for (int k = 0; k < kLists; ++k) {
        list[k] = reinterpret_cast<uint32_t*>(base + off);
        off += up(4 * kListArrays * cap);
    }
    ctl = reinterpret_cast<PipeCtl*>(base + off);
    capacity = cap;
}

}  // namespace txp

namespace txd {

using txk::BatchTex;
using txp::ClusterRec;
using txp::PipeCtl;

using txp::kLists;
using txp::kListA;
using txp::kListB;
using txp::kListC;
using txp::kSearchWaves;
constexpr uint32_t key_bit(int list) { return 1u << (5 + list); }

__device__ __forceinline__ const BatchTex& tex_at(const BatchTex* tex, const BatchTex& tex0, uint32_t i)
{
    return tex ? tex[i] : tex0;
}

// The counters of this run, cleared by the first workgroup of the classify
// pass: the kernels that use them start when it has ended.
__device__ __forceinline__ void clear_counters(PipeCtl* __restrict__ ctl, int lane)
{
    constexpr int words = sizeof(PipeCtl) / 4;
    static_assert(words <= 64, "one word per lane");
    if (blockIdx.x == 0 && lane < words) reinterpret_cast<uint32_t*>(ctl)[lane] = 0u;
}

// ClusterFit block on one lane: its record in slot r, and its key.
template <int FMT, int ALG>
__device__ __forceinline__ uint32_t write_record_lane(ClusterRec* __restrict__ recs, uint32_t r,
                                                      const LaneSet& S, const uint32_t (&out)[4],
                                                      float vx, float vy, float vz, const FitParams& fp, uint32_t tex_idx, uint32_t block)
{
    const bool need4 = !(FMT == BC1 && S.transparent);
    const uint32_t info = (uint32_t)S.n | ((S.transparent ? 1u : 0u) << 8) | ((uint32_t)FMT << 12) |
                          ((ALG == ITERATIVE_CLUSTER_FIT ? 8u : 1u) << 16);
    uint4* const q = reinterpret_cast<uint4*>(recs + r);
#pragma unroll
    for (int p = 0; p < 16; p += 4) q[p / 4] = make_uint4(S.pix(p), S.pix(p + 1), S.pix(p + 2), S.pix(p + 3));
#pragma unroll
    for (int p = 0; p < 16; p += 4)
        q[4 + p / 4] = make_uint4(__float_as_uint(S.wt(p)), __float_as_uint(S.wt(p + 1)), __float_as_uint(S.wt(p + 2)),
                                  __float_as_uint(S.wt(p + 3)));
    q[8] = make_uint4((uint32_t)S.lowest, (uint32_t)(S.lowest >> 32), S.first | (S.inc << 16), info);
    q[9] = make_uint4(out[0], out[1], __float_as_uint(vx), __float_as_uint(vy));
    q[10] = make_uint4(__float_as_uint(vz), __float_as_uint(FLT_MAX), __float_as_uint(fp.wr), __float_as_uint(fp.wg));
    q[11] = make_uint4(__float_as_uint(fp.wb), tex_idx, block, 0u);
    // ClusterFit: list C (all of the block's searches in one pass);
    // IterativeClusterFit: the 3-colour search for BC1 (list A) and the
    // 4-colour one unless transparent (list B)
    uint32_t key = (uint32_t)S.n;
    if (ALG == CLUSTER_FIT) {
        key |= key_bit(kListC);
    } else {
        if (FMT == BC1) key |= key_bit(kListA);
        if (need4) key |= key_bit(kListB);
    }
    return key;
}

// Blocks [first, first + count) of one texture, one per lane, 64 at a time.
// Single-colour and range-fit blocks are finished here; ClusterFit blocks
// become records in slots [slot0, slot0 + count).  Block
// b of the pixel grid (a texture, or a level of a chain) is block b + block0 of
// the output.
struct PixelGrid {
    const uint8_t* rgba;
    uint32_t width, height, blocks_wide;
};

template <int FMT, int ALG, class Grid>
__device__ __forceinline__ void classify_chunk(const Grid& G, const BatchTex& T, uint32_t tex_idx, uint32_t first, uint32_t count,
                                               uint32_t slot0, uint32_t block0, const LaneTables& LT, LaneBlockLds& LB, int lane,
                                               ClusterRec* recs, uint32_t* keys)
{
    const FitParams fp{T.wr, T.wg, T.wb, T.weigh_alpha};
    for (uint32_t off = 0; off < count; off += 64) {
        const uint32_t k = off + (uint32_t)lane;
        uint32_t key = 0;
        if (k < count) {
            const uint32_t b = first + k;
            uint32_t px[16];
            const uint32_t valid = fetch_block_lane(G.rgba, G.width, G.height, b % G.blocks_wide,
                                                    b / G.blocks_wide, px);
            uint32_t w[4];
            LaneSet S;
            float vx, vy, vz;
            const int kind = encode_front_lane<FMT, ALG>(px, valid, fp, LT, LB, lane, w, S, vx, vy, vz);
            if (kind == KIND_CLUSTER) {
                key = write_record_lane<FMT, ALG>(recs, slot0 + k, S, w, vx, vy, vz, fp, tex_idx, block0 + b);
            } else if (FMT == BC1) {
                *reinterpret_cast<uint2*>(T.out + ((size_t)block0 + b) * 8u) = make_uint2(w[0], w[1]);
            } else {
                *reinterpret_cast<uint4*>(T.out + ((size_t)block0 + b) * 16u) = make_uint4(w[0], w[1], w[2], w[3]);
            }
            keys[slot0 + k] = key;
        }
    }
}

// Classify over the heavy chunks (BC1/BC2/BC3 textures) of a batch, each
// workgroup taking chunks blockIdx.x, blockIdx.x + gridDim.x, ...  A chunk
// covers blocks [first, first + count) of one texture and record slots
// [slot0, slot0 + count).
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void k_pipe_classify(
    const BatchTex* __restrict__ tex, const uint4* __restrict__ chunks, uint32_t nchunks,
    ClusterRec* __restrict__ recs, uint32_t* __restrict__ keys, PipeCtl* __restrict__ ctl)
{
    __shared__ LaneTables LT;
    __shared__ LaneBlockLds LB;
    const int lane = (int)threadIdx.x;
    clear_counters(ctl, lane);
    fill_lane_tables(LT, lane);
    group_sync();
    // chunks hold similar work, so a plain grid-stride loop balances them
    // (a shared work counter would serialise thousands of atomics at launch)
    for (uint32_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
        const uint4 ch = chunks[c];
        const BatchTex& T = tex[ch.x];
        switch (T.variant) {
        case 0: classify_chunk<BC1, RANGE_FIT>(T, T, ch.x, ch.y, ch.z, ch.w, 0u, LT, LB, lane, recs, keys); break;
        case 1: classify_chunk<BC1, CLUSTER_FIT>(T, T, ch.x, ch.y, ch.z, ch.w, 0u, LT, LB, lane, recs, keys); break;
        case 2: classify_chunk<BC1, ITERATIVE_CLUSTER_FIT>(T, T, ch.x, ch.y, ch.z, ch.w, 0u, LT, LB, lane, recs, keys); break;
        case 3: classify_chunk<BC2, RANGE_FIT>(T, T, ch.x, ch.y, ch.z, ch.w, 0u, LT, LB, lane, recs, keys); break;
        case 4: classify_chunk<BC2, CLUSTER_FIT>(T, T, ch.x, ch.y, ch.z, ch.w, 0u, LT, LB, lane, recs, keys); break;
        case 5: classify_chunk<BC2, ITERATIVE_CLUSTER_FIT>(T, T, ch.x, ch.y, ch.z, ch.w, 0u, LT, LB, lane, recs, keys); break;
        case 6: classify_chunk<BC3, RANGE_FIT>(T, T, ch.x, ch.y, ch.z, ch.w, 0u, LT, LB, lane, recs, keys); break;
        case 7: classify_chunk<BC3, CLUSTER_FIT>(T, T, ch.x, ch.y, ch.z, ch.w, 0u, LT, LB, lane, recs, keys); break;
        default: classify_chunk<BC3, ITERATIVE_CLUSTER_FIT>(T, T, ch.x, ch.y, ch.z, ch.w, 0u, LT, LB, lane, recs, keys); break;
        }
    }
}

// The same for one texture, or the levels of a chain: chunks of chunk_blocks
// blocks, none of them over two levels; slots and output blocks count through
// the chain.  A kernel of its own per format and algorithm: the batch kernel
// holds nine variants.
template <int FMT, int ALG>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void k_pipe_classify_one(
    BatchTex tex0, txk::ChainTable chain, uint32_t nchunks, uint32_t chunk_blocks, ClusterRec* __restrict__ recs,
    uint32_t* __restrict__ keys, PipeCtl* __restrict__ ctl)
{
    __shared__ LaneTables LT;
    __shared__ LaneBlockLds LB;
    const int lane = (int)threadIdx.x;
    clear_counters(ctl, lane);
    fill_lane_tables(LT, lane);
    group_sync();
    for (uint32_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
        PixelGrid G{tex0.rgba, tex0.width, tex0.height, tex0.blocks_wide};
        uint32_t f = c * chunk_blocks, n = tex0.nblocks, block0 = 0;
        if (chain.count) {
            const uint32_t k = chain_level(chain, c);
            const txk::ChainTable::Level& v = chain.level[k];
            f = (c - chain.first[k]) * chunk_blocks;
            n = v.nblocks;
            block0 = v.block0;
            G = PixelGrid{v.rgba, v.width, v.height, v.blocks_wide};
        }
        classify_chunk<FMT, ALG>(G, tex0, 0u, f, min(chunk_blocks, n - f), block0 + f, block0, LT, LB, lane, recs,
                                 keys);
    }
}

// Where position p of a part lies in its list's arrays of nslots entries.
__device__ __forceinline__ size_t part_at(uint32_t part, uint32_t p, uint32_t nslots)
{
    return (size_t)(part >> 1) * nslots + (part & 1u ? nslots - 1u - p : p);
}

// The records of one slot segment into the lists: a counting sort by colour
// count, 16 first, in LDS, and a range of each part reserved with one atomic.
// A part is thus sorted run by run, not as a whole; a whole sort took a
// histogram in the classify pass, its reset and a sum over its copies here
// (reset 4.5 us, bin 11, against 7 now).
__global__ __launch_bounds__(256) void k_pipe_bin(const uint32_t* __restrict__ keys, uint32_t nslots,
                                                  PipeCtl* __restrict__ ctl, uint32_t* __restrict__ list_a,
                                                  uint32_t* __restrict__ list_b, uint32_t* __restrict__ list_c)
{
    constexpr uint32_t kPer = txp::kBinSeg / 256, kParts = txp::kListParts;
    __shared__ uint32_t cnt[kLists][17], off[kLists][17], base[kLists][kParts];
    uint32_t* const lists[kLists] = {list_a, list_b, list_c};
    const uint32_t t = threadIdx.x;
    if (t < kLists * 17) (&cnt[0][0])[t] = 0u;
    uint32_t key[kPer], rank[kPer][kLists];
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
        const uint64_t r = (uint64_t)blockIdx.x * txp::kBinSeg + i * 256u + t;
        key[i] = r < nslots ? keys[r] : 0u;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i)
        for (int k = 0; k < kLists; ++k)
            if (key[i] & key_bit(k)) rank[i][k] = atomicAdd(&cnt[k][key[i] & 31u], 1u);
    __syncthreads();
    // the second wave reserves the ranges while the first sums, for each
    // count, the larger ones of its part
    if (t >= 64u && t < 64u + kLists * kParts) {
        const uint32_t k = (t - 64u) / kParts, part = (t - 64u) % kParts;
        uint32_t n = 0;
#pragma unroll
        for (uint32_t m = 0; m <= 16; ++m) n += txp::part_of(m) == part ? cnt[k][m] : 0u;
        base[k][part] = n ? atomicAdd(&ctl->count[k][part], n) : 0u;
    } else if (t < kLists * 17) {
        const uint32_t k = t / 17u, n = t % 17u;
        uint32_t sum = 0;
#pragma unroll
        for (uint32_t m = 1; m <= 16; ++m) sum += m > n && txp::part_of(m) == txp::part_of(n) ? cnt[k][m] : 0u;
        off[k][n] = sum;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
        const uint32_t r = blockIdx.x * txp::kBinSeg + i * 256u + t, n = key[i] & 31u;
        const uint32_t part = txp::part_of(n);
        for (int k = 0; k < kLists; ++k)
            if (key[i] & key_bit(k)) lists[k][part_at(part, base[k][part] + off[k][n] + rank[i][k], nslots)] = r;
    }
}

// One list as a search reads it.
struct RecList {
    const uint32_t* __restrict__ slots;
    uint32_t nslots, end[txp::kListParts];  // end: positions up to and with each part

    __device__ RecList(const uint32_t* s, uint32_t n, const PipeCtl* __restrict__ ctl, int k) : slots(s), nslots(n)
    {
        uint32_t sum = 0;
        for (uint32_t i = 0; i < txp::kListParts; ++i) end[i] = sum += ctl->count[k][i];
    }
    __device__ uint32_t total() const { return end[txp::kListParts - 1]; }
    // Record slot at position p < total().
    __device__ uint32_t at(uint32_t p) const
    {
        uint32_t part = 0, start = 0;
#pragma unroll
        for (uint32_t i = 0; i + 1 < txp::kListParts; ++i) {
            const bool past = p >= end[i];
            part = past ? i + 1 : part;
            start = past ? end[i] : start;
        }
        return slots[part_at(part, p - start, nslots)];
    }
};

// The block of record R into its group's LDS: lane l writes the point that
// pixel l opens, if it does (colourset.rs:45-97 in pixel order).  Returns the
// pixel's point index, -1 when it is excluded.
__device__ __forceinline__ int load_points(const ClusterRec& R, GroupLds& L, int l)
{
    const uint32_t first = R.masks & 0xFFFFu, inc = R.masks >> 16;
    if ((first >> l) & 1u) {
        float x, y, z;
        rgb_point(R.px[l], x, y, z);
        L.pts[__popc(first & ((1u << l) - 1u))] = make_float4(x, y, z, R.wt[l]);
    }
    const uint32_t low = (R.lowest[l >> 3] >> (4 * (l & 7))) & 15u;
    return (inc >> l) & 1u ? __popc(first & ((1u << low) - 1u)) : -1;
}

// A searched block's state that the split loops do not read, in GroupLds::keep
// (the loops hold most of the 128 registers of a lane): its output fields,
// read with the rest of the record when the group takes it (not behind a load
// at emit time), its record slot, and three words that hold the principal axis
// until the first ordering is built, then the best split's endpoints and key.
enum { kKeepTex = 0, kKeepBlock = 1, kKeepHalf = 2, kKeepRec = 4, kKeepAxis = 5, kKeepEnds = 5, kKeepKey = 7 };

// Result of a finished block: the output block, or (NC = 3 for an opaque BC1
// block) the 3-colour result kept in the record for the 4-colour pass.
template <int NC>
__device__ __forceinline__ void emit_block(const BatchTex* __restrict__ tex, const BatchTex& tex0,
                                           ClusterRec* __restrict__ recs, uint32_t info, const GroupLds& L, int l,
                                           int n, int remap, float lb_err, float thr, int lb_it)
{
    const uint32_t fmt = (info >> 12) & 15u;
    uint32_t lo = 0, hi = 0;
    const bool won = lb_err < thr;
    if (won) {
        write_packed(NC == 4, L.keep[kKeepEnds], L.keep[kKeepEnds + 1],
                     split_index<NC>(L, n, remap, L.keep[kKeepKey], lb_it), l, lo, hi);
    } else if (NC == 4 && fmt == BC1) {
        lo = L.keep[kKeepHalf];  // compress3's block
        hi = L.keep[kKeepHalf + 1];
    }
    if (l == 0) {
        uint8_t* const out = tex_at(tex, tex0, L.keep[kKeepTex]).out;
        const size_t block = L.keep[kKeepBlock];
        if (NC == 3) {
            if ((info >> 8) & 1u) {
                *reinterpret_cast<uint2*>(out + block * 8u) = make_uint2(lo, hi);
            } else {
                ClusterRec& R = recs[L.keep[kKeepRec]];
                R.fit3_err = won ? lb_err : thr;
                R.half[0] = lo;
                R.half[1] = hi;
            }
        } else if (fmt == BC1) {
            *reinterpret_cast<uint2*>(out + block * 8u) = make_uint2(lo, hi);
        } else {
            *reinterpret_cast<uint4*>(out + block * 16u) =
                make_uint4(L.keep[kKeepHalf], L.keep[kKeepHalf + 1], lo, hi);
        }
    }
}

// Lane 0's value of v (the lane that took a wave's list positions).
__device__ __forceinline__ uint32_t lane0(uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, 0); }

// Takes `nwant` (1..4) list positions for one wave from its workgroup's run
// [next, end), packed as (end << 32) | next in LDS and shared by the
// workgroup's 16 groups.  Executed by one lane.  A wave that finds the run
// empty takes the refill lock, reserves the next `refill` positions from
// the shared cursor and installs them; the other waves wait for the lock
// to drop (its holder waits on nothing).  The positions come in up to
// nwant consecutive pieces and are returned in order in pos[0..nwant).
// Positions past the list's end are handed out like any other; their
// groups go idle.
__device__ __forceinline__ void take_positions(uint64_t* run, uint32_t* refilling, uint32_t* __restrict__ cursor,
                                               uint32_t cursor_base, uint32_t refill, uint32_t nwant,
                                               uint32_t (&pos)[4])
{
    uint32_t got = 0;
    while (got < nwant) {
        uint64_t w = __hip_atomic_load(run, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
        const uint32_t next = (uint32_t)w, end = (uint32_t)(w >> 32);
        if (next < end) {
            const uint32_t k = min(nwant - got, end - next);
            if (__hip_atomic_compare_exchange_strong(run, &w, ((uint64_t)end << 32) | (next + k), __ATOMIC_ACQ_REL,
                                                     __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP)) {
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i)
                    if (i >= got && i < got + k) pos[i] = next + (i - got);
                got += k;
            }
            continue;
        }
        uint32_t unlocked = 0u;
        if (__hip_atomic_compare_exchange_strong(refilling, &unlocked, 1u, __ATOMIC_ACQ_REL, __ATOMIC_ACQUIRE,
                                                 __HIP_MEMORY_SCOPE_WORKGROUP)) {
            // only the lock holder installs a run, and no taker changes an
            // empty one, so a run still empty here stays empty until the store
            w = __hip_atomic_load(run, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
            if ((uint32_t)w >= (uint32_t)(w >> 32)) {
                const uint32_t fresh = atomicAdd(cursor, refill) + cursor_base;
                __hip_atomic_store(run, ((uint64_t)(fresh + refill) << 32) | fresh, __ATOMIC_RELEASE,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            __hip_atomic_store(refilling, 0u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        } else {
            __builtin_amdgcn_s_sleep(1);
        }
    }
}

// Persistent search: each 16-lane group pulls records and runs the block's
// ordering iterations independently (cluster.rs:174-249 / 301-389).  NC = 3:
// BC1's compress3, whose result goes to the record (or, for a BC1 block with
// transparent pixels, straight to the output).  NC = 4: compress4 from the
// 3-colour result (BC1) or from nothing (BC2/BC3), then the output block.
//
// Each step has two phases.  Ordering phase: groups without a pending search
// build their next ordering; an ordering equal to an earlier one ends that
// block at once (cluster.rs:176-178, 303-305), and the group pulls its next record and
// tries again, so no group enters the search phase empty-handed while records
// remain.  Search phase: every group with a fresh ordering evaluates its
// candidate splits; the candidate loop runs as long as the largest colour
// count among them needs, and the records are sorted by colour count.
//
// A workgroup is kSearchWaves waves (4 groups each) sharing one run of list
// positions: a group takes one position at a time from it, so near the end
// of the list no group holds records that an idle group could have taken,
// while the shared cursor still sees one atomic per 16 positions.  The waves
// are otherwise independent (no workgroup barrier after the set-up).
template <int NC>
__global__ __launch_bounds__(64 * kSearchWaves) __attribute__((amdgpu_waves_per_eu(4))) void k_pipe_search(
    const BatchTex* __restrict__ tex, BatchTex tex0, ClusterRec* __restrict__ recs, const uint32_t* __restrict__ slots,
    uint32_t nslots, PipeCtl* __restrict__ ctl)
{
    constexpr int kList = NC == 3 ? kListA : kListB;
    const RecList list(slots, nslots, ctl, kList);
    uint32_t* const cursor = &ctl->cursor[kList];
    __shared__ GroupLds lds[4 * kSearchWaves];
    __shared__ uint64_t run;
    __shared__ uint32_t refilling;
    const int lane = (int)(threadIdx.x & 63u), g = lane >> 4, l = lane & 15;
    GroupLds& L = lds[4 * (threadIdx.x >> 6) + g];
    const uint32_t total = list.total();
    // refills of kRefill positions: at most one per group of the workgroup
    // and at most the records per wave, so a short list still spreads over
    // every workgroup; the first run of each workgroup is fixed by its index
    // (no atomic burst at launch) and refills come from the shared cursor,
    // offset past those runs
    const uint32_t kRefill = min(16u, max(4u, total / (kSearchWaves * gridDim.x)));
    const uint32_t kFirst = kSearchWaves * kRefill;
    const uint32_t cursor_base = gridDim.x * kFirst;
    if (threadIdx.x == 0) {
        const uint32_t first = blockIdx.x * kFirst;
        run = ((uint64_t)(first + kFirst) << 32) | first;
        refilling = 0u;
    }
    __syncthreads();

    bool idle = false, need = true, ready = false;
    uint32_t info = 0;
    int it = 0, lb_it = 0, remap = -1;
    float thr = FLT_MAX, lb_err = FLT_MAX;
    FitParams fp{0.0f, 0.0f, 0.0f, 0u};
    for (;;) {
        // ---- ordering phase
        for (;;) {
            // groups without a block take the next record
            if (wave_any(need && !idle)) {
                const bool take = need && !idle;
                const uint64_t want = __ballot(take && l == 0);
                const uint32_t nwant = (uint32_t)__popcll(want);
                const uint32_t rank = (uint32_t)__popcll(want & ((1ull << (uint32_t)(g * 16)) - 1ull));
                uint32_t pos[4] = {0u, 0u, 0u, 0u};
                if (lane == 0) take_positions(&run, &refilling, cursor, cursor_base, kRefill, nwant, pos);
                const uint32_t p0 = lane0(pos[0]), p1 = lane0(pos[1]), p2 = lane0(pos[2]), p3 = lane0(pos[3]);
                const uint32_t p = rank == 0u ? p0 : rank == 1u ? p1 : rank == 2u ? p2 : p3;
                if (take) {
                    if (p >= total) {
                        idle = true;
                    } else {
                        const uint32_t r = list.at(p);
                        const ClusterRec& R = recs[r];
                        remap = load_points(R, L, l);
                        info = R.info;
                        fp = FitParams{R.w[0], R.w[1], R.w[2], 0u};
                        thr = NC == 4 ? R.fit3_err : FLT_MAX;
                        lb_err = thr;
                        lb_it = 0;
                        it = 0;
                        if (l == 0) {
                            uint4* const keep = reinterpret_cast<uint4*>(L.keep);
                            keep[0] = make_uint4(R.tex, R.block, R.half[0], R.half[1]);
                            keep[1] = make_uint4(r, __float_as_uint(R.axis[0]), __float_as_uint(R.axis[1]),
                                                 __float_as_uint(R.axis[2]));
                        }
                        need = false;
                    }
                }
                group_sync();
            }
            const bool todo = !idle && !ready;
            if (!wave_any(todo)) break;
            const int n = (int)(info & 31u);
            float axx = __uint_as_float(L.keep[kKeepAxis]), axy = __uint_as_float(L.keep[kKeepAxis + 1]),
                  axz = __uint_as_float(L.keep[kKeepAxis + 2]);
            if (it > 0) ends_axis(L.keep[kKeepEnds], L.keep[kKeepEnds + 1], axx, axy, axz);
            const bool unique = ordering_step(L, l, n, todo, it, axx, axy, axz);
            ready = ready || unique;
            const bool repeated = todo && !unique;
            if (wave_any(repeated)) {
                if (repeated) {
                    emit_block<NC>(tex, tex0, recs, info, L, l, n, remap, lb_err, thr, lb_it);
                    need = true;
                }
            }
        }
        if (!wave_any(ready)) break;
        // ---- search phase
        float be;
        uint32_t bc;
        const int n = (int)(info & 31u);
        search_step<NC>(L, l, n, ready, fp, be, bc);
        bool fin = false;
        if (ready) {
            ready = false;
            const bool better = be < lb_err;
            uint32_t sa = 0, sb = 0;  // best_start = best_end = 0 until a split beats the threshold
            if (better) {
                lb_err = be;
                lb_it = it;
                split_endpoints<NC>(L, n, bc, sa, sb);
            }
            if ((better || it == 0) && l == 0) {
                L.keep[kKeepEnds] = sa;
                L.keep[kKeepEnds + 1] = sb;
                L.keep[kKeepKey] = bc;
            }
            fin = lb_it != it || it + 1 >= (int)((info >> 16) & 15u);
            if (!fin) ++it;
        }
        group_sync();
        if (wave_any(fin)) {
            if (fin) {
                emit_block<NC>(tex, tex0, recs, info, L, l, n, remap, lb_err, thr, lb_it);
                need = true;
            }
        }
    }
}

// ClusterFit records (colourfit.rs:44-60 with a single ordering per search,
// cluster.rs:152-417): the four groups of a wave pull a record each and run
// the block's searches on it side by side, exactly as the direct kernel
// does -- compress3 and then, unless the block is transparent, compress4 for
// BC1; compress4 for BC2/BC3.  With one ordering per search there is nothing
// to gain from letting the groups run independently, and for BC1 one pull
// serves both searches.  Records are sorted by colour count, so the four
// candidate loops have the same length.  As in k_pipe_search, the
// workgroup's kSearchWaves waves take their positions, four per step, from
// one shared run, so at the end of the list no wave holds steps that an
// idle wave could have run.
// A list too short for refills of four steps (64 positions a workgroup) has no
// refills: workgroup i of G owns steps i, i + G, i + 2G, ..., and its run
// counts those.  All waves finish a step at about the same time, and refills of
// one step queued on the cursor: 31,000 BC3 records took 139 us, now 88.  With
// full refills the cursor's balance is the better one: 65,000 BC1 and 97,000
// BC2 records take 203 and 250 us with it, 212 and 255 dealt out.
__global__ __launch_bounds__(64 * kSearchWaves) __attribute__((amdgpu_waves_per_eu(4))) void k_pipe_cluster(
    const BatchTex* __restrict__ tex, BatchTex tex0, const ClusterRec* __restrict__ recs,
    const uint32_t* __restrict__ slots, uint32_t nslots, PipeCtl* __restrict__ ctl)
{
    const RecList list(slots, nslots, ctl, kListC);
    uint32_t* const cursor = &ctl->cursor[kListC];
    __shared__ GroupLds lds[4 * kSearchWaves];
    __shared__ uint64_t run;
    __shared__ uint32_t refilling;
    const int lane = (int)(threadIdx.x & 63u), g = lane >> 4, l = lane & 15;
    GroupLds& L = lds[4 * (threadIdx.x >> 6) + g];
    const uint32_t total = list.total();
    // refills of four steps for one wave; the first run of each workgroup is
    // fixed by its index, refills come from the shared cursor, offset past
    // those runs
    const uint32_t kRefill = 16u, kFirst = kSearchWaves * kRefill;
    const uint32_t cursor_base = gridDim.x * kFirst;
    const bool dealt = total < kFirst * gridDim.x;
    if (threadIdx.x == 0) {
        const uint32_t first = dealt ? 0u : blockIdx.x * kFirst;
        run = ((uint64_t)(dealt ? ~0u : first + kFirst) << 32) | first;
        refilling = 0u;
    }
    __syncthreads();
    for (;;) {
        uint32_t pos[4] = {0u, 0u, 0u, 0u};
        if (lane == 0) take_positions(&run, &refilling, cursor, cursor_base, kRefill, 4u, pos);
        const uint32_t p0 = lane0(pos[0]), p1 = lane0(pos[1]), p2 = lane0(pos[2]), p3 = lane0(pos[3]);
        uint32_t p = g == 0 ? p0 : g == 1 ? p1 : g == 2 ? p2 : p3;
        if (dealt) p = ((p >> 2) * gridDim.x + blockIdx.x) * 4u + (p & 3u);
        const bool has = p < total;
        if (!wave_any(has)) break;
        ColourSet cs{0, -1, false};
        FitParams fp{0.0f, 0.0f, 0.0f, 0u};
        float axx = 0.0f, axy = 0.0f, axz = 0.0f;
        uint32_t fmt = BC1;
        if (has) {
            const ClusterRec& R = recs[list.at(p)];
            cs.remap = load_points(R, L, l);
            const uint32_t info = R.info;
            fmt = (info >> 12) & 15u;
            cs.n = (int)(info & 31u);
            cs.transparent = ((info >> 8) & 1u) != 0u;
            fp = FitParams{R.w[0], R.w[1], R.w[2], 0u};
            axx = R.axis[0];
            axy = R.axis[1];
            axz = R.axis[2];
            if (l == 0) *reinterpret_cast<uint4*>(L.keep) = make_uint4(R.tex, R.block, R.half[0], R.half[1]);
        }
        group_sync();
        float best = FLT_MAX;
        uint32_t lo = 0, hi = 0;  // all-zero block if no candidate wins (colourfit.rs:44-60)
        run_cluster<3, 1>(L, cs, l, has && fmt == BC1, axx, axy, axz, fp, best, lo, hi);
        run_cluster<4, 1>(L, cs, l, has && !(fmt == BC1 && cs.transparent), axx, axy, axz, fp, best, lo, hi,
                          has && fmt == BC1);
        if (has && l == 0) {
            const uint4 keep = *reinterpret_cast<const uint4*>(L.keep);  // texture, block, alpha half
            uint8_t* const out = tex_at(tex, tex0, keep.x).out;
            if (fmt == BC1)
                *reinterpret_cast<uint2*>(out + (size_t)keep.y * 8u) = make_uint2(lo, hi);
            else
                *reinterpret_cast<uint4*>(out + (size_t)keep.y * 16u) = make_uint4(keep.z, keep.w, lo, hi);
        }
    }
}

}  // namespace txd

namespace txp {

namespace {

template <int FMT, int ALG>
void launch_classify_one(const PipeLaunch& p, const PipeBufs& b, hipStream_t s)
{
    hipLaunchKernelGGL((txd::k_pipe_classify_one<FMT, ALG>), dim3(p.classify_grid), dim3(64), 0, s, p.tex0, p.chain,
                       p.nchunks, p.chunk_blocks, b.recs, b.keys, b.ctl);
}

hipError_t launch_classify(const PipeLaunch& p, const PipeBufs& b, hipStream_t s)
{
    if (p.d_tex) {
        hipLaunchKernelGGL(txd::k_pipe_classify, dim3(p.classify_grid), dim3(64), 0, s, p.d_tex, p.d_chunks,
                           p.nchunks, b.recs, b.keys, b.ctl);
        return hipGetLastError();
    }
    switch (p.tex0.variant) {
    case 1: launch_classify_one<0, 1>(p, b, s); break;
    case 2: launch_classify_one<0, 2>(p, b, s); break;
    case 4: launch_classify_one<1, 1>(p, b, s); break;
    case 5: launch_classify_one<1, 2>(p, b, s); break;
    case 7: launch_classify_one<2, 1>(p, b, s); break;
    case 8: launch_classify_one<2, 2>(p, b, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_pipeline(const PipeLaunch& p, const PipeBufs& b, hipStream_t s, hipEvent_t* marks)
{
    if (p.nslots > b.capacity || p.nslots > 0xFFFFFFFFull) return hipErrorInvalidValue;
    auto mark = [&](int i) { return marks ? hipEventRecord(marks[i], s) : hipSuccess; };
    if (p.nchunks == 0 || p.nslots == 0) {
        for (int i = 0; i < 5; ++i)
            if (mark(i) != hipSuccess) return hipErrorUnknown;
        return hipGetLastError();
    }
    if (mark(0) != hipSuccess) return hipErrorUnknown;
    // no pass is launched on the counters, keys or lists of one that was not
    hipError_t e = launch_classify(p, b, s);
    if (e != hipSuccess) return e;
    if (mark(1) != hipSuccess) return hipErrorUnknown;
    const uint32_t bin_grid = (uint32_t)((p.nslots + kBinSeg - 1) / kBinSeg);
    const uint32_t search_wgs = (p.search_grid + kSearchWaves - 1) / kSearchWaves;
    hipLaunchKernelGGL(txd::k_pipe_bin, dim3(bin_grid), dim3(256), 0, s, b.keys, (uint32_t)p.nslots, b.ctl, b.list[kListA],
                       b.list[kListB], b.list[kListC]);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (mark(2) != hipSuccess) return hipErrorUnknown;
    if (p.before_search && (e = hipStreamWaitEvent(s, p.before_search, 0)) != hipSuccess) return e;
    if (p.lists & (1u << kListC))
        hipLaunchKernelGGL(txd::k_pipe_cluster, dim3(search_wgs), dim3(64 * kSearchWaves), 0, s, p.d_tex, p.tex0, b.recs,
                           b.list[kListC], (uint32_t)p.nslots, b.ctl);
    if (p.lists & (1u << kListA))
        hipLaunchKernelGGL(txd::k_pipe_search<3>, dim3(search_wgs), dim3(64 * kSearchWaves), 0, s, p.d_tex, p.tex0, b.recs,
                           b.list[kListA], (uint32_t)p.nslots, b.ctl);
    if (mark(3) != hipSuccess) return hipErrorUnknown;
    if (p.lists & (1u << kListB))
        hipLaunchKernelGGL(txd::k_pipe_search<4>, dim3(search_wgs), dim3(64 * kSearchWaves), 0, s, p.d_tex, p.tex0, b.recs,
                           b.list[kListB], (uint32_t)p.nslots, b.ctl);
    if (mark(4) != hipSuccess) return hipErrorUnknown;
    return hipGetLastError();
}

}  // namespace txp
