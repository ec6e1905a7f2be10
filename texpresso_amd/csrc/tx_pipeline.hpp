// tx_pipeline.hpp -- the binned ClusterFit pipeline (host-side interface).
//
//   classify -> bin -> search<3> (BC1) -> search<4>
//
// classify: alpha, colour set and fit choice for every block, one block per
//   lane; single-colour and range-fit blocks are finished here, ClusterFit
//   blocks become a ClusterRec.
// bin: the records into one list per pass, many-coloured ones first and
//   neighbours of nearly one distinct-colour count n
//   (list A: BC1 IterativeClusterFit records for the 3-colour search; list
//   B: records that need the 4-colour search -- BC1 IterativeClusterFit
//   without transparency, BC2/BC3 IterativeClusterFit; list C: ClusterFit
//   records of every format, which get all their searches in one pass).
// search<NC>: persistent waves; each 16-lane group pulls the next record
//   from its list and runs that block's ordering iterations on its own, so
//   blocks with one ordering and blocks with several share a wave without
//   waiting for each other, and neighbouring records have about the same n
//   (the same number of candidate rounds).
// cluster: ClusterFit (a single ordering per search): each group pulls a
//   record and runs its searches on it (BC1: 3-colour then 4-colour).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "bcn_kernels.hpp"

namespace txp {

// One ClusterFit block between the passes: three 64-byte pieces, written whole
// by the classify lane that owns the block.  The points stay in pixel order
// as classify holds them; the search's lane l turns pixel l into its point.
struct __align__(64) ClusterRec {
    uint32_t px[16];     // the block's RGBA8 pixels
    float wt[16];        // sqrt(weight) of the point a pixel opens, 0 for the others
    uint32_t lowest[2];  // nibble p: the lowest pixel of pixel p's colour
    uint32_t masks;      // pixels that open a point | pixels of the set << 16
    uint32_t info;       // n | transparent << 8 | format << 12 | iterations << 16
    uint32_t half[2];    // BC2/BC3: alpha half of the block; BC1: ClusterFit::best_compressed after compress3
    float axis[3];       // principal axis
    float fit3_err;      // ClusterFit::best_error after compress3
    float w[3];          // Params::weights
    uint32_t tex;        // texture index
    uint32_t block;      // block index within the texture (or through the chain)
    uint32_t pad;
};
static_assert(sizeof(ClusterRec) == 192, "record layout");
// the classify pass stores the tail as four 16-byte words starting at lowest
static_assert(offsetof(ClusterRec, lowest) == 128 && offsetof(ClusterRec, half) == 144 &&
                  offsetof(ClusterRec, axis) == 152 && offsetof(ClusterRec, fit3_err) == 164 &&
                  offsetof(ClusterRec, w) == 168 && offsetof(ClusterRec, tex) == 180 &&
                  offsetof(ClusterRec, block) == 184,
              "record tail layout");

enum { kListA = 0, kListB = 1, kListC = 2, kLists = 3 };

// The bin pass takes kBinSeg consecutive record slots per workgroup.
constexpr uint32_t kBinSeg = 1024;

// A list's records lie in six parts by colour count, handed out in order: 16
// colours from the front of the list's first array up, 15 from its end down,
// 14 and 13 likewise in the second array, 10-12 and the others in the third.
// So groups of a wave, which draw from runs far apart in the list, nearly
// always search equally long candidate lists, and the long records come
// first.  (IterativeClusterFit search of a 2048^2 texture: 873 us with a list
// sorted as a whole, 890 with six parts, 895 with four, 929 with two; the
// whole sort cost 10 us more before the search.)
constexpr uint32_t kListParts = 6, kListArrays = 3;
constexpr uint32_t part_of(uint32_t n) { return n >= 13u ? 16u - n : n >= 10u ? 4u : 5u; }

// Counters of one pipeline run, cleared by the classify pass (which does not
// use them).
struct PipeCtl {
    uint32_t count[kLists][kListParts];  // records in each part
    uint32_t cursor[kLists];             // positions the search has handed out
};

struct PipeBufs {
    ClusterRec* recs = nullptr;          // capacity records; slot = the block's position among the chunks
    uint32_t* keys = nullptr;            // capacity: n | in list L << (5 + L); 0 = no record
    uint32_t* list[kLists] = {nullptr};  // kListArrays arrays of `capacity` record slots each
    PipeCtl* ctl = nullptr;
    uint64_t capacity = 0;

    // bytes of device memory for `cap` records (one allocation, 256-aligned parts)
    static constexpr size_t bytes_for(uint64_t cap)
    {
        return align256(sizeof(ClusterRec) * cap) + align256(4 * cap) + kLists * align256(4 * kListArrays * cap) +
               align256(sizeof(PipeCtl));
    }
    static constexpr size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }
    // carves the parts out of one allocation of bytes_for(cap) bytes
    void carve(uint8_t* base, uint64_t cap);
};

// Resident waves per CU: classify (single-wave workgroups, one block per
// lane) is limited by registers and LDS (8 KiB of pixel and weight copies
// per workgroup), the searches by LDS and registers (4 x 2544 B per wave,
// so that four search workgroups of kSearchWaves waves take a CU's 160 KiB);
// both fit 4 waves per SIMD.
constexpr uint32_t kClassifyWavesPerCu = 16;
constexpr uint32_t kSearchWavesPerCu = 16;
constexpr uint32_t kSearchWaves = 4;  // waves per search workgroup (sharing one run of list positions)

struct PipeLaunch {
    const txk::BatchTex* d_tex;  // texture descriptors, with d_chunks (null: only `tex0`)
    txk::BatchTex tex0;          // the texture when d_tex is null (ClusterFit or IterativeClusterFit)
    const uint4* d_chunks;       // heavy chunks (texture, first block, count, first record slot) of
                                 // at most kClassifyBlocks blocks; null with d_tex: implicit chunks of tex0
    txk::ChainTable chain;       // count > 0: the levels of a chain, tex0 holding what they share and the
                                 // output; implicit chunks, already numbered
    uint32_t nchunks;            // heavy chunks
    uint32_t chunk_blocks;       // size of the implicit chunks
    uint64_t nslots;             // record slots the chunks cover (<= capacity)
    uint32_t classify_grid;      // persistent 64-thread workgroups of classify
    uint32_t search_grid;        // persistent 64-thread workgroups of each search
    uint32_t lists;              // bit L set: records may go to list L (its search is launched)
    hipEvent_t before_search;    // when given, the searches start after it
};

// Blocks of a chunk that the classify pass takes in one step, one per lane of
// its wave.  Larger chunks are listed as chunks of this size, so that the steps
// are shared out among the workgroups (a small batch tuned with 128-block
// chunks would otherwise leave half the waves idle and take the others twice
// as long) and a large tuned size costs nothing.
constexpr uint32_t kClassifyBlocks = 64;

// The lists a texture's records can go to: ClusterFit -> C; BC1
// IterativeClusterFit -> A and B; BC2/BC3 IterativeClusterFit -> B; RangeFit
// -> none (classify finishes those blocks).
inline uint32_t lists_for(uint32_t format, uint32_t algorithm)
{
    if (algorithm == 0 || format > 2) return 0u;
    if (algorithm == 1) return 1u << kListC;
    return format == 0 ? (1u << kListA) | (1u << kListB) : 1u << kListB;
}

// Launches classify, bin and the searches on `s`.  With `marks`
// (5 events), marks[0] is recorded before classify, marks[1] after it,
// marks[2] after bin, marks[3] after the ClusterFit pass and the 3-colour
// search (recorded even when there are none) and marks[4] after the
// 4-colour search.
hipError_t launch_pipeline(const PipeLaunch& p, const PipeBufs& b, hipStream_t s, hipEvent_t* marks = nullptr);

}  // namespace txp
