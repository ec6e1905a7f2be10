// bcn_kernels.hpp -- host-side launch interface of the BC1-BC5 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace txk {

struct EncodeArgs {
    int format;           // tx_format
    int algorithm;        // tx_algorithm
    const uint8_t* rgba;  // device, 4-byte aligned, width*height*4 bytes
    uint32_t width, height;
    uint32_t blocks_wide;
    uint64_t nblocks;  // output blocks; blocks past the image are fully masked
    uint8_t* out;      // device, nblocks * block_size bytes
    float wr, wg, wb;
    uint32_t weigh_alpha;
    bool may_overlap;  // on a caller's stream, where calls on others may run beside this one
    bool over_bus;     // rgba is host memory that the kernels read over the bus
};

// Groups per block of the direct kernels.  A split search on 16 lanes takes a
// wave 17 us (30-100 us for IterativeClusterFit) however few blocks there are;
// on 32 or 64 lanes it takes half or a quarter, but a wave then holds 2 or 1
// blocks and repeats what comes before the search.  Measured us for teams of 1
// / 2 / 4 groups (BC1 ClusterFit): 27.5 / 18.5 / 14.4 at 256 blocks, 28.2 /
// 23.4 / 20.8 at 2304, 27.9 / 23.4 / 24.8 at 3136, 33.8 / 29.0 / 35.2 at 5184,
// 34.2 / 33.9 / 40.3 at 6400.  BC1 and BC3 IterativeClusterFit, several
// searches a block: 120 / 68 / 48 and 99 / 61 / 39 at 256 blocks, 174 / 137 /
// 130 and 174 / 134 / 116 at 9216, 164 / 140 / 150 and 178 / 147 / 136 at
// 12544, 190 / 170 / 190 and 197 / 169 / 168 at 16384.
// Those times are of calls one after another.  A longer team does more work in
// all (its groups repeat the front), which calls that overlap on several
// streams pay for: IterativeClusterFit on 8 streams, us a call for teams of 1 /
// 2 / 4, BC1 37 / 28 / 36 and BC3 46 / 36 / 43 at 7056 blocks, 38 / 31 / 39 and
// 47 / 39 / 48 at 7744, 42 / 39 / 50 and 53 / 47 / 59 at 9216.  So where a call
// may overlap others (a texture on a caller's stream) the line of four lies
// where teams of four still beat single groups on 8 streams; alone, such a call
// of 7168..10240 blocks takes up to 1.3 times as long as with four (BC1 64 -> 71
// us and BC3 70 -> 90 at 7744 blocks, 75 -> 76 and 79 -> 89 at 9216; single
// groups took 121 and 172, 129 and 169).  The other lines are those of calls one
// after another, since what teams of two gain alone is more than they lose on 8
// streams (groups of 1 / 2, alone and on 8: IterativeClusterFit BC3 16,384 blocks
// 147 / 127 and 87 / 90, 30,625 210 / 197 and 151 / 164, BC1 30,625 171 / 150 and
// 109 / 117; ClusterFit BC3 6084 30.8 / 28.0 and 19.0 / 21.5, BC1 34.7 / 30.0 and
// 18.0 / 15.9).  Pictures of few colours have short searches and pay for the front
// alone (8 levels a channel, IterativeClusterFit BC3, groups of 1 / 2 / 4: 5625
// blocks 22.7 / 21.2 / 24.2 and on 8 streams 8.5 / 9.7 / 13.7, 16,384 23.9 / 30.5
// and 14.6 / 22.1).  A chain's one launch, which replaces its levels in series,
// keeps these lines on any stream.
inline int team_groups(int algorithm, uint64_t nblocks, bool may_overlap)
{
    const bool iterative = algorithm == 2;
    if (nblocks <= (iterative ? (may_overlap ? 7168u : 10240u) : 2560u)) return 4;
    return nblocks <= (iterative ? 32768u : 6144u) ? 2 : 1;
}

// RangeFit textures of up to this many blocks take the 16-lane groups, larger
// ones a block per lane.  A wave of 64 blocks takes the time of their longest
// serial chain, 9-10 us however few they are, 3 us more with point weights from
// alpha (each lane then compares its 16 pixels pair by pair) and, for BC3, 3 us
// more with partly masked blocks; a group's time follows its block's colours.
// Measured us, groups / lanes, of seeded noise, and of the same with three
// quarters of its tiles flat ("mixed"):
//   BC1          2304 blocks 10.9 /  9.8, mixed 10.2 / 11.5;  4096 11.1 /  9.8, mixed 10.3 / 9.9
//   BC2          1024 blocks  8.9 /  9.1;  2304  9.4 /  9.1;  4096  9.7 /  9.1
//   BC3          2304 blocks  9.7 / 10.0, mixed  9.6 / 11.4;  4096 10.0 / 10.0;  6400 10.5 /  9.9
//   BC3, a side no multiple of 4
//                6561 blocks 10.5 / 12.4;  9409 13.3 / 12.7, 10,201 mixed 12.3 / 14.2;  12,321 14.3 / 12.7
//   weighed by alpha, BC1 / BC2 / BC3
//                8100 blocks 11.4 / 12.8,  9.9 / 12.0, 10.5 / 12.9;  12,100 12.9 / 12.8, 11.8 / 12.1,
//                13.4 / 13.0;  14,400 16.2 / 12.8, 14.9 / 12.0, 16.3 / 13.0
//   a side below 4, BC1 / BC2
//                 512 blocks  5.9 / 9.4,  5.3 / 8.6;  5000 8.1 / 9.6, 7.5 / 8.8;  10,000 9.6 / 9.3, 9.4 / 8.5
// Pictures of few colours keep the groups ahead to 12,000 blocks and more (BC1
// with 8 levels a channel 6.9 / 11.3 at 2304, 8.5 / 10.1 at 12,100).
// Input read over the bus is fetched 16 bytes at a time by a group and in long
// runs by the lanes, so there the line lies lower (whole host calls, groups /
// lanes: BC1 25.7 / 24.4 at 256 blocks, 26.9 / 25.3 at 576, 28.2 / 25.7 at 1024,
// of few colours 22.1 / 25.2, 23.0 / 25.4 and 23.7 / 26.0; weighed 28.2 / 28.6
// at 1024, 30.6 / 29.4 at 1600; BC3 67.6 / 48.2 at 8281), except for sides below
// 4, whose rows are long (2000 blocks 24.2 / 26.0, 4000 weighed 27.6 / 32.4).
inline uint64_t range_group_blocks(const EncodeArgs& a)
{
    const bool bc3 = a.format == 2;
    if (a.over_bus && a.width >= 4 && a.height >= 4) return a.weigh_alpha ? 1280 : 512;
    if (a.weigh_alpha) return 12288;
    if (bc3 && ((a.width | a.height) & 3u)) return 10240;
    if (a.width < 4 || a.height < 4) return 8192;
    return bc3 ? 5120 : 2560;
}

struct BlockListArgs {
    int format;
    int algorithm;
    const uint8_t* blocks;  // device, 64 bytes (16 RGBA8 pixels) per block
    const uint32_t* masks;  // device, one valid-pixel mask per block
    uint64_t nblocks;
    uint8_t* out;  // device, nblocks * block_size bytes
    float wr, wg, wb;
    uint32_t weigh_alpha;
};

// The levels of a mip chain encoded by one launch; their blocks lie back to
// back in the output, level after level.
constexpr uint32_t kMaxChainLevels = 32;
struct ChainTable {
    struct Level {
        const uint8_t* rgba;  // device, 4-byte aligned
        uint32_t width, height, blocks_wide, nblocks;
        uint32_t block0;  // blocks of the levels before it
    };
    uint32_t count;
    uint32_t first[kMaxChainLevels];  // first workgroup (or chunk) of each level, set by the launcher
    Level level[kMaxChainLevels];

    // Numbers the levels' workgroups of `per_group` blocks; returns how many.
    uint64_t number(uint32_t per_group)
    {
        uint64_t n = 0;
        for (uint32_t k = 0; k < count; ++k) {
            first[k] = (uint32_t)n;
            n += ((uint64_t)level[k].nblocks + per_group - 1) / per_group;
        }
        return n;
    }
};

// One texture of a persistent batch launch, as the device reads it.
struct BatchTex {
    const uint8_t* rgba;
    uint8_t* out;
    uint32_t width, height, blocks_wide, nblocks;
    uint32_t variant;  // 3*format + algorithm (BC4: 9, BC5: 10)
    uint32_t pad;
    float wr, wg, wb;
    uint32_t weigh_alpha;
};

// Blocks per chunk of an alpha-only (BC4/BC5) texture encoded one block per
// lane: 8 steps of 64 blocks.
constexpr uint32_t kLightChunkBlocks = 512;

// Launch shape of the alpha-only kernel.  One block per lane: 4-wave
// workgroups, up to 8 per CU, whose waves take pieces of `steps` steps (1, 2, 4
// or 8) of a chunk: as small as leaves each wave at most one (a whole chunk
// takes a wave 35 us, so a small batch is cut finer).  More pieces than waves
// would be drawn from the counter, whose thousands of atomics take longer than
// the work, so only whole chunks are (BC4, 540,672 blocks in chunks of 512: 117
// us in pieces of one step from the counter, 55 in whole chunks, 35 in pieces of
// two).  Nor is a chunk cut `beside` the lockstep encoder over whole chunks of the
// same batch, whose waves stay where they are placed: thousands of short waves
// that fill the GPU ahead of them leave some SIMDs a wave more than others (12
// textures of four formats, 229,086 colour blocks in 1790 chunks of 128,
// ClusterFit 1125 us with the alpha-only chunks cut, 904 with whole ones, RangeFit
// 394 / 347).  Where the colour chunks are cut as well, the shorter waves are the
// better ones (6 textures, 96,455 colour blocks, RangeFit 135 / 149).  16 lanes
// per block: the LDS encoder's workgroups over whole chunks.
struct AlphaShape {
    uint32_t grid, steps;
    uint32_t pieces(uint32_t nlight) const { return steps ? nlight * (kLightChunkBlocks / 64u / steps) : nlight; }
};
inline AlphaShape alpha_shape(uint32_t cus, uint32_t nlight, uint32_t alpha_lanes, uint32_t groups_per_cu,
                              uint32_t waves_per_group, bool beside = false)
{
    AlphaShape a{0, 0};
    if (alpha_lanes != 16) {
        a.steps = kLightChunkBlocks / 64u;
        while (!beside && a.steps > 1 && 2 * (uint64_t)a.pieces(nlight) <= (uint64_t)cus * 32) a.steps /= 2;
    }
    const uint64_t want = alpha_lanes == 16 ? ((uint64_t)nlight + waves_per_group - 1) / waves_per_group
                                            : ((uint64_t)a.pieces(nlight) + 3) / 4;
    const uint64_t cap = alpha_lanes == 16 ? (uint64_t)cus * groups_per_cu : (uint64_t)cus * 8;
    a.grid = (uint32_t)(want < 1 ? 1 : want < cap ? want : cap);
    return a;
}

// Launch shape of the LDS encoder over `nheavy` chunks, the largest of
// `largest` blocks, with at most max_groups workgroups: with fewer chunks than
// waves each chunk is cut into per_chunk pieces of `span` blocks (a multiple of
// 4) so that more of the waves have work.  `largest` counts the chunks as they
// are: a tuning may name any size up to 2^32 - 4, and sizes this near 2^32 are
// rounded up in 64 bits.
struct HeavyShape {
    uint32_t grid, per_chunk, span;
};
inline HeavyShape heavy_shape(uint64_t max_groups, uint32_t nheavy, uint32_t waves_per_group, uint32_t largest)
{
    const uint64_t quads = largest ? ((uint64_t)largest + 3) / 4 : 1;
    uint64_t per = nheavy ? max_groups * waves_per_group / nheavy : 1;
    per = per < 1 ? 1 : per < quads ? per : quads;
    const uint64_t span = 4 * ((quads + per - 1) / per);
    HeavyShape h;
    h.span = (uint32_t)(span < 0xFFFFFFFCull ? span : 0xFFFFFFFCull);
    h.per_chunk = (uint32_t)((4 * quads + h.span - 1) / h.span);
    const uint64_t want = ((uint64_t)nheavy * h.per_chunk + waves_per_group - 1) / waves_per_group;
    h.grid = (uint32_t)(want < 1 ? 1 : want < max_groups ? want : max_groups);
    return h;
}

// Counter reset + persistent kernels over chunks {texture, first block,
// block count, 0}: the first `nheavy` chunks (any format) go to the LDS
// encoder (workgroups of `waves_per_group` = 1, 2 or 4 waves), the
// next `nlight` (BC4/BC5 only) to the alpha-only launch (launch_alpha_chunks),
// on `s_light` when given (fork/join through the two events) or after the
// heavy kernel on `s`.  d_counter holds two counters.
hipError_t launch_batch_raw(const BatchTex* d_tex, const uint4* d_chunks, uint32_t nheavy, uint32_t nlight,
                            uint32_t* d_counter, HeavyShape heavy, AlphaShape light, uint32_t waves_per_group,
                            uint32_t alpha_lanes, hipStream_t s, hipStream_t s_light, hipEvent_t fork,
                            hipEvent_t join);

// Persistent kernel over the BC4/BC5 chunks [first, first + nlight):
// alpha_lanes = 1 runs one block per lane (k_batch_light, 4-wave
// workgroups); 16 runs a 16-lane group per block (k_batch with
// `waves_per_group` waves per workgroup).  `d_counter` is its work counter
// (not reset here; not used when alpha_needs_counter() says so).
hipError_t launch_alpha_chunks(const BatchTex* d_tex, const uint4* d_chunks, uint32_t first, uint32_t nlight,
                               uint32_t* d_counter, AlphaShape shape, uint32_t alpha_lanes, uint32_t waves_per_group,
                               hipStream_t s);

// Whether the alpha-only kernel draws work from its counter: not when one
// block per lane leaves each wave at most one piece.
inline bool alpha_needs_counter(AlphaShape shape, uint32_t nlight, uint32_t alpha_lanes)
{
    return alpha_lanes == 16 || (uint64_t)shape.pieces(nlight) > (uint64_t)shape.grid * 4;
}

// Counter reset (d_counter[0..1], where it is needed) + the alpha-only kernel
// over chunks [first, first + nlight) on `s`.
hipError_t launch_batch_light(const BatchTex* d_tex, const uint4* d_chunks, uint32_t first, uint32_t nlight,
                              uint32_t* d_counter, AlphaShape shape, uint32_t alpha_lanes, uint32_t waves_per_group,
                              hipStream_t s);

// Clears d_counter[0..1] on `s` (a kernel: replay-safe inside graphs).
hipError_t reset_counters(uint32_t* d_counter, hipStream_t s);

// Launch shapes that keep every grid dimension within its limit (2^32
// work-items in x, 2^16 workgroups in y) whatever the texture size.  The
// one-pass encoders take `groups` workgroups as a 2-D grid of rows of at
// most 2^16 and index workgroup y * gridDim.x + x (a grid-stride loop
// instead made the compiler keep more registers live and cost the lockstep
// kernel a wave per SIMD); the decoder caps its tile grid and walks larger
// images grid-stride; the mip levels take a launch per 2^23 columns of
// tiles (more than one above 2^29 texels wide) and walk rows grid-stride.
constexpr uint64_t kGroupsPerRow = 1ull << 16;
constexpr uint64_t kMaxGroups2d = kGroupsPerRow * 65535ull;
constexpr uint64_t kMaxDecodeTilesX = 1ull << 16;  // 256-block tiles of the decoder per grid row
constexpr uint64_t kMaxDecodeTilesY = 1ull << 14;
constexpr uint64_t kMaxMipTilesX = 1ull << 23;     // 64 x 64 source tiles of the mip levels per grid row
constexpr uint64_t kMaxMipTilesY = 1ull << 14;

inline uint32_t capped_grid(uint64_t groups, uint64_t cap) { return (uint32_t)(groups < cap ? groups : cap); }

inline dim3 grid_2d(uint64_t groups)
{
    const uint64_t x = groups < kGroupsPerRow ? groups : kGroupsPerRow;
    return dim3((uint32_t)x, (uint32_t)((groups + x - 1) / x));
}

hipError_t launch_encode(const EncodeArgs& a, hipStream_t s);
// The same kernels over every level of a chain in one launch: `a` holds the
// format, algorithm, weights, output and the total block count (below 2^32).
hipError_t launch_encode_chain(const EncodeArgs& a, const ChainTable& levels, hipStream_t s);
hipError_t launch_encode_blocks(const BlockListArgs& a, hipStream_t s);
hipError_t launch_decode(int format, const uint8_t* data, uint32_t w, uint32_t h, uint8_t* out, hipStream_t s);
// The elementary-operation check (tx_util_elementary): d_tables holds
// 256 + 17 + 4096 floats; the three per-value outputs hold n entries each.
hipError_t launch_elementary(const float* d_in, uint32_t n, float* d_tables, float* d_snap31, float* d_snap63,
                             int32_t* d_round255, hipStream_t s);
// The reciprocal check (tx_util_reciprocal): n values in and out.
hipError_t launch_reciprocal(const float* d_in, uint32_t n, float* d_out, hipStream_t s);
// Levels 1..nout (1 <= nout <= kMipLevelsPerLaunch) of the RGBA8 image src
// (w x h, 4-byte aligned) back to back into dst: 2x2 box of the level above,
// edge clamp, (sum + 2) >> 2; level k is max(1, w >> k) x max(1, h >> k).
constexpr uint32_t kMipLevelsPerLaunch = 6;
constexpr uint32_t kMipTile = 64;  // source texels per side of a workgroup's tile
// Grid of the launch that starts at tile column col0 (col0 * kMipTile < w).
inline dim3 mip_grid(uint32_t w, uint32_t h, uint64_t col0)
{
    return dim3(capped_grid(((uint64_t)w + kMipTile - 1) / kMipTile - col0, kMaxMipTilesX),
                capped_grid(((uint64_t)h + kMipTile - 1) / kMipTile, kMaxMipTilesY));
}
hipError_t launch_mip_levels(const uint8_t* src, uint32_t w, uint32_t h, uint32_t nout, uint8_t* dst, hipStream_t s);

}  // namespace txk
