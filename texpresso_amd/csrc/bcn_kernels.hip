// bcn_kernels.hip -- kernels and launchers of the BC1-BC5 codec (gfx950).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bcn_device.hpp"
#include "bcn_kernels.hpp"
#include "bcn_lane.hpp"

#pragma clang fp contract(off)

namespace txd {

// ------------------------------------------------------------------ encode

template <int FMT>
__device__ __forceinline__ void store_block(uint8_t* out, uint64_t b, const uint32_t (&w)[4])
{
    if (FMT == BC1 || FMT == BC4)
        *reinterpret_cast<uint2*>(out + b * 8u) = make_uint2(w[0], w[1]);
    else
        *reinterpret_cast<uint4*>(out + b * 16u) = make_uint4(w[0], w[1], w[2], w[3]);
}

// Index of this workgroup in a grid_2d launch (workgroup y * gridDim.x + x;
// below 2^32 since y < 2^16 and x <= 2^16).
__device__ __forceinline__ uint32_t group_index() { return blockIdx.y * gridDim.x + blockIdx.x; }

// One image as the one-pass encoders see it: a texture, or a level of a chain.
struct Image {
    const uint8_t* rgba;
    uint32_t width, height, blocks_wide;
    uint64_t nblocks;
    uint8_t* out;
};

// Level of workgroup `group` and that workgroup's number within the level.
template <int FMT>
__device__ __forceinline__ Image chain_image(const txk::ChainTable& chain, uint8_t* out, uint32_t& group)
{
    const uint32_t k = chain_level(chain, group);
    const txk::ChainTable::Level& v = chain.level[k];
    group -= chain.first[k];
    constexpr size_t bs = FMT == BC1 || FMT == BC4 ? 8u : 16u;
    return Image{v.rgba, v.width, v.height, v.blocks_wide, v.nblocks, out + v.block0 * bs};
}

// One wave per 4 / T consecutive output blocks, each held by T 16-lane groups
// that share its split searches.
template <int FMT, int ALG, int T>
__device__ __forceinline__ void encode_groups(const Image& im, uint32_t group, const FitParams& fp, GroupLds* lds)
{
    const int tid = (int)threadIdx.x, g = tid >> 4, l = tid & 15;
    // the last row of a 2-D grid may hold groups past the texture: all their
    // blocks are not live, as in a part-filled last wave
    const uint64_t b = (uint64_t)group * (4u / T) + (uint64_t)(g / T);
    const bool live = b < im.nblocks;
    const uint32_t bx = live ? (uint32_t)(b % im.blocks_wide) : 0u;
    const uint32_t by = live ? (uint32_t)(b / im.blocks_wide) : 0u;
    bool valid;
    const uint32_t px = fetch_pixel(im.rgba, im.width, im.height, bx, by, live, l, valid);
    uint32_t w[4];
    encode_block<FMT, ALG, T>(px, valid, fp, lds[g], g, l, w);
    if (live && l == 0 && g % T == 0) store_block<FMT>(im.out, b, w);
}

// Plain per-texture launch, and the same over the levels of a chain.
template <int FMT, int ALG, int T>
__global__ __launch_bounds__(64) void k_encode(Image im, FitParams fp)
{
    __shared__ GroupLds lds[4];
    encode_groups<FMT, ALG, T>(im, group_index(), fp, lds);
}

template <int FMT, int ALG, int T>
__global__ __launch_bounds__(64) void k_encode_chain(txk::ChainTable chain, uint8_t* __restrict__ out, FitParams fp)
{
    __shared__ GroupLds lds[4];
    uint32_t group = group_index();
    const Image im = chain_image<FMT>(chain, out, group);
    encode_groups<FMT, ALG, T>(im, group, fp, lds);
}

// BC4 / BC5: one block per lane (alpha codebooks are integer work on 16
// values; a lane's 16 dword loads keep many bytes in flight, and neighbouring
// lanes read neighbouring 16-byte row segments).
template <int FMT>
__device__ __forceinline__ void encode_alpha_lanes(const Image& im, uint32_t group)
{
    const uint64_t b = (uint64_t)group * blockDim.x + threadIdx.x;
    if (b >= im.nblocks) return;
    uint32_t px[16];
    const uint32_t valid = fetch_block_lane(im.rgba, im.width, im.height, (uint32_t)(b % im.blocks_wide),
                                            (uint32_t)(b / im.blocks_wide), px);
    uint32_t w[4];
    encode_alpha_lane<FMT>(px, valid, w);
    store_block<FMT>(im.out, b, w);
}

template <int FMT>
__global__ __launch_bounds__(256) void k_encode_alpha(Image im)
{
    encode_alpha_lanes<FMT>(im, group_index());
}

template <int FMT>
__global__ __launch_bounds__(256) void k_encode_alpha_chain(txk::ChainTable chain, uint8_t* __restrict__ out)
{
    uint32_t group = group_index();
    const Image im = chain_image<FMT>(chain, out, group);
    encode_alpha_lanes<FMT>(im, group);
}

// RangeFit (BC1/BC2/BC3): one block per lane, the front of the pipeline's
// classify pass (alpha, colour set, principal axis, then the single-colour or
// range fit) without its record path.  A RangeFit block is a few thousand
// mostly serial operations; on a 16-lane group every fold would run on all 16
// lanes, which pays below range_group_blocks() only.  Single-wave workgroups (the wave's LDS copies of the
// block pixels and weights): of four waves they were 3-5 % faster where the
// blocks fill whole rounds of the GPU (2048^2 23.6 -> 22.8 us) and 3 % slower
// between (344,000 blocks 31.1 -> 32.0 us).
template <int FMT>
__device__ __forceinline__ void encode_range_lanes(const Image& im, uint32_t group, const FitParams& fp,
                                                   LaneTables& LT, LaneBlockLds& LB)
{
    const int lane = (int)threadIdx.x;
    const uint64_t base = (uint64_t)group * 64u;
    if (base >= im.nblocks) return;
    fill_lane_tables(LT, lane);
    group_sync();
    const uint64_t b = base + (uint64_t)lane;
    if (b < im.nblocks) {
        uint32_t px[16];
        const uint32_t valid = fetch_block_lane(im.rgba, im.width, im.height, (uint32_t)(b % im.blocks_wide),
                                                (uint32_t)(b / im.blocks_wide), px);
        uint32_t w[4];
        LaneSet S;
        float vx, vy, vz;
        encode_front_lane<FMT, RANGE_FIT>(px, valid, fp, LT, LB, lane, w, S, vx, vy, vz);
        store_block<FMT>(im.out, b, w);
    }
}

template <int FMT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void k_encode_range_lane(Image im,
                                                                                                  FitParams fp)
{
    __shared__ LaneTables LT;
    __shared__ LaneBlockLds LB;
    encode_range_lanes<FMT>(im, group_index(), fp, LT, LB);
}

template <int FMT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void k_encode_range_chain(
    txk::ChainTable chain, uint8_t* __restrict__ out, FitParams fp)
{
    __shared__ LaneTables LT;
    __shared__ LaneBlockLds LB;
    uint32_t group = group_index();
    const Image im = chain_image<FMT>(chain, out, group);
    encode_range_lanes<FMT>(im, group, fp, LT, LB);
}

// Explicit block list (Format::compress_block_masked over many blocks): block
// b's 16 pixels are the 64 bytes at blocks + 64*b, its mask is masks[b].  T as
// in k_encode.
template <int FMT, int ALG, int T>
__global__ __launch_bounds__(64) void k_encode_blocks(const uint8_t* __restrict__ blocks,
                                                      const uint32_t* __restrict__ masks, uint64_t nblocks,
                                                      uint8_t* __restrict__ out, FitParams fp)
{
    __shared__ GroupLds lds[4];
    const int tid = (int)threadIdx.x, g = tid >> 4, l = tid & 15;
    const uint64_t b = (uint64_t)group_index() * (4u / T) + (uint64_t)(g / T);
    const bool live = b < nblocks;
    const uint32_t mask = live ? masks[b] : 0u;
    const bool valid = live && ((mask >> l) & 1u);
    const uint32_t px = valid ? reinterpret_cast<const uint32_t*>(blocks + 64 * b)[l] : 0u;
    uint32_t w[4];
    encode_block<FMT, ALG, T>(px, valid, fp, lds[g], g, l, w);
    if (live && l == 0 && g % T == 0) store_block<FMT>(out, b, w);
}

// ------------------------------------------------------------------ decode

// Format::decompress_block (colourblock.rs:96-169, alpha.rs:53-68, 258-304)
// with one block per lane.  A row of four pixels is worked on as four byte
// planes: the row's indices are spread to one per byte and each plane is one
// byte permute of its palette (4 entries for a colour channel, 8 for an alpha
// codebook); eight more permutes turn the planes into four RGBA pixels.

// v / 3, v / 5, v / 7 for the interpolated values (v <= 765, 1275, 1785)
__device__ __forceinline__ uint32_t div3(uint32_t v) { return __umul24(v, 21846u) >> 16; }
__device__ __forceinline__ uint32_t div5(uint32_t v) { return __umul24(v, 13108u) >> 16; }
__device__ __forceinline__ uint32_t div7(uint32_t v) { return __umul24(v, 9363u) >> 16; }

__device__ __forceinline__ uint32_t bytes4(uint32_t a, uint32_t b, uint32_t c, uint32_t d)
{
    return a | (b << 8) | (c << 16) | (d << 24);
}

// Four 2-, 3- or 4-bit fields of x, one per byte.
__device__ __forceinline__ uint32_t spread2(uint32_t x)
{
    const uint32_t t = (x | (x << 12)) & 0x000F000Fu;
    return (t | (t << 6)) & 0x03030303u;
}
__device__ __forceinline__ uint32_t spread3(uint32_t x)
{
    const uint32_t t = (x | (x << 10)) & 0x003F003Fu;
    return (t | (t << 5)) & 0x07070707u;
}
__device__ __forceinline__ uint32_t spread4(uint32_t x)
{
    const uint32_t t = (x | (x << 8)) & 0x00FF00FFu;
    return (t | (t << 4)) & 0x0F0F0F0Fu;
}

// alpha.rs:258-304: the codebook of an 8-byte alpha block, entries 0-3 in lo
// and 4-7 in hi, and the 12 index bits of row y.
struct AlphaBlock {
    uint32_t lo, hi, i0, i1;  // indices of rows 0-1 and 2-3 (24 bits each)

    __device__ AlphaBlock(uint32_t w0, uint32_t w1)
    {
        const uint32_t a0 = w0 & 255u, a1 = (w0 >> 8) & 255u;
        uint32_t c[8] = {a0, a1};
        if (a0 <= a1) {
#pragma unroll
            for (uint32_t i = 1; i < 5; ++i) c[1 + i] = div5((5u - i) * a0 + i * a1);
            c[6] = 0u;
            c[7] = 255u;
        } else {
#pragma unroll
            for (uint32_t i = 1; i < 7; ++i) c[1 + i] = div7((7u - i) * a0 + i * a1);
        }
        lo = bytes4(c[0], c[1], c[2], c[3]);
        hi = bytes4(c[4], c[5], c[6], c[7]);
        i0 = (w0 >> 16) | (w1 << 16);
        i1 = w1 >> 8;
    }
    __device__ uint32_t row(int y) const
    {
        const uint32_t i = __builtin_amdgcn_ubfe(y < 2 ? i0 : i1, 12 * (y & 1), 12);
        return __builtin_amdgcn_perm(hi, lo, spread3(i));
    }
};

// colourblock.rs:96-169: the palette of a colour block, one word per channel,
// and its index bits.
struct ColourBlock {
    uint32_t r, g, b, a, idx;

    __device__ ColourBlock(uint32_t ends, uint32_t indices, bool is_bc1) : idx(indices)
    {
        const uint32_t e0 = ends & 0xFFFFu, e1 = ends >> 16;
        const bool three = is_bc1 && e0 <= e1;
        auto channel = [&](uint32_t x, uint32_t y) {
            const uint32_t c2 = three ? (x + y) >> 1 : div3(2u * x + y);
            const uint32_t c3 = three ? 0u : div3(x + 2u * y);
            return bytes4(x, y, c2, c3);
        };
        auto wide5 = [](uint32_t v) { return (v << 3) | (v >> 2); };
        auto wide6 = [](uint32_t v) { return (v << 2) | (v >> 4); };
        r = channel(wide5(e0 >> 11), wide5(e1 >> 11));
        g = channel(wide6((e0 >> 5) & 63u), wide6((e1 >> 5) & 63u));
        b = channel(wide5(e0 & 31u), wide5(e1 & 31u));
        a = three ? 0x00FFFFFFu : 0xFFFFFFFFu;
    }
    __device__ uint32_t select(int y) const { return spread2((idx >> (8 * y)) & 255u); }
};

// 16 bytes stored where only 4-byte alignment is given (the rows of an image
// whose width is no multiple of 4).
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));

// The words of the block at p, which may have any alignment: with p % 4 == m,
// the aligned words around it (each holds at least one of the block's bytes)
// shifted into place.
template <int WORDS>
__device__ __forceinline__ void load_block(const uint8_t* p, uint32_t m, uint32_t (&w)[4])
{
    if (m == 0) {
        if (WORDS == 4) {
            const u32x4_a4 v = *reinterpret_cast<const u32x4_a4*>(p);
            w[0] = v[0]; w[1] = v[1]; w[2] = v[2]; w[3] = v[3];
        } else {
            const u32x2_a4 v = *reinterpret_cast<const u32x2_a4*>(p);
            w[0] = v[0]; w[1] = v[1];
        }
        return;
    }
    const uint32_t* q = reinterpret_cast<const uint32_t*>(p - m);
    uint32_t prev = q[0];
#pragma unroll
    for (int i = 0; i < WORDS; ++i) {
        const uint32_t next = q[i + 1];
        w[i] = __builtin_amdgcn_alignbyte(next, prev, m);
        prev = next;
    }
}

template <int FMT>
__device__ __forceinline__ void decode_block(const uint32_t (&w)[4], uint32_t (&rows)[4][4])
{
    constexpr bool colour = FMT == BC1 || FMT == BC2 || FMT == BC3;
    const ColourBlock C(colour ? w[FMT == BC1 ? 0 : 2] : 0u, colour ? w[FMT == BC1 ? 1 : 3] : 0u, FMT == BC1);
    const AlphaBlock A0(w[0], w[1]), A1(FMT == BC5 ? w[2] : 0u, FMT == BC5 ? w[3] : 0u);
#pragma unroll
    for (int y = 0; y < 4; ++y) {
        uint32_t r, g, b, a = 0xFFFFFFFFu;
        if (colour) {
            const uint32_t sel = C.select(y);
            r = __builtin_amdgcn_perm(0u, C.r, sel);
            g = __builtin_amdgcn_perm(0u, C.g, sel);
            b = __builtin_amdgcn_perm(0u, C.b, sel);
            if (FMT == BC1) a = __builtin_amdgcn_perm(0u, C.a, sel);
            if (FMT == BC2) {
                const uint32_t q = spread4((w[y >> 1] >> (16 * (y & 1))) & 0xFFFFu);
                a = q | (q << 4);
            }
            if (FMT == BC3) a = A0.row(y);
        } else {
            r = A0.row(y);
            g = FMT == BC5 ? A1.row(y) : r;
            b = FMT == BC5 ? 0u : r;
        }
        const uint32_t rg01 = __builtin_amdgcn_perm(g, r, 0x05010400u), rg23 = __builtin_amdgcn_perm(g, r, 0x07030602u);
        const uint32_t ba01 = __builtin_amdgcn_perm(a, b, 0x05010400u), ba23 = __builtin_amdgcn_perm(a, b, 0x07030602u);
        rows[y][0] = __builtin_amdgcn_perm(ba01, rg01, 0x05040100u);
        rows[y][1] = __builtin_amdgcn_perm(ba01, rg01, 0x07060302u);
        rows[y][2] = __builtin_amdgcn_perm(ba23, rg23, 0x05040100u);
        rows[y][3] = __builtin_amdgcn_perm(ba23, rg23, 0x07060302u);
    }
}

// One block per lane; a wave covers 2^shift x 2^(6 - shift) blocks (64 in a
// row unless the image is narrower), so its block loads and the four row
// stores are runs of neighbouring 16-byte pieces.  Bound by memory: 4096^2 BC3
// (84 MB) takes 13.1 us, 6.4 TB/s (the 256 MB last-level cache holds part of
// the pixels); the form with one pixel per lane and byte loads from the block
// took 51.8 us.  Grids smaller than the image walk it grid-stride in both
// directions.
template <int FMT>
__global__ __launch_bounds__(256) void k_decode(const uint8_t* __restrict__ data, uint32_t width, uint32_t height,
                                                uint32_t blocks_wide, uint32_t blocks_high, uint32_t shift,
                                                uint8_t* __restrict__ out)
{
    constexpr uint32_t bs = (FMT == BC1 || FMT == BC4) ? 8u : 16u;
    const uint32_t misaligned = (uint32_t)(uintptr_t)data & 3u;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t lx = lane & ((1u << shift) - 1u), ly = (wave << (6u - shift)) + (lane >> shift);
    const uint32_t step_y = gridDim.y << (8u - shift), step_x = gridDim.x << shift;
    for (uint32_t by = (blockIdx.y << (8u - shift)) + ly; by < blocks_high; by += step_y) {
        for (uint32_t bx = (blockIdx.x << shift) + lx; bx < blocks_wide; bx += step_x) {
            uint32_t w[4], rows[4][4];
            load_block<(int)bs / 4>(data + ((size_t)by * blocks_wide + bx) * bs, misaligned, w);
            decode_block<FMT>(w, rows);
            uint32_t* o = reinterpret_cast<uint32_t*>(out) + (size_t)by * 4u * width + (size_t)bx * 4u;
            const uint32_t nx = min(4u, width - bx * 4u), ny = min(4u, height - by * 4u);
#pragma unroll
            for (uint32_t y = 0; y < 4; ++y) {
                if (y < ny) {
                    if (nx == 4u) {
                        const u32x4_a4 v = {rows[y][0], rows[y][1], rows[y][2], rows[y][3]};
                        *reinterpret_cast<u32x4_a4*>(o) = v;
                    } else {
#pragma unroll
                        for (uint32_t x = 0; x < 3; ++x)
                            if (x < nx) o[x] = rows[y][x];
                    }
                }
                o += width;
            }
        }
    }
}

// The exactly specified elementary operations of the encoder, evaluated by
// the device functions the kernels use, for an exhaustive check against a
// host IEEE binary32 evaluation: u8/255 (unit8), the sqrt(count) table the
// one-block-per-lane front fills (fill_lane_tables), sqrtf(k / 256) of the
// alpha-weighted point weights (k = 1..4096, the range of the summed
// (alpha + 1) values), and for each input value the 5- and 6-bit grid snap
// (snap, range.rs / cluster.rs) and roundf clamped to [0, 255]
// (f32_to_i32_clamped, math.rs:100-102).  tables: 256 + 17 + 4096 floats.
__global__ __launch_bounds__(64) void k_elementary(const float* __restrict__ in, uint32_t n, float* __restrict__ tables,
                                                   float* __restrict__ snap31, float* __restrict__ snap63,
                                                   int32_t* __restrict__ round255)
{
    __shared__ LaneTables T;
    const int lane = (int)threadIdx.x;
    if (blockIdx.x == 0) {
        fill_lane_tables(T, lane);
        group_sync();
        for (int i = lane; i < 256; i += 64) tables[i] = unit8((uint32_t)i);
        if (lane < 17) tables[256 + lane] = T.sqc[lane];
        for (int k = lane + 1; k <= 4096; k += 64) tables[256 + 17 + (k - 1)] = sqrtf((float)k / 256.0f);
    }
    for (uint32_t i = blockIdx.x * 64u + (uint32_t)lane; i < n; i += gridDim.x * 64u) {
        const float v = in[i];
        snap31[i] = snap(v, 31.0f, 1.0f / 31.0f);
        snap63[i] = snap(v, 63.0f, 1.0f / 63.0f);
        round255[i] = f32_to_i32_clamped(v, 255);
    }
}

// recip() of each input, for the same check.
__global__ __launch_bounds__(64) void k_reciprocal(const float* __restrict__ in, uint32_t n, float* __restrict__ out)
{
    for (uint32_t i = blockIdx.x * 64u + threadIdx.x; i < n; i += gridDim.x * 64u) out[i] = recip(in[i]);
}

}  // namespace txd

// ---------------------------------------------------------------- launchers

namespace {

txd::Image image_of(const txk::EncodeArgs& a)
{
    return txd::Image{a.rgba, a.width, a.height, a.blocks_wide, a.nblocks, a.out};
}
txd::FitParams fit_of(const txk::EncodeArgs& a) { return txd::FitParams{a.wr, a.wg, a.wb, a.weigh_alpha}; }

// Workgroups of `per_group` blocks for a texture, or for the levels of a chain
// (which it numbers); 0 when there is nothing to launch or the grid's limit is
// exceeded (`e` says which).
uint64_t groups_for(const txk::EncodeArgs& a, txk::ChainTable* chain, uint32_t per_group, hipError_t& e)
{
    const uint64_t groups = chain ? chain->number(per_group) : (a.nblocks + per_group - 1) / per_group;
    e = groups > txk::kMaxGroups2d ? hipErrorInvalidValue : hipSuccess;
    return e == hipSuccess ? groups : 0;
}

// Every launcher takes the chain by pointer, null for a single texture.
template <int FMT, int ALG, int T>
hipError_t launch_encode_n(const txk::EncodeArgs& a, txk::ChainTable* chain, hipStream_t s)
{
    hipError_t e;
    const uint64_t groups = groups_for(a, chain, 4 / T, e);
    if (groups == 0) return e;
    if constexpr (ALG != 0) {  // a chain's RangeFit blocks are encoded one per lane
        if (chain) {
            hipLaunchKernelGGL((txd::k_encode_chain<FMT, ALG, T>), txk::grid_2d(groups), dim3(64), 0, s, *chain, a.out,
                               fit_of(a));
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((txd::k_encode<FMT, ALG, T>), txk::grid_2d(groups), dim3(64), 0, s, image_of(a), fit_of(a));
    return hipGetLastError();
}

template <int FMT, int ALG>
hipError_t launch_encode_t(const txk::EncodeArgs& a, txk::ChainTable* chain, hipStream_t s)
{
    switch (txk::team_groups(ALG, a.nblocks, a.may_overlap)) {
    case 4: return launch_encode_n<FMT, ALG, 4>(a, chain, s);
    case 2: return launch_encode_n<FMT, ALG, 2>(a, chain, s);
    default: return launch_encode_n<FMT, ALG, 1>(a, chain, s);
    }
}

template <int FMT>
hipError_t launch_encode_range(const txk::EncodeArgs& a, txk::ChainTable* chain, hipStream_t s)
{
    hipError_t e;
    const uint64_t groups = groups_for(a, chain, 64, e);
    if (groups == 0) return e;
    if (chain)
        hipLaunchKernelGGL((txd::k_encode_range_chain<FMT>), txk::grid_2d(groups), dim3(64), 0, s, *chain, a.out,
                           fit_of(a));
    else
        hipLaunchKernelGGL((txd::k_encode_range_lane<FMT>), txk::grid_2d(groups), dim3(64), 0, s, image_of(a),
                           fit_of(a));
    return hipGetLastError();
}

template <int FMT>
hipError_t launch_encode_f(const txk::EncodeArgs& a, txk::ChainTable* chain, hipStream_t s)
{
    switch (a.algorithm) {
    case 0:
        if (!chain && a.nblocks <= txk::range_group_blocks(a)) return launch_encode_n<FMT, 0, 1>(a, nullptr, s);
        return launch_encode_range<FMT>(a, chain, s);
    case 1: return launch_encode_t<FMT, 1>(a, chain, s);
    default: return launch_encode_t<FMT, 2>(a, chain, s);
    }
}

template <int FMT>
hipError_t launch_encode_alpha(const txk::EncodeArgs& a, txk::ChainTable* chain, hipStream_t s)
{
    hipError_t e;
    const uint64_t groups = groups_for(a, chain, 256, e);
    if (groups == 0) return e;
    if (chain)
        hipLaunchKernelGGL((txd::k_encode_alpha_chain<FMT>), txk::grid_2d(groups), dim3(256), 0, s, *chain, a.out);
    else
        hipLaunchKernelGGL((txd::k_encode_alpha<FMT>), txk::grid_2d(groups), dim3(256), 0, s, image_of(a));
    return hipGetLastError();
}

hipError_t launch_encode_any(const txk::EncodeArgs& a, txk::ChainTable* chain, hipStream_t s)
{
    switch (a.format) {
    case 0: return launch_encode_f<0>(a, chain, s);
    case 1: return launch_encode_f<1>(a, chain, s);
    case 2: return launch_encode_f<2>(a, chain, s);
    case 3: return launch_encode_alpha<3>(a, chain, s);
    case 4: return launch_encode_alpha<4>(a, chain, s);
    default: return hipErrorInvalidValue;
    }
}

template <int FMT, int ALG, int T>
hipError_t launch_blocks_n(const txk::BlockListArgs& a, hipStream_t s)
{
    if (a.nblocks > 4 * txk::kMaxGroups2d) return hipErrorInvalidValue;
    const uint64_t groups = (a.nblocks * T + 3) / 4;
    if (groups == 0) return hipSuccess;
    hipLaunchKernelGGL((txd::k_encode_blocks<FMT, ALG, T>), txk::grid_2d(groups), dim3(64), 0, s, a.blocks, a.masks,
                       a.nblocks, a.out, txd::FitParams{a.wr, a.wg, a.wb, a.weigh_alpha});
    return hipGetLastError();
}

template <int FMT, int ALG>
hipError_t launch_blocks_t(const txk::BlockListArgs& a, hipStream_t s)
{
    if constexpr (ALG != 0) {
        const int t = txk::team_groups(ALG, a.nblocks, false);
        if (t == 4) return launch_blocks_n<FMT, ALG, 4>(a, s);
        if (t == 2) return launch_blocks_n<FMT, ALG, 2>(a, s);
    }
    return launch_blocks_n<FMT, ALG, 1>(a, s);
}

template <int FMT>
hipError_t launch_blocks_f(const txk::BlockListArgs& a, hipStream_t s)
{
    switch (a.algorithm) {
    case 0: return launch_blocks_t<FMT, 0>(a, s);
    case 1: return launch_blocks_t<FMT, 1>(a, s);
    default: return launch_blocks_t<FMT, 2>(a, s);
    }
}

template <int FMT>
hipError_t launch_decode_t(const uint8_t* data, uint32_t w, uint32_t h, uint8_t* out, hipStream_t s)
{
    if (w == 0 || h == 0) return hipSuccess;
    const uint32_t bw = (w + 3) / 4, bh = (h + 3) / 4;
    uint32_t shift = 0;  // a wave's row of blocks: the image's width, rounded up to a power of two, at most 64
    while (shift < 6 && (1u << shift) < bw) ++shift;
    const uint64_t tx = 1ull << shift, ty = 1ull << (8 - shift);
    const dim3 grid(txk::capped_grid((bw + tx - 1) / tx, txk::kMaxDecodeTilesX),
                    txk::capped_grid((bh + ty - 1) / ty, txk::kMaxDecodeTilesY));
    hipLaunchKernelGGL((txd::k_decode<FMT>), grid, dim3(256), 0, s, data, w, h, bw, bh, shift, out);
    return hipGetLastError();
}

}  // namespace

namespace txk {

hipError_t launch_encode(const EncodeArgs& a, hipStream_t s) { return launch_encode_any(a, nullptr, s); }

hipError_t launch_encode_chain(const EncodeArgs& a, const ChainTable& levels, hipStream_t s)
{
    ChainTable chain = levels;
    return launch_encode_any(a, &chain, s);
}

hipError_t launch_encode_blocks(const BlockListArgs& a, hipStream_t s)
{
    switch (a.format) {
    case 0: return launch_blocks_f<0>(a, s);
    case 1: return launch_blocks_f<1>(a, s);
    case 2: return launch_blocks_f<2>(a, s);
    case 3: return launch_blocks_t<3, 0>(a, s);
    case 4: return launch_blocks_t<4, 0>(a, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_elementary(const float* d_in, uint32_t n, float* d_tables, float* d_snap31, float* d_snap63,
                             int32_t* d_round255, hipStream_t s)
{
    const uint32_t groups = (uint32_t)std::min<uint64_t>(4096, std::max<uint64_t>(1, ((uint64_t)n + 63) / 64));
    hipLaunchKernelGGL(txd::k_elementary, dim3(groups), dim3(64), 0, s, d_in, n, d_tables, d_snap31, d_snap63,
                       d_round255);
    return hipGetLastError();
}

hipError_t launch_reciprocal(const float* d_in, uint32_t n, float* d_out, hipStream_t s)
{
    const uint32_t groups = (uint32_t)std::min<uint64_t>(4096, std::max<uint64_t>(1, ((uint64_t)n + 63) / 64));
    hipLaunchKernelGGL(txd::k_reciprocal, dim3(groups), dim3(64), 0, s, d_in, n, d_out);
    return hipGetLastError();
}

hipError_t launch_decode(int format, const uint8_t* data, uint32_t w, uint32_t h, uint8_t* out, hipStream_t s)
{
    switch (format) {
    case 0: return launch_decode_t<0>(data, w, h, out, s);
    case 1: return launch_decode_t<1>(data, w, h, out, s);
    case 2: return launch_decode_t<2>(data, w, h, out, s);
    case 3: return launch_decode_t<3>(data, w, h, out, s);
    case 4: return launch_decode_t<4>(data, w, h, out, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace txk
