// tx_mips.hip -- device mip-chain generation (the step before the encoder
// when a caller needs every level; texpresso itself encodes one level, and
// its CLI writes level 0 only, cli/src/main.rs:148-160).
//
// Level k has size max(1, w >> k) x max(1, h >> k); each texel of level k+1
// is the rounded mean of a 2x2 box of level k with edge clamp,
// (a + b + c + d + 2) >> 2 per channel.  A side larger than 1 halves with its
// odd last texel left out, so a texel of level k depends on the 2^k x 2^k
// texels of level 0 at its place only, and the clamp acts on sides of 1 alone.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bcn_kernels.hpp"

namespace txd {

constexpr uint32_t kTile = txk::kMipTile;  // source texels per side of a workgroup's tile

typedef uint32_t mip4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t mip2 __attribute__((ext_vector_type(2), aligned(4)));

// (a + b + c + d + 2) >> 2 per byte: the even and the odd bytes as two 16-bit
// lanes of a word each.
__device__ __forceinline__ uint32_t mean4(uint32_t a, uint32_t b, uint32_t c, uint32_t d)
{
    constexpr uint32_t m = 0x00FF00FFu;
    const uint32_t e = (a & m) + (b & m) + (c & m) + (d & m) + 0x00020002u;
    const uint32_t o = ((a >> 8) & m) + ((b >> 8) & m) + ((c >> 8) & m) + ((d >> 8) & m) + 0x00020002u;
    return ((e >> 2) & m) | (((o >> 2) & m) << 8);
}

// Levels 1..nout (nout <= 6) of the w x h image src in the columns of tiles
// from col0 on, one 64 x 64 source tile per workgroup: each thread averages 4 x 4 texels into 2 x 2 of level 1 and
// one of level 2, and the tile's 16 x 16 texels of level 2 go down to one
// texel of level 6 through LDS on the first wave.  The levels lie back to
// back in dst.  Bound by memory: the source is read once and no level is read
// back.  4096 x 2048 (45 MB) takes 12.1 us in two launches (3.7 TB/s); one
// dependent launch per level, a texel per thread with four 4-byte loads, took
// 44.6 us.
__global__ __launch_bounds__(256) void k_mip_levels(const uint32_t* __restrict__ src, uint32_t w, uint32_t h,
                                                    uint32_t nout, uint32_t* __restrict__ dst, uint32_t col0)
{
    __shared__ uint32_t lds[16][17];
    const uint32_t tx = threadIdx.x & 15u, ty = threadIdx.x >> 4;
    const uint32_t w1 = max(1u, w >> 1), h1 = max(1u, h >> 1), w2 = max(1u, w1 >> 1), h2 = max(1u, h1 >> 1);
    const uint32_t col = col0 + blockIdx.x, x0 = col * kTile + 4u * tx;
    for (uint64_t tile = blockIdx.y; tile * kTile < h; tile += gridDim.y) {
        const uint32_t y0 = (uint32_t)tile * kTile + 4u * ty;
        uint32_t p[4][4];
        if (x0 + 4u <= w) {
            // past the last row, that row again
#pragma unroll
            for (uint32_t y = 0; y < 4; ++y) {
                const mip4 v = *reinterpret_cast<const mip4*>(src + (size_t)min(y0 + y, h - 1u) * w + x0);
#pragma unroll
                for (uint32_t x = 0; x < 4; ++x) p[y][x] = v[x];
            }
        } else {
#pragma unroll
            for (uint32_t y = 0; y < 4; ++y)
#pragma unroll
                for (uint32_t x = 0; x < 4; ++x)
                    p[y][x] = src[(size_t)min(y0 + y, h - 1u) * w + min(x0 + x, w - 1u)];
        }
        uint32_t a[2][2];
        uint32_t* out = dst;
#pragma unroll
        for (uint32_t y = 0; y < 2; ++y) {
#pragma unroll
            for (uint32_t x = 0; x < 2; ++x)
                a[y][x] = mean4(p[2 * y][2 * x], p[2 * y][2 * x + 1], p[2 * y + 1][2 * x], p[2 * y + 1][2 * x + 1]);
            const uint32_t ox = x0 / 2u, oy = y0 / 2u + y;
            if (oy < h1) {
                uint32_t* const o = out + (size_t)oy * w1 + ox;
                if (ox + 1u < w1) *reinterpret_cast<mip2*>(o) = mip2{a[y][0], a[y][1]};
                else if (ox < w1) o[0] = a[y][0];
            }
        }
        if (nout < 2u) continue;
        // a side of 1 repeats its only row or column
        if (w1 == 1u) a[0][1] = a[0][0], a[1][1] = a[1][0];
        if (h1 == 1u) a[1][0] = a[0][0], a[1][1] = a[0][1];
        const uint32_t c = mean4(a[0][0], a[0][1], a[1][0], a[1][1]);
        out += (size_t)w1 * h1;
        if (x0 / 4u < w2 && y0 / 4u < h2) out[(size_t)(y0 / 4u) * w2 + x0 / 4u] = c;
        if (nout < 3u) continue;
        lds[ty][tx] = c;
        __syncthreads();
        if (threadIdx.x < 64u) {
            // level k from level k-1 in lds: `side` texels a side of the tile
            uint32_t pw = w2, ph = h2;
            for (uint32_t k = 3, side = 8; k <= nout; ++k, side >>= 1) {
                out += (size_t)pw * ph;
                const uint32_t nw = max(1u, pw >> 1), nh = max(1u, ph >> 1);
                const uint32_t lx = threadIdx.x & 7u, ly = threadIdx.x >> 3;
                const uint32_t xb = pw == 1u ? 0u : 1u, yb = ph == 1u ? 0u : 1u;
                const bool in = lx < side && ly < side;
                uint32_t m = 0;
                if (in)
                    m = mean4(lds[2u * ly][2u * lx], lds[2u * ly][2u * lx + xb], lds[2u * ly + yb][2u * lx],
                              lds[2u * ly + yb][2u * lx + xb]);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (in) lds[ly][lx] = m;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                const uint32_t ox = col * side + lx, oy = (uint32_t)tile * side + ly;
                if (in && ox < nw && oy < nh) out[(size_t)oy * nw + ox] = m;
                pw = nw;
                ph = nh;
            }
        }
        __syncthreads();
    }
}

// One level, a texel per thread with four 4-byte loads: where the tiles serve
// badly (mip_levels_apart).
__global__ __launch_bounds__(256) void k_mip_level(const uint32_t* __restrict__ src, uint32_t w, uint32_t h,
                                                   uint32_t* __restrict__ dst, uint32_t nw, uint32_t nh)
{
    const uint32_t x = blockIdx.x * 64u + (threadIdx.x & 63u);
    if (x >= nw) return;
    const uint32_t x0 = min(2u * x, w - 1u), x1 = min(2u * x + 1u, w - 1u);
    for (uint32_t y = blockIdx.y * 4u + (threadIdx.x >> 6); y < nh; y += gridDim.y * 4u) {
        const size_t y0 = (size_t)min(2u * y, h - 1u) * w, y1 = (size_t)min(2u * y + 1u, h - 1u) * w;
        dst[(size_t)y * nw + x] = mean4(src[y0 + x0], src[y0 + x1], src[y1 + x0], src[y1 + x1]);
    }
}

}  // namespace txd

namespace txk {

namespace {

// Whether nout levels of a w x h image go by a launch each.  A tile's threads
// read 16-byte runs, which straddle cache lines when rows start at any 4-byte
// address: where one level is all, so that reading the source once saves
// nothing, a texel per thread is faster (4095 x 2047 8.6 us, 11.0 in tiles; 4096
// x 2048 7.3 and 5.8).  And of an image below 16 rows a tile uses 64 threads or
// fewer, so its time grows with the width where a launch stays at its 3 us (10^6
// x 2, three levels 9.4 us, 19.2 in tiles; 300,000 x 7 9.3 and 7.5, one level 3.6
// and 6.2; 100,000 x 1, three levels 9.5 and 4.1).
bool mip_levels_apart(uint32_t w, uint32_t h, uint32_t nout)
{
    if (w >= 1u << 29) return false;  // the tiles' launches are cut by width
    if (nout == 1 && w >= 64 && (w & 3u)) return true;
    return h < 16 && w >= nout << 18;
}

hipError_t launch_mips_apart(const uint32_t* src, uint32_t w, uint32_t h, uint32_t nout, uint32_t* dst, hipStream_t s)
{
    for (uint32_t k = 0; k < nout; ++k) {
        const uint32_t nw = std::max(1u, w >> 1), nh = std::max(1u, h >> 1);
        const dim3 grid((nw + 63u) / 64u, capped_grid(((uint64_t)nh + 3) / 4, kMaxMipTilesY));
        hipLaunchKernelGGL(txd::k_mip_level, grid, dim3(256), 0, s, src, w, h, dst, nw, nh);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        src = dst;
        dst += (size_t)nw * nh;
        w = nw;
        h = nh;
    }
    return hipSuccess;
}

}  // namespace

hipError_t launch_mip_levels(const uint8_t* src, uint32_t w, uint32_t h, uint32_t nout, uint8_t* dst, hipStream_t s)
{
    if (w == 0 || h == 0 || nout == 0 || nout > kMipLevelsPerLaunch) return hipErrorInvalidValue;
    if (mip_levels_apart(w, h, nout))
        return launch_mips_apart(reinterpret_cast<const uint32_t*>(src), w, h, nout, reinterpret_cast<uint32_t*>(dst),
                                 s);
    for (uint64_t col0 = 0; col0 * kMipTile < w; col0 += kMaxMipTilesX) {
        hipLaunchKernelGGL(txd::k_mip_levels, mip_grid(w, h, col0), dim3(256), 0, s,
                           reinterpret_cast<const uint32_t*>(src), w, h, nout, reinterpret_cast<uint32_t*>(dst),
                           (uint32_t)col0);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace txk
