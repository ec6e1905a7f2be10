// bcn_lane.hpp -- front half of a BC1/BC2/BC3 block with the whole block on
// one lane: alpha, colour set, principal axis, and the single-colour and
// range fits (lib.rs:188-230, colourset.rs:35-112, math.rs:44-97,
// single.rs:100-164, range.rs:44-192).
//
// The 16-lane-group front (encode_front) spreads a block over 16 lanes, which
// suits the colour-set comparisons but repeats every serial fold (centroid,
// covariance, eight power-iteration steps, the range fit's point loops) on
// all 16 lanes.  Here each lane owns one block, so a wave runs 64 blocks and
// each serial step is done once per block.  The arithmetic is the same
// expression for expression: points are visited in point order (first
// occurrence order, i.e. increasing pixel index), so every fold matches.
#pragma once
#include "bcn_device.hpp"

namespace txd {

// sqrtf(count) of the unweighted point weights, filled once per workgroup.
struct LaneTables {
    float sqc[17];
};

__device__ __forceinline__ void fill_lane_tables(LaneTables& T, int lane)
{
    if (lane < 17) T.sqc[lane] = sqrtf((float)lane);
}

// Per-wave LDS of the lane front: the pixels and point weights of every
// lane's block, pixel-major with the lane fastest (each access by the wave is
// 64 consecutive words, free of bank conflicts).  Rolled loops over pixels
// read them here by index.
struct LaneBlockLds {
    uint32_t px[16][64];
    float w[16][64];
};

// The colour set of one block on one lane (colourset.rs:35-112).  Pixels are
// kept in pixel order; a point is the first included pixel of its colour.
struct LaneSet {
    LaneBlockLds* L;
    int lane;
    uint32_t first;     // bit p: pixel p opens a point
    uint32_t inc;       // bit p: pixel p is in the set
    uint64_t lowest;    // nibble p: the lowest pixel of pixel p's colour
    int n;
    bool transparent;

    __device__ uint32_t pix(int p) const { return L->px[p][lane]; }
    __device__ float wt(int p) const { return L->w[p][lane]; }  // sqrt(weight), 0 off the points
};

// Pixel p's colour as a comparison key: its RGB when included, otherwise a
// value no colour has (so it matches nothing).
__device__ __forceinline__ uint32_t colour_key(uint32_t px, uint32_t inc, int p)
{
    return ((inc >> p) & 1u) ? (px & 0xFFFFFFu) : 0x1000000u + (uint32_t)p;
}

// Batcher's odd-even merge sort of 16 values, ascending: 63 compare-exchange
// steps, straight-line once unrolled (the network sorts every 0/1 input, so
// it sorts every input).
__device__ __forceinline__ void sort16(uint32_t (&k)[16])
{
#pragma unroll
    for (int p = 1; p < 16; p <<= 1)
#pragma unroll
        for (int d = p; d >= 1; d >>= 1)
#pragma unroll
            for (int j = d % p; j + d < 16; j += 2 * d)
#pragma unroll
                for (int i = 0; i < d; ++i)
                    if (i + j + d < 16 && (i + j) / (2 * p) == (i + j + d) / (2 * p)) {
                        const uint32_t a = k[i + j], b = k[i + j + d];
                        k[i + j] = min(a, b);
                        k[i + j + d] = max(a, b);
                    }
}

// colourset.rs:35-112 on one lane, unweighted points (weigh_colour_by_alpha
// off): the 16 keys (colour << 4 | pixel; an excluded pixel's colour is a
// value no colour has) sorted put each colour's pixels in one run, lowest
// pixel first.  The run's first pixel opens the colour's point when it is in
// the set (it is the lowest pixel of that colour); every pixel of the run has
// it as its lowest same-colour pixel; the point's weight is sqrtf(run
// length).  Same sets and weights as the pairwise compares of the weighted
// form below.
template <int FMT>
__device__ __forceinline__ void colour_set_lane_sorted(const uint32_t (&px)[16], uint32_t inc, const LaneTables& T,
                                                       LaneBlockLds& L, int lane, LaneSet& S)
{
    uint32_t k[16];
#pragma unroll
    for (int p = 0; p < 16; ++p) k[p] = (colour_key(px[p], inc, p) << 4) | (uint32_t)p;
    sort16(k);
    uint32_t first = 0, head = 0, cnt = 0;
    uint64_t lowest = 0;
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        const uint32_t i = k[s] & 15u;
        const bool start = s == 0 || (k[s] >> 4) != (k[s - 1] >> 4);
        head = start ? i : head;
        cnt = start ? 1u : cnt + 1u;
        const bool in = (inc >> i) & 1u;
        first |= (start && in ? 1u : 0u) << i;
        lowest |= (uint64_t)head << (4 * i);
        // weights: the run's first pixel holds sqrt(pixels so far), so its
        // run's last pixel leaves the full count; every other pixel 0, and an
        // excluded pixel (a run of its own) 0
        L.w[i][lane] = start && in ? T.sqc[1] : 0.0f;
        if (!start) L.w[head][lane] = T.sqc[cnt];
    }
    S.lowest = lowest;
    S.first = first;
    S.n = __popc(first);
}

// colourset.rs:35-112 on one lane.  Unweighted points take the sorted form
// above.  Weighted ones: for each pixel p, same = the pixels with p's colour (p
// included); p opens a point when none of them is lower (a pixel's point index
// counts the points opened below its lowest same-colour pixel), whose weight is
// the sum of (alpha + 1) / 256 over those pixels (exact in binary32), then sqrtf.
template <int FMT>
__device__ __forceinline__ void colour_set_lane(const uint32_t (&px)[16], uint32_t valid, const FitParams& fp,
                                                const LaneTables& T, LaneBlockLds& L, int lane, LaneSet& S)
{
    S.L = &L;
    S.lane = lane;
    uint32_t inc = 0, transp = 0;
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        const uint32_t a = px[p] >> 24;
        const bool v = (valid >> p) & 1u;
        inc |= (v && !(FMT == BC1 && a < 128u) ? 1u : 0u) << p;
        transp |= (v && a < 128u ? 1u : 0u) << p;
        L.px[p][lane] = px[p];
    }
    S.inc = inc;
    S.transparent = FMT == BC1 && transp != 0;
    if (!fp.weigh_alpha) {
        colour_set_lane_sorted<FMT>(px, inc, T, L, lane, S);
        return;
    }
    uint32_t first = 0;
    uint64_t lowest = 0;
    uint32_t keys[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) keys[m] = colour_key(px[m], inc, m);
    // the pixel loop stays rolled (pixel p comes from LDS) and the 16
    // compares against the register copies are unrolled
#pragma unroll 1
    for (int p = 0; p < 16; ++p) {
        const uint32_t kp = colour_key(L.px[p][lane], inc, p);
        uint32_t same = 0, asum = 0;
        // e = 1 when the keys match: keys are below 2^25, so for distinct keys
        // (difference - 1) never has bit 31 set.  (The test is always true here.
        // Without it the compiler orders this block otherwise and what follows
        // lies 4 bytes earlier, by which BC1 RangeFit of 1366 x 767, a wave per
        // SIMD and bound by instruction fetch, took 13.0 us instead of 12.7.)
        if (fp.weigh_alpha) {
#pragma unroll
            for (int m = 0; m < 16; ++m) {
                const uint32_t e = ((kp ^ keys[m]) - 1u) >> 31;
                same |= e << m;
                asum += e * ((px[m] >> 24) + 1u);
            }
        }
        const bool in = (inc >> p) & 1u;
        const bool opens = in && (same & ((1u << p) - 1u)) == 0u;
        first |= (opens ? 1u : 0u) << p;
        lowest |= (uint64_t)__builtin_ctz(same) << (4 * p);
        float w = 0.0f;
        if (opens) w = sqrtf((float)asum / 256.0f);
        L.w[p][lane] = w;
    }
    S.lowest = lowest;
    S.first = first;
    S.n = __popc(first);
}

// math.rs:44-97 over the points of a lane's set (same folds as
// principal_axis).  The folds run over all 16 pixels, unrolled, with the
// colours converted from the pixel registers (a rolled loop over LDS copies
// waits out two LDS reads per step, most of its time): a pixel that opens no
// point has w = 0, so its terms are +0 or -0 and adding them leaves the
// (never negative-zero) accumulators unchanged.
__device__ __forceinline__ void principal_axis_lane(const LaneSet& S, const uint32_t (&px)[16], float& vx, float& vy,
                                                    float& vz)
{
    float total = 0.0f, cx = 0.0f, cy = 0.0f, cz = 0.0f;
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        float x, y, z;
        rgb_point(px[p], x, y, z);
        const float w = S.wt(p);
        total = total + w;
        cx = cx + x * w;
        cy = cy + y * w;
        cz = cz + z * w;
    }
    if (total > FLT_EPSILON) {
        cx = cx / total;
        cy = cy / total;
        cz = cz / total;
    }
    float c0 = 0.0f, c1 = 0.0f, c2 = 0.0f, c3 = 0.0f, c4 = 0.0f, c5 = 0.0f;
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        float x, y, z;
        rgb_point(px[p], x, y, z);
        const float w = S.wt(p);
        const float ax = x - cx, ay = y - cy, az = z - cz;
        const float bx = ax * w, by = ay * w, bz = az * w;
        c0 = c0 + ax * bx;
        c1 = c1 + ax * by;
        c2 = c2 + ax * bz;
        c3 = c3 + ay * by;
        c4 = c4 + ay * bz;
        c5 = c5 + az * bz;
    }
    vx = 1.0f; vy = 1.0f; vz = 1.0f;
#pragma unroll
    for (int it = 0; it < 8; ++it) {
        float wx = c0 * vx, wy = c1 * vx, wz = c2 * vx;
        wx = c1 * vy + wx; wy = c3 * vy + wy; wz = c4 * vy + wz;
        wx = c2 * vz + wx; wy = c4 * vz + wy; wz = c5 * vz + wz;
        const float a = fmaxf(wx, fmaxf(wy, wz));
        const float r = 1.0f / a;
        vx = wx * r; vy = wy * r; vz = wz * r;
    }
}

// colourblock.rs:58-94 with all 16 indices on one lane (pixel p in bits
// 2p..2p+1 of `idx`).
__device__ __forceinline__ void write_packed_lane(bool four, uint32_t a, uint32_t b, uint32_t idx, uint32_t& lo,
                                                  uint32_t& hi)
{
    if (!four) {
        if (a > b) {  // write3: a <= b, swap palette slots 0 and 1
            const uint32_t t = a; a = b; b = t;
            idx ^= ~(idx >> 1) & 0x55555555u;  // 0 <-> 1 where the high bit is clear
        }
    } else {
        if (a < b) {  // write4: a >= b, index ^ 1
            const uint32_t t = a; a = b; b = t;
            idx ^= 0x55555555u;
        } else if (a == b) {
            idx = 0u;
        }
    }
    lo = a | (b << 16);
    hi = idx;
}

// Two index bits per pixel: `in` for pixels of the set, 3 for the others.
__device__ __forceinline__ uint32_t spread_index(uint32_t inc, uint32_t in)
{
    uint32_t m2 = 0;
#pragma unroll
    for (int p = 0; p < 16; ++p) m2 |= ((inc >> p) & 1u ? 3u : 0u) << (2 * p);
    return ((in * 0x55555555u) & m2) | (0xFFFFFFFFu & ~m2);
}

// single.rs:100-164 (same steps as single_fit)
template <int FMT>
__device__ __forceinline__ void single_fit_lane(const LaneSet& S, uint32_t& lo, uint32_t& hi)
{
    // point 0 is the lowest pixel that opens a point; round(255 * (u / 255)) is
    // the byte u again
    const uint32_t q = S.pix(__builtin_ctz(S.first));
    const int cr = (int)(q & 255u), cg = (int)((q >> 8) & 255u), cb = (int)((q >> 16) & 255u);
    uint32_t best = 0xFFFFFFFFu;
    uint32_t s = 0, e = 0, index = 0;
    if (FMT == BC1) {
        const uint32_t err = single_endpoints(0, 1, cr, cg, cb, s, e, index);
        if (err < best) {
            write_packed_lane(false, s, e, spread_index(S.inc, index), lo, hi);
            best = err;
        }
    }
    if (FMT != BC1 || !S.transparent) {
        const uint32_t err = single_endpoints(2, 3, cr, cg, cb, s, e, index);
        if (err < best)
            write_packed_lane(true, s, e, spread_index(S.inc, index), lo, hi);
    }
}

// range.rs:44-192 (same steps as range_fit): the index of every included
// pixel is that of its colour, which is its point's.  The pixel loops are
// unrolled over the pixel registers and free of branches, so that a pixel's
// arithmetic runs beside its neighbours': a range fit is a few thousand
// dependent operations per lane, and a launch of up to 65,536 blocks has one
// wave per SIMD to hide them.
template <int FMT>
__device__ __forceinline__ void range_fit_lane(const LaneSet& S, const uint32_t (&pix)[16], const FitParams& fp,
                                               float px, float py, float pz, uint32_t& lo, uint32_t& hi)
{
    // extremes of the projections over the points, in point order from point
    // 0: a new minimum first, else a new maximum
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, e0 = 0.0f, e1 = 0.0f, e2 = 0.0f;
    float mn = 0.0f, mx = 0.0f;
    bool any = false;
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        float x, y, z;
        rgb_point(pix[p], x, y, z);
        const float d = x * px + y * py + z * pz;
        const bool pt = (S.first >> p) & 1u;
        const bool lower = pt & (!any | (d < mn));
        const bool upper = pt & (!any | (!lower & (d > mx)));
        s0 = lower ? x : s0; s1 = lower ? y : s1; s2 = lower ? z : s2;
        mn = lower ? d : mn;
        e0 = upper ? x : e0; e1 = upper ? y : e1; e2 = upper ? z : e2;
        mx = upper ? d : mx;
        any = any | pt;
    }
    s0 = snap(s0, 31.0f, 1.0f / 31.0f); s1 = snap(s1, 63.0f, 1.0f / 63.0f); s2 = snap(s2, 31.0f, 1.0f / 31.0f);
    e0 = snap(e0, 31.0f, 1.0f / 31.0f); e1 = snap(e1, 63.0f, 1.0f / 63.0f); e2 = snap(e2, 31.0f, 1.0f / 31.0f);

    // range.rs:104-141 for the 3-colour pass (BC1) and the 4-colour pass (not
    // used for BC1 with transparent pixels) in one loop over the pixels: the
    // two codebooks share codes 0 and 1 (the snapped start and end), so each
    // pixel's distances to them are computed once and serve both passes.
    // Each pass keeps its own first strict minimum per pixel (codes in
    // index order) and its own error folded in point order, exactly as two
    // separate passes would.
    const bool do3 = FMT == BC1;
    const bool do4 = !(FMT == BC1 && S.transparent);
    const float t2 = 2.0f / 3.0f, t1 = 1.0f / 3.0f;
    const float h0 = s0 * 0.5f + e0 * 0.5f, h1 = s1 * 0.5f + e1 * 0.5f, h2 = s2 * 0.5f + e2 * 0.5f;
    const float f0 = s0 * t2 + e0 * t1, f1 = s1 * t2 + e1 * t1, f2 = s2 * t2 + e2 * t1;
    const float g0 = s0 * t1 + e0 * t2, g1 = s1 * t1 + e1 * t2, g2 = s2 * t1 + e2 * t2;
    auto dist_to = [&](float x, float y, float z, float cx, float cy, float cz) {
        const float dx = fp.wr * (x - cx);
        const float dy = fp.wg * (y - cy);
        const float dz = fp.wb * (z - cz);
        return dx * dx + dy * dy + dz * dz;
    };
    float error3 = 0.0f, error4 = 0.0f;
    uint32_t idx3 = 0, idx4 = 0;
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        float x, y, z;
        rgb_point(pix[p], x, y, z);
        const float d0 = dist_to(x, y, z, s0, s1, s2);
        const float d1 = dist_to(x, y, z, e0, e1, e2);
        // codes 0 and 1: the first strict minimum starts from FLT_MAX
        float m01 = FLT_MAX;
        uint32_t k01 = 0;
        if (d0 < m01) m01 = d0;
        if (d1 < m01) {
            m01 = d1;
            k01 = 1;
        }
        const bool in = (S.inc >> p) & 1u, pt = (S.first >> p) & 1u;
        if (do3) {
            float dist = m01;
            uint32_t k = k01;
            const float d2 = dist_to(x, y, z, h0, h1, h2);
            if (d2 < dist) {
                dist = d2;
                k = 2;
            }
            idx3 |= (in ? k : 3u) << (2 * p);
            error3 = pt ? error3 + dist : error3;
        }
        {
            float dist = m01;
            uint32_t k = k01;
            const float d2 = dist_to(x, y, z, f0, f1, f2);
            if (d2 < dist) {
                dist = d2;
                k = 2;
            }
            const float d3 = dist_to(x, y, z, g0, g1, g2);
            if (d3 < dist) {
                dist = d3;
                k = 3;
            }
            idx4 |= (in ? k : 3u) << (2 * p);
            error4 = pt ? error4 + dist : error4;
        }
    }
    const uint32_t a = pack_565(s0, s1, s2), b = pack_565(e0, e1, e2);
    float best = FLT_MAX;
    if (do3 && error3 < best) {
        write_packed_lane(false, a, b, idx3, lo, hi);
        best = error3;
    }
    if (do4 && error4 < best) write_packed_lane(true, a, b, idx4, lo, hi);
}

// BC2 alpha of one lane's block (alpha.rs:27-51, same steps as bc2_alpha).
__device__ __forceinline__ void bc2_alpha_lane(const uint32_t (&px)[16], uint32_t valid, uint32_t& lo, uint32_t& hi)
{
    lo = hi = 0u;
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        const float af = (float)(px[p] >> 24) * (15.0f / 255.0f);
        uint32_t q = (uint32_t)f32_to_i32_clamped(af, 15);
        if (!((valid >> p) & 1u)) q = 0;
        if (p < 8) lo |= q << (4 * p);
        else hi |= q << (4 * (p - 8));
    }
}

// Front of one block on one lane: the alpha half in out[0..1] (BC2/BC3),
// the colour set in S, and for single-colour and range-fit blocks the
// finished colour half in out.  Returns the fit kind; for KIND_CLUSTER the
// principal axis comes back in (vx, vy, vz).
template <int FMT, int ALG>
__device__ __forceinline__ int encode_front_lane(const uint32_t (&px)[16], uint32_t valid, const FitParams& fp,
                                                 const LaneTables& T, LaneBlockLds& L, int lane, uint32_t (&out)[4],
                                                 LaneSet& S, float& vx, float& vy, float& vz)
{
    out[0] = out[1] = out[2] = out[3] = 0;
    colour_set_lane<FMT>(px, valid, fp, T, L, lane, S);
    if (FMT == BC2) bc2_alpha_lane(px, valid, out[0], out[1]);
    // BC3 alpha from the pixel registers; a block with masked pixels (the last
    // row and column of an image) takes the rolled form over the LDS copies
    if (FMT == BC3) {
        if (valid == 0xFFFFu) bc3_alpha_full<16>([&](int p) { return (int)(px[p] >> 24); }, out[0], out[1]);
        else bc3_alpha_core<1>([&](int p) { return (int)(S.pix(p) >> 24); }, valid, out[0], out[1]);
    }
    const int kind = S.n == 1 ? KIND_SINGLE : (ALG == RANGE_FIT || S.n == 0) ? KIND_RANGE : KIND_CLUSTER;
    uint32_t lo = 0, hi = 0;
    vx = vy = vz = 0.0f;
    if (kind == KIND_SINGLE) single_fit_lane<FMT>(S, lo, hi);
    if (ALG == RANGE_FIT) {
        if (kind == KIND_RANGE) {
            principal_axis_lane(S, px, vx, vy, vz);
            range_fit_lane<FMT>(S, px, fp, vx, vy, vz, lo, hi);
        }
    } else {
        if (kind == KIND_CLUSTER) principal_axis_lane(S, px, vx, vy, vz);
        if (kind == KIND_RANGE) empty_fit<FMT>(lo, hi);
    }
    set_colour<FMT>(out, lo, hi);
    return kind;
}

}  // namespace txd
