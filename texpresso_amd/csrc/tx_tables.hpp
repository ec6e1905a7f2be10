// tx_tables.hpp -- compile-time tables for the BC1-BC5 encoder.
//
// Both tables are computed by constexpr functions, so the device copy
// (__constant__) and the host copy are the same bytes by construction.
//
// 1. Single-colour lookup (replaces lib/src/colourfit/single_lut.rs:52-1086).
//    For a channel value t in 0..255 the table gives, per palette slot s in
//    {0, 2}, the quantised endpoints (start, end) and the distance `error`
//    between t and the closest value that slot can reproduce.  The tables are
//    regenerated from the BC1 endpoint expansion: every (start, end) pair is
//    expanded to 8 bits, each palette slot records the first pair that hits a
//    value exactly, and the remaining values are filled by repeated nearest
//    neighbour relaxation (t+1 before t-1), adding 1 to the error per step.
//
// 2. ClusterFit candidate lists (the split loops of
//    lib/src/colourfit/cluster.rs:182-236 and 309-380).  compress4 searches
//    the splits (i, j, k) with 0 <= i < n, i <= j <= n, max(j,1) <= k <= n;
//    compress3 the splits (i, j) with 0 <= i < n, max(i,1) <= j <= n.
//    A split's key, i << 26 | j << 21 | k << 16 (k = 0 for compress3), orders
//    splits as the reference's loops visit them, so the smallest (error, key)
//    is the reference's first strict minimum.
//
//    For one j the splits form a rectangle of i and k values.  The list for n
//    cuts it into tiles of 2 x 2 splits (i, i+1) x (k, k+1), which share what
//    depends on (i, j) or on (j, k) alone, and single splits for the odd row
//    and column.  Both lists are in key order (of a tile's first split).  An
//    entry holds the byte offsets of the prefix-table rows it reads in 16-bit
//    halves:
//      tile:   {soff(i,j) | soff(i+1,j) << 16, soff(j,k) | soff(j,k+1) << 16, key | 16 i}
//      single: {soff(i,j) | soff(j,k) << 16, key | 16 i}
//    (part0 = S[0][i] lives at entry i, and S[0][i+1] right after it).
//    The prefix table S[a][b], a <= b <= 16, is stored compactly: every
//    empty range S[a][a] (all zero) shares offset 0, row 0 (S[0][b], b >= 1)
//    sits at offsets 1..16 so that part0 = S[0][i] is at offset i, and rows
//    a = 1..15 (b = a+1..16) follow: 137 entries in all.
#pragma once
#include <stdint.h>

namespace txt {

constexpr int soff(int a, int b)
{
    return a == b ? 0 : a == 0 ? b : 17 + 16 * (a - 1) - (((a - 1) * a) >> 1) + (b - a - 1);
}
constexpr int kSEntries = 137;  // soff(15, 16) + 1
constexpr int kCand4 = 967;       // compress4 splits for 16 colours
constexpr int kCand3 = 151;       // compress3 splits for 16 colours

constexpr uint32_t split_key(int i, int j, int k)
{
    return ((uint32_t)i << 26) | ((uint32_t)j << 21) | ((uint32_t)k << 16);
}
constexpr int key_i(uint32_t key) { return (int)(key >> 26); }
constexpr int key_j(uint32_t key) { return (int)((key >> 21) & 31u); }
constexpr int key_k(uint32_t key) { return (int)((key >> 16) & 31u); }
constexpr uint32_t kKeyNextI = 1u << 26;  // from (i, j, k) to (i + 1, j, k)
constexpr uint32_t kKeyNextK = 1u << 16;  // from (i, j, k) to (i, j, k + 1)

struct SingleLut {
    uint8_t v[4][256][6];  // [5_3, 6_3, 5_4, 6_4][value][start0,end0,err0,start1,end1,err1]
};

struct SplitTile {
    uint32_t o1, o2, key;
};
struct SplitOne {
    uint32_t o, key;
};
struct SplitList {
    uint16_t start, len;  // entries [start, start + len)
};
struct SplitLists {
    SplitList tiles, ones;
};

// Rows (i) and columns (k) of the rectangle of splits with this j.
constexpr int rect_rows(int n, int j) { return (j < n - 1 ? j : n - 1) + 1; }
constexpr int rect_col0(int j) { return j > 1 ? j : 1; }
constexpr int rect_cols(int n, int j) { return n - rect_col0(j) + 1; }

// Tiles of the n-colour list: as many as fill whole trips of a group's 16
// lanes (the rest of the rectangle stays single splits), and none below
// kTileMinColours, where the tiles' own loop costs what they save (per lane:
// 10 colours 3 tiles and 6 single splits, 9 colours 2 and 6 against 14).
constexpr int kTileMinColours = 10;

constexpr int tiles_for(int n)
{
    int c = 0;
    if (n >= kTileMinColours)
        for (int j = 0; j <= n; ++j) c += (rect_rows(n, j) / 2) * (rect_cols(n, j) / 2);
    return c & ~15;
}
constexpr int splits4_for(int n)
{
    int c = 0;
    for (int j = 0; n > 0 && j <= n; ++j) c += rect_rows(n, j) * rect_cols(n, j);
    return c;
}
constexpr int splits3_for(int n)
{
    int c = 0;
    for (int i = 0; i < n; ++i) c += n - rect_col0(i) + 1;
    return c;
}
constexpr int ones_for(int n) { return splits4_for(n) - 4 * tiles_for(n); }
template <class F>
constexpr int sum_to_16(F f)
{
    int c = 0;
    for (int n = 0; n <= 16; ++n) c += f(n);
    return c;
}
constexpr int kTiles = sum_to_16(tiles_for), kOnes4 = sum_to_16(ones_for), kOnes3 = sum_to_16(splits3_for);
constexpr int kTiles16 = tiles_for(16), kOnes16 = ones_for(16);

struct CandTables {
    SplitTile tile[kTiles];
    SplitOne one4[kOnes4];
    SplitOne one3[kOnes3];
    SplitLists lists4[17], lists3[17];  // by colour count
};

constexpr void build_lut_one(int bits, int colours, uint8_t (&out)[256][6])
{
    int st[3][256] = {}, en[3][256] = {}, er[3][256] = {};
    bool ok[3][256] = {};
    // slots 0 and 2 of the palette are the ones the encoder uses; slot 1 is
    // tracked only to keep the iteration identical in shape
    const int levels = 1 << bits;
    for (int v1 = 0; v1 < levels; ++v1) {
        for (int v2 = 0; v2 < levels; ++v2) {
            const int a = (v1 << (8 - bits)) | (v1 >> (2 * bits - 8));
            const int b = (v2 << (8 - bits)) | (v2 >> (2 * bits - 8));
            const int c2 = colours == 3 ? (a + b) / 2 : (2 * a + b) / 3;
            const int codes[3] = {a, b, c2};
            for (int s = 0; s < 3; ++s) {
                const int t = codes[s];
                if (!ok[s][t]) {
                    ok[s][t] = true;
                    st[s][t] = v1;
                    en[s][t] = v2;
                    er[s][t] = 0;
                }
            }
        }
    }
    for (bool changed = true; changed;) {
        changed = false;
        for (int s = 0; s < 3; ++s) {
            for (int t = 0; t < 256; ++t) {
                for (int q = 0; q < 2; ++q) {
                    const int nt = q == 0 ? t + 1 : t - 1;
                    if (nt < 0 || nt > 255 || !ok[s][nt]) continue;
                    if (!ok[s][t] || er[s][nt] + 1 < er[s][t]) {
                        ok[s][t] = true;
                        st[s][t] = st[s][nt];
                        en[s][t] = en[s][nt];
                        er[s][t] = er[s][nt] + 1;
                        changed = true;
                    }
                }
            }
        }
    }
    for (int t = 0; t < 256; ++t) {
        out[t][0] = (uint8_t)st[0][t];
        out[t][1] = (uint8_t)en[0][t];
        out[t][2] = (uint8_t)er[0][t];
        out[t][3] = (uint8_t)st[2][t];
        out[t][4] = (uint8_t)en[2][t];
        out[t][5] = (uint8_t)er[2][t];
    }
}

constexpr SingleLut make_single_lut()
{
    SingleLut L{};
    build_lut_one(5, 3, L.v[0]);
    build_lut_one(6, 3, L.v[1]);
    build_lut_one(5, 4, L.v[2]);
    build_lut_one(6, 4, L.v[3]);
    return L;
}

// The tiles of the n-colour list, numbered in key order of their first splits:
// `of` is the number of the tile that split (i, j, k) lies in, kTiles if none.
struct TileMap {
    uint16_t no[8][17][9] = {};
    int n = 0;

    constexpr explicit TileMap(int colours) : n(colours)
    {
        int c = 0;
        for (int i = 0; i < n; i += 2)
            for (int j = i; j <= n; ++j)
                for (int k = rect_col0(j); k <= n; k += 2) {
                    const bool whole = i + 1 < rect_rows(n, j) && k + 1 <= n;
                    no[i / 2][j][(k - rect_col0(j)) / 2] = (uint16_t)(whole && c < tiles_for(n) ? c++ : kTiles);
                }
    }
    constexpr int of(int i, int j, int k) const { return no[i / 2][j][(k - rect_col0(j)) / 2]; }
};

constexpr CandTables make_cand_tables()
{
    CandTables T{};
    int nt = 0, n4 = 0, n3 = 0;
    for (int n = 0; n <= 16; ++n) {
        const TileMap map(n);
        T.lists4[n].tiles.start = (uint16_t)nt;
        T.lists4[n].ones.start = (uint16_t)n4;
        T.lists3[n].ones.start = (uint16_t)n3;
        for (int i = 0; i < n; ++i)
            for (int j = i; j <= n; ++j) {
                const uint32_t io = 16u * (uint32_t)i, o1 = 16u * (uint32_t)soff(i, j);
                for (int k = rect_col0(j); k <= n; ++k) {
                    const uint32_t o2 = 16u * (uint32_t)soff(j, k);
                    const bool tiled = map.of(i, j, k) < kTiles;
                    if (tiled && i % 2 == 0 && (k - rect_col0(j)) % 2 == 0)
                        T.tile[nt++] = SplitTile{o1 | (16u * (uint32_t)soff(i + 1, j)) << 16,
                                                 o2 | (16u * (uint32_t)soff(j, k + 1)) << 16, split_key(i, j, k) | io};
                    else if (!tiled)
                        T.one4[n4++] = SplitOne{o1 | o2 << 16, split_key(i, j, k) | io};
                }
                if (j >= 1) T.one3[n3++] = SplitOne{o1, split_key(i, j, 0) | io};
            }
        T.lists4[n].tiles.len = (uint16_t)(nt - T.lists4[n].tiles.start);
        T.lists4[n].ones.len = (uint16_t)(n4 - T.lists4[n].ones.start);
        T.lists3[n].ones.len = (uint16_t)(n3 - T.lists3[n].ones.start);
    }
    return T;
}

// Whether the lists of n colours hold every split exactly once, in key order.
constexpr bool lists_cover(const CandTables& T, int n)
{
    bool seen[16][17][17] = {};
    int count = 0;
    bool ok = true;
    uint32_t last = 0;
    auto see = [&](uint32_t key, int di, int dk) {
        bool& s = seen[key_i(key) + di][key_j(key)][key_k(key) + dk];
        ok = ok && !s && key_i(key) + di <= key_j(key) && key_j(key) <= key_k(key) && key_k(key) + dk <= n;
        s = true;
        ++count;
    };
    for (int e = 0; e < T.lists4[n].tiles.len; ++e) {
        const uint32_t key = T.tile[T.lists4[n].tiles.start + e].key;
        for (int p = 0; p < 4; ++p) see(key, p / 2, p % 2);
        ok = ok && key >= last;
        last = key;
    }
    last = 0;
    for (int e = 0; e < T.lists4[n].ones.len; ++e) {
        const uint32_t key = T.one4[T.lists4[n].ones.start + e].key;
        see(key, 0, 0);
        ok = ok && key > last;
        last = key;
    }
    return ok && count == splits4_for(n);
}
constexpr bool all_lists_cover()
{
    const CandTables T = make_cand_tables();
    bool ok = true;
    for (int n = 0; n <= 16; ++n) ok = ok && lists_cover(T, n);
    return ok;
}
static_assert(all_lists_cover(), "each list holds its splits once, in key order");

// 3. Unit-weight split constants.  When a block has 16 distinct colours and
//    every point weight is exactly 1 (no duplicates, no alpha weighting),
//    the weight components of the split sums are exact integers fixed by
//    the split alone: part0.w = i, part1.w = j - i, part2.w = k - j,
//    xsum.w = 16.  alpha2_sum, beta2_sum, alphabeta_sum and the factor of
//    cluster.rs:193-202 / 325-335 are then the same numbers for every such
//    block.  They are evaluated here with the kernel's own expressions
//    (constant evaluation is IEEE binary32 with round-to-nearest-even and no
//    contraction, like the device code), one entry per split of the
//    16-colour lists of CandTables in their order (tiles: one array per
//    split of the tile, row (i, k), (i, k+1), (i+1, k), (i+1, k+1)), so the
//    device reads bit-identical values instead of recomputing them.
struct UnitSplit {
    float a2, b2, ab, factor;
};

struct UnitTables {
    UnitSplit tile[4][kTiles16];
    UnitSplit one4[kOnes16];
    UnitSplit one3[kCand3];
};

constexpr UnitSplit unit_split4(int i, int j, int k)
{
    const float p0w = (float)i, p1w = (float)(j - i), p2w = (float)(k - j), xsw = 16.0f;
    const float p3w = ((xsw - p2w) - p1w) - p0w;
    const float n19 = 1.0f / 9.0f, n49 = 4.0f / 9.0f;
    const float a2 = p2w * n19 + (p1w * n49 + p0w);
    const float b2 = p1w * n19 + (p2w * n49 + p3w);
    const float ab = (2.0f / 9.0f) * (p1w + p2w);
    return UnitSplit{a2, b2, ab, 1.0f / ((a2 * b2) - ab * ab)};
}

constexpr UnitSplit unit_split3(int i, int j)
{
    const float p0w = (float)i, p1w = (float)(j - i), xsw = 16.0f;
    const float p2w = (xsw - p1w) - p0w;
    const float hw = p1w * 0.25f;
    const float a2 = hw + p0w, b2 = hw + p2w, ab = hw;
    return UnitSplit{a2, b2, ab, 1.0f / ((a2 * b2) - ab * ab)};
}

constexpr UnitTables make_unit_tables()
{
    const CandTables C = make_cand_tables();
    UnitTables U{};
    for (int e = 0; e < kTiles16; ++e) {
        const uint32_t key = C.tile[C.lists4[16].tiles.start + e].key;
        for (int p = 0; p < 4; ++p) U.tile[p][e] = unit_split4(key_i(key) + p / 2, key_j(key), key_k(key) + p % 2);
    }
    for (int e = 0; e < kOnes16; ++e) {
        const uint32_t key = C.one4[C.lists4[16].ones.start + e].key;
        U.one4[e] = unit_split4(key_i(key), key_j(key), key_k(key));
    }
    for (int e = 0; e < kCand3; ++e) {
        const uint32_t key = C.one3[C.lists3[16].ones.start + e].key;
        U.one3[e] = unit_split3(key_i(key), key_j(key));
    }
    return U;
}

static_assert(splits4_for(16) == kCand4 && splits3_for(16) == kCand3 && kTiles16 == 192 && kOnes16 == 199,
              "split counts of 16 colours");
static_assert(soff(0, 16) == 16 && soff(1, 2) == 17 && soff(15, 16) == kSEntries - 1, "compact prefix table");

}  // namespace txt
