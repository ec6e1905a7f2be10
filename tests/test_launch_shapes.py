"""Launch shapes computed on the host, without a GPU: for every chunk size and
number of chunks a batch may have, the pieces of the lockstep encoder's launch
cover each chunk, and the piece count fits the kernel's 32 bits; alpha-only chunks are cut
only as far as each wave gets at most one piece; the grid of
the mip levels stays within a launch's limits for every image size; and the
lines of the direct kernels' teams and of RangeFit's groups."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <stdio.h>
#include "bcn_kernels.hpp"
int main()
{
    unsigned long long groups; unsigned n, wpg, largest;
    while (scanf("%llu %u %u %u", &groups, &n, &wpg, &largest) == 4) {
        if (groups == 0) {  // the mip levels of an n x wpg image: launches, widest grid, its rows
            unsigned launches = 0, x = 0, y = 0;
            unsigned long long covered = 0;
            while (covered * txk::kMipTile < n) {
                const dim3 g = txk::mip_grid(n, wpg, covered);
                x = g.x > x ? g.x : x;
                y = g.y;
                covered += g.x;
                ++launches;
            }
            if (covered != (n + 63ull) / 64) launches = 0;
            printf("%u %u %u\n", launches, x, y);
            continue;
        }
        if (groups == 3) {  // the alpha-only launch of n chunks on wpg CUs: grid, steps, whether it draws work
            const txk::AlphaShape s = txk::alpha_shape(wpg, n, 1, 12, 1);
            printf("%u %u %u\n", s.grid, s.steps, (unsigned)txk::alpha_needs_counter(s, n, 1));
            continue;
        }
        if (groups == 4) {  // the same beside the lockstep encoder
            const txk::AlphaShape s = txk::alpha_shape(wpg, n, 1, 12, 1, true);
            printf("%u %u %u\n", s.grid, s.steps, (unsigned)txk::alpha_needs_counter(s, n, 1));
            continue;
        }
        if (groups == 2) {  // blocks up to which RangeFit takes groups: format, width, height + 2^31 if weighed
            txk::EncodeArgs a{};
            a.format = n;
            a.width = wpg;
            a.height = largest & 0x7FFFFFFFu;
            a.weigh_alpha = largest >> 31;
            printf("%u 0 0\n", (unsigned)txk::range_group_blocks(a));
            continue;
        }
        if (groups == 5) {  // the same for input read over the bus
            txk::EncodeArgs a{};
            a.format = n;
            a.width = wpg;
            a.height = largest & 0x7FFFFFFFu;
            a.weigh_alpha = largest >> 31;
            a.over_bus = true;
            printf("%u 0 0\n", (unsigned)txk::range_group_blocks(a));
            continue;
        }
        if (groups == 1) {  // the team of algorithm n for wpg blocks, on the library's and on a caller's stream
            printf("%d %d 0\n", txk::team_groups(n, wpg, false), txk::team_groups(n, wpg, true));
            continue;
        }
        const txk::HeavyShape h = txk::heavy_shape(groups, n, wpg, largest);
        printf("%u %u %u\n", h.grid, h.per_chunk, h.span);
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    d = tmp_path_factory.mktemp("shapes")
    src, exe = d / "shapes.cpp", d / "shapes"
    src.write_text(SOURCE)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "texpresso_amd", "csrc"), str(src), "-o", str(exe)], check=True)

    def run(rows):
        out = subprocess.run([str(exe)], input="".join("%d %d %d %d\n" % r for r in rows), text=True, check=True,
                             stdout=subprocess.PIPE).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


def test_heavy_pieces_cover_every_chunk(shapes):
    sizes = [4, 8, 60, 64, 68, 128, 4096, 1 << 20, 1 << 30, (1 << 31) - 4, 1 << 31, (1 << 31) + 4, 0xFFFFFFC0,
             0xFFFFFFC4, 0xFFFFFFF8, 0xFFFFFFFC]
    rows = [(256 * g, n, w, c) for g in (1, 12, 64) for w in (1, 2, 4) for c in sizes
            for n in (1, 2, 3, 7, 100, 2000, 3071, 3072, 3073, 100000)]
    for (groups, n, wpg, chunk), (grid, per_chunk, span) in zip(rows, shapes(rows)):
        case = (groups, n, wpg, chunk, grid, per_chunk, span)
        assert per_chunk >= 1 and span >= 4 and span % 4 == 0, case
        assert per_chunk * span >= chunk > (per_chunk - 1) * span, case
        assert n * per_chunk < 1 << 32 and n * per_chunk <= max(n, groups * wpg), case
        assert 1 <= grid <= groups, case


def test_no_chunks_and_single_blocks(shapes):
    # no chunks at all (a batch without colour textures), and chunks below one step
    for grid, per_chunk, span in shapes([(3072, 0, 1, 0), (3072, 0, 4, 0), (3072, 1, 1, 1), (3072, 1, 2, 3)]):
        assert (grid, per_chunk, span) == (1, 1, 4)


def test_mip_grid_within_launch_limits(shapes):
    sides = [1, 63, 64, 65, 4096, (1 << 29) - 1, 1 << 29, (1 << 29) + 1, 1 << 30, (1 << 30) + 1, 0x7FFFFFFF]
    rows = [(0, w, h, 0) for w in sides for h in sides]
    for (_, w, h, _), (launches, widest, y) in zip(rows, shapes(rows)):
        assert widest * 256 < 1 << 32 and 1 <= y < 1 << 16 and y <= (h + 63) // 64, (w, h)
        assert launches == ((w + 63) // 64 + (1 << 23) - 1) >> 23, (w, h)


def test_team_lines(shapes):
    # (algorithm, blocks): team on the library's own stream, team on a caller's
    want = {(1, 1): (4, 4), (1, 2560): (4, 4), (1, 2561): (2, 2), (1, 6144): (2, 2), (1, 6145): (1, 1),
            (2, 1): (4, 4), (2, 7168): (4, 4), (2, 7169): (4, 2), (2, 10240): (4, 2), (2, 10241): (2, 2),
            (2, 32768): (2, 2), (2, 32769): (1, 1)}
    got = shapes([(1, alg, n, 0) for alg, n in want])
    assert {k: v[:2] for k, v in zip(want, got)} == want


def test_range_lines(shapes):
    w = 1 << 31  # weighed by alpha
    want = {(0, 256, 256): 2560, (1, 256, 256): 2560, (2, 256, 256): 5120, (0, 257, 255): 2560, (2, 257, 256): 10240,
            (2, 256, 255): 10240, (0, 3, 8192): 8192, (1, 8192, 1): 8192, (2, 3, 8192): 10240, (0, 256, 256 + w): 12288,
            (1, 1, 64 + w): 12288, (2, 257, 256 + w): 12288}
    got = shapes([(2, fmt, width, height) for fmt, width, height in want])
    assert {k: v[0] for k, v in zip(want, got)} == want


def test_alpha_pieces(shapes):
    rows = [(3, n, cus, 0) for cus in (256, 304) for n in (1, 2, 3, 24, 1023, 1024, 1025, 1500, 2048, 2049, 4096, 4097,
                                                           8192, 8193, 20000, 1 << 23)]
    for (_, n, cus, _), (grid, steps, draws) in zip(rows, shapes(rows)):
        waves, pieces = 32 * cus, n * (8 // steps)
        case = (n, cus, grid, steps, draws)
        assert steps in (1, 2, 4, 8) and grid == min((pieces + 3) // 4, waves // 4), case
        assert bool(draws) == (pieces > 4 * grid) == (n > waves), case
        if steps > 1:  # a finer cut would leave a wave more than one piece
            assert 2 * pieces > waves, case


def test_alpha_chunks_whole_beside_the_lockstep_encoder(shapes):
    rows = [(4, n, cus, 0) for cus in (256, 304) for n in (1, 2, 3, 24, 460, 1024, 8192, 8193, 20000)]
    for (_, n, cus, _), (grid, steps, draws) in zip(rows, shapes(rows)):
        case = (n, cus, grid, steps, draws)
        assert steps == 8 and grid == min((n + 3) // 4, 8 * cus), case
        assert bool(draws) == (n > 32 * cus), case


def test_range_lines_over_the_bus(shapes):
    w = 1 << 31  # weighed by alpha
    want = {(0, 256, 256): 512, (2, 256, 256): 512, (2, 257, 256): 512, (1, 256, 256 + w): 1280, (0, 4, 4): 512,
            (0, 3, 8192): 8192, (1, 8192, 1): 8192, (2, 3, 8192): 10240, (1, 1, 64 + w): 12288}
    got = shapes([(5, fmt, width, height) for fmt, width, height in want])
    assert {k: v[0] for k, v in zip(want, got)} == want
