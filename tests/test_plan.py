"""The rules that cut the passes into blocks (csrc/bl_plan.hpp), compiled on
their own with the host compiler and compared with a search over the choices
that a rule has, over the sizes that the solver takes."""
import os
import subprocess

import pytest

from .blgpu_import import PKG

MAIN = r"""
#include <cstdio>
#include <cstring>
#include "bl_plan.hpp"
using namespace blgpu;
int main() {
    char k[16];
    int a, b, c, d, e;
    while (std::scanf("%15s %d %d %d %d %d", k, &a, &b, &c, &d, &e) == 6) {
        if (!std::strcmp(k, "dct")) {
            const DctPlan p = dct_plan(a, b, (size_t)c, d, e);
            std::printf("%d %d\n", p.lines, p.waves);
        }
        if (!std::strcmp(k, "march")) {  // element size, eddy viscosity, nx, ny, nz; 256 compute units
            const int res = a == 4 ? march_resident<float>(b) : march_resident<double>(b);
            const int tiles = a == 4 ? march_tiles<float>(c + 1, d + 1) : march_tiles<double>(c + 1, d + 1);
            std::printf("%d %d %d\n", march_chunk(e - 1, tiles, 256, res), tiles, res);
        }
        if (!std::strcmp(k, "takes"))
            std::printf("%d %d %d %d\n", dct_takes_fp64(a, b), dct_takes_mixed(a, b), dct_holds(a, b, 8), dct_holds(a, b, 4));
        if (!std::strcmp(k, "thomas")) std::printf("%d\n", thomas_resident(a));
        if (!std::strcmp(k, "steps")) std::printf("%d\n", fewest_plane_steps(a, b, c, d).planes);
        if (!std::strcmp(k, "vfilter")) std::printf("%d\n", a == 4 ? vfilter_resident<float>() : vfilter_resident<double>());
    }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN)
    exe = str(d / "plan")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(PKG, "csrc"), str(d / "main.cpp"), "-o", exe],
                   check=True)

    def ask(rows):
        text = "".join(" ".join(str(v) for v in r) + "\n" for r in rows)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(int(v) for v in line.split()) for line in out.splitlines()]

    return ask


def factor(n):
    n1 = max(a for a in range(1, int(n ** 0.5) + 1) if n % a == 0)
    return n1, n // n1


@pytest.mark.parametrize("es", [4, 8])
def test_x_transform_plan(plan, es):
    """Lengths with a factor past 31: where the blocks fill the chip, more than
    four products of step C go to eight waves, and no number of lines up to a
    full column tile (and that fits 80 KB) takes fewer wave slots per line."""
    lengths = [n for n in range(32, 1300) if factor(n)[1] > 31 and factor(n)[1] <= 256]
    for n, (lines, waves) in zip(lengths, plan([("dct", n, factor(n)[0], es, 40000, 256) for n in lengths])):
        n1, n2 = factor(n)
        k1 = n1 // 2 + 1
        line = es * (n + 1 + 2 * k1 * (n2 | 1))

        def products(lb):
            return (lb * k1 + 15) // 16 * ((n2 // 2 + 16) // 16)

        def slots(lb):
            p = products(lb)
            w = 8 if p > 4 else 4
            return (p + w - 1) // w * w

        assert lines == 1 or lines * line <= 81920
        assert waves == (8 if products(lines) > 4 else 4), n
        most = max(2, (15 + k1) // k1)
        best = min(slots(lb) / lb for lb in range(1, most + 1) if lb == 1 or lb * line <= 81920)
        assert slots(lines) / lines <= best * 1.0001, (n, lines)


def test_x_transform_plan_small(plan):
    """Two lines in two waves for two factors of up to 31; blocks of eight waves,
    and of fewer lines, where a grid has too few lines for the chip."""
    assert plan([("dct", 812, 28, 8, 49000, 256)]) == [(2, 2)]
    assert plan([("dct", 961, 31, 4, 10, 256)]) == [(2, 2)]
    full, = plan([("dct", 127, 1, 8, 40000, 256)])
    few, = plan([("dct", 127, 1, 8, 1536, 256)])
    assert few[0] == (full[0] + 1) // 2 and few[1] == 8 and full[1] == 4


@pytest.mark.parametrize("es", [4, 8])
def test_x_transform_plan_waves(plan, es):
    """Eight waves for four products or fewer only while all blocks reside at once
    (16 waves per compute unit in FP64, 24 in FP32); with many lines and a first
    factor past 7, no more lines that fit a quarter of the LDS fill the four waves'
    products better (16 x 32 points: three lines in four products, not two)."""
    lengths = [n for n in range(32, 1100) if factor(n)[1] > 31 and factor(n)[1] <= 256]
    counts = [256, 432, 1170, 1536, 2360, 3774, 5568, 12288, 25542]
    rows = [("dct", n, factor(n)[0], es, c, 256) for n in lengths for c in counts]
    for (_, n, n1, _, c, _), (lines, waves) in zip(rows, plan(rows)):
        n2, k1 = n // n1, n1 // 2 + 1
        line = es * (n + 1 + 2 * k1 * (n2 | 1))

        def products(lb):
            return (lb * k1 + 15) // 16 * ((n2 // 2 + 16) // 16)

        blocks = (c + lines - 1) // lines
        if waves == 8 and products(lines) <= 4:
            assert blocks * 8 <= 256 * (24 if es == 4 else 16), (n, c)
        if c == 25542 and k1 > 4 and products(lines) <= 4:
            assert products(lines + 1) > 4 or (lines + 1) * line > 40960 or c // (lines + 1) < 2048, (n, lines)


def test_march_plan(plan):
    """The z chunk of the RK march: no other chunk takes fewer plane steps in
    sequence (rounds of the blocks that reside by their LDS, at most three, times
    chunk + 2) while the launch is of up to six blocks per compute unit.  An FP64
    block with an eddy viscosity holds ten planes of 66 x 10, so two reside, and
    278x266x34 goes in one round."""
    shapes = [(278, 266, 34), (161, 57, 42), (390, 244, 57), (292, 206, 196), (716, 261, 63), (24, 16, 8), (5, 4, 5)]
    shapes += [(60 + 37 * i, 20 + 23 * i % 270, 8 + 41 * i % 230) for i in range(20)]
    rows = [("march", es, les, *s) for s in shapes for es in (4, 8) for les in (0, 1)]
    for (_, es, les, nx, ny, nz), (chunk, tiles, res) in zip(rows, plan(rows)):
        plane = 66 * (4 * (3 if es == 4 else 2) + 2)
        assert res == min(3, 163840 // (es * (plane * (10 if les else 7) + 4 * 64 + 8 * (plane // 66 - 2))))
        assert res == (2 if es == 8 and les else 3)
        nk = nz - 1
        steps = {c: -(-tiles * -(-nk // c) // (256 * res)) * (c + 2) for c in range(1, nk + 1)}
        blocks = tiles * -(-nk // chunk)
        if blocks <= 6 * 256:
            least = min(steps.values())
            few = [c for c in steps if steps[c] == least and tiles * -(-nk // c) <= 6 * 256]
            assert not few or chunk == min(few), (es, les, nx, ny, nz)
        if (es, les, nx) == (8, 1, 278):
            assert blocks <= 256 * res


def test_filter_plan(plan):
    """The velocity filter of the dynamic model: blocks of four waves, of which a
    compute unit holds four with up to 128 registers (FP32 fields) and two with up to
    256 (FP64; the kernel's launch bounds are these figures), and the chunk of the
    fewest plane steps among them, the shortest of equal ones up to a block count."""
    assert plan([("vfilter", 4, 0, 0, 0, 0), ("vfilter", 8, 0, 0, 0, 0)]) == [(4,), (2,)]
    rows = [("steps", nk, tiles, slots, most, 0) for nk in (3, 24, 62, 97) for tiles in (1, 18, 130, 192, 700)
            for slots in (512, 1024) for most in (0, 1536)]
    for (_, nk, tiles, slots, most, _), (chunk,) in zip(rows, plan(rows)):
        steps = {c: -(-tiles * -(-nk // c) // slots) * (c + 2) for c in range(1, nk + 1)}
        equal = [c for c in steps if steps[c] == min(steps.values())]
        few = [c for c in equal if tiles * -(-nk // c) <= most]
        assert chunk == (min(few) if few else max(equal))


def test_y_solve_plan(plan):
    """Blocks of the y solve per compute unit: eight waves by their registers, and
    each block, whatever its waves, has 40 KB of LDS, so four blocks at most."""
    for p, (n,) in zip(range(1, 9), plan([("thomas", p, 0, 0, 0, 0) for p in range(1, 9)])):
        assert n == min(8 // p, 163840 // 40960)


def test_x_transform_lengths_taken(plan):
    """FP64 takes the lengths that it always took (two 16-byte lines, their spectra and
    the roots of both factors in 64 KB, or factors of up to 32), mixed precision factors
    of up to 256 on the same kernels; and every length taken is one that the kernels
    hold: the small division's range and one line of either direction in 160 KB."""
    lengths = list(range(3, 5000))
    for n, (fp64, mixed, holds64, holds32) in zip(lengths, plan([("takes", n, factor(n)[0], 0, 0, 0) for n in lengths])):
        n1, n2 = factor(n)
        k1 = n1 // 2 + 1
        assert fp64 == ((n1 <= 32 and k1 <= 16 and n2 <= 32) or 16 * (2 * n + 2 * k1 * n2 + n1 + n2) <= 65536)
        spec = 2 * k1 * (n2 | 1)
        for es, holds in ((8, holds64), (4, holds32)):
            if holds:
                assert k1 <= 128 and k1 * n2 < 16384 and es * (max(n + 1, spec) + spec) <= 163840, n
        assert not fp64 or holds64
        assert not mixed or holds32
        assert mixed == (n2 <= 256 and holds32)
