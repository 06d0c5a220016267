"""The grouping of bricks into MP tiles (group_run of lbx_mp.h), compiled for the
host with an address checker: runs of bricks after a lattice's last tile read no
entry of the tiles' cuts, which has one per tile, and the tiles are those of a
plain restatement."""
import os
import random
import re
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "laboetie_amd", "csrc")

MAIN = r"""
int main() {
    uint32_t n, run, cases;
    if (scanf("%u", &cases) != 1) return 2;
    for (; cases > 0; --cases) {
        if (scanf("%u %u", &n, &run) != 2) return 2;
        uint32_t* count = (uint32_t*)malloc(n * sizeof(uint32_t));
        for (uint32_t o = 0; o < n; ++o)
            if (scanf("%u", count + o) != 1) return 2;
        const auto none = [](uint32_t, uint32_t, uint32_t, uint32_t) {};
        uint32_t tiles = 0, old = 0, at = 0;
        for (uint32_t o = 0; o < n; o += run)
            tiles += group_run(count, o, o + run < n ? o + run : n, nullptr, 0, none).tiles;
        uint8_t* split = (uint8_t*)malloc(tiles ? tiles : 1);  // one entry per tile
        for (uint32_t t = 0; t < tiles; ++t) split[t] = (uint8_t)((t * 2654435761u >> 16) % 9);
        printf("%u", tiles);
        for (uint32_t o = 0; o < n; o += run) {
            const RunTiles k = group_run(count, o, o + run < n ? o + run : n, split, old,
                                         [&](uint32_t b, uint32_t, uint32_t tile, uint32_t acc) {
                                             printf(" %u:%u:%u", b, at + tile, acc);
                                         });
            at += k.tiles;
            old += k.unsplit;
        }
        printf(" %u %u\n", at, old);
        free(split);
        free(count);
    }
}
"""


def restated(count, run):
    """(unsplit tiles, [(brick, tile, place)], tiles)"""
    unsplit, rows, tiles = 0, [], 0
    for o0 in range(0, len(count), run):
        groups = []
        for o in range(o0, min(len(count), o0 + run)):
            if count[o]:
                if not groups or sum(count[b] for b in groups[-1]) + count[o] > 256:
                    groups.append([])
                groups[-1].append(o)
        for g in groups:
            exponent = ((unsplit * 2654435761 & 0xFFFFFFFF) >> 16) % 9
            unsplit += 1
            part, pos, at = None, 0, 0
            for b in g:
                p = (pos << exponent) >> 8
                if p != part:
                    tiles, at, part = tiles + 1, 0, p
                rows.append((b, tiles - 1, at))
                at += count[b]
                pos += count[b]
    return unsplit, rows, tiles


def test_grouping_on_the_host(tmp_path):
    text = open(os.path.join(CSRC, "lbx_mp.h")).read()
    body = re.search(r"struct RunTiles \{.*?\n\};\n.*?\n\}\n", text, re.S).group(0)
    src = tmp_path / "group.cpp"
    src.write_text("#include <cstdint>\n#include <cstdio>\n#include <cstdlib>\n#define __device__\n"
                   "#define __forceinline__ inline\n#define __restrict__\n"
                   "static constexpr uint32_t kMpTile = 256;\n" + body + MAIN)
    exe = tmp_path / "group"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wno-unknown-pragmas", "-fsanitize=address", "-o", str(exe),
                    str(src)], check=True)
    rng = random.Random(7)
    cases = [([0] * 40, 8), ([256, 0, 0], 1), ([], 4), ([0, 5] + [0] * 300, 128)]
    for _ in range(200):
        run = rng.choice([1, 5, 8, 128, 256])
        fill, top = rng.random(), rng.choice([3, 40, 154, 256])
        count = [rng.randint(1, top) if rng.random() < fill else 0 for _ in range(rng.randint(0, 700))]
        cases.append((count + [0] * (run * rng.randint(0, 3)), run))  # runs after the last tile
    cases = [(c, r) for c, r in cases if c]
    feed = "\n".join([str(len(cases))] + [f"{len(c)} {r} " + " ".join(map(str, c)) for c, r in cases])
    out = subprocess.run([str(exe)], input=feed, capture_output=True, text=True)
    assert out.returncode == 0, out.stderr[-2000:]
    for (c, r), line in zip(cases, out.stdout.splitlines()):
        unsplit, rows, tiles = restated(c, r)
        f = line.split()
        assert int(f[0]) == unsplit and int(f[-1]) == unsplit and int(f[-2]) == tiles
        assert [tuple(map(int, x.split(":"))) for x in f[1:-2]] == rows
