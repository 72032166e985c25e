"""Which reconstructions take their table into LDS (vq_amd/csrc/resident_rules.hpp): the rules are compiled by g++ and
asked for sizes up to the limits of the entry points.  What they admit has its places within a run in 32 bits and its
groups within a grid's second dimension; what they refuse goes to the gather kernels, which take any size."""
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAIN = """
#include <cstdio>
#include "resident_rules.hpp"
int main() {
    long long n; int what, a, b, c;  // what: 0 decode to f32, 1 to binary16, 2 residual sums
    while (scanf("%d %lld %d %d %d", &what, &n, &a, &b, &c) == 5)
        printf("%d\\n", what == 2 ? vq::rvq_recon_columns(n, a, b, c) : vq::decode_resident_blocks(what, n, a, b, c));
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rules") / "rules")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-x", "c++", "-", "-I", os.path.join(ROOT, "vq_amd", "csrc"),
                    "-o", exe], input=MAIN, text=True, check=True)

    def ask(cases):
        text = "\n".join(" ".join(str(int(v)) for v in c) for c in cases)
        return [int(v) for v in subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split()]
    return ask


def _decode_ok(f16, n, m, sd, k, G):
    pieces, block = sd // (8 if f16 else 4), k * sd * (2 if f16 else 4)
    groups = -(-m // G)
    for mg in {min(G, m), m - (groups - 1) * G}:  # a whole group, the last one
        rows = min(n, max(1, 1024 * (4 if f16 else 8) // (mg * pieces)))  # of a run, as k_decode_resident takes them
        if (rows - 1) * m * pieces + mg * pieces > 2 ** 32 or (groups > 1 and mg * pieces % 4):  # (64-byte shares)
            return False
    return sd % (8 if f16 else 4) == 0 and block * G <= 128 * 1024 and groups <= 65535


def test_decode_at_the_limits(rules):
    rng = random.Random(1)
    edges = [(1 << e) + d for e in range(8, 24) for d in (-1, 0, 1, 5)] + [1064961, 532481, 8_388_612]
    cases = [(f16, n, m, sd, k) for f16 in (0, 1) for m in edges for sd in (4, 8, 16, 24) for k in (1, 5, 256, 2048)
             for n in (1, 2, 5, 100, 4096, 8192, 1 << 20, 1 << 31)]
    cases += [(rng.random() < 0.5, int(2 ** rng.uniform(0, 32)), int(2 ** rng.uniform(0, 24)), rng.choice([4, 8, 8, 16, 32, 100, 512]),
               int(2 ** rng.uniform(0, 16))) for _ in range(20_000)]
    got = rules(cases)
    assert sum(G > 0 for G in got) > 1000
    assert [c for c, G in zip(cases, got) if G and not _decode_ok(*c, G)] == []


def test_decode_of_ordinary_sizes(rules):
    """(binary16, n, m, sub_dim, k): column blocks per group."""
    want = {(1, 1_000_000, 16, 8, 256): 16, (1, 300_000, 16, 8, 1024): 8, (0, 300_000, 16, 4, 1024): 8, (1, 200_000, 12, 8, 256): 12,
            (1, 66_000, 20, 8, 2048): 4, (1, 262_144, 10, 8, 100): 10, (1, 6, 500_000, 8, 2048): 0, (0, 4096, 8_388_612, 4, 1): 0,
            # shares of a row that end inside a half line, few pieces, no room in LDS
            (1, 1_000_000, 10, 8, 1024): 0, (1, 1_000_000, 17, 8, 2048): 0, (1, 32_000, 16, 8, 256): 0, (1, 1_000_000, 16, 8, 2049): 0,
            # a table that the vector cache holds, also with rows beyond the memory-side cache
            (1, 400_000, 16, 8, 16): 0, (0, 800_000, 16, 4, 200): 0, (0, 800_000, 16, 4, 256): 16, (1, 1_000_000, 16, 8, 16): 16,
            # more than one piece to a centroid
            (1, 130_000, 8, 16, 256): 0, (1, 1_000_000, 8, 16, 256): 8, (0, 400_000, 16, 8, 256): 0, (0, 1_000_000, 16, 8, 256): 16,
            (0, 300_000, 16, 8, 512): 0, (0, 1_000_000, 16, 8, 512): 8, (1, 1_000_000, 10, 12, 256): 0}
    assert rules(list(want)) == list(want.values())


def _recon_ok(n, stages, k, dim, G):
    groups = -(-dim // G)
    for cols in {G, dim - (groups - 1) * G}:
        rows = min(n, max(1, 2048 // (cols // 8)))  # of a run, as k_rvq_recon_resident takes them
        if cols % 8 or (rows - 1) * (dim // 8) + cols // 8 > 2 ** 32:
            return False
    return 4 * stages * k * G <= 128 * 1024 and groups <= 65535


def test_residual_sums(rules):
    rng = random.Random(2)
    dims = [(1 << e) + d for e in range(3, 31) for d in (-8, 0, 8, 24)] + [32 * 65535, 32 * 65535 + 8, 16 * 65535 + 16]
    cases = [(2, n, stages, k, dim) for dim in dims if dim > 0 for stages in (1, 2, 4, 8, 255) for k in (1, 8, 100, 256, 300)
             for n in (1, 3, 2048, 1 << 20)]
    cases += [(2, int(2 ** rng.uniform(0, 32)), rng.randint(1, 40), int(2 ** rng.uniform(0, 10)), rng.randint(1, 500)) for _ in range(5000)]
    got = rules(cases)
    assert sum(G > 0 for G in got) > 1000
    assert [c for c, G in zip(cases, got) if G and not _recon_ok(*c[1:], G)] == []
    want = {(200_000, 4, 256, 128): 32, (1_000_000, 8, 256, 256): 16, (200_000, 6, 256, 200): 16, (100_000, 2, 256, 256): 64,
            (400_000, 2, 256, 72): 0, (100_000, 2, 16, 136): 136, (100_000, 9, 256, 64): 0, (100_000, 4, 256, 100): 0,
            (1, 4, 256, 32 * 65535 + 32): 0}
    assert rules([(2, *c) for c in want]) == list(want.values())
