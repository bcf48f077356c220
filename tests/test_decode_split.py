"""How the decode path splits a call over the compute units (host/decode_split.h), on the CPU over every shape
that the run-wise kernels take and 1 to 8 tokens."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

DOWN = r"""
#include <cstdio>
#include "decode_split.h"
int main() {
    for (unsigned cus : {256u, 304u, 64u})
        for (unsigned max_rows : {32u, 24u})
            for (unsigned E = 256; E <= 4096; E += 256)
                for (unsigned F = 128; F <= 1024; F += 128)
                    for (unsigned U = 1; U <= 16; ++U)
                        for (unsigned n = 1; n <= 8; ++n)
                            std::printf("%u %u %u %u %u %u %u\n", cus, max_rows, E, F, U, n,
                                        gyro::decode_down_rows(E, F, U, n, cus, max_rows));
}
"""

BLOCKS = r"""
#include <cstdio>
#include "decode_split.h"
int main() {
    for (unsigned cus : {256u, 304u, 64u, 32u})
        for (unsigned E : {1024u, 2048u})
            for (unsigned n = 2; n <= 8; ++n)
                std::printf("%u %u %u %u\n", cus, E, n, gyro::decode_blocks_per_lane(E, n, cus));
}
"""


def lines(tmp_path, program):
    src, exe = tmp_path / "split.cpp", tmp_path / "split"
    src.write_text(program)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", str(ROOT / "gyro-dx_amd" / "host"), "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True, timeout=100).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]


def takes(E, F, U, R):
    """What a moe_decode_down_g group of R rows holds: whole groups, its items and its sums."""
    return E % R == 0 and U * (F // 128) * 2 * ((R + 1) // 2) <= 1024 and R * U <= 512


def test_down_rows(tmp_path):
    """Rows are within the kernel's limits, and never make more rounds than the most rows up to E / CUs that the
    kernel takes."""
    for cus, max_rows, E, F, U, n, R in lines(tmp_path, DOWN):
        case = (cus, max_rows, E, F, U, n, R)
        assert 1 <= R <= max_rows and takes(E, F, U, R), case
        plain = min(max_rows, max(1, E // cus))
        while not takes(E, F, U, plain):
            plain -= 1
        assert -(-(E // R) * n // cus) <= -(-(E // plain) * n // cus), (case, plain)


def test_down_rows_examples(tmp_path):
    rows = {k[2:6]: k[6] for k in lines(tmp_path, DOWN) if k[0] == 256 and k[1] == 32}
    assert rows[2560, 640, 10, 1] == 10 and rows[2560, 640, 10, 2] == 20 and rows[2560, 640, 10, 3] == 10
    assert rows[1024, 256, 2, 8] == 32 and rows[3840, 768, 16, 1] == 8 and rows[256, 1024, 16, 1] == 1


def test_blocks_per_lane(tmp_path):
    """Four or two blocks where their groups fill 7/8 of whole rounds of the device's own units."""
    got = {k[:3]: k[3] for k in lines(tmp_path, BLOCKS)}
    for (cus, E, n), r in got.items():
        fills = [b for b in (4, 2) if 8 * (E * n // (8 * b)) >= 7 * cus * -(-E * n // (8 * b) // cus)]
        assert r == (fills[0] if fills else 0), (cus, E, n, r)
    assert [got[256, 2048, n] for n in range(2, 9)] == [2, 0, 4, 0, 2, 4, 4]
    assert [got[256, 1024, n] for n in range(2, 9)] == [0, 0, 2, 0, 0, 4, 4]
