"""The engine's threaded host copies (host/copy_pool.h) on the CPU, under AddressSanitizer: copies at the sizes
where the plan changes, and a transfer that fails with copies posted. Once the failing block is
left, its destination and source may be freed or used for something else, so no helper may touch them."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <cstdio>
#include <memory>
#include <stdexcept>
#include "copy_pool.h"
using gyro::CopyPool;

static int fail(const char *what, long a) { return std::printf("%s %ld\n", what, a), 1; }

int main() {
    CopyPool pool;
    for (long n : {0L, 1L, 131071L, 131072L, 1048575L, 1048576L, 1048577L, 2097152L, 5000001L}) {
        std::vector<unsigned char> a(n), b(n);
        for (long i = 0; i < n; ++i) a[i] = (unsigned char)(i * 7 + n);
        pool.copy(b.data(), a.data(), n);
        if (a != b) return fail("copy of", n);
    }
    constexpr long kPart = 2 << 20, kParts = 8, kBytes = kPart * kParts;
    for (int round = 0; round < 60; ++round) {
        std::unique_ptr<unsigned char[]> src(new unsigned char[kBytes]), dst(new unsigned char[kBytes]);
        std::memset(src.get(), 1, kBytes);
        const long posted = 1 + round % (kParts - 1);
        try {  // a download whose wait for a later part fails
            CopyPool::Scope scope(pool);
            for (long i = 0; i < kParts; ++i) {
                if (i == posted) throw std::runtime_error("wait");
                pool.post(dst.get() + i * kPart, src.get() + i * kPart, round & 1 ? kPart : CopyPool::kPiece);
            }
            pool.finish();
        } catch (const std::runtime_error &) {
        }
        std::memset(dst.get(), 2, kBytes);
        src.reset();
        std::vector<unsigned char> a(1 << 20, 3), b(1 << 20);
        pool.copy(b.data(), a.data(), a.size());  // must not resume what the failed block had queued
        if (a != b) return fail("copy after a failure, round", round);
        for (long i = 0; i < kBytes; ++i)
            if (dst[i] != 2) return fail("written after the failure, byte", i);
    }
    std::puts("ok");
}
"""


def test_copies_and_failed_transfers(tmp_path):
    src, exe = tmp_path / "pool.cpp", tmp_path / "pool"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-fsanitize=address", "-I", str(ROOT / "gyro-dx_amd" / "host"),
                    "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.stdout, r.stderr[-2000:])
