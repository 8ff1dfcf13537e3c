"""The split of a wave's candidate cells into slices, host and device share it:
the slices of every accepted number of candidates follow each other from 0 to
the total, and no step of a slice's loop passes 2^32 (it would never end)."""
import os
import subprocess

from conftest import ROOT

SOURCE = r"""
#include <cstdio>
#include <vector>
#include "hr_slices.h"
using namespace hr;
static int bad(const char* what, uint64_t total, uint64_t s)
{
    std::printf("%s: total %llu slice %llu\n", what, (unsigned long long)total, (unsigned long long)s);
    return 1;
}
int main()
{
    std::vector<uint64_t> totals;
    for (uint64_t t = kPairsHeavy; t < kPairsHeavy + 20000; ++t) totals.push_back(t);
    for (int b = 14; b <= 32; ++b)
        for (int64_t d = -2100; d <= 2100; ++d) {
            const uint64_t t = (1ull << b) + d;
            if (t <= kPairsWaveMax) totals.push_back(t);
        }
    for (uint64_t d = 0; d < 5000; ++d) totals.push_back((uint64_t)kPairsWaveMax - d);
    uint64_t x = 88172645463325252ull;
    for (int i = 0; i < 200000; ++i) {
        x ^= x << 13; x ^= x >> 7; x ^= x << 17;
        const uint64_t t = x % kPairsWaveMax;
        if (t >= kPairsHeavy) totals.push_back(t);
    }
    for (uint64_t total : totals) {
        const uint32_t n = slice_len((uint32_t)total);
        if (n % kSliceStep || n < kSliceMin) return bad("length", total, 0);
        uint64_t at = 0;
        for (uint32_t s = 0; s < kPairSlices; ++s) {
            if ((uint64_t)s * n > 0xFFFFFFFFull) return bad("begin past 2^32", total, s);
            const uint32_t b = slice_begin((uint32_t)total, s);
            if (b >= total) continue;
            const uint32_t e = slice_end((uint32_t)total, s);
            if (b != at || e <= b || e > total) return bad("gap", total, s);
            at = e;
            // the loop's last step, and the first one that is not taken
            const uint64_t last = b + ((uint64_t)(e - b) - 1) / kSliceStep * kSliceStep;
            if (last + kSliceStep > 0xFFFFFFFFull) return bad("step past 2^32", total, s);
            // an owner of the last candidates is found in that step, one of those before is not
            if (!owns_in_step((uint32_t)last, (uint32_t)(total - last), (uint32_t)last)) return bad("owner", total, s);
            if (last && owns_in_step(0u, (uint32_t)last, (uint32_t)last)) return bad("owner before", total, s);
            if (owns_in_step((uint32_t)last, 0u, (uint32_t)last)) return bad("owner of none", total, s);
        }
        if (at != total) return bad("end", total, kPairSlices);
    }
    if (pairs_count_or_refuse(kPairsWaveMax, 7u) != 7u || pairs_count_or_refuse(kPairsWaveMax + 1u, 7u) != ~0u) return 1;
    std::printf("%zu totals\n", totals.size());
    return 0;
}
"""


def test_slices_tile_every_accepted_total(tmp_path):
    src, exe = tmp_path / "slices.cpp", tmp_path / "slices"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "happyray_amd", "csrc"), str(src), "-o",
                           str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
