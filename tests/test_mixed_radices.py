"""The host-side planning of the mixed-radix kernel (afft_mixed_plan.cpp), compiled into a small program with
its table of butterfly costs made writable: for every length, the radices it chooses multiply to the
length and fit the threads, with the costs as they are and with others."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "accelerate-fft_amd"))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "plan_under_test.cpp"
using namespace afft;

int main()
{
    long bad = 0, found = 0;
    for (int dtype = 0; dtype < 2; ++dtype)
        for (int E : {16, 32, kMixWide})
            for (int symmetric = 0; symmetric < (E == kMixWide ? 1 : 2); ++symmetric)
                for (int threads : {256, 512, 1024})
                    for (int64_t n = 2; n <= 16384; ++n) {
                        MixShape s;
                        const int most = E == kMixWide ? mixed_wide_radix(dtype) : kMixMaxRadix;
                        if (!mixed_radices(n, symmetric, E, threads, s, most)) continue;
                        ++found;
                        int64_t product = 1;
                        bool ok = s.npass >= 1 && s.npass <= kMixMaxPasses;
                        for (int i = 0; ok && i < s.npass; ++i) {
                            const int r = s.radix[i];
                            product *= r;
                            ok = r >= 2 && r <= most && n / r <= (int64_t)mixed_butterflies(E, r) * threads &&
                                 (r <= 16 || r == 17 || r == 19 || r == 23 || r == 29 || r == 31);
                        }
                        if (symmetric) ok = ok && s.npass >= 2 && s.radix[0] == s.radix[s.npass - 1];
                        if (!ok || product != n) {
                            if (bad++ < 5) std::printf("type %d E %d symmetric %d threads %d n %ld\n", dtype, E, symmetric, threads, (long)n);
                        }
                    }
    // padded lengths: long enough, products of 2, 3 and 5, with equal ends
    for (int dtype = 0; dtype < 2; ++dtype)
        for (int64_t n = 2; n <= (dtype ? 4096 : 8192); ++n) {
            const int64_t m = mixed_chirpz_length(dtype, n, dtype ? 8192 : 16384, 160 * 1024);
            MixShape s;
            int64_t q = m;
            for (int p : {2, 3, 5})
                while (q && q % p == 0) q /= p;
            if (m < 2 * n - 1 || q != 1 || !mixed_radices(m, true, 16, dtype ? 512 : 1024, s))
                if (bad++ < 10) std::printf("type %d padded length of %ld: %ld\n", dtype, (long)n, (long)m);
        }
    // a search that finds nothing within the best cost so far ends without radices, whatever the costs
    std::srand(7);
    for (int t = 0; t < 50; ++t) {
        for (int r = 2; r <= kMixMaxRadix; ++r) kButterflyCost[r] = 7 + 10.0 * std::rand() / RAND_MAX;
        for (int64_t n = 4; n <= 4096; ++n) {
            int64_t q = n, product = 1;
            for (int p : {2, 3, 5})
                while (q % p == 0) q /= p;
            MixShape s;
            if (q != 1 || !mixed_radices(n, true, 16, 512, s)) continue;
            for (int i = 0; i < s.npass; ++i) product *= s.radix[i];
            if (product != n && bad++ < 10) std::printf("costs %d: n %ld, product %ld\n", t, (long)n, (long)product);
        }
    }
    std::printf("%ld found, %ld bad\n", found, bad);
    return bad || found < 10000;
}
"""


def test_radices_of_every_length(tmp_path):
    import build
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    src, exe = str(tmp_path / "radices.hip"), str(tmp_path / "radices")
    with open(os.path.join(build.CSRC, "afft_mixed_plan.cpp")) as f:
        plan = f.read()
    assert "const double kButterflyCost[" in plan
    with open(tmp_path / "plan_under_test.cpp", "w") as f:
        f.write(plan.replace("const double kButterflyCost[", "double kButterflyCost[").replace("../../include/", ""))
    with open(src, "w") as f:
        f.write(PROGRAM)
    r = subprocess.run([build.HIPCC] + build.COMMON + ["-I" + build.CSRC, src, "-o", exe], capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:]
