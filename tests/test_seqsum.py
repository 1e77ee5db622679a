"""The parallel form of rmsnorm's in-order double sum (stream-_amd/csrc/es_hip_seqsum.h, src/es_engine.c:189-194): the header
is compiled for the CPU, put together as the kernel does (approximate prefix sums, runs composed by a scan, events added one
by one) and compared bit for bit with adding the squares one after another."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HDR_DIR = os.path.join(ROOT, "stream-_amd", "csrc")

PROG = r"""
#define ESQ_SEQSUM_QUAL static inline
#include "es_hip_seqsum.h"
#include <math.h>
#include <random>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <vector>
constexpr int PER = 8;
// one row as the kernel adds it, threads of 8 terms; runs: terms that were not added one by one
static double parallel(const std::vector<float> &x, bool &ok, long &runs) {
    const int nt = ((int)x.size() + PER - 1) / PER;
    std::vector<double> pre(nt + 1, 0.0);
    std::vector<std::vector<double>> q(nt, std::vector<double>(PER, 0.0));
    for (int t = 0; t < nt; t++) {
        double s = 0.0;
        for (int k = 0; k < PER; k++) {
            const size_t e = (size_t)t * PER + k;
            const double d = e < x.size() ? x[e] : 0.0f;
            q[t][k] = d * d;
            s += q[t][k];
        }
        pre[t + 1] = pre[t] + s;
    }
    double sum = 0.0;
    ok = true;
    SeqRun run{0.0, 0.0, 0};
    bool some = false;
    uint32_t b = 0;
    for (int t = 0; t < nt; t++) {
        if (seq_is_run(pre[t], pre[t + 1])) {
            double a[PER];
            memcpy(a, q[t].data(), sizeof a);
            b = seq_binade(pre[t]);
            run = seq_join(run, seq_run(a, b));   // pairs joined left to right; the law below covers the scan's pairing
            some = true;
            runs += PER;
            continue;
        }
        if (some) sum = seq_add_run(sum, run, b, ok);
        for (int k = 0; k < PER; k++) sum += q[t][k];
        run = SeqRun{0.0, 0.0, 0};
        some = false;
    }
    if (some) sum = seq_add_run(sum, run, b, ok);
    return sum;
}
static bool same(const SeqRun &a, const SeqRun &b) { return a.a0 == b.a0 && a.a1 == b.a1 && a.e == b.e; }
int main() {
    std::mt19937 g(7);
    std::normal_distribution<float> N(0, 1);
    std::uniform_real_distribution<double> U(0, 1);
    long rows = 0, bad = 0, refused = 0, runs = 0, terms = 0, law = 0;
    for (int it = 0; it < 20000; it++) {
        const int fam = it % 9, n = fam == 8 ? 16384 : 32 * (1 + (int)(U(g) * 96));
        if (fam == 8 && it % 90 != 8) continue;
        std::vector<float> x(n);
        for (int i = 0; i < n; i++) {
            float v = N(g);
            if (fam == 1) v = (float)(int)(v * 4.0f);                         // small integers: ties, zeros
            if (fam == 2) v = ldexpf(v, (int)(U(g) * 80) - 40);               // magnitudes all over
            if (fam == 3) v = ldexpf(1.0f, (int)(U(g) * 6));                  // powers of two: exact binade edges
            if (fam == 4) v *= 1e-30f;
            if (fam == 5) v *= i == n / 2 ? 3e4f : 1.0f;                      // an outlier
            if (fam == 6) v = ldexpf(1.0f + (float)((int)(U(g) * 3)) * 0x1p-23f, (int)(U(g) * 2) * 14);   // odd low bits: ties
            if (fam == 7) v = i < n / 3 ? 0.0f : 0x1p-26f * v + (i == n / 3 ? 1.0f : 0.0f);   // terms near half a unit of the sum
            x[i] = v;
        }
        double want = 0.0;
        for (float v : x) { const double d = v; want += d * d; }
        bool ok;
        const double got = parallel(x, ok, runs);
        rows++;
        terms += n;
        if (!ok) refused++;
        else if (memcmp(&got, &want, 8)) {
            if (bad++ < 3) printf("family %d n %d: %a, in order %a\n", fam, n, got, want);
        }
        if (it == 0) {   // small terms lost in order, not among themselves: the check at the runs' ends refuses the row
            std::vector<float> y(2048, 0x1p-28f);
            double left = 1.0 - 0x1p-53, s = 0.0;
            for (int i = 0; i < 16; i++) {
                float v = (float)sqrt(left);
                while ((double)v * v > left) v = nextafterf(v, 0.0f);
                y[i] = v;
                left -= (double)v * v;
            }
            for (float v : y) s += (double)v * v;
            const double p = parallel(y, ok, runs);
            if (ok) { printf("not refused: %a, in order %a\n", p, s); bad++; }
        }
        // composition is associative, also across ties
        double a[3][PER];
        for (auto &r : a)
            for (double &v : r) v = floor(U(g) * 9) * 0.25;
        const uint32_t b = seq_binade(0x1p51 + 0.0);   // unit 0.5: quarters tie
        const SeqRun A = seq_run(a[0], b), B = seq_run(a[1], b), C = seq_run(a[2], b);
        if (!same(seq_join(seq_join(A, B), C), seq_join(A, seq_join(B, C)))) law++;
    }
    printf("rows %ld bad %ld refused %ld law %ld in runs %.3f\n", rows, bad, refused, law, (double)runs / terms);
    return bad || law;
}
"""


@pytest.fixture(scope="module")
def prog(tmp_path_factory):
    d = tmp_path_factory.mktemp("seqsum")
    src, exe = d / "chk.cpp", d / "chk"
    src.write_text(PROG)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", HDR_DIR, "-o", str(exe), str(src)], check=True)
    return str(exe)


def test_parallel_sum_equals_the_in_order_sum(prog):
    r = subprocess.run([prog], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    f = r.stdout.split()
    assert f[f.index("bad") + 1] == "0" and f[f.index("law") + 1] == "0"
    assert int(f[f.index("refused") + 1]) <= int(f[f.index("rows") + 1]) // 100
