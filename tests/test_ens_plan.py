"""The prediction that chooses the ensemble's sweep shapes (csrc/zq3d_ens_plan.h), compiled with g++: for runs of tiles
of any lengths it is the end time of a one-by-one simulation of eight XCDs of 32 CUs, and a run of a
billion tiles costs no more than a short one."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "zq3d_ens_plan.h"
#include <cmath>
#include <cstdio>
#include <functional>
#include <queue>
#include <random>
using namespace zq3d;
static double one_by_one(const std::vector<EnsRun>& runs) {
    std::priority_queue<double, std::vector<double>, std::greater<double>> xcd[8];
    for (auto& q : xcd)
        for (int c = 0; c < 32; c++) q.push(0.0);
    double last = 0.0;
    size_t i = 0;
    for (const EnsRun& r : runs)
        for (long long k = 0; k < r.n; k++, i++) {
            auto& q = xcd[i % 8];
            const double end = q.top() + r.us;
            q.pop();
            q.push(end);
            last = std::max(last, end);
        }
    return last;
}
int main() {
    std::mt19937 rng(5);
    for (int it = 0; it < 3000; it++) {
        std::vector<EnsRun> runs;
        double us = 60.0;
        const int n = 1 + (int)(rng() % 12);
        for (int k = 0; k < n; k++) {
            us *= 0.4 + 0.6 * (rng() % 1000) / 1000.0;
            const int most = rng() % 3 == 0 ? 4000 : 300;
            runs.push_back(EnsRun{us, (long long)(rng() % most)});
        }
        const double a = ens_fill_us(runs), b = one_by_one(runs);
        if (std::fabs(a - b) > 1e-9 * (1.0 + b)) return std::printf("case %d: %.12g, one by one %.12g\n", it, a, b), 1;
    }
    if (ens_fill_us({}) != 0.0) return std::printf("no tiles\n"), 1;
    const double big = ens_fill_us({{2.0, 256LL * 1000000000 + 1}, {1.0, 256LL * 1000000000}});
    if (std::fabs(big - 3e9) > 4.0) return std::printf("long runs: %.12g\n", big), 1;
    std::printf("ok\n");
    return 0;
}
"""


def test_prediction_is_the_one_by_one_simulation(tmp_path):
    src = tmp_path / "plan.cpp"
    src.write_text(SRC)
    exe = str(tmp_path / "plan")
    inc = os.path.join(ROOT, "zq_smokesimulation_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", inc, str(src), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
