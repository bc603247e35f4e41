// How the SpMM goes about the panels of a weight, on the CPU.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <random>
#include <vector>

#include "csrc/spmm_launch.h"
#include "csrc/weight_internal.h"

using namespace shflbw;

namespace {

std::vector<int> indptr_of(int X, const std::function<int(int)>& kept)
{
    std::vector<int> p(1, 0);
    for (int i = 0; i < X; i++) p.push_back(p.back() + kept(i));
    return p;
}

// Work of the larger part over half of the work, a panel counting as 280 kept vectors more.
double larger_part(const std::vector<int>& p, int first)
{
    const int X = (int)p.size() - 1;
    const double a = p[first] + 280.0 * first, all = p[X] + 280.0 * X;
    return 2 * std::max(a, all - a) / all;
}

// The two parts of the panels are even in work, not in number, or there are none.
int parts_are_even()
{
    std::mt19937 rng(3);
    int bad = 0, uneven = 0, none = 0;
    auto check = [&](const std::vector<int>& p, const char* what) {
        const int X = (int)p.size() - 1, first = spmm_half_panels(p.data(), X);
        double least = X < 2 ? 2 : larger_part(p, 1);
        for (int i = 2; i < X; i++) least = std::min(least, larger_part(p, i));
        const bool ok = first ? first > 0 && first < X && larger_part(p, first) <= std::max(1.03, least) && least <= 1.05 : least > 1.03;
        if (!ok && bad++ < 8) printf("Failed: %s, %d panels: %d in the first part\n", what, X, first);
        none += first == 0, uneven += first && first != X / 2;
    };
    for (int X : {1, 2, 3, 5, 9, 24, 32, 33, 40, 64, 65, 128, 264}) {
        check(indptr_of(X, [&](int) { return 400; }), "panels of one length");
        check(indptr_of(X, [&](int i) { return i < X / 2 ? 900 : 450; }), "a first half of twice the length");
        check(indptr_of(X, [&](int i) { return 1200 - 800 * i / X; }), "falling lengths");
        check(indptr_of(X, [&](int i) { return i == X - 1 ? 6000 : 700; }), "one long panel");
        check(indptr_of(X, [&](int i) { return i ? 0 : 20000; }), "nothing in all but the first panel");
        check(indptr_of(X, [&](int) { return 0; }), "nothing");
        for (int t = 0; t < 50; t++) check(indptr_of(X, [&](int) { return (int)(rng() % 2000); }), "any lengths");
    }
    printf("parts: %d not in the middle, %d times none, %d wrong\n", uneven, none, bad);
    return bad + (uneven < 50) + (none < 20);
}

// The launch of a product with the 256-column variant of block height 128 (of another one: its wide variant) on 256 compute units.
SpmmLaunchArgs launch_of(int V, int K, int N, const std::vector<int>& indptr, bool permuted, bool residual)
{
    const int X = (int)indptr.size() - 1;
    shflbw_spmm_state s;
    memset(&s, 0, sizeof(s));
    s.args.M = X * V, s.args.N = N, s.args.K = K;
    s.args.D = (void*)(uintptr_t)0x10000; // whole lines; never dereferenced
    s.args.A_row_indices = permuted ? indptr.data() : nullptr;
    s.args.alpha = 1.f, s.args.beta = residual ? 1.f : 0.f;
    s.brow = V, s.ldb_bytes = N * 2;
    for (int i = 0; i < X; i++) s.groups += (indptr[i + 1] - indptr[i] + 63) / 64;
    s.half_panels = spmm_half_panels(indptr.data(), X);
    SpmmLaunchArgs a;
    fill_spmm_launch_args(&s, 256, &a);
    return a;
}

} // namespace

// test_spmm_plan: the checks above.  test_spmm_plan launch V K N permuted residual < kept vectors of every panel: whether C is streamed, panels
// of the first half (0: not in halves).
int main(int argc, char** argv)
{
    if (argc == 7 && !strcmp(argv[1], "launch")) {
        std::vector<int> p(1, 0);
        for (int n; scanf("%d", &n) == 1;) p.push_back(p.back() + n);
        const bool residual = atoi(argv[6]);
        const SpmmLaunchArgs a = launch_of(atoi(argv[2]), atoi(argv[3]), atoi(argv[4]), p, atoi(argv[5]), residual);
        printf("%d %d\n", residual && streams_c(a), panel_halves(a, 32) ? a.half_panels : 0);
        return 0;
    }
    const int bad = parts_are_even();
    printf(bad ? "FAILED\n" : "ALL PASSED\n");
    return bad != 0;
}
