// The planner of the convolution's patch form on the CPU: what a workgroup of the cut it picks would read from LDS, for
// seeded random layers.  The walk below restates the kernel's addressing (position -> column offset, kept column -> row).
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "csrc/spconv_patch.h"

using namespace shflbw;

namespace {

struct Layer {
    int V, F, C, R, S, permuted, B, H, W, stride;
    double density;
};

ConvPatchProblem problem(const Layer& l)
{
    return ConvPatchProblem{l.V, l.F, l.C, l.R, l.S, l.density * l.R * l.S * l.C, l.permuted, l.B, l.H, l.W,
                            (l.H + 2 * (l.R / 2) - l.R) / l.stride + 1, (l.W + 2 * (l.S / 2) - l.S) / l.stride + 1, l.stride, 256};
}

// Ordinary layers, and (one in four) the corners: strides as wide as the filter, filters of one row, narrow maps.
Layer random_layer(std::mt19937& rng)
{
    auto pick = [&](std::initializer_list<int> v) { return v.begin()[rng() % v.size()]; };
    Layer l{};
    l.V = pick({16, 32, 64, 128});
    l.F = l.V * (1 + (int)(rng() % 16));
    l.C = 8 * (1 + (int)(rng() % 64));
    l.permuted = rng() % 2;
    l.B = 1 + (int)(rng() % 64);
    l.density = 0.05 + (rng() % 100) / 110.0;
    if (rng() % 4) {
        l.R = pick({1, 3, 3, 5, 7}), l.S = rng() % 4 ? l.R : pick({1, 2, 3, 4, 7});
        l.H = 3 + (int)(rng() % 56), l.W = rng() % 2 ? l.H : 3 + (int)(rng() % 56);
        l.stride = 1 + (int)(rng() % 3);
    } else {
        l.R = pick({1, 1, 2, 7}), l.S = pick({1, 2, 5, 6, 7, 9, 11});
        l.H = 1 + (int)(rng() % 24), l.W = 1 + (int)(rng() % 24);
        l.stride = 1 + (int)(rng() % 11);
    }
    if (l.H + 2 * (l.R / 2) < l.R || l.W + 2 * (l.S / 2) < l.S) return random_layer(rng);
    return l;
}

// One byte past the last one that any lane of the kernel reads from the patch, counted from its first row.
long patch_end(const Layer& l, const ConvPatchPlan& p)
{
    long col = 0;
    for (int pos = 0; pos < 8 * p.col_blocks; pos++) {
        const int i = pos / p.row_len, j = pos % p.row_len;
        if (i < p.tile_h) col = std::max(col, (long)(i * p.step_h * p.patch_w + j * p.step_w) * 8);
    }
    long row = (long)l.C * p.pitch; // the row of zeros
    for (int r = 0; r < l.R; r++)
        for (int s = 0; s < l.S; s++) row = std::max(row, (l.C - 1L) * p.pitch + (r * p.patch_w + s) * 8);
    return row + col + 8;
}

int reads_stay_inside()
{
    std::mt19937 rng(2024);
    int bad = 0, taken = 0;
    for (int t = 0; t < 20000; t++) {
        // first the one-row filter whose stride leaves one output column per unit
        const Layer l = t == 0 ? Layer{32, 32, 8, 1, 7, 1, 4, 4, 7, 7, 0.5} : random_layer(rng);
        ConvPatchPlan p;
        if (!conv_patch_plan(problem(l), &p)) continue;
        taken++;
        const long place = 128 * p.col_blocks, end = patch_end(l, p);
        if (place + end > p.lds_bytes || p.lds_bytes > CONV_PATCH_LDS_MAX) {
            if (bad++ < 5)
                printf("Failed: V %d F %d C %d %dx%d map %dx%d stride %d: reads to %ld of %d bytes\n", l.V, l.F, l.C, l.R, l.S, l.H, l.W,
                       l.stride, place + end, p.lds_bytes);
        }
    }
    printf("reads: %d cuts, %d past the LDS of the workgroup\n", taken, bad);
    return bad + (taken < 5000);
}

// The order of a panel's kept columns by the rule as it is stated at ConvPatchOrder, one start pair at a time.
struct PlainOrder {
    uint32_t foot;
    int group;

    uint32_t row(int s) const { return s ? (foot << s) | (foot >> (32 - s)) : foot; }

    void tilings(std::vector<int>& shifts, uint32_t used, std::vector<std::vector<int>>& found) const
    {
        if ((int)shifts.size() == group) {
            found.push_back(shifts);
            return;
        }
        const uint32_t lowest = ~used & (used + 1);
        for (int s = 1; s < 32 && found.size() < 3; s++)
            if ((row(s) & lowest) && !(row(s) & used)) {
                shifts.push_back(s);
                tilings(shifts, used | row(s), found);
                shifts.pop_back();
            }
    }

    std::vector<int> of(const std::vector<int>& pair_of) const
    {
        std::vector<int> order;
        std::vector<std::vector<int>> left(32), found;
        for (size_t i = pair_of.size(); i-- > 0;) left[pair_of[i]].push_back((int)i);
        auto take = [&](int s) { order.push_back(left[s].back()), left[s].pop_back(); };
        std::vector<int> shifts{0};
        tilings(shifts, foot, found);
        while (true) { // the tiling and shift whose scarcest member has the most rows left, the first of equals
            int best = 0, at = 0, shift = 0;
            for (size_t t = 0; t < found.size(); t++)
                for (int s = 0; s < 32; s++) {
                    int least = 1 << 30;
                    for (int d : found[t]) least = std::min(least, (int)left[(s + d) & 31].size());
                    if (least > best) best = least, at = (int)t, shift = s;
                }
            if (!best) break;
            for (; best > 0; best--)
                for (int d : found[at]) take((shift + d) & 31);
        }
        while (order.size() < pair_of.size()) { // a row that meets the fewest rows of its group; of those the one with most rows left
            std::vector<int> touched(32, 0);
            for (int g = 0; g < group && order.size() < pair_of.size(); g++) {
                int pick = -1, meets = 0;
                for (int s = 0; s < 32; s++) {
                    if (left[s].empty()) continue;
                    int worst = 0;
                    for (int b = 0; b < 32; b++)
                        if (row(s) >> b & 1) worst = std::max(worst, touched[b]);
                    if (pick < 0 || worst < meets || (worst == meets && left[s].size() > left[pick].size())) pick = s, meets = worst;
                }
                for (int b = 0; b < 32; b++) touched[b] += row(pick) >> b & 1;
                take(pick);
            }
        }
        return order;
    }
};

int orders_follow_the_rule()
{
    std::mt19937 rng(7);
    int bad = 0;
    for (int t = 0; t < 3000; t++) {
        const int group = rng() % 2 ? 4 : 8, n = (int)(rng() % (t % 10 ? 90 : 700)), step = 1 + (int)(rng() % 31);
        uint32_t foot = 0; // a row of positions `step` pairs apart, or (one in four) positions anywhere
        for (int i = 0; i < 32 / group; i++) foot |= 1u << (t % 4 ? i * step & 31 : (int)(rng() % 32));
        std::vector<int> pair_of(n), order;
        const int spread = rng() % 3 ? 32 : 1 + (int)(rng() % 32); // some panels keep few start pairs
        for (int& s : pair_of) s = (int)(rng() % spread);
        ConvPatchOrder(foot, group).of(pair_of, order);
        if (order != PlainOrder{foot, group}.of(pair_of) && bad++ < 5) printf("Failed: order of %d rows, foot %08x, groups of %d\n", n, foot, group);
    }
    printf("orders: %d differ from the rule\n", bad);
    return bad;
}

// With shapes to choose from, the plan has one of them; with its own shape among them it is the plan it would be without.
int plans_keep_to_held_shapes()
{
    std::mt19937 rng(99);
    int bad = 0, other = 0;
    for (int t = 0; t < 3000; t++) {
        Layer l = random_layer(rng);
        const ConvPatchProblem q = problem(l);
        const int rows = conv_patch_unit_rows(l.V);
        ConvPatchPlan free{}, p{};
        if (!conv_patch_plan(q, &free)) continue;
        const ConvPatchShape own = conv_patch_shape(rows, free);
        std::vector<ConvPatchShape> held;
        if (conv_patch_plan(q, &p, &held)) bad++;
        // shapes of the same layer over other maps, as a filter that serves them holds them
        for (int i = 0; i < 4; i++) {
            Layer m = l;
            m.B = 1 + (int)(rng() % 64), m.H = l.R + (int)(rng() % 40), m.W = l.S + (int)(rng() % 40);
            if (conv_patch_plan(problem(m), &p) && !(conv_patch_shape(rows, p) == own)) held.push_back(conv_patch_shape(rows, p));
        }
        if (conv_patch_plan(q, &p, &held)) {
            other++;
            bad += std::find(held.begin(), held.end(), conv_patch_shape(rows, p)) == held.end() || p.lds_bytes > CONV_PATCH_LDS_MAX ||
                   128 * p.col_blocks + patch_end(l, p) > p.lds_bytes;
        }
        held.push_back(own);
        bad += !conv_patch_plan(q, &p, &held) || memcmp(&p, &free, sizeof(p)) != 0;
    }
    printf("held shapes: %d plans with another shape, %d wrong\n", other, bad);
    return bad + (other < 500);
}

// Wide cuts are a further choice of the patch form: a layer that takes the form without them takes it with them.
int wide_cuts_keep_the_form()
{
    // permuted layers whose wide cut is estimated ahead of the best other one by its own weights, and behind the plane forms without them
    std::vector<Layer> layers{{64, 1984, 184, 1, 1, 1, 32, 38, 26, 1, 22.6 / 184}, {64, 1984, 168, 1, 1, 1, 23, 38, 38, 1, 0.06},
                              {32, 1920, 304, 1, 1, 1, 57, 19, 19, 1, 0.19},       {128, 1920, 328, 1, 1, 1, 31, 31, 31, 1, 0.09},
                              {32, 1984, 120, 1, 1, 1, 46, 29, 29, 1, 0.22}};
    std::mt19937 rng(11);
    auto spread = [&](int lo, int hi) { return std::exp(std::log((double)lo) + rng() % 10000 / 10000.0 * std::log((double)hi / lo)); };
    for (int t = 0; t < 2500; t++) {
        Layer l{};
        l.V = 16 << rng() % 4;
        l.F = std::max(512 / l.V + 1, (int)(spread(512, 2048) / l.V)) * l.V;
        l.C = 8 * (int)spread(2, 128);
        l.R = l.S = 1 + 2 * (int)(rng() % 3);
        if (rng() % 6 == 0) l.R = 1, l.S = 7;
        l.permuted = 1, l.B = (int)spread(1, 128), l.H = (int)spread(5, 56), l.W = rng() % 2 ? l.H : (int)spread(5, 56);
        l.stride = rng() % 10 < 7 ? 1 : 2, l.density = spread(5, 50) / 100;
        layers.push_back(l);
    }
    int bad = 0, wide = 0;
    for (const Layer& l : layers) {
        ConvPatchPlan with{}, without{};
        if (!conv_patch_plan(problem(l), &without, nullptr, false)) continue;
        bad += without.deep == CONV_PATCH_WIDE;
        if (!conv_patch_plan(problem(l), &with) || (without.preferred && !with.preferred)) {
            if (bad++ < 8)
                printf("Failed: V %d F %d C %d %dx%d map %d x %dx%d stride %d density %g: the plane forms take it from a wide cut\n", l.V, l.F, l.C,
                       l.R, l.S, l.B, l.H, l.W, l.stride, l.density);
        }
        wide += with.deep == CONV_PATCH_WIDE;
    }
    printf("wide cuts: %d layers, %d left to the plane forms for one\n", wide, bad);
    return bad + (wide < 500);
}

// Where a wide cut and the chunks are estimated alike the layer stays in chunks (these were 1.03 to 1.23 times as long on wide cuts).
int ties_stay_in_chunks()
{
    int bad = 0;
    for (const Layer& l : {Layer{64, 576, 144, 1, 1, 1, 9, 46, 5, 1, 0.122}, Layer{64, 576, 32, 3, 3, 1, 12, 6, 24, 1, 0.058},
                           Layer{64, 576, 24, 1, 1, 1, 8, 15, 17, 1, 0.144}, Layer{64, 576, 24, 1, 1, 1, 3, 25, 25, 1, 0.198},
                           Layer{64, 576, 16, 1, 7, 1, 3, 19, 44, 1, 0.247}, Layer{64, 576, 16, 1, 1, 1, 12, 12, 12, 1, 0.106},
                           Layer{64, 576, 64, 1, 1, 1, 4, 23, 23, 1, 0.257}, Layer{64, 576, 16, 1, 7, 1, 13, 31, 6, 1, 0.096}}) {
        ConvPatchPlan p{};
        bad += !conv_patch_plan(problem(l), &p) || p.deep == CONV_PATCH_WIDE;
    }
    printf("ties: %d on wide cuts\n", bad);
    return bad;
}

} // namespace

// test_patch_plan: the checks above.  test_patch_plan cut V F C R S nnzb permuted B H W stride: the cut of one layer, as
// rows of a row unit, 32-column blocks, waves, row units of a wave, parts of the kept columns, workgroups of a column tile.
int main(int argc, char** argv)
{
    if (argc == 13 && !strcmp(argv[1], "cut")) {
        int v[11];
        for (int i = 0; i < 11; i++) v[i] = atoi(argv[2 + i]);
        Layer l{v[0], v[1], v[2], v[3], v[4], v[6], v[7], v[8], v[9], v[10], 0};
        ConvPatchProblem q = problem(l);
        q.kept_per_panel = (double)v[5] / (l.F / l.V);
        ConvPatchPlan p{};
        if (!conv_patch_plan(q, &p)) return 1;
        printf("%d %d %d %d %d %d %d\n", conv_patch_unit_rows(l.V), p.col_blocks, p.waves, p.panels_per_wave, p.ksplit, p.chunks, p.deep);
        return 0;
    }
    const int bad = reads_stay_inside() + orders_follow_the_rule() + plans_keep_to_held_shapes() + wide_cuts_keep_the_form() +
                    ties_stay_in_chunks();
    printf(bad ? "FAILED\n" : "ALL PASSED\n");
    return bad != 0;
}
