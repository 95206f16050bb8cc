// Walks the column kernels' pixel lists (multigpugridder_amd/csrc/mgg_columns.h)
// on the CPU.  "rows": for every row length, the offsets the walk evaluates.
// "range": over random frames, each extreme then climbed to a local maximum,
// the largest and smallest pair-table index along the column that a walk of
// clamp-free slots looks up, per direction of the projection and slots.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <random>
#include <utility>
#include <vector>

#include "mgg_columns.h"

using namespace mgg;

static std::vector<int> walk(int cnt)
{
    std::vector<int> seen;
    const auto add = [&](int e, int n) { for (int q = 0; q < n; q++) seen.push_back(e + q); };
    col_row(cnt, [&](auto first, auto np) { add(decltype(first)::value, decltype(np)::value); },
            [&](int e, auto np) { add(e, decltype(np)::value); });
    return seen;
}

struct Angles { double th, ph, ps; };
struct Reach { int slots; double lo, hi; };

// How far the last index of a column lies below its first: slots are looked up
// in pairs, and one by one.
static double below(int mode, int slots)
{
    const int pairs = col_clamps(mode, slots) ? 0 : 250 * ((slots + 1) / 2 - 1);
    const int singles = col_clamps_single(mode, slots) ? 0 : 125 * (slots - 1);
    return pairs > singles ? pairs : singles;
}

// One frame's slots and its extreme indices, over all places where the column
// can meet the plane (its remainder to the pixel grid and to the voxels).
static Reach reach(int mode, const Angles &p, const std::vector<int> (&walks)[17])
{
    const double st = std::sin(p.th), ct = std::cos(p.th), sp = std::sin(p.ph), cp = std::cos(p.ph);
    const double n[3] = {st * cp, st * sp, ct}, e1[3] = {ct * cp, ct * sp, -st}, e2[3] = {-sp, cp, 0.0};
    double u[3], v[3];
    for (int k = 0; k < 3; k++) {
        u[k] = std::cos(p.ps) * e1[k] + std::sin(p.ps) * e2[k];
        v[k] = -std::sin(p.ps) * e1[k] + std::cos(p.ps) * e2[k];
    }
    int c = 0;
    for (int k = 1; k < 3; k++)
        if (std::fabs(n[k]) > std::fabs(n[c])) c = k;
    const int axes[2] = {(c + 1) % 3, (c + 2) % 3};
    const double l1 = std::fabs(n[0]) + std::fabs(n[1]) + std::fabs(n[2]);
    const double half = (mode == COL_BACK ? 2.0 : 2.0 * l1) / std::fabs(n[c]);
    const int slots = col_slots(mode, (float)(2.0 * half + 1.5e-2));
    double dlo = 1e30, dhi = -1e30;
    for (int dj = -8; dj < 8; dj++) {
        double lo = -8.0, hi = 7.0;
        for (int a : axes) {
            const double L = col_list_reach((float)u[a], (float)v[a]);
            if (std::fabs(u[a]) < 1e-6) {
                if (std::fabs(v[a] * dj) > L) hi = -9.0;
            } else {
                const double x = (-L - v[a] * dj) / u[a], y = (L - v[a] * dj) / u[a];
                lo = std::fmax(lo, std::ceil(std::fmin(x, y)));
                hi = std::fmin(hi, std::floor(std::fmax(x, y)));
            }
        }
        const int cnt = (int)(hi - lo) + 1;
        if (cnt <= 0) continue;
        for (int e : walks[cnt]) {
            const double d = (lo + e) * u[c] + dj * v[c];
            dlo = std::fmin(dlo, d);
            dhi = std::fmax(dhi, d);
        }
    }
    // slot 0 lies in (half - 1, half] beyond where the column meets the plane
    // (plus 5e-3 for rounding); the transpose counts the other way
    const double f = 0.5 * (std::fabs(u[c]) + std::fabs(v[c]));
    if (mode == COL_ADJOINT) { const double t = dlo; dlo = -dhi; dhi = -t; }
    return {slots, 250.0 + 125.0 * (dlo - f + half + 5e-3 - 1.0) - 0.5 - below(mode, slots),
            250.0 + 125.0 * (dhi + f + half + 5e-3) + 0.5};
}

int main(int argc, char **argv)
{
    std::vector<int> walks[17];
    for (int cnt = 0; cnt <= 16; cnt++) walks[cnt] = walk(cnt);
    if (argc > 1 && !std::strcmp(argv[1], "rows")) {
        for (int cnt = 0; cnt <= 16; cnt++) {
            std::printf("%d", cnt);
            for (int e : walks[cnt]) std::printf(" %d", e);
            std::printf("\n");
        }
        return 0;
    }
    std::mt19937_64 gen(1);
    std::uniform_real_distribution<double> uni(0.0, 1.0);
    std::normal_distribution<double> gauss;
    for (int mode : {COL_BACK, COL_ADJOINT}) {
        struct Best { double value = -1e30; Angles at{}; };
        std::map<std::pair<int, int>, std::vector<Best>> best;  // (slots, sign), eight starts each
        for (int t = 0; t < 400000; t++) {
            const Angles p{std::acos(2.0 * uni(gen) - 1.0), 2.0 * M_PI * uni(gen), 2.0 * M_PI * uni(gen)};
            const Reach r = reach(mode, p, walks);
            if (col_clamps(mode, r.slots) && col_clamps_single(mode, r.slots)) continue;
            for (int sign : {-1, 1}) {
                auto &list = best[{r.slots, sign}];
                list.resize(8);
                Best &b = list[t % 8];
                const double val = sign > 0 ? r.hi : -r.lo;
                if (val > b.value) b = {val, p};
            }
        }
        for (auto &[key, list] : best) {
            double top = -1e30;
            for (Best &b : list) {
                double step = 0.1;
                for (int it = 0; it < 4000; it++) {
                    const Angles q{b.at.th + step * gauss(gen), b.at.ph + step * gauss(gen), b.at.ps + step * gauss(gen)};
                    const Reach r = reach(mode, q, walks);
                    const double val = key.second > 0 ? r.hi : -r.lo;
                    if (r.slots == key.first && val > b.value) b = {val, q};
                    else if (it % 200 == 199) step *= 0.6;
                }
                top = std::fmax(top, b.value);
            }
            std::printf("%d %d %d %.3f %d %d\n", mode, key.first, key.second, key.second * top, ct_lo(mode), ct_hi(mode));
        }
    }
    return 0;
}
