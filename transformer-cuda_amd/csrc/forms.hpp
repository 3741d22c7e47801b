// forms.hpp - which form of an attention kernel a call takes where two of them compute the same
// stage.  Host only.
#pragma once

#include <algorithm>

namespace tcamd {

enum class Stage { Fwd, Dq, Dkdv };

// Estimated time, in the unit of `cost`, that 256 CUs take for the jobs of `heads` heads with costs
// cost(0) >= cost(1) >= ... >= cost(n - 1) each (their sum: sum), longest first: halfway between the
// even share and rounds of 256 jobs that end with their longest.  `paired`: the even share alone.
template <class Cost>
double makespan(Cost cost, int n, double sum, int heads, bool paired) {
    constexpr int kCus = 256;
    const double even = std::max(cost(0), sum * heads / kCus);
    const long long jobs = static_cast<long long>(n) * heads;
    if (paired) return even;
    if (jobs > 64 * kCus) return even + 0.25 * cost(0);  // the rounds' ends in the limit
    double rounds = 0.0;
    for (long long j = 0; j < jobs; j += kCus) rounds += cost(static_cast<int>(j / heads));
    return 0.5 * (even + rounds);
}

// fp32: a stage on shared tiles (flash_*_f32_shared_kernel: 128 rows per workgroup, which walks
// their range of 32-row tiles by itself), or on the persistent per-wave kernel, whose four waves
// share out the range of every 32 rows.  Shared tiles are read once for 128 rows instead of 32, but
// 128 rows are a coarse unit: with fewer than two workgroups a CU, or an uneven last round, the
// time is that of the longest range.  So both times are estimated: tile steps for the shared form,
// a quarter of them and a merge's worth for the other; `merge`, the price of a step of it and the
// shared form's start are fitted to some 710 shapes of each d, from B*H 1 to 400 and T 33 to 2048,
// measured in both forms.  The times over all of them are within 0.6% of the better forms'.  Of the
// slower picks, the forward and dQ have 4 to 11 of more than 5%, of 19% at most.  dK/dV
// goes by one rule with and without dS, whose dK and dV are the same bits: as writing dS costs the
// per-wave form more, the rule leaves it earlier than dK/dV alone would.
// Measured (us, shared -> per-wave):
//   d 64    B*H 8 T 1024, fwd 78 -> 23       B*H 27 T 777, dQ 89 -> 73       B*H 48 T 1024, dK/dV 189 -> 140
//           B*H 200 T 100, fwd 13 -> 16      B*H 256 T 230, dK/dV 58 -> 70   B*H 96 T 1024, fwd 135 -> 138
//           B*H 56 T 1024, dK/dV 203 -> 160, the whole dS-first backward 294 -> 270
//           B*H 144 T 600, dK/dV 143 -> 155, dS-first 215 -> 273
//   d 128   B*H 16 T 2048, fwd 273 -> 179    B*H 144 T 64, fwd 13 -> 20      B*H 256 T 128, dK/dV 50 -> 78
//           B*H 27 T 777, dQ 162 -> 122      B*H 32 T 2048, fwd 293 -> 345
// d 64 beyond T 2048: the shared form's static block order balances long causal ranges worse than
// the queue (B1 H12 T8192 forward 886 per-wave, 1086 shared).  d 32: B8 H12 T1024 forward 72
// per-wave, 74 shared.
inline bool on_shared_tiles(Stage stage, int D, int T, int BH) {
    if (D == 32 || (D == 64 && T > 2048)) return false;
    struct Fit {
        double merge, step, start;
    };
    static constexpr Fit kFit[2][3] = {{{0.5, 1.0, 1.0}, {0.5, 0.85, 1.5}, {1.0, 1.025, 1.0}},
                                       {{1.5, 0.975, 1.5}, {1.0, 0.75, 1.0}, {0.5, 1.325, 1.0}}};
    const Fit& f = kFit[D == 128][static_cast<int>(stage)];
    const int nt = (T - 1) / 32 + 1, nb = (T - 1) / 128 + 1;
    // workgroup b of a head: 4 (b + 1) steps, the last one nt
    const auto shared = [&](int r) { return std::min(4.0 * (nb - r), static_cast<double>(nt)); };
    const double shared_sum = 2.0 * nb * (nb - 1.0) + nt;
    // task i: the waves' share of its i + 1 steps
    const auto wave = [&](int r) { return (nt - r + 3) / 4 + f.merge; };
    const double q = nt / 4, rest = nt % 4;
    const double wave_sum = 2.0 * q * (q + 1.0) + rest * (q + 1.0) + f.merge * nt;
    // two workgroups a CU, all resident and nearly full, in serpentine order: each CU has a long and
    // a short one (B*H 64 T 1024 d 64 dQ 130 shared, 146 per-wave); other whole rounds in
    // heaviest-first order give every CU about the same mix too
    const long long nblk = static_cast<long long>(nb) * BH;
    if (nblk == 512 && static_cast<long long>(T) * BH >= 512 * 128 * 85 / 100) return true;
    const bool paired = nblk >= 512 && nblk % 256 == 0;
    return f.start + makespan(shared, nb, shared_sum, BH, paired) <
           f.step * makespan(wave, nt, wave_sum, BH, false);
}

}  // namespace tcamd
