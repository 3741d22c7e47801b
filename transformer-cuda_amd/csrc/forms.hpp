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

// bf16 (planes = 1) and three planes: whether a stage's waves share out the streamed rows of one
// 32-row block (flash_*_split_kernel) instead of each walking the whole range of its own 32 rows of
// 128.  Sharing ends with the longest range / 4, but copies every tile for 32 rows instead of 128:
// it is the faster form while 128-row workgroups leave CUs idle, and up to more of them the longer
// the ranges are, as copying is then the smaller part.  So the limit on 128-row workgroups is a line
// in T, bounded where the chip is filled either way; up to `from` keys there is too little to share
// (equal times).  The lines lie between the last shapes that gain and the first that lose in 780
// shapes of each type and d, from B*H 1 to 400 and T 33 to 8192, measured in both forms: none loses
// more than 5%.  Measured (us, 128-row workgroups -> shared rows; number of workgroups):
//   bf16 d 32   B*H 12 T 1531 (144), fwd 15.7 -> 8.8, dQ 19.0 -> 9.9, dK/dV 21.7 -> 12.4
//               B*H 48 T 777 (336), fwd 9.7 -> 8.5, dQ 12.0 -> 10.5, dK/dV 14.3 -> 12.5
//   bf16 d 64   B*H 12 T 1531 (144), fwd 20.2 -> 11.8, dQ 26.3 -> 15.0, dK/dV 27.7 -> 19.4
//               B*H 27 T 777 (189), fwd 12.5 -> 11.8, dQ 16.0 -> 16.8, dK/dV 18.2 -> 20.4
//   bf16 d 128  B*H 12 T 1024 (96), fwd 27.6 -> 15.2, dQ 33.7 -> 22.5, dK/dV 32.2 -> 27.4
//               B*H 27 T 449 (108), fwd 15.2 -> 14.9, dQ 18.7 -> 20.7, dK/dV 19.5 -> 24.2
//   three planes, the whole backward: d 32   B*H 16 T 2048 (256) 173 -> 127, B*H 80 T 230 (160) 31 -> 36
//               d 64   B*H 12 T 1531 (144) 162 -> 146, B*H 24 T 1024 (192) 114 -> 126
inline bool on_split_rows(Stage stage, int planes, int D, int T, int BH) {
    struct Line {
        int from, base, per, most;
    };
    static constexpr Line kBf16[3][3] = {  // d 32, 64, 128
        {{256, 224, 8, 480}, {256, 190, 4, 576}, {256, 244, 15, 384}},
        {{256, 92, 8, 320}, {256, 72, 8, 320}, {256, 60, 9, 208}},
        {{256, 97, 16, 224}, {256, 32, 8, 192}, {256, 33, 11, 128}}};
    static constexpr Line kThree[2][2] = {  // d 32, 64: forward, backward
        {{288, 120, 7, 256}, {128, 94, 5, 256}}, {{256, 104, 10, 256}, {128, 108, 32, 144}}};
    const long long nblk = static_cast<long long>(BH) * ((T - 1) / 128 + 1);
    const int d = D == 32 ? 0 : D == 64 ? 1 : 2;
    if (planes == 3 && stage != Stage::Fwd && T <= 128) return nblk <= (D == 32 ? 48 : 64);
    const Line& l = planes == 3 ? kThree[d][stage != Stage::Fwd] : kBf16[d][static_cast<int>(stage)];
    return T > l.from && nblk <= std::min(l.base + T / l.per, l.most);
}

}  // namespace tcamd
