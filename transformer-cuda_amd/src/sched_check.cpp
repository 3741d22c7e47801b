// sched_check.cpp - host-only checks of the block orders the bf16 and three-plane kernels use
// to turn a workgroup id into (head, block), and of the host rule that picks head groups.
//
// For every order (plain, descending, serpentine, grouped) and a range of grid shapes:
//   * the map is a bijection from [0, BH*nb) onto the (head, block) pairs: no block is
//     skipped or computed twice;
//   * when BH % 8 == 0, workgroup i (which the dispatcher sends to XCD i % 8) gets a head of
//     that XCD, [x*BH/8, (x+1)*BH/8), so a head's tiles stay in one L2;
//   * in the plain and grouped orders, an XCD's workgroups take the blocks heaviest first
//     (non-increasing causal work) within a head, and a group's blocks all come before the
//     next group's.
// And head_group at the bench shapes, with the resident capacities the occupancy query
// reports for those kernels on MI355X; and the forms that on_shared_tiles and on_split_rows pick at
// shapes where one form measured clearly faster.  Prints "sched_check: all passed" on success.
//
// sched_check form STAGE D T BH prints the fp32 form of a call instead (STAGE: fwd, dq, dkdv),
// sched_check form STAGE PLANES D T BH the bf16 (PLANES 1) or three-plane (3) form, and
// sched_check tile M N BATCH K SLICES ARRAYS the GEMM's tile and slices of K (at most SLICES).
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "bf16_tile.hpp"
#include "forms.hpp"
#include "gemm_planes.hpp"
#include "sched.hpp"

using tcamd::head_group;
using tcamd::Stage;
using tcamd::bf16t::map_block;
using tcamd::bf16t::map_block_grouped;

static int failures = 0;

#define CHECK(cond, ...)                                     \
    do {                                                     \
        if (!(cond)) {                                       \
            std::printf("FAIL %s:%d: ", __FILE__, __LINE__); \
            std::printf(__VA_ARGS__);                        \
            std::printf("\n");                               \
            if (++failures > 20) std::exit(1);               \
        }                                                    \
    } while (0)

// order: 0 plain, 1 serpentine, 2 grouped (G)
static void check_order(int BH, int nb, bool descending, int order, int G) {
    std::vector<int> seen(static_cast<size_t>(BH) * nb, 0);
    const int hpx = BH / 8;
    // per head: the last block seen (heaviest first); per XCD: the last group seen
    std::vector<int> last(BH, -1);
    std::vector<int> last_group(8, -1);
    for (int id = 0; id < BH * nb; ++id) {
        int bh = -1, b = -1;
        if (order == 2)
            map_block_grouped(id, BH, nb, G, descending, bh, b);
        else
            map_block(id, BH, nb, descending, order == 1, bh, b);
        CHECK(bh >= 0 && bh < BH && b >= 0 && b < nb,
              "BH %d nb %d order %d G %d id %d -> (%d, %d)", BH, nb, order, G, id, bh, b);
        if (bh < 0 || bh >= BH || b < 0 || b >= nb) continue;
        ++seen[static_cast<size_t>(bh) * nb + b];
        if (BH % 8 == 0) {
            CHECK(bh / hpx == id % 8, "BH %d nb %d order %d G %d: id %d (XCD %d) -> head %d",
                  BH, nb, order, G, id, id % 8, bh);
        }
        if (order != 1) {
            // heaviest first within a head: ascending blocks (key-parallel, block 0 the
            // heaviest) or descending ones (query-parallel, the last block the heaviest)
            if (last[bh] >= 0)
                CHECK(descending ? b < last[bh] : b > last[bh],
                      "BH %d nb %d order %d G %d: head %d block %d after %d", BH, nb, order, G,
                      bh, b, last[bh]);
            last[bh] = b;
        }
        if (order == 2 && G > 0 && BH % 8 == 0 && hpx % G == 0) {
            const int x = id % 8, g = (bh - x * hpx) / G;
            CHECK(g >= last_group[x], "BH %d nb %d G %d: XCD %d back to group %d after %d", BH,
                  nb, G, x, g, last_group[x]);
            last_group[x] = g;
        }
    }
    for (size_t i = 0; i < seen.size(); ++i)
        CHECK(seen[i] == 1, "BH %d nb %d order %d G %d: (head %zu, block %zu) mapped %d times",
              BH, nb, order, G, i / nb, i % nb, seen[i]);
}

// fp32 shapes where one form is the faster one by 8% and more: us on shared tiles and per-wave.
static void check_f32_forms() {
    const struct {
        Stage stage;
        int D, T, BH;
        double shared, per_wave;
    } measured[] = {
        {Stage::Fwd, 64, 100, 64, 13, 7},
        {Stage::Fwd, 64, 100, 200, 13, 16},
        {Stage::Fwd, 64, 128, 256, 14, 16},
        {Stage::Fwd, 64, 230, 256, 31, 38},
        {Stage::Fwd, 64, 777, 27, 61, 37},
        {Stage::Fwd, 64, 1024, 8, 78, 23},
        {Stage::Fwd, 64, 2048, 16, 152, 91},
        {Stage::Fwd, 64, 512, 256, 83, 105},
        {Stage::Fwd, 128, 64, 144, 13, 20},
        {Stage::Fwd, 128, 100, 64, 21, 12},
        {Stage::Fwd, 128, 100, 200, 23, 37},
        {Stage::Fwd, 128, 128, 256, 25, 41},
        {Stage::Fwd, 128, 777, 27, 108, 67},
        {Stage::Fwd, 128, 1024, 8, 139, 43},
        {Stage::Fwd, 128, 2048, 16, 273, 179},
        {Stage::Fwd, 128, 512, 256, 183, 269},
        {Stage::Dq, 64, 100, 64, 19, 12},
        {Stage::Dq, 64, 230, 256, 47, 51},
        {Stage::Dq, 64, 777, 27, 89, 73},
        {Stage::Dq, 64, 1024, 8, 115, 61},
        {Stage::Dq, 64, 2048, 16, 226, 180},
        {Stage::Dq, 128, 100, 64, 33, 20},
        {Stage::Dq, 128, 100, 200, 35, 38},
        {Stage::Dq, 128, 128, 256, 38, 42},
        {Stage::Dq, 128, 777, 27, 162, 122},
        {Stage::Dq, 128, 1024, 8, 210, 108},
        {Stage::Dq, 128, 1200, 96, 572, 525},
        {Stage::Dq, 128, 2048, 16, 414, 321},
        {Stage::Dkdv, 64, 100, 64, 23, 12},
        {Stage::Dkdv, 64, 100, 200, 24, 27},
        {Stage::Dkdv, 64, 230, 256, 58, 70},
        {Stage::Dkdv, 64, 777, 27, 123, 71},
        {Stage::Dkdv, 64, 600, 144, 143, 155},
        {Stage::Dkdv, 64, 1024, 8, 150, 45},
        {Stage::Dkdv, 64, 2048, 16, 294, 182},
        {Stage::Dkdv, 64, 512, 256, 179, 200},
        {Stage::Dkdv, 128, 64, 144, 24, 36},
        {Stage::Dkdv, 128, 100, 64, 43, 21},
        {Stage::Dkdv, 128, 100, 200, 46, 66},
        {Stage::Dkdv, 128, 128, 256, 50, 78},
        {Stage::Dkdv, 128, 777, 27, 230, 136},
        {Stage::Dkdv, 128, 1024, 8, 285, 85},
        {Stage::Dkdv, 128, 2048, 16, 563, 365},
        {Stage::Dkdv, 128, 512, 256, 412, 526},
        {Stage::Dq, 64, 1024, 64, 130, 146},
        {Stage::Dq, 64, 2048, 32, 240, 276},
        {Stage::Dq, 128, 129, 256, 72, 55},
        // the whole dS-first backward
        {Stage::Dkdv, 64, 64, 144, 24, 30},
        {Stage::Dkdv, 64, 100, 64, 37, 25},
        {Stage::Dkdv, 64, 100, 200, 41, 50},
        {Stage::Dkdv, 64, 128, 256, 44, 56},
        {Stage::Dkdv, 64, 230, 256, 89, 127},
        {Stage::Dkdv, 64, 777, 27, 174, 119},
        {Stage::Dkdv, 64, 600, 144, 215, 273},
        {Stage::Dkdv, 64, 1024, 8, 212, 104},
        {Stage::Dkdv, 64, 1200, 96, 490, 588},
        {Stage::Dkdv, 64, 2048, 16, 415, 305},
        {Stage::Dkdv, 64, 512, 256, 283, 365},
        {Stage::Dkdv, 128, 64, 144, 41, 53},
        {Stage::Dkdv, 128, 100, 64, 64, 41},
        {Stage::Dkdv, 128, 100, 200, 70, 91},
        {Stage::Dkdv, 128, 128, 256, 75, 104},
        {Stage::Dkdv, 128, 777, 27, 310, 218},
        {Stage::Dkdv, 128, 1024, 8, 383, 182},
        {Stage::Dkdv, 128, 2048, 16, 757, 562},
        {Stage::Dkdv, 128, 512, 256, 580, 700},
    };
    for (const auto& m : measured)
        CHECK(tcamd::on_shared_tiles(m.stage, m.D, m.T, m.BH) == (m.shared < m.per_wave),
              "stage %d d %d T %d B*H %d takes the slower form (%.0f us shared, %.0f per-wave)",
              static_cast<int>(m.stage), m.D, m.T, m.BH, m.shared, m.per_wave);
    // the sizes at which the entry points stop, and B*H * workgroups beyond 2^31
    for (int st = 0; st < 3; ++st)
        for (int D : {32, 64, 128})
            for (int T : {1, 31, 33, 128, 129, 2048, 2049, 1 << 20, 2147483647})
                for (int BH : {1, 7, 65535}) (void)tcamd::on_shared_tiles(static_cast<Stage>(st), D, T, BH);
}

// The same for sharing rows among a workgroup's waves (three planes: the forward, and the whole
// backward).
static void check_split_rows() {
    const struct {
        Stage stage;
        int planes, D, T, BH;
        double block, split;
    } measured[] = {
        {Stage::Fwd, 1, 32, 1531, 12, 15.7, 8.8},   {Stage::Fwd, 1, 32, 1531, 48, 15.9, 17.8},
        {Stage::Dq, 1, 32, 2048, 16, 24.4, 12.8},   {Stage::Dkdv, 1, 32, 1531, 48, 24.9, 29.2},
        {Stage::Fwd, 1, 64, 1531, 12, 20.2, 11.8},  {Stage::Fwd, 1, 64, 1024, 24, 15.0, 12.3},
        {Stage::Fwd, 1, 64, 777, 48, 12.8, 16.2},   {Stage::Dq, 1, 64, 1531, 12, 26.3, 15.0},
        {Stage::Dq, 1, 64, 777, 27, 16.0, 16.8},    {Stage::Dkdv, 1, 64, 300, 36, 9.5, 10.0},
        {Stage::Dkdv, 1, 64, 777, 12, 17.1, 13.3},  {Stage::Dkdv, 1, 64, 777, 27, 18.2, 20.4},
        {Stage::Fwd, 1, 128, 2048, 12, 50.3, 39.3}, {Stage::Fwd, 1, 128, 777, 27, 22.5, 28.7},
        {Stage::Dq, 1, 128, 449, 27, 18.7, 20.7},   {Stage::Dq, 1, 128, 1024, 12, 33.7, 22.5},
        {Stage::Dkdv, 1, 128, 449, 27, 19.5, 24.2}, {Stage::Dkdv, 1, 128, 4096, 4, 108.5, 73.7},
        {Stage::Fwd, 3, 32, 257, 64, 15.6, 17.5},   {Stage::Fwd, 3, 32, 1531, 12, 50.8, 30.7},
        {Stage::Dkdv, 3, 32, 230, 80, 30.5, 36.4},  {Stage::Dkdv, 3, 32, 777, 27, 73.8, 60.2},
        {Stage::Fwd, 3, 64, 230, 80, 24.6, 29.1},   {Stage::Fwd, 3, 64, 1531, 12, 75.1, 54.0},
        {Stage::Dkdv, 3, 64, 777, 12, 90.0, 69.1},  {Stage::Dkdv, 3, 64, 1024, 24, 113.6, 126.0},
        {Stage::Dkdv, 3, 64, 100, 40, 24.5, 21.7},
    };
    for (const auto& m : measured)
        CHECK(tcamd::on_split_rows(m.stage, m.planes, m.D, m.T, m.BH) == (m.split < m.block),
              "stage %d planes %d d %d T %d B*H %d takes the slower form (%.1f us in 128-row "
              "workgroups, %.1f split)",
              static_cast<int>(m.stage), m.planes, m.D, m.T, m.BH, m.block, m.split);
    for (int st = 0; st < 3; ++st)
        for (int planes : {1, 3})
            for (int D : {32, 64})
                for (int T : {1, 128, 256, 257, 8192, 2147483647})
                    for (int BH : {1, 65535})
                        (void)tcamd::on_split_rows(static_cast<Stage>(st), planes, D, T, BH);
}

// STAGE D T BH, or STAGE PLANES D T BH
static int print_form(int n, char** a) {
    const char* names[] = {"fwd", "dq", "dkdv"};
    for (int st = 0; st < 3; ++st)
        if (std::strcmp(a[0], names[st]) == 0) {
            const Stage stage = static_cast<Stage>(st);
            int x[4] = {};
            for (int i = 1; i < n; ++i) x[i - 1] = std::atoi(a[i]);
            if (n == 4)
                std::printf("%s\n", tcamd::on_shared_tiles(stage, x[0], x[1], x[2]) ? "shared"
                                                                                    : "per-wave");
            else
                std::printf("%s\n", tcamd::on_split_rows(stage, x[0], x[1], x[2], x[3]) ? "split"
                                                                                         : "block");
            return 0;
        }
    return 2;
}

static int print_tile(char** a) {
    int x[6];
    for (int i = 0; i < 6; ++i) x[i] = std::atoi(a[i]);
    const tcamd::gemm::Plan p = tcamd::gemm::pick_tile(x[0], x[1], x[2], x[3], x[4], x[5]);
    const tcamd::gemm::TileRate& t = tcamd::gemm::kTiles[p.tile];
    std::printf("%dx%d %d\n", t.bm, t.bn, p.slices);
    return 0;
}

int main(int argc, char** argv) {
    if (argc == 8 && std::strcmp(argv[1], "tile") == 0) return print_tile(argv + 2);
    if ((argc == 6 || argc == 7) && std::strcmp(argv[1], "form") == 0)
        return print_form(argc - 2, argv + 2);
    const int bhs[] = {1, 3, 8, 12, 16, 24, 64, 96, 128, 256, 384};
    const int nbs[] = {1, 2, 7, 8, 16, 33, 64};
    for (int BH : bhs)
        for (int nb : nbs)
            for (int desc = 0; desc < 2; ++desc) {
                check_order(BH, nb, desc != 0, 0, 0);
                check_order(BH, nb, desc != 0, 1, 0);
                for (int G : {0, 1, 2, 4, 8, 16, 32}) check_order(BH, nb, desc != 0, 2, G);
            }

    // head_group(BH, nblk, resident): the groups the bench workloads get.
    // Config 3 (B16 H16 T2048 d64): bf16 dK/dV, 16 key blocks, two workgroups per CU.
    CHECK(head_group(256, 16, 512) == 8, "config 3 dK/dV: %d", head_group(256, 16, 512));
    // Config 3 forward: 16 query blocks, four workgroups per CU.
    CHECK(head_group(256, 16, 1024) == 16, "config 3 forward: %d", head_group(256, 16, 1024));
    // B16 H16 T1024 dK/dV: 8 key blocks, so a group of 8 heads fills the slots once; 16.
    CHECK(head_group(256, 8, 512) == 16, "B16 H16 T1024 dK/dV: %d", head_group(256, 8, 512));
    // B16 H16 T512 dK/dV: no group below 32 heads fills the slots twice.
    CHECK(head_group(256, 4, 512) == 0, "B16 H16 T512 dK/dV: %d", head_group(256, 4, 512));
    // Config 2 (B8 H12): 12 heads per XCD, no power of two >= 8 divides them.
    CHECK(head_group(96, 8, 512) == 0, "config 2: %d", head_group(96, 8, 512));
    // Config 4 (B2 H16 T8192 d128): 4 heads per XCD, below the smallest group.
    CHECK(head_group(32, 64, 256) == 0, "config 4: %d", head_group(32, 64, 256));
    // Heads not a multiple of the XCD count.
    CHECK(head_group(100, 64, 512) == 0, "BH 100: %d", head_group(100, 64, 512));
    // G stays below the heads per XCD (G = hpx is the plain order).
    CHECK(head_group(64, 64, 256) == 0, "BH 64: %d", head_group(64, 64, 256));

    check_f32_forms();
    check_split_rows();

    if (failures) {
        std::printf("sched_check: %d failures\n", failures);
        return 1;
    }
    std::printf("sched_check: all passed\n");
    return 0;
}
