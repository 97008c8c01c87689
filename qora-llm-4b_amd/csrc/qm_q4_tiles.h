// qm_q4_tiles.h -- the workgroup tiles of the Q4 prefill GEMM, shared by the
// device code (one kernel per entry and operand type) and the host (which
// tile a call takes).
//
// Tile (MI, NJ, WN, WK): 16 MI rows x 16 NJ WN columns, WN waves side by side
// over the columns and WK groups of them, each on its own share of k.  NST
// LDS stages of 64 rows of k; OCC waves per SIMD the kernel is compiled for.
// The four figures are nanoseconds per stage measured on an MI355X (256 CUs)
// over m = 4 .. 8192 at the projections' k and n: of a workgroup alone on its
// CU, and per workgroup where a CU has several, for an f16 and a bf16 x (the
// bf16 form converts W once more).
//
// X(MI, NJ, WN, WK, NST, OCC, alone f16, shared f16, alone bf16, shared bf16)
#pragma once
#include <stdint.h>

// tiles with an even WN: the gate/up form takes these (half of the waves hold
// the gate weight's columns, half the up weight's)
#define QM_Q4_TILES_PAIRED(X)                             \
    X(1, 2, 2, 4, 3, 4, 446, 438, 643, 545)               \
    X(3, 2, 2, 4, 2, 4, 637, 618, 808, 668)               \
    X(4, 2, 2, 4, 3, 2, 779, 959, 942, 996)               \
    X(4, 2, 4, 2, 3, 4, 718, 651, 850, 713)               \
    X(4, 4, 2, 4, 3, 2, 1242, 1506, 1462, 1552)           \
    X(6, 4, 2, 4, 2, 2, 1658, 1936, 1824, 1949)           \
    X(6, 4, 4, 1, 3, 2, 904, 732, 1038, 819)              \
    X(6, 4, 4, 2, 3, 2, 1432, 1643, 1686, 1743)           \
    X(8, 4, 4, 1, 3, 2, 1098, 912, 1230, 954)             \
    X(8, 4, 4, 2, 3, 2, 1737, 2042, 1967, 2084)
#define QM_Q4_TILES_SINGLE(X)                             \
    X(1, 2, 1, 16, 3, 4, 878, 1456, 1185, 1456)           \
    X(1, 2, 1, 8, 3, 4, 440, 512, 647, 580)               \
    X(2, 2, 1, 8, 3, 2, 618, 962, 789, 899)               \
    X(3, 2, 1, 8, 2, 2, 780, 1197, 959, 1066)             \
    X(4, 2, 1, 8, 2, 2, 952, 1425, 1132, 1248)

// Above this k the tiles' 32-bit lane offsets do not reach (128 rows of x);
// the (1, 2, 2, 4) tile has a form with 64-bit addresses.
#define QM_Q4_GEMM_MAX_K32 (1 << 23)

#ifndef __HIP_DEVICE_COMPILE__
namespace qm_q4 {

struct Tile {
    const char* name;            // kernel name suffix
    int32_t mi, nj, wn, wk;
    int32_t alone[2], shared[2]; // [x is bf16]
};

#define QM_Q4_TILE_ROW(MI, NJ, WN, WK, NST, OCC, AF, SF, AB, SB) \
    {"m" #MI "n" #NJ "w" #WN "k" #WK, MI, NJ, WN, WK, {AF, AB}, {SF, SB}},
constexpr Tile kTiles[] = {QM_Q4_TILES_PAIRED(QM_Q4_TILE_ROW) QM_Q4_TILES_SINGLE(QM_Q4_TILE_ROW)};
#undef QM_Q4_TILE_ROW
constexpr int kBigTile = 0;      // the tile of the form with 64-bit lane offsets
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);

inline int64_t tile_grid(const Tile& t, int64_t m, int64_t n, bool gate_up) {
    const int64_t rows = 16 * t.mi, cols = 16 * t.nj * (gate_up ? t.wn / 2 : t.wn);
    return (m + rows - 1) / rows * ((n + cols - 1) / cols);
}

// The tile a call takes: the one with the least estimated time, stages per
// workgroup times the measured time of a stage times the workgroups of the
// busiest CU.  It weighs what pulls both ways: a large tile dequantizes and
// loads less per product, a small one, or one that splits k over its waves,
// fills the CUs and shortens the chain of stages when there are few rows.
// Over the measured sizes the choice was within 1% of the best of these tiles
// on average (15% at worst).
inline int pick_tile(int64_t m, int64_t k, int64_t n, bool bf16, bool gate_up, int num_cu) {
    int best = -1;
    int64_t best_ns = 0;
    for (int i = 0; i < kNumTiles; ++i) {
        const Tile& t = kTiles[i];
        if (gate_up && t.wn % 2) continue;
        const int64_t stages = ((k / 32 + 1) / 2 + t.wk - 1) / t.wk;
        const int64_t per_cu = (tile_grid(t, m, n, gate_up) + num_cu - 1) / num_cu;
        const int64_t shared = per_cu * t.shared[bf16];
        const int64_t ns = stages * (per_cu == 1 || shared < t.alone[bf16] ? t.alone[bf16] : shared);
        if (best < 0 || ns < best_ns) {
            best = i;
            best_ns = ns;
        }
    }
    return best;
}

}  // namespace qm_q4
#endif
