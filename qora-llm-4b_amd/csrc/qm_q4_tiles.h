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
// Gate/up needs two equal halves of a workgroup, one per weight: of the WN
// waves side by side, or of the k-groups where WN is 1.
//
// X(MI, NJ, WN, WK, NST, OCC, alone f16, shared f16, alone bf16, shared bf16)
#pragma once
#include <stdint.h>

#define QM_Q4_TILES_ONE_WAVE(X)                 \
    X(1, 2, 1, 8, 3, 4, 424, 445, 595, 546)     \
    X(1, 2, 1, 16, 2, 4, 733, 1161, 1061, 1320) \
    X(1, 4, 1, 8, 2, 4, 608, 690, 994, 921)     \
    X(2, 2, 1, 8, 2, 2, 488, 731, 680, 787)     \
    X(2, 4, 1, 8, 2, 2, 787, 1092, 1100, 1207)  \
    X(3, 2, 1, 8, 2, 2, 623, 903, 773, 890)     \
    X(3, 4, 1, 8, 2, 2, 1058, 1370, 1285, 1426) \
    X(4, 2, 1, 8, 2, 2, 792, 1105, 896, 1031)   \
    X(5, 4, 1, 4, 2, 1, 932, 1050, 1008, 1068)  \
    X(6, 4, 1, 4, 2, 1, 1075, 1210, 1097, 1170)
// no call takes its gate/up form with an f16 x: not built
#define QM_Q4_TILES_GATE_UP_BF16(X)             \
    X(8, 4, 1, 4, 2, 1, 1348, 1463, 1364, 1442)
#define QM_Q4_TILES_PAIRED(X)                   \
    X(3, 2, 2, 4, 2, 4, 641, 627, 797, 669)     \
    X(4, 2, 4, 2, 3, 4, 696, 649, 864, 715)     \
    X(6, 4, 2, 4, 2, 2, 1650, 1967, 1797, 1931) \
    X(6, 4, 4, 1, 3, 2, 888, 734, 1006, 812)    \
    X(6, 4, 4, 2, 3, 2, 1427, 1652, 1681, 1760) \
    X(8, 4, 4, 1, 3, 2, 1089, 907, 1220, 942)   \
    X(8, 4, 4, 2, 3, 2, 1736, 2032, 1992, 2105)
// an odd number of k-groups: no gate/up form
#define QM_Q4_TILES_ODD(X)                      \
    X(4, 4, 1, 7, 2, 2, 1220, 1597, 1378, 1508)

// Above this k the tiles' 32-bit lane offsets do not reach (128 rows of x);
// the first tile has a form with 64-bit ones.
#define QM_Q4_GEMM_MAX_K32 (1 << 23)

#ifndef __HIP_DEVICE_COMPILE__
namespace qm_q4 {

struct Tile {
    const char* name;            // kernel name suffix
    int32_t mi, nj, wn, wk;
    int32_t gate_up;             // gate/up forms: 1 for an f16 x, 2 for a bf16 one
    int32_t alone[2], shared[2]; // [x is bf16]
};

#define QM_Q4_TILE_ROW(GU, MI, NJ, WN, WK, AF, SF, AB, SB) \
    {"m" #MI "n" #NJ "w" #WN "k" #WK, MI, NJ, WN, WK, GU, {AF, AB}, {SF, SB}},
#define QM_Q4_ROW_GATE_UP(MI, NJ, WN, WK, NST, OCC, ...) QM_Q4_TILE_ROW(3, MI, NJ, WN, WK, __VA_ARGS__)
#define QM_Q4_ROW_GATE_UP_BF16(MI, NJ, WN, WK, NST, OCC, ...) QM_Q4_TILE_ROW(2, MI, NJ, WN, WK, __VA_ARGS__)
#define QM_Q4_ROW_PLAIN(MI, NJ, WN, WK, NST, OCC, ...) QM_Q4_TILE_ROW(0, MI, NJ, WN, WK, __VA_ARGS__)
constexpr Tile kTiles[] = {QM_Q4_TILES_ONE_WAVE(QM_Q4_ROW_GATE_UP) QM_Q4_TILES_GATE_UP_BF16(QM_Q4_ROW_GATE_UP_BF16)
                           QM_Q4_TILES_PAIRED(QM_Q4_ROW_GATE_UP) QM_Q4_TILES_ODD(QM_Q4_ROW_PLAIN)};
#undef QM_Q4_ROW_PLAIN
#undef QM_Q4_ROW_GATE_UP_BF16
#undef QM_Q4_ROW_GATE_UP
#undef QM_Q4_TILE_ROW
constexpr int kBigTile = 0;      // the tile of the form with 64-bit lane offsets
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);

inline bool has_gate_up(const Tile& t, bool bf16) { return t.gate_up >> bf16 & 1; }

inline int64_t tile_grid(const Tile& t, int64_t m, int64_t n, bool gate_up) {
    const int64_t rows = 16 * t.mi, cols = 16 * t.nj * (gate_up && t.wn > 1 ? t.wn / 2 : t.wn);
    return (m + rows - 1) / rows * ((n + cols - 1) / cols);
}

// The tile a call takes: the one with the least estimated time, stages per
// workgroup times the measured time of a stage times the workgroups of the
// busiest CU.  It weighs what pulls both ways: a large tile dequantizes and
// loads less per product, a small one, or one that splits k over its waves,
// fills the CUs and shortens the chain of stages when there are few rows.
// Over the measured sizes the choice was within 1% of the best of these tiles
// on average (20% at worst).  From k = 512 on no size of a sweep over 14
// weight shapes and 1 to 8192 rows took longer than with the dequantize-to-LDS
// form these tiles replace; below, where a call is little more than its launch
// and epilogue, the best of them take 0.1 to 0.9 us more than that form did at
// some sizes (1200 x 32 x 2560 5.3 -> 6.1 us, 1 x 128 x 32 1.8 -> 2.3).
inline int pick_tile(int64_t m, int64_t k, int64_t n, bool bf16, bool gate_up, int num_cu) {
    int best = -1;
    int64_t best_ns = 0;
    for (int i = 0; i < kNumTiles; ++i) {
        const Tile& t = kTiles[i];
        if (gate_up && !has_gate_up(t, bf16)) continue;
        const int64_t groups = gate_up && t.wn == 1 ? t.wk / 2 : t.wk;
        const int64_t stages = ((k / 32 + 1) / 2 + groups - 1) / groups;
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
