// The host's choices of kernel, asked line by line on stdin:
//   rows S num_cu mode            -> 16-row groups per block of the GQA prefill
//   tile m k n bf16 gate_up num_cu -> the Q4 GEMM's tile
//   built t                       -> tile t's name and gate/up forms (1 f16, 2 bf16); "-" past the last
#include <iostream>
#include <string>

#include "qm_gqa_plan.h"
#include "qm_q4_tiles.h"

int main() {
    std::string what;
    while (std::cin >> what) {
        int64_t a, b, c, d, e, f;
        if (what == "rows" && std::cin >> a >> b >> c) {
            std::cout << qm_plan::gqp_row_groups(static_cast<int32_t>(a), static_cast<int32_t>(b), c) << "\n";
        } else if (what == "tile" && std::cin >> a >> b >> c >> d >> e >> f) {
            std::cout << qm_q4::kTiles[qm_q4::pick_tile(a, b, c, d != 0, e != 0, static_cast<int>(f))].name << "\n";
        } else if (what == "built" && std::cin >> a) {
            if (a < qm_q4::kNumTiles) std::cout << qm_q4::kTiles[a].name << " " << qm_q4::kTiles[a].gate_up << "\n";
            else std::cout << "-\n";
        } else {
            return 1;
        }
    }
    return 0;
}
