// The host's choices of kernel, asked line by line on stdin:
//   rows S num_cu mode -> 16-row groups per block of the GQA prefill
#include <iostream>
#include <string>

#include "qm_gqa_plan.h"

int main() {
    std::string what;
    while (std::cin >> what) {
        if (what != "rows") return 1;
        int64_t S, cus, mode;
        if (!(std::cin >> S >> cus >> mode)) return 1;
        std::cout << qm_plan::gqp_row_groups(static_cast<int32_t>(S), static_cast<int32_t>(cus), mode) << "\n";
    }
    return 0;
}
