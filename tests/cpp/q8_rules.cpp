// Prints what the size rules of csrc/dsx_q8_0_rules.hpp say, one answer per line of stdin (CPU; driven by
// tests/test_q8_0_rules.py): "gemm hidden inter n_expert n_used tokens cus", "gate_up ..." and "dense hidden inter 0 0 tokens cus" ->
// columns per work item; "wide items_of_64 items_of_128 row_tiles slots 0 0" -> 1 where the items of 128 columns are taken.
#include <cstdio>
#include <cstring>

#include "../../deepstrix_amd/csrc/dsx_q8_0_rules.hpp"

int main() {
    char what[16];
    unsigned v[6];
    while (std::scanf("%15s %u %u %u %u %u %u", what, &v[0], &v[1], &v[2], &v[3], &v[4], &v[5]) == 7) {
        if (std::strcmp(what, "gemm") == 0) std::printf("%u\n", dsx::q8_gemm_columns({v[0], v[1], v[2], v[3]}, v[4], v[5]));
        else if (std::strcmp(what, "gate_up") == 0) {
            const dsx::Q8Shape s{v[0], v[1], v[2], v[3]};
            std::printf("%u\n", dsx::q8_gate_up_columns(s, v[4], dsx::q8_gemm_columns(s, v[4], v[5])));
        } else if (std::strcmp(what, "dense") == 0) std::printf("%u\n", dsx::q8_dense_columns(v[0], v[1], v[4], v[5]));
        else if (std::strcmp(what, "wide") == 0) std::printf("%d\n", (int)dsx::q8_takes_wide_items(v[0], v[1], v[2], v[3]));
        else return 1;
    }
    return 0;
}
