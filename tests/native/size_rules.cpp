// Test harness: the library's rules on sizes (gf_internal.h), evaluated on
// the CPU.  usage: size_rules <rule> <numbers>...
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../garfield_amd/csrc/gf_internal.h"

int main(int argc, char** argv) {
    auto u = [&](int i) { return i < argc ? uint32_t(std::strtoul(argv[i], nullptr, 10)) : 0u; };
    const char* rule = argc > 1 ? argv[1] : "";
    if (!std::strcmp(rule, "first_pairs"))
        std::printf("%zu\n", gf::bf_first_pairs(u(2), u(3), u(4), u(5), u(6), u(7)));
    else if (!std::strcmp(rule, "float_item_tiles"))
        std::printf("%u\n", gf::bf_float_item_tiles(u(2) != 0, u(3), u(4), u(5), u(6)));
    else if (!std::strcmp(rule, "pad_records_fit"))
        std::printf("%d\n", int(gf::bf_pad_records_fit(std::strtoull(argv[2], nullptr, 10), std::strtoull(argv[3], nullptr, 10))));
    else
        return 2;
    return 0;
}
