// Prints what the library's host side decides for a call, without a GPU: linked from the library's own objects, because
// these functions are not part of its exported surface.  Run by tests/test_host_rules.py.
//
//   host_checks split BATCH HEADS KV_HEADS HEAD_DIM KV_BF16 LENGTH SOURCE CAUSAL    attention_split: splits, keys per split
#include "nn/ops_internal.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>

namespace {

int split(char** arg) {
    int splits = 0, chunk = 0;
    auto at = [&](int i) { return std::atoll(arg[i]); };
    dl::detail::attention_split(at(0), at(1), at(2), at(3), at(4) != 0, at(5), at(6), at(7) != 0, splits, chunk);
    std::printf("%d %d\n", splits, chunk);
    return 0;
}

} // namespace

int main(int argc, char** argv) {
    if (argc == 10 && std::strcmp(argv[1], "split") == 0) return split(argv + 2);
    std::fprintf(stderr, "usage: host_checks split BATCH HEADS KV_HEADS HEAD_DIM KV_BF16 LENGTH SOURCE CAUSAL\n");
    return 2;
}
