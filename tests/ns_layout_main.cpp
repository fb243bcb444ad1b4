// Reads trees (a line each: the left child's item per item, -1: a leaf) and writes a line each: steps, seven top items, then item and
// following place of every place.
#include "../catboost_amd/csrc/ns_layout.h"

#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>

int main() {
    std::string line;
    cbamd::TNsTreeLayout layout;  // the same for all of them, as in an evaluator
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::vector<uint32_t> left;
        for (long item; in >> item;) {
            left.push_back(item < 0 ? cbamd::kNsNoItem : static_cast<uint32_t>(item));
        }
        cbamd::LayOutNsTree(left, &layout);
        std::printf("%u", layout.Steps);
        for (uint32_t item : layout.TopItems) {
            std::printf(" %d", static_cast<int>(item));
        }
        for (size_t at = 0; at < layout.Items.size(); ++at) {
            std::printf(" %u %u", layout.Items[at], layout.Next[at]);
        }
        std::printf("\n");
    }
    return 0;
}
