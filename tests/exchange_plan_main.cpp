// Prints the host tables of the exchange kernels for a model read from a file (test_exchange_kernel.py): all numbers
// as text, one array per line.
#include <cstdio>
#include <fstream>
#include <vector>

#include "../catboost_amd/csrc/exchange_plan.h"

int main(int argc, char** argv) {
    if (argc != 2 && argc != 3) {  // a second argument: only the steps of the rounds, and those with the busiest waves' groups
        return 2;
    }
    std::ifstream in(argv[1]);
    size_t treeCount = 0;
    uint32_t buckets = 0, maxDepth = 0, six = 0, tiled = 0;
    in >> treeCount >> buckets >> maxDepth >> six >> tiled;
    std::vector<uint32_t> columnOf(tiled ? buckets : 0);
    for (uint32_t& column : columnOf) {
        in >> column;
    }
    std::vector<cbamd::TExchangeTree> trees(treeCount);
    std::vector<std::vector<double>> leaves(treeCount);
    for (size_t t = 0; t < treeCount; ++t) {
        size_t levels = 0;
        in >> levels;
        for (size_t d = 0; d < levels; ++d) {
            cbamd::TExchangeLevel level;
            in >> level.Bucket >> level.Add >> level.Xor >> level.IsXor >> level.Lopsided;
            trees[t].Levels.push_back(level);
        }
        for (size_t i = 0; i < size_t(1) << levels; ++i) {
            double value = 0.0;
            in >> value;
            leaves[t].push_back(value);
        }
    }
    std::vector<cbamd::TExchangeColumn> columns;
    std::vector<uint32_t> pieces(tiled * cbamd::kExchangeTilePieces);
    for (uint32_t& piece : pieces) {
        in >> piece;
    }
    for (size_t c = 0; c < tiled * cbamd::kExchangeTileColumns; ++c) {
        cbamd::TExchangeColumn column;
        size_t values = 0;
        in >> column.Used >> column.OneHot >> column.RowByte >> values;
        column.Values.resize(values);
        for (uint32_t& v : column.Values) {
            in >> v;
        }
        if (column.Used && !column.OneHot) {
            cbamd::MakeExchangeGrid(six != 0, &column);
        }
        columns.push_back(column);
    }
    if (!in) {
        return 3;
    }
    cbamd::TExchangePlan plan;
    if (!cbamd::BuildExchangePlan(trees, buckets, maxDepth, six != 0, columnOf, &plan)) {
        std::printf("refused\n");
        return 0;
    }
    if (argc == 3) {
        std::printf("%u %u\n", plan.Rounds * cbamd::kExchangeRoundSteps, plan.CompareSteps);
        return 0;
    }
    std::printf("%u\n", plan.Rounds);
    for (const auto* table : {tiled ? &plan.FusedWaveTable : &plan.WaveTable, &plan.Records, &plan.ExtraRows}) {
        for (uint32_t v : *table) {
            std::printf("%u ", v);
        }
        std::printf("\n");
    }
    for (const cbamd::TExchangeLeafRow& row : plan.LeafRows) {
        for (uint32_t i = 0; i < 1u << maxDepth; ++i) {
            uint32_t leaf = 0;
            for (uint32_t bit = 0; bit < 8; ++bit) {
                const uint32_t level = row.Levels >> 4 * bit & 15;
                leaf |= level != cbamd::kExchangeNoLevel ? (i >> bit & 1) << level : 0;
            }
            std::printf("%.17g ", row.Tree != cbamd::kExchangeNoTree ? leaves[row.Tree][leaf] : 0.0);
        }
    }
    std::printf("\n");
    std::vector<uint32_t> table, oneHot;
    if (tiled != 0 && cbamd::BuildExchangeTiles(columns, pieces, six != 0, &table, &oneHot)) {
        for (const auto* t : {&table, &oneHot}) {
            for (uint32_t v : *t) {
                std::printf("%u ", v);
            }
            std::printf("\n");
        }
    }
    return 0;
}
