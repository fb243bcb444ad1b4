// Host tables of the exchange kernels (gen_eval_exchange_kernel.py): one-dimensional oblivious models of depth <= 8 whose
// bins of 256 documents fit the registers of a workgroup's sixteen waves (64 buckets each).
//
// Every wave compares the levels that look at its own buckets and packs their results, one bit per document, into dwords:
// a *group* is MaxDepth levels (8 or 6), whose bits stand in different positions of a byte per document. The dwords meet in
// LDS slots; the wave that sums a tree picks the tree's bits out of the dwords of its levels' groups, the bit at position p
// from the dword that the tree's row names for p. Two levels must therefore stand in different positions if they belong to one tree or to
// one group: a proper edge colouring of the multigraph trees x groups (an edge is a level), whose degrees are at most
// MaxDepth, and such a graph has one with MaxDepth colours (Koenig).
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

namespace cbamd {

constexpr uint32_t kExchangeWaves = 16;          // waves per workgroup, one workgroup per CU
constexpr uint32_t kExchangeWaveBuckets = 64;    // bins registers per wave
constexpr uint32_t kExchangeRoundSteps = 4;      // trees that a wave sums between two barriers
constexpr uint32_t kExchangeSlots = 224;         // LDS slots of 256 bytes for the groups' dwords
constexpr uint32_t kExchangeGroupDwords = 16;    // a group's row: per place (register | xor byte << 8, added bytes); the first dword
                                                 // also slot * 256 << 16, the third one the flags
constexpr uint32_t kExchangeXorFlag = 0x80000000u;   // a level of the group xors
constexpr uint32_t kExchangeMoreFlag = 0x40000000u;  // another group in this step, from the wave's row of extra ones
constexpr uint32_t kExchangeSkipFlag = 0x20000000u;  // no group in this step
constexpr uint32_t kExchangeEarlyRows = 3;       // rows of the groups before the first step that are fetched together
constexpr uint32_t kExchangeTreeDwords = 8;      // a tree's row: per place the byte offset of the slot that holds its level's group
// per round and wave: four group rows, four tree rows
constexpr uint32_t kExchangeRecordDwords = kExchangeRoundSteps * (kExchangeGroupDwords + kExchangeTreeDwords);
constexpr uint32_t kExchangeWaveDwords = 80;     // per wave: 64 bucket offsets in bytes, offset of its first extra group row in
                                                 // bytes, how many of those come before the first step

// Fused kernels: tiles of sixteen pieces of four neighbouring columns, the bins of a tile's 64 columns in a buffer in LDS
constexpr uint32_t kExchangeTiles = 16;
constexpr uint32_t kExchangeTilePieces = 16, kExchangePieceColumns = 4;
constexpr uint32_t kExchangeTileColumns = kExchangeTilePieces * kExchangePieceColumns;
constexpr uint32_t kExchangeColumnBytes = 260;   // of the buffer
constexpr uint32_t kExchangeNoColumn = ~0u;

struct TExchangeLevel {
    uint32_t Bucket = 0;
    uint32_t Add = 0;       // byte added to the (xored) bin: the level's result is the carry into bit 7
    uint32_t Xor = 0;       // seven bits
    bool IsXor = false;
    float Lopsided = 0.0f;  // 0: splits the documents evenly
};

struct TExchangeTree {
    std::vector<TExchangeLevel> Levels;
};

// Where a row of 1 << maxDepth leaf values comes from
constexpr uint32_t kExchangeNoTree = ~0u, kExchangeNoLevel = 15;
struct TExchangeLeafRow {
    uint32_t Tree = kExchangeNoTree;  // none: a row of zeros
    uint32_t Levels = ~0u;            // four bits per bit of the row's index: the level of the model whose result that bit is, or
                                      // kExchangeNoLevel: the bit is another group's, the values are the same for either
};

struct TExchangePlan {
    uint32_t Rounds = 0;
    uint32_t CompareSteps = 0;        // the rounds' steps and what the wave with the most groups of a round compares beyond them: a
                                      // bucket's levels are all its wave's, so a model that looks at few buckets most takes longer
    std::vector<uint32_t> WaveTable;  // [wave][kExchangeWaveDwords]
    std::vector<uint32_t> FusedWaveTable;  // the same with the registers' columns in the buffer for the buckets' offsets
    std::vector<uint32_t> Records;    // [round + 1][wave][kExchangeRecordDwords]: rows are fetched ahead
    std::vector<uint32_t> ExtraRows;  // [wave][its extra groups][kExchangeGroupDwords], and kExchangeEarlyRows spare ones
    std::vector<TExchangeLeafRow> LeafRows;  // [round + 1][wave][step]
};

// maxDepth: 6 or 8, at least the deepest tree's. six: all bins are at most 63, and the levels of even places in a group
// have their results in bit 6. Tree t of pair p = t / 2 is summed by wave p % 16, the last tree of an odd number by wave 0
// behind its others: the sums and their order are the pair-tile kernel's. columnOf: empty, or per bucket tile * 64 + column for
// a fused kernel (registers 4 t .. 4 t + 3 of a wave then hold buckets of tile t). Returns false if the model does not fit (too many
// buckets, or groups that no slot is left for).
bool BuildExchangePlan(const std::vector<TExchangeTree>& trees, uint32_t bucketCount, uint32_t maxDepth, bool six,
                       const std::vector<uint32_t>& columnOf, TExchangePlan* plan);

// A column of a tile of the fused kernels
struct TExchangeColumn {
    bool Used = false, OneHot = false;
    uint32_t RowByte = 0;                // one-hot: where it is in a row
    std::vector<uint32_t> Values;        // bits of the sorted borders, or hashes
    float Scale = 0.0f, Bias = 0.0f;     // the borders' grid (MakeExchangeGrid), its search steps and the borders below each of its cells
    uint32_t Steps = 0;
    std::vector<uint32_t> Start;
};

constexpr uint32_t kExchangeMaxSteps = 4;

// cells of a column's grid: what its 768 bytes of tables have room for beside 64 or 128 borders
constexpr uint32_t ExchangeGridCells(bool six) {
    return six ? 512 : 256;
}

// The grid over a column's sorted borders: a value's cell is fma(clamp(fma(value, Scale, Bias), 0, 1), cells - 1, 2^23) - 2^23, in fp32,
// which rises with the value; so the borders of lower cells are below the value and those of higher cells are not.
void MakeExchangeGrid(bool six, TExchangeColumn* column);

// Tables of the fused kernels (gen_eval_exchange_kernel.py): infos and images of the tiles, and the one-hot columns' records.
// columns: [tile][64]; pieces: [tile][16] byte offsets in a row. Returns false if a column's borders or steps do not fit.
bool BuildExchangeTiles(const std::vector<TExchangeColumn>& columns, const std::vector<uint32_t>& pieces, bool six,
                        std::vector<uint32_t>* table, std::vector<uint32_t>* oneHot);

}  // namespace cbamd
