// Device code of the HIP evaluator (gfx950, wave64).
//
// Quantized layout ("bins"): documents are grouped in blocks of 256; inside a block one wave
// lane owns the four documents {lane, lane + 64, lane + 128, lane + 192} and keeps their bins of
// one bucket in one dword, so
//     bins[((block * buckets + bucket) * 64 + lane) * 4 + j]  is the bin of document
//     block * 256 + j * 64 + lane.
// A wave reads or writes the 256 bytes of one (block, bucket) pair with a single coalesced dword
// access per lane, and per-document results (doc = base + j * 64 + lane) are coalesced as well.
// Bin values are those of the reference's BinarizeFeatures (cpu/quantization.h:333-529):
// float bucket -> number of borders strictly below the value, one-hot bucket -> 1 + index of the
// matching value (0 when none).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace cbamd::dev {

constexpr int kDocsPerBlock = 256;
constexpr int kWave = 64;
constexpr int kBucketFlagNanToInf = 1;  // HasNans && NanValueTreatment == AsTrue
constexpr int kBucketFlagOneHot = 2;
constexpr uint32_t kXcdCount = 8;       // accelerator dies of an MI355X, each with its own L2
constexpr int kBucketTile = 16;         // buckets binarized per workgroup (small: ~20 KB of LDS, 7 workgroups per CU)
constexpr int kMaxBucketValues = 256;   // 254 values, padded

constexpr int kBucketFlagCtr = 4;        // bucket of a CTR feature: filled by CtrBinarizeKernel

struct TBinarizeTables {
    uint32_t BucketCount;          // buckets the binarize kernels fill: float and one-hot features
    uint32_t BucketPitch;          // buckets per document block in `bins` (those and the CTR buckets)
    const uint32_t* BucketSrc;     // source column of the bucket in the chosen layout
    const uint32_t* BucketOffset;  // [BucketCount + 1] offsets into Values
    const uint32_t* BucketFlags;
    const uint32_t* Values;        // float borders (sorted ascending) or one-hot values, as bits
    // float buckets, row binarize kernel: a uniform grid of kLutCells cells over the bucket's borders
    // gives the search a start and a short window instead of the whole border array
    const uint4* Grid;             // per bucket: lowest border, cells per unit (both fp32 bits), search steps, 0
    const uint32_t* Lut;           // per bucket kLutCells bytes: first border the search looks at, per cell
};

struct TTreeTables {
    const uint32_t* Splits;       // per tree split / node: bucket | xorMask << 16 | splitIdx << 24
    const uint32_t* TreeStart;    // first split (oblivious) or first node (non-symmetric) of a tree
    const uint32_t* TreeSize;     // depth (oblivious) or node count (non-symmetric)
    const uint32_t* FirstLeaf;    // index of the tree's first value in Leaves
    const uint32_t* StepNodes;    // non-symmetric: left diff | right diff << 16
    const uint32_t* NodeToLeaf;   // non-symmetric: value index of a terminal node
    const double* Leaves;
    const double* Bias;
    double Scale;
    int Dim;
};

// number of sorted borders strictly below v; `borders` holds 1 << LOG2P entries, the real ones
// first and +inf after them
template <int LOG2P>
__device__ __forceinline__ uint32_t CountBelow(const uint32_t* borders, float v) {
    const uint32_t* p = borders;
#pragma unroll
    for (uint32_t step = 1u << (LOG2P - 1); step >= 1; step >>= 1) {
        const float b = __uint_as_float(p[step - 1]);
        p = (b < v) ? p + step : p;
    }
    return static_cast<uint32_t>(p - borders);
}

constexpr int kLutCells = 256;

// Cell of a value in a bucket's grid: (v - lo) * scale, truncated, negative and NaN to 0, at most
// kLutCells - 1. Subtract and multiply are separate roundings, and the host computes the borders'
// cells with the very same operations (GridCell in hip_evaluator.hip), so cell(b) <= cell(v)
// whenever b <= v: every border in a lower cell is below v, every border in a higher cell above.
__device__ __forceinline__ uint32_t GridCell(float v, float lo, float scale) {
    const float t = __fmul_rn(__fsub_rn(v, lo), scale);
    uint32_t c;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(c) : "v"(t));  // saturating, NaN -> 0
    return min(c, static_cast<uint32_t>(kLutCells - 1));
}

// Number of borders strictly below v, searching only the window the value's cell points at:
// `lut[cell]` borders are known to be below v, the next 2 * topStep - 1 entries hold every border of
// the cell (and then higher ones or the +inf padding, which never count).
__device__ __forceinline__ uint32_t CountBelowInCell(const uint32_t* borders, const uint8_t* lut, float lo, float scale,
                                                     uint32_t topStep, float v) {
    const uint32_t* p = borders + lut[GridCell(v, lo, scale)];
    for (uint32_t step = topStep; step >= 1; step >>= 1) {
        const float b = __uint_as_float(p[step - 1]);
        p = (b < v) ? p + step : p;
    }
    return static_cast<uint32_t>(p - borders);
}

__device__ __forceinline__ uint32_t OneHotBin(const uint32_t* values, uint32_t count, uint32_t v) {
    uint32_t bin = 0;
    for (uint32_t i = 0; i < count; ++i) {
        bin |= (values[i] == v) ? (i + 1) : 0u;
    }
    return bin;
}

// The borders and search tables of the buckets b0 .. b0 + nb of a binarize workgroup (256 threads) into LDS, empty
// slots as +inf. All loads of a step are issued before the first is waited for: with a few workgroups per CU this
// prologue, two dependent loads for each of a thread's sixteen values, is not hidden otherwise: the whole
// call is 5 % shorter for 4M documents of 300 features with 254 borders and 500 non-symmetric trees, 2.5 % for 100 003
// documents of 60 features and 500 trees of three dimensions, 2 % for a CTR model of 1M documents.
template <int LOG2P>
__device__ __forceinline__ void LoadBucketTables(const TBinarizeTables& tab, uint32_t b0, uint32_t nb, uint32_t tid,
                                                 uint32_t* sValues, uint32_t* sLut) {
    constexpr uint32_t kSlots = 1u << LOG2P;
    constexpr int kPerThread = kBucketTile * kSlots / 256, kLutPerThread = kBucketTile * (kLutCells / 4) / 256;
    const uint32_t lutDwords = nb * (kLutCells / 4);
    uint32_t lut[kLutPerThread], begin[kPerThread], end[kPerThread], value[kPerThread];
#pragma unroll
    for (int n = 0; n < kPerThread; ++n) {
        const uint32_t bucket = b0 + min((tid + n * 256) >> LOG2P, nb - 1);
        begin[n] = tab.BucketOffset[bucket];
        end[n] = tab.BucketOffset[bucket + 1];
    }
#pragma unroll
    for (int n = 0; n < kLutPerThread; ++n) {
        lut[n] = tab.Lut[static_cast<size_t>(b0) * (kLutCells / 4) + min(tid + n * 256, lutDwords - 1)];
    }
#pragma unroll
    for (int n = 0; n < kPerThread; ++n) {
        const uint32_t k = (tid + n * 256) & (kSlots - 1);
        value[n] = 0x7f800000u;  // +inf
        if (k < end[n] - begin[n]) {
            value[n] = tab.Values[begin[n] + k];
        }
    }
#pragma unroll
    for (int n = 0; n < kLutPerThread; ++n) {
        sLut[tid + n * 256] = lut[n];
    }
#pragma unroll
    for (int n = 0; n < kPerThread; ++n) {
        sValues[tid + n * 256] = value[n];
    }
}

constexpr int kTilePitch = kDocsPerBlock + 1;  // dwords per bucket row of the transposed tile

// Row-major input: floats[doc * stride + column]; hashed categorical values either bit-cast in
// the same row (CATS_MATRIX == false) or in cats[doc * catStride + column].
// One workgroup owns kBucketTile buckets and walks `blocksPerGroup` consecutive 256-document
// blocks: the bucket values stay in LDS (1 << LOG2P slots per bucket, every bucket of the model
// has fewer values than that), each block's 256 x kBucketTile feature tile is fetched with row-contiguous
// loads into registers one block ahead, transposed through a padded LDS tile and binarized by a
// branch-free binary search; a wave writes the 256 bytes of one (block, bucket) pair at once.
// Rows past the last document are read as the last document (their bins are never used).
// grid = ceil(doc blocks / blocksPerGroup) * ceil(buckets / kBucketTile), block = 256 threads,
// dynamic LDS = (kBucketTile << LOG2P) * 4 + kBucketTile * kLutCells + kBucketTile * kTilePitch * 4 bytes.
template <int LOG2P, bool CATS_MATRIX>
__global__ __launch_bounds__(256) void BinarizeRowsKernel(const float* __restrict__ floats, uint32_t stride,
                                                          const int32_t* __restrict__ cats, uint32_t catStride,
                                                          uint32_t docCount, TBinarizeTables tab,
                                                          uint32_t blocksPerGroup, uint32_t* __restrict__ bins) {
    constexpr uint32_t kSlots = 1u << LOG2P;
    constexpr int kRowsPerPass = 256 / kBucketTile;        // rows per pass of 256 threads
    constexpr int kPasses = kDocsPerBlock / kRowsPerPass;  // values per thread and block
    extern __shared__ uint32_t sBinarize[];
    uint32_t* sValues = sBinarize;                           // [kBucketTile][kSlots]
    uint32_t* sLut = sBinarize + kBucketTile * kSlots;       // [kBucketTile][kLutCells / 4]
    uint32_t* sTile = sLut + kBucketTile * (kLutCells / 4);  // [kBucketTile][kTilePitch]

    const uint32_t tid = threadIdx.x;
    const uint32_t tileCount = (tab.BucketCount + kBucketTile - 1) / kBucketTile;
    // Workgroups go round-robin to the 8 XCDs, each with an L2 of its own. The bucket tiles of one
    // document group share cache lines (a row piece of 128 bytes is not line aligned), so they are
    // given to workgroups of the same XCD that start one after the other: XCD x owns a contiguous
    // range of the work list.
    const uint32_t perXcd = gridDim.x / kXcdCount, extra = gridDim.x % kXcdCount;
    const uint32_t xcd = blockIdx.x % kXcdCount;
    const uint32_t work = xcd * perXcd + min(xcd, extra) + blockIdx.x / kXcdCount;
    const uint32_t b0 = (work % tileCount) * kBucketTile;
    const uint32_t nb = min(static_cast<uint32_t>(kBucketTile), tab.BucketCount - b0);
    const uint32_t blockCount = (docCount + kDocsPerBlock - 1) / kDocsPerBlock;
    const uint32_t blockBegin = (work / tileCount) * blocksPerGroup;
    const uint32_t blockEnd = min(blockBegin + blocksPerGroup, blockCount);

    LoadBucketTables<LOG2P>(tab, b0, nb, tid, sValues, sLut);

    // role of this thread while loading: bucket `myB` of rows myRow0, myRow0 + 8, ...; threads of
    // buckets past the end of the model re-read the last bucket and their values are ignored
    const uint32_t myB = tid % kBucketTile;
    const uint32_t myRow0 = tid / kBucketTile;
    const uint32_t mySrcBucket = b0 + min(myB, nb - 1);
    const uint32_t mySrc = tab.BucketSrc[mySrcBucket];
    const uint32_t* myBase = reinterpret_cast<const uint32_t*>(floats);
    uint32_t myStride = stride;
    if (CATS_MATRIX && (tab.BucketFlags[mySrcBucket] & kBucketFlagOneHot) != 0) {
        myBase = reinterpret_cast<const uint32_t*>(cats);
        myStride = catStride;
    }
    uint32_t* myTileSlot = sTile + myB * kTilePitch + myRow0;

    uint32_t regs[kPasses];
#define CBAMD_LOAD_BLOCK(blockIndex)                                                                   \
    do {                                                                                               \
        const uint32_t firstDoc = (blockIndex) * kDocsPerBlock;                                        \
        if (firstDoc + kDocsPerBlock <= docCount) {                                                    \
            const uint32_t* rowPtr = myBase + static_cast<size_t>(firstDoc + myRow0) * myStride + mySrc; \
            _Pragma("unroll") for (int i = 0; i < kPasses; ++i) {                                      \
                regs[i] = rowPtr[static_cast<size_t>(i) * kRowsPerPass * myStride];                    \
            }                                                                                          \
        } else {                                                                                       \
            _Pragma("unroll") for (int i = 0; i < kPasses; ++i) {                                      \
                const uint32_t doc = min(firstDoc + myRow0 + i * kRowsPerPass, docCount - 1);          \
                regs[i] = myBase[static_cast<size_t>(doc) * myStride + mySrc];                         \
            }                                                                                          \
        }                                                                                              \
    } while (0)

    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    // the buckets this wave binarizes in every block (wave, wave + 4, ...) and their grids
    constexpr int kBucketsPerWave = kBucketTile / (256 / kWave);
    uint32_t myFlags[kBucketsPerWave], myTopStep[kBucketsPerWave];
    float myLo[kBucketsPerWave], myScale[kBucketsPerWave];
#pragma unroll
    for (int k = 0; k < kBucketsPerWave; ++k) {
        const uint32_t bucket = b0 + min(wave + k * (256 / kWave), nb - 1);
        const uint4 grid = tab.Grid[bucket];
        myFlags[k] = __builtin_amdgcn_readfirstlane(tab.BucketFlags[bucket]);
        myLo[k] = __uint_as_float(__builtin_amdgcn_readfirstlane(grid.x));
        myScale[k] = __uint_as_float(__builtin_amdgcn_readfirstlane(grid.y));
        const uint32_t steps = __builtin_amdgcn_readfirstlane(grid.z);
        myTopStep[k] = steps ? 1u << (steps - 1) : 0u;
    }
    if (blockBegin < blockEnd) {
        CBAMD_LOAD_BLOCK(blockBegin);
    }
    for (uint32_t block = blockBegin; block < blockEnd; ++block) {
        __syncthreads();  // the previous block's tile has been consumed (and sValues is complete)
#pragma unroll
        for (int i = 0; i < kPasses; ++i) {
            myTileSlot[i * kRowsPerPass] = regs[i];
        }
        __syncthreads();
        if (block + 1 < blockEnd) {
            CBAMD_LOAD_BLOCK(block + 1);  // in flight while this block is binarized
        }
        // this lane's dword of the block's first bucket of the tile; bucket bb sits bb * 256 bytes further
        uint32_t* blockBins = bins + (static_cast<size_t>(block) * tab.BucketPitch + b0) * kWave + lane;
#pragma unroll
        for (int k = 0; k < kBucketsPerWave; ++k) {
            const uint32_t bb = wave + k * (256 / kWave);
            if (bb >= nb) {
                break;
            }
            const uint32_t* values = sValues + bb * kSlots;
            const uint32_t* column = sTile + bb * kTilePitch + lane;
            uint32_t packed = 0;
            if (myFlags[k] & kBucketFlagOneHot) {
                const uint32_t count = tab.BucketOffset[b0 + bb + 1] - tab.BucketOffset[b0 + bb];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    packed |= OneHotBin(values, count, column[j * kWave]) << (8 * j);
                }
            } else {
                // the lane's four documents go through the search side by side: one pass of the loop
                // control and one LDS round trip per step for all four (CountBelowInCell, four at once)
                const uint8_t* lut = reinterpret_cast<const uint8_t*>(sLut + bb * (kLutCells / 4));
                float v[4];
                uint32_t below[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v[j] = __uint_as_float(column[j * kWave]);
                }
                if (myFlags[k] & kBucketFlagNanToInf) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        v[j] = isnan(v[j]) ? __uint_as_float(0x7f800000u) : v[j];
                    }
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    below[j] = static_cast<uint32_t>(lut[GridCell(v[j], myLo[k], myScale[k])]) * 4;  // byte offsets
                }
                const uint8_t* valueBytes = reinterpret_cast<const uint8_t*>(values);
                for (uint32_t step4 = __builtin_amdgcn_readfirstlane(myTopStep[k]) * 4; step4 >= 4; step4 >>= 1) {
                    const uint8_t* probe = valueBytes + step4 - 4;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float b = *reinterpret_cast<const float*>(probe + below[j]);
                        below[j] += (b < v[j]) ? step4 : 0u;
                    }
                }
                packed = (below[0] >> 2) | (below[1] << 6) | (below[2] << 14) | (below[3] << 22);
            }
            blockBins[bb * kWave] = packed;
        }
    }
#undef CBAMD_LOAD_BLOCK
}

// Column-major input: floats[column * stride + doc] (categorical hashes bit-cast in their column). The work of a
// workgroup is that of BinarizeRowsKernel - kBucketTile buckets, their borders and search tables in LDS,
// `blocksPerGroup` consecutive 256-document blocks, every wave a bucket at a time for the block's 256 documents,
// a lane its four documents side by side - without the tile: a lane's values are neighbours of the other lanes' in
// the column, so they are loaded straight into registers, all buckets of the wave's turn before the first search.
// grid = ceil(doc blocks / blocksPerGroup) * ceil(buckets / kBucketTile), block = 256 threads,
// dynamic LDS = (kBucketTile << LOG2P) * 4 + kBucketTile * kLutCells bytes.
template <int LOG2P>
__global__ __launch_bounds__(256) void BinarizeColumnsKernel(const float* __restrict__ floats, size_t stride,
                                                             uint32_t docCount, TBinarizeTables tab,
                                                             uint32_t blocksPerGroup, uint32_t* __restrict__ bins) {
    constexpr uint32_t kSlots = 1u << LOG2P;
    extern __shared__ uint32_t sBinarize[];
    uint32_t* sValues = sBinarize;                      // [kBucketTile][kSlots]
    uint32_t* sLut = sBinarize + kBucketTile * kSlots;  // [kBucketTile][kLutCells / 4]
    const uint32_t tid = threadIdx.x;
    const uint32_t tileCount = (tab.BucketCount + kBucketTile - 1) / kBucketTile;
    const uint32_t b0 = (blockIdx.x % tileCount) * kBucketTile;
    const uint32_t nb = min(static_cast<uint32_t>(kBucketTile), tab.BucketCount - b0);
    const uint32_t blockCount = (docCount + kDocsPerBlock - 1) / kDocsPerBlock;
    const uint32_t blockBegin = (blockIdx.x / tileCount) * blocksPerGroup;
    const uint32_t blockEnd = min(blockBegin + blocksPerGroup, blockCount);
    LoadBucketTables<LOG2P>(tab, b0, nb, tid, sValues, sLut);
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    constexpr int kBucketsPerWave = kBucketTile / (256 / kWave);
    uint32_t myFlags[kBucketsPerWave], myTopStep[kBucketsPerWave], myCount[kBucketsPerWave];
    float myLo[kBucketsPerWave], myScale[kBucketsPerWave];
    const uint32_t* myColumn[kBucketsPerWave];
#pragma unroll
    for (int k = 0; k < kBucketsPerWave; ++k) {
        const uint32_t bucket = b0 + min(wave + k * (256 / kWave), nb - 1);
        const uint4 grid = tab.Grid[bucket];
        myFlags[k] = __builtin_amdgcn_readfirstlane(tab.BucketFlags[bucket]);
        myLo[k] = __uint_as_float(__builtin_amdgcn_readfirstlane(grid.x));
        myScale[k] = __uint_as_float(__builtin_amdgcn_readfirstlane(grid.y));
        const uint32_t steps = __builtin_amdgcn_readfirstlane(grid.z);
        myTopStep[k] = steps ? 1u << (steps - 1) : 0u;
        myCount[k] = __builtin_amdgcn_readfirstlane(tab.BucketOffset[bucket + 1] - tab.BucketOffset[bucket]);
        myColumn[k] = reinterpret_cast<const uint32_t*>(floats) +
                      static_cast<size_t>(__builtin_amdgcn_readfirstlane(tab.BucketSrc[bucket])) * stride;
    }
    __syncthreads();  // the tables are in LDS
    for (uint32_t block = blockBegin; block < blockEnd; ++block) {
        // documents past the last one are read as the last one (their bins are never used)
        uint32_t doc[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            doc[j] = min(block * kDocsPerBlock + j * kWave + lane, docCount - 1);
        }
        uint32_t raw[kBucketsPerWave][4];
#pragma unroll
        for (int k = 0; k < kBucketsPerWave; ++k) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                raw[k][j] = myColumn[k][doc[j]];
            }
        }
        uint32_t* blockBins = bins + (static_cast<size_t>(block) * tab.BucketPitch + b0) * kWave + lane;
#pragma unroll
        for (int k = 0; k < kBucketsPerWave; ++k) {
            const uint32_t bb = wave + k * (256 / kWave);
            if (bb >= nb) {
                break;
            }
            const uint32_t* values = sValues + bb * kSlots;
            uint32_t packed = 0;
            if (myFlags[k] & kBucketFlagOneHot) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    packed |= OneHotBin(values, myCount[k], raw[k][j]) << (8 * j);
                }
            } else {
                const uint8_t* lut = reinterpret_cast<const uint8_t*>(sLut + bb * (kLutCells / 4));
                float v[4];
                uint32_t below[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v[j] = __uint_as_float(raw[k][j]);
                }
                if (myFlags[k] & kBucketFlagNanToInf) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        v[j] = isnan(v[j]) ? __uint_as_float(0x7f800000u) : v[j];
                    }
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    below[j] = static_cast<uint32_t>(lut[GridCell(v[j], myLo[k], myScale[k])]) * 4;  // byte offsets
                }
                const uint8_t* valueBytes = reinterpret_cast<const uint8_t*>(values);
                for (uint32_t step4 = __builtin_amdgcn_readfirstlane(myTopStep[k]) * 4; step4 >= 4; step4 >>= 1) {
                    const uint8_t* probe = valueBytes + step4 - 4;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float b = *reinterpret_cast<const float*>(probe + below[j]);
                        below[j] += (b < v[j]) ? step4 : 0u;
                    }
                }
                packed = (below[0] >> 2) | (below[1] << 6) | (below[2] << 14) | (below[3] << 22);
            }
            blockBins[bb * kWave] = packed;
        }
    }
}

// ---- CTR (target statistics) features -------------------------------------------------------
// What TStaticCtrProvider::CalcCtrs (catboost/libs/model/static_ctr_provider.cpp:14-131) and the
// binarization of its results (cpu/quantization.h:304-325) do per block, done per document here. A CTR's value
// depends on the document only through the row of the learned statistics that the hash of its projection finds, so
// the host computes the bins of every row once, when the tables are uploaded (BuildCtrTables in hip_evaluator.hip):
// all CTR features of one projection share one hash table whose entries hold the hash and, a byte each, the bins of
// the projection's buckets. An empty entry holds the bins of a hash that no table knows.
struct TCtrGroupDev {             // the CTR features of one projection
    uint32_t ItemBegin, ItemEnd;  // the projection: entries of TCtrTablesDev::Items
    uint32_t FirstPiece;          // the group's table in TCtrTablesDev::Table, in pieces of 16 bytes
    uint32_t HashMask;            // entries of the table - 1
    uint32_t EntryPieces;         // pieces of an entry: hash low, hash high, then the bins
    uint32_t FirstBucket;         // of the group's list in TCtrTablesDev::Buckets
    uint32_t BucketCount;
    uint32_t Unused;
};

constexpr uint32_t kCtrItemCat = 0;       // hashed categorical value of column SrcFlat / SrcSplit
constexpr uint32_t kCtrItemBinGe = 1;     // float split: bin of bucket SrcFlat >= Value
constexpr uint32_t kCtrItemBinEq = 2;     // one-hot split: bin of bucket SrcFlat == Value

struct TCtrItemDev {
    uint32_t Kind, SrcFlat, SrcSplit, Value;  // a categorical item keeps its row of the staged tile in Value
};

struct TCtrTablesDev {
    const TCtrGroupDev* Groups;
    const TCtrItemDev* Items;
    const uint4* Table;
    const uint32_t* Buckets;  // per byte of an entry's bins the bucket it goes to
    // the categorical columns the projections read, as flat and as categorical feature indexes
    const uint32_t* CatColumnsFlat;
    const uint32_t* CatColumnsSplit;
    uint32_t CatColumnCount;
    uint32_t GroupCount;
};

// hashed categorical values of a batch: Base[doc * DocStride + column * ColumnStride]
struct TCatSource {
    const uint32_t* Base;
    size_t DocStride, ColumnStride;
    uint32_t SplitColumns;  // columns are categorical feature indexes (not flat feature indexes)
};

// CalcHash(a, b) = magic * (a + magic * b), catboost/libs/model/hash.h:11-14, as magic * a + magic^2 * b
constexpr uint64_t kCtrMagic = 0x4906ba494954cb65ull;
constexpr uint64_t kCtrMagicSquared = kCtrMagic * kCtrMagic;

// b: a hashed categorical value, sign-extended
__device__ __forceinline__ uint64_t CtrHashOfCat(uint32_t v) {
    constexpr uint32_t kLow = static_cast<uint32_t>(kCtrMagicSquared), kHigh = static_cast<uint32_t>(kCtrMagicSquared >> 32);
    const uint64_t product = static_cast<uint64_t>(v) * kLow;
    const uint32_t high = static_cast<uint32_t>(product >> 32) + v * kHigh - (static_cast<int32_t>(v) < 0 ? kLow : 0u);
    return (static_cast<uint64_t>(high) << 32) | static_cast<uint32_t>(product);
}

// The bins of a lane's four documents ({lane, lane + 64, lane + 128, lane + 192} of the block) in the buckets of CTR
// features. What bounds it is the gathers of table entries (a line of L2 each for tables beyond the L1): one 16-byte
// read finds and answers a lookup of up to eight buckets, where a table per CTR feature, its rows and a division and a
// count of borders per feature took five times as long (1M documents, 16 categorical columns, 24 projections with 96 CTR
// features: 620 us then; 87 to 97 now, three batches in turn; with tables half full instead of a quarter the call takes 252
// us instead of 215).
// grid = (document blocks, shares of the groups), 4 waves per workgroup, each wave a run of the share's groups.
// TILE: the block's hashed categorical values are staged once per workgroup into LDS ([column][document]); without
// it (more than kCtrMaxTileColumns columns) they are read from the batch where a projection needs them.
constexpr uint32_t kCtrMaxTileColumns = 60;
constexpr uint32_t kCtrTilePitch = kDocsPerBlock + 4;  // 16 columns * 4 documents, stored at once, fall on 64 banks

template <bool TILE>
__global__ __launch_bounds__(256) void CtrBinarizeKernel(TCatSource cats, uint32_t docCount, TCtrTablesDev ctr,
                                                         uint32_t bucketPitch, uint32_t groupsPerShare,
                                                         uint32_t* __restrict__ bins) {
    extern __shared__ uint32_t sCats[];  // [CatColumnCount][kCtrTilePitch]
    const uint32_t block = blockIdx.x, tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t firstDoc = block * kDocsPerBlock;
    // documents past the last one are read as the last one (their bins are never used)
    if (TILE) {
        const uint32_t columns = ctr.CatColumnCount;
        const uint32_t* columnList = cats.SplitColumns ? ctr.CatColumnsSplit : ctr.CatColumnsFlat;
        if (cats.ColumnStride == 1) {  // sixteen columns of a row side by side
            for (uint32_t c = tid % 16; c < columns; c += 16) {
                const uint32_t* column = cats.Base + columnList[c];
#pragma unroll 4
                for (uint32_t d = tid / 16; d < kDocsPerBlock; d += 16) {
                    sCats[c * kCtrTilePitch + d] = column[static_cast<size_t>(min(firstDoc + d, docCount - 1)) * cats.DocStride];
                }
            }
        } else {
            const size_t doc = min(firstDoc + tid, docCount - 1);
            for (uint32_t c = 0; c < columns; ++c) {
                sCats[c * kCtrTilePitch + tid] = cats.Base[doc * cats.DocStride + columnList[c] * cats.ColumnStride];
            }
        }
        __syncthreads();
    }
    const uint32_t* blockBins = bins + static_cast<size_t>(block) * bucketPitch * kWave + lane;
    const uint32_t shareBegin = blockIdx.y * groupsPerShare;
    const uint32_t shareEnd = min(shareBegin + groupsPerShare, ctr.GroupCount);
    const uint32_t groupsPerWave = (shareEnd - shareBegin + 3) / 4;
    const uint32_t end = min(shareBegin + (wave + 1) * groupsPerWave, shareEnd);
    for (uint32_t g = shareBegin + wave * groupsPerWave; g < end; ++g) {
        const TCtrGroupDev group = ctr.Groups[g];
        uint64_t hash[4] = {0, 0, 0, 0};
        for (uint32_t i = group.ItemBegin; i < group.ItemEnd; ++i) {
            const TCtrItemDev item = ctr.Items[i];
            if (item.Kind == kCtrItemCat) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    uint32_t v;
                    if (TILE) {
                        v = sCats[item.Value * kCtrTilePitch + j * kWave + lane];
                    } else {
                        const size_t column = cats.SplitColumns ? item.SrcSplit : item.SrcFlat;
                        const size_t doc = min(firstDoc + j * kWave + lane, docCount - 1);
                        v = cats.Base[doc * cats.DocStride + column * cats.ColumnStride];
                    }
                    const uint64_t h = CtrHashOfCat(v);
                    hash[j] = i == group.ItemBegin ? h : kCtrMagic * hash[j] + h;
                }
            } else {
                const uint32_t word = blockBins[item.SrcFlat * kWave];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t bin = (word >> (8 * j)) & 0xffu;
                    const bool holds = item.Kind == kCtrItemBinGe ? bin >= item.Value : bin == item.Value;
                    hash[j] = kCtrMagic * hash[j] + (holds ? kCtrMagicSquared : 0u);
                }
            }
        }
        // the four documents' first probes are in flight together; at most half of a table's entries are taken (a quarter where
        // the tables are small together), so that every probe sequence ends at its hash or at an empty entry (all ones) soon
        const uint4* table = ctr.Table + group.FirstPiece;
        uint32_t at[4];
        uint4 entry[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            at[j] = static_cast<uint32_t>(hash[j]) & group.HashMask;
            entry[j] = table[static_cast<size_t>(at[j]) * group.EntryPieces];
        }
        // (a round of further probes goes through all four documents: a loop for each waited for up to four chains of
        // loads one after the other. CTR launch of 1M documents, 24 projections: 125 -> 107 us.)
        for (;;) {
            bool open[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                open[j] = (entry[j].x != static_cast<uint32_t>(hash[j]) || entry[j].y != static_cast<uint32_t>(hash[j] >> 32)) &&
                          (entry[j].x & entry[j].y) != 0xffffffffu;
            }
            if (!(open[0] || open[1] || open[2] || open[3])) {
                break;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (open[j]) {
                    at[j] = (at[j] + 1) & group.HashMask;
                    entry[j] = table[static_cast<size_t>(at[j]) * group.EntryPieces];
                }
            }
        }
        // bytes of four documents and four buckets -> a dword of four documents per bucket
        const uint32_t* buckets = ctr.Buckets + group.FirstBucket;
        const auto store = [&](uint32_t first, uint32_t d0, uint32_t d1, uint32_t d2, uint32_t d3) {
            const uint32_t low01 = __builtin_amdgcn_perm(d1, d0, 0x05010400u), high01 = __builtin_amdgcn_perm(d1, d0, 0x07030602u);
            const uint32_t low23 = __builtin_amdgcn_perm(d3, d2, 0x05010400u), high23 = __builtin_amdgcn_perm(d3, d2, 0x07030602u);
            const uint32_t out[4] = {__builtin_amdgcn_perm(low23, low01, 0x05040100u), __builtin_amdgcn_perm(low23, low01, 0x07060302u),
                                     __builtin_amdgcn_perm(high23, high01, 0x05040100u), __builtin_amdgcn_perm(high23, high01, 0x07060302u)};
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                if (first + k < group.BucketCount) {
                    bins[(static_cast<size_t>(block) * bucketPitch + buckets[first + k]) * kWave + lane] = out[k];
                }
            }
        };
        store(0, entry[0].z, entry[1].z, entry[2].z, entry[3].z);
        if (group.BucketCount > 4) {
            store(4, entry[0].w, entry[1].w, entry[2].w, entry[3].w);
        }
        for (uint32_t piece = 1; piece < group.EntryPieces; ++piece) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                entry[j] = table[static_cast<size_t>(at[j]) * group.EntryPieces + piece];
            }
            const uint32_t first = piece * 16 - 8;
            store(first, entry[0].x, entry[1].x, entry[2].x, entry[3].x);
            store(first + 4, entry[0].y, entry[1].y, entry[2].y, entry[3].y);
            store(first + 8, entry[0].z, entry[1].z, entry[2].z, entry[3].z);
            store(first + 12, entry[0].w, entry[1].w, entry[2].w, entry[3].w);
        }
    }
}

// Final value of one output cell: Scale * sum (+ Bias[k] when the range starts at tree 0),
// as ApplyScaleAndBias (catboost/libs/model/scale_and_bias.cpp:4-50). No fused multiply-add.
__device__ __forceinline__ double Finish(double sum, double scale, double bias, bool addBias) {
    double r = __dmul_rn(scale, sum);
    if (addBias) {
        r = __dadd_rn(r, bias);
    }
    return r;
}

// Copies of a document block's bins into LDS by a workgroup of THREADS threads. A workgroup of the tile kernels has its
// CU to itself or shares it with one other, so nothing else hides the loads: eight of them per thread are issued before
// the first is stored, where a plain loop waits for every one. 4M documents * 500 non-symmetric trees over 300 features
// 7.01 -> 6.50 ms, 970 640 documents * 2934 trees of depth 6 over 614 features (EvalObliviousRowTileKernel) 2.87 -> 2.59.
template <int THREADS, typename T, typename TStore>
__device__ __forceinline__ void CopyInBatches(const T* __restrict__ src, uint32_t count, uint32_t tid, const TStore& store) {
    constexpr int kBatch = 8;
    for (uint32_t first = tid; first < count; first += kBatch * THREADS) {
        T v[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            v[j] = src[min(first + j * THREADS, count - 1)];  // past the end: the last piece again, not stored
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            if (first + j * THREADS < count) {
                store(first + j * THREADS, v[j]);
            }
        }
    }
}

// All `rows` of a block (256 bytes each), row r to the 64 dwords from tile + 64 * place(r) on; four rows that start at a
// multiple of four have places behind each other. In pieces of 16 bytes per lane, four rows to a wave's request, which go
// into LDS without passing through registers, so that every request is on its way before the first has arrived; dword by dword
// where the bins start at an address that does not allow it (a caller's buffer). A wave's requests have arrived behind
// AwaitTile(); a barrier is the caller's. (Through registers, eight pieces to a batch, the compiler moved each load
// behind the test of its own store: a trip to memory per piece. EvalNonSymmetricLdsKernel,
// 1M documents * 500 trees over 300 features 1.240 -> 1.205 ms; launches of the other kernels: EvalObliviousRowTileKernel, 300 000 documents *
// 100 trees of depth 8 over 500 56.5 -> 52.7 us, 500 000 * 500 trees 213 -> 205, EvalObliviousDeepTileKernel, 100 000 * 50 trees of depth 12 over
// 500 23.6 -> 23.0, its pairs, three dimensions over 200, 41.0 -> 39.8, EvalNonSymmetricTileKernel 55.3 -> 54.4; LeafIndexesTileKernel, whole
// call, 100 000 * 200 trees of depth 8 over 560 141.1 -> 126.7.)
template <int THREADS, typename TPlace>
__device__ __forceinline__ void RequestTile(const uint32_t* src, uint32_t rows, uint32_t tid, uint32_t* tile, const TPlace& place) {
    if ((reinterpret_cast<uintptr_t>(src) & 15) == 0) {
        const uint32_t lane = tid & (kWave - 1);
        for (uint32_t row = __builtin_amdgcn_readfirstlane(tid / kWave) * 4; row < rows; row += THREADS / kWave * 4) {
            if (row + lane / 16 < rows) {
                __builtin_amdgcn_global_load_lds(
                    reinterpret_cast<const __attribute__((address_space(1))) void*>(reinterpret_cast<uintptr_t>(src + row * kWave + lane * 4)),
                    (__attribute__((address_space(3))) void*)(tile + place(row) * kWave), 16, 0, 0);
            }
        }
    } else {
        CopyInBatches<THREADS>(src, rows * kWave, tid, [&](uint32_t i, uint32_t v) { tile[place(i / kWave) * kWave + i % kWave] = v; });
    }
}

__device__ __forceinline__ void AwaitTile() {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
}

template <int THREADS>
__device__ __forceinline__ void CopyTile(const uint32_t* src, uint32_t rows, uint32_t tid, uint32_t* tile) {
    RequestTile<THREADS>(src, rows, tid, tile, [](uint32_t row) { return row; });
    AwaitTile();
}

// Oblivious trees, any model: one wave per 256-document block, four documents per lane, leaf
// sums kept in registers in fp64 and accumulated in tree order (as the CPU evaluator does).
// DCHUNK output dimensions are accumulated per pass over the trees.
// mode: kEvalContinue - the sums start from the raw sums of earlier trees found in `out`; kEvalRaw - store raw
// sums (neither scaled nor biased) for a launch that continues them; `addBias` tells the launch that finishes
// whether the whole range started at tree 0 (0 no, 1 yes, 2: this launch is the whole range, treeBegin tells).
// grid = ceil(doc blocks / 4), block = 256 threads.
constexpr uint32_t kEvalContinue = 1;
constexpr uint32_t kEvalRaw = 2;

template <int DCHUNK>
__global__ __launch_bounds__(256) void EvalObliviousKernel(const uint32_t* __restrict__ bins, size_t docCount,
                                                           uint32_t bucketCount, TTreeTables tt, uint32_t treeBegin,
                                                           uint32_t treeEnd, double* out, uint32_t mode,
                                                           uint32_t addBiasFlag) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const size_t block = static_cast<size_t>(blockIdx.x) * (256 / kWave) + threadIdx.x / kWave;
    const size_t blockCount = (docCount + kDocsPerBlock - 1) / kDocsPerBlock;
    if (block >= blockCount) {
        return;
    }
    const uint32_t* myBins = bins + block * bucketCount * kWave + lane;
    const int dim = tt.Dim;
    const bool addBias = addBiasFlag == 2 ? treeBegin == 0 : addBiasFlag != 0;
    for (int d0 = 0; d0 < dim; d0 += DCHUNK) {
        double acc[4][DCHUNK];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const size_t doc = block * kDocsPerBlock + j * kWave + lane;
#pragma unroll
            for (int k = 0; k < DCHUNK; ++k) {
                acc[j][k] = 0.0;
                if ((mode & kEvalContinue) && doc < docCount && (DCHUNK == 1 || d0 + k < dim)) {
                    acc[j][k] = out[doc * dim + d0 + k];
                }
            }
        }
        for (uint32_t t = treeBegin; t < treeEnd; ++t) {
            const uint32_t first = tt.TreeStart[t];
            const uint32_t depth = tt.TreeSize[t];
            uint32_t idx0 = 0, idx1 = 0, idx2 = 0, idx3 = 0;
            for (uint32_t d = 0; d < depth; ++d) {
                const uint32_t sp = tt.Splits[first + d];
                const uint32_t w = myBins[(sp & 0xffffu) * kWave];
                const uint32_t x = (sp >> 16) & 0xffu;
                const uint32_t s = sp >> 24;
                idx0 |= static_cast<uint32_t>(((w & 0xffu) ^ x) >= s) << d;
                idx1 |= static_cast<uint32_t>((((w >> 8) & 0xffu) ^ x) >= s) << d;
                idx2 |= static_cast<uint32_t>((((w >> 16) & 0xffu) ^ x) >= s) << d;
                idx3 |= static_cast<uint32_t>(((w >> 24) ^ x) >= s) << d;
            }
            const double* leaf = tt.Leaves + tt.FirstLeaf[t] + d0;
            const uint32_t idx[4] = {idx0, idx1, idx2, idx3};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const double* p = leaf + static_cast<size_t>(idx[j]) * dim;
#pragma unroll
                for (int k = 0; k < DCHUNK; ++k) {
                    if (DCHUNK == 1 || d0 + k < dim) {
                        acc[j][k] = __dadd_rn(acc[j][k], p[k]);
                    }
                }
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const size_t doc = block * kDocsPerBlock + j * kWave + lane;
            if (doc < docCount) {
#pragma unroll
                for (int k = 0; k < DCHUNK; ++k) {
                    if (DCHUNK == 1 || d0 + k < dim) {
                        out[doc * dim + d0 + k] =
                            (mode & kEvalRaw) ? acc[j][k] : Finish(acc[j][k], tt.Scale, tt.Bias[d0 + k], addBias);
                    }
                }
            }
        }
    }
}

// Small batches on the register-resident kernels: every slice of the trees left its raw sums in
// partials[slice][count]; adds them in slice order and finishes like ApplyScaleAndBias. One thread per value.
// What bounds it: the latency of the loads. A loop of load and add had one in flight; now IN_FLIGHT are (a whole turn past the last
// slice reads that one again), in workgroups of one wave, which a batch of 17 000 documents spreads over every CU. Sixteen for many
// slices; evaluation (register kernel and this one) of 1000 trees of depth 6, 32 slices: 17 000 documents 22.2 -> 16.1 us, 100 000 48.2 ->
// 43.6; of 500 trees and three dimensions, 16 slices, 21.8 -> 17.6 and 41.5 -> 39.4. Workgroups of four waves 16.3 and 43.9, 19.2 and 40.5; 32
// loads 16.0 and 43.7, 18.3 and 40.7. Three up to kFewSlices, where most of sixteen would be of the last slice; 200 000 documents, one in
// flight, three, sixteen: two slices of three dimensions 22.1, 22.1, 25.0 us, four 31.2, 30.3, 32.3, ten of one 30.7, 29.6, 30.0.
constexpr uint32_t kFewSlices = 10;

template <uint32_t IN_FLIGHT>
__global__ __launch_bounds__(64) void CombineSlicesKernel(const double* __restrict__ partials, uint32_t slices,
                                                           size_t count, double scale, const double* __restrict__ bias,
                                                           int dim, double* __restrict__ out) {
    const size_t i = static_cast<size_t>(blockIdx.x) * 64 + threadIdx.x;
    if (i >= count) {
        return;
    }
    double sum = partials[i];
    for (uint32_t first = 1; first < slices; first += IN_FLIGHT) {
        double part[IN_FLIGHT];
#pragma unroll
        for (uint32_t k = 0; k < IN_FLIGHT; ++k) {
            part[k] = partials[min(first + k, slices - 1) * count + i];
        }
#pragma unroll
        for (uint32_t k = 0; k < IN_FLIGHT; ++k) {
            if (first + k < slices) {
                sum = __dadd_rn(sum, part[k]);
            }
        }
    }
    out[i] = Finish(sum, scale, bias[i % static_cast<size_t>(dim)], true);
}

// ---- small batches of oblivious models: one launch from the features to the results ---------
// A batch of a few thousand documents does not fill the chip, and its time is that of launches and of chains of dependent
// loads, so it takes one kernel that compares the features with the splits' borders directly (no bins) and writes the
// finished values; it may read the features from, and write the results to, pinned host memory. The values of the model's
// features of a workgroup's documents go to LDS (a cell each); a tree is a row of sixteen dwords, eight levels' cells and
// eight borders. The trees are summed in slices and the slices in slice order: those of CombineSlicesKernel, or, for models
// that the register kernels do not take, the partial sums of the kernel that larger batches take (each slice the trees of
// one, brought to one length with null trees), so that a document's value does not depend on which kernel took it. The
// sixteen sums of 1000 trees over 700 buckets against slices of 32 trees: 24 us and 22 for 2048 documents, 62 and 60 for
// 16384 (49 and 60 on the binarize and pair-tile kernels). Two forms:
//   FewDocumentsKernel  a workgroup per document, a lane per tree; the leaf values meet in LDS, where a thread per slice
//                       adds its slice. What bounds it: the chain of loads cell -> feature -> leaf value, a few us.
//   SmallBatchKernel    a workgroup per sixteen documents; a row of sixteen lanes (lane = document) walks a slice, the
//                       lane's dword of a tree's row is handed round with DPP row broadcasts (every lane reading the
//                       whole row would hold the texture path for 64 cycles per tree and wave). What bounds it: vector
//                       issue, some 40 instructions per four trees * sixteen documents at two waves per SIMD.
struct TSmallCell {       // a cell of the tile
    uint32_t SrcFlat;     // column in flat rows or columns
    uint32_t SrcSplit;    // column of the float (kind 0, 1) or categorical (kind 2) matrix
    uint32_t Kind;        // 0: the value; 1: the value, NaN as +inf; 2: 1 where the hash is Value, else 0
    uint32_t Value;
};

struct TSmallTables {
    const TSmallCell* Cells;
    const uint32_t* TreeRows;   // [trees + kSmallNullTrees null trees][16]: levels' cells, borders
    const uint32_t* FirstLeaf;  // of a tree in Leaves, the null trees' too
    const double* Leaves;
    const double* Bias;
    double Scale;
    uint32_t CellCount;
    uint32_t Dim;
    uint32_t TreeCount;
    uint32_t SliceTrees;
    uint32_t SliceCount;
};

struct TSmallSource {     // value of feature f of document d: Floats[d * DocStride + f * ColumnStride], in dwords
    const uint32_t* Floats;
    size_t DocStride, ColumnStride;
    const uint32_t* Cats;  // split rows: the hashed categorical values, else null
    size_t CatStride;
    uint32_t Split;        // split rows: columns are float and categorical indexes
};

constexpr int kSmallDocs = 16;                   // documents of a workgroup of SmallBatchKernel
constexpr int kSmallTurn = 16;                   // trees that one of its lanes has in flight, one dimension at a time
constexpr int kSmallNullTrees = 2 * kSmallTurn;
constexpr int kSmallThreads = 512;
constexpr int kFewThreads = 1024;

// Dwords between two documents of SmallBatchKernel's tile, [document][cell] so that a level's cell is one byte offset in
// both kernels. Odd multiples of four: the sixteen documents of a cell fall on sixteen of the 64 banks.
__host__ __device__ __forceinline__ uint32_t SmallDocPitch(uint32_t cells) {
    return (cells + 3) / 8 * 8 + 4;
}

__device__ __forceinline__ uint32_t SmallCellValue(const TSmallSource& src, const TSmallCell& c, size_t doc) {
    uint32_t v;
    if (src.Split && c.Kind == 2) {
        v = src.Cats[doc * src.CatStride + c.SrcSplit];
    } else {
        v = src.Floats[doc * src.DocStride + (src.Split ? c.SrcSplit : c.SrcFlat) * src.ColumnStride];
    }
    if (c.Kind == 1) {
        v = isnan(__uint_as_float(v)) ? 0x7f800000u : v;
    } else if (c.Kind == 2) {
        v = v == c.Value ? 0x3f800000u : 0u;
    }
    return v;
}

// Start and end of a workgroup on the device's wall clock: stamps[workgroup][2]. (One pair for the launch, minimum and
// maximum by atomics, held a launch of 256 workgroups back by some 5 us.)
__device__ __forceinline__ void SmallStamp(ulonglong2* stamps, unsigned long long began) {
    stamps[blockIdx.y * gridDim.x + blockIdx.x] = make_ulonglong2(began, wall_clock64());
}

// How a host call of few documents learns that a workgroup is done: its results are in (coherent, pinned) host memory when its
// flag is the ticket. Looking at the flags is shorter than waiting until the launch is retired.
struct TSmallDone {
    uint32_t* Flags;  // [workgroup]; null: the end of the launch says so
    uint32_t Ticket;
};

// (The second argument is SmallBatchKernel's number of documents; here the grid has it.)
// grid = (documents, ceil(dim / DIMS)), block = whole waves, at most kFewThreads; dynamic LDS = CellCount * 4 rounded up
// to 8 + DIMS * SliceCount * (SliceTrees + 2) * 8 bytes.
template <int DEPTH, int DIMS>
__global__ __launch_bounds__(kFewThreads) void FewDocumentsKernel(TSmallSource src, uint32_t, TSmallTables tab,
                                                                  double* __restrict__ out, ulonglong2* __restrict__ stamps,
                                                                  TSmallDone done) {
    extern __shared__ uint32_t sSmall[];
    const unsigned long long began = wall_clock64();
    const uint32_t tid = threadIdx.x, threads = blockDim.x;
    const uint32_t doc = blockIdx.x, d0 = blockIdx.y * DIMS;
    const uint32_t pitch = tab.SliceTrees + 1;  // the slices' values, one behind another, fall on different banks
    double* values = reinterpret_cast<double*>(sSmall + (tab.CellCount + 1) / 2 * 2);  // [k][slice][pitch]
    double* sums = values + static_cast<size_t>(DIMS) * tab.SliceCount * pitch;        // [k][slice]
    uint4 cells[2], borders[2];
    uint32_t first = 0;
    const auto fetch = [&](uint32_t t) {
        const uint4* row = reinterpret_cast<const uint4*>(tab.TreeRows) + static_cast<size_t>(t) * 4;
        cells[0] = row[0];
        borders[0] = row[2];
        cells[1] = row[1];
        borders[1] = row[3];
        first = tab.FirstLeaf[t];
    };
    fetch(min(tid, tab.TreeCount - 1));  // in flight while the cells are filled
    for (uint32_t i = tid; i < tab.CellCount; i += threads) {
        sSmall[i] = SmallCellValue(src, tab.Cells[i], doc);
    }
    __syncthreads();
    const uint8_t* tile = reinterpret_cast<const uint8_t*>(sSmall);
    for (uint32_t t = tid; t < tab.TreeCount; t += threads) {
        if (t != tid) {
            fetch(t);
        }
        const uint32_t at[8] = {cells[0].x, cells[0].y, cells[0].z, cells[0].w, cells[1].x, cells[1].y, cells[1].z, cells[1].w};
        const uint32_t border[8] = {borders[0].x, borders[0].y, borders[0].z, borders[0].w,
                                    borders[1].x, borders[1].y, borders[1].z, borders[1].w};
        uint32_t idx = 0;
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            const float x = *reinterpret_cast<const float*>(tile + at[d]);
            idx |= (x > __uint_as_float(border[d]) ? 1u : 0u) << d;
        }
        const double* p = tab.Leaves + first + static_cast<size_t>(idx) * tab.Dim + d0;
        const uint32_t slice = t / tab.SliceTrees, cell = slice * pitch + (t - slice * tab.SliceTrees);
#pragma unroll
        for (int k = 0; k < DIMS; ++k) {
            if (DIMS == 1 || d0 + k < tab.Dim) {
                values[k * tab.SliceCount * pitch + cell] = p[k];
            }
        }
    }
    __syncthreads();
    const uint32_t dims = DIMS == 1 ? 1 : min(static_cast<uint32_t>(DIMS), tab.Dim - d0);
    for (uint32_t i = tid; i < tab.SliceCount * dims; i += threads) {
        const uint32_t slice = i % tab.SliceCount;
        const uint32_t count = min(tab.SliceTrees, tab.TreeCount - slice * tab.SliceTrees);
        const double* v = values + static_cast<size_t>(i) * pitch;
        double sum = 0.0;
#pragma unroll 8
        for (uint32_t t = 0; t < count; ++t) {
            sum = __dadd_rn(sum, v[t]);
        }
        sums[i] = sum;
    }
    __syncthreads();
    if (tid < dims) {
        const double* v = sums + tid * tab.SliceCount;
        double sum = v[0];
#pragma unroll 8
        for (uint32_t slice = 1; slice < tab.SliceCount; ++slice) {
            sum = __dadd_rn(sum, v[slice]);
        }
        out[static_cast<size_t>(doc) * tab.Dim + d0 + tid] = Finish(sum, tab.Scale, tab.Bias[d0 + tid], true);
        if (tid == 0) {
            SmallStamp(stamps, began);
        }
        if (done.Flags != nullptr) {
            __threadfence_system();  // the results, which lanes of this one wave wrote, and the stamps first
            if (tid == 0) {
                __hip_atomic_store(done.Flags + blockIdx.y * gridDim.x + blockIdx.x, done.Ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
    }
}

// the value of lane N of the lane's row of sixteen
template <int N>
__device__ __forceinline__ uint32_t RowBroadcast(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x150 + N, 0xf, 0xf, true));
}

// leaf indexes of trees FIRST .. FIRST + 3 of a turn; level d decides bit d
template <int D, int FIRST, int N>
__device__ __forceinline__ void SmallLevels(const uint8_t* docTile, const uint32_t (&row)[N], uint32_t (&idx)[4]) {
    if constexpr (D >= 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float x = *reinterpret_cast<const float*>(docTile + RowBroadcast<D>(row[FIRST + i]));
            idx[i] = idx[i] + idx[i] + (x > __uint_as_float(RowBroadcast<8 + D>(row[FIRST + i])) ? 1u : 0u);
        }
        SmallLevels<D - 1, FIRST>(docTile, row, idx);
    }
}

// The leaf values of a turn's trees, four trees at a time: the scheduler would otherwise start the reads of all of them
// and spill. `leafOfLane`: first leaf of tree i in lane i of the row.
template <int DEPTH, int DIMS, int FIRST, int N>
__device__ __forceinline__ void SmallLeafValues(const uint8_t* docTile, const uint32_t (&row)[N], uint32_t leafOfLane,
                                                const double* leaves, uint32_t dim, uint32_t dimsLeft, double (&value)[N][DIMS]) {
    if constexpr (FIRST < N) {
        uint32_t idx[4] = {0, 0, 0, 0};
        SmallLevels<DEPTH - 1, FIRST>(docTile, row, idx);
        const uint32_t leaf[4] = {RowBroadcast<FIRST>(leafOfLane), RowBroadcast<FIRST + 1>(leafOfLane),
                                  RowBroadcast<FIRST + 2>(leafOfLane), RowBroadcast<FIRST + 3>(leafOfLane)};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const double* p = leaves + (DIMS == 1 ? leaf[i] + idx[i] : leaf[i] + static_cast<size_t>(idx[i]) * dim);
#pragma unroll
            for (int k = 0; k < DIMS; ++k) {
                value[FIRST + i][k] = DIMS == 1 || static_cast<uint32_t>(k) < dimsLeft ? p[k] : 0.0;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        SmallLeafValues<DEPTH, DIMS, FIRST + 4>(docTile, row, leafOfLane, leaves, dim, dimsLeft, value);
    }
}

// grid = (ceil(documents / 16), ceil(dim / DIMS)), block = kSmallThreads: 32 slices at a time;
// dynamic LDS = 16 * SmallDocPitch(CellCount) * 4 + SliceCount * 16 * DIMS * 8 bytes.
template <int DEPTH, int DIMS>
__global__ __launch_bounds__(kSmallThreads) void SmallBatchKernel(TSmallSource src, uint32_t docCount, TSmallTables tab,
                                                                  double* __restrict__ out, ulonglong2* __restrict__ stamps) {
    // trees of a turn: their rows, and the leaf values of the turn before, are in flight together
    constexpr int kTurn = kSmallTurn / DIMS;
    static_assert(2 * kTurn <= kSmallNullTrees, "rows are fetched up to a turn past the last one");
    extern __shared__ uint32_t sSmall[];
    const unsigned long long began = wall_clock64();
    constexpr uint32_t threads = kSmallThreads;
    const uint32_t tid = threadIdx.x;
    const uint32_t firstDoc = blockIdx.x * kSmallDocs;
    const uint32_t docs = min(static_cast<uint32_t>(kSmallDocs), docCount - firstDoc);
    const uint32_t d0 = blockIdx.y * DIMS;
    const uint32_t lane = tid % kSmallDocs;
    const uint32_t docPitch = SmallDocPitch(tab.CellCount);
    double* sums = reinterpret_cast<double*>(sSmall + docPitch * kSmallDocs);  // [slice][k][document]
    uint32_t next[kTurn], nextLeaf;
    const auto fetch = [&](uint32_t t) {
#pragma unroll
        for (int i = 0; i < kTurn; ++i) {
            next[i] = tab.TreeRows[static_cast<size_t>(t + i) * 16 + lane];
        }
        nextLeaf = tab.FirstLeaf[t + lane % kTurn];  // lane i: tree i's
    };
    fetch(min(tid / kSmallDocs * tab.SliceTrees, tab.TreeCount));  // in flight while the tile is filled
    // Neighbouring threads read neighbouring addresses: cells of a document, or documents of a column. A thread's cells of
    // a turn are asked for together, then their values: two trips to memory for up to 256 (128) cells.
    constexpr uint32_t kCells = 4;
    if (src.ColumnStride == 1) {
        constexpr uint32_t kDocs = kSmallDocs / (kSmallThreads / kWave);
        for (uint32_t cell = tid % kWave; cell < tab.CellCount; cell += kCells * kWave) {
            TSmallCell c[kCells];
            uint32_t v[kCells][kDocs];
#pragma unroll
            for (uint32_t i = 0; i < kCells; ++i) {
                c[i] = tab.Cells[min(cell + i * kWave, tab.CellCount - 1)];
            }
#pragma unroll
            for (uint32_t i = 0; i < kCells; ++i) {
#pragma unroll
                for (uint32_t j = 0; j < kDocs; ++j) {
                    v[i][j] = SmallCellValue(src, c[i], firstDoc + min(tid / kWave * kDocs + j, docs - 1));
                }
            }
#pragma unroll
            for (uint32_t i = 0; i < kCells; ++i) {
#pragma unroll
                for (uint32_t j = 0; j < kDocs; ++j) {
                    if (cell + i * kWave < tab.CellCount) {
                        sSmall[(cell + i * kWave) + (tid / kWave * kDocs + j) * docPitch] = v[i][j];
                    }
                }
            }
        }
    } else {
        constexpr uint32_t kRows = kSmallThreads / kSmallDocs;
        for (uint32_t cell = tid / kSmallDocs; cell < tab.CellCount; cell += kCells * kRows) {
            TSmallCell c[kCells];
            uint32_t v[kCells];
#pragma unroll
            for (uint32_t i = 0; i < kCells; ++i) {
                c[i] = tab.Cells[min(cell + i * kRows, tab.CellCount - 1)];
            }
#pragma unroll
            for (uint32_t i = 0; i < kCells; ++i) {
                v[i] = SmallCellValue(src, c[i], firstDoc + min(lane, docs - 1));
            }
#pragma unroll
            for (uint32_t i = 0; i < kCells; ++i) {
                if (cell + i * kRows < tab.CellCount) {
                    sSmall[(cell + i * kRows) + lane * docPitch] = v[i];
                }
            }
        }
    }
    __syncthreads();
    const uint8_t* docTile = reinterpret_cast<const uint8_t*>(sSmall + lane * docPitch);  // (documents past the last one: the last one again)
    const double* leaves = tab.Leaves + d0;
    for (uint32_t slice = tid / kSmallDocs; slice < tab.SliceCount; slice += threads / kSmallDocs) {
        const uint32_t begin = slice * tab.SliceTrees;
        const uint32_t end = min(begin + tab.SliceTrees, tab.TreeCount);
        if (slice != tid / kSmallDocs) {
            fetch(begin);
        }
        double acc[DIMS], value[kTurn][DIMS];
#pragma unroll
        for (int k = 0; k < DIMS; ++k) {
            acc[k] = 0.0;
        }
        // Slices are a multiple of a turn, or the whole model: trees past the end of it are null trees, whose leaf is zero.
        const auto add = [&] {
#pragma unroll
            for (int i = 0; i < kTurn; ++i) {
#pragma unroll
                for (int k = 0; k < DIMS; ++k) {
                    acc[k] = __dadd_rn(acc[k], value[i][k]);
                }
            }
        };
        for (uint32_t t = begin; t < end; t += kTurn) {
            uint32_t row[kTurn];
#pragma unroll
            for (int i = 0; i < kTurn; ++i) {
                row[i] = next[i];
            }
            const uint32_t leafOfLane = nextLeaf;
            if (t + kTurn < end) {
                fetch(t + kTurn);
            }
            if (t > begin) {
                add();  // the values of the turn before
            }
            SmallLeafValues<DEPTH, DIMS, 0>(docTile, row, leafOfLane, leaves, tab.Dim, tab.Dim - d0, value);
        }
        add();
#pragma unroll
        for (int k = 0; k < DIMS; ++k) {
            sums[(slice * DIMS + k) * kSmallDocs + lane] = acc[k];
        }
    }
    __syncthreads();
    if (tid < kSmallDocs * DIMS) {
        const uint32_t k = tid / kSmallDocs;
        if (lane < docs && d0 + k < tab.Dim) {
            double sum = sums[tid];
#pragma unroll 8
            for (uint32_t slice = 1; slice < tab.SliceCount; ++slice) {
                sum = __dadd_rn(sum, sums[slice * DIMS * kSmallDocs + tid]);
            }
            out[static_cast<size_t>(firstDoc + lane) * tab.Dim + d0 + k] = Finish(sum, tab.Scale, tab.Bias[d0 + k], true);
        }
        if (tid == 0) {
            SmallStamp(stamps, began);
        }
    }
}

// Packed tree table of the tile kernel: 16 dwords per tree. Slots 0..7 hold the tree's levels
// (slot d = split d, unused levels padded with a split that is false for every bin), slot 8 the
// index of the tree's first leaf value. A level is
//   7-bit form: bucket << 8 | (128 - splitIdx)          (all bins and split indexes <= 127, no xor)
//   8-bit form: bucket << 16 | xorMask << 8 | splitIdx
constexpr int kPackedTreeDwords = 16;
constexpr int kPackedFirstLeafSlot = 8;

// Bit 7 of every byte of the result tells whether (bin ^ xorMask) >= splitIdx for the four
// documents packed in `a`. 7-bit form: adding (128 - splitIdx) to every byte carries into bit 7
// exactly when bin >= splitIdx. 8-bit form: the unsigned compare is the carry out of
// x + ~splitIdx + 1 taken per byte, x = bin ^ xorMask:
//   carry = (x & ns) | ((x | ns) & low), ns = ~splitIdx, low = (x & 0x7f) + (ns & 0x7f) + 1.
template <bool SEVEN_BIT>
__device__ __forceinline__ uint32_t CompareBytes(uint32_t a, uint32_t level) {
    if (SEVEN_BIT) {
        return a + (level & 0xffu) * 0x01010101u;
    }
    const uint32_t s = level & 0xffu;
    const uint32_t x = a ^ (((level >> 8) & 0xffu) * 0x01010101u);
    const uint32_t ns = (~s) & 0xffu;
    const uint32_t low = (x & 0x7f7f7f7fu) + ((ns & 0x7fu) + 1u) * 0x01010101u;
    const uint32_t nsr = ns * 0x01010101u;
    return (x & nsr) | ((x | nsr) & low);
}

// byte offset of a level's bucket inside the LDS tile (256 bytes per bucket)
template <bool SEVEN_BIT>
__device__ __forceinline__ uint32_t LevelTileOffset(uint32_t level) {
    return SEVEN_BIT ? (level & 0xffffff00u) : ((level >> 16) << 8);
}

// Leaf indexes of one tree for the four documents of a lane, one byte each: MAXD levels, every
// one an LDS dword read, a byte-parallel compare and a shift-in of the four result bits (the
// first split ends up in bit 0).
template <bool SEVEN_BIT, int MAXD>
__device__ __forceinline__ uint32_t TreeIndexes(const uint8_t* laneTile, uint32_t packedRow) {
    uint32_t idx4 = 0;
#pragma unroll
    for (int d = 0; d < MAXD; ++d) {
        const uint32_t level = __builtin_amdgcn_readlane(packedRow, d);
        const uint32_t a = *reinterpret_cast<const uint32_t*>(laneTile + LevelTileOffset<SEVEN_BIT>(level));
        const uint32_t r = CompareBytes<SEVEN_BIT>(a, level);
        idx4 = (r & 0x80808080u) | ((idx4 >> 1) & 0x7f7f7f7fu);
    }
    return idx4 >> (8 - MAXD);
}

// The same for four trees whose packed rows sit side by side in the lanes of `packedRows` (kPackedTreeDwords lanes
// each): all LDS reads of the four trees are in flight before the first compare.
template <bool SEVEN_BIT, int MAXD>
__device__ __forceinline__ void FourTreesIndexes(const uint8_t* laneTile, uint32_t packedRows, uint32_t (&idx)[4]) {
    uint32_t a[4][MAXD];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int d = 0; d < MAXD; ++d) {
            const uint32_t level = __builtin_amdgcn_readlane(packedRows, i * kPackedTreeDwords + d);
            a[i][d] = *reinterpret_cast<const uint32_t*>(laneTile + LevelTileOffset<SEVEN_BIT>(level));
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t idx4 = 0;
#pragma unroll
        for (int d = 0; d < MAXD; ++d) {
            const uint32_t level = __builtin_amdgcn_readlane(packedRows, i * kPackedTreeDwords + d);
            const uint32_t r = CompareBytes<SEVEN_BIT>(a[i][d], level);
            idx4 = (r & 0x80808080u) | ((idx4 >> 1) & 0x7f7f7f7fu);
        }
        idx[i] = idx4 >> (8 - MAXD);
    }
}

// Oblivious trees of depth <= MAXD <= 8 whose bins fit an LDS tile: one workgroup of kTileWaves
// waves per 256-document block. The block's bins (buckets x 256 bytes) are copied to LDS once;
// the waves share the tile and split the trees among themselves (tree t goes to wave
// t % kTileWaves), four documents per lane. A wave fetches a tree's packed row with one 64-byte
// load (two trees ahead) and broadcasts the levels from it. Per-wave partial sums (fp64) are added
// in wave order through an LDS accumulator behind the tile, and the last wave writes the results.
//
// Leaf values. DCHUNK == 1 (one-dimensional models): `leaves` is the model's array and slot 8 of a
// packed row the tree's first value. DCHUNK > 1: `leaves` is a copy padded to DCHUNK values per
// leaf, one run of (leaf count) x DCHUNK values per tree and chunk of DCHUNK dimensions (zeros
// behind the last dimension); slot 9 is the tree's first padded value and slot 10 its leaf count.
// A lane adds all DCHUNK values of a leaf without looking at the dimension; only the final store
// does. LEAF_LDS: every wave copies the (1 << MAXD) * DCHUNK values of its current tree and chunk
// into a private LDS region with row-contiguous 16-byte loads, one tree ahead through registers
// when that takes at most 8 loads per lane, and gathers from there; otherwise the values are
// gathered straight from global memory. `leaves` must be readable for (1 << MAXD) * DCHUNK values
// past the first value of the last tree.
// WAVES waves share a block (tree t goes to wave t % WAVES): kTileWaves, or kWideTileWaves when the
// tile is so large that only one workgroup fits a CU: the waves of a workgroup wait on LDS round trips
// most of the time, and sixteen of them hide what eight cannot (400 buckets: 1.75 instead of 2.79 ms).
// grid = doc blocks, block = 64 * WAVES threads, dynamic LDS = buckets * 256 (rounded up to
// 8) + 256 * DCHUNK * 8 [+ WAVES * (1 << MAXD) * DCHUNK * 8 with LEAF_LDS] bytes.
constexpr int kTileWaves = 8;
constexpr int kWideTileWaves = 16;
constexpr int kPackedPaddedLeafSlot = 9;
constexpr int kPackedLeafCountSlot = 10;

template <bool SEVEN_BIT, int MAXD, int DCHUNK, bool LEAF_LDS, int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(2, 4))) void EvalObliviousTileKernel(
    const uint32_t* __restrict__ bins, size_t docCount, uint32_t bucketCount, const uint32_t* __restrict__ packedTrees,
    const double* __restrict__ leaves, const double* __restrict__ bias, double scale, int dim, uint32_t treeBegin,
    uint32_t treeEnd, double* __restrict__ out) {
    static_assert(DCHUNK == 1 || DCHUNK % 2 == 0, "padded leaf rows are copied in 16-byte pairs");
    constexpr uint32_t kTreeDoubles = (1u << MAXD) * DCHUNK;    // values of one tree and chunk in LDS
    constexpr uint32_t kTreePairs = kTreeDoubles / 2;
    constexpr int kPairsPerLane = static_cast<int>((kTreePairs + kWave - 1) / kWave);
    constexpr bool kPrefetch = kPairsPerLane <= 8;  // registers of the copy that runs one tree ahead
    constexpr int kPrefetchRegs = kPrefetch ? kPairsPerLane : 1;
    constexpr int kFirstSlot = DCHUNK == 1 ? kPackedFirstLeafSlot : kPackedPaddedLeafSlot;
    extern __shared__ uint32_t sTile[];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const size_t block = blockIdx.x;
    const uint32_t tileDwords = bucketCount * kWave;
    const uint32_t* src = bins + block * tileDwords;
    CopyTile<64 * WAVES>(src, bucketCount, tid, sTile);
    const bool addBias = treeBegin == 0;
    const uint8_t* laneTile = reinterpret_cast<const uint8_t*>(sTile) + lane * 4;
    const uint32_t slot = lane & (kPackedTreeDwords - 1);
    double* sRed = reinterpret_cast<double*>(sTile + ((tileDwords + 1) & ~1u));
    double* sLeaf = sRed + kDocsPerBlock * DCHUNK + wave * kTreeDoubles;  // per-wave leaf region
    for (int d0 = 0; d0 < dim; d0 += DCHUNK) {
        __syncthreads();  // tile is loaded / the previous chunk's accumulator has been read
        const uint32_t chunk = static_cast<uint32_t>(d0) / DCHUNK;
        double acc[4][DCHUNK];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int k = 0; k < DCHUNK; ++k) {
                acc[j][k] = 0.0;
            }
        }
        double2 pref[kPrefetchRegs];
#pragma unroll
        for (int i = 0; i < kPrefetchRegs; ++i) {
            pref[i] = {0.0, 0.0};
        }
        // first value of this chunk of the tree whose packed row is `rowValue`
#define CBAMD_TREE_VALUES(rowValue)                                                               \
    (leaves + __builtin_amdgcn_readlane(rowValue, kFirstSlot) +                                   \
     (DCHUNK == 1 ? 0u : chunk * __builtin_amdgcn_readlane(rowValue, kPackedLeafCountSlot) * DCHUNK))
#define CBAMD_FETCH_LEAVES(rowValue)                                                              \
    do {                                                                                          \
        const double2* src2 = reinterpret_cast<const double2*>(CBAMD_TREE_VALUES(rowValue));     \
        _Pragma("unroll") for (int i = 0; i < kPrefetchRegs; ++i) {                               \
            if (static_cast<uint32_t>(i + 1) * kWave <= kTreePairs || i * kWave + lane < kTreePairs) { \
                pref[i] = src2[i * kWave + lane];                                                 \
            }                                                                                     \
        }                                                                                         \
    } while (0)
        // packed rows are fetched two trees ahead so that the next tree's row has arrived by the
        // time its leaf values are requested
#define CBAMD_FETCH_ROW(tree) \
    ((tree) < treeEnd ? packedTrees[static_cast<size_t>(tree) * kPackedTreeDwords + slot] : 0u)
        uint32_t t = treeBegin + wave;
        uint32_t row = CBAMD_FETCH_ROW(t);
        uint32_t rowNext = CBAMD_FETCH_ROW(t + WAVES);
        if (LEAF_LDS && kPrefetch && t < treeEnd) {
            CBAMD_FETCH_LEAVES(row);
        }
        while (t < treeEnd) {
            const uint32_t tNext = t + WAVES;
            const uint32_t rowNext2 = CBAMD_FETCH_ROW(tNext + WAVES);
            const double* leaf = CBAMD_TREE_VALUES(row);
            if (LEAF_LDS) {
                // publish this tree's leaf values in the wave's region; the previous tree's gathers
                // were issued before these stores and LDS serves one wave's requests in order
                double2* dst2 = reinterpret_cast<double2*>(sLeaf);
                if (kPrefetch) {
#pragma unroll
                    for (int i = 0; i < kPrefetchRegs; ++i) {
                        if (static_cast<uint32_t>(i + 1) * kWave <= kTreePairs || i * kWave + lane < kTreePairs) {
                            dst2[i * kWave + lane] = pref[i];
                        }
                    }
                    if (tNext < treeEnd) {
                        CBAMD_FETCH_LEAVES(rowNext);
                    }
                } else {
                    const double2* src2 = reinterpret_cast<const double2*>(leaf);
                    for (uint32_t i = lane; i < kTreePairs; i += kWave) {
                        dst2[i] = src2[i];
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                leaf = sLeaf;
            }
            const uint32_t idx4 = TreeIndexes<SEVEN_BIT, MAXD>(laneTile, row);
            if (DCHUNK == 1) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    acc[j][0] = __dadd_rn(acc[j][0], leaf[(idx4 >> (8 * j)) & 0xffu]);
                }
            } else {
                // the DCHUNK values of the next document's leaf are requested before the current
                // document's are added (the scheduling fences keep the two groups apart)
                double val[2][DCHUNK];
#pragma unroll
                for (int k = 0; k < DCHUNK; ++k) {
                    val[0][k] = leaf[(idx4 & 0xffu) * DCHUNK + k];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (j < 3) {
#pragma unroll
                        for (int k = 0; k < DCHUNK; ++k) {
                            val[(j + 1) & 1][k] = leaf[((idx4 >> (8 * (j + 1))) & 0xffu) * DCHUNK + k];
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int k = 0; k < DCHUNK; ++k) {
                        acc[j][k] = __dadd_rn(acc[j][k], val[j & 1][k]);
                    }
                }
            }
            if (LEAF_LDS) {
                __builtin_amdgcn_wave_barrier();
            }
            t = tNext;
            row = rowNext;
            rowNext = rowNext2;
        }
#undef CBAMD_FETCH_ROW
#undef CBAMD_FETCH_LEAVES
#undef CBAMD_TREE_VALUES
        // waves add their partial sums in wave order into the LDS accumulator; the last wave
        // finishes the values and writes them out
        for (uint32_t w = 0; w + 1 < WAVES; ++w) {
            if (wave == w) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
#pragma unroll
                    for (int k = 0; k < DCHUNK; ++k) {
                        double* cell = sRed + (j * kWave + lane) * DCHUNK + k;
                        *cell = (w == 0) ? acc[j][k] : __dadd_rn(*cell, acc[j][k]);
                    }
                }
            }
            __syncthreads();
        }
        if (wave == WAVES - 1) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const size_t doc = block * kDocsPerBlock + j * kWave + lane;
#pragma unroll
                for (int k = 0; k < DCHUNK; ++k) {
                    if (doc < docCount && (DCHUNK == 1 || d0 + k < dim)) {
                        const double sum = __dadd_rn(sRed[(j * kWave + lane) * DCHUNK + k], acc[j][k]);
                        out[doc * dim + d0 + k] = Finish(sum, scale, bias[d0 + k], addBias);
                    }
                }
            }
        }
    }
}

// One-dimensional oblivious models whose bins do not fit the 256-document tile (more than ~600
// buckets): the same scheme on half a block. A workgroup copies the bins of 128 documents
// (buckets x 128 bytes, two documents per lane: documents (2 * half + j) * 64 + lane of the block)
// and its waves split the trees; everything else is EvalObliviousTileKernel with DCHUNK == 1 and
// leaf values through LDS. `leaves` holds (1 << MAXD) values per tree at a fixed pitch.
// The packed rows come in the form chosen per tree (bit 31 of slot kPackedFormSlot): the 7-bit form
// when the tree has no one-hot split and all float bins of the model fit 7 bits, else the 8-bit form;
// a model with a few one-hot splits pays the longer compare only in the trees that have them.
// A 7-bit row holds what a level needs ready for use, so that a level costs two lane reads and no scalar
// arithmetic: slot d the byte offset of the level's bucket in the half tile (bucket * 128), slot 8 + d
// (128 - splitIdx) * 0x0101. An 8-bit row holds bucket << 16 | xorMask << 8 | splitIdx in slot d.
// grid = 2 * doc blocks, block = 64 * kTileWaves threads, dynamic LDS = buckets * 128 (rounded up
// to 8) + 128 * 8 + kTileWaves * (1 << MAXD) * 8 bytes.
constexpr int kPackedFormSlot = 8;  // mixed table, bit 31: clear = 7-bit form, set = 8-bit form

template <bool SEVEN_BIT, int MAXD>
__device__ __forceinline__ uint32_t TreeIndexesPair(const uint8_t* laneTile, uint32_t packedRow) {
    uint32_t idx2 = 0;
#pragma unroll
    for (int d = 0; d < MAXD; ++d) {
        uint32_t r;
        if (SEVEN_BIT) {
            const uint32_t a = *reinterpret_cast<const uint16_t*>(laneTile + __builtin_amdgcn_readlane(packedRow, d));
            r = a + __builtin_amdgcn_readlane(packedRow, 8 + d);
        } else {
            const uint32_t level = __builtin_amdgcn_readlane(packedRow, d);
            const uint32_t a = *reinterpret_cast<const uint16_t*>(laneTile + (LevelTileOffset<false>(level) >> 1));
            r = CompareBytes<false>(a, level);
        }
        // bits 7 and 15 from r, the rest from the shifted index: one v_bfi. What a sum carries past bit 15
        // moves down one bit per level and is replaced when it reaches bit 15.
        idx2 = (r & 0x8080u) | ((idx2 >> 1) & ~0x8080u);
    }
    return (idx2 & 0xffffu) >> (8 - MAXD);
}

template <int MAXD>
__global__ __launch_bounds__(64 * kTileWaves) void EvalObliviousHalfTileKernel(
    const uint16_t* __restrict__ bins, size_t docCount, uint32_t bucketCount, const uint32_t* __restrict__ packedMixed,
    const double* __restrict__ leaves, const double* __restrict__ bias, double scale, uint32_t treeBegin,
    uint32_t treeEnd, double* __restrict__ out) {
    constexpr uint32_t kTreePairs = (1u << MAXD) / 2;
    constexpr int kPrefetchRegs = static_cast<int>((kTreePairs + kWave - 1) / kWave);
    extern __shared__ uint32_t sTile[];
    uint16_t* sTile16 = reinterpret_cast<uint16_t*>(sTile);
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const size_t block = blockIdx.x >> 1;
    const uint32_t half = blockIdx.x & 1;
    const uint32_t tileWords = bucketCount * kWave;
    const uint16_t* src = bins + block * tileWords * 2 + half;
    for (uint32_t i = tid; i < tileWords; i += 64 * kTileWaves) {
        sTile16[i] = src[2 * i];
    }
    const bool addBias = treeBegin == 0;
    const uint8_t* laneTile = reinterpret_cast<const uint8_t*>(sTile) + lane * 2;
    const uint32_t slot = lane & (kPackedTreeDwords - 1);
    double* sRed = reinterpret_cast<double*>(sTile + ((tileWords / 2 + 1) & ~1u));
    double* sLeaf = sRed + 2 * kWave + wave * (1u << MAXD);  // per-wave leaf region
    __syncthreads();  // tile is loaded
    double acc[2] = {0.0, 0.0};
    // A wave has only one partner on its SIMD here (the tile leaves room for one workgroup per CU),
    // so what it needs from global memory is requested kAhead of its trees ahead: the packed row
    // and the leaf values ((1 << MAXD) doubles per tree at a fixed pitch) of tree t + kAhead * 8
    // go into the registers that tree t has just given up.
    constexpr int kAhead = 4;
    uint32_t rows[kAhead];
    double2 pref[kAhead][kPrefetchRegs];
#define CBAMD_FETCH_TREE(k, tree)                                                                 \
    do {                                                                                          \
        const uint32_t fetchTree = (tree);                                                        \
        rows[k] = 0u;                                                                             \
        if (fetchTree < treeEnd) {                                                                \
            rows[k] = packedMixed[static_cast<size_t>(fetchTree) * kPackedTreeDwords + slot];     \
            const double2* src2 = reinterpret_cast<const double2*>(leaves) + static_cast<size_t>(fetchTree) * kTreePairs; \
            _Pragma("unroll") for (int i = 0; i < kPrefetchRegs; ++i) {                           \
                if (static_cast<uint32_t>(i + 1) * kWave <= kTreePairs || i * kWave + lane < kTreePairs) { \
                    pref[k][i] = src2[i * kWave + lane];                                          \
                }                                                                                 \
            }                                                                                     \
        }                                                                                         \
    } while (0)
    uint32_t t = treeBegin + wave;
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
#pragma unroll
        for (int i = 0; i < kPrefetchRegs; ++i) {
            pref[k][i] = {0.0, 0.0};
        }
        CBAMD_FETCH_TREE(k, t + k * kTileWaves);
    }
    while (t < treeEnd) {
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            if (t < treeEnd) {
                // publish this tree's leaf values in the wave's region; the previous tree's gathers
                // were issued before these stores and LDS serves one wave's requests in order
                double2* dst2 = reinterpret_cast<double2*>(sLeaf);
#pragma unroll
                for (int i = 0; i < kPrefetchRegs; ++i) {
                    if (static_cast<uint32_t>(i + 1) * kWave <= kTreePairs || i * kWave + lane < kTreePairs) {
                        dst2[i * kWave + lane] = pref[k][i];
                    }
                }
                const uint32_t row = rows[k];
                CBAMD_FETCH_TREE(k, t + kAhead * kTileWaves);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                uint32_t idx2;
                if (__builtin_amdgcn_readlane(row, kPackedFormSlot) >> 31) {
                    idx2 = TreeIndexesPair<false, MAXD>(laneTile, row);
                } else {
                    idx2 = TreeIndexesPair<true, MAXD>(laneTile, row);
                }
                acc[0] = __dadd_rn(acc[0], sLeaf[idx2 & 0xffu]);
                acc[1] = __dadd_rn(acc[1], sLeaf[(idx2 >> 8) & 0xffu]);
                __builtin_amdgcn_wave_barrier();
                t += kTileWaves;
            }
        }
    }
#undef CBAMD_FETCH_TREE
    // waves add their partial sums in wave order into the LDS accumulator; the last wave
    // finishes the values and writes them out
    for (uint32_t w = 0; w + 1 < kTileWaves; ++w) {
        if (wave == w) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                double* cell = sRed + j * kWave + lane;
                *cell = (w == 0) ? acc[j] : __dadd_rn(*cell, acc[j]);
            }
        }
        __syncthreads();
    }
    if (wave == kTileWaves - 1) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const size_t doc = block * kDocsPerBlock + (2 * half + j) * kWave + lane;
            if (doc < docCount) {
                out[doc] = Finish(__dadd_rn(sRed[j * kWave + lane], acc[j]), scale, bias[0], addBias);
            }
        }
    }
}

// The same half tile with two trees in flight per wave: lanes 0..31 evaluate one tree and lanes 32..63 the
// next one, each lane for four documents of the tile (one LDS dword: the bins of documents
// (2 * half + j) * 64 + 2 * m + i, byte 2 * i + j, for lane m of either group), so a level costs one LDS read
// and one byte-parallel compare for 2 x 128 (tree, document) pairs instead of 128. Needs every bin of the
// tile below 128 (the 7-bit compare; a one-hot level xors first: (bin ^ (~value & 0x7f)) + 1 carries into
// bit 7 exactly when bin == value).
// `pairRows` holds sixteen 8-byte entries per tree, one per lane of a row of sixteen lanes: entry d < 8 the byte offset
// of level d's bucket in the tile (bucket * 128) and the xor byte four times, entry 8 + d the value added to each of the
// four bins (the byte four times) and 0. Levels past the tree's depth are zero (bucket 0, add 0: never true). A lane
// holds one entry of its group's tree, and the levels take their operands from the row's lanes by DPP (row_newbcast),
// which costs no instruction of its own: 512 bytes per pair over the vector memory path, where a packed row in every
// lane took 2 KB beside the 4 KB of leaf values, and an instruction per level fewer than unpacking it (two on a one-hot level). The wave
// publishes the trees' leaf values (1 << MAXD doubles per tree, a pair's side by side in `leaves`) in its own LDS
// region, one tree after the other: before the gathers the two groups swap half of their indexes, so that every lane
// has two documents of either tree (documents j * 64 + 2 * m + group, j = 0, 1), gathers them from the first tree's
// values, and the second tree's then go to the same place (LDS serves a wave's requests in order). With 2 KB per wave
// instead of a pair's 4 KB sixteen waves find room beside the widest tile instead of eight. That is what the kernel
// lacked: a wave issues an instruction about every nine cycles, and two waves per SIMD left half of the SIMD's issue
// cycles empty. 10M documents * 5000 trees of depth 8 over 1016 buckets, whole call with 10.3 ms of binarize: 57.1 ms with
// eight waves, 51.1 with sixteen, 49.4 with the rows by DPP, 46.9 with the tile in 16-byte pieces. What is left per pair
// and CU, of 115 cycles: vector issue 82, LDS about 78 (32 of them the values going in, 30 the gathers), vector memory 72
// (the values' 4 KB at 64 bytes a cycle): 128 documents share a copy of 256 values, and no wider tile fits.
// The tile of a workgroup that has its CU to itself arrives while nothing else runs there: it is read in 16-byte pieces,
// eight per thread in flight (two bytes a load from bins that do not start at such an address, or through `tileMap`).
// Waves take the pairs round robin; a last tree without a partner is done by wave 0 with both groups on the same tree
// and its values added once. Partial sums (one per wave) are added in a fixed order at the end. The fetches run
// kPairAhead rounds ahead of the walk without looking at the tree range: both tables end with kPairTreePadding trees'
// worth of zeros (a null tree's levels read row 0).
// With `tileMap` the tile has rowCount rows (MapTileBins) and the offsets in pairRows name rows, not buckets.
// The two halves of a block read the same lines of `bins`, two bytes of every four, so they go to workgroups of one
// XCD that start one after the other (workgroups go round-robin to the XCDs).
// grid = 2 * doc blocks, block = 64 * kPairWaves threads, dynamic LDS = rows * 128 (rounded up to 16) +
// kPairWaves * max(1 << MAXD, 128) * 8 bytes (the leaf regions, later the partial sums).
constexpr uint32_t kPairRowXorFlag = 1u << 23;  // slot 0 of a tree's row in registers: some level xors
constexpr int kPairRowDwords = 32;
constexpr int kPairWaves = 16;
constexpr int kPairAhead = 3;
constexpr int kPairTreePadding = 2 * kPairWaves * kPairAhead;

// Rows of a tile that splits the buckets of more than 127 values in two (`tileMap`, a dword per row: bits 0-15 the
// bucket, bits 16.. what becomes of its bins: 0 as they are, 1 min(bin, 127), 2 max(bin - 127, 0)), byte-parallel.
// A split "bin >= s" of such a bucket then reads the first row (s <= 127) or the second (with s - 127), and every
// level of the model is a 7-bit compare.
// A one-hot bucket of more than 127 values (bins 1 + index of the value) takes two rows as well: the bins up to 127
// as they are and 0 for the others (kTileMapOneHotLow), and bin - 127 for the bins from 128 on, 0 for the others
// (kTileMapHigh does exactly that); "bin == v" reads the first row for v <= 127 and the second, with v - 127,
// otherwise: both are 7-bit equalities against a value that is not 0.
constexpr uint32_t kTileMapLow = 1, kTileMapHigh = 2, kTileMapOneHotLow = 3;

__device__ __forceinline__ uint32_t MapTileBins(uint32_t bins4, uint32_t mode) {
    const uint32_t high = bins4 & 0x80808080u;  // bytes above 127
    if (mode == kTileMapLow) {
        return (bins4 | (high - (high >> 7))) & 0x7f7f7f7fu;
    }
    if (mode == kTileMapOneHotLow) {
        return bins4 & ~((high >> 7) * 0xffu);
    }
    if (mode == kTileMapHigh) {
        return ((bins4 & 0x7f7f7f7fu) + 0x01010101u) & ((high >> 7) * 0xffu);
    }
    return bins4;
}

// The rows of a tile with `tileMap` (MapTileBins), a wave per row, eight rows of a wave in flight; load(i) and
// store(row, bins) take the dword (or the half of it) that is the lane's.
template <int WAVES, typename TLoad, typename TStore>
__device__ __forceinline__ void CopyMappedRows(const uint32_t* __restrict__ tileMap, uint32_t rowCount, uint32_t wave,
                                               const TLoad& load, const TStore& store) {
    constexpr int kBatch = 8;
    for (uint32_t first = wave; first < rowCount; first += kBatch * WAVES) {
        uint32_t entry[kBatch], bins4[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            entry[j] = tileMap[min(first + j * WAVES, rowCount - 1)];  // past the end: the last row again, not stored
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            bins4[j] = load(entry[j] & 0xffffu);
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            if (first + j * WAVES < rowCount) {
                store(first + j * WAVES, MapTileBins(bins4[j], entry[j] >> 16));
            }
        }
    }
}

// The value that lane N of each row of sixteen lanes holds, in every lane of the row.
template <int N>
__device__ __forceinline__ uint32_t FromRowLane(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x150 + N, 0xf, 0xf, true));
}

// The walk of the pair-tile kernel, in two halves: the LDS reads of a tree's levels (laneOffset is the lane's offset
// inside a row of the tile, which starts at LDS address 0: the kernel has no other LDS), and the leaf indexes of four
// documents, one per byte, from what they returned. `row` is the lane's entry of pairRows.
// SIX: every bin of the tile is below 64. The even levels then carry the byte (64 - split), so that their result
// lands in bit 6 while the following level's lands in bit 7, and a pair of levels joins the index with one shift
// and two bit-field inserts (a one-hot level on an even position xors with the low six bits of its mask).
template <int MAXD, int D = 0>
__device__ __forceinline__ void ReadPairLevels(uint32_t laneOffset, uint32_t row, uint32_t (&a)[MAXD]) {
    if constexpr (D < MAXD) {
        a[D] = *reinterpret_cast<const __attribute__((address_space(3))) uint32_t*>(FromRowLane<D>(row) + laneOffset);
        ReadPairLevels<MAXD, D + 1>(laneOffset, row, a);
    }
}

template <int MAXD, int D = 0>
__device__ __forceinline__ void XorPairLevels(uint32_t xors, uint32_t (&a)[MAXD]) {
    if constexpr (D < MAXD) {
        a[D] ^= FromRowLane<D>(xors);
        XorPairLevels<MAXD, D + 1>(xors, a);
    }
}

template <int MAXD, int D = 0>
__device__ __forceinline__ void AddPairLevels(uint32_t adds, uint32_t (&a)[MAXD]) {
    if constexpr (D < MAXD) {
        a[D] += FromRowLane<8 + D>(adds);
        AddPairLevels<MAXD, D + 1>(adds, a);
    }
}

template <int MAXD, bool SIX>
__device__ __forceinline__ uint32_t WalkPairLevels(uint2 row, uint32_t (&r)[MAXD]) {
    if (__any(row.y != 0)) {
        XorPairLevels<MAXD>(row.y, r);
    }
    AddPairLevels<MAXD>(row.x, r);
    uint32_t idx4 = 0;
    if constexpr (SIX) {
        static_assert(MAXD % 2 == 0, "levels in pairs");
#pragma unroll
        for (int d = 0; d < MAXD; d += 2) {
            // bit 7 of the odd level, bit 6 of the even one; below them what is left of the even level's sum, which
            // only the first pair lets through: those six bits leave the byte with the shifts that follow (MAXD 8)
            // or end below the six bits that index the leaves (MAXD 6)
            const uint32_t pair = (r[d + 1] & 0x80808080u) | (r[d] & 0x7f7f7f7fu);
            idx4 = d == 0 ? pair : (pair & 0xc0c0c0c0u) | ((idx4 >> 2) & 0x3f3f3f3fu);
        }
    } else {
#pragma unroll
        for (int d = 0; d < MAXD; ++d) {
            idx4 = (r[d] & 0x80808080u) | (idx4 >> 1);
        }
    }
    return idx4;
}

template <bool XOR, int MAXD>
__device__ __forceinline__ uint32_t PairTreeIndexes(const uint8_t* laneTile, const uint4 (&desc)[4]) {
    const uint32_t offs[8] = {desc[0].x, desc[0].y, desc[0].z, desc[0].w, desc[1].x, desc[1].y, desc[1].z, desc[1].w};
    const uint32_t adds[8] = {desc[2].x, desc[2].y, desc[2].z, desc[2].w, desc[3].x, desc[3].y, desc[3].z, desc[3].w};
    uint32_t a[MAXD];
#pragma unroll
    for (int d = 0; d < MAXD; ++d) {
        // rows of trees that never xor hold the plain offset
        a[d] = *reinterpret_cast<const uint32_t*>(laneTile + (XOR ? offs[d] & 0x007fffffu : offs[d]));
    }
    // one wait for the eight reads instead of one per read: LDS returns them in order a few cycles apart, and
    // every wait takes an issue slot (lgkmcnt 0, the other counters untouched)
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_sched_barrier(0);
    uint32_t idx4 = 0;
#pragma unroll
    for (int d = 0; d < MAXD; ++d) {
        uint32_t v = a[d];
        if (XOR) {
            v ^= __builtin_amdgcn_perm(offs[d], offs[d], 0x03030303u);  // the xor byte four times
        }
        // the level's four result bits go to bit 7 of the bytes; earlier levels move down one bit and never
        // reach the byte below within eight levels
        idx4 = ((v + adds[d]) & 0x80808080u) | (idx4 >> 1);
    }
    return idx4;
}

template <int MAXD, bool SIX>
__global__ __launch_bounds__(64 * kPairWaves) void EvalObliviousPairTileKernel(
    const uint16_t* __restrict__ bins, size_t docCount, uint32_t bucketCount, const uint32_t* __restrict__ tileMap,
    uint32_t rowCount, const uint2* __restrict__ pairRows, const double2* __restrict__ leaves2,
    const double* __restrict__ bias, double scale, uint32_t treeBegin, uint32_t treeEnd, double* __restrict__ out) {
    constexpr uint32_t kLeaves = 1u << MAXD;
    constexpr int kLeafRegs = MAXD == 8 ? 4 : 1;       // 16-byte pieces of a pair's 2 * kLeaves leaf values per lane
    constexpr int kPublishRegs = MAXD == 8 ? 2 : 1;    // pieces that go to LDS at a time: one tree's, or both trees'
    constexpr uint32_t kRegion = MAXD == 8 ? kLeaves : 2 * kLeaves;  // doubles of a wave's region
    static_assert(MAXD == 8 || MAXD == 6, "64 or 256 leaves per tree");
    // s_waitcnt for the level reads and, issued before them, the last round's gathers: only the stores behind them
    // stay under way (lgkmcnt in bits 8-11; vmcnt and expcnt untouched)
    constexpr int kWaitForLevelReads = 0xc07f | (kPublishRegs << 8);
    extern __shared__ uint32_t sTile[];
    uint16_t* sTile16 = reinterpret_cast<uint16_t*>(sTile);
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    // sixteen workgroups take eight blocks, one per XCD, their first halves before their second ones; the blocks of a
    // last group that is not full come half by half
    const uint32_t turn = blockIdx.x / (2 * kXcdCount), inTurn = blockIdx.x % (2 * kXcdCount);
    const bool wholeTurn = gridDim.x - turn * (2 * kXcdCount) >= 2 * kXcdCount;
    const size_t block = turn * kXcdCount + (wholeTurn ? inTurn % kXcdCount : inTurn >> 1);
    const uint32_t half = wholeTurn ? inTurn / kXcdCount : inTurn & 1;
    const uint32_t tileWords = rowCount * kWave;  // rowCount = bucketCount without a map
    const uint16_t* src = bins + block * (bucketCount * kWave) * 2 + half;
    const uint32_t group = lane >> 5;
    const uint32_t tileBytes = (tileWords * 2 + 15) & ~15u;
    double* leafArea = reinterpret_cast<double*>(reinterpret_cast<uint8_t*>(sTile) + tileBytes);
    double2* sLeafWave2 = reinterpret_cast<double2*>(leafArea + wave * kRegion) + lane;
    // LDS addresses of the first and the second tree's values
    const uint32_t leafFirst = tileBytes + wave * kRegion * 8, leafSecond = leafFirst + (MAXD == 8 ? 0 : kLeaves * 8);
    const uint32_t laneOffset = (lane & 31) * 4;
    const uint32_t treeCount = treeEnd - treeBegin;
    const uint32_t pairCount = treeCount / 2;
    double acc[2] = {0.0, 0.0};
    constexpr int kAhead = kPairAhead;
    uint2 rows[kAhead];
    double2 pref[kAhead][kLeafRegs];
    // what a lane fetches of the pair that starts at tree `first`: its entry of its group's row and its pieces of
    // the two trees' leaf values
    const uint2* myRows = pairRows + group * 16 + (lane & 15);
    const double2* myLeaves = leaves2 + lane;
#define CBAMD_FETCH_PAIR(k, first)                                                                 \
    do {                                                                                           \
        rows[k] = myRows[static_cast<size_t>(first) * 16];                                         \
        /* the row first: its levels are read before the leaf values go to LDS */                 \
        __builtin_amdgcn_sched_barrier(0);                                                         \
        const double2* values = myLeaves + static_cast<size_t>(first) * (kLeaves / 2);             \
        _Pragma("unroll") for (int i = 0; i < kLeafRegs; ++i) {                                    \
            pref[k][i] = values[i * kWave];                                                        \
        }                                                                                          \
        __builtin_amdgcn_sched_barrier(0);                                                         \
    } while (0)
    uint32_t p = wave;
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
        // (written before the loads so that the arrays stay in registers)
#pragma unroll
        for (int i = 0; i < kLeafRegs; ++i) {
            pref[k][i] = {0.0, 0.0};
        }
        CBAMD_FETCH_PAIR(k, treeBegin + 2 * (p + k * kPairWaves));
    }
    // the tile, behind the requests for the first pairs
    if (tileMap == nullptr && (reinterpret_cast<uintptr_t>(bins) & 15) == 0) {
        const uint4* src4 = reinterpret_cast<const uint4*>(src - half);
        const uint32_t select = half ? 0x07060302u : 0x05040100u;  // the upper or the lower halves of two dwords
        CopyInBatches<64 * kPairWaves>(src4, tileWords / 4, tid, [&](uint32_t i, const uint4& v) {
            reinterpret_cast<uint2*>(sTile)[i] = make_uint2(__builtin_amdgcn_perm(v.y, v.x, select), __builtin_amdgcn_perm(v.w, v.z, select));
        });
    } else if (tileMap == nullptr) {
        for (uint32_t i = tid; i < tileWords; i += 64 * kPairWaves) {
            sTile16[i] = src[2 * i];
        }
    } else {
        CopyMappedRows<kPairWaves>(
            tileMap, rowCount, wave, [&](uint32_t bucket) { return uint32_t(src[2 * (bucket * kWave + lane)]); },
            [&](uint32_t row, uint32_t bins2) { sTile16[row * kWave + lane] = static_cast<uint16_t>(bins2); });
    }
    __syncthreads();  // tile is loaded

    // pieces of the pair's leaf values into the wave's LDS region: gathers of what it held were issued before these
    // stores, and LDS serves one wave's requests in order
#define CBAMD_PUBLISH(k, begin)                                                                    \
    do {                                                                                           \
        __builtin_amdgcn_wave_barrier();                                                           \
        _Pragma("unroll") for (int i = 0; i < kPublishRegs; ++i) {                                 \
            sLeafWave2[i * kWave] = pref[k][(begin) + i];                                          \
        }                                                                                          \
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");                                     \
        __builtin_amdgcn_wave_barrier();                                                           \
    } while (0)
    // The indexes of the pair, four documents of its group's tree per lane, then two documents of either tree:
    // first and second tree's in the low sixteen bits of idxA and idxB.
#define CBAMD_WALK(k, levelBins, idxA, idxB)                                                       \
    do {                                                                                           \
        uint32_t idx4 = WalkPairLevels<MAXD, SIX>(rows[k], levelBins);                             \
        if constexpr (MAXD == 6) {                                                                 \
            idx4 &= 0xfcfcfcfcu;                                                                   \
        }                                                                                          \
        const auto swapped = __builtin_amdgcn_permlane32_swap(idx4, idx4 >> 16, false, false);     \
        idxA = swapped[0];                                                                         \
        idxB = swapped[1];                                                                         \
    } while (0)
    // the leaf value that byte j of idx names: eight times its index (two times the byte with 64 leaves, whose index is
    // in the upper six bits) and the values' address in one instruction
#define CBAMD_LEAF(base, idx, j)                                                                   \
    (*reinterpret_cast<const __attribute__((address_space(3))) double*>(                           \
        __builtin_amdgcn_udot4(idx, (MAXD == 8 ? 8u : 2u) << (8 * (j)), base, false)))

    // One round of a wave: the leaf values that the previous round gathered are added once this round's level reads,
    // issued behind them, have returned; the gathers go out last, and the registers of this pair take the pair kAhead
    // rounds ahead.
    double gathered[2][2] = {{0.0, 0.0}, {0.0, 0.0}};
#define CBAMD_PAIR_ROUND(k)                                                                        \
    do {                                                                                           \
        uint32_t levelBins[MAXD], idxA, idxB;                                                      \
        ReadPairLevels<MAXD>(laneOffset, rows[k].x, levelBins);                                    \
        __builtin_amdgcn_sched_barrier(0);                                                         \
        CBAMD_PUBLISH(k, 0);                                                                       \
        __builtin_amdgcn_sched_barrier(0);                                                         \
        __builtin_amdgcn_s_waitcnt(kWaitForLevelReads);                                            \
        __builtin_amdgcn_sched_barrier(0);                                                         \
        _Pragma("unroll") for (int j = 0; j < 2; ++j) {                                            \
            acc[j] = __dadd_rn(__dadd_rn(acc[j], gathered[0][j]), gathered[1][j]);                 \
        }                                                                                          \
        CBAMD_WALK(k, levelBins, idxA, idxB);                                                      \
        _Pragma("unroll") for (int j = 0; j < 2; ++j) {                                            \
            gathered[0][j] = CBAMD_LEAF(leafFirst, idxA, j);                                       \
        }                                                                                          \
        if constexpr (MAXD == 8) {                                                                 \
            CBAMD_PUBLISH(k, kLeafRegs / 2);                                                       \
        }                                                                                          \
        _Pragma("unroll") for (int j = 0; j < 2; ++j) {                                            \
            gathered[1][j] = CBAMD_LEAF(leafSecond, idxB, j);                                      \
        }                                                                                          \
        __builtin_amdgcn_sched_barrier(0);                                                         \
        CBAMD_FETCH_PAIR(k, treeBegin + 2 * (p + kAhead * kPairWaves));                            \
        p += kPairWaves;                                                                           \
    } while (0)

    static_assert(kAhead == 3, "the rounds below are written out for three register sets");
    // whole turns of the three register sets without a branch between the rounds, so that the waits for
    // the loads count only the loads that are older than the one needed
    while (p + 2 * kPairWaves < pairCount) {
        CBAMD_PAIR_ROUND(0);
        CBAMD_PAIR_ROUND(1);
        CBAMD_PAIR_ROUND(2);
    }
    if (p < pairCount) {
        CBAMD_PAIR_ROUND(0);
        if (p < pairCount) {
            CBAMD_PAIR_ROUND(1);
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        acc[j] = __dadd_rn(__dadd_rn(acc[j], gathered[0][j]), gathered[1][j]);
    }
    if ((treeCount & 1) && wave == 0) {
        // the last tree has no partner: both groups walk it (its row and its leaf values, twice with 64 leaves)
        rows[0] = pairRows[static_cast<size_t>(treeEnd - 1) * 16 + (lane & 15)];
        const double2* values = leaves2 + static_cast<size_t>(treeEnd - 1) * (kLeaves / 2);
#pragma unroll
        for (int i = 0; i < kPublishRegs; ++i) {
            pref[0][i] = values[(i * kWave + lane) & (kLeaves / 2 - 1)];
        }
        uint32_t levelBins[MAXD], idxA, idxB;
        ReadPairLevels<MAXD>(laneOffset, rows[0].x, levelBins);
        CBAMD_PUBLISH(0, 0);
        CBAMD_WALK(0, levelBins, idxA, idxB);
        static_cast<void>(idxB);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            acc[j] = __dadd_rn(acc[j], CBAMD_LEAF(leafFirst, idxA, j));
        }
    }
#undef CBAMD_PAIR_ROUND
#undef CBAMD_FETCH_PAIR
#undef CBAMD_PUBLISH
#undef CBAMD_WALK
#undef CBAMD_LEAF
    __syncthreads();  // every wave is through with its leaf region: the area now takes the partial sums
    // partial sums as [wave][document of the tile], then one thread per document adds the sixteen
    double* sRed = leafArea;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        sRed[wave * 128 + j * kWave + 2 * (lane & 31) + group] = acc[j];
    }
    __syncthreads();
    if (tid < 128) {
        double sum = sRed[tid];
#pragma unroll
        for (int part = 1; part < kPairWaves; ++part) {
            sum = __dadd_rn(sum, sRed[part * 128 + tid]);
        }
        const size_t doc = block * kDocsPerBlock + (2 * half + (tid >> 6)) * kWave + (tid & 63);
        if (doc < docCount) {
            out[doc] = Finish(sum, scale, bias[0], treeBegin == 0);
        }
    }
}

// The same with four trees per wave on a quarter of a block, for models whose rows do not fit the half tile: the
// tile holds the bins of 64 documents (documents quarter * 64 + l of the block in byte l of a row), lanes 16 g ..
// 16 g + 15 walk tree g of a quad of trees, each lane for the four documents of one dword. The rows are
// sixteen dwords per tree in every lane of its group: slot d the byte offset of level d's bucket (bucket * 64) | xor byte
// << 24, slot 8 + d the value added to the bins, slot 0 also kPairRowXorFlag. Rows and leaf values are fetched three rounds ahead, so both tables end with
// kQuadTreePadding null trees.
// WAVES = 8, or 4 when the rows leave LDS for four waves' regions only.
// grid = 4 * doc blocks, block = 64 * WAVES threads, dynamic LDS = rows * 64 (rounded up to 16) +
// WAVES * 4 * (1 << MAXD) * 8 bytes (the leaf regions, later the partial sums).
constexpr int kQuadTreePadding = 4 * kTileWaves * kPairAhead;
static_assert(kPairTreePadding <= kQuadTreePadding, "the tables of the two kernels are padded alike");

template <int MAXD, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void EvalObliviousQuadTileKernel(
    const uint8_t* __restrict__ bins, size_t docCount, uint32_t bucketCount, const uint32_t* __restrict__ tileMap,
    uint32_t rowCount, const uint4* __restrict__ pairRows, const double2* __restrict__ leaves2,
    const double* __restrict__ bias, double scale, uint32_t treeBegin, uint32_t treeEnd, double* __restrict__ out) {
    constexpr uint32_t kLeaves = 1u << MAXD;
    constexpr int kLeafRegs = MAXD == 8 ? 8 : 2;  // 16-byte pieces of a quad's 4 * kLeaves leaf values per lane
    static_assert(MAXD == 8 || MAXD == 6, "64 or 256 leaves per tree");
    extern __shared__ uint32_t sTile[];
    uint8_t* sTile8 = reinterpret_cast<uint8_t*>(sTile);
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const size_t block = blockIdx.x >> 2;
    const uint32_t quarter = blockIdx.x & 3;
    const uint32_t tileBytesUsed = rowCount * kWave;  // rowCount = bucketCount without a map
    const uint8_t* src = bins + block * (bucketCount * kWave) * 4 + quarter;
    if (tileMap == nullptr) {
        for (uint32_t i = tid; i < tileBytesUsed; i += 64 * WAVES) {
            sTile8[i] = src[4 * i];
        }
    } else {
        for (uint32_t row = wave; row < rowCount; row += WAVES) {
            const uint32_t entry = tileMap[row];
            const uint32_t bin = src[4 * ((entry & 0xffffu) * kWave + lane)];
            sTile8[row * kWave + lane] = static_cast<uint8_t>(MapTileBins(bin, entry >> 16));
        }
    }
    const uint32_t group = lane >> 4;
    const uint32_t tileBytes = (tileBytesUsed + 15) & ~15u;
    double* leafArea = reinterpret_cast<double*>(reinterpret_cast<uint8_t*>(sTile) + tileBytes);
    double2* sLeafWave2 = reinterpret_cast<double2*>(leafArea + wave * 4 * kLeaves);
    const double* sLeafMine = leafArea + wave * 4 * kLeaves + group * kLeaves;
    const uint8_t* laneTile = reinterpret_cast<const uint8_t*>(sTile) + (lane & 15) * 4;
    __syncthreads();  // tile is loaded

    const uint32_t treeCount = treeEnd - treeBegin;
    const uint32_t pairCount = treeCount / 4;  // whole quads of trees
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    constexpr int kAhead = kPairAhead;
    uint4 rows[kAhead][4];
    double2 pref[kAhead][kLeafRegs];
    // what a lane fetches of the quad that starts at tree `first`: its group's row and its pieces of the
    // four trees' leaf values
    const uint4* myRows = pairRows + group * 4;
    const double2* myLeaves = leaves2 + lane;
#define CBAMD_FETCH_PAIR(k, first)                                                                 \
    do {                                                                                           \
        const uint4* row = myRows + static_cast<size_t>(first) * 4;                                \
        _Pragma("unroll") for (int i = 0; i < 4; ++i) {                                            \
            rows[k][i] = row[i];                                                                   \
        }                                                                                          \
        const double2* values = myLeaves + static_cast<size_t>(first) * (kLeaves / 2);             \
        _Pragma("unroll") for (int i = 0; i < kLeafRegs; ++i) {                                    \
            pref[k][i] = values[i * kWave];                                                        \
        }                                                                                          \
    } while (0)
    // the quad's leaf values into the wave's LDS region (the previous quad's gathers were issued before these
    // stores and LDS serves one wave's requests in order), then the levels: four leaf indexes per lane
#define CBAMD_PUBLISH_AND_WALK(k, idx4)                                                            \
    do {                                                                                           \
        _Pragma("unroll") for (int i = 0; i < kLeafRegs; ++i) {                                    \
            sLeafWave2[i * kWave + lane] = pref[k][i];                                             \
        }                                                                                          \
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");                                     \
        __builtin_amdgcn_wave_barrier();                                                           \
        const uint32_t flags =                                                                     \
            __builtin_amdgcn_readlane(rows[k][0].x, 0) | __builtin_amdgcn_readlane(rows[k][0].x, 16) | \
            __builtin_amdgcn_readlane(rows[k][0].x, 32) | __builtin_amdgcn_readlane(rows[k][0].x, 48); \
        if (flags & kPairRowXorFlag) {                                                             \
            idx4 = PairTreeIndexes<true, MAXD>(laneTile, rows[k]);                                 \
        } else {                                                                                   \
            idx4 = PairTreeIndexes<false, MAXD>(laneTile, rows[k]);                                \
        }                                                                                          \
    } while (0)

    // One round of a wave: the leaf values that the previous round gathered are added while this round's LDS
    // reads are under way; the registers of this quad take the quad kAhead rounds ahead as soon as every level
    // has read them (the loads then land in those registers), and the gathers go out last.
    constexpr int kLoadsBehind = 2 * (4 + kLeafRegs);
    constexpr int kWaitLoads = 0x0f70 | (kLoadsBehind & 15) | ((kLoadsBehind >> 4) << 14);  // vmcnt(kLoadsBehind)
    double gathered[4] = {0.0, 0.0, 0.0, 0.0};
#define CBAMD_PAIR_ROUND(k)                                                                        \
    do {                                                                                           \
        uint32_t idx4;                                                                             \
        /* one wait for this quad's loads: those of the two quads behind it stay in flight */       \
        __builtin_amdgcn_s_waitcnt(kWaitLoads);                                                    \
        __builtin_amdgcn_sched_barrier(0);                                                         \
        CBAMD_PUBLISH_AND_WALK(k, idx4);                                                           \
        _Pragma("unroll") for (int q = 0; q < 4; ++q) {                                            \
            acc[q] = __dadd_rn(acc[q], gathered[q]);                                               \
        }                                                                                          \
        __builtin_amdgcn_sched_barrier(0);                                                         \
        CBAMD_FETCH_PAIR(k, treeBegin + 4 * (p + kAhead * WAVES));                            \
        __builtin_amdgcn_sched_barrier(0);                                                         \
        _Pragma("unroll") for (int q = 0; q < 4; ++q) {                                            \
            gathered[q] = sLeafMine[(idx4 >> (8 * q + 8 - MAXD)) & (kLeaves - 1)];                 \
        }                                                                                          \
        __builtin_amdgcn_wave_barrier();                                                           \
        p += WAVES;                                                                           \
    } while (0)

    uint32_t p = wave;
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
        // (written before the loads so that the arrays stay in registers)
#pragma unroll
        for (int i = 0; i < kLeafRegs; ++i) {
            pref[k][i] = {0.0, 0.0};
        }
        CBAMD_FETCH_PAIR(k, treeBegin + 4 * (p + k * WAVES));
    }
    static_assert(kAhead == 3, "the rounds below are written out for three register sets");
    // whole turns of the three register sets without a branch between the rounds, so that the waits for
    // the loads count only the loads that are older than the one needed
    while (p + 2 * WAVES < pairCount) {
        CBAMD_PAIR_ROUND(0);
        CBAMD_PAIR_ROUND(1);
        CBAMD_PAIR_ROUND(2);
    }
    if (p < pairCount) {
        CBAMD_PAIR_ROUND(0);
        if (p < pairCount) {
            CBAMD_PAIR_ROUND(1);
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        acc[q] = __dadd_rn(acc[q], gathered[q]);
    }
    const uint32_t rest = treeCount & 3;
    if (rest && wave == 0) {
        // the last one to three trees: a group without a tree of its own walks the last one and adds nothing
        const uint32_t base = treeEnd - rest;
        const uint4* row = pairRows + static_cast<size_t>(base + min(group, rest - 1)) * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            rows[0][i] = row[i];
        }
#pragma unroll
        for (int i = 0; i < kLeafRegs; ++i) {
            const uint32_t piece = i * kWave + lane;  // of the four trees' regions, kLeaves / 2 pieces each
            const uint32_t tree = base + min(piece / (kLeaves / 2), rest - 1);
            pref[0][i] = leaves2[static_cast<size_t>(tree) * (kLeaves / 2) + piece % (kLeaves / 2)];
        }
        uint32_t idx4;
        CBAMD_PUBLISH_AND_WALK(0, idx4);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double v = sLeafMine[(idx4 >> (8 * q + 8 - MAXD)) & (kLeaves - 1)];
            acc[q] = __dadd_rn(acc[q], group < rest ? v : 0.0);
        }
        __builtin_amdgcn_wave_barrier();
    }
#undef CBAMD_PAIR_ROUND
#undef CBAMD_FETCH_PAIR
#undef CBAMD_PUBLISH_AND_WALK
    __syncthreads();  // every wave is through with its leaf region: the area now takes the partial sums
    // partial sums as [wave][group][document of the tile], then one thread per document adds the thirty-two
    double* sRed = leafArea;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        // byte q of a lane's dword: document 4 * (lane & 15) + q of the tile
        sRed[(wave * 4 + group) * kWave + 4 * (lane & 15) + q] = acc[q];
    }
    __syncthreads();
    if (tid < kWave) {
        double sum = sRed[tid];
#pragma unroll
        for (int part = 1; part < 4 * WAVES; ++part) {
            sum = __dadd_rn(sum, sRed[part * kWave + tid]);
        }
        const size_t doc = block * kDocsPerBlock + quarter * kWave + tid;
        if (doc < docCount) {
            out[doc] = Finish(sum, scale, bias[0], treeBegin == 0);
        }
    }
}

// Models of 7-bit bins whose 256-document tile fits LDS, one tree per wave: the walk of
// EvalObliviousPairTileKernel on the whole tile. A tree's row is `tileRows` (the quad-tile kernel's format with
// bucket * 256 as the byte offset); its address is the same in every lane, so it comes through scalar loads
// and a level is an LDS read and three vector instructions with no lane reads and no scalar arithmetic. The
// leaf values go through the wave's LDS region; rows and values are fetched kPairAhead rounds ahead without
// looking at the tree range (both tables end with kRowTilePadding trees' worth of zeros). Waves take the trees
// round robin; their partial sums are added in wave order through an accumulator in LDS at the end.
// Leaf values: one dimension: (1 << MAXD) values per tree. Several dimensions: a workgroup sums DIMS (2 or 4)
// of them at a time, slice after slice of the model's dimensions over the same tile, every slice with another
// walk of the trees; `leaves2` is [slice][tree][piece][leaf] pairs of values (16 bytes: dimensions 2 * piece and
// 2 * piece + 1 of the slice, zeros past the model's last dimension), sliceStride pairs per slice. A wave's
// 16-byte gathers of one piece then spread over all groups of four LDS banks, which leaf rows of 32 bytes would
// not.
// With `tileMap` the tile has rowCount rows (MapTileBins) and the offsets in tileRows name rows, not buckets.
// grid = doc blocks, block = 64 * WAVES, dynamic LDS = rows * 256 (rounded up to 16) + 256 * DIMS * 8 (the
// accumulator) + WAVES * (1 << MAXD) * DIMS * 8 bytes (the leaf regions).
constexpr int kRowTilePadding = kWideTileWaves * kPairAhead;
static_assert(kRowTilePadding <= kPairTreePadding, "the two kernels share the padded leaf table");

template <int MAXD, int WAVES, int DIMS>
__global__ __launch_bounds__(64 * WAVES) void EvalObliviousRowTileKernel(
    const uint32_t* __restrict__ bins, size_t docCount, uint32_t bucketCount, const uint32_t* __restrict__ tileMap,
    uint32_t rowCount, const uint4* __restrict__ tileRows, const double2* __restrict__ leaves2,
    const double* __restrict__ bias, double scale, uint32_t dim, size_t sliceStride, uint32_t treeBegin,
    uint32_t treeEnd, double* __restrict__ out) {
    constexpr uint32_t kLeaves = 1u << MAXD;
    constexpr uint32_t kTreePieces = kLeaves * DIMS / 2;     // 16-byte pieces of a tree's leaf values (of a slice)
    constexpr int kLeafRegs = kTreePieces > kWave ? static_cast<int>(kTreePieces / kWave) : 1;
    constexpr uint32_t kPieceMask = kTreePieces - 1;         // 32 pieces: the upper lanes repeat the lower lanes' pieces
    constexpr int kPairsPerLeaf = DIMS > 1 ? DIMS / 2 : 1;
    constexpr bool kPipelined = DIMS <= 2;  // the values gathered in a round are added during the next one
    static_assert(MAXD == 8 || MAXD == 6, "64 or 256 leaves per tree");
    static_assert(DIMS == 1 || DIMS == 2 || DIMS == 4, "one value or whole pairs per leaf");
    static_assert(WAVES <= kWideTileWaves, "the tables are padded for that many waves");
    extern __shared__ uint32_t sTile[];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const size_t block = blockIdx.x;
    const uint32_t tileDwords = rowCount * kWave;  // rowCount = bucketCount without a map
    const uint32_t* src = bins + block * (bucketCount * kWave);
    if (tileMap == nullptr) {
        CopyTile<64 * WAVES>(src, rowCount, tid, sTile);
    } else {
        CopyMappedRows<WAVES>(
            tileMap, rowCount, wave, [&](uint32_t bucket) { return src[bucket * kWave + lane]; },
            [&](uint32_t row, uint32_t bins4) { sTile[row * kWave + lane] = bins4; });
    }
    const uint32_t tileBytes = (tileDwords * 4 + 15) & ~15u;
    double* sRed = reinterpret_cast<double*>(reinterpret_cast<uint8_t*>(sTile) + tileBytes);  // [DIMS][256 documents]
    double* leafArea = sRed + kDocsPerBlock * DIMS;
    double2* sLeafWave2 = reinterpret_cast<double2*>(leafArea + wave * kLeaves * DIMS);
    const double* sLeafMine = leafArea + wave * kLeaves * DIMS;
    const uint8_t* laneTile = reinterpret_cast<const uint8_t*>(sTile) + lane * 4;
    const uint32_t treeCount = treeEnd - treeBegin;
    constexpr int kAhead = kPairAhead;
    static_assert(kAhead == 3, "the rounds below are written out for three register sets");

#define CBAMD_FETCH_TREE(k, tree)                                                                  \
    do {                                                                                           \
        const uint4* row = tileRows + static_cast<size_t>(tree) * 4;                               \
        _Pragma("unroll") for (int i = 0; i < 4; ++i) {                                            \
            rows[k][i] = row[i];                                                                   \
        }                                                                                          \
        const double2* values = myLeaves + static_cast<size_t>(tree) * kTreePieces;                \
        _Pragma("unroll") for (int i = 0; i < kLeafRegs; ++i) {                                    \
            pref[k][i] = values[i * kWave];                                                        \
        }                                                                                          \
    } while (0)
    // the tree's leaf values into the wave's LDS region (the previous tree's gathers were issued before these
    // stores and LDS serves one wave's requests in order), then the levels: four leaf indexes per lane
#define CBAMD_PUBLISH_AND_WALK(k, idx4)                                                            \
    do {                                                                                           \
        _Pragma("unroll") for (int i = 0; i < kLeafRegs; ++i) {                                    \
            sLeafWave2[(i * kWave + lane) & kPieceMask] = pref[k][i];                              \
        }                                                                                          \
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");                                     \
        __builtin_amdgcn_wave_barrier();                                                           \
        if (__builtin_amdgcn_readfirstlane(rows[k][0].x) & kPairRowXorFlag) {                      \
            idx4 = PairTreeIndexes<true, MAXD>(laneTile, rows[k]);                                 \
        } else {                                                                                   \
            idx4 = PairTreeIndexes<false, MAXD>(laneTile, rows[k]);                                \
        }                                                                                          \
    } while (0)
    // One round of a wave, as in the two-tree kernel: the values that the previous round gathered are added
    // while this round's LDS reads are under way, the registers of this tree take the tree kAhead rounds ahead
    // as soon as every level has read them, and the gathers go out last.
    constexpr int kLoadsBehind = 2 * kLeafRegs;  // vector loads of the two rounds behind the one that is waited for
    constexpr int kWaitLoads = 0x0f70 | (kLoadsBehind & 15) | ((kLoadsBehind >> 4) << 14);  // vmcnt(kLoadsBehind)
#define CBAMD_TREE_ROUND(k)                                                                        \
    do {                                                                                           \
        uint32_t idx4;                                                                             \
        __builtin_amdgcn_s_waitcnt(kWaitLoads);                                                    \
        __builtin_amdgcn_sched_barrier(0);                                                         \
        CBAMD_PUBLISH_AND_WALK(k, idx4);                                                           \
        if constexpr (kPipelined) {                                                                \
            _Pragma("unroll") for (int q = 0; q < 4; ++q) {                                        \
                _Pragma("unroll") for (int c = 0; c < DIMS; ++c) {                                 \
                    acc[q][c] = __dadd_rn(acc[q][c], gathered[q][c]);                              \
                }                                                                                  \
            }                                                                                      \
        }                                                                                          \
        __builtin_amdgcn_sched_barrier(0);                                                         \
        CBAMD_FETCH_TREE(k, treeBegin + p + kAhead * WAVES);                                       \
        __builtin_amdgcn_sched_barrier(0);                                                         \
        _Pragma("unroll") for (int q = 0; q < 4; ++q) {                                            \
            const uint32_t leaf = (idx4 >> (8 * q + 8 - MAXD)) & (kLeaves - 1);                    \
            if constexpr (DIMS == 1) {                                                             \
                gathered[q][0] = sLeafMine[leaf];                                                  \
            } else {                                                                               \
                _Pragma("unroll") for (int piece = 0; piece < kPairsPerLeaf; ++piece) {            \
                    const double2 pair = reinterpret_cast<const double2*>(sLeafMine)[piece * kLeaves + leaf]; \
                    gathered[q][2 * piece] = pair.x;                                               \
                    gathered[q][2 * piece + 1] = pair.y;                                           \
                }                                                                                  \
            }                                                                                      \
        }                                                                                          \
        if constexpr (!kPipelined) {                                                               \
            /* four dimensions: no registers for values in flight across a round */               \
            _Pragma("unroll") for (int q = 0; q < 4; ++q) {                                        \
                _Pragma("unroll") for (int c = 0; c < DIMS; ++c) {                                 \
                    acc[q][c] = __dadd_rn(acc[q][c], gathered[q][c]);                              \
                    gathered[q][c] = 0.0;                                                          \
                }                                                                                  \
            }                                                                                      \
        }                                                                                          \
        __builtin_amdgcn_wave_barrier();                                                           \
        p += WAVES;                                                                                \
    } while (0)

    const uint32_t slices = (dim + DIMS - 1) / DIMS;
    for (uint32_t slice = 0; slice < slices; ++slice) {
        __syncthreads();  // tile is loaded / the previous slice's accumulator has been read
        double acc[4][DIMS], gathered[4][DIMS];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int c = 0; c < DIMS; ++c) {
                acc[q][c] = 0.0;
                gathered[q][c] = 0.0;
            }
        }
        uint4 rows[kAhead][4];
        double2 pref[kAhead][kLeafRegs];
        const double2* myLeaves = leaves2 + slice * sliceStride + (lane & kPieceMask);
        uint32_t p = wave;
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            // (written before the loads so that the arrays stay in registers)
#pragma unroll
            for (int i = 0; i < kLeafRegs; ++i) {
                pref[k][i] = {0.0, 0.0};
            }
            CBAMD_FETCH_TREE(k, treeBegin + p + k * WAVES);
        }
        // whole turns of the three register sets without a branch between the rounds, so that the waits for
        // the loads count only the loads that are older than the one needed
        while (p + 2 * WAVES < treeCount) {
            CBAMD_TREE_ROUND(0);
            CBAMD_TREE_ROUND(1);
            CBAMD_TREE_ROUND(2);
        }
        if (p < treeCount) {
            CBAMD_TREE_ROUND(0);
            if (p < treeCount) {
                CBAMD_TREE_ROUND(1);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int c = 0; c < DIMS; ++c) {
                acc[q][c] = __dadd_rn(acc[q][c], gathered[q][c]);
            }
        }
        // waves add their partial sums in wave order into the LDS accumulator; the last wave finishes the values
        // and writes them out (byte q of a lane's dword: document q * 64 + lane)
        for (uint32_t w = 0; w + 1 < WAVES; ++w) {
            if (wave == w) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
#pragma unroll
                    for (int c = 0; c < DIMS; ++c) {
                        double* cell = sRed + c * kDocsPerBlock + q * kWave + lane;
                        *cell = (w == 0) ? acc[q][c] : __dadd_rn(*cell, acc[q][c]);
                    }
                }
            }
            __syncthreads();
        }
        if (wave == WAVES - 1) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const size_t doc = block * kDocsPerBlock + q * kWave + lane;
#pragma unroll
                for (int c = 0; c < DIMS; ++c) {
                    const uint32_t d = slice * DIMS + c;
                    if (doc < docCount && d < dim) {
                        const double sum = __dadd_rn(sRed[c * kDocsPerBlock + q * kWave + lane], acc[q][c]);
                        out[doc * dim + d] = Finish(sum, scale, bias[d], treeBegin == 0);
                    }
                }
            }
        }
    }
#undef CBAMD_TREE_ROUND
#undef CBAMD_FETCH_TREE
#undef CBAMD_PUBLISH_AND_WALK
}

// One-dimensional models of depth 9 to 16 on the same tile, one tree per wave: the walk of the row-tile kernel
// in two halves. `deepRows` holds 32 dwords per tree: the first sixteen as in tileRows for the levels 0..7, the
// second sixteen for the levels 8..8 + HIGH - 1 (levels past the tree's depth: row 0, add 0, never true; the
// flag of slot 0 says whether any level of the tree xors). The two halves give a byte per document each,
// together the leaf index; a tree's table has up to 512 KB, so the leaf values are gathered from global memory,
// `leaves` + firstLeaf[tree], and added one round later. Rows come two rounds ahead (scalar loads: the address
// is the same in every lane). Both tables end with kRowTilePadding null trees.
// grid = doc blocks, block = 64 * WAVES, dynamic LDS = rows * 256 (rounded up to 16) + 256 * 8 bytes.
template <int HIGH, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void EvalObliviousDeepTileKernel(
    const uint32_t* __restrict__ bins, size_t docCount, uint32_t bucketCount, const uint32_t* __restrict__ tileMap,
    uint32_t rowCount, const uint4* __restrict__ deepRows, const uint32_t* __restrict__ firstLeaf,
    const double* __restrict__ leaves, const double* __restrict__ bias, double scale, uint32_t treeBegin,
    uint32_t treeEnd, double* __restrict__ out) {
    static_assert(HIGH == 4 || HIGH == 8, "levels 8..11 or 8..15 in the second half");
    extern __shared__ uint32_t sTile[];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const size_t block = blockIdx.x;
    const uint32_t tileDwords = rowCount * kWave;  // rowCount = bucketCount without a map
    const uint32_t* src = bins + block * (bucketCount * kWave);
    if (tileMap == nullptr) {
        CopyTile<64 * WAVES>(src, rowCount, tid, sTile);
    } else {
        CopyMappedRows<WAVES>(
            tileMap, rowCount, wave, [&](uint32_t bucket) { return src[bucket * kWave + lane]; },
            [&](uint32_t row, uint32_t bins4) { sTile[row * kWave + lane] = bins4; });
    }
    const uint32_t tileBytes = (tileDwords * 4 + 15) & ~15u;
    double* sRed = reinterpret_cast<double*>(reinterpret_cast<uint8_t*>(sTile) + tileBytes);  // [256 documents]
    const uint8_t* laneTile = reinterpret_cast<const uint8_t*>(sTile) + lane * 4;
    const uint32_t treeCount = treeEnd - treeBegin;
    __syncthreads();  // tile is loaded

    double acc[4] = {0.0, 0.0, 0.0, 0.0}, gathered[4] = {0.0, 0.0, 0.0, 0.0};
    uint4 rows[2][2][4];
    uint32_t first[2];
#define CBAMD_FETCH_DEEP(k, tree)                                                                  \
    do {                                                                                           \
        const uint4* row = deepRows + static_cast<size_t>(tree) * 8;                               \
        _Pragma("unroll") for (int i = 0; i < 4; ++i) {                                            \
            rows[k][0][i] = row[i];                                                                \
            rows[k][1][i] = row[4 + i];                                                            \
        }                                                                                          \
        first[k] = firstLeaf[tree];                                                                \
    } while (0)
#define CBAMD_DEEP_ROUND(k)                                                                        \
    do {                                                                                           \
        uint32_t low4, high4;                                                                      \
        if (__builtin_amdgcn_readfirstlane(rows[k][0][0].x) & kPairRowXorFlag) {                   \
            low4 = PairTreeIndexes<true, 8>(laneTile, rows[k][0]);                                 \
            high4 = PairTreeIndexes<true, HIGH>(laneTile, rows[k][1]);                             \
        } else {                                                                                   \
            low4 = PairTreeIndexes<false, 8>(laneTile, rows[k][0]);                                \
            high4 = PairTreeIndexes<false, HIGH>(laneTile, rows[k][1]);                            \
        }                                                                                          \
        const double* treeLeaves = leaves + __builtin_amdgcn_readfirstlane(first[k]);              \
        _Pragma("unroll") for (int q = 0; q < 4; ++q) {                                            \
            acc[q] = __dadd_rn(acc[q], gathered[q]);                                               \
        }                                                                                          \
        _Pragma("unroll") for (int q = 0; q < 4; ++q) {                                            \
            const uint32_t leaf = ((low4 >> (8 * q)) & 0xffu) |                                    \
                                  (((high4 >> (8 * q + 8 - HIGH)) & ((1u << HIGH) - 1)) << 8);     \
            gathered[q] = treeLeaves[leaf];                                                        \
        }                                                                                          \
        CBAMD_FETCH_DEEP(k, treeBegin + p + 2 * WAVES);                                            \
        p += WAVES;                                                                                \
    } while (0)

    uint32_t p = wave;
    CBAMD_FETCH_DEEP(0, treeBegin + p);
    CBAMD_FETCH_DEEP(1, treeBegin + p + WAVES);
    while (p + WAVES < treeCount) {
        CBAMD_DEEP_ROUND(0);
        CBAMD_DEEP_ROUND(1);
    }
    if (p < treeCount) {
        CBAMD_DEEP_ROUND(0);
    }
#undef CBAMD_DEEP_ROUND
#undef CBAMD_FETCH_DEEP
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        acc[q] = __dadd_rn(acc[q], gathered[q]);
    }
    // waves add their partial sums in wave order into the LDS accumulator; the last wave finishes the values
    // and writes them out (byte q of a lane's dword: document q * 64 + lane)
    for (uint32_t w = 0; w + 1 < WAVES; ++w) {
        if (wave == w) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                double* cell = sRed + q * kWave + lane;
                *cell = (w == 0) ? acc[q] : __dadd_rn(*cell, acc[q]);
            }
        }
        __syncthreads();
    }
    if (wave == WAVES - 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const size_t doc = block * kDocsPerBlock + q * kWave + lane;
            if (doc < docCount) {
                out[doc] = Finish(__dadd_rn(sRed[q * kWave + lane], acc[q]), scale, bias[0], treeBegin == 0);
            }
        }
    }
}

// EvalObliviousDeepTileKernel for models of several dimensions: the same tile, rows and walk; a workgroup sums two
// dimensions, those from blockIdx.y * 2 on (every slice of the dimensions walks the trees again). `leaves` holds the
// values slice by slice, [slice][tree][leaf][2] (zeros past the last dimension), `firstLeaf` counts leaves and
// `sliceLeaves` is the number of leaves of all trees, so that a leaf's two values come with one 16-byte load:
// gathered as two strided doubles from the model's own table the kernel was no faster than the plain one (the
// gathers' way through the texture path is what it waits for). A kernel of its own: as a template parameter of
// the one-dimensional kernel the second dimension cost that kernel 5 %.
// grid = (doc blocks, ceil(dim / 2)), block = 64 * WAVES, dynamic LDS = rows * 256 (rounded up to 16) + 2 * 256 * 8 bytes.
template <int HIGH, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void EvalObliviousDeepTilePairsKernel(
    const uint32_t* __restrict__ bins, size_t docCount, uint32_t bucketCount, const uint32_t* __restrict__ tileMap,
    uint32_t rowCount, const uint4* __restrict__ deepRows, const uint32_t* __restrict__ firstLeaf,
    const double* __restrict__ leaves, const double* __restrict__ bias, double scale, uint32_t dim, uint32_t sliceLeaves,
    uint32_t treeBegin, uint32_t treeEnd, double* __restrict__ out) {
    static_assert(HIGH == 4 || HIGH == 8, "levels 8..11 or 8..15 in the second half");
    constexpr int DIMS = 2;
    const uint32_t d0 = blockIdx.y * DIMS;
    leaves += static_cast<size_t>(blockIdx.y) * sliceLeaves * 2;
    extern __shared__ uint32_t sTile[];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const size_t block = blockIdx.x;
    const uint32_t tileDwords = rowCount * kWave;  // rowCount = bucketCount without a map
    const uint32_t* src = bins + block * (bucketCount * kWave);
    if (tileMap == nullptr) {
        CopyTile<64 * WAVES>(src, rowCount, tid, sTile);
    } else {
        CopyMappedRows<WAVES>(
            tileMap, rowCount, wave, [&](uint32_t bucket) { return src[bucket * kWave + lane]; },
            [&](uint32_t row, uint32_t bins4) { sTile[row * kWave + lane] = bins4; });
    }
    const uint32_t tileBytes = (tileDwords * 4 + 15) & ~15u;
    double* sRed = reinterpret_cast<double*>(reinterpret_cast<uint8_t*>(sTile) + tileBytes);  // [DIMS][256 documents]
    const uint8_t* laneTile = reinterpret_cast<const uint8_t*>(sTile) + lane * 4;
    const uint32_t treeCount = treeEnd - treeBegin;
    __syncthreads();  // tile is loaded

    double acc[4][DIMS], gathered[4][DIMS];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int c = 0; c < DIMS; ++c) {
            acc[q][c] = 0.0;
            gathered[q][c] = 0.0;
        }
    }
    uint4 rows[2][2][4];
    uint32_t first[2];
#define CBAMD_FETCH_DEEP2(k, tree)                                                                  \
    do {                                                                                           \
        const uint4* row = deepRows + static_cast<size_t>(tree) * 8;                               \
        _Pragma("unroll") for (int i = 0; i < 4; ++i) {                                            \
            rows[k][0][i] = row[i];                                                                \
            rows[k][1][i] = row[4 + i];                                                            \
        }                                                                                          \
        first[k] = firstLeaf[tree];                                                                \
    } while (0)
#define CBAMD_DEEP_ROUND2(k)                                                                        \
    do {                                                                                           \
        uint32_t low4, high4;                                                                      \
        if (__builtin_amdgcn_readfirstlane(rows[k][0][0].x) & kPairRowXorFlag) {                   \
            low4 = PairTreeIndexes<true, 8>(laneTile, rows[k][0]);                                 \
            high4 = PairTreeIndexes<true, HIGH>(laneTile, rows[k][1]);                             \
        } else {                                                                                   \
            low4 = PairTreeIndexes<false, 8>(laneTile, rows[k][0]);                                \
            high4 = PairTreeIndexes<false, HIGH>(laneTile, rows[k][1]);                            \
        }                                                                                          \
        const double* treeLeaves = leaves + static_cast<size_t>(__builtin_amdgcn_readfirstlane(first[k])) * DIMS; \
        _Pragma("unroll") for (int q = 0; q < 4; ++q) {                                            \
            _Pragma("unroll") for (int c = 0; c < DIMS; ++c) {                                     \
                acc[q][c] = __dadd_rn(acc[q][c], gathered[q][c]);                                  \
            }                                                                                      \
        }                                                                                          \
        _Pragma("unroll") for (int q = 0; q < 4; ++q) {                                            \
            const uint32_t leaf = ((low4 >> (8 * q)) & 0xffu) |                                    \
                                  (((high4 >> (8 * q + 8 - HIGH)) & ((1u << HIGH) - 1)) << 8);     \
            const double2 pair = reinterpret_cast<const double2*>(treeLeaves)[leaf];               \
            gathered[q][0] = pair.x;                                                               \
            gathered[q][1] = pair.y;                                                               \
        }                                                                                          \
        CBAMD_FETCH_DEEP2(k, treeBegin + p + 2 * WAVES);                                            \
        p += WAVES;                                                                                \
    } while (0)

    uint32_t p = wave;
    CBAMD_FETCH_DEEP2(0, treeBegin + p);
    CBAMD_FETCH_DEEP2(1, treeBegin + p + WAVES);
    while (p + WAVES < treeCount) {
        CBAMD_DEEP_ROUND2(0);
        CBAMD_DEEP_ROUND2(1);
    }
    if (p < treeCount) {
        CBAMD_DEEP_ROUND2(0);
    }
#undef CBAMD_DEEP_ROUND2
#undef CBAMD_FETCH_DEEP2
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int c = 0; c < DIMS; ++c) {
            acc[q][c] = __dadd_rn(acc[q][c], gathered[q][c]);
        }
    }
    // waves add their partial sums in wave order into the LDS accumulator; the last wave finishes the values
    // and writes them out (byte q of a lane's dword: document q * 64 + lane)
    for (uint32_t w = 0; w + 1 < WAVES; ++w) {
        if (wave == w) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
#pragma unroll
                for (int c = 0; c < DIMS; ++c) {
                    double* cell = sRed + c * kDocsPerBlock + q * kWave + lane;
                    *cell = (w == 0) ? acc[q][c] : __dadd_rn(*cell, acc[q][c]);
                }
            }
        }
        __syncthreads();
    }
    if (wave == WAVES - 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const size_t doc = block * kDocsPerBlock + q * kWave + lane;
#pragma unroll
            for (int c = 0; c < DIMS; ++c) {
                if (doc < docCount && d0 + c < dim) {
                    out[doc * dim + d0 + c] = Finish(__dadd_rn(sRed[c * kDocsPerBlock + q * kWave + lane], acc[q][c]), scale,
                                                     bias[d0 + c], treeBegin == 0);
                }
            }
        }
    }
}

__device__ __forceinline__ uint32_t BinOfDoc(const uint8_t* bins, size_t doc, uint32_t bucketCount, uint32_t bucket) {
    const size_t block = doc / kDocsPerBlock;
    const uint32_t r = static_cast<uint32_t>(doc % kDocsPerBlock);
    return bins[((block * bucketCount + bucket) * kWave + (r % kWave)) * 4 + r / kWave];
}

// Walks one non-symmetric tree for one document; returns the terminal node id
// (CalcIndexesNonSymmetric, cpu/evaluator_impl.cpp:462-493).
__device__ __forceinline__ uint32_t WalkNonSymmetric(const uint8_t* bins, size_t doc, uint32_t bucketCount,
                                                     const TTreeTables& tt, uint32_t tree) {
    uint32_t node = tt.TreeStart[tree];
    for (;;) {
        const uint32_t sp = tt.Splits[node];
        const uint32_t st = tt.StepNodes[node];
        const uint32_t b = BinOfDoc(bins, doc, bucketCount, sp & 0xffffu);
        const bool right = ((b ^ ((sp >> 16) & 0xffu)) >= (sp >> 24));
        const uint32_t diff = right ? (st >> 16) : (st & 0xffffu);
        if (diff == 0) {
            return node;
        }
        node += diff;
    }
}

// Non-symmetric trees: one thread per document. grid = ceil(docs / 256), block = 256.
template <int DCHUNK>
__global__ __launch_bounds__(256) void EvalNonSymmetricKernel(const uint8_t* __restrict__ bins, size_t docCount,
                                                              uint32_t bucketCount, TTreeTables tt, uint32_t treeBegin,
                                                              uint32_t treeEnd, double* __restrict__ out) {
    const size_t doc = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (doc >= docCount) {
        return;
    }
    const int dim = tt.Dim;
    const bool addBias = treeBegin == 0;
    for (int d0 = 0; d0 < dim; d0 += DCHUNK) {
        double acc[DCHUNK];
#pragma unroll
        for (int k = 0; k < DCHUNK; ++k) {
            acc[k] = 0.0;
        }
        for (uint32_t t = treeBegin; t < treeEnd; ++t) {
            const uint32_t node = WalkNonSymmetric(bins, doc, bucketCount, tt, t);
            const double* p = tt.Leaves + tt.NodeToLeaf[node] + d0;
#pragma unroll
            for (int k = 0; k < DCHUNK; ++k) {
                if (DCHUNK == 1 || d0 + k < dim) {
                    acc[k] = __dadd_rn(acc[k], p[k]);
                }
            }
        }
#pragma unroll
        for (int k = 0; k < DCHUNK; ++k) {
            if (DCHUNK == 1 || d0 + k < dim) {
                out[doc * dim + d0 + k] = Finish(acc[k], tt.Scale, tt.Bias[d0 + k], addBias);
            }
        }
    }
}

// Non-symmetric trees over an LDS tile of bins: one workgroup of kTileWaves waves per
// 256-document block, the waves split the trees in groups of kNsGroup consecutive trees, four
// documents per lane walk the trees of a group side by side (4 * kNsGroup independent chains).
// The trees come re-laid level by level: an entry is 8 bytes,
//   x: NO_XOR   bucket << 8 | splitIdx << 24          (bucket << 8 = offset of the bucket in the tile)
//      else     bucket | xorMask << 16 | splitIdx << 24
//   y: byte offset (entry index * 8, relative to the tree's first entry) of the left child in the
//      low half and of the right child in the high half.
// A terminal entry has x = 0 (true for every bin), its own offset as right child and, in the low
// half of y, the index of its leaf relative to the tree's first leaf. All lanes take the same
// number of steps (the height of the tallest tree of the group): a lane that has reached its leaf
// stays there. Since
// the lanes of a wave are always on the same level, their gathers of a step fall into the few
// cache lines of that level.
// treeRows: 4 dwords per tree: first entry, height, first leaf value, unused.
// grid = doc blocks, block = 64 * kTileWaves, dynamic LDS = buckets * 256 (rounded up to 8) +
// 256 * DCHUNK * 8 bytes.
constexpr int kNsGroup = 4;

template <bool NO_XOR, int DCHUNK>
__global__ __launch_bounds__(64 * kTileWaves) void EvalNonSymmetricTileKernel(
    const uint32_t* __restrict__ bins, size_t docCount, uint32_t bucketCount, const uint2* __restrict__ entries,
    const uint4* __restrict__ treeRows, const double* __restrict__ leaves, const double* __restrict__ bias, double scale,
    int dim, uint32_t treeBegin, uint32_t treeEnd, double* __restrict__ out) {
    extern __shared__ uint32_t sTile[];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const size_t block = blockIdx.x;
    const uint32_t tileDwords = bucketCount * kWave;
    const uint32_t* src = bins + block * tileDwords;
    CopyTile<64 * kTileWaves>(src, bucketCount, tid, sTile);
    const bool addBias = treeBegin == 0;
    const uint8_t* laneTile = reinterpret_cast<const uint8_t*>(sTile) + lane * 4;
    double* sRed = reinterpret_cast<double*>(sTile + ((tileDwords + 1) & ~1u));
    for (int d0 = 0; d0 < dim; d0 += DCHUNK) {
        __syncthreads();  // tile is loaded / the previous chunk's accumulator has been read
        double acc[4][DCHUNK];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int k = 0; k < DCHUNK; ++k) {
                acc[j][k] = 0.0;
            }
        }
        // a wave walks kNsGroup trees at a time (trees t0 .. t0 + kNsGroup - 1), i.e. 4 * kNsGroup
        // independent chains per lane, to cover the latency of the entry gathers
        for (uint32_t t0 = treeBegin + wave * kNsGroup; t0 < treeEnd; t0 += kTileWaves * kNsGroup) {
            const char* base[kNsGroup];
            uint32_t firstLeaf[kNsGroup];
            uint32_t height = 0;
#pragma unroll
            for (int g = 0; g < kNsGroup; ++g) {
                // trees past the end walk tree t0 again and are not added
                const uint4 row = treeRows[t0 + g < treeEnd ? t0 + g : t0];
                base[g] = reinterpret_cast<const char*>(entries + __builtin_amdgcn_readfirstlane(row.x));
                height = max(height, static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(row.y)));
                firstLeaf[g] = __builtin_amdgcn_readfirstlane(row.z);
            }
            uint32_t off[kNsGroup][4];
#pragma unroll
            for (int g = 0; g < kNsGroup; ++g) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    off[g][j] = 0;
                }
            }
            for (uint32_t step = 0; step < height; ++step) {
                uint2 node[kNsGroup][4];
#pragma unroll
                for (int g = 0; g < kNsGroup; ++g) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        node[g][j] = *reinterpret_cast<const uint2*>(base[g] + off[g][j]);
                    }
                }
#pragma unroll
                for (int g = 0; g < kNsGroup; ++g) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint32_t x = node[g][j].x;
                        uint32_t bin;
                        if (NO_XOR) {
                            bin = laneTile[(x & 0xffffffu) + j];
                        } else {
                            bin = laneTile[((x & 0xffffu) << 8) + j] ^ ((x >> 16) & 0xffu);
                        }
                        const uint32_t shift = bin >= (x >> 24) ? 16u : 0u;
                        off[g][j] = (node[g][j].y >> shift) & 0xffffu;
                    }
                }
            }
#pragma unroll
            for (int g = 0; g < kNsGroup; ++g) {
                if (t0 + g < treeEnd) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint2 last = *reinterpret_cast<const uint2*>(base[g] + off[g][j]);
                        const uint32_t leafRel = last.y & 0xffffu;
                        const double* p = leaves + firstLeaf[g] +
                                          (DCHUNK == 1 ? leafRel : leafRel * static_cast<uint32_t>(dim)) + d0;
#pragma unroll
                        for (int k = 0; k < DCHUNK; ++k) {
                            if (DCHUNK == 1 || d0 + k < dim) {
                                acc[j][k] = __dadd_rn(acc[j][k], p[k]);
                            }
                        }
                    }
                }
            }
        }
        // waves add their partial sums in wave order into the LDS accumulator; the last wave
        // finishes the values and writes them out
        for (uint32_t w = 0; w + 1 < kTileWaves; ++w) {
            if (wave == w) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
#pragma unroll
                    for (int k = 0; k < DCHUNK; ++k) {
                        double* cell = sRed + (j * kWave + lane) * DCHUNK + k;
                        *cell = (w == 0) ? acc[j][k] : __dadd_rn(*cell, acc[j][k]);
                    }
                }
            }
            __syncthreads();
        }
        if (wave == kTileWaves - 1) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const size_t doc = block * kDocsPerBlock + j * kWave + lane;
#pragma unroll
                for (int k = 0; k < DCHUNK; ++k) {
                    if (doc < docCount && (DCHUNK == 1 || d0 + k < dim)) {
                        const double sum = __dadd_rn(sRed[(j * kWave + lane) * DCHUNK + k], acc[j][k]);
                        out[doc * dim + d0 + k] = Finish(sum, scale, bias[d0 + k], addBias);
                    }
                }
            }
        }
    }
}

// Non-symmetric models whose trees have at most kNsLdsEntries entries (a split by a xor mask is two of plain bins): as EvalNonSymmetricTileKernel, but a
// wave walks its trees out of a copy in its own LDS region (an LDS gather costs a fraction of a gather from global memory).
// Trees are grouped into units of up to kNsUnitTrees trees and ENTRIES entries; a wave takes a unit at a time and walks its
// trees side by side (4 documents x kNsUnitTrees chains per lane).
// The top three levels of a tree are the same seven nodes for every document. They come with the unit's row in scalar
// registers, padded to seven where a branch ends early (a node that is false for every bin), and are compared byte-parallel,
// four documents to an instruction: a read of the bucket's bins and a v_lerp_u8 per node, whose bit 7 says bin >= split,
// and selects by those bits. The three bits of a document choose one of the tree's first eight entries, its exits. Units without a
// node on the third level leave that level out: with its four reads a tree, 1M documents, 500 trees of one level over 20 features took
// 431 us a call where now 411, 300 of two levels and two dimensions (500 001 documents, 100 features) 205 and now 186.
// A compact entry is one dword:
//   bits 0-7 splitIdx, bits 8-17 the 256-byte LDS row that holds the bucket's bins (so entry & 0x3ff00 is its
//   address), bits 21-31 index of the left child relative to the unit's first entry.
// Both addresses of a step take one instruction: the bin's is (entry & 0x3ff00) | lane offset, the pair's the
// funnel shift {wave, entry} >> 19, because wave w keeps its entries at LDS address w * 8 KB. Regions shorter than
// 8 KB leave gaps, and the rows of the bins fill them: NsLdsTileRow() says where bucket b goes, for the copy of
// the tile here and for the entries on the host.
// The two children of a node sit side by side at an even index, so one 8-byte LDS read, issued together with the read of
// the node's bin, brings both and the compare only selects: one LDS round trip per level. A terminal entry points at its own
// pair and compares so that it selects itself (even index: splitIdx 255, false for every bin;
// odd index: splitIdx 0, true for every bin, which no real split has). The next unit's entries
// are fetched into registers while the current unit is walked: sixteen bytes per lane and whole rounds of
// the wave, with neither bounds nor branches - every unit starts at a multiple of four entries and `entries`
// ends with ENTRIES spare ones (a copy written with a test per round cost a taken branch each way per round,
// a tenth of the kernel's time). valuesByEntry holds the leaf value of every terminal entry, indexed like
// `entries`. One dimension: ENTRIES zeros behind them, which the trees that a unit lacks and those outside of the call's range
// read; a unit's values are requested behind its walk and added after the next unit's walk, and no load of them depends on a branch, so
// that the wait for a unit's entries does not wait for the values requested behind them. Behind a wave's last unit no entries are
// fetched: a region's 4 KB and more, with one again 1M documents, 100 trees of depth 3 over 60 features took 202 us, now 191.
// What bounds it: the walk's LDS reads and vector issue together (7.4 cycles of a CU for 64 chains' step; without bank conflicts
// 6 % of the launch less, without the bins' reads 8 %, without the selects 12 %), and the values' gathers (12 of them a unit, some
// 8 %). Whole call, with the root alone compared once for a lane's documents, the steps from there on, and values that a branch
// guarded, and now: 4M documents, 500 trees of depth 10 over 300 features 6033 -> 5445 us; 1M, 500 of depth 6 over 60 686 -> 589, 300
// of depth 8 over 150 675 -> 606, 500 of depth 9 over 20 (600 000 documents) 549 -> 491; three dimensions, 500 000 documents, 300
// of depth 8 over 100 418 -> 413.
// unitRows: 32 dwords per unit: first entry, steps behind the exits, first entry of the wave's next unit (WAVES on), first entry
// of the second tree relative to the unit's, that of the third tree | number of trees << 16, and the model's numbers
// of the three trees: a call for the trees [treeBegin, treeEnd) adds the values of those only and passes over
// the units that hold none of them; from dword 8 on eight dwords per tree, its seven nodes by level (children of node n: 2 n + 1
// and 2 n + 2): LDS row of the bins << 8 | (256 - splitIdx), low byte 0: false for every bin; the eighth dword of the first tree: no
// node of the unit's trees is on the third level.
// Models of several dimensions: a workgroup sums DIMS of them, those from blockIdx.y * DIMS on (every slice of
// the dimensions walks the trees again), and valuesByEntry is [slice][entryCount] rows of DIMS values (zeros past
// the last dimension), so that a leaf's values come with one aligned load; those of the range's trees are read and added right behind
// the unit's walk, with the other waves of the SIMD to cover the wait.
// grid = (doc blocks, ceil(dim / DIMS)), block = 64 * WAVES, dynamic LDS = NsLdsTileRows(buckets, WAVES, ENTRIES) * 256
// + 256 * 8 * DIMS bytes; no other LDS in the kernel.
constexpr int kNsLdsEntries = 2048;
constexpr int kNsUnitTrees = 3;
constexpr int kNsUnitDwords = 32;

// The 256-byte LDS row of bucket b's bins: the 8 KB of a wave start with its entries (entries / 64 rows) and the
// rows that are left take bins; the other buckets follow the last wave's 8 KB.
__host__ __device__ constexpr uint32_t NsLdsTileRow(uint32_t bucket, uint32_t waves, uint32_t entries) {
    const uint32_t regionRows = entries / 64, gapRows = 32 - regionRows;
    const uint32_t divisor = gapRows ? gapRows : 1;  // regions of 8 KB leave no gap
    return bucket < gapRows * waves ? 32 * (bucket / divisor) + regionRows + bucket % divisor
                                    : 32 * waves + bucket - gapRows * waves;
}

// Rows of LDS up to the end of the bins
__host__ __device__ constexpr uint32_t NsLdsTileRows(uint32_t buckets, uint32_t waves, uint32_t entries) {
    const uint32_t gapRows = (32 - entries / 64) * waves;
    return 32 * waves + (buckets > gapRows ? buckets - gapRows : 0);
}

// A load of a scalar from an LDS address given as a number (the dynamic LDS of a kernel without other LDS
// starts at 0).
template <class T>
__device__ __forceinline__ T LdsLoad(uint32_t address) {
    return *reinterpret_cast<const __attribute__((address_space(3))) T*>(address);
}

__device__ __forceinline__ double LeafRowValue(const double2& row, int k) {
    return k == 0 ? row.x : row.y;
}

__device__ __forceinline__ double LeafRowValue(const double4& row, int k) {
    return k == 0 ? row.x : k == 1 ? row.y : k == 2 ? row.z : row.w;
}

// Bits of `ones` where those of `mask` are set, of `zeros` elsewhere: v_bitop3 of vector registers, which takes half the time of
// the v_bfi that the expression compiles to.
__device__ __forceinline__ uint32_t SelectBits(uint32_t mask, uint32_t ones, uint32_t zeros) {
    uint32_t r;
    asm("v_bitop3_b32 %0, %1, %2, %3 bitop3:0xca" : "=v"(r) : "v"(mask), "v"(ones), "v"(zeros));
    return r;
}

// (bits & mask) | base, in the same class of instruction
__device__ __forceinline__ uint32_t AndOr(uint32_t bits, uint32_t mask, uint32_t base) {
    uint32_t r;
    asm("v_bitop3_b32 %0, %1, %2, %3 bitop3:0xea" : "=v"(r) : "v"(bits), "v"(mask), "v"(base));
    return r;
}

template <int WAVES, int ENTRIES, int DIMS>
__global__ __launch_bounds__(64 * WAVES) void EvalNonSymmetricLdsKernel(
    const uint32_t* __restrict__ bins, size_t docCount, uint32_t bucketCount, const uint32_t* __restrict__ entries,
    const uint32_t* __restrict__ unitRows, uint32_t unitCount, const double* __restrict__ valuesByEntry,
    const double* __restrict__ bias, double scale, uint32_t dim, uint32_t entryCount, uint32_t treeBegin,
    uint32_t treeEnd, uint32_t wholeModel, double* __restrict__ out) {
    constexpr int kFetch = ENTRIES / (4 * kWave);  // rounds of a wave's copy, sixteen bytes per lane
    static_assert(ENTRIES <= kNsLdsEntries && ENTRIES % (4 * kWave) == 0, "a region holds whole rounds of a wave's copy");
    static_assert((32 - ENTRIES / 64) % 4 == 0, "the tile is requested four rows at a time");
    extern __shared__ uint32_t sTile[];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const size_t block = blockIdx.x;
    const uint32_t tileDwords = bucketCount * kWave;
    const uint32_t* src = bins + block * tileDwords;
    const uint32_t laneOff = lane * 4;
    double* sRed = reinterpret_cast<double*>(sTile + NsLdsTileRows(bucketCount, WAVES, ENTRIES) * kWave);
    uint32_t* sEntries = sTile + wave * kNsLdsEntries;  // 8 KB per wave, the first ENTRIES * 4 bytes of them
    const uint32_t bucketMask = 0x3ff00u;
    // A unit's entries come as whole rounds, whatever its size: a unit starts at a multiple of four entries and
    // the table ends with ENTRIES spare ones, so the copy needs neither a bound nor a branch (entries past the
    // unit's are never followed).
    using TEntries4 = uint32_t __attribute__((ext_vector_type(4)));
    TEntries4 fetched[kFetch];
    const auto fetchUnit = [&](uint32_t firstEntry) {
        const TEntries4* source = reinterpret_cast<const TEntries4*>(entries + firstEntry) + lane;
#pragma unroll
        for (int i = 0; i < kFetch; ++i) {
            fetched[i] = source[i * kWave];
        }
    };
    // whether a unit holds a tree of the call's range
    const auto anyWanted = [&](uint32_t unit) {
        const uint32_t* r = unitRows + unit * kNsUnitDwords;
        const uint32_t trees = r[4] >> 16, range = treeEnd - treeBegin;
        return r[5] - treeBegin < range || (trees > 1 && r[6] - treeBegin < range) || (trees > 2 && r[7] - treeBegin < range);
    };
    const auto skipUnwanted = [&](uint32_t unit) {
        while (unit < unitCount && !anyWanted(unit)) {
            unit += WAVES;
        }
        return unit;
    };

    RequestTile<64 * WAVES>(src, bucketCount, tid, sTile, [](uint32_t bucket) { return NsLdsTileRow(bucket, WAVES, ENTRIES); });
    const auto unitBehind = [&](uint32_t unit) { return wholeModel ? unit + WAVES : skipUnwanted(unit + WAVES); };
    uint32_t u = wholeModel ? wave : skipUnwanted(wave);
    uint32_t row[kNsUnitDwords];
    const auto loadRow = [&](uint32_t unit) {
#pragma unroll
        for (int i = 0; i < kNsUnitDwords; ++i) {
            row[i] = unitRows[unit * kNsUnitDwords + i];
        }
    };
    if (u < unitCount) {
        loadRow(u);
        fetchUnit(row[0]);
    }
    AwaitTile();
    __syncthreads();  // tile is loaded

    double acc[4][DIMS];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int k = 0; k < DIMS; ++k) {
            acc[j][k] = 0.0;
        }
    }
    // one dimension: a unit's values are requested behind its walk and added behind the next unit's
    double pending[kNsUnitTrees][4];
#pragma unroll
    for (int g = 0; g < kNsUnitTrees; ++g) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            pending[g][j] = 0.0;
        }
    }
    const auto addPending = [&]() {
#pragma unroll
        for (int g = 0; g < kNsUnitTrees; ++g) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[j][0] = __dadd_rn(acc[j][0], pending[g][j]);
            }
        }
    };
    uint32_t next = unitBehind(u);
    const uint32_t d0 = blockIdx.y * DIMS;
    const double* sliceValues = valuesByEntry + static_cast<size_t>(blockIdx.y) * entryCount * DIMS;
    const uint32_t mask80 = 0x80808080u, maskC0 = 0xc0c0c0c0u;
    while (u < unitCount) {
        const uint32_t first = row[0], steps = row[1], trees = row[4] >> 16;
        // trees the unit does not have walk its first tree again; their values are not added
        const uint32_t start[kNsUnitTrees] = {0u, row[3], row[4] & 0xffffu};
        bool wanted[kNsUnitTrees];
#pragma unroll
        for (int g = 0; g < kNsUnitTrees; ++g) {
            wanted[g] = static_cast<uint32_t>(g) < trees && row[5 + g] - treeBegin < treeEnd - treeBegin;
        }
        // the previous unit's reads were issued before these stores and LDS serves one wave in order
#pragma unroll
        for (int i = 0; i < kFetch; ++i) {
            reinterpret_cast<TEntries4*>(sEntries)[i * kWave + lane] = fetched[i];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (next < unitCount) {
            fetchUnit(wholeModel ? row[2] : unitRows[next * kNsUnitDwords]);
        }
        // the top levels
        uint32_t path[kNsUnitTrees];  // a document's three results in bits 5 to 7 of its byte
        const auto compareTop = [&](auto levels) {
            constexpr int kNodes = (1 << decltype(levels)::value) - 1;
            uint32_t bins4[kNsUnitTrees][kNodes];
#pragma unroll
            for (int g = 0; g < kNsUnitTrees; ++g) {
#pragma unroll
                for (int n = 0; n < kNodes; ++n) {
                    bins4[g][n] = LdsLoad<uint32_t>((row[8 + 8 * g + n] & bucketMask) | laneOff);
                }
            }
#pragma unroll
            for (int g = 0; g < kNsUnitTrees; ++g) {
                uint32_t side[kNodes];  // bit 7 of every byte: the document goes right
#pragma unroll
                for (int n = 0; n < kNodes; ++n) {
                    side[n] = __builtin_amdgcn_lerp(bins4[g][n], (row[8 + 8 * g + n] & 0xffu) * 0x01010101u, 0);
                }
                const uint32_t second = SelectBits(side[0], side[2], side[1]);
                uint32_t third = 0;
                if constexpr (kNodes == 7) {
                    third = SelectBits(side[0], SelectBits(second, side[6], side[5]), SelectBits(second, side[4], side[3]));
                }
                path[g] = SelectBits(maskC0, SelectBits(mask80, side[0], second >> 1), third >> 2);
            }
        };
        if (row[15] != 0) {
            compareTop(std::integral_constant<int, 2>());
        } else {
            compareTop(std::integral_constant<int, 3>());
        }
        uint32_t entry[kNsUnitTrees][4];
#pragma unroll
        for (int g = 0; g < kNsUnitTrees; ++g) {
            const uint32_t exits = wave * (kNsLdsEntries * 4) + start[g] * 4;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                entry[g][j] = LdsLoad<uint32_t>(AndOr(path[g] >> (8 * j + 3), 0x1cu, exits));
            }
        }
        loadRow(min(next, unitCount - 1));
        for (uint32_t step = 0; step < steps; ++step) {
            uint64_t pair[kNsUnitTrees][4];  // the two children of a chain's node, left in the low half
            uint32_t bin[kNsUnitTrees][4];
#pragma unroll
            for (int g = 0; g < kNsUnitTrees; ++g) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t e = entry[g][j];
                    // bits 18-20 of an entry are clear: e >> 19 is the byte offset of the pair of children in
                    // the wave's region, whose number comes in from above (kNsLdsEntries * 4 = 1 << 13)
                    pair[g][j] = LdsLoad<uint64_t>(__builtin_amdgcn_alignbit(wave, e, 19));
                    bin[g][j] = LdsLoad<uint8_t>(AndOr(e, bucketMask, laneOff) + j);
                }
            }
#pragma unroll
            for (int g = 0; g < kNsUnitTrees; ++g) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    entry[g][j] = static_cast<uint32_t>(bin[g][j] >= (entry[g][j] & 0xffu) ? pair[g][j] >> 32 : pair[g][j]);
                }
            }
        }
        // eight times a terminal entry's place in the unit: that of its pair, and one more for the right one (splitIdx 0, else 255)
        uint32_t place[kNsUnitTrees][4];
#pragma unroll
        for (int g = 0; g < kNsUnitTrees; ++g) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                place[g][j] = (entry[g][j] >> 18) | (~entry[g][j] & 8u);
            }
        }
        if constexpr (DIMS == 1) {
            addPending();
#pragma unroll
            for (int g = 0; g < kNsUnitTrees; ++g) {
                // the requests stay behind the sums: the values then have the same registers in every turn, where other ones
                // would be waited for and moved
                asm volatile("" : "+v"(acc[0][0]), "+v"(acc[1][0]), "+v"(acc[2][0]), "+v"(acc[3][0]), "+v"(place[g][0]), "+v"(place[g][1]),
                                  "+v"(place[g][2]), "+v"(place[g][3]));
                const char* from = reinterpret_cast<const char*>(valuesByEntry + (wanted[g] ? first : entryCount));
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    pending[g][j] = *reinterpret_cast<const double*>(from + place[g][j]);
                }
            }
        } else {
#pragma unroll
            for (int g = 0; g < kNsUnitTrees; ++g) {
                if (wanted[g]) {
                    using TLeafRow = typename std::conditional<DIMS == 2, double2, double4>::type;
                    TLeafRow value[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        value[j] = reinterpret_cast<const TLeafRow*>(sliceValues)[first + place[g][j] / 8];
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
#pragma unroll
                        for (int k = 0; k < DIMS; ++k) {
                            acc[j][k] = __dadd_rn(acc[j][k], LeafRowValue(value[j], k));
                        }
                    }
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
        u = next;
        next = unitBehind(u);
    }
    if constexpr (DIMS == 1) {
        addPending();
    }
    // waves add their partial sums in wave order into the LDS accumulator; the last wave
    // finishes the values and writes them out
    for (uint32_t w = 0; w + 1 < WAVES; ++w) {
        if (wave == w) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int k = 0; k < DIMS; ++k) {
                    double* cell = sRed + (k * 4 + j) * kWave + lane;
                    *cell = (w == 0) ? acc[j][k] : __dadd_rn(*cell, acc[j][k]);
                }
            }
        }
        __syncthreads();
    }
    if (wave == WAVES - 1) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const size_t doc = block * kDocsPerBlock + j * kWave + lane;
#pragma unroll
            for (int k = 0; k < DIMS; ++k) {
                if (doc < docCount && d0 + k < dim) {
                    out[doc * dim + d0 + k] =
                        Finish(__dadd_rn(sRed[(k * 4 + j) * kWave + lane], acc[j][k]), scale, bias[d0 + k], treeBegin == 0);
                }
            }
        }
    }
}

// Leaf indexes [doc][tree - treeBegin] for both tree kinds (CalcLeafIndexesGeneric,
// cpu/evaluator.h:174-253; non-symmetric numbering cpu/evaluator_impl.cpp:626-633).
__global__ __launch_bounds__(256) void LeafIndexesKernel(const uint8_t* __restrict__ bins, size_t docCount,
                                                         uint32_t bucketCount, TTreeTables tt, int oblivious,
                                                         uint32_t treeBegin, uint32_t treeEnd,
                                                         uint32_t* __restrict__ out) {
    const size_t doc = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (doc >= docCount) {
        return;
    }
    const size_t treeCount = treeEnd - treeBegin;
    for (uint32_t t = treeBegin; t < treeEnd; ++t) {
        uint32_t result;
        if (oblivious) {
            const uint32_t first = tt.TreeStart[t];
            const uint32_t depth = tt.TreeSize[t];
            uint32_t idx = 0;
            for (uint32_t d = 0; d < depth; ++d) {
                const uint32_t sp = tt.Splits[first + d];
                const uint32_t b = BinOfDoc(bins, doc, bucketCount, sp & 0xffffu);
                idx |= static_cast<uint32_t>((b ^ ((sp >> 16) & 0xffu)) >= (sp >> 24)) << d;
            }
            result = idx;
        } else {
            const uint32_t node = WalkNonSymmetric(bins, doc, bucketCount, tt, t);
            result = (tt.NodeToLeaf[node] - tt.FirstLeaf[t]) / static_cast<uint32_t>(tt.Dim);
        }
        out[doc * treeCount + (t - treeBegin)] = result;
    }
}

// Leaf indexes of oblivious trees of depth <= MAXD <= 8 whose 256-document tile of bins fits LDS: the byte-parallel walk
// of the tile kernels (four documents per lane, a tree per wave and turn, its levels broadcast from a lane's register), and
// rows of the output written whole. What bounds it is the output, four bytes per document and tree. A workgroup of eight
// waves takes a block of 256 documents and a share of the trees in groups of 64: wave w walks trees 8 w .. 8 w + 7 of
// the group, four at a time, turns the four bytes of four trees into the four bytes of a document (a 4 x 4 transpose of
// bytes) and leaves them in LDS, a ring of 128 trees per document, a byte each; then sixteen threads write 64 indexes of
// a document, 16 bytes a thread. The 64 indexes are those that fill whole 128-byte lines of the output, up to 31 trees
// behind the group, which the ring still holds: rows of 4 * trees bytes start anywhere in a line, and lines written in two
// parts cost the memory twice. 200 000 documents * 1000 trees of depth 6 over 100 features: 466 us with a workgroup per
// block and 4-byte stores, 227 with shares and 16-byte stores, 165 with whole lines, one after another on one box; traced in
// whole calls 183 us (4.4 TB/s), back to back 200.
// A share is some groups of 64 trees: the grid is blocks * shares, so that a batch of a few hundred blocks still fills
// the chip a few times over (one workgroup per block left a last generation nearly empty).
// GROUP = 32 is for tiles that leave less than 33 KB of LDS (509 to 576 buckets): half the trees per group, a line of a
// document at a time, a ring of 64 trees in 16 KB. Its documents' rings have no spare dword between them; each starts a
// dword further on than that of four documents before, so that the lanes' stores fall on all banks. 200 000 documents * 500
// trees of depth 8, whole call: 540 buckets 250 us, 2540 through LeafIndexesKernel; 508 buckets, groups of 64, 251.
// packedTrees as in EvalObliviousTileKernel. block = 512 threads, dynamic LDS = buckets * 256 + 256 * LeafIndexPitch * 4.
// STREAM: the stores of whole lines are nontemporal: an output larger than the memory-side cache (256 MB) goes past the
// caches. 200 000 documents * 1000 trees (800 MB), whole call: 242 -> 219 us with three outputs in turn, 240 -> 181 with one. A
// smaller output keeps plain stores: its next reader finds it in that cache (60 000 * 700, 168 MB, call and a reduction
// over the indexes: 138 us, 154 with nontemporal stores). Those of a share's first and last group are plain always: they write
// parts of lines (nontemporal as well: 219 -> 226 and 181 -> 221).
constexpr int kLeafIndexGroup = 64;
constexpr int kLeafIndexSmallGroup = 32;
constexpr int kLeafIndexThreads = 512;
constexpr int kLeafIndexLine = 32;                        // dwords of a line of the output

// dwords between two documents' rings of two groups of trees
__host__ __device__ constexpr int LeafIndexPitch(int group) {
    return group == kLeafIndexSmallGroup ? 2 * group / 4 : 2 * group / 4 + 1;
}

template <bool STREAM>
__device__ __forceinline__ void StoreQuad(uint32_t* to, const uint4& quad) {
    typedef uint32_t TQuad __attribute__((ext_vector_type(4)));
    if (STREAM) {
        __builtin_nontemporal_store(TQuad{quad.x, quad.y, quad.z, quad.w}, reinterpret_cast<TQuad*>(to));
    } else {
        *reinterpret_cast<uint4*>(to) = quad;
    }
}

template <bool SEVEN_BIT, int MAXD, int GROUP, bool STREAM>
__global__ __launch_bounds__(kLeafIndexThreads) void LeafIndexesTileKernel(
    const uint32_t* __restrict__ bins, uint32_t docCount, uint32_t bucketCount, const uint32_t* __restrict__ packedTrees,
    uint32_t treeBegin, uint32_t treeEnd, uint32_t shares, uint32_t shareTrees, uint32_t* __restrict__ out) {
    extern __shared__ uint32_t sTile[];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    // the shares of a block go to one XCD one after the other, so that they read its bins from one L2
    const uint32_t perXcd = gridDim.x / kXcdCount, extra = gridDim.x % kXcdCount;
    const uint32_t xcd = blockIdx.x % kXcdCount;
    const uint32_t work = xcd * perXcd + min(xcd, extra) + blockIdx.x / kXcdCount;
    const uint32_t block = work / shares;
    // A share ends, document by document, where a line ends; the next one walks the trees of a line more in front.
    const bool firstShare = work % shares == 0, lastShare = work % shares == shares - 1;
    const int32_t lead = firstShare ? 0 : kLeafIndexLine;
    const uint32_t firstTree = treeBegin + (work % shares) * shareTrees - lead;
    const int32_t count = lastShare ? treeEnd - firstTree : shareTrees + lead;  // trees that are walked
    CopyTile<kLeafIndexThreads>(bins + static_cast<size_t>(block) * (bucketCount * kWave), bucketCount, tid, sTile);
    uint32_t* ring = sTile + bucketCount * kWave;
    const uint8_t* laneTile = reinterpret_cast<const uint8_t*>(sTile) + lane * 4;
    const size_t treeCount = treeEnd - treeBegin;
    const uint32_t blockDocs = min(static_cast<uint32_t>(kDocsPerBlock), docCount - block * kDocsPerBlock);
    uint32_t* blockOut = out + static_cast<size_t>(block) * kDocsPerBlock * treeCount + (firstTree - treeBegin);
    constexpr int kWaves = kLeafIndexThreads / kWave;
    constexpr int kPerWave = GROUP / kWaves;
    constexpr int kRing = 2 * GROUP / 4, kPitch = LeafIndexPitch(GROUP);  // dwords of a document's ring, and to the next one
    constexpr uint32_t kDocThreads = GROUP / 4;                           // threads that write a document
    constexpr uint32_t kDocsPerPass = kLeafIndexThreads / kDocThreads;
    // where the ring of document d of the block starts, the same for every kWave documents
    const auto ringStart = [](uint32_t d) { return kPitch == kRing ? d / 4 : 0u; };
    static_assert(kPitch != kRing || (kWave / 4 % kRing == 0 && kDocsPerPass / 4 % kRing == 0), "documents that share a start");
    // the packed rows of the wave's trees of a group, four trees to a register, fetched a group ahead; trees past
    // the share are walked as its last tree and not written
    uint32_t rows[kPerWave / 4];
    const auto fetchRows = [&](int32_t group) {
#pragma unroll
        for (int q = 0; q < kPerWave / 4; ++q) {
            const int32_t t = min(group + static_cast<int32_t>(wave * kPerWave + q * 4 + lane / kPackedTreeDwords), count - 1);
            rows[q] = packedTrees[static_cast<size_t>(firstTree + t) * kPackedTreeDwords + lane % kPackedTreeDwords];
        }
    };
    fetchRows(0);
    for (int32_t group = 0; group < count; group += GROUP) {
        __syncthreads();  // the tile is loaded; the previous group's indexes are written
#pragma unroll
        for (int q = 0; q < kPerWave / 4; ++q) {
            uint32_t idx[4];
            FourTreesIndexes<SEVEN_BIT, MAXD>(laneTile, rows[q], idx);
            const uint32_t low01 = __builtin_amdgcn_perm(idx[1], idx[0], 0x05010400u);  // documents 0 and 1, trees 0 and 1
            const uint32_t high01 = __builtin_amdgcn_perm(idx[1], idx[0], 0x07030602u);
            const uint32_t low23 = __builtin_amdgcn_perm(idx[3], idx[2], 0x05010400u);
            const uint32_t high23 = __builtin_amdgcn_perm(idx[3], idx[2], 0x07030602u);
            uint32_t* cell = ring + lane * kPitch + (group / 4 + wave * (kPerWave / 4) + q + ringStart(lane)) % kRing;
            cell[0 * kWave * kPitch] = __builtin_amdgcn_perm(low23, low01, 0x05040100u);
            cell[1 * kWave * kPitch] = __builtin_amdgcn_perm(low23, low01, 0x07060302u);
            cell[2 * kWave * kPitch] = __builtin_amdgcn_perm(high23, high01, 0x05040100u);
            cell[3 * kWave * kPitch] = __builtin_amdgcn_perm(high23, high01, 0x07060302u);
        }
        __syncthreads();
        fetchRows(group + GROUP);
        const int32_t done = min(group + GROUP, count);  // trees whose indexes are in the ring
        const int32_t quadTree = group + static_cast<int32_t>(tid % kDocThreads) * 4;
        // the indexes of trees `tree` .. tree + 3 of the document whose ring is `cells` and starts at `start`
        const auto ringQuad = [&](const uint32_t* cells, uint32_t start, int32_t tree) {
            const uint32_t at = static_cast<uint32_t>(tree + 4 * kRing) / 4 + start;
            const uint32_t bytes = __builtin_amdgcn_alignbyte(cells[(at + 1) % kRing], cells[at % kRing],
                                                              static_cast<uint32_t>(tree) & 3u);
            return make_uint4(bytes & 0xffu, (bytes >> 8) & 0xffu, (bytes >> 16) & 0xffu, bytes >> 24);
        };
        if (group > 0 && (done < count || !lastShare)) {
            // inside a row: a group's whole lines per document (fewer behind a share's last, shorter group)
            uint32_t* row = blockOut + (tid / kDocThreads) * treeCount;
            const uint32_t* cells = ring + (tid / kDocThreads) * kPitch;
            const int32_t groupTrees = done - group;
#pragma unroll
            for (uint32_t pass = 0; pass < kDocsPerBlock / kDocsPerPass; ++pass) {
                const int32_t behind = static_cast<int32_t>((reinterpret_cast<uintptr_t>(row) / 4) % kLeafIndexLine);
                const uint4 quad = ringQuad(cells, ringStart(tid / kDocThreads), quadTree - behind);
                if (pass * kDocsPerPass + tid / kDocThreads < blockDocs && quadTree - group < groupTrees) {
                    StoreQuad<STREAM>(row + (quadTree - behind), quad);
                }
                row += kDocsPerPass * treeCount;
                cells += kDocsPerPass * kPitch;
            }
            continue;
        }
        for (uint32_t d = tid / kDocThreads; d < blockDocs; d += kDocsPerPass) {
            uint32_t* row = blockOut + d * treeCount;
            const int32_t behind = static_cast<int32_t>((reinterpret_cast<uintptr_t>(row) / 4) % kLeafIndexLine);
            // whole lines only, but for the row's first and last
            const int32_t begin = group > 0 ? group - behind : firstShare ? 0 : lead - behind;
            const int32_t end = done == count && lastShare ? count : done - behind;
            for (int32_t tree = quadTree - behind; tree < end; tree += GROUP) {
                const uint4 quad = ringQuad(ring + d * kPitch, ringStart(d), tree);
                if (tree >= begin && tree + 4 <= end) {
                    *reinterpret_cast<uint4*>(row + tree) = quad;
                } else {
                    const uint32_t values[4] = {quad.x, quad.y, quad.z, quad.w};
#pragma unroll
                    for (int32_t i = 0; i < 4; ++i) {
                        if (tree + i >= begin && tree + i < end) {
                            row[tree + i] = values[i];
                        }
                    }
                }
            }
        }
    }
}

// Re-lays bins out as the reference does: blocks of 128 documents, [block][bucket][doc in block],
// the last block packed with its own document count (cpu/quantization.h:357-365).
__global__ __launch_bounds__(256) void ExportBinsKernel(const uint8_t* __restrict__ bins, size_t docCount,
                                                        uint32_t bucketCount, uint8_t* __restrict__ out) {
    const size_t doc = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (doc >= docCount) {
        return;
    }
    const size_t refBlockStart = doc / 128 * 128;
    const size_t inBlock = doc - refBlockStart;
    const size_t blockDocs = min(static_cast<size_t>(128), docCount - refBlockStart);
    for (uint32_t b = 0; b < bucketCount; ++b) {
        out[refBlockStart * bucketCount + b * blockDocs + inBlock] = BinOfDoc(bins, doc, bucketCount, b);
    }
}

// ---- prediction types on the device --------------------------------------------------------
// TEvalResultProcessor::PostprocessBlock (catboost/libs/model/eval_processing.h:174-240) over blocks of
// min(128, total documents) documents, with the reference's exponent (fmath::expd_v / fmath::expd,
// contrib/libs/fmath/fmath.hpp:474-512, 565-648). The library is compiled without contraction, so each
// operation rounds on its own like the CPU's.

struct TFastExpDev {
    const unsigned long long* Mantissa;  // 2048 mantissas of 2^(i / 2048)
    double Scale, InvScale;              // 2048 / ln 2 and its reciprocal
};

// the arithmetic both forms share; `indexBits`: table index in bits 0..10, binary exponent above
__device__ __forceinline__ double FastExpCore(const TFastExpDev& c, double x, double rounded, unsigned long long indexBits) {
    constexpr int kTableBits = 11;
    const double kMagic = static_cast<double>(3ull << 51);
    constexpr unsigned long long kAdjust = (1ull << (kTableBits + 10)) - (1ull << kTableBits);
    const unsigned long long mantissa = c.Mantissa[indexBits & ((1u << kTableBits) - 1)];
    const unsigned long long power = (((indexBits + kAdjust) >> kTableBits) << 52) | mantissa;
    double t = rounded - kMagic;
    t = t * c.InvScale;
    t = t - x;
    double y = 3.0000000027955394 - t;
    y = y * (t * t);
    y = y * 0.16666666685227835064;
    y = y - t;
    y = y + 1.0;
    return y * __longlong_as_double(static_cast<long long>(power));
}

// element `index` of a run of `count` values handed to the exponent at once: the first count & ~3 take
// the vector form (clamped argument, NaN -> upper clamp), the rest the scalar form (0 / +inf outside)
__device__ __forceinline__ double FastExpAt(const TFastExpDev& c, double v, size_t index, size_t count) {
    const double kMagic = static_cast<double>(3ull << 51);
    if (index < (count & ~size_t(3))) {
        v = v < 709.78272569338397 ? v : 709.78272569338397;
        v = v > -708.39641853226408 ? v : -708.39641853226408;
        double d = v * c.Scale;
        d = d + kMagic;
        return FastExpCore(c, v, d, static_cast<unsigned long long>(__double_as_longlong(d)));
    }
    if (v <= -708.39641853226408) {
        return 0.0;
    }
    if (v >= 709.78271289338397) {
        return __longlong_as_double(0x7ff0000000000000ll);
    }
    double d = v * c.Scale;
    d = d + kMagic;
    const long long low = static_cast<long long>(static_cast<int>(static_cast<unsigned int>(__double_as_longlong(d))));
    return FastExpCore(c, v, d, static_cast<unsigned long long>(low));
}

constexpr int kPredRaw = 0, kPredExponent = 1, kPredRmseWithUncertainty = 2, kPredProbability = 3, kPredClass = 4,
              kPredMultiProbability = 5;  // EApiPredictionType, catboost/libs/model_interface/c_api.h:50-57

// One thread per document of a chunk that starts at document `firstDoc` of `totalDocs`.
// raw[doc * dim + k] -> out (doc values for Class, doc * dim values otherwise). raw == out is allowed
// except for Class with dim > 1. Softmax, and Class and MultiProbability of many dimensions, have the kernels below.
__global__ __launch_bounds__(256) void ApplyPredictionTypeKernel(int type, uint32_t dim, size_t firstDoc,
                                                                 size_t totalDocs, size_t docCount, TFastExpDev c,
                                                                 const double* raw, double* out) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= docCount) {
        return;
    }
    const size_t doc = firstDoc + i;
    const size_t blockSize = totalDocs < 128 ? totalDocs : 128;
    const size_t inBlock = doc % blockSize;
    const size_t blockDocs = min(blockSize, totalDocs - (doc - inBlock));  // documents of this document's block
    const double* r = raw + i * dim;
    if (type == kPredClass) {
        if (dim == 1) {
            out[i] = r[0] > 0.0 ? 1.0 : 0.0;
        } else {
            uint32_t best = 0;
            double top = r[0];
            for (uint32_t k = 1; k < dim; ++k) {
                const double v = r[k];
                if (top < v) {  // std::max_element: the first largest
                    top = v;
                    best = k;
                }
            }
            out[i] = static_cast<double>(best);
        }
        return;
    }
    double* o = out + i * dim;
    if (dim == 1) {
        const double v = r[0];
        if (type == kPredProbability) {
            o[0] = 1. / (1. + FastExpAt(c, -v, inBlock, blockDocs));
        } else if (type == kPredExponent) {
            o[0] = FastExpAt(c, v, inBlock, blockDocs);
        } else {
            o[0] = v;
        }
        return;
    }
    if (type == kPredRmseWithUncertainty) {
        for (uint32_t k = 0; k < dim; ++k) {
            double v = r[k];
            if (k == 1) {
                v = FastExpAt(c, v * 2.0, 0, 1);
            }
            o[k] = v;
        }
    } else if (type == kPredMultiProbability) {
        for (uint32_t k = 0; k < dim; ++k) {
            o[k] = 1. / (1. + FastExpAt(c, -r[k], inBlock * dim + k, blockDocs * dim));
        }
    } else {
        for (uint32_t k = 0; k < dim; ++k) {
            o[k] = r[k];
        }
    }
}

// CalcSoftmax (eval_processing.h:15-27) of two to eight dimensions, a document's values in the registers of its thread; raw == out
// is allowed. In loops over a dimension of the call's every exponential was stored and, as out may be raw, loaded again for the
// division, and no load went past a store, so they waited for memory; here a document's loads are in flight together. A launch:
// 100 000 documents of three dimensions 4.3 -> 2.7 us, 500 000 of eight 92.3 -> 17.8 (64 MB; a copy takes 12), 1 000 000 of two
// 11.9 -> 6.4. Eight dimensions are 16 registers per array; more take the kernel below. A kernel of its own, since its registers
// cost the other types' waves (Class of 1 000 000 documents of two dimensions 4.0 -> 4.5 us with both in one).
template <uint32_t DIM>
__global__ __launch_bounds__(256) void SoftmaxKernel(size_t docCount, TFastExpDev c, const double* raw, double* out) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= docCount) {
        return;
    }
    const double* r = raw + i * DIM;
    double* o = out + i * DIM;
    double v[DIM];
#pragma unroll
    for (uint32_t k = 0; k < DIM; ++k) {
        v[k] = r[k];
    }
    double top = v[0];
#pragma unroll
    for (uint32_t k = 1; k < DIM; ++k) {
        top = top < v[k] ? v[k] : top;
    }
    double sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < DIM; ++k) {
        v[k] = FastExpAt(c, v[k] - top, k, DIM);
        sum += v[k];
    }
#pragma unroll
    for (uint32_t k = 0; k < DIM; ++k) {
        o[k] = v[k] / sum;
    }
}

// f(k, r[k]) for k = 0 .. dim - 1, the loads of a turn of eight in flight together and before what f stores in its places of r
template <typename F>
__device__ __forceinline__ void ForEachInTurns(const double* r, uint32_t dim, const F& f) {
    constexpr uint32_t kTurn = 8;
    for (uint32_t first = 0; first < dim; first += kTurn) {
        double v[kTurn];
#pragma unroll
        for (uint32_t j = 0; j < kTurn; ++j) {
            v[j] = r[min(first + j, dim - 1)];
        }
#pragma unroll
        for (uint32_t j = 0; j < kTurn; ++j) {
            if (first + j < dim) {
                f(first + j, v[j]);
            }
        }
    }
}

// Many dimensions: softmax of more than eight (its exponentials computed twice, which costs less than storing and loading them),
// Class and MultiProbability from the two lines on. Arguments as ApplyPredictionTypeKernel, whose loop has one load in flight.
// Workgroups of one wave: few documents of many dimensions spread over every CU. A launch, that loop -> this kernel: Class of
// 500 000 documents of eight dimensions 9.5 -> 7.1 us (400 000 of five 4.2 -> 4.4, 1 000 000 of two 4.0 -> 5.9), MultiProbability of
// 500 000 of eight 65 -> 28, 15 000 of four 3.3 -> 2.8 (100 000 of three 3.4 -> 3.5); softmax of 200 000 of ten 51 -> 22,
// of 20 000 of a hundred 114 -> 55 (71 with workgroups of four waves).
constexpr uint32_t kManyDimsClass = 8, kManyDimsMultiProbability = 4;

__global__ __launch_bounds__(64) void ApplyPredictionTypeManyKernel(int type, uint32_t dim, size_t firstDoc, size_t totalDocs,
                                                                    size_t docCount, TFastExpDev c, const double* raw, double* out) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= docCount) {
        return;
    }
    const double* r = raw + i * dim;
    double* o = out + i * dim;
    if (type == kPredMultiProbability) {
        const size_t doc = firstDoc + i;
        const size_t blockSize = totalDocs < 128 ? totalDocs : 128;
        const size_t inBlock = doc % blockSize;
        const size_t blockDocs = min(blockSize, totalDocs - (doc - inBlock));  // documents of this document's block
        ForEachInTurns(r, dim, [&](uint32_t k, double v) {
            o[k] = 1. / (1. + FastExpAt(c, -v, inBlock * dim + k, blockDocs * dim));
        });
        return;
    }
    uint32_t best = 0;
    double top = r[0];
    ForEachInTurns(r, dim, [&](uint32_t k, double v) {
        if (top < v) {  // std::max_element: the first largest
            top = v;
            best = k;
        }
    });
    if (type == kPredClass) {
        out[i] = static_cast<double>(best);
        return;
    }
    double sum = 0;
    ForEachInTurns(r, dim, [&](uint32_t k, double v) { sum += FastExpAt(c, v - top, k, dim); });
    ForEachInTurns(r, dim, [&](uint32_t k, double v) { o[k] = FastExpAt(c, v - top, k, dim) / sum; });
}

// Leaf values of a model in another layout, a workgroup per row: what other kernels' tables of them are made of, once per model. On the
// host each table was a second pass over the leaves and a transfer of them: building an evaluator of 1000 trees of depth 8 over 200
// features (one such table) 3.25 -> 2.45 ms, of 2000 of depth 6 and ten dimensions 7.7 -> 5.9. A launch takes 6 us for 2 MB of leaf values
// read and written, 8 for 10 MB, 21 for 10 MB in ten dimensions (a lane writes ten values in a row).
struct TLeafRow {
    uint64_t Destination;  // of its first value, in values
    uint32_t Source;       // of the tree's first value
    uint32_t Levels;       // four bits per bit of the row's index: the bit of the tree's leaf index that it is, or kLeafRowNoLevel
    uint32_t Leaves;       // of the row that are the tree's, the others are zeros
    uint32_t Pitch;        // leaves of the row, with kLeafRowFolded
};
constexpr uint32_t kLeafRowNoLevel = 15, kLeafRowInOrder = 0x76543210u;
constexpr uint32_t kLeafRowFolded = 0x80000000u;  // index i of the row stands at i ^ (i >> 1)

__global__ __launch_bounds__(64) void PlaceLeavesKernel(const TLeafRow* __restrict__ rows, uint32_t dim, const double* __restrict__ leaves,
                                                        double* __restrict__ out) {
    const TLeafRow row = rows[blockIdx.x];
    for (uint32_t leaf = threadIdx.x; leaf < (row.Pitch & ~kLeafRowFolded); leaf += 64) {
        uint32_t from = 0;
#pragma unroll
        for (uint32_t bit = 0; bit < 8; ++bit) {
            const uint32_t level = row.Levels >> 4 * bit & 15;
            from |= level != kLeafRowNoLevel ? (leaf >> bit & 1) << level : 0u;
        }
        for (uint32_t k = 0; k < dim; ++k) {
            out[row.Destination + static_cast<size_t>(row.Pitch & kLeafRowFolded ? leaf ^ (leaf >> 1) : leaf) * dim + k] =
                leaf < row.Leaves ? leaves[row.Source + static_cast<size_t>(from) * dim + k] : 0.0;
        }
    }
}

__global__ void FillBiasKernel(double* __restrict__ out, size_t count, const double* __restrict__ bias, int dim) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < count) {
        out[i] = bias[i % dim];
    }
}

// Clears `dwords` 32-bit words. A kernel rather than hipMemsetAsync, so that callers may capture the
// launch into a HIP graph.
__global__ void FillZeroKernel(uint32_t* __restrict__ out, size_t dwords) {
    const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < dwords; i += stride) {
        out[i] = 0;
    }
}

}  // namespace cbamd::dev
