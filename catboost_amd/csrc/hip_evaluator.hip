// Host side of the HIP evaluator: model upload, kernel launches, host staging.
#include "hip_evaluator.h"
#include "exchange_plan.h"
#include "fast_exp.h"
#include "kernels.hip.h"
#include "ns_layout.h"

#include <hip/hip_ext.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <future>
#include <iterator>
#include <limits>
#include <map>
#include <numeric>
#include <string>
#include <system_error>
#include <thread>
#include <tuple>
#include <vector>

// Bin buffer of the entry point that allocates nothing (THipEvaluator::CalcDeviceNoAlloc): every GPU the
// library runs on holds one copy of this array, at its own address, until the process ends. In host code
// the name is only a handle for hipGetSymbolAddress; kernels get the address that call returns.
static __device__ __align__(256) unsigned char scratch[cbamd::THipEvaluator::kNoAllocScratchBytes];

namespace cbamd {

namespace {

void HipCheck(hipError_t e, const char* what) {
    if (e != hipSuccess) {
        throw TModelError(std::string("HIP error in ") + what + ": " + hipGetErrorString(e));
    }
}
#define HIP_CHECK(expr) HipCheck((expr), #expr)

template <typename T>
class TDeviceVec {
public:
    TDeviceVec() = default;
    ~TDeviceVec() { Reset(); }
    TDeviceVec(const TDeviceVec&) = delete;
    TDeviceVec& operator=(const TDeviceVec&) = delete;

    void Reset() {
        if (Ptr) {
            (void)hipFree(Ptr);
            Ptr = nullptr;
            Cap = 0;
        }
    }
    void Upload(const std::vector<T>& host) {
        Reserve(std::max<size_t>(host.size(), 1));
        if (!host.empty()) {
            HIP_CHECK(hipMemcpy(Ptr, host.data(), host.size() * sizeof(T), hipMemcpyHostToDevice));
        }
    }
    // grow-only
    void Reserve(size_t count) {
        if (count > Cap) {
            Reset();
            HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&Ptr), count * sizeof(T)));
            Cap = count;
        }
    }
    T* Get() const { return Ptr; }
    size_t Capacity() const { return Cap; }

private:
    T* Ptr = nullptr;
    size_t Cap = 0;
};

template <typename T, unsigned FLAGS = hipHostMallocDefault>
class TPinnedVec {
public:
    ~TPinnedVec() { Reset(); }
    void Reset() {
        if (Ptr) {
            (void)hipHostFree(Ptr);
            Ptr = nullptr;
            Cap = 0;
        }
    }
    // true: the memory is new
    bool Reserve(size_t count) {
        if (count <= Cap) {
            return false;
        }
        Reset();
        HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&Ptr), count * sizeof(T), FLAGS));
        Cap = count;
        return true;
    }
    T* Get() const { return Ptr; }

private:
    T* Ptr = nullptr;
    size_t Cap = 0;
};

// The calling thread's current device for as long as this lives; its own again afterwards.
class TDeviceGuard {
public:
    explicit TDeviceGuard(int deviceId) {
        HIP_CHECK(hipGetDevice(&Previous));
        HIP_CHECK(hipSetDevice(deviceId));
    }
    ~TDeviceGuard() { (void)hipSetDevice(Previous); }
    TDeviceGuard(const TDeviceGuard&) = delete;
    TDeviceGuard& operator=(const TDeviceGuard&) = delete;

private:
    int Previous = 0;
};

// Calls that a capture elsewhere in the process would forbid (waits, copies) on streams of this file's own, which no
// capture knows: this thread may make them for as long as this lives.
class TCaptureGuard {
public:
    TCaptureGuard() { HIP_CHECK(hipThreadExchangeStreamCaptureMode(&Mode)); }
    ~TCaptureGuard() { (void)hipThreadExchangeStreamCaptureMode(&Mode); }
    TCaptureGuard(const TCaptureGuard&) = delete;
    TCaptureGuard& operator=(const TCaptureGuard&) = delete;

private:
    hipStreamCaptureMode Mode = hipStreamCaptureModeRelaxed;
};

// A kernel that uses more than 64 KB of dynamic LDS has to be told so once (per device); the largest size asked
// for so far is remembered, so that the attribute is not set again on every launch.
// The code object of the assembly kernels, loaded once per device and kept for the life of the process: every
// evaluator of a device shares it (a few megabytes of code and some milliseconds of loading otherwise per model).
hipModule_t SharedRegModule(const void* image) {
    static std::mutex lock;
    static std::vector<std::pair<int, hipModule_t>> loaded;
    int device = 0;
    HIP_CHECK(hipGetDevice(&device));
    std::lock_guard<std::mutex> guard(lock);
    for (const auto& item : loaded) {
        if (item.first == device) {
            return item.second;
        }
    }
    hipModule_t module = nullptr;
    HIP_CHECK(hipModuleLoadData(&module, image));
    loaded.emplace_back(device, module);
    return module;
}

void EnsureDynamicLds(const void* kernel, size_t bytes) {
    if (bytes <= 64 * 1024) {
        return;
    }
    static std::mutex lock;
    static std::vector<std::pair<std::pair<int, const void*>, size_t>> granted;
    int device = 0;
    HIP_CHECK(hipGetDevice(&device));
    std::lock_guard<std::mutex> guard(lock);
    for (auto& item : granted) {
        if (item.first.first == device && item.first.second == kernel) {
            if (item.second >= bytes) {
                return;
            }
            HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
            item.second = bytes;
            return;
        }
    }
    HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
    granted.push_back({{device, kernel}, bytes});
}

// Address of `scratch` on a device, asked for once per device, with that device current.
uint8_t* NoAllocScratchOfCurrentDevice(int deviceId) {
    static std::mutex lock;
    static std::vector<uint8_t*> perDevice;
    std::lock_guard<std::mutex> guard(lock);
    if (perDevice.size() <= static_cast<size_t>(deviceId)) {
        perDevice.resize(static_cast<size_t>(deviceId) + 1, nullptr);
    }
    if (perDevice[deviceId] == nullptr) {
        void* ptr = nullptr;
        HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        CBAMD_ENSURE(ptr != nullptr, "the device holds no copy of the no-allocation bin buffer");
        perDevice[deviceId] = static_cast<uint8_t*>(ptr);
    }
    return perDevice[deviceId];
}

// Code object of the register-resident evaluate kernels (assembled from the output of
// gen_eval_reg_kernel.py at build time).
alignas(4096) const unsigned char kEvalRegCodeObject[] = {
#include "eval_reg_kernel_co.inc"
};

// Must match gen_eval_reg_kernel.py: kernel arguments, variants, trees per LDS buffer.
struct TEvalRegArgs {
    const void* Bins;
    const void* Rows;
    const void* Leaves;
    void* Out;
    uint32_t DocCount;
    uint32_t BlockCount;
    uint32_t TreeBlocks;
    uint32_t Flags;
    double Scale;
    const double* Bias;
    uint32_t BucketCount;
    uint32_t Dim;
    uint32_t FirstDim;
    uint32_t StoreDims;
};
static_assert(sizeof(TEvalRegArgs) == 80, "kernel argument block shared by the register-resident and the fused kernels");

struct TEvalRegLaunchArgs {
    TEvalRegArgs Reg;
    uint32_t TreeBlocksPerSlice;  // one slice: all tree blocks
    uint32_t SlicesPerGroup;      // slices of a workgroup (grid.y * SlicesPerGroup cover the trees)
    const uint32_t* RegMap;       // read when Reg.Flags has kRegFlagMapped: where each bins register comes from
};
static_assert(sizeof(TEvalRegLaunchArgs) == 96, "kernel argument block of the register-resident kernels");
constexpr uint32_t kRegFlagMapped = 8;
constexpr uint32_t kRegFlagPlainTable = 16;  // kernels of several dimensions and 64 leaves: the leaf table is not folded
constexpr uint32_t kRegFlagPairTable = 32;   // kernels of four and six dimensions and 64 leaves: nor that, but in pieces of two dimensions
// what a mapped bins register holds of its bucket's bins (bits 16.. of a map entry)
constexpr uint32_t kRegMapAsIs = 0, kRegMapLow = 1, kRegMapHigh = 2;  // bin, min(bin, 127), max(bin - 127, 0)

// argument block of the exchange kernels (gen_eval_exchange_kernel.py)
struct TEvalExchangeArgs {
    const void* Bins;
    const void* WaveTable;
    const void* Records;
    const void* ExtraRows;
    const void* Leaves;
    double* Out;
    const double* Bias;
    double Scale;
    uint32_t DocCount;
    uint32_t Rounds;
    uint32_t BlockBytes;
    uint32_t Unused;
};
static_assert(sizeof(TEvalExchangeArgs) == 80, "kernel argument block of the exchange kernels");
struct TFusedExchangeArgs {
    TEvalExchangeArgs Walk;  // no bins; the wave table of the fused kernels
    const float* Rows;
    const void* Tiles;
    uint32_t StrideBytes;
    uint32_t TileCount;
    const void* OneHot;
};
static_assert(sizeof(TFusedExchangeArgs) == 112, "kernel argument block of the fused exchange kernels");
constexpr int kFusedExchange = 3;  // FusedLayoutFor: flat rows, the fused exchange kernel

struct TEvalRegVariant {
    uint32_t Buckets;
    uint32_t Waves;
    uint32_t Pitch;   // dimensions per launch = doubles per leaf row
    uint32_t Leaves;  // leaf rows per tree (64: trees of depth <= 6)
    bool Mixed;       // 32-dword level tables, compare form chosen per tree
    bool Six;         // every bin at most 64: even levels compare into bit 6, two levels share a merge
    bool Folds;       // the leaf tables are folded (64 leaves: or as they are, by a flag)
    bool PairWalk;    // 64 leaves: or in pieces of two dimensions, by another
    const char* Name;
};
// kEvalRegVariants: gen_eval_reg_kernel.py's kernels, those of fewer registers first, with what their leaf tables have to look like;
// ExchangeFoldsLeaves: whether the exchange kernels of a depth read folded rows. Written by the generator beside the kernels.
#include "eval_reg_tables.inc"
constexpr int kRegMaxDepth = 10;  // deepest tree of the register kernels (one-dimensional models; 8 otherwise)

// Fused kernels (binarize + evaluate in one launch, bins only ever in registers): shapes of
// gen_eval_reg_kernel.py's FUSED_SHAPES, each in a plain and a six-bit form, and each of these in a form that
// walks six levels instead of eight (models of depth <= 6), listed before the eight-level form of its shape.
struct TFusedVariant {
    uint32_t Buckets;  // bins registers = 16 per unit of sixteen columns
    uint32_t Waves;
    bool Six;
    uint32_t Levels;
    const char* Name;
    bool Columns = false;  // column-major documents
};
constexpr TFusedVariant kFusedVariants[] = {
    {64, 8, false, 6, "cbamd_fused_b64_w8_d6"},
    {64, 8, true, 6, "cbamd_fused_b64_w8_d6_s"},
    {64, 8, false, 8, "cbamd_fused_b64_w8"},
    {64, 8, true, 8, "cbamd_fused_b64_w8_s"},
    {80, 8, false, 6, "cbamd_fused_b80_w8_d6"},
    {80, 8, true, 6, "cbamd_fused_b80_w8_d6_s"},
    {80, 8, false, 8, "cbamd_fused_b80_w8"},
    {80, 8, true, 8, "cbamd_fused_b80_w8_s"},
    {208, 4, false, 6, "cbamd_fused_b208_w4_d6"},
    {208, 4, true, 6, "cbamd_fused_b208_w4_d6_s"},
    {208, 4, false, 8, "cbamd_fused_b208_w4"},
    {208, 4, true, 8, "cbamd_fused_b208_w4_s"},
    {64, 8, false, 6, "cbamd_fused_cols_b64_w8_d6", true},
    {64, 8, true, 6, "cbamd_fused_cols_b64_w8_d6_s", true},
    {64, 8, false, 8, "cbamd_fused_cols_b64_w8", true},
    {64, 8, true, 8, "cbamd_fused_cols_b64_w8_s", true},
    {80, 8, false, 6, "cbamd_fused_cols_b80_w8_d6", true},
    {80, 8, true, 6, "cbamd_fused_cols_b80_w8_d6_s", true},
    {80, 8, false, 8, "cbamd_fused_cols_b80_w8", true},
    {80, 8, true, 8, "cbamd_fused_cols_b80_w8_s", true},
    {160, 4, false, 6, "cbamd_fused_cols_b160_w4_d6", true},
    {160, 4, true, 6, "cbamd_fused_cols_b160_w4_d6_s", true},
    {160, 4, false, 8, "cbamd_fused_cols_b160_w4", true},
    {160, 4, true, 8, "cbamd_fused_cols_b160_w4_s", true},
    {208, 4, false, 6, "cbamd_fused_cols_b208_w4_d6", true},
    {208, 4, true, 6, "cbamd_fused_cols_b208_w4_d6_s", true},
    {208, 4, false, 8, "cbamd_fused_cols_b208_w4", true},
    {208, 4, true, 8, "cbamd_fused_cols_b208_w4_s", true},
};
constexpr uint32_t kLateStartCus = 256;     // CUs of the device whose second workgroups the fused kernels of rows start late
constexpr uint32_t kFusedUnitColumns = 16;
constexpr uint32_t kFusedUnitDwords = 40;   // sixteen lo, sixteen scale, flags, padding
constexpr uint32_t kFusedMaxSteps = 4;
constexpr size_t kFusedImageBytes = 32 * 1024;
constexpr size_t kFusedLutOffset = 16 * 1024;

struct TEvalFusedArgs {
    TEvalRegArgs Reg;       // Bins: the delay of the CUs' second workgroups (rows); Leaves: the border table images, then the leaf table
    const void* Floats;
    const void* Units;
    uint32_t StrideBytes;
    uint32_t UnitCount;
};
static_assert(sizeof(TEvalFusedArgs) == 104, "kernel argument block of the fused kernels");

// Trees of a slice of a small batch: two of the kernels' tree blocks, and not fewer than 32 trees (kernels with
// large leaf tables have blocks of 2 or 4 trees, and a slice costs a partial sum per document)
uint32_t RegSliceTrees(uint32_t treeBlock) {
    return std::max(2 * treeBlock, 32u);
}

// Slices that one workgroup of a sliced launch walks. The chip holds `resident` workgroups at a time (two to four per CU, by
// the variant's registers and LDS), and a workgroup pays for its bins, its first tables and its end what about one slice
// costs: the number with the cheapest sum over the generations is taken (half a slice to two and a half as the price
// measured the same). A slice per workgroup -> this rule, 1000 trees of depth 8 over 200 features, whole device call:
// 50 000 documents 99 -> 78 us, 100 000 151 -> 100, 200 000 255 -> 157; 20 000 (no more workgroups than fit) 62 -> 57.
// Two per CU assumed where three fit: 100 003 documents of 500 trees and three dimensions 87.3 us instead of 81.3.
uint32_t RegSlicesPerGroup(size_t groups, uint32_t slices, size_t resident) {
    uint32_t best = 1;
    size_t bestCost = std::numeric_limits<size_t>::max();
    for (uint32_t k = 1; k <= slices; ++k) {
        const size_t generations = (groups * ((slices + k - 1) / k) + resident - 1) / resident;
        const size_t cost = generations * (k + 1);
        if (cost < bestCost) {
            best = k;
            bestCost = cost;
        }
    }
    return best;
}

// Whether a variant's leaf tables are folded for trees of this depth: leaf l at l ^ (l >> 1)
bool FoldsLeaves(const TEvalRegVariant& v, int depth) {
    return v.Folds && (v.Leaves == 256 || depth == 6);
}

// ... or, of 64 leaves, hold pieces of two dimensions, 16 bytes per leaf (those of 256 leaves always do)
bool PairsDimensions(const TEvalRegVariant& v, int depth) {
    return v.Pitch > 1 && (v.Leaves == 256 || (v.PairWalk && depth <= 4));
}

// trees per LDS buffer of a variant: a power of two, at most 16, buffer at most 32 KB
uint32_t RegTreeBlock(const TEvalRegVariant& v) {
    uint32_t block = 16;
    while (block > 1 && block * v.Leaves * v.Pitch * 8 > 32 * 1024) {
        block /= 2;
    }
    return block;
}

// The variant for a model: one-dimensional models take the smallest register file that holds
// their buckets; others the pitch that needs the fewest launches (then the smallest such pitch).
// mixed: the model has one-hot splits, or bins above 128 that stay in one register.
const TEvalRegVariant* PickRegVariant(uint32_t buckets, uint32_t dim, uint32_t maxDepth, bool mixed, bool six,
                                      uint32_t minVariantBuckets = 0) {
    const TEvalRegVariant* best = nullptr;
    uint32_t bestLaunches = 0;
    // A model of several dimensions with more buckets than the kernels of two and more dimensions hold (they
    // need registers for their sums) takes the one-dimensional kernels, a launch per dimension: every launch
    // walks the trees again, which still is several times faster than leaving the registers.
    for (int onePerLaunch = 0; onePerLaunch < 2 && !best; ++onePerLaunch) {
        if (onePerLaunch && dim == 1) {
            break;
        }
        for (const auto& v : kEvalRegVariants) {
            // trees of depth <= 6: 64 leaf rows and six levels
            const bool shallow = maxDepth <= 6;
            const uint32_t leaves = maxDepth > 8 ? 1024u : shallow ? 64u : 256u;
            if (buckets > v.Buckets || v.Buckets < minVariantBuckets || (dim == 1 || onePerLaunch) != (v.Pitch == 1) ||
                v.Leaves != leaves || v.Mixed != mixed || v.Six != six) {
                continue;
            }
            const uint32_t launches = (dim + v.Pitch - 1) / v.Pitch;
            if (!best || launches < bestLaunches || (launches == bestLaunches && dim > 1 && v.Pitch < best->Pitch)) {
                best = &v;
                bestLaunches = launches;
            }
        }
    }
    return best;
}

}  // namespace

// The end of a stage (binarize, evaluate) as an event that the stage's last launch carries: the event of a dispatch costs
// nothing, where one that is recorded behind it is a packet of its own between two kernels. A stage whose last launch does
// not take the event has it recorded. A kernel of 60 us and the wait for it: 73.5 us with start and end recorded, 71.0 with
// the launch's event; kernels of 60 and 20 us with three recorded events 98.2, 91.6 with the launches' events. Whole calls:
// 100 003 documents of three dimensions 93.2 -> 91.1 us, a fused call of 1M documents 108.7 -> 107.3.
struct THipEvaluator::TStageEnd {
    hipEvent_t Event = nullptr;
    hipEvent_t Take() {
        const hipEvent_t e = Event;
        Event = nullptr;
        return e;
    }
    void Close(hipStream_t s) {
        if (const hipEvent_t e = Take()) {
            HIP_CHECK(hipEventRecord(e, s));
        }
    }
};

namespace {

hipEvent_t TakeEnd(THipEvaluator::TStageEnd* end) {
    return end ? end->Take() : nullptr;
}

// a launch that carries `end` (a plain one without: those may be captured)
template <typename TKernel, typename... TArgs>
void LaunchWithEnd(TKernel kernel, dim3 grid, dim3 block, size_t lds, hipStream_t s, hipEvent_t end, TArgs... args) {
    if (end) {
        hipExtLaunchKernelGGL(kernel, grid, block, static_cast<uint32_t>(lds), s, nullptr, end, 0, args...);
    } else {
        hipLaunchKernelGGL(kernel, grid, block, lds, s, args...);
    }
}

// The same for a kernel of the code object, `args` its argument block. (gridX * threads has 32 bits, which a batch of less than 2^29
// documents does not leave: 1024 threads for 256 documents at the most.)
template <typename TArgs>
void LaunchModuleWithEnd(hipFunction_t kernel, uint32_t gridX, uint32_t gridY, uint32_t threads, hipStream_t s, hipEvent_t end,
                         TArgs& args) {
    size_t size = sizeof(args);
    void* config[] = {HIP_LAUNCH_PARAM_BUFFER_POINTER, &args, HIP_LAUNCH_PARAM_BUFFER_SIZE, &size, HIP_LAUNCH_PARAM_END};
    if (end) {  // (this call counts work-items, the other workgroups)
        HIP_CHECK(hipExtModuleLaunchKernel(kernel, gridX * threads, gridY, 1, threads, 1, 1, 0, s, nullptr, config, nullptr, end, 0));
    } else {
        HIP_CHECK(hipModuleLaunchKernel(kernel, gridX, gridY, 1, threads, 1, 1, 0, s, nullptr, config));
    }
}

// Diagnostic switches, read from the environment when an evaluator is built (cb_hip_evaluator.h lists them) and
// only in a process that sets CATBOOST_AMD_TEST_SWITCHES=1: a production process that happens to have one of the
// names in its environment keeps the default kernels. They choose between kernels that give the same results;
// tests use them to reach every kernel with one model.
struct TKernelSwitches {
    bool RegKernel = true;        // CATBOOST_AMD_REG_KERNEL=0: no register-resident assembly kernels
    bool RegSix = true;           // CATBOOST_AMD_REG_SIX=0: no six-bit form of those kernels, nor of the pair-tile kernel
    bool CtrTile = true;          // CATBOOST_AMD_CTR_TILE=0: the plain CTR kernel instead of the tile kernel
    uint32_t RegMinBuckets = 0;   // CATBOOST_AMD_REG_MIN_BUCKETS=n: only register kernels that hold n buckets or more
    bool Fused = true;            // CATBOOST_AMD_FUSED=0: binarize and evaluate always as two launches
    bool SmallBatch = true;       // CATBOOST_AMD_SMALL_BATCH=0: small batches are not spread over slices of the trees
    bool LevelOrder = true;       // CATBOOST_AMD_LEVEL_ORDER=0: register kernels keep the model's order of a tree's levels
    bool PairTile = true;         // CATBOOST_AMD_PAIR_TILE=0: the half-tile kernel with one tree per wave
    bool Exchange = true;         // CATBOOST_AMD_EXCHANGE=0: the pair-tile kernel for batches of every size
    bool RowTile = true;          // CATBOOST_AMD_ROW_TILE=0: the tile kernel that broadcasts a tree's levels from a lane
    bool RegSplit = true;         // CATBOOST_AMD_REG_SPLIT=0: a bucket keeps to one register: more than 127 values send a model to the mixed kernels
    uint32_t NsWaves = 0;         // CATBOOST_AMD_NS_WAVES=4|6|8|10|11|12|16: shapes of the non-symmetric LDS kernel with so many waves or none
    uint32_t FlagTicket = 0;      // CATBOOST_AMD_FLAG_TICKET=n: the first ticket of few host documents' flags is n + 1; their waits are counted
    bool CountFlagged = false;
    uint32_t FlagWaitUs = 200;    // CATBOOST_AMD_FLAG_WAIT_US=n: microseconds after which such a call waits for its launch instead

    static TKernelSwitches FromEnvironment() {
        const auto off = [](const char* name) {
            const char* v = std::getenv(name);
            return v != nullptr && v[0] == '0';
        };
        TKernelSwitches k;
        const char* gate = std::getenv("CATBOOST_AMD_TEST_SWITCHES");
        if (gate == nullptr || gate[0] != '1') {
            return k;
        }
        k.RegKernel = !off("CATBOOST_AMD_REG_KERNEL");
        k.RegSix = !off("CATBOOST_AMD_REG_SIX");
        k.CtrTile = !off("CATBOOST_AMD_CTR_TILE");
        k.Fused = !off("CATBOOST_AMD_FUSED");
        k.LevelOrder = !off("CATBOOST_AMD_LEVEL_ORDER");
        k.SmallBatch = !off("CATBOOST_AMD_SMALL_BATCH");
        k.PairTile = !off("CATBOOST_AMD_PAIR_TILE");
        k.Exchange = !off("CATBOOST_AMD_EXCHANGE");
        k.RowTile = !off("CATBOOST_AMD_ROW_TILE");
        k.RegSplit = !off("CATBOOST_AMD_REG_SPLIT");
        if (const char* v = std::getenv("CATBOOST_AMD_NS_WAVES")) {
            k.NsWaves = static_cast<uint32_t>(std::strtoul(v, nullptr, 10));
        }
        if (const char* v = std::getenv("CATBOOST_AMD_FLAG_TICKET")) {
            k.FlagTicket = static_cast<uint32_t>(std::strtoul(v, nullptr, 10));
            k.CountFlagged = true;
        }
        if (const char* v = std::getenv("CATBOOST_AMD_FLAG_WAIT_US")) {
            k.FlagWaitUs = static_cast<uint32_t>(std::strtoul(v, nullptr, 10));
        }
        if (const char* v = std::getenv("CATBOOST_AMD_REG_MIN_BUCKETS")) {
            k.RegMinBuckets = static_cast<uint32_t>(std::strtoul(v, nullptr, 10));
        }
        return k;
    }
};

// log2 of the LDS slots per bucket of the row binarize kernel: the smallest count that still
// exceeds the largest bucket of the model
int BinarizeLog2Slots(uint32_t maxBucketValues) {
    return maxBucketValues < 32 ? 5 : maxBucketValues < 64 ? 6 : maxBucketValues < 128 ? 7 : 8;
}

// Host twin of dev::GridCell: the same two roundings and the same truncation.
uint32_t GridCell(float v, float lo, float scale) {
    volatile float d = v - lo;
    volatile float t = d * scale;
    const float tt = t;
    if (!(tt > 0.0f)) {
        return 0;
    }
    if (tt >= 4294967296.0f) {
        return dev::kLutCells - 1;
    }
    return std::min<uint32_t>(static_cast<uint32_t>(tt), dev::kLutCells - 1);
}

// The uniform grid over a float bucket's sorted borders that starts the border search: lowest border,
// cells per unit, the search steps that cover the tallest cell, and per cell the number of borders in
// lower cells (what a search in that cell may skip).
struct TBucketGrid {
    float Lo = 0.0f;
    float Scale = 0.0f;
    uint32_t Steps = 0;
    uint32_t Start[dev::kLutCells] = {};
};

// Steps and starts from the borders of each cell
void SetGridStarts(const uint32_t* population, TBucketGrid* g) {
    const uint32_t tallest = *std::max_element(population, population + dev::kLutCells);
    while ((1u << g->Steps) - 1 < tallest) {
        ++g->Steps;
    }
    uint32_t start = 0;
    for (int c = 0; c < dev::kLutCells; ++c) {
        g->Start[c] = start;
        start += population[c];
    }
}

TBucketGrid MakeBucketGrid(const std::vector<float>& borders) {
    TBucketGrid g;
    if (borders.empty()) {
        return g;
    }
    g.Lo = borders.front();
    const float span = borders.back() - g.Lo;
    if (std::isfinite(g.Lo) && std::isfinite(span) && span > 0.0f) {
        g.Scale = static_cast<float>(dev::kLutCells) / span;
        if (!std::isfinite(g.Scale)) {
            g.Scale = 0.0f;
        }
    } else {
        g.Lo = 0.0f;
    }
    uint32_t population[dev::kLutCells] = {};
    for (float x : borders) {
        ++population[GridCell(x, g.Lo, g.Scale)];
    }
    SetGridStarts(population, &g);
    return g;
}

// The grid of the fused kernels: a value's cell is the nearest whole number of 255 times its place, clamped to 0 .. 1, in fp32. The place
// rises with the value, so the borders of lower cells are below the value and those of higher cells are not.
TBucketGrid MakeFusedGrid(const std::vector<float>& borders, bool columnMajor) {
    TBucketGrid g;
    if (borders.empty()) {
        return g;
    }
    const float span = borders.back() - borders.front();
    const float scale = 1.0f / span, bias = -borders.front() * scale;
    if (std::isfinite(span) && span > 0.0f && std::isfinite(scale) && std::isfinite(bias)) {
        g.Lo = columnMajor ? bias : borders.front();
        g.Scale = scale;
    }
    uint32_t population[dev::kLutCells] = {};
    for (float x : borders) {
        const float place = columnMajor ? std::fma(x, g.Scale, g.Lo) : (x - g.Lo) * g.Scale;
        const double clamped = place > 0.0f ? std::min(place, 1.0f) : 0.0f;  // (NaN: 0)
        ++population[static_cast<uint32_t>(std::nearbyint(clamped * (dev::kLutCells - 1)))];
    }
    SetGridStarts(population, &g);
    return g;
}

constexpr size_t kMaxTileLdsBytes = 160 * 1024;

// Batches of SmallBatchKernel and FewDocumentsKernel, in documents times passes over the dimensions; beyond come the binarize
// and register kernels in slices of the trees, for some models before (TakesSmallBatchOnDevice). FewDocumentsKernel against SmallBatchKernel: 512 documents 18 against 21 us, 1024 24 against 21.
constexpr size_t kSmallBatchDocs = 16384;
constexpr size_t kFewDocs = 640;
// ... of host calls, whose features are at most so many bytes: more go through the pipeline of chunks
constexpr size_t kSmallHostBytes = size_t(16) << 20;

// Workgroups up to which a host batch's launch sets flags: every one of them orders its results before its flag, over PCIe.
// 1000 trees of depth 6 over 100 features, whole call with the launch's event and with flags: 1 row 20.6 and 18.3 us, 4 rows
// 20.5 and 18.5, 16 20.8 and 19.8, 24 21.0 and 20.2, 200 23.6 and 28.3.
constexpr size_t kFlaggedGroups = 16;

// Workgroups wanted of a leaf index launch: 200 000 documents * 1000 trees (782 blocks, 2 workgroups per CU) take 225 us as
// 782 workgroups, 200 as 2346, 216 as 4692 (shorter runs of a row, the bins read more often), launches back to back.
constexpr size_t kLeafIndexWorkgroups = 2048;

// Size of all tables of CTR bins together up to which they are (usually) at most a quarter full instead of half: three times
// an L2. Half and a quarter full, 1M documents, whole call: 36 projections of 1000 hashes (2.3 MB a quarter full) 408 and
// 315 us, 4000 (9 MB) 459 and 421, 8000 (19 MB) 527 and 561, 16 000 (38 MB) 624 and 687; 12 projections of 8000 (6 MB) 225 and
// 208, 16 000 (13 MB) 247 and 245, 32 000 (25 MB) 274 and 293, 115 000 (100 MB) 356 and 352. (Batches of 100 000 documents
// gain up to 10 % at any of these sizes, by 7 to 14 us.)
constexpr size_t kCtrRoomyBytes = size_t(12) << 20;

// The cache between the L2s and HBM. What is larger is not found there by its next reader.
constexpr size_t kMemorySideCacheBytes = size_t(256) << 20;

// LDS of the tile kernel without leaf regions: the bins of 256 documents and the accumulator
size_t TileLdsBytes(uint32_t buckets, int dchunk) {
    return ((static_cast<size_t>(buckets) * dev::kDocsPerBlock + 7) & ~size_t(7)) +
           static_cast<size_t>(dev::kDocsPerBlock) * dchunk * sizeof(double);
}

// LDS of EvalNonSymmetricLdsKernel: 8 KB per wave (its entries, then rows of bins), the other rows of bins, the
// accumulator
size_t NsLdsKernelBytes(uint32_t buckets, uint32_t waves, uint32_t entries, uint32_t dims) {
    return static_cast<size_t>(dev::NsLdsTileRows(buckets, waves, entries)) * 256 + dev::kDocsPerBlock * sizeof(double) * dims;
}

// dimensions that one workgroup of EvalNonSymmetricLdsKernel sums (a model of more walks its trees once per slice)
uint32_t NsLdsDims(int dim) {
    return dim == 1 ? 1 : dim == 2 ? 2 : 4;
}

// Few buckets leave LDS for larger regions (fewer units, larger trees) at a given number of waves, and 249 to 312 buckets
// for ten or eleven waves where trees of more than 1536 entries would leave eight. Evaluate launch, 500 000 documents, 500 trees
// of depth 10 over 100 features: 580 us with eight waves of 2048 entries, 544 with twelve of 1536, 506 with twelve of 2048, 508 with
// sixteen of 1536, 484 with sixteen of 2048; over 300 features 598 with eight, 559 with ten, 544 with eleven of 1792, 557 with
// twelve of 1536; 1M, 500 of depth 6 over 60 753 with eight, 630 with twelve of 1536, 546 with sixteen of 1024; three dimensions, 500 000, 300 of
// depth 8 over 100 408 with eight, 369 with twelve of 1536, 351 with sixteen of 1024.
// The model's shape is the one with the least steps / speed. Steps (a unit takes as many as its tallest tree, and the three top levels for
// three more) per time, relative to eight waves, measured over eight models of depth 6 to 10, 100 to 300 features, one to three dimensions:
//   16 x 1024 1.16 .. 1.38   16 x 1536 1.09 .. 1.34   16 x 2048 1.20 .. 1.23   12 x 1536 1.11 .. 1.23   12 x 2048 1.09 .. 1.15
//   11 x 1792 1.08 .. 1.17   10 x 2048 1.05 .. 1.09   (counting the top levels as no step or as five: the same within 0.04)
// (a region that is fuller takes longer per step, so a shape's speed falls as its units shrink). The figures below were set on
// two models and a walk that began at the root; they still give seven of these eight the fastest shape and one (depth 10 over 300
// features) the second, 2 % behind. Of five models of 20 to 60 features two had a faster one: there two workgroups of eight waves
// share a CU (100 trees of depth 8 over 50 features 163 us against the 189 of the 16 x 1024 that is taken, 500 of depth 9 over 20 476 against
// 487), which the rule does not know.
// The shapes of EvalNonSymmetricLdsKernel, most waves first.
struct TNsLdsShape {
    uint32_t Waves;
    uint32_t Entries;
    double Speed;  // steps per unit of time, relative to the 8-wave shape
};
constexpr TNsLdsShape kNsLdsShapes[] = {{16, 1024, 1.45}, {16, 1536, 1.37}, {16, 2048, 1.35}, {12, 1536, 1.26}, {12, 2048, 1.2},
                                        {11, 1792, 1.08}, {10, 2048, 1.04}, {8, 2048, 1.0},   {6, 2048, 0.8},   {4, 2048, 0.55}};

// Calls `tryShape` with the waves and the entries of one shape after another until it returns true.
template <typename TTry, size_t... I>
bool LaunchOfShape(const TTry& tryShape, std::index_sequence<I...>) {
    return (tryShape(std::integral_constant<int, kNsLdsShapes[I].Waves>(), std::integral_constant<int, kNsLdsShapes[I].Entries>()) || ...);
}

// A unit of EvalNonSymmetricLdsKernel: up to three trees that a wave walks side by side out of its LDS region
struct TNsUnit {
    uint32_t Trees[dev::kNsUnitTrees];
    uint32_t TreeCount;
    uint32_t Entries;
    uint32_t Height;
};

// The trees (rows: first entry, steps behind the exits, entry count, unused) by falling height, the order in which PackNsUnits takes them
std::vector<uint32_t> OrderNsTrees(const std::vector<uint32_t>& rows, size_t treeCount) {
    std::vector<uint32_t> order(treeCount);
    std::iota(order.begin(), order.end(), 0u);
    std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) {
        return rows[a * 4 + 1] != rows[b * 4 + 1] ? rows[a * 4 + 1] > rows[b * 4 + 1] : rows[a * 4 + 2] > rows[b * 4 + 2];
    });
    return order;
}

// Groups the trees into units of at most `limit` entries. A unit takes as many steps as its tallest tree, so the trees go in by
// falling height, and every tree joins the fullest of the recently opened units that still has room for it (trees need not be
// neighbours in the model: the kernel's sums are partial sums per wave anyway). False when a tree exceeds the limit.
bool PackNsUnits(const std::vector<uint32_t>& rows, const std::vector<uint32_t>& order, uint32_t limit, std::vector<TNsUnit>* units) {
    if (std::any_of(order.begin(), order.end(), [&](uint32_t t) { return rows[t * 4 + 2] > limit; })) {
        return false;
    }
    constexpr size_t kWindow = 64;  // open units looked at per tree
    std::vector<size_t> open;
    for (const uint32_t t : order) {
        const uint32_t size = rows[t * 4 + 2];
        size_t best = open.size();
        for (size_t i = open.size() > kWindow ? open.size() - kWindow : 0; i < open.size(); ++i) {
            const TNsUnit& unit = (*units)[open[i]];
            if (unit.Entries + size <= limit && (best == open.size() || unit.Entries > (*units)[open[best]].Entries)) {
                best = i;
            }
        }
        if (best == open.size()) {
            TNsUnit unit{};
            unit.Height = rows[t * 4 + 1];
            units->push_back(unit);
            open.push_back(units->size() - 1);
        }
        TNsUnit& unit = (*units)[open[best]];
        unit.Trees[unit.TreeCount++] = t;
        unit.Entries += size;
        if (unit.TreeCount == static_cast<uint32_t>(dev::kNsUnitTrees)) {
            open.erase(open.begin() + static_cast<std::ptrdiff_t>(best));
        }
    }
    return true;
}

// Dimensions that a workgroup of the row-tile kernel sums at a time. Two: the sums, the values in flight and three
// trees' worth of values fetched ahead then fit a wave's registers at sixteen waves. A walk for four dimensions takes
// 1.8 times as long (C3's trees over 300 features: 3.6 against 2.06 ms), so only models of three or four dimensions
// with 64 leaves per tree take it, for one walk instead of two.
uint32_t RowTileDims(uint32_t maxDepth, int dim) {
    return dim == 1 ? 1 : maxDepth <= 6 && (dim == 3 || dim == 4) ? 4 : 2;
}

// LDS of the row-tile kernel: 256 documents' bins, the accumulator, a tree's leaf values per wave
size_t RowTileLdsBytes(uint32_t buckets, uint32_t maxDepth, uint32_t dims, uint32_t waves) {
    const size_t leaves = maxDepth <= 6 ? 64 : 256;
    return ((static_cast<size_t>(buckets) * 256 + 15) & ~size_t(15)) + dev::kDocsPerBlock * dims * sizeof(double) +
           static_cast<size_t>(waves) * leaves * dims * sizeof(double);
}

// Waves per workgroup of the row-tile kernel: eight when two workgroups then share a CU, else sixteen if LDS
// has room for their regions, else eight; 0 when the tile leaves no room for eight regions.
uint32_t RowTileWaves(uint32_t buckets, uint32_t maxDepth, int dim) {
    const uint32_t dims = RowTileDims(maxDepth, dim);
    if (2 * RowTileLdsBytes(buckets, maxDepth, dims, dev::kTileWaves) <= kMaxTileLdsBytes) {
        return dev::kTileWaves;
    }
    if (RowTileLdsBytes(buckets, maxDepth, dims, dev::kWideTileWaves) <= kMaxTileLdsBytes) {
        return dev::kWideTileWaves;
    }
    return RowTileLdsBytes(buckets, maxDepth, dims, dev::kTileWaves) <= kMaxTileLdsBytes ? dev::kTileWaves : 0;
}

// LDS of the deep-tile kernel: 256 documents' bins and the accumulator
size_t DeepTileLdsBytes(uint32_t rows, int dims) {
    return ((static_cast<size_t>(rows) * 256 + 15) & ~size_t(15)) + static_cast<size_t>(dims) * dev::kDocsPerBlock * sizeof(double);
}

// dimensions that a workgroup of the deep-tile kernel sums per walk of the trees
int DeepTileDims(int dim) {
    return dim == 1 ? 1 : 2;
}

// LDS of the quad-tile kernel: 64 documents' bins, then per wave the leaf values of four trees (later the partial sums)
size_t QuadTileLdsBytes(uint32_t rows, int maxd, uint32_t waves) {
    return ((static_cast<size_t>(rows) * 64 + 15) & ~size_t(15)) +
           static_cast<size_t>(waves) * 4 * (size_t(1) << maxd) * sizeof(double);
}

// Waves per workgroup of the quad-tile kernel: eight, or four when the rows leave room for no more; 0: no room
uint32_t QuadTileWaves(uint32_t rows, int maxd) {
    return QuadTileLdsBytes(rows, maxd, 8) <= kMaxTileLdsBytes ? 8u : QuadTileLdsBytes(rows, maxd, 4) <= kMaxTileLdsBytes ? 4u : 0u;
}

// LDS of the pair-tile kernel: 128 documents' bins, then per wave the leaf values of one tree of 256 leaves or two of 64;
// the same area takes one partial sum per wave and document at the end
size_t PairTileLdsBytes(uint32_t buckets, int maxd) {
    return ((static_cast<size_t>(buckets) * 128 + 15) & ~size_t(15)) +
           static_cast<size_t>(dev::kPairWaves) * std::max<size_t>(size_t(1) << maxd, 128) * sizeof(double);
}

// Trees from which the pair-tile kernel is the faster of it and the tile kernel where both could take a model of one dimension, by the
// evaluate launch for 100 000 and 1M documents, tile and pair-tile: 625 buckets, ranges of 300 trees of depth 8 53 and 54, 431 and 456 us, 600
// trees 89 and 82, 722 and 660; 100 of depth 6 28 and 27, 232 and 232, 200 39 and 32, 312 and 266. 620 buckets, one of more than 127 values,
// 400 trees of depth 8 74 and 80, 606 and 631 us, 600 90 and 83, 715 and 656; 300 of these and 8000 trees 1011 and 791, 8040 and 6083.
// (Up to 32 768 documents, a workgroup per CU, the pair-tile kernel is ahead with any number: 300 trees 28 and 17.)
constexpr uint32_t PairTrees(uint32_t maxDepth) {
    return maxDepth <= 6 ? 150 : 500;
}

// dimensions the tile kernel accumulates per pass over the trees (and the pitch of its padded leaf rows)
int TileChunk(int dim) {
    return dim == 1 ? 1 : dim == 2 ? 2 : dim <= 4 ? 4 : dim <= 8 ? 8 : dim <= 12 ? 12 : 16;
}

// Level-order tables of non-symmetric trees for EvalNonSymmetricTileKernel (its comment has the
// entry format). The walk they encode is CalcIndexesNonSymmetric, cpu/evaluator_impl.cpp:462-493:
// from a node, the chosen side's diff leads to the next node and a zero diff ends the walk at the
// node's own leaf (NonSymmetricNodeIdToLeafId). A zero side becomes a terminal entry of its own.
// usable = false when a tree does not fit the 16-bit offsets of an entry.
// The compact tables (EvalNonSymmetricLdsKernel) are filled when the model, of any dimension, has at most 1023 buckets and
// no tree above dev::kNsLdsEntries entries (one-hot splits count two).
void BuildLevelOrderTrees(const TModelTrees& trees, int dim, const std::vector<uint32_t>& firstLeaf,
                          TDeviceVec<uint32_t>* entriesOut, TDeviceVec<uint32_t>* rowsOut, bool* usable, bool* noXor,
                          std::vector<uint32_t>* compactEntries, std::vector<uint32_t>* compactRows, std::vector<uint32_t>* topNodes,
                          std::vector<double>* valuesByEntry, bool* compactUsable) {
    struct TItem {
        uint32_t Node;        // model node, or the parent node of a synthetic terminal
        bool Terminal;
        bool Second = false;     // the second test of a one-hot split taken apart (see unfold)
        uint32_t LeftEntry = 0;  // of a second test: the entry of the split's left side
        int64_t CopyOf = -1;     // an entry that repeats an earlier one of the tree: same test, same children
    };
    struct TUnfolded {
        std::vector<TItem> Order;                                // breadth first, the two children of an entry side by side
        std::vector<uint32_t> Level;
        std::vector<std::pair<uint32_t, uint32_t>> Children;     // entry index of (false side, true side); terminals: unused
        uint32_t Height = 0;
        bool Fits = true;
    };
    // Breadth-first order of a tree's entries. A tree whose nodes share children (the loader only checks that
    // every step stays inside the tree) unfolds into more entries than it has nodes, up to 2^depth: the walk
    // stops as soon as the entries no longer fit the 16-bit offsets, and the model goes to the kernel that
    // follows the step nodes.
    // splitOneHot: the compact entries only know "bin >= splitIdx". A one-hot split, bin == v, becomes two of
    // them: "bin >= v" (false: the model's left side) and behind its true side "bin >= v + 1" (false: the
    // model's right side, the bins are equal; true: the left side again). The entry of the left side is
    // repeated there, not its subtree: the copy names the same pair of children.
    const auto unfold = [&](uint32_t root, bool splitOneHot, TUnfolded* unfolded) {
        TUnfolded& u = *unfolded;
        u.Order.clear();
        u.Level.clear();
        u.Children.clear();
        u.Height = 0;
        u.Order.push_back({root, false});
        u.Level.push_back(0);
        for (size_t i = 0; i < u.Order.size() && u.Order.size() * 8 <= 0xffffu; ++i) {
            if (u.Order[i].CopyOf >= 0) {
                const size_t original = static_cast<size_t>(u.Order[i].CopyOf);  // an earlier index: already visited
                const int64_t keep = u.Order[i].CopyOf;
                u.Order[i] = u.Order[original];
                u.Order[i].CopyOf = keep;
                u.Children.push_back(u.Children[original]);
                if (u.Order[i].Terminal) {
                    u.Height = std::max(u.Height, u.Level[i]);
                }
                continue;
            }
            const TItem item = u.Order[i];
            const auto& st = trees.NonSymmetricStepNodes[item.Node];
            const bool terminal = item.Terminal || (!item.Second && st.LeftSubtreeDiff == 0 && st.RightSubtreeDiff == 0);
            u.Order[i].Terminal = terminal;
            if (terminal) {
                u.Height = std::max(u.Height, u.Level[i]);
                u.Children.emplace_back(0, 0);
                continue;
            }
            const uint32_t diffs[2] = {st.LeftSubtreeDiff, st.RightSubtreeDiff};
            const auto pushSide = [&](int side) {
                const uint32_t index = static_cast<uint32_t>(u.Order.size());
                if (diffs[side] == 0) {
                    u.Order.push_back({item.Node, true});
                } else {
                    u.Order.push_back({item.Node + diffs[side], false});
                }
                u.Level.push_back(u.Level[i] + 1);
                return index;
            };
            const bool oneHot = splitOneHot && trees.RepackedBins[item.Node].XorMask != 0;
            uint32_t child[2];
            if (!oneHot) {
                child[0] = pushSide(0);
                child[1] = pushSide(1);
            } else if (!item.Second) {
                child[0] = pushSide(0);
                child[1] = static_cast<uint32_t>(u.Order.size());
                TItem second{item.Node, false};
                second.Second = true;
                second.LeftEntry = child[0];
                u.Order.push_back(second);
                u.Level.push_back(u.Level[i] + 1);
            } else {
                child[0] = pushSide(1);
                child[1] = static_cast<uint32_t>(u.Order.size());
                TItem copy{item.Node, false};
                copy.CopyOf = item.LeftEntry;
                u.Order.push_back(copy);
                u.Level.push_back(u.Level[i] + 1);
            }
            u.Children.emplace_back(child[0], child[1]);
        }
        u.Fits = u.Order.size() * 8 <= 0xffffu;
    };
    const size_t treeCount = trees.GetTreeCount();
    *noXor = true;
    for (const auto& rb : trees.RepackedBins) {
        *noXor = *noXor && rb.XorMask == 0;
    }
    std::vector<uint32_t> entries, rows(treeCount * 4, 0);
    *usable = true;
    *compactUsable = trees.EffectiveBinFeaturesBucketCount <= 1023;
    compactRows->assign(treeCount * 4, 0);
    TUnfolded plain, split;  // (these are filled anew by every tree)
    std::vector<uint32_t> left;
    TNsTreeLayout layout;
    for (size_t t = 0; t < treeCount && *usable; ++t) {
        const uint32_t root = static_cast<uint32_t>(trees.TreeStartOffsets[t]);
        const size_t firstEntry = entries.size() / 2;
        unfold(root, false, &plain);
        if (!plain.Fits) {
            *usable = false;
            break;
        }
        const std::vector<TItem>& order = plain.Order;
        const auto& children = plain.Children;
        for (size_t i = 0; i < order.size(); ++i) {
            const TItem item = order[i];
            uint32_t x, y;
            if (item.Terminal) {
                const uint32_t leafRel = (trees.NonSymmetricNodeIdToLeafId[item.Node] - firstLeaf[t]) / static_cast<uint32_t>(dim);
                if (leafRel > 0xffffu) {
                    *usable = false;
                    break;
                }
                x = 0;
                y = leafRel | (static_cast<uint32_t>(i * 8) << 16);
            } else {
                const auto& rb = trees.RepackedBins[item.Node];
                x = *noXor ? (static_cast<uint32_t>(rb.FeatureIndex) << 8) | (static_cast<uint32_t>(rb.SplitIdx) << 24)
                           : static_cast<uint32_t>(rb.FeatureIndex) | (static_cast<uint32_t>(rb.XorMask) << 16) |
                                 (static_cast<uint32_t>(rb.SplitIdx) << 24);
                y = (children[i].first * 8) | ((children[i].second * 8) << 16);
            }
            entries.push_back(x);
            entries.push_back(y);
        }
        rows[t * 4 + 0] = static_cast<uint32_t>(firstEntry);
        rows[t * 4 + 1] = plain.Height;
        rows[t * 4 + 2] = firstLeaf[t];
        // compact layout: the top nodes apart, the eight exits behind them, then pairs of children, so that every pair starts even
        if (!*compactUsable || !*usable) {
            *compactUsable = false;
            continue;
        }
        if (!*noXor) {
            unfold(root, true, &split);
        }
        const TUnfolded& compact = *noXor ? plain : split;
        *compactUsable = compact.Fits && compact.Order.size() + 1 <= static_cast<size_t>(dev::kNsLdsEntries);
        if (!*compactUsable) {
            continue;
        }
        const auto splitOf = [&](size_t i) {
            const auto& rb = trees.RepackedBins[compact.Order[i].Node];
            if (rb.XorMask == 0) {
                return static_cast<uint32_t>(rb.SplitIdx);
            }
            // a one-hot split holds ~value in its xor mask (and 255 as its split index)
            return ((~static_cast<uint32_t>(rb.XorMask)) & 0xffu) + (compact.Order[i].Second ? 1u : 0u);
        };
        const auto bucketOf = [&](size_t i) { return static_cast<uint32_t>(trees.RepackedBins[compact.Order[i].Node].FeatureIndex); };
        left.resize(compact.Order.size());
        for (size_t i = 0; i < left.size(); ++i) {
            left[i] = compact.Order[i].Terminal ? kNsNoItem : compact.Children[i].first;  // the true side always follows the false side
        }
        LayOutNsTree(left, &layout);
        // the seven nodes of the top levels; false for every bin where there is none
        for (const uint32_t i : layout.TopItems) {
            *compactUsable = *compactUsable && (i == kNsNoItem || splitOf(i) <= 255);
            topNodes->push_back(i == kNsNoItem ? 0u : bucketOf(i) << 8 | (256u - splitOf(i)));
        }
        topNodes->push_back(0u);
        const std::vector<uint32_t>& placed = layout.Items;
        const size_t count = (placed.size() + 7) / 8 * 8;  // (a tree's exits start at a multiple of 32 bytes)
        (*compactRows)[t * 4 + 0] = static_cast<uint32_t>(compactEntries->size());
        (*compactRows)[t * 4 + 1] = layout.Steps;
        (*compactRows)[t * 4 + 2] = static_cast<uint32_t>(count);
        *compactUsable = *compactUsable && count <= static_cast<size_t>(dev::kNsLdsEntries);
        compactEntries->resize(compactEntries->size() + count);
        valuesByEntry->resize(compactEntries->size() * dim, 0.0);
        uint32_t* entryAt = compactEntries->data() + compactEntries->size() - count;
        double* valueAt = valuesByEntry->data() + valuesByEntry->size() - count * dim;
        for (uint32_t at = 0; at < count; ++at) {
            if (at >= placed.size()) {
                entryAt[at] = NsTerminalEntry(at);
            } else if (compact.Order[placed[at]].Terminal) {
                entryAt[at] = NsTerminalEntry(layout.Next[at]);
                std::copy_n(trees.LeafValues.data() + trees.NonSymmetricNodeIdToLeafId[compact.Order[placed[at]].Node], dim, valueAt + static_cast<size_t>(at) * dim);
            } else {
                const uint32_t split = splitOf(placed[at]);
                *compactUsable = *compactUsable && split <= 255;
                entryAt[at] = (split & 0xffu) | bucketOf(placed[at]) << 8 | layout.Next[at] << 21;
            }
        }
    }
    *compactUsable = *compactUsable && *usable;
    if (*usable) {
        entriesOut->Upload(entries);
        rowsOut->Upload(rows);
    }
}

// Where the kernels read the model's features in a caller's data: the positions stored in the model, or
// those positions sent through a feature layout. The vector sizes a caller must provide follow the
// reference without a layout (the last feature of each list decides, model.h:494-541) and are the
// largest position read plus one with a layout.
struct TFeaturePositions {
    const TFeatureLayout* Layout = nullptr;
    size_t FlatVectorSize = 0;
    size_t MinFloatSize = 0;
    size_t MinCatSize = 0;

    TFeaturePosition Of(const TFloatFeature& f) const {
        return Layout ? Layout->Remap(f) : TFeaturePosition{f.Index, f.FlatIndex};
    }
    TFeaturePosition Of(const TCatFeature& c) const {
        return Layout ? Layout->Remap(c) : TFeaturePosition{c.Index, c.FlatIndex};
    }

    TFeaturePositions(const TModelTrees& trees, const TFeatureLayout* layout)
        : Layout(layout && layout->Defined() ? layout : nullptr)
    {
        if (!Layout) {
            FlatVectorSize = trees.GetFlatFeatureVectorExpectedSize();
            MinFloatSize = trees.MinimalSufficientFloatFeaturesVectorSize;
            MinCatSize = trees.MinimalSufficientCatFeaturesVectorSize;
            return;
        }
        for (const auto& f : trees.FloatFeatures) {
            if (f.UsedInModel() && f.Index >= 0 && f.FlatIndex >= 0) {
                const TFeaturePosition p = Of(f);
                FlatVectorSize = std::max(FlatVectorSize, static_cast<size_t>(p.FlatIndex) + 1);
                MinFloatSize = std::max(MinFloatSize, static_cast<size_t>(p.Index) + 1);
            }
        }
        for (const auto& c : trees.CatFeatures) {
            if (c.UsedInModel && c.Index >= 0 && c.FlatIndex >= 0) {
                const TFeaturePosition p = Of(c);
                FlatVectorSize = std::max(FlatVectorSize, static_cast<size_t>(p.FlatIndex) + 1);
                MinCatSize = std::max(MinCatSize, static_cast<size_t>(p.Index) + 1);
            }
        }
    }
};

// work(0) ... work(count - 1) on at most `threads` threads of the host, sixteen at the most; the first exception of any of
// them is thrown here.
template <typename TWork>
void RunOnThreads(size_t count, size_t threads, const TWork& work) {
    threads = std::min({threads, count, size_t(16), size_t(std::max(1u, std::thread::hardware_concurrency()))});
    std::atomic<size_t> next{0};
    std::exception_ptr failure;
    std::mutex failureLock;
    const auto take = [&] {
        for (size_t i; (i = next++) < count;) {
            try {
                work(i);
            } catch (...) {
                std::lock_guard<std::mutex> guard(failureLock);
                failure = failure ? failure : std::current_exception();
                next = count;
            }
        }
    };
    std::vector<std::thread> pool;
    pool.reserve(threads);
    try {
        for (size_t t = 1; t < threads; ++t) {
            pool.emplace_back(take);
        }
    } catch (const std::system_error&) {
        // fewer threads than asked for
    }
    take();
    for (auto& thread : pool) {
        thread.join();
    }
    if (failure) {
        std::rethrow_exception(failure);
    }
}

// Host tables of the exchange kernels, which take longer than all others of such a model together: made on threads of their own
// meanwhile. Building an evaluator of 5000 trees of depth 8 over 1016 features 16 -> 7.5 ms (with their leaf values copied on the device; the
// plan alone 9 -> 4 ms, one of its threads), 3.1 without them.
struct TExchangeTables {
    std::vector<TExchangeTree> Trees;
    std::vector<TExchangeColumn> Columns;      // fused form: none if the model does not qualify
    std::vector<uint32_t> ColumnOf, Pieces;
    uint32_t BucketCount = 0, MaxDepth = 0;
    bool Six = false;

    TExchangePlan Plan;
    std::vector<uint32_t> Tiles, OneHot;
    bool Planned = false, Tiled = false;

    void Build() {
        RunOnThreads(2, 2, [&](size_t part) {
            if (part == 0) {
                Planned = BuildExchangePlan(Trees, BucketCount, MaxDepth, Six, ColumnOf, &Plan);
            } else if (!Columns.empty()) {
                for (TExchangeColumn& column : Columns) {
                    if (column.Used && !column.OneHot) {
                        MakeExchangeGrid(Six, &column);
                    }
                }
                Tiled = BuildExchangeTiles(Columns, Pieces, Six, &Tiles, &OneHot);
            }
        });
    }
};

// One feature's value of one row of its table, static_ctr_provider.cpp:52-126: one branch per CTR type, the row null
// where the table does not know the hash. Single roundings throughout, as TModelCtr::Calc (online_ctr.h:290-293).
float CtrValueOfRow(const TModelCtr& ctr, const TCtrValueTable& table, const uint8_t* row) {
    const auto counter = [&](size_t i) {
        uint32_t v;
        std::memcpy(&v, row + 4 * i, 4);
        return v;
    };
    const auto asFloat = [](uint32_t v) { return static_cast<float>(static_cast<int32_t>(v)); };
    const int classes = table.TargetClassesCount;
    switch (ctr.Base.CtrType) {
        case ECtrType::BinarizedTargetMeanValue:
        case ECtrType::FloatTargetMeanValue: {
            if (!row) {
                return ctr.Calc(0.f, 0.f);
            }
            float sum;
            std::memcpy(&sum, row, 4);
            return ctr.Calc(sum, asFloat(counter(1)));
        }
        case ECtrType::Counter:
        case ECtrType::FeatureFreq:
            return ctr.Calc(row ? asFloat(counter(0)) : 0.f, static_cast<float>(table.CounterDenominator));
        case ECtrType::Buckets: {
            if (!row) {
                return ctr.Calc(0.f, 0.f);
            }
            uint32_t total = 0;
            for (int c = 0; c < classes; ++c) {
                total += counter(c);
            }
            return ctr.Calc(asFloat(counter(ctr.TargetBorderIdx)), asFloat(total));
        }
        case ECtrType::Borders: {
            if (!row) {
                return ctr.Calc(0.f, 0.f);
            }
            if (classes <= 2) {
                return ctr.Calc(asFloat(counter(1)), asFloat(counter(0) + counter(1)));
            }
            uint32_t good = 0, total = 0;
            for (int c = 0; c < classes; ++c) {
                total += counter(c);
                good += c > ctr.TargetBorderIdx ? counter(c) : 0u;
            }
            return ctr.Calc(asFloat(good), asFloat(total));
        }
    }
    return 0.f;
}

// The rows of a table in the order in which TDenseIndexHashView::GetIndex (helpers/dense_hash_view.h:46-56) would come
// upon them: `found(hash, row)` for every bucket that a look-up of its own hash reaches before an empty bucket.
template <typename TFound>
void ForEachCtrRow(const TCtrValueTable& table, const TFound& found) {
    const size_t bucketCount = table.IndexHashRaw.size() / 12, mask = bucketCount - 1;
    const auto bucket = [&](size_t at, uint64_t* hash, uint32_t* row) {
        std::memcpy(hash, table.IndexHashRaw.data() + 12 * at, 8);
        std::memcpy(row, table.IndexHashRaw.data() + 12 * at + 8, 4);
    };
    constexpr uint64_t kEmpty = ~uint64_t(0);
    uint64_t hash;
    uint32_t row;
    size_t start = 0;
    for (; start < bucketCount; ++start) {
        bucket(start, &hash, &row);
        if (hash == kEmpty) {
            break;
        }
    }
    size_t run = 0;  // taken buckets between the last empty one and this one
    for (size_t i = 1; i < bucketCount; ++i) {
        const size_t at = (start + i) & mask;
        bucket(at, &hash, &row);
        if (hash == kEmpty) {
            run = 0;
            continue;
        }
        if (((at - hash) & mask) <= run) {
            found(hash, row);
        }
        ++run;
    }
}

// Device tables of the model's CTR features (TStaticCtrProvider, catboost/libs/model/static_ctr_provider.cpp):
// per projection a descriptor, the projection itself (SetupBinFeatureIndexes, :142-178, resolved to bucket
// numbers and input columns) and one hash table that holds, per hash that any of the projection's tables of learned
// statistics knows, the bins of all the projection's CTR features (dev::TCtrGroupDev). Every row index and class index
// is checked here, so a damaged model fails at load instead of reading out of bounds.
// Appends one bucket entry per 254 borders of a CTR feature to the binarize bucket tables.
struct TCtrDeviceTables {
    TDeviceVec<uint32_t> Groups, Items, Table, Buckets, CatColumnsFlat, CatColumnsSplit;
    uint32_t CatColumnCount = 0;
    uint32_t GroupCount = 0;
};

void BuildCtrTables(const TModelTrees& trees, const TFeaturePositions& positions,
                    const std::vector<TCtrValueTable>& tables, std::vector<uint32_t>* srcFlat,
                    std::vector<uint32_t>* srcSplit, std::vector<uint32_t>* offsets, std::vector<uint32_t>* flags,
                    std::vector<uint32_t>* values, TCtrDeviceTables* result) {
    static_assert(sizeof(dev::TCtrGroupDev) == 32 && sizeof(dev::TCtrItemDev) == 16, "device CTR records changed size");
    std::vector<dev::TCtrGroupDev> groups;
    std::vector<dev::TCtrItemDev> items;
    std::vector<uint32_t> catColumnsFlat, catColumnsSplit;  // distinct categorical columns of all projections
    std::vector<bool> tableChecked(tables.size(), false);
    std::vector<uint32_t> tableRows(tables.size(), 0);

    // first bucket of every used float feature and of every one-hot feature
    std::vector<uint32_t> floatFirstBucket(trees.FloatFeatures.size(), 0), oneHotFirstBucket(trees.OneHotFeatures.size(), 0);
    uint32_t bucket = 0;
    for (size_t i = 0; i < trees.FloatFeatures.size(); ++i) {
        floatFirstBucket[i] = bucket;
        bucket += static_cast<uint32_t>((trees.FloatFeatures[i].Borders.size() + kMaxValuesPerBin - 1) / kMaxValuesPerBin);
    }
    for (size_t i = 0; i < trees.OneHotFeatures.size(); ++i) {
        oneHotFirstBucket[i] = bucket;
        bucket += static_cast<uint32_t>((trees.OneHotFeatures[i].Values.size() + kMaxValuesPerBin - 1) / kMaxValuesPerBin);
    }

    // the features: their tables, checked, and their buckets
    struct TFeature {
        size_t Table = 0;
        size_t RowBytes = 0;
        uint32_t FirstBucket = 0, BucketCount = 0;
    };
    std::vector<TFeature> features;
    std::vector<std::vector<size_t>> groupFeatures;
    for (const auto& feature : trees.CtrFeatures) {
        const TModelCtr& ctr = feature.Ctr;
        size_t t = 0;
        while (t < tables.size() && !(tables[t].ModelCtrBase == ctr.Base)) {
            ++t;
        }
        CBAMD_ENSURE(t < tables.size(), "Model has a CTR feature without its table of learned statistics");
        const TCtrValueTable& table = tables[t];
        const size_t bucketCount = table.IndexHashRaw.size() / 12;
        CBAMD_ENSURE(table.IndexHashRaw.size() % 12 == 0 && bucketCount > 0 && (bucketCount & (bucketCount - 1)) == 0 &&
                         bucketCount <= (size_t(1) << 31),
                     "Dense hash view must have 2^k buckets");
        // bytes of one row and the class indexes the CTR reads (static_ctr_provider.cpp:52-126)
        size_t rowBytes = 0;
        switch (ctr.Base.CtrType) {
            case ECtrType::BinarizedTargetMeanValue:
            case ECtrType::FloatTargetMeanValue:
                rowBytes = 8;
                break;
            case ECtrType::Counter:
            case ECtrType::FeatureFreq:
                rowBytes = 4;
                break;
            case ECtrType::Buckets:
                CBAMD_ENSURE(table.TargetClassesCount > 0 && ctr.TargetBorderIdx >= 0 &&
                                 ctr.TargetBorderIdx < table.TargetClassesCount,
                             "CTR target border index out of range");
                rowBytes = 4 * static_cast<size_t>(table.TargetClassesCount);
                break;
            case ECtrType::Borders:
                if (table.TargetClassesCount > 2) {
                    CBAMD_ENSURE(ctr.TargetBorderIdx >= 0 && ctr.TargetBorderIdx < table.TargetClassesCount,
                                 "CTR target border index out of range");
                    rowBytes = 4 * static_cast<size_t>(table.TargetClassesCount);
                } else {
                    rowBytes = 8;
                }
                break;
        }
        if (!tableChecked[t]) {
            tableChecked[t] = true;
            bool hasEmpty = false;
            uint32_t maxRow = 0;
            bool anyRow = false;
            for (size_t b = 0; b < bucketCount; ++b) {
                uint32_t w[3];
                std::memcpy(w, table.IndexHashRaw.data() + 12 * b, 12);
                if ((w[0] & w[1]) == 0xffffffffu) {
                    hasEmpty = true;
                } else {
                    maxRow = std::max(maxRow, w[2]);
                    anyRow = true;
                }
            }
            CBAMD_ENSURE(hasEmpty, "CTR index hash table has no empty bucket");
            CBAMD_ENSURE(maxRow != 0xffffffffu || !anyRow, "CTR value table is shorter than its index");
            tableRows[t] = anyRow ? maxRow + 1 : 0;
        }
        CBAMD_ENSURE(static_cast<size_t>(tableRows[t]) * rowBytes <= table.CTRBlob.size(),
                     "CTR value table is shorter than its index");
        TFeature f;
        f.Table = t;
        f.RowBytes = rowBytes;
        f.FirstBucket = static_cast<uint32_t>(srcFlat->size());
        for (size_t begin = 0; begin < feature.Borders.size(); begin += kMaxValuesPerBin) {
            const size_t end = std::min(begin + kMaxValuesPerBin, feature.Borders.size());
            std::vector<float> b;
            for (size_t i = begin; i < end; ++i) {
                if (!std::isnan(feature.Borders[i])) {
                    b.push_back(feature.Borders[i]);
                }
            }
            std::sort(b.begin(), b.end());
            for (float x : b) {
                uint32_t bits;
                std::memcpy(&bits, &x, 4);
                values->push_back(bits);
            }
            offsets->push_back(static_cast<uint32_t>(values->size()));
            srcFlat->push_back(0);
            srcSplit->push_back(0);
            flags->push_back(dev::kBucketFlagCtr);
        }
        f.BucketCount = static_cast<uint32_t>(srcFlat->size()) - f.FirstBucket;
        size_t g = 0;
        while (g < groupFeatures.size() &&
               !(trees.CtrFeatures[groupFeatures[g].front()].Ctr.Base.Projection == ctr.Base.Projection)) {
            ++g;
        }
        if (g == groupFeatures.size()) {
            groupFeatures.emplace_back();
        }
        groupFeatures[g].push_back(features.size());
        features.push_back(f);
    }

    std::vector<uint32_t> buckets;
    for (const std::vector<size_t>& members : groupFeatures) {
        const TFeatureCombination& projection = trees.CtrFeatures[members.front()].Ctr.Base.Projection;
        dev::TCtrGroupDev group{};
        group.ItemBegin = static_cast<uint32_t>(items.size());
        for (int catIndex : projection.CatFeatures) {
            const TCatFeature* cat = nullptr;
            for (const auto& c : trees.CatFeatures) {
                if (c.Index == catIndex && c.UsedInModel) {
                    cat = &c;
                }
            }
            CBAMD_ENSURE(cat != nullptr && cat->FlatIndex >= 0 && cat->Index >= 0,
                         "CTR projection refers to an unknown or unused categorical feature");
            const TFeaturePosition at = positions.Of(*cat);
            CBAMD_ENSURE(static_cast<size_t>(at.FlatIndex) < positions.FlatVectorSize &&
                             static_cast<size_t>(at.Index) < positions.MinCatSize,
                         "categorical feature position exceeds the model's feature vector size");
            uint32_t tileRow = 0;
            while (tileRow < catColumnsSplit.size() && catColumnsSplit[tileRow] != static_cast<uint32_t>(at.Index)) {
                ++tileRow;
            }
            if (tileRow == catColumnsSplit.size()) {
                catColumnsFlat.push_back(static_cast<uint32_t>(at.FlatIndex));
                catColumnsSplit.push_back(static_cast<uint32_t>(at.Index));
            }
            items.push_back({dev::kCtrItemCat, static_cast<uint32_t>(at.FlatIndex), static_cast<uint32_t>(at.Index), tileRow});
        }
        for (const auto& split : projection.BinFeatures) {
            bool found = false;
            for (size_t i = 0; i < trees.FloatFeatures.size() && !found; ++i) {
                const auto& ff = trees.FloatFeatures[i];
                if (ff.Index != split.FloatFeature) {
                    continue;
                }
                for (size_t b = 0; b < ff.Borders.size(); ++b) {
                    if (ff.Borders[b] == split.Split) {
                        const uint32_t at = floatFirstBucket[i] + static_cast<uint32_t>(b / kMaxValuesPerBin);
                        items.push_back({dev::kCtrItemBinGe, at, at, static_cast<uint32_t>(b % kMaxValuesPerBin) + 1});
                        found = true;
                        break;
                    }
                }
            }
            CBAMD_ENSURE(found, "CTR projection refers to a float split the model does not have");
        }
        for (const auto& split : projection.OneHotFeatures) {
            bool found = false;
            for (size_t i = 0; i < trees.OneHotFeatures.size() && !found; ++i) {
                const auto& oh = trees.OneHotFeatures[i];
                if (oh.CatFeatureIndex != split.CatFeatureIdx) {
                    continue;
                }
                for (size_t v = 0; v < oh.Values.size(); ++v) {
                    if (oh.Values[v] == split.Value) {
                        const uint32_t at = oneHotFirstBucket[i] + static_cast<uint32_t>(v / kMaxValuesPerBin);
                        items.push_back({dev::kCtrItemBinEq, at, at, static_cast<uint32_t>(v % kMaxValuesPerBin) + 1});
                        found = true;
                        break;
                    }
                }
            }
            CBAMD_ENSURE(found, "CTR projection refers to a one-hot split the model does not have");
        }
        group.ItemEnd = static_cast<uint32_t>(items.size());
        group.FirstBucket = static_cast<uint32_t>(buckets.size());
        for (size_t i : members) {
            for (uint32_t k = 0; k < features[i].BucketCount; ++k) {
                buckets.push_back(features[i].FirstBucket + k);
            }
            group.BucketCount += features[i].BucketCount;
        }
        group.EntryPieces = (8 + group.BucketCount + 15) / 16;
        groups.push_back(group);
    }

    // What the groups' tables take when the hashes of a projection's largest table fill at most half of one. Members of one
    // table follow each other, so that each table is gone through once.
    std::vector<std::vector<size_t>> groupOrder(groups.size());
    std::vector<size_t> groupEntries(groups.size(), 2);
    size_t indexBytes = 0;
    for (const TCtrValueTable& t : tables) {
        indexBytes += t.IndexHashRaw.size();
    }
    RunOnThreads(groups.size(), indexBytes >> 20, [&](size_t g) {
        const std::vector<size_t>& members = groupFeatures[g];
        std::vector<size_t>& order = groupOrder[g];
        order.resize(members.size());
        std::iota(order.begin(), order.end(), size_t(0));
        std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return features[members[a]].Table < features[members[b]].Table; });
        size_t keys = 0;  // of the largest table
        for (size_t i = 0; i < order.size(); ++i) {
            const size_t t = features[members[order[i]]].Table;
            if (i == 0 || t != features[members[order[i - 1]]].Table) {
                size_t rows = 0;
                ForEachCtrRow(tables[t], [&](uint64_t, uint32_t) { ++rows; });
                keys = std::max(keys, rows);
            }
        }
        while (groupEntries[g] < 2 * keys) {
            groupEntries[g] *= 2;
        }
    });
    // A quarter where all tables together then take no more than kCtrRoomyBytes: a wave's lookups take as many rounds as the
    // longest of its 256 probe sequences.
    size_t tableBytes = 0;
    for (size_t g = 0; g < groups.size(); ++g) {
        tableBytes += groupEntries[g] * groups[g].EntryPieces * 16;
    }
    if (2 * tableBytes <= kCtrRoomyBytes) {
        for (size_t& entries : groupEntries) {
            entries *= 2;
        }
    }

    // the table of group g: entries of a hash and its bins
    const auto buildTable = [&](size_t g) {
        dev::TCtrGroupDev& group = groups[g];
        const std::vector<size_t>& members = groupFeatures[g];
        std::vector<uint32_t> table, firstByte;  // ... of every member's bins in an entry
        uint32_t bytes = 0;
        for (size_t i : members) {
            firstByte.push_back(bytes);
            bytes += features[i].BucketCount;
        }
        // the bins of member i for a row of its table (null: unknown hash)
        const auto fillBins = [&](size_t i, const uint8_t* row, uint8_t* bins) {
            const TFeature& f = features[members[i]];
            const float value = CtrValueOfRow(trees.CtrFeatures[members[i]].Ctr, tables[f.Table], row);
            for (uint32_t k = 0; k < f.BucketCount; ++k) {
                const uint32_t begin = (*offsets)[f.FirstBucket + k], end = (*offsets)[f.FirstBucket + k + 1];
                const float* borders = reinterpret_cast<const float*>(values->data());
                // the number of borders below the value (none below a NaN)
                bins[firstByte[i] + k] = static_cast<uint8_t>(std::lower_bound(borders + begin, borders + end, value) - (borders + begin));
            }
        };
        const size_t entryDwords = 4 * static_cast<size_t>(group.EntryPieces);
        std::vector<uint32_t> unknown(entryDwords, 0);
        unknown[0] = unknown[1] = 0xffffffffu;
        for (size_t i = 0; i < members.size(); ++i) {
            fillBins(i, nullptr, reinterpret_cast<uint8_t*>(unknown.data() + 2));
        }
        // Tables of one projection were learned on the same documents and know the same hashes; where they do not, the
        // union may pass half of the entries, and the table is built again with twice as many.
        const std::vector<size_t>& order = groupOrder[g];
        size_t entries = groupEntries[g];
        const auto build = [&] {
            CBAMD_ENSURE(entries <= (size_t(1) << 31), "CTR tables are too large");
            table.clear();
            table.reserve(entries * entryDwords);
            for (size_t e = 0; e < entries; ++e) {
                table.insert(table.end(), unknown.begin(), unknown.end());
            }
            group.HashMask = static_cast<uint32_t>(entries - 1);
            std::vector<uint32_t> filledBy(entries, 0);  // a hash that a damaged table holds twice: the first one counts
            size_t taken = 0;
            bool fits = true;
            for (size_t first = 0, last = 0; first < order.size(); first = last) {
                const size_t t = features[members[order[first]]].Table;
                while (last < order.size() && features[members[order[last]]].Table == t) {
                    ++last;
                }
                ForEachCtrRow(tables[t], [&](uint64_t hash, uint32_t row) {
                    size_t at = static_cast<size_t>(hash) & (entries - 1);
                    const auto hashAt = [&] {
                        const uint32_t* e = table.data() + at * entryDwords;
                        return e[0] | (static_cast<uint64_t>(e[1]) << 32);
                    };
                    while (hashAt() != hash && hashAt() != ~uint64_t(0)) {
                        at = (at + 1) & (entries - 1);
                    }
                    uint32_t* entry = table.data() + at * entryDwords;
                    if (hashAt() != hash) {
                        if (!fits || 2 * (taken + 1) > entries) {
                            fits = false;
                            return;
                        }
                        ++taken;
                        entry[0] = static_cast<uint32_t>(hash);
                        entry[1] = static_cast<uint32_t>(hash >> 32);
                    }
                    if (filledBy[at] == last) {
                        return;
                    }
                    filledBy[at] = static_cast<uint32_t>(last);
                    for (size_t i = first; i < last; ++i) {
                        fillBins(order[i], tables[t].CTRBlob.data() + static_cast<size_t>(row) * features[members[order[i]]].RowBytes,
                                 reinterpret_cast<uint8_t*>(entry + 2));
                    }
                });
            }
            return fits;
        };
        while (!build()) {
            entries *= 2;
        }
        return table;
    };
    // The groups' tables, side by side on the host's threads: 8 categorical columns of 400 000 values each and 4 pairs of
    // them, 48 CTR features, 0.10 s; 0.87 on one thread.
    std::vector<std::vector<uint32_t>> groupTables(groups.size());
    RunOnThreads(groups.size(), indexBytes >> 18, [&](size_t g) { groupTables[g] = buildTable(g); });
    size_t pieces = 0;
    for (size_t g = 0; g < groups.size(); ++g) {
        CBAMD_ENSURE(pieces < (size_t(1) << 32), "CTR tables are too large");
        groups[g].FirstPiece = static_cast<uint32_t>(pieces);
        pieces += groupTables[g].size() / 4;
    }
    result->Table.Reserve(4 * pieces);
    for (size_t g = 0; g < groups.size(); ++g) {
        HIP_CHECK(hipMemcpy(result->Table.Get() + 4 * static_cast<size_t>(groups[g].FirstPiece), groupTables[g].data(),
                            groupTables[g].size() * 4, hipMemcpyHostToDevice));
        groupTables[g] = {};
    }
    const auto upload = [](const void* data, size_t bytes, TDeviceVec<uint32_t>* out) {
        std::vector<uint32_t> raw(std::max<size_t>(bytes / 4, 1), 0);
        if (bytes) {
            std::memcpy(raw.data(), data, bytes);
        }
        out->Upload(raw);
    };
    upload(groups.data(), groups.size() * sizeof(dev::TCtrGroupDev), &result->Groups);
    upload(items.data(), items.size() * sizeof(dev::TCtrItemDev), &result->Items);
    upload(buckets.data(), buckets.size() * 4, &result->Buckets);
    result->CatColumnsFlat.Upload(catColumnsFlat);
    result->CatColumnsSplit.Upload(catColumnsSplit);
    result->CatColumnCount = static_cast<uint32_t>(catColumnsFlat.size());
    result->GroupCount = static_cast<uint32_t>(groups.size());
}

}  // namespace

int GetHipDeviceCount() {
    int n = 0;
    const hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess) {
        throw TModelError(std::string("HIP runtime reports no usable device: ") + hipGetErrorString(e));
    }
    return n;
}

struct THipEvaluator::TImpl {
    int DeviceId = 0;
    uint32_t CuCount = 0;
    // flags of few host documents (the switches of tests): first ticket, longest wait, calls that their flags ended
    uint32_t FlagTicket = 0, FlagWaitUs = 200;
    bool CountFlagged = false;
    std::atomic<uint64_t> FlaggedCalls{0};
    hipStream_t Stream = nullptr;
    uint8_t* NoAllocScratch = nullptr;  // this device's copy of the file-scope array `scratch`
    bool Oblivious = true;
    uint32_t RealBucketCount = 0;  // buckets of the model; the device layout uses max(1, this)
    uint32_t LayoutBuckets = 1;
    uint32_t BinarizeBuckets = 0;  // float and one-hot buckets: what the binarize kernels fill
    uint32_t CtrCount = 0;         // CTR features; their buckets follow and CtrBinarizeKernel fills them
    size_t FlatVectorSize = 0;
    size_t MinFloatSize = 0;
    size_t MinCatSize = 0;
    bool HasCats = false;
    uint32_t MaxBucketValues = 0;  // largest number of borders / one-hot values in one bucket
    uint32_t MaxDepth = 0;         // deepest oblivious tree
    bool HasOneHot = false;

    // binarize tables
    TDeviceVec<uint32_t> BucketSrcFlat, BucketSrcSplit, BucketOffset, BucketFlags, Values;
    TDeviceVec<uint32_t> BucketGrid;  // 4 dwords per bucket: lowest border, cells per unit, search steps, 0
    TDeviceVec<uint32_t> BucketLut;   // kLutCells bytes per bucket
    TDeviceVec<unsigned long long> ExpMantissa;  // the table of the prediction types' exponent
    TCtrDeviceTables Ctr;
    bool CtrTileUsable = false;  // the projections' categorical columns fit the LDS tile of CtrBinarizeKernel
    // tree tables
    TDeviceVec<uint32_t> Splits, TreeStart, TreeSize, FirstLeaf, StepNodes, NodeToLeaf;
    TDeviceVec<double> Leaves, Bias;
    TDeviceVec<uint32_t> PackedTrees;  // tile kernel: 16 dwords per oblivious tree of depth <= 8
    TDeviceVec<uint32_t> PackedMixed;  // half-tile kernel: packed rows in the form chosen per tree
    TDeviceVec<double> HalfTileLeaves; // half-tile kernel: 64 or 256 leaf values per tree at a fixed pitch
    TDeviceVec<uint32_t> PairRows;     // pair-tile kernel: 32 dwords per tree, empty when the model does not qualify
    bool PairSix = false;              // ... in the six-bit form (every bin below 64)
    TDeviceVec<uint32_t> ExchangeWaves, ExchangeRecords, ExchangeExtra;  // exchange kernel (exchange_plan.h)
    TDeviceVec<double> ExchangeLeaves;
    uint32_t ExchangeRounds = 0;
    double ExchangeGeneration = 0.0;   // how many generations of the pair-tile kernel's workgroups one of its own lasts
    bool FusedExchangeBalanced = false;  // few enough levels look at the same buckets for the fused form
    bool PairBeforeTile = false;       // the tile kernel would hold the model's bins, but the pair-tile kernel takes it
    hipFunction_t ExchangeFunction = nullptr;  // nullptr: the model does not qualify
    std::string ExchangeName;
    TDeviceVec<uint32_t> FusedExchangeWaves, FusedExchangeTiles, FusedExchangeOneHot;  // its form that makes the bins from flat rows
    uint32_t FusedExchangeTileCount = 0;
    hipFunction_t FusedExchangeFunction = nullptr;
    std::string FusedExchangeName;
    TDeviceVec<uint32_t> QuadRows;     // quad-tile kernel: 16 dwords per tree, 64 bytes per row of the tile
    TDeviceVec<uint32_t> TileRows;     // row-tile kernel (whole tile, one tree per wave): the same with 256 bytes per bucket
    TDeviceVec<double> TileLeaves;     // its leaf values: [slice of the dimensions][tree][pair of dimensions][leaf][2]
    size_t TileSliceStride = 0;        // 16-byte pairs of TileLeaves per slice
    TDeviceVec<uint32_t> DeepRows;     // deep-tile kernel (depth 9 to 16): 32 dwords per tree, two halves of the row-tile form
    TDeviceVec<uint32_t> DeepFirstLeaf;  // and the trees' first leaf values in Leaves (one dimension) or first leaves in DeepLeaves
    TDeviceVec<double> DeepLeaves;       // several dimensions: [slice of two][tree][leaf][2]
    uint32_t DeepSliceLeaves = 0;        // leaves of all trees
    TDeviceVec<uint32_t> TileMap;      // rows of the tile of the row-tile or pair-tile kernel when buckets of more than
                                       // 127 values take two; empty: a row per bucket
    uint32_t TileRowCount = 0;
    TDeviceVec<double> LeavesPadded;   // tile kernel, multi-dimensional: [tree][chunk][leaf][TileChunk(dim)]
    bool PackedSevenBit = false;
    bool LeavesPairAligned = false;  // every tree's first leaf value sits at an even index
    double Scale = 1.0;
    int Dim = 1;
    std::vector<double> HostBias;

    // non-symmetric trees re-laid level by level for the tile kernel
    bool NsTileUsable = false;
    bool NsNoXor = false;
    TDeviceVec<uint32_t> NsEntries;  // pairs of dwords
    TDeviceVec<uint32_t> NsRows;     // 4 dwords per tree
    bool NsLdsUsable = false;        // compact entries walked out of LDS (xor masks as splits of their own)
    TDeviceVec<uint32_t> NsCompactEntries;
    TDeviceVec<uint32_t> NsCompactRows;  // dev::kNsUnitDwords per unit of trees
    uint32_t NsUnitCount = 0;
    uint32_t NsEntryCount = 0;       // entries of all units: rows of NsValuesByEntry per slice of the dimensions (NsSliceRows)
    TNsLdsShape NsLdsShape{0, 0};    // waves and entries per region of EvalNonSymmetricLdsKernel for this model
    TDeviceVec<double> NsValuesByEntry;

    // register-resident kernels (one-dimensional 7-bit oblivious models of depth <= 8 whose
    // buckets fit the register file): level rows and leaf values at a fixed pitch per tree
    bool RegKernelUsable = false;
    bool SmallBatchSlices = true;  // small batches: slices of the trees on workgroups of their own
    hipModule_t RegModule = nullptr;  // the device's shared module (SharedRegModule), not owned
    hipFunction_t RegFunction = nullptr;
    uint32_t RegWaves = 0;
    uint32_t RegTreeBlocks = 0;
    uint32_t RegTreeBlockSize = 16;   // trees per LDS buffer of the chosen kernel
    uint32_t RegRowDwords = 16;       // dwords of a tree's level table
    size_t RegLaunchLeaves = 0;  // doubles of the leaf table of one launch
    TDeviceVec<uint32_t> RegRows;
    TDeviceVec<double> RegLeaves;  // [launch][tree][leaf row][pitch]
    TDeviceVec<double> RegBias;    // the bias, readable for a whole pitch behind every dimension
    // The launches of a pass over the trees: the kernel's pitch in dimensions each, the last one with the narrowest kernel that
    // holds what is left (ten dimensions: six, then four instead of six of which two are padding).
    struct TRegLaunch {
        hipFunction_t Function = nullptr;
        const char* Name = "";
        uint32_t Waves = 0;
        uint32_t FirstDim = 0;
        uint32_t StoreDims = 1;
        uint32_t TreeBlock = 16;         // trees per LDS buffer of this kernel
        uint32_t GroupsPerCu = 1;        // workgroups that a CU holds at a time
        uint32_t Flags = 0;              // kRegFlagPlainTable or none
        size_t TreeLeafDoubles = 0;      // doubles of a tree in Leaves
        const double* Leaves = nullptr;  // the launch's leaf table
    };
    std::vector<TRegLaunch> RegLaunches;
    TDeviceVec<double> RegTailLeaves;  // leaf table of a last launch that uses another kernel
    // Models without xor masks whose buckets hold more than 128 values: such a bucket takes two bins registers,
    // min(bin, 127) and max(bin - 127, 0), so that every level is a 7-bit compare (the kernels' register map)
    TDeviceVec<uint32_t> RegMap;

    // fused kernels, per layout (0: flat rows, 1: split rows of a model without categorical features, 2: flat columns)
    struct TFused {
        hipFunction_t Function = nullptr;
        uint32_t Waves = 0;
        const char* Name = "";
        uint32_t UnitCount = 0;
        TDeviceVec<uint32_t> Rows;    // level rows that name bins registers of the fused layout
        TDeviceVec<uint32_t> Units;   // unit records
        TDeviceVec<uint8_t> Table;    // border table images, then a copy of the leaf table
    };
    std::shared_ptr<TFused> Fused[3];  // null: two launches
    // Below about one wave per SIMD a fused launch lasts as long as one wave's binarize phase and tree walk,
    // and two launches (the binarize kernel spreads a block over many waves) are shorter.
    size_t FusedMinDocs() const {
        return SmallBatchSlices ? size_t(1024) * dev::kDocsPerBlock : 0;
    }
    // Column-major documents of models with few buckets and few trees: a fused launch loads and searches sixteen columns
    // whatever the model has of them, and there is little else to do. Two launches against one, trees of depth 6, 4M documents:
    // one bucket, 30 trees 55 and 78 us, 300 trees 233 and 243; four buckets, 30 trees 67 and 78, 100 trees 120 and 128; eight,
    // 30 trees 83 and 83, 300 trees 261 and 249; twelve, 30 trees 98 and 88. 530 000 documents: one bucket, 30 trees 25 and 29,
    // eight, 100 trees 42.8 and 43.5. (Smaller batches' trees would be cut into slices, one more launch: 500 000 documents,
    // one bucket, 100 trees 45 and 33.)
    bool FewColumnsForFused(size_t docCount, size_t treeCount) const {
        return SmallBatchSlices && docCount >= (size_t(1) << 19) && BinarizeBuckets < 12 && BinarizeBuckets * treeCount < 1600;
    }
    // Column-major batches that leave CUs without a workgroup of the fused shapes of eight waves, which last as long as one
    // workgroup's walk whatever the batch: two launches with the trees in slices fill the chip and save about 0.3 us per 1000
    // trees and 1000 documents below 460 000, at the price of the bins' way through memory and two more launches, about 8 us and a
    // quarter of one per bucket. Beyond 192 workgroups the slices take another generation of them. Slices and fused, depth 6:
    // 262 144 documents, 8 buckets, 200 trees 40 and 42 us, 20 buckets, 600 trees 68 and 93, 60, 1000 trees 113 and 145, 80, 300
    // trees 73 and 71; 300 000, 8 buckets, 200 trees 48 and 43, 20, 600 trees 83 and 94, 60, 300 trees 76 and 67; 350 000, 20, 600
    // trees 86 and 94, 80, 1000 trees of depth 8 165 and 166; 390 000, 20, 600 trees 90 and 94, 60, 1000 trees 150 and 146; 420 000,
    // 20, 600 trees 107 and 94. (The shape of 160 over 92 buckets, 1000 trees: 262 144 121 and 124, 350 000 160 and 150.)
    bool SlicesBeforeFusedColumns(size_t docCount, size_t treeCount) const {
        return Fused[2]->Waves == 8 && docCount < size_t(192) * 8 * dev::kDocsPerBlock &&
               (460000 - docCount) * treeCount > 26000000 + 830000 * size_t(BinarizeBuckets);
    }
    const char* RegKernelName = "";

    // small-batch kernel: tree rows of sixteen dwords, and from these dwords on the cells of its tile and the first leaves
    bool SmallUsable = false;
    uint32_t SmallCellCount = 0;
    TDeviceVec<uint32_t> SmallTable;
    TDeviceVec<dev::TLeafRow> LeafRows;  // of the copies of the leaf values (kept: to free them there would take 40 to 60 us)
    TDeviceVec<double> SmallLeaves;    // the leaf values, a tree's in the order of its levels in those rows
    size_t SmallCellsAt = 0, SmallFirstLeafAt = 0;
    // rows of the table without the null trees at its end, and those of a slice: a slice of the register kernels' (the whole
    // model when it is too short for slices), or a partial sum of SumOrder() with null trees up to the length of the longest
    uint32_t SmallTreeCount = 0, SmallSliceTrees = 0;
    uint32_t SmallSliceCount() const { return (SmallTreeCount + SmallSliceTrees - 1) / SmallSliceTrees; }

    // The order in which a whole-model launch of EvalQuantizedDevice adds the trees of an oblivious model of depth <= 8 that
    // the register kernels do not take: partial sums, each in tree order, added one after the other.
    struct TSumOrder {
        uint32_t Waves = 1;     // of a workgroup
        uint32_t Side = 1;      // consecutive trees that a wave takes at a time; a last group that is not full is wave 0's
        bool PerTree = false;   // ... each to a sum of its own
        uint32_t Parts() const { return PerTree ? Waves * Side : Waves; }
        uint32_t PartOf(size_t tree, size_t treeCount) const {
            const size_t group = tree / Side;
            const size_t wave = (group + 1) * Side <= treeCount ? group % Waves : 0;
            return static_cast<uint32_t>(PerTree ? wave * Side + tree % Side : wave);
        }
    };
    TSumOrder SumOrder() const;

    // The exchange kernel instead of the pair-tile kernel, whose sums it gives: a workgroup per block of 256 documents where the other
    // has one per half block, one per CU in both. A generation of its workgroups lasts as long as 1.2 to 1.45 generations of the
    // other's (trees of depth 7 and 8) or 1.6 to 1.8 (up to 6), measured with 500 to 5000 trees; the batch decides how many of
    // each there are. 5000 trees of depth 8 over 1016 features, evaluate launch, pair-tile -> exchange: 33 000 documents
    // 240 -> 170 us, 66 000 363 -> 334, 130 000 493 -> 351, 1M 3633 -> 2659; 2000 of depth 5 over 700: 50 000 documents 61 -> 52 us,
    // 130 000 124 -> 113, 1M 887 -> 810, but 66 000 88 -> 96 and 140 000 147 -> 155, which stay where they were.
    bool TakesExchangeKernel(size_t docCount) const {
        if (ExchangeFunction == nullptr || docCount >= (size_t(1) << 29)) {
            return false;
        }
        const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
        const size_t generations = (blocks + CuCount - 1) / CuCount, others = (2 * blocks + CuCount - 1) / CuCount;
        return static_cast<double>(generations) * ExchangeGeneration < static_cast<double>(others);
    }

    // The fused form instead of a binarize launch and either kernel. A generation of its workgroups takes some 50 us longer (per 1000
    // columns), whatever part of the CUs has one; a binarize launch takes 70 us per 65 536 documents. Whole call over 1016 features,
    // two launches -> fused, by the share of the generations' places that have a workgroup: 0.50 (66 000 documents), 500 trees
    // 146 -> 150 us, 5000 trees 441 -> 457; 0.69 (90 000) 182 -> 168 and 469 -> 464, but 2000 trees of depth 5 over 700 features (pair-tile)
    // 181 -> 190; 0.77 (50 000) 96 -> 89 and 251 -> 247; 0.99 (130 000) 234 -> 192 and 525 -> 484.
    // (anyBatchSize: also where the two launches are the faster)
    bool TakesFusedExchangeKernel(size_t docCount, bool anyBatchSize) const {
        const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
        return FusedExchangeFunction != nullptr && docCount < (size_t(1) << 29) &&
               (anyBatchSize || (FusedExchangeBalanced && blocks * 10 >= (blocks + CuCount - 1) / CuCount * CuCount * 7));
    }

    // What a model's levels on few buckets cost the exchange kernels. A CU's walk over 256 documents takes, in us, 11 and 0.0335 per tree
    // of depth 7 or 8 (13 and 0.021 up to 6), the pair-tile kernel's two 17 and 0.047 (18 and 0.021). When the busiest waves have `turns`
    // groups to compare for a step, it takes 8 and 0.0188 (0.0165) * turns per tree, where that is more. Whole calls for 1M
    // documents, binarize and pair-tile launches, binarize and exchange, fused, by the share of the levels on one bucket (and turns): 2000 trees of
    // depth 8 over 1016 features, 10 % (1.9) 2708, 2305, 2076 us; 16 % (2.7) 2717, 2687, 2483; 20 % (3.3) 2733, 3018, 2778; 30 % (4.7)
    // 2714, 3832, 3572; 2000 of depth 6 over 700, 7 % (1.5) 1672, 1603, 1412; 10 % (2.0) 1665, 1687, 1590; 13 % (2.4) 1686, 1844, 1836; 500 of
    // depth 8 over 600, 30 % (4.2) 1246, 1254, 1087. The fused form saves more of a binarize launch than it takes itself, 19 us for 65 536
    // documents of 1000 columns, whatever the walk does.
    void SetExchangeCosts(size_t trees, double turns) {
        const bool shallow = MaxDepth <= 6;
        const double count = static_cast<double>(trees), even = shallow ? 13.0 + 0.021 * count : 11.0 + 0.0335 * count;
        const double walk = std::max(even, 8.0 + (shallow ? 0.0165 : 0.0188) * turns * count);
        const double pairs = shallow ? 18.0 + 0.021 * count : 17.0 + 0.047 * count;
        ExchangeGeneration = (shallow ? 1.8 : 1.45) * walk / even;
        FusedExchangeBalanced = walk - pairs <= 0.019 * LayoutBuckets;
    }

    TEvalExchangeArgs ExchangeArgs(size_t docCount, double* results) const {
        return {nullptr, ExchangeWaves.Get(), ExchangeRecords.Get(), ExchangeExtra.Get(), ExchangeLeaves.Get(), results, Bias.Get(), Scale,
                static_cast<uint32_t>(docCount), ExchangeRounds, LayoutBuckets * dev::kDocsPerBlock, 0};
    }

    // The tile kernel takes the model, or a range of its trees (of kernels on bins in an LDS tile of whole blocks, the one without a tree's
    // row in registers).
    bool TileFits(uint32_t rangeTrees = ~0u) const {
        return (!PairBeforeTile || rangeTrees < PairTrees(MaxDepth)) && TileLdsBytes(LayoutBuckets, TileChunk(Dim)) <= kMaxTileLdsBytes;
    }

    int SmallDims() const { return Dim == 1 ? 1 : Dim == 2 ? 2 : 4; }
    uint32_t SmallPasses() const { return static_cast<uint32_t>((Dim + SmallDims() - 1) / SmallDims()); }
    size_t SmallLdsBytes() const {
        const size_t tile = static_cast<size_t>(dev::SmallDocPitch(SmallCellCount)) * dev::kSmallDocs * 4;
        return tile + static_cast<size_t>(SmallSliceCount()) * dev::kSmallDocs * SmallDims() * 8;
    }
    size_t FewLdsBytes() const {
        return (static_cast<size_t>(SmallCellCount) + 1) / 2 * 8 +
               static_cast<size_t>(SmallSliceCount()) * (SmallSliceTrees + 2) * SmallDims() * 8;
    }
    // of the batches that TakesSmallBatchKernel lets through
    bool TakesFewDocumentsKernel(size_t docCount) const {
        return docCount * SmallPasses() <= kFewDocs && FewLdsBytes() <= kMaxTileLdsBytes;
    }

    // Staging of the calls that own their buffers (CalcDevice and the host entry points): a call borrows a
    // context - a stream, a bin buffer and two slots of pinned and device staging memory - from a small pool,
    // so that a few callers of one evaluator run side by side and later ones wait for a free context.
    struct THostSlot {
        TPinnedVec<float> PinnedFloats;
        TPinnedVec<int32_t> PinnedCats;
        TPinnedVec<double> PinnedResults;
        // flags of the workgroups of a small host batch and its results, which the host looks at while the launch runs
        TPinnedVec<double, hipHostMallocCoherent> SmallMemory;
        uint32_t* SmallFlags() const { return reinterpret_cast<uint32_t*>(SmallMemory.Get()); }
        double* SmallResults() const { return SmallMemory.Get() + kFlaggedGroups * sizeof(uint32_t) / sizeof(double); }
        uint32_t SmallTicket = 0;
        size_t SmallGroups = 0;  // workgroups of the running launch
        TPinnedVec<uint32_t> PinnedIndexes;
        TPinnedVec<uint8_t> PinnedExport;
        TDeviceVec<float> StageFloats;
        TDeviceVec<int32_t> StageCats;
        TDeviceVec<double> StageResults;
        TDeviceVec<uint32_t> StageIndexes;
        TDeviceVec<uint8_t> StageExport;
        // binarize start, binarize end, evaluate end, results on the host, features on the device
        hipEvent_t Ev[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
    };
    // Start and end of every workgroup of a small-batch launch. (In pinned memory, which the kernel would write over PCIe,
    // they cost a call 0.2 to 0.6 us; an event in front of the launch cost 19 us.) LastKernelTimes of one thread may read
    // those of a call that has returned while another thread's call runs on the same context: a launch takes a buffer that
    // nobody else refers to.
    struct TSmallStamps {
        TDeviceVec<unsigned long long> Values;
        size_t Count = 0;
    };
    struct THostContext {
        hipStream_t Stream = nullptr;
        hipStream_t CopyStream = nullptr;  // features of the next chunk, while the kernels of the one before run on Stream;
                                           // made by the first call of several chunks
        TDeviceVec<uint8_t> ScratchBins;
        TDeviceVec<double> SlicePartials;  // raw sums per slice of the trees (small batches)
        THostSlot Slots[2];
        hipEvent_t Ev[3] = {nullptr, nullptr, nullptr};
        std::vector<std::shared_ptr<TSmallStamps>> Stamps;  // of this context's launches; at most one more than refer to them
        std::shared_ptr<TSmallStamps> RunningStamps;        // those that the running launch writes
        bool Busy = false;

        TSmallStamps& StampsForLaunch(size_t workgroups) {
            RunningStamps.reset();
            for (const auto& stamps : Stamps) {
                if (stamps.use_count() == 1) {
                    RunningStamps = stamps;
                }
            }
            if (!RunningStamps) {
                RunningStamps = Stamps.emplace_back(std::make_shared<TSmallStamps>());
            }
            RunningStamps->Values.Reserve(2 * workgroups);
            RunningStamps->Count = workgroups;
            return *RunningStamps;
        }

        // The stream for the features of a call's chunks.
        hipStream_t CopiesOf(bool severalChunks) {
            if (!severalChunks) {
                return Stream;
            }
            if (CopyStream == nullptr) {
                HIP_CHECK(hipStreamCreateWithFlags(&CopyStream, hipStreamNonBlocking));
            }
            return CopyStream;
        }
        // What Stream does from here on finds the slot's features, sent on `copies`, on the device.
        void AwaitCopies(int slot, hipStream_t copies) {
            if (copies != Stream) {
                HIP_CHECK(hipEventRecord(Slots[slot].Ev[4], copies));
                HIP_CHECK(hipStreamWaitEvent(Stream, Slots[slot].Ev[4], 0));
            }
        }

        THostContext() {
            try {
                HIP_CHECK(hipStreamCreateWithFlags(&Stream, hipStreamNonBlocking));
                for (auto& e : Ev) {
                    HIP_CHECK(hipEventCreate(&e));
                }
                for (auto& slot : Slots) {
                    for (auto& e : slot.Ev) {
                        HIP_CHECK(hipEventCreate(&e));
                    }
                }
            } catch (...) {
                Release();  // the destructor does not run for a constructor that throws
                throw;
            }
        }
        ~THostContext() {
            Release();
        }
        void Release() {
            for (hipStream_t s : {CopyStream, Stream}) {
                if (s) {
                    (void)hipStreamSynchronize(s);
                }
            }
            for (auto& e : Ev) {
                if (e) {
                    (void)hipEventDestroy(e);
                }
            }
            for (auto& slot : Slots) {
                for (auto& e : slot.Ev) {
                    if (e) {
                        (void)hipEventDestroy(e);
                    }
                }
            }
            for (hipStream_t* s : {&CopyStream, &Stream}) {
                if (*s) {
                    (void)hipStreamDestroy(*s);
                    *s = nullptr;
                }
            }
        }
        THostContext(const THostContext&) = delete;
        THostContext& operator=(const THostContext&) = delete;
    };
    static constexpr size_t kMaxHostContexts = 4;
    std::mutex ContextLock;
    std::condition_variable ContextFree;
    std::vector<std::unique_ptr<THostContext>> Contexts;
    std::shared_ptr<const TSmallStamps> LastSmallStamps;  // the last call's if it was a small batch; under TimesLock
    hipStream_t TimesStream = nullptr;                    // reads them
    std::mutex TimesStreamLock;

    // A context of the pool for the time of one call.
    class TContextLease {
    public:
        explicit TContextLease(TImpl& impl)
            : Impl(impl)
        {
            std::unique_lock<std::mutex> guard(Impl.ContextLock);
            for (;;) {
                for (auto& c : Impl.Contexts) {
                    if (!c->Busy) {
                        Context = c.get();
                        break;
                    }
                }
                if (!Context && Impl.Contexts.size() < kMaxHostContexts) {
                    Impl.Contexts.emplace_back(new THostContext);
                    Context = Impl.Contexts.back().get();
                }
                if (Context) {
                    Context->Busy = true;
                    return;
                }
                Impl.ContextFree.wait(guard);
            }
        }
        ~TContextLease() {
            {
                std::lock_guard<std::mutex> guard(Impl.ContextLock);
                Context->Busy = false;
            }
            Impl.ContextFree.notify_one();
        }
        THostContext& operator*() const { return *Context; }
        THostContext* operator->() const { return Context; }

    private:
        TImpl& Impl;
        THostContext* Context = nullptr;
    };

    dev::TBinarizeTables BinarizeTables(bool flat) const {
        dev::TBinarizeTables t;
        t.BucketCount = BinarizeBuckets;
        t.BucketPitch = LayoutBuckets;
        t.BucketSrc = flat ? BucketSrcFlat.Get() : BucketSrcSplit.Get();
        t.BucketOffset = BucketOffset.Get();
        t.BucketFlags = BucketFlags.Get();
        t.Values = Values.Get();
        t.Grid = reinterpret_cast<const uint4*>(BucketGrid.Get());
        t.Lut = BucketLut.Get();
        return t;
    }
    dev::TCtrTablesDev CtrTables() const {
        dev::TCtrTablesDev t;
        t.Groups = reinterpret_cast<const dev::TCtrGroupDev*>(Ctr.Groups.Get());
        t.Items = reinterpret_cast<const dev::TCtrItemDev*>(Ctr.Items.Get());
        t.Table = reinterpret_cast<const uint4*>(Ctr.Table.Get());
        t.Buckets = Ctr.Buckets.Get();
        t.CatColumnsFlat = Ctr.CatColumnsFlat.Get();
        t.CatColumnsSplit = Ctr.CatColumnsSplit.Get();
        t.CatColumnCount = Ctr.CatColumnCount;
        t.GroupCount = Ctr.GroupCount;
        return t;
    }
    dev::TTreeTables TreeTables() const {
        dev::TTreeTables t;
        t.Splits = Splits.Get();
        t.TreeStart = TreeStart.Get();
        t.TreeSize = TreeSize.Get();
        t.FirstLeaf = FirstLeaf.Get();
        t.StepNodes = StepNodes.Get();
        t.NodeToLeaf = NodeToLeaf.Get();
        t.Leaves = Leaves.Get();
        t.Bias = Bias.Get();
        t.Scale = Scale;
        t.Dim = Dim;
        return t;
    }
    hipStream_t Pick(void* stream) const { return stream ? static_cast<hipStream_t>(stream) : Stream; }

    // Also runs when the evaluator's constructor throws half way (a refused model), so that the
    // stream, the events and the code object of a partly built evaluator are released.
    ~TImpl() {
        (void)hipSetDevice(DeviceId);
        if (Stream) {
            (void)hipStreamSynchronize(Stream);
        }
        Contexts.clear();
        for (hipStream_t s : {Stream, TimesStream}) {
            if (s) {
                (void)hipStreamDestroy(s);
            }
        }
    }
};

THipEvaluator::THipEvaluator(const TModelTrees& trees, int deviceId, const std::vector<TCtrValueTable>* ctrTables,
                             const TFeatureLayout* layout)
    : Impl(new TImpl)
{
    const TFeaturePositions positions(trees, layout);
    const TKernelSwitches switches = TKernelSwitches::FromEnvironment();
    const int deviceCount = GetHipDeviceCount();
    CBAMD_ENSURE(deviceCount > 0, "no HIP device found: the HIP evaluator needs an AMD GPU");
    CBAMD_ENSURE(deviceId >= 0 && deviceId < deviceCount, "HIP device id out of range");
    HIP_CHECK(hipSetDevice(deviceId));
    TImpl& m = *Impl;
    m.DeviceId = deviceId;
    int cus = 0;
    HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, deviceId));
    m.CuCount = static_cast<uint32_t>(cus);
    m.SmallBatchSlices = switches.SmallBatch;
    m.FlagTicket = switches.FlagTicket;
    m.CountFlagged = switches.CountFlagged;
    m.FlagWaitUs = switches.FlagWaitUs;
    m.NoAllocScratch = NoAllocScratchOfCurrentDevice(deviceId);
    HIP_CHECK(hipStreamCreateWithFlags(&m.Stream, hipStreamNonBlocking));
    TreeCount = trees.GetTreeCount();
    ApproxDimension = trees.ApproxDimension;
    BucketCount = trees.EffectiveBinFeaturesBucketCount;
    m.Oblivious = trees.IsOblivious();
    m.RealBucketCount = BucketCount;
    m.LayoutBuckets = std::max<uint32_t>(1, BucketCount);
    m.FlatVectorSize = positions.FlatVectorSize;
    m.MinFloatSize = positions.MinFloatSize;
    m.MinCatSize = positions.MinCatSize;
    m.HasCats = trees.UsedCatFeaturesCount > 0;
    m.Dim = trees.ApproxDimension;
    m.Scale = trees.Scale;
    m.HostBias = trees.Bias;
    {
        const TFastExpConstants constants = FastExpConstants();
        m.ExpMantissa.Upload(std::vector<unsigned long long>(constants.Mantissa, constants.Mantissa + 2048));
    }

    // ---- binarize tables: one entry per bucket, float buckets first, then one-hot buckets, in
    // the order of BinarizeFeatures (cpu/quantization.h:366-409, 54-79). Borders are sorted inside
    // each bucket (the bin is a count, so order does not matter) and NaN borders, which never
    // compare below anything, are dropped.
    std::vector<uint32_t> srcFlat, srcSplit, offsets, flags, values;
    offsets.push_back(0);
    for (const auto& f : trees.FloatFeatures) {
        if (!f.UsedInModel()) {
            continue;
        }
        CBAMD_ENSURE(f.FlatIndex >= 0 && f.Index >= 0, "float feature without a position");
        // the vector sizes come from the last feature of each list (as in the reference); a feature
        // that points past them would make the kernels read behind a caller's row
        const TFeaturePosition at = positions.Of(f);
        CBAMD_ENSURE(static_cast<size_t>(at.FlatIndex) < m.FlatVectorSize && static_cast<size_t>(at.Index) < m.MinFloatSize,
                     "float feature position exceeds the model's feature vector size");
        for (size_t begin = 0; begin < f.Borders.size(); begin += kMaxValuesPerBin) {
            const size_t end = std::min(begin + kMaxValuesPerBin, f.Borders.size());
            std::vector<float> b;
            for (size_t i = begin; i < end; ++i) {
                if (!std::isnan(f.Borders[i])) {
                    b.push_back(f.Borders[i]);
                }
            }
            std::sort(b.begin(), b.end());
            for (float x : b) {
                uint32_t bits;
                std::memcpy(&bits, &x, 4);
                values.push_back(bits);
            }
            offsets.push_back(static_cast<uint32_t>(values.size()));
            srcFlat.push_back(static_cast<uint32_t>(at.FlatIndex));
            srcSplit.push_back(static_cast<uint32_t>(at.Index));
            const bool nanToInf = f.HasNans && f.NanValueTreatment == ENanValueTreatment::AsTrue;
            flags.push_back(nanToInf ? dev::kBucketFlagNanToInf : 0);
        }
    }
    for (const auto& oh : trees.OneHotFeatures) {
        const TCatFeature* cat = nullptr;
        for (const auto& c : trees.CatFeatures) {
            if (c.Index == oh.CatFeatureIndex && c.UsedInModel) {
                cat = &c;
            }
        }
        CBAMD_ENSURE(cat != nullptr, "one-hot feature refers to an unknown or unused categorical feature");
        CBAMD_ENSURE(cat->FlatIndex >= 0 && cat->Index >= 0, "categorical feature without a position");
        const TFeaturePosition at = positions.Of(*cat);
        CBAMD_ENSURE(static_cast<size_t>(at.FlatIndex) < m.FlatVectorSize && static_cast<size_t>(at.Index) < m.MinCatSize,
                     "categorical feature position exceeds the model's feature vector size");
        for (size_t begin = 0; begin < oh.Values.size(); begin += kMaxValuesPerBin) {
            const size_t end = std::min(begin + kMaxValuesPerBin, oh.Values.size());
            for (size_t i = begin; i < end; ++i) {
                values.push_back(static_cast<uint32_t>(oh.Values[i]));
            }
            offsets.push_back(static_cast<uint32_t>(values.size()));
            srcFlat.push_back(static_cast<uint32_t>(at.FlatIndex));
            srcSplit.push_back(static_cast<uint32_t>(at.Index));
            flags.push_back(dev::kBucketFlagOneHot);
        }
    }
    m.BinarizeBuckets = static_cast<uint32_t>(srcFlat.size());
    CBAMD_ENSURE(m.BinarizeBuckets == trees.CtrFirstBucket, "internal error: bucket count mismatch");
    if (!trees.CtrFeatures.empty()) {
        CBAMD_ENSURE(ctrTables != nullptr, "Model has CTR features but no tables of learned statistics");
        BuildCtrTables(trees, positions, *ctrTables, &srcFlat, &srcSplit, &offsets, &flags, &values, &m.Ctr);
        m.CtrCount = static_cast<uint32_t>(trees.CtrFeatures.size());
        m.CtrTileUsable = m.Ctr.CatColumnCount <= dev::kCtrMaxTileColumns && switches.CtrTile;
    }
    CBAMD_ENSURE(srcFlat.size() == BucketCount, "internal error: bucket count mismatch");
    for (size_t b = 0; b + 1 < offsets.size(); ++b) {
        m.MaxBucketValues = std::max(m.MaxBucketValues, offsets[b + 1] - offsets[b]);
    }
    m.HasOneHot = !trees.OneHotFeatures.empty();
    if (m.Oblivious) {
        for (int d : trees.TreeSizes) {
            m.MaxDepth = std::max<uint32_t>(m.MaxDepth, static_cast<uint32_t>(d));
        }
    }
    if (BucketCount == 0) {  // keep the device tables non-empty; the binarize kernel is skipped
        srcFlat.push_back(0);
        srcSplit.push_back(0);
        offsets.push_back(0);
        flags.push_back(0);
    }
    // grid and search window of every float bucket (dev::CountBelowInCell)
    {
        const uint32_t slots = 1u << BinarizeLog2Slots(m.MaxBucketValues);
        const size_t bucketRows = offsets.size() - 1;
        std::vector<uint32_t> grid(bucketRows * 4, 0), lut(bucketRows * (dev::kLutCells / 4), 0);
        for (size_t b = 0; b < bucketRows; ++b) {
            const uint32_t n = offsets[b + 1] - offsets[b];
            if ((flags[b] & dev::kBucketFlagOneHot) || n == 0) {
                continue;
            }
            std::vector<float> borders(n);
            std::memcpy(borders.data(), values.data() + offsets[b], n * sizeof(float));
            const TBucketGrid g = MakeBucketGrid(borders);
            const float lo = g.Lo, scale = g.Scale;
            const uint32_t steps = g.Steps;
            CBAMD_ENSURE((1u << steps) <= slots, "internal error: search window exceeds the bucket's slots");
            uint8_t* cells = reinterpret_cast<uint8_t*>(lut.data() + b * (dev::kLutCells / 4));
            for (int c = 0; c < dev::kLutCells; ++c) {
                // a lower start only adds borders known to be below the value; it keeps the window inside the slots
                cells[c] = static_cast<uint8_t>(std::min(g.Start[c], slots - (1u << steps)));
            }
            std::memcpy(&grid[b * 4 + 0], &lo, 4);
            std::memcpy(&grid[b * 4 + 1], &scale, 4);
            grid[b * 4 + 2] = steps;
        }
        m.BucketGrid.Upload(grid);
        m.BucketLut.Upload(lut);
    }
    m.BucketSrcFlat.Upload(srcFlat);
    m.BucketSrcSplit.Upload(srcSplit);
    m.BucketOffset.Upload(offsets);
    m.BucketFlags.Upload(flags);
    m.Values.Upload(values);

    // ---- tree tables
    std::vector<uint32_t> splits(trees.RepackedBins.size());
    for (size_t i = 0; i < splits.size(); ++i) {
        const auto& rb = trees.RepackedBins[i];
        CBAMD_ENSURE(rb.FeatureIndex < m.LayoutBuckets, "internal error: split refers to a missing bucket");
        splits[i] = static_cast<uint32_t>(rb.FeatureIndex) | (static_cast<uint32_t>(rb.XorMask) << 16) |
                    (static_cast<uint32_t>(rb.SplitIdx) << 24);
    }
    std::vector<uint32_t> treeStart(trees.TreeStartOffsets.begin(), trees.TreeStartOffsets.end());
    std::vector<uint32_t> treeSize(trees.TreeSizes.begin(), trees.TreeSizes.end());
    std::vector<uint32_t> firstLeaf(trees.TreeFirstLeafOffsets.size());
    for (size_t t = 0; t < firstLeaf.size(); ++t) {
        CBAMD_ENSURE(trees.TreeFirstLeafOffsets[t] <= std::numeric_limits<uint32_t>::max(), "model has too many leaf values");
        firstLeaf[t] = static_cast<uint32_t>(trees.TreeFirstLeafOffsets[t]);
    }
    std::vector<uint32_t> steps(trees.NonSymmetricStepNodes.size());
    for (size_t i = 0; i < steps.size(); ++i) {
        steps[i] = static_cast<uint32_t>(trees.NonSymmetricStepNodes[i].LeftSubtreeDiff) |
                   (static_cast<uint32_t>(trees.NonSymmetricStepNodes[i].RightSubtreeDiff) << 16);
    }
    m.Splits.Upload(splits);
    m.TreeStart.Upload(treeStart);
    m.TreeSize.Upload(treeSize);
    m.FirstLeaf.Upload(firstLeaf);
    m.StepNodes.Upload(steps);
    m.NodeToLeaf.Upload(trees.NonSymmetricNodeIdToLeafId);
    m.Bias.Upload(trees.Bias);

    // How unevenly a level splits the documents, 0 (two halves) to 0.5, estimated from the rank of its border among the feature's borders
    // (borders are quantiles of the training data). Kernels take a tree's levels in any order, leaf tables permuted to match.
    const auto lopsidedness = [&](const TRepackedBin& rb) {
        const uint32_t n = offsets[rb.FeatureIndex + 1] - offsets[rb.FeatureIndex];
        const bool oneHot = (flags[rb.FeatureIndex] & dev::kBucketFlagOneHot) != 0 || rb.XorMask != 0;
        const double share = oneHot ? 0.05 : static_cast<double>(rb.SplitIdx) / (n + 1.0);
        return switches.LevelOrder ? std::fabs(share - 0.5) : 0.0;
    };

    // Order of a tree's levels in the tables of the register and small-batch kernels (levelOrder[t][position] = level of the
    // model). The leaf gathers of a wave meet in the LDS banks that the low bits of the leaf indexes choose; lanes with the
    // same index share one access, lanes that differ only in high bits wait for each other. So the levels
    // that split the documents most evenly go to the low bits and the lopsided ones, on which most lanes
    // agree, to the high bits: fewer lanes of a bank then differ. The sums and their order do not change.
    std::vector<std::array<uint8_t, kRegMaxDepth>> levelOrder;
    if (m.Oblivious && m.MaxDepth <= kRegMaxDepth) {
        levelOrder.resize(TreeCount);
        for (size_t t = 0; t < TreeCount; ++t) {
            double keys[kRegMaxDepth];
            for (int d = 0; d < trees.TreeSizes[t]; ++d) {
                const double key = lopsidedness(trees.RepackedBins[trees.TreeStartOffsets[t] + d]);
                int at = d;
                for (; at > 0 && key < keys[at - 1]; --at) {
                    keys[at] = keys[at - 1];
                    levelOrder[t][at] = levelOrder[t][at - 1];
                }
                keys[at] = key;
                levelOrder[t][at] = static_cast<uint8_t>(d);
            }
        }
    }

    // Leaf values in other layouts are copied by a kernel from those on the device, when all tables stand (PlaceLeavesKernel).
    std::vector<dev::TLeafRow> leafRows;
    std::vector<std::pair<double*, size_t>> leafCopies;  // where, and how many rows of leafRows up to there
    const auto placeLeaves = [&](TDeviceVec<double>* to, size_t size) {  // leafRows has got the rows
        to->Reserve(std::max<size_t>(size, 1));
        leafCopies.emplace_back(to->Get(), leafRows.size());
    };

    TExchangeTables exchangeTables;
    std::future<void> exchangeBuilt;
    const auto finishExchange = [&] {
        exchangeBuilt.get();
        const TExchangeTables& x = exchangeTables;
        if (!x.Planned) {
            return;
        }
        const std::string shape = std::string(x.MaxDepth == 6 ? "d6" : "d8") + (x.Six ? "_s" : "");
        if (x.Tiled) {
            m.FusedExchangeWaves.Upload(x.Plan.FusedWaveTable);
            m.FusedExchangeTiles.Upload(x.Tiles);
            m.FusedExchangeOneHot.Upload(x.OneHot);
            m.FusedExchangeTileCount = static_cast<uint32_t>(x.Pieces.size()) / kExchangeTilePieces;
            m.FusedExchangeName = "cbamd_fused_exchange_" + shape;
            HIP_CHECK(hipModuleGetFunction(&m.FusedExchangeFunction, SharedRegModule(kEvalRegCodeObject), m.FusedExchangeName.c_str()));
        }
        m.ExchangeRounds = x.Plan.Rounds;
        m.SetExchangeCosts(TreeCount, static_cast<double>(x.Plan.CompareSteps) / (x.Plan.Rounds * kExchangeRoundSteps));
        m.ExchangeWaves.Upload(x.Plan.WaveTable);
        m.ExchangeRecords.Upload(x.Plan.Records);
        m.ExchangeExtra.Upload(x.Plan.ExtraRows);
        const size_t pitch = size_t(1) << x.MaxDepth;
        for (size_t r = 0; r < x.Plan.LeafRows.size(); ++r) {
            const TExchangeLeafRow& row = x.Plan.LeafRows[r];
            const bool tree = row.Tree != kExchangeNoTree;
            leafRows.push_back({r * pitch, tree ? firstLeaf[row.Tree] : 0u, row.Levels, tree ? static_cast<uint32_t>(pitch) : 0u,
                                static_cast<uint32_t>(pitch) | (ExchangeFoldsLeaves(x.MaxDepth) ? dev::kLeafRowFolded : 0u)});
        }
        placeLeaves(&m.ExchangeLeaves, x.Plan.LeafRows.size() * pitch);
        m.ExchangeName = "cbamd_eval_exchange_" + shape;
        HIP_CHECK(hipModuleGetFunction(&m.ExchangeFunction, SharedRegModule(kEvalRegCodeObject), m.ExchangeName.c_str()));
    };

    // The kernels that keep a tree's row in registers (two trees per wave on half a tile, one on a whole tile)
    // compare 7 bits. Their tile has a row per bucket, and two for a bucket of more than 127 values, which the
    // kernel makes while it copies the bins to LDS (tileMap): min(bin, 127) and max(bin - 127, 0) for a float
    // bucket, the bins up to 127 (0 for the others) and bin - 127 from 128 on (0 for the others) for a one-hot bucket.
    std::vector<uint32_t> tileRowOfBucket(offsets.size(), 0), tileMap;
    const bool tileRowsUsable = true;
    bool tileRowsSplit = false;
    for (size_t b = 0; b + 1 < offsets.size(); ++b) {
        tileRowOfBucket[b] = static_cast<uint32_t>(tileMap.size());
        if (offsets[b + 1] - offsets[b] <= 127) {
            tileMap.push_back(static_cast<uint32_t>(b));
        } else {
            const bool oneHot = (flags[b] & dev::kBucketFlagOneHot) != 0;
            tileMap.push_back(static_cast<uint32_t>(b) | ((oneHot ? dev::kTileMapOneHotLow : dev::kTileMapLow) << 16));
            tileMap.push_back(static_cast<uint32_t>(b) | (dev::kTileMapHigh << 16));
            tileRowsSplit = true;
        }
    }
    const uint32_t tileRowCount = static_cast<uint32_t>(tileMap.size());
    // A level of a tree in those kernels' rows: (row of the tile, xor byte, value added to the four bins, xors)
    struct TTileLevel {
        uint32_t Row, Xor, Add;
        bool IsXor;
    };
    const auto tileLevelOf = [&](const TRepackedBin& rb) {
        TTileLevel level = {tileRowOfBucket[rb.FeatureIndex], 0, 0, false};
        if (rb.XorMask != 0 || rb.SplitIdx == 0xff) {
            // one-hot: bin == value, value = ~XorMask; below 128 seven bits of it are enough, a value from 128 on
            // is looked for as value - 127 in the bucket's second row
            uint32_t value = ~static_cast<uint32_t>(rb.XorMask) & 0xffu;
            if (value > 127 && offsets[rb.FeatureIndex + 1] - offsets[rb.FeatureIndex] > 127) {
                level.Row += 1;
                value -= 127;
            }
            level.Xor = ~value & 0x7fu;
            level.Add = 0x01010101u;
            level.IsXor = true;
        } else if (rb.SplitIdx > 127) {
            level.Row += 1;  // the bucket's second row holds max(bin - 127, 0)
            level.Add = (128u - (rb.SplitIdx - 127u)) * 0x01010101u;
        } else {
            level.Add = (128u - rb.SplitIdx) * 0x01010101u;
        }
        return level;
    };
    // Their rows: 16 dwords per tree, slot d the byte offset of level d's row in the tile | xor byte << 24, slot
    // 8 + d the value added to the four bins of a dword.
    const auto rowsInRegisters = [&](uint32_t bucketBytes) {
        std::vector<uint32_t> rows((trees.GetTreeCount() + dev::kQuadTreePadding) * dev::kPackedTreeDwords, 0);
        for (size_t t = 0; t < trees.GetTreeCount(); ++t) {
            uint32_t* row = rows.data() + t * dev::kPackedTreeDwords;
            bool anyXor = false;
            for (int d = 0; d < trees.TreeSizes[t]; ++d) {
                const TTileLevel level = tileLevelOf(trees.RepackedBins[trees.TreeStartOffsets[t] + d]);
                row[d] = level.Row * bucketBytes | level.Xor << 24;
                row[8 + d] = level.Add;
                anyXor = anyXor || level.IsXor;
            }
            if (anyXor) {
                row[0] |= dev::kPairRowXorFlag;
            }
        }
        return rows;
    };

    // The pair-tile kernel's rows: sixteen entries of two dwords per tree, entry d a level's row offset (128-byte rows)
    // and its xor byte four times, entry 8 + d the value added to the four bins of a dword
    const auto pairTileRows = [&](bool six) {
        std::vector<uint32_t> rows((trees.GetTreeCount() + dev::kPairTreePadding) * dev::kPairRowDwords, 0);
        for (size_t t = 0; t < trees.GetTreeCount(); ++t) {
            uint32_t* row = rows.data() + t * dev::kPairRowDwords;
            for (int d = 0; d < trees.TreeSizes[t]; ++d) {
                const TTileLevel level = tileLevelOf(trees.RepackedBins[trees.TreeStartOffsets[t] + d]);
                uint32_t xorByte = level.Xor, addByte = level.Add & 0xffu;
                if (six && d % 2 == 0) {
                    // the six-bit form of an even level: its result goes to bit 6 of the byte
                    if (level.IsXor) {
                        xorByte &= 0x3fu;
                    } else {
                        CBAMD_ENSURE(addByte > 64, "split index beyond the six-bit form");
                        addByte -= 64;
                    }
                }
                row[2 * d] = level.Row * 128u;
                row[2 * d + 1] = xorByte * 0x01010101u;
                row[2 * (8 + d)] = addByte * 0x01010101u;
            }
        }
        return rows;
    };

    // 7-bit compares need every bin and split index to fit 7 bits and no xor mask
    m.PackedSevenBit = m.Oblivious && !m.HasOneHot && m.MaxBucketValues <= 127;
    if (m.Oblivious && m.MaxDepth <= 8) {
        std::vector<uint32_t> packed(trees.GetTreeCount() * dev::kPackedTreeDwords, 0);
        for (size_t t = 0; t < trees.GetTreeCount(); ++t) {
            uint32_t* row = packed.data() + t * dev::kPackedTreeDwords;
            for (int d = 0; d < 8; ++d) {
                if (d < trees.TreeSizes[t]) {
                    const auto& rb = trees.RepackedBins[trees.TreeStartOffsets[t] + d];
                    row[d] = m.PackedSevenBit
                                 ? (static_cast<uint32_t>(rb.FeatureIndex) << 8) | (128u - rb.SplitIdx)
                                 : (static_cast<uint32_t>(rb.FeatureIndex) << 16) |
                                       (static_cast<uint32_t>(rb.XorMask) << 8) | rb.SplitIdx;
                } else {
                    row[d] = m.PackedSevenBit ? 0u : 0xffu;  // a level that is false for every bin
                }
            }
            row[dev::kPackedFirstLeafSlot] = firstLeaf[t];
        }
        if (m.Dim > 1) {
            const size_t pitch = static_cast<size_t>(TileChunk(m.Dim));
            const size_t chunks = (static_cast<size_t>(m.Dim) + pitch - 1) / pitch;
            std::vector<double> padded;
            for (size_t t = 0; t < trees.GetTreeCount(); ++t) {
                const size_t leafCount = size_t(1) << trees.TreeSizes[t];
                CBAMD_ENSURE(padded.size() <= std::numeric_limits<uint32_t>::max(), "model has too many leaf values");
                packed[t * dev::kPackedTreeDwords + dev::kPackedPaddedLeafSlot] = static_cast<uint32_t>(padded.size());
                packed[t * dev::kPackedTreeDwords + dev::kPackedLeafCountSlot] = static_cast<uint32_t>(leafCount);
                const double* values = trees.LeafValues.data() + trees.TreeFirstLeafOffsets[t];
                for (size_t c = 0; c < chunks; ++c) {
                    for (size_t leaf = 0; leaf < leafCount; ++leaf) {
                        for (size_t k = 0; k < pitch; ++k) {
                            const size_t d = c * pitch + k;
                            padded.push_back(d < static_cast<size_t>(m.Dim) ? values[leaf * m.Dim + d] : 0.0);
                        }
                    }
                }
            }
            padded.resize(padded.size() + 256 * pitch, 0.0);  // the kernel copies 256 leaves' worth per tree
            m.LeavesPadded.Upload(padded);
        }
        m.PackedTrees.Upload(packed);
        if (m.Dim == 1) {
            // per-tree form: 7-bit when the tree has no one-hot split and every float bin fits 7 bits
            uint32_t maxFloatValues = 0;
            for (size_t b = 0; b + 1 < offsets.size(); ++b) {
                if (!(flags[b] & dev::kBucketFlagOneHot)) {
                    maxFloatValues = std::max(maxFloatValues, offsets[b + 1] - offsets[b]);
                }
            }
            std::vector<uint32_t> mixed(packed.size(), 0);
            for (size_t t = 0; t < trees.GetTreeCount(); ++t) {
                bool sevenBit = maxFloatValues <= 127;
                for (int d = 0; d < trees.TreeSizes[t]; ++d) {
                    sevenBit = sevenBit && trees.RepackedBins[trees.TreeStartOffsets[t] + d].XorMask == 0;
                }
                uint32_t* row = mixed.data() + t * dev::kPackedTreeDwords;
                for (int d = 0; d < 8; ++d) {
                    if (d < trees.TreeSizes[t]) {
                        const auto& rb = trees.RepackedBins[trees.TreeStartOffsets[t] + d];
                        if (sevenBit) {
                            // ready for use: byte offset of the bucket's row in the half tile, compare constant
                            row[d] = static_cast<uint32_t>(rb.FeatureIndex) * 128u;
                            row[8 + d] = (128u - rb.SplitIdx) * 0x0101u;
                        } else {
                            row[d] = (static_cast<uint32_t>(rb.FeatureIndex) << 16) |
                                     (static_cast<uint32_t>(rb.XorMask) << 8) | rb.SplitIdx;
                        }
                    } else {
                        row[d] = sevenBit ? 0u : 0xffu;  // a split that no bin passes
                    }
                }
                if (!sevenBit) {
                    row[dev::kPackedFormSlot] |= 0x80000000u;
                }
            }
            m.PackedMixed.Upload(mixed);
            // The tile fits LDS up to 632 buckets, but not with the regions of the row-tile kernel beyond 568 rows (trees of depth 7 and 8) or
            // 616: two trees per wave on half a tile there, or the exchange kernel, if the model has trees enough or the latter takes its
            // large batches (a bucket of more than 127 values keeps that off). Few trees on rows of their own: the tile kernel.
            const bool fewTrees = TreeCount < PairTrees(m.MaxDepth);
            m.PairBeforeTile = switches.RowTile && switches.PairTile && PairTileLdsBytes(tileRowCount, 8) <= kMaxTileLdsBytes &&
                               RowTileWaves(tileRowCount, m.MaxDepth, 1) == 0 && !(fewTrees && tileRowsSplit);
            if (!m.TileFits()) {
                const size_t pitch = m.MaxDepth <= 6 ? 64 : 256;
                // zeros at the end: the pair-tile and quad-tile kernels fetch ahead of their trees without a bound
                const size_t rowCount = trees.GetTreeCount() + dev::kQuadTreePadding;
                for (size_t t = 0; t < rowCount; ++t) {
                    leafRows.push_back({t * pitch, t < TreeCount ? firstLeaf[t] : 0u, dev::kLeafRowInOrder,
                                        t < TreeCount ? 1u << trees.TreeSizes[t] : 0u, static_cast<uint32_t>(pitch)});
                }
                placeLeaves(&m.HalfTileLeaves, rowCount * pitch);
                // two trees per wave: every bin of the tile's rows below 128 (the one-hot test then fits 7 bits too)
                const int maxd = m.MaxDepth <= 6 ? 6 : 8;
                const bool pairFits = PairTileLdsBytes(tileRowCount, 8) <= kMaxTileLdsBytes;
                // four trees per wave on a quarter of a block when the rows do not fit the half tile
                const bool quadFits = !pairFits && QuadTileWaves(tileRowCount, maxd) != 0;
                if (switches.PairTile && tileRowsUsable && (pairFits || quadFits)) {
                    if (pairFits) {
                        // every bin below 64: the walk joins two levels at a time
                        m.PairSix = m.MaxBucketValues <= 63 && !tileRowsSplit && switches.RegSix;
                        m.PairRows.Upload(pairTileRows(m.PairSix));
                        if (switches.Exchange && !tileRowsSplit) {
                            TExchangeTables& x = exchangeTables;
                            x.BucketCount = m.LayoutBuckets;
                            x.MaxDepth = static_cast<uint32_t>(maxd);
                            x.Six = m.PairSix;
                            x.Trees.resize(trees.GetTreeCount());
                            for (size_t t = 0; t < x.Trees.size(); ++t) {
                                x.Trees[t].Levels.reserve(trees.TreeSizes[t]);
                                for (int d = 0; d < trees.TreeSizes[t]; ++d) {
                                    const auto& rb = trees.RepackedBins[trees.TreeStartOffsets[t] + d];
                                    const TTileLevel level = tileLevelOf(rb);
                                    x.Trees[t].Levels.push_back({level.Row, level.Add & 0xffu, level.Xor, level.IsXor, static_cast<float>(lopsidedness(rb))});
                                }
                            }
                            // The fused form: the model's columns in pieces of four neighbouring ones, sixteen pieces a tile. A
                            // piece that would leave the row is moved back over its neighbour.
                            bool tiled = switches.Fused && m.CtrCount == 0 && m.BinarizeBuckets == BucketCount && BucketCount > 0 &&
                                         m.FlatVectorSize >= kExchangePieceColumns;
                            std::vector<std::pair<uint32_t, uint32_t>> byColumn;
                            for (uint32_t b = 0; tiled && b < BucketCount; ++b) {
                                byColumn.emplace_back(srcFlat[b], b);
                                tiled = (flags[b] & dev::kBucketFlagNanToInf) == 0 && offsets[b + 1] > offsets[b];
                            }
                            std::sort(byColumn.begin(), byColumn.end());
                            x.ColumnOf.assign(m.LayoutBuckets, kExchangeNoColumn);
                            for (size_t i = 0; tiled && i < byColumn.size(); ++i) {
                                const uint32_t column = byColumn[i].first;
                                if (x.Pieces.empty() || column * 4 >= x.Pieces.back() + 4 * kExchangePieceColumns) {
                                    x.Pieces.push_back(4 * std::min<uint32_t>(column & ~3u, static_cast<uint32_t>(m.FlatVectorSize) - kExchangePieceColumns));
                                }
                                x.ColumnOf[byColumn[i].second] = static_cast<uint32_t>(x.Pieces.size() - 1) * kExchangePieceColumns + column - x.Pieces.back() / 4;
                                tiled = (i == 0 || column != byColumn[i - 1].first) && x.Pieces.size() <= kExchangeTiles * kExchangeTilePieces;
                            }
                            if (tiled) {
                                x.Pieces.resize((x.Pieces.size() + kExchangeTilePieces - 1) / kExchangeTilePieces * kExchangeTilePieces, 0);
                                x.Columns.resize(x.Pieces.size() * kExchangePieceColumns);
                                for (uint32_t b = 0; b < BucketCount; ++b) {
                                    TExchangeColumn& column = x.Columns[x.ColumnOf[b]];
                                    column.Used = true;
                                    column.OneHot = (flags[b] & dev::kBucketFlagOneHot) != 0;
                                    column.RowByte = srcFlat[b] * 4;
                                    column.Values.assign(values.begin() + offsets[b], values.begin() + offsets[b + 1]);
                                }
                            } else {
                                x.ColumnOf.clear();
                            }
                            // (run by get() where there is no thread to be had)
                            exchangeBuilt = std::async(std::launch::async | std::launch::deferred, [&exchangeTables] { exchangeTables.Build(); });
                        }
                    } else {
                        m.QuadRows.Upload(rowsInRegisters(64));
                    }
                    m.TileRowCount = tileRowsSplit ? tileRowCount : m.LayoutBuckets;  // (a model without splits: its one zero bucket)
                    if (tileRowsSplit) {
                        m.TileMap.Upload(tileMap);
                    }
                }
                if (fewTrees && m.PairBeforeTile && exchangeBuilt.valid()) {
                    finishExchange();
                    if (m.ExchangeFunction == nullptr || (m.ExchangeGeneration >= 2.0 && !m.FusedExchangeBalanced)) {
                        m.PairBeforeTile = TileLdsBytes(m.LayoutBuckets, 1) > kMaxTileLdsBytes;
                        if (!m.PairBeforeTile) {
                            m.ExchangeFunction = m.FusedExchangeFunction = nullptr;  // their sums are not the tile kernel's
                        }
                    }
                }
            }
        }
        m.LeavesPairAligned = true;
        for (uint32_t f : firstLeaf) {
            m.LeavesPairAligned = m.LeavesPairAligned && (f % 2 == 0);
        }
    }

    if (!m.Oblivious) {
        std::vector<uint32_t> compactEntries, compactRows, topNodes;
        std::vector<double> valuesByEntry;
        BuildLevelOrderTrees(trees, m.Dim, firstLeaf, &m.NsEntries, &m.NsRows, &m.NsTileUsable, &m.NsNoXor,
                             &compactEntries, &compactRows, &topNodes, &valuesByEntry, &m.NsLdsUsable);
        if (m.NsLdsUsable) {
            // the shape whose units take the least time: more waves hide more of the walk's latency, smaller
            // regions hold fewer trees per unit (kNsLdsShapes)
            m.NsLdsUsable = false;
            double bestCost = 0.0;
            struct TPlan {
                bool Fits = false;
                std::vector<TNsUnit> Units;
            };
            std::map<uint32_t, TPlan> plans;  // by the entries of a region
            const std::vector<uint32_t> order = OrderNsTrees(compactRows, TreeCount);
            for (const TNsLdsShape& shape : kNsLdsShapes) {
                if ((switches.NsWaves != 0 && switches.NsWaves != shape.Waves) ||
                    NsLdsKernelBytes(m.LayoutBuckets, shape.Waves, shape.Entries, NsLdsDims(m.Dim)) > kMaxTileLdsBytes) {
                    continue;
                }
                const auto [known, fresh] = plans.try_emplace(shape.Entries);
                std::vector<TNsUnit>& plan = known->second.Units;
                if (fresh) {
                    known->second.Fits = PackNsUnits(compactRows, order, shape.Entries, &plan);
                }
                if (!known->second.Fits) {
                    continue;  // a tree larger than a region
                }
                uint64_t steps = 0;
                for (const TNsUnit& unit : plan) {
                    steps += unit.Height + 3;  // the top three levels
                }
                const double cost = static_cast<double>(steps) / shape.Speed;
                if (!m.NsLdsUsable || cost < bestCost) {
                    m.NsLdsUsable = true;
                    m.NsLdsShape = shape;
                    bestCost = cost;
                }
            }
            if (m.NsLdsUsable) {
                const std::vector<TNsUnit>& bestUnits = plans[m.NsLdsShape.Entries].Units;
                // the entries in the order of the units; child indexes (bits 21-31) count from the unit's first entry (trees are
                // whole pieces of eight entries, as a wave's copy of a unit, sixteen bytes per lane, needs pieces of four)
                std::vector<uint32_t> entries, units;
                std::vector<double> values;
                entries.reserve(compactEntries.size());
                values.reserve(valuesByEntry.size());
                // the bucket (bits 8-17 of an entry or node) becomes the LDS row of its bins in this shape
                const auto withTileRow = [&](uint32_t entry) {
                    return (entry & ~0x3ff00u) | dev::NsLdsTileRow((entry >> 8) & 0x3ffu, m.NsLdsShape.Waves, m.NsLdsShape.Entries) << 8;
                };
                std::vector<uint32_t> from;
                std::vector<double> old;
                for (const TNsUnit& unit : bestUnits) {
                    const uint32_t first = static_cast<uint32_t>(entries.size());
                    uint32_t start[dev::kNsUnitTrees] = {};
                    uint32_t count = 0;
                    for (uint32_t i = 0; i < unit.TreeCount; ++i) {
                        const uint32_t t = unit.Trees[i];
                        const uint32_t treeFirst = compactRows[t * 4], treeEntries = compactRows[t * 4 + 2];
                        start[i] = count;
                        for (uint32_t e = 0; e < treeEntries; ++e) {
                            entries.push_back(withTileRow(compactEntries[treeFirst + e]) + (count << 21));
                        }
                        const double* value = valuesByEntry.data() + static_cast<size_t>(treeFirst) * m.Dim;
                        values.insert(values.end(), value, value + static_cast<size_t>(treeEntries) * m.Dim);
                        count += treeEntries;
                    }
                    if (unit.Height == 0) {
                        from.clear();
                        for (uint32_t i = 0; i < unit.TreeCount; ++i) {
                            CompactNsExits(entries.data() + first + start[i], &from);
                        }
                        const size_t dim = static_cast<size_t>(m.Dim);
                        old.assign(values.begin() + static_cast<std::ptrdiff_t>(first * dim), values.end());
                        for (size_t r = 0; r < from.size(); ++r) {
                            std::copy_n(old.data() + from[r] * dim, dim, values.data() + (first + r) * dim);
                        }
                    }
                    const uint32_t row[8] = {first, unit.Height, first, start[1], start[2] | (unit.TreeCount << 16),
                                             unit.Trees[0], unit.Trees[1], unit.Trees[2]};
                    units.insert(units.end(), row, row + 8);
                    for (uint32_t i = 0; i < static_cast<uint32_t>(dev::kNsUnitTrees); ++i) {
                        const uint32_t* nodes = topNodes.data() + unit.Trees[i < unit.TreeCount ? i : 0] * 8;  // (a tree too few: the first again)
                        std::transform(nodes, nodes + 8, std::back_inserter(units), withTileRow);
                    }
                    const bool third = std::any_of(unit.Trees, unit.Trees + unit.TreeCount, [&](uint32_t t) {
                        const uint32_t* nodes = topNodes.data() + t * 8;
                        return std::any_of(nodes + 3, nodes + 7, [](uint32_t node) { return (node & 0xffu) != 0; });
                    });
                    units[units.size() - dev::kNsUnitDwords + 15] = third ? 0u : 1u;
                }
                // the first entry of the unit that a unit's wave takes next
                for (size_t u = 0; u + m.NsLdsShape.Waves < bestUnits.size(); ++u) {
                    units[u * dev::kNsUnitDwords + 2] = units[(u + m.NsLdsShape.Waves) * dev::kNsUnitDwords];
                }
                m.NsUnitCount = static_cast<uint32_t>(bestUnits.size());
                m.NsEntryCount = static_cast<uint32_t>(entries.size());
                {
                    // ... in whole regions, whatever the unit's size: spare entries behind the last unit
                    std::vector<uint32_t> padded(entries);
                    padded.resize(entries.size() + m.NsLdsShape.Entries, 255u);
                    m.NsCompactEntries.Upload(padded);
                }
                m.NsCompactRows.Upload(units);
                // [slice of the dimensions][entry][dimension of the slice], zeros past the last dimension and, of one, behind the last entry
                const uint32_t dims = NsLdsDims(m.Dim), slices = (static_cast<uint32_t>(m.Dim) + dims - 1) / dims;
                const size_t sliceRows = NsSliceRows(entries.size(), dims, m.NsLdsShape.Entries);
                if (m.Dim == 1) {
                    values.resize(sliceRows, 0.0);
                } else {
                    std::vector<double> bySlice(slices * sliceRows * dims, 0.0);
                    for (uint32_t slice = 0; slice < slices; ++slice) {
                        for (size_t e = 0; e < entries.size(); ++e) {
                            for (uint32_t k = 0; k < dims && slice * dims + k < static_cast<uint32_t>(m.Dim); ++k) {
                                bySlice[(slice * sliceRows + e) * dims + k] = values[e * m.Dim + slice * dims + k];
                            }
                        }
                    }
                    values.swap(bySlice);
                }
                m.NsValuesByEntry.Upload(values);
            }
        }
    }

    const bool regEnabled = switches.RegKernel;
    // The 7-bit compare "bin + 128 - s carries into bit 7" stays within its byte for bins up to 127 + s, and s is at least 1:
    // buckets of up to 128 values (the usual number of candidate borders; a json model lists them all) need no second
    // register, and in the six-bit form, whose even levels add 64 - s, buckets of up to 64. Only a level that stands for
    // none (constant 0) would then be true for the largest bin: the leaf tables repeat a tree's values in the rows
    // that such levels choose between. 1M documents, 1000 trees of depth 6, 116 buckets of which 20 have 128 values:
    // 136 registers and two waves per SIMD before, 116 and three now, evaluate launch 243 -> 216 us.
    // (The tile kernels keep to 127 and 63 values: their leaf tables have no rows to repeat.)
    const uint32_t sevenBitValues = switches.RegSplit ? 128 : 127;
    const bool regSevenBit = m.Oblivious && !m.HasOneHot && m.MaxBucketValues <= sevenBitValues;
    const bool six = regSevenBit && m.MaxBucketValues <= 64 && switches.RegSix;
    const TEvalRegVariant* variant =
        m.Oblivious && m.MaxDepth <= kRegMaxDepth && TreeCount > 0
            ? PickRegVariant(m.LayoutBuckets, static_cast<uint32_t>(m.Dim), m.MaxDepth, !regSevenBit, six,
                             switches.RegMinBuckets)
            : nullptr;
    // bins registers: one per bucket, or two for the buckets of more than 128 values when that keeps a model
    // without xor masks off the 8-bit compare
    std::vector<uint32_t> firstRegOfBucket(offsets.size(), 0), regMap;
    bool regMapped = false;
    uint32_t maxFloatBucketValues = 0;
    for (size_t b = 0; b + 1 < offsets.size(); ++b) {
        if (!(flags[b] & dev::kBucketFlagOneHot)) {
            maxFloatBucketValues = std::max(maxFloatBucketValues, offsets[b + 1] - offsets[b]);
        }
    }
    if (m.Oblivious && m.MaxDepth <= kRegMaxDepth && TreeCount > 0 && maxFloatBucketValues > sevenBitValues && switches.RegSplit) {
        for (size_t b = 0; b + 1 < offsets.size(); ++b) {
            firstRegOfBucket[b] = static_cast<uint32_t>(regMap.size());
            if ((flags[b] & dev::kBucketFlagOneHot) || offsets[b + 1] - offsets[b] <= sevenBitValues) {
                regMap.push_back(static_cast<uint32_t>(b) | (kRegMapAsIs << 16));
            } else {
                regMap.push_back(static_cast<uint32_t>(b) | (kRegMapLow << 16));
                regMap.push_back(static_cast<uint32_t>(b) | (kRegMapHigh << 16));
            }
        }
        // without one-hot splits the model is all 7-bit now; with them the trees that have none are
        const TEvalRegVariant* splitVariant = PickRegVariant(static_cast<uint32_t>(regMap.size()), static_cast<uint32_t>(m.Dim),
                                                             m.MaxDepth, m.HasOneHot, false, switches.RegMinBuckets);
        if (splitVariant != nullptr) {
            variant = splitVariant;
            regMapped = true;
        }
    }
    const uint32_t regCount = regMapped ? static_cast<uint32_t>(regMap.size()) : m.LayoutBuckets;
    // a thread's 32-bit offset walks through the leaf table of a launch while it is copied to LDS
    const bool regTableAddressable =
        variant && (TreeCount / RegTreeBlock(*variant) + 3) * RegTreeBlock(*variant) * variant->Leaves * variant->Pitch * 8 <
                       (uint64_t(1) << 32) - (1u << 20);
    if (regEnabled && variant && regTableAddressable) {
        m.RegModule = SharedRegModule(kEvalRegCodeObject);
        HIP_CHECK(hipModuleGetFunction(&m.RegFunction, m.RegModule, variant->Name));
        m.RegKernelName = variant->Name;
        const uint32_t block = RegTreeBlock(*variant);
        const size_t pitch = variant->Pitch, rowsPerTree = variant->Leaves;
        const size_t rowDwords = variant->Mixed || variant->Leaves > 256 ? 32 : 16;
        const int rowLevels = variant->Leaves > 256 ? 10 : 8;
        m.RegWaves = variant->Waves;
        m.RegRowDwords = static_cast<uint32_t>(rowDwords);
        m.RegTreeBlocks = static_cast<uint32_t>((TreeCount + block - 1) / block);
        // two blocks of null trees behind the last one: the kernels prefetch that far
        const size_t tableTrees = (static_cast<size_t>(m.RegTreeBlocks) + 2) * block;
        const size_t launches = (static_cast<size_t>(m.Dim) + pitch - 1) / pitch;
        m.RegLaunchLeaves = tableTrees * rowsPerTree * pitch;
        // the last launch: the kernel of the same form with the smallest pitch that holds the dimensions left
        const size_t tailFirst = (launches - 1) * pitch, tailDims = static_cast<size_t>(m.Dim) - tailFirst;
        const TEvalRegVariant* tailVariant = nullptr;
        for (const auto& v : kEvalRegVariants) {
            if (m.Dim > 1 && v.Pitch > 1 && v.Pitch >= tailDims && v.Pitch < pitch && v.Leaves == variant->Leaves &&
                v.Mixed == variant->Mixed && v.Six == variant->Six && v.Waves == variant->Waves &&
                regCount <= v.Buckets && (!tailVariant || v.Pitch < tailVariant->Pitch)) {
                tailVariant = &v;
            }
        }
        const uint32_t tailBlock = tailVariant ? RegTreeBlock(*tailVariant) : block;
        const size_t tailPitch = tailVariant ? tailVariant->Pitch : pitch;
        const size_t tailTableTrees = ((TreeCount + tailBlock - 1) / tailBlock + 2) * tailBlock;
        // tree ranges are cut at blocks of the kernel with the larger block (both are powers of two)
        m.RegTreeBlockSize = std::max(block, tailBlock);
        // A level that stands for none (bucket 0 or the tree's first one, add 0) is true for the bins from 128 on, in the six-bit form
        // from 64 on at its even levels. Nothing may depend on it: the leaf tables repeat a tree's values in all rows that such
        // levels choose between, and the trees that fill up the last block have zeros in all of theirs.
        std::vector<uint32_t> rows(std::max(tableTrees, tailTableTrees) * rowDwords, 0);
        std::vector<double> leaves((tailVariant ? launches - 1 : launches) * m.RegLaunchLeaves, 0.0);
        std::vector<double> tailLeaves(tailVariant ? tailTableTrees * rowsPerTree * tailPitch : 0, 0.0);
        // The register of a level's bins and the split index there: a float bucket that takes two registers answers
        // "bin >= s" in the first for s <= 127 and as "bin - 127 >= s - 127" in the second.
        const auto registerOf = [&](const TRepackedBin& rb) -> std::pair<uint32_t, uint32_t> {
            uint32_t reg = rb.FeatureIndex, splitIdx = rb.SplitIdx;
            if (regMapped) {
                reg = firstRegOfBucket[rb.FeatureIndex];
                if (rb.XorMask == 0 && splitIdx > 127 && !(flags[rb.FeatureIndex] & dev::kBucketFlagOneHot) &&
                    offsets[rb.FeatureIndex + 1] - offsets[rb.FeatureIndex] > sevenBitValues) {
                    reg += 1;
                    splitIdx -= 127;
                }
            }
            return {reg, splitIdx};
        };
        for (size_t t = 0; t < TreeCount; ++t) {
            const int depth = trees.TreeSizes[t];
            const auto levelAt = [&](int position) -> const TRepackedBin& {
                return trees.RepackedBins[trees.TreeStartOffsets[t] + levelOrder[t][position]];
            };
            // 7-bit form: no xor mask in the tree and no bin of its buckets above 128
            bool sevenBit = true;
            for (int d = 0; d < depth; ++d) {
                const auto& rb = levelAt(d);
                sevenBit = sevenBit && rb.XorMask == 0 &&
                           (regMapped || offsets[rb.FeatureIndex + 1] - offsets[rb.FeatureIndex] <= sevenBitValues);
            }
            CBAMD_ENSURE(sevenBit || variant->Mixed, "internal error: tree needs the 8-bit compare");
            uint32_t* row = rows.data() + t * rowDwords;
            if (sevenBit) {
                for (int d = 0; d < depth; ++d) {
                    const auto& rb = levelAt(d);
                    const auto [reg, splitIdx] = registerOf(rb);
                    row[2 * d] = reg;
                    // the level's bit is the carry into bit 7; six-bit kernels want the even levels' in bit 6
                    // (of the first eight levels: levels 8 and 9 of a deep tree are read from bit 7 in every form)
                    row[2 * d + 1] = ((variant->Six && d % 2 == 0 && d < 8 ? 64u : 128u) - splitIdx) * 0x01010101u;
                }
                for (int d = depth; d < rowLevels && depth > 0; ++d) {
                    row[2 * d] = row[0];
                }
            } else {
                for (int d = 0; d < 8; ++d) {
                    // levels past the tree's depth: splitIdx 255, false for every bin (bins are at most 254)
                    uint32_t bucket = 0, xorMask = 0, splitIdx = 255;
                    if (d < depth) {
                        const auto& rb = levelAt(d);
                        std::tie(bucket, splitIdx) = registerOf(rb);
                        xorMask = rb.XorMask;
                    }
                    row[4 * d] = bucket;
                    row[4 * d + 1] = xorMask * 0x01010101u;
                    row[4 * d + 2] = (256u - splitIdx) * 0x01010101u;  // (a split's index is at least 1)
                }
                row[0] |= 0x80000000u;
            }
            const double* values = trees.LeafValues.data() + trees.TreeFirstLeafOffsets[t];
            for (size_t launch = 0; launch < launches; ++launch) {
                const bool tailTable = tailVariant && launch + 1 == launches;
                const size_t launchPitch = tailTable ? tailPitch : pitch;
                double* table = tailTable ? tailLeaves.data() + t * rowsPerTree * tailPitch
                                          : leaves.data() + launch * m.RegLaunchLeaves + t * rowsPerTree * pitch;
                const TEvalRegVariant& kernel = tailTable ? *tailVariant : *variant;
                const bool folds = FoldsLeaves(kernel, m.MaxDepth), pairs = PairsDimensions(kernel, m.MaxDepth);
                for (size_t leaf = 0; leaf < rowsPerTree; ++leaf) {
                    // where the kernel looks for it (the top bit of what it folds comes inverted), and the leaf of the model whose level
                    // bits are these (those behind the tree's levels may be anything)
                    const size_t place = folds ? leaf ^ (leaf >> 1) ^ (rowsPerTree >> 2) : leaf;
                    size_t modelLeaf = 0;
                    for (int d = 0; d < depth; ++d) {
                        modelLeaf |= ((leaf >> d) & 1) << levelOrder[t][d];
                    }
                    // pieces of two dimensions, 16 bytes per leaf, or one per dimension
                    for (size_t k = 0; k < launchPitch && launch * pitch + k < static_cast<size_t>(m.Dim); ++k) {
                        const size_t slot = pairs ? (k / 2) * rowsPerTree * 2 + place * 2 + k % 2 : k * rowsPerTree + place;
                        table[slot] = values[modelLeaf * m.Dim + launch * pitch + k];
                    }
                }
            }
        }
        std::vector<double> biasPadded(static_cast<size_t>(m.Dim) + pitch, 0.0);
        std::copy(m.HostBias.begin(), m.HostBias.end(), biasPadded.begin());
        m.RegRows.Upload(rows);
        m.RegLeaves.Upload(leaves);
        m.RegBias.Upload(biasPadded);
        if (tailVariant) {
            m.RegTailLeaves.Upload(tailLeaves);
        }
        if (regMapped) {
            // an entry per register of the largest kernel, in whole batches of sixteen; the spare ones load bucket 0
            regMap.resize((224 + 15) / 16 * 16, 0);
            m.RegMap.Upload(regMap);
        }
        for (size_t launch = 0; launch < launches; ++launch) {
            TImpl::TRegLaunch l;
            l.FirstDim = static_cast<uint32_t>(launch * pitch);
            l.StoreDims = static_cast<uint32_t>(std::min(pitch, static_cast<size_t>(m.Dim) - launch * pitch));
            l.Waves = variant->Waves;
            if (tailVariant && launch + 1 == launches) {
                HIP_CHECK(hipModuleGetFunction(&l.Function, m.RegModule, tailVariant->Name));
                l.Name = tailVariant->Name;
                l.TreeBlock = tailBlock;
                l.TreeLeafDoubles = rowsPerTree * tailPitch;
                l.Leaves = m.RegTailLeaves.Get();
            } else {
                l.Function = m.RegFunction;
                l.Name = variant->Name;
                l.TreeBlock = block;
                l.TreeLeafDoubles = rowsPerTree * pitch;
                l.Leaves = m.RegLeaves.Get() + launch * m.RegLaunchLeaves;
            }
            const TEvalRegVariant& kernel = tailVariant && launch + 1 == launches ? *tailVariant : *variant;
            l.Flags = FoldsLeaves(kernel, m.MaxDepth) ? 0u : PairsDimensions(kernel, m.MaxDepth) ? kRegFlagPairTable : kRegFlagPlainTable;
            int groupsPerCu = 0;
            HIP_CHECK(hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&groupsPerCu, l.Function, static_cast<int>(64 * l.Waves), 0));
            l.GroupsPerCu = static_cast<uint32_t>(std::max(1, groupsPerCu));
            m.RegLaunches.push_back(l);
        }
        m.RegKernelUsable = true;

        // ---- fused kernels: float-only one-dimensional models in the 7-bit or six-bit form whose rows are
        // at least sixteen columns wide. The bins registers follow the columns of the rows (a unit = sixteen
        // consecutive columns = sixteen registers), so the level rows are rewritten per row layout.
        // Models of the 96-register shape take the fused kernel of 64 or 80 bins registers when their units fit it (112
        // and 128 registers: four waves per SIMD like their evaluate kernel); with more units they stay on two launches
        // (a fused kernel of 96 bins registers would run at three waves per SIMD and is the slower - measured on
        // 50 and 90 buckets). A model on the six-level kernel takes the form of the fused kernel that walks six levels, whose
        // buffers hold 64 trees: null trees up to whole buffers, and two more. (The limit on the table's bytes, which the kernels address by
        // 32 bits, counts 256 rows a tree for either form: some two million trees.)
        const bool fusedCandidate = switches.Fused && !regMapped && !variant->Mixed && variant->Pitch == 1 && variant->Leaves <= 256 && m.Dim == 1 && !m.HasCats &&
                                    m.CtrCount == 0 && m.BinarizeBuckets == BucketCount && BucketCount > 0 &&
                                    (TreeCount / block + 3) * block * 256 * 8 + 16 * kFusedImageBytes < (uint64_t(1) << 32) - (1u << 20);
        const size_t bufferTrees = kFusedImageBytes / (variant->Leaves * sizeof(double));
        const size_t fusedTrees = fusedCandidate ? ((TreeCount + bufferTrees - 1) / bufferTrees + 2) * bufferTrees : 0;
        const size_t fusedLeaves = fusedTrees * variant->Leaves;  // zeros behind the register kernel's
        for (int layoutIndex = 0; layoutIndex < 3 && fusedCandidate; ++layoutIndex) {
            const bool columnMajor = layoutIndex == 2;  // a value is a load of its own: units of any sixteen buckets
            const std::vector<uint32_t>& columns = layoutIndex == 1 ? srcSplit : srcFlat;
            const size_t rowWidth = layoutIndex == 1 ? m.MinFloatSize : m.FlatVectorSize;
            if (rowWidth < kFusedUnitColumns && !columnMajor) {
                continue;
            }
            if (layoutIndex == 1 && m.MinFloatSize == m.FlatVectorSize && srcSplit == srcFlat) {
                m.Fused[1] = m.Fused[0];  // the same rows
                continue;
            }
            std::vector<std::pair<uint32_t, uint32_t>> byColumn;  // (column, bucket)
            for (uint32_t b = 0; b < BucketCount; ++b) {
                byColumn.emplace_back(columns[b], b);
            }
            std::sort(byColumn.begin(), byColumn.end());
            bool distinct = true;
            for (size_t i = 1; i < byColumn.size(); ++i) {
                distinct = distinct && byColumn[i].first != byColumn[i - 1].first;
            }
            if (!distinct && !columnMajor) {
                continue;
            }
            // units: sixteen columns from a used column on, moved back where they would leave the row
            std::vector<uint32_t> unitStart, slotOfBucket(BucketCount, 0);
            for (uint32_t b = 0; b < BucketCount && columnMajor; ++b) {
                slotOfBucket[b] = b;
            }
            if (columnMajor) {
                unitStart.assign((BucketCount + kFusedUnitColumns - 1) / kFusedUnitColumns, 0);
            }
            for (size_t i = 0; i < byColumn.size() && !columnMajor;) {
                const uint32_t start = static_cast<uint32_t>(std::min<size_t>(byColumn[i].first, rowWidth - kFusedUnitColumns));
                const uint32_t unit = static_cast<uint32_t>(unitStart.size());
                unitStart.push_back(start);
                while (i < byColumn.size() && byColumn[i].first < start + kFusedUnitColumns) {
                    slotOfBucket[byColumn[i].second] = unit * kFusedUnitColumns + (byColumn[i].first - start);
                    ++i;
                }
            }
            const TFusedVariant* fused = nullptr;
            for (const auto& v : kFusedVariants) {
                // (of the rows' shapes the wide one is for the models of the wide evaluate kernels; columns over 88
                // buckets: 1M documents, 200 trees 164 us on two launches, 126 on the shape of 160, 1000 trees 329 and 301)
                if (v.Columns == columnMajor && v.Six == variant->Six && unitStart.size() * kFusedUnitColumns <= v.Buckets && !fused &&
                    (variant->Waves == 4 || v.Buckets <= 80 || columnMajor) && variant->Leaves == 1u << v.Levels) {
                    fused = &v;
                }
            }
            if (!fused) {
                continue;
            }
            const uint32_t slots = fused->Six ? 64 : 128;           // border slots of a bucket in an image
            const uint32_t bucketsPerImage = fused->Six ? 64 : 32;
            const uint32_t unitsPerImage = bucketsPerImage / kFusedUnitColumns;
            const uint32_t maxUnits = fused->Buckets / kFusedUnitColumns;
            uint32_t images = (fused->Buckets + bucketsPerImage - 1) / bucketsPerImage;
            images += images % 2;
            std::vector<uint32_t> bucketOfSlot(fused->Buckets, UINT32_MAX);
            for (uint32_t b = 0; b < BucketCount; ++b) {
                bucketOfSlot[slotOfBucket[b]] = b;
            }
            // grids first: the four columns of a load share their number of search steps
            std::vector<TBucketGrid> grids(fused->Buckets);
            std::vector<std::vector<float>> bordersOfSlot(fused->Buckets);
            std::vector<uint32_t> groupSteps(fused->Buckets / 4, 1);
            bool fits = true;
            for (uint32_t slot = 0; slot < fused->Buckets; ++slot) {
                const uint32_t b = bucketOfSlot[slot];
                if (b == UINT32_MAX) {
                    continue;
                }
                const uint32_t n = offsets[b + 1] - offsets[b];
                bordersOfSlot[slot].resize(n);
                std::memcpy(bordersOfSlot[slot].data(), values.data() + offsets[b], n * sizeof(float));
                grids[slot] = MakeFusedGrid(bordersOfSlot[slot], columnMajor);
                groupSteps[slot / 4] = std::max(groupSteps[slot / 4], grids[slot].Steps);
                fits = fits && n <= slots;
            }
            for (uint32_t steps : groupSteps) {
                fits = fits && steps <= kFusedMaxSteps && (1u << steps) <= slots;
            }
            if (!fits) {
                continue;
            }
            // the records of all units the kernel has code for, one more, and the units' byte offsets in a row or every
            // unit's columns (places that no bucket has read the first bucket's)
            const size_t recordDwords = (static_cast<size_t>(maxUnits) + 1) * kFusedUnitDwords;
            std::vector<uint32_t> units(recordDwords + (columnMajor ? (maxUnits + 1) * kFusedUnitColumns : 16), 0);
            std::fill(units.begin() + recordDwords, units.end(), columnMajor ? columns[0] : 0);
            for (size_t u = 0; u < unitStart.size() && !columnMajor; ++u) {
                units[recordDwords + u] = unitStart[u] * 4;
            }
            for (uint32_t b = 0; b < BucketCount && columnMajor; ++b) {
                units[recordDwords + b] = columns[b];
            }
            std::vector<uint8_t> table(images * kFusedImageBytes + fusedLeaves * sizeof(double), 0);
            for (uint32_t slot = 0; slot < fused->Buckets; ++slot) {
                const uint32_t unit = slot / kFusedUnitColumns, column = slot % kFusedUnitColumns;
                uint32_t* record = units.data() + static_cast<size_t>(unit) * kFusedUnitDwords;
                const uint32_t steps = groupSteps[slot / 4], group = column / 4;
                record[32] |= (steps >= 4 ? 1u << group : 0u) | (steps >= 3 ? 16u << group : 0u) | (steps >= 2 ? 256u << group : 0u);
                const uint32_t b = bucketOfSlot[slot];
                if (b == UINT32_MAX) {
                    continue;  // a column no split reads: all-zero record and tables, its register is never indexed
                }
                record[32] |= 4096u << group;
                std::memcpy(&record[column], &grids[slot].Lo, 4);
                std::memcpy(&record[16 + column], &grids[slot].Scale, 4);
                if (flags[b] & dev::kBucketFlagNanToInf) {
                    record[32] |= 0x10000u << column;
                }
                uint8_t* image = table.data() + (unit / unitsPerImage) * kFusedImageBytes;
                const uint32_t local = (unit % unitsPerImage) * kFusedUnitColumns + column;
                uint32_t* borders = reinterpret_cast<uint32_t*>(image + static_cast<size_t>(local) * slots * 4);
                for (uint32_t k = 0; k < slots; ++k) {
                    uint32_t bits = 0x7f800000u;  // +inf behind the real borders
                    if (k < bordersOfSlot[slot].size()) {
                        std::memcpy(&bits, &bordersOfSlot[slot][k], 4);
                    }
                    borders[k] = bits;
                }
                uint8_t* lut = image + kFusedLutOffset + static_cast<size_t>(local) * dev::kLutCells;
                for (int c = 0; c < dev::kLutCells; ++c) {
                    const uint32_t start = std::min(grids[slot].Start[c], slots + 1 - (1u << steps));  // the search ends inside the slots
                    lut[c] = static_cast<uint8_t>(fused->Six ? start * 4 : start);  // the six-bit form stores byte offsets
                }
            }
            std::memcpy(table.data() + images * kFusedImageBytes, leaves.data(), std::min(leaves.size(), fusedLeaves) * sizeof(double));
            // level rows of the same form as the register kernel's, naming bins registers of this layout
            std::vector<uint32_t> fusedRows(rows);
            fusedRows.resize(std::max(fusedRows.size(), fusedTrees * rowDwords), 0);
            for (size_t t = 0; t < TreeCount; ++t) {
                const int depth = trees.TreeSizes[t];
                uint32_t* row = fusedRows.data() + t * rowDwords;
                for (int d = 0; d < depth; ++d) {
                    row[2 * d] = slotOfBucket[trees.RepackedBins[trees.TreeStartOffsets[t] + levelOrder[t][d]].FeatureIndex];
                }
                for (int d = depth; d < 8 && depth > 0; ++d) {
                    row[2 * d] = row[0];
                }
            }
            m.Fused[layoutIndex] = std::make_shared<TImpl::TFused>();
            TImpl::TFused& f = *m.Fused[layoutIndex];
            HIP_CHECK(hipModuleGetFunction(&f.Function, m.RegModule, fused->Name));
            f.Waves = fused->Waves;
            f.Name = fused->Name;
            f.UnitCount = static_cast<uint32_t>(unitStart.size());
            f.Rows.Upload(fusedRows);
            f.Units.Upload(units);
            f.Table.Upload(table);
        }
    }

    // Models that the register kernels do not take, every bin of the tile's rows below 128, the 256-document tile and the leaf
    // regions of eight waves in LDS: a tree's row in registers (EvalObliviousRowTileKernel).
    if (!m.RegKernelUsable && m.Oblivious && m.MaxDepth <= 8 && TreeCount > 0 && switches.RowTile && tileRowsUsable &&
        RowTileWaves(tileRowCount, m.MaxDepth, m.Dim) != 0) {
        const size_t leavesPerTree = m.MaxDepth <= 6 ? 64 : 256;
        const size_t dims = RowTileDims(m.MaxDepth, m.Dim), slices = (static_cast<size_t>(m.Dim) + dims - 1) / dims;
        const size_t tableTrees = TreeCount + dev::kPairTreePadding;  // zeros at the end: the kernel fetches ahead of its trees
        std::vector<double> values(slices * tableTrees * leavesPerTree * dims, 0.0);
        for (size_t t = 0; t < TreeCount; ++t) {
            const double* leaf = trees.LeafValues.data() + trees.TreeFirstLeafOffsets[t];
            for (size_t l = 0; l < (size_t(1) << trees.TreeSizes[t]); ++l) {
                for (size_t d = 0; d < static_cast<size_t>(m.Dim); ++d) {
                    // [slice][tree][pair of dimensions][leaf][dimension of the pair]; one dimension: [tree][leaf]
                    const size_t slice = d / dims, k = d % dims;
                    const size_t slot = dims == 1 ? l : ((k / 2) * leavesPerTree + l) * 2 + k % 2;
                    values[(slice * tableTrees + t) * leavesPerTree * dims + slot] = leaf[l * m.Dim + d];
                }
            }
        }
        m.TileLeaves.Upload(values);
        m.TileSliceStride = tableTrees * leavesPerTree * dims / 2;
        m.TileRows.Upload(rowsInRegisters(256));
        m.TileRowCount = tileRowsSplit ? tileRowCount : m.LayoutBuckets;  // (a model without splits: its one zero bucket)
        if (tileRowsSplit) {
            m.TileMap.Upload(tileMap);
        }
    }

    // Models of depth 9 to 16 that the register kernels do not take (deeper than 10, one-hot splits, several
    // dimensions, more registers than they have): the same tile, a tree's levels in two halves of eight, leaf values
    // gathered from the model's own table, two dimensions per walk (EvalObliviousDeepTileKernel).
    if (!m.RegKernelUsable && m.Oblivious && m.MaxDepth > 8 && m.MaxDepth <= 16 && TreeCount > 0 &&
        switches.RowTile && tileRowsUsable &&
        DeepTileLdsBytes(tileRowsSplit ? tileRowCount : m.LayoutBuckets, DeepTileDims(m.Dim)) <= kMaxTileLdsBytes) {
        const size_t tableTrees = TreeCount + dev::kPairTreePadding;
        std::vector<uint32_t> rows(tableTrees * 32, 0), first(tableTrees, 0);
        for (size_t t = 0; t < TreeCount; ++t) {
            uint32_t* row = rows.data() + t * 32;
            bool anyXor = false;
            for (int d = 0; d < trees.TreeSizes[t]; ++d) {
                const TTileLevel level = tileLevelOf(trees.RepackedBins[trees.TreeStartOffsets[t] + d]);
                uint32_t* half = row + (d < 8 ? 0 : 16);
                const int slot = d % 8;
                half[slot] = level.Row * 256u | level.Xor << 24;
                half[8 + slot] = level.Add;
                anyXor = anyXor || level.IsXor;
            }
            if (anyXor) {
                row[0] |= dev::kPairRowXorFlag;
            }
            first[t] = firstLeaf[t];
        }
        if (m.Dim > 1) {
            // two dimensions of a leaf side by side, slice after slice
            const size_t dim = static_cast<size_t>(m.Dim), slices = (dim + 1) / 2;
            size_t leafCount = 0;
            for (size_t t = 0; t < TreeCount; ++t) {
                first[t] = static_cast<uint32_t>(leafCount);
                leafCount += size_t(1) << trees.TreeSizes[t];
            }
            CBAMD_ENSURE(leafCount < (size_t(1) << 31), "too many leaves for the deep-tile kernel");
            std::vector<double> pairs(slices * leafCount * 2, 0.0);
            for (size_t t = 0; t < TreeCount; ++t) {
                const double* values = trees.LeafValues.data() + trees.TreeFirstLeafOffsets[t];
                for (size_t leaf = 0; leaf < (size_t(1) << trees.TreeSizes[t]); ++leaf) {
                    for (size_t k = 0; k < dim; ++k) {
                        pairs[((k / 2) * leafCount + first[t] + leaf) * 2 + k % 2] = values[leaf * dim + k];
                    }
                }
            }
            m.DeepLeaves.Upload(pairs);
            m.DeepSliceLeaves = static_cast<uint32_t>(leafCount);
        }
        m.DeepRows.Upload(rows);
        m.DeepFirstLeaf.Upload(first);
        m.TileRowCount = tileRowsSplit ? tileRowCount : m.LayoutBuckets;
        if (tileRowsSplit) {
            m.TileMap.Upload(tileMap);
        }
    }

    // ---- small-batch kernel: every split as "cell of the tile above a border"
    if (m.Oblivious && m.MaxDepth <= 8 && TreeCount > 0 && m.CtrCount == 0 && BucketCount > 0) {
        std::vector<dev::TSmallCell> cells;
        std::vector<uint32_t> cellOfBucket(BucketCount, UINT32_MAX);
        std::map<std::pair<uint32_t, uint32_t>, uint32_t> cellOfValue;  // one-hot: (bucket, value's index) -> cell
        // The trees in slices that are added as larger batches' kernels add them: consecutive trees for the register kernels'
        // slices, else the trees of a wave's partial sum.
        std::vector<size_t> order;
        const size_t nullTree = TreeCount;
        if (m.RegKernelUsable) {
            order.resize(TreeCount);
            std::iota(order.begin(), order.end(), size_t(0));
            const uint32_t slice = RegSliceTrees(m.RegTreeBlockSize);
            m.SmallSliceTrees = TreeCount < 2 * static_cast<size_t>(slice) ? static_cast<uint32_t>(TreeCount) : slice;
        } else {
            const TImpl::TSumOrder sums = m.SumOrder();
            std::vector<std::vector<size_t>> parts(sums.Parts());
            size_t longest = 0;
            for (size_t t = 0; t < TreeCount; ++t) {
                std::vector<size_t>& part = parts[sums.PartOf(t, TreeCount)];
                part.push_back(t);
                longest = std::max(longest, part.size());
            }
            while (parts.back().empty()) {
                parts.pop_back();  // sums of zero
            }
            if (parts.size() > 1) {
                longest = (longest + dev::kSmallTurn - 1) / dev::kSmallTurn * dev::kSmallTurn;
            }
            for (std::vector<size_t>& part : parts) {
                part.resize(longest, nullTree);
                order.insert(order.end(), part.begin(), part.end());
            }
            m.SmallSliceTrees = static_cast<uint32_t>(longest);
        }
        m.SmallTreeCount = static_cast<uint32_t>(order.size());
        // rows of null trees at the end, for a last slice that ends inside a turn: no level is above +inf or NaN
        order.resize(order.size() + dev::kSmallNullTrees, nullTree);
        std::vector<uint32_t> rows(order.size() * 16, 0);
        std::vector<uint32_t> first(order.size(), static_cast<uint32_t>(trees.LeafValues.size()));
        // Sixteen documents of a tree read its leaf values together, from as many lines of 128 bytes as the high bits of their indexes
        // differ: the lopsided levels, on which most documents agree, go there (6.9 lines -> 5.2 at depth 8). 1000 trees of depth 8,
        // SmallBatchKernel for 4096 documents 12.5 -> 11.2 us, 16 384 38.7 -> 33.7; of depth 6 25.0 -> 24.0.
        const uint32_t never = 0x7f800000u;
        bool usable = trees.LeafValues.size() < (size_t(1) << 32);
        for (size_t place = 0; place < order.size() && usable; ++place) {
            const size_t t = order[place];
            const int depth = t < TreeCount ? trees.TreeSizes[t] : 0;
            uint32_t* row = rows.data() + place * 16;
            if (t < TreeCount) {
                first[place] = static_cast<uint32_t>(trees.TreeFirstLeafOffsets[t]);
            }
            for (int d = 0; d < 8; ++d) {
                row[8 + d] = never;
                if (d >= depth) {
                    continue;
                }
                const auto& rb = trees.RepackedBins[trees.TreeStartOffsets[t] + levelOrder[t][d]];
                const uint32_t b = rb.FeatureIndex, n = offsets[b + 1] - offsets[b];
                // a damaged model may name a border that is not there: such a split stays with the kernels on bins
                const bool oneHot = (flags[b] & dev::kBucketFlagOneHot) != 0;
                const uint32_t at = oneHot ? static_cast<uint8_t>(~rb.XorMask) : rb.SplitIdx;
                if (at == 0 || at > n || (oneHot ? rb.SplitIdx != 0xff : rb.XorMask != 0)) {
                    usable = false;
                    break;
                }
                uint32_t cell;
                if (oneHot) {
                    // "bin = at", and no other value of the bucket is the same one
                    const uint32_t value = values[offsets[b] + at - 1];
                    usable = usable &&
                             std::count(values.begin() + offsets[b], values.begin() + offsets[b + 1], value) == 1;
                    const auto found = cellOfValue.emplace(std::make_pair(b, at), static_cast<uint32_t>(cells.size()));
                    if (found.second) {
                        cells.push_back({srcFlat[b], srcSplit[b], 2u, value});
                    }
                    cell = found.first->second;
                    row[8 + d] = 0x3f000000u;  // 0.5
                } else {
                    if (cellOfBucket[b] == UINT32_MAX) {
                        cellOfBucket[b] = static_cast<uint32_t>(cells.size());
                        cells.push_back({srcFlat[b], srcSplit[b], (flags[b] & dev::kBucketFlagNanToInf) ? 1u : 0u, 0u});
                    }
                    cell = cellOfBucket[b];
                    row[8 + d] = values[offsets[b] + at - 1];
                }
                row[d] = cell * 4;
            }
        }
        if (usable && !cells.empty()) {
            // one allocation: the rows, the cells, the first leaves
            std::vector<uint32_t> table(std::move(rows));
            m.SmallCellsAt = table.size();
            const uint32_t* cellDwords = reinterpret_cast<const uint32_t*>(cells.data());
            table.insert(table.end(), cellDwords, cellDwords + cells.size() * (sizeof(dev::TSmallCell) / 4));
            m.SmallFirstLeafAt = table.size();
            table.insert(table.end(), first.begin(), first.end());
            m.SmallTable.Upload(table);
            for (size_t t = 0; t < TreeCount; ++t) {
                uint32_t levels = ~0u;
                for (int d = 0; d < trees.TreeSizes[t]; ++d) {
                    levels ^= (dev::kLeafRowNoLevel ^ levelOrder[t][d]) << 4 * d;
                }
                leafRows.push_back({firstLeaf[t], firstLeaf[t], levels, 1u << trees.TreeSizes[t], 1u << trees.TreeSizes[t]});
            }
            leafRows.push_back({trees.LeafValues.size(), 0u, ~0u, 0u, 256u});  // null trees' values
            placeLeaves(&m.SmallLeaves, trees.LeafValues.size() + 256 * static_cast<size_t>(trees.ApproxDimension));
            m.SmallCellCount = static_cast<uint32_t>(cells.size());
            m.SmallUsable = true;
        }
    }

    {
        // the tile kernel copies (1 << 8) * dim doubles per tree: keep that much readable behind the end
        std::vector<double> padded;
        padded.reserve(trees.LeafValues.size() + 256 * static_cast<size_t>(trees.ApproxDimension));
        padded = trees.LeafValues;
        padded.resize(padded.size() + 256 * static_cast<size_t>(trees.ApproxDimension), 0.0);
        m.Leaves.Upload(padded);
    }
    if (exchangeBuilt.valid()) {
        finishExchange();
    }
    if (!leafCopies.empty()) {
        m.LeafRows.Upload(leafRows);
        size_t first = 0;
        for (const auto& [to, end] : leafCopies) {
            hipLaunchKernelGGL(dev::PlaceLeavesKernel, dim3(static_cast<uint32_t>(end - first)), dim3(64), 0, m.Stream, m.LeafRows.Get() + first,
                               static_cast<uint32_t>(m.Dim), static_cast<const double*>(m.Leaves.Get()), to);
            HIP_CHECK(hipGetLastError());
            first = end;
        }
        HIP_CHECK(hipStreamSynchronize(m.Stream));
    }
}

THipEvaluator::~THipEvaluator() = default;

size_t THipEvaluator::QuantizedBytes(size_t docCount) const {
    const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
    return std::max<size_t>(blocks, 1) * Impl->LayoutBuckets * dev::kDocsPerBlock;
}

void THipEvaluator::Synchronize(void* stream) {
    HIP_CHECK(hipStreamSynchronize(Impl->Pick(stream)));
}

namespace {

constexpr uint32_t kBinarizeBlocksPerGroup = 8;

template <int LOG2P, bool CATS_MATRIX>
void LaunchBinarizeRowsPC(size_t blocks, const float* floats, size_t stride, const int32_t* cats, size_t catStride,
                          size_t docCount, const dev::TBinarizeTables& tab, uint32_t* bins, hipStream_t s, hipEvent_t end) {
    const size_t tiles = (tab.BucketCount + dev::kBucketTile - 1) / dev::kBucketTile;
    // A workgroup keeps its tile's borders in LDS over up to kBinarizeBlocksPerGroup document blocks; a smaller batch gives
    // each fewer blocks, so that there are still a few generations of workgroups, whose phases overlap: whole call with about
    // 1024 workgroups and with 4096, 100 000 documents of 250 features, 300 trees 71.9 and 67.3 us, 200 000 119.0 and 111.9,
    // 200 000 of 100 features, four dimensions 94.2 and 91.3, 50 000 of 600 features 91.3 and 87.3; 100 000 of 50 to 200 features
    // the same within 1 %. Tables of 256 slots (20 KB) cost a workgroup more than that gives: a CTR model of 1M documents 364 us with 1024
    // and 373 with 4096. (Column-major batches, which have no tile to fill: 100 000 documents 69.6 and 71.7, so those keep 1024.)
    const uint32_t blocksPerGroup = static_cast<uint32_t>(
        std::max<size_t>(1, std::min<size_t>(kBinarizeBlocksPerGroup, blocks * tiles / (LOG2P < 8 ? 4096 : 1024))));
    const size_t groups = (blocks + blocksPerGroup - 1) / blocksPerGroup;
    CBAMD_ENSURE(groups * tiles < (size_t(1) << 31), "batch is too large for one binarize launch");
    const dim3 grid(static_cast<uint32_t>(groups * tiles));
    const size_t lds = (static_cast<size_t>(dev::kBucketTile) << LOG2P) * 4 +
                       static_cast<size_t>(dev::kBucketTile) * dev::kLutCells +
                       static_cast<size_t>(dev::kBucketTile) * dev::kTilePitch * 4;
    auto kernel = dev::BinarizeRowsKernel<LOG2P, CATS_MATRIX>;
    EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds);
    LaunchWithEnd(kernel, grid, dim3(256), lds, s, end, floats, static_cast<uint32_t>(stride), cats, static_cast<uint32_t>(catStride),
                  static_cast<uint32_t>(docCount), tab, blocksPerGroup, bins);
}

template <int LOG2P>
void LaunchBinarizeRowsP(size_t blocks, const float* floats, size_t stride, const int32_t* cats, size_t catStride,
                         size_t docCount, const dev::TBinarizeTables& tab, uint32_t* bins, hipStream_t s, hipEvent_t end) {
    if (cats != nullptr) {
        LaunchBinarizeRowsPC<LOG2P, true>(blocks, floats, stride, cats, catStride, docCount, tab, bins, s, end);
    } else {
        LaunchBinarizeRowsPC<LOG2P, false>(blocks, floats, stride, cats, catStride, docCount, tab, bins, s, end);
    }
}

// picks the smallest LDS slot count that still exceeds the largest bucket of the model
void LaunchBinarizeRows(uint32_t maxBucketValues, size_t blocks, const float* floats, size_t stride,
                        const int32_t* cats, size_t catStride, size_t docCount, const dev::TBinarizeTables& tab,
                        uint32_t* bins, hipStream_t s, hipEvent_t end) {
    CBAMD_ENSURE(docCount < (size_t(1) << 31) && stride < (size_t(1) << 31) && catStride < (size_t(1) << 31),
                 "batch is too large for one binarize launch");
    if (tab.BucketCount == 0) {
        return;  // a model of CTR features only
    }
    const int log2Slots = BinarizeLog2Slots(maxBucketValues);
    if (log2Slots == 5) {
        LaunchBinarizeRowsP<5>(blocks, floats, stride, cats, catStride, docCount, tab, bins, s, end);
    } else if (log2Slots == 6) {
        LaunchBinarizeRowsP<6>(blocks, floats, stride, cats, catStride, docCount, tab, bins, s, end);
    } else if (log2Slots == 7) {
        LaunchBinarizeRowsP<7>(blocks, floats, stride, cats, catStride, docCount, tab, bins, s, end);
    } else {
        LaunchBinarizeRowsP<8>(blocks, floats, stride, cats, catStride, docCount, tab, bins, s, end);
    }
}

template <int LOG2P>
void LaunchBinarizeColumnsP(size_t blocks, const float* floats, size_t stride, size_t docCount,
                            const dev::TBinarizeTables& tab, uint32_t* bins, hipStream_t s, hipEvent_t end) {
    const size_t tiles = (tab.BucketCount + dev::kBucketTile - 1) / dev::kBucketTile;
    const uint32_t blocksPerGroup = static_cast<uint32_t>(
        std::max<size_t>(1, std::min<size_t>(kBinarizeBlocksPerGroup, blocks * tiles / 1024)));
    const size_t groups = (blocks + blocksPerGroup - 1) / blocksPerGroup;
    CBAMD_ENSURE(groups * tiles < (size_t(1) << 31), "batch is too large for one binarize launch");
    const size_t lds = (static_cast<size_t>(dev::kBucketTile) << LOG2P) * 4 +
                       static_cast<size_t>(dev::kBucketTile) * dev::kLutCells;
    auto kernel = dev::BinarizeColumnsKernel<LOG2P>;
    EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds);
    LaunchWithEnd(kernel, dim3(static_cast<uint32_t>(groups * tiles)), dim3(256), lds, s, end, floats, stride,
                  static_cast<uint32_t>(docCount), tab, blocksPerGroup, bins);
}

// column-major documents: the same choice of LDS slots as for rows
void LaunchBinarizeColumns(uint32_t maxBucketValues, size_t blocks, const float* floats, size_t stride,
                           size_t docCount, const dev::TBinarizeTables& tab, uint32_t* bins, hipStream_t s, hipEvent_t end) {
    CBAMD_ENSURE(docCount < (size_t(1) << 31), "batch is too large for one binarize launch");
    const int log2Slots = BinarizeLog2Slots(maxBucketValues);
    if (log2Slots == 5) {
        LaunchBinarizeColumnsP<5>(blocks, floats, stride, docCount, tab, bins, s, end);
    } else if (log2Slots == 6) {
        LaunchBinarizeColumnsP<6>(blocks, floats, stride, docCount, tab, bins, s, end);
    } else if (log2Slots == 7) {
        LaunchBinarizeColumnsP<7>(blocks, floats, stride, docCount, tab, bins, s, end);
    } else {
        LaunchBinarizeColumnsP<8>(blocks, floats, stride, docCount, tab, bins, s, end);
    }
}

}  // namespace

void THipEvaluator::CheckBatch(const TFeatureBatch& batch, size_t docCount) const {
    const TImpl& m = *Impl;
    CBAMD_ENSURE(batch.Floats != nullptr || (batch.Layout == TFeatureBatch::SplitRows && m.MinFloatSize == 0),
                 "float features pointer is null");
    switch (batch.Layout) {
        case TFeatureBatch::FlatRows:
            CBAMD_ENSURE(batch.Stride >= m.FlatVectorSize, "insufficient flat features vector size: " +
                                                                std::to_string(batch.Stride) + " expected: " +
                                                                std::to_string(m.FlatVectorSize));
            break;
        case TFeatureBatch::SplitRows:
            CBAMD_ENSURE(batch.Stride >= m.MinFloatSize, "insufficient float features vector size: " +
                                                             std::to_string(batch.Stride) + " expected: " +
                                                             std::to_string(m.MinFloatSize));
            if (m.HasCats) {
                CBAMD_ENSURE(batch.Cats != nullptr, "Model has categorical features but no categorical features provided");
                CBAMD_ENSURE(batch.CatStride >= m.MinCatSize, "insufficient cat features vector size: " +
                                                                  std::to_string(batch.CatStride) + " expected: " +
                                                                  std::to_string(m.MinCatSize));
            }
            break;
        case TFeatureBatch::FlatColumns:
            CBAMD_ENSURE(batch.Stride >= docCount, "column stride is shorter than the document count");
            break;
        default:
            CBAMD_ENSURE(false, "unknown feature layout");
    }
}

void THipEvaluator::QuantizeDevice(const TFeatureBatch& batch, size_t docCount, uint8_t* bins, void* stream, TStageEnd* end) {
    TImpl& m = *Impl;
    if (docCount == 0) {
        return;
    }
    hipStream_t s = m.Pick(stream);
    const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
    CBAMD_ENSURE(blocks <= 0x7fffffffu, "too many documents in one batch");
    if (m.RealBucketCount == 0) {
        // a model without splits: one all-zero bucket per block keeps the layout non-empty
        CBAMD_ENSURE(bins != nullptr, "quantized buffer is null");
        const size_t dwords = QuantizedBytes(docCount) / 4;
        hipLaunchKernelGGL(dev::FillZeroKernel, dim3(static_cast<uint32_t>(std::min<size_t>((dwords + 255) / 256, 4096))),
                           dim3(256), 0, s, reinterpret_cast<uint32_t*>(bins), dwords);
        HIP_CHECK(hipGetLastError());
        return;
    }
    CBAMD_ENSURE(bins != nullptr, "quantized buffer is null");
    CheckBatch(batch, docCount);
    const hipEvent_t binarizeEnd = m.CtrCount > 0 || m.BinarizeBuckets == 0 ? nullptr : TakeEnd(end);
    switch (batch.Layout) {
        case TFeatureBatch::FlatRows:
            LaunchBinarizeRows(m.MaxBucketValues, blocks, batch.Floats, batch.Stride, nullptr, 0, docCount,
                               m.BinarizeTables(true), reinterpret_cast<uint32_t*>(bins), s, binarizeEnd);
            break;
        case TFeatureBatch::SplitRows:
            // a model with one-hot buckets always reads them from the categorical matrix here
            LaunchBinarizeRows(m.MaxBucketValues, blocks, batch.Floats, batch.Stride, m.HasCats ? batch.Cats : nullptr,
                               batch.CatStride, docCount, m.BinarizeTables(false), reinterpret_cast<uint32_t*>(bins), s, binarizeEnd);
            break;
        case TFeatureBatch::FlatColumns:
            if (m.BinarizeBuckets > 0) {
                LaunchBinarizeColumns(m.MaxBucketValues, blocks, batch.Floats, batch.Stride, docCount,
                                      m.BinarizeTables(true), reinterpret_cast<uint32_t*>(bins), s, binarizeEnd);
            }
            break;
    }
    HIP_CHECK(hipGetLastError());
    if (m.CtrCount > 0) {
        // the CTR features read the bins written above and the hashed categorical values
        dev::TCatSource cats;
        cats.SplitColumns = batch.Layout == TFeatureBatch::SplitRows ? 1u : 0u;
        if (batch.Layout == TFeatureBatch::SplitRows) {
            cats.Base = reinterpret_cast<const uint32_t*>(batch.Cats);
            cats.DocStride = batch.CatStride;
            cats.ColumnStride = 1;
        } else if (batch.Layout == TFeatureBatch::FlatRows) {
            cats.Base = reinterpret_cast<const uint32_t*>(batch.Floats);
            cats.DocStride = batch.Stride;
            cats.ColumnStride = 1;
        } else {
            cats.Base = reinterpret_cast<const uint32_t*>(batch.Floats);
            cats.DocStride = 1;
            cats.ColumnStride = batch.Stride;
        }
        // shares of the projections: a small batch has fewer blocks than the chip has room for workgroups
        const uint32_t groups = m.Ctr.GroupCount;
        const uint32_t wanted = static_cast<uint32_t>(std::max<size_t>(1, std::min<size_t>((groups + 3) / 4, 2048 / blocks)));
        const uint32_t groupsPerShare = (groups + wanted - 1) / wanted;
        const dim3 grid(static_cast<uint32_t>(blocks), (groups + groupsPerShare - 1) / groupsPerShare);
        if (m.CtrTileUsable) {
            const size_t lds = static_cast<size_t>(std::max<uint32_t>(m.Ctr.CatColumnCount, 1)) * dev::kCtrTilePitch * 4;
            LaunchWithEnd(dev::CtrBinarizeKernel<true>, grid, dim3(256), lds, s, TakeEnd(end), cats, static_cast<uint32_t>(docCount),
                          m.CtrTables(), m.LayoutBuckets, groupsPerShare, reinterpret_cast<uint32_t*>(bins));
        } else {
            LaunchWithEnd(dev::CtrBinarizeKernel<false>, grid, dim3(256), 0, s, TakeEnd(end), cats, static_cast<uint32_t>(docCount),
                          m.CtrTables(), m.LayoutBuckets, groupsPerShare, reinterpret_cast<uint32_t*>(bins));
        }
        HIP_CHECK(hipGetLastError());
    }
}

namespace {


// LDS of the half-tile kernel: 128 documents' bins, the accumulator, the per-wave leaf regions
size_t HalfTileLdsBytes(uint32_t buckets, int maxd) {
    return ((static_cast<size_t>(buckets) * 128 + 7) & ~size_t(7)) + 128 * sizeof(double) +
           static_cast<size_t>(dev::kTileWaves) * (size_t(1) << maxd) * sizeof(double);
}

// LDS of the per-wave leaf regions of the tile kernel
size_t TileLeafLdsBytes(int maxd, int dchunk, int waves = dev::kTileWaves) {
    return static_cast<size_t>(waves) * (size_t(1) << maxd) * dchunk * sizeof(double);
}

// leaf values go through LDS whenever the tile, the accumulator and the per-wave leaf regions
// fit the 160 KB of a CU (gathers from global memory cost ~50 L1 accesses per wave instruction)
bool TileLeavesInLds(uint32_t buckets, int maxd, int dchunk, bool pairAligned) {
    return pairAligned && TileLdsBytes(buckets, dchunk) + TileLeafLdsBytes(maxd, dchunk) <= kMaxTileLdsBytes;
}

// a tile of which only one workgroup fits a CU gets sixteen waves instead of eight, LDS permitting
int TileWaves(uint32_t buckets, int maxd, int dchunk, bool leavesInLds) {
    const size_t narrow = TileLdsBytes(buckets, dchunk) + (leavesInLds ? TileLeafLdsBytes(maxd, dchunk) : 0);
    const size_t wide = TileLdsBytes(buckets, dchunk) + (leavesInLds ? TileLeafLdsBytes(maxd, dchunk, dev::kWideTileWaves) : 0);
    return 2 * narrow > kMaxTileLdsBytes && wide <= kMaxTileLdsBytes ? dev::kWideTileWaves : dev::kTileWaves;
}

// the levels that EvalObliviousTileKernel walks
int TileLevels(uint32_t maxDepth) {
    return maxDepth <= 4 ? 4 : maxDepth <= 6 ? 6 : 8;
}

struct TTileArgs {
    const uint8_t* Bins;
    size_t DocCount;
    uint32_t Buckets;
    const uint32_t* PackedTrees;
    const double* Leaves;
    const double* Bias;
    double Scale;
    int Dim;
    uint32_t TreeBegin, TreeEnd;
    double* Out;
    hipStream_t Stream;
    bool LeavesPairAligned;
};

template <bool SEVEN_BIT, int MAXD, int DCHUNK, bool LEAF_LDS, int WAVES>
void LaunchEvalTileW(const TTileArgs& a) {
    const size_t blocks = (a.DocCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
    const size_t lds = TileLdsBytes(a.Buckets, DCHUNK) + (LEAF_LDS ? TileLeafLdsBytes(MAXD, DCHUNK, WAVES) : 0);
    auto kernel = dev::EvalObliviousTileKernel<SEVEN_BIT, MAXD, DCHUNK, LEAF_LDS, WAVES>;
    EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds);
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(blocks)), dim3(64 * WAVES), lds, a.Stream,
                       reinterpret_cast<const uint32_t*>(a.Bins), a.DocCount, a.Buckets, a.PackedTrees, a.Leaves, a.Bias,
                       a.Scale, a.Dim, a.TreeBegin, a.TreeEnd, a.Out);
}

template <bool SEVEN_BIT, int MAXD, int DCHUNK, bool LEAF_LDS>
void LaunchEvalTileL(const TTileArgs& a) {
    if (TileWaves(a.Buckets, MAXD, DCHUNK, LEAF_LDS) == dev::kWideTileWaves) {
        LaunchEvalTileW<SEVEN_BIT, MAXD, DCHUNK, LEAF_LDS, dev::kWideTileWaves>(a);
    } else {
        LaunchEvalTileW<SEVEN_BIT, MAXD, DCHUNK, LEAF_LDS, dev::kTileWaves>(a);
    }
}

template <bool SEVEN_BIT, int MAXD, int DCHUNK>
void LaunchEvalTile(const TTileArgs& a) {
    if (TileLeavesInLds(a.Buckets, MAXD, DCHUNK, a.LeavesPairAligned)) {
        LaunchEvalTileL<SEVEN_BIT, MAXD, DCHUNK, true>(a);
    } else {
        LaunchEvalTileL<SEVEN_BIT, MAXD, DCHUNK, false>(a);
    }
}

template <bool SEVEN_BIT, int MAXD>
void LaunchEvalTileD(int dchunk, const TTileArgs& a) {
    switch (dchunk) {
        case 1: LaunchEvalTile<SEVEN_BIT, MAXD, 1>(a); break;
        case 2: LaunchEvalTile<SEVEN_BIT, MAXD, 2>(a); break;
        case 4: LaunchEvalTile<SEVEN_BIT, MAXD, 4>(a); break;
        case 8: LaunchEvalTile<SEVEN_BIT, MAXD, 8>(a); break;
        case 12: LaunchEvalTile<SEVEN_BIT, MAXD, 12>(a); break;
        default: LaunchEvalTile<SEVEN_BIT, MAXD, 16>(a); break;
    }
}

template <bool SEVEN_BIT>
void LaunchEvalTileM(uint32_t maxDepth, int dchunk, const TTileArgs& a) {
    switch (TileLevels(maxDepth)) {
        case 4: LaunchEvalTileD<SEVEN_BIT, 4>(dchunk, a); break;
        case 6: LaunchEvalTileD<SEVEN_BIT, 6>(dchunk, a); break;
        default: LaunchEvalTileD<SEVEN_BIT, 8>(dchunk, a); break;
    }
}

template <bool NO_XOR, int DCHUNK>
void LaunchEvalNonSymmetricTileX(const uint8_t* bins, size_t docCount, uint32_t buckets, const uint2* entries,
                                 const uint4* rows, const double* leaves, const double* bias, double scale, int dim,
                                 uint32_t treeBegin, uint32_t treeEnd, double* out, hipStream_t s) {
    const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
    const size_t lds = TileLdsBytes(buckets, DCHUNK);
    auto kernel = dev::EvalNonSymmetricTileKernel<NO_XOR, DCHUNK>;
    EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds);
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(blocks)), dim3(64 * dev::kTileWaves), lds, s,
                       reinterpret_cast<const uint32_t*>(bins), docCount, buckets, entries, rows, leaves, bias, scale, dim,
                       treeBegin, treeEnd, out);
}

template <typename... TArgs>
void LaunchEvalNonSymmetricTile(bool noXor, int dchunk, TArgs... args) {
    if (noXor) {
        switch (dchunk) {
            case 1: LaunchEvalNonSymmetricTileX<true, 1>(args...); break;
            case 4: LaunchEvalNonSymmetricTileX<true, 4>(args...); break;
            default: LaunchEvalNonSymmetricTileX<true, 16>(args...); break;
        }
    } else {
        switch (dchunk) {
            case 1: LaunchEvalNonSymmetricTileX<false, 1>(args...); break;
            case 4: LaunchEvalNonSymmetricTileX<false, 4>(args...); break;
            default: LaunchEvalNonSymmetricTileX<false, 16>(args...); break;
        }
    }
}

template <int DCHUNK>
void LaunchEval(bool oblivious, const uint8_t* bins, size_t docCount, uint32_t buckets, const dev::TTreeTables& tt,
                uint32_t treeBegin, uint32_t treeEnd, double* out, hipStream_t s) {
    const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
    if (oblivious) {
        const uint32_t grid = static_cast<uint32_t>((blocks + 3) / 4);
        hipLaunchKernelGGL(dev::EvalObliviousKernel<DCHUNK>, dim3(grid), dim3(256), 0, s,
                           reinterpret_cast<const uint32_t*>(bins), docCount, buckets, tt, treeBegin, treeEnd, out, 0u, 2u);
    } else {
        hipLaunchKernelGGL(dev::EvalNonSymmetricKernel<DCHUNK>, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, s,
                           bins, docCount, buckets, tt, treeBegin, treeEnd, out);
    }
}

}  // namespace

// One branch per kernel, in the order in which EvalQuantizedDevice comes to them.
THipEvaluator::TImpl::TSumOrder THipEvaluator::TImpl::SumOrder() const {
    const int dchunk = TileChunk(Dim);
    TSumOrder order;
    if (TileRows.Get() != nullptr) {
        order.Waves = RowTileWaves(TileRowCount, MaxDepth, Dim);
    } else if (TileFits()) {
        const int levels = TileLevels(MaxDepth);
        const bool leavesInLds = TileLeavesInLds(LayoutBuckets, levels, dchunk, Dim > 1 || LeavesPairAligned);
        order.Waves = static_cast<uint32_t>(TileWaves(LayoutBuckets, levels, dchunk, leavesInLds));
    } else if (QuadRows.Get() != nullptr) {
        order.Waves = QuadTileWaves(TileRowCount, MaxDepth <= 6 ? 6 : 8);
        order.Side = 4;
        order.PerTree = true;
    } else if (Dim == 1 && HalfTileLeaves.Get() != nullptr && HalfTileLdsBytes(LayoutBuckets, 8) <= kMaxTileLdsBytes) {
        order.Waves = PairRows.Get() != nullptr ? dev::kPairWaves : dev::kTileWaves;
        order.Side = PairRows.Get() != nullptr ? 2 : 1;
    }
    return order;
}

void THipEvaluator::EvalQuantizedDevice(const uint8_t* bins, size_t docCount, size_t treeStart, size_t treeEnd,
                                        double* results, void* stream, TStageEnd* end) {
    TImpl& m = *Impl;
    if (docCount == 0) {
        return;
    }
    hipStream_t s = m.Pick(stream);
    CBAMD_ENSURE(results != nullptr, "results pointer is null");
    if (TreeCount == 0) {
        // a model without trees answers with its bias (cpu/formula_evaluator.cpp:29-41)
        const size_t count = docCount * m.Dim;
        hipLaunchKernelGGL(dev::FillBiasKernel, dim3(static_cast<uint32_t>((count + 255) / 256)), dim3(256), 0, s, results,
                           count, m.Bias.Get(), m.Dim);
        HIP_CHECK(hipGetLastError());
        return;
    }
    CBAMD_ENSURE(treeStart <= treeEnd && treeEnd <= TreeCount, "tree range is out of bounds");
    CBAMD_ENSURE(bins != nullptr, "quantized buffer is null");
    const dev::TTreeTables tt = m.TreeTables();
    const uint32_t tb = static_cast<uint32_t>(treeStart), te = static_cast<uint32_t>(treeEnd);
    if (m.RegKernelUsable) {
        // Bins kept in registers, a launch per group of dimensions (RegLaunches). A launch addresses its results with 32
        // bits, so a very large batch goes in slices of whole document blocks.
        const size_t sliceDocs = ((size_t(1) << 29) - 1) / m.Dim / dev::kDocsPerBlock * dev::kDocsPerBlock;
        if (docCount > sliceDocs) {
            for (size_t first = 0; first < docCount; first += sliceDocs) {
                const size_t n = std::min(sliceDocs, docCount - first);
                EvalQuantizedDevice(bins + first * m.LayoutBuckets, n, treeStart, treeEnd, results + first * m.Dim, stream);
            }
            return;
        }
        // The kernels walk whole blocks of RegTreeBlock trees. A range that starts or ends inside a block has
        // those few trees evaluated by the kernel that follows the model's own tables, before and after the
        // whole blocks: the launches hand on raw sums, each adds its trees in tree order, so the result is the
        // same sequence of additions as one pass over the range.
        const uint32_t block = m.RegTreeBlockSize;
        const uint32_t wholeBegin = (tb + block - 1) / block * block;
        const uint32_t wholeEnd = te == TreeCount ? te : te / block * block;  // null trees pad the model's last block
        const bool biased = treeStart == 0;
        const auto generic = [&](uint32_t begin, uint32_t end, uint32_t mode) {
            const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
            const dim3 grid(static_cast<uint32_t>((blocks + 3) / 4));
            const auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, reinterpret_cast<const uint32_t*>(bins), docCount,
                                   m.LayoutBuckets, tt, begin, end, results, mode, biased ? 1u : 0u);
            };
            if (m.Dim == 1) {
                launch(dev::EvalObliviousKernel<1>);
            } else if (m.Dim == 2) {
                launch(dev::EvalObliviousKernel<2>);
            } else if (m.Dim <= 4) {
                launch(dev::EvalObliviousKernel<4>);
            } else if (m.Dim <= 8) {
                launch(dev::EvalObliviousKernel<8>);
            } else {
                launch(dev::EvalObliviousKernel<16>);
            }
            HIP_CHECK(hipGetLastError());
        };
        if (wholeBegin >= wholeEnd) {
            generic(tb, te, 0);  // fewer trees than a block holds (or none: the bias alone)
            return;
        }
        const bool head = tb < wholeBegin, tail = wholeEnd < te;
        if (head) {
            generic(tb, wholeBegin, dev::kEvalRaw);
        }
        TEvalRegLaunchArgs launchArgs = {};
        TEvalRegArgs& args = launchArgs.Reg;
        args.Bins = bins;
        args.Rows = m.RegRows.Get() + static_cast<size_t>(wholeBegin) * m.RegRowDwords;
        args.Out = results;
        args.DocCount = static_cast<uint32_t>(docCount);
        args.BlockCount = static_cast<uint32_t>((docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock);
        const uint32_t flags = (biased && !tail ? 1u : 0u) | (head ? 2u : 0u) | (tail ? 4u : 0u) | (m.RegMap.Get() != nullptr ? kRegFlagMapped : 0u);
        launchArgs.RegMap = m.RegMap.Get();
        args.Scale = m.Scale;
        args.BucketCount = m.LayoutBuckets;
        args.Dim = static_cast<uint32_t>(m.Dim);
        for (const TImpl::TRegLaunch& l : m.RegLaunches) {
            args.Flags = flags | l.Flags;
            args.TreeBlocks = (wholeEnd - wholeBegin + l.TreeBlock - 1) / l.TreeBlock;
            launchArgs.TreeBlocksPerSlice = args.TreeBlocks;
            launchArgs.SlicesPerGroup = 1;
            args.Leaves = l.Leaves + static_cast<size_t>(wholeBegin) * l.TreeLeafDoubles;
            args.Bias = m.RegBias.Get() + l.FirstDim;
            args.FirstDim = l.FirstDim;
            args.StoreDims = l.StoreDims;
            const uint32_t grid = (args.BlockCount + l.Waves - 1) / l.Waves;
            const bool last = !tail && &l == &m.RegLaunches.back();
            LaunchModuleWithEnd(l.Function, grid, 1, 64 * l.Waves, s, last ? TakeEnd(end) : nullptr, launchArgs);
        }
        if (tail) {
            generic(wholeEnd, te, dev::kEvalContinue);
        }
        return;
    }
    const int dchunk = TileChunk(m.Dim);
    if (m.TileRows.Get() != nullptr) {
        // 7-bit bins, the tile fits: a tree's row in registers
        const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
        const uint32_t waves = RowTileWaves(m.TileRowCount, m.MaxDepth, m.Dim);
        const uint32_t dims = RowTileDims(m.MaxDepth, m.Dim);
        const size_t lds = RowTileLdsBytes(m.TileRowCount, m.MaxDepth, dims, waves);
        const auto launch = [&](auto kernel) {
            EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds);
            hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(blocks)), dim3(64 * waves), lds, s,
                               reinterpret_cast<const uint32_t*>(bins), docCount, m.LayoutBuckets, m.TileMap.Get(),
                               m.TileRowCount, reinterpret_cast<const uint4*>(m.TileRows.Get()),
                               reinterpret_cast<const double2*>(m.TileLeaves.Get()), m.Bias.Get(), m.Scale,
                               static_cast<uint32_t>(m.Dim), m.TileSliceStride, tb, te, results);
        };
        const bool wide = waves == dev::kWideTileWaves;
        if (m.MaxDepth <= 6) {
            if (dims == 1) {
                wide ? launch(dev::EvalObliviousRowTileKernel<6, dev::kWideTileWaves, 1>)
                     : launch(dev::EvalObliviousRowTileKernel<6, dev::kTileWaves, 1>);
            } else if (dims == 2) {
                wide ? launch(dev::EvalObliviousRowTileKernel<6, dev::kWideTileWaves, 2>)
                     : launch(dev::EvalObliviousRowTileKernel<6, dev::kTileWaves, 2>);
            } else {
                wide ? launch(dev::EvalObliviousRowTileKernel<6, dev::kWideTileWaves, 4>)
                     : launch(dev::EvalObliviousRowTileKernel<6, dev::kTileWaves, 4>);
            }
        } else if (dims == 1) {
            wide ? launch(dev::EvalObliviousRowTileKernel<8, dev::kWideTileWaves, 1>)
                 : launch(dev::EvalObliviousRowTileKernel<8, dev::kTileWaves, 1>);
        } else {
            wide ? launch(dev::EvalObliviousRowTileKernel<8, dev::kWideTileWaves, 2>)
                 : launch(dev::EvalObliviousRowTileKernel<8, dev::kTileWaves, 2>);
        }
        HIP_CHECK(hipGetLastError());
        return;
    }
    if (m.Oblivious && m.MaxDepth <= 8 && m.TileFits(tb != 0 || te != TreeCount ? te - tb : ~0u)) {
        // byte-parallel kernel over an LDS tile of bins
        const TTileArgs args{bins, docCount, m.LayoutBuckets, m.PackedTrees.Get(),
                             m.Dim == 1 ? m.Leaves.Get() : m.LeavesPadded.Get(), m.Bias.Get(), m.Scale, m.Dim, tb, te,
                             results, s, m.Dim == 1 ? m.LeavesPairAligned : true};
        if (m.PackedSevenBit) {
            LaunchEvalTileM<true>(m.MaxDepth, dchunk, args);
        } else {
            LaunchEvalTileM<false>(m.MaxDepth, dchunk, args);
        }
        HIP_CHECK(hipGetLastError());
        return;
    }
    if (m.QuadRows.Get() != nullptr) {
        // the rows do not fit the half tile: quarter blocks, four trees per wave
        const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
        const int maxd = m.MaxDepth <= 6 ? 6 : 8;
        const uint32_t waves = QuadTileWaves(m.TileRowCount, maxd);
        const size_t lds = QuadTileLdsBytes(m.TileRowCount, maxd, waves);
        CBAMD_ENSURE(4 * blocks < (size_t(1) << 31), "batch is too large for one evaluate launch");
        const auto launch = [&](auto kernel) {
            EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds);
            hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(4 * blocks)), dim3(64 * waves), lds, s, bins,
                               docCount, m.LayoutBuckets, m.TileMap.Get(), m.TileRowCount,
                               reinterpret_cast<const uint4*>(m.QuadRows.Get()),
                               reinterpret_cast<const double2*>(m.HalfTileLeaves.Get()), m.Bias.Get(), m.Scale, tb, te,
                               results);
        };
        if (maxd == 6) {
            waves == 8 ? launch(dev::EvalObliviousQuadTileKernel<6, 8>) : launch(dev::EvalObliviousQuadTileKernel<6, 4>);
        } else {
            waves == 8 ? launch(dev::EvalObliviousQuadTileKernel<8, 8>) : launch(dev::EvalObliviousQuadTileKernel<8, 4>);
        }
        HIP_CHECK(hipGetLastError());
        return;
    }
    if (m.Oblivious && m.MaxDepth <= 8 && m.Dim == 1 && m.HalfTileLeaves.Get() != nullptr &&
        HalfTileLdsBytes(m.LayoutBuckets, 8) <= kMaxTileLdsBytes) {
        // the bins of a block exceed the 256-document tile: half blocks
        const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
        const int maxd = m.MaxDepth <= 6 ? 6 : 8;
        if (m.TakesExchangeKernel(docCount) && tb == 0 && te == TreeCount && (reinterpret_cast<uintptr_t>(bins) & 3) == 0) {
            TEvalExchangeArgs args = m.ExchangeArgs(docCount, results);
            args.Bins = bins;
            LaunchModuleWithEnd(m.ExchangeFunction, static_cast<uint32_t>(blocks), 1, 64 * kExchangeWaves, s, TakeEnd(end), args);
            return;
        }
        if (m.PairRows.Get() != nullptr) {
            const size_t lds = PairTileLdsBytes(m.TileRowCount, maxd);
            const auto launch = [&](auto kernel) {
                EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds);
                hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(2 * blocks)), dim3(64 * dev::kPairWaves), lds, s,
                                   reinterpret_cast<const uint16_t*>(bins), docCount, m.LayoutBuckets, m.TileMap.Get(),
                                   m.TileRowCount, reinterpret_cast<const uint2*>(m.PairRows.Get()),
                                   reinterpret_cast<const double2*>(m.HalfTileLeaves.Get()), m.Bias.Get(), m.Scale, tb, te,
                                   results);
            };
            if (maxd == 6) {
                m.PairSix ? launch(dev::EvalObliviousPairTileKernel<6, true>) : launch(dev::EvalObliviousPairTileKernel<6, false>);
            } else {
                m.PairSix ? launch(dev::EvalObliviousPairTileKernel<8, true>) : launch(dev::EvalObliviousPairTileKernel<8, false>);
            }
            HIP_CHECK(hipGetLastError());
            return;
        }
        const size_t lds = HalfTileLdsBytes(m.LayoutBuckets, maxd);
        const auto launch = [&](auto kernel) {
            EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds);
            hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(2 * blocks)), dim3(64 * dev::kTileWaves), lds, s,
                               reinterpret_cast<const uint16_t*>(bins), docCount, m.LayoutBuckets, m.PackedMixed.Get(),
                               m.HalfTileLeaves.Get(), m.Bias.Get(), m.Scale, tb, te, results);
        };
        if (maxd == 6) {
            launch(dev::EvalObliviousHalfTileKernel<6>);
        } else {
            launch(dev::EvalObliviousHalfTileKernel<8>);
        }
        HIP_CHECK(hipGetLastError());
        return;
    }
    // A unit holds trees of like height from anywhere in the model, so a range of the trees still walks most
    // units: the kernel that walks the range's trees alone is the faster for about a tenth of them. Evaluate launch, that kernel and this
    // one, three tenths, a fifth and a tenth of the trees: 500 of depth 10 over 300 features (500 000 documents) 483 and 365, 326 and 303, 191
    // and 234 us; 500 of depth 6 over 60 (1M) 552 and 292, 377 and 279, 203 and 215; three dimensions, 300 of depth 8 over 100 (500 000) 293
    // and 196, 204 and 166, 115 and 123; 100 of depth 8 over 50 (1M) 161 and 147, 110 and 142, 71 and 115. (The line is where it was with the
    // walk from the root; of the seven models measured the smallest alone crosses above a fifth.)
    if (!m.Oblivious && m.NsLdsUsable && (treeEnd - treeStart) * 10 >= TreeCount * 3) {
        const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
        const uint32_t dims = NsLdsDims(m.Dim);
        const size_t lds = NsLdsKernelBytes(m.LayoutBuckets, m.NsLdsShape.Waves, m.NsLdsShape.Entries, dims);
        const auto launch = [&](auto kernel) {
            EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds);
            const dim3 grid(static_cast<uint32_t>(blocks), (static_cast<uint32_t>(m.Dim) + dims - 1) / dims);
            hipLaunchKernelGGL(kernel, grid, dim3(64 * m.NsLdsShape.Waves), lds, s,
                               reinterpret_cast<const uint32_t*>(bins), docCount, m.LayoutBuckets,
                               m.NsCompactEntries.Get(), m.NsCompactRows.Get(),
                               m.NsUnitCount, m.NsValuesByEntry.Get(), m.Bias.Get(), m.Scale,
                               static_cast<uint32_t>(m.Dim), m.NsEntryCount, tb, te,
                               static_cast<uint32_t>(treeStart == 0 && treeEnd == TreeCount), results);
        };
        const auto tryShape = [&](auto waves, auto entries) {
            constexpr int W = decltype(waves)::value, E = decltype(entries)::value;
            if (m.NsLdsShape.Waves != W || m.NsLdsShape.Entries != E) {
                return false;
            }
            if (dims == 1) {
                launch(dev::EvalNonSymmetricLdsKernel<W, E, 1>);
            } else if (dims == 2) {
                launch(dev::EvalNonSymmetricLdsKernel<W, E, 2>);
            } else {
                launch(dev::EvalNonSymmetricLdsKernel<W, E, 4>);
            }
            return true;
        };
        const bool launched = LaunchOfShape(tryShape, std::make_index_sequence<std::size(kNsLdsShapes)>());
        CBAMD_ENSURE(launched, "internal error: no kernel of this shape");
        HIP_CHECK(hipGetLastError());
        return;
    }
    if (!m.Oblivious && m.NsTileUsable) {
        const int nsChunk = m.Dim == 1 ? 1 : m.Dim <= 4 ? 4 : 16;
        if (TileLdsBytes(m.LayoutBuckets, nsChunk) <= kMaxTileLdsBytes) {
            LaunchEvalNonSymmetricTile(m.NsNoXor, nsChunk, bins, docCount, m.LayoutBuckets,
                                       reinterpret_cast<const uint2*>(m.NsEntries.Get()),
                                       reinterpret_cast<const uint4*>(m.NsRows.Get()), m.Leaves.Get(), m.Bias.Get(),
                                       m.Scale, m.Dim, tb, te, results, s);
            HIP_CHECK(hipGetLastError());
            return;
        }
    }
    if (m.DeepRows.Get() != nullptr) {
        const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
        const int dims = DeepTileDims(m.Dim);
        const uint32_t slices = (static_cast<uint32_t>(m.Dim) + dims - 1) / dims;
        const size_t lds = DeepTileLdsBytes(m.TileRowCount, dims);
        const bool wide = 2 * lds > kMaxTileLdsBytes;  // one workgroup per CU: sixteen waves
        const dim3 grid(static_cast<uint32_t>(blocks), slices), threads(64 * (wide ? dev::kWideTileWaves : dev::kTileWaves));
        const auto launch = [&](auto kernel) {
            EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds);
            hipLaunchKernelGGL(kernel, grid, threads, lds, s, reinterpret_cast<const uint32_t*>(bins), docCount, m.LayoutBuckets,
                               m.TileMap.Get(), m.TileRowCount, reinterpret_cast<const uint4*>(m.DeepRows.Get()),
                               m.DeepFirstLeaf.Get(), m.Leaves.Get(), m.Bias.Get(), m.Scale, tb, te, results);
        };
        const auto launchPairs = [&](auto kernel) {
            EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds);
            hipLaunchKernelGGL(kernel, grid, threads, lds, s, reinterpret_cast<const uint32_t*>(bins), docCount, m.LayoutBuckets,
                               m.TileMap.Get(), m.TileRowCount, reinterpret_cast<const uint4*>(m.DeepRows.Get()),
                               m.DeepFirstLeaf.Get(), m.DeepLeaves.Get(), m.Bias.Get(), m.Scale, static_cast<uint32_t>(m.Dim),
                               m.DeepSliceLeaves, tb, te, results);
        };
        if (dims == 1) {
            if (m.MaxDepth <= 12) {
                wide ? launch(dev::EvalObliviousDeepTileKernel<4, dev::kWideTileWaves>)
                     : launch(dev::EvalObliviousDeepTileKernel<4, dev::kTileWaves>);
            } else {
                wide ? launch(dev::EvalObliviousDeepTileKernel<8, dev::kWideTileWaves>)
                     : launch(dev::EvalObliviousDeepTileKernel<8, dev::kTileWaves>);
            }
        } else if (m.MaxDepth <= 12) {
            wide ? launchPairs(dev::EvalObliviousDeepTilePairsKernel<4, dev::kWideTileWaves>)
                 : launchPairs(dev::EvalObliviousDeepTilePairsKernel<4, dev::kTileWaves>);
        } else {
            wide ? launchPairs(dev::EvalObliviousDeepTilePairsKernel<8, dev::kWideTileWaves>)
                 : launchPairs(dev::EvalObliviousDeepTilePairsKernel<8, dev::kTileWaves>);
        }
        HIP_CHECK(hipGetLastError());
        return;
    }
    if (m.Dim == 1) {
        LaunchEval<1>(m.Oblivious, bins, docCount, m.LayoutBuckets, tt, tb, te, results, s);
    } else if (m.Dim == 2) {
        LaunchEval<2>(m.Oblivious, bins, docCount, m.LayoutBuckets, tt, tb, te, results, s);
    } else if (m.Dim <= 4) {
        LaunchEval<4>(m.Oblivious, bins, docCount, m.LayoutBuckets, tt, tb, te, results, s);
    } else if (m.Dim <= 8) {
        LaunchEval<8>(m.Oblivious, bins, docCount, m.LayoutBuckets, tt, tb, te, results, s);
    } else {
        LaunchEval<16>(m.Oblivious, bins, docCount, m.LayoutBuckets, tt, tb, te, results, s);
    }
    HIP_CHECK(hipGetLastError());
}

uint32_t THipEvaluator::TreeSlicesFor(size_t docCount) const {
    const TImpl& m = *Impl;
    // (a slice's results are addressed with 32 bits, as a launch's are: models of more than 2047 dimensions can pass that)
    if (!m.RegKernelUsable || !m.SmallBatchSlices || docCount == 0 || docCount >= (size_t(1) << 29) / m.Dim) {
        return 1;
    }
    // Workgroups of a plain launch; below one per CU the launch lasts as long as one wave's walk through the
    // whole model, so the trees are cut into slices with workgroups of their own. A slice is two tree blocks
    // whatever the batch, so that a document's value does not depend on how many documents came with it
    // (as long as the batch is small enough to be sliced at all).
    const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
    const size_t groups = (blocks + m.RegWaves - 1) / m.RegWaves;
    const size_t sliceTrees = RegSliceTrees(m.RegTreeBlockSize);
    if (groups >= 256 || TreeCount < 2 * sliceTrees) {
        return 1;
    }
    return static_cast<uint32_t>((TreeCount + sliceTrees - 1) / sliceTrees);
}

size_t THipEvaluator::TreeSliceScratchDoubles(size_t docCount) const {
    const uint32_t slices = TreeSlicesFor(docCount);
    return slices > 1 ? static_cast<size_t>(slices) * docCount * Impl->Dim : 0;
}

void THipEvaluator::EvalQuantizedSlicedDevice(const uint8_t* bins, size_t docCount, double* results, double* partials,
                                              void* stream, TStageEnd* end) {
    TImpl& m = *Impl;
    const uint32_t slices = TreeSlicesFor(docCount);
    if (slices <= 1) {
        EvalQuantizedDevice(bins, docCount, 0, TreeCount, results, stream, end);
        return;
    }
    CBAMD_ENSURE(bins != nullptr && results != nullptr && partials != nullptr, "null pointer passed to the sliced evaluation");
    hipStream_t s = m.Pick(stream);
    TEvalRegLaunchArgs launchArgs = {};
    TEvalRegArgs& args = launchArgs.Reg;
    args.Bins = bins;
    args.Rows = m.RegRows.Get();
    args.Out = partials;
    args.DocCount = static_cast<uint32_t>(docCount);
    args.BlockCount = static_cast<uint32_t>((docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock);
    const uint32_t flags = 4 | (m.RegMap.Get() != nullptr ? kRegFlagMapped : 0u);  // raw sums per slice
    launchArgs.RegMap = m.RegMap.Get();
    args.Scale = m.Scale;
    args.BucketCount = m.LayoutBuckets;
    args.Dim = static_cast<uint32_t>(m.Dim);
    // a slice is the same number of trees in every launch
    const uint32_t sliceTrees = RegSliceTrees(m.RegTreeBlockSize);
    for (const TImpl::TRegLaunch& l : m.RegLaunches) {
        args.Flags = flags | l.Flags;
        args.TreeBlocks = static_cast<uint32_t>((TreeCount + l.TreeBlock - 1) / l.TreeBlock);
        launchArgs.TreeBlocksPerSlice = sliceTrees / l.TreeBlock;
        args.Leaves = l.Leaves;
        args.Bias = m.RegBias.Get() + l.FirstDim;
        args.FirstDim = l.FirstDim;
        args.StoreDims = l.StoreDims;
        const uint32_t grid = (args.BlockCount + l.Waves - 1) / l.Waves;
        launchArgs.SlicesPerGroup = RegSlicesPerGroup(grid, slices, size_t(256) * l.GroupsPerCu);
        const uint32_t shares = (slices + launchArgs.SlicesPerGroup - 1) / launchArgs.SlicesPerGroup;
        LaunchModuleWithEnd(l.Function, grid, shares, 64 * l.Waves, s, nullptr, launchArgs);
    }
    const size_t count = docCount * m.Dim;
    const auto combine = [&](auto kernel) {
        LaunchWithEnd(kernel, dim3(static_cast<uint32_t>((count + 63) / 64)), dim3(64), 0, s, TakeEnd(end),
                      static_cast<const double*>(partials), slices, count, m.Scale, m.Bias.Get(), m.Dim, results);
    };
    slices <= dev::kFewSlices ? combine(dev::CombineSlicesKernel<3>) : combine(dev::CombineSlicesKernel<16>);
    HIP_CHECK(hipGetLastError());
}

// The largest batch of the small-batch kernel: see kSmallBatchDocs.
bool THipEvaluator::TakesSmallBatchKernel(size_t docCount, size_t treeStart, size_t treeEnd) const {
    const TImpl& m = *Impl;
    return m.SmallUsable && m.SmallBatchSlices && docCount > 0 && docCount * m.SmallPasses() <= kSmallBatchDocs && treeStart == 0 &&
           treeEnd == TreeCount && m.SmallLdsBytes() <= kMaxTileLdsBytes;
}

// ... of calls whose features are on the device. Its time grows with the levels that a document walks, and by a step for every 4096
// documents (a workgroup of sixteen more on every CU), the one of binarize and evaluate launches hardly, so models of many levels
// take those earlier. Whole call, SmallBatchKernel and the launches: 1000 trees of depth 8 over 200 features, 8192 documents 29.5
// and 32.4 us, 10 240 36.2 and 35.4, 12 400 43.2 and 36.9, 16 384 46.3 and 37.5 (columns of 50 features, 8300 documents 34.2 and 35.6, 16 384
// 44.4 and 36.8); 1000 of depth 6 over 100, 12 288 30.1 and 31.5, 12 400 33.5 and 32.7, 16 384 35.3 and 32.8; 500 of depth 6
// over 150, 16 384 28.1 and 30.7, 300 of depth 8 over 60 28.7 and 30.2. (One dimension on the register kernels; both add the same
// slices. Other models keep the one limit.) The columns to binarize are not looked at, and many of them cost the launches more than the lines suppose:
// 12 289 documents, 501 trees of depth 8 over 200 columns 28.6 and 33.1 us, 833 of depth 6 over 222 31.2 and 35.5, where 563 of depth
// 8 over 60 take 31.7 and 28.3. Of 696 batches of 4000 to 16 000 levels and 20 to 222 columns none is longer on the launches with lines at
// 5000 and 6500 levels, and 12.5 and 20 more for every column beyond 100.
bool THipEvaluator::TakesSmallBatchOnDevice(size_t docCount, size_t treeStart, size_t treeEnd) const {
    const TImpl& m = *Impl;
    const size_t levels = TreeCount * static_cast<size_t>(m.MaxDepth);
    const size_t limit = levels <= 4000 ? kSmallBatchDocs : levels <= 6500 ? 12288 : 10240;
    return TakesSmallBatchKernel(docCount, treeStart, treeEnd) && (m.Dim > 1 || TreeSlicesFor(docCount) <= 1 || docCount <= limit);
}

// One launch of the small-batch kernel whose end `stop` marks. `batch` and `results` may be device or pinned host memory.
// `flagged`: the slot whose flags the workgroups of FewDocumentsKernel set (AwaitSmallBatch).
static void LaunchSmallBatch(THipEvaluator::TImpl& m, THipEvaluator::TImpl::THostContext& ctx, const TFeatureBatch& batch,
                             size_t docCount, double* results, hipStream_t s, hipEvent_t stop,
                             THipEvaluator::TImpl::THostSlot* flagged = nullptr) {
    CBAMD_ENSURE(results != nullptr, "results pointer is null");
    dev::TSmallSource src = {};
    src.Floats = reinterpret_cast<const uint32_t*>(batch.Floats);
    const bool columns = batch.Layout == TFeatureBatch::FlatColumns;
    src.DocStride = columns ? 1 : batch.Stride;
    src.ColumnStride = columns ? batch.Stride : 1;
    src.Cats = reinterpret_cast<const uint32_t*>(batch.Cats);
    src.CatStride = batch.CatStride;
    src.Split = batch.Layout == TFeatureBatch::SplitRows ? 1u : 0u;
    dev::TSmallTables tab = {};
    tab.Cells = reinterpret_cast<const dev::TSmallCell*>(m.SmallTable.Get() + m.SmallCellsAt);
    tab.TreeRows = m.SmallTable.Get();
    tab.FirstLeaf = m.SmallTable.Get() + m.SmallFirstLeafAt;
    tab.Leaves = m.SmallLeaves.Get();
    tab.Bias = m.Bias.Get();
    tab.Scale = m.Scale;
    tab.CellCount = m.SmallCellCount;
    tab.Dim = static_cast<uint32_t>(m.Dim);
    tab.TreeCount = m.SmallTreeCount;
    tab.SliceTrees = m.SmallSliceTrees;
    tab.SliceCount = m.SmallSliceCount();
    const uint32_t dims = static_cast<uint32_t>(m.SmallDims());
    const uint32_t passes = m.SmallPasses();
    const auto launch = [&](auto kernel, size_t groups, uint32_t threads, size_t lds, auto... more) {
        const THipEvaluator::TImpl::TSmallStamps& stamps = ctx.StampsForLaunch(groups * passes);
        EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds);
        hipExtLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(groups), passes), dim3(threads), lds, s, nullptr, stop, 0, src,
                              static_cast<uint32_t>(docCount), tab, results, reinterpret_cast<ulonglong2*>(stamps.Values.Get()), more...);
    };
    const auto launchFew = [&](auto kernel) {
        dev::TSmallDone done = {};
        if (flagged != nullptr) {
            const size_t groups = docCount * passes;
            CBAMD_ENSURE(groups <= kFlaggedGroups, "internal error: more workgroups than flags");
            if (++flagged->SmallTicket == 0) {
                std::memset(flagged->SmallFlags(), 0, kFlaggedGroups * sizeof(uint32_t));
                flagged->SmallTicket = 1;
            }
            done.Flags = flagged->SmallFlags();
            done.Ticket = flagged->SmallTicket;
            flagged->SmallGroups = groups;
        }
        launch(kernel, docCount, std::min<uint32_t>(dev::kFewThreads, (tab.TreeCount + 63) / 64 * 64), m.FewLdsBytes(), done);
    };
    const auto launchSmall = [&](auto kernel) {
        launch(kernel, (docCount + dev::kSmallDocs - 1) / dev::kSmallDocs, dev::kSmallThreads, m.SmallLdsBytes());
    };
    const bool shallow = m.MaxDepth <= 6;
    if (m.TakesFewDocumentsKernel(docCount)) {
        if (dims == 1) {
            shallow ? launchFew(dev::FewDocumentsKernel<6, 1>) : launchFew(dev::FewDocumentsKernel<8, 1>);
        } else if (dims == 2) {
            shallow ? launchFew(dev::FewDocumentsKernel<6, 2>) : launchFew(dev::FewDocumentsKernel<8, 2>);
        } else {
            shallow ? launchFew(dev::FewDocumentsKernel<6, 4>) : launchFew(dev::FewDocumentsKernel<8, 4>);
        }
    } else if (dims == 1) {
        shallow ? launchSmall(dev::SmallBatchKernel<6, 1>) : launchSmall(dev::SmallBatchKernel<8, 1>);
    } else if (dims == 2) {
        shallow ? launchSmall(dev::SmallBatchKernel<6, 2>) : launchSmall(dev::SmallBatchKernel<8, 2>);
    } else {
        shallow ? launchSmall(dev::SmallBatchKernel<6, 4>) : launchSmall(dev::SmallBatchKernel<8, 4>);
    }
    HIP_CHECK(hipGetLastError());
}

// Waits for the workgroups of a launch with flags. The launch itself may not have been retired when this returns; what follows
// on its stream is ordered behind it. A launch that takes long (or has failed) is waited for as usual.
static void AwaitSmallBatch(THipEvaluator::TImpl& m, const THipEvaluator::TImpl::THostSlot& slot, hipEvent_t stop) {
    const uint32_t* flags = slot.SmallFlags();
    const auto started = std::chrono::steady_clock::now();
    size_t group = 0;
    for (uint32_t turn = 0; group < slot.SmallGroups; ++turn) {
        if (m.FlagWaitUs != 0 && __atomic_load_n(flags + group, __ATOMIC_ACQUIRE) == slot.SmallTicket) {
            ++group;
        } else if ((turn % 256 == 255 || m.FlagWaitUs == 0) && std::chrono::steady_clock::now() - started >= std::chrono::microseconds(m.FlagWaitUs)) {
            HIP_CHECK(hipEventSynchronize(stop));
            return;
        }
    }
    if (m.CountFlagged) {
        m.FlaggedCalls.fetch_add(1, std::memory_order_relaxed);
    }
}

int THipEvaluator::FusedLayoutFor(int layout, size_t stride, size_t docCount, size_t treeStart, size_t treeEnd, bool anyBatchSize) const {
    const TImpl& m = *Impl;
    const int layoutIndex = layout == TFeatureBatch::FlatRows ? 0 : layout == TFeatureBatch::SplitRows ? 1 : layout == TFeatureBatch::FlatColumns ? 2 : -1;
    if (layoutIndex < 0 || docCount == 0) {
        return -1;
    }
    if (layoutIndex == 0 && treeStart == 0 && treeEnd == TreeCount && stride < (size_t(1) << 20) &&
        m.TakesFusedExchangeKernel(docCount, anyBatchSize)) {
        return kFusedExchange;
    }
    if (!m.Fused[layoutIndex] || treeStart != 0 || treeEnd != TreeCount || docCount >= (size_t(1) << 29) ||
        stride >= (size_t(1) << (layoutIndex == 2 ? 30 : 20))) {
        return -1;
    }
    if (!anyBatchSize && docCount < m.FusedMinDocs()) {
        return -1;
    }
    if (!anyBatchSize && layoutIndex == 2 &&
        (m.FewColumnsForFused(docCount, TreeCount) || (TreeSlicesFor(docCount) > 1 && m.SlicesBeforeFusedColumns(docCount, TreeCount)))) {
        return -1;
    }
    return layoutIndex;
}

bool THipEvaluator::EvalFusedDevice(const TFeatureBatch& batch, size_t docCount, size_t treeStart, size_t treeEnd,
                                    double* results, void* stream, bool anyBatchSize, TStageEnd* end) {
    TImpl& m = *Impl;
    const int layoutIndex = FusedLayoutFor(batch.Layout, batch.Stride, docCount, treeStart, treeEnd, anyBatchSize);
    if (layoutIndex < 0) {
        return false;
    }
    if (layoutIndex == kFusedExchange) {
        CBAMD_ENSURE(results != nullptr, "results pointer is null");
        CheckBatch(batch, docCount);
        TFusedExchangeArgs args = {m.ExchangeArgs(docCount, results), batch.Floats, m.FusedExchangeTiles.Get(),
                                   static_cast<uint32_t>(batch.Stride * sizeof(float)), m.FusedExchangeTileCount, m.FusedExchangeOneHot.Get()};
        args.Walk.WaveTable = m.FusedExchangeWaves.Get();
        const size_t blocks = (docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock;
        LaunchModuleWithEnd(m.FusedExchangeFunction, static_cast<uint32_t>(blocks), 1, 64 * kExchangeWaves, m.Pick(stream), TakeEnd(end), args);
        return true;
    }
    const TImpl::TFused& f = *m.Fused[layoutIndex];
    CBAMD_ENSURE(results != nullptr, "results pointer is null");
    CBAMD_ENSURE(batch.Floats != nullptr, "float features pointer is null");
    if (layoutIndex == 2) {
        CheckBatch(batch, docCount);
    }
    const size_t need = layoutIndex == 0 ? m.FlatVectorSize : layoutIndex == 1 ? m.MinFloatSize : 0;
    CBAMD_ENSURE(batch.Stride >= need, (layoutIndex == 0 ? "insufficient flat features vector size: " : "insufficient float features vector size: ") +
                                           std::to_string(batch.Stride) + " expected: " + std::to_string(need));
    TEvalFusedArgs args = {};
    args.Reg.Rows = f.Rows.Get();
    args.Reg.Leaves = f.Table.Get();
    args.Reg.Out = results;
    args.Reg.DocCount = static_cast<uint32_t>(docCount);
    args.Reg.BlockCount = static_cast<uint32_t>((docCount + dev::kDocsPerBlock - 1) / dev::kDocsPerBlock);
    args.Reg.TreeBlocks = m.RegTreeBlocks;
    args.Reg.Flags = 1;
    args.Reg.Scale = m.Scale;
    args.Reg.Bias = m.RegBias.Get();
    args.Reg.BucketCount = m.LayoutBuckets;
    args.Reg.Dim = 1;
    args.Reg.FirstDim = 0;
    args.Reg.StoreDims = 1;
    args.Floats = batch.Floats;
    args.Units = f.Units.Get();
    args.StrideBytes = static_cast<uint32_t>(batch.Stride * sizeof(float));
    args.UnitCount = f.UnitCount;
    const uint32_t grid = (args.Reg.BlockCount + f.Waves - 1) / f.Waves;
    // Workgroups that start together wait for their rows together and walk their trees together. The second ones of the
    // CUs start when the rows of the first ones have arrived (6 TB/s: early rather than late; 4.5 gives the same within
    // 1 %, with 3.5 batches of one generation lose what they gain), so that one set walks while the other loads; a part of
    // them waits less. Rows from HBM, whole call, without and with the delay: 1M documents of 50 features, trees of depth 6:
    // 10 trees 75.8 and 74.3 us, 100 89.4 and 87.6, 200 105.8 and 102.9, 500 158.7 and 154.9; 700 000 of 200 features, depth 8:
    // 10 trees 152.2 and 152.2, 30 194.6 and 189.2, 500 275.0 and 264.6; 4M of 200 features, 1000 trees 1608 and 1598; rows of
    // 64 features and up to 30 trees lose, 2M documents 127.8 and 130.5. Two to eight callers at a time gain as one does (1M
    // documents of 200 features, 100 trees 248 and 240 us a call).
    // Batches of one generation whose rows arrive at the full rate as they are, as columns do, would only end later: rows
    // of up to a line or two (1M documents of 17 features, 30 trees 36.8 and 38.8 us), and, in the shapes of four waves,
    // rows that are whole pieces of 64 bytes (520 000 documents, 1000 trees of depth 8: 128 features 208.9 and 219.8 us, 160
    // 222.4 and 231.4, 192 220.3 and 232.3; 127 246.7 and 240.8, 145 246.7 and 243.8, 193 261.7 and 258.2; of eight waves: 1M
    // documents of 80 features, 500 trees 177.7 and 172.9). In several generations those rows gain or lose 1 to 2 %, but
    // rows of 512 bytes lose (128 features: 700 000 documents, 100 trees 112.7 and 118.2, 1M, 1000 trees 391.8 and 399.9).
    const bool wholePieces = (reinterpret_cast<uintptr_t>(batch.Floats) | args.StrideBytes) % 64 == 0;
    const bool oneGeneration = grid <= 2 * kLateStartCus;
    const bool fullRate = f.Waves == 4 && wholePieces ? oneGeneration || args.StrideBytes % 512 == 0 : oneGeneration && args.StrideBytes <= 128;
    if (layoutIndex != 2 && m.CuCount == kLateStartCus && !fullRate) {
        const double secondGroups = std::min<double>(kLateStartCus, std::max<double>(kLateStartCus, grid) - kLateStartCus);
        const double rowBytes = std::min(args.StrideBytes, f.UnitCount * kFusedUnitColumns * 4);
        const double loadSeconds = secondGroups * f.Waves * dev::kDocsPerBlock * rowBytes / 6e12, turnSeconds = 4096 / 2.4e9;
        args.Reg.Bins = reinterpret_cast<const void*>(static_cast<uintptr_t>(std::min(loadSeconds / turnSeconds, 64.0)));
    }
    LaunchModuleWithEnd(f.Function, grid, 1, 64 * f.Waves, m.Pick(stream), TakeEnd(end), args);
    return true;
}

std::string THipEvaluator::DescribeKernels(int layout, size_t docCount, size_t stride) const {
    const TImpl& m = *Impl;
    // whole-model calls only: a call for a range of the trees may take other kernels
    if (const int fused = FusedLayoutFor(layout, stride, docCount, 0, TreeCount, false); fused >= 0) {
        return "fused=" + (fused == kFusedExchange ? m.FusedExchangeName : m.Fused[fused]->Name);
    }
    if (TakesSmallBatchOnDevice(docCount, 0, TreeCount)) {
        const bool few = m.TakesFewDocumentsKernel(docCount);
        return std::string("binarize=none;evaluate=") + (few ? "FewDocumentsKernel<" : "SmallBatchKernel<") + std::to_string(m.MaxDepth <= 6 ? 6 : 8) + ", " + std::to_string(m.SmallDims()) +
               ">, " + std::to_string(m.SmallSliceCount()) + " slices of the trees" +
               (m.CountFlagged ? ";flagged=" + std::to_string(m.FlaggedCalls.load()) : "");
    }
    std::string binarize = m.BinarizeBuckets == 0 ? "none"
                           : layout == TFeatureBatch::FlatColumns
                               ? "BinarizeColumnsKernel"
                               : "BinarizeRowsKernel<" + std::to_string(BinarizeLog2Slots(m.MaxBucketValues)) + ">";
    if (m.CtrCount > 0) {
        binarize += m.CtrTileUsable ? "+CtrBinarizeKernel<true>" : "+CtrBinarizeKernel<false>";
    }
    const int dchunk = TileChunk(m.Dim);
    std::string evaluate;
    if (TreeCount == 0) {
        evaluate = "FillBiasKernel";
    } else if (m.RegKernelUsable) {
        evaluate = m.RegKernelName;
        if (m.RegLaunches.size() > 1) {
            const size_t main = m.RegLaunches.size() - (m.RegTailLeaves.Get() != nullptr ? 1 : 0);
            if (main > 1) {
                evaluate += " x " + std::to_string(main) + " launches";
            }
            if (main < m.RegLaunches.size()) {
                evaluate += std::string(" + ") + m.RegLaunches.back().Name;
            }
        }
        const uint32_t slices = TreeSlicesFor(docCount);
        if (slices > 1) {
            evaluate += " x " + std::to_string(slices) + " slices of the trees + CombineSlicesKernel";
        }
    } else if (m.TileRows.Get() != nullptr) {
        evaluate = "EvalObliviousRowTileKernel";
    } else if (m.Oblivious && m.MaxDepth <= 8 && m.TileFits()) {
        evaluate = "EvalObliviousTileKernel";
    } else if (m.QuadRows.Get() != nullptr) {
        evaluate = "EvalObliviousQuadTileKernel";
    } else if (m.Oblivious && m.MaxDepth <= 8 && m.Dim == 1 && m.HalfTileLeaves.Get() != nullptr &&
               !m.TileFits() && HalfTileLdsBytes(m.LayoutBuckets, 8) <= kMaxTileLdsBytes) {
        evaluate = m.PairRows.Get() != nullptr ? "EvalObliviousPairTileKernel" : "EvalObliviousHalfTileKernel";
        if (m.TakesExchangeKernel(docCount)) {
            evaluate = m.ExchangeName;
        }
    } else if (m.DeepRows.Get() != nullptr) {
        evaluate = "EvalObliviousDeepTileKernel";
    } else if (m.Oblivious) {
        evaluate = "EvalObliviousKernel";
    } else if (m.NsLdsUsable) {
        evaluate = "EvalNonSymmetricLdsKernel<" + std::to_string(m.NsLdsShape.Waves) + ", " +
                   std::to_string(m.NsLdsShape.Entries) + (m.Dim > 1 ? ", " + std::to_string(NsLdsDims(m.Dim)) : "") + ">";
    } else if (m.NsTileUsable && TileLdsBytes(m.LayoutBuckets, m.Dim == 1 ? 1 : m.Dim <= 4 ? 4 : 16) <= kMaxTileLdsBytes) {
        evaluate = "EvalNonSymmetricTileKernel";
    } else {
        evaluate = "EvalNonSymmetricKernel";
    }
    return "binarize=" + binarize + ";evaluate=" + evaluate;
}

void THipEvaluator::LeafIndexesQuantizedDevice(const uint8_t* bins, size_t docCount, size_t treeStart, size_t treeEnd,
                                               uint32_t* indexes, void* stream) {
    TImpl& m = *Impl;
    CBAMD_ENSURE(treeStart <= treeEnd && treeEnd <= TreeCount, "tree range is out of bounds");
    if (docCount == 0 || treeStart == treeEnd) {
        return;
    }
    CBAMD_ENSURE(bins != nullptr && indexes != nullptr, "null pointer passed to leaf index calculation");
    hipStream_t s = m.Pick(stream);
    const size_t blocks = (docCount + 255) / 256;
    const auto tileLds = [&](int group) {
        return static_cast<size_t>(m.LayoutBuckets) * dev::kDocsPerBlock + static_cast<size_t>(dev::kDocsPerBlock) * dev::LeafIndexPitch(group) * 4;
    };
    if (m.Oblivious && m.MaxDepth <= 8 && m.PackedTrees.Get() != nullptr &&
        tileLds(dev::kLeafIndexSmallGroup) <= kMaxTileLdsBytes && docCount < (size_t(1) << 31)) {
        const auto launch = [&](auto kernel, int group) {
            // shares of the trees: enough workgroups for the chip's 256 CUs to go through them a few times over
            const size_t groups = (treeEnd - treeStart + group - 1) / group;
            const size_t wanted = std::max<size_t>(1, std::min<size_t>(groups, (kLeafIndexWorkgroups + blocks - 1) / blocks));
            const size_t shareGroups = (groups + wanted - 1) / wanted;
            const size_t shares = (groups + shareGroups - 1) / shareGroups;
            CBAMD_ENSURE(blocks * shares < (size_t(1) << 31), "batch is too large for one leaf index launch");
            EnsureDynamicLds(reinterpret_cast<const void*>(kernel), tileLds(group));
            hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(blocks * shares)), dim3(dev::kLeafIndexThreads), tileLds(group), s,
                               reinterpret_cast<const uint32_t*>(bins), static_cast<uint32_t>(docCount), m.LayoutBuckets,
                               m.PackedTrees.Get(), static_cast<uint32_t>(treeStart), static_cast<uint32_t>(treeEnd),
                               static_cast<uint32_t>(shares), static_cast<uint32_t>(shareGroups * group), indexes);
        };
        const auto launchGroup = [&](auto group) {
            constexpr int G = decltype(group)::value;
            const auto launchStores = [&](auto stream) {
                constexpr bool STREAM = decltype(stream)::value;
                if (m.PackedSevenBit && m.MaxDepth <= 6) {
                    launch(dev::LeafIndexesTileKernel<true, 6, G, STREAM>, G);
                } else if (m.PackedSevenBit) {
                    launch(dev::LeafIndexesTileKernel<true, 8, G, STREAM>, G);
                } else {
                    launch(dev::LeafIndexesTileKernel<false, 8, G, STREAM>, G);
                }
            };
            if (docCount * (treeEnd - treeStart) * sizeof(uint32_t) > kMemorySideCacheBytes) {
                launchStores(std::true_type());
            } else {
                launchStores(std::false_type());
            }
        };
        if (tileLds(dev::kLeafIndexGroup) <= kMaxTileLdsBytes) {
            launchGroup(std::integral_constant<int, dev::kLeafIndexGroup>());
        } else {
            launchGroup(std::integral_constant<int, dev::kLeafIndexSmallGroup>());
        }
        HIP_CHECK(hipGetLastError());
        return;
    }
    hipLaunchKernelGGL(dev::LeafIndexesKernel, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, s, bins, docCount,
                       m.LayoutBuckets, m.TreeTables(), m.Oblivious ? 1 : 0, static_cast<uint32_t>(treeStart),
                       static_cast<uint32_t>(treeEnd), indexes);
    HIP_CHECK(hipGetLastError());
}

void THipEvaluator::ExportQuantizedDevice(const uint8_t* bins, size_t docCount, uint8_t* referenceLayout, void* stream) {
    TImpl& m = *Impl;
    if (docCount == 0 || m.RealBucketCount == 0) {
        return;
    }
    hipStream_t s = m.Pick(stream);
    hipLaunchKernelGGL(dev::ExportBinsKernel, dim3(static_cast<uint32_t>((docCount + 255) / 256)), dim3(256), 0, s, bins,
                       docCount, m.LayoutBuckets, referenceLayout);
    HIP_CHECK(hipGetLastError());
}

void THipEvaluator::ApplyPredictionTypeDevice(int predictionType, size_t firstDoc, size_t totalDocs, size_t docCount,
                                              const double* raw, double* result, void* stream) {
    TImpl& m = *Impl;
    const uint32_t dim = static_cast<uint32_t>(m.Dim);
    CBAMD_ENSURE(predictionType >= dev::kPredRaw && predictionType <= dev::kPredMultiProbability, "unknown prediction type");
    // one dimension: the types TEvalResultProcessor accepts (eval_processing.h:182-204)
    CBAMD_ENSURE(dim > 1 || predictionType == dev::kPredRaw || predictionType == dev::kPredExponent ||
                     predictionType == dev::kPredProbability || predictionType == dev::kPredClass,
                 "unsupported prediction type");
    CBAMD_ENSURE(firstDoc <= totalDocs && docCount <= totalDocs - firstDoc, "document range exceeds the batch");
    CBAMD_ENSURE(firstDoc % 128 == 0, "a chunk must start at a multiple of 128 documents");
    if (docCount == 0) {
        return;
    }
    CBAMD_ENSURE(raw != nullptr && result != nullptr, "prediction buffers are null");
    CBAMD_ENSURE(!(predictionType == dev::kPredClass && dim > 1 && raw == result),
                 "Class of a multi-dimensional model cannot be computed in place");
    HIP_CHECK(hipSetDevice(m.DeviceId));
    hipStream_t s = m.Pick(stream);
    const TFastExpConstants constants = FastExpConstants();
    dev::TFastExpDev c;
    c.Mantissa = m.ExpMantissa.Get();
    c.Scale = constants.Scale;
    c.InvScale = constants.InvScale;
    const auto gridOf = [&](size_t threads) {
        const size_t groups = (docCount + threads - 1) / threads;
        CBAMD_ENSURE(groups <= 0x7fffffffu, "too many documents in one batch");
        return dim3(static_cast<uint32_t>(groups));
    };
    const auto softmax = [&](auto kernel) { hipLaunchKernelGGL(kernel, gridOf(256), dim3(256), 0, s, docCount, c, raw, result); };
    const bool isSoftmax = predictionType == dev::kPredProbability && dim > 1;
    if (isSoftmax && dim <= 8) {
        switch (dim) {
            case 2: softmax(dev::SoftmaxKernel<2>); break;
            case 3: softmax(dev::SoftmaxKernel<3>); break;
            case 4: softmax(dev::SoftmaxKernel<4>); break;
            case 5: softmax(dev::SoftmaxKernel<5>); break;
            case 6: softmax(dev::SoftmaxKernel<6>); break;
            case 7: softmax(dev::SoftmaxKernel<7>); break;
            default: softmax(dev::SoftmaxKernel<8>); break;
        }
    } else if (isSoftmax || (predictionType == dev::kPredClass && dim >= dev::kManyDimsClass) ||
               (predictionType == dev::kPredMultiProbability && dim >= dev::kManyDimsMultiProbability)) {
        hipLaunchKernelGGL(dev::ApplyPredictionTypeManyKernel, gridOf(64), dim3(64), 0, s, predictionType, dim, firstDoc,
                           totalDocs, docCount, c, raw, result);
    } else {
        hipLaunchKernelGGL(dev::ApplyPredictionTypeKernel, gridOf(256), dim3(256), 0, s, predictionType, dim, firstDoc, totalDocs,
                           docCount, c, raw, result);
    }
    HIP_CHECK(hipGetLastError());
}

void THipEvaluator::CalcDevice(const TFeatureBatch& batch, size_t docCount, size_t treeStart, size_t treeEnd,
                               double* results, void* stream) {
    TImpl& m = *Impl;
    HIP_CHECK(hipSetDevice(m.DeviceId));
    TImpl::TContextLease ctx(m);
    hipStream_t s = stream ? static_cast<hipStream_t>(stream) : m.Stream;
    if (TakesSmallBatchOnDevice(docCount, treeStart, treeEnd)) {
        CheckBatch(batch, docCount);
        LaunchSmallBatch(m, *ctx, batch, docCount, results, s, ctx->Ev[2]);
        HIP_CHECK(hipEventSynchronize(ctx->Ev[2]));
        SetLastSmallTimes(&*ctx);
        return;
    }
    TKernelTimes times;
    TStageEnd binarizeEnd{ctx->Ev[1]}, evalEnd{ctx->Ev[2]};
    HIP_CHECK(hipEventRecord(ctx->Ev[0], s));
    if (EvalFusedDevice(batch, docCount, treeStart, treeEnd, results, s, false, &evalEnd)) {
        // one launch does both: its whole duration is reported as the evaluate time
        evalEnd.Close(s);
        HIP_CHECK(hipEventSynchronize(ctx->Ev[2]));
        HIP_CHECK(hipEventElapsedTime(&times.EvalMs, ctx->Ev[0], ctx->Ev[2]));
    } else {
        ctx->ScratchBins.Reserve(QuantizedBytes(docCount));
        const bool sliced = treeStart == 0 && treeEnd == TreeCount && TreeSlicesFor(docCount) > 1;
        if (sliced) {
            ctx->SlicePartials.Reserve(TreeSliceScratchDoubles(docCount));
        }
        QuantizeDevice(batch, docCount, ctx->ScratchBins.Get(), s, &binarizeEnd);
        binarizeEnd.Close(s);
        if (sliced) {
            EvalQuantizedSlicedDevice(ctx->ScratchBins.Get(), docCount, results, ctx->SlicePartials.Get(), s, &evalEnd);
        } else {
            EvalQuantizedDevice(ctx->ScratchBins.Get(), docCount, treeStart, treeEnd, results, s, &evalEnd);
        }
        evalEnd.Close(s);
        HIP_CHECK(hipEventSynchronize(ctx->Ev[2]));
        HIP_CHECK(hipEventElapsedTime(&times.BinarizeMs, ctx->Ev[0], ctx->Ev[1]));
        HIP_CHECK(hipEventElapsedTime(&times.EvalMs, ctx->Ev[1], ctx->Ev[2]));
    }
    SetLastTimes(times);
}

void THipEvaluator::SetSmallBatchSlicing(bool on) {
    Impl->SmallBatchSlices = on;
}

bool THipEvaluator::SmallBatchSlicing() const {
    return Impl->SmallBatchSlices;
}

void THipEvaluator::CalcDeviceNoAlloc(const TFeatureBatch& batch, size_t docCount, size_t treeStart, size_t treeEnd,
                                      double* results, void* stream) {
    TImpl& m = *Impl;
    const size_t maxDocs = kNoAllocScratchBytes / (static_cast<size_t>(m.LayoutBuckets) * dev::kDocsPerBlock) * dev::kDocsPerBlock;
    // the fused kernel keeps the bins in registers: no buffer at all. A batch whose bins do not fit the fixed
    // buffer takes it whatever its size (below the size from which it is the faster as well),
    // and so does one that CalcDevice would cut into slices, which this call has no memory for
    const bool anyBatchSize = docCount > maxDocs || (docCount >= m.FusedMinDocs() && TreeSlicesFor(docCount) > 1);
    if (EvalFusedDevice(batch, docCount, treeStart, treeEnd, results, stream, anyBatchSize)) {
        return;
    }
    CBAMD_ENSURE(docCount <= maxDocs, "batch of " + std::to_string(docCount) + " documents exceeds the fixed bin buffer: at most " +
                                          std::to_string(maxDocs) + " documents per call for this model");
    // every (block, bucket) cell that the evaluate kernels read is written by the binarize kernels of
    // the same call, so nothing of the previous call's contents has to be cleared
    QuantizeDevice(batch, docCount, m.NoAllocScratch, stream);
    EvalQuantizedDevice(m.NoAllocScratch, docCount, treeStart, treeEnd, results, stream);
}

// ---------------------------------------------------------------------------- host staging ----

namespace {

// documents per slot of the staging pipeline: small enough that gathering the next slot on the host
// overlaps the transfer and the kernels of the current one
size_t PipelineDocs(size_t bytesPerDoc) {
    size_t docs = (size_t(64) << 20) / std::max<size_t>(1, bytesPerDoc);
    docs = std::max<size_t>(docs, 4096);
    docs = std::min<size_t>(docs, size_t(1) << 20);
    return docs / dev::kDocsPerBlock * dev::kDocsPerBlock;
}

// Runs `work(begin, end)` over [0, count) on a few threads when the bytes to move make it worthwhile.
template <typename TWork>
void ParallelCopy(size_t count, size_t bytes, const TWork& work) {
    size_t threads = std::min<size_t>(std::max(1u, std::thread::hardware_concurrency()), 16);
    threads = std::min(threads, bytes / (size_t(4) << 20) + 1);
    threads = std::min(threads, std::max<size_t>(count, 1));
    if (threads <= 1) {
        work(size_t(0), count);
        return;
    }
    std::vector<std::thread> pool;
    const size_t per = (count + threads - 1) / threads;
    for (size_t t = 1; t < threads; ++t) {
        pool.emplace_back(work, std::min(count, t * per), std::min(count, (t + 1) * per));
    }
    work(size_t(0), std::min(count, per));
    for (auto& th : pool) {
        th.join();
    }
}

// Fills pinned memory with `count` items of `itemBytes` (rows or columns given by pointer; fill(begin, end)) by a few threads
// and sends it off piece by piece, send(begin, end) from the calling thread as soon as a piece is filled: the bus, which
// bounds these calls, then starts with the first piece instead of behind the last one. The threads take units in order,
// so the pieces get ready one after the other. An eighth of the whole is a piece, 2 to 8 MB (a large batch: 4.05 ms with
// 2 MB, 3.75 with 4, 3.61 with 8; 16 MB: 532, 532 and 564 us). Whole call, one stream and a copy behind the last row -> this:
// 200 000 rows of 200 features 4.41 -> 3.69 ms (57 GB/s on the bus would be 2.8), 60 000 1.82 -> 1.32, 20 000 0.63 -> 0.54.
constexpr size_t kSendUnitBytes = size_t(256) << 10, kSendMinPieceBytes = size_t(2) << 20, kSendMaxPieceBytes = size_t(8) << 20;

template <typename TFill, typename TSend>
void FillAndSend(size_t count, size_t itemBytes, const TFill& fill, const TSend& send) {
    if (count == 0 || itemBytes == 0) {
        return;
    }
    const size_t perUnit = std::max<size_t>(1, kSendUnitBytes / itemBytes), units = (count + perUnit - 1) / perUnit;
    const size_t pieceBytes = std::min(kSendMaxPieceBytes, std::max(kSendMinPieceBytes, count * itemBytes / 8));
    const size_t unitsPerPiece = std::max<size_t>(1, pieceBytes / (perUnit * itemBytes));
    const size_t pieces = (units + unitsPerPiece - 1) / unitsPerPiece;
    std::atomic<size_t> next{0};
    std::vector<std::atomic<size_t>> filled(pieces);  // units of a piece (value-initialized to zero)
    const auto fillNext = [&] {
        const size_t unit = next.fetch_add(1, std::memory_order_relaxed);
        if (unit >= units) {
            return false;
        }
        fill(unit * perUnit, std::min(count, (unit + 1) * perUnit));
        filled[unit / unitsPerPiece].fetch_add(1, std::memory_order_release);
        return true;
    };
    // the threads are started by one of them: that takes as long as a piece or two take on the bus
    const size_t threads = std::min({static_cast<size_t>(std::max(1u, std::thread::hardware_concurrency())), size_t(16), units,
                                     count * itemBytes / (size_t(2) << 20) + 1});
    std::thread first;
    const auto join = [&] {
        next.store(units, std::memory_order_relaxed);  // (only an exception leaves units behind)
        if (first.joinable()) {
            first.join();
        }
    };
    try {
        if (threads > 1) {
            const auto helper = [&] {
                std::vector<std::thread> pool;
                try {
                    pool.reserve(threads);
                    for (size_t t = 2; t < threads && next.load(std::memory_order_relaxed) < units; ++t) {
                        pool.emplace_back([&] {
                            while (fillNext()) {
                            }
                        });
                    }
                } catch (const std::exception&) {
                    // fewer threads then
                }
                while (fillNext()) {
                }
                for (auto& th : pool) {
                    th.join();
                }
            };
            try {
                first = std::thread(helper);
            } catch (const std::system_error&) {
                // the calling thread alone
            }
        }
        bool left = true;
        for (size_t piece = 0; piece < pieces;) {
            const size_t last = std::min(units, (piece + 1) * unitsPerPiece);
            if (filled[piece].load(std::memory_order_acquire) == last - piece * unitsPerPiece) {
                send(piece * unitsPerPiece * perUnit, std::min(count, last * perUnit));
                ++piece;
            } else if (left) {
                left = fillNext();
            } else {
                std::this_thread::yield();
            }
        }
    } catch (...) {
        join();
        throw;
    }
    join();
}

// Rows given by pointer, dense into pinned memory and from there to the device.
template <typename T>
void SendRows(const T* const* rows, size_t count, size_t rowLen, T* pinned, T* device, hipStream_t s) {
    FillAndSend(
        count, rowLen * sizeof(T),
        [=](size_t begin, size_t end) {
            for (size_t d = begin; d < end; ++d) {
                std::memcpy(pinned + d * rowLen, rows[d], rowLen * sizeof(T));
            }
        },
        [=](size_t begin, size_t end) {
            HIP_CHECK(hipMemcpyAsync(device + begin * rowLen, pinned + begin * rowLen, (end - begin) * rowLen * sizeof(T),
                                     hipMemcpyHostToDevice, s));
        });
}

// Copies `count` rows of `rowLen` elements each, given by pointer, into a dense matrix (the copy is
// what bounds the pointer-per-row entry points).
template <typename T>
void GatherRows(const T* const* rows, size_t count, size_t rowLen, T* dst) {
    ParallelCopy(count, count * rowLen * sizeof(T), [=](size_t begin, size_t end) {
        for (size_t d = begin; d < end; ++d) {
            std::memcpy(dst + d * rowLen, rows[d], rowLen * sizeof(T));
        }
    });
}

// documents [begin, begin + n) of columns [first, last), each given by pointer (null: zeros), into [column][n]
void CopyColumns(const float* const* columns, size_t begin, size_t n, size_t first, size_t last, float* dst) {
    for (size_t f = first; f < last; ++f) {
        if (columns[f] != nullptr) {
            std::memcpy(dst + f * n, columns[f] + begin, n * sizeof(float));
        } else {
            std::memset(dst + f * n, 0, n * sizeof(float));
        }
    }
}

// A model without trees answers with its bias whatever the prediction type: the reference fills the result
// array with the bias values in turn and returns before any post-processing (cpu/formula_evaluator.cpp:29-41).
void FillBiasOnly(const std::vector<double>& bias, size_t count, double* results) {
    for (size_t i = 0; i < count; ++i) {
        results[i] = bias.empty() ? 0.0 : bias[i % bias.size()];
    }
}

// The two-slot pipeline of the host entry points: documents go in chunks; while the GPU copies in, runs and
// copies out the chunk of one slot, the host fills and sends the other slot. stage(slot, begin, n) fills the slot's
// pinned memory and enqueues everything up to the event Ev[3] of the slot; collect(slot, begin, n) runs once
// that event has passed.
template <typename TStage, typename TCollect>
void RunPipeline(size_t docCount, size_t chunk, THipEvaluator::TImpl::THostContext& ctx, const TStage& stage, const TCollect& collect) {
    const hipEvent_t done[2] = {ctx.Slots[0].Ev[3], ctx.Slots[1].Ev[3]};
    size_t pendingBegin[2] = {0, 0}, pendingDocs[2] = {0, 0};
    size_t index = 0;
    const auto finish = [&](int slot) {
        if (pendingDocs[slot]) {
            HIP_CHECK(hipEventSynchronize(done[slot]));
            collect(slot, pendingBegin[slot], pendingDocs[slot]);
            pendingDocs[slot] = 0;
        }
    };
    try {
        for (size_t begin = 0; begin < docCount; begin += chunk, ++index) {
            const int slot = static_cast<int>(index & 1);
            const size_t n = std::min(chunk, docCount - begin);
            finish(slot);  // the slot's previous chunk must be out before its buffers are reused
            stage(slot, begin, n);
            pendingBegin[slot] = begin;
            pendingDocs[slot] = n;
        }
        // the (up to) two chunks still in flight, older first
        finish(static_cast<int>(index & 1));
        finish(static_cast<int>((index + 1) & 1));
    } catch (...) {
        // the context goes back to the pool: nothing of this call may touch its buffers any more
        for (hipStream_t s : {ctx.CopyStream, ctx.Stream}) {
            if (s) {
                (void)hipStreamSynchronize(s);
            }
        }
        throw;
    }
}

}  // namespace

void THipEvaluator::SetLastTimes(const TKernelTimes& times) {
    std::lock_guard<std::mutex> guard(TimesLock);
    LastTimes = times;
    Impl->LastSmallStamps.reset();
}

void THipEvaluator::SetLastSmallTimes(void* smallContext) {
    std::lock_guard<std::mutex> guard(TimesLock);
    Impl->LastSmallStamps = static_cast<TImpl::THostContext*>(smallContext)->RunningStamps;
}

TKernelTimes THipEvaluator::LastKernelTimes() const {
    TImpl& m = *Impl;
    std::shared_ptr<const TImpl::TSmallStamps> last;
    {
        std::lock_guard<std::mutex> guard(TimesLock);
        if (!m.LastSmallStamps) {
            return LastTimes;
        }
        last = m.LastSmallStamps;
    }
    // A small-batch launch left its workgroups' clock stamps on the device. They are fetched when somebody asks, on a stream
    // that nothing else uses, while calls go on and publish theirs.
    TDeviceGuard device(m.DeviceId);
    TCaptureGuard capture;
    std::vector<unsigned long long> stamps(2 * last->Count);
    int clockKhz = 0;
    HIP_CHECK(hipDeviceGetAttribute(&clockKhz, hipDeviceAttributeWallClockRate, m.DeviceId));
    {
        std::lock_guard<std::mutex> guard(m.TimesStreamLock);
        if (m.TimesStream == nullptr) {
            HIP_CHECK(hipStreamCreateWithFlags(&m.TimesStream, hipStreamNonBlocking));
        }
        HIP_CHECK(hipMemcpyAsync(stamps.data(), last->Values.Get(), stamps.size() * sizeof(stamps[0]), hipMemcpyDeviceToHost,
                                 m.TimesStream));
        HIP_CHECK(hipStreamSynchronize(m.TimesStream));
    }
    unsigned long long begin = ~0ull, end = 0;
    for (size_t i = 0; i + 1 < stamps.size(); i += 2) {
        begin = std::min(begin, stamps[i]);
        end = std::max(end, stamps[i + 1]);
    }
    TKernelTimes times;
    times.EvalMs = end > begin && clockKhz > 0 ? static_cast<float>(end - begin) / static_cast<float>(clockKhz) : 0.f;
    return times;
}

// Stages one chunk of rows given by pointer (the reference API's float** / hashed int**) and returns the
// batch that describes it on the device.
static TFeatureBatch StageRowChunk(THipEvaluator::TImpl::THostSlot& slot, hipStream_t s, const float* const* rows,
                                   const int32_t* const* catRows, size_t begin, size_t n, size_t needFloats,
                                   size_t needCats, bool flat) {
    if (needFloats) {
        SendRows(rows + begin, n, needFloats, slot.PinnedFloats.Get(), slot.StageFloats.Get(), s);
    }
    if (needCats) {
        SendRows(catRows + begin, n, needCats, slot.PinnedCats.Get(), slot.StageCats.Get(), s);
    }
    TFeatureBatch batch;
    batch.Layout = flat ? TFeatureBatch::FlatRows : TFeatureBatch::SplitRows;
    batch.Floats = slot.StageFloats.Get();
    batch.Stride = needFloats;
    batch.Cats = needCats ? slot.StageCats.Get() : nullptr;
    batch.CatStride = needCats;
    return batch;
}

// What the prediction entry points share once a chunk's features are on the device: binarize, evaluate,
// prediction type, copy back; the slot's events bracket the kernels.
static void RunPredictionChunk(THipEvaluator& ev, THipEvaluator::TImpl::THostContext& ctx, int slotIndex,
                               const TFeatureBatch& batch, size_t begin, size_t n, size_t docCount, size_t stageDocs,
                               size_t treeStart, size_t treeEnd, int predictionType) {
    THipEvaluator::TImpl::THostSlot& slot = ctx.Slots[slotIndex];
    hipStream_t s = ctx.Stream;
    const size_t dim = static_cast<size_t>(ev.GetApproxDimension());
    const size_t outDim = predictionType == dev::kPredClass ? 1 : dim;
    THipEvaluator::TStageEnd binarizeEnd{slot.Ev[1]}, evalEnd{slot.Ev[2]};
    HIP_CHECK(hipEventRecord(slot.Ev[0], s));
    if (ev.FusedLayoutFor(batch.Layout, batch.Stride, n, treeStart, treeEnd, false) >= 0) {
        // one launch does both: its whole duration is reported as the evaluate time, as CalcDevice does
        binarizeEnd.Close(s);
        ev.EvalFusedDevice(batch, n, treeStart, treeEnd, slot.StageResults.Get(), s, false, &evalEnd);
    } else {
        ev.QuantizeDevice(batch, n, ctx.ScratchBins.Get(), s, &binarizeEnd);
        binarizeEnd.Close(s);
        if (treeStart == 0 && treeEnd == ev.GetTreeCount() && ev.TreeSlicesFor(n) > 1) {
            ctx.SlicePartials.Reserve(ev.TreeSliceScratchDoubles(n));
            ev.EvalQuantizedSlicedDevice(ctx.ScratchBins.Get(), n, slot.StageResults.Get(), ctx.SlicePartials.Get(), s, &evalEnd);
        } else {
            ev.EvalQuantizedDevice(ctx.ScratchBins.Get(), n, treeStart, treeEnd, slot.StageResults.Get(), s, &evalEnd);
        }
    }
    evalEnd.Close(s);
    const double* final = slot.StageResults.Get();
    if (predictionType != dev::kPredRaw) {
        // raw values, and behind them room for a prediction type that cannot be computed in place
        double* processed = slot.StageResults.Get() + (outDim == dim ? 0 : stageDocs * dim);
        ev.ApplyPredictionTypeDevice(predictionType, begin, docCount, n, slot.StageResults.Get(), processed, s);
        final = processed;
    }
    HIP_CHECK(hipMemcpyAsync(slot.PinnedResults.Get(), final, n * outDim * sizeof(double), hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipEventRecord(slot.Ev[3], s));
}

// Whether the features of a small host batch go to device memory before the launch, instead of being read from pinned memory
// by the kernel. Rows: the kernel reads them once per pass over the dimensions, so a copy (some 20 us) pays when the
// passes behind the first would move much. Columns: one document's values, or sixteen documents' of a column, are a request
// over PCIe each, so it pays soon. Whole call, 100 columns, read by the kernel and copied: rows, one dimension, 5000
// documents 98 and 117 us; ten dimensions (three passes), 2048 documents 66 and 82, 5000 195 and 157. Columns, 128 documents
// 30 and 37, 512 61 and 45; 1024 (SmallBatchKernel) 50 and 56, 5000 162 and 112; 600 columns, 512 documents 265 and 83.
static bool CopiesSmallHostBatch(const THipEvaluator::TImpl& m, bool columns, size_t docCount) {
    const size_t values = docCount * m.SmallCellCount;
    if (columns) {
        return values > (m.TakesFewDocumentsKernel(docCount) ? size_t(24) << 10 : size_t(144) << 10);
    }
    return values * (m.SmallPasses() - 1) * 4 > (size_t(5) << 19);
}

// A small batch whose features (`floatCount` and `catCount` values) are in the context's pinned memory; the results come to
// pinned memory, too.
static void CalcSmallHostBatch(THipEvaluator& ev, THipEvaluator::TImpl& m, THipEvaluator::TImpl::THostContext& ctx,
                               TFeatureBatch batch, size_t floatCount, size_t catCount, size_t docCount, int predictionType,
                               double* results) {
    THipEvaluator::TImpl::THostSlot& slot = ctx.Slots[0];
    if (CopiesSmallHostBatch(m, batch.Layout == TFeatureBatch::FlatColumns, docCount)) {
        const auto toDevice = [&](auto& stage, auto& pinned, size_t count) {
            stage.Reserve(std::max<size_t>(1, count));
            if (count) {
                HIP_CHECK(hipMemcpyAsync(stage.Get(), pinned.Get(), count * 4, hipMemcpyHostToDevice, ctx.Stream));
            }
        };
        toDevice(slot.StageFloats, slot.PinnedFloats, floatCount);
        batch.Floats = slot.StageFloats.Get();
        if (batch.Cats != nullptr) {
            toDevice(slot.StageCats, slot.PinnedCats, catCount);
            batch.Cats = slot.StageCats.Get();
        }
    }
    const size_t dim = static_cast<size_t>(m.Dim);
    const size_t outDim = predictionType == dev::kPredClass ? 1 : dim;
    const bool raw = predictionType == dev::kPredRaw;
    if (raw && m.TakesFewDocumentsKernel(docCount) && docCount * m.SmallPasses() <= kFlaggedGroups) {
        if (slot.SmallMemory.Reserve(kFlaggedGroups * sizeof(uint32_t) / sizeof(double) + docCount * dim)) {
            std::memset(slot.SmallFlags(), 0, kFlaggedGroups * sizeof(uint32_t));
            slot.SmallTicket = m.FlagTicket;
        }
        LaunchSmallBatch(m, ctx, batch, docCount, slot.SmallResults(), ctx.Stream, slot.Ev[3], &slot);
        AwaitSmallBatch(m, slot, slot.Ev[3]);
        std::memcpy(results, slot.SmallResults(), docCount * dim * sizeof(double));
    } else if (raw) {
        slot.PinnedResults.Reserve(docCount * dim);
        LaunchSmallBatch(m, ctx, batch, docCount, slot.PinnedResults.Get(), ctx.Stream, slot.Ev[3]);
        HIP_CHECK(hipEventSynchronize(slot.Ev[3]));
        std::memcpy(results, slot.PinnedResults.Get(), docCount * dim * sizeof(double));
    } else {
        slot.PinnedResults.Reserve(docCount * dim);
        slot.StageResults.Reserve(docCount * dim);
        LaunchSmallBatch(m, ctx, batch, docCount, slot.StageResults.Get(), ctx.Stream, slot.Ev[3]);
        ev.ApplyPredictionTypeDevice(predictionType, 0, docCount, docCount, slot.StageResults.Get(), slot.PinnedResults.Get(), ctx.Stream);
        HIP_CHECK(hipStreamSynchronize(ctx.Stream));
        std::memcpy(results, slot.PinnedResults.Get(), docCount * outDim * sizeof(double));
    }
}

void THipEvaluator::CalcHostRows(const float* const* rows, size_t rowLen, bool flat, const int32_t* const* catRows,
                                 size_t catRowLen, size_t docCount, size_t treeStart, size_t treeEnd, double* results,
                                 int predictionType) {
    TImpl& m = *Impl;
    const size_t outDim = predictionType == dev::kPredClass ? 1 : static_cast<size_t>(m.Dim);
    // only the columns the model can address are staged
    const size_t needFloats = flat ? m.FlatVectorSize : m.MinFloatSize;
    const size_t needCats = (!flat && m.HasCats) ? m.MinCatSize : 0;
    CBAMD_ENSURE(needFloats == 0 || rows != nullptr, "Model has float features but no float features provided");
    CBAMD_ENSURE(rowLen >= needFloats, (flat ? "insufficient flat features vector size: " : "insufficient float features vector size: ") +
                                           std::to_string(rowLen) + " expected: " + std::to_string(needFloats));
    CBAMD_ENSURE(needCats == 0 || catRows != nullptr, "Model has categorical features but no categorical features provided");
    CBAMD_ENSURE(catRowLen >= needCats, "insufficient cat features vector size: " + std::to_string(catRowLen) +
                                            " expected: " + std::to_string(needCats));
    if (TreeCount == 0) {
        FillBiasOnly(m.HostBias, docCount * outDim, results);
        return;
    }
    HIP_CHECK(hipSetDevice(m.DeviceId));
    TImpl::TContextLease ctx(m);
    if (TakesSmallBatchKernel(docCount, treeStart, treeEnd) && docCount * (needFloats + needCats) * 4 <= kSmallHostBytes) {
        TImpl::THostSlot& slot = ctx->Slots[0];
        slot.PinnedFloats.Reserve(std::max<size_t>(1, docCount * needFloats));
        if (needFloats) {  // a model of categorical features may come without float rows
            GatherRows(rows, docCount, needFloats, slot.PinnedFloats.Get());
        }
        TFeatureBatch batch;
        batch.Layout = flat ? TFeatureBatch::FlatRows : TFeatureBatch::SplitRows;
        batch.Floats = slot.PinnedFloats.Get();
        batch.Stride = needFloats;
        if (needCats) {
            slot.PinnedCats.Reserve(docCount * needCats);
            GatherRows(catRows, docCount, needCats, slot.PinnedCats.Get());
            batch.Cats = slot.PinnedCats.Get();
            batch.CatStride = needCats;
        }
        CalcSmallHostBatch(*this, m, *ctx, batch, docCount * needFloats, docCount * needCats, docCount, predictionType, results);
        SetLastSmallTimes(&*ctx);
        return;
    }
    const size_t chunk = PipelineDocs((needFloats + needCats) * 4);
    const size_t stageDocs = std::min(chunk, docCount);
    for (int i = 0; i < (docCount > chunk ? 2 : 1); ++i) {
        TImpl::THostSlot& slot = ctx->Slots[i];
        slot.PinnedFloats.Reserve(std::max<size_t>(1, stageDocs * needFloats));
        slot.StageFloats.Reserve(std::max<size_t>(1, stageDocs * needFloats));
        if (needCats) {
            slot.PinnedCats.Reserve(stageDocs * needCats);
            slot.StageCats.Reserve(stageDocs * needCats);
        }
        slot.PinnedResults.Reserve(std::max<size_t>(1, stageDocs * m.Dim));
        slot.StageResults.Reserve(std::max<size_t>(1, stageDocs * (m.Dim + 1)));
    }
    ctx->ScratchBins.Reserve(QuantizedBytes(stageDocs));
    TKernelTimes times;
    const hipStream_t copies = ctx->CopiesOf(docCount > chunk);
    RunPipeline(
        docCount, chunk, *ctx,
        [&](int i, size_t begin, size_t n) {
            const TFeatureBatch batch = StageRowChunk(ctx->Slots[i], copies, rows, catRows, begin, n, needFloats, needCats, flat);
            ctx->AwaitCopies(i, copies);
            RunPredictionChunk(*this, *ctx, i, batch, begin, n, docCount, stageDocs, treeStart, treeEnd, predictionType);
        },
        [&](int i, size_t begin, size_t n) {
            TImpl::THostSlot& slot = ctx->Slots[i];
            std::memcpy(results + begin * outDim, slot.PinnedResults.Get(), n * outDim * sizeof(double));
            float a = 0.f, b = 0.f;
            HIP_CHECK(hipEventElapsedTime(&a, slot.Ev[0], slot.Ev[1]));
            HIP_CHECK(hipEventElapsedTime(&b, slot.Ev[1], slot.Ev[2]));
            times.BinarizeMs += a;
            times.EvalMs += b;
        });
    SetLastTimes(times);
}

// Columns by pointer (CalcModelPredictionFlatTransposed): a chunk is staged as a dense [feature][document]
// matrix, the columns copied by a few threads, and goes through the same two-slot pipeline.
void THipEvaluator::CalcHostColumns(const float* const* columns, size_t columnCount, size_t docCount, size_t treeStart,
                                    size_t treeEnd, double* results, int predictionType) {
    TImpl& m = *Impl;
    const size_t outDim = predictionType == dev::kPredClass ? 1 : static_cast<size_t>(m.Dim);
    const size_t need = m.FlatVectorSize;
    CBAMD_ENSURE(columnCount >= need, "Not enough features provided");
    CBAMD_ENSURE(need == 0 || columns != nullptr, "Not enough features provided");
    if (TreeCount == 0) {
        FillBiasOnly(m.HostBias, docCount * outDim, results);
        return;
    }
    HIP_CHECK(hipSetDevice(m.DeviceId));
    TImpl::TContextLease ctx(m);
    if (TakesSmallBatchKernel(docCount, treeStart, treeEnd) && docCount * need * 4 <= kSmallHostBytes) {
        TImpl::THostSlot& slot = ctx->Slots[0];
        slot.PinnedFloats.Reserve(std::max<size_t>(1, docCount * need));
        float* dst = slot.PinnedFloats.Get();
        ParallelCopy(need, need * docCount * sizeof(float),
                     [=](size_t first, size_t last) { CopyColumns(columns, 0, docCount, first, last, dst); });
        TFeatureBatch batch;
        batch.Layout = TFeatureBatch::FlatColumns;
        batch.Floats = slot.PinnedFloats.Get();
        batch.Stride = docCount;
        CalcSmallHostBatch(*this, m, *ctx, batch, docCount * need, 0, docCount, predictionType, results);
        SetLastSmallTimes(&*ctx);
        return;
    }
    const size_t chunk = PipelineDocs(need * 4);
    const size_t stageDocs = std::min(chunk, docCount);
    for (int i = 0; i < (docCount > chunk ? 2 : 1); ++i) {
        TImpl::THostSlot& slot = ctx->Slots[i];
        slot.PinnedFloats.Reserve(std::max<size_t>(1, stageDocs * need));
        slot.StageFloats.Reserve(std::max<size_t>(1, stageDocs * need));
        slot.PinnedResults.Reserve(std::max<size_t>(1, stageDocs * m.Dim));
        slot.StageResults.Reserve(std::max<size_t>(1, stageDocs * (m.Dim + 1)));
    }
    ctx->ScratchBins.Reserve(QuantizedBytes(stageDocs));
    TKernelTimes times;
    const hipStream_t copies = ctx->CopiesOf(docCount > chunk);
    RunPipeline(
        docCount, chunk, *ctx,
        [&](int i, size_t begin, size_t n) {
            TImpl::THostSlot& slot = ctx->Slots[i];
            float* dst = slot.PinnedFloats.Get();
            float* device = slot.StageFloats.Get();
            FillAndSend(
                need, n * sizeof(float), [=](size_t first, size_t last) { CopyColumns(columns, begin, n, first, last, dst); },
                [=](size_t first, size_t last) {
                    HIP_CHECK(hipMemcpyAsync(device + first * n, dst + first * n, (last - first) * n * sizeof(float),
                                             hipMemcpyHostToDevice, copies));
                });
            ctx->AwaitCopies(i, copies);
            TFeatureBatch batch;
            batch.Layout = TFeatureBatch::FlatColumns;
            batch.Floats = slot.StageFloats.Get();
            batch.Stride = n;
            RunPredictionChunk(*this, *ctx, i, batch, begin, n, docCount, stageDocs, treeStart, treeEnd, predictionType);
        },
        [&](int i, size_t begin, size_t n) {
            TImpl::THostSlot& slot = ctx->Slots[i];
            std::memcpy(results + begin * outDim, slot.PinnedResults.Get(), n * outDim * sizeof(double));
            float a = 0.f, b = 0.f;
            HIP_CHECK(hipEventElapsedTime(&a, slot.Ev[0], slot.Ev[1]));
            HIP_CHECK(hipEventElapsedTime(&b, slot.Ev[1], slot.Ev[2]));
            times.BinarizeMs += a;
            times.EvalMs += b;
        });
    SetLastTimes(times);
}

void THipEvaluator::LeafIndexesHostRows(const float* const* rows, size_t rowLen, bool flat,
                                        const int32_t* const* catRows, size_t catRowLen, size_t docCount,
                                        size_t treeStart, size_t treeEnd, uint32_t* indexes) {
    TImpl& m = *Impl;
    CBAMD_ENSURE(treeStart <= treeEnd && treeEnd <= TreeCount, "tree range is out of bounds");
    const size_t treeCount = treeEnd - treeStart;
    const size_t needFloats = flat ? m.FlatVectorSize : m.MinFloatSize;
    const size_t needCats = (!flat && m.HasCats) ? m.MinCatSize : 0;
    CBAMD_ENSURE(needFloats == 0 || rows != nullptr, "Model has float features but no float features provided");
    CBAMD_ENSURE(rowLen >= needFloats, "insufficient float features vector size: " + std::to_string(rowLen) +
                                           " expected: " + std::to_string(needFloats));
    CBAMD_ENSURE(needCats == 0 || catRows != nullptr, "Model has categorical features but no categorical features provided");
    CBAMD_ENSURE(catRowLen >= needCats, "insufficient cat features vector size");
    if (docCount == 0 || treeCount == 0) {
        return;
    }
    HIP_CHECK(hipSetDevice(m.DeviceId));
    TImpl::TContextLease ctx(m);
    const size_t chunk = PipelineDocs((needFloats + needCats + treeCount) * 4);
    const size_t stageDocs = std::min(chunk, docCount);
    for (int i = 0; i < (docCount > chunk ? 2 : 1); ++i) {
        TImpl::THostSlot& slot = ctx->Slots[i];
        slot.PinnedFloats.Reserve(std::max<size_t>(1, stageDocs * needFloats));
        slot.StageFloats.Reserve(std::max<size_t>(1, stageDocs * needFloats));
        if (needCats) {
            slot.PinnedCats.Reserve(stageDocs * needCats);
            slot.StageCats.Reserve(stageDocs * needCats);
        }
        slot.PinnedIndexes.Reserve(stageDocs * treeCount);
        slot.StageIndexes.Reserve(stageDocs * treeCount);
    }
    ctx->ScratchBins.Reserve(QuantizedBytes(stageDocs));
    RunPipeline(
        docCount, chunk, *ctx,
        [&](int i, size_t begin, size_t n) {
            TImpl::THostSlot& slot = ctx->Slots[i];
            hipStream_t s = ctx->Stream;
            const TFeatureBatch batch = StageRowChunk(slot, s, rows, catRows, begin, n, needFloats, needCats, flat);
            QuantizeDevice(batch, n, ctx->ScratchBins.Get(), s);
            LeafIndexesQuantizedDevice(ctx->ScratchBins.Get(), n, treeStart, treeEnd, slot.StageIndexes.Get(), s);
            HIP_CHECK(hipMemcpyAsync(slot.PinnedIndexes.Get(), slot.StageIndexes.Get(), n * treeCount * sizeof(uint32_t),
                                     hipMemcpyDeviceToHost, s));
            HIP_CHECK(hipEventRecord(slot.Ev[3], s));
        },
        [&](int i, size_t begin, size_t n) {
            // 4 bytes per document and tree: the copy out of the pinned buffer bounds this call, so it is shared out
            uint32_t* dst = indexes + begin * treeCount;
            const uint32_t* src = ctx->Slots[i].PinnedIndexes.Get();
            ParallelCopy(n, n * treeCount * sizeof(uint32_t), [=](size_t first, size_t last) {
                std::memcpy(dst + first * treeCount, src + first * treeCount, (last - first) * treeCount * sizeof(uint32_t));
            });
        });
}

void THipEvaluator::QuantizeHostRows(const float* const* rows, size_t rowLen, bool flat, const int32_t* const* catRows,
                                     size_t catRowLen, size_t docCount, uint8_t* referenceLayout) {
    TImpl& m = *Impl;
    const size_t needFloats = flat ? m.FlatVectorSize : m.MinFloatSize;
    const size_t needCats = (!flat && m.HasCats) ? m.MinCatSize : 0;
    CBAMD_ENSURE(needFloats == 0 || rows != nullptr, "Model has float features but no float features provided");
    CBAMD_ENSURE(rowLen >= needFloats, "insufficient float features vector size: " + std::to_string(rowLen) +
                                           " expected: " + std::to_string(needFloats));
    CBAMD_ENSURE(needCats == 0 || catRows != nullptr, "Model has categorical features but no categorical features provided");
    CBAMD_ENSURE(catRowLen >= needCats, "insufficient cat features vector size");
    if (docCount == 0 || m.RealBucketCount == 0) {
        return;
    }
    HIP_CHECK(hipSetDevice(m.DeviceId));
    TImpl::TContextLease ctx(m);
    // chunks end on a multiple of 256 documents, so that the reference's blocks of 128 do not straddle them
    const size_t chunk = PipelineDocs((needFloats + needCats) * 4 + m.RealBucketCount);
    const size_t stageDocs = std::min(chunk, docCount);
    for (int i = 0; i < (docCount > chunk ? 2 : 1); ++i) {
        TImpl::THostSlot& slot = ctx->Slots[i];
        slot.PinnedFloats.Reserve(std::max<size_t>(1, stageDocs * needFloats));
        slot.StageFloats.Reserve(std::max<size_t>(1, stageDocs * needFloats));
        if (needCats) {
            slot.PinnedCats.Reserve(stageDocs * needCats);
            slot.StageCats.Reserve(stageDocs * needCats);
        }
        slot.PinnedExport.Reserve(stageDocs * m.RealBucketCount);
        slot.StageExport.Reserve(stageDocs * m.RealBucketCount);
    }
    ctx->ScratchBins.Reserve(QuantizedBytes(stageDocs));
    RunPipeline(
        docCount, chunk, *ctx,
        [&](int i, size_t begin, size_t n) {
            TImpl::THostSlot& slot = ctx->Slots[i];
            hipStream_t s = ctx->Stream;
            const TFeatureBatch batch = StageRowChunk(slot, s, rows, catRows, begin, n, needFloats, needCats, flat);
            QuantizeDevice(batch, n, ctx->ScratchBins.Get(), s);
            ExportQuantizedDevice(ctx->ScratchBins.Get(), n, slot.StageExport.Get(), s);
            HIP_CHECK(hipMemcpyAsync(slot.PinnedExport.Get(), slot.StageExport.Get(), n * m.RealBucketCount,
                                     hipMemcpyDeviceToHost, s));
            HIP_CHECK(hipEventRecord(slot.Ev[3], s));
        },
        [&](int i, size_t begin, size_t n) {
            std::memcpy(referenceLayout + begin * m.RealBucketCount, ctx->Slots[i].PinnedExport.Get(), n * m.RealBucketCount);
        });
}

}  // namespace cbamd
