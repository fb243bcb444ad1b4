// Where the entries of a non-symmetric tree stand for EvalNonSymmetricLdsKernel: the seven nodes of the top three levels apart, then
// the eight exits that their results choose from, then pairs of children.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace cbamd {

constexpr uint32_t kNsNoItem = UINT32_MAX;
// Items of a tree up to which a leaf of several exits gets a place of its own, see TNsTreeLayout::Next
constexpr size_t kNsSmallTreeItems = 64;

struct TNsTreeLayout {
    uint32_t TopItems[7];         // by level, children of node n: 2 n + 1 and 2 n + 2; kNsNoItem where a branch ended earlier
    std::vector<uint32_t> Items;  // the item at each place; the exits are the places 0 to 7
    // The place that follows: of a node the place of its children's pair, of a leaf the one at which its documents stay. A leaf above the
    // third level is the item of two to eight exits; in a small tree all of them name one place behind the pairs, so that the leaf values of
    // a small tree's documents come from as few lines of memory as its leaves fill. (Each exit its own: 500 001 documents, 300 trees of
    // depth 2 over 100 features, values of three dimensions spread over 256 bytes instead of 128, 322 us a call, now 278.)
    std::vector<uint32_t> Next;
    uint32_t Steps = 0;           // from the exits to the farthest leaf
    std::vector<uint32_t> PlaceOfPair, StepsFrom;  // scratch, by item and by place
};

// left: per item (the root first) the left child's item, which the right child follows; kNsNoItem: a leaf. A layout is filled anew by every
// tree: models have thousands, and allocating five vectors for each takes longer than laying out a tree of one level.
inline void LayOutNsTree(const std::vector<uint32_t>& left, TNsTreeLayout* layout) {
    // the item that a path of `levels` decisions (the root's the highest bit) leads to, a leaf if it ends there earlier
    const auto follow = [&](uint32_t path, int levels) {
        uint32_t item = 0;
        for (int level = levels - 1; level >= 0 && left[item] != kNsNoItem; --level) {
            item = left[item] + (path >> level & 1);
        }
        return item;
    };
    for (uint32_t n = 0; n < 7; ++n) {
        const int level = n == 0 ? 0 : n < 3 ? 1 : 2;
        const uint32_t item = follow(n + 1 - (1u << level), level);
        layout->TopItems[n] = left[item] == kNsNoItem ? kNsNoItem : item;
    }
    // a pair has one place, whichever items name it (those that a one-hot split repeats name their original's)
    std::vector<uint32_t>&items = layout->Items, &next = layout->Next, &placeOfPair = layout->PlaceOfPair, &stepsFrom = layout->StepsFrom;
    items.clear();
    next.clear();
    for (uint32_t exit = 0; exit < 8; ++exit) {
        items.push_back(follow(exit, 3));
    }
    placeOfPair.assign(left.size(), 0);  // by the left child's item; 0: none yet
    bool repeats = false;
    for (uint32_t at = 0; at < items.size(); ++at) {
        const uint32_t child = left[items[at]];
        if (child == kNsNoItem) {
            next.push_back(at);
            continue;
        }
        if (placeOfPair[child] == 0) {
            placeOfPair[child] = static_cast<uint32_t>(items.size());
            items.push_back(child);
            items.push_back(child + 1);
        } else {
            repeats = true;
        }
        next.push_back(placeOfPair[child]);
    }
    // A pair stands behind the place that names it but for repeated ones, whose steps are found by following the names
    stepsFrom.assign(items.size(), repeats ? kNsNoItem : 0);
    const auto follows = [&](const auto& self, uint32_t at) -> uint32_t {
        if (stepsFrom[at] == kNsNoItem) {
            stepsFrom[at] = left[items[at]] == kNsNoItem ? 0 : 1 + std::max(self(self, next[at]), self(self, next[at] + 1));
        }
        return stepsFrom[at];
    };
    for (uint32_t at = static_cast<uint32_t>(items.size()); !repeats && at-- > 0;) {
        if (left[items[at]] != kNsNoItem) {
            stepsFrom[at] = 1 + std::max(stepsFrom[next[at]], stepsFrom[next[at] + 1]);
        }
    }
    layout->Steps = 0;
    for (uint32_t exit = 0; exit < 8; ++exit) {
        layout->Steps = std::max(layout->Steps, follows(follows, exit));
    }
    if (left.size() <= kNsSmallTreeItems) {
        for (uint32_t exit = 0; exit < 8; ++exit) {
            const uint32_t item = items[exit];
            const uint32_t first = static_cast<uint32_t>(std::find(items.begin(), items.begin() + exit, item) - items.begin());
            if (left[item] != kNsNoItem) {
                continue;
            }
            if (first < exit) {
                next[exit] = next[first];
            } else if (std::count(items.begin() + exit + 1, items.begin() + 8, item) > 0) {
                next[exit] = static_cast<uint32_t>(items.size());
                next.push_back(next[exit]);
                items.push_back(item);
            }
        }
    }
}

// A terminal entry at a place: it selects itself from its pair (even: splitIdx 255, odd: splitIdx 0), and names the row of its leaf's values
constexpr uint32_t NsTerminalEntry(uint32_t place) {
    return (place % 2 != 0 ? 0u : 255u) | ((place & ~1u) << 21);
}

// For a unit whose trees all end at their exits, so that nothing walks on from the places that these name: the eight exits of one of its trees
// name rows one behind the other, a row per leaf. `from`: the places whose values the unit's rows take, this tree's put behind the others'. The leaves of the unit's
// trees then fill as few lines as they can: 273 107 documents, 300 trees of one level and two dimensions, a tree's two rows 256 bytes from
// the next one's, 83.3 us a launch, now 81.4; of three levels and three dimensions 151.6 and now 147.3.
inline void CompactNsExits(uint32_t* exits, std::vector<uint32_t>* from) {
    const size_t tree = from->size();
    for (uint32_t exit = 0; exit < 8; ++exit) {
        const uint32_t place = (exits[exit] >> 21) + ((exits[exit] & 0xffu) == 0 ? 1u : 0u);
        const auto known = std::find(from->begin() + static_cast<std::ptrdiff_t>(tree), from->end(), place);
        exits[exit] = NsTerminalEntry(static_cast<uint32_t>(known - from->begin()));
        if (known == from->end()) {
            from->push_back(place);
        }
    }
}

// Rows of the leaf values of a slice of the dimensions. Of one dimension a region's zeros follow, which trees that a unit lacks or that the
// call's range leaves out read; of several such trees' rows are not read at all.
constexpr size_t NsSliceRows(size_t entries, uint32_t dims, uint32_t regionEntries) {
    return dims == 1 ? entries + regionEntries : entries;
}

}  // namespace cbamd
