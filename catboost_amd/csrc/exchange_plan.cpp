#include "exchange_plan.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <future>
#include <numeric>
#include <utility>

namespace cbamd {

namespace {

// A level of the model as an edge of the multigraph trees x groups
struct TEdge {
    uint32_t Tree = 0, Group = 0;
    const TExchangeLevel* Level = nullptr;
    float Lopsided = 0.0f;
    uint8_t ModelLevel = 0;  // which level of its tree
    bool High = false;       // one of the places behind the first five
    int8_t Place = -1;       // place in its group, later the order of the compares
};

// A tree's edges follow one another: all trees are in the order of their steps (At: place of a tree in that order)
struct TTreeEdges {
    std::vector<uint32_t> First;  // per place in the order, and the end
    std::vector<uint32_t> At;
    uint32_t Begin(uint32_t tree) const { return First[At[tree]]; }
    uint32_t End(uint32_t tree) const { return First[At[tree] + 1]; }
};

struct TGroup {
    std::vector<uint32_t> Edges;
    uint32_t FirstRound = ~0u, LastRound = 0;  // rounds whose trees look at it
    uint32_t Slot = 0;
};

// Gives the places behind the first kEvenPlaces to the levels that split the documents unevenly: the five low bits of a leaf index
// choose the pair of LDS banks of a gather, lanes with the same index share an access, and lopsided levels in the high bits
// leave fewer different leaves per bank (borders drawn evenly, 16 lanes a cycle: 12.0 cycles per gather of 64 lanes in the model's order,
// 8.5 so). A tree and a group have at most as many edges on either side as there are places; trees start within that,
// groups are brought there by swapping pairs of a tree's levels, the cheapest first.
constexpr uint32_t kEvenPlaces = 5;

class TSides {
public:
    TSides(std::vector<TEdge>* edges, const TTreeEdges& ofTree, const std::vector<TGroup>& groups, uint32_t places)
        : Edges(*edges), OfTree(ofTree), Groups(groups), Places{kEvenPlaces, places - kEvenPlaces}
        , TreeCount{std::vector<uint8_t>(ofTree.At.size(), 0), std::vector<uint8_t>(ofTree.At.size(), 0)}
        , GroupCount{std::vector<uint8_t>(groups.size(), 0), std::vector<uint8_t>(groups.size(), 0)}, Seen(groups.size(), 0) {
    }

    bool Assign() {
        for (uint32_t t = 0; t < OfTree.At.size(); ++t) {
            const uint32_t begin = OfTree.Begin(t), end = OfTree.End(t);
            for (uint32_t e = begin; e < end; ++e) {
                uint32_t before = 0;  // edges of the tree that come before this one, evenest first
                for (uint32_t o = begin; o < end; ++o) {
                    before += Edges[o].Lopsided < Edges[e].Lopsided || (o < e && Edges[o].Lopsided == Edges[e].Lopsided);
                }
                Edges[e].High = before >= kEvenPlaces;
                Count(e, 1);
            }
        }
        for (uint32_t g = 0; g < Groups.size(); ++g) {
            for (int side = 0; side < 2; ++side) {
                while (GroupCount[side][g] > Places[side]) {
                    if (!Relieve(g, side != 0)) {
                        return false;
                    }
                }
            }
        }
        return true;
    }

private:
    void Count(uint32_t e, int by) {
        TreeCount[Edges[e].High][Edges[e].Tree] += by;
        GroupCount[Edges[e].High][Edges[e].Group] += by;
    }
    void Flip(uint32_t e) {
        Count(e, -1);
        Edges[e].High = !Edges[e].High;
        Count(e, 1);
    }
    float Cost(uint32_t e) const {  // of moving the edge to the other side
        return Edges[e].High ? -Edges[e].Lopsided : Edges[e].Lopsided;
    }

    // One edge of `side` less in group g: along a shortest chain of swaps (an edge of the group leaves `side`, another
    // edge of its tree takes its place there, and so on) that ends at a tree or a group with room.
    bool Relieve(uint32_t g, bool side) {
        Steps.clear();
        At.assign(1, g);
        Via.assign(1, -1);
        Seen[g] = ++Search;
        while (!At.empty()) {
            float bestCost = 0.0f;
            int best = -1;
            Next.clear();
            NextVia.clear();
            for (size_t i = 0; i < At.size(); ++i) {
                for (uint32_t out : Groups[At[i]].Edges) {
                    if (Edges[out].High != side) {
                        continue;
                    }
                    const uint32_t t = Edges[out].Tree;
                    if (TreeCount[!side][t] < Places[!side]) {
                        Steps.push_back({out, ~0u, Via[i]});
                        if (best < 0 || Cost(out) < bestCost) {
                            best = static_cast<int>(Steps.size()) - 1;
                            bestCost = Cost(out);
                        }
                        continue;
                    }
                    for (uint32_t in = OfTree.Begin(t); in < OfTree.End(t); ++in) {
                        const uint32_t to = Edges[in].Group;
                        if (Edges[in].High == side || to == At[i]) {
                            continue;
                        }
                        if (GroupCount[side][to] < Places[side]) {
                            const float cost = Cost(out) + Cost(in);
                            Steps.push_back({out, in, Via[i]});
                            if (best < 0 || cost < bestCost) {
                                best = static_cast<int>(Steps.size()) - 1;
                                bestCost = cost;
                            }
                        } else if (Seen[to] != Search) {
                            Seen[to] = Search;
                            Steps.push_back({out, in, Via[i]});
                            Next.push_back(to);
                            NextVia.push_back(static_cast<int>(Steps.size()) - 1);
                        }
                    }
                }
            }
            if (best >= 0) {
                for (int s = best; s >= 0; s = Steps[s].Parent) {
                    Flip(Steps[s].Out);
                    if (Steps[s].In != ~0u) {
                        Flip(Steps[s].In);
                    }
                }
                return true;
            }
            At.swap(Next);
            Via.swap(NextVia);
        }
        return false;
    }

    struct TStep {
        uint32_t Out, In;  // edges that leave and enter the side
        int Parent;        // step before
    };
    std::vector<TStep> Steps;              // of Relieve
    std::vector<uint32_t> At, Next;        // groups of the frontier and of the next one
    std::vector<int> Via, NextVia;         // steps that led there
    std::vector<TEdge>& Edges;
    const TTreeEdges& OfTree;
    const std::vector<TGroup>& Groups;
    const uint32_t Places[2];
    std::vector<uint8_t> TreeCount[2], GroupCount[2];
    std::vector<uint32_t> Seen;            // per group the last search that had it on a frontier
    uint32_t Search = 0;
};

// Places base .. base + colours - 1 for the edges of one side: each edge takes a place that is free at its tree and at its group, after
// swapping two places along the alternating path that starts at the group when there is no such place.
void Colour(std::vector<TEdge>* edges, size_t treeCount, size_t groupCount, bool high, uint32_t colours, uint32_t base) {
    std::vector<uint32_t> slots((treeCount + groupCount) * colours);  // a colour's edge at a vertex, the trees' first
    std::vector<uint8_t> freeOf(treeCount + groupCount, static_cast<uint8_t>((1u << colours) - 1));
    std::vector<uint32_t> path;
    const auto take = [&](uint32_t e, uint32_t vertex, uint32_t colour) {
        slots[vertex * colours + colour] = e;
        freeOf[vertex] &= ~(1u << colour);
    };
    for (size_t i = 0; i < edges->size(); ++i) {
        TEdge& e = (*edges)[i];
        if (e.High != high) {
            continue;
        }
        const uint32_t tree = e.Tree, group = static_cast<uint32_t>(treeCount) + e.Group;
        uint32_t colour;
        if (const uint32_t both = freeOf[tree] & freeOf[group]; both != 0) {
            colour = __builtin_ctz(both);
        } else {
            // the path from the group along the colours atTree, atGroup, atTree ... never comes to the edge's tree
            const uint32_t atTree = __builtin_ctz(freeOf[tree]), atGroup = __builtin_ctz(freeOf[group]);
            path.clear();
            bool isTree = false;
            uint32_t vertex = group, along = atTree;
            while ((freeOf[vertex] >> along & 1) == 0) {
                path.push_back(slots[vertex * colours + along]);
                isTree = !isTree;
                vertex = isTree ? (*edges)[path.back()].Tree : static_cast<uint32_t>(treeCount) + (*edges)[path.back()].Group;
                along ^= atTree ^ atGroup;
            }
            for (uint32_t p : path) {
                const TEdge& on = (*edges)[p];
                const uint32_t bit = 1u << (on.Place - base);
                freeOf[on.Tree] |= bit;
                freeOf[treeCount + on.Group] |= bit;
            }
            for (uint32_t p : path) {
                TEdge& on = (*edges)[p];
                const uint32_t other = on.Place - base == atTree ? atGroup : atTree;
                on.Place = static_cast<int8_t>(base + other);
                take(p, on.Tree, other);
                take(p, static_cast<uint32_t>(treeCount) + on.Group, other);
            }
            colour = atTree;
        }
        e.Place = static_cast<int8_t>(base + colour);
        take(static_cast<uint32_t>(i), tree, colour);
        take(static_cast<uint32_t>(i), group, colour);
    }
}

}  // namespace

bool BuildExchangePlan(const std::vector<TExchangeTree>& trees, uint32_t bucketCount, uint32_t maxDepth, bool six,
                       const std::vector<uint32_t>& columnOf, TExchangePlan* plan) {
    const size_t treeCount = trees.size();
    // ---- buckets to waves: the busiest first, each to the wave that compares the least
    std::vector<uint32_t> levelsOf(bucketCount, 0);
    for (const TExchangeTree& t : trees) {
        for (const TExchangeLevel& l : t.Levels) {
            if (l.Bucket >= bucketCount) {
                return false;  // a damaged model
            }
            ++levelsOf[l.Bucket];
        }
    }
    std::vector<uint32_t> byLevels;
    for (uint32_t b = 0; b < bucketCount; ++b) {
        if (levelsOf[b] > 0) {
            byLevels.push_back(b);
        }
    }
    if (treeCount == 0 || byLevels.size() > size_t(kExchangeWaves) * kExchangeWaveBuckets) {
        return false;
    }
    std::stable_sort(byLevels.begin(), byLevels.end(), [&](uint32_t a, uint32_t b) { return levelsOf[a] > levelsOf[b]; });
    // (with tiles at most four of a tile's buckets to a wave: there are 64 of them at most)
    const bool tiled = !columnOf.empty();
    const uint32_t tileCount = tiled ? kExchangeTiles : 1, perTile = kExchangeWaveBuckets / tileCount;
    std::vector<uint32_t> waveOf(bucketCount, 0), registerOf(bucketCount, 0);
    std::vector<uint32_t> taken(kExchangeWaves * tileCount, 0);
    std::vector<size_t> load(kExchangeWaves, 0);
    plan->WaveTable.assign(size_t(kExchangeWaves) * kExchangeWaveDwords, 0);
    plan->FusedWaveTable = plan->WaveTable;
    for (uint32_t b : byLevels) {
        const uint32_t tile = tiled ? columnOf[b] / kExchangeTileColumns : 0;
        if (tile >= tileCount) {
            return false;
        }
        uint32_t best = kExchangeWaves;
        for (uint32_t w = 0; w < kExchangeWaves; ++w) {
            if (taken[w * tileCount + tile] < perTile && (best == kExchangeWaves || load[w] < load[best])) {
                best = w;
            }
        }
        if (best == kExchangeWaves) {
            return false;
        }
        waveOf[b] = best;
        registerOf[b] = tile * perTile + taken[best * tileCount + tile]++;
        load[best] += levelsOf[b];
        plan->WaveTable[best * kExchangeWaveDwords + registerOf[b]] = b * 256u;
        if (tiled) {
            plan->FusedWaveTable[best * kExchangeWaveDwords + registerOf[b]] = columnOf[b] % kExchangeTileColumns * kExchangeColumnBytes;
        }
    }

    // ---- trees to the waves that sum them, and to steps
    std::vector<std::vector<uint32_t>> treesOf(kExchangeWaves);
    for (size_t t = 0; t < treeCount / 2 * 2; ++t) {
        treesOf[t / 2 % kExchangeWaves].push_back(static_cast<uint32_t>(t));
    }
    if (treeCount % 2 != 0) {
        treesOf[0].push_back(static_cast<uint32_t>(treeCount - 1));
    }
    size_t longest = 0;
    std::vector<uint32_t> stepOf(treeCount, 0), sumWaveOf(treeCount, 0);
    for (uint32_t w = 0; w < kExchangeWaves; ++w) {
        longest = std::max(longest, treesOf[w].size());
        for (size_t i = 0; i < treesOf[w].size(); ++i) {
            stepOf[treesOf[w][i]] = static_cast<uint32_t>(i);
            sumWaveOf[treesOf[w][i]] = w;
        }
    }
    plan->Rounds = static_cast<uint32_t>((longest + kExchangeRoundSteps - 1) / kExchangeRoundSteps);
    const size_t steps = size_t(plan->Rounds) * kExchangeRoundSteps;

    // ---- levels to groups: a wave's levels in the order of their trees' steps
    std::vector<uint32_t> byStep(treeCount);
    for (size_t t = 0; t < treeCount; ++t) {
        byStep[t] = static_cast<uint32_t>(t);
    }
    std::stable_sort(byStep.begin(), byStep.end(), [&](uint32_t a, uint32_t b) { return stepOf[a] < stepOf[b]; });
    std::vector<TEdge> edges;
    edges.reserve(std::accumulate(levelsOf.begin(), levelsOf.end(), size_t(0)));
    std::vector<TGroup> groups;
    std::vector<std::vector<uint32_t>> groupsOf(kExchangeWaves);
    TTreeEdges edgesOfTree;
    edgesOfTree.At.resize(treeCount);
    for (uint32_t t : byStep) {
        edgesOfTree.At[t] = static_cast<uint32_t>(edgesOfTree.First.size());
        edgesOfTree.First.push_back(static_cast<uint32_t>(edges.size()));
        for (uint32_t d = 0; d < trees[t].Levels.size(); ++d) {
            const TExchangeLevel& level = trees[t].Levels[d];
            const uint32_t w = waveOf[level.Bucket];
            if (groupsOf[w].empty() || groups[groupsOf[w].back()].Edges.size() == maxDepth) {
                groupsOf[w].push_back(static_cast<uint32_t>(groups.size()));
                groups.emplace_back();
                groups.back().Edges.reserve(maxDepth);
            }
            TEdge edge;
            edge.Tree = t;
            edge.Group = groupsOf[w].back();
            edge.Level = &level;
            edge.Lopsided = level.Lopsided;
            edge.ModelLevel = static_cast<uint8_t>(d);
            TGroup& group = groups[edge.Group];
            const uint32_t round = stepOf[t] / kExchangeRoundSteps;
            group.FirstRound = std::min(group.FirstRound, round);
            group.LastRound = std::max(group.LastRound, round);
            group.Edges.push_back(static_cast<uint32_t>(edges.size()));
            edges.push_back(edge);
        }
    }
    edgesOfTree.First.push_back(static_cast<uint32_t>(edges.size()));

    // ---- places in the groups
    if (!TSides(&edges, edgesOfTree, groups, maxDepth).Assign()) {
        return false;
    }
    {
        // of either side on its own, which touch no edge in common: on two threads where there are many
        std::future<void> low = std::async(edges.size() < 8192 ? std::launch::deferred : std::launch::async | std::launch::deferred,
                                           [&] { Colour(&edges, treeCount, groups.size(), false, kEvenPlaces, 0); });
        Colour(&edges, treeCount, groups.size(), true, maxDepth - kEvenPlaces, kEvenPlaces);
        low.get();
    }

    // ---- when a group is compared, and in which slot it stands. A wave compares a group at the end of a step. The barrier of
    // round r stands at the beginning of its last step; behind it come the reads for the next round's first tree. So
    // the last step of round p - 1 and the first three of round p make up *phase* p: a group for the trees of round r
    // is compared in phase r - 1 or before (phase -1: before the first step), and its slot is free again from phase r + 1 on, r
    // the last round that looks at it. As far as slots go a wave compares a group in every step and so stays ahead of the need.
    std::vector<std::vector<uint32_t>> groupsAt(steps * kExchangeWaves), early(kExchangeWaves);
    std::vector<uint32_t> freeSlots;
    for (uint32_t s = kExchangeSlots; s-- > 0;) {
        freeSlots.push_back(s);
    }
    std::vector<std::vector<uint32_t>> freedAfter(plan->Rounds);
    std::vector<size_t> next(kExchangeWaves, 0);
    const int64_t rounds = plan->Rounds;
    plan->CompareSteps = 0;
    for (int64_t phase = -1; phase < rounds; ++phase) {
        std::vector<std::vector<uint32_t>> now(kExchangeWaves);
        const auto nextRound = [&](uint32_t w) {  // first round that needs the wave's next group
            return next[w] < groupsOf[w].size() ? static_cast<int64_t>(groups[groupsOf[w][next[w]]].FirstRound) : rounds + 2;
        };
        const auto place = [&](uint32_t w) {
            TGroup& group = groups[groupsOf[w][next[w]]];
            group.Slot = freeSlots.back();
            freeSlots.pop_back();
            freedAfter[group.LastRound].push_back(group.Slot);
            now[w].push_back(groupsOf[w][next[w]++]);
        };
        for (uint32_t w = 0; w < kExchangeWaves; ++w) {
            while (nextRound(w) <= phase + 1) {
                if (freeSlots.empty()) {
                    return false;
                }
                place(w);
            }
        }
        const int64_t firstStep = std::max<int64_t>(phase * kExchangeRoundSteps - 1, 0);
        const uint32_t stepCount = phase < 0 ? 0 : static_cast<uint32_t>(phase * kExchangeRoundSteps + kExchangeRoundSteps - 1 - firstStep);
        // ahead of the need, not the slots that the next phases' groups may want
        for (uint32_t turn = 0; turn < kExchangeRoundSteps; ++turn) {
            for (uint32_t w = 0; w < kExchangeWaves; ++w) {
                if ((phase < 0 ? turn == 0 : now[w].size() < stepCount) && nextRound(w) <= phase + 2 && freeSlots.size() > 4 * kExchangeWaves) {
                    place(w);
                }
            }
        }
        size_t busiest = 0, together = 0;
        for (const std::vector<uint32_t>& groupsNow : now) {
            busiest = std::max(busiest, groupsNow.size());
            together += groupsNow.size();
        }
        plan->CompareSteps += static_cast<uint32_t>(phase < 0 ? busiest - together / kExchangeWaves : std::max<size_t>(busiest, stepCount));
        for (uint32_t w = 0; w < kExchangeWaves; ++w) {
            for (size_t i = 0; i < now[w].size(); ++i) {
                (phase < 0 ? early[w] : groupsAt[(firstStep + i % stepCount) * kExchangeWaves + w]).push_back(now[w][i]);
            }
        }
        if (phase >= 0) {
            freeSlots.insert(freeSlots.end(), freedAfter[phase].begin(), freedAfter[phase].end());
        }
    }

    // ---- tables
    const auto writeGroup = [&](uint32_t g, uint32_t* row) {
        std::fill(row, row + kExchangeGroupDwords, 0u);
        row[0] = groups[g].Slot * 256u << 16;
        for (uint32_t e : groups[g].Edges) {
            const TEdge& edge = edges[e];
            uint32_t xorByte = edge.Level->Xor, addByte = edge.Level->Add;
            if (six && edge.Place % 2 == 0) {
                // the result goes to bit 6
                if (edge.Level->IsXor) {
                    xorByte &= 0x3fu;
                } else {
                    addByte -= 64;
                }
            }
            row[2 * edge.Place] |= registerOf[edge.Level->Bucket] | xorByte << 8;
            row[2 * edge.Place + 1] = (addByte & 0xffu) * 0x01010101u;
            row[2] |= edge.Level->IsXor ? kExchangeXorFlag : 0u;
        }
    };
    const auto recordOf = [&](size_t step, uint32_t w) {
        return plan->Records.data() + (step / kExchangeRoundSteps * kExchangeWaves + w) * kExchangeRecordDwords;
    };
    plan->Records.assign((size_t(plan->Rounds) + 1) * kExchangeWaves * kExchangeRecordDwords, 0);
    plan->ExtraRows.clear();
    for (uint32_t w = 0; w < kExchangeWaves; ++w) {
        uint32_t* wave = plan->WaveTable.data() + w * kExchangeWaveDwords;
        wave[kExchangeWaveBuckets] = static_cast<uint32_t>(plan->ExtraRows.size() * sizeof(uint32_t));
        wave[kExchangeWaveBuckets + 1] = static_cast<uint32_t>(early[w].size());
        std::copy_n(wave + kExchangeWaveBuckets, 2, plan->FusedWaveTable.data() + w * kExchangeWaveDwords + kExchangeWaveBuckets);
        const auto addExtra = [&](uint32_t g) {
            plan->ExtraRows.resize(plan->ExtraRows.size() + kExchangeGroupDwords);
            uint32_t* row = plan->ExtraRows.data() + plan->ExtraRows.size() - kExchangeGroupDwords;
            writeGroup(g, row);
            return row;
        };
        for (uint32_t g : early[w]) {
            addExtra(g);
        }
        for (size_t step = 0; step < steps; ++step) {
            const std::vector<uint32_t>& at = groupsAt[step * kExchangeWaves + w];
            uint32_t* row = recordOf(step, w) + step % kExchangeRoundSteps * kExchangeGroupDwords;
            if (at.empty()) {
                row[2] = kExchangeSkipFlag;
                continue;
            }
            writeGroup(at[0], row);
            row[2] |= at.size() > 1 ? kExchangeMoreFlag : 0u;
            for (size_t i = 1; i < at.size(); ++i) {
                addExtra(at[i])[2] |= i + 1 < at.size() ? kExchangeMoreFlag : 0u;
            }
        }
    }
    plan->ExtraRows.resize(plan->ExtraRows.size() + kExchangeEarlyRows * kExchangeGroupDwords, 0);
    plan->LeafRows.assign((size_t(plan->Rounds) + 1) * kExchangeWaves * kExchangeRoundSteps, TExchangeLeafRow());
    for (size_t t = 0; t < treeCount; ++t) {
        const size_t step = stepOf[t], inRound = step % kExchangeRoundSteps;
        const uint32_t w = sumWaveOf[t];
        uint32_t* row = recordOf(step, w) + kExchangeRoundSteps * kExchangeGroupDwords + inRound * kExchangeTreeDwords;
        TExchangeLeafRow& leaves = plan->LeafRows[(step / kExchangeRoundSteps * kExchangeWaves + w) * kExchangeRoundSteps + inRound];
        leaves.Tree = static_cast<uint32_t>(t);
        for (uint32_t e = edgesOfTree.Begin(static_cast<uint32_t>(t)); e < edgesOfTree.End(static_cast<uint32_t>(t)); ++e) {
            const TEdge& edge = edges[e];
            row[edge.Place] = groups[edge.Group].Slot * 256u;
            leaves.Levels ^= (kExchangeNoLevel ^ edge.ModelLevel) << 4 * edge.Place;
        }
    }
    return true;
}

void MakeExchangeGrid(bool six, TExchangeColumn* column) {
    const uint32_t cells = ExchangeGridCells(six);
    std::vector<float> borders(column->Values.size());
    std::memcpy(borders.data(), column->Values.data(), borders.size() * sizeof(float));
    column->Scale = column->Bias = 0.0f;
    const float span = borders.empty() ? 0.0f : borders.back() - borders.front();
    if (std::isfinite(span) && span > 0.0f) {
        const float scale = 1.0f / span, bias = -borders.front() * scale;
        if (std::isfinite(scale) && std::isfinite(bias)) {
            column->Scale = scale;
            column->Bias = bias;
        }
    }
    column->Start.assign(cells, 0);
    for (float border : borders) {
        const float place = std::fma(border, column->Scale, column->Bias);
        const float clamped = place > 0.0f ? std::min(place, 1.0f) : 0.0f;  // (NaN: 0)
        const float cell = std::fma(clamped, static_cast<float>(cells - 1), 8388608.0f) - 8388608.0f;
        ++column->Start[static_cast<uint32_t>(cell)];
    }
    const uint32_t tallest = *std::max_element(column->Start.begin(), column->Start.end());
    column->Steps = 0;
    while ((1u << column->Steps) - 1 < tallest) {
        ++column->Steps;
    }
    uint32_t below = 0;
    for (uint32_t& start : column->Start) {
        const uint32_t here = start;
        start = below;
        below += here;
    }
}

bool BuildExchangeTiles(const std::vector<TExchangeColumn>& columns, const std::vector<uint32_t>& pieces, bool six,
                        std::vector<uint32_t>* table, std::vector<uint32_t>* oneHot) {
    constexpr uint32_t kInfoDwords = 4, kOffsetsAt = 64, kHeaderDwords = 320;
    constexpr uint32_t kParameterDwords = 12, kRecordDwords = 16;
    const uint32_t slots = six ? 64 : 128;  // borders of a column, +inf behind the real ones
    const uint32_t cells = ExchangeGridCells(six), columnDwords = slots + cells / 4;
    const uint32_t pieceDwords = kExchangePieceColumns * columnDwords + 4;  // so that the pieces' tables start in different banks
    const uint32_t parametersAt = kExchangeTilePieces * pieceDwords;
    const uint32_t imageDwords = parametersAt + kExchangeTilePieces * kParameterDwords;
    const size_t tiles = columns.size() / kExchangeTileColumns;
    if (tiles == 0 || tiles > kExchangeTiles) {
        return false;
    }
    table->assign(kHeaderDwords + tiles * imageDwords, 0);
    oneHot->clear();
    std::copy(pieces.begin(), pieces.end(), table->begin() + kOffsetsAt);
    for (size_t t = 0; t < tiles; ++t) {
        uint32_t* info = table->data() + t * kInfoDwords;
        uint32_t* image = table->data() + kHeaderDwords + t * imageDwords;
        const TExchangeColumn* tile = columns.data() + t * kExchangeTileColumns;
        std::vector<uint32_t> hot;
        uint32_t steps = 1;
        for (uint32_t c = 0; c < kExchangeTileColumns; ++c) {
            if (tile[c].Used && tile[c].OneHot) {
                hot.push_back(c);
            } else if (tile[c].Used) {
                if (tile[c].Values.size() > slots || tile[c].Steps > kExchangeMaxSteps) {
                    return false;
                }
                steps = std::max(steps, tile[c].Steps);
            }
        }
        info[0] = steps;
        info[1] = static_cast<uint32_t>(hot.size());
        info[2] = static_cast<uint32_t>(oneHot->size() * sizeof(uint32_t));
        for (uint32_t c = 0; c < kExchangeTileColumns; ++c) {
            const bool searched = tile[c].Used && !tile[c].OneHot;
            uint32_t* parameters = image + parametersAt + c / kExchangePieceColumns * kParameterDwords;
            uint32_t* borders = image + c / kExchangePieceColumns * pieceDwords + c % kExchangePieceColumns * columnDwords;
            uint8_t* lut = reinterpret_cast<uint8_t*>(borders + slots);
            for (uint32_t k = 0; k < slots; ++k) {
                borders[k] = searched && k < tile[c].Values.size() ? tile[c].Values[k] : 0x7f800000u;
            }
            if (searched) {
                std::memcpy(parameters + c % kExchangePieceColumns, &tile[c].Scale, 4);
                std::memcpy(parameters + kExchangePieceColumns + c % kExchangePieceColumns, &tile[c].Bias, 4);
                for (uint32_t cell = 0; cell < cells; ++cell) {
                    const uint32_t start = std::min(tile[c].Start[cell], slots + 1 - (1u << steps));  // the search ends inside the slots
                    lut[cell] = static_cast<uint8_t>(six ? start * 4 : start);
                }
            }
            if (c % kExchangePieceColumns == 0) {
                parameters[2 * kExchangePieceColumns] = pieces[(t + 1) % tiles * kExchangeTilePieces + c / kExchangePieceColumns];
            }
        }
        // the one-hot columns: where their records are, then the records (sixteen dwords each, and sixteen per eight values)
        const size_t list = oneHot->size();
        oneHot->resize(list + hot.size(), 0);
        for (size_t k = 0; k < hot.size(); ++k) {
            const TExchangeColumn& column = tile[hot[k]];
            (*oneHot)[list + k] = static_cast<uint32_t>(oneHot->size() * sizeof(uint32_t));
            const size_t chunks = (column.Values.size() + 7) / 8;
            if (chunks == 0) {
                return false;
            }
            const size_t record = oneHot->size();
            oneHot->resize(record + (1 + chunks) * kRecordDwords, 0);
            (*oneHot)[record] = column.RowByte;
            (*oneHot)[record + 1] = hot[k] * kExchangeColumnBytes;
            (*oneHot)[record + 2] = static_cast<uint32_t>(chunks);
            for (size_t i = 0; i < 8 * chunks; ++i) {
                const size_t value = i < column.Values.size() ? i : 0;  // the first one again behind the last
                (*oneHot)[record + kRecordDwords + 2 * i] = column.Values[value];
                (*oneHot)[record + kRecordDwords + 2 * i + 1] = static_cast<uint32_t>(value) + 1;
            }
        }
    }
    if (oneHot->empty()) {
        oneHot->resize(1, 0);
    }
    return true;
}

}  // namespace cbamd
