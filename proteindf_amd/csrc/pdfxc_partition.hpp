// The shape of a grid's bisection, which follows from its number of points
// alone: the nodes of every level and the chunks of their points, and the nodes
// left to one workgroup each.  Plain C++, for the host and the device.
#pragma once

#include <algorithm>
#include <cstdint>
#include <utility>
#include <vector>

namespace pdfxc {

constexpr int kLeafPts = 128;   // points of a block
constexpr int kNodeMax = 4096;  // points of a node that one workgroup cuts in LDS (120 KiB)
constexpr int kChunk = 4096;    // points per workgroup of the level passes
constexpr int kPartThreads = 256;

struct PartNode {
    int lo, hi, mid;
};
struct PartChunk {
    int node, lo, hi;
};
struct LeafNode {
    int lo, hi, buf;
};

struct PartTree {
    std::vector<PartNode> nodes;        // of all levels, a level after the other
    std::vector<PartChunk> chunks;      // node: its number within the level
    std::vector<int> node_off{0}, chunk_off{0};
    std::vector<LeafNode> leaves;
    size_t most = 0;                    // nodes of the fullest level
};

// Positions go up to 2^31 - 129: sums past a node's end are taken in 64 bits.
inline PartTree part_tree(int64_t n) {
    PartTree T;
    std::vector<std::pair<int, int>> cur{{0, (int)n}}, next;
    for (int level = 0; !cur.empty(); ++level) {
        next.clear();
        for (const auto& [lo, hi] : cur) {
            if (hi - lo <= kNodeMax) {
                T.leaves.push_back(LeafNode{lo, hi, level & 1});
                continue;
            }
            const int mid = lo + ((hi - lo + kLeafPts - 1) / kLeafPts / 2) * kLeafPts;
            const int id = (int)T.nodes.size() - T.node_off.back();
            T.nodes.push_back(PartNode{lo, hi, mid});
            for (int64_t k = lo; k < hi; k += kChunk)
                T.chunks.push_back(PartChunk{id, (int)k, (int)std::min<int64_t>(hi, k + kChunk)});
            next.push_back({lo, mid});
            next.push_back({mid, hi});
        }
        if ((int)T.nodes.size() > T.node_off.back()) {
            T.most = std::max(T.most, T.nodes.size() - T.node_off.back());
            T.node_off.push_back((int)T.nodes.size());
            T.chunk_off.push_back((int)T.chunks.size());
        }
        cur.swap(next);
    }
    return T;
}

// f(position) for the points of a chunk that thread t of kPartThreads takes;
// counted within the chunk, whose end may be the last position an int holds
template <typename F>
constexpr void each_point(const PartChunk& C, int t, F f) {
    for (int k = t; k < C.hi - C.lo; k += kPartThreads) f(C.lo + k);
}

}  // namespace pdfxc
