// TEST INFRASTRUCTURE. The collapse of a binary tree into four-wide nodes
// (ratbite_amd/csrc/device/collapse.hpp) on the CPU, one node at a time: the
// indices that the nodes take are checked before anything is written there.
#include <cstring>
#include <vector>

#include "../../ratbite_amd/csrc/device/collapse.hpp"

using namespace rbh;
using namespace rbh::lbvh;

extern "C" {

// Collapses the binary tree `nodes` over n >= 2 triangles (root 0) as
// kernels/lbvh.hip does, into out4 and out4h of max_nodes4(n) nodes; writes[i]
// counts how often index i was taken. Returns the number of four-wide nodes or,
// at an index that is not one of the allocated ones, ~index.
int64_t host_collapse(const BvhNode* nodes, uint32_t n, void* out4, void* out4h, uint32_t* writes) {
    const uint32_t cap = max_nodes4(n);
    std::vector<Bvh4Node> n4(cap);
    std::vector<Bvh4HNode> n4h(cap);   // (aligned, which the caller's arrays need not be)
    std::vector<Open> open{Open{0u, 0, 1u}};
    int64_t count = 0;
    while (!open.empty()) {
        const Open t = open.back();
        open.pop_back();
        if (t.id >= cap) return ~(int64_t)t.id;
        ++writes[t.id];
        ++count;
        Open next[4];
        const uint32_t inner = collapse_node(t, nodes, n4.data(), n4h.data(), next);
        for (uint32_t k = 0; k < inner; ++k) open.push_back(next[k]);
    }
    std::memcpy(out4, n4.data(), cap * sizeof(Bvh4Node));
    std::memcpy(out4h, n4h.data(), cap * sizeof(Bvh4HNode));
    return count;
}

uint32_t host_max_nodes4(uint32_t n) { return max_nodes4(n); }

}  // extern "C"
