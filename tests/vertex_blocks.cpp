// Prints the vertex blocks of a mesh read from stdin: element, vertices,
// elements, most incidences and most slots of a block, then the topology.
// Output: incidences of every slot on one line, then a line per block {first
// slot, slots, first owners index, incidences}.
#include <cstdio>
#include <vector>

#include "oe_host.hpp"

int main() {
    int element, nv, ne, max_inc, max_slots;
    if (std::scanf("%d %d %d %d %d", &element, &nv, &ne, &max_inc, &max_slots) != 5) return 1;
    oe::HostMesh m;
    m.element = static_cast<oe::Element>(element);
    m.xyz.assign(3 * static_cast<size_t>(nv), 0.f);
    m.topo.resize(static_cast<size_t>(ne) * oe::elem_nb_vertices(m.element));
    for (int32_t& v : m.topo)
        if (std::scanf("%d", &v) != 1) return 1;
    const oe::OwnersCSR o =
        oe::build_owners(m, oe::color_dsat(oe::build_primal_graph(m.element, m.topo, nv)), true);
    std::vector<int32_t> blocks, begin;
    oe::build_vertex_blocks(o, max_inc, max_slots, blocks, begin);
    for (int32_t n : o.slot_nb) std::printf("%d ", n);
    std::printf("\n");
    for (size_t i = 0; i < blocks.size(); i += 4)
        std::printf("%d %d %d %d\n", blocks[i], blocks[i + 1], blocks[i + 2], blocks[i + 3]);
    return 0;
}
