/* Packed fetches through the C++ engine, announced beforehand and not: the arrays in the block are those of fetch().
 * tests/test_fetch_packed_early.py compiles, links and runs it. */
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "visualmesh/engine/hip/engine.hpp"
#include "visualmesh/geometry/Sphere.hpp"
#include "visualmesh/mesh.hpp"
#include "visualmesh/model/ring6.hpp"
#include "visualmesh/utility/fourcc.hpp"

int main() {
    using Engine = visualmesh::engine::hip::Engine<float>;
    visualmesh::Mesh<float, visualmesh::model::Ring6> mesh(visualmesh::geometry::Sphere<float>(0.0949f), 1.2f, 3.0f, 5.0f);
    visualmesh::mat4<float> Hoc = {{{{1, 0, 0, 0}}, {{0, 1, 0, 0}}, {{0, 0, 1, 1.2f}}, {{0, 0, 0, 1}}}};
    visualmesh::Lens<float> lens;
    lens.dimensions = {{320, 256}};
    lens.projection = visualmesh::EQUISOLID;
    lens.focal_length = 105;
    lens.centre = {{0, 0}};
    lens.k = {{0, 0}};
    lens.fov = 3.14159265f;
    std::vector<uint8_t> image(320 * 256 * 4);
    for (size_t i = 0; i < image.size(); ++i) image[i] = uint8_t(i * 2654435761u >> 24);

    Engine engine{visualmesh::NetworkStructure<float>()}; /* the sampled channels are the classes */
    engine.announce_packed(nullptr, 0);                   /* nothing staged yet: no effect */
    engine.stage(std::vector<Engine::Frame<visualmesh::model::Ring6>>(2, {&mesh, Hoc, lens, image.data(), visualmesh::fourcc("RGBA")}));
    engine.run();
    const auto want = engine.fetch<visualmesh::model::Ring6>();
    const size_t bytes = engine.packed_size();
    void* const block = vmhip_host_alloc(bytes);
    bool same = block != nullptr && !want[0].global_indices.empty();
    for (int turn = 0; same && turn < 6; ++turn) {
        const bool announced = turn % 3 != 2;
        if (announced) engine.announce_packed(block, bytes);
        std::memset(block, 0xee, bytes);
        engine.run();
        std::vector<vmhip_result> got;
        engine.fetch_packed_async(block, bytes, got);
        engine.fetch_wait();
        for (size_t i = 0; i < want.size(); ++i) {
            const size_t V = want[i].global_indices.size();
            same = same && size_t(got[i].n_visible) == V && !std::memcmp(got[i].pixel_coordinates, want[i].pixel_coordinates.data(), 8 * V)
                   && !std::memcmp(got[i].global_indices, want[i].global_indices.data(), 4 * V)
                   && !std::memcmp(got[i].neighbourhood, want[i].neighbourhood.data(), 4 * 6 * (V + 1))
                   && !std::memcmp(got[i].classifications, want[i].classifications.data(), 4 * want[i].classifications.size());
        }
    }
    engine.announce_packed(block, bytes);
    engine.announce_packed(nullptr, 0); /* withdrawn: the block may go */
    vmhip_host_free(block);
    engine.run();
    std::puts(same ? "ok" : "differ");
    return same ? 0 : 1;
}
