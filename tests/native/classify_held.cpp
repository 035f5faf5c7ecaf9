/* Engine::classify_held: the same arrays as the call by value, left on the device where they are more than the caller asked for, past the kept block where
 * they are more than that may hold. tests/test_classify_held.py compiles, links and runs it. */
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "visualmesh/engine/hip/engine.hpp"
#include "visualmesh/geometry/Sphere.hpp"
#include "visualmesh/mesh.hpp"
#include "visualmesh/model/ring6.hpp"
#include "visualmesh/utility/fourcc.hpp"

using Engine = visualmesh::engine::hip::Engine<float>;
using Mesh = visualmesh::Mesh<float, visualmesh::model::Ring6>;

static bool same(const vmhip_result& got, const visualmesh::ClassifiedMesh<float, 6>& want) {
    const size_t V = want.global_indices.size();
    return size_t(got.n_visible) == V && !std::memcmp(got.pixel_coordinates, want.pixel_coordinates.data(), 8 * V)
           && !std::memcmp(got.global_indices, want.global_indices.data(), 4 * V) && !std::memcmp(got.neighbourhood, want.neighbourhood.data(), 4 * 6 * (V + 1))
           && !std::memcmp(got.classifications, want.classifications.data(), 4 * want.classifications.size());
}

int main() {
    visualmesh::mat4<float> down = {{{{0, 0, 1, 0}}, {{0, 1, 0, 0}}, {{-1, 0, 0, 1.2f}}, {{0, 0, 0, 1}}}}, up = {{{{0, 0, -1, 0}}, {{0, 1, 0, 0}}, {{1, 0, 0, 1.2f}}, {{0, 0, 0, 1}}}};
    visualmesh::Lens<float> lens;
    lens.dimensions = {{640, 640}};
    lens.projection = visualmesh::EQUIDISTANT;
    lens.focal_length = 200;
    lens.centre = {{0, 0}};
    lens.k = {{0, 0}};
    lens.fov = 3.14159265f;
    std::vector<uint8_t> image(640 * 640 * 4);
    for (size_t i = 0; i < image.size(); ++i) image[i] = uint8_t(i * 2654435761u >> 24);
    const uint32_t rgba = visualmesh::fourcc("RGBA");
    const Engine by_value{visualmesh::NetworkStructure<float>()}, engine{visualmesh::NetworkStructure<float>()};
    for (const float k : {2.0f, 27.0f}) { /* some hundred KB; more than 64 MB */
        const Mesh mesh(visualmesh::geometry::Sphere<float>(0.0949f), 1.2f, k, 20.0f);
        const auto want = by_value(mesh, down, lens, image.data(), rgba);
        const size_t V = want.global_indices.size();
        if (V == 0 || (V * 52 > VMHIP_HELD_MOST) != (k == 27.0f)) return std::printf("%zu nodes\n", V), 1;
        for (int turn = 0; turn < 2; ++turn) {
            if (!same(engine.classify_held(mesh, down, lens, image.data(), rgba), want)) return std::printf("held, k %g\n", double(k)), 1;
            const vmhip_result r = engine.classify_held(mesh, down, lens, image.data(), rgba, 1024);
            if (size_t(r.n_visible) != V || r.pixel_coordinates || r.global_indices || r.neighbourhood || r.classifications) return std::printf("on the device, k %g\n", double(k)), 1;
            const auto fetched = engine.fetch<visualmesh::model::Ring6>();
            if (fetched[0].global_indices != want.global_indices || fetched[0].classifications != want.classifications) return std::printf("fetched, k %g\n", double(k)), 1;
        }
        const vmhip_result none = engine.classify_held(mesh, up, lens, image.data(), rgba);
        if (size_t(none.n_visible) != by_value(mesh, up, lens, image.data(), rgba).global_indices.size()) return std::printf("up, k %g\n", double(k)), 1;
    }
    std::puts("ok");
    return 0;
}
