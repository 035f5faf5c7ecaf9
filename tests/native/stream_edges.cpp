/* A batch of a stream of batches that follows other work of its engine: frames staged and never run, a run whose results were never fetched.
 * tests/test_stream_edges.py compiles, links and runs it. */
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "visualmesh/engine/hip/engine.hpp"
#include "visualmesh/geometry/Sphere.hpp"
#include "visualmesh/mesh.hpp"
#include "visualmesh/model/ring6.hpp"
#include "visualmesh/utility/fourcc.hpp"

using Engine = visualmesh::engine::hip::Engine<float>;
using Frames = std::vector<Engine::Frame<visualmesh::model::Ring6>>;
using Wanted = std::vector<visualmesh::ClassifiedMesh<float, 6>>;

struct Scene {
    int width, height;
    visualmesh::Mesh<float, visualmesh::model::Ring6> mesh;
    uint8_t* images;
    size_t n;
    Scene(int w, int h, float k, size_t frames) : width(w), height(h), mesh(visualmesh::geometry::Sphere<float>(0.0949f), 1.2f, k, 8.0f), n(frames) {
        const size_t bytes = size_t(4) * w * h * n;
        images = static_cast<uint8_t*>(vmhip_host_alloc(bytes));
        for (size_t i = 0; i < bytes; ++i) images[i] = uint8_t((i + size_t(w)) * 2654435761u >> 24);
    }
    ~Scene() { vmhip_host_free(images); }
    Frames frames() const {
        visualmesh::Lens<float> lens;
        lens.dimensions = {{width, height}};
        lens.projection = visualmesh::EQUISOLID;
        lens.focal_length = 0.33f * float(width);
        lens.centre = {{0, 0}};
        lens.k = {{0, 0}};
        lens.fov = 3.14159265f;
        Frames out;
        for (size_t i = 0; i < n; ++i) {
            const float pitch = 0.3f + 0.1f * float(i), c = std::cos(pitch), s = std::sin(pitch);
            visualmesh::mat4<float> Hoc = {{{{c, 0, s, 0}}, {{0, 1, 0, 0}}, {{-s, 0, c, 1.2f}}, {{0, 0, 0, 1}}}};
            out.push_back({&mesh, Hoc, lens, images + size_t(4) * width * height * i, visualmesh::fourcc("RGBA")});
        }
        return out;
    }
};

static bool same(const std::vector<vmhip_result>& got, const Wanted& want) {
    if (got.size() != want.size()) return false;
    for (size_t i = 0; i < want.size(); ++i) {
        const size_t V = want[i].global_indices.size();
        if (V == 0 || size_t(got[i].n_visible) != V || std::memcmp(got[i].pixel_coordinates, want[i].pixel_coordinates.data(), 8 * V)
            || std::memcmp(got[i].global_indices, want[i].global_indices.data(), 4 * V) || std::memcmp(got[i].neighbourhood, want[i].neighbourhood.data(), 4 * 6 * (V + 1))
            || std::memcmp(got[i].classifications, want[i].classifications.data(), 4 * want[i].classifications.size()))
            return false;
    }
    return true;
}

static bool stream(const Engine& engine, const Scene& scene, const Wanted& want) {
    std::vector<vmhip_result> got;
    (void) engine.stream_begin(scene.frames(), engine);
    const size_t bytes = engine.packed_size();
    void* const block = vmhip_host_alloc(bytes);
    engine.stream_geometry(block, bytes, got);
    engine.stream_layers();
    engine.stream_images();
    engine.stream_classes();
    engine.stream_end();
    const bool ok = same(got, want);
    vmhip_host_free(block);
    return ok;
}

int main() {
    const Scene large(1280, 1024, 5.0f, 6), small(320, 256, 3.0f, 2);
    visualmesh::NetworkStructure<float> network; /* the sampled channels are the classes */
    const Engine reference(network), engine(network);
    reference.stage(large.frames());
    reference.run();
    const Wanted want_large = reference.fetch<visualmesh::model::Ring6>();
    reference.stage(small.frames());
    reference.run();
    const Wanted want_small = reference.fetch<visualmesh::model::Ring6>();

    for (int turn = 0; turn < 4; ++turn) {
        engine.stage_async(turn % 2 ? small.frames() : large.frames());  // and never run
        if (!stream(engine, turn % 2 ? large : small, turn % 2 ? want_large : want_small)) return std::printf("staged and never run, turn %d\n", turn), 1;
    }
    void* block = nullptr;
    size_t bytes = 0;
    for (int turn = 0; turn < 4; ++turn) {
        engine.stage(large.frames());
        if (turn > 0) engine.announce_packed(block, bytes);
        engine.run();
        if (turn == 0) bytes = engine.packed_size(), block = vmhip_host_alloc(bytes);
        if (!stream(engine, small, want_small)) return std::printf("run and never fetched, turn %d\n", turn), 1;
    }
    engine.stage(large.frames());
    engine.announce_packed(block, bytes);
    engine.run();
    std::vector<vmhip_result> got;
    engine.fetch_packed_async(block, bytes, got);
    engine.fetch_wait();
    if (!same(got, want_large)) return std::puts("a run behind the streams"), 1;
    vmhip_host_free(block);

    std::string names; /* of the kernels of a profiled pass: both parts of it */
    if (vmhip_batch_profile(engine.native_batch(), 1) != VMHIP_OK || !stream(engine, large, want_large)) return std::puts("a profiled stream"), 1;
    const char* name[16] = {};
    float ms[16];
    int64_t units[16];
    int32_t n = 0;
    if (vmhip_batch_profile_read(engine.native_batch(), 16, &n, name, ms, units) != VMHIP_OK) return std::puts("profile_read"), 1;
    for (int i = 0; i < n; ++i) names += std::string(name[i]) + (ms[i] > 0.0f && ms[i] < 5.0f && units[i] > 0 ? " " : "? ");
    if (names != "project compact neighbourhood sample ") return std::printf("profiled: %s\n", names.c_str()), 1;
    std::puts("ok");
    return 0;
}
