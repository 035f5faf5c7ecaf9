/* Pipeline<float> over a library that is not there: the C interface it stands on is played here, with copies that arrive as soon as they may and memory that
 * is overwritten as it is freed, so that what a caller is promised can be tested without a device, and steps can be made to fail.
 * tests/test_pipeline_states.py compiles and runs it, with the name of what is to be tested. */
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "visualmesh/engine/hip/engine.hpp"
#include "visualmesh/geometry/Sphere.hpp"
#include "visualmesh/mesh.hpp"
#include "visualmesh/model/ring6.hpp"

struct vmhip_engine {};
struct vmhip_mesh {};
struct vmhip_batch {
    bool streaming = false, layers = false;
    std::vector<uint32_t> V; /* a frame's fourcc is its number of visible nodes */
    uint8_t* block = nullptr;
};
namespace {
constexpr int NN = 6, CLASSES = 4;
std::vector<std::pair<void*, size_t>> blocks;
std::string failing;      /* the step that fails next */
std::string last_error = "played";
bool fails(const char* step) {
    if (failing != step) return false;
    failing.clear();
    return true;
}
int refused(const char* why) {
    last_error = why;
    return VMHIP_ERR_ARGUMENT;
}
size_t padded(size_t n) { return (n + 255) / 256 * 256; }
size_t geometry(uint32_t V) { return padded(8 * V) + padded(4 * V) + padded(4 * NN * (V + 1)); }
size_t classes(uint32_t V) { return padded(4 * CLASSES * (V + 1)); }
size_t geometry(const vmhip_batch* b) {
    size_t n = 0;
    for (uint32_t V : b->V) n += geometry(V);
    return n;
}
size_t total(const vmhip_batch* b) {
    size_t n = geometry(b);
    for (uint32_t V : b->V) n += classes(V);
    return n;
}
uint8_t mark(const vmhip_batch* b) { return uint8_t(b->V[0]); }
}  // namespace
extern "C" {
const char* vmhip_last_error(void) { return last_error.c_str(); }
int vmhip_engine_create(const vmhip_network*, int32_t, int32_t, vmhip_engine** out) { return *out = new vmhip_engine, VMHIP_OK; }
void vmhip_engine_destroy(vmhip_engine* e) { delete e; }
int32_t vmhip_engine_n_classes(const vmhip_engine*) { return CLASSES; }
int vmhip_mesh_upload(const float*, const int32_t*, int32_t, int32_t, vmhip_mesh** out) { return *out = new vmhip_mesh, VMHIP_OK; }
int vmhip_mesh_attach_tree(vmhip_mesh*, const vmhip_tree_element*, int32_t) { return VMHIP_OK; }
void vmhip_mesh_release(vmhip_mesh* m) { delete m; }
int vmhip_batch_create(vmhip_engine*, vmhip_batch** out) { return *out = new vmhip_batch, VMHIP_OK; }
void vmhip_batch_destroy(vmhip_batch* b) { delete b; }
int vmhip_batch_set_untested(vmhip_batch*, int32_t, const int32_t*, int32_t) { return VMHIP_OK; }
void* vmhip_host_alloc(size_t n) { return blocks.push_back({std::calloc(1, n), n}), blocks.back().first; }
void vmhip_host_free(void* p) {
    for (auto& b : blocks)
        if (b.first == p) std::memset(p, 0xdd, b.second);
}
size_t vmhip_batch_fetch_packed_size(const vmhip_batch* b) { return total(b); }
int vmhip_batch_stream_begin(vmhip_batch* b, vmhip_batch* first, const vmhip_frame* frames, int32_t n, int32_t* n_visible) {
    if (!b || !first || !n_visible) return refused("stream_begin: null argument");
    if (b->streaming) return refused("stream_begin: still under way");
    if (fails("begin")) return VMHIP_ERR_HIP;
    b->V.clear();
    for (int32_t i = 0; i < n; ++i) b->V.push_back(frames[i].fourcc), n_visible[i] = int32_t(frames[i].fourcc);
    b->streaming = true, b->layers = false, b->block = nullptr;
    return VMHIP_OK;
}
int vmhip_batch_stream_geometry(vmhip_batch* b, void* block, size_t bytes, vmhip_result* results) {
    if (!b || !b->streaming || total(b) > bytes) return refused("stream_geometry: no frames under way, or a small block");
    b->block = static_cast<uint8_t*>(block);
    size_t at = 0, at_classes = geometry(b);
    for (size_t i = 0; i < b->V.size(); ++i) {
        const uint32_t V = b->V[i];
        results[i] = vmhip_result{};
        results[i].capacity = results[i].n_visible = int32_t(V);
        results[i].pixel_coordinates = reinterpret_cast<float*>(b->block + at);
        results[i].classifications = reinterpret_cast<float*>(b->block + at_classes);
        at += geometry(V), at_classes += classes(V);
    }
    std::memset(block, mark(b), geometry(b));
    return VMHIP_OK;
}
int vmhip_batch_stream_layers(vmhip_batch* b) {
    if (!b || !b->streaming) return refused("stream_layers: no frames under way");
    if (fails("layers")) return b->streaming = false, VMHIP_ERR_HIP;
    b->layers = true;
    return VMHIP_OK;
}
int vmhip_batch_stream_images(vmhip_batch* b) {
    if (!b || !b->streaming) return refused("stream_images: no frames under way");
    return fails("images") ? VMHIP_ERR_HIP : VMHIP_OK;
}
int vmhip_batch_stream_classes(vmhip_batch* b) {
    if (!b || !b->streaming) return refused("stream_classes: no frames under way");
    if (!b->layers) return b->streaming = false, VMHIP_OK;
    if (fails("classes")) return b->streaming = false, VMHIP_ERR_HIP;
    std::memset(b->block + geometry(b), mark(b), total(b) - geometry(b));
    return VMHIP_OK;
}
int vmhip_batch_stream_end(vmhip_batch* b) { return b->streaming = false, VMHIP_OK; }
/* not reached by a pipeline */
int vmhip_batch_graph_stats(const vmhip_batch*, int64_t*, int64_t*, int64_t*) { return VMHIP_OK; }
int vmhip_batch_stage(vmhip_batch*, const vmhip_frame*, int32_t, int32_t) { std::abort(); }
int vmhip_batch_stage_async(vmhip_batch*, const vmhip_frame*, int32_t, int32_t) { std::abort(); }
int vmhip_batch_classify_begin(vmhip_batch*, const vmhip_frame*, int32_t, vmhip_result*) { std::abort(); }
}

using Engine = visualmesh::engine::hip::Engine<float>;
using Pipeline = visualmesh::engine::hip::Pipeline<float>;
using Frames = std::vector<Engine::Frame<visualmesh::model::Ring6>>;
using Results = std::vector<vmhip_result>;

#define CHECK(what)                                              \
    do {                                                         \
        if (!(what)) {                                           \
            std::printf("line %d: %s\n", __LINE__, #what);       \
            return 1;                                            \
        }                                                        \
    } while (0)

struct Caller {
    visualmesh::Mesh<float, visualmesh::model::Ring6> mesh{visualmesh::geometry::Sphere<float>(0.0949f), 1.2f, 1.0f, 3.0f};
    Pipeline pipe;
    /* a batch of frames of V, V + 1, ... visible nodes */
    Frames batch(uint32_t V, size_t n) {
        visualmesh::mat4<float> Hoc = {{{{1, 0, 0, 0}}, {{0, 1, 0, 0}}, {{0, 0, 1, 1.2f}}, {{0, 0, 0, 1}}}};
        visualmesh::Lens<float> lens;
        lens.dimensions = {{320, 256}};
        lens.projection = visualmesh::EQUISOLID;
        lens.focal_length = 105;
        lens.centre = {{0, 0}};
        lens.k = {{0, 0}};
        lens.fov = 3.14159265f;
        Frames f;
        for (size_t i = 0; i < n; ++i) f.push_back({&mesh, Hoc, lens, this, uint32_t(V + i)});
        return f;
    }
    const Results* submit(uint32_t V, size_t n) { return pipe.submit<visualmesh::model::Ring6>(batch(V, n)); }
    bool throws(uint32_t V, size_t n) {
        try {
            (void) submit(V, n);
        } catch (const std::exception&) {
            return true;
        }
        return false;
    }
    bool flush_throws() {
        try {
            (void) pipe.flush();
        } catch (const std::exception&) {
            return true;
        }
        return false;
    }
    /* the results are those of the batch of `n` frames of V nodes and on, every byte of them */
    static bool are(const Results* r, uint32_t V, size_t n) {
        if (!r || r->size() != n) return false;
        for (size_t i = 0; i < n; ++i) {
            if ((*r)[i].n_visible != int32_t(V + i)) return false;
            const uint8_t* const px = reinterpret_cast<const uint8_t*>((*r)[i].pixel_coordinates);
            const uint8_t* const cls = reinterpret_cast<const uint8_t*>((*r)[i].classifications);
            for (size_t k = 0; k < geometry(uint32_t(V + i)); ++k)
                if (px[k] != uint8_t(V)) return false;
            for (size_t k = 0; k < classes(uint32_t(V + i)); ++k)
                if (cls[k] != uint8_t(V)) return false;
        }
        return true;
    }
};

/* results stay as they are until two more calls, also beside batches that need larger blocks, and while the pipeline drains */
int held() {
    Caller c;
    const Results* last = nullptr;
    for (uint32_t step = 0; step < 9; ++step) {
        const Results* done = c.submit(10 + 20 * step, 2 + step % 3);
        if (last) CHECK(Caller::are(last, 10 + 20 * (step - 3), 2 + (step - 3) % 3));
        CHECK((done != nullptr) == (step >= 2));
        if (done) CHECK(Caller::are(done, 10 + 20 * (step - 2), 2 + (step - 2) % 3));
        last = done;
    }
    const Results* first = c.pipe.flush();
    CHECK(Caller::are(last, 10 + 20 * 6, 2));
    CHECK(Caller::are(first, 10 + 20 * 7, 3));
    const Results* second = c.pipe.flush();
    CHECK(Caller::are(first, 10 + 20 * 7, 3));
    CHECK(Caller::are(second, 10 + 20 * 8, 4));
    CHECK(c.submit(200, 5) == nullptr);
    CHECK(Caller::are(second, 10 + 20 * 8, 4));
    CHECK(Caller::are(c.pipe.flush(), 200, 5));
    CHECK(c.pipe.flush() == nullptr);
    return 0;
}

/* batches without frames, the first one among them */
int empty() {
    for (uint32_t first = 0; first < 4; ++first) {  // batches before the first empty one
        Caller c;
        uint32_t step = 0;
        for (; step < first; ++step) CHECK(Caller::are(c.submit(10 + step, 2), 10 + step - 2, 2) == (step >= 2));
        const Results* done = c.submit(0, 0);
        CHECK(step >= 2 ? Caller::are(done, 10 + step - 2, 2) : done == nullptr);
        CHECK(c.pipe.engine(int(step)).n_classes() == CLASSES);
        for (++step; step < 8; ++step) {
            done = c.submit(10 + step, 2);
            if (step - 2 == first) CHECK(done && done->empty());
            else if (step >= 2) CHECK(Caller::are(done, 10 + step - 2, 2));
            else CHECK(done == nullptr);
        }
        CHECK(Caller::are(c.pipe.flush(), 16, 2));
        CHECK(Caller::are(c.pipe.flush(), 17, 2));
        CHECK(c.pipe.flush() == nullptr);
    }
    return 0;
}

/* a step that fails: the batch is lost, the call that would have returned it says so (the call that submits it, if it never was under way), every other batch comes as it would have */
int failures() {
    const char* steps[] = {"begin", "layers", "images", "classes"};
    for (const std::string step : steps)
        for (uint32_t lost = 0; lost < 4; ++lost) {
            const bool at_once = step == "begin" || step == "layers";
            Caller c;
            std::vector<uint32_t> order; /* what is under way, 0 for the batch that will be missing */
            for (uint32_t turn = 0; turn < 9; ++turn) {
                const uint32_t V = 10 + turn;
                if (turn == lost && at_once) {
                    failing = step;
                    CHECK(c.throws(V, 2));
                    continue; /* as if it had not been submitted */
                }
                order.push_back(turn == lost ? 0 : V);
                if (order.size() > 2 && order[order.size() - 3] == 0) {
                    failing = step == "classes" ? step : failing;
                    CHECK(c.throws(V, 2));
                    CHECK(failing.empty());
                    continue;
                }
                const Results* done = c.submit(V, 2);
                if (turn == lost && step == "images") failing = step; /* fails in the next call, is told by the one after that */
                if (order.size() > 2) CHECK(Caller::are(done, order[order.size() - 3], 2));
                else CHECK(done == nullptr);
            }
            CHECK(Caller::are(c.pipe.flush(), 17, 2));
            CHECK(Caller::are(c.pipe.flush(), 18, 2));
            CHECK(c.pipe.flush() == nullptr);
            CHECK(c.pipe.flush() == nullptr);
        }
    /* while the pipeline drains, and behind that */
    Caller c;
    CHECK(c.submit(20, 2) == nullptr && c.submit(21, 3) == nullptr);
    failing = "classes";
    CHECK(c.flush_throws());
    CHECK(Caller::are(c.pipe.flush(), 21, 3));
    CHECK(c.pipe.flush() == nullptr);
    failing = "begin";
    CHECK(c.throws(22, 2));
    CHECK(c.pipe.flush() == nullptr && c.pipe.flush() == nullptr && c.pipe.flush() == nullptr);
    CHECK(c.submit(23, 2) == nullptr);
    CHECK(Caller::are(c.pipe.flush(), 23, 2));
    CHECK(c.pipe.flush() == nullptr);
    return 0;
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    const int rc = what == "held" ? held() : what == "empty" ? empty() : what == "failures" ? failures() : 2;
    if (rc == 0) std::puts("ok");
    return rc;
}
