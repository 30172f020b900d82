// The C ABI the host layer stands on, in host memory: allocations, transfers and copies are done, ops are counted and not run.
// With it the layer's own bookkeeping (who owns what, what is recorded, what is waited for) runs without a GPU.
// Below it, the questions tests/test_host_layer.py asks; each returns what it found.
#include <cstdlib>
#include <cstring>
#include <memory>
#include <set>

#include "llm.hpp"

struct shv_ctx {
    int unwaited = 0;  // copies since the stream was last waited for
};
struct shv_prerecorded {
    int ops;
};

namespace {
int g_contexts = 0, g_recorded = 0, g_enqueued = 0, g_given = 0;
size_t g_free = size_t(16) << 30;  // what the device claims to have left
std::set<void *> g_memory;
int take(size_t bytes, void **p) {
    *p = std::calloc(1, bytes);
    g_memory.insert(*p);
    return 0;
}
int give(void *p) {
    if (p && !g_memory.erase(p)) return -1;
    g_given++;
    std::free(p);
    return 0;
}
}  // namespace

extern "C" {
const char *shv_last_error(void) { return "the double refuses"; }
int shv_init(int, shv_ctx **out) { return *out = new shv_ctx, g_contexts++, 0; }
void shv_destroy(shv_ctx *c) {
    if (c) g_contexts--;
    delete c;
}
int shv_sync(shv_ctx *c) { return c->unwaited = 0; }
int shv_alloc(shv_ctx *, size_t bytes, void **p) { return take(bytes, p); }
int shv_free(shv_ctx *, void *p) { return give(p); }
int shv_device_props(shv_ctx *, shv_props *p) { return std::memset(p, 0, sizeof *p), p->hbm_bytes = 16ull << 30, 0; }
int shv_block_alloc(int, size_t bytes, size_t keep, void **p) { return bytes + keep > g_free ? SHV_E_NOMEM : take(bytes, p); }
int shv_block_free(int, void *p) { return give(p); }
int shv_block_read(int, void *dst, const void *src, size_t n) { return std::memcpy(dst, src, n), 0; }
int shv_host_alloc(shv_ctx *, size_t bytes, void **p) { return take(bytes, p); }
int shv_host_free(shv_ctx *, void *p) { return give(p); }
int shv_upload_async(shv_ctx *, void *dst, const void *src, size_t n) { return std::memcpy(dst, src, n), 0; }
int shv_download(shv_ctx *c, void *dst, const void *src, size_t n) { return std::memcpy(dst, src, n), c->unwaited = 0; }
int shv_copy(shv_ctx *c, void *dst, const void *src, size_t n) { return std::memmove(dst, src, n), c->unwaited++, 0; }
int shv_zero(shv_ctx *, void *dst, size_t n) { return std::memset(dst, 0, n), 0; }
int shv_upload_words(shv_ctx *, const shv_words *w, int n) {
    for (int i = 0; i < n; i++) std::memcpy(w[i].dst, w[i].src, static_cast<size_t>(w[i].n) * 4);
    return 0;
}
int shv_copy_spans(shv_ctx *c, const shv_span *s, int n) {
    for (int i = 0; i < n; i++) s[i].src ? std::memcpy(s[i].dst, s[i].src, s[i].bytes) : std::memset(s[i].dst, 0, s[i].bytes);
    c->unwaited++;
    return 0;
}
int shv_enqueue(shv_ctx *, uint32_t, const void *, size_t) { return g_enqueued++, 0; }
int shv_dispatch_multi(shv_ctx *, const shv_op *, int, int, uint64_t *ns, uint64_t *) { return *ns = 0; }
int shv_prerecord(shv_ctx *, const shv_op *, int n, shv_prerecorded **out) { return *out = new shv_prerecorded{n}, g_recorded++, 0; }
int shv_prerecorded_submit(shv_ctx *c, shv_prerecorded *, int, uint64_t *ns) { return *ns = 0, c->unwaited = 0; }
int shv_prerecorded_launch(shv_ctx *, shv_prerecorded *) { return 0; }
void shv_prerecorded_destroy(shv_ctx *, shv_prerecorded *p) { delete p; }
int shv_dequant(shv_ctx *, const shv_dequant_args *) { return 0; }
int shv_quantize_q4k(shv_ctx *, const shv_quantize_q4k_args *) { return 0; }
int shv_fill_normal(shv_ctx *, const shv_fill_normal_args *) { return 0; }
int shv_router_fold(shv_ctx *, const shv_router_fold_args *) { return 0; }
int shv_stamp(shv_ctx *, int) { return 0; }
int shv_stamp_elapsed(shv_ctx *, int, int, uint64_t *ns) { return *ns = 0; }
}

namespace {

// a model of four small layers, its graph, and a sequence of six tokens in it
struct Rig {
    std::unique_ptr<llm::Device> dev = std::make_unique<llm::Device>(0);
    std::unique_ptr<llm::Model> model;
    std::unique_ptr<llm::Graph> graph;
    explicit Rig(int nextn = 0) {
        llm::Config c;
        c.NLayer = 4, c.NEmbd = 256, c.NExpert = 4, c.NExpertUsed = 2, c.FFNExpert = 256, c.VocabSize = 512, c.NextN = nextn;
        c.SSMHeadK = 2, c.SSMHeadV = 4, c.NHead = 8, c.NHeadKV = 1;
        model = std::make_unique<llm::Model>(*dev, c);
        llm::GraphOpts o;
        o.NKV = 1024, o.MaxTokens = 16;
        graph = std::make_unique<llm::Graph>(*dev, *model, o);
        graph->Extend({1, 2, 3, 4, 5, 6}, nullptr, static_cast<float *>(nullptr));
    }
    ~Rig() {
        graph.reset();
        model.reset();
        dev.reset();
    }
};

}  // namespace

extern "C" {

// A checkpoint taken, copied, its carry marked, and the first taken again further on: does the copy still hold the mark?
int double_copied_checkpoint() {
    Rig r;
    llm::Checkpoint a;
    r.graph->Checkpoint(a);
    if (!a.on_device) return -1;
    std::memset(a.on_device->ptr, 0x5A, a.on_device->bytes);
    const llm::Checkpoint b = a;
    r.graph->Extend({7, 8}, nullptr, static_cast<float *>(nullptr));
    r.graph->Checkpoint(a);
    const std::vector<float> held = b.on_device->Read();
    for (size_t i = 0; i < held.size() * 4; i++)
        if (reinterpret_cast<const char *>(held.data())[i] != 0x5A) return 0;
    return a.past == 8 && b.past == 6;
}

// One checkpoint taken twice by its own graph: is its memory used again?
int double_own_checkpoint_again() {
    Rig r;
    llm::Checkpoint a;
    r.graph->Checkpoint(a);
    const void *first = a.on_device->ptr;
    r.graph->Checkpoint(a);
    return a.on_device->ptr == first;
}

// Restored by another graph: has that graph finished reading when the call returns, and does it leave the memory alone when it
// takes the checkpoint anew?
int double_restored_elsewhere() {
    Rig r, other;
    llm::Checkpoint a;
    r.graph->Checkpoint(a);
    other.graph->Restore(a);
    if (other.dev->ctx()->unwaited) return 0;
    const int before = g_given;
    other.graph->Checkpoint(a);
    return g_given == before + 1;  // given back, which waits for the device, and other memory taken
}

// A checkpoint that outlives its model: the contexts still there, and a thousand times the allocations beside the checkpoint's own.
int double_checkpoint_outlives_its_model() {
    const size_t before = g_memory.size();
    llm::Checkpoint a;
    {
        Rig r;
        r.graph->Checkpoint(a);
    }
    return g_contexts + 1000 * static_cast<int>(g_memory.size() - before - 1);
}

// A checkpoint on a device with `free_mb` of its 16 GB left: 1 in device memory, 0 whole in host memory, and restored from there.
int double_checkpoint_where_free(int free_mb) {
    Rig r;
    llm::Checkpoint a;
    g_free = static_cast<size_t>(free_mb) << 20;
    r.graph->Checkpoint(a);
    g_free = static_cast<size_t>(16) << 30;
    r.graph->Restore(a);
    return a.on_device ? 1 : a.dn.empty() ? -1 : 0;
}

// The draft's cells over prompts of every length from 1 to 130: how many sequences of ops were recorded for them.
int double_recordings_for_cells() {
    Rig r(1);
    llm::MTPHead head(*r.dev, *r.model, r.graph->Head(), 4, 1024, 1);
    std::vector<float> rows(130 * 256);
    const int before = g_recorded;
    for (int n = 1; n <= 130; n++) {
        head.Reset();
        head.WriteCells(rows.data(), std::vector<int32_t>(n, 7), 0);
        if (head.Past() != n) return -1;
    }
    return g_recorded - before;
}
}
