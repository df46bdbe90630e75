// CPU stand-ins for the C ABI calls a blob converter makes, with queues that run nothing until somebody waits for them:
// compiled together with the host sources by tests/test_converter_queues_cpu.py.  A launch that writes memory of the
// converter's which a launch still waiting in another queue uses, or reads what that one has yet to write, is counted; so is
// page-locked memory that holds something else when a launch reads it than when the launch was made.  Test infrastructure only.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <iterator>
#include <map>
#include <vector>

#include "rocm_device.h"

namespace {
typedef std::pair<const char *, size_t> Range;
struct Op {
    std::vector<Range> reads, writes;
    std::vector<char> had;  // what page-locked memory the launch reads held
};
std::map<void *, std::vector<Op>> g_queues;
std::map<const char *, size_t> g_device, g_host;  // the converter's allocations
int g_conflicts = 0, g_launches = 0, g_device_syncs = 0;

bool Inside(const std::map<const char *, size_t> &m, const void *p) {
    auto it = m.upper_bound((const char *)p);
    return it != m.begin() && (const char *)p < std::prev(it)->first + std::prev(it)->second;
}
bool Overlap(const std::vector<Range> &a, const std::vector<Range> &b) {
    for (auto &x : a)
        for (auto &y : b)
            if (x.first < y.first + y.second && y.first < x.first + x.second)
                return true;
    return false;
}
void Drain(void *q) {
    for (auto &op : g_queues[q])
        if (!op.had.empty())
            g_conflicts += memcmp(op.reads[0].first, op.had.data(), op.had.size()) != 0;
    g_queues[q].clear();
}
Op Make(void *q, const void *src, size_t src_bytes, void *dst, size_t dst_bytes) {
    Op op;
    if (Inside(g_device, src) || Inside(g_host, src))
        op.reads.push_back({(const char *)src, src_bytes});
    if (Inside(g_host, src))
        op.had.assign((const char *)src, (const char *)src + src_bytes);
    if (Inside(g_device, dst))
        op.writes.push_back({(const char *)dst, dst_bytes});
    for (auto &kv : g_queues)
        if (kv.first != q)
            for (auto &other : kv.second)
                g_conflicts += Overlap(op.writes, other.reads) || Overlap(op.writes, other.writes) || Overlap(op.reads, other.writes);
    return op;
}
int Launch(void *q, const void *src, size_t src_bytes, void *dst, size_t dst_bytes) {
    ++g_launches;
    g_queues[q].push_back(Make(q, src, src_bytes, dst, dst_bytes));
    return 0;
}
int Allocate(std::map<const char *, size_t> &m, void **p, size_t bytes) {
    *p = calloc(1, bytes);
    m[(const char *)*p] = bytes;
    return *p ? 0 : 2;
}
}  // namespace

extern "C" {
int tnn_rocm_malloc(void **p, size_t bytes) { return Allocate(g_device, p, bytes); }
int tnn_rocm_malloc_host(void **p, size_t bytes) { return Allocate(g_host, p, bytes); }
int tnn_rocm_device_sync(void *) {
    ++g_device_syncs;
    for (auto &kv : g_queues)
        Drain(kv.first);
    return 0;
}
// freeing waits for the device, as hipFree and hipHostFree do
int tnn_rocm_free(void *p) { return p ? (--g_device_syncs, tnn_rocm_device_sync(nullptr), g_device.erase((const char *)p), free(p), 0) : 0; }
int tnn_rocm_free_host(void *p) { return p ? (--g_device_syncs, tnn_rocm_device_sync(nullptr), g_host.erase((const char *)p), free(p), 0) : 0; }
int tnn_rocm_stream_sync(void *q) { return Drain(q), 0; }
int tnn_rocm_memcpy_h2d(void *dst, const void *src, size_t bytes, void *q) {
    Drain(q);
    Make(q, src, bytes, dst, bytes);
    return memcpy(dst, src, bytes), 0;
}
int tnn_rocm_copy_mapped(void *dst, const void *src, size_t bytes, void *q) { return Launch(q, src, bytes, dst, bytes); }
int tnn_rocm_memcpy_d2d(void *dst, const void *src, size_t bytes, void *q) { return Launch(q, src, bytes, dst, bytes); }
int tnn_rocm_cast(void *q, int, const void *src, int, void *dst, size_t n) { return Launch(q, src, n * 4, dst, n * 2); }
int tnn_rocm_binary(void *q, int, int, const void *, const int *, int, const void *b, const int *bd, int rank, void *y, const int *yd, int) {
    size_t nb = 4, ny = 4;
    for (int i = 0; i < rank; ++i)
        nb *= bd[i], ny *= yd[i];
    return Launch(q, b, nb, y, ny);
}
}

using namespace TNN_NS;

int main() {
    struct Case {
        DataType type;
        DimsVector dims;
        bool scaled, device_mat;
    } cases[] = {
        {DATA_TYPE_FLOAT, {1, 64}, false, false},          // fetched from a page-locked slot
        {DATA_TYPE_HALF, {1, 64}, false, false},           // converted out of a slot
        {DATA_TYPE_HALF, {1, 3, 100, 1000}, false, false}, // converted out of the device staging buffer
        {DATA_TYPE_HALF, {1, 3, 8, 8}, true, true},        // device mat: scaled in the staging buffer, operands in another
    };
    int queues[3], bad = 0;
    for (auto &c : cases) {
        BlobDesc desc;
        desc.name        = "x";
        desc.device_type = DEVICE_ROCM;
        desc.data_type   = c.type;
        desc.dims        = c.dims;
        const size_t n   = (size_t)DimsVectorUtils::Count(c.dims);
        std::vector<char> memory(n * 4);
        BlobHandle handle;
        handle.base = memory.data();
        Blob blob(desc, handle);
        BlobConverter converter(&blob);
        std::vector<std::vector<float>> given;
        for (int i = 0; i < 200; ++i)
            given.push_back(std::vector<float>(n, (float)(i + 1)));
        MatConvertParam param;
        // one queue for some calls, then others in turn, and back
        for (int i = 0; i < (n > 1000 ? 12 : 200); ++i) {
            Mat mat(c.device_mat ? DEVICE_ROCM : DEVICE_NAIVE, NCHW_FLOAT, c.dims, given[i].data());
            if (c.scaled)
                param.scale = {(float)i, 2.f, 3.f}, param.bias = {1.f, (float)i, 0.f};
            void *q   = &queues[i % 20 == 3 ? 1 : i % 7 == 5 ? 2 : 0];
            Status st = converter.ConvertFromMatAsync(mat, param, q);
            if (st != TNN_OK) {
                printf("conversion failed: %s\n", st.description().c_str());
                return 2;
            }
        }
        tnn_rocm_device_sync(nullptr);
        printf("type %d, %zu elements: launches %d, conflicts %d\n", (int)c.type, n, g_launches, g_conflicts);
        bad += g_conflicts + (g_launches == 0);
        g_conflicts = g_launches = 0;
    }
    // a program that keeps to one queue is never made to wait for the device
    g_device_syncs = 0;
    BlobDesc desc;
    desc.name = "y", desc.device_type = DEVICE_ROCM, desc.data_type = DATA_TYPE_FLOAT, desc.dims = {1, 64};
    std::vector<float> memory(64), value(64, 1.f);
    BlobHandle handle;
    handle.base = memory.data();
    Blob blob(desc, handle);
    BlobConverter converter(&blob);
    for (int i = 0; i < 50; ++i) {
        Mat mat(DEVICE_NAIVE, NCHW_FLOAT, desc.dims, value.data());
        converter.ConvertFromMatAsync(mat, MatConvertParam(), &queues[0]);
    }
    tnn_rocm_stream_sync(&queues[0]);
    printf("one queue: device syncs %d, conflicts %d\n", g_device_syncs, g_conflicts);
    return bad || g_device_syncs || g_conflicts ? 1 : 0;
}
