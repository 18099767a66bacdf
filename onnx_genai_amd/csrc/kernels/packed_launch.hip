// One launch for the nodes of a recorded step that read the same activations.
//
// A stream capture records the calls of one stream as a chain, so each node of a step waits for the one before it, though the step's data
// asks for less: q, k and v read one input, and so do gate and up of a model that was exported without fused nodes. A launch that depends on another costs
// about 2 us before it has read a byte, more than half the time of such a node of a 0.5B model.
// A node that could run beside the one recorded just before it is therefore not recorded as a launch of its own: it becomes a further row of that launch's
// grid, with its own columns, bias and result; every row is as long as the widest node's, and workgroups beyond a row's columns read nothing. Each keeps its own split of K, so its sums are those of a launch by itself, bit for bit.
// 24 layers of a 0.5B model at one row, f16, block 32: 169 launches 585 us, 97 launches 393.
// What may join: the capture's only open end is the launch recorded last (anything recorded in between, by whomever, is another end); the same kernel
// build, activations, rows, K, split of K and result type; and no result of one that is an input or a result of the other.
// A node that cannot join still gets something out of the launch before it, where that one is short (its own weights are few, and waiting for them is
// what it does): further rows of its grid read the first weights of the new node ahead (weights_ahead.hiph).
// The recorded node gets new arguments and a larger grid while the capture is open (hipGraphKernelNodeSetParams), so the graph is complete after every call
// and nothing is left to do when the capture ends.
#include <mutex>
#include <new>

#include "packed_launch.hiph"

struct RocmStepTail {
    std::mutex mu;
    unsigned long long capture = 0;
    hipGraphNode_t node = nullptr;          // NULL: nothing to join
    mnb::PackedLaunch launch;               // as it stands in `node`
    hipGraphNode_t before = nullptr;        // the launch in front of it, if that reads its weights ahead
    mnb::PackedLaunch before_launch;
};

namespace mnb {
namespace {

// The one node that the next operation on `stream` would depend on.
bool open_end(hipStream_t stream, unsigned long long* capture, hipGraphNode_t* node)
{
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    const hipGraphNode_t* ends = nullptr;
    size_t count = 0;
    if (hipStreamGetCaptureInfo_v2(stream, &status, capture, nullptr, &ends, &count) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if (status != hipStreamCaptureStatusActive || count != 1) return false;
    *node = ends[0];
    return true;
}

struct Range {
    uintptr_t begin, end;
};
bool meet(const Range& a, const Range& b) { return a.begin < b.end && b.begin < a.end; }
Range range(const void* p, int64_t elements, int dtype)
{
    const uintptr_t at = reinterpret_cast<uintptr_t>(p);
    return p ? Range{at, at + static_cast<uintptr_t>(elements) * (dtype == ROCM_DT_F32 ? 4 : 2)} : Range{0, 0};
}
Range result(const PackedParams& p, const PackedNode& node) { return range(node.y, static_cast<int64_t>(p.m) * node.n, p.rest.y_dtype); }
Range bias(const PackedParams& p, const PackedNode& node)
{
    return range(node.bias, (node.bias_dtype & ROCM_BIAS_PER_ROW) ? static_cast<int64_t>(p.m) * node.n : node.n, node.bias_dtype & 0xff);
}

// `to` with the node of `add` as a further row, or false: they do not go together.
bool joined(const PackedLaunch& to, const PackedLaunch& add, PackedLaunch* out)
{
    const PackedParams &p = to.p, &q = add.p;
    const uint32_t one = 1u << 24;                         // (the rows so far)
    if (to.nodes < 1 || to.nodes == kMaxNodes || add.nodes != 1 || to.kernel != add.kernel || to.threads != add.threads || to.lds != add.lds) return false;
    if (p.a != q.a || p.m != q.m || p.k != q.k || p.groups != q.groups || p.split != q.split + (to.nodes - 1) * one || p.rest.y_dtype != q.rest.y_dtype) return false;
    const PackedNode& node = q.rest.nodes[0];
    const Range a = range(q.a, static_cast<int64_t>(q.m) * q.k, ROCM_DT_F16), y = result(q, node), b = bias(q, node);
    if (meet(y, a)) return false;
    for (int i = 0; i < to.nodes; ++i) {
        const Range other = result(p, p.rest.nodes[i]);
        if (meet(y, other) || meet(a, other) || meet(b, other) || meet(y, bias(p, p.rest.nodes[i]))) return false;
    }
    *out = to;
    if (to.nodes == 1) {
        out->p.packed_up = node.packed;
        out->p.n_up = node.n;
    }
    out->p.rest.nodes[out->nodes++] = node;
    out->p.split += one;
    if (out->grid < add.grid) out->grid = add.grid;
    // every row of the grid is as long as the widest node's: not where the workgroups without columns would be most of many
    int64_t busy = 0;
    for (int i = 0; i < out->nodes; ++i) busy += (static_cast<int64_t>(out->p.rest.nodes[i].n) + 15) / 16;
    return static_cast<int64_t>(out->grid) * out->nodes <= 2 * busy + 512;
}

// Launches that read no more weights than this leave the memory idle for long enough to read the next one's, up to this many together (bytes, as in
// swiglu.hip: the memory's rate and the size of the near caches set them). Steps of a 0.5B model at
// one row and of a 7B model at one / 16 rows: 392, 1,117 / 1,538 us with nothing read ahead here, 388, 1,115 / 1,527 with launches of at most 1 MB, 387, 1,114 / 1,528 of
// 5 MB, 383, 1,112 / 1,527 of 10 MB; 14, 18 or 22 MB together are level to 0.5 %.
constexpr uint64_t kShortLaunch = 10000000, kAheadTogether = 18000000;

uint64_t bytes_read(const PackedLaunch& l)
{
    uint64_t columns = 0;
    for (int i = 0; i < (l.nodes > 1 ? l.nodes : 1); ++i) columns += (static_cast<uint64_t>(l.p.rest.nodes[i].n) + 15) / 16;
    return columns * l.stream;
}

unsigned grid_rows(const PackedLaunch& l)
{
    const unsigned rows = l.p.rows();
    const WeightsAhead& w = l.p.rest.ahead;
    if (w.workgroups == 0) return rows;
    const uint64_t blocks = w.from + static_cast<uint64_t>(w.workgroups) * w.parts * (w.second ? 2 : 1);
    return static_cast<unsigned>((blocks + l.grid - 1) / l.grid);
}

// `before` with the first weights of `next` read ahead, or false.
bool reads_ahead(const PackedLaunch& before, const PackedLaunch& next, PackedLaunch* out)
{
    const uint64_t own = bytes_read(before);
    if (!before.carries || next.stream == 0 || own > kShortLaunch) return false;
    RocmWeightsAhead ahead{};
    ahead.first = next.p.packed;
    ahead.second = next.nodes > 1 && next.grid % kXcds == 0 ? next.p.packed_up : nullptr;      // (its workgroups lie on the same XCDs then)
    ahead.bytes = next.stream;
    ahead.workgroups = next.grid;
    for (int i = 0; i < (ahead.second ? 2 : 1); ++i) {
        const uint32_t columns = (static_cast<uint32_t>(next.p.rest.nodes[i].n) + 15u) / 16u;
        if (columns < ahead.workgroups) ahead.workgroups = columns;
    }
    *out = before;
    (void)plan_weights_ahead(ahead, kAheadTogether - own, before.threads, before.p.rows() * before.grid, before.grid, &out->p.rest.ahead);
    return out->p.rest.ahead.workgroups != 0 && grid_rows(*out) <= 65535;
}

// The launch of `nodes`, as one after the other would be recorded.
bool launch_of(const RocmStepNodes& nodes, PackedLaunch* out)
{
    for (int i = 0; i < nodes.nodes; ++i) {
        PackedLaunch one{};
        one.p.packed = static_cast<const uint8_t*>(nodes.packed[i]);
        one.p.n = nodes.columns[i];
        one.p.split = 1u << 24;
        one.p.rest.nodes[0] = PackedNode{nullptr, nullptr, one.p.packed, one.p.n, ROCM_DT_F32};
        one.grid = (static_cast<unsigned>(one.p.n) + 15u) / 16u;
        one.threads = nodes.threads;
        one.carries = true;
        one.nodes = 1;
        one.stream = nodes.stream;
        const PackedLaunch before = *out;
        if (i == 0) *out = one;
        else if (!joined(before, one, out)) return false;
    }
    return true;
}

}  // namespace

int start_packed(const PackedLaunch& launch, hipStream_t stream, RocmStepTail* tail)
{
    auto arguments = [](PackedParams& p, void* (&to)[11]) {
        void* const all[11] = {&p.a, &p.packed, &p.packed_up, &p.gamma, &p.m, &p.k, &p.n, &p.n_up, &p.groups, &p.split, &p.rest};
        for (int i = 0; i < 11; ++i) to[i] = all[i];
    };
    void* args[11];
    auto alone = [&] {
        PackedParams p = launch.p;
        arguments(p, args);
        return static_cast<int>(hipLaunchKernel(launch.kernel, dim3(launch.grid), dim3(launch.threads), args, launch.lds, stream));
    };
    if (!tail) return alone();
    std::lock_guard<std::mutex> lock(tail->mu);
    unsigned long long capture = 0;
    hipGraphNode_t node = nullptr;
    // What a recorded node launches becomes `l`; on failure it is what it was.
    auto replaced = [&](hipGraphNode_t at, PackedLaunch& l) {
        arguments(l.p, args);
        hipKernelNodeParams params{};
        params.func = const_cast<void*>(l.kernel);
        params.gridDim = dim3(l.grid, grid_rows(l));
        params.blockDim = dim3(l.threads);
        params.sharedMemBytes = static_cast<unsigned>(l.lds);
        params.kernelParams = args;
        if (hipGraphKernelNodeSetParams(at, &params) == hipSuccess) return true;
        (void)hipGetLastError();
        return false;
    };
    const bool behind = tail->node && open_end(stream, &capture, &node) && capture == tail->capture && node == tail->node;
    PackedLaunch changed;
    if (behind && joined(tail->launch, launch, &changed) && replaced(node, changed)) {
        tail->launch = changed;
        if (changed.nodes == 2 && tail->before && reads_ahead(tail->before_launch, tail->launch, &changed)) (void)replaced(tail->before, changed);
        return 0;
    }
    tail->before = nullptr;
    if (behind && reads_ahead(tail->launch, launch, &changed) && replaced(node, changed)) {
        tail->before = node;
        tail->before_launch = tail->launch;                // (without what it reads ahead)
    }
    tail->node = nullptr;
    const int rc = alone();
    if (rc == 0 && open_end(stream, &capture, &node)) {
        tail->capture = capture;
        tail->node = node;
        tail->launch = launch;
    }
    return rc;
}

}  // namespace mnb

extern "C" RocmStepTail* rocm_step_tail_create(void) { return new (std::nothrow) RocmStepTail(); }
extern "C" void rocm_step_tail_destroy(RocmStepTail* tail) { delete tail; }
extern "C" void rocm_step_tail_reset(RocmStepTail* tail)
{
    if (!tail) return;
    std::lock_guard<std::mutex> lock(tail->mu);
    tail->node = tail->before = nullptr;
}
extern "C" int rocm_step_reads(const RocmStepNodes* nodes, const RocmStepNodes* next, uint32_t x, uint32_t y, RocmStepReads* out)
{
    mnb::PackedLaunch launch{}, behind{}, changed{};
    auto shared = [](const RocmStepNodes* of, mnb::PackedLaunch* to) { return of->nodes >= 1 && of->nodes <= mnb::kMaxNodes && mnb::launch_of(*of, to); };
    if (!shared(nodes, &launch) || (next && !shared(next, &behind))) return -1;
    if (next && mnb::reads_ahead(launch, behind, &changed)) launch = changed;
    const mnb::PackedParams& p = launch.p;
    *out = RocmStepReads{launch.grid, mnb::grid_rows(launch), p.rest.ahead.workgroups, 0, 0};
    if (x >= out->grid || y >= out->rows) return -1;
    if (y >= p.rows()) {                                                                       // (rows as the kernel tells them apart)
        mnb::ahead_range(p.rest.ahead, y * p.rest.ahead.grid + x, launch.threads, &out->first, &out->bytes);
        return 0;
    }
    const int n = y == 0 ? p.n : y == 1 ? p.n_up : p.rest.nodes[y].n;
    const uint8_t* const packed = y == 0 ? p.packed : y == 1 ? p.packed_up : p.rest.nodes[y].packed;
    if (!mnb::has_columns(x, n)) return 0;
    out->first = reinterpret_cast<uintptr_t>(packed) + static_cast<uint64_t>(x) * launch.stream;
    out->bytes = launch.stream;
    return 0;
}

extern "C" uint64_t rocm_weights_ahead_reads(const RocmWeightsAhead* next, uint64_t budget, uint32_t threads, uint32_t blocks, uint32_t block, RocmStepReads* out)
{
    mnb::WeightsAhead w;
    const uint64_t all = mnb::plan_weights_ahead(*next, budget, threads, blocks, 0, &w);
    *out = RocmStepReads{0, 0, w.workgroups, 0, 0};
    mnb::ahead_range(w, block, threads, &out->first, &out->bytes);
    return all;
}
