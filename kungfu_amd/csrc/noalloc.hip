// kf_hip_matmul_noalloc: kf_hip_matmul for callers that cannot allocate device memory (code under HIP graph capture,
// tight serving loops, harnesses that forbid hipMalloc). The activation scratch that kf_hip_matmul takes as an
// argument is instead a file-scope device array of KF_NOALLOC_SCRATCH_BYTES, one copy per GPU, held until the process
// ends. No reference counterpart.
//
// In host code the array's name is only a host-side stand-in, not a device address: every host use goes through the
// device address that hipGetSymbolAddress returns, looked up once per device (with that device current) on the
// device's first call and kept per device.
#include "kf_host.h"
#include "kf_knobs.h"
#include <hip/hip_runtime.h>

#include <algorithm>
#include <deque>
#include <mutex>
#include <set>
#include <vector>

#include "../../include/kf_hip.h"
#include "kf_layout.h"

void kf_set_error(const char* fmt, ...);

namespace {

static __device__ __align__(256) uint8_t scratch[KF_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;

// The device address of `scratch` on `dev` (looked up on first use), or nullptr with the error recorded
void* scratch_ptr(int dev) {
    static std::mutex mu;
    static void* ptr[kMaxDevices] = {};
    if (dev < 0 || dev >= kMaxDevices) {
        kf_set_error("device %d: at most %d devices", dev, kMaxDevices);
        return nullptr;
    }
    std::lock_guard<std::mutex> g(mu);
    if (!ptr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            kf_set_error("hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
            (void)hipGetLastError();  // the failure is reported here, not by the next launch's error check
            return nullptr;
        }
        ptr[dev] = p;
    }
    return ptr[dev];
}

}  // namespace

extern "C" size_t kf_hip_noalloc_scratch_bytes(void) { return KF_NOALLOC_SCRATCH_BYTES; }

extern "C" int kf_hip_matmul_noalloc(uint32_t ty, const void* w, int n_in, int n_out, const float* x, int rows, const float* bias,
                                     const float* res, float* y, void* stream) {
    if (rows < 0 || n_in <= 0) {
        kf_set_error("%d rows of %d columns", rows, n_in);
        return KF_E_INVALID;
    }
    const size_t need = kf_hip_act_bytes(rows, n_in);
    if (need > KF_NOALLOC_SCRATCH_BYTES) {
        kf_set_error("%d rows of %d columns need %zu bytes of activation scratch, the no-allocation entry point holds %zu", rows, n_in, need,
                     (size_t)KF_NOALLOC_SCRATCH_BYTES);
        return KF_E_INVALID;
    }
    int dev = 0;
    const hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        kf_set_error("hipGetDevice: %s", hipGetErrorString(e));
        return KF_E_HIP;
    }
    void* act = scratch_ptr(dev);
    if (!act) return KF_E_HIP;
    // quant_act writes every byte of the scratch that the product reads, so nothing is cleared between calls
    return kf_hip_matmul(ty, w, n_in, n_out, x, rows, act, bias, res, y, stream);
}

// ------------------------------------------------------------------------------------------------ split-K scratch
// The split products' partial tiles and tickets (kf_host.h): static, so nothing is allocated and the addresses never
// change. Each device has its own copy, found with hipGetSymbolAddress once per device. Stream slots go to (device,
// stream) pairs on first use and come back through kf_hip_release_stream. A stream under graph capture gets the
// graph slot instead: a captured graph keeps the address it recorded and may be replayed on any stream, so it must
// never share a slot with direct launches, which hold stream slots only.
// Within one capture the slot goes from product to product only along the graph's own order: the nodes recorded at the
// end of the last product that used it have to be ancestors of the next one. Branches forked over several streams of
// a capture run at the same time in a replay, and two products there would write over each other's partials.
static __device__ __align__(256) uint8_t split_scratch[KF_SPLIT_SLOTS * KF_SPLIT_SCRATCH + KF_SPLIT_SPARES * KF_SPLIT_SPARE];

namespace {
// A capture that has used the graph slot: its id, the nodes its last use ended with, and whether a product of it is
// being recorded right now
struct GraphUse {
    unsigned long long id;
    bool busy;
    std::vector<hipGraphNode_t> last;
};
constexpr size_t KF_GRAPH_USES = 64;  // captures remembered per device; more of them at once are not expected

std::mutex g_split_mu;
std::map<int, uint8_t*> g_split_base;                       // per device

// Slots given to (device, stream) pairs
struct SlotPool {
    int count;
    std::map<std::pair<int, hipStream_t>, int> held;
    std::map<int, unsigned> taken;  // per device: bit i set when slot i is held

    // the stream's slot, a free one if it has none yet; -1: every one is held by another stream
    int take(int dev, hipStream_t s) {
        const auto it = held.find({dev, s});
        if (it != held.end()) return it->second;
        unsigned& t = taken[dev];
        for (int i = 0; i < count; i++)
            if (!(t & (1u << i))) {
                t |= 1u << i;
                held[{dev, s}] = i;
                return i;
            }
        return -1;
    }
    void give_back(int dev, hipStream_t s) {
        const auto it = held.find({dev, s});
        if (it == held.end()) return;
        taken[dev] &= ~(1u << it->second);
        held.erase(it);
    }
};
SlotPool g_stream_slots{KF_SPLIT_STREAM_SLOTS, {}, {}}, g_spare_slots{KF_SPLIT_SPARES, {}, {}};
std::map<int, std::deque<GraphUse>> g_graph_uses;           // per device, the newest last

// A stream's capture: its id and the nodes that whatever it records next will depend on
bool capture_front(hipStream_t s, unsigned long long* id, std::vector<hipGraphNode_t>* front) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    const hipGraphNode_t* deps = nullptr;
    size_t n = 0;
    if (hipStreamGetCaptureInfo_v2(s, &cs, id, nullptr, &deps, &n) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if (cs != hipStreamCaptureStatusActive) return false;
    front->assign(deps, deps + (deps ? n : 0));
    return true;
}

// Whether every node of `want` is in `front` or an ancestor of it. The search goes breadth first from the front: in a
// capture on one stream the last use lies a few nodes back.
bool all_before(const std::vector<hipGraphNode_t>& want, const std::vector<hipGraphNode_t>& front) {
    std::set<hipGraphNode_t> left(want.begin(), want.end()), seen(front.begin(), front.end());
    std::deque<hipGraphNode_t> at(front.begin(), front.end());
    std::vector<hipGraphNode_t> deps;
    while (!left.empty() && !at.empty()) {
        const hipGraphNode_t node = at.front();
        at.pop_front();
        left.erase(node);
        size_t n = 0;
        if (hipGraphNodeGetDependencies(node, nullptr, &n) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        if (n == 0) continue;
        deps.resize(n);
        if (hipGraphNodeGetDependencies(node, deps.data(), &n) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        for (size_t i = 0; i < n; i++)
            if (seen.insert(deps[i]).second) at.push_back(deps[i]);
    }
    return left.empty();
}

// The slot for a product on `s`, null if there is none for it. `take`: the product is launched next (under capture the
// slot is then busy until split_done).
void* split_slot(hipStream_t s, bool graph, bool take, bool* capturing) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cs) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    *capturing = cs != hipStreamCaptureStatusNone;
    if (*capturing && (!graph || kf_knob_on(KF_KNOB_CAPTURE_NO_SPLIT))) return nullptr;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    std::lock_guard<std::mutex> g(g_split_mu);
    auto b = g_split_base.find(dev);
    if (b == g_split_base.end()) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(split_scratch)) != hipSuccess || !p) {
            (void)hipGetLastError();
            return nullptr;
        }
        b = g_split_base.emplace(dev, static_cast<uint8_t*>(p)).first;
    }
    if (*capturing) {
        unsigned long long id = 0;
        std::vector<hipGraphNode_t> front;
        if (!capture_front(s, &id, &front)) return nullptr;
        auto& uses = g_graph_uses[dev];
        auto u = std::find_if(uses.begin(), uses.end(), [&](const GraphUse& x) { return x.id == id; });
        if (u != uses.end() && (u->busy || !all_before(u->last, front))) return nullptr;
        if (take) {
            if (u == uses.end()) {
                if (uses.size() == KF_GRAPH_USES) uses.pop_front();
                uses.push_back(GraphUse{id, true, {}});
            } else {
                u->busy = true;
            }
        }
        return b->second + (size_t)KF_SPLIT_STREAM_SLOTS * KF_SPLIT_SCRATCH;
    }
    const bool main = graph || g_stream_slots.held.count({dev, s});
    const int i = (main ? g_stream_slots : g_spare_slots).take(dev, s);
    if (i < 0) return nullptr;  // every slot held by another stream: the scratch-free form
    return b->second + (main ? i * KF_SPLIT_SCRATCH : KF_SPLIT_SLOTS * KF_SPLIT_SCRATCH + i * KF_SPLIT_SPARE);
}
}  // namespace

KfSplit::KfSplit(hipStream_t s, bool graph) : stream_(s), capturing_(false), p_(static_cast<char*>(split_slot(s, graph, true, &capturing_))) {}

bool KfSplit::ready(hipStream_t s, bool graph) {
    bool capturing = false;
    return split_slot(s, graph, false, &capturing) != nullptr;
}

// Under capture: the product is recorded, its nodes are the slot's last use. Where they cannot be read the slot stays
// busy, and the rest of this capture runs without it.
KfSplit::~KfSplit() {
    if (!p_ || !capturing_) return;
    int dev = 0;
    unsigned long long id = 0;
    std::vector<hipGraphNode_t> front;
    if (hipGetDevice(&dev) != hipSuccess || !capture_front(stream_, &id, &front)) {
        (void)hipGetLastError();
        return;
    }
    std::lock_guard<std::mutex> g(g_split_mu);
    for (GraphUse& u : g_graph_uses[dev])
        if (u.id == id) {
            u.last = front;
            u.busy = false;
        }
}

extern "C" int kf_hip_release_stream(void* stream) {
    const hipStream_t s = static_cast<hipStream_t>(stream);
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        kf_set_error("hipGetDevice: %s", hipGetErrorString(e));
        return KF_E_HIP;
    }
    std::lock_guard<std::mutex> g(g_split_mu);
    if (!g_stream_slots.held.count({dev, s}) && !g_spare_slots.held.count({dev, s})) return KF_OK;
    // a slot is free only once the stream's products that use it have ended
    e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
        kf_set_error("hipStreamSynchronize: %s", hipGetErrorString(e));
        return KF_E_HIP;
    }
    g_stream_slots.give_back(dev, s);
    g_spare_slots.give_back(dev, s);
    return KF_OK;
}
