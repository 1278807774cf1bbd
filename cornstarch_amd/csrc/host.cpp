// Host side of the attention entry points in native code: argument checks, the caches of the last mask's flags and plan,
// output allocation, the autograd node and the calls into libbam_hip.so.  Python keeps the public functions and whatever
// is not in the usual form (other layouts, head dims that are no multiple of 8, error reporting): every function here answers
// None for those and the caller takes its general path.
//
// Why native: a short forward + backward (2 x 283 tokens) kept the GPU busy for 84 us but took 300 us in Python (now 75) --
// argument marshalling through ctypes, an event and a copy on a side stream for the plan's pair count, and a Python
// autograd function whose backward runs on the engine's thread.
#include <torch/extension.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/Exceptions.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <sched.h>

#include <atomic>
#include <cmath>
#include <mutex>
#include <vector>

#include "../../include/bam_hip.h"

namespace py = pybind11;
using at::Tensor;
using c10::optional;
using torch::autograd::variable_list;

namespace {

struct BamFailure : std::runtime_error {
    using std::runtime_error::runtime_error;
};

void check(int rc, const char* what) {
    if (rc != BAM_OK)
        throw BamFailure(std::string(what) + " failed (" + std::to_string(rc) + "): " + bam_last_error());
}

typedef c10::hip::HIPStream Stream;
Stream current_stream(c10::Device device) { return c10::hip::getCurrentHIPStream(device.index()); }
bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }

// ------------------------------------------------------------------ pair counts
// The number of pairs of a plan is device data; the last launch of the plan builder stores it, under a tag, to a word of
// pinned host memory that belongs to the plan, and a backward that needs it polls that word.  A word goes back to the
// pool once its value has arrived (or, if nobody waited for it, once a later look finds it there), so a late store can
// never land in a word that has a new owner.
class CountWords {
public:
    struct Word {
        uint64_t* at = nullptr;
        uint32_t tag = 0;
    };
    Word take() {
        std::lock_guard<std::mutex> hold(mutex_);
        sweep();
        if (free_.empty()) {
            uint64_t* slab = nullptr;
            check(bam_host_words_alloc(&slab, kSlab), "bam_host_words_alloc");
            slabs_.push_back(slab);
            for (int i = 0; i < kSlab; ++i) free_.push_back(slab + i);
        }
        Word w{free_.back(), ++tag_ == 0 ? ++tag_ : tag_};
        free_.pop_back();
        return w;
    }
    void give_back(Word w, bool arrived) {
        std::lock_guard<std::mutex> hold(mutex_);
        if (arrived || has_arrived(w))
            free_.push_back(w.at);
        else
            pending_.push_back(w);
    }
    static bool has_arrived(const Word& w) { return (uint32_t)(__atomic_load_n(w.at, __ATOMIC_ACQUIRE) >> 32) == w.tag; }
    // every word back in the pool: the memory can go (process end)
    void release() {
        std::lock_guard<std::mutex> hold(mutex_);
        sweep();
        if (free_.size() != slabs_.size() * kSlab) return;
        for (uint64_t* s : slabs_) bam_host_words_free(s);
        slabs_.clear();
        free_.clear();
    }

private:
    static constexpr int kSlab = 256;
    void sweep() {
        for (size_t i = 0; i < pending_.size();)
            if (has_arrived(pending_[i])) {
                free_.push_back(pending_[i].at);
                pending_[i] = pending_.back();
                pending_.pop_back();
            } else {
                ++i;
            }
    }
    std::mutex mutex_;
    std::vector<uint64_t*> slabs_, free_;
    std::vector<Word> pending_;
    uint32_t tag_ = 0;
};
CountWords& count_words() {
    static CountWords* w = new CountWords;  // never destroyed: plans may outlive static destruction
    return *w;
}

// ------------------------------------------------------------------ plan
struct PlanCore {
    Tensor workspace, flags;
    int64_t flags_version = -1;
    bam_plan plan = {};
    CountWords::Word word;
    optional<Stream> stream;  // where the builder was launched
    std::atomic<int64_t> pairs{-1};
    std::atomic<int32_t> rows_known{BAM_ROWS_UNKNOWN};

    PlanCore() = default;
    PlanCore(const PlanCore&) = delete;
    ~PlanCore() {
        if (word.at != nullptr) count_words().give_back(word, pairs.load() >= 0);
    }
    // Not while capturing: every replay would store to the word again, whoever owns it by then, and the caches would hold
    // a plan that nothing has computed yet.  A plan built before the capture is used in it like any other.
    void prepare(Tensor ws, Stream s) {
        if (capturing()) throw BamFailure("a plan cannot be built while a graph is captured: run the call once before");
        workspace = std::move(ws);
        stream = s;
        word = count_words().take();
    }
    // a launch of the builder failed: whether the word will be written is unknown, so it is never handed out again
    void abandon() { word.at = nullptr; }
    // waits for the value; call without the GIL
    int64_t wait_pairs() {
        if (pairs.load() >= 0) return pairs.load();
        if (word.at == nullptr) throw BamFailure("the plan has no pair count");
        for (int64_t n = 0; !CountWords::has_arrived(word); ++n) {
            if (n < 4096) {
                __builtin_ia32_pause();
                continue;
            }
            sched_yield();
            // the stream has run dry and the value is still not there: its launch failed
            if (n % 4096 == 0 && stream->query() && !CountWords::has_arrived(word))
                throw BamFailure("the pair count of a plan never arrived");
        }
        look();
        return pairs.load();
    }
    // takes the value if it is there
    void look() {
        if (pairs.load() >= 0 || word.at == nullptr || !CountWords::has_arrived(word)) return;
        const uint32_t value = (uint32_t)__atomic_load_n(word.at, __ATOMIC_ACQUIRE);
        const bool sorted = plan.rows != nullptr, moved = sorted && value >> 31, left = sorted && (value >> 30 & 1);
        rows_known.store(moved && !left ? BAM_ROWS_MOVED : left && !moved ? BAM_ROWS_LEFT : BAM_ROWS_UNKNOWN);
        pairs.store(sorted ? value & 0x3FFFFFFFu : value);
    }
};

// A Python object held by native state that may be destroyed on any thread.
std::shared_ptr<PyObject> hold(const py::object& o) {
    return std::shared_ptr<PyObject>(py::object(o).release().ptr(), [](PyObject* p) {
        if (!Py_IsInitialized() || _Py_IsFinalizing()) return;  // (a thread that asks for the lock then is ended where it stands)
        py::gil_scoped_acquire gil;
        Py_DECREF(p);
    });
}

PyObject* g_plan_type = nullptr;   // Python's subclass of PlanCore
PyObject* g_error_type = nullptr;  // Python's BamError

struct Plan {  // a plan and the Python object it lives in
    std::shared_ptr<PlanCore> core;
    std::shared_ptr<PyObject> obj;
    explicit operator bool() const { return (bool)core; }
    py::object py_object() const { return obj ? py::reinterpret_borrow<py::object>(obj.get()) : py::none(); }
};
Plan new_plan() {
    py::object o = py::reinterpret_borrow<py::object>(g_plan_type)();
    return Plan{o.cast<std::shared_ptr<PlanCore>>(), hold(o)};
}
Plan plan_of(const py::object& o) {
    if (o.is_none()) return {};
    return Plan{o.cast<std::shared_ptr<PlanCore>>(), hold(o)};
}

void hip_check(hipError_t e, const char* what) {
    if (e == hipSuccess) return;
    (void)hipGetLastError();
    throw BamFailure(std::string(what) + ": " + hipGetErrorString(e));
}

// What one call computed and a later one may find again (flags, plan, gathered index arrays), and the stream that computes it.  A
// later call on that stream just uses it.  On another one it first waits for an event behind the launches, and the caching allocator
// learns that this stream uses the memory too.  An event costs the stream it is recorded on 4.7 us, so it is recorded when the first
// such call asks; a stream that torch does not own may be gone by then, or share its handle with another, and gets it at once.
// A call under capture makes the graph an owner: its replays read the results after the caches have moved on.
class Prepared : public std::enable_shared_from_this<Prepared> {
    typedef std::shared_ptr<Prepared> Held;

public:
    // after the launches
    Prepared(Stream stream, std::vector<Tensor> results, std::shared_ptr<PlanCore> plan)
        : stream_(stream), results_(std::move(results)), plan_(std::move(plan)) {
        if (plan_) results_.push_back(plan_->workspace);
        if (external()) record();
    }
    Prepared(const Prepared&) = delete;
    ~Prepared() {
        if (event_ != nullptr) (void)hipEventDestroy(event_);
    }
    // Call before the results are used on the current stream.  False: they cannot be, the caller has to compute its own.
    bool use() {
        const Stream now = current_stream(stream_.device());
        const bool captured = now.stream() != nullptr && capturing(), elsewhere = now != stream_ || external();
        if (!captured && !elsewhere) return true;
        const std::lock_guard<std::mutex> lock(mutex_);
        if (elsewhere && !done_) {
            const c10::DeviceGuard guard(stream_.device());
            const c10::hip::HIPStreamCaptureModeGuard relaxed(hipStreamCaptureModeRelaxed);
            if (event_ == nullptr) {
                hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
                if (stream_.stream() != nullptr) hip_check(hipStreamIsCapturing(stream_.stream(), &status), "state of a stream");
                if (status != hipStreamCaptureStatusNone) return false;  // (the event would become part of that graph)
                record();
            }
            if (captured) {  // (replays run on any stream: the results are there before the capture goes on)
                hip_check(hipEventSynchronize(event_), "wait for a plan");
                done_ = true;
            } else if (hipEventQuery(event_) == hipSuccess) {
                done_ = true;
            } else {
                (void)hipGetLastError();
                hip_check(hipStreamWaitEvent(now.stream(), event_, 0), "wait for a plan");
            }
        }
        if (captured)
            give_to_graph(now);
        else
            for (const Tensor& t : results_) t.record_stream(c10::Stream::unpack3(now.id(), now.device_index(), c10::DeviceType::CUDA));
        return true;
    }
    // What graphs that are gone owned.  (The runtime lets go of it where the last graph is destroyed, under its own locks: there
    // the reference only changes hands.)
    static void collect() {
        std::vector<Held*> gone;
        {
            const std::lock_guard<std::mutex> lock(dropped_mutex());
            gone.swap(dropped());
        }
        for (Held* h : gone) delete h;
    }
    static int64_t held_by_graphs() { return held_.load(); }

private:
    // (the id of a stream of torch's own is not its handle, except for the default stream, whose handle is null)
    bool external() const { return stream_.stream() != nullptr && stream_.id() == reinterpret_cast<int64_t>(stream_.stream()); }
    void record() {
        const c10::DeviceGuard guard(stream_.device());
        hip_check(hipEventCreateWithFlags(&event_, hipEventDisableTiming), "event behind a plan");
        hip_check(hipEventRecord(event_, stream_.stream()), "event behind a plan");
    }
    static std::mutex& dropped_mutex() {
        static std::mutex* m = new std::mutex;  // never destroyed: a graph may outlive static destruction
        return *m;
    }
    static std::vector<Held*>& dropped() {
        static auto* v = new std::vector<Held*>;
        return *v;
    }
    static void drop(void* held) {
        const std::lock_guard<std::mutex> lock(dropped_mutex());
        dropped().push_back(static_cast<Held*>(held));
        --held_;
    }
    // The graph that `stream` is being captured into, and what is instantiated from it, own a reference through a user object.
    void give_to_graph(const Stream& stream) {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        unsigned long long id = 0;
        hipGraph_t graph = nullptr;
        hip_check(hipStreamGetCaptureInfo_v2(stream.stream(), &status, &id, &graph, nullptr, nullptr), "graph of a capture");
        if (graph == graph_ && id == capture_) return;
        auto held = std::make_unique<Held>(shared_from_this());
        hipUserObject_t owner = nullptr;
        hip_check(hipUserObjectCreate(&owner, held.get(), &Prepared::drop, 1, hipUserObjectNoDestructorSync), "owner of a plan");
        held.release();
        ++held_;
        const hipError_t e = hipGraphRetainUserObject(graph, owner, 1, hipGraphUserObjectMove);
        if (e != hipSuccess) (void)hipUserObjectRelease(owner, 1);
        hip_check(e, "owner of a plan");
        graph_ = graph;
        capture_ = id;
    }
    static inline std::atomic<int64_t> held_{0};
    const Stream stream_;
    std::vector<Tensor> results_;
    const std::shared_ptr<PlanCore> plan_;
    std::mutex mutex_;
    hipEvent_t event_ = nullptr;
    bool done_ = false;
    hipGraph_t graph_ = nullptr;  // the last one that became an owner, and its capture
    unsigned long long capture_ = 0;
};

// ------------------------------------------------------------------ caches (one entry each; guarded by the GIL)
// An entry belongs to the very memory it was computed from: it keeps that tensor alive and compares address, shape,
// strides, device and version counter.
struct Cached {
    Tensor owner, flags;
    uint32_t version = 0;
    Plan plan;
    std::shared_ptr<Prepared> prepared;
    // whether this is the entry of `t`; flags and plan are then ready for the current stream
    bool hit(const Tensor& t) const { return matches(t) && (!prepared || prepared->use()); }
    bool matches(const Tensor& t) const {
        return !t.is_inference() && owner.defined() && flags.defined() && owner.data_ptr() == t.data_ptr() && owner.sizes() == t.sizes() &&
               owner_strides == t.strides() && version == t._version() && owner.device() == t.device();
    }
    std::vector<int64_t> owner_strides;  // (the owner's own may be changed in place)
};
Cached g_bitfield, g_mask;

void store(Cached& slot, const Tensor& owner, const Tensor& flags, Plan plan, const Stream& stream) {
    Prepared::collect();
    if (owner.is_inference()) return;  // no version counter: nothing would tell that it has been written to
    if (stream.stream() != nullptr && capturing()) return;  // (flags without a plan: replays compute them, in the graph's memory)
    Cached fresh;
    fresh.owner = owner;
    fresh.owner_strides = owner.strides().vec();
    fresh.flags = flags;
    fresh.version = owner._version();
    fresh.prepared = std::make_shared<Prepared>(stream, std::vector<Tensor>{flags}, plan.core);
    fresh.plan = std::move(plan);
    std::swap(slot, fresh);  // the old entry goes after the new one is in place: its end may run Python code, which may call here
}

// What the caller of a lookup works with: a copy, as the entry itself may be replaced whenever Python code can run (the end
// of the entry it replaced, a garbage collection), by another thread or by a finalizer of this one.
struct Flags {
    Tensor flags;
    Plan plan;
};

bool plain(const Tensor& t) {  // an ordinary tensor: no subclass, no functorch wrapper, no forward-mode tangent
    return !t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                                     c10::DispatchKey::FuncTorchGradWrapper})) &&
           !t._fw_grad(0).defined();
}

bool bitfield_ready(const Tensor& bf) {
    return bf.is_cuda() && bf.scalar_type() == at::kLong && bf.dim() == 2 && bf.stride(1) == 1 && bf.size(0) > 0 &&
           bf.size(1) > 0 && !bf.is_inference() && plain(bf);
}

// From here on the plan's rows are sorted (where the segments are many).  A sequence with few segments, whose rows stay, pays the
// launch that finds that out: 4 us, which may be 2 % of the shortest forward over 16384 tokens (4 heads, D 32) and is at most 0.7 %
// from here on.  Many segments gain 5 to 28 %: forward + backward of 65536 tokens with 200 segments 62.9 -> 47.7 ms, forward alone
// of 32768 tokens with 60, 16 / 4 heads, D 64 1920 -> 1730 us.  Shorter ones with many segments would gain as well (8192 tokens with
// 30: 1873 -> 1678) and do without, as nobody knows how many there are before that launch.
constexpr int64_t kSortedRows = 32768;

// flags (and plan, up to 131072 tokens) of an int64 (B, S) mask on the GPU
Flags bitfield_flags(const Tensor& mask) {
    if (g_bitfield.hit(mask)) return {g_bitfield.flags, g_bitfield.plan};
    const Tensor bf = mask.stride(1) == 1 ? mask : mask.contiguous();
    const c10::DeviceGuard guard(bf.device());
    const int64_t B = bf.size(0), S = bf.size(1);
    const Stream stream = current_stream(bf.device());
    const c10::InferenceMode ordinary(false);  // (an entry made in inference mode also serves calls outside)
    Tensor flags = at::empty({B, (S + 127) / 128, (S + 31) / 32}, bf.options().dtype(at::kChar));
    const bool sorted = S >= kSortedRows && B * ((S + 31) / 32) * ((S + 127) / 128) < (int64_t)1 << 30 && B <= 65535;
    int64_t bytes = bam_plan_workspace_bytes((int)B, (int)S);
    if (sorted) check(bam_sorted_plan_workspace_bytes((int)B, (int)S, &bytes), "bam_sorted_plan_workspace_bytes");
    Plan plan;
    if (bytes > 0) {
        plan = new_plan();
        PlanCore& c = *plan.core;
        c.prepare(at::empty({bytes}, bf.options().dtype(at::kByte)), stream);
        const auto build = sorted ? bam_tile_plan_sorted_counted : bam_tile_plan_counted;
        const int rc = build(bf.data_ptr<int64_t>(), bf.stride(0), flags.data_ptr<int8_t>(), flags.stride(0),
                             flags.stride(1), c.workspace.data_ptr(), bytes, (int)B, (int)S, &c.plan, c.word.at, c.word.tag,
                             stream.stream());
        if (rc != BAM_OK) c.abandon();
        check(rc, "bam_tile_plan");
        c.flags = flags;
        c.flags_version = flags._version();
    } else {
        check(bam_tile_flags(bf.data_ptr<int64_t>(), bf.stride(0), flags.data_ptr<int8_t>(), flags.stride(0), flags.stride(1),
                             (int)B, (int)S, stream.stream()),
              "bam_tile_flags");
    }
    store(g_bitfield, mask, flags, plan, stream);
    return {flags, plan};
}

bool mask_ready(const Tensor& mask, int64_t B, int64_t Sq, int64_t Sk) {
    return mask.is_cuda() && mask.scalar_type() == at::kBool && mask.dim() == 3 && mask.size(0) == B && mask.size(1) == Sq &&
           mask.size(2) == Sk && mask.is_contiguous() && (reinterpret_cast<uintptr_t>(mask.data_ptr()) & 3) == 0 &&
           !mask.is_inference() && plain(mask);
}

// the same for a materialized mask that satisfies mask_ready
Flags mask_flags(const Tensor& mask) {
    if (g_mask.hit(mask)) return {g_mask.flags, g_mask.plan};
    const c10::DeviceGuard guard(mask.device());
    const int64_t B = mask.size(0), Sq = mask.size(1), Sk = mask.size(2);
    const Stream stream = current_stream(mask.device());
    const c10::InferenceMode ordinary(false);
    Tensor flags = at::empty({B, (Sq + 127) / 128, (Sk + 31) / 32}, mask.options().dtype(at::kChar));
    const int64_t bytes = bam_mask_plan_workspace_bytes((int)B, (int)Sq, (int)Sk);
    Plan plan;
    Tensor ws;
    if (bytes > 0) {
        try {
            ws = at::empty({bytes}, mask.options().dtype(at::kByte));
        } catch (const c10::OutOfMemoryError&) {  // no room for a quarter of the mask: flags only, the kernels read its bytes
        }
    }
    const uint8_t* bytes_of = (const uint8_t*)mask.data_ptr();
    if (ws.defined()) {
        plan = new_plan();
        PlanCore& c = *plan.core;
        c.prepare(ws, stream);
        const int rc = bam_mask_tile_plan_counted(bytes_of, flags.data_ptr<int8_t>(), flags.stride(0), flags.stride(1),
                                                  ws.data_ptr(), bytes, (int)B, (int)Sq, (int)Sk, &c.plan, c.word.at, c.word.tag,
                                                  stream.stream());
        if (rc != BAM_OK) c.abandon();
        check(rc, "bam_mask_tile_plan");
        c.flags = flags;
        c.flags_version = flags._version();
    } else {
        check(bam_mask_tile_flags(bytes_of, flags.data_ptr<int8_t>(), flags.stride(0), flags.stride(1), (int)B, (int)Sq, (int)Sk,
                                  stream.stream()),
              "bam_mask_tile_flags");
    }
    store(g_mask, mask, flags, plan, stream);
    return {flags, plan};
}

// ------------------------------------------------------------------ calls
bool head_dim_ready(int64_t d) { return d > 0 && d <= 128 && d % 8 == 0; }

// the kernels' layout rules: unit stride along D, 16-byte aligned rows
bool rows_ready(const Tensor& t, int64_t elems) {
    return t.stride(3) == 1 && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0 && t.stride(0) % elems == 0 &&
           t.stride(1) % elems == 0 && t.stride(2) % elems == 0;
}

bool qkv_ready(const Tensor& q, const Tensor& k, const Tensor& v) {
    if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) return false;
    const auto type = q.scalar_type();
    if (!q.is_cuda() || (type != at::kHalf && type != at::kBFloat16) || k.scalar_type() != type || v.scalar_type() != type ||
        k.device() != q.device() || v.device() != q.device() || !plain(q) || !plain(k) || !plain(v))
        return false;
    return head_dim_ready(q.size(3)) && k.sizes() == v.sizes() && k.size(0) == q.size(0) && k.size(3) == q.size(3) &&
           q.numel() > 0 && k.numel() > 0 && q.size(2) % k.size(2) == 0 && rows_ready(q, 8) && rows_ready(k, 8) && rows_ready(v, 8);
}

bam_tensor tensor4(const Tensor& t) { return bam_tensor{t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)}; }

// bias: 4-dimensional, broadcastable to (B, Hq, Sq, Sk), its last two dimensions (1 or Sq, Sk)
bool make_bias(const Tensor& bias, const Tensor& q, int64_t Sk, bam_bias& out) {
    const int64_t B = q.size(0), Sq = q.size(1), Hq = q.size(2);
    if (!bias.is_cuda() || bias.device() != q.device() || bias.dim() != 4 || bias.stride(3) != 1 ||
        (bias.scalar_type() != at::kFloat && bias.scalar_type() != q.scalar_type()) || bias.size(3) != Sk ||
        (bias.size(2) != 1 && bias.size(2) != Sq) || (bias.size(1) != 1 && bias.size(1) != Hq) ||
        (bias.size(0) != 1 && bias.size(0) != B) || bias.requires_grad() || !plain(bias))
        return false;
    auto stride = [&](int d, int64_t full) { return bias.size(d) == full && full != 1 ? bias.stride(d) : (int64_t)0; };
    // (a dimension of size 1 keeps its own stride where nothing is broadcast: it is never multiplied by more than 0)
    out = bam_bias{bias.data_ptr(), stride(0, B), stride(1, Hq), stride(2, Sq), bias.scalar_type() == at::kFloat ? 1 : 0};
    return true;
}

struct Call {  // one attention problem: sizes, mask source, bias, plan
    int mode = BAM_MASK_BITFIELD;
    const Tensor* bf = nullptr;
    const bam_index_view* index = nullptr;
    const Tensor* mask = nullptr;
    const Tensor* flags = nullptr;
    const bam_bias* bias = nullptr;
    const bam_plan* plan = nullptr;
    double scale = 0;
};

bam_attn attn_args(const Call& c, const Tensor& q, const Tensor& k, const Tensor& v) {
    bam_attn a = {};
    a.q = tensor4(q);
    a.k = tensor4(k);
    a.v = tensor4(v);
    a.mode = c.mode;
    if (c.bf != nullptr) {
        a.bf = c.bf->data_ptr<int64_t>();
        a.bf_stride_b = c.bf->stride(0);
    }
    a.index = c.index;
    a.mask = c.mask != nullptr ? (const uint8_t*)c.mask->data_ptr() : nullptr;
    a.flags = c.flags->data_ptr<int8_t>();
    a.flags_stride_b = c.flags->stride(0);
    a.flags_stride_m = c.flags->stride(1);
    a.bias = c.bias;
    a.plan = c.plan;
    a.B = (int)q.size(0);
    a.Sq = (int)q.size(1);
    a.Sk = (int)k.size(1);
    a.Hq = (int)q.size(2);
    a.Hkv = (int)k.size(2);
    a.D = (int)q.size(3);
    a.dtype = q.scalar_type() == at::kBFloat16 ? BAM_DTYPE_BF16 : BAM_DTYPE_F16;
    a.scale = (float)c.scale;
    return a;
}

std::pair<Tensor, Tensor> run_forward(const Call& c, const Tensor& q, const Tensor& k, const Tensor& v) {
    const c10::DeviceGuard guard(q.device());
    const at::NoGradGuard no_grad;
    Tensor o = at::empty_like(q);
    Tensor lse = at::empty({q.size(0), q.size(2), (q.size(1) + 127) / 128 * 128}, q.options().dtype(at::kFloat));
    bam_attn a = attn_args(c, q, k, v);
    a.o = tensor4(o);
    a.lse = lse.data_ptr<float>();
    check(bam_attn_fwd(&a, current_stream(q.device()).stream()), "bam_attn_fwd");
    return {o, lse};
}

// dq, dk, dv: written in the dtype of q, or (accumulate) fp32 and added to.  The plan's dS hand-over: Python decides on the
// workspace (it may not fit, or be taken in runs of heads) once the pair count is there.
void run_backward(Call c, const Plan& plan, const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                  const Tensor& lse, const Tensor& dq, const Tensor& dk, const Tensor& dv, bool accumulate) {
    const c10::DeviceGuard guard(q.device());
    const at::NoGradGuard no_grad;
    const bool scaled = q.size(3) <= 64 && c.bias == nullptr;
    Tensor delta = at::empty({(scaled ? 2 : 1) * lse.numel()}, lse.options());  // and the scaled lse
    bam_plan desc = {};  // (its own copy: what is known of the rows may still change)
    if (plan) {
        plan.core->look();
        desc = plan.core->plan;
        desc.rows_known = plan.core->rows_known.load();
        c.plan = &desc;
    }
    bam_attn a = attn_args(c, q, k, v);
    a.o = tensor4(o);
    a.dout = tensor4(dout);
    a.dq = tensor4(dq);
    a.dk = tensor4(dk);
    a.dv = tensor4(dv);
    a.lse = lse.data_ptr<float>();
    a.delta = delta.data_ptr<float>();
    if (scaled) a.lse_scaled = a.delta + lse.numel();
    a.accumulate = accumulate ? 1 : 0;
    Tensor ws;
    // Small problems take no dS workspace and are launched without waiting for the plan's count; where the count decides, it is waited
    // for and asked again.
    int takes_ds = 0;
    check(bam_attn_bwd_takes_ds(&a, &takes_ds), "bam_attn_bwd_takes_ds");
    auto wait_pairs = [&]() {
        optional<py::gil_scoped_release> release;
        if (PyGILState_Check()) release.emplace();
        return plan.core->wait_pairs();
    };
    if (takes_ds) {
        a.pairs = wait_pairs();
        desc.rows_known = plan.core->rows_known.load();
        check(bam_attn_bwd_takes_ds(&a, &takes_ds), "bam_attn_bwd_takes_ds");
    }
    if (takes_ds) {
        py::gil_scoped_acquire gil;
        py::tuple got = plan.py_object().attr("backward_workspace")(a.B, a.Hq, a.Hkv, a.D, a.Sk, c.bias == nullptr);
        a.head_runs = got[0].cast<int>();
        if (!got[1].is_none()) {
            ws = got[1].cast<Tensor>();
            a.ds_workspace = ws.data_ptr();
            a.ds_capacity = plan.core->pairs.load();
        }
    }
    Tensor parts;  // (given back to the caching allocator on return: the launches that use it are on the current stream)
    check(bam_attn_bwd_parts(&a, &a.parts_bytes), "bam_attn_bwd_parts");
    if (a.parts_bytes > 0) {
        try {
            parts = at::empty({a.parts_bytes}, q.options().dtype(at::kByte));
            a.parts_workspace = parts.data_ptr();
        } catch (const c10::OutOfMemoryError&) {  // no room for it right now: one part, as without a workspace
        }
    }
    check(bam_attn_bwd(&a, current_stream(q.device()).stream()), "bam_attn_bwd");
    // The count of a small problem is waited for behind its launches, which the GPU works on meanwhile: a plan whose launch failed is
    // refused by the backward here as well, and not by whatever synchronizes next.
    if (plan && a.D > 64 && a.Sk <= 131072) wait_pairs();
}

// ------------------------------------------------------------------ autograd
struct AttentionBackward : public torch::autograd::Node {
    using SavedVariable = torch::autograd::SavedVariable;
    SavedVariable q, k, v, o, lse, bias, mask, flags;  // mask: the bitfields, or the materialized mask
    Plan plan;
    int mode = BAM_MASK_BITFIELD;
    bool has_bias = false;
    at::ScalarType type = at::kHalf;  // of q
    int64_t Sk = 0, Hkv = 0;
    double scale = 0;

    std::string name() const override { return "BitfieldAttentionFunctionBackward"; }
    void release_variables() override {
        const std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable* s : {&q, &k, &v, &o, &lse, &bias, &mask, &flags}) s->reset_data();
        plan = Plan();
    }
    // A C++ exception reaches the caller of the engine as a plain RuntimeError (this module's translator is not on that way);
    // a Python error passes through it as what it is.
    variable_list apply(variable_list&& grads) override {
        try {
            return compute(std::move(grads));
        } catch (const BamFailure& e) {
            py::gil_scoped_acquire gil;
            PyErr_SetString(g_error_type != nullptr ? g_error_type : PyExc_RuntimeError, e.what());
            raise_python_error();
        } catch (py::error_already_set& e) {
            py::gil_scoped_acquire gil;
            e.restore();
            raise_python_error();
        }
    }

private:
    [[noreturn]] static void raise_python_error() {
        python_error e;
        e.persist();
        throw e;
    }
    variable_list compute(variable_list&& grads) {
        if (!grads[0].defined()) return variable_list(3);
        const at::NoGradGuard no_grad;
        Tensor q_, k_, v_, o_, lse_, bias_, mask_, flags_;
        Plan plan_;
        {  // (another thread's backward through the same graph may be releasing them)
            const std::lock_guard<std::mutex> lock(mutex_);
            q_ = q.unpack(), k_ = k.unpack(), v_ = v.unpack(), o_ = o.unpack(shared_from_this()), lse_ = lse.unpack();
            bias_ = bias.unpack(), mask_ = mask.unpack(), flags_ = flags.unpack();
            plan_ = plan;
        }
        Tensor dout = grads[0];
        if (dout.scalar_type() != type) dout = dout.to(type);
        if (!rows_ready(dout, 8)) dout = dout.contiguous();
        // What the forward saved has been through the user's saved-tensor hooks, if there are any.  Another layout is copied
        // into the kernels' form; with another shape, type or device the kernels would compute something else.
        const int64_t B = dout.size(0), Sq = dout.size(1), Hq = dout.size(2), D = dout.size(3);
        auto expect = [&](const Tensor& t, at::ScalarType st, at::IntArrayRef sizes, const char* what) {
            if (!t.defined() || t.device() != dout.device() || t.scalar_type() != st || t.sizes() != sizes || !plain(t))
                throw BamFailure(std::string("the saved ") + what + " came back from its hooks with another shape, type or device");
        };
        auto expect_rows = [&](Tensor& t, at::IntArrayRef sizes, const char* what) {
            expect(t, type, sizes, what);
            if (!rows_ready(t, 8)) t = t.clone(at::MemoryFormat::Contiguous);  // (also where only the address is not aligned)
        };
        expect_rows(q_, dout.sizes(), "q");
        expect_rows(k_, {B, Sk, Hkv, D}, "k");
        expect_rows(v_, {B, Sk, Hkv, D}, "v");
        expect_rows(o_, dout.sizes(), "o");
        expect(lse_, at::kFloat, {B, Hq, (Sq + 127) / 128 * 128}, "lse");
        lse_ = lse_.contiguous();
        expect(flags_, at::kChar, {B, (Sq + 127) / 128, (Sk + 31) / 32}, "flags");
        if (flags_.stride(2) != 1) flags_ = flags_.contiguous();
        if (mode == BAM_MASK_BITFIELD) {
            expect(mask_, at::kLong, {B, Sk}, "mask");
            if (mask_.stride(1) != 1) mask_ = mask_.contiguous();
        } else {
            expect(mask_, at::kBool, {B, Sq, Sk}, "mask");
            if (!mask_.is_contiguous() || (reinterpret_cast<uintptr_t>(mask_.data_ptr()) & 3) != 0)
                mask_ = mask_.clone(at::MemoryFormat::Contiguous);
        }
        Tensor dq = at::empty_like(q_), dk = at::empty_like(k_), dv = at::empty_like(v_);
        Call c;
        bam_bias desc;
        c.mode = mode;
        c.bf = mode == BAM_MASK_BITFIELD ? &mask_ : nullptr;
        c.mask = mode == BAM_MASK_DENSE ? &mask_ : nullptr;
        c.flags = &flags_;
        c.scale = scale;
        if (has_bias) {
            if (bias_.defined() && bias_.dim() == 4 && bias_.stride(3) != 1) bias_ = bias_.contiguous();
            if (!bias_.defined() || !make_bias(bias_, q_, Sk, desc))
                throw BamFailure("the saved bias came back from its hooks with another shape, type or device");
            c.bias = &desc;
        }
        run_backward(c, plan_, dout, q_, k_, v_, o_, lse_, dq, dk, dv, false);
        return {dq, dk, dv};
    }
};

Tensor attention(Call c, const Plan& plan, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& mask,
                 const optional<Tensor>& bias) {
    if (plan) c.plan = &plan.core->plan;
    auto [o, lse] = run_forward(c, q, k, v);
    if (at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())) {
        auto node = std::shared_ptr<AttentionBackward>(new AttentionBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(q, k, v));
        node->q = torch::autograd::SavedVariable(q, false);
        node->k = torch::autograd::SavedVariable(k, false);
        node->v = torch::autograd::SavedVariable(v, false);
        node->lse = torch::autograd::SavedVariable(lse, false);
        if (bias) node->bias = torch::autograd::SavedVariable(*bias, false);
        node->has_bias = (bool)bias;
        node->mask = torch::autograd::SavedVariable(mask, false);
        node->flags = torch::autograd::SavedVariable(*c.flags, false);
        node->plan = plan;
        node->mode = c.mode;
        node->type = q.scalar_type();
        node->Sk = k.size(1);
        node->Hkv = k.size(2);
        node->scale = c.scale;
        torch::autograd::set_history(o, node);
        node->o = torch::autograd::SavedVariable(o, true);
    }
    return o;
}

double scale_or_default(optional<double> scale, int64_t d) {
    return scale && *scale != 0.0 ? *scale : 1.0 / std::sqrt((double)d);
}

// bitfield_attn_func
optional<Tensor> bitfield_attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& bf,
                                    const optional<Tensor>& bias, optional<double> scale) {
    if (!qkv_ready(q, k, v) || !bitfield_ready(bf) || bf.device() != q.device() || bf.size(0) != q.size(0) ||
        q.size(1) != k.size(1) || bf.size(1) != k.size(1))
        return c10::nullopt;
    Call c;
    bam_bias desc;
    if (bias) {
        if (!make_bias(*bias, q, k.size(1), desc)) return c10::nullopt;
        c.bias = &desc;
    }
    const auto [flags, plan] = bitfield_flags(bf);
    if (plan && plan.core->flags.unsafeGetTensorImpl() != flags.unsafeGetTensorImpl()) return c10::nullopt;
    c.bf = &bf;
    c.flags = &flags;
    c.scale = scale_or_default(scale, q.size(3));
    return attention(c, plan, q, k, v, bf, bias);
}

// flash_attn_func
optional<Tensor> masked_attention(const Tensor& q, const Tensor& k, const Tensor& v, const optional<Tensor>& bias,
                                  const Tensor& mask, optional<double> scale) {
    if (!qkv_ready(q, k, v) || !mask_ready(mask, q.size(0), q.size(1), k.size(1)) || mask.device() != q.device())
        return c10::nullopt;
    Call c;
    bam_bias desc;
    if (bias) {
        if (!make_bias(*bias, q, k.size(1), desc)) return c10::nullopt;
        c.bias = &desc;
    }
    const auto [flags, plan] = mask_flags(mask);
    c.mode = BAM_MASK_DENSE;
    c.mask = &mask;
    c.flags = &flags;
    c.scale = scale_or_default(scale, q.size(3));
    return attention(c, plan, q, k, v, mask, bias);
}

// The forward / backward of the private entry points.  `index`: address of a bam_index_view (0 = none).
bool make_call(Call& c, bam_bias& desc, const optional<Tensor>& bf, int64_t index, const optional<Tensor>& mask, bool dense,
               const Tensor& flags, const optional<Tensor>& bias, double scale, const Tensor& q, const Tensor& k) {
    if (!flags.is_cuda() || flags.dim() != 3 || flags.scalar_type() != at::kChar || flags.stride(2) != 1) return false;
    c.mode = dense ? BAM_MASK_DENSE : index != 0 ? BAM_MASK_INDEXED : BAM_MASK_BITFIELD;
    if (c.mode == BAM_MASK_BITFIELD) {
        if (!bf || !bf->is_cuda() || bf->dim() != 2 || bf->scalar_type() != at::kLong || bf->stride(1) != 1) return false;
        c.bf = &*bf;
    }
    c.index = reinterpret_cast<const bam_index_view*>(index);
    c.mask = mask ? &*mask : nullptr;
    c.flags = &flags;
    c.scale = scale;
    if (bias) {
        if (!make_bias(*bias, q, k.size(1), desc)) return false;
        c.bias = &desc;
    }
    return true;
}

py::object forward(const Tensor& q, const Tensor& k, const Tensor& v, const optional<Tensor>& bf, int64_t index,
                   const optional<Tensor>& mask, bool dense, const Tensor& flags, const optional<Tensor>& bias, double scale,
                   const py::object& plan) {
    Call c;
    bam_bias desc;
    if (!qkv_ready(q, k, v) || !make_call(c, desc, bf, index, mask, dense, flags, bias, scale, q, k)) return py::none();
    const Plan p = plan_of(plan);
    if (p) c.plan = &p.core->plan;
    auto [o, lse] = run_forward(c, q, k, v);
    return py::make_tuple(o, lse);
}

py::object backward(Tensor dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse,
                    optional<Tensor> dq, optional<Tensor> dk, optional<Tensor> dv, bool accumulate, const optional<Tensor>& bf,
                    int64_t index, const optional<Tensor>& mask, bool dense, const Tensor& flags, const optional<Tensor>& bias,
                    double scale, const py::object& plan) {
    Call c;
    bam_bias desc;
    if (!qkv_ready(q, k, v) || !make_call(c, desc, bf, index, mask, dense, flags, bias, scale, q, k)) return py::none();
    const auto type = q.scalar_type(), out_type = accumulate ? at::kFloat : type;
    if (dout.dim() != 4 || dout.sizes() != q.sizes() || dout.scalar_type() != type || !dout.is_cuda() || o.dim() != 4 ||
        o.sizes() != q.sizes() || o.scalar_type() != type || !rows_ready(o, 8) || !lse.is_contiguous() ||
        lse.scalar_type() != at::kFloat)
        return py::none();
    if (!rows_ready(dout, 8)) dout = dout.contiguous();
    if (!dq) dq = at::empty_like(q);
    if (!dk) dk = at::empty_like(k);
    if (!dv) dv = at::empty_like(v);
    for (const auto& [g, x] : {std::pair<const Tensor&, const Tensor&>(*dq, q), {*dk, k}, {*dv, v}})
        if (g.dim() != 4 || g.sizes() != x.sizes() || g.scalar_type() != out_type || !rows_ready(g, accumulate ? 4 : 8))
            return py::none();
    run_backward(c, plan_of(plan), dout, q, k, v, o, lse, *dq, *dk, *dv, accumulate);
    return py::make_tuple(*dq, *dk, *dv);
}

// Index-tensor attention: gathers bitfields and positions of rows and keys, fills the bam_index_view at `view` and builds
// the plan.  -> (the arrays as a Prepared, plan or None)
py::tuple index_view(const Tensor& bf, const Tensor& idx_q, const Tensor& idx_k, int64_t view) {
    const c10::DeviceGuard guard(bf.device());
    const Stream stream = current_stream(bf.device());
    const int64_t B = bf.size(0), Sq = idx_q.numel(), Sk = idx_k.numel();
    Tensor bits = at::empty({B * (Sq + Sk)}, bf.options());
    Tensor pos = at::empty({Sq + Sk}, bf.options().dtype(at::kInt));
    int64_t* qb = bits.data_ptr<int64_t>();
    int* qp = pos.data_ptr<int>();
    bam_index_view& iv = *reinterpret_cast<bam_index_view*>(view);
    iv = bam_index_view{qb, qb + B * Sq, qp, qp + Sq, Sq, Sk, (int32_t)Sq, (int32_t)Sk};
    const int64_t bytes = bam_plan_workspace_bytes_rect((int)B, (int)Sq, (int)Sk);
    Plan plan;
    if (bytes > 0) {
        plan = new_plan();
        PlanCore& c = *plan.core;
        c.prepare(at::empty({bytes}, bf.options().dtype(at::kByte)), stream);
        const int rc = bam_gather_plan_indexed(bf.data_ptr<int64_t>(), bf.stride(0), (int)bf.size(1), idx_q.data_ptr<int64_t>(),
                                               idx_k.data_ptr<int64_t>(), &iv, c.workspace.data_ptr(), bytes, (int)B, &c.plan,
                                               c.word.at, c.word.tag, stream.stream());
        if (rc != BAM_OK) c.abandon();
        check(rc, "bam_gather_plan_indexed");
    } else {  // no plan for so many rows
        check(bam_gather_bitfields(bf.data_ptr<int64_t>(), bf.stride(0), (int)bf.size(1), idx_q.data_ptr<int64_t>(), (int)Sq, qb,
                                   Sq, qp, (int)B, stream.stream()),
              "bam_gather_bitfields");
        check(bam_gather_bitfields(bf.data_ptr<int64_t>(), bf.stride(0), (int)bf.size(1), idx_k.data_ptr<int64_t>(), (int)Sk,
                                   qb + B * Sq, Sk, qp + Sq, (int)B, stream.stream()),
              "bam_gather_bitfields");
    }
    return py::make_tuple(std::make_shared<Prepared>(stream, std::vector<Tensor>{bits, pos}, plan.core), plan.py_object());
}

// Counters of the decode step's merge, zero between calls, one set per stream: the calls of a stream run in order, those
// of different streams may overlap.  32 KiB per stream that has decoded; given back when the process ends.
constexpr int64_t kDecodeCounters = 8192;
std::mutex g_counters_mutex;
std::vector<std::pair<void*, Tensor>> g_counters;
// None while capturing: the library does not use them there, and a set made then would live in the graph's memory and be
// cleared by its replays.  None on hipStreamPerThread: one handle, another stream in each thread.
uint32_t* decode_counters(const Tensor& like, const Stream& stream) {
    if (capturing() || stream.stream() == hipStreamPerThread) return nullptr;
    std::lock_guard<std::mutex> guard(g_counters_mutex);
    for (const auto& [s, t] : g_counters)
        if (s == (void*)stream.stream() && t.device() == like.device()) return (uint32_t*)t.data_ptr();
    if (g_counters.size() >= 64) return nullptr;
    g_counters.emplace_back((void*)stream.stream(), at::zeros({kDecodeCounters}, like.options().dtype(at::kInt)));
    return (uint32_t*)g_counters.back().second.data_ptr();
}

// Decode step: query (B, Hq, 1, D), key / value (B, Hkv, Sk, D) -> (B, 1, Hq, D)
optional<Tensor> decode(const Tensor& q, const Tensor& k, const Tensor& v, optional<double> scaling, int64_t window,
                        double softcap) {
    if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) return c10::nullopt;
    const auto type = q.scalar_type();
    const int64_t B = q.size(0), Hq = q.size(1), D = q.size(3), Hkv = k.size(1), Sk = k.size(2);
    if (!q.is_cuda() || (type != at::kHalf && type != at::kBFloat16) || k.scalar_type() != type || v.scalar_type() != type ||
        k.device() != q.device() || v.device() != q.device() || q.size(2) != 1 || k.sizes() != v.sizes() || k.size(0) != B ||
        k.size(3) != D || !head_dim_ready(D) || q.numel() == 0 || k.numel() == 0 || Hq % Hkv != 0 || q.stride(3) != 1 ||
        !rows_ready(k, 8) || !rows_ready(v, 8) || !plain(q) || !plain(k) || !plain(v))
        return c10::nullopt;
    const c10::DeviceGuard guard(q.device());
    const at::NoGradGuard no_grad;
    Tensor out = at::empty({B, 1, Hq, D}, q.options());
    const int64_t bytes = bam_decode_workspace_bytes((int)B, (int)Sk, (int)Hq, (int)Hkv, (int)D, (int)window);
    const Stream stream = current_stream(q.device());
    Tensor ws;
    uint32_t* counters = nullptr;
    if (bytes > 0) {
        ws = at::empty({bytes}, q.options().dtype(at::kByte));
        counters = decode_counters(q, stream);
    }
    check(bam_decode_counted(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), q.stride(0), q.stride(1), k.stride(0), k.stride(2),
                     k.stride(1), v.stride(0), v.stride(2), v.stride(1), Hq * D, D, (int)B, (int)Sk, (int)Hq, (int)Hkv, (int)D,
                     (float)(scaling ? *scaling : 1.0 / std::sqrt((double)D)),
                     type == at::kBFloat16 ? BAM_DTYPE_BF16 : BAM_DTYPE_F16, (int)window, (float)softcap,
                     bytes > 0 ? ws.data_ptr() : nullptr, bytes, counters, kDecodeCounters, stream.stream()),
          "bam_decode");
    return out;
}

}  // namespace

PYBIND11_MODULE(_bam_host, m) {
    py::register_exception_translator([](std::exception_ptr p) {
        try {
            if (p) std::rethrow_exception(p);
        } catch (const BamFailure& e) {
            PyErr_SetString(g_error_type != nullptr ? g_error_type : PyExc_RuntimeError, e.what());
        }
    });
    py::class_<PlanCore, std::shared_ptr<PlanCore>>(m, "PlanCore")
        .def(py::init<>())
        .def_readonly("workspace", &PlanCore::workspace)
        .def_property_readonly("flags", [](const PlanCore& c) -> py::object {
            return c.flags.defined() ? py::cast(c.flags) : py::none();
        })
        .def_readonly("flags_version", &PlanCore::flags_version)
        .def_property_readonly("struct_address", [](const PlanCore& c) { return (int64_t)&c.plan; })
        .def("ds_pairs", &PlanCore::wait_pairs, py::call_guard<py::gil_scoped_release>());
    py::class_<Prepared, std::shared_ptr<Prepared>>(m, "Prepared").def("use", &Prepared::use);
    // once, by the Python layer: its subclass of PlanCore and the exception its callers expect
    m.def("setup", [](py::object plan_type, py::object error_type) {
        g_plan_type = plan_type.release().ptr();
        g_error_type = error_type.release().ptr();
    });
    m.def("bitfield_attention", &bitfield_attention);
    m.def("masked_attention", &masked_attention);
    m.def("forward", &forward);
    m.def("backward", &backward);
    m.def("index_view", &index_view);
    m.def("decode", &decode);
    // (flags, plan) of a mask; None where the general path has to make the mask contiguous (or complain) first
    m.def("bitfield_flags", [](const Tensor& bf) -> py::object {
        if (!bitfield_ready(bf)) return py::none();
        return py::cast(bitfield_flags(bf).flags);
    });
    m.def("bitfield_flags_general", [](const Tensor& bf) { return bitfield_flags(bf).flags; });
    m.def("mask_flags", [](const Tensor& mask, int64_t B, int64_t Sq, int64_t Sk) -> py::object {
        if (!mask_ready(mask, B, Sq, Sk)) return py::none();
        const Flags f = mask_flags(mask);
        return py::make_tuple(f.flags, f.plan.py_object());
    });
    // the plan cached with these very flags, if `bf` is still the unchanged mask they were computed from
    m.def("plan_for", [](const Tensor& flags, const Tensor& bf) -> py::object {
        const Cached& c = g_bitfield;
        if (!c.plan || !c.plan.core->flags.defined() || flags.data_ptr() != c.plan.core->flags.data_ptr() ||
            flags.sizes() != c.plan.core->flags.sizes() || !c.flags.is_same(c.plan.core->flags) || !c.hit(bf))
            return py::none();
        return c.plan.py_object();
    });
    m.def("cached_bitfield_flags", []() -> py::object {
        const Tensor flags = g_bitfield.flags;
        if (g_bitfield.prepared) g_bitfield.prepared->use();
        return flags.defined() ? py::cast(flags) : py::none();
    });
    m.def("cached_bitfield_plan", []() { return g_bitfield.plan.py_object(); });
    m.def("set_cached_bitfield_flags", [](optional<Tensor> flags) {
        Cached fresh;
        if (flags) {
            fresh = g_bitfield;
            fresh.flags = *flags;
        }
        std::swap(g_bitfield, fresh);
    });
    m.def("forget_bitfield", []() {
        Cached gone;
        std::swap(g_bitfield, gone);
    });
    m.def("forget_mask", []() {
        Cached gone;
        std::swap(g_mask, gone);
    });
    m.def("decode_counter_sets", []() { return g_counters.size(); });
    m.def("held_by_graphs", []() {
        Prepared::collect();
        return Prepared::held_by_graphs();
    });
    m.def("release_memory", []() {
        Prepared::collect();
        count_words().release();
        g_counters.clear();
    });
    // what tells a tensor (and its contents) from another for the caches that live in Python
    m.def("tensor_key", [](const Tensor& t) {
        std::string key;
        auto put = [&](int64_t x) { key.append((const char*)&x, sizeof(x)); };
        put((int64_t)t.data_ptr());
        put((int64_t)t._version());
        put(((int64_t)t.device().type() << 32) | (uint8_t)t.device().index());
        put((int64_t)t.scalar_type());
        for (int64_t x : t.sizes()) put(x);
        for (int64_t x : t.strides()) put(x);
        return py::bytes(key);
    });
}
