#include <chrono>
#include "exec.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <functional>
#include <future>
#include <set>

namespace he::exec {

// ---------------------------------------------------------------------------------------------------------
// Device pool
// ---------------------------------------------------------------------------------------------------------
static std::atomic<DevicePool*> g_pool{nullptr};

DevicePool& DevicePool::global() {
    static DevicePool* pool = [] {
        DevicePool* p = new DevicePool();  // never destroyed: tensors may outlive static destruction order
        g_pool.store(p, std::memory_order_release);
        return p;
    }();
    return *pool;
}

void DevicePool::poll_if_created() {
    if (DevicePool* p = g_pool.load(std::memory_order_acquire)) p->poll();
}

SharedEvent::~SharedEvent() {
    if (e) DevicePool::global().recycle(e);
}

void DevicePool::end_scope_after(uint64_t scope, EventRef done) {
    std::lock_guard<std::mutex> lk(mu_);
    pending_.push_back({scope, std::move(done)});
}

void DevicePool::recycle(hipEvent_t event) {
    std::lock_guard<std::mutex> lk(mu_);
    spare_events_.push_back(event);
}

void DevicePool::poll() {
    // Oldest first, and no further than the first execution that is still running: a host that runs many
    // executions ahead of the device would otherwise query every one of them on every allocation. Executions of
    // one thread finish in order; another thread's younger ones wait for the next poll at worst.
    std::vector<EventRef> passed;  // let go of outside the lock: the last holder's release takes it again
    {
        std::lock_guard<std::mutex> lk(mu_);
        while (!pending_.empty() && hipEventQuery(pending_.front().second->e) == hipSuccess) {
            if (blocks_.stream_is_live(pending_.front().first)) blocks_.end_stream(pending_.front().first);
            passed.push_back(std::move(pending_.front().second));
            pending_.pop_front();
        }
    }
}

EventRef DevicePool::take_event() {
    auto ev = std::make_shared<SharedEvent>();
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (!spare_events_.empty()) {
            ev->e = spare_events_.back();
            spare_events_.pop_back();
            return ev;
        }
    }
    HE_HIP(hipEventCreateWithFlags(&ev->e, hipEventDisableTiming));
    return ev;
}

uint64_t DevicePool::begin_scope(uint64_t thread) {
    poll();
    std::lock_guard<std::mutex> lk(mu_);
    uint64_t parent = 0;
    if (thread) {
        auto it = thread_last_scope_.find(thread);
        if (it != thread_last_scope_.end() && blocks_.stream_is_live(it->second)) parent = it->second;
    }
    const uint64_t s = blocks_.begin_stream(parent);
    if (thread) thread_last_scope_[thread] = s;
    return s;
}

void DevicePool::end_scope(uint64_t scope) {
    std::lock_guard<std::mutex> lk(mu_);
    if (blocks_.stream_is_live(scope)) blocks_.end_stream(scope);
}

size_t DevicePool::live_scopes() {
    std::lock_guard<std::mutex> lk(mu_);
    return blocks_.num_streams();
}

void DevicePool::note_locked(Tensor& t, uint64_t scope) {
    size_t kept = 0;
    bool present = false;
    for (uint64_t s : t.used)
        if (blocks_.stream_is_live(s)) {
            t.used[kept++] = s;
            present = present || s == scope;
        }
    t.used.resize(kept);
    if (!present) t.used.push_back(scope);
}

void DevicePool::note_use(Tensor& t, uint64_t scope) {
    std::lock_guard<std::mutex> lk(mu_);
    note_locked(t, scope);
}

void DevicePool::note_uses(const std::vector<TensorRef>& tensors, uint64_t scope) {
    std::lock_guard<std::mutex> lk(mu_);
    for (auto& t : tensors)
        if (t) note_locked(*t, scope);
}

Allocation DevicePool::allocate(size_t bytes, uint64_t scope) {
    // sizes are rounded up to the alignment so that small requests do not fragment the pages (device.rs:104-108)
    const uint64_t size = std::max<uint64_t>((bytes + kAlign - 1) / kAlign * kAlign, kAlign);
    Allocation a;
    for (int attempt = 0; attempt < 2; attempt++) {
        if (attempt == 1) poll();  // blocks of executions that have finished since become available
        std::lock_guard<std::mutex> lk(mu_);
        if (blocks_.allocate(size, kAlign, scope, &a.block)) {
            a.ptr = page_base_[a.block.page] + a.block.start;
            reuses_++;
            return a;
        }
    }
    // a new page: at least 1 GiB, a power of two (device.rs:144-154)
    uint64_t page = kMinPage;
    while (page < size) page *= 2;
    void* base = nullptr;
    HE_HIP(hipMalloc(&base, page));
    std::lock_guard<std::mutex> lk(mu_);
    const alloc::PageId id = blocks_.add_page(page);
    if (page_base_.size() <= id) page_base_.resize(id + 1);
    page_base_[id] = (char*)base;
    driver_bytes_ += page;
    driver_allocs_++;
    HE_REQUIRE(blocks_.allocate(size, kAlign, scope, &a.block), HE_ERR_INTERNAL, "a new page does not hold the allocation");
    a.ptr = page_base_[a.block.page] + a.block.start;
    return a;
}

void DevicePool::release(const Allocation& a, uint64_t owner, const std::vector<uint64_t>& used) {
    if (!a.ptr) return;
    std::lock_guard<std::mutex> lk(mu_);
    alloc::Block b = a.block;
    b.in_use.clear();
    if (owner && blocks_.stream_is_live(owner)) b.in_use.insert(owner);
    for (uint64_t s : used)
        if (blocks_.stream_is_live(s)) b.in_use.insert(s);
    blocks_.deallocate(std::move(b));
}

void DevicePool::stats(uint64_t* driver_bytes, uint64_t* driver_allocs, uint64_t* reuses) {
    std::lock_guard<std::mutex> lk(mu_);
    *driver_bytes = driver_bytes_;
    *driver_allocs = driver_allocs_;
    *reuses = reuses_;
}

// ---------------------------------------------------------------------------------------------------------
// Tensors
// ---------------------------------------------------------------------------------------------------------
Tensor::~Tensor() {
    if (ready && uploaded) (void)hipEventSynchronize(ready->e);  // the copy that fills the block may still be queued
    Allocation a;
    a.ptr = ptr;
    a.block = block;
    DevicePool::global().release(a, scope, used);
}

TensorRef allocate_tensor(int dtype, size_t len, uint64_t scope) {
    auto t = std::make_shared<Tensor>();
    t->dtype = dtype;
    t->len = len;
    t->bytes = storage_bytes(dtype, len);
    t->scope = scope;
    Allocation a = DevicePool::global().allocate(t->bytes, scope);
    t->ptr = a.ptr;
    t->block = std::move(a.block);
    return t;
}

namespace {
struct Staging {
    void* host = nullptr;
    size_t capacity = 0;
    hipEvent_t done = nullptr;
};
struct Streams {
    int device = 0;
    std::vector<hipStream_t> s;
    EventRef exec_end;  // end of this thread's latest execution (recorded on s[0] after it joined the others)
    bool has_run = false;
    hipStream_t h2d = nullptr, d2h = nullptr;
    void* landing = nullptr;  // pinned, kSmallDownload bytes: where small results arrive
    std::vector<Staging> staging;  // pinned upload buffers, reused once their copy has finished
};
// A pinned buffer of at least `bytes` whose previous copy (if any) has completed.
Staging& staging_buffer(Streams& st, size_t bytes) {
    for (Staging& b : st.staging)
        if (b.capacity >= bytes && hipEventQuery(b.done) == hipSuccess) return b;
    // drop finished buffers that are too small before growing: keeps at most a few per thread
    for (size_t i = 0; i < st.staging.size();) {
        if (hipEventQuery(st.staging[i].done) == hipSuccess) {
            (void)hipHostFree(st.staging[i].host);
            (void)hipEventDestroy(st.staging[i].done);
            st.staging[i] = st.staging.back();
            st.staging.pop_back();
        } else {
            i++;
        }
    }
    Staging b;
    b.capacity = std::max<size_t>(bytes, 1u << 20);
    HE_HIP(hipHostMalloc(&b.host, b.capacity, hipHostMallocDefault));
    HE_HIP(hipEventCreateWithFlags(&b.done, hipEventDisableTiming));
    st.staging.push_back(b);
    return st.staging.back();
}
std::unique_ptr<Streams> make_streams() {
    auto st = std::make_unique<Streams>();
    HE_HIP(hipGetDevice(&st->device));
    // HELIUM_HIP_STREAMS=<1..4>: how many streams the independent instructions of a step fan out over
    const char* env = getenv("HELIUM_HIP_STREAMS");
    const int n = env ? std::max(1, std::min(4, atoi(env))) : 4;
    for (int i = 0; i < n; i++) {
        hipStream_t x;
        HE_HIP(hipStreamCreateWithFlags(&x, hipStreamNonBlocking));
        st->s.push_back(x);
    }
    HE_HIP(hipStreamCreateWithFlags(&st->h2d, hipStreamNonBlocking));
    HE_HIP(hipStreamCreateWithFlags(&st->d2h, hipStreamNonBlocking));
    return st;
}
// A small pool of non-blocking streams per host thread (helium/src/cuda/context.rs:112-125), with the pinned buffers that go
// with it. A thread that ends leaves its own to the next one that begins, which carries on where they are: its executions come
// after the other's on the same stream, and so may take the memory that those have freed (DevicePool::begin_scope: the pool's
// thread token is the set's address). A thread's address as the token would be taken up by another thread's, whose streams are
// in no order with the first one's.
Streams& thread_streams() {
    struct Spare {
        std::mutex mu;
        std::vector<std::unique_ptr<Streams>> sets;
    };
    static Spare* spare = new Spare();  // never destroyed: threads may end after static destruction
    struct Mine {
        std::unique_ptr<Streams> st;
        ~Mine() {
            if (!st) return;
            std::lock_guard<std::mutex> lk(spare->mu);
            spare->sets.push_back(std::move(st));
        }
    };
    static thread_local Mine mine;
    if (!mine.st) {
        int device = 0;
        HE_HIP(hipGetDevice(&device));
        std::lock_guard<std::mutex> lk(spare->mu);
        for (auto& set : spare->sets)
            if (set->device == device) {
                mine.st = std::move(set);
                std::swap(set, spare->sets.back());
                spare->sets.pop_back();
                break;
            }
    }
    if (!mine.st) mine.st = make_streams();
    return *mine.st;
}
}  // namespace

namespace {
// Whether nothing of this thread's executions is still running: a copy may then go on the main stream, and whoever reads what
// it brings - or what it takes - needs no wait between streams, which costs the device about 10 us.
bool main_stream_is_idle(Streams& st) { return !st.has_run || hipEventQuery(st.exec_end->e) == hipSuccess; }

// Small results leave through a kernel that writes them to pinned host memory: a copy engine takes 15 us for 4 KB (23 us into
// pageable memory), the kernel and the wait for it 8.
constexpr size_t kSmallDownload = 64 << 10;
const char* kCopyOutSource = R"HIP(
extern "C" __global__ __launch_bounds__(256) void copy_out(const unsigned* __restrict__ from, unsigned* __restrict__ to, unsigned words) {
    for (unsigned i = blockIdx.x * 256u + threadIdx.x; i < words; i += gridDim.x * 256u) to[i] = from[i];
}
)HIP";
void download_small(Streams& st, const Tensor& t, void* dst, hipStream_t stream) {
    static JitKernel kernel(kCopyOutSource, "copy_out");
    if (!st.landing) HE_HIP(hipHostMalloc(&st.landing, kSmallDownload, hipHostMallocDefault));
    // (whole words: blocks are 256-byte granules)
    uint32_t words = (uint32_t)((t.bytes + 3) / 4);
    const void* from = t.ptr;
    void* argv[] = {&from, &st.landing, &words};
    const uint32_t grid[3] = {(words + 255) / 256, 1, 1}, block[3] = {256, 1, 1};
    kernel.launch(grid, block, 0, stream, argv);
    HE_HIP(hipStreamSynchronize(stream));
    memcpy(dst, st.landing, t.bytes);
}
}  // namespace

TensorRef create_tensor_with_data(const void* data, int dtype, size_t len) {
    TensorRef t = allocate_tensor(dtype, len, 0);
    Streams& st = thread_streams();
    const hipStream_t stream = main_stream_is_idle(st) ? st.s[0] : st.h2d;
    if (t->bytes) {
        // staged through pinned memory so that the copy is asynchronous (tensor_storage.rs:83-110)
        Staging& b = staging_buffer(st, t->bytes);
        memcpy(b.host, data, t->bytes);
        HE_HIP(hipMemcpyAsync(t->ptr, b.host, t->bytes, hipMemcpyHostToDevice, stream));
        HE_HIP(hipEventRecord(b.done, stream));
    }
    t->uploaded = true;
    t->ready = DevicePool::global().take_event();
    t->ready->on = stream;
    HE_HIP(hipEventRecord(t->ready->e, stream));
    return t;
}

void download_tensor(const TensorRef& t, void* dst) {
    Streams& st = thread_streams();
    // the latest execution's own result: nothing that it does not need is ahead of a copy on the main stream
    const bool latest = t->ready && t->ready == st.exec_end;
    const hipStream_t stream = latest ? st.s[0] : st.d2h;
    if (t->ready && !latest) HE_HIP(hipStreamWaitEvent(stream, t->ready->e, 0));
    if (t->bytes && t->bytes <= kSmallDownload) {
        download_small(st, *t, dst, stream);
        return;
    }
    if (t->bytes) HE_HIP(hipMemcpyAsync(dst, t->ptr, t->bytes, hipMemcpyDeviceToHost, stream));
    HE_HIP(hipStreamSynchronize(stream));
}

// ---------------------------------------------------------------------------------------------------------
// execute_graph
// ---------------------------------------------------------------------------------------------------------
namespace {
// HELIUM_HIP_EXEC_TIMING=1: host time per section of execute_graph, averaged and printed every 100 calls.
struct HostTimer {
    static bool on() {
        static const bool v = getenv("HELIUM_HIP_EXEC_TIMING") != nullptr;
        return v;
    }
    std::chrono::steady_clock::time_point t = std::chrono::steady_clock::now();
    double acc[8] = {0};
    void lap(int i) {
        if (!on()) return;
        auto n = std::chrono::steady_clock::now();
        acc[i] += std::chrono::duration<double, std::micro>(n - t).count();
        t = n;
    }
    void report() {
        if (!on()) return;
        static thread_local double sum[8] = {0};
        static thread_local int calls = 0;
        for (int i = 0; i < 8; i++) sum[i] += acc[i];
        if (++calls % 100 != 0) return;
        fprintf(stderr, "[exec timing] per graph, us: setup %.1f, storage and launches %.1f, finish %.1f\n", sum[2] / 100, sum[4] / 100, sum[5] / 100);
        for (double& v : sum) v = 0;
    }
};
// Join events of an execution are destroyed one execution later on the same thread: by then they were recorded and
// waited on long ago.
void retire_join_events(const std::vector<hipEvent_t>& events) {
    static thread_local std::vector<hipEvent_t> garbage;
    for (hipEvent_t e : garbage) (void)hipEventDestroy(e);
    garbage = events;
}
std::atomic<int> g_fan_out{1};

// Whether the independent instructions of a step are worth a stream each. Putting work on a second stream costs a
// join before and after it: on this runtime a hipStreamWaitEvent takes the host 15-20 us for the first stream that
// waits on an event and about 7 us for each further one, and the device a few microseconds per dependent queue. What
// it can gain is the time of instructions too small to fill the chip, which then run beside each other (or under an
// instruction that does fill it): an instruction that moves more than a few MiB already uses every CU or all of the
// memory bandwidth, and two of those side by side finish when they would have finished one after the other.
//
// `shares`: the instructions that would share launches (can_share_launch) count as one that does the work of all.
bool fan_out_pays(const plan::Step& step, const ir::OpGraph& g, const std::function<bool(const plan::Instr&, double)>& shares) {
    if (step.instrs.size() < 2) return false;
    constexpr double kLaunchUs = 4, kBytesPerUs = 2e6, kNarrowBytes = 4 << 20, kJoinUs = 20;
    double narrow_sum = 0, narrow_max = 0, shared = 0;
    bool wide = false;
    for (auto& instr : step.instrs) {
        double bytes = 0;
        for (NodeId n : instr->inputs()) bytes += (double)storage_bytes(g.get(n).desc.dtype, (size_t)ir::num_elements(g.get(n).desc.shape));
        for (NodeId n : instr->outputs()) bytes += (double)storage_bytes(g.get(n).desc.dtype, (size_t)ir::num_elements(g.get(n).desc.shape));
        if (bytes > kNarrowBytes) {
            wide = true;
            continue;
        }
        if (shares(*instr, bytes)) {
            shared += bytes / kBytesPerUs;
            continue;
        }
        const double us = kLaunchUs + bytes / kBytesPerUs;
        narrow_sum += us;
        narrow_max = std::max(narrow_max, us);
    }
    if (shared > 0) {
        narrow_sum += kLaunchUs + shared;
        narrow_max = std::max(narrow_max, kLaunchUs + shared);
    }
    const double gain = wide ? narrow_sum : narrow_sum - narrow_max;
    return gain > 2 * kJoinUs;
}
// The same with the launches that the instructions can share. Only a step that fans out if they share none is looked at that
// closely: whether one can is known by its kernel, so the kernels of its small instructions are compiled here.
//
// A step of 30 independent instructions: 250 us over four streams and 29 us with shared launches at 64 KB to 1 MB each, 12 of
// them 91 and 22 us. (It is so up to the 4 MB above, too: 16 of 2 MB 110 and 23 us. Those keep fanning out, as it is laid down
// for HE_OPT_STREAM_FAN_OUT.)
bool fan_out_pays(const plan::Step& step, const ir::OpGraph& g) {
    constexpr double kSharesBytes = 1 << 20;
    if (!fan_out_pays(step, g, [](const plan::Instr&, double) { return false; })) return false;
    std::vector<std::future<void>> jobs;
    for (auto& instr : step.instrs)
        if (instr->kind() == plan::InstrKind::Pointwise && !instr->compiled()) jobs.push_back(std::async(std::launch::async, [instr] { instr->precompile(); }));
    for (auto& j : jobs) j.get();
    return fan_out_pays(step, g, [](const plan::Instr& instr, double bytes) { return bytes <= kSharesBytes && !instr.absorbed() && can_share_launch(instr); });
}

// The side stream. A training step ends in many chains that nothing else waits for: a filter gradient, the launch that
// adds up its partial tiles, the optimizer's update of that filter. On one stream each of them holds up the chain
// that everything else hangs on (the data gradients); on a second stream they run beside it - matrix-core work under
// the memory-bound kernels of the next layers, and the other way round. The split: the instruction that nothing reads
// and that the most work leads up to ends the main chain; every instruction it does not depend on, directly or
// indirectly, runs on the side (no main instruction reads what a side instruction writes, by construction) - the small
// ones too: keeping those of less than 10 us that read main results only on the main stream measured 0.5% slower.
// HELIUM_HIP_SIDE_STREAM=0 switches the side stream off, =1 on for plans of any size.
void side_stream_split(Prepared* pr) {
    const char* env = tuning::get("HELIUM_HIP_SIDE_STREAM");
    if (env && atoi(env) == 0) return;
    const bool forced = env && atoi(env) != 0;
    for (uint8_t f : pr->fan_out)
        if (f) return;  // a plan whose steps fan out keeps to that scheme
    Prepared::Side S;
    for (auto& step : pr->plan->steps)
        for (auto& instr : step.instrs)
            if (!instr->absorbed()) {
                S.index[instr.get()] = S.order.size();
                S.order.push_back(instr.get());
            }
    const size_t n = S.order.size();
    if (n < 3) return;
    const ir::OpGraph& g = *pr->graph;
    auto bytes_of = [&](NodeId id) { return (double)storage_bytes(g.get(id).desc.dtype, (size_t)ir::num_elements(g.get(id).desc.shape)); };
    constexpr double kLaunchUs = 4, kBytesPerUs = 2e6, kWorthUs = 200, kDeviceBoundUs = 10;
    std::map<NodeId, uint32_t> made_by;
    std::vector<double> cost(n);
    S.deps.resize(n);
    S.dependents.resize(n);
    for (size_t i = 0; i < n; i++) {
        double bytes = 0;
        std::set<uint32_t> from;
        for (NodeId in : S.order[i]->all_inputs()) {
            bytes += bytes_of(in);
            auto it = made_by.find(in);
            if (it != made_by.end() && it->second != i) from.insert(it->second);
        }
        for (uint32_t d : from) {
            S.deps[i].push_back(d);
            S.dependents[d].push_back((uint32_t)i);
        }
        for (NodeId out : S.order[i]->all_outputs()) {
            bytes += bytes_of(out);
            made_by[out] = (uint32_t)i;
        }
        cost[i] = kLaunchUs + bytes / kBytesPerUs;
    }
    auto ancestors = [&](size_t of) {
        std::vector<uint8_t> in(n, 0);
        std::vector<uint32_t> stack{(uint32_t)of};
        in[of] = 1;
        while (!stack.empty()) {
            const uint32_t cur = stack.back();
            stack.pop_back();
            for (uint32_t d : S.deps[cur])
                if (!in[d]) {
                    in[d] = 1;
                    stack.push_back(d);
                }
        }
        return in;
    };
    std::vector<uint8_t> main_set;
    double main_cost = -1;
    for (size_t s = 0; s < n; s++) {
        if (!S.dependents[s].empty()) continue;
        std::vector<uint8_t> in = ancestors(s);
        double c = 0;
        for (size_t i = 0; i < n; i++)
            if (in[i]) c += cost[i];
        if (c >= main_cost) {
            main_cost = c;
            main_set.swap(in);
        }
    }
    S.side.assign(n, 0);
    double side_cost = 0;
    for (size_t i = 0; i < n; i++) {
        if (main_set[i]) continue;
        S.side[i] = 1;
        side_cost += cost[i];
    }
    // Early instructions (side value 2): small main-chain instructions that read nothing but the graph's inputs (or each
    // other) - a filter converted to the multiplicands' type ahead of its convolution - and whose first reader comes
    // well into the execution. Each would hold the main stream for a launch's latency; the side stream runs them all at
    // the start instead, and the main stream waits for them once, ahead of the first instruction that reads one.
    size_t early = 0;
    if (!tuning::get("HELIUM_HIP_NO_EARLY_INSTRS")) {
        constexpr double kEarlyUs = 20, kLeadUs = 100;
        std::vector<double> before(n + 1, 0);  // main-stream work ahead of each position
        for (size_t i = 0; i < n; i++) before[i + 1] = before[i] + (S.side[i] ? 0 : cost[i]);
        for (size_t i = 0; i < n; i++) {
            if (S.side[i] || cost[i] >= kEarlyUs || S.dependents[i].empty()) continue;
            bool sources_only = true;
            for (uint32_t d : S.deps[i]) sources_only = sources_only && S.side[d] == 2;
            uint32_t first_reader = (uint32_t)n;
            for (uint32_t d : S.dependents[i]) first_reader = std::min(first_reader, d);
            if (!sources_only || (!forced && before[first_reader] < kLeadUs)) continue;
            S.side[i] = 2;
            early++;
        }
    }
    if (getenv("HELIUM_HIP_PLAN_DEBUG")) {
        size_t count = 0;
        for (uint8_t f : S.side) count += f == 1;
        fprintf(stderr, "[plan] side stream: %zu of %zu launching instructions, about %.0f us beside %.0f us; %zu early instructions\n", count, n, side_cost,
                main_cost, early);
    }
    if (side_cost == 0 || (!forced && side_cost < kWorthUs)) return;
    // An execution that the host cannot keep ahead of (it needs 8-10 us per launch, and 15-20 more per wait between
    // streams) gains nothing from a second stream and loses the waits: the training step at batch 4 to 16, where the
    // estimate is 6 to 8 us of device time per launch, ran up to 1.5x slower with it; at 11 us (batch 32) and above it
    // gains 7-12%.
    if (!forced && (main_cost + side_cost) / (double)n < kDeviceBoundUs) return;
    pr->side = std::move(S);
}
}  // namespace

void assign_streams(Prepared* pr) {
    for (auto& step : pr->plan->steps) pr->fan_out.push_back(fan_out_pays(step, *pr->graph));
    side_stream_split(pr);
    for (size_t i = 0; i < pr->side.order.size(); i++)
        if (pr->side.side[i] == 1 && pr->side.order[i]->kind() == plan::InstrKind::Gemm) pr->side.order[i]->runs_beside_main_chain();
}

void set_stream_fan_out(int mode) {
    HE_REQUIRE(mode >= 0 && mode <= 2, HE_ERR_INVALID, "stream fan-out is 0 (never), 1 (where it pays) or 2 (always)");
    g_fan_out.store(mode);
}

std::shared_ptr<const Prepared> prepare(const ir::OpGraph& graph_in) {
    auto pr = std::make_shared<Prepared>();
    auto graph = std::make_shared<ir::OpGraph>(graph_in);
    graph->optimize();
    pr->graph = plan::graph_for_execution(graph);
    if (pr->graph->has_origins()) {
        for (NodeId in : pr->graph->inputs()) pr->input_of[pr->graph->origin(in)] = in;
        for (NodeId out : pr->graph->outputs()) pr->caller_output[out] = pr->graph->origin(out);
    }
    pr->plan = plan::generate_cached_plan(pr->graph);
    // tensors that survive the plan get their ready event recorded (enumerate_output_tensors, cuda.rs:142-153)
    for (auto& step : pr->plan->steps) {
        for (auto& instr : step.instrs)
            for (NodeId o : instr->outputs()) pr->alive.insert(o);
        for (NodeId r : step.tensors_to_release) pr->alive.erase(r);
    }
    // (ahead of the kernels: a product that will run beside the main chain is built for that)
    assign_streams(pr.get());
    // begin_execute (cuda.rs:98-139): compile every kernel of the plan up front, in parallel (cuda.rs:262-270)
    std::vector<std::future<void>> jobs;
    for (auto& step : pr->plan->steps)
        for (auto& instr : step.instrs)
            if (!instr->compiled()) jobs.push_back(std::async(std::launch::async, [instr] { instr->precompile(); }));
    for (auto& j : jobs) j.get();
    build_schedule(pr.get());
    if (getenv("HELIUM_HIP_PLAN_DEBUG") && pr->schedule) {
        uint64_t bytes = 0;
        for (uint64_t b : pr->schedule->blocks) bytes += b;
        fprintf(stderr, "[plan] schedule: %d instructions, %zu launches, %.1f MB of intermediate values in %zu blocks\n", pr->schedule->instrs,
                pr->schedule->launches.size(), bytes / 1e6, pr->schedule->blocks.size());
    }
    if (getenv("HELIUM_HIP_PLAN_DEBUG")) {
        size_t fanned = 0, multi = 0;
        for (size_t k = 0; k < pr->plan->steps.size(); k++) {
            fanned += pr->fan_out[k];
            multi += pr->plan->steps[k].instrs.size() > 1;
        }
        fprintf(stderr, "[plan] %zu steps, %zu with several instructions, %zu of them fan out over streams\n", pr->plan->steps.size(), multi, fanned);
    }
    return pr;
}

namespace {
// The thread's streams wait for a tensor that something outside this execution fills (an upload, another thread's graph).
void wait_for_tensor(const Tensor& t, hipStream_t stream, hipStream_t main, ExecStats* stats) {
    // What the main stream recorded is ahead of this execution there; the side stream has waited for the end of the thread's
    // previous execution, which an upload can come after.
    if (!t.ready || (t.ready->on == main && (stream == main || !t.uploaded)) || t.ready_seen.load(std::memory_order_acquire)) return;
    // a producer seen finished once stays finished: no wait is queued for it again
    if (hipEventQuery(t.ready->e) == hipSuccess) {
        const_cast<Tensor&>(t).ready_seen.store(true, std::memory_order_release);
        return;
    }
    HE_HIP(hipStreamWaitEvent(stream, t.ready->e, 0));
    stats->event_waits++;
}

// HELIUM_HIP_INSTR_TIMING=<n>: every launch is timed on its own (the device is drained before and after it), and the n
// slowest of the second execution are listed with the bytes they read and write. A debugging aid: it serialises.
struct LaunchTimes {
    static int wanted() {
        static const int n = getenv("HELIUM_HIP_INSTR_TIMING") ? atoi(getenv("HELIUM_HIP_INSTR_TIMING")) : 0;
        return n;
    }
    struct Time {
        double us;
        size_t launch;
    };
    std::vector<Time> times;
    std::chrono::steady_clock::time_point t0;
    void start() {
        HE_HIP(hipDeviceSynchronize());
        t0 = std::chrono::steady_clock::now();
    }
    void stop(size_t launch) {
        HE_HIP(hipDeviceSynchronize());
        times.push_back({std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count(), launch});
    }
    void report(const Schedule& S) {
        static std::atomic<int> reports{0};
        if (times.empty() || reports.fetch_add(1) != 1) return;  // the second execution: kernels are compiled and loaded by then
        std::sort(times.begin(), times.end(), [](const Time& a, const Time& b) { return a.us > b.us; });
        double total = 0;
        for (auto& t : times) total += t.us;
        fprintf(stderr, "[instr timing] %zu launches, %.1f us in all; slowest:\n", times.size(), total);
        for (int i = 0; i < wanted() && i < (int)times.size(); i++) {
            const Schedule::Launch& L = S.launches[times[i].launch];
            int64_t bytes = 0;
            for (uint32_t a : L.args) bytes += (int64_t)S.slots[a].bytes;
            fprintf(stderr, "  #%-4zu %8.1f us %8.1f MB %6.2f TB/s  %s\n", times[i].launch, times[i].us, bytes / 1e6, bytes / times[i].us / 1e6,
                    L.kernel ? L.kernel->describe().substr(0, 320).c_str() : "permute");
        }
    }
};

NamedTensors execute_scheduled(const Prepared& prepared, const NamedTensors& inputs, bool one_stream, ExecStats* stats) {
    HostTimer ht;
    const Schedule& S = *prepared.schedule;
    DevicePool& pool = DevicePool::global();
    Streams& st = thread_streams();
    const hipStream_t main = st.s[0];
    const bool use_side = S.uses_side && !one_stream && st.s.size() >= 2 && !LaunchTimes::wanted();
    static const bool launch_events = getenv("HELIUM_HIP_NO_LAUNCH_EVENTS") == nullptr;
    ExecStats local;
    std::vector<TensorRef> tensors(S.slots.size());  // the caller's and the results
    for (auto& in : inputs) {
        auto it = std::lower_bound(S.inputs.begin(), S.inputs.end(), in.first, [](const Schedule::Named& a, NodeId n) { return a.node < n; });
        if (it != S.inputs.end() && it->node == in.first) tensors[it->slot] = in.second;
    }
    for (auto& in : S.inputs) HE_REQUIRE(tensors[in.slot], HE_ERR_INVALID, "missing storage for input node %u", in.node);
    EventRef done = pool.take_event();
    done->on = main;
    const uint64_t scope = pool.begin_scope((uint64_t)(uintptr_t)&st);
    bool done_recorded = false, side_used = false, side_joined = false;
    std::vector<EventRef> events;  // of this execution, given back when it has been queued
    auto record = [&](hipStream_t on) {
        events.push_back(pool.take_event());
        HE_HIP(hipEventRecord(events.back()->e, on));
        return events.back()->e;
    };
    auto join_side = [&] {
        if (!side_used || side_joined) return;
        HE_HIP(hipStreamWaitEvent(main, record(st.s[1]), 0));
        local.event_waits++;
        side_joined = true;
    };
    std::vector<TensorRef> blocks(S.blocks.size());
    try {
        pool.note_uses(tensors, scope);
        ht.lap(2);
        hipEvent_t main_end = nullptr, early_end = nullptr;  // what the next wait of the other stream is for
        std::vector<void*> ptrs;
        LaunchTimes timing;
        for (size_t i = 0; i < S.launches.size(); i++) {
            const Schedule::Launch& L = S.launches[i];
            for (uint32_t b : L.opens_blocks) blocks[b] = allocate_tensor(HE_U32, (size_t)(S.blocks[b] / 4), scope);
            for (uint32_t r : L.opens_results) tensors[r] = allocate_tensor(S.slots[r].dtype, S.slots[r].len, scope);
            const bool on_side = use_side && L.stream == 1;
            const hipStream_t stream = on_side ? st.s[1] : main;
            if (on_side) {
                // the side stream's first work of this execution comes after the end of the thread's previous one
                if (!side_used && st.has_run) HE_HIP(hipStreamWaitEvent(stream, st.exec_end->e, 0));
                side_used = true;
                if (L.waits_for_main) {
                    HE_HIP(hipStreamWaitEvent(stream, main_end, 0));
                    local.event_waits++;
                }
            } else if (use_side && L.waits_for_early) {
                HE_HIP(hipStreamWaitEvent(stream, early_end, 0));
                local.event_waits++;
            }
            for (uint32_t in : L.new_inputs) wait_for_tensor(*tensors[in], stream, main, &local);
            const bool closes = L.closes && launch_events;
            if (closes) {
                join_side();
                set_pending_stop_event(done->e);
            } else if (use_side && L.marks_end && launch_events) {
                events.push_back(pool.take_event());
                main_end = events.back()->e;
                set_pending_stop_event(main_end);
            }
            ptrs.resize(L.args.size());
            for (size_t a = 0; a < L.args.size(); a++) {
                const Schedule::Slot& s = S.slots[L.args[a]];
                ptrs[a] = s.where == Schedule::Slot::Arena ? (char*)blocks[s.block]->ptr + s.offset : tensors[L.args[a]]->ptr;
            }
            if (LaunchTimes::wanted()) timing.start();
            try {
                if (L.kernel) L.kernel->execute(ptrs.data(), stream);
                else L.permute->execute(ptrs[0], ptrs[1], stream);
            } catch (...) {
                (void)take_pending_stop_event();
                throw;
            }
            if (LaunchTimes::wanted()) timing.stop(i);
            // (still pending: a launch too large for the entry point that takes an event)
            const bool taken = take_pending_stop_event() == nullptr;
            if (closes) done_recorded = taken;
            else if (use_side && L.marks_end && !(taken && launch_events)) main_end = record(stream);
            if (use_side && i + 1 == S.early_launches) early_end = record(stream);
            for (uint32_t b : L.closes_blocks) blocks[b].reset();
        }
        ht.lap(4);
        join_side();
        // Drop of the executor (cuda.rs:232-260): when everything queued above has run, the scope's freed blocks become available
        // to everyone. The main stream carries the event the pool polls.
        if (!done_recorded) HE_HIP(hipEventRecord(done->e, main));
        timing.report(S);
    } catch (...) {
        // The scope must end, and only after the work already queued.
        try {
            side_joined = false;
            join_side();
            HE_HIP(hipEventRecord(done->e, main));
            st.exec_end = done;
            st.has_run = true;
            pool.end_scope_after(scope, done);
        } catch (...) {
            (void)hipDeviceSynchronize();
            pool.end_scope(scope);
        }
        throw;
    }
    // The same event orders this thread's next execution after this one, and it is the ready event of every tensor the caller
    // gets (enumerate_output_tensors, cuda.rs:142-153, records one per tensor).
    for (size_t i = 0; i < S.slots.size(); i++)
        if (S.slots[i].where == Schedule::Slot::Result) tensors[i]->ready = done;
    st.exec_end = done;
    st.has_run = true;
    pool.end_scope_after(scope, std::move(done));
    local.steps = S.steps;
    local.instrs = S.instrs;
    local.streams_used = side_used ? 2 : 1;
    if (stats) *stats = local;
    NamedTensors result;
    result.reserve(S.outputs.size());
    for (auto& o : S.outputs) result.emplace_back(o.node, tensors[o.slot]);
    ht.lap(5);
    ht.report();
    return result;
}
}  // namespace

NamedTensors execute_prepared(const Prepared& prepared, const NamedTensors& named_inputs, ExecStats* stats) {
    const int fan_mode = g_fan_out.load();
    if (prepared.schedule && fan_mode != 2) return execute_scheduled(prepared, named_inputs, fan_mode == 0, stats);
    // Step by step, the instructions of a step over the thread's streams.
    // The ids of a rewritten graph differ from the caller's: inputs are renamed on the way in, outputs on the way out
    std::map<NodeId, TensorRef> inputs;
    for (auto& kv : named_inputs) {
        if (prepared.input_of.empty()) {
            inputs[kv.first] = kv.second;
            continue;
        }
        auto it = prepared.input_of.find(kv.first);
        if (it != prepared.input_of.end()) inputs[it->second] = kv.second;
    }
    const std::shared_ptr<const ir::OpGraph>& graph = prepared.graph;
    const std::shared_ptr<const plan::Plan>& plan = prepared.plan;
    const std::set<NodeId>& alive = prepared.alive;
    DevicePool& pool = DevicePool::global();
    Streams& st = thread_streams();
    for (NodeId in : graph->inputs())
        HE_REQUIRE(inputs.count(in), HE_ERR_INVALID, "missing storage for input node %u", in);
    const uint64_t scope = pool.begin_scope((uint64_t)(uintptr_t)&st);
    std::map<NodeId, TensorRef> tensors = inputs;
    {
        std::vector<TensorRef> held;
        for (auto& kv : inputs) held.push_back(kv.second);
        pool.note_uses(held, scope);
    }
    ExecStats local;
    std::set<const Tensor*> synced;        // input tensors whose ready event a stream already waited on
    std::vector<size_t> prev_streams;      // streams the previous step ran on
    std::vector<hipEvent_t> events;        // join events of this execution
    std::map<size_t, std::set<hipEvent_t>> waited_for;  // per stream: the events it has been made to wait for
    std::set<size_t> used_streams;
    // Every stream in `cur` waits for the end of the previous step on every other stream it ran on. The events are
    // recorded here, before the new step enqueues anything, so they mark exactly the end of that step.
    auto join = [&](const std::vector<size_t>& cur) {
        for (size_t p : prev_streams) {
            bool needed = false;
            for (size_t w : cur) needed = needed || w != p;
            if (!needed) continue;
            hipEvent_t e;
            HE_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
            events.push_back(e);
            HE_HIP(hipEventRecord(e, st.s[p]));
            for (size_t w : cur)
                if (w != p) {
                    HE_HIP(hipStreamWaitEvent(st.s[w], e, 0));
                    local.event_waits++;
                }
        }
    };
    // An execution whose steps hold one instruction each runs on stream 0 alone: its last launch can carry the
    // execution's event itself.
    auto step_width = [&](size_t k) {
        const plan::Step& step = plan->steps[k];
        const bool fan = !step.in_order && (fan_mode == 2 || (fan_mode == 1 && prepared.fan_out[k]));
        return fan ? std::min(step.instrs.size(), st.s.size()) : std::min<size_t>(step.instrs.size(), 1);
    };
    const plan::Instr* closing = nullptr;
    {
        bool one_stream = true;
        for (size_t k = 0; k < plan->steps.size(); k++) {
            auto& step = plan->steps[k];
            one_stream = one_stream && step_width(k) <= 1;
            for (auto& instr : step.instrs)
                if (!instr->absorbed()) closing = instr.get();  // (an absorbed instruction launches nothing)
        }
        if (!one_stream || getenv("HELIUM_HIP_NO_LAUNCH_EVENTS")) closing = nullptr;
    }
    EventRef done = pool.take_event();
    done->on = st.s[0];
    bool done_recorded = false;
    // One instruction on stream `w` of the thread's pool: storage for what it writes, waits for inputs made outside
    // this execution, its launches.
    auto run_instr = [&](const plan::Instr& instr, size_t w, std::vector<const Tensor*>& waited) {
        hipStream_t stream = st.s[w];
        // a stream's first work of this execution comes after the end of the thread's previous execution
        // (stream 0 carried that end itself)
        if (used_streams.insert(w).second && w != 0 && st.has_run) {
            HE_HIP(hipStreamWaitEvent(stream, st.exec_end->e, 0));
            waited_for[w].insert(st.exec_end->e);
        }
        for (NodeId out : instr.all_outputs()) {
            const ir::Descriptor& d = graph->get(out).desc;
            tensors[out] = allocate_tensor(d.dtype, (size_t)ir::num_elements(d.shape), scope);
        }
        for (NodeId in : instr.all_inputs()) {
            auto it = tensors.find(in);
            HE_REQUIRE(it != tensors.end(), HE_ERR_INTERNAL, "missing storage for node %u", in);
            // tensors made outside this execution carry a ready event (uploads, earlier graphs)
            if (inputs.count(in) && !synced.count(it->second.get())) {
                Tensor& t = *it->second;
                // a producer seen finished once stays finished: no wait is queued for it again
                if (t.ready && !t.ready_seen.load(std::memory_order_acquire)) {
                    if (hipEventQuery(t.ready->e) == hipSuccess) {
                        t.ready_seen.store(true, std::memory_order_release);
                    } else if (waited_for[w].insert(t.ready->e).second) {
                        // (one wait per event and stream: the tensors a previous execution returned share its end event,
                        // and a wait costs the host 15-20 us on a stream other than the one that recorded the event)
                        HE_HIP(hipStreamWaitEvent(stream, t.ready->e, 0));
                        local.event_waits++;
                    }
                }
                waited.push_back(it->second.get());
            }
        }
        if (&instr == closing) set_pending_stop_event(done->e);
        try {
            instr.execute([&](NodeId n) -> void* { return tensors.at(n)->ptr; }, stream);
        } catch (...) {
            (void)take_pending_stop_event();
            throw;
        }
        // taken by the instruction's last launch, or still pending (a launch too large for that entry point)
        if (&instr == closing) done_recorded = take_pending_stop_event() == nullptr;
        local.instrs++;
    };
    // Whatever happens below, the scope must end, and only after the work already queued: a failing instruction leaves
    // earlier launches running on up to four streams. On failure stream 0 is ordered after every stream this execution
    // used, the end event is recorded there as usual, and the error goes on to the caller.
    try {
    for (size_t step_no = 0; step_no < plan->steps.size(); step_no++) {
        auto& step = plan->steps[step_no];
        for (NodeId r : step.tensors_to_release) tensors.erase(r);
        if (step.instrs.empty()) continue;
        local.steps++;
        std::vector<const Tensor*> waited;
        // Instructions of one step are independent: they fan out over the stream pool where that pays.
        const size_t width = step_width(step_no);
        std::vector<size_t> cur(width);
        for (size_t w = 0; w < width; w++) cur[w] = w;
        join(cur);
        for (size_t i = 0; i < step.instrs.size(); i++) {
            const plan::Instr& instr = *step.instrs[i];
            if (instr.absorbed()) continue;  // run, and its outputs allocated, by the instruction that carries it
            run_instr(instr, i % width, waited);
        }
        // every stream of the next steps is ordered after this step's streams, so one wait per tensor is enough
        synced.insert(waited.begin(), waited.end());
        prev_streams = cur;
    }
    } catch (...) {
        try {
            prev_streams.assign(used_streams.begin(), used_streams.end());
            join({0});
            HE_HIP(hipEventRecord(done->e, st.s[0]));
            st.exec_end = done;
            st.has_run = true;
            pool.end_scope_after(scope, done);
        } catch (...) {
            (void)hipDeviceSynchronize();
            pool.end_scope(scope);
        }
        retire_join_events(events);
        throw;
    }
    // Drop of the executor (cuda.rs:232-260): when everything queued above has run, the scope's freed blocks
    // become available to everyone. Stream 0 joins the last step and carries the event the pool polls.
    join({0});
    if (!done_recorded) HE_HIP(hipEventRecord(done->e, st.s[0]));
    // The same event orders this thread's next execution after this one, and it is the ready event of every tensor
    // that outlives the plan (enumerate_output_tensors, cuda.rs:142-153, records one per tensor).
    for (NodeId out : alive) tensors.at(out)->ready = done;
    st.exec_end = done;
    st.has_run = true;
    pool.end_scope_after(scope, std::move(done));
    retire_join_events(events);
    local.streams_used = (int)used_streams.size();
    if (stats) *stats = local;

    NamedTensors result;
    for (NodeId out : graph->outputs()) {
        NodeId from = graph->inbound(out)[0];
        auto it = tensors.find(from);
        HE_REQUIRE(it != tensors.end(), HE_ERR_INTERNAL, "output node %u has no storage", out);
        result.emplace_back(prepared.caller_output.empty() ? out : prepared.caller_output.at(out), it->second);
    }
    std::sort(result.begin(), result.end(), [](const auto& a, const auto& b) { return a.first < b.first; });
    return result;
}

}  // namespace he::exec
