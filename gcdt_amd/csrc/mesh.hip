// gfx950 kernels and host drivers of the mesh phases: scans, sampling,
// bitmap ("boostmap") location, parallel insertion rounds, flip rounds,
// leaf compaction and adjacency construction.
#include <algorithm>
#include <atomic>
#include <climits>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "mesh.hpp"

namespace gcdt {

// ================================================================== context

// Values of each tunable that a GPU parity test covers (the autotuner's
// candidates, plus tail thresholds 0 and 2^20 that force one round path).
// Anything else is refused, by gcdt_set_tunable and by the environment
// overrides alike.
bool tunable_cleared(const std::string& name, int v)
{
    if (name == "tail_threshold")
        return v == 0 || v == 1024 || v == 2048 || v == 4096 || v == 8192 || v == 16384 || v == (1 << 20);
    if (name == "grid_cap") return v == 2048 || v == 4096 || v == 8192 || v == 16384;
    if (name == "flip_items" || name == "ins_items") return v == 1 || v == 2 || v == 4;
    if (name == "pivot" || name == "single_tester" || name == "validate") return v == 0 || v == 1;
    return false;
}

Tunables& Tunables::get()
{
    static Tunables t = [] {
        Tunables x;
        auto env = [&](const char* var, const char* name, int* dst) {
            const char* e = getenv(var);
            if (!e) return;
            char* end = nullptr;
            long v = strtol(e, &end, 10);
            if (end == e || *end != 0 || v < INT_MIN || v > INT_MAX || !tunable_cleared(name, (int)v)) {
                x.env_error += std::string(var) + "=" + e + " is not a cleared value; ";
                return;
            }
            *dst = (int)v;
        };
        env("GCDT_TAIL_THRESHOLD", "tail_threshold", &x.tail_threshold);
        env("GCDT_PIVOT", "pivot", &x.pivot);
        env("GCDT_SINGLE_TESTER", "single_tester", &x.single_tester);
        env("GCDT_VALIDATE", "validate", &x.validate);
        env("GCDT_GRID_CAP", "grid_cap", &g_grid_cap);
        return x;
    }();
    return t;
}

thread_local std::vector<PendingFree>* g_defer = nullptr;
int g_grid_cap = kMaxGrid;

thread_local Arena* g_arena = nullptr;

void Arena::require(size_t bytes) const
{
    if (bytes > cap)
        throw Error(GCDT_ERR_SCRATCH, "the scratch array (" + std::to_string(cap) + " bytes) is too small for this "
                                      "input: " + std::to_string(bytes) + " bytes needed so far");
}

void* Arena::take(size_t bytes)
{
    const size_t len = size(bytes);
    require(top + len);
    void* p = base + top;
    top += len;
    if (top > high) high = top;
    return p;
}

void Arena::give(void* p, size_t bytes)
{
    size_t off = (size_t)((char*)p - base), end = off + size(bytes);
    if (end != top) {
        if (nfreed < kFreed) {
            freed_off[nfreed] = off;
            freed_end[nfreed] = end;
            nfreed++;
        }
        return;  // a full list leaves the block in use until the call ends
    }
    top = off;
    for (bool again = true; again;) {
        again = false;
        for (int i = 0; i < nfreed; i++)
            if (freed_end[i] == top) {
                top = freed_off[i];
                freed_off[i] = freed_off[--nfreed];
                freed_end[i] = freed_end[nfreed];
                again = true;
                break;
            }
    }
}

void hold_to(DBuf<int>& pad, size_t top)
{
    if (g_arena && g_arena->top < top) pad.alloc((top - g_arena->top) / sizeof(int));
}

void* dev_take(size_t bytes)
{
    if (g_arena) return g_arena->take(bytes);
    void* p = getMemCacheRef().getMemByAbtrtSize(bytes);
    if (!p) throw Error(GCDT_ERR_OOM, "device pool allocation failed");
    return p;
}

void dev_give(void* p, size_t bytes)
{
    if (!p) return;
    if (g_arena && g_arena->owns(p)) g_arena->give(p, bytes);
    else if (g_defer) g_defer->push_back({p, bytes});
    else getMemCacheRef().releaseAbtrtMem(p, bytes);
}

namespace {
// Pinned counter mirrors and snapshot rings, reused across solves: allocating
// and freeing pinned memory per call costs more than a small solve and
// hipHostFree waits for the whole device, which would serialise solves that
// run on different streams.
std::mutex g_host_mu;
std::vector<HostSlot> g_host_free;
}  // namespace

HostSlot take_host_slot()
{
    {
        std::lock_guard<std::mutex> g(g_host_mu);
        if (!g_host_free.empty()) {
            HostSlot h = g_host_free.back();
            g_host_free.pop_back();
            return h;
        }
    }
    HostSlot h{};
    GCDT_HIP(hipHostMalloc((void**)&h.hcnt, sizeof(int) * C_NUM, hipHostMallocDefault));
    // written by kernels (round-begin snapshots): coherent, so the writes reach
    // host memory without a cache flush; sequence number 0 is never issued
    GCDT_HIP(hipHostMalloc((void**)&h.hring, sizeof(unsigned long long) * 2 * C_NUM,
                           hipHostMallocMapped | hipHostMallocCoherent));
    memset(h.hring, 0, sizeof(unsigned long long) * 2 * C_NUM);
    GCDT_HIP(hipHostGetDevicePointer((void**)&h.hring_dev, h.hring, 0));
    return h;
}

Ctx::Ctx(hipStream_t s, const HostSlot* fixed) : st(s)
{
    if (!Tunables::get().env_error.empty()) throw Error(GCDT_ERR_INVALID, Tunables::get().env_error);
    tail_threshold = Tunables::get().tail_threshold;
    pivot = Tunables::get().pivot;
    single_tester = Tunables::get().single_tester;
    flip_items = Tunables::get().flip_items;
    ins_items = Tunables::get().ins_items;
    dcnt.alloc(C_NUM);
    // on a fixed array below everything that is given back before them
    if (g_arena) {
        ring.ensure(ROUND_SETS * ROUND_INTS);
        scan_sums.ensure(ARENA_SCAN_SUMS);
    }
    HostSlot h = fixed ? *fixed : take_host_slot();
    fixed_slot = fixed != nullptr;
    hcnt = h.hcnt;
    hring = h.hring;
    hring_dev = h.hring_dev;
    if (st) {
        prev_defer = g_defer;
        g_defer = &deferred;
    }
    zero_counters();
}

Ctx::~Ctx()
{
    if (st) {
        // every kernel of this solve has finished before its blocks go back
        (void)hipStreamSynchronize(st);
        g_defer = prev_defer;
        for (auto& f : deferred) getMemCacheRef().releaseAbtrtMem(f.p, f.bytes);
        deferred.clear();
    }
    if (hcnt && !fixed_slot) {
        std::lock_guard<std::mutex> g(g_host_mu);
        g_host_free.push_back(HostSlot{hcnt, hring, hring_dev});
    }
}

// One counter into a snapshot slot: one 64-bit store at system scope, so the
// host never sees a value without its sequence number.
__device__ inline void snap_store(unsigned long long* dst, unsigned seq, int v)
{
    __hip_atomic_store(dst, ((unsigned long long)seq << 32) | (unsigned)v, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ inline void round_snap_store(const RoundSnap& s)
{
    if (s.dst && blockIdx.x == 0 && threadIdx.x < C_NUM) {
        const int j = threadIdx.x;
        snap_store(&s.dst[j], s.seq, j == S_ERR ? *s.err : (j < ROUND_WORDS ? s.set[j * ROUND_LINE] : 0));
    }
}

__global__ __launch_bounds__(kBlock) void k_rounds_start(int* ring, int next, int base)
{
    static_assert(ROUND_INTS == kBlock, "a workgroup per set");
    const int i = blockIdx.x * kBlock + threadIdx.x;
    ring[i] = i == R_NEXT ? next : (i == ROUND_INTS + R_BASE ? base : 0);
}

// the counters straight into the mapped pinned ring (a kernel costs less
// than a copy-engine transfer)
__global__ void k_snap(const int* cnt, unsigned long long* dst, unsigned seq)
{
    snap_store(&dst[threadIdx.x], seq, cnt[threadIdx.x]);
}

namespace {
// process-wide, so a slot reused by another context never matches old words
std::atomic<unsigned> g_snap_seq{0};
}  // namespace

unsigned Ctx::snap_begin(int slot)
{
    unsigned s = ++g_snap_seq;
    if (s == 0) s = ++g_snap_seq;
    ring_seq[slot] = s;
    return s;
}

void Ctx::snapshot(int slot)
{
    unsigned seq = snap_begin(slot);
    k_snap<<<1, C_NUM, 0, st>>>(dcnt.p, snap_dst(slot), seq);
    GCDT_LAUNCH_CHECK();
}

const int* Ctx::wait_snapshot(int slot)
{
    const unsigned long long* p = hring + C_NUM * slot;
    const unsigned want = ring_seq[slot];
    int* out = hsnap[slot];
    auto complete = [&]() {
        for (int i = 0; i < C_NUM; i++) {
            unsigned long long v = __atomic_load_n(p + i, __ATOMIC_ACQUIRE);
            if ((unsigned)(v >> 32) != want) return false;
            out[i] = (int)(unsigned)v;
        }
        return true;
    };
    for (unsigned spin = 1;; ++spin) {
        if (complete()) return out;
        if ((spin & 1023) == 0) {
            // the words can be missing only while their kernel is queued or
            // running: a device error or a drained stream without them ends
            // the wait
            hipError_t e = hipStreamQuery(st);
            if (e == hipSuccess) {
                if (complete()) return out;
                throw Error(GCDT_ERR_INTERNAL, "counter snapshot missing");
            }
            if (e != hipErrorNotReady) GCDT_HIP(e);
        }
    }
}

void Ctx::rounds_start(int next, int base)
{
    ring.ensure(ROUND_SETS * ROUND_INTS);
    k_rounds_start<<<ROUND_SETS, kBlock, 0, st>>>(ring.p, next, base);
    GCDT_LAUNCH_CHECK();
}

void Ctx::rounds_turn(int r)
{
    // half way through one half of the ring the other half is cleared: its
    // rounds are done and read, and it comes into use half a half later
    constexpr int half = ROUND_SETS / 2;
    if (r % half == half / 2 && r > half)
        fill_i32(*this, ring.p + (r / half % 2 ? 0 : half * ROUND_INTS), 0, half * ROUND_INTS);
}

RoundSnap Ctx::round_snap(int r)
{
    RoundSnap s;
    s.seq = snap_begin(r & 1);
    s.dst = snap_dst(r & 1);
    s.set = round_set(r);
    s.err = dcnt.p + C_ERR;
    return s;
}

// through the mapped ring and a poll: a copy and a stream synchronisation cost
// the host 15-20 us, this 8
void Ctx::read(int i, int k)
{
    snapshot(0);
    const int* h = wait_snapshot(0);
    for (int j = i; j < i + k; j++) hcnt[j] = h[j];
}

__global__ void k_set1(int* p, int v) { *p = v; }

void Ctx::set(int i, int v)
{
    k_set1<<<1, 1, 0, st>>>(dcnt.p + i, v);
    GCDT_LAUNCH_CHECK();
}

void Ctx::zero_counters() { fill_i32(*this, dcnt.p, 0, C_NUM); }

void Ctx::check_err()
{
    int e = get(C_ERR);
    if (e == 0) return;
    int status = GCDT_ERR_INTERNAL;
    if (e & MERR_CAPACITY) status = GCDT_ERR_CAPACITY;
    else if (e & (MERR_LOCATE | MERR_DUPLICATE)) status = GCDT_ERR_LOCATE;
    else if (e & MERR_CROSSING) status = GCDT_ERR_CROSSING;
    else if (e & MERR_SCRATCH) status = GCDT_ERR_SCRATCH;
    else if (e & MERR_INVALID) status = GCDT_ERR_INVALID;
    throw Error(status, "device consistency flag " + std::to_string(e));
}

// ================================================================== live kernel timing

namespace {
struct ProfRec {
    std::string name;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> ev;
    long long launches = 0;
    long long items = 0;
};
std::mutex g_prof_mu;
bool g_prof_on = false;
std::string g_prof_only;            // time only this kernel when not empty
std::vector<ProfRec> g_prof;
std::vector<hipEvent_t> g_ev_pool;  // events are reused across resets

bool take_event(hipEvent_t* e)
{
    if (!g_ev_pool.empty()) {
        *e = g_ev_pool.back();
        g_ev_pool.pop_back();
        return true;
    }
    return hipEventCreate(e) == hipSuccess;
}
}  // namespace

ProfScope::ProfScope(const char* name, hipStream_t s, long long items) : st(s)
{
    // no events (and no bookkeeping that allocates) inside an arena call
    if (!g_prof_on || g_arena) return;
    std::lock_guard<std::mutex> g(g_prof_mu);
    if (!g_prof_only.empty() && g_prof_only != name) return;
    for (size_t i = 0; i < g_prof.size(); i++)
        if (g_prof[i].name == name) slot = (int)i;
    if (slot < 0) {
        g_prof.push_back(ProfRec{name, {}, 0, 0});
        slot = (int)g_prof.size() - 1;
    }
    hipEvent_t a, b;
    if (!take_event(&a)) {
        slot = -1;
        return;
    }
    if (!take_event(&b)) {
        g_ev_pool.push_back(a);
        slot = -1;
        return;
    }
    (void)hipEventRecord(a, st);
    g_prof[slot].ev.push_back({a, b});
    g_prof[slot].launches++;
    g_prof[slot].items += items;
}

ProfScope::~ProfScope()
{
    if (slot < 0) return;
    std::lock_guard<std::mutex> g(g_prof_mu);
    (void)hipEventRecord(g_prof[slot].ev.back().second, st);
}

void prof_enable(bool on)
{
    std::lock_guard<std::mutex> g(g_prof_mu);
    g_prof_on = on;
}

void prof_reset()
{
    std::lock_guard<std::mutex> g(g_prof_mu);
    for (auto& r : g_prof)
        for (auto& e : r.ev) {
            (void)hipEventSynchronize(e.second);
            g_ev_pool.push_back(e.first);
            g_ev_pool.push_back(e.second);
        }
    g_prof.clear();
}

void prof_add_items(const char* name, long long items)
{
    if (!g_prof_on) return;
    std::lock_guard<std::mutex> g(g_prof_mu);
    for (auto& r : g_prof)
        if (r.name == name) {
            r.items += items;
            return;
        }
    // an item count without timed launches of its own (work done inside
    // another kernel's launches)
    g_prof.push_back(ProfRec{name, {}, 0, items});
}

void prof_only(const char* name)
{
    std::lock_guard<std::mutex> g(g_prof_mu);
    g_prof_only = name ? name : "";
}

// total ms, launches and items of one kernel (synchronises its events)
bool prof_read(const char* name, double* ms, long long* launches, long long* items)
{
    std::lock_guard<std::mutex> g(g_prof_mu);
    for (auto& r : g_prof) {
        if (r.name != name) continue;
        double t = 0;
        for (auto& e : r.ev) {
            (void)hipEventSynchronize(e.second);
            float f = 0;
            (void)hipEventElapsedTime(&f, e.first, e.second);
            t += f;
        }
        *ms = t;
        *launches = r.launches;
        *items = r.items;
        return true;
    }
    return false;
}

int prof_names(char* buf, int cap)
{
    std::lock_guard<std::mutex> g(g_prof_mu);
    std::string all;
    for (auto& r : g_prof) {
        all += r.name;
        all += ';';
    }
    if (buf && cap > 0) {
        int n = (int)std::min<size_t>(all.size(), (size_t)cap - 1);
        memcpy(buf, all.data(), n);
        buf[n] = 0;
    }
    return (int)all.size();
}

// ================================================================== primitives

__global__ __launch_bounds__(kBlock) void k_fill_i32(int* p, int v, long long n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ __launch_bounds__(kBlock) void k_fill_u64(unsigned long long* p, unsigned long long v, long long n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}

void fill_i32(Ctx& c, int* p, int v, long long n)
{
    if (n <= 0) return;
    k_fill_i32<<<grid_for(n), kBlock, 0, c.st>>>(p, v, n);
    GCDT_LAUNCH_CHECK();
}

void fill_u64(Ctx& c, unsigned long long* p, unsigned long long v, long long n)
{
    if (n <= 0) return;
    k_fill_u64<<<grid_for(n), kBlock, 0, c.st>>>(p, v, n);
    GCDT_LAUNCH_CHECK();
}

__global__ __launch_bounds__(kBlock) void k_fill_jobs(FillJobs f)
{
    const long long i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x, step = (long long)gridDim.x * blockDim.x;
    for (int j = 0; j < f.njobs; j++) {
        int* p = f.job[j].p;
        const long long n = f.job[j].n;
        const int v = f.job[j].v;
        const bool wide = ((unsigned long long)p & 15) == 0;  // buffers start 256-byte aligned, counters need not
        const long long n4 = wide ? n / 4 : 0;
        for (long long i = i0; i < n4; i += step) ((int4*)p)[i] = make_int4(v, v, v, v);
        for (long long i = 4 * n4 + i0; i < n; i += step) p[i] = v;
    }
}

void fill_jobs(Ctx& c, const FillJobs& f)
{
    long long most = 0;
    for (int j = 0; j < f.njobs; j++) most = std::max(most, f.job[j].n);
    if (most == 0) return;
    k_fill_jobs<<<grid_for((most + 3) / 4), kBlock, 0, c.st>>>(f);
    GCDT_LAUNCH_CHECK();
}

constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_TILE = kBlock * SCAN_ITEMS;
constexpr int SCAN_PAD(int i) { return i + (i >> 4); }

__device__ inline int block_excl_scan(int v, int& total)
{
    __shared__ int wsum[kBlock / 64];
    int lane = __lane_id(), w = threadIdx.x >> 6;
    int wt;
    int ex = wave_excl_scan(v, wt);
    if (lane == 0) wsum[w] = wt;
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < kBlock / 64; i++) {
        int s = wsum[i];
        if (i < w) base += s;
        tot += s;
    }
    __syncthreads();
    total = tot;
    return base + ex;
}

__global__ __launch_bounds__(kBlock) void k_scan_tile_sums(const int* in, long long n, int* sums)
{
    long long base = (long long)blockIdx.x * SCAN_TILE;
    int s = 0;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        long long i = base + (long long)j * kBlock + threadIdx.x;
        if (i < n) s += in[i];
    }
    int tot;
    block_excl_scan(s, tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

__global__ __launch_bounds__(1024) void k_scan_sums(int* sums, int nt, int* total, int* total2)
{
    __shared__ int wsum[16];
    __shared__ int carry_s;
    if (threadIdx.x == 0) carry_s = 0;
    __syncthreads();
    for (int base = 0; base < nt; base += 1024) {
        int i = base + threadIdx.x;
        int v = i < nt ? sums[i] : 0;
        int lane = __lane_id(), w = threadIdx.x >> 6;
        int wt;
        int ex = wave_excl_scan(v, wt);
        if (lane == 0) wsum[w] = wt;
        __syncthreads();
        int pre = 0, tot = 0;
        for (int q = 0; q < 16; q++) {
            if (q < w) pre += wsum[q];
            tot += wsum[q];
        }
        int carry = carry_s;
        if (i < nt) sums[i] = carry + pre + ex;
        __syncthreads();
        if (threadIdx.x == 0) carry_s = carry + tot;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (total) *total = carry_s;
        if (total2) *total2 = carry_s;
    }
}

// OWN: sums[] holds the tiles' own totals and each workgroup adds up those
// before it (and the last one writes the grand total); else sums[] is scanned.
template <bool INCL, bool OWN>
__global__ __launch_bounds__(kBlock) void k_scan_apply(const int* in, int* out, long long n, const int* sums, int* total,
                                                       int* total2)
{
    __shared__ int tile[SCAN_PAD(SCAN_TILE)];
    __shared__ int s_pre;
    long long base = (long long)blockIdx.x * SCAN_TILE;
    if (OWN) {
        int v = 0, tot;
        for (int i = threadIdx.x; i < (int)blockIdx.x; i += kBlock) v += sums[i];
        block_excl_scan(v, tot);
        if (threadIdx.x == 0) {
            s_pre = tot;
            if (blockIdx.x == gridDim.x - 1) {
                if (total) *total = tot + sums[blockIdx.x];
                if (total2) *total2 = tot + sums[blockIdx.x];
            }
        }
        __syncthreads();
    } else if (threadIdx.x == 0) {
        s_pre = sums[blockIdx.x];
    }
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        int li = j * kBlock + threadIdx.x;
        long long i = base + li;
        tile[SCAN_PAD(li)] = i < n ? in[i] : 0;
    }
    __syncthreads();
    int v[SCAN_ITEMS];
    int s = 0;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        v[j] = tile[SCAN_PAD(threadIdx.x * SCAN_ITEMS + j)];
        s += v[j];
    }
    int tot;
    const int pre = block_excl_scan(s, tot);  // its barriers order s_pre too
    int run = s_pre + pre;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        run += INCL ? v[j] : 0;
        tile[SCAN_PAD(threadIdx.x * SCAN_ITEMS + j)] = run;
        run += INCL ? 0 : v[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        int li = j * kBlock + threadIdx.x;
        long long i = base + li;
        if (i < n) out[i] = tile[SCAN_PAD(li)];
    }
}

// A whole scan of up to SCAN_ONE ints in one workgroup.
constexpr int SCAN_ONE = 16384;

template <bool INCL>
__global__ __launch_bounds__(1024) void k_scan_one(const int* in, int* out, int n, int* total, int* total2)
{
    __shared__ int wsum[16];
    int carry = 0;
    for (int base = 0; base < n; base += 4096) {
        const int i = base + 4 * (int)threadIdx.x;
        int v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = i + j < n ? in[i + j] : 0;
        int wt;
        const int sum = v[0] + v[1] + v[2] + v[3];
        const int ex = wave_excl_scan(sum, wt);
        if (__lane_id() == 0) wsum[threadIdx.x >> 6] = wt;
        __syncthreads();
        int pre = 0, tot = 0;
        for (int q = 0; q < 16; q++) {
            if (q < (int)(threadIdx.x >> 6)) pre += wsum[q];
            tot += wsum[q];
        }
        int run = carry + pre + ex;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            run += INCL ? v[j] : 0;
            if (i + j < n) out[i + j] = run;
            run += INCL ? 0 : v[j];
        }
        carry += tot;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (total) *total = carry;
        if (total2) *total2 = carry;
    }
}

long long scan_scratch_ints(long long n) { return (n + SCAN_TILE - 1) / SCAN_TILE + 1; }

// Exclusive (inclusive when incl) scan of in[0..n) into out[0..n); the total
// goes to dcnt[C_TOTAL] and, when total_at_end, also to out[n] (out must then
// hold n+1 ints).
static void scan_impl(Ctx& c, const int* in, int* out, long long n, bool total_at_end, bool incl = false)
{
    if (n <= 0) {
        c.set(C_TOTAL, 0);
        if (total_at_end) {
            k_set1<<<1, 1, 0, c.st>>>(out, 0);
            GCDT_LAUNCH_CHECK();
        }
        return;
    }
    int *total = c.dcnt.p + C_TOTAL, *total2 = total_at_end ? out + n : nullptr;
    long long nt = (n + SCAN_TILE - 1) / SCAN_TILE;
    int* sums;
    if (c.ext_scratch) {
        if (c.ext_scratch_bytes < sizeof(int) * (size_t)(nt + 1))
            throw Error(GCDT_ERR_SCRATCH, "caller scratch too small for a scan of " + std::to_string(n));
        sums = c.ext_scratch;
    } else {
        c.scan_sums.ensure((size_t)nt + 1);
        sums = c.scan_sums.p;
    }
    // one launch up to SCAN_ONE ints; two up to 4,096 tiles, whose totals every
    // workgroup can add up itself; else a launch between them for the totals
    if (n <= SCAN_ONE) {
        if (incl)
            k_scan_one<true><<<1, 1024, 0, c.st>>>(in, out, (int)n, total, total2);
        else
            k_scan_one<false><<<1, 1024, 0, c.st>>>(in, out, (int)n, total, total2);
        GCDT_LAUNCH_CHECK();
        return;
    }
    k_scan_tile_sums<<<(unsigned)nt, kBlock, 0, c.st>>>(in, n, sums);
    GCDT_LAUNCH_CHECK();
    if (nt <= 4096) {
        if (incl)
            k_scan_apply<true, true><<<(unsigned)nt, kBlock, 0, c.st>>>(in, out, n, sums, total, total2);
        else
            k_scan_apply<false, true><<<(unsigned)nt, kBlock, 0, c.st>>>(in, out, n, sums, total, total2);
        GCDT_LAUNCH_CHECK();
        return;
    }
    k_scan_sums<<<1, 1024, 0, c.st>>>(sums, (int)nt, total, total2);
    GCDT_LAUNCH_CHECK();
    if (incl)
        k_scan_apply<true, false><<<(unsigned)nt, kBlock, 0, c.st>>>(in, out, n, sums, nullptr, nullptr);
    else
        k_scan_apply<false, false><<<(unsigned)nt, kBlock, 0, c.st>>>(in, out, n, sums, nullptr, nullptr);
    GCDT_LAUNCH_CHECK();
}

void scan_excl(Ctx& c, const int* in, int* out, long long n) { scan_impl(c, in, out, n, false); }
void scan_incl(Ctx& c, const int* in, int* out, long long n) { scan_impl(c, in, out, n, false, true); }
void scan_excl_total(Ctx& c, const int* in, int* out, long long n) { scan_impl(c, in, out, n, true); }

// ================================================================== square / sample

constexpr int GRID_R = (1 << 30) - 1;

__device__ inline void square_corners(int2* pts, int n)
{
    pts[n] = make_int2(0, 0);
    pts[n + 1] = make_int2(GRID_R, 0);
    pts[n + 2] = make_int2(GRID_R, GRID_R);
    pts[n + 3] = make_int2(0, GRID_R);
}

// rawMesh.cu:16-21: (N,N+1,N+3) and (N+1,N+2,N+3) split along the anti-diagonal
__device__ inline void square_seeds(int3* tri, int3* adj, int n)
{
    tri[0] = make_int3(n, n + 1, n + 3);
    tri[1] = make_int3(n + 1, n + 2, n + 3);
    adj[0] = make_int3(1, -1, -1);
    adj[1] = make_int3(-1, 0, -1);
}

__global__ void k_init_square(int2* pts, int3* tri, int3* adj, int n)
{
    square_corners(pts, n);
    square_seeds(tri, adj, n);
}

__device__ inline bool point_inside(int2 p) { return p.x > 0 && p.y > 0 && p.x < GRID_R && p.y < GRID_R; }

__global__ __launch_bounds__(kBlock) void k_check_points(const int2* pts, int n, int* err)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        if (!point_inside(pts[i])) atomicOr(err, MERR_INVALID);
}

void check_points(Ctx& c, const int2* pts, int n)
{
    if (n <= 0) return;
    k_check_points<<<grid_for(n), kBlock, 0, c.st>>>(pts, n, c.dcnt.p + C_ERR);
    GCDT_LAUNCH_CHECK();
    c.check_err();
}

void init_square(Ctx& c, int2* pts, int3* tri, int3* adj, int n)
{
    k_init_square<<<1, 1, 0, c.st>>>(pts, tri, adj, n);
    GCDT_LAUNCH_CHECK();
}

__global__ void k_write_corners(int2* pts, int n) { square_corners(pts, n); }

void write_corners(Ctx& c, int2* pts, int n)
{
    k_write_corners<<<1, 1, 0, c.st>>>(pts, n);
    GCDT_LAUNCH_CHECK();
}

constexpr int LOG_SAMPLE = 8;   // math_base.cuh:24 logSample
constexpr int LOG_BITMAP = 10;  // math_base.cuh:25 logBitmap
constexpr int SAMPLE_CELLS = 1 << (2 * LOG_SAMPLE);
constexpr int BITMAP_CELLS = 1 << (2 * LOG_BITMAP);

// Cell grid of the point-location bitmap ("boostmap") that the reference's entry
// points build and read: 1024x1024 cells over the square (math_base.cuh:25
// logBitmap).
struct GridOne {
    static constexpr int LOG = LOG_BITMAP;
    __device__ long long tri_base(const int3&) const { return 0; }
    __device__ long long pt_base(int) const { return 0; }
};

template <class G>
__device__ inline long long pt_cell(const G& g, int p, int2 P)
{
    return g.pt_base(p) + ((long long)(P.x >> (30 - G::LOG)) << G::LOG) + (P.y >> (30 - G::LOG));
}

__global__ __launch_bounds__(kBlock) void k_sample_cells(const int2* pts, int n, int* cellmin)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        int2 p = pts[i];
        int cell = ((p.x >> (30 - LOG_SAMPLE)) << LOG_SAMPLE) + (p.y >> (30 - LOG_SAMPLE));
        atomicMin(&cellmin[cell], (int)i);
    }
}

__global__ __launch_bounds__(kBlock) void k_sample_flags(const int* cellmin, int* flags)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < SAMPLE_CELLS; i += gridDim.x * blockDim.x)
        flags[i] = cellmin[i] != INT_MAX;
}

__global__ __launch_bounds__(kBlock) void k_sample_emit(const int2* pts, const int* cellmin, const int* offs, int* ids,
                                                        int2* spts)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < SAMPLE_CELLS; i += gridDim.x * blockDim.x) {
        int p = cellmin[i];
        if (p != INT_MAX) {
            int o = offs[i];
            if (ids) ids[o] = p;
            if (spts) spts[o] = pts[p];
        }
    }
}

int sample_points(Ctx& c, const int2* pts, int n, int* sample_ids, int2* sample_pts)
{
    DBuf<int> cellmin(SAMPLE_CELLS), offs(SAMPLE_CELLS + 1);
    fill_i32(c, cellmin.p, INT_MAX, SAMPLE_CELLS);
    if (n > 0) {
        k_sample_cells<<<grid_for(n), kBlock, 0, c.st>>>(pts, n, cellmin.p);
        GCDT_LAUNCH_CHECK();
    }
    k_sample_flags<<<grid_for(SAMPLE_CELLS), kBlock, 0, c.st>>>(cellmin.p, offs.p);
    GCDT_LAUNCH_CHECK();
    scan_excl(c, offs.p, offs.p, SAMPLE_CELLS);
    k_sample_emit<<<grid_for(SAMPLE_CELLS), kBlock, 0, c.st>>>(pts, cellmin.p, offs.p, sample_ids, sample_pts);
    GCDT_LAUNCH_CHECK();
    return c.get(C_TOTAL);
}

// ================================================================== Morton order

// 20-bit Morton code of the 1024x1024 cell of a 2^30-grid point
__device__ inline unsigned morton_cell(int2 p)
{
    unsigned x = (unsigned)p.x >> 20, y = (unsigned)p.y >> 20;
    x = (x | (x << 8)) & 0x00FF00FFu;
    x = (x | (x << 4)) & 0x0F0F0F0Fu;
    x = (x | (x << 2)) & 0x33333333u;
    x = (x | (x << 1)) & 0x55555555u;
    y = (y | (y << 8)) & 0x00FF00FFu;
    y = (y | (y << 4)) & 0x0F0F0F0Fu;
    y = (y | (y << 2)) & 0x33333333u;
    y = (y | (y << 1)) & 0x55555555u;
    return x | (y << 1);
}

// ---------------------------------------------------------------- order inside cells

// Counting sorts place the elements of one bucket in the order their atomics
// arrived.  Where that order reaches a decision (point ids key the insertion
// claims, triangle ids key the flip claims), each bucket's range is then
// reordered by a key of its own elements -- the input index of a point, the
// sorted vertex ids of a triangle -- so the order is the same on every run.
// The scatter writes one slot per position: (element, bucket) for triangles,
// (element, bucket, x, y) for points.  A bucket of up to CELL_RANK_MAX (256)
// elements is ranked by one lane per element, its key
// against every key of the bucket (all staged in LDS by the workgroup); buckets
// of up to CELL_BLOCK_MAX by one workgroup's bitonic sort in LDS; larger ones,
// which the count passes flag, by a merge sort of all their elements
// (cell_reorder_huge).
#ifndef GCDT_CELL_RANK_MAX
#define GCDT_CELL_RANK_MAX 256
#endif
#ifndef GCDT_CELL_BLOCK_MAX
#define GCDT_CELL_BLOCK_MAX 2048
#endif
constexpr int CELL_RANK_MAX = GCDT_CELL_RANK_MAX;
constexpr int CELL_BLOCK_MAX = GCDT_CELL_BLOCK_MAX;
static_assert(CELL_RANK_MAX <= CELL_BLOCK_MAX, "bucket caps");

// Points: the key is the input index; a position holds (index, cell, x, y),
// so placing a point writes its coordinates, its index and the inverse map
// without gathering the point again.
struct CellKeyPoint {
    struct Key {
        int a;
    };
    using Slot = int4;
    const int2* pts;  // input points (for the paths that place by element)
    int* perm;        // sorted position -> input index
    int2* out;        // sorted points
    int* inv;         // input index -> sorted position
    __device__ Key of(int e) const { return Key{e}; }
    __device__ static Key max_key() { return Key{INT_MAX}; }
    __device__ static bool less(const Key& x, const Key& y) { return x.a < y.a; }
    __device__ void put(long long pos, const Slot& e) const
    {
        perm[pos] = e.x;
        out[pos] = make_int2(e.z, e.w);
        inv[e.x] = (int)pos;
    }
    __device__ void put_elem(long long pos, int el) const
    {
        perm[pos] = el;
        out[pos] = pts[el];
        inv[el] = (int)pos;
    }
};

// Leaves: the key is the triangle's vertex ids, smallest first; a position
// holds (triangle, cell) and placing writes the triangle id and its
// destination.
struct CellKeyTri {
    const int3* tri;
    int* src;   // sorted position -> triangle
    int* dest;  // triangle -> sorted position
    using Key = int3;
    using Slot = int2;
    __device__ void put(long long pos, const Slot& e) const { put_elem(pos, e.x); }
    __device__ void put_elem(long long pos, int el) const
    {
        src[pos] = el;
        dest[el] = (int)pos;
    }
    __device__ Key of(int e) const
    {
        const int3 t = tri[e];
        const int a = min(t.x, min(t.y, t.z)), c = max(t.x, max(t.y, t.z));
        return make_int3(a, t.x + t.y + t.z - a - c, c);
    }
    __device__ static Key max_key() { return make_int3(INT_MAX, INT_MAX, INT_MAX); }
    __device__ static bool less(const Key& x, const Key& y)
    {
        return x.x < y.x || (x.x == y.x && (x.y < y.y || (x.y == y.y && x.z < y.z)));
    }
};

// eb[s] = (element, bucket, ...) at position s; a bucket's range is
// [end[b-1], end[b]) (end: inclusive scan).  Places (KF::put) each element of a
// bucket of up to CELL_RANK_MAX at its rank in the bucket's key order and
// every other element where it is; a bucket's first lane lists a bucket of
// CELL_RANK_MAX + 1 .. CELL_BLOCK_MAX for the workgroup pass.  The workgroup
// first stages the keys of every position its ranked buckets cover (its own
// kBlock positions and the parts of its edge buckets beyond them, at most
// CELL_RANK_MAX - 1 on either side), so the rank loops read only LDS.
template <class KF>
__global__ __launch_bounds__(kBlock) void k_cell_rank(KF kf, const int* end, const typename KF::Slot* eb, long long n,
                                                     int* big, int* nbig)
{
    using Key = typename KF::Key;
    using Slot = typename KF::Slot;
    __shared__ Key sk[kBlock + 2 * (CELL_RANK_MAX - 1)];
    __shared__ int s_lo, s_hi;
    for (long long s0 = (long long)blockIdx.x * kBlock; s0 < n; s0 += (long long)gridDim.x * kBlock) {
        const long long s = s0 + threadIdx.x;
        Slot e{};
        long long a = 0, k = 0;
        if (s < n) {
            e = eb[s];
            a = e.y ? end[e.y - 1] : 0;
            k = end[e.y] - a;
        }
        const bool rank = s < n && k > 1 && k <= CELL_RANK_MAX;
        if (threadIdx.x == 0) {
            s_lo = kBlock;
            s_hi = 0;
        }
        __syncthreads();
        // window [lo, hi) relative to s0: lo >= -(CELL_RANK_MAX - 1),
        // hi <= kBlock + CELL_RANK_MAX - 1
        {
            // one LDS atomic per wave: the wave's own bounds first
            int wl = rank ? (int)(a - s0) : kBlock, wh = rank ? (int)(a + k - s0) : 0;
            for (int d = 32; d > 0; d >>= 1) {
                wl = min(wl, __shfl_down(wl, d, 64));
                wh = max(wh, __shfl_down(wh, d, 64));
            }
            if (__lane_id() == 0 && wl < wh) {
                atomicMin(&s_lo, wl);
                atomicMax(&s_hi, wh);
            }
        }
        __syncthreads();
        const int lo = s_lo, hi = s_hi;
        // a lane stages its own key when its cell is ranked (the keys of
        // unranked positions are never read); the parts of the edge cells
        // beyond the workgroup's positions are staged in turn
        if (rank) sk[(int)threadIdx.x - lo] = kf.of(e.x);
        for (int t = lo + (int)threadIdx.x; t < 0; t += kBlock) sk[t - lo] = kf.of(eb[s0 + t].x);
        for (int t = kBlock + (int)threadIdx.x; t < hi; t += kBlock) sk[t - lo] = kf.of(eb[s0 + t].x);
        __syncthreads();
        bool list = false;
        if (s < n) {
            long long pos = s;
            if (rank) {
                const Key mine = sk[s - s0 - lo];
                const Key* w = sk + (a - s0 - lo);
                int r = 0;
                for (int q = 0; q < (int)k; q++) r += KF::less(w[q], mine) ? 1 : 0;
                pos = a + r;
            }
            kf.put(pos, e);
            list = s == a && k > CELL_RANK_MAX && k <= CELL_BLOCK_MAX;
        }
        const int p = wave_alloc(list ? 1 : 0, nbig);
        if (list) big[p] = e.y;
        __syncthreads();
    }
}

// one workgroup per listed bucket: a bitonic sort in LDS, padded to a power of
// two with largest keys, of the bucket's elements into its range of out[]
template <class KF>
__global__ __launch_bounds__(kBlock) void k_cell_sort_block(KF kf, const int* end, const int* big, const int* nbig,
                                                              const typename KF::Slot* eb)
{
    using Key = typename KF::Key;
    __shared__ int se[CELL_BLOCK_MAX];
    __shared__ Key sk[CELL_BLOCK_MAX];
    const int nb = *nbig;
    for (int q = blockIdx.x; q < nb; q += gridDim.x) {
        const int b = big[q];
        const int a = b ? end[b - 1] : 0, k = end[b] - a;
        int np2 = 1;
        while (np2 < k) np2 <<= 1;
        for (int i = threadIdx.x; i < np2; i += kBlock) {
            const int el = i < k ? eb[a + i].x : -1;
            se[i] = el;
            sk[i] = i < k ? kf.of(el) : KF::max_key();
        }
        for (int size = 2; size <= np2; size <<= 1) {
            for (int stride = size >> 1; stride > 0; stride >>= 1) {
                __syncthreads();
                for (int i = threadIdx.x; i < (np2 >> 1); i += kBlock) {
                    const int lo = 2 * i - (i & (stride - 1)), hi = lo + stride;
                    const bool up = (lo & size) == 0;
                    if (KF::less(sk[hi], sk[lo]) == up) {
                        const Key tk = sk[lo];
                        sk[lo] = sk[hi];
                        sk[hi] = tk;
                        const int te = se[lo];
                        se[lo] = se[hi];
                        se[hi] = te;
                    }
                }
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < k; i += kBlock) kf.put_elem(a + i, se[i]);
        __syncthreads();
    }
}

// Buckets of more than CELL_BLOCK_MAX elements (a dense cluster: the count
// passes flag them, so the common solve never takes this path) are sorted
// together as (bucket, key, element) items: the items of every such bucket,
// compacted in position order, are sorted in chunks of CELL_BLOCK_MAX in LDS
// and then merged pairwise, each item placing itself in the merged run by a
// binary search of the other run (keys are unique); item j of the sorted
// array goes back to the j-th flagged position.
template <class KF>
struct CellItem {
    typename KF::Key key;
    int bucket;
    int elem;
};

template <class KF>
__device__ inline bool item_less(const CellItem<KF>& x, const CellItem<KF>& y)
{
    return x.bucket < y.bucket || (x.bucket == y.bucket && KF::less(x.key, y.key));
}

template <class SLOT>
__global__ __launch_bounds__(kBlock) void k_cell_huge_flags(const int* end, const SLOT* eb, long long n, int* flag)
{
    for (long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x; s < n; s += (long long)gridDim.x * blockDim.x) {
        const int b = eb[s].y;
        flag[s] = end[b] - (b ? end[b - 1] : 0) > CELL_BLOCK_MAX ? 1 : 0;
    }
}

template <class KF>
__global__ __launch_bounds__(kBlock) void k_cell_huge_gather(KF kf, const typename KF::Slot* eb, long long n,
                                                             const int* flag,
                                                             const int* off, CellItem<KF>* items, int* pos)
{
    for (long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x; s < n; s += (long long)gridDim.x * blockDim.x) {
        if (!flag[s]) continue;
        const typename KF::Slot e = eb[s];
        const int j = off[s];
        items[j] = CellItem<KF>{kf.of(e.x), e.y, e.x};
        pos[j] = (int)s;
    }
}

// one workgroup per chunk of CELL_BLOCK_MAX items: bitonic sort in LDS, the
// last chunk padded with items above every real one
template <class KF>
__global__ __launch_bounds__(kBlock) void k_cell_chunk_sort(CellItem<KF>* items, long long m)
{
    using Item = CellItem<KF>;
    __shared__ Item sv[CELL_BLOCK_MAX];
    const long long nchunks = (m + CELL_BLOCK_MAX - 1) / CELL_BLOCK_MAX;
    for (long long q = blockIdx.x; q < nchunks; q += gridDim.x) {
        const long long a = q * CELL_BLOCK_MAX;
        const int k = (int)min((long long)CELL_BLOCK_MAX, m - a);
        int np2 = 1;
        while (np2 < k) np2 <<= 1;
        for (int i = threadIdx.x; i < np2; i += kBlock)
            sv[i] = i < k ? items[a + i] : Item{KF::max_key(), INT_MAX, -1};
        for (int size = 2; size <= np2; size <<= 1) {
            for (int stride = size >> 1; stride > 0; stride >>= 1) {
                __syncthreads();
                for (int i = threadIdx.x; i < (np2 >> 1); i += kBlock) {
                    const int lo = 2 * i - (i & (stride - 1)), hi = lo + stride;
                    const bool up = (lo & size) == 0;
                    if (item_less<KF>(sv[hi], sv[lo]) == up) {
                        const Item t = sv[lo];
                        sv[lo] = sv[hi];
                        sv[hi] = t;
                    }
                }
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < k; i += kBlock) items[a + i] = sv[i];
        __syncthreads();
    }
}

// runs of w sorted items, merged in pairs: an item at index i of its run goes
// to the pair's start + i + (items of the other run below it)
template <class KF>
__global__ __launch_bounds__(kBlock) void k_cell_merge(const CellItem<KF>* in, CellItem<KF>* out, long long m,
                                                       long long w)
{
    for (long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x; j < m; j += (long long)gridDim.x * blockDim.x) {
        const long long run = j / w, base = (run & ~1LL) * w;
        const long long o0 = (run ^ 1) * w, o1 = min(o0 + w, m);
        const CellItem<KF> x = in[j];
        long long lo = o0, hi = o1 > o0 ? o1 : o0;
        while (lo < hi) {
            const long long mid = (lo + hi) >> 1;
            if (item_less<KF>(in[mid], x)) lo = mid + 1;
            else hi = mid;
        }
        out[base + (j - run * w) + (lo - o0)] = x;
    }
}

template <class KF>
__global__ __launch_bounds__(kBlock) void k_cell_huge_put(KF kf, const CellItem<KF>* items, const int* pos, long long m)
{
    for (long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x; j < m; j += (long long)gridDim.x * blockDim.x)
        kf.put_elem(pos[j], items[j].elem);
}

template <class KF>
static void cell_reorder_huge(Ctx& c, const KF& kf, const int* end, const typename KF::Slot* eb, long long n)
{
    DBuf<int> flag((size_t)n), off((size_t)n + 1);  // the scan writes its total at off[n]
    k_cell_huge_flags<typename KF::Slot><<<grid_for(n), kBlock, 0, c.st>>>(end, eb, n, flag.p);
    GCDT_LAUNCH_CHECK();
    scan_excl_total(c, flag.p, off.p, n);
    const long long m = c.get(C_TOTAL);
    if (m <= 0) return;
    DBuf<CellItem<KF>> a((size_t)m), b((size_t)m);
    DBuf<int> pos((size_t)m);
    k_cell_huge_gather<KF><<<grid_for(n), kBlock, 0, c.st>>>(kf, eb, n, flag.p, off.p, a.p, pos.p);
    GCDT_LAUNCH_CHECK();
    flag.release();
    off.release();
    k_cell_chunk_sort<KF><<<1024, kBlock, 0, c.st>>>(a.p, m);
    GCDT_LAUNCH_CHECK();
    CellItem<KF>*x = a.p, *y = b.p;
    for (long long w = CELL_BLOCK_MAX; w < m; w <<= 1) {
        k_cell_merge<KF><<<grid_for(m), kBlock, 0, c.st>>>(x, y, m, w);
        GCDT_LAUNCH_CHECK();
        std::swap(x, y);
    }
    k_cell_huge_put<KF><<<grid_for(m), kBlock, 0, c.st>>>(kf, x, pos.p, m);
    GCDT_LAUNCH_CHECK();
}

// What the count passes leave in C_HUGE: CELL_LARGE when a bucket holds more than
// CELL_RANK_MAX elements, CELL_HUGE when one holds more than CELL_BLOCK_MAX.
enum : int { CELL_LARGE = 1, CELL_HUGE = 2 };
__device__ inline void count_large(int r, int* huge)
{
    if (r == CELL_RANK_MAX) atomicOr(huge, CELL_LARGE);
    if (r == CELL_BLOCK_MAX) atomicOr(huge, CELL_HUGE);
}

// eb[0..n): (element, bucket, ...), grouped by bucket.  Each element is
// placed (KF::put) at its position in the reordered order.  large: C_HUGE of
// the count pass; C_NQ was cleared before it.
template <class KF>
static void cell_reorder(Ctx& c, const KF& kf, const int* end, const typename KF::Slot* eb, long long n, int large)
{
    if (n <= 0) return;
    // a list entry per bucket above the rank cap: at most n / (cap + 1)
    DBuf<int> big((size_t)(n / (CELL_RANK_MAX + 1) + 1));
    k_cell_rank<KF><<<grid_for(n), kBlock, 0, c.st>>>(kf, end, eb, n, big.p, c.dcnt.p + C_NQ);
    GCDT_LAUNCH_CHECK();
    if (large & CELL_LARGE) {
        k_cell_sort_block<KF><<<1024, kBlock, 0, c.st>>>(kf, end, big.p, c.dcnt.p + C_NQ, eb);
        GCDT_LAUNCH_CHECK();
    }
    if (large & CELL_HUGE) cell_reorder_huge(c, kf, end, eb, n);
}

// Counting sort of points by 20-bit Morton cell: the count pass keeps the
// value its atomicAdd returns (the point's arrival rank in its cell) in
// inv[], the scatter writes (index, cell, x, y) at the cell's start plus that
// rank, and the per-cell reorder places each point by input index, writing
// the sorted points, perm and the inverse map.
// Points outside the square are flagged here and land in some cell (the caller
// fails before they are used).
__device__ inline int morton_cell_any(int2 p) { return (int)(morton_cell(p) & (BITMAP_CELLS - 1)); }

__global__ __launch_bounds__(kBlock) void k_morton_count(const int2* pts, int n, int* cnt, int* rank, int* huge, int* err)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const int2 p = pts[i];
        if (!point_inside(p)) atomicOr(err, MERR_INVALID);
        const int r = atomicAdd(&cnt[morton_cell_any(p)], 1);
        rank[i] = r;
        count_large(r, huge);
    }
}

// cell_end holds the inclusive scan of the counts: cell c starts at
// cell_end[c - 1] (0 for c = 0).
__global__ __launch_bounds__(kBlock) void k_morton_scatter(const int2* pts, int n, const int* cell_end,
                                                           const int* rank, int4* eb)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const int2 p = pts[i];
        const int cell = morton_cell_any(p);
        const int pos = (cell ? cell_end[cell - 1] : 0) + rank[i];
        eb[pos] = make_int4((int)i, cell, p.x, p.y);
    }
}

void morton_order(Ctx& c, const int2* pts, int n, int2* out, int* perm, int* inv, int* cell_end)
{
    FillJobs f;
    f.add(cell_end, 0, BITMAP_CELLS + 1);
    f.add(c.dcnt.p + C_HUGE, 0, 1);
    f.add(c.dcnt.p + C_NQ, 0, 1);
    fill_jobs(c, f);
    if (n <= 0) return;
    k_morton_count<<<grid_for(n), kBlock, 0, c.st>>>(pts, n, cell_end, inv, c.dcnt.p + C_HUGE, c.dcnt.p + C_ERR);
    GCDT_LAUNCH_CHECK();
    scan_incl(c, cell_end, cell_end, BITMAP_CELLS);
    DBuf<int4> eb((size_t)n);
    k_morton_scatter<<<grid_for(n), kBlock, 0, c.st>>>(pts, n, cell_end, inv, eb.p);
    GCDT_LAUNCH_CHECK();
    c.read(0, C_NUM);
    if (c.hcnt[C_ERR]) c.check_err();
    // inv held the arrival ranks; placing rewrites it as the inverse map
    cell_reorder(c, CellKeyPoint{pts, perm, out, inv}, cell_end, eb.p, n, c.hcnt[C_HUGE]);
}

// Sample of Morton-ordered points: the 256x256 sample cell with Morton index
// m covers the 16 consecutive 20-bit cells [16m, 16m+16), i.e. the sorted
// range [end[16m-1], end[16m+15]).  Its sample is its extreme point towards
// the nearer edges of the square: the smallest (x, y) in lexicographic order,
// with x taken as -x in the right half of the square and y as -y in the top
// half.  Any point of the cell serves location; the extreme one does not
// depend on the order of the sorted range, and on collinear rows and columns
// -- a lattice, or points clamped to the square's edge -- it puts the samples
// on the outermost lines, so the points between two samples split the edge
// joining them instead of fanning out from a sample off the line (a fan that
// Lawson flips unwind one row per round).
__device__ inline int sample_range_start(const int* cell_end, int m)
{
    return m ? cell_end[16 * m - 1] : 0;
}

__global__ __launch_bounds__(kBlock) void k_sample_morton_flags(const int* cell_end, int* flags)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < SAMPLE_CELLS; i += gridDim.x * blockDim.x)
        flags[i] = cell_end[16 * i + 15] > sample_range_start(cell_end, i);
}

// one wave per sample cell: its extreme point over the cell's sorted range
__global__ __launch_bounds__(kBlock) void k_sample_morton_emit(const int2* pts, const int* cell_end, const int* offs,
                                                               int* ids)
{
    const int lane = __lane_id();
    const int nwaves = (gridDim.x * blockDim.x) >> 6;
    for (int m = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; m < SAMPLE_CELLS; m += nwaves) {
        const int a = sample_range_start(cell_end, m), b = cell_end[16 * m + 15];
        if (b <= a) continue;  // wave-uniform
        // the cell's column and row (even and odd bits of its Morton index)
        unsigned cx = 0, cy = 0;
        for (int bit = 0; bit < 8; bit++) {
            cx |= (((unsigned)m >> (2 * bit)) & 1u) << bit;
            cy |= (((unsigned)m >> (2 * bit + 1)) & 1u) << bit;
        }
        const unsigned fx = cx >= 128 ? ~0u : 0u, fy = cy >= 128 ? ~0u : 0u;
        unsigned long long best = ~0ull;
        int bi = a;
        for (int i = a + lane; i < b; i += 64) {
            const int2 p = pts[i];
            const unsigned long long k = ((unsigned long long)((unsigned)p.x ^ fx) << 32) | ((unsigned)p.y ^ fy);
            if (k < best) {
                best = k;
                bi = i;
            }
        }
        unsigned long long w = best;
        for (int off = 32; off > 0; off >>= 1) {
            const unsigned long long o = __shfl(w, lane ^ off, 64);
            w = o < w ? o : w;
        }
        // points are distinct: exactly one lane holds the minimum
        const unsigned long long owner = __ballot(best == w);
        const int src = __ffsll((long long)owner) - 1;
        const int id = __shfl(bi, src, 64);
        if (lane == 0) ids[offs[m]] = id;
    }
}

int sample_points_morton(Ctx& c, const int2* pts, const int* cell_end, int* sample_ids, int* offs)
{
    k_sample_morton_flags<<<grid_for(SAMPLE_CELLS), kBlock, 0, c.st>>>(cell_end, offs);
    GCDT_LAUNCH_CHECK();
    scan_excl(c, offs, offs, SAMPLE_CELLS);
    // one wave per sample cell
    k_sample_morton_emit<<<grid_for(64LL * SAMPLE_CELLS), kBlock, 0, c.st>>>(pts, cell_end, offs, sample_ids);
    GCDT_LAUNCH_CHECK();
    return c.get(C_TOTAL);
}

__global__ __launch_bounds__(kBlock) void k_relabel_pairs(const int2* in, int C, const int* inv, int n, int2* out)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < C; i += (long long)gridDim.x * blockDim.x) {
        int2 e = in[i];
        // ids outside [0,n) are kept and rejected later by the constraint checks
        e.x = (e.x >= 0 && e.x < n) ? inv[e.x] : e.x;
        e.y = (e.y >= 0 && e.y < n) ? inv[e.y] : e.y;
        out[i] = e;
    }
}

__global__ __launch_bounds__(kBlock) void k_unmap_tris(int3* tri, int T, const int* perm, int n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < T; i += (long long)gridDim.x * blockDim.x) {
        int3 t = tri[i];
        t.x = t.x < n ? perm[t.x] : t.x;
        t.y = t.y < n ? perm[t.y] : t.y;
        t.z = t.z < n ? perm[t.z] : t.z;
        tri[i] = t;
    }
}

void relabel_pairs(Ctx& c, const int2* in, int C, const int* inv, int n, int2* out)
{
    if (C <= 0) return;
    k_relabel_pairs<<<grid_for(C), kBlock, 0, c.st>>>(in, C, inv, n, out);
    GCDT_LAUNCH_CHECK();
}

void unmap_tris(Ctx& c, int3* tri, int T, const int* perm, int n)
{
    if (T <= 0 || n <= 0) return;
    k_unmap_tris<<<grid_for(T), kBlock, 0, c.st>>>(tri, T, perm, n);
    GCDT_LAUNCH_CHECK();
}

// ================================================================== location

// initTriangle, rawMesh.cu:37-57: side of the anti-diagonal (R,0)-(0,R)
__global__ __launch_bounds__(kBlock) void k_locate_two(const int2* pts, int n, int* loc, int* pend)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        int o = orient2d(make_int2(GRID_R, 0), make_int2(0, GRID_R), pts[i]);
        loc[i] = o > 0 ? 3 : (o < 0 ? 4 + 3 : 0);  // tri 0 inside / tri 1 inside / edge opposite vertex 0 of tri 0
        pend[i] = (int)i;
    }
}

__global__ __launch_bounds__(kBlock) void k_seed_square(int2* pts, int n, int3* tri, int3* adj, const int* ids, int nids,
                                                        int* loc, int* pend)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        square_corners(pts, n);
        square_seeds(tri, adj, n);
    }
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < nids; i += (long long)gridDim.x * blockDim.x) {
        int p = ids[i];
        int o = orient2d(make_int2(GRID_R, 0), make_int2(0, GRID_R), pts[p]);
        loc[p] = o > 0 ? 3 : (o < 0 ? 4 + 3 : 0);
        pend[i] = p;
    }
}

void seed_square(Ctx& c, int2* pts, int n, int3* tri, int3* adj, const int* ids, int nids, int* loc, int* pend)
{
    k_seed_square<<<grid_for(nids), kBlock, 0, c.st>>>(pts, n, tri, adj, ids, nids, loc, pend);
    GCDT_LAUNCH_CHECK();
}

int locate_two(Ctx& c, const int2* pts, int n, int* loc, int* pend)
{
    if (n > 0) {
        k_locate_two<<<grid_for(n), kBlock, 0, c.st>>>(pts, n, loc, pend);
        GCDT_LAUNCH_CHECK();
    }
    return n;
}

__global__ __launch_bounds__(kBlock) void k_mark_vertices(const int3* tri, int T, int n, int* isv)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < T; i += (long long)gridDim.x * blockDim.x) {
        int3 t = tri[i];
        if (t.x < n) isv[t.x] = 1;
        if (t.y < n) isv[t.y] = 1;
        if (t.z < n) isv[t.z] = 1;
    }
}

// initTriangleBoost, rawMesh.cu:59-152: scan the triangles listed for the
// point's bitmap cell; the first whose closed region holds the point wins.
template <class G>
__global__ __launch_bounds__(kBlock) void k_locate_bitmap(G g, const int2* pts, int n, const int* isv, const int3* tri,
                                                          const int* bm_off, const int* bm_tri, int* loc, int* pend,
                                                          int* npend, int* err)
{
    __shared__ int s_buf[STAGE_CAP];
    __shared__ int s_base;
    Staged<STAGE_CAP> sp(s_buf, &s_base, pend, npend);
    TILE_LOOP(base, n, kBlock)
    {
        long long i = base + threadIdx.x;
        bool want = false;
        if (i < n) {
            int p = (int)i;
            if (isv[p]) {
                loc[p] = -1;
            } else {
                int2 P = pts[p];
                long long cell = pt_cell(g, p, P);
                int r = -1, t = -1;
                for (int j = bm_off[cell], e = bm_off[cell + 1]; j < e; j++) {
                    t = bm_tri[j];
                    int3 tv = tri[t];
                    r = classify(pts[tv.x], pts[tv.y], pts[tv.z], P);
                    if (r >= 0 || r == -2) break;
                }
                if (r >= 0) {
                    loc[p] = t * 4 + r;
                    want = true;
                } else {
                    loc[p] = -1;
                    atomicOr(err, r == -2 ? MERR_DUPLICATE : MERR_LOCATE);
                }
            }
        }
        int slot = sp.reserve(want ? 1 : 0);
        if (want) s_buf[slot] = (int)i;
    }
    sp.flush();
}

template <class G>
static int locate_bitmap_g(Ctx& c, const G& g, const int2* pts, int n, const int3* tri, int T, const int* bm_off,
                           const int* bm_tri, int* loc, int* isv, int* pend)
{
    k_mark_vertices<<<grid_for(T), kBlock, 0, c.st>>>(tri, T, n, isv);
    GCDT_LAUNCH_CHECK();
    c.set(C_NPEND, 0);
    if (n > 0) {
        ProfScope ps("locate_bitmap", c.st, n);
        k_locate_bitmap<G><<<grid_for(n), kBlock, 0, c.st>>>(g, pts, n, isv, tri, bm_off, bm_tri, loc, pend,
                                                             c.dcnt.p + C_NPEND, c.dcnt.p + C_ERR);
        GCDT_LAUNCH_CHECK();
    }
    c.read(0, C_NUM);
    if (c.hcnt[C_ERR]) c.check_err();
    return c.hcnt[C_NPEND];
}

int locate_bitmap(Ctx& c, const int2* pts, int n, const int3* tri, int T, const int* bm_off, const int* bm_tri,
                  int* loc, int* isv, int* pend)
{
    return locate_bitmap_g(c, GridOne{}, pts, n, tri, T, bm_off, bm_tri, loc, isv, pend);
}

// vertex -> a triangle of the mesh that has it (set for the mesh's vertices only)
__global__ __launch_bounds__(kBlock) void k_vertex_tri(const int3* tri, int T, int* vt)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < T; i += (long long)gridDim.x * blockDim.x) {
        const int3 t = tri[i];
        vt[t.x] = (int)i;
        vt[t.y] = (int)i;
        vt[t.z] = (int)i;
    }
}

// The sample of a point's own cell: of the whole square (sample_points_morton),
// or the first point of the instance's 16x16 cell (batch_sample_sorted).
struct CellSampleOne {
    const int *ids, *offs;
    __device__ int of(int, int2 P) const { return ids[offs[morton_cell(P) >> (2 * (LOG_BITMAP - LOG_SAMPLE))]]; }
};

struct CellSampleInst {
    const int *vinst, *cbase, *lvl, *cell_end;
    __device__ int of(int p, int2 P) const
    {
        const int inst = vinst[p], sh = 2 * (lvl[inst] - 4);
        const int f0 = cbase[inst] + ((int)(morton_cell(P) >> 12) << sh);  // 4 of 10 levels
        return f0 ? cell_end[f0 - 1] : 0;
    }
};

// A thread per point: from its cell's sample, across any edge that has the
// point strictly outside, to the triangle whose closed region holds it (on a
// Delaunay mesh such a walk ends).  Which of an edge's two triangles a point
// on it is recorded in does not matter (closeness_rank_edge).  Bound by the
// chain of loads, so it reads the sample mesh's flip records: one 64-byte line
// a triangle, where triangle and neighbours and then the three vertices were
// two loads in a row.
template <class S>
__global__ __launch_bounds__(kBlock) void k_locate_walk(S smp, const int2* pts, int n, const FRec* rec, int T,
                                                        const int* vt, int* loc, int* pend, int* npend, int* err)
{
    __shared__ int s_buf[STAGE_CAP];
    __shared__ int s_base;
    Staged<STAGE_CAP> sp(s_buf, &s_base, pend, npend);
    TILE_LOOP(base, n, kBlock)
    {
        const long long i = base + threadIdx.x;
        bool want = false;
        if (i < n) {
            const int p = (int)i;
            const int2 P = pts[p];
            const int v = smp.of(p, P);
            int r = -1, t = vt[v];
            if (v != p) {
                for (int g = 0; g < T && t >= 0; g++) {
                    const FRec x = rec_load(&rec[t]);
                    const int2 A = x.p[0], B = x.p[1], C = x.p[2];
                    const int o0 = orient2d(B, C, P), o1 = orient2d(C, A, P), o2 = orient2d(A, B, P);
                    if (o0 >= 0 && o1 >= 0 && o2 >= 0) {
                        const int z = (o0 == 0) + (o1 == 0) + (o2 == 0);
                        r = z == 0 ? 3 : (z > 1 ? -2 : (o0 == 0 ? 0 : (o1 == 0 ? 1 : 2)));
                        break;
                    }
                    t = o0 < 0 ? x.a.x : (o1 < 0 ? x.a.y : x.a.z);
                }
                want = true;  // also when not found: the list's length is known to the host
                if (r < 0) atomicOr(err, r == -2 ? MERR_DUPLICATE : MERR_LOCATE);
            }
            loc[p] = r >= 0 ? t * 4 + r : -1;
        }
        const int slot = sp.reserve(want ? 1 : 0);
        if (want) s_buf[slot] = (int)i;
    }
    sp.flush();
}

template <class S>
static void locate_walk_s(Ctx& c, const S& smp, const int2* pts, int n, long long nv, const int3* tri, const FRec* rec,
                          int T, int* loc, int* pend)
{
    if (n <= 0) return;
    DBuf<int> vt((size_t)nv);
    k_vertex_tri<<<grid_for(T), kBlock, 0, c.st>>>(tri, T, vt.p);
    GCDT_LAUNCH_CHECK();
    ProfScope ps("locate_walk", c.st, n);
    k_locate_walk<S><<<grid_for(n), kBlock, 0, c.st>>>(smp, pts, n, rec, T, vt.p, loc, pend, c.dcnt.p + C_NPEND,
                                                       c.dcnt.p + C_ERR);
    GCDT_LAUNCH_CHECK();
}

void locate_walk(Ctx& c, const int2* pts, int n, const int3* tri, const FRec* rec, int T, const int* ids,
                 const int* offs, int* loc, int* pend)
{
    locate_walk_s(c, CellSampleOne{ids, offs}, pts, n, (long long)n + 4, tri, rec, T, loc, pend);
}

void locate_walk_batch(Ctx& c, const int2* pts, const int* vinst, const int* cbase, const int* lvl, const int* cell_end,
                       long long NP, int K, const int3* tri, const FRec* rec, int T, int* loc, int* pend)
{
    locate_walk_s(c, CellSampleInst{vinst, cbase, lvl, cell_end}, pts, (int)NP, NP + 4LL * K, tri, rec, T, loc, pend);
}

// ================================================================== insertion rounds

// The claimed-triangle list of a round: the claim whose atomicMax finds a key
// of an older epoch is the triangle's first this round and appends it, so
// every claimed triangle is listed once and the split step walks these
// triangles instead of every pending point.
__device__ inline bool claim_first(unsigned long long old, unsigned epoch)
{
    return (unsigned)(old >> 44) != (epoch & 0xfffffu);
}

// Wave-combined claims: consecutive lanes that target the same triangle form
// a run (the pending list stays in near-Morton order, so early rounds have
// long runs); a segmented max over each run leaves the run's highest key in
// its first lane, which issues the run's only atomic.  *f1 / *f2 report
// whether this lane's claims on t / t2 came first this round.  All lanes must
// be active.
__device__ inline void claim_combined_w(unsigned long long* claim, int t, int t2, unsigned long long key,
                                        unsigned epoch, bool* f1, bool* f2)
{
    const int lane = __lane_id();
    const int prev = __shfl_up(t, 1, 64);
    const bool head = lane == 0 || prev != t;
    const unsigned long long heads = __ballot(head);
    const unsigned long long after = heads & ~((2ull << lane) - 1);
    const int end = after ? __ffsll((long long)after) - 2 : 63;  // last lane of this lane's run
    unsigned long long v = t >= 0 ? key : 0ull;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        unsigned long long o = __shfl_down(v, d, 64);
        if (lane + d <= end) v = o > v ? o : v;
    }
    *f1 = head && t >= 0 && claim_first(atomicMax(&claim[t], v), epoch);
    *f2 = t2 >= 0 && claim_first(atomicMax(&claim[t2], key), epoch);
}

// Claims of `epoch` for up to IT points per thread (l: their places, < 0 none;
// close: their closeness there), appending first-claimed triangles to wl.
// Block-uniform: every thread of the block calls it.
template <int IT>
__device__ inline void claim_items(const Ins& s, const int (&p)[IT], const int (&l)[IT], const unsigned (&close)[IT],
                                   unsigned epoch, Staged<STAGE_CAP>& sw)
{
    int wt[2 * IT];
    int nq = 0;
#pragma unroll
    for (int j = 0; j < IT; j++) {
        int t = -1, t2 = -1;
        unsigned long long key = 0;
        if (l[j] >= 0) {
            const int k = l[j] & 3;
            t = l[j] >> 2;
            key = ins_key(p[j], k < 3, close[j], epoch);
            if (k < 3) t2 = ins_edge_neighbour(s, t, k);
        }
        bool f1, f2;
        claim_combined_w(s.claim, t, t2, key, epoch, &f1, &f2);
        wt[2 * j] = f1 ? t : -1;
        wt[2 * j + 1] = f2 ? t2 : -1;
        nq += (wt[2 * j] >= 0) + (wt[2 * j + 1] >= 0);
    }
    int b = sw.reserve(nq);
#pragma unroll
    for (int j = 0; j < 2 * IT; j++)
        if (wt[j] >= 0) sw.buf[b++] = wt[j];
}

// The first tile's entries of a list, read beside its length (which a launch
// otherwise waits for alone): entries past the length are read and not used.
template <int IT>
__device__ inline void first_tile(const int* list, long long cap, long long bid, int (&v)[IT])
{
#pragma unroll
    for (int j = 0; j < IT; j++) {
        const long long i = bid * kBlock * IT + j * kBlock + threadIdx.x;
        v[j] = list && i < cap ? list[i] : 0;
    }
}
#define TILE_ITEM(list, first, base, bid, i, j, IT) \
    ((base) == (long long)(bid)*kBlock * (IT) ? (first)[j] : (list)[i])

// First claims of a run of rounds (later rounds claim inside k_ins_reloc).
__global__ __launch_bounds__(kBlock) void k_ins_claim_w(Ins s, const int* list, const int* cnt, unsigned epoch, int* wl,
                                                        int* nw, int wcap)
{
    __shared__ int s_buf[STAGE_CAP];
    __shared__ int s_base;
    Staged<STAGE_CAP> sw(s_buf, &s_base, wl, nw, wcap, s.err, MERR_CAPACITY);
    int n = *cnt;
    TILE_LOOP(base, n, kBlock)
    {
        long long i = base + threadIdx.x;
        int p[1] = {-1}, l[1] = {-1};
        unsigned close[1] = {0};
        if (i < n) {
            p[0] = list[i];
            l[0] = s.loc[p[0]];
            if (l[0] >= 0) {
                const int3 tv = s.m.tri[l[0] >> 2];
                close[0] = ins_close(s, s.m.pts[tv.x], s.m.pts[tv.y], s.m.pts[tv.z], s.m.pts[p[0]], p[0], l[0] & 3);
            }
        }
        claim_items<1>(s, p, l, close, epoch, sw);
    }
    sw.flush();
}

// Items per thread of the block-appending list kernels: 1, 2 or 4 (tunable;
// more items amortise the block-wide append, fewer keep more waves in flight).
template <class F>
void with_items(int v, F&& f)
{
    if (v == 1) f(std::integral_constant<int, 1>{});
    else if (v == 2) f(std::integral_constant<int, 2>{});
    else f(std::integral_constant<int, 4>{});
}

// Splits for the round's claimed triangles: a triangle's claim word names its
// winning point; an on-edge winner splits from its own triangle (loc), not
// from the second one it claimed.
template <int INS_ITEMS>
__global__ __launch_bounds__(kBlock) void k_ins_split(Ins s, const int* list, const int* cnt, int lcap, int* set,
                                                      RoundSnap snap)
{
    round_snap_store(snap);
    int pre[INS_ITEMS];
    first_tile(list, lcap, blockIdx.x, pre);
    int n = min(*cnt, lcap);  // an overfull list has flagged MERR_CAPACITY
    const int first = set[R_BASE];
    TILE_LOOP(base, n, kBlock * INS_ITEMS)
    {
        int pp[INS_ITEMS], ll[INS_ITEMS], need[INS_ITEMS];
        int tot = 0;
#pragma unroll
        for (int j = 0; j < INS_ITEMS; j++) {
            long long i = base + (long long)j * kBlock + threadIdx.x;
            pp[j] = -1;
            need[j] = 0;
            if (i < n) {
                const int t = TILE_ITEM(list, pre, base, blockIdx.x, i, j, INS_ITEMS);
                const unsigned long long w = s.claim[t];
                const int p = (int)(unsigned)w;
                const int l = s.loc[p];
                if (l >= 0 && (l >> 2) == t) {
                    const int k = l & 3;
                    pp[j] = p;
                    ll[j] = l;
                    need[j] = k == 3 ? 3 : (s.claim[A3(s.m, t, k)] == w ? 4 : 0);
                }
            }
            tot += need[j];
        }
        int b = first + block_alloc<kBlock>(tot, &set[R_NEW]);
#pragma unroll
        for (int j = 0; j < INS_ITEMS; j++) {
            if (need[j]) {
                if (b + need[j] > s.cap) atomicOr(s.err, MERR_CAPACITY);
                else ins_split_at(s, pp[j], ll[j], b);
                b += need[j];
            }
        }
    }
}

// rounds of at most this many points settle and relocate in workgroups of their
// own: both halves are then on the chip at once
#ifndef GCDT_INS_SPLIT_MAX
#define GCDT_INS_SPLIT_MAX 131072
#endif
constexpr int INS_SPLIT_MAX = GCDT_INS_SPLIT_MAX;

// Outer adjacency of the round's new triangles (their slots follow from the
// round's counters), then the relocation of the pending points, fused with the
// next round's claims (epoch next_ep) and its claimed-triangle list.  Only the
// claims of on-edge points read adjacency, and they resolve entries that this
// launch has not settled yet (ins_edge_neighbour).  The slots of the next round
// begin where this round's end.
//
// split: even workgroups relocate, odd ones settle.  Both are chains of three to
// five trips to memory, which a small round is made of (12 rounds of 20,000
// points 124 -> 105 us); a large one is better off settling first, while the
// lines that the splits wrote are near (10M points 2.70 ms, split 3.14).
template <int INS_ITEMS>
__global__ __launch_bounds__(kBlock) void k_ins_reloc(Ins s, const int* list, const int* cnt, int lcap, int split, int* list2,
                                                      unsigned next_ep, int* wl, int wcap, int* set, int* next_set)
{
    __shared__ int s_buf[STAGE_CAP], s_buf2[STAGE_CAP];
    __shared__ int s_base, s_base2;
    Staged<STAGE_CAP> sl(s_buf, &s_base, list2, &set[R_NEXT]),
        sw(s_buf2, &s_base2, wl, &set[R_NW], wcap, s.err, MERR_CAPACITY);
    const long long bid = split ? blockIdx.x >> 1 : blockIdx.x, nblk = split ? gridDim.x >> 1 : gridDim.x;
    int pre[INS_ITEMS];
    first_tile(list, lcap, bid, pre);
    if (!split || (blockIdx.x & 1)) {
        const int tb = set[R_BASE], te = tb + set[R_NEW];
        if (bid == 0 && threadIdx.x == 0) next_set[R_BASE] = te;
        for (long long i = bid * kBlock + threadIdx.x + tb; i < min(te, s.cap); i += nblk * kBlock) ins_fix(s, (int)i);
        if (split) return;
    }
    int n = *cnt;
    for (long long base = bid * kBlock * INS_ITEMS; base < n; base += nblk * kBlock * INS_ITEMS) {
        int p[INS_ITEMS], l[INS_ITEMS];
        unsigned close[INS_ITEMS];
        int tot = 0;
#pragma unroll
        for (int j = 0; j < INS_ITEMS; j++) {
            long long i = base + (long long)j * kBlock + threadIdx.x;
            l[j] = -1;
            if (i < n) {
                p[j] = TILE_ITEM(list, pre, base, bid, i, j, INS_ITEMS);
                const int at = s.loc[p[j]];
                int to = at;
                if (at >= 0 && ins_relocate_at<CLAIM_LAUNCH, true>(s, p[j], &to, &close[j])) {
                    if (to != at) s.loc[p[j]] = to;
                    l[j] = to;
                }
            }
            tot += l[j] >= 0;
        }
        int b = sl.reserve(tot);
#pragma unroll
        for (int j = 0; j < INS_ITEMS; j++)
            if (l[j] >= 0) s_buf[b++] = p[j];
        claim_items<INS_ITEMS>(s, p, l, close, next_ep, sw);
    }
    flush_both(sl, sw);
}

// ---- persistent single-workgroup tail: all remaining insertion rounds in one
// launch (block barriers between the phases, LDS counters for the lists)
constexpr int TAIL_BS = 1024;

// What a persistent tail hands to the host ring in place of the counters: one
// word per thread, the others 0.
__device__ inline void tail_snap(const RoundSnap& snap, int n, int r, int err, int ntri, int flips, int props)
{
    const int j = threadIdx.x;
    if (j >= C_NUM) return;
    int v = j == C_TAIL_N ? n : j == C_TAIL_R ? r : j == C_TAIL_ERR ? err : j == C_NTRI ? ntri : j == C_TAIL_F ? flips : j == C_TAIL_P ? props : 0;
    if (j == C_ERR) v = __hip_atomic_load(snap.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    snap_store(&snap.dst[j], snap.seq, v);
}

// Insertion rounds of at most INS_LIST points in one workgroup.  A round is a
// chain of waits, so it is kept short: the list holds each point with its place
// and closeness, in LDS; the claims stay in the workgroup's own L2; two
// barriers a round; and a point that has moved claims its new triangle from the
// vertices it was just located by, while the last waves settle the outer
// adjacency of the round's new triangles (ins_edge_neighbour).
// Returns the points left (0 unless the round limit or an error stops it).
// Up to 4,096 points, where the tail starts by default and the two lists fill
// 96 KB: 2,100 points from the seeds 235 -> 112 us, of which the first seven
// rounds are 10 us each, bound by one CU's instruction rate, and the last six 3
// us each, a chain of about six trips to its L2.
#ifndef GCDT_INS_LIST
#define GCDT_INS_LIST 4096
#endif
constexpr int INS_LIST = GCDT_INS_LIST;

struct InsList {
    int p[INS_LIST];
    int l[INS_LIST];
    unsigned close[INS_LIST];
};

// p's claims (l < 0: none).  Combined over runs of lanes as claim_combined_w
// (all lanes active): 2,100 points on the same few triangles are 31 us of
// atomics on one word without it.
__device__ inline void ins_claim_wg(const Ins& s, int p, int l, unsigned close, unsigned ep)
{
    const int lane = __lane_id();
    const int t = l < 0 ? -1 : l >> 2, k = l & 3;
    const unsigned long long key = ins_key(p, k < 3, close, ep);
    const int prev = __shfl_up(t, 1, 64);
    const bool head = lane == 0 || prev != t;
    const unsigned long long heads = __ballot(head);
    const unsigned long long after = heads & ~((2ull << lane) - 1);
    const int end = after ? __ffsll((long long)after) - 2 : 63;  // last lane of this lane's run
    unsigned long long v = key;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long o = __shfl_down(v, d, 64);
        if (lane + d <= end) v = o > v ? o : v;
    }
    if (t < 0) return;
    if (head) at_max_wg(&s.claim[t], v);
    if (k < 3) {
        const int t2 = ins_edge_neighbour(s, t, k);
        if (t2 >= 0) at_max_wg(&s.claim[t2], key);
    }
}

__device__ inline int ins_short_rounds(const Ins& s, const int* P, int n, InsList* s_list, int* s_np, int* s_nt, unsigned& ep,
                                       int max_rounds, int& r, int& err)
{
    for (int i0 = 0; i0 < n; i0 += TAIL_BS) {
        const int i = i0 + (int)threadIdx.x;
        int p = -1, l = -1;
        unsigned close = 0;
        if (i < n) {
            p = P[i];
            l = s.loc[p];
            if (l >= 0) {
                const int3 tv = s.m.tri[l >> 2];
                close = ins_close(s, s.m.pts[tv.x], s.m.pts[tv.y], s.m.pts[tv.z], s.m.pts[p], p, l & 3);
            }
            s_list[0].p[i] = p;
            s_list[0].l[i] = l;
            s_list[0].close[i] = close;
        }
        ins_claim_wg(s, p, l, close, ep);
    }
    if (threadIdx.x < 2) s_np[threadIdx.x] = 0;
    int tb = *s_nt;
    __syncthreads();
    for (int q = 0; n > 0 && r < max_rounds; q ^= 1) {
        InsList &in = s_list[q], &out = s_list[q ^ 1];
        for (int i0 = 0; i0 < n; i0 += TAIL_BS) {
            const int i = i0 + (int)threadIdx.x;
            int p = -1, l = -1, need = 0;
            if (i < n) {
                p = in.p[i];
                l = in.l[i];
            }
            if (l >= 0) {
                const int t = l >> 2, k = l & 3;
                const unsigned long long key = ins_key(p, k < 3, in.close[i], ep);
                if (ld_u64_wg(&s.claim[t]) == key)
                    need = k == 3 ? 3 : (ld_u64_wg(&s.claim[A3(s.m, t, k)]) == key ? 4 : 0);
            }
            const int b = wave_alloc(need, s_nt);
            if (need) {
                if (b + need > s.cap) {
                    atomicOr(s.err, MERR_CAPACITY);
                } else {
                    ins_split_at(s, p, l, b);
                    in.l[i] = -1;
                }
            }
        }
        __syncthreads();
        const int te = min(*s_nt, s.cap);
        if (threadIdx.x == 0) s_np[q ^ 1] = 0;
        for (int c = tb + TAIL_BS - 1 - (int)threadIdx.x; c < te; c += TAIL_BS) ins_fix(s, c);
        for (int i0 = 0; i0 < n; i0 += TAIL_BS) {
            const int i = i0 + (int)threadIdx.x;
            int p = -1, l = -1;
            unsigned close = 0;
            if (i < n) {
                p = in.p[i];
                l = in.l[i];
                close = in.close[i];
            }
            const bool keep = l >= 0 && ins_relocate_at<CLAIM_WG, false>(s, p, &l, &close);
            const int b = wave_alloc(keep ? 1 : 0, &s_np[q]);
            if (keep) {
                out.p[b] = p;
                out.l[b] = l;
                out.close[b] = close;
            }
            ins_claim_wg(s, p, keep ? l : -1, close, ep + 1);
        }
        __syncthreads();
        const int n2 = s_np[q];
        if (n2 >= n && te == tb) {
            err = 1;
            break;
        }
        n = n2;
        tb = te;
        ep++;
        r++;
    }
    return n;
}

// set: the counters of the launched round that made the list P (the host has
// not waited for them), or null: n points and ntri triangles
__global__ __launch_bounds__(TAIL_BS) void k_ins_tail(Ins s, int* P, int* P2, int n, int ntri, const int* set,
                                                      unsigned epoch0, int max_rounds, RoundSnap snap)
{
    if (set) {
        n = set[R_NEXT];
        ntri = set[R_BASE] + set[R_NEW];
    }
    __shared__ int s_np, s_nt, s_tb, s_np2[2];
    __shared__ InsList s_list[2];
    unsigned ep = epoch0;
    int r = 0, err = 0;
    if (threadIdx.x == 0) s_nt = ntri;
    __syncthreads();
    while (n > 0 && r < max_rounds) {
        if (n <= INS_LIST) {
            n = ins_short_rounds(s, P, n, s_list, s_np2, &s_nt, ep, max_rounds, r, err);
            break;
        }
        for (int i = threadIdx.x; i < n; i += TAIL_BS) ins_claim(s, P[i], ep);
        if (threadIdx.x == 0) {
            s_np = 0;
            s_tb = s_nt;
        }
        __syncthreads();
        for (int i0 = 0; i0 < n; i0 += TAIL_BS) {
            const int i = i0 + (int)threadIdx.x;
            const int p = i < n ? P[i] : -1;
            const int need = p >= 0 ? ins_need(s, p, ep) : 0;
            const int b = wave_alloc(need, &s_nt);
            if (need) {
                if (b + need > s.cap) atomicOr(s.err, MERR_CAPACITY);
                else ins_split(s, p, b);
            }
        }
        __syncthreads();
        int tb = s_tb, te = min(s_nt, s.cap);
        for (int c = tb + (int)threadIdx.x; c < te; c += TAIL_BS) ins_fix(s, c);
        __syncthreads();
        for (int i0 = 0; i0 < n; i0 += TAIL_BS) {
            const int i = i0 + (int)threadIdx.x;
            const int p = i < n ? P[i] : -1;
            const bool keep = p >= 0 && ins_relocate(s, p);
            const int b = wave_alloc(keep ? 1 : 0, &s_np);
            if (keep) P2[b] = p;
        }
        __syncthreads();
        int n2 = s_np;
        if (n2 >= n && te == tb) {
            err = 1;
            break;
        }
        n = n2;
        int* tmp = P;
        P = P2;
        P2 = tmp;
        ep++;
        r++;
        __syncthreads();
    }
    __syncthreads();
    tail_snap(snap, n, r, err, s_nt, 0, 0);
}

int insert_rounds(Ctx& c, const Ins& s_in, DBuf<int>& pend, DBuf<int>& pend2, int npend, int ntri, int* rounds)
{
    Ins s = s_in;
    s.pivot = c.pivot;
    int* P = pend.p;   // input list of the next round to launch
    int* P2 = pend2.p;
    int r = 0;
    int est = npend;  // estimate of the next round's input size (exact for the first)
    int nt = ntri;
    bool done = npend == 0;
    // Rounds are launched one ahead of the host's knowledge of their input
    // size: each round's counters are snapshot asynchronously and read after
    // the next round is queued, so the GPU does not wait for the host.
    int n_in = npend;  // input of the round whose counters are read next
    int nw_in = 0;     // and the triangles claimed for it (0: not known)
    auto check_round = [&](const int* h) {
        if (h[S_ERR]) c.check_err();
        if (n_in > 0 && h[S_NEXT] >= n_in && h[S_NEW] == 0)
            throw Error(GCDT_ERR_INTERNAL, "insertion round without progress");
        // exact list lengths of the round, for per-item bytes of the timed kernels
        prof_add_items("ins_split", nw_in);
        prof_add_items("ins_reloc", n_in);
        n_in = h[S_NEXT];
        nw_in = h[S_NW];
        nt = h[S_BASE] + h[S_NEW];
        if (n_in == 0) done = true;
        est = n_in;
    };
    // Claimed-triangle lists: every pending point claims at most two
    // triangles, and each claimed triangle is listed once per round.
    DBuf<int> wa, wb;
    int* W = nullptr;   // triangles claimed for the round being launched
    int* W2 = nullptr;  // triangles claimed for the round after it
    long long wcap = std::min<long long>(2LL * npend, s.cap) + 1;
    if (!done && est > c.tail_threshold) {
        wa.ensure((size_t)wcap);
        wb.ensure((size_t)wcap);
        W = wa.p;
        W2 = wb.p;
        c.rounds_start(npend, ntri);
        // the first round's claims; later rounds claim inside the relocation
        ProfScope ps("ins_claim", c.st, est);
        k_ins_claim_w<<<grid_for(est), kBlock, 0, c.st>>>(s, P, c.round_set(0) + R_NEXT, c.epoch + 1, W2,
                                                          c.round_set(0) + R_NW, (int)wcap);
        GCDT_LAUNCH_CHECK();
    }
    while (!done && est > c.tail_threshold) {
        if (++r > 100000) throw Error(GCDT_ERR_NOT_CONVERGED, "insertion rounds did not converge");
        unsigned ep = c.next_epoch();
        c.rounds_turn(r);
        int *in = c.round_set(r - 1), *set = c.round_set(r);
        // round r - 1 goes to the host with round r's first kernel
        const RoundSnap snap = r > 1 ? c.round_snap(r - 1) : RoundSnap{};
        std::swap(W, W2);
        with_items(c.ins_items, [&](auto it) {
            constexpr int IT = decltype(it)::value;
            ProfScope ps("ins_split", c.st, 0);
            k_ins_split<IT><<<grid_for((est + IT - 1) / IT), kBlock, 0, c.st>>>(s, W, in + R_NW, (int)wcap, set, snap);
            GCDT_LAUNCH_CHECK();
        });
        with_items(c.ins_items, [&](auto it) {
            constexpr int IT = decltype(it)::value;
            ProfScope ps("ins_reloc", c.st, 0);
            const int split = est <= INS_SPLIT_MAX;
            k_ins_reloc<IT><<<grid_for((est + IT - 1) / IT) << split, kBlock, 0, c.st>>>(
                s, P, in + R_NEXT, npend, split, P2, ep + 1, W2, (int)wcap, set, c.round_set(r + 1));
            GCDT_LAUNCH_CHECK();
        });
        std::swap(P, P2);
        if (r >= 2) check_round(c.round_wait(r - 1));  // round r is queued
    }
    if (!done) {
        // finish in one persistent workgroup, which reads the last launched
        // round's counters itself (a wait here idles the GPU for 10 us)
        prof_add_items("ins_split", r ? nw_in : 0);
        prof_add_items("ins_reloc", r ? n_in : 0);
        unsigned ep0 = c.epoch + 1;
        RoundSnap snap = c.round_snap(0);
        {
            ProfScope ps("ins_tail", c.st, est);
            k_ins_tail<<<1, TAIL_BS, 0, c.st>>>(s, P, P2, est, nt, r ? c.round_set(r) : nullptr, ep0, 1 << 20, snap);
            GCDT_LAUNCH_CHECK();
        }
        const int* h = c.round_wait(0);
        if (h[C_ERR]) c.check_err();
        if (h[C_TAIL_ERR]) throw Error(GCDT_ERR_INTERNAL, "insertion round without progress (tail)");
        r += h[C_TAIL_R];
        c.epoch += (unsigned)h[C_TAIL_R];
        if (h[C_TAIL_N] != 0) throw Error(GCDT_ERR_NOT_CONVERGED, "insertion tail did not converge");
        nt = h[C_NTRI];
    }
    if (rounds) *rounds = r;
    if (nt > s.cap) throw Error(GCDT_ERR_CAPACITY, "triangle capacity exceeded");
    return nt;
}

// ================================================================== flip rounds

// Claims of the short rounds of one persistent workgroup, in an LDS hash
// table instead of the records' claim words (device-scope atomics and
// atomic loads there cost a trip to the memory side each; these rounds are
// chains of such trips).  Open addressing on the triangle id.  Tags (-1) and
// keys (0) of a table are cleared before the round that uses it.
constexpr int LCL_CAP = 2048;      // entries per table
constexpr int LCL_MAX_LIST = 512;  // rounds of at most this many items use it (2 claims per item)

struct LdsClaims {
    int* tag;
    unsigned long long* key;
    static constexpr bool kMeta = true;
    __device__ void propose(const FlipP& f, int t, int n, unsigned long long k) const
    {
        max(f, t, k);
        max(f, n, k);
    }
    __device__ void max(const FlipP& f, int t, unsigned long long k) const
    {
        unsigned h = hash32((uint32_t)t) & (LCL_CAP - 1);
        for (int probe = 0; probe < LCL_CAP; probe++) {
            int g = tag[h];
            if (g == -1) g = atomicCAS(&tag[h], -1, t);
            if (g == -1 || g == t) {
                atomicMax(&key[h], k);
                return;
            }
            h = (h + 1) & (LCL_CAP - 1);
        }
        atomicOr(f.err, MERR_CAPACITY);
    }
    __device__ unsigned long long find(int t) const
    {
        unsigned h = hash32((uint32_t)t) & (LCL_CAP - 1);
        for (int probe = 0; probe < LCL_CAP; probe++) {
            int g = tag[h];
            if (g == t) return key[h];
            if (g == -1) return 0ull;
            h = (h + 1) & (LCL_CAP - 1);
        }
        return 0ull;
    }
    template <bool COH>
    __device__ unsigned long long get(const FlipP&, int t, unsigned long long) const
    {
        return find(t);
    }
    template <bool COH>
    __device__ unsigned long long load(const FlipP&, int t) const
    {
        return find(t);
    }
};

// Flip engines: the array-per-field layout (short lists on a mesh whose
// arrays stay in place) and the packed 64-byte records (whole-mesh rounds).
// Both keep the same claims protocol; apply() sets mark = epoch + 1 on the
// two triangles of a flip.
struct EngSoA {
    static constexpr bool kFused = false;
    Flip f;
    __device__ bool test(int t, unsigned ep, bool all, bool single) const { return flip_test(f, t, ep, all, single); }
    __device__ bool fixtest(int t, unsigned ep, bool all, bool single) const { return test(t, ep, all, single); }
    // multi-launch rounds: the proposal list holds triangles
    __device__ int propose(int t, unsigned ep, bool all, bool single) const { return test(t, ep, all, single) ? t : -1; }
    __device__ int apply_round(int q, unsigned ep, int* t, int* nn) const
    {
        *t = q;
        return apply<false>(q, ep, nn);
    }
    // no LDS claims for this layout (the persistent tail never asks for them)
    __device__ bool fixtest_l(int t, unsigned ep, const LdsClaims&) const { return test(t, ep, false, false); }
    __device__ int apply_l(int t, unsigned ep, int* nn, const LdsClaims&) const { return apply<true>(t, ep, nn); }
    template <bool COH>
    __device__ int apply(int t, unsigned ep, int* nn) const
    {
        int res = flip_apply<COH>(f, t, ep, nn);
        if (res == 2) {
            f.mark[t] = (int)ep + 1;
            f.mark[*nn] = (int)ep + 1;
        }
        return res;
    }
    __device__ void fix(int t, unsigned ep) const { flip_fix(f, t, ep); }
    __device__ void set_mark(int t, int v) const { f.mark[t] = v; }
};

struct EngPacked {
    // the test launch also settles the previous round's flips (flip_fixtest_p)
    static constexpr bool kFused = true;
    FlipP f;
    PeerClaims pc;  // of the multi-launch rounds
    // multi-launch rounds: the proposal list holds 3 t + edge
    __device__ int propose(int t, unsigned ep, bool all, bool single) const
    {
        int k;
        return flip_fixtest_p(f, t, ep, all, single, pc, &k) ? 3 * t + k : -1;
    }
    __device__ int apply_round(int q, unsigned ep, int* t, int* nn) const
    {
        *t = (int)((unsigned)q / 3u);
        return flip_apply_peer(f, q, ep, nn, pc);
    }
    __device__ bool test(int t, unsigned ep, bool all, bool single) const
    {
        return flip_test_p(f, t, ep, all, single);
    }
    __device__ bool fixtest(int t, unsigned ep, bool all, bool single) const
    {
        return flip_fixtest_p(f, t, ep, all, single);
    }
    __device__ bool fixtest_l(int t, unsigned ep, const LdsClaims& cl) const
    {
        return flip_fixtest_p(f, t, ep, false, false, cl);
    }
    __device__ int apply_l(int t, unsigned ep, int* nn, const LdsClaims& cl) const
    {
        return flip_apply_p<true>(f, t, ep, nn, cl);
    }
    template <bool COH>
    __device__ int apply(int t, unsigned ep, int* nn) const
    {
        return flip_apply_p<COH>(f, t, ep, nn);
    }
    __device__ void fix(int t, unsigned ep) const { flip_fix_p(f, t, ep); }
    __device__ void set_mark(int t, int v) const { f.r[t].meta = rec_with_mark(f.r[t].meta, v); }
};

// Tests the listed triangles; the ones that propose a flip are appended to
// `prop`, the only list the apply step reads.
template <class E, int FT_ITEMS>
__global__ __launch_bounds__(kBlock) void k_flip_test(E e, const int* list, const int* cnt, int lcap, unsigned epoch,
                                                      int single, int* prop, int* nprop, int cap, int* eflag,
                                                      RoundSnap snap)
{
    round_snap_store(snap);
    __shared__ int s_buf[STAGE_CAP];
    __shared__ int s_base;
    // a triangle proposes at most once per round, so `prop` (cap entries)
    // cannot overflow; a miscount flags MERR_CAPACITY instead of writing past it
    Staged<STAGE_CAP> sp(s_buf, &s_base, prop, nprop, cap, eflag, MERR_CAPACITY);
    int pre[FT_ITEMS];
    first_tile(list, lcap, blockIdx.x, pre);
    int n = min(*cnt, lcap);
    TILE_LOOP(base, n, kBlock * FT_ITEMS)
    {
        int q[FT_ITEMS];
        int nq = 0;
#pragma unroll
        for (int j = 0; j < FT_ITEMS; j++) {
            q[j] = -1;
            long long i = base + (long long)j * kBlock + threadIdx.x;
            if (i < n) {
                q[j] = e.propose(list ? TILE_ITEM(list, pre, base, blockIdx.x, i, j, FT_ITEMS) : (int)i, epoch, list == nullptr, single != 0);
            }
            nq += q[j] >= 0;
        }
        int b = sp.reserve(nq);
#pragma unroll
        for (int j = 0; j < FT_ITEMS; j++)
            if (q[j] >= 0) s_buf[b++] = q[j];
    }
    sp.flush();
}

// The same for short lists of packed records, whose time is the chain of trips
// to memory: four lanes share a triangle, one an edge, and the proposal (or -1)
// of entry i goes to prop[i], so that no list is appended to (20,000 points, 23
// rounds: 220 -> 116 us).
__global__ __launch_bounds__(kBlock) void k_flip_test_short(FlipP f, PeerClaims cl, const int* list, const int* cnt, int lcap,
                                                            unsigned epoch, int single, int* prop, RoundSnap snap)
{
    round_snap_store(snap);
    const int k = (int)threadIdx.x & 3, lead = (int)threadIdx.x & 60;
    const long long i0 = (long long)blockIdx.x * (kBlock / 4) + (threadIdx.x >> 2);
    const int pre = list && i0 < lcap ? list[i0] : 0;
    const int n = min(*cnt, lcap);
    TILE_LOOP(base, n, kBlock / 4)
    {
        const long long i = base + (threadIdx.x >> 2);
        int t = -1, nn = -1;
        bool hit = false;
        if (i < n) {
            t = list ? (i == i0 ? pre : list[i]) : (int)i;
            const FRec r = rec_load(&f.r[t]);
            FRec rn;
            hit = k < 3 && flip_fixtest_edge(f, t, r, k, epoch, list == nullptr, single != 0, &nn, &rn);
        }
        const unsigned m = (unsigned)(__ballot(hit) >> lead) & 7u;
        const int cand = m ? __ffsll((long long)m) - 1 : 3;
        if (i < n && k == cand) {
            if (cand < 3) cl.propose(f, t, nn, ((unsigned long long)epoch << 32) | (unsigned)(3 * t + cand));
            prop[i] = cand < 3 ? 3 * t + cand : -1;
        }
    }
}

// holes: entries of the list are proposals or -1; their number goes to *nprop.
template <class E, int FA_ITEMS>
__global__ __launch_bounds__(kBlock) void k_flip_apply(E e, const int* list, const int* cnt, int holes, int* nprop,
                                                       unsigned epoch, int* list2, int* cnt2, int* flipped, int* nflip,
                                                       int cap, int* eflag)
{
    __shared__ int s_buf[STAGE_CAP], s_buf2[E::kFused ? 1 : STAGE_CAP];
    __shared__ int s_base, s_base2;
    // each triangle enters the next list at most once per round (a lost
    // proposer that keeps its own claim is flipped by no one), so both lists
    // hold at most cap entries; a miscount flags MERR_CAPACITY
    Staged<STAGE_CAP> sq(s_buf, &s_base, list2, cnt2, cap, eflag, MERR_CAPACITY),
        sf(s_buf2, &s_base2, flipped, nflip, cap, eflag, MERR_CAPACITY);
    __shared__ int s_nf, s_np;  // fused engines need only the number of flipped triangles
    if (E::kFused && threadIdx.x == 0) s_nf = s_np = 0;
    int flips = 0, props = 0;
    int pre[FA_ITEMS];
    first_tile(list, cap, blockIdx.x, pre);
    int n = min(*cnt, cap);
    TILE_LOOP(base, n, kBlock * FA_ITEMS)
    {
        int qa[FA_ITEMS], qb[FA_ITEMS];
        int nq = 0, nf = 0;
#pragma unroll
        for (int j = 0; j < FA_ITEMS; j++) {
            qa[j] = -1;
            qb[j] = -1;
            long long i = base + (long long)j * kBlock + threadIdx.x;
            if (i < n) {
                int t, nn = -1;
                const int q = TILE_ITEM(list, pre, base, blockIdx.x, i, j, FA_ITEMS);
                if (q >= 0) {
                    int res = e.apply_round(q, epoch, &t, &nn);
                    if (res == 1) e.set_mark(t, (int)epoch + 1);
                    if (res == 1 || res == 2) qa[j] = t;
                    if (res == 2) qb[j] = nn;
                    props++;
                }
            }
            nq += (qa[j] >= 0) + (qb[j] >= 0);
            nf += (qb[j] >= 0) ? 2 : 0;
        }
        int b = sq.reserve(nq);
        int fb = E::kFused ? 0 : sf.reserve(nf);
        flips += nf;
#pragma unroll
        for (int j = 0; j < FA_ITEMS; j++) {
            if (qa[j] >= 0) s_buf[b++] = qa[j];
            if (qb[j] >= 0) {
                s_buf[b++] = qb[j];
                if (!E::kFused) {
                    s_buf2[fb++] = qa[j];
                    s_buf2[fb++] = qb[j];
                }
            }
        }
    }
    sq.flush();
    if (E::kFused) {  // after the barrier in flush
        wave_alloc(flips, &s_nf);
        if (holes) wave_alloc(props, &s_np);
        __syncthreads();
        if (threadIdx.x == 0 && s_nf) atomicAdd(nflip, s_nf);
        if (threadIdx.x == 0 && s_np) atomicAdd(nprop, s_np);
    } else {
        sf.flush();
    }
}

template <class E>
__global__ __launch_bounds__(kBlock) void k_flip_fix(E e, const int* list, const int* cnt, int cap, unsigned epoch)
{
    int n = min(*cnt, cap);
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        e.fix(list[i], epoch);
}

// One flip round of at most SHORT_MAX triangles in one workgroup: its list and
// the listed triangles' records stay in LDS from round to round (kept: the
// records are there), four lanes share a triangle, one an edge, and whoever
// tested the edge that wins flips it from the records it holds.  Only the
// neighbour slots are read again for that: the test settles them, in records
// of other lanes too.  Returns the length of the next list; lf receives the
// flipped triangles, *nf their count.
//
// Such a round is a chain of waits: list, record, neighbours, up to three
// in-circle tests in a row (0.4 us each for a lone wave), claims, and in the
// apply list, record, neighbour and stores again: 3 us in that form, 1.9 in this
// (10M clustered points: 6.5 -> 4.3 ms in 1,100 to 2,200 rounds).
#ifndef GCDT_SHORT_MAX
#define GCDT_SHORT_MAX (TAIL_BS / 4)
#endif
constexpr int SHORT_MAX = GCDT_SHORT_MAX;
static_assert(4 * SHORT_MAX <= TAIL_BS, "four lanes a triangle");

__device__ inline int short_round(const FlipP& f, int* list, FRec* rec, bool kept, int n, unsigned ep,
                                  const LdsClaims& cl, const LdsClaims& next, int* n2, int* nf, int q, int* lf)
{
    const int i = (int)threadIdx.x >> 2, k = (int)threadIdx.x & 3;
    const int lane = (int)threadIdx.x & 63, lead = lane & ~3;
    const bool on = ((int)(threadIdx.x & ~63u) >> 2) < n;  // the wave has a triangle
    int t = -1, nn = -1, cand = 3;
    FRec r, rn;
    unsigned long long key = 0ull;
    if (on) {
        bool hit = false;
        if (i < n && k < 3) {
            t = list[i];
            r = kept ? rec_load(&rec[i]) : rec_load(&f.r[t]);
            hit = flip_fixtest_edge(f, t, r, k, ep, false, false, &nn, &rn);
        }
        const unsigned m = (unsigned)(__ballot(hit) >> lead) & 7u;
        cand = m ? __ffsll((long long)m) - 1 : 3;
        t = __shfl(t, lead, 64);
        nn = __shfl(nn, lead + cand, 64);
        key = ((unsigned long long)ep << 32) | (unsigned)(3 * t + cand);
        if (cand != 3 && k < 2) cl.max(f, k == 0 ? t : nn, key);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        n2[q ^ 1] = 0;
        nf[q ^ 1] = 0;
    }
    for (int j = threadIdx.x; j < LCL_CAP; j += TAIL_BS) {
        next.tag[j] = -1;
        next.key[j] = 0ull;
    }
    if (on) {
        const unsigned long long own = cand != 3 && k < 2 ? cl.find(k == 0 ? t : nn) : 0ull;
        const unsigned long long ct = __shfl(own, lead, 64), cn = __shfl(own, lead + 1, 64);
        int res = 0;  // as flip_apply_p
        if (cand != 3) {
            if (ct == key) res = cn == key ? 2 : 1;
            else res = (ct >> 32) == ep && cl.find((int)((ct & 0xffffffffu) / 3)) == ct ? 3 : 1;
        }
        int b = wave_alloc(k == 0 ? (res == 1 ? 1 : res == 2 ? 2 : 0) : 0, &n2[q]);
        const int w = wave_alloc(k == 0 && res == 2 ? 2 : 0, &nf[q]);
        b = __shfl(b, lead, 64);
        if (k == 0 && res == 2) {
            lf[w] = t;
            lf[w + 1] = nn;
        }
        if (res == 1 && k == 0) {
            list[b] = t;
            r.a = f.r[t].a;
            if (b < SHORT_MAX) rec_store(&rec[b], r.v, r.a, r.p[0], r.p[1], r.p[2], r.meta, r.stamp, 0ull);
        } else if (res == 2 && k == cand) {
            r.a = f.r[t].a;
            rn.a = f.r[nn].a;
            flip_records(&f.r[t], &f.r[nn], t, r, k, nn, rn, ep, key);
            list[b] = t;
            list[b + 1] = nn;
            if (b + 1 < SHORT_MAX) flip_records(&rec[b], &rec[b + 1], t, r, k, nn, rn, ep, key);
        }
    }
    __syncthreads();
    return n2[q];
}

// Persistent single-workgroup tail of the flip rounds.
// set: the counters of the launched round that made the list A, or null: n.
template <class E>
__global__ __launch_bounds__(TAIL_BS) void k_flip_tail(E e, int* A, int* B, int* lf, int n, const int* set, int cap,
                                                       unsigned epoch0, int max_rounds, int* eflag, RoundSnap snap)
{
    // round counters double-buffered by round parity: a round's pair is reset
    // after the round's first barrier, which every thread passes only after
    // reading the pair two rounds back
    __shared__ int s_n2[2], s_nf[2];
    // claims of rounds with at most LCL_MAX_LIST items (fused engines), one
    // table per round parity: the other one is cleared while a round applies
    __shared__ int s_tag[2][LCL_CAP];
    __shared__ unsigned long long s_key[2][LCL_CAP];
    // list and records of the rounds of at most SHORT_MAX triangles
    __shared__ int s_list[E::kFused ? 2 * SHORT_MAX : 1];
    __shared__ int4 s_rec[E::kFused ? SHORT_MAX * (sizeof(FRec) / sizeof(int4)) : 1];
    unsigned ep = epoch0;  // A, B and lf hold cap entries each, n <= cap
    int r = 0, err = 0, flips = 0, props = 0;
    if (set) {
        n = min(set[R_NEXT], cap);
        flips = set[R_FLIP] / 2;
        props = set[R_PROP];
        // the highest-keyed proposal always wins both of its triangles
        if (n > 0 && flips == 0) {
            err = 1;
            max_rounds = 0;
        }
    }
    int nf = 0;
    if (threadIdx.x == 0) {
        s_n2[0] = 0;
        s_nf[0] = 0;
    }
    // LDS starts with whatever the CU held before: clear tags and keys
    for (int i = threadIdx.x; i < 2 * LCL_CAP; i += TAIL_BS) {
        (&s_tag[0][0])[i] = -1;
        (&s_key[0][0])[i] = 0ull;
    }
    __syncthreads();
    while (n > 0 && r < max_rounds) {
        if constexpr (E::kFused) {
            if (n <= SHORT_MAX) {
                for (int i = threadIdx.x; i < n; i += TAIL_BS) s_list[i] = A[i];
                __syncthreads();
                for (bool kept = false; n > 0 && n <= SHORT_MAX && r < max_rounds; kept = true) {
                    const int q = r & 1;
                    const int n2 = short_round(e.f, s_list, (FRec*)s_rec, kept, n, ep, LdsClaims{s_tag[q], s_key[q]},
                                               LdsClaims{s_tag[q ^ 1], s_key[q ^ 1]}, s_n2, s_nf, q, lf);
                    nf = s_nf[q];
                    if (n2 > 0 && nf == 0) {
                        err = 1;
                        break;
                    }
                    flips += nf / 2;
                    n = n2;
                    ep++;
                    r++;
                }
                if (err) break;
                if (n > SHORT_MAX) {
                    for (int i = threadIdx.x; i < n; i += TAIL_BS) A[i] = s_list[i];
                    __syncthreads();
                }
                continue;
            }
        }
        const int q = r & 1;
        const bool lds = E::kFused && n <= LCL_MAX_LIST;
        const LdsClaims cl{s_tag[q], s_key[q]};
        // fused engines settle the previous round's flips while testing
        for (int i = threadIdx.x; i < n; i += TAIL_BS) {
            if (lds) e.fixtest_l(A[i], ep, cl);
            else if (E::kFused) e.fixtest(A[i], ep, false, false);
            else e.test(A[i], ep, false, false);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            s_n2[q ^ 1] = 0;
            s_nf[q ^ 1] = 0;
        }
        for (int i = threadIdx.x; i < LCL_CAP; i += TAIL_BS) {
            s_tag[q ^ 1][i] = -1;
            s_key[q ^ 1][i] = 0ull;
        }
        // block-uniform trip count, so each wave reserves its appends with
        // one LDS atomic per counter
        for (int i0 = 0; i0 < n; i0 += TAIL_BS) {
            const int i = i0 + (int)threadIdx.x;
            int t = -1, nn = -1, res = 0;
            if (i < n) {
                t = A[i];
                res = lds ? e.apply_l(t, ep, &nn, cl) : e.template apply<true>(t, ep, &nn);
            }
            const int b = wave_alloc(res == 1 ? 1 : res == 2 ? 2 : 0, &s_n2[q]);
            const int w = wave_alloc(res == 2 ? 2 : 0, &s_nf[q]);
            if (res == 1) {
                if (b < cap) B[b] = t;
                e.set_mark(t, (int)ep + 1);
            } else if (res == 2) {
                if (b + 1 < cap) {
                    B[b] = t;
                    B[b + 1] = nn;
                }
                if (w + 1 < cap) {
                    lf[w] = t;
                    lf[w + 1] = nn;
                }
            }
        }
        __syncthreads();
        int n2 = s_n2[q];
        nf = s_nf[q];
        if (n2 > cap || nf > cap) {  // cannot happen (one entry per triangle): flagged, not written
            if (threadIdx.x == 0) atomicOr(eflag, MERR_CAPACITY);
            n = 0;
            break;
        }
        if (!E::kFused) {
            for (int i = threadIdx.x; i < nf; i += TAIL_BS) e.fix(lf[i], ep);
            __syncthreads();
        }
        if (n2 > 0 && nf == 0) {
            err = 1;
            break;
        }
        flips += nf / 2;
        n = n2;
        int* tmp = A;
        A = B;
        B = tmp;
        ep++;
        r++;
    }
    if (E::kFused && n > 0 && nf > 0) {
        // stopped at the round limit with the last round's flips unsettled
        for (int i = threadIdx.x; i < nf; i += TAIL_BS) e.fix(lf[i], ep - 1);
        __syncthreads();
    }
    __syncthreads();
    tail_snap(snap, n, r, err, 0, flips, props);
}

template <class E>
__global__ __launch_bounds__(kBlock) void k_mark_list(E e, const int* list, int n, int v)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        e.set_mark(list ? list[i] : (int)i, v);
}

__global__ __launch_bounds__(kBlock) void k_iota(int* p, int n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        p[i] = (int)i;
}

__global__ __launch_bounds__(kBlock) void k_pack_faces(const int3* __restrict__ tri, const int3* __restrict__ adj,
                                                       const int* __restrict__ cflag, const int2* __restrict__ pts,
                                                       int T, FRec* __restrict__ r)
{
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < T; t += (long long)gridDim.x * blockDim.x) {
        FRec x;
        x.v = tri[t];
        x.a = adj[t];
        x.p[0] = pts[x.v.x];
        x.p[1] = pts[x.v.y];
        x.p[2] = pts[x.v.z];
        rec_store(&r[t], x.v, x.a, x.p[0], x.p[1], x.p[2], (cflag ? cflag[t] & 7 : 0) | FREC_NOCAND | FREC_NOPARTNER,
                  0, 0ull);
    }
}

__global__ __launch_bounds__(kBlock) void k_unpack_faces(const FRec* __restrict__ r, int T, int3* __restrict__ tri,
                                                         int3* __restrict__ adj, int* __restrict__ cflag)
{
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < T; t += (long long)gridDim.x * blockDim.x) {
        const FRec x = rec_load(&r[t]);
        tri[t] = x.v;
        adj[t] = x.a;
        if (cflag) cflag[t] = x.meta & 7;
    }
}

namespace {

// The two-tester rounds of at most this many triangles run in one persistent
// workgroup; larger ones as launches of their own.  A workgroup takes about
// 50 us for a round of 2,000 to 4,000 triangles and 10 us for 700; a launched
// round takes 16 us at either size (4.2M lattice, line at 512 / 1,024 / 2,048:
// 10.97 / 10.92 / 12.06 ms).
#ifndef GCDT_FLIP_WG_LIST
#define GCDT_FLIP_WG_LIST 1024
#endif
constexpr int FLIP_WG_LIST = GCDT_FLIP_WG_LIST;

// Rounds of at most this many triangles test by edges (k_flip_test_short): a
// launch of 2,000 to 30,000 takes 5.0 us for 9.6.  Larger ones are bound by
// atomics and lines instead; between here and 500,000 the two forms measure the
// same.
#ifndef GCDT_FLIP_SHORT_MAX
#define GCDT_FLIP_SHORT_MAX 65536
#endif
constexpr int FLIP_SHORT_MAX = GCDT_FLIP_SHORT_MAX;

// Rounds of test / apply / fix over a triangle list until no edge needs a
// flip.  Round 1 reads `init` (or the implicit list of all T triangles); later
// rounds alternate between two device lists whose lengths stay on the device
// (the rounds' counter ring); the host checks round r-1 while round r is
// queued.  Lists above the tail threshold are tested by the lower of an edge's
// two active triangles (single tester); from there on every listed triangle
// tests, in launched rounds down to FLIP_WG_LIST triangles and then in one
// persistent workgroup.  Where the rounds change over decides which flips
// meet in a round, and with them the slots of the result, so the threshold is
// the tunable's alone; FLIP_WG_LIST changes nothing but the time.
template <class E>
long long flip_driver(Ctx& c, E e, int T, const int* init, int ninit, int* rounds)
{
    DBuf<int> la(T), lb(T), lf(T), lp(T);
    DBuf<int> prop;  // PeerClaims: a byte per triangle
    if constexpr (E::kFused) {
        prop.alloc((size_t)T / 4 + 1);
        e.pc.prop = (unsigned char*)prop.p;
    }
    const int* act = init;
    int* nxt = la.p;
    int* other = lb.p;
    int est = init ? ninit : T;
    if (est > std::min(c.tail_threshold, FLIP_WG_LIST)) c.rounds_start(est, 0);
    if (init) {
        k_mark_list<E><<<grid_for(ninit), kBlock, 0, c.st>>>(e, init, ninit, (int)c.epoch + 1);
        GCDT_LAUNCH_CHECK();
    }
    long long flips = 0;
    long long settled = 0;  // fused engines: flipped triangles settled inside test launches
    int r = 0;
    bool done = est == 0;
    int n_in = est;   // input of the round whose counters are read next
    int n_flip = 0;   // flipped triangles of the last round read
    auto check_round = [&](const int* h) {
        if (h[S_ERR]) c.check_err();
        // the highest-keyed proposal always wins both of its triangles
        if (h[S_NEXT] > 0 && h[S_FLIP] == 0) throw Error(GCDT_ERR_INTERNAL, "flip round without progress");
        n_flip = h[S_FLIP];
        flips += n_flip / 2;
        settled += n_flip;
        prof_add_items("flip_test", n_in);
        prof_add_items("flip_apply", h[S_PROP]);
        if (!E::kFused) prof_add_items("flip_fix", n_flip);  // else settled by the next test launch
        n_in = h[S_NEXT];
        if (n_in == 0) done = true;
        est = n_in;
    };
    auto launch_rounds = [&](int down_to, int single) {
        while (!done && est > down_to) {
            if (++r > 1000000) throw Error(GCDT_ERR_NOT_CONVERGED, "flip rounds did not converge");
            unsigned ep = c.next_epoch();
            c.rounds_turn(r);
            int *in = c.round_set(r - 1), *set = c.round_set(r);
            // round r - 1 goes to the host with round r's first kernel
            const RoundSnap snap = r > 1 ? c.round_snap(r - 1) : RoundSnap{};
            if constexpr (E::kFused) {
                // tags 1..250 in turn; all bytes are cleared before a tag comes again
                if ((r - 1) % 250 == 0) fill_i32(c, prop.p, 0, (long long)prop.n);
                e.pc.tag = (unsigned char)(1 + (r - 1) % 250);
            }
            with_items(c.flip_items, [&](auto it) {
                constexpr int IT = decltype(it)::value;
                bool holes = false;
                if constexpr (E::kFused) holes = est <= FLIP_SHORT_MAX;
                if (holes) {
                    if constexpr (E::kFused) {
                        ProfScope ps("flip_test", c.st, 0);
                        k_flip_test_short<<<grid_for(4LL * est), kBlock, 0, c.st>>>(
                            e.f, e.pc, act, in + R_NEXT, (init && act == init) ? ninit : T, ep, single, lp.p, snap);
                        GCDT_LAUNCH_CHECK();
                    }
                } else {
                    ProfScope ps("flip_test", c.st, 0);
                    k_flip_test<E, IT><<<grid_for((est + IT - 1) / IT), kBlock, 0, c.st>>>(
                        e, act, in + R_NEXT, (init && act == init) ? ninit : T, ep, single, lp.p, set + R_PROP, T,
                        c.dcnt.p + C_ERR, snap);
                    GCDT_LAUNCH_CHECK();
                }
                {
                    ProfScope ps("flip_apply", c.st, 0);
                    k_flip_apply<E, IT><<<grid_for((est + IT - 1) / IT), kBlock, 0, c.st>>>(
                        e, lp.p, holes ? in + R_NEXT : set + R_PROP, holes, set + R_PROP, ep, nxt, set + R_NEXT, lf.p,
                        set + R_FLIP, T, c.dcnt.p + C_ERR);
                    GCDT_LAUNCH_CHECK();
                }
            });
            if (!E::kFused) {
                ProfScope ps("flip_fix", c.st, 0);
                k_flip_fix<E><<<grid_for(est), kBlock, 0, c.st>>>(e, lf.p, set + R_FLIP, T, ep);
                GCDT_LAUNCH_CHECK();
            }
            act = nxt;
            std::swap(nxt, other);
            if (r >= 2) check_round(c.round_wait(r - 1));  // round r is queued
        }
    };
    launch_rounds(c.tail_threshold, c.single_tester);
    if (!done) {
        launch_rounds(FLIP_WG_LIST, 0);
        if (done) r--;  // the round queued ahead had no input: the workgroup would not have run it
    }
    // the last round's flips are settled by the tail: flipped triangles are in
    // the next list, so a round with flips is never the last
    if (E::kFused && r) prof_add_items("flip_test_fix", settled);
    if (!done) {
        // the rest in one persistent workgroup, which reads the last launched
        // round's counters itself
        const int last = r;
        unsigned ep0 = c.epoch + 1;
        if (!act) {  // small mesh: materialise the implicit list
            k_iota<<<grid_for(est), kBlock, 0, c.st>>>(lb.p, est);
            GCDT_LAUNCH_CHECK();
            act = lb.p;
            nxt = la.p;
        } else if (init && act == init) {
            // the tail alternates its two lists: work on a copy of the
            // caller's list
            GCDT_HIP(hipMemcpyAsync(lb.p, init, sizeof(int) * (size_t)ninit, hipMemcpyDeviceToDevice, c.st));
            act = lb.p;
            nxt = la.p;
        }
        RoundSnap snap = c.round_snap(0);
        {
            ProfScope ps("flip_tail", c.st, est);
            k_flip_tail<E><<<1, TAIL_BS, 0, c.st>>>(e, (int*)act, nxt, lf.p, est, last ? c.round_set(last) : nullptr, T,
                                                    ep0, 1 << 20, c.dcnt.p + C_ERR, snap);
            GCDT_LAUNCH_CHECK();
        }
        const int* h = c.round_wait(0);
        if (h[C_ERR]) c.check_err();
        if (h[C_TAIL_ERR]) throw Error(GCDT_ERR_INTERNAL, "flip round without progress (tail)");
        r += h[C_TAIL_R];
        c.epoch += (unsigned)h[C_TAIL_R];
        flips += h[C_TAIL_F];
        if (last) {
            prof_add_items("flip_test", n_in);
            prof_add_items("flip_apply", h[C_TAIL_P]);
            if (!E::kFused) prof_add_items("flip_fix", 2LL * h[C_TAIL_F]);
        }
        if (h[C_TAIL_N] != 0) throw Error(GCDT_ERR_NOT_CONVERGED, "flip tail did not converge");
    }
    if (rounds) *rounds = r;
    return flips;
}

}  // namespace

long long flip_rounds_records(Ctx& c, FRec* rec, const Mesh& m, int T, int* rounds)
{
    if (T <= 0) {
        if (rounds) *rounds = 0;
        return 0;
    }
    EngPacked e;
    e.f = FlipP{rec, c.dcnt.p + C_ERR};
    long long flips = flip_driver(c, e, T, nullptr, 0, rounds);
    {
        ProfScope ps("flip_unpack", c.st, T);
        k_unpack_faces<<<grid_for(T), kBlock, 0, c.st>>>(rec, T, m.tri, m.adj, m.cflag);
        GCDT_LAUNCH_CHECK();
    }
    return flips;
}

long long flip_rounds(Ctx& c, const Mesh& m, int T, const int* init, int ninit, int* rounds)
{
    if (T <= 0) {
        if (rounds) *rounds = 0;
        return 0;
    }
    if (!init) {
        // whole mesh: packed records for the rounds, written back at the end
        DBuf<FRec> rec(T);
        {
            ProfScope ps("flip_pack", c.st, T);
            k_pack_faces<<<grid_for(T), kBlock, 0, c.st>>>(m.tri, m.adj, m.cflag, m.pts, T, rec.p);
            GCDT_LAUNCH_CHECK();
        }
        return flip_rounds_records(c, rec.p, m, T, rounds);
    }
    DBuf<unsigned long long> claim(T);
    DBuf<int> stamp(T), partner(T), cand(T), mark(T);
    FillJobs f;
    f.add(claim.p, 0, 2LL * T);
    f.add(stamp.p, 0, T);
    f.add(mark.p, 0, T);
    fill_jobs(c, f);
    EngSoA e;
    e.f.m = m;
    e.f.claim = claim.p;
    e.f.stamp = stamp.p;
    e.f.partner = partner.p;
    e.f.cand = cand.p;
    e.f.mark = mark.p;
    e.f.err = c.dcnt.p + C_ERR;
    return flip_driver(c, e, T, init, ninit, rounds);
}

// ================================================================== batches of instances

// instance of each point (binary search over the point offsets)
__global__ __launch_bounds__(kBlock) void k_batch_vinst(const long long* off, int K, long long NP, int* vinst)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < NP; i += (long long)gridDim.x * blockDim.x) {
        int lo = 0, hi = K;  // last instance with off[inst] <= i
        while (lo + 1 < hi) {
            int mid = (lo + hi) >> 1;
            if (off[mid] <= i) lo = mid;
            else hi = mid;
        }
        vinst[i] = lo;
    }
}

// corners NP+4i..NP+4i+3 and the two triangles 2i, 2i+1 of every instance
__global__ __launch_bounds__(kBlock) void k_batch_init(int2* pts, int3* tri, int3* adj, int K, long long NP)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < K; i += (long long)gridDim.x * blockDim.x) {
        int c = (int)(NP + 4 * i);
        pts[c] = make_int2(0, 0);
        pts[c + 1] = make_int2(GRID_R, 0);
        pts[c + 2] = make_int2(GRID_R, GRID_R);
        pts[c + 3] = make_int2(0, GRID_R);
        int t = (int)(2 * i);
        tri[t] = make_int3(c, c + 1, c + 3);
        tri[t + 1] = make_int3(c + 1, c + 2, c + 3);
        adj[t] = make_int3(t + 1, -1, -1);
        adj[t + 1] = make_int3(-1, t, -1);
    }
}

// constraint vertex ids: instance-local -> global; ids outside the instance
// become -1 (rejected by the constraint checks)
__global__ __launch_bounds__(kBlock) void k_batch_cons(const int2* in, const long long* coff, const long long* poff, int K,
                                                       long long NC, int2* out)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < NC; i += (long long)gridDim.x * blockDim.x) {
        int lo = 0, hi = K;
        while (lo + 1 < hi) {
            int mid = (lo + hi) >> 1;
            if (coff[mid] <= i) lo = mid;
            else hi = mid;
        }
        long long base = poff[lo], n = poff[lo + 1] - poff[lo];
        int2 e = in[i];
        e.x = (e.x >= 0 && e.x < n) ? (int)(base + e.x) : -1;
        e.y = (e.y >= 0 && e.y < n) ? (int)(base + e.y) : -1;
        out[i] = e;
    }
}

// scatter the global mesh back into per-instance lists with local vertex ids.
// Leaves are in vertex order and point ids instance-major, so an instance's
// triangles fill one range of slots [first, last] (flips and cavities reuse
// slots in place): a triangle's place in its list is its slot minus first,
// the same on every run.  A range that does not hold exactly the instance's
// triangle count flags MERR_INTERNAL_COUNT.
__device__ inline int batch_inst_of(int3 t, const int* vinst, long long NP)
{
    return t.x < NP ? vinst[t.x] : (int)((t.x - NP) >> 2);
}

// the ends of each instance's run of slots, where the instance changes (one
// store per end; a split run stores an end twice and fails the count check)
__global__ __launch_bounds__(kBlock) void k_batch_span(const int3* tri, int T, const int* vinst, long long NP,
                                                       int* first, int* last)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < T; i += (long long)gridDim.x * blockDim.x) {
        const int inst = batch_inst_of(tri[i], vinst, NP);
        if (i == 0 || batch_inst_of(tri[i - 1], vinst, NP) != inst) first[inst] = (int)i;
        if (i == T - 1 || batch_inst_of(tri[i + 1], vinst, NP) != inst) last[inst] = (int)i;
    }
}

__global__ __launch_bounds__(kBlock) void k_batch_out(const int3* tri, int T, const int* vinst, const int* perm,
                                                      const long long* poff, const long long* toff, long long NP,
                                                      const int* first, const int* last, int3* out, int* err)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < T; i += (long long)gridDim.x * blockDim.x) {
        const int3 t = tri[i];
        const int inst = batch_inst_of(t, vinst, NP);
        const long long base = poff[inst], n = poff[inst + 1] - poff[inst];
        if ((long long)last[inst] - first[inst] + 1 != toff[inst + 1] - toff[inst]) {
            atomicOr(err, MERR_INTERNAL_COUNT);
            continue;
        }
        auto local = [&](int v) -> int {
            return v < NP ? (int)((perm ? perm[v] : v) - base) : (int)(n + ((v - NP) & 3));
        };
        out[toff[inst] + (i - first[inst])] = make_int3(local(t.x), local(t.y), local(t.z));
    }
}

void batch_vinst(Ctx& c, const long long* off, int K, long long NP, int* vinst)
{
    if (NP <= 0) return;
    k_batch_vinst<<<grid_for(NP), kBlock, 0, c.st>>>(off, K, NP, vinst);
    GCDT_LAUNCH_CHECK();
}

// Batch points counting-sorted by instance, then by the Morton order of a
// per-instance grid of 4^L cells (L in [4, 10], about one cell per point, the
// instance's cells numbered from cbase[i]): instance ranges are kept,
// neighbours in the plane become neighbours in memory down to single points,
// and each 16x16 cell of an instance is a contiguous range whose first point
// is a sample.  The same one-atomic counting sort as morton_order: ranks in
// inv[], then an inclusive scan, then a gather of each cell's start.
struct BatchCells {
    const int* vinst;
    const int* cbase;
    const int* lvl;
    __device__ int cell(int i, int2 p) const
    {
        int inst = vinst[i];
        return cbase[inst] + (int)(morton_cell(p) >> (2 * (10 - lvl[inst])));
    }
};

// points by (instance, fine cell), each cell in input order (the count,
// scatter and per-cell reorder of the single solve's Morton order)
__global__ __launch_bounds__(kBlock) void k_batch_cell_count(BatchCells b, const int2* pts, long long NP, int* cnt,
                                                             int* rank, int* huge)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < NP; i += (long long)gridDim.x * blockDim.x) {
        const int r = atomicAdd(&cnt[b.cell((int)i, pts[i])], 1);
        rank[i] = r;
        count_large(r, huge);
    }
}

__global__ __launch_bounds__(kBlock) void k_batch_cell_scatter(BatchCells b, const int2* pts, long long NP,
                                                               const int* cell_end, const int* rank, int4* eb)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < NP; i += (long long)gridDim.x * blockDim.x) {
        const int2 p = pts[i];
        const int cell = b.cell((int)i, p);
        const int pos = (cell ? cell_end[cell - 1] : 0) + rank[i];
        eb[pos] = make_int4((int)i, cell, p.x, p.y);
    }
}

void batch_order(Ctx& c, const int2* pts, const int* vinst, const int* cbase, const int* lvl, long long NP,
                 long long ncells, int2* out, int* perm, int* inv, int* cell_end)
{
    FillJobs f;
    f.add(cell_end, 0, ncells + 1);
    f.add(c.dcnt.p + C_HUGE, 0, 1);
    f.add(c.dcnt.p + C_NQ, 0, 1);
    fill_jobs(c, f);
    if (NP <= 0) return;
    BatchCells b{vinst, cbase, lvl};
    k_batch_cell_count<<<grid_for(NP), kBlock, 0, c.st>>>(b, pts, NP, cell_end, inv, c.dcnt.p + C_HUGE);
    GCDT_LAUNCH_CHECK();
    scan_incl(c, cell_end, cell_end, ncells);
    DBuf<int4> eb((size_t)NP);
    k_batch_cell_scatter<<<grid_for(NP), kBlock, 0, c.st>>>(b, pts, NP, cell_end, inv, eb.p);
    GCDT_LAUNCH_CHECK();
    cell_reorder(c, CellKeyPoint{pts, perm, out, inv}, cell_end, eb.p, NP, c.get(C_HUGE));
}

// Sorted range of 16x16 cell c (Morton index) of instance i: the fine cells
// [cbase + (c << 2(L-4)), cbase + ((c+1) << 2(L-4))).
__device__ inline int2 coarse_range(const int* cbase, const int* lvl, const int* cell_end, long long idx)
{
    int inst = (int)(idx >> 8), c = (int)(idx & 255);
    int sh = 2 * (lvl[inst] - 4);
    int f0 = cbase[inst] + (c << sh), f1 = cbase[inst] + ((c + 1) << sh);
    return make_int2(f0 ? cell_end[f0 - 1] : 0, cell_end[f1 - 1]);
}

__global__ __launch_bounds__(kBlock) void k_range_flags(const int* cbase, const int* lvl, const int* cell_end,
                                                        long long ncoarse, int* flags)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < ncoarse; i += (long long)gridDim.x * blockDim.x) {
        int2 r = coarse_range(cbase, lvl, cell_end, i);
        flags[i] = r.y > r.x;
    }
}

__global__ __launch_bounds__(kBlock) void k_range_emit(const int* cbase, const int* lvl, const int* cell_end,
                                                       const int* offs, long long ncoarse, int* ids)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < ncoarse; i += (long long)gridDim.x * blockDim.x) {
        int2 r = coarse_range(cbase, lvl, cell_end, i);
        if (r.y > r.x) ids[offs[i]] = r.x;
    }
}

int batch_sample_sorted(Ctx& c, const int* cbase, const int* lvl, const int* cell_end, int K, int* ids)
{
    long long ncoarse = (long long)K << 8;
    DBuf<int> offs((size_t)ncoarse + 1);
    k_range_flags<<<grid_for(ncoarse), kBlock, 0, c.st>>>(cbase, lvl, cell_end, ncoarse, offs.p);
    GCDT_LAUNCH_CHECK();
    scan_excl(c, offs.p, offs.p, ncoarse);
    k_range_emit<<<grid_for(ncoarse), kBlock, 0, c.st>>>(cbase, lvl, cell_end, offs.p, ncoarse, ids);
    GCDT_LAUNCH_CHECK();
    return c.get(C_TOTAL);
}

// Listed points located in their instance's two seed triangles (the side of
// the anti-diagonal).
__global__ __launch_bounds__(kBlock) void k_batch_locate_ids(const int2* pts, const int* vinst, const int* ids, int n,
                                                             int* loc, int* pend)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        int p = ids[i];
        int t0 = 2 * vinst[p];
        int o = orient2d(make_int2(GRID_R, 0), make_int2(0, GRID_R), pts[p]);
        loc[p] = o > 0 ? t0 * 4 + 3 : (o < 0 ? (t0 + 1) * 4 + 3 : t0 * 4 + 0);
        pend[i] = p;
    }
}

void batch_locate_ids(Ctx& c, const int2* pts, const int* vinst, const int* ids, int n, int* loc, int* pend)
{
    if (n <= 0) return;
    k_batch_locate_ids<<<grid_for(n), kBlock, 0, c.st>>>(pts, vinst, ids, n, loc, pend);
    GCDT_LAUNCH_CHECK();
}

void batch_init(Ctx& c, int2* pts, int3* tri, int3* adj, int K, long long NP)
{
    k_batch_init<<<grid_for(K), kBlock, 0, c.st>>>(pts, tri, adj, K, NP);
    GCDT_LAUNCH_CHECK();
}

void batch_cons(Ctx& c, const int2* in, const long long* coff, const long long* poff, int K, long long NC, int2* out)
{
    if (NC <= 0) return;
    k_batch_cons<<<grid_for(NC), kBlock, 0, c.st>>>(in, coff, poff, K, NC, out);
    GCDT_LAUNCH_CHECK();
}

void batch_out(Ctx& c, const int3* tri, int T, const int* vinst, const int* perm, const long long* poff,
               const long long* toff, long long NP, int K, int3* out)
{
    DBuf<int> first(K), last(K);
    fill_i32(c, first.p, INT_MAX, K);
    fill_i32(c, last.p, -1, K);
    k_batch_span<<<grid_for(T), kBlock, 0, c.st>>>(tri, T, vinst, NP, first.p, last.p);
    GCDT_LAUNCH_CHECK();
    k_batch_out<<<grid_for(T), kBlock, 0, c.st>>>(tri, T, vinst, perm, poff, toff, NP, first.p, last.p, out,
                                                  c.dcnt.p + C_ERR);
    GCDT_LAUNCH_CHECK();
    c.check_err();
}

// ================================================================== flags -> list

__global__ __launch_bounds__(kBlock) void k_flag_scatter(const int* flags, const int* off, int n, int* list)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        if (flags[i]) list[off[i]] = (int)i;
}

int flags_to_list(Ctx& c, const int* flags, int n, int* list)
{
    DBuf<int> off((size_t)n + 1);
    scan_excl(c, flags, off.p, n);
    k_flag_scatter<<<grid_for(n), kBlock, 0, c.st>>>(flags, off.p, n, list);
    GCDT_LAUNCH_CHECK();
    return c.get(C_TOTAL);
}

// ================================================================== phase check

// Per-triangle checks of a mesh between phases (the "validate" tunable):
// bits of C_VAL name what failed, C_VAL_FIRST the lowest failing triangle.
enum : int { VAL_IDS = 1, VAL_CW = 2, VAL_ADJ = 4, VAL_CFLAG = 8, VAL_DELAUNAY = 16 };

__global__ __launch_bounds__(kBlock) void k_validate_mesh(const int2* pts, long long nv, const int3* tri,
                                                          const int3* adj, const int* cflag, int T, int delaunay,
                                                          int* bad, int* first)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < T; i += (long long)gridDim.x * blockDim.x) {
        const int3 v = tri[i];
        int f = 0;
        if (v.x < 0 || v.y < 0 || v.z < 0 || v.x >= nv || v.y >= nv || v.z >= nv) {
            f = VAL_IDS;
        } else {
            const int2 A = pts[v.x], B = pts[v.y], C = pts[v.z];
            if (orient2d(A, B, C) <= 0) f |= VAL_CW;
            const int3 a = adj[i];
            const int cf = cflag ? cflag[i] : 0;
            for (int k = 0; k < 3; k++) {
                const int n = get3(a, k);
                if (n < 0) continue;  // the bounding square's sides
                if (n >= T) {
                    f |= VAL_ADJ;
                    continue;
                }
                const int u = get3(v, nx3(k)), w = get3(v, pv3(k));
                const int3 nt = tri[n];
                if (!has2(nt, u, w)) {
                    f |= VAL_ADJ;
                    continue;
                }
                const int j = slot_other(nt, u, w);
                if (get3(adj[n], j) != (int)i) {
                    f |= VAL_ADJ;
                    continue;
                }
                const int ck = (cf >> k) & 1;
                if (cflag && ck != ((cflag[n] >> j) & 1)) f |= VAL_CFLAG;
                const int o = get3(nt, j);
                if (delaunay && !ck && n > i && (o < 0 || o >= nv || incircle(A, B, C, pts[o]) > 0)) f |= VAL_DELAUNAY;
            }
        }
        if (f) {
            atomicOr(bad, f);
            atomicMin(first, (int)i);
        }
    }
}

void check_mesh(Ctx& c, const int2* pts, long long nv, const int3* tri, const int3* adj, const int* cflag, int T,
                bool delaunay, int* failed, int* first)
{
    *failed = 0;
    *first = -1;
    if (T <= 0) return;
    c.set(C_VAL, 0);
    c.set(C_VAL_FIRST, INT_MAX);
    k_validate_mesh<<<grid_for(T), kBlock, 0, c.st>>>(pts, nv, tri, adj, cflag, T, delaunay ? 1 : 0, c.dcnt.p + C_VAL,
                                                      c.dcnt.p + C_VAL_FIRST);
    GCDT_LAUNCH_CHECK();
    c.read(C_VAL, 2);
    *failed = c.hcnt[C_VAL];
    if (*failed) *first = c.hcnt[C_VAL_FIRST];
}

void validate_mesh(Ctx& c, const char* phase, const Mesh& m, long long nv, int T, bool delaunay)
{
    if (!Tunables::get().validate || T <= 0) return;
    int f = 0, first = -1;
    check_mesh(c, m.pts, nv, m.tri, m.adj, m.cflag, T, delaunay, &f, &first);
    if (!f) return;
    std::string what;
    const char* names[] = {"vertex ids", "orientation", "adjacency", "constraint bits", "local Delaunay"};
    for (int b = 0; b < 5; b++)
        if (f & (1 << b)) what += std::string(what.empty() ? "" : ", ") + names[b];
    throw Error(GCDT_ERR_INTERNAL, std::string("mesh check after ") + phase + " failed (" + what + "), first at triangle " +
                                       std::to_string(first));
}

void validate_records(Ctx& c, const char* phase, const FRec* rec, const Mesh& m, long long nv, int T, bool delaunay)
{
    if (!Tunables::get().validate || T <= 0) return;
    k_unpack_faces<<<grid_for(T), kBlock, 0, c.st>>>(rec, T, m.tri, m.adj, m.cflag);
    GCDT_LAUNCH_CHECK();
    validate_mesh(c, phase, m, nv, T, delaunay);
}

// ================================================================== leaves

__global__ __launch_bounds__(kBlock) void k_leaf_flags(const int* sons, int T, int* flags)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < T; i += (long long)gridDim.x * blockDim.x)
        flags[i] = sons[i] == -1;
}

__global__ __launch_bounds__(kBlock) void k_leaf_scatter(const int3* tri, const int3* adj, const int* sons, const int* off,
                                                         int T, int3* tri2, int3* adj2, long long cap, int* err)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < T; i += (long long)gridDim.x * blockDim.x) {
        if (sons[i] != -1) continue;
        int o = off[i];
        if (o >= cap) {
            atomicOr(err, MERR_CAPACITY);
            continue;
        }
        tri2[o] = tri[i];
        if (adj && adj2) {
            int3 a = adj[i];
            a.x = a.x >= 0 ? off[a.x] : -1;
            a.y = a.y >= 0 ? off[a.y] : -1;
            a.z = a.z >= 0 ? off[a.z] : -1;
            adj2[o] = a;
        }
    }
}

// Leaves in Morton order of their centroid's 1024^2 cell (the reference's
// reorderFaces, kernel.cu:1886-1964, done as a counting sort fused with the
// compaction): neighbouring triangles end up near each other in memory.
// Sort key of a leaf for the compacted mesh order: the Morton cell of its
// centroid on the 2048x2048 grid over the square (about five leaves per cell
// at 10M points, so nearly every cell is ranked lane by lane).
#ifndef GCDT_LEAF_CELL_BITS
#define GCDT_LEAF_CELL_BITS 11
#endif
constexpr int LEAF_CELL_BITS = GCDT_LEAF_CELL_BITS;
constexpr long long LEAF_CELLS = 1LL << (2 * LEAF_CELL_BITS);
__device__ inline unsigned morton_cell_leaf(int2 p)
{
    unsigned x = (unsigned)p.x >> (30 - LEAF_CELL_BITS), y = (unsigned)p.y >> (30 - LEAF_CELL_BITS);
    unsigned r = 0;
    for (int b = 0; b < LEAF_CELL_BITS; b++) r |= (((x >> b) & 1u) << (2 * b)) | (((y >> b) & 1u) << (2 * b + 1));
    return r;
}
// Small meshes sort by a coarser grid of about one cell per leaf (4^bits
// cells, so that clearing and scanning the counts costs no more than the
// leaves do) and order each coarse cell by fine cell first: the same order.
struct LeafKeyOne {
    int shift;  // 2 * (LEAF_CELL_BITS - bits)
    __device__ int key(const int3&, int2 g) const { return (int)(morton_cell_leaf(g) >> shift); }
};
static int leaf_bits(long long nleaf)
{
    int b = 5;
    while (b < LEAF_CELL_BITS && (1LL << (2 * b)) < nleaf) b++;
    return b;
}
__device__ inline int2 centroid(const int2* pts, const int3& t)
{
    const int2 a = pts[t.x], b = pts[t.y], c = pts[t.z];
    return make_int2((int)(((long long)a.x + b.x + c.x) / 3), (int)(((long long)a.y + b.y + c.y) / 3));
}

// CellKeyTri with the leaf's fine cell before its vertex ids
struct CellKeyTriFine {
    const int3* tri;
    const int2* pts;
    int* src;
    int* dest;
    using Key = int4;
    using Slot = int2;
    __device__ void put(long long pos, const Slot& e) const { put_elem(pos, e.x); }
    __device__ void put_elem(long long pos, int el) const
    {
        src[pos] = el;
        dest[el] = (int)pos;
    }
    __device__ Key of(int e) const
    {
        const int3 t = tri[e];
        const int a = min(t.x, min(t.y, t.z)), c = max(t.x, max(t.y, t.z));
        return make_int4((int)morton_cell_leaf(centroid(pts, t)), a, t.x + t.y + t.z - a - c, c);
    }
    __device__ static Key max_key() { return make_int4(INT_MAX, INT_MAX, INT_MAX, INT_MAX); }
    __device__ static bool less(const Key& x, const Key& y)
    {
        if (x.x != y.x) return x.x < y.x;
        return x.y < y.y || (x.y == y.y && (x.z < y.z || (x.z == y.z && x.w < y.w)));
    }
};

// The count pass keeps each leaf's rank within its cell in rank[]; the dest
// pass adds the cell's start to it without a second atomic.
template <class KEY>
__global__ __launch_bounds__(kBlock) void k_leaf_cells(KEY kf, const int2* pts, const int3* tri, const int* sons, int T,
                                                       int* cnt, int* cellof, int* rank, int* huge)
{
    WAVE_LOOP(i, T)
    {
        int cell = -1;
        if (i < T && sons[i] == -1) {
            const int3 t = tri[i];
            cell = kf.key(t, centroid(pts, t));
        }
        // consecutive leaves were allocated together and mostly share a cell
        int r = wave_run_add(cnt, cell);
        if (cell >= 0) {
            cellof[i] = cell;
            rank[i] = r;
            count_large(r, huge);
        }
    }
}

// dest[] holds the ranks on entry and the arrival-order destinations on exit
// (-1 for dead triangles); eb[] gets (leaf, cell) at each destination.  The
// per-cell reorder then writes the final destinations and their inverse.
__global__ __launch_bounds__(kBlock) void k_leaf_dest(const int* sons, const int* cellof, int T, const int* start,
                                                      int* dest, int2* eb, long long cap)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < T; i += (long long)gridDim.x * blockDim.x) {
        int d = sons[i] == -1 ? start[cellof[i]] + dest[i] : -1;
        dest[i] = d;
        if (d >= 0 && d < cap) eb[d] = make_int2((int)i, cellof[i]);
    }
}

// Leaves into packed flip records (the coordinates gathered here, so the flips
// need no pack pass over a freshly written mesh).  Walks the destinations in
// order and gathers each one's leaf, so the 64-byte writes are contiguous and
// the reads do the scattering.
__global__ __launch_bounds__(kBlock) void k_leaf_move(const int3* tri, const int3* adj, const int* dest,
                                                      const int* src, int n, const int2* pts, FRec* rec)
{
    for (long long o = (long long)blockIdx.x * blockDim.x + threadIdx.x; o < n; o += (long long)gridDim.x * blockDim.x) {
        int i = src[o];
        int3 a = adj[i];
        a.x = a.x >= 0 ? dest[a.x] : -1;
        a.y = a.y >= 0 ? dest[a.y] : -1;
        a.z = a.z >= 0 ? dest[a.z] : -1;
        const int3 v = tri[i];
        rec_store(&rec[o], v, a, pts[v.x], pts[v.y], pts[v.z], FREC_NOCAND | FREC_NOPARTNER, 0, 0ull);
    }
}

// CK: the order inside a cell.  The records are allocated last, when what the
// sort needs is gone: a batch of many small instances, nearly all of whose
// points are in its samples, would peak here otherwise.  (A fixed array counts
// them all.)
template <class CK, class KEY>
static int filter_leaves_sorted(Ctx& c, CK ck, const KEY& kf, long long ncells, const int2* pts, const int3* tri,
                                const int3* adj, DBuf<int>& sons, int T, DBuf<FRec>& rec, long long nleaf)
{
    if (g_arena) rec.alloc((size_t)nleaf);
    DBuf<int> cnt((size_t)ncells + 1), cellof(T > 0 ? T : 1), dest(T > 0 ? T : 1);
    FillJobs f;
    f.add(cnt.p, 0, ncells + 1);
    f.add(c.dcnt.p + C_HUGE, 0, 1);
    f.add(c.dcnt.p + C_NQ, 0, 1);
    fill_jobs(c, f);
    k_leaf_cells<KEY><<<grid_for(T), kBlock, 0, c.st>>>(kf, pts, tri, sons.p, T, cnt.p, cellof.p, dest.p,
                                                        c.dcnt.p + C_HUGE);
    GCDT_LAUNCH_CHECK();
    scan_excl_total(c, cnt.p, cnt.p, ncells);
    c.read(0, C_NUM);
    const int n = c.hcnt[C_TOTAL], large = c.hcnt[C_HUGE];
    if (n != nleaf)
        throw Error(GCDT_ERR_INTERNAL, "leaf count " + std::to_string(n) + " != " + std::to_string(nleaf));
    DBuf<int> src(n > 0 ? n : 1);
    {
        DBuf<int2> eb(n > 0 ? n : 1);
        k_leaf_dest<<<grid_for(T), kBlock, 0, c.st>>>(sons.p, cellof.p, T, cnt.p, dest.p, eb.p, nleaf);
        GCDT_LAUNCH_CHECK();
        cellof.release();
        sons.release();
        // each cell's leaves by their vertex ids (the count pass placed them
        // in arrival order); cnt holds the cells' starts, cnt[c + 1] their ends
        ck.tri = tri;
        ck.src = src.p;
        ck.dest = dest.p;
        cell_reorder(c, ck, cnt.p + 1, eb.p, n, large);
    }
    cnt.release();
    rec.ensure((size_t)nleaf);
    if (n > 0) {
        ProfScope ps("leaf_move", c.st, n);
        k_leaf_move<<<grid_for(n), kBlock, 0, c.st>>>(tri, adj, dest.p, src.p, n, pts, rec.p);
        GCDT_LAUNCH_CHECK();
    }
    return n;
}

int filter_leaves_morton_rec(Ctx& c, const int2* pts, const int3* tri, const int3* adj, DBuf<int>& sons, int T,
                             DBuf<FRec>& rec, long long nleaf)
{
    // on a fixed array, where the longer keys of a crowded coarse cell count, for
    // the smallest meshes only
    const int b = g_arena && nleaf > 65536 ? LEAF_CELL_BITS : leaf_bits(nleaf);
    const LeafKeyOne key{2 * (LEAF_CELL_BITS - b)};
    if (b == LEAF_CELL_BITS)
        return filter_leaves_sorted(c, CellKeyTri{}, key, LEAF_CELLS, pts, tri, adj, sons, T, rec, nleaf);
    CellKeyTriFine ck{};
    ck.pts = pts;
    return filter_leaves_sorted(c, ck, key, 1LL << (2 * b), pts, tri, adj, sons, T, rec, nleaf);
}

// Batch meshes: instance-major, then the Morton order of the centroid's cell
// in the instance's own grid of 4^L cells (the point order's cells, about one
// point each), so a cell holds a few leaves and its reorder stays in one wave.
struct LeafKeyInst {
    const int* vinst;
    const int* cbase;
    const int* lvl;
    long long NP;  // corners of instance i are NP + 4i .. NP + 4i + 3
    __device__ int key(const int3& t, int2 g) const
    {
        const int inst = t.x < NP ? vinst[t.x] : (int)((t.x - NP) >> 2);
        return cbase[inst] + (int)(morton_cell(g) >> (2 * (10 - lvl[inst])));
    }
};

int filter_leaves_inst_rec(Ctx& c, const int2* pts, const int* vinst, const int* cbase, const int* lvl,
                           long long ncells, long long NP, const int3* tri, const int3* adj, DBuf<int>& sons, int T,
                           DBuf<FRec>& rec, long long nleaf)
{
    return filter_leaves_sorted(c, CellKeyTri{}, LeafKeyInst{vinst, cbase, lvl, NP}, ncells, pts, tri, adj, sons, T,
                                rec, nleaf);
}

int filter_leaves(Ctx& c, const int3* tri, const int3* adj, const int* sons, int T, int3* tri2, int3* adj2,
                  long long cap)
{
    DBuf<int> off((size_t)T + 1);
    k_leaf_flags<<<grid_for(T), kBlock, 0, c.st>>>(sons, T, off.p);
    GCDT_LAUNCH_CHECK();
    scan_excl(c, off.p, off.p, T);
    k_leaf_scatter<<<grid_for(T), kBlock, 0, c.st>>>(tri, adj, sons, off.p, T, tri2, adj2, cap, c.dcnt.p + C_ERR);
    GCDT_LAUNCH_CHECK();
    int n = c.get(C_TOTAL);
    c.check_err();
    return n;
}

// ================================================================== bitmap

template <int LOG>
__device__ inline void tri_cells(int2 A, int2 B, int2 C, int& x0, int& y0, int& x1, int& y1)
{
    constexpr int sh = 30 - LOG;
    x0 = min(A.x, min(B.x, C.x)) >> sh;
    x1 = max(A.x, max(B.x, C.x)) >> sh;
    y0 = min(A.y, min(B.y, C.y)) >> sh;
    y1 = max(A.y, max(B.y, C.y)) >> sh;
}

// Closed triangle vs closed box, exact (separating-axis test: the box axes,
// then each triangle edge with all four corners strictly outside).
// Same predicate as the reference's intersect(), boostmap.cu:30-66.
__device__ inline bool tri_meets_box(int2 A, int2 B, int2 C, int bx0, int by0, int bx1, int by1)
{
    if (max(A.x, max(B.x, C.x)) < bx0 || min(A.x, min(B.x, C.x)) > bx1) return false;
    if (max(A.y, max(B.y, C.y)) < by0 || min(A.y, min(B.y, C.y)) > by1) return false;
    int2 q[4] = {make_int2(bx0, by0), make_int2(bx1, by0), make_int2(bx1, by1), make_int2(bx0, by1)};
    int2 P[3] = {A, B, C};
#pragma unroll
    for (int e = 0; e < 3; e++) {
        int2 u = P[e], v = P[(e + 1) % 3];
        bool out = true;
#pragma unroll
        for (int j = 0; j < 4; j++) out &= orient2d(u, v, q[j]) < 0;
        if (out) return false;
    }
    return true;
}

template <class G>
__global__ __launch_bounds__(kBlock) void k_bm_count(G g, const int2* pts, const int3* tri, int T, int* cnt)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < T; i += (long long)gridDim.x * blockDim.x) {
        int3 t = tri[i];
        int x0, y0, x1, y1;
        tri_cells<G::LOG>(pts[t.x], pts[t.y], pts[t.z], x0, y0, x1, y1);
        cnt[i] = (x1 - x0 + 1) * (y1 - y0 + 1);
    }
}

__device__ inline int upper_bound_i(const int* a, int n, long long x)
{
    int lo = 0, hi = n;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (a[mid] <= x) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

template <class G>
__global__ __launch_bounds__(kBlock) void k_bm_test(G g, const int2* pts, const int3* tri, const int* off, int T,
                                                    long long npairs, int* cellcnt, int* ord, int* cellof)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < npairs; i += (long long)gridDim.x * blockDim.x) {
        int t = upper_bound_i(off, T + 1, i) - 1;
        int local = (int)(i - off[t]);
        int3 tv = tri[t];
        int2 A = pts[tv.x], B = pts[tv.y], C = pts[tv.z];
        int x0, y0, x1, y1;
        tri_cells<G::LOG>(A, B, C, x0, y0, x1, y1);
        int h = y1 - y0 + 1;
        int cx = x0 + local / h, cy = y0 + local % h;
        constexpr int sh = 30 - G::LOG;
        bool hit = tri_meets_box(A, B, C, cx << sh, cy << sh, ((cx + 1) << sh) - 1, ((cy + 1) << sh) - 1);
        int cell = (int)(g.tri_base(tv) + ((long long)cx << G::LOG) + cy);
        cellof[i] = cell;
        ord[i] = hit ? atomicAdd(&cellcnt[cell], 1) : -1;
    }
}

__global__ __launch_bounds__(kBlock) void k_bm_fill(const int* off, int T, long long npairs, const int* ord,
                                                    const int* cellof, const int* cell_off, int* bm)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < npairs; i += (long long)gridDim.x * blockDim.x) {
        int o = ord[i];
        if (o < 0) continue;
        int t = upper_bound_i(off, T + 1, i) - 1;
        bm[cell_off[cellof[i]] + o] = t;
    }
}

template <class G>
static void build_bitmap_g(Ctx& c, const G& g, long long ncells, const int2* pts, const int3* tri, int T,
                           int** offsets, int** tris, int* ntris)
{
    DBuf<int> off((size_t)T + 1);
    k_bm_count<G><<<grid_for(T), kBlock, 0, c.st>>>(g, pts, tri, T, off.p);
    GCDT_LAUNCH_CHECK();
    scan_excl_total(c, off.p, off.p, T);
    long long npairs = c.get(C_TOTAL);
    DBuf<int> ord(npairs), cellof(npairs);
    DBuf<int> cell_off((size_t)ncells + 1);
    fill_i32(c, cell_off.p, 0, ncells + 1);
    if (npairs > 0) {
        k_bm_test<G><<<grid_for(npairs), kBlock, 0, c.st>>>(g, pts, tri, off.p, T, npairs, cell_off.p, ord.p,
                                                            cellof.p);
        GCDT_LAUNCH_CHECK();
    }
    scan_excl_total(c, cell_off.p, cell_off.p, ncells);
    int total = c.get(C_TOTAL);
    DBuf<int> bm(total > 0 ? total : 1);
    if (npairs > 0) {
        k_bm_fill<<<grid_for(npairs), kBlock, 0, c.st>>>(off.p, T, npairs, ord.p, cellof.p, cell_off.p, bm.p);
        GCDT_LAUNCH_CHECK();
    }
    // hand the buffers to the caller; they are released with the sizes
    // (ncells + 1) ints and `total` ints
    *offsets = cell_off.detach();
    *tris = bm.detach();
    *ntris = total;
}

void build_bitmap(Ctx& c, const int2* pts, const int3* tri, int T, int** offsets, int** tris, int* ntris)
{
    build_bitmap_g(c, GridOne{}, BITMAP_CELLS, pts, tri, T, offsets, tris, ntris);
}

template <class G>
__global__ __launch_bounds__(kBlock) void k_bm_pairs(G, const int2* pts, const int3* tri, int T, unsigned long long* total)
{
    unsigned long long n = 0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < T; i += (long long)gridDim.x * blockDim.x) {
        const int3 t = tri[i];
        int x0, y0, x1, y1;
        tri_cells<G::LOG>(pts[t.x], pts[t.y], pts[t.z], x0, y0, x1, y1);
        n += (unsigned long long)((x1 - x0 + 1) * (y1 - y0 + 1));
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) n += __shfl_down(n, d, 64);
    if (__lane_id() == 0 && n) atomicAdd(total, n);
}

// By the buffers of build_bitmap: only where the triangles' cells fit and their
// entries (no more than the pairs of triangle and cell) might not, the bitmap
// itself tells.
void require_bitmap(Ctx& c, const int2* pts, const int3* tri, int T, size_t top, size_t more)
{
    if (!g_arena) return;
    static_assert(C_TOTAL % 2 == 0, "an aligned 64-bit word");
    FillJobs f;
    f.add(c.dcnt.p + C_TOTAL, 0, 2);
    fill_jobs(c, f);
    k_bm_pairs<GridOne><<<grid_for(T), kBlock, 0, c.st>>>(GridOne{}, pts, tri, T, (unsigned long long*)(c.dcnt.p + C_TOTAL));
    GCDT_LAUNCH_CHECK();
    c.read(C_TOTAL, 2);
    const size_t npairs = ((size_t)(unsigned)c.hcnt[C_TOTAL + 1] << 32) | (unsigned)c.hcnt[C_TOTAL];
    const size_t cells = top + Arena::size(sizeof(int) * ((size_t)T + 1)) + 2 * Arena::size(sizeof(int) * npairs) +
                         Arena::size(sizeof(int) * (BITMAP_CELLS + 1));
    g_arena->require(cells);
    if (cells + Arena::size(sizeof(int) * npairs) + more <= g_arena->cap) return;
    DBuf<int> pad;
    hold_to(pad, top);
    int *bo, *bt, nbt;
    build_bitmap(c, pts, tri, T, &bo, &bt, &nbt);
    g_arena->require(g_arena->top + more);
    dev_give(bo, sizeof(int) * (BITMAP_CELLS + 1));
    dev_give(bt, sizeof(int) * (size_t)(nbt > 0 ? nbt : 1));
}

// ================================================================== adjacency from a triangle list

__global__ __launch_bounds__(kBlock) void k_adj_count(const int3* tri, int T, int* cnt)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < 3LL * T; i += (long long)gridDim.x * blockDim.x) {
        int t = (int)(i / 3), k = (int)(i % 3);
        int3 tv = tri[t];
        int u = get3(tv, nx3(k)), v = get3(tv, pv3(k));
        atomicAdd(&cnt[min(u, v)], 1);
    }
}

__global__ __launch_bounds__(kBlock) void k_adj_fill(const int3* tri, int T, const int* off, int* cur, int* bucket)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < 3LL * T; i += (long long)gridDim.x * blockDim.x) {
        int t = (int)(i / 3), k = (int)(i % 3);
        int3 tv = tri[t];
        int u = get3(tv, nx3(k)), v = get3(tv, pv3(k));
        int key = min(u, v);
        bucket[off[key] + atomicAdd(&cur[key], 1)] = (int)i;
    }
}

__global__ __launch_bounds__(kBlock) void k_adj_match(const int3* tri, int T, const int* off, const int* bucket, int* adj)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < 3LL * T; i += (long long)gridDim.x * blockDim.x) {
        int t = (int)(i / 3), k = (int)(i % 3);
        int3 tv = tri[t];
        int u = get3(tv, nx3(k)), v = get3(tv, pv3(k));
        int key = min(u, v);
        int r = -1;
        for (int j = off[key], e = off[key + 1]; j < e; j++) {
            int h = bucket[j];
            if (h == (int)i) continue;
            int3 w = tri[h / 3];
            int kk = h % 3;
            if (get3(w, nx3(kk)) == v && get3(w, pv3(kk)) == u) {
                r = h / 3;
                break;
            }
        }
        adj[i] = r;
    }
}

__global__ __launch_bounds__(kBlock) void k_cons_mark(const int3* tri, const int* off, const int* bucket, const int2* cons,
                                                      int C, int* cflag)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < C; i += (long long)gridDim.x * blockDim.x) {
        int2 e = cons[i];
        int key = min(e.x, e.y), other = max(e.x, e.y);
        for (int j = off[key], f = off[key + 1]; j < f; j++) {
            int h = bucket[j];
            int3 w = tri[h / 3];
            int kk = h % 3;
            int a = get3(w, nx3(kk)), b = get3(w, pv3(kk));
            if (max(a, b) == other) atomicOr(&cflag[h / 3], 1 << kk);
        }
    }
}

void build_adjacency(Ctx& c, const int3* tri, int T, int nv, int3* adj)
{
    DBuf<int> off((size_t)nv + 1), cur(nv), bucket(3LL * T);
    fill_i32(c, off.p, 0, nv + 1);
    fill_i32(c, cur.p, 0, nv);
    k_adj_count<<<grid_for(3LL * T), kBlock, 0, c.st>>>(tri, T, off.p);
    GCDT_LAUNCH_CHECK();
    scan_excl_total(c, off.p, off.p, nv);
    k_adj_fill<<<grid_for(3LL * T), kBlock, 0, c.st>>>(tri, T, off.p, cur.p, bucket.p);
    GCDT_LAUNCH_CHECK();
    k_adj_match<<<grid_for(3LL * T), kBlock, 0, c.st>>>(tri, T, off.p, bucket.p, (int*)adj);
    GCDT_LAUNCH_CHECK();
}

void mark_constraint_edges(Ctx& c, const int3* tri, const int3* adj, int T, int nv, const int2* cons, int C, int* cflag)
{
    (void)adj;
    DBuf<int> off((size_t)nv + 1), cur(nv), bucket(3LL * T);
    fill_i32(c, off.p, 0, nv + 1);
    fill_i32(c, cur.p, 0, nv);
    k_adj_count<<<grid_for(3LL * T), kBlock, 0, c.st>>>(tri, T, off.p);
    GCDT_LAUNCH_CHECK();
    scan_excl_total(c, off.p, off.p, nv);
    k_adj_fill<<<grid_for(3LL * T), kBlock, 0, c.st>>>(tri, T, off.p, cur.p, bucket.p);
    GCDT_LAUNCH_CHECK();
    if (C > 0) {
        k_cons_mark<<<grid_for(C), kBlock, 0, c.st>>>(tri, off.p, bucket.p, cons, C, cflag);
        GCDT_LAUNCH_CHECK();
    }
}

}  // namespace gcdt
