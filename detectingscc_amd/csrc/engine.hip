// engine.hip -- the SCC phase engine: device-resident graph and state, the
// vHong / wHong / vSlota / wSlota phase orders, phase timing, and the C ABI
// for the device engine.
//
// The reference drives every phase from the host with a 1-byte D2H after
// each kernel (scc_WCC.cu:683-686).  Here queue counts and fixpoint flags
// live on the device: a direction-optimised search decides each level on
// the device and the host queues windows of levels per look at the
// counters; the reference mappings queue `check_every` levels; trim-1
// queues several passes per look; other fixpoints look once per sweep.
// A look is a one-workgroup kernel that publishes the counters into
// mapped host memory, on which the host spins.
#include <chrono>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include <algorithm>

#include "batch.h"
#include "engine.h"
#include "host_util.h"
#include "merge.h"

namespace sccamd {

#define HIP_TRY(call)                                                                       \
    do {                                                                                    \
        hipError_t _e = (call);                                                             \
        if (_e != hipSuccess)                                                               \
            return fail(SCC_ERR_DEVICE, "%s failed: %s (%s:%d)", #call, hipGetErrorString(_e), \
                        __FILE__, __LINE__);                                                \
    } while (0)

static const char *const kPhaseNames[SCC_PHASE_COUNT] = {
    "trim1", "trim2", "pivot", "reach", "update", "wcc", "color", "local", "merge", "label"};

const char *phase_name(int p) { return (p >= 0 && p < SCC_PHASE_COUNT) ? kPhaseNames[p] : "?"; }

Engine::~Engine() { release(); }

void Engine::release()
{
    if (device >= 0) (void)hipSetDevice(device);
    auto f = [](void *p) {
        if (p) (void)hipFree(p);
    };
    f(g.Fr); f(g.Fc); f(g.Br); f(g.Bc); f(g.F1); f(g.B1); f(g.DP);
    f(st.cls); f(st.lab); f(st.aux); f(st.fvis); f(st.bvis); f(st.piv);
    for (int i = 0; i < 2; i++) {
        f(st.qf[i]); f(st.qb[i]);
    }
    for (int i = 0; i < 3; i++) {
        f(st.bigf[i]); f(st.bigb[i]); f(st.bigoff_f[i]); f(st.bigoff_b[i]);
    }
    f(st.pivlist); f(st.stamp); f(st.part); f(st.ctr); f(st.bred); f(d_tmp8);
    drop_spare();
    for (auto &b : buf) {
        f(b.p);
        b = DevBuf();
    }
    f(low_buf.p);
    low_buf = DevBuf();
    sub.reset();
    f(small_q);
    small_q = nullptr;
    if (h_ctr) (void)hipHostFree(h_ctr);
    if (h_pub) (void)hipHostFree(h_pub);
    h_pub = nullptr;
    d_pub = nullptr;
    for (auto e : events) (void)hipEventDestroy(e);
    events.clear();
    if (stream) (void)hipStreamDestroy(stream);
    g = DevGraph();
    st = DevState();
    d_tmp8 = nullptr;
    h_ctr = nullptr;
    stream = nullptr;
    capV = capE = 0;
}

scc_status Engine::init(int dev)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0)
        return fail(SCC_ERR_DEVICE, "no HIP device available");
    if (dev < 0 || dev >= n) return fail(SCC_ERR_INVALID, "device %d out of range (0..%d)", dev, n - 1);
    device = dev;
    HIP_TRY(hipSetDevice(dev));
    scc_status ns = noalloc_init(dev);
    if (ns != SCC_OK) return ns;
    HIP_TRY(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    HIP_TRY(hipHostMalloc((void **)&h_ctr, CT(kCtrLines) * sizeof(uint32_t), hipHostMallocDefault));
    HIP_TRY(hipMalloc((void **)&st.ctr, CT(kCtrLines) * sizeof(uint32_t)));
    // on the engine's stream: it does not wait for the null stream, where a
    // memset may still be queued (behind another engine's kernels, say) when
    // this call returns, and would then clear the counters of a later run
    (void)hipGetLastError();   // an earlier call's error, the caller's own perhaps, is not this launch's
    k_fill_u32(stream, st.ctr, 0u, CT(kCtrLines));
    HIP_TRY(hipGetLastError());
    // counters published into mapped, coherent host memory: C_COUNT lines
    // plus one line for the sequence word (without it, read-backs copy and
    // synchronise the stream)
    if (hipHostMalloc((void **)&h_pub, 2 * CT(C_COUNT + 1) * sizeof(uint32_t),
                      hipHostMallocMapped | hipHostMallocCoherent) == hipSuccess) {
        std::memset(h_pub, 0, 2 * CT(C_COUNT + 1) * sizeof(uint32_t));
        if (hipHostGetDevicePointer((void **)&d_pub, h_pub, 0) != hipSuccess) {
            (void)hipGetLastError();
            (void)hipHostFree(h_pub);
            h_pub = nullptr;
            d_pub = nullptr;
        }
    } else {
        (void)hipGetLastError();
        h_pub = nullptr;
    }
    HIP_TRY(hipMalloc((void **)&small_q, 4 * (SMALL_V + 2) * sizeof(uint32_t)));
    int rate_khz = 0;
    if (hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, dev) == hipSuccess && rate_khz > 0)
        ticks_per_ms = (double)rate_khz;
    // diagnostic: SCC_TRACE_LEVELS=1 prints every host decision of a search
    const char *tr = std::getenv("SCC_TRACE_LEVELS");
    trace_levels = tr && tr[0] == '1';
    // a bound on the scratch and optional arrays, past which the engine acts
    // as where the device has no more memory
    const char *limit = std::getenv("SCC_SCRATCH_LIMIT");
    if (limit && limit[0]) extra_limit = std::strtoull(limit, nullptr, 10);
    return SCC_OK;
}

template <class T> static hipError_t dalloc(T **p, size_t n)
{
    return hipMalloc((void **)p, sizeof(T) * (n ? n : 1));
}

// Whether a graph of V vertices and E arcs fits the arrays as allocated.  The
// queues' slot regions depend on V through the grid sizes: a smaller graph in
// a larger context must fit the queues too (they grow with V, and this keeps
// it so).
bool Engine::fits(uint32_t V, uint32_t E) const
{
    const bool queues_fit = std::max(queue_words(V), trim_list_words(V)) <= qf_words && queue_words(V) <= qb_words;
    return V <= capV && E <= capE && queues_fit;
}

// (Re)allocate device arrays for V vertices and E arcs.
scc_status Engine::reserve(uint32_t V, uint32_t E)
{
    HIP_TRY(hipSetDevice(device));
    if (fits(V, E)) return SCC_OK;
    uint32_t nV = V > capV ? V : capV, nE = E > capE ? E : capE;
    // keep the context, drop the arrays
    auto f = [](void *p) {
        if (p) (void)hipFree(p);
    };
    f(g.Fr); f(g.Fc); f(g.Br); f(g.Bc); f(g.F1); f(g.B1); f(g.DP);
    f(st.cls); f(st.lab); f(st.aux); f(st.fvis); f(st.bvis); f(st.piv);
    for (int i = 0; i < 2; i++) {
        f(st.qf[i]); f(st.qb[i]);
    }
    for (int i = 0; i < 3; i++) {
        f(st.bigf[i]); f(st.bigb[i]); f(st.bigoff_f[i]); f(st.bigoff_b[i]);
    }
    f(st.pivlist); f(st.stamp); f(st.part); f(st.bred); f(d_tmp8);
    (void)give_back();
    uint32_t *ctr = st.ctr;
    g = DevGraph();
    st = DevState();
    st.ctr = ctr;
    capV = capE = 0;
    has_graph = has_part = ran = false;   // the caller sets them again, unless the allocation fails
    const size_t nv = (size_t)nV + 1;
    const size_t nwords = 2 * ((nv + 63) / 64);
    hipError_t e = hipSuccess;
    auto A = [&](hipError_t r) {
        if (r != hipSuccess && e == hipSuccess) e = r;
    };
    A(dalloc(&g.Fr, nv + 1)); A(dalloc(&g.Br, nv + 1));
    A(dalloc(&g.Fc, nE)); A(dalloc(&g.Bc, nE));
    A(dalloc(&g.F1, nv)); A(dalloc(&g.B1, nv)); A(dalloc(&g.DP, nv));
    A(dalloc(&st.cls, nv)); A(dalloc(&st.lab, nv)); A(dalloc(&st.aux, nv));
    A(dalloc(&st.fvis, 2 * nwords)); A(dalloc(&st.bvis, 2 * nwords));
    A(dalloc(&st.piv, 3 * nv + 3));
    // the FW queues also hold the trim-1 lists; sized for the largest of
    // nV and V (slot regions follow the grid sizes of the graph uploaded)
    qf_words = std::max({queue_words(nV), trim_list_words(nV), queue_words(V), trim_list_words(V)});
    qb_words = std::max(queue_words(nV), queue_words(V));
    for (int i = 0; i < 2; i++) {
        A(dalloc(&st.qf[i], qf_words)); A(dalloc(&st.qb[i], qb_words));
    }
    // a hub list holds vertices of degree >= LB_BIG only
    const size_t nhub = std::min<size_t>(nv, (size_t)nE / LB_BIG + 1);
    for (int i = 0; i < 3; i++) {
        A(dalloc(&st.bigf[i], nhub)); A(dalloc(&st.bigb[i], nhub));
        A(dalloc(&st.bigoff_f[i], nhub)); A(dalloc(&st.bigoff_b[i], nhub));
    }
    // d_tmp8 also holds the single-class trim's live bitmap (live_bits())
    A(dalloc(&st.pivlist, nv)); A(dalloc(&st.stamp, nv)); A(dalloc(&st.part, nv + 1));
    A(dalloc(&d_tmp8, std::max(nv, 4 * (nwords + 2))));
    A(dalloc(&st.bred, 2 * (size_t)VIS_BLOCKS));
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(e == hipErrorOutOfMemory ? SCC_ERR_NOMEM : SCC_ERR_DEVICE,
                    "Error: Not enough memory on GPU (V=%u E=%u): %s", nV, nE, hipGetErrorString(e));
    }
    st.nwords = (uint32_t)nwords;
    capV = nV;
    capE = nE;
    k_fill_u32(stream, st.stamp, 0u, nv);   // no epoch is 0
    trim_epoch = 0;
    return SCC_OK;
}

// Words of the first mirror buffer's sequence line that hold the upload
// check's results, one per direction.
constexpr int kCheckWord = 16;

// Host-side validation of the reference layout: a malformed CSR must be
// rejected before any kernel indexes with it.
static scc_status validate_csr(uint32_t V, uint32_t E, const uint32_t *R, const uint32_t *C,
                               const char *name)
{
    if (R[0] != 0 || R[1] != 0 || R[V + 1] != E)
        return fail(SCC_ERR_INVALID, "%s row array must start 0,0 and end at E=%u", name, E);
    std::atomic<int> bad{0};
    parallel_chunks((uint64_t)V + 1, [&](uint64_t b, uint64_t e, int) {
        for (uint64_t v = b; v < e; v++)
            if (R[v] > R[v + 1]) bad = 1;
    });
    if (bad) return fail(SCC_ERR_INVALID, "%s row array is not monotone", name);
    parallel_chunks(E, [&](uint64_t b, uint64_t e, int) {
        for (uint64_t i = b; i < e; i++)
            if (C[i] < 1 || C[i] > V) bad = 1;
    });
    if (bad) return fail(SCC_ERR_INVALID, "%s column entry outside [1, %u]", name, V);
    return SCC_OK;
}

// Second set of graph arrays, of the first set's capacity, for uploads that
// are checked on the device: the graph that is there stays whole until the
// new one has passed.  Bounded; without it the host checks before the copy.
static constexpr uint64_t kSpareMax = 2ull << 30;   // bytes

bool Engine::spare_set()
{
    if (spare.Fr) return true;
    const size_t rows = (size_t)capV + 2;
    const uint64_t bytes = 8 * ((uint64_t)rows + capE);
    if (bytes > kSpareMax || extra_bytes() + bytes > extra_limit) return false;
    hipError_t e[4] = {dalloc(&spare.Fr, rows), dalloc(&spare.Br, rows), dalloc(&spare.Fc, capE),
                       dalloc(&spare.Bc, capE)};
    for (hipError_t r : e)
        if (r != hipSuccess) {
            (void)hipGetLastError();
            drop_spare();
            return false;
        }
    return true;
}

uint64_t Engine::extra_bytes() const
{
    uint64_t n = low_buf.cap + (spare.Fr ? 8 * ((uint64_t)capV + 2 + capE) : 0);
    for (const auto &b : buf) n += b.cap;
    return n;
}

bool Engine::give_back()
{
    if (!spare.Fr && !low_buf.p) return false;
    (void)hipSetDevice(device);
    (void)hipStreamSynchronize(stream);
    drop_spare();
    if (low_buf.p) (void)hipFree(low_buf.p);
    low_buf = DevBuf();
    return true;
}

void Engine::drop_spare()
{
    for (uint32_t *p : {spare.Fr, spare.Br, spare.Fc, spare.Bc})
        if (p) (void)hipFree(p);
    spare = DevGraph();
}

// The arrays are checked before any kernel of a run indexes with them: from
// kDeviceCheck vertices or arcs on by the device after the copy, in an array
// set that no run sees before it has passed; on the host before the copy
// below that, and where the first set has to grow or no second one can be had
// while an earlier graph is held.  What the device finds wrong the host check
// names.  Upload with the host's passes (whose threads start at 4,096
// entries) and with the device's: 1,000 vertices and 4,000 arcs 52 and 49 us,
// 2,000 and 8,000 560 and 69, 60,000 and 240,000 1,219 and 118, 2^20 and 2^23
// 4,185 and 2,574.
static constexpr uint32_t kDeviceCheck = 4096;

scc_status Engine::upload(uint32_t V, uint32_t E, const uint32_t *Fr, const uint32_t *Fc,
                          const uint32_t *Br, const uint32_t *Bc, bool checked)
{
    if (!Fr || !Br || (E && (!Fc || !Bc))) return fail(SCC_ERR_INVALID, "null graph array");
    if (V >= (1u << 30)) return fail(SCC_ERR_INVALID, "V=%u exceeds 2^30-1", V);
    auto host_check = [&]() {
        const scc_status c = validate_csr(V, E, Fr, Fc, "Fr/Fc");
        return c != SCC_OK ? c : validate_csr(V, E, Br, Bc, "Br/Bc");
    };
    scc_status s;
    HIP_TRY(hipSetDevice(device));
    const bool keep = has_graph;   // a graph that a rejected upload leaves in place
    const bool on_device = !checked && d_pub && std::max(V, E) >= kDeviceCheck && (!keep || (fits(V, E) && spare_set()));
    if (!checked && !on_device && (s = host_check()) != SCC_OK) return s;
    if ((s = reserve(V, E)) != SCC_OK) {
        const scc_status c = on_device ? host_check() : SCC_OK;
        return c != SCC_OK ? c : s;
    }
    DevGraph &to = on_device && keep ? spare : g;
    uint32_t *const flag = h_pub ? h_pub + CT(C_COUNT) + kCheckWord : nullptr;
    if (on_device) {
        flag[0] = flag[1] = 0;
        (void)hipGetLastError();   // an earlier call's
    }
    const uint32_t *const rows[2] = {Fr, Br}, *const cols[2] = {Fc, Bc};
    uint32_t *const drows[2] = {to.Fr, to.Br}, *const dcols[2] = {to.Fc, to.Bc};
    for (int d = 0; d < 2; d++) {
        HIP_TRY(hipMemcpyAsync(drows[d], rows[d], sizeof(uint32_t) * ((size_t)V + 2), hipMemcpyHostToDevice, stream));
        if (E) HIP_TRY(hipMemcpyAsync(dcols[d], cols[d], sizeof(uint32_t) * E, hipMemcpyHostToDevice, stream));
        if (on_device) {
            k_check_csr(stream, drows[d], dcols[d], V, E, d_pub + CT(C_COUNT) + kCheckWord + d);
            HIP_TRY(hipGetLastError());   // a check that did not run finds nothing wrong
        }
    }
    HIP_TRY(hipStreamSynchronize(stream));
    if (on_device && (flag[0] || flag[1])) {
        const scc_status c = host_check();
        return c != SCC_OK ? c : fail(SCC_ERR_INVALID, "the graph arrays changed during the upload");
    }
    if (&to == &spare) {
        std::swap(g.Fr, spare.Fr);
        std::swap(g.Fc, spare.Fc);
        std::swap(g.Br, spare.Br);
        std::swap(g.Bc, spare.Bc);
    }
    g.V = V;
    g.E = E;
    has_graph = true;
    has_part = false;
    ran = false;
    return SCC_OK;
}

// Partition ids are remapped to dense 0..K-1 (order kept) so that the local
// classes 3*id stay inside the pivot table.
scc_status Engine::upload_partition(const uint32_t *part)
{
    if (!has_graph) return fail(SCC_ERR_NOTREADY, "no graph uploaded");
    std::vector<uint32_t> ids(part + 1, part + 1 + g.V);
    std::sort(ids.begin(), ids.end());
    ids.erase(std::unique(ids.begin(), ids.end()), ids.end());
    std::vector<uint32_t> dense((size_t)g.V + 2, 0);
    parallel_chunks(g.V, [&](uint64_t b, uint64_t e, int) {
        for (uint64_t v = b + 1; v <= e; v++)
            dense[v] = (uint32_t)(std::lower_bound(ids.begin(), ids.end(), part[v]) - ids.begin());
    });
    // on the engine's stream (non-blocking, so not ordered with the null
    // stream): after any queued work that reads the partition, before the
    // next run's; the synchronisation keeps `dense` alive until copied
    HIP_TRY(hipMemcpyAsync(st.part, dense.data(), sizeof(uint32_t) * ((size_t)g.V + 2), hipMemcpyHostToDevice,
                           stream));
    HIP_TRY(hipStreamSynchronize(stream));
    num_parts = (uint32_t)ids.size();
    has_part = true;
    return SCC_OK;
}

scc_status Engine::adopt_begin(uint32_t V, uint32_t E)
{
    if (V >= (1u << 30)) return fail(SCC_ERR_INVALID, "V=%u exceeds 2^30-1", V);
    has_graph = has_part = ran = false;
    scc_status s = reserve(V, E);
    if (s != SCC_OK) return s;
    g.V = V;
    g.E = E;
    return SCC_OK;
}

void Engine::adopt_end()
{
    has_graph = true;
    has_part = false;
    ran = false;
}

// Adopt a graph that is already in device memory (copied device to device).
// Used for the quotient graph, whose CSR is built by kernels and valid by
// construction.
scc_status Engine::upload_device(uint32_t V, uint32_t E, const uint32_t *dFr, const uint32_t *dFc,
                                 const uint32_t *dBr, const uint32_t *dBc, hipStream_t from)
{
    if (V >= (1u << 30)) return fail(SCC_ERR_INVALID, "V=%u exceeds 2^30-1", V);
    scc_status s;
    if ((s = reserve(V, E)) != SCC_OK) return s;
    g.V = V;
    g.E = E;
    HIP_TRY(hipStreamSynchronize(from));
    HIP_TRY(hipMemcpyAsync(g.Fr, dFr, sizeof(uint32_t) * ((size_t)V + 2), hipMemcpyDeviceToDevice, stream));
    HIP_TRY(hipMemcpyAsync(g.Br, dBr, sizeof(uint32_t) * ((size_t)V + 2), hipMemcpyDeviceToDevice, stream));
    if (E) {
        HIP_TRY(hipMemcpyAsync(g.Fc, dFc, sizeof(uint32_t) * E, hipMemcpyDeviceToDevice, stream));
        HIP_TRY(hipMemcpyAsync(g.Bc, dBc, sizeof(uint32_t) * E, hipMemcpyDeviceToDevice, stream));
    }
    has_graph = true;
    has_part = false;
    ran = false;
    return SCC_OK;
}

template <class T> scc_status Engine::scratch(DevBuf &b, size_t n, T **out)
{
    const size_t bytes = sizeof(T) * (n ? n : 1);
    if (b.cap < bytes) {
        if (b.p) (void)hipFree(b.p);
        b.p = nullptr;
        b.cap = 0;
        // past the bound it asks for more than any device has, which the runtime refuses
        auto get = [&] { return hipMalloc(&b.p, extra_bytes() + bytes > extra_limit ? SIZE_MAX / 4 : bytes); };
        // an allocation that fails is tried again without the optional arrays
        hipError_t e = get();
        if (e != hipSuccess) {
            (void)hipGetLastError();   // not to be taken for a launch's
            if (give_back()) e = get();
        }
        if (e != hipSuccess) {
            (void)hipGetLastError();
            b.p = nullptr;
            return fail(SCC_ERR_NOMEM, "Error: Not enough memory on GPU (%zu scratch bytes)", bytes);
        }
        b.cap = bytes;
    }
    *out = static_cast<T *>(b.p);
    return SCC_OK;
}

// Both words of every counter line into host memory the GPU writes
// directly, then the sequence number (system-scope release).
// Words of each counter line the host reads: 32- and 64-bit counters use
// words 0..1, the search state (DirState) words 0..kDirStateWords-1.
constexpr int kPubWords = kDirStateWords;

// A spread counter is published as its own word plus its slots (the work
// units, which only a run with sizes counts, if `wide`).
__global__ void publish_ctr_kernel(const uint32_t *ctr, uint32_t *pub, uint32_t seq, int wide)
{
    const uint32_t i = threadIdx.x;
    if (i < C_COUNT) {
        for (int w = 0; w < kPubWords; w++) pub[CT(i) + w] = ctr[CT(i) + w];
        if (spread_index((int)i) >= 0 && !wide_counter((int)i)) {
            uint32_t t = ctr[CT(i)];
            for (int j = 0; j < kSpread; j++) t += ctr[CSLOT((int)i, j)];
            pub[CT(i)] = t;
        } else if (wide && wide_counter((int)i)) {
            uint64_t t = *reinterpret_cast<const uint64_t *>(ctr + CT(i));
            for (int j = 0; j < kSpread; j++) t += *reinterpret_cast<const uint64_t *>(ctr + CSLOT((int)i, j));
            pub[CT(i)] = (uint32_t)t;
            pub[CT(i) + 1] = (uint32_t)(t >> 32);
        }
    }
    __threadfence_system();
    __syncthreads();
    if (i == 0) __hip_atomic_store(pub + CT(C_COUNT), seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The host reads the counters of everything queued before a publication.
// With the published mirror it spins on the sequence word (a few
// microseconds after the last kernel) instead of a copy plus a stream
// synchronisation (about 25 us); after kPublishWaitMs it synchronises the
// stream anyway, which also reports any device error.  The mirror has two
// buffers, publication k going to buffer k & 1, so one publication may be
// queued behind the one the host waits for (pipelined search windows): a
// caller waits for publication k before it queues k + 2.
static constexpr double kPublishWaitMs = 2000.0;
static constexpr size_t kPubBuffer = CT(C_COUNT + 1);   // words of one buffer, sequence word last

uint32_t Engine::publish_ctr()
{
    const uint32_t seq = ++pub_seq;
    if (h_pub) publish_ctr_kernel<<<1, 64, 0, stream>>>(st.ctr, d_pub + (seq & 1) * kPubBuffer, seq,
                                                       search_stats ? 1 : 0);
    return seq;
}

scc_status Engine::wait_ctr(uint32_t seq)
{
    if (!h_pub) {
        HIP_TRY(hipMemcpyAsync(h_ctr, st.ctr, CT(kCtrLines) * sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
        HIP_TRY(hipStreamSynchronize(stream));
        for (int i = 0; i < C_COUNT; i++)
            if (spread_index(i) >= 0) {
                uint64_t t = h_ctr[CT(i)] | ((uint64_t)h_ctr[CT(i) + 1] << 32);
                for (int j = 0; j < kSpread; j++)
                    t += h_ctr[CSLOT(i, j)] | ((uint64_t)h_ctr[CSLOT(i, j) + 1] << 32);
                h_ctr[CT(i)] = (uint32_t)t;
                if (wide_counter(i)) h_ctr[CT(i) + 1] = (uint32_t)(t >> 32);
            }
        return SCC_OK;
    }
    HIP_TRY(hipGetLastError());
    const uint32_t *buf = h_pub + (seq & 1) * kPubBuffer;
    const uint32_t *flag = buf + CT(C_COUNT);
    const auto t0 = std::chrono::steady_clock::now();
    for (uint64_t spin = 0; __atomic_load_n(flag, __ATOMIC_ACQUIRE) != seq; spin++) {
        if ((spin & 1023) == 1023 &&
            std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count() > kPublishWaitMs) {
            HIP_TRY(hipStreamSynchronize(stream));
            if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) != seq)
                return fail(SCC_ERR_DEVICE, "counter publication %u did not arrive", seq);
            break;
        }
        __builtin_ia32_pause();
    }
    for (int i = 0; i < C_COUNT; i++)
        for (int w = 0; w < kPubWords; w++) h_ctr[CT(i) + w] = buf[CT(i) + w];
    return SCC_OK;
}

scc_status Engine::read_ctr() { return wait_ctr(publish_ctr()); }

// Zero counters [first, first+n), both words of each (64-bit counters too)
// and the slots of spread counters.
__global__ void zero_ctr_kernel(uint32_t *ctr, uint32_t first, uint32_t n)
{
    if (threadIdx.x < n) {
        const int c = (int)(first + threadIdx.x);
        ctr[CT(c)] = 0;
        ctr[CT(c) + 1] = 0;
        if (spread_index(c) >= 0)
            for (int j = 0; j < kSpread; j++) ctr[CSLOT(c, j)] = 0;
    }
}

void Engine::zero_ctr(int first, int n)
{
    zero_ctr_kernel<<<1, 64, 0, stream>>>(st.ctr, (uint32_t)first, (uint32_t)n);
}

void Engine::mark(int phase, bool force)
{
    if (phase >= 0 && !phase_marks && !force) return;
    if (nmarks == events.size()) {
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess) return;
        events.push_back(e);
    }
    (void)hipEventRecord(events[nmarks], stream);
    mark_phase.resize(nmarks + 1);
    mark_phase[nmarks] = phase;
    nmarks++;
}

// Phase times: the interval between consecutive marks belongs to the
// phase of the earlier mark (-1 = untimed).
void Engine::collect_times(scc_stats *s)
{
    for (int p = 0; p < SCC_PHASE_COUNT; p++) s->ms_phase[p] = 0;
    s->ms_scc = 0;
    if (nmarks < 2) return;
    (void)hipEventSynchronize(events[nmarks - 1]);
    for (size_t i = 0; i + 1 < nmarks; i++) {
        float ms = 0;
        (void)hipEventElapsedTime(&ms, events[i], events[i + 1]);
        if (mark_phase[i] >= 0 && phase_marks) s->ms_phase[mark_phase[i]] += ms;
        s->ms_scc += ms;
    }
}

uint32_t Engine::bpd(int W) const
{
    uint64_t b = ((uint64_t)g.V + 1) * (uint64_t)W / 256 + 1;
    return (uint32_t)(b > 2048 ? 2048 : b);
}

void Engine::init_vis(bool elect_first, bool use_live_bits)
{
    k_init_vis(stream, g, st, elect_first, use_live_bits ? live_bits() : nullptr);
    do_seeded = elect_first ? 2 : 0;
}

// The level-L arguments of direction d (0 = FW, 1 = BW): queues alternate
// with the level, counts and hub lists rotate through three slots.
DirArgs Engine::dir_args(int d, uint32_t level) const
{
    DirArgs D;
    const int in = level & 1, out = in ^ 1;
    const int hub = d ? C_BIGB : C_BIGF;
    const int cur = level % 3, prev = (level + 2) % 3, next = (level + 1) % 3;
    D.R = d ? g.Br : g.Fr;
    D.C = d ? g.Bc : g.Fc;
    D.vis = d ? st.bvis : st.fvis;
    D.qin = d ? st.qb[in] : st.qf[in];
    D.qout = d ? st.qb[out] : st.qf[out];
    D.cnt = st.ctr + CT(d ? C_BWCNT : C_FWCNT);
    D.cslot = st.ctr + CSLOT(d ? C_BWCNT : C_FWCNT, 0);
    D.big = d ? st.bigb[cur] : st.bigf[cur];
    D.bigoff = d ? st.bigoff_b[cur] : st.bigoff_f[cur];
    D.bigc = reinterpret_cast<unsigned long long *>(st.ctr + CT(hub + cur));
    D.pbig = d ? st.bigb[prev] : st.bigf[prev];
    D.pbigoff = d ? st.bigoff_b[prev] : st.bigoff_f[prev];
    D.pbigc = reinterpret_cast<unsigned long long *>(st.ctr + CT(hub + prev));
    D.bigc_zero = reinterpret_cast<unsigned long long *>(st.ctr + CT(hub + next));
    return D;
}

// FW and/or BW search from the seeded queues until both frontiers are
// empty, `K` levels per look at the counters (reference mappings and LB).
scc_status Engine::reach(bool fw, bool bw, bool single, int expand, int W, uint32_t *levels_out)
{
    if (!fw && !bw) return SCC_OK;
    if (expand == SCC_EXPAND_DO) return reach_do(fw, bw, single, levels_out);
    do_seeded = 0;   // the seeded state is for a direction-optimised search only
    // levels queued past the end of the search are no-ops, so a look at the
    // counters every 8 levels costs at most 7 empty launches
    const int K = check_every > 0 ? check_every : 8;
    zero_ctr(C_BIGF, 6);   // both directions' hub lists start empty
    const uint32_t blocks = bpd(expand == SCC_EXPAND_VWARP ? W : 1);
    uint32_t level = 0;
    for (;;) {
        LevelArgs a;
        std::memset(&a, 0, sizeof a);
        a.cls = st.cls;
        a.level = (int)level;
        if (fw) a.d[a.ndirs++] = dir_args(0, level);
        if (bw) a.d[a.ndirs++] = dir_args(1, level);
        k_expand_level(stream, a, expand, W, single, blocks);
        level++;
        if (level % K != 0) continue;
        scc_status s = read_ctr();
        if (s != SCC_OK) return s;
        bool any = false;
        for (int d = 0; d < 2; d++) {
            if (!(d ? bw : fw)) continue;
            const uint32_t nf = h_ctr[CT((d ? C_BWCNT : C_FWCNT) + level % 3)];
            const uint64_t hubs = *reinterpret_cast<const unsigned long long *>(
                h_ctr + CT((d ? C_BIGB : C_BIGF) + (level + 2) % 3)) >> 32;
            any |= nf || hubs;
        }
        if (!any) break;
        // every level claims at least one vertex, so V+1 levels bound a search
        if (level > limit()) return no_convergence("reachability");
    }
    if (levels_out) *levels_out += level;
    return SCC_OK;
}

// Direction-optimised search.  Each level is one launch whose workgroups
// choose top-down or bottom-up per direction on the device (dir_decide), so
// the host queues a window of levels per look at the counters: kDoWindow
// levels on the full grid (kFirstWindow for a single-class search, the
// first of a decomposition: power-law graphs finish it within that many
// levels), or kSpecLevels levels on a grid sized for a few times the
// current frontier while every direction is top-down, has no hubs pending,
// grew at most kSpecRise-fold since the previous look and would have to
// grow kSpecGrowth-fold more to reach the bottom-up switch point
// (high-diameter graphs run thousands of small levels; such a window may
// not switch to bottom-up).  From the second look on the windows are
// pipelined: the next one is queued before the host reads the counters of
// the last, so the GPU does not wait for the host (its parameters come from
// the look before); a search that ends in its first window pays nothing
// for that.
// Levels queued past the end of the search are no-ops.
static constexpr int kDoWindow = 4;
// 6: the first searches of R-MAT scales 22 and 24 take 6 levels, so a
// window of 8 ran two no-op launches (about 4.5 us each on 2,048
// workgroups); a first search of 7 or more levels pays one more look
static constexpr int kFirstWindow = 6;
static constexpr int kSpecLevels = 16;
static constexpr int64_t kSpecGrowth = 8;
static constexpr int64_t kSpecRise = 2;

// The rows of a low-degree graph (this decomposition's degree pass has seen
// no vertex of more than LOW_DEG arcs one way), made on first use by a
// search; null if there is no memory for them (32 bytes per vertex).
bool Engine::low_rows_ok() const
{
    return deg_known && !h_ctr[CT(C_DEG4)] && !low_denied;
}

uint4 *Engine::low_rows()
{
    uint4 *rows = nullptr;
    if (scratch(low_buf, 2 * ((size_t)g.V + 1), &rows) != SCC_OK) {
        low_denied = true;
        return nullptr;
    }
    k_low_rows(stream, g, rows, rows + g.V + 1);
    return rows;
}

scc_status Engine::reach_do(bool fw, bool bw, bool single, uint32_t *levels_out, uint32_t max_levels, bool *done)
{
    int dirs[2], nd = 0;   // argument position -> direction
    if (fw) dirs[nd++] = 0;
    if (bw) dirs[nd++] = 1;
    const uint32_t full = do_blocks(g.V, nd);
    if (do_seeded != nd) k_do_begin(stream, st.ctr, nd);
    do_seeded = 0;
    DoArgs a;
    std::memset(&a, 0, sizeof a);
    a.cls = st.cls;
    a.ctr = st.ctr;
    a.V = g.V;
    a.ndirs = nd;
    a.qcap = slot_cap(g.V, full);   // bottom-up levels run on the full grid only
    a.count = search_stats && single ? 1 : 0;   // the first search of a run with sizes
    for (int i = 0; i < nd; i++) {
        a.PR[i] = dirs[i] ? g.Fr : g.Br;
        a.PC[i] = dirs[i] ? g.Fc : g.Bc;
        a.PF[i] = dirs[i] ? g.F1 : g.B1;
    }
    uint32_t level = 0;
    bool low = false;   // queue low-degree levels
    bool thorough = false;   // max_levels does not hold: there have been low-degree levels
    auto queue = [&](int window, uint32_t blocks) {
        a.bu_ok = blocks == full;
        a.low_next = single && deg_known && !low_denied;
        for (int k = 0; k < window; k++, level++) {
            for (int i = 0; i < nd; i++) a.d[i] = dir_args(dirs[i], level);
            a.level = (int)level;
            if (low) k_low_level(stream, a, blocks);
            else k_do_level(stream, a, single, blocks);
        }
    };
    queue(single ? kFirstWindow : kDoWindow, full);
    uint32_t seen = level, seq = publish_ctr();
    int window = 0;   // nothing is queued ahead of the first look
    bool narrow_ok = true;
    uint32_t blocks = full;
    int64_t nf_prev[2] = {0, 0};
    for (;;) {
        const bool ahead = window > 0;
        uint32_t seen_next = seen, seq_next = seq;
        if (ahead) {
            queue(window, blocks);
            seen_next = level;
            seq_next = publish_ctr();
        }
        scc_status s = wait_ctr(seq);
        if (s != SCC_OK) return s;
        // the state level `seen` would compute: levels 0..seen-1 ran
        const int64_t nlive = h_ctr[CT(C_NLIVE)];
        bool any = false, spec = true, thin = single && low_rows_ok();
        int64_t nf_max = 0;
        uint32_t end = 0;
        for (int i = 0; i < nd; i++) {
            const int d = dirs[i];
            const uint32_t last = seen - 1;
            const DirState prev = load_dir_state(h_ctr, last == 0 ? 0 : last & 1, i);
            const uint32_t nf = h_ctr[CT((d ? C_BWCNT : C_FWCNT) + seen % 3)];
            const uint32_t hubs = (uint32_t)(*reinterpret_cast<const unsigned long long *>(
                                                 h_ctr + CT((d ? C_BIGB : C_BIGF) + last % 3)) >> 32);
            const DirState next = dir_decide(prev, nf, hubs, (uint32_t)nlive, seen, true);
            if (trace_levels)
                std::fprintf(stderr, "[scc reach] after level %u: %s %s %u (hubs %u), visited %llu\n", last,
                             d ? "bw" : "fw",
                             next.mode == DIR_OFF ? "done" : next.mode == DIR_BU ? "BU" : "TD",
                             prev.mode == DIR_OFF ? 0u : nf, prev.mode == DIR_TD ? hubs : 0u,
                             (unsigned long long)next.visited);
            if (next.mode == DIR_OFF) {
                end = std::max(end, next.end);
                continue;
            }
            any = true;
            const int64_t remaining = nlive - (int64_t)next.visited;
            thin &= next.mode == DIR_TD && (int64_t)nf * kToBottomUp * kSpecGrowth <= remaining;
            if (next.mode == DIR_BU || (prev.mode == DIR_TD && hubs) || !nf_prev[i] ||
                (int64_t)nf > nf_prev[i] * kSpecRise || (int64_t)nf * kToBottomUp * kSpecGrowth > remaining)
                spec = false;
            nf_prev[i] = nf;
            nf_max = std::max<int64_t>(nf_max, nf);
        }
        if (!any) {
            // a window queued meanwhile runs as no-ops; its counters are
            // published into the other buffer, which nothing waits for
            if (levels_out) *levels_out += end + h_ctr[CT(C_NLEVELS)] + h_ctr[CT(C_NLEVELS) + 1];
            if (done) *done = true;
            return SCC_OK;
        }
        if (done && !thorough && seen >= max_levels) {
            if (levels_out) *levels_out += seen;
            *done = false;
            return SCC_OK;
        }
        // every level claims at least one vertex, so V+1 levels bound a search
        if (seen > limit()) return no_convergence("reachability");
        // Narrow frontiers: every active direction top-down from a top-down
        // level, no hubs pending, a frontier that fits the workgroup's LDS.
        // The narrow kernel continues from `level` (everything before it is
        // queued) and rewrites that level's input; nothing is queued behind
        // it until the host has read where it stopped.  After a narrow run at
        // least one window of device-wide levels runs before the next one.
        // A single-class search does not use it: its top-down levels go on
        // expanding narrow frontiers inside the device-wide launch (local
        // continuation), which is faster on every high-diameter graph
        // measured (a 20,000-vertex cycle 50 -> 25 ms, the 4096^2 grid
        // 29 -> 27.6 ms) and leaves power-law searches unchanged.
        bool narrow = narrow_ok && !single;
        for (int i = 0; i < nd && narrow; i++) {
            const int d = dirs[i];
            const uint32_t last = seen - 1;
            const DirState prev = load_dir_state(h_ctr, last == 0 ? 0 : last & 1, i);
            if (prev.mode == DIR_OFF) continue;
            const uint32_t nf = h_ctr[CT((d ? C_BWCNT : C_FWCNT) + seen % 3)];
            const uint32_t hubs = (uint32_t)(*reinterpret_cast<const unsigned long long *>(
                                                 h_ctr + CT((d ? C_BIGB : C_BIGF) + last % 3)) >> 32);
            narrow = prev.mode == DIR_TD && !hubs && nf <= narrow_cap();
        }
        narrow_ok = true;
        if (narrow) {
            for (int i = 0; i < nd; i++) a.d[i] = dir_args(dirs[i], level);
            a.level = (int)level;
            k_narrow_levels(stream, a, single);
            seen = level;
            seq = publish_ctr();
            window = 0;
            narrow_ok = false;
            nf_prev[0] = nf_prev[1] = 0;
            continue;
        }
        // A search that is still narrow after the first window, on a graph
        // of at most LOW_DEG arcs per vertex and direction: its rows go into
        // arrays of their own (0.22 ms for 16.8M vertices, and a hop then
        // takes 0.5 to 0.75 us instead of 1.25 to 2.1) and its levels run as
        // low-degree levels.
        low = thin;
        if (low && !a.A[0]) {
            uint4 *rows = low_rows();
            for (int i = 0; i < nd && rows; i++) a.A[i] = rows + (dirs[i] ? (size_t)g.V + 1 : 0);
            low = rows != nullptr;
        }
        window = spec ? kSpecLevels : kDoWindow;
        thorough |= low;
        // no level is queued past the bound (level <= max_levels: the first window fits it)
        if (done && !thorough) window = (int)std::min<uint32_t>((uint32_t)window, max_levels - level);
        blocks = full;
        if (low) blocks = (uint32_t)std::min<int64_t>(full, std::max<int64_t>(128, (nf_max * 2 + 31) / 32));
        else if (spec) blocks = (uint32_t)std::min<int64_t>(full, std::max<int64_t>(32, (nf_max * 4 + 255) / 256));
        if (!ahead) {   // after the first look: queue now, ahead from then on
            queue(window, blocks);
            seen_next = level;
            seq_next = publish_ctr();
        }
        seen = seen_next;
        seq = seq_next;
    }
}

// trim-1 to its fixpoint (scc_WCC.cu:680-687), or one pass.  After the
// first sweep each pass re-checks the neighbours of the previous pass's
// removals (listed alternately in the FW queue buffers, which are free
// outside a search) until a pass removes nothing; a pass that follows one
// removing more than 1/kTrimSweepShare of the vertices sweeps instead.  The
// kernel makes that choice from the list count, so the host queues
// kTrimQueued passes per look at the counters.
static constexpr uint32_t kTrimSweepShare = 32;
static constexpr uint32_t kTrimQueued = 4;

scc_status Engine::trim1(bool fixpoint, bool single, bool none_dead, bool wait, bool labels)
{
    mark(SCC_PHASE_TRIM1);
    // a fresh state comes straight from the state initialisation, which
    // zeroed every counter line (the removal-list counts and their slots too)
    if (!none_dead) zero_ctr(C_TLIST, 3);
    // the single-class live bitmap lives in the byte scratch array, free
    // during a decomposition; the first pivot round reads it
    uint32_t *live = single ? live_bits() : nullptr;
    const bool degree_first = fixpoint && single && none_dead;
    deg_known |= degree_first && few_arcs(g);
    const bool eager = labels || !degree_first;   // lazy: the live bitmap alone (no class or label writes)
    k_trim1(stream, g, st, st.qf[1], st.qf[0], 0u, 0, kTrimSweepShare, live, degree_first, eager);
    uint32_t pass = 1;
    if (!wait) {
        // one batch of passes and no look at the counters: the SCCs do not
        // depend on how far trimming got (what a fixpoint would still remove,
        // the phases after the first search remove), and the GPU goes on to
        // the next phase without waiting for the host
        for (uint32_t k = 0; fixpoint && k < kTrimQueued; k++, pass++) {
            if (++trim_epoch == 0) {
                k_fill_u32(stream, st.stamp, 0u, (uint64_t)g.V + 1);
                trim_epoch = 1;
            }
            k_trim1(stream, g, st, st.qf[(pass + 1) & 1], st.qf[pass & 1], trim_epoch, pass, kTrimSweepShare, live,
                    true, eager);
        }
        return SCC_OK;
    }
    while (fixpoint) {
        for (uint32_t k = 0; k < kTrimQueued; k++, pass++) {
            if (++trim_epoch == 0) {   // wrapped: no stale stamp may match a new epoch
                k_fill_u32(stream, st.stamp, 0u, (uint64_t)g.V + 1);
                trim_epoch = 1;
            }
            k_trim1(stream, g, st, st.qf[(pass + 1) & 1], st.qf[pass & 1], trim_epoch, pass, kTrimSweepShare, live,
                    true, eager);
        }
        scc_status s = read_ctr();
        if (s != SCC_OK) return s;
        // the next pass's input: what the last queued pass removed
        if (!h_ctr[CT(C_TLIST + pass % 3)]) break;
        // every pass but the last removes a vertex
        if (pass > limit()) return no_convergence("trim-1");
    }
    if (!fixpoint) return read_ctr();
    return SCC_OK;
}

uint64_t Engine::limit() const { return (uint64_t)g.V + 8; }

scc_status Engine::no_convergence(const char *what)
{
    return fail(SCC_ERR_DEVICE, "%s did not converge within %llu iterations", what,
                (unsigned long long)limit());
}

// One pivot round: elect, seed, FW||BW, update.  Returns live count.
scc_status Engine::pivot_round(bool first, int expand, int W, scc_stats *stats, uint32_t *live, int canon,
                               bool use_live_bits, bool lazy)
{
    lazy = lazy && first;
    mark(SCC_PHASE_PIVOT);
    init_vis(first, first && use_live_bits);
    if (!first) {
        k_elect(stream, g, st);
        k_select(stream, g, st);
        do_seeded = 2;
    }
    mark(SCC_PHASE_REACH, first);   // the first search is always timed
    const int first_mark = (int)nmarks - 1;
    scc_status s = reach(true, true, first, expand, W, &stats->levels);
    if (s != SCC_OK) return s;
    mark(SCC_PHASE_UPDATE, first);
    if (first) {
        first_reach_marks[0] = first_mark;
        first_reach_marks[1] = (int)nmarks - 1;
        if (search_stats) k_reach_stats(stream, g, st);
    }
    // C_LIVE is clear: in the first round (one pivot at most) from the state
    // initialisation, later from the seeding
    // the first round's update also takes its SCC's minimum (one pivot)
    if (lazy && use_live_bits) k_update_words(stream, g, st, live_bits());
    else k_update(stream, g, st, first, first && use_live_bits ? live_bits() : nullptr, lazy);
    if (!first) k_clear_piv(stream, st, g.V + 1);   // the first round's update clears its pivot's entries
    if (canon >= 0) {
        // the labels of a decomposition this round finished, in the same
        // look at the counters (a no-op on the device if a vertex is live);
        // in the first round the only non-final label is the pivot's, whose
        // minimum the update left in aux
        mark(SCC_PHASE_LABEL);
        if (lazy && canon == 0) {
            k_label_from_bits(stream, g, st);
        } else if (first) {
            k_canon_apply(stream, g, st, true);
            if (canon) k_sizes(stream, g, st, true);
        } else {
            k_canon(stream, g, st, canon != 0, true);
        }
        mark(-1);
    }
    if ((s = read_ctr()) != SCC_OK) return s;
    *live = h_ctr[CT(C_LIVE)];
    if (first) stats->first_pivot = h_ctr[CT(C_PIV0)];
    return SCC_OK;
}

scc_status Engine::min_label()
{
    mark(SCC_PHASE_WCC);
    k_minlabel_init(stream, g, st);
    scc_status s;
    uint64_t it = 0;
    do {
        if (it) zero_ctr(C_CHANGED, 1);
        k_minlabel_prop(stream, g, st);
        if ((s = read_ctr()) != SCC_OK) return s;
        if (++it > limit()) return no_convergence("min-label propagation");
    } while (h_ctr[CT(C_CHANGED)]);
    k_minlabel_finish(stream, g, st);
    return SCC_OK;
}

scc_status Engine::color_loop(int expand, int W, scc_stats *stats)
{
    scc_status s;
    for (;;) {
        if ((s = read_ctr()) != SCC_OK) return s;
        if (!h_ctr[CT(C_LIVE)]) break;
        if (++stats->rounds > limit()) return no_convergence("colouring rounds");
        mark(SCC_PHASE_COLOR);
        k_color_init(stream, g, st);
        uint64_t it = 0;
        do {
            if (it) zero_ctr(C_CHANGED, 1);
            k_color_prop(stream, g, st);
            if ((s = read_ctr()) != SCC_OK) return s;
            if (++it > limit()) return no_convergence("colour propagation");
        } while (h_ctr[CT(C_CHANGED)]);
        init_vis();
        k_color_roots(stream, g, st);
        do_seeded = 1;
        mark(SCC_PHASE_REACH);
        if ((s = reach(true, false, false, expand, W, &stats->levels)) != SCC_OK) return s;
        mark(SCC_PHASE_UPDATE);
        k_color_finish(stream, g, st);
    }
    return SCC_OK;
}

scc_status Engine::run(const scc_opts &o, scc_stats *out)
{
    if (!has_graph) return fail(SCC_ERR_NOTREADY, "no graph uploaded");
    HIP_TRY(hipSetDevice(device));
    const char A = o.algo;
    if (A != 'g' && A != 'h' && A != 'x' && A != 'y' && A != 'd')
        return fail(SCC_ERR_INVALID, "unknown algorithm '%c'", A);
    if (A == 'd' && !has_part)
        return fail(SCC_ERR_NOTREADY, "detectSCC needs a partition vector (scc_partition_upload)");
    int W = o.warp;
    if (W != 1 && W != 2 && W != 4 && W != 8 && W != 16 && W != 32 && W != 64)
        return fail(SCC_ERR_INVALID, "warp size %d not in {1,2,4,8,16,32,64}", W);
    int expand = o.expand;
    // The automatic mode is the direction-optimised search for every
    // algorithm: the labels do not depend on the expansion, and on R-MAT
    // scale 22 it is 23-42x faster than the reference's mappings, which stay
    // selectable (SCC_EXPAND_VERTEX, or SCC_EXPAND_VWARP with W lanes).
    if (expand == SCC_EXPAND_AUTO) expand = SCC_EXPAND_DO;
    if (expand != SCC_EXPAND_VERTEX && expand != SCC_EXPAND_VWARP && expand != SCC_EXPAND_LB &&
        expand != SCC_EXPAND_DO)
        return fail(SCC_ERR_INVALID, "unknown expand mode %d", expand);
    // the reference uses the virtual warp only for the first pivot's search
    // (scc_WCC.cu:209-317); the main loop uses vertex-per-thread
    const int first_expand = expand;
    const int loop_expand = (expand == SCC_EXPAND_VWARP) ? SCC_EXPAND_VERTEX : expand;
    check_every = o.check_every;
    search_stats = o.sizes != 0;
    phase_marks = o.phase_times != 0;

    scc_stats stats;
    std::memset(&stats, 0, sizeof stats);
    // A small graph in one launch: where nothing asks for the device-wide
    // engine's per-phase times, search counts or mappings (batch.h has the
    // sizes, small_scc_kernel the reason for them).
    if (A != 'd' && expand == SCC_EXPAND_DO && !o.sizes && !o.phase_times && g.V && g.V <= SMALL_V &&
        g.E <= SMALL_E && h_pub) {
        scc_status ss = run_small(A, o.trim1 != 0, o.trim2 != 0, &stats);
        if (ss != SCC_OK) return ss;
        ran = true;
        if (out) *out = stats;
        return SCC_OK;
    }
    nmarks = 0;
    first_reach_marks[0] = first_reach_marks[1] = -1;
    mark(-1);
    const bool hong = (A == 'g' || A == 'x');
    // the first trim-1 pass of Hong and detectSCC starts from the fresh
    // state and writes the per-vertex words itself
    const bool fresh_trim = o.trim1 && (hong || A == 'd');
    // The first-neighbour and degree-product arrays belong to the
    // decomposition, not to the upload: every run builds them from the CSR.
    // The fresh trim's degree pass builds them for the vertices it keeps;
    // any other path builds them for every vertex first.
    deg_known = low_denied = false;
    if (!fresh_trim) k_first_arcs(stream, g);
    k_init_state(stream, g, st, nullptr, !fresh_trim);   // also zeroes the counters
    scc_status s;
    uint32_t live = g.V;
    bool labelled = false;   // the first pivot round finished the decomposition and its labels
    if (A == 'd') {
        if ((s = detect_phases(o, loop_expand, W, &stats, false)) != SCC_OK) return s;
    } else if (hong) {
        // lazy labels: the degree pass and the first update write no labels
        // (nor the members' class words); a decomposition the first round
        // finishes takes its labels from the search's bitmaps, otherwise a
        // fix-up writes what the eager round would have (sizes needs them)
        const bool lazy = o.trim1 && !o.sizes;
        if (o.trim1 && (s = trim1(true, true, true, false, !lazy)) != SCC_OK) return s;
        // the single-class trim just left an exact live bitmap
        if ((s = pivot_round(true, first_expand, W, &stats, &live, o.sizes != 0 ? 1 : 0, o.trim1 != 0, lazy)) !=
            SCC_OK)
            return s;
        labelled = live == 0;
        if (live && lazy) k_label_fixup(stream, g, st, live_bits());
        // with no live vertex left (a power-law graph's first search often
        // takes everything trim-1 left) every later phase removes nothing,
        // elects nothing and changes no label
        if (live) {
            if (o.trim1 && (s = trim1(true)) != SCC_OK) return s;
            if (o.trim2) {
                mark(SCC_PHASE_TRIM2);
                k_trim2(stream, g, st);
            }
            if (o.trim1 && (s = trim1(true)) != SCC_OK) return s;
            if ((s = min_label()) != SCC_OK) return s;
            for (;;) {
                // a round with no live vertex elects nothing and reports live = 0
                if ((s = pivot_round(false, loop_expand, W, &stats, &live)) != SCC_OK) return s;
                if (!live) break;
                // each round finishes at least its pivots' SCCs
                if (++stats.rounds > limit()) return no_convergence("pivot rounds");
            }
        }
    } else {
        // vSlota/wSlota: one trim-1 pass, -q ignored (scc_Coloring.cu:507-508)
        if (o.trim1 && (s = trim1(false, true, false, false)) != SCC_OK) return s;
        if ((s = pivot_round(true, first_expand, W, &stats, &live, -1, o.trim1 != 0)) != SCC_OK) return s;
        if ((s = color_loop(loop_expand, W, &stats)) != SCC_OK) return s;
    }
    if (!labelled) {
        if (A != 'd') {
            mark(SCC_PHASE_LABEL);
            k_canon(stream, g, st, o.sizes != 0);
        } else if (o.sizes) {   // detectSCC labels come out of the merge already canonical
            mark(SCC_PHASE_LABEL);
            k_sizes(stream, g, st);
        }
        mark(-1);
        if ((s = read_ctr()) != SCC_OK) return s;
    }
    if (h_ctr[CT(C_ANOM)])
        return fail(SCC_ERR_DEVICE, "internal invariant violated %u times", h_ctr[CT(C_ANOM)]);
    collect_times(&stats);
    if (first_reach_marks[0] >= 0) {
        float ms = 0;
        (void)hipEventElapsedTime(&ms, events[first_reach_marks[0]], events[first_reach_marks[1]]);
        stats.ms_first_reach = ms;
    }
    auto u64 = [&](int i) { return (uint64_t)h_ctr[CT(i)] | ((uint64_t)h_ctr[CT(i) + 1] << 32); };
    stats.num_sccs = h_ctr[CT(C_NSCC)];
    stats.num_trim1 = h_ctr[CT(C_TRIM1)];
    stats.num_trim2 = h_ctr[CT(C_TRIM2)];
    stats.num_pivot = h_ctr[CT(C_PIVOT)];
    stats.largest = h_ctr[CT(C_LARGEST)];
    stats.first_fw_vertices = u64(C_FWV);
    stats.first_fw_arcs = u64(C_FWE);
    stats.first_bw_vertices = u64(C_BWV);
    stats.first_bw_arcs = u64(C_BWE);
    for (int k = 0; k < 8; k++) stats.first_work[k] = u64(C_WORK + k);
    ran = true;
    if (out) *out = stats;
    return SCC_OK;
}

// The whole decomposition as one launch of one workgroup; the device times
// come from the kernel's own clock reads.
scc_status Engine::run_small(char algo, bool trim1, bool trim2, scc_stats *stats)
{
    SmallArgs a;
    a.V = g.V;
    a.E = g.E;
    a.cfg = batch_cfg(trim1, trim2, algo == 'h' || algo == 'y');
    a.seq = ++pub_seq;
    a.Fr = g.Fr;
    a.Fc = g.Fc;
    a.Br = g.Br;
    a.Bc = g.Bc;
    a.lab = st.lab;
    a.aux = st.aux;
    a.pivlist = st.pivlist;
    a.q = small_q;
    a.pub = d_pub + (a.seq & 1) * kPubBuffer;
    a.piv = st.piv;
    k_small(stream, a);
    scc_status s = wait_ctr(a.seq);
    if (s != SCC_OK) return s;
    if (h_ctr[CT(C_ANOM)]) return fail(SCC_ERR_DEVICE, "internal invariant violated: a class without a pivot");
    auto ms = [&](int i) {
        return (double)((uint64_t)h_ctr[CT(i)] | ((uint64_t)h_ctr[CT(i) + 1] << 32)) / ticks_per_ms;
    };
    stats->num_sccs = h_ctr[CT(C_NSCC)];
    stats->num_trim1 = h_ctr[CT(C_TRIM1)];
    stats->num_trim2 = h_ctr[CT(C_TRIM2)];
    stats->num_pivot = h_ctr[CT(C_PIVOT)];
    stats->first_pivot = h_ctr[CT(C_PIV0)];
    stats->rounds = h_ctr[CT(C_NPIV)];
    stats->levels = h_ctr[CT(C_NLEVELS)];
    stats->ms_scc = ms(C_FWV);
    stats->ms_first_reach = ms(C_BWV);
    return SCC_OK;
}

// detectSCC's search across the partitions runs where more than 1 in
// kCrossShare of up to 2^16 sampled arcs lead to another partition
// (k_cross_sample, about 6 us).  With fewer the local SCCs are whole
// partitions and their quotient graph is small: 2^20 vertices in 200
// communities with no arc between them 822 us with the search and 690
// without, with 1 arc in 10,000 between them 1,855 and 840; with 1 in 1,000
// it is 587 with it and 1,018 without.
// On a low-degree graph it runs to its end: a hop takes 0.5 to 0.75 us there
// (expand_low_kernel), and the local SCCs and the quotient graph of such a
// graph are as deep in sum (the 1024^2 grid of 0.7 in 16 blocks of rows 5.6
// ms against 18.4, in random partitions 11 ms against 9.7 s, a cycle of 20,000
// in 50 parts 9.8 against 55).  Otherwise it is given up if it has not ended
// after kDetectLevels levels: on a high-diameter graph the local SCCs and
// their quotient graph may be the shorter way.  Where most arcs cross, the
// local SCCs are small and the quotient graph nearly as deep, and it gets
// kDetectDeep.  A level is one launch, and narrow ones go on for up to 64 hops
// each, so a search that is given up has cost at most about 1,000 hops of 1.3
// to 2.1 us, or 3,000.
static constexpr uint32_t kCrossShare = 2048;
static constexpr uint32_t kDetectLevels = 16, kDetectDeep = 48;

// detectSCC (scc_WCC.cu:1000-1617): trim-1, the search across the
// partitions, then, of what it leaves, trim-2 and trim-1 (1122-1173), local
// SCCs per (partition, class) (1175-1269) and the merge as a quotient-graph
// SCC computed by a second engine on the same device.  With local_only there
// is no search, and the canonical local labels are left in lab.
scc_status Engine::detect_phases(const scc_opts &o, int expand, int W, scc_stats *stats, bool local_only)
{
    if (!has_part) return fail(SCC_ERR_NOTREADY, "detectSCC needs a partition vector");
    scc_status s;
    if (!local_only) k_cross_sample(stream, g, st);   // the next look at the counters brings it
    if (o.trim1 && (s = trim1(true, true, true)) != SCC_OK) return s;
    if (!local_only && !o.trim1 && (s = read_ctr()) != SCC_OK) return s;
    // the live bitmap stays exact up to the second trim-1 (every live vertex
    // is in class 0 so far): from the trim-1 above, or from the class words
    bool bits = o.trim1 != 0;
    // Most graphs that are partitioned have one SCC across most partitions:
    // it is searched for first, over all the vertices, and trim-2, the local
    // SCCs and the quotient graph are those of what it leaves, often nothing
    // (on 8.4M vertices trim-2 alone took 300 us of class tests on vertices
    // that the search takes)
    bool found = false;
    uint32_t left = 0;
    const uint32_t cross = h_ctr[CT(C_CROSS)], sampled = h_ctr[CT(C_CROSS) + 1];
    if (!local_only && (uint64_t)cross * kCrossShare > sampled) {
        mark(SCC_PHASE_MERGE);
        if (!bits) k_live_bits(stream, g, st, live_bits());
        const uint32_t bound = 2 * (uint64_t)cross > sampled ? kDetectDeep : kDetectLevels;
        if ((s = detect_search(bound, stats, &found, &left)) != SCC_OK) return s;
        if (found) k_detect_members(stream, g, st, live_bits(), left == 0);
        if (found && !left) return SCC_OK;
        if (found) k_live_bits(stream, g, st, live_bits());
        bits = true;
    }
    if (o.trim2) {
        // nothing reads the bitmap after trim-2
        mark(SCC_PHASE_TRIM2);
        k_trim2(stream, g, st, bits ? live_bits() : nullptr);
    }
    // every live vertex is still in class 0 (trim-2 only removes), so the
    // second fixpoint runs single-class too: its first pass rebuilds the
    // live bitmap from the class words, and it tests neighbours in the bitmap
    if (o.trim1 && (s = trim1(true, true)) != SCC_OK) return s;
    mark(SCC_PHASE_LOCAL);
    uint32_t *tbits;
    if ((s = scratch(buf[0], st.nwords, &tbits)) != SCC_OK) return s;
    k_local_init(stream, g, st, tbits);
    uint32_t live = 0;
    for (;;) {
        if ((s = pivot_round(false, expand, W, stats, &live)) != SCC_OK) return s;
        if (!live) break;
        if (++stats->rounds > limit()) return no_convergence("local rounds");
    }
    mark(SCC_PHASE_LABEL);
    k_canon(stream, g, st, false);
    if (local_only) return SCC_OK;
    mark(SCC_PHASE_MERGE);
    const uint32_t *qlab = nullptr, *qid = nullptr, *rep = nullptr;
    if ((s = merge_quotient(tbits, stats, &qid, &rep, &qlab)) != SCC_OK) return s;
    zero_ctr(C_NSCC, 1);
    k_q_map(stream, g, st, tbits, qid, qlab, rep);
    return SCC_OK;
}

// FW and BW from one pivot over every live vertex (classes ignored; they are
// all still in class 0), in the live bitmap, for at most max_levels levels.
scc_status Engine::detect_search(uint32_t max_levels, scc_stats *stats, bool *found, uint32_t *left)
{
    init_vis(true, true);
    const bool counted = search_stats;
    search_stats = false;   // the work units are those of a first search
    scc_status s = reach_do(true, true, true, &stats->levels, max_levels, found);
    search_stats = counted;
    if (s != SCC_OK || !*found) return s;
    zero_ctr(C_LIVE, 1);
    k_detect_found(stream, g, st, live_bits());
    if ((s = read_ctr()) != SCC_OK) return s;
    *left = h_ctr[CT(C_LIVE)];
    return SCC_OK;
}

// The quotient graph of the local SCCs of the vertices not in tbits and its
// SCCs: qid (local SCC of each representative), rep (its vertex) and the
// labels of the quotient vertices (null: no arcs between them).
scc_status Engine::merge_quotient(const uint32_t *tbits, scc_stats *stats, const uint32_t **qid_out,
                                  const uint32_t **rep_out, const uint32_t **qlab_out)
{
    scc_status s;
    const size_t nv = (size_t)g.V + 1;
    uint32_t *isrep, *qid, *rep, *Qr, *QBr, *tiles;
    if ((s = scratch(buf[1], nv, &isrep)) != SCC_OK || (s = scratch(buf[2], nv, &qid)) != SCC_OK ||
        (s = scratch(buf[3], nv, &rep)) != SCC_OK || (s = scratch(buf[6], nv + 1, &Qr)) != SCC_OK ||
        (s = scratch(buf[7], nv + 1, &QBr)) != SCC_OK ||
        (s = scratch(buf[8], scan_tile_count(nv + 1), &tiles)) != SCC_OK)
        return s;
    *qid_out = qid;
    *rep_out = rep;
    k_q_mark(stream, g, st, tbits, isrep);
    k_exscan(stream, isrep, qid, nv, tiles);
    uint32_t last[2];
    HIP_TRY(hipMemcpyAsync(&last[0], qid + g.V, 4, hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipMemcpyAsync(&last[1], isrep + g.V, 4, hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    const uint32_t QV = last[0] + last[1];
    if (QV) {
        // quotient arcs as sorted 64-bit keys: each vertex's quotient id,
        // the keys of the arcs between different local SCCs, and two radix
        // sorts into the rows of both directions.  The keys go straight into
        // the (grow-only) buffer an earlier merge left; only a first merge,
        // or one whose keys did not fit, counts them first.
        uint32_t *qv;
        unsigned long long *qn;
        if ((s = scratch(buf[11], nv, &qv)) != SCC_OK || (s = scratch(buf[12], 1, &qn)) != SCC_OK) return s;
        k_q_vid(stream, g, st, tbits, qid, qv);
        auto read_count = [&](unsigned long long *out) -> scc_status {
            HIP_TRY(hipMemcpyAsync(out, qn, sizeof *out, hipMemcpyDeviceToHost, stream));
            HIP_TRY(hipStreamSynchronize(stream));
            return SCC_OK;
        };
        unsigned long long qe = 0;
        uint64_t *keys = static_cast<uint64_t *>(buf[13].p);
        uint64_t kcap = buf[13].cap / sizeof(uint64_t);
        for (int attempt = 0;; attempt++) {
            k_fill_u32(stream, reinterpret_cast<uint32_t *>(qn), 0u, 2);
            if (kcap) k_q_keys(stream, true, g, qv, qn, keys, kcap);
            else k_q_keys(stream, false, g, qv, qn, nullptr, 0);
            if ((s = read_count(&qe)) != SCC_OK) return s;
            if (qe > 0xFFFFFFFFull) return fail(SCC_ERR_INVALID, "quotient graph has %llu arcs", qe);
            if (kcap && qe <= kcap) break;   // every key written
            if (attempt == 2) return fail(SCC_ERR_DEVICE, "quotient arc count changed between passes");
            if ((s = scratch(buf[13], std::max<uint64_t>(qe, 1), &keys)) != SCC_OK) return s;
            kcap = buf[13].cap / sizeof(uint64_t);
        }
        const uint32_t QE = (uint32_t)qe;
        if (QE) {
            uint32_t *Qc, *QBc;
            uint64_t *sorted;
            void *tmp;
            const size_t tmp_bytes = csr_sort_bytes(QV, QE);
            if ((s = scratch(buf[9], QE, &Qc)) != SCC_OK || (s = scratch(buf[10], QE, &QBc)) != SCC_OK ||
                (s = scratch(buf[14], QE, &sorted)) != SCC_OK ||
                (s = scratch(buf[15], tmp_bytes, reinterpret_cast<uint8_t **>(&tmp))) != SCC_OK)
                return s;
            if ((s = csr_from_keys(stream, QV, QE, keys, sorted, tmp, tmp_bytes, Qr, Qc, QBr, QBc)) != SCC_OK)
                return s;
            k_q_rep(stream, g, isrep, qid, rep);
            if (!sub) {
                sub.reset(new Engine());
                if ((s = sub->init(device)) != SCC_OK) return s;
            }
            s = sub->upload_device(QV, QE, Qr, Qc, QBr, QBc, stream);
            if (s == SCC_ERR_NOMEM && give_back()) s = sub->upload_device(QV, QE, Qr, Qc, QBr, QBc, stream);
            if (s != SCC_OK) return s;
            scc_opts so;
            scc_opts_default(&so);
            so.algo = 'g';
            so.expand = SCC_EXPAND_DO;
            so.sizes = 0;
            scc_stats sst;
            if ((s = sub->run(so, &sst)) != SCC_OK) return s;
            // its labels are read on this engine's stream: a small graph's
            // counters arrive before its kernel has ended
            HIP_TRY(hipStreamSynchronize(sub->stream));
            *qlab_out = sub->st.lab;
            stats->levels += sst.levels;
        }
    }
    return SCC_OK;
}

// The condensation DAG of the last run: node k = the SCC with the k-th
// smallest canonical label, an arc per distinct pair of SCCs joined by an
// arc.  The quotient kernels of the detectSCC merge count and place the arcs
// between different SCCs on the device (no vertex excluded: an empty
// finished bitmap); the host sorts, removes parallel arcs and builds the
// reverse rows.
scc_status Engine::condense(scc_host_graph *out, uint32_t *node_of)
{
    if (!ran) return fail(SCC_ERR_NOTREADY, "no completed run");
    std::memset(out, 0, sizeof *out);
    const size_t nv = (size_t)g.V + 1;
    uint32_t *none, *isrep, *qid, *cout, *cin, *Qr, *QBr, *tiles;
    scc_status s;
    if ((s = scratch(buf[0], st.nwords, &none)) != SCC_OK || (s = scratch(buf[1], nv, &isrep)) != SCC_OK ||
        (s = scratch(buf[2], nv, &qid)) != SCC_OK || (s = scratch(buf[4], nv + 1, &cout)) != SCC_OK ||
        (s = scratch(buf[5], nv + 1, &cin)) != SCC_OK || (s = scratch(buf[6], nv + 1, &Qr)) != SCC_OK ||
        (s = scratch(buf[7], nv + 1, &QBr)) != SCC_OK ||
        (s = scratch(buf[8], scan_tile_count(nv + 1), &tiles)) != SCC_OK)
        return s;
    k_fill_u32(stream, none, 0u, st.nwords);
    k_q_mark(stream, g, st, none, isrep);
    k_exscan(stream, isrep, qid, nv, tiles);
    std::vector<uint32_t> hq(nv), hlab(nv), hrep(nv);
    HIP_TRY(hipMemcpyAsync(hq.data(), qid, sizeof(uint32_t) * nv, hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipMemcpyAsync(hrep.data(), isrep, sizeof(uint32_t) * nv, hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipMemcpyAsync(hlab.data(), st.lab, sizeof(uint32_t) * nv, hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    const uint32_t QV = hq[g.V] + hrep[g.V];
    if (node_of) {
        node_of[0] = 0;
        for (uint32_t v = 1; v <= g.V; v++) node_of[v] = hq[hlab[v]] + 1;
    }
    std::vector<uint32_t> src, dst;
    if (QV) {
        k_fill_u32(stream, cout, 0, (uint64_t)QV + 2);
        k_fill_u32(stream, cin, 0, (uint64_t)QV + 2);
        k_q_arcs(stream, 0, g, st, none, qid, cout, cin, nullptr, nullptr);
        k_exscan(stream, cout, Qr, (uint64_t)QV + 2, tiles);
        k_exscan(stream, cin, QBr, (uint64_t)QV + 2, tiles);
        std::vector<uint32_t> hr((size_t)QV + 2);
        HIP_TRY(hipMemcpyAsync(hr.data(), Qr, sizeof(uint32_t) * hr.size(), hipMemcpyDeviceToHost, stream));
        HIP_TRY(hipStreamSynchronize(stream));
        const uint32_t QE = hr[QV + 1];
        if (QE) {
            uint32_t *Qc, *QBc;
            if ((s = scratch(buf[9], QE, &Qc)) != SCC_OK || (s = scratch(buf[10], QE, &QBc)) != SCC_OK)
                return s;
            HIP_TRY(hipMemcpyAsync(cout, Qr, sizeof(uint32_t) * ((size_t)QV + 2), hipMemcpyDeviceToDevice, stream));
            HIP_TRY(hipMemcpyAsync(cin, QBr, sizeof(uint32_t) * ((size_t)QV + 2), hipMemcpyDeviceToDevice, stream));
            k_q_arcs(stream, 1, g, st, none, qid, cout, cin, Qc, QBc);
            dst.resize(QE);
            HIP_TRY(hipMemcpyAsync(dst.data(), Qc, sizeof(uint32_t) * QE, hipMemcpyDeviceToHost, stream));
            HIP_TRY(hipStreamSynchronize(stream));
            src.resize(QE);
            for (uint32_t q = 1; q <= QV; q++)
                for (uint32_t i = hr[q]; i < hr[q + 1]; i++) src[i] = q;
        }
    }
    scc_host_graph dag;
    const uint32_t none_arc = 0;
    if ((s = scc_csr_from_arcs(QV, src.size(), src.empty() ? &none_arc : src.data(),
                               dst.empty() ? &none_arc : dst.data(), &dag)) != SCC_OK)
        return s;
    // parallel arcs out: rows are sorted, so keep the first of each run
    auto dedupe = [&](uint32_t *R, uint32_t *C) {
        uint32_t w = 0;
        for (uint32_t v = 1; v <= QV; v++) {
            const uint32_t b = R[v], e = R[v + 1];
            R[v] = w;
            for (uint32_t i = b; i < e; i++)
                if (i == b || C[i] != C[i - 1]) C[w++] = C[i];
        }
        R[QV + 1] = w;
        return w;
    };
    const uint32_t E1 = dedupe(dag.Fr, dag.Fc), E2 = dedupe(dag.Br, dag.Bc);
    if (E1 != E2) {
        scc_host_graph_free(&dag);
        return fail(SCC_ERR_DEVICE, "condensation rows disagree (%u forward, %u reverse arcs)", E1, E2);
    }
    dag.E = E1;
    *out = dag;
    return SCC_OK;
}

scc_status Engine::labels(uint32_t *lab)
{
    if (!ran) return fail(SCC_ERR_NOTREADY, "no completed run");
    HIP_TRY(hipMemcpyAsync(lab, st.lab, sizeof(uint32_t) * ((size_t)g.V + 1), hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return SCC_OK;
}

// The size histogram of the last run, on the device (k_size_histogram): sizes
// from the canonical labels, then the per-size counts and their non-zero
// entries (at most floor(sqrt(2V)) + 1 distinct sizes: the sizes of distinct
// SCCs sum to at most V).  *ms is the device time of its four passes.
scc_status Engine::histogram(uint64_t *pairs, uint32_t cap, uint32_t *npairs, double *ms)
{
    if (!ran) return fail(SCC_ERR_NOTREADY, "no completed run");
    HIP_TRY(hipSetDevice(device));
    uint32_t kmax = 1;
    while ((uint64_t)kmax * (kmax + 1) / 2 <= g.V) kmax++;
    // the number of pairs found, a pad word, then the pairs
    uint64_t *dn;
    scc_status s;
    if ((s = scratch(buf[11], 2 * (size_t)kmax + 2, &dn)) != SCC_OK) return s;
    uint64_t *const dpairs = dn + 2;
    if (events.size() < 2) {
        for (size_t i = events.size(); i < 2; i++) {
            hipEvent_t e;
            HIP_TRY(hipEventCreate(&e));
            events.push_back(e);
        }
    }
    nmarks = 0;   // the run's phase marks are already collected
    HIP_TRY(hipEventRecord(events[0], stream));
    k_size_histogram(stream, g, st, st.aux, dpairs, kmax, reinterpret_cast<uint32_t *>(dn));
    HIP_TRY(hipEventRecord(events[1], stream));
    // the count and the first pairs in one copy (a power-law graph has a few
    // dozen sizes), the rest in another
    const size_t first = std::min<size_t>(kmax, 255);
    std::vector<uint64_t> h(2 * first + 2);
    HIP_TRY(hipMemcpyAsync(h.data(), dn, sizeof(uint64_t) * h.size(), hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    const uint32_t n = (uint32_t)h[0];
    if (n > kmax) return fail(SCC_ERR_DEVICE, "%u distinct SCC sizes exceed the bound %u", n, kmax);
    if (n > first) {
        h.resize(2 * (size_t)n + 2);
        HIP_TRY(hipMemcpyAsync(h.data() + 2 + 2 * first, dpairs + 2 * first, sizeof(uint64_t) * 2 * (n - first),
                               hipMemcpyDeviceToHost, stream));
        HIP_TRY(hipStreamSynchronize(stream));
    }
    float t = 0;
    (void)hipEventElapsedTime(&t, events[0], events[1]);
    if (ms) *ms = t;
    std::vector<std::pair<uint64_t, uint64_t>> v(n);
    for (uint32_t i = 0; i < n; i++) v[i] = {h[2 * i + 2], h[2 * i + 3]};
    std::sort(v.begin(), v.end());
    for (uint32_t i = 0; i < n && i < cap; i++) {
        pairs[2 * i] = v[i].first;
        pairs[2 * i + 1] = v[i].second;
    }
    *npairs = n;
    return SCC_OK;
}

// --------------------------------------------------- phase entries ---

scc_status Engine::phase_begin(const uint8_t *dead)
{
    if (!has_graph) return fail(SCC_ERR_NOTREADY, "no graph uploaded");
    HIP_TRY(hipSetDevice(device));
    ran = false;
    phase_marks = true;   // the phase entry points time their phase
    deg_known = low_denied = false;
    if (dead) HIP_TRY(hipMemcpyAsync(d_tmp8, dead, (size_t)g.V + 1, hipMemcpyHostToDevice, stream));
    k_first_arcs(stream, g);
    k_init_state(stream, g, st, dead ? d_tmp8 : nullptr);   // also zeroes the counters
    return SCC_OK;
}

scc_status Engine::fetch8(uint8_t *out)
{
    HIP_TRY(hipMemcpyAsync(out, d_tmp8, (size_t)g.V + 1, hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return SCC_OK;
}

scc_status Engine::fetch32(uint32_t *out, const uint32_t *src)
{
    HIP_TRY(hipMemcpyAsync(out, src, sizeof(uint32_t) * ((size_t)g.V + 1), hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return SCC_OK;
}

scc_status Engine::phase_local(uint32_t *out)
{
    if (!has_part) return fail(SCC_ERR_NOTREADY, "no partition uploaded");
    scc_status s;
    if ((s = phase_begin(nullptr)) != SCC_OK) return s;
    nmarks = 0;
    scc_opts o;
    scc_opts_default(&o);
    // trim-2 would finish a 2-cycle whose ends lie in different partitions as
    // one pair: a global SCC but two local ones.  Trim-1 removes only
    // vertices that are singletons locally as well.
    o.trim2 = 0;
    scc_stats tmp;
    std::memset(&tmp, 0, sizeof tmp);
    if ((s = detect_phases(o, SCC_EXPAND_DO, 1, &tmp, true)) != SCC_OK) return s;
    if ((s = fetch32(out, st.lab)) != SCC_OK) return s;
    out[0] = 0;
    return SCC_OK;
}

scc_status Engine::phase_trim1(const uint8_t *dead, uint8_t *removed)
{
    scc_status s;
    if ((s = phase_begin(dead)) != SCC_OK) return s;
    nmarks = 0;
    if ((s = trim1(true, true, dead == nullptr)) != SCC_OK) return s;
    k_export_removed(stream, g, st, d_tmp8);
    if ((s = fetch8(removed)) != SCC_OK) return s;
    if (dead)
        for (uint32_t v = 0; v <= g.V; v++) removed[v] = removed[v] && !dead[v];
    return SCC_OK;
}

scc_status Engine::phase_trim2(const uint8_t *dead, uint32_t *pair)
{
    scc_status s;
    if ((s = phase_begin(dead)) != SCC_OK) return s;
    k_trim2(stream, g, st);
    std::vector<uint32_t> cls((size_t)g.V + 1);
    if ((s = fetch32(cls.data(), st.cls)) != SCC_OK) return s;
    if ((s = fetch32(pair, st.lab)) != SCC_OK) return s;
    for (uint32_t v = 0; v <= g.V; v++)
        pair[v] = (v == 0 || cls[v] != DEAD || (dead && dead[v])) ? 0u : (pair[v] & ~LAB_FINAL);
    return SCC_OK;
}

scc_status Engine::phase_first_pivot(const uint8_t *dead, uint32_t *pivot)
{
    scc_status s;
    if ((s = phase_begin(dead)) != SCC_OK) return s;
    init_vis(true);
    if ((s = read_ctr()) != SCC_OK) return s;
    *pivot = 0;
    if (h_ctr[CT(C_NPIV)] > 1) return fail(SCC_ERR_DEVICE, "first-pivot election chose %u vertices", h_ctr[CT(C_NPIV)]);
    if (h_ctr[CT(C_NPIV)] == 1) {
        HIP_TRY(hipMemcpyAsync(pivot, st.pivlist, sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
        HIP_TRY(hipStreamSynchronize(stream));
    }
    return SCC_OK;
}

scc_status Engine::phase_reach(uint32_t src, int dir, int expand, int W, const uint8_t *dead,
                               uint8_t *out, uint32_t *levels, double *ms)
{
    if (!has_graph) return fail(SCC_ERR_NOTREADY, "no graph uploaded");
    if (src < 1 || src > g.V) return fail(SCC_ERR_INVALID, "source %u outside [1, %u]", src, g.V);
    if (dead && dead[src]) return fail(SCC_ERR_INVALID, "source %u is marked dead", src);
    if (expand == SCC_EXPAND_AUTO) expand = SCC_EXPAND_VERTEX;
    if (expand < SCC_EXPAND_VERTEX || expand > SCC_EXPAND_DO)
        return fail(SCC_ERR_INVALID, "unknown expand mode %d", expand);
    if (W != 1 && W != 2 && W != 4 && W != 8 && W != 16 && W != 32 && W != 64)
        return fail(SCC_ERR_INVALID, "warp size %d not in {1,2,4,8,16,32,64}", W);
    scc_status s;
    if ((s = phase_begin(dead)) != SCC_OK) return s;
    init_vis();
    k_seed_single(stream, st, src, dir);
    nmarks = 0;
    mark(SCC_PHASE_REACH);
    uint32_t lv = 0;
    if ((s = reach(dir == 0, dir != 0, true, expand, W, &lv)) != SCC_OK) return s;
    mark(-1);
    scc_stats tmp;
    collect_times(&tmp);
    if (ms) *ms = tmp.ms_scc;
    if (levels) *levels = lv;
    k_export_visited(stream, g, st, dir, d_tmp8);
    return fetch8(out);
}

scc_status Engine::phase_min_label(const uint8_t *dead, uint32_t *out)
{
    scc_status s;
    if ((s = phase_begin(dead)) != SCC_OK) return s;
    k_minlabel_init(stream, g, st);
    uint64_t it = 0;
    do {
        if (it) zero_ctr(C_CHANGED, 1);
        k_minlabel_prop(stream, g, st);
        if ((s = read_ctr()) != SCC_OK) return s;
        if (++it > limit()) return no_convergence("min-label propagation");
    } while (h_ctr[CT(C_CHANGED)]);
    if ((s = fetch32(out, st.cls)) != SCC_OK) return s;
    for (uint32_t v = 0; v <= g.V; v++)
        if (out[v] == DEAD || v == 0) out[v] = 0;
    return SCC_OK;
}

scc_status Engine::phase_max_color(const uint8_t *dead, uint32_t *out)
{
    scc_status s;
    if ((s = phase_begin(dead)) != SCC_OK) return s;
    k_color_init(stream, g, st);
    uint64_t it = 0;
    do {
        if (it) zero_ctr(C_CHANGED, 1);
        k_color_prop(stream, g, st);
        if ((s = read_ctr()) != SCC_OK) return s;
        if (++it > limit()) return no_convergence("colour propagation");
    } while (h_ctr[CT(C_CHANGED)]);
    return fetch32(out, st.aux);
}

} // namespace sccamd
