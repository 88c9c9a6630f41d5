// kernels_batch.hip -- many independent graphs in one persistent launch.
//
// The reference runs one graph per process with a host round trip after
// every kernel (scc_WCC.cu:683-686).  Here each workgroup pops a graph index
// from a device work queue (largest graphs first) and runs the whole SCC
// pipeline for that graph on its own, with workgroup barriers between the
// phases and every queue count and fixpoint flag in LDS.  Nothing goes back
// to the host until the batch is done.
//
// Phase orders are the reference's: vHong (scc_WCC.cu:573-998) and vSlota
// (scc_Coloring.cu:403-701).  The first round (trim-1, the first pivot's FW
// and BW search) has one class only and runs on bitmaps; a graph that it
// finishes gets its labels from them.  Otherwise the vertices it left are
// listed, and the later phases run over that list.  Per graph the
// configuration word selects the algorithm and the trims (with the workgroup
// size chosen by the autotuner per size and degree bucket).
//
// What bounds it: one graph's chain of dependent loads (a workgroup waits
// for some hundreds of them one after another) and, for the large graphs of
// a batch, HBM (6.5 GB for the 4.4 GB of the 4,096-graph mix).  Hence:
// several chunks' loads in flight per lane (four 64-vertex chunks and all
// their list walks side by side: 2.45 -> 1.95 ms on the mix, although its
// registers leave one 1,024-lane workgroup per CU instead of two), the two
// directions of a search on two halves of the waves, a frontier's arcs
// balanced over its wave, hubs over the workgroup, bottom-up levels where
// the degree pays for them, no gather of first neighbours where trim-1 would
// remove little, and nothing run for vertices that are finished.  The mix
// (47.6M vertices, 434M arcs, 1,024 lanes) 11.1 -> 1.8 ms; 700 graphs of 2^8
// to 2^12 vertices with 256 lanes 1.31 -> 0.17 ms.
//
// Layout: graph i's per-vertex arrays start at slot voff[i] (a multiple of
// 64, so bitmap words never straddle two graphs) and span V_i+2 slots; its
// column arrays start at eoff[i]; its pivot table spans 3*(V_i+2) keys from
// 3*voff[i].  Vertex ids inside a graph are local (1..V_i).
#include "batch.h"

namespace sccamd {

// cfg word: bit 0 trim-1, bit 1 trim-2, bit 2 Slota (colouring) instead of Hong
__host__ __device__ inline bool cfg_t1(uint32_t c) { return c & 1u; }
__host__ __device__ inline bool cfg_t2(uint32_t c) { return (c >> 1) & 1u; }
__host__ __device__ inline bool cfg_slota(uint32_t c) { return (c >> 2) & 1u; }

namespace {

__device__ __forceinline__ uint32_t ln() { return threadIdx.x & 63u; }

// A value every lane holds alike (read from LDS, say), as a scalar: the
// views' pointers and the loop bounds then live in scalar registers.
__device__ __forceinline__ uint32_t uni(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }

__device__ __forceinline__ uint64_t bkey_deg(uint32_t outdeg, uint32_t indeg, uint32_t v)
{
    uint64_t p = (uint64_t)outdeg * (uint64_t)indeg;
    p = p > 0xFFFFFFFFull ? 0xFFFFFFFFull : p;
    return (p << 32) | (uint64_t)(0xFFFFFFFFu - v);
}

__device__ __forceinline__ uint64_t bkey(const uint32_t *Fr, const uint32_t *Br, uint32_t v)
{
    return bkey_deg(Fr[v + 1] - Fr[v], Br[v + 1] - Br[v], v);
}

__device__ __forceinline__ uint32_t bkey_vertex(uint64_t k) { return 0xFFFFFFFFu - (uint32_t)k; }

__device__ __forceinline__ bool bbit(const uint32_t *bm, uint32_t v) { return (bm[v >> 5] >> (v & 31)) & 1u; }

// A frontier vertex of at least HUB_DEG arcs is walked by the whole
// workgroup (one lane group alone would walk the pivot of a power-law graph
// for hundreds of steps); up to HUB_CAP of them per level.
constexpr uint32_t HUB_DEG = 512;
constexpr uint32_t HUB_CAP = 128;

// Levels of at most 64 frontier vertices and NARROW_ARCS arcs are run by one
// wave per direction, without workgroup barriers and with the frontier in
// LDS (g_narrow).
constexpr uint32_t NARROW_ARCS = 256;

// what a graph's run counted (scc_stats has the meanings)
struct GraphStats {
    uint32_t trim1, trim2, pivots, first_pivot, rounds, levels;
    uint64_t search_ticks;   // the first search, wall clock
};

// per-workgroup scratch in LDS
struct Lds {
    uint32_t graph;
    uint32_t tail[2];         // entries in the FW and BW queues
    uint32_t npiv;
    uint32_t nact;            // listed vertices
    uint32_t nhub;
    uint32_t anom;            // a class without a recorded pivot was seen
    uint32_t red[2][16];
    unsigned long long key;
    uint32_t hub[HUB_CAP];    // vertex | direction << 31
    uint32_t near[2][NARROW_ARCS];   // per direction, the frontier of a narrow level
    uint32_t nlo[2];          // where the frontier begins in the queue after the narrow levels
    uint32_t nlev[2];         // and how many there were
    GraphStats st;            // written by thread 0
};

// one graph's views
struct G1 {
    uint32_t V;
    uint32_t E;
    const uint32_t *Fr, *Fc, *Br, *Bc;
    uint32_t *cls, *lab, *aux;
    uint32_t *live, *fvis, *bvis;   // one bit per vertex
    uint32_t *seen;                 // two such bitmaps (g_trim_listed), one after the other
    uint64_t *piv;
    // four arrays of V+2 words: 0 and 2 are the FW and BW queues (each
    // vertex enters a search's queue once, so a queue is never reused within
    // a search), 1 holds the first out-neighbours and then (batch) the list
    // of the vertices the first round left, 3 the live bitmap of a graph too
    // large for LDS
    uint32_t *q;
    __device__ __forceinline__ uint32_t *queue(uint32_t k) const { return q + (size_t)k * (V + 2); }
    __device__ __forceinline__ uint32_t *f1() const { return queue(1); }
    __device__ __forceinline__ uint32_t *b1() const { return aux; }   // first in-neighbours (first round only)
    uint32_t *list;   // the vertices the first round left, V+2 words
    uint32_t *pivlist;
};

// Workgroup sum; L.red is double-buffered by `k`, so consecutive sums with
// alternating k need one barrier each.
template <int BS> __device__ __forceinline__ uint32_t wg_sum(Lds &L, uint32_t x, uint32_t k)
{
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
    if (ln() == 0) L.red[k][threadIdx.x >> 6] = x;
    __syncthreads();
    uint32_t t = 0;
    for (int w = 0; w < BS / 64; w++) t += L.red[k][w];
    return uni(t);
}

template <int BS> __device__ __forceinline__ uint32_t wg_sum1(Lds &L, uint32_t x)
{
    __syncthreads();
    const uint32_t t = wg_sum<BS>(L, x, 0);
    __syncthreads();
    return t;
}

template <int BS> __device__ __forceinline__ uint32_t wg_min1(Lds &L, uint32_t x)
{
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t y = __shfl_xor(x, o);
        x = y < x ? y : x;
    }
    __syncthreads();
    if (ln() == 0) L.red[0][threadIdx.x >> 6] = x;
    __syncthreads();
    uint32_t t = DEAD;
    for (int w = 0; w < BS / 64; w++) t = L.red[0][w] < t ? L.red[0][w] : t;
    __syncthreads();
    return uni(t);
}

// a[i] for a per-vertex array (i < 2^30, so the byte offset fits 32 bits and
// the address is a scalar base and one vector register)
__device__ __forceinline__ uint32_t at(const uint32_t *a, uint32_t i)
{
    return *reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(a) + (uint32_t)(i << 2));
}

__device__ __forceinline__ void put(uint32_t *a, uint32_t i, uint32_t x)
{
    *reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(a) + (uint32_t)(i << 2)) = x;
}

// LDS-counter push (wave-aggregated over the active lanes)
__device__ __forceinline__ void lpush(bool p, uint32_t v, uint32_t *q, uint32_t *cnt)
{
    const uint64_t act = __ballot(1);
    const uint64_t m = __ballot(p);
    if (!m) return;
    const int leader = __ffsll((unsigned long long)act) - 1;
    uint32_t b = 0;
    if ((int)ln() == leader) b = atomicAdd(cnt, (uint32_t)__popcll(m));
    b = __shfl(b, leader);
    if (p) put(q, b + (uint32_t)__popcll(m & ((1ull << ln()) - 1)), v);
}

// Per-vertex list walks: a step loads GK columns and then issues every
// probe of the step before using any (indexes past the end repeat the last
// arc, which changes no minimum, maximum or existence test).  A walk of
// one arc per step waits for two dependent loads per arc.
constexpr uint32_t GK = 2;

// For each of a lane's K lists, a vertex of C[k][i[k]..e[k]) whose bit is set
// in bm, 0 if none (i == e: nothing to look up; all 64 lanes of the wave
// call).  The lane's lists are walked side by side, GK arcs of each in
// flight, for ROW_LANE arcs; what is left of longer lists the wave walks
// together, one list after the other: a lane alone took milliseconds for a
// power-law graph's hub whose neighbours are nearly all unset, and its graph
// finished last by as much.
constexpr uint32_t ROW_LANE = 32;

template <uint32_t K>
__device__ __forceinline__ void g_any_bit(const uint32_t *const (&C)[K], uint32_t (&i)[K], const uint32_t (&e)[K],
                                          const uint32_t *bm, uint32_t (&hit)[K])
{
    uint32_t own[K];
    bool any = false;
#pragma unroll
    for (uint32_t k = 0; k < K; k++) {
        hit[k] = 0;
        own[k] = min(e[k], i[k] + ROW_LANE);
        any |= i[k] < e[k];
    }
    while (any) {
        uint32_t w[K][GK];
#pragma unroll
        for (uint32_t k = 0; k < K; k++) {
#pragma unroll
            for (uint32_t n = 0; n < GK; n++) w[k][n] = 0;   // the dummy: never set
            if (!hit[k] && i[k] < own[k]) {
#pragma unroll
                for (uint32_t n = 0; n < GK; n++) w[k][n] = C[k][min(i[k] + n, e[k] - 1)];
            }
        }
        any = false;
#pragma unroll
        for (uint32_t k = 0; k < K; k++) {
#pragma unroll
            for (uint32_t n = 0; n < GK; n++)
                if (!hit[k] && bbit(bm, w[k][n])) hit[k] = w[k][n];
            i[k] = hit[k] ? own[k] : min(i[k] + GK, own[k]);
            any |= i[k] < own[k];
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < K; k++) {
        uint64_t todo = __ballot(!hit[k] && i[k] < e[k]);
        while (todo) {
            const int l = __ffsll((unsigned long long)todo) - 1;
            todo &= todo - 1;
            const uint32_t end = (uint32_t)__builtin_amdgcn_readlane((int)e[k], l);
            uint32_t found = 0;
            for (uint32_t j = (uint32_t)__builtin_amdgcn_readlane((int)i[k], l); !found && j < end; j += 128) {
                const uint32_t w0 = C[k][min(j + ln(), end - 1)], w1 = C[k][min(j + 64 + ln(), end - 1)];
                const uint32_t w = bbit(bm, w0) ? w0 : bbit(bm, w1) ? w1 : 0u;
                const uint64_t m = __ballot(w != 0);
                if (m) found = (uint32_t)__builtin_amdgcn_readlane((int)w, __ffsll((unsigned long long)m) - 1);
            }
            if ((int)ln() == l) hit[k] = found;
        }
    }
}

// Whether some arc of C[i..e) leads to a vertex of class c (all 64 lanes of
// the wave call).  As in g_any_bit the wave takes what is left of a long row
// together: with a lane alone on it, 4,096 vertices with one of 3,900
// out-arcs took 42.4 ms by colouring (now 2.3) and, where trim-1 peels a long
// path in front of such a row, 196 ms (now 21).
__device__ __forceinline__ bool g_any_cls(const uint32_t *C, uint32_t i, uint32_t e, const uint32_t *cls,
                                          uint32_t c)
{
    bool hit = false;
    const uint32_t own = min(e, i + ROW_LANE);
    for (; !hit && i < own; i += GK) {
        uint32_t w[GK];
#pragma unroll
        for (uint32_t k = 0; k < GK; k++) w[k] = C[min(i + k, e - 1)];
#pragma unroll
        for (uint32_t k = 0; k < GK; k++) hit |= cls[w[k]] == c;
    }
    uint64_t todo = __ballot(!hit && i < e);
    while (todo) {
        const int l = __ffsll((unsigned long long)todo) - 1;
        todo &= todo - 1;
        const uint32_t end = (uint32_t)__builtin_amdgcn_readlane((int)e, l);
        const uint32_t cl = (uint32_t)__builtin_amdgcn_readlane((int)c, l);
        bool found = false;
        for (uint32_t j = (uint32_t)__builtin_amdgcn_readlane((int)i, l); !found && j < end; j += 128) {
            const uint32_t w0 = C[min(j + ln(), end - 1)], w1 = C[min(j + 64 + ln(), end - 1)];
            found = __any(cls[w0] == cl || cls[w1] == cl);
        }
        if ((int)ln() == l) hit = found;
    }
    return hit;
}

// m combined with a[w] over the arcs C[i..e): the largest (MAX) or the
// smallest; long rows as in g_any_cls
template <bool MAX> __device__ __forceinline__ uint32_t g_pick(uint32_t m, uint32_t x)
{
    return MAX ? (x > m ? x : m) : (x < m ? x : m);
}

template <bool MAX>
__device__ __forceinline__ uint32_t g_fold(const uint32_t *C, uint32_t i, uint32_t e, const uint32_t *a, uint32_t m)
{
    const uint32_t own = min(e, i + ROW_LANE);
    for (; i < own; i += GK) {
        uint32_t w[GK];
#pragma unroll
        for (uint32_t k = 0; k < GK; k++) w[k] = C[min(i + k, e - 1)];
#pragma unroll
        for (uint32_t k = 0; k < GK; k++) m = g_pick<MAX>(m, a[w[k]]);
    }
    uint64_t todo = __ballot(i < e);
    while (todo) {
        const int l = __ffsll((unsigned long long)todo) - 1;
        todo &= todo - 1;
        const uint32_t end = (uint32_t)__builtin_amdgcn_readlane((int)e, l);
        uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)m, l);
        for (uint32_t j = (uint32_t)__builtin_amdgcn_readlane((int)i, l); j < end; j += 128) {
            const uint32_t w0 = C[min(j + ln(), end - 1)], w1 = C[min(j + 64 + ln(), end - 1)];
            x = g_pick<MAX>(g_pick<MAX>(x, a[w0]), a[w1]);
        }
        for (int o = 32; o > 0; o >>= 1) x = g_pick<MAX>(x, (uint32_t)__shfl_xor((int)x, o));
        if ((int)ln() == l) m = x;
    }
    return m;
}

// ------------------------------------------------- the first round ---
// A wave owns the 64-vertex chunks w, w + BS/64, ... and with them the two
// words of each bitmap, which it writes with plain stores.

// Degrees: the live bitmap (vertices with an in- and an out-arc; all of them
// with the trims off) and the best pivot key among them, which goes to
// L.key.  Returns the number of vertices that are not live.
constexpr uint32_t DEG_CHUNKS = 4;

template <int BS> __device__ __forceinline__ uint32_t g_degrees(Lds &L, const G1 &g, bool trim)
{
    const uint32_t nch = (g.V + 64) / 64;
    unsigned long long best = 0;
    uint32_t gone = 0;
    for (uint32_t c0 = uni(threadIdx.x >> 6); c0 < nch; c0 += DEG_CHUNKS * (BS / 64)) {
        uint32_t fb[DEG_CHUNKS], fe[DEG_CHUNKS], bb[DEG_CHUNKS], be[DEG_CHUNKS];
#pragma unroll
        for (uint32_t h = 0; h < DEG_CHUNKS; h++) {
            const uint32_t v = (c0 + h * (BS / 64)) * 64 + ln(), vv = v <= g.V ? v : 0u;   // row 0 is empty
            fb[h] = at(g.Fr, vv);
            fe[h] = at(g.Fr, vv + 1);
            bb[h] = at(g.Br, vv);
            be[h] = at(g.Br, vv + 1);
        }
#pragma unroll
        for (uint32_t h = 0; h < DEG_CHUNKS; h++) {
            const uint32_t ch = c0 + h * (BS / 64), v = ch * 64 + ln();
            const bool in = v >= 1 && v <= g.V;
            const bool alive = in && (!trim || (fe[h] > fb[h] && be[h] > bb[h]));
            gone += in && !alive;
            const uint64_t m = __ballot(alive);
            if (ch < nch && ln() < 2) g.live[2 * ch + ln()] = ln() ? (uint32_t)(m >> 32) : (uint32_t)m;
            if (alive) {
                const unsigned long long k = bkey_deg(fe[h] - fb[h], be[h] - bb[h], v);
                best = k > best ? k : best;
            }
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long x = __shfl_xor(best, o);
        best = x > best ? x : best;
    }
    if (ln() == 0 && best) atomicMax(&L.key, best);
    return wg_sum1<BS>(L, gone);
}

// trim-1 (scc_kernels.cu:187-233) on the live bitmap.  A vertex tests its
// first in- and out-neighbour (pass 0 gathers them); where one is gone it
// walks the list and keeps the live neighbour it finds as its first one,
// which the next pass and the bottom-up levels then test.  A pass reads
// every live vertex's first neighbours, so it stops when a pass removes less
// than 1/TRIM_STOP of the vertices: what a fixpoint would still remove (the
// long chains of a sparse graph, a few vertices per pass for dozens of
// passes) is left to the list phases, whose passes read the listed vertices
// only (stopping at 1/128 instead of 1/32 of the vertices, and not at all,
// made the mix's sparsest graphs its last to end).  A graph of which the
// degrees alone removed less than 1/TRIM_MIN is not trimmed here at all: the
// gather of its first neighbours, one line of columns per vertex and
// direction, costs more than what it would remove (mix 3.05 -> 2.69 ms).
constexpr uint32_t TRIM_CHUNKS = 4;
constexpr uint32_t TRIM_STOP = 32;
// LISTED: queue 0 lists what the last pass removed, for g_trim_listed.
constexpr uint32_t TRIM_MIN = 8;

template <int BS, bool LISTED> __device__ __forceinline__ void g_trim_bits(Lds &L, const G1 &g)
{
    const uint32_t nch = (g.V + 64) / 64;
    uint32_t *F1 = g.f1(), *B1 = g.b1();
    for (uint32_t pass = 0; pass <= g.V; pass++) {   // each pass removes a vertex or ends
        if (LISTED) {
            __syncthreads();
            if (threadIdx.x == 0) L.tail[0] = 0;
            __syncthreads();
        }
        uint32_t removed = 0;                        // wave-uniform
        for (uint32_t c0 = uni(threadIdx.x >> 6); c0 < nch; c0 += TRIM_CHUNKS * (BS / 64)) {
            uint32_t word[TRIM_CHUNKS], pin[TRIM_CHUNKS], pout[TRIM_CHUNKS];
            bool any = false;
#pragma unroll
            for (uint32_t h = 0; h < TRIM_CHUNKS; h++) {
                const uint32_t ch = c0 + h * (BS / 64);
                word[h] = ch < nch ? g.live[2 * ch + (ln() >> 5)] : 0u;
                any |= word[h] != 0;
            }
            if (!__ballot(any)) continue;
            if (pass == 0) {
                uint32_t fb[TRIM_CHUNKS], bb[TRIM_CHUNKS];
#pragma unroll
                for (uint32_t h = 0; h < TRIM_CHUNKS; h++) {
                    const uint32_t v = (c0 + h * (BS / 64)) * 64 + ln(), vv = v <= g.V ? v : 0u;
                    fb[h] = at(g.Fr, vv);
                    bb[h] = at(g.Br, vv);
                }
#pragma unroll
                for (uint32_t h = 0; h < TRIM_CHUNKS; h++) {
                    pin[h] = pout[h] = 0;
                    if ((word[h] >> (ln() & 31)) & 1u) {   // live: both lists have an arc
                        pin[h] = g.Bc[bb[h]];
                        pout[h] = g.Fc[fb[h]];
                    }
                }
#pragma unroll
                for (uint32_t h = 0; h < TRIM_CHUNKS; h++) {
                    const uint32_t v = (c0 + h * (BS / 64)) * 64 + ln();
                    if ((word[h] >> (ln() & 31)) & 1u) {
                        put(B1, v, pin[h]);
                        put(F1, v, pout[h]);
                    }
                }
            } else {
#pragma unroll
                for (uint32_t h = 0; h < TRIM_CHUNKS; h++) {
                    const uint32_t v = (c0 + h * (BS / 64)) * 64 + ln(), vv = v <= g.V ? v : 0u;
                    pin[h] = at(B1, vv);
                    pout[h] = at(F1, vv);
                }
            }
            // lists 2h and 2h + 1: chunk h's in- and out-list, where the first
            // neighbour is gone (a vertex that is not live has no entry in B1
            // and F1)
            const uint32_t *C[2 * TRIM_CHUNKS];
            uint32_t i[2 * TRIM_CHUNKS], e[2 * TRIM_CHUNKS], x[2 * TRIM_CHUNKS];
            bool walk = false;
#pragma unroll
            for (uint32_t h = 0; h < TRIM_CHUNKS; h++) {
                const bool alive = (word[h] >> (ln() & 31)) & 1u;
                C[2 * h] = g.Bc;
                C[2 * h + 1] = g.Fc;
                x[2 * h] = !alive || bbit(g.live, pin[h]);
                x[2 * h + 1] = !alive || bbit(g.live, pout[h]);
                walk |= !x[2 * h] || !x[2 * h + 1];
            }
            if (__ballot(walk)) {
#pragma unroll
                for (uint32_t h = 0; h < TRIM_CHUNKS; h++) {
                    const uint32_t v = (c0 + h * (BS / 64)) * 64 + ln();
                    const uint32_t ri = x[2 * h] ? 0u : v, ro = x[2 * h + 1] ? 0u : v;   // row 0 is empty
                    i[2 * h] = at(g.Br, ri);
                    e[2 * h] = at(g.Br, ri + 1);
                    i[2 * h + 1] = at(g.Fr, ro);
                    e[2 * h + 1] = at(g.Fr, ro + 1);
                }
                uint32_t y[2 * TRIM_CHUNKS];
                g_any_bit<2 * TRIM_CHUNKS>(C, i, e, g.live, y);
#pragma unroll
                for (uint32_t h = 0; h < TRIM_CHUNKS; h++) {
                    const uint32_t v = (c0 + h * (BS / 64)) * 64 + ln();
                    if (y[2 * h]) put(B1, v, y[2 * h]);
                    if (y[2 * h + 1]) put(F1, v, y[2 * h + 1]);
                    x[2 * h] |= y[2 * h];
                    x[2 * h + 1] |= y[2 * h + 1];
                }
#pragma unroll
                for (uint32_t h = 0; h < TRIM_CHUNKS; h++) {
                    const uint32_t ch = c0 + h * (BS / 64);
                    const bool out = !x[2 * h] || !x[2 * h + 1];
                    const uint64_t m = __ballot(out);
                    if (LISTED) lpush(out, ch * 64 + ln(), g.queue(0), &L.tail[0]);
                    const uint32_t mw = ln() < 32 ? (uint32_t)m : (uint32_t)(m >> 32);
                    if ((ln() & 31) == 0 && mw) g.live[2 * ch + (ln() >> 5)] = word[h] & ~mw;
                    removed += (uint32_t)__popcll(m);
                }
            }
        }
        if ((uint64_t)wg_sum<BS>(L, ln() == 0 ? removed : 0u, pass & 1) * TRIM_STOP <= g.V) break;
    }
    __syncthreads();
}

// no vertex visited (finished ones are told apart by their class)
template <int BS> __device__ __forceinline__ void g_clear_vis(const G1 &g)
{
    const uint32_t nw = 2 * ((g.V + 64) / 64);
    for (uint32_t i = threadIdx.x; i < nw; i += BS) {
        g.fvis[i] = 0;
        g.bvis[i] = 0;
    }
}

// A live neighbour w (0: none) that lost an out-arc (d = 1) or in-arc (d = 0)
// goes too, and is listed in queue 0, unless another live arc that way is
// left.  The first lane to mark w in `seen` looks: whatever else w lost, it
// lost before this pass.  (Without the marks every one of a thousand parallel
// arcs walked the row.)  All 64 lanes of the wave call.
__device__ __forceinline__ void g_recheck(Lds &L, const G1 &g, uint32_t d, uint32_t w, uint32_t *seen)
{
    const uint32_t *R = d ? g.Fr : g.Br, *const C[1] = {d ? g.Fc : g.Bc};
    const uint32_t bit = 1u << (w & 31);
    const bool look = bbit(g.live, w) && !bbit(seen, w) && !(atomicOr(&seen[w >> 5], bit) & bit);
    if (!__ballot(look)) return;
    const uint32_t r = look ? w : 0u;   // row 0 is empty
    uint32_t i[1] = {at(R, r)}, x[1];
    const uint32_t e[1] = {at(R, r + 1)};
    g_any_bit<1>(C, i, e, g.live, x);
    const bool gone = look && !x[0] && (atomicAnd(&g.live[w >> 5], ~bit) & bit);
    lpush(gone, w, g.queue(0), &L.tail[0]);
}

// Every vertex that is not live and has arcs, in queue 0.
template <int BS> __device__ __forceinline__ void g_list_gone(Lds &L, const G1 &g)
{
    __syncthreads();
    if (threadIdx.x == 0) L.tail[0] = 0;
    __syncthreads();
    for (uint32_t v = threadIdx.x; v <= g.V; v += BS)
        lpush(!bbit(g.live, v) && (at(g.Fr, v + 1) > at(g.Fr, v) || at(g.Br, v + 1) > at(g.Br, v)), v, g.queue(0),
              &L.tail[0]);
}

// trim-1 on to its fixpoint, from the removed vertices in queue 0 that no
// pass has followed up yet.  The arcs of many vertices are balanced over
// their wave, as in g_expand; few vertices get several waves each.
template <int BS> __device__ __forceinline__ void g_trim_listed(Lds &L, const G1 &g)
{
    const uint32_t *q = g.queue(0);
    const uint32_t wv = uni(threadIdx.x >> 6), nwv = BS / 64, d = wv & 1, w = wv >> 1, nw = nwv / 2;
    const uint32_t *R = d ? g.Br : g.Fr, *C = d ? g.Bc : g.Fc;
    const uint32_t nb = 2 * ((g.V + 64) / 64);
    uint32_t *seen = g.seen + d * nb;
    __syncthreads();
    for (uint32_t lo = 0, hi = uni(L.tail[0]); lo != hi;) {   // each pass but the last lists a vertex
        for (uint32_t i = threadIdx.x; i < 2 * nb; i += BS) g.seen[i] = 0;
        __syncthreads();   // and every lane has read the tail
        const uint32_t n = hi - lo;
        if (n < nw) {
            const uint32_t each = nw / n;   // waves per vertex and side
            if (w / each < n) {
                const uint32_t u = at(q, lo + w / each);
                for (uint32_t j = at(R, u) + 64 * (w % each), end = at(R, u + 1); j < end; j += 64 * each)
                    g_recheck(L, g, d, j + ln() < end ? C[j + ln()] : 0u, seen);
            }
        } else {
            const uint32_t per = min(64u, (n + nw - 1) / nw);
            for (uint32_t t = lo + per * w; t < hi; t += per * nw) {
                const uint32_t u = ln() < per && t + ln() < hi ? at(q, t + ln()) : 0u;   // row 0 is empty
                const uint32_t b = at(R, u), deg = at(R, u + 1) - b;
                uint32_t sum = deg;   // inclusive
                for (int o = 1; o < 64; o <<= 1) {
                    const uint32_t y = __shfl_up(sum, o);
                    if ((int)ln() >= o) sum += y;
                }
                const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)sum, 63);
                const uint32_t start = b - (sum - deg);   // arc j of the tile is C[start + j], modulo 2^32
                for (uint32_t j0 = 0; j0 < total; j0 += 64) {
                    const uint32_t j = j0 + ln();
                    uint32_t own = 0;
#pragma unroll
                    for (uint32_t o = 32; o >= 1; o >>= 1)
                        own += (uint32_t)__shfl((int)sum, (int)(own + o - 1)) <= j ? o : 0u;
                    const uint32_t st = __shfl(start, (int)own);   // past the end `own` is 63, and the load is skipped
                    g_recheck(L, g, d, j < total ? C[st + j] : 0u, seen);
                }
            }
        }
        __syncthreads();
        lo = hi;
        hi = uni(L.tail[0]);
    }
    __syncthreads();
}

// The arcs of frontier entries [lo, hi) of direction d's queue.  SINGLE: every live vertex is in one class, a neighbour is taken
// if it is live and not visited; otherwise if it is in the vertex's class
// (a finished vertex is in none) and not visited.
template <bool SINGLE>
__device__ __forceinline__ bool g_claim(const G1 &g, uint32_t *vis, uint32_t w, uint32_t c)
{
    const uint32_t bit = 1u << (w & 31);
    const uint32_t word = vis[w >> 5];
    const bool ok = SINGLE ? (g.live[w >> 5] & ~word & bit) != 0 : (!(word & bit) && g.cls[w] == c);
    return ok && !(atomicOr(&vis[w >> 5], bit) & bit);
}

// A wave takes up to 64 frontier vertices, scans their degrees and walks
// their arcs one after the other with all lanes (consecutive lanes read
// consecutive columns, EXP_UNR steps in flight), whatever the degree mix: an
// arc's vertex is the first lane whose running degree sum exceeds the arc's
// index, found with six shuffles.  w of nw: this wave among the waves that
// work on this direction.
constexpr uint32_t EXP_UNR = 2;

template <bool SINGLE>
__device__ __forceinline__ void g_expand(Lds &L, const G1 &g, uint32_t d, uint32_t lo, uint32_t hi, uint32_t w,
                                         uint32_t nw)
{
    const uint32_t *R = d ? g.Br : g.Fr, *C = d ? g.Bc : g.Fc;
    uint32_t *vis = d ? g.bvis : g.fvis, *q = g.queue(2 * d);
    const uint32_t per = min(64u, (hi - lo + nw - 1) / nw);   // vertices per wave and step
    for (uint32_t t = lo + per * w; t < hi; t += per * nw) {
        const uint32_t v = ln() < per && t + ln() < hi ? at(q, t + ln()) : 0u;   // row 0 is empty
        const uint32_t b = at(R, v);
        uint32_t n = at(R, v + 1) - b;
        const uint32_t c = SINGLE ? 0u : g.cls[v];
        if (n >= HUB_DEG) {
            const uint32_t k = atomicAdd(&L.nhub, 1u);
            if (k < HUB_CAP) {
                L.hub[k] = v | (d << 31);
                n = 0;
            }
        }
        uint32_t sum = n;   // inclusive
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(sum, o);
            if ((int)ln() >= o) sum += y;
        }
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)sum, 63);
        const uint32_t start = b - (sum - n);   // arc j of the tile is C[start + j], modulo 2^32
        for (uint32_t j0 = 0; j0 < total; j0 += 64 * EXP_UNR) {
            uint32_t x[EXP_UNR], cx[EXP_UNR];
            bool ok[EXP_UNR];
#pragma unroll
            for (uint32_t u = 0; u < EXP_UNR; u++) {
                const uint32_t j = j0 + u * 64 + ln();
                uint32_t own = 0;
#pragma unroll
                for (uint32_t o = 32; o >= 1; o >>= 1)
                    own += (uint32_t)__shfl((int)sum, (int)(own + o - 1)) <= j ? o : 0u;
                // past the end `own` is 63, and the load is skipped
                const uint32_t st = __shfl(start, (int)own);
                cx[u] = SINGLE ? 0u : __shfl(c, (int)own);
                ok[u] = j < total;
                x[u] = 0;
                if (ok[u]) x[u] = C[st + j];
            }
#pragma unroll
            for (uint32_t u = 0; u < EXP_UNR; u++)
                lpush(ok[u] && g_claim<SINGLE>(g, vis, x[u], cx[u]), x[u], q, &L.tail[d]);
        }
    }
}

// The hubs the level listed, a workgroup's width of arcs at a time (between
// two barriers).
template <int BS, bool SINGLE> __device__ __forceinline__ void g_hubs(Lds &L, const G1 &g)
{
    const uint32_t nh = uni(min(L.nhub, HUB_CAP));
    for (uint32_t k = 0; k < nh; k++) {
        const uint32_t e = uni(L.hub[k]), v = e & 0x7FFFFFFFu, d = e >> 31;
        const uint32_t *R = d ? g.Br : g.Fr, *C = d ? g.Bc : g.Fc;
        uint32_t *vis = d ? g.bvis : g.fvis;
        const uint32_t c = SINGLE ? 0u : g.cls[v];
        for (uint32_t j = at(R, v) + threadIdx.x, end = at(R, v + 1); j < end; j += BS) {
            const uint32_t w = C[j];
            lpush(g_claim<SINGLE>(g, vis, w, c), w, g.queue(2 * d), &L.tail[d]);
        }
    }
}

// Top-down levels of direction d while they are narrow, by the calling wave
// alone: the frontier is queue entries [lo, hi), hi - lo <= 64.  A level is
// two dependent loads (rows, columns) and LDS work, about 1.5 us against 3 to
// 4 us for a level of the whole workgroup with its barriers and queue in
// global memory; the first and last levels of nearly every search, and all
// of a long cycle's, are narrow.  Ends when the frontier is empty or no
// longer narrow: L.tail[d] has then grown by the vertices claimed, and the
// frontier is queue entries [L.nlo[d], L.tail[d]) (the entries of the levels
// in between are not written; nothing reads them).
template <bool SINGLE>
__device__ __forceinline__ void g_narrow(Lds &L, const G1 &g, uint32_t d, uint32_t lo, uint32_t hi)
{
    const uint32_t *R = d ? g.Br : g.Fr, *C = d ? g.Bc : g.Fc;
    uint32_t *vis = d ? g.bvis : g.fvis, *q = g.queue(2 * d), *near = L.near[d];
    uint32_t n = hi - lo, tail = hi, levels = 0;
    uint32_t v = ln() < n ? at(q, lo + ln()) : 0u;   // row 0 is empty
    for (;;) {
        const uint32_t b = at(R, v), deg = at(R, v + 1) - b;
        const uint32_t c = SINGLE ? 0u : g.cls[v];
        // any degree over the bound ends the loop before sums can wrap
        uint32_t sum = min(deg, NARROW_ARCS + 1);
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(sum, o);
            if ((int)ln() >= o) sum += y;
        }
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)sum, 63);
        if (total > NARROW_ARCS) break;
        const uint32_t start = b - (sum - deg);
        uint32_t m = 0;   // vertices claimed
        for (uint32_t j0 = 0; j0 < total; j0 += 64) {
            const uint32_t j = j0 + ln();
            uint32_t own = 0;
#pragma unroll
            for (uint32_t o = 32; o >= 1; o >>= 1) own += (uint32_t)__shfl((int)sum, (int)(own + o - 1)) <= j ? o : 0u;
            const uint32_t st = __shfl(start, (int)own), cx = SINGLE ? 0u : __shfl(c, (int)own);
            uint32_t x = 0;
            if (j < total) x = C[st + j];
            const bool claimed = j < total && g_claim<SINGLE>(g, vis, x, cx);
            const uint64_t mask = __ballot(claimed);
            if (claimed) near[m + (uint32_t)__popcll(mask & ((1ull << ln()) - 1))] = x;
            m += (uint32_t)__popcll(mask);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        tail += m;
        n = m;
        levels++;
        if (m > 64) {
            for (uint32_t i = ln(); i < m; i += 64) put(q, tail - m + i, near[i]);
            break;
        }
        if (m == 0) break;
        v = ln() < m ? near[ln()] : 0u;
        __builtin_amdgcn_wave_barrier();   // every entry is read before the next level's are written
    }
    if (n <= 64 && ln() < n) put(q, tail - n + ln(), v);
    if (ln() == 0) {
        L.tail[d] = tail;
        L.nlo[d] = tail - n;
        L.nlev[d] = levels;
    }
}

// The narrow levels of both directions, one wave each; returns false (and
// does nothing) unless every direction left is narrow.
template <int BS, bool SINGLE>
__device__ __forceinline__ bool g_narrow_both(Lds &L, const G1 &g, uint32_t (&lo)[2], uint32_t (&hi)[2])
{
    if (hi[0] - lo[0] > 64 || hi[1] - lo[1] > 64) return false;
    const uint32_t wv = uni(threadIdx.x >> 6);
    if (wv < 2 && (wv ? hi[1] != lo[1] : hi[0] != lo[0]))
        g_narrow<SINGLE>(L, g, wv, wv ? lo[1] : lo[0], wv ? hi[1] : hi[0]);
    __syncthreads();
    uint32_t levels = 0;
    for (uint32_t d = 0; d < 2; d++) {
        if (lo[d] == hi[d]) continue;
        lo[d] = uni(L.nlo[d]);
        hi[d] = uni(L.tail[d]);
        levels = max(levels, uni(L.nlev[d]));
    }
    if (threadIdx.x == 0) L.st.levels += levels;
    __syncthreads();
    return true;
}

// A bottom-up level of direction d: a live vertex not yet visited joins if
// one of its parents is visited: its first parent, if trim-1 has left the
// array of them (`first`), or one of its row.  A parent that joins in this same level may or may not
// be seen; if not, it is in the queue that the next level starts from.
// A level goes bottom-up when its frontier holds more than 1/BU_SWITCH of
// the vertices left to visit (1/BU_BURST right after growing kBurst-fold), in
// graphs of at least BU_DEGREE arcs per vertex.  The share is larger than
// the single-graph engine's 1/16: here a top-down claim is an LDS operation,
// while a bottom-up level walks the list of nearly every vertex whose first
// parent is not visited (mix: 1/16 2.93 ms, 1/4 2.77, 1/2 2.69, 1/1 2.66,
// untrimmed 4.5 to 4.6).  In sparser graphs a whole search top-down costs
// less than two bottom-up sweeps: 63,665 vertices of 2.07 arcs 1.20 -> 0.66
// ms for the search; from 8 arcs on it costs more (mix 1.91 -> 2.32 ms with
// BU_DEGREE at 8).
// 64-vertex chunks a wave takes side by side in a bottom-up level: their
// lists' loads are in flight together, but a step lasts as long as the
// longest list of all of them.  A batch, whose workgroups share the memory's
// latency, takes four (mix 1.84 ms; two 1.88, one 1.99); the small-graph
// kernel, alone on its CU and with graphs under 15,000 arcs in LDS, one (999
// vertices 45 us with four, 41 with two, 39 with one; 16,384 and 139,000
// arcs 101, 98, 95.5).
constexpr uint32_t BU_CHUNKS = 4;
constexpr uint64_t BU_SWITCH = 3, BU_BURST = 8, BU_DEGREE = 3;

template <uint32_t BUC>
__device__ __forceinline__ void g_bottom_up(Lds &L, const G1 &g, uint32_t d, uint32_t w, uint32_t nw,
                                            bool first)
{
    const uint32_t *R = d ? g.Fr : g.Br, *C = d ? g.Fc : g.Bc, *P = d ? g.f1() : g.b1();
    uint32_t *vis = d ? g.bvis : g.fvis, *q = g.queue(2 * d);
    const uint32_t nch = (g.V + 64) / 64;
    for (uint32_t c0 = w; c0 < nch; c0 += BUC * nw) {
        uint32_t word[BUC], cand[BUC], p[BUC];
        bool any = false;
#pragma unroll
        for (uint32_t h = 0; h < BUC; h++) {
            const uint32_t ch = c0 + h * nw, i = 2 * ch + (ln() >> 5);
            word[h] = ch < nch ? vis[i] : ~0u;
            cand[h] = ch < nch ? g.live[i] & ~word[h] : 0u;
            any |= cand[h] != 0;
        }
        if (!__ballot(any)) continue;
        if (first) {
#pragma unroll
            for (uint32_t h = 0; h < BUC; h++) {
                const uint32_t v = (c0 + h * nw) * 64 + ln();
                p[h] = at(P, v <= g.V ? v : 0u);
            }
        }
        bool hit[BUC], more[BUC];
        bool anym = false;
#pragma unroll
        for (uint32_t h = 0; h < BUC; h++) {
            const bool is = (cand[h] >> (ln() & 31)) & 1u;
            hit[h] = first && is && bbit(vis, p[h]);   // a live vertex has a first parent
            more[h] = is && !hit[h];
            anym |= more[h];
        }
        if (__ballot(anym)) {
            const uint32_t *Ck[BUC];
            uint32_t b[BUC], e[BUC], x[BUC];
#pragma unroll
            for (uint32_t h = 0; h < BUC; h++) {
                const uint32_t r = more[h] ? (c0 + h * nw) * 64 + ln() : 0u;   // row 0 is empty
                Ck[h] = C;
                b[h] = at(R, r);
                e[h] = at(R, r + 1);
            }
            g_any_bit<BUC>(Ck, b, e, vis, x);
#pragma unroll
            for (uint32_t h = 0; h < BUC; h++) hit[h] |= x[h] != 0;
        }
#pragma unroll
        for (uint32_t h = 0; h < BUC; h++) {
            const uint32_t ch = c0 + h * nw;
            const uint64_t m = __ballot(hit[h]);
            if (!m) continue;
            const uint32_t mw = ln() < 32 ? (uint32_t)m : (uint32_t)(m >> 32);
            if ((ln() & 31) == 0 && mw) vis[2 * ch + (ln() >> 5)] = word[h] | mw;
            lpush(hit[h], ch * 64 + ln(), q, &L.tail[d]);
        }
    }
}

// The waves of a level that has both directions to run are split between
// them (the two searches do not touch each other's state, so their chains of
// loads overlap); with one direction left every wave works on it.
template <int BS, class Level>
__device__ __forceinline__ void g_both(const uint32_t *lo, const uint32_t *hi, Level level)
{
    const uint32_t wv = uni(threadIdx.x >> 6), nwv = BS / 64;
    if (lo[0] != hi[0] && lo[1] != hi[1]) level(wv & 1, wv >> 1, nwv / 2);
    else level(lo[0] != hi[0] ? 0u : 1u, wv, nwv);
}

// The first pivot's FW and BW search, each level of a direction top-down or
// bottom-up (`dense`: the graph has the arcs for it).
template <int BS, uint32_t BUC>
__device__ __forceinline__ void g_first_search(Lds &L, const G1 &g, uint32_t nlive, bool first, bool dense)
{
    uint32_t lo[2] = {0, 0}, hi[2] = {1, 1}, prev[2] = {1, 1};
    bool bu[2] = {false, false};
    for (uint32_t level = 0; level <= g.V; level++) {   // each level claims a vertex or ends
        if (!bu[0] && !bu[1] && g_narrow_both<BS, true>(L, g, lo, hi)) {
            prev[0] = hi[0] - lo[0];
            prev[1] = hi[1] - lo[1];
        }
        if (lo[0] == hi[0] && lo[1] == hi[1]) break;
        if (threadIdx.x == 0) L.st.levels++;
        g_both<BS>(lo, hi, [&](uint32_t d, uint32_t w, uint32_t nw) {
            if (d ? bu[1] : bu[0]) g_bottom_up<BUC>(L, g, d, w, nw, first);
            else g_expand<true>(L, g, d, d ? lo[1] : lo[0], d ? hi[1] : hi[0], w, nw);
        });
        __syncthreads();
        if (uni(L.nhub)) {
            g_hubs<BS, true>(L, g);
            __syncthreads();
            if (threadIdx.x == 0) L.nhub = 0;
        }
        for (uint32_t d = 0; d < 2; d++) {
            if (lo[d] == hi[d]) continue;
            lo[d] = hi[d];
            hi[d] = uni(L.tail[d]);
            const uint64_t nf = hi[d] - lo[d], left = nlive - hi[d];
            if (!bu[d])
                bu[d] = dense && nf * (nf > kBurst * (uint64_t)prev[d] ? BU_BURST : BU_SWITCH) > left &&
                        nf * kBottomUpFloor >= nlive;
            else
                bu[d] = nf * kToTopDown >= nlive;
            prev[d] = (uint32_t)nf;
        }
        __syncthreads();   // every lane has read the tails and the hub count
    }
}

// ----------------------------------------------- the later phases ---
// Over the `n` vertices the first round left (g.list), in classes.

#define LIST_LOOP(v)                                                                        \
    for (uint32_t _i = threadIdx.x, v; _i < n && (v = at(list, _i), true); _i += BS)
// with all 64 lanes of a wave in every step; past the end v is 0, the dummy,
// which is dead, has no colour and whose row is empty
#define WAVE_LIST_LOOP(v)                                                                   \
    for (uint32_t _i = threadIdx.x & ~63u, v; _i < n && (v = _i + ln() < n ? at(list, _i + ln()) : 0u, true); _i += BS)

template <int BS> __device__ __forceinline__ void g_trim1(Lds &L, const G1 &g, uint32_t n)
{
    const uint32_t *list = g.list;
    for (uint32_t pass = 0; pass <= g.V; pass++) {   // each pass removes a vertex or ends
        uint32_t removed = 0;
        WAVE_LIST_LOOP(v)
        {
            // class and both rows' offsets together; a dead vertex scans
            // empty ranges, so the offsets are used on every path and are
            // not loaded after the class test or the first scan
            const uint32_t c = g.cls[v];
            const uint32_t bb = at(g.Br, v), be = at(g.Br, v + 1), fb = at(g.Fr, v), fe = at(g.Fr, v + 1);
            const bool act = c != DEAD;
            const bool kin = g_any_cls(g.Bc, bb, act ? be : bb, g.cls, c);
            const bool keep = g_any_cls(g.Fc, fb, kin ? fe : fb, g.cls, c);
            if (act && !keep) {   // its label is still the v | LAB_FINAL it was listed with
                __hip_atomic_store(&g.cls[v], DEAD, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                removed++;
            }
        }
        const uint32_t n1 = wg_sum<BS>(L, removed, pass & 1);
        if (!n1) break;
        if (threadIdx.x == 0) L.st.trim1 += n1;
    }
    __syncthreads();
}

__device__ __forceinline__ int g_deg2(const uint32_t *R, const uint32_t *C, const uint32_t *cls,
                                      uint32_t v, uint32_t c, uint32_t *k)
{
    int d = 0;
    for (uint32_t i = at(R, v), e = at(R, v + 1); i < e; i++) {
        const uint32_t w = C[i];
        if (cls[w] != c) continue;
        if (++d == 2) return 2;
        *k = w;
    }
    return d;
}

__device__ __forceinline__ bool g_arc(const uint32_t *R, const uint32_t *C, uint32_t v, uint32_t k)
{
    for (uint32_t i = at(R, v), e = at(R, v + 1); i < e; i++)
        if (C[i] == k) return true;
    return false;
}

// trim-2 (scc_kernels.cu:236-357), claim by CAS on the smaller id
template <int BS> __device__ __forceinline__ void g_trim2(Lds &L, const G1 &g, uint32_t n)
{
    const uint32_t *list = g.list;
    LIST_LOOP(v)
    {
        const uint32_t c = g.cls[v];
        if (c == DEAD) continue;
        uint32_t k = 0, kk = 0;
        bool hit = g_deg2(g.Br, g.Bc, g.cls, v, c, &k) == 1 && g_arc(g.Fr, g.Fc, v, k) &&
                   g_deg2(g.Br, g.Bc, g.cls, k, c, &kk) == 1;
        if (!hit) {
            k = 0;
            hit = g_deg2(g.Fr, g.Fc, g.cls, v, c, &k) == 1 && g_arc(g.Br, g.Bc, v, k) &&
                  g_deg2(g.Fr, g.Fc, g.cls, k, c, &kk) == 1;
        }
        if (hit) {
            const uint32_t lo = v < k ? v : k, hi = v < k ? k : v;
            if (atomicCAS(&g.cls[lo], c, DEAD) == c) {
                atomicAdd(&L.st.trim2, 1u);
                g.lab[lo] = lo | LAB_FINAL;
                g.lab[hi] = lo | LAB_FINAL;
                __hip_atomic_store(&g.cls[hi], DEAD, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
    }
    __syncthreads();
}

// FW and, with do_bw, BW top-down levels from the seeded queues
template <int BS> __device__ __forceinline__ void g_reach(Lds &L, const G1 &g, bool do_bw)
{
    uint32_t lo[2] = {0, 0};
    uint32_t hi[2] = {uni(L.tail[0]), do_bw ? uni(L.tail[1]) : 0u};
    __syncthreads();
    for (uint32_t level = 0; level <= g.V; level++) {   // each level claims a vertex or ends
        g_narrow_both<BS, false>(L, g, lo, hi);
        if (lo[0] == hi[0] && lo[1] == hi[1]) break;
        if (threadIdx.x == 0) L.st.levels++;
        g_both<BS>(lo, hi, [&](uint32_t d, uint32_t w, uint32_t nw) {
            g_expand<false>(L, g, d, d ? lo[1] : lo[0], d ? hi[1] : hi[0], w, nw);
        });
        __syncthreads();
        if (uni(L.nhub)) {
            g_hubs<BS, false>(L, g);
            __syncthreads();
            if (threadIdx.x == 0) L.nhub = 0;
        }
        for (uint32_t d = 0; d < 2; d++) {
            if (lo[d] == hi[d]) continue;
            lo[d] = hi[d];
            hi[d] = uni(L.tail[d]);
        }
        __syncthreads();
    }
}

// One pivot per live class, seeded in both directions.
template <int BS> __device__ __forceinline__ void g_pivots(Lds &L, const G1 &g, uint32_t n)
{
    const uint32_t *list = g.list;
    // a wave whose live lanes share a class does one atomic
    unsigned long long *piv = reinterpret_cast<unsigned long long *>(g.piv);
    for (uint32_t i0 = threadIdx.x & ~63u; i0 < n; i0 += BS) {
        const uint32_t v = i0 + ln() < n ? at(list, i0 + ln()) : 0u;   // vertex 0, the dummy, is dead
        const uint32_t c = g.cls[v];
        const bool ok = c != DEAD;
        const uint64_t live = __ballot(ok);
        if (!live) continue;
        const int lead = __ffsll((unsigned long long)live) - 1;
        const uint32_t c0 = __shfl(c, lead);
        unsigned long long k = ok ? bkey(g.Fr, g.Br, v) : 0ull;
        if (__all(!ok || c == c0)) {
            for (int o = 32; o > 0; o >>= 1) {
                const unsigned long long x = __shfl_xor(k, o);
                k = x > k ? x : k;
            }
            if ((int)ln() == lead && k > __hip_atomic_load(&piv[c0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                atomicMax(&piv[c0], k);
        } else if (ok && k > __hip_atomic_load(&piv[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
            atomicMax(&piv[c], k);
        }
    }
    if (threadIdx.x == 0) L.npiv = 0;
    __syncthreads();
    LIST_LOOP(v)
    {
        const uint32_t c = g.cls[v];
        const bool win = c != DEAD && g.piv[c] == bkey(g.Fr, g.Br, v);
        if (win) {
            atomicOr(&g.fvis[v >> 5], 1u << (v & 31));
            atomicOr(&g.bvis[v >> 5], 1u << (v & 31));
        }
        lpush(win, v, g.pivlist, &L.npiv);
    }
    __syncthreads();
    const uint32_t np = uni(L.npiv);
    for (uint32_t i = threadIdx.x; i < np; i += BS) {
        g.queue(0)[i] = g.pivlist[i];
        g.queue(2)[i] = g.pivlist[i];
    }
    if (threadIdx.x == 0) {
        L.tail[0] = np;
        L.tail[1] = np;
        L.st.pivots += np;   // each finds its SCC
    }
    __syncthreads();
}

// update (scc_kernels.cu:124-142) + clear the next round's pivot slots, if
// there is one
template <int BS> __device__ __forceinline__ uint32_t g_update(Lds &L, const G1 &g, uint32_t n)
{
    const uint32_t *list = g.list;
    uint32_t live = 0;
    LIST_LOOP(v)
    {
        const uint32_t c = g.cls[v];
        if (c == DEAD) continue;
        uint32_t p = bkey_vertex(g.piv[c]);
        if (p - 1u >= g.V) {   // every live class elects a pivot; keep indices in range if not
            L.anom = 1;
            p = v;
        }
        const uint32_t f = bbit(g.fvis, v), b = bbit(g.bvis, v);
        if (f && b) {
            g.lab[v] = p;
            g.cls[v] = DEAD;
        } else {
            g.cls[v] = 3u * p + f + 2u * b;
            live++;
        }
    }
    const uint32_t left = wg_sum1<BS>(L, live);
    if (!left) return 0;   // nothing reads the keys of a graph that is done
    for (uint32_t i = threadIdx.x; i < L.npiv; i += BS) {
        const uint32_t p = g.pivlist[i];
        g.piv[3ull * p] = 0;
        g.piv[3ull * p + 1] = 0;
        g.piv[3ull * p + 2] = 0;
    }
    __syncthreads();
    return left;
}

// "WCC" min reachable label with pointer jumping (scc_kernels.cu:477-536)
template <int BS> __device__ __forceinline__ void g_minlabel(Lds &L, const G1 &g, uint32_t n)
{
    const uint32_t *list = g.list;
    LIST_LOOP(v)
        if (g.cls[v] != DEAD) g.cls[v] = v;
    __syncthreads();
    for (uint32_t it = 0; it <= g.V; it++) {   // labels only decrease
        uint32_t changed = 0;
        WAVE_LIST_LOOP(v)
        {
            // label and row offsets together (an inactive lane folds an
            // empty range, so the offsets are used on every path)
            const uint32_t m0 = g.cls[v], b = at(g.Fr, v), e = at(g.Fr, v + 1);
            const bool act = m0 != DEAD;
            uint32_t m = g_fold<false>(g.Fc, b, act ? e : b, g.cls, m0);
            if (!act) continue;
            for (int jump = 0; jump < 32; jump++) {
                const uint32_t x = g.cls[m];
                if (x >= m) break;
                m = x;
            }
            if (m < m0) {
                __hip_atomic_store(&g.cls[v], m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                changed = 1;
            }
        }
        if (!wg_sum<BS>(L, changed, it & 1)) break;
    }
    __syncthreads();
    LIST_LOOP(v)
    {
        const uint32_t m = g.cls[v];
        if (m == DEAD) continue;
        if (m == v) g.piv[3ull * v] = 0;
        g.cls[v] = 3u * m;
    }
    __syncthreads();
}

// vSlota colouring loop (scc_Coloring.cu:590-637); aux is 0 for every
// vertex outside the list
template <int BS> __device__ __forceinline__ void g_color_loop(Lds &L, const G1 &g, uint32_t n)
{
    const uint32_t *list = g.list;
    uint32_t live = n;
    for (uint32_t round = 0; live && round <= g.V; round++) {   // a round finishes >= 1 SCC
        LIST_LOOP(v)
            g.aux[v] = g.cls[v] != DEAD ? v : 0u;
        __syncthreads();
        for (uint32_t it = 0; it <= g.V; it++) {   // colours only increase
            uint32_t changed = 0;
            WAVE_LIST_LOOP(v)
            {
                // as in g_minlabel
                const uint32_t m0 = g.aux[v], b = at(g.Fr, v), e = at(g.Fr, v + 1);
                const bool act = m0 != 0;
                uint32_t m = g_fold<true>(g.Fc, b, act ? e : b, g.aux, m0);
                if (!act) continue;
                for (int jump = 0; jump < 32; jump++) {
                    const uint32_t x = g.aux[m];
                    if (x <= m) break;
                    m = x;
                }
                if (m > m0) {
                    __hip_atomic_store(&g.aux[v], m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    changed = 1;
                }
            }
            if (!wg_sum<BS>(L, changed, it & 1)) break;
        }
        __syncthreads();
        g_clear_vis<BS>(g);
        if (threadIdx.x == 0) L.tail[0] = 0;
        __syncthreads();
        LIST_LOOP(v)
        {
            bool root = false;
            if (g.cls[v] != DEAD) {
                const uint32_t c = g.aux[v];
                g.cls[v] = c;
                root = c == v;
                if (root) atomicOr(&g.fvis[v >> 5], 1u << (v & 31));
            }
            lpush(root, v, g.queue(0), &L.tail[0]);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            L.st.pivots += L.tail[0];   // each root finds its SCC
            L.st.rounds++;
        }
        g_reach<BS>(L, g, false);
        uint32_t lv = 0;
        LIST_LOOP(v)
        {
            const uint32_t c = g.cls[v];
            if (c == DEAD) continue;
            if (bbit(g.fvis, v)) {
                g.lab[v] = c;
                g.cls[v] = DEAD;
            } else {
                lv++;
            }
        }
        live = wg_sum1<BS>(L, lv);
    }
}

// Canonical labels of the listed vertices; returns their number of SCCs.
// The minimum per label: the lanes of a wave that share its first label
// combine, the others go lane by lane, and the guard reads the current
// minimum at agent scope (the CU's L1 may hold a stale copy), so a large SCC
// costs about one atomic per wave instead of one per vertex.  Combining up to
// four labels per step made the pass 70 us on 16,384 vertices in 5,466 SCCs,
// so 55.
template <int BS> __device__ __forceinline__ uint32_t g_canon(Lds &L, const G1 &g, uint32_t n)
{
    const uint32_t *list = g.list;
    LIST_LOOP(v)
        g.aux[v] = DEAD;
    __syncthreads();
    for (uint32_t i0 = threadIdx.x & ~63u; i0 < n; i0 += BS) {
        const uint32_t v = i0 + ln() < n ? at(list, i0 + ln()) : 0u;
        const uint32_t l = v ? g.lab[v] : LAB_FINAL;
        bool pending = !(l & LAB_FINAL);
        const uint64_t pm = __ballot(pending);
        if (!pm) continue;
        const int lead = __ffsll((unsigned long long)pm) - 1;
        const uint32_t rl = (uint32_t)__builtin_amdgcn_readlane((int)l, lead);
        const bool mine = pending && l == rl;
        uint32_t m = mine ? v : DEAD;
        for (int o = 32; o > 0; o >>= 1) {
            const uint32_t x = __shfl_xor(m, o);
            m = x < m ? x : m;
        }
        if ((int)ln() == lead && m < __hip_atomic_load(&g.aux[rl], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMin(&g.aux[rl], m);
        pending = pending && !mine;
        if (pending && v < __hip_atomic_load(&g.aux[l], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMin(&g.aux[l], v);
    }
    __syncthreads();
    uint32_t roots = 0;
    LIST_LOOP(v)
    {
        const uint32_t l = g.lab[v];
        const uint32_t r = (l & LAB_FINAL) ? (l & ~LAB_FINAL) : g.aux[l];
        g.lab[v] = r;
        roots += r == v;
    }
    return wg_sum1<BS>(L, roots);
}

// The whole pipeline of one graph; returns its number of SCCs.  Inlined once
// per place the views may be in, so that accesses to LDS are LDS instructions.
//
// Under Hong's order the small-graph kernel reports the pivot and the counts
// of trim-1's fixpoint, as the device-wide engine does.  FULL 2 trims that
// far before the first search, and so does FULL 1 where it sweeps anyway.
// Otherwise FULL 1 searches first: a pivot on a cycle is none that trim-1
// would have removed, and the list phases then remove and count the same
// vertices (none of them lies on a path between two that stay, so the search
// puts those into the same classes).  After an SCC of one vertex it trims, and
// searches again if the pivot went.  Trimming first where the graph is in LDS
// takes 999 vertices from 50.5 to 46.5 us; outside it 16,384 vertices and
// 139,000 arcs take 126 us so and 122 searched first.
template <int BS, uint32_t BUC = BU_CHUNKS, int FULL = 0>
__device__ __forceinline__ uint32_t g_solve(Lds &L, const G1 &g, uint32_t cfg)
{
    const uint32_t nch = (g.V + 64) / 64, nw = 2 * nch;
    if (threadIdx.x == 0) {
        L.key = 0;
        L.nhub = 0;
        L.nact = 0;
        L.anom = 0;
        L.st = GraphStats();
    }
    __syncthreads();
    const uint32_t ndeg = g_degrees<BS>(L, g, cfg_t1(cfg));
    // (never with the trims off; FULL: colouring trims once, as in the device-wide engine)
    const bool first = (uint64_t)ndeg * TRIM_MIN > g.V && !(FULL && cfg_slota(cfg));
    if (first) g_trim_bits<BS, FULL != 0>(L, g);
    const bool full = FULL && cfg_t1(cfg) && !cfg_slota(cfg);
    bool trim = full && (FULL == 2 || first);
    if (trim) {
        if (!first) g_list_gone<BS>(L, g);   // else queue 0 holds what the last sweep removed
        g_trim_listed<BS>(L, g);
    }
    uint32_t nlive, p0, nmem, root;
    for (;;) {
        uint32_t nl = 0;
        for (uint32_t i = threadIdx.x; i < nw; i += BS) {
            nl += (uint32_t)__popc(g.live[i]);
            g.fvis[i] = 0;
            g.bvis[i] = 0;
        }
        nlive = wg_sum1<BS>(L, nl);
        // the best key of the degree pass may name a vertex the trim removed
        if (nlive && !bbit(g.live, bkey_vertex(L.key))) {
            __syncthreads();
            if (threadIdx.x == 0) L.key = 0;
            __syncthreads();
            unsigned long long best = 0;
            for (uint32_t v = threadIdx.x; v <= g.V; v += BS)
                if (bbit(g.live, v)) {
                    const unsigned long long k = bkey(g.Fr, g.Br, v);
                    best = k > best ? k : best;
                }
            for (int o = 32; o > 0; o >>= 1) {
                const unsigned long long x = __shfl_xor(best, o);
                best = x > best ? x : best;
            }
            if (ln() == 0 && best) atomicMax(&L.key, best);
            __syncthreads();
        }
        p0 = nlive ? uni(bkey_vertex(L.key)) : 0u;
        if (nlive) {
            if (threadIdx.x == 0) {
                g.fvis[p0 >> 5] |= 1u << (p0 & 31);
                g.bvis[p0 >> 5] |= 1u << (p0 & 31);
                g.queue(0)[0] = p0;
                g.queue(2)[0] = p0;
                L.tail[0] = 1;
                L.tail[1] = 1;
            }
            __syncthreads();
            const uint64_t t0 = wall_clock64();
            g_first_search<BS, BUC>(L, g, nlive, first, g.E >= BU_DEGREE * (uint64_t)g.V);
            if (threadIdx.x == 0) {
                L.st.search_ticks = wall_clock64() - t0;
                L.st.first_pivot = p0;
                L.st.pivots = 1;
            }
        }
        // the pivot's SCC: its size, its smallest vertex
        uint32_t members = 0, least = DEAD;
        for (uint32_t i = threadIdx.x; i < nw; i += BS) {
            const uint32_t m = g.live[i] & g.fvis[i] & g.bvis[i];
            members += (uint32_t)__popc(m);
            if (m && least == DEAD) least = 32 * i + (uint32_t)(__ffs(m) - 1);
        }
        nmem = wg_sum1<BS>(L, members);
        root = wg_min1<BS>(L, least);
        if (!full || trim || nmem != 1) break;
        g_list_gone<BS>(L, g);
        g_trim_listed<BS>(L, g);
        trim = true;
        if (bbit(g.live, p0)) {   // what the trim removed had no part in the search
            nl = 0;
            for (uint32_t i = threadIdx.x; i < nw; i += BS) nl += (uint32_t)__popc(g.live[i]);
            nlive = wg_sum1<BS>(L, nl);
            break;
        }
        if (threadIdx.x == 0) L.st = GraphStats();
    }
    const uint32_t singles = g.V - nlive;   // trim-1's
    if (threadIdx.x == 0) L.st.trim1 = singles;
    if (nmem == nlive) {
        for (uint32_t v = threadIdx.x; v <= g.V; v += BS) g.lab[v] = bbit(g.live, v) ? root : v;
        return singles + (nmem ? 1u : 0u);
    }
    // Vertices are left: their classes and the list of them.  Every other
    // label is final.  Class 3 p0 + k needs its pivot key cleared.
    const bool slota = cfg_slota(cfg);
    uint32_t *list = g.list;   // the first out-neighbours are not needed any more
    for (uint32_t c0 = uni(threadIdx.x >> 6); c0 < nch; c0 += BS / 64) {
        const uint32_t v = c0 * 64 + ln(), i = 2 * c0 + (ln() >> 5), sh = ln() & 31;
        const uint32_t lw = g.live[i], f = (g.fvis[i] >> sh) & 1u, b = (g.bvis[i] >> sh) & 1u;
        const bool alive = (lw >> sh) & 1u, rest = alive && !(f && b);
        if (v <= g.V) {
            g.lab[v] = alive && !rest ? root : (rest ? v | LAB_FINAL : v);
            g.cls[v] = rest ? 3u * p0 + f + 2u * b : DEAD;
            if (slota) g.aux[v] = 0;
        }
        lpush(rest, v, list, &L.nact);
    }
    if (threadIdx.x < 3) g.piv[3ull * p0 + threadIdx.x] = 0;
    __syncthreads();
    const uint32_t n = uni(L.nact);
    if (!slota) {
        if (cfg_t1(cfg)) g_trim1<BS>(L, g, n);
        if (cfg_t2(cfg)) {
            g_trim2<BS>(L, g, n);
            if (cfg_t1(cfg)) g_trim1<BS>(L, g, n);
        }
        g_minlabel<BS>(L, g, n);
        for (uint32_t round = 0; round <= g.V + 1; round++) {
            g_clear_vis<BS>(g);
            __syncthreads();
            g_pivots<BS>(L, g, n);
            g_reach<BS>(L, g, true);
            if (!g_update<BS>(L, g, n)) break;
            if (threadIdx.x == 0) L.st.rounds++;
        }
    } else {
        g_color_loop<BS>(L, g, n);
    }
    return singles + (nmem ? 1u : 0u) + g_canon<BS>(L, g, n);
}

} // namespace

// LDS tiers.  A graph whose bitmaps (live, FW and BW visited) fit `words`
// words each keeps them in LDS, so probes and claims are LDS operations (a
// device-wide atomic costs a share of a chip-wide rate of about 10 G/s); a
// graph whose class words fit `cls_words` keeps those in LDS as well for the
// phases after the first round.  Larger graphs use their slots in global
// memory.  The tiers leave room for several workgroups per CU:
// (their number is set by registers before LDS at 1,024 and 512 lanes):
//   1,024 lanes: bitmaps up to 2^16 vertices, classes up to 2^13 (58 KB)
//     512 lanes: bitmaps up to 2^16, classes up to 2^12 (42 KB)
//     256 lanes: bitmaps up to 2^16, classes up to 2^11 (34 KB)
template <int BS> struct BTier;
template <> struct BTier<1024> {
    static constexpr uint32_t words = 2 * ((65536 + 64) / 64);
    static constexpr uint32_t cls_words = (1u << 13) + 2;
};
template <> struct BTier<512> {
    static constexpr uint32_t words = 2 * ((65536 + 64) / 64);
    static constexpr uint32_t cls_words = (1u << 12) + 2;
};
template <> struct BTier<256> {
    static constexpr uint32_t words = 2 * ((65536 + 64) / 64);
    static constexpr uint32_t cls_words = (1u << 11) + 2;
};

// At least four waves per SIMD (128 vector registers): a second 512-lane
// workgroup then fits a CU (mix at 512 lanes 2.54 -> 1.67 ms); 1,024 lanes
// need as many anyway, 256 lanes do not change.
template <int BS>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(4))) void batch_scc_kernel(BatchDev B, uint32_t first, uint32_t count)
{
    __shared__ Lds L;
    __shared__ uint32_t s_bits[3][BTier<BS>::words];
    __shared__ uint32_t s_cls[BTier<BS>::cls_words];
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) L.graph = atomicAdd(B.next, 1u);
        __syncthreads();
        const uint32_t k = uni(L.graph);
        if (k >= count) break;
        const uint32_t gi = B.order[first + k];
        const uint64_t vo = B.voff[gi], eo = B.eoff[gi];
        const uint32_t cfg = B.cfg[gi];
        const uint64_t t0 = wall_clock64();
        G1 g;
        g.V = B.Vn[gi];
        g.E = (uint32_t)(B.eoff[gi + 1] - eo);
        g.Fr = B.Fr + vo;
        g.Br = B.Br + vo;
        g.Fc = B.Fc + eo;
        g.Bc = B.Bc + eo;
        g.lab = B.lab + vo;
        g.aux = B.aux + vo;
        g.piv = B.piv + 3 * vo;
        g.q = B.q + 4 * vo;
        g.list = g.queue(1);
        g.pivlist = B.pivlist + vo;
        uint32_t n;
        if (2 * ((g.V + 64) / 64) > BTier<BS>::words) {
            g.live = g.queue(3);
            g.fvis = B.fvis + vo / 32;
            g.bvis = B.bvis + vo / 32;
            g.cls = B.cls + vo;
            n = g_solve<BS>(L, g, cfg);
        } else {
            g.live = s_bits[0];
            g.fvis = s_bits[1];
            g.bvis = s_bits[2];
            if (g.V + 1 > BTier<BS>::cls_words) {
                g.cls = B.cls + vo;
                n = g_solve<BS>(L, g, cfg);
            } else {
                g.cls = s_cls;
                n = g_solve<BS>(L, g, cfg);
            }
        }
        if (threadIdx.x == 0) {
            B.nscc[gi] = L.anom ? BATCH_ANOMALY : n;
            B.tstart[gi] = t0;
            B.tend[gi] = wall_clock64();
        }
    }
}

// ------------------------------------------------ one small graph ---
// A resident graph of at most SMALL_V vertices and SMALL_E arcs as one
// launch of one workgroup, instead of the device-wide engine's chain of
// about 19 launches and two looks at the counters (100 to 150 us on graphs
// of this size, 300 and more where the first round leaves vertices).  Where
// the whole CSR and the work arrays fit LDS they are copied there first, so
// a level's dependent loads are LDS reads.  The counters the host waits for
// are written to its mapped memory by the kernel itself.
// Whole calls, one workgroup against the device-wide engine, at 2, 4, 8 and
// 16 arcs per vertex: 1,000 vertices 58 / 39 / 29 / 26 us against 120 / 112 /
// 123 / 98, 8,000 vertices 125 / 90 / 78 / 56 against 407 / 134 / 116 / 107,
// 16,384 vertices 193 / 139 / 94 / 87 against 388 / 149 / 121 / 108; at
// 32,768 vertices it would be 250 against 148 at 4 arcs.  Structured graphs
// of 16,384 vertices: a 0.7 grid 524 against 734, islands of up to nine 713
// against 2,140, rings of 16 1,230 against 6,660, a path 54,000 against
// 74,000, a chain of 2-cycles 62,000 against 207,000.  Slower here are a
// cycle (14.7 against 9.7 ms, 4,096 vertices 3.6 against 2.1: a hop of the
// device-wide engine's low-degree levels is one memory trip, a narrow level
// two; nothing known before the launch tells it from a path) and, with the
// trims off, a star without a cycle (207 against 186): one CU does all its
// scattered key accesses.  What is left after the first round is listed in
// LDS beside the class words (16,384 vertices in 5,466 SCCs 358 -> 344).
constexpr uint32_t SMALL_LDS = 36864;   // words: class words, list and marks, or all of a graph that fits

__global__ __launch_bounds__(1024) void small_scc_kernel(SmallArgs a)
{
    __shared__ Lds L;
    constexpr uint32_t words = 2 * ((SMALL_V + 64) / 64);
    __shared__ uint32_t s_bits[3 * words];
    __shared__ uint32_t s_mem[SMALL_LDS];
    static_assert(2 * SMALL_V + 3 + 2 * words <= SMALL_LDS, "class words, list of vertices left and marks fit");
    const uint64_t t0 = wall_clock64();
    G1 g;
    g.V = a.V;
    g.E = a.E;
    g.lab = a.lab;
    g.piv = a.piv;
    g.pivlist = a.pivlist;
    g.live = s_bits;
    g.fvis = s_bits + words;
    g.bvis = s_bits + 2 * words;
    g.cls = s_mem;
    uint32_t n;
    const uint64_t nr = (uint64_t)a.V + 2;
    if (8 * nr + 2 * (uint64_t)a.E <= SMALL_LDS) {
        uint32_t *Fr = s_mem + nr, *Br = Fr + nr, *Fc = Br + nr, *Bc = Fc + a.E;
        g.aux = Bc + a.E;
        g.q = g.aux + nr;   // 4 * nr words
        g.list = g.queue(1);
        g.seen = s_bits + words;   // the visited bitmaps, free until the search
        for (uint32_t i = threadIdx.x; i < nr; i += 1024) {
            Fr[i] = a.Fr[i];
            Br[i] = a.Br[i];
        }
        for (uint32_t i = threadIdx.x; i < a.E; i += 1024) {
            Fc[i] = a.Fc[i];
            Bc[i] = a.Bc[i];
        }
        g.Fr = Fr;
        g.Br = Br;
        g.Fc = Fc;
        g.Bc = Bc;
        __syncthreads();
        n = g_solve<1024, 1, 2>(L, g, a.cfg);
    } else {
        g.Fr = a.Fr;
        g.Br = a.Br;
        g.Fc = a.Fc;
        g.Bc = a.Bc;
        g.aux = a.aux;
        g.q = a.q;
        g.list = s_mem + SMALL_V + 1;
        g.seen = s_mem + 2 * SMALL_V + 3;
        n = g_solve<1024, 1, 1>(L, g, a.cfg);
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    uint32_t *p = a.pub;
    p[CT(C_NSCC)] = n;
    p[CT(C_TRIM1)] = L.st.trim1;
    p[CT(C_TRIM2)] = L.st.trim2;
    p[CT(C_PIVOT)] = L.st.pivots;
    p[CT(C_PIV0)] = L.st.first_pivot;
    p[CT(C_ANOM)] = L.anom;
    p[CT(C_NPIV)] = L.st.rounds;
    p[CT(C_NLEVELS)] = L.st.levels;
    const uint64_t all = wall_clock64() - t0, search = L.st.search_ticks;
    p[CT(C_FWV)] = (uint32_t)all;
    p[CT(C_FWV) + 1] = (uint32_t)(all >> 32);
    p[CT(C_BWV)] = (uint32_t)search;
    p[CT(C_BWV) + 1] = (uint32_t)(search >> 32);
    __threadfence_system();
    __hip_atomic_store(p + CT(C_COUNT), a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

void k_small(hipStream_t s, const SmallArgs &a) { small_scc_kernel<<<1, 1024, 0, s>>>(a); }

uint32_t batch_cfg(bool trim1, bool trim2, bool slota)
{
    return (trim1 ? 1u : 0u) | (trim2 ? 2u : 0u) | (slota ? 4u : 0u);
}

int batch_occupancy(int block)
{
    int n = 0;
    hipError_t e;
    if (block == 1024)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, batch_scc_kernel<1024>, 1024, 0);
    else if (block == 512)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, batch_scc_kernel<512>, 512, 0);
    else
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, batch_scc_kernel<256>, 256, 0);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return 1;
    }
    return n < 1 ? 1 : n;
}

void k_batch(hipStream_t s, const BatchDev &B, uint32_t first, uint32_t count, int block, uint32_t grid)
{
    if (!count) return;
    if (block == 1024)
        batch_scc_kernel<1024><<<grid, 1024, 0, s>>>(B, first, count);
    else if (block == 512)
        batch_scc_kernel<512><<<grid, 512, 0, s>>>(B, first, count);
    else
        batch_scc_kernel<256><<<grid, 256, 0, s>>>(B, first, count);
}

} // namespace sccamd
