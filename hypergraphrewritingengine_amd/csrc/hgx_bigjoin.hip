// hgx_bigjoin.hip -- the join over one large state (tens of thousands of edges and up), where
// the state does not fit LDS: the match-join stress workload, one rewriting step of one big
// state (hgx_match_count, and hgx_match_count_noalloc over a fixed device scratch).
//
// Index (the role of SignatureIndex / InvertedVertexIndex, hypergraph/src/index.cpp:45-80): a CSR
// keyed by (vertex, pivot position) -> ascending edge ids, over the positions the rule's join
// pivots on and the edges of the arities it wants there. One pass over the edges counts the lists
// (the counter's old value is an entry's place in its list), marks the seeds, and counts the edges
// of each vertex tuple in a hash table (for closing edges, below); one scan places lists, tuples
// and seeds; a second pass writes the entries, and a third puts each list in ascending order by
// counting an entry's smaller neighbours (long lists in LDS, the longest by a bit set of the edges
// there). Above
// kIndexPlaceEdges edges the lists come from a stable radix sort of (list, edge) pairs instead.
//
// Join (join_core.hpp:143-208), breadth first: the partial matches of depth d (d edges in join
// order) are a frontier held in HBM, in lexicographic order. Depth d+1 takes every (partial,
// candidate) pair -- candidates from the CSR list of the pivot vertex, ascending -- as one item:
// the items are numbered by a scan of the per-partial list lengths and dealt to workgroups in
// tiles. A test pass writes one bit per item and the survivors of each tile, a scan of the tile
// counts places every tile, and a place pass writes the items whose bit is set, in item order.
// Item order is (partial, ascending candidate), so the final match list is in the order of a
// serial depth-first join over ascending candidates -- the oracle's order. A last pattern edge
// that closes (every vertex bound earlier) has no depth of its own: the items of the depth before
// it look its tuple up. The work per depth is spread over all its candidates, not one thread per
// seed.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstring>
#include <vector>

#include "hgx_bigjoin.hpp"
#include "hgx_device.hpp"
#include "hgx_kernels.hpp"
#include "hgx_runtime.hpp"

namespace hgx {

constexpr uint32_t BJ_THREADS = 256;
constexpr uint32_t BJ_WAVES = BJ_THREADS / WAVE;
constexpr uint32_t BJ_IPT = 4;                            // items per thread per tile
constexpr uint32_t BJ_TILE = BJ_THREADS * BJ_IPT;         // items per workgroup tile
constexpr uint32_t BJ_WORDS = BJ_TILE / WAVE;             // survivor words per tile
constexpr uint32_t BJ_STAGE_Q = 4096;                     // partials a tile looks through for its lists
constexpr uint32_t BJ_STAGE_W = 2048;                     // words of their edges and vertices
constexpr uint32_t BJ_TILE_BYTES = 8 * (BJ_WORDS + 4);    // device memory of a tile

// ---- index -------------------------------------------------------------------------------

// Zero fill: a kernel, so the join's stream holds kernels and copies only.
__global__ void k_bj_zero(uint32_t* p, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// The key of a vertex tuple (arity, vertices), vertex i given by x(i): equal tuples have equal
// keys; the join verifies every vertex of a candidate, so a collision costs a rejected candidate,
// never a wrong match.
template <class X>
__device__ __forceinline__ uint64_t tuple_key(uint32_t a, X x) {
    uint64_t h = 0x9E3779B97F4A7C15ULL ^ a;
    for (uint32_t i = 0; i < a; ++i) h = mix64(h ^ ((uint64_t)x(i) + 0x632BE59BD9B4E019ULL * (i + 1)));
    return h;
}
// The table holds the key's upper half (0 marks an empty place); its lower half picks the place.
__device__ __forceinline__ uint32_t tuple_tag(uint64_t key) {
    const uint32_t t = (uint32_t)(key >> 32);
    return t ? t : 1u;
}

// Whether edges of arity a are listed at pivot position number u, and whether the tuple table
// holds edges of arity a.
__device__ __forceinline__ bool bj_listed(const BJView& v, uint32_t u, uint32_t a) {
    return a < 32 && ((v.uar[u] >> a) & 1u);
}
__device__ __forceinline__ bool bj_tabled(const BJView& v, uint32_t a) { return a < 32 && ((v.tar >> a) & 1u); }

// One count at cnt[k] for each lane with `in`; returns the value before. The lanes that share the
// first lane's counter add once, so a hub costs an atomic per wave and not one per edge (a star of
// 1 million edges took 12.4 ms with one each).
__device__ __forceinline__ uint32_t bj_add(uint32_t* cnt, uint64_t k, bool in) {
    uint32_t r = 0;
    for (uint32_t round = 0; round < 2; ++round) {
        const uint64_t left = __ballot(in);
        if (!left) break;
        const uint32_t first = (uint32_t)__builtin_ctzll(left);
        const uint64_t same = __ballot(in && k == wave_lane_u64(k, first));
        if (!(same & (same - 1))) break;
        uint32_t base = 0;
        if (lane_id() == first) base = atomicAdd(&cnt[k], (uint32_t)__popcll(same));
        base = __shfl(base, (int)first, WAVE);
        if ((same >> lane_id()) & 1u) {
            r = base + lanes_below(same);
            in = false;
        }
    }
    return in ? atomicAdd(&cnt[k], 1u) : r;
}

// First pass over the edges: list and tuple counts, each entry's place in its list (arrival
// order), and the seeds -- the edges that fit pattern edge order[0]: its arity, and its repeated
// variables (match_core.hpp:32-49) -- as one bit per edge and a count per workgroup. Bound by the
// latency of the counters' atomics, one edge per thread. A triangle join over 200,000 binary edges:
// 35 us here, 19 in the place pass and 14 in the order pass, 79 us with the scan; a histogram with
// stable sorts of the (list, edge) and (tuple key, edge) pairs and a compaction of the seeds took
// 45 launches and about 380 us.
__global__ __launch_bounds__(BJ_THREADS) void k_bj_count(BJView v, BJIndex x) {
    __shared__ uint32_t wn[BJ_WAVES];
    const uint32_t e = blockIdx.x * BJ_THREADS + threadIdx.x;
    const uint32_t lane = lane_id(), w = threadIdx.x / WAVE;
    bool seed = false;
    const bool edge = e < v.m;
    const uint32_t a = edge ? v.ar[e] : 0u;
    const uint32_t* ve = v.ev + (size_t)(edge ? e : 0u) * v.A;
    for (uint32_t u = 0; u < v.U; ++u) {                  // every lane: bj_add works across the wave
        const bool in = edge && bj_listed(v, u, a);
        const uint32_t r = bj_add(x.cnt, in ? (uint64_t)ve[v.upos[u]] * v.U + u : 0ull, in);
        if (in) x.rank[(size_t)e * v.U + u] = r;
    }
    if (v.full) {
        const bool in = edge && bj_tabled(v, a);
        uint32_t h = 0;
        if (in) {
            const uint64_t key = tuple_key(a, [&](uint32_t i) { return ve[i]; });
            const uint32_t tag = tuple_tag(key);
            h = (uint32_t)key & v.tmask;
            for (;;) {                                    // the table has twice the edges' places
                uint32_t was = __hip_atomic_load(&x.tslot[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (was == 0) was = atomicCAS(&x.tslot[h], 0u, tag);
                if (was == 0 || was == tag) break;
                h = (h + 1) & v.tmask;
            }
            x.tplace[e] = h;
        }
        const uint32_t r = bj_add(x.cnt, x.tcnt0 + h, in);
        if (in) x.trank[e] = r;
    }
    if (edge) {
        const DRule& R = v.R;
        const uint32_t p = R.order[0];
        seed = a == R.la[p];
        for (uint32_t i = 0; seed && i < a; ++i) {
            const uint32_t s = R.jsrc[0][i];
            if (s != 0xFFu) seed = ve[i] == ve[s & 15u];
        }
    }
    const uint64_t bal = __ballot(seed);
    if (lane == 0) {
        if (e < v.m) x.smask[e / WAVE] = bal;
        wn[w] = (uint32_t)__popcll(bal);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t n = 0;
        for (uint32_t k = 0; k < BJ_WAVES; ++k) n += wn[k];
        x.cnt[x.scnt0 + blockIdx.x] = n;
    }
}

// Second pass, over the scanned counts: the entries to their lists in arrival order (a list of one
// is done), or (SORT) the (list, edge) pairs a stable sort orders; the seeds in edge order; the
// longest list, and the lists too long to order by counting. Bound by its scattered reads and
// writes.
template <bool SORT>
__global__ __launch_bounds__(BJ_THREADS) void k_bj_place_index(BJView v, BJIndex x) {
    __shared__ uint32_t wmax[2 * BJ_WAVES];
    const uint32_t e = blockIdx.x * BJ_THREADS + threadIdx.x;
    const uint32_t lane = lane_id(), w = threadIdx.x / WAVE;
    uint32_t longest = 0, tuples = 0;
    if (e < v.m) {
        const uint32_t a = v.ar[e];
        auto entry = [&](uint32_t list, uint32_t base, uint32_t n, uint32_t r) {
            if (SORT) return;
            x.un[base + r] = e;
            if (n == 1) x.idx[base] = e;
            if (r == 0 && n > kIndexWave) x.longq[atomicAdd(&x.scal[2], 1u)] = list;
        };
        for (uint32_t u = 0; u < v.U; ++u) {
            const size_t s = (size_t)e * v.U + u;
            const bool in = bj_listed(v, u, a);
            const uint32_t list = in ? v.ev[(size_t)e * v.A + v.upos[u]] * v.U + u : x.nkeys;
            if (in) {
                const uint32_t lo = v.off[list], n = v.off[list + 1] - lo, r = x.rank[s];
                if (r == 0) longest = n > longest ? n : longest;
                entry(list, lo, n, r);
            }
            if (SORT) { x.rank[s] = list; x.un[s] = e; }
        }
        const bool in = bj_tabled(v, a);
        if (in && !SORT) {
            const uint32_t h = x.tplace[e], lo = v.toff[h] - v.toff[0];
            tuples = v.toff[h + 1] - v.toff[h];
            entry(x.nkeys + 1 + h, x.tbase + lo, tuples, x.trank[e]);
        }
        if (SORT && v.full) {
            if (!in) x.tplace[e] = v.tmask + 1;
            x.un[x.tbase + e] = e;
        }
        const uint64_t sm = x.smask[e / WAVE];
        if ((sm >> lane) & 1u) {
            uint32_t o = v.off[x.scnt0 + blockIdx.x] - v.off[x.scnt0] + lanes_below(sm);
            for (uint32_t k = 0; k < w; ++k) o += (uint32_t)__popcll(x.smask[e / WAVE - w + k]);
            x.seeds[o] = e;
        }
    }
    longest = wave_max_u32(longest);
    tuples = wave_max_u32(tuples);
    if (lane == 0) { wmax[w] = longest; wmax[BJ_WAVES + w] = tuples; }
    __syncthreads();
    if (threadIdx.x < 2) {                                // (few workgroups raise a maximum)
        uint32_t most = 0;
        for (uint32_t k = 0; k < BJ_WAVES; ++k) {
            const uint32_t y = wmax[threadIdx.x * BJ_WAVES + k];
            most = y > most ? y : most;
        }
        uint32_t* to = &x.scal[threadIdx.x ? 3 : 1];
        if (most > __hip_atomic_load(to, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(to, most);
        if (blockIdx.x == 0 && threadIdx.x == 0) x.scal[0] = v.off[x.scnt0 + gridDim.x] - v.off[x.scnt0];
    }
}

// Third pass: an entry's place in its list is the number of smaller edges there. At most
// kIndexShort reads per entry, from the cache lines its neighbours read too.
__global__ __launch_bounds__(BJ_THREADS) void k_bj_order(BJView v, BJIndex x) {
    const uint32_t e = blockIdx.x * BJ_THREADS + threadIdx.x;
    if (e >= v.m) return;
    const uint32_t a = v.ar[e];
    auto place = [&](uint32_t base, uint32_t n) {
        if (n < 2 || n > kIndexShort) return;
        uint32_t below = 0;
#pragma unroll 4
        for (uint32_t i = 0; i < n; ++i) below += x.un[base + i] < e ? 1u : 0u;
        x.idx[base + below] = e;
    };
    for (uint32_t u = 0; u < v.U; ++u) {
        if (!bj_listed(v, u, a)) continue;
        const uint32_t list = v.ev[(size_t)e * v.A + v.upos[u]] * v.U + u, lo = v.off[list];
        place(lo, v.off[list + 1] - lo);
    }
    if (bj_tabled(v, a)) {
        const uint32_t h = x.tplace[e];
        place(x.tbase + v.toff[h] - v.toff[0], v.toff[h + 1] - v.toff[h]);
    }
}

// Lists of more than kIndexShort and at most kIndexWave entries, a wave each: the list in LDS, an
// entry's place again the smaller edges there, four a read. Lists of 240 in a state of 1 million
// edges: 0.31 ms the whole join; 0.63 with k_bj_order reading them from memory for each entry.
__global__ __launch_bounds__(BJ_THREADS) void k_bj_order_wave(BJView v, BJIndex x, uint64_t lists) {
    __shared__ __align__(16) uint32_t buf[BJ_WAVES][kIndexWave];
    const uint32_t lane = lane_id();
    uint32_t* own = buf[threadIdx.x / WAVE];
    // neighbouring lists to different waves, so few long ones still spread over the chip
    const uint64_t waves = (uint64_t)gridDim.x * BJ_WAVES;
    for (uint64_t g = (uint64_t)blockIdx.x * BJ_WAVES + threadIdx.x / WAVE; g < lists; g += waves * WAVE) {
        const uint64_t i = g + lane * waves;
        uint32_t lo = 0, n = 0;
        if (i < lists) {
            const uint64_t list = i < x.nkeys ? i : i + 1;
            lo = i < x.nkeys ? v.off[list] : x.tbase + v.off[list] - v.toff[0];
            n = v.off[list + 1] - v.off[list];
        }
        for (uint64_t todo = __ballot(n > kIndexShort && n <= kIndexWave); todo; todo &= todo - 1) {
            const int l = __builtin_ctzll(todo);
            const uint32_t at = (uint32_t)__builtin_amdgcn_readlane((int)lo, l);
            const uint32_t len = (uint32_t)__builtin_amdgcn_readlane((int)n, l);
            for (uint32_t j = lane; j < ((len + 3) & ~3u); j += WAVE) own[j] = j < len ? x.un[at + j] : 0xFFFFFFFFu;
            wave_sync();
            for (uint32_t j = lane; j < len; j += WAVE) {
                const uint32_t e = own[j];
                uint32_t below = 0;
                for (uint32_t k = 0; k < len; k += 4) {
                    const uint4 y = *(const uint4*)(own + k);
                    below += (y.x < e ? 1u : 0u) + (y.y < e ? 1u : 0u) + (y.z < e ? 1u : 0u) + (y.w < e ? 1u : 0u);
                }
                x.idx[at + below] = e;
            }
            wave_sync();
        }
    }
}

// The long lists, a workgroup each: their edges as a bit set over all edges in LDS (words of 32),
// read back in order. At most kIndexPlaceEdges edges, so the set fits 128 KB.
__global__ __launch_bounds__(1024) void k_bj_order_long(BJView v, BJIndex x, uint32_t n_long) {
    extern __shared__ uint8_t lds[];
    uint32_t* set = (uint32_t*)lds;
    __shared__ uint32_t wn[16];
    const uint32_t tid = threadIdx.x, lane = lane_id(), w = tid / WAVE;
    const uint32_t words = (v.m + 31) / 32, per = (words + 15) / 16;      // a wave's share
    const uint32_t b = w * per < words ? w * per : words, e = b + per < words ? b + per : words;
    for (uint32_t q = blockIdx.x; q < n_long; q += gridDim.x) {
        const uint32_t list = x.longq[q];
        const uint32_t lo = list < x.nkeys ? v.off[list] : x.tbase + v.off[list] - v.toff[0];
        const uint32_t n = v.off[list + 1] - v.off[list];
        for (uint32_t i = tid; i < words; i += 1024) set[i] = 0;
        __syncthreads();
        for (uint32_t i = tid; i < n; i += 1024) {
            const uint32_t y = x.un[lo + i];
            atomicOr(&set[y >> 5], 1u << (y & 31u));
        }
        __syncthreads();
        uint32_t c = 0;
        for (uint32_t i = b + lane; i < e; i += WAVE) c += (uint32_t)__popc(set[i]);
        c = wave_sum_u32(c);
        if (lane == 0) wn[w] = c;
        __syncthreads();
        uint32_t o = lo;
        for (uint32_t k = 0; k < w; ++k) o += wn[k];
        for (uint32_t i0 = b; i0 < e; i0 += WAVE) {
            const uint32_t i = i0 + lane;
            uint32_t s = i < e ? set[i] : 0u;
            const uint32_t inc = wave_incl_scan_u32((uint32_t)__popc(s));
            uint32_t at = o + inc - (uint32_t)__popc(s);
            for (; s; s &= s - 1) x.idx[at++] = i * 32 + (uint32_t)__ffs((int)s) - 1;
            o += (uint32_t)__builtin_amdgcn_readlane((int)inc, WAVE - 1);
        }
        __syncthreads();
    }
}

// ---- join --------------------------------------------------------------------------------

// The edges with a vertex tuple: where their list begins in tidx, and how many.
__device__ __forceinline__ uint32_t bj_find(const BJView& v, uint64_t key, uint32_t& lo) {
    const uint32_t tag = tuple_tag(key);
    uint32_t h = (uint32_t)key & v.tmask;
    for (;;) {                                            // the table has empty places
        const uint32_t s = v.tslot[h];
        if (s == tag) { lo = v.toff[h] - v.toff[0]; return v.toff[h + 1] - v.toff[h]; }
        if (s == 0) return 0;
        h = (h + 1) & v.tmask;
    }
}

// Candidate list of each partial of depth d: [lo, lo + cnt) of the pivot vertex's CSR list, of the
// tuple index for a closing edge, or every edge when pattern edge order[d] shares no bound
// variable. cnt[P] = 0 ends the scan's input.
__global__ void k_bj_range(BJView v, uint32_t d, const uint32_t* F, uint64_t P, uint32_t* lo, uint32_t* cnt) {
    const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q > P) return;
    if (q == P) { cnt[q] = 0; return; }
    const DRule& R = v.R;
    const uint32_t pv = R.piv[d];
    auto vertex = [&](uint32_t i) {                       // bound at an earlier depth
        const uint32_t s = R.jsrc[d][i];
        return v.ev[(size_t)F[q * d + (s >> 4)] * v.A + (s & 15u)];
    };
    uint32_t l = 0, n = v.m;
    if ((v.full >> d) & 1u) {
        n = bj_find(v, tuple_key(R.la[R.order[d]], vertex), l);
    } else if (pv != 0xFFu) {
        const uint32_t key = vertex(pv) * v.U + v.dpos[d];
        l = v.off[key];
        n = v.off[key + 1] - l;
    }
    lo[q] = l;
    cnt[q] = n;
}

// Last q in [a, b) with start[q] <= t, given start[a] <= t < start[b].
__device__ __forceinline__ uint64_t bj_owner(const uint64_t* start, uint64_t a, uint64_t b, uint64_t t) {
    while (b - a > 1) {
        const uint64_t mid = (a + b) >> 1;
        if (start[mid] <= t) a = mid; else b = mid;
    }
    return a;
}
// The same over start[0..P] by a whole wave, 64 probes a round.
__device__ __forceinline__ uint64_t bj_owner_wave(const uint64_t* start, uint64_t P, uint64_t t) {
    const uint32_t lane = lane_id();
    uint64_t a = 0, b = P;
    while (b - a > 1) {
        const uint64_t step = (b - a + WAVE - 1) / WAVE, p = a + step * lane;
        const uint64_t in = __ballot(lane == 0 || (p < b && start[p] <= t));
        a += step * (uint64_t)(__popcll(in) - 1);
        b = a + step < b ? a + step : b;
    }
    return a;
}

struct BJLevel {
    uint32_t d;               // depth being added (1 .. n-1)
    uint32_t turn;            // which of found[0..1] holds the matches before this call
    const uint32_t* F;        // [P * d] partials, join order
    uint64_t P;
    const uint32_t* lo;       // [P]
    const uint64_t* start;    // [P + 1] scan of the list lengths; start[P] = items (device)
    uint64_t ntiles;          // tiles provisioned: an upper bound of the items' tiles
    uint64_t* tile_cnt;       // [ntiles + 1] survivors per tile (the last 0)
    const uint64_t* tile_off; // [ntiles + 1] their scan
    uint64_t* tile_q;         // [2 * ntiles] a tile's first and last partial
    uint64_t* mask;           // [ntiles * BJ_WORDS] one bit per item: it survives
    uint32_t* Fn;             // inner depth: the next frontier [S * (d+1)]
    uint32_t* out;            // last depth: matches, n_lhs edges each in pattern order
    uint64_t cap;             //   (room for cap matches in all)
    uint64_t* found;          // [3] device: matches, by turns, and algorithmic bytes
};

// Bookkeeping of a depth: the matches found (by turns: other workgroups still read the old count),
// and the algorithmic bytes (the candidate reads of every item, the partials' lists, the frontier
// or the matches written).
__device__ __forceinline__ void bj_tally(const BJView& v, const BJLevel& L, bool last) {
    const uint64_t s = L.tile_off[L.ntiles], t = L.start[L.P];
    const uint32_t n = v.R.n_lhs, a = v.R.la[v.R.order[L.d]];
    uint64_t bytes = t * 4ull * (1ull + a) + L.P * (4ull * L.d + 12ull);
    if (last) {
        const uint64_t before = L.found[L.turn];
        const uint64_t cap = L.out ? L.cap : 0, room = cap > before ? cap - before : 0;
        bytes += (s < room ? s : room) * 4ull * n;
        L.found[L.turn ^ 1u] = before + s;
    } else {
        bytes += s * 4ull * (L.d + 1);
    }
    L.found[2] += bytes;
}
__global__ void k_bj_tally(BJView v, BJLevel L) { bj_tally(v, L, true); }

// A tile's view of its items in LDS. A set bit of `bits` begins the (nonempty) list of the next
// partial, so item i belongs to list number popcount(bits up to i) - 1: no search per item.
struct BJTile {
    uint64_t bits[BJ_WORDS];
    uint64_t sum[BJ_WORDS + 1];
    uint64_t q[2];
    uint32_t pre[BJ_WORDS + 1];
    uint32_t cofs[BJ_TILE];           // per list: candidate of the tile's item i at cofs + i
    uint32_t word[BJ_STAGE_W];        // per list: bj_word of its partial
    uint16_t ci[BJ_TILE];             // per list: its partial, from the tile's first
};
struct BJStaged { bool lists, words; uint32_t per; };

// Word k of partial q at depth d: its d edges, then the vertex each slot of pattern edge order[d]
// must carry, then (a closing edge follows) of order[d + 1]; 0 where no earlier depth binds it.
__device__ __forceinline__ uint32_t bj_word(const BJView& v, const BJLevel& L, uint64_t q, uint32_t k) {
    const uint32_t d = L.d;
    const uint32_t* part = L.F + q * d;
    if (k < d) return part[k];
    k -= d;
    uint32_t at = d;
    const uint32_t pa = v.R.la[v.R.order[d]];
    if (k >= pa) { k -= pa; at = d + 1; }
    const uint32_t s = v.R.jsrc[at][k];
    if (s == 0xFFu || (s >> 4) >= d) return 0;
    return v.ev[(size_t)part[s >> 4] * v.A + (s & 15u)];
}

// The lists of partials [q0, q0 + nq) over the tile's items [t0, ..) into LDS, when they fit.
template <bool CLOSE>
__device__ __forceinline__ BJStaged bj_stage(const BJView& v, const BJLevel& L, BJTile& S, uint64_t t0, uint64_t q0,
                                             uint64_t nq) {
    const uint32_t tid = threadIdx.x;
    const uint32_t per = L.d + v.R.la[v.R.order[L.d]] + (CLOSE ? (uint32_t)v.R.la[v.R.order[L.d + 1]] : 0u);
    if (nq > BJ_STAGE_Q) return BJStaged{false, false, per};
    if (tid < BJ_WORDS) S.bits[tid] = 0;
    __syncthreads();
    for (uint32_t i = tid; i < (uint32_t)nq; i += BJ_THREADS) {
        const uint64_t s = L.start[q0 + i];
        if (L.start[q0 + i + 1] == s) continue;
        const uint32_t at = s > t0 ? (uint32_t)(s - t0) : 0u;
        atomicOr((unsigned long long*)&S.bits[at / WAVE], 1ull << (at % WAVE));
    }
    __syncthreads();
    if (tid < WAVE) {
        const uint32_t c = tid < BJ_WORDS ? (uint32_t)__popcll(S.bits[tid]) : 0u;
        const uint32_t inc = wave_incl_scan_u32(c);
        if (tid < BJ_WORDS) S.pre[tid + 1] = inc;
        if (tid == 0) S.pre[0] = 0;
    }
    __syncthreads();
    for (uint32_t i = tid; i < (uint32_t)nq; i += BJ_THREADS) {
        const uint64_t s = L.start[q0 + i];
        if (L.start[q0 + i + 1] == s) continue;
        const uint32_t at = s > t0 ? (uint32_t)(s - t0) : 0u;
        const uint32_t r = S.pre[at / WAVE] + (uint32_t)__popcll(S.bits[at / WAVE] & ((1ull << (at % WAVE)) - 1ull));
        S.ci[r] = (uint16_t)i;
        S.cofs[r] = L.lo[q0 + i] + (uint32_t)(t0 - s);
    }
    __syncthreads();
    const uint32_t words = S.pre[BJ_WORDS] * per;
    if (words > BJ_STAGE_W) return BJStaged{true, false, per};
    for (uint32_t i = tid; i < words; i += BJ_THREADS) S.word[i] = bj_word(v, L, q0 + S.ci[i / per], i % per);
    __syncthreads();
    return BJStaged{true, true, per};
}

// One item: its partial, where the partial's words begin in BJTile::word (or kNotStaged), its
// candidate.
constexpr uint32_t kNotStaged = 0xFFFFFFFFu;
struct BJItem {
    uint64_t q;
    uint32_t w, e;
};
__device__ __forceinline__ uint32_t bj_word(const BJView& v, const BJLevel& L, const BJTile& S, const BJItem& it,
                                            uint32_t k) {
    return it.w != kNotStaged ? S.word[it.w + k] : bj_word(v, L, it.q, k);
}
template <bool CLOSE>
__device__ __forceinline__ BJItem bj_item(const BJView& v, const BJLevel& L, const BJTile& S, const BJStaged st,
                                          uint64_t t0, uint32_t i) {
    BJItem it;
    uint32_t c;
    it.w = kNotStaged;
    if (st.lists) {
        const uint32_t k = i / WAVE;
        const uint32_t r = S.pre[k] + (uint32_t)__popcll(S.bits[k] & (~0ull >> (63u - i % WAVE))) - 1u;
        it.q = S.q[0] + S.ci[r];
        c = S.cofs[r] + i;
        if (st.words) it.w = r * st.per;
    } else {
        it.q = bj_owner(L.start, S.q[0], S.q[1] + 1, t0 + i);
        c = L.lo[it.q] + (uint32_t)(t0 + i - L.start[it.q]);
    }
    const uint32_t d = L.d;
    it.e = (v.full >> d) & 1u ? v.tidx[c] : v.R.piv[d] == 0xFFu ? c : v.idx[c];
    return it;
}

// Whether an item's candidate fits: it has the arity, is not already in the partial
// (edge-injective) and agrees with every binding the partial and its own earlier slots fixed
// (vertex-non-injective: distinct variables may share a vertex). v.chk[d] holds the slots with
// something to compare -- a pivot's list holds it already -- and bit d of v.chk_ar whether the
// candidate's arity is not the list's own.
__device__ __forceinline__ bool bj_fits(const BJView& v, const BJLevel& L, const BJTile& S, const BJItem& it) {
    const DRule& R = v.R;
    const uint32_t d = L.d;
    auto word = [&](uint32_t k) { return bj_word(v, L, S, it, k); };
    if (((v.chk_ar >> d) & 1u) && v.ar[it.e] != R.la[R.order[d]]) return false;
    for (uint32_t k = 0; k < d; ++k)
        if (word(k) == it.e) return false;
    const uint32_t* x = v.ev + (size_t)it.e * v.A;
    for (uint32_t c = v.chk[d]; c; c &= c - 1) {
        const uint32_t i = (uint32_t)__builtin_ctz(c), s = R.jsrc[d][i];
        if (x[i] != ((s >> 4) < d ? word(d + i) : x[s & 15u])) return false;
    }
    return true;
}

// The closing edges of an item that fits: their list, and (bj_closes) whether one of it fits.
__device__ __forceinline__ uint32_t bj_closing(const BJView& v, const BJLevel& L, const BJTile& S, const BJItem& it,
                                               uint32_t& lo) {
    const DRule& R = v.R;
    const uint32_t d = L.d, pa = R.la[R.order[d]], a = R.la[R.order[d + 1]];
    const uint32_t* x = v.ev + (size_t)it.e * v.A;
    return bj_find(v, tuple_key(a, [&](uint32_t i) {
        const uint32_t s = R.jsrc[d + 1][i];
        return (s >> 4) == d ? x[s & 15u] : bj_word(v, L, S, it, d + pa + i);
    }), lo);
}
__device__ __forceinline__ bool bj_closes(const BJView& v, const BJLevel& L, const BJTile& S, const BJItem& it,
                                          uint32_t c) {
    const DRule& R = v.R;
    const uint32_t d = L.d, pa = R.la[R.order[d]], a = R.la[R.order[d + 1]];
    auto word = [&](uint32_t k) { return bj_word(v, L, S, it, k); };
    if (c == it.e || v.ar[c] != a) return false;
    for (uint32_t k = 0; k < d; ++k)
        if (word(k) == c) return false;
    for (uint32_t i = 0; i < a; ++i) {
        const uint32_t s = R.jsrc[d + 1][i];
        const uint32_t want = (s >> 4) == d ? v.ev[(size_t)it.e * v.A + (s & 15u)] : word(d + pa + i);
        if (v.ev[(size_t)c * v.A + i] != want) return false;
    }
    return true;
}

// Test pass over the items of a depth, a tile per workgroup iteration: one bit per item and the
// survivors of each tile (with CLOSE, the matches the survivors' closing edges make). The number
// of items is read on the device (the scan's total), so no host round trip sizes the launch;
// tiles past it count zero. Bound by the latency of the candidate reads (and, with CLOSE, of the
// candidate's vertices and the table), so tiles are small to keep many waves in flight. The
// triangles of 200,000 edges over 20,000 vertices (2 million items): 65 us with the closing edge
// looked up here; a frontier of all 2 million wedges, in two halves for a scratch that does not
// hold it, its candidate lists and their scan took 400 us. 250,000 items of a ternary wedge: 10.7
// us, with one bit per item; three searches per item and slots for 16 survivors a tile, then a
// second pass over the tiles with more, took 33 and 28.
template <bool CLOSE>
__global__ __launch_bounds__(BJ_THREADS) void k_bj_test(BJView v, BJLevel L) {
    __shared__ BJTile S;
    const uint32_t tid = threadIdx.x, lane = lane_id(), w = tid / WAVE;
    const uint64_t T = L.start[L.P];
    if (blockIdx.x == 0 && tid == 0) L.tile_cnt[L.ntiles] = 0;
    for (uint64_t tile = blockIdx.x; tile < L.ntiles; tile += gridDim.x) {
        const uint64_t t0 = tile * BJ_TILE;
        if (t0 >= T) {                                    // the same for the whole workgroup
            if (tid == 0) L.tile_cnt[tile] = 0;
            continue;
        }
        const uint64_t t1 = t0 + BJ_TILE < T ? t0 + BJ_TILE : T;
        if (w < 2) {
            const uint64_t q = bj_owner_wave(L.start, L.P, w ? t1 - 1 : t0);
            if (lane == 0) { S.q[w] = q; L.tile_q[2 * tile + w] = q; }
        }
        __syncthreads();
        const uint64_t q0 = S.q[0];
        const BJStaged st = bj_stage<CLOSE>(v, L, S, t0, q0, S.q[1] - q0 + 1);
        const uint32_t n = (uint32_t)(t1 - t0);
        uint64_t found = 0;
        BJItem it[BJ_IPT];                                // the candidates' reads in flight together
#pragma unroll
        for (uint32_t k = 0; k < BJ_IPT; ++k) {
            const uint32_t i = k * BJ_THREADS + tid;
            it[k] = bj_item<CLOSE>(v, L, S, st, t0, i < n ? i : n - 1);
        }
#pragma unroll
        for (uint32_t k = 0; k < BJ_IPT; ++k) {
            bool ok = k * BJ_THREADS + tid < n && bj_fits(v, L, S, it[k]);
            if (CLOSE && ok) {
                uint32_t lo = 0, c = 0;
                const uint32_t len = bj_closing(v, L, S, it[k], lo);
                for (uint32_t j = 0; j < len; ++j) c += bj_closes(v, L, S, it[k], v.tidx[lo + j]) ? 1u : 0u;
                ok = c != 0;
                found += c;
            }
            const uint64_t bal = __ballot(ok);
            if (lane == 0) {
                L.mask[tile * BJ_WORDS + k * BJ_WAVES + w] = bal;
                if (!CLOSE) found += (uint64_t)__popcll(bal);
            }
        }
        if (CLOSE) found = wave_sum_u64(found);
        if (lane == 0) S.sum[w] = found;
        __syncthreads();
        if (tid == 0) {
            uint64_t s = 0;
            for (uint32_t k = 0; k < BJ_WAVES; ++k) s += S.sum[k];
            L.tile_cnt[tile] = s;
        }
        __syncthreads();
    }
}

// Place pass: the surviving items of each tile, in item order, to the next frontier or (LAST) the
// match list. A tile with few survivors finds their partials by a search, without staging. Bound by
// the latency of that chain (9 us for 250,000 survivors, 30 for 1,000 triangles in as many tiles).
template <bool LAST, bool CLOSE>
__global__ __launch_bounds__(BJ_THREADS) void k_bj_place(BJView v, BJLevel L) {
    __shared__ BJTile S;
    const uint32_t tid = threadIdx.x, lane = lane_id(), w = tid / WAVE;
    const uint32_t d = L.d, n = v.R.n_lhs;
    const uint64_t base = LAST ? L.found[L.turn] : 0;
    for (uint64_t tile = blockIdx.x; tile < L.ntiles; tile += gridDim.x) {
        const uint64_t off = base + L.tile_off[tile];
        if (L.tile_cnt[tile] == 0 || (LAST && off >= L.cap)) continue;    // (the whole workgroup)
        const uint64_t t0 = tile * BJ_TILE;
        const uint64_t* mask = L.mask + tile * BJ_WORDS;
        if (tid < WAVE) {
            const uint64_t c = tid < BJ_WORDS ? (uint64_t)__popcll(mask[tid]) : 0ull;
            const uint64_t inc = wave_incl_scan_u64(c);
            if (tid < BJ_WORDS) S.sum[tid + 1] = inc;
            if (tid == 0) S.sum[0] = 0;
            if (tid < 2) S.q[tid] = L.tile_q[2 * tile + tid];
        }
        __syncthreads();
        const uint64_t q0 = S.q[0];
        BJStaged st{false, false, 0};
        if (S.sum[BJ_WORDS] > BJ_TILE / 16) st = bj_stage<CLOSE>(v, L, S, t0, q0, S.q[1] - q0 + 1);
        uint64_t before[BJ_IPT];                          // CLOSE: matches of the wave's earlier items,
        BJItem item[BJ_IPT];                              //   the items,
        uint32_t first[BJ_IPT], len[BJ_IPT];              //   their closing edges
        if (CLOSE) {
#pragma unroll
            for (uint32_t k = 0; k < BJ_IPT; ++k) {
                const uint32_t i = k * BJ_THREADS + tid;
                uint32_t c = 0;
                first[k] = len[k] = 0;
                if ((mask[k * BJ_WAVES + w] >> lane) & 1u) {
                    item[k] = bj_item<CLOSE>(v, L, S, st, t0, i);
                    len[k] = bj_closing(v, L, S, item[k], first[k]);
                    for (uint32_t j = 0; j < len[k]; ++j)
                        c += bj_closes(v, L, S, item[k], v.tidx[first[k] + j]) ? 1u : 0u;
                }
                const uint64_t inc = wave_incl_scan_u64((uint64_t)c);
                before[k] = inc - c;
                if (k == 0) __syncthreads();              // every wave has read the survivors' sums
                if (lane == WAVE - 1) S.sum[k * BJ_WAVES + w + 1] = inc;
            }
            __syncthreads();
            if (tid < WAVE) {
                const uint64_t inc = wave_incl_scan_u64(tid < BJ_WORDS ? S.sum[tid + 1] : 0ull);
                if (tid < BJ_WORDS) S.sum[tid + 1] = inc;
            }
            __syncthreads();
        }
#pragma unroll
        for (uint32_t k = 0; k < BJ_IPT; ++k) {
            const uint32_t i = k * BJ_THREADS + tid;
            const uint64_t m = mask[k * BJ_WAVES + w];
            if (!((m >> lane) & 1u)) continue;
            const BJItem it = CLOSE ? item[k] : bj_item<CLOSE>(v, L, S, st, t0, i);
            auto word = [&](uint32_t x) { return bj_word(v, L, S, it, x); };
            uint64_t g = off + S.sum[k * BJ_WAVES + w] + (CLOSE ? before[k] : (uint64_t)lanes_below(m));
            if (CLOSE) {
                for (uint32_t j = 0; j < len[k]; ++j) {
                    const uint32_t c = v.tidx[first[k] + j];
                    if (!bj_closes(v, L, S, it, c)) continue;
                    if (g >= L.cap) break;
                    uint32_t* o = L.out + g * n;
                    for (uint32_t x = 0; x < d; ++x) o[v.R.order[x]] = word(x);
                    o[v.R.order[d]] = it.e;
                    o[v.R.order[d + 1]] = c;
                    ++g;
                }
            } else if (LAST) {
                if (g >= L.cap) continue;
                uint32_t* o = L.out + g * n;
                for (uint32_t x = 0; x < d; ++x) o[v.R.order[x]] = word(x);
                o[v.R.order[d]] = it.e;
            } else {
                uint32_t* o = L.Fn + g * (d + 1);
                for (uint32_t x = 0; x < d; ++x) o[x] = word(x);
                o[d] = it.e;
            }
        }
        __syncthreads();
    }
    if (blockIdx.x == 0 && tid == 0) bj_tally(v, L, LAST);
}

}  // namespace hgx

namespace hgx {

struct BJCast64 {
    __host__ __device__ uint64_t operator()(uint32_t x) const { return x; }
};

template <class T>
static T* bget(BJMem& m, size_t n) { return (T*)m.get(sizeof(T) * (n ? n : 1)); }

template <class T>
static T read1(const T* d, hipStream_t st) {
    T x{};
    HIP_TRY(hipMemcpyAsync(&x, d, sizeof(T), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    return x;
}

// exclusive sums over n + 1 entries (the last input zero): out[n] is the total
template <class In, class Out>
static void bj_scan_of(BJMem& m, In in, Out* out, uint64_t n, hipStream_t st) {
    if (n + 1 > 0x7FFFFFFFull) throw Error{HGX_ERR_UNSUPPORTED, "join scan above 2^31 entries"};
    size_t tmp = 0;
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, in, out, (int)(n + 1), st));
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(m.get(tmp), tmp, in, out, (int)(n + 1), st));
}
static void bj_scan(BJMem& m, const uint32_t* in, uint64_t* out, uint64_t n, hipStream_t st) {
    bj_scan_of(m, hipcub::TransformInputIterator<uint64_t, BJCast64, const uint32_t*>(in, BJCast64()), out, n, st);
}

static uint32_t blocks_for(uint64_t n, uint32_t threads) { return (uint32_t)std::max<uint64_t>(1, (n + threads - 1) / threads); }

// Which positions the join pivots on, which depths close, and what each depth compares.
static void bj_plan(BJView& v) {
    const DRule& R = v.R;
    v.U = 0;
    v.full = v.tar = v.chk_ar = 0;
    for (uint32_t d = 1; d < R.n_lhs; ++d) {
        const uint32_t a = R.la[R.order[d]], pv = R.piv[d];
        bool all = true;                                  // every slot bound by earlier depths
        v.chk[d] = 0;
        for (uint32_t i = 0; i < a; ++i) {
            const uint32_t s = R.jsrc[d][i];
            all &= s != 0xFFu && (s >> 4) < d;
            if (s != 0xFFu) v.chk[d] |= 1u << i;
        }
        if (all) {
            v.full |= 1u << d;
            v.tar |= 1u << a;
            v.chk_ar |= 1u << d;
            continue;
        }
        if (pv == 0xFFu) { v.chk_ar |= 1u << d; continue; }
        v.chk[d] &= ~(1u << pv);
        uint32_t u = 0;
        while (u < v.U && v.upos[u] != pv) ++u;
        if (u == v.U) { v.upos[v.U++] = (uint8_t)pv; v.uar[u] = 0; }
        v.uar[u] |= 1u << a;
        v.dpos[d] = (uint8_t)u;
    }
    for (uint32_t d = 1; d < R.n_lhs; ++d)                // a list of several arities
        if (!((v.chk_ar >> d) & 1u) && (v.uar[v.dpos[d]] & (v.uar[v.dpos[d]] - 1u))) v.chk_ar |= 1u << d;
}

// The index of a state held on the device as ev [m * A], ar [m], vertex ids below nv, and the
// seeds. One read back: the seeds and the longest list.
static void bj_index(BJRun& J, uint32_t nv, uint64_t* n_seeds, uint32_t** seeds, hipEvent_t built) {
    BJMem& mem = *J.mem;
    BJView& v = J.v;
    hipStream_t st = J.st;
    const uint32_t m = v.m;
    if ((uint64_t)nv * v.A >= 0xFFFFFFF0ull || (uint64_t)m * v.A >= 0x7FFFFFF0ull)
        throw Error{HGX_ERR_UNSUPPORTED, "index above 2^31 vertex slots"};
    bj_plan(v);
    if (!m) v.full = v.tar = 0;
    const bool sort = m > kIndexPlaceEdges;
    const uint64_t nkeys = (uint64_t)nv * v.U, slots = (uint64_t)m * v.U, tm = v.full ? m : 0;
    uint64_t tcap = 0;
    if (v.full)
        for (tcap = 1; tcap < 2ull * m; tcap <<= 1) {}    // load factor <= 1/2
    v.tmask = (uint32_t)(tcap - 1);
    const uint32_t blocks = blocks_for(m, BJ_THREADS);
    BJIndex x{};
    x.nkeys = (uint32_t)nkeys;
    x.tcnt0 = nkeys + 1;
    x.scnt0 = x.tcnt0 + (v.full ? tcap + 1 : 0);
    const uint64_t ncnt = x.scnt0 + blocks + 1;
    // one zeroed region: matches by turns and bytes, scalars, counts, the tuple table
    const uint64_t zeroed = 6 + 4 + ncnt + tcap;
    uint32_t* z = bget<uint32_t>(mem, zeroed);
    J.acc = (uint64_t*)z;
    x.scal = z + 6;
    x.cnt = x.scal + 4;
    x.tslot = x.cnt + ncnt;
    uint32_t* off = bget<uint32_t>(mem, ncnt);
    x.rank = bget<uint32_t>(mem, slots);
    x.un = bget<uint32_t>(mem, slots + tm);
    x.idx = bget<uint32_t>(mem, slots + tm);
    x.tbase = (uint32_t)slots;
    x.tplace = bget<uint32_t>(mem, tm);
    x.trank = bget<uint32_t>(mem, tm);
    x.longq = bget<uint32_t>(mem, (slots + tm) / kIndexWave + 1);
    x.smask = bget<uint64_t>(mem, ((uint64_t)m + WAVE - 1) / WAVE);
    x.seeds = *seeds = bget<uint32_t>(mem, m);
    v.off = off;
    v.toff = off + x.tcnt0;
    v.idx = x.idx;
    v.tidx = x.idx + slots;
    v.tslot = x.tslot;
    hipLaunchKernelGGL(k_bj_zero, dim3(blocks_for(zeroed, 256)), dim3(256), 0, st, z, zeroed);
    if (m) {
        hipLaunchKernelGGL(k_bj_count, dim3(blocks), dim3(BJ_THREADS), 0, st, v, x);
        if (ncnt <= 0x7FFFFFFFull) {
            bj_scan_of(mem, x.cnt, off, ncnt - 1, st);
        } else {                                          // readers take differences within a part
            bj_scan_of(mem, x.cnt, off, nkeys, st);
            if (v.full) bj_scan_of(mem, x.cnt + x.tcnt0, off + x.tcnt0, tcap, st);
            bj_scan_of(mem, x.cnt + x.scnt0, off + x.scnt0, blocks, st);
        }
        if (!sort) {
            hipLaunchKernelGGL(k_bj_place_index<false>, dim3(blocks), dim3(BJ_THREADS), 0, st, v, x);
            hipLaunchKernelGGL(k_bj_order, dim3(blocks), dim3(BJ_THREADS), 0, st, v, x);
        } else {
            hipLaunchKernelGGL(k_bj_place_index<true>, dim3(blocks), dim3(BJ_THREADS), 0, st, v, x);
            // keys to kout, edges to idx; keys are at most their largest (the entries in no list)
            auto sorted = [&](const uint32_t* kin, const uint32_t* vin, uint32_t* vout, uint64_t n, uint64_t largest) {
                if (!n) return;
                int bits = 1;
                while (bits < 32 && (largest >> bits) != 0) ++bits;
                uint32_t* kout = bget<uint32_t>(mem, n);
                size_t tmp = 0;
                HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, kin, kout, vin, vout, (int)n, 0, bits, st));
                HIP_TRY(hipcub::DeviceRadixSort::SortPairs(mem.get(tmp), tmp, kin, kout, vin, vout, (int)n, 0, bits, st));
            };
            sorted(x.rank, x.un, x.idx, slots, nkeys);
            sorted(x.tplace, x.un + slots, x.idx + slots, tm, tcap);
        }
        HIP_TRY(hipGetLastError());
    }
    if (built) HIP_TRY(hipEventRecord(built, st));
    uint32_t hs[4] = {0, 0, 0, 0};
    HIP_TRY(hipMemcpyAsync(hs, x.scal, sizeof(hs), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    if (!sort && std::max(hs[1], hs[3]) > kIndexShort) {
        const uint64_t lists = nkeys + tcap;
        hipLaunchKernelGGL(k_bj_order_wave, dim3((uint32_t)std::min<uint64_t>((lists + BJ_WAVES - 1) / BJ_WAVES, J.grid)),
                           dim3(BJ_THREADS), 0, st, v, x, lists);
    }
    if (hs[2])
        hipLaunchKernelGGL(k_bj_order_long, dim3(std::min<uint32_t>(hs[2], J.grid)), dim3(1024), (m + 31) / 32 * 4, st,
                           v, x, hs[2]);
    HIP_TRY(hipGetLastError());
    *n_seeds = hs[0];
    J.maxlist = hs[1];
    // read the state twice, write and read the places, the entries and the offsets
    J.index_bytes += 2ull * m * (4ull * v.A + 1) + (slots + tm) * 4ull * 5 + ncnt * 12ull + tcap * 4ull;
}

// Extends the partials F (P of them, d edges each) by pattern edge order[d], and on to the last
// depth; splits F in two, in order, when the items or the next frontier would outgrow the memory
// at hand. The host learns a depth's survivors only where it must size the next frontier; the
// last depth writes its matches at the device-side running count and leaves the host nothing to
// wait for.
static void bj_depth(BJRun& J, uint32_t d, const uint32_t* F, uint64_t P) {
    BJMem& mem = *J.mem;
    const uint32_t n = J.v.R.n_lhs;
    const bool close = d + 2 == n && ((J.v.full >> (d + 1)) & 1u);
    const bool last = d + 1 == n || close;
    const size_t mk = mem.mark();
    auto halves = [&] {
        mem.rewind(mk);
        bj_depth(J, d, F, P / 2);
        bj_depth(J, d, F + (P / 2) * d, P - P / 2);
    };
    uint32_t* lo = bget<uint32_t>(mem, P);
    uint32_t* cnt = bget<uint32_t>(mem, P + 1);
    uint64_t* start = bget<uint64_t>(mem, P + 1);
    hipLaunchKernelGGL(k_bj_range, dim3(blocks_for(P + 1, 256)), dim3(256), 0, J.st, J.v, d, F, P, lo, cnt);
    bj_scan(mem, cnt, start, P, J.st);
    // tiles to provision: the longest candidate list bounds every partial's; an exact count (one
    // round trip) only when that bound is loose beyond use or too much to hold
    const bool full = (J.v.full >> d) & 1u;
    const uint64_t per = J.v.R.piv[d] == 0xFFu ? (uint64_t)J.v.m : std::max<uint64_t>(1, J.maxlist);
    uint64_t ntiles = (P * per + BJ_TILE - 1) / BJ_TILE;
    // a closing edge has about one candidate per partial: the exact count, not the list bound
    if (full || P * per / std::max<uint64_t>(1, P) != per || ntiles > ((uint64_t)1 << 20) ||
        ntiles * BJ_TILE_BYTES > mem.left() / 2) {
        const uint64_t T = read1(start + P, J.st);
        ntiles = (T + BJ_TILE - 1) / BJ_TILE;
    }
    if (ntiles == 0) { mem.rewind(mk); return; }
    if (P > 1 && ntiles * BJ_TILE_BYTES > mem.left()) { halves(); return; }
    BJLevel L{};
    L.d = d; L.F = F; L.P = P; L.lo = lo; L.start = start; L.ntiles = ntiles;
    L.tile_cnt = bget<uint64_t>(mem, ntiles + 1);
    uint64_t* toff = bget<uint64_t>(mem, ntiles + 1);
    L.tile_off = toff;
    L.tile_q = bget<uint64_t>(mem, 2 * ntiles);
    L.mask = bget<uint64_t>(mem, ntiles * BJ_WORDS);
    L.out = J.out; L.cap = J.cap; L.found = J.acc; L.turn = J.turn;
    const uint32_t grid = (uint32_t)std::min<uint64_t>(ntiles, J.grid);
    if (close) hipLaunchKernelGGL(k_bj_test<true>, dim3(grid), dim3(BJ_THREADS), 0, J.st, J.v, L);
    else hipLaunchKernelGGL(k_bj_test<false>, dim3(grid), dim3(BJ_THREADS), 0, J.st, J.v, L);
    HIP_TRY(hipGetLastError());
    bj_scan_of(mem, (const uint64_t*)L.tile_cnt, toff, ntiles, J.st);
    if (last) {
        if (!J.out) hipLaunchKernelGGL(k_bj_tally, dim3(1), dim3(1), 0, J.st, J.v, L);
        else if (close) hipLaunchKernelGGL((k_bj_place<true, true>), dim3(grid), dim3(BJ_THREADS), 0, J.st, J.v, L);
        else hipLaunchKernelGGL((k_bj_place<true, false>), dim3(grid), dim3(BJ_THREADS), 0, J.st, J.v, L);
        HIP_TRY(hipGetLastError());
        J.turn ^= 1u;
        mem.rewind(mk);
        return;
    }
    const uint64_t S = read1(toff + ntiles, J.st);
    if (S == 0) { mem.rewind(mk); return; }
    // the next frontier, the next depth's lists and scan, and its tiles
    const uint64_t tiles = (S * std::max<uint64_t>(1, J.maxlist) / BJ_TILE + 2) * BJ_TILE_BYTES;
    const uint64_t need = S * (4ull * (d + 1) + 16ull) + std::min<uint64_t>(tiles, mem.room() / 4);
    if (need > mem.room()) {
        if (P == 1) throw Error{HGX_ERR_CAPACITY, "one partial match of the join has more extensions than memory holds"};
        halves();
        return;
    }
    L.Fn = bget<uint32_t>(mem, S * (d + 1));
    hipLaunchKernelGGL((k_bj_place<false, false>), dim3(grid), dim3(BJ_THREADS), 0, J.st, J.v, L);
    HIP_TRY(hipGetLastError());
    bj_depth(J, d + 1, L.Fn, S);
    mem.rewind(mk);
}

// All matches of rule R in the state (ev, ar) on the device: the index and seeds, the depths.
void bj_match(BJRun& J, uint32_t nv, float* ms_index, float* ms_join, bool timed) {
    BJMem& mem = *J.mem;
    if (!mem.arena) {
        // a fixed region: refuse a state whose index alone cannot fit before launching anything
        const uint64_t nkeys = (uint64_t)nv * J.v.A, slots = (uint64_t)J.v.m * J.v.A;
        const uint64_t need = (nkeys + 1) * 16ull + slots * 16ull + (uint64_t)J.v.m * 93ull + (1ull << 20);
        if (need > mem.cap - mem.used)
            throw Error{HGX_ERR_CAPACITY, "a state of " + std::to_string(J.v.m) + " edges needs " +
                                              std::to_string(need >> 20) + " MiB for its index, more than the " +
                                              std::to_string(mem.cap >> 20) + " MiB fixed scratch"};
    }
    hipEvent_t t0 = nullptr, t1 = nullptr, t2 = nullptr;
    if (timed) {
        HIP_TRY(hipEventCreate(&t0)); HIP_TRY(hipEventCreate(&t1)); HIP_TRY(hipEventCreate(&t2));
        HIP_TRY(hipEventRecord(t0, J.st));
    }
    uint64_t P0 = 0;
    uint32_t* seeds = nullptr;
    bj_index(J, nv, &P0, &seeds, t1);
    J.turn = 0;
    J.alg_bytes += (uint64_t)J.v.m * (4ull * J.v.A + 1) + P0 * 4ull;
    if (J.v.R.n_lhs == 1) {
        if (J.out && P0) {
            const uint64_t k = std::min(P0, J.cap);
            HIP_TRY(hipMemcpyAsync(J.out, seeds, sizeof(uint32_t) * k, hipMemcpyDeviceToDevice, J.st));
        }
        J.found = P0;
    } else if (P0) {
        bj_depth(J, 1, seeds, P0);
    }
    if (timed) HIP_TRY(hipEventRecord(t2, J.st));
    uint64_t acc[3] = {0, 0, 0};
    HIP_TRY(hipMemcpyAsync(acc, J.acc, sizeof(acc), hipMemcpyDeviceToHost, J.st));
    HIP_TRY(hipStreamSynchronize(J.st));
    if (J.v.R.n_lhs > 1) J.found = acc[J.turn];
    J.alg_bytes += acc[2];
    if (timed) {
        HIP_TRY(hipEventElapsedTime(ms_index, t0, t1));
        HIP_TRY(hipEventElapsedTime(ms_join, t1, t2));
        (void)hipEventDestroy(t0); (void)hipEventDestroy(t1); (void)hipEventDestroy(t2);
    }
}

}  // namespace hgx

using namespace hgx;

extern "C" int hgx_match_count(hgx_ctx* ctx, const uint8_t* rules, uint32_t rules_len, uint32_t n_rules,
                               uint32_t rule, const uint32_t* edge_offsets, const uint32_t* vertices,
                               uint32_t n_edges, uint64_t* count, uint32_t* match_edges, uint64_t cap,
                               float* device_ms) {
    if (!ctx || !rules || !count || (n_edges && (!edge_offsets || !vertices)) || rule >= n_rules)
        return HGX_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> g(ctx->mu);
    return guarded(ctx, [&]() -> int {
        HIP_TRY(hipSetDevice(ctx->device));
        hgx_run_desc d{};
        d.rules = rules; d.rules_len = rules_len; d.n_rules = n_rules; d.steps = 0;
        d.edge_offsets = edge_offsets; d.vertices = vertices; d.n_edges = n_edges;
        RunHost h = parse_run(&d, false);              // validates rules and arities, renumbers
        const DRule R = h.rules[rule];
        const uint32_t m = h.root_ne(0);
        uint32_t A = 1;
        for (uint32_t e = 0; e < m; ++e) A = std::max(A, h.arity(e));
        for (int i = 0; i < R.n_lhs; ++i) A = std::max<uint32_t>(A, R.la[i]);
        const uint32_t nv = std::max(1u, h.root_nv[0]);
        std::vector<uint32_t> ev((size_t)m * A, 0);
        std::vector<uint8_t> ar(m);
        for (uint32_t e = 0; e < m; ++e) {
            ar[e] = (uint8_t)h.arity(e);
            for (uint32_t k = 0; k < h.arity(e); ++k) ev[(size_t)e * A + k] = h.verts[h.edge_vb[e] + k];
        }
        hipStream_t s = ctx->stream;
        Arena arena(ctx->pool.get());
        BJMem mem;
        mem.arena = &arena;
        uint32_t* d_ev = bget<uint32_t>(mem, (size_t)m * A);
        uint8_t* d_ar = bget<uint8_t>(mem, m);
        h2d(d_ev, ev.data(), ev.size(), s);
        h2d(d_ar, ar.data(), ar.size(), s);
        BJRun J{};
        J.st = s; J.mem = &mem; J.grid = ctx->num_cu * 8;
        J.v.R = R; J.v.ev = d_ev; J.v.ar = d_ar; J.v.m = m; J.v.A = A;
        uint32_t* d_out = nullptr;
        float ms_index = 0, ms_join = 0;
        if (match_edges && cap && cap * R.n_lhs * 4ull > (256ull << 20)) {
            // a large caller buffer: count first, then hold only the matches there are
            BJRun C = J;
            Arena counting(ctx->pool.get());
            BJMem cm;
            cm.arena = &counting;
            C.mem = &cm;
            bj_match(C, nv, &ms_index, &ms_join, false);
            cap = std::min<uint64_t>(cap, std::max<uint64_t>(1, C.found));
        }
        if (match_edges && cap) {
            d_out = bget<uint32_t>(mem, cap * R.n_lhs);
            J.out = d_out; J.cap = cap;
        }
        bj_match(J, nv, &ms_index, &ms_join, true);
        const uint64_t total = J.found;
        if (d_out && total) d2h(match_edges, d_out, std::min(cap, total) * R.n_lhs, s);
        HIP_TRY(hipStreamSynchronize(s));
        if (device_ms) device_ms[0] = ms_index + ms_join;
        if (ctx->prof.on) {
            auto& si = ctx->prof.acc["bigjoin_index"];
            std::snprintf(si.name, sizeof(si.name), "bigjoin_index");
            si.launches += 1; si.total_ms += ms_index; si.items += m; si.alg_bytes += J.index_bytes;
            auto& sj = ctx->prof.acc["bigjoin_join"];
            std::snprintf(sj.name, sizeof(sj.name), "bigjoin_join");
            sj.launches += 1; sj.total_ms += ms_join; sj.items += m; sj.alg_bytes += J.alg_bytes;
        }
        *count = total;
        return HGX_OK;
    });
}

