// hgx_kernels.hip -- gfx950 kernels of one multiway generation.
//
//   k_match<false>   SCAN -> EXPAND -> SINK join, counting matches per state
//   k_match<true>    the same join, writing match records in the deterministic order
//   k_match_bits     both over small binary states, by bit sets
//   k_match_lists    both over larger binary states that fit the LDS, by lists per position
//   k_expand         rewrite + WL hash, one team per child state
//                    (k_expand_small, k_expand_large: children of one arity)
//   k_record         each child's event, causal masks and records, its hash into its request's
//                    state map, and the request's counters
//   k_branchial      sibling-event overlap pairs, one wave per parent state (k_branchial_count:
//                    only their number, where counters are cheaper than bit sets; k_brl_*: the
//                    sorted per-edge lists for parents above 128 edges)
//   k_wl_states      WL hash of given states (roots, and the hgx_wl_hash_batch entry point)
//   small helpers    per-run totals, count masking, map rehash
//
// Every kernel is wave64-native: one team (a wave, or the waves of a workgroup for large
// states) owns one state or one child, stages that state's
// edges in LDS and cooperates through ballots, mbcnt prefix sums and LDS atomics. There is no
// MFMA: nothing here is a dense contraction.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <type_traits>

#include "hgx_device.hpp"
#include "hgx_kernels.hpp"
#include "hgx_wl.hpp"
#include "hgx_wl_small.hpp"
#include "hgx_wl_large.hpp"

namespace hgx {

// Logical block index with consecutive indices kept on one XCD (blocks are dealt to the 8
// XCDs round-robin), so neighbouring children -- which share their parent's edges -- hit the
// same L2. gridDim.x is a multiple of 8 for every launch that uses it.
__device__ inline uint32_t xcd_block() {
    const uint32_t g = gridDim.x, b = blockIdx.x;
    return (b % 8u) * (g / 8u) + b / 8u;
}

// ------------------------------------------------------------------------------------------
// The join. A wave owns one parent state, whose edges are staged in LDS. For each rule of the
// state's run:
//   SCAN    lanes test every edge against the first position of the rule's join order
//           (arity + the repetitions the pattern demands, match_core.hpp:32-49) and the seed
//           list is compacted in edge order with a ballot + mbcnt prefix.
//   EXPAND  each lane extends one seed depth-first over the remaining positions in join order,
//           trying candidates in ascending edge order (join_core.hpp:143-180): edge-injective,
//           vertex-non-injective.
//   SINK    per-lane match counts are prefix-summed across the wave so every match lands at
//           its place in the order (state, rule, seed, depth-first) -- the order the oracle
//           enumerates, so event numbering is identical across engines and runs.
// ------------------------------------------------------------------------------------------

// Counts. A state's matches, a round's and a run's tally are added in 64 bits, and a state stops being
// counted once it passes what its run may still take -- its cap or, without one, the 2^32 - 1 a count
// holds: the run's generation is then refused whatever the other states hold. A seed is given up at
// kSeedMany (the last depth adds at most 65,535 between two looks) and stands for 2^32.
constexpr uint64_t kNoBudget = 0xFFFFFFFFull;     // MatchArgs::budget of a run without a cap
constexpr uint32_t kSeedMany = 0xFFFE0000u;
// Without a cap only counts above this are added to the run's tally: the adds of one run's 300 k states
// to one word took 4 ms, and the few that matter for 2^32 are large.
constexpr uint64_t kTallyMany = 4096;
__device__ __forceinline__ uint64_t seed_count(uint32_t c) { return c < kSeedMany ? c : kNoBudget + 1; }
__device__ __forceinline__ uint32_t stored_count(uint64_t n) { return n < kNoBudget ? (uint32_t)n : (uint32_t)kNoBudget; }
__device__ __forceinline__ void add_tally(const MatchArgs& a, uint32_t run, bool capped, uint64_t n) {
    if (capped ? n != 0 : n > kTallyMany) atomicAdd(&a.run_acc[run], (unsigned long long)n);
}

// Per-lane depth-first state: the edge bound at each depth, the bound-variable mask on entry to
// each depth, the next candidate and the end of the candidate range at each depth, and the
// variable bindings. Rules up to 16 LHS edges and variable ids up to 31 keep it per lane in
// private memory (JoinLaneBig); the common rules -- at most 4 LHS edges, variables below 16 --
// keep it in LDS, interleaved across the wave (element i of a lane at word i * 64 + lane), so
// every step of the depth-first search is an LDS access rather than a private-memory one.
template <int KM, int VM>
struct JoinLaneT {
    uint32_t matched[KM];
    uint32_t smask[KM + 1];
    uint32_t cidx[KM];
    uint32_t chi[KM];
    uint32_t bind[VM];
};
using JoinLaneBig = JoinLaneT<16, 32>;

struct LaneArr {
    uint32_t* p;            // this lane's element 0
    __device__ __forceinline__ uint32_t& operator[](uint32_t i) const { return p[i * WAVE]; }
};
struct JoinLaneLds {
    static constexpr uint32_t WORDS = 4 + 5 + 4 + 4 + 16;
    LaneArr matched, smask, cidx, chi, bind;
    __device__ __forceinline__ void at(uint32_t* block, uint32_t lane) {
        matched.p = block + lane;
        smask.p = matched.p + 4 * WAVE;
        cidx.p = smask.p + 5 * WAVE;
        chi.p = cidx.p + 4 * WAVE;
        bind.p = chi.p + 4 * WAVE;
    }
};

template <class Bind>
__device__ __forceinline__ bool bind_edge(const uint32_t* ev, uint32_t ea, const uint8_t* pv, uint32_t pa,
                                 Bind bind, uint32_t& mask) {   // match_core.hpp:32-49
    if (ea != pa) return false;
    for (uint32_t i = 0; i < ea; ++i) {
        const uint32_t var = pv[i], bit = 1u << var;
        if (mask & bit) { if (bind[var] != ev[i]) return false; }
        else { bind[var] = ev[i]; mask |= bit; }
    }
    return true;
}

// Candidates of depth d: the incidence list of the pivot vertex (a vertex the pattern edge
// shares with the bound prefix; the list holds every edge containing it, ascending), or every
// edge when the pattern edge shares nothing. Either way the candidates are tried in ascending
// edge order, so the matches come out in the same order as an all-edge scan.
template <class JoinLane>
__device__ __forceinline__ void cand_range(const DRule& R, uint32_t d, const JoinLane& L, const uint32_t* iend,
                                  uint32_t ne, uint32_t& lo, uint32_t& hi) {
    const uint32_t pv = R.piv[d];
    if (pv == 0xFFu) { lo = 0; hi = ne; return; }
    const uint32_t x = L.bind[R.lv[R.order[d]][pv]];
    lo = x ? iend[x - 1] : 0u;
    hi = iend[x];
}

// Depth-first completion of one seed; returns the number of matches. With q_out != nullptr
// every match is written at out_base + k (the k-th match of this seed).
template <class JoinLane>
__device__ __forceinline__ uint32_t join_seed(const DRule& R, const uint32_t* sv, const uint8_t* sa,
                                     uint32_t ne, uint32_t A, const uint32_t* iend, const uint16_t* ie,
                                     uint32_t seed, JoinLane& L,
                                     uint16_t* q_out, uint32_t K, uint32_t out_base,
                                     uint32_t* par_out, uint32_t* rule_out, uint32_t* cne_out,
                                     uint32_t parent, uint32_t rule_id, uint32_t child_ne) {
    const uint32_t n = R.n_lhs;
    uint32_t mask = 0;
    if (!bind_edge(sv + seed * A, sa[seed], R.lv[R.order[0]], R.la[R.order[0]], L.bind, mask))
        return 0;
    uint32_t found = 0;
    L.matched[0] = seed;
    if (n == 1) {
        if (q_out) {
            q_out[(size_t)out_base * K + R.order[0]] = (uint16_t)seed;
            par_out[out_base] = parent; rule_out[out_base] = rule_id; cne_out[out_base] = child_ne;
        }
        return 1;
    }
    L.smask[1] = mask;
    cand_range(R, 1, L, iend, ne, L.cidx[1], L.chi[1]);
    uint32_t d = 1;
    while (d >= 1) {
        const uint32_t p = R.order[d];
        const bool indexed = R.piv[d] != 0xFFu;
        bool advanced = false;
        while (L.cidx[d] < L.chi[d]) {
            const uint32_t j = L.cidx[d]++;
            const uint32_t e = indexed ? (uint32_t)ie[j] : j;
            bool taken = false;
            for (uint32_t t = 0; t < d; ++t) taken |= (L.matched[t] == e);
            if (taken) continue;
            uint32_t m = L.smask[d];
            if (!bind_edge(sv + e * A, sa[e], R.lv[p], R.la[p], L.bind, m)) continue;
            L.matched[d] = e;
            if (d + 1 == n) {
                if (q_out) {
                    const size_t o = (size_t)(out_base + found);
                    for (uint32_t t = 0; t < n; ++t) q_out[o * K + R.order[t]] = (uint16_t)L.matched[t];
                    par_out[o] = parent; rule_out[o] = rule_id; cne_out[o] = child_ne;
                }
                if (++found == kSeedMany && !q_out) return found;
                continue;
            }
            L.smask[d + 1] = m;
            cand_range(R, d + 1, L, iend, ne, L.cidx[d + 1], L.chi[d + 1]);
            ++d;
            advanced = true;
            break;
        }
        if (!advanced) --d;
    }
    return found;
}

// Order of two matches of one state, as a full join emits them: rule, then the edge
// positions in the rule's join order (q arrays are in LHS order).
__device__ __forceinline__ bool match_less(const DRule* rules, uint32_t ra, const uint16_t* qa, uint32_t rb,
                                  const uint16_t* qb) {
    if (ra != rb) return ra < rb;
    const DRule& R = rules[ra];
    for (uint32_t t = 0; t < R.n_lhs; ++t) {
        const uint32_t o = R.order[t];
        if (qa[o] != qb[o]) return qa[o] < qb[o];
    }
    return false;
}

// Delta matches (find_delta_matches, hypergraph/include/hypergraph/pattern_matcher.hpp:493-537):
// pattern edge p bound to child edge `anchor` (a produced edge), the rest completed depth-first
// in the anchored order aord[p]. LHS positions below p take kept edges only (positions below
// `kept`), so a match that uses produced edges is found exactly once -- from its lowest LHS
// position holding a produced edge. With d_out the k-th match is written at d_out + k * stride
// as (rule, edge positions in LHS order).
template <class JoinLane>
__device__ __forceinline__ uint32_t join_anchor(const DRule& R, uint32_t p, const uint32_t* sv, const uint8_t* sa,
                                       uint32_t ne, uint32_t A, const uint32_t* iend, const uint16_t* ie,
                                       uint32_t kept, uint32_t anchor, JoinLane& L, uint16_t* d_out,
                                       uint32_t stride, uint32_t rule_id) {
    const uint32_t n = R.n_lhs;
    const uint8_t* ord = R.aord[p];
    const uint8_t* piv = R.apiv[p];
    uint32_t mask = 0;
    if (!bind_edge(sv + anchor * A, sa[anchor], R.lv[p], R.la[p], L.bind, mask)) return 0;
    L.matched[0] = anchor;
    auto range = [&](uint32_t d, uint32_t& lo, uint32_t& hi) {
        const uint32_t pv = piv[d];
        if (pv == 0xFFu) { lo = 0; hi = ne; return; }
        const uint32_t x = L.bind[R.lv[ord[d]][pv]];
        lo = x ? iend[x - 1] : 0u;
        hi = iend[x];
    };
    uint32_t found = 0;
    if (n == 1) {
        if (d_out) { d_out[0] = (uint16_t)rule_id; d_out[1 + p] = (uint16_t)anchor; }
        return 1;
    }
    L.smask[1] = mask;
    range(1, L.cidx[1], L.chi[1]);
    uint32_t d = 1;
    while (d >= 1) {
        const uint32_t pe = ord[d];
        const bool indexed = piv[d] != 0xFFu;
        const uint32_t lim = pe < p ? kept : ne;      // candidates ascend: stop at the limit
        bool advanced = false;
        while (L.cidx[d] < L.chi[d]) {
            const uint32_t j = L.cidx[d]++;
            const uint32_t e = indexed ? (uint32_t)ie[j] : j;
            if (e >= lim) { L.cidx[d] = L.chi[d]; break; }
            bool taken = false;
            for (uint32_t t = 0; t < d; ++t) taken |= (L.matched[t] == e);
            if (taken) continue;
            uint32_t m = L.smask[d];
            if (!bind_edge(sv + e * A, sa[e], R.lv[pe], R.la[pe], L.bind, m)) continue;
            L.matched[d] = e;
            if (d + 1 == n) {
                if (d_out) {
                    uint16_t* o = d_out + (size_t)found * stride;
                    o[0] = (uint16_t)rule_id;
                    for (uint32_t t = 0; t < n; ++t) o[1 + ord[t]] = (uint16_t)L.matched[t];
                }
                if (++found == kSeedMany && !d_out) return found;
                continue;
            }
            L.smask[d + 1] = m;
            range(d + 1, L.cidx[d + 1], L.chi[d + 1]);
            ++d;
            advanced = true;
            break;
        }
        if (!advanced) --d;
    }
    return found;
}

// Depth-first completion of one seed with the search state in registers, for rules of at most
// N = 4 LHS edges: every depth is its own template level, so the edges bound so far are a
// register array indexed by constants, and a variable's value is read from the vertex slot
// where it was first bound (DRule::jsrc) instead of from a binding table. Same candidates in
// the same order as join_seed, so the same matches in the same order.
template <int N>
__device__ __forceinline__ uint32_t pick(const uint32_t (&m)[N], uint32_t d) {
    uint32_t r = m[0];
#pragma unroll
    for (int k = 1; k < N; ++k) r = (d == (uint32_t)k) ? m[k] : r;
    return r;
}

struct RegJoinOut {
    uint16_t* q;
    uint32_t K, base, *parent, *rule, *cne;
    uint32_t state, rule_id, child_ne;
};

template <int N, int D, bool OUT>
__device__ __forceinline__ uint32_t reg_join(const DRule& R, const uint32_t* sv, const uint8_t* sa, uint32_t ne,
                                             uint32_t A, const uint32_t* iend, const uint16_t* ie,
                                             uint32_t (&m)[N], const RegJoinOut& o, uint32_t found) {
    if constexpr (D == N) {
        if constexpr (OUT) {
            const size_t at = (size_t)(o.base + found);
#pragma unroll
            for (int t = 0; t < N; ++t) o.q[at * o.K + R.order[t]] = (uint16_t)m[t];
            o.parent[at] = o.state; o.rule[at] = o.rule_id; o.cne[at] = o.child_ne;
        }
        return found + 1;
    } else {
        const uint32_t pe = R.order[D], pa = R.la[pe];
        uint32_t lo = 0, hi = ne;
        const uint32_t pv = R.piv[D];
        const bool indexed = pv != 0xFFu;
        if (indexed) {
            const uint32_t src = R.jsrc[D][pv];
            const uint32_t x = sv[pick<N>(m, src >> 4) * A + (src & 15u)];
            lo = x ? iend[x - 1] : 0u;
            hi = iend[x];
        }
        for (uint32_t j = lo; j < hi; ++j) {
            const uint32_t e = indexed ? (uint32_t)ie[j] : j;
            bool ok = sa[e] == pa;
#pragma unroll
            for (int t = 0; t < D; ++t) ok &= (m[t] != e);
            if (!ok) continue;
            for (uint32_t i = 0; i < pa && ok; ++i) {
                const uint32_t src = R.jsrc[D][i];
                if (src == 0xFFu) continue;
                const uint32_t sd = src >> 4, si = src & 15u;
                const uint32_t want = sd == (uint32_t)D ? sv[e * A + si] : sv[pick<N>(m, sd) * A + si];
                ok = sv[e * A + i] == want;
            }
            if (!ok) continue;
            m[D] = e;
            found = reg_join<N, D + 1, OUT>(R, sv, sa, ne, A, iend, ie, m, o, found);
            if (!OUT && D + 1 < N && found >= kSeedMany) return found;   // (the last depth adds at most 65,535)
        }
        return found;
    }
}

template <int N, bool OUT>
__device__ __forceinline__ uint32_t reg_join_seed(const DRule& R, const uint32_t* sv, const uint8_t* sa,
                                                  uint32_t ne, uint32_t A, const uint32_t* iend,
                                                  const uint16_t* ie, uint32_t seed, const RegJoinOut& o) {
    uint32_t m[N];
#pragma unroll
    for (int t = 0; t < N; ++t) m[t] = 0xFFFFFFFFu;
    m[0] = seed;
    return reg_join<N, 1, OUT>(R, sv, sa, ne, A, iend, ie, m, o, 0u);
}

// seeds already satisfy position order[0]'s pattern (the SCAN checks it)
template <bool OUT>
__device__ __forceinline__ uint32_t reg_join_any(const DRule& R, const uint32_t* sv, const uint8_t* sa,
                                                 uint32_t ne, uint32_t A, const uint32_t* iend,
                                                 const uint16_t* ie, uint32_t seed, const RegJoinOut& o) {
    switch (R.n_lhs) {
        case 1: return reg_join_seed<1, OUT>(R, sv, sa, ne, A, iend, ie, seed, o);
        case 2: return reg_join_seed<2, OUT>(R, sv, sa, ne, A, iend, ie, seed, o);
        case 3: return reg_join_seed<3, OUT>(R, sv, sa, ne, A, iend, ie, seed, o);
        default: return reg_join_seed<4, OUT>(R, sv, sa, ne, A, iend, ie, seed, o);
    }
}

uint32_t match_lds_per_wave(uint32_t max_ne, uint32_t max_nextv, uint32_t A, uint32_t KL, uint32_t dmax,
                            bool small, uint32_t team, bool lanes) {
    auto al = [](uint32_t b) { return (b + 7u) & ~7u; };
    // + 64: carving slack; + 64: the team's reduction words at the end
    uint32_t b = al(max_ne * A * 4) + al(max_ne) + al(max_ne * 2) + al((max_nextv + 1) * 4) +
                 al(max_ne * A * 2) * 2 + al(max_ne * A * 4) + 128;
    if (small) b += (lanes ? JoinLaneLds::WORDS * WAVE * 4 * team : 0u) + 2 * (uint32_t)sizeof(DRule);
    if (dmax) b += al(dmax * (KL + 1) * 2) + al(dmax * 2) + al((dmax + 1) * 4);
    return b;
}

// W is the team: one wave per state (W = 1, up to four per workgroup, each with its own
// workspace) or the W waves of a workgroup sharing one state and one workspace (large states,
// whose workspace would otherwise leave a CU one or two waves). The one-wave passes are held to
// four waves per SIMD (128 registers): at five (96) the emit pass spilled 19 registers and 96
// bytes per lane to scratch -- 25 MB of writes per launch instead of 3 MB -- and config 2 ran 3%
// slower, while the batched pass timed alike under both bounds (both measured on binary states, which
// have kernels of their own now).
// GWS: the workspace is a per-workgroup slice of global memory (a.scratch) -- the same code for
// states too large for LDS, with W = 8. G < 64 (with W = 1): sub-wave teams, 64 / G states per
// wave, each team with its own workspace, for small states whose seeds would leave most of a
// wave's lanes idle.
template <bool EMIT, class JoinLane, uint32_t W, bool GWS = false, uint32_t G = 64>
__global__ __launch_bounds__(W == 1 ? 256 : 64 * W, W == 1 ? 4 : 1) void k_match(MatchArgs a) {
    using TM = typename TeamSel<W, G>::type;
    extern __shared__ uint8_t lds[];
    constexpr uint32_t N = TM::N;
    const uint32_t w = threadIdx.x / WAVE, l = lane_id();
    const uint32_t ti = W == 1 ? threadIdx.x / G : 0;         // team within the workgroup
    uint8_t* p;
    if constexpr (GWS) p = a.scratch + (size_t)blockIdx.x * a.lds_per_wave;
    else p = lds + (W == 1 ? (size_t)ti * a.lds_per_wave : 0);
    const TM tm((uint64_t*)(p + a.lds_per_wave - 64));         // the workspace's last 64 bytes
    const uint32_t A = a.P.A;
    uint32_t* sv = (uint32_t*)carve(p, a.max_ne * A * 4);      // vertices
    uint8_t* sa = carve(p, a.max_ne);                           // arity
    uint16_t* seeds = (uint16_t*)carve(p, a.max_ne * 2);
    uint32_t* iend = (uint32_t*)carve(p, (a.max_nextv + 1) * 4); // incidence list ends per vertex
    uint16_t* ie = (uint16_t*)carve(p, a.max_ne * A * 2);       // incidence lists
    uint16_t* ie2 = (uint16_t*)carve(p, a.max_ne * A * 2);      // the same, before ordering
    uint32_t* iown = (uint32_t*)carve(p, a.max_ne * A * 4);     // vertex owning each list slot
    const uint32_t dstride = a.KL + 1;                          // delta match: rule + positions
    uint16_t* dlist = (uint16_t*)carve(p, a.dmax * dstride * 2);   // empty when dmax = 0
    uint16_t* dperm = (uint16_t*)carve(p, a.dmax * 2);
    uint32_t* dhist = (uint32_t*)carve(p, a.dmax ? (a.dmax + 1) * 4 : 0);
    JoinLane L;
    // Small rules (<= 4 LHS edges, <= 2 rules per request): the request's rules staged in LDS per
    // state, so every pattern read in the depth-first search is an LDS read.
    constexpr bool SMALL = std::is_same<JoinLane, JoinLaneLds>::value;
    DRule* lr = nullptr;
    if constexpr (SMALL) {
        // one lane-interleaved block per wave; only the forwarding path's anchored joins use it
        // (the full join keeps its search in registers and checks seeds by first-binding slot)
        const uint32_t lane_words = a.fwd_n ? JoinLaneLds::WORDS * WAVE * W : 0u;
        L.at((uint32_t*)carve(p, lane_words * 4) + (W == 1 || !lane_words ? 0 : w * JoinLaneLds::WORDS * WAVE), l);
        lr = (DRule*)carve(p, 2 * sizeof(DRule));
    }

    // States strided over the teams: neighbouring states (often one request's, of similar size)
    // go to different teams, which balances the launch better than contiguous chunks do.
    const uint32_t tpb = W == 1 ? (blockDim.x / WAVE) * (WAVE / G) : 1;   // teams per workgroup
    const uint32_t teams = gridDim.x * tpb;
    const uint32_t n_items = a.nrange ? a.n_items : a.P.n;
    // The count pass visits the states scattered over the launch, so each request's states are
    // counted at an even pace from start to end: a request over its cap passes it with most of
    // its states still ahead, and those are skipped at the tally check below (in launch order a
    // request's states are counted at once, and the check stops few). Blocks of
    // kCountSpreadBlock consecutive states stay together: neighbouring small states share cache
    // lines, which one state at a time would fetch again for each.
    const bool spread = !EMIT && a.spread > 1;
    const uint32_t nblk = (n_items + kCountSpreadBlock - 1) / kCountSpreadBlock;
    const uint32_t n_loop = spread ? nblk * kCountSpreadBlock : n_items;
    for (uint32_t ls = blockIdx.x * tpb + (W == 1 ? ti : 0); ls < n_loop; ls += teams) {
        uint32_t li = ls;
        if (spread) {
            li = (uint32_t)((uint64_t)(ls / kCountSpreadBlock) * a.spread % nblk) * kCountSpreadBlock +
                 ls % kCountSpreadBlock;
            if (li >= n_items) continue;                        // the last block's tail
        }
        uint32_t s = li;
        if (a.nrange) {                                         // subset: logical -> state
            uint32_t lo = 0, hi = a.nrange;
            while (hi - lo > 1) { const uint32_t mid = (lo + hi) >> 1; if (a.rpre[mid] <= li) lo = mid; else hi = mid; }
            s = a.rb[lo] + (li - a.rpre[lo]);
        }
        // the state's record and its request's flags in two rounds of independent loads
        const uint32_t run = a.P.run[s];
        const uint32_t ne = a.P.ne[s];
        const uint64_t eo = a.P.eoff[s];
        const uint32_t nvid = a.P.nextv[s];                     // labels are < nvid
        const uint8_t active = a.active[run] && (!a.smask || a.smask[s]);
        const uint64_t budget = EMIT ? 0 : (uint64_t)a.budget[run];
        // the run's tally moves under other teams: one read, shared, so the team agrees
        const bool capped = budget != kNoBudget;
        const uint64_t tally = EMIT ? 0 : tm.bcast(tm.leader() ? (uint64_t)a.run_acc[run] : 0ull);
        if (!active || (!EMIT && tally > budget)) {
            if (!EMIT && tm.leader()) { a.cnt[s] = 0; a.state_edges[s] = 0; }
            continue;
        }
        for (uint32_t i = tm.r; i < ne * A; i += N) sv[i] = a.P.ev[eo * A + i];
        for (uint32_t i = tm.r; i < ne; i += N) sa[i] = a.P.ar[eo + i];
        for (uint32_t v = tm.r; v <= nvid; v += N) iend[v] = 0;
        tm.sync();
        // Incidence index (vertex -> ascending edges, one entry per (vertex, edge)): counting
        // sort with LDS atomics, then each list put in edge order.
        for (uint32_t e = tm.r; e < ne; e += N)
            for (uint32_t k = 0; k < sa[e]; ++k) {
                const uint32_t x = sv[e * A + k];
                bool dup = false;
                for (uint32_t k2 = 0; k2 < k; ++k2) dup |= (sv[e * A + k2] == x);
                if (!dup) atomicAdd(&iend[x], 1u);
            }
        tm.sync();
        const uint32_t nslot = tm.excl_scan_lds(iend, nvid + 1);    // iend[x] = start of x's list
        // The emit pass writes matches in the full join's order, and the delta joins of the
        // forwarding path (join_anchor) stop a list at the first edge past their limit: both need
        // each list in ascending edge order. The count pass's full join enumerates every
        // candidate of a list, whatever its order, and joins over the lists as filled.
        const bool sorted = EMIT || s < a.fwd_n;
        if (sorted)
            for (uint32_t x = tm.r; x < nvid; x += N)
                for (uint32_t i = iend[x]; i < iend[x + 1]; ++i) iown[i] = x;
        tm.sync();
        for (uint32_t e = tm.r; e < ne; e += N)
            for (uint32_t k = 0; k < sa[e]; ++k) {
                const uint32_t x = sv[e * A + k];
                bool dup = false;
                for (uint32_t k2 = 0; k2 < k; ++k2) dup |= (sv[e * A + k2] == x);
                if (!dup) ie2[atomicAdd(&iend[x], 1u)] = (uint16_t)e;   // -> iend[x] = end
            }
        tm.sync();
        // each list into ascending edge order: an entry's place is the number of smaller entries
        // of its list, so a hub vertex's list is placed by as many lanes as it has entries
        if (sorted) {
            for (uint32_t j = tm.r; j < nslot; j += N) {
                const uint32_t x = iown[j];
                const uint32_t b = x ? iend[x - 1] : 0u, n = iend[x] - b;
                const uint16_t key = ie2[j];
                uint32_t r = 0;
#pragma unroll 4
                for (uint32_t i = 0; i < n; ++i) r += ie2[b + i] < key ? 1u : 0u;
                ie[b + r] = key;
            }
            tm.sync();
        }
        const uint16_t* il = sorted ? ie : ie2;

        const DRun& RN = a.runs[run];
        const DRule* rules;
        if constexpr (SMALL) {
            // the whole rules when forwarding (anchored orders), else the prefix the full join
            // reads (DRule puts those fields first)
            const uint32_t pw = a.fwd_n ? (uint32_t)(sizeof(DRule) / 4) : (uint32_t)(offsetof(DRule, lv) / 4);
            const uint32_t words = RN.n_rules * pw;
            for (uint32_t i = tm.r; i < words; i += N) {
                const uint32_t r = i / pw, k = i - r * pw;
                ((uint32_t*)&lr[r])[k] = ((const uint32_t*)&RN.rules[r])[k];
            }
            tm.sync();
            rules = lr;
        } else {
            rules = RN.rules;
        }
        uint64_t total = 0;
        uint64_t edges_sum = 0;                                // count pass: edges of the children
        bool stop = false;
        uint32_t out = EMIT ? (uint32_t)a.moff[s] : 0u;
        bool full = true;
        if (s < a.fwd_n) {
            // ---- incremental forwarding (parallel_evolution.cpp:591-756): the parent's
            //      matches that avoid the consumed edges, plus delta joins at the produced
            //      edges, merged into the full join's order ----
            const DRule& CR = rules[a.pm_rule[s]];
            const uint32_t nc = CR.n_lhs, nprod = CR.n_rhs;
            const uint32_t kept = ne - nprod;                   // kept edges come first
            const uint16_t* cq = a.pm_q + (size_t)s * a.pm_K;  // consumed, parent positions
            const uint32_t par = a.pm_parent[s];
            const uint64_t lb = a.pm_moff[par], le = a.pm_moff[par + 1];
            uint32_t ncombo = 0;                                // (rule, anchor, produced edge)
            for (uint32_t r = 0; r < RN.n_rules; ++r) ncombo += rules[r].n_lhs * nprod;
            auto combo = [&](uint32_t i, uint32_t& r, uint32_t& pp, uint32_t& j) {
                r = 0;
                while (i >= rules[r].n_lhs * nprod) { i -= rules[r].n_lhs * nprod; ++r; }
                pp = i / nprod;
                j = i % nprod;
            };
            uint64_t nd = 0;
            uint64_t de = 0;                                    // child edges of the delta matches
            for (uint32_t base = 0; base < ncombo; base += N) {
                const uint32_t i = base + tm.r;
                uint32_t c = 0;
                if (i < ncombo) {
                    uint32_t r, pp, j;
                    combo(i, r, pp, j);
                    c = join_anchor(rules[r], pp, sv, sa, ne, A, iend, il, kept, kept + j, L, nullptr, 0, 0);
                    de += (uint64_t)c * (ne - rules[r].n_lhs + rules[r].n_rhs);
                }
                nd += tm.sum64(seed_count(c));
            }
            if (!EMIT || (a.dmax && nd <= a.dmax)) {
                full = false;
                if (EMIT) {
                    uint32_t o = 0;
                    for (uint32_t base = 0; base < ncombo; base += N) {
                        const uint32_t i = base + tm.r;
                        uint32_t c = 0, r = 0, pp = 0, j = 0;
                        if (i < ncombo) {
                            combo(i, r, pp, j);
                            c = join_anchor(rules[r], pp, sv, sa, ne, A, iend, il, kept, kept + j, L, nullptr, 0, 0);
                        }
                        uint32_t round;
                        const uint32_t inc = tm.incl_scan(c, round);
                        if (c)
                            join_anchor(rules[r], pp, sv, sa, ne, A, iend, il, kept, kept + j, L,
                                        dlist + (size_t)(o + inc - c) * dstride, dstride, r);
                        o += round;
                    }
                    tm.sync();
                    for (uint32_t i = tm.r; i < nd; i += N) {        // rank = place in order
                        const uint16_t* di = dlist + (size_t)i * dstride;
                        uint32_t rank = 0;
                        for (uint32_t j = 0; j < nd; ++j) {
                            const uint16_t* dj = dlist + (size_t)j * dstride;
                            rank += match_less(rules, dj[0], dj + 1, di[0], di + 1) ? 1u : 0u;
                        }
                        dperm[rank] = (uint16_t)i;
                    }
                    for (uint32_t i = tm.r; i <= nd; i += N) dhist[i] = 0;
                    tm.sync();
                }
                uint32_t nf = 0;
                for (uint64_t base = lb; base < le; base += N) {
                    const uint64_t m = base + tm.r;
                    bool fw = false;
                    uint32_t rm = 0, nm = 0;
                    uint16_t qm[16];
                    if (m < le) {
                        rm = a.pm_rule[m];
                        nm = rules[rm].n_lhs;
                        fw = true;
                        for (uint32_t t = 0; t < nm; ++t) {
                            const uint32_t x = a.pm_q[m * a.pm_K + t];
                            uint32_t below = 0;
                            for (uint32_t u = 0; u < nc; ++u) {
                                const uint32_t y = cq[u];
                                fw &= (x != y);
                                below += (y < x) ? 1u : 0u;
                            }
                            qm[t] = (uint16_t)(x - below);   // position among the kept edges
                        }
                    }
                    uint32_t nround;
                    const uint32_t at = tm.compact(fw, nround);
                    if (!EMIT && fw) de += ne - nm + rules[rm].n_rhs;
                    if (EMIT && fw) {
                        uint32_t lo = 0, hi = nd;                   // delta matches before it
                        while (lo < hi) {
                            const uint32_t mid = (lo + hi) >> 1;
                            const uint16_t* dm = dlist + (size_t)dperm[mid] * dstride;
                            if (match_less(rules, dm[0], dm + 1, rm, qm)) lo = mid + 1; else hi = mid;
                        }
                        const uint32_t o2 = out + nf + at + lo;
                        for (uint32_t t = 0; t < nm; ++t) a.M.q[(size_t)o2 * a.M.K + t] = qm[t];
                        a.M.parent[o2] = s;
                        a.M.rule[o2] = rm;
                        a.M.cne[o2] = ne - nm + rules[rm].n_rhs;
                        atomicAdd(&dhist[lo], 1u);
                    }
                    nf += nround;
                }
                if (EMIT) {
                    tm.sync();
                    tm.excl_scan_lds(dhist, nd + 1);          // dhist[k + 1] = forwarded before delta k
                    for (uint32_t k = tm.r; k < nd; k += N) {
                        const uint16_t* dm = dlist + (size_t)dperm[k] * dstride;
                        const uint32_t rr = dm[0], nm = rules[rr].n_lhs;
                        const uint32_t o2 = out + dhist[k + 1] + k;
                        for (uint32_t t = 0; t < nm; ++t) a.M.q[(size_t)o2 * a.M.K + t] = dm[1 + t];
                        a.M.parent[o2] = s;
                        a.M.rule[o2] = rr;
                        a.M.cne[o2] = ne - nm + rules[rr].n_rhs;
                    }
                    tm.sync();
                } else {
                    total = nf + nd;
                    edges_sum = tm.sum64(de);
                    if (tm.leader()) add_tally(a, run, capped, total);
                }
            }
        }
        for (uint32_t r = 0; full && r < RN.n_rules && !stop; ++r) {
            const DRule& R = rules[r];
            const uint32_t p0 = R.order[0];
            const uint32_t child_ne = ne - R.n_lhs + R.n_rhs;
            // SCAN: compact the seeds of position order[0] in edge order.
            uint32_t nseed = 0;
            for (uint32_t base = 0; base < ne; base += N) {
                const uint32_t e = base + tm.r;
                bool ok = false;
                if (e < ne && sa[e] == R.la[p0]) {
                    if constexpr (SMALL) {
                        // repeated pattern variables: each position equals its first binding's
                        ok = true;
                        for (uint32_t i = 0; i < R.la[p0]; ++i) {
                            const uint32_t src = R.jsrc[0][i];
                            if (src != 0xFFu) ok &= sv[e * A + i] == sv[e * A + (src & 15u)];
                        }
                    } else {
                        uint32_t m = 0;
                        ok = bind_edge(sv + e * A, sa[e], R.lv[p0], R.la[p0], L.bind, m);
                    }
                }
                uint32_t nround;
                const uint32_t at = tm.compact(ok, nround);
                if (ok) seeds[nseed + at] = (uint16_t)e;
                nseed += nround;
            }
            tm.sync();
            // EXPAND + SINK, 64 seeds per round.
            uint16_t* sc = (SMALL && a.seedcnt && s >= a.fwd_n) ? a.seedcnt + 2 * eo + (size_t)r * ne : nullptr;
            for (uint32_t base = 0; base < nseed; base += N) {
                const uint32_t i = base + tm.r;
                uint32_t c = 0;
                if (i < nseed) {
                    if constexpr (SMALL) {
                        const uint32_t kept = (EMIT && sc) ? sc[i] : 0xFFFFu;
                        c = kept != 0xFFFFu ? kept
                                            : reg_join_any<false>(R, sv, sa, ne, A, iend, il, seeds[i], RegJoinOut{});
                        if (!EMIT && sc) sc[i] = (uint16_t)(c < 0xFFFFu ? c : 0xFFFFu);
                    } else {
                        c = join_seed(R, sv, sa, ne, A, iend, il, seeds[i], L, nullptr, 0, 0, nullptr, nullptr,
                                      nullptr, 0, 0, 0);
                    }
                }
                if (EMIT) {
                    uint32_t round;
                    const uint32_t inc = tm.incl_scan(c, round);
                    if (i < nseed && c) {
                        if constexpr (SMALL) {
                            const RegJoinOut ro{a.M.q, a.M.K, out + inc - c, a.M.parent, a.M.rule, a.M.cne,
                                                s, r, child_ne};
                            reg_join_any<true>(R, sv, sa, ne, A, iend, il, seeds[i], ro);
                        } else {
                            join_seed(R, sv, sa, ne, A, iend, il, seeds[i], L, a.M.q, a.M.K, out + inc - c,
                                      a.M.parent, a.M.rule, a.M.cne, s, r, child_ne);
                        }
                    }
                    out += round;
                } else {
                    // The run's shared tally: once it passes what the run may still take, the
                    // generation is over the cap whatever the other states hold, so stop. Every
                    // state's count equals what it added, so the totals stay over the cap.
                    const uint64_t round = tm.sum64(seed_count(c));
                    total += round;
                    edges_sum += round * child_ne;
                    if ((base + N >= nseed && r + 1 >= RN.n_rules) || (!capped && total <= kTallyMany)) {
                        // the state's last round, or one not worth it: nothing to stop, no wait
                        if (tm.leader()) add_tally(a, run, capped, round);
                    } else {
                        unsigned long long before = 0;
                        if (tm.leader() && round) before = atomicAdd(&a.run_acc[run], (unsigned long long)round);
                        before = tm.bcast(before);
                        if (before + round > budget) { stop = true; break; }
                    }
                }
            }
            tm.sync();
        }
        if (!EMIT && tm.leader()) {
            a.cnt[s] = stored_count(total);
            a.state_edges[s] = edges_sum;
        }
    }
}


// ------------------------------------------------------------------------------------------
// The join over small binary states by bit sets: states of at most 64 * NW edges and 255 vertex labels,
// every edge binary, rules of at most 4 LHS edges. Per (position, vertex) a set of the edges holding
// the vertex there, one bit an edge, in LDS; the candidates of a depth are the intersection of the
// sets of its bound positions (and the loops where the pattern edge repeats its variable) less the
// edges in use, so no candidate is tested, the ascending order is the bits', and the last depth
// counts by population count. Matches and their order are k_match's. What bounded k_match here were
// chains of LDS reads per candidate -- list entry, edge, rule tables; this one is bound by the state's
// loads and the building of the sets (batched pass: count 4.10 -> 0.85 ms, emit 1.80 -> 0.36).
// ------------------------------------------------------------------------------------------

template <uint32_t NW>
struct BitSet {
    uint64_t w[NW];
};

template <uint32_t NW>
struct BitJoin {
    const uint64_t* inc0;      // [labels][NW]
    const uint64_t* inc1;
    const uint16_t* ev;        // edges: first vertex | second << 8
    BitSet<NW> all, loops;
    uint32_t bj[4];
};

// The edges bound so far and their vertices, by value and by constant depth: registers.
struct Bound {
    uint32_t e0, e1, e2, e3, v0, v1, v2, v3;
    template <int D>
    __device__ __forceinline__ void set(uint32_t x, uint32_t v) {
        if constexpr (D == 1) { e1 = x; v1 = v; }
        else if constexpr (D == 2) { e2 = x; v2 = v; }
        else { e3 = x; v3 = v; }
    }
};

// Candidates of depth D, whose binding word is b.
template <uint32_t NW, int D>
__device__ __forceinline__ BitSet<NW> bit_cands(const BitJoin<NW>& J, uint32_t b, const Bound& B) {
    auto value = [&](uint32_t src) {                 // a bound position's vertex
        const uint32_t d = (src >> 1) & 3u;
        uint32_t x = B.v0;
        // (masks, not selects: a select of two members makes the struct live in memory)
        if (D > 1) { const uint32_t m = 0u - (uint32_t)(d == 1); x = (x & ~m) | (B.v1 & m); }
        if (D > 2) { const uint32_t m = 0u - (uint32_t)(d == 2); x = (x & ~m) | (B.v2 & m); }
        return (src & 8u) ? x >> 8 : x & 0xFFu;
    };
    BitSet<NW> m = J.all;
    if (b & 1u) {
        const uint64_t* s = J.inc0 + value(b) * NW;
#pragma unroll
        for (uint32_t k = 0; k < NW; ++k) m.w[k] &= s[k];
    }
    if (b & 16u) {
        const uint64_t* s = J.inc1 + value(b >> 4) * NW;
#pragma unroll
        for (uint32_t k = 0; k < NW; ++k) m.w[k] &= s[k];
    }
#pragma unroll
    for (uint32_t k = 0; k < NW; ++k) {
        if (b & 256u) m.w[k] &= J.loops.w[k];
        auto drop = [&](uint32_t e) { if (NW == 1 || (e >> 6) == k) m.w[k] &= ~(1ull << (e & 63u)); };
        drop(B.e0);
        if (D > 1) drop(B.e1);
        if (D > 2) drop(B.e2);
    }
    return m;
}

// Completions of depths D..N-1; OUT writes each as the found-th match of `o`, else counts.
template <uint32_t NW, int N, int D, bool OUT>
__device__ __forceinline__ uint32_t bit_join(const BitJoin<NW>& J, Bound B, const RegJoinOut& o, uint32_t found) {
    if constexpr (D == N) {
        if constexpr (OUT) {
            const size_t at = (size_t)(o.base + found);
            if (N == 2 && o.K == 2) {                 // the pair in one word
                const bool swap = ((J.bj[0] >> 12) & 3u) != 0;
                ((uint32_t*)o.q)[at] = swap ? (B.e1 | B.e0 << 16) : (B.e0 | B.e1 << 16);
            } else {
                uint16_t* q = o.q + at * o.K;
                q[(J.bj[0] >> 12) & 3u] = (uint16_t)B.e0;
                if (N > 1) q[(J.bj[1] >> 12) & 3u] = (uint16_t)B.e1;
                if (N > 2) q[(J.bj[2] >> 12) & 3u] = (uint16_t)B.e2;
                if (N > 3) q[(J.bj[3] >> 12) & 3u] = (uint16_t)B.e3;
            }
            o.parent[at] = o.state; o.rule[at] = o.rule_id; o.cne[at] = o.child_ne;
        }
        return found + 1;
    } else {
        const BitSet<NW> m = bit_cands<NW, D>(J, J.bj[D], B);
#pragma unroll
        for (uint32_t k = 0; k < NW; ++k) {
            if constexpr (D + 1 == N && !OUT) {
                found += (uint32_t)__popcll(m.w[k]);
            } else {
                for (uint64_t w = m.w[k]; w; w &= w - 1) {
                    const uint32_t e = k * 64 + (uint32_t)__builtin_ctzll(w);
                    B.template set<D>(e, D + 1 < N ? J.ev[e] : 0u);
                    found = bit_join<NW, N, D + 1, OUT>(J, B, o, found);
                }
            }
        }
        return found;
    }
}

template <uint32_t NW, bool OUT>
__device__ __forceinline__ uint32_t bit_join_any(const BitJoin<NW>& J, uint32_t n_lhs, uint32_t seed, uint32_t sv,
                                                 const RegJoinOut& o) {
    const Bound B{seed, 0, 0, 0, sv, 0, 0, 0};
    switch (n_lhs) {
        case 1: return bit_join<NW, 1, 1, OUT>(J, B, o, 0u);
        case 2: return bit_join<NW, 2, 1, OUT>(J, B, o, 0u);
        case 3: return bit_join<NW, 3, 1, OUT>(J, B, o, 0u);
        default: return bit_join<NW, 4, 1, OUT>(J, B, o, 0u);
    }
}

uint32_t match_bits_lds(uint32_t max_ne, uint32_t max_nextv, uint32_t nw) {
    return (2 * max_nextv * nw * 8 + ((2 * max_ne + 7u) & ~7u) + 15u) & ~15u;
}

template <bool EMIT, uint32_t NW, uint32_t G>
__global__ __launch_bounds__(256) void k_match_bits(MatchArgs a) {
    using TM = typename TeamSel<1, G>::type;
    extern __shared__ uint8_t lds[];
    constexpr uint32_t N = TM::N;
    const uint32_t tpb = (blockDim.x / WAVE) * (WAVE / G), ti = threadIdx.x / G;
    uint8_t* p = lds + (size_t)ti * a.lds_per_wave;
    const TM tm(nullptr);
    const uint32_t A = a.P.A, NL = a.max_nextv;
    uint64_t* inc0 = (uint64_t*)carve(p, NL * NW * 8);
    uint64_t* inc1 = (uint64_t*)carve(p, NL * NW * 8);
    uint16_t* ev = (uint16_t*)carve(p, a.max_ne * 2);

    // states strided over the teams, the count pass's scattered in blocks, as in k_match
    const uint32_t teams = gridDim.x * tpb;
    const uint32_t n_items = a.nrange ? a.n_items : a.P.n;
    const bool spread = !EMIT && a.spread > 1;
    const uint32_t nblk = (n_items + kCountSpreadBlock - 1) / kCountSpreadBlock;
    const uint32_t n_loop = spread ? nblk * kCountSpreadBlock : n_items;
    for (uint32_t ls = blockIdx.x * tpb + ti; ls < n_loop; ls += teams) {
        uint32_t s = ls;
        if (spread) {
            s = (uint32_t)((uint64_t)(ls / kCountSpreadBlock) * a.spread % nblk) * kCountSpreadBlock +
                ls % kCountSpreadBlock;
            if (s >= n_items) continue;                         // the last block's tail
        }
        if (a.nrange) {                                         // subset: logical -> state
            uint32_t lo = 0, hi = a.nrange;
            while (hi - lo > 1) { const uint32_t mid = (lo + hi) >> 1; if (a.rpre[mid] <= s) lo = mid; else hi = mid; }
            s = a.rb[lo] + (s - a.rpre[lo]);
        }
        const uint32_t run = a.P.run[s];
        const uint32_t ne = a.P.ne[s];
        const uint64_t eo = a.P.eoff[s];
        const uint32_t nvid = a.P.nextv[s];                     // labels are < nvid
        const uint32_t nm = EMIT ? a.cnt[s] : 0u;
        const uint8_t active = a.active[run] && (!a.smask || a.smask[s]);
        const uint64_t budget = EMIT ? 0 : (uint64_t)a.budget[run];
        const uint64_t tally = EMIT ? 0 : tm.bcast(tm.leader() ? (uint64_t)a.run_acc[run] : 0ull);
        if (!active || (EMIT ? nm == 0 : tally > budget)) {
            if (!EMIT && tm.leader()) { a.cnt[s] = 0; a.state_edges[s] = 0; }
            continue;
        }
        const DRun& RN = a.runs[run];
        const DRule* rules = RN.rules;
        const uint32_t n_rules = RN.n_rules;
        tm.sync();
        for (uint32_t i = tm.r; i < nvid * NW; i += N) { inc0[i] = 0; inc1[i] = 0; }
        tm.sync();
        BitJoin<NW> J;
        J.inc0 = inc0; J.inc1 = inc1; J.ev = ev;
#pragma unroll
        for (uint32_t k = 0; k < NW; ++k) {
            J.loops.w[k] = 0;
            J.all.w[k] = ne >= 64 * (k + 1) ? ~0ull : ne > 64 * k ? (1ull << (ne - 64 * k)) - 1ull : 0ull;
        }
        for (uint32_t base = 0; base < ne; base += N) {
            const uint32_t e = base + tm.r;
            uint32_t x = 0, y = 1;
            if (e < ne) {
                if (A == 2) { const uint2 v = ((const uint2*)a.P.ev)[eo + e]; x = v.x; y = v.y; }
                else { x = a.P.ev[(eo + e) * A]; y = a.P.ev[(eo + e) * A + 1]; }
                ev[e] = (uint16_t)(x | y << 8);
                atomicOr((unsigned long long*)&inc0[x * NW + (e >> 6)], 1ull << (e & 63u));
                atomicOr((unsigned long long*)&inc1[y * NW + (e >> 6)], 1ull << (e & 63u));
            }
            const uint64_t lb = tm.ballot(e < ne && x == y) << (base & 63u);
#pragma unroll
            for (uint32_t k = 0; k < NW; ++k)
                if ((base >> 6) == k) J.loops.w[k] |= lb;
        }
        tm.sync();
        const uint64_t room = budget - tally;                  // count pass: matches the run may still take
        uint64_t total = 0;
        uint64_t edges_sum = 0;                                // count pass: edges of the children
        uint32_t out = EMIT ? (uint32_t)a.moff[s] : 0u;
        for (uint32_t r = 0; r < n_rules && (EMIT || total <= room); ++r) {
            const DRule& R = rules[r];
            if (!R.bits_ok) continue;                           // a pattern edge that is not binary
            const uint32_t n_lhs = R.n_lhs, child_ne = ne - n_lhs + R.n_rhs;
#pragma unroll
            for (int d = 0; d < 4; ++d) J.bj[d] = R.bj[d];
            // one rule's matches fit 32 bits (255 * 254 * 253 * 252); a sum past what is left has one
            // lane past its share, so the sum is formed only then
            const uint32_t left = (uint32_t)(room - total), share = left / N;
            uint32_t mine = 0;
            for (uint32_t base = 0; base < ne; base += N) {
                const uint32_t seed = base + tm.r;
                const uint32_t sv = seed < ne ? ev[seed] : 0u;
                const bool ok = seed < ne && (!(J.bj[0] & 256u) || (sv & 0xFFu) == sv >> 8);
                const uint32_t c = ok ? bit_join_any<NW, false>(J, n_lhs, seed, sv, RegJoinOut{}) : 0u;
                mine += c;
                if (!EMIT && tm.any(mine > share) && tm.sum(mine) > left) break;
                if constexpr (EMIT) {
                    uint32_t round;
                    const uint32_t inc = tm.incl_scan(c, round);
                    if (c) {
                        const RegJoinOut ro{a.M.q, a.M.K, out + inc - c, a.M.parent, a.M.rule, a.M.cne, s, r, child_ne};
                        bit_join_any<NW, true>(J, n_lhs, seed, sv, ro);
                    }
                    out += round;
                }
            }
            if constexpr (!EMIT) {
                const uint32_t sum = tm.sum(mine);
                total += sum;
                edges_sum += (uint64_t)sum * child_ne;
            }
        }
        if (!EMIT && tm.leader()) {
            a.cnt[s] = stored_count(total);
            a.state_edges[s] = edges_sum;
            // the run's shared tally: past what the run may still take its other states are skipped
            add_tally(a, run, budget != kNoBudget, total);
        }
    }
}

template <uint32_t NW>
static hipError_t launch_match_bits_nw(const MatchArgs& a, bool emit, uint32_t grid, uint32_t wpb, uint32_t lanes,
                                       hipStream_t st) {
    const dim3 g(grid), b(64 * wpb);
    const size_t lds = (size_t)a.lds_per_wave * wpb * (64 / lanes);
    switch (lanes + (emit ? 1 : 0)) {
        case 16: hipLaunchKernelGGL((k_match_bits<false, NW, 16>), g, b, lds, st, a); break;
        case 17: hipLaunchKernelGGL((k_match_bits<true, NW, 16>), g, b, lds, st, a); break;
        case 32: hipLaunchKernelGGL((k_match_bits<false, NW, 32>), g, b, lds, st, a); break;
        case 33: hipLaunchKernelGGL((k_match_bits<true, NW, 32>), g, b, lds, st, a); break;
        case 64: hipLaunchKernelGGL((k_match_bits<false, NW, 64>), g, b, lds, st, a); break;
        case 65: hipLaunchKernelGGL((k_match_bits<true, NW, 64>), g, b, lds, st, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

uint32_t launch_grid(uint32_t items, uint32_t wpb, uint32_t grid_cap);

hipError_t launch_match_bits(const MatchArgs& a, bool emit, uint32_t grid_cap, uint32_t wpb, hipStream_t st,
                             uint32_t lanes) {
    const uint32_t items = a.nrange ? a.n_items : a.P.n;
    if (!items) return hipSuccess;
    const uint32_t nw = match_bits_words(a.max_ne);
    if (!nw || a.max_nextv > kMatchBitsLabels || a.scratch || a.fwd_n || a.P.A < 2) return hipErrorInvalidValue;
    const uint32_t grid = launch_grid(items, wpb * (64 / lanes), grid_cap);
    return nw == 1 ? launch_match_bits_nw<1>(a, emit, grid, wpb, lanes, st)
           : nw == 2 ? launch_match_bits_nw<2>(a, emit, grid, wpb, lanes, st)
                     : launch_match_bits_nw<4>(a, emit, grid, wpb, lanes, st);
}

// ------------------------------------------------------------------------------------------
// The join over larger binary states, up to what the LDS holds (8 bytes an edge and 4 a label), by the W
// waves of a workgroup: the edges as vertex pairs in one word, and per (position, vertex) the list of
// its edges. A depth takes the shorter list of its bound positions and tests the other one, its
// binding words in registers (DRule::bj); a last depth with one bound position and nothing else to
// test counts its list's length less the edges in use. Matches and their order are k_match's: the
// emit pass puts every list in edge order. What bounded k_match here were the chains of LDS reads per
// candidate, and for states past its 25 bytes an edge of LDS a workspace in global memory.
// ------------------------------------------------------------------------------------------

struct ListJoin {
    const uint32_t* ev;        // edges: first vertex | second << 16
    const uint32_t* end;       // per vertex: end of its list at position 0 | at position 1 << 16
    const uint16_t* l0;
    const uint16_t* l1;
    uint32_t ne;
    uint32_t bj[4];
    uint64_t most;             // count pass: a seed with more matches is given up
};

// Matches of a seed: a hub's pass 32 bits from four pattern edges on; one that is written fits.
template <bool OUT>
using ListCount = std::conditional_t<OUT, uint32_t, uint64_t>;

template <int N, int D, bool OUT>
__device__ __forceinline__ ListCount<OUT> list_join(const ListJoin& J, Bound B, const RegJoinOut& o,
                                                    ListCount<OUT> found) {
    if constexpr (D == N) {
        if constexpr (OUT) {
            const size_t at = (size_t)(o.base + found);
            uint16_t* q = o.q + at * o.K;
            q[(J.bj[0] >> 12) & 3u] = (uint16_t)B.e0;
            if (N > 1) q[(J.bj[1] >> 12) & 3u] = (uint16_t)B.e1;
            if (N > 2) q[(J.bj[2] >> 12) & 3u] = (uint16_t)B.e2;
            if (N > 3) q[(J.bj[3] >> 12) & 3u] = (uint16_t)B.e3;
            o.parent[at] = o.state; o.rule[at] = o.rule_id; o.cne[at] = o.child_ne;
        }
        return found + 1;
    } else {
        const uint32_t b = J.bj[D];
        auto value = [&](uint32_t src) {                 // a bound position's vertex
            const uint32_t d = (src >> 1) & 3u;
            uint32_t x = B.v0;
            if (D > 1) { const uint32_t m = 0u - (uint32_t)(d == 1); x = (x & ~m) | (B.v1 & m); }
            if (D > 2) { const uint32_t m = 0u - (uint32_t)(d == 2); x = (x & ~m) | (B.v2 & m); }
            return (src & 8u) ? x >> 16 : x & 0xFFFFu;
        };
        const bool b0 = (b & 1u) != 0, b1 = (b & 16u) != 0, rep = (b & 256u) != 0;
        const uint32_t x0 = b0 ? value(b) : 0u, x1 = b1 ? value(b >> 4) : 0u;
        uint32_t lo = 0, hi = J.ne;
        const uint16_t* list = nullptr;
        if (b0) {
            lo = x0 ? J.end[x0 - 1] & 0xFFFFu : 0u;
            hi = J.end[x0] & 0xFFFFu;
            list = J.l0;
        }
        if (b1) {
            const uint32_t lo1 = x1 ? J.end[x1 - 1] >> 16 : 0u, hi1 = J.end[x1] >> 16;
            if (!b0 || hi1 - lo1 < hi - lo) { lo = lo1; hi = hi1; list = J.l1; }
        }
        if constexpr (D + 1 == N && !OUT) {
            if (b0 != b1 && !rep) {
                // the list less the edges in use that are on it
                auto on = [&](uint32_t v) { return b0 ? (v & 0xFFFFu) == x0 : v >> 16 == x1; };
                uint32_t c = hi - lo - (on(B.v0) ? 1u : 0u);
                if (D > 1) c -= on(B.v1) ? 1u : 0u;
                if (D > 2) c -= on(B.v2) ? 1u : 0u;
                return found + c;
            }
        }
        for (uint32_t j = lo; j < hi; ++j) {
            const uint32_t e = list ? (uint32_t)list[j] : j;
            const uint32_t v = J.ev[e];
            bool ok = e != B.e0;
            if (D > 1) ok &= e != B.e1;
            if (D > 2) ok &= e != B.e2;
            ok &= !b0 || (v & 0xFFFFu) == x0;
            ok &= !b1 || v >> 16 == x1;
            ok &= !rep || (v & 0xFFFFu) == v >> 16;
            if (!ok) continue;
            B.template set<D>(e, v);
            found = list_join<N, D + 1, OUT>(J, B, o, found);
            if (!OUT && D + 1 < N && found > J.most) return found;
        }
        return found;
    }
}

template <bool OUT>
__device__ __forceinline__ ListCount<OUT> list_join_any(const ListJoin& J, uint32_t n_lhs, uint32_t seed, uint32_t sv,
                                                        const RegJoinOut& o) {
    const Bound B{seed, 0, 0, 0, sv, 0, 0, 0};
    switch (n_lhs) {
        case 1: return list_join<1, 1, OUT>(J, B, o, 0u);
        case 2: return list_join<2, 1, OUT>(J, B, o, 0u);
        case 3: return list_join<3, 1, OUT>(J, B, o, 0u);
        default: return list_join<4, 1, OUT>(J, B, o, 0u);
    }
}

// Workspace: edges, list ends, the two lists, a bit per edge and the lists above 16 entries (emit).
struct ListSizes {
    uint32_t NE, NL, NB, NH;
    __host__ __device__ static ListSizes make(uint32_t ne, uint32_t nl) {
        return ListSizes{ne, nl, (ne + 31) / 32, 2 * ne / 17 + 1};
    }
    __host__ __device__ uint32_t bytes() const {
        auto al = [](uint32_t b) { return (b + 7u) & ~7u; };
        return al(4 * NE) + al(4 * (NL + 1)) + 2 * al(2 * NE) + al(4 * NB) + al(4 * NH) + 16 + 128;
    }
};

// The list [lo, hi) of l into ascending order (edge ids are distinct), by the workgroup: marked in a bit
// set and read back in order.
template <class TM>
__device__ __forceinline__ void sort_list_bits(const TM& tm, uint16_t* l, uint32_t lo, uint32_t hi, uint32_t* bits,
                                               uint32_t nb) {
    for (uint32_t i = tm.r; i < nb; i += TM::N) bits[i] = 0;
    tm.sync();
    for (uint32_t j = lo + tm.r; j < hi; j += TM::N) atomicOr(&bits[l[j] >> 5], 1u << (l[j] & 31u));
    tm.sync();
    uint32_t at = lo;
    for (uint32_t base = 0; base < nb; base += TM::N) {
        const uint32_t i = base + tm.r;
        uint32_t w = i < nb ? bits[i] : 0u, round;
        uint32_t o = (uint32_t)__popc(w);
        o = at + tm.incl_scan(o, round) - o;
        for (; w; w &= w - 1) l[o++] = (uint16_t)(i * 32 + (uint32_t)__builtin_ctz(w));
        at += round;
    }
    tm.sync();
}

template <bool EMIT, uint32_t W>
__global__ __launch_bounds__(64 * W) void k_match_lists(MatchArgs a) {
    extern __shared__ uint8_t lds[];
    constexpr uint32_t N = 64 * W;
    const ListSizes z = ListSizes::make(a.max_ne, a.max_nextv);
    uint8_t* p = lds;
    uint32_t* ev = (uint32_t*)carve(p, 4 * z.NE);
    uint32_t* end = (uint32_t*)carve(p, 4 * (z.NL + 1));
    uint16_t* l0 = (uint16_t*)carve(p, 2 * z.NE);
    uint16_t* l1 = (uint16_t*)carve(p, 2 * z.NE);
    uint32_t* bits = (uint32_t*)carve(p, 4 * z.NB);
    uint32_t* hubs = (uint32_t*)carve(p, 4 * z.NH);
    uint32_t* word = (uint32_t*)carve(p, 16);
    const Team<W> tm((uint64_t*)carve(p, 128));
    const uint32_t l = tm.r, A = a.P.A;
    const uint32_t n_items = a.nrange ? a.n_items : a.P.n;
    const bool spread = !EMIT && a.spread > 1;
    const uint32_t nblk = (n_items + kCountSpreadBlock - 1) / kCountSpreadBlock;
    const uint32_t n_loop = spread ? nblk * kCountSpreadBlock : n_items;
    for (uint32_t ls = blockIdx.x; ls < n_loop; ls += gridDim.x) {
        uint32_t s = ls;
        if (spread) {
            s = (uint32_t)((uint64_t)(ls / kCountSpreadBlock) * a.spread % nblk) * kCountSpreadBlock +
                ls % kCountSpreadBlock;
            if (s >= n_items) continue;                         // the last block's tail
        }
        if (a.nrange) {                                         // subset: logical -> state
            uint32_t lo = 0, hi = a.nrange;
            while (hi - lo > 1) { const uint32_t mid = (lo + hi) >> 1; if (a.rpre[mid] <= s) lo = mid; else hi = mid; }
            s = a.rb[lo] + (s - a.rpre[lo]);
        }
        const uint32_t run = a.P.run[s];
        const uint32_t ne = a.P.ne[s];
        const uint64_t eo = a.P.eoff[s];
        const uint32_t nvid = a.P.nextv[s];                     // labels are < nvid
        const uint8_t active = a.active[run] && (!a.smask || a.smask[s]);
        const uint64_t budget = EMIT ? 0 : (uint64_t)a.budget[run];
        // one read of the run's tally, which moves under other workgroups, for all of the team
        const uint64_t tally = EMIT ? 0 : tm.bcast(l == 0 ? (uint64_t)a.run_acc[run] : 0ull);
        if (!active || (EMIT ? a.cnt[s] == 0 : tally > budget)) {
            if (!EMIT && l == 0) { a.cnt[s] = 0; a.state_edges[s] = 0; }
            continue;
        }
        tm.sync();
        for (uint32_t v = l; v <= nvid; v += N) end[v] = 0;
        if (l == 0) word[0] = 0;
        tm.sync();
        for (uint32_t e = l; e < ne; e += N) {
            uint32_t x, y;
            if (A == 2) { const uint2 v = ((const uint2*)a.P.ev)[eo + e]; x = v.x; y = v.y; }
            else { x = a.P.ev[(eo + e) * A]; y = a.P.ev[(eo + e) * A + 1]; }
            ev[e] = x | y << 16;
            atomicAdd(&end[x], 1u);
            atomicAdd(&end[y], 1u << 16);
        }
        tm.sync();
        tm.excl_scan_lds(end, nvid + 1);        // both positions' counts at once: neither sum passes 16 bits
        for (uint32_t e = l; e < ne; e += N) {
            const uint32_t v = ev[e];
            l0[atomicAdd(&end[v & 0xFFFFu], 1u) & 0xFFFFu] = (uint16_t)e;
            l1[atomicAdd(&end[v >> 16], 1u << 16) >> 16] = (uint16_t)e;
        }
        tm.sync();
        if constexpr (EMIT) {
            // every list into edge order: up to 16 entries by a lane, to 64 by a wave, longer ones by
            // the workgroup
            for (uint32_t i = l; i < 2 * nvid; i += N) {
                const uint32_t v = i >> 1, sh = (i & 1u) * 16;
                const uint32_t lo = v ? (end[v - 1] >> sh) & 0xFFFFu : 0u, hi = (end[v] >> sh) & 0xFFFFu;
                if (hi - lo < 2) continue;
                if (hi - lo > 16) { hubs[atomicAdd(&word[0], 1u)] = i; continue; }
                uint16_t* q = sh ? l1 : l0;
                for (uint32_t j = lo + 1; j < hi; ++j) {
                    const uint16_t x = q[j];
                    uint32_t k = j;
                    while (k > lo && q[k - 1] > x) { q[k] = q[k - 1]; --k; }
                    q[k] = x;
                }
            }
            tm.sync();
            const uint32_t nh = word[0];
            for (uint32_t k = l / WAVE; k < nh; k += W) {
                const uint32_t i = hubs[k], v = i >> 1, sh = (i & 1u) * 16;
                const uint32_t lo = v ? (end[v - 1] >> sh) & 0xFFFFu : 0u, n = ((end[v] >> sh) & 0xFFFFu) - lo;
                if (n > WAVE) continue;
                uint16_t* q = sh ? l1 : l0;
                const uint32_t ln = lane_id(), un = (uint32_t)__builtin_amdgcn_readfirstlane((int)n);
                const uint32_t x = ln < n ? q[lo + ln] : 0xFFFFFFFFu;
                uint32_t r = 0;
                for (uint32_t j = 0; j < un; ++j) r += (uint32_t)__builtin_amdgcn_readlane((int)x, (int)j) < x ? 1u : 0u;
                if (ln < n) q[lo + r] = (uint16_t)x;
            }
            for (uint32_t k = 0; k < nh; ++k) {
                const uint32_t i = hubs[k], v = i >> 1, sh = (i & 1u) * 16;
                const uint32_t lo = v ? (end[v - 1] >> sh) & 0xFFFFu : 0u, hi = (end[v] >> sh) & 0xFFFFu;
                if (hi - lo > WAVE) sort_list_bits(tm, sh ? l1 : l0, lo, hi, bits, (ne + 31) / 32);
            }
            tm.sync();
        }
        const DRun& RN = a.runs[run];
        ListJoin J;
        J.ev = ev; J.end = end; J.l0 = l0; J.l1 = l1; J.ne = ne;
        const uint64_t room = budget - tally;                  // count pass: matches the run may still take
        uint64_t total = 0;
        uint64_t edges_sum = 0;                                // count pass: edges of the children
        uint32_t out = EMIT ? (uint32_t)a.moff[s] : 0u;
        for (uint32_t r = 0; r < RN.n_rules && (EMIT || total <= room); ++r) {
            const DRule& R = RN.rules[r];
            if (!R.bits_ok) continue;                           // a pattern edge that is not binary
            const uint32_t n_lhs = R.n_lhs, child_ne = ne - n_lhs + R.n_rhs;
#pragma unroll
            for (int d = 0; d < 4; ++d) J.bj[d] = R.bj[d];
            const uint64_t left = room - total;
            uint64_t mine = 0;
            J.most = EMIT ? kNoBudget : left;
            for (uint32_t base = 0; base < ne; base += N) {
                const uint32_t seed = base + l;
                const uint32_t sv = seed < ne ? ev[seed] : 0u;
                const bool ok = seed < ne && (!(J.bj[0] & 256u) || (sv & 0xFFFFu) == sv >> 16);
                const uint64_t c = ok ? list_join_any<false>(J, n_lhs, seed, sv, RegJoinOut{}) : 0u;
                mine += c;
                // a sum past what is left has one lane past its share; looked at after rounds 1, 2, 4, ..
                // (12,001 edges, 12 rounds: after each one cost the count pass 1 % of a step)
                if (!EMIT && base + N < ne && ((base / N) & (base / N + 1)) == 0 && tm.any(mine > left / N) &&
                    tm.sum64(mine) > left)
                    break;
                if constexpr (EMIT) {
                    uint32_t round;
                    const uint32_t inc = tm.incl_scan((uint32_t)c, round);
                    if (c) {
                        const RegJoinOut ro{a.M.q, a.M.K, out + inc - (uint32_t)c, a.M.parent, a.M.rule, a.M.cne, s, r,
                                            child_ne};
                        list_join_any<true>(J, n_lhs, seed, sv, ro);
                    }
                    out += round;
                }
            }
            if constexpr (!EMIT) {
                const uint64_t sum = tm.sum64(mine);
                total += sum;
                edges_sum += sum * child_ne;
            }
        }
        if (!EMIT && l == 0) {
            a.cnt[s] = stored_count(total);
            a.state_edges[s] = edges_sum;
            add_tally(a, run, budget != kNoBudget, total);
        }
    }
}

uint32_t match_lists_lds(uint32_t max_ne, uint32_t max_nextv) {
    return (ListSizes::make(max_ne, max_nextv).bytes() + 15u) & ~15u;
}

hipError_t launch_match_lists(const MatchArgs& a, bool emit, uint32_t grid, uint32_t team, hipStream_t st) {
    const uint32_t items = a.nrange ? a.n_items : a.P.n;
    if (!items) return hipSuccess;
    if (a.max_ne > 65535 || a.max_nextv > 65535 || a.scratch || a.fwd_n || a.P.A < 2) return hipErrorInvalidValue;
    const dim3 g(grid);
    const size_t lds = a.lds_per_wave;
    switch (team * 2 + (emit ? 1 : 0)) {
        case 16: hipLaunchKernelGGL((k_match_lists<false, 8>), g, dim3(512), lds, st, a); break;
        case 17: hipLaunchKernelGGL((k_match_lists<true, 8>), g, dim3(512), lds, st, a); break;
        case 32: hipLaunchKernelGGL((k_match_lists<false, 16>), g, dim3(1024), lds, st, a); break;
        case 33: hipLaunchKernelGGL((k_match_lists<true, 16>), g, dim3(1024), lds, st, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// Rewrite + hash, one team per child, then the children's records (Rewriter::apply,
// hypergraph/src/rewriter.cpp:11-205, with hgcommon rewrite semantics rewrite_core.hpp:53-87).
// ------------------------------------------------------------------------------------------

// A slot is read before it is claimed: most children repeat a hash already in the map, and a
// plain load that finds it (or another key: keys are only ever written once, 0 -> key) settles
// the probe without an atomic; only an empty-looking slot is claimed by compare-and-swap, whose
// result is authoritative if the load was stale.
__device__ inline bool map_insert(DRun* run, uint64_t h) {
    if (h == 0) return atomicExch(&run->zero_seen, 1u) == 0u;
    const uint32_t mask = run->map_mask;
    uint32_t i = (uint32_t)mix64(h) & mask;
    while (true) {
        // device scope is enough: only this device reads and claims the map
        uint64_t old = __hip_atomic_load(&run->map_keys[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (old == 0)
            old = atomicCAS((unsigned long long*)&run->map_keys[i], 0ull, (unsigned long long)h);
        if (old == 0) return true;
        if (old == h) return false;
        i = (i + 1) & mask;
    }
}

// The hash h of given state i: stored and, for a root, inserted into its run's state map.
__device__ inline void wl_state_done(const WLStatesArgs& a, uint32_t i, uint64_t h) {
    a.out[i] = h;
    if (a.run_of) {
        DRun* RN = &a.runs[a.run_of[i]];
        if (map_insert(RN, h)) {
            atomicAdd((unsigned long long*)&a.ctr[(size_t)a.run_of[i] * CTR_N + CTR_CANON], 1ull);
            atomicAdd((unsigned long long*)&a.ctr[(size_t)a.run_of[i] * CTR_N + CTR_FINGERPRINT],
                      (unsigned long long)mix64(h));
        }
    }
}

// GWS selects the workspace at compile time (global scratch for states too large for LDS), so
// the LDS variant addresses its workspace with LDS instructions rather than flat ones. W is the
// team: W = 1, one wave per child (up to four per workgroup, each with its own workspace);
// W > 1, the workgroup's W waves share one child and one workspace, for large children whose
// workspace would otherwise leave a CU one or two waves. One-wave teams are held to four waves
// per SIMD (about 100 registers, none spilled). When this kernel took the batched workload's
// children too (k_expand_small does now), its expansion was 9.8 ms so, 15.3 ms at three waves and
// 11.1 ms at five.
template <bool GWS, uint32_t W, uint32_t G>
__global__ __launch_bounds__(W == 1 ? 256 : 64 * W, W == 1 ? 4 : 1) void k_expand(ExpandArgs a) {
    using TM = typename TeamSel<W, G>::type;
    extern __shared__ uint8_t lds[];
    const uint32_t tpb = W == 1 ? (blockDim.x / WAVE) * (WAVE / G) : 1;   // teams per workgroup
    const uint32_t w = W == 1 ? threadIdx.x / G : 0;                       // team within the workgroup
    uint8_t* my;
    if constexpr (GWS) my = a.scratch + ((size_t)blockIdx.x * tpb + w) * a.lds_per_wave;
    else my = lds + (size_t)w * a.lds_per_wave;
    const TM tm((uint64_t*)(my + a.lds_per_wave - 64));   // a wave team's reduction words: the last 64 bytes
    const uint32_t PA = a.P.A, A = a.C.A;                  // parent / child vertex strides
    const WLSizes z = expand_sizes(a.max_child_ne, a.max_nv, a.max_nextv, A, a.lean != 0);
    WLSpace s;
    uint8_t* p = my;
    wl_bind(s, p, z, A);
    // Child vertex labels and the label -> local id map live in the hash's srt and nbr regions,
    // which the hash only writes after they are read.
    uint32_t* gv = (uint32_t*)s.srt;                      // [NE * A]
    uint32_t* vmap = (uint32_t*)s.nbr;                    // [max_nextv + 1]

    // Children in chunks of kChunk consecutive ones, dealt round-robin to the teams (2 measured
    // best of 1, 2, 4 and contiguous per-team blocks on the batched workload; 1 and 2 measure
    // alike since the run counters left this kernel): a chunk keeps neighbouring children (one
    // parent) on one team, and the dealing spreads large and small requests' children over all
    // teams.
    constexpr uint32_t kChunk = 2;
    const uint32_t gw = xcd_block() * tpb + w, nw = gridDim.x * tpb;
    uint32_t rr = 0;                                       // range of logical index c (subsets)


    for (uint32_t lc = gw * kChunk; lc < a.n_items; lc += (lc % kChunk == kChunk - 1) ? (nw - 1) * kChunk + 1 : 1) {
        uint32_t c = lc;
        if (a.nrange) {
            if (lc % kChunk == 0 || lc == gw * kChunk) {       // a new chunk: find its range
                uint32_t lo = 0, hi = a.nrange;
                while (hi - lo > 1) { const uint32_t mid = (lo + hi) >> 1; if (a.rpre[mid] <= lc) lo = mid; else hi = mid; }
                rr = lo;
            }
            while (lc >= a.rpre[rr + 1]) ++rr;
            c = a.rb[rr] + (lc - a.rpre[rr]);
        }
        const uint32_t par = a.M.parent[c];
        const uint32_t rid = a.M.rule[c];
        const uint32_t run = a.P.run[par];
        const DRule& R = a.runs[run].rules[rid];
        const uint32_t nl = R.n_lhs, nr = R.n_rhs;
        const uint32_t pne = a.P.ne[par];
        const uint64_t peo = a.P.eoff[par];
        const uint64_t ceo = a.C.eoff[c];
        const uint32_t cne = pne - nl + nr;
        const uint32_t pdep = a.P.depth[par];
        const uint32_t step = pdep + 1;                       // generation of the child
        const uint16_t* q = a.M.q + (size_t)c * a.M.K;
        // Parent edges minus the consumed ones, order kept (SparseBitset::derive).
        uint32_t kept = 0;
        for (uint32_t base = 0; base < pne; base += TM::N) {
            const uint32_t i = base + tm.r;
            bool keep = i < pne;
            if (keep) for (uint32_t t = 0; t < nl; ++t) keep &= (q[t] != i);
            uint32_t n_round;
            const uint32_t at = tm.compact(keep, n_round);
            if (keep) {
                const uint32_t pos = kept + at;
                const uint8_t ar = a.P.ar[peo + i];
                for (uint32_t k = 0; k < A; ++k) {
                    const uint32_t v = k < PA ? a.P.ev[(peo + i) * PA + k] : 0u;
                    a.C.ev[(ceo + pos) * A + k] = v;
                    gv[pos * A + k] = v;
                }
                a.C.ar[ceo + pos] = ar;
                a.C.ps[ceo + pos] = a.P.ps[peo + i];
                s.e_ar[pos] = ar;
            }
            kept += n_round;
        }
        // Produced edges in RHS order; fresh vertices ascending by variable
        // (assign_fresh_consecutive / resolve_rhs_vertices, rewrite_core.hpp:53-87).
        const uint32_t fresh_base = a.P.nextv[par];
        if (tm.r < nr) {
            const uint32_t pos = kept + tm.r;
            const uint32_t ra = R.ra[tm.r];
            for (uint32_t k = 0; k < A; ++k) {
                uint32_t v = 0;
                if (k < ra) {
                    const uint32_t var = R.rv[tm.r][k];
                    if (R.lhs_mask & (1u << var)) {
                        const uint32_t se = q[R.var_src_edge[var]];
                        v = a.P.ev[(peo + se) * PA + R.var_src_pos[var]];
                    } else {
                        v = fresh_base + __popc(R.new_mask & ((1u << var) - 1u));
                    }
                }
                a.C.ev[(ceo + pos) * A + k] = v;
                gv[pos * A + k] = v;
            }
            a.C.ar[ceo + pos] = (uint8_t)ra;
            a.C.ps[ceo + pos] = (uint8_t)step;
            s.e_ar[pos] = (uint8_t)ra;
        }
        tm.sync();
        // Local vertex numbering: ascending label, as the reference's sorted vertex list.
        const uint32_t nextv = fresh_base + R.n_new;
        for (uint32_t v = tm.r; v <= nextv; v += TM::N) vmap[v] = 0;
        tm.sync();
        for (uint32_t e = tm.r; e < cne; e += TM::N)
            for (uint32_t k = 0; k < s.e_ar[e]; ++k) vmap[gv[e * A + k]] = 1;
        tm.sync();
        const uint32_t nv = tm.excl_scan_lds(vmap, nextv + 1);
        for (uint32_t e = tm.r; e < cne; e += TM::N)
            for (uint32_t k = 0; k < A; ++k) s.e_lv[e * A + k] = (uint16_t)(k < s.e_ar[e] ? vmap[gv[e * A + k]] : 0);
        s.nE = cne;
        s.nV = nv;
        tm.sync();
        const uint64_t h = wl_hash_team(s, tm);
        if (tm.leader()) a.C.hash[c] = h;              // the child's other records: k_record
        tm.sync();
    }
}

// k_expand for small children of one arity (at most kSmallMaxEdges edges and kSmallMaxLabels labels, a stride of
// at most 4): the same child, with the hash of hgx_wl_small.hpp. Labels are bytes, so the rewrite leaves its edges in LDS as the hash reads them;
// a kept edge's place is its position less the consumed positions below it (two words of bits), so
// the copy needs no compaction and its loads do not wait for each other.
template <uint32_t UA, uint32_t G>
__global__ __launch_bounds__(256, 5) void k_expand_small(ExpandArgs a) {
    using TM = typename TeamSel<1, G>::type;
    extern __shared__ uint8_t lds[];
    const uint32_t tpb = (blockDim.x / WAVE) * (WAVE / G);                 // teams per workgroup
    const uint32_t w = threadIdx.x / G;
    const TM tm(nullptr);
    const uint32_t l = tm.r;
    const uint32_t PA = UA ? UA : a.P.A, A = UA ? UA : a.C.A;              // parent / child vertex strides
    SmallSpace s;
    small_bind(s, lds + (size_t)w * a.lds_per_wave, SmallSizes::make(a.max_child_ne, a.max_nextv, A), A);

    // Children in chunks of a.chunk consecutive ones, dealt round-robin to the teams: 2 keep a
    // parent's neighbouring children on one team, 1 where the launch has a team for every child.
    const uint32_t chunk = a.chunk;
    const uint32_t gw = xcd_block() * tpb + w, nw = gridDim.x * tpb;
    uint32_t rr = 0;
    for (uint32_t lc = gw * chunk, at = 0; lc < a.n_items;) {
        uint32_t c = lc;
        if (a.nrange) {
            if (at == 0) {                                     // a new chunk: find its range
                uint32_t lo = 0, hi = a.nrange;
                while (hi - lo > 1) { const uint32_t mid = (lo + hi) >> 1; if (a.rpre[mid] <= lc) lo = mid; else hi = mid; }
                rr = lo;
            }
            while (lc >= a.rpre[rr + 1]) ++rr;
            c = a.rb[rr] + (lc - a.rpre[rr]);
        }
        if (++at == chunk) { at = 0; lc += (nw - 1) * chunk + 1; } else ++lc;
        const uint32_t par = a.M.parent[c];
        const uint32_t rid = a.M.rule[c];
        const uint64_t ceo = a.C.eoff[c];
        const uint32_t q_t = l < a.M.K ? a.M.q[(size_t)c * a.M.K + l] : 0u;     // consumed position l
        const uint32_t run = a.P.run[par];
        const uint32_t pne = a.P.ne[par];
        const uint64_t peo = a.P.eoff[par];
        const uint32_t fresh_base = a.P.nextv[par];
        const uint32_t step = a.P.depth[par] + 1u;            // generation of the child
        const DRule& R = a.runs[run].rules[rid];
        const uint32_t nl = R.n_lhs, nr = R.n_rhs;
        const uint32_t ua = UA ? UA : R.la[0];
        const uint32_t cne = pne - nl + nr, kept = pne - nl;
        uint64_t used[4] = {0, 0, 0, 0};                       // consumed positions (below 256)
        for (uint32_t t = 0; t < nl; ++t) {
            const uint32_t q = tm.shfl(q_t, t);
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
                if ((q >> 6) == k) used[k] |= 1ull << (q & 63u);
        }
        // parent edges minus the consumed ones, order kept (SparseBitset::derive)
        for (uint32_t i = l; i < pne; i += TM::N) {
            const uint32_t iw = i >> 6;
            uint32_t below = 0;
            bool keep = true;
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                const uint64_t low = iw > k ? ~0ull : iw == k ? (1ull << (i & 63u)) - 1ull : 0ull;
                below += (uint32_t)__popcll(used[k] & low);
                if (iw == k) keep = !((used[k] >> (i & 63u)) & 1ull);
            }
            if (!keep) continue;
            const uint32_t pos = i - below;
            if constexpr (UA == 2) {
                const uint2 v = ((const uint2*)a.P.ev)[peo + i];
                ((uint2*)a.C.ev)[ceo + pos] = v;
                ((uint16_t*)s.ev)[pos] = (uint16_t)(v.x | (v.y << 8));
            } else {
                for (uint32_t k = 0; k < A; ++k) {
                    const uint32_t v = k < PA ? a.P.ev[(peo + i) * PA + k] : 0u;
                    a.C.ev[(ceo + pos) * A + k] = v;
                    if (k < ua) s.ev[pos * ua + k] = (uint8_t)v;
                }
            }
            a.C.ar[ceo + pos] = (uint8_t)ua;
            a.C.ps[ceo + pos] = a.P.ps[peo + i];
        }
        // produced edges in RHS order; fresh vertices ascending by variable
        // (assign_fresh_consecutive / resolve_rhs_vertices, rewrite_core.hpp:53-87)
        for (uint32_t base = 0; base < nr; base += TM::N) {
            const uint32_t t = base + l;
            const uint32_t pos = kept + t;
            for (uint32_t k = 0; k < A; ++k) {
                uint32_t v = 0, se = 0, var = 0;
                const bool in = t < nr && k < ua;
                if (in) {
                    var = R.rv[t][k];
                    se = R.var_src_edge[var];
                }
                const uint32_t q = tm.shfl(q_t, se);           // every lane of the team takes part
                if (in) {
                    if (R.lhs_mask & (1u << var)) v = a.P.ev[(peo + q) * PA + R.var_src_pos[var]];
                    else v = fresh_base + __popc(R.new_mask & ((1u << var) - 1u));
                    s.ev[pos * ua + k] = (uint8_t)v;
                }
                if (t < nr) a.C.ev[(ceo + pos) * A + k] = v;
            }
            if (t < nr) {
                a.C.ar[ceo + pos] = (uint8_t)ua;
                a.C.ps[ceo + pos] = (uint8_t)step;
            }
        }
        tm.sync();
        const uint32_t nextv = fresh_base + R.n_new;
        const uint64_t h = wl_hash_small<UA>(s, tm, cne, nextv, ua);
        if (tm.leader()) a.C.hash[c] = h;              // the child's other records: k_record
        tm.sync();
    }
}

// k_expand for large children of one arity (past k_expand_small's limits, within hgx_wl_large.hpp's): the
// W waves of a workgroup rewrite one child and hash it with its colours in LDS. ALL: every array of the
// hash in LDS, else the ones walked in order in a slice of a.scratch per workgroup.
template <uint32_t UA, uint32_t W, bool ALL>
__global__ __launch_bounds__(64 * W) void k_expand_large(ExpandArgs a) {
    extern __shared__ uint8_t lds[];
    const uint32_t PA = UA ? UA : a.P.A, A = UA ? UA : a.C.A;              // parent / child vertex strides
    const LargeSizes z = LargeSizes::make(a.max_child_ne, a.max_nextv, A);
    LargeSpace s;
    large_bind<ALL>(s, lds, ALL ? nullptr : a.scratch + (size_t)blockIdx.x * z.rest(), z);
    const Team<W> tm(s.red);
    const uint32_t l = tm.r;
    for (uint32_t lc = xcd_block(); lc < a.n_items; lc += gridDim.x) {
        uint32_t c = lc;
        if (a.nrange) {
            uint32_t lo = 0, hi = a.nrange;
            while (hi - lo > 1) { const uint32_t mid = (lo + hi) >> 1; if (a.rpre[mid] <= lc) lo = mid; else hi = mid; }
            c = a.rb[lo] + (lc - a.rpre[lo]);
        }
        const uint32_t par = a.M.parent[c];
        const uint64_t ceo = a.C.eoff[c];
        const uint32_t run = a.P.run[par];
        const uint32_t pne = a.P.ne[par];
        const uint64_t peo = a.P.eoff[par];
        const uint32_t fresh_base = a.P.nextv[par];
        const DRule& R = a.runs[run].rules[a.M.rule[c]];
        const uint32_t nl = R.n_lhs, nr = R.n_rhs;
        const uint32_t ua = UA ? UA : R.la[0];
        const uint32_t cne = pne - nl + nr, kept = pne - nl;
        if (l < nl) s.q[l] = a.M.q[(size_t)c * a.M.K + l];
        tm.sync();
        // parent edges minus the consumed ones, order kept (SparseBitset::derive)
        for (uint32_t i = l; i < pne; i += 64 * W) {
            bool keep = true;
            uint32_t pos = i;
            for (uint32_t t = 0; t < nl; ++t) {
                const uint32_t q = s.q[t];
                keep &= q != i;
                pos -= q < i ? 1u : 0u;
            }
            if (!keep) continue;
            if constexpr (UA == 2) {
                ((uint2*)a.C.ev)[ceo + pos] = ((const uint2*)a.P.ev)[peo + i];
            } else {
                for (uint32_t k = 0; k < A; ++k) a.C.ev[(ceo + pos) * A + k] = k < PA ? a.P.ev[(peo + i) * PA + k] : 0u;
            }
            a.C.ar[ceo + pos] = (uint8_t)ua;
            a.C.ps[ceo + pos] = a.P.ps[peo + i];
        }
        // produced edges in RHS order; fresh vertices ascending by variable
        // (assign_fresh_consecutive / resolve_rhs_vertices, rewrite_core.hpp:53-87)
        if (l < nr) {
            const uint32_t pos = kept + l;
            for (uint32_t k = 0; k < A; ++k) {
                uint32_t v = 0;
                if (k < ua) {
                    const uint32_t var = R.rv[l][k];
                    if (R.lhs_mask & (1u << var)) v = a.P.ev[(peo + s.q[R.var_src_edge[var]]) * PA + R.var_src_pos[var]];
                    else v = fresh_base + __popc(R.new_mask & ((1u << var) - 1u));
                }
                a.C.ev[(ceo + pos) * A + k] = v;
            }
            a.C.ar[ceo + pos] = (uint8_t)ua;
            a.C.ps[ceo + pos] = (uint8_t)(a.P.depth[par] + 1u);
        }
        tm.sync();
        const uint64_t h = wl_hash_large<UA, ALL>(s, tm, a.C.ev + ceo * A, A, cne, fresh_base + R.n_new, ua);
        if (tm.leader()) a.C.hash[c] = h;              // the child's other records: k_record
        tm.sync();
    }
}

// The hash of given states of one arity each, within the same limits.
template <uint32_t UA, uint32_t W, bool ALL>
__global__ __launch_bounds__(64 * W) void k_wl_large(WLStatesArgs a) {
    extern __shared__ uint8_t lds[];
    const uint32_t A = UA ? UA : a.A;
    const LargeSizes z = LargeSizes::make(a.max_ne, a.max_nv, A);
    LargeSpace s;
    large_bind<ALL>(s, lds, ALL ? nullptr : a.scratch + (size_t)blockIdx.x * z.rest(), z);
    const Team<W> tm(s.red);
    for (uint32_t i = blockIdx.x; i < a.n; i += gridDim.x) {
        const uint64_t e0 = a.state_off[i];
        const uint32_t ne = (uint32_t)(a.state_off[i + 1] - e0);
        tm.sync();
        const uint64_t h = wl_hash_large<UA, ALL>(s, tm, a.ev + e0 * A, A, ne, a.nv[i], UA ? UA : ne ? a.ar[e0] : 2u);
        if (tm.leader()) wl_state_done(a, i, h);
    }
}

uint32_t large_lds(uint32_t max_ne, uint32_t max_nextv, uint32_t A, bool all) {
    const LargeSizes z = LargeSizes::make(max_ne, max_nextv, A);
    return (z.hot() + (all ? z.rest() : 0u) + 15u) & ~15u;
}
uint32_t large_scratch(uint32_t max_ne, uint32_t max_nextv, uint32_t A) { return LargeSizes::make(max_ne, max_nextv, A).rest(); }

template <uint32_t UA, uint32_t W>
static hipError_t launch_expand_large_w(const ExpandArgs& a, uint32_t grid, hipStream_t st) {
    if (a.scratch) hipLaunchKernelGGL((k_expand_large<UA, W, false>), dim3(grid), dim3(64 * W), a.lds_per_wave, st, a);
    else hipLaunchKernelGGL((k_expand_large<UA, W, true>), dim3(grid), dim3(64 * W), a.lds_per_wave, st, a);
    return hipGetLastError();
}

hipError_t launch_expand_large(const ExpandArgs& a, uint32_t grid, uint32_t team, hipStream_t st) {
    if (!a.n_items) return hipSuccess;
    if (!a.lean || a.C.A > 4 || !large_fits(a.max_child_ne, a.max_nextv, a.C.A)) return hipErrorInvalidValue;
    const bool two = a.P.A == 2 && a.C.A == 2;
    switch (team) {
        case 4: return two ? launch_expand_large_w<2, 4>(a, grid, st) : launch_expand_large_w<0, 4>(a, grid, st);
        case 8: return two ? launch_expand_large_w<2, 8>(a, grid, st) : launch_expand_large_w<0, 8>(a, grid, st);
        case 16: return two ? launch_expand_large_w<2, 16>(a, grid, st) : launch_expand_large_w<0, 16>(a, grid, st);
        default: return hipErrorInvalidValue;
    }
}

template <uint32_t UA, uint32_t W>
static hipError_t launch_wl_large_w(const WLStatesArgs& a, uint32_t grid, hipStream_t st) {
    if (a.scratch) hipLaunchKernelGGL((k_wl_large<UA, W, false>), dim3(grid), dim3(64 * W), a.lds_per_wave, st, a);
    else hipLaunchKernelGGL((k_wl_large<UA, W, true>), dim3(grid), dim3(64 * W), a.lds_per_wave, st, a);
    return hipGetLastError();
}

hipError_t launch_wl_large(const WLStatesArgs& a, uint32_t grid, uint32_t team, hipStream_t st) {
    if (!a.n) return hipSuccess;
    if (!a.lean || a.A > 4 || !large_fits(a.max_ne, a.max_nv, a.A)) return hipErrorInvalidValue;
    switch (team) {
        case 4: return a.A == 2 ? launch_wl_large_w<2, 4>(a, grid, st) : launch_wl_large_w<0, 4>(a, grid, st);
        case 8: return a.A == 2 ? launch_wl_large_w<2, 8>(a, grid, st) : launch_wl_large_w<0, 8>(a, grid, st);
        case 16: return a.A == 2 ? launch_wl_large_w<2, 16>(a, grid, st) : launch_wl_large_w<0, 16>(a, grid, st);
        default: return hipErrorInvalidValue;
    }
}

__global__ void k_fill(uint8_t* p, uint32_t word, uint64_t words, uint64_t bytes) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t w = i; w < words; w += stride) ((uint32_t*)p)[w] = word;
    if (i < bytes - words * 4) p[words * 4 + i] = (uint8_t)word;          // the tail bytes
}

// A workgroup per transfer, 16 bytes a thread where both ends allow it. Bound by the round trip to
// host memory (4 us for a pass's two dozen transfers, which were a copy of 5 us each).
__global__ __launch_bounds__(256) void k_move(const Move* moves) {
    const Move m = moves[blockIdx.x];
    static_assert(kMoveBytes == 16 * 256, "one 16-byte read per thread");
    const uint64_t align = (uint64_t)m.dst | (uint64_t)m.src;
    uint64_t done = 0;
    if ((align & 15u) == 0) {
        const uint64_t n = m.bytes / 16;
        if (threadIdx.x < n) ((uint4*)m.dst)[threadIdx.x] = ((const uint4*)m.src)[threadIdx.x];
        done = n * 16;
    } else if ((align & 3u) == 0) {
        const uint64_t n = m.bytes / 4;
        for (uint64_t i = threadIdx.x; i < n; i += 256) ((uint32_t*)m.dst)[i] = ((const uint32_t*)m.src)[i];
        done = n * 4;
    }
    for (uint64_t i = done + threadIdx.x; i < m.bytes; i += 256) ((uint8_t*)m.dst)[i] = ((const uint8_t*)m.src)[i];
}

hipError_t launch_move(const Move* moves, uint32_t n, hipStream_t st) {
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_move, dim3(n), dim3(256), 0, st, moves);
    return hipGetLastError();
}

hipError_t launch_fill(void* p, uint8_t value, uint64_t bytes, hipStream_t st) {
    if (!bytes) return hipSuccess;
    const uint32_t word = 0x01010101u * value;
    // whole 32-bit words from a 4-byte aligned start; the rest bytewise
    uint8_t* b = (uint8_t*)p;
    const uint64_t lead = (4 - ((uintptr_t)b & 3)) & 3;
    if (lead) {
        const uint64_t k = lead < bytes ? lead : bytes;
        hipLaunchKernelGGL(k_fill, dim3(1), dim3(64), 0, st, b, word, (uint64_t)0, k);
        if (k == bytes) return hipGetLastError();
        b += k;
        bytes -= k;
    }
    const uint64_t words = bytes / 4;
    uint64_t blocks = (std::max<uint64_t>(words, 4) + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_fill, dim3((uint32_t)blocks), dim3(256), 0, st, b, word, words, bytes);
    return hipGetLastError();
}

// Calibration read: every 16-byte word of [p, p + words * 16) read once, one sum written, so the
// launch's HBM traffic is known (the bytes read, and 8 written).
__global__ void k_read_calibration(const uint4* p, uint64_t words, unsigned long long* sink) {
    uint64_t acc = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint4 v = p[i];
        acc += (uint64_t)v.x + v.y + v.z + v.w;
    }
    acc = wave_sum_u64(acc);
    if (lane_id() == 0) atomicAdd(sink, (unsigned long long)acc);
}

// Reads 16 bytes at the start of each of `lines` distinct 128-byte lines of the buffer: with n
// lines in the buffer (a power of two) line (i * P) mod n, P odd, is a bijection, so the lines
// read are distinct and spread over the whole buffer.
__global__ void k_read_gather(const uint8_t* p, uint32_t lines, uint32_t mask, unsigned long long* sink) {
    uint64_t acc = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < lines; i += gridDim.x * blockDim.x) {
        const uint32_t l = (uint32_t)(((uint64_t)i * 0x9E3779B1u) & mask);
        const uint4 v = *(const uint4*)(p + (uint64_t)l * 128);
        acc += (uint64_t)v.x + v.y + v.z + v.w;
    }
    acc = wave_sum_u64(acc);
    if (lane_id() == 0) atomicAdd(sink, (unsigned long long)acc);
}

// One device-scope compare-and-swap on the first word of each of `lines` distinct lines (the
// buffer holds no zero word, so every one fails and nothing changes), then one device-scope add
// per thread into 4,096 words of 64-byte stride: the atomics' traffic, for the counters.
__global__ void k_atomic_calibration(uint8_t* p, uint32_t lines, uint32_t mask, unsigned long long* ctr,
                                     unsigned long long* sink) {
    uint64_t acc = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < lines; i += gridDim.x * blockDim.x) {
        const uint32_t l = (uint32_t)(((uint64_t)i * 0x9E3779B1u) & mask);
        acc += atomicCAS((unsigned long long*)(p + (uint64_t)l * 128), 0ull, 1ull);
        atomicAdd(&ctr[(i & 4095u) * 8u], 1ull);
    }
    acc = wave_sum_u64(acc);
    if (lane_id() == 0) atomicAdd(sink, (unsigned long long)acc);
}

hipError_t launch_read_gather(void* p, uint64_t bytes, uint64_t* sink, uint64_t* ctr, hipStream_t st) {
    uint64_t n = 1;                                   // 128-byte lines in the buffer, a power of two
    while (n * 2 * 128 <= bytes) n *= 2;
    if (n < 4) return hipSuccess;
    hipLaunchKernelGGL(k_read_gather, dim3(2048), dim3(256), 0, st, (const uint8_t*)p, (uint32_t)(n / 4),
                       (uint32_t)(n - 1), (unsigned long long*)sink);
    if (hipGetLastError() != hipSuccess) return hipErrorLaunchFailure;
    hipLaunchKernelGGL(k_atomic_calibration, dim3(2048), dim3(256), 0, st, (uint8_t*)p, (uint32_t)(n / 4),
                       (uint32_t)(n - 1), (unsigned long long*)ctr, (unsigned long long*)sink);
    return hipGetLastError();
}

// HGX_OPTION_COUNTER_FLUSH: one streaming read of the flush buffer, whose lines displace every
// line the L2 holds (the sum goes nowhere the host reads; it is kept live by a store into the
// buffer's first word only when it is impossible, i.e. never).
__global__ void k_flush(const uint4* p, uint64_t words) {
    uint64_t acc = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint4 v = p[i];
        acc += (uint64_t)v.x + v.y + v.z + v.w;
    }
    if (acc == 0xFFFFFFFFFFFFFFFFull) ((uint4*)p)[0] = make_uint4(1, 1, 1, 1);
}

hipError_t launch_flush(const void* buf, uint64_t bytes, hipStream_t st) {
    hipLaunchKernelGGL(k_flush, dim3(2048), dim3(256), 0, st, (const uint4*)buf, bytes / 16);
    return hipGetLastError();
}

hipError_t launch_read_calibration(const void* p, uint64_t bytes, uint64_t* sink, hipStream_t st) {
    const uint64_t words = bytes / 16;
    hipLaunchKernelGGL(k_read_calibration, dim3(2048), dim3(256), 0, st, (const uint4*)p, words,
                       (unsigned long long*)sink);
    return hipGetLastError();
}

// A run over its budget stops being counted once the count pass is sure of it, so its total is
// any value above the budget: the decision is what must agree, and below the budget the total.
__global__ void k_plan_check(const uint64_t* tot, const uint64_t* want, const uint32_t* budget, uint32_t n,
                             uint32_t* flag) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t b = budget[i];
    const bool over = tot[i] > b, want_over = want[i] > b;
    if (over != want_over || (!over && tot[i] != want[i])) atomicOr(flag, 1u);
}

hipError_t launch_plan_check(const uint64_t* tot, const uint64_t* want, const uint32_t* budget, uint32_t n,
                             uint32_t* flag, hipStream_t st) {
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_plan_check, dim3((n + 255) / 256), dim3(256), 0, st, tot, want, budget, n, flag);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// Branchial pairs of parents above BR_MAX_EDGES edges. Every (consumed edge slot, match) of such
// a parent becomes one 64-bit key (slot << 32 | match); sorted, the keys of one slot are its consuming
// matches in ascending order. Match i meets each partner j > i through the first of its own
// edges that j also consumes: from its key for that edge, the keys after it with the same slot.
// The work is the entries plus the sum over edges of (matches consuming it)^2 -- not the
// generation's edge count, nor (matches per parent)^2. One thread per match or entry.
// ------------------------------------------------------------------------------------------

__device__ __forceinline__ bool brl_large(const BrListArgs& a, uint32_t m, uint32_t& par) {
    par = a.M.parent[m];
    return a.P.ne[par] > BR_MAX_EDGES && a.cnt[par] >= 2;
}

// Keys and payloads of match m at entries [m*K, m*K + K): (slot << 32 | m, m*K + k) for its
// consumed edges, the sentinel (past every slot) for the rest.
__global__ void k_brl_keys(BrListArgs a) {
    const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= a.M.n) return;
    const uint32_t K = a.M.K;
    uint32_t par, nl = 0;
    if (brl_large(a, m, par)) nl = a.runs[a.P.run[par]].rules[a.M.rule[m]].n_lhs;
    const uint16_t* q = a.M.q + (size_t)m * K;
    for (uint32_t k = 0; k < K; ++k) {
        const uint64_t x = (uint64_t)m * K + k;
        a.key_in[x] = k < nl ? ((a.P.eoff[par] + q[k]) << 32) | m : a.sentinel;
        a.val_in[x] = (uint32_t)x;
    }
}

// Where each (match, k) entry landed in the sorted keys.
__global__ void k_brl_pos(BrListArgs a, uint64_t n) {
    const uint64_t x = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= n || a.key[x] == a.sentinel) return;
    a.pos[a.val[x]] = (uint32_t)x;
}

template <bool EMIT>
__device__ __forceinline__ uint32_t brl_match_pairs(const BrListArgs& a, uint32_t i, uint32_t par, uint32_t run) {
    const DRun& RN = a.runs[run];
    const uint32_t K = a.M.K;
    const uint32_t nl = RN.rules[a.M.rule[i]].n_lhs;
    const uint16_t* qi = a.M.q + (size_t)i * K;
    uint32_t c = 0;
    uint64_t o = 0;
    if (EMIT) {
        const uint32_t mb = (uint32_t)a.moff[par];
        o = a.poff[par] + (a.bo[i] - a.bo[mb]);
    }
    for (uint32_t k = 0; k < nl; ++k) {
        const uint64_t x0 = a.pos[(uint64_t)i * K + k];
        const uint64_t slot = a.key[x0] >> 32;
        for (uint64_t x = x0 + 1; x < a.n_keys && (a.key[x] >> 32) == slot; ++x) {
            const uint32_t j = (uint32_t)a.key[x];
            // count j here only if this is the first of i's edges that j consumes
            const uint16_t* qj = a.M.q + (size_t)j * K;
            const uint32_t nj = RN.rules[a.M.rule[j]].n_lhs;
            bool earlier = false;
            for (uint32_t k2 = 0; k2 < k && !earlier; ++k2)
                for (uint32_t y = 0; y < nj; ++y) earlier |= (qj[y] == qi[k2]);
            if (earlier) continue;
            if (EMIT) {
                a.pairs[2 * o] = RN.ev_base + (i - RN.child_begin);
                a.pairs[2 * o + 1] = RN.ev_base + (j - RN.child_begin);
                ++o;
            }
            ++c;
        }
    }
    return c;
}

// One lane per match; the count pass adds each run's and each parent's pairs once per wave that holds
// some of its matches.
template <bool EMIT>
__global__ void k_brl_pairs(BrListArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t par = INV, run = INV, c = 0;
    if (i < a.M.n && brl_large(a, i, par)) {
        run = a.P.run[par];
        c = brl_match_pairs<EMIT>(a, i, par, run);
        if (!EMIT) a.bc[i] = c;
    } else {
        par = INV;
    }
    if constexpr (!EMIT) {
        for (uint64_t left = __ballot(c != 0); left;) {
            const int u = (int)__builtin_ctzll(left);
            const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)run, u);
            const bool mine = run == r0 && c;
            const uint32_t sum = wave_sum_u32(mine ? c : 0u);
            if (lane_id() == 0)
                atomicAdd((unsigned long long*)&a.ctr[(size_t)r0 * CTR_N + CTR_BRANCHIAL], (unsigned long long)sum);
            left &= ~__ballot(mine);
        }
        if (a.pcnt)
            for (uint64_t left = __ballot(c != 0); left;) {
                const int u = (int)__builtin_ctzll(left);
                const uint32_t p0 = (uint32_t)__builtin_amdgcn_readlane((int)par, u);
                const bool mine = par == p0 && c;
                const uint32_t sum = wave_sum_u32(mine ? c : 0u);
                if (lane_id() == 0) atomicAdd(&a.pcnt[p0], sum);
                left &= ~__ballot(mine);
            }
    }
}

hipError_t launch_brl(const BrListArgs& a, int phase, hipStream_t st) {
    const uint32_t n = a.M.n;
    if (!n) return hipSuccess;
    const dim3 g((n + 255) / 256), b(256);
    switch (phase) {
        case 0: hipLaunchKernelGGL(k_brl_keys, g, b, 0, st, a); break;
        case 1: hipLaunchKernelGGL(k_brl_pos, dim3((uint32_t)((a.n_keys + 255) / 256)), b, 0, st, a, a.n_keys); break;
        case 2: hipLaunchKernelGGL(k_brl_pairs<false>, g, b, 0, st, a); break;
        default: hipLaunchKernelGGL(k_brl_pairs<true>, g, b, 0, st, a); break;
    }
    return hipGetLastError();
}

// The records of a generation's children, one lane per child, after k_expand: the event, its causal
// masks and lineage table, the child's own record, and its identity -- its hash into its request's
// state map (Hypergraph::create_or_get_canonical_state, hypergraph/src/hypergraph.cpp:154-254) --
// with the request's counters. Apart from k_expand because none of it needs a team: there a few lanes
// of each team did it while the hash's registers were live, and its values lived through the hash.
//
// Causal: one triple per consumed edge with a producer; the producers are events of this lineage,
// named by their generation (rewriter.cpp:121-191, causal_graph.cpp:187-234). Transitive reduction: a
// producer is redundant exactly when it is a causal ancestor of another one (an ancestor mask never
// holds the event's own generation, so of any one).
//
// Device-scope atomics are performed beyond the L2 and each moves a whole request over the fabric
// (measured on gfx950: 64 bytes per compare-and-swap, taken or not, 32 per add), and the children of
// one generation that hash alike all find the slot empty before any of them claims it. So a lane
// whose (request, hash) equals a lower lane's in the wave leaves the insert to that lane, and a wave
// keeps the counters of the run its lanes hold (a run's children are contiguous) in registers over
// all of its children, adding them when the run changes, and a workgroup's waves add their last run's
// together: 10.3 M children of one run 2.63 ms with an add per 256 children, 1.06 with one per wave
// of at most 4,096, 0.70 so.
constexpr uint32_t kRecordWaves = 4096;   // at most, so one large run is added to by as many waves
__global__ __launch_bounds__(256) void k_record(ExpandArgs a, uint32_t n, uint32_t chunk) {
    const uint32_t l = lane_id();
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
    const uint32_t first = wave * chunk, end = min(n, first + chunk);
    uint32_t cur = INV;                                   // the run whose counters the lanes hold
    uint32_t events = 0, canon = 0, triples = 0, triples_tr = 0, pairs = 0, pairs_tr = 0;
    uint64_t fp = 0;
    __shared__ uint64_t bsum[4][CTR_BRANCHIAL + 1];       // the waves' last runs: slot CTR_BRANCHIAL holds
    __shared__ uint32_t brun[4];                          //   the fingerprint
    auto add_row = [&](uint32_t r, uint32_t k, uint64_t x) {
        if (x) atomicAdd((unsigned long long*)&a.ctr[(size_t)r * CTR_N + (k == CTR_BRANCHIAL ? CTR_FINGERPRINT : k)],
                         (unsigned long long)x);
    };
    auto flush = [&](bool last) {
        const uint64_t x[CTR_BRANCHIAL + 1] = {wave_sum_u32(events), wave_sum_u32(canon), wave_sum_u32(triples),
                                               wave_sum_u32(pairs), wave_sum_u32(pairs_tr), wave_sum_u32(triples_tr),
                                               wave_sum_u64(fp)};
        if (l == 0) {
            if (last) brun[threadIdx.x / WAVE] = cur;
#pragma unroll
            for (uint32_t k = 0; k <= CTR_BRANCHIAL; ++k) {
                if (last) bsum[threadIdx.x / WAVE][k] = x[k];
                else if (cur != INV) add_row(cur, k, x[k]);
            }
        }
        events = canon = triples = triples_tr = pairs = pairs_tr = 0;
        fp = 0;
    };
    for (uint32_t base = first; base < end; base += WAVE) {
        const uint32_t c = base + l;
        const bool in = c < end;
        uint32_t run = INV, t_n = 0, tt_n = 0, p_n = 0, pt_n = 0;
        uint64_t h = 0;
        if (in) {
            const uint32_t par = a.M.parent[c], rid = a.M.rule[c];
            h = a.C.hash[c];
            run = a.P.run[par];
            const uint32_t pne = a.P.ne[par], nextv = a.P.nextv[par], in_state = a.P.sid[par];
            const uint64_t peo = a.P.eoff[par];
            const uint32_t step = a.P.depth[par] + 1u;    // generation of the child
            const DRun& RN = a.runs[run];
            const DRule& R = RN.rules[rid];
            const uint32_t nl = R.n_lhs, cne = pne - nl + R.n_rhs;
            const uint16_t* q = a.M.q + (size_t)c * a.M.K;
            const uint64_t* plan = a.P.lanc + (size_t)par * a.P.lstride;
            uint64_t prod = 0, anc = 0;                   // producers' generations; their ancestors
            for (uint32_t t = 0; t < nl; ++t) {
                const uint32_t ps = a.P.ps[peo + q[t]];
                if (a.E.cps) a.E.cps[(size_t)c * a.E.cK + t] = (uint8_t)ps;
                if (ps) {
                    prod |= 1ull << ps;
                    anc |= plan[ps - 1];
                    ++t_n;
                }
            }
            uint64_t tr = (RN.flags & 0x100u) ? prod & ~anc : prod;
            anc |= prod;
            if (RN.flags & 0x1u) {
                for (uint32_t t = 0; t < nl; ++t) tt_n += (uint32_t)((tr >> a.P.ps[peo + q[t]]) & 1ull);
            } else {
                prod = 0; tr = 0; anc = 0; t_n = 0;
            }
            p_n = (uint32_t)__popcll(prod);
            pt_n = (uint32_t)__popcll(tr);
            const uint32_t ev_id = RN.ev_base + (c - RN.child_begin);
            a.C.run[c] = run;
            a.C.ne[c] = cne;
            a.C.nextv[c] = nextv + R.n_new;
            a.C.sid[c] = RN.n_roots + ev_id;
            a.C.depth[c] = (uint8_t)step;
            a.E.in_state[c] = in_state;
            a.E.rule[c] = rid;
            a.E.prod[c] = prod;
            a.E.tr[c] = tr;
            // lineage table: the parent's, then this event's ancestor mask
            uint64_t* clan = a.C.lanc + (size_t)c * a.C.lstride;
            for (uint32_t t = 0; t + 1 < step; ++t) clan[t] = plan[t];
            clan[step - 1] = anc;
        }
        bool dup = false;
        for (int k = 0; k < WAVE - 1; ++k) {
            const uint32_t hl = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)h, k);
            const uint32_t hh = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(h >> 32), k);
            const uint32_t rk = (uint32_t)__builtin_amdgcn_readlane((int)run, k);
            dup |= k < (int)l && hl == (uint32_t)h && hh == (uint32_t)(h >> 32) && rk == run;
        }
        const bool fresh = in && !dup && map_insert(&a.runs[run], h);
        const uint64_t f = fresh ? mix64(h) : 0ull;
        for (uint64_t left = __ballot(in); left;) {       // the runs among the lanes, usually one
            const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)run, (int)__builtin_ctzll(left));
            const bool mine = run == r0;
            if (r0 != cur) { flush(false); cur = r0; }
            if (mine) {
                events += 1;
                canon += fresh ? 1u : 0u;
                fp += f;
                triples += t_n; triples_tr += tt_n; pairs += p_n; pairs_tr += pt_n;
            }
            left &= ~__ballot(mine);
        }
    }
    // the workgroup's waves mostly end in one run: one add for them all
    flush(true);
    __syncthreads();
    if (threadIdx.x <= CTR_BRANCHIAL) {
        const uint32_t k = threadIdx.x;
        uint64_t sum = 0;
        for (uint32_t w = 0; w < 4; ++w) {
            if (brun[w] != INV) sum += bsum[w][k];
            if (brun[w] != INV && (w == 3 || brun[w + 1] != brun[w])) { add_row(brun[w], k, sum); sum = 0; }
        }
    }
}

hipError_t launch_record(const ExpandArgs& a, uint32_t n, hipStream_t st) {
    if (!n) return hipSuccess;
    const uint32_t chunk = WAVE * ((n + WAVE * kRecordWaves - 1) / (WAVE * kRecordWaves));
    const uint32_t waves = (n + chunk - 1) / chunk;
    hipLaunchKernelGGL(k_record, dim3((waves + 3) / 4), dim3(256), 0, st, a, n, chunk);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// Branchial pairs: two events of the SAME input state whose consumed edge sets intersect,
// one pair each (causal_graph.cpp:324-351). One wave per parent.
//
// Parents of at most 128 edges: the parent's matches are taken in chunks; for each chunk an
// LDS bitset per edge position marks the chunk's matches that consume it. Match i then meets
// every later match j of the chunk through the OR of the bitsets of its own edges: one popcount
// per 64 candidates instead of one test per pair. A consumed set is NW 64-bit words (one up to
// 64 edges, two up to 128); the bitsets and the cached consumed sets take the same 16 KiB of
// LDS either way, so a two-word parent works in half-size chunks. Larger parents take the
// per-edge match lists above (k_brl_*).
// ------------------------------------------------------------------------------------------

constexpr uint32_t BR_LDS_WORDS = 1024;             // per table: 8 KiB of bitsets, 8 KiB of masks

static uint32_t branchial_lds_per_wave() { return 2 * BR_LDS_WORDS * 8 + 64; }

template <uint32_t NW>
__device__ __forceinline__ void consumed_mask(const BranchialArgs& a, const DRun& RN, uint32_t m,
                                              uint64_t (&msk)[NW]) {
    const uint32_t nl = RN.rules[a.M.rule[m]].n_lhs;
    const uint16_t* q = a.M.q + (size_t)m * a.M.K;
#pragma unroll
    for (uint32_t w = 0; w < NW; ++w) msk[w] = 0;
    for (uint32_t t = 0; t < nl; ++t) {
        const uint32_t e = q[t];
#pragma unroll
        for (uint32_t w = 0; w < NW; ++w)
            if ((e >> 6) == w) msk[w] |= 1ull << (e & 63);
    }
}

// One parent (cnt >= 2 matches from m0): its pairs counted (emit 0) or written (emit 1).
template <uint32_t NW>
__device__ __forceinline__ uint32_t branchial_parent(const BranchialArgs& a, const DRun& RN, uint32_t m0,
                                                     uint32_t cnt, uint32_t ne, uint32_t ev0, uint64_t out,
                                                     uint8_t* my, uint32_t l) {
    constexpr uint32_t WORDS = 16 / NW;              // 64-bit words per edge bitset
    constexpr uint32_t CHUNK = WORDS * 64;           // matches per chunk
    constexpr uint32_t MASKS = BR_LDS_WORDS / NW;    // consumed sets cached in LDS
    uint64_t* bits = (uint64_t*)my;                  // [64 * NW edges][WORDS]
    uint64_t* mcache = bits + BR_LDS_WORDS;          // [MASKS][NW]
    uint32_t total = 0;
    const uint32_t ncache = cnt < MASKS ? cnt : MASKS;
    for (uint32_t i = l; i < ncache; i += WAVE) {
        uint64_t mk[NW];
        consumed_mask<NW>(a, RN, m0 + i, mk);
#pragma unroll
        for (uint32_t w = 0; w < NW; ++w) mcache[i * NW + w] = mk[w];
    }
    wave_sync();
    auto mask_of = [&](uint32_t i, uint64_t (&mk)[NW]) {
        if (i < MASKS) {
#pragma unroll
            for (uint32_t w = 0; w < NW; ++w) mk[w] = mcache[i * NW + w];
        } else {
            consumed_mask<NW>(a, RN, m0 + i, mk);
        }
    };
    for (uint32_t cb = 0; cb < cnt; cb += CHUNK) {
        const uint32_t ce = min(cnt, cb + CHUNK);
        const uint32_t words = (ce - cb + 63) >> 6;
        // only the words this chunk reads: the parent's edges x the chunk's 64-match words
        for (uint32_t x = l; x < ne * words; x += WAVE) {
            const uint32_t e = x / words;
            bits[e * WORDS + (x - e * words)] = 0;
        }
        wave_sync();
        for (uint32_t j = cb + l; j < ce; j += WAVE) {
            const uint32_t r = j - cb;
            uint64_t mj[NW];
            mask_of(j, mj);
#pragma unroll
            for (uint32_t w = 0; w < NW; ++w)
                for (uint64_t mk = mj[w]; mk; mk &= mk - 1)
                    atomicOr((unsigned long long*)&bits[(w * 64 + __builtin_ctzll(mk)) * WORDS + (r >> 6)],
                             1ull << (r & 63));
        }
        wave_sync();
        for (uint32_t base = 0; base < ce; base += WAVE) {
            const uint32_t i = base + l;
            uint32_t c = 0;
            uint64_t mi[NW];
#pragma unroll
            for (uint32_t w = 0; w < NW; ++w) mi[w] = 0;
            auto partners = [&](uint32_t wd) {         // later matches of word wd sharing an edge with i
                const uint32_t jb = cb + wd * 64;
                uint64_t word = 0;
#pragma unroll
                for (uint32_t w = 0; w < NW; ++w)
                    for (uint64_t mk = mi[w]; mk; mk &= mk - 1)
                        word |= bits[(w * 64 + __builtin_ctzll(mk)) * WORDS + wd];
                if (jb <= i) word &= ~((2ull << (i - jb)) - 1ull);
                return word;
            };
            if (i < ce) {
                mask_of(i, mi);
                for (uint32_t wd = 0; wd < words; ++wd) {
                    if (cb + wd * 64 + 63 <= i) continue;
                    c += __popcll(partners(wd));
                }
            }
            if (a.emit) {
                const uint32_t inc = wave_incl_scan_u32(c);
                uint64_t o = out + inc - c;
                if (c) {
                    for (uint32_t wd = 0; wd < words; ++wd) {
                        const uint32_t jb = cb + wd * 64;
                        if (jb + 63 <= i) continue;
                        for (uint64_t word = partners(wd); word; word &= word - 1) {
                            a.pairs[2 * o] = ev0 + i;
                            a.pairs[2 * o + 1] = ev0 + jb + __builtin_ctzll(word);
                            ++o;
                        }
                    }
                }
                out += __shfl(inc, WAVE - 1, WAVE);
            } else {
                total += c;
            }
        }
        wave_sync();
    }
    return total;
}

// The pair counts of parents whose matches consume at most three edges, without the pairs. Two
// matches of a parent that share k edges share k single edges, k (k - 1) / 2 edge pairs and, for
// k = 3, one triple: single - pairs + triples is 1 for k = 1, 2 and 3. So each match adds itself to
// a counter of each of its edges, of its edge pairs (a triangular table) and of its triple (a hash
// table), and the counters' old values, with those signs, are the pairs it makes with earlier
// matches: one pass over the matches, where the bit sets of k_branchial take one to build them and
// one to read them for every 64 matches.
// G lanes per parent: 16 for those of few edges in a generation of enough parents to fill the chip so
// (bound by the latency of a parent's reads, so the parents in flight count), a wave for those of many
// matches, whose time with bit sets grows as the square. Parents in between stay with k_branchial: the
// tables of 65 to 128 edges take all the LDS of its bit sets (those of the batched workload's fifth
// generation 0.23 ms by bit sets, 0.43 by a wave of counts each).
// 300 k parents of one evolution 0.50 -> 0.06 ms; a generation with parents of up to 4,096 matches
// 0.50 -> 0.07; the batched workload's counts 1.25 -> 0.84.
__host__ __device__ inline uint32_t branchial_count_words(uint32_t ne) {
    return ((ne + (ne * (ne - (ne ? 1u : 0u)) / 2 + 1) / 2) + 3u) & ~3u;
}
// Slots of the triples' table for cnt matches: a load of at most a half.
__device__ __forceinline__ uint32_t branchial_slots(uint32_t cnt) {
    uint32_t n = 32;
    while (n < 2 * cnt) n <<= 1;
    return n;
}
// Who counts a parent's pairs: 16 lanes (1), a wave (2) of k_branchial_count, or k_branchial (0).
__device__ __forceinline__ uint32_t branchial_tier(const BranchialArgs& a, uint32_t count_lhs, uint32_t ne, uint32_t cnt) {
    const uint32_t k = count_lhs & 3u;
    if (k == 0) return 0;
    if (ne <= a.few_ne && (k < 3 || cnt <= kBranchialFewTriples)) return 1;
    return cnt > kBranchialMany && (k < 3 || cnt <= kBranchialTriples) ? 2 : 0;
}
template <uint32_t G>
__device__ __forceinline__ uint32_t branchial_count(const BranchialArgs& a, const DRun& RN, uint32_t lhs, uint32_t* tab,
                                                    uint32_t m0, uint32_t cnt, uint32_t ne, uint32_t r) {
    const uint32_t words = branchial_count_words(ne), slots = (lhs & 3u) == 3 ? branchial_slots(cnt) : 0u;
    uint32_t* triples = tab + words;
    for (uint32_t i = r; i < (words + slots) / 4; i += G) ((uint4*)tab)[i] = make_uint4(0, 0, 0, 0);
    wave_sync();
    uint32_t pairs = 0;
    auto edge_pair = [&](uint32_t x, uint32_t y) {
        const uint32_t hi = x > y ? x : y, lo = x > y ? y : x, at = hi * (hi - 1) / 2 + lo, sh = 16 * (at & 1u);
        pairs -= (atomicAdd(&tab[ne + at / 2], 1u << sh) >> sh) & 0xFFFFu;
    };
    for (uint32_t i = r; i < cnt; i += G) {
        const uint32_t m = m0 + i;
        const uint16_t* q = a.M.q + (size_t)m * a.M.K;
        const uint32_t nl = lhs & 4u ? lhs & 3u : RN.rules[a.M.rule[m]].n_lhs;
        const uint32_t x = q[0];
        pairs += atomicAdd(&tab[x], 1u);
        if (nl < 2) continue;
        const uint32_t y = q[1];
        pairs += atomicAdd(&tab[y], 1u);
        edge_pair(x, y);
        if (nl < 3) continue;
        const uint32_t z = q[2];
        pairs += atomicAdd(&tab[z], 1u);
        edge_pair(x, z);
        edge_pair(y, z);
        const uint32_t lo = min(x, min(y, z)), hi = max(x, max(y, z));
        const uint32_t key = (lo << 14 | (x + y + z - lo - hi) << 7 | hi) + 1;     // at most 22 bits
        uint32_t h = (key * 0x9E3779B1u) >> 16 & (slots - 1);
        for (;;) {                                     // (the table is at most half full)
            const uint32_t was = atomicCAS(&triples[h], 0u, key << 10 | 1u);
            if (was == 0) break;
            if (was >> 10 == key) { pairs += atomicAdd(&triples[h], 1u) & 1023u; break; }
            h = (h + 1) & (slots - 1);
        }
    }
    wave_sync();
    return group_sum<G>(pairs);
}
template <uint32_t G>
__global__ __launch_bounds__(G == WAVE ? 64 : 256) void k_branchial_count(BranchialArgs a) {
    extern __shared__ uint8_t lds[];
    constexpr uint32_t GPW = WAVE / G, WPB = G == WAVE ? 1 : 4, SUMS = WPB * GPW;
    __shared__ uint32_t srun[SUMS];
    __shared__ uint64_t ssum[SUMS];
    const uint32_t w = threadIdx.x / WAVE, l = lane_id(), g = l / G, r = l % G;
    uint32_t* tab = (uint32_t*)(lds + (size_t)w * a.lds_per_wave) + g * a.group_words;
    uint32_t cur = INV;                                // the run whose pairs `sum` holds
    uint64_t sum = 0;
    auto add = [&](uint32_t run, uint32_t total) {
        if (run != cur) {
            if (cur != INV && sum && r == 0)
                atomicAdd((unsigned long long*)&a.ctr[(size_t)cur * CTR_N + CTR_BRANCHIAL], (unsigned long long)sum);
            cur = run;
            sum = 0;
        }
        sum += total;
    };
    // 16 lanes look at their parent; a wave, whose parents are rare, at 64 at a time (neighbours, which
    // are often alike, to different waves), and takes those that are its own one by one
    const uint64_t waves = (uint64_t)gridDim.x * WPB;
    for (uint64_t base = (uint64_t)blockIdx.x * WPB + w; base * (WAVE / G) < a.P.n; base += G == WAVE ? waves * WAVE : waves) {
        const uint64_t s = G == WAVE ? base + l * waves : base * GPW + g;
        uint32_t cnt = 0, ne = 0, run = INV, m0 = 0, lhs = 0;
        if (s < a.P.n) cnt = a.cnt[s];
        if (cnt >= 2) {
            ne = a.P.ne[s];
            run = a.P.run[s];
            m0 = (uint32_t)a.moff[s];
            lhs = a.runs[run].count_lhs;
        }
        const bool live = cnt >= 2 && ne <= BR_MAX_EDGES && branchial_tier(a, lhs, ne, cnt) == (G == WAVE ? 2u : 1u);
        if constexpr (G < WAVE) {
            if (live) {
                const uint32_t total = branchial_count<G>(a, a.runs[run], lhs, tab, m0, cnt, ne, r);
                if (r == 0 && a.pcnt) a.pcnt[s] = total;
                add(run, total);
            }
        } else {
            for (uint64_t todo = __ballot(live); todo; todo &= todo - 1) {
                const int at = __builtin_ctzll(todo);
                auto of = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, at); };
                const uint32_t one = of(run);
                const uint32_t total = branchial_count<G>(a, a.runs[one], of(lhs), tab, of(m0), of(cnt), of(ne), r);
                if (r == 0 && a.pcnt) a.pcnt[base + (uint64_t)at * waves] = total;
                add(one, total);
            }
        }
    }
    // one add per workgroup and run (groups hold neighbouring parents, mostly one run's)
    if (r == 0) { srun[w * GPW + g] = cur; ssum[w * GPW + g] = sum; }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t held = INV;
        uint64_t t = 0;
        for (uint32_t k = 0; k <= SUMS; ++k) {
            if (k < SUMS && (srun[k] == INV || srun[k] == held)) {
                if (srun[k] == held) t += ssum[k];
                continue;
            }
            if (held != INV && t)
                atomicAdd((unsigned long long*)&a.ctr[(size_t)held * CTR_N + CTR_BRANCHIAL], (unsigned long long)t);
            if (k < SUMS) { held = srun[k]; t = ssum[k]; }
        }
    }
}

// The pairs of a run are added to its counter once per wave and run (a wave's states are mostly one
// run's): an add per parent, 300 k of them to one evolution's counter, took 3.5 ms where the
// counting itself takes 0.2.
__global__ __launch_bounds__(256) void k_branchial(BranchialArgs a) {
    extern __shared__ uint8_t lds[];
    const uint32_t w = threadIdx.x / WAVE, l = lane_id();
    uint8_t* my = lds + (size_t)w * a.lds_per_wave;
    const uint32_t waves = gridDim.x * (blockDim.x / WAVE);
    uint32_t cur = INV;                                // the run whose pairs `sum` holds
    uint64_t sum = 0;
    auto flush = [&] {
        if (cur != INV && sum && l == 0)
            atomicAdd((unsigned long long*)&a.ctr[(size_t)cur * CTR_N + CTR_BRANCHIAL], (unsigned long long)sum);
        sum = 0;
    };
    for (uint32_t s = blockIdx.x * (blockDim.x / WAVE) + w; s < a.P.n; s += waves) {
        const uint32_t cnt = a.cnt[s];
        const uint32_t ne = a.P.ne[s];
        if (cnt < 2 || ne > BR_MAX_EDGES) { if (a.emit == 0 && a.pcnt && l == 0) a.pcnt[s] = 0; continue; }
        const uint32_t run = a.P.run[s];
        const uint32_t m0 = (uint32_t)a.moff[s];
        const DRun& RN = a.runs[run];
        if (!a.emit && branchial_tier(a, RN.count_lhs, ne, cnt)) continue;
        const uint32_t ev0 = RN.ev_base + (m0 - RN.child_begin);
        const uint64_t out = a.emit ? a.poff[s] : 0;
        const uint32_t total = ne <= 64 ? branchial_parent<1>(a, RN, m0, cnt, ne, ev0, out, my, l)
                                        : branchial_parent<2>(a, RN, m0, cnt, ne, ev0, out, my, l);
        if (!a.emit) {
            const uint32_t tot = wave_sum_u32(total);
            const uint32_t r = (uint32_t)__builtin_amdgcn_readfirstlane((int)run);
            if (r != cur) { flush(); cur = r; }
            sum += tot;
            if (l == 0 && a.pcnt) a.pcnt[s] = tot;
        }
        wave_sync();
    }
    if (!a.emit) flush();
}

// ------------------------------------------------------------------------------------------
// WL hash of explicitly given states (dense local vertex ids per state). Optionally inserts
// each into its run's state map (roots).
// ------------------------------------------------------------------------------------------

template <bool GWS, uint32_t W>
__global__ __launch_bounds__(W == 1 ? 256 : 64 * W) void k_wl_states(WLStatesArgs a) {
    extern __shared__ uint8_t lds[];
    const uint32_t tpb = W == 1 ? blockDim.x / WAVE : 1;    // teams per workgroup
    const uint32_t w = W == 1 ? threadIdx.x / WAVE : 0;     // team within the workgroup
    uint8_t* p;
    if constexpr (GWS) p = a.scratch + ((size_t)blockIdx.x * tpb + w) * a.lds_per_wave;
    else p = lds + (size_t)w * a.lds_per_wave;
    const Team<W> tm((uint64_t*)(p + a.lds_per_wave - 64));   // the workspace's last 64 bytes
    const uint32_t A = a.A;
    const WLSizes z = WLSizes::make(a.max_ne, a.max_nv, A, a.lean != 0);
    WLSpace s;
    wl_bind(s, p, z, A);
    const uint32_t teams = gridDim.x * tpb;
    for (uint32_t i = blockIdx.x * tpb + w; i < a.n; i += teams) {
        const uint64_t e0 = a.state_off[i];
        const uint32_t ne = (uint32_t)(a.state_off[i + 1] - e0);
        for (uint32_t e = tm.r; e < ne; e += Team<W>::N) {
            const uint8_t ar = a.ar[e0 + e];
            s.e_ar[e] = ar;
            for (uint32_t k = 0; k < A; ++k) s.e_lv[e * A + k] = (uint16_t)(k < ar ? a.ev[(e0 + e) * A + k] : 0u);
        }
        s.nE = ne;
        s.nV = a.nv[i];
        tm.sync();
        const uint64_t h = wl_hash_team(s, tm);
        if (tm.leader()) wl_state_done(a, i, h);
        tm.sync();
    }
}

// Admissions of one step: one block per request.
__global__ void k_admit(const AdmitItem* items, uint64_t* ctr) {
    const AdmitItem it = items[blockIdx.x];
    const uint32_t* src = (const uint32_t*)it.rule_src;
    uint32_t* dst = (uint32_t*)it.rule_dst;
    const uint32_t words = it.n_rules * (uint32_t)(sizeof(DRule) / 4);
    for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) dst[i] = src[i];
    for (uint64_t i = threadIdx.x; i < it.map_cap; i += blockDim.x) it.map_keys[i] = 0;
    if (threadIdx.x < CTR_N) ctr[(size_t)it.slot * CTR_N + threadIdx.x] = 0;
}

hipError_t launch_admit(const AdmitItem* items, uint32_t n, uint64_t* ctr, hipStream_t st) {
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_admit, dim3(n), dim3(256), 0, st, items, ctr);
    return hipGetLastError();
}

// One block per prepared request: its roots' records and edges into the generation.
__global__ void k_copy_roots(const RootCopy* items, GenView v) {
    const RootCopy it = items[blockIdx.x];
    const uint64_t e0 = it.eoff[0], e1 = it.eoff[it.n_roots];
    for (uint32_t k = threadIdx.x; k <= it.n_roots; k += blockDim.x) {
        v.eoff[it.dst_state + k] = it.dst_edge + (it.eoff[k] - e0);
        if (k < it.n_roots) {
            v.run[it.dst_state + k] = it.slot;
            v.ne[it.dst_state + k] = it.ne[k];
            v.nextv[it.dst_state + k] = it.nextv[k];
            v.sid[it.dst_state + k] = k;
            v.depth[it.dst_state + k] = 0;
        }
    }
    for (uint64_t e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
        const uint64_t d = it.dst_edge + (e - e0);
        v.ar[d] = it.ar[e];
        v.ps[d] = 0;
        for (uint32_t x = 0; x < v.A; ++x) v.ev[d * v.A + x] = x < it.src_A ? it.ev[e * it.src_A + x] : 0u;
    }
}

hipError_t launch_copy_roots(const RootCopy* items, uint32_t n, const GenView& v, hipStream_t st) {
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_copy_roots, dim3(n), dim3(256), 0, st, items, v);
    return hipGetLastError();
}

// Per-run match totals of a generation: runs' states are contiguous ranges. For each run, its
// children's edges and the edges of its states that have matches (the parents its expansion reads)
// are summed into its slot (zero before the launch), its matches come from the offsets. A wave takes
// kTotalsChunk consecutive states, 64 at a time: lanes of one run keep running sums that are
// added once per chunk, and a group holding several runs is summed by segments with one scan, so
// neither one run of 300 k states (one wave per run: 2.05 ms a pass, so 0.04) nor a generation of
// one state per run (run after run in a chunk: 0.59 ms a batched pass, so 0.10) is left to one
// wave's latency.
constexpr uint32_t kTotalsChunk = 512;
__device__ __forceinline__ void add_run_totals(uint64_t* edges, uint64_t* parent_edges, uint32_t r, uint64_t sum,
                                               uint64_t pe) {
    if (sum) atomicAdd((unsigned long long*)&edges[r], (unsigned long long)sum);
    if (pe) atomicAdd((unsigned long long*)&parent_edges[r], (unsigned long long)pe);
}
__global__ void k_run_totals(const uint64_t* moff, const uint64_t* state_edges, const uint32_t* cnt,
                             const uint32_t* ne, const uint32_t* run, uint32_t n, const uint32_t* run_sbeg,
                             const uint32_t* run_send, uint64_t* tot, uint64_t* edges, uint64_t* parent_edges) {
    const uint32_t c = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE, l = lane_id();
    const uint32_t first = c * kTotalsChunk, end = min(n, first + kTotalsChunk);
    uint64_t sum = 0, pe = 0;                           // this lane's states of run `cur`
    uint32_t cur = INV;
    auto flush = [&] {
        if (cur == INV) return;
        const uint64_t a = wave_sum_u64(sum), b = wave_sum_u64(pe);
        if (l == 0) add_run_totals(edges, parent_edges, cur, a, b);
        sum = pe = 0;
        cur = INV;
    };
    for (uint32_t base = first; base < end; base += WAVE) {
        const uint32_t s = base + l;
        const bool in = s < end;
        const uint32_t r = in ? run[s] : INV;
        const uint64_t se = in ? state_edges[s] : 0;
        const uint64_t ps = in && cnt[s] ? ne[s] : 0;
        if (in && run_sbeg[r] == s) tot[r] = moff[run_send[r]] - moff[s];
        const uint32_t r0 = __shfl(r, 0, WAVE);
        if (__ballot(in && r != r0) == 0) {
            if (r0 != cur) { flush(); cur = r0; }
            sum += se;
            pe += ps;
            continue;
        }
        flush();
        const uint64_t a = wave_incl_scan_u64(se), b = wave_incl_scan_u64(ps);
        const uint32_t prev = __shfl_up(r, 1, WAVE);
        const uint64_t heads = __ballot(l == 0 || r != prev);
        const uint32_t h = 63u - (uint32_t)__clzll((long long)(heads & ((2ull << l) - 1ull)));   // segment's first lane
        const uint64_t a0 = wave_lane_u64(a, h ? h - 1 : 0), b0 = wave_lane_u64(b, h ? h - 1 : 0);
        const bool last = l == WAVE - 1 || ((heads >> (l + 1)) & 1ull);
        if (last && r != INV) add_run_totals(edges, parent_edges, r, a - (h ? a0 : 0), b - (h ? b0 : 0));
    }
    flush();
}

// Zero the counts of states whose run does not advance this generation.
__global__ void k_mask_counts(const uint32_t* run, const uint8_t* active, uint32_t n, uint32_t* cnt) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n && !active[run[s]]) cnt[s] = 0;
}

// Move one run's state map into a larger table.
__global__ void k_rehash(const uint64_t* old_keys, uint32_t old_cap, uint64_t* keys, uint32_t mask) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= old_cap) return;
    const uint64_t h = old_keys[i];
    if (h == 0) return;
    uint32_t j = (uint32_t)mix64(h) & mask;
    while (true) {
        const uint64_t old = atomicCAS((unsigned long long*)&keys[j], 0ull, (unsigned long long)h);
        if (old == 0) return;
        j = (j + 1) & mask;
    }
}

// ------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------

static uint32_t grid_for(uint32_t items, uint32_t per_block, uint32_t cap);
uint32_t launch_grid(uint32_t items, uint32_t wpb, uint32_t grid_cap) { return grid_for(items, wpb, grid_cap); }

static uint32_t grid_for(uint32_t items, uint32_t per_block, uint32_t cap) {
    uint32_t g = (items + per_block - 1) / per_block;
    if (g > cap) g = cap;
    if (g < 8) g = 8;
    return (g + 7u) & ~7u;
}

template <uint32_t G>
static void launch_match_lanes(const MatchArgs& a, bool emit, uint32_t grid, uint32_t wpb, hipStream_t st) {
    const uint32_t threads = 64 * wpb;
    const size_t lds = (size_t)a.lds_per_wave * wpb * (64 / G);
    if (a.small) {
        if (emit) hipLaunchKernelGGL((k_match<true, JoinLaneLds, 1, false, G>), dim3(grid), dim3(threads), lds, st, a);
        else hipLaunchKernelGGL((k_match<false, JoinLaneLds, 1, false, G>), dim3(grid), dim3(threads), lds, st, a);
    } else {
        if (emit) hipLaunchKernelGGL((k_match<true, JoinLaneBig, 1, false, G>), dim3(grid), dim3(threads), lds, st, a);
        else hipLaunchKernelGGL((k_match<false, JoinLaneBig, 1, false, G>), dim3(grid), dim3(threads), lds, st, a);
    }
}

template <uint32_t W>
static void launch_match_team(const MatchArgs& a, bool emit, uint32_t grid, uint32_t wpb, hipStream_t st) {
    const uint32_t threads = W == 1 ? 64 * wpb : 64 * W;
    if constexpr (W == 8) {
        if (a.scratch) {
            if (a.small) {
                if (emit) hipLaunchKernelGGL((k_match<true, JoinLaneLds, 8, true>), dim3(grid), dim3(threads), 0, st, a);
                else hipLaunchKernelGGL((k_match<false, JoinLaneLds, 8, true>), dim3(grid), dim3(threads), 0, st, a);
            } else {
                if (emit) hipLaunchKernelGGL((k_match<true, JoinLaneBig, 8, true>), dim3(grid), dim3(threads), 0, st, a);
                else hipLaunchKernelGGL((k_match<false, JoinLaneBig, 8, true>), dim3(grid), dim3(threads), 0, st, a);
            }
            return;
        }
    }
    const size_t lds = (size_t)a.lds_per_wave * (W == 1 ? wpb : 1);
    if (a.small) {
        if (emit) hipLaunchKernelGGL((k_match<true, JoinLaneLds, W>), dim3(grid), dim3(threads), lds, st, a);
        else hipLaunchKernelGGL((k_match<false, JoinLaneLds, W>), dim3(grid), dim3(threads), lds, st, a);
    } else {
        if (emit) hipLaunchKernelGGL((k_match<true, JoinLaneBig, W>), dim3(grid), dim3(threads), lds, st, a);
        else hipLaunchKernelGGL((k_match<false, JoinLaneBig, W>), dim3(grid), dim3(threads), lds, st, a);
    }
}

hipError_t launch_match(const MatchArgs& a, bool emit, uint32_t grid_cap, uint32_t wpb, uint32_t team,
                        hipStream_t st, uint32_t lanes) {
    const uint32_t items = a.nrange ? a.n_items : a.P.n;
    if (!items) return hipSuccess;
    if (a.scratch && team != 8) return hipErrorInvalidValue;     // global workspaces: 8-wave teams
    if (lanes != 64) {                                           // sub-wave teams: one wave per team set
        if (team != 1 || a.scratch || (lanes != 16 && lanes != 32)) return hipErrorInvalidValue;
        const uint32_t grid = grid_for(items, wpb * (64 / lanes), grid_cap);
        if (lanes == 16) launch_match_lanes<16>(a, emit, grid, wpb, st);
        else launch_match_lanes<32>(a, emit, grid, wpb, st);
        return hipGetLastError();
    }
    const uint32_t grid = grid_for(items, team == 1 ? wpb : 1, grid_cap);
    switch (team) {
        case 1: launch_match_team<1>(a, emit, grid, wpb, st); break;
        case 4: launch_match_team<4>(a, emit, grid, wpb, st); break;
        case 8: launch_match_team<8>(a, emit, grid, wpb, st); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

uint32_t expand_lds_per_wave(uint32_t max_child_ne, uint32_t max_nv, uint32_t max_nextv, uint32_t A, bool lean) {
    const WLSizes z = expand_sizes(max_child_ne, max_nv, max_nextv, A, lean);
    // + 64: carving slack; + 64: the team's reduction words at the end
    return ((z.bytes(A) + 128u) + 15u) & ~15u;
}

template <uint32_t W, uint32_t G>
static void launch_expand_team(const ExpandArgs& a, uint32_t grid, uint32_t wpb, hipStream_t st) {
    const uint32_t threads = W == 1 ? 64 * wpb : 64 * W;
    const size_t lds = a.scratch ? 0 : (size_t)a.lds_per_wave * (W == 1 ? wpb * (64 / G) : 1);
    if constexpr (G == 64) {
        if (a.scratch) { hipLaunchKernelGGL((k_expand<true, W, 64>), dim3(grid), dim3(threads), lds, st, a); return; }
    }
    hipLaunchKernelGGL((k_expand<false, W, G>), dim3(grid), dim3(threads), lds, st, a);
}

uint32_t expand_grid(uint32_t n_items, uint32_t team, uint32_t wpb, uint32_t grid_cap, uint32_t lanes) {
    return grid_for(n_items, team == 1 ? wpb * (64 / lanes) : 1, grid_cap);
}

uint32_t expand_small_lds(uint32_t max_child_ne, uint32_t max_nextv, uint32_t A) {
    return (SmallSizes::make(max_child_ne, max_nextv, A).bytes(A) + 15u) & ~15u;
}

template <uint32_t UA>
static hipError_t launch_expand_small_ua(const ExpandArgs& a, uint32_t grid, uint32_t wpb, uint32_t lanes,
                                         hipStream_t st) {
    const dim3 g(grid), b(64 * wpb);
    const size_t lds = (size_t)a.lds_per_wave * wpb * (64 / lanes);
    switch (lanes) {
        case 64: hipLaunchKernelGGL((k_expand_small<UA, 64>), g, b, lds, st, a); break;
        case 32: hipLaunchKernelGGL((k_expand_small<UA, 32>), g, b, lds, st, a); break;
        case 16: hipLaunchKernelGGL((k_expand_small<UA, 16>), g, b, lds, st, a); break;
        case 8: hipLaunchKernelGGL((k_expand_small<UA, 8>), g, b, lds, st, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_expand_small(const ExpandArgs& a, uint32_t grid_cap, uint32_t wpb, uint32_t lanes, hipStream_t st) {
    if (!a.n_items) return hipSuccess;
    if (!a.lean || a.scratch || a.max_child_ne > kSmallMaxEdges || a.max_nextv > kSmallMaxLabels || a.C.A > 4 ||
        a.M.K > lanes)
        return hipErrorInvalidValue;
    ExpandArgs x = a;
    const uint32_t grid = expand_grid(a.n_items, 1, wpb, grid_cap, lanes);
    x.chunk = (uint64_t)grid * wpb * (64 / lanes) >= a.n_items ? 1u : 2u;
    return x.P.A == 2 && a.C.A == 2 ? launch_expand_small_ua<2>(x, grid, wpb, lanes, st)
                                    : launch_expand_small_ua<0>(x, grid, wpb, lanes, st);
}

hipError_t launch_expand(const ExpandArgs& a, uint32_t grid_cap, uint32_t wpb, uint32_t team, hipStream_t st,
                         uint32_t lanes) {
    if (!a.n_items) return hipSuccess;
    if (lanes != 64 && (team != 1 || a.scratch || (lanes != 16 && lanes != 32))) return hipErrorInvalidValue;
    const uint32_t grid = expand_grid(a.n_items, team, wpb, grid_cap, lanes);
    switch (team * 100 + lanes) {
        case 164: launch_expand_team<1, 64>(a, grid, wpb, st); break;
        case 132: launch_expand_team<1, 32>(a, grid, wpb, st); break;
        case 116: launch_expand_team<1, 16>(a, grid, wpb, st); break;
        case 264: launch_expand_team<2, 64>(a, grid, wpb, st); break;
        case 464: launch_expand_team<4, 64>(a, grid, wpb, st); break;
        case 864: launch_expand_team<8, 64>(a, grid, wpb, st); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_branchial(BranchialArgs a, const BranchialShape& h, uint32_t grid_cap, hipStream_t st) {
    const uint32_t most = h.max_ne < BR_MAX_EDGES ? h.max_ne : BR_MAX_EDGES;
    a.few_ne = 0;
    if (!a.emit && h.counted) {
        if (a.P.n >= kBranchialQuarter) {
            a.few_ne = most < kBranchialFewEdges ? most : kBranchialFewEdges;
            a.group_words = branchial_count_words(a.few_ne) + (h.triples ? 2 * kBranchialFewTriples : 0u);
            a.lds_per_wave = 16 * a.group_words;
            hipLaunchKernelGGL(k_branchial_count<16>, dim3(grid_for(a.P.n, 16, grid_cap)), dim3(256),
                               (size_t)a.lds_per_wave * 4, st, a);
            if (most <= a.few_ne && !h.rest && !h.triples) return hipGetLastError();
        }
        if (h.matches > kBranchialMany) {
            uint32_t cnt = 0;                          // matches of the largest parent with triples
            if (h.triples) for (cnt = 16; cnt < h.triples && cnt < kBranchialTriples;) cnt <<= 1;
            a.group_words = branchial_count_words(most) + 2 * cnt;
            a.lds_per_wave = 4 * a.group_words;
            hipLaunchKernelGGL(k_branchial_count<64>, dim3(grid_for(a.P.n, 1, grid_cap)), dim3(64),
                               a.lds_per_wave, st, a);
        }
    }
    a.lds_per_wave = branchial_lds_per_wave();
    hipLaunchKernelGGL(k_branchial, dim3(grid_for(a.P.n, 2, grid_cap)), dim3(128), (size_t)a.lds_per_wave * 2, st, a);
    return hipGetLastError();
}

uint32_t wl_states_lds_per_wave(uint32_t max_ne, uint32_t max_nv, uint32_t A, bool lean) {
    const WLSizes z = WLSizes::make(max_ne, max_nv, A, lean);
    // + 64: carving slack; + 64: the team's reduction words at the end
    return (z.bytes(A) + 128u + 15u) & ~15u;
}

template <uint32_t W>
static void launch_wl_states_team(const WLStatesArgs& a, uint32_t grid, uint32_t wpb, hipStream_t st) {
    const uint32_t threads = W == 1 ? 64 * wpb : 64 * W;
    const size_t lds = a.scratch ? 0 : (size_t)a.lds_per_wave * (W == 1 ? wpb : 1);
    if (a.scratch) hipLaunchKernelGGL((k_wl_states<true, W>), dim3(grid), dim3(threads), lds, st, a);
    else hipLaunchKernelGGL((k_wl_states<false, W>), dim3(grid), dim3(threads), lds, st, a);
}

uint32_t wl_states_grid(uint32_t n, uint32_t team, uint32_t wpb, uint32_t grid_cap) {
    return grid_for(n, team == 1 ? wpb : 1, grid_cap);
}

hipError_t launch_wl_states(const WLStatesArgs& a, uint32_t grid_cap, uint32_t wpb, uint32_t team, hipStream_t st) {
    if (!a.n) return hipSuccess;
    if (a.large) return launch_wl_large(a, a.large, team, st);
    const uint32_t grid = wl_states_grid(a.n, team, wpb, grid_cap);
    switch (team) {
        case 1: launch_wl_states_team<1>(a, grid, wpb, st); break;
        case 2: launch_wl_states_team<2>(a, grid, wpb, st); break;
        case 4: launch_wl_states_team<4>(a, grid, wpb, st); break;
        case 8: launch_wl_states_team<8>(a, grid, wpb, st); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_run_totals(const uint64_t* moff, const uint64_t* state_edges, const uint32_t* cnt,
                             const uint32_t* ne, const uint32_t* run, uint32_t n, const uint32_t* b,
                             const uint32_t* e, uint64_t* tot, uint64_t* edges, uint64_t* parent_edges,
                             hipStream_t st) {
    if (n == 0) return hipSuccess;
    const uint32_t waves = (n + kTotalsChunk - 1) / kTotalsChunk;
    hipLaunchKernelGGL(k_run_totals, dim3((waves + 3) / 4), dim3(256), 0, st, moff, state_edges, cnt, ne, run, n, b,
                       e, tot, edges, parent_edges);
    return hipGetLastError();
}

hipError_t launch_mask_counts(const uint32_t* run, const uint8_t* active, uint32_t n, uint32_t* cnt,
                              hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_mask_counts, dim3((n + 255) / 256), dim3(256), 0, st, run, active, n, cnt);
    return hipGetLastError();
}

hipError_t launch_rehash(const uint64_t* ok, uint32_t old_cap, uint64_t* keys, uint32_t mask, hipStream_t st) {
    if (!old_cap) return hipSuccess;
    hipLaunchKernelGGL(k_rehash, dim3((old_cap + 255) / 256), dim3(256), 0, st, ok, old_cap, keys, mask);
    return hipGetLastError();
}

}  // namespace hgx
