// hgx_wl_large.hpp -- the WL canonical hash of a large state of one arity (2..4), by the W waves of a
// workgroup.
//
// The same value as wl_hash_team (hgx_wl.hpp; common/include/hgcommon/wl_core.hpp:67-202) for states
// past hgx_wl_small.hpp's limits whose colours fit the LDS: up to about 12,700 vertex labels, 13 to 14
// bytes of LDS a label. Only what is read or added to at random is kept there -- the colours, and one
// array that is in turn the write cursors, the distinct-count set, the sorted long lists and the
// components; the lists, their offsets, the next colours and the edges are walked in order, so they
// stay in global memory (or in LDS too, where everything fits: ALL). The general hash keeps every
// array in one place: 63 bytes a binary edge in LDS, so a CU holds one state of 2,048 edges, and all
// of them in global memory beyond, where its gathers and atomics are round trips to the L2.
// Vertices are named by their labels, as in hgx_wl_small.hpp.
#pragma once

#include "hgx_wl_small.hpp"

namespace hgx {

constexpr uint32_t kLargeMaxLabels = 16383;      // a list entry is (label << 2) | position in 16 bits
constexpr uint32_t kLargeMaxEntries = 65535;     // entries of a state's lists: places in 16 bits

struct LargeSizes {
    uint32_t NL, NN, CAP, NLONG, NHUGE;
    __host__ __device__ static LargeSizes make(uint32_t ne, uint32_t nl, uint32_t A) {
        LargeSizes z;
        z.NL = nl ? nl : 1;
        z.NN = (ne ? ne : 1) * A * (A - 1);
        z.NLONG = z.NN / 9 + 1;
        z.NHUGE = z.NN / 65 + 1;
        // set slots: load factor 0.67 at most, and 0.83 where the LDS does not hold that (10,500 labels:
        // a child 0.70 ms against 0.75, the state 0.29 against 0.31)
        for (uint32_t spare : {z.NL / 2, z.NL / 5}) {
            z.CAP = z.NL + spare + 8;
            if (z.CAP < z.NN / 2 + 1) z.CAP = z.NN / 2 + 1;  // the sorted lists, if all are long
            if (z.hot() <= 160u << 10) break;
        }
        return z;
    }
    // LDS held whatever the layout, and the rest
    __host__ __device__ uint32_t hot() const {
        return 8 * NL + ((4 * CAP + 7u) & ~7u) + ((2 * NHUGE + 7u) & ~7u) + 256;
    }
    __host__ __device__ uint32_t rest() const {
        auto al = [](uint32_t b) { return (b + 7u) & ~7u; };
        return 8 * NL + al(4 * (NL + 1)) + al(2 * NN) + al(2 * NLONG);
    }
};

struct LargeSpace {
    uint64_t* cur;      // [NL] LDS: occurrences per position (16 bits each), then colours
    uint32_t* set;      // [CAP] LDS: cursors; distinct-count set (label + 1); sorted lists; components
    uint32_t* word;     // [4] LDS
    uint16_t* hl;       // [NHUGE] LDS: vertices with lists above 64 entries
    uint64_t* red;      // [16] LDS: the team's reductions
    uint16_t* q;        // [16] LDS: the match's consumed positions
    uint64_t* nxt;      // [NL]
    uint32_t* off;      // [NL + 1]
    uint16_t* nb;       // [NN]
    uint16_t* lv;       // [NLONG] vertices with lists of 9 to 16 entries from the front, to 64 from the back
    uint32_t NL, CAP, NLONG;
};

// ALL: everything in LDS from `lds`; else the arrays walked in order in global memory from `mem`.
template <bool ALL>
__device__ __forceinline__ void large_bind(LargeSpace& s, uint8_t* lds, uint8_t* mem, const LargeSizes& z) {
    s.cur = (uint64_t*)carve(lds, 8 * z.NL);
    s.set = (uint32_t*)carve(lds, 4 * z.CAP);
    s.word = (uint32_t*)carve(lds, 16);
    s.hl = (uint16_t*)carve(lds, 2 * z.NHUGE);
    s.red = (uint64_t*)carve(lds, 128);
    s.q = (uint16_t*)carve(lds, 32);
    uint8_t* p = nullptr;
    if constexpr (ALL) p = lds;
    else p = mem;
    s.nxt = (uint64_t*)carve(p, 8 * z.NL);
    s.off = (uint32_t*)carve(p, 4 * (z.NL + 1));
    s.nb = (uint16_t*)carve(p, 2 * z.NN);
    s.lv = (uint16_t*)carve(p, 2 * z.NLONG);
    s.NL = z.NL;
    s.CAP = z.CAP;
    s.NLONG = z.NLONG;
}

// Number of distinct colours among the labels that edges hold. The table has an odd number of slots and
// is probed in steps of a power of two, so every sequence visits all of them; eight step lengths keep
// chains short at the load that fits beside the colours (neighbouring slots at 0.89: 27-36% of the
// hash).
template <class TM>
__device__ __forceinline__ uint32_t large_ndistinct(const TM& tm, const LargeSpace& s, uint32_t nl, uint32_t cap) {
    for (uint32_t i = tm.r; i < cap; i += TM::N) s.set[i] = 0;
    tm.sync();
    uint32_t cnt = 0;
    for (uint32_t v = tm.r; v < nl; v += TM::N) {
        if (s.off[v + 1] == s.off[v]) continue;
        const uint64_t x = s.cur[v];
        const uint32_t h = ((uint32_t)(x >> 32) ^ (uint32_t)x) * 0x9E3779B1u;
        uint32_t slot = (uint32_t)(((uint64_t)h * cap) >> 32);
        uint32_t step = 16u << (h & 7u);
        while (step >= cap) step >>= 1;
        while (true) {
            const uint32_t old = atomicCAS(&s.set[slot], 0u, v + 1);
            if (old == 0) { ++cnt; break; }
            if (s.cur[old - 1] == x) break;
            slot += step;
            if (slot >= cap) slot -= cap;
        }
    }
    return tm.sum(cnt);
}

// Rank of x among the 16 values of its row (equal ones by lane), i the lane's place in the row: every
// other lane's value comes by in turn.
template <int J>
__device__ __forceinline__ uint32_t row_rank_from(uint64_t x, uint32_t i) {
    if constexpr (J == 16) return 0;
    else {
        const uint64_t y = dpp<kDppRowRor + J>(x);           // from lane i - J, or 16 + i - J
        return ((y < x || (y == x && i >= (uint32_t)J)) ? 1u : 0u) + row_rank_from<J + 1>(x, i);
    }
}
__device__ __forceinline__ uint32_t row_rank(uint64_t x, uint32_t i) { return row_rank_from<1>(x, i); }

// Entries [a0, a0 + 64) of the list [b, b + n) to their places in order, by a wave: every entry's value comes
// by in turn, 64 at a time by lane reads (equal ones by place).
__device__ __forceinline__ void large_rank_unit(const LargeSpace& s, uint16_t* order, uint32_t b, uint32_t n,
                                                uint32_t a0, uint32_t lane) {
    auto entry = [&](uint32_t j) { return (uint32_t)s.nb[b + (j < n ? j : 0u)]; };
    const uint32_t tx = entry(a0 + lane);
    const uint64_t x = fnv(s.cur[tx >> 2], tx & 3u);
    uint32_t r = 0;
    uint32_t ty = entry(lane);
    for (uint32_t c0 = 0; c0 < n; c0 += WAVE) {
        const uint64_t y = fnv(s.cur[ty >> 2], ty & 3u);
        ty = entry(c0 + WAVE + lane);                         // (the next ones' read meanwhile)
        const uint32_t m = n - c0 < WAVE ? n - c0 : WAVE;
        auto at = [&](uint32_t i) {
            return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(y >> 32), (int)i) << 32) |
                   (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)y, (int)i);
        };
        if (c0 < a0) {
#pragma unroll 8
            for (uint32_t i = 0; i < m; ++i) r += at(i) <= x ? 1u : 0u;
        } else if (c0 > a0) {
#pragma unroll 8
            for (uint32_t i = 0; i < m; ++i) r += at(i) < x ? 1u : 0u;
        } else {
#pragma unroll 8
            for (uint32_t i = 0; i < m; ++i) {
                const uint64_t z = at(i);
                r += (z < x || (z == x && i < lane)) ? 1u : 0u;
            }
        }
    }
    if (a0 + lane < n) order[b + r] = (uint16_t)tx;
}

// ev: the state's edges at stride A in global memory; every edge has arity ua (UA when it is known).
template <uint32_t UA, bool ALL, class TM>
__device__ __forceinline__ uint64_t wl_hash_large(LargeSpace s, const TM& tm, const uint32_t* ev, uint32_t A,
                                                  uint32_t nE, uint32_t nl, uint32_t ua_) {
    const uint32_t ua = UA ? UA : ua_;
    const uint32_t l = tm.r;
    constexpr uint32_t N = TM::N;
    if (nE == 0) return EMPTY_STATE_HASH;     // hypergraph.cpp:743-745
    auto edge = [&](uint32_t e, uint32_t (&x)[4]) {
        if constexpr (UA == 2) {
            const uint2 t = ((const uint2*)ev)[e];
            x[0] = t.x; x[1] = t.y;
        } else {
            for (uint32_t p = 0; p < 4; ++p) x[p] = p < ua ? ev[(size_t)e * A + p] : 0u;
        }
    };

    for (uint32_t v = l; v < nl; v += N) s.cur[v] = 0;
    if (l < 3) s.word[l] = 0;
    tm.sync();
    for (uint32_t e = l; e < nE; e += N) {
        uint32_t x[4];
        edge(e, x);
#pragma unroll
        for (uint32_t p = 0; p < (UA ? UA : 4u); ++p)
            if (p < ua) atomicAdd((unsigned long long*)&s.cur[x[p]], 1ull << (16 * p));
    }
    tm.sync();
    // initial colours (wl_core.hpp:93-107), offsets, and the vertices with long lists
    uint32_t mine = 0, nslots = 0;
    for (uint32_t base = 0; base < nl; base += N) {
        const uint32_t v = base + l;
        const uint64_t c = v < nl ? s.cur[v] : 0ull;
        const uint32_t d = (uint32_t)(c & 0xFFFFu) + (uint32_t)((c >> 16) & 0xFFFFu) + (uint32_t)((c >> 32) & 0xFFFFu) +
                           (uint32_t)(c >> 48);
        const uint32_t n = d * (ua - 1);
        mine += d != 0 ? 1u : 0u;
        uint32_t round;
        const uint32_t inc = tm.incl_scan(n, round);
        if (v < nl) {
            const uint32_t o = nslots + inc - n;
            s.off[v] = o;
            s.set[v] = o;                      // write cursor
            uint64_t h = fnv(FNV_OFFSET, d);
#pragma unroll
            for (uint32_t p = 0; p < (UA ? UA : 4u); ++p)
                for (uint32_t i = (uint32_t)(c >> (16 * p)) & 0xFFFFu; i > 0; --i) h = fnv(fnv(h, ua), p);
            s.cur[v] = h;
            if (n > WAVE) s.hl[atomicAdd(&s.word[2], 1u)] = (uint16_t)v;
            else if (n > 16) s.lv[s.NLONG - 1 - atomicAdd(&s.word[1], 1u)] = (uint16_t)v;
            else if (n > 8) s.lv[atomicAdd(&s.word[0], 1u)] = (uint16_t)v;
        }
        nslots += round;
    }
    if (l == 0) s.off[nl] = nslots;
    const uint32_t nV = tm.sum(mine);
    tm.sync();
    const uint32_t nmed = s.word[0], nlong = s.word[1], nhuge = s.word[2];
    for (uint32_t e = l; e < nE; e += N) {
        uint32_t x[4];
        edge(e, x);
        if constexpr (UA == 2) {
            s.nb[atomicAdd(&s.set[x[0]], 1u)] = (uint16_t)((x[1] << 2) | 1u);
            s.nb[atomicAdd(&s.set[x[1]], 1u)] = (uint16_t)(x[0] << 2);
        } else {
            for (uint32_t p = 0; p < ua; ++p) {
                uint32_t o = atomicAdd(&s.set[x[p]], ua - 1);
                for (uint32_t k = 0; k < ua; ++k)
                    if (k != p) s.nb[o++] = (uint16_t)((x[k] << 2) | k);
            }
        }
    }
    tm.sync();
    uint32_t cap = 2 * nV + 1;
    if (cap > s.CAP) cap = (s.CAP - 1) | 1u;
    uint32_t prev_d = large_ndistinct(tm, s, nl, cap);

    // refinement (wl_core.hpp:119-141)
    const uint32_t w = l / WAVE, lane = lane_id();
    for (uint32_t it = 0; it < WL_MAX_ITERS; ++it) {
        tm.sync();
        // Lists above 64 entries: 64 of a list's entries against all of it is a wave's unit of work, dealt
        // to the waves in turn over all lists, the entries left in order in LDS; then a lane folds a list.
        // (One list after another by the workgroup, folded from global memory: 2,000 edges on 40 vertices
        // 1.96 ms, 0.14 so, 0.22 by the general hash; 12,000 on 200 0.56, general 3.0.)
        uint16_t* order = (uint16_t*)s.set;
        uint32_t u = (uint32_t)__builtin_amdgcn_readfirstlane((int)w);
        for (uint32_t k0 = 0; k0 < nhuge; k0 += WAVE) {
            const uint32_t hv = k0 + lane < nhuge ? s.hl[k0 + lane] : s.hl[0];
            const uint32_t hb = s.off[hv], hn = s.off[hv + 1] - hb;
            const uint32_t m = nhuge - k0 < WAVE ? nhuge - k0 : WAVE;
            for (uint32_t k = 0; k < m; ++k) {
                const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)hb, (int)k);
                const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)hn, (int)k);
                const uint32_t units = (n + WAVE - 1) / WAVE;
                for (; u < units; u += N / WAVE) large_rank_unit(s, order, b, n, u * WAVE, lane);
                u -= units;
            }
        }
        if (nhuge) {
            tm.sync();
            for (uint32_t k = l; k < nhuge; k += N) {
                const uint32_t v = s.hl[k], b = s.off[v], e = s.off[v + 1];
                uint64_t h = s.cur[v];
#pragma unroll 8
                for (uint32_t i = b; i < e; ++i) {
                    const uint32_t t = order[i];
                    h = fnv(h, fnv(s.cur[t >> 2], t & 3u));
                }
                s.nxt[v] = h;
            }
        }
        // 9 to 16 entries: four lists a wave, an entry per lane of a row, ranked against the row's
        // others by rotation and folded by shifting them down to its first lane
        for (uint32_t k0 = 4 * w; k0 < nmed; k0 += 4 * (N / WAVE)) {
            const uint32_t k = k0 + (lane >> 4), i = lane & 15u;
            const uint32_t v = k < nmed ? s.lv[k] : 0u;
            const uint32_t b = k < nmed ? s.off[v] : 0u, n = k < nmed ? s.off[v + 1] - b : 0u;
            uint64_t x = ~0ull;
            if (i < n) {
                const uint32_t t = s.nb[b + i];
                x = fnv(s.cur[t >> 2], t & 3u);
            }
            const uint32_t dst = (lane & ~15u) | row_rank(x, i);
            const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_permute((int)(dst << 2), (int)(uint32_t)x);
            const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_permute((int)(dst << 2), (int)(uint32_t)(x >> 32));
            x = ((uint64_t)hi << 32) | lo;
            uint64_t h = s.cur[v];
            for (uint32_t j = 0; j < 16; ++j) {
                h = j < n ? fnv(h, x) : h;
                x = dpp<kDppRowShl + 1>(x);
            }
            if (i == 0 && k < nmed) s.nxt[v] = h;
        }
        // 17 to 64: a list per wave
        for (uint32_t k = w; k < nlong; k += N / WAVE) {
            const uint32_t v = s.lv[s.NLONG - 1 - k];
            const uint32_t b = s.off[v], n = s.off[v + 1] - b;
            uint64_t x = 0;
            if (lane < n) {
                const uint32_t t = s.nb[b + lane];
                x = fnv(s.cur[t >> 2], t & 3u);
            }
            const uint32_t un = (uint32_t)__builtin_amdgcn_readfirstlane((int)n);
            uint32_t r = 0;
            for (uint32_t i = 0; i < un; ++i) {
                const uint64_t y = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), (int)i) << 32) |
                                   (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, (int)i);
                r += (y < x || (y == x && i < lane)) ? 1u : 0u;
            }
            // sorted: lane r takes the entry of rank r
            uint64_t sx;
            {
                const uint32_t dst = lane < n ? r : lane;
                const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_permute((int)(dst << 2), (int)(uint32_t)x);
                const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_permute((int)(dst << 2), (int)(uint32_t)(x >> 32));
                sx = ((uint64_t)hi << 32) | lo;
            }
            uint64_t h = s.cur[v];
            for (uint32_t i = 0; i < un; ++i) {
                const uint64_t y = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(sx >> 32), (int)i) << 32) |
                                   (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)sx, (int)i);
                h = fnv(h, y);
            }
            if (lane == 0) s.nxt[v] = h;
        }
        for (uint32_t v = l; v < nl; v += N) {
            const uint32_t b = s.off[v], n = s.off[v + 1] - b;
            if (n == 0 || n > 8) continue;
            uint64_t h = s.cur[v];
            if (__ballot(n > 3) == 0)
                h = __ballot(n > 2) == 0 ? small_fold<2>(s.nb, s.cur, b, n, h) : small_fold<3>(s.nb, s.cur, b, n, h);
            else if (__ballot(n > 6) == 0)
                h = __ballot(n > 4) == 0 ? small_fold<4>(s.nb, s.cur, b, n, h) : small_fold<6>(s.nb, s.cur, b, n, h);
            else
                h = small_fold<8>(s.nb, s.cur, b, n, h);
            s.nxt[v] = h;
        }
        tm.sync();
        if constexpr (ALL) {
            uint64_t* t = s.cur; s.cur = s.nxt; s.nxt = t;
        } else {
            for (uint32_t v = l; v < nl; v += N)
                if (s.off[v + 1] != s.off[v]) s.cur[v] = s.nxt[v];
            tm.sync();
        }
        const uint32_t d = large_ndistinct(tm, s, nl, cap);
        if (d == prev_d) break;
        prev_d = d;
    }

    // connected components (wl_core.hpp:143-168): the larger root of an edge's ends hooks onto the
    // smaller, then paths halve; at the end a component's labels all name its smallest
    tm.sync();
    uint32_t* comp = s.set;
    for (uint32_t v = l; v < nl; v += N) comp[v] = v;
    tm.sync();
    while (true) {
        bool changed = false;
        for (uint32_t e = l; e < nE; e += N) {
            uint32_t x[4];
            edge(e, x);
            uint32_t a = comp[x[0]];
#pragma unroll
            for (uint32_t p = 1; p < (UA ? UA : 4u); ++p) {
                if (p >= ua) break;
                const uint32_t c = comp[x[p]];
                const uint32_t lo = a < c ? a : c, hi = a < c ? c : a;
                if (lo != hi) { atomicMin(&comp[hi], lo); changed = true; }
                a = lo;
            }
        }
        if (!tm.any(changed)) break;            // (a barrier)
        for (uint32_t k = 0; k < 2; ++k) {
            for (uint32_t v = l; v < nl; v += N) {
                const uint32_t c = comp[v], cc = comp[c];
                if (cc < c) atomicMin(&comp[v], cc);
            }
            tm.sync();
        }
    }

    // folds (wl_core.hpp:170-201). A component's vertex sum is gathered in its root's own entry:
    // roots are only added to, the others only read.
    uint64_t vsum = 0, esum = 0, csum = 0;
    for (uint32_t e = l; e < nE; e += N) {
        uint32_t x[4];
        edge(e, x);
        uint64_t eh = fnv(FNV_OFFSET, ua);
#pragma unroll
        for (uint32_t p = 0; p < (UA ? UA : 4u); ++p)
            if (p < ua) eh = fnv(eh, s.cur[x[p]]);
        esum += splitmix(eh);
    }
    tm.sync();
    bool many = false;
    uint32_t x0[4];
    edge(0, x0);
    const uint32_t c0 = comp[x0[0]];
    for (uint32_t v = l; v < nl; v += N) {
        if (s.off[v + 1] == s.off[v]) continue;
        const uint64_t m = splitmix(s.cur[v]);
        vsum += m;
        s.cur[v] = m;
        many |= comp[v] != c0;
    }
    vsum = tm.sum64(vsum);
    if (tm.any(many)) {                          // (barriers)
        for (uint32_t v = l; v < nl; v += N)
            if (s.off[v + 1] != s.off[v] && comp[v] != v)
                atomicAdd((unsigned long long*)&s.cur[comp[v]], (unsigned long long)s.cur[v]);
        tm.sync();
        for (uint32_t v = l; v < nl; v += N) {
            if (s.off[v + 1] != s.off[v] && comp[v] == v) s.nxt[v] = s.cur[v];
        }
        tm.sync();
        uint64_t* cnt = s.cur;                   // vertices, and edges in the upper half
        for (uint32_t v = l; v < nl; v += N) cnt[v] = 0;
        tm.sync();
        for (uint32_t v = l; v < nl; v += N)
            if (s.off[v + 1] != s.off[v]) atomicAdd((unsigned long long*)&cnt[comp[v]], 1ull);
        for (uint32_t e = l; e < nE; e += N) {
            uint32_t x[4];
            edge(e, x);
            atomicAdd((unsigned long long*)&cnt[comp[x[0]]], 1ull << 32);
        }
        tm.sync();
        for (uint32_t v = l; v < nl; v += N)
            if (s.off[v + 1] != s.off[v] && comp[v] == v)
                csum += splitmix(fnv(fnv(FNV_OFFSET, cnt[v]), s.nxt[v]));
        csum = tm.sum64(csum);
    } else {
        csum = splitmix(fnv(fnv(FNV_OFFSET, ((uint64_t)nE << 32) | nV), vsum));
    }
    esum = tm.sum64(esum);
    uint64_t hash = fnv(FNV_OFFSET, nV);
    hash = fnv(hash, nE);
    hash = fnv(hash, vsum);
    hash = fnv(hash, esum);
    return fnv(hash, csum);
}

}  // namespace hgx
