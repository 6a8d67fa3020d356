// hgx_wl_small.hpp -- the WL canonical hash of a small state of one arity (2..4), by a team of 8 to
// 64 lanes of one wave.
//
// The same value as wl_hash_team (hgx_wl.hpp; common/include/hgcommon/wl_core.hpp:67-202) for states
// of at most 255 edges and 255 vertex labels, every edge of arity ua. What bounds the general
// hash on such states is instruction issue and the LDS round trips between its phases, so this
// one has fewer of both:
//   - vertices are named by their labels (below 256, one byte), not renumbered densely: a label no
//     edge holds has degree 0 and takes part in nothing. The numbering scan, its mark and remap
//     passes and the label arrays are gone, and an edge is ua bytes;
//   - one packed counter per label (8 bits per position) gives degree and initial colour;
//   - vertices of at most 2, 4 or 8 neighbours fold them sorted in registers by the smallest network
//     that fits every lane of the round; only longer lists are rank-sorted through LDS, by the
//     whole team, so one hub does not send every vertex that way;
//   - components hook roots (each pass joins whole trees), and a connected state -- most are -- folds
//     its one component from sums already at hand, without atomics;
//   - the distinct count keeps vertex labels in its set, not colours, and a long list is sorted in
//     the memory of the set and the cursors, both idle then: 2.8 KiB at 64 edges and 80 labels
//     (4.6 KiB in the general lean workspace), so more states are in flight.
#pragma once

#include "hgx_wl.hpp"

namespace hgx {

constexpr uint32_t kSmallMaxEdges = 255, kSmallMaxLabels = 255;

struct SmallSizes {
    uint32_t NE, NL, NN, HT, RB, NX;
    __host__ __device__ static SmallSizes make(uint32_t ne, uint32_t nl, uint32_t A) {
        SmallSizes z;
        z.NE = ne ? ne : 1;
        z.NL = nl ? nl : 1;
        z.NN = z.NE * A * (A - 1);
        const uint32_t nv = z.NL < z.NE * A ? z.NL : z.NE * A;     // vertices that can occur
        z.HT = 64;
        while (z.HT < nv + nv / 4 + 1) z.HT <<= 1;                 // load factor <= 0.8
        uint32_t rb = 12 * z.NL;                                   // component counts and labels
        if (rb < 4 * z.HT) rb = 4 * z.HT;
        if (rb < 2 * z.NN) rb = 2 * z.NN;                          // one list of every entry, by index
        z.RB = (rb + 15u) & ~15u;
        z.NX = z.RB / 8 < z.NN ? z.RB / 8 : z.NN;
        if (z.NX > 255) z.NX = 255;                                // long-list entries, numbered in a byte
        return z;
    }
    __host__ __device__ uint32_t bytes(uint32_t A) const {
        auto al = [](uint32_t b) { return (b + 7u) & ~7u; };
        return RB + 16 * NL + al(2 * (NL + 1)) + al(2 * NN) + 2 * al(NX) + al(4 * (NX / 9 + 1)) + al(NX / 9 + 1) +
               al(NE * A);
    }
};

struct SmallSpace {
    uint64_t* vals;     // [NX] long lists' values while they are sorted; in the same memory (RB bytes):
    uint32_t* set;      //   [HT] the distinct-count set: label + 1 of each colour's first holder
    uint64_t* cnt;      //   [NL] component counts, then
    uint32_t* pc;       //   [NL] occurrences per position (8 bits each), write cursors; component labels
    uint64_t* cur;      // [NL] colours
    uint64_t* nxt;      // [NL] the next round's
    uint16_t* off;      // [NL + 1] CSR of the neighbour lists
    uint16_t* nb;       // [NN] neighbours: (label << 2) | position
    uint8_t* own;       // [NX] long lists: each entry's list
    uint8_t* perm;      // [NX] the entry at each rank
    uint32_t* lt;       // [NX / 9 + 1] each list's place in nb, first entry and length (12, 8, 8 bits)
    uint8_t* lv;        // [NX / 9 + 1] its vertex
    uint8_t* ev;        // [NE * ua] edges
    uint32_t nx;
};

__device__ __forceinline__ void small_bind(SmallSpace& s, uint8_t* p, const SmallSizes& z, uint32_t A) {
    s.vals = (uint64_t*)carve(p, z.RB);
    s.cnt = s.vals;
    s.pc = (uint32_t*)(s.vals + z.NL);
    s.set = (uint32_t*)s.vals;
    s.cur = (uint64_t*)carve(p, 8 * z.NL);
    s.nxt = (uint64_t*)carve(p, 8 * z.NL);
    s.off = (uint16_t*)carve(p, 2 * (z.NL + 1));
    s.nb = (uint16_t*)carve(p, 2 * z.NN);
    s.own = carve(p, z.NX);
    s.perm = carve(p, z.NX);
    s.lt = (uint32_t*)carve(p, 4 * (z.NX / 9 + 1));
    s.lv = carve(p, z.NX / 9 + 1);
    s.ev = carve(p, z.NE * A);
    s.nx = z.NX;
}

// Exact number of distinct colours among the used labels (bit k of `used`: label k * N + rank).
template <class TM>
__device__ __forceinline__ uint32_t small_ndistinct(const TM& tm, const SmallSpace& s, const uint64_t* cur,
                                                    uint32_t nl, uint32_t used, uint32_t mask) {
    for (uint32_t i = tm.r; i <= mask / 4; i += TM::N) ((uint4*)s.set)[i] = make_uint4(0, 0, 0, 0);
    tm.sync();
    uint32_t cnt = 0;
    for (uint32_t v = tm.r, u = used; v < nl; v += TM::N, u >>= 1) {
        if (!(u & 1u)) continue;
        const uint64_t x = cur[v];
        uint32_t slot = (((uint32_t)(x >> 32) ^ (uint32_t)x) * 0x9E3779B1u >> 16) & mask;
        while (true) {
            const uint32_t old = atomicCAS(&s.set[slot], 0u, v + 1);
            if (old == 0) { ++cnt; break; }
            if (cur[old - 1] == x) break;
            slot = (slot + 1) & mask;
        }
    }
    return tm.sum(cnt);
}

#define HGX_CE(a, b) { const uint64_t lo_ = x[a] < x[b] ? x[a] : x[b]; \
                       const uint64_t hi_ = x[a] < x[b] ? x[b] : x[a]; x[a] = lo_; x[b] = hi_; }
// Colour h folded with the values of a list of at most M entries in ascending order.
template <int M>
__device__ __forceinline__ uint64_t small_fold(const uint16_t* nb, const uint64_t* cur, uint32_t b, uint32_t n,
                                               uint64_t h) {
    uint64_t x[M];
#pragma unroll
    for (int i = 0; i < M; ++i) {
        const uint32_t t = nb[(uint32_t)i < n ? b + i : b];
        const uint64_t val = fnv(cur[t >> 2], t & 3u);
        x[i] = (uint32_t)i < n ? val : ~0ull;
    }
    if constexpr (M == 2) { HGX_CE(0, 1) }
    else if constexpr (M == 3) { HGX_CE(0, 1) HGX_CE(0, 2) HGX_CE(1, 2) }
    else if constexpr (M == 4) { HGX_CE(0, 1) HGX_CE(2, 3) HGX_CE(0, 2) HGX_CE(1, 3) HGX_CE(1, 2) }
    else if constexpr (M == 6) {
        HGX_CE(0, 5) HGX_CE(1, 3) HGX_CE(2, 4) HGX_CE(1, 2) HGX_CE(3, 4) HGX_CE(0, 3)
        HGX_CE(2, 5) HGX_CE(0, 1) HGX_CE(2, 3) HGX_CE(4, 5) HGX_CE(1, 2) HGX_CE(3, 4)
    } else {
        static_assert(M == 8, "list lengths with a network");
        sort8(x);
    }
#pragma unroll
    for (int i = 0; i < M; ++i) {
        const uint64_t y = fnv(h, x[i]);
        h = (uint32_t)i < n ? y : h;
    }
    return h;
}
#undef HGX_CE

// Colours of the vertices with long lists (nlong lists, numbered entries [first, total)), into nxt.
template <class TM>
__device__ __forceinline__ void small_long_lists(const TM& tm, const SmallSpace& s, const uint64_t* cur, uint64_t* nxt,
                                                 uint32_t nlong, uint32_t first, uint32_t total) {
    for (uint32_t f = first + tm.r; f < total; f += TM::N) {
        const uint32_t d = s.lt[s.own[f]];
        const uint32_t t = s.nb[(d & 0xFFFu) + f - ((d >> 12) & 0xFFu)];
        s.vals[f] = fnv(cur[t >> 2], t & 3u);
    }
    tm.sync();
    for (uint32_t f = first + tm.r; f < total; f += TM::N) {   // an entry's rank: smaller ones, then by place
        const uint32_t d = s.lt[s.own[f]];
        const uint32_t fo = (d >> 12) & 0xFFu, n = d >> 20;
        const uint64_t x = s.vals[f];
        uint32_t r = fo;
#pragma unroll 4
        for (uint32_t i = fo; i < fo + n; ++i) {
            const uint64_t y = s.vals[i];
            r += (y < x || (y == x && i < f)) ? 1u : 0u;
        }
        s.perm[r] = (uint8_t)f;
    }
    tm.sync();
    for (uint32_t k = tm.r; k < nlong; k += TM::N) {
        const uint32_t d = s.lt[k], v = s.lv[k];
        const uint32_t fo = (d >> 12) & 0xFFu, n = d >> 20;
        uint64_t h = cur[v];
#pragma unroll 4
        for (uint32_t i = fo; i < fo + n; ++i) h = fnv(h, s.vals[s.perm[i]]);
        nxt[v] = h;
    }
    tm.sync();
}

// Table of the lists above 8 and up to nx / 2 entries that begin in the window [lo, lo + window) of such lists'
// entries: number of lists, numbered entries [first, end). Returns the entries of all windows.
template <class TM>
__device__ __forceinline__ uint32_t small_window(const TM& tm, const SmallSpace& s, uint32_t nl, uint32_t lo,
                                                 uint32_t window, uint32_t& nlong, uint32_t& first, uint32_t& end) {
    constexpr uint32_t N = TM::N;
    uint32_t total = 0, start = 0xFFu, stop = 0;               // start, stop: this lane's part
    nlong = 0;
    for (uint32_t base = 0; base < nl; base += N) {
        const uint32_t v = base + tm.r;
        const uint32_t b = v < nl ? s.off[v] : 0u;
        uint32_t n = v < nl ? s.off[v + 1] - b : 0u;
        if (n <= 8 || n > s.nx / 2) n = 0;
        uint32_t round;
        const uint32_t fo = total + tm.incl_scan(n, round) - n - lo;   // (past the window where it is below 0)
        const bool in = n != 0 && fo < window;
        const uint64_t mask = tm.ballot(in);
        if (in) {
            const uint32_t i = nlong + (uint32_t)__popcll(mask & ((1ull << tm.r) - 1ull));
            s.lt[i] = b | (fo << 12) | (n << 20);
            s.lv[i] = (uint8_t)v;
            for (uint32_t j = fo; j < fo + n; ++j) s.own[j] = (uint8_t)i;
            start = fo < start ? fo : start;
            stop = fo + n;
        }
        nlong += (uint32_t)__popcll(mask);
        total += round;
    }
    tm.sync();
    first = 0xFFu - tm.max(0xFFu - start);
    end = tm.max(stop);
    return total;
}

// Lists of more than nx / 2 entries, a few at most: N entries against N at a time by lane reads, the entries
// left in order in the sort area, then folded a lane each.
template <class TM>
__device__ __forceinline__ void small_huge_lists(const TM& tm, const SmallSpace& s, const uint64_t* cur, uint64_t* nxt,
                                                 uint32_t nl) {
    constexpr uint32_t N = TM::N;
    const uint32_t l = tm.r;
    uint16_t* order = (uint16_t*)s.vals;
    bool any = false;
    for (uint32_t base = 0; base < nl; base += N) {
        const uint32_t v0 = base + l;
        for (uint64_t left = tm.ballot(v0 < nl && s.off[v0 + 1] - s.off[v0] > s.nx / 2); left; left &= left - 1) {
            const uint32_t v = base + (uint32_t)__builtin_ctzll(left);
            const uint32_t b = s.off[v], n = s.off[v + 1] - b;
            any = true;
            auto value = [&](uint32_t j) {
                const uint32_t t = s.nb[b + (j < n ? j : 0u)];
                return fnv(cur[t >> 2], t & 3u);
            };
            for (uint32_t a0 = 0; a0 < n; a0 += N) {
                const uint32_t j = a0 + l;
                const uint64_t x = value(j);
                uint32_t r = 0;
                for (uint32_t c0 = 0; c0 < n; c0 += N) {
                    const uint64_t y = value(c0 + l);
                    const uint32_t m = n - c0 < N ? n - c0 : N;
#pragma unroll 4
                    for (uint32_t i = 0; i < m; ++i) {
                        const uint64_t z = ((uint64_t)tm.read_lane((uint32_t)(y >> 32), i) << 32) |
                                           tm.read_lane((uint32_t)y, i);
                        r += (z < x || (z == x && c0 + i < j)) ? 1u : 0u;
                    }
                }
                if (j < n) order[b + r] = s.nb[b + j];
            }
        }
    }
    tm.sync();
    if (!any) return;
    for (uint32_t v = l; v < nl; v += N) {
        const uint32_t b = s.off[v], n = s.off[v + 1] - b;
        if (n <= s.nx / 2) continue;
        uint64_t h = cur[v];
#pragma unroll 4
        for (uint32_t i = b; i < b + n; ++i) {
            const uint32_t t = order[i];
            h = fnv(h, fnv(cur[t >> 2], t & 3u));
        }
        nxt[v] = h;
    }
    tm.sync();
}

// UA: the arity when it is known at compile time, else 0 (then ua).
template <uint32_t UA, class TM>
__device__ __forceinline__ uint64_t wl_hash_small(const SmallSpace& s, const TM& tm, uint32_t nE, uint32_t nl,
                                                  uint32_t ua_) {
    const uint32_t ua = UA ? UA : ua_;
    const uint32_t l = tm.r;
    constexpr uint32_t N = TM::N;
    if (nE == 0) return EMPTY_STATE_HASH;     // hypergraph.cpp:743-745

    for (uint32_t v = l; v < nl; v += N) s.pc[v] = 0;
    tm.sync();
    for (uint32_t e = l; e < nE; e += N) {
        if constexpr (UA == 2) {
            atomicAdd(&s.pc[s.ev[e * 2]], 1u);
            atomicAdd(&s.pc[s.ev[e * 2 + 1]], 1u << 8);
        } else {
            for (uint32_t p = 0; p < ua; ++p) atomicAdd(&s.pc[s.ev[e * ua + p]], 1u << (8 * p));
        }
    }
    tm.sync();
    // Initial colours (wl_core.hpp:93-107: fnv(degree), then each occurrence's (arity, position) in
    // ascending order; nothing truncates at these arities), the lists' offsets, and the long lists:
    // above 8 entries, entries numbered through all of them.
    uint32_t nV = 0, nslots = 0, nlong = 0, nent = 0;
    uint32_t used = 0, shrt = 0;               // bit k: label k * N + l has edges / a short list
    for (uint32_t base = 0, k = 0; base < nl; base += N, ++k) {
        const uint32_t v = base + l;
        const uint32_t c = v < nl ? s.pc[v] : 0u;
        const uint32_t d = (c & 0xFFu) + ((c >> 8) & 0xFFu) + ((c >> 16) & 0xFFu) + (c >> 24);
        const uint32_t n = d * (ua - 1);
        nV += (uint32_t)__popcll(tm.ballot(d != 0));
        used |= (d != 0 ? 1u : 0u) << k;
        shrt |= (d != 0 && n <= 8 ? 1u : 0u) << k;
        uint32_t round;
        const uint32_t inc = tm.incl_scan(n, round);
        const uint32_t o = nslots + inc - n;
        nslots += round;
        if (v < nl) {
            s.off[v] = (uint16_t)o;
            s.pc[v] = o;                       // write cursor
            uint64_t h = fnv(FNV_OFFSET, d);
#pragma unroll
            for (uint32_t p = 0; p < (UA ? UA : 4u); ++p)
                for (uint32_t i = (c >> (8 * p)) & 0xFFu; i > 0; --i) h = fnv(fnv(h, ua), p);
            s.cur[v] = h;
        }
        const uint64_t lng = tm.ballot(n > 8);
        if (lng) {
            uint32_t ents;
            const uint32_t fo = nent + tm.incl_scan(n > 8 ? n : 0u, ents) - n;
            nent += ents;
            const uint32_t i = nlong + (uint32_t)__popcll(lng & ((1ull << l) - 1ull));
            nlong += (uint32_t)__popcll(lng);
            if (n > 8 && fo + n <= s.nx) {
                s.lt[i] = o | (fo << 12) | (n << 20);
                s.lv[i] = (uint8_t)v;
                for (uint32_t j = fo; j < fo + n; ++j) s.own[j] = (uint8_t)i;
            }
        }
    }
    if (l == 0) s.off[nl] = (uint16_t)nslots;
    tm.sync();
    for (uint32_t e = l; e < nE; e += N) {
        if constexpr (UA == 2) {
            const uint32_t x = s.ev[e * 2], y = s.ev[e * 2 + 1];
            const uint32_t ox = atomicAdd(&s.pc[x], 1u), oy = atomicAdd(&s.pc[y], 1u);
            s.nb[ox] = (uint16_t)((y << 2) | 1u);
            s.nb[oy] = (uint16_t)(x << 2);
        } else {
            for (uint32_t p = 0; p < ua; ++p) {
                uint32_t o = atomicAdd(&s.pc[s.ev[e * ua + p]], ua - 1);
                for (uint32_t k = 0; k < ua; ++k)
                    if (k != p) s.nb[o++] = (uint16_t)(((uint32_t)s.ev[e * ua + k] << 2) | k);
            }
        }
    }
    tm.sync();
    uint32_t ht = 64;
    while (ht < nV + nV / 4 + 1) ht <<= 1;
    uint64_t* cur = s.cur;
    uint64_t* nxt = s.nxt;
    uint32_t prev_d = small_ndistinct(tm, s, cur, nl, used, ht - 1);

    // refinement (wl_core.hpp:119-141): the sorted multiset of fnv(colour, position) over the
    // neighbour list, folded in order
    for (uint32_t it = 0; it < WL_MAX_ITERS; ++it) {
        tm.sync();
        if (nent) {
            // Long lists with more entries than are numbered (dense states, high arities): those up to
            // half as many in windows, short enough that the longest list beginning at a window's end
            // still fits; the table is the window's then, formed anew each time. 240 edges on 30
            // vertices, 3.8 k children: 0.33 ms with one list after another, 0.085 so (general 0.19).
            const bool many = nent > s.nx;
            uint32_t first = 0, end = nent, all = 0, window = 0;
            if (many) {
                uint32_t longest = 0;
                for (uint32_t v = l; v < nl; v += N) {
                    const uint32_t n = s.off[v + 1] - s.off[v];
                    if (n <= s.nx / 2 && n > longest) longest = n;
                }
                window = s.nx + 1 - tm.max(longest);
            }
            for (uint32_t lo = 0;;) {
                if (many) all = small_window(tm, s, nl, lo, window, nlong, first, end);
                small_long_lists(tm, s, cur, nxt, nlong, first, end);
                lo += window;
                if (lo >= all) break;
            }
            if (many) small_huge_lists(tm, s, cur, nxt, nl);
        }
        for (uint32_t v = l, u = shrt; v < nl; v += N, u >>= 1) {
            if (!(u & 1u)) continue;
            const uint32_t b = s.off[v], n = s.off[v + 1] - b;
            uint64_t h = cur[v];
            // the smallest network that fits every lane here
            if (__ballot(n > 3) == 0)
                h = __ballot(n > 2) == 0 ? small_fold<2>(s.nb, cur, b, n, h) : small_fold<3>(s.nb, cur, b, n, h);
            else if (__ballot(n > 6) == 0)
                h = __ballot(n > 4) == 0 ? small_fold<4>(s.nb, cur, b, n, h) : small_fold<6>(s.nb, cur, b, n, h);
            else
                h = small_fold<8>(s.nb, cur, b, n, h);
            nxt[v] = h;
        }
        tm.sync();
        uint64_t* t = cur; cur = nxt; nxt = t;
        const uint32_t d = small_ndistinct(tm, s, cur, nl, used, ht - 1);
        if (d == prev_d) break;
        prev_d = d;
    }

    // connected components (wl_core.hpp:143-168): the larger root of an edge's ends hooks onto the
    // smaller, then paths halve; at the end a component's labels all name its smallest
    tm.sync();
    uint32_t* comp = s.pc;
    for (uint32_t v = l; v < nl; v += N) comp[v] = v;
    tm.sync();
    while (true) {
        bool changed = false;
        for (uint32_t e = l; e < nE; e += N) {
            uint32_t a = comp[s.ev[e * ua]];
#pragma unroll
            for (uint32_t p = 1; p < ua; ++p) {
                const uint32_t c = comp[s.ev[e * ua + p]];
                const uint32_t lo = a < c ? a : c, hi = a < c ? c : a;
                if (lo != hi) { atomicMin(&comp[hi], lo); changed = true; }
                a = lo;
            }
        }
        tm.sync();
        if (!tm.any(changed)) break;
        for (uint32_t k = 0; k < 2; ++k) {
            for (uint32_t v = l; v < nl; v += N) {
                const uint32_t c = comp[v], cc = comp[c];
                if (cc != c) comp[v] = cc;
            }
            tm.sync();
        }
    }

    // folds (wl_core.hpp:170-201)
    uint64_t vsum = 0, esum = 0, csum = 0;
    bool many = false;                        // a second component
    const uint32_t c0 = comp[s.ev[0]];
    for (uint32_t v = l, u = used; v < nl; v += N, u >>= 1) {
        if (!(u & 1u)) continue;
        vsum += splitmix(cur[v]);
        many |= comp[v] != c0;
    }
    for (uint32_t e = l; e < nE; e += N) {
        uint64_t eh = fnv(FNV_OFFSET, ua);
#pragma unroll
        for (uint32_t p = 0; p < ua; ++p) eh = fnv(eh, cur[s.ev[e * ua + p]]);
        esum += splitmix(eh);
    }
    if (tm.any(many)) {
        uint64_t* acc_col = nxt;              // the refinement's other buffer, finished with
        uint64_t* acc_cnt = s.cnt;
        for (uint32_t v = l; v < nl; v += N) { acc_col[v] = 0; acc_cnt[v] = 0; }
        tm.sync();
        for (uint32_t v = l, u = used; v < nl; v += N, u >>= 1) {
            if (!(u & 1u)) continue;
            atomicAdd((unsigned long long*)&acc_col[comp[v]], (unsigned long long)splitmix(cur[v]));
            atomicAdd((unsigned long long*)&acc_cnt[comp[v]], 1ull);
        }
        for (uint32_t e = l; e < nE; e += N)
            atomicAdd((unsigned long long*)&acc_cnt[comp[s.ev[e * ua]]], 1ull << 32);
        tm.sync();
        for (uint32_t v = l, u = used; v < nl; v += N, u >>= 1) {
            if (!(u & 1u) || comp[v] != v) continue;
            csum += splitmix(fnv(fnv(FNV_OFFSET, acc_cnt[v]), acc_col[v]));
        }
        csum = tm.sum64(csum);
        vsum = tm.sum64(vsum);
    } else {
        vsum = tm.sum64(vsum);
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
