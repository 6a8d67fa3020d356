// hgx_bigjoin.hpp -- the large-state join's host interface, shared by hgx_match_count and the
// allocation-free entry point: the state and rule as the kernels see them, the device memory
// the join draws from, and the join itself.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "hgx_device.hpp"
#include "hgx_runtime.hpp"

namespace hgx {

// Lists of at most kIndexShort entries are ordered by a thread per entry that counts, of at most
// kIndexWave by a wave per list that counts in LDS (cost n^2 / 64), longer ones by a bit set of the
// edges in LDS (cost of all edges / 32, whatever n). States of at most kIndexPlaceEdges edges have their lists placed and ordered rather
// than sorted: the bit set of 2^20 edges is 128 KB, and the two ways meet there -- wedges of random
// graphs (edges / 10 vertices), whole join: 98 against 128 us at 20,000 edges, 237 / 339 at 500,000,
// 350 / 462 at 1 million, 589 / 600 at 2 million and 1,017 / 966 at 4 million (placed / sorted).
constexpr uint32_t kIndexShort = 32;
constexpr uint32_t kIndexWave = 256;
constexpr uint32_t kIndexPlaceEdges = 1u << 20;

struct BJView {
    DRule R;
    const uint32_t* ev;     // [m * A]
    const uint8_t* ar;      // [m]
    uint32_t m, A;
    // The CSR over the U positions the join pivots on: list vertex * U + u holds, ascending, the
    // edges with the vertex at position upos[u] and an arity in the bit set uar[u].
    uint32_t U;
    uint8_t upos[16];
    uint8_t dpos[16];       // per depth: which of them it pivots on
    uint32_t uar[16];
    const uint32_t* off;    // [lists + 1]
    const uint32_t* idx;    // [entries]
    // What a depth compares of a candidate: the slots, and (bit d of chk_ar) the arity
    uint32_t chk[16];
    uint32_t chk_ar;
    // Closing edges: a depth whose pattern edge has every vertex bound by earlier depths takes its
    // candidates from the edges with exactly that vertex tuple, by an open-addressing table of
    // 32-bit tags (0 empty; a tag shared by two tuples only widens a list's verification). The
    // edges of the tuple at place h are tidx[toff[h] - toff[0] ..], ascending. Bit d of `full`
    // marks such a depth (0: no table), tar is the bit set of their arities.
    uint32_t full, tar, tmask;
    const uint32_t* tslot;  // [tmask + 1]
    const uint32_t* toff;   // [tmask + 2]
    const uint32_t* tidx;
};

// The index while it is built.
struct BJIndex {
    uint32_t nkeys;         // lists of the CSR
    uint64_t tcnt0, scnt0;  // where the tuples' and the seeds' counts begin in cnt
    uint32_t* cnt;          // counts: lists + 1, (tuple table + 1,) workgroups' seeds + 1
    uint32_t* rank;         // [m * U] an entry's place in its list; its list (sorted instead)
    uint32_t* tplace;       // [m] a tuple's place in the table
    uint32_t* trank;        // [m] the edge's place in the tuple's list
    uint32_t* tslot;
    uint32_t* un;           // [m * U + m] list entries in arrival order, tuples' from tbase
    uint32_t* idx;          //   and ascending
    uint32_t tbase;
    uint32_t* longq;        // lists of more than kIndexWave entries (tuple h: nkeys + 1 + h)
    uint64_t* smask;        // one bit per edge: a seed
    uint32_t* seeds;
    uint32_t* scal;         // seeds, longest list, long lists, longest tuple list
};

// Device memory of one join: an Arena, or a fixed region (the allocation-free entry point)
// handed out by a bump pointer that each depth rewinds when its subtree is done.
struct BJMem {
    Arena* arena = nullptr;
    uint8_t* base = nullptr;
    size_t cap = 0, used = 0;
    void* get(size_t bytes) {
        if (arena) return arena->alloc(bytes ? bytes : 1);
        const size_t o = (used + 255) & ~(size_t)255;
        if (o + bytes > cap)
            throw Error{HGX_ERR_CAPACITY, "the join needs more than the " + std::to_string(cap >> 20) +
                                              " MiB of its fixed scratch"};
        used = o + bytes;
        return base + o;
    }
    size_t mark() const { return used; }
    void rewind(size_t m) { if (!arena) used = m; }
    // bytes a depth's tiles may take before it splits its partials in two
    size_t left() const { return arena ? ((size_t)1 << 30) : (cap > used + (1u << 20) ? cap - used - (1u << 20) : 0); }
    // bytes a next frontier may take before the depth splits its partials in two
    size_t room() const { return arena ? ((size_t)1 << 30) : (cap > used + (8u << 20) ? cap - used - (8u << 20) : 0); }
};

struct BJRun {
    hipStream_t st;
    BJView v;
    BJMem* mem;
    uint32_t grid;            // workgroup cap of the item passes
    uint32_t* out;            // matches (device), or null to count
    uint64_t cap = 0;
    uint64_t found = 0;
    uint32_t maxlist = 0;     // the longest candidate list of the index
    uint64_t* acc = nullptr;  // device: matches found (by turns, two), join bytes
    uint32_t turn = 0;        // which of the two holds the matches found so far
    uint64_t index_bytes = 0; // algorithmic bytes of the index build
    uint64_t alg_bytes = 0;   // of the join: adjacency reads of every item, frontiers, matches
};

// All matches of J.v.R in the state J.v (on the device, vertex ids below nv): J.found counts them
// and, with J.out, the first J.cap are written (n_lhs edge ids each, pattern order), in the order
// of a serial depth-first join over ascending candidates. With `timed`, the index and join times.
void bj_match(BJRun& J, uint32_t nv, float* ms_index, float* ms_join, bool timed);

}  // namespace hgx
