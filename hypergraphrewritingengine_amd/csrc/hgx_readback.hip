// hgx_readback.hip -- a result's arrays to the host: states, events, causal pairs, branchial pairs.
//
// A run's states lie in one segment per generation, in state-id order, and its events are its
// states above the roots, so every array is gathered by one kernel over all of the run's segments
// that writes the finished records straight into pinned host memory (the records leave over PCIe as
// they are made; no device staging, so a full HBM budget does not stop a readback). What bounds a
// small result is the count of host round trips -- one launch and one synchronisation per array
// here, where a copy per segment and field took about a hundred copies for four arrays of three
// generations (evolution and readback of 157 states 1.70 -> 0.75 ms; 60 results of a batch 75.5 ->
// 9.1 ms) -- and a large one the bytes over PCIe and into the caller's pages: pieces alternate
// between the two halves of a pinned buffer, the next one filled while the host copies this one
// out (300,405 states, 0.5 M causal and 1.8 M branchial pairs: 14.6 -> 3.7 ms with the evolution).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "hgx_engine.hpp"

namespace hgx {
namespace {

constexpr uint32_t kMaxSegs = HGX_MAX_STEPS + 1;
constexpr uint32_t kRBlock = 256;

// Concatenation of segments of 64-bit words: WL hashes, branchial pairs.
struct GatherSegs {
    const uint64_t* p[kMaxSegs];
    uint64_t first[kMaxSegs + 1];        // words before each segment; [n] = their total
    uint32_t n;
};
struct EventSegs {
    const uint32_t* in[kMaxSegs];        // segment k's events (k > 0), null for the roots
    const uint32_t* rule[kMaxSegs];
    uint32_t first[kMaxSegs + 1];        // first state id of each segment
    uint32_t n;
};
struct CausalSegs {
    const uint32_t* in[kMaxSegs];
    const uint64_t* prod[kMaxSegs];
    const uint64_t* tr[kMaxSegs];
    uint32_t first[kMaxSegs + 1];
    uint32_t n;
};

__global__ __launch_bounds__(kRBlock) void k_read_words(GatherSegs a, uint64_t lo, uint64_t hi, uint64_t* out) {
    const uint64_t i = lo + (uint64_t)blockIdx.x * kRBlock + threadIdx.x;
    if (i >= hi) return;
    uint32_t k = 0;
    while (k + 1 < a.n && i >= a.first[k + 1]) ++k;
    out[i - lo] = a.p[k][i - a.first[k]];
}

// Events [lo, hi) as hgx_event records.
__global__ __launch_bounds__(kRBlock) void k_read_events(EventSegs a, uint32_t lo, uint32_t hi, uint4* out) {
    const uint32_t e = lo + blockIdx.x * kRBlock + threadIdx.x;
    if (e >= hi) return;
    const uint32_t s = e + a.first[1];                   // the event's output state
    uint32_t k = 1;
    while (k + 1 < a.n && s >= a.first[k + 1]) ++k;
    const uint32_t i = s - a.first[k];
    out[e - lo] = make_uint4(a.in[k][i], s, a.rule[k][i], k);
}

// Causal pairs of events [lo, hi), kRBlock events per workgroup: in consumer order, then ascending
// producer generation. A workgroup's pairs are compact in a slot of its own (kRBlock * K pairs, K
// = the run's largest LHS, then as many reduction tags), their number in cnt[workgroup]; the host
// closes the gaps between slots as it copies them out, so the counting pass and scan that one
// compact list would need are not made. Producers are named by generation: the walk up the
// lineage passes one segment per generation, so each step is one load.
__global__ __launch_bounds__(kRBlock) void k_read_causal(CausalSegs a, uint32_t lo, uint32_t hi, uint32_t K,
                                                         uint64_t* pairs, uint8_t* tags, uint32_t* cnt) {
    __shared__ uint32_t wsum[kRBlock / WAVE];
    const uint32_t e = lo + blockIdx.x * kRBlock + threadIdx.x;
    const uint32_t roots = a.first[1];
    uint64_t prod = 0, tr = 0;
    uint32_t x = 0, g = 0;
    if (e < hi) {
        const uint32_t s = e + roots;
        uint32_t k = 1;
        while (k + 1 < a.n && s >= a.first[k + 1]) ++k;
        const uint32_t i = s - a.first[k];
        prod = a.prod[k][i];
        tr = a.tr[k][i];
        x = a.in[k][i];
        g = k - 1;                                       // x is a state of generation g
    }
    const uint32_t n = (uint32_t)__popcll(prod);
    const uint32_t inc = wave_incl_scan_u32(n);
    const uint32_t w = threadIdx.x / WAVE;
    if (lane_id() == WAVE - 1) wsum[w] = inc;
    __syncthreads();
    uint32_t base = inc - n, total = 0;
    for (uint32_t j = 0; j < kRBlock / WAVE; ++j) {
        base += j < w ? wsum[j] : 0u;
        total += wsum[j];
    }
    if (threadIdx.x == 0) cnt[blockIdx.x] = total;
    const uint64_t o = (uint64_t)blockIdx.x * kRBlock * K + base;
    uint32_t at = n;
    while (prod) {
        const uint32_t s = 63u - (uint32_t)__clzll((long long)prod);
        prod &= ~(1ull << s);
        while (g > s) { x = a.in[g][x - a.first[g]]; --g; }   // up to generation s
        --at;
        pairs[o + at] = ((uint64_t)e << 32) | (x - roots);     // (producer, consumer)
        tags[o + at] = (uint8_t)((tr >> s) & 1u);
    }
}

uint32_t blocks_for(uint64_t n) { return (uint32_t)((n + kRBlock - 1) / kRBlock); }

// The calling thread's device for the life of the guard: results may be read by any thread.
struct DeviceGuard {
    int prev = -1;
    explicit DeviceGuard(int dev) {
        HIP_TRY(hipGetDevice(&prev));
        if (prev != dev) HIP_TRY(hipSetDevice(dev));
        else prev = -1;
    }
    ~DeviceGuard() { if (prev >= 0) (void)hipSetDevice(prev); }
};

// Pieces [lo, hi) of n items, at most `per` each: fill(lo, hi, half) queues the kernel that writes
// the piece into a half of the pinned buffer, take(lo, hi, half) copies it out once it is there.
template <class Fill, class Take>
void stream_out(const RunRec& R, uint64_t n, uint64_t per, Fill&& fill, Take&& take) {
    if (!n) return;
    const DeviceGuard dev(R.stage->device());
    StageLease s(*R.stage);
    const uint64_t pieces = (n + per - 1) / per;
    auto hi = [&](uint64_t p) { return std::min(n, (p + 1) * per); };
    try {
        fill(0, hi(0), s.half(0));
        HIP_TRY(hipGetLastError());
        for (uint64_t p = 0; p < pieces; ++p) {
            if (pieces > 1) HIP_TRY(hipEventRecord(s.event(p & 1), R.st));
            if (p + 1 < pieces) {
                fill((p + 1) * per, hi(p + 1), s.half((p + 1) & 1));
                HIP_TRY(hipGetLastError());
            }
            if (pieces > 1) HIP_TRY(hipEventSynchronize(s.event(p & 1)));
            else HIP_TRY(hipStreamSynchronize(R.st));
            take(p * per, hi(p), s.half(p & 1));
        }
    } catch (...) {
        (void)hipStreamSynchronize(R.st);                // no kernel still writes the buffer
        throw;
    }
}

// First state id of each generation's segment; checks that the segments hold the run's states.
template <class S>
void seg_bounds(const RunRec& R, S& a) {
    if (R.segs.size() > kMaxSegs) throw Error{HGX_ERR_DEVICE, "more generations than a result can hold"};
    a.n = (uint32_t)R.segs.size();
    uint64_t o = 0;
    for (uint32_t k = 0; k < a.n; ++k) { a.first[k] = (uint32_t)o; o += R.segs[k].e - R.segs[k].b; }
    a.first[a.n] = (uint32_t)o;
    if (o != R.states) throw Error{HGX_ERR_DEVICE, "a result's generations do not hold its states"};
}

void read_words(const RunRec& R, const GatherSegs& a, uint64_t* out) {
    stream_out(R, a.first[a.n], StageLease::kHalf / 8,
               [&](uint64_t lo, uint64_t hi, uint8_t* h) {
                   hipLaunchKernelGGL(k_read_words, dim3(blocks_for(hi - lo)), dim3(kRBlock), 0, R.st, a, lo, hi,
                                      (uint64_t*)h);
               },
               [&](uint64_t lo, uint64_t hi, const uint8_t* h) { std::memcpy(out + lo, h, 8 * (hi - lo)); });
}

template <class F>
int read_guarded(F&& f) {
    try {
        return f();
    } catch (const Error& e) {
        return e.code;
    } catch (const std::exception&) {
        return HGX_ERR_DEVICE;
    }
}

}  // namespace
}  // namespace hgx

using namespace hgx;

extern "C" int hgx_result_states(const hgx_result* r, uint64_t* hash, uint32_t* step, uint32_t* creator,
                                 uint64_t cap) {
    if (!r || cap < r->run->counts.raw_states) return HGX_ERR_INVALID;
    const RunRec& R = *r->run;
    return read_guarded([&]() -> int {
        EventSegs b{};
        seg_bounds(R, b);
        if (hash) {
            GatherSegs a{};
            for (const Segment& sg : R.segs) {
                if (sg.e == sg.b) continue;
                a.p[a.n] = sg.g->v.hash + sg.b;
                a.first[a.n + 1] = a.first[a.n] + (sg.e - sg.b);
                ++a.n;
            }
            if (a.n) read_words(R, a, hash);
        }
        const uint32_t roots = R.hp->n_roots();
        for (uint32_t k = 0; k < b.n; ++k) {
            if (step) std::fill(step + b.first[k], step + b.first[k + 1], k);
            if (creator)
                for (uint32_t s = b.first[k]; s < b.first[k + 1]; ++s) creator[s] = k ? s - roots : 0xFFFFFFFFu;
        }
        return HGX_OK;
    });
}

extern "C" int hgx_result_events(const hgx_result* r, hgx_event* out, uint64_t cap) {
    static_assert(sizeof(hgx_event) == sizeof(uint4), "one event is one 16-byte record");
    if (!r || (!out && r->run->events) || cap < r->run->events) return HGX_ERR_INVALID;
    const RunRec& R = *r->run;
    return read_guarded([&]() -> int {
        if (!R.events) return HGX_OK;
        EventSegs a{};
        seg_bounds(R, a);
        for (uint32_t k = 1; k < a.n; ++k) {
            a.in[k] = R.segs[k].g->ev.in_state + R.segs[k].b;
            a.rule[k] = R.segs[k].g->ev.rule + R.segs[k].b;
        }
        stream_out(R, R.events, StageLease::kHalf / sizeof(hgx_event),
                   [&](uint64_t lo, uint64_t hi, uint8_t* h) {
                       hipLaunchKernelGGL(k_read_events, dim3(blocks_for(hi - lo)), dim3(kRBlock), 0, R.st, a,
                                          (uint32_t)lo, (uint32_t)hi, (uint4*)h);
                   },
                   [&](uint64_t lo, uint64_t hi, const uint8_t* h) {
                       std::memcpy(out + lo, h, sizeof(hgx_event) * (hi - lo));
                   });
        return HGX_OK;
    });
}

extern "C" int hgx_result_causal(const hgx_result* r, hgx_pair* pairs, uint8_t* in_tr, uint64_t cap) {
    if (!r) return HGX_ERR_INVALID;
    const RunRec& R = *r->run;
    if (!(R.hp->flags & HGX_REC_CAUSAL) || cap < R.counts.causal_pairs) return HGX_ERR_INVALID;
    return read_guarded([&]() -> int {
        if (!R.events) return HGX_OK;
        CausalSegs a{};
        seg_bounds(R, a);
        for (uint32_t k = 1; k < a.n; ++k) {
            const Segment& sg = R.segs[k];
            a.in[k] = sg.g->ev.in_state + sg.b;
            a.prod[k] = sg.g->ev.prod + sg.b;
            a.tr[k] = sg.g->ev.tr + sg.b;
        }
        const uint32_t K = R.hp->max_lhs;
        const uint64_t slot = (uint64_t)kRBlock * K;               // pairs a workgroup's slot holds
        const uint64_t nb = std::min<uint64_t>(StageLease::kHalf / (9 * slot + 4), blocks_for(R.events));
        uint64_t o = 0;
        bool over = false;
        stream_out(R, R.events, nb * kRBlock,
                   [&](uint64_t lo, uint64_t hi, uint8_t* h) {
                       hipLaunchKernelGGL(k_read_causal, dim3(blocks_for(hi - lo)), dim3(kRBlock), 0, R.st, a,
                                          (uint32_t)lo, (uint32_t)hi, K, (uint64_t*)h, h + 8 * slot * nb + 4 * nb,
                                          (uint32_t*)(h + 8 * slot * nb));
                   },
                   [&](uint64_t lo, uint64_t hi, const uint8_t* h) {
                       const uint32_t* cnt = (const uint32_t*)(h + 8 * slot * nb);
                       const uint8_t* tags = h + 8 * slot * nb + 4 * nb;
                       for (uint64_t b = 0; b < blocks_for(hi - lo); ++b) {
                           const uint64_t c = cnt[b];
                           if (over || c > slot || o + c > cap) { over = true; return; }
                           if (pairs) std::memcpy(pairs + o, h + 8 * slot * b, 8 * c);
                           if (in_tr) std::memcpy(in_tr + o, tags + slot * b, c);
                           o += c;
                       }
                   });
        return over ? HGX_ERR_INVALID : HGX_OK;
    });
}

extern "C" int hgx_result_branchial(const hgx_result* r, hgx_pair* pairs, uint64_t cap) {
    if (!r) return HGX_ERR_INVALID;
    const RunRec& R = *r->run;
    if (!(R.hp->flags & HGX_REC_BRANCHIAL) || !(R.hp->flags & HGX_REC_RELATIONS)) return HGX_ERR_INVALID;
    if (cap < R.counts.branchial_pairs) return HGX_ERR_INVALID;
    return read_guarded([&]() -> int {
        GatherSegs a{};
        for (const Segment& sg : R.segs) {
            if (sg.br_e <= sg.br_b || !sg.g->br_pairs) continue;
            if (a.n == kMaxSegs) return HGX_ERR_DEVICE;
            a.p[a.n] = (const uint64_t*)sg.g->br_pairs + sg.br_b;
            a.first[a.n + 1] = a.first[a.n] + (sg.br_e - sg.br_b);
            ++a.n;
        }
        if (!a.n) return HGX_OK;
        if (a.first[a.n] > cap) return HGX_ERR_INVALID;
        read_words(R, a, (uint64_t*)pairs);
        return HGX_OK;
    });
}
