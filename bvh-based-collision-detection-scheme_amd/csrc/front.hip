// BVTT-front kernels for gfx950: self-CD traversal, front generate / UPDATE / KEEP / REORDER,
// front ordering, quality snapshot and check, narrow phase.
//
// Reference behaviour (Source/Project/Mine/ of littlemine/BVH-based-Collision-Detection-Scheme):
//   pure traversal       collision/bvtt_front/BvhCDKernels.cu:17-49
//   generate             collision/bvtt_front/BvttFrontGenerateKernels.cu:51-90
//   UPDATE prune/sprout  collision/bvtt_front/BvttFrontPruneSproutKernels.cu:12-93
//   KEEP                 collision/bvtt_front/BvttFrontKeepKernels.cu:11-58
//   REORDER (balance)    collision/bvtt_front/BvttFrontReorderKernels.cu:27-63, BvttFrontLooseIntra.cu:285-312
//   ordering             collision/bvtt_front/BvttFrontReorderKernels.cu:12-24, collision/auxiliary/FlOrderLog.cu:7-12
//   snapshot / quality   collision/bvtt_front/BvttFrontGenerateKernels.cu:26-49
//   restructure marks    collision/lbvh/LBvhFixedDeformable.cu:216-241, LBvhRestructureKernels.cu:9-35
//   narrow phase         collision/narrow_phase/narrow_phase.cu:8-24 (17-axis SAT written here from the
//                        separating-axis theorem; canonical argument order: lower triangle id first)
//
// Layout and scheduling on gfx950:
//  * Every node visit is one 32-byte record (two 16-byte loads): box + rangex/escape
//    (internal) or box + parent/escape (leaf).
//  * Fronts are SoA (node id, query leaf) so that ordering is a radix sort on the node id
//    with the query as payload: no per-node counters, no atomics, and the bucket starts
//    (the reference's FlOrderLog offsets) come from binary searches on the sorted ids.
//  * Work is distributed grid-stride (consecutive entries per wave64, coalesced SoA loads).
//  * Appends go through a per-wave LDS staging buffer: lanes take slots with a ballot
//    prefix, and one global atomic reserves space for a whole buffer when it is flushed.
//    Capacity is checked before every global write (overflow bit instead of a write).
#include <cstdio>
#include <string>
#include <vector>

#include "bvhcd_internal.hpp"
#include "kernels.hpp"

namespace bvhcd {

constexpr int kWaves = kBlock / 64;
constexpr uint32_t kStage = 256;   // staged entries per wave, single-list kernels
// Per list where the incremental restructure stages three lists (GENERATE and UPDATE: kWalkStage,
// kSproutStage, which leave them more resident waves). A flush is one atomic on a segment counter.
constexpr uint32_t kStage3 = 256;

__device__ inline uint64_t lanes_below() { return (1ull << lane_id()) - 1ull; }

// Per-wave LDS words shared between lanes are reached through pointers typed as LDS: their
// accesses are then ds_read / ds_write. Through generic pointers they would be flat accesses,
// which also count against the vector-memory counter, so waiting for one of them would wait for
// every global load in flight as well.
#define BVHCD_LDS __attribute__((address_space(3)))
typedef volatile BVHCD_LDS int2 lds_int2;
typedef volatile BVHCD_LDS uint32_t lds_u32;

// ---------------------------------------------------------------- output sinks
// Front output (SoA node / query), segmented like the pair lists: kPairSegs counters
// kCntStride words apart, segment g at [g * seg_cap, g * seg_cap + count). The producing kernel
// appends segment-wise; front_finish then gathers the segments into the current buffer.
struct FrontSink {
    uint32_t* cnt;
    uint32_t* node;
    int32_t* query;
    int64_t seg_cap;
    uint32_t ovf_bit;
    // wave-ordered production (null: off): chunk records and per-wave totals
    uint4* chunks = nullptr;
    uint32_t* wave_tot = nullptr;
    uint32_t chunk_seg_cap = 0;
};
struct PairSink {  // int2 list with one counter
    uint32_t* count;
    int2* out;
    uint32_t cap;
    uint32_t ovf_bit;
    __device__ void write(uint32_t o, int2 v) const { out[o] = v; }
};
struct SegPairSink {  // segmented pair list: kPairSegs counters kCntStride words apart
    uint32_t* cnt;
    int2* base;
    int64_t seg_cap;
    uint32_t ovf_bit;
};

// The staging word pair of a wave and list: sfill[0] = staged entries, sfill[1] = rotor that
// picks the segment of the next flush of a segmented list.
template <class Sink>
__device__ void stage_flush(const Sink& sk, uint32_t* ovf, lds_int2* sbuf, lds_u32*, uint32_t f,
                            uint64_t active) {
    const int lane = lane_id();
    const int leader = __ffsll((long long)active) - 1;
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(sk.count, f);
    base = __shfl(base, leader);
    const uint32_t rank = (uint32_t)__popcll(active & lanes_below());
    const uint32_t nact = (uint32_t)__popcll(active);
    bool over = false;
    for (uint32_t i = rank; i < f; i += nact) {
        const uint32_t o = base + i;
        const int2 v = make_int2(sbuf[i].x, sbuf[i].y);
        if (o < sk.cap) sk.write(o, v);
        else over = true;
    }
    if (over) atomicOr(ovf, sk.ovf_bit);
}
// Segmented lists: successive flushes of a wave rotate over the segments, so the appends
// spread over kPairSegs counters and every segment fills evenly whichever workgroups produce
// the entries. The rotor start spreads the waves of one XCD (workgroups b with equal b % 8,
// which a per-XCD split makes neighbours in the data) over all segments too.
template <int W = kWaves>
__device__ inline uint32_t rotor_start() {
    const uint32_t b = blockIdx.x, w = threadIdx.x >> 6;
    return (b / kXcds) * W + w + (b % kXcds) * kXcds;
}
// One flush takes its slots in the rotor's next segment; what does not fit there (the segment
// filled up) is given back to the counter and tries the following segments, so a list overflows
// only once all its segments are full, and every segment counter ends at the entries its segment
// holds. Entries no segment took are counted in word 2 of the list's counter block (the list's
// requested length is the segment counts plus that). Wave-ordered production (chunk records):
// one 64-bit add on the segment counter takes both the slots (low word) and the chunk's seq in
// the segment (high word), and every seq gets its record, which keeps only what its segment
// holds; a record that does not fit drops its chunk (overflow bit) so that the gathered front
// stays dense. sfill[2] counts the wave's recorded entries.
struct SegTake {
    uint32_t g, base, fit;
};
__device__ inline SegTake seg_take(uint32_t* cnt, int64_t seg_cap, const FrontSink* chunked, uint32_t* ovf,
                                   lds_u32* sfill, uint32_t want, uint64_t active) {
    const int leader = __ffsll((long long)active) - 1;
    uint32_t g = 0, base = 0, fit = 0;
    if (lane_id() == leader) {
        g = sfill[1] % kPairSegs;
        sfill[1] = sfill[1] + 1;
        if (chunked) {
            const unsigned long long old =
                atomicAdd(reinterpret_cast<unsigned long long*>(cnt + g * kCntStride), (1ull << 32) | want);
            base = (uint32_t)old;
            const uint32_t seq = (uint32_t)(old >> 32);
            fit = base < (uint64_t)seg_cap ? (uint32_t)min<int64_t>(want, seg_cap - base) : 0u;
            if (seq < chunked->chunk_seg_cap) {
                const uint32_t wave = blockIdx.x * kWaves + (threadIdx.x >> 6);
                chunked->chunks[(int64_t)g * chunked->chunk_seg_cap + seq] = make_uint4(base, wave, sfill[2], fit);
            } else {
                fit = 0u;
                atomicOr(ovf, chunked->ovf_bit);
            }
            sfill[2] = sfill[2] + fit;
        } else {
            base = atomicAdd(cnt + g * kCntStride, want);
            fit = base < (uint64_t)seg_cap ? (uint32_t)min<int64_t>(want, seg_cap - base) : 0u;
        }
        if (fit < want) atomicSub(cnt + g * kCntStride, want - fit);  // slots past the segment's end
    }
    return SegTake{(uint32_t)__shfl((int)g, leader), (uint32_t)__shfl((int)base, leader),
                   (uint32_t)__shfl((int)fit, leader)};
}
__device__ inline void stage_flush(const SegPairSink& sk, uint32_t* ovf, lds_int2* sbuf, lds_u32* sfill,
                                   uint32_t f, uint64_t active) {
    const uint32_t rank = (uint32_t)__popcll(active & lanes_below());
    const uint32_t nact = (uint32_t)__popcll(active);
    uint32_t done = 0;
    for (int a = 0; a < kPairSegs && done < f; ++a) {
        const SegTake t = seg_take(sk.cnt, sk.seg_cap, nullptr, ovf, sfill, f - done, active);
        int2* out = sk.base + (int64_t)t.g * sk.seg_cap + t.base;
        for (uint32_t i = rank; i < t.fit; i += nact) out[i] = make_int2(sbuf[done + i].x, sbuf[done + i].y);
        done += t.fit;
    }
    if (done < f && lane_id() == __ffsll((long long)active) - 1) {
        atomicOr(ovf, sk.ovf_bit);
        atomicAdd(sk.cnt + kDroppedWord, f - done);
    }
}
__device__ inline void stage_flush(const FrontSink& sk, uint32_t* ovf, lds_int2* sbuf, lds_u32* sfill,
                                   uint32_t f, uint64_t active) {
    const uint32_t rank = (uint32_t)__popcll(active & lanes_below());
    const uint32_t nact = (uint32_t)__popcll(active);
    uint32_t done = 0;
    for (int a = 0; a < kPairSegs && done < f; ++a) {
        const SegTake t = seg_take(sk.cnt, sk.seg_cap, sk.chunks ? &sk : nullptr, ovf, sfill, f - done, active);
        const int64_t o = (int64_t)t.g * sk.seg_cap + t.base;
        for (uint32_t i = rank; i < t.fit; i += nact) {
            sk.node[o + i] = (uint32_t)sbuf[done + i].y;
            sk.query[o + i] = sbuf[done + i].x;
        }
        done += t.fit;
    }
    if (done < f && lane_id() == __ffsll((long long)active) - 1) {
        atomicOr(ovf, sk.ovf_bit);
        atomicAdd(sk.cnt + kDroppedWord, f - done);
    }
}

// Called by the currently active lanes of a wave; `pred` selects the lanes that emit `v`.
template <class Sink>
__device__ inline void stage_push(const Sink& sk, uint32_t* ovf, lds_int2* sbuf, lds_u32* sfill,
                                  uint32_t cap, bool pred, int2 v) {
    const uint64_t active = __ballot(1);
    const uint64_t m = __ballot(pred);
    if (m == 0) return;
    uint32_t f = *sfill;
    const uint32_t cnt = (uint32_t)__popcll(m);
    if (f + cnt > cap) {
        stage_flush(sk, ovf, sbuf, sfill, f, active);
        f = 0;
    }
    if (pred) {
        const uint32_t slot = f + (uint32_t)__popcll(m & lanes_below());
        sbuf[slot].x = v.x;
        sbuf[slot].y = v.y;
    }
    if (lane_id() == __ffsll((long long)active) - 1) *sfill = f + cnt;
}

template <class Sink>
__device__ inline void stage_final(const Sink& sk, uint32_t* ovf, lds_int2* sbuf, lds_u32* sfill) {
    const uint32_t f = *sfill;
    if (f) stage_flush(sk, ovf, sbuf, sfill, f, __ballot(1));
    if (lane_id() == 0) *sfill = 0;
}

// Per-block staging storage for up to three lists; fill[list][wave] = {staged, rotor, recorded
// entries of a wave-ordered production}.
template <uint32_t CAP>
struct StagesT {
    int2 buf[3][kWaves][CAP];
    uint32_t fill[3][kWaves][3];
};
using Stages = StagesT<kStage3>;
template <uint32_t CAP>
__device__ inline void stages_init(StagesT<CAP>& st) {
    const int w = threadIdx.x >> 6;
    if (lane_id() < 3) {
        st.fill[lane_id()][w][0] = 0;
        st.fill[lane_id()][w][1] = rotor_start();
        st.fill[lane_id()][w][2] = 0;
    }
}
// End of a wave's production: its recorded total, every wave of the launch writing its own.
__device__ inline void wave_total(const FrontSink& sk, lds_u32* sfill) {
    if (sk.chunks && lane_id() == __ffsll((long long)__ballot(1)) - 1)
        sk.wave_tot[blockIdx.x * kWaves + (threadIdx.x >> 6)] = sfill[2];
}

// Output context of a traversal thread.
struct Out {
    FrontSink fi, fe;
    SegPairSink bp;
    uint32_t* ovf;
    lds_int2* sb[3];
    lds_u32* sf[3];
    uint32_t scap;  // staging entries per wave and list
    const int32_t* lfaces;
    int skip_adj;   // drop pairs of triangles sharing a vertex
    // Broad-phase pairs are kept as leaf (sorted-slot) ids, query first (qi < j): the narrow
    // phase then reads leaf-ordered faces with locality, and maps to triangle ids itself.
    __device__ void pair_push(bool pred, int2 v) const { stage_push(bp, ovf, sb[2], sf[2], scap, pred, v); }
    __device__ void pair_final() const { stage_final(bp, ovf, sb[2], sf[2]); }
    __device__ void pair(int32_t qi, int32_t j) const {
        if (skip_adj && faces_share_vertex(lfaces, qi, j)) return;
        pair_push(true, make_int2(qi, j));
    }
    __device__ void int_entry(int32_t qi, int32_t node) const {
        stage_push(fi, ovf, sb[0], sf[0], scap, true, make_int2(qi, node));
    }
    __device__ void ext_entry(int32_t qi, int32_t leaf) const {
        stage_push(fe, ovf, sb[1], sf[1], scap, true, make_int2(qi, leaf));
    }
    __device__ void final_flush() const {
        stage_final(fi, ovf, sb[0], sf[0]);
        stage_final(fe, ovf, sb[1], sf[1]);
        pair_final();
        wave_total(fi, sf[0]);
        wave_total(fe, sf[1]);
    }
};

// Segmented pair list of kind 0 (broad phase) or 1 (narrow phase).
__device__ inline SegPairSink pair_segments(const DevState& d, int kind, uint32_t ovf_bit) {
    return SegPairSink{d.pcnt + kind * kPairSegs * kCntStride, kind ? d.np : d.bp, d.pair_seg_cap, ovf_bit};
}

// Pair-only kernels (KEEP, batched traversal) stage one list: a third of the LDS, so 8 waves
// per SIMD instead of 6 hide more of the dependent node loads. W = waves per workgroup.
template <int W = kWaves>
struct StagesBPT {
    int2 buf[W][kStage];
    uint32_t fill[W][2];
};
using StagesBP = StagesBPT<>;
template <int W>
__device__ inline void stages_init(StagesBPT<W>& st) {
    const int w = threadIdx.x >> 6;
    if (lane_id() == 0) {
        st.fill[w][0] = 0;
        st.fill[w][1] = rotor_start<W>();
    }
}
template <int W>
__device__ inline Out make_out(StagesBPT<W>& st, const DevState& d) {
    Out o;
    o.fi = FrontSink{nullptr, nullptr, nullptr, 0u, 0u};
    o.fe = o.fi;
    o.bp = pair_segments(d, 0, 4u);
    o.ovf = &d.ctr[C_OVF];
    const int w = threadIdx.x >> 6;
    o.sb[0] = o.sb[1] = nullptr;
    o.sf[0] = o.sf[1] = nullptr;
    o.sb[2] = (lds_int2*)st.buf[w];
    o.sf[2] = (lds_u32*)st.fill[w];
    o.scap = kStage;
    o.lfaces = d.lfaces;
    o.skip_adj = d.skip_adj;
    return o;
}

template <uint32_t CAP>
__device__ inline Out make_out(StagesT<CAP>& st, const FrontSink& fi, const FrontSink& fe, const DevState& d) {
    Out o;
    o.fi = fi;
    o.fe = fe;
    o.bp = pair_segments(d, 0, 4u);
    o.ovf = &d.ctr[C_OVF];
    const int w = threadIdx.x >> 6;
    for (int k = 0; k < 3; ++k) {
        o.sb[k] = (lds_int2*)st.buf[k][w];
        o.sf[k] = (lds_u32*)st.fill[k][w];
    }
    o.scap = CAP;
    o.lfaces = d.lfaces;
    o.skip_adj = d.skip_adj;
    return o;
}

constexpr uint32_t kOpenSample = 16, kOpenMost = 20;
__device__ inline bool node_overlap(const DevState& d, int32_t nd, const Box& q) {
    const float4 lo = d.inode[nd].lo, hi = d.inode[nd].hi;
    return box_overlap(q, lo, hi);
}

// Stackless DFS from encoded node `st` until `stop` (lca-escape encoding). With FRONT, the
// non-overlapping internal nodes and all reached leaves are appended to the next front.
template <bool FRONT>
__device__ uint32_t stackless(const DevState& d, const Out& out, int32_t qi, const Box& q, int32_t st, int32_t stop) {
    uint32_t visits = 0;
    // A correct traversal visits every node at most once; the bound only guards against a
    // corrupted tree (flag 16 reported as a device error instead of a hang).
    const int64_t limit = 2 * d.maxT + 16;
    int64_t steps = 0;
    while (st != stop) {
        if (++steps > limit) {
            atomicOr(&d.ctr[C_OVF], 16u);
            break;
        }
        int32_t j;
        if (!(st & 1)) {
            int32_t nd = st >> 1;
            float4 lo = d.inode[nd].lo, hi = d.inode[nd].hi;
            j = f2i(lo.w);                    // leftmost leaf of the whole left spine
            const int32_t t = d.leaf_par[j];  // bottom of the spine
            bool reached = false;
            for (;;) {
                ++visits;
                if (!box_overlap(q, lo, hi)) break;
                if (nd == t) {
                    reached = true;
                    break;
                }
                ++nd;
                lo = d.inode[nd].lo;
                hi = d.inode[nd].hi;
            }
            if (!reached) {
                if (FRONT) out.int_entry(qi, nd);
                st = f2i(hi.w);
                continue;
            }
        } else {
            j = st >> 1;
        }
        const float4 llo = d.leaf[j].lo, lhi = d.leaf[j].hi;
        ++visits;
        if (box_overlap(q, llo, lhi)) out.pair(qi, j);
        if (FRONT) out.ext_entry(qi, j);
        st = f2i(lhi.w);
    }
    return visits;
}

// A wave's node tests, added to one of the kPairSegs visit words (beside the broad-phase segment
// counters) which pair_totals sums.
__device__ inline void add_visits(const DevState& d, uint32_t v) {
    uint64_t x = v;
    for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off);
    const uint32_t b = blockIdx.x, slot = (b / kXcds * (blockDim.x >> 6) + (threadIdx.x >> 6) + b % kXcds * kXcds) % kPairSegs;
    if (lane_id() == 0 && x) atomicAdd(visit_word(d, slot), (unsigned long long)x);
}

// ---------------------------------------------------------------- host-side front views
struct FrontIn {
    const uint32_t* node[2];
    const int32_t* query[2];
    const uint32_t* size[2];
    uint32_t cap[2];
};

// Segmented output into the spare buffer of `kind` (its counters cleared by front_begin).
static FrontSink next_sink(DevState& d, int kind) {
    const int nb = d.fcur[kind] ^ 1;
    return FrontSink{d.fcnt + kind * kPairSegs * kCntStride, d.fnode[kind][nb], d.fquery[kind][nb],
                     d.front_cap[kind] / kPairSegs, kind ? 2u : 1u};
}
static void front_begin(DevState& d, hipStream_t s) { fill_u32(d.fcnt, 2 * kPairSegs * kCntStride, 0u, s); }

// Gathers the segments of the spare buffer into the current buffer of `kind`, after its first
// `base` entries (base read from *base_word before any block writes, 0 when null); the current
// buffer's size becomes base + total, clamped to the capacity (overflow bit otherwise).
__global__ void __launch_bounds__(kBlock) k_front_compact(DevState d, int kind, const uint32_t* __restrict__ src_node,
                                                          const int32_t* __restrict__ src_query,
                                                          uint32_t* __restrict__ dst_node,
                                                          int32_t* __restrict__ dst_query, const uint32_t* base_word,
                                                          uint32_t* dst_size) {
    __shared__ uint32_t pre[kPairSegs + 1];
    const int64_t seg_cap = d.front_cap[kind] / kPairSegs;
    const uint32_t total = seg_prefix(d.fcnt + kind * kPairSegs * kCntStride, (uint32_t)seg_cap, pre);
    const uint32_t base = base_word ? *base_word : 0u;
    const uint32_t cap = (uint32_t)min(d.front_cap[kind], (int64_t)0xFFFFFFFF);
    const uint32_t room = base < cap ? cap - base : 0u;
    const uint32_t m = min(total, room);
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < m; k += gridDim.x * blockDim.x) {
        const int64_t src = seg_slot(pre, k, seg_cap);
        dst_node[base + k] = src_node[src];
        dst_query[base + k] = src_query[src];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *dst_size = base + m;
        if (m < total) atomicOr(&d.ctr[C_OVF], kind ? 2u : 1u);
        // capacity that would have held every requested entry (an over-estimate after an
        // overflow: slots a full segment refused were asked for again elsewhere)
        const uint32_t* cnt = d.fcnt + kind * kPairSegs * kCntStride;
        uint32_t sum = cnt[kDroppedWord];
        for (int g = 0; g < kPairSegs; ++g) sum += cnt[g * kCntStride];
        d.ctr[kind ? C_FREQ_E : C_FREQ_I] = base + sum;
    }
}
// append: keep the current buffer's entries and add the new ones after them.
static void front_finish(DevState& d, int kind, bool append, hipStream_t s) {
    const int c = d.fcur[kind], nb = c ^ 1;
    uint32_t* size = d.fsize + 2 * kind + c;
    uint32_t* base_word = nullptr;
    if (append) {  // the base is snapshotted: block 0 rewrites *size while others still read
        base_word = d.ctr + (kind ? C_KEPT_E : C_KEPT_I);
        hipMemcpyAsync(base_word, size, sizeof(uint32_t), hipMemcpyDeviceToDevice, s);
    }
    hipLaunchKernelGGL(k_front_compact, dim3(2048), dim3(kBlock), 0, s, d, kind, d.fnode[kind][nb],
                       d.fquery[kind][nb], d.fnode[kind][c], d.fquery[kind][c], base_word, size);
}
// Wave-ordered production: the sinks record chunks, `waves` producing waves (the launch's).
static bool wave_ordered_ok(const DevState& d, int64_t waves) {
    return d.fchunk[0] && d.fchunk[1] && waves <= d.wave_cap;
}
static void record_chunks(DevState& d, FrontSink& sk, int kind) {
    sk.chunks = d.fchunk[kind];
    sk.wave_tot = d.wave_tot[kind];
    sk.chunk_seg_cap = (uint32_t)d.chunk_seg_cap;
}

// Orders a wave-ordered production of `kind` into its current buffer. The chunk records are
// first copied into lists by producing wave (k_chunk_count, a scan of the counts, k_chunk_list,
// each with its offset in the segments, so the next kernel finds the entries in one load); then one
// workgroup per producing wave w loads its chunks straight from the segments (chunk c holds the
// wave's entries c.z .. c.z + count - 1) and orders the run by query with a counting sort in LDS
// on q - per w (the wave's queries are per w .. per w + per - 1), writing it once at the scan of the
// wave totals. The order within a query is not kept (fronts are multisets). A run longer than
// kWaveRunLds entries, or one past the capacity, is written in production order (clamped to the
// capacity; the overflow bit is set and the front stays a dense prefix). The size becomes the
// wave totals' sum, clamped to the capacity.
__global__ void __launch_bounds__(kBlock) k_chunk_count(DevState d, int kind) {
    __shared__ uint32_t pre[kPairSegs + 1];
    const uint32_t nchunks =
        seg_prefix(d.fcnt + kind * kPairSegs * kCntStride + 1, (uint32_t)d.chunk_seg_cap, pre);  // chunk seqs
    for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < nchunks; c += gridDim.x * blockDim.x)
        atomicAdd(&d.wave_nch[d.fchunk[kind][seg_slot(pre, c, d.chunk_seg_cap)].y], 1u);
}
__global__ void __launch_bounds__(kBlock) k_chunk_list(DevState d, int kind) {
    __shared__ uint32_t pre[kPairSegs + 1];
    const uint32_t nchunks =
        seg_prefix(d.fcnt + kind * kPairSegs * kCntStride + 1, (uint32_t)d.chunk_seg_cap, pre);
    const int64_t seg_cap = d.front_cap[kind] / kPairSegs;
    for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < nchunks; c += gridDim.x * blockDim.x) {
        const int64_t slot = seg_slot(pre, c, d.chunk_seg_cap);
        const uint4 ch = d.fchunk[kind][slot];
        const uint64_t src = (uint64_t)((slot / d.chunk_seg_cap) * seg_cap + ch.x);  // in the segments
        d.clist[d.wave_cbase[ch.y] + atomicSub(&d.wave_nch[ch.y], 1u) - 1u] =
            make_uint4((uint32_t)src, (uint32_t)(src >> 32), ch.z, ch.w);
    }
}
constexpr uint32_t kWaveRunLds = 4096;
constexpr int kOrderBlock = 512;  // LDS allows 4 workgroups per CU: 8 waves each fill it
__global__ void __launch_bounds__(kOrderBlock) k_wave_order(DevState d, int kind, uint32_t waves, uint32_t per,
                                                       const uint32_t* __restrict__ src_node,
                                                       const int32_t* __restrict__ src_query,
                                                       uint32_t* __restrict__ dst_node,
                                                       int32_t* __restrict__ dst_query, uint32_t* dst_size) {
    __shared__ uint32_t lnode[kWaveRunLds];
    __shared__ uint32_t lkey[kWaveRunLds];  // (q - per w) << 16 | rank among the run's entries of q
    __shared__ uint32_t cnt[64];
    const uint32_t w = blockIdx.x;
    const uint32_t cap = (uint32_t)min(d.front_cap[kind], (int64_t)0xFFFFFFFF);
    const uint32_t b0 = d.wave_base[w], m = d.wave_tot[kind][w];
    const uint32_t c0 = d.wave_cbase[w], c1 = w + 1 < waves ? d.wave_cbase[w + 1] : d.ctr[C_WAVE_CHUNKS];
    const int lane = lane_id(), wid = threadIdx.x >> 6;
    if (w == 0 && threadIdx.x == 0) {
        const uint32_t total = d.ctr[C_WAVE_TOTAL];
        *dst_size = min(total, cap);
        if (total > cap) atomicOr(&d.ctr[C_OVF], kind ? 2u : 1u);
        const uint32_t* fc = d.fcnt + kind * kPairSegs * kCntStride;
        uint32_t sum = fc[kDroppedWord];
        for (int g = 0; g < kPairSegs; ++g) sum += fc[g * kCntStride];
        d.ctr[kind ? C_FREQ_E : C_FREQ_I] = sum;
    }
    if (m > kWaveRunLds || (uint64_t)b0 + m > cap) {
        for (uint32_t c = c0 + wid; c < c1; c += kOrderBlock / 64) {
            const uint4 ch = d.clist[c];
            const int64_t src = (int64_t)((uint64_t)ch.x | (uint64_t)ch.y << 32);
            for (uint32_t i = lane; i < ch.w; i += 64) {
                const uint32_t o = b0 + ch.z + i;
                if (o < cap) {
                    dst_node[o] = src_node[src + i];
                    dst_query[o] = src_query[src + i];
                }
            }
        }
        return;
    }
    if (threadIdx.x < 64) cnt[threadIdx.x] = 0u;
    __syncthreads();
    const int32_t q0 = (int32_t)(w * per);
    for (uint32_t c = c0 + wid; c < c1; c += kOrderBlock / 64) {
        const uint4 ch = d.clist[c];
        const int64_t src = (int64_t)((uint64_t)ch.x | (uint64_t)ch.y << 32);
        constexpr int kPerLane = kStage3 / 64;  // a chunk is one staging flush
        uint32_t nd[kPerLane];
        int32_t q[kPerLane];
#pragma unroll
        for (int k = 0; k < kPerLane; ++k) {
            const uint32_t i = lane + 64u * k;
            if (i < ch.w) {
                nd[k] = src_node[src + i];
                q[k] = src_query[src + i];
            }
        }
#pragma unroll
        for (int k = 0; k < kPerLane; ++k) {
            const uint32_t i = lane + 64u * k, j = ch.z + i;
            if (i < ch.w && j < m) {
                const uint32_t qo = min((uint32_t)(q[k] - q0), 63u);
                lnode[j] = nd[k];
                lkey[j] = qo << 16 | atomicAdd(&cnt[qo], 1u);
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < 64) {  // exclusive scan of the 64 query counts
        const uint32_t v = cnt[threadIdx.x];
        uint32_t x = v;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t y = __shfl_up(x, off);
            if ((int)threadIdx.x >= off) x += y;
        }
        cnt[threadIdx.x] = x - v;
    }
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < m; j += kOrderBlock) {
        const uint32_t key = lkey[j], qo = key >> 16;
        const uint32_t o = b0 + cnt[qo] + (key & 0xFFFFu);
        dst_node[o] = lnode[j];
        dst_query[o] = q0 + (int32_t)qo;
    }
}

static void front_finish_waves(DevState& d, int kind, int64_t waves, uint32_t per, hipStream_t s) {
    const int c = d.fcur[kind], nb = c ^ 1;  // the production is in the spare buffer's segments
    launch_exscan(d, d.wave_tot[kind], d.wave_base, waves, d.ctr + C_WAVE_TOTAL, s);
    fill_u32(d.wave_nch, waves, 0u, s);
    hipLaunchKernelGGL(k_chunk_count, dim3(512), dim3(kBlock), 0, s, d, kind);
    launch_exscan(d, d.wave_nch, d.wave_cbase, waves, d.ctr + C_WAVE_CHUNKS, s);
    hipLaunchKernelGGL(k_chunk_list, dim3(512), dim3(kBlock), 0, s, d, kind);
    hipLaunchKernelGGL(k_wave_order, dim3((unsigned)waves), dim3(kOrderBlock), 0, s, d, kind, (uint32_t)waves, per,
                       d.fnode[kind][nb], d.fquery[kind][nb], d.fnode[kind][c], d.fquery[kind][c],
                       d.fsize + 2 * kind + c);
}

static FrontIn cur_front(DevState& d) {
    FrontIn f;
    for (int k = 0; k < 2; ++k) {
        const int b = d.fcur[k];
        f.node[k] = d.fnode[k][b];
        f.query[k] = d.fquery[k][b];
        f.size[k] = d.fsize + 2 * k + b;
        f.cap[k] = (uint32_t)std::min<int64_t>(d.front_cap[k], 0xFFFFFFFFll);
    }
    return f;
}
__host__ __device__ inline FrontSink null_sink() { return FrontSink{nullptr, nullptr, nullptr, 0u, 0u}; }

// One 64-lane launch (a kernel, not memsets: the batched frame graph records it): the per-step
// pair counters, the visit counter and the segment counters of both pair lists.
__global__ void k_reset_step(DevState d) { zero_step_counters(d, threadIdx.x); }
static void reset_step_counters(DevState& d, hipStream_t s) {
    static_assert(kPairSegs == 64, "one lane per segment counter");
    hipLaunchKernelGGL(k_reset_step, dim3(1), dim3(kPairSegs), 0, s, d);
}

static unsigned stream_grid() { return 2048; }

// ---------------------------------------------------------------- launch-shape tuning
// The reference picks one block size per kernel from the occupancy API
// (system/CudaDevice/CudaDevice.cu:60-94). Here the grid of the grid-stride kernels,
// KEEP's entries per thread and the workgroup size of KEEP and the narrow phase (2, 4
// or 8 wave64s, their LDS sized to match) are tuned per kernel and size class ceil(log2 n), by
// timing candidates on live data (bvhcd_autotune / bvhcd_batch_autotune). The table is
// process-wide and not locked.
namespace {
constexpr int kClasses = 40;
unsigned g_grid[TK_COUNT][kClasses] = {};
struct TuneTrial {
    int kernel, cls;
    unsigned grid;
    float ms;
};
std::vector<TuneTrial> g_trials;
int size_class(int64_t n) {
    int c = 0;
    while (c < kClasses - 1 && ((int64_t)1 << c) < n) ++c;
    return c;
}
}  // namespace

// The shapes used until a kernel is tuned. n = triangles of the scene (of the querying object for an
// inter-object front). KEEP up to half a million triangles is bound by the length of its dependent rounds,
// and one resident set of workgroups (1536 of 256 threads; 1024 start sooner on the smallest) has the
// fewest; above by throughput, where small workgroups leave the tail early. KEEP and narrow phase, us,
// 1024 x 256 / 1536 x 256 / 16384 x 128 threads: 216k triangles 59 / 59 / -, 272k 70 / 70 / 83, 498k 97 / 96 /
// 102 (8192 x 128), 625k 296 / 288 / 281, 2.1M 845 / 865 / 829 (two entries in flight per thread). From
// 2^22 triangles on larger workgroups: 16384 of 128 / 256 / 512 threads, 8.4M sheets on the boxes 1273 /
// 1204 / 1154, on the records (launch_keep) 803 / 735 / 793; 4.2M on the records 411 / 407 / 437, 2.1M
// 446 / 508 / 636.
// The narrow phase: 4096 x 256 -> 16384 x 256 from a million triangles on, 2.1M 0.253 -> 0.235,
// 8.4M 0.341 -> 0.311; below it is the same within 0.5 us from 1024 workgroups on.
static unsigned default_shape(int kernel, int64_t n) {
    switch (kernel) {
        case TK_KEEP:
            return n <= (1 << 19) ? make_shape(n <= (1 << 17) ? 1024u : 1536u, 2u)
                                  : make_shape(16384u, 2u, n <= (1 << 22) ? 2u : 8u);
        case TK_NARROW: return make_shape(n <= (1 << 19) ? 1024u : n <= (1 << 20) ? 4096u : 16384u, 1u);
        default: return 0xFFFFFFu;  // batched traversal: one group of queries per wave
    }
}
unsigned tuned_shape(int kernel, int64_t n, int64_t queries) {
    const unsigned g = g_grid[kernel][size_class(n)];
    return g ? g : default_shape(kernel, queries ? queries : n);
}
bool shape_set(int kernel, int64_t n) { return g_grid[kernel][size_class(n)] != 0; }
void set_tuned_shape(int kernel, int64_t n, unsigned sh) { g_grid[kernel][size_class(n)] = sh; }
void record_tuning(int kernel, int64_t n, unsigned sh, float ms) {
    g_trials.push_back({kernel, size_class(n), sh, ms});
}
std::string tuning_report() {
    static const char* names[TK_COUNT] = {"k_keep", "k_narrow", "k_batch_cd"};
    std::string r = "kernel size_class grid unroll block ms_per_launch chosen\n";
    char line[160];
    for (const TuneTrial& t : g_trials) {
        snprintf(line, sizeof(line), "%s 2^%d %u %u %u %.4f %s\n", names[t.kernel], t.cls, shape_grid(t.grid),
                 shape_unroll(t.grid), 64u * shape_waves(t.grid), t.ms, g_grid[t.kernel][t.cls] == t.grid ? "*" : "");
        r += line;
    }
    return r;
}

// ---------------------------------------------------------------- per-wave stacks of node tests
constexpr uint32_t kDescStack = 512;
template <int W, uint32_t CAP = kDescStack>
struct DescStack {
    int2 item[W][CAP];  // (query, node << 1 | leaf)
    uint32_t top[W];
};

// Pushes (q, node enc) for the lanes with pred set; returns false for a lane whose item did not
// fit (it must then test that node itself). Called by all active lanes of the wave.
template <uint32_t CAP = kDescStack>
__device__ inline bool desc_push(lds_int2* stk, lds_u32* top, bool pred, int32_t q, int32_t enc) {
    const uint64_t m = __ballot(pred);
    if (m == 0) return true;
    const uint32_t t = *top;
    const uint32_t rank = (uint32_t)__popcll(m & lanes_below());
    const bool fits = t + rank < CAP;
    if (pred && fits) {
        stk[t + rank].x = q;
        stk[t + rank].y = enc;
    }
    const uint32_t pushed = (uint32_t)__popcll(__ballot(pred && fits));
    if (lane_id() == __ffsll((long long)__ballot(1)) - 1) *top = t + pushed;
    return fits || !pred;
}

__device__ inline float lane_perm(int at, float v) { return i2f(__builtin_amdgcn_ds_bpermute(at, f2i(v))); }
// Takes up to one item per active lane off the wave's stack; returns the number taken.
__device__ inline uint32_t desc_pop(lds_int2* stk, lds_u32* top, bool& active, int32_t& q, int32_t& enc) {
    const uint64_t m = __ballot(1);
    const uint32_t t = *top, rank = (uint32_t)__popcll(m & lanes_below());
    const uint32_t take = min(t, (uint32_t)__popcll(m));
    active = rank < take;
    if (active) {
        q = stk[t - 1 - rank].x;
        enc = stk[t - 1 - rank].y;
    }
    __builtin_amdgcn_wave_barrier();
    if (lane_id() == __ffsll((long long)m) - 1) *top = t - take;
    __builtin_amdgcn_wave_barrier();
    return take;
}

// ---------------------------------------------------------------- pure traversal / generate
// Self-CD query leaf i walks the leaves after it, from lca[i + 1] (its record's escape) on: that node's
// subtree, then the subtree at its escape, and so on to the end; inter-object: every query walks the
// whole tree from its root lca[0]. A wave takes `per` queries; the nodes still to be tested lie on its
// LDS stack as (query's lane | kChain for a walk's own nodes, encoded node), and every lane tests one
// per round: a node that does not overlap and every leaf is an entry of the query's front, an
// overlapping node pushes its children, a chain node the next one. The nodes tested, the entries and the
// pairs are those of the queries' own walks. Bound by the latency of the rounds on small scenes, by the
// vector L1 (three divergent 16-byte loads per test) and the staged output on large ones. Against a walk
// per lane, parts of it handed to idle lanes, us: 2.6k triangles 48 -> 36, 41k 62 -> 45, 65k boxes 134 ->
// 101, 130k 152 -> 115, 8.4M 3850 -> 3350.
constexpr uint32_t kWalkStack = 256, kWalkStage = 192;  // 24 resident waves per CU
static_assert(kWalkStage <= kStage3, "k_wave_order's lanes hold a chunk (one flush) of up to kStage3 entries");
constexpr int32_t kChain = 64;
template <bool FRONT>
__global__ void __launch_bounds__(kBlock) k_traverse(int32_t n, uint32_t per, DevState d, FrontSink fi, FrontSink fe) {
    __shared__ StagesT<kWalkStage> st;
    __shared__ DescStack<kWaves, kWalkStack> ds;
    stages_init(st);
    const int w = threadIdx.x >> 6, lane = lane_id();
    if (lane == 0) ds.top[w] = 0;
    lds_int2* stk = (lds_int2*)ds.item[w];
    lds_u32* top = (lds_u32*)&ds.top[w];
    const Out out = make_out(st, fi, fe, d);
    const int32_t nq = d.inter ? d.nq : n - 1;
    const int32_t q0 = (int32_t)((blockIdx.x * kWaves + w) * per), i = q0 + lane;
    const bool query = lane < (int)per && i < nq;
    Box own{};
    int32_t start = -1;
    if (query) {
        const float4 lo = d.qleaf[i].lo, hi = d.qleaf[i].hi;
        own = rec_box(lo, hi);
        start = d.inter ? d.leaf_lca[0] : f2i(hi.w);
    }
    uint32_t visits = 0;
    desc_push<kWalkStack>(stk, top, query && start != -1, lane | kChain, start);
    const int64_t limit = 64 * (2 * d.maxT + 16);
    for (int64_t rounds = 0;; ++rounds) {
        const uint32_t t = *top;
        if (t == 0) break;
        if (rounds > limit) {  // only a corrupted tree gets here (flag 16, a device error)
            if (lane == 0) atomicOr(&d.ctr[C_OVF], 16u);
            break;
        }
        // an item pushes three at most: fewer are taken when the stack is nearly full
        const uint32_t take = max(1u, min(min(t, 64u), (kWalkStack - t) / 2u));
        const bool active = (uint32_t)lane < take;
        int32_t x = 0, enc = 0;
        if (active) {
            x = stk[t - 1 - lane].x;
            enc = stk[t - 1 - lane].y;
        }
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) *top = t - take;
        __builtin_amdgcn_wave_barrier();
        const int32_t nd = enc >> 1, q = q0 + (x & 63);
        const bool leaf = enc & 1;
        float4 lo = make_float4(0.f, 0.f, 0.f, 0.f), hi = lo;
        int4 tp = make_int4(0, 0, 0, 0);
        if (active) {
            const NodeRec* r = leaf ? &d.leaf[nd] : &d.inode[nd];
            lo = r->lo;
            hi = r->hi;
            if (!leaf) tp = d.itopo[nd];
        }
        const int from = (x & 63) << 2;
        const Box qb{lane_perm(from, own.mnx), lane_perm(from, own.mny), lane_perm(from, own.mnz),
                     lane_perm(from, own.mxx), lane_perm(from, own.mxy), lane_perm(from, own.mxz)};
        const bool hit = active && box_overlap(qb, lo, hi);
        visits += active ? 1u : 0u;
        const bool next = active && (x & kChain) && f2i(hi.w) != -1, grow = hit && !leaf;
        const bool ok_n = desc_push<kWalkStack>(stk, top, next, x, f2i(hi.w));
        const bool ok_l = desc_push<kWalkStack>(stk, top, grow, x & 63, tp.x),
                   ok_r = desc_push<kWalkStack>(stk, top, grow, x & 63, tp.y);
        bool pair = hit && leaf;
        if (out.skip_adj && pair) pair = !faces_share_vertex(out.lfaces, q, nd);
        out.pair_push(pair, make_int2(q, nd));
        if (FRONT) {
            stage_push(out.fe, out.ovf, out.sb[1], out.sf[1], out.scap, active && leaf, make_int2(q, nd));
            stage_push(out.fi, out.ovf, out.sb[0], out.sf[0], out.scap, active && !leaf && !hit, make_int2(q, nd));
        }
        // no room (a full stack's last item only): this lane walks what did not fit
        if (grow && !(ok_l && ok_r)) visits += stackless<FRONT>(d, out, q, qb, ok_l ? tp.y : tp.x, f2i(hi.w));
        if (!ok_n) visits += stackless<FRONT>(d, out, q, qb, f2i(hi.w), -1);
    }
    if (FRONT) out.final_flush();
    else out.pair_final();
    add_visits(d, visits);
}

// ---------------------------------------------------------------- pairs of 64 queries at a time
// The overlapping leaf pairs (q, j > q) of a whole tree, without a front. A wave takes `size` (up to 64)
// queries (neighbouring sorted leaves) together and works in two steps:
//  * nodes: the tree from a cut of up to 64 nodes near its root, 64 nodes per round off a per-wave LDS stack, each lane testing
//    one node against the boxes of the 64 queries and dropping subtrees that hold no leaf after the
//    first query. A run of neighbouring leaves can jump (Morton order), and one box around a jump
//    covers everything between: the run is cut at its three widest jumps and a node is tested
//    against the four pieces' boxes (2M-triangle folded cloth: 481 nodes per wave instead of 793,
//    the worst wave 2281 instead of 59425);
//  * leaves: those reached (170 per wave there) are tested against runs of 8 neighbouring queries (RUNS):
//    a leaf per lane against each run's box first, then the 8 queries of the runs it overlaps, 8 such
//    items per step, boxes in LDS; or every lane tests every leaf against its own query, the leaf's box
//    loaded once for the wave through the scalar cache. Hits go to the wave's LDS list.
// Every node test serves 64 queries and every leaf record is fetched once per wave, where a walk
// or a front entry per query fetches two 32-byte records per test. A pair is found exactly when the
// leaves' boxes overlap, as in a query's own walk: a node's box holds its leaves' boxes and a piece's
// box its queries', so no ancestor of an overlapping leaf is dropped. (Boxes given by the caller can
// hold NaN, for which that is not so: they take the walks and fronts.)
// skip_adj: pairs of triangles that share a vertex are removed when the LDS list is flushed (64 pairs
// per step; the query's vertex ids come from its lane).
// Bound by the latency of one round after another on small scenes, by instruction issue on large ones
// (48 % of the VALU and 47 % of the scalar slots busy on 64 scenes of 2.6M triangles). Folded cloths: 180k
// triangles 185 -> 93 us (against the queries' own walks sharing a wave's lanes), 64 scenes of 2.6M
// triangles 1.04 -> 0.56 ms (against a walk per lane). KEEP's test of a front stays where there is one:
// 0.44 ms against 0.66 ms here on the 2M cloth, 13 us against 17 us on 2,560 triangles.
// A group's cut (CUT): the nodes at which its search ended, which cover every leaf the group can meet.
// The tree of the batched scenes stays for the refits between two builds: the build's traversal records
// the groups' cuts, the others start from them instead of from the root (on 64 scenes 24 rounds of nodes
// become 6; 0.61 -> 0.49 ms a refit
// frame) and go on below a node that overlaps by now. A cut of more than kCutCap nodes isn't held,
// its group starts from the root.
enum GroupCut : int { kCutNone = 0, kCutRecord = 1, kCutRead = 2 };
constexpr uint32_t kGroupStack = 512;  // encoded nodes per wave (2 KB)
constexpr int kGroupPieces = 4;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef BVHCD_LDS f32x4 lds_f32x4;
typedef volatile BVHCD_LDS uint16_t lds_u16;
constexpr int kRun = 8;             // neighbouring queries tested together (RUNS)
template <bool RUNS>
struct GroupLds {
    static constexpr uint32_t kStage = RUNS ? 256 : 512;  // staged pairs per wave
    f32x4 leaf[kWaves][RUNS ? 64 : 1][2];   // RUNS: a round's leaves by lane: (lo, id), (hi, -)
    f32x4 query[kWaves][RUNS ? 64 : 1][2];  // and the queries: (lo, -), (hi, last leaf)
    uint16_t item[kWaves][RUNS ? 64 * 64 / kRun : 2];  // run << 6 | lane of the leaf
    uint32_t cand[kWaves][RUNS ? 1 : 128];  // else the leaves' ids
    uint32_t stack[kWaves][kGroupStack];
    int2 pairs[kWaves][kStage];
    uint32_t fill[kWaves][2];          // [1]: segment rotor (stage_flush)
};
typedef const __attribute__((address_space(4))) float4 const_float4;  // loaded through the scalar cache
__device__ inline float lane_f(float v, int lane) {
    return i2f(__builtin_amdgcn_readlane(f2i(v), lane));
}
// Box of each aligned run of 8 lanes, in all its lanes.
template <int CTRL>
__device__ inline float dpp_f(float v) {
    return i2f(__builtin_amdgcn_mov_dpp(f2i(v), CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ inline Box dpp_merge(const Box& b) {
    return box_merge(b, Box{dpp_f<CTRL>(b.mnx), dpp_f<CTRL>(b.mny), dpp_f<CTRL>(b.mnz), dpp_f<CTRL>(b.mxx),
                            dpp_f<CTRL>(b.mxy), dpp_f<CTRL>(b.mxz)});
}
__device__ inline Box run_box(const Box& b) {  // lane ^ 1, lane ^ 2, then the other four
    static_assert(kRun == 8, "two quad permutations and a half-row mirror");
    return dpp_merge<0x141>(dpp_merge<0x4E>(dpp_merge<0xB1>(b)));
}
__device__ inline uint32_t wave_max(uint32_t v) {
    for (int off = 32; off > 0; off >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, off));
    return v;
}
__device__ inline void wave_lds_order() {  // LDS operations of one wave complete in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool BATCH, bool RUNS, int CUT>
__global__ void __launch_bounds__(kBlock) k_group_cd(int32_t n, uint32_t size, DevState d,
                                                     const uint64_t* __restrict__ keys,
                                                     const int32_t* __restrict__ scene_last) {
    constexpr uint32_t kGroupStage = GroupLds<RUNS>::kStage;
    __shared__ GroupLds<RUNS> lds;
    const int w = threadIdx.x >> 6, lane = lane_id();
    lds_u32* const stk = (lds_u32*)lds.stack[w];
    lds_f32x4* const lbox = (lds_f32x4*)lds.leaf[w];
    lds_f32x4* const qbox = (lds_f32x4*)lds.query[w];
    lds_u16* const item = (lds_u16*)lds.item[w];
    lds_u32* const cand = (lds_u32*)lds.cand[w];
    lds_int2* const sb = (lds_int2*)lds.pairs[w];
    lds_u32* const sf = (lds_u32*)lds.fill[w];
    if (lane == 0) sf[1] = rotor_start();
    const SegPairSink sink = pair_segments(d, 0, 4u);
    uint32_t* const ovf = &d.ctr[C_OVF];
    const bool drop_adj = d.skip_adj != 0;
    // each XCD takes one contiguous eighth of the groups; the grid is a multiple of the XCDs
    const uint32_t groups = ((uint32_t)n + size - 1u) / size, share = (groups + kXcds - 1) / kXcds;
    const uint32_t xcd = blockIdx.x % kXcds, end_gi = min((xcd + 1) * share, groups);
    uint32_t visits = 0;
    for (uint32_t gi = xcd * share + (blockIdx.x / kXcds) * kWaves + w; gi < end_gi;  // wave-uniform
         gi += gridDim.x / kXcds * kWaves) {
        const int32_t g0 = (int32_t)(gi * size), q = g0 + lane;
        const bool valid = (uint32_t)lane < size && q < n;
        Box qb = empty_box();
        int32_t after = INT32_MAX, last = n - 1;  // this lane's leaves: (after, last]
        int32_t f0 = 0, f1 = 0, f2 = 0;           // its triangle's vertices
        if (valid) {
            const float4 lo = d.leaf[q].lo, hi = d.leaf[q].hi;
            qb = rec_box(lo, hi);
            after = q;
            if (BATCH) last = scene_last[(int32_t)(keys[q] >> 30)];
            if (drop_adj) {
                f0 = d.lfaces[3 * (int64_t)q];
                f1 = d.lfaces[3 * (int64_t)q + 1];
                f2 = d.lfaces[3 * (int64_t)q + 2];
            }
        }
        // the wave's last leaf (scenes follow one another in leaf order)
        const int32_t glast =
            BATCH ? __builtin_amdgcn_readlane(last, min((int32_t)size - 1, n - 1 - g0)) : n - 1;
        // cut the 64 queries at their widest jumps between box centres
        const float cx = qb.mnx + qb.mxx, cy = qb.mny + qb.mxy, cz = qb.mnz + qb.mxz;
        const float gap = fabsf(__shfl_down(cx, 1) - cx) + fabsf(__shfl_down(cy, 1) - cy) + fabsf(__shfl_down(cz, 1) - cz);
        uint32_t key = lane + 1 < (int)size && q + 1 < n ? (((uint32_t)f2i(gap) & 0x7FFFFFC0u) | (uint32_t)lane) : 0u;
        uint64_t heads = 1ull;  // first lanes of the pieces
#pragma unroll
        for (int c = 1; c < kGroupPieces; ++c) {
            const uint32_t k = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave_max(key));
            if (k == 0u) break;
            heads |= 2ull << (k & 63u);
            if (lane == (int)(k & 63u)) key = 0u;
        }
        const int first = 63 - __clzll((long long)(heads & ((2ull << lane) - 1ull)));  // this lane's piece
        Box pb = qb;
        for (int off = 1; off < 64; off <<= 1) {  // box of the piece up to this lane
            const Box o{__shfl_up(pb.mnx, off), __shfl_up(pb.mny, off), __shfl_up(pb.mnz, off),
                        __shfl_up(pb.mxx, off), __shfl_up(pb.mxy, off), __shfl_up(pb.mxz, off)};
            if (lane - off >= first) pb = box_merge(pb, o);
        }
        Box piece[kGroupPieces];
#pragma unroll
        for (int c = 0; c < kGroupPieces; ++c) {  // wave-uniform (scalar registers)
            const uint64_t rest = heads & (heads - 1ull);  // without its first piece
            const int end = rest ? __ffsll((long long)rest) - 2 : 63;
            piece[c] = Box{lane_f(pb.mnx, end), lane_f(pb.mny, end), lane_f(pb.mnz, end),
                           lane_f(pb.mxx, end), lane_f(pb.mxy, end), lane_f(pb.mxz, end)};
            if (rest) heads = rest;  // fewer pieces: the last one again
        }
        Box run{};
        if (RUNS) {
            run = run_box(qb);
            qbox[2 * lane] = f32x4{qb.mnx, qb.mny, qb.mnz, 0.f};
            qbox[2 * lane + 1] = f32x4{qb.mxx, qb.mxy, qb.mxz, i2f(valid ? last : -1)};
        }

        uint32_t fill = 0;
        auto flush = [&]() {
            uint32_t f = fill;
            if (drop_adj) {  // compacted in place: every step writes below what it has read
                f = 0;
                for (uint32_t b = 0; b < fill; b += 128) {
                    int2 p[2];
                    int32_t v[2][3];
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const uint32_t i = b + 64u * u + lane;
                        p[u] = i < fill ? make_int2(sb[i].x, sb[i].y) : make_int2(g0, g0);
                        const int32_t* fc = d.lfaces + 3 * (int64_t)p[u].y;
                        v[u][0] = fc[0];
                        v[u][1] = fc[1];
                        v[u][2] = fc[2];
                    }
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const int src = p[u].x - g0;
                        const int32_t a0 = __shfl(f0, src), a1 = __shfl(f1, src), a2 = __shfl(f2, src);
                        const bool share = a0 == v[u][0] || a0 == v[u][1] || a0 == v[u][2] || a1 == v[u][0] ||
                                           a1 == v[u][1] || a1 == v[u][2] || a2 == v[u][0] || a2 == v[u][1] ||
                                           a2 == v[u][2];
                        const bool keep = b + 64u * u + lane < fill && !share;
                        const uint64_t m = __ballot(keep);
                        if (keep) {
                            const uint32_t slot = f + (uint32_t)__popcll(m & lanes_below());
                            sb[slot].x = p[u].x;
                            sb[slot].y = p[u].y;
                        }
                        f += (uint32_t)__popcll(m);
                    }
                }
            }
            if (f) stage_flush(sink, ovf, sb, sf, f, ~0ull);
            fill = 0;
        };
        auto emit = [&](bool hit, int32_t qi, int32_t j) {  // room for 64 pairs is the caller's business
            const uint64_t m = __ballot(hit);
            if (m == 0ull) return;
            if (hit) {
                const uint32_t slot = fill + (uint32_t)__popcll(m & lanes_below());
                sb[slot].x = qi;
                sb[slot].y = j;
            }
            fill += (uint32_t)__popcll(m);
        };
        // RUNS: tests the leaves of the lanes with `reached` (box lo, hi, id nd): every run's box against
        // every leaf, a lane each, then the 8 queries of the runs that it overlaps, 8 such items at once
        auto test_runs = [&](bool reached, int32_t nd, const float4& lo, const float4& hi) {
            constexpr int kAtOnce = 2;
            constexpr uint32_t kItems = 64 / kRun;
            if (reached) {
                lbox[2 * lane] = f32x4{lo.x, lo.y, lo.z, i2f(nd)};
                lbox[2 * lane + 1] = f32x4{hi.x, hi.y, hi.z, 0.f};
            }
            uint32_t items = 0;
            for (uint32_t r = 0; r < size; r += kRun) {
                const Box b{lane_f(run.mnx, (int)r), lane_f(run.mny, (int)r), lane_f(run.mnz, (int)r),
                            lane_f(run.mxx, (int)r), lane_f(run.mxy, (int)r), lane_f(run.mxz, (int)r)};
                const bool near = reached && nd > g0 + (int32_t)r && box_overlap(b, lo, hi);
                const uint64_t m = __ballot(near);
                if (near) item[items + (uint32_t)__popcll(m & lanes_below())] = (uint16_t)(r / kRun << 6 | (uint32_t)lane);
                items += (uint32_t)__popcll(m);
            }
            wave_lds_order();
            for (uint32_t k0 = 0; k0 < items; k0 += kAtOnce * kItems) {
                if (fill > kGroupStage - 64u * kAtOnce) flush();
                int32_t qi[kAtOnce], j[kAtOnce];
                bool h[kAtOnce];
#pragma unroll
                for (int u = 0; u < kAtOnce; ++u) {
                    const uint32_t k = k0 + u * kItems + (uint32_t)(lane / kRun);
                    const uint32_t it = item[min(k, items - 1u)], lf = it & 63u, qs = (it >> 6) * kRun + (lane % kRun);
                    const f32x4 a = lbox[2 * lf], b = lbox[2 * lf + 1], c = qbox[2 * qs], e = qbox[2 * qs + 1];
                    j[u] = f2i(a.w);
                    qi[u] = g0 + (int32_t)qs;
                    h[u] = k < items && j[u] > qi[u] && j[u] <= f2i(e.w) &&
                           box_overlap(Box{c.x, c.y, c.z, e.x, e.y, e.z}, make_float4(a.x, a.y, a.z, 0.f),
                                       make_float4(b.x, b.y, b.z, 0.f));
                }
#pragma unroll
                for (int u = 0; u < kAtOnce; ++u) emit(h[u], qi[u], j[u]);
            }
            wave_lds_order();
        };
        // else: tests the first k (<= 64) of the leaves reached, kAtOnce loaded together (what lies past
        // the k-th is some leaf and is not counted)
        auto test_leaves = [&](uint32_t k) {
            constexpr int kAtOnce = 4;
            const int32_t cv = (int32_t)cand[min((uint32_t)lane, k - 1u)];
            for (uint32_t c = 0; c < k; c += kAtOnce) {
                if (fill > kGroupStage - 64u * kAtOnce) flush();
                float4 lo[kAtOnce], hi[kAtOnce];
                int32_t j[kAtOnce];
#pragma unroll
                for (int u = 0; u < kAtOnce; ++u) {
                    j[u] = __builtin_amdgcn_readlane(cv, (int)(c + u));
                    const_float4* r = (const_float4*)(uintptr_t)&d.leaf[j[u]];
                    lo[u] = make_float4(r[0].x, r[0].y, r[0].z, 0.f);
                    hi[u] = make_float4(r[1].x, r[1].y, r[1].z, 0.f);
                }
#pragma unroll
                for (int u = 0; u < kAtOnce; ++u)
                    emit(c + u < k && j[u] > after && (!BATCH || j[u] <= last) && box_overlap(qb, lo[u], hi[u]), q, j[u]);
            }
        };
        uint32_t top = 0, ncand = 0;         // wave-uniform
        uint32_t cn = 0, next = 0, rec = 0;  // the cut's nodes, those taken of them, nodes recorded
        uint32_t ids = 0;                    // the cut's next 64 nodes
        uint32_t* const cut = CUT ? d.cut + (int64_t)gi * kCutCap : nullptr;
        if (CUT == kCutRead) cn = (uint32_t)__builtin_amdgcn_readfirstlane((int)d.cut_cnt[gi]);
        if (CUT == kCutRead && cn <= kCutCap) {
            if ((uint32_t)lane < cn) ids = cut[lane];
        } else {  // from the cut near the root
            cn = 0;
            top = d.top_cut[64];
            stk[lane] = d.top_cut[lane];
        }
        // every node enters the stack at most once; the bound only guards against a corrupted tree
        // (flag 16, reported as a device error, instead of a hang)
        const int64_t limit = 2 * d.maxT + 16;
        for (int64_t round = 0; top > 0 || next < cn; ++round) {
            if (round > limit) {
                if (lane == 0) atomicOr(ovf, 16u);
                break;
            }
            uint32_t take;
            int32_t e = 0;
            if (CUT == kCutRead && next < cn && top < 64u) {
                take = min(cn - next, 64u);
                e = (int32_t)ids;
                next += take;
                ids = next + lane < cn ? cut[next + lane] : 0u;
            } else {
                take = max(1u, min(min(top, 64u), kGroupStack - top));
                top -= take;
                if ((uint32_t)lane < take) e = (int32_t)stk[top + lane];
            }
            const bool act = (uint32_t)lane < take;
            const int32_t nd = e >> 1;
            const bool leaf = e & 1;
            bool hit = false, ends = false;  // ends: the search stops at this node, or walks on below it
            float4 lo = make_float4(0.f, 0.f, 0.f, 0.f), hi = lo;
            int4 tp = make_int4(0, 0, 0, 0);
            if (act) {
                const NodeRec* r = leaf ? &d.leaf[nd] : &d.inode[nd];
                lo = r->lo;
                hi = r->hi;
                if (!leaf) tp = d.itopo[nd];
                ++visits;
                const int32_t begin = leaf ? nd : f2i(lo.w), end = leaf ? nd : tp.w;  // its leaves
                bool any = false;
#pragma unroll
                for (int c = 0; c < kGroupPieces; ++c) any |= box_overlap(piece[c], lo, hi);
                const bool ours = end > g0 && (!BATCH || begin <= glast);
                hit = any && ours;
                ends = ours && (leaf || !any);
            }
            const uint64_t mi = __ballot(hit && !leaf), ml = __ballot(hit && leaf);
            if (mi) {
                const uint32_t slot = top + 2u * (uint32_t)__popcll(mi & lanes_below());
                const bool fits = slot + 2u <= kGroupStack;
                if (hit && !leaf && fits) {
                    stk[slot] = (uint32_t)tp.x;
                    stk[slot + 1] = (uint32_t)tp.y;
                }
                const uint64_t mf = __ballot(hit && !leaf && fits);
                top += 2u * (uint32_t)__popcll(mf);
                ends = ends || (hit && !leaf && !fits);
                // no room (only a full stack's last item, see `take`): the lanes walk that subtree
                for (uint64_t over = mi & ~mf; over; over &= over - 1ull) {
                    const int src = __ffsll((long long)over) - 1;
                    const int32_t stop = __builtin_amdgcn_readlane(f2i(hi.w), src);
                    int32_t cur = valid ? __builtin_amdgcn_readlane(tp.x, src) : stop;
                    int64_t steps = 0;
                    while (__ballot(cur != stop) != 0ull) {
                        if (++steps > limit) {
                            if (lane == 0) atomicOr(ovf, 16u);
                            break;
                        }
                        if (fill > kGroupStage - 64u) flush();
                        bool h = false;
                        int32_t j = 0;
                        if (cur != stop) {
                            const int32_t x = cur >> 1;
                            const NodeRec* r = (cur & 1) ? &d.leaf[x] : &d.inode[x];
                            const float4 a = r->lo, b = r->hi;
                            const bool o = box_overlap(qb, a, b);
                            ++visits;
                            if ((cur & 1) || !o) {
                                h = (cur & 1) && o && x > after && (!BATCH || x <= last);
                                j = x;
                                cur = f2i(b.w);
                            } else {
                                cur = d.itopo[x].x;
                            }
                        }
                        emit(h, q, j);
                    }
                }
            }
            if (CUT == kCutRecord) {
                const uint64_t me = __ballot(ends);
                const uint32_t slot = rec + (uint32_t)__popcll(me & lanes_below());
                if (ends && slot < kCutCap) cut[slot] = (uint32_t)e;
                rec += (uint32_t)__popcll(me);
            }
            if (RUNS) {
                if (ml) test_runs(hit && leaf, nd, lo, hi);
                continue;
            }
            if (ml) {
                if (hit && leaf) cand[ncand + (uint32_t)__popcll(ml & lanes_below())] = (uint32_t)nd;
                ncand += (uint32_t)__popcll(ml);
                wave_lds_order();
            }
            const bool done = top == 0u && next >= cn;
            if (ncand >= 64u || (done && ncand > 0u)) {
                test_leaves(min(ncand, 64u));
                const uint32_t rest = ncand > 64u ? ncand - 64u : 0u;
                if ((uint32_t)lane < rest) cand[lane] = cand[64 + lane];
                wave_lds_order();
                ncand = rest;
                if (done && ncand > 0u) {  // the last round's overhang
                    test_leaves(ncand);
                    ncand = 0;
                }
            }
        }
        flush();
        if (CUT == kCutRecord && lane == 0) d.cut_cnt[gi] = rec;  // above kCutCap: not held
    }
    add_visits(d, visits);
}

// Queries per wave. Small scenes are bound by their heaviest wave, large ones by the node tests, which
// 64 queries share: pure traversal, us, with 64 / 32 / 16 / 8: 2.6k 35 / 26 / 21 / 17, 28k 110 / 62 / 40 /
// 34, 41k 49 / 36 / 30 / 42, 65k 124 / 73 / 47 / 59, 180k 128 / 93 / 100 / 148, 522k 328 / 286 / 320 / 475,
// 718k 363 / 368 / 419 / 642, 2.1M 716 / 866 / 1223 / 1968.
static uint32_t group_size(int32_t n) {
    return n <= 1 << 15 ? 8u : n <= 3 << 15 ? 16u : n <= 5 << 17 ? 32u : 64u;
}
// Workgroups of k_group_cd, one group per wave: the same number for each XCD's share.
static unsigned group_grid(int32_t n) {
    const unsigned g = group_size(n), share = (((unsigned)n + g - 1u) / g + kXcds - 1) / kXcds;
    return kXcds * ((share + kWaves - 1) / kWaves);
}

// Leaf tests by runs of 8 queries (RUNS) up to this many leaves: an eighth of the box tests, but twice
// the LDS and a third fewer resident waves, which larger scenes need (us, runs / every lane its query: 7k
// 48 / 69, 65k 47 / 66, 130k 70 / 88, 318k 136 / 165, 718k 363 / 370, 1.2M 611 / 574, 2.1M 775 / 716).
constexpr int32_t kGroupRuns = 3 << 18;
int64_t cut_groups(int64_t n) { return (n + group_size((int32_t)n) - 1) / group_size((int32_t)n); }
template <bool BATCH, int CUT>
static void launch_group_cd(DevState& d, int32_t n, unsigned grid, const uint64_t* keys, const int32_t* scene_last,
                            hipStream_t s) {
    if (n <= kGroupRuns)
        hipLaunchKernelGGL((k_group_cd<BATCH, true, CUT>), dim3(grid), dim3(kBlock), 0, s, n, group_size(n), d, keys, scene_last);
    else
        hipLaunchKernelGGL((k_group_cd<BATCH, false, CUT>), dim3(grid), dim3(kBlock), 0, s, n, group_size(n), d, keys, scene_last);
}

// Queries of a traversal: the leaves before the last one (self-CD) or the other object's leaves.
static int64_t query_count(const DevState& d, int32_t n) { return d.inter ? d.nq : n - 1; }
// Queries a wave of k_traverse takes. With few waves the longest wave is the kernel's time, with enough of
// them full waves do the least: GENERATE in node order, us, with 64 / 32 / 16 / 8: 2.6k 133 / 113 / 94 / 89,
// 28k 359 / 267 / 214 / 187, 41k 196 / 167 / 148 / 150, 180k 547 / 463 / 438 / 464, 522k 2170 / 1712 / 1518 /
// 1456, 1.2M 3615 / 2943 / 2692 / 2874, 2.1M 4158 / 3730 / 3737 / 4240, 8.4M 10622 / 10953 / 11817 / 14525.
uint32_t walk_queries(int64_t nq) { return nq <= 1 << 15 ? 8u : nq <= 3 << 19 ? 16u : nq <= 1 << 22 ? 32u : 64u; }
static unsigned walk_grid(int64_t nq) { return grid_for(nq, (int)(kWaves * walk_queries(nq))); }
int64_t max_walk_waves(int64_t T) {
    int64_t w = 1;
    for (const int64_t nq : {T, std::min<int64_t>(T, 1 << 22), std::min<int64_t>(T, 3 << 19), std::min<int64_t>(T, 1 << 15)})
        w = std::max<int64_t>(w, (int64_t)walk_grid(nq) * kWaves);
    return w;
}

// Self-CD over boxes made from the vertices.
static bool group_ok(const DevState& d) { return !d.inter && !d.pbox; }

void launch_pure_cd(DevState& d, int32_t n, hipStream_t s) {
    reset_step_counters(d, s);
    const int64_t nq = query_count(d, n);
    if (group_ok(d) && nq > 0)
        launch_group_cd<false, kCutNone>(d, n, group_grid(n), nullptr, nullptr, s);
    else if (nq > 0) {
        hipLaunchKernelGGL(k_traverse<false>, dim3(walk_grid(nq)), dim3(kBlock), 0, s, n, walk_queries(nq), d,
                           null_sink(), null_sink());
    }
}

// ---------------------------------------------------------------- batched scenes
// Self-CD over many scenes in one tree: the sort keys carry the scene id above the 30 Morton
// bits, so every scene is one subtree and its leaves are contiguous; query x of the scene whose
// last leaf is b is paired with the leaves (x, b] only. At most `grid` workgroups, each taking
// groups of its XCD's share in turn. Counters are cleared with a kernel (no memset nodes) so that
// the sequence can be captured in a graph.
void launch_batch_cd(DevState& d, int32_t n, const uint64_t* keys, const int32_t* scene_last, unsigned grid,
                     bool built, hipStream_t s) {
    reset_step_counters(d, s);
    const unsigned g = std::min(group_grid(n), kXcds * std::max(grid / kXcds, 1u));
    if (n < 2) return;
    if (built) launch_group_cd<true, kCutRecord>(d, n, g, keys, scene_last, s);
    else launch_group_cd<true, kCutRead>(d, n, g, keys, scene_last, s);
}

// ---------------------------------------------------------------- ordering
// beg[b] = first position of bucket b in the sorted keys (b in [0, nb]); key count from *dn.
__global__ void __launch_bounds__(kBlock) k_bucket_begin(const uint32_t* __restrict__ keys, const uint32_t* dn,
                                                         uint32_t cap, int32_t nb, uint32_t* __restrict__ beg) {
    const uint32_t m = min(*dn, cap);
    for (int32_t b = blockIdx.x * blockDim.x + threadIdx.x; b <= nb; b += gridDim.x * blockDim.x) {
        uint32_t lo = 0, hi = m;  // first index with keys[idx] >= b
        while (lo < hi) {
            const uint32_t mid = lo + ((hi - lo) >> 1);
            if (keys[mid] < (uint32_t)b) lo = mid + 1;
            else hi = mid;
        }
        beg[b] = lo;
    }
}

static int bits_for(int64_t v) {
    int b = 1;
    while (((int64_t)1 << b) <= v) ++b;
    return b;
}

// Fronts of the learned schedule are not node-ordered; they are sorted by query leaf instead
// (stable, so each query keeps its emission order): neighbouring queries read neighbouring
// nodes, which KEEP's per-XCD split then keeps inside one L2.
static void sort_front_by_query(DevState& d, int kind, int32_t n, hipStream_t s) {
    const int c = d.fcur[kind], o = c ^ 1;
    const bool in_tmp = radix_sort_u32_dev(d, reinterpret_cast<uint32_t*>(d.fquery[kind][c]),
                                           reinterpret_cast<int32_t*>(d.fnode[kind][c]),
                                           reinterpret_cast<uint32_t*>(d.fquery[kind][o]),
                                           reinterpret_cast<int32_t*>(d.fnode[kind][o]), d.front_cap[kind],
                                           d.fsize + 2 * kind + c, bits_for(n - 1), s);
    if (in_tmp) {
        hipMemcpyAsync(d.fsize + 2 * kind + o, d.fsize + 2 * kind + c, sizeof(uint32_t), hipMemcpyDeviceToDevice, s);
        d.fcur[kind] = o;
    }
}
void launch_query_order(DevState& d, int32_t n, hipStream_t s) {
    if (n < 2) return;
    sort_front_by_query(d, 0, n, s);
    sort_front_by_query(d, 1, n, s);
}

// Counting sort by node id (the reference's FlOrderLog::prepare + pureReorderLooseFrontsWithLog,
// FlOrderLog.cu:7-26, BvttFrontReorderKernels.cu:12-24): per-node counts, an exclusive scan
// into the bucket starts intbeg[0..n-1] (internal ids) / extbeg[0..n] (leaves), one scatter
// into the spare buffer. Lanes holding runs of one node id (fronts produced from node-ordered
// fronts keep them together) take their slots with one atomic per run. The order inside a
// bucket is that of the atomics, as in the reference.
__device__ inline uint32_t run_atomic(uint32_t* ctr, bool valid, uint32_t key) {
    const int lane = lane_id();
    const uint64_t vmask = __ballot(valid);
    const uint32_t prev = __shfl_up(key, 1);
    const bool prev_valid = lane > 0 ? ((vmask >> (lane - 1)) & 1ull) != 0 : false;
    const bool start = valid && !(prev_valid && prev == key);
    const uint64_t starts = __ballot(start);
    const uint64_t le = (2ull << lane) - 1ull;  // lanes at or below this one
    const uint64_t upto = starts & le;
    const int s0 = upto ? 63 - __clzll((long long)upto) : lane;  // this lane's run start
    uint32_t base = 0;
    if (start) {  // the run ends at the next start or the next invalid lane
        const uint64_t stop = (starts | ~vmask) & ~le;
        const int e = stop ? __ffsll((long long)stop) - 1 : 64;
        base = atomicAdd(ctr + key, (uint32_t)(e - lane));
    }
    base = __shfl(base, s0);
    return base + (uint32_t)(lane - s0);
}

// The same with every set of equal keys in the wave taken together, one round per distinct key:
// internal fronts put nodes with large subtrees into the fronts of many queries, and their
// counters would otherwise take one contended atomic per entry.
// The rounds only group the lanes: each group's lowest lane issues its atomic and keeps the old
// value, and one shuffle after the last round hands the bases out, so the atomics of all rounds
// are in flight together instead of one round trip per distinct key.
__device__ inline uint32_t match_atomic(uint32_t* ctr, bool valid, uint32_t key) {
    const int lane = lane_id();
    uint64_t todo = __ballot(valid);
    uint32_t base = 0, rank = 0;
    int lead = lane;
    while (todo) {  // wave-uniform
        const int first = __ffsll((long long)todo) - 1;
        const uint32_t k = (uint32_t)__shfl((int)key, first);
        const uint64_t grp = __ballot(key == k) & todo;
        if (lane == first) base = atomicAdd(ctr + k, (uint32_t)__popcll(grp));
        if ((grp >> lane) & 1ull) {
            lead = first;
            rank = (uint32_t)__popcll(grp & lanes_below());
        }
        todo &= ~grp;
    }
    return (uint32_t)__shfl((int)base, lead) + rank;
}
template <bool MATCH>
__device__ inline uint32_t slot_atomic(uint32_t* ctr, bool valid, uint32_t key) {
    return MATCH ? match_atomic(ctr, valid, key) : run_atomic(ctr, valid, key);
}

template <bool MATCH>
__global__ void __launch_bounds__(kBlock) k_order_count(const uint32_t* __restrict__ node, const uint32_t* size,
                                                        uint32_t cap, int32_t nb, uint32_t* __restrict__ cnt) {
    const uint32_t m = min(*size, cap);
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t k0 = blockIdx.x * blockDim.x; k0 < m; k0 += stride) {  // wave-uniform trip count
        const uint32_t k = k0 + threadIdx.x;
        const bool valid = k < m;
        const uint32_t key = valid ? min(node[k], (uint32_t)(nb - 1)) : 0u;
        slot_atomic<MATCH>(cnt, valid, key);
    }
}

// BALANCE (REORDER, internal front): inside each bucket the entries whose node does not overlap
// its query go first (slots from the bucket start up), the overlapping ones last (from the bucket
// end down), as the reference's reorderIntLooseIntraFrontsWithLog does with its back counts
// (BvttFrontReorderKernels.cu:27-63).
template <bool BALANCE, bool MATCH>
__global__ void __launch_bounds__(kBlock) k_order_scatter(DevState d, const uint32_t* __restrict__ node,
                                                          const int32_t* __restrict__ query, const uint32_t* size,
                                                          uint32_t cap, int32_t nb, const uint32_t* __restrict__ beg,
                                                          uint32_t* __restrict__ cur, uint32_t* __restrict__ back,
                                                          uint32_t* __restrict__ dst_node,
                                                          int32_t* __restrict__ dst_query, uint32_t* dst_size) {
    const uint32_t m = min(*size, cap);
    if (blockIdx.x == 0 && threadIdx.x == 0) *dst_size = m;
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t k0 = blockIdx.x * blockDim.x; k0 < m; k0 += stride) {  // wave-uniform trip count
        const uint32_t k = k0 + threadIdx.x;
        const bool valid = k < m;
        uint32_t nd = 0;
        int32_t q = 0;
        if (valid) {
            nd = node[k];
            q = query[k];
        }
        const uint32_t key = min(nd, (uint32_t)(nb - 1));
        bool ov = false;
        if (BALANCE && valid) {
            const float4 qlo = d.qleaf[q].lo, qhi = d.qleaf[q].hi;
            ov = node_overlap(d, (int32_t)key, rec_box(qlo, qhi));
        }
        const uint32_t r = slot_atomic<MATCH>(cur, valid && !ov, key);
        uint32_t o = beg[key] + r;
        if (BALANCE) {
            const uint32_t rb = slot_atomic<MATCH>(back, valid && ov, key);
            if (ov) o = beg[key + 1] - 1u - rb;
        }
        if (valid) {
            dst_node[o] = nd;
            dst_query[o] = q;
        }
    }
}

// One counting sort of a front kind by node id into its spare buffer, which becomes current;
// beg[0..nb] = bucket starts (beg[nb] = size).
static void order_front(DevState& d, int kind, int32_t nb, uint32_t* cnt, uint32_t* beg, bool balance,
                        hipStream_t s) {
    const int c = d.fcur[kind], o = c ^ 1;
    const uint32_t cap = (uint32_t)std::min<int64_t>(d.front_cap[kind], 0xFFFFFFFFll);
    const unsigned g = std::min<unsigned>(grid_for(d.front_cap[kind]), 8192u);
    fill_u32(cnt, nb, 0u, s);
    // internal fronts take equal keys per wave together, external ones (leaves near each query,
    // few repeats) per run of equal neighbours
    if (kind == 0)
        hipLaunchKernelGGL(k_order_count<true>, dim3(g), dim3(kBlock), 0, s, d.fnode[kind][c], d.fsize + 2 * kind + c,
                           cap, nb, cnt);
    else
        hipLaunchKernelGGL(k_order_count<false>, dim3(g), dim3(kBlock), 0, s, d.fnode[kind][c],
                           d.fsize + 2 * kind + c, cap, nb, cnt);
    launch_exscan(d, cnt, beg, nb, beg + nb, s);
    fill_u32(cnt, nb, 0u, s);
    if (balance) {
        fill_u32(d.intback, nb, 0u, s);
        hipLaunchKernelGGL((k_order_scatter<true, true>), dim3(g), dim3(kBlock), 0, s, d, d.fnode[kind][c],
                           d.fquery[kind][c], d.fsize + 2 * kind + c, cap, nb, beg, cnt, d.intback, d.fnode[kind][o],
                           d.fquery[kind][o], d.fsize + 2 * kind + o);
    } else if (kind == 0) {
        hipLaunchKernelGGL((k_order_scatter<false, true>), dim3(g), dim3(kBlock), 0, s, d, d.fnode[kind][c],
                           d.fquery[kind][c], d.fsize + 2 * kind + c, cap, nb, beg, cnt, nullptr, d.fnode[kind][o],
                           d.fquery[kind][o], d.fsize + 2 * kind + o);
    } else {
        hipLaunchKernelGGL((k_order_scatter<false, false>), dim3(g), dim3(kBlock), 0, s, d, d.fnode[kind][c],
                           d.fquery[kind][c], d.fsize + 2 * kind + c, cap, nb, beg, cnt, nullptr, d.fnode[kind][o],
                           d.fquery[kind][o], d.fsize + 2 * kind + o);
    }
    d.fcur[kind] = o;
}

// A freshly generated internal front is radix-sorted instead (3 passes of 8 bits, then the bucket
// starts by binary search): there every query's front holds the few nodes with the largest
// subtrees, and the counting sort's atomics on those nodes' counters contend even when each wave
// takes its equal keys together (measured on the folded 2M-triangle cloth, 46.8 M entries: counting
// 4.7 ms, radix 1.3 ms). So is a generated external front of a large scene: in query order hardly
// any neighbours share a leaf, so the counting sort makes two random atomics per entry (2M cloth,
// 35 M entries: 1.6 ms against 1.0 ms; GENERATE of 522k triangles 2.09 -> 1.97 ms, of 130k 0.53 against
// 0.56 ms). Fronts made by UPDATE are nearly in node order already, where the counting sort is the
// faster one for both kinds (UPDATE of the 2M cloth 3.18 ms, 3.51 with internal and 3.78 with both by
// radix).
constexpr int32_t kRadixExtMin = 1 << 18;
static void radix_order_front(DevState& d, int kind, int32_t nb, uint32_t* beg, hipStream_t s) {
    const int c = d.fcur[kind], o = c ^ 1;
    const bool in_tmp = radix_sort_u32_dev(d, d.fnode[kind][c], d.fquery[kind][c], d.fnode[kind][o], d.fquery[kind][o],
                                           d.front_cap[kind], d.fsize + 2 * kind + c, bits_for(nb - 1), s);
    if (in_tmp) {
        hipMemcpyAsync(d.fsize + 2 * kind + o, d.fsize + 2 * kind + c, sizeof(uint32_t), hipMemcpyDeviceToDevice, s);
        d.fcur[kind] = o;
    }
    const int cc = d.fcur[kind];
    hipLaunchKernelGGL(k_bucket_begin, dim3(grid_for(nb + 1)), dim3(kBlock), 0, s, d.fnode[kind][cc],
                       d.fsize + 2 * kind + cc, (uint32_t)std::min<int64_t>(d.front_cap[kind], 0xFFFFFFFFll), nb, beg);
}

void launch_order_fronts(DevState& d, int32_t n, hipStream_t s, bool generated) {
    if (generated) radix_order_front(d, 0, n - 1, d.intbeg, s);
    else order_front(d, 0, n - 1, d.intcnt, d.intbeg, false, s);
    if (generated && n >= kRadixExtMin) radix_order_front(d, 1, n, d.extbeg, s);
    else order_front(d, 1, n, d.extcnt, d.extbeg, false, s);
}

// Without node ordering, the front comes out ordered by query without a global sort: the
// production is gathered in wave order (each wave's consecutive queries keep their entries
// together, the waves following in query order), then each wave's run is sorted by query.
void launch_generate(DevState& d, int32_t n, hipStream_t s, bool order) {
    reset_step_counters(d, s);
    front_begin(d, s);
    FrontSink fi = next_sink(d, 0), fe = next_sink(d, 1);
    const int64_t nq = query_count(d, n);
    const uint32_t per = walk_queries(nq);
    const unsigned grid = nq > 0 ? walk_grid(nq) : 0u;
    const bool waves = !order && nq > 0 && wave_ordered_ok(d, (int64_t)grid * kWaves);
    if (waves) {
        record_chunks(d, fi, 0);
        record_chunks(d, fe, 1);
    }
    if (nq > 0) hipLaunchKernelGGL(k_traverse<true>, dim3(grid), dim3(kBlock), 0, s, n, per, d, fi, fe);
    if (waves) {
        front_finish_waves(d, 0, (int64_t)grid * kWaves, per, s);
        front_finish_waves(d, 1, (int64_t)grid * kWaves, per, s);
    } else {
        front_finish(d, 0, false, s);
        front_finish(d, 1, false, s);
        if (order && n >= 2) launch_order_fronts(d, n, s, true);
        if (!order) launch_query_order(d, n, s);
    }
    d.front_by_query = order ? 0 : 1;
}

// ---------------------------------------------------------------- UPDATE (prune / sprout)
// One entry per lane and loop iteration (grid-stride, so the wave's entries stay neighbours; the next
// one's words are loaded meanwhile). Pruned entries climb by the parent words beside the node
// records. An overlapping internal entry sprouts: its children go on the wave's LDS stack, from which
// every lane tests one node per round (a node that does not overlap and every leaf is an entry of the
// new front, an overlapping node pushes its children); rounds run while the stack fills the wave, the
// rest waits for more entries. Bound by the latency of the loads that follow one another, so by their
// number and the waves in flight. Against a walk per lane, parts of it handed to idle lanes, and
// climbs by the spine arrays, us: 2.6k triangles 25 -> 18, 41k 78 -> 64, 65k boxes 60 -> 48,
// 130k 89 -> 70, 2.1M 1710 -> 1340 (1860 with half as many waves).
constexpr uint32_t kSproutStack = 256, kSproutStage = 192;  // 24 resident waves per CU
__device__ inline uint32_t sprout_drain(const DevState& d, const Out& out, lds_int2* stk, lds_u32* top, uint32_t least) {
    uint32_t visits = 0;
    const int64_t limit = 64 * (2 * d.maxT + 16);
    for (int64_t rounds = 0;; ++rounds) {
        const uint32_t t = *top;
        if (t < least || t == 0) break;
        if (rounds > limit) {  // only a corrupted tree gets here (flag 16, a device error)
            if (lane_id() == 0) {
                atomicOr(&d.ctr[C_OVF], 16u);
                *top = 0;
            }
            break;
        }
        bool active;
        int32_t q = 0, enc = 0;
        desc_pop(stk, top, active, q, enc);
        const int32_t nd = enc >> 1;
        const bool leaf = enc & 1;
        bool hit = false;
        Box qb{};
        float4 hi = make_float4(0.f, 0.f, 0.f, 0.f);
        int4 tp = make_int4(0, 0, 0, 0);
        if (active) {
            const float4 qlo = d.qleaf[q].lo, qhi = d.qleaf[q].hi;
            const NodeRec* r = leaf ? &d.leaf[nd] : &d.inode[nd];
            const float4 lo = r->lo;
            hi = r->hi;
            if (!leaf) tp = d.itopo[nd];
            qb = rec_box(qlo, qhi);
            hit = box_overlap(qb, lo, hi);
            ++visits;
        }
        const bool grow = hit && !leaf;
        const bool ok_l = desc_push<kSproutStack>(stk, top, grow, q, tp.x),
                   ok_r = desc_push<kSproutStack>(stk, top, grow, q, tp.y);
        bool pair = hit && leaf;
        if (out.skip_adj && pair) pair = !faces_share_vertex(out.lfaces, q, nd);
        out.pair_push(pair, make_int2(q, nd));
        stage_push(out.fe, out.ovf, out.sb[1], out.sf[1], out.scap, active && leaf, make_int2(q, nd));
        stage_push(out.fi, out.ovf, out.sb[0], out.sf[0], out.scap, active && !leaf && !hit, make_int2(q, nd));
        if (grow && !(ok_l && ok_r)) {  // no room: this lane walks what did not fit (never a left child alone)
            visits += stackless<true>(d, out, q, qb, ok_l ? tp.y : tp.x, f2i(hi.w));
        }
    }
    return visits;
}
__global__ void __launch_bounds__(kBlock) k_update(DevState d, FrontIn in, FrontSink fi, FrontSink fe) {
    __shared__ StagesT<kSproutStage> st;
    __shared__ DescStack<kWaves, kSproutStack> ds;
    stages_init(st);
    const int w = threadIdx.x >> 6;
    if (lane_id() == 0) ds.top[w] = 0;
    lds_int2* stk = (lds_int2*)ds.item[w];
    lds_u32* top = (lds_u32*)&ds.top[w];
    const Out out = make_out(st, fi, fe, d);
    const uint32_t ni = min(*in.size[0], in.cap[0]), ne = min(*in.size[1], in.cap[1]), total = ni + ne;
    const uint32_t stride = gridDim.x * blockDim.x;
    uint32_t visits = 0;
    int32_t qn = 0, xn = 0;  // the next iteration's entry, loaded while this one's records are
    auto load_entry = [&](uint32_t k) {
        if (k >= total) return;
        qn = k < ni ? in.query[0][k] : in.query[1][k - ni];
        xn = (int32_t)(k < ni ? in.node[0][k] : in.node[1][k - ni]);
    };
    const uint32_t first = blockIdx.x * blockDim.x + threadIdx.x;
    load_entry(first);
    // wave-uniform trip count: every lane of a wave takes part in the sprout rounds
    for (uint32_t k = first; k - lane_id() < total; k += stride) {
        const bool valid = k < total, internal = k < ni;
        const int32_t q = qn, x = xn;
        Box b{};
        bool hit = false, climb = false;
        int32_t node = x;  // climbing: a node that does not overlap, and its topology
        int4 tp = make_int4(0, 0, 0, 0);
        if (valid) {
            const float4 qlo = d.qleaf[q].lo, qhi = d.qleaf[q].hi;
            const NodeRec* r = internal ? &d.inode[x] : &d.leaf[x];
            const float4 lo = r->lo, hi = r->hi;
            if (internal) tp = d.itopo[x];
            b = rec_box(qlo, qhi);
            hit = box_overlap(b, lo, hi);
            climb = internal && !hit;
            if (!internal) node = f2i(lo.w);  // the leaf's parent
            ++visits;
        }
        load_entry(k + stride);
        bool ext = valid && !internal && hit;
        bool pair = ext;
        if (out.skip_adj && pair) pair = !faces_share_vertex(out.lfaces, q, x);
        if (valid && !internal && !hit && node < 0) ext = true;  // the only leaf: the root's entry stays
        else if (valid && !internal && !hit) {
            const bool right = (d.leaf_mark[x] & 4u) != 0u;
            const int4 pt = d.itopo[node];
            ++visits;
            ext = node_overlap(d, node, b);
            climb = !ext && !right;  // a right child's left sibling's entry climbs
            tp = pt;
        }
        // prune: climb while the parent does not overlap either
        bool keep = false;
        while (climb) {
            const int32_t par = tp.z >> 1;
            if (par < 0) {
                keep = true;
                break;
            }
            const int4 pt = d.itopo[par];
            ++visits;
            keep = node_overlap(d, par, b);
            if (keep || (tp.z & 1)) break;  // from a right child: a left sibling's entry covers the parent
            node = par;
            tp = pt;
        }
        out.pair_push(pair, make_int2(q, x));
        stage_push(out.fe, out.ovf, out.sb[1], out.sf[1], out.scap, ext, make_int2(q, x));
        stage_push(out.fi, out.ovf, out.sb[0], out.sf[0], out.scap, keep, make_int2(q, node));
        // sprout: less than 64 items are left from before, so 128 more fit
        desc_push<kSproutStack>(stk, top, internal && hit, q, tp.x);
        desc_push<kSproutStack>(stk, top, internal && hit, q, tp.y);
        visits += sprout_drain(d, out, stk, top, 64u);
    }
    visits += sprout_drain(d, out, stk, top, 1u);
    out.final_flush();
    add_visits(d, visits);
}

// checkFrontQuality: uses the offsets of the previous ordering (intbeg/extbeg) and the snapshot.
__global__ void __launch_bounds__(kBlock) k_quality(int32_t n, DevState d) {
    const int32_t I = n - 1;
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= I) return;
    const int32_t x = d.int_rx[i], y = d.int_ry[i];
    const int intCnt = (int)(d.intbeg[i + y - x] - d.intbeg[i]);
    const int extCnt = (int)(d.extbeg[y + 1] - d.extbeg[x]);
    const float snap1 = d.snapshot[i] + 1.0f;  // a float sum, as in the reference expression
    if (1.0 * intCnt / extCnt > (double)snap1 - 0.7 * intCnt / (double)d.intbeg[I]) {
        atomicAdd(&d.intrange[i], 1);
        atomicAdd(&d.intrange[i + y - x], -1);
        atomicMin(&d.rtroot[x], i);
    }
}

__global__ void __launch_bounds__(kBlock) k_snapshot(int32_t n, DevState d) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int32_t x = d.int_rx[i], y = d.int_ry[i];
    const uint32_t ic = d.intbeg[i + y - x] - d.intbeg[i];
    const uint32_t ec = d.extbeg[y + 1] - d.extbeg[x];
    d.snapshot[i] = (float)(1.0 * ic / (double)(ec + 1u));
}

void launch_snapshot(DevState& d, int32_t n, hipStream_t s) {
    if (n >= 2) hipLaunchKernelGGL(k_snapshot, dim3(grid_for(n - 1)), dim3(kBlock), 0, s, n, d);
}

void launch_update(DevState& d, int32_t n, int quality, hipStream_t s, bool order) {
    if (!order) quality = 0;  // the quality check reads the ordering's bucket offsets
    reset_step_counters(d, s);
    front_begin(d, s);
    const FrontIn in = cur_front(d);
    FrontSink fi = next_sink(d, 0), fe = next_sink(d, 1);
    hipLaunchKernelGGL(k_update, dim3(stream_grid()), dim3(kBlock), 0, s, d, in, fi, fe);
    front_finish(d, 0, false, s);  // into the input buffers, which k_update is done with
    front_finish(d, 1, false, s);
    if (quality && n >= 2) {
        hipMemsetAsync(d.intrange, 0, sizeof(int32_t) * n, s);
        fill_i32(d.rtroot, n, INT32_MAX, s);
        hipLaunchKernelGGL(k_quality, dim3(grid_for(n - 1)), dim3(kBlock), 0, s, n, d);
    }
    if (order && n >= 2) launch_order_fronts(d, n, s, false);
    if (!order) launch_query_order(d, n, s);
    d.front_by_query = order ? 0 : 1;
}

// ---------------------------------------------------------------- KEEP
// Descents below internal front entries that now overlap their query are shared by the wave:
// instead of one lane walking a subtree while the others wait, the (query, node) pairs still to
// be tested go on a per-wave LDS stack and every lane takes one per round (a round is one
// dependent load: the node's record, and for an overlapping internal node its children). The
// nodes tested and the pairs found are those of the lane's own walk; a stack that is full
// leaves the lane to walk that subtree itself.
// Tests node `enc` against q's box: an overlapping leaf is a pair, an overlapping internal node
// pushes its two children (or, without room, is walked by this lane). Returns the node tests.
__device__ inline uint32_t desc_test(const DevState& d, const Out& out, lds_int2* stk, lds_u32* top,
                                     bool active, int32_t q, int32_t enc) {
    uint32_t visits = 0;
    bool leaf_hit = false, int_hit = false;
    int32_t nd = enc >> 1;
    Box qb{};
    float4 hi = make_float4(0.f, 0.f, 0.f, 0.f);
    if (active) {
        const float4 qlo = d.qleaf[q].lo, qhi = d.qleaf[q].hi;
        qb = rec_box(qlo, qhi);
        const NodeRec* r = (enc & 1) ? &d.leaf[nd] : &d.inode[nd];
        const float4 lo = r->lo;
        hi = r->hi;
        ++visits;
        const bool hit = box_overlap(qb, lo, hi);
        leaf_hit = hit && (enc & 1);
        int_hit = hit && !(enc & 1);
    }
    bool emit = leaf_hit;
    if (out.skip_adj && emit) emit = !faces_share_vertex(out.lfaces, q, nd);
    out.pair_push(emit, make_int2(q, nd));
    int4 tp = make_int4(0, 0, 0, 0);
    if (int_hit) tp = d.itopo[nd];
    const int32_t lc = tp.x, rc = tp.y;
    const bool ok_l = desc_push(stk, top, int_hit, q, lc);
    const bool ok_r = desc_push(stk, top, int_hit, q, rc);
    if (int_hit && !(ok_l && ok_r)) {  // no room: walk what did not fit here (one call site)
        int32_t start = lc, end = f2i(hi.w);  // both children: nd's subtree below nd
        if (ok_l) start = rc;                 // the right child alone
        else if (ok_r) end = (lc & 1) ? d.leaf_lca[(lc >> 1) + 1] : f2i(d.inode[lc >> 1].hi.w);  // the left alone
        visits += stackless<false>(d, out, q, qb, start, end);
    }
    return visits;
}

// Works the wave's stack off, one item per lane and round, while it holds at least `least` items
// (64 between loop iterations: only full rounds, the rest waits for more; 1 at the end). Called
// by all active lanes.
__device__ inline uint32_t desc_drain(const DevState& d, const Out& out, lds_int2* stk, lds_u32* top,
                                      uint32_t least) {
    uint32_t visits = 0;
    const int lane = lane_id();
    // every node is tested at most once per query walk; the bound only guards against a
    // corrupted tree (flag 16, reported as a device error, instead of a hang)
    const int64_t limit = 2 * d.maxT + 16;
    for (int64_t rounds = 0;; ++rounds) {
        const uint32_t t = *top;
        if (t < least || t == 0) break;
        if (rounds > limit) {
            if (lane == __ffsll((long long)__ballot(1)) - 1) {
                atomicOr(&d.ctr[C_OVF], 16u);
                *top = 0;
            }
            break;
        }
        bool active;
        int32_t q = 0, enc = 0;
        desc_pop(stk, top, active, q, enc);
        visits += desc_test(d, out, stk, top, active, q, enc);
    }
    return visits;
}

// KEEP over the current front, U entries per thread per loop iteration with all their loads issued
// together. Bound by the vector L1: a wave's load of 64 different records takes 65 cycles of its CU
// whatever the load's width, so a box in two 16-byte loads costs 130 of the 215 cycles that 64 entries
// take (74 % of the L1's cycles busy, 40 % of the VALU's). On large scenes (Q) the entries are therefore
// tested on 16-byte records, one load each, and the few that those leave open (0.2 %
// on scenes in motion), like the descents,
// on the boxes. Scenes whose coordinates coincide exactly, such as sheets of one grid on one another,
// leave many open: where the last KEEP's records left more than one entry in kOpenMost open (counted by one
// workgroup in kOpenSample), this kernel ends at once and the one without Q that is launched after it
// (otherwise) does the work; the count is handed on until a step without KEEP or REORDER clears it.
// (Both loops in one kernel: 8 % slower.) Records / boxes, us: 3.9 % open 289 / 304 (sheets of 2.1M), 1073 /
// 1209 (of 8.4M); 4.4 % 193 / 197 (cloth of 1.3M), 288 / 331 (of 2.1M); 4.6 % 297 / 305; 5.8 % 305 / 304; 6.3
// % 1179 / 1204; 7.6 % 322 / 301; 8.4 % 1244 / 1212; 13 % 388 / 318. KEEP, us, boxes -> Q: 2.1M triangles
// 432..646 -> 365..596 over ten frames of a front, sheets of 2.9M 375 -> 265, of 8.4M 1150 -> 1033 (without
// shared-vertex pairs) and 937 -> 745; the refit that writes the records takes 16 us (2.1M) and 68 us (8.4M)
// longer. Below a million triangles the gain is within that cost.
// implicit: the current front's shared-vertex head (C_ADJ entries after the last partition) is
// not tested when the last refit found every coordinate finite: its pairs are broad-phase hits
// whatever the positions (both boxes hold the shared vertex) and are counted, not listed.
// W = waves per workgroup (the tuner picks it with the grid and U).
template <int U, int W, bool Q>
__global__ void __launch_bounds__(64 * W) k_keep(DevState d, FrontIn in, int implicit, int otherwise) {
    __shared__ StagesBPT<W> st;
    __shared__ DescStack<W> ds;
    stages_init(st);
    const int w = threadIdx.x >> 6;
    if (lane_id() == 0) ds.top[w] = 0;
    lds_int2* stk = (lds_int2*)ds.item[w];
    lds_u32* stop = (lds_u32*)&ds.top[w];
    const Out out = make_out(st, d);
    uint32_t ni = min(*in.size[0], in.cap[0]), ne = min(*in.size[1], in.cap[1]);
    // with skip_adj the head's pairs are filtered out anyway: skipped and not counted
    const uint32_t head = implicit ? min(d.ctr[C_ADJ], ne) : 0u;
    const uint32_t skip = d.skip_adj || d.ctr[C_NO_IMPLICIT] == 0u ? head : 0u;
    ne -= skip;
    const uint32_t total = ni + ne;
    if (Q || otherwise) {  // the boxes at once: see below
        const uint32_t open = d.ctr[C_KEEP_OPEN];
        const bool boxes = open > total / (kOpenMost * kOpenSample);
        if (Q && boxes && blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(d.pcnt + kOpenWord, open);
        if (Q == boxes) return;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) d.ctr[C_IMPLICIT] = d.skip_adj ? 0u : skip;
    const uint32_t* ext_node = in.node[1] + skip;
    const int32_t* ext_query = in.query[1] + skip;
    uint32_t opened = 0;
    const XcdLoop it = xcd_loop(total);
    const uint32_t stride = it.stride;
    if (it.begin - threadIdx.x >= it.end) return;  // the whole workgroup lies past the end
    uint32_t visits = 0;
    // entries of iteration k0 into (q, nd); -1 past the end
    auto load_entries = [&](uint32_t k0, int32_t* q, int32_t* nd) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t k = k0 + u * stride;
            q[u] = -1;
            nd[u] = 0;
            if (k >= it.end) continue;
            if (k < ni) {
                q[u] = in.query[0][k];
                nd[u] = (int32_t)in.node[0][k];
            } else {
                q[u] = ext_query[k - ni];
                nd[u] = (int32_t)ext_node[k - ni];
            }
        }
    };
    // software pipeline: the next iteration's entries are loaded while this one's node records
    // are in flight, so each iteration waits for one round trip instead of two
    int32_t qn[U], ndn[U];
    load_entries(it.begin, qn, ndn);
    // one loop iteration: test the entries, push the children of now-overlapping nodes, stage pairs
    auto keep_step = [&](uint32_t k0) {
        int32_t q[U], nd[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            q[u] = qn[u];
            nd[u] = ndn[u];
        }
        float4 qlo[Q ? 1 : U], qhi[Q ? 1 : U], lo[Q ? 1 : U], hi[Q ? 1 : U];
        ulonglong2 qa[Q ? U : 1], na[Q ? U : 1];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool internal = k0 + u * stride < ni;
            if (Q) {
                qa[u] = na[u] = make_ulonglong2(0ull, 0ull);
                if (q[u] >= 0) {
                    qa[u] = d.qleafrec[q[u]];
                    na[u] = internal ? d.qnode[nd[u]] : d.qleafrec[nd[u]];
                }
                continue;
            }
            qlo[u] = qhi[u] = lo[u] = hi[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (q[u] >= 0) {
                const NodeRec* r = internal ? &d.inode[nd[u]] : &d.leaf[nd[u]];
                qlo[u] = d.qleaf[q[u]].lo;
                qhi[u] = d.qleaf[q[u]].hi;
                lo[u] = r->lo;
                hi[u] = r->hi;
            }
        }
        load_entries(k0 + U * stride, qn, ndn);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool internal = k0 + u * stride < ni;
            bool hit;
            if (Q) {  // where the grid can't tell, the entry itself goes on the stack for a test of the boxes
                bool open;
                hit = q[u] >= 0 && !q_apart(qa[u], na[u], open);
                const bool later = hit && open;
                opened += later ? 1u : 0u;
                if (!desc_push(stk, stop, later, q[u], nd[u] << 1 | (internal ? 0 : 1))) {  // no room: here
                    const NodeRec *a = &d.qleaf[q[u]], *b = internal ? &d.inode[nd[u]] : &d.leaf[nd[u]];
                    hit = box_overlap(rec_box(a->lo, a->hi), b->lo, b->hi);
                    ++visits;
                } else {
                    hit = hit && !open;
                    visits += q[u] >= 0 && !later ? 1u : 0u;  // an open entry's is counted with its boxes
                }
            } else {
                hit = q[u] >= 0 && box_overlap(rec_box(qlo[u], qhi[u]), lo[u], hi[u]);
                visits += q[u] >= 0 ? 1u : 0u;
            }
            // the node now overlaps: its children go on the wave's stack
            const bool desc = internal && hit;
            int4 tp = make_int4(0, 0, 0, 0);
            if (desc) tp = d.itopo[nd[u]];
            const int32_t lc = tp.x, rc = tp.y;
            const bool ok_l = desc_push(stk, stop, desc, q[u], lc);
            const bool ok_r = desc_push(stk, stop, desc, q[u], rc);
            if (desc && !(ok_l && ok_r)) {  // no room on the stack: this lane walks the subtree
                const int32_t start = ok_l ? rc : lc;
                const float4 a = d.qleaf[q[u]].lo, b = d.qleaf[q[u]].hi;
                visits += stackless<false>(d, out, q[u], rec_box(a, b), start, f2i(d.inode[nd[u]].hi.w));
            }
            bool emit = hit && !internal;
            if (out.skip_adj && emit) emit = !faces_share_vertex(out.lfaces, q[u], nd[u]);
            out.pair_push(emit, make_int2(q[u], nd[u]));
        }
    };
    // The wave stays in the loop until all its lanes are past the end (their entries read as
    // -1), so every drain of the stack runs with the whole wave, from one call site.
    for (uint32_t k0 = it.begin;; k0 += U * stride) {
        const bool last = __ballot(k0 < it.end) == 0;
        if (!last) keep_step(k0);
        visits += desc_drain(d, out, stk, stop, last ? 1u : 64u);
        if (last) break;
    }
    out.pair_final();
    if (Q && blockIdx.x / kXcds % kOpenSample == 0) {
        for (int off = 32; off > 0; off >>= 1) opened += __shfl_xor(opened, off);
        if (lane_id() == 0 && opened)
            atomicAdd(d.pcnt + (blockIdx.x * W + w) % kPairSegs * kCntStride + kOpenWord, opened);
    }
    add_visits(d, visits);
}

// ---------------------------------------------------------------- shared-vertex partition
// Reorders the current external front into [entries whose two triangles share a vertex | the rest]
// and leaves the head's length in C_ADJ; run by KEEP once per front version. One pass: a workgroup
// flags its tile (flags in registers), takes the tile's places with one atomic, the head's from the
// front's start and the rest's from its end, and reads the entries again to place them. A tile keeps
// its order; tiles follow one another about as they are dispatched. Bound by the faces gathered per
// entry (both triangles'), once. The tiles' atomics follow one another, about 30 per us, so that large
// scenes take tiles of 16384 entries, by 1024 threads: the 2M cloth's 35M entries 0.29 -> 0.22 ms against
// 256 threads with four times the rounds, 0.25 ms with tiles of 4096; 8.4M sheets' 74M 0.52 -> 0.43 ms.
// (Counting, a scan and a scatter, each entry tested twice: 0.30 ms; 41k triangles 40 us, here 17.)
constexpr int kAdjItems = 16;  // entries per thread
template <int W>
__global__ void __launch_bounds__(64 * W) k_adj_partition(DevState d, FrontIn in, uint32_t* __restrict__ dst_node,
                                                          int32_t* __restrict__ dst_query, uint32_t* dst_size) {
    constexpr int ITEMS = kAdjItems, B = 64 * W;
    static_assert(ITEMS * W % 64 == 0, "whole waves of counts");
    __shared__ uint32_t cnt[ITEMS * W];  // flagged entries before each round's wave
    __shared__ uint32_t base_head, base_rest;
    const uint32_t ne = min(*in.size[1], in.cap[1]);
    if (blockIdx.x == 0 && threadIdx.x == 0) *dst_size = ne;
    const uint64_t b0 = (uint64_t)blockIdx.x * (B * ITEMS);
    if (b0 >= ne) return;  // block-uniform
    const uint32_t left = (uint32_t)min<uint64_t>(ne - b0, B * ITEMS);  // the tile's entries
    const uint32_t* node = in.node[1] + b0;
    const int32_t* query = in.query[1] + b0;
    const int w = threadIdx.x >> 6;
    uint64_t flags = 0;
#pragma unroll 4
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = r * B + threadIdx.x;
        const bool adj = i < left && leaves_share_vertex(d, query[i], (int32_t)node[i]);
        flags |= adj ? 1ull << r : 0ull;
        const uint64_t m = __ballot(adj);
        if (lane_id() == 0) cnt[r * W + w] = (uint32_t)__popcll(m);
    }
    __syncthreads();
    if (threadIdx.x < 64) {  // exclusive scan of the counts
        uint32_t carry = 0;
        for (int g = 0; g < ITEMS * W; g += 64) {
            const uint32_t v = cnt[g + threadIdx.x];
            uint32_t x = v;
            for (int off = 1; off < 64; off <<= 1) {
                const uint32_t y = __shfl_up(x, off);
                if ((int)threadIdx.x >= off) x += y;
            }
            cnt[g + threadIdx.x] = carry + x - v;
            carry += __shfl(x, 63);
        }
        if (threadIdx.x == 0) {
            const unsigned long long old =
                atomicAdd(reinterpret_cast<unsigned long long*>(d.ctr + C_ADJ),
                          (unsigned long long)carry | (unsigned long long)(left - carry) << 32);
            base_head = (uint32_t)old;
            base_rest = ne - (uint32_t)(old >> 32) - (left - carry);
        }
    }
    __syncthreads();
#pragma unroll 4
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = r * B + threadIdx.x;
        const bool adj = (flags >> r) & 1ull;
        const uint64_t m = __ballot(adj);
        if (i >= left) continue;
        const uint32_t before = cnt[r * W + w] + (uint32_t)__popcll(m & lanes_below());  // flagged ones
        const uint32_t o = adj ? base_head + before : base_rest + (i - before);
        dst_node[o] = node[i];
        dst_query[o] = query[i];
    }
}

void launch_adj_partition(DevState& d, int32_t n, hipStream_t s) {
    const FrontIn in = cur_front(d);
    const int nb = d.fcur[1] ^ 1;
    fill_u32(d.ctr + C_ADJ, 2, 0u, s);
    // tiles of 16384 entries on large scenes: the tiles' atomics follow one another
    const int64_t waves = (d.front_cap[1] + 64 * kAdjItems - 1) / (64 * kAdjItems);
    if (n > (1 << 19))
        hipLaunchKernelGGL(k_adj_partition<16>, dim3(grid_for(waves, 16)), dim3(1024), 0, s, d, in, d.fnode[1][nb],
                           d.fquery[1][nb], d.fsize + 2 + nb);
    else
        hipLaunchKernelGGL(k_adj_partition<4>, dim3(grid_for(waves, 4)), dim3(256), 0, s, d, in, d.fnode[1][nb],
                           d.fquery[1][nb], d.fsize + 2 + nb);
    d.fcur[1] = nb;
    d.adj_version = d.front_version;
}

// sh: a launch shape (make_shape); the shapes' unrolls and workgroup sizes are all instantiated.
template <bool Q>
static void keep_in_shape(unsigned sh, const DevState& d, const FrontIn& in, int implicit, int otherwise, hipStream_t s) {
    const unsigned g = shape_grid(sh), w = shape_waves(sh);
#define BVHCD_KEEP(U, W) hipLaunchKernelGGL((k_keep<U, W, Q>), dim3(g), dim3(64 * W), 0, s, d, in, implicit, otherwise)
    switch (shape_unroll(sh) * 16 + w) {
        case 4 * 16 + 8: BVHCD_KEEP(4, 8); break;
        case 4 * 16 + 2: BVHCD_KEEP(4, 2); break;
        case 4 * 16 + 4: BVHCD_KEEP(4, 4); break;
        case 2 * 16 + 8: BVHCD_KEEP(2, 8); break;
        case 2 * 16 + 2: BVHCD_KEEP(2, 2); break;
        case 2 * 16 + 4: BVHCD_KEEP(2, 4); break;
        case 1 * 16 + 8: BVHCD_KEEP(1, 8); break;
        case 1 * 16 + 2: BVHCD_KEEP(1, 2); break;
        default: BVHCD_KEEP(1, 4); break;
    }
#undef BVHCD_KEEP
}

void launch_keep(DevState& d, int32_t n, hipStream_t s, bool counters_zeroed) {
    // inter-object fronts pair triangles of two objects: no shared vertices, no partition
    const int implicit = d.inter ? 0 : 1;
    if (implicit && d.adj_version != d.front_version) launch_adj_partition(d, n, s);
    if (!counters_zeroed) reset_step_counters(d, s);
    const unsigned sh = tuned_shape(TK_KEEP, n, d.inter ? d.nq : 0);
    const FrontIn in = cur_front(d);
    if (keeps_on_records(d, n)) {
        const bool set = shape_set(TK_KEEP, n), large = n > 1 << 22;
        keep_in_shape<true>(!set && large ? make_shape(16384u, 2u, 4u) : sh, d, in, implicit, 0, s);
        // The boxes, where the records left too much open: in the tuned shape too, so that tuning times the
        // kernel that does the work and a shape that is set holds for both. Untuned, up to 2^22 triangles
        // one resident set of workgroups, as it mostly ends at once (8.4M sheets on the boxes 1281 us, and
        // 1167 in the boxes' own shape, which costs 8 where the records do the work).
        keep_in_shape<false>(set || large ? sh : make_shape(1536u, 2u), d, in, implicit, 1, s);
    } else {
        keep_in_shape<false>(sh, d, in, implicit, 0, s);
    }
}

// ---------------------------------------------------------------- incremental front restructure
// The intent of BvttFrontLooseIntra::restructure (collision/bvtt_front/BvttFrontLooseIntra.cu:330-400,
// separateFronts :172-211, BvttFrontRestructureKernels.cu:12-90; unreachable in the shipped
// intra path): after a subtree rebuild keep the front entries it does not touch and re-walk
// only what it invalidates, instead of regenerating the whole front.
// Each query's front is a cut of the leaves to its right. For a rebuilt subtree R, leaves [a, b]:
//  * an entry strictly inside R of a query outside [a, b] is one piece of that query's cut of R;
//    the piece whose leftmost leaf is a becomes the walk (query, R), the others are dropped;
//  * an entry strictly inside R of a query inside [a, b] is dropped; that query's part inside
//    R is re-walked from lca[q + 1] to R's escape lca[b + 1];
//  * all other entries (outside every rebuilt subtree, at an ancestor, or at R) stay.
// Classification runs on the old topology (rt_of_leaf and the old rangex), before emission.
__global__ void __launch_bounds__(kBlock) k_restr_classify(DevState d, FrontIn in, FrontSink fi, FrontSink fe,
                                                           PairSink tasks) {
    __shared__ Stages st;
    stages_init(st);
    const Out out = make_out(st, fi, fe, d);
    const uint32_t ni = min(*in.size[0], in.cap[0]), ne = min(*in.size[1], in.cap[1]), total = ni + ne;
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < total; k += gridDim.x * blockDim.x) {
        bool task = false;
        int32_t q, r;
        if (k < ni) {
            q = in.query[0][k];
            const int32_t x = (int32_t)in.node[0][k];
            const int32_t lx = d.int_rx[x];
            r = d.rt_of_leaf[lx];
            const bool inside = r >= 0 && x > r;  // x < r: an ancestor of r
            stage_push(fi, out.ovf, out.sb[0], out.sf[0], out.scap, !inside, make_int2(q, x));
            task = inside && d.rt_of_leaf[q] != r && lx == d.int_rx[r];
        } else {
            q = in.query[1][k - ni];
            const int32_t j = (int32_t)in.node[1][k - ni];
            r = d.rt_of_leaf[j];
            const bool inside = r >= 0;
            stage_push(fe, out.ovf, out.sb[1], out.sf[1], out.scap, !inside, make_int2(q, j));
            task = inside && d.rt_of_leaf[q] != r && j == d.int_rx[r];
        }
        stage_push(tasks, out.ovf, out.sb[2], out.sf[2], out.scap, task, make_int2(q, r));
    }
    stage_final(fi, out.ovf, out.sb[0], out.sf[0]);
    stage_final(fe, out.ovf, out.sb[1], out.sf[1]);
    stage_final(tasks, out.ovf, out.sb[2], out.sf[2]);
}

void launch_front_restr_prepare(DevState& d, int32_t n, hipStream_t s) {
    front_begin(d, s);
    const FrontIn in = cur_front(d);
    FrontSink fi = next_sink(d, 0), fe = next_sink(d, 1);
    hipMemsetAsync(d.ctr + C_TASKS, 0, sizeof(uint32_t), s);
    // walks beyond the capacity are counted, not written (ovf bit 0): the caller compares
    // the count with the capacity and regenerates the front instead
    const PairSink tasks{d.ctr + C_TASKS, d.rtasks, (uint32_t)std::min<int64_t>(d.rtask_cap, 0xFFFFFFFFll), 0u};
    if (n >= 2) hipLaunchKernelGGL(k_restr_classify, dim3(stream_grid()), dim3(kBlock), 0, s, d, in, fi, fe, tasks);
    front_finish(d, 0, false, s);
    front_finish(d, 1, false, s);
}

// Walks of the repaired front: (query, rebuilt root) walks first, then every query inside a
// rebuilt run walks its part of that run. Entries append after the kept ones.
__global__ void __launch_bounds__(kBlock) k_restr_walk(DevState d, uint32_t ntasks, int32_t n, FrontSink fi,
                                                       FrontSink fe) {
    __shared__ Stages st;
    stages_init(st);
    const Out out = make_out(st, fi, fe, d);
    const uint32_t total = ntasks + (uint32_t)n;
    uint32_t visits = 0;
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < total; k += gridDim.x * blockDim.x) {
        int32_t q, start, stop;
        if (k < ntasks) {
            const int2 t = d.rtasks[k];
            q = t.x;
            start = t.y << 1;
            stop = d.leaf_lca[d.int_ry[t.y] + 1];
        } else {
            q = (int32_t)(k - ntasks);
            const int32_t r = d.rt_of_leaf[q];
            if (r < 0) continue;
            const int32_t b = d.int_ry[r];
            if (q >= b) continue;
            start = d.leaf_lca[q + 1];
            stop = d.leaf_lca[b + 1];
        }
        const float4 lo = d.leaf[q].lo, hi = d.leaf[q].hi;
        visits += stackless<true>(d, out, q, rec_box(lo, hi), start, stop);
    }
    out.final_flush();
    add_visits(d, visits);
}

void launch_front_restr_apply(DevState& d, int32_t n, uint32_t ntasks, hipStream_t s) {
    reset_step_counters(d, s);
    if (n < 2) return;
    // pairs of the kept entries (KEEP over the kept part only)
    hipMemcpyAsync(d.ctr + C_KEPT_I, d.fsize + d.fcur[0], sizeof(uint32_t), hipMemcpyDeviceToDevice, s);
    hipMemcpyAsync(d.ctr + C_KEPT_E, d.fsize + 2 + d.fcur[1], sizeof(uint32_t), hipMemcpyDeviceToDevice, s);
    FrontIn kept = cur_front(d);
    kept.size[0] = d.ctr + C_KEPT_I;
    kept.size[1] = d.ctr + C_KEPT_E;
    hipLaunchKernelGGL((k_keep<1, kWaves, false>), dim3(stream_grid()), dim3(kBlock), 0, s, d, kept, 0, 0);
    // the walks write segments into the spare buffers, then append after the kept entries
    front_begin(d, s);
    FrontSink fi = next_sink(d, 0), fe = next_sink(d, 1);
    hipLaunchKernelGGL(k_restr_walk, dim3(stream_grid()), dim3(kBlock), 0, s, d, ntasks, n, fi, fe);
    front_finish(d, 0, true, s);
    front_finish(d, 1, true, s);
}

// ---------------------------------------------------------------- REORDER (balance)
// Pairs as in KEEP from the unchanged cut; then the internal front is counting-sorted by node
// with each bucket's non-overlapping entries first. Its bucket starts go to scratch (`cursor`):
// intbeg keeps the last ordering's offsets, which the quality check reads (the front need not
// have been node-ordered since: an incremental restructure appends entries).
void launch_reorder(DevState& d, int32_t n, hipStream_t s, bool counters_zeroed) {
    launch_keep(d, n, s, counters_zeroed);
    if (n < 2) return;
    order_front(d, 0, n - 1, d.intcnt, d.cursor, true, s);
}

// ---------------------------------------------------------------- restructure decision
// intmark = inclusive scan of intrange; outermost flagged roots are rtroot[x] with intmark 1.
__global__ void k_intmark_fix(int32_t I, const int32_t* __restrict__ intrange, int32_t* __restrict__ intmark) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < I) intmark[i] += intrange[i];
}
__global__ void k_select_roots(int32_t n, DevState d) {
    const int32_t x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= n) return;
    const int32_t r = d.rtroot[x];
    if (r != INT32_MAX && d.intmark[r] == 1) {
        const int32_t a = d.int_rx[r], b = d.int_ry[r];
        atomicAdd(&d.ctr[C_RT_SUB], 1u);
        atomicAdd(&d.ctr[C_RT_INT], (uint32_t)(b - a));
        atomicAdd(&d.ctr[C_RT_LEAF], (uint32_t)(b - a + 1));
        // difference array of (root + 1) over the leaf range
        atomicAdd(&d.r_leaf_lo[a], r + 1);
        atomicAdd(&d.r_leaf_lo[b + 1], -(r + 1));
    }
}

void launch_restr_decision(DevState& d, int32_t n, hipStream_t s) {
    const int32_t I = n - 1;
    hipMemsetAsync(d.ctr + C_RT_SUB, 0, sizeof(uint32_t) * 3, s);
    launch_exscan(d, reinterpret_cast<const uint32_t*>(d.intrange), reinterpret_cast<uint32_t*>(d.intmark), I, nullptr,
                  s);
    hipLaunchKernelGGL(k_intmark_fix, dim3(grid_for(I)), dim3(kBlock), 0, s, I, d.intrange, d.intmark);
    hipMemsetAsync(d.r_leaf_lo, 0, sizeof(int32_t) * ((size_t)n + 1), s);
    hipLaunchKernelGGL(k_select_roots, dim3(grid_for(n)), dim3(kBlock), 0, s, n, d);
}

// ---------------------------------------------------------------- narrow phase
__device__ inline float3 ld3(const float* __restrict__ v, int32_t i) {
    return make_float3(v[3 * (int64_t)i], v[3 * (int64_t)i + 1], v[3 * (int64_t)i + 2]);
}
__device__ inline float3 sub3(float3 a, float3 b) { return make_float3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ inline float3 cross3(float3 a, float3 b) {
    return make_float3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ inline float dot3(float3 a, float3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// Projections of both triangles on `ax` overlap (closed intervals).
__device__ inline bool axis_overlap(float3 ax, const float3* p, const float3* q) {
    const float P0 = dot3(ax, p[0]), P1 = dot3(ax, p[1]), P2 = dot3(ax, p[2]);
    const float Q0 = dot3(ax, q[0]), Q1 = dot3(ax, q[1]), Q2 = dot3(ax, q[2]);
    const float mx1 = fmaxf(fmaxf(P0, P1), P2), mn1 = fminf(fminf(P0, P1), P2);
    const float mx2 = fmaxf(fmaxf(Q0, Q1), Q2), mn2 = fminf(fminf(Q0, Q1), Q2);
    return !(mn1 > mx2) && !(mn2 > mx1);
}

// 17 candidate axes: two face normals, 9 edge-edge crosses, 6 in-plane edge normals.
// Coordinates are translated so that the first vertex of P is the origin.
__device__ bool sat_tri_tri(float3 P1, float3 P2, float3 P3, float3 Q1, float3 Q2, float3 Q3) {
    float3 p[3] = {make_float3(0.f, 0.f, 0.f), sub3(P2, P1), sub3(P3, P1)};
    float3 q[3] = {sub3(Q1, P1), sub3(Q2, P1), sub3(Q3, P1)};
    const float3 e[3] = {sub3(p[1], p[0]), sub3(p[2], p[1]), sub3(p[0], p[2])};
    const float3 f[3] = {sub3(q[1], q[0]), sub3(q[2], q[1]), sub3(q[0], q[2])};
    const float3 nrm = cross3(e[0], e[1]), mrm = cross3(f[0], f[1]);
    if (!axis_overlap(nrm, p, q)) return false;
    if (!axis_overlap(mrm, p, q)) return false;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (!axis_overlap(cross3(e[i], f[j]), p, q)) return false;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (!axis_overlap(cross3(e[k], nrm), p, q)) return false;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (!axis_overlap(cross3(f[k], mrm), p, q)) return false;
    return true;
}

// Narrow-phase test of a self-CD broad-phase pair of leaves `lv`; `pr` receives the pair in
// canonical order (the triangle with the lower id first, and as P of the test).
__device__ inline bool narrow_self(const int32_t* __restrict__ prim, const int32_t* __restrict__ lfaces,
                                   const uint8_t* __restrict__ finite, const float* __restrict__ verts, int2 lv,
                                   int2& pr) {
    int32_t ta = prim[lv.x], tb = prim[lv.y], la = lv.x, lb = lv.y;
    if (ta > tb) {
        const int32_t t = ta; ta = tb; tb = t;
        const int32_t l = la; la = lb; lb = l;
    }
    pr = make_int2(ta, tb);
    const int32_t* fa = lfaces + 3 * (int64_t)la;
    const int32_t* fb = lfaces + 3 * (int64_t)lb;
    const int32_t a0 = fa[0], a1 = fa[1], a2 = fa[2], b0 = fb[0], b1 = fb[1], b2 = fb[2];
    // A shared vertex has bitwise-equal translated coordinates on both sides, so while every
    // product stays finite (all |coordinates| <= 1e8) its projection lies in both intervals on
    // every axis: the SAT always reports a hit, and the test is skipped.
    const bool share = a0 == b0 || a0 == b1 || a0 == b2 || a1 == b0 || a1 == b1 || a1 == b2 || a2 == b0 ||
                       a2 == b1 || a2 == b2;
    if (share && finite[la] && finite[lb]) return true;
    return sat_tri_tri(ld3(verts, a0), ld3(verts, a1), ld3(verts, a2), ld3(verts, b0), ld3(verts, b1),
                       ld3(verts, b2));
}

template <int W>
__global__ void __launch_bounds__(64 * W) k_narrow(DevState d) {
    __shared__ int2 sbuf[W][kStage];
    __shared__ uint32_t sfill[W][2];
    __shared__ uint32_t pre[kPairSegs + 1];
    const int w = threadIdx.x >> 6;
    if (lane_id() == 0) {
        sfill[w][0] = 0;
        sfill[w][1] = rotor_start<W>();
    }
    const SegPairSink sink = pair_segments(d, 1, 8u);
    lds_int2* const sb = (lds_int2*)sbuf[w];
    lds_u32* const sf = (lds_u32*)sfill[w];
    const uint32_t npairs = seg_prefix(d.pcnt, (uint32_t)d.pair_seg_cap, pre);
    if (blockIdx.x * blockDim.x >= npairs) return;
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < npairs; k += gridDim.x * blockDim.x) {
        const int2 lv = d.bp[seg_slot(pre, k, d.pair_seg_cap)];  // leaves
        if (d.inter) {  // (query leaf of the other object, leaf of this tree): this tree's triangle is P
            const int32_t* fa = d.lfaces + 3 * (int64_t)lv.y;
            const int32_t* fb = d.qlfaces + 3 * (int64_t)lv.x;
            const bool hit = sat_tri_tri(ld3(d.verts, fa[0]), ld3(d.verts, fa[1]), ld3(d.verts, fa[2]),
                                         ld3(d.qverts, fb[0]), ld3(d.qverts, fb[1]), ld3(d.qverts, fb[2]));
            stage_push(sink, &d.ctr[C_OVF], sb, sf, kStage, hit,
                       make_int2(d.prim_idx[lv.y], d.qprim[lv.x]));
            continue;
        }
        int2 pr;
        const bool hit = narrow_self(d.prim_idx, d.lfaces, d.tri_finite, d.verts, lv, pr);
        stage_push(sink, &d.ctr[C_OVF], sb, sf, kStage, hit, pr);
    }
    stage_final(sink, &d.ctr[C_OVF], sb, sf);
}

void launch_narrow(DevState& d, hipStream_t s, bool counters_zeroed) {
    // kernels, not memsets: the batched frame graph records this
    if (!counters_zeroed) fill_u32(d.pcnt + kPairSegs * kCntStride, kPairSegs * kCntStride, 0u, s);
    const unsigned sh = tuned_shape(TK_NARROW, d.maxT), g = shape_grid(sh);
    switch (shape_waves(sh)) {
        case 8: hipLaunchKernelGGL(k_narrow<8>, dim3(g), dim3(512), 0, s, d); break;
        case 2: hipLaunchKernelGGL(k_narrow<2>, dim3(g), dim3(128), 0, s, d); break;
        default: hipLaunchKernelGGL(k_narrow<4>, dim3(g), dim3(256), 0, s, d); break;
    }
}

// Totals of both segmented pair lists (requested counts: what the segments hold plus what none
// took, so an overflowing list reports what it needed) and their largest segment: ctr[C_BP],
// ctr[C_NP], ctr[C_BP_SEGMAX], ctr[C_NP_SEGMAX]. Implicit (shared-vertex) pairs are added to
// both totals; with a narrow phase they are hits.
__device__ inline void pair_totals(const DevState& d, int narrow) {  // two waves, one per list
    const int kind = threadIdx.x >> 6, g = lane_id();
    const uint32_t* cnt = d.pcnt + kind * kPairSegs * kCntStride;
    uint32_t v = cnt[g * kCntStride] + (g == 0 ? cnt[kDroppedWord] : 0u), m = cnt[g * kCntStride];
    for (int off = 32; off > 0; off >>= 1) {
        v += __shfl_down(v, off);
        m = max(m, __shfl_down(m, off));
    }
    if (kind == 0) {
        uint64_t t = *visit_word(d, g);
        for (int off = 32; off > 0; off >>= 1) t += __shfl_down(t, off);
        if (g == 0) ctr64(d.ctr)[C64_VISITS] = t;
    }
    if (g == 0) {
        const uint32_t impl = d.ctr[C_IMPLICIT];
        if (kind == 1) d.ctr[C_IMPL_NP] = narrow ? impl : 0u;
        const uint32_t total = v + (kind == 0 || narrow ? impl : 0u);
        d.ctr[kind ? C_NP : C_BP] = total;
        d.ctr[kind ? C_NP_SEGMAX : C_BP_SEGMAX] = m;
        if (d.hres) {
            d.hres[kind ? H_NP : H_BP] = total;
            if (kind == 0) d.hres[H_OVF] = d.ctr[C_OVF];
        }
    }
}
__global__ void k_pair_totals(DevState d, int narrow) { pair_totals(d, narrow); }
void launch_pair_totals(DevState& d, hipStream_t s, bool narrow) {
    hipLaunchKernelGGL(k_pair_totals, dim3(1), dim3(128), 0, s, d, narrow ? 1 : 0);
}
void clear_np(DevState& d, hipStream_t s) {
    fill_u32(d.pcnt + kPairSegs * kCntStride, kPairSegs * kCntStride, 0u, s);
}

// Pair k of a list, in the virtual order [listed segments | implicit head of the external front];
// leaf-id pairs (the broad-phase list, the implicit ones) mapped to triangle ids, lower first.
__device__ inline int2 list_pair(const DevState& d, int kind, const uint32_t* pre, uint32_t listed, uint32_t k) {
    int2 p;
    if (k < listed) {
        p = (kind ? d.np : d.bp)[seg_slot(pre, k, d.pair_seg_cap)];
        if (kind == 1) return p;
    } else {
        const int c = d.fcur[1];
        p = make_int2(d.fquery[1][c][k - listed], (int32_t)d.fnode[1][c][k - listed]);
    }
    if (d.inter) return make_int2(d.prim_idx[p.y], d.qprim[p.x]);  // (this tree's triangle, query's)
    const int32_t a = d.prim_idx[p.x], b = d.prim_idx[p.y];
    return a < b ? make_int2(a, b) : make_int2(b, a);
}

// Contiguous copy of pairs [first, first + count) of a list into dst. TOTALS: the totals too, by the
// first workgroup's first two waves, and no copy after an overflow.
template <bool TOTALS>
__global__ void __launch_bounds__(kBlock) k_pair_gather(DevState d, int kind, int2* __restrict__ dst, uint64_t first,
                                                        uint64_t count, int narrow) {
    __shared__ uint32_t pre[kPairSegs + 1];
    const uint32_t listed = seg_prefix(d.pcnt + kind * kPairSegs * kCntStride, (uint32_t)d.pair_seg_cap, pre);
    const uint32_t impl = !TOTALS ? d.ctr[kind ? C_IMPL_NP : C_IMPLICIT] : kind == 0 || narrow ? d.ctr[C_IMPLICIT] : 0u;
    if (TOTALS) {
        if (blockIdx.x == 0 && threadIdx.x < 128) pair_totals(d, narrow);
        if (d.ctr[C_OVF]) return;
    }
    const uint64_t total = (uint64_t)listed + impl;
    const uint64_t end = min(first + count, total);
    for (uint64_t k = first + blockIdx.x * blockDim.x + threadIdx.x; k < end; k += gridDim.x * blockDim.x)
        dst[k - first] = list_pair(d, kind, pre, listed, (uint32_t)k);
}
void launch_pair_gather(DevState& d, int kind, int2* dst, int64_t first, int64_t count, hipStream_t s) {
    hipLaunchKernelGGL(k_pair_gather<false>, dim3(std::min(grid_for(count), 2048u)), dim3(kBlock), 0, s, d, kind, dst,
                       (uint64_t)first, (uint64_t)count, 0);
}
void launch_totals_and_gather(DevState& d, int kind, int2* dst, int64_t cap, bool narrow, hipStream_t s) {
    cap = std::min(cap, d.pair_cap + d.front_cap[1]);  // as many pairs as there can be: the grid follows it
    hipLaunchKernelGGL(k_pair_gather<true>, dim3(std::min(grid_for(cap), 2048u)), dim3(kBlock), 0, s, d, kind, dst,
                       (uint64_t)0, (uint64_t)cap, narrow ? 1 : 0);
}

// ---------------------------------------------------------------- pair-set digest
__device__ inline uint64_t mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__global__ void __launch_bounds__(kBlock) k_digest(DevState d, int kind, uint64_t* out) {
    __shared__ uint32_t pre[kPairSegs + 1];
    const uint32_t listed = seg_prefix(d.pcnt + kind * kPairSegs * kCntStride, (uint32_t)d.pair_seg_cap, pre);
    const uint32_t n = listed + d.ctr[kind ? C_IMPL_NP : C_IMPLICIT];
    uint64_t acc = 0;
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const int2 p = list_pair(d, kind, pre, listed, k);
        acc += mix64(((uint64_t)(uint32_t)p.x << 32) | (uint32_t)p.y);
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off);
    if (lane_id() == 0 && acc) atomicAdd((unsigned long long*)out, (unsigned long long)acc);
}

void launch_digest(DevState& d, int filtered, hipStream_t s) {
    uint64_t* out = ctr64(d.ctr) + C64_DIGEST;
    fill_u32(reinterpret_cast<uint32_t*>(out), 2, 0u, s);
    hipLaunchKernelGGL(k_digest, dim3(1024), dim3(kBlock), 0, s, d, filtered ? 1 : 0, out);
}

}  // namespace bvhcd
