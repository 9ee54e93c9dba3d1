// Full-vocabulary sampling: the reference's slow path (Sampler.cs:41-95), BuildFilteredDistribution
// (:118-163), GreedyWithHistoryPenalties (:421-437), SampleFromDistribution (:564-576) and
// ResampleResidual (:587-618).
//
// The row is materialised in an fp32 work row exactly as the reference copies it, and every stage is
// one pass of a 1024-thread workgroup over that row.  All running sums that the reference evaluates
// left to right go through the exact evaluator in sr_seqsum.h, so probabilities, cut-offs and draws
// carry the reference's bits.
#include <algorithm>
#include <cstddef>

#include "sr_device.h"
#include "sr_kernels.h"
#include "sr_seqsum.h"
#include "sr_types.h"

namespace {

#ifdef SR_PROFILE
#define FPROF(a, slot_, i_) do { if ((a).prof && (slot_) == 0 && threadIdx.x == 0) (a).prof[(i_)] = (unsigned long long)wall_clock64(); } while (0)
// (adds the time since *t_ to stamp i_ and moves *t_ on: for the steps of a loop)
#define FPROF_ADD(a, slot_, i_, t_) do { if ((a).prof && (slot_) == 0 && threadIdx.x == 0) { const unsigned long long now_ = (unsigned long long)wall_clock64(); (a).prof[(i_)] += now_ - (t_); (t_) = now_; } } while (0)
#else
#define FPROF(a, slot_, i_) do { } while (0)
#define FPROF_ADD(a, slot_, i_, t_) do { } while (0)
#endif

constexpr int kT = SR_SEQ_THREADS;
constexpr int kW = SR_SEQ_WAVES;
constexpr int kSmall = SR_FULL_SMALL_CAP;  // survivors sorted inside the kernel
constexpr int kTagIndexBits = 19;          // a find's tag in the walk by slabs: rank << 19 | index
constexpr int kCkpt = 128;                 // tiles of a row whose running sums are kept for the search that follows

struct FullSmem {
    SrSeqSmem seq;
    SrSeq8Smem seq8;
    float lane_sum[SR_SEQ_CHAINS];
    float redf[kW];
    uint32_t redu[kW];
    int redi[kW];
    uint32_t hist[256];
    uint32_t bc[16];
    float ckpt[kCkpt];  // running sum behind every tile of a row's exact sum (SeqMarks)
    float segst[SR_SEG_MAX];  // running sum behind every segment of a prepared row (seg_walk)
    uint32_t segbc[4];
    alignas(16) unsigned long long sortbuf[kSmall];  // (cut_unsorted's tables lie here and are read by vectors of 16 bytes)
    float sprob[kSmall];
    uint32_t tags[kSmall];
    double u;  // the row's uniform (k_full_row)
};
static_assert(offsetof(FullSmem, sortbuf) % 16 == 0 && alignof(FullSmem) % 16 == 0, "whole vectors");

// SR_OUT_AMBIGUOUS of the row at work: any thread that sees a cut or the draw land on its boundary (sr_near /
// sr_stop_near) stores here; the row's flags are written behind a barrier that follows.
#define SR_AMB_WORD 15
#define SR_AMB_IF(cond_) do { if (cond_) sm.bc[SR_AMB_WORD] = 1u; } while (0)

// ---- block reductions ------------------------------------------------------------------------------
__device__ __forceinline__ float blk_max_f(float v, bool* any_nan, FullSmem& sm)
{
    // NaN propagates (TensorPrimitives.Max)
    uint32_t nanf = (v != v) ? 1u : 0u;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        float w = __shfl_xor(v, o);
        uint32_t wn = __shfl_xor(nanf, o);
        v = fmaxf(v, w);
        nanf |= wn;
    }
    __syncthreads();
    if (sr_lane() == 0) { sm.redf[sr_wave_id()] = v; sm.redu[sr_wave_id()] = nanf; }
    __syncthreads();
    float m = sm.redf[0];
    uint32_t n = sm.redu[0];
#pragma unroll
    for (int w = 1; w < kW; w++) { m = fmaxf(m, sm.redf[w]); n |= sm.redu[w]; }
    *any_nan = n != 0u;
    return m;
}
__device__ __forceinline__ int blk_sum_i(int v, FullSmem& sm)
{
    v = sr_wave_sum_i32(v);
    __syncthreads();
    if (sr_lane() == 0) sm.redi[sr_wave_id()] = v;
    __syncthreads();
    int t = 0;
#pragma unroll
    for (int w = 0; w < kW; w++) t += sm.redi[w];
    return t;
}
__device__ __forceinline__ unsigned long long blk_max_u64(unsigned long long v, FullSmem& sm)
{
    v = sr_wave_max_u64(v);
    __syncthreads();
    if (sr_lane() == 0) sm.sortbuf[sr_wave_id()] = v;
    __syncthreads();
    unsigned long long t = 0ull;
#pragma unroll
    for (int w = 0; w < kW; w++) t = sm.sortbuf[w] > t ? sm.sortbuf[w] : t;
    __syncthreads();
    return t;
}
// exclusive scan of one int per thread
__device__ __forceinline__ int blk_excl_scan(int v, int* total, FullSmem& sm)
{
    int incl = sr_wave_incl_scan_i32(v);
    __syncthreads();
    if (sr_lane() == SR_WAVE - 1) sm.redi[sr_wave_id()] = incl;
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kW; w++) {
        int t = sm.redi[w];
        if (w < sr_wave_id()) base += t;
        tot += t;
    }
    *total = tot;
    return base + incl - v;
}


// ---- one pass of the workgroup over a row ---------------------------------------------------------------
// Calls f(value, index) for every element, any order, with 16-byte loads (four in flight per thread) where the
// row allows it; with kWrite the value returned by f is stored back.  The caller synchronises.
template <bool kWrite, typename F>
__device__ __forceinline__ void row_pass(float* p, int n, F f)
{
    const int tid = threadIdx.x;
    const int head = min(n, (int)((4u - (unsigned)(((uintptr_t)p >> 2) & 3u)) & 3u));  // elements before 16-byte alignment
    if (tid < head) {
        const float y = f(p[tid], tid);
        if (kWrite) p[tid] = y;
    }
    float4* p4 = (float4*)(p + head);
    const int nv = (n - head) >> 2;
    auto one = [&](float4& a, int v) __attribute__((always_inline)) {
        const int i = head + 4 * v;
        a.x = f(a.x, i); a.y = f(a.y, i + 1); a.z = f(a.z, i + 2); a.w = f(a.w, i + 3);
    };
    int v = tid;
    for (; v + 3 * kT < nv; v += 4 * kT) {
        float4 a = p4[v], b = p4[v + kT], c = p4[v + 2 * kT], d = p4[v + 3 * kT];
        one(a, v); one(b, v + kT); one(c, v + 2 * kT); one(d, v + 3 * kT);
        if (kWrite) { p4[v] = a; p4[v + kT] = b; p4[v + 2 * kT] = c; p4[v + 3 * kT] = d; }
    }
    for (; v < nv; v += kT) {
        float4 a = p4[v];
        one(a, v);
        if (kWrite) p4[v] = a;
    }
    const int done = head + 4 * nv;
    if (tid < n - done) {
        const float y = f(p[done + tid], done + tid);
        if (kWrite) p[done + tid] = y;
    }
}

// ---- exact left-to-right sum over term(i), i in [0, n) ------------------------------------------------
// term(i) must be >= 0 (or +0 for "skipped").  With kSearch, stops at the first i whose running sum is
// >= target and returns it in *found (else -1).
template <bool kSearch, typename Term>
__device__ __forceinline__ float seq_sum(Term term, int n, float s0, float target, int* found, FullSmem& sm)
{
    float s = s0;
    *found = -1;
    for (int base = 0; base < n; base += SR_SEQ_TILE) {
        float x[SR_SEQ_RUN];
        const int i0 = base + (int)threadIdx.x * SR_SEQ_RUN;
#pragma unroll
        for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = (threadIdx.x < SR_SEQ_ACTIVE && i0 + j < n) ? term(i0 + j) : 0.0f;
        int f;
        sr_seq_tile<kSearch>(x, &s, target, &f, sm.seq);
        if (kSearch && f >= 0) {
            *found = base + f;
            return s;
        }
    }
    return s;
}

// The same over rows in memory.  A thread's SR_SEQ_RUN consecutive terms come in with 16-byte loads when the row
// is 16-byte aligned (one 4-byte load per term makes every load instruction of a wave touch 64 cache lines).
// The whole tiles of an aligned row are loaded kDepth - 1 tiles ahead of the tile that is scanned, into register
// sets that take turns: one workgroup has to keep that much in flight to cover the latency of memory.  Two things
// keep the loads in flight: what is loaded is turned into terms only when its tile is up, and the loop issues the
// same number of loads on every path -- behind the last tile it loads that tile again, to no effect -- because the
// compiler can wait for "all but the newest n loads" only where it can count them, and otherwise waits for all.
//   issue_fast(base, raw)  starts the loads of the whole tile whose first term is `base`, no conditions
//   issue_any(base, raw)   the same for any tile of any row (ragged end, unaligned row)
//   finish(raw, x)         the tile's terms from what was loaded
//
// A sum that is followed by a search over the same terms (residual resampling: Sampler.cs:594-614) leaves marks: the
// running sum behind every tile (SeqMarks::keep, rows of at most kCkpt tiles).  The running sum never decreases, so
// the search's answer lies in the first tile whose mark has reached the target, and the state in front of that tile is
// the mark before it: the search starts there (SeqMarks::from) instead of at the row's first term, and reads one
// tile instead of, on average, half the row.
struct SeqMarks {
    float* keep = nullptr;  // a sum writes the running sum behind tile t to keep[t]
    int from = 0;           // first tile that is looked at; s0 is the running sum in front of it
};
__device__ __forceinline__ bool seq_marks_fit(int n) { return (n + SR_SEQ_TILE - 1) / SR_SEQ_TILE <= kCkpt; }
// the tile at which a search for `target` over the marked row starts, and the running sum in front of it (*s0); behind a
// barrier that follows the sum
__device__ __forceinline__ int seq_marks_find(const float* marks, int n, float target, float* s0)
{
    const int tiles = (n + SR_SEQ_TILE - 1) / SR_SEQ_TILE;
    int t = 0;
    while (t < tiles - 1 && !(marks[t] >= target)) t++;
    *s0 = t > 0 ? marks[t - 1] : 0.0f;
    return t;
}
template <bool kSearch, int kDepth, typename Raw, typename IssueFast, typename IssueAny, typename Finish>
__device__ __forceinline__ float seq_sum_tiles(IssueFast issue_fast, IssueAny issue_any, Finish finish, bool fast_ok, int n,
                                               float s0, float target, int* found, FullSmem& sm, SeqMarks marks = SeqMarks())
{
    float s = s0;
    *found = -1;
    const int n_full = fast_ok ? n / SR_SEQ_TILE : 0;  // whole tiles, taken by the pipelined loop
    const int tb = marks.from;
    if (n_full > tb) {
        Raw r[kDepth];
#pragma unroll
        for (int k = 0; k < kDepth - 1; k++) issue_fast(min(tb + k, n_full - 1) * SR_SEQ_TILE, r[k]);
        for (int t0 = tb; t0 < n_full; t0 += kDepth) {
#pragma unroll
            for (int k = 0; k < kDepth; k++) {
                const int t = t0 + k;
                if (t >= n_full) break;
                issue_fast(min(t + kDepth - 1, n_full - 1) * SR_SEQ_TILE, r[(k + kDepth - 1) % kDepth]);
                float x[SR_SEQ_RUN];
                finish(r[k], x, t * SR_SEQ_TILE);
                int f;
                sr_seq_tile<kSearch>(x, &s, target, &f, sm.seq);
                if (kSearch && f >= 0) {
                    *found = t * SR_SEQ_TILE + f;
                    return s;
                }
                if (!kSearch && marks.keep && threadIdx.x == 0) marks.keep[t] = s;
            }
        }
    }
    for (int base = max(n_full, tb) * SR_SEQ_TILE; base < n; base += SR_SEQ_TILE) {
        Raw r;
        issue_any(base, r);
        float x[SR_SEQ_RUN];
        finish(r, x, base);
        int f;
        sr_seq_tile<kSearch>(x, &s, target, &f, sm.seq);
        if (kSearch && f >= 0) {
            *found = base + f;
            return s;
        }
        if (!kSearch && marks.keep && threadIdx.x == 0) marks.keep[base / SR_SEQ_TILE] = s;
    }
    return s;
}

struct SeqRaw1 { float v[SR_SEQ_RUN]; };
struct SeqRaw2 { float p[SR_SEQ_RUN], q[SR_SEQ_RUN]; };

// SR_SEQ_RUN consecutive elements of an aligned row from index i0 on, all inside the row
__device__ __forceinline__ void seq_load_run_fast(const float* p, int i0, float (&v)[SR_SEQ_RUN])
{
    static_assert(SR_SEQ_RUN % 4 == 0, "whole float4 per thread");
    const float4* vp = (const float4*)(p + i0);
#pragma unroll
    for (int k = 0; k < SR_SEQ_RUN / 4; k++) {
        const float4 a = vp[k];
        v[4 * k] = a.x; v[4 * k + 1] = a.y; v[4 * k + 2] = a.z; v[4 * k + 3] = a.w;
    }
}
// ... of any row, zeros past the row's end
__device__ __forceinline__ void seq_load_run(const float* p, bool aligned, int i0, int n, float (&v)[SR_SEQ_RUN])
{
    if (threadIdx.x >= SR_SEQ_ACTIVE) {  // (these threads carry no terms)
#pragma unroll
        for (int j = 0; j < SR_SEQ_RUN; j++) v[j] = 0.0f;
    } else if (aligned && i0 + SR_SEQ_RUN <= n) {
        seq_load_run_fast(p, i0, v);
    } else {
#pragma unroll
        for (int j = 0; j < SR_SEQ_RUN; j++) v[j] = (i0 + j < n) ? p[i0 + j] : 0.0f;
    }
}

// (every term is multiplied by m1 and then by m2 first: the two normalising factors of a row that was left unscaled)
struct SeqNoWatch {
    __device__ __forceinline__ void operator()(float, int) const {}
};
// watch(x, i) sees every term with its index as it passes (the terms of a tile are looked at before the tile is added)
struct SeqNoMap {
    __device__ __forceinline__ float operator()(float x, int) const { return x; }
};
// map(x, i) stands between a scaled term and the sum: the term that is added (and watched) is what it returns
template <bool kSearch, typename Watch = SeqNoWatch, typename Map = SeqNoMap>
__device__ __forceinline__ float seq_sum_row(const float* p, int n, float s0, float target, int* found, FullSmem& sm,
                                             float m1 = 1.0f, float m2 = 1.0f, Watch watch = Watch(), Map map = Map(),
                                             SeqMarks marks = SeqMarks())
{
    static_assert(SR_SEQ_ACTIVE == SR_SEQ_THREADS, "every thread of the block loads a run");
    const bool aligned = ((uintptr_t)p & 15u) == 0u;
    auto issue_fast = [&](int base, SeqRaw1& r) __attribute__((always_inline)) {
        seq_load_run_fast(p, base + (int)threadIdx.x * SR_SEQ_RUN, r.v);
    };
    auto issue_any = [&](int base, SeqRaw1& r) __attribute__((always_inline)) {
        seq_load_run(p, aligned, base + (int)threadIdx.x * SR_SEQ_RUN, n, r.v);
    };
    auto finish = [&](const SeqRaw1& r, float (&x)[SR_SEQ_RUN], int base) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < SR_SEQ_RUN; j++) {
            x[j] = map(__fmul_rn(__fmul_rn(r.v[j], m1), m2), base + (int)threadIdx.x * SR_SEQ_RUN + j);
            watch(x[j], base + (int)threadIdx.x * SR_SEQ_RUN + j);
        }
    };
    return seq_sum_tiles<kSearch, 3, SeqRaw1>(issue_fast, issue_any, finish, aligned, n, s0, target, found, sm, marks);
}

// ... and over the positive part of the difference of two rows (residual resampling)
template <bool kSearch>
__device__ __forceinline__ float seq_sum_residual(const float* p, const float* q, int n, float s0, float target, int* found,
                                                  FullSmem& sm, float m1 = 1.0f, float m2 = 1.0f, SeqMarks marks = SeqMarks())
{
    const bool aligned = (((uintptr_t)p | (uintptr_t)q) & 15u) == 0u;
    auto issue_fast = [&](int base, SeqRaw2& r) __attribute__((always_inline)) {
        const int i0 = base + (int)threadIdx.x * SR_SEQ_RUN;
        seq_load_run_fast(p, i0, r.p);
        seq_load_run_fast(q, i0, r.q);
    };
    auto issue_any = [&](int base, SeqRaw2& r) __attribute__((always_inline)) {
        const int i0 = base + (int)threadIdx.x * SR_SEQ_RUN;
        seq_load_run(p, aligned, i0, n, r.p);
        seq_load_run(q, aligned, i0, n, r.q);
    };
    auto finish = [&](const SeqRaw2& r, float (&x)[SR_SEQ_RUN], int) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < SR_SEQ_RUN; j++) {
            const float d = __fsub_rn(__fmul_rn(__fmul_rn(r.p[j], m1), m2), r.q[j]);
            x[j] = d > 0.0f ? d : 0.0f;
        }
    };
    return seq_sum_tiles<kSearch, 2, SeqRaw2>(issue_fast, issue_any, finish, aligned, n, s0, target, found, sm, marks);
}

// ---- exact sums prepared by the whole device ---------------------------------------------------------------
// One workgroup adds a row at the rate at which one compute unit reads and scans it (1 MB in ~45 us).  Where the terms
// lie in memory before that workgroup starts, the whole device prepares the sum: the row is cut into segments of
// SR_SEG_TERMS terms, its workgroups leave an approximate sum of every segment (any order), and seg_make_record turns
// every segment into its increment function n -> n + a[n & 1] (sr_seqsum.h) for the binade that the
// approximate prefix predicts for the segment's start.  The workgroup that needs the sum then only walks the
// functions (seg_walk, one wave): a function is applied when the exact running sum in front of its segment lies in the
// binade it was made for and stays there; any other segment -- one in which the sum changes binade (a sum that starts
// at zero does that ~17 times, mostly within the first segments), a prediction that missed -- is added from its terms
// by the wave's own exact scan (sr_seq_wave).  The result never depends on the prediction: only the time does.
__device__ __forceinline__ int seg_count(int n) { return (n + SR_SEG_TERMS - 1) / SR_SEG_TERMS; }
static_assert(SR_SEG_TERMS == SR_WAVE * SR_SEQ_RUN && sizeof(SeqSegFunc) == 96, "one run of 16 terms per lane; six 16-byte loads per record");

struct SegRec {
    uint4 f, g, x0, x1, x2, x3;
};
// (kAgent: the records were written by other workgroups of the same launch)
template <bool kAgent>
__device__ __forceinline__ void seg_load_rec(const SeqSegFunc* funcs, int seg, int nseg, SegRec& r)
{
    const SeqSegFunc* f = funcs + min(seg, nseg - 1);
    if (kAgent) {
        const unsigned long long* q = (const unsigned long long*)f;
        unsigned long long v[12];
#pragma unroll
        for (int i = 0; i < 12; i++) v[i] = sr_load_agent(q + i);
        auto word = [&](int i) -> uint4 { return make_uint4((uint32_t)v[2 * i], (uint32_t)(v[2 * i] >> 32), (uint32_t)v[2 * i + 1], (uint32_t)(v[2 * i + 1] >> 32)); };
        r.f = word(0); r.g = word(1); r.x0 = word(2); r.x1 = word(3); r.x2 = word(4); r.x3 = word(5);
    } else {
        const uint4* q = (const uint4*)f;
        r.f = q[0]; r.g = q[1]; r.x0 = q[2]; r.x1 = q[3]; r.x2 = q[4]; r.x3 = q[5];
    }
    if (seg >= nseg) r.f.w = SR_SEG_ZERO;
}

// The exact running sum over the terms of nseg segments from s0, by the 64 lanes of ONE wave.  With kSearch it stops at the
// first term at which the running sum reaches `target`: *found = its index and the returned value is the running sum at that
// term.  With `states` (not with kSearch) the running sum behind segment g is left at states[g].
// load(segment, x) gives the lane's 16 terms of a segment, wherever the terms come from.
//
// 64 segments at a time, a lane each, the next 64 loading meanwhile.  The segments that are one function with the same
// increment for both parities -- nearly all -- are summed up once (inclusive sums T over the lanes).  The others are known
// beforehand and taken one by one: the exact sum in front of one is a lane read and an addition, its record gives the sum
// behind it; a record that does not fit that sum leaves the segment to be added from its terms.  Only then is it looked at
// whether every segment lay in the binade its record was made for; the first that did not is added from its terms, and what
// follows is done again.  A segment taken by itself costs some 50 instructions of the one wave, 0.1 us, a sum that
// starts at zero has about a dozen; looking for the end of every run of segments as it went, the walk took 0.45 us for each:
// 98 segments of a row of 100,003 entries 5.3 us, and a search over as many 7.5.
// first64: the first 64 records, where the caller has asked for them already.  kFew: there are no more than those.  kNear: they lie in
// shared memory, mostly, and are not asked for ahead (24 registers less).
template <bool kSearch, bool kAgent = false, bool kFew = false, bool kNear = false, typename Load>
__device__ __forceinline__ float seg_walk_from(Load load, int nseg, const SeqSegFunc* funcs, float s0, float target, int* found,
                                               float* states, const SegRec* first64 = nullptr)
{
    const int lane = sr_lane();
    uint32_t sb = (uint32_t)__builtin_amdgcn_readfirstlane((int)sr_f2u(s0));  // the running sum's bits, the same in every lane
    *found = -1;
    SegRec next;
    if (first64) next = *first64;
    else seg_load_rec<kAgent>(funcs, lane, nseg, next);
    for (int base = 0; base < nseg; base += SR_WAVE) {
        if (kNear && base > 0) seg_load_rec<kAgent>(funcs, base + lane, nseg, next);
        const SegRec r = next;
        if (!kFew && !kNear && base + SR_WAVE < nseg) seg_load_rec<kAgent>(funcs, base + SR_WAVE + lane, nseg, next);  // (the next 64 segments' come in meanwhile)
        const uint32_t kind = r.f.w & 0xffu;
        const bool simple = kind == SR_SEG_PLAIN && r.f.x == r.f.y && r.f.x < (1u << 24), split = kind == SR_SEG_SPLIT;
        const unsigned long long stops = ~__ballot(simple || kind == SR_SEG_ZERO);
        const uint32_t T = (uint32_t)sr_wave_incl_scan_i32(simple ? (int)r.f.x : 0);
        uint32_t eb = sr_state_eb(sb), off = sr_state_n(sb, eb);
        uint32_t pre = off, ebv = eb;  // behind a lane's segment the sum is pre + T in the binade ebv
        unsigned long long todo = stops;
        if (sb == 0u && stops != 0ull) {
            // the first segment that has a term, where its record carries the sum behind it
            const int t = (int)__ffsll((long long)stops) - 1;
            const uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)kind, t), Tt = (uint32_t)__builtin_amdgcn_readlane((int)T, t);
            if (k == SR_SEG_EXACT && Tt == 0u) {
                const uint32_t to = (uint32_t)__builtin_amdgcn_readlane((int)r.g.w, t);
                eb = sr_state_eb(to);
                off = sr_state_n(to, eb);
                if (lane >= t) { pre = off; ebv = eb; }
                todo &= todo - 1ull;
            }
        }
        const uint32_t eb1 = kind == SR_SEG_PLAIN || split ? (uint32_t)r.f.z : 0xffffu;
        // One form for both kinds of records, no branch per segment: a plain one has sixteen zeros for the terms of its crossing and a
        // second function that adds nothing.  [lo2, lo2 + size2): the bits of the second function's binade.
        uint32_t odd1 = 0u, inc2 = 0u, odd2 = 0u, lo2 = 0u, size2 = 0u;
        float xs[16] = {};
        if (todo != 0ull) {
            odd1 = r.f.y - r.f.x;
            inc2 = split ? r.g.x : 0u;
            odd2 = split ? r.g.y - r.g.x : 0u;
            const uint32_t eb2 = split ? (uint32_t)r.g.z : eb1;
            lo2 = eb2 > 1u ? eb2 << 23 : 0u;
            size2 = eb2 > 1u ? 1u << 23 : 1u << 24;
            const uint32_t words[16] = {r.x0.x, r.x0.y, r.x0.z, r.x0.w, r.x1.x, r.x1.y, r.x1.z, r.x1.w,
                                        r.x2.x, r.x2.y, r.x2.z, r.x2.w, r.x3.x, r.x3.y, r.x3.z, r.x3.w};
#pragma unroll
            for (int j = 0; j < 16; j++) xs[j] = split ? sr_u2f(words[j]) : 0.0f;
        }
        int pos = 0;  // the segments below were where they were planned
        for (;;) {
            int fix = -1;  // a segment to be added from its terms
            uint32_t before = 0u;
            while (todo != 0ull) {
                const int t = (int)__ffsll((long long)todo) - 1;
                todo &= todo - 1ull;
                const uint32_t Tt = (uint32_t)__builtin_amdgcn_readlane((int)T, t), n = off + Tt;
                before = sr_state_bits(n, eb);
                const uint32_t b1 = before + (r.f.x + (odd1 & (0u - (n & 1u))));
                float acc = sr_u2f(b1);
#pragma unroll
                for (int j = 0; j < 16; j++) acc = __fadd_rn(acc, xs[j]);
                const uint32_t b2 = sr_f2u(acc), b3 = b2 + (inc2 + (odd2 & (0u - (b2 & 1u))));
                // (one comparison each: the record is for the binade the sum is in, the first function ends in it, the second one
                // starts and ends in its own)
                const unsigned long long ok = __ballot(eb1 == eb) & __ballot(b1 < sr_state_bits(1u << 24, eb)) & __ballot(b2 >= lo2) & __ballot(b3 - lo2 < size2);
                const uint32_t to = (uint32_t)__builtin_amdgcn_readlane((int)b3, t);
                if (SR_RARE(((ok >> t) & 1ull) == 0ull || n >= (1u << 24))) {
                    fix = n >= (1u << 24) ? -1 : t;  // (-1: a segment in front of this one left its binade unforeseen)
                    break;
                }
                eb = sr_state_eb(to);
                off = sr_state_n(to, eb) - Tt;
                if (lane >= t) { pre = off; ebv = eb; }
            }
            if (fix < 0) {
                const unsigned long long bad = __ballot(simple && lane >= pos && (eb1 != ebv || pre + T >= (1u << 24)));
                if (SR_USUAL(bad == 0ull)) break;
                // (everything in front of this segment is exact)
                fix = (int)__ffsll((long long)bad) - 1;
                pos = fix + 1;
                before = fix > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)sr_state_bits(pre + T, ebv), fix - 1) : sb;
                todo = pos < SR_WAVE ? stops & (~0ull << pos) : 0ull;
            }
            float x[SR_SEQ_RUN];
            load(base + fix, x);
            int at;
            const uint32_t to = (uint32_t)__builtin_amdgcn_readfirstlane((int)sr_f2u(sr_seq_wave<SR_SEQ_RUN, false>(x, sr_u2f(before), 0.0f, &at)));
            eb = sr_state_eb(to);
            off = sr_state_n(to, eb) - (uint32_t)__builtin_amdgcn_readlane((int)T, fix);
            if (lane >= fix) { pre = off; ebv = eb; }
        }
        const uint32_t ends = sr_state_bits(pre + T, ebv);
        if (!kSearch && states && base + lane < nseg) states[base + lane] = sr_u2f(ends);
        if (kSearch) {
            const unsigned long long reach = __ballot(sr_u2f(ends) >= target && base + lane < nseg);
            if (reach != 0ull) {
                const int t = (int)__ffsll((long long)reach) - 1;
                const uint32_t before = t > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)ends, t - 1) : sb;
                float x[SR_SEQ_RUN];
                load(base + t, x);
                int at;
                const float s = sr_seq_wave<SR_SEQ_RUN, true>(x, sr_u2f(before), target, &at);
                *found = (base + t) * SR_SEG_TERMS + at;
                return s;
            }
        }
        sb = (uint32_t)__builtin_amdgcn_readlane((int)ends, SR_WAVE - 1);
    }
    return sr_u2f(sb);
}

// ... over terms[0, n) in memory
template <bool kSearch>
__device__ __forceinline__ float seg_walk(const float* terms, int n, const SeqSegFunc* funcs, float s0, float target, int* found,
                                          float* states, const SegRec* first64 = nullptr)
{
    const bool aligned = ((uintptr_t)terms & 15u) == 0u;
    const int lane = sr_lane();
    return seg_walk_from<kSearch>([&](int seg, float (&x)[SR_SEQ_RUN]) __attribute__((always_inline)) {
        seq_load_run(terms, aligned, seg * SR_SEG_TERMS + lane * SR_SEQ_RUN, n, x);
    }, seg_count(n), funcs, s0, target, found, states, first64);
}

// The record of one segment (SeqSegFunc) from its terms x (lane l holds the terms 16 l ... 16 l + 15 of the segment) and
// the approximate sum `before` of everything in front of the segment.  One wave.
// With `seg_sum` (>= 0: the approximate sum of the segment's own terms, known beforehand) a segment whose start and
// end lie well inside one binade gets its one function without a look at where inside it the sum would change binade.
// (kAgent: the record will be read by other workgroups of the same launch.  kAbout: seg_sum was not added up from the terms in
// floating point, where a sum is 0 only if every term is, but in whole units or by atomic additions: whether the segment has a
// term at all, the terms say.)
template <bool kAgent = false, bool kAbout = false>
__device__ __forceinline__ void seg_make_record(const float (&x)[SR_SEQ_RUN], int seg, double before, SeqSegFunc* out,
                                                float seg_sum = -1.0f)
{
    const int lane = sr_lane();
    auto put = [&](int i, uint32_t v0, uint32_t v1, uint32_t v2, uint32_t v3) {
        if (kAgent) sr_store_agent_f4((float4*)out + i, sr_u2f(v0), sr_u2f(v1), sr_u2f(v2), sr_u2f(v3));
        else ((uint4*)out)[i] = make_uint4(v0, v1, v2, v3);
    };
    {
        // A segment without a term (masked, or cut) changes no sum whatever its binade.  This is the one thing in a record that no
        // walk looks at again.  (Asked of the terms everywhere, a call of the verifier over 144 rows of 262,144 took 128.5 us, not 126.7.)
        float any = seg_sum;
        if (kAbout || seg_sum < 0.0f) {
            any = sr_max_f32(x[0], x[SR_SEQ_RUN - 1]);
#pragma unroll
            for (int j = 1; j + 1 < SR_SEQ_RUN; j += 2) any = sr_max3_f32(any, x[j], x[j + 1]);
        }
        if (__ballot(any > 0.0f) == 0ull) {
            if (lane == 0) put(0, 0u, 0u, 0u, SR_SEG_ZERO);
            return;
        }
    }
    const bool first = seg == 0 || before == 0.0;  // nothing in front
    if (!first && seg_sum >= 0.0f) {
        const float lo = __double2float_rn(before), hi = lo + seg_sum;
        uint32_t nn;
        int eb_lo, eb_hi;
        sr_split(lo * 0.9999f, &nn, &eb_lo);
        sr_split(hi * 1.0001f, &nn, &eb_hi);
        if (SR_USUAL(eb_lo == eb_hi)) {  // (wave-uniform: both are the same in every lane)
            const SrInc sc = sr_scan_inc<false>(sr_run_inc(x, eb_lo));
            if (lane == SR_WAVE - 1) {
                put(0, sc.a0, sc.a1, (uint32_t)eb_lo, SR_SEG_PLAIN);
                put(1, SR_SEQ_SAT, SR_SEQ_SAT, (uint32_t)eb_lo, 0u);
            }
            return;
        }
    }
    // approximate running sum behind every lane's run (single precision does: a prediction that misses costs time only)
    float own = 0.0f;
#pragma unroll
    for (int j = 0; j < SR_SEQ_RUN; j++) own += x[j];
    const float incl = sr_wave_incl_sum_f32(own);
    const float before_f = __double2float_rn(before);
    const float p_end = before_f + incl;
    uint32_t nn;
    int eb_first, eb_last, eb_mine_end;
    sr_split(before_f, &nn, &eb_first);
    sr_split(__shfl(p_end, SR_WAVE - 1), &nn, &eb_last);
    sr_split(p_end, &nn, &eb_mine_end);
    SeqSegFunc f;
    f.a0 = f.a1 = f.b0 = f.b1 = SR_SEQ_SAT;
    f.eb = eb_first; f.eb2 = eb_last; f.kind = SR_SEG_PLAIN; f.end_bits = 0u;
    int cross = -1;
    if (SR_RARE(first)) {
        // the row's first segment (that has a term) starts from +0 exactly: its end, once and for all
        int dummy;
        const float end = sr_seq_wave<SR_SEQ_RUN, false>(x, 0.0f, 0.0f, &dummy);
        f.kind = SR_SEG_EXACT;
        f.end_bits = sr_f2u(end);
    } else if (eb_first == eb_last) {
        const SrInc sc = sr_scan_inc<false>(sr_run_inc(x, eb_first));
        f.a0 = (uint32_t)__builtin_amdgcn_readlane((int)sc.a0, SR_WAVE - 1);
        f.a1 = (uint32_t)__builtin_amdgcn_readlane((int)sc.a1, SR_WAVE - 1);
    } else {
        // the first lane behind whose run the sum is expected in another binade; everything behind that lane must then
        // lie in the segment's last binade, or the segment is no two functions
        const unsigned long long left = __ballot(eb_mine_end != eb_first);
        cross = left ? (int)__ffsll((long long)left) - 1 : SR_WAVE - 1;
        const int eb_behind = __builtin_amdgcn_readlane(eb_mine_end, cross);
        if (eb_behind == eb_last) {
            SrInc m1, m2;
            m1.a0 = m1.a1 = m2.a0 = m2.a1 = 0u;
            if (lane < cross) m1 = sr_run_inc(x, eb_first);
            if (lane > cross) m2 = sr_run_inc(x, eb_last);
            const SrInc s1 = sr_scan_inc<false>(m1), s2 = sr_scan_inc<false>(m2);
            f.a0 = (uint32_t)__builtin_amdgcn_readlane((int)s1.a0, SR_WAVE - 1);
            f.a1 = (uint32_t)__builtin_amdgcn_readlane((int)s1.a1, SR_WAVE - 1);
            f.b0 = (uint32_t)__builtin_amdgcn_readlane((int)s2.a0, SR_WAVE - 1);
            f.b1 = (uint32_t)__builtin_amdgcn_readlane((int)s2.a1, SR_WAVE - 1);
            f.kind = SR_SEG_SPLIT | ((uint32_t)cross << 8);
        } else {
            cross = -1;
        }
    }
    if (lane == 0) {
        put(0, f.a0, f.a1, (uint32_t)f.eb, f.kind);
        put(1, f.b0, f.b1, (uint32_t)f.eb2, f.end_bits);
    }
    if (lane == cross) {
#pragma unroll
        for (int j = 0; j < 16; j += 4) put(2 + j / 4, sr_f2u(x[j]), sr_f2u(x[j + 1]), sr_f2u(x[j + 2]), sr_f2u(x[j + 3]));
    }
}

// The search that follows a sum over the same terms: the first term at which the running sum reaches `target`, from
// the states the sum left (one wave; -1 when the sum stays below the target).
template <typename Load>
__device__ __forceinline__ int seg_search_states(Load load, int nseg, const float* states, float target, float* at_sum)
{
    int first = nseg;
    for (int g = sr_lane(); g < nseg; g += SR_WAVE)
        if (states[g] >= target) { first = g; break; }
    first = sr_wave_min_i32(first);
    if (first >= nseg) return -1;
    float x[SR_SEQ_RUN];
    load(first, x);
    int at;
    *at_sum = sr_seq_wave<SR_SEQ_RUN, true>(x, first > 0 ? states[first - 1] : 0.0f, target, &at);
    return at >= 0 ? first * SR_SEG_TERMS + at : -1;
}

// TensorPrimitives.Sum in its 256-bit shape: strided lane accumulators seeded with the first vector, the
// ragged tail folded in through an overlapped last vector, pairwise horizontal add.
template <typename Term>
__device__ __forceinline__ float tp_sum(Term term, int n, FullSmem& sm)
{
    int dummy;
    if (n < 4) {
        return seq_sum<false>(term, n, 0.0f, 0.0f, &dummy, sm);
    }
    if (n >= 8) {
        // the eight lane accumulators as eight chains advanced together: one pass over the row
        const int nv = n / 8, rem = n - nv * 8;
        const int g = (int)threadIdx.x & (SR_SEQ_CHAINS - 1), lt = (int)threadIdx.x >> 3;
        const bool extra = rem > 0 && g >= 8 - rem;
        const int cnt = nv + (extra ? 1 : 0);
        float s = 0.0f;
        auto load = [&](int base, float (&x)[SR_SEQ_RUN8]) __attribute__((always_inline)) {
            const int i0 = base + lt * SR_SEQ_RUN8;
            if (i0 + SR_SEQ_RUN8 <= nv) {
#pragma unroll
                for (int j = 0; j < SR_SEQ_RUN8; j++) x[j] = term((i0 + j) * 8 + g);
            } else {
#pragma unroll
                for (int j = 0; j < SR_SEQ_RUN8; j++) {
                    const int i = i0 + j;
                    x[j] = (i < cnt) ? (i < nv ? term(i * 8 + g) : term(n - 8 + g)) : 0.0f;
                }
            }
        };
        // two register sets take turns: no copy, which would wait for the loads, sits between the tiles
        float xa[SR_SEQ_RUN8], xb[SR_SEQ_RUN8];
#pragma unroll
        for (int j = 0; j < SR_SEQ_RUN8; j++) xa[j] = xb[j] = 0.0f;
        load(0, xa);
        for (int base = 0; base < nv + 1; base += 2 * SR_SEQ_CHAIN_TILE) {
            if (base + SR_SEQ_CHAIN_TILE < nv + 1) load(base + SR_SEQ_CHAIN_TILE, xb);
            sr_seq_tile8(xa, &s, sm.seq8);
            if (base + SR_SEQ_CHAIN_TILE >= nv + 1) break;
            if (base + 2 * SR_SEQ_CHAIN_TILE < nv + 1) load(base + 2 * SR_SEQ_CHAIN_TILE, xa);
            sr_seq_tile8(xb, &s, sm.seq8);
        }
        __syncthreads();
        if (lt == 0) sm.lane_sum[g] = s;
        __syncthreads();
        const float l0 = sm.lane_sum[0], l1 = sm.lane_sum[1], l2 = sm.lane_sum[2], l3 = sm.lane_sum[3],
                    l4 = sm.lane_sum[4], l5 = sm.lane_sum[5], l6 = sm.lane_sum[6], l7 = sm.lane_sum[7];
        __syncthreads();
        return __fadd_rn(__fadd_rn(__fadd_rn(l0, l1), __fadd_rn(l2, l3)), __fadd_rn(__fadd_rn(l4, l5), __fadd_rn(l6, l7)));
    }
    const int w = 4;
    const int nv = n / w, rem = n - nv * w;
    float lane_sum[4];
#pragma unroll
    for (int l = 0; l < 4; l++) {
        const bool extra = rem > 0 && l >= w - rem;
        const int cnt = nv + (extra ? 1 : 0);
        auto lt = [&](int i) -> float { return i < nv ? term(i * w + l) : term(n - w + l); };
        lane_sum[l] = seq_sum<false>(lt, cnt, 0.0f, 0.0f, &dummy, sm);
    }
    return __fadd_rn(__fadd_rn(lane_sum[0], lane_sum[1]), __fadd_rn(lane_sum[2], lane_sum[3]));
}

// The same sum over a long row in memory (times mul when do_mul), one wave per lane accumulator.  The row comes in
// through LDS 8,192 entries at a time -- every thread brings two 16-byte pieces, two rounds ahead of the round that is
// added --, laid out chain by chain, and the wave of a chain adds its 1,024 terms of the round with the wave's own
// exact scan (sr_seq_wave_grown): no block-wide step but one barrier per round, so a round costs what its 32 KB take to
// arrive.  The place of term v = 16 l + j of chain g is g * 1024 + 64 j + (l + 2 j) mod 64: the 64 lanes of a wave
// read a term from 64 consecutive places, and the stores of a piece's four entries fall two to a bank.
__device__ __forceinline__ float tp_sum_row(const float* p, int n, float mul, bool do_mul, FullSmem& sm)
{
    constexpr int kRound = 8192;
    static_assert(offsetof(FullSmem, sprob) == offsetof(FullSmem, sortbuf) + sizeof(FullSmem::sortbuf) &&
                  offsetof(FullSmem, tags) == offsetof(FullSmem, sprob) + sizeof(FullSmem::sprob) &&
                  sizeof(FullSmem::sortbuf) + sizeof(FullSmem::sprob) + sizeof(FullSmem::tags) >= 2 * kRound * sizeof(float),
                  "two rounds fit the three arrays, which lie one behind the other");
    static_assert(kRound == 8 * kT, "two 16-byte pieces per thread and round");
    if (n < 2 * kRound || ((uintptr_t)p & 15u) != 0u) {
        if (do_mul) return tp_sum([&](int i) -> float { return __fmul_rn(p[i], mul); }, n, sm);
        return tp_sum([&](int i) -> float { return p[i]; }, n, sm);
    }
    float* buf = (float*)sm.sortbuf;
    const int tid = threadIdx.x, lane = sr_lane(), wave = sr_wave_id();
    const int nv = n / 8, rem = n - nv * 8, body = nv * 8;
    const int rounds = (body + kRound - 1) / kRound;
    auto fetch = [&](int r, float4 (&v)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int x0 = r * kRound + 4 * (tid + h * kT);
            if (x0 + 4 <= body) {
                v[h] = *(const float4*)(p + x0);
            } else {
                v[h].x = x0 < body ? p[x0] : 0.0f;
                v[h].y = x0 + 1 < body ? p[x0 + 1] : 0.0f;
                v[h].z = x0 + 2 < body ? p[x0 + 2] : 0.0f;
                v[h].w = 0.0f;  // (x0 + 3 < body would have taken the other way)
            }
        }
    };
    auto stash = [&](int r, const float4 (&v)[2]) __attribute__((always_inline)) {
        float* b = buf + (r & 1) * kRound;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int t2 = tid + h * kT;  // the piece's number within the round
            const int vec = t2 >> 1, j = vec & 15, l = vec >> 4;
            float* at = b + (4 * (t2 & 1)) * 1024 + 64 * j + ((l + 2 * j) & 63);
            at[0] = do_mul ? __fmul_rn(v[h].x, mul) : v[h].x;
            at[1024] = do_mul ? __fmul_rn(v[h].y, mul) : v[h].y;
            at[2048] = do_mul ? __fmul_rn(v[h].z, mul) : v[h].z;
            at[3072] = do_mul ? __fmul_rn(v[h].w, mul) : v[h].w;
        }
    };
    float sc = 0.0f;
    auto add_round = [&](int r) __attribute__((always_inline)) {
        if (wave < SR_SEQ_CHAINS) {
            const float* b = buf + (r & 1) * kRound + wave * 1024;
            float x[16];
#pragma unroll
            for (int j = 0; j < 16; j++) x[j] = b[64 * j + ((lane + 2 * j) & 63)];
            int dummy;
            sc = sr_seq_wave_grown<16, false>(x, sc, 0.0f, &dummy);
        }
    };
    // (behind the last round the loop fetches that round again, to no effect: the compiler can wait for "all but the
    // newest loads" only where it can count them)
    float4 va[2], vb[2];
    __syncthreads();  // (whoever used the arrays before is done)
    fetch(0, va);
    fetch(min(1, rounds - 1), vb);
    stash(0, va);
    for (int r = 0; r < rounds; r += 2) {
        fetch(min(r + 2, rounds - 1), va);
        __syncthreads();
        add_round(r);
        if (r + 1 >= rounds) break;
        stash(r + 1, vb);
        fetch(min(r + 3, rounds - 1), vb);
        __syncthreads();
        add_round(r + 1);
        if (r + 2 < rounds) stash(r + 2, va);
    }
    if (wave < SR_SEQ_CHAINS) {
        if (rem > 0 && wave >= 8 - rem) {  // the overlapped last vector's entry of this chain
            float x[1];
            const float t = p[n - 8 + wave];
            x[0] = lane == 0 ? (do_mul ? __fmul_rn(t, mul) : t) : 0.0f;
            int dummy;
            sc = sr_seq_wave<1, false>(x, sc, 0.0f, &dummy);
        }
        if (lane == 0) sm.lane_sum[wave] = sc;
    }
    __syncthreads();
    const float l0 = sm.lane_sum[0], l1 = sm.lane_sum[1], l2 = sm.lane_sum[2], l3 = sm.lane_sum[3],
                l4 = sm.lane_sum[4], l5 = sm.lane_sum[5], l6 = sm.lane_sum[6], l7 = sm.lane_sum[7];
    __syncthreads();
    return __fadd_rn(__fadd_rn(__fadd_rn(l0, l1), __fadd_rn(l2, l3)), __fadd_rn(__fadd_rn(l4, l5), __fadd_rn(l6, l7)));
}

// Normalize (Sampler.cs:553-562)
__device__ __forceinline__ void normalize_row(float* p, int n, FullSmem& sm)
{
    const float sum = tp_sum_row(p, n, 1.0f, false, sm);
    if (sum > 0.0f && sum != 1.0f) {
        const float inv = __fdiv_rn(1.0f, sum);
        row_pass<true>(p, n, [&](float x, int) -> float { return __fmul_rn(x, inv); });
    }
    __syncthreads();
}

// k-th largest value of p[0..n) (1-based), p >= 0: FindKthLargest (Sampler.cs:624-645).
// With last_shift = 16 only the upper 16 bits are resolved: the result is then the smallest value of the
// 65536-value bucket that holds the k-th largest.
// Keys above hi_key are left out (they count as absent).
__device__ __forceinline__ float kth_largest(const float* p, int n, int k, FullSmem& sm, int last_shift = 0,
                                             uint32_t hi_key = 0xffffffffu)
{
    uint32_t prefix = 0u, pmask = 0u;
    int need = k;
    for (int shift = 24; shift >= last_shift; shift -= 8) {
        if (threadIdx.x < 256) sm.hist[threadIdx.x] = 0u;
        __syncthreads();
        // Zeros (masked or filtered entries, often most of the row) are left out: they are the smallest keys and
        // only matter when fewer than k entries are positive, and then the answer is zero either way.
        row_pass<false>(const_cast<float*>(p), n, [&](float x, int) -> float {
            const uint32_t key = sr_f2u(x);
            if (key != 0u && (key & pmask) == prefix && key <= hi_key) atomicAdd(&sm.hist[(key >> shift) & 0xffu], 1u);
            return x;
        });
        __syncthreads();
        if (threadIdx.x == 0) {
            int c = 0, d = 255;
            for (; d > 0; d--) {
                if (c + (int)sm.hist[d] >= need) break;
                c += (int)sm.hist[d];
            }
            sm.bc[0] = (uint32_t)d;
            sm.bc[1] = (uint32_t)(need - c);
        }
        __syncthreads();
        prefix |= sm.bc[0] << shift;
        pmask |= 0xffu << shift;
        need = (int)sm.bc[1];
        __syncthreads();
    }
    return sr_u2f(prefix);
}

// The value of lane (lane ^ kMask), moved by the vector unit alone (no LDS): DPP inside rows of 16 lanes, the swaps of
// rows and of wave halves beyond.  Every lane of the wave must be active.
template <int kMask> __device__ __forceinline__ uint32_t lane_xor_u32(uint32_t v)
{
    static_assert(kMask == 1 || kMask == 2 || kMask == 4 || kMask == 8 || kMask == 16 || kMask == 32, "one bit of the lane number");
    if (kMask == 1) return sr_dpp_u32<0xB1>(v);                        // quad_perm [1, 0, 3, 2]
    if (kMask == 2) return sr_dpp_u32<0x4E>(v);                        // quad_perm [2, 3, 0, 1]
    if (kMask == 4) return sr_dpp_u32<0x1B>(sr_dpp_u32<0x141>(v));     // 7 - l inside eight lanes, then 3 - l inside four
    if (kMask == 8) return sr_dpp_u32<0x128>(v);                       // a row rotated by half its length
    if (kMask == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return (sr_lane() & 16) ? r[0] : r[1];
    }
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (sr_lane() & 32) ? r[0] : r[1];
}
// The wave's sums of eight values per lane: lane l returns that of c[l & 7].  (Three exchanges halve what a lane holds, three
// more add up the groups of eight lanes: ten additions where eight sums by themselves take 48.)
__device__ __forceinline__ float wave_sum_8(const float (&c)[8])
{
    const int lane = sr_lane();
    float h[4], q[2];
    const bool b4 = (lane & 4) != 0, b2 = (lane & 2) != 0, b1 = (lane & 1) != 0;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const float keep = b4 ? c[g + 4] : c[g], send = b4 ? c[g] : c[g + 4];
        h[g] = keep + sr_u2f(lane_xor_u32<4>(sr_f2u(send)));
    }
#pragma unroll
    for (int g = 0; g < 2; g++) {
        const float keep = b2 ? h[g + 2] : h[g], send = b2 ? h[g] : h[g + 2];
        q[g] = keep + sr_u2f(lane_xor_u32<2>(sr_f2u(send)));
    }
    float v = (b1 ? q[1] : q[0]) + sr_u2f(lane_xor_u32<1>(sr_f2u(b1 ? q[0] : q[1])));
    v += sr_u2f(lane_xor_u32<8>(sr_f2u(v)));
    v += sr_u2f(lane_xor_u32<16>(sr_f2u(v)));
    v += sr_u2f(lane_xor_u32<32>(sr_f2u(v)));
    return v;
}
template <int kMask> __device__ __forceinline__ unsigned long long lane_xor_key(unsigned long long v)
{
    return ((unsigned long long)lane_xor_u32<kMask>((uint32_t)(v >> 32)) << 32) | (unsigned long long)lane_xor_u32<kMask>((uint32_t)v);
}
template <int kMask> __device__ __forceinline__ uint32_t lane_xor_key(uint32_t v) { return lane_xor_u32<kMask>(v); }

// Bitonic sort (descending) of buf[0 .. n_pow2) in LDS, n_pow2 a power of two <= kSmall, keys of 32 or 64 bits; entries
// that must come last are zero.  All threads call, behind a barrier that follows the last write of the entries.
//
// The entries live in registers, four consecutive ones per thread (a wave holds 256 consecutive entries): strides 1 and
// 2 pair registers of one thread, strides 4..128 pair lanes of one wave, and LDS is needed only for the strides of 256
// and more.  Those come at the start of the last merges (sizes 512 and up); all of them of one merge are done in one
// visit to LDS, by 256 threads that each hold one column (entries c, c + 256, c + 512, ...).
template <typename K>
__device__ __forceinline__ void sort_lds_desc(K* buf, int n_pow2)
{
    constexpr int kRow = 256;                 // entries of one wave
    constexpr int kCols = kSmall / kRow;      // most entries of one column
    static_assert(kRow == 4 * SR_WAVE && kRow * kW >= kSmall && kCols == 16, "the layout described above");
    const int tid = threadIdx.x, wave = sr_wave_id();
    if (n_pow2 <= kRow) {
        // A short list: every entry counts the entries that come before it (equal ones by their place).
        K key = 0;
        int rank = 0;
        if (tid < n_pow2) {
            key = buf[tid];
            for (int j = 0; j < n_pow2; j++) {
                const K o = buf[j];
                rank += (o > key || (o == key && j < tid)) ? 1 : 0;
            }
        }
        __syncthreads();
        if (tid < n_pow2) buf[rank] = key;
        __syncthreads();
        return;
    }
    const int base = 4 * tid;
    const int pe = max(n_pow2, 4);
    const bool wave_has = wave * kRow < pe;   // (the other waves only meet at the barriers)
    K v[4];
    auto load_rows = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = (base + r < n_pow2) ? buf[base + r] : (K)0;
    };
    auto store_rows = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (base + r < n_pow2) buf[base + r] = v[r];
    };
    auto cx = [&](K& lo_i, K& hi_i, bool desc) __attribute__((always_inline)) {  // lo_i is the entry with the smaller index
        const K mx = lo_i > hi_i ? lo_i : hi_i, mn = lo_i > hi_i ? hi_i : lo_i;
        lo_i = desc ? mx : mn;
        hi_i = desc ? mn : mx;
    };
    auto lane_step = [&](auto mask, bool want_max) __attribute__((always_inline)) {
        constexpr int kM = decltype(mask)::value;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const K o = lane_xor_key<kM>(v[r]);
            const K mx = v[r] > o ? v[r] : o, mn = v[r] > o ? o : v[r];
            v[r] = want_max ? mx : mn;
        }
    };
    // the steps of merge size k2 with strides j_first, j_first / 2, ..., 1 (j_first <= 128)
    auto row_steps = [&](int k2, int j_first) __attribute__((always_inline)) {
        const bool desc = (base & k2) == 0;  // (k2 >= 4: the four entries share it; k2 == 2 is handled below)
        if (j_first >= 128) lane_step(std::integral_constant<int, 32>{}, desc == ((base & 128) == 0));
        if (j_first >= 64) lane_step(std::integral_constant<int, 16>{}, desc == ((base & 64) == 0));
        if (j_first >= 32) lane_step(std::integral_constant<int, 8>{}, desc == ((base & 32) == 0));
        if (j_first >= 16) lane_step(std::integral_constant<int, 4>{}, desc == ((base & 16) == 0));
        if (j_first >= 8) lane_step(std::integral_constant<int, 2>{}, desc == ((base & 8) == 0));
        if (j_first >= 4) lane_step(std::integral_constant<int, 1>{}, desc == ((base & 4) == 0));
        if (k2 == 2) {
            cx(v[0], v[1], true);
            cx(v[2], v[3], false);
        } else {
            cx(v[0], v[2], desc);
            cx(v[1], v[3], desc);
            cx(v[0], v[1], desc);
            cx(v[2], v[3], desc);
        }
    };
    if (wave_has) {
        load_rows();
        for (int k2 = 2; k2 <= min(pe, kRow); k2 <<= 1) row_steps(k2, k2 >> 1);
    }
    for (int k2 = 2 * kRow; k2 <= pe; k2 <<= 1) {
        if (wave_has) store_rows();
        __syncthreads();
        if (tid < kRow) {
            const int cols = pe / kRow;  // 2, 4, 8 or 16 entries in this thread's column
            K c[kCols];
#pragma unroll
            for (int a2 = 0; a2 < kCols; a2++) c[a2] = a2 < cols ? buf[tid + a2 * kRow] : (K)0;
#pragma unroll
            for (int ja = kCols / 2; ja >= 1; ja >>= 1) {
                if (ja * kRow * 2 <= k2) {
#pragma unroll
                    for (int a2 = 0; a2 < kCols; a2++)
                        if ((a2 & ja) == 0 && (a2 | ja) < cols) cx(c[a2], c[a2 | ja], ((a2 * kRow) & k2) == 0);
                }
            }
#pragma unroll
            for (int a2 = 0; a2 < kCols; a2++)
                if (a2 < cols) buf[tid + a2 * kRow] = c[a2];
        }
        __syncthreads();
        if (wave_has) {
            load_rows();
            row_steps(k2, kRow / 2);
        }
    }
    if (wave_has) store_rows();
    __syncthreads();
}
__device__ __forceinline__ void sort_small_desc(FullSmem& sm, int n_pow2) { sort_lds_desc(sm.sortbuf, n_pow2); }

template <int ES>
__device__ __forceinline__ float load_logit(const char* rowp, int i)
{
    if (ES == 4) return ((const float*)rowp)[i];
    return sr_bf16_to_f32(((const uint16_t*)rowp)[i]);
}

// A sampled row needs no adjusted copy: the masked, scaled logit is recomputed from the input where it is read (the
// row maximum and the expf pass), which saves one pass over the row and one write of it.  The few ids that a logit
// bias or a history penalty touches are left out of those two passes -- a bitmap of the vocabulary, read beside the
// logits like an allow-mask, names them -- and handled by the kernels that run one workgroup per row: k_full_edits
// computes their adjusted values, keeps them (a.edit_tab: the bitmap, then one float per edit) and folds them into the
// row's maximum; k_full_row writes their expf before it reads the row.  Without the table (the host gives it when the
// batch holds such a row), and for a row with more edits than it takes, the row keeps its adjusted copy.
__device__ __forceinline__ bool row_edits_on_the_fly(const SrRow& rd, const SrFullArgs& a)
{
    return (a.edit_tab != nullptr || a.edits_in_pass) && sr_row_edits_on_the_fly(rd, a.vocab);
}
__device__ __forceinline__ bool row_is_direct(const SrRow& rd, const SrFullArgs& a)
{
    return rd.temperature > 0.0f && (rd.edit_cnt <= 0 || row_edits_on_the_fly(rd, a));
}

// The value of an edited id before the temperature: LogitBias (Sampler.cs:51-58), then the history penalties
// (:367-419), on the masked logit.
__device__ __forceinline__ float edited_logit(float x, const SrEdit& e, const SrRow& rd, bool sampled, bool pen)
{
    if (sampled && e.has_bias) x = __fadd_rn(x, e.bias);
    if (pen && e.occ_all > 0) {
        if (rd.rep != 1.0f)
            for (int o = 0; o < e.occ_win; o++) x = x > 0.0f ? __fdiv_rn(x, rd.rep) : __fmul_rn(x, rd.rep);
        if (rd.presence != 0.0f || rd.frequency != 0.0f)
            x = __fsub_rn(x, __fadd_rn(rd.presence, __fmul_rn(rd.frequency, (float)e.occ_all)));
    }
    return x;
}

// ---- one pass of the grid's x dimension over a row of logits ---------------------------------------------
// The masked (and temperature-scaled) logits of a row, sixteen input bytes per thread and load, four loads in flight;
// body(i, x, c) gets c consecutive values starting at element i (c = 4 or 8 on the vector path, 1 on the scalar
// path that rows with an unaligned start and the last elements of a row take).
template <int ES>
struct RowSource {
    const char* rowp;
    const uint32_t* mrow;
    bool scale;
    float inv_temp;
    const uint32_t* erow = nullptr;  // bitmap of the ids the row's edits touch (body gets the bits of its run), or null
    __device__ __forceinline__ float fix(float x, uint32_t keep) const
    {
        if (!keep) x = SR_NEG_INF;
        return scale ? __fmul_rn(x, inv_temp) : x;
    }
};
template <int ES, typename Body>
__device__ __forceinline__ void stream_row(const RowSource<ES>& src, int n, Body body)
{
    constexpr int E = 16 / ES, kU = 4;
    const int nv = (((uintptr_t)src.rowp & 15u) == 0u) ? n / E : 0;
    const int step = (int)gridDim.x * 256;
    for (int v0 = (int)blockIdx.x * 256 + (int)threadIdx.x; v0 < nv; v0 += step * kU) {
        uint4 raw[kU];
        uint32_t keep[kU], hit[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int v = v0 + u * step;
            raw[u] = make_uint4(0u, 0u, 0u, 0u);
            keep[u] = 0xffu;
            hit[u] = 0u;
            if (v < nv) {
                raw[u] = ((const uint4*)src.rowp)[v];
                if (src.mrow) keep[u] = src.mrow[(v * E) >> 5] >> ((v * E) & 31);
                if (src.erow) hit[u] = (src.erow[(v * E) >> 5] >> ((v * E) & 31)) & ((1u << E) - 1u);
            }
        }
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int v = v0 + u * step;
            if (v >= nv) break;
            float x[E];
            if (ES == 4) {
                x[0] = sr_u2f(raw[u].x); x[1] = sr_u2f(raw[u].y); x[2] = sr_u2f(raw[u].z); x[3] = sr_u2f(raw[u].w);
            } else {
                const uint32_t r[4] = {raw[u].x, raw[u].y, raw[u].z, raw[u].w};
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    x[(2 * q) % E] = sr_u2f(r[q] << 16);
                    x[(2 * q + 1) % E] = sr_u2f(r[q] & 0xffff0000u);
                }
            }
#pragma unroll
            for (int q = 0; q < E; q++) x[q] = src.fix(x[q], (keep[u] >> q) & 1u);
            body(v * E, x, E, hit[u]);
        }
    }
    for (int i = nv * E + (int)blockIdx.x * 256 + (int)threadIdx.x; i < n; i += step) {
        float x[E];
        x[0] = src.fix(load_logit<ES>(src.rowp, i), src.mrow ? (src.mrow[i >> 5] >> (i & 31)) & 1u : 1u);
        body(i, x, 1, src.erow ? (src.erow[i >> 5] >> (i & 31)) & 1u : 0u);
    }
}
// stores c values (c = 1, 4 or 8) at w + i, with 16-byte stores where the address allows
template <int E>
__device__ __forceinline__ void store_run(float* w, int i, const float (&x)[E], int c)
{
    if (c == E && (((uintptr_t)(w + i)) & 15u) == 0u) {
#pragma unroll
        for (int q = 0; q < E; q += 4) *(float4*)(w + i + q) = make_float4(x[q], x[q + 1], x[q + 2], x[q + 3]);
    } else {
#pragma unroll
        for (int q = 0; q < E; q++)
            if (q < c) w[i + q] = x[q];
    }
}

// The histogram of a row's e = expf(x - max) by their upper 16 bits (kHistPos positions: position d holds the keys
// 0x3f80 - d, position 0 is e = 1, the last position everything below): see nucleus_from_histogram
constexpr int kHistPos = 8192;
constexpr uint32_t kHistTopKey = 0x3f80u;
__device__ __forceinline__ void hist_count(uint32_t* hcnt, uint32_t* bad, float e)
{
    if (e > 0.0f) {
        const uint32_t key = sr_f2u(e) >> 16;
        if (key <= kHistTopKey) atomicAdd(&hcnt[min(kHistTopKey - key, (uint32_t)(kHistPos - 1))], 1u);
        else *bad = 1u;  // (no e exceeds 1; if one does, the general way takes the row)
    }
}

// Which rows take which way: asked by the passes over the whole device and by the row's workgroup alike.
// A sampled row that only min-p and top-p cut: the pass over the whole device lists what can be in its nucleus, and the
// row's workgroup finds the cut in that list.  (Not where a verifier reads e in place.)
__device__ __forceinline__ bool row_is_listed(const SrRow& rd, const SrFullArgs& a)
{
    return !a.lazy_scale && (a.mode == 0 || a.prepared) && a.seg_func != nullptr && rd.temperature > 0.0f && sr_row_cut(rd) && !(rd.top_k > 0 && rd.top_k < a.vocab);
}
// A row of the verifier whose drafts are accepted by the ratio test (SpeculativeDecoder.cs:538-548).
__device__ __forceinline__ bool spec_by_ratio(const SrRow& rd)
{
    return !(rd.p_min > 0.0f && rd.p_min < 1.0f) && (rd.flags & SR_ROWBIT_DRAFT_FROM_LOOKUP) == 0u;
}
// the longest list that its workgroup takes
__device__ __forceinline__ int list_cap(bool big) { return big ? SR_LIST_CAP_BIG : SR_LIST_CAP_SMALL; }
// A sampled row that nothing cuts.
__device__ __forceinline__ bool row_is_plain(const SrRow& rd, const SrFullArgs& a)
{
    return a.seg_func != nullptr && rd.temperature > 0.0f && !sr_row_cut(rd) && !(rd.top_k > 0 && rd.top_k < a.vocab);
}
// Rows of the verifier under the ratio test whose e no launch writes down: k_spec_factor makes it for one row of a handful (SrFullState::e_open).
__device__ __forceinline__ bool row_e_open(const SrRow& rd, const SrFullArgs& a)
{
    return a.factor_later && row_is_plain(rd, a) && spec_by_ratio(rd) && rd.edit_cnt == 0 && rd.mask_row < 0;
}
// e of a row: where it stands, or expf(x - max) of its fp32 logits, to the last bit what the pass over the whole device had.
struct ERow {
    const float* e;   // (starts on 16 bytes)
    const float* lg;  // at any address; null: e is there
    float inv_temp, max;
    const uint64_t* tab;  // of expf, in shared memory
    __device__ __forceinline__ float of(float x) const { return sr_expf_neg(__fsub_rn(__fmul_rn(x, inv_temp), max), tab); }
};
__device__ __forceinline__ float row_inv_temp(const SrRow& rd) { return rd.temperature != 1.0f ? __fdiv_rn(1.0f, rd.temperature) : 1.0f; }
// Where e = expf(x - max) of a row lies: in the work row, or, where distributions are handed out and the launches behind k_full_row
// follow, in scratch memory of its own (one place for all rows of a launch, which the host names).
__device__ __forceinline__ float* row_e(const SrFullArgs& a, int slot) { return a.e_rows + (size_t)slot * (size_t)a.e_stride; }
// the walk by slabs over the row itself, for a row in scratch memory that only top-p cuts and whose list was too long
__device__ __forceinline__ bool row_fast_nucleus(const SrRow& rd, const SrFullArgs& a)
{
    const bool use_top_p = rd.top_p < 1.0f && rd.top_p > 0.0f;
    return use_top_p && !(rd.top_k > 0 && rd.top_k < a.vocab) && !(rd.min_p > 0.0f) && a.mode == 0 && a.vocab >= 8 &&
           a.vocab <= (1 << kTagIndexBits) && a.sort_stride >= a.vocab;
}
// the row's maximum in SrFullState: this launch's number in front of the key, and what the word holds of this launch
__device__ __forceinline__ unsigned long long full_maxkey(const SrFullArgs& a, uint32_t key)
{
    return ((unsigned long long)a.seq << 32) | (unsigned long long)key;
}
__device__ __forceinline__ uint32_t full_maxkey_of(const SrFullArgs& a, unsigned long long word)
{
    return (uint32_t)(word >> 32) == a.seq ? (uint32_t)word : 0u;
}

// ---- stage 1: the masked (and temperature-scaled) copy of the row ------------------------------------
template <int ES>
__global__ __launch_bounds__(256) void k_full_prep(SrFullArgs a)
{
    const int slot = blockIdx.y;
    const int row = a.row_list[slot];
    const SrRow rd = a.rows[row];
    float* w = a.work + (size_t)(a.work_by_row ? row : slot) * a.work_stride;
    RowSource<ES> src;
    src.rowp = (const char*)a.logits + (size_t)row * (size_t)a.row_stride * ES;
    src.mrow = (rd.mask_row >= 0) ? a.mask + (size_t)rd.mask_row * a.mask_stride : nullptr;
    src.scale = rd.temperature > 0.0f && rd.temperature != 1.0f;
    src.inv_temp = src.scale ? __fdiv_rn(1.0f, rd.temperature) : 1.0f;
    if (row_is_direct(rd, a)) return;  // the kernels behind read the logits themselves
    stream_row<ES>(src, a.vocab, [&](int i, const float (&x)[16 / ES], int c, uint32_t) { store_run(w, i, x, c); });
}

// ---- stage 2: logit bias and history penalties on the few ids they touch (Sampler.cs:51-58, :367-419)
template <int ES>
__global__ __launch_bounds__(256) void k_full_edits(SrFullArgs a)
{
    const int slot = blockIdx.x;
    const int row = a.row_list[slot];
    const SrRow rd = a.rows[row];
    if (rd.edit_cnt <= 0) return;
    const SrEdit* ed = a.edits + rd.edit_off;
    if (a.edits_in_pass && row_edits_on_the_fly(rd, a)) return;  // (k_full_softmax_seg applies them where it loads the row)
    if (row_edits_on_the_fly(rd, a)) {
        // the row's bitmap (cleared first: the barrier's wait for the stores stands between them and the atomics on
        // the same words), the adjusted and scaled values of its edits, and their share of the row's maximum
        const int words = (a.vocab + 31) / 32;
        uint32_t* tab = a.edit_tab + (size_t)slot * (size_t)a.edit_tab_stride;
        float* vals = (float*)(tab + words);
        for (int i = threadIdx.x; i < words; i += 256) tab[i] = 0u;
        sr_drain_stores();  // (not a fence: a release at device scope writes the whole L2 back)
        __syncthreads();
        const char* rowp = (const char*)a.logits + (size_t)row * (size_t)a.row_stride * ES;
        const uint32_t* mrow = (rd.mask_row >= 0) ? a.mask + (size_t)rd.mask_row * a.mask_stride : nullptr;
        const bool scale = rd.temperature != 1.0f;
        const float inv_temp = scale ? __fdiv_rn(1.0f, rd.temperature) : 1.0f;
        const bool pen = (rd.flags & SR_ROWFLAG_HAS_PENALTY) != 0u;
        uint32_t k = 0u;
        for (int e = threadIdx.x; e < rd.edit_cnt; e += 256) {
            const int id = ed[e].id;
            atomicOr(&tab[id >> 5], 1u << (id & 31));
            float x = load_logit<ES>(rowp, id);
            if (mrow && !((mrow[id >> 5] >> (id & 31)) & 1u)) x = SR_NEG_INF;
            x = edited_logit(x, ed[e], rd, true, pen);
            if (scale) x = __fmul_rn(x, inv_temp);
            vals[e] = x;
            const uint32_t kv = (x != x) ? 0xffffffffu : sr_okey(x);  // NaN propagates (TensorPrimitives.Max)
            k = kv > k ? kv : k;
        }
        k = sr_wave_max_u32(k);
        if (sr_lane() == 0 && k != 0u) atomicMax(&a.state[slot].maxkey, full_maxkey(a, k));
        return;
    }
    const char* rowp = (const char*)a.logits + (size_t)row * (size_t)a.row_stride * ES;
    float* w = a.work + (size_t)(a.work_by_row ? row : slot) * a.work_stride;
    const uint32_t* mrow = (rd.mask_row >= 0) ? a.mask + (size_t)rd.mask_row * a.mask_stride : nullptr;
    const bool sampled = rd.temperature > 0.0f;
    const bool scale = sampled && rd.temperature != 1.0f;
    const float inv_temp = scale ? __fdiv_rn(1.0f, rd.temperature) : 1.0f;
    const bool pen = (rd.flags & SR_ROWFLAG_HAS_PENALTY) != 0u;
    for (int e = threadIdx.x; e < rd.edit_cnt; e += 256) {
        const int id = ed[e].id;
        float x = load_logit<ES>(rowp, id);
        if (mrow && !((mrow[id >> 5] >> (id & 31)) & 1u)) x = SR_NEG_INF;
        x = edited_logit(x, ed[e], rd, sampled, pen);
        if (scale) x = __fmul_rn(x, inv_temp);
        w[id] = x;
    }
}

// ---- stage 2b: the row maximum and expf(x - max) of the sampled rows, spread over the whole device ------
// (Softmax, Sampler.cs:448-459.)  One workgroup per row would spend most of its time in the double-precision
// expf of 150 thousand entries; here every row is cut into up to 64 pieces.
template <int ES>
__global__ __launch_bounds__(256) void k_full_max(SrFullArgs a)
{
    __shared__ uint32_t wmax[4];
    const int slot = blockIdx.y;
    const int row = a.row_list[slot];
    const SrRow rd = a.rows[row];
    if (rd.temperature <= 0.0f) return;  // greedy rows keep their logits
    uint32_t k = 0u;
    auto fold = [&](float v) {
        const uint32_t kv = (v != v) ? 0xffffffffu : sr_okey(v);  // NaN propagates (TensorPrimitives.Max)
        k = kv > k ? kv : k;
    };
    if (row_is_direct(rd, a)) {
        RowSource<ES> src;
        src.rowp = (const char*)a.logits + (size_t)row * (size_t)a.row_stride * ES;
        src.mrow = (rd.mask_row >= 0) ? a.mask + (size_t)rd.mask_row * a.mask_stride : nullptr;
        src.scale = rd.temperature != 1.0f;
        src.inv_temp = src.scale ? __fdiv_rn(1.0f, rd.temperature) : 1.0f;
        // (ids that the row's edits touch are not looked at: k_full_edits has folded their adjusted values in)
        src.erow = rd.edit_cnt > 0 ? a.edit_tab + (size_t)slot * (size_t)a.edit_tab_stride : nullptr;
        stream_row<ES>(src, a.vocab, [&](int, const float (&x)[16 / ES], int c, uint32_t hit) {
#pragma unroll
            for (int q = 0; q < 16 / ES; q++)
                if (q < c && ((hit >> q) & 1u) == 0u) fold(x[q]);
        });
    } else {
        RowSource<4> src;  // the adjusted copy
        src.rowp = (const char*)(a.work + (size_t)(a.work_by_row ? row : slot) * a.work_stride);
        src.mrow = nullptr;
        src.scale = false;
        src.inv_temp = 1.0f;
        stream_row<4>(src, a.vocab, [&](int, const float (&x)[4], int c, uint32_t) {
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (q < c) fold(x[q]);
        });
    }
    k = sr_wave_max_u32(k);
    if (sr_lane() == 0) wmax[sr_wave_id()] = k;
    __syncthreads();
    if (threadIdx.x == 0) {
        k = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
        if (k != 0u) atomicMax(&a.state[slot].maxkey, full_maxkey(a, k));
    }
}
template <int ES>
__global__ __launch_bounds__(256) void k_full_exp(SrFullArgs a)
{
    const int slot = blockIdx.y;
    const int row = a.row_list[slot];
    const SrRow rd = a.rows[row];
    if (rd.temperature <= 0.0f) return;
    const uint32_t mk = full_maxkey_of(a, a.state[slot].maxkey);
    if (mk == 0xffffffffu || mk <= 0x007fffffu) return;  // NaN, or nothing above -inf: the row kernel makes it uniform
    const float m = sr_okey_inv(mk);
    __shared__ uint64_t tab[32];  // the expf table: a lookup per element from global memory is a long dependent load
    if (threadIdx.x < 32) tab[threadIdx.x] = sr_exp2f_tab[threadIdx.x];
    __syncthreads();
    float* w = a.work + (size_t)(a.work_by_row ? row : slot) * a.work_stride;
    if (row_is_direct(rd, a)) {
        RowSource<ES> src;
        src.rowp = (const char*)a.logits + (size_t)row * (size_t)a.row_stride * ES;
        src.mrow = (rd.mask_row >= 0) ? a.mask + (size_t)rd.mask_row * a.mask_stride : nullptr;
        src.scale = rd.temperature != 1.0f;
        src.inv_temp = src.scale ? __fdiv_rn(1.0f, rd.temperature) : 1.0f;
        // (what is written for an id that the row's edits touch does not matter: k_full_row writes it again)
        stream_row<ES>(src, a.vocab, [&](int i, const float (&x)[16 / ES], int c, uint32_t) {
            float e[16 / ES];
#pragma unroll
            for (int q = 0; q < 16 / ES; q++) e[q] = q < c ? sr_expf_tab(__fsub_rn(x[q], m), tab) : 0.0f;
            store_run(w, i, e, c);
        });
    } else {
        RowSource<4> src;  // the adjusted copy, replaced in place
        src.rowp = (const char*)w;
        src.mrow = nullptr;
        src.scale = false;
        src.inv_temp = 1.0f;
        stream_row<4>(src, a.vocab, [&](int i, const float (&x)[4], int c, uint32_t) {
            float e[4];
#pragma unroll
            for (int q = 0; q < 4; q++) e[q] = q < c ? sr_expf_tab(__fsub_rn(x[q], m), tab) : 0.0f;
            store_run(w, i, e, c);
        });
    }
}

// ---- the same in one pass, laid out for a denominator that the whole device prepares ---------------------------
// (launches of rows of SR_SEG_MIN_VOCAB to SR_SEG_MAX x SR_SEG_TERMS entries, at any address: a.seg_func is set.)  A wave takes whole
// segments of SR_SEG_TERMS elements, in the end every lane 16 consecutive ones, and leaves beside e = expf(x - max) the
// record of the segment's exact sum (SeqSegFunc) for the row's workgroup to walk (seg_walk).  The binade that a record is
// made for comes from the segments' approximate sums of e.  The ids that a row's edits touch take their adjusted values as the
// pass loads them (seg_apply_edits), or from the row's adjusted copy, where it keeps one: e is final when the pass has written it.
template <int ES>
struct SegSource {
    const char* rowp;      // the row's logits, or null: the adjusted copy in w
    const uint32_t* mrow;
    const float* w;
    bool scale;
    float inv_temp;
};
template <int ES>
__device__ __forceinline__ SegSource<ES> seg_source(const SrRow& rd, const SrFullArgs& a, int slot, int row)
{
    SegSource<ES> src;
    src.w = a.work + (size_t)(a.work_by_row ? row : slot) * a.work_stride;  // (the adjusted copy, where the row keeps one)
    src.rowp = nullptr;
    src.mrow = nullptr;
    src.scale = false;
    src.inv_temp = 1.0f;
    if (row_is_direct(rd, a)) {
        src.rowp = (const char*)a.logits + (size_t)row * (size_t)a.row_stride * ES;
        src.mrow = (rd.mask_row >= 0) ? a.mask + (size_t)rd.mask_row * a.mask_stride : nullptr;
        src.scale = rd.temperature != 1.0f;
        src.inv_temp = src.scale ? __fdiv_rn(1.0f, rd.temperature) : 1.0f;
    }
    return src;
}
// The wave's segment as it is loaded: vectors of E elements, lane l the vectors l, 64 + l, ... of the segment, so that every
// load instruction of the wave covers consecutive memory.  x[E k + q] is element (k 64 + l) E + q of the segment; -inf past the
// row's end.  fp32: 4.  bf16: 8, or 4 in launches that write e through to memory as they go (out_now), where with eight a store
// instruction leaves every second 16 bytes of its lines to the next one: 64 penalised rows of 151,936 48.3 -> 41.8 us, of 65,537 34.3 -> 30.7, 24 of
// 262,144 42.9 -> 38.6; launches whose e goes to the caches lose 0.5 - 2 % by the narrower loads (32 ragged rows of 100,003 51.9 -> 52.3).
template <int ES, int E> __device__ __forceinline__ uint4 seg_load_vec(const char* p)  // the vector's bits
{
    if (ES * E == 16) return sr_load16<ES>(p);
    const uint2 v = sr_load8<ES>(p);
    return make_uint4(v.x, v.y, 0u, 0u);
}
template <int E>
__device__ __forceinline__ int seg_elem(int seg, int lane, int slot_kq)
{
    return seg * SR_SEG_TERMS + ((slot_kq / E) * SR_WAVE + lane) * E + (slot_kq % E);
}
template <int ES, int E>
__device__ __forceinline__ void seg_load_logits(const SegSource<ES>& src, int seg, int lane, int n, float (&x)[SR_SEQ_RUN])
{
    constexpr int K = SR_SEG_TERMS / (SR_WAVE * E);
    static_assert(K * E == SR_SEQ_RUN, "sixteen elements per lane");
    if (SR_USUAL((seg + 1) * SR_SEG_TERMS <= n)) {
        // a whole segment (all but a row's last): every load is issued before anything is done with one of them
        if (src.rowp) {
            uint4 raw[K];
            uint32_t keep[K];
#pragma unroll
            for (int k = 0; k < K; k++) {
                const int i0 = seg * SR_SEG_TERMS + (k * SR_WAVE + lane) * E;
                raw[k] = seg_load_vec<ES, E>(src.rowp + (size_t)i0 * ES);
            }
            if (src.mrow) {
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const int i0 = seg * SR_SEG_TERMS + (k * SR_WAVE + lane) * E;
                    keep[k] = src.mrow[i0 >> 5] >> (i0 & 31);
                }
            }
#pragma unroll
            for (int k = 0; k < K; k++) {
                float* xv = &x[k * E];
                if (ES == 4) {
                    xv[0] = sr_u2f(raw[k].x); xv[1] = sr_u2f(raw[k].y); xv[2] = sr_u2f(raw[k].z); xv[3] = sr_u2f(raw[k].w);
                } else {
                    const uint32_t r[4] = {raw[k].x, raw[k].y, raw[k].z, raw[k].w};
#pragma unroll
                    for (int q = 0; q < E / 2; q++) {
                        xv[2 * q] = sr_u2f(r[q] << 16);
                        xv[2 * q + 1] = sr_u2f(r[q] & 0xffff0000u);
                    }
                }
            }
            // (each behind one test for the whole row: as selections per element they were a seventh of the pass's instructions
            // in rows that have neither)
            if (src.mrow) {
#pragma unroll
                for (int k = 0; k < K; k++)
#pragma unroll
                    for (int q = 0; q < E; q++) x[k * E + q] = ((keep[k] >> q) & 1u) ? x[k * E + q] : SR_NEG_INF;
            }
            if (src.scale) {
#pragma unroll
                for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = __fmul_rn(x[j], src.inv_temp);
            }
        } else {
            float4 rw[K * E / 4];
#pragma unroll
            for (int k = 0; k < K; k++)
#pragma unroll
                for (int q4 = 0; q4 < E / 4; q4++)
                    rw[k * (E / 4) + q4] = sr_load_f4(src.w + seg * SR_SEG_TERMS + (k * SR_WAVE + lane) * E + 4 * q4);
#pragma unroll
            for (int v = 0; v < K * E / 4; v++) {
                x[4 * v] = rw[v].x; x[4 * v + 1] = rw[v].y; x[4 * v + 2] = rw[v].z; x[4 * v + 3] = rw[v].w;
            }
        }
        return;
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int i0 = seg * SR_SEG_TERMS + (k * SR_WAVE + lane) * E;
        float* xv = &x[k * E];
        if (i0 >= n) {
#pragma unroll
            for (int q = 0; q < E; q++) xv[q] = SR_NEG_INF;
            continue;
        }
        const bool whole = i0 + E <= n;
        if (!src.rowp) {  // the adjusted copy
#pragma unroll
            for (int q4 = 0; q4 < E; q4 += 4) {
                if (whole) {
                    const float4 v = sr_load_f4(src.w + i0 + q4);
                    xv[q4] = v.x; xv[q4 + 1] = v.y; xv[q4 + 2] = v.z; xv[q4 + 3] = v.w;
                } else {
#pragma unroll
                    for (int q = q4; q < q4 + 4; q++) xv[q] = (i0 + q < n) ? src.w[i0 + q] : SR_NEG_INF;
                }
            }
            continue;
        }
        uint32_t keep = (1u << E) - 1u;
        if (src.mrow) keep = src.mrow[i0 >> 5] >> (i0 & 31);
        if (whole) {
            const uint4 v = seg_load_vec<ES, E>(src.rowp + (size_t)i0 * ES);
            if (ES == 4) {
                xv[0] = sr_u2f(v.x); xv[1] = sr_u2f(v.y); xv[2] = sr_u2f(v.z); xv[3] = sr_u2f(v.w);
            } else {
                const uint32_t r[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int q = 0; q < E / 2; q++) {
                    xv[2 * q] = sr_u2f(r[q] << 16);
                    xv[2 * q + 1] = sr_u2f(r[q] & 0xffff0000u);
                }
            }
        } else {
#pragma unroll
            for (int q = 0; q < E; q++) xv[q] = (i0 + q < n) ? load_logit<ES>(src.rowp, i0 + q) : 0.0f;
        }
#pragma unroll
        for (int q = 0; q < E; q++) {
            float v = ((keep >> q) & 1u) ? xv[q] : SR_NEG_INF;
            if (src.scale) v = __fmul_rn(v, src.inv_temp);
            xv[q] = (i0 + q < n) ? v : SR_NEG_INF;
        }
    }
}
// The ids of segment `seg` that the row's edits touch (a row that keeps no adjusted copy): their values in x, as
// seg_load_logits left them, are replaced by the adjusted ones -- LogitBias and the history penalties on the masked
// logit, then the temperature (Sampler.cs:51-58, :367-419).  entry(i, id, e) names the i-th candidate of `count`: an id and
// its place in the row's edit list; 64 candidates at a time, a lane each, then the owners of the hits take them one
// by one.
template <int ES, int E, typename Entry>
__device__ __forceinline__ void seg_apply_edits(const SrFullArgs& a, const SrRow& rd, const SegSource<ES>& src, int seg, int lane,
                                                int count, Entry entry, float (&x)[SR_SEQ_RUN])
{
    const SrEdit* ed = a.edits + rd.edit_off;
    const bool pen = (rd.flags & SR_ROWFLAG_HAS_PENALTY) != 0u;
    const int lo = seg * SR_SEG_TERMS;
    for (int base = 0; base < count; base += SR_WAVE) {
        int id = -1;
        float val = 0.0f;
        if (base + lane < count) {
            int e = 0;
            entry(base + lane, id, e);
            if (id >= lo && id < lo + SR_SEG_TERMS && id < a.vocab) {
                float v = load_logit<ES>(src.rowp, id);
                if (src.mrow && !((src.mrow[id >> 5] >> (id & 31)) & 1u)) v = SR_NEG_INF;
                v = edited_logit(v, ed[e], rd, true, pen);
                val = src.scale ? __fmul_rn(v, src.inv_temp) : v;
            } else {
                id = -1;
            }
        }
        unsigned long long todo = __ballot(id >= 0);
        while (todo != 0ull) {
            const int h = __ffsll((long long)todo) - 1;
            todo &= todo - 1ull;
            const int local = __shfl(id, h) - lo;
            const float vh = __shfl(val, h);
            const int v = local / E, j = (v / SR_WAVE) * E + local % E;
            const bool mine = lane == v % SR_WAVE;
#pragma unroll
            for (int jj = 0; jj < SR_SEQ_RUN; jj++) x[jj] = (mine && jj == j) ? vh : x[jj];
        }
    }
}

// Everything is one launch (k_full_softmax_seg): a wave keeps its segments in registers, so the logits are read once.  The
// workgroups of a row meet twice: each leaves its largest logit, and when it has everyone's computes e = expf(x - max), leaves its
// segments' sums (and, for rows that top-p cuts, its share of the row's mass by size of e), and when it has everyone's makes
// the segments' records from the sums in front of them.  Workgroups start in
// the order of their numbers, a row's side by side, so those that a waiting workgroup waits for are running or next to
// start; the waits are bounded all the same: a workgroup whose wait runs out marks the row (SrFullState::late), leaves its words
// for the others and ends, and the row's own workgroup does the whole row by itself from the logits (row_alone).
// What is left at a meeting carries the launch's number (SrFullArgs::meet), so that the poll that finds it has it: a maximum and a count of
// the row by atomics, polled and then read, were four trips to memory one behind the other, and the atomics of a row queue.  41 meetings in a row on
// their own, us each, atomics and words: 19 workgroups x 64 rows 5.6 and 2.4, 13 x 32 2.7 and 1.3, 32 x 16 3.8 and 2.3; the second,
// whose sums were written through, waited for, counted and read, 4.1 and 2.6, 2.2 and 1.5, 2.8 and 2.0.  Of calls, where the slowest
// workgroup is waited for either way: 16 rows of 262,144 fp32 with distributions 65.0 -> 63.4, 32 ragged bf16 rows of 100,003 52.0 -> 50.8, 64
// penalised rows of 151,936 41.15 -> 40.7.
// Where tokens are all that is asked for, the first meeting also has about the sum of the row's exponentials, relative to its largest: fast
// ones of the logits in the registers, a dozen cycles each.  With it a row whose largest entry decides (row_decided) is done there -- no e, no
// records, no list, nothing for the launches behind --, and any other row that is not cut by its mass needs no second meeting.  us a call,
// before -> now, rows whose largest entry stands out and flat ones (N(0, 1.5^2)): 64 rows of 151,936 under min-p 37.6 -> 14.7 and 49.4 -> 48.5, 16
// of them 28.2 -> 10.8 and 40.1 -> 36.0; 32 bf16 rows of 100,003 under top-p 30.2 -> 13.1 and 680 -> 684, that nothing cuts 50.4 -> 13.1 and 47.5 ->
// 47.2; one row of 151,936 38.3 -> 13.3 and 39.5 -> 37.8, 64 83.7 -> 50.9 (one of them open) and 82.1 -> 80.4.
//
// What bounds it: the vector units (the double-precision expf is 30 instructions an element).  The first pass used to
// take a fast exponential of every element, for approximate sums relative to the segment's own maximum, to save the second
// meeting; the sums come from e itself now, which costs a meeting of 2 - 3 us and a quarter fewer instructions.

constexpr uint32_t kKeyInf = 0xff800000u;  // +inf as an ordered key; above it: a NaN
// a segment's largest value as an ordered key; 0xffffffff = it holds a NaN (which propagates: TensorPrimitives.Max)
__device__ __forceinline__ uint32_t seg_max_key(const float (&x)[SR_SEQ_RUN])
{
    static_assert(SR_SEQ_RUN % 2 == 0, "the first, then two at a time, then the last");
    float m = sr_max_f32(x[0], x[SR_SEQ_RUN - 1]);
    bool nan = false;
#pragma unroll
    for (int j = 1; j + 1 < SR_SEQ_RUN; j += 2) m = sr_max3_f32(m, x[j], x[j + 1]);
#pragma unroll
    for (int j = 0; j < SR_SEQ_RUN; j += 2) nan = nan || __builtin_isunordered(x[j], x[j + 1]);
    return nan ? 0xffffffffu : sr_okey(m);
}
// The mass of a row's e by size: kMassBuckets buckets, eight to a doubling, bucket 0 just below 1, the last one everything
// small.  From the sums over all of the row: the smallest value (as bits) whose bucket still has to be listed for the
// listed entries to hold `share` of the row's mass and a little more; *least = that many entries the list has at least (a
// bucket's mass over its largest value; the values of a bucket differ by an eighth at most).
constexpr int kMassBuckets = 256;
// A workgroup adds up its share in whole numbers: an entry e in (0, 1], x = 0x3f800000 - its bits, is 2^24 - x mod 2^23 units of
// 2^(-24 - k) where k = x >> 23 counts the doublings down from 1, the same for all of a bucket; the upper 17 bits of that, added
// over the 16,384 entries of the largest workgroup, fit 32.  (In shared memory an atomic addition of floats takes a wave
// some 190 cycles here, whatever the addresses: two, four or eight copies of the table changed nothing.  The pass over 64 rows of
// 151,936 at temperature 2, where most entries are counted: 81 us with floats, 34 with whole numbers, 33 without the table.)
constexpr int kMassDrop = 7;
__device__ __forceinline__ uint32_t mass_units(uint32_t x) { return (0x01000000u - (x & 0x7fffffu)) >> kMassDrop; }
__device__ __forceinline__ float mass_of_units(uint32_t units, int bucket)
{
    return (float)units * sr_u2f((uint32_t)(127 - 24 + kMassDrop - (bucket >> 3)) << 23);
}
__device__ __forceinline__ uint32_t mass_list_from(const float (&v)[4], float share, float* least)
{
    static_assert(kMassBuckets == 4 * SR_WAVE, "four buckets per lane");
    const int lane = sr_lane();
    const float own = (v[0] + v[1]) + (v[2] + v[3]);
    const float incl = sr_wave_incl_sum_f32(own);
    const float total = sr_u2f((uint32_t)__builtin_amdgcn_readlane((int)sr_f2u(incl), SR_WAVE - 1));
    const float target = share * total * 1.0005f;
    float c = incl - own;
    int d = kMassBuckets;
#pragma unroll
    for (int q = 3; q >= 0; q--) {
        float upto = c;
#pragma unroll
        for (int k = 0; k <= q; k++) upto += v[k];
        if (upto >= target) d = 4 * lane + q;
    }
    d = sr_wave_min_i32(d);
    float c_least = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; q++)  // (the last bucket's entries are of any size below the others')
        if (4 * lane + q <= min(d, kMassBuckets - 2)) c_least += v[q] * __builtin_amdgcn_rcpf(sr_u2f(0x3f800000u - ((uint32_t)(4 * lane + q) << 20)));
    *least = 0.99f * sr_wave_sum_f32(c_least);  // (sums and reciprocals are rounded)
    if (d >= kMassBuckets - 1) return 1u;  // everything above zero
    return 0x3f800000u - ((uint32_t)(d + 1) << 20) + 1u;
}

// The smallest e that can be a survivor of the row's min-p or so near its threshold that the row counts as ambiguous: the
// probabilities fl(e inv) and the threshold fl(min_p inv) are three roundings apart at most -- where they are normal
// numbers (inv is 1 / 2^20 at least); a smaller min_p bounds nothing.
__device__ __forceinline__ uint32_t min_p_list_from(const SrRow& rd)
{
    return rd.min_p >= 1e-30f ? sr_f2u(__fmul_rn(rd.min_p, 1.0f - 2.0f * SR_AMBIG_REL - 1e-6f)) : 0u;
}

constexpr float kLog2E = 0x1.715476p+0f;
// Whether a row's largest entry, e = 1, is its token: its nucleus is that entry alone, or, in a row that nothing cuts, the draw lands
// on it.  all: about the sum of the row's e, front: of what stands in front of the workgroup that holds the largest, own: of what that one holds
// (fast exponentials: 2e-5 at most).  The exact sums go one by one in fp32 and end near these: an addition is off by 2^-24 of the sum at most, and by the
// smaller of its two operands at most, so n of them by n 2^-24 of the sum and by the mass beside the largest entry, whichever is less; the eight
// accumulators of the final Normalize by n / 8 + 200 roundings.  What lies nearer to a line than that is not decided here, nor is anything that
// could count as ambiguous: draws at either end, cuts beside the threshold, a largest entry that is not the only one (it covers more than half).
__device__ __forceinline__ bool row_decided(const SrRow& rd, int n, float all, float front, float own, float u)
{
    const float by_n = (float)n * 6.3e-8f, beside = fmaxf(all - 1.0f, 0.0f) + 4e-5f * all;
    const float least = (1.0f - 1e-5f) / (all * (1.0f + 4e-5f) + fminf(all * by_n, beside));  // its probability is at least this
    const bool use_top_p = rd.top_p < 1.0f && rd.top_p > 0.0f, use_min_p = rd.min_p > 0.0f;
    bool yes = all < 1e30f && least > 0.505f && u > 2e-6f && u < 1.0f - 4e-6f;
    if (use_min_p) yes = yes && rd.min_p < 0.99f && beside < 0.999f * rd.min_p;  // (nothing else survives)
    if (use_top_p) yes = yes && rd.top_p > 1e-5f && least > rd.top_p;            // (the running sum stops at the first)
    if (!use_top_p && !use_min_p) {
        const float inv = 1.0f / all, off = fminf(by_n, beside * inv) * 1.05f + ((float)(n / 8) + 200.0f) * 6.6e-8f + 8e-5f;
        yes = yes && u > (front + fmaxf(own - 1.0f, 0.0f)) * inv + off && u < (front + 1.0f) * inv - off;
    }
    return yes;
}

// A greedy row that rides along (SrFullArgs::n_greedy): the largest of its masked logits, the first by index among equals, NaN left
// out -- what the selection kernel finds for such a row.  The row's word for it is zero between launches: whoever counts in last
// takes the result and puts the zero back.
template <int ES, int kW, int kS, int E>
__device__ __forceinline__ void seg_greedy(const SrFullArgs& a, const SrRow& rd, int slot, int row, unsigned long long* of_wave)
{
    const int lane = sr_lane(), wave = sr_wave_id(), n = a.vocab, nseg = seg_count(n);
    SegSource<ES> src;
    src.rowp = (const char*)a.logits + (size_t)row * (size_t)a.row_stride * ES;
    src.mrow = (rd.mask_row >= 0) ? a.mask + (size_t)rd.mask_row * a.mask_stride : nullptr;
    src.w = nullptr;
    src.scale = false;
    src.inv_temp = 1.0f;
    const int seg0 = (int)blockIdx.x * (kW * kS) + wave;
    float t[kS][SR_SEQ_RUN];
#pragma unroll
    for (int s = 0; s < kS; s++)
        if (seg0 + s * kW < nseg) seg_load_logits<ES, E>(src, seg0 + s * kW, lane, n, t[s]);
    unsigned long long best = 0ull;  // ordered key << 32 | ~index; 0: nothing above -inf
#pragma unroll
    for (int s = 0; s < kS; s++) {
        const int seg = seg0 + s * kW;
        if (seg >= nseg) continue;
        float m = sr_max_f32(t[s][0], t[s][SR_SEQ_RUN - 1]);
#pragma unroll
        for (int j = 1; j + 1 < SR_SEQ_RUN; j += 2) m = sr_max3_f32(m, t[s][j], t[s][j + 1]);
        const uint32_t k = sr_wave_max_u32(m == m ? sr_okey(m) : 0u);
        if (k <= 0x007fffffu || k < (uint32_t)(best >> 32)) continue;
        const float mk = sr_okey_inv(k);
        int at = 0x7fffffff;
#pragma unroll
        for (int j = SR_SEQ_RUN - 1; j >= 0; j--)
            if (t[s][j] == mk) at = min(at, seg_elem<E>(seg, lane, j));
        at = sr_wave_min_i32(at);
        const unsigned long long found = ((unsigned long long)k << 32) | (unsigned long long)(0xffffffffu - (uint32_t)at);
        best = found > best ? found : best;
    }
    if (lane == 0) of_wave[wave] = best;
    sr_barrier_lds();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 0; w < kW; w++) best = of_wave[w] > best ? of_wave[w] : best;
        // (each atomic's returned value is waited for before the next is issued: whoever counts in last finds the result complete)
        unsigned long long* const sync = a.row_sync + (size_t)slot * SR_ROW_SYNC_STRIDE;
        const unsigned long long s0 = __hip_atomic_fetch_max(sync, (unsigned long long)a.seq << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long s1 = __hip_atomic_fetch_max(sync + 2, best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" : : "v"(s0), "v"(s1) : "memory");
        const unsigned long long was = __hip_atomic_fetch_add(sync, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (((uint32_t)was & 0xffffu) + 1u == gridDim.x) {
            const unsigned long long r = __hip_atomic_exchange(sync + 2, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // (nothing above -inf: every masked logit is -inf and the first index wins)
            a.out_tokens[row] = r != 0ull ? (int)(0xffffffffu - (uint32_t)r) : 0;
            if (a.out_flags) a.out_flags[row] = SR_KFLAG_GREEDY | (r != 0ull ? 0u : SR_KFLAG_DEGENERATE);
        }
    }
}

// kLists: the launch may have rows that list their candidates, and greedy ones (not the verifier's).
// kLater: a verifier's launch with factor_later (144 rows of 131,072, which do without, were 2 us slower with the test in it)
template <int ES, int kW, int kS, bool kLater = false, int E = 16 / ES, bool kLists = kS != 4>
__global__ __launch_bounds__(kW * SR_WAVE, kS == 4 ? 5 : 6) void k_full_softmax_seg(SrFullArgs a)
{
    constexpr int kThreads = kW * SR_WAVE;
    constexpr int K = SR_SEG_TERMS / (SR_WAVE * E);
    static_assert(kW == SR_HALF_BLOCK_SEGS, "a workgroup's segments are whole half blocks");
    const int slot = blockIdx.y, lane = sr_lane(), wave = sr_wave_id();
    const int row = a.row_list[slot];
    const SrRow rd = a.rows[row];
    __shared__ uint64_t tab[32];  // the expf table: a lookup per element from global memory is a long dependent load
    // a wave's segment on its way from the order of the loads to 16 terms a lane: a lane's 16 terms lie together, 16
    // bytes apart from the next lane's, so that neither the stores nor the loads of 16 bytes a lane collide on a bank
    __shared__ float4 turn_all[kW][SR_WAVE * 5];
    float* const share = (float*)&turn_all[0][0];  // every segment's part of the row's sum (behind the second meeting)
    static_assert(SR_SEG_MAX * sizeof(float) <= sizeof(turn_all), "in the same place");
    __shared__ uint32_t mass[kMassBuckets];  // this workgroup's part of the row's mass by size of e (mass_units)
    __shared__ float mass_rest;              // ... of its last bucket
    __shared__ float chains[kS][SR_SEQ_CHAINS];
    __shared__ uint32_t wkey[kW];
    __shared__ float wsum[kW];
    // 0: the row's words came in, and 2: its largest entry decides   1: the row's maximum   2: about the sum of e in front of the workgroup
    __shared__ uint32_t bc[3];
    // the row's edits that fall into this workgroup's segments (id << 32 | place in the row's edit list), and how many
    // there are (more than the list holds: the waves go through the row's whole edit list instead)
    constexpr int kHitCap = 256;
    __shared__ unsigned long long hits[kHitCap];
    __shared__ uint32_t n_hits;
    if (SR_RARE(rd.temperature <= 0.0f)) {  // greedy rows keep their logits where a distribution is asked for
        if (kLists && a.mode == 0) seg_greedy<ES, kW, kS, E>(a, rd, slot, row, hits);
        return;
    }
    const int n = a.vocab, nseg = seg_count(n);
    SrFullState* st = a.state + slot;
    const unsigned long long stamp = (unsigned long long)a.seq << 32;
    unsigned long long* const met_max = a.meet + (size_t)slot * a.meet_stride;  // two words per workgroup
    unsigned long long* const met_sum = met_max + a.meet_sums;                  // ... and per segment
    SeqSegFunc* recs = a.seg_func + (size_t)slot * a.seg_stride;
    float* sums = a.seg_sum + (size_t)slot * a.seg_stride;
    if (threadIdx.x < 32) tab[threadIdx.x] = sr_exp2f_tab[threadIdx.x];
    const SegSource<ES> src = seg_source<ES>(rd, a, slot, row);
    float* const w = row_e(a, slot);
    const bool plain = a.prepared && row_is_plain(rd, a), listed = kLists && row_is_listed(rd, a);
    const bool use_top_p = rd.top_p < 1.0f && rd.top_p > 0.0f;
    const bool out_now = !a.prepared && ((uintptr_t)w & 15u) == 0u, open_e = kLater && row_e_open(rd, a);
    // (a row that min-p cuts as well lists everything down to its threshold: entries on it count for SR_OUT_AMBIGUOUS wherever
    // top-p ends)
    const bool by_mass = listed && use_top_p && !(rd.min_p > 0.0f);
    const bool by_count = listed && !by_mass && a.mode != 0;
    const uint32_t min_p_from = max(min_p_list_from(rd), 1u);
    // a row whose token is all that is asked for: its largest entry may decide
    const bool asks = kLists && a.mode == 0 && !(rd.top_k > 0 && rd.top_k < n);
    // (the row's sum is at least 1: n entries below this make up less than half of what top-p leaves out)
    const float mass_min = (1.0f - rd.top_p) * 0.5f / (float)n;
    if (by_mass || by_count) {
        for (int i = threadIdx.x; i < kMassBuckets; i += kThreads) mass[i] = 0u;
        if (threadIdx.x == 0) mass_rest = 0.0f;
    }
    if (plain && threadIdx.x < kS * SR_SEQ_CHAINS) (&chains[0][0])[threadIdx.x] = 0.0f;

    // A row that keeps no adjusted copy although bias or penalties touch some of its ids: the workgroup looks through
    // the row's edit list for the ids of its own segments, and its waves put the adjusted values in place of what they load
    // (the ids are asked for in front of the logits and looked at behind them: the loads overlap)
    const bool edits = src.rowp != nullptr && rd.edit_cnt > 0;
    const SrEdit* ed = a.edits + rd.edit_off;
    constexpr int kIds = SR_FULL_EDIT_VALUES / kThreads;
    static_assert(kIds * kThreads == SR_FULL_EDIT_VALUES, "every edit of a row without an adjusted copy is looked at");
    int ids[kIds];
    if (edits) {
        if (threadIdx.x == 0) n_hits = 0u;
        sr_barrier_lds();
#pragma unroll
        for (int j = 0; j < kIds; j++) {
            const int e = (int)threadIdx.x + j * kThreads;
            ids[j] = kS != 4 && e < rd.edit_cnt ? ed[e].id : -1;
        }
    }
    // (a wave takes kS segments, the workgroup's waves side by side: every one of its loads is out before the first is used)
    const int seg0 = (int)blockIdx.x * (kW * kS) + wave;
    float t[kS][SR_SEQ_RUN];
#pragma unroll
    for (int s = 0; s < kS; s++)
        if (seg0 + s * kW < nseg) seg_load_logits<ES, E>(src, seg0 + s * kW, lane, n, t[s]);
    if (edits) {
        const int lo = (int)blockIdx.x * (kW * kS) * SR_SEG_TERMS, hi = lo + kW * kS * SR_SEG_TERMS;
#pragma unroll
        for (int j = 0; j < kIds; j++) {
            // (beside four segments there is no room to ask for them ahead)
            if (kS == 4) ids[j] = (int)threadIdx.x + j * kThreads < rd.edit_cnt ? ed[(int)threadIdx.x + j * kThreads].id : -1;
            if (ids[j] >= lo && ids[j] < hi) {
                const uint32_t pos = atomicAdd(&n_hits, 1u);
                if (pos < (uint32_t)kHitCap)
                    hits[pos] = ((unsigned long long)(uint32_t)ids[j] << 32) | (unsigned long long)(uint32_t)((int)threadIdx.x + j * kThreads);
            }
        }
        sr_barrier_lds();
        const bool from_hits = n_hits <= (uint32_t)kHitCap;
#pragma unroll
        for (int s = 0; s < kS; s++)
            if (seg0 + s * kW < nseg)
                seg_apply_edits<ES, E>(a, rd, src, seg0 + s * kW, lane, from_hits ? (int)n_hits : rd.edit_cnt, [&](int i, int& id, int& e) {
                    if (from_hits) {
                        const unsigned long long h = hits[i];
                        id = (int)(h >> 32);
                        e = (int)(uint32_t)h;
                    } else {
                        id = ed[i].id;
                        e = i;
                    }
                }, t[s]);
    }
    double u_row = 0.0;  // (behind the logits: it may come over the bus)
    if (asks && wave == 0) u_row = a.uniforms[(size_t)row * a.uniforms_per_row];
    uint32_t k = 0u;
#pragma unroll
    for (int s = 0; s < kS; s++)
        if (seg0 + s * kW < nseg) k = max(k, seg_max_key(t[s]));
    k = sr_wave_max_u32(k);
    if (lane == 0) wkey[wave] = k;
    if (asks) {
        // about the sum of the wave's exponentials, relative to the wave's largest
        float sum = 0.0f;
        if (k > 0x007fffffu && k < kKeyInf) {
            const float mw = sr_okey_inv(k);
#pragma unroll
            for (int s = 0; s < kS; s++)
                if (seg0 + s * kW < nseg)
#pragma unroll
                    for (int j = 0; j < SR_SEQ_RUN; j++) {
                        sum += __builtin_amdgcn_exp2f((t[s][j] - mw) * kLog2E);
                        if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (a few at a time: the registers are the segments')
                    }
            sum = sr_wave_sum_f32(sum);
        }
        if (lane == 0) wsum[wave] = sum;
    }
    sr_barrier_lds();
    // The first meeting: every workgroup's largest logit, and where the row asks about the sum of its exponentials relative to that, each
    // in a word below the launch's number, which all of the row's workgroups read until it is this launch's.
    auto about = [](uint32_t key, float sum, float m) __attribute__((always_inline)) -> float {
        return key > 0x007fffffu ? sum * __builtin_amdgcn_exp2f((sr_okey_inv(key) - m) * kLog2E) : 0.0f;
    };
    uint32_t k_group = wkey[0];
#pragma unroll
    for (int j = 1; j < kW; j++) k_group = max(k_group, wkey[j]);
    if (wave == 0) {
        float sum = 0.0f;
        if (asks) {
            const float m = sr_okey_inv(k_group);
#pragma unroll
            for (int j = 0; j < kW; j++) sum += about(wkey[j], wsum[j], m);
        }
        if (lane == 0) {
            sr_store_agent(met_max + 2 * blockIdx.x, stamp | (unsigned long long)k_group);
            if (asks) sr_store_agent(met_max + 2 * blockIdx.x + 1, stamp | (unsigned long long)sr_f2u(sum));
        }
    }
    // where the workgroup's largest logit is, should it be the row's token: found while the words are under way
    int top_at = -1;
    if (asks && k == k_group) {
        const float mg = sr_okey_inv(k);
#pragma unroll
        for (int s = 0; s < kS; s++)
            if (seg0 + s * kW < nseg)
#pragma unroll
                for (int j = 0; j < SR_SEQ_RUN; j++) top_at = t[s][j] == mg ? s * SR_SEQ_RUN + j : top_at;
    }
    if (wave == 0) {
        constexpr int kWords = SR_SEG_MAX / (kW * kS) / SR_WAVE > 0 ? SR_SEG_MAX / (kW * kS) / SR_WAVE : 1;  // a lane, of each kind
        k = k_group;
        bool here = true;
        uint32_t key[kWords];
        float part[kWords];
#pragma unroll
        for (int w = 0; w < kWords; w++) {
            const int g = w * SR_WAVE + lane;
            key[w] = 0u;
            part[w] = 0.0f;
            if (g >= (int)gridDim.x) continue;
            bool in = false;
            for (uint32_t it = 0; it < a.row_wait_limit; it++) {
                const unsigned long long v = sr_load_agent(met_max + 2 * g), e = asks ? sr_load_agent(met_max + 2 * g + 1) : v;
                key[w] = (uint32_t)v;
                part[w] = sr_u2f((uint32_t)e);
                if ((uint32_t)(v >> 32) == a.seq && (uint32_t)(e >> 32) == a.seq) { in = true; break; }
                __builtin_amdgcn_s_sleep(1);
            }
            here = here && in;
            k = max(k, key[w]);
        }
        here = __ballot(!here) == 0ull;
        k = sr_wave_max_u32(k);
        bool decided = false;
        float before = 0.0f;
        if (asks && here && k > 0x007fffffu && k < kKeyInf) {
            const float m = sr_okey_inv(k);
            float all = 0.0f;
            int first = (int)gridDim.x;  // the workgroup that holds the largest entry
#pragma unroll
            for (int w = kWords - 1; w >= 0; w--) {
                part[w] = about(key[w], part[w], m);
                const unsigned long long top = __ballot(key[w] == k);
                if (top != 0ull) first = w * SR_WAVE + (int)__ffsll((long long)top) - 1;
            }
            float front = 0.0f, own = 0.0f;
#pragma unroll
            for (int w = 0; w < kWords; w++) {
                const int g = w * SR_WAVE + lane;
                all += part[w];
                before += g < (int)blockIdx.x ? part[w] : 0.0f;
                front += g < first ? part[w] : 0.0f;
                own += g == first ? part[w] : 0.0f;
            }
            before = sr_wave_sum_f32(before);
            decided = row_decided(rd, n, sr_wave_sum_f32(all), sr_wave_sum_f32(front), sr_wave_sum_f32(own), __double2float_rn(u_row));
        }
        if (lane == 0) {
            bc[0] = here ? (decided ? 2u : 1u) : 0u;
            bc[1] = k;
            bc[2] = sr_f2u(before);
            // the wait ran out: the row is left to its own workgroup
            if (!here) sr_store_agent(&st->late, a.seq);
            else if (blockIdx.x == 0) st->maxkey = full_maxkey(a, k);
        }
    }
    __syncthreads();
    if (SR_RARE(bc[0] == 0u)) {
        // (nobody waits for this one)
        if (lane == 0)
#pragma unroll
            for (int s = 0; s < kS; s++)
                if (seg0 + s * kW < nseg) sr_store_agent(met_sum + seg0 + s * kW, stamp);
        return;
    }
    const uint32_t mk = bc[1];
    // A NaN, or nothing above -inf: the row's workgroup makes it uniform.  A maximum of +inf, beside which e is no number where it
    // stands: the row's workgroup takes the row alone, so that every x - max below is at most 0, or -inf.
    if (SR_RARE(mk >= kKeyInf || mk <= 0x007fffffu)) return;
    const float m = sr_okey_inv(mk);
    if (asks && bc[0] == 2u) {
        if (wkey[wave] == mk) {
            if (top_at >= 0) a.out_tokens[row] = seg_elem<E>(seg0 + top_at / SR_SEQ_RUN * kW, lane, top_at % SR_SEQ_RUN);  // (the only one of its value)
            if (lane == 0) {
                if (a.out_flags) a.out_flags[row] = SR_KFLAG_FULL;
                st->decided = a.seq;
            }
        }
        return;
    }

    // e of the wave's segments: written to the row, counted by size, and turned into the order of the sum
    float own[kS];
    float4* const turn = turn_all[wave];
#pragma unroll
    for (int s = 0; s < kS; s++) {
        own[s] = 0.0f;
        const int seg = seg0 + s * kW;
        if (seg >= nseg) continue;
        float e[SR_SEQ_RUN];
        // (a whole segment without a test per element: the 16 chains of a lane then run interleaved)
        if (SR_USUAL((seg + 1) * SR_SEG_TERMS <= n)) {
#pragma unroll
            for (int j = 0; j < SR_SEQ_RUN; j++) e[j] = sr_expf_neg(__fsub_rn(t[s][j], m), tab);
        } else {
#pragma unroll
            for (int j = 0; j < SR_SEQ_RUN; j++) e[j] = seg_elem<E>(seg, lane, j) < n ? sr_expf_neg(__fsub_rn(t[s][j], m), tab) : 0.0f;
        }
#pragma unroll
        for (int k2 = 0; k2 < K; k2++) {
            const int i0 = seg * SR_SEG_TERMS + (k2 * SR_WAVE + lane) * E;
            if (kLater && open_e) continue;
            if (i0 + E <= n) {
#pragma unroll
                for (int q = 0; q < E; q += 4) {
                    // (rows of e start on 16 bytes.  Where no launch behind this one reads all of e, it goes out while the pass goes
                    // on, instead of from the caches at its end: 64 penalised rows of 151,936 33.9 -> 30.8 us)
                    if (out_now) sr_store_agent_f4((float4*)(w + i0 + q), e[k2 * E + q], e[k2 * E + q + 1], e[k2 * E + q + 2], e[k2 * E + q + 3]);
                    else sr_store_f4(w + i0 + q, e[k2 * E + q], e[k2 * E + q + 1], e[k2 * E + q + 2], e[k2 * E + q + 3]);
                }
            } else {
#pragma unroll
                for (int q = 0; q < E; q++)
                    if (i0 + q < n) w[i0 + q] = e[k2 * E + q];
            }
        }
        if (by_mass) {
            // (entries so small that all of them together cannot reach into the nucleus are summed in registers, as the last
            // bucket -- most of a sharp row: shared-memory atomics queue)
            float small = 0.0f;
#pragma unroll
            for (int j = 0; j < SR_SEQ_RUN; j++) {
                const uint32_t x = 0x3f800000u - sr_f2u(e[j]);
                if (e[j] >= mass_min && x < ((uint32_t)(kMassBuckets - 1) << 20)) atomicAdd(&mass[x >> 20], mass_units(x));
                else small += e[j];
            }
            small = sr_wave_sum_f32(small);
            if (lane == 0) unsafeAtomicAdd(&mass_rest, small);
        } else if (by_count) {
            // how many entries the list will have
            int c = 0;
#pragma unroll
            for (int j = 0; j < SR_SEQ_RUN; j++) c += __popcll(__ballot(sr_f2u(e[j]) >= min_p_from));
            if (lane == 0 && c > 0) atomicAdd(&mass[0], (uint32_t)c);
        }
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < SR_SEQ_RUN; j++) sum += e[j];
        own[s] = sr_wave_sum_f32(sum);
        // through shared memory into the order of the sum: lane l gets the terms 16 l ... 16 l + 15 of the segment (only
        // this wave touches its part: the wave's own order of shared-memory operations is all it needs)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
#pragma unroll
        for (int k2 = 0; k2 < K; k2++)
#pragma unroll
            for (int q = 0; q < E; q += 4) {
                const int i = (k2 * SR_WAVE + lane) * E + q;  // the element's place in the segment
                turn[(i >> 4) * 5 + ((i & 15) >> 2)] = make_float4(e[k2 * E + q], e[k2 * E + q + 1], e[k2 * E + q + 2], e[k2 * E + q + 3]);
            }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int k2 = 0; k2 < 4; k2++) {
            const float4 v = turn[lane * 5 + k2];
            t[s][4 * k2] = v.x; t[s][4 * k2 + 1] = v.y; t[s][4 * k2 + 2] = v.z; t[s][4 * k2 + 3] = v.w;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (plain) {
            // the segment's part of the eight lane accumulators of the final Normalize
            float c[SR_SEQ_CHAINS];
#pragma unroll
            for (int g = 0; g < SR_SEQ_CHAINS; g++) c[g] = t[s][g] + t[s][g + 8];
            const float mine = wave_sum_8(c);
            if (lane < SR_SEQ_CHAINS) unsafeAtomicAdd(&chains[s][lane], mine);
        }
    }
    sr_barrier_lds();
    if (by_mass) {
        for (int i = threadIdx.x; i < kMassBuckets; i += kThreads) {
            const float v = i < kMassBuckets - 1 ? mass_of_units(mass[i], i) : mass_rest;
            if (v > 0.0f) unsafeAtomicAdd(a.mass + (size_t)slot * kMassBuckets + i, v);
        }
    } else if (by_count && threadIdx.x == 0 && mass[0] > 0u) {
        unsafeAtomicAdd(a.mass + (size_t)slot * kMassBuckets, (float)mass[0]);  // (a whole number below 2^24)
    }
    if (plain && threadIdx.x < kS * SR_SEQ_CHAINS) {
        const int hb = (int)blockIdx.x * kS + (int)threadIdx.x / SR_SEQ_CHAINS;
        if (hb < a.chain_stride / SR_SEQ_CHAINS)
            a.chain_sum[(size_t)slot * a.chain_stride + (size_t)hb * SR_SEQ_CHAINS + (threadIdx.x & (SR_SEQ_CHAINS - 1))] = (&chains[0][0])[threadIdx.x];
    }
    if (by_mass || by_count) {  // (added to before the workgroup's segments count as in)
        sr_drain_stores();
        __syncthreads();
    }
    // The second one: a word of every segment, its sum -- but where the first has told all there is to ask.
    const bool meets = !asks || by_mass;
    if (!meets) {
        if (lane == 0) {
#pragma unroll
            for (int s = 0; s < kS; s++)
                if (seg0 + s * kW < nseg) share[s * kW + wave] = sums[seg0 + s * kW] = own[s];
        }
    } else if (lane == 0) {
#pragma unroll
        for (int s = 0; s < kS; s++)
            if (seg0 + s * kW < nseg) {
                sr_store_agent(met_sum + seg0 + s * kW, stamp | (unsigned long long)sr_f2u(own[s]));
                sums[seg0 + s * kW] = own[s];  // (for the launches behind)
            }
    }
    for (int g = meets ? (int)threadIdx.x : nseg; g < nseg; g += kThreads) {
        unsigned long long v = 0ull;
        bool in = false;
        for (uint32_t it = 0; it < a.row_wait_limit; it++) {
            v = sr_load_agent(met_sum + g);
            if ((uint32_t)(v >> 32) == a.seq) { in = true; break; }
            __builtin_amdgcn_s_sleep(1);
        }
        if (!in) bc[0] = 0u;
        share[g] = sr_u2f((uint32_t)v);
    }
    __syncthreads();
    if (bc[0] == 0u) {
        if (threadIdx.x == 0) sr_store_agent(&st->late, a.seq);
        return;
    }
    // (the row's mass by size, four buckets a lane, or the length of its list, on its way beside the segments' sums)
    float row_mass[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const float* const mass_at = a.mass + (size_t)slot * kMassBuckets;
    if (by_mass) {
#pragma unroll
        for (int q = 0; q < 4; q++) row_mass[q] = sr_load_agent(mass_at + 4 * lane + q);
    } else if (by_count) {
        row_mass[0] = sr_load_agent(mass_at);
    }
    // what the list of a row that is cut holds: everything that can survive its min-p, or enough of the largest for top-p
    uint32_t from = 0xffffffffu;
    bool too_long = false;
    if (listed) {
        // A list that is longer than the row's workgroup takes is not made: a flat row's held most of the row, eight bytes an
        // entry, for nothing.  Where a distribution is handed out the row goes on from e in the caller's row, and that is put
        // there from here.  Every workgroup of the row comes to the same answer from the same sums.  (Distributions of 16
        // flat rows of 151,936 that min-p cuts: 196 us with the list and a copy of the row by its one workgroup, this 138; the
        // pass over 64 rows of tokens at temperature 2, before its sums were whole numbers, 114 -> 81.  Counting costs 0.8 us of
        // 35 where min-p cuts; tokens alone gain by it only in flat rows, 16 of them 159 -> 136 us, and go without.)
        float least;
        if (by_mass) {
            from = mass_list_from(row_mass, rd.top_p, &least);
        } else {
            from = min_p_from;
            least = row_mass[0];
        }
        too_long = least > (float)list_cap(a.big_slabs != 0);
        if (blockIdx.x == 0 && threadIdx.x == 0) st->list_from = too_long ? 0u : from;
    }
#pragma unroll
    for (int s = 0; s < kS; s++) {
        const int seg = seg0 + s * kW;
        if (seg >= nseg) continue;
        float before = 0.0f;
        for (int g = lane; g < (meets ? seg : s * kW + wave); g += SR_WAVE) before += share[g];
        before = sr_wave_sum_f32(before);
        if (!meets) before += sr_u2f(bc[2]);
        seg_make_record(t[s], seg, (double)before, recs + seg, own[s]);
        if (too_long) {
            if (a.mode != 0) {  // (what is left of the row's last four, k_full_row copies)
                float* const p = a.work + (size_t)(a.work_by_row ? row : slot) * a.work_stride;
                const int i0 = seg * SR_SEG_TERMS + lane * SR_SEQ_RUN;
#pragma unroll
                for (int j = 0; j < SR_SEQ_RUN; j += 4)
                    if (i0 + j + 4 <= n) sr_store_f4(p + i0 + j, t[s][j], t[s][j + 1], t[s][j + 2], t[s][j + 3]);
            }
        } else if (listed) {
            // the segment's entries of the list, in the order of their indices, at the segment's own place in the row's lists
            uint32_t bits = 0u;
#pragma unroll
            for (int j = 0; j < SR_SEQ_RUN; j++) bits |= sr_f2u(t[s][j]) >= from ? 1u << j : 0u;
            const int mine = __popc(bits);
            const int incl = sr_wave_incl_scan_i32(mine);
            if (lane == SR_WAVE - 1) a.seg_cnt[(size_t)slot * a.seg_stride + seg] = (uint32_t)incl;
            size_t at = (size_t)slot * (size_t)a.sort_stride + (size_t)seg * SR_SEG_TERMS + (size_t)(incl - mine);
            if (__ballot(bits != 0u) != 0ull) {
#pragma unroll
                for (int j = 0; j < SR_SEQ_RUN; j++)
                    if ((bits >> j) & 1u) {
                        a.sort_keys_in[at] = sr_f2u(t[s][j]);
                        a.sort_vals_in[at] = seg * SR_SEG_TERMS + lane * SR_SEQ_RUN + j;
                        at++;
                    }
            }
        }
    }
}

// ---- argmax of an fp32 row: first index of the maximum, first NaN wins -------------------------------
__device__ __forceinline__ int row_argmax(const float* w, int n, FullSmem& sm)
{
    unsigned long long best = 0ull;
    row_pass<false>(const_cast<float*>(w), n, [&](float v, int i) -> float {
        const uint32_t k = (v != v) ? 0xffffffffu : sr_okey(v);
        const unsigned long long e = ((unsigned long long)k << 32) | (unsigned long long)(0xffffffffu - (uint32_t)i);
        best = e > best ? e : best;
        return v;
    });
    best = blk_max_u64(best, sm);
    return best ? (int)(0xffffffffu - (uint32_t)(best & 0xffffffffull)) : 0;
}

// first index whose running fp32 sum reaches r = (float)u; last index as the rounding fallback
// (SampleFromDistribution, Sampler.cs:564-576)
__device__ __forceinline__ int draw_from_row(const float* p, int n, double u, FullSmem& sm, float m1 = 1.0f, float m2 = 1.0f)
{
    const float r = __double2float_rn(u);
    int found;
    const float at = seq_sum_row<true>(p, n, 0.0f, r, &found, sm, m1, m2);
    if (threadIdx.x == 0)
        SR_AMB_IF(found >= 0 ? sr_stop_near(at, __fmul_rn(__fmul_rn(p[found], m1), m2), r) : sr_near(at, r));
    return found >= 0 ? found : n - 1;
}

// Final Normalize (Sampler.cs:91-92, :553-562) and draw (:564-576) of a row whose survivors are listed in index order
// in sm.sortbuf[0, m) (~index << 32 | probability bits; an entry with probability bits of zero is no survivor) and
// whose other entries are all zero.  Adding zero changes no running sum, so the eight strided chains of
// TensorPrimitives.Sum (plus its overlapped tail) and the running sum of the draw are taken over the survivors alone,
// in index order: a chain's terms are the survivors whose index falls on it, and the tail's indices lie behind every
// body index, so one order serves all eight chains.  Behind a barrier that follows the last write of the list.
// A list of more than kSmall entries comes through sm.sortbuf a block of kSmall at a time: fill(first, count), called
// by all threads between two barriers, puts the entries [first, first + count) at sm.sortbuf[0, count).  A list that is
// in sm.sortbuf already has m <= kSmall and a fill that does nothing.
struct NoFill {
    __device__ __forceinline__ void operator()(int, int) const {}
};
__device__ __forceinline__ int list_layout(int i) { return (i & ~1023) | ((i & 15) << 6) | ((i >> 4) & 63); }
// ... of at most 64 members, at sm.sortbuf as they come: one thread per chain adds its own, and one thread draws.  What the final Normalize
// multiplies by, 1 where it leaves the values alone.
__device__ __forceinline__ float finish_short_list(const SrFullArgs& a, int n, int m, int row, FullSmem& sm)
{
    const int nv8 = (n / 8) * 8;
    const int tid = threadIdx.x;
    if (tid < SR_SEQ_CHAINS) {
        float s = 0.0f;
        for (int i = 0; i < m; i++) {
            const unsigned long long v = sm.sortbuf[i];
            const int e = (int)(0xffffffffu - (uint32_t)(v >> 32));
            const int chain = e < nv8 ? (e & 7) : e - (n - 8);
            if (chain == tid) s = __fadd_rn(s, sr_u2f((uint32_t)v));
        }
        sm.lane_sum[tid] = s;
    }
    __syncthreads();
    const float l0 = sm.lane_sum[0], l1 = sm.lane_sum[1], l2 = sm.lane_sum[2], l3 = sm.lane_sum[3],
                l4 = sm.lane_sum[4], l5 = sm.lane_sum[5], l6 = sm.lane_sum[6], l7 = sm.lane_sum[7];
    const float sum = __fadd_rn(__fadd_rn(__fadd_rn(l0, l1), __fadd_rn(l2, l3)), __fadd_rn(__fadd_rn(l4, l5), __fadd_rn(l6, l7)));
    const bool scale = sum > 0.0f && sum != 1.0f;
    const float inv = scale ? __fdiv_rn(1.0f, sum) : 1.0f;
    if (a.mode != 1 && tid == 0) {
        const float r = __double2float_rn(sm.u);
        int token = n - 1;
        if (!(r > 0.0f)) {
            token = 0;  // the running sum starts at p[0] >= 0: index 0 reaches a target of zero whatever it holds
        } else {
            float acc = 0.0f;
            bool hit = false;
            for (int i = 0; i < m && !hit; i++) {
                const unsigned long long v = sm.sortbuf[i];
                const float x = sr_u2f((uint32_t)v), xs = scale ? __fmul_rn(x, inv) : x;
                acc = __fadd_rn(acc, xs);
                if (acc >= r) {
                    token = (int)(0xffffffffu - (uint32_t)(v >> 32));
                    hit = true;
                    SR_AMB_IF(sr_stop_near(acc, xs, r));
                }
            }
            if (!hit) SR_AMB_IF(sr_near(acc, r));
        }
        if (a.out_tokens) a.out_tokens[row] = token;
    }
    return inv;
}
template <typename Fill = NoFill>
__device__ __forceinline__ void finish_from_ordered_list(const SrFullArgs& a, float* p, int n, int m, int row, FullSmem& sm,
                                                         Fill fill = Fill(), int cap = kSmall, bool laid_out = false)
{
    // (cap: what a list that is in shared memory already may hold -- kSmall, or 2 kSmall where the launch gave the
    // workgroup the room: the list then runs on from sm.sortbuf through the two arrays behind it)
    constexpr bool kResident = std::is_same<Fill, NoFill>::value;
    constexpr int kPerT = 2 * kSmall / kT;
    unsigned long long* const buf = &sm.sortbuf[0];
    const int cpt = (kResident ? cap : kSmall) / kT;  // entries per thread of the list's new layout
    const int nv8 = (n / 8) * 8;
    const int lane = sr_lane(), wave = sr_wave_id();
    // One wave per chain: it passes over the whole list in index order, sixteen entries per lane at a time, with the
    // entries of the other chains as zeros.
    // A lane's sixteen consecutive entries would all lie in the same LDS banks as every other lane's: inside each
    // thousand entries the list is laid out anew, entry 16 l + j at place 64 j + l.
    // (laid_out: the caller has put its list there that way)
    auto place_of = [](int i) -> int { return list_layout(i); };
    auto lay_out = [&]() __attribute__((always_inline)) {
        static_assert(kSmall == 4 * kT, "four entries per thread, or eight");
        unsigned long long t[kPerT];
#pragma unroll
        for (int r = 0; r < kPerT; r++) t[r] = r < cpt ? buf[cpt * (int)threadIdx.x + r] : 0ull;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kPerT; r++)
            if (r < cpt) buf[place_of(cpt * (int)threadIdx.x + r)] = t[r];
        __syncthreads();
    };
    auto load_terms = [&](int i0, int cnt, int chain, float mul, bool scale, float (&x)[16]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const int i = i0 + j;
            const unsigned long long v = i < cnt ? buf[place_of(i)] : 0ull;
            const int e = (int)(0xffffffffu - (uint32_t)(v >> 32));
            const bool mine = chain < 0 || (e < nv8 ? (e & 7) : e - (n - 8)) == chain;
            const float t = sr_u2f((uint32_t)v);
            x[j] = (i < cnt && mine) ? (scale ? __fmul_rn(t, mul) : t) : 0.0f;
        }
    };
    if (kResident && m <= SR_WAVE) {
        const float inv = finish_short_list(a, n, m, row, sm);
        if (a.mode != 0 && inv != 1.0f) row_pass<true>(p, n, [&](float x, int) -> float { return __fmul_rn(x, inv); });
        return;
    }
    float sc = 0.0f;
    if (kResident && !laid_out) lay_out();
    const int step = kResident ? cap : kSmall;  // (a resident list is one block)
    for (int first = 0; first < m; first += step) {
        const int cnt = min(step, m - first);
        if (!kResident) {
            __syncthreads();
            fill(first, cnt);
            __syncthreads();
            lay_out();
        }
        if (wave < SR_SEQ_CHAINS) {
            for (int b0 = 0; b0 < cnt; b0 += 16 * SR_WAVE) {
                float x[16];
                load_terms(b0 + 16 * lane, cnt, wave, 1.0f, false, x);
                int dummy;
                sc = sr_seq_wave<16, false>(x, sc, 0.0f, &dummy);
            }
        }
    }
    if (wave < SR_SEQ_CHAINS && lane == 0) sm.lane_sum[wave] = sc;
    __syncthreads();
    FPROF(a, blockIdx.x, 18);
    const float l0 = sm.lane_sum[0], l1 = sm.lane_sum[1], l2 = sm.lane_sum[2], l3 = sm.lane_sum[3],
                l4 = sm.lane_sum[4], l5 = sm.lane_sum[5], l6 = sm.lane_sum[6], l7 = sm.lane_sum[7];
    const float sum = __fadd_rn(__fadd_rn(__fadd_rn(l0, l1), __fadd_rn(l2, l3)), __fadd_rn(__fadd_rn(l4, l5), __fadd_rn(l6, l7)));
    const bool scale = sum > 0.0f && sum != 1.0f;
    const float inv = scale ? __fdiv_rn(1.0f, sum) : 1.0f;
    if (a.mode != 0 && scale) row_pass<true>(p, n, [&](float x, int) -> float { return __fmul_rn(x, inv); });
    if (a.mode == 1) return;
    const float r = __double2float_rn(sm.u);
    int token = n - 1;
    bool done = false;  // (what wave 0 knows)
    if (!(r > 0.0f)) {
        token = 0;  // the running sum starts at p[0] >= 0: index 0 reaches a target of zero whatever it holds
        done = true;
    }
    float acc = 0.0f;
    for (int first = 0; first < m; first += step) {
        const int cnt = min(step, m - first);
        if (!kResident) {
            if (wave == 0 && lane == 0) sm.bc[10] = done ? 1u : 0u;
            __syncthreads();
            if (sm.bc[10] != 0u) break;
            fill(first, cnt);
            __syncthreads();
            lay_out();
        }
        if (wave == 0 && !done) {
            for (int b0 = 0; b0 < cnt; b0 += 16 * SR_WAVE) {
                float x[16];
                load_terms(b0 + 16 * lane, cnt, -1, inv, scale, x);
                int f;
                acc = sr_seq_wave<16, true>(x, acc, r, &f);
                if (f >= 0) {
                    const unsigned long long v = buf[place_of(b0 + f)];
                    token = (int)(0xffffffffu - (uint32_t)(v >> 32));
                    done = true;
                    const float t = sr_u2f((uint32_t)v);
                    SR_AMB_IF(lane == 0 && sr_stop_near(acc, scale ? __fmul_rn(t, inv) : t, r));
                    break;
                }
            }
        }
    }
    if (wave == 0 && lane == 0) {
        SR_AMB_IF(!done && sr_near(acc, r));  // (the draw ran off the end of the list: the last index, by the rounding fallback)
        if (a.out_tokens) a.out_tokens[row] = token;
    }
}
// ... of a list in any order, its entries as probability bits << 32 | ~index
__device__ __forceinline__ void finish_from_list(const SrFullArgs& a, float* p, int n, int m, int row, FullSmem& sm)
{
    const int tid = threadIdx.x;
    int P = 2;
    while (P < m) P <<= 1;
    __syncthreads();
    for (int i = tid; i < P; i += kT) {
        const unsigned long long v = sm.sortbuf[i];
        sm.sortbuf[i] = (i < m) ? ((v & 0xffffffffull) << 32) | (v >> 32) : 0ull;  // ~index on top: descending = index ascending
    }
    __syncthreads();
    sort_small_desc(sm, P);
    finish_from_ordered_list(a, p, n, m, row, sm);
}

// Every wave passes over its stretch [w0, w1) of a row (w0 a multiple of 4) and hands the entries for which pred(y, i)
// holds to a sink, in index order -- y being the entry times inv (the entry itself without do_scale).  Returns the
// wave's count.  The loads of the next thousand entries are on their way while a thousand are looked at.
//   sink.reserve(before, count)   room for `count` more finds of this wave, `before` found so far: the first one's place
//   sink.put(place, rank, y bits, index)   rank = the find's number within the wave
// The pass is bound by its instructions, not by memory: about 8 us for a row of 151,936 entries with few finds, 30 us
// when every 256 entries hold some.
struct StretchToSegment {  // at the stretch's own positions of the row's sort segment
    uint32_t* gk;
    int32_t* gi;
    int w0;
    __device__ __forceinline__ int reserve(int before, int) const { return w0 + before; }
    __device__ __forceinline__ void put(int place, int, uint32_t ybits, int i) const { gk[place] = ybits; gi[place] = i; }
};
struct StretchToPool {  // appended to a pool in LDS that all waves share: values to vals, tags to tags
    uint32_t* counter;
    uint32_t* vals;
    uint32_t* tags;
    int cap;  // entries the pool holds
    __device__ __forceinline__ int reserve(int, int count) const
    {
        int b = 0;
        if (sr_lane() == 0) b = (int)atomicAdd(counter, (uint32_t)count);
        return __builtin_amdgcn_readfirstlane(b);
    }
    __device__ __forceinline__ void put(int place, int rank, uint32_t ybits, int i) const
    {
        if (place < cap) { vals[place] = ybits; tags[place] = ((uint32_t)rank << kTagIndexBits) | (uint32_t)i; }
    }
};
struct StretchCount {  // nothing is kept: the wave's count is what list_stretch returns
    __device__ __forceinline__ int reserve(int, int) const { return 0; }
    __device__ __forceinline__ void put(int, int, uint32_t, int) const {}
};
struct StretchFind {  // the index of the wave's find number `target` (none for a negative target)
    int target;
    uint32_t* out;
    __device__ __forceinline__ int reserve(int, int) const { return 0; }
    __device__ __forceinline__ void put(int, int rank, uint32_t, int i) const
    {
        if (rank == target) *out = (uint32_t)i;
    }
};
template <typename Sink, typename Pred>
__device__ __forceinline__ int list_stretch(const float* p, int w0, int w1, bool do_scale, float inv, Sink sink, Pred pred)
{
    const int lane = sr_lane();
    const bool aligned = ((uintptr_t)p & 15u) == 0u;
    int cw = 0;
    auto load = [&](int i0, float (&v)[4][4]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = i0 + u * 256 + 4 * lane;
            if (aligned && i + 4 <= w1) {
                const float4 t = *(const float4*)(p + i);
                v[u][0] = t.x; v[u][1] = t.y; v[u][2] = t.z; v[u][3] = t.w;
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++) v[u][k] = (i + k < w1) ? p[i + k] : 0.0f;
            }
        }
    };
    auto look = [&](int i0, const float (&v)[4][4]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = i0 + u * 256 + 4 * lane;
            float y[4];
            bool pr[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                y[k] = do_scale ? __fmul_rn(v[u][k], inv) : v[u][k];
                pr[k] = i + k < w1 && pred(y[k], i + k);
            }
            if (__ballot(pr[0] || pr[1] || pr[2] || pr[3]) == 0ull) continue;
            int before = 0, total = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const unsigned long long b = __ballot(pr[k]);
                before += (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
                total += __popcll(b);
            }
            int place = sink.reserve(cw, total) + before, rank = cw + before;
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (pr[k]) { sink.put(place, rank, sr_f2u(y[k]), i + k); place++; rank++; }
            cw += total;
        }
    };
    if (w0 >= w1) return 0;
    float va[4][4], vb[4][4];
    load(w0, va);
    for (int i0 = w0; i0 < w1; i0 += 2048) {
        // (the scheduling barriers keep the loads where they are written: left alone, the compiler moves them down
        // to where their values are used, and every thousand entries wait for memory once more)
        if (i0 + 1024 < w1) load(i0 + 1024, vb);
        __builtin_amdgcn_sched_barrier(0);
        look(i0, va);
        if (i0 + 1024 >= w1) break;
        if (i0 + 2048 < w1) load(i0 + 2048, va);
        __builtin_amdgcn_sched_barrier(0);
        look(i0 + 1024, vb);
    }
    return cw;
}

// ---- the nucleus of a row that only top-p cuts, without a pass that writes the row ---------------------------------
// The row holds e = expf(x - max); its probabilities are y = fl(e * inv) (y = e when the sum is 1), which rise with e.
// The caller has counted the e by their upper 16 bits in hcnt (LDS, kHistPos
// positions: position d holds the keys 0x3f80 - d, position 0 is e = 1, the last position everything below).  From the
// counts: the longest run of positions from the top that holds at most kSmall entries (a slab), the first one shortened
// to where a lower bound of its probability mass (count x the position's smallest value) passes top_p with a margin.
// One read of the row lists a slab's entries (every wave takes a stretch of the row; the finds go to a pool in LDS
// with their number within the wave, from which their places in index order follow); their values alone are sorted,
// the exact running sum goes on through them, and slab follows slab until it reaches top_p.  The members -- the values
// above the value at the cut and the first few equal to it by index -- are marked in the last slab's index-ordered
// list, from which a nucleus of one slab is finished; one of several slabs has its members listed by one more read
// of the row into the row's sort segment and is finished from there a block at a time.  Returns kNucleusDone, or
// which general way the row has to go (nothing is written then but LDS and the row's sort segment).
enum NucleusWay : int { kNucleusDone = 0, kNucleusGeneral = 1, kNucleusGeneralNoSlabs = 2 };
constexpr int kNucleusMaxSlabs = 40;
constexpr int kNucleusRowFinish = 4;  // a nucleus that took more slabs than this is finished by passes over the row
// `extra`: 16 kSmall bytes of shared memory beyond sm, or null.  With them a slab holds 2 kSmall entries -- most nuclei of
// a few thousand entries then close in one slab, which is listed by one read of the row and finished from the list,
// where two slabs cost three reads --: the pool of values and tags lies there, and the lists that are sm.sortbuf
// otherwise run on through the two arrays behind it.
__device__ __forceinline__ int nucleus_from_histogram(const SrFullArgs& a, float top_p, const float* p, int n, int slot,
                                                      int row, bool do_scale, float inv, FullSmem& sm, uint32_t* extra)
{
    constexpr int kPer = kHistPos / kT;
    static_assert(kHistPos * 4 <= kSmall * 8 && kHistPos % kT == 0, "the histogram fits the sort buffer");
    static_assert(offsetof(FullSmem, sprob) == offsetof(FullSmem, sortbuf) + sizeof(FullSmem::sortbuf) &&
                  offsetof(FullSmem, tags) == offsetof(FullSmem, sprob) + sizeof(FullSmem::sprob) &&
                  sizeof(FullSmem::sortbuf) + sizeof(FullSmem::sprob) + sizeof(FullSmem::tags) >= 2 * kSmall * sizeof(unsigned long long),
                  "a list of 2 kSmall entries fits the three arrays, which lie one behind the other");
    constexpr int kPerT = 2 * kSmall / kT;  // most entries of a slab per thread
    const int tid = threadIdx.x, lane = sr_lane(), wave = sr_wave_id();
    const int S = extra ? 2 * kSmall : kSmall;  // entries a slab may hold
    const int cpt = S / kT;
    const uint32_t* hcnt = (const uint32_t*)sm.sortbuf;
    uint32_t* sval = extra ? extra : (uint32_t*)sm.sprob;
    uint32_t* const tags = extra ? extra + 2 * kSmall : sm.tags;
    unsigned long long* const list = &sm.sortbuf[0];  // [S]
    [[maybe_unused]] unsigned long long t_step = 0ull;
    FPROF_ADD(a, slot, 16, t_step);
    if (sm.bc[5] != 0u) return kNucleusGeneral;
    // counts and mass bounds (in units of 2^-28) of this thread's positions
    uint32_t mine[kPer], mq[kPer];
    int own = 0;
    uint32_t ownq = 0u;
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int d = tid * kPer + j;
        mine[j] = hcnt[d];
        const float e_low = d < kHistPos - 1 ? sr_u2f((kHistTopKey - (uint32_t)d) << 16) : 0.0f;
        const float y_low = do_scale ? __fmul_rn(e_low, inv) : e_low;
        mq[j] = (uint32_t)fminf((float)mine[j] * y_low * 268435456.0f, 268435456.0f);
        own += (int)mine[j];
        ownq += mq[j];
    }
    int tot, totq;
    const int c0 = blk_excl_scan(own, &tot, sm);
    const uint32_t q0 = (uint32_t)blk_excl_scan((int)ownq, &totq, sm);
    int crowd = 0;  // entries at positions that hold more than a slab (runs of one value, if the row can be walked at all)
#pragma unroll
    for (int j = 0; j < kPer; j++) crowd += mine[j] > (uint32_t)S ? (int)mine[j] : 0;
    const int crowded_total = blk_sum_i(crowd, sm);
    if (tid == 0) { sm.bc[7] = (uint32_t)kHistPos; sm.bc[11] = (uint32_t)tot; }
    __syncthreads();
    {
        const uint32_t target_q = (uint32_t)(top_p * 1.001f * 268435456.0f) + 64u;
        uint32_t q = q0;
        int c = c0, d_first = kHistPos, c_first = 0;
#pragma unroll
        for (int j = 0; j < kPer; j++) {
            q += mq[j];
            c += (int)mine[j];
            if (q >= target_q && d_first == kHistPos) { d_first = tid * kPer + j; c_first = c; }
        }
        if (d_first < kHistPos) {
            atomicMin(&sm.bc[7], (uint32_t)d_first);
            atomicMin(&sm.bc[11], (uint32_t)c_first);  // (counts rise with the positions: the least belongs to the first)
        }
    }
    const int chunk = ((n + kW * 256 - 1) / (kW * 256)) * 256;
    const int w0 = min(n, wave * chunk), w1 = min(n, w0 + chunk);
    uint32_t* gk = a.sort_keys_in + (size_t)slot * a.sort_stride;
    int32_t* gi = a.sort_vals_in + (size_t)slot * a.sort_stride;
    FPROF_ADD(a, slot, 11, t_step);

    // The nucleus is walked from the top, a slab of at most kSmall entries at a time: the positions [d_prev, d_end).
    constexpr int kMaxSlabs = kNucleusMaxSlabs;
    float run = 0.0f;      // exact running sum behind the slabs before
    float hi_y = 0.0f;     // what is left has y <= hi_y (from the second slab on)
    int d_prev = 0;
    int taken = 0;         // entries that the histogram holds at the positions before d_prev
    int found = -1, nc = 0, slab = 0;
    bool all_in = false;
    int runs = 0;              // positions passed as runs of one value
    bool was_capped = false;   // ... after which what is left is bounded from above too
    bool cut_in_run = false;   // the cut fell inside such a run: ycut / idx_last are set by the walk
    uint32_t ycut = 0u;
    int idx_last = -1;         // the last member among the entries equal to the cut value
    uint32_t pv[kPerT];  // the last slab's entries that this thread read from the pool: their values (index and place in
                         // index order stay in the pool's tags)
#pragma unroll
    for (int r = 0; r < kPerT; r++) pv[r] = 0u;
    for (;; slab++) {
        if (slab >= kMaxSlabs) return kNucleusGeneralNoSlabs;  // (the general way would walk the same slabs)
        if (tid == 0) sm.bc[6] = (uint32_t)kHistPos;
        __syncthreads();
        {
            int c = c0, d_first = kHistPos;
#pragma unroll
            for (int j = 0; j < kPer; j++) {
                c += (int)mine[j];
                if (tid * kPer + j >= d_prev && c - taken > S && d_first == kHistPos) d_first = tid * kPer + j;
            }
            if (d_first < kHistPos) atomicMin(&sm.bc[6], (uint32_t)d_first);
        }
        __syncthreads();
        // about how many entries the nucleus holds: a row that would need more slabs than are walked goes the general
        // way at once (its survivors are sorted where they lie)
        if (slab == 0 && runs == 0 && (int)sm.bc[11] - min((int)sm.bc[11], crowded_total) > (kMaxSlabs - 2) * S)
            return kNucleusGeneralNoSlabs;
        const int d_cnt = (int)sm.bc[6], d_mass = (int)sm.bc[7];
        const int d_end = d_mass + 1 > d_prev ? min(d_cnt, d_mass + 1) : d_cnt;
        if (d_end <= d_prev) {
            // One position alone holds more than a slab.  Where all its entries share one probability -- the equal
            // logits of a coarse grid, of bf16 -- no order among them is needed: the running sum goes through them
            // as through so many equal terms, and if the cut falls among them, the members are the first ones by
            // index.  Anything else is left to the general way's sort.
            if (++runs > 256) return kNucleusGeneralNoSlabs;
            const uint32_t key_d = kHistTopKey - (uint32_t)d_prev;
            const bool last_pos = d_prev == kHistPos - 1;
            // the position's distinct probabilities (a few at most, or the row is left to the sort) and their counts
            constexpr int kDistinct = 16;
            uint32_t* dval = sm.hist + 32;
            uint32_t* dcnt = sm.hist + 32 + kDistinct;
            __syncthreads();
            if (tid < 2 * kDistinct) sm.hist[32 + tid] = 0u;
            if (tid == 0) sm.bc[12] = 0u;
            __syncthreads();
            row_pass<false>(const_cast<float*>(p), n, [&](float e, int) -> float {
                const uint32_t k16 = sr_f2u(e) >> 16;
                if (e > 0.0f && (last_pos ? k16 <= key_d : k16 == key_d)) {
                    const uint32_t yb = sr_f2u(do_scale ? __fmul_rn(e, inv) : e);
                    bool placed = false;
                    for (int sl = 0; sl < kDistinct && !placed; sl++) {
                        const uint32_t old = atomicCAS(&dval[sl], 0u, yb);
                        if (old == 0u || old == yb) {
                            atomicAdd(&dcnt[sl], 1u);
                            placed = true;
                        }
                    }
                    if (!placed || yb < 0x00800000u) sm.bc[12] = 1u;  // (too many values, or one below the normal range)
                }
                return e;
            });
            __syncthreads();
            if (sm.bc[12] != 0u) return kNucleusGeneralNoSlabs;
            // from the largest value down (every thread finds the same order)
            uint32_t below = 0xffffffffu;  // values at or above this one are done
            bool cut_here = false;
            for (int round = 0; round < kDistinct; round++) {
                uint32_t mn = 0u;
                int c_run = 0;
                for (int sl = 0; sl < kDistinct; sl++) {
                    const uint32_t v = dval[sl];
                    if (v != 0u && v < below && v > mn) { mn = v; c_run = (int)dcnt[sl]; }
                }
                if (mn == 0u) break;  // all of the position's values are done
                below = mn;
                const float yv = sr_u2f(mn);
                int f;
                run = seq_sum<true>([&](int) -> float { return yv; }, c_run, run, top_p, &f, sm);
                if (f < 0) continue;
                // (a cut inside a run of equal probabilities keeps the first ones by index: the managed sort leaves
                // their order open)
                SR_AMB_IF(f + 1 < c_run || sr_stop_near(run, yv, top_p));
                // the cut falls inside this run: its first f + 1 entries by index are members
                const int cw = list_stretch(p, w0, w1, do_scale, inv, StretchCount{}, [&](float y, int) -> bool { return sr_f2u(y) == mn; });
                __syncthreads();
                if (lane == 0) sm.redi[wave] = cw;
                if (tid == 0) sm.bc[9] = 0xffffffffu;
                __syncthreads();
                int before_w = 0;
#pragma unroll
                for (int w = 0; w < kW; w++) before_w += w < wave ? sm.redi[w] : 0;
                const int target = (f >= before_w && f < before_w + cw) ? f - before_w : -1;
                __syncthreads();
                (void)list_stretch(p, w0, w1, do_scale, inv, StretchFind{target, &sm.bc[9]}, [&](float y, int) -> bool { return sr_f2u(y) == mn; });
                __syncthreads();
                if (sm.bc[9] == 0xffffffffu) return kNucleusGeneralNoSlabs;  // (the counts of the two reads differ: not possible)
                ycut = mn;
                idx_last = (int)sm.bc[9];
                cut_in_run = true;
                cut_here = true;
                break;
            }
            if (cut_here) { nc = 0; break; }
            const uint32_t mn = below;  // the position's smallest value: what is left of the row lies below it
            // the whole run lies inside the nucleus: on to the position behind it
            {
                int c = c0;
#pragma unroll
                for (int j = 0; j < kPer; j++) {
                    c += (int)mine[j];
                    if (tid * kPer + j == d_prev) sm.bc[8] = (uint32_t)c;
                }
            }
            __syncthreads();
            taken = (int)sm.bc[8];
            hi_y = sr_u2f(mn - 1u);  // what is left lies below the run's value
            d_prev = d_prev + 1;
            __syncthreads();
            if (d_prev >= kHistPos) { all_in = true; nc = 0; break; }
            slab--;  // (a run is not one of the slabs that the limit counts; the for's increment puts it back)
            was_capped = true;
            continue;
        }
        {
            int c = c0;
#pragma unroll
            for (int j = 0; j < kPer; j++) {
                c += (int)mine[j];
                if (tid * kPer + j == d_end - 1) sm.bc[8] = (uint32_t)c;
            }
        }
        all_in = d_end >= kHistPos;
        const float c_e = all_in ? 0.0f : sr_u2f(((kHistTopKey - (uint32_t)d_end) << 16) | 0xffffu);
        const float c_y = do_scale ? __fmul_rn(c_e, inv) : c_e;  // taken: y > c_y, which e > c_e follows from
        const bool capped = slab > 0 || was_capped;

        // the slab's entries: every wave lists those of its stretch of the row in a pool in LDS, each with its number
        // within the wave, from which its place in index order follows once all waves' counts are known
        if (tid == 0) sm.bc[4] = 0u;
        __syncthreads();
        const int cw = list_stretch(p, w0, w1, do_scale, inv, StretchToPool{&sm.bc[4], sval, tags, S},
                                    [&](float y, int) -> bool { return y > c_y && !(capped && y > hi_y); });
        if (lane == 0) sm.redi[wave] = cw;
        __syncthreads();
        taken = (int)sm.bc[8];
        nc = (int)sm.bc[4];
        if (nc > S) return kNucleusGeneral;
        FPROF_ADD(a, slot, 12, t_step);
        if (nc > 0) {
            // this thread's entries of the pool; their places in index order take the place of their numbers within
            // the wave in the tags
#pragma unroll
            for (int r = 0; r < kPerT; r++) {
                const int e = r * kT + tid;
                pv[r] = e < nc ? sval[e] : 0u;
                if (e < nc) {
                    const uint32_t tag = tags[e];
                    const int i = (int)(tag & ((1u << kTagIndexBits) - 1u)), w = i / chunk;
                    int off = (int)(tag >> kTagIndexBits);
#pragma unroll
                    for (int k = 0; k < kW - 1; k++) off += k < w ? sm.redi[k] : 0;
                    tags[e] = ((uint32_t)off << kTagIndexBits) | (uint32_t)i;
                }
            }
            // The values are sorted.  A long list is first cut into 4,096 groups of equal width in the values' bit
            // patterns between the slab's bounds -- counted, the counts summed, the values put group by group -- and
            // then every value finds its rank among the values of its group (equal values are interchangeable in the
            // sum that follows): far fewer steps than the sorting network, unless a group holds more than a few dozen.
            const uint32_t bhi = sr_f2u(capped ? hi_y : (do_scale ? __fmul_rn(1.0f, inv) : 1.0f)), blo = sr_f2u(c_y);
            const uint32_t span = bhi >= blo ? bhi - blo : 0xffffffffu;
            const int gshift = span < (uint32_t)kSmall ? 0 : 20 - __clz((int)span);  // (span >> gshift) < kSmall
            auto group_of = [&](uint32_t v) -> uint32_t { return min((bhi - v) >> gshift, (uint32_t)(kSmall - 1)); };
            bool counted = false;
            if (nc > 1024 && bhi >= blo) {
                uint32_t* cur = (uint32_t*)sm.sortbuf;
                uint32_t* grp = cur + kSmall;
                __syncthreads();  // (sval has been read)
#pragma unroll
                for (int r = 0; r < 4; r++) cur[r * kT + tid] = 0u;
                if (tid == 0) sm.bc[12] = 0u;
                __syncthreads();
#pragma unroll
                for (int r = 0; r < kPerT; r++)
                    if (r * kT + tid < nc) atomicAdd(&cur[group_of(pv[r])], 1u);
                __syncthreads();
                uint32_t c4[4];
                int own = 0;
                uint32_t big = 0u;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    c4[r] = cur[4 * tid + r];
                    own += (int)c4[r];
                    big = max(big, c4[r]);
                }
                if (big > 128u) sm.bc[12] = 1u;
                int tot_c;
                int at = blk_excl_scan(own, &tot_c, sm);
                counted = sm.bc[12] == 0u;  // (the scan's barriers lie between the store and this load)
                if (counted) {
#pragma unroll
                    for (int r = 0; r < 4; r++) { cur[4 * tid + r] = (uint32_t)at; at += (int)c4[r]; }
                    __syncthreads();
#pragma unroll
                    for (int r = 0; r < kPerT; r++)
                        if (r * kT + tid < nc) grp[atomicAdd(&cur[group_of(pv[r])], 1u)] = pv[r];
                    __syncthreads();  // cur[g] is now where group g ends
#pragma unroll
                    for (int r = 0; r < kPerT; r++) {
                        const int i = r * kT + tid;
                        if (i < nc) {
                            const uint32_t v = grp[i];
                            const uint32_t g = group_of(v);
                            const int from = g > 0u ? (int)cur[g - 1u] : 0, to = (int)cur[g];
                            int rank = from;
                            for (int j = from; j < to; j++) {
                                const uint32_t o = grp[j];
                                rank += (o > v || (o == v && j < i)) ? 1 : 0;
                            }
                            sval[rank] = v;
                        }
                    }
                    __syncthreads();
                }
            }
            if (!counted) {
                if (nc > kSmall) return kNucleusGeneral;  // (the network sorts kSmall entries at most)
                int P = 2;
                while (P < nc) P <<= 1;
                __syncthreads();
                for (int e = nc + tid; e < P; e += kT) sval[e] = 0u;
                __syncthreads();
                sort_lds_desc(sval, P);
            }
            FPROF_ADD(a, slot, 13, t_step);
            run = seq_sum<true>([&](int i) -> float { return sr_u2f(sval[i]); }, nc, run, top_p, &found, sm);
            if (found >= 0)
                SR_AMB_IF(sr_stop_near(run, sr_u2f(sval[found]), top_p) || (found + 1 < nc && sval[found + 1] == sval[found]));
            FPROF_ADD(a, slot, 14, t_step);
        }
        if (a.prof && slot == 0 && tid == 0) a.prof[15] += 1ull;
        if (found >= 0 || all_in) break;
        hi_y = c_y;
        d_prev = d_end;
    }
    if (found < 0 && !cut_in_run) SR_AMB_IF(sr_near(run, top_p));  // the whole row is the nucleus: barely?

    // the last slab's entries in index order (the sort's scratch memory is free again)
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPerT; r++)
        if (r * kT + tid < nc) {
            const uint32_t tag = tags[r * kT + tid];
            list[tag >> kTagIndexBits] = ((unsigned long long)(0xffffffffu - (tag & ((1u << kTagIndexBits) - 1u))) << 32) | (unsigned long long)pv[r];
        }
    __syncthreads();
    // Members: everything above the value at the cut, and of the entries equal to it the first ones by index.
    if (found >= 0 && !cut_in_run) {
        ycut = sval[found];
        int gt = 0;
        for (int e = tid; e < nc; e += kT) gt += sval[e] > ycut ? 1 : 0;
        const int keep_eq = found + 1 - blk_sum_i(gt, sm);
        unsigned long long ent[kPerT];
        int eqc = 0;
#pragma unroll
        for (int r = 0; r < kPerT; r++) {
            const int e = cpt * tid + r;
            ent[r] = (r < cpt && e < nc) ? list[e] : 0ull;
            eqc += (r < cpt && e < nc && (uint32_t)ent[r] == ycut) ? 1 : 0;
        }
        int tot_eq;
        int rank = blk_excl_scan(eqc, &tot_eq, sm);
#pragma unroll
        for (int r = 0; r < kPerT; r++) {
            const int e = cpt * tid + r;
            if (r < cpt && e < nc) {
                const uint32_t yb = (uint32_t)ent[r];
                const bool keep = yb > ycut || (yb == ycut && rank < keep_eq);
                if (yb == ycut && rank == keep_eq - 1) sm.bc[9] = 0xffffffffu - (uint32_t)(ent[r] >> 32);
                if (yb == ycut) rank++;
                if (!keep) list[e] = ent[r] & 0xffffffff00000000ull;
            }
        }
        __syncthreads();
        idx_last = (int)sm.bc[9];
    }
    if (slab == 0 && runs == 0) {
        finish_from_ordered_list(a, const_cast<float*>(p), n, nc, row, sm, NoFill(), S);
        return kNucleusDone;
    }
    // Several slabs: the members -- known by value and, at the cut value, by index -- are listed by one more read of
    // the row, again in index order in the waves' stretches of the sort segment, and the final Normalize and the draw
    // take them from there a block at a time.
    const float ycut_f = sr_u2f(ycut);
    if (slab >= kNucleusRowFinish || runs > 0) {
        // A nucleus of many thousands of members: listing them and passing over the list, 5 us per thousand, costs more
        // than writing the row -- scaled, everything outside the nucleus zero -- and the two passes over it of the
        // final Normalize and the pass of the draw (about 70 us for 151,936 entries).
        float* w = const_cast<float*>(p);
        row_pass<true>(w, n, [&](float e, int i) -> float {
            const float y = do_scale ? __fmul_rn(e, inv) : e;
            return (y > ycut_f || (y == ycut_f && i <= idx_last)) ? y : 0.0f;
        });
        __syncthreads();
        normalize_row(w, n, sm);
        if (a.mode != 1) {
            const int token = draw_from_row(w, n, sm.u, sm);
            if (tid == 0 && a.out_tokens) a.out_tokens[row] = token;
        }
        return kNucleusDone;
    }
    const int cm = list_stretch(p, w0, w1, do_scale, inv, StretchToSegment{gk, gi, w0},
                                [&](float y, int i) -> bool { return y > ycut_f || (y == ycut_f && i <= idx_last); });
    sr_drain_stores();
    __syncthreads();  // (the last readers of sm.hist are long past; this one orders the stretches' stores before the fills)
    if (lane == 0) sm.hist[wave] = (uint32_t)cm;
    __syncthreads();
    int members = 0;
#pragma unroll
    for (int w = 0; w < kW; w++) members += (int)sm.hist[w];
    FPROF_ADD(a, slot, 17, t_step);
    finish_from_ordered_list(a, const_cast<float*>(p), n, members, row, sm, [&](int first, int cnt) {
        // (all of a thread's loads are on their way before the first of them is waited for)
        int src[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int g = first + min(r * kT + tid, cnt - 1);
            int w = 0, off = 0;
#pragma unroll
            for (int k = 0; k < kW - 1; k++) {
                const int ck = (int)sm.hist[k];
                if (w == k && g >= off + ck) { off += ck; w = k + 1; }
            }
            src[r] = min(n, w * chunk) + (g - off);
        }
        uint32_t yb[4];
        int32_t ix[4];
#pragma unroll
        for (int r = 0; r < 4; r++) { yb[r] = gk[src[r]]; ix[r] = gi[src[r]]; }
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (r * kT + tid < cnt) sm.sortbuf[r * kT + tid] = ((unsigned long long)(0xffffffffu - (uint32_t)ix[r]) << 32) | (unsigned long long)yb[r];
    });
    return kNucleusDone;
}

// ---- the survivors of a row sorted where they lie -------------------------------------------------------------------
// keys[i] (probability bits) and ids[i] (indices) of ns entries in device memory, sorted by descending key, equal keys
// by ascending index, by this workgroup alone: a bitonic network whose comparators all point the same way (a merge
// starts by comparing every entry with its mirror image in the block, then halves), so that a length that is no power of
// two needs no padding in memory -- the entries past the end count as the smallest and never move.  Tiles of kSmall
// entries are sorted and merged in LDS; only the steps that reach across tiles go through memory.  For the rare row
// whose nucleus the walk by slabs cannot close: about 2 ms for 130 thousand survivors.
__device__ __forceinline__ void sort_survivors_in_place(uint32_t* keys, int32_t* ids, int ns, FullSmem& sm)
{
    typedef unsigned long long u64;
    const int tid = threadIdx.x;
    auto ld = [&](int i) -> u64 { return ((u64)keys[i] << 32) | (u64)(0xffffffffu - (uint32_t)ids[i]); };
    auto st = [&](int i, u64 v) { keys[i] = (uint32_t)(v >> 32); ids[i] = (int32_t)(0xffffffffu - (uint32_t)v); };
    auto tile_in = [&](int t0) {
        for (int e = tid; e < kSmall; e += kT) sm.sortbuf[e] = t0 + e < ns ? ld(t0 + e) : 0ull;
        __syncthreads();
    };
    auto tile_out = [&](int t0) {
        for (int e = tid; e < kSmall; e += kT)
            if (t0 + e < ns) st(t0 + e, sm.sortbuf[e]);
        sr_drain_stores();
        __syncthreads();
    };
    __syncthreads();
    for (int t0 = 0; t0 < ns; t0 += kSmall) {
        tile_in(t0);
        sort_lds_desc(sm.sortbuf, kSmall);
        tile_out(t0);
    }
    int total = kSmall;  // the power of two that the network is laid out for
    while (total < ns) total <<= 1;
    for (int k2 = 2 * kSmall; k2 <= total; k2 <<= 1) {
        // every entry of a block's first half against its mirror image in the second
        for (int pr = tid; pr < total / 2; pr += kT) {
            const int blk = pr / (k2 / 2), off = pr - blk * (k2 / 2);
            const int i = blk * k2 + off, j = blk * k2 + k2 - 1 - off;
            if (j < ns) {
                const u64 x = ld(i), y = ld(j);
                if (x < y) { st(i, y); st(j, x); }
            }
        }
        sr_drain_stores();
        __syncthreads();
        // halves, quarters, ... of the block down to the size of a tile
        for (int j2 = k2 / 4; j2 >= kSmall; j2 >>= 1) {
            for (int pr = tid; pr < total / 2; pr += kT) {
                const int i = ((pr & ~(j2 - 1)) << 1) | (pr & (j2 - 1)), j = i | j2;
                if (j < ns) {
                    const u64 x = ld(i), y = ld(j);
                    if (x < y) { st(i, y); st(j, x); }
                }
            }
            sr_drain_stores();
            __syncthreads();
        }
        // the rest of the merge inside every tile
        for (int t0 = 0; t0 < ns; t0 += kSmall) {
            tile_in(t0);
            for (int j2 = kSmall / 2; j2 >= 1; j2 >>= 1) {
                for (int pr = tid; pr < kSmall / 2; pr += kT) {
                    const int i = ((pr & ~(j2 - 1)) << 1) | (pr & (j2 - 1)), j = i | j2;
                    const u64 x = sm.sortbuf[i], y = sm.sortbuf[j];
                    if (x < y) { sm.sortbuf[i] = y; sm.sortbuf[j] = x; }
                }
                __syncthreads();
            }
            tile_out(t0);
        }
    }
}

// ---- the cut of a row whose candidates the pass over the whole device has listed ----------------------------------------
// a.sort_keys_in / a.sort_vals_in hold, per segment, the entries e >= SrFullState::list_from in the order of their indices,
// a.seg_cnt how many.  Their values are sorted in shared memory, the min-p threshold and the exact running sum of
// top-p name the cut, and a nucleus of up to `finish_most` members is normalised and drawn from here; a larger one, and every
// row whose distribution is handed out, is left to the whole device (k_prepared_row): its members
// are known by the value at the cut and, among equal ones, by the last index.
// (One workgroup used to count the row's e into a histogram, read the row once per 8,192 entries of its nucleus to list
// them, and once more to list the members: 113 us a launch of 16 constrained rows of 151,936, of which the listing reads
// -- 600 KB each at what one compute unit takes in -- were two thirds.)
enum ListWay : int { kListDone = 0, kListDeferred = 1, kListGeneral = 2, kListClosed = 3 };
__device__ __forceinline__ int list_place(int i) { return i + (i >> 4); }  // (runs of 16 start in different banks)

__device__ __forceinline__ uint32_t* list_values(uint32_t* more, FullSmem& sm) { return more ? more : (uint32_t*)sm.sortbuf; }

// the row's members are left to the whole device: the factors and the cut, and what k_prepared_row
// needs to know of the sums in front of its blocks
__device__ __forceinline__ void row_deferred(const SrFullArgs& a, SrFullState* st, float inv, float ycut, int idx_last, const FullSmem& sm)
{
    if (threadIdx.x == 0) {
        st->mul1 = inv;
        st->mul2 = 1.0f;
        st->ycut = ycut;
        st->idx_last = idx_last;
        st->u = __double2float_rn(sm.u);  // (the uniform may lie in host memory: fetched once, by k_full_row)
        st->deferred = a.seq;
        a.row_sync[(size_t)(st - a.state) * SR_ROW_SYNC_STRIDE + 1] = (unsigned long long)a.seq << 32;  // nobody has counted in
    }
}

// kPer: most entries of a thread.  (One function for every length spent a microsecond a step on entries that are not there.)
// A list of up to kT entries has its indices in list_ids(sm), in the list's order.
__device__ __forceinline__ uint32_t* list_ids(FullSmem& sm) { return sm.tags + (kSmall - kT); }
// an entry of e in (0, 1] in whole units of 2^-40
__device__ __forceinline__ unsigned long long e_units(uint32_t ebits)
{
    return ((unsigned long long)((ebits & 0x7fffffu) | 0x800000u) << 17) >> min(127u - (ebits >> 23), 63u);
}
// Where the running sum over a long list's probabilities, the largest first, reaches `target`, without the list in order.
// Inside a binade an addition of a term moves the sum by a whole number of its last places, the same number wherever the sum stands -- but for a
// term that falls exactly half way between two --, so the terms of a stretch may come in any order.  The entries are counted by value
// into groups of equal width in the bit patterns; what stands in front of a group is then known to about half a group's width, and
// with it the binade, in which its terms' increments are added up in whole numbers.  In order are only those that need it: the first 32 (the
// sum doubles from term to term), groups in which the sum may change binade, groups that hold a term half way, and the one in which
// it gets to the target.  A walk of one thread's length over those, the stretches between them as one integer each, gives every state exactly;
// it checks that each stretch lies in the binade it was added up for, and what does not fit goes by the sorted list.
// Sorting such a list in shared memory is bound by what one compute unit's banks take: 14,000 entries 33 us and 10 for the sums in order, 7,800
// 20 and 8, 3,000 9 and 6; this 13, 11 and 9 for all of it.  us a call, rows of 151,936 fp32 at temperature 0.6 and top-p 0.95 under masks that leave 0.4, 0.2, 0.1
// of them: one row 92 -> 75, 72 -> 65, 60 -> 58; 64 rows 152 -> 134, 131 -> 123, 117 -> 115.  Two rows to a compute unit, lists of 2,000: 72.6 -> 73.5.
struct ListCut {
    int ns;        // entries that min-p leaves
    int cutoff;    // of which the first so many are members
    uint32_t ebits;  // e of the last member
    float run;     // the sum behind it, or of all entries
    bool found;    // the sum got to the target
};
constexpr int kInOrder = 1024;  // most entries that are put in order
static_assert(kInOrder % 4 == 0 && (SR_LIST_CAP_SMALL + SR_LIST_CAP_SMALL / 16) % 4 == 0, "the tables follow each other on whole vectors");
template <int kPer>
__device__ __forceinline__ bool cut_unsorted(const uint32_t (&ev)[kPer], uint32_t valid, uint32_t from, bool do_scale, float inv, float target, uint32_t* base,
                                             int G, ListCut* cut, FullSmem& sm)
{
    const int tid = threadIdx.x, lane = sr_lane(), wave = sr_wave_id();
    uint32_t* const cnt = base;          // entries of a group, then of all groups in front
    uint32_t* const info = base + G;     // a group's binade, and why its entries are in order
    uint32_t* const inc = base + 2 * G;  // a group's increments, then those of all groups in front
    uint32_t* const list = base + 3 * G; // the entries that are put in order: as they come, sorted, the stretch in front of each, the state behind each
    uint32_t* const sorted = list + kInOrder;
    uint32_t* const gap = sorted + kInOrder;
    uint32_t* const state = gap + kInOrder;
    constexpr uint32_t kOrdered = 0x100u, kHalfWay = 0x200u;
    constexpr int kMost = 4;  // groups of a thread
    auto prob = [&](uint32_t ebits) -> float { return do_scale ? __fmul_rn(sr_u2f(ebits), inv) : sr_u2f(ebits); };
    const uint32_t span = 0x3f800000u - min(from, 0x3f800000u);
    int gshift = 0;
    while ((span >> gshift) >= (uint32_t)G) gshift++;
    auto group_of = [&](uint32_t v) -> uint32_t { return min((0x3f800000u - v) >> gshift, (uint32_t)(G - 1)); };
    const int per = G / kT, g0 = tid * per;
    for (int i = tid; i < G; i += kT) { cnt[i] = 0u; inc[i] = 0u; }
    // 11: a group found by all   12: it does not fit   13: entries in order   14: some group holds a term half way
    if (tid >= 11 && tid <= 14) sm.bc[tid] = tid == 11 ? 0xffffffffu : 0u;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPer; r++)
        if ((valid >> r) & 1u) atomicAdd(&cnt[group_of(ev[r])], 1u);
    __syncthreads();
    {
        int c[kMost], cs = 0;
        float m[kMost], ms = 0.0f;
#pragma unroll
        for (int q = 0; q < kMost; q++) {
            c[q] = q < per ? (int)cnt[g0 + q] : 0;
            const uint32_t middle = 0x3f800000u - ((uint32_t)(g0 + q) << gshift) - ((1u << gshift) >> 1);
            m[q] = c[q] > 0 ? (float)c[q] * prob(middle) : 0.0f;
            cs += c[q];
            ms += m[q];
        }
        const int ci = sr_wave_incl_scan_i32(cs);
        const float mi = sr_wave_incl_sum_f32(ms);
        if (lane == SR_WAVE - 1) { sm.redi[wave] = ci; sm.redf[wave] = mi; }
        __syncthreads();
        int cb = ci - cs, all = 0;
        float mb = mi - ms;
#pragma unroll
        for (int w = 0; w < kW; w++) {
            if (w < wave) { cb += sm.redi[w]; mb += sm.redf[w]; }
            all += sm.redi[w];
        }
        cut->ns = all;
        // (half of a group's width, and what n additions may be off)
        const float off = sr_u2f((uint32_t)(127 - 23 + gshift) << 23) * 0.55f + 3e-4f;
#pragma unroll
        for (int q = 0; q < kMost; q++)
            if (q < per) {
                const uint32_t e0 = sr_f2u(mb * (1.0f - off)) >> 23, e1 = sr_f2u((mb + m[q]) * (1.0f + off)) >> 23;
                info[g0 + q] = (sr_f2u(mb) >> 23) | (cb < 32 || e0 != e1 ? kOrdered : 0u);
                cnt[g0 + q] = (uint32_t)cb;
                cb += c[q];
                mb += m[q];
            }
        if (all == 0) return false;
    }
    __syncthreads();
    auto in_order = [&](uint32_t v) {
        const uint32_t pos = atomicAdd(&sm.bc[13], 1u);
        if (pos < (uint32_t)kInOrder) list[pos] = v;
    };
#pragma unroll
    for (int r = 0; r < kPer; r++)
        if ((valid >> r) & 1u) {
            const uint32_t g = group_of(ev[r]), in = info[g];
            if (in & kOrdered) {
                in_order(ev[r]);
            } else {
                const uint32_t b = (in & 0xffu) << 23;
                const float y = prob(ev[r]);
                const uint32_t even = sr_f2u(__fadd_rn(sr_u2f(b), y)) - b, odd = sr_f2u(__fadd_rn(sr_u2f(b + 1u), y)) - (b + 1u);
                atomicAdd(&inc[g], even);
                if (even != odd) {
                    atomicOr(&info[g], kHalfWay);
                    sm.bc[14] = 1u;
                }
            }
        }
    __syncthreads();
    if (sm.bc[14] != 0u) {
#pragma unroll
        for (int r = 0; r < kPer; r++)
            if (((valid >> r) & 1u) && (info[group_of(ev[r])] & (kOrdered | kHalfWay)) == kHalfWay) in_order(ev[r]);
        __syncthreads();
    }
    const int n = (int)sm.bc[13];
    if (SR_RARE(n > kInOrder - 8)) return false;
    auto put_in_order = [&](int len) {  // list -> sorted, the largest first: every entry against every other, four threads to an entry where they are few
        const int sh = len <= kT / 4 ? 2 : len <= kT / 2 ? 1 : 0, e = tid >> sh;
        const uint32_t v = e < len ? list[e] : 0u;
        int rank = 0;
        for (int j = tid & ((1 << sh) - 1); j < len; j += 1 << sh) {
            const uint32_t o = list[j];
            rank += (o > v) | ((o == v) & (j < e)) ? 1 : 0;
        }
        if (sh > 0) rank += (int)sr_dpp_u32<kDppXor1>((uint32_t)rank);
        if (sh > 1) rank += (int)sr_dpp_u32<kDppXor2>((uint32_t)rank);
        if (e < len && (tid & ((1 << sh) - 1)) == 0) sorted[rank] = v;
    };
    uint32_t all_inc = 0u;
    {
        uint32_t d[kMost], ds = 0u;
#pragma unroll
        for (int q = 0; q < kMost; q++) {
            d[q] = q < per && (info[g0 + q] & (kOrdered | kHalfWay)) == 0u ? inc[g0 + q] : 0u;
            ds += d[q];
        }
        const uint32_t di = (uint32_t)sr_wave_incl_scan_i32((int)ds);
        if (lane == SR_WAVE - 1) sm.redu[wave] = di;
        put_in_order(n);
        __syncthreads();
        uint32_t db = di - ds;
#pragma unroll
        for (int w = 0; w < kW; w++) {
            if (w < wave) db += sm.redu[w];
            all_inc += sm.redu[w];
        }
#pragma unroll
        for (int q = 0; q < kMost; q++)
            if (q < per) { inc[g0 + q] = db; db += d[q]; }
    }
    __syncthreads();
    // The stretch in front of every entry in order, and behind the last one, in increments; beside it the entry's probability.  (Zeros up to a
    // multiple of eight, for the walk.)
    float* const ys = (float*)list;
    auto stretch = [&](int i) -> uint32_t {  // i = 1 ... n
        const uint32_t g = i < n ? group_of(sorted[i]) : (uint32_t)G;
        return (g < (uint32_t)G ? inc[g] : all_inc) - inc[group_of(sorted[i - 1])];
    };
    for (int i = tid; i < ((n + 7) & ~7); i += kT) {
        gap[i] = i > 0 && i < n ? stretch(i) : 0u;
        ys[i] = i < n ? prob(sorted[i]) : 0.0f;
    }
    __syncthreads();
    if (wave == 0) {
        // (one wave, every lane the same; what bounds it is its instructions, two an entry beside the loads and stores)
        uint32_t b = 0u;
        for (int i0 = 0; i0 < n; i0 += 8) {
            const float4 y0 = *(const float4*)(ys + i0), y1 = *(const float4*)(ys + i0 + 4);
            const uint4 d0 = *(const uint4*)(gap + i0), d1 = *(const uint4*)(gap + i0 + 4);
            uint4 t0, t1;
            t0.x = b = sr_f2u(__fadd_rn(sr_u2f(b + d0.x), y0.x));
            t0.y = b = sr_f2u(__fadd_rn(sr_u2f(b + d0.y), y0.y));
            t0.z = b = sr_f2u(__fadd_rn(sr_u2f(b + d0.z), y0.z));
            t0.w = b = sr_f2u(__fadd_rn(sr_u2f(b + d0.w), y0.w));
            t1.x = b = sr_f2u(__fadd_rn(sr_u2f(b + d1.x), y1.x));
            t1.y = b = sr_f2u(__fadd_rn(sr_u2f(b + d1.y), y1.y));
            t1.z = b = sr_f2u(__fadd_rn(sr_u2f(b + d1.z), y1.z));
            t1.w = b = sr_f2u(__fadd_rn(sr_u2f(b + d1.w), y1.w));
            if (lane == 0) {
                *(uint4*)(state + i0) = t0;
                *(uint4*)(state + i0 + 4) = t1;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        int at = -1, kind = 0;
        bool misfit = false;
        uint32_t last = 0u;  // (of lane n mod 64) the sum behind everything
        for (int i0 = 0; i0 <= n && at < 0; i0 += SR_WAVE) {
            const int i = i0 + lane;
            uint32_t before = 0u, d = 0u;
            if (i > 0 && i <= n) {
                before = state[i - 1];
                d = i < n ? gap[i] : stretch(n);
                if (d != 0u) {
                    // the stretch's groups were added up for one binade, and the sum is in it from end to end
                    const uint32_t eb = info[group_of(sorted[i - 1]) + 1u] & 0xffu, eb1 = info[(i < n ? group_of(sorted[i]) : (uint32_t)G) - 1u] & 0xffu;
                    misfit = misfit || d >= (1u << 24) || eb1 != eb || (before >> 23) != eb || ((before + d) >> 23) != eb;
                }
            }
            const bool in_gap = d != 0u && sr_u2f(before + d) >= target, on_it = i < n && sr_u2f(state[min(i, n - 1)]) >= target;
            if (i == n) last = before + d;
            const unsigned long long hit = __ballot(in_gap || on_it);
            if (hit != 0ull) {
                const int l = (int)__ffsll((long long)hit) - 1;
                at = i0 + l;
                kind = ((__ballot(in_gap) >> l) & 1ull) != 0ull ? 2 : 1;
            }
        }
        if (__ballot(misfit) != 0ull && lane == 0) sm.bc[12] = 1u;
        if (kind == 0 && lane == (n & (SR_WAVE - 1))) sm.segbc[2] = last;
        if (kind == 1) {
            const uint32_t g = group_of(sorted[at]);
            int before = 0;  // entries of the same group in front
            for (int j0 = 0; j0 < at; j0 += SR_WAVE) before += __popcll(__ballot(j0 + lane < at && group_of(sorted[min(j0 + lane, n - 1)]) == g));
            if (lane == 0) sm.segbc[2] = cnt[g] + (uint32_t)before + 1u;
        }
        if (lane == 0) {
            sm.segbc[0] = (uint32_t)kind;
            sm.segbc[1] = (uint32_t)at;
        }
    }
    __syncthreads();
    if (SR_RARE(sm.bc[12] != 0u)) return false;
    const int kind = (int)sm.segbc[0], at = (int)sm.segbc[1];
    cut->found = kind != 0;
    if (kind == 0) {
        cut->run = sr_u2f(sm.segbc[2]);
        cut->cutoff = cut->ns;
        cut->ebits = 0u;
        return true;
    }
    if (kind == 1) {
        cut->run = sr_u2f(state[at]);
        cut->cutoff = (int)sm.segbc[2];
        cut->ebits = sorted[at];
        return true;
    }
    // inside a stretch: the group in which the sum gets there, and its entries in order
    const uint32_t gp = group_of(sorted[at - 1]), g_end = at < n ? group_of(sorted[at]) : (uint32_t)G, front = state[at - 1];
    uint32_t first = 0xffffffffu;
#pragma unroll
    for (int q = kMost - 1; q >= 0; q--) {
        const uint32_t g = (uint32_t)(g0 + q);
        if (q < per && g > gp && g < g_end) {
            const uint32_t to = front + ((g + 1u < (uint32_t)G ? inc[g + 1u] : all_inc) - inc[gp]);
            if (sr_u2f(to) >= target) first = g;
        }
    }
    first = sr_wave_min_u32(first);  // (an atomic of every group behind the cut: 8 us)
    if (lane == 0 && first != 0xffffffffu) atomicMin(&sm.bc[11], first);
    if (tid == 0) sm.bc[13] = 0u;
    __syncthreads();
    const uint32_t gc = sm.bc[11];
    if (SR_RARE(gc >= (uint32_t)G)) return false;
#pragma unroll
    for (int r = 0; r < kPer; r++)
        if (((valid >> r) & 1u) && group_of(ev[r]) == gc) in_order(ev[r]);
    __syncthreads();
    const int m = (int)sm.bc[13];
    const uint32_t s0 = front + (inc[gc] - inc[gp]);
    if (SR_RARE(m > kInOrder)) return false;
    put_in_order(m);
    __syncthreads();
    uint32_t b = s0, e = 0u;
    int k = 0;
    for (; k < m; k++) {  // (every thread the same: a few dozen)
        e = sorted[k];
        b = sr_f2u(__fadd_rn(sr_u2f(b), prob(e)));
        if (sr_u2f(b) >= target) break;
    }
    if (SR_RARE(k >= m)) return false;
    cut->run = sr_u2f(b);
    cut->cutoff = (int)cnt[gc] + k + 1;
    cut->ebits = e;
    return true;
}

// Final Normalize and draw (Sampler.cs:91-92, :553-576) of a sampled row whose members are thousands of its list's entries: members holds
// those of the thread, idx their indices; the threads' entries follow each other in the order of the indices.
// The eight accumulators' terms are put side by side, each accumulator's in the order of the indices, so that a wave passes over a thousand terms
// of its own; over all members with the others' as zeros (finish_from_ordered_list) it is eight times as many rounds.  Putting them there takes 3.7 us, so lists of up
// to 4,096 go that way: 3,000 members 9.6 us to the sum and 10.2 that way, 7,800 13.4 and 17.7.
template <int kPer, typename Prob>
__device__ __forceinline__ void finish_members(const SrFullArgs& a, int n, int row, const uint32_t (&ev)[kPer], const int (&idx)[kPer], uint32_t members, Prob prob,
                                               uint32_t* more, FullSmem& sm)
{
    const int lane = sr_lane(), wave = sr_wave_id(), tid = threadIdx.x, nv8 = (n / 8) * 8;
    unsigned long long* const list = sm.sortbuf;  // index << 32 | bits of the probability, at list_layout
    uint32_t* const terms = more ? more : (uint32_t*)sm.sprob;  // the accumulators' terms, at list_place
    static_assert((2 * kSmall + 8 * 16) * 17 / 16 <= SR_LIST_CAP_BIG + SR_LIST_CAP_BIG / 16 && (kSmall + 8 * 16) * 17 / 16 <= 2 * kSmall,
                  "the terms of 8,192 members fit behind 68 KB, of 4,096 in the two arrays behind the list");
    auto chain_of = [&](int i) -> int { return i < nv8 ? i & 7 : i - (n - 8); };
    // members of every accumulator, two counts to a word (8,192 at most), in front of the thread's
    uint32_t cc[4] = {0u, 0u, 0u, 0u}, in[4];
#pragma unroll
    for (int r = 0; r < kPer; r++)
        if ((members >> r) & 1u) {
            const int c = chain_of(idx[r]);
#pragma unroll
            for (int k = 0; k < 4; k++) cc[k] += (c >> 1) == k ? 1u << (16 * (c & 1)) : 0u;
        }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        in[k] = (uint32_t)sr_wave_incl_scan_i32((int)cc[k]);
        if (lane == SR_WAVE - 1) sm.hist[4 * wave + k] = in[k];
        in[k] -= cc[k];
    }
    __syncthreads();  // (and nobody reads what lies in the lists' places any more)
    uint32_t tot[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int w = 0; w < kW; w++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t v = sm.hist[4 * w + k];
            tot[k] += v;
            in[k] += w < wave ? v : 0u;
        }
    int at = 0, m = 0, base = 0, own_base = 0, own_cnt = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        at += (int)(in[k] & 0xffffu) + (int)(in[k] >> 16);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int cnt = (int)((tot[k] >> (16 * h)) & 0xffffu);
            if (lane == 0) sm.hist[128 + 8 * wave + 2 * k + h] = (uint32_t)base;  // (a copy of the wave's own)
            if (wave == 2 * k + h) { own_base = base; own_cnt = cnt; }
            base += (cnt + 15) & ~15;
            m += cnt;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int r = 0; r < kPer; r++)
        if ((members >> r) & 1u) {
            const int c = chain_of(idx[r]);
            uint32_t p = 0u;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                p = (c >> 1) == k ? in[k] : p;
                in[k] += (c >> 1) == k ? 1u << (16 * (c & 1)) : 0u;
            }
            p = (p >> (16 * (c & 1))) & 0xffffu;
            const uint32_t y = sr_f2u(prob(ev[r]));
            terms[list_place((int)(sm.hist[128 + 8 * wave + c] + p))] = y;
            list[list_layout(at)] = ((unsigned long long)(uint32_t)idx[r] << 32) | (unsigned long long)y;
            at++;
        }
    __syncthreads();
    if (wave < SR_SEQ_CHAINS) {
        float sc = 0.0f;
        for (int b0 = 0; b0 < own_cnt; b0 += 16 * SR_WAVE) {
            float x[16];
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const int i = b0 + 16 * lane + j;
                x[j] = i < own_cnt ? sr_u2f(terms[list_place(own_base + i)]) : 0.0f;
            }
            int dummy;
            sc = sr_seq_wave<16, false>(x, sc, 0.0f, &dummy);
        }
        if (lane == 0) sm.lane_sum[wave] = sc;
    }
    __syncthreads();
    const float l0 = sm.lane_sum[0], l1 = sm.lane_sum[1], l2 = sm.lane_sum[2], l3 = sm.lane_sum[3],
                l4 = sm.lane_sum[4], l5 = sm.lane_sum[5], l6 = sm.lane_sum[6], l7 = sm.lane_sum[7];
    const float sum = __fadd_rn(__fadd_rn(__fadd_rn(l0, l1), __fadd_rn(l2, l3)), __fadd_rn(__fadd_rn(l4, l5), __fadd_rn(l6, l7)));
    const bool scale = sum > 0.0f && sum != 1.0f;
    const float inv = scale ? __fdiv_rn(1.0f, sum) : 1.0f, u = __double2float_rn(sm.u);
    if (!(u > 0.0f)) {  // the running sum starts at p[0] >= 0: index 0 reaches a target of zero whatever it holds
        if (tid == 0 && a.out_tokens) a.out_tokens[row] = 0;
        return;
    }
    if (wave != 0) return;
    // (a thousand at a time to where the draw lands: on average half of them.  Records by a wave each and a walk over them: 6.6 us whatever
    // u is, this 2.6 to 4.7)
    float acc = 0.0f;
    int f = -1;
    for (int b0 = 0; b0 < m && f < 0; b0 += 16 * SR_WAVE) {
        float x[16];
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const int i = b0 + 16 * lane + j;
            const float y = i < m ? sr_u2f((uint32_t)list[list_layout(i)]) : 0.0f;
            x[j] = scale ? __fmul_rn(y, inv) : y;
        }
        acc = sr_seq_wave<16, true>(x, acc, u, &f);
        if (f >= 0) f += b0;
    }
    if (lane == 0) {
        int token = n - 1;  // (the draw ran off the end of the list: the last index, by the rounding fallback)
        if (f >= 0) {
            const unsigned long long v = list[list_layout(f)];
            token = (int)(v >> 32);
            const float y = sr_u2f((uint32_t)v);
            SR_AMB_IF(sr_stop_near(acc, scale ? __fmul_rn(y, inv) : y, u));
        } else {
            SR_AMB_IF(sr_near(acc, u));
        }
        if (a.out_tokens) a.out_tokens[row] = token;
    }
}

template <int kPer>
__device__ __forceinline__ int cut_from_list(const SrFullArgs& a, const SrRow& rd, SrFullState* st, float* p, int n, int slot, int row,
                                             bool do_scale, float inv, int N, FullSmem& sm, uint32_t* more)
{
    constexpr bool kOne = kPer == 1;
    const int tid = threadIdx.x, lane = sr_lane(), wave = sr_wave_id();
    const bool use_top_p = rd.top_p < 1.0f && rd.top_p > 0.0f, use_min_p = rd.min_p > 0.0f;
    const int nseg = seg_count(n);
    const uint32_t from = st->list_from;
    const float mp = do_scale ? __fmul_rn(1.0f, inv) : 1.0f;  // the largest probability: the largest e is expf(0) = 1
    const float thr = use_min_p ? __fmul_rn(rd.min_p, mp) : 0.0f;
    uint32_t* const grp = list_values(more, sm);
    uint32_t* const cnt = more ? (uint32_t*)sm.sortbuf : grp + list_place(SR_LIST_CAP_SMALL);
    int* const off = (int*)sm.segst;  // [nseg] where a segment's entries start
    static_assert(SR_LIST_GROUPS_BIG * 4 <= sizeof(FullSmem::sortbuf) + sizeof(FullSmem::sprob) + sizeof(FullSmem::tags) &&
                  (SR_LIST_GROUPS_SMALL + SR_LIST_CAP_SMALL + SR_LIST_CAP_SMALL / 16) * 4 <=
                      sizeof(FullSmem::sortbuf) + sizeof(FullSmem::sprob) + sizeof(FullSmem::tags), "the tables fit the three arrays");
    static_assert((2 * kT + SR_LIST_CAP_SMALL + SR_LIST_CAP_SMALL / 16) * 4 <= sizeof(FullSmem::sortbuf) + sizeof(FullSmem::sprob) + sizeof(FullSmem::tags) - kT * 4,
                  "... and those of a list with its indices leave them alone");
    // (behind the barrier that follows the gathering)
    // A thread takes 2^sh consecutive entries, as few as the list's length allows (always 16: a list of 1,000 kept one wave
    // busy, 12 us).
    int sh = 0;
    if (!kOne)
        while ((kT << sh) < N) sh++;
    const int per = 1 << sh;
    const int G = min(more ? SR_LIST_GROUPS_BIG : SR_LIST_GROUPS_SMALL, kT << (sh + 1));  // groups: two to an entry, where there is room
    const int i0 = tid << sh;
    const int mine = max(0, min(per, N - i0));
    uint32_t ev[kPer];
#pragma unroll
    for (int r = 0; r < kPer; r++) ev[r] = r < mine ? grp[list_place(i0 + r)] : 0u;
    auto prob = [&](uint32_t ebits) -> float { return do_scale ? __fmul_rn(sr_u2f(ebits), inv) : sr_u2f(ebits); };

    bool in_place = false;  // the cut is known from the list as it stands
    ListCut cut = {};
    if (!kOne && use_top_p) {
        uint32_t valid = 0u;
#pragma unroll
        for (int r = 0; r < kPer; r++)
            if (r < mine && use_min_p) {
                const float y = prob(ev[r]);
                SR_AMB_IF(sr_near(y, thr));  // an entry on the threshold
                valid |= y >= thr ? 1u << r : 0u;
            }
        if (!use_min_p) valid = (1u << mine) - 1u;
        static_assert((3 * 4096 + 4 * kInOrder) * 4 <= sizeof(FullSmem::sortbuf) + sizeof(FullSmem::sprob) + sizeof(FullSmem::tags) &&
                      (SR_LIST_CAP_SMALL + SR_LIST_CAP_SMALL / 16 + 3 * 2048 + 4 * kInOrder) * 4 <= sizeof(FullSmem::sortbuf) + sizeof(FullSmem::sprob) + sizeof(FullSmem::tags),
                      "the tables fit");
        in_place = cut_unsorted<kPer>(ev, valid, from, do_scale, inv, rd.top_p, cnt, more ? 4096 : 2048, &cut, sm);
        if (!in_place) __syncthreads();
    }
    if (!kOne && in_place) {
    } else if (kOne && N <= kT / 4) {
        // A short list: every entry against every other, four threads to an entry (lists of 80 to 140: 1.5 us, 6 by groups)
        const int e = tid >> 2;
        const uint32_t v = e < N ? grp[list_place(e)] : 0u;
        int rank = 0;
#pragma unroll 8
        for (int j = tid & 3; j < N; j += 4) {
            const uint32_t o = grp[list_place(j)];
            rank += (o > v) | ((o == v) & (j < e)) ? 1 : 0;
        }
        rank += (int)sr_dpp_u32<kDppXor1>((uint32_t)rank);
        rank += (int)sr_dpp_u32<kDppXor2>((uint32_t)rank);
        __syncthreads();
        if (e < N && (tid & 3) == 0) grp[list_place(rank)] = v;
    } else {
        // Sorted by value: groups of equal width in the bit patterns, counted, placed, and every value ranked inside its group -- a group of one value (the equal logits of a coarse grid) needs no ranks and is
        // told by its neighbours.  (4,096 groups with their extremes counted along: 12 - 20 us for 14,000 entries, most of it the
        // longest group of every wave looked through 16 times.)
        for (int i = tid; i < G; i += kT) cnt[i] = 0u;
        if (tid == 0) sm.bc[12] = 0u;
        __syncthreads();
        const uint32_t span = 0x3f800000u - min(from, 0x3f800000u);
        int gshift = 0;
        while ((span >> gshift) >= (uint32_t)G) gshift++;
        auto group_of = [&](uint32_t v) -> uint32_t { return min((0x3f800000u - v) >> gshift, (uint32_t)(G - 1)); };
#pragma unroll
        for (int r = 0; r < kPer; r++)
            if (r < mine) atomicAdd(&cnt[group_of(ev[r])], 1u);
        __syncthreads();
        {
            // a wave's share of the groups, 64 at a time: the sums inside each 64, one behind the other inside the wave, then what stands
            // in front of it.  (All of them are read before the first is scanned: 16,384 groups took 4.4 us one by one.)
            constexpr int kRuns = kPer == 1 ? 2 : kPer == 4 ? 8 : SR_LIST_GROUPS_BIG / kT;
            const int g0 = wave * (G / kW), runs = G / kT;
            int c[kRuns], incl[kRuns];
#pragma unroll
            for (int q = 0; q < kRuns; q++) c[q] = q < runs ? (int)cnt[g0 + q * SR_WAVE + lane] : 0;
            int in_wave = 0;
#pragma unroll
            for (int q = 0; q < kRuns; q++) incl[q] = sr_wave_incl_scan_i32(c[q]);
#pragma unroll
            for (int q = 0; q < kRuns; q++) {
                c[q] = in_wave + incl[q] - c[q];
                in_wave += __builtin_amdgcn_readlane(incl[q], SR_WAVE - 1);
            }
            if (lane == 0) sm.redi[wave] = in_wave;
            __syncthreads();
            int before = 0;
#pragma unroll
            for (int w = 0; w < kW; w++) before += w < wave ? sm.redi[w] : 0;
#pragma unroll
            for (int q = 0; q < kRuns; q++)
                if (q < runs) cnt[g0 + q * SR_WAVE + lane] = (uint32_t)(before + c[q]);
        }
        __syncthreads();
        uint32_t at[kPer];  // (all places are asked for before the first is used)
#pragma unroll
        for (int r = 0; r < kPer; r++) at[r] = r < mine ? atomicAdd(&cnt[group_of(ev[r])], 1u) : 0u;
#pragma unroll
        for (int r = 0; r < kPer; r++)
            if (r < mine) grp[list_place((int)at[r])] = ev[r];
        __syncthreads();  // cnt[g] is now where group g ends
        constexpr uint32_t kMixed = 0x80000000u;  // (of cnt: the group holds more than one value)
        uint32_t v[kPer];
        uint32_t last = (mine > 0 && i0 > 0) ? grp[list_place(i0 - 1)] : 0u;
#pragma unroll
        for (int r = 0; r < kPer; r++) v[r] = r < mine ? grp[list_place(i0 + r)] : 0u;
#pragma unroll
        for (int r = 0; r < kPer; r++) {
            if (r < mine && v[r] != last && i0 + r > 0 && group_of(v[r]) == group_of(last)) atomicOr(&cnt[group_of(v[r])], kMixed);
            last = v[r];
        }
        __syncthreads();
        int rank[kPer];
#pragma unroll
        for (int r = 0; r < kPer; r++) {
            rank[r] = i0 + r;
            const uint32_t ce = r < mine ? cnt[group_of(v[r])] : 0u;
            if (ce & kMixed) {
                const int i = i0 + r;
                const uint32_t g = group_of(v[r]);
                const int b = g > 0u ? (int)(cnt[g - 1u] & ~kMixed) : 0, e = (int)(ce & ~kMixed);
                if (e - b > 128) sm.bc[12] = 1u;
                int k = b;
                for (int j0 = b; j0 < min(e, b + 128); j0 += 4) {  // (four on their way at a time)
                    uint32_t o[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) o[q] = grp[list_place(min(j0 + q, N - 1))];
#pragma unroll
                    for (int q = 0; q < 4; q++) k += (j0 + q < e) & ((o[q] > v[r]) | ((o[q] == v[r]) & (j0 + q < i))) ? 1 : 0;
                }
                rank[r] = k;
            }
        }
        __syncthreads();
        if (sm.bc[12] != 0u) return kListGeneral;
#pragma unroll
        for (int r = 0; r < kPer; r++)
            if (r < mine) grp[list_place(rank[r])] = v[r];
    }
    // the survivors of min-p (the largest ones)
    int ns = in_place ? cut.ns : N;
    if (use_min_p && !in_place) {
        int c = 0;
#pragma unroll
        for (int r = 0; r < kPer; r++)
            if (r < mine) {
                const float y = prob(ev[r]);
                SR_AMB_IF(sr_near(y, thr));  // an entry on the threshold
                c += y >= thr ? 1 : 0;
            }
        ns = blk_sum_i(c, sm);
    }
    __syncthreads();
    if (ns <= 0) return kListGeneral;
    FPROF(a, slot, 11);
    // The indices of the thread's entries, asked for in front of the cut where there is room to keep them: an entry's place in the
    // list names its segment and its place there.  (A pass over all segments behind the cut, for the members' indices: 5 - 6 us.)
    const int32_t* gi = a.sort_vals_in + (size_t)slot * (size_t)a.sort_stride;
    int idx[kPer];
    auto fetch_indices = [&]() __attribute__((always_inline)) {
        if (kOne) {
            idx[0] = tid < N ? (int)list_ids(sm)[tid] : 0;
            return;
        }
        int sg = 0;
        for (int half = SR_SEG_MAX / 2; half > 0; half >>= 1)  // the last segment that starts at the first entry or in front of it
            if (sg + half < nseg && off[sg + half] <= i0) sg += half;
        int start = off[sg], next = sg + 1 < nseg ? off[sg + 1] : N;
#pragma unroll
        for (int r = 0; r < kPer; r++) {
            idx[r] = 0;
            if (r < mine) {
                while (next <= i0 + r) {  // (ends at the last segment, whose entries end the list)
                    sg++;
                    start = next;
                    next = sg + 1 < nseg ? off[sg + 1] : N;
                }
                idx[r] = gi[(size_t)sg * SR_SEG_TERMS + (size_t)(i0 + r - start)];
            }
        }
    };
    if (kPer <= 4) fetch_indices();
    int found = -1;
    if (!kOne && in_place) {
        found = cut.found ? cut.cutoff - 1 : -1;
        if (found < 0 && from > 1u && min_p_list_from(rd) < from) return kListGeneral;
        if (found >= 0 && from > 1u && prob(from - 1u) >= prob(cut.ebits)) return kListGeneral;
    } else if (use_top_p) {
        auto fetch = [&](int b0, float (&x)[SR_SEQ_RUN]) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < SR_SEQ_RUN; j++) {
                const int i = b0 + lane * SR_SEQ_RUN + j;
                x[j] = i < ns ? prob(grp[list_place(i)]) : 0.0f;
            }
        };
        if (kOne || ns <= SR_SEG_TERMS) {
            if (wave == 0) {
                float x[SR_SEQ_RUN];
                fetch(0, x);
                int at;
                const float s = sr_seq_wave<SR_SEQ_RUN, true>(x, 0.0f, rd.top_p, &at);
                if (lane == 0) { sm.segbc[1] = (uint32_t)at; sm.segbc[2] = sr_f2u(s); }
            }
        } else {
            // a thousand to a wave: their records, as for any long sum, and one wave walks them (one wave by itself: 6.5 us for
            // 3,500; by the workgroup's tiles as many)
            SeqSegFunc* const recs = (SeqSegFunc*)(sm.tags + kSmall / 2);  // (the groups are done with)
            static_assert(SR_LIST_CAP_BIG / SR_SEG_TERMS <= kW && kW * sizeof(SeqSegFunc) <= kSmall * 2 &&
                          (SR_LIST_CAP_SMALL + SR_LIST_CAP_SMALL / 16) * 4 <= sizeof(FullSmem::sortbuf) + sizeof(FullSmem::sprob), "a wave each; the records fit");
            const int nrec = seg_count(ns);
            float x[SR_SEQ_RUN], own = 0.0f;
            if (wave < nrec) {
                fetch(wave * SR_SEG_TERMS, x);
#pragma unroll
                for (int j = 0; j < SR_SEQ_RUN; j++) own += x[j];
                own = sr_wave_sum_f32(own);
                if (lane == 0) sm.redf[wave] = own;
            }
            __syncthreads();
            if (wave < nrec) {
                float before = 0.0f;
#pragma unroll
                for (int w = 0; w < kW; w++) before += w < wave ? sm.redf[w] : 0.0f;
                seg_make_record(x, wave, (double)before, recs + wave, own);
            }
            __syncthreads();
            if (wave == 0) {
                int at;
                const float s = seg_walk_from<true, false, true>([&](int sg, float (&y)[SR_SEQ_RUN]) __attribute__((always_inline)) { fetch(sg * SR_SEG_TERMS, y); },
                                                    nrec, recs, 0.0f, rd.top_p, &at, nullptr);
                if (lane == 0) { sm.segbc[1] = (uint32_t)at; sm.segbc[2] = sr_f2u(s); }
            }
        }
        __syncthreads();
        found = (int)sm.segbc[1];
        // the list ended before the sum was there, and the row goes on behind it
        if (found < 0 && from > 1u && min_p_list_from(rd) < from) return kListGeneral;
        // ... or an entry behind the list's end shares the probability at the cut
        if (found >= 0 && from > 1u && prob(from - 1u) >= prob(grp[list_place(found)])) return kListGeneral;
        if (tid == 0) {
            const float run = sr_u2f(sm.segbc[2]);
            if (found >= 0) {
                const float y = prob(grp[list_place(found)]);
                SR_AMB_IF(sr_stop_near(run, y, rd.top_p) || (found + 1 < ns && prob(grp[list_place(found + 1)]) == y));
            } else {
                SR_AMB_IF(sr_near(run, rd.top_p));
            }
        }
    }
    const int cutoff = found >= 0 ? found + 1 : ns, m = cutoff;
    float ycut;
    bool tie;
    if (!kOne && in_place) {
        // the value at the cut (where nothing was cut, the smallest that is left), and whether an entry behind the cut has it
        if (found >= 0) {
            ycut = prob(cut.ebits);
        } else {
            uint32_t least = 0xffffffffu;
#pragma unroll
            for (int r = 0; r < kPer; r++)
                if (r < mine) {
                    const float y = prob(ev[r]);
                    if (!use_min_p || y >= thr) least = min(least, sr_f2u(y));
                }
            least = sr_wave_min_u32(least);
            if (lane == 0) sm.redu[wave] = least;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < kW; w++) least = min(least, sm.redu[w]);
            ycut = sr_u2f(least);
        }
        int c = 0;
#pragma unroll
        for (int r = 0; r < kPer; r++) c += r < mine && prob(ev[r]) >= ycut ? 1 : 0;
        tie = blk_sum_i(c, sm) > cutoff;
        if (tid == 0) SR_AMB_IF(found >= 0 ? sr_stop_near(cut.run, ycut, rd.top_p) || tie : sr_near(cut.run, rd.top_p));
    } else {
        ycut = prob(grp[list_place(cutoff - 1)]);
        tie = false;
    }
    const bool finish = a.mode == 0 && m <= a.finish_most;
    if (!finish && !a.prepared) return kListGeneral;
    // Members: everything above the value at the cut, and of the entries equal to it the first ones by index -- nearly always all of
    // them: nothing behind the cut has its value.
    if (!in_place) tie = cutoff < ns && prob(grp[list_place(cutoff)]) == ycut;
    if (kPer > 4) fetch_indices();
    uint32_t members = 0u;
    int last_here = -1;
    if (tie) {
        int gt = 0, eq = 0;
#pragma unroll
        for (int r = 0; r < kPer; r++)
            if (r < mine) {
                const float y = prob(ev[r]);
                gt += y > ycut ? 1 : 0;
                eq += y == ycut ? 1 : 0;
            }
        int tot_eq;
        const int eq0 = blk_excl_scan(eq, &tot_eq, sm);
        const int keep_eq = cutoff - blk_sum_i(gt, sm);
        int k = eq0;
#pragma unroll
        for (int r = 0; r < kPer; r++)
            if (r < mine) {
                const float y = prob(ev[r]);
                const bool same = y == ycut;
                if (y > ycut || (same && k < keep_eq)) members |= 1u << r;
                if (same && k == keep_eq - 1) last_here = r;
                k += same ? 1 : 0;
            }
    } else {
#pragma unroll
        for (int r = 0; r < kPer; r++)
            if (r < mine && prob(ev[r]) >= ycut) members |= 1u << r;
    }
    if (kPer > 4 && finish && m > SR_SEG_TERMS) {
        finish_members<kPer>(a, n, row, ev, idx, members, prob, more, sm);
        return kListDone;
    }
    if (finish) {
        // in the order of the list, which is the order of the indices
        int tot;
        int at = blk_excl_scan(__popc(members), &tot, sm);  // (its barriers: the sorted values have been read)
        const bool laid_out = kOne && m > SR_WAVE;
#pragma unroll
        for (int r = 0; r < kPer; r++)
            if ((members >> r) & 1u) {
                sm.sortbuf[laid_out ? list_layout(at) : at] = ((unsigned long long)(0xffffffffu - (uint32_t)idx[r]) << 32) | (unsigned long long)sr_f2u(prob(ev[r]));
                at++;
            }
        __syncthreads();
        finish_from_ordered_list(a, p, n, m, row, sm, NoFill(), m <= kSmall ? kSmall : 2 * kSmall, laid_out);
        return kListDone;
    }
    // Left to the whole device: the members' part of every segment and of every half block of the eight accumulators.  (In whole
    // numbers: an atomic addition of floats in shared memory takes a wave some 190 cycles, 9 us for 5,000 members.)
    if (tid == 0) sm.bc[9] = (uint32_t)n;  // (the last index that is a member of the value at the cut; without a tie all are)
    __syncthreads();                       // (the sorted values have been read)
    unsigned long long* const ssum = sm.sortbuf;
    unsigned long long* const csum = ssum + SR_SEG_MAX;
    static_assert((SR_SEG_MAX + SR_SEG_MAX / SR_HALF_BLOCK_SEGS * SR_SEQ_CHAINS) * 8 <= sizeof(FullSmem::sortbuf), "the sums fit");
    for (int i = tid; i < nseg; i += kT) ssum[i] = 0ull;
    for (int i = tid; i < a.chain_stride; i += kT) csum[i] = 0ull;
    __syncthreads();
    FPROF(a, slot, 12);
    const int nv8 = (n / 8) * 8;
    {
        unsigned long long run = 0ull;  // of the entries of one segment, which follow each other
        int sg = 0;
#pragma unroll
        for (int r = 0; r < kPer; r++)
            if ((members >> r) & 1u) {
                const unsigned long long units = e_units(ev[r]);
                if (idx[r] / SR_SEG_TERMS != sg && run != 0ull) {
                    atomicAdd(&ssum[sg], run);
                    run = 0ull;
                }
                sg = idx[r] / SR_SEG_TERMS;
                run += units;
                if (idx[r] < nv8) atomicAdd(&csum[idx[r] / (SR_HALF_BLOCK_SEGS * SR_SEG_TERMS) * SR_SEQ_CHAINS + (idx[r] & (SR_SEQ_CHAINS - 1))], units);
                if (r == last_here) sm.bc[9] = (uint32_t)idx[r];
            }
        if (run != 0ull) atomicAdd(&ssum[sg], run);
    }
    __syncthreads();
    for (int i = tid; i < nseg; i += kT) a.seg_sum[(size_t)slot * a.seg_stride + i] = (float)ssum[i] * 0x1p-40f;
    for (int i = tid; i < a.chain_stride; i += kT) a.chain_sum[(size_t)slot * a.chain_stride + i] = (float)csum[i] * 0x1p-40f;
    row_deferred(a, st, inv, ycut, (int)sm.bc[9], sm);
    return kListDeferred;
}

// ... of a list of at most 64 entries, a sharp row's: by one wave, an entry a lane.  sm.hist[0, N) holds the values of e, sm.hist[64,
// 64 + N) the indices, in the order of the indices.  (The general way's block-wide steps took 14 us for 20 entries.)
__device__ __forceinline__ int cut_from_short_list(const SrFullArgs& a, const SrRow& rd, SrFullState* st, float* p, int n, int slot, int row,
                                                   bool do_scale, float inv, int N, FullSmem& sm)
{
    const int tid = threadIdx.x, lane = sr_lane();
    const bool use_top_p = rd.top_p < 1.0f && rd.top_p > 0.0f, use_min_p = rd.min_p > 0.0f;
    const uint32_t from = st->list_from;
    if (sr_wave_id() == 0) {
        const float mp = do_scale ? __fmul_rn(1.0f, inv) : 1.0f;  // the largest probability: the largest e is expf(0) = 1
        const float thr = use_min_p ? __fmul_rn(rd.min_p, mp) : 0.0f;
        const float e = lane < N ? sr_u2f(sm.hist[lane]) : 0.0f;
        const int idx = lane < N ? (int)sm.hist[SR_WAVE + lane] : 0;
        const float y = do_scale ? __fmul_rn(e, inv) : e;
        bool amb = lane < N && use_min_p && sr_near(y, thr);
        const bool in = lane < N && !(use_min_p && y < thr);
        const int ns = __popcll(__ballot(in));
        // place in the order of the values, equal ones by index
        const float key = in ? y : -1.0f;
        int rank = 0;
        for (int j = 0; j < N; j++) {
            const float o = sr_u2f((uint32_t)__builtin_amdgcn_readlane((int)sr_f2u(key), j));
            rank += (o > key || (o == key && j < lane)) ? 1 : 0;
        }
        if (in) sm.sprob[rank] = y;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const float sorted = lane < ns ? sm.sprob[lane] : 0.0f;
        auto at = [&](int i) -> float { return sr_u2f((uint32_t)__builtin_amdgcn_readlane((int)sr_f2u(sorted), i)); };
        int found = -1;
        if (use_top_p) {
            float run = 0.0f;
            for (int i = 0; i < ns && found < 0; i++) {
                run = __fadd_rn(run, at(i));
                if (run >= rd.top_p) found = i;
            }
            const float behind = from > 1u ? __fmul_rn(sr_u2f(from - 1u), do_scale ? inv : 1.0f) : -1.0f;
            if (found >= 0 ? behind >= at(found) : from > 1u && min_p_list_from(rd) < from) {
                // the list ended before the sum was there, and the row goes on behind it -- or an entry behind the list's
                // end shares the probability at the cut
                found = -2;
            } else if (found >= 0) {
                amb = amb || sr_stop_near(run, at(found), rd.top_p) || (found + 1 < ns && at(found + 1) == at(found));
            } else {
                amb = amb || sr_near(run, rd.top_p);
            }
        }
        const int cutoff = found >= 0 ? found + 1 : ns;
        const bool member = in && rank < cutoff;
        const unsigned long long ms = __ballot(member);
        if (__ballot(amb) != 0ull && found != -2 && lane == 0) sm.bc[SR_AMB_WORD] = 1u;
        if (member) {
            sm.sortbuf[__popcll(ms & ((1ull << lane) - 1ull))] = ((unsigned long long)(0xffffffffu - (uint32_t)idx) << 32) | (unsigned long long)sr_f2u(y);
            if (rank == cutoff - 1) { sm.bc[9] = (uint32_t)idx; sm.bc[10] = sr_f2u(y); }
        }
        if (lane == 0) sm.segbc[1] = (uint32_t)(found == -2 ? 0 : cutoff);
    }
    __syncthreads();
    const int m = (int)sm.segbc[1];
    if (m <= 0) return kListGeneral;
    if (a.mode == 0) {
        finish_from_ordered_list(a, p, n, m, row, sm);
        return kListDone;
    }
    // The members' sum and the draw are at hand: k_prepared_row has the row to write, nothing to meet for.  (With what it leaves out for
    // rows that their largest entry decides, distributions with tokens, us before and now: 16 rows of 262,144, every third uncut, 67 -> 54, 64 of
    // 151,936 87 -> 74, 16 bf16 rows of 100,003 49 -> 40, one row of 151,936 39 -> 31.)
    const float inv2 = finish_short_list(a, n, m, row, sm);
    row_deferred(a, st, inv, sr_u2f(sm.bc[10]), (int)sm.bc[9], sm);
    if (tid == 0) {
        st->mul2 = inv2;
        st->drawn = a.seq;
    }
    return kListClosed;
}

// A row whose workgroups did not meet (SrFullState::late): everything by this workgroup alone, from the logits -- the adjusted
// row and its maximum as an ordered key (0xffffffff: it holds a NaN), then e in place.  Slow; no launch is known to need it.
__device__ __forceinline__ float row_alone_logit(const SrFullArgs& a, const char* rowp, const uint32_t* mrow, int i)
{
    const float x = a.dtype == 1 ? load_logit<2>(rowp, i) : load_logit<4>(rowp, i);
    return (mrow && !((mrow[i >> 5] >> (i & 31)) & 1u)) ? SR_NEG_INF : x;
}
__device__ __forceinline__ uint32_t row_alone(const SrFullArgs& a, const SrRow& rd, float* p, int n, int row, FullSmem& sm)
{
    const int tid = threadIdx.x;
    const char* rowp = (const char*)a.logits + (size_t)row * (size_t)a.row_stride * (a.dtype == 1 ? 2 : 4);
    const uint32_t* mrow = (rd.mask_row >= 0) ? a.mask + (size_t)rd.mask_row * a.mask_stride : nullptr;
    const bool scale = rd.temperature != 1.0f, pen = (rd.flags & SR_ROWFLAG_HAS_PENALTY) != 0u;
    const float inv_temp = scale ? __fdiv_rn(1.0f, rd.temperature) : 1.0f;
    for (int i = tid; i < n; i += kT) {
        const float x = row_alone_logit(a, rowp, mrow, i);
        p[i] = scale ? __fmul_rn(x, inv_temp) : x;
    }
    sr_drain_stores();
    __syncthreads();
    const SrEdit* ed = a.edits + rd.edit_off;
    for (int e = tid; e < rd.edit_cnt; e += kT) {
        const float x = edited_logit(row_alone_logit(a, rowp, mrow, ed[e].id), ed[e], rd, true, pen);
        p[ed[e].id] = scale ? __fmul_rn(x, inv_temp) : x;
    }
    sr_drain_stores();
    __syncthreads();
    uint32_t k = 0u;
    row_pass<false>(p, n, [&](float x, int) -> float {
        k = max(k, x != x ? 0xffffffffu : sr_okey(x));
        return x;
    });
    k = (uint32_t)(blk_max_u64((unsigned long long)k, sm));
    if (k != 0xffffffffu && k > 0x007fffffu) {
        const float m = sr_okey_inv(k);
        row_pass<true>(p, n, [&](float x, int) -> float { return sr_expf(__fsub_rn(x, m)); });
        sr_drain_stores();
        __syncthreads();
    }
    return k;
}

// ---- stage 3: softmax, top-k, min-p, top-p on the work row --------------------------------------------
// One workgroup per row, one launch: the row is cut, normalised and drawn from here.  A nucleus that the walk by
// slabs cannot close has its survivors compacted into the row's sort segment and sorted there by this workgroup.
// kLater: a verifier's launch with factor_later (what that asks for cost all others 0.7 us here)
template <bool kLater>
__global__ __launch_bounds__(kT) void k_full_row(SrFullArgs a)
{
    __shared__ FullSmem sm;
    const int tid = threadIdx.x;
    const int slot = blockIdx.x;
    const int n = a.vocab;
    SrFullState* st = a.state + slot;
    // What does not hang on the row's descriptor is asked for beside it: the row's state, the first records of its sum (by the
    // wave that will walk them) and how many entries its segments have listed (by the others).
    const uint32_t st_late = st->late, st_list_from = st->list_from, st_decided = st->decided;
    const unsigned long long st_maxkey = st->maxkey;
    // (Whatever `late` says: only a workgroup that had all of the row's words decides, and one that decides has written the token.  Written once
    // more, it could come after the caller has it and has begun the next call: into that one's results, from logits given away.)
    if (st_decided == a.seq) return;
    SegRec first64 = {};
    constexpr int kCntAhead = 4;
    int cnt_ahead[kCntAhead] = {};
    if (a.seg_func) {
        const int nseg = seg_count(n);
        if (sr_wave_id() == 0) {
            seg_load_rec<false>(a.seg_func + (size_t)slot * a.seg_stride, sr_lane(), nseg, first64);
        } else {
#pragma unroll
            for (int q = 0; q < kCntAhead; q++) {
                const int g = q * SR_WAVE + sr_lane();
                cnt_ahead[q] = g < nseg ? (int)a.seg_cnt[(size_t)slot * a.seg_stride + g] : 0;
            }
        }
    }
    const int row = a.row_list[slot];
    const SrRow rd = a.rows[row];
    float* p = a.work + (size_t)(a.work_by_row ? row : slot) * a.work_stride;
    const bool greedy = rd.temperature <= 0.0f;
    const bool use_top_p = rd.top_p < 1.0f && rd.top_p > 0.0f;
    if (tid == 0) {
        sm.bc[SR_AMB_WORD] = 0u;  // (every path that can set it passes a barrier first)
        // what the reader of a row that is not left to it expects: factors of 1
        st->mul1 = st->mul2 = 1.0f;
    }
    // (the next launch of the pass over the whole device finds the row's mass by size at zero)
    if (a.seg_func && tid < kMassBuckets) a.mass[(size_t)slot * kMassBuckets + tid] = 0.0f;

    if (greedy) {
        // Greedy / GreedyWithHistoryPenalties on the adjusted row; distributions become one-hot
        const int am = row_argmax(p, n, sm);
        if (a.mode != 0) {
            __syncthreads();
            row_pass<true>(p, n, [&](float, int i) -> float { return (i == am) ? 1.0f : 0.0f; });
        }
        if (tid == 0) {
            if (a.out_tokens) a.out_tokens[row] = am;
            if (a.out_flags) a.out_flags[row] = SR_KFLAG_GREEDY | SR_KFLAG_FULL;
        }
        return;
    }

    // The uniform may lie in host memory, a trip over the bus: one thread asks for it now and hands it on when the sum is there.
    double u_row = 0.0;
    if (tid == kT - 1 && a.mode != 1) u_row = a.uniforms[(size_t)row * a.uniforms_per_row];
    {
        FPROF(a, slot, 0);
        // Softmax (Sampler.cs:448-472): the maximum and e = expf(x - max) were computed by the kernels before
        const bool alone = a.seg_func != nullptr && (st_late == a.seq || full_maxkey_of(a, st_maxkey) == kKeyInf);
        const bool walked = a.seg_func != nullptr && !alone;
        // (a list that would have been too long was not made)
        const bool has_list = walked && row_is_listed(rd, a) && st_list_from != 0u, plain = walked && row_is_plain(rd, a);
        // A row whose distribution is asked for as well, nothing cuts, and its largest entry decides: k_prepared_row makes neither the
        // records of the draw nor the walk over them (SrFullState::drawn).  It costs nothing here: a wave beside the one that walks.
        const bool asks_draw = !kLater && plain && a.prepared && a.mode == 2;
        float* const e_row = walked ? row_e(a, slot) : p;
        const uint32_t mk = SR_RARE(alone) ? row_alone(a, rd, p, n, row, sm) : full_maxkey_of(a, st_maxkey);
        const bool any_nan = mk == 0xffffffffu;
        const float m = mk == 0u ? SR_NEG_INF : sr_okey_inv(mk);
        FPROF(a, slot, 1);
        uint32_t flags = SR_KFLAG_FULL;
        bool fused = false;  // scaling, min-p and the count of survivors were done in one pass
        int survivors = 0;   // ... this thread's share of the count
        int ns_listed = -1;  // >= 0: the block-wide count, and sm.sortbuf[0, ns_listed) holds the survivors
        bool row_unwritten = false;  // the row still holds expf(x - max): it will be finished from the list
        bool no_slabs = false;       // the nucleus is known to be too large for the walk by slabs
        if (SR_RARE(any_nan || sr_f2u(m) == 0xff800000u)) {
            const float uni = n > 0 ? __fdiv_rn(1.0f, (float)n) : 0.0f;
            row_pass<true>(p, n, [&](float, int) -> float { return uni; });
            flags |= SR_KFLAG_DEGENERATE;
            if (tid == kT - 1) sm.u = u_row;
            __syncthreads();
        } else {
            if (SR_RARE(row_edits_on_the_fly(rd, a) && !a.seg_func)) {
                // the ids that the row's edits touch were left out of the expf pass: their e, from the adjusted values
                // that k_full_edits kept
                const float* vals = (const float*)(a.edit_tab + (size_t)slot * (size_t)a.edit_tab_stride + (n + 31) / 32);
                const SrEdit* ed = a.edits + rd.edit_off;
                for (int e = tid; e < rd.edit_cnt; e += kT) p[ed[e].id] = sr_expf(__fsub_rn(vals[e], m));
                sr_drain_stores();  // (this compute unit has not read these lines before: the loads below find them in L2)
                __syncthreads();
            }
            extern __shared__ uint32_t more_lds[];  // when a.big_slabs, else nothing
            uint32_t* const more = a.big_slabs ? more_lds : nullptr;
            int dummy;
            float sum;
            int n_list = 0;
            if (SR_USUAL(walked)) {
                // the whole device has prepared the sum (k_full_softmax_seg): one wave walks the segments' records while the
                // others fetch the row's list, if it has one
                if (sr_wave_id() == 0) {
                    ERow er;
                    er.e = e_row;
                    er.lg = nullptr;
                    if (kLater && row_e_open(rd, a)) {
                        er.lg = (const float*)a.logits + (size_t)row * (size_t)a.row_stride;
                        er.inv_temp = row_inv_temp(rd);
                        er.max = m;
                        er.tab = (const uint64_t*)sm.sortbuf;  // (no list is fetched beside this walk)
                        if (sr_lane() < 32) ((uint64_t*)sm.sortbuf)[sr_lane()] = sr_exp2f_tab[sr_lane()];
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                        __builtin_amdgcn_wave_barrier();
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                    }
                    const bool aligned = ((uintptr_t)e_row & 15u) == 0u;
                    const float s = seg_walk_from<false>([&](int seg, float (&x)[SR_SEQ_RUN]) __attribute__((always_inline)) {
                        const int i0 = seg * SR_SEG_TERMS + sr_lane() * SR_SEQ_RUN;
                        if (!kLater || !er.lg) {
                            seq_load_run(e_row, aligned, i0, n, x);
                            return;
                        }
                        if (seg * SR_SEG_TERMS + SR_SEG_TERMS <= n) {
#pragma unroll
                            for (int j = 0; j < SR_SEQ_RUN; j += 4) {
                                const float4 l = sr_load_f4(er.lg + i0 + j);
                                x[j] = l.x; x[j + 1] = l.y; x[j + 2] = l.z; x[j + 3] = l.w;
                            }
                        } else {
#pragma unroll
                            for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = er.lg[min(i0 + j, n - 1)];
                        }
#pragma unroll
                        for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = i0 + j < n ? er.of(x[j]) : 0.0f;
                    }, seg_count(n), a.seg_func + (size_t)slot * a.seg_stride, 0.0f, 0.0f, &dummy, nullptr, &first64);
                    if (sr_lane() == 0) sm.segbc[0] = sr_f2u(s);
                } else if (kLater && sr_wave_id() == 1) {
                    // about the same sum, without the roundings of n additions one behind the other (spec_spread)
                    const int nseg = seg_count(n);
                    float about = 0.0f;
                    for (int g = sr_lane(); g < nseg; g += SR_WAVE) about += a.seg_sum[(size_t)slot * a.seg_stride + g];
                    about = sr_wave_sum_f32(about);
                    if (sr_lane() == 0) sm.segbc[3] = sr_f2u(about);
                } else if (asks_draw) {
                    // (where e = 1 stands: the row is not decided unless all others' e add up to less than that)
                    if (sr_wave_id() == 1) {
                        const double u = a.uniforms[(size_t)row * a.uniforms_per_row];
                        const int nseg = seg_count(n), lane = sr_lane();
                        float all = 0.0f, front = 0.0f, own = 0.0f;
                        int top = -1;
                        for (int g0 = 0; g0 < nseg; g0 += SR_WAVE) {
                            const float part = g0 + lane < nseg ? a.seg_sum[(size_t)slot * a.seg_stride + g0 + lane] : 0.0f;
                            const unsigned long long has = __ballot(part >= 1.0f);
                            const int l = has != 0ull ? (int)__ffsll((long long)has) - 1 : SR_WAVE;
                            all += part;
                            front += top < 0 && lane < l ? part : 0.0f;
                            own += top < 0 && lane == l ? part : 0.0f;
                            if (has != 0ull) top = g0 + l;
                        }
                        const bool yes = row_decided(rd, n, sr_wave_sum_f32(all), sr_wave_sum_f32(front), sr_wave_sum_f32(own), __double2float_rn(u));
                        if (lane == 0) sm.segbc[3] = top >= 0 && yes ? 1u : 0u;
                    }
                } else if (has_list) {
                    // where the segments' entries start: every wave adds up the counts for itself and writes all of them, the
                    // same values (a scan by the workgroup, in front of the walk, was two barriers)
                    const int nseg = seg_count(n), lane = sr_lane();
                    int* const off = (int*)sm.segst;
                    static_assert(kCkpt >= SR_WAVE, "a word per entry of a short list");
                    auto count = [&](int g0, int c) __attribute__((always_inline)) {
                        const int incl = sr_wave_incl_scan_i32(c), o = n_list + incl - c, g = g0 + lane;
                        if (g < nseg) off[g] = o;
                        if (sr_wave_id() == 1)  // where every entry of a short list lies
                            for (int k = 0; k < c && o + k < SR_WAVE; k++) ((int*)sm.ckpt)[o + k] = g * SR_SEG_TERMS + k;
                        n_list += __builtin_amdgcn_readlane(incl, SR_WAVE - 1);
                    };
#pragma unroll
                    for (int q = 0; q < kCntAhead; q++)
                        if (q * SR_WAVE < nseg) count(q * SR_WAVE, cnt_ahead[q]);
                    for (int g0 = kCntAhead * SR_WAVE; g0 < nseg; g0 += SR_WAVE)
                        count(g0, g0 + lane < nseg ? (int)a.seg_cnt[(size_t)slot * a.seg_stride + g0 + lane] : 0);
                    if (tid == SR_WAVE) sm.segbc[3] = (uint32_t)n_list;
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                    if (n_list <= SR_WAVE) {
                        const int l = tid - SR_WAVE;
                        if (l < n_list) {
                            const size_t at = (size_t)slot * (size_t)a.sort_stride + (size_t)((const int*)sm.ckpt)[l];
                            sm.hist[l] = a.sort_keys_in[at];
                            sm.hist[SR_WAVE + l] = (uint32_t)a.sort_vals_in[at];
                        }
                    } else if (n_list <= list_cap(more != nullptr)) {
                        uint32_t* const grp = list_values(more, sm);
                        const uint32_t* gk = a.sort_keys_in + (size_t)slot * (size_t)a.sort_stride;
                        const int32_t* gi = a.sort_vals_in + (size_t)slot * (size_t)a.sort_stride;
                        // (four segments' first entries on their way at a time)
                        for (int s0 = sr_wave_id() - 1; s0 < nseg; s0 += 4 * (kW - 1)) {
                            uint32_t v[4], id[4] = {0u, 0u, 0u, 0u};
                            int at[4], len[4];
#pragma unroll
                            for (int q = 0; q < 4; q++) {
                                const int sg = s0 + q * (kW - 1);
                                at[q] = sg < nseg ? off[sg] : 0;
                                len[q] = sg < nseg ? (sg + 1 < nseg ? off[sg + 1] : n_list) - at[q] : 0;
                                v[q] = lane < len[q] ? gk[(size_t)sg * SR_SEG_TERMS + lane] : 0u;
                            }
                            if (n_list <= kT) {
#pragma unroll
                                for (int q = 0; q < 4; q++) {
                                    const int sg = s0 + q * (kW - 1);
                                    id[q] = lane < len[q] ? (uint32_t)gi[(size_t)sg * SR_SEG_TERMS + lane] : 0u;
                                }
                            }
#pragma unroll
                            for (int q = 0; q < 4; q++) {
                                const int sg = s0 + q * (kW - 1);
                                if (lane < len[q]) grp[list_place(at[q] + lane)] = v[q];
                                if (lane < len[q] && n_list <= kT) list_ids(sm)[at[q] + lane] = id[q];
                                for (int i = lane + SR_WAVE; i < len[q]; i += SR_WAVE) {
                                    grp[list_place(at[q] + i)] = gk[(size_t)sg * SR_SEG_TERMS + i];
                                    if (n_list <= kT) list_ids(sm)[at[q] + i] = (uint32_t)gi[(size_t)sg * SR_SEG_TERMS + i];
                                }
                            }
                        }
                    }
                }
                __syncthreads();
                sum = sr_u2f(sm.segbc[0]);
                if (has_list) n_list = (int)sm.segbc[3];
            } else {
                sum = seq_sum_row<false>(p, n, 0.0f, 0.0f, &dummy, sm);
            }
            if (tid == kT - 1) sm.u = u_row;
            __syncthreads();
            FPROF(a, slot, 2);
            const bool do_scale = sum > 0.0f && sum != 1.0f;
            const float inv = do_scale ? __fdiv_rn(1.0f, sum) : 1.0f;
            // (the verifier asks for the factors of few of its positions: k_spec_factor)
            if (plain && (a.prepared || (kLater && spec_by_ratio(rd)))) {
                row_deferred(a, st, inv, -1.0f, 0, sm);
                if (tid == 0) {
                    if (asks_draw) st->drawn = sm.segbc[3] != 0u ? a.seq : 0u;
                    if (kLater) {
                        st->e_open = row_e_open(rd, a) ? a.seq : 0u;
                        st->mul2 = __fdiv_rn(sum, sr_u2f(sm.segbc[3]));
                    }
                    st->flags = flags;
                }
                return;
            }
            if (a.lazy_scale && a.mode == 1 && !(rd.top_k > 0 && rd.top_k < n) && !(rd.min_p > 0.0f) && !use_top_p) {
                // No filter touches the row: its final entries are fmul(fmul(e, inv), inv2) with inv2 from the final
                // Normalize (Sampler.cs:91-92) over the scaled values.  The reader applies the two factors; the row
                // keeps e and is not written again.
                const float sum2 = tp_sum_row(p, n, inv, true, sm);
                const float inv2 = (sum2 > 0.0f && sum2 != 1.0f) ? __fdiv_rn(1.0f, sum2) : 1.0f;
                if (tid == 0) {
                    st->mul1 = inv;
                    st->mul2 = inv2;
                    st->n_survivors = 0;
                    st->flags = flags;
                    if (a.out_flags) a.out_flags[row] = flags;
                }
                return;
            }
            if (has_list) {
                int way = kListGeneral;
                if (n_list > 0 && n_list <= SR_WAVE)
                    way = cut_from_short_list(a, rd, st, p, n, slot, row, do_scale, inv, n_list, sm);
                else if (n_list > 0 && n_list <= list_cap(more != nullptr))
                    way = n_list <= kT ? cut_from_list<1>(a, rd, st, p, n, slot, row, do_scale, inv, n_list, sm, more)
                          : n_list <= 4 * kT ? cut_from_list<4>(a, rd, st, p, n, slot, row, do_scale, inv, n_list, sm, more)
                                             : cut_from_list<SR_LIST_CAP_BIG / kT>(a, rd, st, p, n, slot, row, do_scale, inv, n_list, sm, more);
                if (SR_USUAL(way != kListGeneral)) {
                    FPROF(a, slot, 9);
                    __syncthreads();
                    if (tid == 0) {
                        const uint32_t f = flags | (sm.bc[SR_AMB_WORD] ? SR_KFLAG_AMBIGUOUS : 0u);
                        st->flags = f;
                        if ((way == kListDone || (way == kListClosed && a.mode == 2)) && a.out_flags) a.out_flags[row] = f;
                    }
                    return;
                }
            }
            if (e_row != p) {
                // (a row that goes on here has its probabilities take shape in the caller's row; one whose list was not made has
                // all but the last of e there)
                for (int i = tid + (row_is_listed(rd, a) && st_list_from == 0u ? n & ~3 : 0); i < n; i += kT) p[i] = e_row[i];
                sr_drain_stores();
                __syncthreads();
            }
            const bool fast_nucleus = row_fast_nucleus(rd, a);
            if (fast_nucleus) {
                uint32_t* hcnt = (uint32_t*)sm.sortbuf;
                __syncthreads();
                for (int i = tid; i < kHistPos; i += kT) hcnt[i] = 0u;
                if (tid == 0) sm.bc[5] = 0u;
                __syncthreads();
                row_pass<false>(p, n, [&](float x, int) -> float { hist_count(hcnt, &sm.bc[5], x); return x; });
                __syncthreads();
            }
            const int way = fast_nucleus ? nucleus_from_histogram(a, rd.top_p, p, n, slot, row, do_scale, inv, sm, more) : kNucleusGeneral;
            no_slabs = way == kNucleusGeneralNoSlabs;
            if (way == kNucleusDone) {
                FPROF(a, slot, 9);
                __syncthreads();
                if (tid == 0) {
                    st->n_survivors = 0;
                    st->flags = flags;
                    if (a.out_flags) a.out_flags[row] = flags | (sm.bc[SR_AMB_WORD] ? SR_KFLAG_AMBIGUOUS : 0u);
                }
                return;
            }
            if (!(rd.top_k > 0 && rd.top_k < n) && (rd.min_p > 0.0f || use_top_p)) {
                // No top-k stage in between: the scaling, the min-p cut (Sampler.cs:493-503) and the count of
                // survivors that top-p starts from share one pass.  The largest probability needs no search: the
                // largest e is expf(0) = 1, so it is 1 * (1 / sum).
                const float mp = do_scale ? __fmul_rn(1.0f, inv) : 1.0f;
                const bool use_min_p = rd.min_p > 0.0f;
                const float thr = use_min_p ? __fmul_rn(rd.min_p, mp) : 0.0f;
                int c = 0;
                // A min-p cut leaves few survivors: they are listed while the row is read, which saves the pass that
                // would collect them; a row that is only sampled from (no distribution out) and ends with at most
                // 4,096 survivors is finished from that list and need not be written at all.
                const bool list_now = use_min_p;
                if (list_now) {
                    if (tid == 0) sm.bc[4] = 0u;
                    __syncthreads();
                }
                auto body = [&](float x, int i) -> float {
                    float y = do_scale ? __fmul_rn(x, inv) : x;
                    if (use_min_p) SR_AMB_IF(sr_near(y, thr));  // an entry on the threshold
                    if (use_min_p && y < thr) y = 0.0f;
                    if (y > 0.0f) {
                        c++;
                        if (list_now) {
                            const uint32_t pos = atomicAdd(&sm.bc[4], 1u);
                            if (pos < (uint32_t)kSmall)
                                sm.sortbuf[pos] = ((unsigned long long)sr_f2u(y) << 32) | (unsigned long long)(0xffffffffu - (uint32_t)i);
                        }
                    }
                    return y;
                };
                const bool read_only = list_now && a.mode == 0 && n >= 8;
                if (read_only) {
                    row_pass<false>(p, n, body);
                } else {
                    row_pass<true>(p, n, body);
                }
                survivors = c;
                fused = true;
                if (list_now) {
                    const int ns_now = blk_sum_i(c, sm);
                    if (ns_now <= kSmall) ns_listed = ns_now;
                    row_unwritten = read_only && ns_now > 0 && ns_now <= kSmall;
                    if (read_only && !row_unwritten) {
                        // too many survivors to finish from the list: the scaled row is needed after all
                        row_pass<true>(p, n, [&](float x, int) -> float {
                            float y = do_scale ? __fmul_rn(x, inv) : x;
                            if (use_min_p && y < thr) y = 0.0f;
                            return y;
                        });
                    }
                }
            } else if (do_scale) {
                row_pass<true>(p, n, [&](float x, int) -> float { return __fmul_rn(x, inv); });
            }
            __syncthreads();
        }
        FPROF(a, slot, 3);
        // ApplyTopK + Normalize (Sampler.cs:71-81, :477-488): everything equal to the k-th value survives
        if (rd.top_k > 0 && rd.top_k < n) {
            const float kth = kth_largest(p, n, rd.top_k, sm);
            row_pass<true>(p, n, [&](float x, int) -> float { return x < kth ? 0.0f : x; });
            __syncthreads();
            normalize_row(p, n, sm);
        }
        FPROF(a, slot, 4);
        // ApplyMinP (Sampler.cs:493-503)
        if (rd.min_p > 0.0f && !fused) {
            float mp = 0.0f;
            row_pass<false>(p, n, [&](float x, int) -> float { mp = fmaxf(mp, x); return x; });
            bool nn;
            mp = blk_max_f(mp, &nn, sm);
            const float thr = __fmul_rn(rd.min_p, mp);
            row_pass<true>(p, n, [&](float x, int) -> float {
                SR_AMB_IF(x > 0.0f && sr_near(x, thr));
                return x < thr ? 0.0f : x;
            });
            __syncthreads();
        }
        FPROF(a, slot, 5);
        // ApplyTopP (Sampler.cs:516-551)
        int listed = -1;  // the row's survivors are sm.sortbuf[0, listed)
        if (use_top_p) {
            int cnt = survivors;
            if (!fused) row_pass<false>(p, n, [&](float x, int) -> float { cnt += x > 0.0f ? 1 : 0; return x; });
            int ns;
            ns = blk_sum_i(cnt, sm);
            const bool have_list = ns_listed >= 0;  // (then ns == ns_listed <= kSmall)
            // The nucleus is walked in descending order, a slab of at most kSmall probabilities at a time: the slab
            // is everything above the 65536-value bucket that holds the kSmall-th largest of what is left, it is
            // sorted here and the exact running sum goes on through it from where the slab before ended.  Most
            // nuclei close in the first slab; a masked row without min-p (tens of thousands of survivors) takes a
            // few.  Only a row that makes no progress (more than kSmall probabilities inside one bucket) or needs
            // more than kMaxSlabs slabs has all its survivors sorted (sort_survivors_in_place).
            constexpr int kMaxSlabs = 24;
            // A row that needs several slabs has all their bounds from one histogram of its probabilities' 16-bit keys
            // instead of two select passes per slab.  The histogram is counted in LDS (the slabs' sort buffer, free
            // until the first slab): position d = 0x3fff - key, so that positions ascend as the values fall; 8,192
            // positions reach down to 2^-63, what lies below shares the last one.  Its running sums go to the row's
            // segment of the sort buffers: sums[d] = survivors at positions <= d, and the position that holds the
            // kSmall-th largest of what is left is the first d with sums[d] >= taken + kSmall.
            constexpr int kPos = 8192;
            static_assert(kPos * 4 <= kSmall * 8 && kPos % kT == 0, "the histogram fits the sort buffer");
            constexpr int kPer = kPos / kT;
            uint32_t* sums = a.sort_keys_in + (size_t)slot * a.sort_stride;
            bool use_hist = !have_list && ns > kSmall && a.sort_stride >= kPos && !no_slabs;
            if (use_hist) {
                uint32_t* cnt = (uint32_t*)sm.sortbuf;
                for (int i = tid; i < kPos; i += kT) cnt[i] = 0u;
                if (tid == 0) sm.bc[5] = 0u;
                __syncthreads();
                row_pass<false>(p, n, [&](float v, int) -> float {
                    if (v > 0.0f) {
                        const uint32_t key = sr_f2u(v) >> 16;
                        if (key <= 0x3fffu) atomicAdd(&cnt[min(0x3fffu - key, (uint32_t)(kPos - 1))], 1u);
                        else sm.bc[5] = 1u;  // (no probability is 2 or more; if one is, the slabs take the other way)
                    }
                    return v;
                });
                __syncthreads();
                use_hist = sm.bc[5] == 0u;
                uint32_t mine[kPer];
                int own = 0;
#pragma unroll
                for (int q = 0; q < kPer; q++) { mine[q] = cnt[tid * kPer + q]; own += (int)mine[q]; }
                int tot;
                int upto = blk_excl_scan(own, &tot, sm);
#pragma unroll
                for (int q = 0; q < kPer; q++) { upto += (int)mine[q]; sums[tid * kPer + q] = (uint32_t)upto; }
                // The first slab need not be full: count x the position's smallest value bounds the mass of the
                // positions from below (in units of 2^-28), and the slab ends where that bound passes top-p (+ 0.1 %) --
                // a few hundred entries for a sharp row instead of 4,096 to gather and sort.
                uint32_t ownq = 0u, mq[kPer];
#pragma unroll
                for (int q = 0; q < kPer; q++) {
                    const int d = tid * kPer + q;
                    const float y_low = d < kPos - 1 ? sr_u2f((0x3fffu - (uint32_t)d) << 16) : 0.0f;
                    mq[q] = (uint32_t)fminf((float)mine[q] * y_low * 268435456.0f, 268435456.0f);
                    ownq += mq[q];
                }
                int totq;
                uint32_t uptoq = (uint32_t)blk_excl_scan((int)ownq, &totq, sm);
                if (tid == 0) sm.bc[7] = (uint32_t)kPos;
                __syncthreads();
                const uint32_t target_q = (uint32_t)(rd.top_p * 1.001f * 268435456.0f) + 64u;
                int d_first = kPos;
#pragma unroll
                for (int q = 0; q < kPer; q++) {
                    uptoq += mq[q];
                    if (uptoq >= target_q && d_first == kPos) d_first = tid * kPer + q;
                }
                if (d_first < kPos) atomicMin(&sm.bc[7], (uint32_t)d_first);
                sr_drain_stores();
                __syncthreads();
            }
            const uint32_t d_mass = use_hist ? sm.bc[7] : (uint32_t)kPos;
            FPROF(a, slot, 10);
            [[maybe_unused]] unsigned long long t_step = 0ull;
            FPROF_ADD(a, slot, 16, t_step);
            bool closed = false;
            float run = 0.0f;                  // exact running sum behind the slabs taken so far
            int taken = 0;                     // survivors in those slabs
            uint32_t hi_key = 0xffffffffu;     // what is left are the probabilities with keys <= hi_key
            float c_above = -1.0f;             // the current slab: probabilities strictly above this value ...
            for (int slab = 0; slab < kMaxSlabs && ns > 0 && !closed && !no_slabs; slab++) {
                const bool last_slab = ns - taken <= kSmall;  // everything that is left fits
                if (last_slab) {
                    c_above = 0.0f;
                } else if (use_hist) {
                    const uint32_t target = (uint32_t)(taken + kSmall);
                    // the one thread whose positions hold the first d with sums[d] >= target names it
                    const uint32_t last = sums[tid * kPer + kPer - 1], before = tid > 0 ? sums[tid * kPer - 1] : 0u;
                    if (last >= target && before < target) {
                        int d = tid * kPer + kPer - 1;
#pragma unroll
                        for (int q = kPer - 2; q >= 0; q--)
                            if (sums[tid * kPer + q] >= target) d = tid * kPer + q;
                        sm.bc[5] = (uint32_t)d;
                    }
                    __syncthreads();
                    uint32_t d = sm.bc[5];
                    __syncthreads();
                    if (slab == 0) d = min(d, d_mass + 1u);
                    if (d < (uint32_t)(kPos - 1)) {
                        c_above = sr_u2f(((0x3fffu - d) << 16) | 0xffffu);
                    } else {  // (the shared last position: its keys are not one bucket)
                        use_hist = false;
                        c_above = sr_u2f(sr_f2u(kth_largest(p, n, kSmall, sm, 16, hi_key)) | 0xffffu);
                    }
                } else {
                    c_above = sr_u2f(sr_f2u(kth_largest(p, n, kSmall, sm, 16, hi_key)) | 0xffffu);
                }
                FPROF_ADD(a, slot, 11, t_step);
                int nc;
                if (have_list) {
                    nc = ns;  // (ns <= kSmall: the survivors were listed while the row was scaled)
                } else {
                    if (tid == 0) sm.bc[4] = 0u;
                    __syncthreads();
                    row_pass<false>(p, n, [&](float v, int i) -> float {
                        if (v > c_above && sr_f2u(v) <= hi_key) {
                            const uint32_t pos = atomicAdd(&sm.bc[4], 1u);
                            if (pos < (uint32_t)kSmall)
                                sm.sortbuf[pos] = ((unsigned long long)sr_f2u(v) << 32) | (unsigned long long)(0xffffffffu - (uint32_t)i);
                        }
                        return v;
                    });
                    __syncthreads();
                    nc = (int)sm.bc[4];
                    __syncthreads();
                }
                FPROF_ADD(a, slot, 12, t_step);
                if (nc <= 0 || nc > kSmall) break;  // no progress: the row's survivors are sorted as a whole
                int P = 2;
                while (P < nc) P <<= 1;
                for (int i = nc + tid; i < P; i += kT) sm.sortbuf[i] = 0ull;
                __syncthreads();
                sort_small_desc(sm, P);
                FPROF_ADD(a, slot, 13, t_step);
                for (int i = tid; i < nc; i += kT) sm.sprob[i] = sr_u2f((uint32_t)(sm.sortbuf[i] >> 32));
                __syncthreads();
                int found;
                if (nc <= SR_WAVE) {
                    // a handful of survivors (a row that min-p has cut): one thread adds them the way the scalar loop does
                    if (tid == 0) {
                        float s = run;
                        int f = -1;
                        for (int i = 0; i < nc && f < 0; i++) {
                            s = __fadd_rn(s, sm.sprob[i]);
                            if (s >= rd.top_p) f = i;
                        }
                        sm.segbc[1] = (uint32_t)f;
                        sm.segbc[2] = sr_f2u(s);
                    }
                    __syncthreads();
                    found = (int)sm.segbc[1];
                    run = sr_u2f(sm.segbc[2]);
                    __syncthreads();  // (the words may be written again for the next slab)
                } else {
                    run = seq_sum<true>([&](int i) -> float { return sm.sprob[i]; }, nc, run, rd.top_p, &found, sm);
                }
                if (found >= 0)
                    SR_AMB_IF(sr_stop_near(run, sm.sprob[found], rd.top_p) || (found + 1 < nc && sm.sprob[found + 1] == sm.sprob[found]));
                else if (taken + nc == ns)
                    SR_AMB_IF(sr_near(run, rd.top_p));
                FPROF_ADD(a, slot, 14, t_step);
                if (a.prof && slot == 0 && tid == 0) a.prof[15] += 1ull;
                taken += nc;
                closed = found >= 0 || taken == ns;
                if (closed) {
                    const int cutoff = found >= 0 ? found + 1 : nc;
                    if (!row_unwritten)
                        for (int i = cutoff + tid; i < nc; i += kT)
                            p[0xffffffffu - (uint32_t)(sm.sortbuf[i] & 0xffffffffull)] = 0.0f;
                    __syncthreads();
                    if (taken < ns) {  // everything that was in no slab comes later in the order
                        row_pass<true>(p, n, [&](float x, int) -> float { return x > c_above ? x : 0.0f; });
                        __syncthreads();
                    }
                    if (slab == 0) listed = cutoff;  // the members are all at hand
                } else {
                    hi_key = sr_f2u(c_above);
                }
            }
            if (ns > 0 && !closed) {
                // the nucleus reaches past what the walk by slabs takes: the survivors go to the row's sort segment and
                // are sorted there
                uint32_t* keys = a.sort_keys_in + (size_t)slot * a.sort_stride;
                int32_t* ids = a.sort_vals_in + (size_t)slot * a.sort_stride;
                const bool aligned = ((uintptr_t)p & 15u) == 0u;
                int base = 0;
                for (int i0 = 0; i0 < n; i0 += 4 * kT) {
                    const int i = i0 + 4 * tid;
                    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                    if (aligned && i + 4 <= n) {
                        const float4 t = *(const float4*)(p + i);
                        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
                    } else {
#pragma unroll
                        for (int q = 0; q < 4; q++)
                            if (i + q < n) v[q] = p[i + q];
                    }
                    const int mine = (v[0] > 0.0f ? 1 : 0) + (v[1] > 0.0f ? 1 : 0) + (v[2] > 0.0f ? 1 : 0) + (v[3] > 0.0f ? 1 : 0);
                    int tot;
                    int pos = base + blk_excl_scan(mine, &tot, sm);
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        if (v[q] > 0.0f) { keys[pos] = sr_f2u(v[q]); ids[pos] = i + q; pos++; }
                    base += tot;
                }
                sr_drain_stores();
                sort_survivors_in_place(keys, ids, ns, sm);
                // the nucleus over the sorted survivors (descending probability, ascending index among equal ones)
                int found;
                const float at = seq_sum<true>([&](int i) -> float { return sr_u2f(keys[i]); }, ns, 0.0f, rd.top_p, &found, sm);
                if (tid == 0)
                    SR_AMB_IF(found >= 0 ? (sr_stop_near(at, sr_u2f(keys[found]), rd.top_p) || (found + 1 < ns && keys[found + 1] == keys[found]))
                                         : sr_near(at, rd.top_p));
                const int cutoff = found >= 0 ? found + 1 : ns;
                for (int i = cutoff + tid; i < ns; i += kT) p[ids[i]] = 0.0f;
                __syncthreads();
            }
            if (tid == 0) st->n_survivors = ns;
        } else if (ns_listed > 0 && ns_listed <= kSmall && n >= 8) {
            listed = ns_listed;  // min-p alone: its survivors are the members
        }
        FPROF(a, slot, 6);
        const bool finish_here = listed > 0 && listed <= kSmall && n >= 8;
        if (tid == 0) {
            st->flags = flags;
        }
        if (finish_here) {
            // the nucleus closed inside the kernel and its members are at hand: no pass over the row is needed
            finish_from_list(a, p, n, listed, row, sm);
            FPROF(a, slot, 9);
            __syncthreads();
            if (tid == 0 && a.out_flags) a.out_flags[row] = flags | (sm.bc[SR_AMB_WORD] ? SR_KFLAG_AMBIGUOUS : 0u);
            return;
        }
        __syncthreads();
    }
    FPROF(a, slot, 7);
    // final Normalize (Sampler.cs:91-92)
    normalize_row(p, n, sm);
    FPROF(a, slot, 8);
    int token = -1;
    if (a.mode != 1) {
        token = draw_from_row(p, n, sm.u, sm);
        if (tid == 0 && a.out_tokens) a.out_tokens[row] = token;
    }
    FPROF(a, slot, 9);
    __syncthreads();
    if (tid == 0 && a.out_flags) a.out_flags[row] = st->flags | (sm.bc[SR_AMB_WORD] ? SR_KFLAG_AMBIGUOUS : 0u);
}

// ---- rows left to the whole device: final Normalize and draw (Sampler.cs:91-92, :553-576) --------------------------------
// The members' probabilities y = fl(e inv) are known by the cut (all of them, in a row that nothing cuts).  One launch
// (k_prepared_row), a workgroup per block of 8,192 entries, which it reads once:
//   its waves, one per lane accumulator of TensorPrimitives.Sum, make the records of their 1,024 terms of the block;
//   whoever of the row's workgroups is there last walks the eight accumulators, and the others wait for the factor;
//   then every wave takes a segment: z = fl(y / sum), written where the distribution is handed out, and the segment's record
//   for the running sum of the draw;
//   whoever comes last walks those records to the draw's target.
// What bounds it: the serial chain (data, records, meeting, walk of the accumulators, records, walk of the draw), about a
// third of it trips to memory.  32 ragged bf16 rows of 100,003: 23 us, 16 rows of 262,144 fp32: 33; as three launches --
// each 4 us before its first byte, and the row read twice -- the same steps took 27 and 38.
// The wait is bounded: a workgroup whose wait runs out marks the row (SrFullState::late_behind), counts itself in as if it had done
// its block, and whoever comes last does all blocks of the row again.
template <bool kLogits>
struct PreparedRow {
    ERow row;  // (kLogits: of the verifier, whose e may not be there)
    float inv, ycut;
    int idx_last, n;
    __device__ __forceinline__ float cut(float ev, int i) const  // y, or 0 outside the nucleus
    {
        const float y = __fmul_rn(ev, inv);
        return (y > ycut) | ((y == ycut) & (i <= idx_last)) ? y : 0.0f;  // (no branch per entry)
    }
};
template <bool kLogits>
__device__ __forceinline__ PreparedRow<kLogits> prepared_row(const SrFullArgs& a, const SrFullState* st, int slot, const uint64_t* tab, float inv_temp)
{
    PreparedRow<kLogits> r;
    r.row.e = row_e(a, slot);
    if (kLogits) {
        r.row.lg = st->e_open == a.seq ? (const float*)a.logits + (size_t)slot * (size_t)a.row_stride : nullptr;  // (the verifier's slots are its rows)
        r.row.inv_temp = inv_temp;
        r.row.max = sr_okey_inv((uint32_t)st->maxkey);
        r.row.tab = tab;
    }
    r.inv = st->mul1;
    r.ycut = st->ycut;
    r.idx_last = st->idx_last;
    r.n = a.vocab;
    return r;
}
constexpr int kPrepT = 512;
static_assert(kPrepT / SR_WAVE == SR_SEQ_CHAINS, "a wave per chain, and one per segment");
constexpr int kPrepBlock = SR_SEQ_CHAINS * SR_SEG_TERMS;
// y of the wave's segment of block blk, as it is loaded: lane l the pieces l, 64 + l, ... of four entries
template <bool kLogits>
__device__ __forceinline__ void prepared_load(const PreparedRow<kLogits>& r, int blk, int wave, int lane, float4 (&v)[4], float4* ev = nullptr)
{
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i0 = blk * kPrepBlock + wave * SR_SEG_TERMS + (k * SR_WAVE + lane) * 4;
        v[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (i0 + 4 <= r.n) {
            // (the rows of e start on 16-byte boundaries; what is loaded from the logits becomes e behind all loads)
            v[k] = kLogits && r.row.lg ? sr_load_f4(r.row.lg + i0) : *(const float4*)(r.row.e + i0);
        } else if (i0 < r.n) {
            const float* const from = kLogits && r.row.lg ? r.row.lg : r.row.e;
            v[k].x = from[i0];
            if (i0 + 1 < r.n) v[k].y = from[i0 + 1];
            if (i0 + 2 < r.n) v[k].z = from[i0 + 2];
        }
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i0 = blk * kPrepBlock + wave * SR_SEG_TERMS + (k * SR_WAVE + lane) * 4;
        if (kLogits && r.row.lg) {
            v[k].x = i0 < r.n ? r.row.of(v[k].x) : 0.0f; v[k].y = i0 + 1 < r.n ? r.row.of(v[k].y) : 0.0f;
            v[k].z = i0 + 2 < r.n ? r.row.of(v[k].z) : 0.0f; v[k].w = i0 + 3 < r.n ? r.row.of(v[k].w) : 0.0f;
            ev[k] = v[k];
        }
        v[k].x = r.cut(v[k].x, i0); v[k].y = r.cut(v[k].y, i0 + 1); v[k].z = r.cut(v[k].z, i0 + 2); v[k].w = r.cut(v[k].w, i0 + 3);
    }
}
// z of the wave's segment: to the caller's row where the distribution is handed out, and the segment's record for the draw
template <bool kLogits>
__device__ __forceinline__ void prepared_segment(const SrFullArgs& a, const PreparedRow<kLogits>& r, int slot, int row, int seg, int lane, float4 (&v)[4],
                                                 float before, float inv2, float4* turn, bool drawn)
{
    const int n = r.n;
    float* const p = a.work + (size_t)(a.work_by_row ? row : slot) * a.work_stride;
    if (drawn && r.ycut < 0.0f) {
        // the uncut row's token is its largest entry, e = 1, the only one whose fl(e m1) is m1
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i0 = seg * SR_SEG_TERMS + (k * SR_WAVE + lane) * 4;
            const int at = v[k].x == r.inv ? i0 : v[k].y == r.inv ? i0 + 1 : v[k].z == r.inv ? i0 + 2 : v[k].w == r.inv ? i0 + 3 : -1;
            if (at >= 0) {
                if (a.out_tokens) a.out_tokens[row] = at;
                if (a.out_flags) a.out_flags[row] = a.state[slot].flags;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i0 = seg * SR_SEG_TERMS + (k * SR_WAVE + lane) * 4;
        v[k].x = __fmul_rn(v[k].x, inv2); v[k].y = __fmul_rn(v[k].y, inv2); v[k].z = __fmul_rn(v[k].z, inv2); v[k].w = __fmul_rn(v[k].w, inv2);
        if (a.mode != 0) {
            if (i0 + 4 <= n) {
                sr_store_f4(p + i0, v[k].x, v[k].y, v[k].z, v[k].w);
            } else if (i0 < n) {
                p[i0] = v[k].x;
                if (i0 + 1 < n) p[i0 + 1] = v[k].y;
                if (i0 + 2 < n) p[i0 + 2] = v[k].z;
            }
        }
    }
    if (a.mode == 1 || drawn) return;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i = (k * SR_WAVE + lane) * 4;
        turn[(i >> 4) * 5 + ((i & 15) >> 2)] = v[k];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float t[SR_SEQ_RUN];
    float own = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const float4 q = turn[lane * 5 + k];
        t[4 * k] = q.x; t[4 * k + 1] = q.y; t[4 * k + 2] = q.z; t[4 * k + 3] = q.w;
        own += (q.x + q.y) + (q.z + q.w);
    }
    own = sr_wave_sum_f32(own);
    // (the records of the denominator have been walked: theirs take their place)
    seg_make_record<true>(t, seg, (double)(before * r.inv * inv2), a.seg_func + (size_t)slot * a.seg_stride + seg, own);
}
// kPhase 0: all of it.  1 and 2: up to the factor, and from there on, as two launches of which neither waits, for launches of several
// times the workgroups that the device holds (behind_twice): there the ones that wait keep others out, most of all where a
// row's workgroups do not all fit behind the rows in front of it.
// 3: as 1, for rows whose shares of the accumulators nobody has added up (k_spec_factor): the workgroups meet over them (bounded; what
// stands in front of a block's terms only has to be about right, so a wait that runs out takes an eighth of the segments' sums).
struct PreparedSmem {
    float4 room[SR_SEQ_CHAINS * SR_WAVE * 5];  // the block chain by chain, then every wave's segment on its way to 16 terms a lane
    float lane_sum[SR_SEQ_CHAINS];
    // 0: whether the workgroup is the row's last   1: the factor   2: whether the wait for it ended in time (a word of its own: the
    // waiting thread writes it while others may still have to read the first)
    uint32_t bc[3];
};
template <int kPhase>
__device__ __forceinline__ void prepared_block(const SrFullArgs& a, int slot, PreparedSmem& sm, const uint64_t* tab = nullptr, float inv_temp = 1.0f)
{
    float4* const room = sm.room;
    float* const lane_sum = sm.lane_sum;
    uint32_t* const bc = sm.bc;
    const int blk = blockIdx.x, tid = threadIdx.x, lane = sr_lane(), wave = sr_wave_id();
    SrFullState* st = a.state + slot;
    const int row = kPhase == 3 ? slot : a.row_list[slot];
    const PreparedRow<kPhase == 3> r = prepared_row<kPhase == 3>(a, st, slot, tab, inv_temp);
    const int n = r.n, nv = n / 8, rem = n - nv * 8, body = nv * 8, nblk = (nv + SR_SEG_TERMS - 1) / SR_SEG_TERMS, nseg = seg_count(n);
    unsigned long long* const sync = a.row_sync + (size_t)slot * SR_ROW_SYNC_STRIDE + 1;
    const float* const sums = a.seg_sum + (size_t)slot * a.seg_stride;
    SeqSegFunc* const chain = a.chain_func + ((size_t)slot * SR_SEQ_CHAINS + wave) * a.chain_blocks;
    const int seg = blk * SR_SEQ_CHAINS + wave;
    float4 v[4];
    float4 ev[4];  // (phase 3)
    const bool drawn = kPhase != 3 && st->drawn == a.seq, closed = drawn && !(r.ycut < 0.0f);
    if (closed && kPhase == 1) return;
    prepared_load(r, blk, wave, lane, v, ev);
    if (closed) {
        if (seg < nseg) prepared_segment(a, r, slot, row, seg, lane, v, 0.0f, st->mul2, room, true);
        return;
    }
    // about what stands in front of the block's terms of the wave's chain, and of the wave's segment
    const float* const cs = a.chain_sum + (size_t)slot * a.chain_stride;
    float before = 0.0f, before_seg = 0.0f, own = 0.0f;
    const int hb1 = a.chain_stride / SR_SEQ_CHAINS;
    if (kPhase != 3) {
        for (int hb = lane; hb < 2 * blk; hb += SR_WAVE) before += cs[hb * SR_SEQ_CHAINS + wave];
        if (2 * blk < hb1) own = cs[2 * blk * SR_SEQ_CHAINS + wave];
        if (2 * blk + 1 < hb1) own += cs[(2 * blk + 1) * SR_SEQ_CHAINS + wave];
    }
    if (kPhase != 1 && kPhase != 3 && !a.lazy_scale && a.mode != 1 && !drawn && seg < nseg)
        for (int g = lane; g < seg; g += SR_WAVE) before_seg += sums[g];
    float x[SR_SEQ_RUN];
    if (kPhase != 2 && blk < nblk) {
        // chain by chain in shared memory: the place of term 16 l + j of chain g is g 1024 + 64 j + (l + 2 j) mod 64, so that
        // the lanes of a wave read a term from 64 consecutive places and a piece's stores fall two to a bank
        float* const buf = (float*)room;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int t4 = wave * (SR_SEG_TERMS / 4) + k * SR_WAVE + lane;  // the piece's number within the block
            const int vec = t4 >> 1, j = vec & 15, l = vec >> 4;
            const bool in = blk * kPrepBlock + 4 * t4 < body;  // (body is a multiple of 8)
            float* at = buf + (4 * (t4 & 1)) * 1024 + 64 * j + ((l + 2 * j) & 63);
            at[0] = in ? v[k].x : 0.0f; at[1024] = in ? v[k].y : 0.0f; at[2048] = in ? v[k].z : 0.0f; at[3072] = in ? v[k].w : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = buf[wave * 1024 + 64 * j + ((lane + 2 * j) & 63)];
    }
    if (kPhase == 3) {
        if (blk < nblk) {
#pragma unroll
            for (int j = 0; j < SR_SEQ_RUN; j++) own += x[j];
            own = sr_wave_sum_f32(own);
            if (lane == 0) sr_store_agent(&a.chain_sum[(size_t)slot * a.chain_stride + (size_t)blk * SR_SEQ_CHAINS + wave], own);
        }
        sr_drain_stores();
        __syncthreads();
        if (tid == 0) {
            const unsigned long long was = __hip_atomic_fetch_add(sync, 1ull << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint32_t ok = ((uint32_t)(was >> 16) & 0xffffu) + 1u == gridDim.x ? 1u : 0u;
            for (uint32_t it = 0; ok == 0u && it < a.behind_wait_limit; it++) {
                ok = ((uint32_t)(sr_load_agent(sync) >> 16) & 0xffffu) == gridDim.x ? 1u : 0u;
                if (ok == 0u) __builtin_amdgcn_s_sleep(1);
            }
            bc[0] = ok;
        }
        __syncthreads();
        if (blk < nblk) {
            if (bc[0] != 0u) {
                for (int b = lane; b < blk; b += SR_WAVE) before += sr_load_agent(&cs[b * SR_SEQ_CHAINS + wave]);
            } else {
                for (int g = lane; g < blk * SR_SEQ_CHAINS; g += SR_WAVE) before += sums[g] * (r.inv / SR_SEQ_CHAINS);
            }
        }
    }
    if (kPhase == 3 && r.row.lg) {
        // (behind the meeting: a barrier waits for what is on its way to memory, and this is only needed by whoever counts in last.
        // The rows of e are whole pieces long)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i0 = blk * kPrepBlock + wave * SR_SEG_TERMS + (k * SR_WAVE + lane) * 4;
            if (i0 < n) sr_store_agent_f4((float4*)(const_cast<float*>(r.row.e) + i0), ev[k].x, ev[k].y, ev[k].z, ev[k].w);
        }
    }
    if (kPhase != 2 && blk < nblk) {
        const float by = kPhase == 3 ? 1.0f : r.inv;  // (what phase 3 has added up is normalised already)
        before = sr_wave_sum_f32(before) * by;
        seg_make_record<true, kPhase != 3>(x, blk, (double)before, chain + blk, own * by);  // (k_full_row's own sums)
    }
    bool last_in = false;
    if (kPhase != 2) {
        sr_drain_stores();
        __syncthreads();  // (the workgroup's records are out, and nobody reads the block any more)
        if (tid == 0) {
            const unsigned long long was = __hip_atomic_fetch_add(sync, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            bc[0] = ((uint32_t)was & 0xffffu) + 1u == gridDim.x ? 1u : 0u;
        }
        __syncthreads();
        last_in = bc[0] != 0u;
        if ((kPhase == 1 || kPhase == 3 || a.lazy_scale) && !last_in) return;  // (the last one has all there is to do)
    }
    // the eight accumulators, a wave each: the sum of the members, and 1 over it
    auto normaliser = [&]() __attribute__((always_inline)) -> float {
        int dummy;
        float s = seg_walk_from<false, true>([&](int b, float (&x)[SR_SEQ_RUN]) __attribute__((always_inline)) {
            // (no condition stands between the loads: with one each they wait for each other; a whole block by offsets from one
            // address)
            const int t0 = b * SR_SEG_TERMS + lane * SR_SEQ_RUN;
            const float* const e0 = r.row.e + (size_t)t0 * 8 + wave;
            if ((b + 1) * SR_SEG_TERMS <= nv) {
#pragma unroll
                for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = e0[j * 8];
            } else {
#pragma unroll
                for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = e0[(min(t0 + j, nv - 1) - t0) * 8];
            }
#pragma unroll
            for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = t0 + j < nv ? r.cut(x[j], (t0 + j) * 8 + wave) : 0.0f;
        }, nblk, chain, 0.0f, 0.0f, &dummy, nullptr);
        if (rem > 0 && wave >= 8 - rem) s = __fadd_rn(s, r.cut(r.row.e[n - 8 + wave], n - 8 + wave));  // the overlapped last vector
        if (lane == 0) lane_sum[wave] = s;
        __syncthreads();
        const float l0 = lane_sum[0], l1 = lane_sum[1], l2 = lane_sum[2], l3 = lane_sum[3], l4 = lane_sum[4], l5 = lane_sum[5],
                    l6 = lane_sum[6], l7 = lane_sum[7];
        const float sum = __fadd_rn(__fadd_rn(__fadd_rn(l0, l1), __fadd_rn(l2, l3)), __fadd_rn(__fadd_rn(l4, l5), __fadd_rn(l6, l7)));
        return (sum > 0.0f && sum != 1.0f) ? __fdiv_rn(1.0f, sum) : 1.0f;
    };
    // (phase 3: the row's workgroups, on other dies too, wrote e just now, through to memory.  No cache holds one of these lines from
    // before it was written: rows and blocks start on lines of their own, and nothing in the launch loads e of a position that it has
    // still to write -- spec_e<true>.  Read past the caches by agent-scope loads the blocks that no record fits cost 1.5 us of 127 at 16
    // rows of 262,144 and 8 drafts, 3 of 109 at 64 of 65,536 and 6: eight waves take 4 bytes of every 32 each)
    // Whoever counts in last walks them, and the others wait for the factor.  (All workgroups of the row walking for themselves, the
    // same work: 512 of them, at 16 rows of 262,144, fetched 12 MB of records past the caches and took 2.6 - 8 us for it.)
    unsigned long long* const factor = sync + 2;  // launch number << 32 | the factor's bits
    float inv2 = 1.0f;
    bool here = true;
    if (kPhase == 2) {
        inv2 = st->mul2;
    } else if (last_in) {
        inv2 = normaliser();
        if (tid == 0) {
            st->mul2 = inv2;
            if (kPhase == 3) st->e_open = 0u;
            sr_store_agent(factor, ((unsigned long long)a.seq << 32) | (unsigned long long)sr_f2u(inv2));
        }
        if (kPhase == 1 || kPhase == 3 || a.lazy_scale) return;
    } else {
        if (tid == 0) {
            uint32_t ok = 0u;
            unsigned long long v = 0ull;
            for (uint32_t it = 0; it < a.behind_wait_limit; it++) {
                v = sr_load_agent(factor);
                if ((uint32_t)(v >> 32) == a.seq) { ok = 1u; break; }
                __builtin_amdgcn_s_sleep(1);
            }
            if (ok == 0u) sr_store_agent(&st->late_behind, a.seq);
            bc[2] = ok;
            bc[1] = (uint32_t)v;
        }
        __syncthreads();
        here = bc[2] != 0u;
        inv2 = sr_u2f(bc[1]);
    }
    if (here && seg < nseg) prepared_segment(a, r, slot, row, seg, lane, v, sr_wave_sum_f32(before_seg), inv2, room + wave * SR_WAVE * 5, drawn);
    sr_drain_stores();
    __syncthreads();
    if (tid == 0) {
        const unsigned long long was = __hip_atomic_fetch_add(sync, 1ull << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        bc[0] = ((uint32_t)(was >> 16) & 0xffffu) + 1u == gridDim.x ? (sr_load_agent(&st->late_behind) == a.seq ? 2u : 1u) : 0u;
        if (bc[0] == 2u) bc[1] = (uint32_t)sr_load_agent(factor);
    }
    __syncthreads();
    if (bc[0] == 0u) return;
    if (SR_RARE(bc[0] == 2u)) {
        // some workgroup stopped waiting: all of the row again (everyone has counted in: the factor is there)
        inv2 = sr_u2f(bc[1]);
        for (int b = 0; b < (int)gridDim.x; b++) {
            const int sg = b * SR_SEQ_CHAINS + wave;
            if (sg >= nseg) break;
            prepared_load(r, b, wave, lane, v);
            float front = 0.0f;
            for (int g = lane; g < sg; g += SR_WAVE) front += sums[g];
            prepared_segment(a, r, slot, row, sg, lane, v, sr_wave_sum_f32(front), inv2, room + wave * SR_WAVE * 5, drawn);
        }
        sr_drain_stores();
        __syncthreads();
    }
    if (a.mode == 1 || drawn || wave != 0) return;
    const float u = st->u;
    int found;
    const float at = seg_walk_from<true, true>([&](int sg, float (&x)[SR_SEQ_RUN]) __attribute__((always_inline)) {
        const int i0 = sg * SR_SEG_TERMS + lane * SR_SEQ_RUN;
        seq_load_run(r.row.e, true, i0, n, x);  // (zeros past the end stay zeros)
#pragma unroll
        for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = __fmul_rn(r.cut(x[j], i0 + j), inv2);
    }, nseg, a.seg_func + (size_t)slot * a.seg_stride, 0.0f, u, &found, nullptr);
    if (lane == 0) {
        const bool amb = found >= 0 ? sr_stop_near(at, __fmul_rn(r.cut(r.row.e[found], found), inv2), u) : sr_near(at, u);
        if (a.out_tokens) a.out_tokens[row] = found >= 0 ? found : n - 1;
        if (a.out_flags) a.out_flags[row] = st->flags | (amb ? SR_KFLAG_AMBIGUOUS : 0u);
    }
}

template <int kPhase>
__global__ __launch_bounds__(kPrepT, 4) void k_prepared_row(SrFullArgs a)
{
    __shared__ PreparedSmem sm;
    const int slot = blockIdx.y;
    if (a.state[slot].deferred != a.seq) return;
    prepared_block<kPhase>(a, slot, sm);
}

// ---- SampleTopK (Sampler.cs:216-357) for rows wider than the selection kernel takes -----------------------
// The reference keeps the k + history-length largest raw logits (earlier index first among equals), applies the
// history penalties to those, orders them again (stable), and samples among the first k.  Here the whole row is
// sorted device-wide by (raw logit descending, index ascending), the first `sel` entries are adjusted and sorted
// again, and one workgroup per row walks the result.
// the reference's selection size: k + history length when the row has history penalties (Sampler.cs:224-225)
__device__ __forceinline__ int wide_sel(const SrRow& rd, int vocab)
{
    const long long s = (long long)rd.top_k + ((rd.flags & SR_ROWFLAG_HAS_PENALTY) ? (long long)rd.n_prev : 0ll);
    return (int)(s < (long long)vocab ? s : (long long)vocab);
}
template <int ES>
__global__ __launch_bounds__(256) void k_wide_keys(SrFullArgs a)
{
    const int slot = blockIdx.y;
    const int row = a.row_list[slot];
    const SrRow rd = a.rows[row];
    const char* rowp = (const char*)a.logits + (size_t)row * (size_t)a.row_stride * ES;
    const uint32_t* mrow = (rd.mask_row >= 0) ? a.mask + (size_t)rd.mask_row * a.mask_stride : nullptr;
    uint32_t* keys = a.sort_keys_in + (size_t)slot * a.sort_stride;
    int32_t* ids = a.sort_vals_in + (size_t)slot * a.sort_stride;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < a.vocab; i += gridDim.x * 256) {
        float x = load_logit<ES>(rowp, i);
        if (mrow && !((mrow[i >> 5] >> (i & 31)) & 1u)) x = SR_NEG_INF;
        keys[i] = sr_okey(x);
        ids[i] = i;
    }
}

// the first `sel` sorted entries with the history penalties of SampleTopK applied (Sampler.cs:262-297); entries
// that hold -inf are the reference's unfilled slots (index -1)
__global__ __launch_bounds__(256) void k_wide_adjust(SrFullArgs a)
{
    const int slot = blockIdx.y;
    const int row = a.row_list[slot];
    const SrRow rd = a.rows[row];
    // In place: entry t of the sorted row becomes (adjusted key, t) -- the place in the first order is what the second
    // sort breaks ties by, which makes it the stable sort that the reference's insertion is (Sampler.cs:289-294) --
    // and its token id goes to wide_ids[t].
    uint32_t* keys = a.sort_keys_in + (size_t)slot * a.sort_stride;
    int32_t* ids = a.sort_vals_in + (size_t)slot * a.sort_stride;
    const uint32_t* skeys = keys;
    const int32_t* sids = ids;
    int32_t* tok = a.wide_ids + (size_t)slot * a.sort_stride;
    const int sel = wide_sel(rd, a.vocab);
    const bool pen = (rd.flags & SR_ROWFLAG_HAS_PENALTY) != 0u && rd.edit_cnt > 0;
    const SrEdit* ed = a.edits + rd.edit_off;
    for (int t = blockIdx.x * 256 + threadIdx.x; t < sel; t += gridDim.x * 256) {
        float v = sr_okey_inv(skeys[t]);
        int id = sids[t];
        if (sr_f2u(v) == 0xff800000u) {
            id = -1;
        } else if (pen) {
            int lo = 0;
            if (rd.flags & SR_ROWFLAG_EDITS_SORTED) {
                int hi = rd.edit_cnt;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (ed[mid].id < id) lo = mid + 1; else hi = mid;
                }
            } else {
                // (a row that was meant for the selection kernel and is redone here: its few edits are unsorted)
                while (lo < rd.edit_cnt && ed[lo].id != id) lo++;
            }
            if (lo < rd.edit_cnt && ed[lo].id == id && ed[lo].occ_all > 0) {
                const SrEdit ee = ed[lo];
                if (rd.rep != 1.0f && ee.occ_win > 0) v = v > 0.0f ? __fdiv_rn(v, ee.pen) : __fmul_rn(v, ee.pen);
                v = __fsub_rn(v, __fadd_rn(rd.presence, __fmul_rn(rd.frequency, (float)ee.occ_all)));
            }
        }
        keys[t] = sr_okey(v);
        ids[t] = t;
        tok[t] = id;
    }
}

// One row's (key, id) pairs sorted where they lie by the row's workgroup: descending key, ascending id among equal
// keys.  first != 0: the whole row (ids = token indices: the order the reference's selection keeps, Sampler.cs:232-247);
// else its first `sel` entries after the penalties (ids = places in the first order).
__global__ __launch_bounds__(kT) void k_wide_sort(SrFullArgs a, int first)
{
    __shared__ FullSmem sm;
    const int slot = blockIdx.x;
    const SrRow rd = a.rows[a.row_list[slot]];
    sort_survivors_in_place(a.sort_keys_in + (size_t)slot * a.sort_stride, a.sort_vals_in + (size_t)slot * a.sort_stride,
                            first ? a.vocab : wide_sel(rd, a.vocab), sm);
}

// temperature softmax over the first k entries, min-p, top-p and the draw, all left to right (Sampler.cs:299-356)
__global__ __launch_bounds__(kT) void k_wide_tail(SrFullArgs a)
{
    __shared__ FullSmem sm;
    const int tid = threadIdx.x;
    const int slot = blockIdx.x;
    const int row = a.row_list[slot];
    const SrRow rd = a.rows[row];
    const uint32_t* keys = a.sort_keys_in + (size_t)slot * a.sort_stride;
    const int32_t* pos = a.sort_vals_in + (size_t)slot * a.sort_stride;   // an entry's place in the first order ...
    const int32_t* tok = a.wide_ids + (size_t)slot * a.sort_stride;       // ... names its token id
    float* probs = a.work + (size_t)slot * a.work_stride;
    const int k = min(rd.top_k, wide_sel(rd, a.vocab));
    const float v0 = sr_okey_inv(keys[0]);
    const int id0 = tok[pos[0]];
    if (id0 < 0 || sr_f2u(v0) == 0xff800000u) {
        // nothing above -inf (Sampler.cs:254-255): Greedy over a row of -inf returns index 0
        if (tid == 0) {
            a.out_tokens[row] = 0;
            if (a.out_flags) a.out_flags[row] = SR_KFLAG_TOPK | SR_KFLAG_DEGENERATE;
        }
        return;
    }
    const float inv_temp = rd.temperature == 1.0f ? 1.0f : __fdiv_rn(1.0f, rd.temperature);
    const float mx = __fmul_rn(v0, inv_temp);
    for (int t = tid; t < k; t += kT) {
        const float v = sr_okey_inv(keys[t]);
        probs[t] = sr_f2u(v) == 0xff800000u ? 0.0f : sr_expf(__fsub_rn(__fmul_rn(v, inv_temp), mx));
    }
    __syncthreads();
    int found;
    const float sum = seq_sum_row<false>(probs, k, 0.0f, 0.0f, &found, sm);
    const float inv_sum = sum > 0.0f ? __fdiv_rn(1.0f, sum) : 0.0f;
    __syncthreads();
    row_pass<true>(probs, k, [&](float x, int) -> float { return __fmul_rn(x, inv_sum); });
    __syncthreads();
    int count = k;
    bool amb = false;  // SR_OUT_AMBIGUOUS: a cut or the draw lies on its boundary
    if (rd.min_p > 0.0f) {
        const float thr = __fmul_rn(rd.min_p, probs[0]);
        unsigned long long first = 0ull;  // ~index of the first entry below the threshold
        row_pass<false>(probs, k, [&](float x, int i) -> float {
            if (x < thr) {
                const unsigned long long e = 0xffffffffull - (unsigned long long)(uint32_t)i;
                first = e > first ? e : first;
            }
            return x;
        });
        first = blk_max_u64(first, sm);
        if (first) count = (int)(0xffffffffull - first);
        amb = (count > 0 && sr_near(probs[count - 1], thr)) || (count < k && sr_near(probs[count], thr));
    }
    if (rd.top_p < 1.0f && rd.top_p > 0.0f) {
        const float at = seq_sum_row<true>(probs, count, 0.0f, rd.top_p, &found, sm);
        amb = amb || (found >= 0 ? sr_stop_near(at, probs[found], rd.top_p) : sr_near(at, rd.top_p));
        if (found >= 0) count = found + 1;
    }
    const float kept = seq_sum_row<false>(probs, count, 0.0f, 0.0f, &found, sm);
    const float r = __fmul_rn(__double2float_rn(a.uniforms[(size_t)row * a.uniforms_per_row]), kept);
    const float at = seq_sum_row<true>(probs, count, 0.0f, r, &found, sm);
    amb = amb || (found >= 0 ? sr_stop_near(at, probs[found], r) : sr_near(at, r));
    if (tid == 0) {
        int token = id0;
        if (found >= 0 && tok[pos[found]] >= 0) token = tok[pos[found]];
        a.out_tokens[row] = token;
        if (a.out_flags) a.out_flags[row] = SR_KFLAG_TOPK | (amb ? SR_KFLAG_AMBIGUOUS : 0u);
    }
}

// ---- SampleFromProbs / ResampleResidual on caller-provided distributions ------------------------------
__global__ __launch_bounds__(kT) void k_draw_rows(const float* probs, int64_t stride, int n, const double* uniforms,
                                                   int* out_tokens)
{
    __shared__ FullSmem sm;
    const int row = blockIdx.x;
    const int t = draw_from_row(probs + (size_t)row * stride, n, uniforms[row], sm);
    if (threadIdx.x == 0) out_tokens[row] = t;
}

// residual = max(0, p - q): first the left-to-right sum of the positive residuals, then the first index
// whose running residual reaches (float)u * sum; degenerate residual -> draw from p (Sampler.cs:587-618)
__device__ __forceinline__ int resample_residual_row(const float* p, const float* q, int n, double u, FullSmem& sm,
                                                     float m1 = 1.0f, float m2 = 1.0f)
{
    int dummy;
    auto res = [&](int i) -> float {
        const float r = __fsub_rn(__fmul_rn(__fmul_rn(p[i], m1), m2), q[i]);
        return r > 0.0f ? r : 0.0f;
    };
    SeqMarks marks;
    if (seq_marks_fit(n)) marks.keep = sm.ckpt;
    const float sum = seq_sum_residual<false>(p, q, n, 0.0f, 0.0f, &dummy, sm, m1, m2, marks);
    if (!(sum > 0.0f)) return draw_from_row(p, n, u, sm, m1, m2);  // sum <= 0 or NaN
    const float target = __fmul_rn(__double2float_rn(u), sum);
    // `target <= cum` is only tested on positive residuals: a zero target must not stop on a zero term
    int found;
    if (target <= 0.0f) {
        int first = 0x7fffffff;
        for (int i = threadIdx.x; i < n; i += kT)
            if (res(i) > 0.0f) { first = i; break; }
        first = sr_wave_min_i32(first);
        __syncthreads();
        if (sr_lane() == 0) sm.redi[sr_wave_id()] = first;
        __syncthreads();
        int f = 0x7fffffff;
        for (int w = 0; w < kW; w++) f = min(f, sm.redi[w]);
        __syncthreads();
        return f;  // sum > 0 guarantees a positive residual exists
    }
    float s0 = 0.0f;
    SeqMarks from;
    if (marks.keep) {
        __syncthreads();  // (the marks were written by thread 0)
        from.from = seq_marks_find(sm.ckpt, n, target, &s0);
    }
    seq_sum_residual<true>(p, q, n, s0, target, &found, sm, m1, m2, from);
    if (found >= 0) return found;
    // rounding fallback: the last index with a positive residual
    int last = -1;
    for (int i = threadIdx.x; i < n; i += kT)
        if (res(i) > 0.0f) last = i;
    last = -sr_wave_min_i32(-last);
    __syncthreads();
    if (sr_lane() == 0) sm.redi[sr_wave_id()] = last;
    __syncthreads();
    int l = -1;
    for (int w = 0; w < kW; w++) l = max(l, sm.redi[w]);
    __syncthreads();
    return l;
}

__global__ __launch_bounds__(kT) void k_residual_rows(const float* p, int64_t ps, const float* q, int64_t qs, int n,
                                                       const double* uniforms, int* out_tokens)
{
    __shared__ FullSmem sm;
    const int row = blockIdx.x;
    const int t = resample_residual_row(p + (size_t)row * ps, q + (size_t)row * qs, n, uniforms[row], sm);
    if (threadIdx.x == 0) out_tokens[row] = t;
}

// ... from the residual row itself (res[i] = max(0, fl(fl(p[i] m1) m2) - q[i]), written by k_spec_residual): the same
// terms in the same order, read from one row instead of computed from two
__device__ __forceinline__ int resample_residual_stored(const float* res, const float* p, int n, double u, FullSmem& sm,
                                                        float m1, float m2)
{
    int dummy;
    SeqMarks marks;
    if (seq_marks_fit(n)) marks.keep = sm.ckpt;
    const float sum = seq_sum_row<false>(res, n, 0.0f, 0.0f, &dummy, sm, 1.0f, 1.0f, SeqNoWatch(), SeqNoMap(), marks);
    if (!(sum > 0.0f)) return draw_from_row(p, n, u, sm, m1, m2);  // sum <= 0 or NaN
    const float target = __fmul_rn(__double2float_rn(u), sum);
    auto edge = [&](bool first_one) -> int {  // the first / the last index with a positive residual
        int at = first_one ? 0x7fffffff : -1;
        for (int i = threadIdx.x; i < n; i += kT)
            if (res[i] > 0.0f) {
                at = i;
                if (first_one) break;
            }
        at = first_one ? sr_wave_min_i32(at) : -sr_wave_min_i32(-at);
        __syncthreads();
        if (sr_lane() == 0) sm.redi[sr_wave_id()] = at;
        __syncthreads();
        int f = first_one ? 0x7fffffff : -1;
        for (int w = 0; w < kW; w++) f = first_one ? min(f, sm.redi[w]) : max(f, sm.redi[w]);
        __syncthreads();
        return f;
    };
    if (target <= 0.0f) return edge(true);  // a zero target must not stop on a zero term
    int found;
    float s0 = 0.0f;
    SeqMarks from;
    if (marks.keep) {
        __syncthreads();  // (the marks were written by thread 0)
        from.from = seq_marks_find(sm.ckpt, n, target, &s0);
    }
    seq_sum_row<true>(res, n, s0, target, &found, sm, 1.0f, 1.0f, SeqNoWatch(), SeqNoMap(), from);
    return found >= 0 ? found : edge(false);  // (rounding: the sum of the search fell short of the target)
}

// Every position of a row is filtered with the row's own parameters (SpeculativeDecoder.cs:535): the batch's row
// descriptors, one copy per position, without their allow-masks
__global__ __launch_bounds__(256) void k_expand_rows(const SrRow* src, SrRow* dst, int rows, int positions)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * positions) return;
    SrRow d = src[i / positions];
    d.mask_row = -1;
    dst[i] = d;
}

// The terms of the draw behind a row's accept loop: max(0, fl(fl(p m1) m2) - q) of its first rejected position, or the scaled target
// row of the bonus position
struct SpecTerms {
    const float* p;   // (starts on 16 bytes)
    const float* q;   // at any address; null: the bonus position
    float m1, m2;
    int n;
    __device__ __forceinline__ float term(float pv, float qv) const
    {
        const float sp = __fmul_rn(__fmul_rn(pv, m1), m2), r = q ? __fsub_rn(sp, qv) : sp;
        return q ? (r > 0.0f ? r : 0.0f) : sp;
    }
    __device__ __forceinline__ float at(int i) const { return term(p[i], q ? q[i] : 0.0f); }
    // four consecutive terms from i0, zeros past the end
    __device__ __forceinline__ float4 four(int i0) const
    {
        float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (i0 + 4 <= n) {
            const float4 pv = *(const float4*)(p + i0), qv = q ? sr_load_f4(q + i0) : o;
            o = make_float4(term(pv.x, qv.x), term(pv.y, qv.y), term(pv.z, qv.z), term(pv.w, qv.w));
        } else if (i0 < n) {
            o.x = at(i0);
            if (i0 + 1 < n) o.y = at(i0 + 1);
            if (i0 + 2 < n) o.z = at(i0 + 2);
        }
        return o;
    }
    __device__ __forceinline__ void run(int seg, float (&x)[SR_SEQ_RUN]) const  // a lane's 16 terms of a segment
    {
        float4 v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = four(seg * SR_SEG_TERMS + sr_lane() * SR_SEQ_RUN + 4 * k);
#pragma unroll
        for (int k = 0; k < 4; k++) { x[4 * k] = v[k].x; x[4 * k + 1] = v[k].y; x[4 * k + 2] = v[k].z; x[4 * k + 3] = v[k].w; }
    }
};
// e of token tok at a position of the verifier's batch (its place in the logits is asked for beside the state that says which holds).
// kOpenUnread: in the launch that writes e of open positions, where whoever counts in last reads it behind this: what stands there
// before is not loaded at all, or this die's cache would keep the line as it was.  Behind that launch both places are asked for at
// once (with the branch there too 0.5 - 0.9 us).
template <bool kOpenUnread>
__device__ __forceinline__ float spec_e(const SrSpecArgs& a, const SrRow& rd, size_t slot, int tok, const uint64_t* tab)
{
    const SrFullState* sl = a.state + slot;
    const uint32_t open = sl->e_open;
    const float* const at = a.p_all + slot * (size_t)a.p_stride + tok;
    const float x = a.target_logits[slot * (size_t)a.vocab + tok];
    float there = 0.0f;
    if (!kOpenUnread || open != a.seq) there = *at;
    ERow r;
    r.inv_temp = row_inv_temp(rd);
    r.max = sr_okey_inv((uint32_t)sl->maxkey);
    r.tab = tab;
    const float made = r.of(x);
    return open == a.seq ? made : there;
}
__device__ __forceinline__ void spec_table(uint64_t* tab)  // by the first wave, which uses it first
{
    if (threadIdx.x < 32) tab[threadIdx.x] = sr_exp2f_tab[threadIdx.x];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ float spec_accept(float px, float qx) { return qx > 0.0f ? fminf(1.0f, __fdiv_rn(px, qx)) : (px > 0.0f ? 1.0f : 0.0f); }
// The accept loop of a row under the ratio test needs one element of p and of q per position, no pass over a row:
// one wave walks it ahead of everything else and names the first rejected position, so that the residual row of
// that position -- which the row's workgroup would otherwise compute twice, from two rows, at the rate of one compute
// unit -- can be written by the whole device (k_spec_residual) before k_spec_verify reads it.
__global__ __launch_bounds__(SR_WAVE) void k_spec_walk(SrSpecArgs a)
{
    const int row = blockIdx.x, lane = sr_lane();
    const SrRow rd = a.rows[row];
    const int n = a.vocab, L = a.n_draft;
    const bool true_spec = spec_by_ratio(rd);
    int reject = -1;
    if (true_spec) {
        const float* pr = a.p_all + (size_t)row * (L + 1) * (size_t)a.p_stride;
        const double* u = a.uniforms + (size_t)row * a.uniforms_per_row;
        for (int i0 = 0; i0 < L; i0 += SR_WAVE) {
            const int i = i0 + lane;
            bool stop = false, bad = false;
            if (i < L) {
                const int tok = a.draft_tokens[(size_t)row * L + i];
                bad = (uint32_t)tok >= (uint32_t)n;
                if (!bad) {
                    const SrFullState* sl = a.state + (size_t)row * (L + 1) + i;
                    const float px = __fmul_rn(__fmul_rn(pr[(size_t)i * (size_t)a.p_stride + tok], sl->mul1), sl->mul2);
                    const float qx = a.draft_probs[((size_t)row * L + i) * n + tok];
                    const float acc = spec_accept(px, qx);
                    stop = !(u[i] < (double)acc);  // (every position before it was accepted and drew one uniform)
                }
            }
            const unsigned long long ends = __ballot(stop || bad);
            if (ends != 0ull) {
                const int l = (int)__ffsll((long long)ends) - 1;
                const bool is_bad = ((__ballot(bad) >> l) & 1ull) != 0ull;
                reject = is_bad ? -1 : i0 + l;  // (an id outside the vocabulary ends the row without a correction)
                break;
            }
        }
    }
    if (lane == 0) a.reject[row] = reject;
}

// The terms the row's workgroup will add, written by the whole device: max(0, fl(fl(p m1) m2) - q) of the first rejected
// position.
__global__ __launch_bounds__(256) void k_spec_residual(SrSpecArgs a)
{
    const int row = blockIdx.y;
    const int i = a.reject[row];
    if (i < 0) return;
    const int n = a.vocab, L = a.n_draft;
    SpecTerms t;
    t.p = a.p_all + ((size_t)row * (L + 1) + i) * (size_t)a.p_stride;
    t.q = a.draft_probs + ((size_t)row * L + i) * n;
    const SrFullState* sl = a.state + (size_t)row * (L + 1) + i;
    t.m1 = sl->mul1;
    t.m2 = sl->mul2;
    t.n = n;
    float* const out = a.resid + (size_t)row * (size_t)a.resid_stride;
    for (int x0 = ((int)blockIdx.x * 256 + (int)threadIdx.x) * 4; x0 < n; x0 += (int)gridDim.x * 1024) *(float4*)(out + x0) = t.four(x0);
    // (the rows of a.resid start on 16 bytes and are a multiple of 16 bytes long)
}

// The factors 1 / (sum of the probabilities) of the final Normalize (Sampler.cs:91-92), for the positions that need theirs.  A row
// that nothing cuts has probabilities fl(fl(e m1) m2), m1 = fl(1 / s) with s the sum of e added one behind the other, and m2 hangs on
// the exact sum of all fl(e m1) in the eight accumulators.  About the sum of e, S, is known from the segments' sums to 50
// roundings, so m2 is s / S but for those and the n / 8 additions of an accumulator (all terms are positive): spec_spread(n), 0.2 % at
// 262,144.  Nearly every accept test comes out the same at both ends.  What needs m2 itself: the positions in front of the first
// certain rejection whose test is open, and the position that the row draws from.  k_full_row leaves all of them at s / S
// (SrFullState::deferred), a workgroup per block of a row's 8,192 entries finds those positions for itself, a position a lane, and
// takes them as k_prepared_row takes a row up to the factor.  The positions left at s / S are tested with that.
// So e of the others is read nowhere but at their draft token, and is not written at all (row_e_open).  What bounds it: the chain again, two trips
// for the positions 2.4 us, the block from its logits 10 - 12 us (expf of 16 entries a lane is a third), the meeting 4 - 5, records 3, the
// walk 5.  144 rows of 262,144, us: k_full_softmax_seg 72 -> 59, k_full_row, whose workgroups made the sums of all of them, 48 -> 15, this
// one 28; the call 143 -> 127.  (e stored in front of the meeting, whose barrier waits for it: this kernel 30.)
__device__ __forceinline__ double spec_spread(int n) { return ((double)(n / 8) + 200.0) * (1.1 / 16777216.0) + 1e-6; }
__global__ __launch_bounds__(kPrepT, 4) void k_spec_factor(SrFullArgs a, SrSpecArgs s)
{
    __shared__ PreparedSmem sm;
    __shared__ unsigned long long said;
    __shared__ uint64_t tab[32];
    const int row = blockIdx.y, lane = sr_lane();
    const SrRow rd = s.rows[row];
    if (!spec_by_ratio(rd)) return;
    const int n = s.vocab, L = s.n_draft;  // (L < SR_WAVE)
    if (sr_wave_id() == 0) {
        spec_table(tab);
        bool open = false, ends = false, bad = false;
        if (lane < L) {
            const int tok = s.draft_tokens[(size_t)row * L + lane];
            bad = (uint32_t)tok >= (uint32_t)n;
            if (!bad) {
                const SrFullState* sl = s.state + (size_t)row * (L + 1) + lane;
                const bool any = sl->deferred == a.seq;  // m2 is s / S so far
                const float y = __fmul_rn(spec_e<true>(s, rd, (size_t)row * (L + 1) + lane, tok, tab), sl->mul1);
                const float qx = s.draft_probs[((size_t)row * L + lane) * n + tok];
                const double u = s.uniforms[(size_t)row * s.uniforms_per_row + lane];
                const float acc = spec_accept(__fmul_rn(y, sl->mul2), qx);
                ends = !(u < (double)acc);
                if (any && y > 0.0f) {
                    if (!(qx > 0.0f)) {
                        open = y < 1e-30f;
                    } else {
                        const double ratio = (double)y * (double)sl->mul2 / (double)qx, d = spec_spread(n);
                        const bool low = u < fmin(1.0, ratio * (1.0 - d)), high = u < fmin(1.0, ratio * (1.0 + d));
                        open = low != high || y < 1e-30f || !(ratio >= 1e-30);  // (relative bounds end where numbers lose digits)
                    }
                }
            }
        }
        const unsigned long long end = __ballot(!open && (ends || bad)), wrong = __ballot(bad), undecided = __ballot(open);
        const int last = end != 0ull ? (int)__ffsll((long long)end) - 1 : L;
        unsigned long long pick = undecided & ((1ull << last) - 1ull);
        if (((wrong >> last) & 1ull) == 0ull) pick |= 1ull << last;  // (an id outside the vocabulary ends the row without a draw)
        if (lane == 0) said = pick;
    }
    __syncthreads();
    const float inv_temp = row_inv_temp(rd);
    for (unsigned long long pick = said; pick != 0ull; pick &= pick - 1ull) {
        const int slot = row * (L + 1) + (int)__ffsll((long long)pick) - 1;
        if (a.state[slot].deferred != a.seq) continue;
        prepared_block<3>(a, slot, sm, tab, inv_temp);
        __syncthreads();
    }
}

// ---- launches of which every row is open: nothing cuts, biases or penalises it, and the ratio test decides ------------------------
// An accept test needs p at one token, and p = fl(fl(e m1) m2) is e / S to spec_open_spread(n) whatever the exact sums are: m1 = fl(1 / s), and m2 is s
// / S but for the roundings of the accumulators.  So the pass over all positions needs neither e to the last bit nor a sum in
// order, and no position waits for another's: k_spec_units reads the logits once, a wave a unit of 2,048, and leaves every unit's
// maximum and about its sum of exp(x - maximum), by lane accumulator.  What needs the exact factors -- the positions in front of the
// first certain rejection whose test is open, and the one that is drawn from, one or two of nine -- k_spec_open works out from
// the logits: e, the records of its sum, m1; the records of the eight accumulators over fl(e m1), m2.
// 16 sequences of 8 drafts over 262,144 (144 rows), us: this one 23 (6.6 TB/s; k_full_softmax_seg, with e, two meetings and records, 59),
// k_full_row none (15), k_spec_open 45 (k_spec_factor 28; its chain: tests 3.4, the block from its logits 8, records 5, walk 7, records 5,
// walk 4), k_spec_rows 23 both; the call 127 -> 98.  A further position with an open test is another 25.  A bonus row whose largest entry
// decides (row_decided: the units bound its draw) needs none of it: calls without a rejection 45, 1 x 8 of 262,144 50 -> 17, 16 x 4 of 128,256 62 -> 25.
// A unit's maximum is exact; a term's exponential is v_exp_f32 of a difference rounded once: 2^-24 of the exponent's size, which is
// below 28 for all terms that make up more than 2^-22 of the sum.
// What k_spec_open leaves of a row's tests, behind its meeting point (SrSpecArgs::sync): the positions that it worked out, a bit each; those
// of them whose draft is accepted; the position that ends the row for certain, and above it whether its id lies outside the vocabulary
constexpr int kSpecPicked = 4, kSpecAccepted = 5, kSpecLast = 6;
constexpr unsigned long long kSpecWritten = 1ull << 33;  // ... or that the row's results are written
constexpr int kSpecDone = -2;  // SrSpecArgs::reject of a row whose results are written
// The words behind a position's meeting point (SrFullArgs::row_sync) that count its workgroups in, k_spec_units clears them.  (Not
// those of k_prepared_row and of the greedy rows: other launches of the context find these as they left them.)
constexpr int kOpenFirst = 4, kOpenSecond = 5;
constexpr int kUnitVecs = SR_UNIT_TERMS / (4 * SR_WAVE);
__global__ __launch_bounds__(256) void k_spec_units(SrFullArgs a, SrSpecArgs s)
{
    const int slot = blockIdx.y, lane = sr_lane(), u = (int)blockIdx.x * 4 + sr_wave_id(), n = s.vocab;
    if (blockIdx.x == 0 && threadIdx.x < 2) {  // nobody has counted in
        a.row_sync[(size_t)slot * SR_ROW_SYNC_STRIDE + kOpenFirst + threadIdx.x] = 0ull;
        if (slot % (s.n_draft + 1) == 0 && threadIdx.x == 0) s.sync[(size_t)(slot / (s.n_draft + 1)) * SR_ROW_SYNC_STRIDE + kSpecAccepted] = 0ull;
    }
    if (u >= s.n_units) return;
    const SrRow rd = s.rows[slot / (s.n_draft + 1)];
    const float inv_temp = row_inv_temp(rd);
    const float* const x = s.target_logits + (size_t)slot * (size_t)n;
    float v[kUnitVecs][4];
    const int base = u * SR_UNIT_TERMS + lane * 4;
    if ((u + 1) * SR_UNIT_TERMS <= n) {
#pragma unroll
        for (int k = 0; k < kUnitVecs; k++) {
            const float4 t = sr_load_f4(x + base + k * 4 * SR_WAVE);
            v[k][0] = t.x; v[k][1] = t.y; v[k][2] = t.z; v[k][3] = t.w;
        }
        if (rd.temperature != 1.0f) {
#pragma unroll
            for (int k = 0; k < kUnitVecs; k++)
#pragma unroll
                for (int q = 0; q < 4; q++) v[k][q] = __fmul_rn(v[k][q], inv_temp);
        }
    } else {
#pragma unroll
        for (int k = 0; k < kUnitVecs; k++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int i = base + k * 4 * SR_WAVE + q;
                v[k][q] = i < n ? __fmul_rn(x[i], inv_temp) : SR_NEG_INF;
            }
    }
    float m = v[0][0];
#pragma unroll
    for (int k = 0; k < kUnitVecs; k++) m = sr_max3_f32(sr_max3_f32(m, v[k][0], v[k][1]), v[k][2], v[k][3]);
    m = sr_okey_inv(sr_wave_max_u32(m == m ? sr_okey(m) : 0x007fffffu));  // (a NaN beside numbers is left out here; its exponential is one)
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < kUnitVecs; k++)
#pragma unroll
        for (int q = 0; q < 4; q++) acc[q] += __builtin_amdgcn_exp2f((v[k][q] - m) * kLog2E);
    // lane l holds the terms of the accumulators 4 (l & 1) ... 4 (l & 1) + 3
    float c[SR_SEQ_CHAINS];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        c[q] = (lane & 1) ? 0.0f : acc[q];
        c[4 + q] = (lane & 1) ? acc[q] : 0.0f;
    }
    float chain = wave_sum_8(c);  // (of accumulator lane & 7)
    float sum = sr_wave_sum_f32((acc[0] + acc[1]) + (acc[2] + acc[3]));
    if (!(sum > 0.0f)) {  // (the same in every lane) nothing above -inf, +inf, or a NaN
        bool nan = false;
#pragma unroll
        for (int k = 0; k < kUnitVecs; k++)
#pragma unroll
            for (int q = 0; q < 4; q++) nan = nan || v[k][q] != v[k][q];
        if (__ballot(nan) != 0ull) m = sr_u2f(0x7fc00000u);
        sum = chain = 0.0f;
    }
    const size_t at = (size_t)slot * s.n_units + u;
    if (lane < SR_SEQ_CHAINS) s.unit_chains[at * SR_SEQ_CHAINS + lane] = chain;
    if (lane == 0) s.units[at] = make_float2(m, sum);
}

// A row's units, kUnits a lane: its maximum, and about its sum relative to it.  One wave.
constexpr int kUnitsMost = SR_SEG_MAX * SR_SEG_TERMS / SR_UNIT_TERMS / SR_WAVE, kUnitsFew = 2;
struct SpecRow {
    float max, sum;
    int kind;  // 0: numbers   1: a NaN, or nothing above -inf: the row is uniform   2: +inf
};
template <int kUnits>
__device__ __forceinline__ SpecRow spec_row(const SrSpecArgs& s, size_t slot, float2 (&w)[kUnits])
{
    const int lane = sr_lane();
    SpecRow r;
    float m = SR_NEG_INF;
    bool nan = false;
#pragma unroll
    for (int k = 0; k < kUnits; k++) {
        // (no lane's load behind a condition: they would wait for each other)
        w[k] = make_float2(SR_NEG_INF, 0.0f);
        if (k * SR_WAVE < s.n_units) w[k] = s.units[slot * s.n_units + min(k * SR_WAVE + lane, s.n_units - 1)];
    }
#pragma unroll
    for (int k = 0; k < kUnits; k++)
        if (k * SR_WAVE + lane >= s.n_units) w[k] = make_float2(SR_NEG_INF, 0.0f);
#pragma unroll
    for (int k = 0; k < kUnits; k++) {
        nan = nan || w[k].x != w[k].x;
        m = fmaxf(m, w[k].x);
    }
    r.max = sr_okey_inv(sr_wave_max_u32(sr_okey(m)));
    r.kind = __ballot(nan) != 0ull || r.max == SR_NEG_INF ? 1 : r.max == -SR_NEG_INF ? 2 : 0;
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < kUnits; k++)
        if (k * SR_WAVE < s.n_units) sum += w[k].x > SR_NEG_INF ? w[k].y * __builtin_amdgcn_exp2f((w[k].x - r.max) * kLog2E) : 0.0f;
    r.sum = sr_wave_sum_f32(sum);
    return r;
}
// How far p is from e / S, as a part of it: n / 8 additions of an accumulator and a handful of roundings, and S itself (above).
__device__ __forceinline__ double spec_open_spread(int n) { return ((double)(n / 8) + 200.0) * (1.1 / 16777216.0) + 3e-5; }

// A workgroup per block of a row's 8,192 entries.  Each finds the positions whose factors are asked for by itself (a position a wave,
// from the units), and takes them one by one: e of its block from the logits; the records of its eight segments (what stands in front is
// known from the units: no meeting); counts in, and whoever is there last walks the row's records to s, while the others write e
// and wait for m1 (bounded); then fl(e m1) by accumulator, the records, counts in, and whoever is there last walks those to m2.
// A workgroup whose wait runs out marks the position (SrFullState::late_behind) and counts itself in; the last one then adds the
// accumulators without records.
// one position of a row: e from the logits
struct SpecOpenRow {
    const float* lg;
    const uint64_t* tab;  // of expf, in shared memory
    float inv_temp, max, uniform;
    int kind, n, lane;
    __device__ __forceinline__ float e(float x) const
    {
        const float d = __fsub_rn(__fmul_rn(x, inv_temp), max);
        const float v = d == d ? sr_expf_neg(d, tab) : d;  // (beside +inf, +inf is no number and everything else 0)
        return kind == 1 ? uniform : v;
    }
    // (for the walks' rare segments: a few at a time, beside which the walk keeps its registers)
    template <int kN> __device__ __forceinline__ void all(float (&x)[kN]) const
    {
#pragma unroll
        for (int j = 0; j < kN; j++) {
            x[j] = e(x[j]);
            if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
    }
    // a lane's 16 entries of e of a segment
    __device__ __forceinline__ void run(int sg, float (&x)[SR_SEQ_RUN]) const
    {
        const int i0 = sg * SR_SEG_TERMS + lane * SR_SEQ_RUN;
        if ((sg + 1) * SR_SEG_TERMS <= n) {
#pragma unroll
            for (int j = 0; j < SR_SEQ_RUN; j += 4) {
                const float4 l = sr_load_f4(lg + i0 + j);
                x[j] = l.x; x[j + 1] = l.y; x[j + 2] = l.z; x[j + 3] = l.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = lg[min(i0 + j, n - 1)];
        }
        all(x);
#pragma unroll
        for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = i0 + j < n ? x[j] : 0.0f;
    }
    // ... and of accumulator g of a block: fl(e m1)
    __device__ __forceinline__ void accumulator(int b, int g, float m1, float (&x)[SR_SEQ_RUN]) const
    {
        const int t0 = b * SR_SEG_TERMS + lane * SR_SEQ_RUN, nv = n / 8;
#pragma unroll
        for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = lg[(size_t)min(t0 + j, nv - 1) * 8 + g];
        all(x);
#pragma unroll
        for (int j = 0; j < SR_SEQ_RUN; j++) x[j] = t0 + j < nv ? __fmul_rn(x[j], m1) : 0.0f;
    }
};
__device__ __forceinline__ float spec_m(float sum) { return sum > 0.0f && sum != 1.0f ? __fdiv_rn(1.0f, sum) : 1.0f; }
// All records of a row that others of the launch have made, into shared memory, by the workgroup, where they fit: the waves' trips to
// memory overlap, where the walk of one wave makes them one behind the other.
template <int kThreads>
__device__ __forceinline__ bool stage_records(const SeqSegFunc* recs, int nrec, float4* room, int room_bytes)
{
    const bool fits = nrec * (int)sizeof(SeqSegFunc) <= room_bytes;
    if (fits) {
        const unsigned long long* const from = (const unsigned long long*)recs;
        unsigned long long* const to = (unsigned long long*)room;
        constexpr int kWords = sizeof(SeqSegFunc) / 8, kAhead = 6;
        for (int i0 = threadIdx.x; i0 < nrec * kWords; i0 += kThreads * kAhead) {
            unsigned long long v[kAhead];
#pragma unroll
            for (int k = 0; k < kAhead; k++) v[k] = i0 + k * kThreads < nrec * kWords ? sr_load_agent(from + i0 + k * kThreads) : 0ull;
#pragma unroll
            for (int k = 0; k < kAhead; k++)
                if (i0 + k * kThreads < nrec * kWords) to[i0 + k * kThreads] = v[k];
        }
    }
    __syncthreads();
    return fits;
}

template <int kUnits>  // a lane (eight cost 30 registers that most vocabularies do not need)
__global__ __launch_bounds__(kPrepT, 4) void k_spec_open(SrFullArgs a, SrSpecArgs s)
{
    __shared__ PreparedSmem sm;
    __shared__ uint64_t tab[32];
    __shared__ int test[SR_WAVE];       // of every position   1: its test is open   2: it ends the row   4: an id outside the vocabulary
    __shared__ float seg_own[SR_SEQ_CHAINS];
    const int row = blockIdx.y, blk = blockIdx.x, tid = threadIdx.x, lane = sr_lane(), wave = sr_wave_id();
    const SrRow rd = s.rows[row];
    const int n = s.vocab, L = s.n_draft, nseg = seg_count(n);  // (L < SR_WAVE)
    const int nv = n / 8, rem = n - nv * 8, body = nv * 8, nblk = (nv + SR_SEG_TERMS - 1) / SR_SEG_TERMS;
    SpecOpenRow t;
    t.tab = tab;
    t.inv_temp = row_inv_temp(rd);
    t.n = n;
    t.uniform = __fdiv_rn(1.0f, (float)n);
    if (tid < 32) tab[tid] = sr_exp2f_tab[tid];
    __syncthreads();
    float2 w[kUnits];
    for (int i = wave; i < L; i += SR_SEQ_CHAINS) {
        const size_t slot = (size_t)row * (L + 1) + i;
        const int tok = s.draft_tokens[(size_t)row * L + i];
        const bool bad = (uint32_t)tok >= (uint32_t)n;
        const float x = bad ? 0.0f : s.target_logits[slot * (size_t)n + tok], qx = bad ? 0.0f : s.draft_probs[((size_t)row * L + i) * n + tok];
        const double u = s.uniforms[(size_t)row * s.uniforms_per_row + i];
        const SpecRow r = spec_row(s, slot, w);
        bool open = r.kind != 0, ends = bad;
        if (!bad && r.kind == 0) {
            const float e = sr_expf_neg(__fsub_rn(__fmul_rn(x, t.inv_temp), r.max), tab);
            const double y = (double)e / (double)r.sum;
            if (!(e > 0.0f)) {
                ends = !(u < 0.0);  // (p is 0, whatever the factors are, and so is the ratio)
            } else if (!(qx > 0.0f)) {
                open = y < 1e-29;
                ends = !(u < 1.0);
            } else {
                const double ratio = y / (double)qx, d = spec_open_spread(n);
                const bool low = u < fmin(1.0, ratio * (1.0 - d)), high = u < fmin(1.0, ratio * (1.0 + d));
                open = low != high || y < 1e-29 || !(ratio >= 1e-30);  // (relative bounds end where numbers lose digits)
                ends = !low;
            }
        }
        if (lane == 0) test[i] = (open && !bad ? 1 : 0) | (ends ? 2 : 0) | (bad ? 4 : 0);
    }
    __syncthreads();
    unsigned long long pick;
    int last;
    {
        const int f = lane < L ? test[lane] : 0;
        const unsigned long long end = __ballot((f & 3) == 2), wrong = __ballot((f & 4) != 0), undecided = __ballot((f & 1) != 0);
        last = end != 0ull ? (int)__ffsll((long long)end) - 1 : L;
        pick = undecided & ((1ull << last) - 1ull);
        if (((wrong >> last) & 1ull) == 0ull) pick |= 1ull << last;  // (an id outside the vocabulary ends the row without a draw)
    }
    unsigned long long* const said = s.sync + (size_t)row * SR_ROW_SYNC_STRIDE;
    if (blk == 0 && blockIdx.z == 0 && tid == 0) {
        said[kSpecPicked] = pick;
        said[kSpecLast] = (unsigned long long)last | (last < L && (test[last] & 4) != 0 ? 1ull << 32 : 0ull);
    }
    const bool only_bonus = pick == 1ull << L;  // every draft is accepted for certain
    const float u_bonus = only_bonus ? __double2float_rn(s.uniforms[(size_t)row * s.uniforms_per_row + L]) : 0.0f;
    // (the grid's third dimension: positions side by side)
    auto next = [&](int by) __attribute__((always_inline)) {
        for (int i = 0; i < by; i++) pick &= pick - 1ull;
    };
    for (next((int)blockIdx.z); pick != 0ull; next((int)gridDim.z)) {
        // (what the lane's number gives is worked out here: kept over the whole loop, its dozens of offsets cost that many registers)
        int ln = lane;
        asm volatile("" : "+v"(ln));
        t.lane = ln;
        const int pos = (int)__ffsll((long long)pick) - 1;
        const size_t slot = (size_t)row * (L + 1) + (size_t)pos;
        SrFullState* const st = a.state + slot;
        unsigned long long* const sync = a.row_sync + slot * SR_ROW_SYNC_STRIDE;
        SeqSegFunc* const recs = a.seg_func + slot * a.seg_stride;
        SeqSegFunc* const chain = a.chain_func + (slot * SR_SEQ_CHAINS + wave) * a.chain_blocks;
        float* const e_row = const_cast<float*>(s.p_all) + slot * (size_t)s.p_stride;
        const int seg = blk * SR_SEQ_CHAINS + wave;
        t.lg = s.target_logits + slot * (size_t)n;
        // (all loads of a whole segment without a condition)
        float v[4][4];
        if ((seg + 1) * SR_SEG_TERMS <= n) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float4 x = sr_load_f4(t.lg + seg * SR_SEG_TERMS + (k * SR_WAVE + ln) * 4);
                v[k][0] = x.x; v[k][1] = x.y; v[k][2] = x.z; v[k][3] = x.w;
            }
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int q = 0; q < 4; q++) v[k][q] = t.lg[min(seg * SR_SEG_TERMS + (k * SR_WAVE + ln) * 4 + q, n - 1)];
        }
        // about what stands in front of the block, of all terms and of the wave's accumulator
        constexpr int kBlockUnits = kPrepBlock / SR_UNIT_TERMS;
        float uc[kUnits] = {};
#pragma unroll
        for (int k = 0; k < kUnits; k++)
            if (k * SR_WAVE < blk * kBlockUnits) uc[k] = s.unit_chains[(slot * s.n_units + min(k * SR_WAVE + ln, s.n_units - 1)) * SR_SEQ_CHAINS + wave];
        const SpecRow r = spec_row(s, slot, w);
        t.max = r.max;
        t.kind = __builtin_amdgcn_readfirstlane(r.kind);
        float before = 0.0f, before_chain = 0.0f;
#pragma unroll
        for (int k = 0; k < kUnits; k++)
            if (k * SR_WAVE < blk * kBlockUnits) {
                const float scale = k * SR_WAVE + ln < blk * kBlockUnits && w[k].x > SR_NEG_INF ? __builtin_amdgcn_exp2f((w[k].x - r.max) * kLog2E) : 0.0f;
                before += w[k].y * scale;
                before_chain += uc[k] * scale;
            }
        if (only_bonus && t.kind == 0) {
            // whether the bonus row's largest entry is its token: the same answer in every workgroup
            int first = s.n_units;  // the unit that holds it
#pragma unroll
            for (int k = kUnits - 1; k >= 0; k--) {
                const unsigned long long top = __ballot(w[k].x == r.max);
                if (top != 0ull) first = k * SR_WAVE + (int)__ffsll((long long)top) - 1;
            }
            float front = 0.0f, own_unit = 0.0f;
#pragma unroll
            for (int k = 0; k < kUnits; k++) {
                const float part = w[k].x > SR_NEG_INF ? w[k].y * __builtin_amdgcn_exp2f((w[k].x - r.max) * kLog2E) : 0.0f;
                front += k * SR_WAVE + ln < first ? part : 0.0f;
                own_unit += k * SR_WAVE + ln == first ? part : 0.0f;
            }
            if (row_decided(rd, n, r.sum, sr_wave_sum_f32(front), sr_wave_sum_f32(own_unit), u_bonus)) {
                if (blk == 0 && tid == 0) said[kSpecLast] = (unsigned long long)L | kSpecWritten;
                int at = -1;  // (the only entry of its value: one lane of one workgroup)
#pragma unroll
                for (int k = 0; k < 4; k++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const int i = seg * SR_SEG_TERMS + (k * SR_WAVE + ln) * 4 + q;
                        at = i < n && __fmul_rn(v[k][q], t.inv_temp) == r.max ? i : at;
                    }
                const unsigned long long has = __ballot(at >= 0);
                if (has != 0ull) {
                    const int token = __builtin_amdgcn_readlane(at, (int)__ffsll((long long)has) - 1);
                    int* const out = s.out_tokens + (size_t)row * (L + 1);
                    if (ln < L) out[ln] = s.draft_tokens[(size_t)row * L + ln];
                    if (ln == L) out[ln] = token;
                    if (ln == 0) {
                        s.out_accepted[row] = L;
                        s.reject[row] = kSpecDone;
                    }
                }
                break;
            }
        }
        before = sr_wave_sum_f32(before);
        before_chain = sr_wave_sum_f32(before_chain);
#pragma unroll
        for (int k = 0; k < 4; k++) {
#pragma unroll
            for (int q = 0; q < 4; q++) v[k][q] = t.e(v[k][q]);
#pragma unroll
            for (int q = 0; q < 4; q++) v[k][q] = seg * SR_SEG_TERMS + (k * SR_WAVE + ln) * 4 + q < n ? v[k][q] : 0.0f;
        }
        auto write_e = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int i0 = seg * SR_SEG_TERMS + (k * SR_WAVE + ln) * 4;
                if (i0 < n) sr_store_agent_f4((float4*)(e_row + i0), v[k][0], v[k][1], v[k][2], v[k][3]);  // (the rows of e are whole pieces long)
            }
        };
        auto count_in = [&](int word) __attribute__((always_inline)) -> bool {  // whether this workgroup is the last one
            sr_drain_stores();
            __syncthreads();
            if (tid == 0) sm.bc[0] = (uint32_t)__hip_atomic_fetch_add(sync + word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u == gridDim.x ? 1u : 0u;
            __syncthreads();
            return sm.bc[0] != 0u;
        };
        float m1 = 1.0f, x[SR_SEQ_RUN], own = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++) own += (v[k][0] + v[k][1]) + (v[k][2] + v[k][3]);
        own = sr_wave_sum_f32(own);
        bool here = true;
        if (t.kind == 0) {
            // into the order of the sum, 16 terms a ln
            float4* const turn = sm.room + wave * SR_WAVE * 5;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int i = (k * SR_WAVE + ln) * 4;
                turn[(i >> 4) * 5 + ((i & 15) >> 2)] = make_float4(v[k][0], v[k][1], v[k][2], v[k][3]);
            }
            if (ln == 0) seg_own[wave] = own;
            __syncthreads();
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float4 q = turn[ln * 5 + k];
                x[4 * k] = q.x; x[4 * k + 1] = q.y; x[4 * k + 2] = q.z; x[4 * k + 3] = q.w;
            }
#pragma unroll
            for (int g = 0; g < SR_SEQ_CHAINS; g++) before += g < wave ? seg_own[g] : 0.0f;
            if (seg < nseg) seg_make_record<true>(x, seg, (double)before, recs + seg, own);
            if (count_in(kOpenFirst)) {
                const bool staged = stage_records<kPrepT>(recs, nseg, sm.room, (int)sizeof(sm.room));
                if (wave == 0) {
                    int dummy;
                    auto load = [&](int sg, float (&y)[SR_SEQ_RUN]) __attribute__((always_inline)) { t.run(sg, y); };
                    // (one piece of code for both places)
                    const float f = spec_m(seg_walk_from<false, true, false, true>(load, nseg, staged ? (const SeqSegFunc*)sm.room : recs, 0.0f, 0.0f, &dummy, nullptr));
                    if (ln == 0) {
                        sr_store_agent(sync + 3, ((unsigned long long)a.seq << 32) | (unsigned long long)sr_f2u(f));
                        sm.bc[1] = sr_f2u(f);
                        sm.bc[2] = 1u;
                    }
                }
                write_e();
            } else {
                write_e();
                if (tid == 0) {
                    uint32_t ok = 0u;
                    unsigned long long word = 0ull;
                    for (uint32_t it = 0; it < a.behind_wait_limit; it++) {
                        word = sr_load_agent(sync + 3);
                        if ((uint32_t)(word >> 32) == a.seq) { ok = 1u; break; }
                        __builtin_amdgcn_s_sleep(1);
                    }
                    if (ok == 0u) sr_store_agent(&st->late_behind, a.seq);
                    sm.bc[2] = ok;
                    sm.bc[1] = (uint32_t)word;
                }
            }
            __syncthreads();
            here = sm.bc[2] != 0u;
            m1 = sr_u2f(sm.bc[1]);
        } else {
            write_e();
        }
        if (t.kind != 2 && here && blk < nblk) {
            // chain by chain in shared memory, as in prepared_block
            float* const buf = (float*)sm.room;
            __syncthreads();
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int t4 = wave * (SR_SEG_TERMS / 4) + k * SR_WAVE + ln;
                const int vec = t4 >> 1, j = vec & 15, l = vec >> 4;
                const bool in = blk * kPrepBlock + 4 * t4 < body;
                float* at = buf + (4 * (t4 & 1)) * 1024 + 64 * j + ((l + 2 * j) & 63);
#pragma unroll
                for (int q = 0; q < 4; q++) at[1024 * q] = in ? __fmul_rn(v[k][q], m1) : 0.0f;
            }
            __syncthreads();
            own = 0.0f;
#pragma unroll
            for (int j = 0; j < SR_SEQ_RUN; j++) {
                x[j] = buf[wave * 1024 + 64 * j + ((ln + 2 * j) & 63)];
                own += x[j];
            }
            own = sr_wave_sum_f32(own);
            const float front = t.kind == 0 ? before_chain * m1 : (float)(blk * SR_SEG_TERMS) * t.uniform;
            seg_make_record<true>(x, blk, (double)front, chain + blk, own);
        }
        if (count_in(kOpenSecond)) {
            // (everyone's e, records and marks are out; m1 is there)
            if (tid == 0) {
                sm.bc[2] = sr_load_agent(&st->late_behind) == a.seq ? 1u : 0u;
                if (t.kind == 0) sm.bc[1] = (uint32_t)sr_load_agent(sync + 3);
            }
            __syncthreads();
            if (t.kind == 0) m1 = sr_u2f(sm.bc[1]);
            float m2 = 1.0f;
            if (t.kind != 2) {
                int dummy;
                float sum = 0.0f;
                if (sm.bc[2] == 0u) {
                    sum = seg_walk_from<false, true, false, true>([&](int b, float (&y)[SR_SEQ_RUN]) __attribute__((always_inline)) { t.accumulator(b, wave, m1, y); },
                                                     nblk, chain, 0.0f, 0.0f, &dummy, nullptr);
                } else {
                    for (int b = 0; b < nblk; b++) {  // (some workgroup stopped waiting and made no records)
                        t.accumulator(b, wave, m1, x);
                        sum = sr_seq_wave<SR_SEQ_RUN, false>(x, sum, 0.0f, &dummy);
                    }
                }
                if (rem > 0 && wave >= 8 - rem) sum = __fadd_rn(sum, __fmul_rn(t.e(t.lg[n - 8 + wave]), m1));  // the overlapped last vector
                if (ln == 0) sm.lane_sum[wave] = sum;
                __syncthreads();
                const float* const l = sm.lane_sum;
                m2 = spec_m(__fadd_rn(__fadd_rn(__fadd_rn(l[0], l[1]), __fadd_rn(l[2], l[3])), __fadd_rn(__fadd_rn(l[4], l[5]), __fadd_rn(l[6], l[7]))));
            }
            if (tid == 0) {
                st->mul1 = m1;
                st->mul2 = m2;
                if (pos != last) {  // (an open test: with the factors it is exact)
                    const int tok = s.draft_tokens[(size_t)row * L + pos];
                    const float px = __fmul_rn(__fmul_rn(t.e(t.lg[tok]), m1), m2);
                    if (s.uniforms[(size_t)row * s.uniforms_per_row + pos] < (double)spec_accept(px, s.draft_probs[((size_t)row * L + pos) * n + tok]))
                        __hip_atomic_fetch_or(said + kSpecAccepted, 1ull << pos, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
        __syncthreads();
    }
}

// ---- speculative verification of rows under the ratio test (StepSampled, SpeculativeDecoder.cs:530-559) --------------------
// The accept loop of such a row needs one element of p and of q per position, and the draw behind it one row of terms: max(0,
// fl(fl(p m1) m2) - q) of the first rejected position, or the scaled target row fl(fl(p m1) m2) of the bonus position when every
// draft was accepted.  One launch, a workgroup per eight segments of the row: each finds the position for itself (one wave, a
// position a lane: less than a meeting would cost), makes the terms of its segments, leaves their sums, and when the row's workgroups are
// all there, their records; whoever comes last walks them, draws and writes the row's results.  The terms stay in registers; the
// walk makes those it needs again from p and q.
// What bounds it: the serial chain again (two trips for the position, the terms, a meeting, records, walk, search).  As four
// launches with the terms written and read back: 46 us for 16 rows of 262,144 and 8 drafts.
// The wait is bounded: a workgroup whose wait runs out marks the row and counts itself in, and whoever comes last adds all of the
// row's terms by its own.
// reject[row] = kSpecDone, or -1: the row is k_spec_verify's (other accept rules, a bonus token of a greedy row).
constexpr int kSpecT = 512;
constexpr int kSpecWaves = kSpecT / SR_WAVE;
// the exact running sum (or the search) over all segments from their terms, by one wave; the slow way of the rare cases
template <bool kSearch>
__device__ __forceinline__ float spec_sum_alone(const SpecTerms& t, int nseg, float target, int* found, float* states)
{
    float s = 0.0f;
    *found = -1;
    for (int sg = 0; sg < nseg; sg++) {
        float x[SR_SEQ_RUN];
        t.run(sg, x);
        int at;
        s = sr_seq_wave<SR_SEQ_RUN, kSearch>(x, s, target, &at);
        if (kSearch && at >= 0) {
            *found = sg * SR_SEG_TERMS + at;
            return s;
        }
        if (states && sr_lane() == 0) states[sg] = s;
    }
    return s;
}
// kFrom 1: k_spec_factor was launched in front   2: k_spec_open, which has found the position
template <int kFrom>
__global__ __launch_bounds__(kSpecT, 4) void k_spec_rows(SrSpecArgs a)
{
    __shared__ float4 turn_all[kSpecWaves][SR_WAVE * 5];
    __shared__ float states[SR_SEG_MAX];  // every segment's part of the sum, then the running sum behind every segment
    __shared__ uint32_t bc;
    __shared__ int said[2];
    __shared__ uint64_t tab[32];
    const int row = blockIdx.y, tid = threadIdx.x, lane = sr_lane(), wave = sr_wave_id();
    const SrRow rd = a.rows[row];
    const int n = a.vocab, L = a.n_draft, nseg = seg_count(n);
    unsigned long long* const sync = a.sync + (size_t)row * SR_ROW_SYNC_STRIDE;
    if (!spec_by_ratio(rd)) {
        if (blockIdx.x == 0 && tid == 0) a.reject[row] = -1;
        return;
    }
    const double* const u = a.uniforms + (size_t)row * a.uniforms_per_row;
    if (kFrom == 2) {
        if (tid == 0) {
            const unsigned long long picked = sync[kSpecPicked] & ~sync[kSpecAccepted], last = sync[kSpecLast];
            said[0] = picked != 0ull ? (int)__ffsll((long long)picked) - 1 : (int)(uint32_t)last;
            said[1] = (last & kSpecWritten) != 0ull ? 3 : picked == 0ull ? 2 : said[0] < L ? 0 : 1;
        } else if (tid == SR_WAVE) {
            const unsigned long long was = __hip_atomic_fetch_max(sync, (unsigned long long)a.seq << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("" : : "v"(was) : "memory");
        }
    } else if (wave == 0) {
        if (kFrom == 1) spec_table(tab);
        // the first position that is not accepted: kind 0 rejected, 1 none (position L), 2 an id outside the vocabulary, which
        // ends the row without a correction
        int pos = L, kind = 1;
        for (int i0 = 0; i0 < L; i0 += SR_WAVE) {
            const int i = i0 + lane;
            bool stop = false, bad = false;
            if (i < L) {
                const int tok = a.draft_tokens[(size_t)row * L + i];
                bad = (uint32_t)tok >= (uint32_t)n;
                if (!bad) {
                    const SrFullState* sl = a.state + (size_t)row * (L + 1) + i;
                    const float px = __fmul_rn(__fmul_rn(kFrom == 1 ? spec_e<false>(a, rd, (size_t)row * (L + 1) + i, tok, tab)
                                                            : a.p_all[((size_t)row * (L + 1) + i) * (size_t)a.p_stride + tok], sl->mul1), sl->mul2);
                    const float qx = a.draft_probs[((size_t)row * L + i) * n + tok];
                    const float acc = spec_accept(px, qx);
                    stop = !(u[i] < (double)acc);  // (every position before it was accepted and drew one uniform)
                }
            }
            const unsigned long long ends = __ballot(stop || bad);
            if (ends != 0ull) {
                const int l = (int)__ffsll((long long)ends) - 1;
                pos = i0 + l;
                kind = ((__ballot(bad) >> l) & 1ull) != 0ull ? 2 : 0;
                break;
            }
        }
        if (lane == 0) { said[0] = pos; said[1] = kind; }
    } else if (tid == SR_WAVE) {
        // (the number of the launch: nothing clears the words between launches)
        const unsigned long long was = __hip_atomic_fetch_max(sync, (unsigned long long)a.seq << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" : : "v"(was) : "memory");
    }
    __syncthreads();
    const int pos = said[0], kind = said[1];
    auto results = [&](int correction) __attribute__((always_inline)) {  // (by one wave)
        int* const out = a.out_tokens + (size_t)row * (L + 1);
        for (int i = lane; i <= L; i += SR_WAVE) out[i] = i < pos ? a.draft_tokens[(size_t)row * L + i] : i == pos ? correction : -1;
        if (lane == 0) {
            a.out_accepted[row] = pos;
            a.reject[row] = kSpecDone;
        }
    };
    if (kFrom == 2 && kind == 3) return;
    if (kind == 2) {
        if (blockIdx.x == 0 && wave == 0) results(-1);
        return;
    }
    if (kind == 1 && rd.temperature <= 0.0f) {  // (the bonus token of a greedy row: its argmax)
        if (blockIdx.x == 0 && tid == 0) a.reject[row] = -1;
        return;
    }
    SpecTerms t;
    t.p = a.p_all + ((size_t)row * (L + 1) + pos) * (size_t)a.p_stride;  // (k_spec_factor has seen to it that e is there)
    t.q = kind == 0 ? a.draft_probs + ((size_t)row * L + pos) * n : nullptr;
    {
        const SrFullState* sl = a.state + (size_t)row * (L + 1) + pos;
        t.m1 = sl->mul1;
        t.m2 = sl->mul2;
    }
    t.n = n;
    const int seg = (int)blockIdx.x * kSpecWaves + wave;
    SeqSegFunc* const funcs = a.seg_func + (size_t)row * a.seg_stride;
    float* const sums = a.seg_part + (size_t)row * a.seg_stride;
    float x[SR_SEQ_RUN];
    float own = 0.0f;
    if (seg < nseg) {
        float4 v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = t.four(seg * SR_SEG_TERMS + (k * SR_WAVE + lane) * 4);
        float4* const turn = turn_all[wave];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = (k * SR_WAVE + lane) * 4;
            own += (v[k].x + v[k].y) + (v[k].z + v[k].w);
            turn[(i >> 4) * 5 + ((i & 15) >> 2)] = v[k];
        }
        own = sr_wave_sum_f32(own);
        if (lane == 0) sr_store_agent(&sums[seg], own);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float4 w = turn[lane * 5 + k];
            x[4 * k] = w.x; x[4 * k + 1] = w.y; x[4 * k + 2] = w.z; x[4 * k + 3] = w.w;
        }
    }
    sr_drain_stores();
    __syncthreads();
    if (tid == 0) {
        const unsigned long long was = __hip_atomic_fetch_add(sync, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        uint32_t ok = ((uint32_t)was & 0xffffu) + 1u == gridDim.x ? 1u : 0u;
        for (uint32_t it = 0; ok == 0u && it < a.wait_limit; it++) {
            ok = ((uint32_t)sr_load_agent(sync) & 0xffffu) == gridDim.x ? 1u : 0u;
            if (ok == 0u) __builtin_amdgcn_s_sleep(1);
        }
        if (ok == 0u) sr_store_agent(sync + 1, (unsigned long long)a.seq);
        bc = ok;
    }
    __syncthreads();
    if (bc != 0u) {
        for (int g = tid; g < nseg; g += kSpecT) states[g] = sr_load_agent(&sums[g]);
        __syncthreads();
        if (seg < nseg) {
            float before = 0.0f;
            for (int g = lane; g < seg; g += SR_WAVE) before += states[g];
            before = sr_wave_sum_f32(before);
            seg_make_record<true>(x, seg, (double)before, funcs + seg, own);
        }
    }
    sr_drain_stores();
    __syncthreads();
    if (tid == 0) {
        const unsigned long long was = __hip_atomic_fetch_add(sync, 1ull << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        bc = ((uint32_t)(was >> 16) & 0xffffu) + 1u == gridDim.x ? (sr_load_agent(sync + 1) == (unsigned long long)a.seq ? 2u : 1u) : 0u;
    }
    __syncthreads();
    if (bc == 0u) return;
    const bool alone = bc == 2u;
    // (Not where neither launch stood in front, which takes smaller launches and rows that are cut: 16 x 8 of 50,257 under min-p 54.5
    // us with it and 53.8 without, of 20,011 that nothing touches 48.7 and 48.3, 64 x 4 of 32,768 under top-p 108.3 and 107.8, 1 x 2 of
    // 151,936 44.9 and 45.1.  16 x 8 of 262,144, one sequence under top-p, which has k_spec_factor in front: 231.3 and 231.7.)
    const bool staged = kFrom != 0 && stage_records<kSpecT>(funcs, nseg, &turn_all[0][0], (int)sizeof(turn_all));
    if (wave != 0) return;
    const double ud = u[kind == 0 ? pos + 1 : L];
    const float r = __double2float_rn(ud);
    auto load = [&](int sg, float (&xs)[SR_SEQ_RUN]) __attribute__((always_inline)) { t.run(sg, xs); };
    const SeqSegFunc* const near = (const SeqSegFunc*)&turn_all[0][0];
    int found;
    if (kind == 1) {
        // SampleFromDistribution (Sampler.cs:564-576) over the bonus position
        if (alone) spec_sum_alone<true>(t, nseg, r, &found, nullptr);
        else if (staged) seg_walk_from<true>(load, nseg, near, 0.0f, r, &found, nullptr);
        else seg_walk_from<true, true>(load, nseg, funcs, 0.0f, r, &found, nullptr);
        results(found >= 0 ? found : n - 1);
        return;
    }
    // ResampleResidual (Sampler.cs:587-618)
    int none;
    const float sum = alone ? spec_sum_alone<false>(t, nseg, 0.0f, &none, states) : staged ? seg_walk_from<false>(load, nseg, near, 0.0f, 0.0f, &none, states)
                            : seg_walk_from<false, true>(load, nseg, funcs, 0.0f, 0.0f, &none, states);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (!(sum > 0.0f)) {  // sum <= 0 or NaN: a draw from p
        t.q = nullptr;
        spec_sum_alone<true>(t, nseg, r, &found, nullptr);
        results(found >= 0 ? found : n - 1);
        return;
    }
    const float target = __fmul_rn(r, sum);
    float at_sum;
    found = target > 0.0f ? seg_search_states(load, nseg, states, target, &at_sum) : -1;
    if (found < 0) {
        // a zero target must not stop on a zero term: the first positive one; and where rounding left the sum of the search
        // short of the target, the last positive one
        int edge = target <= 0.0f ? 0x7fffffff : -1;
        for (int i = lane; i < n; i += SR_WAVE)
            if (t.at(i) > 0.0f) {
                edge = i;
                if (target <= 0.0f) break;
            }
        found = target <= 0.0f ? sr_wave_min_i32(edge) : -sr_wave_min_i32(-edge);
    }
    results(found);
}

// ---- speculative verification: the accept loop of StepSampled (SpeculativeDecoder.cs:530-559) ---------
// p_all holds the filtered target distributions of every position, [rows][n_draft + 1][n].
__global__ __launch_bounds__(kT) void k_spec_verify(SrSpecArgs a)
{
    __shared__ FullSmem sm;
    const int row = blockIdx.x;
    const SrRow rd = a.rows[row];
    const int n = a.vocab, L = a.n_draft;
    if (a.reject && a.reject[row] == kSpecDone) return;
    const float* pr = a.p_all + (size_t)row * (L + 1) * (size_t)a.p_stride;
    const float* lg = a.target_logits + (size_t)row * (L + 1) * n;
    const double* u = a.uniforms + (size_t)row * a.uniforms_per_row;
    int* out = a.out_tokens + (size_t)row * (L + 1);
    // SpeculativeDecoder.cs:192 and :538, :549 (`_trueSpecSampling && !usedPld`)
    const bool true_spec = spec_by_ratio(rd);
    for (int i = threadIdx.x; i <= L; i += kT) out[i] = -1;
    __syncthreads();
    int accepted = 0, udraws = 0, correction = -1;
    bool bad_id = false;
    // What the accept tests need of every position -- the draft token, its target and draft probabilities -- is
    // fetched for all positions at once: three dependent loads per position would otherwise line up one behind
    // the other along the walk.
    constexpr int kStage = 1024;
    const bool staged = L <= kStage;
    if (staged) {
        for (int i = (int)threadIdx.x; i < L; i += kT) {
            const int tok = a.draft_tokens[(size_t)row * L + i];
            const SrFullState* sl = a.state + (size_t)row * (L + 1) + i;
            const bool in_range = (uint32_t)tok < (uint32_t)n;  // an id outside the vocabulary is never dereferenced
            sm.sprob[i] = in_range ? __fmul_rn(__fmul_rn(pr[(size_t)i * (size_t)a.p_stride + tok], sl->mul1), sl->mul2) : 0.0f;
            sm.sprob[kStage + i] = (true_spec && in_range) ? a.draft_probs[((size_t)row * L + i) * n + tok] : 0.0f;
            sm.sprob[2 * kStage + i] = __int_as_float(tok);
        }
        for (int i = (int)threadIdx.x; i <= L && i < a.uniforms_per_row; i += kT)
            sm.sortbuf[i] = (unsigned long long)__double_as_longlong(u[i]);
        __syncthreads();
    }
    for (int i = 0; i < L; i++) {
        const float* pd = pr + (size_t)i * (size_t)a.p_stride;
        const float* qd = a.draft_probs + ((size_t)row * L + i) * n;
        const int tok = staged ? __float_as_int(sm.sprob[2 * kStage + i]) : a.draft_tokens[(size_t)row * L + i];
        const SrFullState* sl = a.state + (size_t)row * (L + 1) + i;
        // The managed loop indexes pDist[x_i] (SpeculativeDecoder.cs:536) and throws on an id outside the
        // vocabulary: the row ends here, with -1 where its correction token would stand.
        if ((uint32_t)tok >= (uint32_t)n) { bad_id = true; break; }
        const float px = staged ? sm.sprob[i] : __fmul_rn(__fmul_rn(pd[tok], sl->mul1), sl->mul2);
        bool accept;
        if (true_spec) {
            const float qx = staged ? sm.sprob[kStage + i] : qd[tok];
            const float acc = spec_accept(px, qx);
            const double ui = staged ? __longlong_as_double((long long)sm.sortbuf[udraws]) : u[udraws];
            udraws++;
            accept = ui < (double)acc;
        } else {
            accept = px >= rd.p_min;
            if (!accept) accept = tok == row_argmax(lg + (size_t)i * n, n, sm);  // block-uniform branch
        }
        if (accept) {
            if (threadIdx.x == 0) out[accepted] = tok;
            accepted++;
            continue;
        }
        const float m1 = sl->mul1, m2 = sl->mul2;
        const double uc = u[udraws++];
        if (true_spec && a.reject && a.reject[row] == i)  // the residual row is there already
            correction = resample_residual_stored(a.resid + (size_t)row * (size_t)a.resid_stride, pd, n, uc, sm, m1, m2);
        else
            correction = true_spec ? resample_residual_row(pd, qd, n, uc, sm, m1, m2) : draw_from_row(pd, n, uc, sm, m1, m2);
        break;
    }
    if (correction < 0 && !bad_id) {
        // every draft accepted: bonus token from the last position (greedy rows: its argmax, no draw)
        const float* pd = pr + (size_t)L * (size_t)a.p_stride;
        const SrFullState* sl = a.state + (size_t)row * (L + 1) + L;
        if (rd.temperature <= 0.0f) correction = row_argmax(pd, n, sm);
        else correction = draw_from_row(pd, n, u[udraws++], sm, sl->mul1, sl->mul2);
    }
    if (threadIdx.x == 0) {
        out[accepted] = correction;
        a.out_accepted[row] = accepted;
    }
}

// ---- MtpDecoder.AcceptDraft / SoftmaxProbAt (MtpDecoder.cs:562-596) ------------------------------------
__global__ __launch_bounds__(kT) void k_mtp_verify(const float* logits, int64_t stride, int n, const int* draft,
                                                    float p_min, int* out_argmax, int* out_accept, float* out_prob)
{
    __shared__ FullSmem sm;
    __shared__ double dred[kW];
    const int row = blockIdx.x;
    const float* l = logits + (size_t)row * stride;
    const int am = row_argmax(l, n, sm);
    const int d = draft[row];
    float prob = 0.0f;
    int ok = d == am ? 1 : 0;
    if (!ok && p_min < 1.0f) {
        // max, sum of exp(l - max) in double, ratio cast to float.  The double sum is a tree reduction:
        // it can differ from the reference's left-to-right double sum in the last bits, far below the
        // float result's 1e-5 tolerance.
        float m = l[0];
        for (int i = threadIdx.x; i < n; i += kT) m = fmaxf(m, l[i]);
        bool nn;
        m = blk_max_f(m, &nn, sm);
        double s = 0.0;
        for (int i = threadIdx.x; i < n; i += kT) s += exp((double)__fsub_rn(l[i], m));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        __syncthreads();
        if (sr_lane() == 0) dred[sr_wave_id()] = s;
        __syncthreads();
        double tot = 0.0;
        for (int w = 0; w < kW; w++) tot += dred[w];
        if (tot > 0.0 && d >= 0 && d < n) prob = (float)(exp((double)__fsub_rn(l[d], m)) / tot);
        ok = prob >= p_min ? 1 : 0;
    }
    if (threadIdx.x == 0) {
        out_argmax[row] = am;
        out_accept[row] = ok;
        if (out_prob) out_prob[row] = prob;
    }
}

#ifdef SR_TEST_HOOKS
// The record of every segment of every row of terms (SeqSegFunc), for the binades that the approximate sums predict:
// the sums of the segments in front (part, left by the kernel that wrote the terms) and, inside the segment, of the
// lanes in front.  One wave per segment.
__global__ __launch_bounds__(256) void k_seq_funcs(const float* terms, int64_t stride, int n, const double* part, SeqSegFunc* func,
                                                   int seg_stride)
{
    const int row = blockIdx.y, lane = sr_lane();
    const int seg = (int)blockIdx.x * 4 + sr_wave_id();
    if (seg >= seg_count(n)) return;
    const double* pr = part + (size_t)row * seg_stride;
    double before = 0.0;
    for (int g = lane; g < seg; g += SR_WAVE) before += pr[g];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o);
    const float* t = terms + (size_t)row * (size_t)stride;
    float x[SR_SEQ_RUN];
    seq_load_run(t, ((uintptr_t)t & 15u) == 0u, seg * SR_SEG_TERMS + lane * SR_SEQ_RUN, n, x);
    seg_make_record(x, seg, before, func + (size_t)row * seg_stride + seg);
}

__global__ __launch_bounds__(kT) void k_selftest_seqsum(const float* x, int n, float s0, float target, float* out_sum,
                                                         int* out_idx)
{
    __shared__ FullSmem sm;
    int found;
    float s;
    if (target == target)
        s = seq_sum_row<true>(x, n, s0, target, &found, sm);
    else
        s = seq_sum_row<false>(x, n, s0, 0.0f, &found, sm);
    if (threadIdx.x == 0) { *out_sum = s; *out_idx = found; }
}
// The same sum the prepared way: approximate sums of the segments (times `skew`, to make the predictions miss), the
// segments' records, and the walk of one wave -- the sum with the states it leaves and the search from those states
// (out[0], idx[0]), and the walk that searches by itself (out[1], idx[1]).
__global__ __launch_bounds__(256) void k_selftest_segpart(const float* x, int n, double skew, double* part)
{
    const int seg = (int)blockIdx.x * 4 + sr_wave_id(), lane = sr_lane();
    if (seg >= seg_count(n)) return;
    double acc = 0.0;
    for (int j = 0; j < SR_SEQ_RUN; j++) {
        const int i = seg * SR_SEG_TERMS + lane * SR_SEQ_RUN + j;
        if (i < n) acc += (double)x[i];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if (lane == 0) part[seg] = acc * skew;
}
__global__ __launch_bounds__(kT) void k_selftest_segwalk(const float* x, int n, const SeqSegFunc* funcs, float target, float* out_sum,
                                                          int* out_idx)
{
    __shared__ FullSmem sm;
    if (sr_wave_id() != 0) return;
    int found = -1, found2 = -1;
    const float s = seg_walk<false>(x, n, funcs, 0.0f, 0.0f, &found, sm.segst);
    float s2 = s;
    if (target == target) {
        float at = 0.0f;
        found = seg_search_states([&](int seg, float (&v)[SR_SEQ_RUN]) {
            seq_load_run(x, ((uintptr_t)x & 15u) == 0u, seg * SR_SEG_TERMS + sr_lane() * SR_SEQ_RUN, n, v);
        }, seg_count(n), sm.segst, target, &at);
        s2 = seg_walk<true>(x, n, funcs, 0.0f, target, &found2, nullptr);
    }
    if (sr_lane() == 0) { out_sum[0] = s; out_sum[1] = s2; out_idx[0] = found; out_idx[1] = found2; }
}
#endif

}  // namespace

hipError_t sr_launch_full_prep(const SrFullArgs& a, int n_rows, hipStream_t st)
{
    if (n_rows <= 0) return hipSuccess;
    const int bx = max(1, min(64, (a.vocab + 256 * 16 - 1) / (256 * 16)));
    dim3 grid(bx, n_rows);
    // (the adjusted copy only where some row keeps one: the host knows)
    if (a.dtype == 1) {
        if (a.any_copy) hipLaunchKernelGGL(k_full_prep<2>, grid, dim3(256), 0, st, a);
        if (a.any_edits) hipLaunchKernelGGL(k_full_edits<2>, dim3(n_rows), dim3(256), 0, st, a);
    } else {
        if (a.any_copy) hipLaunchKernelGGL(k_full_prep<4>, grid, dim3(256), 0, st, a);
        if (a.any_edits) hipLaunchKernelGGL(k_full_edits<4>, dim3(n_rows), dim3(256), 0, st, a);
    }
    if (a.seg_func) {
        const int nseg = (a.vocab + SR_SEG_TERMS - 1) / SR_SEG_TERMS;
        // A wave takes one segment, or two where the launch's sampled rows have more segments than half of the device's waves:
        // the workgroups of a row wait for each other between the passes, and fewer of them wait less (16 rows of 262,144
        // fp32: 33 -> 26 us, 64 of 151,936: 55 -> 36).  Below, one and two measure the same, and one starts sooner (a row
        // of 151,936, whole step: 56.6 against 58.9 us).  Four for the verifier's large launches, whose waves keep nothing
        // else in registers (144 rows of 262,144: 98 -> 92 us; 36 rows: 119.6 -> 121.6 a call).
        const long long segs = (long long)(a.n_sampled + a.n_greedy) * nseg;
        const bool four = a.factor_later || (a.lazy_scale && a.dtype != 1 && segs > 12288), two = segs > 3072;
        // ... and four where they take fewer turns of workgroups (five to a compute unit; with two segments a wave six), and where
        // these are the last, or the rows so long that what their last workgroup has too many is little.  Two and four, us: one turn for
        // two, 64 rows of 262,144 fp32 67 and 58 (bf16 68 and 55; cut by nothing or by top-p 110 and 100), 64 of 200,003 57.5 and 54, 96
        // of 151,936 59 and 55.5, 128 64 and 62; more turns, 128 of 262,144 114 and 103 (bf16 114 and 94), 256 214 and 196 (212 and 173),
        // 160 of 200,003 104 and 100.5 (100 and 90), 256 166 both (160 and 145).  As many turns, 64 of 151,936 42 and 50, 160 74 and 85, 96
        // of 262,144 85 and 88 (83 and 78).  Shorter rows, 192 of 151,936 91 and 94, 256 121 and 118, 256 of 131,073 99 and 105,
        // 256 of 100,003 83 and 91, 128 54 both, 200 of 65,537 55 and 56.5.
        const long long sampled = a.n_sampled + a.n_greedy, at_two = 6 * std::max(a.cu_count, 1), at_four = 5 * std::max(a.cu_count, 1);
        const long long turns_two = (sampled * ((nseg + 7) / 8) + at_two - 1) / at_two, turns_four = (sampled * ((nseg + 15) / 16) + at_four - 1) / at_four;
        const bool big = !a.lazy_scale && turns_four < turns_two && (nseg >= 192 || (nseg >= 128 && turns_four == 1));
        const int per_group = 4 * (four || big ? 4 : two ? 2 : 1);
        dim3 fgrid((unsigned)((nseg + per_group - 1) / per_group), n_rows + a.n_greedy);
        if (a.dtype == 1) {
            if (big && !a.prepared) hipLaunchKernelGGL((k_full_softmax_seg<2, 4, 4, false, 4, true>), fgrid, dim3(256), 0, st, a);
            else if (big) hipLaunchKernelGGL((k_full_softmax_seg<2, 4, 4, false, 8, true>), fgrid, dim3(256), 0, st, a);
            else if (!a.prepared && two) hipLaunchKernelGGL((k_full_softmax_seg<2, 4, 2, false, 4>), fgrid, dim3(256), 0, st, a);
            else if (!a.prepared) hipLaunchKernelGGL((k_full_softmax_seg<2, 4, 1, false, 4>), fgrid, dim3(256), 0, st, a);
            else if (two) hipLaunchKernelGGL((k_full_softmax_seg<2, 4, 2>), fgrid, dim3(256), 0, st, a);
            else hipLaunchKernelGGL((k_full_softmax_seg<2, 4, 1>), fgrid, dim3(256), 0, st, a);
        } else {
            if (a.factor_later) hipLaunchKernelGGL((k_full_softmax_seg<4, 4, 4, true>), fgrid, dim3(256), 0, st, a);
            else if (big) hipLaunchKernelGGL((k_full_softmax_seg<4, 4, 4, false, 4, true>), fgrid, dim3(256), 0, st, a);
            else if (four) hipLaunchKernelGGL((k_full_softmax_seg<4, 4, 4>), fgrid, dim3(256), 0, st, a);
            else if (two) hipLaunchKernelGGL((k_full_softmax_seg<4, 4, 2>), fgrid, dim3(256), 0, st, a);
            else hipLaunchKernelGGL((k_full_softmax_seg<4, 4, 1>), fgrid, dim3(256), 0, st, a);
        }
    } else if (a.dtype == 1) {
        hipLaunchKernelGGL(k_full_max<2>, grid, dim3(256), 0, st, a);
        hipLaunchKernelGGL(k_full_exp<2>, grid, dim3(256), 0, st, a);
    } else {
        hipLaunchKernelGGL(k_full_max<4>, grid, dim3(256), 0, st, a);
        hipLaunchKernelGGL(k_full_exp<4>, grid, dim3(256), 0, st, a);
    }
    return hipGetLastError();
}
hipError_t sr_launch_wide_keys(const SrFullArgs& a, int n_rows, hipStream_t st)
{
    if (n_rows <= 0) return hipSuccess;
    dim3 grid(max(1, min(64, (a.vocab + 256 * 16 - 1) / (256 * 16))), n_rows);
    if (a.dtype == 1) hipLaunchKernelGGL(k_wide_keys<2>, grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(k_wide_keys<4>, grid, dim3(256), 0, st, a);
    return hipGetLastError();
}
hipError_t sr_launch_wide_adjust(const SrFullArgs& a, int n_rows, hipStream_t st)
{
    if (n_rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_wide_adjust, dim3(32, n_rows), dim3(256), 0, st, a);
    return hipGetLastError();
}
hipError_t sr_launch_wide_sort(const SrFullArgs& a, int n_rows, int first, hipStream_t st)
{
    hipLaunchKernelGGL(k_wide_sort, dim3((unsigned)n_rows), dim3(kT), 0, st, a, first);
    return hipGetLastError();
}
hipError_t sr_launch_wide_tail(const SrFullArgs& a, int n_rows, hipStream_t st)
{
    if (n_rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_wide_tail, dim3(n_rows), dim3(kT), 0, st, a);
    return hipGetLastError();
}
hipError_t sr_launch_full_row(const SrFullArgs& a, int n_rows, hipStream_t st)
{
    if (n_rows <= 0) return hipSuccess;
    // (longer lists of candidates, slabs of twice the size: see cut_from_list and nucleus_from_histogram)
    static_assert((SR_LIST_CAP_BIG + SR_LIST_CAP_BIG / 16) * 4 >= 16 * kSmall, "room for the slabs as well");
    const unsigned more = a.big_slabs ? (unsigned)((SR_LIST_CAP_BIG + SR_LIST_CAP_BIG / 16) * 4) : 0u;
    if (more) {
        static bool allowed[64] = {};  // (once per device)
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        if (dev < 0 || dev >= 64 || !allowed[dev]) {
            for (const void* k : {(const void*)k_full_row<false>, (const void*)k_full_row<true>}) {
                e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)more);
                if (e != hipSuccess) return e;
            }
            if (dev >= 0 && dev < 64) allowed[dev] = true;
        }
    }
    if (a.factor_later) hipLaunchKernelGGL(k_full_row<true>, dim3(n_rows), dim3(kT), more, st, a);
    else hipLaunchKernelGGL(k_full_row<false>, dim3(n_rows), dim3(kT), more, st, a);
    if (a.prepared) {
        const int nseg = (a.vocab + SR_SEG_TERMS - 1) / SR_SEG_TERMS;
        const dim3 grid((unsigned)((nseg + SR_SEQ_CHAINS - 1) / SR_SEQ_CHAINS), n_rows);
        if (a.behind_twice) {
            hipLaunchKernelGGL(k_prepared_row<1>, grid, dim3(kPrepT), 0, st, a);
            hipLaunchKernelGGL(k_prepared_row<2>, grid, dim3(kPrepT), 0, st, a);
        } else {
            hipLaunchKernelGGL(k_prepared_row<0>, grid, dim3(kPrepT), 0, st, a);
        }
    }
    return hipGetLastError();
}
hipError_t sr_launch_draw_rows(const float* probs, int64_t stride, int n, int rows, const double* u, int* out,
                               hipStream_t st)
{
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_draw_rows, dim3(rows), dim3(kT), 0, st, probs, stride, n, u, out);
    return hipGetLastError();
}
hipError_t sr_launch_residual_rows(const float* p, int64_t ps, const float* q, int64_t qs, int n, int rows,
                                   const double* u, int* out, hipStream_t st)
{
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_residual_rows, dim3(rows), dim3(kT), 0, st, p, ps, q, qs, n, u, out);
    return hipGetLastError();
}
hipError_t sr_launch_expand_rows(const SrRow* src, SrRow* dst, int rows, int positions, hipStream_t st)
{
    if (rows <= 0 || positions <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_expand_rows, dim3((unsigned)((rows * positions + 255) / 256)), dim3(256), 0, st, src, dst, rows, positions);
    return hipGetLastError();
}
static int seg_count_of(int n) { return (n + SR_SEG_TERMS - 1) / SR_SEG_TERMS; }
hipError_t sr_launch_spec_verify(const SrSpecArgs& a, int rows, hipStream_t st)
{
    if (rows <= 0) return hipSuccess;
    SrSpecArgs b = a;
    if (!(b.reject && b.n_draft > 0 && b.draft_probs && rows <= 65535)) {  // (rows are the grid's second dimension)
        b.resid = nullptr;
        b.reject = nullptr;
    } else if (b.seg_func) {
        const dim3 grid((unsigned)((seg_count_of(b.vocab) + kSpecWaves - 1) / kSpecWaves), rows);
        static_assert(kSpecWaves == SR_SEQ_CHAINS && kSpecT == kPrepT, "the same blocks of a row");
        b.open_factors = nullptr;
        if (a.all_open) {
            const dim3 open_grid(grid.x, grid.y, (unsigned)b.open_side);
            hipLaunchKernelGGL(k_spec_units, dim3((unsigned)((b.n_units + 3) / 4), rows * (b.n_draft + 1)), dim3(256), 0, st, *a.open_factors, b);
            if (b.n_units <= kUnitsFew * SR_WAVE) hipLaunchKernelGGL(k_spec_open<kUnitsFew>, open_grid, dim3(kPrepT), 0, st, *a.open_factors, b);
            else hipLaunchKernelGGL(k_spec_open<kUnitsMost>, open_grid, dim3(kPrepT), 0, st, *a.open_factors, b);
            hipLaunchKernelGGL(k_spec_rows<2>, grid, dim3(kSpecT), 0, st, b);
        } else if (a.open_factors) {
            hipLaunchKernelGGL(k_spec_factor, grid, dim3(kPrepT), 0, st, *a.open_factors, b);
            hipLaunchKernelGGL(k_spec_rows<1>, grid, dim3(kSpecT), 0, st, b);
        } else {
            hipLaunchKernelGGL(k_spec_rows<0>, grid, dim3(kSpecT), 0, st, b);
        }
        if (!b.any_other) return hipGetLastError();
    } else {
        const int nseg = seg_count_of(b.vocab);
        hipLaunchKernelGGL(k_spec_walk, dim3(rows), dim3(SR_WAVE), 0, st, b);
        hipLaunchKernelGGL(k_spec_residual, dim3((unsigned)std::min(64, (nseg + 3) / 4), rows), dim3(256), 0, st, b);
    }
    hipLaunchKernelGGL(k_spec_verify, dim3(rows), dim3(kT), 0, st, b);
    return hipGetLastError();
}
hipError_t sr_launch_mtp_verify(const float* logits, int64_t stride, int n, int rows, const int* draft, float p_min,
                                int* out_argmax, int* out_accept, float* out_prob, hipStream_t st)
{
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_mtp_verify, dim3(rows), dim3(kT), 0, st, logits, stride, n, draft, p_min, out_argmax,
                       out_accept, out_prob);
    return hipGetLastError();
}
#ifdef SR_TEST_HOOKS
hipError_t sr_launch_selftest_seqsum(const float* x, int n, float s0, float target, float* out_sum, int* out_idx,
                                     hipStream_t st)
{
    hipLaunchKernelGGL(k_selftest_seqsum, dim3(1), dim3(kT), 0, st, x, n, s0, target, out_sum, out_idx);
    return hipGetLastError();
}
hipError_t sr_launch_selftest_segsum(const float* x, int n, double skew, float target, double* part, SeqSegFunc* funcs,
                                     float* out_sum, int* out_idx, hipStream_t st)
{
    const int nseg = (n + SR_SEG_TERMS - 1) / SR_SEG_TERMS;
    hipLaunchKernelGGL(k_selftest_segpart, dim3((unsigned)((nseg + 3) / 4)), dim3(256), 0, st, x, n, skew, part);
    hipLaunchKernelGGL(k_seq_funcs, dim3((unsigned)((nseg + 3) / 4), 1), dim3(256), 0, st, x, (int64_t)0, n, part, funcs, nseg);
    hipLaunchKernelGGL(k_selftest_segwalk, dim3(1), dim3(kT), 0, st, x, n, funcs, target, out_sum, out_idx);
    return hipGetLastError();
}
#endif
