// Kernel argument blocks and host-callable launchers (one per .hip file).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "sr_types.h"

// out_flags bits written by the kernels; identical to SR_OUT_* of the public header
#define SR_KFLAG_GREEDY (1u << 0)
#define SR_KFLAG_TOPK (1u << 1)
#define SR_KFLAG_FULL (1u << 2)
#define SR_KFLAG_DEGENERATE (1u << 3)
#define SR_KFLAG_AMBIGUOUS (1u << 4)
#define SR_KFLAG_UNSUPPORTED (1u << 31)
// the public bits of SrRow.flags as device code sees them (the public header is not included on the device side)
#define SR_ROWBIT_HAS_LOGIT_BIAS (1u << 0)
#define SR_ROWBIT_DRAFT_FROM_LOOKUP (1u << 1)
// internal bit of SrRow.flags: the row has a history and at least one active penalty
#define SR_ROWFLAG_HAS_PENALTY (1u << 8)
// internal bit: the penalties can only lower a logit, so the scan skips the history ids (scan mask) and
// the row tail fetches their logits by id instead of over-selecting by the history length
#define SR_ROWFLAG_HIST_EXCL (1u << 9)
// the row's edits are sorted by id (else they stand in order of first appearance in the history)
#define SR_ROWFLAG_EDITS_SORTED (1u << 10)

// A sampled full-vocabulary row that keeps no adjusted copy of its logits although bias or penalties touch some ids
// (host and device agree on this: the host provides the rows' tables when a batch holds such a row).
#define SR_FULL_EDIT_VALUES 2048
static inline __host__ __device__ bool sr_row_edits_on_the_fly(const SrRow& rd, int)
{
    return rd.temperature > 0.0f && rd.edit_cnt > 0 && rd.edit_cnt <= SR_FULL_EDIT_VALUES;
}

// min-p or top-p cuts the row
static inline __host__ __device__ bool sr_row_cut(const SrRow& rd) { return rd.min_p > 0.0f || (rd.top_p < 1.0f && rd.top_p > 0.0f); }

#define SR_TK_MAX_XCD 16
struct SrTopkArgs {
    const void* logits;
    int64_t row_stride;      // elements
    int32_t vocab;
    int32_t dtype;           // 0 = f32, 1 = bf16
    int32_t chunks;          // chunk items per row
    int32_t n_rows;          // rows in this launch
    int32_t chunk_vecs;      // 16-byte vectors per chunk, a multiple of 64
    // Workgroup b runs the program progs[b] = (first item, number of items, launch slot of the row it finishes at
    // the end or -1, 1 when its items are exactly that row's chunks): it streams items[first .. first + n) in order.  An item is x = bits 24..30 chunk |
    // bits 0..23 launch slot of the row, y = batch row, z = scan-mask row, w = sel.
    const int4* items;
    const int4* progs;
    int32_t n_workers, n_items;
    int32_t cu_count;        // compute units of the device
    int32_t own_rows;        // every worker's program is one whole row (all its chunks, then its tail)
    uint32_t start_gap;      // ticks of the 100 MHz clock that every compute unit's second worker starts behind its first (0: none)
    int32_t short_lists;     // no row of the launch asks for more than SR_TK_SHORT_SEL entries
    const int32_t* sel_list; // [n_rows] batch row of every launch slot
    const SrRow* rows;
    const SrEdit* edits;
    const uint32_t* mask;
    int64_t mask_stride;     // words
    const uint32_t* scan_mask; // keep-bits of every row in the kernel's access order (SrRow.scan_row)
    int64_t scan_stride;     // 32-bit words per scan row: chunks x threads x SR_TK_MASK_WORDS
    float4* gmax;            // [n_rows][chunks][SR_TK_THREADS]: the four group maxima of every thread of every chunk
    float4* gmax2;           // ... the second largest element of each of those groups
    uint32_t* gpos;          // ... the position of the largest inside its group, 8 bits per group
    uint32_t* gbound;        // [n_rows][chunks][waves][2]: every chunk wave's share of the row's bound and its largest kept
                             // element (ordered keys)
    unsigned long long* cand; // [n_rows][SR_TK_ROW_CAP] (value bits << 32 | index), built by the row's tail
    // Counters, two sets of done_cap entries: a launch counts the chunks of slot s in row_done[parity * done_cap + s]
    // and clears the other set for the launch after it, so that whatever a launch leaves behind never reaches a
    // later one.
    uint32_t* row_done;
    uint32_t done_cap;
    uint32_t parity;
    uint32_t spin_limit;     // polls of a row's counter before its tail stops waiting and selects from the logits alone
    const double* uniforms;
    int32_t uniforms_per_row;
    int32_t* out_tokens;
    uint32_t* out_flags;     // may be null
    unsigned long long* prof; // phase timestamps [chunk items + rows][16] in profiling builds, else unused
};
hipError_t sr_launch_topk(const SrTopkArgs& a, int n_rows, hipStream_t stream);
// Builds scan row i for descs[i]; base_addr / stride_bytes are those of the logits the mask is used with
// (they decide where a row starts inside its first 16-byte vector), epv = 4 (fp32) or 8 (bf16).
// all pieces of an upload in one launch: segs (itself in pinned host memory) lists n pieces
hipError_t sr_launch_scatter(const SrCopyTable& t, hipStream_t stream);
// scan_ids: the n_scan scan rows to build (NULL: rows 0 .. n_scan - 1)
hipError_t sr_launch_pack_allow_mask(const void* logits, int dtype, int rows, int vocab, int64_t row_stride, uint32_t* out,
                                     int64_t out_stride, hipStream_t stream);
// AND of the n (<= SR_MASK_AND_MAX) registered masks ids_host[] into slot dst of the pool; *any (zero before) becomes 1
// when a bit inside the vocabulary is left
#define SR_MASK_AND_MAX 8
hipError_t sr_launch_mask_and(uint32_t* pool, int64_t pool_words, const int32_t* ids_host, int n, int dst, int vocab, uint32_t* any,
                              hipStream_t stream);
// pieces: when not null, the pieces of an upload are put in their places by further workgroups of the same launch (descs, rows
// and edits are then where the host packed them)
hipError_t sr_launch_build_scan_mask(const SrScanDesc* descs, const int32_t* scan_ids, int n_scan, const SrRow* rows, const SrEdit* edits,
                                     const uint32_t* mask, int64_t mask_stride, uint32_t* scan_mask, int64_t scan_stride,
                                     int vocab, int epv, int chunks, int chunk_vecs, unsigned long long base_addr,
                                     long long stride_bytes, const SrCopyTable* pieces, hipStream_t stream);

// What one appended token per row changes (sr_batch_append_tokens): history length and edit count of n_rowp rows,
// n_edits whole edits, n_clears keep-bits of scan masks built with the given geometry.  The lists may lie in pinned host memory.
hipError_t sr_launch_apply_patches(SrRow* rows, const SrRowPatch* rp, int n_rowp, SrEdit* edits, const SrEditPatch* ep,
                                   int n_edits, const SrMaskClear* mc, int n_clears, uint32_t* scan_mask,
                                   int64_t scan_stride, int epv, int chunk_vecs, unsigned long long base_addr,
                                   long long stride_bytes, hipStream_t stream);

struct SrArgmaxArgs {
    const void* logits;
    int64_t row_stride;
    int32_t vocab;
    int32_t dtype;
    int32_t rows;
    int32_t chunks;           // workgroups per row
    int32_t chunk_len;        // elements per chunk, a multiple of the elements of a 16-byte vector
    int32_t vec;              // rows start on 16-byte boundaries: 16-byte loads
    // rows of more than one chunk: [rows] packed (key << 32 | ~idx) and [rows] chunks counted in; both zero before
    // the launch and zero again after it
    unsigned long long* best;
    uint32_t* done;
    int32_t* out_idx;         // may be null
    float* out_val;           // may be null
    unsigned long long* host; // pinned host memory, or null: value bits << 32 | index of every row
};
// fills chunks, chunk_len and vec from the other fields
void sr_argmax_plan(SrArgmaxArgs& a, int cu_count);
// clear_first: best and done may hold anything (a fill precedes the kernel)
hipError_t sr_launch_argmax_rows(const SrArgmaxArgs& a, bool clear_first, hipStream_t stream);
// the current device's copy of the scratch that belongs to the library's code object: SR_ARGMAX_STATIC_ROWS rows
hipError_t sr_argmax_static_scratch(int device, unsigned long long** best, uint32_t** done);

hipError_t sr_launch_selftest_expf(const float* x, float* y, int64_t n, hipStream_t stream);

// ---- full-vocabulary path (sr_full.hip) ---------------------------------------------------------------
struct SrFullState {
    // launch number << 32 | ordered key of the row's largest adjusted logit (0xffffffff = the row holds a NaN; 0 = none
    // yet); short and very long rows raise it with 64-bit atomic maxima: what an earlier launch left is below anything of the
    // present one, so the word needs no clearing between launches
    unsigned long long maxkey;
    uint32_t flags;
    int32_t n_survivors;  // entries with probability > 0 when top-p starts
    float mul1, mul2;     // the row's entries are to be multiplied by these two, in this order (1 unless lazy_scale)
    uint32_t late;        // the number of the last launch in which a workgroup of the row stopped waiting at a meeting point
    uint32_t deferred;    // the number of the last launch that left the row's normalisation and draw to the whole device
    float ycut;           // ... whose members are the probabilities above ycut, and of those equal to it the ones up to idx_last
    int32_t idx_last;
    uint32_t list_from;   // the row's list of candidates holds its e from this value on (as bits); 0: it would have been too long
    uint32_t late_behind; // the number of the last launch in which a workgroup of k_prepared_row stopped waiting for the row's others
    float u;              // the uniform of the draw, of a row left to the whole device
    uint32_t e_open;      // the number of the last launch that did not write the row's e down: its reader takes it from the logits
    uint32_t decided;     // the number of the last launch in which k_full_softmax_seg found the row's token
    uint32_t drawn;       // ... in which k_full_row left the row to the whole device without its draw: of an uncut row that its largest entry
                          // decides (ycut < 0), or of one whose second factor is known as well (mul2)
};
static_assert(sizeof(SrFullState) == 64, "the 8-byte word, aligned, in front");
// SrFullArgs::row_sync, a word per row (rows 256 bytes apart: every workgroup of a row adds to its word and polls it):
// launch number << 32 | workgroups of a greedy row that have counted in.  The number is
// put in by an atomic maximum before the first count of a launch, so nothing clears the words.  The word behind it counts the
// workgroups of k_prepared_row the same way; k_full_row, which leaves the row to them, starts it.  The third one holds what the
// workgroups of a greedy row have found so far (zero between launches), the fourth one the factor that k_prepared_row's workgroups
// wait for, with the launch number above it; k_spec_open's wait for theirs there too, and the fifth and the sixth one count them in at
// their two meeting points (k_spec_units clears both).
#define SR_ROW_SYNC_STRIDE 32

struct SeqSegFunc;
struct SrFullArgs {
    const void* logits;
    int64_t row_stride;
    int32_t vocab;
    int32_t dtype;
    const int32_t* row_list;   // rows handled (device)
    const SrRow* rows;
    const SrEdit* edits;
    const uint32_t* mask;
    int64_t mask_stride;
    float* work;               // fp32 rows: [slot] or, with work_by_row, [row]
    int64_t work_stride;
    int32_t work_by_row;
    int32_t mode;              // 0 = sample, 1 = distribution only, 2 = distribution and sample
    int32_t lazy_scale;        // mode 1 only: rows that no filter touches keep expf(x - max); their two normalising
                               // factors go to state[slot].mul1 / mul2 for the reader to apply
    uint32_t* edit_tab;        // [slot][edit_tab_stride]: per row a bitmap of the ids its edits touch and one float per
    int64_t edit_tab_stride;   // edit (the adjusted value), for sampled rows that keep no adjusted copy; or null
    int32_t any_copy;          // some row keeps an adjusted copy of its logits (greedy rows, rows the table does not take)
    SrFullState* state;        // [slot]
    uint32_t* sort_keys_in;    // [slot][sort_stride]
    int32_t* sort_vals_in;
    int64_t sort_stride;       // entries per row segment in the sort buffers
    int32_t* wide_ids;         // [slot][sort_stride]: wide top-k rows, the token id of every place of the first order
    const double* uniforms;
    int32_t uniforms_per_row;
    int32_t* out_tokens;       // [row], may be null in mode 1
    uint32_t* out_flags;       // [row], may be null
    unsigned long long* prof;  // optional phase timestamps of slot 0 [32] (test hook), normally null
    // The softmax denominators prepared by the whole device (k_full_softmax_seg, seg_walk); seg_func is
    // null where the rows are added by their workgroups (fewer entries than SR_SEG_MIN_VOCAB, or more than SR_SEG_MAX segments).
    SeqSegFunc* seg_func;          // [slot][seg_stride]
    int32_t seg_stride;
    float* seg_sum;                // [slot][seg_stride] about the sum of every segment's e (of its members, in a row that is cut)
    float* chain_sum;              // [slot][chain_stride] ... of every half block's share of each of the eight lane accumulators
    int32_t chain_stride;
    int32_t chain_blocks;
    SeqSegFunc* chain_func;        // [slot][8][chain_blocks]
    float* mass;                   // [slot][256] the row's mass by size of e, or (the first) the length of its list; zero between launches
    uint32_t* seg_cnt;             // [slot][seg_stride] entries of every segment in the row's list (sort_keys_in, sort_vals_in)
    float* e_rows;                 // [slot][e_stride] expf(x - max) of the rows; starts on 16 bytes
    int64_t e_stride;
    int32_t prepared;              // the launches behind k_full_row follow: it may leave rows to the whole device
    int32_t factor_later;          // lazy_scale: mul2 of rows that nothing cuts is left to k_spec_factor, under the ratio test
    int32_t behind_twice;          // k_prepared_row as two launches, the second from the factor on
    int32_t finish_most;           // members up to which k_full_row normalises and draws by itself
    uint32_t seq;                  // the launch's number (never 0): see SrFullState::maxkey
    int32_t n_greedy;              // greedy rows behind the others in row_list, whose token k_full_softmax_seg finds (mode 0)
    int32_t cu_count;              // compute units of the device
    int32_t n_sampled;             // rows of the launch with a temperature above 0 (greedy rows leave the passes at once)
    int32_t any_edits;             // some row of the launch has edits for k_full_edits (else it is not launched)
    int32_t edits_in_pass;         // seg_func is set: sampled rows with up to SR_FULL_EDIT_VALUES edits keep no adjusted copy and
                                   // need no table either (k_full_softmax_seg applies their edits where it loads the row)
    unsigned long long* row_sync;  // [slot * SR_ROW_SYNC_STRIDE]
    // [slot * meet_stride] what k_full_softmax_seg's workgroups leave for each other, the launch's number << 32 above every word (so nothing
    // clears them between launches): a workgroup's largest logit as an ordered key and about the sum of its exponentials relative to that, and from
    // meet_sums on a segment's sum of e
    unsigned long long* meet;
    int32_t meet_stride, meet_sums;
    uint32_t row_wait_limit;       // polls of a row's count before a workgroup of k_full_softmax_seg stops waiting for it
    uint32_t behind_wait_limit;    // ... of k_prepared_row
    int32_t big_slabs;             // k_full_row gets 68 KB of shared memory more: lists of 16,384 candidates, slabs of 8,192 entries
};
hipError_t sr_launch_full_prep(const SrFullArgs& a, int n_rows, hipStream_t st);
hipError_t sr_launch_full_row(const SrFullArgs& a, int n_rows, hipStream_t st);
// SampleTopK by sorts of the whole row (rows beyond the selection kernel's limits): keys of the whole row, the row's
// sort by its own workgroup (first != 0) or that of its adjusted first `sel` entries, the adjustment, the walk over
// the sorted result
hipError_t sr_launch_wide_keys(const SrFullArgs& a, int n_rows, hipStream_t st);
hipError_t sr_launch_wide_adjust(const SrFullArgs& a, int n_rows, hipStream_t st);
hipError_t sr_launch_wide_sort(const SrFullArgs& a, int n_rows, int first, hipStream_t st);
hipError_t sr_launch_wide_tail(const SrFullArgs& a, int n_rows, hipStream_t st);
hipError_t sr_launch_draw_rows(const float* probs, int64_t stride, int n, int rows, const double* u, int* out,
                               hipStream_t st);
hipError_t sr_launch_residual_rows(const float* p, int64_t ps, const float* q, int64_t qs, int n, int rows,
                                   const double* u, int* out, hipStream_t st);

// One segment of SR_SEG_TERMS terms of a row whose exact sum the whole device prepares (seg_make_record, seg_walk in
// sr_full.hip): the increment function n -> n + a[n & 1] of its terms in the binade `eb` (sr_seqsum.h), and for a
// segment in which the running sum is expected to change binade once, inside the 16 terms of lane `cross`: the function
// of the terms in front of those 16 (a0, a1, eb), the 16 terms themselves, and the function of the terms behind them
// (b0, b1) in the binade eb2.  The row's first segment, whose start is known exactly, carries its exact end instead.
#define SR_SEG_PLAIN 0u
#define SR_SEG_EXACT 1u
#define SR_SEG_SPLIT 2u
#define SR_SEG_ZERO 3u   // no term above zero: no sum changes
struct SeqSegFunc {  // 96 bytes
    uint32_t a0, a1;
    int32_t eb;
    uint32_t kind;   // SR_SEG_* | cross << 8
    uint32_t b0, b1;
    int32_t eb2;
    uint32_t end_bits;  // SR_SEG_EXACT: the running sum behind the segment when the sum in front of it is +0
    float x[16];
};
struct SrSpecArgs {
    const SrRow* rows;
    int32_t vocab;
    int32_t n_draft;
    const float* p_all;          // [rows][n_draft + 1][p_stride] filtered target distributions, to be multiplied by ...
    int64_t p_stride;
    const SrFullState* state;    // ... mul1 and mul2 of [rows][n_draft + 1]
    const float* target_logits;  // [rows][n_draft + 1][vocab]
    const float* draft_probs;    // [rows][n_draft][vocab]
    const int32_t* draft_tokens; // [rows][n_draft]
    const double* uniforms;
    int32_t uniforms_per_row;
    int32_t* out_accepted;       // [rows]
    int32_t* out_tokens;         // [rows][n_draft + 1]
    int32_t* reject;             // [rows]: what k_spec_verify needs to know of the launches in front of it
    // rows of up to SR_SEG_MAX segments (k_spec_rows), else null:
    SeqSegFunc* seg_func;        // [rows][seg_stride]: the records of the segments of the terms that the row draws from
    float* seg_part;             // [rows][seg_stride]: about the sum of every segment of them
    int32_t seg_stride;
    unsigned long long* sync;    // [row * SR_ROW_SYNC_STRIDE]: as SrFullArgs::row_sync, and behind it the last launch in which a wait ran out
    uint32_t seq, wait_limit;
    // launches of which every row is one that nothing touches, under the ratio test (k_spec_units, k_spec_open):
    float2* units;               // [rows][n_draft + 1][n_units]: every unit's largest scaled logit (NaN: it holds one) and about its sum of exp(x - that)
    float* unit_chains;          // ... [8]: every lane accumulator's part of the sum
    int32_t n_units;
    int32_t open_side;           // positions of a row that k_spec_open takes side by side
    int32_t all_open;            // the launch is one of these: units are set, open_factors holds what k_spec_open needs
    const SrFullArgs* open_factors;  // on the host: the launch that left factors open (SrFullArgs::factor_later), or null; n_draft < 64
    int32_t any_other;           // some row is not under the ratio test, or greedy: k_spec_verify follows
    // ... and of more:
    float* resid;                // [rows][resid_stride]: max(0, p - q) of the row's first rejected position
    int64_t resid_stride;
};
hipError_t sr_launch_spec_verify(const SrSpecArgs& a, int rows, hipStream_t st);
hipError_t sr_launch_expand_rows(const SrRow* src, SrRow* dst, int rows, int positions, hipStream_t st);
hipError_t sr_launch_mtp_verify(const float* logits, int64_t stride, int n, int rows, const int* draft, float p_min,
                                int* out_argmax, int* out_accept, float* out_prob, hipStream_t st);
hipError_t sr_launch_selftest_seqsum(const float* x, int n, float s0, float target, float* out_sum, int* out_idx,
                                     hipStream_t st);
hipError_t sr_launch_selftest_segsum(const float* x, int n, double skew, float target, double* part, SeqSegFunc* funcs,
                                     float* out_sum, int* out_idx, hipStream_t st);
