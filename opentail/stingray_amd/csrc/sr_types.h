// Structures shared by the host packer and the kernels.
#pragma once
#include <stdint.h>

// How a row is dispatched; mirrors Sampler.Sample (Sampler.cs:17-39 of the reference engine).
enum SrPath : int32_t {
    SR_PATH_GREEDY = 0,      // Temperature <= 0, no history penalty      -> Greedy(masked logits)
    SR_PATH_GREEDY_PEN = 1,  // Temperature <= 0 with history penalties   -> GreedyWithHistoryPenalties
    SR_PATH_TOPK = 2,        // 0 < TopK < vocab and no logit bias        -> SampleTopK
    SR_PATH_FULL = 3,        // everything else                           -> full-vocabulary pipeline
    SR_PATH_TOPK_WIDE = 4    // SampleTopK beyond the selection kernel's limits -> device-wide sort of the row
};

struct SrRow {
    float temperature;
    float top_p;
    float min_p;
    float rep;
    float presence;
    float frequency;
    float p_min;
    int32_t top_k;
    int32_t sel;        // how many of the largest scanned logits the row needs (see the packer)
    int32_t path;       // SrPath
    int32_t edit_off;   // first SrEdit of this row
    int32_t edit_cnt;
    int32_t mask_row;   // row index into the allow-mask array, or -1
    int32_t n_prev;
    uint32_t flags;     // SR_ROW_* from the public header
    int32_t scan_row;   // row index into the scan-mask array (row edges, allow-mask, history ids)
};

// One distinct in-range token id that the row's history or logit bias touches; sorted by id per row where a kernel
// searches them (SR_ROWFLAG_EDITS_SORTED), else in order of first appearance in the history.
struct SrEdit {
    int32_t id;
    float bias;         // LogitBias value (applied first); valid when has_bias
    int32_t occ_win;    // occurrences inside the trailing repetition window
    int32_t occ_all;    // occurrences in the whole history
    float pen;          // powf(repetition_penalty, occ_win), computed with the host libm (1 when unused)
    uint32_t has_bias;
};

// One row of the scan-mask array of the selection kernel: which batch row it is built for, and from what.
struct SrScanDesc {
    int32_t row;
    uint32_t flags;
};
// What sr_batch_append_tokens sends to the device: an edit to be written at a position of the edit array, and a
// keep-bit of a scan-mask row to be cleared (the id entered the row's history).
struct SrEditPatch {
    int32_t index;
    SrEdit edit;
};
// one piece of an upload: bytes that lie in pinned host memory and belong at a device address
struct SrCopySeg {
    const void* src;
    void* dst;
    unsigned long long bytes;
};
// ... and all of them, in a kernel's arguments
#define SR_COPY_SEGS 12
struct SrCopyTable {
    int32_t n;
    int32_t pad;
    SrCopySeg seg[SR_COPY_SEGS];
};
struct SrRowPatch {
    int32_t row;
    int32_t n_prev;
    int32_t edit_cnt;
    int32_t mask_row;  // the row's allow-mask from now on (-1 none); rows of batches without registered masks keep theirs
    int32_t sel;
    int32_t edit_off;  // where the row's edits lie from now on (a row that ran out of room moves to the array's end)
};
struct SrMaskClear {
    int32_t scan_row;
    int32_t row;
    int32_t id;
};
#define SR_SCAN_ALLOW 1u  // start from the row's allow-mask
#define SR_SCAN_HIST 2u   // clear the row's history ids

// Limits of the top-k selection kernel.
#define SR_TK_THREADS 512
#define SR_TK_VEC 19                       // 16-byte vectors of fp32 logits held per thread
#define SR_TK_VEC_BF16 10                  // ... of bf16 logits: the same 40 thousand elements per workgroup
#define SR_ARGMAX_STATIC_ROWS 16384        // rows the argmax entry point that allocates nothing takes per call
#define SR_TK_WINDOW 5                     // ... of which a thread has in flight or in registers at a time
#define SR_TK_WINDOW_OWN 10                // ... when every worker streams one row of its own
#define SR_TK_WINDOW_KEPT 5                // ... and keeps the row's results in registers (the whole chunk in flight, 19, was the setting
                                           // while every chunk ended with a bound loop for the loads to hide; without those loops it
                                           // costs 1.3 us a launch at 256 rows: what is in flight beyond the window only queues.  1,024
                                           // rows of 151,936 fp32, two workers to a compute unit: 3 vectors 118.7 us, 4 115.6, 5 113.9, 7 113.8)
// Bytes that the compute units' first rows hold, over this: ticks of the 100 MHz clock in eight tenths of the time in which 6.8 TB/s
// bring them, after which the second workers start.  None, 0.5, 0.8 and 1.0 of it, us: 1,024 rows of 151,936 fp32 114.2, 109.4, 106.8,
// 107.2; 768 93.9, 82.0, 80.1, 83.4; 520 66.8, 62.5, 62.3, 65.0; 1,024 of bf16 69.4, 67.2, 66.4, 66.4; 600 of 49,152 fp32 40.0, 39.7, 38.2,
// 37.3; 1,024 of 16,384 39.7, 39.2, 38.9, 38.8.  Up to two workers to a compute unit it gains nothing: 512 rows 59.7 and 59.0, 384 50.7
// both, 320 47.6 and 48.0, 512 of bf16 38.8 and 39.5.  That workgroups cu_count ... 2 cu_count - 1 are the compute units' second ones holds
// only where the launch has the device to itself.  Beside another stream that is never idle the wait is lost time, none and 0.8, us a step and in
// brackets until both streams are through: four passes over 64 MB a step, 1,024 rows 183 and 182 (183 and 182), 768 143 and 153 (157 and
// 153), 520 122 and 132 (137 both); a 4,096^3 bf16 product a step, 198 and 202, 176 and 179, 155 and 161.  Beside three small kernels a step
// it gains what it gains alone (114 and 106, 94 and 81, 67 and 64).
#define SR_TK_START_GAP 85000.0
#define SR_TK_MASK_WORDS 3                 // 32-bit keep-words per chunk thread: 19 x 4 and 10 x 8 bits both fit 96
#define SR_TK_GROUPS 4                     // group maxima per thread
#define SR_TK_SHORT_SEL 64                 // a launch whose rows all ask for at most this many entries: see k_topk_rows
#define SR_TK_LONG_SEL 256                 // ... and one of which some row asks for more than this many: see topk_geometry
#define SR_TK_SEL_MAX 2048                 // most entries (candidates + history ids) the row tail sorts
#define SR_TK_ROW_CAP 8192                 // candidates all chunks of a row may hand to its tail (16 per thread)
#define SR_TK_KEPT_CHUNKS 8                 // most of a row whose results a worker keeps in registers, in pairs beyond four
#define SR_TK_MAX_CHUNKS 128               // most workgroups one row is split over

// Full-vocabulary path: nucleus candidates up to this count are sorted inside the row kernel.
#define SR_FULL_SMALL_CAP 4096
#define SR_SEG_TERMS 1024                  // terms per segment of a sum that the whole device prepares (64 lanes x 16)
#define SR_SEG_MIN_VOCAB 4096              // shorter rows are not worth the preparation
#define SR_UNIT_TERMS 2048                 // entries of a row whose largest and whose sum one wave of the verifier's first pass finds
#define SR_HALF_BLOCK_SEGS 4               // segments of a half block of the final Normalize's eight accumulators (4,096 entries)
// Which launches have a second one behind them (k_prepared_row) that spreads their long rows over the whole device.  A row's own
// workgroup costs about the same for one row and for 256; the launch behind it costs 10 to 20 us and what the rows hold
// together.  Measured both ways, us with it against without; sharp and flat are rows over N(0, 1.5^2) with a few large entries at
// top-p 0.9 and temperature 0.6, and at top-p 0.95 and temperature 1.5.
// Tokens of rows that nothing cuts: at every length.  16 rows of 4,608: 34 against 49, of 16,384: 37 against 48, of 49,152: 43
// against 64; 64 rows of 151,936: 91 against 122; 192 (28,608 segments): 199 against 197; 256: 266 against 251.  That only
// top-p cuts, where it finds nothing to do for sharp rows, and where a flat row's nucleus outgrows what its workgroup finishes by
// itself: 1, 16, 64 and 256 rows of 24,576 21, 23, 24, 36 against 20, 21, 22, 30 (sharp) and 81, 102, 110, 144 against 111, 196,
// 207, 231 (flat); of 28,672 21, 24, 25, 39 against 19, 21, 23, 34 and 74, 116, 129, 172 against 103, 225, 240, 267; of 20,480, where
// one flat row or four gain nothing, 21, 22, 24, 34 against 19, 20, 22, 29 and 69, 92, 101, 131 against 65, 151, 188, 211; of 16,384
// 23 against 21 and 76 against 72.  Both kinds of rows together, sharp and flat ones: 16 rows of 31,000 44 against 60 and 131
// against 250, of 20,480 41 against 49 and 103 against 183, of 16,384 40 against 52 and 92 against 73, of 8,192 37 against 57
// and 62 against 55; 256 rows of 31,000 84 against 76 and 251 against 285.
// Distributions: at every length.  16 rows of 4,608 37 against 51, cut by top-p 32 against 82; of 16,384 37 against 47, 33 against 37
// (flat: 77 against 131).  128 rows of 151,936 (19,072 segments) 147 against 158 and 131 against 146, 192 rows 223 against 198 and
// 199 against 196; 160 rows of 131,072 (20,480) 161 both, 136 against 157.
// The verifier, where the workgroup passes over its row once and not three times, so that the number of rows decides: of 65,536 3
// rows 44 against 48, 32 rows 51 against 53, 45 rows 56 against 54; of 131,072 44 against 55, 59 against 68, 72 against 70; of
// 262,144 50 against 74, 88 against 93, 106 against 98; of 32,768 3 rows 40 against 42, 24 rows 47 against 45.
// From so many segments on, fewer where every row has a compute unit to itself in k_full_row, the verifier's second sums are left to
// k_spec_factor instead, and e is not written down: calls of 144 rows (16 sequences of 8 drafts) of 262,144 128 us against 143, 80 rows
// of it 102 against 106, 192 of 151,936 108 against 111, 176 of 131,072 94 against 97, 144 of it (18,432 segments) 88 against 86, 96 of
// 151,936 92 against 85; 448 rows of 65,536 108 against 118, 576 of 32,768 92 against 99, 288 of 50,257 (14,400) 84 against 92, 224 of
// it 78 against 70, 384 of 32,768 (12,288) 84 against 77, 2,304 of 16,384 153 against 210, 768 of it 89 against 83.
// The verifier's launches of rows that nothing touches go by two launches that leave all sums in order to the positions that need them
// (k_spec_units, k_spec_open), not by the pass, the row kernel and what follows them, at every length: where every draft is accepted and the
// bonus rows' largest entries decide, nothing needs them.  Where any sequence of the call rejects a draft, has a test too close to tell, or a flat bonus
// row (N(0, 1.5^2)), some position does need them, and short or few rows pay for it: the host cannot know, and what such calls lose, up to 13 %, is a
// quarter of what the others gain at most.  Sequences x drafts, us with them against without: everything decided; flat bonus rows; every sequence with a
// rejection; every sequence with a close test:
//    1 x 2 of  16,384   14 against 38   39.8 against 35.1   41.4 against 36.5   41.8 against 36.2
//   16 x 8 of  16,384   16 against 44   46.7 against 43.4   48.6 against 43.9   49.6 against 44.2
//    1 x 4 of  32,768   15 against 40   43.8 against 39.7   45.9 against 40.9   46.6 against 41.0
//   16 x 8 of  20,011   21 against 49   50.4 against 47.0   52.0 against 47.7   54.5 against 48.7
//   16 x 8 of  40,000   22 against 54   54.0 against 51.1   54.5 against 51.6   56.4 against 51.9
//    1 x 2 of  49,152   15 against 44   43.2 against 42.6   42.5 against 42.2   44.4 against 42.8
//    1 x 2 of 100,003   18 against 47   46.6 against 42.6   48.5 against 44.5   48.9 against 43.8
//    1 x 4 of 151,936   17 against 48   48.1 against 46.2   48.1 against 49.1   49.9 against 48.1
//   16 x 8 of 262,144   45 against 127   98 against 127  (the pass and k_spec_factor)
#define SR_PREPARED_MIN_SEGS 24        // tokens, rows that are cut
#define SR_PREPARED_MIN_SEGS_MIXED 20  // ... beside rows that are not
#define SR_PREPARED_ROWS_MIXED 128
#define SR_PREPARED_SEGS 32768
#define SR_PREPARED_SEGS_DISTRIBUTIONS 20480
#define SR_PREPARED_MIN_SEGS_VERIFY 64
#define SR_PREPARED_ROWS_VERIFY 32
#define SR_FACTOR_LATER_SEGS 14336
#define SR_FACTOR_LATER_SEGS_FEW 20480
// Distributions of rows that min-p cuts, where no other row asks for that launch: worth it for few long rows.  10, 200, 2,000, 8,000
// and 15,000 entries left, with it against without: one row of 131,072 36, 44, 50, 73, 102 us against 44, 56, 70, 102, 103; 16 rows
// 47, 56, 62, 83, 111 against 49, 61, 76, 110, 110; 32 (4,096 segments) 51, 62, 69, 91, 119 against 56, 68, 82, 118, 119; 64 rows 75, 88,
// 96, 121, 150 against 60, 72, 86, 121, 122; 16 rows of 262,144 59, 69, 77, 96, 124 against 82, 94, 109, 176, 179; 32 of 151,936 (4,768)
// 64, 76, 84, 103, 134 against 62, 74, 88, 130, 131, 48 of them 71, 85, 90, 109, 140 against 65, 76, 91, 132, 133; 16 rows of 98,304
// 45, 53, 58, 82, 112 against 43, 54, 68, 95, 95, of 65,536 40, 49, 54, 78, 105 against 35, 47, 60, 76, 76.  At odd addresses, one row
// of 100,003 37, 46, 51, 75, 102 against 39, 50, 63, 89, 89, 16 rows 45, 55, 59, 83, 111 against 44, 56, 69, 158, 157; 64 rows (6,272)
// 68, 81, 85, 108, 138 against 54, 66, 80, 168, 170; 16 rows of 65,537 41, 50, 54, 79, 106 against 38, 49, 62, 126, 123, one row 35, 45, 49,
// 73, 97 against 32, 45, 56, 72, 71.
#define SR_PREPARED_MIN_SEGS_MIN_P 128
#define SR_PREPARED_MIN_SEGS_MIN_P_ODD 96
#define SR_PREPARED_SEGS_MIN_P 4096
// candidates of a row that k_full_row sorts, and the groups it sorts them by: with a compute unit to itself, and without
#define SR_LIST_CAP_BIG 16384
#define SR_LIST_CAP_SMALL 4096
#define SR_LIST_GROUPS_BIG 16384
#define SR_LIST_GROUPS_SMALL 8192
#define SR_SEG_MAX 1024                    // most segments of such a row: longer rows are added the plain way
