// Host side of the full-vocabulary entry points: the slow path of Sampler.Sample, BuildFilteredDistribution,
// SampleWithDistribution, SampleFromProbs, ResampleResidual, the speculative accept loop and the MTP
// accept test.  Launch sequences only; all arithmetic is in sr_full.hip.
#include <cstring>

#include "sr_host.h"
#include "../../../include/stingray_sampler_test.h"

namespace {

// a row of the verifier whose drafts are accepted by the ratio test
bool by_ratio(const SrRow& r) { return !(r.p_min > 0.0f && r.p_min < 1.0f) && !(r.flags & SR_ROW_DRAFT_FROM_LOOKUP); }

// the number of the next launch (full_state is there)
hipError_t next_launch(sr_ctx* ctx)
{
    if (++ctx->full_seq != 0u) return hipSuccess;
    // the numbers have gone round: nothing of an earlier launch may look like this one's
    hipError_t e = hipMemsetAsync(ctx->full_state.p, 0, ctx->full_state.cap, ctx->stream);
    if (e == hipSuccess && ctx->full_row_sync.p) e = hipMemsetAsync(ctx->full_row_sync.p, 0, ctx->full_row_sync.cap, ctx->stream);
    if (e == hipSuccess && ctx->full_meet.p) e = hipMemsetAsync(ctx->full_meet.p, 0, ctx->full_meet.cap, ctx->stream);
    if (e == hipSuccess && ctx->spec_sync.p) e = hipMemsetAsync(ctx->spec_sync.p, 0, ctx->spec_sync.cap, ctx->stream);
    ctx->full_seq = 1u;
    return e;
}

// Runs the full-vocabulary pipeline for the rows in `list` (device array of n_rows row indices).
//   mode 0: work rows live in ctx scratch, tokens out.   mode 1/2: work rows ARE the caller's probs rows.
int run_full(sr_ctx* ctx, const sr_batch* b, const int32_t* list_dev, int n_rows, bool any_top_p, const void* logits_dev,
             int dtype, int64_t row_stride, int mode, float* probs_dev, int64_t probs_stride, int32_t* out_tokens_dev,
             uint32_t* out_flags_dev, bool lazy_scale = false, const std::vector<SrRow>* host_rows = nullptr, int n_greedy = 0,
             SrFullArgs* factor_later = nullptr)
{
    if (n_rows <= 0) return SR_OK;
    hipStream_t st = ctx->stream;
    const int vocab = b->vocab;
    SrFullArgs a{};
    a.logits = logits_dev;
    a.row_stride = row_stride;
    a.vocab = vocab;
    a.dtype = dtype;
    a.row_list = list_dev;
    a.rows = b->d_rows.as<SrRow>();
    a.edits = b->d_edits.as<SrEdit>();
    a.mask = sr_batch_mask_ptr(b);
    a.mask_stride = sr_batch_mask_stride(b);
    a.mode = mode;
    a.cu_count = ctx->cu_count;
    a.n_greedy = n_greedy;  // (a further n_greedy rows of the list: they need nothing of what follows but a meeting point)
    a.prof = ctx->prof;
    if (mode == 0) {
        const int64_t ws = (vocab + 3) & ~3;
        SR_HIP(ctx, ctx->work.reserve((size_t)n_rows * ws * sizeof(float), st));
        a.work = ctx->work.as<float>();
        a.work_stride = ws;
        a.work_by_row = 0;
    } else {
        a.work = probs_dev;
        a.work_stride = probs_stride;
        a.work_by_row = 1;
    }
    a.lazy_scale = lazy_scale ? 1 : 0;
    // Which of the rows that come here keep an adjusted copy, and which have their edits applied where they are read
    // (the rows of the batch that take this path: every row in modes 1 / 2).
    // Long rows: the softmax denominators are prepared by
    // the pass over the whole device (k_full_softmax_seg) and the rows' workgroups only walk the records.  That pass also
    // applies the edits of the rows without an adjusted copy itself: they need no table and no kernel in front.
    const int nseg = (vocab + SR_SEG_TERMS - 1) / SR_SEG_TERMS;
    const bool seg_mode = vocab >= SR_SEG_MIN_VOCAB && nseg <= SR_SEG_MAX;
    a.edits_in_pass = seg_mode ? 1 : 0;
    bool any_table = false, any_copy = false, any_edits = false, any_list = false, prepared = false, any_plain = false, any_min_p = false;
    int n_sampled = 0, n_seen = 0;
    for (const SrRow& r : (host_rows ? *host_rows : b->h_rows)) {
        if (mode == 0 && r.path != SR_PATH_FULL) continue;
        const bool on_the_fly = sr_row_edits_on_the_fly(r, vocab);
        any_table = any_table || (on_the_fly && !seg_mode);
        n_sampled += r.temperature > 0.0f ? 1 : 0;
        n_seen++;
        any_edits = any_edits || (r.edit_cnt > 0 && !(on_the_fly && seg_mode));
        any_copy = any_copy || !(r.temperature > 0.0f && (r.edit_cnt <= 0 || on_the_fly));
        if (seg_mode && r.temperature > 0.0f && !(r.top_k > 0 && r.top_k < vocab)) {
            any_list = any_list || sr_row_cut(r);
            // Rows that the row kernel may leave to the whole device: those that nothing cuts and, but for the verifier, whose
            // reader takes e where it is, those that only top-p cuts (a few members or tens of thousands).  What a min-p of some
            // size leaves is mostly little, and nobody knows before the launch: tokens of 64 rows of 151,936 with 300 entries left
            // take 51 us with the launch behind and 47 without, with 2,000 102 and 57, with 8,000 119 and 92, since up to 8,192 the row's
            // workgroup then finishes by itself; with 9,000 to 16,000 132 - 156 and 180 - 198, and with 30,000, where it finds nothing to
            // do, 162 and 159.  Distributions: SR_PREPARED_MIN_SEGS_MIN_P, whatever the min-p.
            const bool by_min_p = mode != 0 ? r.min_p > 0.0f : r.min_p >= 0.002f;
            prepared = prepared || (lazy_scale ? !sr_row_cut(r) : !by_min_p);
            any_plain = any_plain || !sr_row_cut(r);
            any_min_p = any_min_p || by_min_p;
        }
    }
    const bool odd_rows = mode != 0 && !lazy_scale && (probs_stride & 3) != 0;
    const long long segs = (long long)n_rows * nseg;
    if (lazy_scale) {
        prepared = prepared && nseg >= SR_PREPARED_MIN_SEGS_VERIFY && n_rows <= SR_PREPARED_ROWS_VERIFY;
        if (factor_later && any_plain && seg_mode && dtype == SR_DTYPE_F32 && segs >= (n_rows > ctx->cu_count ? SR_FACTOR_LATER_SEGS : SR_FACTOR_LATER_SEGS_FEW)) {
            a.factor_later = 1;
            prepared = false;
        }
    } else if (mode != 0) {
        prepared = prepared && segs <= SR_PREPARED_SEGS_DISTRIBUTIONS;
    } else {
        // (any_list: some row is cut)
        const bool mixed = any_plain && nseg >= SR_PREPARED_MIN_SEGS_MIXED && n_rows <= SR_PREPARED_ROWS_MIXED;
        prepared = prepared && ((any_plain && !any_list) || mixed || nseg >= SR_PREPARED_MIN_SEGS) && segs <= SR_PREPARED_SEGS;
    }
    if (mode != 0 && !lazy_scale && any_min_p)
        prepared = prepared || (nseg >= (odd_rows ? SR_PREPARED_MIN_SEGS_MIN_P_ODD : SR_PREPARED_MIN_SEGS_MIN_P) && (long long)n_rows * nseg <= SR_PREPARED_SEGS_MIN_P);
    a.any_copy = any_copy ? 1 : 0;
    a.any_edits = any_edits ? 1 : 0;
    a.n_sampled = (int)((long long)n_sampled * n_rows / std::max(1, n_seen));  // (a verifier's launch has every row several times)
    a.edit_tab = nullptr;
    a.edit_tab_stride = (((int64_t)vocab + 31) / 32 + SR_FULL_EDIT_VALUES + 3) & ~(int64_t)3;
    if (any_table) {
        SR_HIP(ctx, ctx->edit_tab.reserve((size_t)n_rows * (size_t)a.edit_tab_stride * sizeof(uint32_t), st));
        a.edit_tab = ctx->edit_tab.as<uint32_t>();
    }
    // (cleared when new: the rows' maxima carry the number of the launch that wrote them, and the rows' scalars are
    // otherwise left by each launch the way the next one expects them)
    SR_HIP(ctx, ctx->full_state.reserve((size_t)n_rows * sizeof(SrFullState), st, true));
    a.state = ctx->full_state.as<SrFullState>();
    SR_HIP(ctx, next_launch(ctx));
    a.seq = ctx->full_seq;
    a.row_wait_limit = ctx->row_wait_limit;
    a.behind_wait_limit = ctx->behind_wait_limit;
    // sort segments are laid out with the work stride of mode 0; in modes 1/2 use a private stride
    const int64_t seg_stride = (vocab + 3) & ~3;
    if ((int64_t)n_rows * seg_stride >= (int64_t)1 << 31)
        return sr_fail(ctx, SR_ERR_UNSUPPORTED, "full-vocabulary path: rows x vocab exceeds 2^31 entries");
    if (any_top_p || any_list) {
        // a row's segment: scratch of its top-p stage (histogram sums, the members of a long nucleus, and the survivors
        // of a row that the walk by slabs cannot close, sorted there by the row's workgroup)
        const size_t items = (size_t)n_rows * seg_stride;
        SR_HIP(ctx, ctx->sort_k0.reserve(items * 4, st));
        SR_HIP(ctx, ctx->sort_v0.reserve(items * 4, st));
        a.sort_keys_in = ctx->sort_k0.as<uint32_t>();
        a.sort_vals_in = ctx->sort_v0.as<int32_t>();
    }
    // the kernels index sort segments with work_stride; keep both strides equal in mode 0 and pass the
    // segment stride separately otherwise
    a.sort_stride = seg_stride;
    {
        if (seg_mode) {
            const size_t segs = (size_t)n_rows * (size_t)nseg;
            const int half_blocks = (nseg + SR_HALF_BLOCK_SEGS - 1) / SR_HALF_BLOCK_SEGS;
            SR_HIP(ctx, ctx->full_seg_func.reserve(segs * sizeof(SeqSegFunc), st));
            SR_HIP(ctx, ctx->full_seg_sum.reserve(segs * sizeof(float), st));
            SR_HIP(ctx, ctx->full_seg_cnt.reserve(segs * sizeof(uint32_t), st));
            SR_HIP(ctx, ctx->full_mass.reserve((size_t)n_rows * 256 * sizeof(float), st, true));
            SR_HIP(ctx, ctx->full_row_sync.reserve((size_t)(n_rows + n_greedy) * SR_ROW_SYNC_STRIDE * sizeof(unsigned long long), st, true));
            a.row_sync = ctx->full_row_sync.as<unsigned long long>();
            a.meet_sums = (2 * half_blocks + 15) & ~15;
            a.meet_stride = (a.meet_sums + nseg + 15) & ~15;
            SR_HIP(ctx, ctx->full_meet.reserve((size_t)n_rows * (size_t)a.meet_stride * sizeof(unsigned long long), st, true));
            a.meet = ctx->full_meet.as<unsigned long long>();
            a.seg_func = (SeqSegFunc*)ctx->full_seg_func.p;
            a.seg_sum = ctx->full_seg_sum.as<float>();
            a.seg_cnt = ctx->full_seg_cnt.as<uint32_t>();
            a.mass = ctx->full_mass.as<float>();
            a.seg_stride = nseg;
            a.chain_stride = half_blocks * 8;
            a.chain_blocks = (half_blocks + 1) / 2;
            SR_HIP(ctx, ctx->full_chain_sum.reserve((size_t)n_rows * (size_t)a.chain_stride * sizeof(float), st));
            SR_HIP(ctx, ctx->full_chain_func.reserve((size_t)n_rows * 8 * (size_t)a.chain_blocks * sizeof(SeqSegFunc), st));
            a.chain_sum = ctx->full_chain_sum.as<float>();
            a.chain_func = (SeqSegFunc*)ctx->full_chain_func.p;
            a.prepared = prepared ? 1 : 0;
            // Two launches of k_prepared_row in place of one whose workgroups wait, from twice the workgroups on that the device
            // holds, where these are not whole rows.  One and two launches, us: tokens that nothing cuts, 56 rows of
            // 200,064 97 and 90, 64 of 151,936 90 and 83, 192 of 151,936 199 and 180, 96 of 100,003 88.5 and 85, 160 of 50,257 82 and 80;
            // whole rows: 128 of 131,072 130 and 141, 48 of 262,144 122 and 124; fewer workgroups: 48 of 151,936 76.5 and 75.5,
            // beside rows cut by top-p 68 and 70.5.  Distributions of rows that are all cut, whose launch passes memory at most: 48 of
            // 262,144 106 and 100, 128 of 131,072 114 and 112, 128 of 65,536 69 both.
            const int blocks = (half_blocks + 1) / 2, held = 2 * ctx->cu_count;
            a.behind_twice = prepared && !lazy_scale && (long long)n_rows * blocks >= 2 * held &&
                             (any_plain ? blocks >= 7 && held % blocks != 0 : mode != 0 && blocks >= 12) ? 1 : 0;
            // Up to 8,192 members cost the row's workgroup less than the launch behind it (us a call, top-p 0.95 at temperature 0.6 under masks that leave
            // 0.4, 0.2, 0.1, 0.03 of the row, 1,024 and 8,192: 64 rows of 151,936 134 and 134, 123 and 89, 115 and 74, 90 and 67; 200 of 65,536 142 and 99, 133
            // and 83, 133 and 77; one row 75 both, 65 and 63, 58 and 49), but where a row that nothing cuts takes that launch anyway: then it waits
            // for them (every third row of 32 of 100,003 87 and 104, 76 and 87, 71 and 75).  Of short rows more, whatever stands beside them:
            // 256 rows of 12,290, half of them cut to some thousand members, 98 us, with 1,024 134.
            a.finish_most = prepared && any_plain && nseg >= SR_PREPARED_MIN_SEGS ? 1024 : 8192;
            // e = expf(x - max): in the work rows of tokens-only launches and of the verifier (whose reader applies the factors);
            // apart from the caller's rows where the probabilities take shape there
            a.e_rows = a.work;
            a.e_stride = a.work_stride;
            if (mode != 0 && !lazy_scale && prepared) {
                a.e_stride = seg_stride;
                SR_HIP(ctx, ctx->work.reserve((size_t)n_rows * (size_t)a.e_stride * sizeof(float), st));
                a.e_rows = ctx->work.as<float>();
            }
        }
    }
    a.uniforms = sr_batch_uniforms(b);
    a.uniforms_per_row = b->upr;
    a.out_tokens = out_tokens_dev;
    a.out_flags = out_flags_dev;
    // With a compute unit per row the row kernel's workgroups can have more shared memory each: longer lists of candidates
    // and slabs of twice the size.  (With more rows, two workgroups share a compute unit.)
    a.big_slabs = ((any_top_p || any_list) && n_rows <= ctx->cu_count) ? 1 : 0;

    SR_HIP(ctx, sr_launch_full_prep(a, n_rows, st));
    SR_HIP(ctx, sr_launch_full_row(a, n_rows, st));  // (every row is finished by this one launch)
    if (factor_later) *factor_later = a;
    return SR_OK;
}

bool row_uses_top_p(const SrRow& r) { return r.temperature > 0.0f && r.top_p < 1.0f && r.top_p > 0.0f; }

int check_batch_call(sr_ctx* ctx, const sr_batch* b, const void* logits_dev, int dtype, int64_t row_stride, const char* who)
{
    if (!logits_dev) return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, std::string(who) + ": logits is null");
    if (dtype != SR_DTYPE_F32 && dtype != SR_DTYPE_BF16) return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, std::string(who) + ": unknown dtype");
    if (b->vocab <= 0) return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, std::string(who) + ": empty vocabulary");
    if (row_stride < b->vocab) return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, std::string(who) + ": row stride < vocab");
    if (int rc = sr_batch_complete(ctx, b, who)) return rc;
    return sr_batch_masks_valid(ctx, b, who);
}

// identity row list [0, rows) on the device
int identity_list(sr_ctx* ctx, int rows, const int32_t** out)
{
    if (ctx->ident_rows < rows) {
        std::vector<int32_t> h((size_t)rows);
        for (int i = 0; i < rows; i++) h[(size_t)i] = i;
        SR_HIP(ctx, ctx->ident.reserve((size_t)rows * sizeof(int32_t), ctx->stream));
        SR_HIP(ctx, hipMemcpyAsync(ctx->ident.p, h.data(), (size_t)rows * sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream));
        SR_HIP(ctx, hipStreamSynchronize(ctx->stream));
        ctx->ident_rows = rows;
    }
    *out = ctx->ident.as<int32_t>();
    return SR_OK;
}

// The caller's uniforms for a kernel enqueued on the context's stream: copied into pinned memory of the context, which
// the kernel reads in place, so the call neither waits nor depends on the caller's array afterwards.
int upload_uniforms(sr_ctx* ctx, const double* uniforms, int rows, const double** dev)
{
    const size_t bytes = (size_t)rows * sizeof(double);
    SR_HIP(ctx, ctx->uni_ring.begin(ctx->pinned, bytes + 256, ctx->stream, 0, ctx->stream_epoch));
    const void* at = ctx->uni_ring.put(uniforms, bytes);
    if (!at) return sr_fail(ctx, SR_ERR_OUT_OF_MEMORY, "no pinned memory for the uniforms");
    *dev = (const double*)at;
    return SR_OK;
}

}  // namespace

int sr_full_rows_launch(sr_ctx* ctx, const sr_batch* b, const void* logits_dev, int dtype, int64_t row_stride,
                        int32_t* out_tokens_dev, uint32_t* out_flags_dev)
{
    bool any_top_p = false;
    for (int32_t r : b->h_full_list) any_top_p = any_top_p || row_uses_top_p(b->h_rows[(size_t)r]);
    return run_full(ctx, b, b->d_full_list.as<int32_t>(), (int)b->h_full_list.size() - b->full_greedy, any_top_p, logits_dev, dtype,
                    row_stride, 0, nullptr, 0, out_tokens_dev, out_flags_dev, false, nullptr, b->full_greedy);
}

// SampleTopK (Sampler.cs:216-357) for rows whose k + history length exceeds what the selection kernel's row tail
// sorts: the row sorted where it lies by one workgroup, its first k + history-length entries adjusted and sorted
// again, and a walk over the result by the same workgroup.
int sr_wide_rows_launch(sr_ctx* ctx, const sr_batch* b, const int32_t* list_dev, int n_rows, const void* logits_dev,
                        int dtype, int64_t row_stride, int32_t* out_tokens_dev, uint32_t* out_flags_dev)
{
    if (n_rows <= 0) return SR_OK;
    hipStream_t st = ctx->stream;
    const int vocab = b->vocab;
    const int64_t stride = (vocab + 3) & ~3;
    if ((int64_t)n_rows * stride >= (int64_t)1 << 31)
        return sr_fail(ctx, SR_ERR_UNSUPPORTED, "wide top-k rows: rows x vocab exceeds 2^31 entries");
    const size_t items = (size_t)n_rows * (size_t)stride;
    SrFullArgs a{};
    a.logits = logits_dev;
    a.row_stride = row_stride;
    a.vocab = vocab;
    a.dtype = dtype;
    a.row_list = list_dev;
    a.rows = b->d_rows.as<SrRow>();
    a.edits = b->d_edits.as<SrEdit>();
    a.mask = sr_batch_mask_ptr(b);
    a.mask_stride = sr_batch_mask_stride(b);
    SR_HIP(ctx, ctx->work.reserve(items * sizeof(float), st));
    a.work = ctx->work.as<float>();
    a.work_stride = stride;
    SR_HIP(ctx, ctx->sort_k0.reserve(items * 4, st));
    SR_HIP(ctx, ctx->sort_v0.reserve(items * 4, st));
    SR_HIP(ctx, ctx->sort_v1.reserve(items * 4, st));
    a.sort_keys_in = ctx->sort_k0.as<uint32_t>();
    a.sort_vals_in = ctx->sort_v0.as<int32_t>();
    a.wide_ids = ctx->sort_v1.as<int32_t>();
    a.sort_stride = stride;
    a.uniforms = sr_batch_uniforms(b);
    a.uniforms_per_row = b->upr;
    a.out_tokens = out_tokens_dev;
    a.out_flags = out_flags_dev;

    SR_HIP(ctx, sr_launch_wide_keys(a, n_rows, st));
    SR_HIP(ctx, sr_launch_wide_sort(a, n_rows, 1, st));
    SR_HIP(ctx, sr_launch_wide_adjust(a, n_rows, st));
    SR_HIP(ctx, sr_launch_wide_sort(a, n_rows, 0, st));
    SR_HIP(ctx, sr_launch_wide_tail(a, n_rows, st));
    return SR_OK;
}

extern "C" {

int sr_build_distribution_launch(sr_ctx* ctx, const sr_batch* b, const void* logits_dev, int dtype, int64_t row_stride,
                                 float* out_probs_dev, int64_t probs_stride, int32_t probs_len)
{
    if (!ctx || !b) return SR_ERR_NULL_ARGUMENT;
    if (b->rows == 0) return SR_OK;
    if (probs_len != b->vocab)  // Sampler.cs:121-123
        return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "probs length (" + std::to_string(probs_len) + ") must equal logits length (" +
                                                         std::to_string(b->vocab) + ").");
    int rc = check_batch_call(ctx, b, logits_dev, dtype, row_stride, "sr_build_distribution_launch");
    if (rc != SR_OK) return rc;
    if (!out_probs_dev) return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "sr_build_distribution_launch: probs is null");
    if (probs_stride < b->vocab) return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "sr_build_distribution_launch: probs stride < vocab");
    SR_HIP(ctx, hipSetDevice(ctx->device));
    const int32_t* list = nullptr;
    rc = identity_list(ctx, b->rows, &list);
    if (rc != SR_OK) return rc;
    bool any_top_p = false;
    for (const SrRow& r : b->h_rows) any_top_p = any_top_p || row_uses_top_p(r);
    return run_full(ctx, b, list, b->rows, any_top_p, logits_dev, dtype, row_stride, 1, out_probs_dev, probs_stride, nullptr, nullptr);
}

int sr_sample_with_distribution_launch(sr_ctx* ctx, const sr_batch* b, const void* logits_dev, int dtype, int64_t row_stride,
                                       float* out_probs_dev, int64_t probs_stride, int32_t probs_len, int32_t* out_tokens_dev)
{
    if (!ctx || !b) return SR_ERR_NULL_ARGUMENT;
    if (b->rows == 0) return SR_OK;
    if (probs_len != b->vocab)
        return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "probs length (" + std::to_string(probs_len) + ") must equal logits length (" +
                                                         std::to_string(b->vocab) + ").");
    int rc = check_batch_call(ctx, b, logits_dev, dtype, row_stride, "sr_sample_with_distribution_launch");
    if (rc != SR_OK) return rc;
    if (!out_probs_dev || !out_tokens_dev) return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "sr_sample_with_distribution_launch: null output");
    if (probs_stride < b->vocab) return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "sr_sample_with_distribution_launch: probs stride < vocab");
    for (const SrRow& r : b->h_rows)
        if (r.temperature > 0.0f && b->upr < 1)
            return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "sr_sample_with_distribution_launch: a sampled row needs a uniform");
    SR_HIP(ctx, hipSetDevice(ctx->device));
    const int32_t* list = nullptr;
    rc = identity_list(ctx, b->rows, &list);
    if (rc != SR_OK) return rc;
    bool any_top_p = false;
    for (const SrRow& r : b->h_rows) any_top_p = any_top_p || row_uses_top_p(r);
    return run_full(ctx, b, list, b->rows, any_top_p, logits_dev, dtype, row_stride, 2, out_probs_dev, probs_stride, out_tokens_dev, nullptr);
}

int sr_sample_from_probs_launch(sr_ctx* ctx, const float* probs_dev, int32_t rows, int32_t vocab, int64_t probs_stride,
                                const double* uniforms, int32_t* out_tokens_dev)
{
    if (!ctx) return SR_ERR_NULL_ARGUMENT;
    if (!uniforms) return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "rng");  // ArgumentNullException(rng), Sampler.cs:197
    if (rows == 0) return SR_OK;
    if (!probs_dev || !out_tokens_dev) return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "sr_sample_from_probs_launch: null tensor");
    if (rows < 0 || vocab <= 0 || probs_stride < vocab) return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "sr_sample_from_probs_launch: bad shape");
    SR_HIP(ctx, hipSetDevice(ctx->device));
    const double* u = nullptr;
    int rc = upload_uniforms(ctx, uniforms, rows, &u);
    if (rc != SR_OK) return rc;
    SR_HIP(ctx, sr_launch_draw_rows(probs_dev, probs_stride, vocab, rows, u, out_tokens_dev, ctx->stream));
    return SR_OK;
}

int sr_resample_residual_launch(sr_ctx* ctx, const float* p_dev, int32_t p_len, int64_t p_stride, const float* q_dev,
                                int32_t q_len, int64_t q_stride, int32_t rows, const double* uniforms, int32_t* out_tokens_dev)
{
    if (!ctx) return SR_ERR_NULL_ARGUMENT;
    if (!uniforms) return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "rng");  // Sampler.cs:589
    if (p_len != q_len)                                                // Sampler.cs:590-592
        return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT,
                       "p and q must have equal length (" + std::to_string(p_len) + " vs " + std::to_string(q_len) + ").");
    if (rows == 0) return SR_OK;
    if (!p_dev || !q_dev || !out_tokens_dev) return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "sr_resample_residual_launch: null tensor");
    if (rows < 0 || p_len <= 0 || p_stride < p_len || q_stride < q_len)
        return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "sr_resample_residual_launch: bad shape");
    SR_HIP(ctx, hipSetDevice(ctx->device));
    const double* u = nullptr;
    int rc = upload_uniforms(ctx, uniforms, rows, &u);
    if (rc != SR_OK) return rc;
    SR_HIP(ctx, sr_launch_residual_rows(p_dev, p_stride, q_dev, q_stride, p_len, rows, u, out_tokens_dev, ctx->stream));
    return SR_OK;
}


// ---- span-shaped forms: host buffers in, host results out ------------------------------------------------

static int stage_up(sr_ctx* ctx, DeviceBuf& buf, const void* src, size_t bytes)
{
    SR_HIP(ctx, buf.reserve(bytes, ctx->stream));
    SR_HIP(ctx, hipMemcpyAsync(buf.p, src, bytes, hipMemcpyHostToDevice, ctx->stream));
    return SR_OK;
}

static int distribution_host(sr_ctx* ctx, const char* what, bool sample, const float* logits, int32_t rows, int32_t vocab,
                             int64_t row_stride, const sr_row_params* params, const int32_t* hist_ids,
                             const int32_t* hist_offsets, const int32_t* bias_ids, const float* bias_vals,
                             const int32_t* bias_offsets, const double* uniforms, float* out_probs, int64_t probs_stride,
                             int32_t probs_len, int32_t* out_tokens)
{
    if (!ctx) return SR_ERR_NULL_ARGUMENT;
    if (rows == 0) return SR_OK;
    if (probs_len != vocab)  // Sampler.cs:121-123
        return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "probs length (" + std::to_string(probs_len) + ") must equal logits length (" +
                                                         std::to_string(vocab) + ").");
    if (!logits || !params || !out_probs || (sample && !out_tokens))
        return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, std::string(what) + ": null argument");
    if (rows < 0 || vocab <= 0 || row_stride < vocab || probs_stride < vocab)
        return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, std::string(what) + ": bad shape");
    SR_HIP(ctx, hipSetDevice(ctx->device));
    if (!ctx->tmp_batch) {
        int rc = sr_batch_create(ctx, &ctx->tmp_batch);
        if (rc != SR_OK) return rc;
    }
    int rc = sr_batch_upload(ctx->tmp_batch, rows, vocab, params, hist_ids, hist_offsets, bias_ids, bias_vals, bias_offsets,
                             nullptr, 0, nullptr, uniforms, uniforms ? 1 : 0);
    if (rc != SR_OK) return rc;
    const size_t in_bytes = ((size_t)(rows - 1) * (size_t)row_stride + (size_t)vocab) * sizeof(float);
    rc = stage_up(ctx, ctx->host_logits, logits, in_bytes);
    if (rc != SR_OK) return rc;
    const int64_t ps = (vocab + 3) & ~3;
    SR_HIP(ctx, ctx->stage_probs.reserve((size_t)rows * (size_t)ps * sizeof(float), ctx->stream));
    SR_HIP(ctx, ctx->out_tokens.reserve((size_t)rows * sizeof(int32_t), ctx->stream));
    if (sample)
        rc = sr_sample_with_distribution_launch(ctx, ctx->tmp_batch, ctx->host_logits.p, SR_DTYPE_F32, row_stride,
                                                ctx->stage_probs.as<float>(), ps, probs_len, ctx->out_tokens.as<int32_t>());
    else
        rc = sr_build_distribution_launch(ctx, ctx->tmp_batch, ctx->host_logits.p, SR_DTYPE_F32, row_stride,
                                          ctx->stage_probs.as<float>(), ps, probs_len);
    if (rc != SR_OK) return rc;
    SR_HIP(ctx, hipMemcpy2DAsync(out_probs, (size_t)probs_stride * sizeof(float), ctx->stage_probs.p, (size_t)ps * sizeof(float),
                                 (size_t)vocab * sizeof(float), (size_t)rows, hipMemcpyDeviceToHost, ctx->stream));
    if (sample)
        SR_HIP(ctx, hipMemcpyAsync(out_tokens, ctx->out_tokens.p, (size_t)rows * sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
    SR_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return SR_OK;
}

int sr_build_distribution(sr_ctx* ctx, const float* logits, int32_t rows, int32_t vocab, int64_t row_stride,
                          const sr_row_params* params, const int32_t* hist_ids, const int32_t* hist_offsets,
                          const int32_t* bias_ids, const float* bias_vals, const int32_t* bias_offsets, float* out_probs,
                          int64_t probs_stride, int32_t probs_len)
{
    return distribution_host(ctx, "sr_build_distribution", false, logits, rows, vocab, row_stride, params, hist_ids, hist_offsets,
                             bias_ids, bias_vals, bias_offsets, nullptr, out_probs, probs_stride, probs_len, nullptr);
}

int sr_sample_with_distribution(sr_ctx* ctx, const float* logits, int32_t rows, int32_t vocab, int64_t row_stride,
                                const sr_row_params* params, const int32_t* hist_ids, const int32_t* hist_offsets,
                                const int32_t* bias_ids, const float* bias_vals, const int32_t* bias_offsets,
                                const double* uniforms, float* out_probs, int64_t probs_stride, int32_t probs_len,
                                int32_t* out_tokens)
{
    return distribution_host(ctx, "sr_sample_with_distribution", true, logits, rows, vocab, row_stride, params, hist_ids,
                             hist_offsets, bias_ids, bias_vals, bias_offsets, uniforms, out_probs, probs_stride, probs_len,
                             out_tokens);
}

int sr_sample_from_probs(sr_ctx* ctx, const float* probs, int32_t rows, int32_t vocab, int64_t probs_stride,
                         const double* uniforms, int32_t* out_tokens)
{
    if (!ctx) return SR_ERR_NULL_ARGUMENT;
    if (!uniforms) return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "rng");  // ArgumentNullException(rng), Sampler.cs:197
    if (rows == 0) return SR_OK;
    if (!probs || !out_tokens) return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "sr_sample_from_probs: null argument");
    if (rows < 0 || vocab <= 0 || probs_stride < vocab) return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "sr_sample_from_probs: bad shape");
    SR_HIP(ctx, hipSetDevice(ctx->device));
    int rc = stage_up(ctx, ctx->host_logits, probs, ((size_t)(rows - 1) * (size_t)probs_stride + (size_t)vocab) * sizeof(float));
    if (rc != SR_OK) return rc;
    SR_HIP(ctx, ctx->out_tokens.reserve((size_t)rows * sizeof(int32_t), ctx->stream));
    rc = sr_sample_from_probs_launch(ctx, ctx->host_logits.as<float>(), rows, vocab, probs_stride, uniforms, ctx->out_tokens.as<int32_t>());
    if (rc != SR_OK) return rc;
    SR_HIP(ctx, hipMemcpyAsync(out_tokens, ctx->out_tokens.p, (size_t)rows * sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
    SR_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return SR_OK;
}

int sr_resample_residual(sr_ctx* ctx, const float* p, int32_t p_len, int64_t p_stride, const float* q, int32_t q_len,
                         int64_t q_stride, int32_t rows, const double* uniforms, int32_t* out_tokens)
{
    if (!ctx) return SR_ERR_NULL_ARGUMENT;
    if (!uniforms) return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "rng");  // Sampler.cs:589
    if (p_len != q_len)                                                // Sampler.cs:590-592
        return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT,
                       "p and q must have equal length (" + std::to_string(p_len) + " vs " + std::to_string(q_len) + ").");
    if (rows == 0) return SR_OK;
    if (!p || !q || !out_tokens) return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "sr_resample_residual: null argument");
    if (rows < 0 || p_len <= 0 || p_stride < p_len || q_stride < q_len)
        return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "sr_resample_residual: bad shape");
    SR_HIP(ctx, hipSetDevice(ctx->device));
    int rc = stage_up(ctx, ctx->host_logits, p, ((size_t)(rows - 1) * (size_t)p_stride + (size_t)p_len) * sizeof(float));
    if (rc != SR_OK) return rc;
    rc = stage_up(ctx, ctx->stage_probs, q, ((size_t)(rows - 1) * (size_t)q_stride + (size_t)q_len) * sizeof(float));
    if (rc != SR_OK) return rc;
    SR_HIP(ctx, ctx->out_tokens.reserve((size_t)rows * sizeof(int32_t), ctx->stream));
    rc = sr_resample_residual_launch(ctx, ctx->host_logits.as<float>(), p_len, p_stride, ctx->stage_probs.as<float>(), q_len, q_stride,
                                     rows, uniforms, ctx->out_tokens.as<int32_t>());
    if (rc != SR_OK) return rc;
    SR_HIP(ctx, hipMemcpyAsync(out_tokens, ctx->out_tokens.p, (size_t)rows * sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
    SR_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return SR_OK;
}

int sr_spec_verify_launch(sr_ctx* ctx, const sr_batch* b, const float* target_logits_dev, const float* draft_probs_dev,
                          const int32_t* draft_tokens_dev, int32_t n_draft, int32_t* out_accepted_dev, int32_t* out_tokens_dev)
{
    if (!ctx || !b) return SR_ERR_NULL_ARGUMENT;
    if (b->rows == 0) return SR_OK;
    if (n_draft < 0) return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "sr_spec_verify_launch: negative draft length");
    if (int rc = sr_batch_complete(ctx, b, "sr_spec_verify_launch")) return rc;
    if (!target_logits_dev || !out_accepted_dev || !out_tokens_dev || (n_draft > 0 && !draft_tokens_dev))
        return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "sr_spec_verify_launch: null tensor");
    if (n_draft > 0 && !draft_probs_dev) {
        // only rows under the ratio test read q (SpeculativeDecoder.cs:538-543)
        for (int r = 0; r < b->rows; r++) {
            const SrRow& d = b->h_rows[(size_t)r];
            if (by_ratio(d))
                return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "sr_spec_verify_launch: a row under the ratio test needs the draft distributions");
        }
    }
    if (b->vocab <= 0) return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "sr_spec_verify_launch: empty vocabulary");
    if (b->upr < n_draft + 1) return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "sr_spec_verify_launch: needs n_draft + 1 uniforms per row");
    if (b->has_mask) return sr_fail(ctx, SR_ERR_UNSUPPORTED, "sr_spec_verify_launch: allow-masks are not part of speculative verification");
    SR_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    const int rows = b->rows, V = b->vocab, P = n_draft + 1;
    // Every position of a row is filtered with the row's parameters (SpeculativeDecoder.cs:535): expand the
    // batch's row descriptors to rows x positions and build all distributions in one pass.
    if ((int64_t)rows * P * V >= (int64_t)1 << 31)
        return sr_fail(ctx, SR_ERR_UNSUPPORTED, "sr_spec_verify_launch: rows x positions x vocab exceeds 2^31 entries");
    bool any_top_p = false;
    for (int r = 0; r < rows; r++) any_top_p = any_top_p || row_uses_top_p(b->h_rows[(size_t)r]);
    // (made by a kernel, so that the call does not wait for the host; kept with the batch until its descriptors change)
    if (b->spec_positions != P) {
        SR_HIP(ctx, b->spec_rows.reserve((size_t)rows * P * sizeof(SrRow), st));
        SR_HIP(ctx, sr_launch_expand_rows(b->d_rows.as<SrRow>(), b->spec_rows.as<SrRow>(), rows, P, st));
        b->spec_positions = P;
    }
    const int64_t p_stride = ((int64_t)V + 63) & ~(int64_t)63;  // (no row of e shares a cache line with another: k_spec_factor)
    SR_HIP(ctx, ctx->spec_probs.reserve((size_t)rows * P * (size_t)p_stride * sizeof(float), st));
    sr_batch tmp;  // a view: expanded rows, the original edits
    tmp.ctx = ctx;
    tmp.rows = rows * P;
    tmp.vocab = V;
    tmp.upr = 0;
    tmp.d_rows.p = b->spec_rows.p;
    tmp.d_edits.p = b->d_edits.p;
    tmp.mask_stride = 0;
    const int32_t* list = nullptr;
    SrFullArgs full{};
    const bool in_one = n_draft > 0 && n_draft < 64 && draft_probs_dev && rows <= 65535;  // (k_spec_factor: a position a lane)
    // Rows that nothing touches, all of them: k_spec_units and k_spec_open (both sides measured: sr_types.h).  Not the untouched rows of a mixed call:
    // it lasts as long as the cut row's positions, which one workgroup each finishes.  16 x 8 of 262,144, none, one and all sequences
    // under top-p, us: 114, 229, 270; with one, k_full_softmax_seg 59, k_full_row 110, k_spec_factor 38, k_spec_rows 22, where the other
    // way's 23 + 69 + 23 would stand beside a pass and a k_full_row for the cut row's nine positions.
    const int nseg = (V + SR_SEG_TERMS - 1) / SR_SEG_TERMS;
    bool all_open = in_one && V >= SR_SEG_MIN_VOCAB && nseg <= SR_SEG_MAX && (int64_t)rows * P <= 65535;
    for (int r = 0; r < rows && all_open; r++) {
        const SrRow& d = b->h_rows[(size_t)r];
        all_open = d.temperature > 0.0f && by_ratio(d) && !sr_row_cut(d) && !(d.top_k > 0 && d.top_k < V) && d.edit_cnt <= 0 && d.mask_row < 0;
    }
    int rc = all_open ? SR_OK : identity_list(ctx, rows * P, &list);
    if (all_open) {
        const size_t slots = (size_t)rows * (size_t)P;
        const int half_blocks = (nseg + SR_HALF_BLOCK_SEGS - 1) / SR_HALF_BLOCK_SEGS;
        full.seg_stride = nseg;
        full.chain_blocks = (half_blocks + 1) / 2;
        SR_HIP(ctx, ctx->full_state.reserve(slots * sizeof(SrFullState), st, true));
        SR_HIP(ctx, ctx->full_row_sync.reserve(slots * SR_ROW_SYNC_STRIDE * sizeof(unsigned long long), st, true));
        SR_HIP(ctx, ctx->full_seg_func.reserve(slots * (size_t)nseg * sizeof(SeqSegFunc), st));
        SR_HIP(ctx, ctx->full_chain_func.reserve(slots * 8 * (size_t)full.chain_blocks * sizeof(SeqSegFunc), st));
        SR_HIP(ctx, next_launch(ctx));
        full.state = ctx->full_state.as<SrFullState>();
        full.row_sync = ctx->full_row_sync.as<unsigned long long>();
        full.seg_func = (SeqSegFunc*)ctx->full_seg_func.p;
        full.chain_func = (SeqSegFunc*)ctx->full_chain_func.p;
        full.seq = ctx->full_seq;
        full.behind_wait_limit = ctx->behind_wait_limit;
    } else if (rc == SR_OK)
        rc = run_full(ctx, &tmp, list, rows * P, any_top_p, target_logits_dev, SR_DTYPE_F32, V, 1, ctx->spec_probs.as<float>(), p_stride,
                      nullptr, nullptr, true, &b->h_rows, 0, in_one ? &full : nullptr);  // (the verifier applies the normalising factors of unfiltered rows itself)
    tmp.d_rows.p = nullptr;  // borrowed
    tmp.d_edits.p = nullptr;
    if (rc != SR_OK) return rc;
    SrSpecArgs a{};
    a.rows = b->d_rows.as<SrRow>();
    a.vocab = V;
    a.n_draft = n_draft;
    a.p_all = ctx->spec_probs.as<float>();
    a.p_stride = p_stride;
    a.state = ctx->full_state.as<SrFullState>();
    a.target_logits = target_logits_dev;
    a.draft_probs = draft_probs_dev;
    a.draft_tokens = draft_tokens_dev;
    a.uniforms = sr_batch_uniforms(b);
    a.uniforms_per_row = b->upr;
    a.out_accepted = out_accepted_dev;
    a.out_tokens = out_tokens_dev;
    SR_HIP(ctx, ctx->spec_reject.reserve((size_t)rows * sizeof(int32_t), st));
    a.reject = ctx->spec_reject.as<int32_t>();
    a.seg_stride = (V + SR_SEG_TERMS - 1) / SR_SEG_TERMS;
    if (a.seg_stride <= SR_SEG_MAX) {
        SR_HIP(ctx, ctx->seg_part.reserve((size_t)rows * (size_t)a.seg_stride * sizeof(float), st));
        SR_HIP(ctx, ctx->seg_func.reserve((size_t)rows * (size_t)a.seg_stride * sizeof(SeqSegFunc), st));
        // (cleared when new, and when the launches' numbers have gone round: run_full)
        SR_HIP(ctx, ctx->spec_sync.reserve((size_t)rows * SR_ROW_SYNC_STRIDE * sizeof(unsigned long long), st, true));
        a.seg_part = ctx->seg_part.as<float>();
        a.seg_func = (SeqSegFunc*)ctx->seg_func.p;
        a.sync = ctx->spec_sync.as<unsigned long long>();
        a.seq = ctx->full_seq;
        a.wait_limit = ctx->behind_wait_limit;
    } else {  // (longer rows are added by their workgroups alone)
        a.resid_stride = ((int64_t)V + 3) & ~(int64_t)3;
        SR_HIP(ctx, ctx->spec_resid.reserve((size_t)rows * (size_t)a.resid_stride * sizeof(float), st));
        a.resid = ctx->spec_resid.as<float>();
    }
    for (int r = 0; r < rows; r++) {
        const SrRow& d = b->h_rows[(size_t)r];
        if (!by_ratio(d) || !(d.temperature > 0.0f)) a.any_other = 1;
    }
    if (full.factor_later || all_open) a.open_factors = &full;
    if (all_open) {
        a.all_open = 1;
        // as many positions side by side as the device holds workgroups beside the first ones': 16 x 8 of 20,011 and of 40,000 with two open in
        // a row 70 us -> 49 and 68 -> 47.  (Not more: 16 x 8 of 262,144, whose first ones fill it, 105 -> 92 where a row has two, but 44.6 -> 47.3
        // where none has.)
        const long long held = 2 * ctx->cu_count / std::max(1LL, (long long)rows * full.chain_blocks);
        a.open_side = (int)std::max(1LL, std::min({held, (long long)P, 4LL}));
        a.n_units = (V + SR_UNIT_TERMS - 1) / SR_UNIT_TERMS;
        const size_t units = (size_t)rows * (size_t)P * (size_t)a.n_units;
        SR_HIP(ctx, ctx->spec_units.reserve(units * sizeof(float2), st));
        SR_HIP(ctx, ctx->spec_unit_chains.reserve(units * 8 * sizeof(float), st));
        a.units = (float2*)ctx->spec_units.p;
        a.unit_chains = ctx->spec_unit_chains.as<float>();
    }
    SR_HIP(ctx, sr_launch_spec_verify(a, rows, st));
    return SR_OK;
}

int sr_mtp_verify_launch(sr_ctx* ctx, const float* logits_dev, int32_t rows, int32_t vocab, int64_t row_stride,
                         const int32_t* draft_tokens_dev, float p_min, int32_t* out_argmax_dev, int32_t* out_accept_dev,
                         float* out_prob_dev)
{
    if (!ctx) return SR_ERR_NULL_ARGUMENT;
    if (rows == 0) return SR_OK;
    if (!logits_dev || !draft_tokens_dev || !out_argmax_dev || !out_accept_dev)
        return sr_fail(ctx, SR_ERR_NULL_ARGUMENT, "sr_mtp_verify_launch: null tensor");
    if (rows < 0 || vocab <= 0 || row_stride < vocab) return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "sr_mtp_verify_launch: bad shape");
    SR_HIP(ctx, hipSetDevice(ctx->device));
    // p_min <= 0 means "argmax match only" (SamplingParams.SpecDraftPMin, Sampler.cs:791)
    const float pm = p_min > 0.0f ? p_min : 1.0f;
    SR_HIP(ctx, sr_launch_mtp_verify(logits_dev, row_stride, vocab, rows, draft_tokens_dev, pm, out_argmax_dev, out_accept_dev,
                                     out_prob_dev, ctx->stream));
    return SR_OK;
}

#ifdef SR_TEST_HOOKS
// Test hook (include/stingray_sampler_test.h): exact left-to-right sum of x_dev[0..n) from s0
int sr_selftest_seqsum(sr_ctx* ctx, const float* x_dev, int32_t n, float s0, float target, float* out_sum_dev,
                              int32_t* out_idx_dev)
{
    if (!ctx) return SR_ERR_NULL_ARGUMENT;
    SR_HIP(ctx, hipSetDevice(ctx->device));
    SR_HIP(ctx, sr_launch_selftest_seqsum(x_dev, n, s0, target, out_sum_dev, out_idx_dev, ctx->stream));
    return SR_OK;
}
// Test hook: the same sum as the whole device prepares it (segments' records made for predictions that are `skew`
// times the segments' true sums, the walk of one wave): out_sum_dev[0], out_idx_dev[0] from the sum and the search
// over its states, [1] from the walk that searches by itself
int sr_selftest_segsum(sr_ctx* ctx, const float* x_dev, int32_t n, double skew, float target, float* out_sum_dev,
                       int32_t* out_idx_dev)
{
    if (!ctx) return SR_ERR_NULL_ARGUMENT;
    if (n <= 0 || (n + SR_SEG_TERMS - 1) / SR_SEG_TERMS > SR_SEG_MAX) return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "sr_selftest_segsum: length");
    SR_HIP(ctx, hipSetDevice(ctx->device));
    const size_t nseg = (size_t)(n + SR_SEG_TERMS - 1) / SR_SEG_TERMS;
    SR_HIP(ctx, ctx->seg_part.reserve(nseg * sizeof(double), ctx->stream));
    SR_HIP(ctx, ctx->seg_func.reserve(nseg * sizeof(SeqSegFunc), ctx->stream));
    SR_HIP(ctx, sr_launch_selftest_segsum(x_dev, n, skew, target, ctx->seg_part.as<double>(), (SeqSegFunc*)ctx->seg_func.p,
                                          out_sum_dev, out_idx_dev, ctx->stream));
    return SR_OK;
}
// Test hook: the full-vocabulary rows of a batch, and then their last launch once more as if a workgroup of every row had stopped waiting at
// the row's first meeting, with `none` in the results
int sr_selftest_late_rows(sr_ctx* ctx, const sr_batch* b, const void* logits_dev, int dtype, int64_t row_stride, int32_t none, int32_t* out_tokens_dev,
                          uint32_t* out_flags_dev)
{
    if (!ctx || !b) return SR_ERR_NULL_ARGUMENT;
    const int n = (int)b->h_full_list.size();
    if (n != b->rows || b->full_greedy > 0 || !out_tokens_dev || !out_flags_dev)
        return sr_fail(ctx, SR_ERR_INVALID_ARGUMENT, "sr_selftest_late_rows: not a batch of sampled full-vocabulary rows");
    if (int rc = check_batch_call(ctx, b, logits_dev, dtype, row_stride, "sr_selftest_late_rows")) return rc;
    SR_HIP(ctx, hipSetDevice(ctx->device));
    bool any_top_p = false;
    for (const SrRow& r : b->h_rows) any_top_p = any_top_p || row_uses_top_p(r);
    SrFullArgs a{};
    if (int rc = run_full(ctx, b, b->d_full_list.as<int32_t>(), n, any_top_p, logits_dev, dtype, row_stride, 0, nullptr, 0, out_tokens_dev, out_flags_dev,
                          false, nullptr, 0, &a))
        return rc;
    std::vector<SrFullState> state((size_t)n);
    const std::vector<int32_t> nothing((size_t)n, none);
    SR_HIP(ctx, hipMemcpyAsync(state.data(), a.state, (size_t)n * sizeof(SrFullState), hipMemcpyDeviceToHost, ctx->stream));
    SR_HIP(ctx, hipStreamSynchronize(ctx->stream));
    for (SrFullState& s : state) { s.late = a.seq; s.deferred = 0u; }
    SR_HIP(ctx, hipMemcpyAsync(a.state, state.data(), (size_t)n * sizeof(SrFullState), hipMemcpyHostToDevice, ctx->stream));
    SR_HIP(ctx, hipMemcpyAsync(out_tokens_dev, nothing.data(), (size_t)n * sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream));
    SR_HIP(ctx, hipMemcpyAsync(out_flags_dev, nothing.data(), (size_t)n * sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream));
    SR_HIP(ctx, hipStreamSynchronize(ctx->stream));
    SR_HIP(ctx, sr_launch_full_row(a, n, ctx->stream));
    SR_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return SR_OK;
}
#endif  // SR_TEST_HOOKS

}  // extern "C"
