// The HIP runtime calls that the library's host code makes, on host memory, and its kernel launchers without kernels: linked
// with sr_api.cpp and sr_full_host.cpp they make a library of the host side alone, which tests drive without a GPU.
// Allocations are counted and can be made to fail; what a test asks about is kept in `seen`.
#include <cstdlib>
#include <cstring>
#include <map>

#include "../../opentail/stingray_amd/csrc/sr_kernels.h"

namespace {
std::map<void*, size_t> live;  // what hipMalloc and hipHostMalloc have handed out and not taken back
int fail_device = 0, fail_pinned = 0;
struct Seen {
    int64_t scan_builds, stream_waits, launches;
    const double* uniforms;
    const SrRow* rows;
} seen;

hipError_t take(void** p, size_t n, int fail)
{
    if (fail) { *p = nullptr; return hipErrorOutOfMemory; }
    *p = aligned_alloc(256, (n + 255) / 256 * 256 + 256);
    memset(*p, 0xee, n);
    live[*p] = n;
    return hipSuccess;
}
hipError_t give(void* p)
{
    if (p && live.erase(p) == 0) abort();  // (taken back twice, or never handed out)
    free(p);
    return hipSuccess;
}
}  // namespace

extern "C" {
void cpu_fail(int device, int pinned) { fail_device = device; fail_pinned = pinned; }
int64_t cpu_scan_builds() { return seen.scan_builds; }
int64_t cpu_stream_waits() { return seen.stream_waits; }
int64_t cpu_launches() { return seen.launches; }
const double* cpu_uniforms() { return seen.uniforms; }
int cpu_scan_row(int row) { return seen.rows[row].scan_row; }
// bytes of live memory from p on (0: p is in none)
int64_t cpu_live(const void* p)
{
    for (auto& b : live)
        if ((const char*)p >= (const char*)b.first && (const char*)p < (const char*)b.first + b.second)
            return (const char*)b.first + b.second - (const char*)p;
    return 0;
}

hipError_t hipMalloc(void** p, size_t n) { return take(p, n, fail_device); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return take(p, n, fail_pinned); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipHostFree(void* p) { return give(p); }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) { memset(p, 0, sizeof *p); p->multiProcessorCount = 256; return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "an error of the test's"; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t)
{
    for (size_t i = 0; i < h; i++) memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)0x10; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { seen.stream_waits++; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)0x20; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
}

static hipError_t launched() { seen.launches++; return hipSuccess; }
static hipError_t put(const SrCopyTable& t)
{
    for (int i = 0; i < t.n; i++) memcpy(t.seg[i].dst, t.seg[i].src, t.seg[i].bytes);
    return launched();
}
hipError_t sr_launch_scatter(const SrCopyTable& t, hipStream_t) { return put(t); }
hipError_t sr_launch_build_scan_mask(const SrScanDesc*, const int32_t*, int, const SrRow*, const SrEdit*, const uint32_t*, int64_t, uint32_t*,
                                     int64_t, int, int, int, int, unsigned long long, long long, const SrCopyTable* pieces, hipStream_t)
{
    seen.scan_builds++;
    return pieces ? put(*pieces) : launched();
}
hipError_t sr_launch_topk(const SrTopkArgs& a, int, hipStream_t) { seen.uniforms = a.uniforms; seen.rows = a.rows; return launched(); }
hipError_t sr_launch_full_prep(const SrFullArgs& a, int, hipStream_t) { seen.uniforms = a.uniforms; return launched(); }
hipError_t sr_launch_full_row(const SrFullArgs&, int, hipStream_t) { return launched(); }
hipError_t sr_launch_pack_allow_mask(const void*, int, int, int, int64_t, uint32_t*, int64_t, hipStream_t) { return launched(); }
hipError_t sr_launch_mask_and(uint32_t*, int64_t, const int32_t*, int, int, int, uint32_t*, hipStream_t) { return launched(); }
hipError_t sr_launch_apply_patches(SrRow*, const SrRowPatch*, int, SrEdit*, const SrEditPatch*, int, const SrMaskClear*, int, uint32_t*, int64_t, int,
                                   int, unsigned long long, long long, hipStream_t)
{
    return launched();
}
void sr_argmax_plan(SrArgmaxArgs&, int) {}
hipError_t sr_argmax_static_scratch(int, unsigned long long** best, uint32_t** done) { *best = nullptr; *done = nullptr; return hipSuccess; }
hipError_t sr_launch_argmax_rows(const SrArgmaxArgs&, bool, hipStream_t) { return launched(); }
hipError_t sr_launch_wide_keys(const SrFullArgs&, int, hipStream_t) { return launched(); }
hipError_t sr_launch_wide_adjust(const SrFullArgs&, int, hipStream_t) { return launched(); }
hipError_t sr_launch_wide_sort(const SrFullArgs&, int, int, hipStream_t) { return launched(); }
hipError_t sr_launch_wide_tail(const SrFullArgs&, int, hipStream_t) { return launched(); }
hipError_t sr_launch_draw_rows(const float*, int64_t, int, int, const double*, int*, hipStream_t) { return launched(); }
hipError_t sr_launch_residual_rows(const float*, int64_t, const float*, int64_t, int, int, const double*, int*, hipStream_t) { return launched(); }
hipError_t sr_launch_spec_verify(const SrSpecArgs&, int, hipStream_t) { return launched(); }
hipError_t sr_launch_expand_rows(const SrRow*, SrRow*, int, int, hipStream_t) { return launched(); }
hipError_t sr_launch_mtp_verify(const float*, int64_t, int, int, const int*, float, int*, int*, float*, hipStream_t) { return launched(); }
