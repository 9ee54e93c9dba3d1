// Row-wise argmax: Sampler.Greedy (Sampler.cs:442-446) for a [rows x vocab] tensor, the counterpart of
// the reference's llm_argmax_rows (CudaTextKernels.cs:465-479).  Lowest index wins on equal values; a NaN
// element wins outright (first NaN), as TensorPrimitives.IndexOfMax documents.
//
// One launch, grid = rows x chunks.  A workgroup streams its chunk with 16-byte loads (up to eight in
// flight per thread), reduces it to a packed (key << 32 | ~index) and, when the row has more than one chunk,
// folds that into the row's slot with a 64-bit atomic max and counts itself in; the workgroup that counts in
// last writes the row's result and puts slot and counter back to zero, so the scratch of one launch is ready
// for the next without a fill.  Rows of one chunk write their result directly.
//
// This file also holds the scratch of the entry point that allocates nothing: a zero-initialised array in
// device memory that belongs to the library's code object, one copy per GPU.
#include <algorithm>

#include "sr_device.h"
#include "sr_kernels.h"
#include "sr_types.h"

// best[SR_ARGMAX_STATIC_ROWS] (8 bytes each) followed by done[SR_ARGMAX_STATIC_ROWS] (4 bytes each): 192 KiB.
// In host code this name is only a handle for hipGetSymbolAddress, never an address to give a kernel.
static __device__ __align__(256) unsigned long long scratch[SR_ARGMAX_STATIC_ROWS + SR_ARGMAX_STATIC_ROWS / 2];

namespace {
constexpr int kThreads = 256;
constexpr int kUnroll = 4;

typedef uint32_t __attribute__((ext_vector_type(4))) u32x4;

constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices];  // per device: where that device's copy of `scratch` lies

__global__ void k_fill_u32(uint32_t* p, int n, uint32_t v)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

template <int ES> __device__ __forceinline__ float load_elem(const char* p, int64_t i)
{
    if (ES == 4) return ((const float*)p)[i];
    return sr_bf16_to_f32(((const uint16_t*)p)[i]);
}

// An element's order as a signed whole number, the same way back: the bits of a negative number turned round.  +0 is just above -0
// (sr_okey makes them the same), a positive NaN above +inf, a negative one below -inf.
__device__ __forceinline__ uint32_t turned(uint32_t x) { return x ^ ((uint32_t)((int)x >> 31) & 0x7fffffffu); }
typedef short __attribute__((ext_vector_type(2))) i16x2;
__device__ __forceinline__ i16x2 as_i16x2(uint32_t x) { return __builtin_bit_cast(i16x2, x); }
__device__ __forceinline__ i16x2 turned2(uint32_t x)  // two bf16 elements at once
{
    return as_i16x2(x ^ (__builtin_bit_cast(uint32_t, as_i16x2(x) >> (short)15) & 0x7fff7fffu));
}
// What a tile of a thread's vectors holds: its largest and its smallest element in that order.
template <int ES> struct Span;
template <> struct Span<4> {
    int hi, lo;
    __device__ __forceinline__ void start(const u32x4& t) { hi = lo = (int)turned(t[0]); }
    __device__ __forceinline__ void fold(const u32x4& t)
    {
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const int k = (int)turned(t[w]);
            hi = max(hi, k);
            lo = min(lo, k);
        }
    }
    __device__ __forceinline__ int largest() const { return hi; }
    __device__ __forceinline__ bool nan() const { return hi > 0x7f800000 || lo < (int)0x807fffffu; }
};
template <> struct Span<2> {
    i16x2 hi, lo;
    __device__ __forceinline__ void start(const u32x4& t) { hi = lo = turned2(t[0]); }
    __device__ __forceinline__ void fold(const u32x4& t)
    {
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const i16x2 k = turned2(t[w]);
            hi = __builtin_elementwise_max(hi, k);
            lo = __builtin_elementwise_min(lo, k);
        }
    }
    __device__ __forceinline__ int largest() const { return max((int)hi[0], (int)hi[1]); }
    __device__ __forceinline__ bool nan() const { return largest() > 0x7f80 || min((int)lo[0], (int)lo[1]) < (int)(short)0x807f; }
};
// element e of a vector as the bits of an fp32 number
template <int ES> __device__ __forceinline__ uint32_t bits_of(const u32x4& t, int e)
{
    if (ES == 4) return t[e];
    return (e & 1) ? t[e >> 1] & 0xffff0000u : t[e >> 1] << 16;
}
__device__ __forceinline__ bool is_nan_bits(uint32_t x) { return (x & 0x7fffffffu) > 0x7f800000u; }

// kAligned: the rows start on 16-byte boundaries.  What bounds it: memory, where there is enough of it; a launch over little waits for
// its first vectors and for its chunks to come together.  Two tiles of four vectors a thread in turn, the loads of one under the
// folding of the other, two and a half (bf16, in pairs) and four instructions an element; an element's index is looked for only
// where a wave's tile holds more than its tiles before.  Against eight or nine instructions an element, key and index carried along, a
// tile of eight at a time, and element by element in rows at odd addresses, whole calls with host results one behind the other, four buffers
// in turn, both kernels on one card, us: 128 rows of 151,936 bf16 23.2 -> 19.6, 256 30.6 -> 25.8, 1 15.6 -> 13.6, 512 44.1 -> 35.6; 64 rows
// of 100,003 bf16 35.3 -> 17.4, 300 of 100,003 fp32 113 -> 35.8, 1,024 of 20,011 bf16 42.7 -> 21.1.
// (In a run of its own, 128 rows: tiles of eight 27, of six 26.7, of two and three as of four; three to six workgroups to a compute unit
// 24.6 - 25.4 where two took 24.8.  With four instructions an element in the search for the index, in place of two, 24.8.)
template <int ES, bool kAligned> __global__ __launch_bounds__(kThreads) void k_argmax_rows(SrArgmaxArgs a)
{
    __shared__ unsigned long long s_best[kThreads / SR_WAVE];
    constexpr int EPV = 16 / ES;
    const int row = __builtin_amdgcn_readfirstlane((int)(blockIdx.x / (unsigned)a.chunks));
    const int c = (int)blockIdx.x - row * a.chunks;
    const int lo = c * a.chunk_len, hi = min(a.vocab, lo + a.chunk_len);
    const char* rowp = (const char*)a.logits + (size_t)row * (size_t)a.row_stride * ES;
    const int tid = (int)threadIdx.x;
    unsigned long long best = 0ull;  // of the wave: key << 32 | ~index (NaN above everything); 0: no element yet
    const int v_lo = lo / EPV, v_hi = hi / EPV;  // whole vectors; only the row's last chunk can leave elements over
    if (v_lo < v_hi) {
        // (a vector past the chunk's end is the chunk's last one again)
        const int last = v_hi - 1;
        auto load = [&](int base, u32x4 (&t)[kUnroll]) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < kUnroll; j++) {
                const char* const at = rowp + (size_t)min(base + tid + j * kThreads, last) * 16;
                if (kAligned) {
                    t[j] = __builtin_nontemporal_load((const u32x4*)at);
                } else {
                    const uint4 v = sr_load16<ES>(at);
                    t[j] = u32x4{v.x, v.y, v.z, v.w};
                }
            }
        };
        auto fold = [&](int base, const u32x4 (&t)[kUnroll]) __attribute__((always_inline)) {
            Span<ES> s;
            s.start(t[0]);
#pragma unroll
            for (int j = 0; j < kUnroll; j++) s.fold(t[j]);
            const bool nan = __ballot(s.nan()) != 0ull;
            const uint32_t k = sr_wave_max_u32((uint32_t)s.largest() ^ 0x80000000u) ^ 0x80000000u;
            // the largest element's bits, and its key
            const uint32_t bits = ES == 4 ? turned(k) : (k ^ ((uint32_t)((int)k >> 31) & 0x7fffu)) << 16;
            const uint32_t key = nan ? 0xffffffffu : sr_okey(sr_u2f(bits));
            if (key <= (uint32_t)(best >> 32)) return;  // (of equal ones the first stays: its index is lower)
            // (from the last to the first: a comparison and a selection each)
            int code = -1;
            if (nan || (bits << 1) == 0u) {  // (a zero is as large with either sign)
#pragma unroll
                for (int j = kUnroll - 1; j >= 0; j--)
#pragma unroll
                    for (int e = EPV - 1; e >= 0; e--) {
                        const uint32_t x = bits_of<ES>(t[j], e);
                        code = (nan ? is_nan_bits(x) : (x << 1) == 0u) ? j * EPV + e : code;
                    }
            } else {
                const uint32_t half = bits >> 16;
#pragma unroll
                for (int j = kUnroll - 1; j >= 0; j--)
#pragma unroll
                    for (int e = EPV - 1; e >= 0; e--) {
                        const bool is = ES == 4 ? t[j][e] == bits : ((e & 1) ? t[j][e >> 1] >> 16 : t[j][e >> 1] & 0xffffu) == half;
                        code = is ? j * EPV + e : code;
                    }
            }
            uint32_t at = code < 0 ? 0xffffffffu : (uint32_t)min(base + tid + (code / EPV) * kThreads, last) * EPV + (uint32_t)(code % EPV);
            at = ~sr_wave_max_u32(~at);
            best = ((unsigned long long)key << 32) | (unsigned long long)(0xffffffffu - at);
        };
        constexpr int kStep = kUnroll * kThreads;
        u32x4 t0[kUnroll], t1[kUnroll];
        load(v_lo, t0);
        for (int base = v_lo; base < v_hi; base += 2 * kStep) {
            if (base + kStep < v_hi) load(base + kStep, t1);
            fold(base, t0);
            if (base + 2 * kStep < v_hi) load(base + 2 * kStep, t0);
            if (base + kStep < v_hi) fold(base + kStep, t1);
        }
    }
    {
        // the elements behind the row's last whole vector
        const int i = max(lo, v_hi * EPV) + tid;
        unsigned long long own = 0ull;
        if (i < hi) {
            const float v = load_elem<ES>(rowp, i);
            own = ((unsigned long long)(v != v ? 0xffffffffu : sr_okey(v)) << 32) | (unsigned long long)(0xffffffffu - (uint32_t)i);
        }
        if (max(lo, v_hi * EPV) < hi) {  // (fewer than a vector's: one each)
            own = sr_wave_max_u64(own);
            best = own > best ? own : best;
        }
    }

    // (key << 32 | ~index): the largest key wins, among equal keys the lowest index
    if (sr_lane() == 0) s_best[sr_wave_id()] = best;
    __syncthreads();
    if (tid != 0) return;
    for (int w = 1; w < kThreads / SR_WAVE; w++) best = s_best[w] > best ? s_best[w] : best;
    if (a.chunks > 1) {
        // Both are device-scope atomics without a fence (a release fence would write back the whole L2): the maximum
        // is waited for -- its old value comes back -- before the chunk is counted in, so whoever counts in last
        // finds every chunk's maximum in the slot.
        const unsigned long long seen = __hip_atomic_fetch_max(&a.best[row], best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" : : "v"(seen) : "memory");
        const uint32_t before = __hip_atomic_fetch_add(&a.done[row], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (before != (uint32_t)a.chunks - 1u) return;
        best = __hip_atomic_load(&a.best[row], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&a.best[row], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&a.done[row], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const int idx = best ? (int)(0xffffffffu - (uint32_t)(best & 0xffffffffull)) : 0;  // empty row -> 0
    // the original bits: the key's, the same way back; a NaN's and a zero's are fetched (a trip to memory of its own)
    const uint32_t key = (uint32_t)(best >> 32);
    const float val = best == 0ull ? 0.0f : key == 0xffffffffu || key == 0x80000000u ? load_elem<ES>(rowp, idx) : sr_okey_inv(key);
    if (a.host) {
        // The host goes on when it sees its word, in front of this kernel's end: what the device arrays get is written through
        // to memory, not left in this die's L2 for the kernel's end to write back, and waited for, before the word goes out.
        // Whoever reads the arrays behind the call, on whatever stream, finds the results there, and nothing is stored any
        // more to arrays that the caller gives away.  (Two stores and a wait of one thread per row: a call over 128 rows of
        // 151,936 bf16 takes 24.7 us, 24.5 with plain stores behind the word; with a wait for the stream instead it takes 28.6.)
        if (a.out_idx) __hip_atomic_store(&a.out_idx[row], idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (a.out_val) __hip_atomic_store(&a.out_val[row], val, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        // (one store, seen by the host as a whole)
        __hip_atomic_store(&a.host[row], ((unsigned long long)sr_f2u(val) << 32) | (unsigned long long)(uint32_t)idx, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
        return;
    }
    if (a.out_idx) a.out_idx[row] = idx;
    if (a.out_val) a.out_val[row] = val;
}

#ifdef SR_TEST_HOOKS
__global__ void k_selftest_expf(const float* x, float* y, int64_t n)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = sr_expf(x[i]);
}
#endif
}  // namespace

void sr_argmax_plan(SrArgmaxArgs& a, int cu_count)
{
    const int es = a.dtype == 1 ? 2 : 4, epv = 16 / es;
    a.vec = ((uintptr_t)a.logits % 16 == 0 && ((size_t)a.row_stride * es) % 16 == 0) ? 1 : 0;
    // enough workgroups for two per compute unit (64 KB of loads in flight on each, two tiles a thread: what the memory's latency takes at
    // the machine's rate; eight per compute unit, with their dispatch and their atomics, were 5 us slower on 256 rows of
    // 151,936), none with less than one unrolled pass of work
    const int per_pass = kThreads * kUnroll * epv;
    int s = std::max(1, std::min((2 * cu_count + a.rows - 1) / std::max(a.rows, 1), a.vocab / per_pass));
    int len = (a.vocab + s - 1) / s;
    len = (len + epv - 1) / epv * epv;
    a.chunk_len = std::max(len, epv);
    a.chunks = a.vocab > 0 ? (a.vocab + a.chunk_len - 1) / a.chunk_len : 1;
}

hipError_t sr_launch_argmax_rows(const SrArgmaxArgs& a, bool clear_first, hipStream_t stream)
{
    if (a.rows <= 0) return hipSuccess;
    if (clear_first && a.chunks > 1) {
        // best and done are separate arrays: clear each where it is
        hipLaunchKernelGGL(k_fill_u32, dim3((2 * a.rows + 255) / 256), dim3(256), 0, stream, (uint32_t*)a.best, 2 * a.rows, 0u);
        hipLaunchKernelGGL(k_fill_u32, dim3((a.rows + 255) / 256), dim3(256), 0, stream, a.done, a.rows, 0u);
    }
    const dim3 grid((unsigned)a.rows * (unsigned)a.chunks), block(kThreads);
    if (a.dtype == 1) {
        if (a.vec) hipLaunchKernelGGL((k_argmax_rows<2, true>), grid, block, 0, stream, a);
        else hipLaunchKernelGGL((k_argmax_rows<2, false>), grid, block, 0, stream, a);
    } else {
        if (a.vec) hipLaunchKernelGGL((k_argmax_rows<4, true>), grid, block, 0, stream, a);
        else hipLaunchKernelGGL((k_argmax_rows<4, false>), grid, block, 0, stream, a);
    }
    return hipGetLastError();
}

// The address of the current device's copy of the static scratch, looked up once per device.
hipError_t sr_argmax_static_scratch(int device, unsigned long long** best, uint32_t** done)
{
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    void* p = __atomic_load_n(&g_scratch_ptr[device], __ATOMIC_ACQUIRE);
    if (!p) {
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        __atomic_store_n(&g_scratch_ptr[device], p, __ATOMIC_RELEASE);
    }
    *best = (unsigned long long*)p;
    *done = (uint32_t*)((unsigned long long*)p + SR_ARGMAX_STATIC_ROWS);
    return hipSuccess;
}

#ifdef SR_TEST_HOOKS
hipError_t sr_launch_selftest_expf(const float* x, float* y, int64_t n, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_selftest_expf, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, x, y, n);
    return hipGetLastError();
}
#endif
