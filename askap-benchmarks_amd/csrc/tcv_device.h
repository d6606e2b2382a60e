// Device code shared by the tiled gridding and degridding kernels: buffer and
// scalar loads, the tap formats, wave reductions and the work-item source.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "tcv_internal.h"

namespace {

constexpr unsigned kOOB = 0x80000000u;  // byte offset beyond any C buffer we accept

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *p, unsigned bytes)
{
    // word3 0x00020000: raw 32-bit buffer format used for untyped loads on gfx9.
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, 0x00020000);
}

// Load of wave-uniform data that no wave writes while the kernel runs (work
// items, entries, visibilities, plane scales).  Through the constant address
// space the compiler issues a scalar (SMEM) load into SGPRs, instead of a
// vector load, a wait for it and readfirstlane.
template <typename T>
__device__ __forceinline__ T cload(const T *p, int i)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return ((const __attribute__((address_space(4))) T *)p)[i];
#else
    return p[i];   // the host pass only parses device functions
#endif
}

// a * b for 0 <= a, b < 2^24, b wave-uniform: the full-rate 24-bit multiply,
// written as the instruction so that the compiler cannot fold it into a
// neighbouring expression as a quarter-rate 32- or 64-bit multiply
__device__ __forceinline__ int umul24(int a, int b)
{
    int r;
    asm("v_mul_u32_u24 %0, %1, %2" : "=v"(r) : "s"(b), "v"(a));
    return r;
}

// a * b + c (24-bit unsigned a, b; b wave-uniform)
__device__ __forceinline__ unsigned umad24(int a, int b, unsigned c)
{
    unsigned r;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    return r;
}

// a * b + c (24-bit signed a, b; b wave-uniform)
__device__ __forceinline__ unsigned imad24(int a, int b, unsigned c)
{
    unsigned r;
    asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    return r;
}

__device__ __forceinline__ float2 load_c(__amdgpu_buffer_rsrc_t r, unsigned voff)
{
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, 0, 0));
}


// Sum over each 16-lane row of a wave (all lanes must be active): four DPP steps
// leave every lane with its row's sum.
__device__ __forceinline__ float row_sum(float x)
{
    auto dpp = [](float v, auto ctrl) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
            0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xF, 0xF, false));
    };
    x += dpp(x, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
    x += dpp(x, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
    x += dpp(x, std::integral_constant<int, 0x141>{});  // row_half_mirror
    x += dpp(x, std::integral_constant<int, 0x140>{});  // row_mirror
    return x;
}

// Sum over the 64 lanes: the row sums, combined by four readlanes.  The result
// is wave-uniform.
__device__ __forceinline__ float wave_sum(float x)
{
    const int xi = __builtin_bit_cast(int, row_sum(x));
    const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(xi, 0));
    const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(xi, 16));
    const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(xi, 32));
    const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(xi, 48));
    return (r0 + r1) + (r2 + r3);
}

// ---- tap storage ---------------------------------------------------------------
// FP32: complex64 taps (8 B).  FP16: (re, im) half pairs (4 B) scaled by the
// max-abs of their w-plane; accumulation stays FP32.
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

template <bool HALF>
struct Taps;

template <>
struct Taps<false> {
    static constexpr unsigned kBytes = 8;
    __device__ static __forceinline__ float2 load(__amdgpu_buffer_rsrc_t r, unsigned voff)
    {
        return load_c(r, voff);
    }
};

template <>
struct Taps<true> {
    static constexpr unsigned kBytes = 4;
    __device__ static __forceinline__ float2 load(__amdgpu_buffer_rsrc_t r, unsigned voff)
    {
        const half2_t h = __builtin_bit_cast(half2_t, __builtin_amdgcn_raw_buffer_load_b32(r, voff, 0, 0));
        return make_float2((float)h.x, (float)h.y);
    }
};

// Two consecutive taps (one 16-byte load for FP32, 8 bytes for FP16): the
// vector memory path moves data per group of four lanes, so wider loads carry
// twice the taps per unit of L1 throughput.
template <bool HALF>
__device__ __forceinline__ float4 load_pair(__amdgpu_buffer_rsrc_t r, unsigned voff)
{
    if constexpr (!HALF) {
        return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
    } else {
        const uint2 u = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, 0, 0));
        const half2_t a = __builtin_bit_cast(half2_t, u.x), b = __builtin_bit_cast(half2_t, u.y);
        return make_float4((float)a.x, (float)a.y, (float)b.x, (float)b.y);
    }
}

// Four consecutive FP16 taps in one 16-byte load.
struct Quad {
    float2 t0, t1, t2, t3;
};

__device__ __forceinline__ float2 half_tap(unsigned w)
{
    const half2_t h = __builtin_bit_cast(half2_t, w);
    return make_float2((float)h.x, (float)h.y);
}

__device__ __forceinline__ Quad load_quad_half(__amdgpu_buffer_rsrc_t r, unsigned voff)
{
    const uint4 u = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
    return Quad{half_tap(u.x), half_tap(u.y), half_tap(u.z), half_tap(u.w)};
}

// a or b by a lane-dependent flag, as a bit blend: a plain select of two
// struct members can be rewritten by the compiler into an indexed load from
// the stack, which would put the quadruples in scratch memory
__device__ __forceinline__ float blend(bool pickB, float a, float b)
{
    const unsigned m = 0u - (unsigned)pickB;
    return __uint_as_float((__float_as_uint(a) & ~m) | (__float_as_uint(b) & m));
}

// tap i of a quadruple for a lane-dependent i in [0, 4)
__device__ __forceinline__ float2 pick4(const Quad &q, int i)
{
    const bool lo = i & 1, hi = i & 2;
    const float ax = blend(lo, q.t0.x, q.t1.x), ay = blend(lo, q.t0.y, q.t1.y);
    const float bx = blend(lo, q.t2.x, q.t3.x), by = blend(lo, q.t2.y, q.t3.y);
    return make_float2(blend(hi, ax, bx), blend(hi, ay, by));
}

__device__ __forceinline__ int entry_width(int w) { return w & 0xFFFF; }
__device__ __forceinline__ int entry_plane(const int4 &en, const JobDesc &d)
{
    return d.planeTaps > 0 ? en.y / d.planeTaps : (int)((unsigned)en.w >> 16);
}

template <bool HALF>
__device__ __forceinline__ float2 vis_value(const JobDesc &d, const int4 &en)
{
    if constexpr (!HALF) {
        if (!d.data) return make_float2(1.f, 0.f);   // PSF gridding: data == 1 + 0i
        return cload(static_cast<const float2 *>(d.data), en.z);
    } else {
        const half2_t v = cload(static_cast<const half2_t *>(d.data), en.z);
        const float sc = d.dataScale * cload(d.planeScale, entry_plane(en, d));
        return make_float2((float)v.x * sc, (float)v.y * sc);
    }
}

// Work-item source of the persistent kernels: one job (descriptor passed by
// value) or a batch (descriptors in device memory, located through the
// exclusive prefix sum of the jobs' item counts).
template <bool BATCH>
struct ItemSource {
    JobDesc one;
    const JobDesc *jobs;
    const int *prefix;
    int nJobs;
    int *queue;

    // Single job: items are XCD-major with per-XCD queues.  Batch: each XCD
    // walks its share of every job in job order (per-XCD prefix sums after the
    // job prefix, counters at queue[kHeadInts (1 + q)]), then takes from the others.
    int xcd;
    int *bcast;   // one slot per workgroup (kernels that keep LDS for their tile)

    __device__ __forceinline__ int total() const
    {
        if constexpr (BATCH) return __builtin_amdgcn_readfirstlane(prefix[nJobs]);
        else return __builtin_amdgcn_readfirstlane(one.meta[0]);
    }
    // XCD q's share of the items and its i-th item
    __device__ __forceinline__ int share(int q) const
    {
        if constexpr (BATCH) return prefix[(nJobs + 1) * (1 + q) + nJobs];
        else return one.meta[17 + q] - one.meta[16 + q];
    }
    __device__ __forceinline__ int item_of(int q, int i) const
    {
        if constexpr (BATCH) {
            const int *px = prefix + (nJobs + 1) * (1 + q);
            int lo = 0, hi = nJobs;   // px[lo] <= i < px[hi]
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (px[mid] <= i) lo = mid; else hi = mid;
            }
            return prefix[lo] + jobs[lo].meta[16 + q] + (i - px[lo]);
        } else {
            return one.meta[16 + q] + i;
        }
    }
    // Next work item (one lane calls this); >= total() when none is left.  The
    // queues start after the workgroups' first items (first_item), so a list of
    // no more items than workgroups takes no atomics (378 items, 1024 workgroups:
    // gridding 85 us with, 74 without).
    __device__ __forceinline__ int acquire() const
    {
        if (!xcd) return (int)gridDim.x + atomicAdd(queue, 1);
        // own XCD first (hardware XCC_ID register), then steal from the others
        const int x0 = (int)(__builtin_amdgcn_s_getreg((3 << 11) | 20) & 7);
        for (int k = 0; k < 8; ++k) {
            const int q = (x0 + k) & 7;
            const int tot = share(q), taken = ((int)gridDim.x + 7 - q) >> 3;
            if (tot <= taken) continue;
            int *head = BATCH ? queue + kHeadInts * (1 + q) : one.meta + 32 + kHeadInts * q;
            const int i = taken + atomicAdd(head, 1);
            if (i < tot) return item_of(q, i);
        }
        return 0x7fffffff;
    }
    // A workgroup's first item: its own number, or its place in the share of the XCD
    // that workgroups are dealt to in turn (any other deal costs locality alone).
    __device__ __forceinline__ int first() const
    {
        if (!xcd) return (int)blockIdx.x;
        const int q = blockIdx.x & 7, i = blockIdx.x >> 3;
        return i < share(q) ? item_of(q, i) : acquire();
    }
    // item -> (job descriptor, local item index); wave-uniform
    __device__ __forceinline__ void locate(int item, JobDesc &d, int &local) const
    {
        if constexpr (BATCH) {
            int lo = 0, hi = nJobs;   // prefix[lo] <= item < prefix[hi]
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (__builtin_amdgcn_readfirstlane(prefix[mid]) <= item) lo = mid; else hi = mid;
            }
            d = jobs[lo];
            local = item - __builtin_amdgcn_readfirstlane(prefix[lo]);
        } else {
            d = one;
            local = item;
        }
    }
};

// Next work item for the whole workgroup without spending LDS: thread 0
// publishes the item it acquired during the previous one (`next`, taken from
// the queue one item ahead so that the queue's latency overlaps the work) in
// the workgroup's slot and acquires the following one.  Waiting for its memory
// counters completes the store in the CU's L2 before the barrier (a
// device-scope fence would also write back the L2), and the waves, all on the
// same CU, read the slot from that L2.  The caller reaches another barrier
// before thread 0 publishes again, so no wave can miss a value.  Every item
// acquired is processed: the loop ends on the first one past the end.
template <bool BATCH>
__device__ __forceinline__ int acquire_for_block(const ItemSource<BATCH> &src, int &next, int nItems)
{
    if (threadIdx.x == 0) {
        __hip_atomic_store(src.bcast + blockIdx.x, next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_waitcnt(0);   // every counter of this wave drained
    }
    __syncthreads();
    const int item = __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(src.bcast + blockIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    if (threadIdx.x == 0 && item < nItems) next = src.acquire();
    return item;
}

// The first item of a workgroup (thread 0 only; see acquire_for_block).
template <bool BATCH>
__device__ __forceinline__ int first_item(const ItemSource<BATCH> &src)
{
    return threadIdx.x == 0 ? src.first() : 0;
}

}  // namespace
