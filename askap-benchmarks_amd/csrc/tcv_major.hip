// Major-cycle neighbours of the gridder on the device
// (current/tMajorACC/tMajorACC.cc): the shifted 2-D FFT (fftExec), fftFix,
// Hogbom CLEAN (findPeak / subtractPsf / deconvolve) and the visibility
// subtraction.  Everything stays resident in HBM; the Hogbom loop runs without
// a host round trip per iteration.
#include <hip/hip_runtime.h>
#include <hipfft/hipfft.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string>

#include "tcv_internal.h"

namespace {

// ---- shifted FFT ----------------------------------------------------------------
// fftExec rotates the grid by g/2 on both axes, transforms, and rotates back
// (tMajorACC.cc:509-535).  For an even square grid that composition equals
// M . F . M, where M multiplies pixel (x, y) by (-1)^(x+y): rolling by g/2
// before a length-g DFT multiplies bin k by (-1)^k, and rolling after it is
// the DFT of the (-1)^n-modulated input times (-1)^(g/2); on a square grid the
// two (-1)^(g/2) factors cancel.  M is exact (a sign flip), so the shifts cost
// one in-place pass each instead of two copies through a second buffer.
// mode 0: x *= M; mode 1: x = M*x with fftFix folded in (real * scale, imag 0).
__global__ __launch_bounds__(256) void k_checker(float2 *__restrict__ g, int gSize, int mode,
                                                 float scale)
{
    const int y = blockIdx.y;
    const int x0 = (blockIdx.x * blockDim.x + threadIdx.x) * 2;
    if (x0 >= gSize) return;
    float4 *p = reinterpret_cast<float4 *>(g + (size_t)y * gSize + x0);   // gSize even
    float4 v = *p;
    const float s = ((x0 + y) & 1) ? -1.f : 1.f;   // pixel x0; x0 + 1 has the other sign
    if (mode == 0) {
        v.x *= s;
        v.y *= s;
        v.z = -s * v.z;
        v.w = -s * v.w;
    } else {
        v.x = (s * v.x) * scale;
        v.y = 0.f;
        v.z = (-s * v.z) * scale;
        v.w = 0.f;
    }
    *p = v;
}

// fftFix on its own: grid = real(grid) * scale (tMajorACC.cc:620-627).
__global__ __launch_bounds__(256) void k_fft_fix(float2 *__restrict__ g, long long n, float scale)
{
    long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        float2 v = g[i];
        g[i] = make_float2(v.x * scale, 0.f);
    }
}

// data -= model (tMajorACC.cc:1549-1556), complex, 16 B per thread per step.
__global__ __launch_bounds__(256) void k_vis_subtract(float2 *__restrict__ d,
                                                      const float2 *__restrict__ m, long long n)
{
    long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        const float2 a = d[i], b = m[i];
        d[i] = make_float2(a.x - b.x, a.y - b.y);
    }
}

// ---- Hogbom ------------------------------------------------------------------------
// findPeak picks the first pixel of largest |re| (tMajorACC.cc:689-701).  A
// 64-bit key orders pixels the same way under an unsigned max: |v|'s bits (31,
// non-negative floats order like their bit patterns), then the complemented
// index (smaller index wins a tie), then the sign of v (so the signed value
// can be rebuilt from the winning key).  One atomicMax per workgroup.
__device__ __forceinline__ unsigned long long peak_key(float v, unsigned idx)
{
    const unsigned a = __float_as_uint(v) & 0x7fffffffu;
    return ((unsigned long long)a << 33) | ((unsigned long long)(~idx) << 1) |
           (unsigned long long)(v < 0.f ? 1u : 0u);
}
__device__ __forceinline__ unsigned key_index(unsigned long long k)
{
    return ~(unsigned)((k >> 1) & 0xffffffffull);
}
__device__ __forceinline__ float key_value(unsigned long long k)
{
    const float a = __uint_as_float((unsigned)(k >> 33));
    return (k & 1ull) ? -a : a;
}

__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long k)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long t = __shfl_xor(k, o, 64);
        k = t > k ? t : k;
    }
    return k;
}

// workgroup max of k, then one atomicMax into *out (256 threads)
__device__ __forceinline__ void block_peak(unsigned long long k, unsigned long long *out)
{
    __shared__ unsigned long long s[4];
    k = wave_max_u64(k);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) s[wave] = k;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long m = s[0];
        for (int w = 1; w < 4; ++w) m = s[w] > m ? s[w] : m;
        if (m) atomicMax(out, m);
    }
}

// the residual's real plane back into the complex image
__global__ __launch_bounds__(256) void k_real_writeback(float2 *__restrict__ dst,
                                                        const float *__restrict__ src, long long n)
{
    long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) dst[i].x = src[i];
}

struct HogbomArgs {
    float *res;                  // residual real plane, W x W
    const float *psf;            // PSF real plane, PW x PW
    float2 *model;               // complex model image, W x W
    unsigned long long *keys;    // [0..2] rotating residual peaks, [3] PSF peak
    int W, PW;
    float gain;
};

// One Hogbom iteration (tMajorACC.cc:823-838) fused with the next findPeak:
// reads the residual peak of iteration i from keys[i % 3], adds gain * peak to
// the model, subtracts gain * peak * PSF over the overlap (subtractPsf,
// tMajorACC.cc:723-750, including its row offset diffy = ry - px), and
// reduces the updated residual's peak into keys[(i + 1) % 3].  keys[(i + 2) % 3]
// (read by iteration i - 1, written by iteration i + 1) is cleared here.
// Arithmetic is rounded exactly as the reference's float expressions.
template <bool VEC>
__global__ __launch_bounds__(256) void k_hogbom_step(HogbomArgs a, int i)
{
    // no fused multiply-add: each product and difference is rounded on its own,
    // as in the reference's float expressions (plain operators under this
    // pragma; helpers defined elsewhere would carry their own contract flags)
#pragma clang fp contract(off)
    const unsigned long long kc = a.keys[i % 3];
    const unsigned long long kp = a.keys[3];
    const float peak = key_value(kc);
    const int W = a.W, PW = a.PW;
    const unsigned pos = key_index(kc), ppos = key_index(kp);
    const int rx = (int)(pos % (unsigned)W), ry = (int)(pos / (unsigned)W);
    const int px = (int)(ppos % (unsigned)PW), py = (int)(ppos / (unsigned)PW);
    const int diffx = rx - px, diffy = ry - px;   // as in the reference
    const int startx = max(0, rx - px), starty = max(0, ry - py);
    const int stopx = min(W - 1, rx + (PW - px - 1)), stopy = min(W - 1, ry + (PW - py - 1));
    const float amp = a.gain * peak;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        a.model[pos].x = a.model[pos].x + peak * a.gain;
        a.keys[(i + 2) % 3] = 0ull;
    }
    // rows split over blockIdx.y, columns over blockIdx.x: no per-pixel division.
    // kRows rows a step, all their loads issued before any use, so that a
    // thread has that many reads in flight (one at a time left it waiting on
    // memory latency row after row).
    constexpr int kRows = 8;
    unsigned long long best = 0;
    if constexpr (VEC) {
        // W % 4 == 0: four adjacent pixels a thread, one 16-byte residual load
        // and store per row (the PSF row is read per pixel: any alignment)
        for (int x4 = (blockIdx.x * 256 + threadIdx.x) * 4; x4 < W; x4 += gridDim.x * 1024) {
            for (int y0 = blockIdx.y; y0 < W; y0 += gridDim.y * kRows) {
                float4 v[kRows];
                float pv[kRows][4];
                bool sub[kRows][4];
#pragma unroll
                for (int u = 0; u < kRows; ++u) {
                    const int y = y0 + u * (int)gridDim.y;
                    const int sy = y - diffy;
                    const bool rowOk = y < W;
                    const bool rowSub = rowOk && y >= starty && y <= stopy && sy >= 0 && sy < PW;
                    v[u] = rowOk ? *reinterpret_cast<const float4 *>(a.res + (size_t)y * W + x4)
                                 : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const int x = x4 + c;
                        sub[u][c] = rowSub && x >= startx && x <= stopx;
                        pv[u][c] = sub[u][c] ? a.psf[(ptrdiff_t)sy * PW - diffx + x] : 0.f;
                    }
                }
#pragma unroll
                for (int u = 0; u < kRows; ++u) {
                    const int y = y0 + u * (int)gridDim.y;
                    if (y >= W) continue;
                    float vv[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
                    bool any = false;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        if (sub[u][c]) {
                            vv[c] = vv[c] - amp * pv[u][c];
                            any = true;
                        }
                        const unsigned long long k =
                            peak_key(vv[c], (unsigned)y * (unsigned)W + (unsigned)(x4 + c));
                        best = k > best ? k : best;
                    }
                    if (any)
                        *reinterpret_cast<float4 *>(a.res + (size_t)y * W + x4) =
                            make_float4(vv[0], vv[1], vv[2], vv[3]);
                }
            }
        }
        block_peak(best, a.keys + (i + 1) % 3);
        return;
    }
    for (int x = blockIdx.x * 256 + threadIdx.x; x < W; x += gridDim.x * 256) {
        const bool colIn = x >= startx && x <= stopx;
        for (int y0 = blockIdx.y; y0 < W; y0 += gridDim.y * kRows) {
            float v[kRows], pv[kRows];
            bool sub[kRows];
#pragma unroll
            for (int u = 0; u < kRows; ++u) {
                const int y = y0 + u * (int)gridDim.y;
                const int sy = y - diffy;
                const bool rowOk = y < W;
                sub[u] = rowOk && colIn && y >= starty && y <= stopy && sy >= 0 && sy < PW;
                v[u] = rowOk ? a.res[(size_t)y * W + x] : 0.f;
                pv[u] = sub[u] ? a.psf[(ptrdiff_t)sy * PW - diffx + x] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < kRows; ++u) {
                const int y = y0 + u * (int)gridDim.y;
                if (y >= W) continue;
                float vv = v[u];
                if (sub[u]) {
                    vv = vv - amp * pv[u];
                    a.res[(size_t)y * W + x] = vv;
                }
                const unsigned long long k = peak_key(vv, (unsigned)y * (unsigned)W + (unsigned)x);
                best = k > best ? k : best;
            }
        }
    }
    block_peak(best, a.keys + (i + 1) % 3);
}

// Peak of the real parts of a complex image into *key (zeroed beforehand), and
// with PLANE the real parts into a float plane as well: one read of the image.
// Two pixels a load, four loads in flight (4096^2: 36 us alone, 68 us as an
// extraction and a reduction of the plane).
template <bool PLANE>
__global__ __launch_bounds__(256) void k_peak_complex(const float2 *__restrict__ img, long long n,
                                                      float *__restrict__ plane, unsigned long long *key)
{
    constexpr int U = 4;
    const long long pairs = n >> 1, stride = (long long)gridDim.x * 256;
    unsigned best = 0, at = 0;   // |re| bits, index; a thread's indices ascend
    bool any = false;
    float val = 0.f;
    auto take = [&](float v, long long i) {
        const unsigned a = __float_as_uint(v) & 0x7fffffffu;
        if (a > best || !any) {
            best = a;
            at = (unsigned)i;
            val = v;
            any = true;
        }
    };
    for (long long p = blockIdx.x * 256LL + threadIdx.x; p < pairs; p += U * stride) {
        float4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long long q = p + u * stride;
            v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (q < pairs) __builtin_memcpy(&v[u], img + 2 * q, 16);   // images need only 8-byte alignment
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long long q = p + u * stride;
            if (q >= pairs) break;
            if constexpr (PLANE) *reinterpret_cast<float2 *>(plane + 2 * q) = make_float2(v[u].x, v[u].z);
            take(v[u].x, 2 * q);
            take(v[u].z, 2 * q + 1);
        }
    }
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
        const float v = img[n - 1].x;
        if constexpr (PLANE) plane[n - 1] = v;
        take(v, n - 1);
    }
    block_peak(any ? peak_key(val, at) : 0ull, key);
}

// The whole Hogbom loop in one launch, for residuals that fit the registers of
// the workgroups that run together (up to 2^24 pixels: 64 a lane): every thread
// keeps GPT groups of four adjacent residual pixels from the first iteration to
// the last (columns x..x+3 of GPT rows), so an iteration reads only the PSF.  Each iteration ends with one
// exchange among the workgroups: every workgroup publishes its peak in a slot of
// its own and reads all the others' (two sets of slots by turns: a workgroup is
// never more than one iteration ahead of the slowest, which must still find the
// set before).  A slot holds the peak's key and the iteration's number (8 bits)
// in one 64-bit word, so nothing else needs ordering.  The host launches it
// cooperatively, so all workgroups are resident; the waits are bounded all the
// same (another process may hold part of the device), and a launch is done whole
// or not at all: nothing is written until every workgroup has finished the
// iterations and added itself to *agree, and one whose wait runs out marks *agree
// kLost unless all have.  Components wait in LDS until then, kLoopIters at most;
// more iterations take more launches, each of which goes on only where the one
// before was done (*chunks).
// Key: |v| bits << 25 | (2^24 - 1 - index) << 1 | sign, as peak_key orders them.
// Bound: the PSF's read, 67 MB at 4096^2 from the Infinity Cache, and the
// exchange.  13.4 us an iteration at 4096^2, against 35.5 us for
// k_hogbom_step, which also reads and writes the residual (201 MB).
struct HogbomLoop {
    float2 *res;                     // complex residual, W x W (real parts updated)
    const float *psf;                // PSF real plane, PW x PW, kPsfPad floats on each side
    float2 *model;                   // complex model image
    const unsigned long long *psfKey;   // PSF peak (peak_key)
    unsigned long long *slots;       // 2 x kSlots, zeroed
    unsigned long long *first;       // first residual peak (peak_key; the first launch)
    unsigned *agree;                 // workgroups that finished, zeroed
    int *chunks;                     // launches of this call done
    int *hostFail;                   // host flag of a call that doesn't wait (or null)
    unsigned long long polls;        // longest wait (of about a microsecond each)
    int W, PW, niters, chunk;        // chunk: launches before this one
    int C;                           // column groups of four a row, rounded up to a power of two
    float gain;
};
constexpr int kSlots = 1024;
constexpr int kLoopIters = 1024;
constexpr unsigned kLost = 1u << 31;
constexpr int kPsfPad = 64;   // floats before and after the plane that a group of four may read (unused)

__device__ __forceinline__ unsigned long long loop_key(unsigned absBits, unsigned idx, bool neg)
{
    return ((unsigned long long)absBits << 25) | ((unsigned long long)(0xffffffu - idx) << 1) | (neg ? 1u : 0u);
}

template <int GPT>
__global__ __launch_bounds__(1024) void k_hogbom_loop(HogbomLoop a)
{
#pragma clang fp contract(off)
    constexpr int kBlk = GPT < 4 ? GPT : 4;   // groups whose PSF reads are issued together
    __shared__ unsigned s_abs[16];
    __shared__ unsigned long long s_key, s_win[16];
    __shared__ unsigned s_pos[kLoopIters];   // the components (the first workgroup's are used)
    __shared__ float s_amp[kLoopIters];
    __shared__ bool s_done;
    if (*a.chunks != a.chunk) return;   // an earlier launch was not done
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int W = a.W, PW = a.PW, nWG = gridDim.x;
    // the workgroup's threads cover 1024 / C rows of C column groups a step
    const int x = (tid & (a.C - 1)) * 4, rows = 1024 / a.C;
    const int y0 = (int)blockIdx.x * rows + tid / a.C, dy = nWG * rows;   // row i: y0 + i * dy
    float v[GPT][4];
#pragma unroll
    for (int i = 0; i < GPT; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c)
            v[i][c] = y0 + i * dy < W && x + c < W ? a.res[(size_t)(y0 + i * dy) * W + x + c].x : 0.f;
    const unsigned long long kp = *a.psfKey;
    const unsigned ppos = key_index(kp);
    const int px = (int)(ppos % (unsigned)PW), py = (int)(ppos / (unsigned)PW);
    if (tid == 0) s_key = 0ull;
    bool lost = false;
    for (int it = 0; it < max(a.niters, 1) && !lost; ++it) {
        // opaque copies: the rows' positions are worked out again in every
        // iteration instead of being kept in registers across them
        int yb = y0, xa = x;
        asm volatile("" : "+v"(yb), "+v"(xa));
        // this workgroup's peak: the largest |v| first, then its first pixel
        unsigned m = 0;
#pragma unroll
        for (int i = 0; i < GPT; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) m = max(m, __float_as_uint(v[i][c]) & 0x7fffffffu);
        unsigned wm = m;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) wm = max(wm, (unsigned)__shfl_xor((int)wm, o, 64));
        if (lane == 0) s_abs[wave] = wm;
        __syncthreads();
        unsigned bm = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) bm = max(bm, s_abs[w]);
        if (m == bm) {
            unsigned idx = ~0u;
            bool neg = false;
            // a thread's indices ascend with i and c: the first one stays.  (The
            // sign is shifted out: masked as above, the compiler would keep the
            // masked values from there in registers.)
#pragma unroll
            for (int i = GPT - 1; i >= 0; --i)
#pragma unroll
                for (int c = 3; c >= 0; --c)
                    if (__float_as_uint(v[i][c]) << 1 == bm << 1 && yb + i * dy < W && xa + c < W) {
                        idx = (unsigned)(yb + i * dy) * (unsigned)W + (unsigned)(xa + c);
                        neg = v[i][c] < 0.f;
                    }
            if (idx != ~0u) atomicMax(&s_key, loop_key(bm, idx, neg));
        }
        __syncthreads();
        const unsigned long long tag = (unsigned long long)((it + 1) & 0xff) << 56;
        unsigned long long *slots = a.slots + (it & 1) * kSlots;
        if (tid == 0)
            __hip_atomic_store(slots + blockIdx.x, s_key | tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        unsigned long long k = tid < nWG ? ~0ull : 0ull;
        if (tid < nWG) {
            for (unsigned long long n = 0; n < a.polls; ++n) {
                k = __hip_atomic_load(slots + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (k >> 56 == tag >> 56) break;
                k = ~0ull;   // still the wrong one when the wait ends
            }
        }
        if (tid < nWG || wave * 64 < nWG) k = wave_max_u64(k);
        if (lane == 0) s_win[wave] = k;
        __syncthreads();
        unsigned long long win = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) win = s_win[w] > win ? s_win[w] : win;
        // a lost workgroup ends the iteration on pixel 0 with a peak of zero (a break
        // here costs 27 spilled registers)
        lost = win == ~0ull;
        win = lost ? loop_key(0u, 0u, false) : win & ((1ull << 56) - 1);
        const unsigned absBits = (unsigned)(win >> 25), pos = 0xffffffu - (unsigned)((win >> 1) & 0xffffffu);
        const float peak = __uint_as_float(absBits | ((unsigned)(win & 1) << 31));
        if (tid == 0) {
            s_key = 0ull;
            if (it == 0 && a.chunk == 0 && blockIdx.x == 0) *a.first = peak_key(peak, pos);
        }
        if (it == a.niters) break;   // none to do
        const int rx = (int)(pos % (unsigned)W), ry = (int)(pos / (unsigned)W);
        const int diffx = rx - px, diffy = ry - px;   // as in the reference
        const int startx = max(0, rx - px), starty = max(0, ry - py);
        const int stopx = min(W - 1, rx + (PW - px - 1)), stopy = min(W - 1, ry + (PW - py - 1));
        const float amp = a.gain * peak;
        if (tid == 1023) {   // not in a wave that waits for the slots
            s_pos[it] = pos;
            s_amp[it] = amp;
        }
        bool col[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) col[c] = xa + c >= startx && xa + c <= stopx;
        const bool colSome = xa <= stopx && xa + 3 >= startx;
        // row y takes PSF row y - diffy where both exist
        const int yLo = max(starty, diffy), yHi = min(stopy, PW - 1 + diffy);
        const int at0 = (yb - diffy) * PW + (xa - diffx);   // down to -3 and up to PW * PW + 2: see kPsfPad
#pragma unroll
        for (int i0 = 0; i0 < GPT; i0 += kBlk) {
            float4 p[kBlk];
            bool row[kBlk];
#pragma unroll
            for (int b = 0; b < kBlk; ++b) {
                const int y = yb + (i0 + b) * dy;
                row[b] = colSome && y >= yLo && y <= yHi;
                __builtin_memcpy(&p[b], a.psf + (row[b] ? at0 + (i0 + b) * dy * PW : 0), 16);
            }
#pragma unroll
            for (int b = 0; b < kBlk; ++b) {
                const float t[4] = {p[b].x, p[b].y, p[b].z, p[b].w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float u = v[i0 + b][c] - amp * t[c];
                    v[i0 + b][c] = row[b] && col[c] ? u : v[i0 + b][c];
                }
            }
            __builtin_amdgcn_sched_barrier(0);   // PSF reads of kBlk rows in flight: the registers' bound
        }
    }
    if (tid == 0) {
        unsigned n = lost ? atomicOr(a.agree, kLost) | kLost : atomicAdd(a.agree, 1u) + 1;
        for (unsigned long long p = 0; p < a.polls && n != (unsigned)nWG && !(n & kLost); ++p)
            n = __hip_atomic_load(a.agree, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        while (n != (unsigned)nWG && !(n & kLost)) {   // the wait ran out; each turn but the last finds one more
            const unsigned seen = atomicCAS(a.agree, n, n | kLost);
            n = seen == n ? n | kLost : seen;
        }
        s_done = n == (unsigned)nWG;
        if (!s_done && a.hostFail) __hip_atomic_store(a.hostFail, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __syncthreads();
    if (!s_done) return;
    if (blockIdx.x == 0) {
        // a component a thread; the first at a pixel adds all of that pixel's in turn
        if (tid == 0) *a.chunks = a.chunk + 1;
        if (tid < a.niters) {
            const unsigned at = s_pos[tid];
            int j = 0;
            while (j < tid && s_pos[j] != at) ++j;
            if (j == tid) {
                float m = a.model[at].x;
                for (; j < a.niters; ++j)
                    if (s_pos[j] == at) m = m + s_amp[j];
                a.model[at].x = m;
            }
        }
    }
    int yw = y0, xw = x;
    asm volatile("" : "+v"(yw), "+v"(xw));   // addresses worked out anew, not kept since the loads
#pragma unroll
    for (int i = 0; i < GPT; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (yw + i * dy < W && xw + c < W) a.res[(size_t)(yw + i * dy) * W + xw + c].x = v[i][c];
}

int stream_blocks(tcv_ctx *ctx, long long n, int perThread = 1)
{
    const long long want = (n + 256LL * perThread - 1) / (256LL * perThread);
    return (int)std::max<long long>(1, std::min<long long>(want, (long long)ctx->cus * 8));
}

}  // namespace

// ---- host side ---------------------------------------------------------------------

static tcv_status fft_plan(tcv_ctx *ctx, int gSize, hipfftHandle *out)
{
    auto it = ctx->fftPlans.find(gSize);
    if (it != ctx->fftPlans.end()) {
        *out = (hipfftHandle)it->second;
        return TCV_OK;
    }
    hipfftHandle h = nullptr;
    if (hipfftPlan2d(&h, gSize, gSize, HIPFFT_C2C) != HIPFFT_SUCCESS)
        return tcv_fail(ctx, TCV_ERR_DEVICE, "hipfftPlan2d failed for " + std::to_string(gSize));
    if (hipfftSetStream(h, ctx->stream) != HIPFFT_SUCCESS) {
        hipfftDestroy(h);
        return tcv_fail(ctx, TCV_ERR_DEVICE, "hipfftSetStream failed");
    }
    ctx->fftPlans[gSize] = (void *)h;
    *out = h;
    return TCV_OK;
}

void major_release(tcv_ctx *ctx)
{
    for (auto &kv : ctx->fftPlans) hipfftDestroy((hipfftHandle)kv.second);
    ctx->fftPlans.clear();
    for (auto &kv : ctx->fftTwiddles) (void)hipFree(kv.second);
    ctx->fftTwiddles.clear();
    if (ctx->majorWs) (void)hipFree(ctx->majorWs);
    ctx->majorWs = nullptr;
    ctx->majorWsBytes = 0;
    if (ctx->lateFail) (void)hipHostFree(ctx->lateFail);
    ctx->lateFail = nullptr;
}

// grow-only workspace: Hogbom's float planes and peak keys
static tcv_status major_ws(tcv_ctx *ctx, size_t bytes, void **p)
{
    if (ctx->majorWsBytes < bytes) {
        if (ctx->majorWs) TCV_HIP(ctx, hipStreamSynchronize(ctx->stream));
        if (ctx->majorWs) (void)hipFree(ctx->majorWs);
        ctx->majorWs = nullptr;
        ctx->majorWsBytes = 0;
        if (hipMalloc(&ctx->majorWs, bytes) != hipSuccess) {
            (void)hipGetLastError();
            return tcv_fail(ctx, TCV_ERR_NOMEM, "Hogbom workspace of " + std::to_string(bytes) +
                                                    " bytes");
        }
        ctx->majorWsBytes = bytes;
    }
    *p = ctx->majorWs;
    return TCV_OK;
}

// The flag that the kernels of a call which doesn't wait set in host memory; the
// calls that wait for the stream report it (ctx_wait).
static tcv_status late_flag(tcv_ctx *ctx, int **d_flag)
{
    if (!ctx->lateFail) {
        void *p = nullptr;
        if (hipHostMalloc(&p, sizeof(int), hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
            (void)hipGetLastError();
            return tcv_fail(ctx, TCV_ERR_NOMEM, "tcv_hogbom: host flag");
        }
        ctx->lateFail = (int *)p;
        *ctx->lateFail = 0;
    }
    void *d = nullptr;
    TCV_HIP(ctx, hipHostGetDevicePointer(&d, ctx->lateFail, 0));
    *d_flag = (int *)d;
    return TCV_OK;
}

// The one-launch loop: residuals of up to 2^24 pixels (64 registers a lane on
// every CU; the keys' 24-bit index) on devices that launch cooperatively, and PSFs
// whose tap index fits an int.
static int hogbom_groups(const tcv_ctx *ctx, long long width, int *C, unsigned *nWG)
{
    *C = 1;
    while (*C * 4LL < width) *C *= 2;
    if (*C > 1024) return 0;
    const long long rows = 1024 / *C;   // rows a workgroup covers in one step
    for (int gpt = 1; gpt <= 16; gpt *= 2) {
        const long long n = (width + rows * gpt - 1) / (rows * gpt);
        if (n <= std::min(ctx->cus, kSlots)) {
            *nWG = (unsigned)n;
            return gpt;
        }
    }
    return 0;
}

static bool hogbom_loop_fits(const tcv_ctx *ctx, long long width, long long psfWidth)
{
    int C;
    unsigned nWG;
    return ctx->coopLaunch && width <= 4096 && psfWidth <= 32768 && hogbom_groups(ctx, width, &C, &nWG) > 0;
}

static hipError_t launch_hogbom_loop(tcv_ctx *ctx, HogbomLoop a)
{
    unsigned nWG = 0;
    const int gpt = hogbom_groups(ctx, a.W, &a.C, &nWG);
    const void *k = gpt == 1   ? (const void *)k_hogbom_loop<1>
                    : gpt == 2 ? (const void *)k_hogbom_loop<2>
                    : gpt == 4 ? (const void *)k_hogbom_loop<4>
                    : gpt == 8 ? (const void *)k_hogbom_loop<8>
                               : (const void *)k_hogbom_loop<16>;
    void *args[] = {&a};
    return hipLaunchCooperativeKernel(k, dim3(nWG), dim3(1024), args, 0, ctx->stream);
}

static tcv_status fft_run(tcv_ctx *ctx, float *d_grid, int gSize, int forward, int fix, float scale)
{
    if (!ctx) return TCV_ERR_INVALID;
    if (!d_grid || gSize < 2 || (gSize & 1) || gSize > 65534)
        return tcv_fail(ctx, TCV_ERR_INVALID, "fftExec: gSize must be even (the shift is by gSize/2)");
    float2 *g = reinterpret_cast<float2 *>(d_grid);
    // Powers of two of 256 to 4096: two passes of our own with the modulation
    // folded in (4096^2: 121 us, against 281 us of the library's four passes
    // between two of k_checker); other sizes and larger ones through hipFFT.
    if (fft_pow2_supported(gSize)) {
        ProfScope ps(ctx, "fft");
        return fft_pow2_run(ctx, g, gSize, forward, fix, scale);
    }
    hipfftHandle h;
    tcv_status st = fft_plan(ctx, gSize, &h);
    if (st != TCV_OK) return st;
    ProfScope ps(ctx, "fft");
    const dim3 grid((gSize / 2 + 255) / 256, gSize);
    hipLaunchKernelGGL(k_checker, grid, dim3(256), 0, ctx->stream, g, gSize, 0, 1.f);
    TCV_HIP(ctx, hipGetLastError());
    if (hipfftExecC2C(h, (hipfftComplex *)g, (hipfftComplex *)g,
                      forward ? HIPFFT_FORWARD : HIPFFT_BACKWARD) != HIPFFT_SUCCESS)
        return tcv_fail(ctx, TCV_ERR_DEVICE, "hipfftExecC2C failed");
    hipLaunchKernelGGL(k_checker, grid, dim3(256), 0, ctx->stream, g, gSize, fix ? 1 : 0, scale);
    TCV_HIP(ctx, hipGetLastError());
    return TCV_OK;
}

extern "C" {

tcv_status tcv_fft_exec(tcv_ctx *ctx, float *d_grid, int gSize, int forward)
{
    return fft_run(ctx, d_grid, gSize, forward, 0, 1.f);
}

tcv_status tcv_fft_exec_fix(tcv_ctx *ctx, float *d_grid, int gSize, int forward, float scale)
{
    return fft_run(ctx, d_grid, gSize, forward, 1, scale);
}

tcv_status tcv_fft_fix(tcv_ctx *ctx, float *d_grid, long long nPixels, float scale)
{
    if (!ctx) return TCV_ERR_INVALID;
    if (nPixels < 0 || (nPixels && !d_grid)) return tcv_fail(ctx, TCV_ERR_INVALID, "tcv_fft_fix");
    if (!nPixels) return TCV_OK;
    ProfScope ps(ctx, "fft_fix");
    hipLaunchKernelGGL(k_fft_fix, dim3(stream_blocks(ctx, nPixels, 4)), dim3(256), 0, ctx->stream,
                       (float2 *)d_grid, nPixels, scale);
    TCV_HIP(ctx, hipGetLastError());
    return TCV_OK;
}

tcv_status tcv_vis_subtract(tcv_ctx *ctx, float *d_data, const float *d_model, long long nVis)
{
    if (!ctx) return TCV_ERR_INVALID;
    if (nVis < 0 || (nVis && (!d_data || !d_model)))
        return tcv_fail(ctx, TCV_ERR_INVALID, "tcv_vis_subtract");
    if (!nVis) return TCV_OK;
    ProfScope ps(ctx, "vis_subtract");
    hipLaunchKernelGGL(k_vis_subtract, dim3(stream_blocks(ctx, nVis, 4)), dim3(256), 0,
                       ctx->stream, (float2 *)d_data, (const float2 *)d_model, nVis);
    TCV_HIP(ctx, hipGetLastError());
    return TCV_OK;
}

tcv_status tcv_find_peak(tcv_ctx *ctx, const float *d_image, long long nPixels, float *maxVal,
                         long long *maxPos)
{
    if (!ctx) return TCV_ERR_INVALID;
    if (!d_image || nPixels < 1 || nPixels > 0xffffffffLL || !maxVal || !maxPos)
        return tcv_fail(ctx, TCV_ERR_INVALID, "tcv_find_peak: bad argument (1 <= nPixels < 2^32)");
    void *ws;
    tcv_status st = major_ws(ctx, 256, &ws);
    if (st != TCV_OK) return st;
    unsigned long long *key = (unsigned long long *)ws;
    ProfScope ps(ctx, "find_peak");
    st = launch_fill_u32(ctx, key, 0u, 2);
    if (st != TCV_OK) return st;
    hipLaunchKernelGGL(k_peak_complex<false>, dim3(stream_blocks(ctx, nPixels, 8)), dim3(256), 0,
                       ctx->stream, (const float2 *)d_image, nPixels, (float *)nullptr, key);
    TCV_HIP(ctx, hipGetLastError());
    unsigned long long k = 0;
    TCV_HIP(ctx, hipMemcpyAsync(&k, key, 8, hipMemcpyDeviceToHost, ctx->stream));
    if ((st = ctx_wait(ctx)) != TCV_OK) return st;
    const unsigned a = (unsigned)(k >> 33);
    float av;
    std::memcpy(&av, &a, 4);
    *maxVal = (k & 1) ? -av : av;
    *maxPos = k ? (long long)(~(unsigned)((k >> 1) & 0xffffffffull)) : 0;
    return TCV_OK;
}

tcv_status tcv_hogbom(tcv_ctx *ctx, float *d_residual, long long width, const float *d_psf,
                      long long psfWidth, float *d_model, int niters, float gain,
                      float *psfPeakVal, long long *psfPeakPos, float *dirtyPeakVal,
                      long long *dirtyPeakPos)
{
    if (!ctx) return TCV_ERR_INVALID;
    if (!d_residual || !d_psf || !d_model || width < 1 || psfWidth < 1 || niters < 0 ||
        width * width > 0xffffffffLL || psfWidth * psfWidth > 0xffffffffLL)
        return tcv_fail(ctx, TCV_ERR_INVALID, "tcv_hogbom: bad argument (widths below 65536)");
    const long long n = width * width, pn = psfWidth * psfWidth;
    const bool wait = psfPeakVal || psfPeakPos || dirtyPeakVal || dirtyPeakPos;
    // (a few iterations on a small image take less than the cooperative launch: one on
    // 250^2 27 us, 37 by the loop; five on 64^2 43 and 45)
    bool loop = hogbom_loop_fits(ctx, width, psfWidth) && (niters >= 8 || width > 512);
    int launched = 0, done = 0;   // launches of the loop made, and done
    unsigned long long pk = 0, first = 0;
    ProfScope ps(ctx, "hogbom");
    for (;;) {
        // PSF plane | keys, launches done | count of finished workgroups and slots
        // of the loop, or residual plane
        const size_t psfB = ((size_t)(pn + 2 * kPsfPad) * 4 + 255) & ~size_t(255);
        const size_t resB =
            loop ? 256 + 2 * kSlots * sizeof(unsigned long long) : ((size_t)n * 4 + 255) & ~size_t(255);
        void *ws;
        tcv_status st = major_ws(ctx, psfB + 256 + resB, &ws);
        if (st != TCV_OK) return st;
        float *psf = (float *)ws + kPsfPad;
        unsigned long long *keys = (unsigned long long *)((char *)ws + psfB);
        void *rest = (char *)ws + psfB + 256;
        st = launch_fill_u32(ctx, keys, 0u, loop ? 64 + resB / 4 : 64);
        if (st != TCV_OK) return st;
        hipLaunchKernelGGL(k_peak_complex<true>, dim3(stream_blocks(ctx, pn, 8)), dim3(256), 0, ctx->stream,
                           (const float2 *)d_psf, pn, psf, keys + 3);
        TCV_HIP(ctx, hipGetLastError());
        if (loop) {
            HogbomLoop a{(float2 *)d_residual, psf, (float2 *)d_model, keys + 3,
                         (unsigned long long *)((char *)rest + 256), keys, (unsigned *)rest, (int *)(keys + 8),
                         nullptr, ctx->waitPolls, (int)width, (int)psfWidth, 0, 0, 0, gain};
            if (!wait && (st = late_flag(ctx, &a.hostFail)) != TCV_OK) return st;
            do {
                a.chunk = launched;
                a.niters = std::min(niters - launched * kLoopIters, kLoopIters);
                if (launched && (st = launch_fill_u32(ctx, rest, 0u, resB / 4)) != TCV_OK) return st;
                const hipError_t e = launch_hogbom_loop(ctx, a);
                if (e != hipSuccess && !launched) break;   // not launched together: one launch an iteration
                TCV_HIP(ctx, e);
                ++launched;
            } while (launched * (long long)kLoopIters < niters);
            if (!launched) {
                (void)hipGetLastError();
                loop = false;
                continue;
            }
            if (wait) {
                TCV_HIP(ctx, hipMemcpyAsync(&first, keys, 8, hipMemcpyDeviceToHost, ctx->stream));
                TCV_HIP(ctx, hipMemcpyAsync(&pk, keys + 3, 8, hipMemcpyDeviceToHost, ctx->stream));
                TCV_HIP(ctx, hipMemcpyAsync(&done, a.chunks, 4, hipMemcpyDeviceToHost, ctx->stream));
                if ((st = ctx_wait(ctx)) != TCV_OK) return st;
                if (done < launched) {   // a wait ran out: the rest in one launch an iteration
                    loop = false;
                    continue;
                }
            }
            break;
        }
        float *res = (float *)rest;
        hipLaunchKernelGGL(k_peak_complex<true>, dim3(stream_blocks(ctx, n, 8)), dim3(256), 0, ctx->stream,
                           (const float2 *)d_residual, n, res, keys + 0);
        TCV_HIP(ctx, hipGetLastError());
        if (wait && !done) TCV_HIP(ctx, hipMemcpyAsync(&first, keys, 8, hipMemcpyDeviceToHost, ctx->stream));
        HogbomArgs a{res, psf, (float2 *)d_model, keys, (int)width, (int)psfWidth, gain};
        // four pixels a thread when the rows are whole float4s
        const bool vec = width % 4 == 0;
        const long long perRow = vec ? width / 4 : width;
        const int bx = (int)std::min<long long>((perRow + 255) / 256, 64);
        const int by = (int)std::max<long long>(1, std::min<long long>(width, (long long)ctx->cus * 8 / bx));
        for (int i = 0; i < niters - done * kLoopIters; ++i) {
            if (vec)
                hipLaunchKernelGGL(k_hogbom_step<true>, dim3(bx, by), dim3(256), 0, ctx->stream, a, i);
            else
                hipLaunchKernelGGL(k_hogbom_step<false>, dim3(bx, by), dim3(256), 0, ctx->stream, a, i);
        }
        TCV_HIP(ctx, hipGetLastError());
        hipLaunchKernelGGL(k_real_writeback, dim3(stream_blocks(ctx, n, 4)), dim3(256), 0, ctx->stream,
                           (float2 *)d_residual, (const float *)res, n);
        TCV_HIP(ctx, hipGetLastError());
        if (wait) {
            TCV_HIP(ctx, hipMemcpyAsync(&pk, keys + 3, 8, hipMemcpyDeviceToHost, ctx->stream));
            if ((st = ctx_wait(ctx)) != TCV_OK) return st;
        }
        break;
    }
    if (wait) {
        auto val = [](unsigned long long k) {
            const unsigned a2 = (unsigned)(k >> 33);
            float f;
            std::memcpy(&f, &a2, 4);
            return (k & 1) ? -f : f;
        };
        auto pos = [](unsigned long long k) {
            return k ? (long long)(~(unsigned)((k >> 1) & 0xffffffffull)) : 0LL;
        };
        if (psfPeakVal) *psfPeakVal = val(pk);
        if (psfPeakPos) *psfPeakPos = pos(pk);
        if (dirtyPeakVal) *dirtyPeakVal = val(first);
        if (dirtyPeakPos) *dirtyPeakPos = pos(first);
    }
    return TCV_OK;
}

}  // extern "C"
