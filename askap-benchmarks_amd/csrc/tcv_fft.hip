// The shifted 2-D transform of fftExec (current/tMajorACC/tMajorACC.cc:488-546)
// for power-of-two grids of 256 to 4096 pixels a side: two passes over the
// grid, one along the rows and one along the columns, each of which reads and
// writes every pixel once and applies the (-1)^(x+y) modulation (and, on the
// way out, fftFix) to the values it already holds.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "tcv_internal.h"

namespace {

// Twiddle factors of one length n: 16 x 16 factors exp(-2 pi i k r / 256) of
// the second stage at [r * 16 + k], then L x 256 factors exp(-2 pi i k r / n)
// of the third (L = n / 256) at [256 + r * 256 + k], so that neighbouring
// threads (k) read neighbouring factors.  Rounded from double.
constexpr int kTw3 = 256;

typedef unsigned uint2v __attribute__((ext_vector_type(2)));

template <int DIR>
__device__ __forceinline__ float2 cmul(float2 a, float2 w)
{
    if constexpr (DIR < 0) return make_float2(a.x * w.x - a.y * w.y, a.x * w.y + a.y * w.x);
    else return make_float2(a.x * w.x + a.y * w.y, a.y * w.x - a.x * w.y);   // conj(w)
}

template <int DIR>
__device__ __forceinline__ float2 rot(float2 a)   // a * exp(DIR i pi / 2)
{
    if constexpr (DIR < 0) return make_float2(a.y, -a.x);
    else return make_float2(-a.y, a.x);
}

__device__ __forceinline__ float2 add(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 sub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }

template <int DIR>
__device__ __forceinline__ void dft4(float2 &a, float2 &b, float2 &c, float2 &d)
{
    const float2 s0 = add(a, c), d0 = sub(a, c), s1 = add(b, d), d1 = rot<DIR>(sub(b, d));
    a = add(s0, s1);
    b = add(d0, d1);
    c = sub(s0, s1);
    d = sub(d0, d1);
}

// In-place DFT of R values at v[0], v[S], v[2 S], ... (natural order in and out)
template <int R, int S, int DIR>
__device__ __forceinline__ void dft(float2 *v)
{
    constexpr float kC1 = 0.92387953251128675613f, kS1 = 0.38268343236508977173f;   // pi / 8
    constexpr float kH = 0.70710678118654752440f;
    if constexpr (R == 2) {
        const float2 a = v[0], b = v[S];
        v[0] = add(a, b);
        v[S] = sub(a, b);
    } else if constexpr (R == 4) {
        dft4<DIR>(v[0], v[S], v[2 * S], v[3 * S]);
    } else if constexpr (R == 8) {
        // n = n1 + 2 n2, k = k1 + 4 m
        dft4<DIR>(v[0], v[2 * S], v[4 * S], v[6 * S]);
        dft4<DIR>(v[S], v[3 * S], v[5 * S], v[7 * S]);
        float2 o[8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            constexpr float c[4] = {1.f, kH, 0.f, -kH}, s[4] = {0.f, -kH, -1.f, -kH};
            const float2 e = v[2 * k * S];
            float2 t = v[(2 * k + 1) * S];
            if (k) t = cmul<DIR>(t, make_float2(c[k], s[k]));
            o[k] = add(e, t);
            o[k + 4] = sub(e, t);
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k * S] = o[k];
    } else if constexpr (R == 16) {
        // n = n1 + 4 n2, k = k1 + 4 m
#pragma unroll
        for (int n1 = 0; n1 < 4; ++n1) dft4<DIR>(v[n1 * S], v[(n1 + 4) * S], v[(n1 + 8) * S], v[(n1 + 12) * S]);
        // v[n1 + 4 k1] *= exp(-2 pi i n1 k1 / 16)
        v[5 * S] = cmul<DIR>(v[5 * S], make_float2(kC1, -kS1));
        v[6 * S] = cmul<DIR>(v[6 * S], make_float2(kH, -kH));
        v[7 * S] = cmul<DIR>(v[7 * S], make_float2(kS1, -kC1));
        v[9 * S] = cmul<DIR>(v[9 * S], make_float2(kH, -kH));
        v[10 * S] = rot<DIR>(v[10 * S]);
        v[11 * S] = cmul<DIR>(v[11 * S], make_float2(-kH, -kH));
        v[13 * S] = cmul<DIR>(v[13 * S], make_float2(kS1, -kC1));
        v[14 * S] = cmul<DIR>(v[14 * S], make_float2(-kH, -kH));
        v[15 * S] = cmul<DIR>(v[15 * S], make_float2(-kC1, kS1));
        float2 o[16];
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) {
            dft4<DIR>(v[(4 * k1) * S], v[(4 * k1 + 1) * S], v[(4 * k1 + 2) * S], v[(4 * k1 + 3) * S]);
#pragma unroll
            for (int m = 0; m < 4; ++m) o[k1 + 4 * m] = v[(4 * k1 + m) * S];
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k * S] = o[k];
    }
}

__host__ __device__ constexpr int padded(int i) { return i + (i >> 4); }

// One pass.  COLS == 0: rows; each group of N / 16 threads transforms one row.
// COLS > 0: columns, COLS adjacent ones a workgroup (thread = row group x
// column), so that a pixel row's segment is read and written contiguously.
// Every thread keeps 16 values in registers; the stages (radix 16, 16, N / 256,
// self-sorting) exchange them through LDS, real parts first and then imaginary
// parts, so that the buffer (padded by one in 16 against bank conflicts) is
// half as large.
// Bound: memory.  At 4096^2 the row pass takes 45 us (268 MB, 5.9 TB/s) and the
// column pass 76 us: its four columns a workgroup (what 4096 rows leave room
// for at 16 values a thread) are 32-byte segments.  Holding it to 64 registers,
// for two workgroups a CU, left it at 75-84 us.
// OUT 1: times (-1)^(x+y) on input (row pass); 2: on output; 3: on output with
// fftFix (real part * scale, imaginary part 0).
template <int N, int COLS, int DIR, int OUT>
__global__ __launch_bounds__(COLS ? N / 16 * COLS : 256) void k_fft_pass(float2 *__restrict__ g,
                                                                           const float2 *__restrict__ tw,
                                                                           float scale)
{
    constexpr int T = N / 16;                 // threads a transform
    constexpr int L = N / 256;                // radix of the third stage
    constexpr int P = COLS ? COLS : 256 / T;  // transforms a workgroup
    __shared__ float buf[padded(N) * P];
    const int t = threadIdx.x;
    const int j = COLS ? t / P : t % T, c = COLS ? t % P : t / T;
    // one byte offset a thread; value r is r * T (or 256) rows or pixels on, a
    // wave-uniform distance
    unsigned base;
    constexpr unsigned kStep = COLS ? 8u * N : 8u;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(g, 0, 8u * (unsigned)N * (unsigned)N, 0x00020000);
    int sgn;   // parity of x + y for the thread's first value (T and 256 are even)
    if constexpr (COLS > 0) {
        // workgroups whose segments share 128-byte lines run on one XCD
        // (consecutive workgroups go to the eight XCDs in turn)
        constexpr int G = COLS < 16 ? 16 / COLS : 1;
        const int b = blockIdx.x, xcd = b & 7, q = b >> 3;
        const int cb = G > 1 ? ((q / G) * 8 + xcd) * G + q % G : b;
        const int x = cb * COLS + c;
        base = 8u * ((unsigned)j * N + x);
        sgn = (x + j) & 1;
    } else {
        const int y = blockIdx.x * P + c;
        base = 8u * ((unsigned)y * N + j);
        sgn = (y + j) & 1;
    }
    auto slot = [&](int i) { return COLS ? padded(i) * P + c : padded(N) * c + padded(i); };
    float2 v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r)
        v[r] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rs, base, kStep * (r * T), 0));
    if constexpr (OUT == 1) {
        const float s = sgn ? -1.f : 1.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = make_float2(v[r].x * s, v[r].y * s);
    }
    dft<16, 1, DIR>(v);
    // exchange: the values go to `to(r)`, the next stage's come from `from(r)`
    auto exchange = [&](auto to, auto from) {
#pragma unroll
        for (int r = 0; r < 16; ++r) buf[slot(to(r))] = v[r].x;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r].x = buf[slot(from(r))];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 16; ++r) buf[slot(to(r))] = v[r].y;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r].y = buf[slot(from(r))];
    };
    exchange([&](int r) { return j * 16 + r; }, [&](int r) { return j + r * T; });
    const int k = j & 15;
#pragma unroll
    for (int r = 1; r < 16; ++r) v[r] = cmul<DIR>(v[r], tw[r * 16 + k]);
    dft<16, 1, DIR>(v);
    if constexpr (L > 1) {
        __syncthreads();   // the first exchange's last reads
        // butterfly b of the thread (16 / L of them): index jj = j + b T in
        // [0, 256), values v[b + (16 / L) r]
        constexpr int B = 16 / L;
        exchange([&](int r) { return (j >> 4) * 256 + k + r * 16; },
                 [&](int i) { return j + (i % B) * T + (i / B) * 256; });
#pragma unroll
        for (int b = 0; b < B; ++b) {
#pragma unroll
            for (int r = 1; r < L; ++r)
                v[b + B * r] = cmul<DIR>(v[b + B * r], tw[kTw3 + r * 256 + j + b * T]);
            dft<L, B, DIR>(v + b);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float2 o = v[i];
            if constexpr (OUT >= 2) {
                const float s = sgn ? -1.f : 1.f;
                o = OUT == 2 ? make_float2(o.x * s, o.y * s) : make_float2((s * o.x) * scale, 0.f);
            }
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2v, o), rs, base,
                                                  kStep * ((i % B) * T + (i / B) * 256), 0);
        }
    } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float2 o = v[r];
            if constexpr (OUT >= 2) {
                const float s = sgn ? -1.f : 1.f;
                o = OUT == 2 ? make_float2(o.x * s, o.y * s) : make_float2((s * o.x) * scale, 0.f);
            }
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2v, o), rs, base, kStep * (r * T), 0);
        }
    }
}

template <int N, int DIR>
void run_passes(tcv_ctx *ctx, float2 *g, const float2 *tw, int fix, float scale)
{
    constexpr int T = N / 16, P = 256 / T;
    constexpr int COLS = N >= 4096 ? 4 : N == 2048 ? 8 : 16;   // at most 1024 threads
    hipLaunchKernelGGL((k_fft_pass<N, 0, DIR, 1>), dim3(N / P), dim3(256), 0, ctx->stream, g, tw, 1.f);
    if (fix)
        hipLaunchKernelGGL((k_fft_pass<N, COLS, DIR, 3>), dim3(N / COLS), dim3(T * COLS), 0, ctx->stream, g,
                           tw, scale);
    else
        hipLaunchKernelGGL((k_fft_pass<N, COLS, DIR, 2>), dim3(N / COLS), dim3(T * COLS), 0, ctx->stream, g,
                           tw, 1.f);
}

}  // namespace

bool fft_pow2_supported(int n) { return n >= 256 && n <= 4096 && (n & (n - 1)) == 0; }

tcv_status fft_pow2_run(tcv_ctx *ctx, float2 *g, int n, int forward, int fix, float scale)
{
    auto it = ctx->fftTwiddles.find(n);
    if (it == ctx->fftTwiddles.end()) {
        const int L = n / 256;
        std::vector<float2> h(kTw3 + (size_t)L * 256);
        auto w = [](double turn) {
            const double a = -2.0 * M_PI * turn;
            return make_float2((float)std::cos(a), (float)std::sin(a));
        };
        for (int r = 0; r < 16; ++r)
            for (int k = 0; k < 16; ++k) h[r * 16 + k] = w((double)(k * r) / 256.0);
        for (int r = 0; r < L; ++r)
            for (int k = 0; k < 256; ++k) h[kTw3 + r * 256 + k] = w((double)(k * r) / (double)n);
        void *d = nullptr;
        if (hipMalloc(&d, h.size() * sizeof(float2)) != hipSuccess) {
            (void)hipGetLastError();
            return tcv_fail(ctx, TCV_ERR_NOMEM, "FFT twiddle factors");
        }
        if (hipMemcpy(d, h.data(), h.size() * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipFree(d);
            return tcv_fail(ctx, TCV_ERR_DEVICE, "FFT twiddle upload failed");
        }
        it = ctx->fftTwiddles.emplace(n, d).first;
    }
    const float2 *tw = (const float2 *)it->second;
    switch (n) {
#define X(N)                                                       \
    case N:                                                        \
        if (forward) run_passes<N, -1>(ctx, g, tw, fix, scale);    \
        else run_passes<N, 1>(ctx, g, tw, fix, scale);             \
        break;
        X(256) X(512) X(1024) X(2048) X(4096)
#undef X
    default: return tcv_fail(ctx, TCV_ERR_UNSUPPORTED, "FFT length");
    }
    TCV_HIP(ctx, hipGetLastError());
    return TCV_OK;
}
