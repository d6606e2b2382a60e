// Gridding and degridding of narrow kernels.
//
// The tiled kernels give a tile to four or eight waves that walk every entry
// together (gridder) or one entry each (degridder).  An entry of a narrow kernel
// has less work than its own set-up and waits: a 9 x 9 footprint is one load,
// and cost 300 CU cycles to grid and 175 to degrid.  Here
//  * one wave owns a region of the grid in LDS and takes every gridDim-th work item
//    (items are of one size: a queue's atomics, 12 ns each on one address, cost
//    more than they even out);
//  * regions overlap by the widest narrow kernel less one, so every footprint
//    lies inside one region: one entry a visibility, nothing clipped, and
//    degridding stores its result instead of adding parts with atomics;
//  * entries are decoded a lane each, 64 at a time, and their visibilities
//    fetched a block ahead; a lane's place in the footprint is worked out once
//    for a run of entries of one width, so an entry costs a handful of adds
//    beside its multiply-adds; the taps of the next entries are loaded while
//    the present ones are worked on.
// Regions of 32 cells (widths up to 19: 14 cells apart at the widest) keep 18
// gridding waves a CU in flight (8704 bytes of LDS each) and 16 degridding ones, of
// 48 cells (widths up to 31) 8.
//
// Bound: LDS and vector instruction issue (an entry's taps come from the L2s); of
// the gridder's LDS cycles on widths 7-19 60 % are bank conflicts.
// 3.8 M visibilities of widths 7-19 on 4096^2 (509 M grid points): gridder 1860 us
// by tiles, 360 by regions (11 TFLOP/s); degridder 1685 and 264 (15 TFLOP/s).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "tcv_device.h"
#include "tcv_internal.h"

namespace {

// A region of R x R cells in LDS as two planes, even and odd columns: column c of
// row r is cell r * RS + c / 2 of plane c & 1.  Two adjacent cells are then one
// in each plane whatever the column's parity, and the lanes of a wave read and
// write each plane contiguously along a row.  The last column of a plane and
// the cells beyond it are never part of the grid: the cell after a
// footprint of odd width may fall there.  (Rows are 34 dwords apart, 50 in a region of
// 48: a step's rows of a narrow footprint share banks.)
template <int R>
struct Region {
    static constexpr int RS = R / 2 + 1, PC = R * RS;
    static constexpr unsigned PB = PC * 8u;   // bytes a plane
};

// Steps of 64 pairs that footprints take: up to 3 in a region of 32, 4 to 8 in one
// of 48.
constexpr int pairs_of(int s) { return ((s + 1) >> 1) * s; }
static_assert(kRegions[0] == 32 && pairs_of(kRegionWidths[0]) <= 3 * 64, "steps of the smaller regions");
static_assert(kRegions[1] == 48 && pairs_of(kRegionWidths[0] + 1) > 3 * 64 && pairs_of(kRegionWidths[1]) <= 8 * 64,
              "steps of the larger regions");

// Orders this wave's LDS accesses for the compiler (the hardware runs a wave's
// LDS instructions in order): lanes read cells that other lanes wrote.
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float lane_f(float v, int i)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i));
}

// vis_value for an entry per lane
template <bool HALF>
__device__ __forceinline__ float2 lane_value(const JobDesc &d, const int4 &en)
{
    if constexpr (!HALF) {
        if (!d.data) return make_float2(1.f, 0.f);   // PSF gridding: data == 1 + 0i
        return static_cast<const float2 *>(d.data)[en.z];
    } else {
        const half2_t v = static_cast<const half2_t *>(d.data)[en.z];
        const float sc = d.dataScale * d.planeScale[entry_plane(en, d)];
        return make_float2((float)v.x * sc, (float)v.y * sc);
    }
}

// An entry's place in its region: byte offsets of its first cell and of the cell
// after it.
struct Place {
    int a, b;
};
template <int R>
__device__ __forceinline__ Place place_at(int x, int y)
{
    const int c = (y * Region<R>::RS + (x >> 1)) * 8;
    return x & 1 ? Place{c + (int)Region<R>::PB, c + 8} : Place{c, c + (int)Region<R>::PB};
}
template <int R>
__device__ __forceinline__ Place place_of(const int4 &en, int Bx, int By)
{
    return place_at<R>((en.x & 0xFFFF) - Bx, (int)((unsigned)en.x >> 16) - By);
}

// Lane positions in a footprint of width s, walked as the flat index p over its
// wp = ceil(s / 2) pairs of columns a row, step j of a group of G lanes taking
// p = lane % G + G j.  An odd width's last pair has its second cell outside:
// its tap is the next one in the table, times an exact zero.
template <int J>
struct Steps {
    int s = 0, n = 0;      // width and pairs
    unsigned tap[J];       // byte offset from the first tap; kOOB past the end
    unsigned cell[J];      // byte offset from the first cell
    bool out[J];           // the pair's second cell is outside
    bool in[J];            // p < n
};

template <int J, int G, int RS, unsigned TB>
__device__ __forceinline__ void set_steps(Steps<J> &S, int s, int lane)
{
    const int wp = (s + 1) >> 1;
    S.s = s;
    S.n = wp * s;
    const float rw = 1.f / (float)wp;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int p = lane % G + G * j;
        // p + 0.5 is at least 1 / (2 wp) from a multiple of wp
        const int row = (int)(((float)p + 0.5f) * rw), k = p - row * wp;
        S.in[j] = p < S.n;
        S.tap[j] = S.in[j] ? (unsigned)(row * s + 2 * k) * TB : kOOB;
        S.cell[j] = S.in[j] ? (unsigned)(row * RS + k) * 8u : 0u;
        S.out[j] = (s & 1) && k == wp - 1;
    }
}

// The pair of taps at a byte offset; EDGE (the run has an entry at the table's
// end): tap by tap, the one after the table as zero.  The runs that need it are
// compiled apart: a branch here would leave the number of loads in flight open
// and make every use wait for all of them.
template <bool HALF, bool EDGE>
__device__ __forceinline__ float4 pair_at(__amdgpu_buffer_rsrc_t rc, unsigned off, bool out)
{
    if constexpr (!EDGE) return load_pair<HALF>(rc, off);
    constexpr unsigned TB = Taps<HALF>::kBytes;
    const float2 a = Taps<HALF>::load(rc, off);
    const float2 b = Taps<HALF>::load(rc, out || off >= kOOB ? kOOB : off + TB);
    return make_float4(a.x, a.y, b.x, b.y);
}

// The entries [i, i + returned) of a block that share entry i's width
__device__ __forceinline__ int run_length(int width, int i, int m, int lane)
{
    const int s = __builtin_amdgcn_readlane(width, i);
    const unsigned long long same = __ballot(lane < m && width == s) >> i;
    return ~same == 0ull ? 64 - i : __builtin_ctzll(~same);
}

// Adds an entry's taps c to the region: all its cells are read before the first
// is written (a lane's J cells are distinct), so that one wait serves them all.
// Every step but the last is full; the last one's lanes past the end are off.
template <int J>
__device__ __forceinline__ void add_steps(char *lds, const Steps<J> &S, const float4 *c, int A, int B, float dx,
                                          float dy, int nSteps, bool inLast)
{
    float2 u[J], v[J];
    auto on = [&](int j) { return j + 1 < nSteps || (j + 1 == nSteps && inLast); };
#pragma unroll
    for (int j = 0; j < J; ++j)
        if (on(j)) {
            u[j] = *reinterpret_cast<float2 *>(lds + (S.cell[j] + A));
            v[j] = *reinterpret_cast<float2 *>(lds + (S.cell[j] + B));
        }
#pragma unroll
    for (int j = 0; j < J; ++j) {
        u[j].x = fmaf(dx, c[j].x, fmaf(-dy, c[j].y, u[j].x));
        u[j].y = fmaf(dx, c[j].y, fmaf(dy, c[j].x, u[j].y));
        const float wx = fmaf(dx, c[j].z, fmaf(-dy, c[j].w, v[j].x));
        const float wy = fmaf(dx, c[j].w, fmaf(dy, c[j].z, v[j].y));
        v[j].x = S.out[j] ? v[j].x : wx;
        v[j].y = S.out[j] ? v[j].y : wy;
    }
#pragma unroll
    for (int j = 0; j < J; ++j)
        if (on(j)) {
            *reinterpret_cast<float2 *>(lds + (S.cell[j] + A)) = u[j];
            *reinterpret_cast<float2 *>(lds + (S.cell[j] + B)) = v[j];
        }
    wave_order();
}

// ---- gridder ------------------------------------------------------------------
// attic/tConvolveMPI/Benchmark.cc:131-154: the wave adds the entries' footprints
// to its region in entry order, every cell rounded as by the other gridders.
// Four steps of taps are in flight beside the four being added.
template <int R, bool HALF, bool MANY>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(R == 32 ? 5 : 2)))
void k_grid_narrow(JobDesc one, const JobDesc *__restrict__ jobs)
{
    const JobDesc jd = MANY ? jobs[blockIdx.y] : one;
    using T = Region<R>;
    constexpr int RS = T::RS, D = 4;
    constexpr unsigned TB = Taps<HALF>::kBytes;
    __shared__ float2 cells[2 * T::PC];
    const int lane = threadIdx.x;
    const int nItems = __builtin_amdgcn_readfirstlane(jd.meta[0]);
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(jd.C, jd.cBytes);
    const int nTaps = (int)(jd.cBytes / TB);
    const int4 *__restrict__ entries = jd.entries;
    const int gSize = jd.gSize;
    char *const lds = reinterpret_cast<char *>(cells);

    for (int item = blockIdx.x; item < nItems; item += gridDim.x) {
        const int4 it = cload(jd.items, item);
        const int tyi = it.x / jd.nTX, txi = it.x - tyi * jd.nTX;
        const int Bx = txi * jd.strideW, By = tyi * jd.strideH;
        const int last = it.y + it.z - 1;

        auto entry_block = [&](int b) { return entries[min(b + lane, last)]; };
        int4 enC = entry_block(it.y), enN = entry_block(it.y + 64);
        float2 dC = lane_value<HALF>(jd, enC);
        for (int i = lane; i < T::PC; i += 64) reinterpret_cast<float4 *>(cells)[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        wave_order();

        for (int b = it.y; b <= last; b += 64) {
            const float2 dN = lane_value<HALF>(jd, enN);
            const int4 enNN = entry_block(b + 128);
            const int m = min(64, last + 1 - b);
            const Place at = place_of<R>(enC, Bx, By);
            const int width = entry_width(enC.w), tap0 = enC.y;
            // entries [i0, i1) of one width, J steps each
            auto run = [&](auto jTag, auto edgeTag, int s, int i0, int i1) {
                constexpr int J = decltype(jTag)::value, E = J == 1 ? D : J == 2 ? D / 2 : 1;
                constexpr bool EDGE = decltype(edgeTag)::value;
                Steps<J> S;
                set_steps<J, 64, RS, TB>(S, s, lane);
                const int steps = J <= 4 ? J : (S.n + 63) >> 6;
                const bool inLast = lane + 64 * (steps - 1) < S.n;
                auto fill = [&](float4 (&c)[E][J], int i) {
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        // past the run: its last entry again, not added
                        const unsigned off = (unsigned)__builtin_amdgcn_readlane(tap0, min(i + e, i1 - 1)) * TB;
#pragma unroll
                        for (int j = 0; j < J; ++j) c[e][j] = pair_at<HALF, EDGE>(rc, S.tap[j] + off, S.out[j]);
                    }
                };
                auto drain = [&](const float4 (&c)[E][J], int i) {
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        if (i + e >= i1) break;   // wave-uniform
                        add_steps<J>(lds, S, c[e], __builtin_amdgcn_readlane(at.a, i + e),
                                     __builtin_amdgcn_readlane(at.b, i + e), lane_f(dC.x, i + e),
                                     lane_f(dC.y, i + e), steps, inLast);
                    }
                };
                float4 a[E][J], z[E][J];
                fill(a, i0);
                for (int i = i0; i < i1; i += 2 * E) {
                    fill(z, i + E);
                    drain(a, i);
                    fill(a, i + 2 * E);
                    drain(z, i + E);
                }
            };
            for (int i = 0; i < m;) {
                const int s = __builtin_amdgcn_readlane(width, i);
                const int i1 = min(m, i + run_length(width, i, m, lane));
                const int n = ((s + 1) >> 1) * s;
                auto by_edge = [&](auto jTag) {
                    if (__any(lane >= i && lane < i1 && tap0 + s * s >= nTaps)) run(jTag, std::true_type{}, s, i, i1);
                    else run(jTag, std::false_type{}, s, i, i1);
                };
                if constexpr (R == 32) {
                    if (n <= 64) by_edge(std::integral_constant<int, 1>{});
                    else if (n <= 128) by_edge(std::integral_constant<int, 2>{});
                    else by_edge(std::integral_constant<int, 3>{});
                } else {
                    if (n <= 64 * 4) by_edge(std::integral_constant<int, 4>{});
                    else if (n <= 64 * 6) by_edge(std::integral_constant<int, 6>{});
                    else by_edge(std::integral_constant<int, 8>{});
                }
                i = i1;
            }
            enC = enN;
            dC = dN;
            enN = enNN;
        }

        // flush, a lane per float: contiguous atomics (regions overlap)
        const float *f0 = reinterpret_cast<const float *>(cells);
        const int rows = min(R, gSize - By), floats = min(2 * R, 2 * (gSize - Bx));
        float *g0 = reinterpret_cast<float *>(jd.grid + (size_t)By * gSize + Bx);
        for (int q = lane; q < R * R * 2; q += 64) {
            const int r = q / (2 * R), fl = q % (2 * R);
            // float fl of a row: column fl / 2
            const float v = f0[(((fl >> 1) & 1) * T::PC + r * RS + (fl >> 2)) * 2 + (fl & 1)];
            if (v != 0.f && r < rows && fl < floats) unsafeAtomicAdd(g0 + (size_t)r * gSize * 2 + fl, v);
        }
        wave_order();
    }
}

// ---- degridder ----------------------------------------------------------------
// attic/tConvolveMPI/Benchmark.cc:165-193: the region is loaded once an item; a
// group of G lanes takes an entry (G = 16 for footprints of up to 64 pairs, 32
// for up to 128, else 64), so that short footprints share the loads, the
// reduction and the waits of a wave.
template <int R, bool HALF, bool MANY>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(R == 32 ? 4 : 2)))
void k_degrid_narrow(JobDesc one, const JobDesc *__restrict__ jobs)
{
    const JobDesc jd = MANY ? jobs[blockIdx.y] : one;
    using T = Region<R>;
    constexpr int RS = T::RS;
    constexpr unsigned TB = Taps<HALF>::kBytes;
    __shared__ float2 cells[2 * T::PC];
    const int lane = threadIdx.x;
    const int nItems = __builtin_amdgcn_readfirstlane(jd.meta[0]);
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(jd.C, jd.cBytes);
    const int nTaps = (int)(jd.cBytes / TB);
    const int4 *__restrict__ entries = jd.entries;
    const float2 *__restrict__ grid = jd.grid;
    const int gSize = jd.gSize;
    const char *const lds = reinterpret_cast<const char *>(cells);
    for (int i = lane; i < T::PC; i += 64) reinterpret_cast<float4 *>(cells)[i] = make_float4(0.f, 0.f, 0.f, 0.f);

    for (int item = blockIdx.x; item < nItems; item += gridDim.x) {
        const int4 it = cload(jd.items, item);
        const int tyi = it.x / jd.nTX, txi = it.x - tyi * jd.nTX;
        const int Bx = txi * jd.strideW, By = tyi * jd.strideH;
        const int last = it.y + it.z - 1;

        auto entry_block = [&](int b) { return entries[min(b + lane, last)]; };
        int4 enC = entry_block(it.y);
        constexpr int kPairs = R * R / 2, kPer = (kPairs + 63) / 64, kBlk = 5;
        wave_order();
        for (int i0 = 0; i0 < kPer; i0 += kBlk) {
            float4 v[kBlk];
#pragma unroll
            for (int b = 0; b < kBlk; ++b) {
                const int q = lane + 64 * (i0 + b);
                const int row = By + q / (R / 2), col = Bx + 2 * (q % (R / 2));
                v[b] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (q < kPairs && row < gSize && col < gSize) {
                    const float2 *g = grid + (size_t)row * gSize + col;
                    if (col + 1 < gSize) {
                        __builtin_memcpy(&v[b], g, 16);   // 8-byte aligned when gSize or the stride is odd
                    } else {
                        const float2 a = *g;
                        v[b].x = a.x;
                        v[b].y = a.y;
                    }
                }
            }
#pragma unroll
            for (int b = 0; b < kBlk; ++b) {
                const int q = lane + 64 * (i0 + b);
                if (q < kPairs) {
                    const int c = (q / (R / 2)) * RS + q % (R / 2);
                    cells[c] = make_float2(v[b].x, v[b].y);
                    cells[T::PC + c] = make_float2(v[b].z, v[b].w);
                }
            }
        }
        wave_order();

        for (int b = it.y; b <= last; b += 64) {
            const int4 enN = entry_block(b + 64);
            const int m = min(64, last + 1 - b);
            const Place at = place_of<R>(enC, Bx, By);
            const int width = entry_width(enC.w), tap0 = enC.y, pl = HALF ? entry_plane(enC, jd) : 0;
            // entries [i0, i1) of one width, G lanes and J steps each
            auto run = [&](auto gTag, auto jTag, auto edgeTag, int s, int i0, int i1) {
                constexpr int G = decltype(gTag)::value, J = decltype(jTag)::value;
                constexpr bool EDGE = decltype(edgeTag)::value;
                constexpr int E = 64 / G, Q = J <= 3 ? 2 : 1;   // entries a round, rounds in flight
                const int grp = lane / G;
                Steps<J> S;
                set_steps<J, G, RS, TB>(S, s, lane);
                auto entry_of = [&](int i) { return min(i + grp, i1 - 1); };
                auto fill = [&](float4 (&c)[Q][J], int i) {
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        // past the run: its last entry again, not stored
                        const int c0 = G == 64 ? __builtin_amdgcn_readlane(tap0, min(i + q, i1 - 1))
                                               : __shfl(tap0, entry_of(i + q * E), 64);
#pragma unroll
                        for (int j = 0; j < J; ++j)
                            c[q][j] = pair_at<HALF, EDGE>(rc, S.tap[j] + (unsigned)c0 * TB, S.out[j]);
                    }
                };
                auto drain = [&](const float4 (&c)[Q][J], int i) {
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        if (i + q * E >= i1) break;
                        const int k = entry_of(i + q * E);
                        const int A = G == 64 ? __builtin_amdgcn_readlane(at.a, i + q) : __shfl(at.a, k, 64);
                        const int B = G == 64 ? __builtin_amdgcn_readlane(at.b, i + q) : __shfl(at.b, k, 64);
                        float sr = 0.f, si = 0.f;
#pragma unroll
                        for (int j = 0; j < J; ++j) {
                            const float2 u = *reinterpret_cast<const float2 *>(lds + (S.cell[j] + A));
                            const float2 v = *reinterpret_cast<const float2 *>(lds + (S.cell[j] + B));
                            // lanes past the end (of the last steps) and second cells outside
                            // don't count, whatever their taps and cells hold
                            const bool ends = J <= 4 ? j == J - 1 : j >= J / 2;
                            const bool in0 = !ends || S.in[j], in1 = !S.out[j] && in0;
                            const float ur = fmaf(u.x, c[q][j].x, fmaf(-u.y, c[q][j].y, sr));
                            const float ui = fmaf(u.x, c[q][j].y, fmaf(u.y, c[q][j].x, si));
                            sr = in0 ? ur : sr;
                            si = in0 ? ui : si;
                            const float vr = fmaf(v.x, c[q][j].z, fmaf(-v.y, c[q][j].w, sr));
                            const float vi = fmaf(v.x, c[q][j].w, fmaf(v.y, c[q][j].z, si));
                            sr = in1 ? vr : sr;
                            si = in1 ? vi : si;
                        }
                        if constexpr (G == 64) {
                            sr = wave_sum(sr);
                            si = wave_sum(si);
                        } else {
                            sr = row_sum(sr);
                            si = row_sum(si);
                            if constexpr (G == 32) {
                                sr += __shfl_xor(sr, 16, 64);
                                si += __shfl_xor(si, 16, 64);
                            }
                        }
                        const int vis = __shfl(enC.z, k, 64);
                        if constexpr (HALF) {
                            const float ps = jd.planeScale[__shfl(pl, k, 64)];
                            sr *= ps;
                            si *= ps;
                        }
                        if (lane % G == 0 && i + q * E + grp < i1) {
                            if constexpr (MANY) {   // jobs may share their output: added to the cleared values
                                unsafeAtomicAdd(&jd.out[vis].x, sr);
                                unsafeAtomicAdd(&jd.out[vis].y, si);
                            } else {
                                jd.out[vis] = make_float2(sr, si);
                            }
                        }
                    }
                };
                float4 a[Q][J], z[Q][J];
                fill(a, i0);
                for (int i = i0; i < i1; i += 2 * Q * E) {
                    fill(z, i + Q * E);
                    drain(a, i);
                    fill(a, i + 2 * Q * E);
                    drain(z, i + Q * E);
                }
            };
            auto by_edge = [&](auto gTag, auto jTag, int s, int i0, int i1) {
                if (__any(lane >= i0 && lane < i1 && tap0 + s * s >= nTaps))
                    run(gTag, jTag, std::true_type{}, s, i0, i1);
                else
                    run(gTag, jTag, std::false_type{}, s, i0, i1);
            };
            auto by_steps = [&](auto gTag, int s, int i0, int i1, int steps) {
                if (steps == 1) by_edge(gTag, std::integral_constant<int, 1>{}, s, i0, i1);
                else if (steps == 2) by_edge(gTag, std::integral_constant<int, 2>{}, s, i0, i1);
                else if (steps == 3) by_edge(gTag, std::integral_constant<int, 3>{}, s, i0, i1);
                else by_edge(gTag, std::integral_constant<int, 4>{}, s, i0, i1);
            };
            for (int i = 0; i < m;) {
                const int s = __builtin_amdgcn_readlane(width, i);
                const int i1 = min(m, i + run_length(width, i, m, lane));
                const int n = ((s + 1) >> 1) * s;
                using W = std::integral_constant<int, 64>;
                if constexpr (R == 32) {
                    if (n <= 64) by_steps(std::integral_constant<int, 16>{}, s, i, i1, (n + 15) / 16);
                    else if (n <= 128) by_steps(std::integral_constant<int, 32>{}, s, i, i1, (n + 31) / 32);
                    else by_edge(W{}, std::integral_constant<int, 3>{}, s, i, i1);
                } else {
                    if (n <= 64 * 4) by_edge(W{}, std::integral_constant<int, 4>{}, s, i, i1);
                    else if (n <= 64 * 6) by_edge(W{}, std::integral_constant<int, 6>{}, s, i, i1);
                    else by_edge(W{}, std::integral_constant<int, 8>{}, s, i, i1);
                }
                i = i1;
            }
            enC = enN;
        }
        wave_order();
    }
}

}  // namespace

// The kernels of a region size; many: FP32 storage, a job to each blockIdx.y.
static auto narrow_kernel(int region, bool half, bool degrid, bool many) -> void (*)(JobDesc, const JobDesc *)
{
#define X(R)                                                                                   \
    if (region == R)                                                                           \
        return many ? (degrid ? k_degrid_narrow<R, false, true> : k_grid_narrow<R, false, true>) \
               : half ? (degrid ? k_degrid_narrow<R, true, false> : k_grid_narrow<R, true, false>) \
                      : (degrid ? k_degrid_narrow<R, false, false> : k_grid_narrow<R, false, false>);
    X(32) X(48)
#undef X
    return nullptr;
}

tcv_status launch_narrow(tcv_ctx *ctx, const JobDesc &jd, int region, bool half, bool degrid)
{
    const auto k = narrow_kernel(region, half, degrid, false);
    if (!k) return tcv_fail(ctx, TCV_ERR_UNSUPPORTED, "region size not built");
    int per = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void *)k, 64, 0) != hipSuccess || per < 1) per = 1;
    ProfScope ps(ctx, degrid ? (half ? "degrid_tiled_half" : "degrid_tiled") : (half ? "grid_tiled_half" : "grid_tiled"));
    hipLaunchKernelGGL(k, dim3(std::max(1, ctx->cus) * per), dim3(64), 0, ctx->stream, jd, (const JobDesc *)nullptr);
    TCV_HIP(ctx, hipGetLastError());
    return TCV_OK;
}

tcv_status launch_narrow_many(tcv_ctx *ctx, const JobDesc *d_jobs, int nJobs, int region, bool degrid)
{
    const auto k = narrow_kernel(region, false, degrid, true);
    if (!k) return tcv_fail(ctx, TCV_ERR_UNSUPPORTED, "region size not built");
    int per = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void *)k, 64, 0) != hipSuccess || per < 1) per = 1;
    // four times the resident waves among the jobs, 16 at least to a job: an uneven
    // job's waves end early and leave their place to the next one's
    const int full = std::max(1, ctx->cus) * per;
    const int x = std::min(full, std::max(16, 4 * full / nJobs));
    ProfScope ps(ctx, degrid ? "degrid_batch" : "grid_batch");
    for (int j0 = 0; j0 < nJobs; j0 += 65535) {
        hipLaunchKernelGGL(k, dim3(x, std::min(nJobs - j0, 65535)), dim3(64), 0, ctx->stream, JobDesc{}, d_jobs + j0);
        TCV_HIP(ctx, hipGetLastError());
    }
    return TCV_OK;
}
