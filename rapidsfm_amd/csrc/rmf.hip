// rmf.hip - per-cell affine RANSAC match filter.
//
// Reference: rmf::cudaRansacMatchFilter (RansacMatchFilter.cu:394-419) and its
// kernels kernelFindBestAffineForCells (:196-279),
// kernelTryBestAffineOfOtherCellsAndVote (:281-338) and kernelComputeVotes
// (:341-391); host side RansacMatchFilter::getInlierMask (RansacMatchFilter.cpp:40-135).
// Semantics kept: 3x3-cell neighbourhoods, 3 distinct draws per hypothesis
// from the glibc LCG, Gauss elimination without pivoting, scale gate
// det in [1/16, 16], inlier radius threshold * min(sqrt(det), 1), strict
// best-count per thread, the CTA tree reduction of CtaReducer::findMax, and a
// vote for every inlier of a cell whose best affine has >= 6 inliers.
// Deliberate differences (determinism): the LCG seed is an argument instead of
// clock(); a cell with fewer than 9 neighbourhood matches stores a NaN affine
// (the reference leaves it unwritten); every thread votes with the CTA-best
// count (the reference tests partial per-thread counts before a barrier).
#include "internal.hpp"
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

namespace rsfm_amd {
namespace rmf {

constexpr int kCta = 128;
constexpr uint32_t kMinInliers = 6;

// a cell's 3 x 3 neighbourhood: its matches are three runs of the cell-ordered
// array, one per cell row (cells of a row are consecutive)
struct Cells {
    uint32_t start[3], end[3];  // end: of the runs' concatenation
    uint32_t sum;
};

__device__ inline void cells_init(Cells& c, const uint32_t* bounds, uint32_t cols, uint32_t rows, uint32_t bx, uint32_t by)
{
    c.sum = 0;
    const uint32_t n0 = bx > 0 ? bx - 1 : 0, n1 = min(bx + 1, cols - 1);
#pragma unroll
    for (int t = 0; t < 3; t++) {
        const int m = (int)by - 1 + t;
        c.start[t] = 0;
        if (m >= 0 && m < (int)rows) {
            c.start[t] = bounds[(uint32_t)m * cols + n0];
            c.sum += bounds[(uint32_t)m * cols + n1 + 1] - c.start[t];
        }
        c.end[t] = c.sum;
    }
}

// place of the neighbourhood's idx-th match (idx < sum)
__device__ inline uint32_t cells_map(const Cells& c, uint32_t idx)
{
    if (idx < c.end[0]) return c.start[0] + idx;
    if (idx < c.end[1]) return c.start[1] + (idx - c.end[0]);
    return c.start[2] + (idx - c.end[1]);
}

__device__ inline float sq_threshold(const float T[6], float threshold)
{
    const float sqrScale = T[0] * T[4] - T[1] * T[3];
    const float scale = sqrtf(sqrScale);
    const float s = (1.f < scale) ? 1.f : scale;  // std::min(scale, 1.f), NaN kept
    const float th = threshold * s;
    return th * th;
}

__device__ inline bool is_inlier(const float T[6], float4 p, float sq)
{
    const float d0 = ((T[0] * p.x + T[1] * p.y) + T[2]) - p.z;
    const float d1 = ((T[3] * p.x + T[4] * p.y) + T[5]) - p.w;
    return d0 * d0 + d1 * d1 < sq;
}

// Inlier counts of one affine per lane over a neighbourhood, by the matrix
// cores. d0 = T0 x + T1 y + T2 - x' and d1 are matrix products with f16 halves
// (22 bits) of the coordinates about the neighbourhood's first match and of the
// coefficients, ten of K = 16 slots each; s = d0^2 + d1^2 - sq then differs from
// the FP32 test's by at most the model's c (below), so s < -c and s > c have
// the exact outcome and only tests between are done by is_inlier. Four vector
// instructions per test instead of seventeen: v_fma twice, v_alignbit (sign
// bits, one popcount per 32 tests) and, per four tests, the least |s| less c
// (v_min3, v_min, v_sub, v_alignbit).
// 64 pairs of about 4000 matches in 16 x 12 cells, 256 hypotheses: best affine
// 327 -> 126 us, votes 284 -> 110 us (the exact test per lane and match had 17
// instructions and its match's load in the chain).
// The bound, u = 2^-24, M = the largest magnitudes in the neighbourhood about
// its first match, m the same in pixels: a staged term is off by 13 u (the
// subtraction, two splits of 2^-22, the dropped lo * lo), the matrix unit's
// FP32 sum by 10 u of the terms' magnitudes (assumed; 5.9 u measured), halves below
// f16's normal range by 2^-14 absolute; the exact expression rounds at most
// 3 u (|T0| mx + |T1| my) + 2 u (|T2| + mx').
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
constexpr uint32_t kTiles = 16, kChunk = kTiles * 16;  // matches staged at a time
constexpr float kScale = 64.f;                         // coefficients are staged times 2^6
constexpr float kFar = 32768.f;

struct Half2 {
    _Float16 h, l;
};
__device__ inline Half2 split(float x)
{
    asm("" : "+v"(x));  // one rounding for both uses of x (no v_fma_mixlo_f16)
    Half2 r;
    r.h = (_Float16)x;
    r.l = (_Float16)(x - (float)r.h);
    return r;
}

struct CountSmem {
    v4h tile[kTiles][64];             // matches as matrix operands, [lane] = (match, K group)
    float4 raw[kChunk];               // the same matches as they are
    v4h model[kCta / 64][2][2][64];   // [wave][d0, d1][K group][model]
    float T[kCta / 64][6][64];
    float sq[kCta / 64][64];
    float big[kCta / 64][4];
};

// a neighbourhood's centre (its first match) and largest magnitudes about it
struct Frame {
    float cx, cy, cz, cw, x, y, z, w;
    bool odd;  // coordinates beyond the bound: every test is exact
};

// largest value of the wave (float or uint32_t)
template <class V>
__device__ inline V wave_max(V x)
{
    const auto most = [](V a, V b) {
        if constexpr (std::is_same_v<V, float>) return fmaxf(a, b);
        else return max(a, b);
    };
    const auto dpp = [](V v, auto k) {
        return __builtin_bit_cast(V, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(k)::value, 0xF, 0xF, true));
    };
    x = most(x, dpp(x, std::integral_constant<int, 0xB1>{}));   // quad_perm: neighbour
    x = most(x, dpp(x, std::integral_constant<int, 0x4E>{}));   // quad_perm: other pair
    x = most(x, dpp(x, std::integral_constant<int, 0x141>{}));  // row_half_mirror
    x = most(x, dpp(x, std::integral_constant<int, 0x140>{}));  // row_mirror
    uint32_t u = __builtin_bit_cast(uint32_t, x);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    x = most(__builtin_bit_cast(V, (uint32_t)a[0]), __builtin_bit_cast(V, (uint32_t)a[1]));
    u = __builtin_bit_cast(uint32_t, x);
    const auto b = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return most(__builtin_bit_cast(V, (uint32_t)b[0]), __builtin_bit_cast(V, (uint32_t)b[1]));
}

__device__ inline void frame_add(Frame& f, const float4& p)
{
    f.x = fmaxf(f.x, fabsf(p.x - f.cx));
    f.y = fmaxf(f.y, fabsf(p.y - f.cy));
    f.z = fmaxf(f.z, fabsf(p.z - f.cz));
    f.w = fmaxf(f.w, fabsf(p.w - f.cw));
    f.odd = f.odd || !(fabsf(p.x) + fabsf(p.y) + fabsf(p.z) + fabsf(p.w) < 1e6f);
}

// match i of the chunk (valid: there is one) to S.tile: K groups
// {x.h x.h x.l 64}, {y.h y.h y.l 64}, {x'.h x'.l y'.h y'.l}, {pad, 1024, 0, 0}
__device__ __forceinline__ void stage_match(CountSmem& S, const Frame& f, uint32_t i, bool valid, const float4& p)
{
    const _Float16 z = (_Float16)0.f;
    const Half2 x = split(p.x - f.cx), y = split(p.y - f.cy), u = split(p.z - f.cz), v = split(p.w - f.cw);
    v4h* t = S.tile[i >> 4] + (i & 15);
    t[0] = valid ? v4h{x.h, x.h, x.l, (_Float16)kScale} : v4h{z, z, z, z};
    t[16] = valid ? v4h{y.h, y.h, y.l, (_Float16)kScale} : v4h{z, z, z, z};
    t[32] = valid ? v4h{u.h, u.l, v.h, v.l} : v4h{z, z, z, z};
    t[48] = valid ? v4h{z, (_Float16)1024.f, z, z} : v4h{(_Float16)kFar, z, z, z};
}

// The neighbourhood's frame and, when it fits one chunk, its matches staged
// (each is loaded once). All threads of the workgroup call it; c.sum > 0.
__device__ __forceinline__ Frame stage_cell(CountSmem& S, const Cells& c, const float4* __restrict__ m)
{
    constexpr uint32_t kPer = kChunk / kCta;
    const uint32_t tid = threadIdx.x;
    const bool one = c.sum <= kChunk;
    float4 p[kPer];
    if (one) {
#pragma unroll
        for (uint32_t u = 0; u < kPer; u++) p[u] = m[cells_map(c, min(tid + u * kCta, c.sum - 1))];
    }
    const float4 o = m[cells_map(c, 0)];
    Frame f{o.x, o.y, o.z, o.w, 0.f, 0.f, 0.f, 0.f, false};
    if (one) {
#pragma unroll
        for (uint32_t u = 0; u < kPer; u++) frame_add(f, p[u]);
    } else {
        for (uint32_t k = tid; k < c.sum; k += kCta) frame_add(f, m[cells_map(c, k)]);
    }
    f.x = wave_max(f.odd ? 1e6f : f.x);
    f.y = wave_max(f.y);
    f.z = wave_max(f.z);
    f.w = wave_max(f.w);
    if ((tid & 63) == 0) {
        S.big[tid >> 6][0] = f.x;
        S.big[tid >> 6][1] = f.y;
        S.big[tid >> 6][2] = f.z;
        S.big[tid >> 6][3] = f.w;
    }
    if (one) {
#pragma unroll
        for (uint32_t u = 0; u < kPer; u++) {
            const uint32_t i = tid + u * kCta;
            if (i < ((c.sum + 15) & ~15u)) {
                stage_match(S, f, i, i < c.sum, p[u]);
                S.raw[i] = p[u];
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kCta / 64; w++) {
        f.x = fmaxf(f.x, S.big[w][0]);
        f.y = fmaxf(f.y, S.big[w][1]);
        f.z = fmaxf(f.z, S.big[w][2]);
        f.w = fmaxf(f.w, S.big[w][3]);
    }
    f.odd = !(fmaxf(fmaxf(f.x, f.y), fmaxf(f.z, f.w)) < 30000.f);
    return f;
}

// matches [at, at + kChunk) of a longer neighbourhood
__device__ __forceinline__ void stage_chunk(CountSmem& S, const Cells& c, const Frame& f, const float4* __restrict__ m, uint32_t at)
{
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kChunk; i += kCta) {
        const float4 p = m[cells_map(c, min(at + i, c.sum - 1))];
        stage_match(S, f, i, at + i < c.sum, p);
        S.raw[i] = p;
    }
    __syncthreads();
}

// inliers of the lane's affine T (live: it has any) over the neighbourhood;
// every thread of the workgroup calls it
__device__ __forceinline__ uint32_t count_inliers(CountSmem& S, const Cells& c, const Frame& f, const float T[6], bool live,
                                         const float4* __restrict__ m, float threshold)
{
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, q = lane >> 4;
    const float sq = sq_threshold(T, threshold);
    live = live && sq > 0.f;  // false for NaN too: such a model has no inliers
    if (f.odd) {
        uint32_t cnt = 0;
        if (live)
            for (uint32_t k = 0; k < c.sum; k++) cnt += is_inlier(T, m[cells_map(c, k)], sq);
        return cnt;
    }
    // the model about the frame's centre, its operands and c
    const float t0 = fabsf(T[0]), t1 = fabsf(T[1]), t3 = fabsf(T[3]), t4 = fabsf(T[4]);
    const double o0 = (double)T[0] * f.cx + (double)T[1] * f.cy + ((double)T[2] - f.cz);
    const double o1 = (double)T[3] * f.cx + (double)T[4] * f.cy + ((double)T[5] - f.cw);
    const float a0 = (float)fabs(o0), a1 = (float)fabs(o1);
    const float px = f.x + fabsf(f.cx), py = f.y + fabsf(f.cy), pz = f.z + fabsf(f.cz), pw = f.w + fabsf(f.cw);
    const float u = 5.9604645e-8f;
    // an inlier's x' is within the threshold of the model's value: larger ones do not reach the boundary
    const float th = sqrtf(sq);
    const float z0 = t0 * f.x + t1 * f.y + a0, z1 = t3 * f.x + t4 * f.y + a1;
    const float e0 = u * (23.f * (z0 + fminf(f.z, z0 + 2.f * th)) + 3.f * (t0 * px + t1 * py) + 2.f * (fabsf(T[2]) + pz)) +
                     6.2e-5f * (t0 + t1 + 3.f) + 1e-6f * (f.x + f.y);
    const float e1 = u * (23.f * (z1 + fminf(f.w, z1 + 2.f * th)) + 3.f * (t3 * px + t4 * py) + 2.f * (fabsf(T[5]) + pw)) +
                     6.2e-5f * (t3 + t4 + 3.f) + 1e-6f * (f.x + f.y);
    const float cc = 1.05f * (2.f * th * (e0 + e1) + e0 * e0 + e1 * e1 + 16.f * u * sq);
    // a model that maps the whole neighbourhood further from its matches than the
    // threshold (another cell's, extrapolated) has no inlier: in exact arithmetic
    // d0 is at least a0 - (t0 x + t1 y + z) throughout, and e0 holds the FP32
    // expression's own roundings, which for a steep model exceed the threshold;
    // the second th and e0 and the 1e-4 are for the roundings of these lines
    if (a0 * 0.9999f > t0 * f.x + t1 * f.y + f.z + 2.f * (th + e0) || a1 * 0.9999f > t3 * f.x + t4 * f.y + f.w + 2.f * (th + e1))
        live = false;
    // beyond f16's range: every test of the model is open
    const bool open = live && !(fmaxf(fmaxf(t0, t1), fmaxf(t3, t4)) < 500.f && fmaxf(a0, a1) < 30000.f && sq < 1e8f && cc < 1e8f);
    const bool use = live && !open;
    {
        const float k = use ? kScale : 0.f, k1 = use ? 1.f : 0.f;
        const Half2 x0 = split(T[0] * k), y0 = split(T[1] * k), x1 = split(T[3] * k), y1 = split(T[4] * k);
        const Half2 w0 = split((float)o0 * k1), w1 = split((float)o1 * k1);
        S.model[wave][0][0][lane] = use ? v4h{x0.h, x0.l, x0.h, w0.h} : v4h{0, 0, 0, 0};
        S.model[wave][0][1][lane] = use ? v4h{y0.h, y0.l, y0.h, w0.l} : v4h{0, 0, 0, 0};
        S.model[wave][1][0][lane] = use ? v4h{x1.h, x1.l, x1.h, w1.h} : v4h{0, 0, 0, 0};
        S.model[wave][1][1][lane] = use ? v4h{y1.h, y1.l, y1.h, w1.l} : v4h{0, 0, 0, 0};
#pragma unroll
        for (int k6 = 0; k6 < 6; k6++) S.T[wave][k6][lane] = T[k6];
        S.sq[wave][lane] = sq;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // operands of the wave's four blocks of 16 models; -sq and c in units of
    // (64 px)^2. A dead model's third group makes d0 huge; an open one has
    // s = 0, c = 1.
    v4h m0[4], m1[4];
    float sqn[4], cs[4];
    const _Float16 z = (_Float16)0.f, one = (_Float16)-kScale;
#pragma unroll
    for (int b = 0; b < 4; b++) {
        const int src = b * 16 + (int)c16;
        const float bs = __shfl(use ? sq * (kScale * kScale) : 0.f, src);
        const float bc = __shfl(use ? cc * (kScale * kScale) : (open ? 1.f : 0.f), src);
        const bool dead = __shfl(live ? 0 : 1, src) != 0, any = __shfl(use ? 1 : 0, src) != 0;
        sqn[b] = -bs;
        cs[b] = bc;
        if (q < 2) {
            m0[b] = S.model[wave][0][q][src];
            m1[b] = S.model[wave][1][q][src];
        } else if (q == 2) {
            m0[b] = any ? v4h{one, one, z, z} : v4h{z, z, z, z};
            m1[b] = any ? v4h{z, z, one, one} : v4h{z, z, z, z};
        } else {
            m0[b] = v4h{(_Float16)kFar, dead ? (_Float16)kFar : z, z, z};
            m1[b] = v4h{z, z, z, z};
        }
    }
    uint32_t acc[4] = {0, 0, 0, 0};
    for (uint32_t at = 0; at < c.sum; at += kChunk) {
        if (c.sum > kChunk) stage_chunk(S, c, f, m, at);
        const uint32_t tiles = min(kTiles, (c.sum - at + 15) / 16);
        for (uint32_t g0 = 0; g0 < tiles; g0 += 8) {
            const uint32_t nt = min(8u, tiles - g0);
            uint32_t in[4] = {0, 0, 0, 0}, near[4] = {0, 0, 0, 0};
            for (uint32_t t = 0; t < nt; t++) {
                const v4h a = S.tile[g0 + t][lane];
                const v4f zero = {0.f, 0.f, 0.f, 0.f};
                v4f d0[4], d1[4];
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    d0[b] = __builtin_amdgcn_mfma_f32_16x16x16f16(a, m0[b], zero, 0, 0, 0);
                    d1[b] = __builtin_amdgcn_mfma_f32_16x16x16f16(a, m1[b], zero, 0, 0, 0);
                }
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    float s[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        s[j] = fmaf(d1[b][j], d1[b][j], fmaf(d0[b][j], d0[b][j], sqn[b]));
                        in[b] = __builtin_amdgcn_alignbit(in[b], __float_as_uint(s[j]), 31);
                    }
                    const float low = fminf(fminf(fminf(fabsf(s[0]), fabsf(s[1])), fabsf(s[2])), fabsf(s[3])) - cs[b];
                    near[b] = __builtin_amdgcn_alignbit(near[b], __float_as_uint(low), 31);
                }
            }
            // open groups of four tests, each by its lane, exactly
            while (__any((near[0] | near[1] | near[2] | near[3]) != 0)) {
                uint32_t w = 0, k = 0;
#pragma unroll
                for (int b = 3; b >= 0; b--)
                    if (near[b]) {
                        w = near[b];
                        k = b;
                    }
                if (w) {
                    const uint32_t bit = (uint32_t)__ffs((int)w) - 1u, src = k * 16 + c16;
                    float M[6];
#pragma unroll
                    for (int k6 = 0; k6 < 6; k6++) M[k6] = S.T[wave][k6][src];
                    const float ms = S.sq[wave][src];
                    const uint32_t i = (g0 + nt - 1 - bit) * 16 + 4 * q;
                    uint32_t a = 0;
#pragma unroll
                    for (uint32_t j = 0; j < 4; j++)
                        a += at + i + j < c.sum && is_inlier(M, S.raw[i + j], ms) ? 1u : 0u;
#pragma unroll
                    for (int b = 0; b < 4; b++)
                        if ((uint32_t)b == k) {
                            near[b] &= w - 1;
                            in[b] &= ~(15u << (4 * bit));
                            acc[b] += a;
                        }
                }
            }
#pragma unroll
            for (int b = 0; b < 4; b++) acc[b] += (uint32_t)__popc(in[b]);
        }
    }
    // sums over the lane groups; the lane's model is number lane % 16 of block lane / 16
    uint32_t mine = 0;
#pragma unroll
    for (int b = 0; b < 4; b++) {
        uint32_t a = acc[b];
        a += (uint32_t)__shfl_xor((int)a, 16);
        a += (uint32_t)__shfl_xor((int)a, 32);
        if (q == (uint32_t)b) mine = a;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return live ? mine : 0u;
}

// solveGaussElim semantics (SfmUtils.hpp:156-184): no pivoting, 3x3 with two right-hand sides
__device__ inline void solve_gauss3(float Ab[3][5], float X[3][2])
{
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const float inv = 1.f / Ab[i][i];
#pragma unroll
        for (int j = i + 1; j < 3; j++) {
            const float factor = Ab[j][i] * inv;
#pragma unroll
            for (int k = i + 1; k < 5; k++) Ab[j][k] = Ab[j][k] - factor * Ab[i][k];
        }
    }
#pragma unroll
    for (int r = 0; r < 3; r++) {
        X[r][0] = Ab[r][3];
        X[r][1] = Ab[r][4];
    }
#pragma unroll
    for (int i = 2; i >= 0; i--) {
        const float inv = 1.f / Ab[i][i];
        X[i][0] = X[i][0] * inv;
        X[i][1] = X[i][1] * inv;
#pragma unroll
        for (int j = i - 1; j >= 0; j--) {
            const float factor = Ab[j][i];
            X[j][0] = X[j][0] - factor * X[i][0];
            X[j][1] = X[j][1] - factor * X[i][1];
        }
    }
}

__device__ inline uint32_t lcg(uint32_t& s)
{
    s = (s * 1103515245u + 12345u) & 0x7fffffffu;
    return s;
}

struct Reducer {
    uint32_t cnt[kCta / 64], order[kCta / 64];
    float aff[6];
};

// CtaReducer::findMax: the largest count; among equals its tree (thread t keeps
// its value unless t + mid holds a strictly larger count, mid = 64 .. 1) leaves
// the thread whose reversed index is lowest. The winner's count and affine are
// returned to every thread. Count and order are reduced one after the other: a
// key of both in 32 bits would leave the count 25.
__device__ __forceinline__ void cta_find_max(Reducer& R, uint32_t& cnt, float T[6])
{
    static_assert(kCta == 128, "seven index bits, two waves");
    const uint32_t mine = 128u - (__brev(threadIdx.x) >> 25);
    const uint32_t most = wave_max(cnt), first = wave_max(cnt == most ? mine : 0u);
    if ((threadIdx.x & 63) == 0) {
        R.cnt[threadIdx.x >> 6] = most;
        R.order[threadIdx.x >> 6] = first;
    }
    __syncthreads();
    const uint32_t c0 = R.cnt[0], c1 = R.cnt[1], o0 = R.order[0], o1 = R.order[1];
    const bool second = c1 > c0 || (c1 == c0 && o1 > o0);
    if (mine == (second ? o1 : o0))
#pragma unroll
        for (int q = 0; q < 6; q++) R.aff[q] = T[q];
    __syncthreads();
    cnt = second ? c1 : c0;
#pragma unroll
    for (int q = 0; q < 6; q++) T[q] = R.aff[q];
}

struct CellSmem {
    Reducer R;
    CountSmem C;
};

// one cell (bx, by): the best of nbTests affine hypotheses
__device__ __forceinline__ void best_affine_cell(CellSmem& S, float* __restrict__ affine, const float4* __restrict__ m,
                                        const uint32_t* __restrict__ bounds, uint32_t cols, uint32_t rows,
                                        uint32_t nbTests, float threshold, uint32_t seed, uint32_t bx, uint32_t by)
{
    Cells c;
    cells_init(c, bounds, cols, rows, bx, by);
    const uint32_t rank = by * cols + bx;
    if (c.sum < 9) {
        if (threadIdx.x < 6) affine[rank * 6 + threadIdx.x] = __builtin_nanf("");
        return;
    }
    const Frame f = stage_cell(S.C, c, m);
    float best[6] = {1.f, 0.f, 0.f, 0.f, 1.f, 0.f};
    uint32_t bestCnt = 0;
    uint32_t st = seed + (kCta * rank + threadIdx.x) * 22695477u;
    for (uint32_t h0 = 0; h0 < nbTests; h0 += kCta) {
        bool live = h0 + threadIdx.x < nbTests;
        float T[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (live) {
            uint32_t idx[3];
            uint32_t got = 0;
            while (got < 3) {
                const uint32_t v = lcg(st) % c.sum;
                bool dup = false;
                for (uint32_t q = 0; q < got; q++) dup |= idx[q] == v;
                if (!dup) idx[got++] = v;
            }
            float Ab[3][5];
#pragma unroll
            for (int r = 0; r < 3; r++) {
                const float4 p = c.sum <= kChunk ? S.C.raw[idx[r]] : m[cells_map(c, idx[r])];
                Ab[r][0] = p.x;
                Ab[r][1] = p.y;
                Ab[r][2] = 1.f;
                Ab[r][3] = p.z;
                Ab[r][4] = p.w;
            }
            float X[3][2];
            solve_gauss3(Ab, X);
#pragma unroll
            for (int r = 0; r < 3; r++) {
                T[r] = X[r][0];
                T[3 + r] = X[r][1];
            }
            const float sqrScale = T[0] * T[4] - T[1] * T[3];
            if (sqrScale < 0.0625f || sqrScale > 16.f || !isfinite(sqrScale)) live = false;
        }
        const uint32_t k = count_inliers(S.C, c, f, T, live, m, threshold);
        if (k > bestCnt) {
            bestCnt = k;
#pragma unroll
            for (int q = 0; q < 6; q++) best[q] = T[q];
        }
    }
    cta_find_max(S.R, bestCnt, best);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int q = 0; q < 6; q++) affine[rank * 6 + q] = best[q];
    }
}

__global__ __launch_bounds__(kCta, 4) void best_affine_kernel(float* __restrict__ affine, const float4* __restrict__ m,
                                                           const uint32_t* __restrict__ bounds, uint32_t cols,
                                                           uint32_t rows, uint32_t nbTests, float threshold, uint32_t seed)
{
    __shared__ CellSmem S;
    best_affine_cell(S, affine, m, bounds, cols, rows, nbTests, threshold, seed, blockIdx.x, blockIdx.y);
}

__device__ inline void vote(uint32_t* votesWords, uint32_t idx)
{
    atomicAdd(votesWords + (idx >> 2), 1u << (8 * (idx & 3)));
}

// one cell: its own affine (or, with tryOther, the best of every cell's affine
// on its neighbourhood) votes for its inliers when it explains >= 6 of them
__device__ __forceinline__ void vote_cell(CellSmem& S, uint32_t* __restrict__ votesWords, const float* __restrict__ affine,
                                 const float4* __restrict__ m, const uint32_t* __restrict__ bounds, uint32_t cols,
                                 uint32_t rows, float threshold, bool tryOther, uint32_t bx, uint32_t by)
{
    Cells c;
    cells_init(c, bounds, cols, rows, bx, by);
    if (c.sum < kMinInliers) return;  // nobody can explain that many
    const uint32_t rank = by * cols + bx;
    const uint32_t nCells = tryOther ? cols * rows : 1u;
    const Frame f = stage_cell(S.C, c, m);
    float best[6];
#pragma unroll
    for (int q = 0; q < 6; q++) best[q] = affine[rank * 6 + q];
    uint32_t bestCnt = 0;
    for (uint32_t n0 = 0; n0 < nCells; n0 += kCta) {
        const uint32_t n = n0 + threadIdx.x;
        const bool live = n < nCells;
        float T[6];
#pragma unroll
        for (int q = 0; q < 6; q++) T[q] = affine[(tryOther && live ? n : rank) * 6 + q];
        const uint32_t k = count_inliers(S.C, c, f, T, live, m, threshold);
        if (k > bestCnt) {
            bestCnt = k;
#pragma unroll
            for (int q = 0; q < 6; q++) best[q] = T[q];
        }
    }
    cta_find_max(S.R, bestCnt, best);
    if (bestCnt < kMinInliers) return;
    const float sq = sq_threshold(best, threshold);
    for (uint32_t k = threadIdx.x; k < c.sum; k += kCta) {
        const uint32_t mi = cells_map(c, k);
        if (is_inlier(best, c.sum <= kChunk ? S.C.raw[k] : m[mi], sq)) vote(votesWords, mi);
    }
}

__global__ __launch_bounds__(kCta, 4) void vote_kernel(uint32_t* __restrict__ votesWords, const float* __restrict__ affine,
                                                    const float4* __restrict__ m, const uint32_t* __restrict__ bounds,
                                                    uint32_t cols, uint32_t rows, float threshold, bool tryOther)
{
    __shared__ CellSmem S;
    vote_cell(S, votesWords, affine, m, bounds, cols, rows, threshold, tryOther, blockIdx.x, blockIdx.y);
}

// ---------------------------------------------------------------------------
// Batched form (no reference counterpart: the reference bins each pair's
// matches on the host and runs one pair per call with a blocking sync,
// RansacMatchFilter.cpp:42-133). Per pair: device binning with the
// reference's rule and order, the two cell kernels over all pairs in one
// launch each, then the mask (votes >= minVotes) and an in-place stable
// compaction of the gathered pairs and matches with the kept count.
constexpr int kBinThreads = 1024;
constexpr int kBinWaves = kBinThreads / 64;
constexpr uint32_t kMaxCells = 1024;

__device__ inline uint32_t task_n(const BatchTask& T) { return min(*T.count, T.nHost); }

// cell of a point: the reference's ceil rule, clamped (RansacMatchFilter.cpp:47-52)
__device__ inline uint32_t cell_of(float x, float y, const BatchTask& T)
{
    const float cw = (float)T.cellWidth;
    const float fi = fminf(fmaxf(ceilf(y / cw), 0.f), (float)T.rows - 1.f);
    const float fj = fminf(fmaxf(ceilf(x / cw), 0.f), (float)T.cols - 1.f);
    return (uint32_t)fi * T.cols + (uint32_t)fj;
}

struct BinSmem {
    uint32_t cnt[kMaxCells];
    uint32_t cursor[kMaxCells];
    uint16_t waveCnt[kBinWaves][kMaxCells];
    uint32_t scan[kBinWaves];
};

// one workgroup per task: votes cleared, cell counts, bounds (exclusive
// prefix, cells in row-major order), then a stable scatter: points in index
// order, a point's slot = its cell's start + earlier points of the same cell
// (peer groups from ballots inside a wave, per-wave cell counts across the waves of a
// round of 1024 points, a running cursor across rounds); 64 tasks of about 4000
// points 39 -> 19 us with peer groups by the cell number's bits and the cell
// prefix by wave scans
template <class Src>
__global__ __launch_bounds__(kBinThreads) void bin_kernel(const Src batch)
{
    __shared__ BinSmem S;
    const BatchTask& T = batch[blockIdx.x];
    const uint32_t n = task_n(T);
    const uint32_t nCells = T.cols * T.rows;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (uint32_t w = tid; w < (T.nHost + 3) / 4; w += kBinThreads) reinterpret_cast<uint32_t*>(T.votes)[w] = 0;
    for (uint32_t c = tid; c < kMaxCells; c += kBinThreads) S.cnt[c] = 0;
    __syncthreads();
    for (uint32_t i = tid; i < n; i += kBinThreads) {
        const float4 p = T.pts[i];
        atomicAdd(&S.cnt[cell_of(p.x, p.y, T)], 1u);
    }
    __syncthreads();
    // exclusive prefix over the cells (nCells <= kMaxCells = kBinThreads)
    const uint32_t v = tid < nCells ? S.cnt[tid] : 0u;
    uint32_t inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)inc, o);
        if (lane >= (uint32_t)o) inc += y;
    }
    if (lane == 63) S.scan[wave] = inc;
    __syncthreads();
    for (uint32_t w = 0; w < wave; w++) inc += S.scan[w];
    if (tid < nCells) {
        const uint32_t start = inc - v;
        S.cursor[tid] = start;
        T.bounds[tid] = start;
    }
    if (tid == 0) T.bounds[nCells] = n;
    __syncthreads();
    for (uint32_t base = 0; base < n; base += kBinThreads) {
        const uint32_t i = base + tid;
        const bool valid = i < n;
        float4 p = make_float4(0.f, 0.f, 0.f, 0.f);
        uint32_t cell = ~0u;
        if (valid) {
            p = T.pts[i];
            cell = cell_of(p.x, p.y, T);
        }
        for (uint32_t c = lane; c < nCells; c += 64) S.waveCnt[wave][c] = 0;
        // lanes of this wave with the same cell: those that agree on every bit of
        // its number (one ballot a bit; one per distinct cell took up to 64)
        uint64_t peers = __ballot(valid);
        for (uint32_t k = 0; (1u << k) < nCells; k++) {
            const bool bit = (cell >> k) & 1u;
            const uint64_t set = __ballot(bit);
            peers &= bit ? set : ~set;
        }
        const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
        const uint32_t rank = (uint32_t)__popcll(peers & below);
        __syncthreads();  // waveCnt cleared by every wave
        if (valid && rank == 0) S.waveCnt[wave][cell] = (uint16_t)__popcll(peers);
        __syncthreads();
        if (valid) {
            uint32_t pos = S.cursor[cell] + rank;
            for (uint32_t w = 0; w < wave; w++) pos += S.waveCnt[w][cell];
            T.reordered[pos] = p;
            T.pos[i] = pos;
        }
        __syncthreads();
        for (uint32_t c = tid; c < nCells; c += kBinThreads) {
            uint32_t add = 0;
            for (uint32_t w = 0; w < kBinWaves; w++) add += S.waveCnt[w][c];
            S.cursor[c] += add;
        }
        __syncthreads();
    }
}

template <class Src>
__global__ __launch_bounds__(kCta, 4) void best_affine_batch_kernel(const Src batch, BatchParams prm)
{
    __shared__ CellSmem S;
    const BatchTask& T = batch[blockIdx.z];
    if (blockIdx.x >= T.cols || blockIdx.y >= T.rows || task_n(T) < 16) return;
    best_affine_cell(S, T.affine, T.reordered, T.bounds, T.cols, T.rows, prm.nbTests, T.threshold, T.seed, blockIdx.x,
                     blockIdx.y);
}

template <class Src>
__global__ __launch_bounds__(kCta, 4) void vote_batch_kernel(const Src batch, BatchParams prm)
{
    __shared__ CellSmem S;
    const BatchTask& T = batch[blockIdx.z];
    if (blockIdx.x >= T.cols || blockIdx.y >= T.rows || task_n(T) < 16) return;
    vote_cell(S, reinterpret_cast<uint32_t*>(T.votes), T.affine, T.reordered, T.bounds, T.cols, T.rows, T.threshold,
              prm.tryOther != 0, blockIdx.x, blockIdx.y);
}

// one workgroup per task: keep[i] = votes of point i >= minVotes; the kept
// points (and matches) move to the front in index order, in place (a round
// reads all of its 1024 entries before any is written, and writes only below
// the next round's first entry); the count becomes the kept count
template <class Src>
__global__ __launch_bounds__(kBinThreads) void compact_kernel(const Src batch, BatchParams prm)
{
    __shared__ uint32_t sWave[kBinWaves];
    __shared__ uint32_t sBase;
    const BatchTask& T = batch[blockIdx.x];
    const uint32_t n = task_n(T);
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) sBase = 0;
    __syncthreads();
    for (uint32_t base = 0; base < n; base += kBinThreads) {
        const uint32_t i = base + tid;
        bool keep = false;
        float4 p = make_float4(0.f, 0.f, 0.f, 0.f);
        rsfm_valid_match mv{};
        if (i < n) {
            keep = n >= 16 && T.votes[T.pos[i]] >= prm.minVotes;
            p = T.pts[i];
            if (T.matches) mv = T.matches[i];
            if (T.mask) T.mask[i] = keep ? 1 : 0;
        }
        const uint64_t b = __ballot(keep);
        const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
        if (lane == 0) sWave[wave] = (uint32_t)__popcll(b);
        __syncthreads();
        uint32_t off = sBase;
        for (uint32_t w = 0; w < wave; w++) off += sWave[w];
        if (keep) {
            const uint32_t o = off + (uint32_t)__popcll(b & below);
            T.pts[o] = p;
            if (T.matches) T.matches[o] = mv;
        }
        __syncthreads();
        if (tid == 0) {
            uint32_t t = 0;
            for (uint32_t w = 0; w < kBinWaves; w++) t += sWave[w];
            sBase += t;
        }
        __syncthreads();
    }
    if (T.mask)
        for (uint32_t i = n + tid; i < T.nHost; i += kBinThreads) T.mask[i] = 0;
    if (tid == 0) *T.count = sBase;
}

int launch_batch_table(const BatchTask* tasks, uint32_t nTasks, uint32_t maxCols, uint32_t maxRows, const BatchParams& p,
                       hipStream_t stream)
{
    if (nTasks == 0) return RSFM_OK;
    const InTable<BatchTask> src{tasks};
    bin_kernel<<<nTasks, kBinThreads, 0, stream>>>(src);
    RSFM_CHECK(check_launch("rmf bin table"));
    best_affine_batch_kernel<<<dim3(maxCols, maxRows, nTasks), kCta, 0, stream>>>(src, p);
    RSFM_CHECK(check_launch("rmf best affine table"));
    vote_batch_kernel<<<dim3(maxCols, maxRows, nTasks), kCta, 0, stream>>>(src, p);
    RSFM_CHECK(check_launch("rmf vote table"));
    compact_kernel<<<nTasks, kBinThreads, 0, stream>>>(src, p);
    return check_launch("rmf compact table");
}

size_t batch_workspace_bytes(uint32_t nPts, uint32_t nCells)
{
    return align_up((size_t)nPts * 16, 256) + align_up((size_t)nPts * 4, 256) + align_up(((size_t)nCells + 1) * 4, 256) +
           align_up((size_t)nCells * 24, 256) + align_up(((size_t)nPts + 3) / 4 * 4, 256);
}

void place_workspace(BatchTask& t, uint8_t*& ws)
{
    const uint32_t nCells = t.cols * t.rows;
    t.reordered = reinterpret_cast<float4*>(ws);
    ws += align_up((size_t)t.nHost * 16, 256);
    t.pos = reinterpret_cast<uint32_t*>(ws);
    ws += align_up((size_t)t.nHost * 4, 256);
    t.bounds = reinterpret_cast<uint32_t*>(ws);
    ws += align_up(((size_t)nCells + 1) * 4, 256);
    t.affine = reinterpret_cast<float*>(ws);
    ws += align_up((size_t)nCells * 24, 256);
    t.votes = ws;
    ws += align_up(((size_t)t.nHost + 3) / 4 * 4, 256);
}

int make_batch_task(const rsfm_rmf_task& t, uint32_t cellCols, float relativeThreshold, BatchTask& out)
{
    RSFM_RETURN_IF(t.imgWidth <= 0 || t.imgHeight <= 0, RSFM_ERR_INVALID, "rmf batch: bad image size");
    RSFM_RETURN_IF(t.nbPtsDev == nullptr, RSFM_ERR_INVALID, "rmf batch: nbPtsDev (device count) is required");
    RSFM_RETURN_IF(t.nbPts > 0 && t.pts == nullptr, RSFM_ERR_INVALID, "rmf batch: pts is null");
    RSFM_RETURN_IF(reinterpret_cast<uintptr_t>(t.pts) % 16, RSFM_ERR_INVALID, "rmf batch: pts must be 16-byte aligned");
    const uint32_t mx = (uint32_t)std::max(t.imgWidth, t.imgHeight);
    const uint32_t cw = div_up(mx, cellCols);
    const uint32_t cols = div_up((uint32_t)t.imgWidth, cw), rows = div_up((uint32_t)t.imgHeight, cw);
    RSFM_RETURN_IF(cols * rows > kMaxCells, RSFM_ERR_INVALID, "rmf batch: more than 1024 cells");
    out = BatchTask{};
    out.pts = reinterpret_cast<float4*>(t.pts);
    out.matches = t.matches;
    out.count = t.nbPtsDev;
    out.nHost = t.nbPts;
    out.mask = t.inlierMask;
    out.cols = cols;
    out.rows = rows;
    out.cellWidth = cw;
    out.threshold = (float)cw * relativeThreshold;
    out.seed = t.seed;
    return RSFM_OK;
}

__global__ void zero_words_kernel(uint32_t* p, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

}  // namespace rmf
}  // namespace rsfm_amd

using namespace rsfm_amd;

extern "C" int rsfm_rmf_filter(uint8_t* votes, float* affineScratch, const rsfm_pt_pair* matches, uint32_t nbMatches,
                               const uint32_t* bounds, uint32_t cols, uint32_t rows, uint32_t nbRansacTests,
                               float threshold, int tryOtherAffines, uint32_t seed, hipStream_t stream)
{
    RSFM_RETURN_IF(reinterpret_cast<uintptr_t>(votes) % 4, RSFM_ERR_INVALID, "rmf: votes must be 4-byte aligned");
    RSFM_RETURN_IF(nbMatches > 0 && (votes == nullptr || matches == nullptr || bounds == nullptr || affineScratch == nullptr),
                   RSFM_ERR_INVALID, "rmf: null pointer");
    RSFM_RETURN_IF(cols == 0 || rows == 0, RSFM_ERR_INVALID, "rmf: cols and rows must be >= 1");
    RSFM_RETURN_IF(reinterpret_cast<uintptr_t>(matches) % 16, RSFM_ERR_INVALID, "rmf: matches must be 16-byte aligned");
    if (nbMatches == 0) return RSFM_OK;
    const uint32_t words = div_up(nbMatches, 4);
    rmf::zero_words_kernel<<<div_up(words, 256), 256, 0, stream>>>(reinterpret_cast<uint32_t*>(votes), words);
    RSFM_CHECK(check_launch("rmf zero votes"));
    if (nbMatches < 16) return RSFM_OK;
    const dim3 grid(cols, rows);
    const float4* m = reinterpret_cast<const float4*>(matches);
    rmf::best_affine_kernel<<<grid, rmf::kCta, 0, stream>>>(affineScratch, m, bounds, cols, rows, nbRansacTests,
                                                            threshold, seed);
    RSFM_CHECK(check_launch("rmf best affine"));
    rmf::vote_kernel<<<grid, rmf::kCta, 0, stream>>>(reinterpret_cast<uint32_t*>(votes), affineScratch, m, bounds, cols,
                                                     rows, threshold, tryOtherAffines != 0);
    return check_launch("rmf vote");
}

// host binning of RansacMatchFilter::getInlierMask (RansacMatchFilter.cpp:42-67)
extern "C" int rsfm_rmf_bin_host(int imgWidth, int imgHeight, uint32_t cellCols, const rsfm_pt_pair* matches,
                                 uint32_t nbMatches, uint32_t* cols, uint32_t* rows, uint32_t* cellWidth,
                                 rsfm_pt_pair* reordered, uint32_t* bounds, uint32_t* order)
{
    RSFM_RETURN_IF(imgWidth <= 0 || imgHeight <= 0 || cellCols == 0, RSFM_ERR_INVALID, "rmf bin: bad image size");
    const uint32_t mx = (uint32_t)std::max(imgWidth, imgHeight);
    const uint32_t cw = div_up(mx, cellCols);
    const uint32_t c = div_up((uint32_t)imgWidth, cw), r = div_up((uint32_t)imgHeight, cw);
    const uint32_t nCells = c * r;
    RSFM_RETURN_IF(nbMatches > 0 && (matches == nullptr || cols == nullptr || rows == nullptr || cellWidth == nullptr ||
                                     reordered == nullptr || bounds == nullptr || order == nullptr),
                   RSFM_ERR_INVALID, "rmf bin: null argument");
    for (uint32_t k = 0; k < nbMatches; k++)
        RSFM_RETURN_IF(!std::isfinite(matches[k].x0) || !std::isfinite(matches[k].y0), RSFM_ERR_INVALID,
                       "rmf bin: non-finite keypoint coordinate at match " + std::to_string(k));
    std::vector<uint32_t> cell(nbMatches), cnt(nCells + 1, 0);
    for (uint32_t k = 0; k < nbMatches; k++) {
        const float fi = std::min(std::max(std::ceil(matches[k].y0 / (float)cw), 0.f), (float)r - 1.f);
        const float fj = std::min(std::max(std::ceil(matches[k].x0 / (float)cw), 0.f), (float)c - 1.f);
        cell[k] = (uint32_t)fi * c + (uint32_t)fj;
        cnt[cell[k] + 1]++;
    }
    for (uint32_t i = 0; i < nCells; i++) cnt[i + 1] += cnt[i];
    std::copy(cnt.begin(), cnt.end(), bounds);
    for (uint32_t k = 0; k < nbMatches; k++) {
        const uint32_t p = cnt[cell[k]]++;
        reordered[p] = matches[k];
        order[p] = k;
    }
    *cols = c;
    *rows = r;
    *cellWidth = cw;
    return RSFM_OK;
}

extern "C" int rsfm_rmf_filter_batch_workspace_size(const rsfm_rmf_task* tasks, size_t nbTasks, uint32_t cellCols,
                                                    size_t* bytes)
{
    RSFM_RETURN_IF(bytes == nullptr || (nbTasks > 0 && tasks == nullptr), RSFM_ERR_INVALID, "rmf batch: null argument");
    RSFM_RETURN_IF(cellCols == 0, RSFM_ERR_INVALID, "rmf batch: cellCols must be >= 1");
    size_t total = 0;
    for (size_t i = 0; i < nbTasks; i++) {
        rmf::BatchTask t;
        RSFM_CHECK(rmf::make_batch_task(tasks[i], cellCols, 1.f, t));
        total += rmf::batch_workspace_bytes(t.nHost, t.cols * t.rows);
    }
    *bytes = total;
    return RSFM_OK;
}

extern "C" int rsfm_rmf_filter_batch(const rsfm_rmf_task* tasks, size_t nbTasks, uint32_t cellCols,
                                     uint32_t nbRansacTests, float relativeThreshold, uint32_t minVotes,
                                     int tryOtherAffines, void* workspace, size_t workspaceBytes, hipStream_t stream)
{
    using namespace rmf;
    size_t need = 0;
    RSFM_CHECK(rsfm_rmf_filter_batch_workspace_size(tasks, nbTasks, cellCols, &need));
    RSFM_RETURN_IF(workspaceBytes < need, RSFM_ERR_INVALID,
                   "rmf batch: workspace too small (" + std::to_string(workspaceBytes) + " < " + std::to_string(need) + ")");
    RSFM_RETURN_IF(need > 0 && (workspace == nullptr || reinterpret_cast<uintptr_t>(workspace) % 256),
                   RSFM_ERR_INVALID, "rmf batch: workspace must be non-null and 256-byte aligned");
    RSFM_RETURN_IF(!(relativeThreshold > 0.f), RSFM_ERR_INVALID, "rmf batch: threshold must be > 0");
    const BatchParams prm{nbRansacTests, minVotes, tryOtherAffines};
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    constexpr size_t kMax = 32;
    for (size_t b = 0; b < nbTasks; b += kMax) {
        const size_t n = std::min(kMax, nbTasks - b);
        ByValue<BatchTask, kMax> batch{};
        uint32_t maxCols = 0, maxRows = 0;
        for (size_t i = 0; i < n; i++) {
            RSFM_CHECK(make_batch_task(tasks[b + i], cellCols, relativeThreshold, batch.t[i]));
            place_workspace(batch.t[i], ws);
            maxCols = std::max(maxCols, batch.t[i].cols);
            maxRows = std::max(maxRows, batch.t[i].rows);
        }
        bin_kernel<<<(uint32_t)n, kBinThreads, 0, stream>>>(batch);
        RSFM_CHECK(check_launch("rmf bin"));
        best_affine_batch_kernel<<<dim3(maxCols, maxRows, (uint32_t)n), kCta, 0, stream>>>(batch, prm);
        RSFM_CHECK(check_launch("rmf best affine batch"));
        vote_batch_kernel<<<dim3(maxCols, maxRows, (uint32_t)n), kCta, 0, stream>>>(batch, prm);
        RSFM_CHECK(check_launch("rmf vote batch"));
        compact_kernel<<<(uint32_t)n, kBinThreads, 0, stream>>>(batch, prm);
        RSFM_CHECK(check_launch("rmf compact"));
    }
    return RSFM_OK;
}
