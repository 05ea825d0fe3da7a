// ransac.hip - batched fundamental-matrix RANSAC hypothesis fitting and scoring.
//
// Reference path: ransac<F,8> (ransac.hpp:115-163) driving
// findEpipolarityRansacWithInsufficientTiePts<0> (ImagePair.cpp:148-204):
// per hypothesis the sample sanity gate (ImagePair.cpp:160-177), the 8-point
// fit (legacy/geometry.hpp:216-259) and the inlier count of
// checkEpipolarTransformation (legacy/geometry.cpp:55-86) over all points.
// Sample indices are an input (the reference draws them from a
// random_device-seeded engine), so a fixed index set gives one defined
// inlier count per hypothesis.
//
// GPU layout: a workgroup of four or eight wavefronts fits its hypotheses one
// per lane (fgeom::fit8) into LDS, then counts their inliers over all
// correspondences with the matrix-core screen of screen.hpp (fundamental
// matrices) or one lane per hypothesis (homographies, four wavefronts).
#include "internal.hpp"
#include "fgeom.hpp"
#include "hgeom.hpp"
#include "screen.hpp"
#include <algorithm>

namespace rsfm_amd {
namespace ransac {

constexpr int kThreads = 256;
constexpr int kMaxTasks = 32;

typedef ByValue<DevTask, kMaxTasks> Batch;

__device__ inline uint32_t task_n(const DevTask& T) { return T.nDev ? min(*T.nDev, T.nHost) : T.nHost; }

// Model kinds of the hypothesis kernels: 0 / 1 = fundamental matrix from 8
// points with the two-sided / Sampson test, 2 = homography from 4 points with
// checkProjectiveTransformation's test.
template <int kMode>
constexpr int sample_size() { return kMode == 2 ? 4 : 8; }

template <int kMode>
__device__ inline bool model_inlier(const float M[9], float4 p, float t2)
{
    if constexpr (kMode == 2) return hgeom::inlier_h(M, p, t2);
    else return fgeom::inlier<kMode>(M, p, t2);
}

// sanity gate of ImagePair.cpp:167-177 (and :366-374 for H): any two samples
// closer than the threshold in either image reject the hypothesis
template <int kN>
__device__ inline bool sane(const float4 p[kN], float s0, float s1)
{
    if (s0 <= 0.f && s1 <= 0.f) return true;
    bool ok = true;
#pragma unroll
    for (int i = 0; i < kN; i++)
#pragma unroll
        for (int j = 0; j < i; j++) {
            const float dx0 = p[i].x - p[j].x, dy0 = p[i].y - p[j].y;
            const float dx1 = p[i].z - p[j].z, dy1 = p[i].w - p[j].w;
            if (dx0 * dx0 + dy0 * dy0 < s0 || dx1 * dx1 + dy1 * dy1 < s1) ok = false;
        }
    return ok;
}

// fit of hypothesis h; false when out of range, insane or degenerate
template <int kMode>
__device__ inline bool fit_hypothesis(const DevTask& T, uint32_t n, uint32_t h, float s0, float s1, float M[9])
{
    constexpr int kN = sample_size<kMode>();
    if (h >= T.H || n < (uint32_t)kN) return false;
    float4 p[kN];
    bool inRange = true;
#pragma unroll
    for (int i = 0; i < kN; i++) {
        const uint32_t k = T.idx[(size_t)h * kN + i];
        inRange = inRange && k < n;
        p[i] = T.pts[k < n ? k : 0];
    }
    if (!inRange || !sane<kN>(p, s0, s1)) return false;
    if constexpr (kMode == 2) return fgeom::fit_h4(p, M);
    else return fgeom::fit8(p, M);
}

// Scoring: one lane per hypothesis; a workgroup holds 64 hypotheses and
// kScoreWaves wavefronts. Wavefront 0 fits the 64 models in registers and
// shares them through LDS; then each wavefront walks its own contiguous part
// of the correspondences in index order (all lanes read the same
// correspondence, so the loop body is VALU work only), and the partial counts
// are summed through LDS. Splitting the points keeps enough wavefronts per
// SIMD to hide load and dependency latency: one wavefront per 64 hypotheses
// gives only two per SIMD for 32 pairs of 4096 hypotheses.
constexpr int kScoreThreads = 64;
#ifndef RSFM_SCORE_WAVES
#define RSFM_SCORE_WAVES 4
#endif
constexpr int kScoreWaves = RSFM_SCORE_WAVES;
constexpr int kScoreBlock = kScoreThreads * kScoreWaves;

// points [beg, end) of wavefront w of `waves`: contiguous parts starting on multiples of 8
__device__ inline void wave_range(uint32_t n, uint32_t w, uint32_t waves, uint32_t& beg, uint32_t& end)
{
    const uint32_t part = ((n + waves - 1) / waves + 7u) & ~7u;
    beg = min(n, w * part);
    end = min(n, beg + part);
}

// number of inliers of model F among P[0, m): the next eight points are in
// flight while the current eight are tested
template <int kMode>
__device__ inline uint32_t count_inliers(const float F[9], const float4* __restrict__ P, uint32_t m, float t2)
{
    auto test4 = [&](const float4& a, const float4& b, const float4& c, const float4& d) -> uint32_t {
        return (model_inlier<kMode>(F, a, t2) ? 1u : 0u) + (model_inlier<kMode>(F, b, t2) ? 1u : 0u) +
               (model_inlier<kMode>(F, c, t2) ? 1u : 0u) + (model_inlier<kMode>(F, d, t2) ? 1u : 0u);
    };
    uint32_t cnt = 0, i = 0;
    if (m >= 8) {
        float4 c0 = P[0], c1 = P[1], c2 = P[2], c3 = P[3], c4 = P[4], c5 = P[5], c6 = P[6], c7 = P[7];
        for (; i + 16 <= m; i += 8) {
            const float4* __restrict__ Q = P + i + 8;  // one address per trip, immediate offsets
            const float4 n0 = Q[0], n1 = Q[1], n2 = Q[2], n3 = Q[3];
            const float4 n4 = Q[4], n5 = Q[5], n6 = Q[6], n7 = Q[7];
            cnt += test4(c0, c1, c2, c3) + test4(c4, c5, c6, c7);
            c0 = n0;
            c1 = n1;
            c2 = n2;
            c3 = n3;
            c4 = n4;
            c5 = n5;
            c6 = n6;
            c7 = n7;
        }
        cnt += test4(c0, c1, c2, c3) + test4(c4, c5, c6, c7);
        i += 8;
    }
    for (; i < m; i++) cnt += model_inlier<kMode>(F, P[i], t2) ? 1u : 0u;
    return cnt;
}

template <int kMode, class Src>
__global__ __launch_bounds__(kScoreBlock) void score_kernel(const Src batch, float t2, float s0, float s1)
{
    const Wg3 wg = xcd_local_block();  // all hypothesis blocks of a pair share one L2
    const DevTask& T = batch[wg.y];
    if (wg.x * kScoreThreads >= T.H) return;
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t h = wg.x * kScoreThreads + lane;
    const uint32_t n = task_n(T);
    __shared__ float sF[9][kScoreThreads];
    __shared__ uint32_t sOk[kScoreThreads];
    __shared__ uint32_t sCnt[kScoreWaves][kScoreThreads];
    float F[9];
    if (w == 0) {
        const bool ok = fit_hypothesis<kMode>(T, n, h, s0, s1, F);
#pragma unroll
        for (int q = 0; q < 9; q++) sF[q][lane] = ok ? F[q] : 0.f;
        sOk[lane] = ok ? 1u : 0u;
    }
    __syncthreads();
    const bool ok = sOk[lane] != 0;
#pragma unroll
    for (int q = 0; q < 9; q++) F[q] = sF[q][lane];
    uint32_t cnt = 0;
    if (ok) {
        uint32_t beg, end;
        wave_range(n, w, kScoreWaves, beg, end);
        // the offset is hidden from the uniformity analysis so the loads take
        // the vector memory path (in-order vmcnt, so the prefetch overlaps);
        // all 64 lanes read the same address, one cache line per wavefront
        uint32_t base = beg;
        asm volatile("" : "+v"(base));
        cnt = count_inliers<kMode>(F, T.pts + base, end - beg, t2);
    }
    sCnt[w][lane] = cnt;
    __syncthreads();
    if (w != 0 || h >= T.H) return;
    uint32_t total = 0;
#pragma unroll
    for (int k = 0; k < kScoreWaves; k++) total += sCnt[k][lane];
    T.counts[h] = ok ? total : 0u;
    if (T.models) {
#pragma unroll
        for (int q = 0; q < 9; q++) T.models[(size_t)h * 9 + q] = F[q];
    }
}

// Box of the pair's points for the screen, by the calling waves' nThreads
// threads (t of them): per-wave parts into S.part.
template <class Sm>
__device__ inline void box_scan(Sm& S, const float4* __restrict__ P, uint32_t n, uint32_t t, uint32_t nThreads)
{
    screen::BoxPart b;
    screen::box_init(b);
    uint32_t i = t;
    for (; i + 3 * nThreads < n; i += 4 * nThreads) {
        const float4 p0 = P[i], p1 = P[i + nThreads], p2 = P[i + 2 * nThreads], p3 = P[i + 3 * nThreads];
        screen::box_add(b, p0);
        screen::box_add(b, p1);
        screen::box_add(b, p2);
        screen::box_add(b, p3);
    }
    for (; i < n; i += nThreads) screen::box_add(b, P[i]);
    screen::box_wave_reduce(b);
    if ((threadIdx.x & 63) == 0) S.part[threadIdx.x >> 6] = b;
}

// the whole box from the parts of waves [first, kWaves)
template <class Sm>
__device__ inline screen::Box box_join(const Sm& S, uint32_t first, uint32_t n)
{
    screen::BoxPart b = S.part[first];
    for (uint32_t w = first + 1; w < Sm::kWaves; w++) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            b.lo[k] = fminf(b.lo[k], S.part[w].lo[k]);
            b.hi[k] = fmaxf(b.hi[k], S.part[w].hi[k]);
        }
        b.odd |= S.part[w].odd;
    }
    return screen::box_finish(b, n);
}

// Scoring of fundamental matrices: a workgroup of kWaves wavefronts (eight in
// the wide form, four in the narrow one, see launch_score) holds 64 kFit
// hypotheses, fitted one per lane by its first kFit wavefronts while the others
// scan the pair's box; then the wavefronts count the inliers of 16 kNB
// hypotheses each, kSplit of them sharing the points, with the matrix-core
// screen. Coordinates that the screen's bound does not cover (not finite, above
// 2^20, all equal) take the exact loop.

template <int kMode, int kWaves, int kFit, int kNB, class Src>
__global__ __launch_bounds__(64 * kWaves, 4) void score_screen_kernel(const Src batch, float t2, float s0, float s1)
{
    constexpr uint32_t kHyp = 64 * kFit;
    constexpr uint32_t kGroups = kHyp / (16 * kNB);       // waves with models of their own
    constexpr int kSplit = kWaves / kGroups;
    static_assert(kGroups * kSplit == kWaves && kFit < kWaves, "waves and hypotheses");
    const Wg3 wg = xcd_local_block();  // all hypothesis blocks of a pair share one L2
    const DevTask& T = batch[wg.y];
    if (wg.x * kHyp >= T.H) return;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const uint32_t n = task_n(T);
    __shared__ screen::Smem<kWaves, 2> S;
    __shared__ float sF[9][kHyp];
    __shared__ uint32_t sOk[kHyp], sCnt[kHyp];
    if (w < kFit) {
        float F[9];
        const bool ok = fit_hypothesis<kMode>(T, n, wg.x * kHyp + tid, s0, s1, F);
#pragma unroll
        for (int q = 0; q < 9; q++) sF[q][tid] = ok ? F[q] : 0.f;
        sOk[tid] = ok ? 1u : 0u;
        sCnt[tid] = 0u;
    }
    else box_scan(S, T.pts, n, tid - kHyp, 64 * kWaves - kHyp);
    __syncthreads();
    if (n >= (uint32_t)sample_size<kMode>()) {
        const screen::Box box = box_join(S, kFit, n);
        auto model = [&](uint32_t k, float F[9]) {
#pragma unroll
            for (int q = 0; q < 9; q++) F[q] = sF[q][k];
            return sOk[k] != 0;
        };
        if (!box.odd) {
            screen::v8h be[kNB], bq[kMode == 1 ? 1 : 2][kNB];
            float d2[kNB], cc[kNB];
            const uint32_t base = (w % kGroups) * 16 * kNB;
            screen::load_models<kMode, kNB>(S, box, base, 16 * kNB, t2, model, be, bq, d2, cc);
            screen::count_points<kMode, kNB, kSplit>(S, box, T.pts, n, t2, base, w / kGroups, be, bq, d2, cc, sCnt, model);
        } else {
            uint32_t beg, end;
            wave_range(n, w, kWaves, beg, end);
            for (uint32_t g = 0; g < (uint32_t)kFit; g++) {
                float F[9];
                if (!model(g * 64 + lane, F)) continue;
                const uint32_t c = count_inliers<kMode>(F, T.pts + beg, end - beg, t2);
                if (c) atomicAdd(&sCnt[g * 64 + lane], c);
            }
        }
    }
    __syncthreads();
    const uint32_t h = wg.x * kHyp + tid;
    if (tid >= kHyp || h >= T.H) return;
    T.counts[h] = sOk[tid] ? sCnt[tid] : 0u;
    if (T.models) {
#pragma unroll
        for (int q = 0; q < 9; q++) T.models[(size_t)h * 9 + q] = sF[q][tid];
    }
}

// best hypothesis (largest count, lowest index among equals) and its inlier
// mask: 16 wavefronts per task, the maximum key through wave shuffles and one
// LDS round, the mask four points per thread and trip with the loads first
constexpr int kBestThreads = 1024;

template <int kMode, class Src>
__global__ __launch_bounds__(kBestThreads) void best_kernel(const Src batch, float t2, float s0, float s1)
{
    const DevTask& T = batch[blockIdx.x];
    const uint32_t n = task_n(T);
    constexpr int kWaves = kBestThreads / 64;
    __shared__ uint64_t sKey[kWaves];
    __shared__ float sF[9];
    __shared__ uint32_t sOk;
    const uint32_t tid = threadIdx.x;
    uint64_t key = 0;  // (count << 32) | ~h : max count, then lowest h
    for (uint32_t h = tid; h < T.H; h += kBestThreads) {
        const uint64_t k = ((uint64_t)T.counts[h] << 32) | (uint32_t)~h;
        key = k > key ? k : key;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint64_t k = __shfl_xor(key, o);
        key = k > key ? k : key;
    }
    if ((tid & 63) == 0) sKey[tid >> 6] = key;
    __syncthreads();
    if (tid == 0) {
        uint64_t bk = 0;
        for (int w = 0; w < kWaves; w++) bk = sKey[w] > bk ? sKey[w] : bk;
        const uint32_t bestH = T.H ? ~(uint32_t)bk : 0u;
        const uint32_t bestC = (uint32_t)(bk >> 32);
        float F[9];
        bool ok = T.H > 0 && bestC > 0;
        if (T.models != nullptr) {
            // the scorer stored every model; a nonzero count means its fit succeeded
            if (ok)
                for (int q = 0; q < 9; q++) F[q] = T.models[(size_t)bestH * 9 + q];
        } else {
            ok = ok && fit_hypothesis<kMode>(T, n, bestH, s0, s1, F);
        }
        for (int q = 0; q < 9; q++) sF[q] = ok ? F[q] : 0.f;
        sOk = ok;
        if (T.best) {
            T.best[0] = T.H ? bestH : ~0u;
            T.best[1] = bestC;
        }
    }
    __syncthreads();
    if (!T.mask) return;
    float F[9];
    for (int q = 0; q < 9; q++) F[q] = sF[q];
    const bool ok = sOk != 0;
    for (uint32_t i0 = tid; i0 < T.nHost; i0 += 4 * kBestThreads) {
        float4 p[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint32_t i = i0 + u * kBestThreads;
            if (ok && i < n) p[u] = T.pts[i];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint32_t i = i0 + u * kBestThreads;
            if (i < T.nHost) T.mask[i] = (ok && i < n) ? (uint8_t)model_inlier<kMode>(F, p[u], t2) : 0;
        }
    }
}

// ---------------------------------------------------------------------------
// 7-point hypotheses (the sampling model of findEpipolarityDegensac,
// degensac.cpp:113-150): each sample of 7 indices gives up to three F
// (fgeom::fit7); a hypothesis scores as its best model (most inliers, first
// on ties), which is also the model reported for it.
constexpr int kMaxF7 = 3;

__device__ inline bool sane7(const float4 p[7], float s0, float s1)
{
    if (s0 <= 0.f && s1 <= 0.f) return true;
    bool ok = true;
#pragma unroll
    for (int i = 0; i < 7; i++)
#pragma unroll
        for (int j = 0; j < i; j++) {
            const float dx0 = p[i].x - p[j].x, dy0 = p[i].y - p[j].y;
            const float dx1 = p[i].z - p[j].z, dy1 = p[i].w - p[j].w;
            if (dx0 * dx0 + dy0 * dy0 < s0 || dx1 * dx1 + dy1 * dy1 < s1) ok = false;
        }
    return ok;
}

// the seven points of sample h, false if it is to be rejected
__device__ inline bool load_sample7(const DevTask& T, uint32_t n, uint32_t h, float s0, float s1, float4 p[7])
{
    if (h >= T.H || n < 7) return false;
    bool inRange = true;
#pragma unroll
    for (int i = 0; i < 7; i++) {
        const uint32_t k = T.idx[(size_t)h * 7 + i];
        inRange = inRange && k < n;
        p[i] = T.pts[k < n ? k : 0];
    }
    return inRange && sane7(p, s0, s1);
}

// 7-point scoring. A workgroup takes kS7Samples samples, one per lane of its
// first two wavefronts: every such lane reduces its sample to a cubic while the
// others scan the pair's box; the cubic's one or three root intervals are
// bisected in FP64 by the other six wavefronts, an interval a lane (chains of up
// to 80 dependent steps; one after the other on the sample's own lane they took
// 30 us more); the sample's lane makes the models of the roots, up to three, and
// the workgroup's M models are listed in LDS in sample order (a scan of the model
// counts). Wavefront w then counts the inliers of models 16 R w .. (R = ceil(M /
// 128), at most three blocks of 16) over all points with the matrix-core screen. A
// sample with one real root thus takes one model slot instead of three (about 2.5
// models per sample with 8K-keypoint pairs). Each sample then reports its best
// model (most inliers, the first on ties) and that count. 32 pairs x 4096 samples
// x 1400 points on average, two-sided test: 468 -> 288 us with the screen instead
// of the exact test on every point, -> 259 with the bisections spread.
constexpr uint32_t kS7Samples = 128;
constexpr int kS7Waves = 8, kS7Block = 64 * kS7Waves;
constexpr uint32_t kS7MaxModels = kS7Samples * kMaxF7;
static_assert(kS7Samples % 64 == 0 && kS7Block == (1 + kMaxF7) * kS7Samples, "a lane per sample and per interval");

// the wave's 16 R models (base, count of them) over all points
template <int kMode, int R, class Sm, class Model>
__device__ inline void count7(Sm& S, const screen::Box& box, const float4* __restrict__ P, uint32_t n, float t2,
                              uint32_t base, uint32_t count, uint32_t* cnt, Model model)
{
    screen::v8h be[R], bq[kMode == 1 ? 1 : 2][R];
    float d2[R], cc[R];
    screen::load_models<kMode, R>(S, box, base, count, t2, model, be, bq, d2, cc);
    screen::count_points<kMode, R, 1>(S, box, P, n, t2, base, 0, be, bq, d2, cc, cnt, model);
}

template <int kMode, class Src>
__global__ __launch_bounds__(kS7Block, 4) void score7_kernel(const Src batch, float t2, float s0, float s1)
{
    const Wg3 wg = xcd_local_block();
    const DevTask& T = batch[wg.y];
    if (wg.x * kS7Samples >= T.H) return;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const uint32_t h = wg.x * kS7Samples + tid;
    const uint32_t n = task_n(T);
    __shared__ screen::Smem<kS7Waves, 1> S;  // two workgroups per CU
    // the cubics and their roots, then the models
    union Fit {
        struct {
            double a[4][kS7Samples], e[4][kS7Samples], root[kMaxF7][kS7Samples];
            uint8_t intervals[kS7Samples], has[kMaxF7][kS7Samples];
        } s;
        float F[9][kS7MaxModels];
    };
    __shared__ Fit fit;
    float (&sF)[9][kS7MaxModels] = fit.F;
    __shared__ uint32_t sCnt[kS7MaxModels];
    __shared__ uint32_t sWaveModels[kS7Samples / 64];
    for (uint32_t k = tid; k < kS7MaxModels; k += kS7Block) sCnt[k] = 0u;
    fgeom::Basis7 basis;
    int ni = 0;
    if (tid < kS7Samples) {
        float4 p[7];
        double a[4], e[4];
        if (load_sample7(T, n, h, s0, s1, p) && fgeom::fit7_cubic(p, basis, a)) {
            ni = fgeom::cubic_intervals(a, e);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                fit.s.a[k][tid] = a[k];
                fit.s.e[k][tid] = e[k];
            }
        }
        fit.s.intervals[tid] = (uint8_t)ni;
    } else {
        box_scan(S, T.pts, n, tid - kS7Samples, kS7Block - kS7Samples);
    }
    __syncthreads();
    if (tid >= kS7Samples) {
        const uint32_t i = tid / kS7Samples - 1, s = tid % kS7Samples;
        if (i < fit.s.intervals[s]) {
            double a[4], x = 0.0;
#pragma unroll
            for (int k = 0; k < 4; k++) a[k] = fit.s.a[k][s];
            fit.s.has[i][s] = fgeom::interval_root(a, fit.s.e[i][s], fit.s.e[i + 1][s], x);
            fit.s.root[i][s] = x;
        }
    }
    __syncthreads();
    float Fw[kMaxF7][9];  // written with a running index
    int nm = 0;
    if (ni > 0) {
        double roots[kMaxF7];
        int nr = 0;
        for (int i = 0; i < ni; i++)
            if (fit.s.has[i][tid]) fgeom::append_root(roots, nr, fit.s.root[i][tid]);
        nm = fgeom::fit7_models(basis, roots, nr, Fw);
    }
    // the models' place in the list: prefix of nm in lane order (the lanes
    // past the samples add nothing)
    uint32_t inc = (uint32_t)nm;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)inc, o);
        if (lane >= (uint32_t)o) inc += y;
    }
    if (lane == 63 && w < kS7Samples / 64) sWaveModels[w] = inc;
    __syncthreads();
    uint32_t off = inc - (uint32_t)nm;
#pragma unroll
    for (uint32_t k = 0; k < kS7Samples / 64; k++) off += k < w ? sWaveModels[k] : 0u;
#pragma unroll
    for (int mi = 0; mi < kMaxF7; mi++)
        if (mi < nm)
#pragma unroll
            for (int q = 0; q < 9; q++) sF[q][off + mi] = Fw[mi][q];
    __syncthreads();
    uint32_t M = 0;
#pragma unroll
    for (uint32_t k = 0; k < kS7Samples / 64; k++) M += sWaveModels[k];
    const uint32_t R = (M + 16 * (uint32_t)kS7Waves - 1) / (16 * (uint32_t)kS7Waves);
    if (R > 0) {
        const screen::Box box = box_join(S, kS7Samples / 64, n);
        auto model = [&](uint32_t k, float F[9]) {
#pragma unroll
            for (int q = 0; q < 9; q++) F[q] = sF[q][k];
            return true;
        };
        if (!box.odd) {
            const uint32_t base = w * 16 * R, count = M > base ? min(M - base, 16 * R) : 0u;
            switch (R) {
                case 1: count7<kMode, 1>(S, box, T.pts, n, t2, base, count, sCnt, model); break;
                case 2: count7<kMode, 2>(S, box, T.pts, n, t2, base, count, sCnt, model); break;
                default: count7<kMode, 3>(S, box, T.pts, n, t2, base, count, sCnt, model); break;
            }
        } else {
            uint32_t beg, end;
            wave_range(n, w, (uint32_t)kS7Waves, beg, end);
            for (uint32_t k = lane; k < M; k += 64) {
                float F[9];
                model(k, F);
                const uint32_t c = count_inliers<kMode>(F, T.pts + beg, end - beg, t2);
                if (c) atomicAdd(&sCnt[k], c);
            }
        }
    }
    __syncthreads();
    if (tid >= kS7Samples || h >= T.H) return;
    uint32_t best = 0;
    int bm = 0;
    for (int mi = 0; mi < nm; mi++) {
        const uint32_t cm = sCnt[off + mi];
        if (mi == 0 || cm > best) {
            best = cm;
            bm = mi;
        }
    }
    T.counts[h] = nm ? best : 0u;
    if (T.models) {
#pragma unroll
        for (int q = 0; q < 9; q++) T.models[(size_t)h * 9 + q] = nm ? sF[q][off + bm] : 0.f;
    }
}

// best 7-point hypothesis (largest count, lowest index), and the mask of its best
// model where one is asked for. The model is read if the scorer stored it; else
// it is solved again and the sample's models recounted, which a caller that takes
// no mask does not pay (32 pairs x 4096 samples: 50 -> 7 us).
template <int kMode, class Src>
__global__ __launch_bounds__(kThreads) void best7_kernel(const Src batch, float t2, float s0, float s1)
{
    const DevTask& T = batch[blockIdx.x];
    const uint32_t n = task_n(T);
    __shared__ uint64_t sKey[kThreads];
    __shared__ uint32_t sRed[kMaxF7][kThreads];
    __shared__ float sFs[kMaxF7][9];
    __shared__ int sNm;
    uint64_t key = 0;
    for (uint32_t h = threadIdx.x; h < T.H; h += kThreads) {
        const uint64_t k = ((uint64_t)T.counts[h] << 32) | (uint32_t)~h;
        key = k > key ? k : key;
    }
    sKey[threadIdx.x] = key;
    __syncthreads();
    for (int s = kThreads / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) sKey[threadIdx.x] = max(sKey[threadIdx.x], sKey[threadIdx.x + s]);
        __syncthreads();
    }
    const uint64_t bk = sKey[0];
    const uint32_t bestH = T.H ? ~(uint32_t)bk : 0u;
    const uint32_t bestC = (uint32_t)(bk >> 32);
    if (threadIdx.x == 0 && T.best) {
        T.best[0] = T.H ? bestH : ~0u;
        T.best[1] = bestC;
    }
    if (!T.mask) return;
    const bool found = T.H > 0 && bestC > 0;
    if (threadIdx.x == 0) {
        float Fs[kMaxF7][9];
        float4 p[7];
        int nm = 0;
        if (found && T.models) {
            for (int q = 0; q < 9; q++) Fs[0][q] = T.models[(size_t)bestH * 9 + q];
            nm = 1;
        } else if (found && load_sample7(T, n, bestH, s0, s1, p)) {
            nm = fgeom::fit7(p, Fs);
        }
        for (int m = 0; m < kMaxF7; m++)
            for (int q = 0; q < 9; q++) sFs[m][q] = m < nm ? Fs[m][q] : 0.f;
        sNm = nm;
    }
    __syncthreads();
    const int nm = sNm;
    int bm = 0;
    if (nm > 1) {
        // counts of the two or three models of the best sample
        uint32_t c[kMaxF7] = {0, 0, 0};
        for (uint32_t i = threadIdx.x; i < n; i += kThreads) {
            const float4 p = T.pts[i];
            for (int m = 0; m < nm; m++) c[m] += fgeom::inlier<kMode>(sFs[m], p, t2) ? 1u : 0u;
        }
        for (int m = 0; m < kMaxF7; m++) sRed[m][threadIdx.x] = c[m];
        __syncthreads();
        for (int s = kThreads / 2; s > 0; s >>= 1) {
            if (threadIdx.x < s)
                for (int m = 0; m < kMaxF7; m++) sRed[m][threadIdx.x] += sRed[m][threadIdx.x + s];
            __syncthreads();
        }
        for (int m = 1; m < nm; m++)
            if (sRed[m][0] > sRed[bm][0]) bm = m;
    }
    float F[9];
    for (int q = 0; q < 9; q++) F[q] = sFs[bm][q];
    for (uint32_t i = threadIdx.x; i < T.nHost; i += kThreads)
        T.mask[i] = (nm > 0 && i < n) ? (uint8_t)fgeom::inlier<kMode>(F, T.pts[i], t2) : 0;
}

// ---------------------------------------------------------------------------
// device sampler: hypothesis h of stream `seed` draws 8 distinct indices in
// [0, n) from a splitmix64 sequence seeded by (seed, h), rejecting repeats
__device__ inline uint64_t splitmix(uint64_t& s)
{
    s += 0x9E3779B97F4A7C15ull;
    uint64_t z = s;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

constexpr int kSampleMaxTasks = 32;
typedef ByValue<SampleTask, kSampleMaxTasks> SampleBatch;

__global__ void sample_kernel(uint32_t* idx, uint32_t H, uint32_t nHost, const uint32_t* nDev, uint64_t seed);

template <class Src>
__global__ void sample_batch_kernel(const Src batch)
{
    const SampleTask& T = batch[blockIdx.y];
    if (blockIdx.x * blockDim.x >= T.H) return;
    // same draw as sample_kernel, task taken from the batch
    const uint32_t h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= T.H) return;
    const uint32_t n = T.nDev ? min(*T.nDev, T.nHost) : T.nHost;
    const uint32_t k = T.k;
    uint32_t* out = T.idx + (size_t)h * k;
    if (n < k) {
        for (uint32_t i = 0; i < k; i++) out[i] = ~0u;
        return;
    }
    uint64_t s = T.seed ^ ((uint64_t)h * 0xD1B54A32D192ED03ull);
    uint32_t v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        v[i] = ~0u;
        if ((uint32_t)i >= k) continue;
        for (;;) {
            const uint32_t c = (uint32_t)(splitmix(s) % n);
            bool dup = false;
#pragma unroll
            for (int j = 0; j < i; j++) dup |= v[j] == c;
            if (!dup) {
                v[i] = c;
                break;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 8; i++)
        if ((uint32_t)i < k) out[i] = v[i];
}

// ---- weighted sampler for learned proposals (no reference counterpart; the
// reference draws uniformly, ransac.hpp:23-82). Weights become integers
// q_i = round(clamp(w_i, 0, 1) * 65536) with an exact u64 inclusive prefix, so
// the draw is reproducible bit for bit on the CPU. Hypothesis h uses the same
// splitmix64 stream as the uniform sampler: r = next % total selects the first
// i with cdf[i] > r (probability q_i / total); repeats are rejected (draws
// without replacement), at most kMaxWeightedDraws draws per hypothesis, after
// which it is marked ~0u. total == 0 falls back to the uniform draw.
constexpr uint32_t kMaxWeightedDraws = 512;

struct WSampleTask {
    uint32_t* idx;
    uint32_t H;
    uint32_t nHost;
    const uint32_t* nDev;
    const float* w;
    uint64_t* cdf;
    uint64_t seed;
};
struct WSampleBatch {
    WSampleTask t[kSampleMaxTasks];
};

__device__ inline uint32_t quant_weight(float w) { return (uint32_t)(fminf(fmaxf(w, 0.f), 1.f) * 65536.f + 0.5f); }

// one 1024-thread workgroup per task: cdf[i] = sum_{k <= i} q_k
__global__ __launch_bounds__(1024) void weight_scan_kernel(const WSampleBatch batch)
{
    const WSampleTask& T = batch.t[blockIdx.x];
    const uint32_t n = T.nDev ? min(*T.nDev, T.nHost) : T.nHost;
    __shared__ uint64_t sWave[16];
    __shared__ uint64_t sCarry;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) sCarry = 0;
    __syncthreads();
    for (uint32_t base = 0; base < n; base += 4096) {
        // each thread owns 4 consecutive entries
        const uint32_t i0 = base + 4 * tid;
        uint64_t q[4];
#pragma unroll
        for (int k = 0; k < 4; k++) q[k] = i0 + k < n ? quant_weight(T.w[i0 + k]) : 0;
        q[1] += q[0];
        q[2] += q[1];
        q[3] += q[2];
        // inclusive scan of the thread totals across the wave
        uint64_t x = q[3];
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint64_t y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        if (lane == 63) sWave[wave] = x;
        __syncthreads();
        uint64_t waveOff = 0;
        for (int w = 0; w < wave; w++) waveOff += sWave[w];
        const uint64_t off = sCarry + waveOff + x - q[3];
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (i0 + k < n) T.cdf[i0 + k] = off + q[k];
        __syncthreads();
        if (tid == 1023) sCarry = off + q[3];
        __syncthreads();
    }
}

// x mod d with m = (2^64 - 1) / d: the product's high word is the quotient or one
// less, since m >= 2^64 / d - 1 and x < 2^64
__device__ inline uint64_t mod_by(uint64_t x, uint64_t d, uint64_t m)
{
    const uint64_t r = x - __umul64hi(x, m) * d;
    return r >= d ? r - d : r;
}

constexpr uint32_t kTable = 2048;  // entries of the LDS table, 16 KB

// Steps of kDraws binary searches side by side for the first i with at[i] > r[k] in
// lo[k] .. hi[k], which holds one. A search that has ended (lo = hi) stays where it is.
template <int kDraws, class Array>
__device__ __forceinline__ void search_steps(const Array& at, uint32_t steps, const uint64_t (&r)[kDraws],
                                             uint32_t (&lo)[kDraws], uint32_t (&hi)[kDraws])
{
    for (; steps > 0; steps--)
#pragma unroll
        for (int k = 0; k < kDraws; k++) {
            const uint32_t mid = lo[k] + ((hi[k] - lo[k]) >> 1);
            if (at[mid] > r[k]) hi[k] = mid;
            else lo[k] = mid + 1;
        }
}

// c[k] = first i with cdf[i] > r[k], every r[k] < cdf[n - 1]: among the last entries of the
// 2^shift long blocks (table, nb of them), then in the block
template <int kDraws>
__device__ __forceinline__ void find_draws(const uint64_t (&table)[kTable], uint32_t nb, uint32_t shift,
                                           const uint64_t* __restrict__ cdf, uint32_t n, const uint64_t (&r)[kDraws],
                                           uint32_t (&c)[kDraws])
{
    uint32_t hi[kDraws];
#pragma unroll
    for (int k = 0; k < kDraws; k++) {
        c[k] = 0;
        hi[k] = nb - 1;
    }
    search_steps<kDraws>(table, 32 - __clz((int)(nb - 1)), r, c, hi);
    if (shift == 0) return;
#pragma unroll
    for (int k = 0; k < kDraws; k++) {
        c[k] <<= shift;
        hi[k] = c[k] + min(n - 1 - c[k], (1u << shift) - 1u);
    }
    search_steps<kDraws>(cdf, shift, r, c, hi);
}

// One hypothesis a lane. A draw is a chain of log2 n dependent loads, each of 64
// addresses apart: the prefix sums, thinned to kTable entries, are searched in LDS, the
// first eight draws side by side, and only repeats are drawn again one at a time; the
// remainder of a draw takes a multiplication instead of a 64-bit division. 12 tasks x 4096
// hypotheses over 2400 weights: 24 us with each draw after the other in global memory, 21
// side by side there, 14 so.
constexpr int kWSampleThreads = 256;
__global__ __launch_bounds__(kWSampleThreads) void weighted_sample_kernel(const WSampleBatch batch)
{
    const WSampleTask& T = batch.t[blockIdx.y];
    if (blockIdx.x * kWSampleThreads >= T.H) return;
    const uint32_t h = blockIdx.x * kWSampleThreads + threadIdx.x;
    const uint32_t n = T.nDev ? min(*T.nDev, T.nHost) : T.nHost;
    uint32_t* out = T.idx + (size_t)h * 8;
    if (n < 8) {
        if (h < T.H)
            for (int i = 0; i < 8; i++) out[i] = ~0u;
        return;
    }
    __shared__ uint64_t table[kTable];
    uint32_t shift = 0;
    while (((n - 1) >> shift) >= kTable) shift++;
    const uint32_t nb = ((n - 1) >> shift) + 1;
    for (uint32_t i = threadIdx.x; i < nb; i += kWSampleThreads) table[i] = T.cdf[i + 1 < nb ? ((i + 1) << shift) - 1 : n - 1];
    __syncthreads();
    if (h >= T.H) return;
    const uint64_t total = table[nb - 1], d = total ? total : n, m = ~0ull / d;
    uint64_t s = T.seed ^ ((uint64_t)h * 0xD1B54A32D192ED03ull);
    uint32_t v[8], count = 0, draws = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = ~0u;  // no index
    auto accept = [&](uint32_t c) {
        bool dup = false;
#pragma unroll
        for (int j = 0; j < 8; j++) dup |= v[j] == c;
        if (dup) {
            draws++;
            return;
        }
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = (uint32_t)j == count ? c : v[j];
        count++;
    };
    {
        uint64_t r[8];
        uint32_t c[8];
#pragma unroll
        for (int k = 0; k < 8; k++) r[k] = mod_by(splitmix(s), d, m);
        if (total) find_draws<8>(table, nb, shift, T.cdf, n, r, c);
#pragma unroll
        for (int k = 0; k < 8; k++) accept(total ? c[k] : (uint32_t)r[k]);
    }
    while (count < 8) {
        if (draws >= kMaxWeightedDraws) {
            for (int k = 0; k < 8; k++) out[k] = ~0u;
            return;
        }
        const uint64_t r[1] = {mod_by(splitmix(s), d, m)};
        uint32_t c[1];
        if (total) find_draws<1>(table, nb, shift, T.cdf, n, r, c);
        accept(total ? c[0] : (uint32_t)r[0]);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) out[i] = v[i];
}

__global__ void sample_kernel(uint32_t* idx, uint32_t H, uint32_t nHost, const uint32_t* nDev, uint64_t seed)
{
    const uint32_t h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= H) return;
    const uint32_t n = nDev ? min(*nDev, nHost) : nHost;
    uint32_t* out = idx + (size_t)h * 8;
    if (n < 8) {
        for (int i = 0; i < 8; i++) out[i] = ~0u;
        return;
    }
    uint64_t s = seed ^ ((uint64_t)h * 0xD1B54A32D192ED03ull);
    uint32_t v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        for (;;) {
            const uint32_t c = (uint32_t)(splitmix(s) % n);
            bool dup = false;
#pragma unroll
            for (int j = 0; j < i; j++) dup |= v[j] == c;
            if (!dup) {
                v[i] = c;
                break;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 8; i++) out[i] = v[i];
}

int launch_sample_table(const SampleTask* tasks, uint32_t nTasks, uint32_t maxH, hipStream_t stream)
{
    if (nTasks == 0 || maxH == 0) return RSFM_OK;
    sample_batch_kernel<<<dim3(div_up(maxH, 256), nTasks), 256, 0, stream>>>(InTable<SampleTask>{tasks});
    return check_launch("sample table");
}

// Scores of nTasks tasks of at most maxH hypotheses; kind = model kind. A
// 256-hypothesis workgroup stages each point for four times the models of a
// 64-hypothesis one, which in turn keeps more workgroups in flight: at 12
// pairs x 4096 hypotheses x 1300-2400 points (192 or 768 workgroups) the wide
// form takes 53 us and the narrow one 58 us, at one pair (16 or 64) only the
// narrow one spreads the fits. 32 pairs x 4096 x 2454 points: 208 -> 98 us
// against one exact test per lane and trip (VALU issue 93% busy; 46.6 M vector
// instructions instead of 110 M), 64 pairs of the affine-filtered batch 218 ->
// 139 us.
constexpr uint32_t kWideMin = 128;
template <class Src>
static int launch_score(const Src& src, uint32_t nTasks, uint32_t maxH, float t2, int kind, float s0, float s1,
                        hipStream_t stream, const char* name)
{
    if (kind == 2) {
        score_kernel<2><<<dim3(div_up(maxH, kScoreThreads), nTasks), kScoreBlock, 0, stream>>>(src, t2, s0, s1);
    } else if (div_up(maxH, 256) * nTasks >= kWideMin) {
        const dim3 grid(div_up(maxH, 256), nTasks);
        if (kind == 0) score_screen_kernel<0, 8, 4, 2><<<grid, 512, 0, stream>>>(src, t2, s0, s1);
        else score_screen_kernel<1, 8, 4, 4><<<grid, 512, 0, stream>>>(src, t2, s0, s1);
    } else {
        const dim3 grid(div_up(maxH, 64), nTasks);
        if (kind == 0) score_screen_kernel<0, 4, 1, 1><<<grid, 256, 0, stream>>>(src, t2, s0, s1);
        else score_screen_kernel<1, 4, 1, 1><<<grid, 256, 0, stream>>>(src, t2, s0, s1);
    }
    return check_launch(name);
}

int launch_score_table(const DevTask* tasks, uint32_t nTasks, uint32_t maxH, float threshold, int mode,
                       float minSepSq0, float minSepSq1, hipStream_t stream, bool withBest)
{
    RSFM_RETURN_IF(mode != 0 && mode != 1, RSFM_ERR_INVALID, "ransac: mode must be 0 or 1");
    if (nTasks == 0) return RSFM_OK;
    const float t2 = threshold * threshold;
    const InTable<DevTask> src{tasks};
    if (maxH > 0) RSFM_CHECK(launch_score(src, nTasks, maxH, t2, mode, minSepSq0, minSepSq1, stream, "ransac score table"));
    if (!withBest) return RSFM_OK;
    if (mode == 0) best_kernel<0><<<nTasks, kBestThreads, 0, stream>>>(src, t2, minSepSq0, minSepSq1);
    else best_kernel<1><<<nTasks, kBestThreads, 0, stream>>>(src, t2, minSepSq0, minSepSq1);
    return check_launch("ransac best table");
}

int launch_score7_table(const DevTask* tasks, uint32_t nTasks, uint32_t maxH, float threshold, int mode,
                        float minSepSq0, float minSepSq1, hipStream_t stream)
{
    RSFM_RETURN_IF(mode != 0 && mode != 1, RSFM_ERR_INVALID, "ransac7: mode must be 0 or 1");
    if (nTasks == 0) return RSFM_OK;
    const float t2 = threshold * threshold;
    const InTable<DevTask> src{tasks};
    if (maxH > 0) {
        const dim3 grid(div_up(maxH, kS7Samples), nTasks);
        if (mode == 0) score7_kernel<0><<<grid, kS7Block, 0, stream>>>(src, t2, minSepSq0, minSepSq1);
        else score7_kernel<1><<<grid, kS7Block, 0, stream>>>(src, t2, minSepSq0, minSepSq1);
        RSFM_CHECK(check_launch("ransac7 score table"));
    }
    if (mode == 0) best7_kernel<0><<<nTasks, kThreads, 0, stream>>>(src, t2, minSepSq0, minSepSq1);
    else best7_kernel<1><<<nTasks, kThreads, 0, stream>>>(src, t2, minSepSq0, minSepSq1);
    return check_launch("ransac7 best table");
}

}  // namespace ransac
}  // namespace rsfm_amd

using namespace rsfm_amd;

namespace rsfm_amd {
namespace ransac {
// score + best over batches of at most kMaxTasks tasks; kind = model kind
// (0 / 1 fundamental matrix, 2 homography)
static int run_hypotheses(const rsfm_ransac_task* tasks, size_t nbTasks, float threshold, int kind, float minSepSq0,
                          float minSepSq1, hipStream_t stream, const char* name)
{
    RSFM_RETURN_IF(nbTasks > 0 && tasks == nullptr, RSFM_ERR_INVALID, std::string(name) + ": tasks is null");
    RSFM_RETURN_IF(!(threshold > 0.f), RSFM_ERR_INVALID, std::string(name) + ": threshold must be > 0");
    const float t2 = threshold * threshold;
    for (size_t b = 0; b < nbTasks; b += kMaxTasks) {
        const size_t n = std::min<size_t>(kMaxTasks, nbTasks - b);
        Batch batch{};
        uint32_t maxH = 0;
        for (size_t i = 0; i < n; i++) {
            const rsfm_ransac_task& t = tasks[b + i];
            RSFM_RETURN_IF(t.nbHyp > 0 && (t.sampleIdx == nullptr || t.counts == nullptr), RSFM_ERR_INVALID,
                           std::string(name) + ": sampleIdx/counts must be set when nbHyp > 0");
            RSFM_RETURN_IF(t.nbPts > 0 && t.pts == nullptr, RSFM_ERR_INVALID, std::string(name) + ": pts is null");
            RSFM_RETURN_IF(reinterpret_cast<uintptr_t>(t.pts) % 16, RSFM_ERR_INVALID,
                           std::string(name) + ": pts must be 16-byte aligned");
            batch.t[i] = DevTask{reinterpret_cast<const float4*>(t.pts), t.nbPtsDev, t.nbPts, t.nbHyp, t.sampleIdx,
                                 t.counts, t.models, t.best, t.inlierMask};
            maxH = std::max(maxH, t.nbHyp);
        }
        if (maxH > 0) RSFM_CHECK(launch_score(batch, (uint32_t)n, maxH, t2, kind, minSepSq0, minSepSq1, stream, name));
        bool anyBest = false;
        for (size_t i = 0; i < n; i++) anyBest |= batch.t[i].best != nullptr || batch.t[i].mask != nullptr;
        if (anyBest) {
            if (kind == 0) best_kernel<0><<<(uint32_t)n, kBestThreads, 0, stream>>>(batch, t2, minSepSq0, minSepSq1);
            else if (kind == 1) best_kernel<1><<<(uint32_t)n, kBestThreads, 0, stream>>>(batch, t2, minSepSq0, minSepSq1);
            else best_kernel<2><<<(uint32_t)n, kBestThreads, 0, stream>>>(batch, t2, minSepSq0, minSepSq1);
            RSFM_CHECK(check_launch(name));
        }
    }
    return RSFM_OK;
}
}  // namespace ransac
}  // namespace rsfm_amd

extern "C" int rsfm_ransac_f8(const rsfm_ransac_task* tasks, size_t nbTasks, float threshold, int mode,
                              float minSepSq0, float minSepSq1, hipStream_t stream)
{
    RSFM_RETURN_IF(mode != 0 && mode != 1, RSFM_ERR_INVALID, "ransac: mode must be 0 (two-sided line) or 1 (Sampson)");
    return ransac::run_hypotheses(tasks, nbTasks, threshold, mode, minSepSq0, minSepSq1, stream, "ransac");
}

extern "C" int rsfm_ransac_h4(const rsfm_ransac_task* tasks, size_t nbTasks, float threshold, float minSepSq0,
                              float minSepSq1, hipStream_t stream)
{
    return ransac::run_hypotheses(tasks, nbTasks, threshold, 2, minSepSq0, minSepSq1, stream, "ransac_h4");
}

extern "C" int rsfm_ransac_sample_indices(uint32_t* sampleIdx, uint32_t nbHyp, uint32_t nbPts,
                                          const uint32_t* nbPtsDev, uint64_t seed, hipStream_t stream)
{
    if (nbHyp == 0) return RSFM_OK;
    RSFM_RETURN_IF(sampleIdx == nullptr, RSFM_ERR_INVALID, "sample_indices: sampleIdx is null");
    ransac::sample_kernel<<<div_up(nbHyp, 256), 256, 0, stream>>>(sampleIdx, nbHyp, nbPts, nbPtsDev, seed);
    return check_launch("ransac sample_indices");
}

namespace {
int sample_batch(const rsfm_sample_task* tasks, size_t nbTasks, uint32_t k, hipStream_t stream)
{
    using namespace ransac;
    RSFM_RETURN_IF(nbTasks > 0 && tasks == nullptr, RSFM_ERR_INVALID, "sample batch: tasks is null");
    RSFM_RETURN_IF(k < 4 || k > 8, RSFM_ERR_INVALID, "sample batch: sampleSize must be in [4, 8]");
    for (size_t b = 0; b < nbTasks; b += kSampleMaxTasks) {
        const size_t n = std::min<size_t>(kSampleMaxTasks, nbTasks - b);
        SampleBatch batch{};
        uint32_t maxH = 0;
        for (size_t i = 0; i < n; i++) {
            const rsfm_sample_task& t = tasks[b + i];
            RSFM_RETURN_IF(t.nbHyp > 0 && t.sampleIdx == nullptr, RSFM_ERR_INVALID, "sample batch: sampleIdx is null");
            batch.t[i] = SampleTask{t.sampleIdx, t.nbHyp, t.nbPts, t.nbPtsDev, t.seed, k};
            maxH = std::max(maxH, t.nbHyp);
        }
        if (maxH == 0) continue;
        sample_batch_kernel<<<dim3(div_up(maxH, 256), (uint32_t)n), 256, 0, stream>>>(batch);
        RSFM_CHECK(check_launch("ransac sample_indices_batch"));
    }
    return RSFM_OK;
}
}  // namespace

extern "C" int rsfm_ransac_sample_indices_batch(const rsfm_sample_task* tasks, size_t nbTasks, hipStream_t stream)
{
    return sample_batch(tasks, nbTasks, 8, stream);
}

extern "C" int rsfm_ransac_sample_indices_batch_k(const rsfm_sample_task* tasks, size_t nbTasks, uint32_t sampleSize,
                                                  hipStream_t stream)
{
    return sample_batch(tasks, nbTasks, sampleSize, stream);
}

extern "C" int rsfm_ransac_sample_weighted_batch(const rsfm_weighted_sample_task* tasks, size_t nbTasks,
                                                 hipStream_t stream)
{
    using namespace ransac;
    RSFM_RETURN_IF(nbTasks > 0 && tasks == nullptr, RSFM_ERR_INVALID, "weighted sample: tasks is null");
    for (size_t b = 0; b < nbTasks; b += kSampleMaxTasks) {
        const size_t n = std::min<size_t>(kSampleMaxTasks, nbTasks - b);
        WSampleBatch batch{};
        uint32_t maxH = 0;
        for (size_t i = 0; i < n; i++) {
            const rsfm_weighted_sample_task& t = tasks[b + i];
            RSFM_RETURN_IF(t.nbHyp > 0 && t.sampleIdx == nullptr, RSFM_ERR_INVALID,
                           "weighted sample: sampleIdx is null");
            RSFM_RETURN_IF(t.nbPts > 0 && (t.weights == nullptr || t.cdf == nullptr), RSFM_ERR_INVALID,
                           "weighted sample: weights/cdf null");
            RSFM_RETURN_IF(reinterpret_cast<uintptr_t>(t.cdf) % 8 != 0, RSFM_ERR_INVALID,
                           "weighted sample: cdf must be 8-byte aligned");
            batch.t[i] = WSampleTask{t.sampleIdx, t.nbHyp, t.nbPts, t.nbPtsDev, t.weights, t.cdf, t.seed};
            maxH = std::max(maxH, t.nbHyp);
        }
        weight_scan_kernel<<<(uint32_t)n, 1024, 0, stream>>>(batch);
        RSFM_CHECK(check_launch("weighted sample scan"));
        if (maxH == 0) continue;
        weighted_sample_kernel<<<dim3(div_up(maxH, (uint32_t)kWSampleThreads), (uint32_t)n), kWSampleThreads, 0, stream>>>(batch);
        RSFM_CHECK(check_launch("weighted sample"));
    }
    return RSFM_OK;
}

extern "C" int rsfm_ransac_f7(const rsfm_ransac_task* tasks, size_t nbTasks, float threshold, int mode, float minSepSq0,
                              float minSepSq1, hipStream_t stream)
{
    using namespace ransac;
    RSFM_RETURN_IF(nbTasks > 0 && tasks == nullptr, RSFM_ERR_INVALID, "ransac7: tasks is null");
    RSFM_RETURN_IF(mode != 0 && mode != 1, RSFM_ERR_INVALID, "ransac7: mode must be 0 (two-sided line) or 1 (Sampson)");
    RSFM_RETURN_IF(!(threshold > 0.f), RSFM_ERR_INVALID, "ransac7: threshold must be > 0");
    const float t2 = threshold * threshold;
    for (size_t b = 0; b < nbTasks; b += kMaxTasks) {
        const size_t n = std::min<size_t>(kMaxTasks, nbTasks - b);
        Batch batch{};
        uint32_t maxH = 0;
        for (size_t i = 0; i < n; i++) {
            const rsfm_ransac_task& t = tasks[b + i];
            RSFM_RETURN_IF(t.nbHyp > 0 && (t.sampleIdx == nullptr || t.counts == nullptr), RSFM_ERR_INVALID,
                           "ransac7: sampleIdx/counts must be set when nbHyp > 0");
            RSFM_RETURN_IF(t.nbPts > 0 && t.pts == nullptr, RSFM_ERR_INVALID, "ransac7: pts is null");
            RSFM_RETURN_IF(reinterpret_cast<uintptr_t>(t.pts) % 16, RSFM_ERR_INVALID, "ransac7: pts must be 16-byte aligned");
            batch.t[i] = DevTask{reinterpret_cast<const float4*>(t.pts), t.nbPtsDev, t.nbPts, t.nbHyp, t.sampleIdx,
                                 t.counts, t.models, t.best, t.inlierMask};
            maxH = std::max(maxH, t.nbHyp);
        }
        if (maxH > 0) {
            const dim3 grid(div_up(maxH, kS7Samples), (uint32_t)n);
            if (mode == 0) score7_kernel<0><<<grid, kS7Block, 0, stream>>>(batch, t2, minSepSq0, minSepSq1);
            else score7_kernel<1><<<grid, kS7Block, 0, stream>>>(batch, t2, minSepSq0, minSepSq1);
            RSFM_CHECK(check_launch("ransac7 score"));
        }
        bool anyBest = false;
        for (size_t i = 0; i < n; i++) anyBest |= batch.t[i].best != nullptr || batch.t[i].mask != nullptr;
        if (anyBest) {
            if (mode == 0) best7_kernel<0><<<(uint32_t)n, kThreads, 0, stream>>>(batch, t2, minSepSq0, minSepSq1);
            else best7_kernel<1><<<(uint32_t)n, kThreads, 0, stream>>>(batch, t2, minSepSq0, minSepSq1);
            RSFM_CHECK(check_launch("ransac7 best"));
        }
    }
    return RSFM_OK;
}
