// screen.hpp - matrix-core screening of the epipolar inlier tests.
//
// A hypothesis scorer asks, for every (model F, correspondence) pair, for the
// outcome of fgeom::inlier in FP32 with its fixed rounding. On the vector ALUs
// that is 20 to 37 instructions per pair. Here both sides of the comparison
// come from f16 matrix products instead, with a bound on how far they can be
// off; only the pairs whose outcome the bound leaves open are tested by
// fgeom::inlier itself, so every outcome, hence every count, is the exact
// test's.
//
// Both sides are linear in monomials of the point: e = x1^T F x0 has the nine
// products of (X0, Y0, 1) and (X1, Y1, 1); the squared line normals are
// quadratic forms, 1 + 5 monomials per image. (X, Y) are the coordinates
// centred on the pair's bounding box and scaled to [-1, 1]. Monomials and
// coefficients are split into two f16 halves (22 bits), and the products
// hi*hi, hi*lo, lo*hi fill the K = 32 of one v_mfma_f32_16x16x32_f16: three
// slots per monomial, two for a constant, 26 slots for e and exactly 32 for
// the normals. A 16-point x 16-model block takes two of them (three for the
// two-sided test) and leaves each lane four tests of four vector instructions:
// s = e^2 - D (v_fma), its sign bit collected (v_alignbit; one popcount per 32
// tests), g = |s| - 2 d |e| (v_fma) and, per four tests, their least g compared
// with 2 c (v_min3, v_min, v_sub, v_alignbit).
//
// The bound. Per model, with every quantity scaled alike: S = sum of the
// largest magnitudes of e's terms over the box, Qs the normals' (threshold
// included), Q the largest D over the box.
//  - a staged monomial is off by at most 5 roundings of FP32 and the split's
//    2^-22, a coefficient by 2^-24 + 2^-22, the dropped lo*lo term by 2^-22:
//    18 * 2^-24 per term; a half below f16's normal range adds at most 2^-14
//    absolute on either side (counted whether or not subnormals are kept);
//  - the matrix unit's FP32 accumulation is not documented. It was measured, at up
//    to 5.9 * 2^-24 of the sum of the terms' magnitudes over 3e7 random dot products
//    (uniform, split, spread over 12 binades, cancelling, subnormal; an operand
//    below f16's normal range counts as 2^-14); 10 is assumed, and a test takes
//    the same measurement again;
//  - the exact test's own roundings, from its expressions (make_coef).
// With d and c the sums of these for e and for D (d^2 and the comparison's own
// roundings in c), the exact e^2 - D differs from the screen's by at most
// 2 d |e| + c where it is near zero, so a test with g > c has the exact
// outcome. The others are open and are done by the exact test in groups of the
// lane's four: 2e-4 to 3e-4 of all tests are in such a group at 70% outliers,
// 2e-3 to 3e-3 at 30%, 1e-2 to 2e-2 at 5% (600 and 2454 points, 8 points a model;
// 7-point models up to 1.3e-3 at 70%).
#pragma once
#include "common.hpp"
#include "fgeom.hpp"

namespace rsfm_amd {
namespace screen {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr float kOne = 1024.f;     // monomials are staged times 2^10, away from f16's subnormals
constexpr float kFar = 32768.f;    // coefficient that makes e huge: padding points, rejected models
constexpr uint32_t kMaxPoints = 1u << 23;  // a queued test packs the point in 23 bits, the model in 9
constexpr uint32_t kQueue = 128;           // open tests per wave

// the pair's bounding box: centres, half extents after scaling (at most 1) and
// largest magnitudes in pixels of the four coordinates, scales of the two
// images; odd: coordinates that the bound does not cover
struct Box {
    float c[4], x[4], m[4], s[2];
    uint32_t odd;
};

struct BoxPart {
    float lo[4], hi[4];
    uint32_t odd;
};

__device__ inline void box_init(BoxPart& b)
{
#pragma unroll
    for (int k = 0; k < 4; k++) {
        b.lo[k] = __builtin_inff();
        b.hi[k] = -__builtin_inff();
    }
    b.odd = 0;
}

__device__ inline void box_add(BoxPart& b, const float4& p)
{
    const float v[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        b.lo[k] = fminf(b.lo[k], v[k]);
        b.hi[k] = fmaxf(b.hi[k], v[k]);
        b.odd |= !(fabsf(v[k]) <= 1048576.f);
    }
}

__device__ inline void box_wave_reduce(BoxPart& b)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            b.lo[k] = fminf(b.lo[k], __shfl_xor(b.lo[k], o));
            b.hi[k] = fmaxf(b.hi[k], __shfl_xor(b.hi[k], o));
        }
        b.odd |= (uint32_t)__shfl_xor((int)b.odd, o);
    }
}

__device__ inline Box box_finish(const BoxPart& b, uint32_t n)
{
    Box r;
    r.odd = b.odd | (n > kMaxPoints - 1024);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        r.c[k] = 0.5f * (b.lo[k] + b.hi[k]);
        r.m[k] = fmaxf(fabsf(b.lo[k]), fabsf(b.hi[k]));
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        float h = 0.f;
#pragma unroll
        for (int k = 2 * i; k < 2 * i + 2; k++) h = fmaxf(h, fmaxf(b.hi[k] - r.c[k], r.c[k] - b.lo[k]));
        r.s[i] = h > 0.f ? 1.f / h : 1.f;
#pragma unroll
        for (int k = 2 * i; k < 2 * i + 2; k++) r.x[k] = fmaxf(b.hi[k] - r.c[k], r.c[k] - b.lo[k]) * r.s[i];
        // below this the exact test's own values reach FP32's subnormals
        if (!(fmaxf(r.m[2 * i], r.m[2 * i + 1]) >= 0.0009765625f) || !(h >= 1e-6f)) r.odd = 1;
    }
    return r;
}

struct Half2 {
    _Float16 h, l;
};
__device__ inline Half2 split(float x)
{
    // opaque, so that a product is not converted from its unrounded value in one
    // place (v_fma_mixlo_f16) and from the rounded one in another
    asm("" : "+v"(x));
    Half2 r;
    r.h = (_Float16)x;
    r.l = (_Float16)(x - (float)r.h);
    return r;
}

// the point's two operands for lane group q (K slots 8q .. 8q + 7): e's
// monomials {X1X0, X1Y0 | Y1X0, Y1Y0 | X0, Y0 | X1, Y1} and the normals'
// {X0X0, X0Y0, Y0Y0 | X0, Y0, 1 | the same of image 1}
__device__ inline void point_operands(const Box& B, float4 p, bool valid, int q, v8h& oe, v8h& od)
{
    const float X0 = (p.x - B.c[0]) * B.s[0], Y0 = (p.y - B.c[1]) * B.s[0];
    const float X1 = (p.z - B.c[2]) * B.s[1], Y1 = (p.w - B.c[3]) * B.s[1];
    const float on = valid ? kOne : 0.f;
    const float u = q == 0 ? X1 * on : (q == 1 ? Y1 * on : on);
    const Half2 a = split(u * (q == 3 ? X1 : X0)), b = split(u * (q == 3 ? Y1 : Y0));
    const _Float16 one = (_Float16)on, pad = (_Float16)(kOne - on), zero = (_Float16)0.f;
    oe = v8h{a.h, a.h, a.l, b.h, b.h, b.l, q == 0 ? one : (q == 1 ? pad : zero), q < 2 ? one : zero};
    const float x = q >= 2 ? X1 : X0, y = q >= 2 ? Y1 : Y0;
    const bool odd = (q & 1) != 0;
    const float w = odd ? on : x * on;
    const Half2 c = split(w * x), d = split(w * y), f = split(y * (y * on));
    od = v8h{c.h, c.h, c.l, d.h, d.h, d.l, odd ? f.l : f.h, odd ? one : f.h};
}

// coefficients of one model, scaled by powers of two: e's nine in F's order,
// the normals' {xx, xy, yy, x, y} per image and their constants, 2 d and c
struct Coef {
    float e[9];
    float q[2][5];
    float k[2];  // mode 1: k[0] = the sum's constant; mode 0: one per image
    float d2, c;
    bool far;  // rejected model: never an inlier
};

__device__ inline double pow2d(int e) { return __longlong_as_double((long long)(1023 + e) << 52); }
__device__ inline int expo(double x) { return (int)((__double_as_longlong(x) >> 52) & 0x7FF) - 1022; }  // |x| < 2^expo

template <int kMode>
__device__ inline Coef make_coef(const Box& B, const float F[9], bool ok, float t2)
{
    Coef r;
    r.far = !ok;
    const double g0 = 1.0 / (double)B.s[0], g1 = 1.0 / (double)B.s[1];
    const double c0x = B.c[0], c0y = B.c[1], c1x = B.c[2], c1y = B.c[3];
    double A[3][3], G[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const double f0 = F[3 * i], f1 = F[3 * i + 1], f2 = F[3 * i + 2];
        A[i][0] = f0 * g0;
        A[i][1] = f1 * g0;
        A[i][2] = f0 * c0x + f1 * c0y + f2;
    }
    // largest monomials: (x0, y0, 1) and (x1, y1, 1), scaled and in pixels
    const double e0[3] = {B.x[0], B.x[1], 1.0}, e1[3] = {B.x[2], B.x[3], 1.0};
    const double m0[3] = {B.m[0], B.m[1], 1.0}, m1[3] = {B.m[2], B.m[3], 1.0};
    double S = 0.0, top = 0.0;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        G[0][j] = A[0][j] * g1;
        G[1][j] = A[1][j] * g1;
        G[2][j] = c1x * A[0][j] + c1y * A[1][j] + A[2][j];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            S += fabs(G[i][j]) * e1[i] * e0[j];
            top = fmax(top, fabs(G[i][j]));
        }
    }
    // squared normals times t^2: l1 = F x0 (image 0's monomials), l0 = F^T x1;
    // their sum of term magnitudes, and their largest value: a convex function's, at a corner of the box
    double Q[2][6], sum[2] = {0.0, 0.0}, most[2] = {0.0, 0.0}, topQ = 0.0;
    double nrm[2][2];  // largest |normal component| of l1, l0 in pixels
    const double w[2] = {(double)t2 / (g1 * g1), (double)t2 / (g0 * g0)};
#pragma unroll
    for (int m = 0; m < 2; m++) {
        double a[2][3];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) a[i][j] = m == 0 ? G[i][j] : G[j][i];
        Q[m][0] = w[m] * (a[0][0] * a[0][0] + a[1][0] * a[1][0]);
        Q[m][1] = 2.0 * w[m] * (a[0][0] * a[0][1] + a[1][0] * a[1][1]);
        Q[m][2] = w[m] * (a[0][1] * a[0][1] + a[1][1] * a[1][1]);
        Q[m][3] = 2.0 * w[m] * (a[0][0] * a[0][2] + a[1][0] * a[1][2]);
        Q[m][4] = 2.0 * w[m] * (a[0][1] * a[0][2] + a[1][1] * a[1][2]);
        Q[m][5] = w[m] * (a[0][2] * a[0][2] + a[1][2] * a[1][2]);
        const double* x = m == 0 ? e0 : e1;
        sum[m] = fabs(Q[m][0]) * x[0] * x[0] + fabs(Q[m][1]) * x[0] * x[1] + fabs(Q[m][2]) * x[1] * x[1] +
                 fabs(Q[m][3]) * x[0] + fabs(Q[m][4]) * x[1] + fabs(Q[m][5]);
#pragma unroll
        for (int k = 0; k < 6; k++) topQ = fmax(topQ, fabs(Q[m][k]));
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const double cx = k & 1 ? x[0] : -x[0], cy = k & 2 ? x[1] : -x[1];
            const double u0 = a[0][0] * cx + a[0][1] * cy + a[0][2], u1 = a[1][0] * cx + a[1][1] * cy + a[1][2];
            most[m] = fmax(most[m], w[m] * (u0 * u0 + u1 * u1));
        }
        const double px = m == 0 ? 1.0 / g1 : 1.0 / g0;
#pragma unroll
        for (int i = 0; i < 2; i++) nrm[m][i] = px * (fabs(a[i][0]) * x[0] + fabs(a[i][1]) * x[1] + fabs(a[i][2]));
    }
    // the exact test's roundings, in units of 2^-24: of e (P), of t^2 n (N).
    // l0a = x1 F0 + (y1 F3 + F6) and its like lose at most their terms' and
    // partial sums' magnitudes; e = l0a x0 + (l0b y0 + l0c) adds those of its own
    double P, N;
    {
        double f[9];
#pragma unroll
        for (int k = 0; k < 9; k++) f[k] = fabs((double)F[k]);
        constexpr double kMul = kMode == 0 ? 1.0 : 0.0;  // products are rounded by themselves
        auto line = [&](double a, double b, double c, const double x[3], double most) {
            return kMul * (a * x[0] + b * x[1]) + (b * x[1] + c) + most;
        };
        const double lc = m1[0] * f[2] + m1[1] * f[5] + f[8];
        const double r0a = line(f[0], f[3], f[6], m1, nrm[1][0]), r0b = line(f[1], f[4], f[7], m1, nrm[1][1]);
        const double r0c = line(f[2], f[5], f[8], m1, lc);
        const double r1a = line(f[0], f[1], f[2], m0, nrm[0][0]), r1b = line(f[3], f[4], f[5], m0, nrm[0][1]);
        const double b1 = nrm[1][1] * m0[1];
        P = r0a * m0[0] + r0b * m0[1] + r0c + kMul * (nrm[1][0] * m0[0] + b1) + (b1 + lc);
        N = 2.0 * (double)t2 * (r0a * nrm[1][0] + r0b * nrm[1][1] + r1a * nrm[0][0] + r1b * nrm[0][1]);
    }
    // scale: e's coefficients below 2^10, the normals' (2^(2k + 10) of theirs) below 2^13
    const int ks = 10 - expo(top), kq = (2 - expo(topQ)) >> 1;
    const int k = ks < kq ? ks : kq;
    const double u = 5.9604644775390625e-8;  // 2^-24
    const double Qs = kMode == 1 ? sum[0] + sum[1] : fmax(sum[0], sum[1]);
    const double Qm = kMode == 1 ? most[0] + most[1] : fmin(most[0], most[1]);
    const bool inRange = k > -400 && k < 400 && top > 0.0 && topQ > 0.0 && S < 1e30 && Qs < 1e30 && P < 1e30 && N < 1e30;
    const double ik = inRange ? pow2d(-k) : 1.0, ik2 = inRange ? pow2d(-2 * k) : 1.0;
    const double de = 28.0 * u * S + u * P + 9.0 * 6.2e-5 * ik + 9.0 * u * top;
    const double dq = 28.0 * u * Qs + u * N + 12.0 * 6.2e-5 * 9.765625e-4 * ik2 + 12.0 * u * topQ;
    const double c = 1.01 * (dq + de * de + 12.0 * u * (Qm + dq));
    // with kOne = 2^10 in every staged monomial the matrix unit leaves e times
    // 2^(k + 10) and D times 2^(2k + 20)
    const double sk = inRange ? pow2d(k) : 0.0, sq = inRange ? pow2d(2 * k) : 0.0;
    // out of range: every test of the model stays open
    const bool open = !inRange || !(c * sq < 1e20) || !(de * sk < 1e15);
    const bool use = ok && !open;
    // chosen, not multiplied by zero: out of range they may be infinite or NaN
    auto coef = [&](double x, double f) { return use ? (float)(x * f) : 0.f; };
    const double fq = sq * kOne;
#pragma unroll
    for (int i = 0; i < 9; i++) r.e[i] = coef(G[i / 3][i % 3], sk);
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
        for (int i = 0; i < 5; i++) r.q[m][i] = coef(Q[m][i], fq);
    if (kMode == 1) {
        r.k[0] = coef(Q[0][5] + Q[1][5], fq);
        r.k[1] = 0.f;
    } else {
        r.k[0] = coef(Q[0][5], fq);
        r.k[1] = coef(Q[1][5], fq);
    }
    // an open model has e = D = 0, so g = 0 < c; a padding point has e = kFar kOne, and
    // where its square is below a very large c it is one of an open group, which knows n
    r.d2 = use ? (float)(2.02 * de * sk * kOne) : 0.f;
    r.c = use ? (float)(c * sq * kOne * kOne) : 1.f;
    return r;
}

// the model's operands for lane group q
__device__ inline v8h model_e(const Coef& c, int q)
{
    const _Float16 z = (_Float16)0.f;
    const float a = q == 0 ? c.e[0] : (q == 1 ? c.e[3] : (q == 2 ? c.e[6] : c.e[2]));
    const float b = q == 0 ? c.e[1] : (q == 1 ? c.e[4] : (q == 2 ? c.e[7] : c.e[5]));
    const Half2 x = split(a), y = split(b), k = split(c.e[8]);
    const _Float16 f = (_Float16)(c.far ? kFar : 0.f);
    return v8h{x.h, x.l, x.h, y.h, y.l, y.h, q == 0 ? k.h : (q == 1 ? (_Float16)kFar : z), q == 0 ? k.l : (q == 1 ? f : z)};
}
// the squared normals of image m's monomials (m = 0, 1), or both (m = 2)
__device__ inline v8h model_q(const Coef& c, int q, int m)
{
    const int im = q >> 1;
    const bool odd = (q & 1) != 0, on = m == 2 || m == im;
    const float a = !on ? 0.f : (im ? c.q[1][odd ? 3 : 0] : c.q[0][odd ? 3 : 0]);
    const float b = !on ? 0.f : (im ? c.q[1][odd ? 4 : 1] : c.q[0][odd ? 4 : 1]);
    const float d = !on ? 0.f : (im ? c.q[1][2] : c.q[0][2]);
    const Half2 x = split(a), y = split(b), w = split(d), k = split(m == 1 ? c.k[1] : c.k[0]);
    return v8h{x.h, x.l, x.h, y.h, y.l, y.h, w.h, odd ? (im ? k.l : k.h) : w.l};
}

// LDS of one workgroup of kWaveCount waves; chunks of kPerWave 16-point tiles
// staged by each wave
template <uint32_t kWaveCount, uint32_t kPerWave>
struct Smem {
    static constexpr uint32_t kWaves = kWaveCount, kPer = kPerWave, kTiles = kPer * kWaves, kChunk = kTiles * 16;
    v8h stage[2][kTiles][2][64];  // [buffer][tile][e, normals][lane]
    uint32_t queue[kWaves][kQueue];
    BoxPart part[kWaves];
};
static_assert(sizeof(v8h) == 16, "operand of one lane");

// the wave's models base .. base + count (at most 16 kNB): lane i computes model
// base + i, and the blocks' operands are gathered through LDS, kRB blocks of 16
// at a time. get(k, F) gives model k, false if rejected.
template <int kMode, int kNB, class Sm, class Get>
__device__ inline void load_models(Sm& S, const Box& B, uint32_t base, uint32_t count, float t2, Get get,
                                   v8h (&be)[kNB], v8h (&bq)[kMode == 1 ? 1 : 2][kNB], float (&d2)[kNB], float (&cc)[kNB])
{
    static_assert(kNB <= 4, "one model per lane");
    constexpr int kOps = kMode == 1 ? 2 : 3;
    constexpr int kRB = (int)(sizeof(S.stage) / (Sm::kWaves * kOps * 64 * sizeof(v8h)));
    static_assert(kRB >= 1, "exchange area");
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6, c16 = lane & 15;
    v8h* X = &S.stage[0][0][0][0] + w * (kRB * kOps * 64);  // [block][operand][lane]
    float F[9];
    bool ok = false;
    if (lane < count) ok = get(base + lane, F);
    if (!ok)
#pragma unroll
        for (int k = 0; k < 9; k++) F[k] = 0.f;
    const Coef c = make_coef<kMode>(B, F, ok, t2);
#pragma unroll
    for (int b = 0; b < kNB; b++) {
        d2[b] = -__shfl(c.d2, b * 16 + (int)c16);
        cc[b] = __shfl(c.c, b * 16 + (int)c16);
    }
#pragma unroll
    for (int r = 0; r < kNB; r += kRB) {
        const int mine = (int)(lane >> 4) - r;
        if (mine >= 0 && mine < kRB) {
            v8h* Y = X + mine * (kOps * 64);
#pragma unroll
            for (int g = 0; g < 4; g++) {
                Y[g * 16 + c16] = model_e(c, g);
                if constexpr (kMode == 1) {
                    Y[64 + g * 16 + c16] = model_q(c, g, 2);
                } else {
                    Y[64 + g * 16 + c16] = model_q(c, g, 0);
                    Y[128 + g * 16 + c16] = model_q(c, g, 1);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int b = 0; b < kRB; b++)
            if (r + b < kNB) {
                be[r + b] = X[b * (kOps * 64) + lane];
                bq[0][r + b] = X[b * (kOps * 64) + 64 + lane];
                if constexpr (kMode == 0) bq[1][r + b] = X[b * (kOps * 64) + 128 + lane];
            }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// The points of P against the wave's kNB blocks of 16 models (model base +
// 16 b + lane % 16); certain inliers and the open tests' exact ones are added
// to cnt[] in LDS. kSplit waves hold the same models and share the tiles: this
// one takes tiles part, part + kSplit, ... Every wave of the workgroup calls it
// (the points are staged together); model(k, F) loads model k for an exact test.
template <int kMode, int kNB, int kSplit, class Sm, class Model>
__device__ inline void count_points(Sm& S, const Box& B, const float4* __restrict__ P, uint32_t n, float t2,
                                    uint32_t base, uint32_t part, const v8h (&be)[kNB], const v8h (&bq)[kMode == 1 ? 1 : 2][kNB],
                                    const float (&d2)[kNB], const float (&cc)[kNB], uint32_t* cnt,
                                    Model model)
{
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6, c16 = lane & 15, q = lane >> 4;
    constexpr uint32_t kPer = Sm::kPer, kTiles = Sm::kTiles, kChunk = Sm::kChunk;
    constexpr uint32_t kTurn = kTiles / kSplit < 8 ? kTiles / kSplit : 8;  // tiles per 32 sign bits
    const uint32_t nChunks = (n + kChunk - 1) / kChunk;
    uint32_t acc[kNB];
#pragma unroll
    for (int b = 0; b < kNB; b++) acc[b] = 0;
    float4 p[kPer];
    auto fetch = [&](uint32_t c) {
#pragma unroll
        for (uint32_t u = 0; u < kPer; u++) p[u] = P[min(c * kChunk + (w * kPer + u) * 16 + c16, n - 1)];
    };
    auto stage = [&](uint32_t c) {
#pragma unroll
        for (uint32_t u = 0; u < kPer; u++) {
            const uint32_t t = w * kPer + u;
            v8h oe, od;
            point_operands(B, p[u], c * kChunk + t * 16 + c16 < n, (int)q, oe, od);
            S.stage[c & 1][t][0][lane] = oe;
            S.stage[c & 1][t][1][lane] = od;
        }
    };
    uint32_t* queue = S.queue[w];
    uint32_t qn = 0;
    // the queue's entries [first, first + m): four points of a model each
    auto exact = [&](uint32_t first, uint32_t m) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (lane < m) {
            const uint32_t id = queue[first + lane], k = id >> 23, i = id & (kMaxPoints - 1);
            float F[9];
            model(k, F);
            uint32_t a = 0;
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) a += fgeom::inlier<kMode>(F, P[min(i + j, n - 1)], t2) && i + j < n ? 1u : 0u;
            if (a) atomicAdd(&cnt[k], a);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    fetch(0);
    __syncthreads();  // the operand exchange of load_models used the staging area
    stage(0);
    if (nChunks > 1) fetch(1);
    __syncthreads();
    for (uint32_t c = 0; c < nChunks; c++) {
        if (c + 1 < nChunks) stage(c + 1);
        if (c + 2 < nChunks) fetch(c + 2);
        const uint32_t tiles = min(kTiles, (n - c * kChunk + 15) / 16);
        for (uint32_t t0 = part; t0 < tiles; t0 += kTurn * kSplit) {
            // sign bits of s (four a tile) and of the least g less c (one), the last in bit 0
            uint32_t in[kNB], near[kNB];
#pragma unroll
            for (int b = 0; b < kNB; b++) in[b] = near[b] = 0;
            const uint32_t nt = min(kTurn, (tiles - t0 + kSplit - 1) / kSplit);
            v8h oe = S.stage[c & 1][t0][0][lane], od = S.stage[c & 1][t0][1][lane];
            for (uint32_t t = 0; t < nt; t++) {
                v4f e[kNB], d[kNB], d1[kNB];
                const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int b = 0; b < kNB; b++) {
                    e[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(oe, be[b], zero, 0, 0, 0);
                    d[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(od, bq[0][b], zero, 0, 0, 0);
                    if constexpr (kMode == 0) d1[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(od, bq[1][b], zero, 0, 0, 0);
                }
                // the next tile's operands, in flight under this tile's tests
                const uint32_t tn = min(t0 + (t + 1) * kSplit, kTiles - 1);
                oe = S.stage[c & 1][tn][0][lane];
                od = S.stage[c & 1][tn][1][lane];
#pragma unroll
                for (int b = 0; b < kNB; b++) {
                    float g[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float D = kMode == 0 ? fminf(d[b][j], d1[b][j]) : d[b][j];
                        const float s = fmaf(e[b][j], e[b][j], -D);
                        in[b] = __builtin_amdgcn_alignbit(in[b], __float_as_uint(s), 31);
                        g[j] = fmaf(d2[b], fabsf(e[b][j]), fabsf(s));
                    }
                    const float low = fminf(fminf(fminf(g[0], g[1]), g[2]), g[3]) - cc[b];
                    near[b] = __builtin_amdgcn_alignbit(near[b], __float_as_uint(low), 31);
                }
            }
            bool any = false;
#pragma unroll
            for (int b = 0; b < kNB; b++) any |= near[b] != 0;
            // the turn's open groups, one per lane and trip, to the wave's queue;
            // their sign bits do not count
            while (__any(any)) {
                uint32_t m = 0, k = 0;
#pragma unroll
                for (int b = kNB - 1; b >= 0; b--)
                    if (near[b]) {
                        m = near[b];
                        k = b;
                    }
                const uint32_t bit = (uint32_t)__ffs((int)m) - 1u;
                any = false;
#pragma unroll
                for (int b = 0; b < kNB; b++) {
                    if (m && (uint32_t)b == k) {
                        near[b] &= m - 1;
                        in[b] &= ~(15u << (4 * bit));
                    }
                    any |= near[b] != 0;
                }
                const uint64_t who = __ballot(m != 0);
                if (m)
                    queue[qn + __builtin_amdgcn_mbcnt_hi((uint32_t)(who >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)who, 0u))] =
                        ((base + 16 * k + c16) << 23) | (c * kChunk + (t0 + (nt - 1 - bit) * kSplit) * 16 + 4 * q);
                qn += (uint32_t)__popcll(who);
                if (qn >= 64) {
                    qn -= 64;
                    exact(qn, 64);
                }
            }
#pragma unroll
            for (int b = 0; b < kNB; b++) acc[b] += (uint32_t)__popc(in[b]);
        }
        __syncthreads();
    }
    if (qn) exact(0, qn);
#pragma unroll
    for (int b = 0; b < kNB; b++) {
        uint32_t a = acc[b];
        a += (uint32_t)__shfl_xor((int)a, 16);
        a += (uint32_t)__shfl_xor((int)a, 32);
        if (q == 0 && a) atomicAdd(&cnt[base + 16 * b + c16], a);
    }
}

}  // namespace screen
}  // namespace rsfm_amd
