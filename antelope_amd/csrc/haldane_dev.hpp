// haldane_dev.hpp - device helpers shared by the 2-band (Haldane) kernels:
// wave-level reductions, the Bloch-vector state of one k point and the time
// sample of the currents (antelope.cpp:307-333 with SBEs.h:694-760).
#pragma once

#include "sbe_internal.hpp"

namespace sbe {
namespace dev {

// ------------------------------------------- RK tableaus (SBEs.h:395-416)
template <int RK> struct Coef;
template <> struct Coef<4> {
    static constexpr int S = 4;
    static constexpr double a[4][4] = {{0, 0, 0, 0}, {0.5, 0, 0, 0}, {0, 0.5, 0, 0}, {0, 0, 1.0, 0}};
    static constexpr double b[4] = {1.0 / 6.0, 2.0 / 6.0, 2.0 / 6.0, 1.0 / 6.0};
    static constexpr double c[4] = {0.0, 0.5, 0.5, 1.0};
};
template <> struct Coef<5> {
    static constexpr int S = 6;
    static constexpr double a[6][6] = {
        {0, 0, 0, 0, 0, 0},
        {0.25, 0, 0, 0, 0, 0},
        {3. / 32., 9. / 32., 0, 0, 0, 0},
        {1932. / 2197., -7200. / 2197., 7296. / 2197., 0, 0, 0},
        {439. / 216., -8., 3680. / 513., -845. / 4104., 0, 0},
        {-8. / 27., 2., -3544. / 2565., 1859. / 4104., -11. / 40., 0}};
    static constexpr double b[6] = {16. / 135., 0, 6656. / 12825., 28561. / 56430., -9. / 50., 2. / 55.};
    static constexpr double c[6] = {0.0, 0.25, 3. / 8., 12. / 13., 1.0, 0.5};
};

// Stage bookkeeping of a tableau: the stage at c = 1 (the next step's sample
// time), or -1; for each stage, an earlier stage (>= 1) at the same c, or -1.
template <int RK>
__host__ __device__ constexpr int stage_at_one()
{
    for (int i = 1; i < Coef<RK>::S; ++i)
        if (Coef<RK>::c[i] == 1.0) return i;
    return -1;
}
template <int RK>
__host__ __device__ constexpr int same_time_stage(int i)
{
    for (int j = 1; j < i; ++j)
        if (Coef<RK>::c[j] == Coef<RK>::c[i]) return j;
    return -1;
}

// --------------------------------------------------- wave-level reduction
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// a <- rows {0,1} of a and rows {0,1} of b; b <- rows {2,3} of a and b
__device__ __forceinline__ void swap32(double &a, double &b)
{
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    a = __hiloint2double(hi[0], lo[0]);
    b = __hiloint2double(hi[1], lo[1]);
}

// a <- even rows of a and b; b <- odd rows of a and b
__device__ __forceinline__ void swap16(double &a, double &b)
{
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    a = __hiloint2double(hi[0], lo[0]);
    b = __hiloint2double(hi[1], lo[1]);
}

// The sums of v[0..7] over the 64 lanes of the wave, each in eight lanes: lane l ends with
// the total of v[sum8_value(l)], and the lanes of a value are numbered 0..7 by sum8_member.
// Requires all 64 lanes.
__device__ __forceinline__ int sum8_value(int lane) { return (lane & 3) | ((lane >> 2) & 4); }
__device__ __forceinline__ int sum8_member(int lane) { return ((lane >> 2) & 3) | ((lane >> 3) & 4); }
constexpr unsigned long long kSum8First = 0x0000111100001111ull;  // the lanes of value 0

// On the matrix pipe, which these kernels leave idle: the 4x4x4 FP64 MFMA of four blocks
// (lane l = j + 4 b + 16 i) with A = v_q and B = ones in column q adds v_q's four rows of
// lanes into column q, so four values share one accumulator; a second one with A = ones
// adds the rows of that. The four blocks of a row are added with DPP. 10 MFMAs and 8 VALU
// additions and moves, against 45 VALU instructions of a reduce-scatter by permlane swaps
// and DPP, but a longer way to the sums. A value that is not
// finite meets the others' zeros and makes all eight NaN: only for sums whose reader refuses such a row.
__device__ __forceinline__ double wave_sum8(const double v[8])
{
    const int lane = __lane_id();
    double s[2] = {0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const double e = (lane & 3) == q ? 1.0 : 0.0;
        s[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(v[q], e, s[0], 0, 0, 0);
        s[1] = __builtin_amdgcn_mfma_f64_4x4x4f64(v[4 + q], e, s[1], 0, 0, 0);
    }
    s[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(1.0, s[0], 0.0, 0, 0, 0);
    s[1] = __builtin_amdgcn_mfma_f64_4x4x4f64(1.0, s[1], 0.0, 0, 0, 0);
    double x = (lane & 16) != 0 ? s[1] : s[0];
    x += dpp_f64<0x128>(x);  // row_ror:8
    x += dpp_f64<0x124>(x);  // row_ror:4
    return x;
}

// Sum each of v[0..7] over the 64 lanes of the wave by swaps and DPP (reduce-scatter):
// lane l ends with the total of v[reduce8_value(l)] (value q ^ 2 eight lanes away, in DPP's reach). Requires
// all 64 lanes. The faster of the two in the
// fixed-step length-gauge kernels, us a step, swaps and matrix pipe: FP64 RK4 40^2 k points 0.634 and 0.649,
// 300^2 1.10 and 1.12, 1000^2 8.7 and 9.9; FP32 300^2 0.99 and 1.03; 64 solves of 200^2 408 and 421 ms (FP64),
// 291 and 307 (FP32).
__device__ __forceinline__ int reduce8_value(int lane) { return ((lane >> 3) & 4) | ((lane >> 2) & 2) | ((lane >> 4) & 1); }
__device__ __forceinline__ double wave_reduce8(double v[8])
{
    const int lane = __lane_id();
    // lane bit 5: permlane32 swap + add
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        double a = v[j], b = v[j + 4];
        swap32(a, b);
        v[j] = a + b;  // lanes 0-31: v[j], lanes 32-63: v[j+4]
    }
    // lane bit 4: permlane16 swap + add
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        double a = v[2 * j], b = v[2 * j + 1];
        swap16(a, b);
        v[j] = a + b;  // even rows: v[2j], odd rows: v[2j+1]
    }
    // lane bit 3: rotate by 8 inside each 16-lane row (= lane ^ 8)
    const bool hi = (lane & 8) != 0;
    const double keep = hi ? v[1] : v[0];
    const double send = hi ? v[0] : v[1];
    double x = keep + dpp_f64<0x128>(send);  // row_ror:8
    // eight consecutive lanes now share a value: all-reduce over the low 3 bits
    x += dpp_f64<0x141>(x);  // row_half_mirror (i <-> 7-i)
    x += dpp_f64<0x4E>(x);   // quad_perm [2,3,0,1]
    x += dpp_f64<0xB1>(x);   // quad_perm [1,0,3,2]
    return x;
}

// -------------------------------------------------------- model kernels
template <typename R>
struct Vec3 {
    R x, y, z;
};

// d(k+A) from the six phases e_j = e^{i(k+A).v_j} (a_0..a_2 then b_0..b_2)
template <typename R>
__device__ __forceinline__ Vec3<R> dvec(const R er[6], const R ei[6], R t1, R c3, R M0)
{
    Vec3<R> d;
    d.x = t1 * (er[0] + er[1] + er[2]);
    d.y = t1 * (ei[0] + ei[1] + ei[2]);
    d.z = M0 - c3 * (ei[3] + ei[4] + ei[5]);
    return d;
}

template <typename R> struct StateT;
template <> struct StateT<double> {
    using T = double;
    static constexpr int kComp = 0;
};
template <> struct StateT<float> {
    using T = float;
    static constexpr int kComp = 1;
};

// explicit fused multiply-add: the same inputs give the same bits wherever
// it is inlined (no contraction left to the compiler)
__device__ __forceinline__ float fmar(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmar(double a, double b, double c) { return __builtin_fma(a, b, c); }

// 1/x from the hardware reciprocal: FP64 with one cubic step (residual e: r (1 + e + e^2),
// the estimate's error cubed), FP32 with a Newton step
__device__ __forceinline__ double rcp_nr(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    const double e = fmar(-x, r, 1.0);
    return fmar(r, fmar(e, e, e), r);
}
__device__ __forceinline__ float rcp_nr(float x)
{
    const float r = __builtin_amdgcn_rcpf(x);
    return fmar(r, fmar(-x, r, 1.0f), r);
}
// 1/sqrt(x) and 1/x together: FP64 the hardware root with a cubic step, its square corrected by
// one residual; FP32 the hardware root (1 ulp) and rcp_nr
__device__ __forceinline__ void rsqrt_rcp(double x, double &q, double &inv)
{
    const double q0 = __builtin_amdgcn_rsq(x);
    const double e = fmar(-(x * q0), q0, 1.0);
    q = fmar(q0 * e, fmar(0.375, e, 0.5), q0);
    const double i0 = q * q;
    inv = fmar(i0, fmar(-x, i0, 1.0), i0);
}
__device__ __forceinline__ void rsqrt_rcp(float x, float &q, float &inv)
{
    q = __builtin_amdgcn_rsqf(x);
    inv = rcp_nr(x);
}

// complex product (a + ib)(c + id)
template <typename R>
__device__ __forceinline__ void cmul(R a, R b, R c, R d, R &re, R &im)
{
    re = a * c - b * d;
    im = a * d + b * c;
}

// Per-k registers of one lane.
template <typename R>
struct KPoint {
    R er[6], ei[6];     // e^{i k.v_j} (a_0..a_2, b_0..b_2)
    R n, sx, sy, sz;    // Bloch state
    R cn, cx, cy, cz;   // Kahan compensation (FP32 state only)
    double w;
};

// Everything a k point needs at one time t: the phases e^{i(k+A(t)).v_j},
// d(k+A), |d|^2, 1/|d|^2 and 1/|d|. One function computes it wherever it is
// needed, with explicit FMAs, so equal inputs give equal bits. At a gap closing
// (d = 0) the inverses are finite and meet d = 0 in every product.
template <typename R>
struct Phases {
    R ar[3], ai[3];  // t1 e^{i(k+A).a_j}
    R br[3], bi[3];  // e^{i(k+A).b_j}
    Vec3<R> d;
    R sb;            // sum of bi
    R dd, inv, q;
};

template <typename R> __device__ __forceinline__ R smallest();  // far below any |d|^2 but invertible
template <> __device__ __forceinline__ double smallest<double>() { return 1e-300; }
template <> __device__ __forceinline__ float smallest<float>() { return 1e-36f; }

template <typename R>
__device__ __forceinline__ Phases<R> phases_at(const KPoint<R> &p, const R *row, R c3, R M0)
{
    Phases<R> e;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        e.ar[j] = fmar(p.er[j], row[2 * j], -(p.ei[j] * row[2 * j + 1]));
        e.ai[j] = fmar(p.er[j], row[2 * j + 1], p.ei[j] * row[2 * j]);
        e.br[j] = fmar(p.er[j + 3], row[6 + 2 * j], -(p.ei[j + 3] * row[7 + 2 * j]));
        e.bi[j] = fmar(p.er[j + 3], row[7 + 2 * j], p.ei[j + 3] * row[6 + 2 * j]);
    }
    e.d.x = e.ar[0] + e.ar[1] + e.ar[2];
    e.d.y = e.ai[0] + e.ai[1] + e.ai[2];
    e.sb = e.bi[0] + e.bi[1] + e.bi[2];
    e.d.z = fmar(-c3, e.sb, M0);
    e.dd = fmar(e.d.x, e.d.x, fmar(e.d.y, e.d.y, e.d.z * e.d.z));
    rsqrt_rcp(e.dd > smallest<R>() ? e.dd : smallest<R>(), e.q, e.inv);
    return e;
}

// Half of the stage right-hand side at d (kap = -(g1 - g2)/2 / |d|^2):
// f/2 = d x y - (g2/2) y + ((g2 - g1)/2) (y.d / |d|^2) d, each component one FMA chain.
template <bool DEPH, typename R>
__device__ __forceinline__ Vec3<R> half_rhs(const Vec3<R> &d, R kap, const Vec3<R> &y, R gh2)
{
    Vec3<R> f;
    if (DEPH) {
        const R c = kap * fmar(y.x, d.x, fmar(y.y, d.y, y.z * d.z));
        f.x = fmar(c, d.x, fmar(d.y, y.z, fmar(-d.z, y.y, -(gh2 * y.x))));
        f.y = fmar(c, d.y, fmar(d.z, y.x, fmar(-d.x, y.z, -(gh2 * y.y))));
        f.z = fmar(c, d.z, fmar(d.x, y.y, fmar(-d.y, y.x, -(gh2 * y.z))));
    } else {
        f.x = fmar(d.y, y.z, -(d.z * y.y));
        f.y = fmar(d.z, y.x, -(d.x * y.z));
        f.z = fmar(d.x, y.y, -(d.y * y.x));
    }
    return f;
}

// Time sample of one k point at t_n (antelope.cpp:307-333 with
// SBEs.h:694-760), from the state nn, s and the phases at t_n: adds
// w x (inter_x, inter_y, intra_x, intra_y, s_x, s_y, s_z, s.dhat) to v (FP64), the
// currents without the factor sum8_scale applies to the k sums. Every value is linear in the
// state, so the weight multiplies the four components once; the honeycomb vectors
// (Haldane.h:134-143) turn the derivatives of d0 and d into differences of phases,
//   d/dkx = a0 sqrt3/2 (-(ai3 - ai2), ar3 - ar2, -c3 (2 br1 - br2 - br3)), d0: -c0 (2 bi1 - bi2 - bi3)
//   d/dky = a0/2 (dy - 3 ai1, 3 ar1 - dx, -3 c3 (br2 - br3)),              d0: -3 c0 (bi2 - bi3)
// Evaluated in the state precision R; the k sum is always FP64. Branch-free
// so the scheduler can interleave it with the RK chain.
template <typename R>
__device__ __forceinline__ void sample_state(const Phases<R> &e, double wk, R n, R x, R y, R z, const HaldaneArgs &a,
                                             double v[8])
{
    const R c3 = static_cast<R>(a.c3), c0 = static_cast<R>(a.c0), w = static_cast<R>(wk);
    const Vec3<R> &d = e.d;
    const R nn = n * w, s_x = x * w, s_y = y * w, s_z = z * w;
    const R xx = e.ai[1] - e.ai[2], yx = e.ar[2] - e.ar[1];
    const R zx = -c3 * fmar(R(2), e.br[0], -(e.br[1] + e.br[2]));
    const R ox = -c0 * fmar(R(3), e.bi[0], -e.sb);
    const R xy = fmar(R(-3), e.ai[0], d.y), yy = fmar(R(3), e.ar[0], -d.x);
    const R zy = R(-3) * c3 * (e.br[1] - e.br[2]), oy = R(-3) * c0 * (e.bi[1] - e.bi[2]);
    const R sd = fmar(s_x, d.x, fmar(s_y, d.y, s_z * d.z));
    const R g = sd * e.inv;
    const R tx = fmar(s_x, xx, fmar(s_y, yx, s_z * zx));  // s . d_x d
    const R ty = fmar(s_x, xy, fmar(s_y, yy, s_z * zy));
    const R px = g * fmar(d.x, xx, fmar(d.y, yx, d.z * zx));  // (s.dh)(dh.d_x d)
    const R py = g * fmar(d.x, xy, fmar(d.y, yy, d.z * zy));
    // inter = -(s.d_a d - px), intra = -(n d_a d0 + px)
    v[0] += static_cast<double>(tx - px);
    v[1] += static_cast<double>(ty - py);
    v[2] += static_cast<double>(fmar(nn, ox, px));
    v[3] += static_cast<double>(fmar(nn, oy, py));
    v[4] += static_cast<double>(s_x);
    v[5] += static_cast<double>(s_y);
    v[6] += static_cast<double>(s_z);
    v[7] += static_cast<double>(e.dd > R(0) ? sd * e.q : -s_z);
}

// Which of the two a kernel takes, and the lanes of a value
template <bool SWAPS>
struct Sum8 {
    static constexpr unsigned long long kFirst = SWAPS ? 0xffull : kSum8First;  // the lanes of value 0
    static __device__ __forceinline__ int value(int lane) { return SWAPS ? reduce8_value(lane) : sum8_value(lane); }
    static __device__ __forceinline__ int member(int lane) { return SWAPS ? lane & 7 : sum8_member(lane); }
    static __device__ __forceinline__ double total(double v[8]) { return SWAPS ? wave_reduce8(v) : wave_sum8(v); }
    // of value q the total of value q ^ 2 (row_ror:8, quad_perm [2,3,0,1])
    static __device__ __forceinline__ double other_pair(double x) { return dpp_f64<SWAPS ? 0x128 : 0x4E>(x); }
};

// the factor of this lane's value in the k sums of sample_state
template <bool SWAPS>
__device__ __forceinline__ double sum8_scale(const HaldaneArgs &a, int lane)
{
    const int v = Sum8<SWAPS>::value(lane);
    if (v > 3) return 1.0;
    return (v & 1 ? -0.5 : -0.86602540378443864676) * a.va[0][1];  // va[0] = (0, a0)
}

// The k sums of a sample in this lane's value: inter and intra as they are, or (GenCurrent) the
// total current in the first pair and nothing in the second.
template <bool SWAPS>
__device__ __forceinline__ double sample_sums(double v[8], double scale, bool inter_intra, int lane)
{
    double r = Sum8<SWAPS>::total(v) * scale;
    if (!inter_intra) {  // uniform
        const double o = Sum8<SWAPS>::other_pair(r);  // values 0 <-> 2, 1 <-> 3
        const int q = Sum8<SWAPS>::value(lane);
        r = q > 3 ? r : (q < 2 ? r + o : 0.0);
    }
    return r;
}

template <typename R>
__device__ __forceinline__ void time_sample(const KPoint<R> &p, const Phases<R> &e, const HaldaneArgs &a, double v[8])
{
    sample_state(e, p.w, p.n - p.cn, p.sx - p.cx, p.sy - p.cy, p.sz - p.cz, a, v);
}

}  // namespace dev
}  // namespace sbe
