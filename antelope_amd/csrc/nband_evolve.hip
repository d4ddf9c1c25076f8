// nband_evolve.hip - time-fused LengthWannier steps for N <= 8, classical RK4 and
// fixed-step RK5: one launch runs every step it has matrices for, with rho and
// the eigenvectors in registers.
//
// The reference's step (SBEs.h:596-624, stage right-hand side :762-861, sample
// :694-760) on the register tiles of tile_small.hpp: N <= 4 takes four k points
// per wave, N <= 8 one, one matrix element per lane. The matrices come from a
// source:
//  * AnalyticSource: H(k + A(t)) and J are trigonometric sums (analytic_terms.hpp).
//    A lane keeps its element's coefficients p_t, q_t turned by e^{ik.v_t} once per
//    launch, so a stage's H is 4 FMAs per term against the k-independent
//    cos / sin(A.v_t) of a table row; a launch covers a chunk of the pulse.
//  * BoxSource: the second-pass outputs of the separable Fourier sums of a run of
//    steps (nb_launch_box_steps); the last pass, X = sum_m E1[k1][m] T2[m], is
//    M1 complex multiply-adds per element here, its rows loaded one evaluation
//    ahead into registers.
//
// Bound by latency: a wave's step is one serial chain of small products (the
// eigenvector refinements above all), so the split that pays is many waves with
// little in each. Measured over 502 steps: bilayer Haldane (4 bands), 64 x 48 k,
// RK5: 5.2 ms in one launch against 123 ms in 7,000 launches of the 16x16-tile stage,
// sample and model kernels; MoS2 (3 bands), 72 x 72 k, RK4: 4.6 ms against 103 ms.
#include <cmath>

#include "haldane_setup.hpp"
#include "tile_eig.hpp"

namespace sbe {
namespace {

using namespace tile;
using dev::Coef;

constexpr int kWaves = 4;  // waves per block: one partial row per block and step

// what the step loop needs beside the source: steps [s0, s1), the first step's row of the partial
// sums, the energies [k][lam_pitch]
struct EvolveRun {
    int64_t s0, s1, row0;
    double dt;
    double *lam;
    int lam_pitch, lam_valid;
};

// doubles per table row: at t_n H's (cos, sin) pairs and, times the gradients,
// those of J_x, J_y, J_z; then H's pairs at the tableau's other distinct times
template <int RK>
constexpr int mid_times() { return RK == 4 ? 1 : 4; }
template <int RK, int NT>
constexpr int row_len() { return (8 + 2 * mid_times<RK>()) * NT; }

// table[n - step0][...]
__global__ __launch_bounds__(256) void evolve_table_kernel(const TableArgs laser, const double *__restrict__ A, const EvolveTerms w,
                                                           int mids, int nt_pad, double *__restrict__ tab)
{
    const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int t = static_cast<int>(id % nt_pad);
    const int64_t q = id / nt_pad;
    const int u = static_cast<int>(q % (1 + mids));
    const int64_t n = q / (1 + mids);
    if (n >= laser.nsteps) return;
    const int64_t step = laser.step0 + n;
    double a[3];
    if (A) {
        for (int i = 0; i < 3; ++i) a[i] = A[(step * (1 + mids) + u) * 3 + i];
    } else {
        dev::field_at(laser, laser.atmin + laser.dt * static_cast<double>(step) + laser.c[u] * laser.dt, a);
    }
    double s = 0.0, c = 0.0;
    if (t < w.T) sincos(a[0] * w.vec[t][0] + a[1] * w.vec[t][1] + a[2] * w.vec[t][2], &s, &c);
    double *row = tab + n * (8 + 2 * mids) * nt_pad;
    if (u > 0) {
        row += (6 + 2 * u) * nt_pad;
        row[2 * t] = c;
        row[2 * t + 1] = s;
        return;
    }
    row[2 * t] = c;
    row[2 * t + 1] = s;
    for (int ax = 0; ax < 3; ++ax) {
        const double g = t < w.T ? w.grad[t][ax] : 0.0;
        row[(2 + 2 * ax) * nt_pad + 2 * t] = g * c;
        row[(2 + 2 * ax) * nt_pad + 2 * t + 1] = g * s;
    }
}

// lane j of each quad's value in every lane of the quad
template <int J>
__device__ __forceinline__ double quad_bcast(double x)
{
    return lane_move<J * 0x55>(x);
}

// The population of the m-th lowest band for this lane's column index m, from the
// energies and populations per column (ties by index): every column's pair
// passes by in turn.
template <int Q>
__device__ __forceinline__ double ranked_population(double lam, double p, int N)
{
    const int c = Shape<SmallTile<Q>>::col(), q4 = c & ~3;
    double lq[4 * Q], pq[4 * Q];
    int id[4 * Q];
    auto quad = [&](double l, double v, int base, int sgn, int o) {
        lq[o] = quad_bcast<0>(l), lq[o + 1] = quad_bcast<1>(l), lq[o + 2] = quad_bcast<2>(l), lq[o + 3] = quad_bcast<3>(l);
        pq[o] = quad_bcast<0>(v), pq[o + 1] = quad_bcast<1>(v), pq[o + 2] = quad_bcast<2>(v), pq[o + 3] = quad_bcast<3>(v);
        for (int j = 0; j < 4; ++j) id[o + j] = base + sgn * j;
    };
    quad(lam, p, q4, 1, 0);
    if (Q == 2)  // lane l ^ 7: column (1 - q, 3 - j)
        quad(lane_move<kHalfMirror>(lam), lane_move<kHalfMirror>(p), (4 - q4) + 3, -1, 4);
    double out = 0.0;
#pragma unroll
    for (int x = 0; x < 4 * Q; ++x) {
        int rank = 0;
#pragma unroll
        for (int y = 0; y < 4 * Q; ++y)
            rank += id[y] < N && ((lq[y] < lq[x]) || (lq[y] == lq[x] && id[y] < id[x]));
        if (id[x] < N && rank == c) out = pq[x];
    }
    return out;
}

// ------------------------------------------------------------ sources --
// Per wave: which k point and element a lane works for, and the matrices of the
// current step. herm(): H~ is Hermitian and equal to H. pair(u): H~^T's tile (the
// commutator's A operand) and H at the u-th of the tableau's later distinct times
// (the last, u = mids, is t_n + dt); issue(u) / issue_j() start the loads the next
// pair / currents will need.
template <int Q, int RK, int NT>
struct AnalyticSource {
    using T = SmallTile<Q>;
    static constexpr bool kHerm = true;
    static constexpr int R = row_len<RK, NT>(), kMids = mid_times<RK>();
    static_assert(R <= 64 * kWaves, "a row is fetched by one thread per value");
    const NbEvolve &e;
    double *rows;  // LDS [3][R]: table rows n, n + 1, n + 2 by n mod 3
    double pr[NT], pi[NT], qr[NT], qi[NT];
    cd m0, sc;
    int sl, sn, sf;  // slots of this step's row and the next two
    bool fetch = false;
    double ahead = 0.0;

    __device__ AnalyticSource(const NbArgs &a, const NbEvolve &ev, double *lds, int64_t kk, bool in, int el)
        : e(ev), rows(lds)
    {
        const double kx = a.kpts[3 * kk], ky = a.kpts[3 * kk + 1], kz = a.kpts[3 * kk + 2];
        const int nn = a.N * a.N;
        const cd zero = make_double2(0.0, 0.0);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            double s = 0.0, co = 0.0;
            cd p = zero, q = zero;
            if (t < e.terms.T) {
                sincos(kx * e.terms.vec[t][0] + ky * e.terms.vec[t][1] + kz * e.terms.vec[t][2], &s, &co);
                if (in) {
                    p = e.coef[(1 + 2 * t) * nn + el];
                    q = e.coef[(2 + 2 * t) * nn + el];
                }
            }
            pr[t] = p.x * co + q.x * s;
            pi[t] = p.y * co + q.y * s;
            qr[t] = q.x * co - p.x * s;
            qi[t] = q.y * co - p.y * s;
        }
        m0 = in ? e.coef[el] : zero;
        sc = in ? e.coef[(1 + 2 * e.terms.T) * nn + el] : zero;
        for (int x = threadIdx.x; x < 2 * R; x += 64 * kWaves)
            rows[((e.s0 + x / R) % 3) * R + x % R] = e.table[x];
        __syncthreads();
        sl = static_cast<int>(e.s0 % 3);
        sn = sl == 2 ? 0 : sl + 1;
        sf = sn == 2 ? 0 : sn + 1;
    }
    __device__ T hmat(const double *r) const
    {
        T H;
        double x = m0.x, y = m0.y;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const double co = r[2 * t], s = r[2 * t + 1];
            x = fma(pr[t], co, fma(qr[t], s, x));
            y = fma(pi[t], co, fma(qi[t], s, y));
        }
        H.re[0] = x;
        H.im[0] = y;
        return H;
    }
    __device__ void start(T &Ht, T &H) { Ht = H = hmat(rows + sl * R); }
    __device__ void begin(int64_t step)
    {
        fetch = threadIdx.x < R && step + 2 <= e.s1;
        ahead = fetch ? e.table[(step + 2 - e.s0) * R + threadIdx.x] : 0.0;
    }
    __device__ void current(int ax, double &jr, double &ji) const
    {
        jr = ji = 0.0;
        if (ax == 2 && !e.jz) return;
        const double *r = rows + sl * R + (2 + 2 * ax) * NT;
        double x = 0.0, y = 0.0;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const double co = r[2 * t], s = r[2 * t + 1];
            x = fma(qr[t], co, fma(-pr[t], s, x));
            y = fma(qi[t], co, fma(-pi[t], s, y));
        }
        jr = sc.x * x - sc.y * y;
        ji = sc.x * y + sc.y * x;
    }
    // past the step's barrier every wave has left step n - 1, whose slot takes row n + 2
    __device__ void after_barrier()
    {
        if (fetch) rows[sf * R + threadIdx.x] = ahead;
    }
    __device__ void issue(int) {}
    __device__ void issue_j(int64_t) {}
    __device__ void pair(int u, T &Ht, T &H) { Ht = H = hmat(u < kMids ? rows + sl * R + (8 + 2 * u) * NT : rows + sn * R); }
    __device__ void advance()
    {
        sl = sn;
        sn = sf;
        sf = sn == 2 ? 0 : sn + 1;
    }
};

template <int Q, int RK, int MM>
struct BoxSource {
    using T = SmallTile<Q>;
    static constexpr bool kHerm = false;
    static constexpr int kMids = mid_times<RK>();
    const NbBoxRun &e;
    const bool jz;
    int64_t off, nn, mstride;  // this lane's element in a second-pass output, per matrix and per row m
    int M1;
    cd w[MM];                  // E1[k1][m], 0 past M1, off the matrix and for holes of the k box
    cd raw[3 * MM];
    int64_t step = 0;

    __device__ BoxSource(const NbArgs &a, const NbBoxRun &ev, int k1, int64_t col, bool on, int el)
        : e(ev), jz(ev.jz != 0), nn(a.N * a.N), M1(a.boxM[0])
    {
        mstride = static_cast<int64_t>(a.boxK[1]) * a.boxK[2] * a.bcols;
        off = col * a.bcols + el;
#pragma unroll
        for (int m = 0; m < MM; ++m)
            w[m] = on && m < M1 ? a.boxE[0][static_cast<int64_t>(k1) * M1 + m] : make_double2(0.0, 0.0);
    }
    __device__ const cd *ring(int64_t s) const
    {
        return e.ring + ((s % e.nring + e.nring) % e.nring) * e.t2_stride;
    }
    __device__ void load(const cd *src, int n)
    {
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (j < n)
#pragma unroll
                for (int m = 0; m < MM; ++m) raw[j * MM + m] = src[off + j * nn + (m < M1 ? m : 0) * mstride];
    }
    __device__ cd form(int j) const
    {
        double re = 0.0, im = 0.0;
#pragma unroll
        for (int m = 0; m < MM; ++m) {
            const cd x = raw[j * MM + m];
            re = fma(w[m].x, x.x, fma(-w[m].y, x.y, re));
            im = fma(w[m].x, x.y, fma(w[m].y, x.x, im));
        }
        return make_double2(re, im);
    }
    __device__ void take(T &Ht, T &H)
    {
        const cd t = form(0), h = form(1);
        T X;
        X.re[0] = t.x, X.im[0] = t.y;
        H.re[0] = h.x, H.im[0] = h.y;
        Ht = transpose(X, nullptr);  // H~ need not be Hermitian: its transpose, not its conjugate
    }
    __device__ void start(T &Ht, T &H)
    {
        load(ring(e.s0 - 1), 2);
        take(Ht, H);
        step = e.s0;
        issue_j(step);
    }
    __device__ void begin(int64_t s) { step = s; }
    __device__ void issue_j(int64_t s)
    {
        if (s < e.s0 + e.ns) load(e.tj + (s - e.s0) * e.t2_stride, jz ? 3 : 2);
    }
    __device__ void current(int ax, double &jr, double &ji) const
    {
        jr = ji = 0.0;
        if (ax == 2 && !jz) return;
        const cd v = form(ax);
        jr = v.x;
        ji = v.y;
    }
    __device__ void after_barrier() {}
    __device__ void issue(int u)
    {
        load(u < kMids ? e.th + ((step - e.s0) * kMids + u) * e.t2_stride : ring(step), 2);
    }
    __device__ void pair(int, T &Ht, T &H) { take(Ht, H); }
    __device__ void advance() {}
};

// ---------------------------------------------------------------- steps --
// Steps [s0, s1) of the lane's k point kk (valid: the block's, else a stand-in of
// weight 0 that is not stored): rho, the eigenvectors and the energies in, and out.
// on: the element is inside the N x N matrix. sums: LDS [2][kWaves][nv].
template <int Q, int RK, class SRC>
__device__ __forceinline__ void evolve_steps(const NbArgs &a, SRC &src, const EvolveRun &e, int64_t kk, bool valid, bool in,
                                             bool load, double *sums, cd *__restrict__ rho, cd *__restrict__ Ust,
                                             double *__restrict__ partials)
{
    using T = SmallTile<Q>;
    constexpr int KW = Q == 1 ? 4 : 1, kMids = mid_times<RK>();
    const int N = a.N, nn = N * N, nv = a.nv;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = Shape<T>::row(0), c = Shape<T>::col(), b = (lane >> 2) & 3;
    const int el = in ? i * N + c : 0;
    const double wk = valid ? a.weight[kk] : 0.0;
    cd *const none = nullptr;

    T Rh, U, Ut, Ht, H;
    {
        const cd v = in && load ? rho[kk * nn + el] : make_double2(0.0, 0.0);
        const cd u = in && load ? Ust[kk * nn + el] : make_double2(i == c ? 1.0 : 0.0, 0.0);
        Rh.re[0] = v.x, Rh.im[0] = v.y;
        U.re[0] = u.x, U.im[0] = u.y;
        Ut = transpose(U, none);
    }
    src.start(Ht, H);  // at t_n; carried from step to step
    double lam = 0.0;
    if (e.lam_valid) lam = load ? e.lam[kk * e.lam_pitch + c] : 0.0;
    else eig_refine(H, U, Ut, N, none, true, SRC::kHerm, &lam);

    const double dt = e.dt, g12 = a.gam1 - a.gam2;
    const bool deph = a.deph != 0;
    // the band-diagonal part enters the dephasing only where T1 and T2 differ
    auto deriv = [&](const T &Y, const T &Hc, const T &V, const T &Vt) {
        T M{};
        double d;
        if (deph && g12 != 0.0) M = band_diag(Y, V, Vt, d);
        return stage_derivative_m<SRC::kHerm>(a, Y, Hc, M, none);
    };
    auto refine = [&](const T &Hs, T &V, T &Vt) {
        if (deph && g12 != 0.0) eig_refine(Hs, V, Vt, N, none, true, SRC::kHerm);
    };

    for (int64_t step = e.s0; step < e.s1; ++step) {
        src.begin(step);
        // ---- sample at t_n
        double pc;
        const T M = band_diag(Rh, U, Ut, pc);
        double v[8];
        v[6] = v[7] = 0.0;
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            double jr, ji;
            src.current(ax, jr, ji);
            // Re Tr(rho J) = Re sum conj(rho_ij) J_ij and the same with rho's band-diagonal part
            const double tot = Rh.re[0] * jr + Rh.im[0] * ji;
            const double intra = a.inter_intra ? M.re[0] * jr + M.im[0] * ji : 0.0;
            v[ax] = in ? (tot - intra) * wk : 0.0;
            v[3 + ax] = in ? intra * wk : 0.0;
        }
        src.issue(0);
        double *mine = sums + ((step & 1) * kWaves + w) * nv;
        {
            const double cur = dev::wave_sum8(v);
            if (dev::sum8_value(lane) < 6) mine[dev::sum8_value(lane)] = cur;  // eight lanes hold each
            double pop = ranked_population<Q>(lam, pc, N) * wk;
            double rr = Rh.re[0] * wk, ri = Rh.im[0] * wk;
            if (KW == 4) {  // over the wave's four k points
                pop += lane_move<kRor8>(pop);
                pop += lane_move<kRor4>(pop);
                rr += lane_move<kRor8>(rr);
                rr += lane_move<kRor4>(rr);
                ri += lane_move<kRor8>(ri);
                ri += lane_move<kRor4>(ri);
            }
            const bool lead = KW == 1 || b == 0;
            if (lead && i == 0 && c < N) mine[6 + c] = pop;
            if (lead && in) {
                mine[6 + N + 2 * el] = rr;
                mine[6 + N + 2 * el + 1] = ri;
            }
        }
        // one barrier a step: the sums written before it are added below while the other buffer
        // takes the next step's
        __syncthreads();
        src.after_barrier();
        {
            double *out = partials + (e.row0 + step - e.s0) * static_cast<int64_t>(gridDim.x) * nv +
                          static_cast<int64_t>(blockIdx.x) * nv;
            const double *s = sums + (step & 1) * kWaves * nv;
            for (int x = tid; x < nv; x += 64 * kWaves) out[x] = ((s[x] + s[nv + x]) + s[2 * nv + x]) + s[3 * nv + x];
        }
        // ---- stages
        T X = stage_derivative_m<SRC::kHerm>(a, Rh, Ht, M, none);
        if constexpr (RK == 4) {
            T Acc, Y;
            axpy_tile(Acc, X, dt / 6.0, Rh);
            axpy_tile(Y, X, 0.5 * dt, Rh);
            src.pair(0, Ht, H);
            src.issue(kMids);
            refine(H, U, Ut);
            X = deriv(Y, Ht, U, Ut);
            axpy_tile(Acc, X, dt / 3.0, Acc);
            axpy_tile(Y, X, 0.5 * dt, Rh);
            X = deriv(Y, Ht, U, Ut);
            axpy_tile(Acc, X, dt / 3.0, Acc);
            axpy_tile(Y, X, dt, Rh);
            src.pair(kMids, Ht, H);
            src.issue_j(step + 1);
            eig_refine(H, U, Ut, N, none, true, SRC::kHerm, &lam);
            X = deriv(Y, Ht, U, Ut);
            axpy_tile(Rh, X, dt / 6.0, Acc);
        } else {
            // c = 0, 1/4, 3/8, 12/13, 1, 1/2: the last stage starts its eigenvectors from those at
            // 3/8, the step's own go on to the next sample
            using C = Coef<5>;
            T Kd[6], Vm, Vmt, Hc;
            Kd[0] = X;
            auto input = [&](int s) {
                T Y = Rh;
#pragma unroll
                for (int j = 0; j < 5; ++j)
                    if (j < s && C::a[s][j] != 0.0) axpy_tile(Y, Kd[j], dt * C::a[s][j], Y);
                return Y;
            };
            src.pair(0, Hc, H);
            src.issue(1);
            refine(H, U, Ut);
            Kd[1] = deriv(input(1), Hc, U, Ut);
            src.pair(1, Hc, H);
            src.issue(2);
            refine(H, U, Ut);
            Kd[2] = deriv(input(2), Hc, U, Ut);
            Vm = U;
            Vmt = Ut;
            src.pair(2, Hc, H);
            src.issue(kMids);
            refine(H, U, Ut);
            Kd[3] = deriv(input(3), Hc, U, Ut);
            src.pair(kMids, Ht, H);
            src.issue(3);
            eig_refine(H, U, Ut, N, none, true, SRC::kHerm, &lam);
            Kd[4] = deriv(input(4), Ht, U, Ut);
            src.pair(3, Hc, H);
            src.issue_j(step + 1);
            refine(H, Vm, Vmt);
            Kd[5] = deriv(input(5), Hc, Vm, Vmt);
#pragma unroll
            for (int j = 0; j < 6; ++j)
                if (C::b[j] != 0.0) axpy_tile(Rh, Kd[j], dt * C::b[j], Rh);
        }
        src.advance();
    }
    if (valid && in) {
        rho[kk * nn + el] = make_double2(Rh.re[0], Rh.im[0]);
        Ust[kk * nn + el] = make_double2(U.re[0], U.im[0]);
    }
    if (valid && i == 0) e.lam[kk * e.lam_pitch + c] = lam;
}

template <int Q, int RK, int NT>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2))) void nb_evolve_kernel(
    const NbArgs a, const NbEvolve e, cd *__restrict__ rho, cd *__restrict__ Ust, double *__restrict__ partials)
{
    using T = SmallTile<Q>;
    extern __shared__ double evolve_lds[];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int64_t unit = static_cast<int64_t>(blockIdx.x) * kWaves + w;
    const int64_t k = Q == 1 ? unit * 4 + ((lane >> 2) & 3) : unit;
    const bool valid = k < a.nk;  // lanes past the last k point repeat it with weight 0
    const int64_t kk = valid ? k : a.nk - 1;
    const int i = Shape<T>::row(0), c = Shape<T>::col();
    const bool in = i < a.N && c < a.N;
    AnalyticSource<Q, RK, NT> src(a, e, evolve_lds, kk, in, in ? i * a.N + c : 0);
    const EvolveRun run{e.s0, e.s1, 0, e.dt, e.lam, 8, e.lam_valid};
    evolve_steps<Q, RK>(a, src, run, kk, valid, in, true, evolve_lds + 3 * row_len<RK, NT>(), rho, Ust, partials);
}

// Wannier models on a product k grid: a wave's k points differ along a1 (one (k2, k3)
// column, so its second-pass rows are shared), neighbouring units run along a1 too
template <int Q, int RK, int MM>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2))) void nb_box_evolve_kernel(
    const NbArgs a, const NbBoxRun e, cd *__restrict__ rho, cd *__restrict__ Ust, double *__restrict__ partials)
{
    using T = SmallTile<Q>;
    extern __shared__ double evolve_lds[];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int K1 = a.boxK[0], K2 = a.boxK[1], K3 = a.boxK[2];
    const int g1 = Q == 1 ? (K1 + 3) / 4 : K1;  // units per column
    const int64_t unit = static_cast<int64_t>(blockIdx.x) * kWaves + w;
    const int64_t ncol = static_cast<int64_t>(K2) * K3;
    const bool there = unit < g1 * ncol;
    const int64_t col = there ? unit / g1 : 0;
    const int g = there ? static_cast<int>(unit - col * g1) : 0;
    const int k1 = Q == 1 ? 4 * g + ((lane >> 2) & 3) : g;
    // a k block of the grid leaves holes in its box (k map -1): zero matrices, nothing stored
    const int64_t kmap = there && k1 < K1 ? a.box_kinv[(static_cast<int64_t>(k1) * K2 * K3) + col] : -1;
    const bool valid = kmap >= 0;
    const int i = Shape<T>::row(0), c = Shape<T>::col();
    const bool in = i < a.N && c < a.N;
    BoxSource<Q, RK, MM> src(a, e, valid ? k1 : 0, col, valid && in, in ? i * a.N + c : 0);
    const EvolveRun run{e.s0, e.s0 + e.ns, e.row0, e.dt, e.lam, 16, e.lam_valid};
    evolve_steps<Q, RK>(a, src, run, valid ? kmap : 0, valid, in, valid, evolve_lds, rho, Ust, partials);
}

template <int Q, int RK, int NT>
hipError_t launch(const NbArgs &a, const NbEvolve &e, double2 *rho, double2 *U, double *partials, hipStream_t s)
{
    const size_t lds = sizeof(double) * (3 * row_len<RK, NT>() + 2 * kWaves * a.nv);
    nb_evolve_kernel<Q, RK, NT><<<dim3(static_cast<unsigned>(e.nblocks)), 64 * kWaves, lds, s>>>(a, e, rho, U, partials);
    return hipGetLastError();
}

template <int RK, int NT>
hipError_t launch_q(const NbArgs &a, const NbEvolve &e, double2 *rho, double2 *U, double *partials, hipStream_t s)
{
    return a.N <= 4 ? launch<1, RK, NT>(a, e, rho, U, partials, s) : launch<2, RK, NT>(a, e, rho, U, partials, s);
}

template <int RK>
hipError_t launch_rk(const NbArgs &a, const NbEvolve &e, double2 *rho, double2 *U, double *partials, hipStream_t s)
{
    switch (evolve_padded_terms(e.terms.T)) {
    case 3: return launch_q<RK, 3>(a, e, rho, U, partials, s);
    case 6: return launch_q<RK, 6>(a, e, rho, U, partials, s);
    default: return launch_q<RK, 9>(a, e, rho, U, partials, s);
    }
}

template <int Q, int RK>
hipError_t launch_box(const NbArgs &a, const NbBoxRun &e, double2 *rho, double2 *U, double *partials, hipStream_t s)
{
    const size_t lds = sizeof(double) * 2 * kWaves * a.nv;
    const dim3 grid(static_cast<unsigned>(e.nblocks));
    if (a.boxM[0] <= 3) nb_box_evolve_kernel<Q, RK, 3><<<grid, 64 * kWaves, lds, s>>>(a, e, rho, U, partials);
    else if (a.boxM[0] <= 5) nb_box_evolve_kernel<Q, RK, 5><<<grid, 64 * kWaves, lds, s>>>(a, e, rho, U, partials);
    else nb_box_evolve_kernel<Q, RK, 7><<<grid, 64 * kWaves, lds, s>>>(a, e, rho, U, partials);
    return hipGetLastError();
}

}  // namespace

int box_evolve_blocks(int N, const int K[3])
{
    const int64_t units = static_cast<int64_t>(N <= 4 ? (K[0] + 3) / 4 : K[0]) * K[1] * K[2];
    return static_cast<int>((units + kWaves - 1) / kWaves);
}

hipError_t launch_box_evolve(const NbArgs &a, const NbBoxRun &e, int rk_order, double2 *rho, double2 *U, double *partials,
                             hipStream_t s)
{
    if (!a.box || a.N < 1 || a.N > 8 || a.boxM[0] > kNbFusedMaxM1 || e.ns < 1 || e.nring < 1 || e.s0 < 0 ||
        e.nblocks != box_evolve_blocks(a.N, a.boxK))
        return hipErrorInvalidValue;
    if (rk_order == SBE_RK4)
        return a.N <= 4 ? launch_box<1, 4>(a, e, rho, U, partials, s) : launch_box<2, 4>(a, e, rho, U, partials, s);
    if (rk_order == SBE_RK5_FEHLBERG)
        return a.N <= 4 ? launch_box<1, 5>(a, e, rho, U, partials, s) : launch_box<2, 5>(a, e, rho, U, partials, s);
    return hipErrorInvalidValue;
}

int evolve_blocks(int N, int64_t nk)
{
    const int64_t per = N <= 4 ? 4 * kWaves : kWaves;
    return static_cast<int>((nk + per - 1) / per);
}

hipError_t launch_evolve_table(const TableArgs &laser, const double *A, const EvolveTerms &t, int rk_order, double *tab, hipStream_t s)
{
    const int mids = evolve_times(rk_order) - 1, ntp = evolve_padded_terms(t.T);
    if (laser.nsteps < 1 || laser.nstage != 1 + mids || (!A && laser.npulses > kMaxDevicePulses)) return hipErrorInvalidValue;
    const int64_t n = laser.nsteps * (1 + mids) * ntp;
    evolve_table_kernel<<<dim3(static_cast<unsigned>((n + 255) / 256)), 256, 0, s>>>(laser, A, t, mids, ntp, tab);
    return hipGetLastError();
}

hipError_t launch_evolve(const NbArgs &a, const NbEvolve &e, int rk_order, double2 *rho, double2 *U, double *partials,
                         hipStream_t s)
{
    if (a.N < 1 || a.N > 8 || e.terms.T > kEvolveMaxTerms || e.s1 <= e.s0 || e.nblocks != evolve_blocks(a.N, a.nk))
        return hipErrorInvalidValue;
    if (rk_order == SBE_RK4) return launch_rk<4>(a, e, rho, U, partials, s);
    if (rk_order == SBE_RK5_FEHLBERG) return launch_rk<5>(a, e, rho, U, partials, s);
    return hipErrorInvalidValue;
}

}  // namespace sbe
