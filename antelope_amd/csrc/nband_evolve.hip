// nband_evolve.hip - time-fused LengthWannier steps of the analytic classes
// (N <= 8), classical RK4 and fixed-step RK5: one launch runs every step of a
// chunk with rho, the eigenvectors and the model in registers.
//
// The reference's step (SBEs.h:596-624, stage right-hand side :762-861, sample
// :694-760) on the register tiles of tile_small.hpp: N <= 4 takes four k points
// per wave, N <= 8 one, one matrix element per lane. H(k + A(t)) and J are
// trigonometric sums (analytic_terms.hpp): a lane keeps its element's
// coefficients p_t, q_t turned by e^{ik.v_t} once per launch, so a stage's H is
// 4 FMAs per term against the k-independent cos / sin(A.v_t) of a table row, and
// nothing of a step touches HBM but the row of k sums.
//
// Bound by latency: a wave's step is one serial chain of small products (the
// eigenvector refinements above all), so the split that pays is many waves with
// little in each. 64 x 48 k points, bilayer Haldane (4 bands), RK5, 502 steps:
// see the figures at launch_evolve.
#include <cmath>

#include "haldane_dev.hpp"
#include "tile_eig.hpp"

namespace sbe {
namespace {

using namespace tile;
using dev::Coef;

constexpr int kWaves = 4;  // waves per block: one partial row per block and step

// doubles per table row: at t_n H's (cos, sin) pairs and, times the gradients,
// those of J_x, J_y, J_z; then H's pairs at the tableau's other distinct times
template <int RK>
constexpr int mid_times() { return RK == 4 ? 1 : 4; }
template <int RK, int NT>
constexpr int row_len() { return (8 + 2 * mid_times<RK>()) * NT; }

// table[n][...] for n in [0, nt]: A [nt + 1][1 + mids][3]
__global__ __launch_bounds__(256) void evolve_table_kernel(const double *__restrict__ A, const EvolveTerms w, int mids,
                                                           int nt_pad, int64_t rows, double *__restrict__ tab)
{
    const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int t = static_cast<int>(id % nt_pad);
    const int64_t q = id / nt_pad;
    const int u = static_cast<int>(q % (1 + mids));
    const int64_t n = q / (1 + mids);
    if (n >= rows) return;
    const double *a = A + (n * (1 + mids) + u) * 3;
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

template <int Q, int RK, int NT>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2))) void nb_evolve_kernel(
    const NbArgs a, const NbEvolve e, cd *__restrict__ rho, cd *__restrict__ Ust, double *__restrict__ partials)
{
    using T = SmallTile<Q>;
    constexpr int KW = Q == 1 ? 4 : 1;  // k points per wave
    constexpr int R = row_len<RK, NT>();
    static_assert(R <= 64 * kWaves, "a row is fetched by one thread per value");
    extern __shared__ double evolve_lds[];
    double *rows = evolve_lds;                  // [3][R]: table rows n, n + 1, n + 2 by n mod 3
    double *sums = evolve_lds + 3 * R;          // [2][kWaves][nv]
    const int N = a.N, nn = N * N, nv = a.nv;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = Shape<T>::row(0), c = Shape<T>::col(), b = (lane >> 2) & 3;
    const int64_t k = (static_cast<int64_t>(blockIdx.x) * kWaves + w) * KW + (KW == 4 ? b : 0);
    const bool valid = k < a.nk;  // lanes past the block's k points repeat the last one with weight 0
    const int64_t kk = valid ? k : a.nk - 1;
    const double wk = valid ? a.weight[kk] : 0.0;
    const bool in = i < N && c < N;
    const int el = in ? i * N + c : 0;

    // this element's coefficients, turned by the phases of k
    double pr[NT], pi[NT], qr[NT], qi[NT];
    const double kx = a.kpts[3 * kk], ky = a.kpts[3 * kk + 1], kz = a.kpts[3 * kk + 2];
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
    const cd m0 = in ? e.coef[el] : zero, sc = in ? e.coef[(1 + 2 * e.terms.T) * nn + el] : zero;
    auto hmat = [&](const double *r) {
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
    };
    auto jmat = [&](const double *r, double &jr, double &ji) {  // r: the axis's gradient pairs
        double x = 0.0, y = 0.0;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const double co = r[2 * t], s = r[2 * t + 1];
            x = fma(qr[t], co, fma(-pr[t], s, x));
            y = fma(qi[t], co, fma(-pi[t], s, y));
        }
        jr = sc.x * x - sc.y * y;
        ji = sc.x * y + sc.y * x;
    };

    T Rh, U, Ut;
    {
        const cd v = in ? rho[kk * nn + el] : zero;
        const cd u = in ? Ust[kk * nn + el] : make_double2(i == c ? 1.0 : 0.0, 0.0);
        Rh.re[0] = v.x, Rh.im[0] = v.y;
        U.re[0] = u.x, U.im[0] = u.y;
        Ut = transpose(U, nullptr);
    }
    for (int x = tid; x < 2 * R; x += 64 * kWaves) rows[((e.s0 + x / R) % 3) * R + x % R] = e.table[e.s0 * R + x];
    __syncthreads();
    int sl = static_cast<int>(e.s0 % 3);  // this step's row slot
    T H = hmat(rows + sl * R);            // at t_n, carried from step to step
    double lam = 0.0;
    if (e.lam_valid) lam = e.lam[kk * 8 + c];
    else eig_refine(H, U, Ut, N, static_cast<cd *>(nullptr), 1e-8, true, true, &lam);

    const double dt = e.dt, g12 = a.gam1 - a.gam2;
    const bool deph = a.deph != 0;
    // the band-diagonal part enters the dephasing only where T1 and T2 differ
    auto deriv = [&](const T &Y, const T &Hs, const T &V, const T &Vt) {
        T M{};
        double d;
        if (deph && g12 != 0.0) M = band_diag(Y, V, Vt, d);
        return stage_derivative_m<true>(a, Y, Hs, M, static_cast<cd *>(nullptr));
    };
    auto refine = [&](const T &Hs, T &V, T &Vt) {
        if (deph && g12 != 0.0) eig_refine(Hs, V, Vt, N, static_cast<cd *>(nullptr), 1e-8, true, true);
    };

    for (int64_t step = e.s0; step < e.s1; ++step) {
        const double *row = rows + sl * R;
        const int sn = sl == 2 ? 0 : sl + 1, sf = sn == 2 ? 0 : sn + 1;  // slots of the next two rows
        const double *next = rows + sn * R;
        const bool fetch = tid < R && step + 2 <= e.nt;
        const double ahead = fetch ? e.table[(step + 2) * R + tid] : 0.0;
        // ---- sample at t_n
        double pc;
        const T M = band_diag(Rh, U, Ut, pc);
        double v[8];
        v[6] = v[7] = 0.0;
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            double jr = 0.0, ji = 0.0;
            if (ax < 2 || e.jz) jmat(row + (2 + 2 * ax) * NT, jr, ji);
            // Re Tr(rho J) = Re sum conj(rho_ij) J_ij and the same with rho's band-diagonal part
            const double tot = Rh.re[0] * jr + Rh.im[0] * ji;
            const double intra = a.inter_intra ? M.re[0] * jr + M.im[0] * ji : 0.0;
            v[ax] = (tot - intra) * wk;
            v[3 + ax] = intra * wk;
        }
        double *mine = sums + ((step & 1) * kWaves + w) * nv;
        {
            const double cur = dev::wave_reduce8(v);
            if ((lane & 7) == 0 && (lane >> 3) < 6) mine[lane >> 3] = cur;
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
        // one barrier a step: past it every wave has left step n - 1, whose row slot takes row n + 2,
        // and the sums written before it are added below while the other buffer takes step n + 1's
        __syncthreads();
        if (fetch) rows[sf * R + tid] = ahead;
        {
            double *out = partials + ((step - e.s0) * gridDim.x + blockIdx.x) * static_cast<int64_t>(nv);
            const double *s = sums + (step & 1) * kWaves * nv;
            for (int x = tid; x < nv; x += 64 * kWaves) out[x] = ((s[x] + s[nv + x]) + s[2 * nv + x]) + s[3 * nv + x];
        }
        // ---- stages
        T X = stage_derivative_m<true>(a, Rh, H, M, static_cast<cd *>(nullptr));
        if constexpr (RK == 4) {
            T Acc, Y;
            axpy_tile(Acc, X, dt / 6.0, Rh);
            axpy_tile(Y, X, 0.5 * dt, Rh);
            H = hmat(row + 8 * NT);
            refine(H, U, Ut);
            X = deriv(Y, H, U, Ut);
            axpy_tile(Acc, X, dt / 3.0, Acc);
            axpy_tile(Y, X, 0.5 * dt, Rh);
            X = deriv(Y, H, U, Ut);
            axpy_tile(Acc, X, dt / 3.0, Acc);
            axpy_tile(Y, X, dt, Rh);
            H = hmat(next);
            eig_refine(H, U, Ut, N, static_cast<cd *>(nullptr), 1e-8, true, true, &lam);
            X = deriv(Y, H, U, Ut);
            axpy_tile(Rh, X, dt / 6.0, Acc);
        } else {
            // c = 0, 1/4, 3/8, 12/13, 1, 1/2: the last stage starts its eigenvectors from those at
            // 3/8, the step's own go on to the next sample
            using C = Coef<5>;
            T Kd[6], Vm, Vmt, Hs;
            Kd[0] = X;
            auto input = [&](int s) {
                T Y = Rh;
#pragma unroll
                for (int j = 0; j < 5; ++j)
                    if (j < s && C::a[s][j] != 0.0) axpy_tile(Y, Kd[j], dt * C::a[s][j], Y);
                return Y;
            };
            Hs = hmat(row + 8 * NT);
            refine(Hs, U, Ut);
            Kd[1] = deriv(input(1), Hs, U, Ut);
            Hs = hmat(row + 10 * NT);
            refine(Hs, U, Ut);
            Kd[2] = deriv(input(2), Hs, U, Ut);
            Vm = U;
            Vmt = Ut;
            Hs = hmat(row + 12 * NT);
            refine(Hs, U, Ut);
            Kd[3] = deriv(input(3), Hs, U, Ut);
            H = hmat(next);
            eig_refine(H, U, Ut, N, static_cast<cd *>(nullptr), 1e-8, true, true, &lam);
            Kd[4] = deriv(input(4), H, U, Ut);
            Hs = hmat(row + 14 * NT);
            refine(Hs, Vm, Vmt);
            Kd[5] = deriv(input(5), Hs, Vm, Vmt);
#pragma unroll
            for (int j = 0; j < 6; ++j)
                if (C::b[j] != 0.0) axpy_tile(Rh, Kd[j], dt * C::b[j], Rh);
        }
        sl = sn;
    }
    if (valid && in) {
        rho[k * nn + el] = make_double2(Rh.re[0], Rh.im[0]);
        Ust[k * nn + el] = make_double2(U.re[0], U.im[0]);
    }
    if (valid && i == 0) e.lam[k * 8 + c] = lam;
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

}  // namespace

int evolve_blocks(int N, int64_t nk)
{
    const int64_t per = N <= 4 ? 4 * kWaves : kWaves;
    return static_cast<int>((nk + per - 1) / per);
}

hipError_t launch_evolve_table(const double *A, const EvolveTerms &t, int rk_order, int64_t rows, double *tab, hipStream_t s)
{
    const int mids = evolve_times(rk_order) - 1, ntp = evolve_padded_terms(t.T);
    const int64_t n = rows * (1 + mids) * ntp;
    evolve_table_kernel<<<dim3(static_cast<unsigned>((n + 255) / 256)), 256, 0, s>>>(A, t, mids, ntp, rows, tab);
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
