// nband_velocity.hip - time-fused VelocityHamiltonian steps for N <= 16: steps
// [s0, s1) in one launch (SBEs.h:787-805,862-871: the band-basis
// H = sum_a A_a(t) P_a + diag(E)), classical RK4 or fixed-step RK5.
//
// A wave owns its k points for every step - one on 16x16 tiles (N > 8) or on 4x4
// quadrants (N <= 8), four for N <= 4 (tile_small.hpp) - with pMatrix, E, the
// occupations, rho and the stage derivatives in registers, so only the per-step
// partial rows reach HBM. A block's W waves add their sample sums in LDS into one
// row per step, in wave order, behind one barrier a step (two buffers). A at the
// stage times comes from a table of the whole pulse ([nt][stages][3], the host's
// values), read with uniform loads.
//
// Bound by the serial chain of one k point (a product and a transpose per stage).
// Wannier N = 12, 16 x 15 x 4 k, RK5: 6.4 us per step against 14.4 us with one
// launch per step (12.1 us of kernel), which also wrote and read rho and pMatrix
// every step.
#include "haldane_dev.hpp"
#include "tile_eig.hpp"

namespace sbe {
namespace {

using namespace tile;
using dev::Coef;

// the matrix element of register r, transposed (t) or as stored; 0 outside N x N
template <class T>
__device__ __forceinline__ T load_any(const cd *M, int N, bool t)
{
    const int c = Shape<T>::col();
    T X;
#pragma unroll
    for (int r = 0; r < Shape<T>::E; ++r) {
        const int i = Shape<T>::row(r);
        cd v = make_double2(0.0, 0.0);
        if (i < N && c < N) v = t ? M[c * N + i] : M[i * N + c];
        X.re[r] = v.x;
        X.im[r] = v.y;
    }
    return X;
}

template <class T>
constexpr int k_per_wave() { return Shape<T>::kSize == 4 ? 4 : 1; }
template <class T>
constexpr int tb_len() { return Shape<T>::kSize == 16 ? 16 * kTpad : 0; }  // complex of a wave's transpose buffer

template <class T, int RK, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2))) void nb_vel_fused_kernel(
    const NbArgs a, const NbVelFused f, const cd *__restrict__ P, const double *__restrict__ Eocc,
    cd *__restrict__ rho, double *__restrict__ partials)
{
    using C = Coef<RK>;
    constexpr int E = Shape<T>::E, S = C::S, KW = k_per_wave<T>();
    extern __shared__ cd vel_lds[];
    const int N = a.N, nn = N * N, nv = a.nv;
    const int c = Shape<T>::col(), lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int b = (lane >> 2) & 3;
    const int64_t k = (static_cast<int64_t>(blockIdx.x) * W + w) * KW + (KW == 4 ? b : 0);
    const bool active = k < a.nk;
    const int64_t kk = active ? k : a.nk - 1;  // past the last k point: its copy at weight 0, not stored
    const int64_t ks = a.nk_stride * nn;
    cd *buf = vel_lds + w * tb_len<T>();
    double *red = reinterpret_cast<double *>(vel_lds + W * tb_len<T>());  // [2][W][nv]
    // pMatrix_a read transposed: not Hermitian for the model classes whose J is not
    T R = load_any<T>(rho + kk * nn, N, false);
    const T Px = load_any<T>(P + kk * nn, N, true), Py = load_any<T>(P + ks + kk * nn, N, true),
            Pz = load_any<T>(P + 2 * ks + kk * nn, N, true);
    const double Ec = c < N ? Eocc[kk * 2 * N + c] : 0.0;      // E of band c
    const double oc = c < N ? Eocc[kk * 2 * N + N + c] : 0.0;  // occupation of band c
    const double wk = active ? a.weight[kk] : 0.0;
    const double dt = f.dt;
    for (int64_t step = f.s0; step < f.s1; ++step) {
        // ---- sample at t_n: band populations, currents Tr(rho P_a) split into the
        // diagonal (intraband) and off-diagonal parts, rho sums
        double v[8];
        v[6] = v[7] = 0.0;
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            const T &Pa = ax == 0 ? Px : (ax == 1 ? Py : Pz);
            double inter = 0.0, intra = 0.0;
#pragma unroll
            for (int r = 0; r < E; ++r) {
                const double val = R.re[r] * Pa.re[r] - R.im[r] * Pa.im[r];  // Re(rho_ij P_ji)
                if (Shape<T>::row(r) == c && a.inter_intra) intra += val;
                else inter += val;
            }
            v[ax] = inter * wk;
            v[3 + ax] = intra * wk;
        }
        const double cur = dev::wave_sum8(v);
        double *mine = red + ((step & 1) * W + w) * nv;
        if (dev::sum8_value(lane) < 6) mine[dev::sum8_value(lane)] = cur;  // eight lanes hold each
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const int i = Shape<T>::row(r);
            double rr = R.re[r] * wk, ri = R.im[r] * wk;
            if (KW == 4) {  // over the wave's four k points
                rr += lane_move<kRor8>(rr);
                rr += lane_move<kRor4>(rr);
                ri += lane_move<kRor8>(ri);
                ri += lane_move<kRor4>(ri);
            }
            if (i < N && c < N && (KW == 1 || b == 0)) {
                mine[6 + N + 2 * (i * N + c)] = rr;
                mine[6 + N + 2 * (i * N + c) + 1] = ri;
                if (i == c) mine[6 + c] = rr;
            }
        }
        // the sums of this buffer are added below while the other takes the next step's; the barrier
        // of the step after next comes before this one is written again
        __syncthreads();
        double *row = partials + ((step - f.s0) * f.nblocks + blockIdx.x) * static_cast<int64_t>(nv);
        const double *sm = red + (step & 1) * W * nv;
        for (int x = threadIdx.x; x < nv; x += 64 * W) {
            double sum = sm[x];
#pragma unroll
            for (int q = 1; q < W; ++q) sum += sm[q * nv + x];
            row[x] = sum;
        }
        // ---- the stages
        const double *At = f.A + step * (3 * S);
        T Kd[S], Acc;
#pragma unroll
        for (int st = 0; st < S; ++st) {
            T Y = R;
            if constexpr (RK == 4) {
                if (st > 0) axpy_tile(Y, Kd[st - 1], dt * C::a[st][st - 1], R);
            } else {
#pragma unroll
                for (int j = 0; j < st; ++j)
                    if (C::a[st][j] != 0.0) axpy_tile(Y, Kd[j], dt * C::a[st][j], Y);
            }
            const double A0 = At[3 * st], A1 = At[3 * st + 1], A2 = At[3 * st + 2];
            T M;  // H^T = sum_a A_a P_a^T + diag(E)
#pragma unroll
            for (int r = 0; r < E; ++r) {
                M.re[r] = A0 * Px.re[r] + A1 * Py.re[r] + A2 * Pz.re[r] + (Shape<T>::row(r) == c ? Ec : 0.0);
                M.im[r] = A0 * Px.im[r] + A1 * Py.im[r] + A2 * Pz.im[r];
            }
            const T Q = cmm(M, false, Y);  // H y
            const T Qt = transpose(Q, buf);
            T &X = Kd[st];
#pragma unroll
            for (int r = 0; r < E; ++r) {
                const double dr = Q.re[r] - Qt.re[r], di = Q.im[r] + Qt.im[r];
                double xr = di, xi = -dr;  // -i (H y - (H y)^dag)
                if (a.deph) {
                    const bool dg = Shape<T>::row(r) == c;
                    const double gm = dg ? a.gam1 : a.gam2;
                    xr -= gm * (Y.re[r] - (dg ? oc : 0.0));
                    xi -= gm * Y.im[r];
                }
                X.re[r] = xr;
                X.im[r] = xi;
            }
            if constexpr (RK == 4) axpy_tile(st == S - 1 ? R : Acc, X, dt * C::b[st], st == 0 ? R : Acc);
        }
        if constexpr (RK != 4) {
#pragma unroll
            for (int j = 0; j < S; ++j)
                if (C::b[j] != 0.0) axpy_tile(R, Kd[j], dt * C::b[j], R);
        }
    }
    if (active) {
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const int i = Shape<T>::row(r);
            if (i < N && c < N) rho[k * nn + i * N + c] = make_double2(R.re[r], R.im[r]);
        }
    }
}

template <class T, int RK, int W>
hipError_t launch(const NbArgs &a, const NbVelFused &f, const double2 *P, const double *Eocc, double2 *rho,
                  double *partials, hipStream_t s)
{
    const size_t lds = sizeof(double2) * W * tb_len<T>() + sizeof(double) * 2 * W * a.nv;
    const hipError_t e = allow_lds(reinterpret_cast<const void *>(&nb_vel_fused_kernel<T, RK, W>), lds);
    if (e != hipSuccess) return e;
    nb_vel_fused_kernel<T, RK, W><<<dim3(static_cast<unsigned>(f.nblocks)), 64 * W, lds, s>>>(a, f, P, Eocc, rho, partials);
    return hipGetLastError();
}

template <int RK>
hipError_t launch_rk(const NbArgs &a, const NbVelFused &f, const double2 *P, const double *Eocc, double2 *rho,
                     double *partials, hipStream_t s)
{
    if (a.N <= 4) return launch<SmallTile<1>, RK, 4>(a, f, P, Eocc, rho, partials, s);
    if (a.N <= 8) return launch<SmallTile<2>, RK, 4>(a, f, P, Eocc, rho, partials, s);
    return f.waves == 4 ? launch<Tile, RK, 4>(a, f, P, Eocc, rho, partials, s)
                        : launch<Tile, RK, 8>(a, f, P, Eocc, rho, partials, s);
}

}  // namespace

// k points per block: N <= 8 four waves; N <= 16 eight, or four where blocks of eight would be
// fewer than the CUs (a wave then has a SIMD to itself)
int vel_fused_waves(int N, int64_t nk) { return N <= 8 || (nk + 7) / 8 < 256 ? 4 : 8; }
int64_t vel_fused_blocks(int N, int64_t nk)
{
    const int64_t per = vel_fused_waves(N, nk) * (N <= 4 ? 4 : 1);
    return (nk + per - 1) / per;
}

hipError_t nb_launch_vel_fused(const NbArgs &a, const NbVelFused &f, int rk_order, const double2 *P, const double *Eocc,
                               double2 *rho, double *partials, hipStream_t s)
{
    if (a.N < 1 || a.N > 16 || f.nblocks != vel_fused_blocks(a.N, a.nk) || f.waves != vel_fused_waves(a.N, a.nk) ||
        f.s1 < f.s0)
        return hipErrorInvalidValue;
    if (rk_order == SBE_RK4) return launch_rk<4>(a, f, P, Eocc, rho, partials, s);
    if (rk_order == SBE_RK5_FEHLBERG) return launch_rk<5>(a, f, P, Eocc, rho, partials, s);
    return hipErrorInvalidValue;
}

}  // namespace sbe
