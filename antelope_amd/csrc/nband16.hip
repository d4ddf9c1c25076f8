// nband16.hip - N-band (Wannier) stage and sample kernels for N <= 16 with
// every matrix in MFMA registers.
//
// Same mathematics as nb_rhs_kernel / nb_sample_kernel (SBEs.h:762-861 RHS,
// SBEs.h:694-760 currents), restructured for one 16x16 FP64 MFMA tile per
// matrix and one wave per k point:
//  * A 16x16 complex matrix is a Tile: lane l = c + 16 g holds the elements
//    (g + 4r, c), r = 0..3 - the D layout of v_mfma_f64_16x16x4f64. Bands
//    beyond N are zero padding (identity in the eigenvectors).
//  * C = A B runs as four real MFMAs per K block of 4. The B operand of
//    block kb is register kb of B's tile; the A operand is register kb of
//    A^T's tile. For Hermitian A (H, H~, rho) and for A = X^dag that is
//    the conjugate of A's own tile, so products of that form need no data
//    movement; a transpose (U^T, T^dag) goes through a padded 16x17 LDS
//    buffer of the wave, conflict-free.
//  * Eigenvectors U(k + A(t)) are refined from the stored ones (warm start)
//    by rotations written as matrix products, second order in the Jacobi
//    angles (eig_refine). The columns keep the order of the warm start (bands
//    are followed continuously); the sample kernel ranks them by eigenvalue,
//    as the reference's ascending zheevr order.
//  * The dephasing U (Gamma o (U^dag y U)) U^dag is g2 y + (g1 - g2)
//    U diag(U^dag y U) U^dag (Gamma = g1 on the diagonal, g2 off it): one
//    product y U, a column reduction and one product U diag(d) U^dag.
//  * Currents: Tr(rho J_a) elementwise; the intraband part sum_i
//    (U^dag rho U)_ii (U^dag J_a U)_ii from the products rho U and J_a U.
//    J_a (and pMatrix_a below) is read transposed and used as a general
//    matrix: some model classes' current matrices are not Hermitian.
//  * VelocityHamiltonian gauge (band basis): one product H y per stage with
//    H = sum_a A_a P_a + diag(E) formed elementwise, the stage derivatives
//    kept in registers.
#include <cmath>
#include <map>
#include <mutex>

#include "haldane_dev.hpp"
#include "nband.hpp"
#include "tile_eig.hpp"

namespace sbe {
namespace {

using namespace tile;


// Stage i: y = rho + sum_j dt a_ij k_j; k_i = f(y); after the last stage
// rho += sum_i dt b_i k_i. PAIR: stage sg and the next stage sg2 at the same
// time (RK4's c = 1/2, 1/2) in one pass, sharing H~, U and rho in registers;
// sg2's input takes sg's derivative from registers. Two waves a SIMD: at three (168 registers) the
// refinement spills 46 to 58 of them to scratch (SPLIT16, 16 bands, 48x48x8 k points, 16 RK5 steps: 41.6 ms
// at three, 38.0 at two, and 39.3 before the refinement was second order).
template <bool PAIR>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void nb16_rhs_kernel(
    const NbArgs a, const NbStage sg, const NbStage sg2, const cd *__restrict__ mats, cd *__restrict__ rho,
    cd *__restrict__ kbuf, cd *__restrict__ Ust)
{
    __shared__ cd buf[16 * kTpad];
    const int64_t k = blockIdx.x;
    if (k >= a.nk) return;
    const int N = a.N, nn = N * N;
    const int64_t kstride = a.nk_stride * nn;
    cd *rk = rho + k * nn;
    // rho is read again where needed rather than held across the stages (registers)
    Tile Y = load_tile(rk, N);
    for (int j = 0; j < sg.stage; ++j) {
        if (sg.a[j] == 0.0) continue;
        const Tile Kj = load_tile(kbuf + j * kstride + k * nn, N);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            Y.re[r] += sg.a[j] * Kj.re[r];
            Y.im[r] += sg.a[j] * Kj.im[r];
        }
    }
    const Tile HtT = load_tile_t(mats + k * nn, N);  // mat 0: H~ = H + E.D, transposed (A operand)
    Tile U, Ut;
    if (a.deph) {
        U = load_tile(Ust + k * nn, N, true);
        Ut = transpose(U, buf);
        if (!sg.ureuse) {  // eigenvectors at this stage time, warm-started
            const Tile H = load_tile(mats + a.nk_stride * nn + k * nn, N);  // mat 1: H
            eig_refine(H, U, Ut, N, buf);
            store_tile(Ust + k * nn, U, N);
        }
    }
    Tile X = stage_derivative(a, Y, HtT, U, Ut, buf);
    store_tile(kbuf + sg.stage * kstride + k * nn, X, N);
    const NbStage &fin = PAIR ? sg2 : sg;  // the stage whose derivative X holds at the end
    if (PAIR) {
        Tile Y2 = load_tile(rk, N);
        for (int j = 0; j < sg2.stage; ++j) {
            if (sg2.a[j] == 0.0) continue;
            const Tile Kj = j == sg.stage ? X : load_tile(kbuf + j * kstride + k * nn, N);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                Y2.re[r] += sg2.a[j] * Kj.re[r];
                Y2.im[r] += sg2.a[j] * Kj.im[r];
            }
        }
        X = stage_derivative(a, Y2, HtT, U, Ut, buf);
        store_tile(kbuf + sg2.stage * kstride + k * nn, X, N);
    }
    if (fin.last) {
        Tile Rn = load_tile(rk, N);
        for (int j = 0; j < fin.nstage; ++j) {
            if (fin.b[j] == 0.0) continue;
            const Tile Kj = j == fin.stage ? X : load_tile(kbuf + j * kstride + k * nn, N);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                Rn.re[r] += fin.b[j] * Kj.re[r];
                Rn.im[r] += fin.b[j] * Kj.im[r];
            }
        }
        store_tile(rk, Rn, N);
    }
}

// ------------------------------------------------------------ sample --
// Observables at t_n (mats slots 1..4: H, J_x, J_y, J_z at k + A(t_n)); each wave walks
// k = wave, wave + G, ... and writes one row of partial sums
// [inter(3) intra(3) pop(N) rho(2 N^2)], as nb_sample_kernel.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void nb16_sample_kernel(const NbArgs a, const cd *__restrict__ mats,
                                                         const cd *__restrict__ rho, double *__restrict__ partials,
                                                         int64_t step_local, cd *__restrict__ Ust, int ureuse)
{
    __shared__ cd buf[16 * kTpad];
    const int N = a.N, nn = N * N;
    const int c = lane_c(), g = lane_g();
    const int lane = threadIdx.x;
    double racc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    double cur[6] = {0, 0, 0, 0, 0, 0};
    double pop = 0.0;  // lane m < N: population of the m-th lowest band
    for (int64_t k = blockIdx.x; k < a.nk; k += gridDim.x) {
        const double w = a.weight[k];
        const Tile R = load_tile(rho + k * nn, N);
        const Tile H = load_tile(mats + a.nk_stride * nn + k * nn, N);  // mat 1: H
        Tile U = load_tile(Ust + k * nn, N, true);
        if (!ureuse) {  // eigenvectors at k + A(t_n), warm-started from the last ones
            Tile Ut = transpose(U, buf);
            eig_refine(H, U, Ut, N, buf);
            store_tile(Ust + k * nn, U, N);
        }
        // band energies (for the ascending order) and populations of U's columns
        const double lam = col_dot(U, cmm(H, true, U));
        const double p = col_dot(U, cmm(R, true, U));
        int rank = 0;  // rank of column c among the N energies, ties by index
        for (int j = 0; j < N; ++j) {
            const double lj = __shfl(lam, j, 64);
            rank += (lj < lam) || (lj == lam && j < c);
        }
        for (int j = 0; j < N; ++j) {
            const int rj = __shfl(rank, j, 64);
            const double pj = __shfl(p, j, 64);
            if (rj == lane) pop += pj * w;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            racc[2 * r] += R.re[r] * w;
            racc[2 * r + 1] += R.im[r] * w;
        }
        for (int ax = 0; ax < 3; ++ax) {
            // mats 2..4: J_a, read transposed: some model classes' J is not Hermitian
            const Tile Jt = load_tile_t(mats + (2 + ax) * a.nk_stride * nn + k * nn, N);
            double tot = 0.0;  // Re Tr(rho J) = sum_ij Re(rho_ij J_ji)
#pragma unroll
            for (int r = 0; r < 4; ++r) tot += R.re[r] * Jt.re[r] - R.im[r] * Jt.im[r];
            tot = wave_sum(tot);
            double intra = 0.0;
            if (a.inter_intra) {
                const double jd = col_dot(U, cmm(Jt, false, U));  // Re (U^dag J U)_cc
                intra = wave_sum(lane < 16 && c < N ? p * jd : 0.0);
            }
            cur[ax] += (tot - intra) * w;
            cur[3 + ax] += intra * w;
        }
    }
    double *row = partials + (step_local * gridDim.x + blockIdx.x) * static_cast<int64_t>(a.nv);
    if (lane < 6) {
        double v = 0.0;
#pragma unroll
        for (int q = 0; q < 6; ++q)
            if (lane == q) v = cur[q];
        row[lane] = v;
    }
    if (lane < N) row[6 + lane] = pop;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = g + 4 * r;
        if (i < N && c < N) {
            row[6 + N + 2 * (i * N + c)] = racc[2 * r];
            row[6 + N + 2 * (i * N + c) + 1] = racc[2 * r + 1];
        }
    }
}

// ------------------------------------------------- velocity gauge ----
// One time step of the VelocityHamiltonian gauge (SBEs.h:762-861 with the
// band-basis H = sum_a A_a(t) P_a + diag(E)), as nb_vel_step_kernel: the
// sample at t_n, S stages with the derivatives in registers, the update.
// Each wave walks k = wave, wave + G, ... and writes one row of partial sums.
template <int S>
__global__ __launch_bounds__(64) void nb16_vel_step_kernel(const NbArgs a, const NbVelStep v,
                                                           const cd *__restrict__ P, const double *__restrict__ Eocc,
                                                           cd *__restrict__ rho, double *__restrict__ partials,
                                                           int64_t step_local)
{
    __shared__ cd buf[16 * kTpad];
    const int N = a.N, nn = N * N;
    const int c = lane_c(), g = lane_g();
    const int lane = threadIdx.x;
    const int64_t ks = a.nk_stride * nn;
    double racc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    double cur[6] = {0, 0, 0, 0, 0, 0};
    double pop = 0.0;
    for (int64_t k = blockIdx.x; k < a.nk; k += gridDim.x) {
        const double w = a.weight[k];
        const Tile R = load_tile(rho + k * nn, N);
        // pMatrix_a read transposed: not Hermitian for the model classes whose J is not
        const Tile Px = load_tile_t(P + k * nn, N), Py = load_tile_t(P + ks + k * nn, N),
                   Pz = load_tile_t(P + 2 * ks + k * nn, N);
        const double Ec = c < N ? Eocc[k * 2 * N + c] : 0.0;       // E of band c
        const double oc = c < N ? Eocc[k * 2 * N + N + c] : 0.0;   // occupation of band c
        // ---- sample at t_n: band populations, currents Tr(rho P_a) split
        // into the diagonal (intraband) and off-diagonal parts, rho sums
        double lr[4], lc;
        diag_bcast(R, lr, lc);
        if (lane < N) pop += lc * w;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            racc[2 * r] += R.re[r] * w;
            racc[2 * r + 1] += R.im[r] * w;
        }
        for (int ax = 0; ax < 3; ++ax) {
            const Tile &Pa = ax == 0 ? Px : (ax == 1 ? Py : Pz);
            double inter = 0.0, intra = 0.0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double val = R.re[r] * Pa.re[r] - R.im[r] * Pa.im[r];  // Re(rho_ij P_ji)
                if (g + 4 * r == c && a.inter_intra) intra += val;
                else inter += val;
            }
            cur[ax] += wave_sum(inter) * w;
            cur[3 + ax] += wave_sum(intra) * w;
        }
        // ---- RK stages
        Tile Kd[S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            Tile Y = R;
#pragma unroll
            for (int j = 0; j < s; ++j) {
                if (v.a[s][j] == 0.0) continue;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    Y.re[r] += v.a[s][j] * Kd[j].re[r];
                    Y.im[r] += v.a[s][j] * Kd[j].im[r];
                }
            }
            const double A0 = v.A[s][0], A1 = v.A[s][1], A2 = v.A[s][2];
            Tile M;  // H^T = sum_a A_a P_a^T + diag(E)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                M.re[r] = A0 * Px.re[r] + A1 * Py.re[r] + A2 * Pz.re[r] + (g + 4 * r == c ? Ec : 0.0);
                M.im[r] = A0 * Px.im[r] + A1 * Py.im[r] + A2 * Pz.im[r];
            }
            const Tile T = cmm(M, false, Y);  // H y
            const Tile Tt = transpose(T, buf);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double dr = T.re[r] - Tt.re[r], di = T.im[r] + Tt.im[r];
                double xr = di, xi = -dr;  // -i (H y - (H y)^dag)
                if (a.deph) {
                    const bool dg = g + 4 * r == c;
                    const double gm = dg ? a.gam1 : a.gam2;
                    xr -= gm * (Y.re[r] - (dg ? oc : 0.0));
                    xi -= gm * Y.im[r];
                }
                Kd[s].re[r] = xr;
                Kd[s].im[r] = xi;
            }
        }
        Tile Rn = R;
#pragma unroll
        for (int j = 0; j < S; ++j) {
            if (v.b[j] == 0.0) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                Rn.re[r] += v.b[j] * Kd[j].re[r];
                Rn.im[r] += v.b[j] * Kd[j].im[r];
            }
        }
        store_tile(rho + k * nn, Rn, N);
    }
    double *row = partials + (step_local * gridDim.x + blockIdx.x) * static_cast<int64_t>(a.nv);
    if (lane < 6) {
        double vv = 0.0;
#pragma unroll
        for (int q = 0; q < 6; ++q)
            if (lane == q) vv = cur[q];
        row[lane] = vv;
    }
    if (lane < N) row[6 + lane] = pop;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = g + 4 * r;
        if (i < N && c < N) {
            row[6 + N + 2 * (i * N + c)] = racc[2 * r];
            row[6 + N + 2 * (i * N + c) + 1] = racc[2 * r + 1];
        }
    }
}


// ------------------------------------------------- fused RK step -----
// One RK4 or RK5 step per launch (SBEs.h:596-624 with the stage right-hand side of
// SBEs.h:762-861 and the sample of SBEs.h:694-760), for a product k grid with
// separable Fourier sums. Block = four k points that share (k2, k3) and differ
// along a1, one wave each. The sums' last pass (along a1),
//   X(k1, k2, k3) = sum_m E1[k1][m] T2[m][k2][k3],
// runs here: the block stages T2's M1 rows of its column for two matrices at a
// time in LDS and every wave forms its own tiles from them, so H~, H and J of
// the three times of a step are read once per column instead of written and
// read back per k point. Per wave and step: the sample at t_n (U, rho and the
// band energies from the last step), stage 1 at t_n, stages 2 and 3 at
// t_n + dt/2 (eigenvectors refined there), stage 4 at t_n + dt (eigenvectors
// refined for the next sample); rho, U and the energies are the only per-k
// HBM traffic. The waves' sample sums are added in LDS in wave order into
// one partial row per block.
//
// Bound by the FP64 pipe, which MFMA and VALU share: of the 64 thousand cycles that a SIMD spends
// on a k point 32 are MFMA (32 products) and about 15 VALU; the rest are waits for LDS, barriers and MFMA
// results that the second wave of the SIMD does not cover. Two staging slots instead of four let two
// blocks of four waves share a CU (one of eight before): while one waits at a barrier the
// other has products to do. That and one fixed chunk of every staged row per wave, in place
// of a chunk list with a division per load (3800 scalar instructions per k point), took
// 48x48x8 with 16 bands from 371 to 329 ms, 628 steps; six wave sums in one (wave_sum8) are
// part of it. (In kernel time 308 ms then and 317 since the refinement ends degenerate bands in a unitary basis.)
//
// RK5 (Fehlberg): the same blocks and staging over five later times; the six stage
// derivatives stay in registers, so one wave has a SIMD to itself (512 registers). One launch
// instead of fourteen: 247 -> 105 us a step on 24x24 k points, 2162 -> 1600 on 48x48x8,
// 16 bands; 207 -> 83 on 14x14, 12 bands.

// dynamic LDS of a block: the waves' transpose buffers (which also hold a wave's sample
// sums once), then two staging slots of kNbFusedMaxM1 x 256 complex each (row m of the
// second-pass output at m * 256, so the m offsets are immediates). The slots fill straight
// from global memory (global_load_lds); their tiles are formed into registers first, so they
// fill again while the block computes.
constexpr int kFusedW = kNbFusedWaves;
constexpr int kFusedPitch = 256;
constexpr int kFusedBuf = 16 * kTpad;  // complex per wave
static_assert(64 * kFusedW >= 256, "a wave per chunk of a 16 x 16 matrix");
static_assert(2 * kFusedBuf >= 6 + 16 + 2 * 256, "a wave's sample sums fit its transpose buffer");

__device__ __forceinline__ cd *fused_slot(cd *lds, int slot)
{
    return lds + kFusedW * kFusedBuf + slot * (kNbFusedMaxM1 * kFusedPitch);
}

// This wave's share of filling slot 0 with matrix j0 of src0 and slot 1 with j1 of src1
// (src1 may be null), rows m < M1 of column col: wave w takes chunk w of 64 complex of
// every row (N N <= 256), each lane one element straight to LDS; their completion is
// counted by vmcnt (fused_wait).
__device__ __forceinline__ void stage_async(const NbArgs &a, cd *lds, const cd *src0, int j0, const cd *src1, int j1,
                                            int64_t col, int w, int lane)
{
    const int nn = a.N * a.N, M1 = a.boxM[0];
    const int64_t mstride = static_cast<int64_t>(a.boxK[1]) * a.boxK[2] * a.bcols;
    const int ij = w * 64 + lane;
    if (ij < nn) {
#pragma unroll
        for (int slot = 0; slot < 2; ++slot) {
            if (slot && !src1) break;
            const cd *src = (slot ? src1 : src0) + col * a.bcols + (slot ? j1 : j0) * nn + ij;
            cd *dst = fused_slot(lds, slot) + w * 64;
#pragma unroll
            for (int m = 0; m < kNbFusedMaxM1; ++m) {
                if (m < M1) {
                    __builtin_amdgcn_global_load_lds(src, dst + m * kFusedPitch, 16, 0, 0);
                    src += mstride;
                }
            }
        }
    }
}

// every wave's staging loads have landed and every wave is past its last reads
__device__ __forceinline__ void fused_wait()
{
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
}

// this lane's elements of X = sum_m E1[m] Y[m] from a staging slot, in the order of
// operations of the a1 pass of the separable sums. The row loop keeps its branch at M1:
// without it (rows clamped, factors 0) the reads of a whole tile are in flight at once and
// their registers spill (48x48x8, 16 bands: 329 ms against 357).
__device__ __forceinline__ Tile form_tile(const cd *ys, const cd *e1, int M1, int N)
{
    const int c = lane_c(), g = lane_g();
    int off[4];
    bool ok[4];
    double re[4], im[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = g + 4 * r;
        ok[r] = i < N && c < N;
        off[r] = ok[r] ? i * N + c : 0;
        re[r] = im[r] = 0.0;
    }
#pragma unroll
    for (int m = 0; m < kNbFusedMaxM1; ++m) {
        if (m < M1) {
            const cd w = e1[m];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const cd x = ys[m * kFusedPitch + off[r]];
                re[r] = fma(w.x, x.x, fma(-w.y, x.y, re[r]));
                im[r] = fma(w.x, x.y, fma(w.y, x.x, im[r]));
            }
        }
    }
    Tile T;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        T.re[r] = ok[r] ? re[r] : 0.0;
        T.im[r] = ok[r] ? im[r] : 0.0;
    }
    return T;
}

// x of lane j (j uniform over the wave)
__device__ __forceinline__ double lane_value(double x, int j)
{
    const int lo = __builtin_amdgcn_readlane(__double2loint(x), j);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(x), j);
    return __hiloint2double(hi, lo);
}

// HERM: H~ and H are Hermitian to rounding (NbArgs::herm), so a tile's conjugate is its transpose's tile
template <int RK, bool HERM>
__global__ __launch_bounds__(64 * kFusedW) __attribute__((amdgpu_waves_per_eu(RK == 4 ? 2 : 1))) void nb16_step_kernel(
    const NbArgs a, const NbFused f, cd *__restrict__ rho, cd *__restrict__ Ust, double *__restrict__ partials)
{
    extern __shared__ cd step_lds[];
    const int N = a.N, nn = N * N;
    const int c = lane_c(), g = lane_g(), lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int K1 = a.boxK[0], K2 = a.boxK[1], K3 = a.boxK[2], M1 = a.boxM[0];
    // blocks of one column adjacent in dispatch order on one XCD (blocks go round robin
    // over the eight XCDs), so the column's T2 rows are shared through that XCD's L2
    const int nb = static_cast<int>(gridDim.x), b = static_cast<int>(blockIdx.x);
    const int lin = nb % 8 == 0 ? (b % 8) * (nb / 8) + b / 8 : b;
    const int col = lin / f.g1, grp = lin - col * f.g1;
    const int k2 = col / K3, k3 = col - k2 * K3;
    const int k1 = grp * kFusedW + w;
    // a k block of the grid leaves holes in its box (k map -1): those waves only stage
    const int64_t kmap = k1 < K1 ? a.box_kinv[(static_cast<int64_t>(k1) * K2 + k2) * K3 + k3] : -1;
    const bool active = kmap >= 0;
    const int64_t k = active ? kmap : 0;
    cd *buf = step_lds + w * kFusedBuf;
    const double dt = f.dt;
    // this wave's a1 factors E1[k1][m] in LDS (read as broadcasts by every tile formed)
    cd *e1 = fused_slot(step_lds, 2) + w * kNbFusedMaxM1;
    if (lane < M1) e1[lane] = a.boxE[0][static_cast<int64_t>(active ? k1 : 0) * M1 + lane];

    auto form_ht = [&](int slot) {
        const Tile T = form_tile(fused_slot(step_lds, slot), e1, M1, N);
        return HERM ? T : transpose(T, buf);
    };
    Tile R, U, Ut, Y, Acc, Ht, X;
    double lam = 0.0, p = 0.0;
    double pop = 0.0;
    const double wk = active ? a.weight[k] : 0.0;
    const bool need_h = !f.u_valid || !f.lam_valid;
    // staging order: [H(t_n) if needed] [J_x J_y] [J_z H~(t_n)] [H~ H at t + dt/2] [H~ H at t + dt]
    if (need_h) stage_async(a, step_lds, f.t2_prev, 1, nullptr, 0, col, w, lane);
    else stage_async(a, step_lds, f.t2_j, 0, f.t2_j, 1, col, w, lane);
    if (active) {
        R = load_tile(rho + k * nn, N);
        U = load_tile(Ust + k * nn, N, true);
        Ut = transpose(U, buf);
    }
    // ---- sample at t_n
    if (need_h) {  // eigenvectors / energies at t_n from H(t_n)
        fused_wait();
        if (active) {
            const Tile H = form_tile(fused_slot(step_lds, 0), e1, M1, N);
            if (!f.u_valid) eig_refine(H, U, Ut, N, buf);
            lam = col_dot(U, cmm(H, true, U));
        }
        __syncthreads();  // slots read
        stage_async(a, step_lds, f.t2_j, 0, f.t2_j, 1, col, w, lane);
    } else if (active) {
        lam = f.lam[k * 16 + c];
    }
    // rho's band-diagonal part: the populations, the intraband currents Tr(M J) and
    // stage 1's dephasing
    Tile M;
    if (active) {
        M = band_diag(R, U, Ut, p);  // p: populations of U's columns
        int rank = 0;                // rank of column c among the N energies, ties by index
        for (int j = 0; j < N; ++j) {
            const double lj = lane_value(lam, j);
            rank += (lj < lam) || (lj == lam && j < c);
        }
        // lane rank(c) receives column c's population (forward permute; lanes c < N)
        {
            const int dst = (lane < N ? rank : lane) * 4;  // byte address of the receiving lane
            const int lo = __builtin_amdgcn_ds_permute(dst, __double2loint(p));
            const int hi = __builtin_amdgcn_ds_permute(dst, __double2hiint(p));
            if (lane < N) pop = __hiloint2double(hi, lo) * wk;
        }
    }
    // Re Tr(rho J_a) = Re sum_ij conj(rho_ij) J_ij (rho Hermitian; J need not be) and
    // Re Tr(M J_a) = sum_c p_c Re (U^dag J_a U)_cc the same way, elementwise on J's tile:
    // this lane's part of the inter and intra sums, summed over the wave together
    double cur[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    auto current = [&](int ax, const Tile &J) {
        double tot = 0.0, intra = 0.0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            tot += R.re[r] * J.re[r] + R.im[r] * J.im[r];
            intra += M.re[r] * J.re[r] + M.im[r] * J.im[r];
        }
        if (!a.inter_intra) intra = 0.0;
        cur[ax] = (tot - intra) * wk;
        cur[3 + ax] = intra * wk;
    };
    fused_wait();  // [J_x J_y]
    if (active) {
        current(0, form_tile(fused_slot(step_lds, 0), e1, M1, N));
        current(1, form_tile(fused_slot(step_lds, 1), e1, M1, N));
    }
    __syncthreads();  // slots read
    stage_async(a, step_lds, f.t2_j, 2, f.t2_prev, 0, col, w, lane);
    fused_wait();  // [J_z H~]
    if (active) {
        current(2, form_tile(fused_slot(step_lds, 0), e1, M1, N));
        Ht = form_ht(1);
    }
    // ---- the block's sample sums: one partial row, waves added in order
    {
        double *red = reinterpret_cast<double *>(step_lds);  // a transpose buffer per wave
        double *mine = reinterpret_cast<double *>(buf);
        const double v = dev::wave_sum8(cur);
        const int q = dev::sum8_value(lane);
        if (q < 6) mine[q] = v;  // eight lanes hold each
        if (lane < N) mine[6 + lane] = pop;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = g + 4 * r;
            if (i < N && c < N) {
                mine[6 + N + 2 * (i * N + c)] = active ? R.re[r] * wk : 0.0;
                mine[6 + N + 2 * (i * N + c) + 1] = active ? R.im[r] * wk : 0.0;
            }
        }
        __syncthreads();  // slots read, sums written
        stage_async(a, step_lds, f.t2_half, 0, f.t2_half, 1, col, w, lane);
        double *row = partials + (f.step_local * nb + b) * static_cast<int64_t>(a.nv);
        for (int u = threadIdx.x; u < a.nv; u += blockDim.x) {
            double sum = 0.0;
#pragma unroll
            for (int j = 0; j < kFusedW; ++j) sum += red[j * 2 * kFusedBuf + u];
            row[u] = sum;
        }
        __syncthreads();  // sums read: the transpose buffers are free
    }
    // ---- stage 1 at t_n
    if (active) X = stage_derivative_m<HERM>(a, R, Ht, M, buf);
    if constexpr (RK == 4) {
    if (active) {
        axpy_tile(Acc, X, dt / 6.0, R);
        axpy_tile(Y, X, 0.5 * dt, R);
    }
    // ---- stages 2 and 3 at t_n + dt/2
    fused_wait();  // [H~ H at t + dt/2]
    Tile H;
    if (active) {
        Ht = form_ht(0);
        if (a.deph) H = form_tile(fused_slot(step_lds, 1), e1, M1, N);
    }
    __syncthreads();  // slots read
    stage_async(a, step_lds, f.t2_end, 0, f.t2_end, 1, col, w, lane);
    if (active) {
        // (within the step only: the columns' unitarity is left to the refinement at its end)
        if (a.deph) eig_refine(H, U, Ut, N, buf, false, HERM);
        Tile Mh{};
        double dd;
        if (a.deph) Mh = band_diag(Y, U, Ut, dd);
        X = stage_derivative_m<HERM>(a, Y, Ht, Mh, buf);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            Acc.re[r] = fma(dt / 3.0, X.re[r], Acc.re[r]);
            Acc.im[r] = fma(dt / 3.0, X.im[r], Acc.im[r]);
        }
        axpy_tile(Y, X, 0.5 * dt, R);
        if (a.deph) Mh = band_diag(Y, U, Ut, dd);
        X = stage_derivative_m<HERM>(a, Y, Ht, Mh, buf);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            Acc.re[r] = fma(dt / 3.0, X.re[r], Acc.re[r]);
            Acc.im[r] = fma(dt / 3.0, X.im[r], Acc.im[r]);
        }
        axpy_tile(Y, X, dt, R);
    }
    // ---- stage 4 at t_n + dt; eigenvectors and energies for the next sample
    fused_wait();  // [H~ H at t + dt]
    if (active) {
        Ht = form_ht(0);
        H = form_tile(fused_slot(step_lds, 1), e1, M1, N);
        eig_refine(H, U, Ut, N, buf, true, HERM, &lam);
        Tile Me{};
        double dd;
        if (a.deph) Me = band_diag(Y, U, Ut, dd);
        X = stage_derivative_m<HERM>(a, Y, Ht, Me, buf);
        axpy_tile(R, X, dt / 6.0, Acc);
    }
    } else {
        // c = 0, 1/4, 3/8, 12/13, 1, 1/2: the last stage starts its eigenvectors from those at 3/8,
        // the step's own go on to the next sample
        using C = dev::Coef<5>;
        Tile Kd[6], Vm, Vmt, H;
        Kd[0] = X;
        auto input = [&](int st) {
            Tile Yi = R;
#pragma unroll
            for (int j = 0; j < 5; ++j)
                if (j < st && C::a[st][j] != 0.0) axpy_tile(Yi, Kd[j], dt * C::a[st][j], Yi);
            return Yi;
        };
        // H~, H of the time staged last; the slots then take those of src (if given)
        auto pair = [&](const cd *src) {
            fused_wait();
            if (active) {
                Ht = form_ht(0);
                H = form_tile(fused_slot(step_lds, 1), e1, M1, N);
            }
            __syncthreads();  // slots read
            if (src) stage_async(a, step_lds, src, 0, src, 1, col, w, lane);
        };
        auto deriv = [&](int st, const Tile &V, const Tile &Vt) {
            const Tile Yi = input(st);
            Tile Md{};
            double dd;
            if (a.deph) Md = band_diag(Yi, V, Vt, dd);
            Kd[st] = stage_derivative_m<HERM>(a, Yi, Ht, Md, buf);
        };
        const cd *mid = f.t2_half;
#pragma unroll
        for (int st = 1; st <= 3; ++st) {  // 1/4, 3/8, 12/13
            pair(st < 3 ? mid + st * f.mid_stride : f.t2_end);
            if (active) {
                if (a.deph) eig_refine(H, U, Ut, N, buf, true, HERM);
                deriv(st, U, Ut);
                if (st == 2) {
                    Vm = U;
                    Vmt = Ut;
                }
            }
        }
        pair(mid + 3 * f.mid_stride);
        if (active) {
            eig_refine(H, U, Ut, N, buf, true, HERM, &lam);
            deriv(4, U, Ut);
        }
        pair(nullptr);
        if (active) {
            if (a.deph) eig_refine(H, Vm, Vmt, N, buf, true, HERM);
            deriv(5, Vm, Vmt);
#pragma unroll
            for (int j = 0; j < 6; ++j)
                if (C::b[j] != 0.0) axpy_tile(R, Kd[j], dt * C::b[j], R);
        }
    }
    if (active) {
        store_tile(rho + k * nn, R, N);
        store_tile(Ust + k * nn, U, N);
        if (lane < 16) f.lam[k * 16 + c] = lam;
    }
}


}  // namespace

hipError_t nb16_launch_vel_step(const NbArgs &a, const NbVelStep &v, const double2 *P, const double *Eocc,
                                double2 *rho, double *partials, int64_t step_local, hipStream_t s)
{
    if (a.N > 16) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(a.sample_waves));
    if (v.nstage == 4) nb16_vel_step_kernel<4><<<grid, 64, 0, s>>>(a, v, P, Eocc, rho, partials, step_local);
    else if (v.nstage == 6) nb16_vel_step_kernel<6><<<grid, 64, 0, s>>>(a, v, P, Eocc, rho, partials, step_local);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t nb16_launch_rhs(const NbArgs &a, const NbStage &sg, const double2 *mats, double2 *rho, double2 *kbuf,
                           double2 *U, hipStream_t s)
{
    if (a.N > 16) return hipErrorInvalidValue;
    nb16_rhs_kernel<false><<<dim3(static_cast<unsigned>(a.nk)), 64, 0, s>>>(a, sg, sg, mats, rho, kbuf, U);
    return hipGetLastError();
}

hipError_t nb16_launch_rhs_pair(const NbArgs &a, const NbStage &sg, const NbStage &sg2, const double2 *mats,
                                double2 *rho, double2 *kbuf, double2 *U, hipStream_t s)
{
    if (a.N > 16) return hipErrorInvalidValue;
    nb16_rhs_kernel<true><<<dim3(static_cast<unsigned>(a.nk)), 64, 0, s>>>(a, sg, sg2, mats, rho, kbuf, U);
    return hipGetLastError();
}

hipError_t nb16_launch_sample(const NbArgs &a, const double2 *mats, const double2 *rho, double *partials,
                              int64_t step_local, double2 *U, int ureuse, hipStream_t s)
{
    if (a.N > 16) return hipErrorInvalidValue;
    nb16_sample_kernel<<<dim3(static_cast<unsigned>(a.sample_waves)), 64, 0, s>>>(a, mats, rho, partials, step_local,
                                                                                 U, ureuse);
    return hipGetLastError();
}

// dynamic LDS beyond the default limit: raise the kernel's limit, once per device and kernel
hipError_t allow_lds(const void *kernel, size_t lds)
{
    if (lds <= (size_t(64) << 10)) return hipSuccess;
    static std::mutex mu;
    static std::map<std::pair<int, const void *>, size_t> raised;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lk(mu);
    size_t &have = raised[{dev, kernel}];
    if (have < lds) {
        e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        if (e != hipSuccess) return e;
        have = lds;
    }
    return hipSuccess;
}

template <int RK, bool HERM>
static hipError_t launch_step(const NbArgs &a, const NbFused &f, double2 *rho, double2 *U, double *partials,
                              hipStream_t s)
{
    constexpr size_t lds = sizeof(double2) * static_cast<size_t>(
        kFusedW * kFusedBuf + 2 * kNbFusedMaxM1 * kFusedPitch + kFusedW * kNbFusedMaxM1);
    const hipError_t e = allow_lds(reinterpret_cast<const void *>(&nb16_step_kernel<RK, HERM>), lds);
    if (e != hipSuccess) return e;
    nb16_step_kernel<RK, HERM><<<dim3(static_cast<unsigned>(f.nblocks)), 64 * kFusedW, lds, s>>>(a, f, rho, U, partials);
    return hipGetLastError();
}

hipError_t nb16_launch_step(const NbArgs &a, const NbFused &f, int rk_order, double2 *rho, double2 *U, double *partials,
                            hipStream_t s)
{
    if (a.N > 16 || !a.box || a.boxM[0] < 1 || a.boxM[0] > kNbFusedMaxM1 || f.nblocks < 1) return hipErrorInvalidValue;
    if (rk_order == SBE_RK4)
        return a.herm ? launch_step<4, true>(a, f, rho, U, partials, s) : launch_step<4, false>(a, f, rho, U, partials, s);
    if (rk_order == SBE_RK5_FEHLBERG)
        return a.herm ? launch_step<5, true>(a, f, rho, U, partials, s) : launch_step<5, false>(a, f, rho, U, partials, s);
    return hipErrorInvalidValue;
}

}  // namespace sbe
