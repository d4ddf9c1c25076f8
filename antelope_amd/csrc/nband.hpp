// nband.hpp - N-band (Wannier) path: kernel arguments and launchers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace sbe {

// Matrix kinds an evaluation of the Fourier sums can produce.
enum : int { kMatHtilde = 0, kMatH0 = 1, kMatJx = 2, kMatJy = 3, kMatJz = 4 };

constexpr int kNbMaxBands = 32;

struct NbArgs {
    int N;                 // bands
    int nr;                // lattice vectors R
    int nval;
    int fermi;             // Fermi-Dirac initial occupations
    double fermi_energy;
    int inter_intra;
    int deph;              // any dephasing on (T1 or T2)
    double gam1, gam2;     // 1/T1, 1/T2 (0 = off)
    int64_t nk, nk_stride;
    int nv;                // values per sample row: 6 + N + 2 N^2
    int sample_waves;      // rows of the per-step partial sums
    const double *kpts;    // [nk_stride][3]
    const double *weight;  // [nk_stride]
    const double *rcart;   // [nr][3] cartesian R (bohr)
    const double *rweight; // [nr] 1/degeneracy
    const double2 *ham;    // [nr][N][N]
    const double2 *pos;    // [nr][3][N][N]
    int herm;              // ham and pos are Hermitian, X(-R) = X(R)^dag: H and H~ are too (to rounding)
    // FP16-split Fourier sums (SBE_PREC_SPLIT16): halves as raw 16-bit words
    int split16;
    int nr_pad;            // nr rounded up to the MFMA K (32)
    int64_t bcols;         // columns of the B planes (4 N^2 rounded up to 64)
    const uint16_t *p16;   // e^{ik.R}: planes [re_hi, re_lo, im_hi, im_lo][nk_stride][nr_pad]
    uint16_t *b16;         // B of one evaluation: planes [re_hi, re_lo, im_hi, im_lo][bcols][nr_pad]
    double2 *b64;          // FP64 form: B of one evaluation [nr_pad][bcols]
    double hmax, pmax, rmax;  // max |H(R)|, max |r(R)|, max |R_a| (scales of B)
    int velocity;          // VelocityHamiltonian gauge (band basis at k)
    // analytic tight-binding class (SBE_MODEL_WILSON_MASS ... SBE_MODEL_TMDC):
    // H and J come from analytic.hpp instead of the Fourier sums; 0 = Wannier
    int model_kind;
    double mparams[24];
    int tile16;            // N <= 16: stage and sample kernels with the matrices in MFMA registers
    // Separable Fourier sums (FP64 form, product k grids): R = n1 a1 + n2 a2 + n3 a3 on the
    // lattice box lo_i <= n_i < lo_i + M_i, theta_i = k.a_i taking K_i values per axis
    int box;
    int boxM[3], boxK[3];
    const int32_t *box_r;     // [M1][M2][M3] index into the R list, -1 where the box has no R
    const double2 *boxE[3];   // [K_i][M_i] e^{i n theta}, n = lo_i + m
    const int32_t *box_kinv;  // [K1][K2][K3] k index of this block, -1 where absent
    double2 *box_b;           // B on the box [M1 M2 M3][bcols]
    double2 *box_t1;          // first pass  [M1][M2][K3][bcols]
    double2 *box_t2;          // second pass [M1][K2][K3][bcols]
    // isDipoleZero (Wannier90.h:180-194): the sums take the phase of R + tau_n - tau_m
    // (tau_n = Re <0n|r|0n>) and no E.D term
    int dzero;
    double tau[kNbMaxBands][3];
};

// One evaluation of the Fourier sums at k + A(t) with field E(t).
struct NbEval {
    double A[3], E[3];
    int nmat;
    int mats[5];
};

// One RK stage: coefficients already multiplied by dt.
struct NbStage {
    int stage, nstage, last;
    int ureuse;   // the stored eigenvectors belong to this stage's H (same time)
    double a[8];  // dt a_{stage,j}
    double b[8];  // dt b_j (used when last)
};

// One whole RK4 or RK5 step of the LengthWannier gauge for N <= 16 on a product k grid
// with separable Fourier sums (nb16_step_kernel): the last pass of the sums
// (along a1) runs inside the step kernel, from the second pass's output of
// each evaluation time, so the matrices never reach HBM. t2_* are that output,
// [M1][K2][K3][bcols] with the evaluation's matrices side by side in the columns.
constexpr int kNbFusedWaves = 4;  // k points along a1 per block (one wave each)
constexpr int kNbFusedMaxM1 = 7;  // lattice vectors along a1 staged in LDS
struct NbFused {
    const double2 *t2_prev;  // H~, H at t_n
    const double2 *t2_j;     // J_x, J_y, J_z at t_n
    const double2 *t2_half;  // H~, H at t_n + dt/2 (RK5: at c = 1/4, 3/8, 12/13, 1/2, mid_stride apart)
    int64_t mid_stride;
    const double2 *t2_end;   // H~, H at t_n + dt
    double *lam;             // [nk_stride][16] band energies at the stored eigenvectors' time
    int u_valid;             // the stored eigenvectors belong to H(t_n)
    int lam_valid;           // lam belongs to them
    double dt;
    int64_t step_local;      // row block of the partial sums
    int g1;                  // blocks per (k2, k3) column: ceil(K1 / kNbFusedWaves)
    int nblocks;             // g1 K2 K3: partial rows per step
};
// dynamic LDS beyond the default limit: raises the kernel's limit, once per device and kernel (nband16.hip)
hipError_t allow_lds(const void *kernel, size_t lds);
hipError_t nb16_launch_step(const NbArgs &a, const NbFused &f, int rk_order, double2 *rho, double2 *U, double *partials,
                            hipStream_t s);
// the separable sums of one evaluation up to the second pass: t2 [M1][K2][K3][bcols]
hipError_t nb_launch_box_t2(const NbArgs &a, const NbEval &ev, double2 *t2, hipStream_t s);
// the same for nev <= 4 evaluations in three launches, each with its own scratch b
// [cells][bcols], t1 [M1][M2][K3][bcols] and output t2
hipError_t nb_launch_box_t2_multi(const NbArgs &a, int nev, const NbEval *evs, double2 *const *b, double2 *const *t1,
                                  double2 *const *t2, hipStream_t s);
// The separable sums up to the second pass for a run of RK steps [s0, s0 + ns) in three
// launches (bform, the passes along a3 and a2), evaluation e = (mids + 2) sl + typ: typ 0 J at
// t_n into tj + sl t2_stride, typ 1..mids H~ H at the tableau's times between t_n and t_n + dt
// (RK4: dt/2; RK5: dt/4, 3dt/8, 12dt/13, dt/2) into th + (mids sl + typ - 1) t2_stride, the last
// H~ H at t_n + dt into ring + (step mod nring) t2_stride (the pair of the step before s0 stays
// in the ring when nring > ns); per evaluation scratch b + e b_stride, t1 + e t1_stride. laser:
// [nt][mids + 2][6], A and E at t_n, the times between and t_n + dt.
struct NbBoxSteps {
    const double *laser;
    int64_t s0;
    int ns, nring, mids;
    double2 *b, *t1, *tj, *th, *ring;
    int64_t b_stride, t1_stride, t2_stride;  // elements
};
hipError_t nb_launch_box_steps(const NbArgs &a, const NbBoxSteps &d, hipStream_t s);
// The same with the pass along a1 as well, each evaluation's matrices into out[e]
// ([nmat][nk_stride][N][N]; the padding k points are not written)
hipError_t nb_launch_box_mats_multi(const NbArgs &a, int nev, const NbEval *evs, double2 *const *b, double2 *const *t1,
                                    double2 *const *t2, double2 *const *out, hipStream_t s);

// Up to four evaluations of the dense sums in one launch (Wannier models with at most
// kNbDenseMultiMaxR lattice vectors; P = e^{ik.R} [nk_stride][nr]), each into out[e]
// ([nmat][nk_stride][N][N]; the padding k points are not written)
constexpr int kNbDenseMultiMaxR = 32;
hipError_t nb_launch_dense_multi(const NbArgs &a, int nev, const NbEval *evs, const double2 *P, double2 *const *out,
                                 hipStream_t s);

// The matrices of steps [s0, s0 + ns) of the RK4 LengthWannier gauge in one launch
// (the dense sums, the same R lists): J at t_n into j [ns][3][slot], H~ (and H with
// dephasing) at t_n + dt/2 into half [ns][2][slot], H~ and H at t_n + dt into the ring
// [nring][2][slot] at step mod nring (the pair of the step before s0 is kept there when
// nring > ns). laser: [nt][3][6], A and E at t_n, t_n + dt/2, t_n + dt.
struct NbDenseSteps {
    const double *laser;
    int64_t s0;
    int ns, nring, deph;
    int64_t slot;  // nk_stride N^2
    double2 *j, *half, *ring;
};
hipError_t nb_launch_dense_steps(const NbArgs &a, const NbDenseSteps &d, const double2 *P, hipStream_t s);

// One whole RK4 step of the LengthWannier gauge for 16 < N <= 32 (nb32_step_kernel):
// four waves per k point, each one 16x16 quadrant of every matrix; the matrices of the
// step's times from the Fourier-sum outputs ([nk_stride][N][N] each, j: [3][nk_stride][N][N]).
constexpr int kNb32MaxBlocks = 256;  // blocks of the N <= 32 step: one per CU, k points walked in turn
struct NbStep32 {
    const double2 *ht_prev, *h_prev;  // H~, H at t_n (h_prev read when u_valid or lam_valid is 0)
    const double2 *j;                 // J_x, J_y, J_z at t_n
    const double2 *ht_half, *h_half;  // at t_n + dt/2
    const double2 *ht_end, *h_end;    // at t_n + dt
    double *lam;                      // [nk_stride][32] band energies at the stored eigenvectors' time
    int u_valid, lam_valid;
    double dt;
    int64_t step_local;
};
hipError_t nb32_launch_step(const NbArgs &a, const NbStep32 &f, int nblocks, double2 *rho, double2 *U, double *partials,
                            hipStream_t s);

// Time-fused VelocityHamiltonian steps for N <= 16, RK4 or RK5 (nb_vel_fused_kernel):
// steps [s0, s1) in one launch, one partial row per block and step.
struct NbVelFused {
    const double *A;  // [nt][stages][3]: A(t_n + c_s dt)
    int64_t s0, s1;
    double dt;
    int nblocks;      // partial rows per step: vel_fused_blocks for N <= 16, nk above
    int waves;        // N <= 16: vel_fused_waves
};
int vel_fused_waves(int N, int64_t nk);
int64_t vel_fused_blocks(int N, int64_t nk);
hipError_t nb_launch_vel_fused(const NbArgs &a, const NbVelFused &f, int rk_order, const double2 *P, const double *Eocc,
                               double2 *rho, double *partials, hipStream_t s);
// the same for 16 < N <= 32, RK4: one block of four waves per k point (nblocks = nk)
constexpr int64_t kNb32VelMaxK = 1024;
hipError_t nb32_launch_vel_fused(const NbArgs &a, const NbVelFused &f, const double2 *P, const double *Eocc,
                                 double2 *rho, double *partials, hipStream_t s);

// Time-fused LengthWannier steps of the analytic classes with N <= 8
// (nb_evolve_kernel): steps [s0, s1) in one launch, one partial row per block and step.
constexpr int kEvolveMaxTerms = 9;
struct EvolveTerms {  // analytic_terms.hpp
    int T;
    double vec[kEvolveMaxTerms][3], grad[kEvolveMaxTerms][3];
};
struct NbEvolve {
    EvolveTerms terms;
    const double2 *coef;   // [1 + 2 T + 1][N][N]: m0, (p_t, q_t) per term, the current's element factors
    const double *table;   // [s1 - s0 + 1][row]: cos / sin(A.v_t) at the distinct times of step s0 on
    int jz;                // any z current
    int64_t s0, s1;
    double dt;
    int nblocks;
    double *lam;           // [nk_stride][8] band energies at the stored eigenvectors' time
    int lam_valid;         // the stored eigenvectors and lam belong to t_{s0}
};
// distinct stage times of a step (t_n first, t_n + dt being the next step's), the padded
// number of terms of the kernels, doubles per table row and blocks of a launch
inline int evolve_times(int rk_order) { return rk_order == 4 ? 2 : 5; }
inline int evolve_padded_terms(int T) { return T <= 3 ? 3 : (T <= 6 ? 6 : 9); }
inline int evolve_row_len(int rk_order, int T) { return (6 + 2 * evolve_times(rk_order)) * evolve_padded_terms(T); }
int evolve_blocks(int N, int64_t nk);
// the table of rows n in [step0, step0 + nsteps) of the laser at its times t_n + c_u dt, or (A
// not null) from A of the whole pulse at them, [n][times][3]
struct TableArgs;
hipError_t launch_evolve_table(const TableArgs &laser, const double *A, const EvolveTerms &t, int rk_order, double *tab, hipStream_t s);
hipError_t launch_evolve(const NbArgs &a, const NbEvolve &e, int rk_order, double2 *rho, double2 *U, double *partials,
                         hipStream_t s);

// The same for Wannier models with N <= 8 on the separable Fourier sums: steps [s0, s0 + ns),
// whose second-pass outputs are in place (NbBoxSteps), one partial row per block and step.
struct NbBoxRun {
    const double2 *tj, *th, *ring;
    int64_t t2_stride;
    int nring, ns;
    int64_t s0, row0;      // row0: the first step's row of the partial sums
    int jz;                // any z current
    double dt;
    int nblocks;
    double *lam;           // [nk_stride][16]
    int lam_valid;
};
int box_evolve_blocks(int N, const int K[3]);
hipError_t launch_box_evolve(const NbArgs &a, const NbBoxRun &e, int rk_order, double2 *rho, double2 *U, double *partials,
                             hipStream_t s);

// One time step of the VelocityHamiltonian gauge: A at the stage times and
// the tableau (coefficients already multiplied by dt).
struct NbVelStep {
    int nstage;
    double A[7][3];  // A(t_n + c_i dt), i < nstage
    double a[7][7];  // dt a_ij
    double b[7];     // dt b_i
};

size_t nb_lds_bytes(int N);
// LDS of the velocity step kernel; p_lds keeps the k point's pMatrix in LDS
size_t nb_vel_lds_bytes(int N, int nstage, bool p_lds);
// per k: U, E and pMatrix_a = U^dag J_a U from mats {H, J_x, J_y, J_z} at k;
// rho = diag(occupations). P [3][nk_stride][N][N], Eocc [nk_stride][2N] (E, occ)
hipError_t nb_launch_vel_init(const NbArgs &a, const double2 *mats, double2 *P, double *Eocc, double2 *U,
                              double2 *rho, hipStream_t s);
// U^dag rho U per k with U = eig(H) (H: [nk_stride][N][N]), the phase rule of the velocity set-up
hipError_t nb_launch_band_export(const NbArgs &a, const double2 *H, const double2 *rho, double2 *out, hipStream_t s);
// sample at t_n, then one RK step, for every k (partials row step_local)
hipError_t nb_launch_vel_step(const NbArgs &a, const NbVelStep &v, const double2 *P, const double *Eocc, double2 *rho,
                              double *partials, int64_t step_local, bool p_lds, hipStream_t s);
hipError_t nb_launch_phase(const NbArgs &a, double2 *P, hipStream_t s);
// SPLIT16: e^{ik.R} split into FP16 hi/lo planes once per context
hipError_t nb_launch_psplit(const NbArgs &a, const double2 *P, uint16_t *p16, hipStream_t s);
hipError_t nb_launch_fourier(const NbArgs &a, const NbEval &ev, const double2 *P, double2 *out, hipStream_t s);
// analytic classes: the same matrices [mat][nk_stride][N][N] at k + A (analytic.hip)
hipError_t nb_launch_model(const NbArgs &a, const NbEval &ev, double2 *out, hipStream_t s);
hipError_t nb_launch_init(const NbArgs &a, const double2 *H0, double2 *rho, double2 *U, hipStream_t s);
hipError_t nb_launch_sample(const NbArgs &a, const double2 *mats, const double2 *rho, double *partials,
                            int64_t step_local, double2 *U, int ureuse, hipStream_t s);
hipError_t nb_launch_rhs(const NbArgs &a, const NbStage &sg, const double2 *mats, double2 *rho, double2 *kbuf,
                         double2 *U, hipStream_t s);
// N <= 16 forms of the two above (nband16.hip)
hipError_t nb16_launch_rhs(const NbArgs &a, const NbStage &sg, const double2 *mats, double2 *rho, double2 *kbuf,
                           double2 *U, hipStream_t s);
hipError_t nb16_launch_sample(const NbArgs &a, const double2 *mats, const double2 *rho, double *partials,
                              int64_t step_local, double2 *U, int ureuse, hipStream_t s);
// two consecutive stages at the same time in one launch (RK4's c = 1/2, 1/2)
hipError_t nb16_launch_rhs_pair(const NbArgs &a, const NbStage &sg, const NbStage &sg2, const double2 *mats,
                                double2 *rho, double2 *kbuf, double2 *U, hipStream_t s);
hipError_t nb16_launch_vel_step(const NbArgs &a, const NbVelStep &v, const double2 *P, const double *Eocc,
                                double2 *rho, double *partials, int64_t step_local, hipStream_t s);

}  // namespace sbe
