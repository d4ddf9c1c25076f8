// tile_eig.hpp - the per-k operations of the N-band RK stage and sample on
// register tiles (tile16.hpp, tile_small.hpp): warm-started eigenvectors, the
// band-diagonal part of a matrix, the stage derivative. T is the tile type;
// buf is the wave's LDS transpose buffer (16x16 tiles; unused by small ones).
#pragma once

#include "nband.hpp"
#include "tile_small.hpp"

namespace sbe {
namespace tile {

// U <- U (3I - U^dag U) / 2 (Newton-Schulz: unitarity error e -> ~e^2);
// returns e = max |U^dag U - I| before the step (over the wave)
template <class T>
__device__ __forceinline__ double orthonormalize(T &U, T &Ut, cd *buf)
{
    const int c = Shape<T>::col();
    const T G = cmm(U, true, U);
    T S;
    double e = 0.0;
#pragma unroll
    for (int r = 0; r < Shape<T>::E; ++r) {
        const bool dg = Shape<T>::row(r) == c;
        const double dr = G.re[r] - (dg ? 1.0 : 0.0);
        e = fmax(e, fmax(fabs(dr), fabs(G.im[r])));
        S.re[r] = (dg ? 1.5 : 0.0) - 0.5 * G.re[r];
        S.im[r] = -0.5 * G.im[r];
    }
    U = cmm(Ut, false, S);
    Ut = transpose(U, buf);
    return wave_max_dpp(e);
}

// 1 / (D/2 + s sqrt(D^2/4 + w2)), s = the sign of D (sgn). 16x16 tiles divide and
// take the root; small tiles take the hardware estimates with one Newton step
// each (1e-15 relative): an angle's own error is second order in the eigenvectors.
template <class T>
__device__ __forceinline__ double inv_angle(double D, double w2, double s)
{
    const double x = 0.25 * D * D + w2;
    if (Shape<T>::E > 1) return 1.0 / (0.5 * D + s * sqrt(x));
    double q = __builtin_amdgcn_rsq(x);
    q = q * fma(-0.5 * x * q, q, 1.5);
    const double y = fma(s * x, q, 0.5 * D);
    const double v = __builtin_amdgcn_rcp(y);
    return v * fma(-y, v, 2.0);
}

// Warm-started eigenvectors of the Hermitian part of H (as zheevr, which
// reads one triangle; H from FP16-split sums is Hermitian only to their
// error): U (and its transpose Ut) in, refined U, Ut out.
// small: max|K| below which the last round is U (I + K) (its neglected K^2/2 and the
// next round's O(K^2) residual are the eigenvectors' error); ortho: end with a
// Newton-Schulz step (U unitary to rounding rather than to O(small^2))
// herm: Hin is Hermitian to rounding already (FP64 sums), no symmetrization; lam_out:
// this lane's column of diag(U^dag H U) before the last rotation (the band energies to
// O(max|K|^2), for ranking)
template <class T>
__device__ void eig_refine(const T &Hin, T &U, T &Ut, int N, cd *buf, double small_tol = 1e-8, bool ortho = true,
                           bool herm = false, double *lam_out = nullptr)
{
    constexpr int E = Shape<T>::E;
    const int c = Shape<T>::col();
    T H = Hin;
    if (!herm) {
        const T Ht = transpose(Hin, buf);
#pragma unroll
        for (int r = 0; r < E; ++r) {
            H.re[r] = 0.5 * (Hin.re[r] + Ht.re[r]);
            H.im[r] = 0.5 * (Hin.im[r] - Ht.im[r]);
        }
    }
    T W = cmm(U, true, cmm(H, true, U));  // U^dag (H U)
    double lam_last = 0.0;
    for (int it = 0; it < 30; ++it) {
        double lam_r[E], lam_c;
        diag_bcast(W, lam_r, lam_c);
        lam_last = lam_c;
        T K;
        double kmax = 0.0;
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const int i = Shape<T>::row(r);
            K.re[r] = 0.0;
            K.im[r] = 0.0;
            const double w2 = W.re[r] * W.re[r] + W.im[r] * W.im[r];
            // (small tiles: squares below 1e-280 would leave the root's estimate's range)
            if (i != c && i < N && c < N && w2 > (E > 1 ? 0.0 : 1e-280)) {
                const double D = lam_c - lam_r[r];
                const double s = (D > 0.0 || (D == 0.0 && i < c)) ? 1.0 : -1.0;
                const double inv = inv_angle<T>(D, w2, s);
                K.re[r] = W.re[r] * inv;
                K.im[r] = W.im[r] * inv;
                kmax = fmax(kmax, K.re[r] * K.re[r] + K.im[r] * K.im[r]);  // |K|^2 here, the root once below
            }
        }
        kmax = sqrt(wave_max_dpp(kmax));
        if (kmax == 0.0) break;
        if (kmax > 0.5) {  // far from converged (a cold-like start): damped rotations
            const double f = 0.5 / kmax;
#pragma unroll
            for (int r = 0; r < E; ++r) {
                K.re[r] *= f;
                K.im[r] *= f;
            }
        }
        T V;
        const bool small = kmax < small_tol;
        if (small) {  // I + K: the neglected K^2 / 2 is below 1e-16
#pragma unroll
            for (int r = 0; r < E; ++r) {
                V.re[r] = K.re[r] + (Shape<T>::row(r) == c ? 1.0 : 0.0);
                V.im[r] = K.im[r];
            }
        } else {  // I + K + K^2/2, unitary to |K|^4 / 4; K^T's tile is -conj(K)
            T Kn;
#pragma unroll
            for (int r = 0; r < E; ++r) {
                Kn.re[r] = -K.re[r];
                Kn.im[r] = -K.im[r];
            }
            const T K2 = cmm(Kn, true, K);
#pragma unroll
            for (int r = 0; r < E; ++r) {
                V.re[r] = K.re[r] + 0.5 * K2.re[r] + (Shape<T>::row(r) == c ? 1.0 : 0.0);
                V.im[r] = K.im[r] + 0.5 * K2.im[r];
            }
        }
        U = cmm(Ut, false, V);  // U V
        Ut = transpose(U, buf);
        if (small) break;
        if (kmax > 1e-3) {  // V far from unitary: restore U fully, then W from H itself
            for (int q = 0; q < 8; ++q)
                if (orthonormalize(U, Ut, buf) < 1e-8) break;
            W = cmm(U, true, cmm(H, true, U));
        } else {
            W = cmm(V, true, cmm(W, true, V));  // V^dag (W V)
        }
    }
    if (ortho) orthonormalize(U, Ut, buf);
    if (lam_out) *lam_out = lam_last;
}

// The band-diagonal part of y, U diag(U^dag y U) U^dag, and this lane's column
// of its diagonal d = (U^dag y U)_cc (two products)
template <class T>
__device__ __forceinline__ T band_diag(const T &Y, const T &U, const T &Ut, double &d)
{
    const T G = cmm(Y, true, U);  // y U
    d = col_dot(U, G);            // (U^dag y U)_cc
    double dr[Shape<T>::E];
    col_to_row(&U, d, dr);
    T Ud;  // (U diag(d))^T's tile: row i of U^T times d_i
#pragma unroll
    for (int r = 0; r < Shape<T>::E; ++r) {
        Ud.re[r] = Ut.re[r] * dr[r];
        Ud.im[r] = Ut.im[r] * dr[r];
    }
    return cmm(Ud, false, Ut, true);  // U diag(d) U^dag (B = U^dag: tile conj(U^T))
}

// The stage derivative at y given H~^T's tile (HERM: H~'s own tile, H~ Hermitian, so
// that H~^T's tile is its conjugate) and (dephasing on) y's band-diagonal part M:
// -i(H~ y - (H~ y)^dag) - g2 y - (g1 - g2) M.
template <bool HERM, class T>
__device__ __forceinline__ T stage_derivative_m(const NbArgs &a, const T &Y, const T &HtT, const T &M, cd *buf)
{
    const T P = cmm(HtT, HERM, Y);  // H~ y
    const T Pt = transpose(P, buf);
    T X;  // -i (P - P^dag)
#pragma unroll
    for (int r = 0; r < Shape<T>::E; ++r) {
        const double dr = P.re[r] - Pt.re[r], di = P.im[r] + Pt.im[r];
        X.re[r] = di;
        X.im[r] = -dr;
    }
    if (a.deph) {
        const double g2 = a.gam2, g12 = a.gam1 - a.gam2;
#pragma unroll
        for (int r = 0; r < Shape<T>::E; ++r) {
            X.re[r] -= g2 * Y.re[r] + g12 * M.re[r];
            X.im[r] -= g2 * Y.im[r] + g12 * M.im[r];
        }
    }
    return X;
}

// The same with U, U^T given (M formed here when dephasing)
template <class T>
__device__ __forceinline__ T stage_derivative(const NbArgs &a, const T &Y, const T &HtT, const T &U, const T &Ut, cd *buf)
{
    T M{};
    if (a.deph) {
        double d;
        M = band_diag(Y, U, Ut, d);
    }
    return stage_derivative_m<false>(a, Y, HtT, M, buf);
}

// Y = B + s X
template <class T>
__device__ __forceinline__ void axpy_tile(T &Y, const T &X, double s, const T &B)
{
#pragma unroll
    for (int r = 0; r < Shape<T>::E; ++r) {
        Y.re[r] = fma(s, X.re[r], B.re[r]);
        Y.im[r] = fma(s, X.im[r], B.im[r]);
    }
}

}  // namespace tile
}  // namespace sbe
