// tile_small.hpp - complex N x N FP64 matrices for N <= 4 and N <= 8 as
// register tiles of v_mfma_f64_4x4x4_4b_f64, one complex element per lane.
//
// That instruction multiplies four independent 4x4 blocks. Lane l = j + 4 b +
// 16 i holds element (i, j) of block b (D layout, also the B operand's layout;
// the A operand's layout is that of A^T, so it is A^T's tile).
//  * SmallTile<1> (N <= 4): block b is the matrix of k point b of the wave's
//    four; a complex product is four instructions for four k points.
//  * SmallTile<2> (N <= 8): block b = 2 p + q is quadrant (p, q) of one k
//    point's matrix; a complex product is eight instructions, and the operand
//    quadrants move between the blocks with DPP moves of whole 4-lane banks.
// A 16x16 tile (tile16.hpp) spends 16 instructions of 64 cycles on a product
// whatever N is; these take 4 x 16 cycles for four k points and 8 x 16 cycles
// for one, so the matrix pipe is not spent on padding.
// A transpose is a product with the identity (exact), with no LDS traffic.
#pragma once

#include <hip/hip_runtime.h>

#include "tile16.hpp"

namespace sbe {
namespace tile {

template <int Q>
struct SmallTile {
    double re[1], im[1];
};

// x with the lanes of the banks in BANKS replaced by the DPP move CTRL of x
template <int CTRL, int BANKS>
__device__ __forceinline__ double bank_move(double old, double x)
{
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(x), CTRL, 0xf, BANKS, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(x), CTRL, 0xf, BANKS, false);
    return __hiloint2double(hi, lo);
}
template <int CTRL>
__device__ __forceinline__ double lane_move(double x)
{
    return bank_move<CTRL, 0xf>(x, x);
}
constexpr int kXor1 = 0xB1, kXor2 = 0x4E;  // quad_perm [1,0,3,2], [2,3,0,1]
constexpr int kHalfMirror = 0x141;         // lane l <-> l ^ 7
constexpr int kMirror = 0x140;             // lane l <-> l ^ 15
constexpr int kRor4 = 0x124, kRor8 = 0x128;
constexpr int kShl4 = 0x104, kShr4 = 0x114;

// ---- element of this lane: row(r), col()
template <class T>
struct Shape;
template <>
struct Shape<Tile> {
    static constexpr int E = 4, kSize = 16;
    static __device__ __forceinline__ int row(int r) { return lane_g() + 4 * r; }
    static __device__ __forceinline__ int col() { return lane_c(); }
};
template <int Q>
struct Shape<SmallTile<Q>> {
    static constexpr int E = 1, kSize = 4 * Q;
    static __device__ __forceinline__ int row(int)
    {
        const int i = (threadIdx.x >> 4) & 3;
        return Q == 1 ? i : i + 4 * ((threadIdx.x >> 3) & 1);
    }
    static __device__ __forceinline__ int col()
    {
        const int j = threadIdx.x & 3;
        return Q == 1 ? j : j + 4 * ((threadIdx.x >> 2) & 1);
    }
};

__device__ __forceinline__ double mfma4(double a, double b, double c) { return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0); }
template <int NEG>
__device__ __forceinline__ double mfma4n(double a, double b, double c)
{
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, NEG);
}

// C = A B; Aop is A^T's tile (tile16.hpp), CA and CB conjugate the operands
template <bool CA, bool CB>
__device__ __forceinline__ SmallTile<1> cmm_t(const SmallTile<1> &A, const SmallTile<1> &B)
{
    constexpr int kNegRe2 = (CA != CB) ? 0 : 1, kNegIm1 = CB ? 2 : 0, kNegIm2 = CA ? 1 : 0;
    SmallTile<1> C;
    C.re[0] = mfma4(A.re[0], B.re[0], 0.0);
    C.im[0] = mfma4n<kNegIm1>(A.re[0], B.im[0], 0.0);
    C.re[0] = mfma4n<kNegRe2>(A.im[0], B.im[0], C.re[0]);
    C.im[0] = mfma4n<kNegIm2>(A.im[0], B.re[0], C.im[0]);
    return C;
}

// C_pq = A_pp B_pq + A_p(1-p) B_(1-p)q: the first term takes B where it lies, the
// second B's rows of quadrants exchanged (one DPP move per word). A^T's tile holds
// A_pr^T in block (r, p): the A operands are its blocks [0,0,3,3] and [2,2,1,1].
__device__ __forceinline__ double quad_diag(double x) { return bank_move<kShl4, 0x4>(bank_move<kShr4, 0x2>(x, x), x); }

template <bool CA, bool CB>
__device__ __forceinline__ SmallTile<2> cmm_t(const SmallTile<2> &A, const SmallTile<2> &B)
{
    constexpr int kNegRe2 = (CA != CB) ? 0 : 1, kNegIm1 = CB ? 2 : 0, kNegIm2 = CA ? 1 : 0;
    const double ar0 = quad_diag(A.re[0]), ai0 = quad_diag(A.im[0]), br0 = B.re[0], bi0 = B.im[0];
    const double ar1 = quad_diag(lane_move<kRor8>(A.re[0])), ai1 = quad_diag(lane_move<kRor8>(A.im[0]));
    const double br1 = lane_move<kRor8>(B.re[0]), bi1 = lane_move<kRor8>(B.im[0]);
    SmallTile<2> C;
    C.re[0] = mfma4(ar0, br0, 0.0);
    C.im[0] = mfma4n<kNegIm1>(ar0, bi0, 0.0);
    C.re[0] = mfma4n<kNegRe2>(ai0, bi0, C.re[0]);
    C.im[0] = mfma4n<kNegIm2>(ai0, br0, C.im[0]);
    C.re[0] = mfma4(ar1, br1, C.re[0]);
    C.im[0] = mfma4n<kNegIm1>(ar1, bi1, C.im[0]);
    C.re[0] = mfma4n<kNegRe2>(ai1, bi1, C.re[0]);
    C.im[0] = mfma4n<kNegIm2>(ai1, br1, C.im[0]);
    return C;
}

template <int Q>
__device__ __forceinline__ SmallTile<Q> cmm(const SmallTile<Q> &A, bool conjA, const SmallTile<Q> &B, bool conjB = false)
{
    if (conjA) return conjB ? cmm_t<true, true>(A, B) : cmm_t<true, false>(A, B);
    return conjB ? cmm_t<false, true>(A, B) : cmm_t<false, false>(A, B);
}

// X^T: each 4x4 block as the A operand against the identity (1 x + 0 exactly),
// the off-diagonal quadrants (blocks 1 and 2) exchanged
__device__ __forceinline__ double transpose_value(double x, bool quads)
{
    if (quads) x = bank_move<kShr4, 0x4>(bank_move<kShl4, 0x2>(x, x), x);
    const double one = ((threadIdx.x >> 4) & 3) == (threadIdx.x & 3) ? 1.0 : 0.0;
    return mfma4(x, one, 0.0);
}
template <int Q>
__device__ __forceinline__ SmallTile<Q> transpose(const SmallTile<Q> &X, cd *)
{
    SmallTile<Q> T;
    T.re[0] = transpose_value(X.re[0], Q == 2);
    T.im[0] = transpose_value(X.im[0], Q == 2);
    return T;
}

// sum over the rows of this lane's column / over the columns of its row
template <int Q>
__device__ __forceinline__ double col_sum(double x)
{
    x = add32(add16(x));
    if (Q == 2) x += lane_move<kRor8>(x);
    return x;
}
template <int Q>
__device__ __forceinline__ double row_sum(double x)
{
    x += lane_move<kXor1>(x);
    x += lane_move<kXor2>(x);
    if (Q == 2) x += lane_move<kHalfMirror>(x);
    return x;
}

// Re sum_i conj(X_ic) Y_ic for this lane's column c (the diagonal of X^dag Y)
template <int Q>
__device__ __forceinline__ double col_dot(const SmallTile<Q> &X, const SmallTile<Q> &Y)
{
    return col_sum<Q>(X.re[0] * Y.re[0] + X.im[0] * Y.im[0]);
}

// a column value (the same in every row) at this lane's row indices
template <int Q>
__device__ __forceinline__ void col_to_row(const SmallTile<Q> *, double d, double out[1])
{
    out[0] = row_sum<Q>(Shape<SmallTile<Q>>::row(0) == Shape<SmallTile<Q>>::col() ? d : 0.0);
}
__device__ __forceinline__ void col_to_row(const Tile *, double d, double out[4])
{
    const int g = lane_g();
#pragma unroll
    for (int r = 0; r < 4; ++r) out[r] = __shfl(d, 4 * r + g, 64);
}

template <int Q>
__device__ __forceinline__ void diag_bcast(const SmallTile<Q> &W, double lam_r[1], double &lam_c)
{
    const double dv = Shape<SmallTile<Q>>::row(0) == Shape<SmallTile<Q>>::col() ? W.re[0] : 0.0;
    lam_c = col_sum<Q>(dv);
    lam_r[0] = row_sum<Q>(dv);
}

// maximum over the wave, in every lane, without LDS
__device__ __forceinline__ double wave_max_dpp(double v)
{
    double a, b;
    pair32(v, a, b);
    v = fmax(a, b);
    pair16(v, a, b);
    v = fmax(a, b);
    v = fmax(v, lane_move<kMirror>(v));
    v = fmax(v, lane_move<kHalfMirror>(v));
    v = fmax(v, lane_move<kXor2>(v));
    v = fmax(v, lane_move<kXor1>(v));
    return v;
}

}  // namespace tile
}  // namespace sbe
