// Device routine shared by the panel kernel and the batched fit: Cholesky
// factor and inverse of one 64x64 block held in LDS by one 256-thread
// workgroup. Header-only so each kernel file inlines it.
#pragma once

#include <hip/hip_runtime.h>

namespace gpamd::k
{
namespace b64
{

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

// 1/sqrt(d) from the hardware estimate y (relative error below 2^-22) and
// e = 1 - d y^2: y (1 + e/2 + 3/8 e^2), whose error is of the order of e^3.
// A non-positive or NaN d gives NaN or infinity.
__device__ __forceinline__ double rsqrt_correct(double y, double e) { return fma(e * y, fma(e, 0.375, 0.5), y); }

__device__ __forceinline__ double rsqrt_refined(double d)
{
    const double y = __builtin_amdgcn_rsq(d);
    return rsqrt_correct(y, fma(-(d * y), y, 1.0));
}

// Lane L of each 16-lane row of the wavefront, on every lane of that row
// (one v_mov_b64_dpp row_newbcast).
template <int L>
__device__ __forceinline__ double row_bcast(double v)
{
    static_assert(L >= 0 && L < 16, "a row has 16 lanes");
    constexpr int ROW_NEWBCAST = 0x150;
    const long long b = __double_as_longlong(v);
    return __longlong_as_double(__builtin_amdgcn_update_dpp(0ll, b, ROW_NEWBCAST + L, 0xf, 0xf, true));
}

// Columns C .. C + COUNT - 1 of the rows d and r minus dj, rj (column J,
// scaled) times dj's entries in those columns: v_fmac_f64 takes the row
// broadcast as its operand, so a column costs two instructions. The wait is
// the one a DPP operand needs after a vector write of its register; the
// compiler does not add it for operands of inline assembly.
template <int C, int COUNT>
__device__ __forceinline__ void eliminate_columns(double (&d)[16], double (&r)[16], double dj, double rj)
{
    if constexpr (COUNT == 4)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %0, -%8, %8 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, -%8, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %2, -%8, %8 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %3, -%8, %9 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %4, -%8, %8 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %5, -%8, %9 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %6, -%8, %8 row_newbcast:%13 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %7, -%8, %9 row_newbcast:%13 row_mask:0xf bank_mask:0xf"
            : "+v"(d[C]), "+v"(r[C]), "+v"(d[C + 1]), "+v"(r[C + 1]), "+v"(d[C + 2]), "+v"(r[C + 2]), "+v"(d[C + 3]), "+v"(r[C + 3])
            : "v"(dj), "v"(rj), "n"(C), "n"(C + 1), "n"(C + 2), "n"(C + 3));
    else if constexpr (COUNT >= 1)
    {
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %0, -%2, %2 row_newbcast:%4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, -%2, %3 row_newbcast:%4 row_mask:0xf bank_mask:0xf"
            : "+v"(d[C]), "+v"(r[C])
            : "v"(dj), "v"(rj), "n"(C));
        eliminate_columns<C + 1, COUNT - 1>(d, r, dj, rj);
    }
}

// The next (up to) four columns from C on, kept where they stand.
template <int C>
__device__ __forceinline__ void eliminate_next(double (&d)[16], double (&r)[16], double dj, double rj)
{
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (C < 16)
        eliminate_columns<C, (16 - C < 4 ? 16 - C : 4)>(d, r, dj, rj);
    __builtin_amdgcn_sched_barrier(0);
}

// Pivots J .. 15 of a 16x16 diagonal block. Lane l holds row l % 16 of the
// block in d (every 16-lane row of the wavefront a copy, so a pivot column's
// entries reach all lanes by row broadcasts) and one further row in r, whose
// panel solve runs in the same pass. inv: 1/sqrt of pivot J; pivot: lane
// l's pivot l % 16. The next pivot's 1/sqrt is a chain of dependent
// operations: it starts as soon as its column is updated, and the other
// columns' updates are issued in its waits.
template <int J>
__device__ __forceinline__ void eliminate(double (&d)[16], double (&r)[16], double inv, double &pivot, int l16)
{
    d[J] *= inv;
    r[J] *= inv;
    if constexpr (J < 15)
    {
        const double dj = d[J], rj = r[J];
        eliminate_columns<J + 1, 1>(d, r, dj, rj);
        __builtin_amdgcn_sched_barrier(0);
        const double djj = row_bcast<J + 1>(d[J + 1]);
        double y = __builtin_amdgcn_rsq(djj);
        eliminate_next<J + 2>(d, r, dj, rj);
        const double t = djj * y;
        eliminate_next<J + 6>(d, r, dj, rj);
        const double e = fma(-t, y, 1.0);
        eliminate_next<J + 10>(d, r, dj, rj);
        y = rsqrt_correct(y, e);
        eliminate_next<J + 14>(d, r, dj, rj);
        pivot = l16 == J + 1 ? djj : pivot;
        eliminate<J + 1>(d, r, y, pivot, l16);
    }
}

// 16x16 tile (tr, tc) of D from row and column `base` on, minus
// D[.., o .. o + 15] D[.., o .. o + 15]^T. A diagonal tile's strict upper
// triangle is scratch.
template <int S>
__device__ __forceinline__ void rank16(double (*D)[S], int base, int tr, int tc, int o, int lm, int lk)
{
    // accumulator: lane holds column lm, rows lk + 4 e
    double c[4];
#pragma unroll
    for (int e = 0; e < 4; e++)
        c[e] = D[base + tr * 16 + lk + 4 * e][base + tc * 16 + lm];
    v4d acc = { 0.0, 0.0, 0.0, 0.0 };
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(D[base + tr * 16 + lm][o + k0 + lk], D[base + tc * 16 + lm][o + k0 + lk], acc, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; e++)
        D[base + tr * 16 + lk + 4 * e][base + tc * 16 + lm] = c[e] - acc[e];
}

// s += L_it W_tj over 16x16 blocks.
template <int S>
__device__ __forceinline__ void inverse_sum(double (*D)[S], double (*W)[S], int i, int t, int j, int lm, int lk, v4d &s)
{
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 4)
        s = __builtin_amdgcn_mfma_f64_16x16x4f64(D[i * 16 + lm][t * 16 + k0 + lk], W[t * 16 + k0 + lk][j * 16 + lm], s, 0, 0, 0);
}

// W_ij = -W_ii s: the B operand of k-step 4e (row 4e + lk, column lm) is
// exactly this lane's accumulator entry e.
template <int S>
__device__ __forceinline__ void inverse_block(double (*W)[S], int i, int j, int lm, int lk, const v4d &s)
{
    v4d acc = { 0.0, 0.0, 0.0, 0.0 };
#pragma unroll
    for (int e = 0; e < 4; e++)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(W[i * 16 + lm][i * 16 + 4 * e + lk], s[e], acc, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; e++)
        W[i * 16 + lk + 4 * e][j * 16 + lm] = -acc[e];
}

}  // namespace b64

// Cholesky factor and inverse of one 64x64 block held in LDS, by one
// workgroup of 256 threads, in four 16-wide steps. The chain of 64 pivots
// bounds it, so everything else runs beside the chain:
//  * wavefront 0 eliminates a step's 16 pivots in registers, one matrix row
//    per lane: the diagonal block's rows (a copy in each 16-lane row of the
//    wavefront), and in lanes 16 .. 63 the rows below it, which leave the
//    pass solved, in lanes 0 .. 15 the identity rows e_s, which leave it as
//    e_s L^-T, column s of the diagonal block's inverse. A pivot's reciprocal
//    square root is a refined hardware estimate;
//  * after the step the four wavefronts update the next step's 16 columns on
//    the matrix cores, one 16x16 tile each;
//  * wavefronts 1 .. 3 apply the rest of the update, and form the inverse's
//    off-diagonal blocks W_ij = -W_ii sum_{t=j}^{i-1} L_it W_tj (two chained
//    matrix-core products whose intermediate never leaves registers), row i
//    while wavefront 0 is at step i + 1; of the last row only the product
//    with W_33 is left for the end.
// Measured on MI355X, one workgroup alone on its CU: 16 700 cycles (33 000
// when readlane broadcasts fed one register set and the inverse followed the
// factor), of which 2 500 per step are the elimination (156 per pivot: its 36
// instructions at 4 cycles each, the chain hidden in them).
// D and W are 16-byte aligned, with an even row stride S. On exit D holds L in its lower triangle (the strict upper triangle is
// scratch), W holds L^-1 on and below the diagonal (exact zeros above it
// inside the 16x16 diagonal blocks, the 16x16 blocks above those untouched).
// A non-positive pivot stores the smallest failing global column in *info.
template <int S>
__device__ __forceinline__ void factor_block64(double (*D)[S], double (*W)[S], int *info, int col0)
{
    using b64::d2;
    using b64::v4d;
    constexpr int NB = 64;
    static_assert(S >= NB && S % 2 == 0, "rows of pairs");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lm = lane & 15, lk = lane >> 4;
    v4d s3 = { 0.0, 0.0, 0.0, 0.0 };  // wavefront j + 1: sum_{t=j}^{2} L_3t W_tj
#pragma unroll
    for (int kb = 0; kb < 4; kb++)
    {
        const int o = kb * 16;
        if (wave == 0)
        {
            const bool below = lane >= 16 && o + lane < NB;
            double d[16], r[16];
#pragma unroll
            for (int t = 0; t < 16; t += 2)
            {
                const d2 v = *reinterpret_cast<const d2 *>(&D[o + lm][o + t]);
                const d2 w = *reinterpret_cast<const d2 *>(&D[below ? o + lane : o][o + t]);
#pragma unroll
                for (int q = 0; q < 2; q++)
                {
                    d[t + q] = v[q];
                    r[t + q] = below ? w[q] : (lane == t + q ? 1.0 : 0.0);
                }
            }
            double pivot = b64::row_bcast<0>(d[0]);
            b64::eliminate<0>(d, r, b64::rsqrt_refined(pivot), pivot, lm);
            if (lane < 16 || below)
            {
#pragma unroll
                for (int t = 0; t < 16; t += 2)
                    *reinterpret_cast<d2 *>(&D[o + lane][o + t]) = lane < 16 ? d2{ d[t], d[t + 1] } : d2{ r[t], r[t + 1] };
            }
            if (lane < 16)
            {
                // zeros above the inverse's diagonal come out exact: e_s has
                // none before column s
#pragma unroll
                for (int t = 0; t < 16; t++)
                    W[o + t][o + lane] = r[t];
                if (!(pivot > 0.0))
                    atomicMin(info, col0 + o + lane);
            }
        }
        else
        {
            const int j = wave - 1;
            if (kb == 1)  // step 0: the tiles beyond column block 1
                b64::rank16(D, 16, j == 0 ? 1 : 2, j == 2 ? 2 : 1, 0, lm, lk);
            if (kb == 2 && j == 2)  // step 1: the last tile
                b64::rank16(D, 32, 1, 1, 16, lm, lk);
            if (kb >= 2 && j < kb - 1)  // the inverse's row kb - 1
            {
                v4d s = { 0.0, 0.0, 0.0, 0.0 };
                for (int t = j; t < kb - 1; t++)
                    b64::inverse_sum(D, W, kb - 1, t, j, lm, lk, s);
                b64::inverse_block(W, kb - 1, j, lm, lk, s);
                // the lanes read each other's entries of that block next
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
            if (kb == 3)
                for (int t = j; t < 3; t++)
                    b64::inverse_sum(D, W, 3, t, j, lm, lk, s3);
        }
        __syncthreads();
        if (kb < 3)
        {
            if (wave < 3 - kb)
                b64::rank16(D, o + 16, wave, 0, o, lm, lk);
            __syncthreads();
        }
    }
    if (wave > 0)
        b64::inverse_block(W, 3, wave - 1, lm, lk, s3);
    __syncthreads();
}

}  // namespace gpamd::k
