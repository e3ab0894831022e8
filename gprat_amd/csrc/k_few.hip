// X L^-T for few rows X (a handful of test points' rows of K*), on FP64 matrix
// cores straight from global memory.
//
// Stepping through L in the factorisation's panels: V_J = X_J W_J^T with the
// panel's kept inverse, then X[:, later] -= V_J L[later, J]^T. With 16 to 64
// rows the step's work is reading L's column panel once, so a 16 x 16 output
// tile per workgroup and its K range split over eight wavefronts keep enough
// loads in flight; both operands of the update are contiguous in k, so a lane
// takes four consecutive k of its row as two 16-byte loads (the four matrix
// instructions of a 16-deep group take k in the order 4 (lane / 16) + t) and
// no LDS stage is needed. The eight partial tiles are added in a fixed order.
#include <algorithm>

#include "kernels.hpp"

namespace gpamd::k
{
namespace
{

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

constexpr int WAVES = 8;
constexpr int THREADS = 64 * WAVES;
constexpr int FEW = 16;  // edge of an output tile

struct Args
{
    const double *V;  // left operand: rows contiguous in k
    long ldv;
    const double *M;  // right operand: rows contiguous in k (L), or k-major (the inverse)
    long ldm;
    const double *C;  // subtracted from (update) or null
    double *out;
    long ldo;
    int K;
};

// Output tile (rows 16 C blockIdx.y .., columns 16 blockIdx.x ..): CT tiles of
// 16 rows that share the right operand. KMAJOR: M(column, k) at [k ldm +
// column], lower triangular (k ends with the tile); else at [column ldm + k].
template <int CT, bool KMAJOR>
__global__ __launch_bounds__(THREADS) void k_few_rows(Args a)
{
    __shared__ double part[WAVES][CT][4][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lm = lane & 15, lk = lane >> 4;
    const long col = static_cast<long>(blockIdx.x) * FEW;
    const long row = static_cast<long>(blockIdx.y) * FEW * CT;
    const int K = KMAJOR ? min(a.K, static_cast<int>(col) + FEW) : a.K;
    const int groups = K / 16, per = (groups + WAVES - 1) / WAVES;
    const int g0 = min(groups, w * per), g1 = min(groups, g0 + per);
    v4d acc[CT];
#pragma unroll
    for (int c = 0; c < CT; c++)
        acc[c] = v4d{ 0.0, 0.0, 0.0, 0.0 };
    const double *v = a.V + (row + lm) * a.ldv + 4 * lk;
    const double *m = KMAJOR ? a.M + static_cast<long>(4 * lk) * a.ldm + col + lm : a.M + (col + lm) * a.ldm + 4 * lk;
#pragma unroll 4
    for (int g = g0; g < g1; g++)
    {
        double b[4];
        if constexpr (KMAJOR)
        {
#pragma unroll
            for (int t = 0; t < 4; t++)
                b[t] = m[static_cast<long>(16 * g + t) * a.ldm];
        }
        else
        {
            const d2 lo = *reinterpret_cast<const d2 *>(m + 16 * g), hi = *reinterpret_cast<const d2 *>(m + 16 * g + 2);
            b[0] = lo[0];
            b[1] = lo[1];
            b[2] = hi[0];
            b[3] = hi[1];
        }
#pragma unroll
        for (int c = 0; c < CT; c++)
        {
            const double *vc = v + static_cast<long>(FEW * c) * a.ldv + 16 * g;
            const d2 lo = *reinterpret_cast<const d2 *>(vc), hi = *reinterpret_cast<const d2 *>(vc + 2);
            const double x[4] = { lo[0], lo[1], hi[0], hi[1] };
#pragma unroll
            for (int t = 0; t < 4; t++)
                acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t], b[t], acc[c], 0, 0, 0);
        }
    }
    // accumulator: lane holds column lm, rows lk + 4 e
#pragma unroll
    for (int c = 0; c < CT; c++)
#pragma unroll
        for (int e = 0; e < 4; e++)
            part[w][c][e][lane] = acc[c][e];
    __syncthreads();
    for (int t = threadIdx.x; t < CT * 256; t += THREADS)
    {
        const int c = t >> 8, e = (t >> 6) & 3, l = t & 63;
        double s = part[0][c][e][l];
#pragma unroll
        for (int q = 1; q < WAVES; q++)
            s += part[q][c][e][l];
        const long at = (row + FEW * c + (l >> 4) + 4 * e) * a.ldo + col + (l & 15);
        a.out[at] = a.C ? a.C[at] - s : s;
    }
}

template <bool KMAJOR>
void launch(hipStream_t s, const Args &a, int rows, int cols)
{
    // as many 16-row tiles per workgroup as the rows allow: they share L's loads
    const int tiles = rows / FEW;
    const unsigned gx = static_cast<unsigned>(cols / FEW);
    if (tiles % 4 == 0)
        hipLaunchKernelGGL((k_few_rows<4, KMAJOR>), dim3(gx, tiles / 4), dim3(THREADS), 0, s, a);
    else if (tiles % 2 == 0)
        hipLaunchKernelGGL((k_few_rows<2, KMAJOR>), dim3(gx, tiles / 2), dim3(THREADS), 0, s, a);
    else
        hipLaunchKernelGGL((k_few_rows<1, KMAJOR>), dim3(gx, tiles), dim3(THREADS), 0, s, a);
    GP_CHECK_LAUNCH();
}

}  // namespace

void few_rows_solve(hipStream_t s, const double *L, long lda, const double *Wpanel, int width, int n, double *X, double *V, long ldx, int rows)
{
    require(n > 0 && n % 16 == 0 && width > 0 && width % 16 == 0 && rows > 0 && rows % FEW == 0 && lda >= n && ldx >= n, "few_rows_solve: bad shape");
    require(lda % 2 == 0 && ldx % 2 == 0 && reinterpret_cast<uintptr_t>(L) % 16 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0
                && reinterpret_cast<uintptr_t>(V) % 16 == 0,
            "few_rows_solve: operands must be 16-byte aligned");
    require(rows / FEW <= 65535, "few_rows_solve: too many rows");
    for (int J = 0; J * width < n; J++)
    {
        const int j0 = J * width, nb = std::min(width, n - j0), j1 = j0 + nb;
        launch<true>(s, Args{ X + j0, ldx, Wpanel + static_cast<long>(J) * width * width, width, nullptr, V + j0, ldx, nb }, rows, nb);
        if (j1 < n)
            launch<false>(s, Args{ V + j0, ldx, L + static_cast<long>(j1) * lda + j0, lda, X + j1, X + j1, ldx, nb }, rows, n - j1);
    }
}

}  // namespace gpamd::k
