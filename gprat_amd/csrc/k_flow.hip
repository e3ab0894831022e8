// Cholesky factorisation as one launch: 64x64 tiles as a dataflow.
//
// The launch-per-step schedule pays two launches and their gaps for each 64
// columns of the diagonal-block chain; below some ten thousand columns that
// chain, not the matrix cores, sets the time. Here workgroups take tasks from
// a device counter and wait for the tiles they need on progress counters, so a
// step of the chain costs a factor, two block products and one hand-over
// between workgroups.
//
// Block columns come in panels of PANEL. A tile of panel p is left-looking
// over panels p - 1 and p (acc = sum_k L_ik L_jk^T in registers, at most
// 2 PANEL - 1 products, then L_ij = (A_ij - acc) W_jj^T); panels 0 .. p - 2
// have been subtracted from A_ij before, one update task each. Task order: the
// first diagonal block, then per block column j of panel p
//  * the pair L(j+1, j) and the diagonal block j + 1 (one task: the chain),
//    the tiles (i, j) below it, and column j of the rows that ride along
//    below the matrix (right-hand sides: they leave as B L^-T);
//  * a PANEL-th of panel p - 1's updates of the tiles right of panel p,
//    nearest columns first: they fill the device while the chain runs.
// Every task depends only on tasks with smaller numbers, which have been
// taken by running workgroups, so every wait ends whatever else holds the
// device; a spin limit turns a lost update into an error instead of a hang.
//
// progress[r] counts the finished tiles of row r from its first one on (L_rr
// counts too): a tile needs progress[i] > k and progress[j] > k for its k-th
// product and progress[j] > j for W_jj. applied[r][c] counts the panels
// subtracted from tile (r, c). Results are written with ordinary stores, made
// visible by a write-back of the L2 that has ended before the counter moves
// (publish), and read after an agent-scope acquire.
//
// Measured on MI355X: a step of the chain takes 14.5 us when nothing else runs
// (factor 8, the two products 2.9, stores and hand-over 2.5), 25 to 40 us
// beside a full device. A fit (assembly and alpha included) at n = 1024 / 2048 /
// 4992 / 8192 takes 0.37 / 0.69 / 2.34 / 6.30 ms (panel schedule: 0.76 / 1.59 /
// 4.35 / 8.72), the last's factorisation at 32 TF/s: a 64x64 tile's products
// read 64 KB of operands for 0.5 MFLOP.
#include <algorithm>
#include <climits>

#include "block64.hpp"
#include "block_mfma.hpp"
#include "kernels.hpp"

namespace gpamd::k
{
namespace
{

struct FlowArgs
{
    double *A;
    long lda;
    double *X;
    int nb, ne, nu, solve;
    double *Winv;
    int *info, *queue, *progress, *applied;
    int tasks;
};

constexpr int NB = 64;
constexpr int THREADS = 256;
constexpr int PANEL = FLOW_PANEL;
// polls before a wait gives up, and how often it looks whether another has
// (a poll takes of the order of a microsecond: more than ten seconds)
constexpr int SPIN_LIMIT = 1 << 24;
constexpr int SPIN_LOOK = 1 << 10;

__global__ __launch_bounds__(THREADS) void k_flow_init(FlowArgs a, long counters)
{
    const long i = static_cast<long>(blockIdx.x) * THREADS + threadIdx.x;
    if (i == 0)
        *a.info = INT_MAX;
    // the queue, progress and applied counters lie one after another
    if (i < counters)
        a.queue[i] = a.solve && i >= 1 && i <= a.nb ? a.nb : 0;
}

__device__ __forceinline__ int load_counter(const int *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Waits until counters p and q have reached `need`, and r `need_r`; returns the
// smaller of p and q (at least `need`). Everything the counted tasks wrote is
// then visible to the workgroup. words: two alternating result words in LDS.
__device__ __forceinline__ int wait_for(const FlowArgs &a, const int *p, const int *q, int need, const int *r, int need_r, int *words, int &turn)
{
    int *word = words + (turn & 1);
    turn++;
    if (threadIdx.x == 0)
    {
        int v = min(load_counter(p), load_counter(q)), u = load_counter(r);
        for (int spins = 1; v < need || u < need_r; spins++)
        {
            if (spins >= SPIN_LIMIT)
                atomicMin(a.info, FLOW_STALLED);
            if (spins % SPIN_LOOK == 0 && load_counter(a.info) == FLOW_STALLED)
            {
                v = max(v, need);
                break;
            }
            // several columns away: poll seldom, so that hundreds of waiting
            // workgroups leave the counters' cache lines to the chain
            if (v < need - 1)
                __builtin_amdgcn_s_sleep(64);
            else
                __builtin_amdgcn_s_sleep(2);
            v = min(load_counter(p), load_counter(q));
            u = load_counter(r);
        }
        *word = v;
    }
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    return *word;
}

__device__ __forceinline__ int wait_for(const FlowArgs &a, const int *p, const int *q, int need, int *words, int &turn)
{
    return wait_for(a, p, q, need, p, 0, words, turn);
}

// This workgroup's stores are visible to whoever sees the counter at
// `value`: every wavefront's have reached the L2 at the barrier, and the L2 is
// written back before the counter moves. The write-back and the wait for it
// are written out in one piece: the compiler's release store (clang of ROCm
// 7.2) leaves that wait out wherever it knows of no other vector memory
// operation in flight, as it did after the chain's L(j + 1, j). The counter
// then overtook the tile: beside other kernels, whose dirty lines make a
// write-back long, the next diagonal step read old elements of it (a fit of
// n = 9000 was off by 3e-6 with requests of a server in flight).
__device__ __forceinline__ void publish(int *p, int value)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
    {
        asm volatile("buffer_wbl2 sc1\n\ts_waitcnt vmcnt(0)" ::: "memory");
        __hip_atomic_store(p, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// acc += A A^T beside mfma_nt_acc's A B^T, from the same staged rows.
__device__ __forceinline__ void mfma_pair(const double *A, const double *B, blk::v4d (&ab)[2][2], blk::v4d (&aa)[2][2], int tid)
{
    const int lane = tid & 63, w = tid >> 6;
    const int lm = lane & 15, lk = lane >> 4;
    const int r0 = (w >> 1) * 32, c0 = (w & 1) * 32;
#pragma unroll 4
    for (int k0 = 0; k0 < NB; k0 += 4)
    {
        double a[2], b[2], t[2];
#pragma unroll
        for (int i = 0; i < 2; i++)
        {
            a[i] = A[(r0 + i * 16 + lm) * blk::XS + k0 + lk];
            b[i] = B[(c0 + i * 16 + lm) * blk::XS + k0 + lk];
            t[i] = A[(c0 + i * 16 + lm) * blk::XS + k0 + lk];
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
            {
                ab[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], ab[i][j], 0, 0, 0);
                aa[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], t[j], aa[i][j], 0, 0, 0);
            }
    }
}

// Block products k0 .. k1 - 1 of two block rows through the LDS stages, the
// next pair of blocks on its way while the current one is multiplied.
template <class F>
__device__ __forceinline__ void stream_blocks(const double *ri, const double *rj, long lda, int k0, int k1, double *buf0, double *buf1, int tid, F product)
{
    blk::d2 va[8], vb[8];
    blk::load_block(ri + static_cast<long>(NB) * k0, lda, va, tid);
    blk::load_block(rj + static_cast<long>(NB) * k0, lda, vb, tid);
    for (int k = k0; k < k1; k++)
    {
        __syncthreads();  // every wavefront is done with the previous pair
        blk::store_block(buf0, va, tid);
        blk::store_block(buf1, vb, tid);
        __syncthreads();
        if (k + 1 < k1)
        {
            blk::load_block(ri + static_cast<long>(NB) * (k + 1), lda, va, tid);
            blk::load_block(rj + static_cast<long>(NB) * (k + 1), lda, vb, tid);
        }
        __builtin_amdgcn_sched_barrier(0);
        product();
    }
}

// buf[r][c] (stride XS) = s - acc at this lane's accumulator positions.
__device__ __forceinline__ void stage_difference(double *buf, const double (&s)[16], const blk::v4d (&acc)[2][2], int tid)
{
    int q = 0;
    blk::for_each(acc, [&](int r, int c, double v) { buf[r * blk::XS + c] = s[q++] - v; }, tid);
}

// The thread's index, hidden from the compiler: what follows from it is not
// carried from task to task (the addresses of a task's block operations, kept
// across the task loop, filled 188 more registers). The factorisation still
// spills 105 of its 256 registers: the diagonal task keeps addresses and
// accumulators in scratch (440 bytes a lane). The launch on a given factor
// spills none.
__device__ __forceinline__ int own_thread()
{
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

__device__ __forceinline__ double *row_of(const FlowArgs &a, int i)
{
    return i < a.nb ? a.A + static_cast<long>(NB) * i * a.lda : a.X + static_cast<long>(NB) * (i - a.nb) * a.lda;
}
__device__ __forceinline__ int *applied_of(const FlowArgs &a, int i, int j) { return a.applied + static_cast<long>(i) * a.nb + j; }

// L = S W^T for W lower triangular (buf S and W staged, stride XS): wavefront
// w owns rows 16 w .. 16 w + 15, column block c needs k < 16 (c + 1) only.
__device__ __forceinline__ void solve_product(const double *S, const double *W, blk::v4d (&acc)[4], int tid)
{
    const int lane = tid & 63, w = tid >> 6;
    const int lm = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int c = 0; c < 4; c++)
        acc[c] = blk::v4d{ 0.0, 0.0, 0.0, 0.0 };
#pragma unroll
    for (int kc = 0; kc < 4; kc++)
#pragma unroll
        for (int k0 = 16 * kc; k0 < 16 * kc + 16; k0 += 4)
        {
            const double a = S[(16 * w + lm) * blk::XS + k0 + lk];
#pragma unroll
            for (int c = kc; c < 4; c++)
                acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, W[(16 * c + lm) * blk::XS + k0 + lk], acc[c], 0, 0, 0);
        }
}

// f(row, column, value) over a solve_product's results.
template <class F>
__device__ __forceinline__ void for_each_solved(const blk::v4d (&acc)[4], int tid, F f)
{
    const int lane = tid & 63, w = tid >> 6;
    const int lm = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int e = 0; e < 4; e++)
            f(16 * w + lk + 4 * e, 16 * c + lm, acc[c][e]);
}

// D -= L L^T for D and L staged (stride XS), the ten 16x16 tiles on and below
// the diagonal dealt to the four wavefronts (3, 3, 2, 2).
__device__ __forceinline__ void subtract_square(double *D, const double *L, int tid)
{
    const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lm = lane & 15, lk = lane >> 4;
    constexpr int rows[4][3] = { { 0, 3, 3 }, { 1, 3, 3 }, { 1, 2, -1 }, { 2, 2, -1 } };
    constexpr int cols[4][3] = { { 0, 0, 1 }, { 0, 2, 3 }, { 1, 0, -1 }, { 1, 2, -1 } };
#pragma unroll
    for (int v = 0; v < 4; v++)
    {
        if (w != v)
            continue;
        blk::v4d acc[3];
        double d[3][4];
#pragma unroll
        for (int t = 0; t < 3; t++)
            if (rows[v][t] >= 0)
            {
                acc[t] = blk::v4d{ 0.0, 0.0, 0.0, 0.0 };
#pragma unroll
                for (int e = 0; e < 4; e++)
                    d[t][e] = D[(16 * rows[v][t] + lk + 4 * e) * blk::XS + 16 * cols[v][t] + lm];
            }
#pragma unroll
        for (int k0 = 0; k0 < NB; k0 += 4)
#pragma unroll
            for (int t = 0; t < 3; t++)
                if (rows[v][t] >= 0)
                    acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(L[(16 * rows[v][t] + lm) * blk::XS + k0 + lk],
                                                                  L[(16 * cols[v][t] + lm) * blk::XS + k0 + lk], acc[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 3; t++)
            if (rows[v][t] >= 0)
            {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    D[(16 * rows[v][t] + lk + 4 * e) * blk::XS + 16 * cols[v][t] + lm] = d[t][e] - acc[t][e];
            }
    }
}

typedef __attribute__((address_space(3))) double lds_double;

// Out of line: the elimination's registers stay out of the tasks' allocation.
__device__ __noinline__ void factor_staged(lds_double *d, lds_double *w, int *info, int col0)
{
    factor_block64(reinterpret_cast<double(*)[blk::XS]>((double *)d), reinterpret_cast<double(*)[blk::XS]>((double *)w), info, col0);
}

// The columns' panels start their products here (see above).
__device__ __forceinline__ int first_product(int column) { return max(0, (column / PANEL - 1) * PANEL); }

// L(j+1, j) and the diagonal block j + 1 (q = j + 1 >= 1), or block 0: the
// chain, at a raised wave priority beside the other tasks of its CU.
__device__ __forceinline__ void diagonal_task(const FlowArgs &a, int q, double *buf0, double *buf1, int *words, int &turn)
{
    const int tid = own_thread();
    double *rq = row_of(a, q);
    double *dst = rq + static_cast<long>(NB) * q;
    double d[16];
    __builtin_amdgcn_s_setprio(2);
    if (q == 0)
        blk::load_at_acc(dst, a.lda, d, tid);
    else
    {
        const int j = q - 1;
        const double *rj = row_of(a, j);
        blk::v4d off[2][2], dia[2][2];
        blk::zero(off);
        blk::zero(dia);
        double *lqj = rq + static_cast<long>(NB) * j;
        // the stored values first: their latency is then not the chain's
        if (q / PANEL >= 2)
            wait_for(a, applied_of(a, q, q), applied_of(a, q, q), q / PANEL - 1, applied_of(a, q, j), j / PANEL - 1, words, turn);
        double s[16];
        blk::load_at_acc(lqj, a.lda, s, tid);
        blk::load_at_acc(dst, a.lda, d, tid);
        const int pair = first_product(q);  // both tiles' products from here on
        for (int k = first_product(j); k < j;)
        {
            const int k1 = min(k < pair ? min(j, pair) : j, wait_for(a, a.progress + q, a.progress + j, k + 1, words, turn));
            if (k < pair)
                stream_blocks(rq, rj, a.lda, k, k1, buf0, buf1, tid, [&] { blk::mfma_nt_acc(buf0, buf1, off, tid); });
            else
                stream_blocks(rq, rj, a.lda, k, k1, buf0, buf1, tid, [&] { mfma_pair(buf0, buf1, off, dia, tid); });
            k = k1;
        }
        __syncthreads();
        stage_difference(buf0, s, off, tid);
        int e = 0;
        blk::for_each(dia, [&](int, int, double v) { d[e++] -= v; }, tid);
        wait_for(a, a.progress + j, a.progress + j, j + 1, words, turn);
        blk::stage_block(buf1, a.Winv + static_cast<long>(j) * NB * NB, NB, tid);
        __syncthreads();
        blk::v4d l[4];
        solve_product(buf0, buf1, l, tid);
        __syncthreads();
        for_each_solved(l, tid,
                        [&](int r, int c, double v)
                        {
                            buf0[r * blk::XS + c] = v;
                            lqj[static_cast<long>(r) * a.lda + c] = v;
                        });
    }
    blk::v4d pos[2][2];
    int e = 0;
    blk::for_each(pos, [&](int r, int c, double) { buf1[r * blk::XS + c] = c <= r ? d[e] : 0.0; e++; }, tid);
    __syncthreads();
    if (q > 0)
    {
        subtract_square(buf1, buf0, tid);
        publish(a.progress + q, q);  // its barrier: the differences are in place
    }
    factor_staged((lds_double *)buf1, (lds_double *)buf0, a.info, NB * q);
    // the inverse first: the next step waits for it, nothing in this launch for L_qq
    double *w = a.Winv + static_cast<long>(q) * NB * NB;
#pragma unroll
    for (int s = 0; s < NB * NB / 2 / THREADS; s++)
    {
        const int t = tid + THREADS * s, r = t >> 5, c = (t & 31) * 2;
        const blk::d2 v = *reinterpret_cast<const blk::d2 *>(buf0 + r * blk::XS + c);
        *reinterpret_cast<blk::d2 *>(w + r * NB + c) = blk::d2{ c <= r ? v[0] : 0.0, c + 1 <= r ? v[1] : 0.0 };
    }
    publish(a.progress + q, q + 1);
    __builtin_amdgcn_s_setprio(0);
    for (int t = tid; t < NB * NB; t += THREADS)
    {
        const int r = t >> 6, c = t & 63;
        if (c <= r)
            dst[static_cast<long>(r) * a.lda + c] = buf1[r * blk::XS + c];
    }
}

// The unit row (its block column) at place `x` of a list of rows below the
// matrix, or -1.
__device__ __forceinline__ int extra_unit(const FlowArgs &a, int x) { return x < a.ne - a.nu ? -1 : x - (a.ne - a.nu); }

// Tile (i, j) off the diagonal. unit >= 0: a row that starts from the identity
// in block column `unit`. SOLVE: the factor is given.
template <bool SOLVE>
__device__ __forceinline__ void off_task(const FlowArgs &a, int i, int j, int unit, double *buf0, double *buf1, int *words, int &turn)
{
    const int tid = own_thread();
    double *ri = row_of(a, i);
    const double *rj = row_of(a, j);
    double *dst = ri + static_cast<long>(NB) * j;
    blk::v4d acc[2][2];
    blk::zero(acc);
    const int before = j / PANEL - 1;                     // panels subtracted by update tasks
    const bool stored = unit < 0 || unit / PANEL < before;  // the tile has a stored value
    // the stored value, and a given factor's inverse block, first: their
    // latency is then not the chain's
    double s[16];
    if (stored)
    {
        if (before >= 1)
            wait_for(a, applied_of(a, i, j), applied_of(a, i, j), before, words, turn);
        blk::load_at_acc(dst, a.lda, s, tid);
    }
    else
    {
        int e = 0;
        blk::for_each(acc, [&](int r, int c, double) { s[e++] = (j == unit && r == c) ? 1.0 : 0.0; }, tid);
    }
    const double *wj = a.Winv + static_cast<long>(j) * NB * NB;
    blk::d2 vw[8];
    if (SOLVE)
        blk::load_block(wj, NB, vw, tid);
    for (int k = max(first_product(j), unit); k < j;)
    {
        const int k1 = min(j, wait_for(a, a.progress + i, a.progress + j, k + 1, words, turn));
        stream_blocks(ri, rj, a.lda, k, k1, buf0, buf1, tid, [&] { blk::mfma_nt_acc(buf0, buf1, acc, tid); });
        k = k1;
    }
    __syncthreads();
    stage_difference(buf0, s, acc, tid);
    if (SOLVE)
        blk::store_block(buf1, vw, tid);
    else
    {
        wait_for(a, a.progress + j, a.progress + j, j + 1, words, turn);
        blk::stage_block(buf1, wj, NB, tid);
    }
    __syncthreads();
    blk::v4d l[4];
    solve_product(buf0, buf1, l, tid);
    for_each_solved(l, tid, [&](int r, int c, double v) { dst[static_cast<long>(r) * a.lda + c] = v; });
    publish(a.progress + i, j + 1);
}

// Tile (i, j) -= panel p's products.
__device__ __forceinline__ void update_task(const FlowArgs &a, int i, int j, int p, int unit, double *buf0, double *buf1, int *words, int &turn)
{
    const int tid = own_thread();
    double *dst = row_of(a, i) + static_cast<long>(NB) * j;
    const int k0 = max(p * PANEL, unit), k1 = (p + 1) * PANEL;
    const bool stored = unit < 0 || unit / PANEL < p;
    blk::v4d acc[2][2];
    blk::zero(acc);
    wait_for(a, a.progress + i, a.progress + j, k1, applied_of(a, i, j), stored ? p : 0, words, turn);
    stream_blocks(row_of(a, i), row_of(a, j), a.lda, k0, k1, buf0, buf1, tid, [&] { blk::mfma_nt_acc(buf0, buf1, acc, tid); });
    double s[16];
    if (stored)
        blk::load_at_acc(dst, a.lda, s, tid);
    else
    {
#pragma unroll
        for (int e = 0; e < 16; e++)
            s[e] = 0.0;
    }
    int e = 0;
    blk::for_each(acc, [&](int r, int c, double v) { dst[static_cast<long>(r) * a.lda + c] = s[e++] - v; }, tid);
    publish(applied_of(a, i, j), p + 1);
}

// Rows below the matrix: nu that start from the identity (X's first nu), then
// ne - nu others. A task list has the others first. Those that panel p's
// updates of later columns reach:
__host__ __device__ __forceinline__ int updated_extra(int ne, int nu, int p)
{
    const int reach = (p + 1) * PANEL;
    return (ne - nu) + (reach < nu ? reach : nu);
}

// Tasks of block column j: its tiles and its share of panel j / PANEL - 1's
// updates [*u0, *u0 + *updates). Column c has own_tiles of the matrix's rows
// from block `from` on (none when L is given).
__host__ __device__ __forceinline__ int own_tiles(const FlowArgs &a, int from) { return a.solve ? 0 : a.nb - from; }
__host__ __device__ __forceinline__ int column_tiles(const FlowArgs &a, int j)
{
    return own_tiles(a, j + 1) + (a.ne - a.nu) + (j + 1 < a.nu ? j + 1 : a.nu);
}
__host__ __device__ __forceinline__ void column_updates(const FlowArgs &a, int j, long *u0, int *updates)
{
    const int p = j / PANEL - 1, m = a.nb - (p + 2) * PANEL;
    *u0 = 0;
    *updates = 0;
    if (p < 0 || m <= 0)
        return;
    const long all = (a.solve ? 0 : static_cast<long>(m) * (m + 1) / 2) + static_cast<long>(m) * updated_extra(a.ne, a.nu, p);
    const int c = j % PANEL;
    // rounded up: the first tile, which the next panel's first diagonal
    // block needs, is in the first share
    const long lo = (all * c + PANEL - 1) / PANEL, hi = (all * (c + 1) + PANEL - 1) / PANEL;
    *u0 = lo;
    *updates = static_cast<int>(hi - lo);
}

// SOLVE: the rows below a given factor only (a.solve).
template <bool SOLVE>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(2))) void k_flow(FlowArgs a)
{
    __shared__ alignas(16) double buf0[NB * blk::XS];
    __shared__ alignas(16) double buf1[NB * blk::XS];
    __shared__ int words[2];
    __shared__ int next;
    int turn = 0;
    int j = 0, first = a.solve ? 0 : 1;  // the current column and its first task's number
    long u0 = 0;
    int updates = 0, tiles = column_tiles(a, 0);
    for (;;)
    {
        __syncthreads();  // the previous task's LDS reads are done
        if (threadIdx.x == 0)
            next = atomicAdd(a.queue, 1);
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(next);
        if (t >= a.tasks)
            return;
        if constexpr (!SOLVE)
            if (t == 0)
            {
                diagonal_task(a, 0, buf0, buf1, words, turn);
                continue;
            }
        // task numbers only grow: the walk is incremental
        while (t >= first + tiles + updates)
        {
            first += tiles + updates;
            j++;
            tiles = column_tiles(a, j);
            column_updates(a, j, &u0, &updates);
        }
        const int idx = t - first, below = own_tiles(a, j + 1);
        if (!SOLVE && idx < below)
        {
            if (idx == 0)
                diagonal_task(a, j + 1, buf0, buf1, words, turn);
            else
                off_task<SOLVE>(a, j + 1 + idx, j, -1, buf0, buf1, words, turn);
        }
        else if (idx < tiles)
        {
            const int u = extra_unit(a, idx - below);
            off_task<SOLVE>(a, a.nb + (u >= 0 ? u : a.nu + idx - below), j, u, buf0, buf1, words, turn);
        }
        else
        {
            const int p = j / PANEL - 1, extra = updated_extra(a.ne, a.nu, p);
            long u = u0 + (idx - tiles);
            int c = (p + 2) * PANEL;
            while (u >= own_tiles(a, c) + extra)
                u -= own_tiles(a, c++) + extra;
            const int r = static_cast<int>(u), own = own_tiles(a, c);
            const int e = r < own ? -1 : extra_unit(a, r - own);
            update_task(a, r < own ? c + r : a.nb + (e >= 0 ? e : a.nu + r - own), c, p, e, buf0, buf1, words, turn);
        }
    }
}

// One 64x64 tile of K^-1 = WT WT^T per workgroup (i >= j; the sum starts at
// block i, where row i of WT does; tiles in row order, so the longest sums
// first), then k_grad_partial's sums over it.
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(2))) void k_flow_gradient(const double *WT, long ldw, int nb, const double *__restrict__ x,
                                                                                                   const double *__restrict__ alpha, int r, double scale,
                                                                                                   double fl, double sv, int n, double *__restrict__ part)
{
    __shared__ alignas(16) double buf0[NB * blk::XS];
    __shared__ alignas(16) double buf1[NB * blk::XS];
    const int tid = threadIdx.x;
    const long t = blockIdx.x;
    int ti = static_cast<int>((sqrt(8.0 * static_cast<double>(t) + 1.0) - 1.0) / 2.0);
    while (static_cast<long>(ti) * (ti + 1) / 2 > t)
        ti--;
    while (static_cast<long>(ti + 1) * (ti + 2) / 2 <= t)
        ti++;
    const int tj = static_cast<int>(t - static_cast<long>(ti) * (ti + 1) / 2);
    blk::v4d acc[2][2];
    blk::zero(acc);
    stream_blocks(WT + static_cast<long>(NB) * ti * ldw, WT + static_cast<long>(NB) * tj * ldw, ldw, ti, nb, buf0, buf1, tid,
                  [&] { blk::mfma_nt_acc(buf0, buf1, acc); });
    __syncthreads();
    blk::for_each(acc, [&](int rr, int c, double v) { buf0[rr * blk::XS + c] = v; });
    __syncthreads();
    const int c = tid % NB;
    const long j = static_cast<long>(tj) * NB + c;
    double s[5] = { 0.0, 0.0, 0.0, 0.0, 0.0 };
    if (j < n)
    {
        const double aj = alpha[j];
        for (int rr = tid / NB; rr < NB; rr += THREADS / NB)
        {
            const long i = static_cast<long>(ti) * NB + rr;
            if (i >= n || i < j)
                continue;
            const double kij = buf0[rr * blk::XS + c];
            const double D = scale * window_sqdist(x, i, x, j, r);
            const double e = exp(D);
            const double dkl = fl * D * e;
            const double dkv = e * sv;
            const double w = (i == j) ? 1.0 : 2.0;
            const double aa = alpha[i] * aj;
            s[0] += w * kij * dkl;
            s[1] += w * kij * dkv;
            s[2] += w * aa * dkl;
            s[3] += w * aa * dkv;
            if (i == j)
                s[4] += kij;
        }
    }
    double(*red)[THREADS] = reinterpret_cast<double(*)[THREADS]>(buf1);
#pragma unroll
    for (int q = 0; q < 5; q++)
        red[q][tid] = s[q];
    __syncthreads();
    for (int w = THREADS / 2; w > 0; w >>= 1)
    {
        if (tid < w)
            for (int q = 0; q < 5; q++)
                red[q][tid] += red[q][tid + w];
        __syncthreads();
    }
    if (tid < 5)
        part[t * 5 + tid] = red[tid][0];
}

// Partial sums of a 64x64 tile (i, j), i >= j, of V V^T over one of gridDim.y
// shares of V's 64-blocks, then their fixed-order sum subtracted from both
// halves of S. The tiles alone would leave most of the device idle (36 for
// 512 rows), so the shares are cut to about one workgroup slot each.
__device__ __forceinline__ void triangle_tile(int t, int &i, int &j)
{
    i = static_cast<int>((sqrt(8.0 * static_cast<double>(t) + 1.0) - 1.0) / 2.0);
    while (i * (i + 1) / 2 > t)
        i--;
    while ((i + 1) * (i + 2) / 2 <= t)
        i++;
    j = t - i * (i + 1) / 2;
}

__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(2))) void k_row_products(const double *V, long ldv, int nb, double *__restrict__ part)
{
    __shared__ alignas(16) double buf0[NB * blk::XS];
    __shared__ alignas(16) double buf1[NB * blk::XS];
    const int tid = threadIdx.x;
    int i, j;
    triangle_tile(blockIdx.x, i, j);
    const int per = (nb + gridDim.y - 1) / gridDim.y;
    const int k0 = min(nb, static_cast<int>(blockIdx.y) * per), k1 = min(nb, k0 + per);
    blk::v4d acc[2][2];
    blk::zero(acc);
    if (k0 < k1)
        stream_blocks(V + static_cast<long>(NB) * i * ldv, V + static_cast<long>(NB) * j * ldv, ldv, k0, k1, buf0, buf1, tid,
                      [&] { blk::mfma_nt_acc(buf0, buf1, acc); });
    double *p = part + (static_cast<long>(blockIdx.x) * gridDim.y + blockIdx.y) * (NB * NB);
    blk::for_each(acc, [&](int r, int c, double v) { p[r * NB + c] = v; });
}

__global__ __launch_bounds__(THREADS) void k_row_products_subtract(const double *__restrict__ part, int shares, double *__restrict__ S, long lds)
{
    int i, j;
    triangle_tile(blockIdx.x, i, j);
    const double *p = part + static_cast<long>(blockIdx.x) * shares * (NB * NB);
    const int e = blockIdx.y * THREADS + threadIdx.x;
    double s = 0.0;
#pragma unroll 4
    for (int q = 0; q < shares; q++)
        s += p[static_cast<long>(q) * (NB * NB) + e];
    const long r = static_cast<long>(NB) * i + (e >> 6), c = static_cast<long>(NB) * j + (e & 63);
    const double v = S[r * lds + c] - s;
    S[r * lds + c] = v;
    if (i != j)
        S[c * lds + r] = v;
}

__global__ __launch_bounds__(THREADS) void k_pack_square(const double *__restrict__ S, long lds, int n, double *__restrict__ out)
{
    for (int c = threadIdx.x; c < n; c += THREADS)
        out[static_cast<long>(blockIdx.x) * n + c] = S[blockIdx.x * lds + c];
}

}  // namespace

long flow_counters(int nb, int ne) { return 1 + (static_cast<long>(nb) + ne) * (1 + nb); }

// Workgroups of a launch: enough for the work to keep up with the chain
// (products of 64x64 blocks, 4 us each with two workgroups on a CU, over 15 us
// per block column, 8 on a given factor), and some that wait ahead; more only
// share the chain's CU and poll. Two workgroups' LDS fit a CU. Measured on
// MI355X (one call, 128 / 192 / 256 / 384 / 512 workgroups, us):
//   n = 1024 m = 1024 330 351 363 379 393     n = 2048 m = 1024 733 704 730 808 860
//   n = 3000 m = 64 - 1006 1005 1072 1147     n = 4096 m = 16 1797 1584 1523 1622 1723
//   n = 6144 m = 16 - 3757 3380 3173 3177     n = 8192 m = 16 - 8291 7085 6252 6056
static long flow_workgroups(const FlowCall &f, int cus)
{
    const double nb = f.nb, ne = f.ne - f.nu, nu = f.nu;
    const double rows = (f.solve ? 0.0 : nb / 6) + ne / 2 + nu / 6;  // products per column and block row of columns
    const double need = rows * nb * (f.solve ? 4.0 / 8 : 4.0 / 15);
    const long wgs = static_cast<long>((need + 80) / 64 + 0.5) * 64;
    return std::clamp<long>(wgs, std::min(cus / 2, 128), 2L * cus);
}

void flow_cholesky(hipStream_t s, const FlowCall &f, int cus)
{
    require(f.nb >= 1 && f.ne >= 0 && f.lda % 2 == 0 && f.lda >= static_cast<long>(NB) * f.nb, "flow_cholesky: bad shape");
    require(f.nu >= 0 && f.nu <= f.ne && f.nu <= f.nb, "flow_cholesky: more unit rows than columns");
    require(f.ne == 0 || (f.X != nullptr && reinterpret_cast<uintptr_t>(f.X) % 16 == 0), "flow_cholesky: bad rows below the matrix");
    require(reinterpret_cast<uintptr_t>(f.A) % 16 == 0 && reinterpret_cast<uintptr_t>(f.Winv) % 16 == 0,
            "flow_cholesky: operands must be 16-byte aligned");
    require(!f.solve || f.ne > 0, "flow_cholesky: nothing to solve");
    const long counters = flow_counters(f.nb, f.ne);
    FlowArgs a{ f.A, f.lda, f.X, f.nb, f.ne, f.nu, f.solve ? 1 : 0, f.Winv, f.info, f.counters, f.counters + 1, f.counters + 1 + f.nb + f.ne, 0 };
    long tasks = f.solve ? 0 : 1;
    for (int j = 0; j < f.nb; j++)
    {
        long u0;
        int updates;
        column_updates(a, j, &u0, &updates);
        tasks += column_tiles(a, j) + updates;
    }
    // every running workgroup may add one number past the last task
    require(tasks < (1L << 30), "flow_cholesky: too many tiles");
    a.tasks = static_cast<int>(tasks);
    hipLaunchKernelGGL(k_flow_init, dim3(static_cast<unsigned>(ceil_div(counters, THREADS))), dim3(THREADS), 0, s, a, counters);
    GP_CHECK_LAUNCH();
    const long wgs = std::min<long>(tasks, flow_workgroups(f, cus));
    if (f.solve)
        hipLaunchKernelGGL(k_flow<true>, dim3(static_cast<unsigned>(wgs)), dim3(THREADS), 0, s, a);
    else
        hipLaunchKernelGGL(k_flow<false>, dim3(static_cast<unsigned>(wgs)), dim3(THREADS), 0, s, a);
    GP_CHECK_LAUNCH();
}

static int row_product_shares(int n, int m)
{
    const long tiles = static_cast<long>(m / NB) * (m / NB + 1) / 2;
    return static_cast<int>(std::clamp<long>(512 / tiles, 1, ceil_div(n / NB, 4)));
}

long row_products_scratch(int n, int m)
{
    return static_cast<long>(m / NB) * (m / NB + 1) / 2 * row_product_shares(n, m) * NB * NB;
}

void subtract_row_products(hipStream_t s, const double *V, long ldv, int n, double *S, long lds, int m, double *part)
{
    require(n > 0 && n % NB == 0 && m > 0 && m % NB == 0 && ldv % 2 == 0 && ldv >= n && lds >= m, "subtract_row_products: bad shape");
    require(reinterpret_cast<uintptr_t>(V) % 16 == 0, "subtract_row_products: operand must be 16-byte aligned");
    const int shares = row_product_shares(n, m);
    const long tiles = static_cast<long>(m / NB) * (m / NB + 1) / 2;
    require(tiles < (1L << 24), "subtract_row_products: too many rows");
    hipLaunchKernelGGL(k_row_products, dim3(static_cast<unsigned>(tiles), shares), dim3(THREADS), 0, s, V, ldv, n / NB, part);
    GP_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_row_products_subtract, dim3(static_cast<unsigned>(tiles), NB * NB / THREADS), dim3(THREADS), 0, s, part, shares, S, lds);
    GP_CHECK_LAUNCH();
}

void pack_square(hipStream_t s, const double *S, long lds, int n, double *out)
{
    require(n >= 1 && lds >= n, "pack_square: bad shape");
    hipLaunchKernelGGL(k_pack_square, dim3(static_cast<unsigned>(n)), dim3(THREADS), 0, s, S, lds, n, out);
    GP_CHECK_LAUNCH();
}

long flow_gradient_tiles(int n_pad) { return static_cast<long>(n_pad / NB) * (n_pad / NB + 1) / 2; }

void flow_gradient(hipStream_t s, const double *WT, long ldw, int n_pad, const double *x, const double *alpha, int r, SEK sek, double sig_l,
                   double sig_v, int n, double *part, double *out)
{
    const long tiles = flow_gradient_tiles(n_pad);
    require(n >= 1 && n <= n_pad && n_pad % NB == 0 && ldw % 2 == 0 && ldw >= n_pad && tiles < (1L << 31), "flow_gradient: bad shape");
    require(reinterpret_cast<uintptr_t>(WT) % 16 == 0, "flow_gradient: operand must be 16-byte aligned");
    const double fl = -2.0 * sek.vertical / sek.lengthscale * sig_l;
    hipLaunchKernelGGL(k_flow_gradient, dim3(static_cast<unsigned>(tiles)), dim3(THREADS), 0, s, WT, ldw, n_pad / NB, x, alpha, r, sek.scale(), fl,
                       sig_v, n, part);
    GP_CHECK_LAUNCH();
    gradient_reduce(s, part, tiles, out);
}

}  // namespace gpamd::k
