// FP32 matrix-core products for the mixed-precision path: the trailing
// update of the factorisation and the variance solve.
//
// The factored FP64 panel is first copied to FP32 in k-major order
// (P[k][row], `panel_to_f32t`), so both operands of C -= A B^T are read as
// contiguous 16-byte row segments and land in LDS without a transpose.
// One workgroup (4 wavefronts) owns a 128x128 tile (short solve products:
// 64x64); each wavefront accumulates a quarter in FP32 on
// v_mfma_f32_16x16x4f32 over 16-deep LDS slabs (double buffered), and the
// epilogue subtracts the FP32 product from the FP64 matrix. The slabs go from
// memory straight into LDS; they are shallow (32 KiB of LDS per workgroup,
// also for the small tile, whose slabs are 32 deep so that a copy's latency is
// paid half as often), and with a 168-register budget a CU holds three
// workgroups. On MI355X the variance solve's updates ran at 124 TF/s staged
// through registers (118 with 32-deep slabs and two workgroups); the direct
// copies took a variance request at n = 24000 with 8192 columns from 155.4 to
// 143.8 ms, with the FP64 residual product's, and the mixed request at
// n = 32768 from 406.8 to 398.0.
#include "kernels.hpp"

namespace gpamd::k
{
namespace
{

typedef float v4f __attribute__((ext_vector_type(4)));
constexpr int THREADS = 256;

// Tile shapes: B x B elements of C per workgroup, one quarter per wavefront,
// over D-deep slabs. The sums run in the same k order in both, so an element
// does not depend on the shape that computed it.
template <int B, int D>
struct Tile
{
    static constexpr int BM = B, BK = D;
    static constexpr int Q = B / 2, NI = B / 32;        // a wavefront's quarter, in elements and 16-wide blocks
    static constexpr int LPT = D * B / (THREADS * 4);  // 16-byte copies per lane per operand slab
    static constexpr int SLAB = D * B;                 // floats of LDS per slab
};
using Large = Tile<128, 16>;
using Small = Tile<64, 32>;
constexpr int BM = Large::BM;

// C (op)= A B with A(i, k) = A[k * lda + i] and B(k, j) = B[k * ldb + j]
// (both operands k-major, as the panel copies are), FP32 products and sums.
template <class TC>
struct Params32
{
    const float *A;
    long lda;
    const float *B;
    long ldb;
    TC *C;
    long ldc;
    int M, N, K;
    int lower;  // only i + diag_off >= j
    long diag_off;
    int set;  // C = acc instead of C -= acc
    int max_wgs;  // > 0: at most this many workgroups, looping over tiles
    int k_to_row;  // A(i, k) known zero for k > i: each row tile stops K at its last row
    int k_from_row;  // A(i, k) known zero for k < i: each row tile starts K at its first row
    int *queue;    // capped: tile counter (0 at launch) or null for fixed shares
    int tiles;     // capped: tiles holding part of the update
};

// One operand's slabs, copied from memory straight into LDS (no staging
// registers, no LDS writes ahead of the products' reads): every copy moves
// 16 bytes per lane to 1 KiB of consecutive LDS, that is 256 / BM k-rows, so
// the rows cannot be padded. The four k-slots of a read fall into disjoint
// banks because row k holds column c at c ^ 16 (k mod 4), which the lanes
// arrange by choosing what they fetch. Columns past the operand's edge are
// clamped to its last group of four; they only feed accumulators the
// epilogue never stores.
template <class S>
struct DirectSlab32
{
    static constexpr int ROWS = 256 / S::BM;  // k-rows per copy
    const float *p[S::LPT];  // what the lane fetches in each of its wavefront's copies
    long step;               // from one slab to the next
    int first;               // the wavefront's first copy

    __device__ __forceinline__ void init(const float *origin, long ld, int rows, int tid)
    {
        step = S::BK * ld;
        first = __builtin_amdgcn_readfirstlane(tid >> 6) * S::LPT;
        const int kk = (tid & 63) / (S::BM / 4), c = (tid & 63) % (S::BM / 4) * 4;
#pragma unroll
        for (int s = 0; s < S::LPT; s++)
        {
            const int k = (first + s) * ROWS + kk;
            p[s] = origin + k * ld + min(c ^ 16 * (k & 3), rows - 4);
        }
    }

    // T: 16-byte aligned LDS; p moves on to the next slab
    __device__ __forceinline__ void fetch(float *T)
    {
#pragma unroll
        for (int s = 0; s < S::LPT; s++)
        {
            using lds_ptr = __attribute__((address_space(3))) float *;
            const unsigned dst = static_cast<unsigned>(reinterpret_cast<unsigned long>((lds_ptr)(T + (first + s) * 256)));
            // no output register: the data goes to LDS at m0 + 16 lane; a
            // write of m0 needs one wait state before its use. m0 is named as
            // written, so that a value of the compiler's there is set again
            // (it is nobody's to preserve, which is what clang warns of)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                         :
                         : "s"(__builtin_amdgcn_readfirstlane(dst)), "v"(p[s])
                         : "memory", "m0");
#pragma clang diagnostic pop
            p[s] += step;
        }
    }

    // this wavefront's copies are in LDS (a barrier shows them to the others)
    static __device__ __forceinline__ void landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
};

template <class S>
__device__ __forceinline__ void mfma_slab32(const float *As, const float *Bs, int wr, int wc, int lm, int lk, v4f (&acc)[S::NI][S::NI])
{
#pragma unroll
    for (int kq = 0; kq < S::BK / 4; kq++)
    {
        float a[S::NI], b[S::NI];
#pragma unroll
        for (int i = 0; i < S::NI; i++)
            a[i] = As[(kq * 4 + lk) * S::BM + ((wr * S::Q + i * 16) ^ 16 * lk) + lm];
#pragma unroll
        for (int j = 0; j < S::NI; j++)
            b[j] = Bs[(kq * 4 + lk) * S::BM + ((wc * S::Q + j * 16) ^ 16 * lk) + lm];
#pragma unroll
        for (int i = 0; i < S::NI; i++)
#pragma unroll
            for (int j = 0; j < S::NI; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
}

// C (op)= acc over one wavefront's quarter of a tile, element (i, j, e) at
// cw + (16 i + e) ldc + 16 j. C is read and written through the same
// pointer, so the compiler keeps every element's load, wait and store in
// program order; the loads of a 16-row strip are therefore all issued before
// its first store (one memory latency per strip, not sixteen). FULL: an
// interior tile (no edge, wholly inside the lower band), no predicates.
template <bool FULL, int NI, class TC>
__device__ __forceinline__ void store_quarter32(const Params32<TC> &p, const v4f (&acc)[NI][NI], TC *cw, int rb, int cb, int rows_a, int rows_b,
                                                long r0, long c0)
{
#pragma unroll
    for (int i = 0; i < NI; i++)
    {
        bool ok[4 * NI];
#pragma unroll
        for (int j = 0; j < NI; j++)
#pragma unroll
            for (int e = 0; e < 4; e++)
            {
                const int rr = rb + i * 16 + e, cc = cb + j * 16;
                ok[j * 4 + e] = FULL || ((rr < rows_a) & (cc < rows_b) & !(p.lower && r0 + rr + p.diag_off < c0 + cc));
            }
        TC cv[4 * NI];
        if (!p.set)
        {
#pragma unroll
            for (int j = 0; j < NI; j++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    cv[j * 4 + e] = ok[j * 4 + e] ? cw[static_cast<long>(i * 16 + e) * p.ldc + j * 16] : TC(0);
        }
#pragma unroll
        for (int j = 0; j < NI; j++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (ok[j * 4 + e])
                    cw[static_cast<long>(i * 16 + e) * p.ldc + j * 16]
                        = p.set ? static_cast<TC>(acc[i][j][e]) : cv[j * 4 + e] - static_cast<TC>(acc[i][j][e]);
    }
}

// One tile of C at (r0, c0).
// part 0: the tile's whole K range; parts 1 and 2: its first and second
// half (in slabs), for C -= updates only.
template <class S, class TC>
__device__ __forceinline__ void gemm_tile32(const Params32<TC> &p, long r0, long c0, float (*As)[S::SLAB], float (*Bs)[S::SLAB], int part = 0)
{
    constexpr int BM = S::BM, BK = S::BK, NI = S::NI;
    const int rows_a = static_cast<int>(min(static_cast<long>(BM), p.M - r0));
    const int rows_b = static_cast<int>(min(static_cast<long>(BM), p.N - c0));

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wr = wave >> 1, wc = wave & 1;
    const int lm = lane & 15, lk = lane >> 4;

    v4f acc[NI][NI];
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++)
            acc[i][j] = v4f{ 0.0f, 0.0f, 0.0f, 0.0f };

    const int kmax = p.k_to_row ? static_cast<int>(min(static_cast<long>(p.K), r0 + BM)) : p.K;
    const int kmin = p.k_from_row ? static_cast<int>(min(static_cast<long>(kmax), r0)) : 0;
    const int half = (kmax / BK / 2) * BK;
    const int k0 = part == 2 ? half : kmin, k1 = part == 1 ? half : kmax;
    if (k1 > k0)
    {
        DirectSlab32<S> da, db;
        da.init(p.A + r0 + static_cast<long>(k0) * p.lda, p.lda, rows_a, tid);
        db.init(p.B + c0 + static_cast<long>(k0) * p.ldb, p.ldb, rows_b, tid);
        da.fetch(As[0]);
        db.fetch(Bs[0]);
        da.landed();
        __syncthreads();

        int buf = 0;
        const int steps = (k1 - k0) / BK;
        for (int t = 1; t < steps; t++)
        {
            da.fetch(As[buf ^ 1]);
            db.fetch(Bs[buf ^ 1]);
            // the copies stay ahead of this slab's products
            __builtin_amdgcn_sched_barrier(0);
            mfma_slab32<S>(As[buf], Bs[buf], wr, wc, lm, lk, acc);
            __builtin_amdgcn_sched_barrier(0);
            da.landed();
            __syncthreads();
            buf ^= 1;
        }
        mfma_slab32<S>(As[buf], Bs[buf], wr, wc, lm, lk, acc);
    }

    // Accumulator layout of the 16x16x4 f32 MFMA on gfx950: lane holds
    // column (lane % 16) and rows 4 (lane / 16) + e, e = 0..3.
    const bool full = rows_a == BM && rows_b == BM && (!p.lower || r0 + p.diag_off >= c0 + BM - 1);
    const int er = wr * S::Q + lk * 4, ec = wc * S::Q + lm;
    TC *cw = p.C + (r0 + er) * p.ldc + c0 + ec;
    if (full)
        store_quarter32<true, NI>(p, acc, cw, er, ec, rows_a, rows_b, r0, c0);
    else
        store_quarter32<false, NI>(p, acc, cw, er, ec, rows_a, rows_b, r0, c0);
}

// The solves' products, one workgroup per tile, row-major. ROLE only
// separates profiler names: 1 diagonal step, 2 update.
template <class S, int ROLE>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(3))) void k_gemm_f32_solve(Params32<float> p)
{
    __shared__ alignas(16) float As[2][S::SLAB];
    __shared__ alignas(16) float Bs[2][S::SLAB];
    const unsigned gx = (p.N + S::BM - 1) / S::BM;
    gemm_tile32<S, float>(p, static_cast<long>(blockIdx.x / gx) * S::BM, static_cast<long>(blockIdx.x % gx) * S::BM, As, Bs);
}

// The factorisation's trailing update (FP64 C). Tiles are numbered
// row-major; a launch with fewer workgroups than tiles loops over them
// (tile w, w + G, ...).
template <class TC>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(3))) void k_gemm_f32_tn(Params32<TC> p)
{
    __shared__ alignas(16) float As[2][Large::SLAB];
    __shared__ alignas(16) float Bs[2][Large::SLAB];
    const int gx = (p.N + BM - 1) / BM;
    const int gy = (p.M + BM - 1) / BM;
    // The tiles holding part of the update (for a lower update, those
    // touching the band) are numbered row by row, neighbours in flight
    // together. With a queue, each workgroup takes the next tile number from
    // a device counter when it is ready (one that starts late or shares its
    // CU takes fewer); without one, workgroup w takes w, w + G, .... For C -=
    // updates the tiles numbered G/2 .. G-1 run as two K halves, the second
    // when the workgroup has nothing else left, so the two workgroups of a
    // CU do not reach their epilogues together; the choice depends only on
    // tile numbers, so rounding does not depend on scheduling. An uncapped
    // launch has a workgroup per tile and splits none.
    __shared__ int next;
    const int G = gridDim.x;
    long first_r = -1, first_c = 0;  // this workgroup's deferred second half
    auto row_tiles = [&](int tr)
    {
        if (!p.lower)
            return gx;
        const long last = static_cast<long>(tr) * BM + (BM - 1) + p.diag_off;
        return last < 0 ? 0 : static_cast<int>(min(static_cast<long>(gx), last / BM + 1));
    };
    // one loop, one copy of the tile's code: with a copy for each way to take
    // a tile the kernel spilled 103 registers (now 32, around the epilogue)
    int tr = 0, row_first = 0, nc = gy > 0 ? row_tiles(0) : 0;  // the current tile row; tile numbers only grow
    for (int t = blockIdx.x;; t += G)
    {
        if (p.queue)
        {
            __syncthreads();  // the previous tile's `next` reads are done
            if (threadIdx.x == 0)
                next = atomicAdd(p.queue, 1);
            __syncthreads();
            t = __builtin_amdgcn_readfirstlane(next);
        }
        const bool done = t >= p.tiles;
        if (done && first_r < 0)
            break;
        long r0 = first_r, c0 = first_c;
        int part = 2, last = 2;  // with no other tile left: the deferred half
        if (!done)
        {
            while (t >= row_first + nc && tr + 1 < gy)
            {
                row_first += nc;
                nc = row_tiles(++tr);
            }
            r0 = static_cast<long>(tr) * BM;
            c0 = static_cast<long>(t - row_first) * BM;
            const bool whole = p.set || p.max_wgs <= 0 || t < G / 2 || t >= G;
            part = whole ? 0 : 1;
            last = part;
            if (!whole && first_r >= 0)
                last = 2;  // a second split tile for this workgroup: both halves now
            else if (!whole)
            {
                first_r = r0;
                first_c = c0;
            }
        }
        // the same for all lanes: the tile's addresses stay in scalar registers
        r0 = __builtin_amdgcn_readfirstlane(static_cast<int>(r0));
        c0 = __builtin_amdgcn_readfirstlane(static_cast<int>(c0));
        for (; part <= last; part++)
        {
            __syncthreads();  // the previous tile's last slab has been read by every wavefront
            gemm_tile32<Large, TC>(p, r0, c0, As, Bs, part);
        }
        if (done)
            break;
    }
}

// P[k][r] = (T) A[(r0 + r) * lda + p0 + k] for r < R, k < W, through a
// 64x64 LDS tile so both the FP64 reads and the k-major writes are coalesced;
// with `back`, the same FP64 values are also copied to back[r * ldback + k].
template <class T>
__global__ __launch_bounds__(THREADS) void k_panel_to_t(const double *__restrict__ A, long lda, long r0, long p0, int R, int W,
                                                         T *__restrict__ P, long ldp, double *__restrict__ back, long ldback)
{
    __shared__ T t[64][65];
    const long rb = static_cast<long>(blockIdx.x) * 64, kb = static_cast<long>(blockIdx.y) * 64;
    const int c = threadIdx.x & 63, q = threadIdx.x >> 6;
    for (int rr = q; rr < 64; rr += 4)
    {
        const long r = rb + rr, k = kb + c;
        const double v = (r < R && k < W) ? A[(r0 + r) * lda + p0 + k] : 0.0;
        t[rr][c] = static_cast<T>(v);
        if (back && r < R && k < W)
            back[r * ldback + k] = v;
    }
    __syncthreads();
    for (int kk = q; kk < 64; kk += 4)
    {
        const long k = kb + kk, r = rb + c;
        if (k < W && r < R)
            P[k * ldp + r] = t[c][kk];
    }
}

}  // namespace

template <class T>
static void panel_to_t(hipStream_t s, const double *A, long lda, long r0, long p0, int R, int W, T *P, long ldp, double *back, long ldback)
{
    require(R >= 0 && W >= 0 && ldp >= R, "panel copy: bad shape");
    if (R == 0 || W == 0)
        return;
    dim3 grid(static_cast<unsigned>(ceil_div(R, 64)), static_cast<unsigned>(ceil_div(W, 64)));
    require(grid.y <= 65535, "panel copy: panel too wide");
    require(!back || ldback >= W, "panel copy: bad copy-back layout");
    hipLaunchKernelGGL(k_panel_to_t<T>, grid, dim3(THREADS), 0, s, A, lda, r0, p0, R, W, P, ldp, back, ldback);
    GP_CHECK_LAUNCH();
}

void panel_to_f32t(hipStream_t s, const double *A, long lda, long r0, long p0, int R, int W, float *P, long ldp, double *back, long ldback)
{
    panel_to_t<float>(s, A, lda, r0, p0, R, W, P, ldp, back, ldback);
}

void panel_to_f64t(hipStream_t s, const double *A, long lda, long r0, long p0, int R, int W, double *P, long ldp, double *back, long ldback)
{
    panel_to_t<double>(s, A, lda, r0, p0, R, W, P, ldp, back, ldback);
}

template <class TC>
static void check_f32(const Params32<TC> &p)
{
    require(p.K % Large::BK == 0, "FP32 product: K must be a multiple of 16");
    require(p.M % 4 == 0 && p.N % 4 == 0 && p.lda % 4 == 0 && p.ldb % 4 == 0
                && reinterpret_cast<uintptr_t>(p.A) % 16 == 0 && reinterpret_cast<uintptr_t>(p.B) % 16 == 0,
            "FP32 product: operand rows must come in aligned groups of four");
    require(static_cast<long>(Large::BK) * std::max(p.lda, p.ldb) + BM < (1L << 31), "FP32 product: operand too tall");
}

void gemm_f32_trailing(hipStream_t s, const float *P, long ldp, long a_off, long b_off, double *C, long ldc, int M, int N, int K, long diag_off,
                       int max_wgs, int *queue)
{
    if (M <= 0 || N <= 0)
        return;
    Params32<double> p{ P + a_off, ldp, P + b_off, ldp, C, ldc, M, N, K, 1, diag_off, 0, max_wgs, 0, 0, queue, 0 };
    check_f32(p);
    const long gx = ceil_div(static_cast<long>(N), static_cast<long>(BM)), gy = ceil_div(static_cast<long>(M), static_cast<long>(BM));
    require(gx * gy < (1L << 31), "FP32 product: too many tiles for one launch");
    // tiles holding part of the update, counted as the capped kernel numbers them
    long active = 0;
    for (long tr = 0; tr < gy; tr++)
    {
        const long last = tr * BM + (BM - 1) + diag_off;
        active += last < 0 ? 0 : std::min(gx, last / BM + 1);
    }
    if (active == 0)
        return;
    require(active < (1L << 30), "FP32 product: too many tiles");
    p.tiles = static_cast<int>(active);
    if (p.max_wgs <= 0 || p.max_wgs >= active)
    {
        p.max_wgs = 0;  // no cap, or one that does not bind: one workgroup per tile
        p.queue = nullptr;
    }
    dim3 grid(static_cast<unsigned>(p.max_wgs > 0 ? p.max_wgs : p.tiles));
    hipLaunchKernelGGL(k_gemm_f32_tn<double>, grid, dim3(THREADS), 0, s, p);
    GP_CHECK_LAUNCH();
}

// The solves' products take 64x64 tiles where 128x128 ones would number at
// most this many. A diagonal step is 6 tile rows of 128 (72 tiles for 1536
// columns: under a third of the CUs, each alone with its 2048 matrix cycles
// per slab), and an update near the end of its sweep is as short; a quarter
// tile per workgroup fills the CUs and evens out the last wave. Above it the
// operands, read twice as often, cost more than the last wave does. Variance
// requests on MI355X (128x128 tiles only / small up to 400 / 1000 /
// 2000 / always): n = 12000, 300 columns 7.63 / 4.85 / 4.85 / 4.84 ms,
// 1500 columns 11.55 / 10.03 / 9.85 / 9.84, 8192 columns 42.4 / 41.7 / 41.6 /
// 41.7; n = 24000, 700 columns 22.95 / - / 18.58 / 18.24 / 18.26, 8192
// columns 155.9 / - / 155.8 / 155.4 / 158.1 (slabs still staged through
// registers; since then 4.46, 9.11, 38.8, 16.99 and 143.8). A diagonal step at 1536 columns
// went from 53 to 18 us, a third of that from leaving out the half of W_J
// that is zero.
constexpr long SMALL_TILE_LIMIT = 2048;

template <class S, int ROLE>
static void launch_solve(hipStream_t s, const Params32<float> &p)
{
    const long tiles = ceil_div(static_cast<long>(p.N), static_cast<long>(S::BM)) * ceil_div(static_cast<long>(p.M), static_cast<long>(S::BM));
    require(tiles < (1L << 31), "FP32 product: too many tiles for one launch");
    hipLaunchKernelGGL((k_gemm_f32_solve<S, ROLE>), dim3(static_cast<unsigned>(tiles)), dim3(THREADS), 0, s, p);
    GP_CHECK_LAUNCH();
}

void gemm_f32_tn(hipStream_t s, const float *A, long lda, const float *B, long ldb, float *C, long ldc, int M, int N, int K, bool set,
                 Triangle a)
{
    if (M <= 0 || N <= 0)
        return;
    Params32<float> p{ A, lda, B, ldb, C, ldc, M, N, K, 0, 0, set ? 1 : 0, 0, a == Triangle::Lower, a == Triangle::Upper, nullptr, 0 };
    check_f32(p);
    const long large = ceil_div(static_cast<long>(N), static_cast<long>(BM)) * ceil_div(static_cast<long>(M), static_cast<long>(BM));
    const bool small = K % Small::BK == 0 && large <= SMALL_TILE_LIMIT;
    if (set)
        small ? launch_solve<Small, 1>(s, p) : launch_solve<Large, 1>(s, p);
    else
        small ? launch_solve<Small, 2>(s, p) : launch_solve<Large, 2>(s, p);
}

}  // namespace gpamd::k
