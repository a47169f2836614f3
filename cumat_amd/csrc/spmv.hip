// spmv.hip -- CSR and ELLPACK sparse matrix-vector products and the Jacobi
// diagonal extraction.
//   CSR:     replaces CSRMVKernel_StaticBatches + ProductAssignment
//            (cuMat/src/SparseProductEvaluation.h:43-139)
//   ELLPACK: replaces ELLPACKMVKernel_StaticBatches
//            (cuMat/src/SparseProductEvaluation.h:194-324)
//   Jacobi:  replaces ExtractDiagonalOp over SparseMatrix::coeff +
//            cwiseInverseCheck (cuMat/src/ConjugateGradient.h:228-230)
#include "bcsr.hpp"
#include "spmv_core.hpp"
#include "spmv_wave.hpp"

#include <algorithm>
#include <type_traits>

namespace cm {

constexpr int SPMV_BS = 256;
constexpr int SPMV_EPT = 8;   // staged non-zeros per lane (8 per row on average)
// Vectors are multiplied together from this many (wavefronts x vectors) on; below,
// a launch of one vector each has more loads in flight. Us, apart / together:
// narrow rows (5 points) FP32 4 vectors of 200 k rows (12.5 k) 8.3 / 9.0, 3 of 400 k
// (18.8 k) 10.7 / 10.6; windows (1 to 39 entries) FP32 4 of 60 k (3.8 k) 13.2 / 17.5, 3
// of 100 k (4.7 k) 18.0 / 16.9, 8 of 60 k (7.5 k) 22.8 / 18.7, 27 points FP64 4 of 60 k
// 17.3 / 19.0, 3 of 100 k 21.6 / 19.6; ELLPACK (a thread takes a row) with 27 slots 4
// of 30 k (1.9 k) 12.0 / 11.5, 8 of 10 k (1.3 k) 7.3 / 9.0, 4 of 60 k (3.8 k) 13.4 / 11.8.
constexpr long long SPMV_MULTI_WAVES = 16384, SPMV_MULTI_WIDE = 4500, ELL_MULTI_WAVES = 3072;

template <typename VT, typename T>
__global__ __launch_bounds__(SPMV_BS) void csr_spmv_kernel(int rows, int cols, int nnz,
                                                           const int* __restrict__ JA,
                                                           const int* __restrict__ IA,
                                                           const VT* __restrict__ vals, int vals_batched,
                                                           const T* __restrict__ x, int x_batched,
                                                           T* __restrict__ y, int mode)
{
    constexpr int WPB = SPMV_BS / 64;
    __shared__ T lds[WPB][SPMV_EPT * 64];
    T* slice = lds[threadIdx.x >> 6];
    const int lane = threadIdx.x & 63;
    const int b = blockIdx.y;
    const VT* v = vals + (vals_batched ? (long long)b * nnz : 0);
    const T* xb = x + (x_batched ? (long long)b * cols : 0);
    T* yb = y + (long long)b * rows;
    ChunkWalk w(div_up_dev(rows, 64), WPB);
    if (!w.valid()) return;  // wave-uniform; no block barrier below
    WaveChunk<VT, SPMV_EPT> cur, nxt;
    chunk_load(cur, JA, IA, v, w.cur * 64, rows);
    for (;;) {
        const int nc = w.peek_next();
        const bool more = nc < w.hi;
        if (more) chunk_load(nxt, JA, IA, v, nc * 64, rows);  // in flight during the gathers below
        const T acc = chunk_compute<VT, T, SPMV_EPT>(cur, JA, IA, v, [xb](int c) { return xb[c]; }, slice);
        if (lane < cur.nr) {
            T* yy = yb + cur.r0 + lane;
            if (mode == CM_ASSIGN) __builtin_nontemporal_store(acc, yy);
            else *yy = assign_mode<T>(mode, *yy, acc);
        }
        if (!more) break;
        cur = nxt;
        w.next();
    }
}

// The product of NB vectors that share the matrix values (blockIdx.y counts
// groups of NB; the last group may hold fewer): the chunk's indices and values
// are read once and stay in registers while one vector after the other is
// gathered and summed. Same sums as csr_spmv_kernel. Measured on MI355X, us, a
// launch of one vector each / together: 1024^2 FP32 2 vectors 24.2 / 19.9, 4
// 45.1 / 29.2, 8 84.6 / 50.8; 100^3 FP64 7 points 3 vectors 64.3 / 39.9. One
// vector stays with csr_spmv_kernel: the same code here takes 68 registers
// instead of 62, one wavefront less per SIMD, and 62 us instead of 44 at 2048^2.
template <typename VT, typename T, int NB>
__global__ __launch_bounds__(SPMV_BS, sizeof(T) == 4 ? 8 : 4) void csr_spmv_multi_kernel(int rows, int cols, int batches,
                                                           const int* __restrict__ JA,
                                                           const int* __restrict__ IA,
                                                           const VT* __restrict__ vals,
                                                           const T* __restrict__ x, T* __restrict__ y, int mode)
{
    constexpr int WPB = SPMV_BS / 64;
    __shared__ T lds[WPB][SPMV_EPT * 64];
    T* slice = lds[threadIdx.x >> 6];
    const int lane = threadIdx.x & 63;
    const int b0 = blockIdx.y * NB;
    const int nb = NB == 1 ? 1 : min(NB, batches - b0);  // a vector past the last one repeats the group's first
    const VT* v = vals;
    const T* xb = x + (long long)b0 * cols;
    T* yb = y + (long long)b0 * rows;
    ChunkWalk w(div_up_dev(rows, 64), WPB);
    if (!w.valid()) return;  // wave-uniform; no block barrier below
    WaveChunk<VT, SPMV_EPT> cur, nxt;
    chunk_load(cur, JA, IA, v, w.cur * 64, rows);
    for (;;) {
        const int nc = w.peek_next();
        const bool more = nc < w.hi;
        if (more) chunk_load(nxt, JA, IA, v, nc * 64, rows);  // in flight during the gathers below
        T acc[NB];
        chunk_compute_multi<VT, T, SPMV_EPT, NB>(
            cur, JA, IA, v, [=](int b, int c) { return xb[(b < nb ? (long long)b * cols : 0) + c]; }, slice, acc);
        if (lane < cur.nr) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if (b >= nb) break;
                T* yy = yb + (long long)b * rows + cur.r0 + lane;
                if (mode == CM_ASSIGN) __builtin_nontemporal_store(acc[b], yy);
                else *yy = assign_mode<T>(mode, *yy, acc[b]);
            }
        }
        if (!more) break;
        cur = nxt;
        w.next();
    }
}

// Rows of more than SPMV_EPT entries on average: every chunk of 64 rows is
// taken in windows of SPMV_EPT * 64 entries. Chunks with a row of more than
// SPMV_ROW_MAX entries go row by row: one lane would add such a row while the
// others wait, and beyond 64 entries its error would exceed the row by row
// form's (chunk_windows).
//
// Row by row, a row of 27 entries is one load per lane, 37 lanes idle, and a
// wave reduction; the next row's loads wait for it. Measured on MI355X, us, row
// by row / windows: 27 points, 572 k rows, FP64 136 / 45.5 (one vector), 332 /
// 67.3 (three, the windows read once for all), FP32 107 / 34.1; 200 k rows of 1
// to 39 entries FP32 41.5 / 19.3. Without the next window's loads in flight
// 54.8, 78.8, 46.5 and 23.8.
//
// A window holds 512 / L rows of L entries, so that many lanes add while the
// others wait: with L the windows' instructions grow, and once the wavefronts
// fill the chip (SPMV_CROWD) those count. Us, row by row / windows, one vector
// of 400 k rows: FP32 L = 32 63 / 60, 40 73 / 71, 48 83 / 88, 64 106 / 123; FP64 48
// 127 / 115. Three vectors apart, 5.4 M entries: FP32 27 91 / 64, 32 60 / 65, 48 55 /
// 72, FP64 40 104 / 92, 48 96 / 94, 64 62 / 88. Hence the limits on a chunk's mean.
// Fewer wavefronts wait for memory (one vector of 5.4 M entries FP32 48 38 / 26),
// and vectors together share the loads (three of 400 k rows FP32 48 234 / 172, FP64 64
// 341 / 319).
constexpr int SPMV_ROW_MAX = 64;
constexpr long long SPMV_CROWD = 3072;
template <typename T> constexpr int SPMV_CROWD_MEAN = sizeof(T) == 8 ? 44 : 30;
template <typename VT, typename T, int NB>
__global__ __launch_bounds__(SPMV_BS) void csr_spmv_wide_kernel(int rows, int cols, int nnz, int batches,
                                                                const int* __restrict__ JA,
                                                                const int* __restrict__ IA,
                                                                const VT* __restrict__ vals, int vals_batched,
                                                                const T* __restrict__ x, int x_batched,
                                                                T* __restrict__ y, int mode, int window_max)
{
    constexpr int WPB = SPMV_BS / 64;
    __shared__ T lds[WPB][SPMV_EPT * 64 + 8];
    T* slice = lds[threadIdx.x >> 6];
    const int lane = threadIdx.x & 63;
    const int b0 = blockIdx.y * NB;
    const int nb = NB == 1 ? 1 : min(NB, batches - b0);
    const VT* v = vals + (vals_batched ? (long long)b0 * nnz : 0);
    const T* xb = x + (x_batched ? (long long)b0 * cols : 0);
    T* yb = y + (long long)b0 * rows;
    auto xg = [=](int b, int c) { return xb[(b < nb ? (long long)b * cols : 0) + c]; };
    for (ChunkWalk w(div_up_dev(rows, 64), WPB); w.valid(); w.next()) {
        const int r0 = w.cur * 64, nr = min(64, rows - r0);
        const int s = JA[r0], e = JA[r0 + nr];
        const int rb = lane < nr ? JA[r0 + lane] : 0, re = lane < nr ? JA[r0 + lane + 1] : 0;
        T acc[NB];
        if (e - s <= window_max && wave_reduce<OpMax>(re - rb) <= SPMV_ROW_MAX)
            chunk_windows<VT, T, SPMV_EPT, NB>(s, e, rb, re, IA, v, xg, slice, acc);
        else
            chunk_rows<VT, T, NB>(nr, rb, re, IA, v, xg, acc);
        if (lane < nr) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if (b >= nb) break;
                T* yy = yb + (long long)b * rows + r0 + lane;
                if (mode == CM_ASSIGN) __builtin_nontemporal_store(acc[b], yy);
                else *yy = assign_mode<T>(mode, *yy, acc[b]);
            }
        }
    }
}

// ELLPACK kernels: NB vectors that share the matrix values are multiplied
// together (blockIdx.y counts groups; the last may hold fewer), so a slot's
// index and value are read once for them; same sums as one vector at a time.
// Measured on MI355X, us: 1000^2 5 slots FP32 8 vectors 65 -> 29, 80^3 27
// slots FP64 4 vectors 125 -> 57.

// Rows of at most MAXW slots: every slot's index and value load is issued
// at once, then the gathers, then the adds in slot order (the same sums as
// ell_spmv_kernel; 2048^2 width 5: 36.3 -> 34.6 us).
template <typename T, int MAXW, int NB>
__global__ void ell_spmv_w_kernel(int rows, int cols, int npr, int batches, const int* __restrict__ idx,
                                  const T* __restrict__ vals, int vals_batched, const T* __restrict__ x,
                                  int x_batched, T* __restrict__ y, int mode)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const int b0 = blockIdx.y * NB;
    const int nb = NB == 1 ? 1 : min(NB, batches - b0);
    const T* v = vals + (vals_batched ? (long long)b0 * rows * npr : 0);
    const T* xb = x + (x_batched ? (long long)b0 * cols : 0);
    int c[MAXW];
    T a[MAXW], g[MAXW];
#pragma unroll
    for (int j = 0; j < MAXW; ++j) {
        const bool ok = j < npr;  // uniform
        c[j] = ok ? __builtin_nontemporal_load(idx + r + (long long)rows * j) : -1;
        a[j] = ok ? __builtin_nontemporal_load(v + r + (long long)rows * j) : T(0);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (b >= nb) break;
        const T* xv = xb + (long long)b * cols;
#pragma unroll
        for (int j = 0; j < MAXW; ++j) g[j] = c[j] >= 0 ? xv[c[j]] : T(0);
        T acc = T(0);
#pragma unroll
        for (int j = 0; j < MAXW; ++j)
            if (c[j] >= 0) acc += a[j] * g[j];
        T* yy = y + r + (long long)rows * (b0 + b);
        *yy = (mode == CM_ASSIGN) ? acc : assign_mode<T>(mode, *yy, acc);
    }
}

template <typename T, int NB>
__global__ void ell_spmv_kernel(int rows, int cols, int npr, int batches, const int* __restrict__ idx,
                                const T* __restrict__ vals, int vals_batched,
                                const T* __restrict__ x, int x_batched, T* __restrict__ y, int mode)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const int b0 = blockIdx.y * NB;
    const int nb = NB == 1 ? 1 : min(NB, batches - b0);  // a vector past the last one repeats the group's first
    const T* v = vals + (vals_batched ? (long long)b0 * rows * npr : 0);
    const T* xb = x + (x_batched ? (long long)b0 * cols : 0);
    T acc[NB];
    const T* xv[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        acc[b] = T(0);
        xv[b] = xb + (b < nb ? (long long)b * cols : 0);
    }
    // column-major: the k-th entries of consecutive rows are contiguous.
    // Four entries' index and value loads are issued together (streamed
    // once: non-temporal), then gathered and added in k order, skipping
    // padding (index < 0)
    int k = 0;
    for (; k + 4 <= npr; k += 4) {
        int c[4];
        T a[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            c[j] = __builtin_nontemporal_load(idx + r + (long long)rows * (k + j));
            a[j] = __builtin_nontemporal_load(v + r + (long long)rows * (k + j));
        }
        T g[NB][4];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int j = 0; j < 4; ++j) g[b][j] = c[j] >= 0 ? xv[b][c[j]] : T(0);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (c[j] >= 0) acc[b] += a[j] * g[b][j];
    }
    for (; k < npr; ++k) {
        const int c = idx[r + (long long)rows * k];
        if (c < 0) continue;
        const T a = v[r + (long long)rows * k];
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] += a * xv[b][c];
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (b >= nb) break;
        T* yy = y + r + (long long)rows * (b0 + b);
        *yy = (mode == CM_ASSIGN) ? acc[b] : assign_mode<T>(mode, *yy, acc[b]);
    }
}

template <typename T>
__global__ void csr_inverse_diagonal_kernel(int rows, int nnz, const int* __restrict__ JA,
                                            const int* __restrict__ IA, const T* __restrict__ vals,
                                            int vals_batched, T* __restrict__ inv)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const int b = blockIdx.y;
    const T* v = vals + (vals_batched ? (long long)b * nnz : 0);
    T d = T(0);
    for (int k = JA[r]; k < JA[r + 1]; ++k)
        if (IA[k] == r) { d = v[k]; break; }
    inv[r + (long long)rows * b] = (d == T(0)) ? T(1) : T(1) / d;
}

template <typename VT, typename T>
static int launch_csr(cm_ctx_t ctx, int rows, int cols, int nnz, int batches, const int* JA,
                      const int* IA, const void* vals, int vb, const void* x, int xb, void* y, int mode)
{
    // grid cap: 8 resident blocks per CU (the wave limit at 256 threads);
    // CUMAT_SPMV_GRID overrides it for tuning sweeps
    static const int gmax = [] {
        const char* s = getenv("CUMAT_SPMV_GRID");
        return (s && atoi(s) >= 8) ? atoi(s) : 2048;
    }();
    const int g = walk_grid(div_up(div_up(rows, 64), SPMV_BS / 64), gmax);
    // more entries than a chunk holds: the windows
    const bool wide = nnz > (long long)SPMV_EPT * rows;
#define CM_WIDE(NB)                                                                                             \
    csr_spmv_wide_kernel<VT, T, NB><<<dim3(g, (batches + NB - 1) / NB), SPMV_BS, 0, ctx->stream>>>(             \
        rows, cols, nnz, batches, JA, IA, (const VT*)vals, vb, (const T*)x, xb, (T*)y, mode, window_max)
#define CM_MULTI(NB)                                                                                            \
    csr_spmv_multi_kernel<VT, T, NB><<<dim3(g, (batches + NB - 1) / NB), SPMV_BS, 0, ctx->stream>>>(            \
        rows, cols, batches, JA, IA, (const VT*)vals, (const T*)x, (T*)y, mode)
    // vectors that share the values are multiplied together, as long as the
    // groups still fill the chip (a wavefront takes 64 rows)
    const long long waves = (long long)div_up(rows, 64) * batches;
    const int nb = (vb || !xb || waves < (wide ? SPMV_MULTI_WIDE : SPMV_MULTI_WAVES)) ? 1 : std::min(batches, 4);
    const int window_max = 64 * (nb == 1 && waves >= SPMV_CROWD ? SPMV_CROWD_MEAN<T> : SPMV_ROW_MAX);
    if (nb == 1 && wide) CM_WIDE(1);
    else if (nb == 1)
        csr_spmv_kernel<VT, T><<<dim3(g, batches), SPMV_BS, 0, ctx->stream>>>(
            rows, cols, nnz, JA, IA, (const VT*)vals, vb, (const T*)x, xb, (T*)y, mode);
    else if (nb == 2 && wide) CM_WIDE(2);
    else if (nb == 2) CM_MULTI(2);
    else if (nb == 3 && wide) CM_WIDE(3);
    else if (nb == 3) CM_MULTI(3);
    else if (wide) CM_WIDE(4);
    else CM_MULTI(4);
#undef CM_WIDE
#undef CM_MULTI
    CM_LAUNCH_CHECK();
    return CM_OK;
}

template <typename T, int NB>
static void launch_ell_nb(cm_ctx_t ctx, int rows, int cols, int npr, int batches, const int* idx, const void* vals,
                          int vb, const void* x, int xb, void* y, int mode)
{
    const dim3 grid(div_up(rows, 256), (batches + NB - 1) / NB);
    if constexpr (std::is_same<T, float>::value)
        if (npr <= 8) {
            ell_spmv_w_kernel<T, 8, NB><<<grid, 256, 0, ctx->stream>>>(rows, cols, npr, batches, idx, (const T*)vals,
                                                                       vb, (const T*)x, xb, (T*)y, mode);
            return;
        }
    ell_spmv_kernel<T, NB><<<grid, 256, 0, ctx->stream>>>(rows, cols, npr, batches, idx, (const T*)vals, vb,
                                                          (const T*)x, xb, (T*)y, mode);
}

template <typename T>
static void launch_ell(cm_ctx_t ctx, int rows, int cols, int npr, int batches, const int* idx, const void* vals,
                       int vb, const void* x, int xb, void* y, int mode)
{
    // together where the groups still fill the chip (as the CSR product; a thread takes a row)
    const bool multi = !vb && xb && (long long)rows * batches >= 64 * ELL_MULTI_WAVES;
    const int nb = multi ? std::min(batches, 4) : 1;
    if (nb == 4) launch_ell_nb<T, 4>(ctx, rows, cols, npr, batches, idx, vals, vb, x, xb, y, mode);
    else if (nb == 3) launch_ell_nb<T, 3>(ctx, rows, cols, npr, batches, idx, vals, vb, x, xb, y, mode);
    else if (nb == 2) launch_ell_nb<T, 2>(ctx, rows, cols, npr, batches, idx, vals, vb, x, xb, y, mode);
    else launch_ell_nb<T, 1>(ctx, rows, cols, npr, batches, idx, vals, vb, x, xb, y, mode);
}

}  // namespace cm

extern "C" {

int cm_csr_spmv(cm_ctx_t ctx, int val_dtype, int vec_dtype, int rows, int cols, int nnz, int batches,
                const int* JA, const int* IA, const void* vals, int vals_batched, const void* x,
                int x_batched, void* y, int mode)
{
    CM_API_BEGIN
    CM_TRY(cm::resolve(ctx, &ctx));
    CM_REQUIRE(rows >= 0 && cols >= 0 && nnz >= 0 && batches >= 1, CM_E_DIM,
               "cm_csr_spmv: bad sizes rows=%d cols=%d nnz=%d batches=%d", rows, cols, nnz, batches);
    CM_REQUIRE(mode >= CM_ASSIGN && mode <= CM_OR, CM_E_ARG, "cm_csr_spmv: bad mode %d", mode);
    cm::count(CM_CNT_EVAL_MATMUL_SPARSE);
    cm::count(CM_CNT_EVAL_ANY);
    if (rows == 0) return CM_OK;
    CM_REQUIRE(JA && y && (nnz == 0 || (IA && vals && x)), CM_E_ARG, "cm_csr_spmv: NULL pointer");
    if (val_dtype == CM_F32 && vec_dtype == CM_F32)
        return cm::launch_csr<float, float>(ctx, rows, cols, nnz, batches, JA, IA, vals, vals_batched, x,
                                            x_batched, y, mode);
    if (val_dtype == CM_F64 && vec_dtype == CM_F64)
        return cm::launch_csr<double, double>(ctx, rows, cols, nnz, batches, JA, IA, vals, vals_batched, x,
                                              x_batched, y, mode);
    if (val_dtype == CM_I32 && vec_dtype == CM_I32)
        return cm::launch_csr<int, int>(ctx, rows, cols, nnz, batches, JA, IA, vals, vals_batched, x,
                                        x_batched, y, mode);
    if (val_dtype == CM_BF16 && vec_dtype == CM_F32)
        return cm::launch_csr<unsigned short, float>(ctx, rows, cols, nnz, batches, JA, IA, vals,
                                                     vals_batched, x, x_batched, y, mode);
    return cm::fail(CM_E_UNSUPPORTED, "cm_csr_spmv: unsupported dtype pair (%d,%d)", val_dtype, vec_dtype);
    CM_API_END
}

int cm_ell_spmv(cm_ctx_t ctx, int dtype, int rows, int cols, int nnz_per_row, int batches,
                const int* indices, const void* vals, int vals_batched, const void* x, int x_batched,
                void* y, int mode)
{
    CM_API_BEGIN
    CM_TRY(cm::resolve(ctx, &ctx));
    CM_REQUIRE(rows >= 0 && cols >= 0 && nnz_per_row >= 0 && batches >= 1, CM_E_DIM,
               "cm_ell_spmv: bad sizes");
    CM_REQUIRE(mode >= CM_ASSIGN && mode <= CM_OR, CM_E_ARG, "cm_ell_spmv: bad mode %d", mode);
    cm::count(CM_CNT_EVAL_MATMUL_SPARSE);
    cm::count(CM_CNT_EVAL_ANY);
    if (rows == 0) return CM_OK;
    if (dtype == CM_F32)
        cm::launch_ell<float>(ctx, rows, cols, nnz_per_row, batches, indices, vals, vals_batched, x, x_batched, y, mode);
    else if (dtype == CM_F64)
        cm::launch_ell<double>(ctx, rows, cols, nnz_per_row, batches, indices, vals, vals_batched, x, x_batched, y, mode);
    else if (dtype == CM_I32)
        cm::launch_ell<int>(ctx, rows, cols, nnz_per_row, batches, indices, vals, vals_batched, x, x_batched, y, mode);
    else
        return cm::fail(CM_E_UNSUPPORTED, "cm_ell_spmv: unsupported dtype %d", dtype);
    CM_LAUNCH_CHECK();
    return CM_OK;
    CM_API_END
}

int cm_csr_inverse_diagonal(cm_ctx_t ctx, int dtype, int rows, int nnz, int batches, const int* JA,
                            const int* IA, const void* vals, int vals_batched, void* invdiag)
{
    CM_API_BEGIN
    CM_TRY(cm::resolve(ctx, &ctx));
    CM_REQUIRE(rows >= 0 && batches >= 1, CM_E_DIM, "cm_csr_inverse_diagonal: bad sizes");
    cm::count(CM_CNT_EVAL_CWISE);
    cm::count(CM_CNT_EVAL_ANY);
    if (rows == 0) return CM_OK;
    dim3 grid(cm::div_up(rows, 256), vals_batched ? batches : 1);
    if (dtype == CM_F32)
        cm::csr_inverse_diagonal_kernel<float><<<grid, 256, 0, ctx->stream>>>(
            rows, nnz, JA, IA, (const float*)vals, vals_batched, (float*)invdiag);
    else if (dtype == CM_F64)
        cm::csr_inverse_diagonal_kernel<double><<<grid, 256, 0, ctx->stream>>>(
            rows, nnz, JA, IA, (const double*)vals, vals_batched, (double*)invdiag);
    else
        return cm::fail(CM_E_UNSUPPORTED, "cm_csr_inverse_diagonal: unsupported dtype %d", dtype);
    CM_LAUNCH_CHECK();
    return CM_OK;
    CM_API_END
}

int cm_bcsr_spmv(cm_ctx_t ctx, int block_dim, int rows, int cols, int nnz, int batches, const int* JA,
                 const int* IA, const float* vals, int vals_batched, const float* x, int x_batched, float* y,
                 int mode)
{
    CM_API_BEGIN
    CM_TRY(cm::resolve(ctx, &ctx));
    CM_REQUIRE(block_dim >= 2 && block_dim <= 4, CM_E_UNSUPPORTED, "cm_bcsr_spmv: block dimension %d (2..4)",
               block_dim);
    CM_REQUIRE(rows >= 0 && cols >= 0 && nnz >= 0 && batches >= 1 && batches <= 65535, CM_E_DIM,
               "cm_bcsr_spmv: bad sizes rows=%d cols=%d nnz=%d batches=%d (1..65535)", rows, cols, nnz, batches);
    CM_REQUIRE(mode >= CM_ASSIGN && mode <= CM_DIV, CM_E_ARG, "cm_bcsr_spmv: bad mode %d", mode);
    cm::count(CM_CNT_EVAL_MATMUL_SPARSE);
    cm::count(CM_CNT_EVAL_ANY);
    if (rows == 0) return CM_OK;
    CM_REQUIRE(JA && y && (nnz == 0 || (IA && vals && x)), CM_E_ARG, "cm_bcsr_spmv: NULL pointer");
    CM_REQUIRE((((uintptr_t)vals | (uintptr_t)x | (uintptr_t)y) & 15) == 0, CM_E_ARG,
               "cm_bcsr_spmv: blocks and vectors must be 16-byte aligned (float4 entries)");
    cm::launch_bcsr_spmv(ctx->stream, block_dim, rows, batches, JA, IA, (const cm::bc_f4*)vals,
                         vals_batched ? (long long)nnz * block_dim : 0, (const cm::bc_f4*)x,
                         x_batched ? (long long)cols : 0, (cm::bc_f4*)y, mode);
    CM_LAUNCH_CHECK();
    return CM_OK;
    CM_API_END
}

int cm_bcsr_inverse_diagonal(cm_ctx_t ctx, int block_dim, int rows, int nnz, int batches, const int* JA,
                             const int* IA, const float* vals, int vals_batched, float* invdiag)
{
    CM_API_BEGIN
    CM_TRY(cm::resolve(ctx, &ctx));
    CM_REQUIRE(block_dim >= 2 && block_dim <= 4, CM_E_UNSUPPORTED,
               "cm_bcsr_inverse_diagonal: block dimension %d (2..4)", block_dim);
    CM_REQUIRE(rows >= 0 && nnz >= 0 && batches >= 1 && batches <= 65535, CM_E_DIM,
               "cm_bcsr_inverse_diagonal: bad sizes");
    cm::count(CM_CNT_EVAL_CWISE);
    cm::count(CM_CNT_EVAL_ANY);
    if (rows == 0) return CM_OK;
    CM_REQUIRE(JA && invdiag && (nnz == 0 || (IA && vals)), CM_E_ARG, "cm_bcsr_inverse_diagonal: NULL pointer");
    CM_REQUIRE((((uintptr_t)vals | (uintptr_t)invdiag) & 15) == 0, CM_E_ARG,
               "cm_bcsr_inverse_diagonal: blocks and entries must be 16-byte aligned");
    cm::launch_bcsr_invdiag(ctx->stream, block_dim, rows, vals_batched ? batches : 1, JA, IA,
                            (const cm::bc_f4*)vals, vals_batched ? (long long)nnz * block_dim : 0,
                            (cm::bc_f4*)invdiag);
    CM_LAUNCH_CHECK();
    return CM_OK;
    CM_API_END
}

}  // extern "C"
