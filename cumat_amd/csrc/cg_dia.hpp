// cg_dia.hpp -- the CG iteration's product with the matrix laid out by
// diagonals.
//
// A solve reads its matrix once per iteration, and at CG's sizes that read
// is what K1 costs: 8 bytes per stored FP32 entry (value and column index),
// LDS traffic to turn the entries' order into rows, and gathers of single p
// values. The matrices CG is used for mostly come from grids, whose entries
// lie on a few diagonals (5 and 7 points: 5 and 7, 27 points: 27). Such a
// matrix needs no column index at all: diagonal d of row i multiplies
// p[i + off[d]], a lane takes consecutive rows, and both the values and p
// are read with contiguous wide loads and no LDS.
//
// The solve lays the matrix out itself, on its own stream, once it is known
// to run for long enough: after every chunk of CG_CHUNK iterations from the
// second on, the last two residuals that the host has heard of tell how many more a solve at that rate needs (cg_dia_pays). Then
// cg_dia_detect_kernel collects the distinct offsets of a sample of rows and
// cg_dia_convert_kernel writes the diagonals, checking every stored entry. A
// chunk later, which is queued meanwhile, K1 uses the diagonals if every entry
// fitted. The residuals decide, not the clock, so a solve switches at the same
// iteration and gives the same bits every time. A row's products are added in ascending column
// order, as the CSR product adds them (with fused multiply-adds); slots that
// a row does not store hold 0 (their p is read inside the batch's own
// vector, so a batch never meets another's values).
//
// Detection and conversion take 28 + 110 us at 160^3 (the gain of 4 iterations),
// 17 + 6 at 512^2, 9 + 4 at 128^2; the detection of a matrix without diagonals
// 15. Queued after the first chunk of every solve they made short ones slower:
// 160^3 with 8 iterations 915 -> 1060 us, with 22 2140 -> 2290; now 915 and 2140
// (58 iterations: 5350 without the layout, 4190 with it from iteration 24 on,
// 4540 now, since the residuals of the first 24 foretell an earlier end).
#pragma once
#include <climits>
#include <cmath>

#include "cm_common.hpp"
#include "spmv_core.hpp"

namespace cm {

constexpr int CG_DIA_MAX = 32;     // diagonals
// Unknowns (n x batches) from which the three-launch form takes the layout:
// below, an iteration is three launches whatever K1 reads, and the layout's 40
// us stay (32^2 13.4 us per iteration without, 13.6 with, 200 iterations; two
// systems of 48^2 15.2 and 13.6).
constexpr long long CG_DIA_MIN = 2048;
constexpr int CG_DIA_SAMPLE = 2048;  // rows the detection looks at
constexpr int CG_DIA_DETECT_BS = 1024;
constexpr int CG_DIA_BS = 256;
// Iterations that have to be left, counted from the last residual that the host
// has heard of, for the layout to pay: 16 of them pass before it is in use, and
// the layout costs the gain of 4 (160^3) to about 40 (512^2, 13.8 and 13.3 us an
// iteration). From CG_DIA_LARGE unknowns on the bytes bind. A residual falls ever
// more slowly at first, so the prediction is short rather than long: at 160^3 a
// solve of 58 iterations counts as 17 more after 16.
constexpr int CG_DIA_PAYS = 64, CG_DIA_PAYS_LARGE = 16;
constexpr long long CG_DIA_LARGE = 1 << 19;

// Whether a solve that came from distance a to distance b (largest |r|^2 over
// the threshold) in one chunk needs 'pays' more iterations from b on at that
// rate. A residual that does not fall, and a tolerance of zero, mean yes.
inline bool cg_dia_pays(float a, float b, int pays)
{
    if (!(b < a)) return true;
    return !(CG_CHUNK * std::log((double)b) < pays * std::log((double)a / (double)b));
}

// What the detection found; written by the device into host-mapped memory
// (so that the host reads it without a copy) and into device memory (for
// the conversion, which is queued before the host knows).
struct DiaPlan {
    int count;  // distinct offsets, ascending in off; 0: more than CG_DIA_MAX, or too sparse
    int bad;    // the conversion met an entry outside the diagonals
    int ready;  // the conversion has ended (in the host's copy)
    int off[CG_DIA_MAX];
};

// The diagonals the two-launch form is built for (a row's operands stay in
// registers).
__host__ __device__ inline bool cg_dia_iter_takes(int count) { return count == 3 || count == 5 || count == 7; }

// One block: the distinct column - row offsets of at most CG_DIA_SAMPLE rows
// spread over the matrix, sorted. cap: elements of one batch's diagonals the
// conversion may write (rows padded to ld). Rows are far apart, so their pages
// cost most of the time. The loops stay rolled: the code runs
// once, and unrolled loads of eight entries, whose instructions have to be
// fetched too, took 24 and 40 us at 512^2 and 160^3.
static __global__ __launch_bounds__(CG_DIA_DETECT_BS) void cg_dia_detect_kernel(int n, const int* __restrict__ JA,
                                                                         const int* __restrict__ IA, long long ld,
                                                                         long long cap, int fused,
                                                                         DiaPlan* __restrict__ plan,
                                                                         DiaPlan* __restrict__ host)
{
    __shared__ int tab[CG_DIA_MAX];
    __shared__ int over;
    const int tid = threadIdx.x;
    if (tid < CG_DIA_MAX) tab[tid] = INT_MIN;
    if (tid == 0) over = 0;
    __syncthreads();
    const int ns = min(n, CG_DIA_SAMPLE);
    for (int s = tid; s < ns; s += CG_DIA_DETECT_BS) {
        const int row = ns > 1 ? (int)((long long)s * (n - 1) / (ns - 1)) : 0;
        const int b = JA[row], e = JA[row + 1];
        if (e - b > CG_DIA_MAX) {
            over = 1;
            continue;
        }
        for (int k = b; k < e; ++k) {
            const int o = IA[k] - row;
            int t = 0;
            for (; t < CG_DIA_MAX; ++t) {
                int cur = *(volatile int*)&tab[t];
                if (cur == INT_MIN) cur = atomicCAS(&tab[t], INT_MIN, o);
                if (cur == o || cur == INT_MIN) break;
                if (t == 8 && *(volatile int*)&over) break;
            }
            if (t == CG_DIA_MAX) over = 1;
        }
    }
    __syncthreads();
    if (tid >= 64) return;
    const int v = tid < CG_DIA_MAX ? tab[tid] : INT_MIN;
    int cnt = __popcll(__ballot(v != INT_MIN));
    if (over || cnt * ld > cap || (fused && !cg_dia_iter_takes(cnt))) cnt = 0;
    if (cnt && v != INT_MIN) {
        int rank = 0;
        for (int a = 0; a < CG_DIA_MAX; ++a) rank += tab[a] != INT_MIN && tab[a] < v;
        plan->off[rank] = host->off[rank] = v;
    }
    if (tid == 0) {
        plan->bad = host->bad = 0;
        plan->count = host->count = cnt;
    }
}

// dia[(b * count + d) * ld + i] = the entry of row i on diagonal d, 0 where
// the row stores none (and for i >= n). A row whose entries are not a
// strictly ascending subset of the plan's offsets marks the plan bad.
template <typename VT>
__global__ __launch_bounds__(CG_DIA_BS) void cg_dia_convert_kernel(int n, const int* __restrict__ JA,
                                                                   const int* __restrict__ IA,
                                                                   const VT* __restrict__ vals, long long vstride,
                                                                   long long ld, VT* __restrict__ dia, const DiaPlan* __restrict__ plan,
                                                                   DiaPlan* __restrict__ host)
{
    const long long i = (long long)blockIdx.x * CG_DIA_BS + threadIdx.x;
    const int cnt = plan->count;
    if (cnt == 0 || i >= ld) return;
    const VT* v = vals + blockIdx.y * vstride;
    VT* o = dia + blockIdx.y * (cnt * ld) + i;
    int k = i < n ? JA[i] : 0;
    const int e = i < n ? JA[i + 1] : 0;
    int c = k < e ? IA[k] : -1;
    for (int d = 0; d < cnt; ++d) {
        VT a = VT(0);
        if (k < e && c - (int)i == plan->off[d]) {
            a = v[k];
            ++k;
            c = k < e ? IA[k] : -1;
        }
        o[d * ld] = a;
    }
    if (k != e) host->bad = 1;
}

// Behind the conversion in the stream.
static __global__ void cg_dia_ready_kernel(DiaPlan* __restrict__ host) { host->ready = 1; }

// Arguments of the product: everything that does not change between
// iterations.
struct DiaArgs {
    int count;
    long long ld, bstride;  // elements between diagonals / between the batches' values (0: shared)
    int off[CG_DIA_MAX];
};

template <typename VT, typename T>
__device__ __forceinline__ T dia_value(VT v)
{
    return (T)v;
}
template <>
__device__ __forceinline__ float dia_value<unsigned short, float>(unsigned short v)
{
    return bf16_to_float(v);
}

// tmp = A p for NB consecutive batches that share the values, and their
// per-block partial p.tmp. A lane takes U rows CG_DIA_BS apart, so every load
// of a wavefront is 64 consecutive elements. D: the diagonals at compile time,
// or -CH for A.count of them in CH chains. Up to 8 entries the CSR product adds a
// row in one chain, and so does this; longer rows it adds in a wavefront's tree,
// and here the diagonals go round four chains, from 27 on eight (rms error in eps
// of the terms' magnitudes, uniform FP32 terms, CSR / one chain / four or eight:
// 13 diagonals 0.343 / 0.471 / 0.331, 21 0.362 / 0.598 / 0.346, 27 0.336 / 0.653 /
// 0.327, 32 0.343 / 0.698 / 0.339).
//
// Bound by the bytes: (values + p + Ap) of 160^3 with 7 diagonals are 148 MB.
// Measured on MI355X, us per launch, CSR product -> this one: 160^3 FP32
// 59.1 -> 24.5 (6.0 TB/s); 512^2 with 8 right-hand sides 16.9 -> 6.8; 16
// systems of 256^2 with their own values 10.7 -> 6.6 (the last two out of
// the last-level cache). Four consecutive rows per lane, 16-byte loads: 25.2,
// 16.8 and 13.2: p + off is then mostly not 16-byte aligned, and such loads
// run at a fraction of the rate. Rows per lane (whole solve, ms, U = 1 / 2 /
// 4): 160^3 73.6 / 73.5 / 72.3; 512^2 x 8 40.4 / 39.8 / 40.4; 16 x 256^2 41.9 /
// 42.8 / 43.9: four pay where a block still has several steps to take. Two
// batches per thread against one: 0.5 % of a solve; four: slower.
inline int cg_dia_chains(int count) { return count <= 8 ? 1 : (count <= 26 ? 4 : 8); }
template <typename VT, typename T, int D, int U, int NB>
__global__ __launch_bounds__(CG_DIA_BS) void cg_dia_kernel(int n, const DiaArgs A, const VT* __restrict__ dia,
                                                           const T* __restrict__ p, T* __restrict__ tmp,
                                                           T* __restrict__ part, CgState<T>* st,
                                                           const T* __restrict__ diag)
{
    const int b0 = blockIdx.y * NB;
    bool idle = true;
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        cg_k1_snapshot(st, b0 + q);
        idle = idle && batch_inactive(st, b0 + q);
    }
    if (idle) return;
    __shared__ T red[CG_DIA_BS / 64];
    const VT* db = dia + blockIdx.y * A.bstride;
    const T* pb = p + (long long)b0 * n;
    T* tb = tmp + (long long)b0 * n;
    constexpr int CH = D > 0 ? 1 : -D;          // chains of a row
    constexpr int STEP = CH > 4 ? CH : 4;       // diagonals whose loads are in flight together
    const int cnt = D > 0 ? D : A.count;
    T s[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) s[q] = T(0);
    for (RowBlockWalk w(blockIdx.x, gridDim.x, div_up_dev(n, CG_DIA_BS * U)); w.valid(); w.next()) {
        const long long first = (long long)w.cur * (CG_DIA_BS * U);
        const long long i = first + threadIdx.x;
        // the block's rows and every p they meet lie inside the vector
        const bool inside = first + A.off[0] >= 0 && first + CG_DIA_BS * U + A.off[cnt - 1] <= n &&
                            first + CG_DIA_BS * U <= n;
        if (inside) {
            T acc[NB][U][CH];
#pragma unroll
            for (int q = 0; q < NB; ++q)
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int k = 0; k < CH; ++k) acc[q][u][k] = T(0);
            auto add = [&](int d, int k) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const T a = dia_value<VT, T>(db[d * A.ld + i + u * CG_DIA_BS]);
#pragma unroll
                    for (int q = 0; q < NB; ++q)
                        acc[q][u][k] += a * pb[(long long)q * n + i + u * CG_DIA_BS + A.off[d]];
                }
            };
            if constexpr (D > 0) {
#pragma unroll
                for (int d = 0; d < D; ++d) add(d, 0);
            } else {
                int d = 0;
                for (; d + STEP <= cnt; d += STEP)
#pragma unroll
                    for (int k = 0; k < STEP; ++k) add(d + k, k % CH);
#pragma unroll
                for (int k = 0; k < STEP - 1; ++k)
                    if (d + k < cnt) add(d + k, k % CH);
            }
#pragma unroll
            for (int h = CH / 2; h > 0; h /= 2)
#pragma unroll
                for (int q = 0; q < NB; ++q)
#pragma unroll
                    for (int u = 0; u < U; ++u)
#pragma unroll
                        for (int k = 0; k < h; ++k) acc[q][u][k] += acc[q][u][k + h];
#pragma unroll
            for (int q = 0; q < NB; ++q)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const long long row = i + u * CG_DIA_BS;
                    const T own = pb[(long long)q * n + row];
                    if (diag) acc[q][u][0] += diag[row] * own;
                    tb[(long long)q * n + row] = acc[q][u][0];
                    s[q] += own * acc[q][u][0];
                }
        } else {
            for (int u = 0; u < U; ++u) {
                const long long row = i + u * CG_DIA_BS;
                if (row >= n) break;
#pragma unroll
                for (int q = 0; q < NB; ++q) {
                    T chain[CH];
#pragma unroll
                    for (int k = 0; k < CH; ++k) chain[k] = T(0);
                    for (int d0 = 0; d0 < cnt; d0 += CH)
#pragma unroll
                        for (int k = 0; k < CH; ++k) {
                            const int d = d0 + k;
                            if (d >= cnt) break;
                            // a slot the row does not store holds 0: any p of this vector will do
                            const long long col = min(max(row + A.off[d], 0ll), (long long)n - 1);
                            chain[k] += dia_value<VT, T>(db[d * A.ld + row]) * pb[(long long)q * n + col];
                        }
#pragma unroll
                    for (int h = CH / 2; h > 0; h /= 2)
#pragma unroll
                        for (int k = 0; k < h; ++k) chain[k] += chain[k + h];
                    T acc = chain[0];
                    const T own = pb[(long long)q * n + row];
                    if (diag) acc += diag[row] * own;
                    tb[(long long)q * n + row] = acc;
                    s[q] += own * acc;
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        const T v = block_reduce<OpSum, CG_DIA_BS>(s[q], red);
        if (threadIdx.x == 0) part[(long long)(b0 + q) * gridDim.x + blockIdx.x] = v;
    }
}

// Rows per lane: four from this many rows on, where a grid of CG_GMAX blocks
// still takes whole steps; below, two (more blocks).
constexpr int CG_DIA_U4_ROWS = 1 << 21;
inline int cg_dia_rows_per_block(int n) { return CG_DIA_BS * (n >= CG_DIA_U4_ROWS ? 4 : 2); }

template <typename VT, typename T, int D, int U>
static void launch_cg_dia_u(hipStream_t stream, int n, int B, int G, const DiaArgs& A, const VT* dia, const T* p,
                            T* tmp, T* part, CgState<T>* st, const T* diag)
{
    // batches that share the values in pairs: the values are read once for both
    if (!A.bstride && B % 2 == 0)
        cg_dia_kernel<VT, T, D, U, 2><<<dim3(G, B / 2), CG_DIA_BS, 0, stream>>>(n, A, dia, p, tmp, part, st, diag);
    else
        cg_dia_kernel<VT, T, D, U, 1><<<dim3(G, B), CG_DIA_BS, 0, stream>>>(n, A, dia, p, tmp, part, st, diag);
}

template <typename VT, typename T>
static void launch_cg_dia(hipStream_t stream, int n, int B, int G, const DiaArgs& A, const VT* dia, const T* p, T* tmp,
                          T* part, CgState<T>* st, const T* diag)
{
    const int chains = cg_dia_chains(A.count);
#define CM_DIA(U)                                                                                              \
    if (A.count == 5) launch_cg_dia_u<VT, T, 5, U>(stream, n, B, G, A, dia, p, tmp, part, st, diag);           \
    else if (A.count == 7) launch_cg_dia_u<VT, T, 7, U>(stream, n, B, G, A, dia, p, tmp, part, st, diag);      \
    else if (chains == 1) launch_cg_dia_u<VT, T, -1, U>(stream, n, B, G, A, dia, p, tmp, part, st, diag);      \
    else if (chains == 4) launch_cg_dia_u<VT, T, -4, U>(stream, n, B, G, A, dia, p, tmp, part, st, diag);      \
    else launch_cg_dia_u<VT, T, -8, U>(stream, n, B, G, A, dia, p, tmp, part, st, diag)
    if (n >= CG_DIA_U4_ROWS) {
        CM_DIA(4);
    } else {
        CM_DIA(2);
    }
#undef CM_DIA
}

}  // namespace cm
