// spmv_wave.hpp -- wavefront-level, software-pipelined CSR SpMV core.
//
// The unit of work is a chunk of 64 consecutive rows owned by one wavefront
// (lane l sums row r0 + l). For a chunk whose non-zeros fit the lane budget
// (EPT per lane, i.e. EPT average non-zeros per row), the wavefront
//   1. loads the chunk's column indices and values with fully coalesced
//      loads, EPT per lane, plus each lane's row bounds;
//   2. gathers x at those columns and parks the products in its private LDS
//      slice (no workgroup barrier: only this wavefront touches the slice);
//   3. sums each lane's row sequentially in CSR order (the reference's
//      summation order, cuMat/src/SparseProductEvaluation.h:55-87).
// Step 1 of the NEXT chunk is issued before steps 2-3 of the current one, so
// index/value loads of one chunk overlap the gathers of the previous one and
// every wavefront keeps two chunks of loads in flight.
// Chunks with more non-zeros fall back to one row at a time per wavefront
// (chunk_rows); a matrix with many of them has a kernel of its own
// (chunk_windows).
// Chunks are assigned so that each XCD owns a contiguous range of rows:
// stencil neighbours of a chunk are then resident in the same L2.
#pragma once
#include "cm_common.hpp"

namespace cm {

template <typename VT, int EPT>
struct WaveChunk {
    int r0, nr, s, e;
    int rb, re;  // this lane's row bounds
    int col[EPT];
    VT v[EPT];
};

// Chunk walk of one wavefront over NC chunks: XCD x (= block % 8) owns chunks
// [x*NC/8, (x+1)*NC/8); its GW/8 wavefronts stride through that range.
struct ChunkWalk {
    int cur, hi, step;
    __device__ ChunkWalk(int NC, int waves_per_block)
    {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int G = gridDim.x;                  // multiple of 8
        const int x = blockIdx.x & 7;
        const int lw = (blockIdx.x >> 3) * waves_per_block + wave;
        const int lo = (int)(((long long)NC * x) >> 3);
        hi = (int)(((long long)NC * (x + 1)) >> 3);
        step = (G >> 3) * waves_per_block;
        cur = lo + lw;
    }
    __device__ bool valid() const { return cur < hi; }
    __device__ int peek_next() const { return cur + step; }
    __device__ void next() { cur += step; }
};

template <bool NT, typename X>
__device__ __forceinline__ X ld_matrix(const X* p)
{
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}

// NT: which matrix streams are loaded non-temporally (streaming: bit 0 the
// column indices, bit 1 the values). A single product streams a matrix that
// is not read again soon; an iterative solver reads the same matrix every
// iteration, and plain loads let the 256 MB last-level cache keep part of it
// from one iteration to the next.
template <typename VT, int EPT, int NT = 3>
__device__ __forceinline__ void chunk_load(WaveChunk<VT, EPT>& C, const int* __restrict__ JA,
                                           const int* __restrict__ IA, const VT* __restrict__ vals, int r0,
                                           int nrows)
{
    const int lane = threadIdx.x & 63;
    C.r0 = r0;
    C.nr = min(64, nrows - r0);
    C.s = JA[r0];
    C.e = JA[r0 + C.nr];
    C.rb = (lane < C.nr) ? JA[r0 + lane] : 0;
    C.re = (lane < C.nr) ? JA[r0 + lane + 1] : 0;
    if (C.e - C.s <= EPT * 64) {
#pragma unroll
        for (int j = 0; j < EPT; ++j) {
            const int k = C.s + lane + 64 * j;
            const bool ok = k < C.e;
            C.col[j] = ok ? ld_matrix<(NT & 1) != 0>(IA + k) : 0;
            C.v[j] = ok ? ld_matrix<(NT & 2) != 0>(vals + k) : VT(0);
        }
    }
}

// A chunk one row at a time (lanes stride the row, fixed-order DPP reduction),
// for the NB vectors xg(b, col): an entry is read once and multiplied with all
// of them. Row lane: entries [rb, re); out[b] is (A x_b)[row lane].
//
// Long rows are one chain of loads per wavefront, so four steps' loads are in
// flight. Measured on MI355X, us, 400 k rows of 5 entries and a hundred of 20000,
// three vectors, a launch of one vector each / one vector after the other / this:
// FP32 150 / 330 / 151, FP64 171 / 450 / 173; one vector 132 -> 63 and 153 -> 86.
template <typename VT, typename T, int NB, typename XG>
__device__ __forceinline__ void chunk_rows(int nr, int rb, int re, const int* __restrict__ IA,
                                           const VT* __restrict__ vals, XG xg, T (&out)[NB])
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int b = 0; b < NB; ++b) out[b] = T(0);
    for (int i = 0; i < nr; ++i) {
        const int a = __builtin_amdgcn_readlane(rb, i), e = __builtin_amdgcn_readlane(re, i);
        T s[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) s[b] = T(0);
        int k = a + lane;
        // four steps' loads in flight, added in the same order
        for (; k - lane + 256 <= e; k += 256) {
            int c[4];
            T v[4], x[NB][4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                c[u] = IA[k + 64 * u];
                v[u] = Load<VT, T>::get(vals, k + 64 * u);
            }
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int u = 0; u < 4; ++u) x[b][u] = xg(b, c[u]);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int u = 0; u < 4; ++u) s[b] += v[u] * x[b][u];
        }
        for (; k < e; k += 64) {
            const int c = IA[k];
            const T v = Load<VT, T>::get(vals, k);
#pragma unroll
            for (int b = 0; b < NB; ++b) s[b] += v * xg(b, c);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const T r = wave_reduce<OpSum>(s[b]);
            if (lane == i) out[b] = r;
        }
    }
}

// The same through windows of EPT * 64 entries: a window's entries are loaded
// and multiplied like a narrow chunk's, and a lane adds the part of its row
// that lies in the window. Row lane: entries [rb, re). slice: EPT * 64 + 8
// elements.
//
// A row is added in blocks of eight, each a tree, and a window's blocks go round
// four partial sums. In one chain each of four, as before, the error grew with the
// row: rms in eps of the sum of the terms' magnitudes, FP32, row by row / four
// chains / this: uniform terms 32 entries 0.347 / 0.370 / 0.347, 64 0.347 / 0.405
// / 0.347; normal 32 0.150 / 0.163 / 0.150, 64 0.116 / 0.145 / 0.116.
template <typename VT, typename T, int EPT, int NB, typename XG>
__device__ __forceinline__ void chunk_windows(int s, int end, int rb, int re, const int* __restrict__ IA,
                                              const VT* __restrict__ vals, XG xg, T* slice, T (&out)[NB])
{
    constexpr int WIN = EPT * 64;
    const int lane = threadIdx.x & 63;
    T part[NB][4];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q) part[b][q] = T(0);
    int ncol[EPT];
    VT nv[EPT];
    auto load = [&](int w0) {
#pragma unroll
        for (int j = 0; j < EPT; ++j) {
            const int k = w0 + lane + 64 * j;
            const bool ok = k < end;
            ncol[j] = ok ? __builtin_nontemporal_load(IA + k) : 0;
            nv[j] = ok ? __builtin_nontemporal_load(vals + k) : VT(0);
        }
    };
    load(s);
    for (int w0 = s; w0 < end; w0 += WIN) {
        int col[EPT];
        VT v[EPT];
#pragma unroll
        for (int j = 0; j < EPT; ++j) {
            col[j] = ncol[j];
            v[j] = nv[j];
        }
        if (w0 + WIN < end) load(w0 + WIN);  // in flight during this window's gathers
        const int a = max(rb, w0) - w0, e = min(re, w0 + WIN) - w0;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            T xv[EPT];
#pragma unroll
            for (int j = 0; j < EPT; ++j) xv[j] = (w0 + lane + 64 * j < end) ? xg(b, col[j]) : T(0);
#pragma unroll
            for (int j = 0; j < EPT; ++j) slice[lane + 64 * j] = Load<VT, T>::get(v, j) * xv[j];
            __builtin_amdgcn_wave_barrier();  // as in chunk_compute
            auto four = [&](int k) { return (slice[k] + slice[k + 1]) + (slice[k + 2] + slice[k + 3]); };
            int k = a;
            for (; k + 32 <= e; k += 32)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    part[b][q] += four(k + 8 * q) + four(k + 8 * q + 4);
                    // 32 reads in flight would take the registers of a wavefront or two
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
            for (int q = 0; q < 3; ++q)
                if (k + 8 <= e) {
                    part[b][q] += four(k) + four(k + 4);
                    k += 8;
                }
            if (k < e) {
                T t = T(0);
                if (k + 4 <= e) {
                    t = four(k);
                    k += 4;
                }
                const T t0 = k < e ? slice[k] : T(0), t1 = k + 1 < e ? slice[k + 1] : T(0),
                        t2 = k + 2 < e ? slice[k + 2] : T(0);
                part[b][3] += t + ((t0 + t1) + t2);
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) out[b] = (part[b][0] + part[b][1]) + (part[b][2] + part[b][3]);
}

// chunk_compute for NB vectors: the chunk's indices and values stay in
// registers while one vector after the other is gathered and summed; the sums
// are those of chunk_compute.
template <typename VT, typename T, int EPT, int NB, typename XG>
__device__ __forceinline__ void chunk_compute_multi(const WaveChunk<VT, EPT>& C, const int* __restrict__ JA,
                                                    const int* __restrict__ IA, const VT* __restrict__ vals, XG xg,
                                                    T* slice, T (&out)[NB])
{
    const int lane = threadIdx.x & 63;
    if (C.e - C.s > EPT * 64) {
        chunk_rows<VT, T, NB>(C.nr, C.rb, C.re, IA, vals, xg, out);
        return;
    }
    const int a = C.rb - C.s, e = C.re - C.s;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        T xv[EPT];
#pragma unroll
        for (int j = 0; j < EPT; ++j) {
            const int k = C.s + lane + 64 * j;
            xv[j] = (k < C.e) ? xg(b, C.col[j]) : T(0);
        }
#pragma unroll
        for (int j = 0; j < EPT; ++j) {
            const int k = C.s + lane + 64 * j;
            if (k < C.e) slice[k - C.s] = Load<VT, T>::get(C.v, j) * xv[j];
        }
        __builtin_amdgcn_wave_barrier();  // as in chunk_compute
        T acc = T(0);
        if (lane < C.nr && a < e) {
            acc = slice[a];
            for (int k = a + 1; k < e; ++k) acc += slice[k];
        }
        out[b] = acc;
        __builtin_amdgcn_wave_barrier();
    }
}

// Returns (A x)[r0 + lane] (0 for lanes beyond the chunk). 'slice' is this
// wavefront's LDS slice of EPT*64 elements. XG(col) yields x[col].
template <typename VT, typename T, int EPT, typename XG>
__device__ __forceinline__ T chunk_compute(const WaveChunk<VT, EPT>& C, const int* __restrict__ JA,
                                           const int* __restrict__ IA, const VT* __restrict__ vals, XG xg,
                                           T* slice)
{
    const int lane = threadIdx.x & 63;
    T acc = T(0);
    if (C.e - C.s <= EPT * 64) {
        T xv[EPT];
#pragma unroll
        for (int j = 0; j < EPT; ++j) {
            const int k = C.s + lane + 64 * j;
            xv[j] = (k < C.e) ? xg(C.col[j]) : T(0);
        }
#pragma unroll
        for (int j = 0; j < EPT; ++j) {
            const int k = C.s + lane + 64 * j;
            if (k < C.e) slice[k - C.s] = Load<VT, T>::get(C.v, j) * xv[j];
        }
        // LDS operations of one wavefront complete in issue order, so the
        // reads below see every lane's write; the wave barrier only keeps
        // the compiler from moving code across this point.
        __builtin_amdgcn_wave_barrier();
        const int a = C.rb - C.s, b = C.re - C.s;
        if (lane < C.nr && a < b) {
            acc = slice[a];
            for (int k = a + 1; k < b; ++k) acc += slice[k];
        }
        __builtin_amdgcn_wave_barrier();
    } else {
        // dense chunk: one row at a time, lanes stride the row
        for (int i = 0; i < C.nr; ++i) {
            const int a = JA[C.r0 + i], b = JA[C.r0 + i + 1];
            T s = T(0);
            for (int k = a + lane; k < b; k += 64) s += Load<VT, T>::get(vals, k) * xg(IA[k]);
            s = wave_reduce<OpSum>(s);
            if (lane == i) acc = s;
        }
    }
    return acc;
}

}  // namespace cm
