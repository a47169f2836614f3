// rxcol.hpp -- the virtual order of a reduction of an expression, and the
// reductions along strided axes (rxcol.hip).
#pragma once
#include "cwise_core.hpp"
#include "jit.hpp"

namespace cm {

constexpr int RX_BS = 256;
constexpr int RX_JIT_DECLINED = 1;

// Virtual order: up to three kept axes (kdim / kaxis, innermost first, in
// the output layout's order) and up to three reduced axes (rdim / raxis).
// Axis ids: 0 row, 1 column, 2 batch.
struct RxShape {
    long long kdim[3], rdim[3];
    int kaxis[3], raxis[3];
    int nk, nr;
    long long L, nseg;
};

// Arguments of the generated reduction kernel cm_jit_reduce.
struct JitRxArgs {
    const void* leaf[CM_CWISE_MAX_LEAVES];
    void* partials;
    void* out;
    long long L, chunk;
    int nchunk, pad;
};

// How one reduction is spelled in generated source.
struct RxNames {
    const char* op;     // cm::OpSum ...
    const char* acc;    // accumulation type
    const char* store;  // stored type
    const char* get;    // register -> accumulation type
    std::string identity;
};

// Launches the generated reduction with lanes along the kept axes where the
// expression's memory lies that way (rx_column_wins); RX_JIT_DECLINED
// elsewhere. Same chunks, partials and bits as reduce_expr_kernel. flat: every
// leaf lies in the virtual order or is a broadcast scalar (P.leaf_scalar).
int rx_column_launch(cm_ctx_t ctx, const CwProgram& P, const RxShape& SH, const RxNames& N, bool wide, bool spread,
                     bool flat, long long nchunk, long long chunk, void* partials, void* out);

}  // namespace cm
