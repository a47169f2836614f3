// cwise_tile.hip -- generated component-wise kernels for programs that read
// a leaf across its memory order (a transposed view in a destination of the
// other layout: 0.5 * (A + A^T), a row-major operand in a column-major
// assignment).
//
// Evaluated in the destination's order, such a leaf costs a cache line per
// element. Here a block evaluates a tile of 64 x 64 elements: each transposed
// leaf's part of the tile is read with lanes along that leaf's contiguous
// axis into LDS (rows of 65 elements, so both directions are free of bank
// conflicts) and taken from there in the destination's order; every other
// leaf and the destination are accessed in runs of 64 elements as before. The
// program runs per element on the same operands in the same way as in
// jit_cwise_flat and the interpreter (cwise_ops.hpp), so the bits are the
// same.
//
// What bounds it: the bytes, each leaf once; a leaf that also appears
// untransposed is read a second time through the caches. Measured on MI355X,
// (A + A^T) * 0.5, us, gathering / tiled: FP32 1021 x 1021 x 61 420 -> 132
// (3.8 TB/s), 1024 x 1024 x 64 -> 82 (6.5), 4096^2 113 -> 31, 8000^2 504 ->
// 117, 64 x 64 x 4000 42 -> 22; FP64 2048 x 2048 x 4 205 -> 61. Whole
// batches per XCD against tiles dealt to all: 1021 x 1021 x 61 132 / 138.
// Tiles along a diagonal: 8000^2 123 -> 146, others the same.
#include "cwise_tile.hpp"

#include <cinttypes>
#include <cstring>

namespace cm {

namespace {

constexpr int TILE = 64;
constexpr int PER = TILE * TILE / 256;  // elements per thread
// Tiles of LDS a block may hold: four of 4-byte, two of 8-byte elements
// (66 KB: two blocks per CU still fit).
constexpr int TILE_LDS_WORDS = 4;

// A leaf read across the destination's order: contiguous along the
// destination's slow axis (s) and a stride of at least 16 elements along its
// fast axis (f). Below that stride a wavefront's gather still uses most of
// every line it touches.
bool transposed(long long sf, long long ss)
{
    return ss == 1 && (sf >= 16 || sf <= -16);
}

}  // namespace

// Which leaves the tiled kernel stages; 0: the program has none, or a shape
// or leaf it does not take.
unsigned cwise_tile_mask(const CwProgram& P, bool wide)
{
    if (!P.dst_direct) return 0;
    const long long F = P.row_order ? P.cols : P.rows, S = P.row_order ? P.rows : P.cols;
    // narrower matrices would leave half of every tile empty
    if (F < TILE / 2 || S < TILE / 2) return 0;
    unsigned mask = 0;
    int tiles = 0;
    for (int l = 0; l < P.nleaves; ++l) {
        const cm_leaf& L = P.leaves[l];
        if (L.kind != CM_LEAF_STRIDED) return 0;
        if (L.dtype != CM_F32 && L.dtype != CM_I32 && L.dtype != CM_BOOL && !(wide && L.dtype == CM_F64)) return 0;
        if (((P.leaf_scalar | P.leaf_direct) >> l) & 1) continue;
        if (!transposed(P.row_order ? L.sc : L.sr, P.row_order ? L.sr : L.sc)) continue;
        mask |= 1u << l;
        tiles += L.dtype == CM_F64 ? 2 : 1;
    }
    return tiles <= TILE_LDS_WORDS ? mask : 0;
}

// Source and key. Strides and shape are constants of the source.
// nt: streaming stores.
int jit_cwise_tile_source(const CwProgram& P, unsigned mask, bool wide, bool nt, std::string& key, std::string& body)
{
    const int dt = P.dst_dtype;
    if (dt != CM_F32 && dt != CM_I32 && dt != CM_BOOL && !(wide && dt == CM_F64)) return JIT_DECLINED;
    const long long F = P.row_order ? P.cols : P.rows, S = P.row_order ? P.rows : P.cols;
    char buf[512];
    snprintf(buf, sizeof(buf), "cwtile%c%c|d%d|m%d|%lld,%lld,%lld,%d|%x|", wide ? 'w' : 'n', nt ? 't' : 'p', dt, P.mode, P.rows, P.cols,
             P.batches, P.row_order, mask);
    key = buf;
    std::string lds, stage, fill, direct, loads, scalars, names[CM_CWISE_MAX_LEAVES];
    const char* namep[CM_CWISE_MAX_LEAVES];
    for (int l = 0; l < P.nleaves; ++l) {
        const cm_leaf& L = P.leaves[l];
        const long long sf = P.row_order ? L.sc : L.sr, ss = P.row_order ? L.sr : L.sc;
        const char* type = L.dtype == CM_BOOL ? "unsigned char" : (L.dtype == CM_F64 ? "uint64_t" : "uint32_t");
        snprintf(buf, sizeof(buf), "L%d,%lld,%lld,%lld|", L.dtype, (long long)L.sr, (long long)L.sc, (long long)L.sb);
        key += buf;
        const std::string n = std::to_string(l);
        if ((P.leaf_scalar >> l) & 1) {
            names[l] = "c" + n;
            scalars += std::string("    const R c") + n + " = (R)((const " + type + "*)A.leaf[" + n + "])[0];\n";
        } else if ((mask >> l) & 1) {
            const char* word = L.dtype == CM_F64 ? "uint64_t" : "uint32_t";
            names[l] = "(R)t" + n + "[lane * PITCH + w + 4 * k]";
            lds += std::string("    __shared__ ") + word + " t" + n + "[TILE * PITCH];\n";
            stage += std::string("    ") + word + " g" + n + "[PER];\n";
            snprintf(buf, sizeof(buf),
                     "    { const %s* p = (const %s*)A.leaf[%d] + b * %lldll + (ts0 + lane);\n#pragma unroll\n"
                     "      for (int k = 0; k < PER; ++k) g%d[k] = (ts0 + lane < S && f0 + w + 4 * k < F)"
                     " ? (%s)p[(f0 + w + 4 * k) * %lldll] : 0; }\n",
                     type, type, l, (long long)L.sb, l, word, sf);
            stage += buf;
            fill += "#pragma unroll\n    for (int k = 0; k < PER; ++k) t" + n + "[(w + 4 * k) * PITCH + lane] = g" + n +
                    "[k];\n";
        } else {
            names[l] = "v" + n + "[k]";
            direct += "    R v" + n + "[PER];\n";
            snprintf(buf, sizeof(buf),
                     "    { const %s* p = (const %s*)A.leaf[%d] + b * %lldll + (f0 + lane) * %lldll;\n#pragma unroll\n"
                     "      for (int k = 0; k < PER; ++k) v%d[k] = (f0 + lane < F && ts0 + w + 4 * k < S)"
                     " ? (R)p[(ts0 + w + 4 * k) * %lldll] : 0; }\n",
                     type, type, l, (long long)L.sb, sf, l, ss);
            loads += buf;
        }
        namep[l] = names[l].c_str();
    }
    for (int i = 0; i < P.ncode; ++i) {
        const cm_instr& I = P.code[i];
        uint64_t fb;
        memcpy(&fb, &I.fimm, 8);
        snprintf(buf, sizeof(buf), "%d,%d,%d,%d,%d,%d,%" PRIx64 ",%" PRIx64 ";", I.opcode, I.dtype, I.fn, I.src, I.arg,
                 I.flags, fb, (uint64_t)I.iimm);
        key += buf;
    }
    std::string prog;
    if (!jit::program_body(P, namep, prog)) return JIT_DECLINED;
    // the interpreter's store_elem
    const char* store;
    if (nt) store = dt == CM_F64 ? "__builtin_nontemporal_store(getd(acc), p);"
                                 : (dt == CM_F32 ? "__builtin_nontemporal_store(getf(acc), p);"
                                                 : "__builtin_nontemporal_store(geti(acc), p);");
    else if (dt == CM_F64) store = "const double v = getd(acc); *p = (MODE == CM_ASSIGN) ? v : assign1<double>(MODE, *p, v);";
    else if (dt == CM_F32) store = "const float v = getf(acc); *p = (MODE == CM_ASSIGN) ? v : assign1<float>(MODE, *p, v);";
    else if (dt == CM_I32) store = "const int v = geti(acc); *p = (MODE == CM_ASSIGN) ? v : assign1<int>(MODE, *p, v);";
    else
        store = "int v = geti(acc) != 0; if (MODE == CM_AND) v = v && *p; else if (MODE == CM_OR) v = v || *p; "
                "*p = (unsigned char)v;";
    const char* dtype = dt == CM_F64 ? "double" : (dt == CM_F32 ? "float" : (dt == CM_I32 ? "int" : "unsigned char"));
    const long long nf = (F + TILE - 1) / TILE, ns = (S + TILE - 1) / TILE;
    snprintf(buf, sizeof(buf),
             "typedef %s R;\nconstexpr int TILE = %d, PITCH = %d, PER = %d, MODE = %d;\n"
             "constexpr long long F = %lldll, S = %lldll, NF = %lldll, NT = %lldll, NB = %lldll;\n",
             wide ? "uint64_t" : "uint32_t", TILE, TILE + 1, PER, P.mode, F, S, nf, nf * ns, (long long)P.batches);
    body = std::string("struct JitTileArgs { const void* leaf[") + std::to_string(CM_CWISE_MAX_LEAVES) +
           "]; void* dst; int by_xcd, pad; };\n" + buf +
           "extern \"C\" __global__ __launch_bounds__(256) void cm_jit_cwise_tile(const JitTileArgs A)\n{\n" + lds +
           "    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);\n"
           // by_xcd: block h runs on XCD h % 8, which takes whole batches, so
           // that a matrix and its transposed reads meet in one L2
           "    const long long h = blockIdx.x;\n"
           "    const long long m = A.by_xcd ? (h & 7) + 8 * ((h >> 3) / NT) : h / NT;\n"
           "    const long long tile = A.by_xcd ? (h >> 3) % NT : h % NT;\n"
           "    if (m >= NB) return;\n"
           "    const long long b = m, ft = tile % NF, f0 = ft * TILE, ts0 = tile / NF * TILE;\n" + scalars + direct + loads + stage +
           fill + "    __syncthreads();\n"
           "    " + dtype + "* const q = (" + dtype + "*)A.dst + b * (F * S) + (f0 + lane);\n"
           "    if (f0 + lane >= F) return;\n"
           "#pragma unroll\n"
           "    for (int k = 0; k < PER; ++k) {\n"
           "        if (ts0 + w + 4 * k >= S) break;\n"
           "        R acc = 0, t = 0, s0 = 0, s1 = 0, s2 = 0, s3 = 0;\n"
           "        (void)t; (void)s0; (void)s1; (void)s2; (void)s3;\n"
           + prog +
           "        " + dtype + "* const p = q + (ts0 + w + 4 * k) * F;\n"
           "        { " + store + " }\n"
           "    }\n"
           "}\n";
    return CM_OK;
}

struct JitTileArgs {
    const void* leaf[CM_CWISE_MAX_LEAVES];
    void* dst;
    int by_xcd, pad;
};

int jit_cwise_tile(cm_ctx_t ctx, const CwProgram& P, bool wide)
{
    const unsigned mask = cwise_tile_mask(P, wide);
    if (!mask) return JIT_DECLINED;
    // streaming stores where every run of 64 elements is whole lines (4096^2
    // FP32 35 -> 31 us, 64^2 x 4000 28 -> 22; with columns of 1021 elements, 132
    // -> 141, two blocks write a part of the same line)
    const long long run = (P.row_order ? P.cols : P.rows) * (long long)dtype_size(P.dst_dtype);
    const bool nt = P.mode == CM_ASSIGN && P.dst_dtype != CM_BOOL && run % 128 == 0 && ((uintptr_t)P.dst & 127) == 0;
    std::string sig("cwtile");
    jit::sig_add(sig, (int)wide);
    jit::sig_add(sig, (int)nt);
    jit::sig_add(sig, mask);
    jit::sig_add(sig, P.dst_dtype);
    jit::sig_add(sig, P.mode);
    jit::sig_add(sig, P.row_order);
    jit::sig_add(sig, P.rows);
    jit::sig_add(sig, P.cols);
    jit::sig_add(sig, P.batches);
    jit::sig_add(sig, P.leaf_scalar);
    jit::sig_add(sig, P.nleaves);
    for (int l = 0; l < P.nleaves; ++l) {
        const cm_leaf& L = P.leaves[l];
        jit::sig_add(sig, L.dtype);
        jit::sig_add(sig, L.sr);
        jit::sig_add(sig, L.sc);
        jit::sig_add(sig, L.sb);
    }
    jit::sig_add(sig, P.ncode);
    for (int i = 0; i < P.ncode; ++i) {
        const cm_instr& I = P.code[i];
        jit::sig_add(sig, I.opcode);
        jit::sig_add(sig, I.dtype);
        jit::sig_add(sig, I.fn);
        jit::sig_add(sig, I.src);
        jit::sig_add(sig, I.arg);
        jit::sig_add(sig, I.flags);
        jit::sig_add(sig, I.fimm);
        jit::sig_add(sig, I.iimm);
    }
    jit::Kernel k;
    if (jit::find_sig(sig, &k) != 0) {
        std::string key, body;
        if (jit_cwise_tile_source(P, mask, wide, nt, key, body) != CM_OK) return JIT_DECLINED;
        if (jit::get(key, body, "cm_jit_cwise_tile", &k) != 0) return JIT_DECLINED;
        jit::put_sig(sig, k);
    }
    JitTileArgs A;
    memset(&A, 0, sizeof(A));
    for (int l = 0; l < P.nleaves; ++l) A.leaf[l] = P.leaves[l].ptr;
    A.dst = P.dst;
    // whole batches per XCD where there are enough of them to balance
    A.by_xcd = P.batches >= 16;
    const long long F = P.row_order ? P.cols : P.rows, S = P.row_order ? P.rows : P.cols;
    const long long tiles = ((F + TILE - 1) / TILE) * ((S + TILE - 1) / TILE);
    const long long blocks = tiles * (A.by_xcd ? (P.batches + 7) / 8 * 8 : P.batches);
    if (blocks >= (1ll << 31)) return JIT_DECLINED;
    if (jit::launch(k, (unsigned)blocks, 256, ctx->stream, &A, sizeof(A)) != 0)
        return fail(CM_E_HIP, "cm_cwise_eval: launch of the generated kernel failed");
    count(CM_CNT_KERNEL_LAUNCH);
    return CM_OK;
}

}  // namespace cm
