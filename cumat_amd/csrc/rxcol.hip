// rxcol.hip -- generated reductions of expressions along strided axes.
//
// The reductions of redexpr.hip put a wavefront's lanes along the reduced
// axes. Where those are strided in memory and a kept axis is contiguous (the
// column sum of a column-major matrix, a batch sum), every lane then touches
// a cache line of its own: 15 us of traffic took 365 us. Here a lane owns one
// kept element and walks the reduced axes, so a wavefront's loads are
// consecutive elements, and the coordinates of the walk are the same for all
// lanes (scalar registers).
//
// The result keeps the bits of reduce_expr_kernel: a lane folds the elements
// exactly as the 256 threads and the block reduction of that kernel would.
// Thread t's elements are known (spread or consecutive mapping, pass after
// pass), and the reduction's tree over the threads is fixed (fold_ops.hpp):
//   16 threads   the butterfly as thread 0 of the row sees it, i.e. a plain
//                binary tree over the threads in the order ROW_ORDER
//   4 rows       (a op b) op (c op d)
//   wavefronts   one after the other.
// So the threads of a row are visited in ROW_ORDER and merged with a stack of
// four partial results. Rows without elements are the identity. The 16 rows
// of 16 threads are split over the wavefronts of a block (UNITS of them) and
// combined in LDS.
//
// What bounds it: the bytes for long folds over many kept elements, the
// latency of a lane's loads (up to 32 in flight) where few are kept. Measured
// on MI355X, us, lanes along the fold / along the kept axes: squared deviation
// from the mean, FP32 3000 x 5000 x 3 over columns 365 -> 49 (3.7 TB/s), over
// batches 8790 -> 61; 1024 x 1024 x 64 over columns 457 -> 48 (5.6 TB/s), over
// batches 856 -> 65, over both 347 -> 198; FP64 1000 x 1000 x 32 over columns
// 277 -> 49. 200000 contiguous segments of 50: 160 -> 44. One pass of loads in
// flight instead of four: over both 225; four threads' loads: 209, and short
// folds slower.
#include "rxcol.hpp"

#include <cstring>

namespace cm {

namespace {

// elements a leaf steps per unit of (row, column, batch)
void strides_of(const cm_leaf& L, long long (&s)[3])
{
    s[0] = L.sr;
    s[1] = L.sc;
    s[2] = L.sb;
}

// Whether lanes along the kept axes read the expression's full leaves (those
// that vary along kept and reduced axes) in longer runs than lanes along the
// reduced axes would: more of them are contiguous there, over at least MIN_RUN
// elements (half a 128-byte line).
bool rx_column_wins(const CwProgram& P, const RxShape& SH)
{
    constexpr long long MIN_RUN = 16;
    auto run = [&](const long long (&s)[3], const long long* dim, const int* axis, int n) {
        long long r = 1;
        for (int a = 0; a < n; ++a) {
            if (dim[a] <= 1) continue;
            if (s[axis[a]] != r) break;
            r *= dim[a];
        }
        return r;
    };
    int kept = 0, reduced = 0;
    for (int l = 0; l < P.nleaves; ++l) {
        long long s[3];
        strides_of(P.leaves[l], s);
        bool vk = false, vr = false;
        for (int a = 0; a < SH.nk; ++a) vk = vk || (SH.kdim[a] > 1 && s[SH.kaxis[a]] != 0);
        for (int a = 0; a < SH.nr; ++a) vr = vr || (SH.rdim[a] > 1 && s[SH.raxis[a]] != 0);
        if (!vk || !vr) continue;
        if (run(s, SH.kdim, SH.kaxis, SH.nk) >= MIN_RUN) ++kept;
        if (run(s, SH.rdim, SH.raxis, SH.nr) >= MIN_RUN) ++reduced;
    }
    return kept > reduced;
}

// Contiguous segments: up to this length, and from this many of them on, a
// lane for each beats a block for each (below, the blocks are few enough).
constexpr long long SHORT_FOLD = 128, MANY_SEGMENTS = 32768;
// Fewer wavefronts than this leave most of the chip idle: 100 kept elements, 4
// chunks of 1600 took 23 us against 17 with lanes along the fold.
constexpr long long MIN_WAVES = 256;

// Wavefronts that share a segment's rows: all 16 rows where each then still
// has a full pass of elements, fewer for short folds (whose other rows are
// empty).
int units_for(long long len)
{
    return len >= 512 ? 16 : (len >= 128 ? 4 : 1);
}

}  // namespace

// Source and key of the kernel. Shape, strides and types are constants of the
// source, addresses, chunks and the segment count are arguments. flat (short
// segments of a flat program): the extents are arguments as well, so that one
// kernel serves a program of every size; element j of segment s is s * L + j.
int jit_reduce_column_source(const CwProgram& P, const RxShape& SH, const RxNames& N, bool wide, bool spread, bool flat,
                             int units, std::string& key, std::string& body)
{
    char buf[512];
    const int V = wide ? 4 : 8;
    const bool one = SH.L <= (spread ? 4 : V);
    key = std::string(flat ? "rxcolf" : "rxcol") + (one ? "1" : "n") + (wide ? "64" : "32") + (spread ? "s" : "c") + std::to_string(units) + "|" + N.op + "|" +
          N.acc + "|" + N.store + "|k";
    // kept coordinates of the lane's segment (once), reduced coordinates of
    // element j (uniform: scalar registers)
    std::string kept, red;
    for (int a = 0; a < SH.nk && !flat; ++a) {
        snprintf(buf, sizeof(buf), "%lld@%d,", SH.kdim[a], SH.kaxis[a]);
        key += buf;
        snprintf(buf, sizeof(buf), "    { const long long q = w_ / %lldll; k3[%d] = w_ - q * %lldll; w_ = q; }\n", SH.kdim[a],
                 SH.kaxis[a], SH.kdim[a]);
        kept += buf;
    }
    key += "r";
    const bool narrow = SH.L < 4294967295ll;
    for (int a = 0; a < SH.nr && !flat; ++a) {
        snprintf(buf, sizeof(buf), "%lld@%d,", SH.rdim[a], SH.raxis[a]);
        key += buf;
        if (a + 1 == SH.nr)
            snprintf(buf, sizeof(buf), "                    r3[%d] = (long long)j_;\n", SH.raxis[a]);
        else
            snprintf(buf, sizeof(buf), "                    { const auto q = j_ / %lld%s; r3[%d] = (long long)(j_ - q * %lld%s); j_ = q; }\n",
                     SH.rdim[a], narrow ? "u" : "ull", SH.raxis[a], SH.rdim[a], narrow ? "u" : "ull");
        red += buf;
    }
    key += "|";
    const long long dim[3] = {P.rows, P.cols, P.batches};
    bool is_red[3] = {false, false, false};
    for (int a = 0; a < SH.nr; ++a) is_red[SH.raxis[a]] = true;
    int varying = 0;
    std::string decls, bases, loads, scalars, names[CM_CWISE_MAX_LEAVES];
    const char* namep[CM_CWISE_MAX_LEAVES];
    for (int l = 0; l < P.nleaves; ++l) {
        const cm_leaf& L = P.leaves[l];
        if (L.dtype != CM_F32 && L.dtype != CM_I32 && L.dtype != CM_BOOL && !(wide && L.dtype == CM_F64))
            return RX_JIT_DECLINED;
        if (L.kind != CM_LEAF_STRIDED) return RX_JIT_DECLINED;
        long long s[3];
        strides_of(L, s);
        if (flat) snprintf(buf, sizeof(buf), "L%d%c|", L.dtype, (P.leaf_scalar >> l) & 1 ? 's' : 'd');
        else snprintf(buf, sizeof(buf), "L%d,%lld,%lld,%lld|", L.dtype, s[0], s[1], s[2]);
        key += buf;
        const char* type = L.dtype == CM_BOOL ? "unsigned char" : (L.dtype == CM_F64 ? "uint64_t" : "uint32_t");
        std::string koff, roff;
        if (flat && !((P.leaf_scalar >> l) & 1)) {
            koff = "w_ * A.L";
            roff = "e_";
        }
        for (int a = 0; a < 3 && !flat; ++a) {
            if (s[a] == 0 || dim[a] <= 1) continue;
            std::string& o = is_red[a] ? roff : koff;
            snprintf(buf, sizeof(buf), "%s%s3[%d] * %lldll", o.empty() ? "" : " + ", is_red[a] ? "r" : "k", a, s[a]);
            o += buf;
        }
        const std::string n = std::to_string(l);
        snprintf(buf, sizeof(buf), "    const %s* const b%d = (const %s*)A.leaf[%d] + (%s);\n", type, l, type, l,
                 koff.empty() ? "0" : koff.c_str());
        bases += buf;
        if (roff.empty()) {  // does not vary along the fold
            names[l] = "c" + n;
            scalars += "    const R c" + n + " = (R)b" + n + "[0];\n";
        } else {
            names[l] = "v" + n + "[k]";
            decls += "                R v" + n + "[PP * V];\n";
            ++varying;
            loads += "                    v" + n + "[k] = (R)b" + n + "[" + roff + "];\n";
        }
        namep[l] = names[l].c_str();
    }
    for (int i = 0; i < P.ncode; ++i) {
        const cm_instr& I = P.code[i];
        uint64_t fb;
        memcpy(&fb, &I.fimm, 8);
        snprintf(buf, sizeof(buf), "%d,%d,%d,%d,%d,%d,%llx,%llx;", I.opcode, I.dtype, I.fn, I.src, I.arg, I.flags,
                 (unsigned long long)fb, (unsigned long long)I.iimm);
        key += buf;
    }
    std::string prog;
    if (!jit::program_body(P, namep, prog)) return RX_JIT_DECLINED;
    // passes whose loads are in flight together: four of one varying leaf, two
    // of two or three, where a thread has that many
    int pp = varying <= 1 ? 4 : (varying <= 3 ? 2 : 1);
    if (SH.L < 2ll * pp * 256 * V) pp = 1;
    const std::string load_text = std::string("const ") + (narrow ? "unsigned" : "unsigned long long") + " e_ = (" +
                                  (narrow ? "unsigned" : "unsigned long long") +
                                  ")EL(p0 + k / V * 256 * V, k % V); auto j_ = e_; (void)j_; long long r3[3] = {0, 0, 0}; " + red + loads;
    const std::string fold_text = "R acc = 0, t = 0, s0 = 0, s1 = 0, s2 = 0, s3 = 0; "
                                  "(void)t; (void)s0; (void)s1; (void)s2; (void)s3;\n" + prog +
                                  "v = OP::apply(v, (TT)" + N.get + "(acc)); ";
    auto define = [](const char* name, const std::string& text) {
        std::string one = std::string("#define ") + name + " ";
        for (char ch : text)
            if (ch == '\n') one += ' ';
            else one += ch;
        return one + "\n";
    };
    const int waves = units >= 4 ? units : 4, tiles = waves / units;
    snprintf(buf, sizeof(buf),
             "typedef %s TT;\ntypedef %s SS;\ntypedef %s OP;\ntypedef %s R;\n"
             "constexpr int V = %d, PP = %d, UNITS = %d, TILES = %d;\nconstexpr bool ONE = %s;\n",
             N.acc, N.store, N.op, wide ? "uint64_t" : "uint32_t", V, pp, units, tiles, one ? "true" : "false");
    body = std::string("struct JitRxArgs { const void* leaf[") + std::to_string(CM_CWISE_MAX_LEAVES) +
           "]; void* partials; void* out; long long L, chunk, nseg; int nchunk, pad; };\n" + buf +
           (spread ? "#define FIRST(t) ((long long)((t) >> 6) * 512 + ((t) & 63) * 4)\n"
                     "#define EL(j0, k) ((j0) + ((k) >> 2) * 256 + ((k) & 3))\n"
                   : "#define FIRST(t) ((long long)(t) * V)\n#define EL(j0, k) ((j0) + (k))\n") +
           define("LOADS", load_text) + define("FOLD", fold_text) +
           "extern \"C\" __global__ __launch_bounds__(" + std::to_string(64 * waves) +
           ") void cm_jit_reduce(const JitRxArgs A)\n{\n"
           "    __shared__ TT rows[UNITS > 1 ? UNITS * 64 : 1];\n"
           "    const int lane = threadIdx.x & 63;\n"
           "    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);\n"
           "    const int unit = wave % UNITS;\n"
           "    const int c = blockIdx.x % A.nchunk;\n"
           "    const long long s = ((long long)(blockIdx.x / A.nchunk) * TILES + wave / UNITS) * 64 + lane;\n"
           "    const bool ok = s < A.nseg;\n"
           "    long long w_ = ok ? s : A.nseg - 1;\n"
           "    long long k3[3] = {0, 0, 0};\n" + kept + bases + scalars +
           "    const long long beg = c * A.chunk;\n"
           "    const long long end = min(A.L, beg + A.chunk);\n"
           "    const TT identity = " + N.identity + ";\n"
           "    TT r4[4] = {identity, identity, identity, identity}, whole = identity;\n"
           "    for (int row = unit * (16 / UNITS); row < (unit + 1) * (16 / UNITS); ++row) {\n"
           "        TT v = identity, a0 = identity, a1 = identity, a2 = identity, a3 = identity;\n"
           "        if (beg + FIRST(row * 16) < end)\n"
           "        for (int i = 0; i < (ONE ? 1 : 16); ++i) {\n"
           // ROW_ORDER, one hexadecimal digit per visit
           "            const int t = row * 16 + (int)((0xba98cdef45673210ull >> (4 * i)) & 15);\n"
           "            v = identity;\n"
           "            for (long long p0 = beg + FIRST(t); p0 < end; p0 += 256 * V) {\n" + decls
           + (pp > 1 ? "                for (; EL(p0 + (PP - 1) * 256 * V, V - 1) < end; p0 += PP * 256 * V) {\n"
                       "#pragma unroll\n"
                       "                    for (int k = 0; k < PP * V; ++k) { LOADS }\n"
                       "#pragma unroll\n"
                       "                    for (int k = 0; k < PP * V; ++k) { FOLD }\n"
                       "                }\n"
                       "                if (p0 >= end) break;\n"
                     : "") +
           // whole passes need no test per element
           "                if (EL(p0, V - 1) < end) {\n"
           "#pragma unroll\n"
           "                    for (int k = 0; k < V; ++k) { LOADS }\n"
           "#pragma unroll\n"
           "                    for (int k = 0; k < V; ++k) { FOLD }\n"
           "                } else {\n"
           "#pragma unroll\n"
           "                    for (int k = 0; k < V; ++k) if (EL(p0, k) < end) { LOADS }\n"
           "#pragma unroll\n"
           "                    for (int k = 0; k < V; ++k) if (EL(p0, k) < end) { FOLD }\n"
           "                }\n"
           "            }\n"
           // one thread has all elements: every other merge adds an identity, and
           // the first of them settles the result
           "            if (ONE) v = OP::apply(v, identity);\n"
           "            else if (!(i & 1)) a0 = v;\n"
           "            else {\n"
           "                v = OP::apply(a0, v);\n"
           "                if (!(i & 2)) a1 = v;\n"
           "                else {\n"
           "                    v = OP::apply(a1, v);\n"
           "                    if (!(i & 4)) a2 = v;\n"
           "                    else {\n"
           "                        v = OP::apply(a2, v);\n"
           "                        if (!(i & 8)) a3 = v;\n"
           "                        else v = OP::apply(a3, v);\n"
           "                    }\n"
           "                }\n"
           "            }\n"
           "        }\n"
           "        if (ONE) { whole = v; break; }\n"
           "        if (UNITS == 16) { whole = v; continue; }\n"
           "        const int x = row & 3;\n"
           "        if (x == 0) r4[0] = v; else if (x == 1) r4[1] = v; else if (x == 2) r4[2] = v;\n"
           "        else {\n"
           "            v = OP::apply(OP::apply(r4[0], r4[1]), OP::apply(r4[2], v));\n"
           "            whole = row == 3 || UNITS == 4 ? v : OP::apply(whole, v);\n"
           "        }\n"
           "    }\n"
           "    if (UNITS > 1) {\n"
           "        rows[unit * 64 + lane] = whole;\n"
           "        __syncthreads();\n"
           "        if (unit != 0) return;\n"
           "#pragma unroll\n"
           "        for (int w = 0; w < 4; ++w) {\n"
           "            TT x;\n"
           "            if (UNITS == 16)\n"
           "                x = OP::apply(OP::apply(rows[w * 256 % (UNITS * 64) + lane], rows[(w * 256 + 64) % (UNITS * 64) + lane]),\n"
           "                              OP::apply(rows[(w * 256 + 128) % (UNITS * 64) + lane], rows[(w * 256 + 192) % (UNITS * 64) + lane]));\n"
           "            else x = rows[w * 64 + lane];\n"
           "            whole = w ? OP::apply(whole, x) : x;\n"
           "        }\n"
           "    }\n"
           "    if (!ok) return;\n"
           "    if (A.nchunk == 1) ((SS*)A.out)[s] = (SS)whole;\n"
           "    else ((TT*)A.partials)[s * A.nchunk + c] = whole;\n"
           "}\n";
    return CM_OK;
}

namespace {

// JitRxArgs with the segment count
struct JitRxColArgs {
    const void* leaf[CM_CWISE_MAX_LEAVES];
    void* partials;
    void* out;
    long long L, chunk, nseg;
    int nchunk, pad;
};

}  // namespace

int rx_column_launch(cm_ctx_t ctx, const CwProgram& P, const RxShape& SH, const RxNames& N, bool wide, bool spread,
                     bool flat, long long nchunk, long long chunk, void* partials, void* out)
{
    // also many short segments, whatever their layout: a block per segment
    // costs 0.8 ns a segment with hardly a thread at work
    const bool many_short = SH.L <= SHORT_FOLD && SH.nseg >= MANY_SEGMENTS;
    // before the signature is looked up: a vector as a diagonal has the strides
    // of the same vector broadcast over the columns
    for (int l = 0; l < P.nleaves; ++l)
        if (P.leaves[l].kind != CM_LEAF_STRIDED) return RX_JIT_DECLINED;
    if (!many_short && !rx_column_wins(P, SH)) return RX_JIT_DECLINED;
    const int units = units_for(chunk < SH.L ? chunk : SH.L);
    if ((SH.nseg + 63) / 64 * nchunk * units < MIN_WAVES) return RX_JIT_DECLINED;
    // short segments of a flat program need no shape in the source
    flat = flat && many_short;
    // everything the generator reads
    std::string sig(flat ? "rxcolf" : "rxcol");
    sig += N.op;
    sig += N.acc;
    sig += N.store;
    jit::sig_add(sig, (int)wide);
    jit::sig_add(sig, (int)spread);
    jit::sig_add(sig, units);
    jit::sig_add(sig, (int)(SH.L <= (spread ? 4 : (wide ? 4 : 8))));
    jit::sig_add(sig, flat ? P.leaf_scalar : 0u);
    jit::sig_add(sig, SH.nk);
    jit::sig_add(sig, SH.nr);
    for (int a = 0; a < 3 && !flat; ++a) {
        jit::sig_add(sig, a < SH.nk ? SH.kdim[a] : 0ll);
        jit::sig_add(sig, a < SH.nk ? SH.kaxis[a] : -1);
        jit::sig_add(sig, a < SH.nr ? SH.rdim[a] : 0ll);
        jit::sig_add(sig, a < SH.nr ? SH.raxis[a] : -1);
    }
    jit::sig_add(sig, P.nleaves);
    for (int l = 0; l < P.nleaves; ++l) {
        const cm_leaf& L = P.leaves[l];
        jit::sig_add(sig, L.dtype);
        jit::sig_add(sig, L.kind);
        if (flat) continue;
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
        if (jit_reduce_column_source(P, SH, N, wide, spread, flat, units, key, body) != CM_OK) return RX_JIT_DECLINED;
        if (jit::get(key, body, "cm_jit_reduce", &k) != 0) return RX_JIT_DECLINED;
        jit::put_sig(sig, k);
    }
    const int waves = units >= 4 ? units : 4, tiles = waves / units;
    const long long blocks = (SH.nseg + 64ll * tiles - 1) / (64ll * tiles) * nchunk;
    if (blocks >= (1ll << 31)) return RX_JIT_DECLINED;
    JitRxColArgs A;
    memset(&A, 0, sizeof(A));
    for (int l = 0; l < P.nleaves; ++l) A.leaf[l] = P.leaves[l].ptr;
    A.partials = partials;
    A.out = out;
    A.L = SH.L;
    A.chunk = chunk;
    A.nseg = SH.nseg;
    A.nchunk = (int)nchunk;
    if (jit::launch(k, (unsigned)blocks, 64 * waves, ctx->stream, &A, sizeof(A)) != 0)
        return fail(CM_E_HIP, "cm_reduce_expr: launch of the generated kernel failed");
    count(CM_CNT_KERNEL_LAUNCH);
    return CM_OK;
}

}  // namespace cm
