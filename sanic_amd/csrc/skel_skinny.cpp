// Contractions over few rows: the Plain(Add) carriers of skel_gemm.cpp (RMSNorm-fused projection,
// dot, int4 group-quantized matmul) when one workgroup's rows do not fill a GEMM tile — a decode
// batch, a short prompt — so the weight stream is the work and the MFMAs are nearly free.
//
// Structure required: gemm_plan's, with row leaves that are stored bf16 runs, a contraction factor
// hi + lo bf16 hold exactly (one bf16 value or the product of two) and a weight that is stored
// bf16 with k or n contiguous, or packed 4-bit q·s ± z with s and z constant over 32 k or more.
//
// Kernel shape: a workgroup owns 16·MT rows × BN columns and its waves split K into stages (256
// bytes of each weight row, 128 for 4-bit; SK rows of a [K, N] weight). A wave requests the row
// runs and then the weights of its stages as whole 128-byte lines, builds its A fragments while
// the weights are in flight, and turns each stage into B fragments through an LDS slot of its own;
// no barrier until the waves' partial tiles meet in LDS, summed in wave order. Above 32 rows also
// as 64 × 32 "tall" tiles, where the rows' own reads would pass the weights': x then takes the
// weights' way through LDS, and the next stage is requested once this one is there. A 4-bit weight goes
// to the MFMA as the integer q (exact in bf16) and each group folds as s·Σ x·q ± z·Σ x, Σ x from
// the matrix cores as well. (The weights pass through registers: with direct-to-LDS transfers in
// flight the compiler waits for all of them before the first row run is used.)
//
// The bound is the weight stream, above 32 rows the arithmetic between its stages. Generic fold → here, K = 2048,
// N = 8192, launches on one weight (33.6 MB, which the Infinity Cache holds; 4-bit 9.5 MB): M = 8 [N, K]
// weights 25 → 7.6 µs, [K, N] weights 11.5 µs (14.8 before the two halves of each line met on one XCD);
// 4-bit, M = 16: 246 → 5.8 µs. On three weights in turn 8.8 µs (3.8 TB/s) and 8.1. K = 8192, N = 2048,
// M = 8: 14.2 µs. Tall tiles, 32-row ones or GEMM tiles → here: 4-bit, M = 33, N = 8192 14.9 → 10.5 µs;
// K = 1968, N = 1088, M = 300 23.8 → 18.8: 170 workgroups, whose CUs issue vector instructions about
// half of the time (every column block forms the hi + lo pairs of its x·g) and take 14 bytes a
// clock that miss L1 (the GEMM's tiles 28).
#include <algorithm>
#include <functional>
#include <numeric>
#include <regex>

#include "emit.h"
#include "skeletons.h"

namespace sanic {

namespace {

// `run` consecutive elements along `var` from a multiple of `run` are consecutive in memory.
bool contiguous_runs(const Access& acc, int var, int64_t run) {
    int64_t stride = 0;
    for (auto& t : acc.addr.terms) {
        if (t.var != var) continue;
        if (t.div == 1 && (t.mod == 0 || t.mod % run == 0)) stride += t.coef;
        else if (t.div % run != 0) return false;
    }
    return stride == 1;
}

// The packed 4-bit input of an elementwise weight tree, with its coordinates.
bool packed_access(const sanic_program_desc* d, int node, const std::vector<Sym>& c, const std::vector<int64_t>& ext, Access& out) {
    const sanic_node& n = d->nodes[node];
    if (n.kind == SANIC_NODE_INPUT) return (n.dtype == SANIC_U4 || n.dtype == SANIC_I4) && sym_access(d, node, c, ext, out);
    if (n.kind == SANIC_NODE_REINDEX || n.kind == SANIC_NODE_VIEW) {
        std::vector<Sym> sc;
        return sym_child_coords(d, node, c, ext, sc) && packed_access(d, n.in[0], sc, ext, out);
    }
    if (n.kind != SANIC_NODE_MAP) return false;
    for (int k = 0; k < n.n_in; k++) {
        const sanic_node& m = d->nodes[n.in[k]];
        std::vector<Sym> cc(m.rank);
        for (int j = 0; j < m.rank; j++) cc[j] = m.shape[j] == 1 ? Sym() : c[n.rank - m.rank + j];
        if (packed_access(d, n.in[k], cc, ext, out)) return true;
    }
    return false;
}

std::string str(int64_t v) { return std::to_string(v); }

}  // namespace

// A K of many stages under few output points: here and in the GEMM a workgroup walks its columns'
// whole K, the split fold gives every point up to 64 workgroups. Estimates in µs, of a round of
// workgroups here (stages of 1024 k over 8 waves, 512 of a [K, N] weight) and of the fold. Here and
// there: [N, K], M = 2, N = 16, K = 65536 33 and 28, 131072 82 and 29; M = 2, N = 64, K = 131072 87 and 111;
// M = 8, N = 16, K = 131072 115 and 110, 196608 177 and 115; M = 16, N = 16, K = 131072 154 and 222, 196608
// 234 and 223; [K, N], M = 2, N = 32, K = 65536 66 and 56, 131072 149 and 80; M = 2, N = 64, K = 65536 134 and
// 172, 131072 274 and 205; M = 8, N = 32, K = 196608 278 and 470.
bool split_fold_faster(const sanic_program_desc* d, int si) {
    GemmPlan P;
    if (!gemm_plan(d, si, P) || !P.rslots.empty() || P.M > 16 || P.K < 32768) return false;
    const sanic_stage& st = d->stages[si];
    const sanic_node& wn = d->nodes[st.leaf[P.w]];
    std::vector<Sym> cw(wn.rank);
    for (int j = 0; j < wn.rank; j++) cw[j] = st.bind[P.w][j] == SANIC_BIND_STREAM ? Sym::var(1) : st.bind[P.w][j] == P.ndim ? Sym::var(0) : Sym();
    Access w;
    if (!sched_is_auto(st.sched) || !sym_access(d, st.leaf[P.w], cw, {P.N, P.K}, w)) return false;
    const double points = (double)(P.M * P.N), m = (double)P.M, k = (double)P.K;
    if (contiguous_runs(w, 1, 8)) return 2.0 + 0.82 * points < k / 1024.0 * (0.5 + 0.042 * m);
    return 2.0 + 0.82 * points + 6.5e-6 * k * points < k / 512.0 * ((P.N > 32 ? 1.02 : 0.54) + 0.018 * m);
}

bool lower_skinny(const sanic_program_desc* d, int si, LoweredStage& out, bool gemm_too) {
    GemmPlan P;
    if (!gemm_plan(d, si, P)) return false;
    const sanic_stage& st = d->stages[si];
    const sanic_carrier& c = st.carrier;
    const int64_t M = P.M, N = P.N, K = P.K;
    int factors = 0;
    if (!sched_is_auto(st.sched) || !exact_in_two(d, st, c.into[P.cslots[0]], P.w, factors)) return false;
    if (N < 16) return false;

    // ── the weight ──
    const sanic_node& wn = d->nodes[st.leaf[P.w]];
    std::vector<Sym> cw(wn.rank);
    for (int j = 0; j < wn.rank; j++) {
        int b = st.bind[P.w][j];
        cw[j] = b == SANIC_BIND_STREAM ? Sym::var(1) : b == P.ndim ? Sym::var(0) : Sym();
    }
    Access wacc;
    bool packed = false, kn = false, negB = false, hasB = false;
    int64_t unit = 0;                                // k over which a 4-bit group's s and z hold
    if (sym_access(d, st.leaf[P.w], cw, {N, K}, wacc)) {
        if (wacc.dtype != SANIC_BF16) return false;
        if (!contiguous_runs(wacc, 1, 8)) {
            if (!contiguous_runs(wacc, 0, 8)) return false;
            kn = true;
        }
    } else {
        std::vector<int> gb, gd;
        std::vector<std::string> qv;
        std::string A_, B_;
        Code l1, d1;
        if (!render_weight_affine(d, st.leaf[P.w], cw, {N, K}, l1, d1, "nn", "k0", "_p", gb, gd, qv, A_, B_, negB, unit, false)) return false;
        if (unit % 32 || K % 32 || !packed_access(d, st.leaf[P.w], cw, {N, K}, wacc) || !contiguous_runs(wacc, 1, 32)) return false;
        hasB = !B_.empty();
        unit = std::gcd(unit, (int64_t)256);
        if (unit == 0) unit = 256;
        packed = true;
    }
    // The GEMM's own tiles (groups under 64 are its slowest; it has no others for them)
    const bool aligned = M % 64 == 0 && N % 32 == 0 && K % 64 == 0, narrow = packed && unit < 64;
    if (aligned && !narrow) return false;
    const bool signed4 = packed && wacc.dtype == SANIC_I4;
    const int run = packed ? 32 : 8;                 // elements of a 16-byte chunk

    // ── the rows ──
    Renderer R(d);
    std::vector<std::vector<Sym>> crow;
    std::vector<bool> moves;                         // the row leaf depends on the row
    for (int l : P.rows) {
        const sanic_node& ln = d->nodes[st.leaf[l]];
        std::vector<Sym> cr(ln.rank);
        bool mv = false;
        for (int j = 0; j < ln.rank; j++) {
            int b = st.bind[l][j];
            cr[j] = b == SANIC_BIND_STREAM ? Sym::var(1) : b == P.mdim ? Sym::var(0) : Sym();
            mv |= b == P.mdim;
        }
        std::vector<int> rb, rd;
        bool rok = true, rc = true;
        std::string rr;
        Code l1, d1;
        render_weight_run(d, st.leaf[l], cr, {M, K}, l1, d1, "mm", "k0", "_p", rb, rd, rok, rc, rr, false);
        if (!rok || !rc || rr.empty()) return false;
        crow.push_back(cr);
        moves.push_back(mv);
    }
    // A is one stored leaf: its runs go to the MFMA as loaded
    int raw_row = -1;
    {
        const sanic_expr& e = d->exprs[c.into[P.cslots[0]]];
        if (e.op == SANIC_OP_MUL)
            for (int k = 0; k < 2; k++) {
                const sanic_expr &a = d->exprs[k ? e.b : e.a], &b = d->exprs[k ? e.a : e.b];
                if (a.op == SANIC_EX_ITEM && a.index == P.w && b.op == SANIC_EX_ITEM)
                    for (size_t li = 0; li < P.rows.size(); li++)
                        if (P.rows[li] == b.index) raw_row = (int)li;
            }
    }
    const bool split = raw_row < 0;
    const int SR = (int)P.rslots.size();
    if (packed && SR) return false;

    // ── tile ──
    // "Tall" tiles: 64 rows × 32 columns whose x goes through LDS as the weights do (whole lines of
    // each row; fragment loads would take 64 bytes of 16 rows each).
    Access xacc;
    int tall_row = -1;
    bool tall = M > 32 && N >= 32 && !narrow;
    for (size_t li = 0; li < P.rows.size(); li++)
        if (moves[li]) {
            tall &= tall_row < 0 && sym_access(d, st.leaf[P.rows[li]], crow[li], {M, K}, xacc) && contiguous_runs(xacc, 1, 8);
            tall_row = (int)li;
        }
    tall &= tall_row >= 0;
    auto columns = [&](int64_t mb) {
        int bn = kn ? 64 : 32;
        while (bn > (kn ? 32 : 16) && (mb * ((N + bn - 1) / bn) < 200 || N < bn)) bn /= 2;
        return bn;
    };
    // Up to 32 rows a GEMM tile is half empty (M = 32: 13.4 µs here, 15.0 there). Above, the least of
    // three estimates in µs, rounds of workgroups over the 256 CUs at what a round measured. Per 2048 k:
    // 32-row tiles 9.5 (4-bit 6.5, in groups of 32 10.7), tall ones 12.5 (4-bit 8.5; rows that start
    // off a line cost them 4 more), an eighth to a quarter more for a [K, N] weight. Per 64-deep K step
    // of the GEMM: 0.3 (64 × 32), 0.55 (128 × 32), 0.68 (128 × 64), 1.05 (128 × 128), 4-bit 0.43 and
    // 0.52 (groups of 32, whole tiles only, 0.52 and 0.68), beside 5 for its operand launch. K = 2048,
    // N = 8192, 4-bit: M = 50 tall 12.6, GEMM 15.1, M = 100 23.5 and 17.7. N = 1088, K = 1968: M = 200
    // 13.6 in 32-row tiles, 18.8 tall, 22.9 GEMM; M = 400 24.6, 18.8, 25.0. N = 4000, K = 1536, M = 100:
    // 17.4 in 32-row tiles, 13.3 tall. 4-bit groups of 32, N = 3264, K = 1408, M = 64: 10.3, GEMM 11.8.
    // They hold at K = 8192, N = 2048, with the norm (32-row, tall, GEMM): M = 40 26.8 / 31.3 / 35.4, M = 100
    // 38.9 / 41.5 / 56.6, M = 200 72.8 / 45.5 / 58.7, M = 300 106 / 75.5 / 62.3; the least is taken in each.
    if (M > 32) {
        const double kd = (double)K / 2048.0;
        auto rounds = [](int64_t blocks) { return (double)((blocks + 255) / 256); };
        const int64_t mb2 = (M + 31) / 32, bn2 = columns(mb2), mb4 = (M + 63) / 64;
        const double small = 3.0 + rounds(mb2 * ((N + bn2 - 1) / bn2)) * kd * (narrow ? 10.7 : packed ? 6.5 : 9.5) * (kn ? 1.25 : 1.0);
        const double high = 3.0 + rounds(mb4 * ((N + 31) / 32)) * kd * (packed ? 8.5 : 12.5) * (kn ? 1.125 : 1.0) + (K % 64 ? 4.0 : 0.0);
        const int64_t bm = M > 64 ? 128 : 64, mb = (M + bm - 1) / bm;
        int64_t bn = 128;
        while (bn > 32 && mb * (N / bn) < 256) bn /= 2;
        const double step = narrow ? (bm == 64 ? 0.52 : 0.68) : bn == 128 ? 1.05 : bn == 64 ? 0.68 : bm == 64 ? (packed ? 0.43 : 0.3) : packed ? 0.52 : 0.55;
        const double gemm = (split ? 5.0 : narrow ? 1.5 : 0.0) + rounds(mb * ((N + bn - 1) / bn)) * (double)((K + 63) / 64) * step;
        if (gemm_too && N >= bn && (!narrow || aligned) && gemm < std::min(small, tall ? high : small)) return false;
        tall &= high < small;
    }
    if (!tall) tall_row = -1;
    const int MT = tall ? 4 : M > 16 ? 2 : 1;
    const int64_t NMB = (M + 16 * MT - 1) / (16 * MT);
    const int BN = tall ? 32 : columns(NMB);
    if (N < BN) return false;
    const int64_t NNB = (N + BN - 1) / BN;
    const int NT = BN / 16;
    const int SK = kn || tall ? 64 : packed ? 256 : 128;          // k of a stage
    const int64_t ST = (K + SK - 1) / SK;
    // 16 waves with one stage each where that covers K (128 registers a lane hold one stage), else
    // 8 waves (256 registers) with the next stage requested ahead of each stage's arithmetic
    const int WMAX = ST <= 16 && !tall ? 16 : 8;
    const int ITER = (int)((ST + WMAX - 1) / WMAX), NW = (int)((ST + ITER - 1) / ITER);
    const int SB = kn ? SK * BN * 2 : BN * (packed ? SK / 2 : SK * 2);   // LDS bytes of a stage
    const int ND = SB / 1024;                                     // loads of a stage, 1 KB a wave each
    const int LPR = kn ? BN / 8 : SK / run;                       // 16-byte chunks of an LDS row
    const int RPI = 64 / LPR;                                     // rows of a load
    const bool tail = K % SK != 0;
    const int NTH = NW * 64, RBM = 16 * MT;
    const int XB = tall ? RBM * SK * 2 : 0, NX = XB / 1024;       // x of a stage: LDS bytes, loads
    const int64_t red = (int64_t)NW * MT * NT * 1024;
    const int64_t lds = std::max<int64_t>((int64_t)NW * (SB + XB), red);
    if (tall && unit > SK) unit = SK;
    const int STEPS = SK / 32, UNITS = packed ? SK / (int)unit : 1;

    Code k;
    k.indent = 1;
    k.line("__shared__ __attribute__((aligned(1024))) unsigned char lds[" + str(lds) + "];");
    if (SR) k.line("__shared__ float rs_lds[" + str(NW * RBM * SR) + "];");
    k.line("const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);");
    k.line("const int l16 = lane & 15, lq = lane >> 4;");
    k.line("const idx_t m0 = (idx_t)(blockIdx.x / " + str(NNB) + ") * " + str(RBM) + ";");
    // 32 columns of a [K, N] weight are half a 128-byte line: the two blocks of a line 8 apart, on one
    // XCD, whose L2 then fetches the line once
    k.line("const int nbi = blockIdx.x % " + str(NNB) + ";");
    k.line("const idx_t n_own = (idx_t)(" + (kn && BN == 32 && NNB >= 16 ? "nbi < " + str(NNB / 16 * 16) + " ? nbi / 16 * 16 + nbi % 8 * 2 + nbi / 8 % 2 : nbi" : std::string("nbi")) + ") * " + str(BN) + ";");
    // the last column block starts BN columns before the end and stores only its own columns
    k.line("const idx_t n0 = " + (N % BN ? "n_own < " + str(N - BN) + " ? n_own : (idx_t)" + str(N - BN) : std::string("n_own")) + ";");
    for (int mt = 0; mt < MT; mt++) {
        const std::string r = "(m0 + " + str(mt * 16) + " + l16)";
        k.line("const idx_t mm" + str(mt) + " = " + (M % RBM ? r + " < " + str(M) + " ? " + r + " : (idx_t)" + str(M - 1) : r) + ";");
    }
    k.line("f32x4 acc[" + str(MT) + "][" + str(NT) + "];");
    k.line("#pragma unroll");
    k.line("for (int i = 0; i < " + str(MT) + "; ++i)");
    k.line("  #pragma unroll");
    k.line("  for (int j = 0; j < " + str(NT) + "; ++j) acc[i][j] = (f32x4){0, 0, 0, 0};");
    for (int s = 0; s < SR; s++)
        for (int mt = 0; mt < MT; mt++) k.line("float rp" + str(s) + "_" + str(mt) + " = 0.0f;");
    if (packed) k.line("const bf16x8 ones8 = __builtin_bit_cast(bf16x8, (sanic_u32x4){0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});");
    const std::string wp = R.param(wacc.buffer);
    // What a lane holds of a stage between its request and its use: the row runs, the weights'
    // 16-byte chunks and, 4-bit, the words of the groups' s and z.
    std::vector<int> aoff(P.rows.size());
    int NA = 0;
    for (size_t li = 0; li < P.rows.size(); li++) {
        if ((int)li == tall_row) continue;
        aoff[li] = NA;
        NA += STEPS * (moves[li] ? MT : 1);
    }
    auto aix = [&](size_t li, int j, int mt) { return (int)li == tall_row ? "xf_" + str(j) + "_" + str(mt) : std::string(tall ? "cur[" : "ar[") + str(aoff[li] + j * (moves[li] ? MT : 1) + (moves[li] ? mt : 0)) + "]"; };
    std::vector<std::string> zname, ztype;           // held words, in order of appearance
    std::vector<std::vector<std::pair<std::string, std::string>>> sz(UNITS);
    std::vector<std::string> szdc(UNITS);
    Code rq, wq;                                      // the request's row and group loads; its weight loads
    rq.indent = wq.indent = 2;
    const std::string sk = "(idx_t)s * " + str(SK) + " + ";
    for (int j = 0; j < STEPS; j++) {
        std::string k0 = "kr" + str(j);
        rq.line("const idx_t " + k0 + " = " + sk + str(j * 32) + " + lq * 8;");
        if (tail) {
            rq.line("const idx_t kc" + str(j) + " = " + k0 + " < " + str(K) + " ? " + k0 + " : (idx_t)" + str(K - 8) + ";");
            k0 = "kc" + str(j);
        }
        for (size_t li = 0; li < P.rows.size(); li++)
            for (int mt = 0; mt < (moves[li] ? MT : 1); mt++) {
                if ((int)li == tall_row) continue;
                const std::string sfx = "_" + str(j) + "_" + str(mt) + "_" + str(li);
                std::vector<int> rb, rd;
                bool rok = true, rc = true;
                std::string rr;
                Code l1, d1;
                l1.indent = d1.indent = rq.indent;
                render_weight_run(d, st.leaf[P.rows[li]], crow[li], {M, K}, l1, d1, "mm" + str(mt), k0, sfx, rb, rd, rok, rc, rr, false);
                for (size_t b = 0; b < rb.size(); b++)
                    rq.line("const " + std::string(ctype_of(rd[b])) + "* __restrict__ wb" + str(b) + sfx + " = " + R.param(rb[b]) + ";");
                rq.s << l1.str();
                rq.line("ar[" + str(aoff[li] + j * (moves[li] ? MT : 1) + (moves[li] ? mt : 0)) + "] = " + rr + ";");
            }
    }
    if (packed)
        for (int u = 0; u < UNITS; u++)
            for (int nt = 0; nt < NT; nt++) {
                const std::string sfx = "_z" + str(u) + "_" + str(nt), ku = "ku" + sfx;
                rq.line("const idx_t " + ku + " = " + (tail ? sk + str(u * unit) + " < " + str(K) + " ? " + sk + str(u * unit) + " : (idx_t)" + str(K - 32) : sk + str(u * unit)) + ";");
                std::vector<int> gb, gd;
                std::vector<std::string> qv;
                std::string A_, B_;
                bool nb = false;
                int64_t ud = 0;
                Code l1, d1;
                l1.indent = rq.indent;
                d1.indent = 3;
                render_weight_affine(d, st.leaf[P.w], cw, {N, K}, l1, d1, "(n0 + " + str(nt * 16) + " + l16)", ku, sfx, gb, gd, qv, A_, B_, nb, ud, false, true);
                for (size_t b = 0; b < gb.size(); b++)
                    rq.line("const " + std::string(ctype_of(gd[b])) + "* __restrict__ wb" + str(b) + sfx + " = " + R.param(gb[b]) + ";");
                const std::string text = l1.str();
                rq.s << text;
                static const std::regex re(R"(const (unsigned short|float) (\w+) = )");
                for (auto m = std::sregex_iterator(text.begin(), text.end(), re); m != std::sregex_iterator(); ++m) {
                    rq.line("z" + str(zname.size()) + " = " + (*m)[2].str() + ";");
                    zname.push_back((*m)[2]);
                    ztype.push_back((*m)[1]);
                    szdc[u] += "      const " + ztype.back() + " " + zname.back() + (tall ? " = zc" : " = z") + str(zname.size() - 1) + ";\n";
                }
                szdc[u] += d1.str();
                sz[u].push_back({A_, B_});
            }
    if (tall) {
        // x: rows of the block (a row past the last repeats it), whole 128-byte lines
        rq.line("#pragma unroll");
        rq.line("for (int i = 0; i < " + str(NX) + "; ++i) {");
        rq.line("  const int r = i * 8 + lane / 8, ch = (lane % 8) ^ (r & 7);");
        const std::string mr = "(m0 + r)", kk = "(" + sk + "ch * 8)";
        rq.line("  const idx_t mm = " + (M % RBM ? mr + " < " + str(M) + " ? " + mr + " : (idx_t)" + str(M - 1) : mr) + ", kk = " + (tail ? kk + " < " + str(K) + " ? " + kk + " : (idx_t)" + str(K - 8) : kk) + ";");
        rq.line("  xr[i] = *(const sanic_u32x4_any*)(" + R.param(xacc.buffer) + " + " + xacc.addr.render({"mm", "kk"}) + ");");
        rq.line("}");
    }
    wq.line("#pragma unroll");
    wq.line("for (int i = 0; i < " + str(ND) + "; ++i) {");
    wq.indent++;
    wq.line("const int r = i * " + str(RPI) + " + lane / " + str(LPR) + ", ch = (lane % " + str(LPR) + ") ^ (r & " + str(LPR - 1) + ");");
    {
        std::string kk = kn ? "(" + sk + "r)" : "(" + sk + "ch * " + str(run) + ")";
        if (tail) kk = "(" + kk + " < " + str(K) + " ? " + kk + " : (idx_t)" + str(K - (kn ? 1 : run)) + ")";
        wq.line("const idx_t kk = " + kk + ", nn = " + (kn ? "(n0 + ch * 8)" : "(n0 + r)") + ";");
        wq.line("const unsigned char* src = (const unsigned char*)(" + wp + ") + " + (packed ? "(" + wacc.addr.render({"nn", "kk"}) + " >> 1)" : wacc.addr.render({"nn", "kk"}) + " * 2") + ";");
        wq.line("wr[i] = __builtin_nontemporal_load((const sanic_u32x4_any*)src);");
    }
    wq.indent--;
    wq.line("}");
    std::string zargs, zdecl;
    for (size_t z = 0; z < zname.size(); z++) zargs += ", " + ztype[z] + "& z" + str(z);
    const std::string params = "int s, sanic_u32x4 (&ar)[" + str(std::max(NA, 1)) + "], " + (tall ? "sanic_u32x4 (&xr)[" + str(NX) + "], " : std::string()) + "sanic_u32x4 (&wr)[" + str(ND) + "]" + zargs;
    k.line("auto request = [&](" + params + ") {");
    k.s << rq.str();
    // (the row runs ahead of the weights: loads complete in issue order)
    k.line("  __builtin_amdgcn_sched_barrier(0);");
    k.s << wq.str();
    k.line("  __builtin_amdgcn_sched_barrier(0);");
    k.line("};");
    k.line("auto consume = [&](" + params + (tall ? ", int next" : "") + ") {");
    k.indent++;
    // A fragments (and the row slots): while the weights are in flight, or of a tall tile a step at a time
    auto own = [&](int j) { return sk + str(j * 32) + " + lq * 8 < " + str(K); };
    const char* comp[4] = {"x", "y", "z", "w"};
    auto fragment = [&](int j, int mt) {
            const std::string fs = "_" + str(j) + "_" + str(mt);
            auto item = [&, j, mt](int e) {
                return [&, j, mt, e](int i) -> std::string {
                    for (size_t li = 0; li < P.rows.size(); li++)
                        if (P.rows[li] == i)
                            return "__uint_as_float(" + (e % 2 ? aix(li, j, mt) + "." + comp[e / 2] + " & 0xFFFF0000u" : aix(li, j, mt) + "." + comp[e / 2] + " << 16") + ")";
                    return "0.0f";
                };
            };
            k.line("sanic_u32x4 ah" + fs + (split ? ", al" + fs : "") + ";");
            k.line("{");
            R.memo.emplace_back();
            if (!split) {
                k.line("ah" + fs + " = " + aix(raw_row, j, mt) + ";");
            } else {
                std::vector<std::string> v(8);
                for (int e = 0; e < 8; e++) v[e] = expr_rest(R, k, c.into[P.cslots[0]], P.w, item(e));
                for (int q = 0; q < 4; q++)
                    k.line("{ unsigned h1, l1; split_bf16(" + v[2 * q] + ", " + v[2 * q + 1] + ", h1, l1); ah" + fs + "[" + str(q) + "] = h1; al" + fs + "[" + str(q) + "] = l1; }");
            }
            if (tail) k.line("if (!(" + own(j) + ")) { ah" + fs + " = (sanic_u32x4){0, 0, 0, 0}; " + (split ? "al" + fs + " = ah" + fs + "; " : "") + "}");
            for (int sl = 0; sl < SR; sl++)
                for (int e = 0; e < 8; e++) {
                    const std::string v = expr_rest(R, k, c.into[P.rslots[sl]], -1, item(e));
                    k.line("rp" + str(sl) + "_" + str(mt) + " += " + (tail ? own(j) + " ? " + v + " : 0.0f" : v) + ";");
                }
            R.memo.pop_back();
            k.line("}");
    };
    if (!tall)
        for (int j = 0; j < STEPS; j++)
            for (int mt = 0; mt < MT; mt++) fragment(j, mt);
    k.line("__builtin_amdgcn_sched_barrier(0);");
    // the stage through this wave's LDS slot (its own reads of the last one are done)
    k.line("unsigned char* slot = lds + wv * " + str(SB + XB) + ";");
    if (tall) {
        k.line("#pragma unroll");
        k.line("for (int i = 0; i < " + str(NX) + "; ++i) *(sanic_u32x4*)(slot + " + str(SB) + " + i * 1024 + lane * 16) = xr[i];");
    }
    const std::string write = "for (int i = 0; i < " + str(ND) + "; ++i) *(sanic_u32x4*)(slot + i * 1024 + lane * 16) = wr[i];";
    k.line("#pragma unroll");
    k.line(write);
    if (tall) {
        // the stage is in LDS: its registers take the next one while this one is folded
        if (NA) {
            k.line("sanic_u32x4 cur[" + str(NA) + "];");
            k.line("#pragma unroll");
            k.line("for (int i = 0; i < " + str(NA) + "; ++i) cur[i] = ar[i];");
        }
        for (size_t z = 0; z < zname.size(); z++) k.line("const " + ztype[z] + " zc" + str(z) + " = z" + str(z) + ";");
        std::string zs;
        for (size_t z = 0; z < zname.size(); z++) zs += ", z" + str(z);
        k.line("__builtin_amdgcn_sched_barrier(0);");
        k.line("request(next, ar, xr, wr" + zs + ");");
    }
    const int per = packed ? (int)unit / 32 : STEPS;      // steps of a fold unit
    for (int j = 0; j < STEPS; j++) {
        const int u = packed ? j / per : 0;
        if (packed && j % per == 0) {
            k.line("{");
            k.line("f32x4 tq[" + str(MT) + "][" + str(NT) + "], xq[" + str(MT) + "];");
            k.line("#pragma unroll");
            k.line("for (int i = 0; i < " + str(MT) + "; ++i) {");
            k.line("  xq[i] = (f32x4){0, 0, 0, 0};");
            k.line("  #pragma unroll");
            k.line("  for (int n = 0; n < " + str(NT) + "; ++n) tq[i][n] = (f32x4){0, 0, 0, 0};");
            k.line("}");
        }
        k.line("{");
        k.indent++;
        k.line("bf16x8 bf[" + str(NT) + "];");
        if (kn) {
            // [k][n] rows, read transposed: in each 16-lane group source lane s reads 4 columns
            // 4·(s % 4) of row base + s / 4, lane i gets those 4 rows of column i. Requested and
            // waited for in one asm block.
            k.line("sanic_s16x4 bt[" + str(2 * NT) + "];");
            k.line("const int br = " + str(j * 32) + " + lq * 8 + (l16 >> 2);");
            std::string body, outs, ins;
            for (int i = 0; i < 2 * NT; i++) {
                const int nt = i / 2, h = i % 2;
                k.line("const unsigned ba" + str(i) + " = (unsigned)(size_t)(__attribute__((address_space(3))) const unsigned char*)(slot + (br + " + str(4 * h) + ") * " + str(BN * 2) +
                       " + (((" + str(nt * 2) + " + ((l16 & 3) >> 1)) ^ ((br + " + str(4 * h) + ") & " + str(LPR - 1) + ")) * 8 + (l16 & 1) * 4) * 2);");
                body += "ds_read_b64_tr_b16 %" + str(i) + ", %" + str(2 * NT + i) + "\\n\\t";
                outs += std::string(i ? ", " : "") + "\"=&v\"(bt[" + str(i) + "])";
                ins += std::string(i ? ", " : "") + "\"v\"(ba" + str(i) + ")";
            }
            k.line("asm volatile(\"" + body + "s_waitcnt lgkmcnt(0)\" : " + outs + " : " + ins + " : \"memory\");");
            for (int nt = 0; nt < NT; nt++)
                k.line("bf[" + str(nt) + "] = __builtin_bit_cast(bf16x8, (sanic_s16x8)__builtin_shufflevector(bt[" + str(2 * nt) + "], bt[" + str(2 * nt + 1) + "], 0, 1, 2, 3, 4, 5, 6, 7));");
        } else if (packed) {
            for (int nt = 0; nt < NT; nt++) {
                k.line("{");
                k.line("  const unsigned w = *(const unsigned*)(slot + (" + str(nt * 16) + " + l16) * " + str(LPR * 16) + " + ((" + str(j) + " ^ (l16 & " + str(LPR - 1) + ")) * 16) + lq * 4);");
                k.line("  unsigned ev = w & 0x0F0F0F0Fu, od = (w >> 4) & 0x0F0F0F0Fu;");
                k.line("  asm(\"\" : \"+v\"(ev), \"+v\"(od));");
                std::string words;
                for (int q = 0; q < 4; q++) {
                    const std::string off = signed4 ? " - 8.0f" : "";
                    const std::string e = "(float)((ev >> " + str(8 * q) + ") & 0xFFu)" + off, o = "(float)((od >> " + str(8 * q) + ") & 0xFFu)" + off;
                    words += std::string(q ? ", " : "") + "pk_bf16(" + e + ", " + o + ")";
                }
                k.line("  bf[" + str(nt) + "] = __builtin_bit_cast(bf16x8, (sanic_u32x4){" + words + "});");
                k.line("}");
            }
        } else {
            for (int nt = 0; nt < NT; nt++)
                k.line("bf[" + str(nt) + "] = *(const bf16x8*)(slot + ((" + str(nt * 16) + " + l16) * " + str(LPR) + " + ((" + str(j * 4) + " + lq) ^ (l16 & " + str(LPR - 1) + "))) * 16);");
        }
        for (int mt = 0; mt < MT; mt++) {
            const std::string ms = str(mt), fs = "_" + str(j) + "_" + ms;
            if (tall) {
                // (row tiles past the last row are left out)
                if (M % RBM && mt) k.line("if (m0 + " + str(mt * 16) + " < " + str(M) + ") {");
                k.line("const sanic_u32x4 xf" + fs + " = *(const sanic_u32x4*)(slot + " + str(SB) + " + ((" + str(mt * 16) + " + l16) * 8 + ((" + str(j * 4) + " + lq) ^ (l16 & 7))) * 16);");
                fragment(j, mt);
            }
            for (int h = 0; h < (split ? 2 : 1); h++) {
                const std::string af = std::string("__builtin_bit_cast(bf16x8, ") + (h ? "al" : "ah") + fs + ")";
                for (int nt = 0; nt < NT; nt++) {
                    const std::string a = (packed ? "tq[" : "acc[") + ms + "][" + str(nt) + "]";
                    k.line(a + " = __builtin_amdgcn_mfma_f32_16x16x32_bf16(" + af + ", bf[" + str(nt) + "], " + a + ", 0, 0, 0);");
                }
                if (packed) k.line("xq[" + ms + "] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(" + af + ", ones8, xq[" + ms + "], 0, 0, 0);");
            }
            if (tall && M % RBM && mt) k.line("}");
        }
        k.indent--;
        k.line("}");
        if (packed && j % per == per - 1) {
            k.s << szdc[u];
            for (int nt = 0; nt < NT; nt++) {
                const auto& p = sz[u][nt];
                k.line("#pragma unroll");
                k.line("for (int i = 0; i < " + str(MT) + "; ++i)");
                k.line("  #pragma unroll");
                k.line("  for (int r = 0; r < 4; ++r) {");
                const std::string a = "acc[i][" + str(nt) + "][r]", t = "fmaf(" + p.first + ", tq[i][" + str(nt) + "][r], " + a + ")";
                k.line("    " + a + " = " + (hasB ? "fmaf(" + std::string(negB ? "-" : "") + p.second + ", xq[i][r], " + t + ")" : t) + ";");
                k.line("  }");
            }
            k.line("}");
        }
    }
    k.indent--;
    k.line("};");
    // wave wv takes stages wv, wv + NW, ...; a request past the last stage repeats that one
    auto hold = [&](const std::string& t) {
        k.line("sanic_u32x4 ar" + t + "[" + str(std::max(NA, 1)) + "], wr" + t + "[" + str(ND) + "];");
        if (tall) k.line("sanic_u32x4 xr" + t + "[" + str(NX) + "];");
        for (size_t z = 0; z < zname.size(); z++) k.line(ztype[z] + " z" + t + str(z) + ";");
    };
    auto call = [&](const std::string& fn, const std::string& s, const std::string& t) {
        std::string zs;
        for (size_t z = 0; z < zname.size(); z++) zs += ", z" + t + str(z);
        const std::string next = tall && fn.find("consume") != std::string::npos ? ", stage(it + 1)" : "";
        k.line(fn + "(" + s + ", ar" + t + (tall ? ", xr" + t : std::string()) + ", wr" + t + zs + next + ");");
    };
    const std::string last = str(ST - 1);
    k.line("auto stage = [&](int it) { const int s = wv + it * " + str(NW) + "; return s < " + str(ST) + " ? s : " + last + "; };");
    hold("a");
    call("request", "stage(0)", "a");
    if (tall) {
        k.line("for (int it = 0; it < " + str(ITER) + "; ++it) {");
        k.indent++;
        k.line("if (wv + it * " + str(NW) + " < " + str(ST) + ") {");
        call("  consume", "stage(it)", "a");
        k.line("}");
        k.indent--;
        k.line("}");
    } else if (ITER == 1) {
        call("consume", "wv", "a");
    } else {
        hold("b");
        k.line("for (int it = 0; it < " + str(ITER) + "; it += 2) {");
        k.indent++;
        call("request", "stage(it + 1)", "b");
        k.line("if (wv + it * " + str(NW) + " < " + str(ST) + ") {");
        call("  consume", "stage(it)", "a");
        k.line("}");
        call("request", "stage(it + 2)", "a");
        k.line("if (wv + (it + 1) * " + str(NW) + " < " + str(ST) + ") {");
        call("  consume", "stage(it + 1)", "b");
        k.line("}");
        k.indent--;
        k.line("}");
    }
    // the waves' partial tiles meet in LDS (over the stages' slots, once every wave is done)
    for (int s = 0; s < SR; s++)
        for (int mt = 0; mt < MT; mt++) {
            const std::string r = "rp" + str(s) + "_" + str(mt);
            k.line(r + " = sanic_rows_sum(" + r + ");");
            k.line("if (lane < 16) rs_lds[(wv * " + str(RBM) + " + " + str(mt * 16) + " + lane) * " + str(SR) + " + " + str(s) + "] = " + r + ";");
        }
    k.line("__syncthreads();");
    k.line("float* part = (float*)lds;");
    k.line("#pragma unroll");
    k.line("for (int i = 0; i < " + str(MT) + "; ++i)");
    k.line("  #pragma unroll");
    k.line("  for (int j = 0; j < " + str(NT) + "; ++j)");
    k.line("    #pragma unroll");
    k.line("    for (int r = 0; r < 4; ++r) part[(((wv * " + str(MT) + " + i) * " + str(NT) + " + j) * 4 + r) * 64 + lane] = acc[i][j][r];");
    k.line("__syncthreads();");
    k.line("for (int e = tid; e < " + str(RBM * BN) + "; e += " + str(NTH) + ") {");
    k.indent++;
    k.line("const int row = e / " + str(BN) + ", col = e % " + str(BN) + ";");
    k.line("const idx_t gm = m0 + row, gn = n0 + col;");
    k.line("if (gm >= " + str(M) + " || gn < n_own) continue;");
    k.line("const int at = (((row / 16) * " + str(NT) + " + col / 16) * 4 + row % 4) * 64 + (row % 16) / 4 * 16 + col % 16;");
    std::vector<std::string> gc(st.rank, "0");
    gc[P.mdim] = "gm";
    gc[P.ndim] = "gn";
    for (int j = 0; j < st.rank; j++) k.line("const idx_t g" + str(j) + " = " + gc[j] + ";");
    auto sum = [&](const std::string& arr, int64_t stride, const std::string& ix) {
        std::string s;
        for (int w = 0; w < NW; w++) s = w ? "(" + s + " + " + arr + "[" + str(w * stride) + " + " + ix + "])" : arr + "[" + ix + "]";
        return s;
    };
    k.line("float fs" + str(P.cslots[0]) + " = " + sum("part", MT * NT * 256, "at") + ";");
    for (int s = 0; s < SR; s++) k.line("float fs" + str(P.rslots[s]) + " = " + sum("rs_lds", RBM * SR, "row * " + str(SR) + " + " + str(s)) + ";");
    // Infinities and NaNs: the hi + lo split of an infinity and zeroed operands beside one do not
    // carry it as the fold does, so a point whose sum is not finite is folded again
    k.line("if (!(__builtin_fabsf(fs" + str(P.cslots[0]) + ") <= 3.402823466e38f)) {");
    k.indent++;
    emit_point_fold(R, k, st, "pf");
    for (int s = 0; s < c.slots; s++) k.line("fs" + str(s) + " = pf" + str(s) + ";");
    k.indent--;
    k.line("}");
    R.memo.emplace_back();
    std::string f = R.expr(k, c.project, "", "", "", "fs");
    k.line("const float fold_v = " + f + ";");
    std::string v = "fold_v";
    if (st.epilogue >= 0) {
        R.fold_var = "fold_v";
        v = R.value(k, st.epilogue, gc);
    }
    R.memo.pop_back();
    std::string lin;
    for (int j = 0; j < st.rank; j++)
        lin = j == 0 ? "(idx_t)(" + gc[0] + ")" : "(" + lin + " * " + str(st.grid[j]) + " + (idx_t)(" + gc[j] + "))";
    k.line(store_stmt(R.param(st.out_buffer), lin, st.out_dtype, v, false, d->buffers[st.out_buffer].scale));
    k.indent--;
    k.line("}");

    const std::string kname = "sanic_rows_" + str(M) + "x" + str(N) + "x" + str(K);
    std::ostringstream src;
    src << kPrelude;
    src << "typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8;\n";
    src << "typedef short sanic_s16x4 __attribute__((ext_vector_type(4)));\n";
    src << "typedef short sanic_s16x8 __attribute__((ext_vector_type(8)));\n";
    src << "typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;\n";
    src << kSplitBf16;
    src << "typedef unsigned sanic_u32x4_any __attribute__((ext_vector_type(4), aligned(1)));\n";
    src << R.args_struct({});
    src << "extern \"C\" __global__ void __launch_bounds__(" << NTH << ") " << kname << "(Args a) {\n" << R.entry() << k.str() << "}\n";
    out.kernel_kind = "skeleton:gemm_rows[" + str(RBM) + "x" + str(BN) + (split ? ",a2" : "") + (packed ? unit < 64 ? ",g32" : ",grp" : "") + (kn ? ",kn" : "") + ",w" + str(NW) + "x" + str(ITER) + "]";
    out.variants = 1;
    out.source = src.str();
    out.launches.push_back({kname, "", dim3((unsigned)(NMB * NNB)), dim3((unsigned)NTH), 0, R.arg_list()});
    return true;
}

}  // namespace sanic
