// FlashAttention prefill skeleton: the online-softmax (m, ℓ, o) carrier over the key axis on
// bf16 MFMA (v_mfma_f32_16x16x32_bf16), for stages whose query grid has a head axis and a
// query-row axis (the causal / sliding-window prefill of the reference's
// scaled_dot_product_attention, /root/reference/src/nn.rs:27-105, folded as
// /root/reference/tests/laws.rs:108-126).
//
// Structure required (read from the carrier and the leaves, never from names): the carrier of
// skel_attention.cpp (a Plain(Max) score slot, ExpShifted slots with constant or value `into`);
// the score leaf = one in-body contraction Σ_d Q·K (both affine bf16 views with d contiguous,
// the head entering K as ⌊h/rep⌋) with scalar factors and additive mask terms around it; the
// value leaf an affine bf16 view.
//
// Any number of rows and keys with row-major V; whole tiles (rows % 128 = 0, keys % 64 = 0) with
// V^T. Kernel shape (one workgroup = one head × 128 query rows, 4 waves × 32 rows; 64 rows, 4
// waves × 16, for lengths off those tiles):
//   S^T = K·Q^T per 64-key tile (so a lane owns one query column: the running max, the sum and
//   the O rescale are lane-local, with one 4-lane shuffle per tile for the max);
//   O^T += V^T·P^T with P packed to bf16 in registers (the MFMA k-order is chosen to match the
//   S^T accumulator layout, so P never goes through LDS);
//   K and V tiles go from global memory straight into a ring of three LDS buffers, two tiles
//   ahead; Q stays in registers; exp2 with log2(e) folded; the −∞ guard of the
//   carrier's combine on the rescale; tiles outside every row's honest window are skipped and
//   tiles entirely inside it skip the mask arithmetic;
//   blockIdx → (KV head, query head, query block) places all query heads of one KV head on one
//   XCD (blockIdx mod 8) so their K/V stay in that XCD's L2, heaviest causal blocks first.
#include <algorithm>
#include <cmath>

#include <functional>
#include <regex>

#include "emit.h"
#include "skeletons.h"

namespace sanic {

namespace {

// Up to this many scores (128 × 128) attention with f32 operands stays with the generic fold.
const int64_t kFoldScores = 128 * 128;

struct FlashPlan {
    int sleaf = -1, vleaf = -1, max_slot = -1;
    std::vector<int> vec_slots, scalar_slots;
    std::vector<double> scalar_into;
    int hdim = -1, qdim = -1, edim = -1;
    int64_t NH = 1, NQ = 1, E = 1, T = 1, HD = 1;
    int rep = 1;
    int dot_reduce = -1;
    Access qacc, kacc, vacc;
    // a query side that is an elementwise expression (RoPE'd Q, say) rather than one affine
    // view: rendered per element once per workgroup, at coordinates qcoords over the vars
    // {0: head, 1: key, 2: d, 3: query row}
    bool qexpr = false;
    bool ragged = false;      // rows not a multiple of 128 or keys not a multiple of 64
    int qnode = -1;
    std::vector<Sym> qcoords;
};

bool has_reduce_below(const sanic_program_desc* d, int node) {
    std::vector<int> st{node};
    while (!st.empty()) {
        int i = st.back();
        st.pop_back();
        if (d->nodes[i].kind == SANIC_NODE_REDUCE || d->nodes[i].kind == SANIC_NODE_SCAN) return true;
        for (int q = 0; q < d->nodes[i].n_in; q++) st.push_back(d->nodes[i].in[q]);
    }
    return false;
}

bool sym_is_var(const Sym& s, int& var) {
    if (s.c0 != 0 || s.terms.size() != 1) return false;
    const SymTerm& t = s.terms[0];
    if (t.coef != 1 || t.div != 1 || t.mod != 0) return false;
    var = t.var;
    return true;
}

// address = c0 + Σ terms; returns per-var coefficient (div 1, no mod) and the h term's div
bool split_addr(const Sym& a, int nvars, std::vector<int64_t>& coef, int& hdiv, int64_t& hcoef) {
    coef.assign(nvars, 0);
    hdiv = 0;
    hcoef = 0;
    for (auto& t : a.terms) {
        if (t.mod) return false;
        if (t.var == 0 && t.div != 1) {
            if (hdiv) return false;
            hdiv = (int)t.div;
            hcoef = t.coef;
            continue;
        }
        if (t.div != 1) return false;
        coef[t.var] += t.coef;
    }
    return true;
}

bool find_flash_dot(const sanic_program_desc* d, int node, const std::vector<Sym>& c, const std::vector<int64_t>& ext,
                    FlashPlan& P) {
    const sanic_node& n = d->nodes[node];
    if (n.kind == SANIC_NODE_MAP) {
        int found = 0;
        for (int k = 0; k < n.n_in; k++) {
            const sanic_node& m = d->nodes[n.in[k]];
            bool has_reduce = false;
            std::vector<int> st{n.in[k]};
            while (!st.empty()) {
                int i = st.back(); st.pop_back();
                if (d->nodes[i].kind == SANIC_NODE_REDUCE || d->nodes[i].kind == SANIC_NODE_SCAN) has_reduce = true;
                for (int q = 0; q < d->nodes[i].n_in; q++) st.push_back(d->nodes[i].in[q]);
            }
            if (!has_reduce) continue;
            int lead = n.rank - m.rank;
            std::vector<Sym> cc(m.rank);
            for (int j = 0; j < m.rank; j++) cc[j] = m.shape[j] == 1 ? Sym() : c[lead + j];
            if (!find_flash_dot(d, n.in[k], cc, ext, P)) return false;
            found++;
        }
        return found == 1;
    }
    if (n.kind != SANIC_NODE_REDUCE || n.op != SANIC_MON_ADD) return false;
    const sanic_node& mp = d->nodes[n.in[0]];
    if (mp.kind != SANIC_NODE_MAP || mp.op != SANIC_OP_MUL) return false;
    // vars: 0 = head, 1 = key (stream), 2 = contraction d, 3 = query row
    std::vector<Sym> mc;
    for (int j = 0, o = 0; j < mp.rank; j++) mc.push_back(j == n.dim ? Sym::var(2) : c[o++]);
    std::vector<int64_t> ext4 = {ext[0], ext[1], mp.shape[n.dim], ext[3]};
    int kside = -1;
    std::vector<std::vector<Sym>> cc(2);
    for (int k = 0; k < 2; k++) {
        const sanic_node& ch = d->nodes[mp.in[k]];
        int lead = mp.rank - ch.rank;
        cc[k].resize(ch.rank);
        bool moves = false;
        for (int j = 0; j < ch.rank; j++) {
            cc[k][j] = ch.shape[j] == 1 ? Sym() : mc[lead + j];
            for (auto& t : cc[k][j].terms) moves |= t.var == 1;
        }
        if (moves) {
            if (kside >= 0) return false;
            kside = k;
        }
    }
    if (kside < 0) return false;
    if (!sym_access(d, mp.in[kside], cc[kside], ext4, P.kacc)) return false;
    if (!sym_access(d, mp.in[1 - kside], cc[1 - kside], ext4, P.qacc)) {
        if (has_reduce_below(d, mp.in[1 - kside])) return false;
        P.qexpr = true;
        P.qnode = mp.in[1 - kside];
        P.qcoords = cc[1 - kside];
    }
    P.dot_reduce = node;
    P.HD = mp.shape[n.dim];
    return true;
}

// How a window edge moves with the query row: `dir` 0 not at all, 1 rising, −1 falling, 2 one of
// the two (by a factor known at run time). `convex` and `concave`: made of lines of whole slopes by
// maxima, or by minima. A straight edge is both.
struct EdgeForm {
    int dir = 0;
    bool convex = true, concave = true;
};

bool join_edges(const EdgeForm& x, const EdgeForm& y, EdgeForm& out) {
    if (x.dir && y.dir && (x.dir != y.dir || x.dir == 2)) return false;
    out = {x.dir ? x.dir : y.dir, x.convex && y.convex, x.concave && y.concave};
    return true;
}

EdgeForm turned(const EdgeForm& e) { return {e.dir == 2 ? 2 : -e.dir, e.concave, e.convex}; }

std::vector<Sym> kid_coords(const sanic_program_desc* d, int node, int k, const std::vector<Sym>& c) {
    const sanic_node& n = d->nodes[node];
    const sanic_node& m = d->nodes[n.in[k]];
    std::vector<Sym> cc(m.rank);
    for (int j = 0; j < m.rank; j++) cc[j] = m.shape[j] == 1 ? Sym() : c[n.rank - m.rank + j];
    return cc;
}

bool sym_form(const Sym& s, int row, EdgeForm& out) {
    out = EdgeForm();
    for (auto& t : s.terms) {
        if (t.var != row || !t.coef) continue;
        if (t.mod || !join_edges(out, {t.coef > 0 ? 1 : -1, t.div == 1, t.div == 1}, out)) return false;
    }
    return true;
}

// The form of an edge at coordinates `c` over the grid's variables, of which `row` is the query row;
// false for an edge that is not known to move one way.
bool edge_form(const sanic_program_desc* d, int node, const std::vector<Sym>& c, const std::vector<int64_t>& ext, int row, EdgeForm& out) {
    const sanic_node& n = d->nodes[node];
    bool moves = false;
    for (auto& s : c)
        for (auto& t : s.terms) moves |= t.var == row;
    out = EdgeForm();
    if (!moves || n.kind == SANIC_NODE_CONST) return true;
    if (n.kind == SANIC_NODE_IOTA) return sym_form(c[0], row, out);
    if (n.kind == SANIC_NODE_COORDINATE) return sym_form(c[n.dim], row, out);
    if (n.kind == SANIC_NODE_VIEW || n.kind == SANIC_NODE_REINDEX) {
        std::vector<Sym> sc;
        return sym_child_coords(d, node, c, ext, sc) && edge_form(d, n.in[0], sc, ext, row, out);
    }
    if (n.kind != SANIC_NODE_MAP) return false;
    EdgeForm e[2];
    for (int k = 0; k < n.n_in; k++)
        if (k > 1 || !edge_form(d, n.in[k], kid_coords(d, node, k, c), ext, row, e[k])) return false;
    switch (n.op) {
    case SANIC_OP_ADD: return join_edges(e[0], e[1], out);
    case SANIC_OP_SUB: return join_edges(e[0], turned(e[1]), out);
    case SANIC_OP_NEG: out = turned(e[0]); return true;
    case SANIC_OP_ROUND_F32: out = e[0]; return true;
    case SANIC_OP_MAX:
    case SANIC_OP_MIN:
        if (!join_edges(e[0], e[1], out)) return false;
        (n.op == SANIC_OP_MAX ? out.concave : out.convex) &= !out.dir;
        return true;
    case SANIC_OP_MUL:
    case SANIC_OP_DIV: {
        // one side moves, the other scales it
        const int k = e[0].dir ? 0 : 1;
        if (e[1 - k].dir || (n.op == SANIC_OP_DIV && k)) return false;
        out = e[k];
        if (!out.dir) return true;
        const sanic_node& f = d->nodes[n.in[1 - k]];
        if (f.kind != SANIC_NODE_CONST) {
            out = {2, false, false};
            return true;
        }
        if (!std::isfinite(f.value) || (n.op == SANIC_OP_DIV && f.value == 0.0)) return false;
        if (f.value == 0.0) out = EdgeForm();
        if (f.value < 0.0) out = turned(out);
        const bool whole = n.op == SANIC_OP_MUL && f.value == std::floor(f.value);
        if (out.dir && !whole) out.convex = out.concave = false;
        return true;
    }
    default: return false;
    }
}

// The coordinates of a window edge over the grid's variables.
std::vector<Sym> edge_coords(const WindowBound& w) {
    std::vector<Sym> c(w.bind.size());
    for (size_t j = 0; j < c.size(); j++)
        if (w.bind[j] >= 0) c[j] = Sym::var(w.bind[j]);
    return c;
}

// A block's and a wave's key range is the union of its first and last row's windows, and its fully
// visible tiles their intersection. That holds for the rows between if each side's edges all move one
// way, and if no window between is empty (which stands for the whole stream) where those two are
// not: sure where one side stands still or the two move apart, and where they move together if the
// lower edges are convex and the upper ones concave.
bool window_between_rows(const sanic_program_desc* d, const sanic_stage& st, int qdim) {
    const std::vector<int64_t> ext(st.grid, st.grid + st.rank);
    EdgeForm side[2];
    for (auto& w : honest_window(d, st)) {
        EdgeForm e;
        const bool low = w.kind == WindowBound::LO_CEIL;
        if (!edge_form(d, w.node, edge_coords(w), ext, qdim, e) || !join_edges(side[low], e, side[low])) return false;
    }
    const EdgeForm &hi = side[0], &lo = side[1];
    if (!hi.dir || !lo.dir) return true;
    return hi.dir != 2 && lo.dir != 2 && (hi.dir != lo.dir || (lo.convex && hi.concave));
}

// The value of a window edge at a query row, where it is made of constants and the row alone.
double edge_at(const sanic_program_desc* d, int node, const std::vector<Sym>& c, const std::vector<int64_t>& ext, int qdim, double row, bool& known) {
    const sanic_node& n = d->nodes[node];
    auto at = [&](const Sym& s) {
        double v = (double)s.c0;
        for (auto& t : s.terms) {
            if (t.var != qdim) known = false;
            int64_t x = (int64_t)row / t.div;
            v += (double)(t.coef * (t.mod ? x % t.mod : x));
        }
        return v;
    };
    if (n.kind == SANIC_NODE_CONST) return n.value;
    if (n.kind == SANIC_NODE_COORDINATE) return at(c[n.dim]);
    if (n.kind == SANIC_NODE_IOTA) return at(c[0]);
    std::vector<Sym> sc;
    if ((n.kind == SANIC_NODE_VIEW || n.kind == SANIC_NODE_REINDEX) && sym_child_coords(d, node, c, ext, sc))
        return edge_at(d, n.in[0], sc, ext, qdim, row, known);
    if (n.kind == SANIC_NODE_MAP && n.n_in <= 2) {
        double v[2] = {0.0, 0.0};
        for (int k = 0; k < n.n_in; k++) v[k] = edge_at(d, n.in[k], kid_coords(d, node, k, c), ext, qdim, row, known);
        switch (n.op) {
        case SANIC_OP_ADD: return v[0] + v[1];
        case SANIC_OP_SUB: return v[0] - v[1];
        case SANIC_OP_MUL: return v[0] * v[1];
        case SANIC_OP_DIV: return v[0] / v[1];
        case SANIC_OP_MAX: return std::max(v[0], v[1]);
        case SANIC_OP_MIN: return std::min(v[0], v[1]);
        case SANIC_OP_NEG: return -v[0];
        default: break;
        }
    }
    known = false;
    return 0.0;
}

// The most keys that a block of `rows` query rows sees between them, over the first, the middle and
// the last block (all, where an edge is not known here).
int64_t longest_window(const sanic_program_desc* d, const sanic_stage& st, int qdim, int64_t nq, int64_t rows) {
    const std::vector<int64_t> ext(st.grid, st.grid + st.rank);
    const auto win = honest_window(d, st);
    int64_t most = 0;
    for (int64_t r0 : {(int64_t)0, nq / 2, std::max<int64_t>(0, nq - rows)}) {
        const int64_t r1 = std::min(nq, r0 + rows) - 1;
        double lo = 0.0, hi = (double)st.stream;
        for (auto& w : win) {
            bool known = true;
            const auto c = edge_coords(w);
            const double a = edge_at(d, w.node, c, ext, qdim, (double)r0, known), b = edge_at(d, w.node, c, ext, qdim, (double)r1, known);
            if (!known) continue;
            if (w.kind == WindowBound::LO_CEIL) lo = std::max(lo, std::min(a, b));
            else hi = std::min(hi, std::max(a, b) + 1.0);
        }
        most = std::max(most, hi > lo ? (int64_t)(hi - lo) : st.stream);
    }
    return most;
}

// The attention structure of a stage: carrier, dims and the affine K and V (any storage dtype).
bool attention_plan(const sanic_program_desc* d, int si, FlashPlan& P) {
    const sanic_stage& st = d->stages[si];
    if (st.kind != SANIC_STAGE_FUSED || st.n_leaves != 2) return false;
    const sanic_carrier& c = st.carrier;
    P = FlashPlan();
    for (int k = 0; k < c.slots; k++)
        if (c.kind[k].kind == SANIC_SLOT_PLAIN && c.kind[k].monoid == SANIC_MON_MAX) {
            if (P.max_slot >= 0) return false;
            P.max_slot = k;
        }
    if (P.max_slot < 0) return false;
    const sanic_expr& mi = d->exprs[c.into[P.max_slot]];
    if (mi.op != SANIC_EX_ITEM) return false;
    P.sleaf = mi.index;
    for (int k = 0; k < c.slots; k++) {
        if (k == P.max_slot) continue;
        if (c.kind[k].kind != SANIC_SLOT_EXP_SHIFTED || c.kind[k].ref_slot != P.max_slot) return false;
        const sanic_expr& e = d->exprs[c.into[k]];
        if (e.op == SANIC_EX_ITEM && e.index != P.sleaf) {
            if (P.vleaf >= 0 && P.vleaf != e.index) return false;
            P.vleaf = e.index;
            P.vec_slots.push_back(k);
        } else if (e.op == SANIC_EX_CONST) {
            P.scalar_slots.push_back(k);
            P.scalar_into.push_back(e.value);
        } else {
            return false;
        }
    }
    if (P.vleaf < 0 || P.vec_slots.size() != 1) return false;
    const sanic_node& sl = d->nodes[st.leaf[P.sleaf]];
    const sanic_node& vl = d->nodes[st.leaf[P.vleaf]];
    std::vector<bool> in_s(st.rank, false), in_v(st.rank, false);
    for (int j = 0; j < sl.rank; j++) if (st.bind[P.sleaf][j] >= 0) in_s[st.bind[P.sleaf][j]] = true;
    for (int j = 0; j < vl.rank; j++) if (st.bind[P.vleaf][j] >= 0) in_v[st.bind[P.vleaf][j]] = true;
    std::vector<int> qdims;
    for (int j = 0; j < st.rank; j++) {
        if (st.grid[j] == 1) continue;
        if (in_v[j] && !in_s[j]) {
            if (P.edim >= 0) return false;
            P.edim = j;
        } else {
            qdims.push_back(j);
        }
    }
    if (P.edim < 0 || qdims.empty() || qdims.size() > 2) return false;
    // the head dim (none for a single head) is the one the value leaf reads; the query row is
    // read only by the score
    for (int j : qdims) {
        if (in_v[j]) P.hdim = j;
        else P.qdim = j;
    }
    if (P.qdim < 0 || (P.hdim < 0) != (qdims.size() == 1)) return false;
    P.NH = P.hdim < 0 ? 1 : st.grid[P.hdim];
    P.NQ = st.grid[P.qdim];
    P.E = st.grid[P.edim];
    P.T = st.stream;
    std::vector<Sym> scs(sl.rank);
    for (int j = 0; j < sl.rank; j++) {
        int b = st.bind[P.sleaf][j];
        scs[j] = b == SANIC_BIND_STREAM ? Sym::var(1) : b == P.hdim ? Sym::var(0) : b == P.qdim ? Sym::var(3) : Sym();
    }
    if (!find_flash_dot(d, st.leaf[P.sleaf], scs, {P.NH, P.T, 1, P.NQ}, P)) return false;
    std::vector<Sym> vcs(vl.rank);
    for (int j = 0; j < vl.rank; j++) {
        int b = st.bind[P.vleaf][j];
        vcs[j] = b == SANIC_BIND_STREAM ? Sym::var(1) : b == P.hdim ? Sym::var(0) : b == P.edim ? Sym::var(2) : Sym();
    }
    if (!sym_access(d, st.leaf[P.vleaf], vcs, {P.NH, P.T, P.E}, P.vacc)) return false;
    return window_between_rows(d, st, P.qdim);
}

bool flash_plan(const sanic_program_desc* d, int si, FlashPlan& P) {
    if (!attention_plan(d, si, P)) return false;
    const sanic_stage& st = d->stages[si];
    if ((!P.qexpr && P.qacc.dtype != SANIC_BF16) || P.kacc.dtype != SANIC_BF16 || P.vacc.dtype != SANIC_BF16) return false;
    if (P.HD != 64 || P.E != 64) return false;
    P.ragged = P.NQ % 128 != 0 || P.T % 64 != 0 || P.hdim < 0;
    // Q: (h, d, i) with d contiguous; K: (⌊h/rep⌋, t, d) with d contiguous; V: (⌊h/rep⌋, t, e)
    std::vector<int64_t> qc, kc, vc;
    int qh, kh, vh;
    int64_t qhc, khc, vhc;
    if (!P.qexpr && (!split_addr(P.qacc.addr, 4, qc, qh, qhc) || qh != 0 || qc[2] != 1 || qc[1] != 0)) return false;
    if (!split_addr(P.kacc.addr, 4, kc, kh, khc)) return false;
    if (!split_addr(P.vacc.addr, 3, vc, vh, vhc)) return false;
    if (kc[2] != 1 || kc[3] != 0 || (vc[2] != 1 && vc[1] != 1)) return false;
    int repk = kh ? kh : (kc[0] ? 1 : (int)P.NH);
    int repv = vh ? vh : (vc[0] ? 1 : (int)P.NH);
    if (repk != repv) return false;
    P.rep = repk;
    if (P.ragged) {
        // They go here only where the schedule is the backend's to choose and
        // the tile rows are whole 16-byte chunks of row-major K and V
        if (!sched_is_auto(st.sched) || vc[2] != 1) return false;
        // A row block's keys are one CU's here: a few query rows over a long cache go to the kernel
        // below, which gives each block of 16 rows up to 8 workgroups. Here and there, µs: no head axis,
        // 17 rows over 1024 keys 12.2 and 8.3, 16 over 4096 34.4 and 13.8, 4 over 65536 525 and 121 (the
        // split fold 403); 32 heads of 16 rows (32 blocks of 16) 12.8 and 10.4 over 1024, of 32 (64) 12.8 and
        // 11.7, of 64 (128) 13.8 and 14.7, over 4096 36.0 and 38.3
        if (!P.qexpr && !lean_scratch() && P.NH * ((P.NQ + 15) / 16) <= 64 && P.T >= 1024 && P.T >= 4 * P.NQ && P.NH * P.NQ * P.T > kFoldScores) return false;
        for (int64_t v : {kc[0], kc[1], khc, P.kacc.addr.c0, vc[0], vc[1], vhc, P.vacc.addr.c0})
            if (v % 8) return false;
        if (!P.qexpr)
            for (int64_t v : {qc[0], qc[3], P.qacc.addr.c0})
                if (v % 8) return false;
    }
    return true;
}

// On tiles every row sees entirely, the score must be `dot · c` (the additive mask terms are
// zero there): read c off the leaf so the tile can fold the scale into the exp2 argument.
bool full_score_scale(const sanic_program_desc* d, int node, int dot, const std::vector<WindowBound>& win, double& c) {
    const sanic_node& n = d->nodes[node];
    if (node == dot) { c = 1.0; return true; }
    if (n.kind != SANIC_NODE_MAP) return false;
    if (n.op == SANIC_OP_ADD) {
        for (int k = 0; k < 2; k++)
            for (auto& w : win)
                if (n.in[k] == w.where_node) return full_score_scale(d, n.in[1 - k], dot, win, c);
        return false;
    }
    if (n.op == SANIC_OP_MUL) {
        for (int k = 0; k < 2; k++) {
            const sanic_node& o = d->nodes[n.in[1 - k]];
            if (o.kind == SANIC_NODE_CONST && o.rank == 0) {
                double inner;
                if (!full_score_scale(d, n.in[k], dot, win, inner)) return false;
                c = inner * o.value;
                return true;
            }
        }
    }
    return false;
}

}  // namespace

bool lower_flash_prefill(const sanic_program_desc* d, int si, int64_t& scratch, LoweredStage& out) {
    FlashPlan P;
    if (!flash_plan(d, si, P)) return false;
    const sanic_stage& st = d->stages[si];
    const sanic_carrier& c = st.carrier;
    const int64_t NH = P.NH, NQ = P.NQ, T = P.T, E = P.E, HD = P.HD;
    // Lengths off the tiles (a prompt nobody padded) and a single head were folded in f32 by the generic fold: here
    // the softmax weights, and a query side that is an expression, go to the MFMA as sums of bf16 terms:
    // two (16 significant bits) where the output is bf16, whose rounding is 128 times theirs, else three
    // (24 bits, the fold's own). RMS error against 64 bits, fold and here, 2 heads, S = 1000: f32 output
    // 2.5e-8 and 2.3e-8, float16 2.43e-5 and bf16 1.94e-4 in both. One query tile per wave holds the other
    // terms in the registers the second tile had (two: 117 VGPRs) and gives short prompts twice the
    // workgroups. 32/8 heads, S = 1000, window 256, with the RoPE stages: 20.0 ms in the generic fold (it
    // forms q·k again for each of the 64 value columns) → 20.1 µs. Three terms, 32/8 heads, S = 1000,
    // causal: 18.1 → 20.9 µs; 8/2 heads, S = 4000: 53 → 60.
    const int NP = !P.ragged ? 1 : st.out_dtype == SANIC_BF16 ? 2 : 3;   // bf16 terms of a softmax weight
    const int fvar = P.ragged ? 0 : d->stages[si].sched.variant;
    // Launches that leave CUs short of waves: 64-row blocks (up to 512 of 128 rows; 32 heads, S = 2048
    // 58 → 47 µs, S = 4096, 1024 blocks, 108 against 123), and KS teams of 4 waves per block, each with
    // every KS-th key tile, merged in LDS at the end — a wave's tile takes ≈ 1.5 µs of dependent phases
    // whatever else the CU does, so the key loop's length is the time. One, 2 and 4 teams: 4/1 heads,
    // S = 2048 40 / 30 / 24 µs; 8 heads, S = 4096 75 / 53 / 51; 16 heads, S = 2048 (512 blocks) 44 / 35 / 37;
    // 16 heads, S = 4096 (1024 blocks) 78 / 70 / 87, S = 2048, 32 heads 47 / 49 / 63; and with few tiles the
    // merge costs more: 6 tiles (S = 1000, window 256) 20 / 22 / 29, 2 tiles 11.6 / 12.4.
    // Each team keeps a running maximum of its own, so on whole tiles, where the weights are one bf16
    // term, their rounding is against other reference points than in the 128-row form: outputs differ
    // by 1e-3 of their RMS (the bf16 of the weights), RMS error against 64 bits 1.11e-4 here and 1.19e-4 there
    // (2 heads, S = 2048), 8.9e-5 and 9.1e-5 (8 heads, S = 4096).
    const bool few = P.ragged || (NH * (NQ / 128) <= 512 && (fvar == 0 || fvar == 3));
    const int QT = few ? 1 : 2;                      // 16-row query tiles per wave
    const int RB = 64 * QT;                          // query rows per workgroup (a team's 4 waves)
    const int64_t NQB = (NQ + RB - 1) / RB;
    const int64_t tiles = longest_window(d, st, P.qdim, NQ, RB) / 64 + 1;
    int KS = 1;
    if (few && tiles >= 12 && NH * NQB <= 256) KS = 4;
    else if (few && ((tiles >= 8 && NH * NQB <= 512) || (tiles >= 48 && NH * NQB <= 1024))) KS = 2;
    const int NBUF = KS > 1 ? 2 : 3;                 // LDS buffers of a team's tile ring
    const std::string KSs = std::to_string(KS), step = std::to_string(64 * KS);
    const std::string QTs = std::to_string(QT), RBs = std::to_string(RB);
    // the last row or key of the operands, where a tile runs past it
    auto row_clamp = [&](const std::string& r) { return P.ragged ? "sanic_min(" + r + ", (idx_t)" + std::to_string(NQ - 1) + ")" : "(" + r + ")"; };
    auto key_clamp = [&](const std::string& r) { return P.ragged ? "sanic_min(" + r + ", (idx_t)" + std::to_string(T - 1) + ")" : "(" + r + ")"; };
    std::vector<int64_t> qc, kc, vc;
    int qh, kh, vh;
    int64_t qhc, khc, vhc;
    if (!P.qexpr) split_addr(P.qacc.addr, 4, qc, qh, qhc);
    split_addr(P.kacc.addr, 4, kc, kh, khc);
    split_addr(P.vacc.addr, 3, vc, vh, vhc);
    const bool v_rows = vc[2] == 1;                  // V[t, e] rows (else V^T with t contiguous)
    auto hterm = [&](const std::vector<int64_t>& cf, int div, int64_t hcf) {
        // address contribution of head hh
        if (div) return "(hh / " + std::to_string(div) + ") * " + std::to_string(hcf);
        return "hh * " + std::to_string(cf[0]);
    };

    Renderer R(d);
    // score functions: the leaf with its contraction replaced by `dotv`; the "full" variant also
    // drops the additive mask terms (used only on tiles every row sees entirely)
    auto win = honest_window(d, st);
    const sanic_node& sl = d->nodes[st.leaf[P.sleaf]];
    std::vector<std::string> lc(sl.rank);
    for (int j = 0; j < sl.rank; j++) {
        int b = st.bind[P.sleaf][j];
        lc[j] = b == SANIC_BIND_STREAM ? "kj" : b == P.hdim ? "hh" : b == P.qdim ? "qi" : "0";
    }
    Renderer Rs(d);
    Rs.take_buffers(R);
    Code sp, sf;
    sp.indent = sf.indent = 1;
    Rs.subst[P.dot_reduce] = "dotv";
    std::string vpart = Rs.value(sp, st.leaf[P.sleaf], lc);
    std::string entry_part = Rs.entry();
    Renderer Rf(d);
    Rf.take_buffers(Rs);
    Rf.subst[P.dot_reduce] = "dotv";
    for (auto& w : win) Rf.subst[w.where_node] = "0.0f";
    std::string vfull = Rf.value(sf, st.leaf[P.sleaf], lc);
    std::string entry_full = Rf.entry();
    R.take_buffers(Rf);
    double scale_c = 0.0;
    const bool scale_known = full_score_scale(d, st.leaf[P.sleaf], P.dot_reduce, win, scale_c) && scale_c > 0.0;

    // window edges per query row (for tile skipping / full-tile detection)
    Code wc;
    wc.indent = 1;
    Renderer Rw(d);
    Rw.take_buffers(R);
    std::vector<std::string> gcw(st.rank, "0");
    if (P.hdim >= 0) gcw[P.hdim] = "hh";
    gcw[P.qdim] = "qrow";
    {
        Code tmp;
        tmp.indent = 1;
        // emit_window names grid coords g<j>
        for (int j = 0; j < st.rank; j++) tmp.line("const idx_t g" + std::to_string(j) + " = " + gcw[j] + ";");
        emit_window(Rw, tmp, st, win, "wlo", "whi");
        wc.s << tmp.str();
    }
    R.take_buffers(Rw);

    // finish: project (+ epilogue) and the narrowing store of one output point
    Renderer Ro(d);
    Ro.take_buffers(R);
    Code fo;
    fo.indent = 1;
    {
        for (int sl2 = 0; sl2 < c.slots; sl2++) fo.line("const float fs" + std::to_string(sl2) + " = fs[" + std::to_string(sl2) + "];");
        std::string f = Ro.expr(fo, c.project, "", "", "", "fs");
        fo.line("const float fold_v = " + f + ";");
        std::vector<std::string> gc(st.rank, "0");
        if (P.hdim >= 0) gc[P.hdim] = "hh";
        gc[P.qdim] = "qi";
        gc[P.edim] = "ee";
        std::string v = "fold_v";
        if (st.epilogue >= 0) {
            Ro.fold_var = "fold_v";
            v = Ro.value(fo, st.epilogue, gc);
        }
        std::string lin;
        for (int j = 0; j < st.rank; j++)
            lin = j == 0 ? "(idx_t)(" + gc[0] + ")" : "(" + lin + " * " + std::to_string(st.grid[j]) + " + (idx_t)(" + gc[j] + "))";
        fo.line(store_stmt(Ro.param(st.out_buffer), lin, st.out_dtype, v, false, d->buffers[st.out_buffer].scale));
    }
    R.take_buffers(Ro);
    if (P.qexpr) {
        // register the expression's buffers before the argument struct is written
        Code scratch_code;
        R.memo.emplace_back();
        std::vector<std::string> cs;
        for (auto& sy : P.qcoords) cs.push_back(sy.render({"hh", "(idx_t)0", "dd", "qrow"}));
        R.value(scratch_code, P.qnode, cs);
        R.memo.pop_back();
    }
    std::string qp = P.qexpr ? std::string() : R.param(P.qacc.buffer), kp = R.param(P.kacc.buffer), vp = R.param(P.vacc.buffer);

    std::ostringstream src;
    src << kPrelude;
    src << "typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8;\n";
    src << "typedef short sanic_s16x4 __attribute__((ext_vector_type(4)));\n";
    src << "typedef short sanic_s16x8 __attribute__((ext_vector_type(8)));\n";
    src << "typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;\n";
    // tiling variants for the measured tuner: {3 workgroups per CU, 2 per CU, key range split
    // in two}. The split form gives every (head, query block) two workgroups, each folding half
    // of the block's key tiles; they exchange their (m, ℓ, o) partials through scratch and the
    // second to arrive combines them (the carrier's ExpShifted combine with its −∞ guard) and
    // projects. It evens out launches whose equal-sized blocks overfill the resident slots.
    int SPL = fvar == 2 ? 2 : 1;
    if (P.ragged) {
        // register every buffer the element-by-element fold reads before the argument struct is written
        Code scratch_code;
        emit_point_fold(R, scratch_code, st, "pf");
    }
    src << (SPL > 1 ? R.args_struct({"float* __restrict__ scratch", "unsigned* counters"}) : R.args_struct({}));
    src << kSplitBf16;
    src << "__device__ __forceinline__ idx_t sanic_min(idx_t a, idx_t b) { return a < b ? a : b; }\n";
    if (NP == 3)
        src << "__device__ __forceinline__ void split3_bf16(float x, float y, unsigned& hi, unsigned& mid, unsigned& lo) {\n"
               "  const unsigned h = pk_bf16(x, y);\n"
               "  hi = h;\n"
               "  split_bf16(x - __uint_as_float(h << 16), y - __uint_as_float(h & 0xFFFF0000u), mid, lo);\n}\n";
    // max across the 4 lane groups of a query column (lanes l, l^16, l^32, l^48): gfx950
    // permlane swaps, no LDS round trip
    // compiler-visible maxima: the compiler forms v_max3_f32 itself and, unlike for inline asm
    // (which it cannot see into), inserts the wait states a VALU read of a fresh MFMA result
    // needs; an asm max placed right after the MFMA read stale accumulator registers
    src << "__device__ __forceinline__ float hmax(float a, float b) {\n"
           "  return __builtin_fmaxf(a, b);\n}\n";
    src << "__device__ __forceinline__ float hmax3(float a, float b, float c) {\n"
           "  return __builtin_fmaxf(__builtin_fmaxf(a, b), c);\n}\n";
    src << "__device__ __forceinline__ float wave_max_x4(float v) {\n"
           "  auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);\n"
           "  v = hmax(__uint_as_float(r32[0]), __uint_as_float(r32[1]));\n"
           "  auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);\n"
           "  return hmax(__uint_as_float(r16[0]), __uint_as_float(r16[1]));\n}\n";
    src << "__device__ __forceinline__ float wave_sum_x4(float v) {\n"
           "  auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);\n"
           "  v = __uint_as_float(r32[0]) + __uint_as_float(r32[1]);\n"
           "  auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);\n"
           "  return __uint_as_float(r16[0]) + __uint_as_float(r16[1]);\n}\n";
    src << "__device__ __forceinline__ float score_part(const Args& a, float dotv, int hh, int qi, int kj) {\n"
        << entry_part << sp.str() << "  return " << vpart << ";\n}\n";
    src << "__device__ __forceinline__ float score_full(const Args& a, float dotv, int hh, int qi, int kj) {\n"
        << entry_full << sf.str() << "  return " << vfull << ";\n}\n";
    src << "__device__ __forceinline__ void window(const Args& a, idx_t hh, idx_t qrow, idx_t& lo, idx_t& hi) {\n"
        << Rw.entry() << wc.str() << "  lo = wlo; hi = whi;\n}\n";
    // the same bounds before an empty window is widened to the whole stream; true = non-empty
    bool raw_ok = true;
    {
        static const std::regex reset(R"(\n *if \(whi <= wlo\) \{ wlo = 0; whi = \d+; \})");
        const std::string raw = std::regex_replace(wc.str(), reset, "");
        // without the reset line removed, window_raw could not tell an empty window: edge
        // tiles then take the rendered leaf
        if (raw == wc.str() && wc.str().find("whi <= wlo") != std::string::npos) raw_ok = false;
        src << "__device__ __forceinline__ bool window_raw(const Args& a, idx_t hh, idx_t qrow, idx_t& lo, idx_t& hi) {\n"
            << Rw.entry() << raw << "  lo = wlo; hi = whi;\n  return whi > wlo;\n}\n";
    }
    src << "__device__ __forceinline__ void finish(const Args& a, const float* fs, idx_t hh, idx_t qi, idx_t ee) {\n"
        << Ro.entry() << fo.str() << "}\n";

    const std::string kname = "sanic_flash_h" + std::to_string(NH) + "_s" + std::to_string(NQ) + "_t" + std::to_string(T);
    Code k;
    k.indent = 1;
    // K and V tiles in a ring of three LDS buffers, filled straight from global memory
    // (global_load_lds, no register staging) two tiles ahead of the MFMAs. Rows are 128 bytes
    // unpadded with the 16-byte chunk index XORed by (row mod 8): a padded stride would put the
    // 16 rows of one fragment read into 2-way bank conflicts on gfx950, and the direct loads
    // write each wave's 1 KB contiguously, so the swizzle is applied to the source addresses.
    k.line("__shared__ __attribute__((aligned(16))) unsigned short kv_lds[" + std::to_string(KS * NBUF) + "][2][64 * 64];");
    // (the wave index through a scalar register: the LDS destinations of the direct loads and
    // the wave's row range are then scalar arithmetic)
    k.line("const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6)" + std::string(KS > 1 ? " & 3, kg = __builtin_amdgcn_readfirstlane(tid >> 8)" : "") + ";");
    k.line("const int l16 = lane & 15, lq = lane >> 4;");
    // XCD-aware block order: blockIdx mod 8 picks the KV head group, heaviest query blocks first
    const int64_t NKV = NH / P.rep;
    const int64_t NB = NH * NQB;
    if (SPL > 1) {
        k.line("const idx_t bid = blockIdx.x % " + std::to_string(NB) + ";");   // partners share an XCD
        k.line("const int part = (int)(blockIdx.x / " + std::to_string(NB) + ");");
    } else {
        k.line("const idx_t bid = blockIdx.x;");
    }
    if (NKV % 8 == 0 || NKV == 8) {
        k.line("const idx_t kvh = bid % " + std::to_string(NKV) + ", rest = bid / " + std::to_string(NKV) + ";");
        k.line("const idx_t hh = kvh * " + std::to_string(P.rep) + " + rest % " + std::to_string(P.rep) + ";");
        k.line("const idx_t qb = " + std::to_string(NQB - 1) + " - rest / " + std::to_string(P.rep) + ";");
    } else {
        k.line("const idx_t hh = bid % " + std::to_string(NH) + ";");
        k.line("const idx_t qb = " + std::to_string(NQB - 1) + " - bid / " + std::to_string(NH) + ";");
    }
    k.line("const idx_t q0 = qb * " + RBs + " + wv * " + std::to_string(16 * QT) + ";");   // this wave's query rows
    // block and wave key ranges from the honest window of the first and last rows
    k.line("idx_t blo_a, bhi_a, blo_b, bhi_b, wlo_a, whi_a, wlo_b, whi_b;");
    k.line("window(a, hh, qb * " + RBs + ", blo_a, bhi_a);");
    k.line("window(a, hh, " + row_clamp("qb * " + RBs + " + " + std::to_string(RB - 1)) + ", blo_b, bhi_b);");
    k.line("window(a, hh, " + row_clamp("q0") + ", wlo_a, whi_a);");
    k.line("window(a, hh, " + row_clamp("q0 + " + std::to_string(16 * QT - 1)) + ", wlo_b, whi_b);");
    if (SPL > 1) {
        k.line("const idx_t klo0 = (blo_a < blo_b ? blo_a : blo_b) / 64 * 64;");
        k.line("const idx_t khi0 = bhi_a > bhi_b ? bhi_a : bhi_b;");
        k.line("const idx_t ntl = khi0 > klo0 ? (khi0 - klo0 + 63) / 64 : 0;");
        k.line("const idx_t klo = klo0 + (part * ntl / 2) * 64;");
        k.line("const idx_t khi = part == 0 ? (klo0 + (ntl / 2) * 64 < khi0 ? klo0 + (ntl / 2) * 64 : khi0) : khi0;");
    } else {
        k.line("const idx_t klo = (blo_a < blo_b ? blo_a : blo_b) / 64 * 64;");
        k.line("const idx_t khi = bhi_a > bhi_b ? bhi_a : bhi_b;");
    }
    k.line("const idx_t wlo = wlo_a < wlo_b ? wlo_a : wlo_b, whi = whi_a > whi_b ? whi_a : whi_b;");
    k.line("const idx_t flo = wlo_a > wlo_b ? wlo_a : wlo_b;");
    // (a first or last row with no visible key stands for the whole stream and says nothing of
    // the rows between: no tile is then full)
    if (raw_ok) {
        k.line("idx_t re_lo, re_hi;");
        k.line("const bool wne = window_raw(a, hh, " + row_clamp("q0") + ", re_lo, re_hi) & window_raw(a, hh, " + row_clamp("q0 + " + std::to_string(16 * QT - 1)) + ", re_lo, re_hi);");
        k.line("const idx_t fhi = !wne ? 0 : whi_a < whi_b ? whi_a : whi_b;");
    } else {
        k.line("const idx_t fhi = whi_a < whi_b ? whi_a : whi_b;");
    }
    // the bounds are wave-uniform (they depend on the block and wave only): held in scalar
    // registers, the key loop's control and the tile classification run on the scalar unit
    k.line("const int klo_s = __builtin_amdgcn_readfirstlane((int)klo), khi_s = __builtin_amdgcn_readfirstlane((int)khi);");
    k.line("const int wlo_s = __builtin_amdgcn_readfirstlane((int)wlo), whi_s = __builtin_amdgcn_readfirstlane((int)whi);");
    k.line("const int flo_s = __builtin_amdgcn_readfirstlane((int)flo), fhi_s = __builtin_amdgcn_readfirstlane((int)fhi);");
    // Edge tiles, per element: inside a row's honest window the score is the unmasked form
    // (the full-tile identity); outside it −1e30 instead of the rendered mask (a finite mask
    // gives that same value for any score below ~1e22; a −∞ mask differs only while a row has
    // seen no visible key). Once a row has seen a visible key either weighs exactly 0, and what
    // a row accumulated before that is scaled by α = exp(−1e30 − m) = 0 on its first visible
    // tile, so the result is the same bit for bit — provided every row of the wave has a
    // non-empty window (else the rendered leaf per element). A finite value, not −∞, keeps
    // fully masked tiles at α = 1 (no rescale pass).
    // (the row bounds are recomputed on edge tiles only: kept live across the loop they cost
    // registers the window configuration spills)
    // (variant 3 takes the rendered leaf on every edge tile: the reference form the fast path
    // is tested against bit for bit)
    const bool edge_on = raw_ok && fvar != 3;
    // two values as the packed bf16 terms w[0] (+ w[1] (+ w[2])), component i
    auto split = [&](const std::string& x, const std::string& y, const std::string& w, const std::string& i) {
        if (NP == 1) return "  " + w + "[0][" + i + "] = pk_bf16(" + x + ", " + y + ");";
        if (NP == 2) return "  { unsigned h1, l1; split_bf16(" + x + ", " + y + ", h1, l1); " + w + "[0][" + i + "] = h1; " + w + "[1][" + i + "] = l1; }";
        return "  { unsigned h1, m1, l1; split3_bf16(" + x + ", " + y + ", h1, m1, l1); " + w + "[0][" + i + "] = h1; " + w + "[1][" + i + "] = m1; " + w + "[2][" + i + "] = l1; }";
    };
    // Q^T as the B operand (lane = query column l16 (+16·qt), d-slots lq·8 + 0..7 (+32·ds)),
    // held in registers for the whole key loop, loaded once from global memory
    k.line("bf16x8 qf[" + QTs + "][2];");
    const int NQT = P.qexpr ? NP : 1;                // bf16 terms of a query value
    for (int h = 1; h < NQT; h++) k.line("bf16x8 q" + std::to_string(h) + "[" + QTs + "][2];");
    for (int qt = 0; qt < QT; qt++)
        k.line("const idx_t qr" + std::to_string(qt) + " = " + row_clamp("q0 + " + std::to_string(qt * 16) + " + l16") + ";");
    if (!P.qexpr) {
        k.line("#pragma unroll");
        k.line("for (int qt = 0; qt < " + QTs + "; ++qt)");
        k.line("  #pragma unroll");
        k.line("  for (int ds = 0; ds < 2; ++ds)");
        k.line("    qf[qt][ds] = *(const bf16x8*)(" + qp + " + " + std::to_string(P.qacc.addr.c0) + " + " + hterm(qc, qh, qhc) +
               " + " + row_clamp("q0 + qt * 16 + l16") + " * " + std::to_string(qc[3]) + " + (ds * 4 + lq) * 8);");
    }
    // An expression query side is rendered element by element (the lane's 2 × 16 values), once
    // per workgroup, after the first K/V transfers are requested so its loads and arithmetic
    // overlap them; each value goes to the MFMA rounded to bf16 (RNE), the operand width.
    // The vectorised form's loads go out first, where the plain Q load would (loads complete in
    // issue order, so the rotation's operands are not queued behind the first K/V tiles), and
    // its arithmetic after the transfers are requested; the per-element form runs after them.
    Code q_lc, q_dc;
    bool q_runs = false;
    std::vector<std::string> q_vals[2][2];
    if (P.qexpr) {
        q_lc.indent = q_dc.indent = k.indent + 1;
        bool ok = true;
        for (int qt = 0; qt < QT && ok; qt++)
            for (int ds = 0; ds < 2 && ok; ds++) {
                const std::string sfx = "_q" + std::to_string(qt) + std::to_string(ds);
                const std::vector<std::string> vars = {"hh", "(idx_t)0", "((idx_t)lq * 8 + " + std::to_string(ds * 32) + ")",
                                                       "qr" + std::to_string(qt)};
                std::vector<int> bufs, dts;
                q_vals[qt][ds] = render_run(d, P.qnode, P.qcoords, {NH, T, HD, NQ}, vars, 2, q_lc, q_dc, sfx, bufs, dts, ok);
                for (size_t b = 0; b < bufs.size() && ok; b++)
                    k.line("const " + std::string(ctype_of(dts[b])) + "* __restrict__ rb" + std::to_string(b) + sfx + " = " + R.param(bufs[b]) + ";");
            }
        q_runs = ok;
        // the loads right away, as the plain Q load would be
        if (q_runs) k.s << q_lc.str();
    }
    auto emit_qexpr = [&]() {
        auto q_split = [&](int qt, int ds, const std::string* v) {
            k.line("{");
            k.line("  sanic_u32x4 w_[" + std::to_string(NP) + "];");
            for (int q = 0; q < 4; q++) k.line(split(v[2 * q], v[2 * q + 1], "w_", std::to_string(q)));
            const std::string ix = "[" + std::to_string(qt) + "][" + std::to_string(ds) + "]";
            for (int h = 0; h < NP; h++) k.line("  q" + (h ? std::to_string(h) : "f") + ix + " = __builtin_bit_cast(bf16x8, w_[" + std::to_string(h) + "]);");
            k.line("}");
        };
        if (q_runs) {
            k.s << q_dc.str();
            for (int qt = 0; qt < QT; qt++)
                for (int ds = 0; ds < 2; ds++) {
                    const auto& v = q_vals[qt][ds];
                    if (NQT > 1) { q_split(qt, ds, v.data()); continue; }
                    k.line("qf[" + std::to_string(qt) + "][" + std::to_string(ds) + "] = __builtin_bit_cast(bf16x8, (sanic_u32x4){pk_bf16(" + v[0] + ", " + v[1] +
                           "), pk_bf16(" + v[2] + ", " + v[3] + "), pk_bf16(" + v[4] + ", " + v[5] + "), pk_bf16(" + v[6] + ", " + v[7] + ")});");
                }
            return;
        }
        for (int qt = 0; qt < QT; qt++) {
            k.line("{");
            k.indent++;
            k.line("const idx_t qrow = qr" + std::to_string(qt) + ";");
            R.memo.emplace_back();
            std::string vals[2][8];
            for (int ds = 0; ds < 2; ds++)
                for (int j = 0; j < 8; j++) {
                    const std::string dd = "((idx_t)lq * 8 + " + std::to_string(ds * 32 + j) + ")";
                    std::vector<std::string> cs;
                    for (auto& sy : P.qcoords) cs.push_back(sy.render({"hh", "(idx_t)0", dd, "qrow"}));
                    vals[ds][j] = R.value(k, P.qnode, cs);
                }
            R.memo.pop_back();
            for (int ds = 0; ds < 2; ds++) {
                if (NQT > 1) { q_split(qt, ds, vals[ds]); continue; }
                std::string pk = "(sanic_u32x4){";
                for (int q = 0; q < 4; q++)
                    pk += std::string(q ? ", " : "") + "pk_bf16(" + vals[ds][2 * q] + ", " + vals[ds][2 * q + 1] + ")";
                k.line("qf[" + std::to_string(qt) + "][" + std::to_string(ds) + "] = __builtin_bit_cast(bf16x8, " + pk + "});");
            }
            k.indent--;
            k.line("}");
        }
    };
    k.line("f32x4 o[4][" + QTs + "];");
    k.line("#pragma unroll");
    k.line("for (int dt = 0; dt < 4; ++dt)");
    k.line("  #pragma unroll");
    k.line("  for (int qt = 0; qt < " + QTs + "; ++qt) o[dt][qt] = (f32x4){0, 0, 0, 0};");
    k.line("float m_run[" + QTs + "];");
    // row sums ℓ accumulate on the matrix cores: a row of ones times P^T (same bf16 P as O)
    k.line("f32x4 lsum[" + QTs + "];");
    k.line("#pragma unroll");
    k.line("for (int qt = 0; qt < " + QTs + "; ++qt) { m_run[qt] = -__builtin_huge_valf(); lsum[qt] = (f32x4){0, 0, 0, 0}; }");
    k.line("const bf16x8 ones = {0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80};");
    const double LOG2E = 1.4426950408889634;
    // Lazy reference max: the running max moves only when a tile's max exceeds it by more than
    // TAU (natural-log units, so every p stays below 2^8): the online softmax is exact for any
    // reference point, and rescaling O and ℓ becomes rare. Only when the projection does not
    // read the max slot itself.
    std::function<bool(int)> reads_f = [&](int e) -> bool {
        const sanic_expr& x = d->exprs[e];
        if (x.op == SANIC_EX_F) return x.index == P.max_slot;
        if (x.op >= SANIC_EX_CONST) return false;
        for (int ch : {x.a, x.b, x.c}) if (ch >= 0 && reads_f(ch)) return true;
        return false;
    };
    const bool lazy = !reads_f(c.project);
    const double TAU = 8.0 / LOG2E;
    // One tile (K: 64 keys × 64 d; V rows [key][e] or V^T rows [e][key] as they lie in memory)
    // into ring buffer b: wave w's transfer u fills LDS rows 8(w + 4u) .. +7, lane l landing on
    // row 8(w + 4u) + l/8, chunk l%8 — so it fetches global chunk (l%8) ^ (l/8) of that row.
    // Four transfers per lane per tile, counted by vmcnt like any global load.
    std::string kbase = std::to_string(P.kacc.addr.c0) + " + " + hterm(kc, kh, khc);
    std::string vbase = std::to_string(P.vacc.addr.c0) + " + " + hterm(vc, vh, vhc);
    const std::string krow = key_clamp("tt + r"), vsrc = v_rows ? krow + " * " + std::to_string(vc[1]) + " + c * 8"
                                                                 : "(idx_t)r * " + std::to_string(vc[2]) + " + tt + c * 8";
    // The direct transfer moves aligned 16-byte chunks; a caller may bind K or V at any element,
    // and the lengths that come here from the generic fold keep taking such a binding: its chunks
    // pass through registers, complete in LDS before the barrier that publishes the tile.
    if (P.ragged) k.line("const bool chunks = (((size_t)(" + kp + ") | (size_t)(" + vp + ")) & 15) == 0;");
    k.line("auto fetch = [&](idx_t tt, int b) {");
    k.line("  #pragma unroll");
    k.line("  for (int u = 0; u < 2; ++u) {");
    k.line("    const int r = 8 * (wv + 4 * u) + (lane >> 3), c = (lane & 7) ^ (lane >> 3);");
    if (P.ragged) {
        k.line("    if (!chunks) {");
        k.line("      const unsigned short* kq = " + kp + " + " + kbase + " + " + krow + " * " + std::to_string(kc[1]) + " + c * 8;");
        k.line("      const unsigned short* vq = " + vp + " + " + vbase + " + " + vsrc + ";");
        k.line("      for (int i = 0; i < 8; ++i) {");
        k.line("        kv_lds[b][0][(wv + 4 * u) * 512 + lane * 8 + i] = kq[i];");
        k.line("        kv_lds[b][1][(wv + 4 * u) * 512 + lane * 8 + i] = vq[i];");
        k.line("      }");
        k.line("      asm volatile(\"s_waitcnt lgkmcnt(0)\" ::: \"memory\");");
        k.line("      continue;");
        k.line("    }");
    }
    k.line("    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(" + kp + " + " + kbase + " + " + krow + " * " +
           std::to_string(kc[1]) + " + c * 8), (__attribute__((address_space(3))) void*)(&kv_lds[b][0][(wv + 4 * u) * 512]), 16, 0, 0);");
    k.line("    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(" + vp + " + " + vbase + " + " + vsrc +
           "), (__attribute__((address_space(3))) void*)(&kv_lds[b][1][(wv + 4 * u) * 512]), 16, 0, 0);");
    k.line("  }");
    k.line("};");
    k.line("if (klo_s < khi_s) {");
    k.indent++;
    if (KS > 1) {
        k.line("int buf = kg * " + std::to_string(NBUF) + ";");
        k.line("if (klo_s + 64 * kg < khi_s) fetch(klo_s + 64 * kg, buf);");
    } else {
        k.line("fetch(klo_s, 0);");
        k.line("if (klo_s + 64 < khi_s) fetch(klo_s + 64, 1);");
    }
    if (P.qexpr) emit_qexpr();
    if (KS > 1) {
        // every team runs every iteration (the barriers are the workgroup's); past its last tile it
        // neither fetches nor folds
        k.line("for (int tb = klo_s; tb < khi_s; tb += " + step + ") {");
        k.indent++;
        k.line("const int t0 = tb + 64 * kg;");
    } else {
        k.line("int buf = 0;");
        k.line("for (int t0 = klo_s; t0 < khi_s; t0 += 64) {");
        k.indent++;
    }
    // this tile's transfers have landed for every wave (only the next tile's four may still be
    // in flight; loads complete in issue order). The buffer the transfer below refills was read
    // in the previous iteration: this barrier orders every wave's reads of it before the refill,
    // so the refill must stay after the barrier. The asm carries the memory clobber that keeps
    // the compiler from moving LDS accesses across the barrier.
    if (KS > 1) {
        k.line("asm volatile(\"s_waitcnt vmcnt(0)\\n\\ts_barrier\" ::: \"memory\");");
        k.line("if (t0 + " + step + " < khi_s) fetch(t0 + " + step + ", buf ^ 1);");
    } else {
    k.line("if (t0 + 64 < khi_s) asm volatile(\"s_waitcnt vmcnt(4)\\n\\ts_barrier\" ::: \"memory\");");
    k.line("else asm volatile(\"s_waitcnt vmcnt(0)\\n\\ts_barrier\" ::: \"memory\");");
    k.line("if (t0 + 128 < khi_s) fetch(t0 + 128, buf == 0 ? 2 : buf - 1);");
    }
    // wave-uniform tile classification (scalar branches)
    k.line("const int live = t0 < whi_s && t0 + 64 > wlo_s;");   // some row sees it
    k.line("if (live) {");
    k.indent++;
    k.line("const int full = t0 >= flo_s && t0 + 64 <= fhi_s;");  // every row sees all
    // S^T tiles: kt (16 keys) × qt (16 queries), contraction over d in 2 steps of 32
    // both query tiles' scores first: each K fragment is read from LDS once for the two tiles
    // (measured: 2% over re-reading it per tile, the kernel being bound by LDS and MFMA issue).
    // The split variant and the rendered-mask reference variant keep one query tile's scores
    // live at a time (with both live they spill 12–13 registers); the products are the same
    // MFMAs in the same order either way.
    const bool s_both = QT == 2 && SPL == 1 && fvar != 3;
    k.line("f32x4 s[4][" + QTs + "];");
    k.line("sanic_u32x4 pw[" + QTs + "][2][" + std::to_string(NP) + "];");
    auto scores = [&](bool both) {
        k.line("#pragma unroll");
        k.line("for (int kt = 0; kt < 4; ++kt) {");
        k.line(both ? "  s[kt][0] = (f32x4){0, 0, 0, 0};" : "  s[kt][qt] = (f32x4){0, 0, 0, 0};");
        if (both) k.line("  s[kt][1] = (f32x4){0, 0, 0, 0};");
        k.line("  #pragma unroll");
        k.line("  for (int ds = 0; ds < 2; ++ds) {");
        k.line("    const bf16x8 ka = *(const bf16x8*)(&kv_lds[buf][0][(kt * 16 + l16) * 64 + (((ds * 4 + lq) ^ (l16 & 7)) * 8)]);");
        if (both) {
            k.line("    #pragma unroll");
            k.line("    for (int qt = 0; qt < 2; ++qt) {");
        } else {
            k.line("    {");
        }
        k.line("      s[kt][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, qf[qt][ds], s[kt][qt], 0, 0, 0);");
        for (int h = 1; h < NQT; h++) k.line("      s[kt][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, q" + std::to_string(h) + "[qt][ds], s[kt][qt], 0, 0, 0);");
        k.line("    }");
        k.line("  }");
        k.line("}");
    };
    if (s_both) scores(true);
    // online softmax per query column (lane-local; the max reduces across the 4 lane groups)
    k.line("#pragma unroll");
    k.line("for (int qt = 0; qt < " + QTs + "; ++qt) {");
    k.indent++;
    if (!s_both) scores(false);
    k.line("const int qi = (int)" + row_clamp("(q0 + qt * 16 + l16)") + ";");
    k.line("float sv[16];");
    k.line("float p[16];");
    k.line("float mn, alpha;");
    if (scale_known) {
        // full tiles: score = dot·c, so max and exp2 work on the raw dot (c > 0)
        k.line("if (full) {");
        k.indent++;
        // 16 → 1 in 8 three-input maxes
        k.line("const float ma = hmax3(s[0][qt][0], s[0][qt][1], s[0][qt][2]), mb_ = hmax3(s[0][qt][3], s[1][qt][0], s[1][qt][1]);");
        k.line("const float mc = hmax3(s[1][qt][2], s[1][qt][3], s[2][qt][0]), md = hmax3(s[2][qt][1], s[2][qt][2], s[2][qt][3]);");
        k.line("const float me = hmax3(s[3][qt][0], s[3][qt][1], s[3][qt][2]);");
        k.line("float mt = hmax3(hmax3(ma, mb_, mc), hmax3(md, me, s[3][qt][3]), ma);");
        // Common case: no lane's scores move its row's running max (every lane's own maximum
        // within the rescale threshold, the running max finite). Then mn = m_run and alpha = 1
        // exactly, as the general form below would find, without the cross-lane reduction,
        // the rescale factor's exp2 or the rescale.
        const std::string keep = lazy ? "m_run[qt] + " + flit(TAU) : std::string("m_run[qt]");
        k.line("if (__all(mt * " + flit(scale_c) + " <= " + keep + " && m_run[qt] > -1e29f)) {");
        k.line("  mn = m_run[qt];");
        k.line("  alpha = 1.0f;");
        k.line("  const float mb = mn * " + flit(LOG2E) + ";");
        k.line("  #pragma unroll");
        k.line("  for (int kt = 0; kt < 4; ++kt)");
        k.line("    #pragma unroll");
        k.line("    for (int r = 0; r < 4; ++r) p[kt * 4 + r] = __builtin_amdgcn_exp2f(fmaf(s[kt][qt][r], " + flit(scale_c * LOG2E) + ", -mb));");
        k.line("} else {");
        k.indent++;
        k.line("mt = wave_max_x4(mt) * " + flit(scale_c) + ";");
        k.line(lazy ? "mn = mt > m_run[qt] + " + flit(TAU) + " ? mt : m_run[qt];" : "mn = fmaxf(m_run[qt], mt);");
        k.line("alpha = m_run[qt] == -__builtin_huge_valf() ? 0.0f : __builtin_amdgcn_exp2f((m_run[qt] - mn) * " + flit(LOG2E) + ");");
        k.line("if (__all(mn > -1e29f)) {");
        k.line("  const float mb = mn * " + flit(LOG2E) + ";");
        k.line("  #pragma unroll");
        k.line("  for (int kt = 0; kt < 4; ++kt)");
        k.line("    #pragma unroll");
        k.line("    for (int r = 0; r < 4; ++r) p[kt * 4 + r] = __builtin_amdgcn_exp2f(fmaf(s[kt][qt][r], " + flit(scale_c * LOG2E) + ", -mb));");
        k.line("} else {");
        k.line("  #pragma unroll");
        k.line("  for (int kt = 0; kt < 4; ++kt)");
        k.line("    #pragma unroll");
        k.line("    for (int r = 0; r < 4; ++r) p[kt * 4 + r] = mn == -__builtin_huge_valf() ? 0.0f : __builtin_amdgcn_exp2f((s[kt][qt][r] * " + flit(scale_c) + " - mn) * " + flit(LOG2E) + ");");
        k.line("}");
        k.indent--;
        k.line("}");
        k.indent--;
        k.line("} else {");
        k.indent++;
    } else {
        k.line("{");
        k.indent++;
    }
    // partial tiles (and scores of any other shape): the rendered leaf per element
    // (full and edge_fast are wave-uniform: one branch per tile, not a select per element)
    // (the key indices are formed here, in the branch that uses them: the compiler would
    // otherwise hoist them ahead of the full-tile branch)
    k.line("int kb = t0 + lq * 4;");
    k.line("asm volatile(\"\" : \"+v\"(kb));");
    k.line("int elo = -1, ehi = 0x7fffffff;");
    if (edge_on) {
        k.line("if (!full) {");
        k.line("  idx_t rl, rh;");
        k.line("  const bool ok = window_raw(a, hh, qi, rl, rh);");
        k.line("  if (__all(ok)) { elo = (int)rl; ehi = (int)rh; } else { elo = 0x7fffffff; }");
        k.line("}");
    } else {
        k.line("if (!full) elo = 0x7fffffff;");
    }
    k.line("if (elo != 0x7fffffff) {");
    k.line("  #pragma unroll");
    k.line("  for (int kt = 0; kt < 4; ++kt)");
    k.line("    #pragma unroll");
    k.line("    for (int r = 0; r < 4; ++r) {");
    k.line("      const int kj = kb + kt * 16 + r;");
    k.line("      const float sf = score_full(a, s[kt][qt][r], (int)hh, qi, " + std::string(P.ragged ? "kj < " + std::to_string(T) + " ? kj : " + std::to_string(T - 1) : "kj") + ");");
    k.line("      sv[kt * 4 + r] = kj >= elo && kj < ehi ? sf : -1e30f;");
    k.line("    }");
    k.line("} else {");
    k.line("  #pragma unroll");
    k.line("  for (int kt = 0; kt < 4; ++kt)");
    k.line("    #pragma unroll");
    if (P.ragged) {
        // keys past the last weigh nothing
        k.line("    for (int r = 0; r < 4; ++r) {");
        k.line("      const int kj = kb + kt * 16 + r;");
        k.line("      const float sp = score_part(a, s[kt][qt][r], (int)hh, qi, kj < " + std::to_string(T) + " ? kj : " + std::to_string(T - 1) + ");");
        k.line("      sv[kt * 4 + r] = kj < " + std::to_string(T) + " ? sp : -__builtin_huge_valf();");
        k.line("    }");
    } else {
        k.line("    for (int r = 0; r < 4; ++r) sv[kt * 4 + r] = score_part(a, s[kt][qt][r], (int)hh, qi, kb + kt * 16 + r);");
    }
    k.line("}");
    k.line("float mt = fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]));");
    k.line("#pragma unroll");
    k.line("for (int i = 4; i < 16; i += 2) mt = fmaxf(mt, fmaxf(sv[i], sv[i + 1]));");
    k.line("mt = wave_max_x4(mt);");
    k.line(lazy ? "mn = mt > m_run[qt] + " + flit(TAU) + " ? mt : m_run[qt];" : "mn = fmaxf(m_run[qt], mt);");
    // the carrier's guarded rescale: a side whose max is −∞ weighs 0
    k.line("alpha = m_run[qt] == -__builtin_huge_valf() ? 0.0f : __builtin_amdgcn_exp2f((m_run[qt] - mn) * " + flit(LOG2E) + ");");
    // Fast form exp2(s·log2e − m·log2e) (one FMA) while every row of the wave has a moderate
    // max; when some row's max is a masked score (≈ −1e30) or −∞ the fused form does not
    // cancel exactly, so (s − m)·log2e is used for that tile.
    k.line("if (__all(mn > -1e29f)) {");
    k.line("  const float mb = mn * " + flit(LOG2E) + ";");
    k.line("  #pragma unroll");
    k.line("  for (int i = 0; i < 16; ++i) p[i] = __builtin_amdgcn_exp2f(fmaf(sv[i], " + flit(LOG2E) + ", -mb));");
    k.line("} else {");
    k.line("  #pragma unroll");
    k.line("  for (int i = 0; i < 16; ++i) p[i] = mn == -__builtin_huge_valf() ? 0.0f : __builtin_amdgcn_exp2f((sv[i] - mn) * " + flit(LOG2E) + ");");
    k.line("}");
    k.indent--;
    k.line("}");
    k.line("m_run[qt] = mn;");
    k.line("if (!__all(alpha == 1.0f)) {");   // the running max moved for some row: rescale
    k.line("  #pragma unroll");
    k.line("  for (int dt = 0; dt < 4; ++dt) { o[dt][qt][0] *= alpha; o[dt][qt][1] *= alpha; o[dt][qt][2] *= alpha; o[dt][qt][3] *= alpha; }");
    k.line("  lsum[qt] *= alpha;");
    k.line("}");
    // P^T as the B operand for key step ks: slots 0..3 = keys 32ks + lq·4 + r (tile 2ks),
    // slots 4..7 = keys 32ks + 16 + lq·4 + r (tile 2ks+1); two slots per dword, RNE in hardware
    k.line("#pragma unroll");
    k.line("for (int ks = 0; ks < 2; ++ks) {");
    for (int q = 0; q < 4; q++) k.line(split("p[8 * ks + " + std::to_string(2 * q) + "]", "p[8 * ks + " + std::to_string(2 * q + 1) + "]", "pw[qt][ks]", std::to_string(q)));
    k.line("}");
    k.indent--;
    k.line("}");
    auto weight = [&](const std::string& qt, const std::string& ks, int h) {
        return "__builtin_bit_cast(bf16x8, pw[" + qt + "][" + ks + "][" + std::to_string(h) + "])";
    };
    // O^T += V^T · P^T ; V^T A operand: row e = dt·16 + l16, keys in the same slot order
    k.line("#pragma unroll");
    k.line("for (int ks = 0; ks < 2; ++ks) {");
    for (int qt = 0; qt < QT; qt++)
        for (int h = 0; h < NP; h++) {
            const std::string q = std::to_string(qt);
            k.line("  lsum[" + q + "] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, " + weight(q, "ks", h) + ", lsum[" + q + "], 0, 0, 0);");
        }
    k.line("}");
    if (v_rows) {
        // V rows in LDS, read transposed (ds_read_b64_tr_b16): in each 16-lane group, source
        // lane s reads 4 values of e at key row (base + s/4), e = dt·16 + 4·(s%4); lane i then
        // holds keys base + 0..3 of e = dt·16 + i — slots 0..3, and base + 16 gives slots 4..7
        // (row + 16 has the same swizzle as row). The reads are issued from inline asm, two
        // value tiles (8 reads) at a time, each group completed by an explicit lgkmcnt wait
        // that the fragments pass through: the compiler's own form of this read waits for
        // every outstanding direct-to-LDS transfer first (vmcnt(0), i.e. the next tile's
        // prefetch), which the loop-top barrier already orders for this buffer.
        k.line("sanic_s16x4 vt[4][2][2];");
        auto vreads = [&](int dt0) {
            for (int dt = dt0; dt < dt0 + 2; dt++)
                for (int ks = 0; ks < 2; ks++) {
                    const std::string ix = "[" + std::to_string(dt) + "][" + std::to_string(ks) + "]";
                    k.line("{");
                    k.line("  const int vrow = " + std::to_string(ks * 32) + " + lq * 4 + (l16 >> 2), vcol = " + std::to_string(dt * 16) + " + (l16 & 3) * 4;");
                    k.line("  const unsigned va_ = (unsigned)(size_t)((__attribute__((address_space(3))) const unsigned short*)&kv_lds[buf][1][vrow * 64 + (((vcol >> 3) ^ (vrow & 7)) << 3) + (vcol & 7)]);");
                    k.line("  asm volatile(\"ds_read_b64_tr_b16 %0, %1\" : \"=v\"(vt" + ix + "[0]) : \"v\"(va_));");
                    k.line("  asm volatile(\"ds_read_b64_tr_b16 %0, %1 offset:2048\" : \"=v\"(vt" + ix + "[1]) : \"v\"(va_));");
                    k.line("}");
                }
        };
        auto vwait = [&](int dt0) {
            std::string ops;
            for (int dt = dt0; dt < dt0 + 2; dt++)
                for (int ks = 0; ks < 2; ks++)
                    for (int h = 0; h < 2; h++)
                        ops += std::string(ops.empty() ? "" : ", ") + "\"+v\"(vt[" + std::to_string(dt) + "][" + std::to_string(ks) + "][" + std::to_string(h) + "])";
            k.line("asm volatile(\"s_waitcnt lgkmcnt(0)\" : " + ops + ");");
        };
        auto vmfma = [&](int dt0) {
            for (int dt = dt0; dt < dt0 + 2; dt++)
                for (int ks = 0; ks < 2; ks++) {
                    const std::string ix = "[" + std::to_string(dt) + "][" + std::to_string(ks) + "]";
                    const std::string va = "__builtin_bit_cast(bf16x8, (sanic_s16x8)__builtin_shufflevector(vt" + ix + "[0], vt" + ix + "[1], 0, 1, 2, 3, 4, 5, 6, 7))";
                    for (int qt = 0; qt < QT; qt++)
                        for (int h = 0; h < NP; h++) {
                            const std::string ov = "o[" + std::to_string(dt) + "][" + std::to_string(qt) + "]";
                            k.line(ov + " = __builtin_amdgcn_mfma_f32_16x16x32_bf16(" + va + ", " + weight(std::to_string(qt), std::to_string(ks), h) + ", " + ov + ", 0, 0, 0);");
                        }
                }
        };
        vreads(0);
        vwait(0);
        vreads(2);
        vmfma(0);
        vwait(2);
        vmfma(2);
    }
    if (!v_rows) {
    k.line("#pragma unroll");
    k.line("for (int dt = 0; dt < 4; ++dt)");
    k.line("  #pragma unroll");
    k.line("  for (int ks = 0; ks < 2; ++ks) {");
    {
        k.line("    const int vrow = dt * 16 + l16, vcol = ks * 32 + lq * 4;");
        k.line("    const unsigned short* vr = &kv_lds[buf][1][vrow * 64 + (((vcol >> 3) ^ (vrow & 7)) << 3) + (vcol & 7)];");
        k.line("    const unsigned short* vr2 = &kv_lds[buf][1][vrow * 64 + ((((vcol + 16) >> 3) ^ (vrow & 7)) << 3) + (vcol & 7)];");
        k.line("    const uint2 lo4 = *(const uint2*)(vr), hi4 = *(const uint2*)(vr2);");
        k.line("    const bf16x8 va = __builtin_bit_cast(bf16x8, (sanic_u32x4){lo4.x, lo4.y, hi4.x, hi4.y});");
    }
    for (int qt = 0; qt < QT; qt++) {
        const std::string q = std::to_string(qt);
        k.line("    o[dt][" + q + "] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, " + weight(q, "ks", 0) + ", o[dt][" + q + "], 0, 0, 0);");
    }
    k.line("  }");
    }
    k.indent--;
    k.line("}");
    k.line(KS > 1 ? "buf ^= 1;" : "buf = buf == 2 ? 0 : buf + 1;");
    k.indent--;
    k.line("}");
    k.indent--;
    k.line("}");
    if (KS > 1) {
        // the teams' carriers meet in LDS (over the tile rings, once every wave is done with them):
        // the first team's waves take the others' in order, by the ExpShifted combine with its −∞ guard
        const std::string slots = std::to_string(18 * QT * 64);
        k.line("__syncthreads();");
        k.line("float* mg = (float*)kv_lds + lane;");
        k.line("if (kg > 0) {");
        k.line("  float* to = mg + ((kg - 1) * 4 + wv) * " + slots + ";");
        k.line("  #pragma unroll");
        k.line("  for (int qt = 0; qt < " + QTs + "; ++qt) {");
        k.line("    #pragma unroll");
        k.line("    for (int i = 0; i < 16; ++i) to[(qt * 18 + i) * 64] = o[i / 4][qt][i % 4];");
        k.line("    to[(qt * 18 + 16) * 64] = m_run[qt];");
        k.line("    to[(qt * 18 + 17) * 64] = lsum[qt][0];");
        k.line("  }");
        k.line("}");
        k.line("__syncthreads();");
        k.line("if (kg > 0) return;");
        k.line("#pragma unroll");
        k.line("for (int g = 0; g < " + std::to_string(KS - 1) + "; ++g) {");
        k.line("  const float* from = mg + (g * 4 + wv) * " + slots + ";");
        k.line("  #pragma unroll");
        k.line("  for (int qt = 0; qt < " + QTs + "; ++qt) {");
        k.line("    const float mo = from[(qt * 18 + 16) * 64], M = __builtin_fmaxf(m_run[qt], mo);");
        k.line("    const float ws = m_run[qt] == -__builtin_huge_valf() ? 0.0f : __builtin_amdgcn_exp2f((m_run[qt] - M) * " + flit(LOG2E) + ");");
        k.line("    const float wo = mo == -__builtin_huge_valf() ? 0.0f : __builtin_amdgcn_exp2f((mo - M) * " + flit(LOG2E) + ");");
        k.line("    lsum[qt][0] = __builtin_fmaf(lsum[qt][0], ws, from[(qt * 18 + 17) * 64] * wo);");
        k.line("    m_run[qt] = M;");
        k.line("    #pragma unroll");
        k.line("    for (int i = 0; i < 16; ++i) o[i / 4][qt][i % 4] = __builtin_fmaf(o[i / 4][qt][i % 4], ws, from[(qt * 18 + i) * 64] * wo);");
        k.line("  }");
        k.line("}");
    }
    int64_t soff = -1;
    if (SPL > 1) {
        // partials [block][part][36][256 lanes] (o in accumulator order, m, ℓ), and one arrival
        // counter per block, re-armed by the combining workgroup
        soff = scratch;
        const int64_t pbytes = NB * 2 * 36 * 256 * 4;
        scratch += pbytes;
        k.line("{");
        k.indent++;
        k.line("float* pw = a.scratch + ((idx_t)bid * 2 + part) * 9216 + tid;");
        k.line("#pragma unroll");
        k.line("for (int dt = 0; dt < 4; ++dt)");
        k.line("  #pragma unroll");
        k.line("  for (int qt = 0; qt < 2; ++qt)");
        k.line("    #pragma unroll");
        k.line("    for (int r = 0; r < 4; ++r) sanic_st(pw + ((dt * 2 + qt) * 4 + r) * 256, o[dt][qt][r]);");
        k.line("for (int qt = 0; qt < 2; ++qt) { sanic_st(pw + (32 + qt) * 256, m_run[qt]); sanic_st(pw + (34 + qt) * 256, lsum[qt][0]); }");
        k.line("unsigned* cnt = a.counters + bid;");
        emit_arrival(k, "sp_last", "tid", "cnt", "2u");
        k.line("if (!sp_last) return;");
        k.line("if (tid == 0) sanic_st(cnt, 0u);");
        // the combine always takes part 0's values as the left operand of one explicit fma
        // (a·wa + b·wb with the product b·wb rounded first), so the rounding does not depend on
        // which half arrived last
        k.line("const float* pr = a.scratch + ((idx_t)bid * 2 + (1 - part)) * 9216 + tid;");
        k.line("#pragma unroll");
        k.line("for (int qt = 0; qt < 2; ++qt) {");
        k.line("  const float mo = sanic_ld(pr + (32 + qt) * 256), lo = sanic_ld(pr + (34 + qt) * 256);");
        k.line("  const float M = __builtin_fmaxf(m_run[qt], mo);");
        k.line("  const float ws = m_run[qt] == -__builtin_huge_valf() ? 0.0f : __builtin_amdgcn_exp2f((m_run[qt] - M) * " + flit(LOG2E) + ");");
        k.line("  const float wo = mo == -__builtin_huge_valf() ? 0.0f : __builtin_amdgcn_exp2f((mo - M) * " + flit(LOG2E) + ");");
        k.line("  const bool p0 = part == 0;");
        k.line("  lsum[qt][0] = p0 ? __builtin_fmaf(lsum[qt][0], ws, lo * wo) : __builtin_fmaf(lo, wo, lsum[qt][0] * ws);");
        k.line("  m_run[qt] = M;");
        k.line("  #pragma unroll");
        k.line("  for (int dt = 0; dt < 4; ++dt)");
        k.line("    #pragma unroll");
        k.line("    for (int r = 0; r < 4; ++r) {");
        k.line("      const float ov = sanic_ld(pr + ((dt * 2 + qt) * 4 + r) * 256);");
        k.line("      o[dt][qt][r] = p0 ? __builtin_fmaf(o[dt][qt][r], ws, ov * wo) : __builtin_fmaf(ov, wo, o[dt][qt][r] * ws);");
        k.line("    }");
        k.line("}");
        k.indent--;
        k.line("}");
    }
    // finish: the row sum across the 4 lane groups, then project per output point. A point is stored once
    // where the epilogue reads a buffer, since the output may be bound to that buffer (the branch
    // ahead of the stores takes 0.2 µs of 18 at S = 1000, window 256).
    std::set<int> epilogue_reads;
    if (st.epilogue >= 0) collect_inputs(d, st.epilogue, epilogue_reads);
    const bool once = P.ragged && !epilogue_reads.empty();
    k.line("#pragma unroll");
    k.line("for (int qt = 0; qt < " + QTs + "; ++qt) {");
    k.indent++;
    k.line("const float lt = lsum[qt][0];");
    k.line("const idx_t qi = q0 + qt * 16 + l16;");
    if (P.ragged) {
        k.line("if (qi >= " + std::to_string(NQ) + ") continue;");
        k.line("bool odd = !(__builtin_fabsf(lt) <= 3.402823466e38f);");
        if (once) {
            k.line("#pragma unroll");
            k.line("for (int p = 0; p < 16; ++p) odd |= !(__builtin_fabsf(o[p / 4][qt][p % 4]) <= 3.402823466e38f);");
            k.line("if (!odd) {");
        }
    }
    k.line("#pragma unroll");
    k.line("for (int dt = 0; dt < 4; ++dt)");
    k.line("  #pragma unroll");
    k.line("  for (int r = 0; r < 4; ++r) {");
    k.line("    float fs[" + std::to_string(c.slots) + "];");
    k.line("    fs[" + std::to_string(P.max_slot) + "] = m_run[qt];");
    for (size_t s = 0; s < P.scalar_slots.size(); s++)
        k.line("    fs[" + std::to_string(P.scalar_slots[s]) + "] = " + flit(P.scalar_into[s]) + " * lt;");
    k.line("    fs[" + std::to_string(P.vec_slots[0]) + "] = o[dt][qt][r];");
    if (P.ragged && !once) k.line("    odd |= !(__builtin_fabsf(o[dt][qt][r]) <= 3.402823466e38f);");
    k.line("    finish(a, fs, hh, qi, dt * 16 + lq * 4 + r);");
    k.line("  }");
    if (P.ragged) {
        // Infinities and NaNs: a masked key of the same tile weighs 0 here, and 0 · ∞ is not what the
        // fold over the honest window gives; a lane with such a sum folds its points again
        k.line(once ? "} else {" : "if (odd) {");
        k.line("  #pragma nounroll");
        k.line("  for (int p = 0; p < 16; ++p) {");
        k.indent += 2;
        std::vector<std::string> gc(st.rank, "0");
        if (P.hdim >= 0) gc[P.hdim] = "hh";
        gc[P.qdim] = "qi";
        gc[P.edim] = "(p / 4 * 16 + lq * 4 + p % 4)";
        for (int j = 0; j < st.rank; j++) k.line("const idx_t g" + std::to_string(j) + " = " + gc[j] + ";");
        emit_point_fold(R, k, st, "pf");
        std::string arr;
        for (int sl2 = 0; sl2 < c.slots; sl2++) arr += (sl2 ? ", pf" : "pf") + std::to_string(sl2);
        k.line("const float fs[" + std::to_string(c.slots) + "] = {" + arr + "};");
        k.line("finish(a, fs, hh, qi, " + gc[P.edim] + ");");
        k.indent -= 2;
        k.line("  }");
        k.line("}");
    }
    k.indent--;
    k.line("}");

    // three waves per SIMD: the softmax of one wave overlaps the MFMAs of the others (the
    // register cap costs a few spilled values outside the inner loop)
    // tiling variants for the measured tuner: workgroups per CU {3, 2}
    int occ = fvar == 1 ? 2 : 3;
    if (KS > 1) occ = 4;
    src << "extern \"C\" __global__ void __launch_bounds__(" << 256 * KS << ", " << occ << ") " << kname << "(Args a) {\n" << R.entry() << k.str() << "}\n";
    out.kernel_kind = "skeleton:flash_prefill[rep " + std::to_string(P.rep) + (P.ragged ? ",any length" : "") + "]" + (SPL > 1 ? "+split2" : "") + (KS > 1 ? "+teams" + KSs : "");
    out.source = src.str();
    out.variants = P.ragged ? 1 : 4;
    std::vector<Arg> args = R.arg_list();
    if (SPL > 1) {
        args.push_back({Arg::SCRATCH, soff});
        args.push_back({Arg::COUNTERS, take_counters(NB)});
    }
    out.launches.push_back({kname, "", dim3((unsigned)(NB * SPL)), dim3((unsigned)(256 * KS)), 0, args});
    return true;
}

// ───────────────────────── float32 attention ───────────────────────────────────────────────
// The same carrier with operands that bf16 MFMAs do not hold: f32 Q, K or V (bf16 ones beside
// them widen on load), head sizes a multiple of 16, any lengths, f32 MFMAs (16x16x4) and expf
// throughout, so nothing is narrower than the generic fold's arithmetic.
//
// One workgroup = one head × 16 query rows; its 8 waves take every 8th tile of 16 keys, each with
// a running (m, ℓ, o) of its own, and merge in LDS by the carrier's combine in wave order. Sᵀ =
// K·Qᵀ, so a lane owns one query column and its P values are the next MFMA's B operand as they
// stand; K and V rows come straight from global memory (whole rows per 16 lanes), one tile ahead.
// The bound is the f32 MFMA rate and the softmax arithmetic of a row block's CU, so where the row
// blocks leave CUs idle up to 8 workgroups share one, a run of its key tiles each, and the last to
// arrive merges their partials in order. S = 1024, d = 64, causal: 1099 µs in the generic fold,
// which forms q·k for each of the 64 value columns; 18.6 with one workgroup per row block, 10.6
// with 4 (256 in all; 11.8 with 512, 13.1 with 128).
bool lower_flash_f32(const sanic_program_desc* d, int si, int64_t& scratch, LoweredStage& out) {
    FlashPlan P;
    if (!attention_plan(d, si, P)) return false;
    const sanic_stage& st = d->stages[si];
    const sanic_carrier& c = st.carrier;
    if (!sched_is_auto(st.sched) || P.qexpr) return false;
    auto wide = [](int dt) { return dt == SANIC_F32 || dt == SANIC_BF16; };
    if (!wide(P.qacc.dtype) || !wide(P.kacc.dtype) || !wide(P.vacc.dtype)) return false;
    const int64_t NH = P.NH, NQ = P.NQ, T = P.T, E = P.E, HD = P.HD;
    if (HD % 16 || E % 16 || HD > 128 || E > 128 || (E / 16 & (E / 16 - 1))) return false;
    // (no measured line: S = 128 takes 22.3 µs at d = 64 and 8.1 at d = 32 in the fold, 7.1 and 4.9 here.
    // The lowering of a 128 × 128 program is the fold with its own choice of schedule, and its test
    // states that)
    if (NH * NQ * T <= kFoldScores) return false;
    std::vector<int64_t> qc, kc, vc;
    int qh, kh, vh;
    int64_t qhc, khc, vhc;
    if (!split_addr(P.qacc.addr, 4, qc, qh, qhc) || !split_addr(P.kacc.addr, 4, kc, kh, khc) || !split_addr(P.vacc.addr, 3, vc, vh, vhc)) return false;
    if (qc[2] != 1 || qc[1] != 0 || kc[2] != 1 || kc[3] != 0 || vc[2] != 1) return false;
    const int ET = (int)(E / 16), DS = (int)(HD / 4);      // value tiles; contraction steps
    const int NWV = 8;
    auto S = [](int64_t v) { return std::to_string(v); };

    Renderer R(d), Rs(d), Ro(d), Rw(d);     // the kernel, and its score, store and window functions
    auto win = honest_window(d, st);
    const sanic_node& sl = d->nodes[st.leaf[P.sleaf]];
    std::vector<std::string> lc(sl.rank);
    for (int j = 0; j < sl.rank; j++) {
        int b = st.bind[P.sleaf][j];
        lc[j] = b == SANIC_BIND_STREAM ? "kj" : b == P.hdim && b >= 0 ? "hh" : b == P.qdim ? "qi" : "0";
    }
    Code sp, wc, fo, k;
    sp.indent = wc.indent = fo.indent = k.indent = 1;
    Rs.subst[P.dot_reduce] = "dotv";
    const std::string vpart = Rs.value(sp, st.leaf[P.sleaf], lc);
    Rw.take_buffers(Rs);
    for (int j = 0; j < st.rank; j++) wc.line("const idx_t g" + S(j) + " = " + (j == P.hdim ? "hh" : j == P.qdim ? "qrow" : "0") + ";");
    emit_window(Rw, wc, st, win, "wlo", "whi");
    Ro.take_buffers(Rw);
    std::vector<std::string> gc(st.rank, "0");
    if (P.hdim >= 0) gc[P.hdim] = "hh";
    gc[P.qdim] = "qi";
    gc[P.edim] = "ee";
    {
        const std::string f = Ro.expr(fo, c.project, "", "", "", "fs");
        fo.line("const float fold_v = " + f + ";");
        std::string v = "fold_v";
        if (st.epilogue >= 0) {
            Ro.fold_var = "fold_v";
            v = Ro.value(fo, st.epilogue, gc);
        }
        std::string lin;
        for (int j = 0; j < st.rank; j++)
            lin = j == 0 ? "(idx_t)(" + gc[0] + ")" : "(" + lin + " * " + S(st.grid[j]) + " + (idx_t)(" + gc[j] + "))";
        fo.line(store_stmt(Ro.param(st.out_buffer), lin, st.out_dtype, v, false, d->buffers[st.out_buffer].scale));
    }
    R.take_buffers(Ro);
    auto base = [&](const Access& acc, const std::vector<int64_t>& cf, int div, int64_t hcf) {
        const std::string h = div ? "(hh / " + S(div) + ") * " + S(hcf) : "hh * " + S(cf[0]);
        return R.param(acc.buffer) + " + " + S(acc.addr.c0) + " + " + h;
    };
    // n consecutive elements at p as floats into x[0..n)
    auto load = [&](const Access& acc, const std::string& p, int n, const std::string& x) {
        if (acc.dtype == SANIC_F32) {
            const int w = n % 4 == 0 ? 4 : n;      // 1, 2 or runs of 4
            for (int i = 0; i < n; i += w) {
                if (w == 1) { k.line(x + "[" + S(i) + "] = (" + p + ")[" + S(i) + "];"); continue; }
                k.line("{ const sanic_f32x" + S(w) + "_any t_ = *(const sanic_f32x" + S(w) + "_any*)(" + p + " + " + S(i) + ");");
                for (int j = 0; j < w; j++) k.line("  " + x + "[" + S(i + j) + "] = t_[" + S(j) + "];");
                k.line("}");
            }
        } else {
            for (int i = 0; i < n; i++) k.line(x + "[" + S(i) + "] = sanic_bf16((" + p + ")[" + S(i) + "]);");
        }
    };
    const int64_t NQB = (NQ + 15) / 16, NB = NH * NQB, NBP = (NB + 7) / 8 * 8;
    const int SPL = lean_scratch() ? 1 : (int)std::max<int64_t>(1, std::min<int64_t>({8, 256 / NB, (T + 127) / 128}));
    // the workgroups of a row block are NBP apart, a multiple of 8: on one XCD
    const bool xl = SPL > 1 && xcd_local_enabled();
    const std::string stx = xl ? "sanic_stx" : "sanic_st", ldx = xl ? "sanic_ldx" : "sanic_ld";
    const int64_t PSZ = 16 * E + 32;                  // floats of a partial: o, m, ℓ
    const int64_t soff = scratch;
    if (SPL > 1) scratch += (NB * SPL * PSZ * 4 + 255) / 256 * 256;
    k.line("__shared__ float o_lds[" + S(NWV) + "][" + S(E) + "][17], m_lds[" + S(NWV) + "][16], l_lds[" + S(NWV) + "][16];");
    k.line("const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);");
    k.line("const int l16 = lane & 15, lq = lane >> 4;");
    // the longest (last) row blocks first
    k.line("const int bid = blockIdx.x % " + S(SPL > 1 ? NBP : NB) + ", part = blockIdx.x / " + S(SPL > 1 ? NBP : NB) + ";");
    if (SPL > 1 && NBP != NB) k.line("if (bid >= " + S(NB) + ") return;");
    k.line("const idx_t hh = bid % " + S(NH) + ", q0 = (" + S(NQB - 1) + " - bid / " + S(NH) + ") * 16;");
    k.line("const idx_t qlast = q0 + 15 < " + S(NQ) + " ? q0 + 15 : (idx_t)" + S(NQ - 1) + ";");
    k.line("idx_t alo, ahi, blo, bhi;");
    k.line("window(a, hh, q0, alo, ahi);");
    k.line("window(a, hh, qlast, blo, bhi);");
    k.line("int klo = __builtin_amdgcn_readfirstlane((int)(alo < blo ? alo : blo)) / 16 * 16, khi = __builtin_amdgcn_readfirstlane((int)(ahi > bhi ? ahi : bhi));");
    if (SPL > 1) {
        // as many of them as have a tile for each wave
        k.line("const int nt = (khi - klo + 15) / 16, nsp = nt <= 8 ? 1 : nt >= " + S(8 * SPL) + " ? " + S(SPL) + " : (nt + 7) / 8;");
        k.line("if (part >= nsp) return;");
        k.line("const int per = (nt + nsp - 1) / nsp * 16;");
        k.line("klo += part * per;");
        k.line("khi = klo + per < khi ? klo + per : khi;");
    }
    k.line("const int qi = (int)(q0 + l16 < qlast ? q0 + l16 : qlast);");
    // step s contracts d = lq·DS + s: a lane's operands of all steps are one contiguous run
    k.line("float qv[" + S(DS) + "];");
    load(P.qacc, "(" + base(P.qacc, qc, qh, qhc) + " + (idx_t)qi * " + S(qc[3]) + " + lq * " + S(DS) + ")", DS, "qv");
    k.line("f32x4 o[" + S(ET) + "];");
    for (int e = 0; e < ET; e++) k.line("o[" + S(e) + "] = (f32x4){0, 0, 0, 0};");
    k.line("float m = -__builtin_huge_valf(), l = 0.0f;");
    // K row of key t0 + l16 (run lq); V rows of keys t0 + lq·4 + r, values l16·ET .. + ET
    k.line("auto fetch = [&](int t0, float (&kv)[" + S(DS) + "], float (&vv)[4][" + S(ET) + "]) {");
    k.indent++;
    k.line("const idx_t kt = t0 + l16 < " + S(T) + " ? t0 + l16 : " + S(T - 1) + ";");
    load(P.kacc, "(" + base(P.kacc, kc, kh, khc) + " + kt * " + S(kc[1]) + " + lq * " + S(DS) + ")", DS, "kv");
    for (int r = 0; r < 4; r++) {
        k.line("const idx_t vt" + S(r) + " = t0 + lq * 4 + " + S(r) + " < " + S(T) + " ? t0 + lq * 4 + " + S(r) + " : " + S(T - 1) + ";");
        load(P.vacc, "(" + base(P.vacc, vc, vh, vhc) + " + vt" + S(r) + " * " + S(vc[1]) + " + l16 * " + S(ET) + ")", ET, "vv[" + S(r) + "]");
    }
    k.indent--;
    k.line("};");
    k.line("auto fold = [&](int t0, float (&kv)[" + S(DS) + "], float (&vv)[4][" + S(ET) + "]) {");
    k.indent++;
    k.line("f32x4 s0 = (f32x4){0, 0, 0, 0}, s1 = (f32x4){0, 0, 0, 0};");
    for (int s = 0; s < DS; s++)
        k.line(std::string(s % 2 ? "s1" : "s0") + " = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[" + S(s) + "], qv[" + S(s) + "], " + (s % 2 ? "s1" : "s0") + ", 0, 0, 0);");
    k.line("float sv[4], p[4];");
    k.line("#pragma unroll");
    k.line("for (int r = 0; r < 4; ++r) {");
    k.line("  const int kj = t0 + lq * 4 + r;");
    k.line("  const float x = score(a, s0[r] + s1[r], (int)hh, qi, kj < " + S(T) + " ? kj : " + S(T - 1) + ");");
    k.line("  sv[r] = kj < " + S(T) + " ? x : -__builtin_huge_valf();");
    k.line("}");
    k.line("const float mt = sanic_rows_max(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3])));");
    k.line("const float mn = fmaxf(m, mt);");
    // the carrier's guarded rescale: a side whose max is −∞ weighs 0
    k.line("const float alpha = m == -__builtin_huge_valf() ? 0.0f : expf(m - mn);");
    k.line("#pragma unroll");
    k.line("for (int r = 0; r < 4; ++r) p[r] = sv[r] == -__builtin_huge_valf() ? 0.0f : expf(sv[r] - mn);");
    k.line("m = mn;");
    k.line("l = l * alpha + ((p[0] + p[1]) + (p[2] + p[3]));");
    for (int e = 0; e < ET; e++) k.line("o[" + S(e) + "] *= alpha;");
    for (int r = 0; r < 4; r++)
        for (int e = 0; e < ET; e++)
            k.line("o[" + S(e) + "] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[" + S(r) + "][" + S(e) + "], p[" + S(r) + "], o[" + S(e) + "], 0, 0, 0);");
    k.indent--;
    k.line("};");
    k.line("float ka[" + S(DS) + "], kb[" + S(DS) + "], va[4][" + S(ET) + "], vb[4][" + S(ET) + "];");
    const std::string step = S(16 * NWV);
    k.line("int t = klo + wv * 16;");
    k.line("if (t < khi) fetch(t, ka, va);");
    k.line("for (; t < khi; t += 2 * " + step + ") {");
    k.line("  if (t + " + step + " < khi) fetch(t + " + step + ", kb, vb);");
    k.line("  fold(t, ka, va);");
    k.line("  if (t + " + step + " >= khi) break;");
    k.line("  if (t + 2 * " + step + " < khi) fetch(t + 2 * " + step + ", ka, va);");
    k.line("  fold(t + " + step + ", kb, vb);");
    k.line("}");
    k.line("l = sanic_rows_sum(l);");
    k.line("if (lane < 16) { m_lds[wv][lane] = m; l_lds[wv][lane] = l; }");
    for (int e = 0; e < ET; e++)
        for (int r = 0; r < 4; r++) k.line("o_lds[wv][(lq * 4 + " + S(r) + ") * " + S(ET) + " + " + S(e) + "][l16] = o[" + S(e) + "][" + S(r) + "];");
    k.line("__syncthreads();");
    // one output point from its merged carrier
    k.line("auto point = [&](int row, int ee, float M, float L, float O) {");
    k.indent++;
    k.line("const idx_t qi = q0 + row;");
    k.line("if (qi >= " + S(NQ) + ") return;");
    k.line("float fs" + S(P.max_slot) + " = M;");
    for (size_t s = 0; s < P.scalar_slots.size(); s++) k.line("float fs" + S(P.scalar_slots[s]) + " = " + flit(P.scalar_into[s]) + " * L;");
    k.line("float fs" + S(P.vec_slots[0]) + " = O;");
    // Infinities and NaNs: a masked key weighs 0 here, and 0 · ∞ is not what the fold over the
    // honest window gives; such a point is folded again
    k.line("if (!(__builtin_fabsf(O) <= 3.402823466e38f) || !(__builtin_fabsf(L) <= 3.402823466e38f) || !(__builtin_fabsf(M) <= 3.402823466e38f)) {");
    k.indent++;
    for (int j = 0; j < st.rank; j++) k.line("const idx_t g" + S(j) + " = " + gc[j] + ";");
    emit_point_fold(R, k, st, "pf");
    for (int s = 0; s < c.slots; s++) k.line("fs" + S(s) + " = pf" + S(s) + ";");
    k.indent--;
    k.line("}");
    std::string fargs;
    for (int s = 0; s < c.slots; s++) fargs += ", fs" + S(s);
    k.line("finish(a, hh, qi, ee" + fargs + ");");
    k.indent--;
    k.line("};");
    // n partials in order: M = max m, each weighed by exp(m − M), a side whose m is −∞ by 0
    auto merge = [&](const std::string& n, const std::string& m, const std::string& l, const std::string& o) {
        k.line("float M = -__builtin_huge_valf();");
        k.line("for (int w = 0; w < " + n + "; ++w) M = fmaxf(M, " + m + ");");
        k.line("float L = 0.0f, O = 0.0f;");
        k.line("for (int w = 0; w < " + n + "; ++w) {");
        k.line("  const float mw = " + m + ", x = mw == -__builtin_huge_valf() ? 0.0f : expf(mw - M);");
        k.line("  L = fmaf(x, " + l + ", L);");
        k.line("  O = fmaf(x, " + o + ", O);");
        k.line("}");
    };
    const std::string points = "for (int p = tid; p < " + S(16 * E) + "; p += " + S(64 * NWV) + ") {";
    k.line(points);
    k.indent++;
    k.line("const int ee = p % " + S(E) + ", row = p / " + S(E) + ";");
    merge(S(NWV), "m_lds[w][row]", "l_lds[w][row]", "o_lds[w][ee][row]");
    if (SPL > 1) {
        k.line("if (nsp > 1) {");
        k.line("  float* to = a.scratch + ((idx_t)bid * " + S(SPL) + " + part) * " + S(PSZ) + ";");
        k.line("  " + stx + "(to + p, O);");
        k.line("  if (ee == 0) { " + stx + "(to + " + S(16 * E) + " + row, M); " + stx + "(to + " + S(16 * E + 16) + " + row, L); }");
        k.line("  continue;");
        k.line("}");
    }
    k.line("point(row, ee, M, L, O);");
    k.indent--;
    k.line("}");
    if (SPL > 1) {
        k.line("if (nsp == 1) return;");
        k.line("unsigned* cnt = a.counters + bid;");
        emit_arrival(k, "sanic_last", "tid", "cnt", "(unsigned)nsp", xl);
        k.line("if (!sanic_last) return;");
        k.line("if (tid == 0) sanic_st(cnt, 0u);");
        k.line("const float* from = a.scratch + (idx_t)bid * " + S(SPL * PSZ) + ";");
        k.line(points);
        k.indent++;
        k.line("const int ee = p % " + S(E) + ", row = p / " + S(E) + ";");
        // (every partial requested before the first is used)
        k.line("float pm[" + S(SPL) + "], pl[" + S(SPL) + "], po[" + S(SPL) + "];");
        k.line("#pragma unroll");
        k.line("for (int w = 0; w < " + S(SPL) + "; ++w) {");
        k.line("  const float* f = from + (w < nsp ? w : 0) * " + S(PSZ) + ";");
        k.line("  pm[w] = " + ldx + "(f + " + S(16 * E) + " + row);");
        k.line("  pl[w] = " + ldx + "(f + " + S(16 * E + 16) + " + row);");
        k.line("  po[w] = " + ldx + "(f + p);");
        k.line("}");
        k.line("float M = -__builtin_huge_valf();");
        k.line("#pragma unroll");
        k.line("for (int w = 0; w < " + S(SPL) + "; ++w) { if (w >= nsp) pm[w] = -__builtin_huge_valf(); M = fmaxf(M, pm[w]); }");
        k.line("float L = 0.0f, O = 0.0f;");
        k.line("#pragma unroll");
        k.line("for (int w = 0; w < " + S(SPL) + "; ++w) {");
        k.line("  if (w >= nsp) continue;");
        k.line("  const float x = pm[w] == -__builtin_huge_valf() ? 0.0f : expf(pm[w] - M);");
        k.line("  L = fmaf(x, pl[w], L);");
        k.line("  O = fmaf(x, po[w], O);");
        k.line("}");
        k.line("point(row, ee, M, L, O);");
        k.indent--;
        k.line("}");
    }

    const std::string kname = "sanic_attn32_h" + S(NH) + "_s" + S(NQ) + "_t" + S(T);
    std::ostringstream src;
    src << kPrelude;
    src << "typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;\n";
    src << "typedef float sanic_f32x4_any __attribute__((ext_vector_type(4), aligned(4)));\n";
    src << "typedef float sanic_f32x2_any __attribute__((ext_vector_type(2), aligned(4)));\n";
    src << R.args_struct(SPL > 1 ? std::vector<std::string>{"float* __restrict__ scratch", "unsigned* counters"} : std::vector<std::string>{});
    src << "__device__ __forceinline__ float score(const Args& a, float dotv, int hh, int qi, int kj) {\n"
        << Rs.entry() << sp.str() << "  return " << vpart << ";\n}\n";
    src << "__device__ __forceinline__ void window(const Args& a, idx_t hh, idx_t qrow, idx_t& lo, idx_t& hi) {\n"
        << Rw.entry() << wc.str() << "  lo = wlo; hi = whi;\n}\n";
    src << "__device__ __forceinline__ void finish(const Args& a, idx_t hh, idx_t qi, idx_t ee";
    for (int s = 0; s < c.slots; s++) src << ", float fs" << s;
    src << ") {\n" << Ro.entry() << fo.str() << "}\n";
    src << "extern \"C\" __global__ void __launch_bounds__(" << 64 * NWV << ") " << kname << "(Args a) {\n" << R.entry() << k.str() << "}\n";
    out.kernel_kind = "skeleton:attn_f32[d " + S(HD) + "]" + (SPL > 1 ? "+split" + S(SPL) : "") + (xl ? "+xcd" : "");
    out.source = src.str();
    out.variants = 1;
    std::vector<Arg> args = R.arg_list();
    if (SPL > 1) {
        args.push_back({Arg::SCRATCH, soff});
        args.push_back({Arg::COUNTERS, take_counters(NB)});
    }
    out.launches.push_back({kname, "", dim3((unsigned)(SPL > 1 ? NBP * SPL : NB)), dim3(64 * NWV), 0, args});
    return true;
}

}  // namespace sanic
