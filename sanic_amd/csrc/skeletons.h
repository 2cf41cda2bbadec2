// Structural analysis shared by the skeletons: symbolic affine coordinates and accesses.
#pragma once
#include <functional>
#include <set>
#include <string>
#include <vector>

#include "emit.h"

namespace sanic {

// coef · ((var / div) % mod); mod 0 = none
struct SymTerm {
    int64_t coef;
    int var;
    int64_t div;
    int64_t mod;
};

// c0 + Σ terms: an integer coordinate as a function of kernel variables
struct Sym {
    int64_t c0 = 0;
    std::vector<SymTerm> terms;
    static Sym var(int v);
    std::string render(const std::vector<std::string>& vars) const;
};

// Kernel functions: two floats packed as bf16 (RNE), and as hi + lo bf16 pairs.
extern const char* kSplitBf16;

// An Input read through Reindex/View chains, as element address = Sym.
struct Access {
    int buffer = -1, dtype = -1, node = -1;
    Sym addr;
};

// The element address of `node` at symbolic coordinates `c` (ext = extent of each variable);
// false when the node is not an affine view of one input (or a padded read may go out of
// bounds).
bool sym_access(const sanic_program_desc* d, int node, const std::vector<Sym>& c,
                const std::vector<int64_t>& ext, Access& out);

bool sym_child_coords(const sanic_program_desc* d, int node, const std::vector<Sym>& c,
                      const std::vector<int64_t>& ext, std::vector<Sym>& sc);

void collect_inputs(const sanic_program_desc* d, int node, std::set<int>& bufs);
// match Lt(coordinate, X + 1) (inside a product) with X scalar: the row dim and X's node
bool match_row_cond(const sanic_program_desc* d, int node, int rank, int& dim, int& pos);
// The decode-attention stage that performs in-place row write `si` itself (the K/V cache
// update of this step feeding that attention), or -1.
int attn_absorber(const sanic_program_desc* d, int si);

// One run of 8 of an elementwise leaf (see skeletons.cpp): loads in `lc` through pointers
// rb<i><sfx> for `bufs`, arithmetic in `dc`.
std::vector<std::string> render_run(const sanic_program_desc* d, int node, const std::vector<Sym>& c,
                                    const std::vector<int64_t>& ext, const std::vector<std::string>& vars, int kv,
                                    Code& lc, Code& dc, const std::string& sfx, std::vector<int>& bufs,
                                    std::vector<int>& dtypes, bool& ok);

// One run of 8 of a weight or row leaf at (nn, k0), and a packed 4-bit weight as q·A ± B
// (skeletons.cpp).
std::vector<std::string> render_weight_run(const sanic_program_desc* d, int node, const std::vector<Sym>& c,
                                           const std::vector<int64_t>& ext, Code& lc, Code& dc, const std::string& nn,
                                           const std::string& k0, const std::string& sfx, std::vector<int>& bufs,
                                           std::vector<int>& dtypes, bool& ok, bool& contiguous, std::string& raw_bf16,
                                           bool stream);
bool render_weight_affine(const sanic_program_desc* d, int node, const std::vector<Sym>& c,
                          const std::vector<int64_t>& ext, Code& lc, Code& dc, const std::string& nn,
                          const std::string& k0, const std::string& sfx, std::vector<int>& bufs,
                          std::vector<int>& dtypes, std::vector<std::string>& q, std::string& A, std::string& B,
                          bool& negB, int64_t& uniform_div, bool stream, bool raw_loads = false);

// A Plain(Add) stage over two output axes as a contraction (skel_gemm.cpp): one slot W·rest(row
// items) summed over the stream, the other slots free of W.
struct GemmPlan {
    int mdim = -1, ndim = -1;
    int64_t M = 0, N = 0, K = 0;
    int w = -1;
    std::vector<int> rows;          // row leaves
    std::vector<int> cslots, rslots;
};
bool gemm_plan(const sanic_program_desc* d, int si, GemmPlan& P);
bool exact_in_two(const sanic_program_desc* d, const sanic_stage& st, int e, int w, int& factors);
std::string expr_rest(Renderer& R, Code& code, int e, int w, const std::function<std::string(int)>& item);

bool lower_gemm(const sanic_program_desc* d, int si, int64_t& scratch, LoweredStage& out);
// The generic split fold is faster than either kernel.
bool split_fold_faster(const sanic_program_desc* d, int si);
// `gemm_too`: decline where the GEMM's tiles are estimated to be faster.
bool lower_skinny(const sanic_program_desc* d, int si, LoweredStage& out, bool gemm_too);
bool lower_flash_f32(const sanic_program_desc* d, int si, int64_t& scratch, LoweredStage& out);
bool lower_flash_prefill(const sanic_program_desc* d, int si, int64_t& scratch, LoweredStage& out);
bool lower_attn_decode(const sanic_program_desc* d, int si, int64_t& scratch, LoweredStage& out);

// Lower stage `si` (and the following stages it batches with) onto the gemv skeleton.
bool lower_gemv_group(const sanic_program_desc* d, int si, int64_t& scratch, std::vector<LoweredStage>& out);

}  // namespace sanic
