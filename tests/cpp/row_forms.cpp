// Host-only: every plan of contiguous and every-second-element rows that a register row kernel runs has a kernel. The launcher
// (norm_op.hip) is compiled for the numbers of vectors per thread that the planner (layout.cpp) gives to each form of the rows and refuses others; the
// table below is the launcher's. Rows, row lengths, pitches and addresses on and off the 16-byte grid go through plan_normalize. No GPU call is made.
#include <cstdio>
#include <random>
#include <set>
#include <string>

#include "common.hpp"

using namespace hpt;

enum Kind { SOFTMAX, LAYERNORM, ADD_LAYERNORM, CAUSAL };
static const char* const kNames[] = {"softmax", "layernorm", "add_layernorm", "causal"};
static long seen = 0, bad = 0;

// The numbers of vectors per thread that the launcher has for this plan, and the form's name.
static std::set<int> kernels_of(const NormPlan& p, int size, Kind k, std::string& form) {
    const int full = 16 / size;
    const bool layer = k == LAYERNORM || k == ADD_LAYERNORM;
    int64_t grid = (p.rows + p.rpb - 1) / p.rpb;
    if (layer && grid > p.max_blocks) grid = p.max_blocks;
    if (p.vec == full && p.ua_rows) {
        form = "unaligned";
        if (p.cols < full || size == 8 || (p.sstride == 2 && size != 2) || p.gb_lds == 2 || (p.gb_lds == 1 && size != 2)) return {};
        if (size == 2 && p.sstride == 2) return layer ? std::set<int>{4} : std::set<int>{2, 4};
        if (size == 2 && layer && p.gb_lds) return {3, 4};
        if (size == 2) return k == ADD_LAYERNORM ? std::set<int>{2} : k == LAYERNORM ? std::set<int>{2, 3} : std::set<int>{2, 3, 4};
        if (k == ADD_LAYERNORM) return {2, 3, 4};
        if (k == LAYERNORM) return p.tpr >= 512 ? std::set<int>{3, 4, 5, 6} : std::set<int>{2, 3, 4, 5};
        return {};
    }
    if (p.vec == full && p.shift) {
        form = "masked";
        if (p.sstride != 1 || p.gb_lds || (layer && grid * p.rpb < p.rows && grid < full)) return {};
        if (size == 2 || (size == 4 && k == ADD_LAYERNORM)) return {};
        return layer ? std::set<int>{2, 3, 4} : std::set<int>{2, 3, 4, 5, 6, 7, 8};
    }
    if (layer && p.gb_lds) {
        form = p.gb_lds == 2 ? "gamma and beta from L2" : "gamma and beta in LDS";
        if (p.vec != full || p.sstride != 1) return {};
        if (p.gb_lds == 1) return size == 2 ? std::set<int>{3, 4} : std::set<int>{};
        return size == 2 ? std::set<int>{3, 4, 5, 6} : std::set<int>{3, 4, 5, 6, 7, 8};
    }
    if (p.vec == full && p.sstride == 2 && grid > 512 && k != ADD_LAYERNORM) {
        form = "every second element, walked";
        if (k == LAYERNORM && (size == 4 ? p.tpr == 1024 : size == 2 && p.tpr >= 512)) return {4};
        if (k != LAYERNORM && size == 4 && (p.tpr == 1024 || (p.tpr == 512 && p.nchunk == 8))) return {4, 8};
    }
    form = "plain";
    if (p.vec == full && p.sstride == 1) return {1, 2, 3, 4, 5, 6, 7, 8};
    return p.vec == 1 || p.vec == full ? std::set<int>{1, 2, 4, 8} : std::set<int>{};
}

static void check(const NormPlan& p, int size, Kind k, const char* what) {
    if (p.kind != NormKind::RowReg || p.lds_rows || p.raw_rows || p.interleave != 1 || (p.tile_rows && (k == SOFTMAX || k == LAYERNORM))) return;
    std::string form;
    const std::set<int> kernels = kernels_of(p, size, k, form);
    const int64_t held = (int64_t)p.tpr * p.nchunk * (p.vec > 1 ? p.vec / p.sstride : 1);
    const int64_t need = form == "masked" ? p.cols + p.vec - 1 : p.cols;  // (the vectors that contain the row, wherever it starts)
    ++seen;
    if (kernels.count(p.nchunk) && held >= need && p.tpr * p.rpb <= 1024) return;
    if (++bad <= 20) printf("%s, %s of %d bytes, %s: %s\n", kNames[k], form.c_str(), size, what, describe(p).c_str());
}

int main() {
    std::mt19937_64 rng(1);
    for (int size : {2, 4, 8})
        for (int64_t cols = 1; cols <= 70000; cols += cols < 2100 ? 1 : 1 + (int64_t)(rng() % 120))
            for (int64_t rows : {1, 17, 64, 129, 300, 512, 513, 1025, 2000, 5000, 20000, 200000}) {
                if (rows * cols > (1ll << 32)) continue;
                for (int step : {1, 2})
                    for (int gap : {0, 1, 3, 16 / size})
                        for (int t = 0; t < 3; ++t) {  // output and input off the grid alike, and by different amounts
                            const int io = t == 0 ? 0 : (int)(rng() % (16 / size)), oo = t < 2 ? io : (int)(rng() % (16 / size)), ro = (int)(rng() % (16 / size));
                            const uintptr_t in = (1ull << 40) + io * size, out = (2ull << 40) + oo * size, residual = (3ull << 40) + ro * size;
                            const int64_t shape[2] = {rows, cols}, strides[2] = {cols * step + gap, step};
                            char what[120];
                            snprintf(what, sizeof what, "[%lld, %lld] step %d, %d between rows, off %d %d %d", (long long)rows, (long long)cols, step, gap, io, oo, ro);
                            auto plan = [&](int64_t axis, int dims, bool fused, uintptr_t r) {
                                return plan_normalize((void*)in, (void*)out, shape, strides, 2, axis, dims, size, fused, (void*)r);
                            };
                            check(plan(1, 0, false, 0), size, SOFTMAX, what);
                            check(plan(0, 1, false, 0), size, LAYERNORM, what);
                            check(plan(1, 0, true, 0), size, CAUSAL, what);
                            NormPlan p = plan(0, 1, true, residual);
                            // (as the caller does: masked rows need the residual off the grid like the output)
                            if (!(p.shift && !p.ua_rows && ((residual ^ out) & 15))) check(p, size, ADD_LAYERNORM, what);
                        }
            }
    printf("%ld plans, %ld without a kernel\n", seen, bad);
    return bad != 0;
}
