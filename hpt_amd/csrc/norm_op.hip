// One normalisation kind (softmax, log_softmax or layernorm) for the four
// float dtypes. Compiled once per kind with -DHPT_NORM_KIND=<0...5>.
#include <algorithm>

#include "norm_interleaved.hpp"
#include "transpose_norm.hpp"

#ifndef HPT_NORM_KIND
#error "compile with -DHPT_NORM_KIND=<kind>"
#endif

namespace hpt {

namespace {

constexpr int KIND = HPT_NORM_KIND;

inline int ilog2(int v) {
    int l = 0;
    while ((1 << l) < v) ++l;
    return l;
}

// The row kernel of full vectors for the numbers of vectors per thread that the plan has in this form.
template <class T, int SS, bool SHIFT, bool PF, bool UA, int... NC>
void launch_row_of(const NormPlan& p, const NormArgs& a, dim3 grid, dim3 block, hipStream_t st) {
    const bool done = ((p.nchunk == NC && (row_reg_kernel<KIND, T, 16 / sizeof(T), NC, SS, SHIFT, PF, 0, 1, UA><<<grid, block, 0, st>>>(a), true)) || ...);
    if (!done) fail(HPT_ERR_KERNEL, "row_reg: no kernel of %d vectors per thread in this form", p.nchunk);
}

template <class T, int VEC, int SS = 1, bool PF = false>
void launch_row_reg(const NormPlan& p, const NormArgs& a, dim3 grid, dim3 block, hipStream_t st) {
    // (3, 5, 6 and 7 vectors per thread: rows of whole vectors whose length is 3, 5, 6 or 7 times a power of
    // two - 768, 1536, 2560, 3072, 3584, 5120, 6144 ... - without idle lanes; full-vector rows only)
    if constexpr (VEC > 1 && SS == 1) {
        switch (p.nchunk) {
            case 3: row_reg_kernel<KIND, T, VEC, 3, SS, false, PF><<<grid, block, 0, st>>>(a); return;
            case 5: row_reg_kernel<KIND, T, VEC, 5, SS, false, PF><<<grid, block, 0, st>>>(a); return;
            case 6: row_reg_kernel<KIND, T, VEC, 6, SS, false, PF><<<grid, block, 0, st>>>(a); return;
            case 7: row_reg_kernel<KIND, T, VEC, 7, SS, false, PF><<<grid, block, 0, st>>>(a); return;
            default: break;
        }
    }
    switch (p.nchunk) {
        case 1: row_reg_kernel<KIND, T, VEC, 1, SS, false, PF><<<grid, block, 0, st>>>(a); break;
        case 2: row_reg_kernel<KIND, T, VEC, 2, SS, false, PF><<<grid, block, 0, st>>>(a); break;
        case 4: row_reg_kernel<KIND, T, VEC, 4, SS, false, PF><<<grid, block, 0, st>>>(a); break;
        case 8: row_reg_kernel<KIND, T, VEC, 8, SS, false, PF><<<grid, block, 0, st>>>(a); break;
        default: fail(HPT_ERR_KERNEL, "row_reg: unsupported chunk count %d", p.nchunk);
    }
}

// Rows off the vector grid as unaligned vectors (two-byte types, f32 layernorms).
template <class T> void launch_row_unaligned(const NormPlan& p, const NormArgs& a, dim3 grid, dim3 block, hipStream_t st) {
    constexpr int FULL = 16 / sizeof(T);
    if (a.cols < FULL) fail(HPT_ERR_KERNEL, "row_reg: rows of %lld elements hold no vector", (long long)a.cols);
    if constexpr (sizeof(T) == 2) {
        if (p.sstride == 2) {
            // (every second element; x + residual, whose four vectors spill, where it would stream otherwise)
            if constexpr (KIND == NORM_ADD_LAYERNORM) {
                launch_row_of<T, 2, false, false, true, 4>(p, a, grid, block, st);
            } else if constexpr (KIND == NORM_LAYERNORM) {
                if (p.tpr >= 512) {
                    if (grid.x > 512u) grid.x = 512u;
                    launch_row_of<T, 2, false, true, true, 4>(p, a, grid, block, st);
                } else {
                    launch_row_of<T, 2, false, false, true, 4>(p, a, grid, block, st);
                }
            } else {
                launch_row_of<T, 2, false, false, true, 2, 4>(p, a, grid, block, st);
            }
            return;
        }
        if constexpr (norm_is_layer(KIND)) {
            if (p.gb_lds == 1) {
                const size_t smem = 2 * (size_t)((p.cols + FULL - 1) / FULL) * FULL * sizeof(T);
                if (p.tpr >= 512 && grid.x > 512u) grid.x = 512u;
                if (p.nchunk == 3) row_reg_kernel<KIND, T, FULL, 3, 1, false, false, 1, 1, true><<<grid, block, smem, st>>>(a);
                else if (p.nchunk == 4) row_reg_kernel<KIND, T, FULL, 4, 1, false, false, 1, 1, true><<<grid, block, smem, st>>>(a);
                else fail(HPT_ERR_KERNEL, "row_reg: no kernel of %d vectors per thread in this form", p.nchunk);
                return;
            }
        }
        if constexpr (KIND == NORM_ADD_LAYERNORM) launch_row_of<T, 1, false, false, true, 2>(p, a, grid, block, st);
        else if constexpr (KIND == NORM_LAYERNORM) launch_row_of<T, 1, false, false, true, 2, 3>(p, a, grid, block, st);
        else launch_row_of<T, 1, false, false, true, 2, 3, 4>(p, a, grid, block, st);
    } else if constexpr (sizeof(T) == 4 && KIND == NORM_ADD_LAYERNORM) {
        launch_row_of<T, 1, false, false, true, 2, 3, 4>(p, a, grid, block, st);
    } else if constexpr (sizeof(T) == 4 && KIND == NORM_LAYERNORM) {
        if (p.tpr >= 512) {
            if (grid.x > 512u) grid.x = 512u;
            launch_row_of<T, 1, false, true, true, 3, 4, 5, 6>(p, a, grid, block, st);
        } else {
            launch_row_of<T, 1, false, false, true, 2, 3, 4, 5>(p, a, grid, block, st);
        }
    } else {
        fail(HPT_ERR_KERNEL, "row_reg: rows of this type are no unaligned vectors");
    }
}

// Few, very long rows: several workgroups per row.
template <class T, int VEC, bool UA> void launch_row_split(const NormPlan& p, const NormArgs& a, hipStream_t st) {
    RowSplitArgs r{};
    r.in = a.in;
    r.out = a.out;
    r.gamma = a.gamma;
    r.beta = a.beta;
    r.residual = a.residual;
    r.kept_in = a.kept_in;
    r.rows = a.rows;
    r.cols = a.cols;
    r.eps = a.eps;
    r.inv_cols = a.inv_cols;
    r.S = p.tsplit;
    const int64_t nv = UA ? (a.cols + VEC - 1) / VEC : a.cols / VEC;
    r.chunk_v = (nv + r.S - 1) / r.S;
    r.part = a.scratch;
    const dim3 grid((unsigned)r.S, (unsigned)a.rows);
    row_split_stats_kernel<KIND, T, VEC, UA><<<grid, dim3(256), 0, st>>>(r);
    row_split_apply_kernel<KIND, T, VEC, UA><<<grid, dim3(256), 0, st>>>(r);
}

// Softmax / log_softmax over an axis that is strided in the output too: three passes.
template <class T, int VEC> void launch_col_split(const NormPlan& p, const NormArgs& a, hipStream_t st) {
    TransposedArgs t{};
    t.in = a.in;
    t.out = a.out;
    const int nk = p.kept_in.n;
    const unsigned batch = nk > 1 ? (unsigned)p.kept_in.size[0] : 1u;
    t.R = (int)p.kept_in.size[nk - 1];
    t.cols = (int)p.cols;
    t.S = p.tsplit;
    t.stats = a.scratch;
    t.params = (char*)a.scratch + (size_t)batch * t.S * t.R * 16;
    t.sa = a.sa;
    t.bi = nk > 1 ? p.kept_in.stride[0] : 0;
    t.inv_cols = a.inv_cols;
    using Part = typename RowPartial<KIND, T>::type;
    if constexpr (VEC > 1) {
        if (p.flat_t > 0) {  // narrow inner dim: flat walk (statistics, the shared finalize, apply)
            const unsigned block = (unsigned)((p.flat_t + 63) / 64 * 64);
            const size_t smem = (size_t)p.flat_t * VEC * sizeof(Part);
            const dim3 grid((unsigned)t.S, 1, batch);
            if (p.shift) {  // batch slabs off 16-byte boundaries: unaligned vectors
                col_flat_stats_kernel<KIND, T, VEC, true><<<grid, dim3(block), smem, st>>>(t, p.flat_t);
                transposed_finalize_kernel<KIND, T><<<dim3((unsigned)((t.R + 15) / 16), 1, batch), dim3(16, 16), 0, st>>>(t);
                col_flat_apply_kernel<KIND, T, VEC, true><<<grid, dim3(block), 0, st>>>(t, p.flat_t, t.S);
            } else {
                col_flat_stats_kernel<KIND, T, VEC><<<grid, dim3(block), smem, st>>>(t, p.flat_t);
                transposed_finalize_kernel<KIND, T><<<dim3((unsigned)((t.R + 15) / 16), 1, batch), dim3(16, 16), 0, st>>>(t);
                col_flat_apply_kernel<KIND, T, VEC><<<grid, dim3(block), 0, st>>>(t, p.flat_t, t.S);
            }
            return;
        }
    }
    const unsigned nw = (unsigned)p.tpr;
    const unsigned rg = (unsigned)((t.R + 64 * VEC - 1) / (64 * VEC));
    const bool ua = VEC > 1 && p.shift;  // inner rows off the vector grid: unaligned vectors
    if (ua && t.R < VEC) fail(HPT_ERR_KERNEL, "col-split: an inner row of %d elements holds no vector of %d", t.R, VEC);
    // Inner rows of vectors that do not start on cache lines: neighbours in x share lines, and the grids of the two large passes are dealt to the XCDs in
    // eight equal parts. Us over axis 0, as numbered by the hardware and this: f32 [8190, 4097] 78.4 and 72.3, [8192, 4112] 78.6 and 73.0, [30000, 1001]
    // 69.4 and 65.4, f16 [8190, 4097] 43.8 and 40.2, bf16 [2700, 12001] 39.9 and 38.2. Rows that start on lines lose by it ([8192, 4096]
    // 66.6 and 68.5), and so do inputs below 16 MiB ([2000, 1111] 17.4 and 17.8).
    const bool on_lines = (t.R * (int64_t)sizeof(T)) % 128 == 0 && (t.sa * (int64_t)sizeof(T)) % 128 == 0 && (((uintptr_t)t.in | (uintptr_t)t.out) & 127) == 0;
    const bool shared = VEC > 1 && !on_lines && (int64_t)batch * t.cols * t.R * (int64_t)sizeof(T) >= (16ll << 20);
    auto set_grid = [&](const dim3& g) {
        t.gx = g.x;
        t.gy = g.y;
        const uint64_t n = (uint64_t)g.x * g.y * g.z;
        t.shared = shared && n < (1ull << 31) ? (unsigned)n : 0;
        return g;
    };
    const dim3 sgrid = set_grid(dim3(rg, (unsigned)t.S, batch));
    auto as_grid = [&](auto launch) {  // launch(unaligned, shared)
        if constexpr (VEC > 1) {
            if (ua && t.shared) return launch(std::true_type{}, std::true_type{});
            if (ua) return launch(std::true_type{}, std::false_type{});
            if (t.shared) return launch(std::false_type{}, std::true_type{});
        }
        launch(std::false_type{}, std::false_type{});
    };
    as_grid([&](auto unaligned, auto dealt) {
        transposed_stats_kernel<KIND, T, VEC, decltype(unaligned)::value, decltype(dealt)::value><<<sgrid, dim3(64 * nw), (size_t)nw * VEC * 64 * sizeof(Part), st>>>(t);
    });
    transposed_finalize_kernel<KIND, T><<<dim3((unsigned)((t.R + 15) / 16), 1, batch), dim3(16, 16), 0, st>>>(t);
    // apply: sixteen positions of the axis per workgroup, one batch of four loads per thread; what runs at one time is then
    // one stretch of memory (f32 [8192, 4096] over axis 0, all three passes, 16 / 32 / 48 positions: 65.2, 70.7, 67.4 us;
    // [32768, 1024] 66.3, 68.4, 68.6; f16 [8190, 4097] 42.0, 43.1, 43.1). Where lines are shared eight, so that what an XCD has in flight is a
    // shorter stretch (8 / 16 positions: f32 [8190, 4097] 71.7 and 73.2, [30000, 1001] 65.4 and 66.3, f16 [8190, 4097] 40.3 and 41.2).
    const int64_t most = shared ? 8 : 16;
    int64_t chunks = std::min<int64_t>((t.cols + most - 1) / most, 65535);
    const int chunk = (int)((t.cols + chunks - 1) / chunks);
    chunks = (t.cols + chunk - 1) / chunk;
    const dim3 agrid = set_grid(dim3(rg, (unsigned)chunks, batch));
    as_grid([&](auto unaligned, auto dealt) {
        col_apply_kernel<KIND, T, VEC, decltype(unaligned)::value, decltype(dealt)::value><<<agrid, dim3(256), 0, st>>>(t, chunk);
    });
}

// How many neighbouring workgroups of the column kernels share an XCD, as xcd_order takes it; `whole`: what is right where inner rows
// start on cache lines. The others share the lines between them: equal shares of the launch while input and output together fit the last-level
// cache, runs of 32 (an XCD's units) beyond, which keeps what is in flight in one stretch of memory. Us, softmax over axis 1, as numbered by the
// hardware (col_reg_kernel) or in pairs (col_tall_kernel) and this: f32 [64, 128, 3249] 56.0 and 48.0, [3000, 40, 250] 60.3 and 52.7, f16 [64, 128, 3249]
// 29.7 and 25.1; runs of 32 and shares: f32 [46, 300, 301] 13.9 and 11.4, [64, 512, 510] 35.2 and 36.1, [129, 512, 510] 81.9 and 92.9. On
// cache lines nothing moves ([64, 128, 3136] 40.4 and 40.8).
static int column_run(const ColRegArgs& c, size_t elem_size, int whole) {
    if ((c.L * (int64_t)elem_size) % 128 == 0 && (c.sa * (int64_t)elem_size) % 128 == 0 && (((uintptr_t)c.in | (uintptr_t)c.out) & 127) == 0) return whole;
    const int64_t batch = c.total / c.nvec;
    return batch * c.cols * c.L * (int64_t)elem_size < (48ll << 20) ? kXcdShares : 5;
}

// A short strided axis held in registers (softmax kinds).
// WIDE: twice the vectors per thread (128 registers of raw values instead of 64).
template <class T, int EV, bool WIDE = false> void launch_col_reg(const NormPlan& p, const NormArgs& a, hipStream_t st) {
    constexpr int REGS = (EV * (int)sizeof(T) + 3) / 4;
    constexpr int NC = (64 / REGS > 64 ? 64 : 64 / REGS) * (WIDE ? 2 : 1);
    ColRegArgs c{};
    const int nk = p.kept_in.n;
    c.in = a.in;
    c.out = a.out;
    c.sa = a.sa;
    c.bi = nk > 1 ? p.kept_in.stride[0] : 0;
    c.L = p.kept_in.size[nk - 1];
    c.nvec = p.shift ? (c.L + EV - 1) / EV : c.L / EV;
    c.total = (nk > 1 ? p.kept_in.size[0] : 1) * c.nvec;
    c.cols = (int)p.cols;
    c.ty_log2 = ilog2(p.tpr);  // thread rows per inner position
    if (p.tpr > 16 || c.cols > NC * p.tpr)
        fail(HPT_ERR_KERNEL, "col-reg: axis of %d does not fit %d thread rows of %d vectors", c.cols, p.tpr, NC);
    const int64_t tx = 256 / p.tpr;
    const dim3 grid((unsigned)((c.total + tx - 1) / tx));
    c.blocks = grid.x;
    // (Up to eight bytes per thread of inner rows that a workgroup holds whole share lines at its ends only, and the numbering costs more: us, dealt and as they
    // come, f32 [472, 176, 9] 11.6 and 10.4, [776, 144, 15] 11.5 and 10.7; but [36, 1000, 157] 17.8 and 23.2, f64 pairs
    // [100, 60, 33] 12.7 and 15.5.)
    constexpr bool kNarrow = EV * sizeof(T) <= 8;
    c.run_log2 = kNarrow && c.nvec < tx ? 0 : column_run(c, sizeof(T), p.shift ? 5 : 0);  // (unaligned with every row on a line: only a batch is off it)
    if constexpr (EV > 1) {
        if (p.shift && c.run_log2) {
            col_reg_kernel<KIND, T, EV, NC, true, true><<<grid, dim3(256), 0, st>>>(c);
            return;
        }
    }
    if constexpr (EV > 1 && kNarrow) {
        if (p.shift) {
            col_reg_kernel<KIND, T, EV, NC, true, false><<<grid, dim3(256), 0, st>>>(c);
            return;
        }
    }
    if (EV > 1 && p.shift) fail(HPT_ERR_KERNEL, "col-reg: unaligned vectors of %d as they come", EV);
    if (c.run_log2) col_reg_kernel<KIND, T, EV, NC, false, true><<<grid, dim3(256), 0, st>>>(c);
    else col_reg_kernel<KIND, T, EV, NC><<<grid, dim3(256), 0, st>>>(c);
}

// Whether the result of col_tall_kernel leaves through the caches. Segments that do not end on 64 bytes share what memory writes at once
// with their neighbours: non-temporal, both parts go out by themselves. Through the cache, with neighbours on one XCD, they meet there. Us, non-temporal
// and cached: f32 [512, 512, 510] 333 and 255, [512, 512, 500] 328 and 285, [46, 1000, 500] 66.0 and 47.9, [116, 512, 500] 74.1 and 51.4, [64, 512, 510] 37.8 and 29.9,
// [84, 200, 1001] 34.1 and 32.6, f16, whole vectors, [131, 512, 1000] 81.3 and 67.3, [66, 512, 1000] 47.4 and 37.1. Whole vectors from 20 MiB of four bytes and 48 of two on (below,
// where the last-level cache takes either, f32 [67, 256, 250] 12.3 and 14.4), but not whole 64-byte pieces ([512, 512, 528] 219 and 243).
// Unaligned vectors, of which a row's last one is stored in elements, only of four bytes (f16, 150 MiB: [250, 400, 501] 1.28 times the time, [800, 300, 301] 1.16) and only where a
// segment is a part of an inner row, so that rows share less than segments do: [655, 256, 50] 21.1 and 23.0, [1273, 256, 37] 23.0 and 24.5, [421, 256, 90] 20.5 and 22.6, but
// [463, 200, 130] 23.1 and 22.1, [310, 300, 90] 19.7 and 18.9. Those from 34 MiB on (16 vectors of a row per workgroup: 26; ratio cached / non-temporal of 200 columns at 21, 28, 36, 46, 90 MiB, rows of
// 201: 1.09, 1.10, 0.93, 0.87, 0.90; of 300: 1.06, 0.94, 0.82, 0.85, 0.83), and of 48 to 96 MiB from an axis of 160 on ([167, 160, 706] 37.0 and 33.4, [143, 129, 706] 25.8 and 27.5).
template <class T> bool tall_stores_cached(const NormPlan& p, const ColRegArgs& c) {
    if ((c.L * (int64_t)sizeof(T)) % 64 == 0 && ((uintptr_t)c.out & 63) == 0) return false;
    const int64_t mib = c.total / c.nvec * c.cols * c.L * (int64_t)sizeof(T) >> 20;
    if (!p.shift) return mib >= (sizeof(T) == 2 ? 48 : 20);
    const int tx = p.tall / p.tpr;  // vectors of an inner row per workgroup
    if (sizeof(T) == 2 || 8 * c.L < 9 * tx * (16 / (int)sizeof(T))) return false;
    return mib >= (tx == 16 ? 26 : 34) && (c.cols >= 160 || mib < 48 || mib >= 96);
}

// NT threads, TX of them along the inner dim, NC vectors each.
template <class T, int NT, int TX, int NC> bool launch_col_tall_as(const NormPlan& p, ColRegArgs& c, hipStream_t st) {
    if (p.tall != NT || p.tpr != NT / TX || p.nchunk != NC || c.cols > NT / TX * NC) return false;
    const dim3 grid((unsigned)((c.total + TX - 1) / TX));
    c.blocks = grid.x;
    const bool cached = tall_stores_cached<T>(p, c);
    if constexpr (sizeof(T) == 4) {
        if (p.shift && cached) {
            col_tall_kernel<KIND, T, NT, TX, NC, true, true><<<grid, dim3(NT), 0, st>>>(c);
            return true;
        }
    }
    if (p.shift) col_tall_kernel<KIND, T, NT, TX, NC, true><<<grid, dim3(NT), 0, st>>>(c);
    else if (cached) col_tall_kernel<KIND, T, NT, TX, NC, false, true><<<grid, dim3(NT), 0, st>>>(c);
    else col_tall_kernel<KIND, T, NT, TX, NC><<<grid, dim3(NT), 0, st>>>(c);
    return true;
}

template <class T> void launch_col_tall(const NormPlan& p, const NormArgs& a, hipStream_t st) {
    constexpr int EV = 16 / sizeof(T);
    ColRegArgs c{};
    const int nk = p.kept_in.n;
    c.in = a.in;
    c.out = a.out;
    c.sa = a.sa;
    c.bi = nk > 1 ? p.kept_in.stride[0] : 0;
    c.L = p.kept_in.size[nk - 1];
    c.nvec = (c.L + EV - 1) / EV;
    c.total = (nk > 1 ? p.kept_in.size[0] : 1) * c.nvec;
    c.cols = (int)p.cols;
    c.run_log2 = column_run(c, sizeof(T), 1);
    if (c.L < EV || p.vec != EV || (!p.shift && c.L % EV != 0)) fail(HPT_ERR_KERNEL, "col-reg: inner rows of %lld elements are not whole vectors", (long long)c.L);
    bool done = false;
    if constexpr (sizeof(T) == 4) {
        done = launch_col_tall_as<T, 1024, 32, 8>(p, c, st) || launch_col_tall_as<T, 1024, 16, 8>(p, c, st) || launch_col_tall_as<T, 1024, 16, 16>(p, c, st);
    } else if constexpr (sizeof(T) == 2) {
        done = launch_col_tall_as<T, 512, 16, 8>(p, c, st) || launch_col_tall_as<T, 512, 16, 16>(p, c, st) || launch_col_tall_as<T, 1024, 16, 16>(p, c, st);
    }
    if (!done) fail(HPT_ERR_KERNEL, "col-reg: no kernel of %d threads holds an axis of %d in %d rows of %d vectors", p.tall, c.cols, p.tpr, p.nchunk);
}

// The transposed forms (kinds 0..2 only).
template <class T> void launch_transposed(const NormPlan& p, const NormArgs& a, hipStream_t st) {
    constexpr int FULL = 16 / sizeof(T);
    if (p.kind == NormKind::TransposedTile) {
        TileArgs t{};
        t.in = a.in;
        t.out = a.out;
        t.gamma = a.gamma;
        t.beta = a.beta;
        const int nk = p.kept_in.n;
        const unsigned batch = nk > 1 ? (unsigned)p.kept_in.size[0] : 1u;
        t.R = (int)p.kept_in.size[nk - 1];
        t.cols = (int)p.cols;
        t.sa = a.sa;
        t.bi = nk > 1 ? p.kept_in.stride[0] : 0;
        t.eps = a.eps;
        t.inv_cols = a.inv_cols;
        t.rg_log2 = ilog2(p.tpr);
        const unsigned blocks = (unsigned)((t.R + p.tpr * FULL - 1) / (p.tpr * FULL));
        // On the vector grid the workgroups that share a line: one (rgN = 8 and more), two or four. Off it neighbours share a line at any rgN: four, or
        // eight of two-byte rows (us, softmax, stored [columns, rows]: f32 [2001, 8001] 42.5 and 37.8, [1001, 8191] 21.0 and 18.5, [4001, 4001] 40.1 and
        // 38.1, f16 [2049, 8191] 26.7 and 23.8, [501, 16001] 14.2 and 12.9). Eight neighbours on one XCD also read and write longer stretches, which
        // counts where every compute unit has a workgroup: f32 [4096, 4096] 32.3 and 30.8, [3000, 6000] 49.5 and 47.3, two-byte rows of up to 2048 columns f16 [2048, 8192] 17.6 and
        // 16.3, [2000, 12000] 29.2 and 27.9; not f32 [4000, 2048] 23.6 and 24.5, [1728, 6016] 16.9 and 17.3, f16 [3000, 8000] 34.3 and 35.3, [1024, 8192] 9.7 and 9.8.
        const bool long_stretch = p.tpr == 4 && (sizeof(T) == 2 ? p.rpb <= 8 && (int64_t)t.R * t.cols >= (16ll << 20) : blocks >= 256 && (int64_t)t.R * t.cols >= (12ll << 20));
        if (p.shift) t.share_log2 = p.tpr == 2 ? 2 : (sizeof(T) == 2 && p.tpr == 4 ? 3 : 2);
        else t.share_log2 = p.tpr >= 8 ? 0 : (p.tpr == 4 ? (long_stretch ? 3 : 1) : 2);
        if (p.shift) {
            transposed_tile_kernel<KIND, T, true><<<dim3(blocks, batch), dim3(64u * (unsigned)p.rpb), 0, st>>>(t);
            return;
        }
        if constexpr (std::is_same<T, float>::value && KIND != NORM_LAYERNORM) {
            if (p.wide_sum) {
                transposed_tile_kernel<KIND, T, false, true><<<dim3(blocks, batch), dim3(64u * (unsigned)p.rpb), 0, st>>>(t);
                return;
            }
        }
        transposed_tile_kernel<KIND, T><<<dim3(blocks, batch), dim3(64u * (unsigned)p.rpb), 0, st>>>(t);
        return;
    }
    if (p.kind == NormKind::Transposed) {
        constexpr int TILE = 8 * FULL;
        TransposedArgs t{};
        t.in = a.in;
        t.out = a.out;
        t.gamma = a.gamma;
        t.beta = a.beta;
        const int nk = p.kept_in.n;
        const unsigned batch = nk > 1 ? (unsigned)p.kept_in.size[0] : 1u;
        t.R = (int)p.kept_in.size[nk - 1];
        t.cols = (int)p.cols;
        t.S = p.tsplit;
        // scratch: [batch][S][R] partial statistics (16 bytes each at most), then [batch][3][R] numbers
        t.stats = a.scratch;
        t.params = (char*)a.scratch + (size_t)batch * t.S * t.R * 16;
        t.sa = a.sa;
        t.bi = nk > 1 ? p.kept_in.stride[0] : 0;
        t.eps = a.eps;
        t.inv_cols = a.inv_cols;
        t.nw = p.tpr;
        const int tiles = (t.cols + TILE - 1) / TILE;
        const unsigned rt = (unsigned)((t.R + TILE - 1) / TILE);
        const unsigned rg = (unsigned)((t.R + 64 * FULL - 1) / (64 * FULL));
        using Part = typename RowPartial<KIND, T>::type;
        const unsigned nw = (unsigned)p.tpr;  // wavefronts per workgroup of the statistics pass
        const dim3 sgrid(rg, (unsigned)t.S, batch);
        const size_t slds = (size_t)nw * FULL * 64 * sizeof(Part);
        if (p.shift) transposed_stats_kernel<KIND, T, FULL, true><<<sgrid, dim3(64 * nw), slds, st>>>(t);
        else transposed_stats_kernel<KIND, T><<<sgrid, dim3(64 * nw), slds, st>>>(t);
        transposed_finalize_kernel<KIND, T><<<dim3((unsigned)((t.R + 15) / 16), 1, batch), dim3(16, 16), 0, st>>>(t);
        // (more column blocks than a grid has in y, from 2^22 four-byte columns on: one launch after the other)
        for (int blocks = (tiles + 1) / 2; t.y0 < blocks; t.y0 += 65535) {
            const dim3 agrid((rt + 3) / 4, (unsigned)std::min(blocks - t.y0, 65535), batch);
            // off the vector grid neighbours share lines: eight of them in a row on one XCD (us, softmax, stored [columns, rows]: f32 [8190, 4097]
            // 103.4 and 94.7, f16 59.0 and 50.4, [8192, 4100] 49.8 and 46.2, [5001, 4001] 37.1 and 37.1)
            const uint64_t n = (uint64_t)agrid.x * agrid.y * agrid.z;
            t.gx = agrid.x;
            t.gy = agrid.y;
            t.shared = n < (1ull << 31) ? (unsigned)n : 0;
            if (p.shift) transposed_apply_kernel<KIND, T, true><<<agrid, dim3(256), 0, st>>>(t);
            else transposed_apply_kernel<KIND, T><<<agrid, dim3(256), 0, st>>>(t);
        }
        return;
    }
}

template <class T> void launch_t(const NormPlan& p, NormArgs a, hipStream_t st) {
    constexpr int FULL = 16 / sizeof(T);
    if (p.kind == NormKind::Empty) return;
    a.tpr = p.tpr;
    a.tpr_log2 = ilog2(p.tpr);
    a.rpb = p.rpb;
    a.inv_cols = 1.0 / (double)p.cols;
    dim3 grid((unsigned)((p.rows + p.rpb - 1) / p.rpb));
    dim3 block((unsigned)(p.tpr * p.rpb));
    if (p.kind == NormKind::Col && p.slab_tile > 0) {
        if constexpr (FULL > 1 && (KIND == NORM_SOFTMAX || KIND == NORM_LOGSOFTMAX)) {
            launch_slabs<KIND, T>(p, a, st);
        } else {
            fail(HPT_ERR_KERNEL, "slab tiles are a softmax plan");
        }
        return;
    }
    if (p.kind == NormKind::Col && p.group_tile > 0) {
        if constexpr (FULL > 1 && (KIND == NORM_SOFTMAX || KIND == NORM_LOGSOFTMAX)) {
            const int64_t batch = p.kept_in.size[0];
            a.rpb = p.group_tile;
            // a very narrow inner dim with groups of a multiple of 128 bytes: the lanes' group starts collide in LDS
            const bool padded = p.kept_in.size[1] * (int64_t)sizeof(T) <= 16 && (p.cols * p.kept_in.size[1] * (int64_t)sizeof(T)) % 128 == 0;
            const dim3 ggrid((unsigned)((batch + p.group_tile - 1) / p.group_tile));
            if (padded) norm_group_tile_kernel<KIND, T, FULL, true><<<ggrid, dim3(256), 0, st>>>(a, (int)p.kept_in.size[1], batch);
            else norm_group_tile_kernel<KIND, T, FULL, false><<<ggrid, dim3(256), 0, st>>>(a, (int)p.kept_in.size[1], batch);
        } else {
            fail(HPT_ERR_KERNEL, "group tiles are a softmax plan");
        }
        return;
    }
    if (p.kind == NormKind::RowSplit) {
        if constexpr (norm_is_causal(KIND)) {
            fail(HPT_ERR_KERNEL, "row-split has no causal form");
        } else {
            if (p.vec == FULL && FULL > 1 && p.shift) launch_row_split<T, FULL, true>(p, a, st);
            else if (p.vec == FULL && FULL > 1) launch_row_split<T, FULL, false>(p, a, st);
            else launch_row_split<T, 1, false>(p, a, st);
        }
        return;
    }
    if (p.kind == NormKind::ColReg) {
        if constexpr (KIND == NORM_SOFTMAX || KIND == NORM_LOGSOFTMAX) {
            if (p.tall) {
                launch_col_tall<T>(p, a, st);
                return;
            }
            switch (p.vec) {
                case 1: launch_col_reg<T, 1>(p, a, st); break;
                case 2: if constexpr (FULL >= 2) launch_col_reg<T, 2>(p, a, st); break;
                case 4:
                    if constexpr (FULL == 4) {
                        if (p.nchunk == 32) launch_col_reg<T, 4, true>(p, a, st);
                        else launch_col_reg<T, 4>(p, a, st);
                    } else if constexpr (FULL > 4) {
                        launch_col_reg<T, 4>(p, a, st);
                    }
                    break;
                case 8: if constexpr (FULL >= 8) launch_col_reg<T, 8>(p, a, st); break;
                default: fail(HPT_ERR_KERNEL, "col-reg: unsupported vector width %d", p.vec);
            }
        } else {
            fail(HPT_ERR_KERNEL, "col-reg is a softmax plan");
        }
        return;
    }
    if (p.kind == NormKind::ColSplit) {
        if constexpr (KIND == NORM_SOFTMAX || KIND == NORM_LOGSOFTMAX) {
            if (p.vec == FULL && FULL > 1) launch_col_split<T, FULL>(p, a, st);
            else launch_col_split<T, 1>(p, a, st);
        } else {
            fail(HPT_ERR_KERNEL, "col-split is a softmax plan");
        }
        return;
    }
    if (p.kind == NormKind::TransposedTile || p.kind == NormKind::Transposed) {
        // the fused kinds run on the row kernels only (the caller demotes transposed plans)
        if constexpr (KIND > NORM_LAYERNORM) fail(HPT_ERR_KERNEL, "fused normalisation: no transposed kernel for this kind");
        else launch_transposed<T>(p, a, st);
        return;
    }
    if (p.kind == NormKind::RowReg && p.lds_rows) {
        // long rows that stay on chip: registers + LDS; the fused kinds stream
        if constexpr (FULL > 1 && sizeof(T) <= 4 && (KIND == NORM_SOFTMAX || KIND == NORM_LOGSOFTMAX)) {
            // 24 + 8 vectors of a four-byte type (16 + 8 of a two-byte type) per thread and 128 registers:
            // 256 or 512 threads; 48 + 16 (32 + 16) and 256 registers: 512 threads. Shifted four-byte rows:
            // 20 + 8 and 44 + 16.
            constexpr int kRegs = sizeof(T) == 4 ? 24 : 16;
            constexpr int kRegsShift = sizeof(T) == 4 ? 20 : 16;
            constexpr int kBigShift = sizeof(T) == 4 ? 44 : 32;
            if (!p.shift) {
                if (p.nchunk == kRegs + 8 && p.tpr == 256) {
                    row_lds_kernel<KIND, T, kRegs, 8, false, 256, 4><<<grid, dim3(256), 0, st>>>(a);
                    return;
                }
                if (p.nchunk == kRegs + 8 && p.tpr == 512) {
                    row_lds_kernel<KIND, T, kRegs, 8, false, 512, 4><<<grid, dim3(512), 0, st>>>(a);
                    return;
                }
                if (p.nchunk == kRegs + 8 && p.tpr == 1024) {
                    row_lds_kernel<KIND, T, kRegs, 8, false, 1024, 1><<<grid, dim3(1024), 0, st>>>(a);
                    return;
                }
                if (p.nchunk == 2 * kRegs + 16 && p.tpr == 512) {
                    row_lds_kernel<KIND, T, 2 * kRegs, 16, false, 512, 1><<<grid, dim3(512), 0, st>>>(a);
                    return;
                }
            } else {
                if (p.nchunk == kRegsShift + 8 && p.tpr == 256) {
                    row_lds_kernel<KIND, T, kRegsShift, 8, true, 256, 4><<<grid, dim3(256), 0, st>>>(a);
                    return;
                }
                if (p.nchunk == kRegsShift + 8 && p.tpr == 512) {
                    row_lds_kernel<KIND, T, kRegsShift, 8, true, 512, 4><<<grid, dim3(512), 0, st>>>(a);
                    return;
                }
                if (p.nchunk == kRegsShift + 8 && p.tpr == 1024) {
                    row_lds_kernel<KIND, T, kRegsShift, 8, true, 1024, 1><<<grid, dim3(1024), 0, st>>>(a);
                    return;
                }
                if (p.nchunk == kBigShift + 16 && p.tpr == 512) {
                    row_lds_kernel<KIND, T, kBigShift, 16, true, 512, 1><<<grid, dim3(512), 0, st>>>(a);
                    return;
                }
            }
            fail(HPT_ERR_KERNEL, "row_lds: no kernel for %d threads x %d vectors", p.tpr, p.nchunk);
        }
        if constexpr (FULL > 1) {
            // (the fused kinds stream such rows, a full workgroup per row)
            a.tpr = 1024;
            a.tpr_log2 = 10;
            if (p.shift) row_stream_kernel<KIND, T, FULL, true><<<grid, dim3(1024), 0, st>>>(a);
            else row_stream_kernel<KIND, T, FULL><<<grid, dim3(1024), 0, st>>>(a);
        }
        return;
    }
    if (p.kind == NormKind::RowReg && p.raw_rows) {
        // two-byte softmax rows of 98305 ... 131072 elements: the raw row in registers, sixteen vectors per
        // thread; the fused kinds stream
        if constexpr (sizeof(T) == 2 && (KIND == NORM_SOFTMAX || KIND == NORM_LOGSOFTMAX)) {
            if (grid.x > 512u) grid.x = 512u;
            row_raw_kernel<KIND, T, 16><<<grid, dim3(1024), 0, st>>>(a);
        } else {
            if (p.vec == FULL) row_stream_kernel<KIND, T, FULL><<<grid, block, 0, st>>>(a);
            else row_stream_kernel<KIND, T, 1><<<grid, block, 0, st>>>(a);
        }
        return;
    }
    if (p.kind == NormKind::RowReg && p.interleave != 1) {
        // (these kernels are compiled in a translation unit of their own)
        if constexpr (KIND == NORM_SOFTMAX || KIND == NORM_LOGSOFTMAX) launch_interleaved_rows<KIND, T>(p, a, grid, block, st);
        else fail(HPT_ERR_KERNEL, "interleaved rows are a softmax plan");
        return;
    }
    if (p.kind == NormKind::RowReg) {
        // Layernorm workgroups walk the rows (gamma / beta stay in registers);
        // softmax has nothing to reuse across rows and runs one row per group.
        if constexpr (FULL > 1 && KIND <= NORM_LAYERNORM) {
            if (p.tile_rows > 0) {
                a.rpb = p.tile_rows;
                a.tpr = 1;
                while (a.tpr < 64 && a.tpr * 8 < p.cols) a.tpr <<= 1;
                a.tpr_log2 = ilog2(a.tpr);
                // (the lanes' sweeps are unrolled to exactly the elements a lane of this row length has: rows of 257 take
                // 5 per lane of 64, and three more steps with every lane masked off cost a fifth of the launch)
                const dim3 tgrid((unsigned)((p.rows + p.tile_rows - 1) / p.tile_rows));
                switch ((int)((p.cols + a.tpr - 1) / a.tpr)) {
                    case 1: norm_tile_kernel<KIND, T, FULL, 1><<<tgrid, dim3(256), 0, st>>>(a); break;
                    case 2: norm_tile_kernel<KIND, T, FULL, 2><<<tgrid, dim3(256), 0, st>>>(a); break;
                    case 3: norm_tile_kernel<KIND, T, FULL, 3><<<tgrid, dim3(256), 0, st>>>(a); break;
                    case 4: norm_tile_kernel<KIND, T, FULL, 4><<<tgrid, dim3(256), 0, st>>>(a); break;
                    case 5: norm_tile_kernel<KIND, T, FULL, 5><<<tgrid, dim3(256), 0, st>>>(a); break;
                    case 6: norm_tile_kernel<KIND, T, FULL, 6><<<tgrid, dim3(256), 0, st>>>(a); break;
                    case 7: norm_tile_kernel<KIND, T, FULL, 7><<<tgrid, dim3(256), 0, st>>>(a); break;
                    case 8: norm_tile_kernel<KIND, T, FULL, 8><<<tgrid, dim3(256), 0, st>>>(a); break;
                    default: fail(HPT_ERR_KERNEL, "norm_tile: %d elements per lane", (int)((p.cols + a.tpr - 1) / a.tpr));
                }
                return;
            }
        }
        unsigned walkers = (unsigned)p.max_blocks;
        if constexpr (KIND == NORM_ADD_LAYERNORM && std::is_same<T, f16_t>::value) {
            // Three vectors per thread in 96 registers: five workgroups of 256 threads per compute unit and not four (bf16 takes 101), so
            // four rounds of them where every one still walks some rows (us, 3072 and this: [13107, 5120] 71.5 and 68.6, [20000, 3072] 64.5 and 61.7,
            // [52428, 1536] 82.8 and 79.8; of 5000 workgroups 30.4 and 33.6, 7000 40.3 and 40.3).
            if (p.gb_lds == 1 && p.nchunk == 3 && p.tpr < 512 && !p.shift && grid.x >= 7500) walkers = 5120;
        }
        if (norm_is_layer(KIND) && grid.x > walkers) grid.x = walkers;
        if constexpr (FULL > 1) {
            // Rows off the vector grid: as unaligned vectors, or as the aligned vectors that contain them.
            if (p.vec == FULL && p.ua_rows) {
                launch_row_unaligned<T>(p, a, grid, block, st);
                return;
            }
            if (p.vec == FULL && p.shift) {
                // shifted rows: a thread's gamma / beta fit every row it walks only if those rows share
                // their misalignment, i.e. the row step is a whole number of vectors
                if (norm_is_layer(KIND) && (int64_t)grid.x * p.rpb < p.rows) {
                    if (grid.x >= (unsigned)FULL) grid.x -= grid.x % FULL;
                    else fail(HPT_ERR_KERNEL, "row_reg: shifted rows need a row step of whole vectors");
                }
                // (the plan's numbers of vectors: layernorm rows while the masks fit beside them)
                if constexpr (sizeof(T) == 2 || (sizeof(T) == 4 && KIND == NORM_ADD_LAYERNORM)) fail(HPT_ERR_KERNEL, "row_reg: rows of this type and kind are unaligned vectors");
                else if constexpr (norm_is_layer(KIND)) launch_row_of<T, 1, true, false, false, 2, 3, 4>(p, a, grid, block, st);
                else launch_row_of<T, 1, true, false, false, 2, 3, 4, 5, 6, 7, 8>(p, a, grid, block, st);
                return;
            }
        }
        if constexpr (FULL > 1 && norm_is_layer(KIND)) {
            if (p.gb_lds == 2 && p.vec == FULL && p.sstride == 1 && !p.shift) {
                // gamma / beta from L2 in the last sweep: one row per group of threads, nothing carried between rows
                // (rows of 512 or 1024 threads: 512 workgroups walk the rows and prefetch)
                const bool pf = p.tpr >= 512 && KIND != NORM_ADD_LAYERNORM;
                if (pf && grid.x > 512u) grid.x = 512u;
#define HPT_L2GB_CASE(N)                                                                                  \
    case 2 * N: row_reg_kernel<KIND, T, FULL, N, 1, false, false, 2><<<grid, block, 0, st>>>(a); return; \
    case 2 * N + 1: row_reg_kernel<KIND, T, FULL, N, 1, false, true, 2><<<grid, block, 0, st>>>(a); return;
                if constexpr (sizeof(T) >= 4) {  // (two-byte rows of seven or eight vectors per thread spill: not planned)
                    switch (p.nchunk * 2 + (pf ? 1 : 0)) {
                        HPT_L2GB_CASE(7) HPT_L2GB_CASE(8)
                        default: break;
                    }
                }
                switch (p.nchunk * 2 + (pf ? 1 : 0)) {
                    HPT_L2GB_CASE(3) HPT_L2GB_CASE(4) HPT_L2GB_CASE(5) HPT_L2GB_CASE(6)
                    default: fail(HPT_ERR_KERNEL, "row_reg: unsupported chunk count %d with gamma / beta from L2", p.nchunk);
                }
#undef HPT_L2GB_CASE
            }
        }
        if constexpr (FULL > 1 && sizeof(T) == 2 && norm_is_layer(KIND)) {
            if (p.gb_lds == 1 && p.vec == FULL && p.sstride == 1 && !p.shift && p.nchunk >= 3 && p.nchunk <= 4) {
                const size_t smem = 2 * (size_t)p.cols * sizeof(T);
                if (p.tpr >= 512 && KIND != NORM_ADD_LAYERNORM) {
                    if (grid.x > 512u) grid.x = 512u;
                    if (p.nchunk == 3) row_reg_kernel<KIND, T, FULL, 3, 1, false, true, 1><<<grid, block, smem, st>>>(a);
                    else row_reg_kernel<KIND, T, FULL, 4, 1, false, true, 1><<<grid, block, smem, st>>>(a);
                } else {
                    if (p.nchunk == 3) row_reg_kernel<KIND, T, FULL, 3, 1, false, false, 1><<<grid, block, smem, st>>>(a);
                    else row_reg_kernel<KIND, T, FULL, 4, 1, false, false, 1><<<grid, block, smem, st>>>(a);
                }
                return;
            }
        }
        if constexpr (FULL > 1 && KIND != NORM_ADD_LAYERNORM) {
            // Long rows: 512 large workgroups that walk the rows and prefetch the next one. Measured
            // (TB/s, without -> with): f32 [3355, 10000] layernorm 3.6 -> 5.1, softmax 3.2 -> 4.2;
            // f32 [2048, 16384] 4.4 -> 5.2 / 4.1 -> 4.8; f16 [1024, 32768] softmax 3.9 -> 4.3. Two-byte
            // softmax rows of 512 threads are the exception (4.6 -> 4.2): they fit three to a compute
            // unit and do better one row per workgroup.
            if (p.vec == FULL && p.sstride == 1 && p.tpr >= 512 &&
                (sizeof(T) >= 4 || p.tpr == 1024 || norm_is_layer(KIND))) {
                if (grid.x > 512u) grid.x = 512u;
                launch_row_reg<T, FULL, 1, true>(p, a, grid, block, st);
                return;
            }
        }
        if constexpr (FULL > 1 && KIND != NORM_ADD_LAYERNORM) {
            // (every second element: the same walk, where a workgroup has more than one row. us, [:, ::2] of the stored, without and with: f32
            // of 1024 threads, or 512 with eight vectors, [1472, 15296] layernorm 36.2 and 34.5, causal 24.2 and 21.7, [2000, 10240] causal 19.9 and 17.6,
            // f16 layernorm [1000, 16384] 14.7 and 11.8, [4000, 8704] 28.1 and 25.5; but of 512 threads with four vectors, three of whose workgroups
            // fit a unit, f32 [3456, 8192] softmax 31.0 and 32.4, f64 layernorm [3456, 8192] 77.0 and 84.4, and f16 softmax [597, 14904] 7.7 and 8.2)
            if (p.vec == FULL && p.sstride == 2 && grid.x > 512u) {
                if constexpr (sizeof(T) == 4 && KIND == NORM_LAYERNORM) {
                    if (p.tpr == 1024) {
                        grid.x = 512u;
                        launch_row_of<T, 2, false, true, false, 4>(p, a, grid, block, st);
                        return;
                    }
                } else if constexpr (sizeof(T) == 4) {
                    if (p.tpr == 1024 || (p.tpr == 512 && p.nchunk == 8)) {
                        grid.x = 512u;
                        launch_row_of<T, 2, false, true, false, 4, 8>(p, a, grid, block, st);
                        return;
                    }
                } else if constexpr (sizeof(T) == 2 && KIND == NORM_LAYERNORM) {
                    if (p.tpr >= 512) {
                        grid.x = 512u;
                        launch_row_of<T, 2, false, true, false, 4>(p, a, grid, block, st);
                        return;
                    }
                }
            }
        }
        if (p.vec == FULL && p.sstride == 2 && FULL > 1) launch_row_reg<T, FULL, 2>(p, a, grid, block, st);
        else if (p.vec == FULL) launch_row_reg<T, FULL>(p, a, grid, block, st);
        else launch_row_reg<T, 1>(p, a, grid, block, st);
        return;
    }
    if constexpr (FULL > 1) {
        if (p.vec == FULL && p.shift) {
            row_stream_kernel<KIND, T, FULL, true><<<grid, block, 0, st>>>(a);
            return;
        }
    }
    if (p.vec == FULL) row_stream_kernel<KIND, T, FULL><<<grid, block, 0, st>>>(a);
    else row_stream_kernel<KIND, T, 1><<<grid, block, 0, st>>>(a);
}

// FloatBinaryType<TI> of the integer types (hpt-types/src/type_promote.rs)
template <class TI> struct PromotedOf { using type = f16_t; };  // bool, i8, i16, u8, u16
template <> struct PromotedOf<int32_t> { using type = float; };
template <> struct PromotedOf<uint32_t> { using type = float; };
template <> struct PromotedOf<int64_t> { using type = double; };
template <> struct PromotedOf<uint64_t> { using type = double; };

template <class TI> void launch_promoting_t(const NormPlan& p, NormArgs a, hipStream_t st) {
    using T = typename PromotedOf<TI>::type;
    constexpr int FULL = 16 / sizeof(T);
    if (p.kind == NormKind::Empty) return;
    if constexpr (KIND > NORM_LAYERNORM) {
        fail(HPT_ERR_DTYPE, "fused normalisation: the input must have a float dtype");
    } else {
        if (p.kind != NormKind::RowStream && p.kind != NormKind::Generic)
            fail(HPT_ERR_KERNEL, "promoted input: the plan was not restricted to the streaming row kernel");
        a.tpr = p.tpr;
        a.tpr_log2 = ilog2(p.tpr);
        a.rpb = p.rpb;
        a.inv_cols = 1.0 / (double)p.cols;
        const dim3 grid((unsigned)((p.rows + p.rpb - 1) / p.rpb));
        const dim3 block((unsigned)(p.tpr * p.rpb));
        if (p.vec == FULL && FULL > 1) row_stream_kernel<KIND, T, FULL, false, TI><<<grid, block, 0, st>>>(a);
        else row_stream_kernel<KIND, T, 1, false, TI><<<grid, block, 0, st>>>(a);
    }
}

}  // namespace

template <> NormLaunchFn norm_promoting_launcher<HPT_NORM_KIND>(int in_dtype) {
    switch (in_dtype) {
        case HPT_BOOL: return &launch_promoting_t<bool8>;
        case HPT_I8: return &launch_promoting_t<int8_t>;
        case HPT_I16: return &launch_promoting_t<int16_t>;
        case HPT_I32: return &launch_promoting_t<int32_t>;
        case HPT_I64: return &launch_promoting_t<int64_t>;
        case HPT_U8: return &launch_promoting_t<uint8_t>;
        case HPT_U16: return &launch_promoting_t<uint16_t>;
        case HPT_U32: return &launch_promoting_t<uint32_t>;
        case HPT_U64: return &launch_promoting_t<uint64_t>;
        default: return nullptr;
    }
}

template <> NormLaunchFn norm_launcher<HPT_NORM_KIND>(int dtype) {
    switch (dtype) {
        case HPT_F16: return &launch_t<f16_t>;
        case HPT_BF16: return &launch_t<bf16_t>;
        case HPT_F32: return &launch_t<float>;
        case HPT_F64: return &launch_t<double>;
        default: return nullptr;
    }
}

}  // namespace hpt
