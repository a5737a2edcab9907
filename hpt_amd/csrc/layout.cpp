// Host-side shape logic: axis normalisation, dimension coalescing and the
// choice of kernel family and launch shape for reductions and normalisations.
//
// The reference prepares a reduction by coalescing dims, grouping them by
// "reduced or kept" and permuting the reduced axes last
// (hpt/src/backends/cpu/utils/reduce/reduce_template.rs:165-253,
// hpt/src/backends/common/reduce.rs:44-96,
// hpt/src/backends/cpu/utils/reduce/reduce_utils.rs:23-56) and then splits on
// "does a reduced axis have stride 1" (hpt/src/backends/common/reduce.rs:24-33).
// The same preparation is done here, generalised to any strides: whichever
// group (kept or reduced) owns the smallest stride decides which way the lanes
// of a wavefront run, so that they always walk memory in address order.
#include <algorithm>
#include <cstring>

#include "common.hpp"

namespace hpt {

void process_axes(const int64_t* axes, int naxes, int ndim, int64_t* out) {
    for (int i = 0; i < naxes; ++i) {
        int64_t a = axes[i];
        for (int j = 0; j < i; ++j)
            if (axes[j] == a) fail(HPT_ERR_PARAM, "Axis %lld is duplicated", (long long)a);
        int64_t v = a < 0 ? a + ndim : a;
        if (ndim > 0 && (v < 0 || v >= ndim))
            fail(HPT_ERR_SHAPE, "Dimension out of range: expected in 0..%d, got %lld", ndim,
                 (long long)v);
        out[i] = v;
    }
    // Two spellings of one axis (-1 and ndim-1) are the same axis.
    for (int i = 0; i < naxes; ++i)
        for (int j = 0; j < i; ++j)
            if (out[j] == out[i]) fail(HPT_ERR_PARAM, "Axis %lld is duplicated", (long long)axes[i]);
}

int reduce_out_dtype(int op, int in) {
    if (in < 0 || in >= HPT_DTYPE_COUNT) fail(HPT_ERR_DTYPE, "invalid dtype %d", in);
    switch (op) {
        case HPT_SUM: case HPT_PROD: case HPT_MAX: case HPT_MIN: case HPT_NANSUM:
        case HPT_NANPROD: case HPT_REDUCEL1: case HPT_SUM_SQUARE:
            return in;
        case HPT_ALL: case HPT_ANY:
            return HPT_BOOL;
        case HPT_MEAN: case HPT_REDUCEL2: case HPT_REDUCEL3: case HPT_LOGSUMEXP:
            // FloatBinaryType<T>: hpt-types/src/promotion/normal_promote/_*.rs
            switch (in) {
                case HPT_BOOL: case HPT_I8: case HPT_I16: case HPT_U8: case HPT_U16: case HPT_F16:
                    return HPT_F16;
                case HPT_I32: case HPT_U32: case HPT_F32: return HPT_F32;
                case HPT_BF16: return HPT_BF16;
                default: return HPT_F64;
            }
        default:
            fail(HPT_ERR_PARAM, "invalid reduce op %d", op);
    }
}

static int64_t iabs(int64_t v) { return v < 0 ? -v : v; }

static int64_t pow2_floor(int64_t v) {
    int64_t p = 1;
    while (p <= v / 2) p *= 2;
    return p;
}
static int64_t pow2_ceil(int64_t v) {
    int64_t p = 1;
    while (p < v && p < ((int64_t)1 << 62)) p *= 2;
    return p;
}

// Append (size, stride) to `d`, merging with the previous entry when the two
// are one dense run: prev.stride == stride * size.
static void push_merged(Dims& d, int64_t size, int64_t stride) {
    if (size == 1) return;
    if (d.n > 0 && d.stride[d.n - 1] == stride * size) {
        d.size[d.n - 1] *= size;
        d.stride[d.n - 1] = stride;
        return;
    }
    if (d.n == kMaxDims)
        fail(HPT_ERR_SHAPE, "view has more than %d non-mergeable dims in one group", kMaxDims);
    d.size[d.n] = size;
    d.stride[d.n] = stride;
    ++d.n;
}

// Largest power-of-two vector width (in elements, at most 16 bytes) that every
// access of the form data + sum(idx_i * stride_i) + inner*1 can use: the base
// address, every other stride and the inner length must be multiples of it.
// Kernels are built for two widths only: the full 16-byte vector or one element.
static int legal_vec(const void* data, size_t elem_size, int64_t inner_len, const Dims& a,
                     const Dims& b, int skip_a_last, int skip_b_last) {
    const int v = (int)(16 / elem_size);
    if (v <= 1) return 1;
    bool ok = ((uintptr_t)data % 16) == 0 && inner_len % v == 0;
    for (int i = 0; ok && i < a.n - skip_a_last; ++i) ok = a.stride[i] % v == 0;
    for (int i = 0; ok && i < b.n - skip_b_last; ++i) ok = b.stride[i] % v == 0;
    return ok ? v : 1;
}

// How many blocks of 256 threads keep an MI355X busy: 256 CUs, each able to
// hold 8 such blocks.
constexpr int64_t kBlocksToFill = 2048;
constexpr int64_t kComputeUnits = 256;  // MI355X

// Slices of the reduced range for `groups` workgroups that share it: the count that fills one, two ... `most` rounds of
// compute units to nine tenths, or the one that comes closest.
static int64_t full_rounds(int64_t groups, int64_t most = 4) {
    int64_t best = 1;
    double best_fill = 0;
    for (int64_t r = 1; r <= most; ++r) {
        const int64_t S = r * kComputeUnits / groups;
        const double fill = (double)(S * groups) / (double)(r * kComputeUnits);
        if (S >= 1 && fill > best_fill) {
            best = S;
            best_fill = fill;
        }
        if (fill >= 0.9) break;
    }
    return best;
}

// Column reductions below this take the plans for small inputs; the partials of those that are split stay below
// the second figure.
constexpr int64_t kSmallColBytes = 8ll << 20;
constexpr size_t kSmallColScratch = 1u << 20;
// Accumulators of a column workgroup's threads, in bytes: more of them take longer to fold than their loads save (argmax of one-byte types, sixteen of eight bytes per
// thread, over axis 0, us, this and twice as many: u8 [2628, 53] 12.0 and 13.7, [1283, 54] 9.6 and 11.7, [300, 20000] 7.9 and 8.5, [2208, 103] 10.8 and 14.9).
constexpr size_t kColAccs = 64u << 10;

ReducePlan plan_reduce(const void* data, const int64_t* shape, const int64_t* strides, int ndim,
                       const int64_t* axes, int naxes, size_t elem_size, size_t acc_size, bool heavy, bool spare_scratch) {
    ReducePlan p;
    bool is_red[kMaxRank] = {};
    for (int i = 0; i < naxes; ++i) is_red[axes[i]] = true;

    p.K = 1;
    p.R = 1;
    for (int i = 0; i < ndim; ++i) (is_red[i] ? p.R : p.K) *= shape[i];
    if (p.K == 0) {
        p.kind = ReduceKind::Empty;
        return p;
    }
    if (p.R == 0) {
        p.kind = ReduceKind::Identity;
        return p;
    }

    // kept dims keep their logical order (the output is contiguous in it)
    for (int i = 0; i < ndim; ++i)
        if (!is_red[i]) push_merged(p.kept, shape[i], strides[i]);
    // reduced dims may be visited in any order: sort by |stride| descending
    int order[kMaxRank], nr = 0;
    for (int i = 0; i < ndim; ++i)
        if (is_red[i] && shape[i] != 1) order[nr++] = i;
    std::stable_sort(order, order + nr,
                     [&](int a, int b) { return iabs(strides[a]) > iabs(strides[b]); });
    for (int i = 0; i < nr; ++i) push_merged(p.red, shape[order[i]], strides[order[i]]);

    int64_t sr = p.red.n ? iabs(p.red.stride[p.red.n - 1]) : INT64_MAX;
    int64_t sk = p.kept.n ? iabs(p.kept.stride[p.kept.n - 1]) : INT64_MAX;

    // the lean kernels index with 32-bit integers and form sums of two such values
    // (chunk starts plus chunk lengths, positions plus batch steps): stay below 2^30
    const int64_t kI32 = 1 << 30;
    if (p.red.n > 0 && (p.kept.n == 0 || sr <= sk)) {
        // ---- Row: lanes walk the reduced index space ---------------------
        p.kind = ReduceKind::Row;
        int64_t rin = p.red.size[p.red.n - 1];
        p.vec = 1;
        if (p.red.stride[p.red.n - 1] == 1)
            p.vec = legal_vec(data, elem_size, rin, p.kept, p.red, 0, 1);
        p.lean = p.red.n == 1 && p.kept.n <= 1 && p.K <= kI32 && rin <= kI32 &&
                 iabs(p.red.stride[0]) <= kI32;
        if (p.lean && p.red.stride[0] == 2 && elem_size <= 8 &&
            legal_vec(data, elem_size, rin * 2, p.kept, p.red, 0, 1) > 1) {
            // every second element along the row: full vectors, even positions kept
            p.vec = (int)(16 / elem_size);
            p.sstride = 2;
        }
        const int full = (int)(16 / elem_size);
        if (p.lean && p.kept.n == 1 && p.sstride == 1 && full > 1 && p.red.stride[0] == 1 && p.kept.stride[0] == rin &&
            (uintptr_t)data % 16 == 0 && rin * (int64_t)elem_size <= (rin % full == 0 ? 512 : 4096) && p.K * rin * (int64_t)elem_size >= (4ll << 20)) {
            // Short rows laid back to back ([N, 3], [N, 33], [N, 100]): a lane per row (or a few) reads
            // 4..12-byte pieces at a stride. Instead a workgroup brings 16 KiB of consecutive rows into
            // LDS with aligned 128-bit loads, whatever the row length, and the rows are summed from there.
            // Rows of whole vectors gain up to 512 bytes (f32 [N, 100]: 3.4 -> 5.9 TB/s; from 2 KiB on the
            // direct kernel is as fast or faster), other rows up to 4 KiB (f32 [N, 257]: 3.3 -> 5.5).
            const int64_t tile_bytes = 16 << 10;
            int64_t rows = tile_bytes / (rin * (int64_t)elem_size);
            rows -= rows % full;  // tiles start on 16-byte boundaries
            if (rows >= full) {
                p.row_tile = (int)rows;
                p.vec = full;
                p.tpr = (int)std::min<int64_t>(64, pow2_ceil((rin + 7) / 8));
                p.rpb = 256 / p.tpr;
                p.split = p.split_q = p.split_i = 1;
                return p;
            }
        }
        if (p.lean && p.vec == 1 && full > 1 && p.sstride == 1 && p.red.stride[0] == 1 && rin >= 64 * full &&
            (uintptr_t)data % elem_size == 0) {
            // Long contiguous rows whose length, pitch or base is off the 16-byte grid (the sum of a
            // whole array of odd length): the kernel peels each row's first elements up to a 16-byte
            // boundary and its last ones, and reads everything between as aligned vectors.
            p.ragged = true;
            p.vec = full;
        }
        if (p.vec == 1 && full > 1 && p.sstride == 1 && p.red.stride[p.red.n - 1] == 1 && rin >= full &&
            (uintptr_t)data % elem_size == 0) {
            // Shorter contiguous runs off the grid (the batch-norm sums of [N, C, 7, 7]: runs of 49):
            // unaligned 128-bit loads from the run's start on, the last one taken from the run's end.
            p.unaligned = true;
            p.vec = full;
        }
        int64_t nv = p.unaligned ? (p.R / rin) * ((rin + full - 1) / full) : p.R / (p.vec / p.sstride);  // vector loads per output
        // About 8 vector loads per lane; groups of one or two wavefronts per row
        // stream best (each wavefront walks its own long run of the row), and
        // only very long rows get a whole workgroup.
        p.tpr = (int)std::min<int64_t>(128, pow2_ceil((nv + 7) / 8));
        if (nv >= 128 * 64) p.tpr = nv >= 1024 * 32 ? 1024 : 256;
        // from four loads per thread on a whole workgroup per row streams a little better than half of
        // one (f16 [4096, 8192] rows: 12.2 -> 11.8 us); rows with peeled ends are better off with fewer
        // lanes idling through the ends
        else if (nv >= 256 * 4 && !p.ragged) p.tpr = 256;
        int block = std::max(256, p.tpr);
        p.rpb = block / p.tpr;
        int64_t blocks = (p.K + p.rpb - 1) / p.rpb;
        p.split = p.split_q = p.split_i = 1;
        if (blocks < kBlocksToFill / 4) {
            // Too few outputs to fill the chip: a whole workgroup per output when that leaves
            // each thread 8 loads or more, then several workgroups of 256 threads
            // per output, each with a long contiguous share (>= 16 loads per
            // thread, 8 when there are many outputs to amortise the second stage over); about
            // 512 workgroups in all is the measured sweet spot.
            if (p.tpr < 256 && nv >= 256 * 8) {
                p.tpr = 256;
                p.rpb = 1;
            }
            // What is small keeps to one launch, up to 1024 threads per output with four vectors each or more: the second launch costs what
            // sixteen vectors per thread do (us per call in two launches of 256 threads and in one: argmax of f32 [1, 37568] 10.8 and 7.4, bf16 [10, 116377] 10.9 and
            // 7.3, sum of all of f32 [4, 104, 12, 12] 10.7 and 7.6; device us of one launch, 256 and 1024 threads: bf16 [28, 46592] argmax 7.3 and
            // 4.9, f32 [40, 28, 26, 26] over all but the channels 11.4 and 6.8).
            // (Half as many of one-byte argmin / argmax, whose sixteen elements per vector take longer than their load: u8 [131072] 7.9 and 7.2, [204894] 8.0 and 10.2,
            // [262128] 8.3 and 12.8; without scratch to spare they stay in one.)
            const bool small = nv <= 16 * 1024 && p.K * nv * 16 <= (4ll << 20);
            p.small_split = small && nv > 8 * 1024 && elem_size == 1 && acc_size >= 8 && spare_scratch;
            if (small && !p.small_split) {
                // Not where the first lanes of a row would have four vectors and most of the others three: a wavefront then goes through whole batches and
                // remainder, twice the instructions to fetch (device us, eight and four per thread: argmax of u8 [30, 3200] 3.1 and 5.6, f32 [30, 800] 2.3 and 3.2; from
                // 3.5 of them on eight are uneven too, bf16 [30, 960] 2.4 and 2.3). Nor where up to four workgroups would become more, on XCDs that have yet to
                // fetch all of it: sum of f32 [200, 68] 1.9 and 2.3, [30, 1024] 1.9 and 2.5. (From 1024 vectors on what is in flight counts for more.)
                const int t4 = (int)std::min<int64_t>(1024, pow2_ceil((nv + 3) / 4));
                const int rpb4 = std::max(256, t4) / t4;
                const bool uneven = nv > 3 * t4 && 2 * nv <= 7 * t4, spread = blocks <= 4 && (p.K + rpb4 - 1) / rpb4 > 4;
                if (nv >= 1024 || (!uneven && !spread)) p.tpr = std::max(p.tpr, t4);
                p.rpb = std::max(256, p.tpr) / p.tpr;
                return p;
            }
            int64_t want = std::max<int64_t>(1, 512 / p.K);  // (never just over two rounds of the compute units)
            int64_t can = nv / (256 * (p.K >= 64 ? 8 : 16));
            int64_t split = std::min<int64_t>(std::min(want, can), 4096);
            if (split > 1) {
                p.tpr = 256;
                p.rpb = 1;
                int64_t rout = p.R / rin;
                int64_t sq = std::min(split, rout);
                int64_t si = std::max<int64_t>(1, split / sq);
                int64_t can_i = std::max<int64_t>(1, (rin / (p.vec / p.sstride)) / p.tpr);
                si = std::min(si, can_i);
                p.split_q = (int)sq;
                p.split_i = (int)si;
                p.split = (int)(sq * si);
            }
        }
    } else {
        // ---- Col: lanes walk the outputs -----------------------------------
        p.kind = ReduceKind::Col;
        const int nk = p.kept.n;
        // A reduction over the MIDDLE axis of a contiguous [B, C, L] whose inner dim divides the 16-byte vector (L = 2
        // or 4 four-byte elements; 2, 4 or 8 two-byte ones): the [C, L] slab is one ROW of C * L elements for the lean
        // row kernel, an element's place in its vector names its output, and a thread keeps L accumulators. Lanes
        // along L would idle, and the flat walk takes two launches.
        {
            const int64_t full = elem_size <= 16 ? (int64_t)(16 / elem_size) : 1;
            if (nk == 2 && p.red.n == 1 && full > 1 && p.kept.stride[1] == 1 && p.kept.size[1] > 1 && p.kept.size[1] <= 8 && full % p.kept.size[1] == 0 &&
                p.red.stride[0] == p.kept.size[1] && p.kept.stride[0] == p.R * p.kept.size[1] && p.R > 64 &&
                (p.R * p.kept.size[1]) % full == 0 && p.R * p.kept.size[1] * (int64_t)elem_size <= (128 << 10) &&
                p.kept.size[0] >= 256 && p.K * p.R * (int64_t)elem_size >= (4ll << 20) && ((uintptr_t)data & 15) == 0) {
                const int64_t L = p.kept.size[1];
                const int64_t shp[2] = {p.kept.size[0], p.R * L}, str[2] = {p.R * L, 1}, ax[1] = {1};
                ReducePlan q = plan_reduce(data, shp, str, 2, ax, 1, elem_size, acc_size, heavy, spare_scratch);
                if (q.kind == ReduceKind::Row && q.lean && q.vec == full && !q.ragged && !q.unaligned && q.sstride == 1 &&
                    q.split == 1 && !q.row_tile) {
                    q.interleave = (int)L;
                    q.K = p.K;
                    q.R = p.R;
                    q.kept = p.kept;
                    q.red = p.red;
                    return q;
                }
            }
        }
        // Two kept dims of which the FIRST is the contiguous one (a reduction over the last axis of a
        // permuted view): the lanes must run along that one. List it last; the kernel then scatters
        // its (few) outputs instead of gathering its (many) inputs.
        if (nk == 2 && p.red.n <= 1 && iabs(p.kept.stride[0]) < iabs(p.kept.stride[1]) && p.kept.size[1] <= 65535 &&
            p.kept.size[0] <= kI32 && p.R <= kI32 && iabs(p.kept.stride[0]) <= kI32) {
            std::swap(p.kept.size[0], p.kept.size[1]);
            std::swap(p.kept.stride[0], p.kept.stride[1]);
            p.kept_swapped = true;
        }
        // The same slabs with an inner dim of 3, 5, 6 or 7 elements (points, colours): a row of the kernel whose
        // lanes, in multiples of L, keep an accumulator per vector place. Mid-sized slabs, many of them: groups up to
        // 2 KiB go through LDS tiles (f32 [30000, 100, 3] 9.1 us there against 13.5 here; above, against the flat walk,
        // [20000, 200, 3] 23.1 -> 12.4), few long ones through the flat walk.
        {
            const int64_t full = elem_size <= 8 ? (int64_t)(16 / elem_size) : 1;
            const int64_t L = nk == 2 ? p.kept.size[1] : 0;
            if (nk == 2 && !p.kept_swapped && p.red.n == 1 && full > 1 && p.kept.stride[1] == 1 && L >= 3 && L <= 7 && full % L != 0 &&
                p.red.stride[0] == L && p.kept.stride[0] == p.R * L && p.R * L * (int64_t)elem_size > 2048 &&
                p.R * L * (int64_t)elem_size <= (256 << 10) && p.kept.size[0] >= 512 &&
                p.K * p.R * (int64_t)elem_size >= (4ll << 20) && ((uintptr_t)data % elem_size) == 0) {
                p.kind = ReduceKind::Row;
                p.mod_rows = (int)L;
                p.vec = (int)full;
                p.tpr = p.R * L / full >= 1024 ? 256 : 64;
                p.rpb = 256 / p.tpr;
                return p;
            }
        }
        int64_t kin = nk ? p.kept.size[nk - 1] : 1;
        p.vec = 1;
        if (nk && p.kept.stride[nk - 1] == 1)
            p.vec = legal_vec(data, elem_size, kin, p.kept, p.red, 1, 0);
        const int64_t outer = nk > 1 ? p.kept.size[0] : 1;
        p.lean = p.red.n <= 1 && nk <= 2 && outer <= 65535 && kin <= kI32 && p.R <= kI32 &&
                 (nk == 0 || iabs(p.kept.stride[nk - 1]) <= kI32);
        if (p.kept_swapped && !p.lean) {  // the general kernel numbers its outputs in kept order: undo
            std::swap(p.kept.size[0], p.kept.size[1]);
            std::swap(p.kept.stride[0], p.kept.stride[1]);
            p.kept_swapped = false;
            kin = p.kept.size[nk - 1];
            p.vec = 1;
            if (p.kept.stride[nk - 1] == 1) p.vec = legal_vec(data, elem_size, kin, p.kept, p.red, 1, 0);
        }
        if (p.lean && nk && p.kept.stride[nk - 1] == 2 && elem_size <= 8 &&
            legal_vec(data, elem_size, kin * 2, p.kept, p.red, 1, 0) > 1) {
            // neighbouring outputs sit at every second position: full vectors, even positions kept
            p.vec = (int)(16 / elem_size);
            p.sstride = 2;
        }
        const int full = (int)(16 / elem_size);
        {
            // Small groups laid back to back ([outer, R, kin] with R * kin elements of at most 2 KiB and
            // rows of kin shorter than a wavefront of vectors): 16 KiB tiles of whole groups through LDS.
            const int64_t G = p.R * kin;
            if (nk == 2 && !p.kept_swapped && p.red.n == 1 && full > 1 && p.sstride == 1 && p.kept.stride[1] == 1 &&
                p.red.stride[0] == kin && p.kept.stride[0] == G && (uintptr_t)data % 16 == 0 &&
                G * (int64_t)elem_size <= 2048 && kin * (int64_t)elem_size < 1024 && p.R >= 2 && p.R <= 256 &&
                p.K * p.R * (int64_t)elem_size >= (4ll << 20) && p.kept.size[0] >= 1024) {
                int64_t groups = (16 << 10) / (G * (int64_t)elem_size);
                groups -= groups % full;  // tiles start on 16-byte boundaries
                if (groups >= full) {
                    p.group_tile = (int)groups;
                    p.vec = full;
                    p.lean = true;
                    p.split = 1;
                    p.bx = 256;
                    p.by = 1;
                    p.chunk = 0;
                    return p;
                }
            }
        }
        if (p.lean && nk && !p.kept_swapped && p.vec < full && p.sstride == 1 && full > 1 && p.kept.stride[nk - 1] == 1 &&
            p.red.n == 1 && p.red.stride[0] == kin && (uintptr_t)data % elem_size == 0 &&
            outer * kin * p.R * (int64_t)elem_size >= (8ll << 20)) {
            // (slabs that start off 16-byte boundaries take the same vectors unaligned)
            const bool slabs_aligned = (uintptr_t)data % 16 == 0 && (outer == 1 || p.kept.stride[0] % full == 0);
            // A contiguous [R, kin] slab whose rows are not whole vectors (kin = 3, 33, 257): walk it
            // as a FLAT array of aligned vectors. With a stride between a thread's visits that is a
            // multiple of kin, every vector slot of every thread stays on one column.
            int64_t g = kin, b = full;
            while (b) { int64_t t = g % b; g = b; b = t; }
            const int64_t kp = kin / g;  // threads per period: kp * full elements = full rows
            int64_t tmax = std::min<int64_t>(1024, (int64_t)((64u << 10) / ((size_t)full * acc_size)));
            // (each slab must be worth at least two periods of the walk: small slabs, of which there are
            // many, take fewer threads each)
            tmax = std::min(tmax, kin * p.R / (2 * full));
            if (kp <= tmax && tmax >= 64) {
                p.flat_t = (int)(kp * (tmax / kp));
                p.vec = full;
                p.unaligned = !slabs_aligned;
                const int64_t per_iter = (int64_t)p.flat_t * full;
                const int64_t iters = (kin * p.R + per_iter - 1) / per_iter;
                int64_t cap = std::max<int64_t>(1, (int64_t)((64ll << 20) / acc_size) / p.K);
                // one large workgroup per compute unit measured best (256: 4.4 TB/s, 512: 3.8, 128: 3.7)
                int64_t split = std::min<int64_t>(iters / 4, std::max<int64_t>(1, 256 / outer));
                p.split = (int)std::max<int64_t>(1, std::min(split, cap));
                p.bx = (p.flat_t + 63) / 64 * 64;
                p.by = 1;
                p.chunk = 0;
                return p;
            }
            // Wider rows (kin = 4097, 50257): a period of full / g rows spans several workgroups; every
            // vector slot is one (row phase, column) pair, so no fold inside the workgroup is needed and
            // the partials are [slice][phase][K].
            const int64_t phases = full / g;
            // (Shorter elements, whose periods are eight rows and more, are faster as unaligned columns, below, where those take
            // them: us, sum over axis 0, f16 [8190, 4097] 21.9 and 16.4, [2700, 5001] 19.1 and 10.8; [16, 512, 4097] over axis 1 22.5 and 19.0.)
            const int64_t xb = (kp + 1023) / 1024;
            if (slabs_aligned && kp > tmax && p.R >= 16 * phases && xb <= 65535 && kin * phases <= kI32 && (elem_size >= 4 || p.R < 256)) {
                p.flat_t = (int)(((kp + xb - 1) / xb + 63) / 64 * 64);
                p.flat_xb = (int)xb;
                p.flat_phases = (int)phases;
                p.vec = full;
                const int64_t periods = p.R / phases;
                int64_t cap = std::max<int64_t>(1, (int64_t)((64ll << 20) / acc_size) / (p.K * phases));
                int64_t slices = std::min<int64_t>(periods / 4, std::max<int64_t>(1, 256 / (outer * xb)));
                slices = std::max<int64_t>(1, std::min(slices, cap));
                p.split = (int)(slices * phases);
                // One slab of four-byte elements and more is launched in workgroups of 256 threads (rows of more than 128 of them:
                // 512), one per compute unit, which leave fewer partials than the plan has room for (scratch is sized, and refused,
                // by `split`): a thousand threads each left a fifth of the units idle at xb = 5, and most of the fold was partials. Us,
                // sum over axis 0: f32 [8190, 4097] 31.2 -> 26.2, [4097, 8190] 31.1 -> 25.2, [2700, 5001] 19.8 -> 14.5, [700, 50257] the same.
                // Several slabs keep the large ones (i32 [12, 128, 4225] over axis 1 11.2, 12.2 in small ones).
                if (outer == 1 && elem_size >= 4) {
                    p.flat_w = (kp + 255) / 256 > 128 ? 512 : 256;
                    p.flat_slices = (int)std::min(slices, full_rounds((kp + p.flat_w - 1) / p.flat_w));
                }
                p.bx = p.flat_t;
                p.by = 1;
                p.chunk = 0;
                return p;
            }
        }
        // Rows that are not whole, aligned vectors (an odd inner length, a base or pitch off 16 bytes):
        // a lane still takes `full` neighbouring outputs, with unaligned 128-bit loads (global memory
        // takes them; now and then one touches two lines) instead of one element at a time - eight
        // times the bytes in flight per lane for f16. The last lane of a row takes its vector from the row's end
        // backwards, so a row holds one at least (kin >= full).
        // (Worth it when a row is a few wavefronts of such lanes and enough is reduced into each output
        // that the lane's outputs, which it then writes one by one, are a small part of the traffic.)
        const int64_t bytes = p.K * p.R * (int64_t)elem_size;
        const bool small = p.lean && bytes < kSmallColBytes;
        const bool ua_ok = p.lean && nk && p.vec == 1 && p.sstride == 1 && full > 1 && p.kept.stride[nk - 1] == 1 && (uintptr_t)data % elem_size == 0;
        int64_t kv = 0, xblocks = 0;  // vector columns the lanes spread over, column blocks
        auto columns = [&](bool ua) {
            p.unaligned = ua;
            if (ua) p.vec = full;
            kv = ((p.lean ? kin : p.K) + (ua ? full - 1 : 0)) / (p.vec / p.sstride);
            p.bx = (int)std::min<int64_t>(64, pow2_ceil(kv));
            // A row of vector columns that is not a whole number of wavefronts (96: hidden size 768 in two-byte
            // elements) would leave the last wavefront of every row partly idle: narrower column blocks
            // (32 or 16 lanes, two or four reduced positions per wavefront) that divide it better.
            // Over axis 1, TB/s: f16 [128, 512, 1280] 4.7 -> 6.1, [512, 197, 768] 5.0 -> 5.7, f32 [256, 512, 320] 5.0 -> 6.2.
            if (kv > 64) {
                auto waste = [&](int64_t b) { return (kv + b - 1) / b * b - kv; };
                for (int b = 32; b >= 16; b >>= 1)
                    if (waste(p.bx) * 8 > kv && waste(b) < waste(p.bx)) p.bx = b;
            }
            xblocks = (kv + p.bx - 1) / p.bx * (p.lean ? outer : 1);
        };
        // One wavefront per 64 vector columns streams best when there are enough
        // columns (measured: 832 wavefronts with 128 loads each reach 5.9 TB/s);
        // with fewer, thread rows and then workgroups split the reduced range:
        // r-partitions so that about 768 wavefronts run, each with >= 16 loads.
        const int64_t kWavesWanted = 768;
        auto need_of = [&]() { return (kWavesWanted + xblocks - 1) / xblocks; };
        const int64_t can = std::max<int64_t>(1, p.R / 16);
        // One launch, thread rows meet in LDS: a workgroup is at least one wavefront.
        auto rows_in_one_launch = [&]() {
            const int64_t base = 64 / p.bx, rp = std::min(need_of(), can);
            if (rp <= 1) return base;
            int64_t by = std::min<int64_t>(pow2_ceil(rp), 1024 / p.bx / base) * base;
            while (by > base && p.bx * by * (p.vec / p.sstride) * acc_size > kColAccs) by /= 2;
            return by;
        };
        columns(ua_ok && kin >= 256 && p.R >= 256);
        if (small) {
            // Below 8 MiB the time is the chain of dependent batches of loads of one lane, and the compute units that
            // stand idle: 16-lane column blocks (256-byte segments of each row) make more workgroups of them, and up
            // to 1024 threads share a block's rows. Where that still leaves a lane more than 24 rows (three batches of
            // eight loads; a second launch costs as much: f32 [1216, 225], 19 rows, 6.4 us in one launch, 7.3 in two, in cache;
            // 48 single elements, [7482, 3] 5.3 and 7.1, [10304, 4] 5.8 and 7.2),
            // the rows are dealt over workgroups too, about 12 to a lane. Over axis 0, us before -> now:
            // f32 [12608, 128] 109 -> 8.3 (in one launch 33.9), f16 [2315, 363] 197 -> 8.8 (16.1), f32 [5440, 45] 28.3 -> 7.3
            // (15.5), bf16 [34112, 40] 57 -> 8.2. (Device time of both launches.)
            // Where the plan above already leaves a lane few rows with less than 1024 threads to fold, the narrower blocks
            // only add to the fold: it stays from 4 (fewer mean more threads than the rows need) to 12 rows of vectors or 20 of
            // single elements per lane, and single elements become unaligned vectors, from two lanes per row on, beyond 24
            // (us, as was and in narrow blocks: f64 [9, 3008] 2.7 and 3.6, i32 [33, 118] 2.3 and 3.5, u8 [136, 3096] 3.8 and 5.8, f32
            // [960, 199] 5.4 and 7.0; but f32 [676, 120], 21 rows, 9.8 and 7.6, [176, 4992], 11 rows by 1024 threads, 6.8 and
            // 5.7, i32 [187, 8], one row, 3.7 and 2.6).
            if (!p.unaligned) {
                const int64_t by = rows_in_one_launch(), rows = (p.R + by - 1) / by;
                if (ua_ok && kin >= 2 * full && p.R >= 64 && rows > 24) {
                    columns(true);
                } else if (p.bx * by < 1024 && rows >= 4 && rows <= (p.vec > 1 ? 12 : 20)) {
                    p.by = (int)by;
                    p.split = 1;
                    p.chunk = p.R;
                    return p;
                }
            }
            // (Eight lanes, a line of each row, and 128 thread rows where 64 would leave a lane more than twelve rows: up to 2048 of them stay in
            // one launch. Over axis 0, us per call, sixteen lanes and eight: f16 [1536, 1000] 11.1 and 7.9, [1021, 3001] 10.2 and 7.4, bf16 [1344, 2368] 9.1 and
            // 7.6, f32 [1400, 900] every second 11.4 and 7.7; in two launches and in one [2040, 384] 9.6 and 8.8, [1800, 1001] 9.6 and 7.8. Longer columns are more than one
            // compute unit brings in: f32 [2100, 900] 10.9 and 11.1, f16 [3000, 1200] every second 11.0 and 14.6. Beyond 1536 rows so are inputs of more than
            // 7 MiB (f16 [2040, 2000] 10.9 and 11.4), whole vectors of rows that do not start on cache lines, which a block reads as two half lines each (f32 [1800, 300] 9.5 and 10.2,
            // [2040, 700] 9.8 and 12.3, [2040, 900] every second 9.8 and 12.3, bf16 [2040, 1800] 9.5 and 12.6), and accumulators of eight bytes that fill 64 KiB (argmax of f16 [2040, 1024] 10.2 and 11.6).
            // The accumulators of one-byte argmin / argmax allow 64 thread rows, so eight lanes up to 1024 rows: u8, argmax, sixteen and eight: [850, 1152] 10.4 and
            // 8.5, [1000, 256] 9.6 and 8.5; [1200, 900] 11.0 and 14.6, [1600, 397] 10.7 and 13.9, [1821, 144] 10.1 and 14.1.
            const size_t lane_accs = (p.vec / p.sstride) * acc_size;
            const bool off_lines = !p.unaligned && (((uintptr_t)data | (uintptr_t)(p.red.stride[0] * (int64_t)elem_size)) & 127) != 0;
            const int64_t most8 = std::min<int64_t>(16 * std::min<int64_t>(128, kColAccs / (8 * lane_accs)),
                                                    bytes > (7ll << 20) || off_lines || (acc_size >= 8 && 1024 * lane_accs >= kColAccs) ? 1536 : 2048);
            const bool eight = p.vec > 1 && p.R > 768 && p.R <= most8;
            while (p.bx > (eight ? 8 : 16) && xblocks < kComputeUnits && p.R >= 32) {
                p.bx /= 2;
                xblocks = (kv + p.bx - 1) / p.bx * outer;
            }
            const int rows_per_wave = 64 / p.bx, uv = p.vec / p.sstride;
            int64_t by = pow2_ceil((p.R + 7) / 8);
            by = std::min(by, rows_per_wave * pow2_ceil((2048 + xblocks - 1) / xblocks));
            by = std::max<int64_t>(rows_per_wave, std::min<int64_t>(by, 1024 / p.bx));
            while (by > rows_per_wave && p.bx * by * uv * acc_size > kColAccs) by /= 2;
            p.by = (int)by;
            p.split = 1;
            if ((p.R + by - 1) / by > (p.vec > 1 ? 24 : 48) && spare_scratch) {
                // workgroups of 256 threads: the more rows share a workgroup, the longer its fold through LDS
                const int64_t sby = std::min<int64_t>(by, std::max(rows_per_wave, 256 / p.bx));
                const int64_t cap = (int64_t)(kSmallColScratch / acc_size) / p.K;
                const int64_t split = std::min({(p.R + sby * 12 - 1) / (sby * 12), (1024 + xblocks - 1) / xblocks, cap});
                if (split * sby > 2 * by) {
                    p.by = (int)sby;
                    p.split = (int)split;
                    p.small_split = true;
                }
            }
            p.chunk = (p.R + p.split - 1) / p.split;
            return p;
        }
        const int base_by = 64 / p.bx;  // a workgroup is at least one wavefront
        const int uv = p.vec / p.sstride;
        p.by = base_by;
        p.split = 1;
        const int64_t need = need_of(), rp = std::min(need, can);
        if (rp > 1) {
            if (bytes >= kSmallColBytes) {
                // Large input: partition over WORKGROUPS first, so that the partitions land
                // on different CUs (48 workgroups of 1024 threads leave 208 CUs idle), and
                // fold the partials in a second launch.
                int64_t cap = std::max<int64_t>(1, (int64_t)((64ll << 20) / acc_size) / p.K);
                if (need > 64) {
                    // Very few column blocks (a narrow inner dim: [N, 3], [N, 33]): aim for ~2048
                    // wavefronts, eight per workgroup (measured best: [32768, 1024] f32 4.7 TB/s with sixteen, 5.3
                    // with eight), up to 256 workgroups per column block.
                    const int64_t slices = std::min((2048 + xblocks - 1) / xblocks, can);
                    int64_t by_waves = std::min<int64_t>(8, pow2_floor(slices));
                    while (by_waves > 1 && 64 * by_waves * uv * acc_size > kColAccs) by_waves /= 2;
                    p.split = (int)std::min<int64_t>(std::min<int64_t>((slices + by_waves - 1) / by_waves, 256), cap);
                    p.by = (int)by_waves * base_by;
                } else {
                    // A power of two of partitions (an even share of a power-of-two axis: whole batches
                    // of eight loads, nobody left with a short last batch), up to four of them as
                    // thread rows of one workgroup: a quarter of the partials, and with four or fewer
                    // no second launch at all. f16 [4096, 8192][:, ::2] over axis 0, 48 workgroup
                    // slices -> 16 of four thread rows: 17.9 -> 14.6 us; f32 [512, 65536] over axis 0,
                    // 3 slices -> one launch of four thread rows: 4.9 -> 6.1 TB/s.
                    // (An op that spends a dozen instructions per element - an exponential, f64 squares of f32
                    // data - needs a second wavefront per SIMD to run beside the loads: eight thread rows. f32
                    // [8192, 4096] over axis 0, us with 4 / 8 thread rows x 16 splits: sum 25.1 / 25.4,
                    // sum_square 27.7 / 25.8, logsumexp 34.7 / 28.4.)
                    const int64_t parts = std::min<int64_t>(pow2_ceil(rp), pow2_floor(can));
                    const int64_t by = std::min<int64_t>(parts, heavy ? 8 : 4);
                    p.split = (int)std::max<int64_t>(1, std::min<int64_t>(parts / by, cap));
                    p.by = (int)by * base_by;
                }
            } else {
                p.by = (int)rows_in_one_launch();
            }
        }
        // Workgroups of several wavefronts each live as long as the launch does, one (or two ...) per
        // compute unit: a count just over a multiple of the 256 compute units leaves a few units with one
        // workgroup more than the rest, and everybody waits for those. f32 [6553, 5120] over axis 0, 20
        // column blocks x splits (workgroups): 12 (240) 24.9 us, 13 (260) 32.0, 16 (320) 29.0, 25 (500)
        // 25.2, 26 (520) 30.1; f32 [43690, 768], 3 column blocks: 85 (255) 26.7 us, 86 (258) 35.6.
        // So the split moves to the nearest count that fills whole rounds of compute units.
        if (p.split > 1 && p.by * p.bx >= 128) {
            const int64_t total = xblocks * p.split;
            const int64_t rounds = (total + kComputeUnits - 1) / kComputeUnits;
            if (total * 10 < rounds * kComputeUnits * 9) {  // less than 90 % of its rounds filled
                int64_t best = p.split, best_dist = -1;
                for (int64_t r = std::max<int64_t>(1, rounds - 1); r <= rounds; ++r) {
                    const int64_t cand = r * kComputeUnits / xblocks;
                    if (cand < 1 || cand > 256 || p.R / (cand * (p.by / base_by)) < 8) continue;
                    const int64_t dist = cand > p.split ? cand - p.split : p.split - cand;
                    if (best_dist < 0 || dist < best_dist) {
                        best = cand;
                        best_dist = dist;
                    }
                }
                const int64_t cap2 = std::max<int64_t>(1, (int64_t)((64ll << 20) / acc_size) / p.K);
                p.split = (int)std::min(best, cap2);
            }
        }
        p.chunk = (p.R + p.split - 1) / p.split;
    }
    return p;
}

static void describe_dims(std::string& s, const char* name, const Dims& d) {
    s += name;
    s += "=[";
    char buf[64];
    for (int i = 0; i < d.n; ++i) {
        snprintf(buf, sizeof buf, "%s%lld:%lld", i ? "," : "", (long long)d.size[i],
                 (long long)d.stride[i]);
        s += buf;
    }
    s += "]";
}

std::string describe(const ReducePlan& p) {
    char buf[256];
    std::string s;
    switch (p.kind) {
        case ReduceKind::Empty: return "empty";
        case ReduceKind::Identity: return "identity";
        case ReduceKind::Row:
            snprintf(buf, sizeof buf, "row%s%s vec=%d tpr=%d rpb=%d rows=%lld cols=%lld split=%d(%dx%d) ",
                     p.row_tile ? "-tile" : p.ragged ? "-ragged" : (p.lean || p.mod_rows) ? "" : "-general", p.sstride == 2 ? "-step2" : p.unaligned ? "-unaligned" : p.interleave > 1 ? "-interleaved" : p.mod_rows ? "-modular" : "", p.vec, p.tpr, p.rpb,
                     (long long)p.K, (long long)p.R, p.split, p.split_q, p.split_i);
            break;
        case ReduceKind::Col:
            snprintf(buf, sizeof buf, "col%s%s vec=%d bx=%d by=%d outs=%lld red=%lld split=%d ",
                     p.group_tile ? "-group-tile" : p.flat_xb ? "-flat-wide" : p.flat_t ? (p.unaligned ? "-flat-unaligned" : "-flat") : p.kept_swapped ? "-swapped" : p.unaligned ? "-unaligned" : p.lean ? "" : "-general",
                     p.sstride == 2 ? "-step2" : "", p.vec,
                     p.flat_t ? p.flat_t : p.bx, p.by,
                     (long long)p.K, (long long)p.R, p.split);
            break;
    }
    s = buf;
    if (p.flat_w) s += "as=" + std::to_string(p.flat_w) + "x" + std::to_string(p.flat_slices * p.flat_phases) + " ";
    describe_dims(s, "kept", p.kept);
    s += " ";
    describe_dims(s, "red", p.red);
    return s;
}

// ---- normalisation ---------------------------------------------------------

// Softmax rows held in registers and LDS (row_lds_kernel): the smallest of its three launch shapes whose
// slots hold the `nvec` vectors of a row's vector grid; false when none does. 24 + 8 vectors of a four-byte
// type (16 + 8 of a two-byte type) per thread, 256 or 512 threads; twice that per thread, 512 threads.
// Shifted four-byte rows keep four vectors fewer in registers (20 + 8, 44 + 16): the masks of the row ends
// beside 24 or 48 vectors spilled 30 registers, and the spills' traffic showed in the HBM counters (f32
// [640, 50257]: 1.22 times the algorithmic bytes; the aligned [640, 50304]: 1.00).
static bool lds_row_shape(NormPlan& p, int64_t nvec, size_t elem_size, bool shift) {
    const int per = elem_size == 4 ? (shift ? 28 : 32) : 24;
    const int big = elem_size == 4 ? (shift ? 60 : 64) : 48;
    if (nvec <= 256 * per) {
        p.tpr = 256;
        p.nchunk = per;
    } else if (nvec <= 512 * per) {
        p.tpr = 512;
        p.nchunk = per;
    } else if (nvec <= 1024 * per) {
        // one workgroup fills the compute unit either way; sixteen wavefronts of 128 registers keep more loads and
        // stores in flight than eight of 256 (f32 [1024, 128256] log_softmax 217 -> 208 us, f16 [2048, 151936] 262 -> 249,
        // f32 [1024, 100277] 183 -> 171, [2048, 69632] 237 -> 224)
        p.tpr = 1024;
        p.nchunk = per;
    } else if (nvec <= 512 * big) {
        p.tpr = 512;
        p.nchunk = big;
    } else {
        return false;
    }
    p.kind = NormKind::RowReg;
    p.lds_rows = 1;
    p.rpb = 1;
    return true;
}

// Softmax over an axis of up to 1024 elements with a contiguous inner dim of L: whether 512 or 1024 threads that hold it in whole
// vectors (col_tall_kernel) are ahead of the plan `p` (`found`: register columns of 256 threads, else three launches), and
// that plan in `p` if so. Us over axis 1, as it was and this:
//   four bytes, 129 ... 256 elements  [64, 129, 256] 9.8 and 6.8, [6, 200, 8200] 21.2 and 17.4, [20, 129, 8001] 48.8 and 34.2; where inner rows are
//     whole 256-byte segments the register columns read what they need of every line too, and stay once there is more than a round of
//     workgroups ([730, 256, 64] 20.1 and 25.7, [1930, 256, 64] 47.4 and 53.5, [21, 138, 3136] 14.9 and 19.4; 98 shapes 0.98x, below a round 1.03x). In 257 ... 399
//     workgroups ([16, 222, 2240] 13.8 and 15.4, 24 shapes 1.02x with eight slower) and inner rows of a few vectors ([8181, 208, 12] 33.2 and 43.3)
//     likewise
//   257 ... 512  [1, 335, 58050] 88.6 and 45.2, [200, 335, 100] 29.0 and 19.6, [6, 512, 8200] 75.6 and 51.6; odd inner rows of 27 ... 52 MiB in all stay for
//     inputs that the last-level cache still holds ([16, 512, 1001] 22.3 and 23.9, [128, 512, 129] 23.9 and 27.6, [8, 512, 3001] 28.2 and 30.7, [24, 400,
//     1001] 22.2 and 24.0); from memory they would gain there too (260 shapes 1.25x). Where inner rows
//     are whole 256-byte segments the 128-register form stays below 128 MiB and for very long rows ([16, 512, 2048] 25.3 and
//     29.5, [1, 512, 262144] 212 and 215; [512, 512, 512] 210 and 190, [64, 512, 1024] 53.2 and 50.1)
//   513 ... 1024  [64, 777, 256] 28.3 and 21.5, [16, 1024, 2048] 92.2 and 53.4; one workgroup fills a compute unit, so there must be enough of
//     them, of rows that are not short: [4, 1000, 1000] 16.8 and 18.9, [200, 1000, 100] 66.2 and 72.2
//   two bytes, 65 ... 256  [64, 100, 256] 10.1 and 5.7, [16, 100, 1001] 13.4 and 6.4; [64, 256, 2048] 26.0 and 29.6, [100, 256, 1024] 26.1 and 25.1
//   257 ... 512  [100, 335, 500] 35.7 and 23.9, [512, 512, 512] 128 and 105; not with inner rows of up to 32 elements that
//     the register columns take in pieces of four, or short odd ones ([4200, 311, 16] 23.4 and 29.1, [2289, 334, 28] 32.6 and 38.9, [489, 353, 11] 11.9 and 16.3;
//     others [2032, 330, 10] 21.6 and 15.4, [5810, 323, 17] 56.7 and 51.1), nor, where they are whole 128-byte segments, with the second of a unit's two
//     workgroups in less than half of the units ([22, 455, 3392] 28.0 and 31.6, [15, 415, 2624] 18.6 and 20.0; but [18, 259, 2816], 396 workgroups, 16.0 and
//     14.6, [866, 477, 64] 24.5 and 22.0), or few workgroups where the register columns' pieces are aligned and these are not ([18, 410, 180] 13.3 and 14.7)
//   513 ... 1024  [512, 513, 24] 21.2 and 15.1, [64, 1000, 256] 28.4 and 22.1, [16, 1000, 2048] 38.1 and 28.4; [4, 777, 1000] 13.4 and 19.1; three
//     launches for odd rows of 1024 and more ([19, 596, 3822] 60.4 and 70.6, [1, 513, 58050] 38.5 and 42.6, [20, 1000, 1501] 40.6 and 51.3; up to 640
//     elements within a round [12, 600, 2051] 27.0 and 23.1), for very long ones, and the flat walk where the last of several rounds is a fifth empty
//     ([536, 896, 180] 121.8 and 149.0), for odd rows of 512 ... 1023 a third ([40, 777, 1001] 46.7 and 56.5, but [90, 600, 517] 53.3 and 46.1, [180, 777, 517]
//     149 and 108; below 64 [966, 544, 35] 47.0 and 38.3); where three launches have whole vectors of wide inner rows, they are
//     ahead in 257 ... 399 workgroups and 513 ... 899 (8 and 10 shapes 0.89x and 1.00x, then 27 0.96x; up to a round 24 1.11x, 400 ... 512 1.15x)
//   three launches for too few positions, any of these  [8, 129, 64] 10.7 and 5.5, two bytes [4, 65, 1000] 10.9 and 5.1, [1, 300, 200] 10.9 and 9.1
static bool tall_columns(NormPlan& p, bool found, const void* in_data, const void* out_data, int64_t sa, int64_t sb, int64_t L, int64_t batch,
                         size_t elem_size) {
    const int64_t vec = 16 / (int64_t)elem_size;
    if ((elem_size != 2 && elem_size != 4) || L < vec || (((uintptr_t)in_data | (uintptr_t)out_data) % elem_size) != 0) return false;
    const bool grid = L % vec == 0 && sa % vec == 0 && sb % vec == 0 && (((uintptr_t)in_data | (uintptr_t)out_data) & 15) == 0;
    int64_t threads = 1024, tx = 16, nc = 8;
    if (elem_size == 4) {
        tx = p.cols <= 256 ? 32 : 16;
        nc = p.cols <= 512 ? 8 : 16;
    } else {
        threads = p.cols <= 512 ? 512 : 1024;
        nc = p.cols <= 256 ? 8 : 16;
    }
    const int64_t blocks = (batch * ((L + vec - 1) / vec) + tx - 1) / tx;
    if (blocks * threads >= (1ll << 32)) return false;  // work-items of one launch
    const bool whole_segments = found && p.vec == 4 && p.nchunk == 32 && elem_size == 4;  // the 128-register form
    const int64_t bytes = p.cols * L * batch * (int64_t)elem_size;
    // (the compute units that got a workgroup more than the others are waited for: 257 ... 400 of them, and two-byte ones of 1024 threads, of which
    // a unit holds one, whenever the last round is a fifth empty)
    const bool part_of_a_round = blocks > kComputeUnits && blocks < 400;
    const int64_t rounds = (blocks + kComputeUnits - 1) / kComputeUnits;
    if (p.cols > 512) {
        if (elem_size == 4 ? (blocks < 192 || L < 256) : blocks < 96) return false;
        if (elem_size == 2 && !grid && L >= 64 && L < 64 * vec && (p.cols * L) % vec == 0 && rounds > 1 && blocks * 5 < rounds * kComputeUnits * 4) return false;
        if (elem_size == 2 && !grid && L >= 64 * vec) {
            if (batch == 1 || (rounds > 1 && blocks * 3 < rounds * kComputeUnits * 2)) return false;
            if (L >= 128 * vec && (rounds > 1 || p.cols > 640)) return false;  // (what else there is has unaligned vectors there, not the flat walk)
        }
        if (elem_size == 2 && grid && L >= 320 && (part_of_a_round || (blocks > 2 * kComputeUnits && blocks < 900) || (L > 8192 && blocks > kComputeUnits))) return false;
    } else if (!found) {
        // (odd inner rows of a wavefront of vectors and more: tests name the three passes)
        if (p.cols > 256 && !grid && L >= 64 * vec) return false;
    } else if (elem_size == 4) {
        if (p.cols <= 128 || L <= 16) return false;
        if (whole_segments && (p.cols <= 256 || L > 16384 || bytes < (128ll << 20))) return false;
        if (p.cols <= 256 && grid && (L % 64 == 0 ? blocks > kComputeUnits : part_of_a_round)) return false;
        if (!grid && p.cols > 320 && L >= 96 && bytes >= (27ll << 20) && bytes < (52ll << 20)) return false;
    } else {
        if (p.cols <= 64 || (grid && p.cols > 128 && p.cols <= 256 && L >= 1024 && bytes >= (64ll << 20))) return false;
        const bool short_rows = L <= 32 && L != 24 && (L % 4 == 0 || (L < 16 && L % 2 == 1));
        const bool half_a_round = (blocks > kComputeUnits && blocks < 360) || (blocks > 2 * kComputeUnits && blocks < 600);
        if (p.cols > 256 && (short_rows || (L % 64 == 0 && half_a_round) || (!grid && !p.shift && blocks < 128 && L > 32))) return false;
    }
    p.kind = NormKind::ColReg;
    p.tall = (int)threads;
    p.vec = (int)vec;
    p.shift = grid ? 0 : 1;
    p.nchunk = (int)nc;
    p.tpr = (int)(threads / tx);
    return true;
}

NormPlan plan_normalize(const void* in_data, const void* out_data, const int64_t* shape,
                        const int64_t* strides, int ndim, int64_t axis, int n_norm_dims,
                        size_t elem_size, bool fused, const void* residual) {
    NormPlan p;
    int64_t total = 1;
    for (int i = 0; i < ndim; ++i) total *= shape[i];
    if (total == 0 || ndim == 0) {
        p.kind = NormKind::Empty;
        return p;
    }
    // contiguous output strides
    int64_t ostr[kMaxRank];
    {
        int64_t s = 1;
        for (int i = ndim - 1; i >= 0; --i) {
            ostr[i] = s;
            s *= shape[i];
        }
    }
    bool is_norm[kMaxRank] = {};
    if (n_norm_dims > 0)
        for (int i = ndim - n_norm_dims; i < ndim; ++i) is_norm[i] = true;
    else
        is_norm[axis] = true;

    // Row dims: merged only where input AND output are both one dense run.
    p.rows = 1;
    for (int i = 0; i < ndim; ++i) {
        if (is_norm[i]) continue;
        p.rows *= shape[i];
        if (shape[i] == 1) continue;
        int n = p.kept_in.n;
        if (n > 0 && p.kept_in.stride[n - 1] == strides[i] * shape[i] &&
            p.kept_out.stride[n - 1] == ostr[i] * shape[i]) {
            p.kept_in.size[n - 1] *= shape[i];
            p.kept_in.stride[n - 1] = strides[i];
            p.kept_out.size[n - 1] *= shape[i];
            p.kept_out.stride[n - 1] = ostr[i];
        } else {
            if (n == kMaxDims)
                fail(HPT_ERR_SHAPE, "view has more than %d non-mergeable row dims", kMaxDims);
            p.kept_in.size[n] = p.kept_out.size[n] = shape[i];
            p.kept_in.stride[n] = strides[i];
            p.kept_out.stride[n] = ostr[i];
            p.kept_in.n = p.kept_out.n = n + 1;
        }
    }
    // Normalised dims keep their logical order (gamma/beta and the output index by it).
    p.cols = 1;
    for (int i = 0; i < ndim; ++i) {
        if (!is_norm[i]) continue;
        p.cols *= shape[i];
        push_merged(p.norm_in, shape[i], strides[i]);
    }
    // Output stride along the (flattened) normalised index.
    p.out_axis_stride = 1;
    if (n_norm_dims <= 0) p.out_axis_stride = ostr[axis];
    if (p.cols == 1) {
        // one element per row: still a legal call. The axis has no extent, so neither of its strides
        // matters: say 1 and the row plans (one lane per "row") take it, whatever the axis was.
        p.norm_in.n = 1;
        p.norm_in.size[0] = 1;
        p.norm_in.stride[0] = 1;
        p.out_axis_stride = 1;
    }

    const int64_t sa = p.norm_in.n == 1 ? p.norm_in.stride[0] : 0;  // input stride along the row
    const int max_vec = (int)(16 / elem_size);

    // default: one group of lanes per row, striding along the row
    p.kind = NormKind::Generic;
    p.vec = 1;
    p.tpr = (int)std::min<int64_t>(1024, pow2_ceil((p.cols + 3) / 4));
    if (p.tpr > 64 && p.tpr < 256) p.tpr = 256;
    p.rpb = std::max(1, 256 / p.tpr);

    if (p.norm_in.n == 1 && p.out_axis_stride == 1) {
        // rows are contiguous in the output
        // input contiguous along the rows, output along the axis (a transposed view): register tiles in
        // one pass, or statistics pass + register-tile transpose; unaligned vectors (shift) where a pitch, a
        // length or a base is off the 16-byte grid. The rows went element by element then, one cache line per
        // lane and load: device us, rows x columns, softmax and layernorm: f16 15552 x 1470 206 and 226 -> 31.7 and 30.7,
        // f16 2066 x 11011 248 and 262 -> 50.7 and 49.7, f32 2557 x 2644 97 and 102 -> 25.7 and 24.4, f32 6966 x 368
        // 32 and 36 -> 11.4 and 11.3, f16 1279 x 432 9.6 and 10.6 -> 6.9 and 6.6.
        const int nk = p.kept_in.n;
        const int v = max_vec;
        const bool lies_transposed = sa > 1 && nk >= 1 && nk <= 2 && p.kept_in.stride[nk - 1] == 1 && v > 1 &&
                                     (nk == 1 || p.kept_in.size[0] <= 65535) &&
                                     p.kept_in.size[nk - 1] <= (1 << 30) && p.cols <= (1 << 30) &&  // 32-bit positions
                                     p.kept_in.size[nk - 1] >= 8 * v && p.cols >= 8 * v;
        const bool on_grid = lies_transposed && p.kept_in.size[nk - 1] % v == 0 && p.cols % v == 0 && sa % v == 0 &&
                             (nk == 1 || p.kept_in.stride[0] % v == 0) &&
                             ((uintptr_t)in_data % 16) == 0 && ((uintptr_t)out_data % 16) == 0;
        // (columns that overlap, of a view made by hand, keep the forms below)
        if (lies_transposed && (on_grid || sa >= p.kept_in.size[nk - 1])) {
            // Single pass when 16 vectors per thread hold (16 * rgN bytes of rows) x (all
            // columns): rgN lanes along the rows, 1024 / rgN thread columns of 16 columns
            // each, 4096 columns at most. Long row segments where they leave enough workgroups; a
            // matrix too small for that is cut into segments of 64 and 32 bytes, which still beats three launches
            // by far (device us, three passes -> one; rows x columns): f32 3200 x 224 softmax 21.5 -> 5.6, layernorm
            // 12.6 -> 4.9; f16 5184 x 2048 24.7 -> 17.2, 21 -> 16.0; f32 300 x 1001 18.6 -> 7.5; bf16 511 x 2001
            // 22 -> 12.6; f32 200 x 3300 layernorm 14.2 -> 10.8 and, where the few workgroups have most columns to
            // walk, 129 x 4000 14.0 (and two gaps between launches) -> 14.6. Beyond 4096 columns 32-byte segments gain
            // nothing (f16 2048 x 8192 28.0 -> 26.3, f32 333 x 8000 layernorm 17 -> 25): three passes. Matrices on the grid
            // below 16384 elements keep three passes only because tests name that plan; in time they lose as well
            // (f32 64 x 100 softmax 13.8 -> 4.8).
            const int64_t R = p.kept_in.size[nk - 1];
            const int64_t batch = nk > 1 ? p.kept_in.size[0] : 1;
            const int64_t cgroups = (p.cols + 15) / 16;
            auto blocks_of = [&](int rg) { return (R + rg * v - 1) / (rg * v) * batch; };
            int rgN = 16;
            while (rgN >= 4 && cgroups * rgN > 1024) rgN >>= 1;
            if (rgN > 8 && blocks_of(rgN) < 256) rgN = 8;
            // Sums of exponentials of f32 rows: f64, but for matrices on the vector grid that fill the chip with long
            // segments, where a thread's 16 of a row are added in f32 and the conversions would show (f32
            // 6080 x 2752 38.3 -> 39.6 us).
            const bool wide_sum = !on_grid || blocks_of(rgN) < 128;
            if (rgN > 4 && blocks_of(rgN) < 192) rgN = 4;
            if (rgN == 4 && blocks_of(rgN) < 128) rgN = 2;
            const bool tile = cgroups * 4 <= 1024 && (!on_grid || blocks_of(rgN) >= 128 || total >= 16384);
            // Few rows off the grid: a group of lanes per row (the general form) reads single elements at a stride, but has
            // every row in a workgroup of its own at once. It is ahead of few tiles of two-byte rows beyond 256 columns, whose 16
            // rows share a workgroup (device us, lanes and tile: bf16 85 x 3255 softmax 10.1 and 15.6, 207 x 1238 7.4 and 9.6, 107 x
            // 288 5.6 and 7.5, f16 138 x 3583 12.5 and 15.0; layernorm bf16 183 x 1189 8.0 and 9.6, f16 goes either way, 137 x 579 6.5
            // and 7.0, 176 x 1854 9.7 and 7.7; 24 tiles and more gain mostly: f16 478 x 339 7.1 and 6.6, bf16 504 x 1201 11.2 and 8.7,
            // but 492 x 288 softmax 6.3 and 7.6; wider types always: f32 163 x 1691 10.2 and 9.9, f64 493 x 16 6.2 and 5.0), and of three
            // launches for few and not too long rows (f32 83 x 5029 softmax 16.2 and 20.9, 40 x 6207 17.2 and 20.0, 35 x 15104
            // 30.8 and 26.2; layernorm 51 x 4736 15.3 and 14.8, 96 x 7241 19.8 and 16.7; two-byte 113 x 4181 layernorm 13.8 and 20.3,
            // 122 x 12359 28.0 and 22.2, softmax 88 x 9461 21.2 and 24.1, 90 x 13253 27.6 and 27.4; f64 18 x 5625 17.4 and 15.0). From
            // 129 to about 256 rows the lanes are still ahead (f32 146 x 5018 17.1 and 22.1, 207 x 6398 22.7 and 23.4), but tests
            // name the three passes there.
            const int64_t longest = (n_norm_dims > 0 ? 4608 : 6656) * (elem_size == 2 ? 3 : 2) / 2;
            const bool lanes = !on_grid && elem_size <= 4 && (tile ? elem_size == 2 && p.cols > 256 && blocks_of(rgN) < 24 : p.rows <= 128 && p.cols < longest);
            if (!lanes) {
                p.vec = v;
                p.shift = on_grid ? 0 : 1;
                if (tile) {
                    p.kind = NormKind::TransposedTile;
                    p.wide_sum = wide_sum;
                    p.tpr = rgN;
                    const int64_t cols_per_wave = 16 * (64 / rgN);
                    p.rpb = (int)((p.cols + cols_per_wave - 1) / cols_per_wave);
                    return p;
                }
                p.kind = NormKind::Transposed;
                // statistics pass: a wavefront covers 64*v rows, every one keeps at least 32 columns. Its loads are in flight two batches
                // deep, so one workgroup per compute unit is enough (us, two and one, stored [columns, rows]: f32 [8192, 8192] softmax 145 and
                // 130, layernorm 144 and 130, [6000, 6000] 98.4 and 92.7, 92.1 and 89.3; f16 [8192, 8192] layernorm 78.7 and 72.6; f64 [8192, 4096] softmax
                // 152 and 134, though [6000, 6000] 156 and 166). Two-byte softmax, twice the arithmetic per byte, keeps two (f16 [16384, 4096] 74.7
                // and 76.7, [6000, 6000] 57.5 and 60.4), unless that many would leave wavefronts too few columns: then what there is fills
                // one round and not a part of the second (f16 [5001, 4001] softmax, 312 workgroups and 256, 41.3 and 39.0).
                const int64_t groups = (R + 64 * v - 1) / (64 * v) * batch;
                const int64_t want = elem_size == 2 && n_norm_dims <= 0 ? 512 / groups : full_rounds(groups, 2);
                int64_t S = std::max<int64_t>(1, std::min<int64_t>(want, p.cols / 128));
                if (S < want && S * groups > kComputeUnits && S * groups * 10 < 2 * kComputeUnits * 9) S = kComputeUnits / groups;
                p.tsplit = (int)std::min<int64_t>(S, 64);
                // Wavefronts per workgroup of the statistics pass: four, one per SIMD, stream a large input. Where half of the compute units
                // have no workgroup and a wavefront of four would walk 16 ... 63 columns, the pass is that chain of loads and exponentials, and eight halve it
                // (us, four and eight, softmax, stored [columns, rows]: f16 [6208, 163] 18.1 and 16.3, f32 [7533, 203] 17.4 and 17.0, bf16 [16000, 256] 25.5 and
                // 20.8; not the f64 sums of layernorm, f16 [6208, 163] 16.5 and 17.0, f32 [12000, 400] 18.3 and 18.9).
                const int64_t slices = p.tsplit;
                p.tpr = n_norm_dims <= 0 && slices * groups <= kComputeUnits / 2 && p.cols >= 64 * slices && p.cols < 256 * slices ? 8 : 4;
                p.scratch_bytes = (size_t)p.rows * p.tsplit * 16 + (size_t)p.rows * 3 * 8;
                return p;
            }
        }
        if (sa >= 1 && sa <= 4) {
            // vector width: input and output must both allow it
            int v = 1;
            if (sa == 1) {
                Dims none;
                int vi = legal_vec(in_data, elem_size, p.cols, p.kept_in, none, 0, 0);
                int vo = legal_vec(out_data, elem_size, p.cols, p.kept_out, none, 0, 0);
                v = std::min(std::min(vi, vo), max_vec);
            } else if (sa == 2 && max_vec >= 2) {
                // every second element: load full vectors, keep the even positions
                Dims none;
                const int uv = max_vec / 2;
                int vi = legal_vec(in_data, elem_size, p.cols * 2, p.kept_in, none, 0, 0);
                bool out_ok = ((uintptr_t)out_data % (uv * elem_size)) == 0 && p.cols % uv == 0;
                // few rows of up to 4096 elements: single elements have up to four times the threads, and there is room for all of them (f16
                // [340, 1763] stored layernorm 4.4, 5.6 as vectors, [389, 3853] 6.1 and 6.6, softmax [340, 1763] 3.8 and 4.2; from 1.3
                // million elements on, or 0.6 million for softmax of short rows, the vectors are ahead)
                const int64_t elements = p.rows * p.cols;
                const bool few = !fused && p.cols <= 4096 && (n_norm_dims > 0 ? elements < 1300000 : p.cols < 1024 && elements < 600000);
                if (vi == max_vec && out_ok) {
                    v = max_vec;
                    p.sstride = 2;
                } else if (elem_size == 2 && p.cols >= 640 && (p.cols + uv - 1) / uv <= 4096 && !(fused && n_norm_dims > 0 && p.cols <= 8192) && !few &&
                           ((uintptr_t)in_data % elem_size) == 0 && ((uintptr_t)out_data % elem_size) == 0) {
                    // Two-byte rows off the vector grid: the same vectors unaligned (us, every second of the stored, single elements and
                    // this: f16 [3456, 7897] causal 27.6 and 19.9, layernorm 30.9 and 28.3, [2000, 16383] softmax 39.8 and 28.8. f32 goes either way:
                    // softmax [2000, 16383] 53.6 and 47.6, with sums over more elements of a lane, [3456, 7897] 32.3 and 35.7; x + residual keeps
                    // single elements up to 1024 threads' eight, its four vectors spill: f16 [3456, 7897] 35.2, 52.1 as vectors, [7598, 3853] 30.1, 54.8, though bf16
                    // [1745, 10870] 36.2 and 32.7; longer rows would stream: bf16 [110, 23911] 16.4, 10.2 as vectors, f16 [71, 23142] 15.1 and 10.8).
                    v = max_vec;
                    p.sstride = 2;
                    p.shift = 1;
                    p.ua_rows = 1;
                }
            }
            p.vec = v;
            // Rows that start off 16-byte boundaries (odd row lengths): the row kernels can still move
            // aligned vectors and mask the two ends of a row, provided input and output rows are
            // misaligned by the same amount: equal bases and row pitches modulo 16 bytes.
            // (few, very long rows are shared among workgroups below, element by element). Measured: the
            // register kernel gains from this between about 16 and 2048 vectors per row (f32 [130561, 257]
            // softmax 3.5 -> 4.9 TB/s, [8190, 4097] 3.1 -> 4.1); shorter rows are mostly row ends and stay
            // element-wise, longer ones stream (two sweeps) at the same speed.
            if (sa == 1 && v == 1 && max_vec > 1 && p.cols >= 16 * max_vec && !(p.rows <= 128 && p.cols >= 16384)) {
                bool same = (((uintptr_t)in_data ^ (uintptr_t)out_data) & 15) == 0 && ((uintptr_t)in_data % elem_size) == 0;
                for (int i = 0; i < p.kept_in.n; ++i)
                    if (((p.kept_in.stride[i] - p.kept_out.stride[i]) * (int64_t)elem_size) % 16 != 0) same = false;
                const int64_t nvs = (p.cols + 2 * (max_vec - 1)) / max_vec;
                // (two-byte layernorm keeps two vectors per thread, so its rows stay in registers up to 1024
                // vectors, 512 threads; f16 [8190, 4097] 1.9 -> 2.2 TB/s, [5461, 6145] 1.9 -> 2.8 against streaming)
                // Softmax rows beyond the register kernel's 2048 shifted vectors stay on chip in registers and
                // LDS (row_lds_kernel, whose vector grid starts on the 128-byte line that holds the row's first
                // element) up to 122846 four-byte or 196545 two-byte elements; they streamed before (two reads).
                // Measured (TB/s): f32 [4096, 30522] 3.5 -> 5.55, [2048, 50257] 4.45 -> 5.3, [1024, 100277] 3.7 -> 4.55;
                // f16 [8192, 32001] 4.0 -> 5.55, [4096, 50257] 4.35 -> 5.2, [2048, 98001] 4.2 -> 4.9.
                if (same && n_norm_dims <= 0 && nvs > 2048 && (elem_size == 2 || elem_size == 4) &&
                    lds_row_shape(p, (p.cols + 128 / (int64_t)elem_size + max_vec - 2) / max_vec, elem_size, true)) {
                    p.vec = max_vec;
                    p.shift = 1;
                    return p;
                }
                // Two-byte rows and f32 layernorm rows as unaligned vectors from the row's start on, whatever the alignments of input,
                // output and residual: no masks but at a row's last vector, and gamma / beta per column as in aligned rows. Us, aligned
                // vectors that contain the row and this: bf16 [17616, 2202] softmax 40.9 and 33.0, [28550, 805] log_softmax 21.2 and 18.2,
                // causal [32, 1001, 1001] 26.9 and 20.7; f16 layernorm [8190, 4097] 59.7 and 33.7, [14245, 561] 14.4 and 11.2, [2000, 12001]
                // (streamed) 31.4 and 22.7; f32 layernorm [8190, 4097] 60.4 and 49.6, [3000, 9001] (streamed) 61.6 and 43.9. The f32 softmax
                // is as fast as that of aligned rows ([16000, 2051] 45.3, [16000, 2052] 47.2).
                // The masked aligned vectors, whose stores are whole lines, are ahead for f32 layernorm of few rows alone ([485, 3090] 6.1 and 6.6 us,
                // [336, 4458] 6.5 and 6.9). With more rows and inputs that come from memory they are level, 46 shapes 0.99x, and with inputs
                // that the last-level cache holds behind: f32 layernorm [7163, 1015] 13.4 and 12.3, [2603, 2161] 13.4 and 10.9, x + residual [2545, 1238]
                // 10.0 and 9.0, f16 softmax [1131, 16150] 19.4 and 16.2, [5806, 7142] 0.81x (from memory 42 two-byte shapes 1.01x, x + residual 40 shapes 0.94x).
                // Input and output off the grid by different amounts took single elements: they stay where stores across lines cost more than
                // they save, short rows (f32 layernorm [61855, 97] 15.5 and 17.4, x + residual [55813, 215] 17.7 and 19.4; two-byte
                // x + residual is level from memory and ahead as vectors in the cache, bf16 [142052, 176] 38.6 and 33.7), and layernorm of few (f32 [1425, 263] 4.3 and 5.2, [178, 2100] 4.9 and 5.5).
                const int64_t nvu = (p.cols + max_vec - 1) / max_vec;
                bool unaligned = (elem_size == 2 || (elem_size == 4 && n_norm_dims > 0)) && ((uintptr_t)in_data % elem_size) == 0 &&
                                 ((uintptr_t)out_data % elem_size) == 0 && nvu <= (elem_size == 4 ? 4096 : 2048);
                if (unaligned && same && elem_size == 4 && !fused) {
                    unaligned = p.cols <= 256 || p.rows > 512 || nvs > 2048;
                } else if (unaligned && !same && n_norm_dims > 0) {
                    if (fused) unaligned = elem_size == 2 || p.cols >= 256 || (p.cols >= 128 && p.cols % 4 == 0);
                    else unaligned = (elem_size == 2 || (p.cols >= 128 && (p.cols <= 192 || p.cols >= 256))) &&
                                     (p.cols >= (elem_size == 2 ? 1024 : 4096) || p.rows * p.cols * (int64_t)elem_size >= (3ll << 20));
                }
                if (unaligned) {
                    v = max_vec;
                    p.vec = v;
                    p.shift = 1;
                    p.ua_rows = 1;
                } else if (same && nvs > ((n_norm_dims > 0 && elem_size == 2) ? 1024 : 2048)) {
                    p.kind = NormKind::RowStream;
                    p.vec = max_vec;
                    p.shift = 1;
                    p.tpr = p.cols >= 4096 * max_vec ? 1024 : 256;
                    p.rpb = 1;
                    return p;
                }
                if (same && !p.ua_rows) {
                    v = max_vec;
                    p.vec = v;
                    p.shift = 1;
                }
            }
            // vector loads per row (shifted rows: one more than the row's own length needs)
            int64_t nv = p.ua_rows ? (p.cols + v / p.sstride - 1) / (v / p.sstride) : p.shift ? (p.cols + 2 * (v - 1)) / v : p.cols / (v / p.sstride);
            const bool masks = p.shift && !p.ua_rows;  // the kernel masks both ends of every row
            // Few, very long contiguous rows: share each row among workgroups. (One workgroup per
            // row would leave a chip of 256 compute units mostly idle.)
            if (sa == 1 && !p.shift && p.rows <= 128 && p.cols >= 16384 && p.cols % v == 0) {
                if (v == 1 && max_vec > 1 && ((uintptr_t)in_data % elem_size) == 0 && ((uintptr_t)out_data % elem_size) == 0) {
                    // rows off the 16-byte grid: unaligned vectors, the last one from the row's end backwards
                    v = max_vec;
                    p.vec = v;
                    p.shift = 1;
                }
                const int64_t nvec = (p.cols + v - 1) / v;
                int64_t S = std::min<int64_t>(512, std::max<int64_t>(1, 1024 / p.rows));
                S = std::min<int64_t>(S, std::max<int64_t>(1, nvec / 1024));  // at least 4 vectors per thread
                if (S >= 2) {
                    p.kind = NormKind::RowSplit;
                    p.tsplit = (int)S;
                    p.scratch_bytes = (size_t)p.rows * S * 24;
                    return p;
                }
                if (p.shift) {  // not worth splitting: back to element-wise rows
                    p.shift = 0;
                    p.vec = v = 1;
                }
            }
            // A row fits the registers of a workgroup up to 8 vectors per thread; layernorm also keeps
            // gamma and beta there (the eight-vector form spills), so it stops at four and streams
            // longer rows (two sweeps; gamma / beta as vectors).
            // Two-byte types hold eight elements per vector: with gamma and beta beside the row, sixteen
            // elements per thread is what fits 128 registers, i.e. two vectors (four of a stride-2 row).
            bool ln_half = n_norm_dims > 0 && v > 1 && elem_size == 2;
            // Two-byte layernorm rows of 640 ... 16384 elements: gamma / beta go to LDS (at most 64 KiB)
            // and the row takes three or four vectors per thread like any other. Measured, f16 (TB/s): [6553, 5120]
            // 3.5 -> 4.6, [4096, 8192] 4.7 -> 5.0, [2730, 12288] 3.2 -> 4.6, [2048, 16384] 3.8 -> 4.6; [65536, 1024]
            // 5.0 -> 5.4, [32768, 2048] 4.6 -> 5.3, [74898, 896] 4.5 -> 5.2, [104857, 640] 4.5 -> 4.9 (shorter rows lose:
            // [131072, 512] 4.9 -> 4.5).
            // (With a residual's vectors beside the row's, gamma / beta in registers spill from the third vector on: beyond 256
            // elements, us: f16 [14245, 560] 20.9 -> 12.5, [14245, 561] 28.9 -> 13.9, [30000, 384] 22.8 -> 16.4; bf16 [30000, 256] 11.4, 14.8 this way.)
            // (Few unaligned rows that would take four vectors per thread keep them in registers, two vectors and twice the threads: f16 [121, 6149] 5.9
            // and 6.5, [428, 7001] 7.9 and 8.1; not three: [250, 3000] 6.3 and 5.6.)
            const bool few_unaligned = p.ua_rows && !fused && p.rows <= 512 && nv > 3 * pow2_ceil((nv + 3) / 4);
            if (ln_half && p.sstride == 1 && !masks && nv * v >= (fused ? 264 : 640) && nv * v <= 16384 && !few_unaligned) {
                p.gb_lds = 1;
                ln_half = false;
            }
            const int64_t per = ln_half ? 2 * p.sstride : 4;
            const int64_t reg_limit = ln_half ? 1024 * per : (n_norm_dims > 0 && v > 1) ? 4096 : 8192;
            // Softmax rows beyond eight vectors per thread of a four-byte type (four of a two-byte type) stay on
            // chip in registers and LDS, one read instead of the streaming kernel's two: row_lds_kernel, up to
            // 131072 four-byte or 196608 two-byte elements. Two-byte rows of 98305 ... 131072 elements keep the
            // raw row in the registers of 1024 threads (sixteen vectors each), which measured faster there.
            // (Layernorm in such a kernel, with gamma / beta from L2 in the last sweep, spilled 60 to 130
            // registers and ran at 1.6-3.3 TB/s: such rows stream, at 3.0-3.4.)
            // Measured (TB/s; before: 1024 threads with 8 + 8 vectors staged through registers, the raw-row
            // kernel, or streaming): f32 [640, 50304] 4.35 -> 5.05, [2048, 50304] 5.05 -> 5.35, [2048, 40960]
            // 4.9 -> 5.35, [1024, 128256] 3.75 -> 4.7; f16 [4096, 50304] 4.75 -> 5.55, [4096, 65536] 5.0 -> 5.6,
            // [2048, 98304] 4.45 -> 5.1, [2048, 151936] 4.25 -> 4.55.
            if (n_norm_dims <= 0 && v == max_vec && p.sstride == 1 && !p.shift) {
                const bool raw16 = elem_size == 2 && nv > 12288 && nv <= 16384;
                if (raw16) {
                    p.kind = NormKind::RowReg;
                    p.raw_rows = 1;
                    p.tpr = 1024;
                    p.rpb = 1;
                    p.nchunk = 16;
                    return p;
                }
                // (the causal softmax has no such kernel: its rows stay with the register kernel while they fit)
                if ((elem_size == 4 ? nv > 8192 : elem_size == 2 && nv > 4096) && !(fused && nv <= reg_limit) &&
                    lds_row_shape(p, nv, elem_size, false))
                    return p;
            }
            // Layernorm rows beyond that (up to 32768 four-byte, 49152 two-byte or 16384 eight-byte elements) still fit
            // the registers of 512 or 1024 threads when gamma / beta do not sit beside them: those are read again for
            // every row, vector by vector in the last sweep, from L2. One read of the row instead of the streaming
            // kernel's two. Measured (% of the HBM peak, streaming -> this): f32 [1771, 18944] 39 -> 60, [1310, 25600]
            // 37 -> 57, [1024, 32768] 43 -> 62; f16 [1771, 18944] 27 -> 55, [1310, 25600] 28 -> 43, [1024, 32768] 33 -> 50.
            // (Two-byte rows of seven or eight vectors per thread spill. Where the forms above exist they are as fast
            // or faster: f32 [4096, 8192] 67.5 against 68, [2730, 12288] 68 against 65; f16 [4096, 8192] 59 against 53.)
            if (n_norm_dims > 0 && v == max_vec && v > 1 && p.sstride == 1 && !p.shift && !p.gb_lds && nv > reg_limit) {
                int t = 1024;
                if (elem_size == 2 && nv <= 512 * 5) t = 512;  // f16 [1771, 18944]: 512 x 5 55 %, 1024 x 3 45 %
                const int64_t c = (nv + t - 1) / t;
                // (layernorm(x + residual) holds the residual's vectors beside the row's: fewer fit before it spills)
                if (c <= (fused ? (elem_size == 2 ? 4 : 6) : (elem_size == 2 ? 6 : 8))) {
                    p.kind = NormKind::RowReg;
                    p.gb_lds = 2;
                    p.tpr = t;
                    p.nchunk = (int)c;
                    p.rpb = 1;
                    return p;
                }
            }
            if (nv <= reg_limit) {
                p.kind = NormKind::RowReg;
                // Short rows laid back to back: the plain kinds move whole 16 KiB tiles through LDS
                // (aligned vectors both ways whatever the row length); the fused kinds keep the
                // register plan made below.
                // Measured (TB/s, registers -> tile): f32 softmax [N, 8] 4.0 -> 5.9, [N, 33] 3.5 -> 5.5,
                // [N, 100] 4.0 -> 5.7, [N, 197] 4.5 -> 5.4; f32 layernorm [N, 33] 3.3 -> 5.1, [N, 100]
                // 3.3 -> 5.4; f16 softmax [N, 33] 2.1 -> 4.0, [N, 64] 2.1 -> 4.8. Rows of whole vectors
                // from 512 bytes on (and two-byte layernorm rows of whole vectors) are as fast or faster
                // from registers.
                const int64_t row_bytes = p.cols * (int64_t)elem_size;
                const bool whole = p.cols % max_vec == 0;
                const bool gains = whole ? (row_bytes >= 32 && row_bytes < 512 && !(elem_size == 2 && n_norm_dims > 0)) : true;
                if (sa == 1 && max_vec > 1 && gains && p.kept_in.n == 1 && p.kept_in.stride[0] == p.cols &&
                    (((uintptr_t)in_data | (uintptr_t)out_data) & 15) == 0 && p.cols <= 512 &&
                    p.rows * row_bytes >= (4ll << 20)) {
                    int64_t rows = (16 << 10) / (p.cols * (int64_t)elem_size);
                    rows -= rows % max_vec;
                    if (rows >= max_vec) p.tile_rows = (int)rows;
                }
                // about four 128-bit vectors per thread; rows that only allow single elements
                // take eight per thread (fewer, busier threads: a 257-element row stays in one
                // wavefront instead of four that meet in LDS)
                p.tpr = (int)std::min<int64_t>(1024, v > 1 ? pow2_ceil((nv + per - 1) / per) : pow2_ceil((nv + 7) / 8));
                if (p.tpr > 64 && p.tpr < 256 && !(ln_half && p.tpr == 128)) p.tpr = 256;
                // A row just over a power of two (4097: 1026 vectors) would take twice the threads with half of
                // them idle: softmax (no gamma / beta beside the row) of 4-byte types takes half the threads and five
                // vectors each. Measured (TB/s): f32 [8190, 4097] 4.6 -> 5.1, [8192, 4100] 4.6 -> 5.7, [4096, 8200]
                // 4.1 -> 4.9, [4000, 10000] 4.7 -> 5.1; f16 [8192, 8200] loses (4.7 -> 3.0: eight widened vectors spill).
                if (n_norm_dims <= 0 && v > 1 && elem_size >= 4 && p.tpr >= 512 && nv <= (p.tpr / 2) * 5) p.tpr /= 2;
                int64_t nc = (nv + p.tpr - 1) / p.tpr;
                p.nchunk = (int)std::max<int64_t>(1, pow2_ceil(nc));
                // Threads per row and vectors per thread are powers of two so far, which leaves a quarter
                // to a third of the lanes idle on rows of 3, 5, 6 or 7 times a power of two - the hidden
                // sizes 768, 1536, 2560, 3072, 5120, 6144, 12288. Aligned rows of whole vectors may take 3
                // (any type) or 5, 6, 7 (4- and 8-byte softmax; layernorm up to 6) vectors per thread: the
                // fewest slots win; among equals, rows of up to 256 threads (layernorm: 512) with the fewest
                // vectors per thread, else the fewest threads. Measured, TB/s: f32 softmax [21845, 1536]
                // 256 x 2 4.7 -> 128 x 3 6.0, [5461, 6144] 512 x 4 4.8 -> 256 x 6 5.8, [2730, 12288] 4.3 -> 5.2;
                // f32 layernorm [13107, 2560] 256 x 4 4.5 -> 128 x 5 5.5, [6553, 5120] 4.7 -> 5.6 (256 x 5),
                // [10922, 3072] 4.9 -> 5.7 (256 x 3); f16 softmax [21845, 3072] 256 x 2 4.5 -> 128 x 3 5.9,
                // [13107, 5120] 4.7 -> 5.8 (256 x 3); f16 layernorm [87381, 768] 4.1 -> 5.0 (32 x 3), [43690, 1536]
                // 3.9 -> 4.9 (64 x 3). (Two-byte rows of five vectors or more per thread lose: layernorm spills.)
                // (gamma / beta in LDS: three or four vectors per thread. Five lose to three with twice the threads, idle
                // lanes and all - f16, % of the HBM peak: [29127, 1152] 58 -> 66.5, [13107, 2560] 58 -> 64, [6553, 5120]
                // 56 -> 62, [3640, 9216] 53 -> 58, [3276, 10240] 39 -> 61)
                // (Rows of odd length, covered by aligned vectors: softmax alike - f16 [116306, 577] 3.6 -> 4.1,
                // [44739, 1500] 4.2 -> 4.9, f32 [8190, 4097] 4.4 -> 5.3, [16000, 2051] 4.3 -> 5.5; layernorm, which
                // carries the masks and the unaligned gamma / beta besides, only up to what it had: more spills.)
                if (v == max_vec && v > 1 && p.sstride == 1 && !p.tile_rows) {
                    const int maxc = n_norm_dims > 0 && masks ? (elem_size == 2 ? 2 : 4)
                                                                : elem_size == 2 ? (ln_half ? 3 : 4)
                                                                : (n_norm_dims > 0 ? (fused ? 4 : 6) : 8);
                    // (layernorm(x + residual) holds the residual's vectors beside the row's: with five or six
                    // per thread it spills - f32 [2730, 12288] 3.1 TB/s)
                    const int pref_tpr = n_norm_dims > 0 ? 512 : 256;
                    // (gamma / beta in LDS: the form exists for three to five vectors per thread only)
                    int64_t best = p.gb_lds ? INT64_MAX : (int64_t)p.tpr * p.nchunk;
                    int bt = p.gb_lds ? 0 : p.tpr, bc = p.nchunk;
                    bool base_stands = !p.gb_lds;  // the shape chosen above is still the best one
                    for (int t = p.gb_lds ? 32 : 16; t <= 1024; t <<= 1) {
                        const int64_t c = std::max<int64_t>((nv + t - 1) / t, p.gb_lds ? 3 : 1);
                        if (c > maxc) continue;
                        const int64_t slots = t * c;
                        bool take = slots < best;
                        if (!take && bt && slots == best && t != bt) {
                            // equal: a row inside the preferred width beats one outside it; inside, the wider row
                            // (fewer vectors per thread) wins, outside, the narrower one (f32 softmax [4096, 8192]
                            // 512 x 4 5.3 -> 256 x 8 5.7 TB/s, [2048, 16384] 1024 x 4 4.8 -> 512 x 8 5.2). The shape
                            // chosen above only gives way when it lies outside the preferred width.
                            const bool in_t = t <= pref_tpr, in_b = bt <= pref_tpr;
                            take = in_t != in_b ? in_t : (in_t ? t > bt : t < bt);
                            if (base_stands && in_b) take = false;
                        }
                        if (take) {
                            best = slots;
                            bt = t;
                            bc = (int)c;
                            base_stands = false;
                        }
                    }
                    if (bt) {
                        p.tpr = bt;
                        p.nchunk = bc;
                    }
                    // Softmax rows beyond 2048 vectors that still leave a sixteenth of those slots idle (threads
                    // come in powers of two): row_lds_kernel's 256 threads take slots in steps of 256 vectors.
                    // Measured (TB/s): f32 [4096, 16388] 4.8 -> 5.15; f16 [8192, 16392] 4.2 -> 5.45. (Full rows
                    // gain nothing: f32 [4096, 32768] 5.55 -> 5.55, f16 [8192, 32768] 5.75 -> 5.35.)
                    if (n_norm_dims <= 0 && !fused && !p.shift && nv > (elem_size == 2 ? 1024 : 2048) && (elem_size == 2 || elem_size == 4) &&
                        (int64_t)p.tpr * p.nchunk - nv >= nv / 16 && lds_row_shape(p, nv, elem_size, false))
                        return p;
                }
                int block = std::max(256, p.tpr);
                p.rpb = block / p.tpr;
                // Layernorm workgroups walk the rows; how many of them is best depends on how many a compute unit
                // can hold. f32 rows of four vectors per thread (gamma and beta beside them: ~100 registers, four
                // workgroups of 256 threads per compute unit) do best with THREE per compute unit, rows of two vectors
                // with six. Measured, us (768 / 1024 / 1536 workgroups): [8192, 4096] 45.7 / 47.6 / 47.5, [32768, 1024]
                // 45.1 / 46.2 / 47.1, [65536, 512] 45.0 / 46.4 / 47.4; [16384, 2048] 52.9 / 47.5 / 46.3, [8192, 2048]
                // 29.1 / 26.2 / 25.2, [8192, 1536] 26.9 / 23.1 / 20.3. Two-byte rows prefetch their next row and stay at 1024.
                // Two-byte rows with gamma / beta in LDS, up to four vectors per thread: three times as many workgroups
                // as a compute unit holds at once, so that one that ends early is replaced (with 1024 a workgroup walks
                // 10 or 11 row pairs and the last step runs two thirds empty). Measured, us (1024 / 1536 / 3072 / all rows):
                // f16 [21845, 3072] 52.1 / 50.5 / 48.6 / 51.0, [16384, 4096] 50.7 / 54.3 / 48.6 / 51.3, [65536, 1024]
                // 49.0 / 49.9 / 47.3 / 46.4; rows of five vectors per thread do best with 1024 ([13107, 5120] 53.2 / 61.9 / 59.2 / 64.2).
                if (n_norm_dims > 0 && p.gb_lds && p.nchunk <= 4 && p.tpr < 512) p.max_blocks = 3072;
                if (n_norm_dims > 0 && elem_size == 4 && v > 1 && p.tpr <= 256) {
                    // (Few rows: with 1024 every workgroup of [1024, 4096] has one row instead of one or two -
                    // 9.7 -> 8.3 us; [1536, 4096] 13.1 -> 11.6, [3072, 4096] 20.9 -> 20.5, from 4096 rows on no difference.)
                    if (p.nchunk >= 4) p.max_blocks = (p.rows + p.rpb - 1) / p.rpb > 3072 ? 768 : 1024;
                    else if (p.nchunk == 2) p.max_blocks = 1536;
                }
            } else {
                p.kind = NormKind::RowStream;
                p.tpr = 1024;
                p.rpb = 1;
                if (p.sstride == 2) {  // the streaming kernel gathers stride-2 rows element by element
                    p.vec = 1;
                    p.sstride = 1;
                    p.shift = p.ua_rows = 0;
                }
            }
            return p;
        }
    }
    if (p.norm_in.n == 1 && p.out_axis_stride > 1 && n_norm_dims <= 0) {
        // Softmax over an axis that is not the last: the inner kept dim is contiguous in the output.
        // When it is in the input too, three passes spread over the whole chip: partial statistics
        // (lanes along the inner dim, the axis dealt over wavefronts and workgroups), finalize, apply.
        const int nk = p.kept_in.n;
        const int64_t slab_bytes = p.cols * sa * (int64_t)elem_size, slabs = nk == 2 ? p.kept_in.size[0] : 0;
        const bool is_slab = nk == 2 && max_vec > 1 && p.cols >= 2 && sa == p.kept_in.size[1] && p.kept_in.stride[1] == 1 &&
                             p.kept_out.stride[1] == 1 && p.kept_in.size[1] == p.out_axis_stride &&
                             p.kept_in.stride[0] == p.cols * sa && p.kept_out.stride[0] == p.cols * sa &&
                             ((uintptr_t)in_data % elem_size) == 0 && ((uintptr_t)out_data % elem_size) == 0;
        // One workgroup per slab, the slab in its registers: the fewest threads (a multiple of L / gcd(L, vector) of them
        // take part) that hold it in four vectors each, up to eight of 1024 threads. (Two vectors and twice the threads:
        // f32 [5592, 2000, 3] 49.2 -> 70.2 us, [500, 512, 16] 11.0 -> 13.0, nothing gains more than noise.) Not where the
        // slabs times their threads reach the 2^32 work-items that a launch may have.
        int slab_threads = 0, slab_chunk = 0;
        auto slab_fits = [&]() {
            const int64_t nv = (p.cols * sa + max_vec - 1) / max_vec;
            int64_t g = sa, b = max_vec;
            while (b) { const int64_t t = g % b; g = b; b = t; }
            const int64_t lp = sa / g;
            for (int64_t t = 64; t <= 1024; t <<= 1) {
                const int64_t act = t / lp * lp;
                if (sa > t || act == 0) continue;
                int64_t nc = (nv + act - 1) / act;
                if (nc > 8 || (nc > 4 && t < 1024)) continue;
                if (nc == 5 || nc == 7) ++nc;  // (kernels exist for 1, 2, 3, 4, 6 and 8)
                slab_threads = (int)t;
                slab_chunk = (int)nc;
                return slabs < (1ll << 32) / t;
            }
            return false;
        };
        // A very narrow inner dim. The general forms leave lanes idle or walk an axis serially there, and take three
        // launches below 4 MiB. us before -> slab: f32 [201, 1639, 4] 92 -> 6.3, bf16 [112, 4044, 8] 128 -> 10.0,
        // f16 [112, 3904, 6] 43 -> 8.6, f32 [2048, 128, 2] 17.3 -> 4.1, bf16 [693, 488, 5] 14.4 -> 6.0, f32 [2511, 963, 8]
        // 45 -> 29.5, bf16 [8, 4000, 4] 12.3 -> 6.5. Up to 64 KiB, and to the 128 KiB that fit a workgroup where the alternative
        // is not the flat walk (f32 [32, 4096, 8] 38.8 -> 9.2).
        const bool narrow = is_slab && sa <= 8 && p.cols >= 64 &&
                            slab_bytes <= (slabs * slab_bytes < (8ll << 20) ? (128 << 10) : (64 << 10)) && slab_fits();
        // Small groups laid back to back (a contiguous [batch, cols, L] tensor with cols * L elements of at
        // most 2 KiB: softmax over 4 heads of 64, over the 2 of [N, 2, 3]): lanes along L would idle and a
        // lane per (batch, inner) pair reads single elements at a stride. A workgroup stages 16 KiB of whole
        // groups in LDS with aligned vectors, one lane per pair normalises its column there, and the
        // tile leaves as it came.
        if (nk == 2 && max_vec > 1 && p.cols >= 2 && sa == p.kept_in.size[1] && p.kept_in.stride[1] == 1 &&
            p.kept_out.stride[1] == 1 && p.kept_in.size[1] == p.out_axis_stride &&
            p.kept_in.stride[0] == p.cols * sa && p.kept_out.stride[0] == p.cols * sa &&
            p.cols * sa * (int64_t)elem_size <= 2048 && sa * (int64_t)elem_size < 512 && p.kept_in.size[0] >= 1024 &&
            p.rows * p.cols * (int64_t)elem_size >= (4ll << 20) && (((uintptr_t)in_data | (uintptr_t)out_data) & 15) == 0 &&
            // (a lane walks its column alone: the longer ones are better off with a wavefront per group, as slabs -
            // us: bf16 [5986, 125, 3] 15.1 -> 8.2, f32 [13254, 87, 5] 18.0 -> 13.1; with an inner dim that divides the vector
            // as interleaved rows, below: bf16 [9408, 216, 4] 25.5 -> 9.7)
            !(narrow && (elem_size == 2 ? p.cols > 96 : elem_size == 4 && sa >= 3))) {
            int64_t groups = (16 << 10) / (p.cols * sa * (int64_t)elem_size);
            groups -= groups % max_vec;  // tiles start on 16-byte boundaries
            if (groups >= max_vec) {
                p.kind = NormKind::Col;
                p.inner = p.out_axis_stride;
                p.group_tile = (int)groups;
                p.vec = max_vec;
                return p;
            }
        }
        // Slabs whose inner dim divides the vector (2 or 4 four-byte elements; 2, 4 or 8 two-byte ones; 2 of eight bytes):
        // the slab is a ROW of cols * L elements for the register row kernel, which keeps one maximum and one sum per
        // place in the vector - one read and one write, no round trip through LDS.
        // An inner dim of two vectors (8 four-byte heads, 16 two-byte ones) likewise, where the axis is too long for the
        // register columns (which are faster up to 1024: f32 [2048, 512, 16] 22.1 against 28.3 us; beyond, against the
        // slab and the flat walk, f32 [1000, 2048, 8] 60.0 -> 31.1): a thread's vectors all hold the same places, and
        // only threads two apart are folded together.
        if (nk == 2 && max_vec > 1 && p.cols > 64 && sa > 1 && sa == p.kept_in.size[1] &&
            (max_vec % sa == 0 || (sa == 2 * max_vec && p.cols > 1024) || ((sa == 3 || sa == 5 || sa == 6 || sa == 7) && max_vec % sa != 0)) &&
            p.kept_in.stride[1] == 1 && p.kept_out.stride[1] == 1 && p.kept_in.size[1] == p.out_axis_stride &&
            p.kept_in.stride[0] == p.cols * sa && p.kept_out.stride[0] == p.cols * sa && (p.cols * sa) % max_vec == 0 &&
            p.cols * sa * (int64_t)elem_size <= (128 << 10) && p.kept_in.size[0] >= 256 &&
            p.rows * p.cols * (int64_t)elem_size >= (4ll << 20) && (((uintptr_t)in_data | (uintptr_t)out_data) & 15) == 0) {
            const int64_t shp[2] = {p.kept_in.size[0], p.cols * sa}, str[2] = {p.cols * sa, 1};
            NormPlan q = plan_normalize(in_data, out_data, shp, str, 2, 1, 0, elem_size, fused);
            if (q.kind == NormKind::RowReg && q.vec == max_vec && q.sstride == 1 && !q.shift && !q.tile_rows && !q.gb_lds &&
                !q.lds_rows && !q.raw_rows && q.tpr * max_vec >= sa) {
                if (max_vec % sa == 0 || sa == 2 * max_vec) {
                    q.interleave = (int)sa;
                    return q;
                }
                // An inner dim of 3, 5, 6 or 7: the largest multiple of it of a row's lanes take part, so that all of a
                // lane's vectors start at the same place modulo the inner dim; the lane keeps a (max, sum) per vector
                // place and the places are rotated into softmaxes, folded, and rotated back.
                // (Inputs with an inner dim of 5, 6 or 7 are faster as slabs, us: f32 [4000, 512, 7] 29.3 -> 23.2,
                // f16 [11264, 488, 6] 39.7 -> 25.2, [11008, 576, 5] 44.5 -> 25.3; with 3 there is no difference: f32
                // [5592, 2000, 3] 48.9 and 49.2. The line at 40 MiB is not where the times cross: tests name the plan of smaller
                // ones, f16 [700, 4000, 6] of 32 MiB the largest, and they are faster as slabs as well - that one 32.0 -> 19.4,
                // f32 [2900, 512, 7] 24.2 -> 18.3, [300, 512, 7] 9.8 -> 5.7, f16 [4000, 576, 5] 19.9 -> 13.1.)
                const int64_t act = q.tpr / sa * sa, nvr = p.cols * sa / max_vec;
                const int64_t nc = (nvr + act - 1) / act;
                const bool as_slab = narrow && sa >= 5 && slabs * slab_bytes >= (40ll << 20);
                if (nc <= 8 && !as_slab) {
                    q.interleave = -(int)sa;
                    q.nchunk = (int)nc;
                    return q;
                }
            }
        }
        // Wider ones, at least 256 of them. (Two-byte inner dims of 9 ... 20 elements, and four-byte ones of whole vectors,
        // go either way by a few points and keep the register columns.)
        const bool mid_slab = is_slab && p.cols > 64 && slab_bytes <= (64 << 10) && slabs >= 256 && slabs * slab_bytes >= (4ll << 20) &&
                              sa * (int64_t)elem_size <= ((p.cols > 1024 || (elem_size == 4 && sa % max_vec != 0)) ? (elem_size == 4 && sa % max_vec != 0 ? 48 : 32) : 12);
        if (narrow || (mid_slab && slab_fits())) {
            p.kind = NormKind::Col;
            p.inner = p.out_axis_stride;
            p.slab_tile = slab_threads;
            p.nchunk = slab_chunk;
            p.vec = max_vec;
            return p;
        }
        if (nk >= 1 && nk <= 2 && p.kept_in.stride[nk - 1] == 1 && p.kept_out.stride[nk - 1] == 1 &&
            p.kept_in.size[nk - 1] == p.out_axis_stride && p.kept_in.size[nk - 1] <= (1 << 30) && p.cols <= (1 << 30) &&
            (nk == 1 || p.kept_in.size[0] <= 65535)) {
            const int64_t L = p.kept_in.size[nk - 1];
            const int64_t batch = nk > 1 ? p.kept_in.size[0] : 1;
            // A SHORT axis (softmax over the channels of [B, 21, H, W]): a thread keeps the whole axis of
            // its inner positions in registers, up to 64 registers of raw values: one read, one write.
            // The widest vector that the axis length leaves room for and the layout allows is taken.
            if (p.cols <= 1024 && p.cols > 1) {
                // (two-byte types: vectors of at least 8 bytes, or the loads are too many and too small)
                // (... unless the axis is so short that one thread holds it anyway)
                // (... or the inner dim so narrow that the alternative, lanes along it, would leave most idle:
                // f16 [4097, 12, 96, 5] over axis 2, 0.4 -> 1.3 TB/s)
                bool found = false;
                for (int ev = max_vec; !found && ev >= ((elem_size == 2 && p.cols > 16 && L >= 64) ? 4 : 1); ev /= 2) {
                    const int64_t regs = std::max<int64_t>(1, ev * (int64_t)elem_size / 4);
                    int64_t nc_max = std::min<int64_t>(64, 64 / regs);
                    const size_t vb = (size_t)ev * elem_size;
                    // thread rows that share an inner position when the axis is longer than one thread holds
                    int64_t ty = pow2_ceil((p.cols + nc_max - 1) / nc_max);
                    // A four-byte axis of 257 ... 512 elements fits sixteen thread rows only as 8-byte pieces, i.e.
                    // 128-byte segments of each inner row per workgroup, fetched by sixteen workgroups on eight XCDs at
                    // different moments. With 128 registers of raw values per thread instead of 64 the pieces are whole
                    // vectors and the segments 256 bytes (f32 [512, 512, 512] over axis 0 or 1: 4.8 TB/s before).
                    if (ty > 16 && elem_size == 4 && ev == 4 && p.cols <= 512 && L % 64 == 0) {
                        nc_max = 32;
                        ty = 16;
                    }
                    // Likewise 129 ... 256 elements: eight thread rows of 128 registers read 512-byte segments where sixteen
                    // of 64 read 256-byte ones. f32 [256, 256, 256] over axis 0 / 1, five processes each, us: 26.3-29.1 /
                    // 23.6-28.9 (which end depends on where the allocator put the buffers) -> 25.2-25.7 / 25.2-26.9.
                    // (65 ... 128 elements the same way, four thread rows, lose: C3 [64, 128, 56, 56] over the channels 41.3 -> 44.6 us)
                    if (ty == 16 && nc_max == 16 && elem_size == 4 && ev == 4 && p.cols > 128 && L % 128 == 0) {
                        nc_max = 32;
                        ty = 8;
                    }
                    // enough threads to fill the chip: inner positions x thread rows
                    if (!(ty <= 16 && p.rows / ev * ty >= 8 * 1024)) continue;
                    // (a long axis of two-byte elements that only fits with sixteen thread rows of 4-byte pieces: the
                    // three-pass flat walk is faster, f16 [512, 768, 60] 1.3 -> 2.1 TB/s, [768, 1024, 33] 1.0 -> 2.3;
                    // f32 single elements are not: [2048, 1024, 8] 4.0 against 2.3)
                    if (ty == 16 && elem_size == 2 && ev <= 2 && sa == L && L <= 1024 * max_vec &&
                        batch * p.cols * L * (int64_t)elem_size >= (8ll << 20))
                        continue;
                    if (L % ev == 0 && sa % ev == 0 && (nk == 1 || p.kept_in.stride[0] % ev == 0) &&
                        (p.cols * L) % ev == 0 && ((uintptr_t)in_data % vb) == 0 && ((uintptr_t)out_data % vb) == 0) {
                        p.kind = NormKind::ColReg;
                        p.vec = ev;
                        p.nchunk = (int)nc_max;
                        p.tpr = (int)ty;
                        found = true;
                        continue;
                    }
                    // an inner dim that is not whole, aligned vectors of this width (odd L, odd strides): the
                    // same vectors unaligned beat narrower aligned ones
                    if (ev > 1 && L >= 8 * ev && ((uintptr_t)in_data % elem_size) == 0 && ((uintptr_t)out_data % elem_size) == 0) {
                        p.kind = NormKind::ColReg;
                        p.vec = ev;
                        p.shift = 1;
                        p.nchunk = (int)nc_max;
                        p.tpr = (int)ty;
                        found = true;
                    }
                }
                if (tall_columns(p, found, in_data, out_data, sa, nk > 1 ? p.kept_in.stride[0] : 0, L, batch, elem_size) || found) return p;
            }
            int v = max_vec;
            const bool vec_ok = v > 1 && L % v == 0 && sa % v == 0 && (nk == 1 || p.kept_in.stride[0] % v == 0) &&
                                ((uintptr_t)in_data % 16) == 0 && ((uintptr_t)out_data % 16) == 0;
            if (!vec_ok) v = 1;
            p.kind = NormKind::ColSplit;
            p.vec = v;
            // A narrow inner dim (or one that is not whole vectors) leaves most lanes idle: walk the
            // contiguous [cols, L] slab as a flat array of aligned vectors instead.
            // (Lanes along the inner dim, below, once it is some wavefronts of vectors: one read of the statistics pass deep in
            // flight and stores in address order beat the flat walk's one large workgroup per compute unit. Softmax over axis 0,
            // us, flat and below: f32 128 MiB, inner 1280 75.3 and 71.0, 2048 73.4 and 65.8, 3000 82.3 and 75.1, 1001 81.3 and 77.7; 32 MiB,
            // 512 25.5 and 24.3, 1000 28.3 and 25.3, 2000 29.5 and 23.4, 384 27.1 and 28.4; two-byte 64 MiB, 384 43.5 and 41.9, 600 (a second
            // wavefront that is nearly empty) 48.3 and 50.9, 1024 42.3 and 37.5, 3000 50.8 and 41.2, 1001 48.8 and 43.0; 24 MiB, 320 29.6 and
            // 23.4, 600 28.6 and 25.3, 257 27.7 and 37.8. From 64 MiB on f32 of 512 ... 1024 goes either way (512 72.6 and 69.2, 704 75.0 and 74.3, 1000
            // 74.2 and 75.7, 1024 72.6 and 67.8), and tests name the flat walk there and for odd slabs of 1001.)
            const int64_t all_bytes = batch * p.cols * L * (int64_t)elem_size;
            const int64_t lanes = L / max_vec;
            bool wide = vec_ok && L > 1024 * max_vec;
            if (elem_size == 4) wide = vec_ok ? L > 1024 || (L >= 512 && all_bytes < (64ll << 20)) : L >= 768 && batch == 1;
            else if (elem_size == 2) wide = vec_ok ? L >= 320 && (all_bytes < (44ll << 20) || lanes * 3 >= (lanes + 63) / 64 * 64 * 2) : L >= 768 && batch == 1;
            if (max_vec > 1 && !wide && sa == L && ((uintptr_t)in_data % elem_size) == 0 &&
                ((uintptr_t)out_data % elem_size) == 0 && batch * p.cols * L * (int64_t)elem_size >= (8ll << 20)) {
                // (slabs that start off 16-byte boundaries take the same vectors unaligned: `shift`)
                const bool aligned = ((uintptr_t)in_data % 16) == 0 && ((uintptr_t)out_data % 16) == 0 &&
                                     (batch == 1 || (p.kept_in.stride[0] % max_vec == 0 && (p.cols * L) % max_vec == 0));
                int64_t g = L, b = max_vec;
                while (b) { int64_t t = g % b; g = b; b = t; }
                const int64_t lp = L / g;  // threads per period
                int64_t tmax = std::min<int64_t>(1024, (64 << 10) / (max_vec * (elem_size >= 4 ? 16 : 8)));
                // (each batch slab must be worth at least two periods of the walk: small slabs, of which there
                // are many, take fewer threads each)
                tmax = std::min(tmax, p.cols * L / (2 * max_vec));
                if (lp <= tmax && tmax >= 64) {
                    p.flat_t = (int)(lp * (tmax / lp));
                    p.vec = max_vec;
                    p.shift = aligned ? 0 : 1;
                    const int64_t periods = p.cols * L / ((int64_t)p.flat_t * max_vec);
                    p.tsplit = (int)std::max<int64_t>(1, std::min<int64_t>(periods / 4, std::max<int64_t>(1, 256 / batch)));
                    p.scratch_bytes = (size_t)p.rows * p.tsplit * 16 + (size_t)p.rows * 3 * 8;
                    return p;
                }
            }
            // Inner rows that are not whole, aligned vectors and too wide for the flat walk (an odd inner length of
            // thousands): a lane still takes a vector's worth of neighbouring inner positions, unaligned, instead of one
            // element (a wavefront then reads 1 KiB per axis position, not 128 or 256 bytes). Below a wavefront of vectors
            // the single elements already cover the inner row in one step.
            if (!vec_ok && max_vec > 1 && L >= 64 * max_vec && ((uintptr_t)in_data % elem_size) == 0 &&
                ((uintptr_t)out_data % elem_size) == 0) {
                v = max_vec;
                p.vec = v;
                p.shift = 1;
            }
            // One workgroup per compute unit for the statistics pass (its loads are in flight two batches deep), or the
            // two if they leave fewer units idle (not three: f64 [1344, 8248], 7 and 11 slices, 60.3 and 64.3 us, f32 [1344, 16500] 55.6 and 57.5).
            const int64_t groups = (L + 64 * v - 1) / (64 * v) * batch;
            if (v > 1) {
                p.tsplit = (int)std::min(full_rounds(groups, 2), std::max<int64_t>(1, p.cols / 32));
                // (beyond 64 partials per row the finalize pass grows: 64 columns each then, f32 [8122, 76] 16.3 -> 15.9 us)
                if (p.tsplit > 64) p.tsplit = (int)std::max<int64_t>(64, std::min<int64_t>(p.tsplit, p.cols / 64));
            } else {
                // Single elements, of which a wavefront has little to read and its last lanes often nothing: two workgroups per unit, up to
                // 64 partials per row, 128 or 256 of a long axis (us, full rounds and this: f16 [2056, 271] 10.1 and 9.2, [4270, 268] 12.1 and 11.3, f32 [7353,
                // 79] 14.4 and 13.3, [4100, 63] 64 10.8, 128 11.2; [13675, 122] 64 17.3, 128 16.6; [138341, 11]
                // 128 30.4, 256 26.4, [81669, 10] 22.2 and 20.5, f64 [68163, 15] 31.8 and 29.2).
                p.tsplit = (int)std::max<int64_t>(1, std::min<int64_t>({512 / groups, p.cols / 32, p.cols >= 50000 ? 256 : p.cols >= 10000 ? 128 : 64}));
            }
            p.tpr = elem_size == 2 && v > 1 && p.cols >= 128 * p.tsplit ? 8 : 4;  // wavefronts per workgroup of the statistics pass
            p.scratch_bytes = (size_t)p.rows * p.tsplit * 16 + (size_t)p.rows * 3 * 8;
            return p;
        }
        p.kind = NormKind::Col;
        p.inner = p.out_axis_stride;
        if (p.rows >= 1024) {
            // every lane owns one row; neighbouring lanes are neighbours in memory
            p.tpr = 1;
            p.rpb = 256;
        }
        return p;
    }
    return p;
}

void demote_to_generic(NormPlan& p) {
    p.kind = NormKind::Generic;
    p.raw_rows = 0;
    p.lds_rows = 0;
    p.group_tile = 0;
    p.slab_tile = 0;
    p.gb_lds = 0;
    p.tile_rows = 0;
    p.flat_t = 0;
    p.vec = 1;
    p.shift = 0;
    p.ua_rows = 0;
    p.tall = 0;
    p.sstride = 1;
    p.nchunk = 1;
    p.scratch_bytes = 0;
    p.tpr = (int)std::min<int64_t>(1024, pow2_ceil((p.cols + 3) / 4));
    if (p.tpr > 64 && p.tpr < 256) p.tpr = 256;
    p.rpb = std::max(1, 256 / p.tpr);
}

void restrict_to_row_stream(NormPlan& p) {
    if (p.kind == NormKind::Empty) return;
    const bool rows_on_grid = (p.kind == NormKind::RowReg || p.kind == NormKind::RowStream) && p.vec > 1 &&
                              p.sstride == 1 && !p.shift && p.norm_in.n == 1 && p.norm_in.stride[0] == 1 &&
                              p.out_axis_stride == 1;
    const int vec = rows_on_grid ? p.vec : 1;
    demote_to_generic(p);
    if (!rows_on_grid) return;
    p.kind = NormKind::RowStream;
    p.vec = vec;
    p.tpr = (int)std::min<int64_t>(1024, pow2_ceil((p.cols / vec + 3) / 4));
    if (p.tpr > 64 && p.tpr < 256) p.tpr = 256;
    p.rpb = std::max(1, 256 / p.tpr);
}

std::string describe(const NormPlan& p) {
    static const char* names[] = {"empty", "rowreg", "rowstream", "rowsplit", "col", "col-split", "transposed", "transposed-tile", "col-reg", "generic"};
    char buf[256];
    snprintf(buf, sizeof buf, "%s%s%s rows=%lld cols=%lld vec=%d tpr=%d rpb=%d nchunk=%d ostride=%lld ",
             names[(int)p.kind], p.sstride == 2 ? "-step2" : (p.flat_t ? (p.shift ? "-flat-unaligned" : "-flat") : (p.shift ? ((p.kind == NormKind::RowSplit || p.kind == NormKind::ColReg || p.kind == NormKind::ColSplit || p.kind == NormKind::Transposed || p.kind == NormKind::TransposedTile) ? "-unaligned" : (p.lds_rows ? "-lds-shift" : "-shift")) : (p.gb_lds == 2 ? "-l2gb" : p.gb_lds ? "-ldsgb" : (p.raw_rows ? "-raw" : (p.lds_rows ? "-lds" : ""))))), p.tile_rows ? "+tile" : (p.interleave > 1 ? "-interleaved" : p.interleave < 0 ? "-modular" : p.group_tile ? "-group-tile" : (p.slab_tile ? "-slab" : "")), (long long)p.rows, (long long)p.cols, p.vec, p.tpr, p.rpb,
             p.nchunk, (long long)p.out_axis_stride);
    std::string s = buf;
    if (p.ua_rows) s += "unaligned ";
    if (p.kind == NormKind::ColSplit || p.kind == NormKind::Transposed) s += "split=" + std::to_string(p.tsplit) + " ";
    if (p.kind == NormKind::RowReg) s += "max_blocks=" + std::to_string(p.max_blocks) + " ";  // (layernorm walks its rows)
    describe_dims(s, "rows_in", p.kept_in);
    s += " ";
    describe_dims(s, "norm_in", p.norm_in);
    return s;
}

// ---- elementwise ------------------------------------------------------------------

EwPlan plan_elementwise(const void* out_data, const int64_t* shape, int ndim, int nin, const void* const* in_data,
                        const int64_t* const* in_strides, size_t elem_size, bool allow_transpose) {
    EwPlan p;
    p.nin = nin;
    p.total = 1;
    for (int i = 0; i < ndim; ++i) p.total *= shape[i];
    if (p.total == 0) return p;
    // coalesce: drop size-1 dims; merge dim i into i+1 when every operand (and the
    // contiguous output, which always can) steps over dim i+1 exactly once per step of i
    for (int i = 0; i < ndim; ++i) {
        if (shape[i] == 1) continue;
        bool merge = p.n > 0;
        if (merge) {
            for (int k = 0; k < nin; ++k)
                if (p.stride[k][p.n - 1] != in_strides[k][i] * shape[i]) merge = false;
        }
        if (merge) {
            p.size[p.n - 1] *= shape[i];
            for (int k = 0; k < nin; ++k) p.stride[k][p.n - 1] = in_strides[k][i];
        } else {
            if (p.n == kMaxDims)
                fail(HPT_ERR_SHAPE, "elementwise: the view does not coalesce to %d dims or fewer", kMaxDims);
            p.size[p.n] = shape[i];
            for (int k = 0; k < nin; ++k) p.stride[k][p.n] = in_strides[k][i];
            ++p.n;
        }
    }
    if (p.n == 0) {  // a single element
        p.n = 1;
        p.size[0] = 1;
        for (int k = 0; k < nin; ++k) p.stride[k][0] = 1;
    }
    p.kind = EwKind::Inner;
    const int full = (int)(16 / elem_size);
    const int last = p.n - 1;
    auto aligned = [&](const void* ptr) { return ((uintptr_t)ptr % 16) == 0; };
    // vectors along the innermost dim: every operand is either contiguous there (stride 1,
    // with 16-byte aligned base and outer strides) or broadcast there (stride 0)
    bool vec_ok = full > 1 && p.size[last] % full == 0 && aligned(out_data);
    for (int k = 0; k < nin && vec_ok; ++k) {
        const int64_t s = p.stride[k][last];
        if (s == 1) {
            if (!aligned(in_data[k])) vec_ok = false;
            for (int i = 0; i < last; ++i)
                if (p.stride[k][i] % full != 0) vec_ok = false;
        } else if (s != 0) {
            vec_ok = false;
        }
    }
    if (vec_ok) {
        p.vec = full;
        return p;
    }
    // copy of a view whose innermost stride is 2: full vectors in, the even positions kept
    if (nin == 1 && full > 1 && p.stride[0][last] == 2 && p.size[last] % full == 0 && aligned(out_data) &&
        aligned(in_data[0])) {
        bool ok = true;
        for (int i = 0; i < last; ++i)
            if (p.stride[0][i] % full != 0) ok = false;
        if (ok) {
            p.vec = full;
            p.sstride = 2;
            return p;
        }
    }
    // copy of a view whose contiguous dim is not the innermost one: transpose in registers
    if (allow_transpose && nin == 1 && full > 1 && p.stride[0][last] != 1 && p.stride[0][last] != 0) {
        int t = -1;
        for (int i = 0; i < last; ++i)
            if (p.stride[0][i] == 1) t = i;
        if (t >= 0 && p.n <= 6) {
            bool ok = aligned(out_data) && aligned(in_data[0]) && p.size[last] % full == 0 && p.size[t] % full == 0 &&
                      p.size[last] >= 2 * full && p.size[t] >= 2 * full && p.size[last] <= (1 << 30) &&
                      p.size[t] <= (1 << 30);
            for (int i = 0; i < p.n; ++i)
                if (i != t && p.stride[0][i] % full != 0) ok = false;
            // the remaining dims ride on blockIdx.z
            int64_t others = 1;
            for (int i = 0; i < p.n; ++i)
                if (i != t && i != last) others *= p.size[i];
            if (ok && others <= 65535) {
                p.kind = EwKind::Transpose;
                p.vec = full;
                p.tdim = t;
                p.tmask = 1;
                p.tile_lds = p.size[last] >= 16 * full && p.size[t] >= 16 * full;
            }
        }
    }
    // binary op with an operand (or both) whose contiguous dim is not the innermost one (a + b.t()): whole
    // tiles of those operands are transposed through LDS; an operand in the output's own layout (or
    // broadcast along the innermost dim) is read as the result is written
    if (allow_transpose && nin == 2 && full > 1 && full <= 8 && p.n <= 6) {
        int mask = 0;
        for (int k = 0; k < 2; ++k)
            if (p.stride[k][last] != 1 && p.stride[k][last] != 0) mask |= 1 << k;
        int t = -1;
        for (int i = 0; i < last && mask; ++i) {
            bool all = true;
            for (int k = 0; k < 2; ++k)
                if ((mask >> k & 1) && p.stride[k][i] != 1) all = false;
            if (all) t = i;
        }
        if (t >= 0) {
            bool ok = aligned(out_data) && p.size[last] % full == 0 && p.size[t] % full == 0 && p.size[last] >= 16 * full &&
                      p.size[t] >= 16 * full && p.size[last] <= (1 << 30) && p.size[t] <= (1 << 30);
            for (int k = 0; k < 2 && ok; ++k) {
                const bool transposed = mask >> k & 1;
                if (!transposed && p.stride[k][last] == 0) continue;  // single elements, splat
                if (!aligned(in_data[k])) ok = false;
                for (int i = 0; i < p.n; ++i)
                    if (i != (transposed ? t : last) && p.stride[k][i] % full != 0) ok = false;
            }
            int64_t others = 1;
            for (int i = 0; i < p.n; ++i)
                if (i != t && i != last) others *= p.size[i];
            if (ok && others <= 65535) {
                p.kind = EwKind::Transpose;
                p.vec = full;
                p.tdim = t;
                p.tmask = mask;
                p.tile_lds = true;
            }
        }
    }
    return p;
}

std::string describe(const EwPlan& p) {
    static const char* names[] = {"empty", "inner", "transpose"};
    char buf[128];
    snprintf(buf, sizeof buf, "%s%s vec=%d total=%lld dims=[", names[(int)p.kind], p.sstride == 2 ? "-step2" : "", p.vec,
             (long long)p.total);
    std::string s = buf;
    for (int i = 0; i < p.n; ++i) {
        snprintf(buf, sizeof buf, "%s%lld:", i ? "," : "", (long long)p.size[i]);
        s += buf;
        for (int k = 0; k < p.nin; ++k) {
            snprintf(buf, sizeof buf, "%s%lld", k ? "/" : "", (long long)p.stride[k][i]);
            s += buf;
        }
    }
    s += "]";
    if (p.kind == EwKind::Transpose) {
        snprintf(buf, sizeof buf, " tdim=%d%s%s", p.tdim, p.nin == 2 ? (p.tmask == 3 ? " both" : p.tmask == 1 ? " lhs" : " rhs") : "",
                 p.tile_lds ? " lds" : "");
        s += buf;
    }
    return s;
}

}  // namespace hpt
