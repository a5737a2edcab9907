// Softmax over the middle axis of contiguous [batch, C, L] slabs with a narrow L, one workgroup per slab.
#pragma once
#include "norm_kernels.hpp"

namespace hpt {

// The slab is read as a flat array of 16-byte vectors, unaligned where it starts off the grid; the `act` threads that
// take part are a multiple of L / gcd(L, VEC), so every place of a thread's vectors stays on one column (an inner
// index) for the whole walk. A thread keeps its NC vectors in registers and a running maximum, then a sum, per place;
// a workgroup's places meet in LDS, where groups of 2^g_log2 lanes share a column. One read and one write, whole
// vectors, no per-element walk through LDS at stride L (which bounded the form before: three dependent loops over the
// axis per column). Bound by latency up to a few MB - load, two folds, store - and by memory beyond.
// us, softmax over C of [batch, C, L], staged slab -> now: bf16 [432, 2596, 8] 32 -> 14.4, bf16 [640, 3286, 6] 41 -> 19.5,
// f32 [2240, 1408, 8] 80 -> 38.1 (5.3 TB/s), f32 [2688, 1931, 6] 85 -> 46.8 (5.3 TB/s), f32 [1024, 3692, 3] 36 -> 21.8.
template <int KIND, class T, int NC>
__global__ void __launch_bounds__(1024) norm_slab_kernel(const T* in, T* outp, int C, int L, int act, int g_log2) {
    static_assert(KIND == NORM_SOFTMAX || KIND == NORM_LOGSOFTMAX, "a softmax kernel");
    using CT = typename Elem<T>::Wide;
    using ST = typename StatType<T>::type;
    constexpr int VEC = 16 / sizeof(T);
    constexpr bool kLog = norm_is_log(KIND);
    constexpr bool kKeepExp = !kLog && sizeof(T) == sizeof(CT);  // exp(x - max) fits back into the vectors
    extern __shared__ __align__(16) unsigned char smem_raw[];
    ST* slots = reinterpret_cast<ST*>(smem_raw);                 // act * VEC places
    CT* maxs = reinterpret_cast<CT*>(slots + act * VEC);         // L columns
    CT* norms = maxs + L;
    CT* mslots = reinterpret_cast<CT*>(slots);

    const int t = threadIdx.x;
    const int n = C * L;
    const T* src = in + (int64_t)blockIdx.x * n;
    T* dst = outp + (int64_t)blockIdx.x * n;
    const int nvec = n / VEC, tail = n - nvec * VEC;
    const bool on = t < act;

    // every load goes out, from an index clamped into the slab
    Pack<T, VEC> v[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) v[c] = load_pack_unaligned<T, VEC>(src + (int64_t)min(t + c * act, nvec - 1) * VEC);
    const int tail_t = nvec % act, tail_c = nvec / act;
    if (tail) {  // the last, partial vector: places past the end hold -inf, which adds nothing
        Pack<T, VEC> e;
#pragma unroll
        for (int j = 0; j < VEC; ++j) e.v[j] = src[min(nvec * VEC + j, n - 1)];
#pragma unroll
        for (int j = 0; j < VEC; ++j) e.v[j] = j < tail ? e.v[j] : Elem<T>::narrow(neg_inf<CT>());
#pragma unroll
        for (int c = 0; c < NC; ++c)
            if (c == tail_c && t == tail_t) v[c] = e;
    }
    const int last = nvec + (tail ? 1 : 0);  // vectors that count
    bool ok[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) ok[c] = on && t + c * act < last;

    // Fold the places of column `col` over the workgroup: slot p holds column p % L.
    const int fold_col = t >> g_log2, fold_lane = t & ((1 << g_log2) - 1), rows = act * VEC / L;
    CT m[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) m[j] = neg_inf<CT>();
#pragma unroll
    for (int c = 0; c < NC; ++c)
        if (ok[c]) {
#pragma unroll
            for (int j = 0; j < VEC; ++j) m[j] = MaxC<CT>::comb(m[j], Elem<T>::widen(v[c].v[j]));
        }
    if (on) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) mslots[t * VEC + j] = m[j];
    }
    __syncthreads();
    if (fold_col < L) {
        CT r = neg_inf<CT>();
        for (int q = fold_lane; q < rows; q += 1 << g_log2) r = MaxC<CT>::comb(r, mslots[q * L + fold_col]);
        r = group_reduce<MaxC<CT>>(r, 1 << g_log2);
        if (fold_lane == 0) maxs[fold_col] = r;
    }
    __syncthreads();
    int col[VEC];
    col[0] = t * VEC % L;
#pragma unroll
    for (int j = 1; j < VEC; ++j) col[j] = col[j - 1] + 1 == L ? 0 : col[j - 1] + 1;
    ST s[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
        m[j] = maxs[col[j]];
        s[j] = 0;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
        if (ok[c]) {
#pragma unroll
            for (int j = 0; j < VEC; ++j) {
                const CT e = exp_ct<T>(Elem<T>::widen(v[c].v[j]) - m[j]);
                s[j] += (ST)e;
                if constexpr (kKeepExp) v[c].v[j] = Elem<T>::narrow(e);
            }
        }
    if (on) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) slots[t * VEC + j] = s[j];
    }
    __syncthreads();
    if (fold_col < L) {
        ST r = 0;
        for (int q = fold_lane; q < rows; q += 1 << g_log2) r += slots[q * L + fold_col];
        r = group_reduce<SumC<ST>>(r, 1 << g_log2);
        if (fold_lane == 0) norms[fold_col] = kLog ? log_ct<T>((CT)r) : (CT)1 / (CT)r;
    }
    __syncthreads();
    CT k[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) k[j] = norms[col[j]];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        if (!ok[c]) continue;
        Pack<T, VEC> o;
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            const CT x = Elem<T>::widen(v[c].v[j]);
            CT y;
            if constexpr (kLog) y = (x - m[j]) - k[j];
            else if constexpr (kKeepExp) y = x * k[j];
            else y = exp_ct<T>(x - m[j]) * k[j];
            o.v[j] = Elem<T>::narrow(y);
        }
        const int iv = t + c * act;
        if (iv < nvec) {
            store_pack_unaligned_stream<T, VEC>(dst + (int64_t)iv * VEC, o);
        } else {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                if (j < tail) dst[nvec * VEC + j] = o.v[j];
        }
    }
}

}  // namespace hpt
