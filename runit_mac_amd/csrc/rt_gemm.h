// rt_gemm.h — what the batched GEMMs of k_gemm.hip and k_gemmw.hip share: the
// inputs their activation preparations take and the K-split partial sums.
#pragma once
#include "rt_device.h"
#include "rt_shared.h"

// The row of a preparation given as the K-split partial sums of the GEMM
// that produced it ([chunk][split][crow][K], as k_gemm_split_sum reads
// them): x = Σ part (SILU: silu(Σ part)·Σ part2), then res + x; written to y
// when given.
struct PrepSum {
    const float* part;
    const float* part2;
    const float* res;
    float* y;
    uint32_t splits, crow;
    uint32_t full, nch;  // wide GEMM: its first `full` tiles are unsplit (wide_splits)
};

// p[0] + p[ss] + ... (splits terms, in order), four loads in flight (a loop
// that waited for each took 8.7 µs at 16 splits of 37×3584)
RT_DEV f32x4 split_add(const float* __restrict__ p, size_t ss, uint32_t splits) {
    f32x4 v = *(const f32x4*)p, t1, t2, t3;
    for (uint32_t sp = 1; sp < splits; sp += 4) {
        const uint32_t r = splits - sp;
        const float* q = p + sp * ss;
        const f32x4 t0 = *(const f32x4*)q;
        if (r > 1) t1 = *(const f32x4*)(q + ss);
        if (r > 2) t2 = *(const f32x4*)(q + 2 * ss);
        if (r > 3) t3 = *(const f32x4*)(q + 3 * ss);
        v += t0;
        if (r > 1) v += t1;
        if (r > 2) v += t2;
        if (r > 3) v += t3;
    }
    return v;
}

// K splits of the 256-column tile that holds column n of chunk ch in the
// partial sums of a wide GEMM (k_gemmw.hip): tiles in the order [column tile]
// [chunk], the first `full` of them unsplit.
RT_DEV uint32_t wide_splits(uint32_t full, uint32_t splits, uint32_t n, uint32_t tile, uint32_t nch, uint32_t ch) {
    return n / tile * nch + ch < full ? 1 : splits;
}

// The row of a preparation given as the split partials of the multi-query
// attention (k_attn_mq_f32_hd*, parts-only, one sequence): element (head h,
// d) of row r is column qi = r·G + h mod G of KV head h / G, merged over the
// nsp key ranges as that kernel's last workgroup merges them.
struct PrepAttn {
    const float* part;
    const float* ml;
    uint32_t nsp, G, hd, cgs;
};
