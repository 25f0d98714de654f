// Rows of doubles.  The reference's dtype dispatch admits double (src/ops/all_reduce_fusion.cpp:29-33, two
// elements per 16-byte vector); what must come out is what its torch-eager composition computes for double
// tensors (test/test_all_reduce_fusion.py:23-28,75):
//   x   = ((0 + p_0) + ... + p_{N-1}) + residual_in        all in double, rank order          -> residual_out
//   rs  = 1 / sqrt( sum(float(x)^2) / H + eps )             fp32: RMSNorm.forward squares x.float()
//   y   = gamma * (x * double(rs))                          double                              -> norm_out
// No quantized output for this type.  One or four 16-byte vectors per thread as planned (vecs_per_thread_f64 says which and what
// it measured), two only on request (tune_vecs_per_thread); the row kernel's geometry and XCD-aware row mapping.  Bound by
// memory: 4 x [2048, 2048] moves 235 MB.  As in the row kernel the partials are added as they arrive and gamma of several
// vectors is requested once the row's registers are free; residual_out is stored as soon as it is known, or with the row's
// other output in launches of few bytes (kEarlyStoreBytes).  N == 0: the sum was staged (part[0] holds it), as in the row
// kernel; reduce_kernel_f64 is that stage A.  With a stage the sums are stored to it; OWNED sums rows == owner (mod N) only
// and reads the others' sums from the stage.
#include <hip/hip_runtime.h>

#include "tde_rows.h"

namespace tde {

__device__ __forceinline__ void unpack_f64(u32x4 raw, double (&d)[2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t lo = raw[2 * i], hi = raw[2 * i + 1]; // copied to scalars before the bit cast
        const uint64_t w = ((uint64_t)hi << 32) | lo;
        d[i] = __builtin_bit_cast(double, w);
    }
}

__device__ __forceinline__ u32x4 pack_f64(const double (&d)[2]) {
    u32x4 raw;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint64_t w = __builtin_bit_cast(uint64_t, d[i]);
        raw[2 * i] = (uint32_t)w;
        raw[2 * i + 1] = (uint32_t)(w >> 32);
    }
    return raw;
}

// residual_out is stored as soon as it is known in launches whose rows together have this many bytes, and with the normed row
// in shorter ones, whose rows are all in flight at once and should finish loading first.  Late against early, four vectors
// per thread: 2 x 300 rows of 2048 -10 %, 2 x 900 of 1024 -11 %, 4 x 900 of 600 -10 %; 4 x 2048 rows of 2048 +3.3 %, 8 x 2048 of 600 +2.8 %.
constexpr int64_t kEarlyStoreBytes = 9 << 20;

template <int N, int VPT, int FORM = kFormPlain, bool SHIFTED = false>
__global__ void __launch_bounds__(1024 / VPT) row_kernel_f64(const RowArgs a) {
    constexpr bool OWNED = FORM == kFormOwned, STAGED = FORM == kFormStaged;
    constexpr int NP = (N == 0) ? 1 : N;
    extern __shared__ __attribute__((aligned(16))) float lds_dyn[]; // squares (two per vector), then block sums
    float *const lds_img = lds_dyn;
    float *const lds_bs = lds_dyn + (uint32_t)a.threads_per_row * a.rows_per_block * (VPT * 2);
    const int tid = threadIdx.x;
    const int tpr = a.threads_per_row;
    const int group = a.row_group(__builtin_amdgcn_readfirstlane(tid >> 6));
    int t = tid - group * tpr; // of the row group; of SHIFTED rows the row's first vector of this thread, as soon as the row is known
    const uint32_t row_bytes = (uint32_t)a.hidden() * 8u;
    uint32_t off[VPT];
#pragma unroll
    for (int j = 0; j < VPT; ++j) off[j] = (uint32_t)(j * tpr + t) * 16u;

    const void *part[NP];
    partial_addresses(a, a.address(kPtrStage), part);
    const rsrc_t gamma_rsrc = row_rsrc(a.ptr(kPtrGamma), 0, row_bytes);

    // the grid covers every row; each XCD takes runs of consecutive row groups (xcd_chunked_block)
    int64_t row = (int64_t)xcd_chunked_block(blockIdx.x, a.chunked_blocks, a.xcd_chunk) * a.rows_per_block + group;

    bool sum_is_new = STAGED;
    if constexpr (OWNED) row = owned_first_row<N>(row, a.tokens, a.owner, sum_is_new);
    const uint32_t bytes = (row < a.tokens) ? row_bytes : 0u;
    const int64_t row_byte = row * (int64_t)row_bytes;
    const int shift = SHIFTED ? a.row_shift(row_byte) : 0;
    if constexpr (SHIFTED) {
        t = first_vector_of<true>(t, shift, tpr);
#pragma unroll
        for (int j = 0; j < VPT; ++j) off[j] = (uint32_t)(j * tpr + t) * 16u;
    }
    const auto load_row = [&](const void *base, u32x4(&v)[VPT]) {
        const rsrc_t rs = row_rsrc(base, row_byte, bytes);
#pragma unroll
        for (int j = 0; j < VPT; ++j) v[j] = rsrc_load16(rs, off[j]);
    };
    u32x4 praw[NP][VPT], rraw[VPT], graw[VPT];
    if (!OWNED || sum_is_new) {
#pragma unroll
        for (int r = 0; r < NP; ++r) load_row(part[r], praw[r]);
    } else {
        load_row(a.ptr(kPtrStage), praw[0]);
    }
    load_row(a.ptr(kPtrResidualIn), rraw);
    const auto load_gamma = [&] {
#pragma unroll
        for (int j = 0; j < VPT; ++j) graw[j] = __builtin_amdgcn_raw_buffer_load_b128(gamma_rsrc, (int)off[j], 0, kAuxDefault);
    };
    if constexpr (VPT == 1) load_gamma();
    else __builtin_amdgcn_sched_barrier(0);

    const SumLayout<VPT, 2, false> sums(lds_img, lds_bs, a.hidden(), tpr, a.rows_per_block, group);
    sumsq_clear(sums, t);
    const RowLength<> length(a.hidden());

    // The partials are summed rank by rank, as they arrive.
    double acc[VPT][2];
    if (N == 0 || (OWNED && !sum_is_new)) {
#pragma unroll
        for (int j = 0; j < VPT; ++j) unpack_f64(praw[0][j], acc[j]); // the staged sum
    } else {
#pragma unroll
        for (int r = 0; r < N; ++r) {
#pragma unroll
            for (int j = 0; j < VPT; ++j) {
                double p[2];
                unpack_f64(praw[r][j], p);
                acc[j][0] = (r == 0 ? 0.0 : acc[j][0]) + p[0];
                acc[j][1] = (r == 0 ? 0.0 : acc[j][1]) + p[1];
            }
            if constexpr (VPT > 1) __builtin_amdgcn_sched_barrier(0);
        }
    }
    double x[VPT][2];
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        double res[2];
        unpack_f64(rraw[j], res);
        x[j][0] = acc[j][0] + res[0];
        x[j][1] = acc[j][1] + res[1];
    }
    const bool early = a.tokens * (int64_t)row_bytes >= kEarlyStoreBytes;
    const auto store_row = [&](const void *base, const double(&v)[VPT][2]) {
        const rsrc_t rs = row_rsrc(base, row_byte, bytes);
#pragma unroll
        for (int j = 0; j < VPT; ++j) rsrc_store16(rs, off[j], pack_f64(v[j]));
    };
    const auto store_sums = [&] {
        if (sum_is_new) store_row(a.ptr(kPtrStage), acc);
        if (early) store_row(a.ptr(kPtrResidualOut), x);
    };
    // Behind the request for gamma: what a wavefront loads is waited for behind the stores it issued before.
    if constexpr (VPT == 1) store_sums();
    uint32_t landed = 0;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const float f0 = (float)x[j][0], f1 = (float)x[j][1];
        const float sq[2] = {f0 * f0, f1 * f1};
        landed = __builtin_bit_cast(uint32_t, sq[0]);
        put_squares(sums.img + (j * tpr + (VPT == 1 ? t : not_before(t, landed))) * 2, sq);
    }
    if (sums.n != sums.chained) {
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            const float f0 = (float)x[j][0], f1 = (float)x[j][1];
            const float sq[2] = {f0 * f0, f1 * f1};
            split_left(sums, j * tpr + t, sq);
        }
    }
    if constexpr (VPT > 1) {
        __builtin_amdgcn_sched_barrier(0);
        load_gamma();
        store_sums();
    }
    const int t_behind = thread_of<SHIFTED>(VPT == 1 ? t : not_before(t, landed), shift, tpr);
    const float sumsq = sumsq_torch_order<SHIFTED>(sums, t_behind, tpr, 0, t_behind & (kWave - 1));
    const float rs = reciprocal_rms(sumsq, length, a.eps);

    const rsrc_t norm_out = row_rsrc(a.ptr(kPtrNorm), row_byte, bytes);
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        double g[2], y[2];
        unpack_f64(graw[j], g);
        y[0] = g[0] * (x[j][0] * (double)rs);
        y[1] = g[1] * (x[j][1] * (double)rs);
        rsrc_store16(norm_out, off[j], pack_f64(y));
    }
    if (!early) store_row(a.ptr(kPtrResidualOut), x);
}

// Stage A for doubles: the reduce kernel's spans (ReduceSpan), sums in double from +0 in rank order.
template <int N, int U>
__global__ void __launch_bounds__(256) reduce_kernel_f64(const RowArgs a, const ReduceSpan sp) {
    constexpr uint32_t SPAN = 256u * U * 16u; // bytes per workgroup
    const void *part[N];
    partial_addresses(a, sp.table, part);
    const int64_t bid = xcd_chunked_block(blockIdx.x, sp.chunked_blocks, sp.xcd_chunk);
    const int64_t k = bid / sp.spans_per_row;
    const int64_t in_row = (bid - k * sp.spans_per_row) * SPAN;
    const int64_t base = (sp.first_row + k * sp.row_step) * sp.row_bytes + in_row;
    const int64_t left = sp.row_bytes - in_row;
    const uint32_t bytes = left < (int64_t)SPAN ? (uint32_t)left : SPAN;
    u32x4 raw[U][N];
#pragma unroll
    for (int r = 0; r < N; ++r) {
        const rsrc_t rs = row_rsrc(part[r], base, bytes);
#pragma unroll
        for (int u = 0; u < U; ++u) raw[u][r] = rsrc_load16(rs, (uint32_t)(u * 256 + threadIdx.x) * 16u);
    }
    const rsrc_t out = row_rsrc(a.ptr(kPtrStage), base, bytes);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        double acc[2] = {0.0, 0.0};
#pragma unroll
        for (int r = 0; r < N; ++r) {
            double p[2];
            unpack_f64(raw[u][r], p);
            acc[0] += p[0];
            acc[1] += p[1];
        }
        __builtin_amdgcn_raw_buffer_store_b128(pack_f64(acc), out, (int)((u * 256 + threadIdx.x) * 16), 0, kAuxDefault);
    }
}

hipError_t launch_reduce_f64(int n, const RowArgs &a, uint64_t table, int64_t row_bytes, int64_t first_row, int64_t row_step, int64_t rows,
                             hipStream_t s) {
    constexpr int U = 4;
    constexpr int64_t span = 256 * U * 16;
    ReduceSpan sp{row_bytes, first_row, row_step, (row_bytes + span - 1) / span, rows == 1 ? 16u : 1u, 0u, table};
    const int64_t blocks = rows * sp.spans_per_row;
    if (blocks <= 0) return hipSuccess;
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;
    sp.chunked_blocks = chunked_blocks(blocks, sp.xcd_chunk);
    const dim3 grid((unsigned)blocks), block(256);
    switch (n) {
    case 2: return launch_kernel<reduce_kernel_f64<2, U>>(grid, block, 0, s, a, sp);
    case 4: return launch_kernel<reduce_kernel_f64<4, U>>(grid, block, 0, s, a, sp);
    case 8: return launch_kernel<reduce_kernel_f64<8, U>>(grid, block, 0, s, a, sp);
    }
    return hipErrorInvalidValue;
}

template <int N, int VPT, bool SHIFTED = false>
hipError_t launch_rows_f64_nv(const RowArgs &a, const Geometry &g, hipStream_t s) {
    const dim3 grid((unsigned)g.grid), block((unsigned)g.block_threads);
    const size_t lds = (size_t)g.lds_bytes; // sumsq_lds_bytes(g.block_threads, VPT, 2): doubles are never limited per CU
    if constexpr (N != 0) {
        if (!SHIFTED && a.line_mask != 0) return launch_rows_f64_nv<N, VPT, true>(a, g, s);
        if (g.form == kFormOwned) return launch_kernel<row_kernel_f64<N, VPT, kFormOwned, SHIFTED>>(grid, block, lds, s, a);
        if (g.form == kFormStaged) return launch_kernel<row_kernel_f64<N, VPT, kFormStaged, SHIFTED>>(grid, block, lds, s, a);
    }
    return launch_kernel<row_kernel_f64<N, VPT, kFormPlain, SHIFTED>>(grid, block, lds, s, a);
}

template <int N>
hipError_t launch_rows_f64_n(const RowArgs &a, const Geometry &g, hipStream_t s) {
    switch (g.vpt) {
    case 1: return launch_rows_f64_nv<N, 1>(a, g, s);
    case 2: return launch_rows_f64_nv<N, 2>(a, g, s);
    case 4: return launch_rows_f64_nv<N, 4>(a, g, s);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_rows_f64(int n, const RowArgs &a, const Geometry &g, hipStream_t s) {
    switch (n) {
    case 0: return launch_rows_f64_n<0>(a, g, s);
    case 2: return launch_rows_f64_n<2>(a, g, s);
    case 4: return launch_rows_f64_n<4>(a, g, s);
    case 8: return launch_rows_f64_n<8>(a, g, s);
    }
    return hipErrorInvalidValue;
}

} // namespace tde
