// Rows of up to 32 16-byte vectors (256 elements of 2 bytes, 128 floats): two or four of them share a wavefront.
//
// row_kernel gives every row wavefronts of its own, and what bounds it on many short rows is the instructions of those
// wavefronts (some 400 to 800 each, whatever their lanes hold), not memory.  Here a row takes a slot of 32 lanes, or of 16 up to 16
// vectors, one vector per lane, and everything that a row's lanes exchange stays inside the wavefront: no workgroup
// barrier.  The arithmetic is row_kernel's step by step, the sum of squares in torch's order included.
//
// us per launch, one row to a wavefront -> here: 2 x [53362, 120] bf16 -> fp8 26.2 -> 17.0, 4 x [26063, 120] 14.3 -> 9.6, 8 x [15262, 128]
// 10.3 -> 8.9 (4.5 TB/s), 2 x [31761, 192] 14.7 -> 11.2, 8 x [3958, 72] fp16 -> int8 5.2 -> 3.9, 2 x [25, 36] fp32 3.2 -> 2.7.
// Four wavefronts to a workgroup with slots of 16 lanes, two with slots of 32 (1 % over four: less of a buffer in one piece, shorter
// queues); chunks of the XCD mapping from 4 to 64 workgroups measure the same within 1 %, launch order 2 % more.
#include "tde_rows.h"

namespace tde {

namespace {

// Lane n of each 16-lane row, in all of them.
template <int n>
__device__ __forceinline__ float row16_lane(float v) {
    return dpp_move<0x150 + n>(v); // row_newbcast
}

// The sum of a row's squares in the order that sumsq_torch_order (tde_rows.h) describes.  A row of up to 256 floats is one block:
// chain (m, k) has up to eight terms, and each 16-lane row sums all 32 chains, lane 4m + k both (m, k) and (m + 4, k), so a
// slot of 32 lanes does it twice and nothing crosses 16-lane rows.
//   img   the slot's squares, one float per element it holds
//   left  the floats from `chained` to n, whose places in img hold zeros
template <int VECF>
__device__ __forceinline__ float slot_sum(const float *img, const float *left, int n, int chained, int slot, int lane) {
    constexpr int TERMS = VECF; // of a chain, with 32 lanes; half of them with 16
    const int m = lane >> 2 & 3, k = lane & 3;
    const float *src = img + 8 * k + m;
    float lo = src[0], hi = src[4];
#pragma unroll
    for (int i = 1; i < TERMS / 2; ++i) {
        lo += src[32 * i];
        hi += src[32 * i + 4];
    }
    if (slot == 32) {
#pragma unroll
        for (int i = TERMS / 2; i < TERMS; ++i) {
            lo += src[32 * i];
            hi += src[32 * i + 4];
        }
    }
    float p = quad_bcast<0x00>(lo), q = quad_bcast<0x00>(hi); // of vector lanes m and m + 4
    float sum = 0.0f;                                         // the scalars left over
    if (n != chained) {
        const int vectors = n >> 3 & 3;
        for (int l = 0; l < vectors; ++l) {
            p += left[8 * l + m];
            q += left[8 * l + m + 4];
        }
        if constexpr (VECF != 8) {
            if (n < 8) { // four scalars: four interleaved sums of one each
                sum = left[0] + left[1];
                sum += left[2];
                sum += left[3];
            } else {
                for (int e = n & ~7; e < n; ++e) sum += left[e - chained];
            }
        }
    }
    p += quad_bcast<0x55>(lo);
    q += quad_bcast<0x55>(hi);
    p += quad_bcast<0xAA>(lo);
    q += quad_bcast<0xAA>(hi);
    p += quad_bcast<0xFF>(lo);
    q += quad_bcast<0xFF>(hi);
    sum = VECF == 8 ? row16_lane<0>(p) : sum + row16_lane<0>(p);
    sum += row16_lane<4>(p);
    sum += row16_lane<8>(p);
    sum += row16_lane<12>(p);
    sum += row16_lane<0>(q);
    sum += row16_lane<4>(q);
    sum += row16_lane<8>(q);
    sum += row16_lane<12>(q);
    return sum;
}

// Maximum over the lanes of a slot, or of a group of them.
__device__ __forceinline__ uint32_t lanes_max(uint32_t v, int lanes) {
    v = row16_max(v);
    if (lanes == 32) v = max_u32(v, (uint32_t)__shfl_xor((int)v, 16, kWave));
    return v;
}

// E, N, Q, FORM as in row_kernel (kFormPlain, kFormStaged or kFormOwned); T-typed rows are written where the launch has a buffer for
// them.  a.threads_per_row is the slot, a.rows_per_block a multiple of the rows of a wavefront.
template <class E, int N, int Q, int FORM>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) short_row_kernel(const RowArgs a) {
    constexpr bool OWNED = FORM == kFormOwned;
    constexpr int VEC = E::VEC;
    constexpr int NP = (N == 0) ? 1 : N;
    // Dynamic LDS: the workgroup's squares (one float per element it holds), then 32 floats per row for what the chains leave.
    extern __shared__ __attribute__((aligned(16))) float lds_dyn[];

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int slot = a.threads_per_row;
    const int slot_shift = slot == 32 ? 5 : 4;
    const int rows = kWave >> slot_shift; // of this wavefront
    const int in_slot = lane & (slot - 1), nth = lane >> slot_shift;
    const int hidden = a.hidden();
    const uint32_t row_bytes = (uint32_t)hidden * E::BYTES;

    const void *part[NP];
    partial_addresses(a, a.address(kPtrStage), part);

    // Everything is addressed from the wavefront's first row on, with owned rows (whose order is another) from the first of their
    // window on: `place` is the row of this lane from there, `held` how many rows there are from there.
    const int64_t first = (int64_t)xcd_chunked_block(blockIdx.x, a.chunked_blocks, a.xcd_chunk) * a.rows_per_block + wave * rows;
    int64_t base = first;
    uint32_t place = (uint32_t)nth;
    bool sum_is_new = FORM == kFormStaged;
    constexpr int WINDOW = kOwnedRun * (N == 0 ? 1 : N); // whole wavefronts
    if constexpr (OWNED) {
        base = first / WINDOW * WINDOW;
        place = (uint32_t)(owned_first_row<N>(first + nth, a.tokens, a.owner, sum_is_new) - base);
    }
    const int64_t left_rows = a.tokens - base;
    const int64_t most = OWNED ? WINDOW : rows;
    const uint32_t held = left_rows <= 0 ? 0u : (uint32_t)(left_rows < most ? left_rows : most);
    const bool here = place < held && (uint32_t)in_slot * 16u < row_bytes;
    const uint32_t off = here ? place * row_bytes + (uint32_t)in_slot * 16u : kPastEnd;
    const int64_t base_byte = base * (int64_t)row_bytes;
    const uint32_t bytes = held * row_bytes;

    // ---- loads: all of them ahead of the first addition ----------------------------------------------
    u32x4 p[NP], staged = u32x4{0, 0, 0, 0};
    bool any_new = true;
    if constexpr (OWNED) {
        staged = rsrc_load16(row_rsrc(a.ptr(kPtrStage), base_byte, bytes), sum_is_new ? kPastEnd : off);
        any_new = __builtin_amdgcn_ballot_w64(sum_is_new) != 0; // one in N wavefronts, and those at a window's seam
#pragma unroll
        for (int r = 0; r < NP; ++r) p[r] = u32x4{0, 0, 0, 0};
    }
    if (any_new) {
        const uint32_t from = OWNED && !sum_is_new ? kPastEnd : off;
#pragma unroll
        for (int r = 0; r < NP; ++r) p[r] = rsrc_load16(row_rsrc(part[r], base_byte, bytes), from);
    }
    const u32x4 residual = rsrc_load16(row_rsrc(a.ptr(kPtrResidualIn), base_byte, bytes), off);
    const u32x4 gamma_raw = __builtin_amdgcn_raw_buffer_load_b128(row_rsrc(a.ptr(kPtrGamma), 0, row_bytes), in_slot * 16, 0, kAuxDefault);
    const RowLength<> length(hidden);

    // ---- reduce, residual add, sum of squares --------------------------------------------------------
    u32x4 sraw;
    if constexpr (N == 0) {
        sraw = p[0];
    } else {
        float acc[VEC];
#pragma unroll
        for (int r = 0; r < NP; ++r) accumulate<E>(p[r], acc, r == 0);
        sraw = E::pack(acc);
        if constexpr (OWNED) {
#pragma unroll
            for (int i = 0; i < 4; ++i) sraw[i] = sum_is_new ? sraw[i] : staged[i];
        }
    }
    const u32x4 xraw = added<E>(sraw, residual);
    float *const img = lds_dyn + wave * (kWave * VEC);
    float *const left = lds_dyn + (uint32_t)slot * a.rows_per_block * VEC + (wave * rows + nth) * 32;
    float sq[VEC];
    squares_of<E>(xraw, sq);
    put_squares(img + lane * VEC, sq);
    const int chained = hidden & ~31;
    if (hidden != chained) {
        const uint32_t behind = (uint32_t)(in_slot * VEC - chained);
        if (behind < (uint32_t)(hidden - chained)) {
            const float zeros[VEC] = {};
            put_squares(img + lane * VEC, zeros);
            put_squares(left + behind, sq);
        }
    }
    wave_lds_fence();
    const float rs = reciprocal_rms(slot_sum<VEC>(img + nth * slot * VEC, left, hidden, chained, slot, lane), length, a.eps);

    // ---- normalize, outputs --------------------------------------------------------------------------
    const u32x4 nraw = normed<E>(xraw, gamma_raw, rs);
    if (FORM == kFormStaged || (OWNED && any_new))
        rsrc_store16(row_rsrc(a.ptr(kPtrStage), base_byte, bytes), sum_is_new ? off : kPastEnd, sraw);
    if (Q == TDE_QUANT_NONE || a.address(kPtrNorm) != 0) rsrc_store16(row_rsrc(a.ptr(kPtrNorm), base_byte, bytes), off, nraw);
    rsrc_store16(row_rsrc(a.ptr(kPtrResidualOut), base_byte, bytes), off, xraw);

    if constexpr (Q != TDE_QUANT_NONE) {
        constexpr bool DYNAMIC = Q != TDE_QUANT_FP8_STATIC;
        const Normed<E> y(nraw);
        float scale[1];
        bool fast;
        if constexpr (DYNAMIC) {
            constexpr bool GROUP = Q == TDE_QUANT_FP8_GROUP;
            constexpr int LANES_PER_GROUP = TDE_QUANT_GROUP / VEC; // 16 (2-byte types) or 32 (fp32: whole rows)
            const float amax = y.largest();
            uint32_t m[1] = {lanes_max(__builtin_bit_cast(uint32_t, amax) & 0x7fffffffu, GROUP ? LANES_PER_GROUP : slot)};
            fast = scales_of_largest<Q>(m, scale);
            const uint32_t scales = GROUP ? (uint32_t)hidden / TDE_QUANT_GROUP : 1u; // of a row
            const bool writes = here && (GROUP ? (in_slot & (LANES_PER_GROUP - 1)) == 0 : in_slot == 0);
            const uint32_t at = place * scales + (GROUP ? (uint32_t)in_slot / LANES_PER_GROUP : 0u);
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, scale[0]), row_rsrc(a.ptr(kPtrScale), base * scales * 4, held * scales * 4u),
                                                  (int)(writes ? at * 4u : kPastEnd), 0, kAuxDefault);
        } else {
            scale[0] = a.static_scale;
            fast = static_scale_is_fast(a.static_scale);
        }
        const rsrc_t q_out = row_rsrc(a.ptr(kPtrCodes), base * (int64_t)hidden, held * (uint32_t)hidden);
        const uint32_t code_off = here ? place * (uint32_t)hidden + (uint32_t)in_slot * VEC : kPastEnd;
        auto quantize = [&](auto use_fast) {
            constexpr bool FAST = decltype(use_fast)::value;
            const float div = (Q == TDE_QUANT_FP8_STATIC || scale[0] > 0.0f) ? scale[0] : 1.0f;
            Divisor<E> divisor;
            if (FAST) divisor = Divisor<E>(div);
            uint32_t codes[VEC / 4];
            codes_of<E, Q, FAST>(y, divisor, div, codes);
            if constexpr (VEC == 8) {
                const u32x2 w = {codes[0], codes[1]};
                __builtin_amdgcn_raw_buffer_store_b64(w, q_out, (int)code_off, 0, kAuxStore);
            } else {
                __builtin_amdgcn_raw_buffer_store_b32(codes[0], q_out, (int)code_off, 0, kAuxStore);
            }
        };
        if (__builtin_expect(fast, 1)) quantize(std::true_type{});
        else quantize(std::false_type{});
    }
}

template <class E, int N, int Q>
hipError_t launch_form(const RowArgs &a, const Geometry &g, hipStream_t s) {
    const dim3 grid((unsigned)g.grid), block((unsigned)g.block_threads);
    const auto launch = [&](auto form) -> hipError_t {
        constexpr auto kernel = short_row_kernel<E, N, Q, decltype(form)::value>;
        if ((size_t)g.lds_bytes > kDefaultMaxDynamicLds) {
            const hipError_t e = allow_large_lds<kernel>();
            if (e != hipSuccess) return e;
        }
        return launch_kernel<kernel>(grid, block, (size_t)g.lds_bytes, s, a);
    };
    if constexpr (N != 0) {
        if (g.form == kFormStaged) return launch(std::integral_constant<int, kFormStaged>{});
        if (g.form == kFormOwned) return launch(std::integral_constant<int, kFormOwned>{});
    }
    return launch(std::integral_constant<int, kFormPlain>{});
}

template <class E, int N>
hipError_t launch_quant(int q, const RowArgs &a, const Geometry &g, hipStream_t s) {
    switch (q) {
    case TDE_QUANT_NONE: return launch_form<E, N, TDE_QUANT_NONE>(a, g, s);
    case TDE_QUANT_FP8_TOKEN: return launch_form<E, N, TDE_QUANT_FP8_TOKEN>(a, g, s);
    case TDE_QUANT_FP8_GROUP: return launch_form<E, N, TDE_QUANT_FP8_GROUP>(a, g, s);
    case TDE_QUANT_INT8_TOKEN: return launch_form<E, N, TDE_QUANT_INT8_TOKEN>(a, g, s);
    case TDE_QUANT_FP8_STATIC: return launch_form<E, N, TDE_QUANT_FP8_STATIC>(a, g, s);
    }
    return hipErrorInvalidValue;
}

template <class E>
hipError_t launch_ranks(int n, int q, const RowArgs &a, const Geometry &g, hipStream_t s) {
    switch (n) {
    case 0: return launch_quant<E, 0>(q, a, g, s);
    case 2: return launch_quant<E, 2>(q, a, g, s);
    case 4: return launch_quant<E, 4>(q, a, g, s);
    case 8: return launch_quant<E, 8>(q, a, g, s);
    }
    return hipErrorInvalidValue;
}

} // namespace

hipError_t launch_short_rows(int dtype, int n, int q, const RowArgs &a, const Geometry &g, hipStream_t s) {
    switch (dtype) {
    case TDE_BF16: return launch_ranks<ElemBF16>(n, q, a, g, s);
    case TDE_F16: return launch_ranks<ElemF16>(n, q, a, g, s);
    case TDE_F32: return launch_ranks<ElemF32>(n, q, a, g, s);
    }
    return hipErrorInvalidValue;
}

} // namespace tde
