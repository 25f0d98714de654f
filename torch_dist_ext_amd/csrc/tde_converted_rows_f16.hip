// fp16 row kernels that convert to fp32 and back in instructions of their own, four partials and four vectors per thread.
//
// What bounds a long launch is memory, and how well memory serves it depends on when the stores of one row meet the loads of the
// next.  With the mixed-precision arithmetic of the other kernels (tde_rows.h: fma_mix) they meet sooner, and rows of four vectors per
// thread, whole lines, lost 0.5 to 2.5 % by it.  us, mixed -> converted: 4 x [13542, 7168] -> static fp8 197.3 -> 193.3, [12184, 7552] 202.2 -> 198.2,
// [20000, 7168] beside a stage 373.5 -> 369.1, [17047, 7272] -> static fp8 255.3 -> 248.7, [22526, 7296] -> fp8 325.7 -> 322.9.
//
// This file is compiled without v_fma_mix* (_build.py): they would round x * rs, multiplied in fp32 and converted, once instead of twice.
#include "tde_rows.h"

namespace tde {

namespace {

struct ElemF16Converted : ElemF16 {
    static constexpr bool MIXED = false;
    static __device__ __forceinline__ u32x4 pack(const float (&f)[VEC]) {
        u32x4 raw;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f16x2 h = {(_Float16)f[2 * i], (_Float16)f[2 * i + 1]};
            raw[i] = __builtin_bit_cast(uint32_t, h);
        }
        return raw;
    }
};

template <int Q, bool WN, int FORM, bool SHIFTED>
hipError_t launch(const RowArgs &a, const Geometry &g, hipStream_t s) {
    constexpr auto kernel = row_kernel<ElemF16Converted, 4, 4, Q, WN, FORM, SHIFTED>;
    if ((size_t)g.lds_bytes > kDefaultMaxDynamicLds) {
        const hipError_t e = allow_large_lds<kernel>();
        if (e != hipSuccess) return e;
    }
    return launch_kernel<kernel>(dim3((unsigned)g.grid), dim3((unsigned)g.block_threads), (size_t)g.lds_bytes, s, a);
}

template <bool SHIFTED>
hipError_t launch_quant(int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s) {
    switch (q) {
    case TDE_QUANT_NONE:
        return g.form == kFormStaged ? launch<TDE_QUANT_NONE, true, kFormStaged, SHIFTED>(a, g, s) : launch<TDE_QUANT_NONE, true, kFormPlain, SHIFTED>(a, g, s);
    case TDE_QUANT_FP8_TOKEN:
        return wn ? launch<TDE_QUANT_FP8_TOKEN, true, kFormPlain, SHIFTED>(a, g, s) : launch<TDE_QUANT_FP8_TOKEN, false, kFormPlain, SHIFTED>(a, g, s);
    case TDE_QUANT_FP8_GROUP:
        if constexpr (!SHIFTED) // rows of whole groups are whole lines
            return wn ? launch<TDE_QUANT_FP8_GROUP, true, kFormPlain, false>(a, g, s) : launch<TDE_QUANT_FP8_GROUP, false, kFormPlain, false>(a, g, s);
        break;
    case TDE_QUANT_INT8_TOKEN:
        return wn ? launch<TDE_QUANT_INT8_TOKEN, true, kFormPlain, SHIFTED>(a, g, s) : launch<TDE_QUANT_INT8_TOKEN, false, kFormPlain, SHIFTED>(a, g, s);
    case TDE_QUANT_FP8_STATIC:
        return wn ? launch<TDE_QUANT_FP8_STATIC, true, kFormPlain, SHIFTED>(a, g, s) : launch<TDE_QUANT_FP8_STATIC, false, kFormPlain, SHIFTED>(a, g, s);
    }
    return hipErrorInvalidValue;
}

} // namespace

hipError_t launch_converted_rows_f16(int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s) {
    return a.line_mask != 0 ? launch_quant<true>(q, wn, a, g, s) : launch_quant<false>(q, wn, a, g, s);
}

} // namespace tde
