// Row kernels for gfx950 (MI355X): N-way partial reduce + residual add + RMSNorm + dynamic quant,
// one pass per row with the row held in registers.
//
// Arithmetic contract (what the reference's torch-eager composition computes,
// test/test_all_reduce_fusion.py:23-28,75-76, with the reduce order of
// src/common/all_reduce_fusion_impl.h:280-298):
//   s   = T( ((0 + p_0) + p_1) + ... + p_{N-1} )      fp32 accumulate in rank order, one rounding to T
//   x   = T( float(s) + float(residual_in) )           -> residual_out            (impl.h:271-278)
//   rs  = 1 / sqrt( sum(float(x)^2) / H + eps )        fp32, IEEE divide and sqrt; the sum in the order of
//                                                      torch's CPU reduction (sumsq_torch_order below)
//   y1  = T( float(x) * rs )
//   y   = T( float(gamma) * float(y1) )                -> norm_out
//   per-token fp8 : scale = amax|y| / 448, code = e4m3( clamp(float(y)/scale, +-448) )
//   per-group fp8 : the same over each 128-column group
//   per-token int8: scale = amax|y| / 127, code = clamp(rne(float(y)/scale), +-127)
//   static fp8    : code = e4m3( clamp(float(y)/static_scale, +-448) ), no scale written
//
// Included by one translation unit per element type; nothing here is exported.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "tde_abi.h"

namespace tde {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;
constexpr int kMaxWavesPerBlock = 16;
constexpr int kMaxKernelRanks = 8;

// Kernel argument block, passed by value.  A launch with 128 bytes of arguments or more costs the host 0.6-0.7 us more
// than one with less on some machines (3.6 us against 2.9; on others 2.5 either way), a tenth of a decode-size call: so
// the device addresses are packed to the 48 bits they have -- as a buffer resource takes them, 32 low bits and 16 high --
// and the kernels read neither the grid's nor the workgroup's size, which would come in 256 bytes of hidden arguments.
// Unpacking is one scalar instruction per address.
enum : int { kPtrPart = 0, kPtrResidualIn = kMaxKernelRanks, kPtrResidualOut, kPtrNorm, kPtrGamma, kPtrCodes, kPtrScale, kPtrStage, kPtrs };

struct RowArgs {
    uint32_t lo[kPtrs];
    uint32_t hi[(kPtrs + 1) / 2]; // two per word; the last half word is `hidden`
    uint16_t threads_per_row;     // multiple of 64; short rows (tde_short_rows.hip): 16 or 32 lanes of a wavefront
    uint8_t rows_per_block;       // at most 16
    uint8_t xcd_chunk;            // workgroups per XCD chunk of the row mapping (power of two; 0 or 1 = rows in launch order)
    int64_t tokens;
    float eps;
    float static_scale;
    uint32_t chunked_blocks; // workgroups the XCD mapping permutes: the whole groups of 8 * xcd_chunk of the grid
    uint8_t owner : 3;       // OWNED row kernels: rows == owner (mod N) are summed here, the others are read from the stage
    uint8_t line_mask : 5;   // row_shift()
    uint8_t table_mask;      // bit r: partial r's address is entry r of a device pointer table.  The table's own address
                             // stands in the stage's place: a launch has one or the other
    uint16_t wave_step; // 32768 / wavefronts per row + 1: row_group()

    __host__ __device__ uint64_t address(int i) const {
        return ((uint64_t)((i & 1) ? hi[i >> 1] >> 16 : hi[i >> 1] & 0xffffu) << 32) | lo[i];
    }
    __host__ __device__ void *ptr(int i) const { return reinterpret_cast<void *>(address(i)); }
    // wave / wavefronts per row, for the at most 16 wavefronts of a workgroup (a division takes 25 instructions ahead of the
    // first load)
    __host__ __device__ int row_group(int wave) const { return wave * wave_step >> 15; }
    __host__ __device__ int hidden() const { return (int)(hi[kPtrs >> 1] >> 16); }
    // By how many vectors the row that starts at byte `row_byte` is moved along its threads (SHIFTED row kernels): thread t of the
    // row group takes vectors (t - shift) mod threads_per_row first.  line_mask: how many vectors a 128-byte line of the
    // narrowest buffer holds, less one (7 of T-typed rows, 15 or 31 of codes); 0: rows stay in place.
    __host__ __device__ int row_shift(int64_t row_byte) const { return (int)((uint32_t)row_byte >> 4 & line_mask); }
    void set(int i, const void *p) {
        const uint64_t v = reinterpret_cast<uint64_t>(p);
        lo[i] = (uint32_t)v;
        set_half(i, (uint32_t)(v >> 32));
    }
    void set_hidden(int64_t h) { set_half(kPtrs, (uint32_t)h); }

private:
    void set_half(int i, uint32_t v) {
        const int shift = (i & 1) * 16;
        hi[i >> 1] = (hi[i >> 1] & ~(0xffffu << shift)) | ((v & 0xffffu) << shift);
    }
};
static_assert(sizeof(RowArgs) == 120 && (kPtrs & 1) == 1, "below 128 bytes, and a half word left for `hidden`");

// The partials' addresses: from the argument block, or (one uniform branch, batched scalar loads) from the device pointer
// table for the entries the host does not know.
// Ahead of it the fields that are needed a little later, or the compiler would fetch each where it is used and wait three times
// for the scalar cache before the first load.  8 x [1, 4096] bf16, from a wavefront's start to its last request: 1132 cycles, with
// this and the row group without a division 1020 (8 x [128, 4096] 4.52 -> 4.47 us, 2 x [700, 4096] fp16 6.28 -> 6.18).
typedef const __attribute__((address_space(4))) uint64_t *table_t;
template <int NP>
__device__ __forceinline__ void partial_addresses(const RowArgs &a, uint64_t table, const void *(&part)[NP]) {
    asm volatile("; all arguments at once" ::"s"(a.tokens), "s"(a.eps), "s"(a.static_scale), "s"(a.chunked_blocks),
                 "s"((uint32_t)a.table_mask));
#pragma unroll
    for (int r = 0; r < NP; ++r) part[r] = a.ptr(kPtrPart + r);
    if (a.table_mask != 0) {
#pragma unroll
        for (int r = 0; r < NP; ++r) {
            const void *from_table = reinterpret_cast<const void *>(((table_t)table)[r]);
            part[r] = (a.table_mask >> r & 1) ? from_table : part[r];
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Element traits: a 16-byte vector <-> VEC floats.  pack() rounds to nearest even.
// ---------------------------------------------------------------------------------------------
struct ElemBF16 {
    static constexpr int VEC = 8;
    static constexpr int BYTES = 2;
    static constexpr bool MIXED = false;
    static __device__ __forceinline__ void unpack(u32x4 raw, float (&f)[VEC]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[2 * i] = __builtin_bit_cast(float, raw[i] << 16);
            f[2 * i + 1] = __builtin_bit_cast(float, raw[i] & 0xffff0000u);
        }
    }
    static __device__ __forceinline__ u32x4 pack(const float (&f)[VEC]) {
        u32x4 raw;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f32x2 v = {f[2 * i], f[2 * i + 1]};
            raw[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
        }
        return raw;
    }
};

struct ElemF16 {
    static constexpr int VEC = 8;
    static constexpr int BYTES = 2;
    static constexpr bool MIXED = true; // see fma_mix
    static __device__ __forceinline__ void unpack(u32x4 raw, float (&f)[VEC]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t w = raw[i]; // copy first: bit_cast applied straight to a vector element reads lane 0
            const f16x2 h = __builtin_bit_cast(f16x2, w);
            f[2 * i] = (float)h[0];
            f[2 * i + 1] = (float)h[1];
        }
    }
    static __device__ __forceinline__ u32x4 pack(const float (&f)[VEC]) {
        u32x4 raw;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float lo = f[2 * i], hi = f[2 * i + 1];
            // one rounding here and one in the operation before it: never one instruction that rounds its exact result once
            asm("" : "+v"(lo), "+v"(hi));
            f32x2 v = {lo, hi};
            raw[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
        }
        return raw;
    }
};

// The same rows with conversions in place of the mixed instructions: longer arithmetic (kFormLong).
struct ElemF16Unmixed : ElemF16 {
    static constexpr bool MIXED = false;
};

struct ElemF32 {
    static constexpr int VEC = 4;
    static constexpr int BYTES = 4;
    static constexpr bool MIXED = false;
    static __device__ __forceinline__ void unpack(u32x4 raw, float (&f)[VEC]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t w = raw[i]; // copy first: bit_cast applied straight to a vector element reads lane 0
            f[i] = __builtin_bit_cast(float, w);
        }
    }
    static __device__ __forceinline__ u32x4 pack(const float (&f)[VEC]) {
        u32x4 raw;
#pragma unroll
        for (int i = 0; i < 4; ++i) raw[i] = __builtin_bit_cast(uint32_t, f[i]);
        return raw;
    }
};

// fp16 rows (E::MIXED) never unpack.  v_fma_mix_f32 takes a half of a packed pair as an fp32 operand, so that a conversion costs
// nothing beside the operation it is for; and where two fp16 numbers are added or multiplied and the result is rounded to fp16,
// the packed instructions, which round once, give the bits of the two roundings of the fp32 operation: a product of two
// has 22 bits and is exact in fp32, and a sum rounded to 24 bits, no fewer than 2 * 11 + 1, never lands on a different side of a
// boundary between two fp16 numbers (Figueroa, "When is double rounding innocuous?", 1995).
// The mixed forms issue at half the rate, so a launch that is bound by instructions of many wavefronts gains from the packed ones
// only; one that waits for a row's chain gains from every instruction left out.  With conversions against this: 2 x [79, 8096] 4.28 -> 4.16 us,
// 4 x [89, 4256] 3.83 -> 3.70, 2 x [1162, 1152] -> int8 4.44 -> 4.33, 2 x [1651, 6328] -> int8 19.85 -> 18.5; 2-3 % up to 40 MB, 0.5 % and less from
// 200 MB on, where four vectors per thread lose up to 2.5 %: four partials convert there (tde_converted_rows_f16.hip), two have a
// limit on workgroups beside a stage (tde_abi.hip).
// HALF: which one of `pair`, 0 or 1.  fma(pair, b, c).
template <int HALF>
__device__ __forceinline__ float fma_mix(uint32_t pair, float b, float c) {
    float r;
    if constexpr (HALF == 0) asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair), "v"(b), "v"(c));
    else asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair), "v"(b), "v"(c));
    return r;
}
// pair + 0, which turns -0 into +0 as the sums that start from 0 do
template <int HALF>
__device__ __forceinline__ float widen_mix(uint32_t pair) {
    float r;
    if constexpr (HALF == 0) asm("v_fma_mix_f32 %0, %1, 1.0, 0 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair));
    else asm("v_fma_mix_f32 %0, %1, 1.0, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair));
    return r;
}
// c + pair, in c's register
template <int HALF>
__device__ __forceinline__ float add_mix(uint32_t pair, float c) {
    if constexpr (HALF == 0) asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel_hi:[1,0,0]" : "+v"(c) : "v"(pair));
    else asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(c) : "v"(pair));
    return c;
}
// pair * b, -0 kept
template <int HALF>
__device__ __forceinline__ float mul_mix(uint32_t pair, float b) {
    float r;
    if constexpr (HALF == 0) asm("v_fma_mix_f32 %0, %1, %2, neg(0) op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair), "v"(b));
    else asm("v_fma_mix_f32 %0, %1, %2, neg(0) op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair), "v"(b));
    return r;
}
template <int HALF>
__device__ __forceinline__ float square_mix(uint32_t pair) {
    float r;
    if constexpr (HALF == 0) asm("v_fma_mix_f32 %0, %1, %1, 0 op_sel_hi:[1,1,0]" : "=v"(r) : "v"(pair));
    else asm("v_fma_mix_f32 %0, %1, %1, 0 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "=v"(r) : "v"(pair));
    return r;
}

// acc = (first ? 0 : acc) + one vector of a partial
template <class E>
__device__ __forceinline__ void accumulate(u32x4 raw, float (&acc)[E::VEC], bool first) {
    if constexpr (E::MIXED) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            acc[2 * i] = first ? widen_mix<0>(raw[i]) : add_mix<0>(raw[i], acc[2 * i]);
            acc[2 * i + 1] = first ? widen_mix<1>(raw[i]) : add_mix<1>(raw[i], acc[2 * i + 1]);
        }
    } else {
        float p[E::VEC];
        E::unpack(raw, p);
#pragma unroll
        for (int i = 0; i < E::VEC; ++i) acc[i] = first ? 0.0f + p[i] : acc[i] + p[i];
    }
}

// T(a + b)
template <class E>
__device__ __forceinline__ u32x4 added(u32x4 a, u32x4 b) {
    if constexpr (E::MIXED) {
        u32x4 sum;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t u = a[i], v = b[i];
            sum[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, u) + __builtin_bit_cast(f16x2, v));
        }
        return sum;
    } else {
        float x[E::VEC], y[E::VEC];
        E::unpack(a, x);
        E::unpack(b, y);
#pragma unroll
        for (int i = 0; i < E::VEC; ++i) x[i] = x[i] + y[i];
        return E::pack(x);
    }
}

template <class E>
__device__ __forceinline__ void squares_of(u32x4 raw, float (&sq)[E::VEC]) {
    if constexpr (E::MIXED) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            sq[2 * i] = square_mix<0>(raw[i]);
            sq[2 * i + 1] = square_mix<1>(raw[i]);
        }
    } else {
        float x[E::VEC];
        E::unpack(raw, x);
#pragma unroll
        for (int i = 0; i < E::VEC; ++i) sq[i] = x[i] * x[i];
    }
}

// T(gamma * T(x * rs)) of one vector.
template <class E>
__device__ __forceinline__ u32x4 normed(u32x4 xraw, u32x4 gamma_raw, float rs) {
    constexpr int VEC = E::VEC;
    float n[VEC];
    if constexpr (E::MIXED) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            n[2 * i] = mul_mix<0>(xraw[i], rs);
            n[2 * i + 1] = mul_mix<1>(xraw[i], rs);
        }
        const u32x4 first = E::pack(n);
        u32x4 y;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t u = first[i], v = gamma_raw[i];
            y[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, v) * __builtin_bit_cast(f16x2, u));
        }
        return y;
    } else {
        float x[VEC], g[VEC];
        E::unpack(xraw, x);
        E::unpack(gamma_raw, g);
#pragma unroll
        for (int i = 0; i < VEC; ++i) n[i] = x[i] * rs;
        E::unpack(E::pack(n), n);
#pragma unroll
        for (int i = 0; i < VEC; ++i) n[i] = g[i] * n[i];
        return E::pack(n);
    }
}

// The largest magnitude of a row's elements: NaN if any of them is, as torch's amax has it (v_max_f32 would drop it).  Two
// elements an instruction, on the values that the quotients need anyway.
__device__ __forceinline__ float max_abs(float acc, float a, float b) {
    float r;
    asm("v_maximum3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(acc), "v"(a), "v"(b));
    return r;
}

// A vector of normed elements on its way to codes: fp32, or as it is where E is MIXED.
template <class E, bool MIXED = E::MIXED>
struct Normed {
    float y[E::VEC];
    Normed() = default;
    __device__ __forceinline__ explicit Normed(u32x4 raw) { E::unpack(raw, y); }
    __device__ __forceinline__ void values(float (&v)[E::VEC]) const {
#pragma unroll
        for (int i = 0; i < E::VEC; ++i) v[i] = y[i];
    }
    __device__ __forceinline__ float largest() const {
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < E::VEC; i += 2) m = max_abs(m, y[i], y[i + 1]);
        return m;
    }
};
template <class E>
struct Normed<E, true> {
    u32x4 raw;
    Normed() = default;
    __device__ __forceinline__ explicit Normed(u32x4 raw_) : raw(raw_) {}
    __device__ __forceinline__ void values(float (&v)[E::VEC]) const { E::unpack(raw, v); }
    __device__ __forceinline__ float largest() const { // of even and odd elements side by side, then of the two
        uint32_t m;
        asm("v_pk_maximum3_f16 %0, %1, %1, %1 neg_lo:[0,0,1] neg_hi:[0,0,1]" : "=v"(m) : "v"(raw[0]));
#pragma unroll
        for (int i = 1; i < 4; ++i) asm("v_pk_maximum3_f16 %0, %0, %1, %1 neg_lo:[0,0,1] neg_hi:[0,0,1]" : "+v"(m) : "v"(raw[i]));
        const f16x2 h = __builtin_bit_cast(f16x2, m);
        const float lo = (float)h[0], hi = (float)h[1];
        return max_abs(lo, hi, hi);
    }
};

// min(max(q, -limit), limit) that keeps NaN, as torch.clamp does.
__device__ __forceinline__ float clamp_keep_nan(float q, float limit) {
    float r;
    asm("v_maximum3_f32 %0, %1, -%2, -%2" : "=v"(r) : "v"(q), "v"(limit));
    asm("v_minimum3_f32 %0, %1, %2, %2" : "=v"(r) : "v"(r), "v"(limit));
    return r;
}

__device__ __forceinline__ uint32_t max_u32(uint32_t a, uint32_t b) { return a > b ? a : b; }

// ---------------------------------------------------------------------------------------------
// 64-lane wavefront reductions: four DPP steps inside each 16-lane row, then the four row
// results are combined through v_readlane.  Every lane ends with the same value.
// ---------------------------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_move_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __builtin_bit_cast(float, dpp_move_u32<CTRL>(__builtin_bit_cast(uint32_t, v)));
}

// Unsigned maximum over each 16-lane row.  The maxima across lanes are taken on the bit patterns of magnitudes: for
// non-negative floats the order of the bits is the order of the values, with every NaN above infinity.
__device__ __forceinline__ uint32_t row16_max(uint32_t v) {
    v = max_u32(v, dpp_move_u32<0xB1>(v));  // quad_perm [1,0,3,2]
    v = max_u32(v, dpp_move_u32<0x4E>(v));  // quad_perm [2,3,0,1]
    v = max_u32(v, dpp_move_u32<0x141>(v)); // row_half_mirror
    v = max_u32(v, dpp_move_u32<0x140>(v)); // row_mirror
    return v;
}

__device__ __forceinline__ float read_lane(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// A value that is the same in every lane.  SCALAR: in a scalar register (the compiler drops __builtin_amdgcn_readfirstlane of what it
// knows to be uniform, and leaves that in a vector register).
template <bool SCALAR>
__device__ __forceinline__ float uniform_value(float v) {
    if constexpr (SCALAR) asm("" : "+v"(v));
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
    v = row16_max(v);
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0), b = (uint32_t)__builtin_amdgcn_readlane((int)v, 16),
                   c = (uint32_t)__builtin_amdgcn_readlane((int)v, 32), d = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
    return max_u32(max_u32(a, b), max_u32(c, d));
}

// Maximum over the wavefronts that share a row.  `slot`: the row's word of LDS, zero before a barrier that every thread has
// passed (0 is the identity: bit patterns of magnitudes).  One barrier.  The four 16-lane rows of a wavefront meet in LDS
// instead of through v_readlane, the wavefronts there instead of in every wavefront once more.
__device__ __forceinline__ uint32_t row_max(uint32_t v, uint32_t *slot, int lane, int waves_per_row) {
    if (waves_per_row == 1) return wave_max(v);
    v = row16_max(v);
    // in assembly, or the compiler would put a reduction over the wavefront in front of it
    if ((lane & 15) == 0)
        asm volatile("ds_max_u32 %0, %1\n\ts_waitcnt lgkmcnt(0)" ::"v"((uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t *)slot), "v"(v) : "memory");
    __syncthreads();
    return *slot;
}

// ---------------------------------------------------------------------------------------------
// Sum of a row's squares in the order of torch's CPU reduction.
//
// The eager composition computes x.float().pow(2).mean(-1) (test/test_all_reduce_fusion.py:25).  On x86 hosts
// torch reduces a contiguous row of n floats with 8-lane vectors and four interleaved vector accumulators
// (its cascade sum): with V = n / 8 vectors, I = V / 4,
//   chain (m, k), m = 0..7, k = 0..3, takes the elements 8 * (4 * i + k) + m, i = 0..I-1;
//   every 16 consecutive i form a block that is summed left to right from zero; the block sums of a chain are
//   summed left to right (a last block shorter than 16 included);
//   p[m] = chain(m,0) + the V % 4 vectors left over + chain(m,1) + chain(m,2) + chain(m,3), left to right;
//   sum  = the n % 8 scalars left over, then p[0] .. p[7], left to right from zero.
// (Rows shorter than 8 floats use four interleaved scalars instead; rows beyond 8192 floats would add a cascade
// level and do not occur: a row has at most 1024 16-byte vectors.)  Following that order makes the reciprocal RMS,
// and with it every normed element, scale and code, bit-identical to the eager composition's.
//
// The row's squares are laid out in LDS in element order (`img`); one thread sums one block of one chain
// (16 reads 32 floats apart), the block sums go through LDS (`bs`), and lanes 4m+k of every wavefront finish chain
// (m, k).  With 8 floats per 16-byte vector (2-byte element types) a block of 64 vectors is exactly what one
// wavefront loaded with one load instruction, so the first step needs no workgroup barrier (WAVE_BLOCKS).
//
// This stands between a row's last load and its first store, where a wavefront pays at least four cycles for every
// instruction of any kind, so nothing in it is guarded element by element: what the chains do not take (V % 4 vectors and n % 8
// scalars) goes to a place of its own (`left`) with zeros in the image, lanes past the row's end hold zeros, and a row's block sums
// are filled up with zeros to a number that has straight-line code (sum_slots).  Adding +0 to a sum of squares changes
// nothing, and neither does leaving out the +0 a sum starts from: a square is never -0.  8 x [1, 4096] bf16: from a
// wavefront's last partial to the reciprocal RMS 2416 -> 1992 cycles with guarded and with straight code, the wait for the
// slowest wavefront in both; launches 2 x [16, 1024] 2.35 -> 2.13 us, 8 x [128, 4096] 4.79 -> 4.53, 4 x [512, 5120] fp16 -> int8
// 8.72 -> 8.27, 2 x [20000, 200] bf16 -> fp8 13.6 -> 11.8.
// ---------------------------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ float quad_bcast(float v) {
    return dpp_move<CTRL>(v);
}

// Dynamic LDS a kernel that calls sumsq_torch_order needs.
inline size_t sumsq_lds_bytes(int block_threads, int vpt, int vec_floats) {
    return ((size_t)block_threads * vpt * vec_floats + 1024) * sizeof(float);
}

// A compute unit of gfx950 has 160 KiB of LDS; a workgroup that asks for this much dynamic LDS (the kernels' 64
// static bytes and the allocation granule fit in the slack) shares its CU with at most `wgs` - 1 others.
constexpr size_t kLdsPerCu = 160 * 1024;
constexpr size_t kDefaultMaxDynamicLds = 64 * 1024; // what a kernel may ask for without raising its attribute
inline size_t lds_bytes_for_workgroups_per_cu(int wgs) { return (kLdsPerCu / (size_t)wgs - 1024) & ~(size_t)255; }

// Raises KERNEL's dynamic-LDS ceiling to (nearly) the whole CU, once per device (a launch asking for more than 64 KiB
// fails otherwise).  Not a stream operation; the first launch of a kernel on a device that needs it pays for it.
template <auto KERNEL>
hipError_t allow_large_lds() {
    static std::atomic<uint64_t> done{0}; // bit d: set on device d
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = (dev >= 0 && dev < 64) ? (uint64_t{1} << dev) : 0;
    if (bit != 0 && (done.load(std::memory_order_acquire) & bit)) return hipSuccess;
    // the most a launch here asks for; the kernel's static LDS must still fit beside it
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(KERNEL), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds_bytes_for_workgroups_per_cu(1));
    if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
    else (void)hipGetLastError(); // reported through the return value, not left behind for the next call
    return e;
}

// One launch.  hipLaunchKernel itself: the <<<>>> form goes through a pushed and popped call configuration and leaves its
// status to hipGetLastError, 0.15 us of host time a launch (2.42 against 2.27 us for an empty kernel).
template <auto KERNEL, class... Args>
hipError_t launch_kernel(dim3 grid, dim3 block, size_t lds, hipStream_t s, const Args &...args) {
    void *ptrs[] = {const_cast<void *>(static_cast<const void *>(&args))...};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void *>(KERNEL), grid, block, ptrs, lds, s);
    if (e != hipSuccess) (void)hipGetLastError(); // reported through the return value, not left behind for the next call
    return e;
}

// Returns `v`, but only once `after` exists: index arithmetic built on the result cannot be hoisted above the
// row loads, whose registers leave no room for it.
__device__ __forceinline__ int not_before(int v, uint32_t after) {
    asm volatile("; index math stays behind the row loads" : "+v"(v) : "v"(after));
    return v;
}

__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Block sums per row as the last step reads them: the number rounded up to one that has straight-line code.  A workgroup's
// slots and its rows' `left` floats (32 each) fit the 1024 floats behind the image: it holds at most 16 blocks in all, so at
// most 16 rows of one slot, 8 of two, 5 of four, 3 of eight or one of more.
__device__ __forceinline__ int sum_slots(int blocks) {
    return blocks <= 1 ? 1 : (blocks <= 2 ? 2 : (blocks <= 4 ? 4 : (blocks <= 8 ? 8 : (blocks <= 12 ? 12 : 16))));
}

// Where a row group's floats lie in LDS; wavefront-uniform, from the row's length and the launch geometry.
//   img  one float per element the group holds (threads * VPT * VECF)
//   bs   32 * slots block sums
//   left the floats from `chained` to n
template <int VPT, int VECF, bool WAVE_BLOCKS>
struct SumLayout {
    float *img, *bs, *left;
    int n, chained; // floats of the row, and how many of them the chains take
    int blocks;     // 512-float blocks that are summed: with WAVE_BLOCKS all that the group holds, else those of the chains
    int slots;

    __device__ __forceinline__ SumLayout(float *lds_img, float *lds_bs, int n_, int tpr, int rows_per_block, int group) {
        n = n_;
        chained = n & ~31;
        blocks = WAVE_BLOCKS ? (tpr >> 6) * VPT : (chained + 511) >> 9;
        slots = sum_slots(blocks);
        img = lds_img + group * (tpr * VPT * VECF);
        bs = lds_bs + group * (slots * 32);
        left = lds_bs + rows_per_block * (slots * 32) + group * 32;
    }
};

// Zeros for the block sums that the last step reads and no thread writes.  Anywhere before the squares are complete: under
// the row's loads.  At most three slots: fewer floats than the group has threads (one slot takes three blocks or none, more
// take five blocks, i.e. 192 threads).
template <int VPT, int VECF, bool WAVE_BLOCKS>
__device__ __forceinline__ void sumsq_clear(const SumLayout<VPT, VECF, WAVE_BLOCKS> &s, int t) {
    if (s.slots != s.blocks && t < (s.slots - s.blocks) * 32) s.bs[s.blocks * 32 + t] = 0.0f;
}

// The squares of one vector (number `vec` of the row) go to their place in the image ...
template <int VECF>
__device__ __forceinline__ void put_squares(float *dst, const float (&sq)[VECF]) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    if constexpr (VECF % 4 == 0) {
#pragma unroll
        for (int c = 0; c < VECF; c += 4) *reinterpret_cast<f32x4 *>(dst + c) = f32x4{sq[c], sq[c + 1], sq[c + 2], sq[c + 3]};
    } else {
#pragma unroll
        for (int c = 0; c < VECF; ++c) dst[c] = sq[c];
    }
}

// ... and from there to the floats that the chains do not take, zeros in their place.  A step of its own behind all of a
// thread's puts: a branch between them keeps the arithmetic of several vectors from overlapping (8 x [2048, 8192] +1.5 %).
template <int VPT, int VECF, bool WAVE_BLOCKS>
__device__ __forceinline__ void split_left(const SumLayout<VPT, VECF, WAVE_BLOCKS> &s, int vec, const float (&sq)[VECF]) {
    const uint32_t behind = (uint32_t)(vec * VECF - s.chained);
    if (behind < (uint32_t)(s.n - s.chained)) {
        const float zeros[VECF] = {};
        put_squares(s.img + vec * VECF, zeros);
        put_squares(s.left + behind, sq);
    }
}

// Sixteen elements of chain `cl` (= 4m + k) 32 floats apart, summed left to right.  GUARD: only the first `terms` (4, 8 or
// 12, or more than that: all) are inside the image.
template <bool GUARD>
__device__ __forceinline__ float chain_block_sum(const float *block, int cl, int terms) {
    const float *src = block + 8 * (cl & 3) + (cl >> 2);
    float v[16];
#pragma unroll
    for (int g = 0; g < 16; g += 4) {
        const bool inside = !GUARD || g == 0 || g < terms;
        const float *from = src + (inside ? 32 * g : 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[g + i] = from[32 * i];
        if (GUARD && g != 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[g + i] = inside ? v[g + i] : 0.0f;
        }
    }
    float acc = v[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) acc += v[i];
    return acc;
}

// A chain's block sums, left to right.  All that could be there are requested before the first is added; what lies in slots that
// are not used is the next row's or nobody's, and inside the 1024 floats for every row (the last of several rows starts at slot
// 16 at most).  Up to eight and up to sixteen have code of their own: always sixteen costs 8 x [1, 4096] 2 %, a switch over every
// number, which the compiler turns into a tree of branches and flags, 4 x [64, 5120] fp16 -> int8 3 % and 4 x [300, 2048] 2 %.
template <int MOST>
__device__ __forceinline__ float chain_sum_of(const float *bs, int cl, int slots) {
    float v[MOST];
#pragma unroll
    for (int b = 0; b < MOST; ++b) v[b] = bs[b * 32 + cl];
    float chain = v[0] + v[1];
    if (slots > 2) chain = (chain + v[2]) + v[3];
    if (slots > 4) {
#pragma unroll
        for (int b = 4; b < 8; ++b) chain += v[b];
    }
    if constexpr (MOST == 16) {
#pragma unroll
        for (int b = 8; b < 12; ++b) chain += v[b];
        if (slots > 12) {
#pragma unroll
            for (int b = 12; b < 16; ++b) chain += v[b];
        }
    }
    return chain;
}
__device__ __forceinline__ float chain_sum(const float *bs, int cl, int slots) {
    if (slots == 1) return bs[cl];
    return slots > 8 ? chain_sum_of<16>(bs, cl, slots) : chain_sum_of<8>(bs, cl, slots);
}

// Waits for the wavefronts that share a row; one wavefront alone only for its own LDS traffic.
__device__ __forceinline__ void row_barrier(int waves_per_row) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if (waves_per_row > 1) __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// After every thread of the row group has put its squares: the sum, the same value in every thread.
// Contains workgroup barriers when a row spans several wavefronts: all threads of the workgroup must call it together.
// wave: the wavefront's number in its row group.
// t, lane: the thread's place in its row group and wavefront.  SHIFTED: the row may be moved along its threads (RowArgs::row_shift).
template <bool SHIFTED, int VPT, int VECF, bool WAVE_BLOCKS>
__device__ __forceinline__ float sumsq_torch_order(const SumLayout<VPT, VECF, WAVE_BLOCKS> &s, int t, int tpr, int wave, int lane) {
    const int waves_per_row = tpr >> 6;
    const int cl = lane & 31;
    if constexpr (WAVE_BLOCKS) {
        static_assert(VECF == 8, "one wavefront load = one block of 64 eight-float vectors");
        // Block j * waves_per_row + wave is what this wavefront wrote for its vector j: no other wavefront is involved, unless
        // the row has been moved.
        if constexpr (SHIFTED) row_barrier(waves_per_row);
        else wave_lds_fence();
        if constexpr (VPT == 1) {
            // one block per wavefront: both of its halves sum it
            s.bs[wave * 32 + cl] = chain_block_sum<false>(s.img + 512 * wave, cl, 16);
        } else {
            // two blocks at a time, one per half of the wavefront; their reads and sums interleave
            float sum[VPT / 2];
            int b[VPT / 2];
#pragma unroll
            for (int k = 0; k < VPT / 2; ++k) {
                b[k] = ((lane >> 5) + 2 * k) * waves_per_row + wave;
                sum[k] = chain_block_sum<false>(s.img + 512 * b[k], cl, 16);
            }
#pragma unroll
            for (int k = 0; k < VPT / 2; ++k) s.bs[b[k] * 32 + cl] = sum[k];
        }
    } else {
        row_barrier(waves_per_row);
        // one thread per chain and block: the group has at least 32 threads per block of its chains
        if (t < 32 * s.blocks) {
            const int b = t >> 5;
            const int terms = (tpr * VPT * VECF - 512 * b) >> 5;
            float sum;
            if (((tpr * VPT * VECF) & 511) == 0) sum = chain_block_sum<false>(s.img + 512 * b, cl, 16);
            else sum = chain_block_sum<true>(s.img + 512 * b, cl, terms);
            s.bs[t] = sum;
        }
    }
    row_barrier(waves_per_row);

    // Lane 4m + k of every wavefront sums the blocks of chain (m, k); the quad then holds the four chains of m.
    const float chain = chain_sum(s.bs, cl, s.slots);
    float p = quad_bcast<0x00>(chain);
    float sum = 0.0f; // the scalars left over
    if (s.n != s.chained) {
        const int m = cl >> 2, L = (s.n >> 3) & 3;
        for (int l = 0; l < L; ++l) p += s.left[8 * l + m];
        if (s.n < 8) {
            // four interleaved scalars, the first of them also takes what is left over
            sum = s.left[0];
            if (s.n < 4) {
                for (int e = 1; e < s.n; ++e) sum += s.left[e];
            } else {
                for (int e = 4; e < s.n; ++e) sum += s.left[e];
                sum += s.left[1];
                sum += s.left[2];
                sum += s.left[3];
            }
        } else if constexpr (VECF != 8) {
            for (int e = s.n & ~7; e < s.n; ++e) sum += s.left[e - s.chained];
        }
    }
    p += quad_bcast<0x55>(chain);
    p += quad_bcast<0xAA>(chain);
    p += quad_bcast<0xFF>(chain);
    float q[8];
#pragma unroll
    for (int mm = 0; mm < 8; ++mm) q[mm] = read_lane(p, 4 * mm);
    __builtin_amdgcn_sched_barrier(0); // read one by one each would be waited for
    sum = VECF == 8 ? q[0] : sum + q[0]; // 2-byte types: whole vectors of eight floats, no scalars left over
#pragma unroll
    for (int mm = 1; mm < 8; ++mm) sum += q[mm];
    return sum;
}

// 1/d from an approximation within one unit in the last place: correctly rounded unless d is all ones and the approximation
// half a unit low (2^23 mantissas of d and both neighbours of 1/d, on the host: unit_test_rounding.cpp).
__host__ __device__ __forceinline__ float refined_reciprocal(float d, float approx) {
    return __builtin_fmaf(__builtin_fmaf(-d, approx, 1.0f), approx, approx);
}

// y / d, correctly rounded, for a divisor shared by many elements.  `rcp` must be the correctly
// rounded 1/d.  q0 = RN(y*rcp) is within one ulp of the quotient; the residual y - q0*d is exact
// in one fma; adding residual*rcp back in a second fma rounds to the correctly rounded quotient
// (Markstein's division theorem) as long as nothing underflows.  Callers take this path only when
// d is far from the subnormal and overflow ranges and use a plain division otherwise.
// The residual is taken as q0*d - y and subtracted, not as y - q0*d and added: the same value for every non-zero y,
// and for y = -0 the result is then -0 like the quotient's (the other form ends in (+0) + (-0) = +0).
__host__ __device__ __forceinline__ float div_shared(float y, float d, float rcp) {
    const float q0 = y * rcp;
    const float e = __builtin_fmaf(q0, d, -y);
    return __builtin_fmaf(-e, rcp, q0);
}

// A row's length and its reciprocal, correctly rounded (no row length is all ones in 24 bits), for reciprocal_rms.  They live
// through the load phase.  SCALAR: in scalar registers, where the vector registers are all taken there.
template <bool SCALAR = false>
struct RowLength {
    float h, rcp;
    __device__ __forceinline__ explicit RowLength(int hidden) {
        h = uniform_value<SCALAR>((float)hidden);
        rcp = uniform_value<SCALAR>(refined_reciprocal(h, __builtin_amdgcn_rcpf(h)));
    }
};

// 1 / sqrt(m) with the root and its reciprocal each rounded as the IEEE operation, from y, an approximation of 1 / sqrt(m).
// The root by Markstein's iteration on g ~ sqrt(m) and y ~ 1 / (2 sqrt(m)) ("Computation of elementary functions on the IBM
// RISC System/6000 processor", 1990), which leaves 1/sqrt(m) in 2y.  That is not yet 1/g, which g's own rounding has moved by
// up to half a unit: two steps of Newton's, or the reciprocal is a unit off for three of 2^24 mantissas.  They start a unit high:
// below 1/g the last step ends in a tie for g all ones and rounds it down.  Right for every mantissa and every y up to three
// units off (on the host, unit_test_rounding.cpp).
__host__ __device__ __forceinline__ float reciprocal_of_root(float m, float y) {
    float g = m * y;
    y *= 0.5f;
    const float e = __builtin_fmaf(-y, g, 0.5f);
    g = __builtin_fmaf(g, e, g);
    y = __builtin_fmaf(y, e, y);
    g = __builtin_fmaf(__builtin_fmaf(-g, g, m), y, g); // sqrt(m)
    return refined_reciprocal(g, refined_reciprocal(g, y * (2.0f + 0x1p-22f)));
}

// 1 / sqrt(sumsq / length + eps) with every step rounded as the IEEE operation: 17 instructions where two divisions and a square
// root are 45.  Outside [2^-60, 2^100], and for NaN, the plain operations.  (Inside it no step
// underflows: a mean small enough for that leaves m == eps.)
template <class Length>
__device__ __forceinline__ float reciprocal_rms(float sumsq, Length length, float eps) {
    const float m = div_shared(sumsq, length.h, length.rcp) + eps;
    constexpr uint32_t LOW = (127u - 60u) << 23, HIGH = (127u + 100u) << 23;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(__builtin_bit_cast(uint32_t, m) - LOW > HIGH - LOW) != 0, 0))
        return 1.0f / __builtin_sqrtf(sumsq / length.h + eps); // in every lane, also of rows inside the range: the same bits
    return reciprocal_of_root(m, __builtin_amdgcn_rsqf(m));
}

// Every buffer is device (global) memory: the few accesses that do not go through a buffer resource
// are typed as address space 1, so they never take the flat aperture check.
#define TDE_GLOBAL __attribute__((address_space(1)))

// Row-sized buffer resources.  A row is addressed as (wavefront-uniform 128-bit resource in SGPRs)
// + (32-bit lane offset in one VGPR).  The resource's size is the row's byte length, or 0 for a row
// past the end: the hardware then returns zeros for loads and drops stores, so neither partially
// filled wavefronts nor tail rows need a branch.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
constexpr int kRsrcFlags = 0x00020000; // raw buffer, 32-bit data format (gfx9 family encoding)
constexpr int kAuxStream = 2; // nt on loads and stores: streamed once, do not keep in cache.
// Measured on MI355X with inputs and outputs rotated far beyond the 256 MB memory-side cache:
// nt loads 7.0 vs 6.4 TB/s read ceiling; nt stores 1-2 % faster than sc1 and 8 % faster than the
// default policy on the 6:1 read/write mix.  (With outputs small enough to stay in that cache,
// sc1 stores measure faster; that is not the HBM-bound case.)
constexpr int kAuxStore = 2;
constexpr int kAuxDefault = 0;

__device__ __forceinline__ rsrc_t row_rsrc(const void *base, int64_t byte_off, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)(static_cast<const char *>(base) + byte_off), 0, (int)bytes,
                                             kRsrcFlags);
}
__device__ __forceinline__ u32x4 rsrc_load16(rsrc_t r, uint32_t off) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, kAuxStream);
}
__device__ __forceinline__ void rsrc_store16(rsrc_t r, uint32_t off, u32x4 v) {
    __builtin_amdgcn_raw_buffer_store_b128(v, r, (int)off, 0, kAuxStore);
}

// Pack VEC fp32 values (already clamped to +-448) to OCP e4m3 bytes, round to nearest even.
template <int VEC>
__device__ __forceinline__ void pack_fp8(const float (&q)[VEC], uint32_t (&out)[VEC / 4]) {
#pragma unroll
    for (int w = 0; w < VEC / 4; ++w) {
        int word = 0;
        word = __builtin_amdgcn_cvt_pk_fp8_f32(q[4 * w], q[4 * w + 1], word, false);
        word = __builtin_amdgcn_cvt_pk_fp8_f32(q[4 * w + 2], q[4 * w + 3], word, true);
        out[w] = (uint32_t)word;
    }
}

// Round to int8 codes, ties to even.  BOUNDED: every q is finite and rounds to a code; adding 1.5 * 2^23 then rounds it and leaves
// the code in the low byte.  Otherwise q has been clamped and NaN becomes 0.
template <int VEC, bool BOUNDED>
__device__ __forceinline__ void pack_int8(const float (&q)[VEC], uint32_t (&out)[VEC / 4]) {
    const auto code = [](float v) {
        if constexpr (BOUNDED) return __builtin_bit_cast(uint32_t, v + 0x1.8p23f);
        else return (uint32_t)(int)__builtin_rintf(v);
    };
#pragma unroll
    for (int w = 0; w < VEC / 4; ++w) {
        const uint32_t lo = __builtin_amdgcn_perm(code(q[4 * w + 1]), code(q[4 * w]), 0x0c0c0400u);
        const uint32_t hi = __builtin_amdgcn_perm(code(q[4 * w + 3]), code(q[4 * w + 2]), 0x04000c0cu);
        out[w] = lo | hi;
    }
}

// What turns a row's elements into codes: the divisor, and its reciprocal in the form that quotient() takes.
//
// Elements of 2 bytes have at most 11 significant bits, and their quotient only has to land on the right side of a code's
// boundary, which has at most 8: the product with a reciprocal in two words, rounded once, gives the same codes as the
// correctly rounded quotient in two instructions instead of three.  Its relative error of 2^-44 could only matter where y lies
// within 2^5 units (of 49 bits) of (2 M +- 1) * d for a boundary M; with d = j 2^20 + r (2^17 for int8) that needs
// M r = -+j with M >= 16 >= j (128), i.e. all ones in d, and even there no code differs as long as the approximation is 1/d
// correctly rounded, which gfx950's is (test_codes_of_every_element_gpu.py).  hi is below 1/d by more than half a unit and lo > 0:
// a numerator of -0 keeps its sign, and of infinity its infinity.  (On the host, for every other mantissa of d, both neighbours
// of 1/d as the approximation and the elements beside every boundary: unit_test_rounding.cpp.)
// fp32 elements take the correctly rounded quotient (div_shared).
template <class E>
struct Divisor {
    float d, hi, lo; // fp32 elements: hi is 1/d correctly rounded

    Divisor() = default;
    __device__ __forceinline__ explicit Divisor(float d_) : Divisor(d_, __builtin_amdgcn_rcpf(d_)) {}
    __host__ __device__ __forceinline__ Divisor(float d_, float approx) {
        d = d_;
        const float r = refined_reciprocal(d, approx);
        if constexpr (E::BYTES == 2) {
            hi = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r) - 1u);
            lo = __builtin_fmaf(-d, hi, 1.0f) * r;
        } else {
            hi = r;
            lo = 0.0f;
        }
    }
    __host__ __device__ __forceinline__ float quotient(float y) const {
        if constexpr (E::BYTES == 2) return __builtin_fmaf(y, hi, y * lo);
        else return div_shared(y, d, hi);
    }
    __device__ __forceinline__ void quotients(const Normed<E> &y, float (&q)[E::VEC]) const {
        if constexpr (E::MIXED) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                q[2 * i] = fma_mix<0>(y.raw[i], hi, mul_mix<0>(y.raw[i], lo));
                q[2 * i + 1] = fma_mix<1>(y.raw[i], hi, mul_mix<1>(y.raw[i], lo));
            }
        } else {
#pragma unroll
            for (int i = 0; i < E::VEC; ++i) q[i] = quotient(y.y[i]);
        }
    }
};

// The largest code of a mode.
template <int Q>
constexpr float kQuantMax = Q == TDE_QUANT_INT8_TOKEN ? 127.0f : 448.0f;

// The dynamic scales of a thread's vectors from the bit patterns of their largest magnitudes.  Returns one wavefront-uniform decision
// for all of them, so the common path carries no per-lane branch: whether every divisor is far from the subnormal and overflow
// ranges, as its quotients need.  A largest magnitude that is NaN or infinite takes the plain division too.
template <int Q, int SCALES>
__device__ __forceinline__ bool scales_of_largest(uint32_t (&m)[SCALES], float (&scale)[SCALES]) {
    constexpr float QMAX = kQuantMax<Q>;
    uint64_t unsafe = 0;
    constexpr uint32_t LOW = (127u - 50u) << 23, HIGH = (127u + 60u) << 23; // 2^-50 to 2^60
#pragma unroll
    for (int j = 0; j < SCALES; ++j)
        unsafe |= __builtin_amdgcn_ballot_w64(m[j] - LOW > HIGH - LOW) & __builtin_amdgcn_ballot_w64(m[j] != 0u);
    const bool fast = unsafe == 0;
#pragma unroll
    for (int j = 0; j < SCALES; ++j) scale[j] = div_shared(__builtin_bit_cast(float, m[j]), QMAX, 1.0f / QMAX);
    if (__builtin_expect(!fast, 0)) {
#pragma unroll
        for (int j = 0; j < SCALES; ++j) {
            asm volatile("; not computed beside the fast one" : "+v"(m[j]));
            scale[j] = __builtin_bit_cast(float, m[j]) / QMAX;
        }
    }
    return fast;
}
__device__ __forceinline__ bool static_scale_is_fast(float scale) {
    return __builtin_amdgcn_readfirstlane(scale >= 0x1p-60f && scale <= 0x1p60f) != 0;
}

// The codes of one vector's elements.  FAST: `divisor` is div's; otherwise the plain division.
template <class E, int Q, bool FAST>
__device__ __forceinline__ void codes_of(const Normed<E> &y, const Divisor<E> &divisor, float div, uint32_t (&codes)[E::VEC / 4]) {
    constexpr int VEC = E::VEC;
    constexpr float QMAX = kQuantMax<Q>;
    float q[VEC];
    if constexpr (FAST && Q == TDE_QUANT_FP8_STATIC && E::BYTES != 2) {
        // A caller's scale can be far below the row's values (the dynamic scales cannot: |y| <= QMAX * scale).
        // Beyond twice the largest code the quotient clamps to QMAX whatever it is, so where its correction
        // would see inf - inf, y is cut there.
#pragma unroll
        for (int i = 0; i < VEC; ++i) q[i] = divisor.quotient(clamp_keep_nan(y.y[i], 2.0f * QMAX * div));
    } else if constexpr (FAST) {
        divisor.quotients(y, q);
    } else {
        y.values(q);
#pragma unroll
        for (int i = 0; i < VEC; ++i) q[i] = q[i] / div;
    }
    // Dynamic scales: the quotient is within 1e-4 of +-QMAX at most, which the conversions below round to
    // the largest code; nothing to clamp
    if constexpr (!FAST || Q == TDE_QUANT_FP8_STATIC) {
#pragma unroll
        for (int i = 0; i < VEC; ++i) q[i] = clamp_keep_nan(q[i], QMAX);
    }
    if constexpr (Q == TDE_QUANT_INT8_TOKEN)
        pack_int8<VEC, FAST>(q, codes);
    else
        pack_fp8<VEC>(q, codes);
}

// Which row group a workgroup takes.  Workgroups are handed to the 8 XCDs round-robin, so in launch order
// every XCD (every L2) walks all of every buffer in 16 KiB steps.  Remapped in groups of 8*chunk, XCD k
// instead takes `chunk` consecutive row groups of each group, i.e. a contiguous piece of every buffer:
// measured 0.5-1.5 % faster with chunks of 8-16 rows (c3 58.4 -> 57.5 us), slower again beyond 64, and 2 %
// slower when each XCD owns one contiguous eighth of the tensor.  A grid tail shorter than a group keeps
// launch order, so the mapping stays one-to-one.
// `chunked`: the workgroups in whole groups, chunked_blocks(grid, chunk).
inline uint32_t chunked_blocks(int64_t grid, uint32_t chunk) { return chunk > 1 ? (uint32_t)grid & ~(8u * chunk - 1u) : 0u; }
__device__ __forceinline__ uint32_t xcd_chunked_block(uint32_t bid, uint32_t chunked, uint32_t chunk) {
    if (chunk > 1) {
        const uint32_t span = 8u * chunk; // power of two
        if (bid < chunked) {
            const uint32_t w = bid & (span - 1u);
            bid = (bid - w) + (w & 7u) * chunk + (w >> 3);
        }
    }
    return bid;
}

// The row that comes i-th in a launch whose rows == owner (mod N) read N partials and the others one staged sum: in each
// window of kOwnedRun * N rows first all of the former, then the others, each in order.  In plain order the long rows
// would meet the same few compute units again and again (workgroups go to the units of an XCD in turn, and N divides
// their number): 8 x [2048, 8192] bf16 -> fp8 35.3 us, 28.2 us in this order.  Windows of a quarter of the length cost 0 to
// 20 % (8 x [5000, 1024] fp16 11.1 -> 14.1 us, 4 x [2048, 8192] 30.5 -> 31.9) and gain 3-4 % on two shapes (2 x [8192, 4096]
// 53.8 -> 52.2, fp32 rows of 532).
constexpr int kOwnedRun = 1024;
template <int N>
__device__ __forceinline__ int64_t owned_first_row(int64_t i, int64_t tokens, int owner, bool &owned) {
    const int64_t window = i / (kOwnedRun * N) * (kOwnedRun * N);
    const int64_t left = tokens - window;
    const int rows = left < kOwnedRun * N ? (int)left : kOwnedRun * N; // of this window; i is past the end if it is <= 0
    const int n_owned = (rows - owner + N - 1) / N;
    const int k = (int)(i - window), other = k - n_owned;
    owned = other < 0;
    if (owned) return window + k * N + owner;
    const int in_span = other % (N - 1);
    return window + other / (N - 1) * N + in_span + (in_span >= owner ? 1 : 0);
}

// The loads of one row: N partial vectors and one residual vector per owned 16-byte column slot.
template <int NP, int VPT>
struct RowLoads {
    u32x4 p[VPT][NP];
    u32x4 r[VPT];
};

// SHIFTED kernels, rows of which start anywhere in a line of memory.  In place, thread t takes vectors t, t + tpr, ... of its row, and what
// each of the row's wavefronts loads and stores begins inside a line whose other part is a neighbour's: nine lines of memory for
// eight lines' worth of data, and stores that are merged, or not, with another wavefront's.  So the row is moved along its threads
// until its wavefronts begin on lines (RowArgs::row_shift), the vectors that fall off the end on the first threads; the row's
// own first and last line are all it still shares.
// Rates in memory, in place -> moved -> the next longer row of whole lines, 12000 rows of 511 vectors: 2 x doubles 5.88 -> 6.26 -> 6.30 TB/s,
// 2 x bf16 5.79 -> 6.14 -> 6.23, 2 x bf16 -> fp8 5.82 -> 6.22 -> 6.27, 4 x fp32 6.10 -> 6.37 -> 6.40, 4 x bf16 -> fp8 staged 5.95 -> 6.25 -> 6.30.
// As a template parameter: the same code without it, a shift of zero, costs launches of whole lines 0.07 us.
template <bool SHIFTED>
__device__ __forceinline__ int first_vector_of(int thread, int shift, int tpr) {
    if constexpr (!SHIFTED) return thread;
    const int v = thread - shift;
    return v < 0 ? v + tpr : v;
}
template <bool SHIFTED>
__device__ __forceinline__ int thread_of(int first_vector, int shift, int tpr) {
    if constexpr (!SHIFTED) return first_vector;
    const int t = first_vector + shift;
    return t >= tpr ? t - tpr : t;
}

// ---------------------------------------------------------------------------------------------
// The row kernel.
//   E      element traits
//   N      number of partials summed per element; N == 0 means "the sum was staged":
//          part[0] already holds s (a T-typed [tokens,hidden] buffer)
//   VPT    16-byte vectors per thread per row (1, 2 or 4)
//   Q      tde_quant
//   WN     write the T-typed normed row (always true for Q == NONE)
//   FORM   kFormWide: compiled for two wavefronts per SIMD (256 registers) instead of three, with gamma requested ahead
//          of the row also for eight partials: two workgroups per CU whose gamma never waits.  Never more than two wavefronts,
//          also where the registers would hold three (fp16 and fp32, 168 and 166 of them: 8 x rows of 600 to 1024 vectors, 1024 to
//          6200 of them, 0.983 of the time, single ones 0.953).  Launched for eight
//          partials with four vectors per thread at 4 to 24 workgroups per CU, to 16 where only codes of a dynamic
//          scale are stored (Geometry::form).
//          kFormStaged: both launches of TDE_ALGO_STAGED in one: the sums are also stored to the stage.
//          kFormOwned: both launches of TDE_ALGO_STAGED_OWNED in one: rows == owner (mod N) are summed from the
//          partials and their sums stored to the stage, every other row's sum is read from the stage
//          kFormLong: fp16 with conversions instead of mixed-precision instructions and packed ones for the rest, for long launches of four partials with
//          four vectors per thread that store codes of per-token scales alone, rows of up to 832 vectors.  What bounds those is memory, and it is served
//          best when the arithmetic holds a row's stores back from the next rows' loads: launches alone, 4 x [32768, 5120] -> int8 takes 341.8 us
//          with the mixed instructions, 339.3 all converted and 334.9 so (as a call of the operator 336.5 either way).  The other long launches of
//          such rows are ahead all converted (tde_converted_rows_f16.hip)
//   SHIFTED rows that are not whole lines of memory, in launches long enough to gain from it (rows_are_shifted)
// Block layout: rows_per_block row groups of threads_per_row threads; thread t of a row group
// owns vectors t, t + threads_per_row, ... (coalesced 1 KiB per wavefront per load) of its row,
// moved along the threads by row_shift() vectors where the row does not start on a line of memory.
// ---------------------------------------------------------------------------------------------
enum : int { kFormPlain = 0, kFormWide = 1, kFormStaged = 2, kFormOwned = 3, kFormLong = 4 };

template <class E, int FORM> struct Arithmetic { typedef E type; };
template <> struct Arithmetic<ElemF16, kFormLong> { typedef ElemF16Unmixed type; };

template <class E, int N, int VPT, int Q, bool WN, int FORM = kFormPlain, bool SHIFTED = false>
__global__ void __launch_bounds__(1024 / VPT)
    // Owned rows of eight partials with two vectors per thread fit eight wavefronts per SIMD without being told, but for fp16: with the mixed
    // instructions it takes 68 registers and seven, and rows of 513 to 575 vectors (29 launches) were 1.2 % behind conversions on average, single ones
    // 4 to 5; with 60 registers and eight 0 to 0.2 %.
    __attribute__((amdgpu_waves_per_eu(VPT == 1 ? 8 : (VPT == 2 ? (E::MIXED && N == 8 && FORM == kFormOwned ? 8 : 5) : (FORM == kFormWide ? 2 : (FORM == kFormOwned ? 4 : 3))), FORM == kFormWide ? 2 : 8)))
    row_kernel(const RowArgs a) {
    constexpr bool WIDE = FORM == kFormWide, OWNED = FORM == kFormOwned;
    constexpr int VEC = E::VEC;
    typedef typename Arithmetic<E, FORM>::type A;
    constexpr int NP = (N == 0) ? 1 : N;
    // residual_out is stored behind the reductions, ahead of the codes: as soon as the sum is known it is 2.4 % slower on
    // 2 x [1257, 6144] static and 7 % on 4 x [512, 5120], behind all codes in one burst 1.7 % on 4 x [32768, 5120] and 1 % on 8 x
    // [2048, 8192] staged.  With a static scale, and where a stage is stored too, it goes out with the normed row already: 1 % and
    // 0.6 % faster there; elsewhere the same, but 2 x [700, 4096] fp16 -> fp8 10 % slower.
    // Dynamic LDS: the workgroup's squares (one float per element it holds), then 1024 floats of block sums.
    extern __shared__ __attribute__((aligned(16))) float lds_dyn[];
    float *const lds_img = lds_dyn;
    float *const lds_bs = lds_dyn + (uint32_t)a.threads_per_row * a.rows_per_block * (VPT * VEC);
    __shared__ uint32_t lds_max[kMaxWavesPerBlock]; // one per row group

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tpr = a.threads_per_row;
    const int waves_per_row = tpr >> 6;
    const int group = a.row_group(wave); // uniform inside a wavefront
    const int first_wave = group * waves_per_row;
    const uint32_t row_bytes = (uint32_t)a.hidden() * E::BYTES;

    const void *part[NP];
    partial_addresses(a, a.address(kPtrStage), part);

    // One workgroup, one group of rows: the grid covers every row (no loop; a looping wavefront waits for its
    // own stores, a fresh workgroup does not).
    int64_t row = (int64_t)xcd_chunked_block(blockIdx.x, a.chunked_blocks, a.xcd_chunk) * a.rows_per_block + group;
    bool sum_is_new = FORM == kFormStaged; // the row's sums go to the stage as well
    if constexpr (OWNED) row = owned_first_row<N>(row, a.tokens, a.owner, sum_is_new);

    // Thread t of the row group owns vectors t, t + tpr, ... of the row, which is first moved along the threads.
    const int shift = SHIFTED ? a.row_shift(row * (int64_t)row_bytes) : 0;
    const int t_row = first_vector_of<SHIFTED>(tid - group * tpr, shift, tpr);
    uint32_t lane_off[VPT]; // byte offset of this thread's vector j inside a row
#pragma unroll
    for (int j = 0; j < VPT; ++j) lane_off[j] = (uint32_t)(j * tpr + t_row) * 16u;
// The row's first vector of this thread and the lane index, rebuilt from the first load offset where they are needed:
// the thread id itself does not stay in a register through the load phase, which has none to spare.
#define TDE_T ((int)(lane0 >> 4))
// The same, not before `after` is there: with several vectors per thread the row loads leave no registers for LDS addresses.
#define TDE_T_BEHIND(after) (VPT == 1 ? TDE_T : not_before(TDE_T, after))
#define TDE_LANE (((int)(lane0 >> 4) + shift) & (kWave - 1))

    auto issue_loads = [&](RowLoads<NP, VPT> &d, int64_t row) {
        const uint32_t bytes = (row < a.tokens) ? row_bytes : 0u;
        const int64_t row_byte = row * (int64_t)row_bytes;
        if constexpr (!OWNED) {
#pragma unroll
            for (int r = 0; r < NP; ++r) {
                const rsrc_t rs = row_rsrc(part[r], row_byte, bytes);
#pragma unroll
                for (int j = 0; j < VPT; ++j) d.p[j][r] = rsrc_load16(rs, lane_off[j]);
            }
        }
        const rsrc_t rr = row_rsrc(a.ptr(kPtrResidualIn), row_byte, bytes);
#pragma unroll
        for (int j = 0; j < VPT; ++j) d.r[j] = rsrc_load16(rr, lane_off[j]);
    };

    // The row's loads go out before anything else touches memory -- except gamma where it pays to have it first:
    // with up to four partials of a 2-byte type, several vectors per thread and a dynamic scale, the registers are
    // there to hold gamma through the load phase, and requested ahead of the row (it is served from L2) it is never
    // waited for behind the row's own traffic.  Measured against requesting it after the accumulate phase, alternating
    // two builds in one process: 4 x [32768, 5120] fp16 -> int8 per token -1.0 %, 4 x [8192, 7168] bf16 -> fp8 per
    // token -1.4 %, 2 x [8192, 8192] -0.6 %, 4 x [2048, 7168] -0.7 %; with per-group scales 4 x [8192, 7168] -1.1 %,
    // 2 x [9000, 7168] -0.6 %; with T-typed output or fp32 rows equal to +0.4 %, so those keep the late request.
    // With eight partials the 16 registers are one too many for three wavefronts per SIMD (169 against 168: spilling
    // costs 2 us on 8 x [2048, 8192], and gamma ahead of the row for three of the four vectors gains 0.1 us); the WIDE
    // instantiation takes them and runs two workgroups per CU: 8 x [2048, 8192] bf16 -> fp8 56.8 us against 57.3,
    // -0.8 % from 1024 to 4096 rows, -1.5 % for rows of 7168, -2.2 % for 4096 rows of 2048, nothing from 6144 rows on
    // (where the launch is limited to two workgroups per CU anyway) and +0.8 to +1.8 % below 1024 rows.  The other
    // eight-partial kernels gain less but none loses (per-group scales -1.0 %, T-typed output -0.3 to -0.8 %, fp32 rows
    // -0.2 to -0.9 %), so WIDE carries gamma ahead of the row for all of them.
    const rsrc_t gamma_rsrc = row_rsrc(a.ptr(kPtrGamma), 0, row_bytes);
    constexpr bool GAMMA_FIRST =
        VPT > 1 && N != 0 && !OWNED &&
        (WIDE || (N <= 4 && E::BYTES == 2 && (Q == TDE_QUANT_FP8_TOKEN || Q == TDE_QUANT_INT8_TOKEN || Q == TDE_QUANT_FP8_GROUP)));
    u32x4 gamma_first[GAMMA_FIRST ? VPT : 1];
    if constexpr (GAMMA_FIRST) {
#pragma unroll
        for (int j = 0; j < VPT; ++j)
            gamma_first[j] = __builtin_amdgcn_raw_buffer_load_b128(gamma_rsrc, (int)lane_off[j], 0, kAuxDefault);
        __builtin_amdgcn_sched_barrier(0);
    }
    RowLoads<NP, VPT> cur;
    issue_loads(cur, row);
    u32x4 gamma_early = u32x4{0, 0, 0, 0};
    if constexpr (VPT == 1) {
        __builtin_amdgcn_sched_barrier(0);
        gamma_early = __builtin_amdgcn_raw_buffer_load_b128(gamma_rsrc, (int)lane_off[0], 0, kAuxDefault);
    }
    // From here on only the first offset stays in a register (the compiler cannot see where it came from, so it
    // keeps neither the thread index nor the other offsets alive through the load phase); the others are one
    // addition away.
    uint32_t lane0 = lane_off[0];
    asm volatile("" : "+v"(lane0));
    const uint32_t vec_stride = (uint32_t)tpr * 16u;
    const SumLayout<VPT, VEC, E::BYTES == 2> sums(lds_img, lds_bs, a.hidden(), tpr, a.rows_per_block, group);
    sumsq_clear(sums, TDE_T);
    if constexpr (Q == TDE_QUANT_FP8_TOKEN || Q == TDE_QUANT_INT8_TOKEN) lds_max[group] = 0u; // for row_max
    // Scalar registers for owned rows: with eight partials and four vectors per thread their 128 vector registers spilled one
    // otherwise (4 bytes a lane to scratch and back; 8 x [2048, 8192] 27.32 -> 27.24 us).
    const RowLength<OWNED> length(a.hidden());
#define TDE_OFF(j) (lane0 + (uint32_t)(j) * vec_stride)

    {
        const bool row_ok = row < a.tokens;
        const uint32_t bytes = row_ok ? row_bytes : 0u;
        const int64_t row_byte = row * (int64_t)row_bytes; // wavefront-uniform

        // ---- reduce, residual add, sum of squares ------------------------------------------------
        const rsrc_t res_out = row_rsrc(a.ptr(kPtrResidualOut), row_byte, bytes);
        u32x4 xraw[VPT];
        // With four vectors per thread, or one, the partials are summed rank by rank as they arrive (the memory system
        // returns a wavefront's loads in the order it issued them), so that only the last partial's additions are
        // left when the row is complete.  The order of every element's additions is the same either way.  With two
        // vectors per thread the accumulators cost more occupancy than the overlap returns (8 partials, 1024 rows of
        // 5120: 21.5 us against 20.4), so those variants sum vector by vector.  With one vector per thread (the
        // decode-size geometries) waiting rank by rank is worth 0.5-1.5 % up to 512 rows and nothing beyond.
        constexpr bool RANK_MAJOR = !OWNED && (N >= 4 && (VPT >= 4 || VPT == 1));
        u32x4 sraw[VPT]; // the row's sums, rounded to T
        if constexpr (OWNED) {
            // Four partials of fp16 with four vectors per thread: decided by a scalar where T-typed rows alone are stored.  As a mask of lanes the
            // compiler lets the two ways of loading share registers, and these kernels then waited for the residual ahead of the partials: 58 launches
            // 0.3 % slower on average, of 250 to 500 rows 3 to 13 % (4 x [283, 6272] 6.29 us against 5.62).  Beside codes the same wait happens to pay,
            // 1.5 % on average; of other types and row lengths nothing waits, and a scalar moves single launches by up to 11 % either way.
            constexpr bool SCALAR = E::MIXED && N == 4 && VPT == 4 && Q == TDE_QUANT_NONE;
            const bool sum_here = SCALAR ? __builtin_amdgcn_readfirstlane((int)sum_is_new) != 0 : sum_is_new;
            if (sum_here) {
                // At most four partials in flight per vector: each one's registers are loaded with the partial four
                // ranks on as soon as it has been added.  That keeps the kernel within 128 registers, four wavefronts
                // per SIMD, which the rows that only read the stage need to have enough loads in flight (limited to
                // two or three workgroups per CU 8 x [2048, 8192] takes 29.4 and 28.6 us instead of 28.2).
                constexpr int B = N < 4 ? N : 4;
                u32x4 p[VPT][B];
                float acc[VPT][VEC];
                auto request = [&](int r) {
                    const rsrc_t rs = row_rsrc(part[r], row_byte, bytes);
#pragma unroll
                    for (int j = 0; j < VPT; ++j) p[j][r % B] = rsrc_load16(rs, TDE_OFF(j));
                };
#pragma unroll
                for (int r = 0; r < B; ++r) request(r);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int r = 0; r < N; ++r) {
#pragma unroll
                    for (int j = 0; j < VPT; ++j) accumulate<A>(p[j][r % B], acc[j], r == 0);
                    if (r + B < N) request(r + B);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int j = 0; j < VPT; ++j) sraw[j] = E::pack(acc[j]);
            } else {
                const rsrc_t rs = row_rsrc(a.ptr(kPtrStage), row_byte, bytes);
#pragma unroll
                for (int j = 0; j < VPT; ++j) sraw[j] = rsrc_load16(rs, TDE_OFF(j));
            }
        }
        float racc[RANK_MAJOR ? VPT : 1][VEC];
        if constexpr (RANK_MAJOR) {
            __builtin_amdgcn_sched_barrier(0);
            // The first two partials are taken together, vector by vector: their eight sums fit the registers the
            // two vectors arrived in, so the accumulators cost no registers while all other loads are in flight.
#pragma unroll
            for (int j = 0; j < VPT; ++j) {
                accumulate<A>(cur.p[j][0], racc[j], true);
                accumulate<A>(cur.p[j][1], racc[j], false);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int r = 2; r < NP; ++r) {
#pragma unroll
                for (int j = 0; j < VPT; ++j) accumulate<A>(cur.p[j][r], racc[j], false);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            if constexpr (OWNED) {
                // above
            } else if constexpr (N == 0) {
                sraw[j] = cur.p[j][0];
            } else if constexpr (RANK_MAJOR) {
                sraw[j] = E::pack(racc[j]);
            } else {
                float acc[VEC];
#pragma unroll
                for (int r = 0; r < NP; ++r) accumulate<A>(cur.p[j][r], acc, r == 0);
                sraw[j] = E::pack(acc);
            }
            xraw[j] = added<A>(sraw[j], cur.r[j]);
            float sq[VEC];
            squares_of<A>(xraw[j], sq);
            put_squares(sums.img + (j * tpr + TDE_T_BEHIND(xraw[j][0])) * VEC, sq);
        }
        if (sums.n != sums.chained) {
#pragma unroll
            for (int j = 0; j < VPT; ++j) {
                float sq[VEC];
                squares_of<A>(xraw[j], sq);
                split_left(sums, j * tpr + TDE_T_BEHIND(xraw[j][0]), sq);
            }
        }
        // gamma (shared by all rows, served from L2).  With several vectors per thread it is requested
        // only now (unless it went out first, see GAMMA_FIRST): the registers of the row loads are free
        // again, and the reduction below covers its latency.  With one vector per thread registers are
        // plentiful and it was requested right behind the row loads (shortest dependent chain for small,
        // latency-bound inputs).
        u32x4 gamma_raw[VPT];
        if constexpr (GAMMA_FIRST) {
#pragma unroll
            for (int j = 0; j < VPT; ++j) gamma_raw[j] = gamma_first[j];
        } else if constexpr (VPT > 1) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < VPT; ++j)
                gamma_raw[j] = __builtin_amdgcn_raw_buffer_load_b128(gamma_rsrc, (int)TDE_OFF(j), 0, kAuxDefault);
        } else {
            gamma_raw[0] = gamma_early;
        }
        // The stage behind the gamma request: a wavefront's loads and stores are waited for in order, and gamma would
        // otherwise wait for these stores.
        if (sum_is_new) {
            const rsrc_t stage = row_rsrc(a.ptr(kPtrStage), row_byte, bytes);
#pragma unroll
            for (int j = 0; j < VPT; ++j) rsrc_store16(stage, TDE_OFF(j), sraw[j]);
        }
        const int t_behind = thread_of<SHIFTED>(TDE_T_BEHIND(xraw[VPT - 1][0]), shift, tpr);
        const float sumsq = sumsq_torch_order<SHIFTED>(sums, t_behind, tpr, wave - first_wave, t_behind & (kWave - 1));
        const float rs = reciprocal_rms(sumsq, length, a.eps);

        // ---- normalize ------------------------------------------------------------------------------
        constexpr bool DYNAMIC = Q != TDE_QUANT_NONE && Q != TDE_QUANT_FP8_STATIC;
        constexpr bool EARLY_RESIDUAL = Q == TDE_QUANT_FP8_STATIC || (Q != TDE_QUANT_NONE && FORM == kFormStaged);
        constexpr int QUANT_VPT = Q == TDE_QUANT_NONE ? 1 : VPT;
        Normed<A> y[QUANT_VPT]; // what is quantized
        float amax[VPT];         // largest magnitude per vector
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            const u32x4 nraw = normed<A>(xraw[j], gamma_raw[j], rs);
            if constexpr (Q == TDE_QUANT_NONE || WN) {
                const rsrc_t norm_out = row_rsrc(a.ptr(kPtrNorm), row_byte, bytes);
                rsrc_store16(norm_out, TDE_OFF(j), nraw);
            }
            if constexpr (Q != TDE_QUANT_NONE) y[j] = Normed<A>(nraw);
            if constexpr (DYNAMIC) amax[j] = y[j].largest();
            if constexpr (EARLY_RESIDUAL) rsrc_store16(res_out, TDE_OFF(j), xraw[j]);
        }

        if constexpr (Q == TDE_QUANT_NONE) {
#pragma unroll
            for (int j = 0; j < VPT; ++j) rsrc_store16(res_out, TDE_OFF(j), xraw[j]);
        }

        // ---- quant epilogue -------------------------------------------------------------------------
        if constexpr (Q != TDE_QUANT_NONE) {
            constexpr int SCALES = Q == TDE_QUANT_FP8_GROUP ? VPT : 1; // a thread's vectors lie in groups of their own
            float scale[SCALES];
            bool fast;
            if constexpr (DYNAMIC) {
                uint32_t m[SCALES];
                if constexpr (Q == TDE_QUANT_FP8_GROUP) {
#pragma unroll
                    for (int j = 0; j < VPT; ++j) {
                        m[j] = row16_max(__builtin_bit_cast(uint32_t, amax[j]) & 0x7fffffffu);
                        if constexpr (TDE_QUANT_GROUP / VEC == 32) m[j] = max_u32(m[j], (uint32_t)__shfl_xor((int)m[j], 16, kWave));
                    }
                } else {
#pragma unroll
                    for (int j = 1; j < VPT; ++j) amax[0] = max_abs(amax[0], amax[j], amax[j]);
                    m[0] = row_max(__builtin_bit_cast(uint32_t, amax[0]) & 0x7fffffffu, lds_max + group, TDE_LANE, waves_per_row);
                }
                fast = scales_of_largest<Q>(m, scale);
            } else {
                scale[0] = a.static_scale;
                fast = static_scale_is_fast(a.static_scale);
            }
            if constexpr (Q == TDE_QUANT_FP8_GROUP) {
                constexpr int LANES_PER_GROUP = TDE_QUANT_GROUP / VEC; // 16 (2-byte types) or 32 (fp32)
                const int64_t groups_per_row = a.hidden() / TDE_QUANT_GROUP;
                const rsrc_t sc_out = row_rsrc(a.ptr(kPtrScale), row * groups_per_row * 4, row_ok ? (uint32_t)groups_per_row * 4u : 0u);
                if ((TDE_LANE & (LANES_PER_GROUP - 1)) == 0) {
#pragma unroll
                    for (int j = 0; j < VPT; ++j)
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, scale[j]), sc_out,
                                                              (int)((TDE_OFF(j) / 16u / LANES_PER_GROUP) * 4u), 0, kAuxDefault);
                }
            } else if constexpr (DYNAMIC) {
                if (row_ok && TDE_T == 0) ((TDE_GLOBAL float *)a.ptr(kPtrScale))[row] = scale[0];
            }
            const rsrc_t q_out = row_rsrc(a.ptr(kPtrCodes), row * (int64_t)a.hidden(), row_ok ? (uint32_t)a.hidden() : 0u);
            if constexpr (!EARLY_RESIDUAL) {
#pragma unroll
                for (int j = 0; j < VPT; ++j) rsrc_store16(res_out, TDE_OFF(j), xraw[j]);
            }
            auto quantize = [&](auto use_fast) {
                constexpr bool FAST = decltype(use_fast)::value;
                Divisor<A> divisor;
#pragma unroll
                for (int j = 0; j < VPT; ++j) {
                    const float sc = scale[SCALES == 1 ? 0 : j];
                    const float div = (Q == TDE_QUANT_FP8_STATIC || sc > 0.0f) ? sc : 1.0f;
                    if (FAST && (SCALES > 1 || j == 0)) divisor = Divisor<A>(div);
                    uint32_t codes[VEC / 4];
                    codes_of<A, Q, FAST>(y[j], divisor, div, codes);
                    const uint32_t code_off = (TDE_OFF(j) / 16u) * (uint32_t)VEC;
                    if constexpr (VEC == 8) {
                        const u32x2 w = {codes[0], codes[1]};
                        __builtin_amdgcn_raw_buffer_store_b64(w, q_out, (int)code_off, 0, kAuxStore);
                    } else {
                        __builtin_amdgcn_raw_buffer_store_b32(codes[0], q_out, (int)code_off, 0, kAuxStore);
                    }
                }
            };
            if (__builtin_expect(fast, 1))
                quantize(std::true_type{});
            else
                quantize(std::false_type{});
        }
    }
}
#undef TDE_T
#undef TDE_T_BEHIND
#undef TDE_LANE
#undef TDE_OFF

// Stage A of the staged algorithm: s = T(sum of partials) for every element, no row structure.
// One workgroup of 256 threads reduces a contiguous span of 256*U vectors (U vectors per thread,
// all N*U loads in flight before the first add) and exits; spans past the end are cut by the buffer
// resource's size, so there is no loop and no tail branch.  U = 4 is the faster choice over the whole
// tensor (8 partials x 32 MiB: 50.5 us against 52.9 us with U = 2); for single 16 KiB rows it would
// leave one workgroup per row, and U = 2 (two per row) measures slightly faster there.
// Which bytes stage A covers: `row_bytes` long rows first_row, first_row + row_step, ...; each row is cut
// into spans_per_row spans.  The whole tensor as one long "row" (first_row 0) is the all-rows form; the
// reference's two-shot share of one rank is rows == rank (mod nranks) (impl.h:365-366).
struct ReduceSpan {
    int64_t row_bytes;
    int64_t first_row;
    int64_t row_step;
    int64_t spans_per_row;
    uint32_t xcd_chunk; // spans each XCD takes in a row (xcd_chunked_block); 16 over whole tensors, 1 for single rows
    uint32_t chunked_blocks;
    uint64_t table; // device pointer table of the partials that RowArgs::table_mask names
};

template <class E, int N, int U>
__global__ void __launch_bounds__(256) reduce_kernel(const RowArgs a, const ReduceSpan sp) {
    constexpr int VEC = E::VEC;
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
        float acc[VEC];
#pragma unroll
        for (int r = 0; r < N; ++r) accumulate<E>(raw[u][r], acc, r == 0);
        // The staged sum is re-read by stage B right away: default (cacheable) store.
        __builtin_amdgcn_raw_buffer_store_b128(E::pack(acc), out, (int)((u * 256 + threadIdx.x) * 16), 0, kAuxDefault);
    }
}

// ---------------------------------------------------------------------------------------------
// Host-side launch geometry shared by tde_plan and the launchers.
// ---------------------------------------------------------------------------------------------
struct Geometry {
    int wgs_per_cu; // limit on resident workgroups per compute unit (0 = none), enforced through lds_bytes
    int lds_bytes;  // dynamic LDS of the row kernel's launch: its own, padded for wgs_per_cu
    int vec_elems;
    int nvec;
    int vpt;
    int threads_per_row; // below 64: short rows, several to a wavefront
    int rows_per_block;
    int block_threads;
    int64_t grid;
    int xcd_chunk;
    int line_mask; // RowArgs::line_mask
    int form;  // which instantiation of the row kernel (kFormPlain, kFormWide, kFormStaged, kFormOwned, kFormLong)
    bool converted; // fp16: tde_converted_rows_f16.hip
};

// Per-dtype launchers, defined in tde_rows_<dtype>.hip.
hipError_t launch_rows_bf16(int n, int vpt, int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s);
hipError_t launch_rows_f16(int n, int vpt, int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s);
hipError_t launch_rows_f32(int n, int vpt, int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s);
// The same for rows that are moved along their threads (a.line_mask), in tde_shifted_rows_<dtype>.hip; n != 0, no per-group scales.
hipError_t launch_shifted_rows_bf16(int n, int vpt, int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s);
hipError_t launch_shifted_rows_f16(int n, int vpt, int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s);
hipError_t launch_shifted_rows_f32(int n, int vpt, int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s);
// fp16, four partials, four vectors per thread, rows in place or moved: plain and, T-typed output only, staged.
hipError_t launch_converted_rows_f16(int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s);
hipError_t launch_reduce_bf16(int n, const RowArgs &a, uint64_t table, int64_t row_bytes, int64_t first_row, int64_t row_step, int64_t rows, hipStream_t s);
hipError_t launch_reduce_f16(int n, const RowArgs &a, uint64_t table, int64_t row_bytes, int64_t first_row, int64_t row_step, int64_t rows, hipStream_t s);
hipError_t launch_reduce_f32(int n, const RowArgs &a, uint64_t table, int64_t row_bytes, int64_t first_row, int64_t row_step, int64_t rows, hipStream_t s);

// Rows of up to 32 vectors, several to a wavefront (tde_short_rows.hip; not doubles).  The normed rows go where the arguments have a
// buffer for them.
constexpr int kShortRowVecs = 32;
constexpr uint32_t kPastEnd = 0x7ffffff0u; // an offset beyond every resource of theirs: loads give zeros, stores are dropped
inline size_t short_rows_lds_bytes(int block_threads, int rows_per_block, int vec_floats) {
    return ((size_t)block_threads * vec_floats + (size_t)rows_per_block * 32) * sizeof(float);
}
hipError_t launch_short_rows(int dtype, int n, int q, const RowArgs &a, const Geometry &g, hipStream_t s);

// Rows of doubles (tde_rows_f64.hip): no quantized output.
hipError_t launch_rows_f64(int n, const RowArgs &a, const Geometry &g, hipStream_t s);
hipError_t launch_reduce_f64(int n, const RowArgs &a, uint64_t table, int64_t row_bytes, int64_t first_row, int64_t row_step, int64_t rows, hipStream_t s);

// Traffic skeleton of the row kernel (tde_probe.hip): same geometry and bytes, no arithmetic.
hipError_t launch_traffic(int n, int vpt, int code_bytes, bool wn, const RowArgs &a, const Geometry &g, uint32_t row_bytes, uint32_t parts,
                          hipStream_t s);

// Instantiation + dispatch body used by the three per-dtype translation units.
template <class E, bool SHIFTED, int N, int VPT>
hipError_t launch_rows_nv(int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s) {
    const dim3 grid((unsigned)g.grid), block((unsigned)g.block_threads);
    const size_t lds = (size_t)g.lds_bytes; // sumsq_lds_bytes of this geometry, padded where the launch limits workgroups per CU
#define TDE_LAUNCH_FORM(QM, WNB, FORM)                                                                   \
    {                                                                                                    \
        if (lds > kDefaultMaxDynamicLds) {                                                               \
            const hipError_t e = allow_large_lds<row_kernel<E, N, VPT, QM, WNB, FORM, SHIFTED>>();       \
            if (e != hipSuccess) return e;                                                               \
        }                                                                                                \
        return launch_kernel<row_kernel<E, N, VPT, QM, WNB, FORM, SHIFTED>>(grid, block, lds, s, a);     \
    }
#define TDE_LAUNCH(QM, WNB)                                                                              \
    if constexpr (N == 8 && VPT == 4) {                                                                  \
        if (g.form == kFormWide) TDE_LAUNCH_FORM(QM, WNB, kFormWide)                                     \
    }                                                                                                    \
    if constexpr (N == 4 && VPT == 4 && E::MIXED && !WNB && (QM == TDE_QUANT_FP8_TOKEN || QM == TDE_QUANT_INT8_TOKEN)) { \
        if (g.form == kFormLong) TDE_LAUNCH_FORM(QM, WNB, kFormLong)                                     \
    }                                                                                                    \
    if constexpr (N != 0) {                                                                              \
        if (g.form == kFormStaged) TDE_LAUNCH_FORM(QM, WNB, kFormStaged)                                 \
        if (g.form == kFormOwned) TDE_LAUNCH_FORM(QM, WNB, kFormOwned)                                   \
    }                                                                                                    \
    TDE_LAUNCH_FORM(QM, WNB, kFormPlain)
    switch (q) {
    case TDE_QUANT_NONE: TDE_LAUNCH(TDE_QUANT_NONE, true)
    case TDE_QUANT_FP8_TOKEN:
        if (wn) { TDE_LAUNCH(TDE_QUANT_FP8_TOKEN, true) } else { TDE_LAUNCH(TDE_QUANT_FP8_TOKEN, false) }
    case TDE_QUANT_FP8_GROUP:
        if constexpr (!SHIFTED) { // rows of whole groups are whole lines
            if (wn) { TDE_LAUNCH(TDE_QUANT_FP8_GROUP, true) } else { TDE_LAUNCH(TDE_QUANT_FP8_GROUP, false) }
        }
        break;
    case TDE_QUANT_INT8_TOKEN:
        if (wn) { TDE_LAUNCH(TDE_QUANT_INT8_TOKEN, true) } else { TDE_LAUNCH(TDE_QUANT_INT8_TOKEN, false) }
    case TDE_QUANT_FP8_STATIC:
        if (wn) { TDE_LAUNCH(TDE_QUANT_FP8_STATIC, true) } else { TDE_LAUNCH(TDE_QUANT_FP8_STATIC, false) }
    }
#undef TDE_LAUNCH
#undef TDE_LAUNCH_FORM
    return hipErrorInvalidValue;
}

template <class E, bool SHIFTED, int N>
hipError_t launch_rows_n(int vpt, int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s) {
    if (vpt == 1) return launch_rows_nv<E, SHIFTED, N, 1>(q, wn, a, g, s);
    if (vpt == 2) return launch_rows_nv<E, SHIFTED, N, 2>(q, wn, a, g, s);
    if (vpt == 4) return launch_rows_nv<E, SHIFTED, N, 4>(q, wn, a, g, s);
    return hipErrorInvalidValue;
}

template <class E, bool SHIFTED>
hipError_t launch_rows_e(int n, int vpt, int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s) {
    switch (n) {
    case 0:
        if constexpr (!SHIFTED) return launch_rows_n<E, false, 0>(vpt, q, wn, a, g, s);
        break;
    case 2: return launch_rows_n<E, SHIFTED, 2>(vpt, q, wn, a, g, s);
    case 4: return launch_rows_n<E, SHIFTED, 4>(vpt, q, wn, a, g, s);
    case 8: return launch_rows_n<E, SHIFTED, 8>(vpt, q, wn, a, g, s);
    }
    return hipErrorInvalidValue;
}

template <class E, int N, int U>
hipError_t launch_reduce_nu(const RowArgs &a, uint64_t table, int64_t row_bytes, int64_t first_row, int64_t row_step, int64_t rows,
                            hipStream_t s) {
    constexpr int64_t span = 256 * U * 16;
    ReduceSpan sp{row_bytes, first_row, row_step, (row_bytes + span - 1) / span, rows == 1 ? 16u : 1u, 0u, table};
    const int64_t blocks = rows * sp.spans_per_row;
    if (blocks <= 0) return hipSuccess;
    if (blocks > 0x7fffffff) return hipErrorInvalidValue; // grid dimension limit
    sp.chunked_blocks = chunked_blocks(blocks, sp.xcd_chunk);
    return launch_kernel<reduce_kernel<E, N, U>>(dim3((unsigned)blocks), dim3(256), 0, s, a, sp);
}

template <class E, int N>
hipError_t launch_reduce_n(const RowArgs &a, uint64_t table, int64_t row_bytes, int64_t first_row, int64_t row_step, int64_t rows,
                           hipStream_t s) {
    if (N >= 8 && row_bytes <= 256 * 4 * 16) return launch_reduce_nu<E, N, 2>(a, table, row_bytes, first_row, row_step, rows, s);
    return launch_reduce_nu<E, N, 4>(a, table, row_bytes, first_row, row_step, rows, s);
}

// Stage A over rows first_row, first_row + row_step, ... (`rows` of them), each row_bytes long.
template <class E>
hipError_t launch_reduce_e(int n, const RowArgs &a, uint64_t table, int64_t row_bytes, int64_t first_row, int64_t row_step, int64_t rows,
                           hipStream_t s) {
    switch (n) {
    case 2: return launch_reduce_n<E, 2>(a, table, row_bytes, first_row, row_step, rows, s);
    case 4: return launch_reduce_n<E, 4>(a, table, row_bytes, first_row, row_step, rows, s);
    case 8: return launch_reduce_n<E, 8>(a, table, row_bytes, first_row, row_step, rows, s);
    }
    return hipErrorInvalidValue;
}

} // namespace tde
