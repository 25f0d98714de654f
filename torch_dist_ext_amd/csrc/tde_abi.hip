// C ABI of libtde_hip.so: validation, launch geometry, kernel dispatch and the emulated peer
// workspace.  Declarations and the reference interfaces they replace are in include/tde_abi.h.
#include <hip/hip_runtime.h>

#include <algorithm>

#include <cstdint>
#include <cstring>
#include <mutex>
#include <new>

#include "tde_abi.h"
#include "tde_rows.h"

// Stage buffer of tde_reduce_rms_static_stage: part of the library's device image, one copy per GPU, held
// until the process ends.  Host code never uses this name as an address: static_stage_ptr() asks the
// runtime for the current device's copy once and keeps the answer.
static __device__ __align__(256) unsigned char scratch[TDE_STATIC_STAGE_BYTES];

namespace {

thread_local int g_last_hip_error = 0;

int hip_fail(hipError_t e) {
    g_last_hip_error = (int)e;
    return TDE_EHIP;
}

int elem_bytes(int dtype) {
    switch (dtype) {
    case TDE_BF16:
    case TDE_F16: return 2;
    case TDE_F32: return 4;
    case TDE_F64: return 8;
    }
    return 0;
}

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device (looked up on the first call per device).
int static_stage_ptr(void **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    if (dev < 0 || dev >= kMaxDevices) return TDE_EINVAL;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e);
        if (ptr == nullptr) return TDE_EINVAL;
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return TDE_OK;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

constexpr int kMaxBlock = 1024;
constexpr int64_t kLoadsInFlightPerCu = 128 * 1024; // target for the limit on resident workgroups (see validate)
// launches with fewer workgroups per compute unit are not limited: 24 with 8 partials, 32 with 4 (whose launches are
// shorter), i.e. 6144 and 8192 workgroups on the 256 CUs of an unpartitioned MI355X; launches of either that store little (few_stores) also
// from 16 to 30.  (From 30 to 32 four partials that store little would gain 2 to 4.5 % from it as well -- 33 launches of 7680 to 8191 rows -- and are
// planned without, which test_abi_host.py and test_workgroup_limits.py pin.)
constexpr int64_t kLimitFromWorkgroupsPerCu8 = 24, kLimitFromWorkgroupsPerCu4 = 32;
constexpr int64_t kFewStoresFrom = 16, kFewStoresUntil = 30;
constexpr int kDefaultComputeUnits = 256; // MI355X; used when no device can be asked (planning on a host without one)

// Compute units of the current device, asked once per device and thread (no lock on the launch path).
int compute_units() {
    thread_local int cached_dev = -1, cached_cu = 0;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) {
        (void)hipGetLastError();
        return kDefaultComputeUnits;
    }
    if (dev != cached_dev) {
        int cu = 0;
        if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cu <= 0) {
            (void)hipGetLastError();
            cu = kDefaultComputeUnits;
        }
        cached_dev = dev;
        cached_cu = cu;
    }
    return cached_cu;
}

// The row counts in the rules for vectors per thread below were swept on 256 compute units.  What they mark is how many rows
// each unit gets -- a launch's time rises in steps, with every further workgroup on the fullest unit, and the steps lie at
// different counts for workgroups of different sizes -- so a device (or partition) with another number of units is asked for
// the same rows per unit.
int64_t rows_as_on_256_units(int64_t tokens, int64_t cus) {
    return cus == 256 ? tokens : tokens / cus * 256 + tokens % cus * 256 / cus;
}

// Whether every row starts and ends on a 128-byte line.  Other rows share their first and last line with their neighbours, and
// several vectors per thread (fewer wavefronts, whose stores lie further apart in time) then lose 2-6 % of a long launch that stores
// much: 2 x 16384 rows of 608 vectors, T-typed output, +3.1 % over one vector per thread, of 609 -3.1 %.
// (Rows left in place; where rows are shifted, below, the rules stated for either kind are within 0.7 % of the best choice.)
bool rows_of_whole_lines(int64_t nvec) { return nvec % 8 == 0; }

// Vectors per thread for rows of doubles in one launch (4 partials x 2048 rows of 2048 in all: 38.5 -> 38.0 us; 2 x 900 rows of
// 1700: 15.3 -> 13.2).  Four against one, swept over 2/4/8 partials x rows of 128 to 1024 vectors x 256 to 32768 rows (some 5000
// launches of other sizes): 1-20 % faster while the launch's steps (one workgroup more on the fullest compute unit) favour
// the narrow workgroups, which ends at the row counts below; beyond them 1-9 % slower.  By wavefronts of a row with one
// vector per thread; rows that fill their lanes, or nearly (13 and 14 wavefronts), gain the longest.
int vecs_per_thread_f64(const tde_problem *p, int64_t nvec, int64_t t) {
    const bool two = p->nranks == 2, four = p->nranks == 4, many = p->nranks >= 8, full = nvec % 256 == 0;
    const bool staged = p->algo == TDE_ALGO_STAGED, owned = p->algo == TDE_ALGO_STAGED_OWNED;
    if (staged || owned) { // swept with the stage: the one launch moves a stream more, or its rows read two streams only
        if (many && !owned && nvec >= 128 && nvec <= 320 && t >= (nvec < 256 ? 8192 : 256)) return 4; // 3-4 %
        if (nvec < 256 || t < 256) return 1;
        if (two && nvec > 576 && nvec <= 640) return 4;            // ten wavefronts per row: 3-13 % at any length
        if (many && owned && nvec > 640 && nvec <= 768) return 4; // 700 vectors: 3-6 % at any length
        return t < (full || nvec > 768 ? (many ? 6144 : 3072) : 1536) ? 4 : 1;
    }
    if (many && nvec >= 128 && nvec < 256) return t >= 8192 ? 4 : 1; // 2-6 %
    if (nvec < 256 || t < 256) return 1;
    const bool lines = rows_of_whole_lines(nvec);
    // the fifth workgroup per unit: four vectors 1-8 % behind in rows of up to eight wavefronts
    const bool fifth = t > 1024 && t <= 1216, fifth_long = t > 1024 && t <= 1280;
    int64_t until = 0;
    switch ((nvec + 63) / 64) {
    case 4: return two ? (t <= 2048 ? 4 : 1) : (many ? (t <= 1024 || (t >= 2304 && t < 6144) ? 4 : 1) : (t <= 2048 && !fifth_long ? 4 : 1));
    case 5: return t <= (two && !lines ? 640 : 1024) || (t > 1280 && t <= 1536) || (many && t >= 1728) ? 4 : 1;
    case 6: until = (lines || two ? fifth_long : fifth) ? 0 : 1536; break;
    case 7: until = !two && fifth ? 0 : (four ? 1408 : 1536); break;
    case 8:
        if (full && t >= 1792) until = many ? 6144 : (four ? 2049 : 0);
        else until = (many && fifth) || (four && fifth_long) ? 0 : 1536;
        break;
    case 9: until = two ? 1281 : (four ? 1025 : (lines ? 1536 : 768)); break;
    case 10: until = two ? (lines ? INT64_MAX : 2304) : 1536; break;
    case 11: until = lines || many ? 1536 : (two ? 1025 : 576); break;
    case 12: until = four ? 576 : (lines ? (full ? (two ? 2304 : 6144) : 1536) : (two ? 1025 : 448)); break;
    case 13:
    case 14: until = four && !lines && t >= 640 && t < 768 ? 0 : (many ? 6144 : 3072); break;
    case 15: until = many ? 6144 : 3072; break;
    default: until = many ? 6144 : (lines || nvec > 1016 ? 3072 : (two ? 1281 : 1152)); break;
    }
    return t < until ? 4 : 1;
}

// The same for the norm phase alone (tde_stage_norm, or the second of two launches), which reads two streams whatever the
// number of partials.  Four against one: up to 37 % faster below 1536 rows (ten to twelve wavefronts), 1-6 % slower beyond the
// ends below.
int vecs_per_thread_f64_norm(int64_t nvec, int64_t t) {
    if (nvec < 256 || t < 256) return 1;
    switch ((nvec + 63) / 64) {
    case 4: return t >= 1344 && t <= 3072 ? 4 : 1;
    case 5: return t >= 1344 && t < 1792 ? 4 : 1;
    case 6: return t <= 896 || (t > 1280 && t < 1536) ? 4 : 1;
    case 7:
    case 8:
    case 9:
    case 11:
    case 12: return t < 1536 ? 4 : 1;
    case 10: return rows_of_whole_lines(nvec) || t < 8192 ? 4 : 1;
    case 13:
    case 14: return 4;
    case 15: return t < 4096 ? 4 : 1;
    }
    return t < 1152 ? 4 : 1;
}

// TDE_ALGO_STAGED_OWNED in one launch, per-token scales: most rows read two buffers only, so a row of one vector per thread has
// little in flight for its many wavefronts.  Swept over 2/4/8 partials x rows of 240 to 832 vectors x 300 to 16000 rows
// against one vector per thread: two are 2-19 % faster with six wavefronts per row, 5-18 % with seven (two partials of a
// 2-byte type: nothing), 4-24 % with nine, 8-21 % with ten; with eleven and twelve four are 3-24 % faster with four and
// eight partials, two 4-17 % with two.
int vecs_per_thread_owned(const tde_problem *p, int64_t nvec, int64_t t, int vpt) {
    const bool few = p->nranks == 2;
    switch ((nvec + 63) / 64) {
    case 6: return t >= 1024 && (!few || nvec <= 352) ? 2 : vpt; // two partials, 371 vectors: +3 %
    case 7: return t >= 1024 && (!few || p->dtype == TDE_F32) ? 2 : vpt;
    case 9: return t >= (few ? 4096 : 2048) ? 2 : vpt;
    case 10: return t >= 640 ? 2 : vpt;
    case 11:
    case 12: return t >= (few ? 4096 : 2048) ? (few ? 2 : 4) : vpt;
    }
    return vpt;
}

// Two and four partials in one launch, rows of up to 768 vectors: a row has few loads per wavefront to cover its reduction, so
// fewer wavefronts with more vectors each can be faster.  From sweeps over rows of 64 to 768 vectors x 256 to 32768 rows in
// bf16, fp16 and fp32, every output mode, with and without T-typed rows beside the codes, against one vector per thread (some
// 8000 launches of other sizes, and rows in steps of 32 to 64 where a range ends).  A launch's time rises in steps, with
// every further workgroup on the fullest compute unit; the two geometries' steps lie apart, which is why a range can end at
// a multiple of 256 rows and why the gain inside one goes from a few percent to twenty.
int vecs_per_thread_few_partials(const tde_problem *p, int64_t nvec, int64_t t) {
    const int waves = (int)((nvec + 63) / 64); // of a row, with one vector per thread
    const bool two = p->nranks == 2, f32 = p->dtype == TDE_F32;
    if (p->quant == TDE_QUANT_NONE) {
        // T-typed output is bound by memory either way, and the gain ends with the first steps: two partials 576 to 1279 rows
        // of 656 and 768 vectors -4 to -20 %, 832 to 1536 rows of 400 and 512 -5 to -18 %, 1344 to 1536 of 260 to 384 -10 to -16 %,
        // of 200 to 256 up to -18 % (2048 and 3072 rows), but of 256 +3 to +5 % from 2049 to 2239 rows, all +3 % beyond 3072; four partials
        // 640 to 1023 rows of 400 and 512 -2 to -8 %, 1472 to 1536 and 1900 to 2048 of 200 to 256 -3 to -12 %, with +2 to +4 % from
        // 1600 to 1800 rows and +5 to +14 % beyond 2048.
        if (two && waves >= 11) return t >= 576 && t < 1280 ? 4 : 1;
        if (waves == 7 || waves == 8) return two ? (t >= 832 && t <= 1536 ? 4 : 1) : (t >= 640 && t < 1024 ? 4 : 1);
        if (two && (waves == 5 || waves == 6)) return t >= 1344 && t <= 1536 ? 4 : 1;
        if (waves == 4)
            return two ? (t >= 1536 && t <= 3072 && !(nvec > 240 && t > 2048 && t < 2240) ? 4 : 1)
                       : ((t >= 1472 && t <= 1536) || (t >= 1900 && t <= 2048) ? 4 : 1);
        return 1;
    }
    const bool per_token = p->quant == TDE_QUANT_FP8_TOKEN || p->quant == TDE_QUANT_INT8_TOKEN;
    if (!two) return f32 && per_token && waves == 9 && t >= 1536 ? 2 : 1; // 3-5 %
    // With T-typed rows beside the codes a row moves more, and what several vectors gain without them ends sooner or is left
    // to rows of whole lines; the rules say where two vectors were still no slower than one.
    const bool t_rows = p->write_norm != 0, lines = rows_of_whole_lines(nvec);
    if (!per_token) {
        // Just beyond two rows per unit the wide workgroups of rows of eleven and twelve wavefronts no longer fit at once (two to a
        // unit), and with T-typed rows beside the codes more vectors pay at once.  Time against one vector per thread, two | four,
        // rows of 650, 704 and 768 vectors:
        //   static, 2-byte    544 rows -2 to -6 % | +1 to -8 %, 704 -13 % | -11 %, 767 -14 to -18 % | -12 to -17 %, 896 +3 % | -10 %,
        //                     1024 -1 to -7 % | -13 to -18 %, 1154 +4 % | +4 %, 1257 and 1280 rows of whole lines -1 to -5 % | -5 to -7 %,
        //                     others +2 % | +1 %
        //   static, fp32      544 to 704 rows -5 to +8 % | -5 to -14 %, 767 -3 to -8 % | -15 to -22 %, 1024 -3 % | -3 to -12 %, 1154 +4 % | +4 %,
        //                     1257 and 1280 -1 to -3 % | -1 to -5 %
        //   group, fp32       544 to 704 rows +7 to -14 % | -7 to -16 %, 767 -7 to -20 % | -20 %, 1024 -4 % | -12 %, 1154 +2 % | +3 %, 1280 -4 % | -7 %
        //   group, 2-byte     544 to 704 rows 0 to -15 % | -2 to -11 %, 767 -14 % | -14 %, 1024 -6 % | -11 %, 1280 -4 % | -5 %
        if (waves >= 11 && t_rows && t >= 544 && t < 1280) {
            if ((f32 || p->quant == TDE_QUANT_FP8_STATIC) && (lines || t < 1025)) return 4;
            if (t < 768) return 2;
        }
        // Long launches 1-14 % faster with two (with T-typed rows fp32 1-5 %, a 2-byte type at best nothing).  Rows of eleven and
        // twelve wavefronts: 768 rows 10-15 % faster with two (fp32 up to 9 %), 1024 3-5 %, 1280 2-5 %, around 900 and 1100 rows up to 2 %
        // slower, 1344 to 1400 -1 to +2 %, fp32 0 to -4 %.
        if (waves >= 11 && t >= 768 && t < (f32 || !t_rows ? 1400 : (lines ? 1281 : 1025))) return 2;
        if (t < 4096 || !(waves == 9 || waves >= 11)) return 1;
        return !t_rows || (f32 && (waves < 12 || lines)) || (waves == 11 && lines) ? 2 : 1;
    }
    if (waves >= 11) { // two 2-18 % faster, 544 to 767 rows up to 22 %; 768 vectors of a 2-byte type 1-2 % slower around 2000 rows
        // fp32 beside T-typed rows: with twelve wavefronts two are up to 6 % slower than one from 590 to 700 rows (768 vectors, 640
        // rows: 9.06 us with one, 9.54 with two, 8.19 with four), four 7-21 % faster over the whole band; with eleven two lose nowhere
        // (704 vectors, 640 rows -7 %).  From 768 rows on two are 17 % faster to 4 % slower than one.
        if (t_rows && f32 && waves >= 12 && t >= 544 && t < 768) return 4;
        if (t_rows && !f32 && (waves >= 12 ? t >= 1408 : !lines && t >= 1537)) return 1;
        return t >= 544 && (f32 || waves == 11 || t < 1536 || t >= 2304) ? 2 : 1;
    }
    if (waves == 9) { // 1-20 %; 2-byte types 1-6 % behind from 1344 to 1536 rows
        if (t_rows && !f32 && !lines && t >= 1344) return 1;
        return t >= 1024 && (f32 || t < 1344 || t > 1536) ? 2 : 1;
    }
    if (waves == 6) return t >= 1536 && (!t_rows || t < 3072) ? 2 : 1; // 1-14 %
    if (waves == 7) { // 1-14 %
        const int64_t until = !t_rows || (f32 && lines) ? INT64_MAX : (f32 || lines ? 8192 : 1792);
        return t >= 1536 && t < until ? 2 : 1;
    }
    if (waves == 5) // fp32 3-13 %, others 0-10 %
        return f32 ? (t >= 1536 && (!t_rows || t < (lines ? 16384 : 6144)) ? 2 : 1) : (t >= 16384 && !t_rows ? 2 : 1);
    return 1;
}

// Fused rows of 13 and 14 wavefronts: where several vectors per thread are no slower than one.  Per-token codes gain from 256 rows
// on (1-5 %, from 800 rows 8-20 %).  Several against one elsewhere: eight partials of a 2-byte type with static or group
// scales up to 768 rows +1 to +4 % (rows of whole lines up to 640), with T-typed output and other rows 0 to +3 %; four partials with
// static or group scales 449 to 768 rows +1 to +2 %, with T-typed rows as well +2 to +5 % (and from 3072 rows of a 2-byte type that are
// not whole lines +2 to +5 %); four partials 641 to 768 rows of T-typed output, or of fp32 per-token codes beside T-typed rows, +2 to +5 %;
// fp32 with static or group scales, rows of whole lines up to 384, +1 to +2 %; up to four partials, exactly one row per compute
// unit, T-typed output (four partials of a 2-byte type: static and group scales too) +2 to +6 %.
bool several_vecs_pay(const tde_problem *p, int64_t nvec, int64_t t) {
    if (t < 256) return true;
    const bool f32 = p->dtype == TDE_F32, four = p->nranks == 4, many = p->nranks >= 8, lines = rows_of_whole_lines(nvec);
    const bool none = p->quant == TDE_QUANT_NONE, fixed = p->quant == TDE_QUANT_FP8_GROUP || p->quant == TDE_QUANT_FP8_STATIC;
    if (t == 256 && ((p->nranks <= 4 && none) || (four && fixed && !f32))) return false;
    if (fixed && p->nranks >= 4) {
        if (f32 && lines && !p->write_norm && t < 384) return false;
        if (many) return f32 || t > (lines ? 640 : 768);
        if (!p->write_norm) return f32 || !(t > 448 && t <= 768);
        return f32 ? !(t > 576 && t <= 768) : !(t > 448 && t <= 800) && (lines || t < 3072);
    }
    if (none && many) return f32 || lines || t > 768;
    if (four && (none || (f32 && p->write_norm))) return !(t > (lines ? 680 : 640) && t <= 768);
    return true;
}

int vecs_per_thread(const tde_problem *p, int64_t nvec, int64_t t, bool norm_alone) {
    // Vectors per thread, from sweeps on MI355X over hidden 1024..8192 in steps of 1024, 2/4/8 partials, 128..32768 rows
    // and three output modes (bf16 and fp16 agree); only differences that held on two devices and across the row
    // counts between the swept powers of two are in here.  Four vectors per thread (small workgroups, many loads in
    // flight per thread, few wavefronts to synchronize per row, partials summed while the later ones are still
    // arriving) win on long rows and wherever eight partials meet full wavefronts, two in the longest launches of
    // mid-length rows; elsewhere one vector per thread is as fast or faster.
    const bool staged = p->algo == TDE_ALGO_STAGED;
    int vpt = 1;
    if (nvec > 768) {
        // Few rows are latency-bound and the widest row groups have the shortest dependent chain; from 256 rows
        // up four vectors per thread are 4-13 % faster than one (8 partials, hidden 8192).  With two partials
        // and up to 2048 rows two vectors per thread are another 2-7 % faster.
        vpt = t >= 256 ? 4 : (t >= 128 ? 2 : 1);
        if (p->nranks == 2 && t >= 256 && t <= 2048) vpt = 2;
        // Rows of 13 and 14 wavefronts, 769 to 888 vectors against one per thread: quantized output up to -27 % with two
        // partials, -22 % with four, -15 % with eight, T-typed output -1 to -13 %; but +2 to +6 % in long launches of two
        // and four partials that move more per row (T-typed rows, the stage), and around 1300 staged rows of two partials.
        if (nvec < 896 && p->nranks <= 4) {
            const bool t_typed = p->quant == TDE_QUANT_NONE;
            const int64_t until = t_typed ? (p->dtype == TDE_F32 ? 6144 : 2048 * p->nranks / 2)
                                          : (staged || (p->nranks == 4 && p->quant == TDE_QUANT_FP8_STATIC) ? 12288 : INT64_MAX);
            if (t > until || (staged && p->nranks == 2 && t >= 1024 && t < 1792)) vpt = 1;
        }
        if (nvec < 896 && p->algo <= TDE_ALGO_FUSED && !several_vecs_pay(p, nvec, t)) vpt = 1;
    } else if (nvec == 512 && p->nranks >= 8 && t >= 1024) {
        vpt = t >= 16384 ? 2 : 4; // four: 3-4 % over one; from 16384 rows two are another 4-7 % ahead
    } else if (nvec == 256 && p->nranks >= 8 && t >= 2048) {
        // four: 3-6 % over one (with fewer partials or rows one is 3-16 % faster); from 32768 rows two: another 4-6 %
        vpt = t >= 32768 ? 2 : 4;
    } else if (nvec == 256 && p->nranks == 4 && t >= 32768) {
        vpt = 2; // 3-4 % over one
    } else if (nvec == 768 && p->nranks >= 8 && t >= 2048) {
        // rows of 6144 2-byte elements: twelve wavefronts with one vector each lose to three with four vectors
        // (2048 to 5600 rows: 1.5-2.3 %) and, in long launches, to six with two (3-6 % from 8192 rows)
        if (t >= 8192) vpt = 2;
        else if (t < 5632) vpt = 4;
    } else if (nvec == 768 && p->nranks == 4 && t >= 1024 && t < 2048) {
        vpt = 4; // 1-5 %
    } else if (nvec == 384 && p->nranks >= 8 && t >= 8192 && p->quant != TDE_QUANT_NONE) {
        vpt = t >= 32768 ? 2 : 4; // 4-5 % over one with quantized output; with T-typed output one is 2 % ahead
    } else if (nvec == 128 && p->nranks >= 8 && t >= 4096 && t < 8192) {
        vpt = 2; // 1-3 % over one
    } else if (nvec > 576 && nvec <= 640) {
        // Ten wavefronts per row leave the compute units unevenly filled: from 640 rows up five wavefronts with two
        // vectors each are 5-30 % faster until there are enough rows to even that out (2048 with eight partials,
        // 16384 with four; rows of 640 vectors of two partials 1-4 % at any length).  With four partials
        // and 16384+ rows all three choices are within 1 %; four vectors per thread is the one whose launches take the
        // same time from the first on (with one, launches 5 to 50 of a cold run took up to 30 % longer).  Rows that do not
        // fill two vectors per thread stop gaining sooner: eight partials at 1152 rows (+3 % at 1300); where a row moves more (the stage,
        // T-typed output of four partials) at 1152 to 6144.
        const bool full = nvec == 640, f32 = p->dtype == TDE_F32;
        const bool heavy = !full && (staged || (p->nranks == 4 && p->quant == TDE_QUANT_NONE));
        const int64_t even_from = p->nranks >= 8 ? (full ? 2048 : 1152) : (p->nranks == 4 ? 16384 : INT64_MAX);
        if (heavy) vpt = t >= 640 && t < (p->nranks == 2 ? 6144 : (p->nranks == 4 ? 1792 : 1152)) ? 2 : 1;
        else if (t >= (full || p->nranks < 8 ? 640 : 768) && t < even_from) vpt = 2;
        else if (p->nranks == 4 && t >= even_from) vpt = nvec == 640 ? 4 : 2;
        else if (p->nranks >= 8 && t >= 16384 && nvec == 640) vpt = 2; // eight partials, long launches: 2 % over one
        if (!full && p->algo <= TDE_ALGO_FUSED) {
            // One vector against two: eight partials 776 to 831 rows -1 to -5 % (768 rows +8 to +12 %; fp32 T-typed output +1 to
            // +6 %).  Rows that are not whole lines: four partials from 4096 rows on -1 to -4 %, until the limit on workgroups per
            // compute unit (below) makes two 1-5 % faster again, and with T-typed rows beside the codes from 1281 (static and group
            // scales) or 1792 rows on -1 to -7 % (fp32 per-token codes as without them); two partials, T-typed output from 8192 rows
            // on -1 to -6 % (fp32 from 12288), T-typed rows beside static and group scales of a 2-byte type from 2304, beside
            // per-token codes from 6144.
            const bool fixed = p->quant == TDE_QUANT_FP8_GROUP || p->quant == TDE_QUANT_FP8_STATIC, none = p->quant == TDE_QUANT_NONE;
            const bool beside = !none && p->write_norm != 0, lines = rows_of_whole_lines(nvec);
            if (p->nranks >= 8 && !(f32 && none) && t >= 776 && t < 832) vpt = 1;
            if (p->nranks == 4 && !lines && !none) {
                if (beside && (fixed || !f32) && t >= (fixed && !f32 ? 1281 : 1792)) vpt = 1;
                if ((beside || !f32) && t >= 4096 && t < kLimitFromWorkgroupsPerCu4 * 256) vpt = 1;
            }
            if (p->nranks == 2 && !lines && (none || (beside && !f32)) &&
                t >= (none ? (f32 ? 12288 : 8192) : (fixed ? 2304 : 6144)))
                vpt = 1;
        }
    }
    const bool per_token = p->quant == TDE_QUANT_FP8_TOKEN || p->quant == TDE_QUANT_INT8_TOKEN;
    const bool owned = p->algo == TDE_ALGO_STAGED_OWNED, fused = !staged && !owned;
    // TDE_ALGO_STAGED, up to four partials, T-typed rows or static and group scales: one vector per thread stays 2-6 % ahead of the
    // ranges above between the lengths they were first swept at.
    if (staged && !per_token && p->nranks <= 4 && nvec > 576 && nvec < 896 && nvec != 640) vpt = nvec == 768 ? vpt : 1;
    // Of fp16, whose arithmetic is shorter, two are 0.6 to 2.7 % ahead in long launches of four partials (5632 to 7080 elements, 9000 to 24000 rows).
    if (staged && p->dtype == TDE_F16 && p->quant == TDE_QUANT_NONE && p->nranks == 4 && nvec > 640 && nvec < 896 && t >= 8192) vpt = 2;
    // The norm phase alone keeps one vector per thread where it stores T-typed rows beside the codes and the rows are not whole
    // lines: several are 2-7 % slower there with six and seven wavefronts per row from 4096 rows on, 2-10 % with eleven and twelve.
    const int waves = (int)((nvec + 63) / 64);
    const bool alone_loses = norm_alone && p->write_norm != 0 && !rows_of_whole_lines(nvec) &&
                             (waves == 11 || waves == 12 || ((waves == 6 || waves == 7) && t >= 4096));
    if (owned && per_token && !alone_loses) vpt = vecs_per_thread_owned(p, nvec, t, vpt);
    else if (fused && vpt == 1 && p->nranks <= 4) vpt = vecs_per_thread_few_partials(p, nvec, t);
    return vpt;
}

// Megabytes that a launch moves in T-typed rows, roughly: what the rules for short and for shifted rows go by.
int64_t row_megabytes(const tde_problem *p, int64_t nvec) {
    const int64_t streams = p->algo == TDE_ALGO_STAGED_OWNED ? 4 : p->nranks + 2; // an owned launch reads two streams for most rows
    return (streams * p->tokens * nvec) >> 16;
}

// Rows that share a wavefront (tde_short_rows.hip) against one wavefront each (row_kernel), 1400 launches of 1 to 60000 rows: up to 16
// vectors 4-15 % faster below 4096 rows, 30 % from there and 35-55 % from 16384 rows on (2 x [30046, 152] bf16 -> fp8 15.2 -> 9.3 us); 17
// to 32 vectors 3-8 % faster below 8192 rows and there, where memory begins to bind, 20 % faster to 3 % slower with two and four
// partials (2 x [40459, 192] 18.2 -> 13.5, 4 x [28759, 192] 14.5 -> 14.8).  Eight partials keep memory busy either way: from 8192
// rows of more than 20 vectors on one row to a wavefront is up to 5 % faster (up to 20 vectors 2-8 % slower).  Owned rows, and the norm
// phase alone, read two buffers for most rows and gain more (8 x [45945, 144] 23.4 -> 17.2), but for two kinds of owned launches (2600
// launches): up to four partials, few rows of a 2-byte type and more than 16 vectors, where the wait for the
// partials behind the stage's is all that counts (below 256 rows 1 % slower, single ones 6 %; fp32 4 % faster), and two partials with
// T-typed rows to store, more than 24 vectors long (from 30 MB on 1 to 14 % slower, T-typed output of fp32 from 72 MB; beside per-token
// codes of a 2-byte type level): one row to a wavefront against two, 4 x [1, 240] bf16 -> fp8 2.42 us and 2.53, 2 x [50271, 248] fp16
// 25.5 and 28.7, 2 x [59915, 124] fp32 -> static fp8 and rows 33.0 and 38.3.
bool share_a_wavefront(const tde_problem *p, int64_t nvec, int64_t t, bool norm_alone) {
    if (p->dtype == TDE_F64 || nvec > tde::kShortRowVecs) return false;
    if (p->algo == TDE_ALGO_STAGED_OWNED && !norm_alone && p->nranks <= 4) {
        const bool f32 = p->dtype == TDE_F32, none = p->quant == TDE_QUANT_NONE;
        if (!f32 && nvec > 16 && t < 256) return false;
        const bool rows_out = none || (p->write_norm != 0 && (f32 || p->quant == TDE_QUANT_FP8_STATIC));
        if (p->nranks == 2 && nvec > 24 && rows_out && row_megabytes(p, nvec) >= (f32 && none ? 72 : 30)) return false;
    }
    return nvec <= 20 || p->nranks < 8 || t < 8192 || p->algo == TDE_ALGO_STAGED_OWNED || norm_alone;
}

// Vectors of a line of the narrowest buffer that counts.
int line_vectors(const tde_problem *p) { return p->quant == TDE_QUANT_NONE ? 8 : (p->dtype == TDE_F32 ? 32 : 16); }

// Whether rows that start inside a line are moved along their threads (tde_rows.h: SHIFTED).  A launch pays 0.07 us for it (the row
// is known before its addresses are) and, with 2-byte types, another barrier ahead of the sums; what it gains is 2-8 % of its
// time in memory.  From 3000 launches of 5 to 2200 MB in place and shifted, the same vectors per thread: 10 MB +1.5 %, 20 MB
// 0 to +0.5 %, 40 MB -1.5 % (single ones up to +3.5 % with two and four partials of one vector per thread), 100 MB -2.2 %,
// from 300 MB on -3.3 % (2 x [31779, 3256] bf16 -> static fp8 and T-typed rows 198.4 -> 183.3 us, 4 x [26096, 962] doubles staged
// 285 -> 255, 2 x [30413, 4008] fp32 -> int8 375 -> 323).  Two and four partials of a 2-byte type, four vectors per thread and one wavefront to
// a row: +0.4 to +1.6 % from 28 to 45 MB (2 x [2999, 1776] fp16 10.1 us against 9.9).  Two wavefronts a row: 0 to -0.5 %, 2-byte types nothing.  Eight partials of a 2-byte type, one
// vector per thread: owned rows +0.2 %, up to four wavefronts a row with workgroups limited per unit +0.3 %.
// Rows of whole T-typed lines whose codes start inside lines: two partials -1 to -3 %, others nothing.
bool rows_are_shifted(const tde_problem *p, int64_t nvec, int64_t t, int vpt) {
    const bool owned = p->algo == TDE_ALGO_STAGED_OWNED, staged = p->algo == TDE_ALGO_STAGED, few = p->nranks <= 4;
    const int line = p->nranks == 2 && !staged && !owned ? line_vectors(p) : 8;
    if (nvec % line == 0 || nvec <= tde::kWave) return false;
    const int64_t mb = row_megabytes(p, nvec);
    if (elem_bytes(p->dtype) > 2) return mb >= (nvec <= 128 ? 56 : 32);
    if (nvec <= 128) return false;
    if (!few && vpt == 1 && (owned || (nvec <= 256 && t >= kLimitFromWorkgroupsPerCu8 * 256))) return false;
    return mb >= (owned || (few && (vpt == 1 || (vpt == 4 && nvec <= 256))) ? 56 : 28);
}

// Vectors per thread where rows are shifted and the lengths that vecs_per_thread was swept at do not speak for them (same launches; against
// its choice).
int vecs_per_thread_shifted(const tde_problem *p, int64_t nvec, int64_t t, int vpt) {
    const int waves = (int)((nvec + 63) / 64);
    const bool none = p->quant == TDE_QUANT_NONE;
    if (p->dtype == TDE_F64 || p->algo == TDE_ALGO_STAGED) return vpt;
    if (p->algo == TDE_ALGO_STAGED_OWNED) {
        // Eight partials, rows of five to ten wavefronts: two vectors 2-20 % ahead of one where codes alone are stored (720 launches).  With
        // T-typed rows to store nine and ten wavefronts keep that (1 to 5 %; T-typed output of fp32 rows of nine +-1 %), eight lose 0.5 to 4 %
        // at any length, five to seven from 18 rows per unit on 0.5 to 5 % (T-typed output; of fp32 also beside codes: of
        // 2-byte rows beside codes two stay 0.5 to 6 % ahead): 8 x [17457, 1476] fp32 90.7 us with two, 86.3 with one, [14836, 2144] bf16 54.0 and 53.2, [2123, 4040] fp16 -> int8 and rows 20.8 and 20.0.
        const bool rows_out = none || p->write_norm != 0;
        const bool one = rows_out && (waves == 8 || (waves < 8 && t >= 18 * 256 && (none || p->dtype == TDE_F32)));
        return p->nranks >= 8 && vpt == 1 && waves >= 5 && waves <= 10 && t >= 1200 && !one ? 2 : vpt;
    }
    if (p->nranks == 2) {
        if (!none && waves >= 13 && t >= 2560) return 2; // 2 % over four
        if (none && waves >= 15 && t >= 8192) return 1; // 2-3 % over four
    } else if (p->nranks == 4) {
        if (waves == 15 && vpt == 4 && t <= 2048) return 2; // 2 %
    } else if (vpt == 1) {
        if (waves == 9 || (waves == 6 && !none)) return t >= 8192 ? 2 : 1; // 2-5 %
        if (nvec >= 600) return t >= 2048 ? 4 : 1;                          // 1-3 %; shorter rows leave four's lanes too empty
    }
    return vpt;
}

// `norm_alone`: the geometry of a launch that only norms the rows of the stage.
int validate(const tde_problem *p, tde::Geometry *geo, bool norm_alone = false) {
    if (p == nullptr) return TDE_EINVAL;
    const int eb = elem_bytes(p->dtype);
    if (eb == 0) return TDE_EDTYPE;
    if (!(p->nranks == 2 || p->nranks == 4 || p->nranks == 8)) return TDE_ENRANKS;
    if (p->rank < 0 || p->rank >= p->nranks) return TDE_ERANK;
    if (p->tokens < 0 || p->hidden <= 0) return TDE_ESHAPE;
    if (p->hidden > kMaxBlock * 16) return TDE_EHIDDEN; // also keeps hidden * eb far from overflow
    if ((p->hidden * eb) % 16 != 0) return TDE_ESHAPE;
    if (p->quant < TDE_QUANT_NONE || p->quant > TDE_QUANT_FP8_STATIC) return TDE_EQUANT;
    if (p->quant == TDE_QUANT_FP8_STATIC && !(p->static_scale > 0.0f && p->static_scale <= 3.0e38f)) return TDE_EQUANT;
    if (p->quant == TDE_QUANT_FP8_GROUP && p->hidden % TDE_QUANT_GROUP != 0) return TDE_EQUANT;
    if (p->algo < TDE_ALGO_AUTO || p->algo > TDE_ALGO_STAGED_OWNED) return TDE_EALGO;
    if (p->dtype == TDE_F64 && p->quant != TDE_QUANT_NONE) return TDE_EQUANT; // doubles: no quantized output
    const int vec = 16 / eb;
    const int64_t nvec = p->hidden / vec;
    if (nvec > kMaxBlock) return TDE_EHIDDEN; // as the reference: one 16-byte vector per thread, 1024 threads
    int64_t total_bytes = 0; // tokens * hidden * elem must be addressable with 64-bit signed offsets
    if (__builtin_mul_overflow(p->tokens, p->hidden * eb, &total_bytes)) return TDE_ESHAPE;

    const int cus = compute_units(); // once a call: asking the runtime for the device takes it 50 ns
    const int64_t t = rows_as_on_256_units(p->tokens, cus);
    int vpt = p->dtype != TDE_F64 ? vecs_per_thread(p, nvec, t, norm_alone) : (norm_alone ? vecs_per_thread_f64_norm(nvec, t) : vecs_per_thread_f64(p, nvec, t));
    if (!norm_alone && rows_are_shifted(p, nvec, t, 4)) vpt = vecs_per_thread_shifted(p, nvec, t, vpt);
    if (p->tune_vecs_per_thread != 0) {
        if (p->tune_vecs_per_thread != 1 && p->tune_vecs_per_thread != 2 && p->tune_vecs_per_thread != 4) return TDE_EINVAL;
        vpt = p->tune_vecs_per_thread;
    }
    if (p->tune_rows_per_block < 0) return TDE_EINVAL;
    if (p->tune_workgroups_per_cu < -1 || p->tune_workgroups_per_cu > 8 || p->reserved != 0) return TDE_EINVAL;
    const bool short_rows = p->tune_vecs_per_thread == 0 && p->tune_rows_per_block == 0 && share_a_wavefront(p, nvec, t, norm_alone);
    const int64_t lanes = (nvec + vpt - 1) / vpt;
    const int tpr = short_rows ? (nvec <= 16 ? 16 : 32) : (int)((lanes + 63) / 64 * 64);
    // pack short rows so a workgroup has at least four wavefronts (two of two rows each: 1 % faster than four)
    int rpb = (tpr == 32 ? 128 : 256) / tpr;
    if (rpb * tpr > kMaxBlock / vpt) rpb = (kMaxBlock / vpt) / tpr; // never beyond the kernel's launch bound
    const int least = std::max(1, tde::kWave / tpr); // whole wavefronts
    while (rpb > least && (p->tokens + rpb - 1) / rpb < 2 * cus) rpb /= 2; // keep every CU busy first
    if (rpb < least) rpb = least;
    if (p->tune_rows_per_block > 0 && p->tune_rows_per_block * tpr <= kMaxBlock / vpt) rpb = p->tune_rows_per_block;
    if (p->tokens > 0 && rpb > p->tokens && !short_rows) rpb = (int)p->tokens;
    const int64_t grid = (p->tokens + rpb - 1) / rpb; // one workgroup per group of rows, no loop
    if (grid > 0x7fffffff) return TDE_ESHAPE;

    // Resident workgroups per compute unit.  Left alone, a CU takes as many workgroups as its registers and LDS hold
    // (3-6 here), each with all of its rows' loads in flight.  On MI355X long launches run fastest with 120-160 KiB
    // of loads in flight per CU: more costs 1-8 % from 8192 rows up with 4 or 8 partials (32768 x 8192: 7.5 % with
    // 4 partials, 4.5 % with 8; 16384 rows: 1-3 %; 8192 rows with 8 partials: 1 %), fewer than two workgroups, or than
    // eight wavefronts that have T-typed rows to store, leave the arithmetic of one row uncovered by the loads of another.
    // Short launches (a few generations of workgroups) gain nothing and can lose 1-3 %, and with 2 partials no limit helps.
    // Eight wavefronts are enough for per-group scales on four partials too (two workgroups against three): 4 x [8192, 7168]
    // bf16 119.3 us against 123.2, 4 x [12000, 8192] 198.4 against 205.9, 4 x [32768, 7168] fp16 467 against 503, fp32
    // 4 x [9000, 3584] 124.9 against 127.0.
    const bool staged = p->algo == TDE_ALGO_STAGED || p->algo == TDE_ALGO_STAGED_OWNED;
    int wgs_per_cu = 0;
    const int64_t per_wg = (int64_t)rpb * (p->nranks + 1) * nvec * 16; // bytes of loads one workgroup keeps in flight
    // Only codes of a dynamic scale beside residual_out to store, four vectors per thread and 96 KiB of loads in two workgroups.
    const bool few_stores = vpt == 4 && p->quant != TDE_QUANT_NONE && p->quant != TDE_QUANT_FP8_STATIC && p->write_norm == 0 && 2 * per_wg >= 96 * 1024;
    const bool many_workgroups = grid >= (p->nranks >= 8 ? kLimitFromWorkgroupsPerCu8 : kLimitFromWorkgroupsPerCu4) * cus ||
                                 (few_stores && grid >= kFewStoresFrom * cus && grid < kFewStoresUntil * cus);
    if (p->dtype != TDE_F64 && !staged && p->nranks >= 4 && many_workgroups) {
        const int waves = tpr * rpb / 64;
        const int at_least = std::max(2, (8 + waves - 1) / waves);
        // Eight partials, rows of three wavefronts with one vector per thread, and of four with T-typed output: 96 KiB from 48 workgroups
        // per unit on, 2 to 2.8 % ahead with T-typed output, 1.3 % with codes (of four wavefronts 1 % ahead to 1.6 % behind, shorter
        // launches 2 % ahead to 1 % behind).
        const bool short_many = p->nranks >= 8 && vpt == 1 && nvec > 128 && nvec <= (p->quant == TDE_QUANT_NONE ? 256 : 192) && grid >= 48 * (int64_t)cus;
        const int64_t in_flight = short_many ? 96 * 1024 : kLoadsInFlightPerCu;
        wgs_per_cu = (int)std::min<int64_t>(8, std::max<int64_t>(at_least, (in_flight + per_wg / 2) / per_wg));
        // Two workgroups are enough for few_stores, six wavefronts among them: 4 x [32768, 5120] fp16 -> int8 338.2 us against
        // 342.3 with three, bf16 -> fp8 336.2 against 344.7, per group 338.7 against 339.7; with T-typed output or rows three
        // stay 3 % ahead.  For them the limit pays from 16 workgroups per unit on: 4 x rows of 770 to 1024 vectors, 4096 to 6143 of them -1.3 % (bf16),
        // -2.3 (fp16) and 0 (fp32), 6144 to 7679 -2.5 to -2.9, per group -2 (below 4096 +0.5; static scales +0.5, T-typed output -0.5).  Eight partials
        // then leave the kernel for two wavefronts per SIMD (`wide`, below) for two workgroups of this one: 120 launches of 4096 to 6143 rows of
        // 769 to 1024 vectors -0.5 % on average, single ones -2.2 to +0.6 %.
        if (few_stores) wgs_per_cu = 2;
    }
    // TDE_ALGO_STAGED in one launch reads what the fused launch reads and stores one stream more.  From 16 workgroups per CU
    // on four and eight partials gain from the same 128 KiB, counted with the stage's stores, but never more than four workgroups
    // (56 launches of 4096 to 40188 rows: 2.0 % faster on average, none more than 0.4 % slower; without a limit against with): 8 x [32005, 2512] bf16 -> fp8 322.8 -> 304.2
    // us (three), 8 x [32012, 1032] fp16 137.1 -> 126.0 (four), 8 x [4096, 3000] 51.8 -> 50.0 (two), 8 x [12091, 8192] 396 -> 381 (two),
    // 4 x [30550, 748] fp32 114.5 -> 106.9 (four), 4 x [16384, 8192] 318.1 -> 313.4 (two).  Rows packed more than two to a workgroup
    // lose up to 2 %, two partials with one vector per thread up to 19 % with two and gain nothing with four.  Four workgroups of short
    // rows hold too little: below 68 KiB of loads and stores in four (four partials, rows of up to 180 vectors) six take 0.96 of the
    // time of four with quantized output, single ones 0.86 (70 launches; 4 x [26425, 1144] fp16 -> int8 84.8 -> 74.0 us, 4 x [27056, 316] fp32
    // 46.8 -> 41.6), and more nothing on top; T-typed output alone is 1 % slower with six.
    // Two partials of fp16 with two vectors per thread, whose arithmetic is short: three workgroups 1.5 to 2 % ahead of no limit
    // (2 x [7341 to 24000, 5120], [16000, 4960]; 23 more of 592, 608, 624 and 640 vectors 0.5 to 3 %).  With four vectors per thread and
    // codes to store no limit is up to 3 % behind what the same launch took with conversions in place of mixed instructions, two workgroups 0 to
    // 4 % ahead of it, from 24 per unit on (120 launches; 2 x [22974, 8128] -> static fp8 340.9 -> 327.6 us, [8607, 6976] -> int8 and rows 133.2 ->
    // 126.7); T-typed output loses 1 to 2 % with two.
    // With owned rows, and in the norm phase alone, most rows read two streams, and a limit only costs (25 launches of four and
    // eight partials: up to 50 %).
    if (p->dtype != TDE_F64 && p->algo == TDE_ALGO_STAGED && !norm_alone && p->nranks >= 4 && rpb <= 2 && grid >= 16 * (int64_t)cus) {
        const int64_t moved = (int64_t)rpb * (p->nranks + 2) * nvec * 16;
        const int64_t most = p->quant != TDE_QUANT_NONE && 4 * moved < 68 * 1024 && row_megabytes(p, nvec) >= 56 ? 6 : 4;
        wgs_per_cu = (int)std::min<int64_t>(most, std::max<int64_t>(2, (kLoadsInFlightPerCu + moved / 2) / moved));
    }
    if (p->dtype == TDE_F16 && p->algo == TDE_ALGO_STAGED && !norm_alone && p->nranks == 2 && vpt == 2 && nvec > 576 && nvec <= 640 && grid >= 24 * (int64_t)cus)
        wgs_per_cu = 3;
    if (p->dtype == TDE_F16 && p->algo == TDE_ALGO_STAGED && !norm_alone && p->nranks == 2 && vpt == 4 && p->quant != TDE_QUANT_NONE && grid >= 24 * (int64_t)cus)
        wgs_per_cu = 2;
    if (p->tune_workgroups_per_cu != 0 && p->dtype != TDE_F64) wgs_per_cu = p->tune_workgroups_per_cu < 0 ? 0 : p->tune_workgroups_per_cu;

    // Eight partials, four vectors per thread, no limit asked for or planned, and 4 to 24 workgroups per CU (few_stores: 4 to 16): the
    // row kernel's two-wavefronts-per-SIMD instantiation (tde_rows.h: WIDE) is 0.2-2.2 % faster there; it is
    // reported as the limit of two workgroups per CU that its registers amount to.
    const bool wide = p->nranks == 8 && vpt == 4 && p->dtype != TDE_F64 && !staged && wgs_per_cu == 0 &&
                p->tune_workgroups_per_cu == 0 && grid >= 4 * (int64_t)cus;

    if (geo) {
        geo->wgs_per_cu = wgs_per_cu;
        size_t lds = short_rows ? tde::short_rows_lds_bytes(tpr * rpb, rpb, vec) : tde::sumsq_lds_bytes(tpr * rpb, vpt, vec);
        if (wgs_per_cu > 0) {
            lds = std::max(lds, tde::lds_bytes_for_workgroups_per_cu(wgs_per_cu)); // never with doubles
            // what the launch enforces: a geometry whose own LDS is larger than the padding admits fewer still
            // (64: the kernels' static LDS)
            geo->wgs_per_cu = (int)std::min<size_t>((size_t)wgs_per_cu, tde::kLdsPerCu / (lds + 64));
        }
        geo->lds_bytes = (int)lds;
        geo->vec_elems = vec;
        geo->nvec = (int)nvec;
        geo->vpt = vpt;
        geo->threads_per_row = tpr;
        geo->rows_per_block = rpb;
        geo->block_threads = tpr * rpb;
        geo->grid = grid;
        geo->line_mask = !short_rows && !norm_alone && rows_are_shifted(p, nvec, t, vpt) ? line_vectors(p) - 1 : 0;
        // Row groups per XCD chunk of the row mapping (tde_rows.h: xcd_chunked_block); 16 measured best with 8
        // partials, 8 with 4.
        geo->xcd_chunk = p->nranks >= 8 ? 16 : 8;
        geo->form = wide ? tde::kFormWide : tde::kFormPlain;
        geo->converted = false;
        if (p->dtype == TDE_F16 && p->nranks == 4 && vpt == 4) {
            // Long fp16 launches with longer arithmetic (tde_converted_rows_f16.hip, tde_rows.h: kFormLong).  Mixed instructions against
            // conversions, rows of 768 to 1024 vectors (250 launches): T-typed output from 32 workgroups per unit on (where its own limit
            // begins) 0.3 to 2 % behind, below it level; static scales and rows beside codes from 48 on 0.3 to 1.7 % behind, below it 0.3 %
            // ahead to level; dynamic codes alone, more than 832 vectors, 0.4 to 0.8 % behind; T-typed output beside a
            // stage from 16 on (where that limit begins) 1 to 2 % behind.
            const bool none = p->quant == TDE_QUANT_NONE, per_token = p->quant == TDE_QUANT_FP8_TOKEN || p->quant == TDE_QUANT_INT8_TOKEN;
            const int from = staged ? 16 : (none ? 32 : 48);
            if (grid >= from * (int64_t)cus && (!staged || (p->algo == TDE_ALGO_STAGED && none && !norm_alone))) {
                geo->converted = !(per_token && p->write_norm == 0 && nvec <= 832);
                if (!geo->converted) geo->form = tde::kFormLong;
            }
        }
        if (wide) geo->wgs_per_cu = 2;
    }
    return TDE_OK;
}

int64_t algorithmic_bytes(const tde_problem *p, int64_t *scale_elems) {
    const int64_t e = elem_bytes(p->dtype);
    const int64_t T = p->tokens, H = p->hidden, N = p->nranks;
    int64_t out = 0, scales = 0;
    switch (p->quant) {
    case TDE_QUANT_NONE: out = T * H * e; break;
    case TDE_QUANT_FP8_TOKEN:
    case TDE_QUANT_INT8_TOKEN: scales = T; out = T * H + 4 * scales; break;
    case TDE_QUANT_FP8_GROUP: scales = T * (H / TDE_QUANT_GROUP); out = T * H + 4 * scales; break;
    case TDE_QUANT_FP8_STATIC: out = T * H; break;
    }
    if (p->quant != TDE_QUANT_NONE && p->write_norm) out += T * H * e;
    if (scale_elems) *scale_elems = scales;
    return (N + 1) * T * H * e + H * e + T * H * e + out;
}

// Calibration kernel: plain 16-byte copy (known traffic for scaling the profiler's memory counters,
// and the practical copy ceiling of the device).
__global__ void __launch_bounds__(256) copy_kernel(const void *src, void *dst, int64_t total_vecs) {
    using tde::u32x4;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < total_vecs; v += stride) {
        const u32x4 x = __builtin_nontemporal_load((const TDE_GLOBAL u32x4 *)((const TDE_GLOBAL char *)src + v * 16));
        __builtin_nontemporal_store(x, (TDE_GLOBAL u32x4 *)((TDE_GLOBAL char *)dst + v * 16));
    }
}

// Nothing: what one dispatch costs when it does no work.
__global__ void __launch_bounds__(64) empty_kernel() {}

// Streaming-rate probes: one 256-thread workgroup per 4 KiB, no loop (the shape that measured fastest for
// both directions).  MODE 0 reads only (the loaded words feed a store that never executes for real data),
// 1 writes only, 2 copies.
template <int MODE>
__global__ void __launch_bounds__(256) stream_kernel(const void *src, void *dst, int64_t total_bytes) {
    using tde::u32x4;
    const int64_t base = (int64_t)blockIdx.x * 4096;
    const int64_t left = total_bytes - base;
    const uint32_t bytes = left < 4096 ? (uint32_t)left : 4096u;
    const uint32_t off = threadIdx.x * 16u;
    u32x4 x = {threadIdx.x, blockIdx.x, 0x9e3779b9u, 0x7f4a7c15u};
    if (MODE != 1) x = tde::rsrc_load16(tde::row_rsrc(src, base, bytes), off);
    if (MODE == 0) {
        // keeps the load alive; random data never matches, so nothing is written
        if ((x[0] ^ x[1]) == 0x5bd1e995u && (x[2] ^ x[3]) == 0x27d4eb2fu) tde::rsrc_store16(tde::row_rsrc(dst, 0, 16), 0, x);
    } else {
        __builtin_amdgcn_raw_buffer_store_b128(x, tde::row_rsrc(dst, base, bytes), (int)off, 0, MODE == 1 ? tde::kAuxDefault : tde::kAuxStore);
    }
}

} // namespace

struct tde_workspace {
    int32_t nranks;
    int32_t nblocks;
    int64_t slot_bytes;
    void *slots[TDE_MAX_RANKS];
    void *flags;   // nranks regions of nblocks*nranks ints, zeroed (layout parity only: no kernel here reads them)
    int32_t *cells; // 5 int cells: counter, two-shot clock, one-shot clock, one-shot size, one-shot clear
};

extern "C" {

int tde_abi_version(void) { return TDE_ABI_VERSION; }

const char *tde_status_string(int status) {
    switch (status) {
    case TDE_OK: return "ok";
    case TDE_EINVAL: return "invalid argument (null pointer or malformed struct)";
    case TDE_ENRANKS: return "nranks must be 2, 4 or 8";
    case TDE_EDTYPE: return "unsupported dtype (bf16, f16, f32, f64)";
    case TDE_ESHAPE: return "bad shape: hidden*elem_size must be a positive multiple of 16 bytes, tokens >= 0";
    case TDE_EHIDDEN: return "hidden too large for the one-pass row kernel (max 1024 16-byte vectors per row: 8192 bf16/f16, 4096 f32, 2048 f64)";
    case TDE_EALIGN: return "buffer not 16-byte aligned";
    case TDE_EQUANT: return "bad quant mode, per-group quant with hidden not a multiple of 128, or static scale not > 0";
    case TDE_EALGO: return "bad algorithm, or staged algorithm without a stage buffer";
    case TDE_EHIP: return "HIP runtime error (see tde_last_hip_error)";
    case TDE_ERANK: return "rank outside [0, nranks)";
    case TDE_ENOMEM: return "device allocation failed";
    case TDE_ETOOBIG: return "tokens*hidden*elem_size exceeds the library's static stage (TDE_STATIC_STAGE_BYTES)";
    }
    return "unknown status";
}

int tde_last_hip_error(void) { return g_last_hip_error; }

int tde_probe_copy(void *dst, const void *src, int64_t bytes, void *hip_stream) {
    if (dst == nullptr || src == nullptr || bytes < 0 || bytes % 16 != 0) return TDE_EINVAL;
    if (!aligned16(dst) || !aligned16(src)) return TDE_EALIGN;
    if (bytes == 0) return TDE_OK;
    const int64_t vecs = bytes / 16;
    int64_t blocks = (vecs + 255) / 256;
    if (blocks > compute_units() * 16) blocks = compute_units() * 16;
    hipLaunchKernelGGL(copy_kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(hip_stream), src, dst, vecs);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? TDE_OK : hip_fail(e);
}

int tde_probe_launch(void *hip_stream) {
    hipLaunchKernelGGL(empty_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(hip_stream));
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? TDE_OK : hip_fail(e);
}

int tde_probe_stream(void *dst, const void *src, int64_t bytes, int32_t mode, void *hip_stream) {
    if (dst == nullptr || src == nullptr || bytes < 0 || bytes % 16 != 0 || mode < 0 || mode > 2) return TDE_EINVAL;
    if (!aligned16(dst) || !aligned16(src)) return TDE_EALIGN;
    if (bytes == 0) return TDE_OK;
    const int64_t blocks = (bytes + 4095) / 4096;
    if (blocks > 0x7fffffff) return TDE_ESHAPE;
    hipStream_t s = static_cast<hipStream_t>(hip_stream);
    const dim3 grid((unsigned)blocks), block(256);
    switch (mode) {
    case 0: hipLaunchKernelGGL(stream_kernel<0>, grid, block, 0, s, src, dst, bytes); break;
    case 1: hipLaunchKernelGGL(stream_kernel<1>, grid, block, 0, s, src, dst, bytes); break;
    default: hipLaunchKernelGGL(stream_kernel<2>, grid, block, 0, s, src, dst, bytes); break;
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? TDE_OK : hip_fail(e);
}

int tde_device_info(tde_device_info_out *out) {
    if (out == nullptr) return TDE_EINVAL;
    std::memset(out, 0, sizeof(*out));
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    int cu = 0, khz = 0, bits = 0;
    e = hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return hip_fail(e);
    // Clock and width are optional: a runtime that does not report them leaves zeros.
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeMemoryClockRate, dev) != hipSuccess) khz = 0;
    if (hipDeviceGetAttribute(&bits, hipDeviceAttributeMemoryBusWidth, dev) != hipSuccess) bits = 0;
    (void)hipGetLastError();
    size_t free_b = 0, total_b = 0;
    e = hipMemGetInfo(&free_b, &total_b);
    if (e != hipSuccess) return hip_fail(e);
    out->compute_units = cu;
    out->memory_clock_khz = khz;
    out->memory_bus_bits = bits;
    out->total_memory_bytes = (int64_t)total_b;
    return TDE_OK;
}

int tde_plan(const tde_problem *problem, tde_plan_out *plan) {
    if (plan == nullptr) return TDE_EINVAL;
    tde::Geometry g{};
    const int st = validate(problem, &g);
    if (st != TDE_OK) return st;
    std::memset(plan, 0, sizeof(*plan));
    plan->algo = (problem->algo == TDE_ALGO_STAGED || problem->algo == TDE_ALGO_STAGED_OWNED) ? problem->algo : TDE_ALGO_FUSED;
    plan->reference_algo = (problem->tokens <= 128) ? 1 : 2;
    plan->vec_elems = g.vec_elems;
    plan->block_threads = g.block_threads;
    plan->vecs_per_thread = g.vpt;
    plan->rows_per_block = g.rows_per_block;
    plan->grid_blocks = (int32_t)g.grid;
    plan->xcd_chunk = g.xcd_chunk;
    plan->workgroups_per_cu = g.wgs_per_cu;
    plan->lds_bytes = g.lds_bytes;
    plan->algorithmic_bytes = algorithmic_bytes(problem, &plan->scale_elems);
    return TDE_OK;
}

int tde_plan_route(const tde_problem *problem, tde_route_out *route) {
    if (route == nullptr) return TDE_EINVAL;
    tde::Geometry g{};
    const int st = validate(problem, &g);
    if (st != TDE_OK) return st;
    std::memset(route, 0, sizeof(*route));
    route->kernel = g.threads_per_row < tde::kWave ? TDE_KERNEL_SHORT
                    : g.converted                  ? TDE_KERNEL_CONVERTED
                    : g.form == tde::kFormWide     ? TDE_KERNEL_WIDE
                    : g.form == tde::kFormLong     ? TDE_KERNEL_LONG
                                                   : TDE_KERNEL_ROWS;
    route->lanes_per_row = g.threads_per_row;
    route->moved_to_lines = g.line_mask != 0 ? g.line_mask + 1 : 0;
    return TDE_OK;
}

namespace {
enum : int { kPhaseReduce = 1, kPhaseNorm = 2, kTrafficOnly = 4 };

// Whether a row's norm touches bytes that another row's sum still needs, or the other way round: the stage shares bytes with a
// buffer that the norm reads or writes, or a partial shares bytes with an output.
bool phases_overlap(const tde_problem *p, const tde_buffers *b) {
    const int64_t row = p->hidden * elem_bytes(p->dtype), all = p->tokens * row, codes = p->tokens * p->hidden;
    const int64_t scales = p->tokens * (p->quant == TDE_QUANT_FP8_GROUP ? p->hidden / TDE_QUANT_GROUP : 1) * (int64_t)sizeof(float);
    const auto overlap = [](const void *x, int64_t x_bytes, const void *y, int64_t y_bytes) {
        const uintptr_t u = reinterpret_cast<uintptr_t>(x), v = reinterpret_cast<uintptr_t>(y);
        return u != 0 && v != 0 && u < v + (uintptr_t)y_bytes && v < u + (uintptr_t)x_bytes;
    };
    const auto meets_output = [&](const void *x) {
        return overlap(x, all, b->residual_out, all) || overlap(x, all, b->norm_out, all) || overlap(x, all, b->q_out, codes) ||
               overlap(x, all, b->scale_out, scales);
    };
    bool any = meets_output(b->stage) || overlap(b->stage, all, b->residual_in, all) || overlap(b->stage, all, b->gamma, row);
    for (int r = 0; r < p->nranks; ++r) any = any || meets_output(b->partial[r]);
    return any;
}

int run_phases(const tde_problem *p, const tde_buffers *b, void *hip_stream, int phases, int probe_parts = 7) {
    tde::Geometry g{};
    const int st = validate(p, &g);
    if (st != TDE_OK) return st;
    if (b == nullptr) return TDE_EINVAL;
    if (p->tokens == 0) return TDE_OK; // nothing to do; empty buffers may be null
    const bool quant = p->quant != TDE_QUANT_NONE;
    const bool wn = !quant || p->write_norm != 0;
    const bool staged = p->algo == TDE_ALGO_STAGED || p->algo == TDE_ALGO_STAGED_OWNED;
    const bool traffic = phases == kTrafficOnly;
    if (traffic) {
        if (staged) return TDE_EALGO; // the skeleton mirrors the fused kernel only
        phases = kPhaseReduce | kPhaseNorm;
    }
    const bool both = phases == (kPhaseReduce | kPhaseNorm);
    if (!both && !staged) return TDE_EALGO; // a single phase exists only in the staged algorithms
    const bool reads_partials = !staged || (phases & kPhaseReduce);

    for (int r = 0; reads_partials && r < p->nranks; ++r) {
        if (b->partial[r] == nullptr && b->partial_table == nullptr) return TDE_EINVAL;
        if (!aligned16(b->partial[r])) return TDE_EALIGN;
    }
    if (phases & kPhaseNorm) {
        if (!b->residual_in || !b->residual_out || !b->gamma) return TDE_EINVAL;
        if (wn && !b->norm_out) return TDE_EINVAL;
        if (quant && !b->q_out) return TDE_EINVAL;
        if (quant && p->quant != TDE_QUANT_FP8_STATIC && !b->scale_out) return TDE_EINVAL;
    }
    if (staged && !b->stage) return TDE_EALGO;
    if (!aligned16(b->residual_in) || !aligned16(b->residual_out) || !aligned16(b->gamma) ||
        !aligned16(b->norm_out) || !aligned16(b->stage) || !aligned16(b->partial_table))
        return TDE_EALIGN;
    if (quant && ((reinterpret_cast<uintptr_t>(b->q_out) & 7u) || (reinterpret_cast<uintptr_t>(b->scale_out) & 3u)))
        return TDE_EALIGN;

    bool from_table = false;
    for (int r = 0; reads_partials && r < p->nranks; ++r) from_table = from_table || b->partial[r] == nullptr;
    // The staged algorithms as a whole are one launch of the row kernel that also stores the sums to the stage (owned
    // rows: reads the other rows' sums from it), which saves reading the sums back, a launch and the gap before it.  Both
    // are bound by memory: 8 x [2048, 8192] bf16 -> fp8 takes 63.2 us (6.11 TB/s of what must be moved) against 70.3 us in
    // two launches, with owned rows 28.2 us (5.35 TB/s) against 31.2; 8 x [64, 5120] 5.9 against 9.7 and 5.8 against 7.8,
    // 4 x [13721, 532] fp32 38.5 against 47.3 and 27.3 against 36.3.  A stage that overlaps a buffer the norm reads or
    // writes, or a partial that overlaps an output, keeps the two launches, whose second only starts when every sum has
    // been stored; so do partials that only a device table knows (RowArgs has no room for the table beside the stage, and no torch operator makes such a call).
    const bool one_launch = staged && both && !from_table && !phases_overlap(p, b);
    if (staged && !one_launch) {
        const int alone = validate(p, &g, true);
        if (alone != TDE_OK) return alone;
    }

    hipStream_t stream = static_cast<hipStream_t>(hip_stream);
    tde::RowArgs a{};
    if (reads_partials) {
        for (int r = 0; r < p->nranks; ++r) {
            a.set(tde::kPtrPart + r, b->partial[r]);
            if (b->partial[r] == nullptr) a.table_mask |= (uint8_t)(1u << r);
        }
        if (a.table_mask != 0) a.set(tde::kPtrStage, b->partial_table);
    }
    const uint64_t table = reinterpret_cast<uint64_t>(b->partial_table);
    a.set(tde::kPtrResidualIn, b->residual_in);
    a.set(tde::kPtrResidualOut, b->residual_out);
    a.set(tde::kPtrNorm, wn ? b->norm_out : nullptr);
    a.set(tde::kPtrGamma, b->gamma);
    a.set(tde::kPtrCodes, b->q_out);
    a.set(tde::kPtrScale, b->scale_out);
    a.set_hidden(p->hidden);
    a.threads_per_row = (uint16_t)g.threads_per_row;
    a.wave_step = (uint16_t)(32768 / std::max(1, g.threads_per_row / tde::kWave) + 1);
    a.rows_per_block = (uint8_t)g.rows_per_block;
    a.xcd_chunk = (uint8_t)g.xcd_chunk;
    a.tokens = p->tokens;
    a.eps = p->eps;
    a.static_scale = p->static_scale;
    a.chunked_blocks = tde::chunked_blocks(g.grid, (uint32_t)g.xcd_chunk);
    a.owner = (uint8_t)p->rank;
    a.line_mask = (uint8_t)g.line_mask;

    int n = p->nranks;
    hipError_t e = hipSuccess;
    if (traffic && p->dtype == TDE_F64) return TDE_EDTYPE;
    if (traffic) {
        const int code_bytes = quant ? (elem_bytes(p->dtype) == 4 ? 4 : 8) : 0;
        e = tde::launch_traffic(n, g.vpt, code_bytes, wn, a, g, (uint32_t)g.nvec * 16u, (uint32_t)probe_parts, stream);
        return e == hipSuccess ? TDE_OK : hip_fail(e);
    }
    if (one_launch) {
        a.set(tde::kPtrStage, b->stage);
        g.form = p->algo == TDE_ALGO_STAGED_OWNED ? tde::kFormOwned : tde::kFormStaged;
    } else if (staged && (phases & kPhaseReduce)) {
        a.set(tde::kPtrStage, b->stage);
        // All rows as one span of bytes, or only this rank's share (rows == rank mod nranks) row by row.
        const int64_t row_bytes = (int64_t)g.nvec * 16;
        int64_t span_bytes = p->tokens * row_bytes, first = 0, step = 1, rows = 1;
        if (p->algo == TDE_ALGO_STAGED_OWNED) {
            span_bytes = row_bytes;
            first = p->rank;
            step = p->nranks;
            rows = (p->tokens - p->rank + p->nranks - 1) / p->nranks;
        }
        switch (p->dtype) {
        case TDE_BF16: e = tde::launch_reduce_bf16(n, a, table, span_bytes, first, step, rows, stream); break;
        case TDE_F16: e = tde::launch_reduce_f16(n, a, table, span_bytes, first, step, rows, stream); break;
        case TDE_F32: e = tde::launch_reduce_f32(n, a, table, span_bytes, first, step, rows, stream); break;
        case TDE_F64: e = tde::launch_reduce_f64(n, a, table, span_bytes, first, step, rows, stream); break;
        }
        if (e != hipSuccess) return hip_fail(e);
    }
    if (!(phases & kPhaseNorm)) return TDE_OK;
    if (staged && !one_launch) {
        a.table_mask = 0;
        a.set(tde::kPtrPart, b->stage);
        n = 0;
    }
    if (g.threads_per_row < tde::kWave) {
        e = tde::launch_short_rows(p->dtype, n, p->quant, a, g, stream);
        return e == hipSuccess ? TDE_OK : hip_fail(e);
    }
    const bool shifted = a.line_mask != 0;
    switch (p->dtype) {
    case TDE_BF16: e = (shifted ? tde::launch_shifted_rows_bf16 : tde::launch_rows_bf16)(n, g.vpt, p->quant, wn, a, g, stream); break;
    case TDE_F16:
        e = g.converted ? tde::launch_converted_rows_f16(p->quant, wn, a, g, stream)
                        : (shifted ? tde::launch_shifted_rows_f16 : tde::launch_rows_f16)(n, g.vpt, p->quant, wn, a, g, stream);
        break;
    case TDE_F32: e = (shifted ? tde::launch_shifted_rows_f32 : tde::launch_rows_f32)(n, g.vpt, p->quant, wn, a, g, stream); break;
    case TDE_F64: e = tde::launch_rows_f64(n, a, g, stream); break;
    }
    if (e != hipSuccess) return hip_fail(e);
    return TDE_OK;
}
} // namespace

int tde_reduce_rms(const tde_problem *p, const tde_buffers *b, void *hip_stream) {
    return run_phases(p, b, hip_stream, kPhaseReduce | kPhaseNorm);
}

int tde_stage_reduce(const tde_problem *p, const tde_buffers *b, void *hip_stream) {
    return run_phases(p, b, hip_stream, kPhaseReduce);
}

int tde_stage_norm(const tde_problem *p, const tde_buffers *b, void *hip_stream) {
    return run_phases(p, b, hip_stream, kPhaseNorm);
}

int tde_reduce_rms_static_stage(const tde_problem *p, const tde_buffers *b, void *hip_stream) {
    if (p == nullptr || b == nullptr) return TDE_EINVAL;
    if (p->algo != TDE_ALGO_AUTO && p->algo != TDE_ALGO_STAGED) return TDE_EALGO;
    tde_problem staged = *p;
    staged.algo = TDE_ALGO_STAGED;
    const int st = validate(&staged, nullptr);
    if (st != TDE_OK) return st;
    // validate() has bounded hidden and checked that tokens * hidden * elem does not overflow
    if (p->tokens * p->hidden * elem_bytes(p->dtype) > (int64_t)TDE_STATIC_STAGE_BYTES) return TDE_ETOOBIG;
    void *stage = nullptr;
    const int sp = static_stage_ptr(&stage);
    if (sp != TDE_OK) return sp;
    tde_buffers with_stage = *b;
    with_stage.stage = stage;
    return run_phases(&staged, &with_stage, hip_stream, kPhaseReduce | kPhaseNorm);
}

int tde_probe_rows(const tde_problem *p, const tde_buffers *b, void *hip_stream) {
    return run_phases(p, b, hip_stream, kTrafficOnly);
}

int tde_probe_rows_parts(const tde_problem *p, const tde_buffers *b, int32_t parts, void *hip_stream) {
    if (parts < 1 || parts > 7) return TDE_EINVAL;
    return run_phases(p, b, hip_stream, kTrafficOnly, parts);
}

// ---- emulated peer workspace ----------------------------------------------------------------

int tde_workspace_create(int32_t nranks, int32_t nblocks, int64_t slot_bytes, tde_workspace **out) {
    if (out == nullptr) return TDE_EINVAL;
    *out = nullptr;
    if (!(nranks == 2 || nranks == 4 || nranks == 8)) return TDE_ENRANKS;
    if (nblocks < 1 || nblocks > 65536) return TDE_EINVAL;
    if (slot_bytes <= 0 || slot_bytes % 16 != 0) return TDE_ESHAPE;
    tde_workspace *ws = new (std::nothrow) tde_workspace();
    if (ws == nullptr) return TDE_ENOMEM;
    ws->nranks = nranks;
    ws->nblocks = nblocks;
    ws->slot_bytes = slot_bytes;
    hipError_t e = hipSuccess;
    for (int r = 0; r < nranks && e == hipSuccess; ++r) e = hipMalloc(&ws->slots[r], (size_t)slot_bytes * 2);
    // one flag region per rank, each nblocks * nranks ints as the reference sizes it (src/ops/all_reduce_fusion.cpp:72)
    const size_t flag_bytes = (size_t)nranks * nblocks * nranks * sizeof(int32_t);
    if (e == hipSuccess) e = hipMalloc(&ws->flags, flag_bytes);
    if (e == hipSuccess) e = hipMemset(ws->flags, 0, flag_bytes);
    if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void **>(&ws->cells), 5 * 64);
    if (e == hipSuccess) e = hipMemset(ws->cells, 0, 5 * 64);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess) {
        tde_workspace_destroy(ws);
        g_last_hip_error = (int)e;
        return (e == hipErrorOutOfMemory) ? TDE_ENOMEM : TDE_EHIP;
    }
    *out = ws;
    return TDE_OK;
}

int tde_workspace_destroy(tde_workspace *ws) {
    if (ws == nullptr) return TDE_OK;
    for (int r = 0; r < TDE_MAX_RANKS; ++r)
        if (ws->slots[r]) (void)hipFree(ws->slots[r]);
    if (ws->flags) (void)hipFree(ws->flags);
    if (ws->cells) (void)hipFree(ws->cells);
    delete ws;
    return TDE_OK;
}

void *tde_workspace_slot(const tde_workspace *ws, int32_t r) {
    if (ws == nullptr || r < 0 || r >= ws->nranks) return nullptr;
    return ws->slots[r];
}

void *tde_workspace_stage(const tde_workspace *ws, int32_t r) {
    if (ws == nullptr || r < 0 || r >= ws->nranks) return nullptr;
    return static_cast<char *>(ws->slots[r]) + ws->slot_bytes;
}

int64_t tde_workspace_slot_bytes(const tde_workspace *ws) { return ws ? ws->slot_bytes : 0; }
int32_t tde_workspace_nranks(const tde_workspace *ws) { return ws ? ws->nranks : 0; }

int tde_workspace_fill_table(const tde_workspace *ws, void **table, int32_t entries) {
    if (ws == nullptr || table == nullptr) return TDE_EINVAL;
    const int n = ws->nranks;
    if (entries != 3 * n + 5) return TDE_EINVAL;
    for (int r = 0; r < n; ++r) {
        table[r] = ws->slots[r];
        table[n + r] = static_cast<char *>(ws->flags) + (size_t)r * ws->nblocks * n * sizeof(int32_t);
        table[2 * n + r] = ws->slots[r];
    }
    for (int c = 0; c < 5; ++c) table[3 * n + c] = reinterpret_cast<char *>(ws->cells) + 64 * c;
    return TDE_OK;
}

} // extern "C"
