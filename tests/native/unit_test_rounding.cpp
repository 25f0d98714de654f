// Host check of the row kernels' correctly rounded reciprocals, roots and quotients (csrc/tde_rows.h): the functions that the
// kernels run, with every approximation that the hardware's one-unit instructions may return in place of the instruction.
//   g++-style exit status 0: everything as the plain IEEE operation gives it; otherwise what differs, one line a kind.
#include "tde_rows.h"

#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <thread>
#include <vector>

namespace {

float value(uint32_t bits) {
    float f;
    std::memcpy(&f, &bits, 4);
    return f;
}
uint32_t bits(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    return u;
}

std::atomic<int> failed{0};

// check(i) for i in [0, n): what is wrong is counted, the first found is shown.
template <class F>
void sweep(const char *what, uint32_t n, F wrong) {
    std::atomic<long> count{0};
    std::atomic<uint32_t> at{0};
    std::vector<std::thread> pool;
    for (uint32_t k = 0; k < 8; ++k)
        pool.emplace_back([&, k] {
            for (uint32_t i = k; i < n; i += 8)
                if (wrong(i)) {
                    ++count;
                    at = i;
                }
        });
    for (auto &t : pool) t.join();
    std::printf("%s: %ld of %u wrong, last %08x\n", what, count.load(), n, at.load());
    if (count != 0) failed = 1;
}

// The two floats around 1/d (an instruction with an error of at most one unit returns one of them), or 1/d itself.
void around_reciprocal(float d, float (&out)[2]) {
    const float r = 1.0f / d;
    const double e = std::fma((double)r, (double)d, -1.0); // exact: 48 bits
    out[0] = e > 0.0 ? value(bits(r) - 1) : r;
    out[1] = e < 0.0 ? value(bits(r) + 1) : r;
}

} // namespace

int main() {
    // every mantissa and both parities of the exponent, approximations up to three units off, at the exponents of the kernels' range
    for (int shift : {-30, 0, 49})
        sweep("1/sqrt", 1u << 24, [shift](uint32_t i) {
            const float m = std::ldexp(value(0x3f800000u + i), 2 * shift), want = 1.0f / std::sqrt(m);
            const uint32_t y = bits((float)(1.0 / std::sqrt((double)m)));
            bool wrong = false;
            for (int off = -3; off <= 3; ++off) wrong = wrong || bits(tde::reciprocal_of_root(m, value(y + off))) != bits(want);
            return wrong;
        });
    sweep("1/d", (1u << 23) - 1, [](uint32_t i) { // all ones in d: see below
        const float d = value(0x3f800000u + i);
        float approx[2];
        around_reciprocal(d, approx);
        return bits(tde::refined_reciprocal(d, approx[0])) != bits(1.0f / d) || bits(tde::refined_reciprocal(d, approx[1])) != bits(1.0f / d);
    });
    // the mean: sums of every size over every row length, and sums whose quotient lies next to the middle of two floats
    sweep("sum / h", 8192 * 64, [](uint32_t i) {
        const float h = (float)(i % 8192 + 1), r = 1.0f / h;
        uint32_t x = i * 2654435761u;
        for (int k = 0; k < 64; ++k) {
            x = x * 1664525u + 1013904223u;
            const double middle = (double)value(0x3f800000u + (x >> 9)) + 0x1p-24;
            const uint32_t near = bits((float)(middle * h));
            for (int off = -1; off <= 1; ++off) {
                const float sum = value(near + off);
                if (bits(tde::div_shared(sum, h, r)) != bits(sum / h)) return true;
            }
        }
        return false;
    });
    // fp32 quotients next to every boundary between two codes of either type, for every mantissa of a scale
    std::vector<float> boundaries;
    for (int k = 0; k < 127; ++k) boundaries.push_back(k + 0.5f);
    sweep("y / d", (1u << 23), [&](uint32_t i) {
        const float d = value(0x3f800000u + i), r = 1.0f / d;
        for (float b : boundaries) {
            const uint32_t near = bits(b * d);
            for (int off = -1; off <= 1; ++off) {
                const float y = value(near + off);
                if (bits(tde::div_shared(y, d, r)) != bits(y / d)) return true;
            }
        }
        return false;
    });
    // Codes of 2-byte elements: the elements of 11 bits on both sides of every boundary (those of 8 bits are among these, and the
    // quotient grows with y).  The boundaries of fp8 codes are those of int8 codes times powers of two, which only shift it; the
    // divisors are taken at the ends of the fast range too.  All ones in d: from 1/d as it is correctly rounded, which is what the
    // instruction gives (test_codes_of_every_element_gpu.py has that divisor); from the float below, 2^k / d would be a tie.
    const auto side = [](float q, float b) { return q < b ? -1 : (q > b ? 1 : 0); };
    for (int shift : {0, -60, 59}) {
        const uint32_t step = shift == 0 ? 1 : 61;
        sweep("codes of 2-byte elements", (1u << 23) / step + 1, [&, shift, step](uint32_t i) {
            const uint32_t mantissa = i * step < 0x7fffffu ? i * step : 0x7fffffu;
            const float d = std::ldexp(value(0x3f800000u + mantissa), shift);
            float approx[2];
            around_reciprocal(d, approx);
            if (mantissa == 0x7fffffu) approx[0] = approx[1] = 1.0f / d;
            for (float start : approx) {
                const tde::Divisor<tde::ElemF16> divisor(d, start);
                for (float b : boundaries) {
                    const uint32_t below = bits(b * d) & ~0x1fffu; // 10 bits behind the leading one
                    for (uint32_t off : {0u, 0x2000u}) {
                        const float y = value(below + off);
                        if (side(divisor.quotient(y), b) != side(y / d, b)) return true;
                    }
                }
                if (bits(divisor.quotient(-0.0f)) != 0x80000000u || divisor.quotient(-INFINITY) != -INFINITY || divisor.quotient(INFINITY) != INFINITY) return true;
            }
            return false;
        });
    }
    return failed;
}
