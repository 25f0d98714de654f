// Host check that tde_plan reports the launch that tde_reduce_rms makes: grid, workgroup, dynamic LDS, and the attribute that
// goes with more than 64 KiB of it.  The runtime's entry points on that path are defined here, so the library calls these;
// no device is asked for (a plan without one counts 256 compute units) and nothing is launched.
//   g++-style exit status 0: as reported; otherwise the first differences, one line each.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <map>
#include <set>

#include "tde_abi.h"

namespace {
struct Launch {
    const void *kernel;
    dim3 grid, block;
    size_t lds;
} last;
int launches = 0;
std::map<const void *, int> ceiling; // dynamic LDS that a kernel may ask for, where it was raised
} // namespace

extern "C" hipError_t hipGetDevice(int *device) {
    *device = 0;
    return hipSuccess;
}
extern "C" hipError_t hipDeviceGetAttribute(int *value, hipDeviceAttribute_t attribute, int) {
    *value = attribute == hipDeviceAttributeMultiprocessorCount ? 256 : 0;
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void *kernel, hipFuncAttribute, int value) {
    ceiling[kernel] = value;
    return hipSuccess;
}
extern "C" hipError_t hipLaunchKernel(const void *kernel, dim3 grid, dim3 block, void **, size_t lds, hipStream_t) {
    last = {kernel, grid, block, lds};
    ++launches;
    return hipSuccess;
}

int main() {
    const int64_t rows[] = {1,    16,   128,  512,  768,  1023, 1024, 1257, 2047, 2048, 4095, 4096, 4097,  6143,  6144,  8191, 8192,
                            8193, 10024, 12000, 16383, 16384, 20000, 32768, 40188, 65536};
    const int64_t vectors[] = {1, 2, 63, 64, 65, 127, 128, 129, 192, 256, 257, 320, 384, 512, 513, 576, 613, 614, 615, 640, 641, 704, 768, 769, 832, 896, 1000, 1024};
    const int elem[] = {2, 2, 4, 8}; // TDE_BF16, TDE_F16, TDE_F32, TDE_F64
    long calls = 0, wrong = 0, large = 0;
    std::set<std::pair<int, int>> limits; // (algorithm, limit) met
    for (int dtype = TDE_BF16; dtype <= TDE_F64; ++dtype)
        for (int n = 2; n <= 8; n *= 2)
            for (int quant = TDE_QUANT_NONE; quant <= TDE_QUANT_FP8_STATIC; ++quant)
                for (int wn = 0; wn <= (quant != TDE_QUANT_NONE); ++wn)
                    for (int algo = TDE_ALGO_FUSED; algo <= TDE_ALGO_STAGED_OWNED; ++algo)
                        for (int64_t tokens : rows)
                            for (int64_t nvec : vectors)
                                for (int limit : {0, -1, 1, 2, 8}) {
                                    tde_problem p{};
                                    p.dtype = dtype;
                                    p.nranks = n;
                                    p.tokens = tokens;
                                    p.hidden = nvec * 16 / elem[dtype];
                                    p.eps = 1e-6f;
                                    p.quant = quant;
                                    p.write_norm = wn;
                                    p.algo = algo;
                                    p.static_scale = quant == TDE_QUANT_FP8_STATIC ? 0.5f : 0.0f;
                                    p.tune_workgroups_per_cu = limit;
                                    tde_plan_out plan{};
                                    if (tde_plan(&p, &plan) != TDE_OK) continue; // a mode that the type or the row length has not
                                    // Buffers a terabyte apart, none of them touched: with room between them the staged algorithms
                                    // are one launch.
                                    tde_buffers b{};
                                    const auto at = [](uintptr_t i) { return reinterpret_cast<void *>(i << 40); };
                                    for (int r = 0; r < n; ++r) b.partial[r] = at(1 + r);
                                    b.residual_in = at(16);
                                    b.residual_out = at(17);
                                    b.gamma = at(18);
                                    if (quant == TDE_QUANT_NONE || wn) b.norm_out = at(19);
                                    if (quant != TDE_QUANT_NONE) b.q_out = at(20);
                                    if (quant != TDE_QUANT_NONE && quant != TDE_QUANT_FP8_STATIC) b.scale_out = static_cast<float *>(at(21));
                                    if (algo != TDE_ALGO_FUSED) b.stage = at(22);
                                    const int before = launches, status = tde_reduce_rms(&p, &b, nullptr);
                                    ++calls;
                                    large += plan.lds_bytes > 64 * 1024;
                                    if (limit == 0) limits.insert({algo, plan.workgroups_per_cu});
                                    const bool raised = ceiling.count(last.kernel) != 0 && ceiling[last.kernel] >= (int)last.lds;
                                    // what the reported limit admits by LDS (beside the kernels' 64 static bytes), registers aside
                                    const int admits = (int)(160 * 1024 / (plan.lds_bytes + 64));
                                    const bool two_by_registers = algo == TDE_ALGO_FUSED && n == 8 && plan.vecs_per_thread == 4 && limit == 0 && plan.workgroups_per_cu == 2;
                                    if (status == TDE_OK && launches == before + 1 && last.grid.x == (unsigned)plan.grid_blocks &&
                                        last.block.x == (unsigned)plan.block_threads && last.lds == (size_t)plan.lds_bytes &&
                                        (last.lds <= 64 * 1024 || raised) &&
                                        (plan.workgroups_per_cu == 0 || admits == plan.workgroups_per_cu || two_by_registers))
                                        continue;
                                    if (++wrong <= 20)
                                        std::printf("dtype %d, %d x [%lld, %lld], quant %d, norm %d, algorithm %d, asked %d: plan says %d per unit, %d x %d threads, %d B; launched %u x %u, %zu B%s\n",
                                                    dtype, n, (long long)tokens, (long long)p.hidden, quant, wn, algo, limit, plan.workgroups_per_cu, plan.grid_blocks,
                                                    plan.block_threads, plan.lds_bytes, last.grid.x, last.block.x, last.lds, raised || last.lds <= 64 * 1024 ? "" : ", ceiling not raised");
                                }
    std::printf("%ld calls, %ld with more than 64 KiB, %zu planned limits, %ld wrong\n", calls, large, limits.size(), wrong);
    // the sweep has to reach the limits it is about: fused 2 to 6, staged 2 to 4, none with owned rows
    for (int l : {0, 2, 3, 4, 5, 6}) wrong += limits.count({TDE_ALGO_FUSED, l}) == 0;
    for (int l : {0, 2, 3, 4}) wrong += limits.count({TDE_ALGO_STAGED, l}) == 0;
    for (const auto &l : limits) wrong += l.first == TDE_ALGO_STAGED_OWNED && l.second != 0;
    return wrong != 0;
}
