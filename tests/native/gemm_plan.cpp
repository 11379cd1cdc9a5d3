// kudacuda_amd/csrc/kc_gemm_plan.h for the tests: out = {shape, tokens of a block, splits}.
#include <cstdint>

#include "../../kudacuda_amd/csrc/kc_gemm_plan.h"

extern "C" void gemm_plan(int epi, int64_t m, int64_t n, int64_t k, int64_t offset, int64_t* out) {
    const auto aligned = reinterpret_cast<void*>(uintptr_t{4096});
    kc::Nf4GemmArgs a;
    a.x = static_cast<const uint16_t*>(aligned);
    a.out = reinterpret_cast<uint16_t*>(uintptr_t{4096} + static_cast<uintptr_t>(offset));  // bytes
    for (int i = 0; i < 3; ++i) {
        a.w[i] = static_cast<const uint8_t*>(aligned);
    }
    a.residual = static_cast<const uint16_t*>(aligned);
    a.kcache = a.vcache = static_cast<uint16_t*>(aligned);
    a.rope_cos = a.rope_sin = a.partials = static_cast<float*>(aligned);
    a.partial_floats = kc::kGemmScratchFloats;
    a.m = m;
    a.n = n;
    a.k = k;
    a.q_rows = 2048;
    a.kv_rows = 256;
    const kc::GemmPlan p = kc::gemm_plan(static_cast<kc::GemmEpi>(epi), a);
    out[0] = static_cast<int64_t>(p.shape);
    out[1] = p.tokens;
    out[2] = p.splits;
}
