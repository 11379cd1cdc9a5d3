// Causal GQA attention of a prefill on the matrix cores (16 query heads over 2
// KV heads, head dim 128): m query rows at positions start + r over cache rows
// [0, start + r], online softmax in fp32.
//
// A block owns 8 tokens of one KV head: two waves of 32 columns (4 tokens x the 8
// query heads that share the KV head) times two K-groups that take alternate 64
// keys of a 128-key window; the groups' results meet in LDS at the end.  Per
// window a wave forms S^T = K q^T with v_mfma_f32_32x32x16_bf16 (A = 32 K rows,
// B = its columns, kept in registers), so a lane holds 32 scores of one column:
// the softmax needs one lane-half exchange for the maximum and none for the sum
// before the end.  Those 32 lie in exactly the B layout that P needs for
// out^T = V^T P^T if V^T's keys are stored in that order, so the weights never
// leave their lane.  They enter as three MFMAs, bf16 parts of 8 bits each whose
// sum is the fp32 weight.  Error before the output's rounding, against 64 bits
// (2-norm, random rows; the row kernel's fp32 sums / this / with two parts): 300
// tokens 1.9e-7 / 1.1e-7 / 1.8e-6, 512 after 1024 8.2e-7 / 2.0e-7 / 2.2e-6, 1999
// 3.9e-7 / 1.7e-7 / 1.9e-6; two parts take 46 us a layer at 1999 tokens, three 54.
// The hardware's exp2 (at most 0.78 ulp off below 0, exp2_fixed 0.87) leaves these
// figures as they are; exp2_fixed in its place takes 95 us.
// V is transposed on its way into LDS (4 keys x 8 dims a thread, byte permutes);
// K rows are swizzled by 16-byte piece; the next window's rows are requested
// while one is computed.
//
// Operands are read from LDS a step ahead of their MFMAs and the weights of 16
// keys are formed between the MFMAs of the 16 before, held there by scheduling
// barriers (left to the compiler each read stalled its own MFMA; with two parts
// 1999 tokens 67 -> 43 us).  A wave of the window takes 64 MFMAs and about as long
// in fp32 arithmetic; two waves a SIMD overlap the two.  Work grows with the position:
// blocks are ordered heavy to light, then light to heavy, so the two that share
// a CU add up alike.
//
// Few tokens over a long cache split the windows over blocks (S) and merge
// partials in a second kernel.  Measured per layer (MI355X, us; before = one
// block per query row, fp32 dot products): 1999 tokens 847 -> 54, 512 after 1024
// 288 -> 29 + 5 (merge), 10 after 1961 about 70 -> 8 + 4.
#include "kc_device.h"
#include "kc_kernels.h"

namespace kc {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kHeads = 8;                 // query heads of a KV head
constexpr int kDim = 128;
constexpr int kBlockTokens = 8;           // of a block: two waves of 4 tokens x 8 heads = 32 columns
constexpr int kGroupKeys = 64;            // keys of one K-group (a pair of waves) and window
constexpr int kWindowKeys = 2 * kGroupKeys;
constexpr int kKBytes = kGroupKeys * kDim * 2;
constexpr int kVPitch = kGroupKeys * 2 + 16;  // bytes of a transposed V row
constexpr int kVBytes = kDim * kVPitch;
constexpr int kGroupBytes = kKBytes + kVBytes;
constexpr float kNegInf = -__builtin_huge_valf();

__device__ __forceinline__ float max_halves(float v) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ __forceinline__ float sum_halves(float v) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

// A block's results (columns: 8 tokens from row0 x 8 heads of KV head g) over
// keys [begin, end) in plain fp32: 4 lanes a column, 32 dims each.
__device__ __forceinline__ void careful_rows(const PrefillAttnArgs& a, int g, int row0, int split, int S, int64_t begin,
                                          int64_t end) {
    const int column = static_cast<int>(threadIdx.x) / 4;
    const int d0 = static_cast<int>(threadIdx.x) % 4 * 32;
    const int row = row0 + column / kHeads;
    if (row >= a.m) {
        return;
    }
    const int head = g * kHeads + column % kHeads;
    const int64_t last = a.start + row + 1;
    end = end < last ? end : last;
    float acc[32] = {};
    float m = kNegInf;
    float l = 0.0f;
    const uint16_t* qp = a.q + static_cast<int64_t>(row) * 2048 + head * kDim + d0;
    for (int64_t key = begin; key < end; ++key) {
        const uint16_t* kp = a.kcache + (g * a.capacity + key) * kDim + d0;
        const uint16_t* vp = a.vcache + (g * a.capacity + key) * kDim + d0;
        float dot = 0.0f;
        for (int d = 0; d < 32; ++d) {
            dot = fmaf(bf16_to_f32(qp[d]), bf16_to_f32(kp[d]), dot);
        }
        dot += __shfl_xor(dot, 1, 4);
        dot += __shfl_xor(dot, 2, 4);
        const float sc = dot * a.qk_scale_log2;
        const float m_new = fmaxf(m, sc);
        const float m_sub = m_new == kNegInf ? 0.0f : m_new;
        const float corr = __builtin_amdgcn_exp2f(m - m_sub);
        const float p = __builtin_amdgcn_exp2f(sc - m_sub);
        l = l * corr + p;
        m = m_new;
#pragma unroll
        for (int d = 0; d < 32; ++d) {
            acc[d] = fmaf(p, bf16_to_f32(vp[d]), acc[d] * corr);
        }
    }
    if (S > 1) {
        const int64_t at = (static_cast<int64_t>(row) * 16 + head) * S + split;
#pragma unroll
        for (int d = 0; d < 32; ++d) {
            a.partials[at * kDim + d0 + d] = acc[d];
        }
        a.partials[a.m * 16 * S * kDim + 2 * at] = m;
        a.partials[a.m * 16 * S * kDim + 2 * at + 1] = l;
        return;
    }
#pragma unroll
    for (int d = 0; d < 32; ++d) {
        a.out[static_cast<int64_t>(row) * 2048 + head * kDim + d0 + d] = Bf16::store(acc[d] / l);
    }
}

__global__ __launch_bounds__(256, 2) void prefill_attention_mfma_kernel(PrefillAttnArgs a, int tiles, int S) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[2 * kGroupBytes];
    __shared__ int s_redo;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31;
    const int q = lane >> 5;
    const int cg = wave & 1;   // column group: tokens 4 cg .. + 3 of the block
    const int kg = wave >> 1;  // K-group
    // blocks in order of falling work, the second half rising, so that the two
    // blocks a CU holds together do about the same everywhere
    const int g = static_cast<int>(blockIdx.x) & 1;
    const int i = static_cast<int>(blockIdx.x) >> 1;
    const int split = i % S;
    const int ti = i / S;
    const int half = (tiles + 1) / 2;
    const int tile = ti < half ? tiles - 1 - ti : ti - half;
    const int row0 = tile * kBlockTokens;
    const int M = static_cast<int>(a.m);
    const int64_t total = a.start + M;  // valid cache rows
    const int rows = M - row0 < kBlockTokens ? M - row0 : kBlockTokens;
    const int64_t keys = a.start + row0 + rows;  // of the block's last token
    const int windows = static_cast<int>((keys + kWindowKeys - 1) / kWindowKeys);
    const int per_split = (windows + S - 1) / S;
    const int w_begin = split * per_split;
    const int w_end = w_begin + per_split < windows ? w_begin + per_split : windows;

    const int tok = row0 + 4 * cg + r / kHeads;  // this lane's column
    const int head = g * kHeads + r % kHeads;
    const int row = tok < M ? tok : M - 1;
    const int64_t pos = a.start + row;
    const int64_t first_pos = a.start + row0 + 4 * cg;  // lowest position of the wave's columns

    bf16x8 qf[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        qf[s] = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const uint4*>(a.q + static_cast<int64_t>(row) * 2048 + head * kDim + 16 * s + 8 * q));
    }
    const uint16_t* const kbase = a.kcache + static_cast<int64_t>(g) * a.capacity * kDim;
    const uint16_t* const vbase = a.vcache + static_cast<int64_t>(g) * a.capacity * kDim;
    const int kc = tid & 15;    // 16-byte piece of a K row
    const int kr = tid >> 4;    // K rows kr, kr + 16, ...
    const int vq = tid & 15;    // V: 4 keys 4 vq .. + 3 of a K-group
    const int vd = tid >> 4;    // and dims 8 vd .. + 7
    const int vpos = 32 * (vq / 8) + 16 * (vq % 8 / 4) + 8 * (vq % 2) + 4 * (vq % 4 / 2);

    typedef uint32_t u32x32 __attribute__((ext_vector_type(32)));
    u32x32 kreg = {}, vreg = {};
    const uint32_t last_key = static_cast<uint32_t>(total - 1);
    auto fetch = [&](int w) __attribute__((always_inline)) {
        const uint32_t base = static_cast<uint32_t>(w) * kWindowKeys;
        const uint8_t* const kb = reinterpret_cast<const uint8_t*>(kbase);
        const uint8_t* const vb = reinterpret_cast<const uint8_t*>(vbase);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t key = base + kr + 16 * j;
            const uint4 v = *reinterpret_cast<const uint4*>(kb + ((key < last_key ? key : last_key) * 256 + 16 * kc));
            kreg[4 * j] = v.x;
            kreg[4 * j + 1] = v.y;
            kreg[4 * j + 2] = v.z;
            kreg[4 * j + 3] = v.w;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t key = base + kGroupKeys * (j / 4) + 4 * vq + j % 4;
            const uint4 v = *reinterpret_cast<const uint4*>(vb + ((key < last_key ? key : last_key) * 256 + 16 * vd));
            vreg[4 * j] = v.x;
            vreg[4 * j + 1] = v.y;
            vreg[4 * j + 2] = v.z;
            vreg[4 * j + 3] = v.w;
        }
    };
    // K rows swizzled by 16-byte piece; V transposed, keys in the order of the
    // weights' operand slots.  Rows past the cache's valid ones hold anything:
    // their V is stored as zero (their weights are zero).
    auto stage = [&](int w) __attribute__((always_inline)) {
        const int64_t base = static_cast<int64_t>(w) * kWindowKeys;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int key = kr + 16 * j;
            *reinterpret_cast<uint4*>(smem + (key / kGroupKeys) * kGroupBytes + (key % kGroupKeys) * (kDim * 2) +
                                      ((kc ^ (key & 15)) * 16)) =
                make_uint4(kreg[4 * j], kreg[4 * j + 1], kreg[4 * j + 2], kreg[4 * j + 3]);
        }
        if (base + kWindowKeys > total) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const bool past = base + kGroupKeys * (j / 4) + 4 * vq + j % 4 >= total;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    vreg[4 * j + c] = past ? 0u : vreg[4 * j + c];
                }
            }
        }
#pragma unroll
        for (int gj = 0; gj < 2; ++gj) {
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                // dim d of keys 0..3: half d % 2 of word d / 2 of each row
                const uint32_t sel = d % 2 == 0 ? 0x05040100u : 0x07060302u;
                const uint32_t lo =
                    __builtin_amdgcn_perm(vreg[16 * gj + 4 + d / 2], vreg[16 * gj + d / 2], sel);
                const uint32_t hi =
                    __builtin_amdgcn_perm(vreg[16 * gj + 12 + d / 2], vreg[16 * gj + 8 + d / 2], sel);
                *reinterpret_cast<uint2*>(smem + gj * kGroupBytes + kKBytes + (8 * vd + d) * kVPitch + 2 * vpos) =
                    make_uint2(lo, hi);
            }
        }
    };

    floatx16 acc[4];
    float m_run = kNegInf;
    float l_run = 0.0f;  // this lane's keys only; the halves meet at the end
    const uint8_t* const s_k = smem + kg * kGroupBytes;
    const uint8_t* const s_v = s_k + kKBytes;
    const int kxor = r & 15;
    auto k_read = [&](uint4 (&k)[2], int s) __attribute__((always_inline)) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            k[kt] = *reinterpret_cast<const uint4*>(s_k + (32 * kt + r) * (kDim * 2) + (((2 * s + q) ^ kxor) * 16));
        }
    };
    auto v_read = [&](uint4& v, int dt, int n) __attribute__((always_inline)) {
        v = *reinterpret_cast<const uint4*>(s_v + (32 * dt + r) * kVPitch + 2 * (16 * n + 8 * q));
    };
    if (tid == 0) {
        s_redo = 0;
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
        acc[dt] = floatx16{};
    }
    if (w_begin < w_end) {
        fetch(w_begin);
    }
    for (int w = w_begin; w < w_end; ++w) {
        const int64_t base = static_cast<int64_t>(w) * kWindowKeys;
        __syncthreads();
        stage(w);
        __syncthreads();
        if (w + 1 < w_end) {
            fetch(w + 1);
        }
        const int64_t key0 = base + kg * kGroupKeys;
        // scores of keys key0 + 32 kt + 8 (e / 4) + 4 q + e % 4; each step's K
        // operands are read while the step before is multiplied
        floatx16 sc[2] = {floatx16{}, floatx16{}};
        uint4 kf[2][2];
        k_read(kf[0], 0);
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            if (s < 7) {
                k_read(kf[(s + 1) & 1], s + 1);
            }
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                sc[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kf[s & 1][kt]), qf[s], sc[kt],
                                                                 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        uint4 vf[4];
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
            v_read(vf[dt], dt, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (__builtin_amdgcn_readfirstlane(static_cast<int>(key0 + kGroupKeys > first_pos + 1)) != 0) {
            // keys that some column may not see
            const int rel = static_cast<int>(pos - key0) - 4 * q;
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    sc[kt][e] = 32 * kt + 8 * (e / 4) + e % 4 <= rel ? sc[kt][e] : kNegInf;
                }
            }
        }
        float mx = sc[0][0];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                mx = fmaxf(mx, sc[kt][e]);
            }
        }
        // log2 domain from here on (the scale is positive)
        const float m_new = fmaxf(m_run, max_halves(mx) * a.qk_scale_log2);
        const float m_sub = m_new == kNegInf ? 0.0f : m_new;
        if (__any(m_new != m_run)) {
            const float corr = __builtin_amdgcn_exp2f(m_run - m_sub);
            l_run *= corr;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    acc[dt][e] *= corr;
                }
            }
            m_run = m_new;
        }
        // weights of 16 keys (step n: scores 8 (n % 2) .. + 7 of tile n / 2) as
        // three bf16 parts, pair by pair: 8 bits each, their sum is the fp32
        // weight exactly (both remainders are exact)
        uint32_t hi[2][4], mid[2][4], lo[2][4];
        auto weights = [&](int n, int e) __attribute__((always_inline)) {
            const float p0 =
                __builtin_amdgcn_exp2f(fmaf(sc[n / 2][8 * (n % 2) + 2 * e], a.qk_scale_log2, -m_sub));
            const float p1 =
                __builtin_amdgcn_exp2f(fmaf(sc[n / 2][8 * (n % 2) + 2 * e + 1], a.qk_scale_log2, -m_sub));
            l_run += p0 + p1;
            const uint32_t h = pack2(p0, p1);
            hi[n & 1][e] = h;
            const float r0 = p0 - __uint_as_float(h << 16);
            const float r1 = p1 - __uint_as_float(h & 0xffff0000u);
            const uint32_t m = pack2(r0, r1);
            mid[n & 1][e] = m;
            lo[n & 1][e] = pack2(r0 - __uint_as_float(m << 16), r1 - __uint_as_float(m & 0xffff0000u));
        };
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            weights(0, e);
        }
        __builtin_amdgcn_sched_barrier(0);
        // between a step's MFMAs the next step's weights are formed and each V
        // operand is replaced by the next step's
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const bf16x8 ph = __builtin_bit_cast(bf16x8, make_uint4(hi[n & 1][0], hi[n & 1][1], hi[n & 1][2], hi[n & 1][3]));
            const bf16x8 pm =
                __builtin_bit_cast(bf16x8, make_uint4(mid[n & 1][0], mid[n & 1][1], mid[n & 1][2], mid[n & 1][3]));
            const bf16x8 pl = __builtin_bit_cast(bf16x8, make_uint4(lo[n & 1][0], lo[n & 1][1], lo[n & 1][2], lo[n & 1][3]));
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vf[dt]), ph, acc[dt], 0, 0, 0);
                acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vf[dt]), pm, acc[dt], 0, 0, 0);
                acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vf[dt]), pl, acc[dt], 0, 0, 0);
                if (n < 3) {
                    weights(n + 1, dt);
                    v_read(vf[dt], dt, n + 1);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // Zero weights (hidden keys, the lower parts of a weight) times an infinity or
    // NaN of V are NaN: a block whose result is not finite starts again, key by
    // key in fp32 with hidden keys left out.
    {
        float zero = l_run * 0.0f;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                zero = fmaf(acc[dt][e], 0.0f, zero);
            }
        }
        if (zero != zero) {
            s_redo = 1;
        }
    }
    __syncthreads();
    if (s_redo != 0) {
        careful_rows(a, g, row0, split, S, static_cast<int64_t>(w_begin) * kWindowKeys,
                     static_cast<int64_t>(w_end) * kWindowKeys);
        return;
    }
    // the K-groups' results meet in group 0; the lane's column is formed again
    // (kept over the loop, which uses every register, its values spilled)
    const int fl = static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
    const int fq = fl >> 5;
    const int ftok = row0 + 4 * cg + fl % 32 / kHeads;
    const int fhead = g * kHeads + fl % kHeads;
    l_run = sum_halves(l_run);
    float* const s_acc = reinterpret_cast<float*>(smem);
    float* const s_ml = s_acc + 2 * 64 * 64;
    if (kg == 1) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                reinterpret_cast<float4*>(s_acc)[(cg * 16 + dt * 4 + i4) * 64 + fl] =
                    make_float4(acc[dt][4 * i4], acc[dt][4 * i4 + 1], acc[dt][4 * i4 + 2], acc[dt][4 * i4 + 3]);
            }
        }
        s_ml[cg * 128 + 2 * fl] = m_run;
        s_ml[cg * 128 + 2 * fl + 1] = l_run;
    }
    __syncthreads();
    if (kg == 1) {
        return;
    }
    const float m1 = s_ml[cg * 128 + 2 * fl];
    const float l1 = s_ml[cg * 128 + 2 * fl + 1];
    const float m_all = fmaxf(m_run, m1);
    const float m_sub = m_all == kNegInf ? 0.0f : m_all;
    const float c0 = __builtin_amdgcn_exp2f(m_run - m_sub);
    const float c1 = __builtin_amdgcn_exp2f(m1 - m_sub);
    const float l_all = l_run * c0 + l1 * c1;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            const float4 v = reinterpret_cast<const float4*>(s_acc)[(cg * 16 + dt * 4 + i4) * 64 + fl];
            acc[dt][4 * i4] = acc[dt][4 * i4] * c0 + v.x * c1;
            acc[dt][4 * i4 + 1] = acc[dt][4 * i4 + 1] * c0 + v.y * c1;
            acc[dt][4 * i4 + 2] = acc[dt][4 * i4 + 2] * c0 + v.z * c1;
            acc[dt][4 * i4 + 3] = acc[dt][4 * i4 + 3] * c0 + v.w * c1;
        }
    }
    if (S > 1) {
        if (ftok < M) {
            const int64_t at = (static_cast<int64_t>(ftok) * 16 + fhead) * S + split;
            float* dst = a.partials + at * kDim;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    *reinterpret_cast<float4*>(dst + 32 * dt + 8 * i4 + 4 * fq) =
                        make_float4(acc[dt][4 * i4], acc[dt][4 * i4 + 1], acc[dt][4 * i4 + 2], acc[dt][4 * i4 + 3]);
                }
            }
            if (fq == 0) {
                *reinterpret_cast<float2*>(a.partials + a.m * 16 * S * kDim + 2 * at) = make_float2(m_all, l_all);
            }
        }
        return;
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
        uint32_t h[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            h[e] = pack2(acc[dt][2 * e] / l_all, acc[dt][2 * e + 1] / l_all);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            // lane halves exchange so that each holds 8 consecutive dims
            const auto s0 = __builtin_amdgcn_permlane32_swap(h[4 * j], h[4 * j + 2], false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(h[4 * j + 1], h[4 * j + 3], false, false);
            if (ftok < M) {
                *reinterpret_cast<uint4*>(a.out + static_cast<int64_t>(ftok) * 2048 + fhead * kDim + 32 * dt + 16 * j +
                                          8 * fq) = make_uint4(s0[0], s1[0], s0[1], s1[1]);
            }
        }
    }
}

// The splits of one row and head: 32 lanes of 4 dims x G groups of splits (every
// G-th split each, up to 8 requested together), the groups' sums through LDS.
// grid (m, 16 / (8 / G)), 256 threads.  One thread per (head, dims) over all
// splits took 7.4 us for 16 splits of 10 rows, a chain of memory round trips.
template <int G>
__global__ __launch_bounds__(256) void prefill_attention_merge_kernel(PrefillAttnArgs a, int S) {
    constexpr int kMergeHeads = 8 / G;  // heads of a block
    __shared__ __attribute__((aligned(16))) float s_part[G][kMergeHeads][kDim];
    __shared__ float s_ml[G][kMergeHeads][2];
    const int64_t row = blockIdx.x;
    const int unit = static_cast<int>(threadIdx.x) / 32;
    const int h = unit % kMergeHeads;
    const int grp = unit / kMergeHeads;
    const int head = static_cast<int>(blockIdx.y) * kMergeHeads + h;
    const int d = static_cast<int>(threadIdx.x) % 32 * 4;
    const int64_t at = (row * 16 + head) * S;
    const float* ml = a.partials + a.m * 16 * S * kDim + 2 * at;
    const float* src = a.partials + at * kDim + d;
    float m = kNegInf;
    float l = 0.0f;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int s0 = grp; s0 < S; s0 += 8 * G) {
        float4 p[8];
        float2 w[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int s = s0 + j * G < S ? s0 + j * G : S - 1;
            p[j] = *reinterpret_cast<const float4*>(src + static_cast<int64_t>(s) * kDim);
            w[j] = *reinterpret_cast<const float2*>(ml + 2 * s);
        }
        float m_new = m;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            m_new = fmaxf(m_new, s0 + j * G < S ? w[j].x : kNegInf);
        }
        const float m_sub = m_new == kNegInf ? 0.0f : m_new;
        const float corr = __builtin_amdgcn_exp2f(m - m_sub);
        m = m_new;
        l *= corr;
        v = make_float4(v.x * corr, v.y * corr, v.z * corr, v.w * corr);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (s0 + j * G < S) {  // (a split without keys of this row: weight 0 on zeros)
                const float c = __builtin_amdgcn_exp2f(w[j].x - m_sub);
                l = fmaf(w[j].y, c, l);
                v.x = fmaf(p[j].x, c, v.x);
                v.y = fmaf(p[j].y, c, v.y);
                v.z = fmaf(p[j].z, c, v.z);
                v.w = fmaf(p[j].w, c, v.w);
            }
        }
    }
    if constexpr (G > 1) {
        *reinterpret_cast<float4*>(&s_part[grp][h][d]) = v;
        if (d == 0) {
            s_ml[grp][h][0] = m;
            s_ml[grp][h][1] = l;
        }
        __syncthreads();
        if (grp != 0) {
            return;
        }
        float m_all = m;
#pragma unroll
        for (int o = 1; o < G; ++o) {
            m_all = fmaxf(m_all, s_ml[o][h][0]);
        }
        const float m_sub = m_all == kNegInf ? 0.0f : m_all;
        const float c = __builtin_amdgcn_exp2f(m - m_sub);
        l *= c;
        v = make_float4(v.x * c, v.y * c, v.z * c, v.w * c);
#pragma unroll
        for (int o = 1; o < G; ++o) {
            const float co = __builtin_amdgcn_exp2f(s_ml[o][h][0] - m_sub);
            const float4 p = *reinterpret_cast<const float4*>(&s_part[o][h][d]);
            l = fmaf(s_ml[o][h][1], co, l);
            v.x = fmaf(p.x, co, v.x);
            v.y = fmaf(p.y, co, v.y);
            v.z = fmaf(p.z, co, v.z);
            v.w = fmaf(p.w, co, v.w);
        }
    }
    *reinterpret_cast<uint2*>(a.out + row * 2048 + head * kDim + d) =
        make_uint2(pack2(v.x / l, v.y / l), pack2(v.z / l, v.w / l));
}

}  // namespace

bool prefill_attention_mfma_fits(const PrefillAttnArgs& a) {
    const auto aligned16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    return aligned16(a.q) && aligned16(a.kcache) && aligned16(a.vcache) && aligned16(a.out) && aligned16(a.partials) &&
           a.start + a.m <= (int64_t{1} << 22) && a.qk_scale_log2 > 0.0f;
}

hipError_t launch_prefill_attention_mfma(const PrefillAttnArgs& a, hipStream_t stream) {
    if (a.m < 1 || a.start < 0 || a.start + a.m > a.capacity || a.q == nullptr || a.kcache == nullptr ||
        a.vcache == nullptr || a.out == nullptr) {
        return hipErrorInvalidValue;
    }
    const int64_t tiles = (a.m + kBlockTokens - 1) / kBlockTokens;
    const int64_t windows = (a.start + a.m + kWindowKeys - 1) / kWindowKeys;
    // two blocks a CU: few tokens split their keys over blocks
    int64_t S = a.partials == nullptr ? 1 : 512 / (2 * tiles);
    S = S < windows ? S : windows;
    while (S > 1 && a.m * 16 * S * (kDim + 2) > a.partial_floats) {
        --S;
    }
    S = S > 1 ? S : 1;
    if (S > 1) {
        const int64_t per = (windows + S - 1) / S;
        S = (windows + per - 1) / per;  // no split without windows at the last token
    }
    hipLaunchKernelGGL(prefill_attention_mfma_kernel, dim3(static_cast<unsigned>(2 * tiles * S)), dim3(256), 0, stream, a,
                       static_cast<int>(tiles), static_cast<int>(S));
    const hipError_t status = hipGetLastError();
    if (status != hipSuccess || S == 1) {
        return status;
    }
    if (S > 8) {
        hipLaunchKernelGGL(prefill_attention_merge_kernel<8>, dim3(static_cast<unsigned>(a.m), 16), dim3(256), 0, stream, a,
                           static_cast<int>(S));
    } else {
        hipLaunchKernelGGL(prefill_attention_merge_kernel<1>, dim3(static_cast<unsigned>(a.m), 2), dim3(256), 0, stream, a,
                           static_cast<int>(S));
    }
    return hipGetLastError();
}

}  // namespace kc
