// NF4 GEMM on MFMA for few tokens (gemm_few_plan() says how many): out[m, n] =
// epilogue(sum_k x[m, k] * w[n, k]), w[n, k] = bf16(codebook[code] * absmax),
// fp32 accumulation in v_mfma_f32_32x32x16_bf16.
//
// Work split.  A fragment is 32 weight rows: 32 outputs, 16 gate rows and the up
// rows of the same outputs (kSwiGlu), or 16 dims of a head and their rotary
// partners (kQkvRope), so that every epilogue finds its pair in one lane's sums
// and needs no second launch.  A block has WN fragments and WK K-groups of waves;
// a step is 64 WK of k, K-group g takes its window g.  Blocks own 32 NT tokens.
//
// Who loads.  Four loader waves stage x (and each step's block maxima) for a step
// ahead; the compute waves load codes, the WK waves of a fragment whole lines of
// its rows together, up to four steps ahead, and hand them over through LDS two
// steps ahead.  x and codes are asked for by different waves because a wave's
// loads return in order: with both in one wave, waiting for a step's x waits for
// all codes requested before it.  Loading the codes straight in the operand layout
// (32 bytes of each of 32 rows an instruction, and their maxima as 32 single
// words) held the first step back to 6 us of the 16 a gate/up block takes.
//
// What bounds it: LDS in the steps (16 table reads and 4 NT operand reads of 16
// bytes a lane for 2048 weights of a wave: about 1850 cycles a step of 12 waves at
// NT = 2), and about 4 us around them: launch, first loads under the other blocks'
// weight stream, the K-groups' sums.  Measured (MI355X, us per call, weights cold;
// before = 16-token fragments of kc_prefill.hip, above 64 tokens kc_gemm.hip):
//   tokens              16           32           64          100          128
//   gate/up SwiGLU  13.8 -> 13.0 15.7 -> 13.3 21.5 -> 17.9 27.0 -> 23.2 25.6 -> 22.3
//   q (k 2048)       7.3 ->  6.3  8.1 ->  6.6 10.1 ->  8.3 13.1 ->  8.3 14.2 ->  8.4
//   down (k 11008)  11.8 -> 11.6 12.9 -> 12.3 16.4 -> 15.5 20.2 -> 18.6 21.6 -> 19.5
//   gate alone      13.3 ->  9.1              22.8 -> 12.0
// More tokens, against the tile kernel: the table at gemm_few_plan().
#include "kc_device.h"
#include "kc_gemm_plan.h"

namespace kc {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kWindow = 64;  // k of one window and K-group: one absmax block
constexpr int kQuadPitch = 66;  // float4 slots of one quad of a wave's sums in LDS (64 lanes and a bank offset)

constexpr int kLoaders = 4;     // waves that stage x
struct Codes {
    uint4 c;
    float am;
};

// Row of its weight and the weight (seg) that row `fr` of fragment `unit` is.
template <GemmEpi EPI>
__device__ __forceinline__ int frag_row(const Nf4GemmArgs& a, int unit, int fr, int& seg) {
    if constexpr (EPI == GemmEpi::kSwiGlu) {
        seg = fr >> 4;
        return unit * 16 + (fr & 15);
    } else if constexpr (EPI == GemmEpi::kQkvRope) {
        const int n0 = (unit >> 2) * 128;
        const int q_rows = static_cast<int>(a.q_rows);
        const int kv_rows = static_cast<int>(a.kv_rows);
        seg = n0 < q_rows ? 0 : (n0 < q_rows + kv_rows ? 1 : 2);
        return n0 - (seg == 0 ? 0 : (seg == 1 ? q_rows : q_rows + kv_rows)) + (unit & 3) * 16 + (fr & 15) + (fr >> 4) * 64;
    } else {
        seg = 0;
        return unit * 32 + fr;
    }
}

template <GemmEpi EPI, int WN, int WK, int NT>
__global__ __launch_bounds__(64 * (WN * WK + kLoaders)) void nf4_few_gemm_kernel(Nf4GemmArgs a, int base, int extra) {
    constexpr bool kPair = EPI == GemmEpi::kSwiGlu || EPI == GemmEpi::kQkvRope;
    constexpr int kWaves = WN * WK;
    constexpr int kThreads = 64 * (kWaves + kLoaders);
    constexpr int kLoadThreads = 64 * kLoaders;
    constexpr int kTokens = 32 * NT;
    constexpr int kChunks = 8 * WK;                           // 16-byte pieces of a token row of one step
    constexpr int kPieces = kTokens * kChunks / kLoadThreads; // of all rows, per loader thread
    constexpr int kAms = (32 * kWaves + kLoadThreads - 1) / kLoadThreads;  // block maxima of a step, per loader thread
    constexpr int kSlots = kNf4Slots;
    constexpr int kTableBytes = kNf4PairEntries * 256;
    constexpr int kGroupBytes = kTokens * 128;
    constexpr int kBufBytes = kGroupBytes * WK;
    constexpr int kCodePitch = 32 * WK + 16;
    constexpr int kCodeBytes = 32 * WN * kCodePitch;
    constexpr int kAmBytes = 32 * kWaves * 4;
    constexpr int kAtX = kTableBytes;
    constexpr int kAtCodes = kAtX + 2 * kBufBytes;
    constexpr int kAtAm = kAtCodes + 2 * kCodeBytes;
    constexpr int kTiles = kAtAm + 2 * kAmBytes;
    constexpr int kAccBytes = kWaves * NT * 4 * kQuadPitch * 16;
    constexpr int kLds = kTiles > kAccBytes ? kTiles : kAccBytes;
    static_assert(kPieces * kLoadThreads == kTokens * kChunks && kLoadThreads == kNf4PairEntries && kLds <= 160 * 1024,
                  "whole pieces; one table entry a loader thread; one CU's LDS");
    __shared__ __attribute__((aligned(256))) uint8_t smem[kLds];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = static_cast<int>(a.k);
    const int M = static_cast<int>(a.m);
    const int n_tile = blockIdx.x;
    const int split = blockIdx.y;
    const int m0 = blockIdx.z * kTokens;
    // this split's steps
    const int w_begin = split * base + (split < extra ? split : extra);
    const int w_end = w_begin + base + (split < extra ? 1 : 0);
    const int last = w_end - 1;
    auto clamp_w = [&](int w) { return w < last ? w : last; };
    const int units = static_cast<int>(EPI == GemmEpi::kSwiGlu ? a.n >> 4 : a.n >> 5);

    if (wave >= kWaves) {
        // ---- loader waves: the pair table, then x and the block maxima step by step
        const uint32_t lt = static_cast<uint32_t>(tid) & (kLoadThreads - 1);
        constexpr uint32_t kRowsPerPiece = kLoadThreads / kChunks;  // piece j: token row lt / kChunks + j kRowsPerPiece
        const uint8_t* const xbase = reinterpret_cast<const uint8_t*>(a.x) + static_cast<int64_t>(m0) * K * 2;
        const uint32_t c = lt % kChunks;
        const uint32_t t0 = lt / kChunks;
        const uint32_t rows = static_cast<uint32_t>(M - m0);
        uint32_t xoff[kPieces];
#pragma unroll
        for (uint32_t j = 0; j < kPieces; ++j) {
            const uint32_t t = t0 + j * kRowsPerPiece;
            xoff[j] = (t < rows ? t : rows - 1) * (2 * K) + 16 * c;
        }
        typedef uint32_t pieces __attribute__((ext_vector_type(4 * kPieces)));
        pieces xa = {}, xb = {};
        auto fetch = [&](pieces& xr, int w) __attribute__((always_inline)) {
            const uint8_t* const src = xbase + w * (kWindow * WK * 2);
#pragma unroll
            for (int j = 0; j < kPieces; ++j) {
                const uint4 v = *reinterpret_cast<const uint4*>(src + xoff[j]);
                xr[4 * j] = v.x;
                xr[4 * j + 1] = v.y;
                xr[4 * j + 2] = v.z;
                xr[4 * j + 3] = v.w;
            }
        };
        const float* amrow[kAms];
        float ama[kAms], amb[kAms];
        const float2 pair_entry = reinterpret_cast<const float2*>(kNf4PairTable.v)[lt];
        fetch(xa, w_begin);
#pragma unroll
        for (uint32_t j = 0; j < kAms; ++j) {
            const uint32_t e0 = lt + j * kLoadThreads;
            const uint32_t e = e0 < 32 * kWaves ? e0 : e0 - 32 * kWaves;  // the last threads repeat others
            const int u = n_tile * WN + static_cast<int>(e / (32 * WK));
            int seg;
            const int row = frag_row<EPI>(a, u < units ? u : units - 1, (e / WK) % 32, seg);
            const float* const src = seg == 0 ? a.absmax[0] : (seg == 1 ? a.absmax[1] : a.absmax[2]);
            amrow[j] = src + static_cast<int64_t>(row) * (K >> 6) + e % WK;
        }
        auto am_fetch = [&](float (&am)[kAms], int w) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < kAms; ++j) {
                am[j] = amrow[j][w * WK];
            }
        };
        auto am_stage = [&](const float (&am)[kAms], int buf) __attribute__((always_inline)) {
#pragma unroll
            for (uint32_t j = 0; j < kAms; ++j) {
                const uint32_t e0 = lt + j * kLoadThreads;
                const uint32_t e = e0 < 32 * kWaves ? e0 : e0 - 32 * kWaves;
                *reinterpret_cast<float*>(smem + kAtAm + buf * kAmBytes + e * 4) = am[j];
            }
        };
        am_fetch(ama, w_begin);
        am_fetch(amb, clamp_w(w_begin + 1));
        fetch(xb, clamp_w(w_begin + 1));
        auto stage = [&](const pieces& xr, int buf) __attribute__((always_inline)) {
            uint8_t* const dst = smem + kAtX + buf * kBufBytes + (c / 8) * kGroupBytes + t0 * 128;
#pragma unroll
            for (uint32_t j = 0; j < kPieces; ++j) {
                const uint32_t swz = ((c % 8) ^ ((t0 + j * kRowsPerPiece) & 7)) * 16;
                *reinterpret_cast<uint4*>(dst + j * kRowsPerPiece * 128 + swz) =
                    make_uint4(xr[4 * j], xr[4 * j + 1], xr[4 * j + 2], xr[4 * j + 3]);
            }
        };
#pragma unroll
        for (int j = 0; j < kSlots; ++j) {
            *reinterpret_cast<float2*>(smem + lt * 256 + ((j + lt) & (kSlots - 1)) * 8) = pair_entry;
        }
        stage(xa, 0);
        am_stage(ama, 0);
        am_stage(amb, 1);
        fetch(xa, clamp_w(w_begin + 2));
        am_fetch(ama, clamp_w(w_begin + 2));
        am_fetch(amb, clamp_w(w_begin + 3));
        __syncthreads();
        __syncthreads();  // the compute waves have read codes and maxima of the first step
        for (int w = w_begin; w < w_end; ++w) {
            stage(xb, 1);
            am_stage(ama, 0);
            fetch(xb, clamp_w(w + 3));
            am_fetch(ama, clamp_w(w + 4));
            __syncthreads();
            if (++w >= w_end) {
                break;
            }
            stage(xa, 0);
            am_stage(amb, 1);
            fetch(xa, clamp_w(w + 3));
            am_fetch(amb, clamp_w(w + 4));
            __syncthreads();
        }
        __syncthreads();
    } else {
        // ---- compute waves
        const SlicedLookup cb{reinterpret_cast<const char*>(smem), (tid & (kSlots - 1)) * 8u};
        const int wn = wave % WN;
        const int g = wave / WN;  // K-group
        const int r = lane & 31;
        const int q = lane >> 5;
        const int unit = n_tile * WN + wn < units ? n_tile * WN + wn : units - 1;
        // the fragment's WK waves load its codes of a step together, whole lines of a row
        const int piece = g * 64 + lane;
        const int prow = piece / (2 * WK);
        const int ppart = piece % (2 * WK);
        int seg;
        const int row = frag_row<EPI>(a, unit, prow, seg);
        const uint8_t* const wsel = seg == 0 ? a.w[0] : (seg == 1 ? a.w[1] : a.w[2]);
        const uint8_t* const wrow = wsel + static_cast<int64_t>(row) * (K >> 1) + 16 * ppart;
        uint8_t* const code_in = smem + kAtCodes + (wn * 32 + prow) * kCodePitch + 16 * ppart;
        const uint8_t* const code_out = smem + kAtCodes + (wn * 32 + r) * kCodePitch + 32 * g + 16 * q;
        const uint8_t* const am_out = smem + kAtAm + ((wn * 32 + r) * WK + g) * 4;
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        auto w_fetch = [&](int w) __attribute__((always_inline)) {
            const uint4 v = load_stream(reinterpret_cast<const uint4*>(wrow + w * (32 * WK)));
            return u32x4{v.x, v.y, v.z, v.w};
        };
        auto w_stage = [&](const u32x4& v, int buf) __attribute__((always_inline)) {
            *reinterpret_cast<uint4*>(code_in + buf * kCodeBytes) = make_uint4(v[0], v[1], v[2], v[3]);
        };
        auto w_read = [&](Codes& to, int buf) __attribute__((always_inline)) {
            to.c = *reinterpret_cast<const uint4*>(code_out + buf * kCodeBytes);
            to.am = *reinterpret_cast<const float*>(am_out + buf * kAmBytes);
        };
        u32x4 f0 = w_fetch(w_begin);
        u32x4 f1 = w_fetch(clamp_w(w_begin + 1));
        u32x4 f2 = w_fetch(clamp_w(w_begin + 2));
        u32x4 f3 = w_fetch(clamp_w(w_begin + 3));
        uint32_t boff[4];  // this lane's operand piece of k-step s in a token row
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            boff[s] = kAtX + g * kGroupBytes + r * 128 + (((4 * q + s) ^ (r & 7)) * 16);
        }
        floatx16 acc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            acc[t] = floatx16{};
        }
        w_stage(f0, 0);
        w_stage(f1, 1);
        f0 = w_fetch(clamp_w(w_begin + 4));
        f1 = w_fetch(clamp_w(w_begin + 5));
        __syncthreads();
        Codes c0, c1;
        w_read(c0, 0);
        __syncthreads();  // codes and maxima of the first step are read: their buffers are free
        float2 p[4];  // table values: byte u of the k-step's code word
        bf16x8 A0, A1;
        uint4 B[NT];
        auto look = [&](int u, const Codes& from, int s) __attribute__((always_inline)) {
            const uint32_t w = word_of(from.c, s);
            p[u] = u == 0 ? *cb.template entry<0>(w)
                          : (u == 1 ? *cb.template entry<1>(w)
                                    : (u == 2 ? *cb.template entry<2>(w) : *cb.template entry<3>(w)));
        };
        auto form = [&](int u, bf16x8& A, const Codes& from) __attribute__((always_inline)) {
            A[2 * u] = static_cast<__bf16>(p[u].x * from.am);
            A[2 * u + 1] = static_cast<__bf16>(p[u].y * from.am);
        };
        auto b_read = [&](int t, int bb, int sb) __attribute__((always_inline)) {
            B[t] = *reinterpret_cast<const uint4*>(smem + bb * kBufBytes + t * 32 * 128 + boff[sb]);
        };
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            look(u, c0, 0);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            b_read(t, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            form(u, A0, c0);
            look(u, c0, 1);
        }
        int w = w_begin;
        // One 16-k step of NT MFMAs: between them the next step's weights An are
        // formed, their table values' registers request the step after that (codes
        // cl, word sl), and each x operand is replaced by the next step's.
        auto step = [&](const bf16x8& A, bf16x8& An, const Codes& cl, int sl, const Codes& cn, int bb,
                        int sb) __attribute__((always_inline)) {
            constexpr int kUnits = 4 / NT;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, __builtin_bit_cast(bf16x8, B[t]), acc[t], 0, 0, 0);
#pragma unroll
                for (int u = t * kUnits; u < (t + 1) * kUnits; ++u) {
                    form(u, An, cn);
                    look(u, cl, sl);
                }
                b_read(t, bb, sb);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // Step w (buffers buf): codes of w + 1 are read, those of w + 2 take the place
        // of this step's in LDS, and their registers request w + 6.
        auto window = [&](const Codes& cur, Codes& next, u32x4& f, int buf) __attribute__((always_inline)) {
            w_read(next, buf ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            step(A0, A1, cur, 2, cur, buf, 1);
            w_stage(f, buf);
            f = w_fetch(clamp_w(w + 6));
            __builtin_amdgcn_sched_barrier(0);
            step(A1, A0, cur, 3, cur, buf, 2);
            step(A0, A1, next, 0, cur, buf, 3);
            __syncthreads();
            step(A1, A0, next, 1, next, buf ^ 1, 0);
            ++w;
        };
        while (true) {
            window(c0, c1, f2, 0);
            if (w >= w_end) break;
            window(c1, c0, f3, 1);
            if (w >= w_end) break;
            window(c0, c1, f0, 0);
            if (w >= w_end) break;
            window(c1, c0, f1, 1);
            if (w >= w_end) break;
        }
        __syncthreads();
        float4* const s_sum = reinterpret_cast<float4*>(smem);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                s_sum[((wave * NT + t) * 4 + i4) * kQuadPitch + lane] =
                    make_float4(acc[t][4 * i4], acc[t][4 * i4 + 1], acc[t][4 * i4 + 2], acc[t][4 * i4 + 3]);
            }
        }
    }
    __syncthreads();
    const float4* const s_acc = reinterpret_cast<const float4*>(smem);
    const int S = gridDim.y;

    // columns 8 i4 .. + 7 of fragment f, token tile t, token tr of the tile
    auto sum8 = [&](int f, int t, int i4, int tr, float (&v)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < WK; ++k) {
            const float4* src = s_acc + (((k * WN + f) * NT + t) * 4 + i4) * kQuadPitch + tr;
            const float4 lo = src[0];
            const float4 hi = src[32];
            const float b[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                v[i] = k == 0 ? b[i] : v[i] + b[i];
            }
        }
    };
    if (S > 1 || !kPair) {
        constexpr int kRuns = WN * NT * 32 * 4;
        for (int e = tid; e < kRuns; e += kThreads) {
            const int i4 = e & 3;
            const int tr = (e >> 2) & 31;
            const int t = (e >> 7) % NT;
            const int f = (e >> 7) / NT;
            const int u = n_tile * WN + f;
            const int m = m0 + 32 * t + tr;
            if (m >= M || u >= units) {
                continue;
            }
            float v[8];
            sum8(f, t, i4, tr, v);
            int64_t col;
            if constexpr (EPI == GemmEpi::kSwiGlu) {
                col = static_cast<int64_t>(u) * 16 + 8 * (i4 & 1);
            } else if constexpr (EPI == GemmEpi::kQkvRope) {
                col = static_cast<int64_t>(u / 4) * 128 + u % 4 * 16 + 8 * (i4 & 1) + 64 * (i4 >> 1);
            } else {
                col = static_cast<int64_t>(u) * 32 + 8 * i4;
            }
            if (S > 1) {
                const int64_t plane = EPI == GemmEpi::kSwiGlu ? static_cast<int64_t>(i4 >> 1) * S + split : split;
                float4* dst = reinterpret_cast<float4*>(a.partials + (plane * M + m) * a.n + col);
                dst[0] = make_float4(v[0], v[1], v[2], v[3]);
                dst[1] = make_float4(v[4], v[5], v[6], v[7]);
                continue;
            }
            if constexpr (!kPair) {
                uint32_t o[4];
                const int64_t at = static_cast<int64_t>(m) * a.n + col;
                if constexpr (EPI == GemmEpi::kBias) {
                    uint32_t b[4] = {0, 0, 0, 0};
                    const bool has = a.bias != nullptr;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        b[i / 2] |= static_cast<uint32_t>(has ? a.bias[col + i] : 0) << (16 * (i % 2));
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        o[i] = has ? pack2(v[2 * i] + lo_f32(b[i]), v[2 * i + 1] + hi_f32(b[i]))
                                   : pack2(v[2 * i], v[2 * i + 1]);
                    }
                } else {
                    const uint4 rv = *reinterpret_cast<const uint4*>(a.residual + at);
                    const uint32_t res[4] = {rv.x, rv.y, rv.z, rv.w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t h = pack2(v[2 * i], v[2 * i + 1]);
                        o[i] = pack2(lo_f32(res[i]) + lo_f32(h), hi_f32(res[i]) + hi_f32(h));
                    }
                }
                *reinterpret_cast<uint4*>(a.out + at) = make_uint4(o[0], o[1], o[2], o[3]);
            }
        }
        return;
    }
    if constexpr (kPair) {
        constexpr int kRuns = WN * NT * 32 * 2;
        for (int e = tid; e < kRuns; e += kThreads) {
            const int j = e & 1;
            const int tr = (e >> 1) & 31;
            const int t = (e >> 6) % NT;
            const int f = (e >> 6) / NT;
            const int u = n_tile * WN + f;
            const int m = m0 + 32 * t + tr;
            if (m >= M || u >= units) {
                continue;
            }
            float lo[8], hi[8];
            sum8(f, t, j, tr, lo);
            sum8(f, t, j + 2, tr, hi);
            if constexpr (EPI == GemmEpi::kSwiGlu) {
                uint32_t o[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    o[i] = pack2(silu_fixed(lo[2 * i]) * hi[2 * i], silu_fixed(lo[2 * i + 1]) * hi[2 * i + 1]);
                }
                *reinterpret_cast<uint4*>(a.out + static_cast<int64_t>(m) * a.n + static_cast<int64_t>(u) * 16 + 8 * j) =
                    make_uint4(o[0], o[1], o[2], o[3]);
            } else {
                const int64_t n0 = static_cast<int64_t>(u) / 4 * 128;
                const int sg = n0 < a.q_rows ? 0 : (n0 < a.q_rows + a.kv_rows ? 1 : 2);
                const int64_t at = n0 - (sg == 0 ? 0 : (sg == 1 ? a.q_rows : a.q_rows + a.kv_rows));
                const int64_t head = at / 128;
                const int d = u % 4 * 16 + 8 * j;
                const int64_t pos = a.start + m;
                const uint16_t* bias = sg == 0 ? a.seg_bias[0] : (sg == 1 ? a.seg_bias[1] : a.seg_bias[2]);
                uint32_t ol[4], oh[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (bias != nullptr) {
#pragma unroll
                        for (int x = 0; x < 2; ++x) {
                            lo[2 * i + x] = lo[2 * i + x] + Bf16::load(bias[at + d + 2 * i + x]);
                            hi[2 * i + x] = hi[2 * i + x] + Bf16::load(bias[at + d + 64 + 2 * i + x]);
                        }
                    }
                    ol[i] = pack2(lo[2 * i], lo[2 * i + 1]);
                    oh[i] = pack2(hi[2 * i], hi[2 * i + 1]);
                    if (sg < 2) {
                        const float2 cs = *reinterpret_cast<const float2*>(a.rope_cos + pos * 64 + d + 2 * i);
                        const float2 sn = *reinterpret_cast<const float2*>(a.rope_sin + pos * 64 + d + 2 * i);
                        const float l0 = lo_f32(ol[i]), l1 = hi_f32(ol[i]), h0 = lo_f32(oh[i]), h1 = hi_f32(oh[i]);
                        ol[i] = pack2((l0 * cs.x) - (h0 * sn.x), (l1 * cs.y) - (h1 * sn.y));
                        oh[i] = pack2((h0 * cs.x) + (l0 * sn.x), (h1 * cs.y) + (l1 * sn.y));
                    }
                }
                uint16_t* dst = sg == 0 ? a.out + static_cast<int64_t>(m) * a.q_rows + head * 128 + d
                                        : (sg == 1 ? a.kcache : a.vcache) + (head * a.capacity + pos) * 128 + d;
                *reinterpret_cast<uint4*>(dst) = make_uint4(ol[0], ol[1], ol[2], ol[3]);
                *reinterpret_cast<uint4*>(dst + 64) = make_uint4(oh[0], oh[1], oh[2], oh[3]);
            }
        }
    }
}

template <GemmEpi EPI, int WN, int WK, int NT>
hipError_t launch_few(const Nf4GemmArgs& a, int64_t S, hipStream_t stream) {
    const int64_t fragments = EPI == GemmEpi::kSwiGlu ? a.n / 16 : a.n / 32;
    const int64_t m_tiles = gemm_ceil(a.m, 32 * NT);
    const int64_t n_tiles = gemm_ceil(fragments, WN);
    const int64_t steps = a.k / (kWindow * WK);
    hipLaunchKernelGGL((nf4_few_gemm_kernel<EPI, WN, WK, NT>),
                       dim3(static_cast<unsigned>(n_tiles), static_cast<unsigned>(S), static_cast<unsigned>(m_tiles)),
                       dim3(64 * (WN * WK + kLoaders)), 0, stream, a, static_cast<int>(steps / S),
                       static_cast<int>(steps % S));
    const hipError_t status = hipGetLastError();
    if (status != hipSuccess) {
        return status;
    }
    if (S > 1) {
        return launch_nf4_gemm_reduce(EPI, a, S, stream);
    }
    if (EPI == GemmEpi::kResidualNorm && a.norm_gamma != nullptr) {
        PrefillNormArgs na;  // unsplit: the row norm needs every block's columns
        na.x = a.out;
        na.gamma = a.norm_gamma;
        na.eps = a.eps;
        na.out = a.norm_out;
        na.m = a.m;
        return launch_prefill_norm(na, stream);
    }
    return hipSuccess;
}

template <GemmEpi EPI, int WN>
hipError_t launch_few_tokens(const Nf4GemmArgs& a, const GemmPlan& plan, hipStream_t stream) {
    return plan.tokens == 32 ? launch_few<EPI, WN, 4, 1>(a, plan.splits, stream)
                             : launch_few<EPI, WN, 4, 2>(a, plan.splits, stream);
}

// The shapes that gemm_few_plan() gives an epilogue (the 2048 and 2560 rows of the
// row norm and of q, k and v never need three fragments a block).
template <GemmEpi EPI>
hipError_t launch_few_shape(const Nf4GemmArgs& a, const GemmPlan& plan, hipStream_t stream) {
    if (plan.shape == GemmShape::kFew1) {
        return launch_few_tokens<EPI, 1>(a, plan, stream);
    }
    if (plan.shape == GemmShape::kFew2) {
        return launch_few_tokens<EPI, 2>(a, plan, stream);
    }
    if constexpr (EPI != GemmEpi::kResidualNorm && EPI != GemmEpi::kQkvRope) {
        if (plan.shape == GemmShape::kFew3) {
            return launch_few_tokens<EPI, 3>(a, plan, stream);
        }
    }
    if constexpr (EPI == GemmEpi::kSwiGlu) {
        if (plan.shape == GemmShape::kFew3x128) {
            return launch_few<EPI, 3, 2, 4>(a, plan.splits, stream);
        }
    }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_nf4_few_gemm(GemmEpi epi, const Nf4GemmArgs& a, const GemmPlan& plan, hipStream_t stream) {
    switch (epi) {
        case GemmEpi::kBias:
            return launch_few_shape<GemmEpi::kBias>(a, plan, stream);
        case GemmEpi::kResidual:
            return launch_few_shape<GemmEpi::kResidual>(a, plan, stream);
        case GemmEpi::kSwiGlu:
            return launch_few_shape<GemmEpi::kSwiGlu>(a, plan, stream);
        case GemmEpi::kQkvRope:
            return launch_few_shape<GemmEpi::kQkvRope>(a, plan, stream);
        case GemmEpi::kResidualNorm:
            return launch_few_shape<GemmEpi::kResidualNorm>(a, plan, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace kc
