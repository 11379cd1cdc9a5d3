// NF4 GEMM on MFMA for more tokens than one launch of the 64-token kernels
// (kc_prefill.hip) holds: out[m, n] = epilogue(sum_k x[m, k] * w[n, k]),
// w[n, k] = bf16(codebook[code] * absmax), fp32 accumulation in
// v_mfma_f32_32x32x16_bf16.
//
// Work split.  A wave owns RF fragments of 32 weight rows and NT tiles of 32
// tokens; a block holds WN waves along the rows and WK along k (each K-group
// sums its own 64-wide window of every 64 WK k, the groups' sums meet in LDS at
// the end).  Each wave dequantises its own rows straight into the A operand
// registers, so a weight is formed once per block and 32 NT tokens instead of
// once per 64, and never goes back to LDS; x is staged in LDS once per block.
// Per k a wave reads 64 NT bytes of x operands and 4 * 32 RF bytes of table
// entries from LDS for 2 * 32 RF * 32 NT flops: at RF = 2, NT = 4 LDS and
// matrix core would both be busy all the time, at RF = 1 LDS sets the bound at
// two thirds of the matrix rate, above what the card sustains.
//
// Operand layouts of the 32x32x16 bf16 MFMA (lane l, r = l % 32, q = l / 32):
// A[r][8q + j], B[8q + j][r], D[8 (i / 4) + 4q + i % 4][r].  With A = weights
// and B[k][token] = x, lane half q owns the 32 contiguous k of its half of a
// 64-wide window (one 16-byte load of codes, one absmax); step s of the window
// takes k = 32q + 8s + j from both operands, so every k is summed once.
//
// Software pipeline, one 16-k step: each MFMA is followed by one weight pair of
// the next step formed from its table value, the table read of the step after
// it into the registers just freed, and the next step's x operand once the
// current one's last MFMA is issued; scheduling barriers keep these groups
// together (left to the compiler, every operand was read right before its use:
// 607 instead of 663 TFLOP/s at 1999 tokens of gate/up, before the blocks shared a CU).  x of
// window w + 2 is requested while w + 1 is staged, the codes of w + 2 when w's
// are used up; one barrier a window.
//
// What bounds it: two waves a SIMD are needed to keep the matrix core busy (a
// wave alone issues its ~7 instructions per MFMA in about twice the MFMA's
// time), and a block's prologue (table fill, first operands) and epilogue hide
// only behind another block of the CU.  Hence the shapes in kc_gemm_plan.h.
// Measured at 1999 tokens (MI355X, us per call; before = 64-token launches):
// gate/up SwiGLU 621 -> 207 (869 TFLOP/s; silu by hardware exp2 and reciprocal, up
// to 2.7 ulp off where silu_fixed is 2.0, 201; by silu_fixed itself about 215), down
// 519 -> 112 (807), q/k/v rows 340 -> 43 (486).
#include "kc_device.h"
#include "kc_gemm_plan.h"

namespace kc {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kWindow = 64;     // k of one window and K-group: one absmax block

template <int RF>
struct Codes {
    uint4 c[RF];
    float am[RF];
};

// A fragment's packed column pairs of one token (h[2 i4 + e]: columns 8 i4 +
// 4 q + 2 e and the next) as 8 consecutive columns a lane: o[j] holds columns
// 16 j + 8 q .. + 7 (lane halves q exchanged by lane swaps).
__device__ __forceinline__ void rows16(const uint32_t (&h)[8], uint4 (&o)[2]) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const auto s0 = __builtin_amdgcn_permlane32_swap(h[4 * j], h[4 * j + 2], false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(h[4 * j + 1], h[4 * j + 3], false, false);
        o[j] = make_uint4(s0[0], s1[0], s0[1], s1[1]);
    }
}

// bf16(res + v) of 8 pairs of bf16 values
__device__ __forceinline__ uint4 add8(const uint4& r, const uint4& v) {
    return make_uint4(pack2(lo_f32(r.x) + lo_f32(v.x), hi_f32(r.x) + hi_f32(v.x)),
                      pack2(lo_f32(r.y) + lo_f32(v.y), hi_f32(r.y) + hi_f32(v.y)),
                      pack2(lo_f32(r.z) + lo_f32(v.z), hi_f32(r.z) + hi_f32(v.z)),
                      pack2(lo_f32(r.w) + lo_f32(v.w), hi_f32(r.w) + hi_f32(v.w)));
}

// RoPE of two neighbouring dims (l) and their partners 64 dims on (h)
__device__ __forceinline__ void rotate2(uint32_t& l, uint32_t& h, float c0, float c1, float s0, float s1) {
    const float l0 = lo_f32(l), l1 = hi_f32(l), h0 = lo_f32(h), h1 = hi_f32(h);
    l = pack2((l0 * c0) - (h0 * s0), (l1 * c1) - (h1 * s1));
    h = pack2((h0 * c0) + (l0 * s0), (h1 * c1) + (l1 * s1));
}

// (two waves a SIMD; the pair shape's one block of 4 waves a CU has all registers)
template <GemmEpi EPI, int WN, int WK, int RF, int NT>
__global__ __launch_bounds__(64 * WN * WK, WN * RF > 4 || WK * RF < 4 ? 2 : 1) void nf4_tile_gemm_kernel(Nf4GemmArgs a, int m_tiles, int n_tiles, int S) {
    constexpr int kThreads = 64 * WN * WK;
    constexpr int kTokens = 32 * NT;
    constexpr int kChunks = 8 * WK;                        // 16-byte pieces of a token row of one window
    constexpr int kPieces = kTokens * kChunks / kThreads;  // of them, per thread
    constexpr int kXRows = 2 * WK * kTokens;               // staged rows: buffers, K-groups, tokens
    // entry e of the pair table: 16 slots at byte e * 256; staged row i of x
    // (128 bytes) in the other half of entry i's 256 bytes, further rows after the table
    constexpr bool kShare = kXRows <= kNf4PairEntries;
    constexpr int kRowStride = kShare ? 256 : 128;
    constexpr int kTableBytes = kNf4PairEntries * 256;
    constexpr int kSlots = kShare ? 16 : 32;
    constexpr int kGroupBytes = kTokens * kRowStride;
    constexpr int kBufBytes = kGroupBytes * WK;
    constexpr int kAccBytes = WK == 1 ? 0 : WN * RF * NT * 16 * 64 * 4;
    constexpr int kTiles = kShare ? kTableBytes : kTableBytes + 2 * kBufBytes;
    constexpr int kLds = kTiles > kAccBytes ? kTiles : kAccBytes;
    static_assert(kThreads >= kNf4PairEntries && kPieces * kThreads == kTokens * kChunks, "whole pieces");
    __shared__ __attribute__((aligned(256))) uint8_t smem[kLds];
    uint8_t* const s_x = smem + (kShare ? 128 : kTableBytes);
    const SlicedLookup cb{reinterpret_cast<const char*>(smem), (threadIdx.x & (kSlots - 1)) * 8u};
    const float2 pair_entry = pair_entry_fetch();

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN;
    const int g = wave / WN;  // K-group
    const int r = lane & 31;
    const int q = lane >> 5;
    const int64_t K = a.k;
    const int M = static_cast<int>(a.m);
    const int id = static_cast<int>(xcd_contiguous(blockIdx.x, gridDim.x));
    const int split = id / (m_tiles * n_tiles);
    const int tile = id - split * (m_tiles * n_tiles);
    const int n_tile = tile / m_tiles;
    const int m0 = (tile - n_tile * m_tiles) * kTokens;

    // windows of this split
    const int windows = static_cast<int>(K / (kWindow * WK));
    const int per_split = (windows + S - 1) / S;
    const int w_begin = split * per_split;
    const int w_end = w_begin + per_split < windows ? w_begin + per_split : windows;

    // this wave's two 32-row fragments
    const int64_t unit = static_cast<int64_t>(n_tile) * WN + wn;
    int64_t row[RF];  // each fragment's first row in its weight
    int seg[RF];
    int64_t col[RF];  // and first output column
    bool live;
    if constexpr (EPI == GemmEpi::kSwiGlu && RF == 2) {
        // gate and up rows of the same outputs
        const int64_t n0 = unit * 32;
        live = n0 < a.n;
        row[0] = row[1] = live ? n0 : a.n - 32;
        col[0] = col[1] = n0;
        seg[0] = 0;
        seg[1] = 1;
    } else if constexpr (EPI == GemmEpi::kQkvRope && RF == 2) {
        // a head's dims d .. d + 31 and their rotary partners d + 64 ..
        const int64_t n0 = unit / 2 * 128 + unit % 2 * 32;
        live = n0 < a.n;
        const int64_t at = live ? n0 : a.n - 128;
        seg[0] = seg[1] = at < a.q_rows ? 0 : (at < a.q_rows + a.kv_rows ? 1 : 2);
        row[0] = at - (seg[0] == 0 ? 0 : (seg[0] == 1 ? a.q_rows : a.q_rows + a.kv_rows));
        row[1] = row[0] + 64;
        col[0] = n0;
        col[1] = n0 + 64;
    } else {
        const int64_t n0 = unit * 32 * RF;
        live = n0 < a.n;
#pragma unroll
        for (int f = 0; f < RF; ++f) {
            const int64_t at = (live ? n0 : a.n - 32 * RF) + 32 * f;
            col[f] = n0 + 32 * f;
            seg[f] = EPI != GemmEpi::kQkvRope ? 0 : (at < a.q_rows ? 0 : (at < a.q_rows + a.kv_rows ? 1 : 2));
            row[f] = at - (seg[f] == 0 ? 0 : (seg[f] == 1 ? a.q_rows : a.q_rows + a.kv_rows));
        }
    }
    // uniform bases and 32-bit lane offsets (one tile's rows span < 2^31 bytes)
    const uint8_t* wbase[RF];
    const uint8_t* abase[RF];
#pragma unroll
    for (int f = 0; f < RF; ++f) {
        const uint8_t* w = seg[f] == 0 ? a.w[0] : (seg[f] == 1 ? a.w[1] : a.w[2]);
        const float* am = seg[f] == 0 ? a.absmax[0] : (seg[f] == 1 ? a.absmax[1] : a.absmax[2]);
        wbase[f] = w + row[f] * (K / 2) + 32 * g;
        abase[f] = reinterpret_cast<const uint8_t*>(am + row[f] * (K / 64) + g);
    }
    const uint32_t woff = static_cast<uint32_t>(r * (K / 2) + 16 * q);
    const uint32_t aoff = static_cast<uint32_t>(r * (K / 64) * 4);
    const uint8_t* const xbase = reinterpret_cast<const uint8_t*>(a.x + static_cast<int64_t>(m0) * K);
    uint32_t xoff[kPieces];
    uint32_t xdst[kPieces];
#pragma unroll
    for (int j = 0; j < kPieces; ++j) {
        const int e = tid + j * kThreads;
        const int t = e / kChunks;
        const int c = e % kChunks;
        const int tc = m0 + t < M ? t : M - 1 - m0;
        xoff[j] = static_cast<uint32_t>(tc * K * 2 + 16 * c);
        xdst[j] = (c / 8) * kGroupBytes + t * kRowStride + (((c % 8) ^ (t & 7)) * 16);
    }
    typedef uint32_t pieces __attribute__((ext_vector_type(4 * kPieces)));
    pieces xr = {};
    auto x_fetch1 = [&](int j, int w) __attribute__((always_inline)) {
        const uint4 v = *reinterpret_cast<const uint4*>(xbase + static_cast<int64_t>(w) * (kWindow * WK * 2) + xoff[j]);
        xr[4 * j] = v.x;
        xr[4 * j + 1] = v.y;
        xr[4 * j + 2] = v.z;
        xr[4 * j + 3] = v.w;
    };
    auto x_stage1 = [&](int j, int buf) __attribute__((always_inline)) {
        *reinterpret_cast<uint4*>(s_x + buf * kBufBytes + xdst[j]) =
            make_uint4(xr[4 * j], xr[4 * j + 1], xr[4 * j + 2], xr[4 * j + 3]);
    };
    auto w_fetch1 = [&](Codes<RF>& c, int f, int w) __attribute__((always_inline)) {
        c.c[f] = *reinterpret_cast<const uint4*>(wbase[f] + static_cast<int64_t>(w) * (32 * WK) + woff);
        c.am[f] = *reinterpret_cast<const float*>(abase[f] + static_cast<int64_t>(w) * (WK * 4) + aoff);
    };
    uint32_t boff[4];  // this lane's operand piece of step s in a token row
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        boff[s] = g * kGroupBytes + r * kRowStride + (((4 * q + s) ^ (r & 7)) * 16);
    }

    floatx16 acc[RF][NT];
#pragma unroll
    for (int f = 0; f < RF; ++f) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            acc[f][t] = floatx16{};
        }
    }
    const int last = w_end - 1;
    auto clamp_w = [&](int w) { return w < last ? w : last; };
    Codes<RF> c0, c1;
#pragma unroll
    for (int j = 0; j < kPieces; ++j) {
        x_fetch1(j, w_begin);
    }
#pragma unroll
    for (int f = 0; f < RF; ++f) {
        w_fetch1(c0, f, w_begin);
    }
#pragma unroll
    for (int j = 0; j < kPieces; ++j) {
        x_stage1(j, 0);
    }
    if (tid < kNf4PairEntries) {
#pragma unroll
        for (int j = 0; j < kSlots; ++j) {
            *reinterpret_cast<float2*>(smem + tid * 256 + ((j + tid) & (kSlots - 1)) * 8) = pair_entry;
        }
    }
#pragma unroll
    for (int j = 0; j < kPieces; ++j) {
        x_fetch1(j, clamp_w(w_begin + 1));
    }
#pragma unroll
    for (int f = 0; f < RF; ++f) {
        w_fetch1(c1, f, clamp_w(w_begin + 1));
    }
    __syncthreads();
    float2 p[4 * RF];  // table values: unit u = byte u % 4 of fragment u / 4
    bf16x8 A0[RF], A1[RF];
    uint4 B[NT];
    auto look = [&](int u, const Codes<RF>& c, int s) __attribute__((always_inline)) {
        const uint32_t w = word_of(c.c[u / 4], s);
        p[u] = u % 4 == 0 ? *cb.template entry<0>(w)
                          : (u % 4 == 1 ? *cb.template entry<1>(w)
                                        : (u % 4 == 2 ? *cb.template entry<2>(w) : *cb.template entry<3>(w)));
    };
    auto form = [&](int u, bf16x8 (&A)[RF], const Codes<RF>& c) __attribute__((always_inline)) {
        A[u / 4][2 * (u % 4)] = static_cast<__bf16>(p[u].x * c.am[u / 4]);
        A[u / 4][2 * (u % 4) + 1] = static_cast<__bf16>(p[u].y * c.am[u / 4]);
    };
    auto b_read = [&](int t, int bb, int sb) __attribute__((always_inline)) {
        B[t] = *reinterpret_cast<const uint4*>(s_x + bb * kBufBytes + t * 32 * kRowStride + boff[sb]);
    };
#pragma unroll
    for (int u = 0; u < 4 * RF; ++u) {
        look(u, c0, 0);
    }
#pragma unroll
    for (int u = 0; u < 4 * RF; ++u) {
        form(u, A0, c0);
        look(u, c0, 1);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        b_read(t, 0, 0);
    }
    int buf = 0;
    int w = w_begin;
    // One 16-k step of 2 NT MFMAs.  Between them, a few instructions each so
    // that they issue while the matrix core works: the next step's weights An
    // are formed from their table values, each value's registers then request
    // the step after that (codes cl, step sl), and each x operand is replaced by
    // the next step's as soon as its last MFMA is issued.
    auto step = [&](const bf16x8 (&A)[RF], bf16x8 (&An)[RF], const Codes<RF>& cl, int sl, const Codes<RF>& cn, int bb, int sb,
                    auto&& extra) __attribute__((always_inline)) {
        constexpr int kSteps = RF * NT;
        constexpr int kUnits = 4 * RF / kSteps;
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            const int t = i / RF;
            const int f = i % RF;
            acc[f][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[f], __builtin_bit_cast(bf16x8, B[t]), acc[f][t], 0, 0,
                                                                0);
#pragma unroll
            for (int u = i * kUnits; u < (i + 1) * kUnits; ++u) {
                form(u, An, cn);
                look(u, cl, sl);
            }
            if (f == RF - 1) {
                b_read(t, bb, sb);
            }
            extra(i, kSteps);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto none = [](int, int) __attribute__((always_inline)) {};
    auto window = [&](Codes<RF>& cur, const Codes<RF>& next) __attribute__((always_inline)) {
        const int w2 = clamp_w(w + 2);
        step(A0, A1, cur, 2, cur, buf, 1, none);
        step(A1, A0, cur, 3, cur, buf, 2, [&](int i, int n) __attribute__((always_inline)) {
#pragma unroll
            for (int j = i * kPieces / n; j < (i + 1) * kPieces / n; ++j) {
                x_stage1(j, buf ^ 1);
                x_fetch1(j, w2);
            }
        });
        step(A0, A1, next, 0, cur, buf, 3, none);
        __syncthreads();
        step(A1, A0, next, 1, next, buf ^ 1, 0, [&](int i, int n) __attribute__((always_inline)) {
            if (i % (n / RF) == 0) {
                w_fetch1(cur, i / (n / RF), w2);
            }
        });
        buf ^= 1;
        ++w;
    };
    while (true) {
        window(c0, c1);
        if (w >= w_end) break;
        window(c1, c0);
        if (w >= w_end) break;
    }
    __syncthreads();

    // the K-groups' sums: each group finishes its share of the token tiles and
    // hands the other share over through LDS (free since the loop's last barrier)
    constexpr int kFin = NT / WK;
    floatx16 fin[RF][kFin];
    if constexpr (WK == 1) {
#pragma unroll
        for (int f = 0; f < RF; ++f) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                fin[f][t] = acc[f][t];
            }
        }
    } else {
        float4* const s_acc = reinterpret_cast<float4*>(smem);
#pragma unroll
        for (int f = 0; f < RF; ++f) {
#pragma unroll
            for (int t = 0; t < kFin; ++t) {
                const floatx16 give = g == 0 ? acc[f][kFin + t] : acc[f][t];
                fin[f][t] = g == 0 ? acc[f][t] : acc[f][kFin + t];
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    s_acc[((wave * RF + f) * kFin + t) * 256 + i4 * 64 + lane] =
                        make_float4(give[4 * i4], give[4 * i4 + 1], give[4 * i4 + 2], give[4 * i4 + 3]);
                }
            }
        }
        __syncthreads();
        const int other = wn + (g ^ 1) * WN;
#pragma unroll
        for (int f = 0; f < RF; ++f) {
#pragma unroll
            for (int t = 0; t < kFin; ++t) {
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    const float4 v = s_acc[((other * RF + f) * kFin + t) * 256 + i4 * 64 + lane];
                    fin[f][t][4 * i4] += v.x;
                    fin[f][t][4 * i4 + 1] += v.y;
                    fin[f][t][4 * i4 + 2] += v.z;
                    fin[f][t][4 * i4 + 3] += v.w;
                }
            }
        }
    }
    if (!live) {
        return;
    }
    const int mf = m0 + 32 * kFin * g;  // first token of this wave's share
    // D row 8 i4 + 4 q + e (e = 0..3) of a fragment, column r: four consecutive
    // output columns a lane
    if (S > 1) {
#pragma unroll
        for (int t = 0; t < kFin; ++t) {
            const int m = mf + 32 * t + r;
            if (m < M) {
#pragma unroll
                for (int f = 0; f < RF; ++f) {
                    const int64_t plane = EPI == GemmEpi::kSwiGlu ? static_cast<int64_t>(f) * S + split : split;
                    float* dst = a.partials + (plane * M + m) * a.n + col[f] + 4 * q;
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        *reinterpret_cast<float4*>(dst + 8 * i4) =
                            make_float4(fin[f][t][4 * i4], fin[f][t][4 * i4 + 1], fin[f][t][4 * i4 + 2],
                                        fin[f][t][4 * i4 + 3]);
                    }
                }
            }
        }
        return;
    }
    if constexpr (RF == 1 && EPI == GemmEpi::kQkvRope) {
        return;  // split only: the rotation needs both fragments
    } else if constexpr (EPI == GemmEpi::kSwiGlu) {
#pragma unroll
        for (int t = 0; t < kFin; ++t) {
            const int m = mf + 32 * t + r;
            uint32_t h[8];
            float far = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                far = fmaxf(far, fabsf(fin[0][t][i]));
            }
            if (__any(far >= kSiluNear)) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    h[i] = pack2(silu_fixed(fin[0][t][2 * i]) * fin[1][t][2 * i],
                                 silu_fixed(fin[0][t][2 * i + 1]) * fin[1][t][2 * i + 1]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    h[i] = pack2(silu_near(fin[0][t][2 * i]) * fin[1][t][2 * i],
                                 silu_near(fin[0][t][2 * i + 1]) * fin[1][t][2 * i + 1]);
                }
            }
            uint4 o[2];
            rows16(h, o);
            if (m < M) {
                uint16_t* dst = a.out + static_cast<int64_t>(m) * a.n + col[0] + 8 * q;
                *reinterpret_cast<uint4*>(dst) = o[0];
                *reinterpret_cast<uint4*>(dst + 16) = o[1];
            }
        }
    } else if constexpr (EPI == GemmEpi::kResidual || EPI == GemmEpi::kResidualNorm) {
#pragma unroll
        for (int t = 0; t < kFin; ++t) {
            const int m = mf + 32 * t + r;
            const int64_t at = static_cast<int64_t>(m < M ? m : M - 1) * a.n + col[0] + 8 * q;
            uint4 res[RF][2];
#pragma unroll
            for (int f = 0; f < RF; ++f) {
                res[f][0] = *reinterpret_cast<const uint4*>(a.residual + at + 32 * f);
                res[f][1] = *reinterpret_cast<const uint4*>(a.residual + at + 32 * f + 16);
            }
#pragma unroll
            for (int f = 0; f < RF; ++f) {
                uint32_t h[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    h[i] = pack2(fin[f][t][2 * i], fin[f][t][2 * i + 1]);
                }
                uint4 o[2];
                rows16(h, o);
                if (m < M) {
                    *reinterpret_cast<uint4*>(a.out + at + 32 * f) = add8(res[f][0], o[0]);
                    *reinterpret_cast<uint4*>(a.out + at + 32 * f + 16) = add8(res[f][1], o[1]);
                }
            }
        }
    } else {
        // bias of this lane's columns: the same for every token
        const bool rope = EPI == GemmEpi::kQkvRope;
        const int64_t head = row[0] / 128;
        const int d = static_cast<int>(row[0] % 128);  // 0 or 32; the partner fragment at d + 64
        const uint16_t* bias = a.bias;
        int64_t bcol = col[0];
        if constexpr (rope) {
            bias = a.seg_bias[0];
            bias = seg[0] == 1 ? a.seg_bias[1] : bias;
            bias = seg[0] == 2 ? a.seg_bias[2] : bias;
            bcol = row[0];
        }
        float bv[RF][16] = {};
        if (bias != nullptr) {
#pragma unroll
            for (int f = 0; f < RF; ++f) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    bv[f][i] = Bf16::load(bias[bcol + (rope ? 64 : 32) * f + 8 * (i / 4) + 4 * q + i % 4]);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < kFin; ++t) {
            const int m = mf + 32 * t + r;
            const int mc = m < M ? m : M - 1;
            uint32_t h[RF][8];
#pragma unroll
            for (int f = 0; f < RF; ++f) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    float v0 = fin[f][t][2 * i];
                    float v1 = fin[f][t][2 * i + 1];
                    if (bias != nullptr) {
                        v0 = v0 + bv[f][2 * i];
                        v1 = v1 + bv[f][2 * i + 1];
                    }
                    h[f][i] = pack2(v0, v1);
                }
            }
            uint16_t* dst;
            int64_t step_f;
            if constexpr (rope) {
                const int64_t pos = a.start + mc;
                if (seg[0] < 2) {
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        const float4 cs = *reinterpret_cast<const float4*>(a.rope_cos + pos * 64 + d + 8 * i4 + 4 * q);
                        const float4 sn = *reinterpret_cast<const float4*>(a.rope_sin + pos * 64 + d + 8 * i4 + 4 * q);
                        rotate2(h[0][2 * i4], h[1][2 * i4], cs.x, cs.y, sn.x, sn.y);
                        rotate2(h[0][2 * i4 + 1], h[1][2 * i4 + 1], cs.z, cs.w, sn.z, sn.w);
                    }
                }
                dst = seg[0] == 0 ? a.out + static_cast<int64_t>(mc) * a.q_rows + head * 128 + d
                                  : (seg[0] == 1 ? a.kcache : a.vcache) + (head * a.capacity + pos) * 128 + d;
                step_f = 64;
            } else {
                dst = a.out + static_cast<int64_t>(mc) * a.n + col[0];
                step_f = 32;
            }
#pragma unroll
            for (int f = 0; f < RF; ++f) {
                uint4 o[2];
                rows16(h[f], o);
                if (m < M) {
                    *reinterpret_cast<uint4*>(dst + f * step_f + 8 * q) = o[0];
                    *reinterpret_cast<uint4*>(dst + f * step_f + 8 * q + 16) = o[1];
                }
            }
        }
    }
}

template <GemmEpi EPI, int WN, int WK, int RF, int NT>
hipError_t launch_tile(const Nf4GemmArgs& a, int64_t S, hipStream_t stream) {
    constexpr bool kPairs = EPI == GemmEpi::kSwiGlu && RF == 2;  // gate and up rows share a tile
    constexpr int64_t kRows = (kPairs ? 32 : 32 * RF) * WN;
    const int64_t m_tiles = gemm_ceil(a.m, 32 * NT);
    const int64_t n_tiles = gemm_ceil(a.n, kRows);
    hipLaunchKernelGGL((nf4_tile_gemm_kernel<EPI, WN, WK, RF, NT>), dim3(static_cast<unsigned>(m_tiles * n_tiles * S)),
                       dim3(64 * WN * WK), 0, stream, a, static_cast<int>(m_tiles), static_cast<int>(n_tiles),
                       static_cast<int>(S));
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

// The shapes that gemm_tile_plan() gives an epilogue.
template <GemmEpi EPI>
hipError_t launch_shape(const Nf4GemmArgs& a, const GemmPlan& plan, hipStream_t stream) {
    constexpr bool kPairEpi = EPI == GemmEpi::kSwiGlu || EPI == GemmEpi::kQkvRope;
    if (plan.shape == GemmShape::kWide) {
        return launch_tile<EPI, 4, 1, 2, 4>(a, plan.splits, stream);
    }
    if constexpr (kPairEpi) {
        if (plan.shape == GemmShape::kPair) {
            return launch_tile<EPI, 2, 2, 2, 4>(a, plan.splits, stream);
        }
    } else {
        if (plan.shape == GemmShape::kLow) {
            return launch_tile<EPI, 4, 2, 1, 2>(a, plan.splits, stream);
        }
    }
    if constexpr (EPI != GemmEpi::kSwiGlu) {
        if (plan.shape == GemmShape::kSquare) {
            return launch_tile<EPI, 4, 2, 1, 4>(a, plan.splits, stream);
        }
    }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_nf4_tile_gemm(GemmEpi epi, const Nf4GemmArgs& a, const GemmPlan& plan, hipStream_t stream) {
    switch (epi) {
        case GemmEpi::kBias:
            return launch_shape<GemmEpi::kBias>(a, plan, stream);
        case GemmEpi::kResidual:
            return launch_shape<GemmEpi::kResidual>(a, plan, stream);
        case GemmEpi::kSwiGlu:
            return launch_shape<GemmEpi::kSwiGlu>(a, plan, stream);
        case GemmEpi::kQkvRope:
            return launch_shape<GemmEpi::kQkvRope>(a, plan, stream);
        case GemmEpi::kResidualNorm:
            return launch_shape<GemmEpi::kResidualNorm>(a, plan, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace kc
