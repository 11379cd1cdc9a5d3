// Which kernel takes an NF4 GEMM of several tokens, in which block shape and over
// how many splits of K.  Plain host arithmetic on sizes, types and alignment.
#pragma once

#include "kc_kernels.h"

namespace kc {

enum class GemmShape {
    kParts,    // kc_prefill.hip: launches of up to kGemmMaxTokens tokens
    kFew1,     // kc_gemm_few.hip: 1, 2 or 3 fragments of 32 rows, four K-groups, 32 or 64 tokens
    kFew2,
    kFew3,
    kFew3x128, // three fragments, two K-groups, 128 tokens
    kLow,      // kc_gemm.hip: 128 rows x 64 tokens, 8 waves of one fragment in two K-groups, one block a CU
    kSquare,   // 128 x 128, the same waves
    kPair,     // 128 x 128, 4 waves of two fragments in two K-groups, one block a CU
    kWide,     // 256 x 128, 4 waves, two blocks a CU
};
struct GemmPlan {
    GemmShape shape = GemmShape::kParts;
    int64_t tokens = kGemmMaxTokens;  // of a block
    int64_t splits = 1;               // of K (kParts: its launcher splits)
};

constexpr int64_t kGemmChip = 256;      // blocks that fill the chip, one a CU
constexpr int64_t kGemmLongK = 4096;    // above it a k is long: see gemm_few_plan() and gemm_tile_plan()

inline int64_t gemm_ceil(int64_t a, int64_t b) { return (a + b - 1) / b; }

// At most `want` splits of `steps` steps of K, as far as the fp32 partial tiles
// (gate and up each have theirs) fit the scratch.
inline int64_t gemm_splits(GemmEpi epi, const Nf4GemmArgs& a, int64_t want, int64_t steps) {
    const int64_t planes = epi == GemmEpi::kSwiGlu ? 2 : 1;
    const int64_t fit = a.partial_floats / (planes * a.m * a.n);
    int64_t s = want < steps ? want : steps;
    s = s < fit ? s : fit;
    return s > 1 ? s : 1;
}

// Both kernels read and write 16-byte pieces of aligned rows (n and k are multiples
// of 64 and 128); a tile's lane offsets and the grid fit 32 bits.
inline bool gemm_whole_pieces(GemmEpi epi, const Nf4GemmArgs& a) {
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    if (a.m < 1 || a.m > (int64_t{1} << 24) || a.n < 64 || a.n % 64 != 0 || a.n > (int64_t{1} << 24) || a.k < 128 ||
        a.k % 128 != 0 || a.k > (int64_t{1} << 22) || a.m * a.n > (int64_t{1} << 40) || a.partials == nullptr) {
        return false;
    }
    bool ok = aligned(a.x) && aligned(a.out) && aligned(a.w[0]) && aligned(a.partials);
    if (epi == GemmEpi::kResidual || epi == GemmEpi::kResidualNorm) {
        ok = ok && a.residual != nullptr && aligned(a.residual);
    }
    if (epi == GemmEpi::kSwiGlu || epi == GemmEpi::kQkvRope) {
        ok = ok && aligned(a.w[1]);
    }
    if (epi == GemmEpi::kQkvRope) {
        ok = ok && aligned(a.w[2]) && aligned(a.rope_cos) && aligned(a.rope_sin) && aligned(a.kcache) &&
             aligned(a.vcache) && a.q_rows % 128 == 0 && a.kv_rows % 128 == 0;
    }
    return ok && (epi != GemmEpi::kResidualNorm || a.n == 2048);
}

// Few tokens: whole steps of four windows, and one round of blocks where there are
// more than 64 tokens.  That reaches 384 tokens for q, k and v at once, 512 for
// o_proj, 256 for down, 128 for gate/up; a narrow weight's blocks still make one
// round at thousands.  us per call in this kernel / in the tile kernel:
//   tokens         65           128          256          384          512
//   q  (2048 rows) 8.8 / 12.0   9.0 / 14.6   9.4 / 15.1   11.6 / 18.0  11.6 / 19.2
//   qkv (2560)     8.7 / 12.8   8.9 / 14.6   11.1 / 16.4  11.4 / 19.2
//   down           17.5 / 19.7  19.7 / 22.3  27.6 / 30.1
//   gate/up        21.3 / 25.5  22.4 / 25.8  (129: 39.0 / 38.9)
//   256 rows       7.9 / 9.4    8.0 / 9.8    9.0 / 10.8   (1024: 9.1 / 13.5, 2048: 13.2 / 14.9)
// Past what was looked for: 256 rows at 4096 tokens take 21.7 here, 17.6 there, 64
// rows at 8192 tokens 16.3 and 14.5.
inline GemmPlan gemm_few_plan(GemmEpi epi, const Nf4GemmArgs& a) {
    const bool swiglu = epi == GemmEpi::kSwiGlu;
    GemmPlan p;
    if (a.k % 256 != 0) {
        return p;
    }
    const int64_t fragments = swiglu ? a.n / 16 : a.n / 32;
    const int64_t two = gemm_ceil(fragments, 2);
    const int64_t tiles = a.m <= 32 ? 1 : gemm_ceil(a.m, 64);
    if (a.m > 64 && two * tiles > (a.k > kGemmLongK && !swiglu ? kGemmChip / 2 : kGemmChip)) {
        // gate/up of 65 .. 128 tokens: each weight formed once for all of them (two
        // 64-token tiles of three fragments 31.5 us, this 22.3)
        if (swiglu && a.m <= 128 && gemm_ceil(fragments, 3) <= kGemmChip) {
            p = {GemmShape::kFew3x128, 128, 1};
        }
        return p;
    }
    if (a.m <= 16 && fragments >= 2 * kGemmChip && a.k <= (fragments > 2 * kGemmChip ? 1024 : 768)) {
        // all CUs full of two or three fragments and little k: the blocks' table and sums
        // cost more than in kParts (gate/up of 1 token, 11008 rows: k 256 7.6 / 5.3 us, 512
        // 8.7 / 6.6, 1024 10.6 / 9.1, 1536 even)
        return p;
    }
    p.tokens = a.m <= 32 ? 32 : 64;
    const int64_t steps = a.k / 256;
    const int64_t blocks = fragments * tiles;  // of one fragment
    const bool few_blocks = blocks <= kGemmChip / 8;
    if (a.k > kGemmLongK && !few_blocks && two * tiles <= kGemmChip) {
        // a long k (down) over many blocks: two fragments a block and K over the chip (gate/up
        // of 1024 rows, k 11008, 33 tokens: unsplit 29.8 us, 64-token launches 16.6, this 15)
        p.shape = GemmShape::kFew2;
        p.splits = gemm_splits(epi, a, kGemmChip / (two * tiles), steps);
    } else if (blocks <= kGemmChip) {
        // A step of 256 costs 0.45 us (64 tokens 0.63), a split's partial tiles and reduce
        // launch about 2: K is split past 2048 (2048 rows of 64 tokens, k 4096: 13.3 -> 10.5
        // us, k 2048 8.3 -> 9.2) and, where few blocks leave most of the chip idle, from
        // 1792 (1024 rows, k 2048: 6.9 in two splits, 6.1 in eight; k 1024 6.1 in two, 4.6
        // unsplit).  Splits of one step only up to eight, sixteen at most: their planes cost
        // the reduce (gate/up of 128 rows, k 4096: 8 splits 15 % faster than 16).  A row
        // norm needs a second launch either way, so o_proj splits over the whole chip and
        // norms in its reduce (prefill of 9 layers, us, unsplit -> split: 1 token 505 ->
        // 487, 16 511 -> 490, 48 629 -> 594, 64 643 -> 616)
        p.shape = GemmShape::kFew1;
        if (epi == GemmEpi::kResidualNorm || a.k > 2048 || (a.k > 1536 && few_blocks)) {
            const int64_t most = steps < 16 ? 8 : (steps < 32 ? steps / 2 : 16);
            p.splits = gemm_splits(epi, a, kGemmChip / blocks < most ? kGemmChip / blocks : most, steps);
        }
    } else {
        p.shape = two * tiles <= kGemmChip ? GemmShape::kFew2 : GemmShape::kFew3;
    }
    return p;
}

// The tile kernel's shapes, each with the number of blocks that fill the chip;
// measured on one box (us per call, q = 2560 rows of k 2048, down = 2048 rows of k
// 11008, gate/up = 2 x 11008 rows of k 2048; the columns from 512 on reach here
// with k a multiple of 256, gate/up from 129 tokens and down from 257):
//   tokens            256   512  1024  1999
//   q      wide      26.4  31.2  41.8  43.1
//          square    22.9  25.6  26.5  49.1
//          pair      24.2  27.3  28.3  52.7
//          low       18.7  18.7  31.1  48.3
//   down   wide      38.6  56.5  92.3   163
//          square    31.4  42.4  68.8   114
//          low       30.7  48.9  80.7   155
//   gate/up wide     39.1  65.7   112   207
//           pair     47.4  70.8   144   274
// One fragment a wave cannot hold a gate/up or rotary pair: those epilogues run
// in the split reduce, or in the wide and pair shapes.
inline GemmPlan gemm_tile_plan(GemmEpi epi, const Nf4GemmArgs& a) {
    const auto tiles = [&](int64_t rows, int64_t tokens) { return gemm_ceil(a.n, rows) * gemm_ceil(a.m, tokens); };
    // `blocks` of `rows` rows fill the chip; a step is `windows` windows of 64; no empty split
    const auto plan = [&](GemmShape shape, int64_t rows, int64_t tokens, int64_t blocks, int64_t windows) {
        const int64_t steps = a.k / (64 * windows);
        const int64_t s = gemm_splits(epi, a, blocks / tiles(rows, tokens), steps);
        return GemmPlan{shape, tokens, gemm_ceil(steps, gemm_ceil(steps, s))};
    };
    const int64_t square = tiles(128, 128);
    if (epi == GemmEpi::kSwiGlu) {
        // below half the chip in wide blocks twice as many narrower ones
        return square < kGemmChip / 2 ? plan(GemmShape::kPair, 64, 128, kGemmChip, 2)
                                      : plan(GemmShape::kWide, 128, 128, 2 * kGemmChip, 1);
    }
    if (square > kGemmChip) {
        // a second, mostly empty round of 128 x 128 blocks costs more than fewer, larger blocks
        return plan(GemmShape::kWide, 256, 128, 2 * kGemmChip, 1);
    }
    if (epi == GemmEpi::kQkvRope) {
        // the rotation is in the reduce (two splits or more) or in blocks that hold pairs
        const GemmPlan p = plan(GemmShape::kSquare, 128, 128, kGemmChip, 2);
        return p.splits > 1 ? p : plan(GemmShape::kPair, 128, 128, kGemmChip, 2);
    }
    // few tokens; or a short k in one unsplit round (no partial tiles, no reduce launch)
    return a.m <= 256 || (a.k <= kGemmLongK && tiles(128, 64) <= kGemmChip)
               ? plan(GemmShape::kLow, 128, 64, kGemmChip, 2)
               : plan(GemmShape::kSquare, 128, 128, kGemmChip, 2);
}

// Few tokens (up to 64, more where they still make one round of its blocks) go
// through kc_gemm_few.hip, more through kc_gemm.hip, which forms each weight once per
// 64 or 128 tokens in one launch.  Calls that neither can take (unaligned buffers; k
// no multiple of 256 at up to 64 tokens) go in launches of kGemmMaxTokens rows, whose
// waves keep a 16-row fragment for all of them.
inline GemmPlan gemm_plan(GemmEpi epi, const Nf4GemmArgs& a) {
    if (!gemm_whole_pieces(epi, a)) {
        return GemmPlan{};
    }
    const GemmPlan p = gemm_few_plan(epi, a);
    return p.shape != GemmShape::kParts || a.m <= kGemmMaxTokens ? p : gemm_tile_plan(epi, a);
}

}  // namespace kc
