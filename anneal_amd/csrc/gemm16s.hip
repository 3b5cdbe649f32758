// gemm16s.hip — which f16 contractions the split kernel (gemm16s_cfg.hip) serves, and with which tile and split.
#include "gemm16s.h"

namespace ah {

static bool operand_ok(const void *p, long ld, int t, int rows, int K) {
    if (((uintptr_t)p & 15) || ld % 8) return false;
    if ((t == 0 ? K : rows) % 8) return false;   // the contiguous dimension, in 16-byte loads
    // offsets are 32-bit: the operand, and a stage of 128 rows (or k-rows) of it, stay under 2 GiB
    const long bytes = (t == 0 ? (long)rows * ld : (long)K * ld) * 2;
    return bytes < (1L << 31) && 128 * ld * 2 < (1L << 31);
}

static hipError_t launch_cfg(const GemmDesc &d, const G16SPlan &p, hipStream_t s) {
    switch (p.cfg) {
        case 0: return gemm16s_launch_0(d, p, s);
        case 1: return gemm16s_launch_1(d, p, s);
        case 2: return gemm16s_launch_2(d, p, s);
        case 3: return gemm16s_launch_3(d, p, s);
        case 4: return gemm16s_launch_4(d, p, s);
        case 5: return gemm16s_launch_5(d, p, s);
        case 6: return gemm16s_launch_6(d, p, s);
        case 7: return gemm16s_launch_7(d, p, s);
        default: return gemm16s_launch_8(d, p, s);
    }
}

// Time of a launch in microseconds, as measured: base + load * (stage * stages + tile[epilogue]) + fold * split (the last
// term with K split only), load being how long a CU's share of the workgroups takes against one: workgroups that fill a CU
// run one after another, of those that share it a second one costs `second` - 1 more, and small ones keep adding that.
// Fitted to 213 shapes (M, N, K from 1 to 8192, the three layouts with their layer epilogues, K split 1 to 12 ways, random
// operands rotating through memory) within 8-11% (0.17 for the 256x256 tile, whose overhang varies most); the choice it
// makes is on average 2.9% slower than the best of all configurations, and 1.63 times faster than the whole-tile variants
// and the register-staged kernel it replaces on the 141 of them that the rule below sends here.
struct Cost {
    float base, stage, second, fold, tile[3];   // tile: store and bias, ReLU mask, SGD
    int share;                                  // workgroups that share a CU: 1, 2, or more (3)
};
static constexpr Cost kCost[kG16SConfigs] = {
    {1.00f, 0.41f, 2.00f, 1.91f, {8.1f, 12.8f, 11.6f}, 1},   // 128x128, two wave sets, 4 stages
    {2.96f, 0.37f, 1.66f, 1.49f, {3.4f, 5.2f, 4.5f}, 2},     // 64x128
    {3.24f, 0.27f, 1.64f, 0.65f, {1.9f, 2.6f, 3.1f}, 2},     // 64x64
    {3.63f, 0.35f, 1.75f, 0.60f, {1.6f, 2.2f, 2.6f}, 2},     // 32x64, four wave sets, 128 of K per stage
    {2.98f, 0.36f, 1.61f, 1.42f, {3.4f, 5.3f, 5.2f}, 2},     // 128x64
    {1.00f, 1.35f, 2.00f, 0.00f, {13.3f, 21.5f, 19.6f}, 1},  // 256x256, never split
    {1.00f, 0.62f, 1.58f, 3.72f, {5.5f, 9.5f, 9.8f}, 2},     // 128x128, one wave set, 2 stages
    {1.00f, 0.54f, 1.49f, 2.02f, {3.6f, 5.4f, 5.8f}, 3},     // 64x128, likewise: short K
    {1.00f, 0.44f, 1.34f, 1.03f, {2.9f, 3.7f, 4.4f}, 3},     // 64x64, likewise
};
constexpr int kCUs = 256, kMaxWorkgroups = 1024;   // workgroups beyond which a further split only adds partials

static bool choose(const GemmDesc &d, G16SPlan *best) {
    const int ep = d.epi == EPI_MASK ? 1 : d.epi == EPI_SGD ? 2 : 0;
    const bool ws = d.sk_sync && d.sk_part;
    float low = 1e30f;
    for (int c = 0; c < kG16SConfigs; c++) {
        const G16SCfg &t = kG16SCfg[c];
        const Cost &k = kCost[c];
        const long tiles = (long)((d.M + t.bm - 1) / t.bm) * ((d.N + t.bn - 1) / t.bn);
        const int nk = (d.K + t.bk - 1) / t.bk;
        for (int want : {1, 2, 3, 4, 6, 8, 12}) {
            if (want > nk || (want > 1 && (!ws || k.fold == 0.0f || tiles * want > kMaxWorkgroups))) break;
            const int stages = (nk + want - 1) / want, split = (nk + stages - 1) / stages;   // no split without a stage
            if (split > 1 && (tiles > kSplitKMaxTiles || tiles * split * t.bm * t.bn > d.sk_cap)) break;
            const long q = (tiles * split + kCUs - 1) / kCUs;   // workgroups of the fullest CU
            const float load = k.share == 1 ? (float)q : k.share == 2 ? (float)(q / 2) * k.second + (float)(q % 2)
                                                                     : 1.0f + (float)(q - 1) * (k.second - 1.0f);
            const float us = k.base + load * (k.stage * (float)stages + k.tile[ep]) + (split > 1 ? k.fold * (float)split : 0.0f);
            if (us < low) {
                low = us;
                *best = {c, split, stages};
            }
        }
    }
    return low < 1e30f;
}

// Where the line lies. The whole-tile variants keep the outputs whose tiles they fill whole (256x256 where those number at
// least 224, else 128x128; K a multiple of 64) from 64 128x128 tiles up: 2048 x 1024 x 2048 21.7 / 21.9 / 24.3 us there
// against 19.9 / 23.2 / 24.0 here (NT / N,MN / MN,MN), 2048 x 2048 x 2048 24.5 / 25.2 / 30.9 against 27.4 / 32.3 / 32.0,
// 4096 x 4096 x 2048 62 / 68 / 105 against 75 / 88 / 104. (Between 64 and 96 tiles this kernel is the faster one, 1024 x 1024 x
// 2048 16.0 / 17.3 / 17.7 us against 21.2 / 21.3 / 23.2. They stay there so that a BEAM search over a key of 64 tiles and more
// has candidates: it takes only kernels that add K in the open key's order, and none adds it in this one's.)
//
// They also keep ragged outputs whose epilogue reads no matrix, as only the edge tiles then store element by element; with a
// mask or SGD epilogue they take 1.1 to 2 times as long as this kernel.
//  - Both operands along K (NT): over 272 tiles on average 1.13 times faster (0.92 to 1.36, 75 shapes: 3584 x 7040 x 128 22.8
//    us there against 31.1, 6709 x 6656 x 320 58.8 against 71.7, 905 x 5120 x 1088 21.9 against 27.4), over 192 tiles up to
//    K = 1280 (923 x 3840 x 128 7.2 against 9.0), over 128 with K from 384 (3477 x 768 x 640 12.7 against 14.8). With fewer
//    tiles or a longer K splitting K gains, and past K = 512 with 257 to 272 tiles, which variant 1 puts one to nearly every
//    CU with two stages in flight (3769 x 1056 x 896 18.1 against 16.6; 727 x 5512 x 320 11.5 against 15.1).
//  - The other layouts: over 192 tiles up to K = 192, 257 to 400 up to K = 1280, each 1.05 to 1.16 times faster on average
//    over 48 shapes (3904 x 1280 x 256 N,MN 10.3 against 12.5); beyond, 0.77 to 1.02 times.
static bool whole_tiles(const GemmDesc &d, long t128) {
    if (d.K % 64 || d.epi == EPI_MASK || d.epi == EPI_SGD) return false;
    if (d.ta || d.tb) return t128 > 192 && (d.K <= 192 || (t128 > 256 && t128 <= 400 && d.K <= 1280));
    if (t128 > 256) return t128 > 272 || d.K <= 512;
    return d.K <= 1280 && (t128 > 192 || (t128 > 128 && d.K >= 384));
}
// A K of less than two stages that 64 does not divide goes to the register-staged kernel's 64x64 tiles from 65 to 192 128x128
// ones (NT, likewise): 256 x 5696 x 32 4.6 us there against 5.7, 1044 x 1088 x 56 5.1 against 6.0, 2014 x 1816 x 104 on even, 1.12
// times faster over 45 shapes; with fewer or more tiles the two are within 3%.
static bool register_staged(const GemmDesc &d, long t128) {
    return !d.ta && !d.tb && d.epi != EPI_MASK && d.epi != EPI_SGD && d.K < 128 && d.K % 64 && t128 > 64 && t128 <= 192;
}

bool gemm16s_serves(const GemmDesc &d) {
    if (d.dtype != GEMM_F16 || d.K <= 0 || d.epi == EPI_MSE || d.colsum || d.A2 || d.C2 || (d.ta && !d.tb)) return false;
    if (d.tile || d.variant || d.splits || d.kgroups) return false;   // the caller's choice of kernel
    if (!operand_ok(d.A, d.lda, d.ta, d.M, d.K) || !operand_ok(d.B, d.ldb, d.tb, d.N, d.K)) return false;
    const long t256 = (long)((d.M + 255) / 256) * ((d.N + 255) / 256), t128 = (long)((d.M + 127) / 128) * ((d.N + 127) / 128);
    const int tile = t256 >= 224 ? 256 : 128;
    const uintptr_t al = (uintptr_t)d.C | (uintptr_t)d.aux | (uintptr_t)d.bias | (uintptr_t)d.W32 | (uintptr_t)d.W16 | (uintptr_t)d.gout;
    const bool aligned = d.ldc % 4 == 0 && d.ldaux % 4 == 0 && (al & 15) == 0;
    if (aligned && t128 >= 64 && d.M % tile == 0 && d.N % tile == 0 && d.K % 64 == 0) return false;
    if (aligned && whole_tiles(d, t128)) return false;
    return !register_staged(d, t128);
}

bool gemm16s_try_launch(const GemmDesc &d, hipStream_t s, hipError_t *err) {
    G16SPlan p;
    if (!gemm16s_serves(d) || !choose(d, &p)) return false;
    *err = launch_cfg(d, p, s);
    return true;
}

}  // namespace ah
