// gemm16s_cfg.hip — f16 MFMA contraction with K split across workgroups and any output size (gfx950). Compiled once per
// tile configuration (-DAH_G16S=<n>, kG16SCfg); gemm16s.hip chooses between them.
//
// The whole-tile variants (gemm16_kernel.h) give each 128x128 or 256x256 output tile to one workgroup: an output of few
// tiles leaves most CUs idle behind one long K loop (32 x 4096 x 4096: 32 workgroups, 31 us for 32 MiB of weights), and a
// size that is no multiple of the tile drops to a per-element epilogue (999 x 1000 x 2056 ran the register-staged kernel,
// K % 64 being 8: 16.7 us). Here
//  - the gridDim.y workgroups of a tile each contract a run of K stages; partial tiles are folded by the last to arrive,
//    in split order (the f32 kernels' scheme, gemm.hip), so nobody waits and the sum does not depend on timing;
//  - inside a workgroup KI wave sets share every stage and take its k-steps in turn, so a small tile still has 8 waves;
//    their accumulators are added in set order through LDS;
//  - operands come in by buffer loads straight to LDS, bounded by each operand's size: rows past M or N and k past K read
//    as zeros, so neither has to divide anything but the 8 halves of a load;
//  - the epilogue goes through LDS to 4 consecutive columns per lane, whole vectors where the row admits them and single
//    elements at the edge.
// LDS images, swizzles and fragments are gemm16_kernel.h's (k-contiguous: XOR-swizzled 256-byte super-rows read with
// ds_read_b128; MN-contiguous: stored orientation read with ds_read_b64_tr_b16).
#include "ah_common.h"
#include "gemm16s.h"
#include "gemm_epi.h"

namespace ah {
namespace g16s {

typedef half_t h8 __attribute__((ext_vector_type(8)));
typedef half_t h4 __attribute__((ext_vector_type(4)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s4 lds_s4;

// Byte offset of (row r, 16-byte chunk c) of a k-contiguous stage of BK halves per row.
template <int BK>
__device__ __forceinline__ int koff(int r, int c) {
    constexpr int CH = BK / 8, SR = 16 / CH;
    const int q = r / SR;
    return q * 256 + ((((r % SR) * CH + c) ^ (q & 15)) << 4);
}
// Byte offset of (k-row k, column m) of an MN-contiguous stage of R columns. The swizzle of its 32-byte segments keeps the
// four k-rows of one transposing read in different banks: a k-row of 128 columns spans all 64 banks, one of 64 half of
// them (rows two apart would meet), one of 32 a quarter (four rows already fill the banks).
template <int R>
__device__ __forceinline__ int mn_swz(int k) {
    if constexpr (R >= 128) return ((k & 3) << 1) ^ ((k >> 3) & 1);
    else if constexpr (R == 64) return k & 2;
    else return 0;
}
template <int R>
__device__ __forceinline__ int mnoff(int k, int m) {
    return k * (R * 2) + (((m >> 4) ^ mn_swz<R>(k)) << 5) + ((m & 15) << 1);
}

// Fragment of MI rows from r, k-step s of the stage (one MFMA's k): 32x32x16 lanes hold row l % 32, k = 16 s + 8 (l / 32)
// .. + 7; 16x16x32 lanes row l % 16, k = 32 s + 8 (l / 16) .. + 7.
template <int R, int T, int BK, int MI>
__device__ __forceinline__ h8 frag(const char *img, int r, int s, int lane) {
    constexpr int HI = 64 / MI;   // lane groups along k
    if constexpr (T == 0) {
        return *(const h8 *)(img + koff<BK>(r + lane % MI, HI * s + lane / MI));
    } else {
        const int g = lane >> 4, j = lane & 15;
        const int m = r + (MI == 32 ? 16 * (g & 1) : 0) + 4 * (j & 3);
        const int k = 8 * HI * s + 8 * (MI == 32 ? g >> 1 : g) + (j >> 2);
        const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(img + mnoff<R>(k, m)));
        const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(img + mnoff<R>(k + 4, m)));
        return __builtin_bit_cast(h8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
}

// One 16-byte-per-lane buffer load into LDS (destination LDS address in M0, lane l's bytes at + 16 l). Issued from inline
// asm so the compiler adds no waits of its own; the kernel orders these loads with s_waitcnt vmcnt. A lane whose offset is
// past the descriptor's size gets zeros.
__device__ __forceinline__ void dma16(uint32_t voff, u4 rsrc, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(rsrc), "s"(lds)
                 : "memory", "m0");
}
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// One operand's share of a wave's stage loads: block j (of PER) of the wave is the stage image's 1 KiB block j * NW + wave.
template <int R, int T, int BK, int NW>
struct Fetch {
    static constexpr int NB = R * BK * 2 / 1024, PER = NB / NW;
    static_assert(PER * NW == NB, "an operand's blocks split evenly over the waves");
    uint32_t off[PER];   // the lane's byte offset from the operand's first row (k-contiguous) or k-row at stage 0
    const char *base;
    long size, step;     // operand bytes, bytes per stage
    __device__ __forceinline__ static int chunk(int b, int lane) {   // k-contiguous: the lane's 16-byte chunk of its row
        constexpr int CH = BK / 8;
        return ((lane & 15) ^ ((4 * b + (lane >> 4)) & 15)) % CH;
    }
    // rows: the operand's rows (T 0) or columns (T 1); K its k extent; r0 the tile's first row; kb the first k
    __device__ __forceinline__ void init(const void *p, long ld, int rows, int K, int r0, long kb, int wave, int lane) {
        const long total = T == 0 ? ((long)(rows - 1) * ld + K) * 2 : ((long)(K - 1) * ld + rows) * 2;
        const long skip = T == 0 ? ((long)r0 * ld + kb) * 2 : (kb * ld + r0) * 2;
        base = (const char *)p + skip;
        size = total - skip;
        step = T == 0 ? BK * 2 : (long)BK * ld * 2;
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int b = j * NW + wave;
            if constexpr (T == 0) {
                constexpr int CH = BK / 8, SR = 16 / CH;
                const int q = 4 * b + (lane >> 4), x = (lane & 15) ^ (q & 15);
                off[j] = (uint32_t)(((long)(q * SR + x / CH) * ld + (x % CH) * 8) * 2);
            } else {
                constexpr int ROWS = 512 / R;
                const int kk = b * ROWS + (16 * lane) / (2 * R), pos = ((16 * lane) % (2 * R)) / 16;
                off[j] = (uint32_t)(((long)kk * ld + ((pos >> 1) ^ mn_swz<R>(kk)) * 16 + (pos & 1) * 8) * 2);
            }
        }
    }
    // the descriptor of stage kt, of size 0 from stage nk on (its loads give zeros and read nothing)
    __device__ __forceinline__ u4 rsrc(int kt, int nk) const {
        const long adv = (long)kt * step, left = size - adv;
        const uintptr_t a = (uintptr_t)(base + adv);
        return (u4){(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, kt < nk ? (uint32_t)left : 0u, 0x00020000u};
    }
    // load j of the stage with descriptor r, krem values of k from its first one on, into the image at LDS address img
    __device__ __forceinline__ void issue(int j, u4 r, long krem, uint32_t img, int wave, int lane) const {
        uint32_t o = off[j];
        if constexpr (T == 0) {   // k past K would be the next row's values
            if (krem < BK) o = chunk(j * NW + wave, lane) * 8 < krem ? o : 0x80000000u;
        }
        dma16(o, r, img + (uint32_t)((j * NW + wave) * 1024));
    }
};

template <typename T>
struct V4;
template <> struct V4<float> { typedef floatx4 type; };
template <> struct V4<half_t> { typedef h4 type; };

// n elements (1..4) of 4 consecutive ones at p; vec: the 16- (or 8-) byte access is aligned and n is 4
template <typename T>
__device__ __forceinline__ floatx4 load4(const T *p, bool vec, int n) {
    floatx4 v = {};
    if (vec) {
        const typename V4<T>::type x = *(const typename V4<T>::type *)p;
        v = (floatx4){(float)x[0], (float)x[1], (float)x[2], (float)x[3]};
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (e < n) v[e] = (float)p[e];
    }
    return v;
}
template <typename T>
__device__ __forceinline__ void store4(T *p, const T (&x)[4], bool vec, int n) {
    if (vec) {
        *(typename V4<T>::type *)p = (typename V4<T>::type){x[0], x[1], x[2], x[3]};
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (e < n) p[e] = x[e];
    }
}

// Floats per row of the epilogue's LDS region: the row groups of one accumulator write (two of 32 lanes, or four of 16, 4
// rows apart) fall into different banks.
template <int FN, int MI>
constexpr int kEpiLd = FN * 32 + (MI == 32 ? 8 : 4);

// The wave tile's epilogue, 32 rows at a time through the wave's LDS region. acc(i, j, r): element r of 32x32 block (i, j)
// (MI 32: the MFMA's own layout; MI 16: its four 16x16 blocks, quarter r / 4 by row then column).
template <int EPI, int FM, int FN, int MI, class Acc>
__device__ __forceinline__ void epilogue(const GemmDesc &d, const Acc &acc, int mb, int nb, int lane, char *wlds, bool aligned) {
    constexpr int LD = kEpiLd<FN, MI>, CPR = FN * 8, RPI = 64 / CPR, NR = 32 / RPI;   // lanes per row, rows per pass, passes
    const float sc = d.scale, lr = d.lr;
    float *const st = (float *)wlds;
    const int c4 = (lane % CPR) * 4, n = nb + c4, nv = d.N - n;   // columns left: may be <= 0
    const bool vec = aligned && nv >= 4;
    floatx4 bias = {};
    if constexpr (EPI == EPI_BIAS || EPI == EPI_BIAS_RELU) {
        if (nv > 0) bias = load4((const half_t *)d.bias + n, vec, nv);
    }
#pragma unroll
    for (int i = 0; i < FM; i++) {
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) st[acc_row_mi<MI>(r, lane) * LD + j * 32 + acc_col_mi<MI>(r, lane)] = acc(i, j, r);
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this wave's writes have landed
        __builtin_amdgcn_wave_barrier();
        constexpr int NI = NR < 8 ? NR : 8;   // passes whose inputs are loaded together
#pragma unroll
        for (int t0 = 0; t0 < NR; t0 += NI) {
        floatx4 in[NI];
        if constexpr (EPI == EPI_MASK || EPI == EPI_SGD) {
#pragma unroll
            for (int t = 0; t < NI; t++) {
                const long m = mb + i * 32 + (t0 + t) * RPI + lane / CPR;
                in[t] = (floatx4){};
                if (m < d.M && nv > 0) {
                    if constexpr (EPI == EPI_SGD) in[t] = load4(d.W32 + m * d.ldc + n, vec, nv);
                    else in[t] = load4((const half_t *)d.aux + m * d.ldaux + n, vec, nv);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < NI; t++) {
            const int row = (t0 + t) * RPI + lane / CPR;
            const long m = mb + i * 32 + row;
            const floatx4 a = *(const floatx4 *)(st + row * LD + c4);
            if (m >= d.M || nv <= 0) continue;
            if constexpr (EPI == EPI_SGD) {
                const floatx4 g = sc * a;
                floatx4 w = in[t] - lr * g;
                asm volatile("" : "+v"(w));   // the f16 copy is f16 of the stored f32 value
                const float gs[4] = {g[0], g[1], g[2], g[3]}, ws[4] = {w[0], w[1], w[2], w[3]};
                if (d.gout) store4(d.gout + m * d.ldc + n, gs, vec, nv);
                store4(d.W32 + m * d.ldc + n, ws, vec, nv);
                if (d.W16) {
                    const half_t hs[4] = {(half_t)w[0], (half_t)w[1], (half_t)w[2], (half_t)w[3]};
                    store4((half_t *)d.W16 + m * d.ldc + n, hs, vec, nv);
                }
            } else {
                half_t o[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if constexpr (EPI == EPI_STORE) o[e] = (half_t)(sc * a[e]);
                    else if constexpr (EPI == EPI_MASK) o[e] = (half_t)(relu_dead((half_t)in[t][e]) ? 0.0f : sc * a[e]);
                    else {
                        const half_t z = (half_t)(q16(a[e]) + bias[e]);   // f16(f16(acc) + b)
                        o[e] = EPI == EPI_BIAS_RELU ? relu_tag(z) : z;
                    }
                }
                store4((half_t *)d.C + m * d.ldc + n, o, vec, nv);
            }
        }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// BM x BN tile, BK halves of K per stage, NS stages in flight, WVM x WVN waves per set, KI wave sets, MI x MI MFMAs.
template <int BM, int BN, int BK, int NS, int WVM, int WVN, int KI, int MI, int TA, int TB, int EPI>
__global__ __launch_bounds__(64 * WVM * WVN * KI) void gemm16s_kernel(GemmDesc d, int stages) {
    constexpr int NW = WVM * WVN * KI, SETW = WVM * WVN, SETT = 64 * SETW;
    constexpr int WM = BM / WVM, WN = BN / WVN, FM = WM / 32, FN = WN / 32, FA = WM / MI, FB = WN / MI, NM = FA * FB;
    constexpr int IMGA = BM * BK * 2, STAGE = (BM + BN) * BK * 2, KS = BK / (MI == 32 ? 16 : 32), KW = KS / KI;
    constexpr int EPIW = 32 * kEpiLd<FN, MI> * 4;                                  // epilogue bytes per wave
    constexpr int RED = (KI - 1) * BM * BN * 4, EP = SETW * EPIW;
    constexpr int SM0 = NS * STAGE > RED ? NS * STAGE : RED, SMEM = SM0 > EP ? SM0 : EP;
    static_assert(KW * KI == KS && KW % 2 == 0, "the sets share a stage's k-steps evenly; the next stage opens in slot 0");
    static_assert(KI == 1 || MI == 32, "the sets' fold reads 32x32 blocks");
    __shared__ __attribute__((aligned(1024))) char smem[SMEM];
    __shared__ int ticket;

    const int tiles_n = (d.N + BN - 1) / BN, tiles_m = (d.M + BM - 1) / BM, ntiles = tiles_m * tiles_n;
    int L = blockIdx.x;
    if ((ntiles & 7) == 0) L = (L & 7) * (ntiles >> 3) + (L >> 3);   // runs of tiles per XCD
    constexpr int G = 4;
    const int group = L / (G * tiles_n), gm0 = group * G, gsz = min(G, tiles_m - gm0);
    const int rem = L - group * G * tiles_n, tm = gm0 + rem % gsz, tn = rem / gsz;
    const int m0 = tm * BM, n0 = tn * BN;

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int ki = wave / SETW, sw = wave % SETW;
    const int wm0 = (sw / WVN) * WM, wn0 = (sw % WVN) * WN;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char *)smem;

    const int split = blockIdx.y, nsplit = gridDim.y;
    const long kb = (long)split * stages * BK;
    const int nk = min(stages, (int)((d.K - kb + BK - 1) / BK));   // >= 1: the launcher leaves no split empty
    Fetch<BM, TA, BK, NW> fa;
    Fetch<BN, TB, BK, NW> fb;
    fa.init(d.A, d.lda, d.M, d.K, m0, kb, wave, lane);
    fb.init(d.B, d.ldb, d.N, d.K, n0, kb, wave, lane);
    constexpr int PA = Fetch<BM, TA, BK, NW>::PER, PER = PA + Fetch<BN, TB, BK, NW>::PER;

    floatx16 acc[MI == 32 ? FM : 1][MI == 32 ? FN : 1];
    floatx4 acc4[MI == 16 ? FA : 1][MI == 16 ? FB : 1];
    if constexpr (MI == 32) {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) acc[i][j] = (floatx16){};
    } else {
#pragma unroll
        for (int i = 0; i < FA; i++)
#pragma unroll
            for (int j = 0; j < FB; j++) acc4[i][j] = (floatx4){};
    }
    // The stages 0 .. NS-1 go out at once; from then on stage kt + NS refills stage kt's buffer, one load after every few
    // MFMAs of the k-step that follows the barrier. Past the last stage the loads go on with empty descriptors, so the
    // number in flight, and with it the wait count, is the same in every iteration.
#pragma unroll
    for (int p = 0; p < NS; p++) {
        const long krem = d.K - kb - (long)p * BK;
        const u4 ra = fa.rsrc(p, nk), rb = fb.rsrc(p, nk);
#pragma unroll
        for (int j = 0; j < PA; j++) fa.issue(j, ra, krem, lds0 + p * STAGE, wave, lane);
#pragma unroll
        for (int j = 0; j < PER - PA; j++) fb.issue(j, rb, krem, lds0 + p * STAGE + IMGA, wave, lane);
    }
    h8 a[2][FA], b[2][FB];
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"((NS - 1) * PER) : "memory");
    lds_barrier();
#pragma unroll
    for (int i = 0; i < FA; i++) a[0][i] = frag<BM, TA, BK, MI>(smem, wm0 + MI * i, ki, lane);
#pragma unroll
    for (int j = 0; j < FB; j++) b[0][j] = frag<BN, TB, BK, MI>(smem + IMGA, wn0 + MI * j, ki, lane);
    for (int kt = 0; kt < nk; kt++) {
        const int buf = kt % NS, nbuf = (kt + 1) % NS, kr = kt + NS;
        const char *sa = smem + buf * STAGE, *sb = sa + IMGA;
        const char *na = smem + nbuf * STAGE, *nbp = na + IMGA;
        const long krem = d.K - kb - (long)kr * BK;
        const u4 ra = fa.rsrc(kr, nk), rb = fb.rsrc(kr, nk);
#pragma unroll
        for (int s = 0; s < KW; s++) {
            const int c = s & 1, nx = c ^ 1;
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 < KW) {
#pragma unroll
                for (int i = 0; i < FA; i++) a[nx][i] = frag<BM, TA, BK, MI>(sa, wm0 + MI * i, (s + 1) * KI + ki, lane);
#pragma unroll
                for (int j = 0; j < FB; j++) b[nx][j] = frag<BN, TB, BK, MI>(sb, wn0 + MI * j, (s + 1) * KI + ki, lane);
            } else {
                // stage kt + 1 has landed for this wave once only the NS - 2 younger stages' loads are out; after the
                // barrier for every wave, and every wave has read all of stage kt's fragments
                asm volatile("s_waitcnt vmcnt(%0)" ::"i"((NS - 2) * PER) : "memory");
                lds_barrier();
#pragma unroll
                for (int i = 0; i < FA; i++) a[nx][i] = frag<BM, TA, BK, MI>(na, wm0 + MI * i, ki, lane);
#pragma unroll
                for (int j = 0; j < FB; j++) b[nx][j] = frag<BN, TB, BK, MI>(nbp, wn0 + MI * j, ki, lane);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < NM; t++) {
                if constexpr (MI == 32)
                    acc[t / FB][t % FB] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[c][t / FB], b[c][t % FB], acc[t / FB][t % FB], 0, 0, 0);
                else
                    acc4[t / FB][t % FB] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[c][t / FB], b[c][t % FB], acc4[t / FB][t % FB], 0, 0, 0);
                if (s == KW - 1) {   // loads [t * PER / NM, (t + 1) * PER / NM) of the refill
#pragma unroll
                    for (int f = t * PER / NM; f < (t + 1) * PER / NM; f++) {
                        if (f < PA) fa.issue(f, ra, krem, lds0 + buf * STAGE, wave, lane);
                        else fb.issue(f - PA, rb, krem, lds0 + buf * STAGE + IMGA, wave, lane);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last loads land before the LDS is reused
    __syncthreads();

    if constexpr (KI > 1) {
        // sets 1 .. KI-1 hand their accumulators to set 0: element e of lane l of wave w of set g at [g-1][w][e][l]
        constexpr int NE = FM * FN * 16;
        float *const red = (float *)smem + lane;
        if (ki > 0) {
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) red[(((ki - 1) * SETW + sw) * NE + (i * FN + j) * 16 + r) * 64] = acc[i][j][r];
        }
        __syncthreads();
        if (ki == 0) {
#pragma unroll
            for (int g = 1; g < KI; g++)
#pragma unroll
                for (int i = 0; i < FM; i++)
#pragma unroll
                    for (int j = 0; j < FN; j++)
#pragma unroll
                        for (int r = 0; r < 16; r++) acc[i][j][r] += red[(((g - 1) * SETW + sw) * NE + (i * FN + j) * 16 + r) * 64];
        }
        __syncthreads();   // the epilogue reuses this LDS
    }
    if constexpr (MI == 32) if (nsplit > 1) {
        // Set 0 stores its accumulators as the split's partial with 16-byte sc1 buffer stores (coherent across the XCDs'
        // L2s) and waits for them; the split that draws the tile's last ticket adds all partials in split order, its own
        // from registers. Chunk c of thread t at byte 16 * (c * SETT + t) of its split.
        constexpr int NC = FM * FN * 4, PART = NC * SETT * 16, SC1 = 16;
        const int tid = threadIdx.x, tile = tm * tiles_n + tn;
        int *const count = d.sk_sync + 2 * tile;
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
            d.sk_part + (long)tile * nsplit * (PART / 4), (short)0, nsplit * PART, 0x00020000);
        if (ki == 0) {
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const floatx16 &a = acc[c / (FN * 4)][(c / 4) % FN];
                const int e = (c % 4) * 4;
                const floatx4 v = {a[e], a[e + 1], a[e + 2], a[e + 3]};
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r, split * PART + (c * SETT + tid) * 16, 0, SC1);
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("s_nop 4" ::: "memory");   // before the store's data registers may be rewritten (see gemm.hip)
                __builtin_amdgcn_sched_barrier(0);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        __syncthreads();
        if (threadIdx.x == 0) ticket = ticket_take_atomic_partials(count);
        __syncthreads();
        if (ticket != nsplit - 1) return;
        if (ki == 0) {
#pragma unroll
            for (int bl = 0; bl < FM * FN; bl++) {
                floatx16 &a = acc[bl / FN][bl % FN];
                floatx4 sum[4];
                for (int q = 0; q < nsplit; q++) {
                    floatx4 v[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        if (q == split) v[u] = (floatx4){a[4 * u], a[4 * u + 1], a[4 * u + 2], a[4 * u + 3]};
                        else v[u] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, q * PART + ((bl * 4 + u) * SETT + tid) * 16, 0, SC1));
                    }
#pragma unroll
                    for (int u = 0; u < 4; u++) sum[u] = q == 0 ? v[u] : sum[u] + v[u];
                }
#pragma unroll
                for (int u = 0; u < 4; u++)
#pragma unroll
                    for (int x = 0; x < 4; x++) a[4 * u + x] = sum[u][x];
            }
        }
        if (threadIdx.x == 0) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // next launch
    }
    if (ki > 0) return;
    auto accv = [&](int i, int j, int r) -> float {
        if constexpr (MI == 32) return acc[i][j][r];
        else return acc4[2 * i + (r >> 3)][2 * j + ((r >> 2) & 1)][r & 3];
    };
    const uintptr_t al = (uintptr_t)d.C | (uintptr_t)d.aux | (uintptr_t)d.bias | (uintptr_t)d.W32 | (uintptr_t)d.W16 | (uintptr_t)d.gout;
    epilogue<EPI, FM, FN, MI>(d, accv, m0 + wm0, n0 + wn0, lane, smem + sw * EPIW, (al & 15) == 0 && d.ldc % 4 == 0 && d.ldaux % 4 == 0);
}

#if AH_G16S == 0
constexpr int kNS = 4, kWVM = 2, kWVN = 2, kKI = 2, kMI = 32;   // 128 KiB of stages: one workgroup per CU
#elif AH_G16S == 1
constexpr int kNS = 3, kWVM = 2, kWVN = 2, kKI = 2, kMI = 32;   // 72 KiB: two
#elif AH_G16S == 2
constexpr int kNS = 4, kWVM = 2, kWVN = 2, kKI = 2, kMI = 32;   // 64 KiB: two
#elif AH_G16S == 3
constexpr int kNS = 3, kWVM = 1, kWVN = 2, kKI = 4, kMI = 32;   // 72 KiB: two
#elif AH_G16S == 4
constexpr int kNS = 3, kWVM = 2, kWVN = 2, kKI = 2, kMI = 32;   // 72 KiB: two
#elif AH_G16S == 5
constexpr int kNS = 2, kWVM = 4, kWVN = 2, kKI = 1, kMI = 16;   // 128 KiB: one
#elif AH_G16S == 6
constexpr int kNS = 2, kWVM = 2, kWVN = 2, kKI = 1, kMI = 32;   // 64 KiB: two
#elif AH_G16S == 7
constexpr int kNS = 2, kWVM = 2, kWVN = 2, kKI = 1, kMI = 32;   // 48 KiB: three
#else
constexpr int kNS = 2, kWVM = 2, kWVN = 2, kKI = 1, kMI = 32;   // 32 KiB: five
#endif
constexpr G16SCfg kC = kG16SCfg[AH_G16S];

template <int TA, int TB, int EPI>
static hipError_t launch(const GemmDesc &d, const G16SPlan &p, hipStream_t s) {
    const dim3 grid(((d.M + kC.bm - 1) / kC.bm) * ((d.N + kC.bn - 1) / kC.bn), p.split);
    hipLaunchKernelGGL((gemm16s_kernel<kC.bm, kC.bn, kC.bk, kNS, kWVM, kWVN, kKI, kMI, TA, TB, EPI>), grid, dim3(64 * kWVM * kWVN * kKI), 0,
                       s, d, p.stages);
    return hipGetLastError();
}
template <int TA, int TB>
static hipError_t launch_epi(const GemmDesc &d, const G16SPlan &p, hipStream_t s) {
    switch (d.epi) {
        case EPI_STORE: return launch<TA, TB, EPI_STORE>(d, p, s);
        case EPI_BIAS: return launch<TA, TB, EPI_BIAS>(d, p, s);
        case EPI_BIAS_RELU: return launch<TA, TB, EPI_BIAS_RELU>(d, p, s);
        case EPI_MASK: return launch<TA, TB, EPI_MASK>(d, p, s);
        case EPI_SGD: return launch<TA, TB, EPI_SGD>(d, p, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace g16s

#define AH_G16S_NAME2(n) gemm16s_launch_##n
#define AH_G16S_NAME(n) AH_G16S_NAME2(n)
hipError_t AH_G16S_NAME(AH_G16S)(const GemmDesc &d, const G16SPlan &p, hipStream_t s) {
    if (d.ta == 0 && d.tb == 0) return g16s::launch_epi<0, 0>(d, p, s);
    if (d.ta == 0 && d.tb == 1) return g16s::launch_epi<0, 1>(d, p, s);
    if (d.ta == 1 && d.tb == 1) return g16s::launch_epi<1, 1>(d, p, s);
    return hipErrorInvalidValue;
}

}  // namespace ah
