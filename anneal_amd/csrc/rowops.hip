// rowops.hip — row reductions, loss-gradient epilogues and small elementwise kernels (gfx950).
//
// Softmax cross-entropy: one wave64 per row (a workgroup past 1024 logits), shuffle reductions for the row
// max, the tie count and the exp-sum; the backward follows the reference's op-by-op rules so the gradient through the row
// max (tensor/gradient_ruleset.go:307-320, no stop-gradient in the reference) is reproduced.
//
// Movement chain (config 5): column strips of X held on chip between one read of X and one write of dX; where
// they do not fit, two streaming passes over X in its stored [R, Cc] layout. A Y-row is an
// X-column, so lanes own columns and walk rows: every wave load is a contiguous 1 KiB row segment
// (float4 per lane) and no transpose is ever materialized. Pass 1 keeps online (max, tie count,
// sum e, sum e^2) per column; a per-column finalize folds the row chunks and evaluates the
// backward's per-row scalars; pass 2 re-reads X and writes dX in the same layout.
#include <float.h>

#include <algorithm>
#include <mutex>

#include "ah_common.h"
#include "rowops.h"
#include "softmax_row.h"

namespace ah {

// ── small elementwise kernels ───────────────────────────────────────────────

__global__ void fill_f32_kernel(float *p, long n, float v) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long stride = (long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

// amp * u, u uniform in [-1, 1) from a 32-bit integer hash of (seed, i); optional f16 copy.
__global__ void fill_hash_kernel(float *p, half_t *p16, long n, uint32_t seed, float amp) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long stride = (long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        uint32_t h = (uint32_t)i * 0x9E3779B1u ^ (uint32_t)(i >> 32) ^ seed;
        h ^= h >> 16; h *= 0x7FEB352Du; h ^= h >> 15; h *= 0x846CA68Bu; h ^= h >> 16;
        const float v = amp * ((float)(h >> 8) * (1.0f / 8388608.0f) - 1.0f);
        if (p) p[i] = v;
        if (p16) p16[i] = (half_t)v;
    }
}

__global__ void cast_f32_f16_kernel(const float *src, half_t *dst, long n) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long stride = (long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) dst[i] = (half_t)src[i];
}

// p -= lr * (scale * g); optional f16 copy and gradient output. Parameter.SGDStep (nn.go:69-76).
__global__ void sgd_kernel(float *p, const float *g, long n, float lr, float scale, half_t *p16, float *gout) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long stride = (long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        float gv = scale * g[i];
        if (gout) gout[i] = gv;
        float w = p[i] - lr * gv;
        asm volatile("" : "+v"(w));   // the f16 copy is f16 of the stored f32 value
        p[i] = w;
        if (p16) p16[i] = (half_t)w;
    }
}

// colsum[n] += sum_m G[m, n]   (bias gradient: Expand rule, tensor/gradient_ruleset.go:207-233)
__global__ __launch_bounds__(256) void colsum_kernel(const float *G, int M, int N, long ld, int rows_per_block,
                                                      float *out) {
    __shared__ float red[4][64];
    int col = blockIdx.x * 64 + (threadIdx.x & 63);
    int sub = threadIdx.x >> 6;
    int r0 = blockIdx.y * rows_per_block;
    int r1 = min(M, r0 + rows_per_block);
    float acc = 0.0f;
    if (col < N)
        for (int r = r0 + sub; r < r1; r += 4) acc += G[(long)r * ld + col];
    red[sub][threadIdx.x & 63] = acc;
    __syncthreads();
    if (sub == 0 && col < N) {
        float v = ((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) + red[3][threadIdx.x];
        atomicAdd(out + col, v);
    }
}

// ── softmax cross-entropy ───────────────────────────────────────────────────
// loss = Sum(onehot * logp) * a,  a = f32(-1/B); see the oracle's ora_softmax_ce for the op list.
// The mean loss of a softmax-CE kernel without a second launch: `mine` is a workgroup's sum of its rows' terms (thread 0).
// Workgroup b stores it to slot b; the last to arrive adds the slots, thread t slots t, t + blockDim, ..., then the threads in
// order, so the result does not depend on timing. Arrivals at one counter queue up (256 of them: 4096 x 512 21.0 us a call, so 19.3; without the loss 16.9), so past 16
// workgroups each of 16 counters takes a sixteenth of them, and its last arrival goes on to the root's. ws: the root counter,
// the 16 others (a 128-byte line each, all zero before and after), the slots. red: one float a wave.
constexpr int kSmGroups = 16, kSmLine = 32, kSmSlots = (1 + kSmGroups) * kSmLine;
__device__ __forceinline__ void softmax_loss_fold(float mine, float a, float *loss, float *ws, float *red) {
    __shared__ int last;
    const int n = gridDim.x;
    if (threadIdx.x == 0) {
        __hip_atomic_store(ws + kSmSlots + blockIdx.x, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int g = blockIdx.x % kSmGroups;
        int *const group = (int *)ws + (1 + g) * kSmLine;
        last = 1;
        if (n > kSmGroups) {
            last = ticket_take_atomic_partials(group) == (n - g + kSmGroups - 1) / kSmGroups - 1;
            if (last) __hip_atomic_store(group, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (last) last = ticket_take_atomic_partials((int *)ws) == min(n, kSmGroups) - 1;
    }
    __syncthreads();
    if (!last) return;
    float v = 0.0f;
    for (int i = threadIdx.x; i < n; i += blockDim.x)
        v += __hip_atomic_load(ws + kSmSlots + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)blockDim.x / 64; w++) v += red[w];
        loss[0] = v * a;
        __hip_atomic_store((int *)ws, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Softmax-CE of rows of up to 64 * VPR logits, a wave a row, the row held in registers between its three wave reductions
// (softmax_ce_row reads it from memory four times) and the wave's next row loading meanwhile. Bound by those reductions'
// latency: up to 256 workgroups of 1 to 16 waves, so that a wave has more than one row only past 4096 rows and the loss takes
// at most 256 arrivals (128 workgroups: 16384 x 1024 47.5 us a call for 39.5). Against four reads of the row and a second
// launch for the loss: 4096 x 512 26.1 -> 19.3 us a call, 16384 x 1024 82.0 -> 39.5 (134 MB, 25 us at the copy rate).
constexpr int kSmWaves = 16, kSmBlocks = 256;
template <int VPR>
__global__ __launch_bounds__(64 * kSmWaves) void softmax_ce_kernel(const float *z, const int32_t *labels, int B, int C,
                                                                   float a, float *dz, float *rowloss, float *loss, float *ws) {
    __shared__ float red[kSmWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6, step = gridDim.x * waves;
    int row = blockIdx.x * waves + wave;
    float nv[VPR], sum = 0.0f, col[VPR] = {};   // col: column sums, not asked for here
    if (row < B) softmax_ce_row_load<VPR>(z + (long)row * C, C, lane, nv);
    for (; row < B; row += step) {
        float v[VPR];
#pragma unroll
        for (int j = 0; j < VPR; j++) v[j] = nv[j];
        if (row + step < B) softmax_ce_row_load<VPR>(z + (long)(row + step) * C, C, lane, nv);
        const float rl = softmax_ce_row_regs<VPR>(v, z + (long)row * C, labels[row], C, a, dz + (long)row * C, lane, col);
        if (rowloss && lane == 0) rowloss[row] = rl;
        sum += rl;
    }
    if (!loss) return;
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < waves; w++) sum += red[w];
    __syncthreads();   // red is reused by the fold
    softmax_loss_fold(sum, a, loss, ws, red);
}

// Rows of more than 1024 and up to 512 * VPR logits: a workgroup of 8 waves a row, held in registers. Bound by the three
// workgroup reductions and, with many rows, by memory. One wave a row from memory: 1 x 8192 77.4 us a call, 2000 x
// 8192 164.7; so 17.8 and 40.2.
constexpr int kSmWideThreads = 512, kSmWideWaves = kSmWideThreads / 64;
template <int VPR>
__global__ __launch_bounds__(kSmWideThreads) void softmax_ce_wide_kernel(const float *z, const int32_t *labels, int B, int C,
                                                                         float a, float *dz, float *rowloss, float *loss, float *ws) {
#pragma clang fp contract(off)   // each reference op rounds on its own, as in softmax_ce_row
    __shared__ float red[4][kSmWideWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    auto load = [&](int row, float (&v)[VPR]) {
#pragma unroll
        for (int j = 0; j < VPR; j++) {
            const int c = tid + kSmWideThreads * j;
            v[j] = c < C ? z[(long)row * C + c] : -FLT_MAX;
        }
    };
    auto fold = [&](int k) {   // the waves' sums in order, the same in every thread
        float r = red[k][0];
#pragma unroll
        for (int w = 1; w < kSmWideWaves; w++) r += red[k][w];
        return r;
    };
    float nv[VPR], total = 0.0f;
    int row = blockIdx.x;
    load(row, nv);   // the grid has no more workgroups than rows
    for (; row < B; row += gridDim.x) {
        float v[VPR], e[VPR];
#pragma unroll
        for (int j = 0; j < VPR; j++) v[j] = nv[j];
        if (row + (int)gridDim.x < B) load(row + gridDim.x, nv);
        const int lab = labels[row];
        const bool in = lab >= 0 && lab < C;
        const float zl = in ? z[(long)row * C + lab] : 0.0f;
        float m = -FLT_MAX;
#pragma unroll
        for (int j = 0; j < VPR; j++) m = fmaxf(m, v[j]);
        m = wave_max(m);
        if (lane == 0) red[0][wave] = m;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kSmWideWaves; w++) m = fmaxf(m, red[0][w]);
        float tie = 0.0f, s = 0.0f;
#pragma unroll
        for (int j = 0; j < VPR; j++) {
            e[j] = exp2f((v[j] - m) * AH_INV_LN2);
            if (tid + kSmWideThreads * j < C) {
                tie += v[j] == m ? 1.0f : 0.0f;
                s += e[j];
            }
        }
        tie = wave_sum(tie);
        s = wave_sum(s);
        if (lane == 0) {
            red[1][wave] = tie;
            red[2][wave] = s;
        }
        __syncthreads();
        tie = fold(1);
        s = fold(2);
        const float ls = log2f(s) * AH_LN2;
        const float rl = in ? ((zl - m) - ls) : 0.0f;
        const float gls = in ? -a : 0.0f;
        const float gs = (gls * AH_LN2) * (1.0f / (s * AH_LN2));
        float gm = 0.0f;
#pragma unroll
        for (int j = 0; j < VPR; j++) {
            const int c = tid + kSmWideThreads * j;
            e[j] = (c == lab ? a : 0.0f) + ((gs * e[j]) * AH_LN2) * AH_INV_LN2;
            if (c < C) gm += -e[j];
        }
        gm = wave_sum(gm);
        if (lane == 0) red[3][wave] = gm;
        __syncthreads();   // a wave at the next row's red[0] store has passed here, where all have read red[0]; so for the others
        const float share = fold(3) * (1.0f / tie);
#pragma unroll
        for (int j = 0; j < VPR; j++) {
            const int c = tid + kSmWideThreads * j;
            if (c < C) dz[(long)row * C + c] = v[j] == m ? e[j] + share : e[j];
        }
        if (rowloss && tid == 0) rowloss[row] = rl;
        total += rl;
    }
    if (!loss) return;
    __syncthreads();   // red is reused by the fold
    softmax_loss_fold(total, a, loss, ws, red[0]);
}

// Longer rows: a wave a row, from memory; with the loss up to kSmLongBlocks workgroups, which fill the chip 8 to a CU (512 of
// them left it a quarter full: 4096 x 16384 749 us a call, so 513).
constexpr int kSmLongBlocks = 2048;
__global__ __launch_bounds__(256) void softmax_ce_long_kernel(const float *z, const int32_t *labels, int B, int C,
                                                              float a, float *dz, float *rowloss, float *loss, float *ws) {
    __shared__ float red[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float sum = 0.0f;
    for (int row = blockIdx.x * 4 + wave; row < B; row += gridDim.x * 4) {
        const float rl = softmax_ce_row(z + (long)row * C, labels[row], C, a, dz + (long)row * C, lane);
        if (rowloss && lane == 0) rowloss[row] = rl;
        sum += rl;
    }
    if (!loss) return;
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) sum = ((red[0] + red[1]) + red[2]) + red[3];
    __syncthreads();
    softmax_loss_fold(sum, a, loss, ws, red);
}

// Softmax-CE with the logit gradient's column sums (the output bias gradient) fused in: each wave
// takes rows blockIdx.x * kSmWaves + wave, then every kSmWaves * gridDim.x rows further, holding each
// row in registers, and keeps the column sums of its rows' dz in registers; the block's waves add theirs
// in wave order into partial row blockIdx.x of part[gridDim.x][C] (summed in row order by the step's
// tail), so the result does not depend on timing. With 16 waves per block and up to 256 blocks, a batch
// of up to 4096 rows gives every wave one row: the row's three dependent wave reductions then overlap
// across waves instead of running back to back in one.
template <int VPR>
__global__ __launch_bounds__(64 * kSmWaves) void softmax_ce_cols_kernel(const float *z, const int32_t *labels, int B, int C,
                                                                        float a, float *dz, float *rowloss, float *part) {
    __shared__ float red[kSmWaves][64 * VPR];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float col[VPR];
#pragma unroll
    for (int j = 0; j < VPR; j++) col[j] = 0.0f;
    // the next row's loads are issued before this row's arithmetic, so a wave with several rows keeps
    // one row's loads in flight
    const int step = gridDim.x * kSmWaves;
    int row = blockIdx.x * kSmWaves + wave;
    float nv[VPR];
    if (row < B) softmax_ce_row_load<VPR>(z + (long)row * C, C, lane, nv);
    for (; row < B; row += step) {
        float v[VPR];
#pragma unroll
        for (int j = 0; j < VPR; j++) v[j] = nv[j];
        if (row + step < B) softmax_ce_row_load<VPR>(z + (long)(row + step) * C, C, lane, nv);
        const float rl = softmax_ce_row_regs<VPR>(v, z + (long)row * C, labels[row], C, a, dz + (long)row * C, lane, col);
        if (lane == 0) rowloss[row] = rl;
    }
#pragma unroll
    for (int j = 0; j < VPR; j++) red[wave][lane + 64 * j] = col[j];
    __syncthreads();
    for (int c = threadIdx.x; c < C; c += 64 * kSmWaves) {
        float acc = red[0][c];
        for (int w = 1; w < kSmWaves; w++) acc += red[w][c];
        part[(long)blockIdx.x * C + c] = acc;
    }
}

// MSE loss finalize: f16 reduce narrowing f16(acc) (codegen/lower.go:712) then * scale in f32.
__global__ void mse_finalize_kernel(const float *acc, float scale, float *out) {
    if (threadIdx.x == 0 && blockIdx.x == 0) out[0] = q16(acc[0]) * scale;
}

// ── config 5: movement + row-reduce chain ───────────────────────────────────

// exp2 of a non-positive argument as the bare v_exp_f32: results below 2^-126 flush to zero (they are
// below f32's normal range and change no sum they enter; exp2f's denormal fix-up costs ~5 VALU ops
// per element, which is most of these streaming kernels' per-element work).
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

struct ColStat {
    float m, t, s, q;
};

__device__ __forceinline__ void stat_push(ColStat &st, float y) {
    if (y > st.m) {
        float f = exp2f((st.m - y) * AH_INV_LN2);
        st.s = st.s * f + 1.0f;
        st.q = st.q * (f * f) + 1.0f;
        st.m = y;
        st.t = 1.0f;
    } else {
        float e = exp2f((y - st.m) * AH_INV_LN2);
        st.s += e;
        st.q += e * e;
        st.t += (y == st.m) ? 1.0f : 0.0f;
    }
}

__device__ __forceinline__ ColStat stat_merge(const ColStat &a, const ColStat &b) {
    ColStat r;
    r.m = fmaxf(a.m, b.m);
    float fa = exp2f((a.m - r.m) * AH_INV_LN2), fb = exp2f((b.m - r.m) * AH_INV_LN2);
    if (a.s == 0.0f) fa = 0.0f;
    if (b.s == 0.0f) fb = 0.0f;
    r.s = a.s * fa + b.s * fb;
    r.q = a.q * (fa * fa) + b.q * (fb * fb);
    r.t = (a.m == r.m ? a.t : 0.0f) + (b.m == r.m ? b.t : 0.0f);
    return r;
}

// Pass 1. Block = 4 waves over the same 256 columns (lane owns 4 consecutive columns);
// blockIdx.y selects a chunk of `rch` rows, waves interleave rows within it. Each wave issues 8 row
// loads (8 KiB) before consuming any, so enough bytes are in flight to cover HBM latency.
__global__ __launch_bounds__(256) void chain_stats_kernel(const float *X, int R, int Cc, int rch, ColStat *part) {
    __shared__ ColStat sh[4][256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c0 = blockIdx.x * 256 + lane * 4;
    const int r0 = blockIdx.y * rch, r1 = min(R, r0 + rch);
    ColStat st[4];
#pragma unroll
    for (int u = 0; u < 4; u++) st[u] = ColStat{-FLT_MAX, 0.0f, 0.0f, 0.0f};
    if (c0 < Cc) {
        int r = r0 + wave;
        for (; r + 28 < r1; r += 32) {
            floatx4 v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = *(const floatx4 *)(X + (long)(r + 4 * j) * Cc + c0);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                // Rescale once per 8 rows to the batch max, then accumulate without branches
                // (the element equal to the new max contributes exp2(0) = 1 exactly, as in stat_push).
                float mb = v[0][u];
#pragma unroll
                for (int j = 1; j < 8; j++) mb = fmaxf(mb, v[j][u]);
                if (mb > st[u].m) {
                    const float f = exp2f((st[u].m - mb) * AH_INV_LN2);
                    st[u].s *= f;
                    st[u].q *= f * f;
                    st[u].t = 0.0f;
                    st[u].m = mb;
                }
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const float e = fast_exp2((v[j][u] - st[u].m) * AH_INV_LN2);
                    st[u].s += e;
                    st[u].q += e * e;
                    st[u].t += (v[j][u] == st[u].m) ? 1.0f : 0.0f;
                }
            }
        }
        for (; r < r1; r += 4) {
            floatx4 v = *(const floatx4 *)(X + (long)r * Cc + c0);
#pragma unroll
            for (int u = 0; u < 4; u++) stat_push(st[u], v[u]);
        }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) sh[wave][lane * 4 + u] = st[u];
    __syncthreads();
    int col = blockIdx.x * 256 + threadIdx.x;
    if (col < Cc) {
        ColStat a = stat_merge(stat_merge(sh[0][threadIdx.x], sh[1][threadIdx.x]),
                               stat_merge(sh[2][threadIdx.x], sh[3][threadIdx.x]));
        part[(long)blockIdx.y * Cc + col] = a;
    }
}

// Per-column finalize: fold the chunk partials, then the reference backward's per-row scalars.
// Block = 16 columns x 16 partial groups: group p folds partials p, p+16, ... (coalesced 256-byte rows),
// the 16 group results are merged in a fixed order (deterministic), then one thread per column
// evaluates the scalars. coef[col] = {m, rs, g*r, gsq, gs, share, dg, loss_row}; lossp[block] is the
// block's sum of loss_row (summed by the gradient pass).
constexpr int kFinCols = 16;
constexpr int kFinGroups = 256 / kFinCols;
__global__ __launch_bounds__(256) void chain_finalize_kernel(const ColStat *part, int nchunks, int R, int Cc,
                                                              const float *g, float *coef, float *dg, float *lossp) {
    __shared__ ColStat sh[kFinGroups][kFinCols];
    __shared__ float lsum[kFinCols];
    const int cl = threadIdx.x % kFinCols, grp = threadIdx.x / kFinCols;
    const int col = blockIdx.x * kFinCols + cl;
    ColStat a{-FLT_MAX, 0.0f, 0.0f, 0.0f};
    if (col < Cc)
        for (int k0 = grp; k0 < nchunks; k0 += 8 * kFinGroups) {   // 8 loads in flight, then the merges
            ColStat v[8];
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (k0 + u * kFinGroups < nchunks) v[u] = part[(long)(k0 + u * kFinGroups) * Cc + col];
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (k0 + u * kFinGroups < nchunks) a = stat_merge(a, v[u]);
        }
    sh[grp][cl] = a;
    __syncthreads();
    if (grp == 0) {
        float lrow = 0.0f;
        if (col < Cc) {
#pragma unroll
            for (int k = 1; k < kFinGroups; k++) a = stat_merge(a, sh[k][cl]);
            const float eps = 1e-6f;
            const float rR = 1.0f / (float)R;
            float rs = 1.0f / a.s;
            float sumS = a.s * rs;             // Sum_j e_j * rs
            float sq = a.q * (rs * rs);        // Sum_j (e_j * rs)^2
            float q = sq * rR;
            float T = sqrtf(q + eps);
            float r = 1.0f / T;
            float gi = g[col];
            float gR = gi * sumS;
            float gT = ((-gR) * r) * r;
            float gu = gT * (1.0f / (2.0f * T));
            float gsq = gu * rR;
            float gRs = (gi * r) * a.s + 2.0f * gsq * (rs * a.q);
            float gs = ((-gRs) * rs) * rs;
            float gm = -(AH_LN2 * AH_INV_LN2) * (rs * gRs + gs * a.s);
            float share = gm * (1.0f / a.t);
            float *cf = coef + (long)col * 8;
            lrow = gi * (r * sumS);
            *(floatx4 *)cf = floatx4{a.m, rs, gi * r, gsq};
            *(floatx4 *)(cf + 4) = floatx4{gs, share, r * sumS, lrow};
            dg[col] = r * sumS;
        }
        lsum[cl] = lrow;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float acc = 0.0f;
        for (int k = 0; k < kFinCols; k++) acc += lsum[k];
        lossp[blockIdx.x] = acc;
    }
}

// Pass 2: dX[j, i] from X[j, i] and the per-column scalars; each wave loads its 8 rows before
// computing. Block (0, 0) also sums the finalize blocks' loss partials in a fixed order.
__global__ __launch_bounds__(256) void chain_grad_kernel(const float *X, int R, int Cc, int rch, const float *coef,
                                                          float *dX, const float *lossp, int nlossp, float *loss) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (blockIdx.x == 0 && blockIdx.y == 0 && wave == 0) {
        float acc = 0.0f;
        for (int i = lane; i < nlossp; i += 64) acc += lossp[i];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
        if (lane == 0) loss[0] = acc;
    }
    const int c0 = blockIdx.x * 256 + lane * 4;
    if (c0 >= Cc) return;
    float m[4], rs[4], gr[4], gsq[4], gs[4], sh[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const floatx4 a = *(const floatx4 *)(coef + (long)(c0 + u) * 8);
        const floatx4 b = *(const floatx4 *)(coef + (long)(c0 + u) * 8 + 4);
        m[u] = a[0]; rs[u] = a[1]; gr[u] = a[2]; gsq[u] = a[3]; gs[u] = b[0]; sh[u] = b[1];
    }
    const int r0 = blockIdx.y * rch, r1 = min(R, r0 + rch);
    // 8 rows in flight per wave. X is read with ordinary loads: the stats pass has just streamed it, so
    // much of it is still in the Infinity Cache (a non-temporal load measured 20-30% slower here).
    for (int rb = r0 + wave; rb < r1; rb += 32) {
        floatx4 v[8];
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (rb + 4 * j < r1) v[j] = *(const floatx4 *)(X + (long)(rb + 4 * j) * Cc + c0);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if (rb + 4 * j >= r1) break;
            floatx4 o;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                float y = v[j][u];
                float e = fast_exp2((y - m[u]) * AH_INV_LN2);
                float S = e * rs[u];
                float t2 = gsq[u] * S;
                float gS = (gr[u] + t2) + t2;
                float ge = gS * rs[u] + gs[u];
                float gzs = ((ge * e) * AH_LN2) * AH_INV_LN2;
                o[u] = gzs + ((y == m[u]) ? sh[u] : 0.0f);
            }
            __builtin_nontemporal_store(o, (floatx4 *)(dX + (long)(rb + 4 * j) * Cc + c0));
        }
    }
}

// ── the chain in one pass over HBM: strips of X held on chip ──────────────────────
// Every softmax / RMS row of the chain is one column of X, and dg, the loss terms and dX of a column need only that column.
// A strip of 32 columns (128 bytes of a row: one cache line) is held on chip by `parts` workgroups of consecutive row
// ranges, up to 4096 rows (512 KiB) each: NS float4 slots per thread, 45 in VGPRs and the rest in LDS through LDS-DMA. Each
// workgroup takes its rows' column statistics (max, sum e, sum e^2, ties) while they land; with several parts they are
// exchanged once through memory, 512 bytes a part; then every workgroup evaluates the column's scalars and writes its rows
// of dX from the on-chip copy. HBM sees X read once and dX written once, where the three-kernel chain reads X twice.
//
// Bound by HBM, load phase then store phase. Strips of 16 columns, one workgroup of 8192 rows each, took 70.5 us for 8192 x
// 4096 with X in memory (49 us with X left in the Infinity Cache by the step before): 64-byte row segments use half of each
// line, and only a neighbour on the same XCD can use the rest.
//
// Waiting for the other parts is bounded: a workgroup that has polled `spin` times takes the missing parts' statistics from X
// itself, in the same order, so the result is the same and nothing depends on the parts running together. That holds in place
// too (dX over X, dg over g): the workgroup says that it reads before it looks again which parts are missing, and those wait
// for it before they write (it runs, and itself waits for nobody meanwhile); dg is stored by the last part to leave, after
// every part has read g.
//
// Thread t owns columns 4 (t & 7) .. + 3 of rows (t >> 3) + 64 i of its range: slot 0 the last, possibly partial 64 rows,
// slots 1 .. nfull the whole ones. Every sum is a fixed tree (slots in order, then lanes by xor, waves in order, parts in
// order). Part 0 stores the strip's loss sum; the last strip to arrive (counter, zero before and after) adds them in order.
constexpr int kStripThreads = 512, kStripWaves = kStripThreads / 64, kStripCols = 32, kStripRows = kStripThreads / 8;
constexpr int kStripMaxRegs = 45, kStripMaxSlots = 64;   // float4 slots per thread in VGPRs; in all (19 in LDS: 152 KiB)
constexpr int kStripMaxParts = 16, kStripMaxPartsFull = 4;   // parts whose statistics fit beside the held rows in LDS
constexpr int kStripMaxStrips = 1024;                    // a handle's counters for ah_chain_step_noalloc
constexpr int kStripSpin = 1 << 14;
// A strip's arrival word: a bit for each part that has posted its statistics, and from bit 16 up the count of workgroups that
// read other parts' rows of X. Polls for those readers (some us each) end after kStripReaderSpin, several seconds.
constexpr int kStripReader = 1 << 16, kStripReaderSpin = 1 << 23;
static_assert(kStripMaxParts <= 16, "a bit for each part below the readers' count");

__device__ __forceinline__ float strip_tree_max(float v) {   // over the 8 lanes of a wave with equal lane & 7
    v = fmaxf(v, __shfl_xor(v, 8, 64));
    v = fmaxf(v, __shfl_xor(v, 16, 64));
    return fmaxf(v, __shfl_xor(v, 32, 64));
}
__device__ __forceinline__ float strip_tree_sum(float v) {
    v += __shfl_xor(v, 8, 64);
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

// A thread's running statistics of its four columns: the reference mt its exponentials are taken against (finite: -FLT_MAX
// or above, so that an entry of -inf adds exp2(-inf) = 0), sum e, sum e^2 and the exact running max, from -FLT_MAX. An
// element more than 2^60 above mt (where e^2 could overflow) first moves the reference to itself. The elements equal to the
// max are counted afterwards, and only where a lane met its running max again (a bit of `tie`, kept in scalar registers):
// counting them as they land took 5 of 17 vector operations per element, in a kernel whose vector work shows (8192 x 4096:
// 67.3 us with the count, 59.1 us without any statistics).
struct StripStat {
    float mt[4], se[4], sq[4], mr[4];
    uint64_t tie;
    __device__ __forceinline__ void init(const float (&ref)[4]) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            mt[u] = ref[u];
            se[u] = sq[u] = 0.0f;
            mr[u] = -FLT_MAX;
        }
        tie = 0;
    }
    __device__ __forceinline__ void push(const floatx4 &x) {
        float d[4];
#pragma unroll
        for (int u = 0; u < 4; u++) d[u] = (x[u] - mt[u]) * AH_INV_LN2;
        const float dm = fmaxf(fmaxf(d[0], d[1]), fmaxf(d[2], d[3]));
        if (__builtin_amdgcn_ballot_w64(dm > 60.0f)) {   // wave-uniform, never taken on ordinary data
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (d[u] > 60.0f) {
                    const float f = fast_exp2(-d[u]);
                    se[u] *= f;
                    sq[u] *= f * f;
                    mt[u] = x[u];
                    d[u] = 0.0f;
                }
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const float e = fast_exp2(d[u]);
            se[u] += e;
            sq[u] += e * e;
            tie |= __builtin_amdgcn_ballot_w64(x[u] == mr[u]);
            mr[u] = fmaxf(mr[u], x[u]);
        }
        // materialise the running values after every slot (left free, the compiler runs one sum over all slots before the
        // next, keeping every slot's e live in between)
        asm volatile("" : "+v"(se[0]), "+v"(se[1]), "+v"(se[2]), "+v"(se[3]), "+v"(sq[0]), "+v"(sq[1]), "+v"(sq[2]),
                     "+v"(sq[3]), "+v"(mr[0]), "+v"(mr[1]), "+v"(mr[2]), "+v"(mr[3]));
    }
    // the elements equal to the thread's max, counted over each(f) (f is called with every element of the thread) where any
    // lane of the wave may have more than one, or one of -FLT_MAX; else one set the max, or none did (-inf only, no element)
    template <class Each>
    __device__ __forceinline__ void count(float (&cnt)[4], Each &&each) const {
#pragma unroll
        for (int u = 0; u < 4; u++) cnt[u] = mr[u] > -FLT_MAX ? 1.0f : 0.0f;
        if (tie == 0) return;
#pragma unroll
        for (int u = 0; u < 4; u++) cnt[u] = 0.0f;
        each([&](const floatx4 &x) {
#pragma unroll
            for (int u = 0; u < 4; u++) cnt[u] += x[u] == mr[u] ? 1.0f : 0.0f;
        });
    }
    // the wave's statistics of its columns to red[..][wave][column]: max, then the sums rescaled to it, ties at it
    __device__ __forceinline__ void post(float (*red)[kStripWaves][kStripCols], int wave, int lane, const float (&cnt)[4]) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const float m = strip_tree_max(mr[u]);
            const float f = fast_exp2((mt[u] - m) * AH_INV_LN2);
            const float s = strip_tree_sum(se[u] * f), q = strip_tree_sum(sq[u] * (f * f));
            const float t = strip_tree_sum(mr[u] == m ? cnt[u] : 0.0f);
            if (lane < 8) {
                red[0][wave][4 * lane + u] = m;
                red[1][wave][4 * lane + u] = s;
                red[2][wave][4 * lane + u] = q;
                red[3][wave][4 * lane + u] = t;
            }
        }
    }
};

// n statistics of a column (max, sum e, sum e^2, ties, the sums against their own max) folded in order; at(k, i) reads them.
template <class At>
__device__ __forceinline__ void strip_fold(int n, At &&at, float (&o)[4]) {
    float m = at(0, 0);
    for (int i = 1; i < n; i++) m = fmaxf(m, at(0, i));
    float s = 0.0f, q = 0.0f, t = 0.0f;
    for (int i = 0; i < n; i++) {
        const float mi = at(0, i);
        const float f = fast_exp2((mi - m) * AH_INV_LN2);
        s += at(1, i) * f;
        q += at(2, i) * (f * f);
        t += mi == m ? at(3, i) : 0.0f;
    }
    o[0] = m; o[1] = s; o[2] = q; o[3] = t;
}

// i <= nfull, compared anew at each use: all 64 of a thread's comparisons kept for the later passes overflow the SGPRs.
__device__ __forceinline__ bool strip_in(int i, int nfull) {
    asm volatile("" : "+s"(nfull));
    return i <= nfull;
}

// part_rows: rows per part (a multiple of 64, at most 64 * NS; the last part may have fewer). stats: parts * 128 floats a
// strip. sync: two words a strip, arrivals and departures, zero before and after. in_place: dX or dg shares memory with X or g.
// Up to 16 slots two workgroups share a CU: 4 waves a SIMD, 128 VGPRs. MULTI: more than one part a strip (a strip of one part
// that jumps over the exchange's code takes 0.4 us more: 630 x 276 10.3 us for 9.8).
template <int NS, bool MULTI>
__global__ __launch_bounds__(kStripThreads, NS <= 16 ? 4 : 2) void chain_strip_kernel(const float *X, int R, int Cc, int parts, int part_rows,
                                                                     const float *g, float *dX, float *dg, float *stats,
                                                                     int *sync, float *lossp, int *counter, float *loss,
                                                                     int spin, int in_place) {
    constexpr int kRegs = NS < kStripMaxRegs ? NS : kStripMaxRegs, kLds = NS - kRegs, kProv = NS < 8 ? NS : 8;
    constexpr int kParts = NS > kStripMaxRegs ? kStripMaxPartsFull : kStripMaxParts;
    __shared__ __attribute__((aligned(1024))) floatx4 held[kLds > 0 ? kLds : 1][kStripThreads];
    __shared__ float red[4][kStripWaves][kStripCols];
    __shared__ float pstat[4][MULTI ? kParts : 1][kStripCols];
    __shared__ __attribute__((aligned(16))) float coef[6][kStripCols];   // dX factors A, B, column max, tie share, loss term, dg
    __shared__ int flag;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nstrips = (Cc + kStripCols - 1) / kStripCols;
    // runs of (strip, part) per XCD: a strip's parts start together, and neighbouring strips, which share lines where Cc is
    // no multiple of 32, meet in one L2
    const int L = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (L >= nstrips * parts) return;
    const int strip = MULTI ? L / parts : L, part = L - strip * parts;
    const int q = tid & 7, rl = tid >> 3, c0 = strip * kStripCols, col = c0 + 4 * q;
    const bool colok = col < Cc;   // Cc % 4 == 0: all four columns or none
    const int rbeg = part * part_rows, rows = min(part_rows, R - rbeg), nfull = (rows - 1) / kStripRows;
    const int row0 = nfull * kStripRows + rl;   // slot 0's row
    const bool ok0 = row0 < rows && colok;
    // Buffer accesses from the part's first row and the strip's first column: the lane's offset in one VGPR, the slot's row
    // offset (wave-uniform) in the scalar offset. Lanes without a row or column and slots past nfull get an offset past the
    // descriptor's size: loads give zeros, stores do nothing. The caller guarantees R * Cc * 4 < 2^31.
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    constexpr int kOut = (int)0x80000000;
    const long org = (long)rbeg * Cc + c0;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)(X + org), (short)0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t dr = __builtin_amdgcn_make_buffer_rsrc((void *)(dX + org), (short)0, 0x7fffffff, 0x00020000);
    const float gi = tid < kStripCols && c0 + tid < Cc ? g[c0 + tid] : 0.0f;   // before this part arrives
    const int voff = colok ? (rl * Cc + 4 * q) * 4 : kOut, voff0 = ok0 ? (row0 * Cc + 4 * q) * 4 : kOut;
    const int rstepB = kStripRows * Cc * 4;
    // 1. the rows: register slots first (they are consumed first), then the LDS slots
    floatx4 v[kRegs];
    v[0] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(xr, voff0, 0, 0));
    // the row offset is a running value advanced through an empty asm, here and for the stores, so that only the current one
    // is live (all of them kept overflow the SGPRs into VGPR lanes)
    int soff = 0;
#pragma unroll
    for (int i = 1; i < kRegs; i++) {
        v[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(xr, strip_in(i, nfull) ? voff : kOut, soff, 0));
        soff += rstepB;
        asm volatile("" : "+s"(soff));
    }
#pragma unroll
    for (int j = 0; j < kLds; j++) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void *)&held[j][wave * 64], 16,
                                                     strip_in(kRegs + j, nfull) ? voff : kOut, soff, 0, 0);
        soff += rstepB;
        asm volatile("" : "+s"(soff));
    }
    // 2. statistics while they land, against the max of the thread's first slots
    StripStat st;
    {
        float ref[4];
#pragma unroll
        for (int u = 0; u < 4; u++) ref[u] = ok0 ? fmaxf(-FLT_MAX, v[0][u]) : -FLT_MAX;
#pragma unroll
        for (int i = 1; i < kProv; i++)
            if (strip_in(i, nfull))
#pragma unroll
                for (int u = 0; u < 4; u++) ref[u] = fmaxf(ref[u], v[i][u]);
        st.init(ref);
    }
    if (ok0) st.push(v[0]);
#pragma unroll
    for (int i = 1; i < kRegs; i++)
        if (strip_in(i, nfull)) st.push(v[i]);
    if constexpr (kLds > 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's LDS-DMA has landed (each lane reads its own)
#pragma unroll 2
        for (int j = 0; j < kLds; j++) {
            if (kRegs + j > nfull) break;
            const floatx4 x = *(volatile floatx4 *)&held[j][tid];
            st.push(x);
        }
    }
    float cnt[4];
    st.count(cnt, [&](auto &&f) {
        if (ok0) f(v[0]);
#pragma unroll
        for (int i = 1; i < kRegs; i++)
            if (strip_in(i, nfull)) f(v[i]);
        for (int j = 0; j < kLds && kRegs + j <= nfull; j++) {
            const floatx4 x = *(volatile floatx4 *)&held[j][tid];
            f(x);
        }
    });
    st.post(red, wave, lane, cnt);
    __syncthreads();
    // 3. the part's column statistics, and the other parts'
    float own[4];
    if (tid < kStripCols) strip_fold(kStripWaves, [&](int k, int w) { return red[k][w][tid]; }, own);
    if constexpr (MULTI) {
        float *const mine = stats + ((long)strip * parts + part) * (4 * kStripCols);
        int *const arrive = sync + 2 * strip;
        if (wave == 0) {
            if (lane < kStripCols)
#pragma unroll
                for (int k = 0; k < 4; k++)
                    __hip_atomic_store(mine + k * kStripCols + lane, own[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // performed where the XCDs are coherent, before the arrival; g has been read
            asm volatile("s_waitcnt vmcnt(0)" :: "v"(gi) : "memory");
            if (lane == 0) {
                const int all = (1 << parts) - 1;
                int got = __hip_atomic_fetch_add(arrive, 1 << part, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) | 1 << part;
                for (int k = 0; k < spin && (got & all) != all; k++) {
                    __builtin_amdgcn_s_sleep(4);
                    got = __hip_atomic_load(arrive, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                const bool reads = (got & all) != all;
                if (reads) got = __hip_atomic_fetch_add(arrive, kStripReader, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                flag = (all & ~got) | (reads ? kStripReader : 0);
            }
        }
        __syncthreads();
        const int missing = __builtin_amdgcn_readfirstlane(flag);   // parts, and kStripReader where this one has said that it reads
        // one value a thread and pass, every load in flight at once (a thread that took its column's parts one after the
        // other paid 1.1 us a part: 8192 x 64 in 16 parts: 26.4 us, so 11.3)
        constexpr int kPer = kParts * 4 * kStripCols / kStripThreads;
        const float *const all = stats + (long)strip * parts * (4 * kStripCols);
        float got[kPer];
#pragma unroll
        for (int j = 0; j < kPer; j++)
            got[j] = tid + j * kStripThreads < parts * 4 * kStripCols
                         ? __hip_atomic_load(all + tid + j * kStripThreads, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0f;
#pragma unroll
        for (int j = 0; j < kPer; j++) {
            const int i = tid + j * kStripThreads;
            pstat[i / kStripCols % 4][i / (4 * kStripCols)][i % kStripCols] = got[j];
        }
        __syncthreads();
        if (missing & (kStripReader - 1)) {
            // the missing ones from X, slot for slot in the order their own workgroup takes them
            for (int p = 0; p < parts; p++) {
                if ((missing >> p & 1) == 0) continue;
                const int pb = p * part_rows, pr = min(part_rows, R - pb), pf = (pr - 1) / kStripRows, r0 = pf * kStripRows + rl;
                const bool pok = r0 < pr && colok;
                const float *const px = X + (long)pb * Cc + col;
                auto at = [&](int i) { return colok ? *(const floatx4 *)(px + (long)((i - 1) * kStripRows + rl) * Cc) : (floatx4){}; };
                const floatx4 x0 = pok ? *(const floatx4 *)(px + (long)r0 * Cc) : (floatx4){};
                float ref[4];
#pragma unroll
                for (int u = 0; u < 4; u++) ref[u] = pok ? fmaxf(-FLT_MAX, x0[u]) : -FLT_MAX;
                for (int i = 1; i < kProv && i <= pf; i++) {
                    const floatx4 x = at(i);
#pragma unroll
                    for (int u = 0; u < 4; u++) ref[u] = fmaxf(ref[u], x[u]);
                }
                StripStat o;
                o.init(ref);
                if (pok) o.push(x0);
                for (int i = 1; i <= pf; i++) o.push(at(i));
                o.count(cnt, [&](auto &&f) {
                    if (pok) f(x0);
                    for (int i = 1; i <= pf; i++) f(at(i));
                });
                __syncthreads();   // red is read by the fold before
                o.post(red, wave, lane, cnt);
                __syncthreads();
                if (tid < kStripCols) {
                    float f[4];
                    strip_fold(kStripWaves, [&](int k, int w) { return red[k][w][tid]; }, f);
#pragma unroll
                    for (int k = 0; k < 4; k++) pstat[k][p][tid] = f[k];
                }
            }
        }
        if (tid < kStripCols) strip_fold(parts, [&](int k, int p) { return pstat[k][p][tid]; }, own);
        if (tid == 0) {
            // every thread has its values of X by the fold's last barrier
            if (missing >= kStripReader) __hip_atomic_fetch_add(arrive, -kStripReader, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (in_place)
                for (int k = 0; k < kStripReaderSpin && __hip_atomic_load(arrive, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= kStripReader; k++)
                    __builtin_amdgcn_s_sleep(4);
        }
    }
    // 4. the column's scalars (chain_finalize's rules), the same in every part
    if (tid < kStripCols) {
        const int c = c0 + tid;
        const bool live = c < Cc;
        const float mm = own[0], s_ = own[1], q_ = own[2], t_ = own[3];
        const float eps = 1e-6f, rR = 1.0f / (float)R;
        const float r_s = 1.0f / s_;
        const float sumS = s_ * r_s;
        const float sqq = q_ * (r_s * r_s);
        const float qm = sqq * rR;
        const float T = sqrtf(qm + eps);
        const float r = 1.0f / T;
        const float gR = gi * sumS;
        const float gT = ((-gR) * r) * r;
        const float gu = gT * (1.0f / (2.0f * T));
        const float gsq_ = gu * rR;
        const float gRs = (gi * r) * s_ + 2.0f * gsq_ * (r_s * q_);
        const float gs_ = ((-gRs) * r_s) * r_s;
        const float gm = -(AH_LN2 * AH_INV_LN2) * (r_s * gRs + gs_ * s_);
        // dX = e * (gr * r_s + gs) + e^2 * (2 gsq r_s^2), plus the tie share where x is the max: the per-element backward
        // of S = e * r_s through sum e and sum S^2, with its per-column factors gathered (the reference's op order rounds
        // them per element; the difference is at f32 rounding)
        coef[0][tid] = (gi * r) * r_s + gs_;
        coef[1][tid] = 2.0f * gsq_ * (r_s * r_s);
        coef[2][tid] = mm;
        coef[3][tid] = gm * (1.0f / t_);
        coef[4][tid] = live ? gi * (r * sumS) : 0.0f;
        coef[5][tid] = r * sumS;
        if (!MULTI && live) dg[c] = r * sumS;
    }
    __syncthreads();
    // the last part to leave (every one has arrived by then) stores dg and clears the words for the next launch: one wave's
    // work, not wave 0's, which takes the loss's ticket behind its stores
    if (MULTI && wave == kStripWaves - 1) {
        int gone = 0;
        if (lane == 0) gone = __hip_atomic_fetch_add(sync + 2 * strip + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_readfirstlane(gone) == parts - 1) {
            if (lane < kStripCols && c0 + lane < Cc) dg[c0 + lane] = coef[5][lane];
            if (lane < 2) __hip_atomic_store(sync + 2 * strip + lane, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // 5. dX from the held rows
    {
        const floatx4 a = *(const floatx4 *)&coef[0][4 * q], b = *(const floatx4 *)&coef[1][4 * q],
                      mx = *(const floatx4 *)&coef[2][4 * q], sh = *(const floatx4 *)&coef[3][4 * q];
        auto put = [&](const floatx4 &x, int off, int soff) {
            floatx4 o;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const float e = fast_exp2((x[u] - mx[u]) * AH_INV_LN2);
                o[u] = (a[u] + b[u] * e) * e;
            }
            // a column's maxima are few: most slots of a wave hold none
            if (__builtin_amdgcn_ballot_w64(x[0] == mx[0]) | __builtin_amdgcn_ballot_w64(x[1] == mx[1]) |
                __builtin_amdgcn_ballot_w64(x[2] == mx[2]) | __builtin_amdgcn_ballot_w64(x[3] == mx[3])) {
#pragma unroll
                for (int u = 0; u < 4; u++) o[u] += x[u] == mx[u] ? sh[u] : 0.0f;
            }
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, o), dr, off, soff, 0);
            // Wait states after the 16-byte store before anything may rewrite its data registers: without them a VALU
            // write two instructions later, behind a v_readlane of a spilled SGPR, reached memory in some lanes.
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_nop 4" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        put(v[0], voff0, 0);
        soff = 0;
#pragma unroll
        for (int i = 1; i < kRegs; i++) {
            if (strip_in(i, nfull)) put(v[i], voff, soff);
            soff += rstepB;
            asm volatile("" : "+s"(soff));
        }
        // the LDS slots through volatile loads: else the compiler may keep an earlier pass's reads live for this one
#pragma unroll 2
        for (int j = 0; j < kLds; j++) {
            if (kRegs + j > nfull) break;
            const floatx4 x = *(volatile floatx4 *)&held[j][tid];
            put(x, voff, soff);
            soff += rstepB;
            asm volatile("" : "+s"(soff));
        }
    }
    // 6. loss: the strip's 32 terms in column order, then the strips in order by the last to arrive
    if (part != 0) return;
    if (tid == 0) {
        float a = 0.0f;
        for (int c = 0; c < kStripCols; c++) a += coef[4][c];
        __hip_atomic_store(lossp + strip, a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        flag = ticket_take_atomic_partials(counter);   // lossp[] is written and read as atomics
    }
    __syncthreads();
    if (flag != nstrips - 1 || wave != 0) return;
    const int per = (nstrips + 63) / 64;
    float a = 0.0f;
    for (int k = 0; k < per; k++) {
        const int s2 = lane * per + k;
        if (s2 < nstrips) a += __hip_atomic_load(lossp + s2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    a = wave_sum(a);
    if (lane == 0) {
        loss[0] = a;
        __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Parts per strip and rows per part: the fewest parts of 64 slots that hold the rows (a plan of more than kStripMaxPartsFull
// parts of more than 45 slots does not fit), then more while the workgroups stay within one per CU and each keeps 8 slots (512
// rows). Two workgroups per CU: 4096 x 4096 34.7 us for 31.8, 3008 x 2048 19.9 for 18.4; parts of 256 rows: 512 x 2048 9.3 us
// for 8.8, 1024 x 64 8.6 for 9.8. Against the three kernels this is faster at every shape measured of at most one workgroup
// per CU, from 64 x 64 (6.1 us for 11.3) over 4096 x 64 (10.5 for 14.8), 2048 x 2048 (15.8 for 17.4), 16384 x 64 (13.9 for
// 14.5) and 16384 x 1024 (34.5 for 44.9) to 8192 x 4096. Parts of many rows fill their CU, so one more than 256 of them makes
// a second round, and a round neither loads nor stores all the time: 7000 x 4100 (258 workgroups) 96 us for 74 with X in
// memory and 74 for 71 with it in the Infinity Cache, 8192 x 5120 111 for 104 and 110 for 86, 7000 x 8192 145 for 128 and 142
// for 122; strips of one part and up to 48 slots are on even (3000 x 8196 75 for 71 and 59 for 68). The three kernels take
// those, unless X outgrows the Infinity Cache, which serves their second read of it (16000 x 4096 132 for 148), and X of a few
// rows on more than two rounds (2 x 27724 19.0 for 15.8).
struct StripPlan {
    int parts, rows;
};
static StripPlan strip_plan(int R, int Cc) {
    const int strips = (Cc + kStripCols - 1) / kStripCols;
    auto slots = [&](int parts) { return ((R + parts - 1) / parts + kStripRows - 1) / kStripRows; };
    int parts = 1;
    while (parts < kStripMaxParts && slots(parts) > kStripMaxSlots) parts++;
    while (parts < kStripMaxParts && strips * (parts + 1) <= 256 && slots(parts + 1) >= 8) parts++;
    const int rows = slots(parts) * kStripRows;
    return {(R + rows - 1) / rows, rows};
}

bool chain_resident_fits(int R, int Cc) {
    if (R <= 0 || Cc <= 0 || Cc % 4 || (long)R * Cc * 4 >= (1L << 31)) return false;
    if ((Cc + kStripCols - 1) / kStripCols > kStripMaxStrips) return false;
    const StripPlan p = strip_plan(R, Cc);
    const int strips = (Cc + kStripCols - 1) / kStripCols, slots = p.rows / kStripRows;
    if (slots > (p.parts <= kStripMaxPartsFull ? kStripMaxSlots : kStripMaxRegs)) return false;
    if (R < 8 && strips > 512) return false;
    const bool rounds = strips * p.parts > 256 && slots > (p.parts > 1 ? 32 : 48);
    return !rounds || (Cc % kStripCols == 0 && (long)R * Cc * 4 > 250000000L);
}

template <int NS, bool MULTI>
static void launch_strip_t(const float *X, const float *g, int R, int Cc, const StripPlan &p, float *stats, int *sync,
                           float *lossp, int *counter, float *dX, float *dg, float *loss, int spin, int in_place, hipStream_t s) {
    const int wgs = (Cc + kStripCols - 1) / kStripCols * p.parts;
    hipLaunchKernelGGL((chain_strip_kernel<NS, MULTI>), dim3((wgs + 7) / 8 * 8), dim3(kStripThreads), 0, s, X, R, Cc, p.parts, p.rows, g,
                       dX, dg, stats, sync, lossp, counter, loss, spin, in_place);
}
template <int NS>
static void launch_strip(const float *X, const float *g, int R, int Cc, const StripPlan &p, float *stats, int *sync, float *lossp,
                         int *counter, float *dX, float *dg, float *loss, int spin, int in_place, hipStream_t s) {
    if (p.parts > 1) launch_strip_t<NS, true>(X, g, R, Cc, p, stats, sync, lossp, counter, dX, dg, loss, spin, in_place, s);
    else launch_strip_t<NS, false>(X, g, R, Cc, p, stats, sync, lossp, counter, dX, dg, loss, spin, in_place, s);
}

hipError_t chain_resident(const float *X, const float *g, int R, int Cc, float *arrays, int *sync, int *counter, float *dX,
                          float *dg, float *loss, int spin, hipStream_t s) {
    if (!chain_resident_fits(R, Cc)) return hipErrorInvalidValue;
    const StripPlan p = strip_plan(R, Cc);
    const int strips = (Cc + kStripCols - 1) / kStripCols, slots = p.rows / kStripRows;
    float *lossp = arrays + (p.parts > 1 ? (long)strips * p.parts * 4 * kStripCols : 0);
    // dX or dg over X or g (over part of one: undefined)
    const uintptr_t nx = (uintptr_t)R * Cc * 4, ng = (uintptr_t)Cc * 4;
    auto meet = [](const float *a, uintptr_t na, const float *b, uintptr_t nb) {
        return (uintptr_t)a < (uintptr_t)b + nb && (uintptr_t)b < (uintptr_t)a + na;
    };
    const int in_place = meet(dX, nx, X, nx) || meet(dg, ng, g, ng);
#define AH_STRIP(n) launch_strip<n>(X, g, R, Cc, p, arrays, sync, lossp, counter, dX, dg, loss, spin, in_place, s)
    if (slots <= 4) AH_STRIP(4);
    else if (slots <= 8) AH_STRIP(8);
    else if (slots <= 16) AH_STRIP(16);
    else if (slots <= 32) AH_STRIP(32);
    else if (slots <= kStripMaxRegs) AH_STRIP(kStripMaxRegs);
    else AH_STRIP(kStripMaxSlots);
#undef AH_STRIP
    return hipGetLastError();
}

// ── step tail: bias SGD for several parameters + loss finalize, in one launch ─────
// Each accumulator element (or partial-row entry) is read and re-zeroed by the thread that sums it,
// leaving the accumulators ready for the next step's atomics or partial stores (no zero-fill launch).
__device__ __forceinline__ float block_sum_512(float v, float *red) {   // fixed order: waves, then 8 slots
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7]));
}

__global__ __launch_bounds__(512) void tail_kernel(TailArgs t) {
    static_assert(kTailCols * kTailChunks == 512, "tail block is 512 threads");
    // The loss has a block of its own (the last), so its reduction runs beside the parameters' instead
    // of ahead of one block's share of them.
    const int ncol = gridDim.x - (t.loss_mode != 0 ? 1 : 0);
    if ((int)blockIdx.x == ncol) {
        __shared__ float red[8];
        if (t.loss_mode == 1 && t.loss_parts > 0) {
            // per-wave partials, summed in a fixed order, then the f16(acc) narrowing (lower.go:712)
            float acc = 0.0f;
            int i = threadIdx.x;
            for (; i + 7 * 512 < t.loss_parts; i += 8 * 512) {   // 8 loads in flight, then the zeroing
                float v[8];
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = t.lossacc[i + j * 512];
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    acc += v[j];
                    t.lossacc[i + j * 512] = 0.0f;
                }
            }
            for (; i < t.loss_parts; i += 512) {
                acc += t.lossacc[i];
                t.lossacc[i] = 0.0f;
            }
            acc = block_sum_512(acc, red);
            if (threadIdx.x == 0) {
                t.loss_out[0] = q16(acc) * t.loss_scale;
                if (t.loss_sum) t.loss_sum[0] = acc;
            }
        } else if (t.loss_mode == 1) {
            if (threadIdx.x == 0) {
                if (t.loss_sum) t.loss_sum[0] = t.lossacc[0];
                t.loss_out[0] = q16(t.lossacc[0]) * t.loss_scale;   // f16(acc) narrowing, lower.go:712
                t.lossacc[0] = 0.0f;
            }
        } else if (t.loss_mode == 2) {
            float acc = 0.0f;
            for (int i = threadIdx.x; i < t.nrow; i += 512) acc += t.rowloss[i];
            acc = block_sum_512(acc, red);
            if (threadIdx.x == 0) t.loss_out[0] = acc * t.loss_scale;
        }
        return;
    }
    // kTailCols consecutive elements per block pass, so a half-wave reads 128 contiguous bytes of a
    // partial row; the rows of a partial-row accumulator are split into kTailChunks chunks (up to 16
    // loads in flight per thread), and the chunk sums are combined in a fixed order, so the result is
    // deterministic.
    long total = 0;
    for (int s = 0; s < t.nseg; s++) total += t.seg[s].n;
    __shared__ float part[kTailChunks][kTailCols];
    const int e = threadIdx.x % kTailCols, q = threadIdx.x / kTailCols;
    for (long base = (long)blockIdx.x * kTailCols; base < total; base += (long)ncol * kTailCols) {
        const long i = base + e;
        long k = i;
        int s = 0;
        if (i < total)
            while (k >= t.seg[s].n) { k -= t.seg[s].n; s++; }
        const TailSeg &g = t.seg[s];
        // the parameter's old value is loaded with the gradient partials, not after their sum
        const float pold = (q == 0 && i < total) ? g.p[k] : 0.0f;
        float a = 0.0f;
        if (i < total) {
            if (g.acc_rows > 0) {
                const int rq = (g.acc_rows + kTailChunks - 1) / kTailChunks, r0 = q * rq;
                const int r1 = min(r0 + rq, g.acc_rows);
                float *const col = g.acc + k;
                float p[16] = {};
                for (int r = r0; r < r1; r += 16) {   // rows past r1 are predicated off, so p[] stays in registers
                    float v[16];
#pragma unroll
                    for (int j = 0; j < 16; j++) v[j] = r + j < r1 ? col[(long)(r + j) * g.acc_ld] : 0.0f;
#pragma unroll
                    for (int j = 0; j < 16; j++) {
                        p[j] += v[j];
                        if (r + j < r1 && !g.keep) col[(long)(r + j) * g.acc_ld] = 0.0f;
                    }
                }
#pragma unroll
                for (int w = 8; w > 0; w >>= 1)
#pragma unroll
                    for (int j = 0; j < w; j++) p[j] += p[j + w];
                a = p[0];
            } else if (q == 0) {
                a = g.acc[k];
                if (!g.keep) g.acc[k] = 0.0f;
            }
        }
        part[q][e] = a;
        __syncthreads();
        if (q == 0 && i < total) {
            float sum = 0.0f;
#pragma unroll
            for (int c = 0; c < kTailChunks; c++) sum += part[c][e];
            const float gv = g.scale * sum;
            if (g.gout) g.gout[k] = gv;
            float w = pold - t.lr * gv;
            asm volatile("" : "+v"(w));   // the f16 copy is f16 of the stored f32 value
            g.p[k] = w;
            if (g.p16) g.p16[k] = (half_t)w;
        }
        __syncthreads();
    }
}

hipError_t step_tail(const TailArgs &t, hipStream_t s) {
    long total = 0;
    for (int i = 0; i < t.nseg; i++) total += t.seg[i].n;
    int blocks = (int)std::min<long>(std::max<long>((total + kTailCols - 1) / kTailCols, 1), 2048);
    if (t.loss_mode != 0) blocks++;   // the loss block
    hipLaunchKernelGGL(tail_kernel, dim3(blocks), dim3(kTailCols * kTailChunks), 0, s, t);
    return hipGetLastError();
}

// ── host launchers ──────────────────────────────────────────────────────────

static int grid_for(long n) {
    long g = (n + 255) / 256;
    return (int)(g < 2048 ? (g < 1 ? 1 : g) : 2048);
}

hipError_t fill_f32(float *p, long n, float v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(fill_f32_kernel, dim3(grid_for(n)), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}
hipError_t fill_hash(float *p, half_t *p16, long n, uint32_t seed, float amp, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(fill_hash_kernel, dim3(grid_for(n)), dim3(256), 0, s, p, p16, n, seed, amp);
    return hipGetLastError();
}
hipError_t cast_f32_f16(const float *src, half_t *dst, long n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(cast_f32_f16_kernel, dim3(grid_for(n)), dim3(256), 0, s, src, dst, n);
    return hipGetLastError();
}
hipError_t sgd_update(float *p, const float *g, long n, float lr, float scale, half_t *p16, float *gout,
                      hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(sgd_kernel, dim3(grid_for(n)), dim3(256), 0, s, p, g, n, lr, scale, p16, gout);
    return hipGetLastError();
}
hipError_t colsum_add(const float *G, int M, int N, long ld, float *out, hipStream_t s) {
    if (M <= 0 || N <= 0) return hipSuccess;
    int rpb = 64;
    dim3 grid((N + 63) / 64, (M + rpb - 1) / rpb);
    hipLaunchKernelGGL(colsum_kernel, grid, dim3(256), 0, s, G, M, N, ld, rpb, out);
    return hipGetLastError();
}
hipError_t softmax_ce(const float *z, const int32_t *labels, int B, int C, float a, float *dz, float *rowloss,
                      hipStream_t s, float *loss, float *ws) {
    if (B <= 0) return hipSuccess;
    if (loss && !ws) return hipErrorInvalidValue;
    static_assert(kSoftmaxWsFloats >= kSmSlots + 2 * kSmBlocks && kSoftmaxWsFloats >= kSmSlots + kSmLongBlocks, "one slot a workgroup");
    if (C <= 1024) {
        const int waves = std::min(kSmWaves, (B + kSmBlocks - 1) / kSmBlocks);
        const dim3 grid(std::min(kSmBlocks, (B + waves - 1) / waves)), block(64 * waves);
#define AH_SM(n) hipLaunchKernelGGL(softmax_ce_kernel<n>, grid, block, 0, s, z, labels, B, C, a, dz, rowloss, loss, ws)
        if (C <= 64) AH_SM(1);
        else if (C <= 128) AH_SM(2);
        else if (C <= 256) AH_SM(4);
        else if (C <= 512) AH_SM(8);
        else AH_SM(16);
#undef AH_SM
    } else if (C <= 16 * kSmWideThreads) {
        const dim3 grid(std::min(2 * kSmBlocks, B)), block(kSmWideThreads);
#define AH_SM(n) hipLaunchKernelGGL(softmax_ce_wide_kernel<n>, grid, block, 0, s, z, labels, B, C, a, dz, rowloss, loss, ws)
        if (C <= 4 * kSmWideThreads) AH_SM(4);
        else if (C <= 8 * kSmWideThreads) AH_SM(8);
        else AH_SM(16);
#undef AH_SM
    } else {
        hipLaunchKernelGGL(softmax_ce_long_kernel, dim3(loss ? std::min(kSmLongBlocks, (B + 3) / 4) : (B + 3) / 4), dim3(256), 0, s, z,
                           labels, B, C, a, dz, rowloss, loss, ws);
    }
    return hipGetLastError();
}
int softmax_ce_cols_blocks(int B) {
    const int b = (B + kSmWaves - 1) / kSmWaves;
    return b < kSoftmaxColsMaxBlocks ? (b < 1 ? 1 : b) : kSoftmaxColsMaxBlocks;
}
hipError_t softmax_ce_cols(const float *z, const int32_t *labels, int B, int C, float a, float *dz, float *rowloss,
                           float *part, hipStream_t s) {
    if (B <= 0) return hipSuccess;
    const dim3 grid(softmax_ce_cols_blocks(B)), block(64 * kSmWaves);
    if (C <= 64) hipLaunchKernelGGL(softmax_ce_cols_kernel<1>, grid, block, 0, s, z, labels, B, C, a, dz, rowloss, part);
    else if (C <= 128) hipLaunchKernelGGL(softmax_ce_cols_kernel<2>, grid, block, 0, s, z, labels, B, C, a, dz, rowloss, part);
    else if (C <= 256) hipLaunchKernelGGL(softmax_ce_cols_kernel<4>, grid, block, 0, s, z, labels, B, C, a, dz, rowloss, part);
    else if (C <= 512) hipLaunchKernelGGL(softmax_ce_cols_kernel<8>, grid, block, 0, s, z, labels, B, C, a, dz, rowloss, part);
    else if (C <= kSoftmaxColsMaxC) hipLaunchKernelGGL(softmax_ce_cols_kernel<16>, grid, block, 0, s, z, labels, B, C, a, dz, rowloss, part);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}
hipError_t mse_finalize(const float *acc, float scale, float *out, hipStream_t s) {
    hipLaunchKernelGGL(mse_finalize_kernel, dim3(1), dim3(64), 0, s, acc, scale, out);
    return hipGetLastError();
}

// Workspace: from float 64 either path's arrays; then the strip kernel's counters, the loss's in a line of its own and two a
// strip, zero before the first call and left zero by every call (the three-kernel path touches none). ah_chain_step_noalloc,
// whose arrays serve every shape and every handle of a GPU, passes its handle's counters.
constexpr long kChainHead = 64, kChainLossSync = 32;
long chain_array_floats(int R, int Cc) {
    int nch = (R + kChainStatsRows - 1) / kChainStatsRows;
    const long three = (long)nch * Cc * 4 + (long)Cc * 8 + (Cc + kFinCols - 1) / kFinCols;
    const long strips = (Cc + kStripCols - 1) / kStripCols;   // their loss terms, and the parts' statistics
    return kChainHead + std::max(three, chain_resident_fits(R, Cc) ? strips * (1 + 4L * kStripCols * strip_plan(R, Cc).parts) : 0L);
}
long chain_sync_ints(int Cc) { return kChainLossSync + 2L * ((Cc + kStripCols - 1) / kStripCols); }
long chain_sync_max_ints() { return chain_sync_ints(kStripMaxStrips * kStripCols); }
long chain_workspace_floats(int R, int Cc) { return chain_array_floats(R, Cc) + chain_sync_ints(Cc); }

hipError_t chain_step(const float *X, const float *g, int R, int Cc, float *work, float *dX, float *dg, float *loss,
                      hipStream_t s, int phase, int *sync, int spin) {
    if (Cc % 4 != 0 || R <= 0) return hipErrorInvalidValue;
    if (phase < 0 && chain_resident_fits(R, Cc)) {
        if (!sync) sync = (int *)(work + chain_array_floats(R, Cc));
        return chain_resident(X, g, R, Cc, work + kChainHead, sync + kChainLossSync, sync, dX, dg, loss, spin < 0 ? kStripSpin : spin, s);
    }
    work += kChainHead;
    const int nch = (R + kChainStatsRows - 1) / kChainStatsRows;
    const int nfin = (Cc + kFinCols - 1) / kFinCols;
    ColStat *part = (ColStat *)work;
    float *coef = work + (long)nch * Cc * 4;
    float *lossp = coef + (long)Cc * 8;
    if (phase < 0 || phase == 0)
        hipLaunchKernelGGL(chain_stats_kernel, dim3((Cc + 255) / 256, nch), dim3(256), 0, s, X, R, Cc, kChainStatsRows, part);
    if (phase < 0 || phase == 1)
        hipLaunchKernelGGL(chain_finalize_kernel, dim3(nfin), dim3(256), 0, s, part, nch, R, Cc, g, coef, dg, lossp);
    if (phase < 0 || phase == 2) {
        int nch2 = (R + kChainGradRows - 1) / kChainGradRows;
        hipLaunchKernelGGL(chain_grad_kernel, dim3((Cc + 255) / 256, nch2), dim3(256), 0, s, X, R, Cc, kChainGradRows,
                           coef, dX, lossp, nfin, loss);
    }
    return hipGetLastError();
}

}  // namespace ah

// ── config-5 chain without allocation ───────────────────────────────────────
// The chain's workspace (per-chunk column partials, per-column coefficients, loss partials) lives in a
// file-scope device array instead of a hipMalloc'd buffer, for callers that cannot allocate (graph
// capture, serving loops). Every GPU the library runs on holds its own copy of `scratch` at its own
// address until the process ends; host code must use the address hipGetSymbolAddress returned for the
// current device, never the array's name (which is only a host-side stand-in).
// The chain writes every workspace entry before reading it (chain_stats fills every chunk partial,
// chain_finalize every coefficient and loss partial; the strip kernel every strip's loss sum and every
// part's statistics), so nothing needs clearing between calls. The strip kernel's counters, which a launch
// takes from zero back to zero, are not here but with each device handle: its launches run one after another
// on its stream, whereas launches of two handles that overlap would leave shared counters wrong for good.
namespace ah {
namespace {
constexpr long kChainScratchFloats = 1L << 22;   // 16 MiB: R x Cc up to 16320 x 4096 (config 5, 8192 x 4096, needs 2.13M floats)
constexpr int kMaxDevices = 64;
static __device__ __align__(256) float scratch[kChainScratchFloats];
float *g_scratch_ptr[kMaxDevices];
}  // namespace

long chain_scratch_floats() { return kChainScratchFloats; }

// Looks up this device's copy of `scratch`, with `ordinal` the current device. Called once per device,
// from ah_open; later calls return the stored address.
hipError_t chain_scratch_init(int ordinal, float **out) {
    if (ordinal < 0 || ordinal >= kMaxDevices) return hipErrorInvalidDevice;
    // handles opened from several threads look the address up under one lock (the table is per process)
    static std::mutex mu;
    std::lock_guard<std::mutex> lock(mu);
    if (!g_scratch_ptr[ordinal]) {
        void *p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch_ptr[ordinal] = (float *)p;
    }
    *out = g_scratch_ptr[ordinal];
    return hipSuccess;
}

}  // namespace ah
