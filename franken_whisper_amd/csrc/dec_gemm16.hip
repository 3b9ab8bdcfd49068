// dec_gemm16.hip — gemv_f16 (nn.rs:2346-2460) for many rows at once, on the
// matrix units in the reference's own operation order (gfx950).
//
// dot_f16c (nn.rs:1983-2051) keeps 32 partial sums ("slots"): slot j is an FMA
// chain over element 32c + j of every 32-wide chunk c.  A product of depth one,
// v_mfma_f32_16x16x1_4b_f32, is exactly one FMA per accumulator (one rounding;
// checked bit for bit against fmaf, denormals, infinities and signed zeros
// among the operands), and its four blocks are four slots: 16 outputs x 16 rows
// of each, from 1 weight and 1 activation register.  So a chunk of 16 outputs x
// 16 rows is eight of them instead of 8,192 FMAs whose operands all come from
// registers filled by LDS: the vector kernel (k_gemv16) reads 4 LDS bytes per
// FMA, which bounds it, and re-reads the weights for every few rows.
//
// Layout: weights in k_gemv16's slot order (row, group of 8 / CPL chunks, lane
// p = kh * 8 + l with the slots 8 (kh * CPL + kk) + l, kk < CPL), 16 bytes a
// lane.  Wave part w of SW = 8 / CPL takes p = 4w .. 4w+3 as its four blocks, so
// a wave's load is 64 bytes of each of 16 rows; a block's 8 waves are 8 / SW
// output tiles that share the staged rows.  Rows (or their LayerNorm) are
// staged in LDS as [row][K + 4], permuted per chunk so a lane reads its CPL
// slots at once (conflict-free: a row is 4 banks on).
//
// Operand layouts of the 16x16x1 form: A lane l -> output l % 16, block l / 16;
// B lane l -> row l % 16, block l / 16; accumulator register 4 b + r of lane l ->
// block b, output 4 (l / 16) + r, row l % 16.
#include "fw_dec.h"

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int GX_K = 1280; // the widest rows: 16 of them in LDS

// LDS position of element e (0..31) of a chunk: lane p's CPL slots contiguous
template <int CPL>
__device__ __forceinline__ int gx_pos(int e) {
    const int k = e >> 3, l = e & 7;
    return ((k / CPL) * 8 + l) * CPL + (k % CPL);
}

template <int CPL, bool LN, bool KEYS>
__global__ void __launch_bounds__(512, 2) k_gemm16x(const uint16_t *__restrict__ Wp, const float *__restrict__ bias,
                                                    const float *__restrict__ x, float *y, int N, int K, int ns,
                                                    int ldy, int mode, const float *__restrict__ gelu_tab,
                                                    const float *__restrict__ lnw, const float *__restrict__ lnb,
                                                    fwhip_filter filt, int use_filter, const int *initialp,
                                                    unsigned long long *keys, int nkey) {
    static_assert(CPL == 2 || CPL == 4, "two or four slots a lane");
    constexpr int SW = 8 / CPL, NT = 8 / SW, CPG = 8 / CPL, LPR = 32 / CPL;
    constexpr int NV = CPL == 4 ? 4 : 16; // values a lane hands to the slot tree's last steps
    constexpr int BG = 5; // weight groups in flight
    extern __shared__ __align__(16) float sm[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int part = wave % SW, tl = wave / SW; // slot part, output tile of the block
    const int s0 = blockIdx.y * 16, sn = min(ns - s0, 16);
    const int ldx = K + 4;
    float *xs = sm, *vs = sm + (size_t)sn * ldx; // [sn][ldx]; [8 waves][NV][64]
    const int G = K / (32 * CPG);
    const int ntile = (N + 16 * NT - 1) / (16 * NT);
    const int initial = KEYS && use_filter ? *initialp : 0;
    const int p = part * 4 + (lane >> 4), srow = min(lane & 15, sn - 1);

    uint4 nxt[BG];
    auto load_batch = [&](int tile, int b) {
        const int row = min(tile * 16 * NT + tl * 16 + (lane & 15), N - 1);
        const uint4 *w = (const uint4 *)(Wp + (size_t)row * K) + p;
#pragma unroll
        for (int i = 0; i < BG; i++) {
            const int g = min(b * BG + i, G - 1); // past the last: re-read, unused
            // (the logits head's weights are read once per step: streamed)
            if constexpr (KEYS) nxt[i] = fw_ld_stream(w + (size_t)g * LPR);
            else nxt[i] = w[(size_t)g * LPR];
        }
    };
    // four values of a staged row
    auto put4 = [&](int row, int e0, float4 v) {
        float *d = xs + (size_t)row * ldx + (e0 & ~31);
        d[gx_pos<CPL>((e0 + 0) & 31)] = v.x;
        d[gx_pos<CPL>((e0 + 1) & 31)] = v.y;
        d[gx_pos<CPL>((e0 + 2) & 31)] = v.z;
        d[gx_pos<CPL>((e0 + 3) & 31)] = v.w;
    };
    int tile = blockIdx.x;
    if (tile < ntile) load_batch(tile, 0);
    if constexpr (LN) {
        // K <= 1280: five float4 groups per lane cover a row, one wave per row
        for (int r = wave; r < sn; r += 8) {
            float4 xv[5];
            bool ok[5];
#pragma unroll
            for (int q = 0; q < 5; q++) {
                const int i = lane + q * 64;
                ok[q] = i < (K >> 2);
                xv[q] = ((const float4 *)(x + (size_t)(s0 + r) * K))[ok[q] ? i : 0];
                if (!ok[q]) xv[q] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
            fw_ln_quant_vals<5>(xv, ok, nullptr, lnw, lnb, K, 0, nullptr, nullptr, lane);
#pragma unroll
            for (int q = 0; q < 5; q++)
                if (ok[q]) put4(r, (lane + q * 64) * 4, xv[q]);
        }
    } else {
        const int n4 = K >> 2, tot = sn * n4;
        constexpr int U = 5; // loads in flight
        for (int i0 = threadIdx.x; i0 < tot; i0 += 512 * U) {
            float4 v[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = min(i0 + u * 512, tot - 1), r = i / n4;
                v[u] = ((const float4 *)(x + (size_t)(s0 + r) * K))[i - r * n4];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = i0 + u * 512, r = i / n4;
                if (i < tot) put4(r, (i - r * n4) * 4, v[u]);
            }
        }
    }
    __syncthreads();
    for (; tile < ntile; tile += gridDim.x) {
        // residual values of this thread's outputs, read before the multiply
        constexpr int NO = (NT * 256 + 511) / 512;
        float yo[NO];
        if (mode == 1) {
#pragma unroll
            for (int q = 0; q < NO; q++) {
                const int i = threadIdx.x + q * 512, row = tile * 16 * NT + (i >> 8) * 16 + (i & 15), s = (i >> 4) & 15;
                yo[q] = i < NT * 256 && row < N && s < sn ? y[(size_t)(s0 + s) * ldy + row] : 0.0f;
            }
        }
        v16f acc[CPL];
#pragma unroll
        for (int kk = 0; kk < CPL; kk++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[kk][r] = 0.0f;
        for (int gb = 0; gb < G; gb += BG) {
            uint4 cur[BG];
#pragma unroll
            for (int i = 0; i < BG; i++) cur[i] = nxt[i];
            if (gb + BG < G) load_batch(tile, gb / BG + 1);
            else if (tile + (int)gridDim.x < ntile) load_batch(tile + gridDim.x, 0);
            const float *xc = xs + (size_t)srow * ldx + gb * CPG * 32 + p * CPL;
            // (guarded groups: as one straight line the compiler reads too far ahead, 58 against 44 us
            // for the logits head)
#pragma unroll
            for (int i = 0; i < BG; i++) {
                if (gb + i >= G) break;
                const uint32_t u[4] = {cur[i].x, cur[i].y, cur[i].z, cur[i].w};
#pragma unroll
                for (int cc = 0; cc < CPG; cc++) {
                    float xv[CPL];
                    const float *xp = xc + (i * CPG + cc) * 32;
                    if constexpr (CPL == 4) {
                        const float4 t = *(const float4 *)xp;
                        xv[0] = t.x; xv[1] = t.y; xv[2] = t.z; xv[3] = t.w;
                    } else {
                        const float2 t = *(const float2 *)xp;
                        xv[0] = t.x; xv[1] = t.y;
                    }
#pragma unroll
                    for (int kk = 0; kk < CPL; kk++) {
                        const int f = cc * CPL + kk;
                        const float wf = fw_h2f((uint16_t)(u[f >> 1] >> ((f & 1) * 16)));
                        acc[kk] = __builtin_amdgcn_mfma_f32_16x16x1f32(wf, xv[kk], acc[kk], 0, 0, 0);
                    }
                }
            }
        }
        // ---- slot tree: t_l = (a0 + a1) + (a2 + a3) over k, then ((t0 + t1) +
        // (t2 + t3)) + ((t4 + t5) + (t6 + t7)).  Part w holds kh = w / 2 and l =
        // 4 (w % 2) + block; what it can add by itself it adds, the rest meets
        // in LDS: vs[wave][value][lane], value = block * 4 + r (CPL 4: r).
        float *vw = vs + (size_t)wave * NV * 64 + lane;
        if constexpr (CPL == 4) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float t[4];
#pragma unroll
                for (int b = 0; b < 4; b++)
                    t[b] = (acc[0][b * 4 + r] + acc[1][b * 4 + r]) + (acc[2][b * 4 + r] + acc[3][b * 4 + r]);
                vw[r * 64] = (t[0] + t[1]) + (t[2] + t[3]);
            }
        } else {
#pragma unroll
            for (int r = 0; r < 16; r++) vw[r * 64] = acc[0][r] + acc[1][r];
        }
        __syncthreads();
        // NT tiles x 16 outputs x 16 rows; consecutive threads on consecutive outputs
#pragma unroll
        for (int q = 0; q < NO; q++) {
            const int i = threadIdx.x + q * 512;
            if (i >= NT * 256) break;
            const int o = i & 15, s = (i >> 4) & 15, tt = i >> 8, row = tile * 16 * NT + tt * 16 + o;
            const float *vb = vs + (size_t)tt * SW * NV * 64 + (o >> 2) * 16 + s; // lane (o / 4, s)
            const int r = o & 3;
            auto at = [&](int w, int b) { return vb[((size_t)w * NV + b * 4 + r) * 64]; };
            float v;
            if constexpr (CPL == 4) {
                v = at(0, 0) + at(1, 0);
            } else {
                float h[2];
#pragma unroll
                for (int lh = 0; lh < 2; lh++) {
                    float t[4];
#pragma unroll
                    for (int b = 0; b < 4; b++) t[b] = at(lh, b) + at(lh + 2, b);
                    h[lh] = (t[0] + t[1]) + (t[2] + t[3]);
                }
                v = h[0] + h[1];
            }
            const bool ok = row < N && s < sn;
            if (bias && ok) v = v + bias[row];
            if (ok) {
                float *yp = y + (size_t)(s0 + s) * ldy + row;
                if (mode == 1) *yp = yo[q] + v;
                else if (mode == 2) *yp = fw_gelu(v, gelu_tab);
                else *yp = v;
            }
            if constexpr (KEYS) {
                // 32-row key tiles: two 16-lane groups of consecutive tt; each
                // group's maximum meets the other's in LDS
                unsigned long long k = 0ull;
                if (ok && !(use_filter && dec_masked(row, filt, initial))) k = am_key(v, row);
                k = row16_max_u64(k);
                unsigned long long *ks = (unsigned long long *)(vs + (size_t)8 * NV * 64);
                if (o == 0) ks[tt * 16 + s] = k;
            }
        }
        if constexpr (KEYS) {
            __syncthreads();
            const unsigned long long *ks = (const unsigned long long *)(vs + (size_t)8 * NV * 64);
            if (threadIdx.x < (NT / 2) * 16) {
                const int kt = threadIdx.x >> 4, s = threadIdx.x & 15, kt0 = tile * (NT / 2) + kt;
                const unsigned long long a = ks[2 * kt * 16 + s], b = ks[(2 * kt + 1) * 16 + s];
                if (s < sn && kt0 < nkey) keys[(size_t)(s0 + s) * nkey + kt0] = a > b ? a : b;
            }
        }
        __syncthreads(); // vs is free
    }
}

template <int CPL, bool LN, bool KEYS>
void gx_go(hipStream_t st, int grid_cap, const uint16_t *Wp, const float *bias, const float *x, float *y, int N, int K,
           int ns, int ldy, int mode, const float *gelu_tab, const float *lnw, const float *lnb,
           const fwhip_filter &filt, int use_filter, const int *initialp, unsigned long long *keys, int nkey) {
    constexpr int NT = CPL, NV = CPL == 4 ? 4 : 16;
    const int rows = ns < 16 ? ns : 16;
    const size_t shm = ((size_t)rows * (K + 4) + (size_t)8 * NV * 64 + (KEYS ? 2 * NT * 16 : 0)) * sizeof(float);
    const int ntile = (N + 16 * NT - 1) / (16 * NT);
    hipLaunchKernelGGL((k_gemm16x<CPL, LN, KEYS>), dim3(ntile < grid_cap ? ntile : grid_cap, (ns + 15) / 16), dim3(512),
                       shm, st, Wp, bias, x, y, N, K, ns, ldy, mode, gelu_tab, lnw, lnb, filt, use_filter, initialp,
                       keys, nkey);
}

} // namespace

// Where the matrix form is the faster one (measured against k_gemv16 on MI355X,
// the same bits): the logits head from 6 rows on (51,866 x 1,280: 47 -> 43 us at
// 6, 55 -> 44 at 10, 91 -> 55 at 16, 220 -> 100 at 32; 4 rows 34 against 43), one
// block per CU walking the tiles (two: 49); the other matrices where rows x
// outputs fill the chip (10 rows: fc1 11.9 -> 10.9 us; 16: q/k/v 12.7 -> 11.9, fc1
// 15.1 -> 12.1; 32: cross q 13.9 -> 11.9, q/k/v 20.8 -> 12.4, fc1 28 -> 23; 320:
// d x d 68 -> 43, fc1 254 -> 152).  Rows longer than 1,280 (fc2) gained nothing.
// The other widths were not fitted, but they gain by the same thresholds: whole
// decodes of 6-16 streams at widths 384, 512, 768 and 1,024 1.01-1.19x, prompts of
// 4-200 rows 1.07-2.7x, one to five streams unchanged.  Argmax keys (a logits
// head) are formed in the eight-lane form alone: a vocabulary below 16,384 stays
// with the vector kernel.
bool fw_gemm16x_ok(int N, int K, int ns, bool keys) {
    const int lpr = fw_gemv16_lpr(N, K);
    if (K > GX_K || (lpr != 8 && lpr != 16) || K % (lpr == 8 ? 64 : 128) || (keys && lpr != 8)) return false;
    return N >= 16384 ? ns >= 6 : lpr == 16 && ns >= 10 && (long long)ns * N >= 40960 && (ns >= 40 || N > 1280);
}

// As fw_launch_gemv16 (the same operands, outputs and bits) where fw_gemm16x_ok.
void fw_launch_gemm16x(hipStream_t st, const uint16_t *Wp, const float *bias, const float *x, float *y, int N, int K,
                       int ns, int ldy, int mode, const float *gelu_tab, const float *lnw, const float *lnb,
                       const fwhip_filter *filt, const int *initialp, unsigned long long *keys, int n_cu) {
    fwhip_filter f;
    memset(&f, 0, sizeof f);
    if (filt) f = *filt;
    const int nkey = keys ? fw_gemv16_key_blocks(N, K) : 0, cap = N >= 16384 ? n_cu : 1 << 30;
#define GX(C_, L_, K_)                                                                                      \
    gx_go<C_, L_, K_>(st, cap, Wp, bias, x, y, N, K, ns, ldy, mode, gelu_tab, lnw, lnb, f, filt != nullptr, \
                      initialp, keys, nkey)
    if (fw_gemv16_lpr(N, K) == 8) { // (keys: the logits head)
        if (keys && lnw) GX(4, true, true);
        else if (keys) GX(4, false, true);
        else if (lnw) GX(4, true, false);
        else GX(4, false, false);
    } else {
        if (lnw) GX(2, true, false);
        else GX(2, false, false);
    }
#undef GX
}
