// enc_gemm.hip — the int8 plan's dense contractions on MFMA (gfx950).
//
// C[M,N] = A[M,K] x B[N,K]^T, i8 x i8 -> i32 (v_mfma_i32_32x32x32_i8).  The
// accumulators are exact integers, equal to the reference's maddubs sum minus
// 128*colsum (nn.rs:1537-1771) or its i8 dot (encoder.rs:2524-2606); epilogue
// ((f32)acc * s_x) * s_w (+ b) in the reference's association
// (nn.rs:1660-1700, encoder.rs:2573-2580).  (The f16-pair GEMMs are in
// enc_gemm_f16.hip.)
//
// Two kernels, the same bits: k_gemm_pi8, persistent blocks over 256 x 256, 256 x
// 128 or 128 x 128 tiles, which the encoder runs, and k_gemm_tile, a 128 x 128 tile
// a block with its epilogue on its own, to check the first against
// (FWHIP_GEMM_I8P=0).  In both, K advances 64 bytes per stage, global -> LDS
// directly, and the epilogue is a template parameter so its loops unroll and
// the accumulators stay in registers.
//
// Tile order: the hardware deals blocks round-robin to the 8 XCDs; block ids
// are mapped so each XCD gets a contiguous run of tiles, walked in groups of
// 8 M-tiles (N outer), so an XCD's L2 holds the A rows of its group and one B
// tile at a time.
//
// MFMA operand layouts (gfx950): A lane l -> row l%32, k block (l/32)*16
// bytes; B lane l -> col l%32, same k block; accumulator r of lane l -> row
// (r/4)*8 + (l/32)*4 + r%4, col l%32.
#include <cstdlib>

#include "enc_gemm.h"

__global__ void __launch_bounds__(256) k_split_f16(const float4 *x, size_t n4, uint2 *hi, uint2 *lo, int *ovf) {
    uint32_t of = 0;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) {
        const float4 v = x[i];
        uint16_t h[4], l[4];
        fw_split2(v.x, h[0], l[0], of);
        fw_split2(v.y, h[1], l[1], of);
        fw_split2(v.z, h[2], l[2], of);
        fw_split2(v.w, h[3], l[3], of);
        hi[i] = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
        lo[i] = make_uint2(l[0] | ((uint32_t)l[1] << 16), l[2] | ((uint32_t)l[3] << 16));
    }
    if (of && ovf) *ovf = 1;
}

// n must be a multiple of 4 (rows of d, d % 128 == 0)
void fw_launch_split_f16(hipStream_t st, const float *x, size_t n, uint16_t *hi, uint16_t *lo, int *ovf) {
    const size_t n4 = n / 4;
    size_t g = (n4 + 255) / 256;
    g = g < 8192 ? g : 8192;
    hipLaunchKernelGGL(k_split_f16, dim3((unsigned)g), dim3(256), 0, st, (const float4 *)x, n4, (uint2 *)hi,
                       (uint2 *)lo, ovf);
}

#define GT_BM 128 // k_gemm_tile's block tile
#define GT_BN 128

// Epilogue for the 4 consecutive rows row0..row0+3 of one column.
template <int EPI>
__device__ __forceinline__ void gemm_store4(const FwGemm &g, int row0, int col, const float (&a)[4]) {
    if (col >= g.N) return;
    if constexpr (EPI == FW_EPI_QKV) {
        // head-major split outputs: Q, K as [B, H, T, 64]; V as [B, H, 64, Tp]
        const int d = g.ldc, which = col / d, cc = col - which * d, h = cc >> 6, dd = cc & 63;
        float bias = g.bias ? g.bias[col] : 0.0f;
        float sw = g.sw[col];
        float v[4];
        uint16_t hi[4], lo[4];
        uint32_t of = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            int row = row0 + e;
            float x = a[e];
            x = row < g.M ? x * g.sx[row] * sw : 0.0f;
            if (g.bias) x = x + bias;
            v[e] = x;
            fw_split2(v[e], hi[e], lo[e], of);
        }
        if (of && g.ovf) *g.ovf = 1;
        if (which < 2) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                int row = row0 + e;
                if (row >= g.M) continue;
                int b = row / g.T, t = row - b * g.T;
                size_t o = (((size_t)b * g.H + h) * g.T + t) * 64 + dd;
                g.o16[2 * which][o] = hi[e];
                g.o16[2 * which + 1][o] = lo[e];
            }
        } else {
            // V^T key positions: bits 2 and 3 of the key index swapped within
            // each 16-key group (the attention kernel reads the 8 keys one MFMA
            // lane needs as one chunk); 4-key runs stay contiguous
            int b = row0 / g.T, t = row0 - b * g.T;
            size_t o = (((size_t)b * g.H + h) * 64 + dd) * g.Tp + fw_vt_pos(t);
            if ((t & 3) == 0 && t + 3 < g.T && row0 + 3 < g.M) {
                uint2 ph = make_uint2(hi[0] | ((uint32_t)hi[1] << 16), hi[2] | ((uint32_t)hi[3] << 16));
                uint2 pl = make_uint2(lo[0] | ((uint32_t)lo[1] << 16), lo[2] | ((uint32_t)lo[3] << 16));
                *(uint2 *)(g.o16[4] + o) = ph;
                *(uint2 *)(g.o16[5] + o) = pl;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    int row = row0 + e;
                    if (row >= g.M) continue;
                    int bb = row / g.T, tt = row - bb * g.T;
                    size_t oo = (((size_t)bb * g.H + h) * 64 + dd) * g.Tp + fw_vt_pos(tt);
                    g.o16[4][oo] = hi[e];
                    g.o16[5][oo] = lo[e];
                }
            }
        }
        return;
    } else {
        float bias = g.bias ? g.bias[col] : 0.0f;
        float sw = EPI != FW_EPI_ACC32 ? g.sw[col] : 1.0f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            int row = row0 + e;
            if (row >= g.M) continue;
            size_t o = (size_t)row * g.ldc + col;
            if constexpr (EPI == FW_EPI_ACC32) {
                ((int *)g.C)[o] = (int)a[e];
                continue;
            } else {
                float v = a[e] * g.sx[row] * sw;
                if (g.bias) v = v + bias;
                if constexpr (EPI == FW_EPI_F32) {
                    g.C[o] = v;
                } else if constexpr (EPI == FW_EPI_RESID) {
                    g.C[o] = g.C[o] + v;
                }
            }
        }
    }
}

// Epilogue of a BM x BN block tile: wave (wm, wn) holds TM x TN 32x32
// accumulator tiles.  `lds` (>= 4 * 32 * 33 floats) is free scratch here.
template <int EPI, int BM, int BN>
__device__ __forceinline__ void gemm_epilogue(const FwGemm &g, v16i (&acc)[BM / 64][BN / 64], unsigned char *lds,
                                              int m0, int n0) {
    constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 32, TN = WN / 32;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    if constexpr (EPI == FW_EPI_QKV) {
        // Heavy epilogues: written once, in a runtime loop over this wave's
        // tiles, reading each tile back from a wave-private LDS slab (a fully
        // unrolled copy of such an epilogue per tile is too large to unroll,
        // which would push the accumulators to scratch memory).
        float *slab = (float *)lds + wave * (32 * 33);
        for (int tile = 0; tile < TM * TN; tile++) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
                    if (i * TN + j == tile)
#pragma unroll
                        for (int r = 0; r < 16; r++)
                            slab[((r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)) * 33 + (lane & 31)] = (float)acc[i][j][r];
            // the slab is private to this wave and a wave's LDS accesses run in
            // order: only the compiler must not reorder across this point
            asm volatile("" ::: "memory");
            const int i = tile / TN, j = tile - i * TN;
            const int col = n0 + wn * WN + j * 32 + (lane & 31);
            for (int q = 0; q < 4; q++) {
                const int rl = q * 8 + (lane >> 5) * 4;
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = slab[(rl + e) * 33 + (lane & 31)];
                gemm_store4<EPI>(g, m0 + wm * WM + i * 32 + rl, col, v);
            }
            asm volatile("" ::: "memory");
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int col = n0 + wn * WN + j * 32 + (lane & 31);
            const int rb = m0 + wm * WM + i * 32 + (lane >> 5) * 4; // + q*8 + e
            if constexpr (EPI == FW_EPI_ACC32) {
                // exact i32 accumulators: store the integers themselves
                if (col < g.N)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int row = rb + (r >> 2) * 8 + (r & 3);
                        if (row < g.M) ((int *)g.C)[(size_t)row * g.ldc + col] = acc[i][j][r];
                    }
            } else {
                // One 32x32 tile at a time: every load it needs (row scales,
                // residual values; rows clamped in bounds) is issued before the
                // first store, so the tile waits on memory once, not per element.
                const int colc = col < g.N ? col : g.N - 1;
                const float bias = g.bias ? g.bias[colc] : 0.0f;
                const float sw = g.sw[colc];
                float sx[16], cv[16];
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    int row = rb + (r >> 2) * 8 + (r & 3);
                    row = row < g.M ? row : g.M - 1;
                    sx[r] = g.sx[row];
                    if constexpr (EPI == FW_EPI_RESID) cv[r] = g.C[(size_t)row * g.ldc + colc];
                }
                if (col < g.N) {
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int row = rb + (r >> 2) * 8 + (r & 3);
                        float v = (float)acc[i][j][r] * sx[r] * sw;
                        if (g.bias) v = v + bias;
                        if (row < g.M) {
                            const size_t o = (size_t)row * g.ldc + col;
                            if constexpr (EPI == FW_EPI_F32) {
                                g.C[o] = v;
                            } else if constexpr (EPI == FW_EPI_RESID) {
                                g.C[o] = cv[r] + v;
                            }
                        }
                    }
                }
            }
        }
}

// ---------------------------------------------------------------------------
// One tile per block, 2x2 waves: operands go global -> LDS directly
// (global_load_lds_dwordx4, no staging registers), NS stages in flight, one
// barrier per stage.  LDS rows are 64 bytes with the 16-byte chunks of row r
// XOR-swizzled by (r ^ r>>2) & 3, so the MFMA fragment reads are free of bank
// conflicts.  Each wave loads ROWS/64 row groups of 16 rows per stage (one
// instruction writes 16 rows x 64 bytes = 1 KB contiguous in LDS).
template <int EPI>
__global__ void __launch_bounds__(256) k_gemm_tile(FwGemm g, int ntm, int ntn) {
    constexpr int BM = GT_BM, BN = GT_BN, NS = 3;
    constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 32, TN = WN / 32;
    constexpr int ROWS = BM + BN;
    constexpr int STAGE = ROWS * 64;
    constexpr int LPW = ROWS / 64; // load instructions per wave per stage
    __shared__ __align__(1024) unsigned char lds[NS * STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;

    const int t = gemm_tile_order(g.map);
    constexpr int GM = 8;
    const int gsize = GM * ntn, grp = t / gsize, first_m = grp * GM;
    const int gm = min(ntm - first_m, GM), rr = t - grp * gsize;
    const int m0 = (first_m + rr % gm) * BM, n0 = (rr / gm) * BN;
    const int nsteps = g.K / 64;

    // per-lane source rows of this wave's row groups (fixed over k)
    const unsigned char *src[LPW];
#pragma unroll
    for (int q = 0; q < LPW; q++) {
        const int lr = (wave * LPW + q) * 16 + (lane >> 2); // LDS row
        const int c = (lane & 3) ^ gsw(lr);                  // global chunk for this LDS slot
        if (lr < BM) {
            int gr = m0 + lr;
            gr = gr < g.M ? gr : g.M - 1; // rows past M: in-bounds reload, never stored
            src[q] = (const unsigned char *)g.A + (size_t)gr * g.lda + c * 16;
        } else {
            int gn = n0 + lr - BM;
            gn = gn < g.N ? gn : g.N - 1;
            src[q] = (const unsigned char *)g.B + (size_t)gn * g.ldb + c * 16;
        }
    }
    auto issue = [&](int s) {
        const int sc = s < nsteps ? s : nsteps - 1; // past the end: harmless reload keeps vmcnt uniform
        unsigned char *dst = lds + (s % NS) * STAGE + wave * LPW * 1024;
#pragma unroll
        for (int q = 0; q < LPW; q++)
            __builtin_amdgcn_global_load_lds((const void *)(src[q] + (size_t)sc * 64),
                                             (void __attribute__((address_space(3))) *)(dst + q * 1024), 16, 0, 0);
    };

    v16i acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0;

    // Fragment ping-pong: the two k-substeps (ks) of a stage use register
    // sets 0 and 1; the next substep's LDS reads are issued before the current
    // substep's MFMAs, so fragment latency hides behind MFMA issue.  The stage
    // barrier sits between the substeps of a stage.
    v4i fa[2][TM], fb[2][TN];
    auto ldfrag = [&](int set, int stage, int ks) {
        const unsigned char *tb = lds + (stage % NS) * STAGE;
        const int c = ks * 2 + (lane >> 5);
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const int lr = wm * WM + i * 32 + (lane & 31);
            fa[set][i] = *(const v4i *)(tb + lr * 64 + ((c ^ gsw(lr)) << 4));
        }
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int lr = BM + wn * WN + j * 32 + (lane & 31);
            fb[set][j] = *(const v4i *)(tb + lr * 64 + ((c ^ gsw(lr)) << 4));
        }
    };
    auto mfmas = [&](int set) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[set][i], fb[set][j], acc[i][j], 0, 0, 0);
    };

#pragma unroll
    for (int p = 0; p < NS - 1; p++) issue(p);
    FW_WAIT_VM(LPW * (NS - 2)); // stage 0 landed
    asm volatile("s_barrier" ::: "memory");
    issue(NS - 1);
    ldfrag(0, 0, 0);
    for (int s = 0; s < nsteps; s++) {
        // set 0 was read a full MFMA block ago: completing it here is free and
        // lets the set-1 reads stay in flight under the set-0 MFMAs
        FW_WAIT_LGKM0();
        ldfrag(1, s, 1);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(0);
        __builtin_amdgcn_sched_barrier(0);
        // stage s+1 visible to every wave; buffer (s % NS) is re-filled by
        // stage s+NS once every wave's reads of it have completed.  Run on the
        // last step too (a dummy stage, fragments never used): a branch here
        // would make the compiler wait on the new reads before the set-1 MFMAs.
        FW_WAIT_VM_LGKM0(LPW * (NS - 2));
        asm volatile("s_barrier" ::: "memory");
        issue(s + NS);
        ldfrag(0, s + 1, 0);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(1);
        __builtin_amdgcn_sched_barrier(0);
    }
    FW_WAIT_VM(0);
    __syncthreads(); // LDS is reused by the heavy epilogues
    gemm_epilogue<EPI, BM, BN>(g, acc, lds, m0, n0);
}

// ---------------------------------------------------------------------------
// Persistent int8 GEMM.  A block (one or two to a CU) walks its share of the tile sequence
// through a single flattened (tile, k-step) pipeline: the operand stages of the
// next tile are already in flight while the current tile's epilogue runs, and
// its stores drain to memory under the next tile's MFMAs (a one-tile-per-block
// launch leaves every CU storing at once and the MFMAs idle meanwhile).
//
// Block = NW = WGM x WGN waves (2 per SIMD); block tile BM x BN, wave tile
// (BM/WGM) x (BN/WGN) of 32x32 i8 MFMA tiles; K advances 64 bytes per stage
// through an NS-stage global -> LDS ring (16-byte chunks XOR-swizzled by
// gsw(row)), one barrier per stage.
//
// vmcnt bookkeeping: stage s+1 is known to have landed once at most
// LPW*(NS-2) of this wave's loads are outstanding, which holds while every
// memory operation issued after stage s+1 is a load (loads return in order).
// Stores may complete out of order with loads, so before a tile's epilogue
// issues stores every outstanding load is waited for (vmcnt 0), and loads
// issued after the stores are the only ones later waits count on.
//
// The per-tile row scales sx, column scales sw and bias are staged into LDS
// with the tile's first stage (SCL 256-byte loads per wave, the same number
// for every wave so the counts above stay uniform), into one of SB = 4 slots by
// the tile's number.  A stage is requested NS - 1 steps ahead and a step's
// requests are not ordered against another wave's epilogue of the step before,
// so tile t + SB may start to load from step (t + 1) n + 1 on at the earliest
// (n steps a tile): (SB - 1) n >= NS.  With two slots that held from K = 64 NS
// on, and a tile of K = 128 took the scales of the tile two further on.
//
// What bounds it: a 256 x 256 stage takes 1,550-1,750 cycles for 1,060 of MFMAs
// (the stage barrier with both waves of a SIMD at it; the fragments, 96 KB a stage
// and CU, would be three quarters of the LDS rate if the MFMAs ran back to back and
// are half of it as it is), a tile's epilogue 15,000-18,000 against 35,000 for its
// 20 stages at K 1280 (conversion of the accumulators, store instructions), the
// clock falls to 1.6-1.9 GHz under it.  With the loads and fragment reads between
// the MFMAs instead of after the barrier (10 windows): a kernel back to back with
// itself q/k/v 146 -> 127 us, attn.out 66 -> 56, fc1 150 -> 146, fc2 165 -> 155; in
// the encoder's trace 144 -> 140, 72 -> 68, 158 -> 157, 178 both.
//
// Tile sequence: XCD x (blocks x, x+8, ...) owns a contiguous range of the
// GM=8-grouped tile order, walked by its blocks in lockstep, so the tiles in
// flight on one XCD share A row panels and B column panels in its L2.  With
// `wrows` > 0 (the QKV epilogue) M tiles never straddle a window of wrows rows:
// each window is tiled on its own, so every tile's rows share one window and
// start at a multiple of BM within it.
#define PI8_MIN_K 128
template <int EPI, int BM, int BN, int WGM, int WGN, int NS>
__global__ void __launch_bounds__(64 * WGM * WGN, 2) k_gemm_pi8(FwGemm g, int ntm, int ntn, int ntw) {
    constexpr int NW = WGM * WGN, WM = BM / WGM, WN = BN / WGN, TM = WM / 32, TN = WN / 32;
    constexpr int STAGE = (BM + BN) * 64, LPW = STAGE / 1024 / NW;
    constexpr int SCL = (BM + 2 * BN + 64 * NW - 1) / (64 * NW); // scale loads per wave per tile
    constexpr int SCLN = SCL * NW * 64;                           // floats per slot
    constexpr int SB = 4;                                         // slots
    static_assert((SB - 1) * (PI8_MIN_K / 64) >= NS, "a slot is free before its next tile's scales arrive");
    constexpr bool QKV = EPI == FW_EPI_QKV;
    // wave-private LDS slab: QKV turns 32 x 32 f32 tiles (rows of 40), the
    // index epilogue sends 32 x WN u16 tiles out as whole rows
    constexpr int SLABB = QKV ? 32 * 40 * 4 : (EPI == FW_EPI_F16IDX ? 32 * WN * 2 : 0); // bytes per wave
    static_assert(STAGE % (1024 * NW) == 0, "stage loads must split evenly over waves");
    __shared__ __align__(1024) unsigned char lds[NS * STAGE + SB * SCLN * 4 + NW * SLABB];
    float *scl = (float *)(lds + NS * STAGE);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int G = gridDim.x, xcd = blockIdx.x & 7, loc = blockIdx.x >> 3, nloc = G >> 3;
    const int ntiles = ntm * ntn;
    const int xs = (int)((long long)ntiles * xcd / 8), xe = (int)((long long)ntiles * (xcd + 1) / 8);
    const int my_n = xe - xs > loc ? (xe - xs - loc + nloc - 1) / nloc : 0;
    const int nsteps = g.K / 64;
    const int total = my_n * nsteps;
    if (total == 0) return;
    uint32_t ovf_any = 0; // an f16-pair value past the f16 range (FW_EPI_QKV)
    // tile ti of this block -> first row, valid rows, first column
    auto coords = [&](int ti, int &m0, int &mrows, int &n0) {
        const int t = xs + loc + ti * nloc;
        constexpr int GM = 8;
        const int gsize = GM * ntn, grp = t / gsize, first_m = grp * GM;
        const int gm = min(ntm - first_m, GM), rr = t - grp * gsize;
        const int mt = first_m + rr % gm;
        n0 = (rr / gm) * BN;
        if (ntw > 0) {
            const int w = mt / ntw, tt = mt - w * ntw;
            m0 = w * g.T + tt * BM;
            mrows = min(BM, g.T - tt * BM);
        } else {
            m0 = mt * BM;
            mrows = min(BM, g.M - m0);
        }
    };
    // issue side: tile and step of the next stage to load; per-lane 32-bit
    // offsets from the tile's operand panels, per-lane scale sources
    int it_tile = 0, it_step = 0;
    const unsigned char *pa, *pb;
    uint32_t off[LPW];
    const float *ssrc[SCL];
    auto set_src = [&](int ti) __attribute__((always_inline)) {
        int m0, mrows, n0;
        coords(ti, m0, mrows, n0);
        pa = (const unsigned char *)g.A + (size_t)m0 * g.lda;
        pb = (const unsigned char *)g.B + (size_t)n0 * g.ldb;
#pragma unroll
        for (int q = 0; q < LPW; q++) {
            const int lr = (wave * LPW + q) * 16 + (lane >> 2);
            const int c = (lane & 3) ^ gsw(lr);
            if (lr < BM) off[q] = (uint32_t)min(lr, mrows - 1) * g.lda + c * 16;
            else off[q] = (uint32_t)min(lr - BM, g.N - 1 - n0) * g.ldb + c * 16;
        }
#pragma unroll
        for (int q = 0; q < SCL; q++) {
            const int e = (q * NW + wave) * 64 + lane;
            if (e < BM) ssrc[q] = g.sx + m0 + min(e, mrows - 1);
            else if (e < BM + BN) ssrc[q] = g.sw + min(n0 + e - BM, g.N - 1);
            else ssrc[q] = (g.bias ? g.bias : g.sw) + min(n0 + max(e - BM - BN, 0), g.N - 1);
        }
    };
    set_src(0);
    // load q of stage gs
    auto issue = [&](int gs, int q) __attribute__((always_inline)) {
        unsigned char *dst = lds + (gs % NS) * STAGE + (wave * LPW + q) * 1024;
        const int sc = it_tile < my_n ? it_step : nsteps - 1; // past the last tile: in-bounds reload
        // (a mask, not a choice between the captured pointers, which would keep them in memory)
        const unsigned long long a = (unsigned long long)pa, b = (unsigned long long)pb;
        const unsigned long long base = a + (((wave * LPW + q) * 16 < BM ? 0ull : ~0ull) & (b - a)) + (size_t)sc * 64;
        __builtin_amdgcn_global_load_lds((const void *)((const char *)base + off[q]),
                                         (void __attribute__((address_space(3))) *)dst, 16, 0, 0);
    };
    // after a stage's last load: the scales of a new tile, the next stage
    auto advance = [&]() __attribute__((always_inline)) {
        if (it_step == 0) {
            float *sd = scl + (it_tile % SB) * SCLN + wave * 64;
#pragma unroll
            for (int e = 0; e < SCL; e++)
                __builtin_amdgcn_global_load_lds((const void *)ssrc[e],
                                                 (void __attribute__((address_space(3))) *)(sd + e * NW * 64), 4,
                                                 0, 0);
        }
        if (++it_step == nsteps) {
            if (it_tile < my_n) {
                it_step = 0;
                if (++it_tile < my_n) set_src(it_tile);
            } else {
                it_step = nsteps - 1;
            }
        }
    };

    v16i acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0;
    // fragment x (A tiles, then B tiles) of substep ks of a stage
    constexpr int NF = TM + TN, NM = TM * TN, LH = LPW / 2;
    v4i fr[2][NF];
    auto ldfrag = [&](int set, int stage, int ks, int x) __attribute__((always_inline)) {
        const unsigned char *tb = lds + (stage % NS) * STAGE;
        const int c = ks * 2 + (lane >> 5);
        const int lr = (x < TM ? wm * WM + x * 32 : BM + wn * WN + (x - TM) * 32) + (lane & 31);
        fr[set][x] = *(const v4i *)(tb + lr * 64 + ((c ^ gsw(lr)) << 4));
    };
    // Half a stage: the MFMAs of one substep with the next substep's fragment
    // reads and loads [q0, q1) of a later stage between them (requested all at
    // once after the barrier they hold the wave's MFMAs up).
    auto half = [&](int set, int rstage, int rks, int lstage, int q0, int q1, bool on) __attribute__((always_inline)) {
        int rd = 0, ld = q0;
#pragma unroll
        for (int m = 0; m < NM; m++) {
            const int i = m / TN, j = m % TN;
            acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fr[set][i], fr[set][TM + j], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < NF; u++)
                if (rd < NF && (m + 1) * NF * 4 >= (rd + 1) * NM * 3) ldfrag(set ^ 1, rstage, rks, rd++);
            if (ld < q1 && (m + 1) * (q1 - q0) * 2 >= (ld - q0 + 1) * NM) {
                if (on) issue(lstage, ld);
                ld++;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int u = 0; u < LPW; u++)
            if (ld < q1) {
                if (on) issue(lstage, ld);
                ld++;
            }
    };

#pragma unroll 1
    for (int p = 0; p < NS - 1; p++) {
#pragma unroll
        for (int q = 0; q < LPW; q++) issue(p, q);
        advance();
    }
    FW_WAIT_VM(0);
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int q = 0; q < LH; q++) issue(NS - 1, q);
#pragma unroll
    for (int x = 0; x < NF; x++) ldfrag(0, 0, 0, x);
    const bool has_bias = g.bias != nullptr;
    int tile = 0, s = 0;
    for (int gs = 0; gs < total; gs++) {
        FW_WAIT_LGKM0(); // set 0, read during the last MFMAs
        half(0, gs, 1, gs + NS - 1, LH, LPW, true);
        advance();
        // stage gs+1 visible to every wave.  At a tile's first step it landed
        // before the last epilogue's stores (or in the prologue), which are
        // left to drain.
        if (s == 0) FW_WAIT_LGKM0();
        else FW_WAIT_VM_LGKM0(LPW * (NS - 2));
        asm volatile("s_barrier" ::: "memory");
        const bool last = s == nsteps - 1;
        half(1, gs + 1, 0, gs + NS, 0, LH, !last); // (a tile's last step loads after its stores)
        if (!last) {
            s++;
            continue;
        }
        // ---- epilogue of this block's tile `tile` ----
        FW_WAIT_VM(0);
        int m0, mrows, n0;
        coords(tile, m0, mrows, n0);
        // lane-derived offsets recomputed here from an opaque copy of the lane
        // id, so per-element addresses are not hoisted out of the tile loop
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const float *ssx = scl + (tile % SB) * SCLN, *ssw = ssx + BM, *sbi = ssw + BN;
        // A 32 x WN u16 tile (accumulator layout: element r of lane l is row
        // (r/4)*8 + (l/32)*4 + r%4, column j*32 + l%32), put into this wave's
        // slab one 32-column tile j at a time, then flushed to rows dst + row*ld,
        // row < vrows, as 16-byte runs of whole rows (WN/8 lanes per row).  The
        // slab is private to the wave and a wave's LDS accesses run in order:
        // only the compiler must not reorder them.
        uint16_t *const sl = (uint16_t *)(lds + NS * STAGE + SB * SCLN * 4 + wave * SLABB);
        auto slab_put = [&](int j, const uint16_t (&u)[16]) {
            asm volatile("" ::: "memory");
#pragma unroll
            for (int r = 0; r < 16; r++) sl[((r >> 2) * 8 + (ln >> 5) * 4 + (r & 3)) * WN + j * 32 + (ln & 31)] = u[r];
            asm volatile("" ::: "memory");
        };
        auto slab_flush = [&](uint16_t *dst, size_t ld, int vrows) {
            constexpr int LPR = WN / 8, RPI = 64 / LPR;
            asm volatile("" ::: "memory");
#pragma unroll
            for (int q = 0; q < 32 / RPI; q++) {
                const int row = q * RPI + ln / LPR, ch = ln % LPR;
                const uint4 w = *(const uint4 *)(sl + row * WN + ch * 8);
                if (row < vrows) *(uint4 *)(dst + row * ld + ch * 8) = w;
            }
            asm volatile("" ::: "memory");
        };
        // The residual rows (two 128-byte rows per store) are written
        // non-temporally: they are not read again by this kernel and would only
        // evict operand panels from L2.  F32 rows (the exact mode's q/k/v and fc1) are
        // left in the caches: its attention reads q, k and v many times, one window's
        // scores 226 -> 179 us and values 408 -> 378.  The QKV epilogue's 16-byte runs stay
        // cached so L2 can merge them into lines (non-temporal partial lines
        // measured 1.6x slower).
        if constexpr (EPI == FW_EPI_RESID) {
            static_assert(TM * TN <= 4, "residual values of the wave tile are held in registers");
            // residual values of every element first: one wait, then the stores
            float cv[TM][TN][16];
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int col = min(n0 + wn * WN + j * 32 + (ln & 31), g.N - 1);
                    const int rl = wm * WM + i * 32 + (ln >> 5) * 4;
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int row = m0 + min(rl + (r >> 2) * 8 + (r & 3), mrows - 1);
                        cv[i][j][r] = g.C[(size_t)row * g.ldc + col];
                    }
                }
            FW_WAIT_VM(0);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int cl = wn * WN + j * 32 + (ln & 31), col = n0 + cl;
                    const int rl = wm * WM + i * 32 + (ln >> 5) * 4;
                    const float s2 = ssw[cl], bb = sbi[cl];
                    v4f sr[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) sr[q] = *(const v4f *)(ssx + rl + q * 8);
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int rw = rl + (r >> 2) * 8 + (r & 3);
                        float v = (float)acc[i][j][r] * sr[r >> 2][r & 3] * s2;
                        if (has_bias) v = v + bb;
                        if (rw < mrows && col < g.N) __builtin_nontemporal_store(cv[i][j][r] + v, g.C + (size_t)(m0 + rw) * g.ldc + col);
                    }
                }
        } else if constexpr (EPI == FW_EPI_F16IDX) {
            const bool wide = n0 + BN <= g.N;
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const int r0 = wm * WM + i * 32, vrows = mrows - r0;
                uint16_t u[TN][16];
                bool sent = false;
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int cl = wn * WN + j * 32 + (ln & 31);
                    const int rl = r0 + (ln >> 5) * 4;
                    const float s2 = ssw[cl], bb = sbi[cl];
                    v4f sr[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) sr[q] = *(const v4f *)(ssx + rl + q * 8);
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        float v = (float)acc[i][j][r] * sr[r >> 2][r & 3] * s2;
                        if (has_bias) v = v + bb;
                        const bool in = fabsf(v) < FW_GIDX_LIM;
                        u[j][r] = in ? fw_f2h(v) : (uint16_t)FW_GIDX_SENT;
                        sent |= !in;
                        acc[i][j][r] = __float_as_int(v); // kept for the rare side stores
                    }
                }
                if (__builtin_amdgcn_ballot_w64(sent)) {
                    // values beyond the table's range: exact f32 into the side array
#pragma unroll
                    for (int j = 0; j < TN; j++)
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            const int rw = r0 + (r >> 2) * 8 + (ln >> 5) * 4 + (r & 3);
                            const int col = n0 + wn * WN + j * 32 + (ln & 31);
                            if (u[j][r] == (uint16_t)FW_GIDX_SENT && rw < mrows && col < g.N)
                                g.C[(size_t)(m0 + rw) * g.ldc + col] = __int_as_float(acc[i][j][r]);
                        }
                }
                if (vrows <= 0) continue;
                if (wide) {
#pragma unroll
                    for (int j = 0; j < TN; j++) slab_put(j, u[j]);
                    slab_flush(g.o16[0] + (size_t)(m0 + r0) * g.ldc + n0 + wn * WN, g.ldc, vrows);
                } else {
#pragma unroll
                    for (int j = 0; j < TN; j++)
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            const int rw = (r >> 2) * 8 + (ln >> 5) * 4 + (r & 3);
                            const int col = n0 + wn * WN + j * 32 + (ln & 31);
                            if (rw < vrows && col < g.N) g.o16[0][(size_t)(m0 + r0 + rw) * g.ldc + col] = u[j][r];
                        }
                }
            }
        } else if constexpr (EPI == FW_EPI_F32 || EPI == FW_EPI_ACC32) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int cl = wn * WN + j * 32 + (ln & 31), col = n0 + cl;
                    const int rl = wm * WM + i * 32 + (ln >> 5) * 4;
                    const float s2 = ssw[cl], bb = sbi[cl];
                    v4f sr[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) sr[q] = *(const v4f *)(ssx + rl + q * 8);
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int rw = rl + (r >> 2) * 8 + (r & 3);
                        if (rw < mrows && col < g.N) {
                            const size_t o = (size_t)(m0 + rw) * g.ldc + col;
                            if constexpr (EPI == FW_EPI_ACC32) {
                                ((int *)g.C)[o] = acc[i][j][r];
                            } else {
                                float v = (float)acc[i][j][r] * sr[r >> 2][r & 3] * s2;
                                if (has_bias) v = v + bb;
                                g.C[o] = v;
                            }
                        }
                    }
                }
        } else if constexpr (QKV) {
            float *slab = (float *)(lds + NS * STAGE + SB * SCLN * 4 + wave * SLABB);
            const int wnd = m0 / g.T, tb0 = m0 - wnd * g.T;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int c0 = n0 + wn * WN + j * 32; // 32 columns of one head
                    const int cl = c0 - n0 + (ln & 31), col = n0 + cl;
                    const int rl = wm * WM + i * 32 + (ln >> 5) * 4;
                    const float s2 = ssw[cl], bb = sbi[cl];
                    v4f sr[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) sr[q] = *(const v4f *)(ssx + rl + q * 8);
                    float v[16];
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        v[r] = (float)acc[i][j][r] * sr[r >> 2][r & 3] * s2;
                        if (has_bias) v[r] = v[r] + bb;
                    }
                    if (c0 >= g.N) continue;
                    const int t0 = tb0 + wm * WM + i * 32; // window position of the tile's first row
                    const int vrows = mrows - (wm * WM + i * 32);
                    if (vrows <= 0) continue;
                    int lt = ln; // opaque per tile: addresses are not hoisted over the tiles
                    asm volatile("" : "+v"(lt));
                    qkv_store32(g, slab, v, lt, c0, wnd, t0, vrows, ovf_any);
                }
        }
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] = 0;
#pragma unroll
        for (int q = 0; q < LH; q++) issue(gs + NS, q);
        tile++;
        s = 0;
    }
    FW_WAIT_VM(0);
    if constexpr (EPI == FW_EPI_QKV)
        if (ovf_any && g.ovf) *g.ovf = 1;
}

// ---------------------------------------------------------------------------
template <int EPI>
static void launch_tile(hipStream_t st, const FwGemm &g) {
    const int ntm = (g.M + GT_BM - 1) / GT_BM, ntn = (g.N + GT_BN - 1) / GT_BN;
    hipLaunchKernelGGL(k_gemm_tile<EPI>, dim3(ntm * ntn), dim3(256), 0, st, g, ntm, ntn);
}

// Persistent int8 launch.  256x256 tiles (8 waves of 128x64) or 256x128 (8 of
// 64x64), one block per CU, or 128x128 (4 of 64x64), two; the residual epilogue,
// whose wave tile must fit its residual values in registers, takes the latter
// two.  The grid is a multiple of 8 so block b runs on XCD b % 8.
//
// The choice is the fewest rounds of the CUs, weighted by a round's time
// relative to 256x256 (measured, K 1280, 10 windows: 27 us, 15 for 256x128, 16
// for two 128x128 a CU, less where one a CU suffices: one and two windows' fc2
// 47 -> 39 us).  Used at every width: with it, and the attention and stem that
// came beside it, whole int8 encoder calls of widths 384-1,280 over 1-16 windows of
// 50-1,500 rows ran 1.10-1.37x faster than with the tile by the output's width
// alone, none slower.
template <int EPI, int BM, int BN, int WGM, int WGN, int NS>
static void launch_pi8(hipStream_t st, const FwGemm &g, int ncu, int per_cu) {
    int ntw = 0, ntm;
    if (EPI == FW_EPI_QKV) {
        ntw = (g.T + BM - 1) / BM;
        ntm = (g.M / g.T) * ntw;
    } else {
        ntm = (g.M + BM - 1) / BM;
    }
    const int ntn = (g.N + BN - 1) / BN;
    const int grid = ncu >= 8 ? ncu / 8 * 8 : 8;
    hipLaunchKernelGGL((k_gemm_pi8<EPI, BM, BN, WGM, WGN, NS>), dim3(grid * per_cu), dim3(64 * WGM * WGN), 0, st, g,
                       ntm, ntn, ntw);
}

template <int EPI>
static void launch_pi8_tiles(hipStream_t st, const FwGemm &g, int ncu) {
    auto blocks = [&](int bm, int bn) {
        const long long tm = EPI == FW_EPI_QKV ? (long long)(g.M / g.T) * ((g.T + bm - 1) / bm) : (g.M + bm - 1) / bm;
        return tm * ((g.N + bn - 1) / bn);
    };
    const long long n2 = blocks(128, 128), left = n2 % (2 * ncu);
    const double c0 = (double)((blocks(256, 256) + ncu - 1) / ncu);
    const double c1 = (double)((blocks(256, 128) + ncu - 1) / ncu) * 0.56;
    const double c2 = (double)(n2 / (2 * ncu)) * 0.6 + (left == 0 ? 0.0 : left <= ncu ? 0.42 : 0.6);
    if constexpr (EPI != FW_EPI_RESID)
        if (c0 <= c1 && c0 <= c2) {
            launch_pi8<EPI, 256, 256, 2, 4, 3>(st, g, ncu, 1);
            return;
        }
    if (c1 <= c2) launch_pi8<EPI, 256, 128, 4, 2, 3>(st, g, ncu, 1);
    else launch_pi8<EPI, 128, 128, 2, 2, EPI == FW_EPI_QKV || EPI == FW_EPI_F16IDX ? 3 : 4>(st, g, ncu, 2);
}

bool fw_launch_gemm(hipStream_t st, int kind, const FwGemm &g0) {
    static int map = -1;
    if (map < 0) {
        const char *e = getenv("FWHIP_GEMM_MAP");
        map = e ? atoi(e) : 1;
    }
    FwGemm g = g0;
    g.map = map;
    static int ncu = 0;
    if (!ncu) {
        int dev = 0;
        (void)hipGetDevice(&dev);
        (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
        if (ncu <= 0) ncu = 256;
    }
    static int pi8 = -1;
    if (pi8 < 0) {
        const char *e = getenv("FWHIP_GEMM_I8P");
        pi8 = e ? atoi(e) : 1;
    }
    if (kind == FW_KIND_F16S) return fw_launch_gemm_f16(st, g0, ncu);
    if (g.K % 64) return false;
    if (pi8 && g.K >= PI8_MIN_K &&
        (g.epi != FW_EPI_QKV || (g.T > 0 && g.M % g.T == 0))) {
        switch (g.epi) {
        case FW_EPI_F32: launch_pi8_tiles<FW_EPI_F32>(st, g, ncu); return true;
        case FW_EPI_RESID: launch_pi8_tiles<FW_EPI_RESID>(st, g, ncu); return true;
        case FW_EPI_QKV: launch_pi8_tiles<FW_EPI_QKV>(st, g, ncu); return true;
        case FW_EPI_ACC32: launch_pi8_tiles<FW_EPI_ACC32>(st, g, ncu); return true;
        case FW_EPI_F16IDX: launch_pi8_tiles<FW_EPI_F16IDX>(st, g, ncu); return true;
        default: break;
        }
    }
    switch (g.epi) {
    case FW_EPI_F32: launch_tile<FW_EPI_F32>(st, g); return true;
    case FW_EPI_RESID: launch_tile<FW_EPI_RESID>(st, g); return true;
    case FW_EPI_QKV: launch_tile<FW_EPI_QKV>(st, g); return true;
    case FW_EPI_ACC32: launch_tile<FW_EPI_ACC32>(st, g); return true;
    default: return false;
    }
}
