// enc_gemm_f16.hip — the f16-pair GEMMs on MFMA (gfx950): the conv stem, every
// linear of the f32 plan and the decoder's cross K/V.
//
// C[M,N] = A[M,K] x B[N,K]^T with f32 activations A carried as an f16 pair
// (hi, lo = f16(a - hi)) against f16 weights B (exact: the reference
// dequantizes f16 weights to f32): two v_mfma_f32_32x32x16_f16 per product,
// per-product error <= 2^-22 |a| + 2^-25, f32 accumulation.
//
// What bounds it: operand requests past LDS and, after those, the matrix
// units' power.  A GELU output is an f16 table value, so its lo half is zero
// except where |v| >= 10: the consumer (fc2, conv2) runs over the hi plane and
// then over those K blocks of the lo plane that the producer flagged (FL).  With
// none flagged the bits are those of hi and lo products in turn (a lo product of
// zero adds nothing); with some, all hi products come before the lo ones, the
// same products in another order.  Each run of flagged blocks fills and drains the
// ring anew.  f32 encoder of two layers with values >= 10 in chosen 64-column
// blocks of fc1 (hi and lo always, 128 x 128 tiles: 4,130 us for 8 windows, 830 for
// one): none 2,586 / 595 us, every 16th block 2,636 / 632, every fourth 2,761 / 702,
// every second 2,928 / 792, all 2,946 / 727; one conv1 value >= 10, which turns the
// lo plane on for conv2 as a whole, 2,663 / 642.
//
// Block tile BM x BN, NW waves of 64 x WN as 32x32 MFMA tiles.  K advances 64
// bytes (32 halves) per stage through a ring of global -> LDS stages (16-byte
// chunks XOR-swizzled by gsw(row)), one barrier per stage; the two 16-deep
// substeps' fragments ping-pong in registers.  A 256 x 256 tile asks for 48 KB
// per stage against 96 KB for the same area in 128 x 128 tiles, whose requests
// (64 bytes each) kept the L2 two thirds busy.  A stage of 256 x 256 takes 2,400
// cycles for 2,060 of MFMAs, at the 1.43 GHz the clock falls to under them (1.05
// PFLOP/s).  Measured on MI355X, 12,000 rows (8 windows of large-v3-turbo), with
// 128 x 128 tiles, the GELU table in global memory and both products always, and
// now: q/k/v 349 -> 246 us, attn.out 110 -> 89, fc1 509 -> 328, fc2 399 -> 178,
// conv1 132 -> 83, conv2 343 -> 131 (and its im2col pass is gone), cross K/V 898
// -> 594.
//
// GELU epilogues read the table from LDS (128 KB, over the drained ring): 64
// lanes asking for 64 lines in L1 cost about as long as the products.
//
// MFMA operand layouts (gfx950): A lane l -> row l%32, k block (l/32)*16
// bytes; B lane l -> col l%32, same k block; accumulator r of lane l -> row
// (r/4)*8 + (l/32)*4 + r%4, col l%32.
#include "enc_gemm.h"

#define GF_LOB 128 // lo flags of one 64-row block: one byte per 64 columns, up to 8192

template <int EPI, bool FL, int BM, int BN, int WGM, int WGN>
struct GemmF16 {
    static constexpr int NW = WGM * WGN, WM = BM / WGM, WN = BN / WGN, TM = WM / 32, TN = WN / 32;
    static constexpr bool GELU = EPI == FW_EPI_GELU_SPLIT || EPI == FW_EPI_CONV2;
    static constexpr bool SLAB = EPI == FW_EPI_QKV || EPI == FW_EPI_XKV;
    // planes of A that go through the ring together, its stages
    static constexpr int NA = FL ? 1 : 2, NS = FL ? 4 : 3;
    static constexpr int STAGE = (NA * BM + BN) * 64;
    static constexpr int mx(int a, int b) { return a > b ? a : b; }
    static constexpr int LDS = mx(NS * STAGE, mx(GELU ? 131072 : 0, SLAB ? NW * 5120 : 0));
    static_assert(WM == 64, "lo flags are per 64-row wave tile");
};

template <int EPI, bool FL, int BM, int BN, int WGM, int WGN>
__global__ void __launch_bounds__(64 * WGM * WGN, 2) k_gemm_f16(FwGemm g, int ntm, int ntn, int ntw) {
    typedef GemmF16<EPI, FL, BM, BN, WGM, WGN> C;
    constexpr int NW = C::NW, WM = C::WM, WN = C::WN, TM = C::TM, TN = C::TN;
    __shared__ __align__(1024) unsigned char lds[C::LDS];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WGN, wn = wave % WGN;

    // XCD-contiguous, M-grouped tile order
    const int t = gemm_tile_order(g.map);
    constexpr int GM = 8;
    const int gsize = GM * ntn, grp = t / gsize, first_m = grp * GM;
    const int gm = min(ntm - first_m, GM), rr = t - grp * gsize;
    const int mt = first_m + rr % gm, n0 = (rr / gm) * BN;
    int m0, mrows;
    if (ntw > 0) { // M tiles of their own in every window of g.T rows
        const int w = mt / ntw, tt = mt - w * ntw;
        m0 = w * g.T + tt * BM;
        mrows = min(BM, g.T - tt * BM);
    } else {
        m0 = mt * BM;
        mrows = min(BM, g.M - m0);
    }
    const int nsteps = g.K / 32;
    // row of A that GEMM row r reads (apad extra rows after every window)
    auto arow = [&](int r) __attribute__((always_inline)) { return r + (g.apad ? r / g.T * g.apad : 0); };
    const int ar0 = arow(m0);
    const char *const pA = (const char *)g.A + (size_t)ar0 * g.lda * 2, *const pB = (const char *)g.B + (size_t)n0 * g.ldb * 2;
    const char *const pL = (const char *)g.A2 + (size_t)ar0 * g.lda * 2;

    // (selects between captured variables are written as masks: as a choice of
    // addresses they would keep the variables in memory)
    auto sel = [](bool c) { return c ? ~0ull : 0ull; };
    auto pick2 = [&](unsigned long long a, unsigned long long b, int s) { return (a & sel(s < 128)) | (b & sel(s >= 128)); };
    // FL: which 64-deep K blocks have lo halves, per 64-row block of the tile
    // (bit kb of lom[b]), or for all of A one answer
    unsigned long long lom[BM / 64][2], any[2] = {0, 0};
    if constexpr (FL) {
#pragma unroll
        for (int b = 0; b < BM / 64; b++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (g.lo_in) {
                    const int rb = min((m0 >> 6) + b, (g.M - 1) >> 6);
                    lom[b][h] = __builtin_amdgcn_ballot_w64(g.lo_in[(size_t)rb * GF_LOB + h * 64 + lane] != 0);
                } else {
                    lom[b][h] = sel(*g.lo_any != 0);
                }
                any[h] |= lom[b][h];
            }
    }
    auto has_lo = [&](int s) { return (pick2(any[0], any[1], s) >> ((s >> 1) & 63)) & 1; }; // stage s (64 bytes of K)

    v16f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    // Stages [s0, s1): fill the ring, run, drain.  FL: of the hi plane, or (lo)
    // of the lo plane.
    constexpr int NA = C::NA, NS = C::NS, STAGE = C::STAGE, LPW = STAGE / 1024 / NW;
    static_assert(STAGE % (1024 * NW) == 0, "stage loads must split evenly over waves");
    auto segment = [&](int s0, int s1, bool lo) __attribute__((always_inline)) {
        // per-lane offsets of this wave's row groups (16 rows a load), from a
        // base that is the same for the whole wave
        uint32_t off[LPW];
        unsigned long long base[LPW], lm[LPW][2]; // lm: the K blocks a row group is read in
#pragma unroll
        for (int q = 0; q < LPW; q++) {
            const int lr = (wave * LPW + q) * 16 + (lane >> 2), c = (lane & 3) ^ gsw(lr);
            if (lr < NA * BM) {
                // rows past the tile's last: in-bounds reload, never stored
                off[q] = (uint32_t)(arow(m0 + min(lr % BM, mrows - 1)) - ar0) * g.lda * 2 + c * 16;
            } else {
                off[q] = (uint32_t)(min(n0 + lr - NA * BM, g.N - 1) - n0) * g.ldb * 2 + c * 16;
            }
            const int rg = (wave * LPW + q) * 16;
            const unsigned long long a = (unsigned long long)pA, l = (unsigned long long)pL, b = (unsigned long long)pB;
            base[q] = a + (sel((rg >= BM || (FL && lo)) && rg < NA * BM) & (l - a)) + (sel(rg >= NA * BM) & (b - a));
            if (FL)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    lm[q][h] = sel(!lo || rg >= BM);
#pragma unroll
                    for (int k = 0; k < BM / 64; k++) lm[q][h] |= lom[k][h] & sel(rg >> 6 == k);
                }
        }
        // load q of stage s
        auto issue = [&](int s, int q) __attribute__((always_inline)) {
            const int sc = s < s1 ? s : s1 - 1; // past the end: harmless reload keeps vmcnt uniform
            unsigned char *dst = lds + ((s - s0) % NS) * STAGE + (wave * LPW + q) * 1024;
            unsigned long long bs = base[q] + (unsigned long long)sc * 64;
            uint32_t o = off[q];
            if (FL) {
                // a block without lo halves was never written: zeros instead
                const bool on = (pick2(lm[q][0], lm[q][1], sc) >> ((sc >> 1) & 63)) & 1;
                bs = (bs & sel(on)) | ((unsigned long long)g.zero & sel(!on));
                o = on ? o : 0;
            }
            __builtin_amdgcn_global_load_lds((const void *)((const char *)bs + o),
                                             (void __attribute__((address_space(3))) *)dst, 16, 0, 0);
        };
        // fragment x (A planes and tiles, then B tiles) of substep ks of a stage
        constexpr int NF = NA * TM + TN, NM = NA * TM * TN, LH = LPW / 2;
        v4i fr[2][NF];
        auto ldfrag = [&](int set, int stage, int ks, int x) __attribute__((always_inline)) {
            const unsigned char *tb = lds + ((stage - s0) % NS) * STAGE;
            const int c = ks * 2 + (lane >> 5);
            const int lr = (x < NA * TM ? (x / TM) * BM + wm * WM + (x % TM) * 32 : NA * BM + wn * WN + (x - NA * TM) * 32) +
                           (lane & 31);
            fr[set][x] = *(const v4i *)(tb + lr * 64 + ((c ^ gsw(lr)) << 4));
        };
        // Half a stage: the MFMAs of one substep with the next substep's fragment
        // reads and loads [q0, q1) of a later stage between them, so that
        // neither queue holds a wave's MFMAs up (requested all at once after the
        // barrier they cost 700-900 cycles a stage).  Every accumulator takes hi
        // then lo; the other tiles lie in between.
        auto half = [&](int set, int rstage, int rks, int lstage, int q0, int q1) __attribute__((always_inline)) {
            int rd = 0, ld = q0;
#pragma unroll
            for (int m = 0; m < NM; m++) {
                const int a = m / (TM * TN), i = m / TN % TM, j = m % TN;
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, fr[set][a * TM + i]),
                                                                   __builtin_bit_cast(v8h, fr[set][NA * TM + j]),
                                                                   acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (ld < q1 && (m + 1) * (q1 - q0) >= (ld - q0 + 1) * (NM / 2)) issue(lstage, ld++);
                if (rd < NF && (m + 1) * NF >= (rd + 1) * (NM * 3 / 4)) ldfrag(set ^ 1, rstage, rks, rd++);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (; rd < NF; rd++) ldfrag(set ^ 1, rstage, rks, rd);
        };
#pragma unroll
        for (int p = 0; p < NS - 1; p++)
#pragma unroll
            for (int q = 0; q < LPW; q++) issue(s0 + p, q);
        FW_WAIT_VM(LPW * (NS - 2)); // stage s0 landed
        asm volatile("s_barrier" ::: "memory");
#pragma unroll
        for (int q = 0; q < LH; q++) issue(s0 + NS - 1, q);
#pragma unroll
        for (int x = 0; x < NF; x++) ldfrag(0, s0, 0, x);
        for (int s = s0; s < s1; s++) {
            FW_WAIT_LGKM0(); // set 0, read during the last MFMAs
            half(0, s, 1, s + NS - 1, LH, LPW);
            // stage s+1 visible to every wave; the buffer of stage s is re-filled
            // by stage s+NS once every wave's reads of it have completed (run on
            // the last stage too: dummy loads, fragments never used)
            FW_WAIT_VM_LGKM0(LPW * (NS - 2));
            asm volatile("s_barrier" ::: "memory");
            half(1, s + 1, 0, s + NS, 0, LH);
        }
        FW_WAIT_VM_LGKM0(0);
        __syncthreads(); // the ring is free (next segment, epilogue)
    };
    if constexpr (FL) {
        int s = 0, e = nsteps;
        for (bool lo = false;; lo = true) {
            segment(s, e, lo);
            s = lo ? e : 0;
            if ((any[0] | any[1]) == 0) break;
            while (s < nsteps && !has_lo(s)) s++;
            if (s >= nsteps) break;
            e = s + 1;
            while (e < nsteps && has_lo(e)) e++;
        }
    } else {
        segment(0, nsteps, false);
    }

    // ---- epilogue ----
    if constexpr (C::GELU) {
        const char *tab = (const char *)fw_gelu_tab16(g.gelu_tab);
#pragma unroll
        for (int q = 0; q < 128 / NW; q++)
            __builtin_amdgcn_global_load_lds((const void *)(tab + (size_t)(wave * (128 / NW) + q) * 1024 + lane * 16),
                                             (void __attribute__((address_space(3))) *)(lds + (wave * (128 / NW) + q) * 1024),
                                             16, 0, 0);
    }
    const int col0 = n0 + wn * WN, rw0 = wm * WM; // the wave tile's first column and its first row in the block
    auto rowl = [&](int i, int r) { return rw0 + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3); };
    float bias[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) bias[j] = g.bias ? g.bias[min(col0 + j * 32 + (lane & 31), g.N - 1)] : 0.0f;
    if constexpr (EPI == FW_EPI_RESID) {
        // the residual values of the next 32x32 tile are requested before a tile's stores
        float cv[2][16];
        auto fetch = [&](int x) {
            const int col = min(col0 + (x % TN) * 32 + (lane & 31), g.N - 1);
#pragma unroll
            for (int r = 0; r < 16; r++)
                cv[x & 1][r] = g.C[(size_t)(m0 + min(rowl(x / TN, r), mrows - 1)) * g.ldc + col];
        };
        fetch(0);
#pragma unroll
        for (int x = 0; x < TM * TN; x++) {
            const int i = x / TN, j = x % TN, col = col0 + j * 32 + (lane & 31);
            if (x + 1 < TM * TN) fetch(x + 1);
#pragma unroll
            for (int r = 0; r < 16; r++) {
                float v = acc[i][j][r];
                if (g.bias) v = v + bias[j];
                v = cv[x & 1][r] + v;
                if (rowl(i, r) < mrows && col < g.N) g.C[(size_t)(m0 + rowl(i, r)) * g.ldc + col] = v;
            }
        }
    } else if constexpr (EPI == FW_EPI_QKV || EPI == FW_EPI_XKV) {
        float *slab = (float *)(lds + wave * 5120);
        const int wnd = m0 / g.T, tb0 = m0 - wnd * g.T;
        uint32_t of = 0;
#pragma unroll
        for (int i = 0; i < TM; i++) {
            // XKV: window and position of this lane's K row (lane / 2) and of the first
            // row of its V^T runs
            int kw = 0, kt = 0, vw[4], vt[4];
            if constexpr (EPI == FW_EPI_XKV) {
                const int rb = m0 + rw0 + i * 32;
                kw = (rb + (lane >> 1)) / g.T;
                kt = rb + (lane >> 1) - kw * g.T;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int row = rb + q * 8 + (lane >> 5) * 4;
                    vw[q] = row / g.T;
                    vt[q] = row - vw[q] * g.T;
                }
            }
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int c0 = col0 + j * 32, t0 = tb0 + rw0 + i * 32, vrows = mrows - (rw0 + i * 32);
                if (c0 >= g.N || vrows <= 0) continue;
                int ln = lane; // opaque: addresses are not hoisted over the tiles
                asm volatile("" : "+v"(ln));
                float v[16];
                if constexpr (EPI == FW_EPI_QKV) {
#pragma unroll
                    for (int r = 0; r < 16; r++) v[r] = g.bias ? acc[i][j][r] + bias[j] : acc[i][j][r];
                    qkv_store32(g, slab, v, ln, c0, wnd, t0, vrows, of);
                } else {
                    // column c0 + c = (l * 2 + kv) * d + h * 64 + dd: the 32 columns share l, kv and h
                    const int d = g.ldc, l = c0 / (2 * d), rc = c0 - l * 2 * d, kv = rc >= d ? 1 : 0, cc = rc - kv * d;
                    const int h = cc >> 6, dd0 = cc & 63;
                    auto lh = [&](int w) { return ((size_t)w * g.L + l) * g.H + h; };
                    if (kv == 0) {
                        // K [T, 64] rows through the slab: 16 dims (32 bytes) per lane
                        asm volatile("" ::: "memory");
#pragma unroll
                        for (int r = 0; r < 16; r++)
                            slab[((r >> 2) * 8 + (ln >> 5) * 4 + (r & 3)) * 40 + (ln & 31)] = acc[i][j][r] * g.scale;
                        asm volatile("" ::: "memory");
                        const int row = ln >> 1, half = ln & 1;
                        v4f w4[4];
#pragma unroll
                        for (int q = 0; q < 4; q++) w4[q] = *(const v4f *)(slab + row * 40 + half * 16 + q * 4);
                        asm volatile("" ::: "memory");
                        if (row < vrows) {
                            uint32_t p[8];
#pragma unroll
                            for (int q = 0; q < 8; q++)
                                p[q] = fw_f2h(w4[q >> 1][(q & 1) * 2]) | ((uint32_t)fw_f2h(w4[q >> 1][(q & 1) * 2 + 1]) << 16);
                            uint4 *o = (uint4 *)(g.o16[0] + (lh(kw) * g.T + kt) * 64 + dd0 + half * 16);
                            o[0] = make_uint4(p[0], p[1], p[2], p[3]);
                            o[1] = make_uint4(p[4], p[5], p[6], p[7]);
                        }
                    } else {
                        // V^T [64, T]: a lane's runs of 4 keys (with T % 4 == 0 all in one window)
#pragma unroll
                        for (int q = 0; q < 4; q++) {
                            const int tr = q * 8 + (ln >> 5) * 4;
                            uint16_t u[4];
#pragma unroll
                            for (int e = 0; e < 4; e++) u[e] = fw_f2h(acc[i][j][q * 4 + e] + bias[j]);
                            auto at = [&](int w, int t) {
                                return g.o16[1] + (lh(w) * 64 + dd0 + (ln & 31)) * g.T + t;
                            };
                            if ((g.T & 3) == 0) {
                                if (tr < vrows)
                                    *(uint2 *)at(vw[q], vt[q]) =
                                        make_uint2(u[0] | ((uint32_t)u[1] << 16), u[2] | ((uint32_t)u[3] << 16));
                            } else {
                                int w = vw[q], t = vt[q];
#pragma unroll
                                for (int e = 0; e < 4; e++) {
                                    if (tr + e < vrows) *at(w, t) = u[e];
                                    if (++t == g.T) {
                                        t = 0;
                                        w++;
                                    }
                                }
                            }
                        }
                    }
                }
            }
        }
        if (of && g.ovf) *g.ovf = 1;
    } else if constexpr (C::GELU) {
        const uint16_t *tab = (const uint16_t *)lds;
        FW_WAIT_VM(0);
        __syncthreads(); // the table is in LDS
        if constexpr (EPI == FW_EPI_CONV2) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int col = col0 + j * 32 + (lane & 31), colc = min(col, g.N - 1);
                    int tr[4]; // window position of each 4-row run
                    float ps[16];
#pragma unroll
                    for (int q = 0; q < 4; q++) tr[q] = (m0 + min(rowl(i, q * 4), mrows - 1)) % g.T;
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        int tt = tr[r >> 2] + (r & 3);
                        tt = tt >= g.T ? tt % g.T : tt;
                        ps[r] = g.pos[(size_t)tt * g.ldc + colc];
                    }
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const float v = g.bias ? acc[i][j][r] + bias[j] : acc[i][j][r];
                        const float tv = fw_h2f(tab[fw_f2h(v)]);
                        const float y = v <= -10.0f ? 0.0f : (v >= 10.0f ? v : tv);
                        if (rowl(i, r) < mrows && col < g.N) g.C[(size_t)(m0 + rowl(i, r)) * g.ldc + col] = y + ps[r];
                    }
                }
        } else {
            // hi = the table's f16 value; lo is zero but for v >= 10 (the value
            // itself).  Columns are processed in 64-wide blocks with a lo flag each.
            uint32_t of = 0;
#pragma unroll
            for (int jb = 0; jb < TN / 2; jb++) {
                bool big = false;
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 2 * jb; j < 2 * jb + 2; j++)
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            if (g.bias) acc[i][j][r] = acc[i][j][r] + bias[j];
                            big |= acc[i][j][r] >= 10.0f;
                        }
                const bool flag = __builtin_amdgcn_ballot_w64(big) != 0;
                const int cb = col0 + jb * 64;
                if (cb >= g.N || rw0 >= mrows) continue;
                if (lane == 0) {
                    if (g.lo_out) g.lo_out[(size_t)((m0 + rw0) >> 6) * GF_LOB + (cb >> 6)] = flag ? 1 : 0;
                    if (g.lo_any_out && flag) *g.lo_any_out = 1;
                }
                const bool wlo = flag || g.lo_any_out; // without per-block flags lo is written throughout
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    size_t ro[4]; // output row of each 4-row run's first row
                    int wr[4];    // rows left in that row's window
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const int row = m0 + min(rowl(i, q * 4), mrows - 1);
                        const int w = g.opad ? row / g.T : 0;
                        ro[q] = g.opad ? (size_t)row + (size_t)w * g.opad + 1 : (size_t)row;
                        wr[q] = g.opad ? g.T - (row - w * g.T) : 4;
                    }
#pragma unroll
                    for (int j = 2 * jb; j < 2 * jb + 2; j++) {
                        const int col = col0 + j * 32 + (lane & 31);
                        uint16_t u[16], lw[16];
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            const float v = acc[i][j][r];
                            u[r] = tab[fw_f2h(v)];
                            lw[r] = 0;
                            if (v <= -10.0f) u[r] = 0;
                        }
                        if (flag) {
#pragma unroll
                            for (int r = 0; r < 16; r++)
                                if (acc[i][j][r] >= 10.0f) fw_split2(acc[i][j][r], u[r], lw[r], of);
                        }
                        // two columns per dword: even lanes store row r, odd lanes row r + 1
                        auto put = [&](uint16_t *dst, const uint16_t (&x)[16]) {
#pragma unroll
                            for (int r = 0; r < 16; r += 2) {
                                const uint32_t mine = lane & 1 ? x[r + 1] : x[r], give = lane & 1 ? x[r] : x[r + 1];
                                const uint32_t got = __builtin_amdgcn_mov_dpp(give, FW_DPP_XOR1, 0xf, 0xf, false);
                                const uint32_t word = lane & 1 ? got | (mine << 16) : mine | (got << 16);
                                const int e = (r & 3) + (lane & 1), q = r >> 2;
                                if (rowl(i, q * 4) + e < mrows && col < g.N)
                                    *(uint32_t *)(dst + (ro[q] + e + (e >= wr[q] ? g.opad : 0)) * g.ldc + (col & ~1)) = word;
                            }
                        };
                        put(g.o16[0], u);
                        if (wlo) put(g.o16[1], lw);
                    }
                }
            }
            if (of && g.ovf) *g.ovf = 1;
        }
    }
}

template <int EPI, bool FL, int BM, int BN, int WGM, int WGN>
static void launch_f16(hipStream_t st, const FwGemm &g) {
    int ntw = 0, ntm;
    if (EPI == FW_EPI_QKV) {
        ntw = (g.T + BM - 1) / BM;
        ntm = (g.M / g.T) * ntw;
    } else {
        ntm = (g.M + BM - 1) / BM;
    }
    const int ntn = (g.N + BN - 1) / BN;
    hipLaunchKernelGGL((k_gemm_f16<EPI, FL, BM, BN, WGM, WGN>), dim3(ntm * ntn), dim3(64 * WGM * WGN), 0, st, g, ntm, ntn,
                       ntw);
}

template <int EPI, bool FL>
static void pick_f16(hipStream_t st, const FwGemm &g, int ncu) {
    // q/k/v tiles stop at a window's end (V^T runs of 8 keys); the cross K/V's run
    // over the windows: at 130 frames of 16 streams a window with tiles of its own is
    // 2 of 128 rows for 130 (set_cross + one step 813 -> 764 us, 10 streams of 260
    // frames 676 -> 607, 16 of 400 1,014 -> 957; from 1,500 frames on the same).
    constexpr bool win = EPI == FW_EPI_QKV;
    constexpr bool gelu = EPI == FW_EPI_GELU_SPLIT || EPI == FW_EPI_CONV2;
    // Rounds of the CUs times a round's time relative to 256 x 256 tiles, one
    // block to a CU (measured, 8 windows: both planes 82 us for a round of 256 x
    // 256 at K = 1280, 48 for 256 x 128, 52 for two 128 x 128 a CU; hi plane, fc2:
    // 178, 113, 127; the same weights at every width: whole f32 encoder calls of widths
    // 384-1,280, attention included, ran 1.36-1.54x faster than on 128 x 128 tiles).  A last round of 128 x 128 with one block to a CU costs
    // less than a full one; a GELU epilogue's table allows only one.
    auto blocks = [&](int bm, int bn) {
        const long long tm = win ? (long long)(g.M / g.T) * ((g.T + bm - 1) / bm) : (g.M + bm - 1) / bm;
        return tm * ((g.N + bn - 1) / bn);
    };
    const long long n2 = blocks(128, 128), left = n2 % (2 * ncu);
    const double c0 = (double)((blocks(256, 256) + ncu - 1) / ncu);
    const double c1 = (double)((blocks(256, 128) + ncu - 1) / ncu) * (FL ? 0.62 : 0.58);
    const double c2 = gelu ? (double)((n2 + ncu - 1) / ncu) * (FL ? 0.41 : 0.36)
                           : (double)(n2 / (2 * ncu)) * (FL ? 0.71 : 0.62) +
                                 (left == 0 ? 0.0 : left <= ncu ? 0.5 : FL ? 0.71 : 0.62);
    const int pick = c0 <= c1 && c0 <= c2 ? 0 : c1 < c2 ? 1 : 2;
    if (pick == 0) launch_f16<EPI, FL, 256, 256, 4, 2>(st, g);
    else if (pick == 1) launch_f16<EPI, FL, 256, 128, 4, 2>(st, g);
    else launch_f16<EPI, FL, 128, 128, 2, 2>(st, g);
}

bool fw_launch_gemm_f16(hipStream_t st, const FwGemm &g0, int ncu) {
    FwGemm g = g0;
    g.map = 1;
    if (g.K % 32 || g.N % 32) return false;
    switch (g.epi) {
    case FW_EPI_RESID:
        if (g.lo_in || g.lo_any) pick_f16<FW_EPI_RESID, true>(st, g, ncu);
        else pick_f16<FW_EPI_RESID, false>(st, g, ncu);
        return true;
    case FW_EPI_GELU_SPLIT: pick_f16<FW_EPI_GELU_SPLIT, false>(st, g, ncu); return true;
    case FW_EPI_CONV2: pick_f16<FW_EPI_CONV2, true>(st, g, ncu); return true;
    case FW_EPI_QKV: pick_f16<FW_EPI_QKV, false>(st, g, ncu); return true;
    case FW_EPI_XKV: pick_f16<FW_EPI_XKV, false>(st, g, ncu); return true;
    default: return false;
    }
}
