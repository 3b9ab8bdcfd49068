// enc_gemm.h — what the encoder's int8 and f16-pair GEMM kernels share.
#pragma once
#include "fw_enc.h"

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void fw_split2(float v, uint16_t &hi, uint16_t &lo) {
    asm volatile("" : "+v"(v));
    _Float16 h = (_Float16)v;
    float r = v - (float)h;
    asm volatile("" : "+v"(r));
    hi = __builtin_bit_cast(uint16_t, h);
    lo = __builtin_bit_cast(uint16_t, (_Float16)r);
}
// The same, or-ing into `of` whether the hi half overflows: |v| >= 65520
// rounds to an infinite f16 (65504 is the largest finite one), and the pair
// then carries inf / NaN instead of v.
__device__ __forceinline__ void fw_split2(float v, uint16_t &hi, uint16_t &lo, uint32_t &of) {
    of |= fabsf(v) >= 65520.0f ? 1u : 0u;
    fw_split2(v, hi, lo);
}

// Block id -> tile sequence number.  map 1: the hardware deals blocks
// round-robin to the 8 XCDs, so block ids are remapped to give each XCD a
// contiguous run of the tile sequence; map 0: identity.
__device__ __forceinline__ int gemm_tile_order(int map) {
    const int nb = gridDim.x, bid = blockIdx.x;
    if (!map) return bid;
    const int xcd = bid & 7, loc = bid >> 3, per = nb >> 3, rem = nb & 7;
    return xcd < rem ? xcd * (per + 1) + loc : rem * (per + 1) + (xcd - rem) * per + loc;
}

// LDS rows are 64 bytes; the 16-byte chunk c of row r sits at chunk c ^ gsw(r),
// so MFMA fragment reads (32 rows of one chunk) are free of bank conflicts.
__device__ __forceinline__ int gsw(int r) { return (r ^ (r >> 2)) & 3; }

// One 32 x 32 tile of the fused q/k/v output (columns c0.. of [3d], rows t0.. of
// window wnd, the first vrows of them valid; v: accumulator layout, element r of
// lane l is row (r/4)*8 + (l/32)*4 + r%4, column l%32) as f16 hi/lo pairs.
// Q, K: [B, H, T, 64] rows, written through a wave-private LDS slab (32 rows of
// 40 floats) so each lane stores 16 consecutive dims (32-byte runs).
// V^T: [B, H, 64, Tp] at key positions fw_vt_pos(t); a lane's 8 values
// r = 8c .. 8c+7 sit at 8 consecutive positions (t0 is a multiple of 32), so
// they go out as 16-byte runs.
__device__ __forceinline__ void qkv_store32(const FwGemm &g, float *slab, const float (&v)[16], int ln, int c0,
                                            int wnd, int t0, int vrows, uint32_t &of) {
    const int d = g.ldc;
    const int which = c0 / d, cc = c0 - which * d, h = cc >> 6, dd0 = cc & 63;
    if (which == 2) {
        const int dd = dd0 + (ln & 31);
        uint16_t *vh = g.o16[4] + (((size_t)wnd * g.H + h) * 64 + dd) * g.Tp;
        uint16_t *vl = g.o16[5] + (((size_t)wnd * g.H + h) * 64 + dd) * g.Tp;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int pb = t0 + 16 * c + 8 * (ln >> 5); // first of 8 positions
            uint16_t hi[8], lo[8];
#pragma unroll
            for (int e = 0; e < 8; e++) fw_split2(v[8 * c + e], hi[e], lo[e], of);
            if (16 * c + 16 <= vrows) {
                uint4 ph, pl;
                ph.x = hi[0] | ((uint32_t)hi[1] << 16);
                ph.y = hi[2] | ((uint32_t)hi[3] << 16);
                ph.z = hi[4] | ((uint32_t)hi[5] << 16);
                ph.w = hi[6] | ((uint32_t)hi[7] << 16);
                pl.x = lo[0] | ((uint32_t)lo[1] << 16);
                pl.y = lo[2] | ((uint32_t)lo[3] << 16);
                pl.z = lo[4] | ((uint32_t)lo[5] << 16);
                pl.w = lo[6] | ((uint32_t)lo[7] << 16);
                *(uint4 *)(vh + pb) = ph;
                *(uint4 *)(vl + pb) = pl;
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    // value e is key t0 + 16c + 8*(e/4) + 4*(lane/32) + e%4
                    const int rr = 16 * c + 8 * (e >> 2) + 4 * (ln >> 5) + (e & 3);
                    if (rr < vrows) {
                        const int p = fw_vt_pos(t0 + rr);
                        vh[p] = hi[e];
                        vl[p] = lo[e];
                    }
                }
            }
        }
    } else {
        // the slab is private to this wave and a wave's LDS accesses
        // run in order: only the compiler must not reorder them
        asm volatile("" ::: "memory");
#pragma unroll
        for (int r = 0; r < 16; r++)
            slab[((r >> 2) * 8 + (ln >> 5) * 4 + (r & 3)) * 40 + (ln & 31)] = v[r];
        asm volatile("" ::: "memory");
        const int row = ln >> 1, half = ln & 1;
        v4f w4[4];
#pragma unroll
        for (int q = 0; q < 4; q++) w4[q] = *(const v4f *)(slab + row * 40 + half * 16 + q * 4);
        asm volatile("" ::: "memory");
        if (row < vrows) {
            uint32_t ph[8], pl[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                uint16_t h0, l0, h1, l1;
                fw_split2(w4[q >> 1][(q & 1) * 2], h0, l0, of);
                fw_split2(w4[q >> 1][(q & 1) * 2 + 1], h1, l1, of);
                ph[q] = h0 | ((uint32_t)h1 << 16);
                pl[q] = l0 | ((uint32_t)l1 << 16);
            }
            const size_t o = (((size_t)wnd * g.H + h) * g.T + t0 + row) * 64 + dd0 + half * 16;
            uint4 *qh = (uint4 *)(g.o16[2 * which] + o), *ql = (uint4 *)(g.o16[2 * which + 1] + o);
            qh[0] = make_uint4(ph[0], ph[1], ph[2], ph[3]);
            qh[1] = make_uint4(ph[4], ph[5], ph[6], ph[7]);
            ql[0] = make_uint4(pl[0], pl[1], pl[2], pl[3]);
            ql[1] = make_uint4(pl[4], pl[5], pl[6], pl[7]);
        }
    }
}
