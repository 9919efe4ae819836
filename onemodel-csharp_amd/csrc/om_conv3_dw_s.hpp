// Weight gradient of the 3x3 convolutions with stride 1 and padding 1 on the bf16 matrix cores from exactly split fp32
// operands (om_split.hpp).
//
// The sum runs over pixels, so a fragment holds eight neighbouring pixels of one channel and a tap shifts it by a pixel.
// A workgroup takes 64 output x 32 input channels and walks items of RB output rows x SG groups of eight columns, staging
// g as [plane][co][row][8 SG columns] and x as [plane][ci][row][8 SG + 8 columns], column c of the segment at c + 1: the
// left tap's fragment is one aligned 16-byte read, and the next word gives the other two taps by 16-bit shifts of the packed
// pairs, so nothing is split or staged twice. Wavefront (b, ky) holds the three taps of row ky for 32 output channels: six
// wavefronts and 96 accumulators each, two workgroups a CU, one staging while the other multiplies. Channel strides are odd
// in 16-byte units, for the banks of the fragment reads. Measured with its reduce: 8 x 64 at 57 x 57 42 us. What bounds it: an
// item's loads are not begun while the one before is multiplied (the accumulators leave no registers for them).
#pragma once

#include "om_split.hpp"

namespace oc3w {

using namespace oms;

constexpr int kCo = 64, kCi = 32, kThreads = 384;
// Quads of four columns staged for one channel at most: geometry() keeps RB and SG within them.
constexpr int kGQuads = 18, kXQuads = 48;

// Segments of at most four groups and bands of about eight groups: near-square tiles stage the fewest halo columns.
inline void geometry(int H, int W, int &RB, int &SG, int &bands, int &segs) {
    const int groups = (W + 7) / 8;
    segs = (groups + 3) / 4;
    SG = (groups + segs - 1) / segs;  // 1 .. 4
    RB = 8 / SG < H ? 8 / SG : H;
    bands = (H + RB - 1) / RB;
}

struct Args {
    const float *g, *x;
    float *part;   // [slot][co][tap][ci]
    double *dbp;   // [slot][co], or null
    int cin, cout, H, W, RB, SG, bands, segs, items, per;
};

// 16-byte units of one channel: its rows, made odd.
__host__ __device__ constexpr int g_units(int RB, int SG) { return (RB * SG) | 1; }
__host__ __device__ constexpr int x_units(int RB, int SG) { return ((RB + 2) * (SG + 1)) | 1; }
constexpr int lds_bytes(int RB, int SG) { return 3 * 16 * (kCo * g_units(RB, SG) + kCi * x_units(RB, SG)); }

// One channel's staged quads q, q + TPC, ... (NU of them): `tab` holds each quad's row << 16 | column. r0, c0: the image row
// and column of the first; zeros outside the image. Loads are free of branches, so all fly together: four columns clamped
// into the row (V4: rows of at least four), moved into place when they are taken.
template <int TPC, int NU, bool V4>
struct Quads {
    float v[NU][4];
    __device__ __forceinline__ void load(const float *src, const int *tab, int n, int q, int r0, int c0, int H, int W) {
#pragma unroll
        for (int i = 0; i < NU; i++) {
            const int t = tab[min(q + i * TPC, n - 1)], iy = r0 + (t >> 16), ix = c0 + (t & 0xFFFF);
            const float *s = src + min(max(iy, 0), H - 1) * W;
            if constexpr (V4) {
                const f4u x = *reinterpret_cast<const f4u *>(s + min(max(ix, 0), W - 4));
#pragma unroll
                for (int e = 0; e < 4; e++) v[i][e] = x[e];
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) v[i][e] = s[min(max(ix + e, 0), W - 1)];
            }
        }
    }
    template <class Each>
    __device__ __forceinline__ void store(char *dst, int plane, const int *tab, int n, int q, int r0, int c0, int H, int W,
                                          Each each) {
#pragma unroll
        for (int i = 0; i < NU; i++) {
            const int u = q + i * TPC, t = tab[min(u, n - 1)], iy = r0 + (t >> 16), ix = c0 + (t & 0xFFFF);
            const bool row = (unsigned)iy < (unsigned)H;
            float x[4];
            if (V4 && row && (unsigned)ix <= (unsigned)(W - 4)) {
#pragma unroll
                for (int e = 0; e < 4; e++) x[e] = v[i][e];
            } else {
                const int d = V4 ? ix - min(max(ix, 0), W - 4) : 0;  // the quad starts d columns after what was loaded
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float y = v[i][e];
                    if constexpr (V4) {
#pragma unroll
                        for (int j = 0; j < 4; j++) y = e + d == j ? v[i][j] : y;
                    }
                    x[e] = row && (unsigned)(ix + e) < (unsigned)W ? y : 0.0f;
                }
            }
            if (u >= n) continue;
            each(x);
            uint32_t h0, m0, l0, h1, m1, l1;
            split2(x[0], x[1], h0, m0, l0);
            split2(x[2], x[3], h1, m1, l1);
            *reinterpret_cast<u32x2 *>(dst + u * 8) = u32x2{h0, h1};
            *reinterpret_cast<u32x2 *>(dst + plane + u * 8) = u32x2{m0, m1};
            *reinterpret_cast<u32x2 *>(dst + 2 * plane + u * 8) = u32x2{l0, l1};
        }
    }
};

template <bool V4>
__global__ void __launch_bounds__(kThreads, 3) k_conv3_dw_s(Args a) {
    OM_LDS_POISON();
    extern __shared__ __attribute__((aligned(16))) char sh[];
    const int gu = g_units(a.RB, a.SG) * 16, xu = x_units(a.RB, a.SG) * 16, gplane = kCo * gu, xplane = kCi * xu;
    char *Gs = sh, *Xs = sh + 3 * gplane;
    int lin = blockIdx.x;
    if ((gridDim.x & 7) == 0) lin = (lin & 7) * (gridDim.x >> 3) + (lin >> 3);  // one slot's blocks on one XCD
    const int ncib = a.cin / kCi, ncob = a.cout / kCo, P = a.H * a.W;
    const int cib = lin % ncib, cob = lin / ncib % ncob, slot = lin / ncib / ncob;
    const int co0 = cob * kCo, ci0 = cib * kCi, tid = threadIdx.x;
    const int lane = tid & 63, l32 = lane & 31, hg = lane >> 5, w = tid >> 6, blk = w & 1, ky = w >> 1;
    const int gch = tid / 6, gq = tid % 6, xch = tid / 12, xq = tid % 12;
    const bool do_db = a.dbp && cib == 0;
    const int i0 = slot * a.per, i1 = min(a.items, i0 + a.per), ngrp = a.RB * a.SG;
    __shared__ int gtab[kGQuads], xtab[kXQuads];
    const int gn = a.RB * 2 * a.SG, xn = (a.RB + 2) * 2 * (a.SG + 1);
    if (tid < gn) gtab[tid] = tid / (2 * a.SG) << 16 | tid % (2 * a.SG) * 4;
    if (tid < xn) xtab[tid] = tid / (2 * a.SG + 2) << 16 | tid % (2 * a.SG + 2) * 4;
    __syncthreads();
    double dbs = 0.0;
    floatx16 acc[3], low[3];
#pragma unroll
    for (int t = 0; t < 3; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[t][e] = low[t][e] = 0.0f;
    const char *gl = Gs + (32 * blk + l32) * gu, *xl = Xs + l32 * xu;
    for (int item = i0; item < i1; item++) {
        const int seg = item % a.segs, band = item / a.segs % a.bands, n = item / a.segs / a.bands;
        const int oy = band * a.RB, ox = seg * a.SG * 8;
        Quads<6, kGQuads / 6, V4> gv;
        Quads<12, kXQuads / 12, V4> xv;
        gv.load(a.g + ((int64_t)n * a.cout + co0 + gch) * P, gtab, gn, gq, oy, ox, a.H, a.W);
        xv.load(a.x + ((int64_t)n * a.cin + ci0 + xch) * P, xtab, xn, xq, oy - 1, ox - 1, a.H, a.W);
        __syncthreads();  // the previous item's reads are done
        gv.store(Gs + gch * gu, gplane, gtab, gn, gq, oy, ox, a.H, a.W, [&](const float (&v)[4]) {
            if (do_db) dbs += ((double)v[0] + (double)v[1]) + ((double)v[2] + (double)v[3]);
        });
        xv.store(Xs + xch * xu, xplane, xtab, xn, xq, oy - 1, ox - 1, a.H, a.W, [](const float (&)[4]) {});
        __syncthreads();
#pragma unroll 1
        for (int f = 0; f < ngrp; f += 2) {
            const int grp = min(f + hg, ngrp - 1), r = grp / a.SG, j = grp - r * a.SG;
            const char *gp = gl + grp * 16, *xp = xl + ((r + ky) * (a.SG + 1) + j) * 16;
            u32x4 fg[3], f0[3], f1[3], f2[3];
#pragma unroll
            for (int q = 0; q < 3; q++) {
                fg[q] = *reinterpret_cast<const u32x4 *>(gp + q * gplane);
                f0[q] = *reinterpret_cast<const u32x4 *>(xp + q * xplane);
                const uint32_t nx = *reinterpret_cast<const uint32_t *>(xp + q * xplane + 16);
                if (f + hg >= ngrp) fg[q] = u32x4{0, 0, 0, 0};  // an odd number of groups: nothing for the upper half
#pragma unroll
                for (int e = 0; e < 3; e++) {
                    f1[q][e] = __builtin_amdgcn_alignbit(f0[q][e + 1], f0[q][e], 16);
                    f2[q][e] = f0[q][e + 1];
                }
                f1[q][3] = __builtin_amdgcn_alignbit(nx, f0[q][3], 16);
                f2[q][3] = nx;
            }
            mma6(fg, f0, acc[0], low[0]);
            mma6(fg, f1, acc[1], low[1]);
            mma6(fg, f2, acc[2], low[2]);
        }
    }
    unsigned big = 0;
#pragma unroll
    for (int t = 0; t < 3; t++) {
        finish_sums(acc[t], low[t]);
#pragma unroll
        for (int e = 0; e < 16; e++) note(acc[t][e], big);
    }
    // element e: output channel 8 (e / 4) + 4 hg + e % 4 of the wavefront's 32
    float *dst = a.part + (((int64_t)slot * a.cout + co0 + 32 * blk + 4 * hg) * 9 + 3 * ky) * a.cin + ci0 + l32;
    if (beyond(big)) {  // values the split does not carry: this wavefront's sums on the fp32 instruction, from global memory
        floatx16 s[3];
#pragma unroll
        for (int t = 0; t < 3; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) s[t][e] = 0.0f;
#pragma unroll 1
        for (int item = i0; item < i1; item++) {
            const int seg = item % a.segs, band = item / a.segs % a.bands, n = item / a.segs / a.bands;
            const float *gg = a.g + ((int64_t)n * a.cout + co0 + 32 * blk + l32) * P;
            const float *xx = a.x + ((int64_t)n * a.cin + ci0 + l32) * P;
            const int ox1 = min(a.W, (seg + 1) * a.SG * 8);
#pragma unroll 1
            for (int oy = band * a.RB; oy < min(a.H, (band + 1) * a.RB); oy++) {
                const int iy = oy + ky - 1;
                const bool row = (unsigned)iy < (unsigned)a.H;
                const float *gr = gg + oy * a.W, *xr = xx + (row ? iy : oy) * a.W;
#pragma unroll 1
                for (int ox = seg * a.SG * 8; ox < ox1; ox += 8) {
#pragma unroll
                    for (int j = 0; j < 8; j += 2) {
                        const int px = ox + j + hg;
                        const bool has = px < ox1;
                        const float gv = gr[min(px, a.W - 1)];
#pragma unroll
                        for (int t = 0; t < 3; t++) {
                            const int ix = px + t - 1;
                            const float v = xr[min(max(ix, 0), a.W - 1)];
                            s[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                                has ? gv : 0.0f, has && row && (unsigned)ix < (unsigned)a.W ? v : 0.0f, s[t], 0, 0, 0);
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < 3; t++) take_beyond(acc[t], s[t]);
    }
#pragma unroll
    for (int t = 0; t < 3; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) dst[((int64_t)(8 * (e >> 2) + (e & 3)) * 9 + t) * a.cin] = acc[t][e];
    if (!do_db) return;  // uniform over the workgroup
    __syncthreads();
    double *ds = reinterpret_cast<double *>(sh);
    ds[tid] = dbs;
    __syncthreads();
    if (tid < kCo) {
        double v = ds[6 * tid];
#pragma unroll
        for (int q = 1; q < 6; q++) v += ds[6 * tid + q];
        a.dbp[(int64_t)slot * a.cout + co0 + tid] = v;
    }
}

}  // namespace oc3w
