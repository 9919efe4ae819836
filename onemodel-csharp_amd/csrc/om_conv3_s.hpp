// 3x3 convolutions with stride 1 and padding 1, forward and input gradient, on the bf16 matrix cores from exactly split
// fp32 operands (om_split.hpp).
//
// The fp32 matrix instruction bounded these (81 TFLOP/s at 32 x 64 x 56 x 56, 0.52 of its peak). Split operands suit a
// convolution better than a dense product, since every staged input value serves nine taps times all the block's output
// channels: splitting costs a tenth of the vector work per matrix instruction that it costs there.
//
// A workgroup takes 32 NW output pixels (flattened, so any width works) of one image and 32 CB output channels, and walks
// the input channels 16 at a time. Per chunk it splits the input rows its pixels touch, halo included and zero outside the
// image, into LDS as [plane][row][column][16 channels], and the weights as [tap][plane][co][16 channels]. A fragment is
// one 16-byte read per plane (lane = pixel or output channel, eight channels per lane group), and a tap is a constant shift
// of the lane's pixel address. Units of four channels of one position are loaded by four neighbouring lanes, so the LDS
// stores are contiguous; the next chunk's loads fly while this one is multiplied. A wavefront holds 32 pixels x all the
// block's channels; lanes are pixels, so the stores run along rows.
//
// Measured (us, fp32 kernel before): 32 x 64 -> 64 channels, 56 x 56: forward 99 -> 62 (119 TFLOP/s of fp32 products), dX
// 99 -> 63; 32 x 32 -> 64, 16 x 64: forward and its split sum with pool 29.6 -> 20.2, dX 22 -> 18.0. What bounds it: one workgroup a CU (98 KB
// of LDS) leaves the splitting (6 us of 60) and the epilogue (5) beside idle matrix cores, 416 workgroups make 1.6 rounds
// over 256 CUs, and 42 us remain with nothing but fragment reads and MFMA. Two pixel blocks a wavefront (9 reads for 12
// instructions less, half the wavefronts) measured 65-70.
#pragma once

#include "om_split.hpp"

namespace oc3 {

using namespace oms;

struct Args {
    const float *in, *wt, *bias;
    float *out, *ws;
    int cin, cout, H, W, R, ntile, N, nsplit, cps, acc, relu;
};

__device__ __forceinline__ float relu1(float v) { return v > 0.0f ? v : (v == v ? 0.0f : v); }

// LDS bytes for R staged rows of an image W wide and 32 cb output channels.
constexpr int lds_bytes(int R, int W, int cb) { return R * (W + 2) * 96 + 9 * 32 * cb * 96; }

template <int CB, int NW, int NU, bool FLIP>
__global__ void __launch_bounds__(64 * NW, 2) k_conv3_s(Args a) {
    OM_LDS_POISON();
    constexpr int NT = 64 * NW, BM = 32 * CB, WU = BM * 4;  // WU units of (output channel, four input channels)
    constexpr int NWU = (WU + NT - 1) / NT;
    extern __shared__ __attribute__((aligned(16))) char sh[];
    const int cols = a.W + 2, npos = a.R * cols, xplane = npos * 32, P = a.H * a.W;
    char *Xs = sh, *Ws = sh + 3 * xplane;  // Ws: [tap][plane][BM][32 bytes]
    int lin = blockIdx.x;
    if ((gridDim.x & 7) == 0) lin = (lin & 7) * (gridDim.x >> 3) + (lin >> 3);  // neighbouring tiles on one XCD
    const int ncb = a.cout / BM;
    const int tile = lin % a.ntile, cb = (lin / a.ntile) % ncb, n = (lin / a.ntile / ncb) % a.N, split = lin / a.ntile / ncb / a.N;
    const int c_beg = split * a.cps * 16, c_end = min(a.cin, c_beg + a.cps * 16);
    const int p0 = tile * 32 * NW, co0 = cb * BM, oy0 = p0 / a.W;
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5, w = threadIdx.x >> 6;
    const float *inn = a.in + (int64_t)n * a.cin * P;

    // Units of the staged input: position t / 4, channels 4 (t % 4) .. + 3. xo: element offset in the chunk's planes
    // (-1: zero).
    int xo[NU];
#pragma unroll
    for (int i = 0; i < NU; i++) {
        const int u = threadIdx.x + i * NT, pos = u >> 2, iy = oy0 - 1 + pos / cols, ix = pos % cols - 1;
        const bool in = pos < npos && (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
        xo[i] = in ? 4 * (u & 3) * P + iy * a.W + ix : -1;
    }
    float xv[NU][4], wv[NWU][36];
    auto load = [&](int c0) {
        const float *x = inn + (int64_t)c0 * P;
#pragma unroll
        for (int i = 0; i < NU; i++) {
            const int o = max(xo[i], 0);
#pragma unroll
            for (int e = 0; e < 4; e++) xv[i][e] = x[o + e * P];
        }
#pragma unroll
        for (int i = 0; i < NWU; i++) {
            const int u = min((int)threadIdx.x + i * NT, WU - 1), co = co0 + (u >> 2), q = u & 3;
            if constexpr (FLIP) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float *s = a.wt + ((int64_t)(c0 + 4 * q + e) * a.cout + co) * 9;
                    const f4u v0 = *reinterpret_cast<const f4u *>(s), v1 = *reinterpret_cast<const f4u *>(s + 4);
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        wv[i][9 * e + t] = v0[t];
                        wv[i][9 * e + 4 + t] = v1[t];
                    }
                    wv[i][9 * e + 8] = s[8];
                }
            } else {
                const float *s = a.wt + ((int64_t)co * a.cin + c0 + 4 * q) * 9;
#pragma unroll
                for (int t = 0; t < 9; t++) {
                    const f4u v = *reinterpret_cast<const f4u *>(s + 4 * t);
#pragma unroll
                    for (int e = 0; e < 4; e++) wv[i][4 * t + e] = v[e];
                }
            }
        }
    };
    auto put = [&](char *d, int plane, const float (&x)[4]) {
        uint32_t h0, m0, l0, h1, m1, l1;
        split2(x[0], x[1], h0, m0, l0);
        split2(x[2], x[3], h1, m1, l1);
        *reinterpret_cast<u32x2 *>(d) = u32x2{h0, h1};
        *reinterpret_cast<u32x2 *>(d + plane) = u32x2{m0, m1};
        *reinterpret_cast<u32x2 *>(d + 2 * plane) = u32x2{l0, l1};
    };
    auto store = [&] {
#pragma unroll
        for (int i = 0; i < NU; i++) {
            const int u = threadIdx.x + i * NT;
            if (u >= npos * 4) continue;
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = xo[i] >= 0 ? xv[i][e] : 0.0f;
            put(Xs + u * 8, xplane, x);
        }
#pragma unroll
        for (int i = 0; i < NWU; i++) {
            const int u = threadIdx.x + i * NT;
            if (u >= WU) continue;
#pragma unroll
            for (int t = 0; t < 9; t++) {
                const int s = FLIP ? 8 - t : t;
                const float x[4] = {wv[i][s], wv[i][9 + s], wv[i][18 + s], wv[i][27 + s]};
                put(Ws + t * (3 * BM * 32) + u * 8, BM * 32, x);
            }
        }
    };

    const int p = p0 + 32 * w + l32;  // past the last pixel: any staged place
    const char *xl = Xs + (p < P ? (p / a.W - oy0) * cols + p % a.W : 0) * 32 + g * 16;
    const char *wl = Ws + l32 * 32 + g * 16;
    floatx16 acc[CB], low[CB];
#pragma unroll
    for (int i = 0; i < CB; i++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[i][e] = low[i][e] = 0.0f;
    u32x4 fx[2][3], fw[2][CB][3];
    auto rd = [&](int s, int tap) {
        const int xt = ((tap / 3) * cols + tap % 3) * 32, wt = tap * (3 * BM * 32);
#pragma unroll
        for (int q = 0; q < 3; q++) fx[s][q] = *reinterpret_cast<const u32x4 *>(xl + xt + q * xplane);
#pragma unroll
        for (int i = 0; i < CB; i++)
#pragma unroll
            for (int q = 0; q < 3; q++) fw[s][i][q] = *reinterpret_cast<const u32x4 *>(wl + wt + q * (BM * 32) + i * 1024);
    };
    load(c_beg);
    for (int c0 = c_beg; c0 < c_end; c0 += 16) {
        store();
        __syncthreads();
        load(min(c0 + 16, c_end - 16));  // in flight while this chunk is multiplied (the last one again at the end)
        rd(0, 0);
#pragma unroll
        for (int tap = 0; tap < 9; tap++) {
            if (tap < 8) rd((tap + 1) & 1, tap + 1);
#pragma unroll
            for (int i = 0; i < CB; i++) mma6(fw[tap & 1][i], fx[tap & 1], acc[i], low[i]);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
    }
    unsigned big = 0;
#pragma unroll
    for (int i = 0; i < CB; i++) {
        finish_sums(acc[i], low[i]);
#pragma unroll
        for (int e = 0; e < 16; e++) note(acc[i][e], big);
    }
    if (beyond(big)) {  // values the split does not carry: this wavefront's sums on the fp32 instruction, from global memory
        floatx16 f[CB];
        const int pc = min(p, P - 1), oy = pc / a.W, ox = pc % a.W;
#pragma unroll
        for (int i = 0; i < CB; i++)
#pragma unroll
            for (int e = 0; e < 16; e++) f[i][e] = 0.0f;
#pragma unroll 1
        for (int c0 = c_beg; c0 < c_end; c0 += 2) {
            const int c = c0 + g;
            const float *x = inn + (int64_t)c * P;
            const float *ww = a.wt + (FLIP ? (int64_t)c * a.cout + co0 + l32 : (int64_t)(co0 + l32) * a.cin + c) * 9;
#pragma unroll
            for (int t = 0; t < 9; t++) {
                const int iy = oy + t / 3 - 1, ix = ox + t % 3 - 1;
                const bool in = (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
                const float v = x[in ? iy * a.W + ix : 0];
#pragma unroll
                for (int i = 0; i < CB; i++)  // an infinite weight on the border: NaN
                    f[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(ww[(int64_t)32 * 9 * i * (FLIP ? 1 : a.cin) + (FLIP ? 8 - t : t)],
                                                                  in ? v : 0.0f, f[i], 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < CB; i++) take_beyond(acc[i], f[i]);
    }
    const bool part = a.nsplit > 1;
    float *dst = (part ? a.ws + (int64_t)split * a.N * a.cout * P : a.out) + ((int64_t)n * a.cout + co0) * P + p;
    // element e of block i: channel 32 i + 8 (e / 4) + 4 g + e % 4. Each pass runs over all of them before the next, so that
    // its loads or stores are in flight together.
    auto each = [&](auto f) {
#pragma unroll
        for (int i = 0; i < CB; i++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][e] = f(acc[i][e], 32 * i + 8 * (e >> 2) + (e & 3));
    };
    if (!part && a.bias) {
        const float *b = a.bias + co0 + 4 * g;
        each([&](float v, int co) { return v + b[co]; });
    }
    if (!part && a.relu) each([&](float v, int) { return relu1(v); });
    if (p >= P) return;
    dst += (int64_t)4 * g * P;
    if (!part && a.acc) each([&](float v, int co) { return dst[(int64_t)co * P] + v; });
    each([&](float v, int co) { return dst[(int64_t)co * P] = v; });
}

}  // namespace oc3
