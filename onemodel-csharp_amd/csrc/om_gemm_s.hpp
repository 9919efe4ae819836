// The dense product's kernel: fp32 operands multiplied on the bf16 matrix cores from three parts each that hold all of
// their bits.
//
// What bounds it and why this form: v_mfma_f32_16x16x4_f32 tops out at 157 TFLOP/s, v_mfma_f32_32x32x16_bf16 at 16 times
// that. Every fp32 operand is split exactly into three bf16 values, x = h + m + l (8 + 8 + 8 significand bits, each the
// rounding of what the previous ones leave), and the product keeps the six terms hh, hm, mh, hl, lh, mm; the dropped ml, lm
// and ll are together below 2^-24 (1 + 2^-9) of |x||y| (2^-24.15 found), half an ulp of the product. hh accumulates in one
// fp32 accumulator and the five small terms in another, so the large sum takes one rounding per 16 products instead of one
// per product or four. Against 64-bit sums of normal operands the 2-norm error is 1.1e-7 at K = 384 and 2.7e-7 at 4096, the
// fp32 instruction's 3.5e-7 and 1.1e-6.
//
// Operands are scaled by 2^24 on their way in, so no part of the smallest subnormal underflows, and the sums by 2^-48 on
// their way out (om_split.hpp). What the scaled range does not hold takes the fp32 instruction: infinities, NaN, operands of
// 2^104 and sums of 2^80 leave a non-finite sum, and a wavefront that finds some among its finished sums computes its tile
// again with v_mfma_f32_32x32x2_f32 straight from global memory and takes those sums from there.
//
// A workgroup is MG x KG wavefronts and computes BM x BN = (32 MG) x (32 TN) of C. Each wavefront owns 32 rows and all BN
// columns, so its A fragments are used by no other wavefront: it loads them from global memory straight into the MFMA layout
// and splits them in registers. B is split once per workgroup on its way into LDS, in fragment order (three bf16 planes; a
// wavefront's fragment read is 64 consecutive 16-byte slots), double-buffered with one barrier per 32 k. KG > 1 wavefront
// groups take every KG-th 32-k step each and their sums are added through LDS in group order: a product with few tiles then
// keeps four wavefronts per CU busy.
//
// The MFMA's first operand is B and its second A, so lane l holds C at row l % 32 and columns 8 q + 4 (l / 32) .. + 3 (q =
// 0 .. 3) of each 32 x 32 block.
//
// The k of a 32-step are permuted alike for both operands: lane group g (= l / 32) and element e of 16 hold k = 8 (e / 4) +
// 4 g + e % 4, so a lane's 16-byte loads of a K-contiguous row and its pair's cover 32 consecutive bytes.
#pragma once

#include "om_gemm_core.hpp"
#include "om_split.hpp"

namespace omg {
namespace gs {

using namespace oms;

// ------------------------------------------------------------------------------------------------------------ loads
// Byte offsets from a uniform pointer stay in 32 bits (the host checks them), so a load is one instruction.
__device__ __forceinline__ const float *at(const float *base, unsigned off) {
    return reinterpret_cast<const float *>(reinterpret_cast<const char *>(base) + off);
}
// k clamped below kend, for loads whose value is then dropped.
__device__ __forceinline__ int kclamp(int k, int kend) { return k < kend ? k : kend - 1; }

// A wavefront's 32 rows x 32 k, raw, in quads: quad w holds elements 4 w .. 4 w + 3 of the lane's row l32, straight from
// memory. KC: stored [m][k], else [k][m]. Lanes past the last row read row m - 1; their results are not stored. (Loading
// [m][k] rows eight lanes to a row and changing layout through LDS gave the same times at every size tried.)
template <bool KC>
struct ALoad {
    const float *base;  // element (row r0, k 0)
    int64_t ld;
    int g;
    unsigned off[KC ? 1 : 4];
    __device__ __forceinline__ ALoad(const float *a, int64_t ld_, int r0, int m, int lane) : ld(ld_) {
        const int row = min(lane & 31, m - 1 - r0);
        g = lane >> 5;
        base = a + (KC ? (int64_t)r0 * ld : (int64_t)r0);
        if constexpr (KC) {
            off[0] = 4u * (unsigned)(row * ld + 4 * g);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) off[e] = 4u * (unsigned)((4 * g + e) * ld + row);
        }
    }
    __device__ __forceinline__ void quad(float (&x)[4], int w, int k0) const {
        if constexpr (KC) {
            const f4u v = *reinterpret_cast<const f4u *>(at(base + k0 + 8 * w, off[0]));
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = v[e];
        } else {
            const float *p = base + (int64_t)(k0 + 8 * w) * ld;
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = *at(p, off[e]);
        }
    }
    // The same with elements at or past kend zero.
    __device__ __forceinline__ void quad_tail(float (&x)[4], int w, int k0, int kend) const {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int k = k0 + 8 * w + 4 * g + e, kc = kclamp(k, kend);
            const float v = KC ? *at(base + kc - 4 * g, off[0]) : *at(base + (int64_t)(kc - 4 * g - e) * ld, off[e]);
            x[e] = k < kend ? v : 0.0f;
        }
    }
};

// LDS byte offset of the 8-byte half slot (row, c = k / 4) of plane 0. A block of 32 rows is two 16-k halves of three
// 1 KB planes; slots stand in fragment order with the row XORed so that neither the stores (eight lanes per row, or
// several rows per lane) nor the fragment reads put two 16-byte slots of a phase on the same banks.
__device__ __forceinline__ int bswz(int row, int g, int h) { return (row & 31) ^ (4 * (g + 2 * h)) ^ ((row >> 4) & 3); }
__device__ __forceinline__ int bslot(int row, int c) {
    const int g = c & 1, h = c >> 2;
    return (row >> 5) * 6144 + h * 3072 + (g * 32 + bswz(row, g, h)) * 16 + ((c >> 1) & 1) * 8;
}
// BN rows (columns of C) x 32 k, loaded by NTH threads in units of quads (four k of one row), split and stored. KC:
// stored [n][k], a unit is one quad; else [k][n], a unit is RV rows x 4 k from RV-wide loads. Rows past the last
// column read the last ones again: a KC row column n - 1, an RV-wide load the last RV columns (the epilogue takes the
// quad of such columns from there).
template <int BN, int NTH, bool KC>
struct BLoad {
    static constexpr int RV = KC ? 1 : BN * 2 % NTH == 0 ? 4 : BN * 4 % NTH == 0 ? 2 : 4;
    static constexpr int UNITS = BN * 8 / RV;
    static constexpr int NU = (UNITS + NTH - 1) / NTH;
    static constexpr bool RAGGED = UNITS % NTH != 0;
    static constexpr int QUADS = NU * RV;  // per thread
    const float *base;                     // element (column n0, k 0)
    int64_t ld;
    int t;
    unsigned off[NU];
    int soff[NU];
    __device__ __forceinline__ BLoad(const float *b, int64_t ld_, int n0, int n, int t_) : ld(ld_), t(t_) {
        const int back = KC ? 0 : max(n0 + RV - n, 0);  // a tile with fewer than RV columns starts its loads earlier
        base = b + (KC ? (int64_t)n0 * ld : (int64_t)(n0 - back));
#pragma unroll
        for (int i = 0; i < NU; i++) {
            const int u = min(t + i * NTH, UNITS - 1);
            if constexpr (KC) {
                off[i] = 4u * (unsigned)(min(u >> 3, n - 1 - n0) * ld + 4 * (u & 7));
                soff[i] = bslot(u >> 3, u & 7);
            } else {
                const int q = u % (BN / RV), c = u / (BN / RV);
                off[i] = 4u * (unsigned)(4 * c * ld + shifted(RV * q, n - n0) + back);
                soff[i] = bslot(RV * q, c);
            }
        }
    }
    // First column (relative to n0) of the quad of columns at c when `cols` columns exist from n0 on.
    __device__ __forceinline__ static int shifted(int c, int cols) { return KC ? c : min(c, cols - RV); }
    // Whether unit i exists for this thread (whole wavefronts only).
    __device__ __forceinline__ bool has(int i) const { return !RAGGED || i + 1 < NU || t + i * NTH < UNITS; }
    __device__ __forceinline__ void unit(float (&x)[NU][4 * RV], int i, int k0) const {
        if (!has(i)) return;
        if constexpr (KC) {
            const f4u v = *reinterpret_cast<const f4u *>(at(base + k0, off[i]));
#pragma unroll
            for (int e = 0; e < 4; e++) x[i][e] = v[e];
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) wide(x[i], e, base + (int64_t)(k0 + e) * ld, off[i]);
        }
    }
    __device__ __forceinline__ void wide(float (&x)[4 * RV], int e, const float *p, unsigned o) const {
        if constexpr (RV == 4) {
            const f4u v = *reinterpret_cast<const f4u *>(at(p, o));
#pragma unroll
            for (int r = 0; r < 4; r++) x[4 * r + e] = v[r];
        } else {
            const f2u v = *reinterpret_cast<const f2u *>(at(p, o));
            x[e] = v[0];
            x[4 + e] = v[1];
        }
    }
    __device__ __forceinline__ void unit_tail(float (&x)[NU][4 * RV], int i, int k0, int kend) const {
        if (!has(i)) return;
        const int u = min(t + i * NTH, UNITS - 1), c = KC ? u & 7 : u / (BN / RV);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int k = k0 + 4 * c + e, kc = kclamp(k, kend);
            if constexpr (KC) {
                x[i][e] = *at(base + kc - 4 * c, off[i]);
            } else {
                wide(x[i], e, base + (int64_t)(kc - 4 * c) * ld, off[i]);
            }
            if (k >= kend)
#pragma unroll
                for (int r = 0; r < RV; r++) x[i][4 * r + e] = 0.0f;
        }
    }
    // Splits quad w of this thread and stores it.
    __device__ __forceinline__ void put(const float (&x)[NU][4 * RV], int w, char *buf) const {
        const int i = w / RV, r = w % RV;
        if (!has(i)) return;
        uint32_t h0, m0, l0, h1, m1, l1;
        split2(x[i][4 * r], x[i][4 * r + 1], h0, m0, l0);
        split2(x[i][4 * r + 2], x[i][4 * r + 3], h1, m1, l1);
        char *d = buf + (soff[i] ^ (r * 16));  // rows RV q + r: the XORed slot's low bits take r
        *reinterpret_cast<u32x2 *>(d) = u32x2{h0, h1};
        *reinterpret_cast<u32x2 *>(d + 1024) = u32x2{m0, m1};
        *reinterpret_cast<u32x2 *>(d + 2048) = u32x2{l0, l1};
    }
};

// ---------------------------------------------------------------------------------------------------------- epilogue
// Four consecutive columns of one row. e0 > 0 at a ragged right edge: the first e0 columns are another quad's; a quad
// that does not exist has e0 = 4 and reads a place that does.
struct OutQuad {
    floatx4 v;
    int row, col, e0;
};
__device__ __forceinline__ floatx4 ld4(const float *p) {
    const f4u v = *reinterpret_cast<const f4u *>(p);
    return floatx4{v[0], v[1], v[2], v[3]};
}
template <bool EDGE>
__device__ __forceinline__ void st4(float *p, floatx4 v, int e0) {
    if (!EDGE || e0 == 0) {
        *reinterpret_cast<f4u *>(p) = f4u{v[0], v[1], v[2], v[3]};
        return;
    }
#pragma unroll
    for (int e = 1; e < 4; e++)
        if (e >= e0) p[e] = v[e];
}

// NB quads through alpha, mask, bias, residual, ReLU or GELU terms and accumulation into C (and the MSE's unit gradient
// and squared differences), each step's loads issued together. REF: GELU by the reference's polynomials (long: one quad
// at a time), else the pair of stated error.
template <bool EDGE, bool REF, int NB>
__device__ __forceinline__ void finish(const Params &p, OutQuad (&q)[NB], float *C, const float *mask, double &mse_acc) {
    floatx4 t[NB] = {}, res[NB] = {}, tgt[NB] = {};
    auto gather_to = [&](floatx4(&d)[NB], const float *base, int64_t ld) {
#pragma unroll
        for (int b = 0; b < NB; b++) d[b] = ld4(base + (int64_t)q[b].row * ld + q[b].col);
    };
    auto gather = [&](const float *base, int64_t ld) { gather_to(t, base, ld); };
    // the residual's and the MSE target's loads first, so they land while the earlier terms are formed
    if (p.resid) gather_to(res, p.resid, p.ldr);
    if (p.mse_t) gather_to(tgt, p.mse_t, p.ldc);
    auto each = [&](auto f) {
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float v = q[b].v[e], u = t[b][e];
                f(v, u);
                q[b].v[e] = v;
                t[b][e] = u;
            }
    };
    const float alpha = p.alpha, dsq = p.mse_dsq;
    if (alpha != 1.0f) each([&](float &v, float &) { v = v * alpha; });
    if (mask) {
        gather(mask, p.n);
#pragma unroll
        for (int b = 0; b < NB; b++) q[b].v = q[b].v + t[b];
    }
    if (p.bias) {
        if (p.bias_per_row) {
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const float br = p.bias[q[b].row];
                q[b].v = q[b].v + floatx4{br, br, br, br};
            }
        } else {
            gather(p.bias, 0);
#pragma unroll
            for (int b = 0; b < NB; b++) q[b].v = q[b].v + t[b];
        }
    }
    if (p.resid) {
#pragma unroll
        for (int b = 0; b < NB; b++) q[b].v = q[b].v + res[b];
    }
    auto out2 = [&] {
#pragma unroll
        for (int b = 0; b < NB; b++) st4<EDGE>(p.out2 + (int64_t)q[b].row * p.ld2 + q[b].col, t[b], q[b].e0);
    };
    if (p.epi == EPI_RELU) {
        each([](float &v, float &) { v = v > 0.0f ? v : (v == v ? 0.0f : v); });
    } else if (p.epi == EPI_MUL_AUX) {
        gather(p.aux, p.ldaux);
        each([](float &v, float &u) { v = omd::canon(v * u); });
    } else if (p.epi == (REF ? EPI_GELU_GRAD : EPI_GELU_GRAD_F)) {
        gather(p.aux, p.ldaux);
        each([](float &v, float &u) { v = REF ? omd::gelu_grad(v, u) : omd::gelu_grad_fast(v, u); });
    } else if (p.epi == (REF ? EPI_GELU : EPI_GELU_F)) {
        each([](float &v, float &u) { u = REF ? omd::gelu(v) : omd::gelu_fast(v); });
        out2();
    } else if (p.epi == (REF ? EPI_GELU_SLOPE : EPI_GELU_SLOPE_F)) {
        each([](float &v, float &u) {
            float a, s;
            if constexpr (REF) omd::gelu_and_slope(v, a, s);
            else omd::gelu_and_slope_fast(v, a, s);
            v = a;
            u = s;
        });
        out2();
    }
    if (p.accumulate) {
        gather(C, p.ldc);
#pragma unroll
        for (int b = 0; b < NB; b++) q[b].v = t[b] + q[b].v;
    }
#pragma unroll
    for (int b = 0; b < NB; b++) st4<EDGE>(C + (int64_t)q[b].row * p.ldc + q[b].col, q[b].v, q[b].e0);
    if (p.mse_t) {  // d = stored value - target; the unit gradient 2 (d / n) as (d dsq) + (d dsq); sum of fl(d d)
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const floatx4 d = q[b].v - tgt[b], u = floatx4{dsq * d[0], dsq * d[1], dsq * d[2], dsq * d[3]};
            st4<EDGE>(p.mse_unit + (int64_t)q[b].row * p.ldc + q[b].col, u + u, q[b].e0);
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (!EDGE || e >= q[b].e0) mse_acc += (double)(d[e] * d[e]);
        }
    }
}

// ---------------------------------------------------------------------------------------------------------- the tile
// EXACT: whole tiles, whole 32-k steps, the same number for every k group. Else any shape with at least four columns.
template <int TN, int MG, int KG, bool TA, bool TB, bool EXACT>
__device__ __forceinline__ void tile(const Params &p, int tm, int tn, int zz) {
    constexpr bool BK_ = TB, EDGE = !EXACT;
    constexpr int BM = 32 * MG, BN = 32 * TN, NTG = 64 * MG;
    constexpr int BUF = BN * 192;  // one 32-step of B: three planes of BN x 32 bf16
    constexpr int LDC = BN + 4;                     // floats between the finished tile's rows in LDS
    constexpr int LOOP = 2 * KG * BUF, OUT = KG * BM * LDC * 4;
    constexpr int LDS = LOOP > OUT ? LOOP : OUT;
    __shared__ __attribute__((aligned(16))) char sh[LDS];

    const int z = zz / p.splits, split = zz % p.splits;
    const int outer = z / p.batch_div, inner = z % p.batch_div;
    const float *A = p.a + outer * p.sa_outer + inner * p.sa_inner;
    const float *B = p.b + outer * p.sb_outer + inner * p.sb_inner;
    const int m0 = tm * BM, n0 = tn * BN;
    const int kbeg = split * p.k_split, kend = min(p.k, kbeg + p.k_split);
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = wv / MG, mg = wv % MG, wm0 = mg * 32;
    const int full = (kend - kbeg) / 32, nit = (full + KG - 1) / KG;

    floatx16 acc[TN], low[TN];
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[j][e] = low[j][e] = 0.0f;

    // A wavefront wholly past the last row computes row m - 1, and stores nothing.
    const ALoad<!TA> la(A, p.lda, EDGE ? min(m0 + wm0, p.m - 1) : m0 + wm0, p.m, lane);
    using LB = BLoad<BN, NTG, BK_>;
    const LB lb(B, p.ldb, n0, p.n, threadIdx.x % NTG);
    char *buf = sh + kg * 2 * BUF;
    int roff[2][2];  // [block parity][half]
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int h = 0; h < 2; h++) roff[s][h] = (g * 32 + bswz(32 * s + l32, g, h)) * 16 + h * 3072;

    double cs = 0.0;
    const bool do_cs = TA && p.db && tn == 0;

    float ra[4][4], rb[LB::NU][4 * LB::RV];
    Frag fa[2];
    u32x4 fb[2][3];
    auto rd = [&](u32x4(&f)[3], const char *cur, int j, int h) {
#pragma unroll
        for (int q = 0; q < 3; q++) f[q] = *reinterpret_cast<const u32x4 *>(cur + j * 6144 + q * 1024 + roff[j & 1][h]);
    };
    auto mm = [&](const u32x4(&f)[3], const Frag &a, int j) { mma6(f, a.p, acc[j], low[j]); };
    // Quad w of A into its half's fragment; `have` false (a k group without this step) gives zeros.
    auto split_a = [&](float (&x)[4], int w, bool have) {
        if (EDGE && KG > 1) {
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = have ? x[e] : 0.0f;
        }
        fa[w >> 1].set4(w & 1, x);
        if (TA && do_cs && have)
#pragma unroll
            for (int e = 0; e < 4; e++) cs += (double)x[e];
    };
    // This group's step `it` starts at k = kat(it); loads past its last step repeat a step that exists.
    auto kat = [&](int it) { return kbeg + (it * KG + kg) * 32; };
    if (nit > 0) {
        auto kcl = [&](int it) { return EXACT ? kat(it < nit ? it : nit - 1) : min(kat(it), kbeg + 32 * (full - 1)); };
        auto have = [&](int it) { return EXACT ? it < nit : kat(it) < kbeg + 32 * full; };
#pragma unroll
        for (int i = 0; i < LB::NU; i++) lb.unit(rb, i, kcl(0));
#pragma unroll
        for (int w = 0; w < 4; w++) la.quad(ra[w], w, kcl(0));
#pragma unroll
        for (int w = 0; w < LB::QUADS; w++) {
            lb.put(rb, w, buf);
            if (w % LB::RV == LB::RV - 1) lb.unit(rb, w / LB::RV, kcl(1));
        }
#pragma unroll
        for (int w = 0; w < 2; w++) {
            split_a(ra[w], w, have(0));
            la.quad(ra[w], w, kcl(1));
        }
        __syncthreads();
        rd(fb[0], buf, 0, 0);
        // Step `it` in buffer it & 1 is 2 TN phases of six MFMAs, the first 16-k half over all column blocks, then the
        // second. Between the MFMAs of a phase goes a share of the coming work: the first half's phases split this
        // step's second half of A, the second half's phases the next step's first half, and all but the last put the
        // next step's B into the other buffer. A raw quad is reloaded as soon as it is split, a whole step before it
        // is wanted again. The barrier stands before the last phase, whose fragments are already in registers, so the
        // next step's first fragments load under it.
        constexpr int W = LB::QUADS, PH = 2 * TN;
        for (int it = 0; it < nit; it++) {
            const char *cur = buf + (it & 1) * BUF;
            char *nxt = buf + ((it & 1) ^ 1) * BUF;
            const int k1 = kcl(it + 1), k2 = kcl(it + 2);
#pragma unroll
            for (int ph = 0; ph < PH; ph++) {
                const int h = ph / TN, j = ph % TN;
                if (ph + 1 < PH) {
                    rd(fb[(ph + 1) & 1], cur, (ph + 1) % TN, (ph + 1) / TN);
                } else {
                    __syncthreads();
                    rd(fb[0], nxt, 0, 0);
                }
                mm(fb[ph & 1], fa[h], j);
#pragma unroll
                for (int w = 0; w < W; w++)
                    if (w * (PH - 1) / W == ph) {
                        lb.put(rb, w, nxt);
                        if (w % LB::RV == LB::RV - 1) lb.unit(rb, w / LB::RV, k2);
                    }
#pragma unroll
                for (int w = 0; w < 2; w++)
                    if (j == (w == 0 ? 0 : (TN + 1) / 2)) {
                        const int q = 2 * (h ^ 1) + w;
                        split_a(ra[q], q, have(h == 0 ? it : it + 1));
                        la.quad(ra[q], q, h == 0 ? k1 : k2);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
    }
    if (EDGE && kbeg + 32 * full < kend) {  // the last k % 32, by group 0
        const int k0 = kbeg + 32 * full;
        if (kg == 0) {
#pragma unroll
            for (int i = 0; i < LB::NU; i++) lb.unit_tail(rb, i, k0, kend);
#pragma unroll
            for (int w = 0; w < 4; w++) la.quad_tail(ra[w], w, k0, kend);
#pragma unroll
            for (int w = 0; w < LB::QUADS; w++) lb.put(rb, w, buf);
#pragma unroll
            for (int w = 0; w < 4; w++) split_a(ra[w], w, true);
        }
        __syncthreads();
        if (kg == 0) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    rd(fb[0], buf, j, h);
                    mm(fb[0], fa[h], j);
                }
        }
        __syncthreads();
    }

    unsigned big = 0;
#pragma unroll
    for (int j = 0; j < TN; j++) {
        finish_sums(acc[j], low[j]);
#pragma unroll
        for (int e = 0; e < 16; e++) note(acc[j][e], big);
    }
    if (beyond(big)) {
#pragma unroll
        for (int j = 0; j < TN; j++) {
            // column of the lane's LDS row, as the loads and the epilogue place it
            const int col = 32 * j + l32;
            const int cc = BK_ ? min(col, p.n - 1 - n0) : LB::shifted(col / LB::RV * LB::RV, p.n - n0) + col % LB::RV;
            const float *b = B + (BK_ ? (int64_t)(n0 + cc) * p.ldb : (int64_t)(n0 + cc));
            floatx16 t;
#pragma unroll
            for (int e = 0; e < 16; e++) t[e] = 0.0f;
#pragma unroll 1
            for (int it = 0; it <= nit; it++) {  // the group's steps, then (group 0) the tail
                const bool tail = it == nit;
                const int k0 = tail ? kbeg + 32 * full : kat(it);
                if (tail ? kg != 0 || k0 >= kend : k0 >= kbeg + 32 * full) continue;
#pragma unroll 1
                for (int w = 0; w < 4; w++) {
                    float xa[4];
                    la.quad_tail(xa, w, k0, kend);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int k = k0 + 8 * w + 4 * g + e, kc = kclamp(k, kend);
                        const float v = BK_ ? b[kc] : b[(int64_t)kc * p.ldb];
                        t = __builtin_amdgcn_mfma_f32_32x32x2f32(k < kend ? v : 0.0f, xa[e], t, 0, 0, 0);
                    }
                }
            }
            take_beyond(acc[j], t);
        }
    }

    if constexpr (TA) {
        if (do_cs) {  // uniform over the workgroup
            cs += __shfl_xor(cs, 32, 64);
            double *shd = reinterpret_cast<double *>(sh);
            if (KG > 1) {
                if (kg > 0 && g == 0) shd[(kg - 1) * BM + wm0 + l32] = cs;
                __syncthreads();
            }
            const int row = m0 + wm0 + l32;
            if (kg == 0 && g == 0 && (EXACT || row < p.m)) {
#pragma unroll
                for (int q = 1; q < KG; q++) cs += shd[(q - 1) * BM + wm0 + l32];
                if (p.splits > 1) {
                    p.colsum_ws[(int64_t)split * p.m + row] = cs;
                } else {
                    const float v = (float)cs;
                    p.db[row] = p.db_acc ? p.db[row] + v : v;
                }
            }
            if (KG > 1) __syncthreads();
        }
    }

    // Lane l holds, of column block j, row l32 and columns 8 q + 4 g .. + 3 (q = 0 .. 3). The tile goes through LDS, a
    // copy per k group, so that the epilogue's global accesses run along rows, BN / 4 lanes to a row; the copies are
    // added in group order as they are read.
    float *out = reinterpret_cast<float *>(sh);
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int c = 32 * j + 8 * q + 4 * g;
            float *d = out + (kg * BM + wm0 + l32) * LDC + c;
            const floatx4 v = {acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
            if constexpr (EDGE && !BK_) {
                // RV-wide loads that cross the right edge were moved back onto the last columns
#pragma unroll
                for (int e = 0; e < 4; e += LB::RV) {
                    const int back = c + e - LB::shifted(c + e, p.n - n0);
                    if (back == 0) {
#pragma unroll
                        for (int r = 0; r < LB::RV; r++) d[e + r] = v[e + r];
                    } else if (back < LB::RV) {
#pragma unroll
                        for (int r = 0; r < LB::RV; r++)
                            if (r >= back) d[e + r - back] = v[e + r];
                    }
                }
            } else {
                *reinterpret_cast<floatx4 *>(d) = v;
            }
        }
    __syncthreads();

    float *C = p.c + outer * p.sc_outer + inner * p.sc_inner;
    const float *mask = p.mask ? p.mask + outer * p.mask_outer_stride : nullptr;
    double mse_acc = 0.0;
    constexpr int CQ = BN / 4, NTHR = 64 * MG * KG, NQ = BM * CQ / NTHR, NB = NQ % 4 == 0 ? 4 : NQ % 3 == 0 ? 3 : 2;
    static_assert(BM * CQ % NTHR == 0 && NQ % NB == 0, "the epilogue's quads split evenly");
    // Quads u0, u0 + 1, .. of this thread out of LDS.
    auto fill = [&](auto &q, int u0) {
        int b = 0;
        for (OutQuad &o : q) {
            const int u = threadIdx.x + (u0 + b++) * NTHR, r = u / CQ;
            int c = 4 * (u % CQ), e0 = 0;
            if (EDGE && n0 + c + 4 > p.n) {  // the last, partial quad: read and stored as the last four columns
                e0 = min(n0 + c + 4 - p.n, 4);
                c = p.n - 4 - n0;
            }
            const float *src = out + r * LDC + c;
            floatx4 v = {0.f, 0.f, 0.f, 0.f};
            if (!EDGE || e0 == 0) {
                v = *reinterpret_cast<const floatx4 *>(src);
#pragma unroll
                for (int s = 1; s < KG; s++) v = v + *reinterpret_cast<const floatx4 *>(src + s * BM * LDC);
            } else {
#pragma unroll
                for (int e = 1; e < 4; e++)
                    if (e >= e0) {
                        v[e] = src[e];
#pragma unroll
                        for (int s = 1; s < KG; s++) v[e] = v[e] + src[s * BM * LDC + e];
                    }
            }
            if (EDGE && m0 + r >= p.m) e0 = 4;
            o = OutQuad{v, EDGE ? min(m0 + r, p.m - 1) : m0 + r, n0 + c, e0};
        }
    };
    if (p.splits == 1 && (p.epi == EPI_GELU || p.epi == EPI_GELU_GRAD || p.epi == EPI_GELU_SLOPE)) {
#pragma unroll 1
        for (int u0 = 0; u0 < NQ; u0++) {
            OutQuad q[1];
            fill(q, u0);
            finish<EDGE, true>(p, q, C, mask, mse_acc);
        }
    } else {
#pragma unroll 1
        for (int u0 = 0; u0 < NQ; u0 += NB) {
            OutQuad q[NB];
            fill(q, u0);
            if (p.splits > 1) {
#pragma unroll
                for (int b = 0; b < NB; b++)
                    st4<EDGE>(p.ws + ((int64_t)split * p.m + q[b].row) * p.n + q[b].col, q[b].v, q[b].e0);
            } else {
                finish<EDGE, false>(p, q, C, mask, mse_acc);
            }
        }
    }
    if (p.mse_t) {  // uniform over the launch; every lane of the wavefront is here
        mse_acc = omd::wave_sum(mse_acc);
        if (lane == 0) p.mse_part[MG * KG * blockIdx.x + wv] = mse_acc;
    }
}

template <int TN, int MG, int KG, bool TA, bool TB, bool EXACT>
__global__ void __launch_bounds__(64 * MG * KG, 2) k_gemm_s(Params p) {
    OM_LDS_POISON();
    constexpr int BM = 32 * MG, BN = 32 * TN;
    int tm, tn, zz;
    tile_coords(p, EXACT ? p.n / BN : (p.n + BN - 1) / BN, EXACT ? p.m / BM : (p.m + BM - 1) / BM, tm, tn, zz);
    tile<TN, MG, KG, TA, TB, EXACT>(p, tm, tn, zz);
}

// Weight gradients (TN products) of a group in one launch: workgroup ranges map to products, and inside a range to
// split, tile row and tile column, or (g.band > 0, unsplit groups) to bands of g.band tile rows walked column by
// column, so the workgroups one XCD runs together share operand panels.
template <int TN, int MG, int KG, bool EXACT>
__global__ void __launch_bounds__(64 * MG * KG, 2) k_gemm_s_tn_group(GroupParams g) {
    OM_LDS_POISON();
    constexpr int BM = 32 * MG, BN = 32 * TN;
    const int total = g.start[g.count];
    int lin = blockIdx.x;
    if ((total & 7) == 0) lin = (lin & 7) * (total >> 3) + (lin >> 3);
    int i = 0;
#pragma unroll
    for (int j = 1; j < kMaxGroup; j++)
        if (j < g.count && lin >= g.start[j]) i = j;
    const Params &p = g.p[i];
    const int t = lin - g.start[i];
    const int tiles_n = (p.n + BN - 1) / BN, tiles_m = (p.m + BM - 1) / BM;
    int tm, tn;
    const int zz = t / (tiles_n * tiles_m), q = t % (tiles_n * tiles_m);
    if (g.band > 0) {
        const int per = g.band * tiles_n, b = q / per, rows = min(g.band, tiles_m - b * g.band), r = q - b * per;
        tn = r / rows;
        tm = b * g.band + r % rows;
    } else {
        tn = q % tiles_n;
        tm = q / tiles_n;
    }
    tile<TN, MG, KG, true, false, EXACT>(p, tm, tn, zz);
}

}  // namespace gs

// The tile shapes that are built, in the order of SConfig::id (om_gemm.hip's chooser weighs them).
//   256 x 128, 256 x 96: eight wavefronts, B split once for 256 rows
//   128 x 128, 128 x 96, 128 x 64: four wavefronts, two workgroups to a CU
//   64 x 96, 64 x 64 with four k groups: products with few tiles
//   64 x 64 with two k groups: several to a CU
#define OMG_S_CONFIGS(X) X(0, 4, 8, 1) X(1, 3, 8, 1) X(2, 4, 4, 1) X(3, 3, 4, 1) X(4, 2, 4, 1) X(5, 3, 2, 4) X(6, 2, 2, 4) X(7, 2, 2, 2)
void launch_s_nt(int cfg, bool exact, const Params &p, unsigned grid, hipStream_t st);
void launch_s_nn(int cfg, bool exact, const Params &p, unsigned grid, hipStream_t st);
void launch_s_tn(int cfg, bool exact, const Params &p, unsigned grid, hipStream_t st);
void launch_s_tn_group(int cfg, bool exact, const GroupParams &g, unsigned grid, hipStream_t st);
}  // namespace omg
