// Projections of the one-token step (decode: one row per sequence, M <= 64) at fp32 precision on
// the gfx950 fp16 matrix cores, with the step's neighbouring element-wise work in the epilogue:
//
//   v[m, n] = s[m] * sum_k X[m, k] W[n, k]          W (N, K)
//   s[m]    = 1 / sqrt(sum_j ssq[m, j] * inv_div + eps)    (ssq given; else s = 1)
//
//   EPI_STORE  Y[m, n] = v + beta * Y[m, n]
//   EPI_CONV   columns c0 .. c0+C-1 go through the depthwise causal-conv update + SiLU (the
//              Mamba conv1d on one new token, state (M, C, Kc-1) shifted in place) into Yc;
//              the other columns are stored to Y
//   EPI_RESID  Y[m, n] += v (the residual add); then, when g2 is given, the next RMSNorm's
//              operand xg[m, n] = Y[m, n] * g2[n] (in fragment order, below) and the row's
//              partial sum of squares over the tile's 16 columns, ssq_out[m, n / 16]
//   EPI_HEAD   Y[m, n] = v (the LM head's logits) and, per row and workgroup, the largest logit
//              with the lowest index among equal maxima (NaN never wins) as a (value, index)
//              pair; a row's pairs are merged by head_argmax_kernel (head.hip)
//   Yf         EPI_CONV: the conv outputs also written in fragment order, the operand of the
//              step's next projection (the Mamba-1 step's x_proj as its own launch)
//   xpart      EPI_CONV: that next projection summed over each conv tile's 16 channels (one
//              partial row per tile and row), so that no launch of its own is needed: the
//              Mamba-1 step's state update adds the partials
//
// The RMSNorms of the step are carried this way: the producer of a row writes x * g and
// partial sums of x^2 per 16 columns, and the consumer's epilogue applies 1 / rms(x) as the
// row scale s[m]; the gated norm's y * silu(z) * g and its partial sums come from the state
// update (ssd.hip). The partial sums are added in a fixed order, identical in every
// workgroup, so s[m] is the same wherever it is formed and every result is deterministic.
//
// Split. As in gemm_h3.hip: a row of an operand is scaled by a power of two so that its largest
// magnitude lies in [2^14, 2^15) and each element is held as fp16 hi + lo; a product is three
// v_mfma_f32_16x16x32_f16 (lo hi, hi lo, hi hi) into fp32 sums, scaled back exactly. W is packed
// once per load (launch_pack_step, gemm_h3.hip: a scale per row); X arrives in fp32 and each wave
// scales and splits its own k range of it in registers, while its W is still on the way from HBM.
// Range: as there, every output is held against what the split may have lost of elements far
// below their row's largest (W: the packing's rho; X: 2^-25 of each scaled element). Its measure is
// the waves' partial sums taken by magnitude, which are small together only if the operands really
// are that far apart. Such an output, and one that is not finite (elements that are inf or NaN
// become NaN), is formed again from the fp32 operands.
//
// Operand order. X is in fragment order (frag_off in glue.hpp): the 1 KB of a (16-row tile,
// 16-wide k-block) is contiguous, lane-major, lane 16 q + i holding row i, k = 4 q .. + 3, so one
// b128 load per lane brings 8 full lines. Two k-blocks make one MFMA operand of 32 k: elements
// 0 .. 3 of lane (q, i) are k = 4 q .. + 3 of the first block, elements 4 .. 7 those of the second;
// W's packed blocks (hi and lo, 1 KB each) use the same order of k.
//
// Decomposition. What bounds a step projection is bringing W (18 MB for a 4384 x 1024 in_proj)
// from HBM once with everything in flight at once: 256 CUs at 6 TB/s and 2 us of latency is
// 48 KB a CU. A workgroup of eight waves owns 16 MT rows x 16 columns and all of K; wave w takes
// an eighth of K, issues all its X and W loads up front, keeps the split X in registers (128 at
// most) and, when there are more column tiles than CUs, walks tiles of
// stride gridDim with the next tile's W in flight. The waves' partial tiles meet in LDS, added in
// wave order. MT covers all rows when that still gives every CU a workgroup (W then crosses the
// L2 once, where 16 x 16 tiles had each W line requested by four row tiles); otherwise the row
// tiles of a column tile are workgroups of their own, on one XCD (ids 8 apart), sharing W in L2.
//
// Measured (MI355X, weights cold, fp32 MFMA tiles of 16 x 16 -> this): 64 x 4384 x 1024 with the
// conv update 14.8 -> 13.2 us, 64 x 3072 x 768 10.4 -> 9.0, the head 64 x 32000 x 1024 49 -> 32.8;
// the narrow ones lose a little, 64 x 1024 x 2048 with the residual 7.5 -> 7.9 and 64 x 768 x 1536
// 6.5 -> 7.0 (every workgroup splits its rows of X anew). The coverage test adds 0.2 to 0.3 us to
// each (decode of 64 sequences, 8 layers: 324 -> 332).
#include <algorithm>

#include "common.hpp"
#include "glue.hpp"

namespace ssm {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

constexpr int kNW = 8;                  // waves per workgroup
constexpr int kNT = 64 * kNW;
constexpr unsigned kOOR = 0x80000000u;  // a buffer offset past every descriptor's range
// EPI_CONV with xpart as a kernel of its own
constexpr int EPI_CONVX = 4;

__device__ __forceinline__ float sum16(float v) {
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 16);
    return v;
}

typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ halfx8 as_h8(u32x4 v) { return __builtin_bit_cast(halfx8, v); }

// Two elements times 2^sh as fp16 hi and lo (round to nearest), packed.
__device__ __forceinline__ void split2(float a, float b, int sh, unsigned& hi, unsigned& lo) {
    const float s0 = __builtin_ldexpf(a, sh), s1 = __builtin_ldexpf(b, sh);
    const halfx2 h = {(_Float16)s0, (_Float16)s1};
    const halfx2 l = {(_Float16)(s0 - (float)h[0]), (_Float16)(s1 - (float)h[1])};
    hi = __builtin_bit_cast(unsigned, h);
    lo = __builtin_bit_cast(unsigned, l);
}

// sum_k X[m, k] W[n, k] from the fp32 operands (X in fragment order) for the lanes with `again`
// set, whose split product will not do: the 16 lanes of a row m share one output at a time, each
// its quads of k in order, then a tree. (All lanes of the wave call it; W rows start anywhere.
// Inline and not unrolled: it takes few registers, where a call had the multi-tile kernels spill.)
__device__ __forceinline__ float step_exact(const float* X, const float* W, int m, int n, int K,
                                         bool again) {
    const int lane = threadIdx.x & 63, l16 = lane & 15;
    unsigned todo = (unsigned)(__ballot(again) >> (lane & 48)) & 0xffffu;
    float out = 0.f;
    while (__any(todo != 0)) {
        const int src = todo ? __builtin_ctz(todo) : 0;
        const float* w = W + (long)__shfl(n, src, 16) * K;
        float s = 0.f;
        if (todo) {
#pragma unroll 1
            for (int k = 4 * l16; k < K; k += 64) {
                const float4 x = *reinterpret_cast<const float4*>(X + frag_off(m, k, K >> 4));
                s = fmaf(x.x, w[k], s);
                s = fmaf(x.y, w[k + 1], s);
                s = fmaf(x.z, w[k + 2], s);
                s = fmaf(x.w, w[k + 3], s);
            }
        }
        s = sum16(s);
        if (todo && l16 == src) out = s;
        todo &= todo - 1;
    }
    return out;
}

// MT row tiles, NC column tiles at a time, KW 32-wide k-blocks per wave and pass; MULTI: a
// workgroup walks several groups of column tiles (K then takes one pass).
template <int MT, int NC, int KW, bool MULTI, int EPI>
__global__ __launch_bounds__(kNT, 2) void stepproj_kernel(StepProj a) {
    constexpr bool CONV = EPI == EPI_CONV || EPI == EPI_CONVX;
    constexpr int ROWS = 16 * MT;
    // epilogue elements of a thread: rows tid / 16 + 32 s, s < RS, of each column tile
    constexpr int RS = (ROWS + 31) / 32, EPT = RS * NC;
    __shared__ float red[MULTI ? 2 : 1][kNW][ROWS][16 * NC + 1];
    __shared__ float sc[64];
    __shared__ float scale[kNW][ROWS];   // the groups' scales per wave and row, summed
    __shared__ float us[EPI == EPI_CONVX ? ROWS : 1][16 * NC + 1];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    // row group tg and first column group: the row groups of a column group are 8 ids apart (one
    // XCD); MULTI workgroups go on to the column groups gstep further
    const int b = blockIdx.x, r8 = b >> 3;
    const int tg = r8 % a.rg;
    const int gstep = (int)gridDim.x / a.rg;
    int tn = NC * ((r8 / a.rg) * 8 + (b & 7));   // first column tile
    if (tn >= a.nt) return;   // (the id space is padded to whole groups of 8 column groups)
    const int slot = tn / NC;   // EPI_HEAD: this workgroup's pair
    const int m0 = tg * ROWS;
    const int KB = a.K >> 4, KB2 = (KB + 1) >> 1;   // 16-wide blocks of X, 32-wide of W

    // ---- operand loads: a wave's k-blocks go in groups of four, each scaled and summed by itself,
    // and the groups' sums are added in order: the same in every workgroup (equal rows of W give
    // equal results) and whether a pass takes two groups or, with more row tiles in the registers,
    // one (a row's result does not depend on the rows beside it). Past 1024 input features two
    // groups are adjacent. (One k-block a wave for up to 256 features, so that the coverage test
    // below has several partial sums to go by, saved the 128-wide preset 1.4 us of 72 a step, but its
    // run-time stride cost every other shape: in_proj of 28 rows 9.5 -> 10.0 us.) Every workgroup reads the same X; those on one XCD start at row
    // tiles of their own.
    constexpr int KG = 4, NG = KW / KG;
    static_assert(KW == KG || KW == 2 * KG, "one or two groups");
    const bool halves = KW == KG && a.npass > 1;   // (uniform) a pass takes one of two adjacent groups
    auto block = [&](int p, int u) __attribute__((always_inline)) {
        if (KW > KG) return KW * (kNW * p + w) + u;
        if (halves) return 2 * KG * (kNW * (p >> 1) + w) + KG * (p & 1) + u;
        return KW * w + u;
    };
    const int irot = (r8 / a.rg) & (MT - 1);
    const auto ra = rsrc(a.X, (unsigned)(a.mt * KB) * 1024u);
    auto load_x = [&](float4 (&x)[MT][KW][2], int p) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int u = 0; u < KW; ++u)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int k16 = 2 * block(p, u) + h;
                    const int tm = tg * MT + ((i + irot) & (MT - 1));
                    x[i][u][h] = bload16<float4>(
                        ra, k16 < KB && tm < a.mt ? (unsigned)(tm * KB + k16) * 1024u + 16u * lane
                                                  : kOOR);
                }
    };
    auto load_w = [&](halfx8 (&wv)[NC][KW][2], int t0, int p) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const int t = t0 + j;
            const auto rw = rsrc((const char*)a.W + (long)t * KB2 * 2048,
                                 t < a.nt ? (unsigned)KB2 * 2048u : 0u);
#pragma unroll
            for (int u = 0; u < KW; ++u) {
                const int kb = block(p, u);
                const unsigned o = kb < KB2 ? (unsigned)kb * 2048u + 16u * lane : kOOR;
#pragma unroll
                for (int h = 0; h < 2; ++h) wv[j][u][h] = ssm::bload16_nt<halfx8>(rw, o + 1024u * h);
            }
        }
    };
    // the split operands, by the row's power of two over the group; ex[g][i] undoes the scale of the
    // accumulator's rows 4 q + r of tile i
    u32x4 xh[MT][KW], xl[MT][KW];   // eight fp16 values each
    int ex[NG][MT][4];
    float scl[MT];                  // of row l16 of tile i: the groups' scales, summed
#pragma unroll
    for (int i = 0; i < MT; ++i) scl[i] = 0.f;
    auto split = [&](const float4 (&x)[MT][KW][2]) __attribute__((always_inline)) {
        // (tile by tile: the first is split while the next one's loads arrive)
#pragma unroll
        for (int gi = 0; gi < NG * MT; ++gi) {
            const int g = gi / MT, i = gi % MT;
            unsigned mx = 0;
#pragma unroll
            for (int u = KG * g; u < KG * (g + 1); ++u)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const float4 v = x[i][u][h];
                    const unsigned m1 = max(__float_as_uint(v.x) & 0x7fffffffu, __float_as_uint(v.y) & 0x7fffffffu);
                    const unsigned m2 = max(__float_as_uint(v.z) & 0x7fffffffu, __float_as_uint(v.w) & 0x7fffffffu);
                    mx = max(mx, max(m1, m2));
                }
            mx = max(mx, (unsigned)__shfl_xor((int)mx, 16));
            mx = max(mx, (unsigned)__shfl_xor((int)mx, 32));
            const int sh = mx ? 141 - min((int)(mx >> 23), 254) : 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) ex[g][i][r] = -__shfl(sh, 4 * q + r);
            scl[i] += mx ? __builtin_ldexpf(1.f, -sh) : 0.f;
            // (an inf gives hi = inf, lo = NaN, and so NaN in every product of its row)
#pragma unroll
            for (int u = KG * g; u < KG * (g + 1); ++u)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const float4 v = x[i][u][h];
                    unsigned h0, l0, h1, l1;
                    split2(v.x, v.y, sh, h0, l0);
                    split2(v.z, v.w, sh, h1, l1);
                    xh[i][u][2 * h] = h0; xh[i][u][2 * h + 1] = h1;
                    xl[i][u][2 * h] = l0; xl[i][u][2 * h + 1] = l1;
                }
        }
    };
    floatx4 out[NC][MT];
    auto multiply = [&](const halfx8 (&wv)[NC][KW][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            floatx4 acc[NC][MT];
#pragma unroll
            for (int j = 0; j < NC; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
            auto mm = [&](int j, int i, u32x4 x, halfx8 y) __attribute__((always_inline)) {
                acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_h8(x), y, acc[j][i], 0, 0, 0);
            };
#pragma unroll
            for (int u = KG * g; u < KG * (g + 1); ++u) {
#pragma unroll
                for (int j = 0; j < NC; ++j)
#pragma unroll
                    for (int i = 0; i < MT; ++i) mm(j, i, xl[i][u], wv[j][u][0]);
#pragma unroll
                for (int j = 0; j < NC; ++j)
#pragma unroll
                    for (int i = 0; i < MT; ++i) mm(j, i, xh[i][u], wv[j][u][1]);
#pragma unroll
                for (int j = 0; j < NC; ++j)
#pragma unroll
                    for (int i = 0; i < MT; ++i) mm(j, i, xh[i][u], wv[j][u][0]);
            }
#pragma unroll
            for (int j = 0; j < NC; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float v = acc[j][i][r];
                        out[j][i][r] += __builtin_ldexpf(v, ex[g][i][r]);
                    }
        }
    };

    float4 xr[MT][KW][2];
    halfx8 w0[NC][KW][2];
    load_x(xr, 0);
    load_w(w0, tn, 0);

    // ---- row scales: eight threads per row, each every eighth partial sum in order
    if (a.ssq) {
        const int srow = tid >> 3, m = m0 + srow;
        const auto rs = rsrc(a.ssq, (unsigned)(a.M * a.nssq) * 4u);
        float t = 0.f;
        if (srow < ROWS) {
            float sp[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int j = 8 * u + (tid & 7);
                sp[u] = bload4(rs, j < a.nssq && m < a.M ? (unsigned)(m * a.nssq + j) * 4u : kOOR);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) t += sp[u];
            for (int j = 64 + (tid & 7); j < a.nssq; j += 8)
                t += bload4(rs, m < a.M ? (unsigned)(m * a.nssq + j) * 4u : kOOR);
        }
        t += __shfl_xor(t, 1);
        t += __shfl_xor(t, 2);
        t += __shfl_xor(t, 4);
        if ((tid & 7) == 0 && srow < ROWS) sc[srow] = 1.f / sqrtf(t * a.inv_div + a.eps);
    } else if (tid < ROWS) {
        sc[tid] = 1.f;
    }

    // greedy pick so far of this thread's rows (EPI_HEAD; columns ascend from tile to tile)
    float best[RS];
    int bidx[RS];
#pragma unroll
    for (int s = 0; s < RS; ++s) { best[s] = -INFINITY; bidx[s] = a.N; }

    // descriptors of the epilogue's inputs (empty where absent: their loads give zeros)
    const auto rwe = rsrc(a.we, (unsigned)a.nt * 64u);
    const auto rcw = rsrc(a.cw, CONV ? (unsigned)(a.C * a.Kc) * 4u : 0u);
    const auto rcb = rsrc(a.cb, CONV && a.cb ? (unsigned)a.C * 4u : 0u);
    const auto rst = rsrc(a.cst, CONV ? (unsigned)(a.M * a.C * (a.Kc - 1)) * 4u : 0u);
    const auto rg2 = rsrc(a.g2, EPI == EPI_RESID && a.g2 ? (unsigned)a.N * 4u : 0u);
    const auto ryy = rsrc(a.Y, EPI == EPI_RESID ? (unsigned)((long)(a.M - 1) * a.ldy + a.N) * 4u : 0u);

    // 2^37 of the rows' scales over all waves, summed when the first tile's waves have met
    static_assert(32 * KG == 128, "the factor 2^-18 of the coverage test");
    float need[RS];
    bool first = true;
    // One column tile: W of its first pass is in wc; the next tile's goes into wnx.
    constexpr int kConvPre = 4;
    constexpr int kXpBlk = kXpartMaxRN / 16 / kNW;   // x_proj column blocks per wave
    auto tile = [&](halfx8 (&wc)[NC][KW][2], halfx8 (&wnx)[NC][KW][2], int buf) __attribute__((always_inline)) {
        // The epilogue's inputs, loaded ahead of the product (they do not depend on it): column
        // en[j] of column tile j, rows as above.
        const int ej = tid & 15;
        int en[NC];
        unsigned wex[NC];   // exponent and loss (rho) of the column's W row
        bool col_ok[NC], in_conv[NC], pre[NC];
        float csv[EPT][kConvPre - 1], cwv[NC][kConvPre], cbv[NC], rsv[EPT], g2v[NC];
        // (through range-checked descriptors: a guarded load would sit behind a branch, and the
        // waits around those branches held the product back: in_proj 21.4 -> 14.7 us)
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            en[j] = 16 * (tn + j) + ej;
            col_ok[j] = en[j] < a.N;
            const int c = en[j] - a.c0;
            in_conv[j] = CONV && col_ok[j] && c >= 0 && c < a.C;
            pre[j] = in_conv[j] && a.Kc <= kConvPre;
            wex[j] = __float_as_uint(bload4(rwe, col_ok[j] ? 4u * en[j] : kOOR));
            if constexpr (CONV) {
                const int Kc1 = a.Kc - 1;
#pragma unroll
                for (int k = 0; k < kConvPre; ++k)
                    cwv[j][k] = bload4(rcw, pre[j] && k < a.Kc ? (unsigned)(c * a.Kc + k) * 4u : kOOR);
                cbv[j] = bload4(rcb, pre[j] ? (unsigned)c * 4u : kOOR);
#pragma unroll
                for (int s = 0; s < RS; ++s) {
                    const int ei = (tid >> 4) + 32 * s, em = m0 + ei;
#pragma unroll
                    for (int k = 0; k < kConvPre - 1; ++k)
                        csv[j * RS + s][k] = bload4(rst, pre[j] && k < Kc1 && ei < ROWS && em < a.M
                                                             ? (unsigned)((em * a.C + c) * Kc1 + k) * 4u
                                                             : kOOR);
                }
            }
            if constexpr (EPI == EPI_RESID) {
                g2v[j] = bload4(rg2, col_ok[j] ? 4u * en[j] : kOOR);
#pragma unroll
                for (int s = 0; s < RS; ++s) {
                    const int ei = (tid >> 4) + 32 * s, em = m0 + ei;
                    rsv[j * RS + s] = bload4(ryy, col_ok[j] && ei < ROWS && em < a.M
                                                      ? (unsigned)((long)em * a.ldy + en[j]) * 4u
                                                      : kOOR);
                }
            }
        }
        // (c0 and C are multiples of 16 with xpart: a column tile is wholly conv or not at all)
        bool xp_tile[NC];
        float wxb[NC][kXpBlk][4];
        if constexpr (EPI == EPI_CONVX) {
            const auto rwx = rsrc(a.wxt, (unsigned)(a.C * a.RN) * 4u);
            // B fragments of the next projection: lane (j, k) of k-step s holds
            // wxt[channel 4 s + k][16 block + j], block w of the wave
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                const int n0 = 16 * (tn + j);
                xp_tile[j] = n0 >= a.c0 && n0 < a.c0 + a.C;
#pragma unroll
                for (int t = 0; t < kXpBlk; ++t)
#pragma unroll
                    for (int s4 = 0; s4 < 4; ++s4) {
                        const int col = 16 * (w + kNW * t) + l16;
                        wxb[j][t][s4] = bload4(rwx, xp_tile[j] && col < a.RN
                                                        ? (unsigned)((n0 - a.c0 + 4 * s4 + q) * a.RN + col) * 4u
                                                        : kOOR);
                    }
            }
        }
#pragma unroll
        for (int j = 0; j < NC; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) out[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
        if constexpr (MULTI) {
            load_w(wnx, tn + NC * gstep, 0);   // past the last tile: an empty range
            multiply(wc);
        } else {
            split(xr);
            multiply(wc);
            for (int p = 1; p < a.npass; ++p) {
                load_x(xr, p);
                load_w(wc, tn, p);
                split(xr);
                multiply(wc);
            }
        }
#pragma unroll
        for (int j = 0; j < NC; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    red[buf][w][16 * ((i + irot) & (MT - 1)) + 4 * q + r][16 * j + l16] = out[j][i][r];
        if (!MULTI || first) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
                if (q == 0) scale[w][16 * ((i + irot) & (MT - 1)) + l16] = scl[i];
        }
        __syncthreads();
        if (!MULTI || first) {
#pragma unroll
            for (int s = 0; s < RS; ++s) {
                const int ei = min((tid >> 4) + 32 * s, ROWS - 1);
                float t = scale[0][ei];
#pragma unroll
                for (int k = 1; k < kNW; ++k) t += scale[k][ei];
                need[s] = t * 0x1p37f;
            }
            first = false;
        }

        float uo[EPT];
#pragma unroll
        for (int e = 0; e < EPT; ++e) {
            const int j = e / RS;
            const int ei = (tid >> 4) + 32 * (e % RS), em = m0 + ei, n = en[j], c = n - a.c0;
            uo[e] = 0.f;
            if (ei >= ROWS) continue;
            float v = red[buf][0][ei][16 * j + ej], mag = fabsf(v);
#pragma unroll
            for (int k = 1; k < kNW; ++k) {
                const float t = red[buf][k][ei][16 * j + ej];
                v += t;
                mag += fabsf(t);
            }
            const bool ok = em < a.M && col_ok[j];
            // The split loses at most 2^15 scale (2^-25 (32 KG) + rho) of an output, which has to
            // be within 2^-22 of its partial sums' magnitudes.
            const bool covered = mag >= need[e % RS] * (0x1p-18f + __uint_as_float(wex[j] & 0xffff0000u));
            v = __builtin_ldexpf(v, (int)(short)wex[j]);
            const bool again = ok && !(covered && __builtin_isfinite(v));
            if (__builtin_expect(__any(again), 0)) {
                const float t = step_exact(a.X, a.Wf, em, n, a.K, again);
                v = again ? t : v;
            }
            v *= sc[ei];
            if constexpr (EPI == EPI_STORE) {
                if (ok) {
                    float* y = a.Y + (long)em * a.ldy + n;
                    *y = a.beta != 0.f ? v + a.beta * *y : v;
                }
            } else if constexpr (EPI == EPI_HEAD) {
                if (ok) a.Y[(long)em * a.ldy + n] = v;
                // (a row's columns ascend with j and from group to group)
                const int s = e % RS;
                if (col_ok[j] && (v > best[s] || (bidx[s] == a.N && v == best[s]))) { best[s] = v; bidx[s] = n; }
            } else if constexpr (CONV) {
                if (ok && !in_conv[j]) a.Y[(long)em * a.ldy + n] = v;
                float u = 0.f;   // the conv output; 0 on padding rows
                const int Kc = a.Kc;
                if (ok && pre[j]) {
                    // same arithmetic order as the conv update kernel (conv1d.hip), on the
                    // prefetched inputs
                    float* st = a.cst + ((long)em * a.C + c) * (Kc - 1);
                    float acc = cbv[j];
#pragma unroll
                    for (int k = 0; k < kConvPre - 1; ++k)
                        if (k < Kc - 1) acc = fmaf(cwv[j][k], csv[e][k], acc);
                    float wl = cwv[j][0];
#pragma unroll
                    for (int k = 1; k < kConvPre; ++k)
                        if (k == Kc - 1) wl = cwv[j][k];
                    acc = fmaf(wl, v, acc);
#pragma unroll
                    for (int k = 1; k < kConvPre - 1; ++k)   // shift the cached inputs down
                        if (k < Kc - 1) st[k - 1] = csv[e][k];
                    if (Kc > 1) st[Kc - 2] = v;
                    u = silu_fast(acc);
                    a.Yc[(long)em * a.ldyc + c] = u;
                } else if (ok && in_conv[j]) {
                    const float* wcv = a.cw + (long)c * Kc;
                    float* st = a.cst + ((long)em * a.C + c) * (Kc - 1);
                    float acc = a.cb ? a.cb[c] : 0.f;
                    for (int k = 0; k < Kc - 1; ++k) {   // taps on the cached inputs, shifting them
                        const float sv = st[k];
                        acc = fmaf(wcv[k], sv, acc);
                        if (k > 0) st[k - 1] = sv;
                    }
                    acc = fmaf(wcv[Kc - 1], v, acc);
                    if (Kc > 1) st[Kc - 2] = v;
                    u = silu_fast(acc);
                    a.Yc[(long)em * a.ldyc + c] = u;
                }
                uo[e] = u;
                // padding rows of the fragment-order copy get zeros for the next projection
                if (a.Yf && in_conv[j] && em < 16 * a.mt) a.Yf[frag_off(em, c, a.C >> 4)] = u;
            } else {   // EPI_RESID
                float o = 0.f;
                if (ok) {
                    o = rsv[e] + v;
                    a.Y[(long)em * a.ldy + n] = o;
                }
                if (a.g2) {
                    // rows past M (up to the tile's 16) get zeros: the next projection reads
                    // whole tiles
                    if (col_ok[j] && em < 16 * a.mt) a.xg[frag_off(em, n, a.nt)] = ok ? o * g2v[j] : 0.f;
                    const float t = sum16(o * o);
                    if (ej == 0 && em < a.M && col_ok[j]) a.ssq_out[(long)em * a.nt + tn + j] = t;
                }
            }
        }
        if constexpr (EPI == EPI_CONVX) {
#pragma unroll
            for (int e = 0; e < EPT; ++e)
                if ((tid >> 4) + 32 * (e % RS) < ROWS)
                    us[(tid >> 4) + 32 * (e % RS)][16 * (e / RS) + ej] = uo[e];
            __syncthreads();
            // D[i][j] = sum_s sum_k u[i][4s + k] wxt[4s + k][j] on the fp32 matrix cores;
            // lane (j, q) holds rows 4q .. 4q + 3
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                if (!xp_tile[j]) continue;   // (uniform over the workgroup)
                const int ct = tn + j - (a.c0 >> 4);
#pragma unroll
                for (int t = 0; t < kXpBlk; ++t) {
                    const int blk = w + kNW * t, col = 16 * blk + l16;
                    if (16 * blk >= a.RN) break;   // wave-uniform
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        if (tg * MT + i >= a.mt) break;
                        floatx4 xa = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int s4 = 0; s4 < 4; ++s4)
                            xa = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                us[16 * i + l16][16 * j + 4 * s4 + q], wxb[j][t][s4], xa, 0, 0, 0);
                        if (col < a.RN) {
                            float* dst = a.xpart + ((long)ct * 16 * a.mt + m0 + 16 * i + 4 * q) * a.RN + col;
#pragma unroll
                            for (int r = 0; r < 4; ++r) dst[(long)r * a.RN] = xa[r];
                        }
                    }
                }
            }
            if constexpr (MULTI) __syncthreads();   // us is written again by the next group
        }
    };
    if constexpr (MULTI) {
        // tiles in pairs, so that each of the two W buffers is named statically. A wave may run
        // one barrier ahead of another: red is double-buffered.
        halfx8 w1[NC][KW][2];
        split(xr);
        for (;;) {
            tile(w0, w1, 0);
            tn += NC * gstep;
            if (tn >= a.nt) break;
            tile(w1, w0, 1);
            tn += NC * gstep;
            if (tn >= a.nt) break;
        }
    } else {
        tile(w0, w0, 0);
    }
    if constexpr (EPI == EPI_HEAD) {
        // a row's best over the workgroup's columns (16 lanes), one pair per row
#pragma unroll
        for (int s = 0; s < RS; ++s) {
            const int ei = (tid >> 4) + 32 * s, em = m0 + ei;
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) {
                const float ov = __shfl_xor(best[s], o, 16);
                const int oi = __shfl_xor(bidx[s], o, 16);
                pick(ov, oi, best[s], bidx[s]);
            }
            if ((tid & 15) == 0 && ei < ROWS && em < a.M) {
                float* dst = a.part + ((long)em * a.nparts + slot) * 2;
                dst[0] = best[s];
                dst[1] = __int_as_float(bidx[s]);
            }
        }
    }
}

// x * g in fragment order and the partial sums of x^2 per 16 columns, for the first RMSNorm
// of the step (d % 16 == 0: every 16-lane group is one row's 16 columns). Rows M .. M16-1
// (the last row tile's padding) are written as zeros.
__global__ __launch_bounds__(256) void xg_ssq_kernel(const float* __restrict__ x, long ldx,
                                                     const float* __restrict__ g,
                                                     float* __restrict__ xg,
                                                     float* __restrict__ ssq, int M, int d) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int m = (int)(i / d), n = (int)(i % d);
    const bool ok = m < M;
    const float v = ok ? x[(long)m * ldx + n] : 0.f;
    xg[frag_off(m, n, d / 16)] = v * g[n];
    const float t = sum16(v * v);
    if (ok && (n & 15) == 0) ssq[(long)m * (d / 16) + n / 16] = t;
}

// The embedding gather of a one-token step fused with the first RMSNorm's operand: hid (M, d)
// = E[ids], xg = hid * g in fragment order and the partial sums of hid^2 per 16 columns, as
// embed_kernel and xg_ssq_kernel would write them one after the other (ids past V flag *bad
// and read row 0). M16 * d threads, d % 16 == 0, so the grid is whole blocks of 256.
__global__ __launch_bounds__(256) void embed_xg_kernel(const uint32_t* __restrict__ ids,
                                                       const float* __restrict__ emb,
                                                       float* __restrict__ hid,
                                                       const float* __restrict__ g,
                                                       float* __restrict__ xg,
                                                       float* __restrict__ ssq, int M, int d,
                                                       int V, int* bad) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int m = (int)(i / d), n = (int)(i % d);
    const bool ok = m < M;
    float v = 0.f;
    if (ok) {
        uint32_t id = ids[m];
        if (id >= (uint32_t)V) {
            if (n == 0) atomicOr(bad, 1);
            id = 0;
        }
        v = emb[(long)id * d + n];
        hid[(long)m * d + n] = v;
    }
    xg[frag_off(m, n, d / 16)] = v * g[n];
    const float t = sum16(v * v);
    if (ok && (n & 15) == 0) ssq[(long)m * (d / 16) + n / 16] = t;
}

// W (N, K) row stride ldw -> W^T (K, N) row-major, out[k N + n] = W[n ldw + k]: the conv
// epilogue's x_proj slice of a tile is then 16 contiguous rows. One thread per element (runs
// once per weight change).
__global__ __launch_bounds__(256) void pack_t_kernel(const float* __restrict__ W, long ldw,
                                                     int N, int K, float* __restrict__ out) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)N * K) return;
    const int k = (int)(i / N), n = (int)(i % N);
    out[i] = W[(long)n * ldw + k];
}

// W (N, K) row-major -> quads, out[((k / 4) N + n) 4 + k % 4] = W[n K + k]: a thread that owns
// row n reads its quads as float4s that are contiguous across a wave (the Mamba-1 step's
// dt_proj rows). One thread per quad (runs once per weight change).
__global__ __launch_bounds__(256) void pack_q4_kernel(const float* __restrict__ W, int N, int K,
                                                      float4* __restrict__ out) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;   // quad index (k / 4) N + n
    if (i >= (long)N * (K / 4)) return;
    const int n = (int)(i % N), k4 = (int)(i / N);
    const float* r = W + (long)n * K + 4 * k4;
    out[i] = make_float4(r[0], r[1], r[2], r[3]);
}

template <int MT, int NC, int KW, bool MULTI>
ssm_status launch_mk(int epi, const StepProj& a, unsigned grid, hipStream_t st) {
    switch (epi) {
        case EPI_STORE: stepproj_kernel<MT, NC, KW, MULTI, EPI_STORE><<<grid, kNT, 0, st>>>(a); break;
        case EPI_CONV:
            if (a.xpart) stepproj_kernel<MT, NC, KW, MULTI, EPI_CONVX><<<grid, kNT, 0, st>>>(a);
            else stepproj_kernel<MT, NC, KW, MULTI, EPI_CONV><<<grid, kNT, 0, st>>>(a);
            break;
        case EPI_HEAD: stepproj_kernel<MT, NC, KW, MULTI, EPI_HEAD><<<grid, kNT, 0, st>>>(a); break;
        default: stepproj_kernel<MT, NC, KW, MULTI, EPI_RESID><<<grid, kNT, 0, st>>>(a); break;
    }
    return check_launch("stepproj");
}

}  // namespace

bool stepproj_ok(int M, int N, int K) {
    return M >= 1 && M <= kStepProjMaxRows && N >= 1 && K >= 16 && K % 16 == 0 &&
           (long)K * 64 < (1L << 31);
}

ssm_status launch_pack_t(const float* W, long ldw, int N, int K, float* out, hipStream_t st) {
    SSM_REQUIRE(W && out && N >= 1 && K >= 1 && ldw >= K, "pack_t: arguments");
    const long n = (long)N * K;
    pack_t_kernel<<<(unsigned)cdiv(n, 256), 256, 0, st>>>(W, ldw, N, K, out);
    return check_launch("pack_t");
}

ssm_status launch_pack_q4(const float* W, int N, int K, float* out, hipStream_t st) {
    SSM_REQUIRE(W && out && N >= 1 && K >= 4 && K % 4 == 0 && ((uintptr_t)out & 15) == 0,
                "pack_q4: arguments");
    const long n = (long)N * (K / 4);
    pack_q4_kernel<<<(unsigned)cdiv(n, 256), 256, 0, st>>>(W, N, K, (float4*)out);
    return check_launch("pack_q4");
}

// Row tiles (rt) and column tiles (nc) per workgroup: as many rows as still give most CUs a
// workgroup (W then crosses the L2 fewer times, but each workgroup loads and splits its rows of
// X). Three and four row tiles go as two groups of two with two column tiles each: half the X
// per workgroup for the same W (64 rows of 4384 x 1024: 14.7 us with all rows and one column
// tile, 13.2 this way). 64 rows of 2048 -> 1024 leave one row tile each, 256 workgroups. per:
// 32-wide k-blocks per wave and pass, what the registers hold of X next to W.
namespace {
constexpr int kStepMaxWG = 256;   // workgroups that walk column groups: one per CU
struct StepPlan {
    int rt, nc, rg, per, npass;
    bool multi;
    unsigned grid;
};
StepPlan step_plan(int M, int N, int K) {
    const int mt = (M + 15) / 16, nt = (N + 15) / 16;
    const int kw = (int)cdiv(cdiv(K, 32), kNW);   // k-blocks per wave
    StepPlan p;
    p.rt = mt <= 1 || (long)nt * cdiv(mt, 2) < 192 ? 1 : 2;
    p.rg = (int)cdiv(mt, p.rt);
    p.nc = p.rt == 2 && p.rg == 2 && nt >= 192 ? 2 : 1;
    p.per = p.rt > 1 || kw <= 4 ? 4 : 8;
    p.npass = kw > 4 && p.per == 4 ? 2 * (int)cdiv(kw, 8) : (int)cdiv(kw, p.per);
    const long groups = cdiv(nt, p.nc), padded = 8L * cdiv(groups, 8);
    p.multi = p.npass == 1 && padded * p.rg > kStepMaxWG && kStepMaxWG % (8 * p.rg) == 0;
    p.grid = p.multi ? (unsigned)kStepMaxWG : (unsigned)(padded * p.rg);
    return p;
}
}  // namespace

int step_head_parts(int M, int N, int K) {
    const StepPlan p = step_plan(M, N, K);
    return p.multi ? (int)p.grid / p.rg : (int)cdiv((N + 15) / 16, p.nc);
}

ssm_status launch_stepproj(int epi, StepProj a, hipStream_t st) {
    SSM_REQUIRE(stepproj_ok(a.M, a.N, a.K) && ((uintptr_t)a.X & 15) == 0 &&
                    ((uintptr_t)a.W & 15) == 0,
                "stepproj: unsupported shape %d x %d x %d", a.M, a.N, a.K);
    SSM_REQUIRE(!a.ssq || (a.nssq >= 1 && a.nssq <= kStepProjMaxSsq), "stepproj: nssq");
    SSM_REQUIRE(epi != EPI_CONV || (a.Kc >= 1 && a.Kc <= 8 && a.cw && a.cst && a.Yc),
                "stepproj: conv epilogue arguments");
    SSM_REQUIRE(epi != EPI_RESID || !a.g2 || (a.xg && a.ssq_out && a.N % 16 == 0),
                "stepproj: residual epilogue arguments");
    SSM_REQUIRE(!a.Yf || (epi == EPI_CONV && a.C % 16 == 0),
                "stepproj: fragment-order copy arguments");
    SSM_REQUIRE(!a.xpart || (epi == EPI_CONV && a.wxt && a.RN >= 1 && a.RN <= kXpartMaxRN &&
                             a.c0 % 16 == 0 && a.C % 16 == 0),
                "stepproj: x_proj partial arguments");
    SSM_REQUIRE(a.Wf && (epi != EPI_HEAD || a.part), "stepproj: arguments");
    // 32-bit offsets of the epilogue's operands
    SSM_REQUIRE((long)a.M * a.C * a.Kc * 4 < (1L << 31) && (long)a.C * a.RN * 4 < (1L << 31) &&
                    (long)a.M * a.ldy * 4 < (1L << 31),
                "stepproj: operand too large");
    a.mt = (a.M + 15) / 16;
    a.nt = (a.N + 15) / 16;
    a.we = (const int*)(a.W + step_ex_off(a.N, a.K));
    const StepPlan p = step_plan(a.M, a.N, a.K);
    a.rg = p.rg; a.npass = p.npass;
    SSM_REQUIRE(epi != EPI_HEAD || a.nparts == step_head_parts(a.M, a.N, a.K),
                "stepproj: head pairs");
    if (p.multi) {
        if (p.nc == 2) return launch_mk<2, 2, 4, true>(epi, a, p.grid, st);
        if (p.rt == 2) return launch_mk<2, 1, 4, true>(epi, a, p.grid, st);
        return p.per == 4 ? launch_mk<1, 1, 4, true>(epi, a, p.grid, st)
                          : launch_mk<1, 1, 8, true>(epi, a, p.grid, st);
    }
    if (p.nc == 2) return launch_mk<2, 2, 4, false>(epi, a, p.grid, st);
    if (p.rt == 2) return launch_mk<2, 1, 4, false>(epi, a, p.grid, st);
    return p.per == 4 ? launch_mk<1, 1, 4, false>(epi, a, p.grid, st)
                      : launch_mk<1, 1, 8, false>(epi, a, p.grid, st);
}

ssm_status launch_embed_xg(const uint32_t* ids, const float* emb, float* hid, const float* g,
                           float* xg, float* ssq, int M, int d, int V, int* bad, hipStream_t st) {
    SSM_REQUIRE(d % 16 == 0 && d / 16 <= kStepProjMaxSsq && M >= 0 && M <= kStepProjMaxRows,
                "embed_xg: d_model %d, rows %d", d, M);
    const long n = (long)((M + 15) / 16) * 16 * d;
    if (n == 0) return SSM_OK;
    embed_xg_kernel<<<(unsigned)cdiv(n, 256), 256, 0, st>>>(ids, emb, hid, g, xg, ssq, M, d, V,
                                                             bad);
    return check_launch("embed_xg");
}

ssm_status launch_xg_ssq(const float* x, long ldx, const float* g, float* xg, float* ssq, int M,
                         int d, hipStream_t st) {
    SSM_REQUIRE(d % 16 == 0 && d / 16 <= kStepProjMaxSsq, "xg_ssq: d_model %d", d);
    const long n = (long)((M + 15) / 16) * 16 * d;
    if (n == 0) return SSM_OK;
    xg_ssq_kernel<<<(unsigned)cdiv(n, 256), 256, 0, st>>>(x, ldx, g, xg, ssq, M, d);
    return check_launch("xg_ssq");
}

}  // namespace ssm
