// Prefill projections on the fp16 matrix cores at fp32 precision: Y = beta * Y + X W^T,
// with X (M, K) and W (N, K) in fp32 (the Linear layers of the model behind model.forward).
//
// Split. Each row of an operand is scaled by a power of two (exact) so that its largest
// magnitude lies in [2^14, 2^15), and each scaled element v is held as two fp16 values,
// hi = fp16(v) and lo = fp16(v - hi), both rounded to nearest: v - hi is exact in fp32, and
// hi + lo is v to 2^-23 |v| or 2^-25 (2^-39 of the row's largest magnitude), whichever is
// larger (2^-25 for each element that may have the latter is kept as the row's rho). The product of a row pair is summed as lo hi + hi lo + hi hi in fp32 accumulators
// (v_mfma_f32_16x16x32_f16, whose products are exact in fp32), leaving out lo lo (2^-22 of a
// product at most); the sum is scaled back exactly in the epilogue. Three MFMAs at 16 times the fp32
// matrix rate replace one, and 3 K / 32 roundings of the running sum replace K / 4.
//
// Range. Elements 2^-17 of their row's largest magnitude and smaller lose bits, which matters
// where the large elements meet zeros or tiny ones, so that the small ones make up the sum.
// Every output is held against rho (below) and, where its sum is not large enough to
// cover the loss, formed again from the fp32 operands on the fp32 matrix cores, 16 x 16 outputs
// at a time: the error is at most (3 K / 32) 2^-24 + 2^-20 of S = sum |x w| for any finite
// operands (or the fp32 product's K / 4 roundings of 2^-24). Normal data takes no such path; the
// tests of its sums cost nothing measurable at 8192 rows, and the packing's counts 1 us of 9 at
// 1000 rows of 2048.
//
// Non-finite values. An inf or NaN element becomes a NaN in hi, so that every output of its
// row (column) comes out NaN; an output that is not finite is formed again in the same way, and
// so gets fp32 arithmetic's own inf or NaN. Rows whose largest magnitude is tiny or huge are
// scaled by ldexp, which covers the whole fp32 range.
//
// Packed order. Both operands are read in the MFMA's own order: the 16-row block rb and the
// 32-k block kb hold two 1 KB fragments (hi, lo), lane 16 q + i of which has row 16 rb + i,
// k = 32 kb + 8 q .. + 7. Weights are packed once per load of the weights, activations by
// pack_h3_kernel before their product (4 bytes per element, as fp32). A fragment goes
// global -> LDS with one 16-byte-per-lane direct load and comes back with one ds_read_b128
// per lane, lane-linear both times: no bank conflicts, no registers, no address arithmetic.
//
// Bound: the fp32 matrix cores peak at 157 TFLOP/s, and the fp32 kernel of gemm.hip ran these
// products at 134-150; three fp16 MFMAs per product peak at about 800, and what limits this
// kernel is the LDS reads per MFMA of the smaller tiles (and the clock under full MFMA load for
// the largest: 1.36 PFLOP/s of fp16 work). Measured on MI355X, fp32 kernel -> this one (the
// packing of X not included; it runs at 5 TB/s), with the relative error against 64 bits:
//   M 8192  N 3072 K 768    282 -> 108 us (358 TFLOP/s)   5.0e-7 -> 3.1e-7
//   M 8192  N 768  K 1536   143 -> 58                     7.0e-7 -> 4.4e-7
//   M 4096  N 8512 K 2048  1066 -> 363 (393)              8.1e-7 -> 5.0e-7
//   M 32768 N 2048 K 4096  3670 -> 1216 (452)             1.2e-6 -> 7.1e-7
//   M 1000  N 4384 K 1024    96 -> 36                     5.7e-7 -> 3.6e-7
// and against hipBLASLt for prompts of 65 to 255 tokens: M 200 N 2048 K 512 10.0 -> 7.4 us.
#include <algorithm>

#include "common.hpp"
#include "glue.hpp"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kKB = 32;              // k per block (one MFMA)
constexpr int kFragB = 1024;         // bytes per fragment
constexpr int kPairB = 2 * kFragB;   // hi and lo of a (row block, k block)
constexpr float kRhoZero = -1e30f;   // rho of a row of zeros: its sums are exact

// ---------------------------------------------------------------- packing
// Workgroup rb packs rows 16 rb .. + 15 (zeros past R): eight waves share the row block's k
// blocks, the block's values stay in registers (KW k blocks per wave) between the row maxima
// and the conversion.
struct PackArgs {
    const float* X; long ldx;
    int R, K, KB;
    char* P;
    int* ex;     // per row: the power of two that undoes the scaling
    float* rho;  // per row: a bound of what hi + lo leave out beyond 2^-23 of each element (scaled)
};

// STEP: the order of k of the one-token step's operand (stepproj.hip: lane (q, i) holds k = 4 q ..
// + 3 of the block's first 16, then of its second 16), and the row's exponent and rho in one word
// (step_ex_off in glue.hpp). VEC: 16-byte loads (rows 16-byte aligned).
template <int KW, bool STEP, bool VEC>
__global__ __launch_bounds__(512) void pack_h3_kernel(PackArgs a) {
    __shared__ unsigned red[8][16];
    __shared__ int rred[8][16];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, i16 = lane & 15;
    const int rb = blockIdx.x;
    const int rows = min(16, a.R - 16 * rb);
    const auto rx = ssm::rsrc(a.X + (long)rb * 16 * a.ldx,
                              (unsigned)(((long)(rows - 1) * a.ldx + a.K) * 4));
    const unsigned row_oor = i16 < rows ? 0u : 0x80000000u;
    const unsigned base = (unsigned)((long)i16 * a.ldx * 4);
    floatx4 v[KW][2];
    unsigned mx = 0;
    // k blocks w, w + 8, ...; per pass KW of them (one pass unless K > 256 KW)
    auto fetch = [&](int kb0) {
#pragma unroll
        for (int u = 0; u < KW; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int k = (kb0 + 8 * u) * kKB + (STEP ? 16 * h + 4 * q : 8 * q + 4 * h);
                const unsigned oor = k < a.K ? row_oor : 0x80000000u;   // (K % 4 == 0)
                const unsigned o = base + (unsigned)k * 4u;
                if constexpr (VEC) {
                    v[u][h] = ssm::bload16<floatx4>(rx, o | oor);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[u][h][e] = ssm::bload4(rx, (o + 4u * e) | oor);
                }
            }
    };
    auto maxima = [&]() {
#pragma unroll
        for (int u = 0; u < KW; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x = v[u][h][e];   // (a bit_cast of the element itself reads [0])
                    const unsigned m = __builtin_bit_cast(unsigned, x) & 0x7fffffffu;
                    mx = max(mx, m);
                }
    };
    const bool once = a.KB <= 8 * KW;
    for (int kb0 = w; kb0 < a.KB; kb0 += 8 * KW) {
        fetch(kb0);
        maxima();
    }
    mx = max(mx, (unsigned)__shfl_xor((int)mx, 16));
    mx = max(mx, (unsigned)__shfl_xor((int)mx, 32));
    if (q == 0) red[w][i16] = mx;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; ++k) mx = max(mx, red[k][i16]);
    // biased exponent of the largest magnitude (inf / NaN rows: the largest finite one)
    const int E = min((int)(mx >> 23), 254);
    const int sh = mx ? 141 - E : 0;
    if (!STEP && w == 0 && q == 0) a.ex[16 * rb + i16] = -sh;
    // What is left out past 2^-23 of an element is 2^-25 at most, and nothing from 2^-2 scaled on:
    // the elements below that are counted, zeros aside (in the doubled bits less one, where a zero
    // is the largest). Three instructions an element; the sum of what is really left out, a quarter
    // of this, took nine (1000 x 2048 8.9 -> 10.4 us).
    const unsigned lim = (unsigned)max(E - 16, 1) << 24;
    int small = 0;
    for (int kb0 = w; kb0 < a.KB; kb0 += 8 * KW) {
        if (!once) fetch(kb0);
#pragma unroll
        for (int u = 0; u < KW; ++u) {
            const int kb = kb0 + 8 * u;
            if (kb >= a.KB) break;
            halfx8 hi, lo;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x = v[u][e >> 2][e & 3];
                const float s = __builtin_ldexpf(x, sh);
                const bool fin = (__builtin_bit_cast(unsigned, x) & 0x7f800000u) != 0x7f800000u;
                const _Float16 hh = (_Float16)s;
                small += 2u * __builtin_bit_cast(unsigned, x) - 1u < lim;
                hi[e] = fin ? hh : (_Float16)__builtin_nanf("");
                lo[e] = fin ? (_Float16)(s - (float)hh) : (_Float16)0.f;
            }
            halfx8* o = reinterpret_cast<halfx8*>(a.P + ((long)rb * a.KB + kb) * kPairB) + lane;
            o[0] = hi;
            o[64] = lo;
        }
    }
    small += __shfl_xor(small, 16);
    small += __shfl_xor(small, 32);
    if (q == 0) rred[w][i16] = small;
    __syncthreads();
    if (w == 0 && q == 0) {
        small = rred[0][i16];
#pragma unroll
        for (int k = 1; k < 8; ++k) small += rred[k][i16];
        const float rho = mx ? 0x1p-25f * (float)small : kRhoZero;
        if constexpr (STEP) {
            const unsigned up = __builtin_bit_cast(unsigned, rho) + (mx ? 0xffffu : 0u);
            a.ex[16 * rb + i16] = (int)((up & 0xffff0000u) | ((unsigned)-sh & 0xffffu));
        } else {
            a.rho[16 * rb + i16] = rho;
        }
    }
}

// ---------------------------------------------------------------- product
struct H3Args {
    const char* Xp; const int* xe; const float* xr;
    const char* Wp; const int* we; const float* wr;
    const float* X; long ldx;      // the fp32 operands (outputs formed again)
    const float* W; long ldw;
    float* Y; long ldy;
    int M, N, K, KB;
    float beta;
    int mt, nt, gm_rows;
    const float* ssq; int nssq; float inv_div, eps;   // row scale, as in gemm.hip
    int gate_c0;                                       // silu from this column on
    int ks, kbs;                                       // split K: slices of kbs k blocks
    float* part;
};

__device__ __forceinline__ void to_lds16(__amdgpu_buffer_rsrc_t r, char* lds, unsigned voff,
                                         unsigned soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds, 16, voff, soff, 0, 0);
}

// At most KEEP of the wave's loads still in flight (vmcnt, in the gfx9 encoding; the other
// counters at their maxima), then the workgroup barrier: the next stage is whole, and every
// wave has finished with the stage read before. The scheduling barriers keep the step's MFMAs
// above the wait.
template <int KEEP>
__device__ __forceinline__ void h3_step() {
    static_assert(KEEP < 64, "vmcnt has six bits");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70 | (KEEP & 15) | ((KEEP >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

// The 16 x 16 outputs of a wave from the fp32 operands, k in [k0, k1), on the fp32 matrix cores:
// x and w are the lane's rows (row / column lane & 15), k quads 4 (lane >> 4) of each 16.
__device__ __forceinline__ floatx4 h3_exact(const float* x, const float* w, int k0, int k1) {
    const int q4 = 4 * ((threadIdx.x & 63) >> 4);
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    constexpr int U = 4;
    for (int k = k0; k < k1; k += 16 * U) {
        float4 xv[U], wv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kk = k + 16 * u + q4;   // (k0, k1 are multiples of 4)
            const bool in = kk < k1;
            xv[u] = in ? *reinterpret_cast<const float4*>(x + kk) : make_float4(0.f, 0.f, 0.f, 0.f);
            wv[u] = in ? *reinterpret_cast<const float4*>(w + kk) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[u].x, wv[u].x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[u].y, wv[u].y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[u].z, wv[u].z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[u].w, wv[u].w, acc, 0, 0, 0);
        }
    }
    return acc;
}

// Whether a running sum is large enough for its split: it bounds S = sum |x w| of the scaled
// operands from below, and 2^15 (rho_x + rho_w) bounds what the split's range leaves out, which is
// then at most 2^-22 S.
__device__ __forceinline__ bool h3_large(float s, float rx, float rw) {
    return fabsf(s) >= 0x1p37f * (rx + rw);
}

// WM x WN waves, each with TI x TJ 16 x 16 tiles: a workgroup owns (16 TI WM) x (16 TJ WN) of
// Y and walks its k blocks through NS LDS stages (each its own LDS object, so that reading one
// does not wait for loads into the others), NS - 1 blocks' fragments in flight while one
// multiplies. Loads past the last block are pushed out of range: the wait counts stay exact.
template <int WM, int WN, int TI, int TJ, int NS, bool BETA, bool RS, bool SPLIT>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_h3_kernel(H3Args a) {
    constexpr int NW = WM * WN, XF = TI * WM, WF = TJ * WN;
    constexpr int BM = 16 * XF, BN = 16 * WF;
    constexpr int NF = 2 * (XF + WF), PER = NF / NW;
    static_assert(NF % NW == 0, "fragments shared out evenly");
    static_assert(NS == 2 || NS == 4, "two or four stages");
    __shared__ __attribute__((aligned(16))) char s0[NF * kFragB];
    __shared__ __attribute__((aligned(16))) char s1[NF * kFragB];
    __shared__ __attribute__((aligned(16))) char s2[NS > 2 ? NF * kFragB : 16];
    __shared__ __attribute__((aligned(16))) char s3[NS > 2 ? NF * kFragB : 16];
    __shared__ float rs[RS ? BM : 1];
    __shared__ int2 words[BM + BN];

    // ---- tile of this workgroup (the order of gemm.hip: consecutive ids per XCD, groups of
    // gm_rows row tiles)
    const int mtv = SPLIT ? a.mt * a.ks : a.mt;
    const int T = mtv * a.nt;
    const int b = blockIdx.x;
    const int xcd = b & 7, per = T >> 3, rem = T & 7;
    const int id = xcd * per + min(xcd, rem) + (b >> 3);
    const int gsz = a.gm_rows * a.nt;
    const int grp = id / gsz, gr = id - grp * gsz;
    const int gm = min(a.gm_rows, mtv - grp * a.gm_rows);
    const int tmv = grp * a.gm_rows + gr % gm, tn = gr / gm;
    const int kz = SPLIT ? tmv / a.mt : 0, tm = SPLIT ? tmv - kz * a.mt : tmv;
    const int kb0 = SPLIT ? kz * a.kbs : 0;
    const int kb1 = SPLIT ? min(kb0 + a.kbs, a.KB) : a.KB;

    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, i16 = lane & 15;
    const int wm = w / WN, wn = w % WN;
    const int m0 = tm * BM, n0 = tn * BN;
    const int rows = min(BM, a.M - m0), cols = min(BN, a.N - n0);
    const unsigned rbs = (unsigned)a.KB * kPairB;   // bytes per packed row block
    const auto rx = ssm::rsrc(a.Xp + (long)(m0 / 16) * rbs, (unsigned)((rows + 15) / 16) * rbs);
    const auto rw = ssm::rsrc(a.Wp + (long)(n0 / 16) * rbs, (unsigned)((cols + 15) / 16) * rbs);

    // wave w loads fragments PER w .. PER w + PER - 1 of a stage: the X row blocks' (hi, lo)
    // pairs, then the W row blocks'; row blocks past the operand read zeros
    unsigned off[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int f = PER * w + u;
        const int r = f < 2 * XF ? f >> 1 : (f - 2 * XF) >> 1;
        off[u] = (unsigned)r * rbs + (f & 1) * kFragB + 16u * lane;
    }
    auto load = [&](char* s, int kb) {
        const unsigned kk = (unsigned)min(kb, kb1) * kPairB;
        const unsigned oor = kb < kb1 ? 0u : 0x80000000u;
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int f = PER * w + u;
            if (f < 2 * XF) to_lds16(rx, s + f * kFragB, off[u] | oor, kk);
            else to_lds16(rw, s + f * kFragB, off[u] | oor, kk);
        }
    };

    // the rows' and columns' exponents and losses, for the test halfway and the epilogue: a word a
    // thread, loaded ahead of the stages (a wait for it does not wait for them)
    static_assert(BM + BN <= 64 * NW, "a word a thread");
    int2 word = make_int2(0, __builtin_bit_cast(int, kRhoZero));
    {
        const int t = threadIdx.x, k = t < BM ? t : t - BM;
        if (k < (t < BM ? rows : cols)) {
            word.x = t < BM ? a.xe[m0 + k] : a.we[n0 + k];
            word.y = __builtin_bit_cast(int, t < BM ? a.xr[m0 + k] : a.wr[n0 + k]);
        }
    }
    auto rho_of = [](int2 v) { return __builtin_bit_cast(float, v.y); };
    auto row_word = [&](int i, int r) { return words[16 * (TI * wm + i) + 4 * q + r]; };
    auto col_word = [&](int j) { return words[BM + 16 * (TJ * wn + j) + i16]; };

    floatx4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    auto frag = [&](const char* s, int f) {
        return *reinterpret_cast<const halfx8*>(s + f * kFragB + 16 * lane);
    };
    constexpr int IH = TI > 4 ? TI / 2 : TI;   // row blocks whose operands are held at a time
    auto compute = [&](const char* s) {
        halfx8 wh[TJ], wl[TJ];
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            wh[j] = frag(s, 2 * (XF + TJ * wn + j));
            wl[j] = frag(s, 2 * (XF + TJ * wn + j) + 1);
        }
#pragma unroll
        for (int h = 0; h < TI; h += IH) {
            halfx8 xh[IH], xl[IH];
#pragma unroll
            for (int i = 0; i < IH; ++i) {
                xh[i] = frag(s, 2 * (TI * wm + h + i));
                xl[i] = frag(s, 2 * (TI * wm + h + i) + 1);
            }
#pragma unroll
            for (int i = 0; i < IH; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j)
                    acc[h + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[i], wh[j], acc[h + i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < IH; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j)
                    acc[h + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[i], wl[j], acc[h + i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < IH; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j)
                    acc[h + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[i], wh[j], acc[h + i][j], 0, 0, 0);
        }
    };

    // The sums are held against the rows' losses halfway (okm: tiles whose sums all are large), and
    // at the end for the others: a row's rho is mostly 0 or a few 2^-26 and its sums 2^27 and more,
    // so an output fails both only where large elements meet small ones.
    static_assert(TI * TJ <= 32, "a bit per tile");
    unsigned okm = 0;
    // (A slice is only part of a sum: its outputs are held against the losses by the finish.)
    const int kbm = SPLIT ? kb1 : kb0 + (kb1 - kb0) / (2 * NS) * NS;   // whole turns of the loop below
    int kb = kb0, end = kbm > kb0 ? kbm : kb1;
    if constexpr (NS == 2) {
        load(s0, kb0);
    } else {
        load(s0, kb0);
        load(s1, kb0 + 1);
        load(s2, kb0 + 2);
    }
    if ((int)threadIdx.x < BM + BN) words[threadIdx.x] = word;
    // lgkmcnt(0): written before the first turn's barrier, past which the words are read
    __builtin_amdgcn_s_waitcnt(0xc07f);
    for (;;) {
        if constexpr (NS == 2) {
            for (; kb < end; kb += 2) {
                h3_step<0>();
                load(s1, kb + 1);
                compute(s0);
                h3_step<0>();
                load(s0, kb + 2);
                if (kb + 1 < kb1) compute(s1);
            }
        } else {
            for (; kb < end; kb += 4) {   // blocks past kb1 multiply zeros
                h3_step<2 * PER>();
                load(s3, kb + 3);
                compute(s0);
                h3_step<2 * PER>();
                load(s0, kb + 4);
                compute(s1);
                h3_step<2 * PER>();
                load(s1, kb + 5);
                compute(s2);
                h3_step<2 * PER>();
                load(s2, kb + 6);
                compute(s3);
            }
        }
        asm volatile("" ::: "memory");   // no read of `words` moves above the turns' barriers
        if (end == kb1) break;
        end = kb1;
        float wr[TJ];
#pragma unroll
        for (int j = 0; j < TJ; ++j) wr[j] = rho_of(col_word(j));
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            float xr[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) xr[r] = rho_of(row_word(i, r));
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                bool ok = true;
#pragma unroll
                for (int r = 0; r < 4; ++r) ok = ok && h3_large(acc[i][j][r], xr[r], wr[j]);
                okm |= ok ? 1u << (i * TJ + j) : 0u;
            }
            __builtin_amdgcn_sched_barrier(0);   // (few registers beside the sums)
        }
    }
    // the loads past the last block end before the LDS they write is given back
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)

    if constexpr (RS) {
        for (int r = threadIdx.x; r < BM; r += 64 * NW) {
            float v = 1.f;
            if (r < rows) {
                const float* p = a.ssq + (long)(m0 + r) * a.nssq;
                float sum = 0.f;
                for (int j = 0; j < a.nssq; ++j) sum += p[j];
                v = rsqrtf(sum * a.inv_div + a.eps);
            }
            rs[r] = v;
        }
        __syncthreads();
    }

    // ---- epilogue: acc[i][j][r] is Y[m0 + 16 (TI wm + i) + 4 q + r][n0 + 16 (TJ wn + j) + i16]
    const long ldo = SPLIT ? a.N : a.ldy;
    float* yo = SPLIT ? a.part + ((long)kz * a.M + m0) * a.N + n0 : a.Y + (long)m0 * a.ldy + n0;
    const auto ry = ssm::rsrc(yo, (unsigned)(((long)(rows - 1) * ldo + cols) * 4));
    int2 ww[TJ];
#pragma unroll
    for (int j = 0; j < TJ; ++j) ww[j] = col_word(j);
    // one output: row scale, beta, gate, store
    auto put = [&](float v, int row, int c) __attribute__((always_inline)) {
        const unsigned o = ((unsigned)(row * ldo + c) * 4u) | (c < cols ? 0u : 0x80000000u);
        if constexpr (!SPLIT) {
            if constexpr (RS) v *= rs[row];
            if constexpr (BETA) v += a.beta * ssm::bload4(ry, o);
            if (n0 + (c & ~15) >= a.gate_c0) v = ssm::silu_fast(v);
        }
        ssm::bstore4(v, ry, o);
    };
    unsigned redo = 0;   // (uniform) tiles with outputs that are not finite or not covered
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        int2 xw[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) xw[r] = row_word(i, r);
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int c = 16 * (TJ * wn + j) + i16;
            float vv[4];
            bool fin = true, open = !SPLIT && !(okm >> (i * TJ + j) & 1);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                vv[r] = __builtin_ldexpf(acc[i][j][r], xw[r].x + ww[j].x);
                fin = fin && __builtin_isfinite(vv[r]);
            }
            if (__any(open || !fin)) {
                bool large = true;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    large = large && h3_large(acc[i][j][r], rho_of(xw[r]), rho_of(ww[j]));
                if (__any(!fin || (open && !large))) redo |= 1u << (i * TJ + j);
            }
            if (!(redo >> (i * TJ + j) & 1)) {
#pragma unroll
                for (int r = 0; r < 4; ++r) put(vv[r], 16 * (TI * wm + i) + 4 * q + r, c);
            }
        }
    }
    // the tiles left out, from the fp32 operands (here no accumulator is live)
    for (; redo; redo &= redo - 1) {
        const int t = __builtin_ctz(redo), i = t / TJ, j = t % TJ;
        const int xrow = min(16 * (TI * wm + i) + i16, rows - 1), c = 16 * (TJ * wn + j) + i16;
        const floatx4 v = h3_exact(a.X + (long)(m0 + xrow) * a.ldx,
                                   a.W + (long)(n0 + min(c, cols - 1)) * a.ldw, kb0 * kKB,
                                   min(kb1 * kKB, a.K));
#pragma unroll
        for (int r = 0; r < 4; ++r) put(v[r], 16 * (TI * wm + i) + 4 * q + r, c);
    }
}

// Split-K finish: Y = epilogue(sum over slices z = 0 .. ks-1 of part[z]), added in slice
// order; the epilogue in the unsplit kernel's order (row scale, beta, gate). Thread
// (row m = blockIdx.y, columns 4 c4 .. 4 c4 + 3); N % 4 == 0. The slices' magnitudes bound S from
// below, against the losses of the row and the columns; an output that they do not cover is formed
// again from the fp32 operands by its wave, 4 k a lane.
__global__ __launch_bounds__(256) void gemm_h3_finish_kernel(H3Args a) {
    const int m = blockIdx.y;
    const int c4 = blockIdx.x * 256 + threadIdx.x;
    const bool in = 4 * c4 < a.N;
    const long MN = (long)a.M * a.N;
    const int cc = in ? c4 : 0;   // (whole waves: an idle lane repeats the first columns)
    const float4* p = reinterpret_cast<const float4*>(a.part + (long)m * a.N) + cc;
    const int xe = a.xe[m];
    const float xr = a.xr[m];
    const int4 we = reinterpret_cast<const int4*>(a.we)[cc];
    const float4 wr = reinterpret_cast<const float4*>(a.wr)[cc];
    float4 v = p[0];
    float4 g = make_float4(fabsf(v.x), fabsf(v.y), fabsf(v.z), fabsf(v.w));
    for (int z = 1; z < a.ks; ++z) {
        const float4 u = p[z * (MN / 4)];
        v.x += u.x; v.y += u.y; v.z += u.z; v.w += u.w;
        g.x += fabsf(u.x); g.y += fabsf(u.y); g.z += fabsf(u.z); g.w += fabsf(u.w);
    }
    float s = 1.f;
    if (a.ssq) {   // same order as the unsplit kernel's row scales
        const float* q = a.ssq + (long)m * a.nssq;
        float sum = 0.f;
        for (int j = 0; j < a.nssq; ++j) sum += q[j];
        s = rsqrtf(sum * a.inv_div + a.eps);
    }
    float o[4] = {v.x, v.y, v.z, v.w};
    const float mag[4] = {g.x, g.y, g.z, g.w}, rho[4] = {wr.x, wr.y, wr.z, wr.w};
    const int ex[4] = {we.x, we.y, we.z, we.w};
    bool again[4];   // (NaN and inf are the slices' own)
#pragma unroll
    for (int e = 0; e < 4; ++e)
        again[e] = in && mag[e] < __builtin_ldexpf(0x1p37f * (xr + rho[e]), xe + ex[e]);
    if (__builtin_expect(__any(again[0] || again[1] || again[2] || again[3]), 0)) {
        const int lane = threadIdx.x & 63;
        const float* x = a.X + (long)m * a.ldx;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            for (unsigned long long todo = __ballot(again[e]); todo; todo &= todo - 1) {
                const int src = __builtin_ctzll(todo);
                const float* w = a.W + (long)(4 * __shfl(c4, src) + e) * a.ldw;
                float t = 0.f;
                for (int k = 4 * lane; k < a.K; k += 256) {   // (K % 4 == 0)
                    const float4 xv = *reinterpret_cast<const float4*>(x + k);
                    const float4 wv = *reinterpret_cast<const float4*>(w + k);
                    t = fmaf(xv.x, wv.x, t);
                    t = fmaf(xv.y, wv.y, t);
                    t = fmaf(xv.z, wv.z, t);
                    t = fmaf(xv.w, wv.w, t);
                }
#pragma unroll
                for (int d = 32; d > 0; d >>= 1) t += __shfl_xor(t, d);
                if (lane == src) o[e] = t;
            }
    }
    if (!in) return;
    float* y = a.Y + (long)m * a.ldy + 4 * c4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int n = 4 * c4 + e;
        float t = o[e];
        if (a.ssq) t *= s;
        if (a.beta != 0.f) t += a.beta * y[e];
        if (n >= a.gate_c0) t = ssm::silu_fast(t);
        y[e] = t;
    }
}

// ---------------------------------------------------------------- choice of tile and split
// Tiles: 256 x 256 on 8 waves, 128 x 128, 128 x 64 and 64 x 64 on 4. What a k block costs a CU
// holding n workgroups was measured on MI355X (us, fit over M 70 .. 32768, N 64 .. 32000, K
// 128 .. 4096): 2.4 n / 0.68 n / 0.37 n / 0.213 n, at least 0.70 and 0.50 for a lone 128 x 128
// or 128 x 64 workgroup (two stages: its loads are then exposed; the 64 x 64 tile keeps
// three blocks in flight and has no such floor). A launch costs about 4 us; a split one the
// finishing launch (1.8 us) and its partials written and read at 5 TB/s more. Per output the
// larger tile is the cheaper (LDS reads per MFMA), so the choice is between idle CUs and that.
struct H3Plan {
    int cfg, ks, kbs;
};

struct H3Tile {
    int bm, bn;
    double per, lone;
};
constexpr H3Tile kTiles[4] = {{256, 256, 2.4, 2.4}, {128, 128, 0.68, 0.70},
                              {128, 64, 0.37, 0.50}, {64, 64, 0.213, 0.213}};

H3Plan pick_h3(int M, int N, int K, size_t part_floats) {
    const int KB = (K + kKB - 1) / kKB;
    H3Plan best{3, 1, KB};
    double cost = 1e300;
    for (int c = 0; c < 4; ++c) {
        const H3Tile& t = kTiles[c];
        const long tiles = ssm::cdiv(M, t.bm) * ssm::cdiv(N, t.bn);
        auto busy = [&](long wgs, int kbs) {
            const long n = ssm::cdiv(wgs, 256);
            return 4.0 + std::max(t.lone, t.per * (double)n) * kbs;
        };
        const double c1 = busy(tiles, KB);
        if (c1 < cost) cost = c1, best = H3Plan{c, 1, KB};
        if (tiles >= 256 || N % 4) continue;
        for (int ks = 2; ks <= KB / 4; ++ks) {
            if ((size_t)ks * M * N > part_floats) break;
            const int kbs = (KB + ks - 1) / ks;
            if ((KB + kbs - 1) / kbs != ks) continue;
            const double cs = busy(tiles * ks, kbs) + 1.8 + 8.0e6 * ks * M * N / 5e12;
            if (cs < cost) cost = cs, best = H3Plan{c, ks, kbs};
        }
    }
    return best;
}

template <int WM, int WN, int TI, int TJ, int NS>
void launch_tile(H3Args a, hipStream_t st) {
    constexpr int BM = 16 * TI * WM, BN = 16 * TJ * WN;
    a.mt = (a.M + BM - 1) / BM;
    a.nt = (a.N + BN - 1) / BN;
    a.gm_rows = 8;
    const dim3 grid((unsigned)(a.mt * a.nt * a.ks)), block(64 * WM * WN);
    const bool beta = a.beta != 0.f;
    if (a.ks > 1) {
        gemm_h3_kernel<WM, WN, TI, TJ, NS, false, false, true><<<grid, block, 0, st>>>(a);
        gemm_h3_finish_kernel<<<dim3((unsigned)((a.N / 4 + 255) / 256), (unsigned)a.M), 256, 0,
                                st>>>(a);
    } else if (a.ssq) {
        if (beta) gemm_h3_kernel<WM, WN, TI, TJ, NS, true, true, false><<<grid, block, 0, st>>>(a);
        else gemm_h3_kernel<WM, WN, TI, TJ, NS, false, true, false><<<grid, block, 0, st>>>(a);
    } else {
        if (beta) gemm_h3_kernel<WM, WN, TI, TJ, NS, true, false, false><<<grid, block, 0, st>>>(a);
        else gemm_h3_kernel<WM, WN, TI, TJ, NS, false, false, false><<<grid, block, 0, st>>>(a);
    }
}

}  // namespace

namespace ssm {

// Offset of the row exponents behind a packed operand's fragments.
static size_t h3_ex_off(int rows, int K) {
    return (size_t)cdiv(rows, 16) * (size_t)cdiv(K, kKB) * kPairB;
}
size_t h3_bytes(int rows, int K) {
    const size_t b = h3_ex_off(rows, K) + (size_t)cdiv(rows, 16) * 16 * (sizeof(int) + sizeof(float));
    return (b + 255) & ~(size_t)255;
}

// ... and of the rows' rho behind the exponents.
static const float* h3_rho(const int* ex, int rows) {
    return (const float*)(ex + cdiv(rows, 16) * 16);
}

bool h3_ok(int M, int N, int K, long ldx, long ldw, long ldy) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 4) return false;
    if (ldx < K || ldw < K || ldy < N || ldx % 4 || ldw % 4) return false;
    // 32-bit offsets inside a tile's descriptors, bit 31 free for the range trick
    const long lim = 1L << 31;
    return 16 * ldx * 4 < lim && 16 * ldw * 4 < lim && 256 * std::max(ldy, (long)N) * 4 < lim &&
           16 * cdiv(K, kKB) * kPairB < lim && (cdiv(M, 64) * cdiv(N, 64)) < (1L << 30) &&
           M < (1 << 30);
}

size_t h3_split_floats(int M, int N, int K) {
    const H3Plan p = pick_h3(M, N, K, (size_t)-1);
    return p.ks > 1 ? (size_t)p.ks * M * N : 0;
}

template <bool STEP, bool VEC>
static ssm_status launch_pack(const PackArgs& a, hipStream_t st) {
    const unsigned grid = (unsigned)cdiv(a.R, 16);
    if (a.KB <= 16) pack_h3_kernel<2, STEP, VEC><<<grid, 512, 0, st>>>(a);
    else if (a.KB <= 32) pack_h3_kernel<4, STEP, VEC><<<grid, 512, 0, st>>>(a);
    else if (a.KB <= 64) pack_h3_kernel<8, STEP, VEC><<<grid, 512, 0, st>>>(a);
    else pack_h3_kernel<16, STEP, VEC><<<grid, 512, 0, st>>>(a);
    return check_launch("pack_h3");
}

ssm_status launch_pack_h3(const float* X, long ldx, int rows, int K, void* packed,
                          hipStream_t st) {
    SSM_REQUIRE(X && packed && rows > 0 && K > 0 && K % 4 == 0 && ldx >= K && ldx % 4 == 0 &&
                    ((uintptr_t)X & 15) == 0 && ((uintptr_t)packed & 15) == 0 &&
                    16 * ldx * 4 < (1L << 31),
                "pack_h3: arguments");
    int* ex = (int*)((char*)packed + h3_ex_off(rows, K));
    const PackArgs a{X, ldx, rows, K, (int)cdiv(K, kKB), (char*)packed, ex,
                     const_cast<float*>(h3_rho(ex, rows))};
    return launch_pack<false, true>(a, st);
}

// The step projection's weights (a layer's weights may start at any float offset).
size_t step_ex_off(int rows, int K) { return h3_ex_off(rows, K) / sizeof(float); }
size_t step_w_floats(int rows, int K) { return h3_bytes(rows, K) / sizeof(float); }
ssm_status launch_pack_step(const float* W, long ldw, int N, int K, float* out, hipStream_t st) {
    SSM_REQUIRE(W && out && N >= 1 && K % 16 == 0 && ldw >= K && ((uintptr_t)out & 15) == 0 &&
                    16 * ldw * 4 < (1L << 31),
                "pack_step: K %d / ldw %ld / alignment", K, ldw);
    const PackArgs a{W, ldw, N, K, (int)cdiv(K, kKB), (char*)out, (int*)(out + step_ex_off(N, K)),
                     nullptr};
    return ((uintptr_t)W & 15) == 0 && ldw % 4 == 0 ? launch_pack<true, true>(a, st)
                                                     : launch_pack<true, false>(a, st);
}

ssm_status launch_gemm_h3(const void* Xp, const float* X, long ldx, const void* Wp,
                          const float* W, long ldw, float* Y, long ldy, int M, int N, int K,
                          float beta, hipStream_t st, const float* ssq, int nssq, float inv_div,
                          float eps, int gate_c0, float* part, size_t part_floats) {
    SSM_REQUIRE(Xp && Wp && X && W && Y && h3_ok(M, N, K, ldx, ldw, ldy),
                "gemm_h3: unsupported shape M %d N %d K %d ld %ld/%ld/%ld", M, N, K, ldx, ldw, ldy);
    SSM_REQUIRE(gate_c0 >= N || gate_c0 % 16 == 0, "gemm_h3: gate column %d", gate_c0);
    SSM_REQUIRE(!ssq || nssq > 0, "gemm_h3: row scale needs nssq > 0");
    const bool ws = part && ((uintptr_t)part & 15) == 0;
    const H3Plan p = pick_h3(M, N, K, ws ? part_floats : 0);
    H3Args a{};
    a.Xp = (const char*)Xp; a.xe = (const int*)((const char*)Xp + h3_ex_off(M, K));
    a.xr = h3_rho(a.xe, M);
    a.Wp = (const char*)Wp; a.we = (const int*)((const char*)Wp + h3_ex_off(N, K));
    a.wr = h3_rho(a.we, N);
    a.X = X; a.ldx = ldx; a.W = W; a.ldw = ldw; a.Y = Y; a.ldy = ldy;
    a.M = M; a.N = N; a.K = K; a.KB = (int)cdiv(K, kKB); a.beta = beta;
    a.ssq = ssq; a.nssq = nssq; a.inv_div = inv_div; a.eps = eps; a.gate_c0 = gate_c0;
    a.ks = p.ks; a.kbs = p.kbs; a.part = part;
    switch (p.cfg) {
        case 0: launch_tile<2, 4, 8, 4, 2>(a, st); break;
        case 1: launch_tile<2, 2, 4, 4, 2>(a, st); break;
        case 2: launch_tile<2, 2, 4, 2, 2>(a, st); break;
        default: launch_tile<2, 2, 2, 2, 4>(a, st); break;
    }
    return check_launch("gemm_h3");
}

}  // namespace ssm
