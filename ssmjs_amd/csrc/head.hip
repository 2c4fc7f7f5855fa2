// The one-token LM head (decode, M <= 64 rows; also the prefill's last positions and short
// forwards), with the final RMSNorm's scale and the greedy pick folded in:
//
//   logits[m, n] = s[m] * sum_k xg[m, k] E[n, k]      E (V, K): the tied embedding
//   s[m]         = 1 / sqrt(sum_j ssq[m, j] * inv_div + eps)
//
// xg = x * g_final (the final RMSNorm's operand, fragment order) and the partial sums ssq come
// from the last layer's out_proj epilogue (stepproj.hip), so the normalised row never goes
// through memory, as with every other norm of the step. The product is a step projection
// (stepproj.hip, EPI_HEAD): 256 workgroups that keep the split rows in registers and stream E
// from HBM. (On the fp32 matrix cores it was bound by their rate: 45 of 48.7 us for 64 x 32000 x
// 1024; now 32.8 us.)
//
// Greedy pick. Each workgroup also writes, per row, the largest logit among its columns with
// the lowest index among equal maxima (NaN never wins), as (value, index) pairs; the finishing
// kernel merges a row's pairs. The merge takes the larger value, or the lower index of equal
// values: a maximum under a total order, so any merge order gives the same pick, which is the
// full-row argmax of the stored logits (glue.hip's argmax_kernel).
#include "common.hpp"
#include "glue.hpp"

namespace ssm {
namespace {

// One workgroup per row: the row's pairs merged by a wave-shuffle and LDS tree.
constexpr int kFin = 256;
__global__ __launch_bounds__(kFin) void head_argmax_kernel(const float* __restrict__ part,
                                                           int nparts, int V,
                                                           uint32_t* __restrict__ out) {
    __shared__ float sv[kFin / 64];
    __shared__ int si[kFin / 64];
    const int row = blockIdx.x;
    const float* p = part + (long)row * nparts * 2;
    float best = -INFINITY;
    int bi = V;
    for (int c = threadIdx.x; c < nparts; c += kFin)
        pick(p[2 * c], __float_as_int(p[2 * c + 1]), best, bi);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(best, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        pick(ov, oi, best, bi);
    }
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) { sv[w] = best; si[w] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < kFin / 64; ++k) pick(sv[k], si[k], best, bi);
        out[row] = bi < V ? (uint32_t)bi : 0u;
    }
}

}  // namespace

bool head_ok(int M, int V, int K) {
    const long nt = (V + 15) / 16;
    return M >= 1 && M <= kStepProjMaxRows && V >= 1 && K >= 16 && K % 16 == 0 &&
           K / 16 <= kStepProjMaxSsq && nt * (K / 16) * 1024 < (1L << 31);
}

int head_parts(int V) { return (int)cdiv(V, 16); }

ssm_status launch_head(const float* xg, const float* ssq, int nssq, float inv_div, float eps,
                       const float* Ep, const float* E, float* y, long ldy, int M, int V, int K,
                       float* part, uint32_t* argmax, hipStream_t st) {
    SSM_REQUIRE(head_ok(M, V, K) && xg && ssq && Ep && E && y && part && ldy >= V && nssq >= 1,
                "head: unsupported arguments (%d x %d x %d)", M, V, K);
    StepProj p;
    p.X = xg; p.W = Ep; p.Wf = E; p.M = M; p.N = V; p.K = K;
    p.ssq = ssq; p.nssq = nssq; p.inv_div = inv_div; p.eps = eps;
    p.Y = y; p.ldy = ldy;
    p.part = part; p.nparts = step_head_parts(M, V, K);
    const ssm_status e = launch_stepproj(EPI_HEAD, p, st);
    if (e != SSM_OK || !argmax) return e;
    head_argmax_kernel<<<(unsigned)M, kFin, 0, st>>>(part, p.nparts, V, argmax);
    return check_launch("head_argmax");
}

}  // namespace ssm
