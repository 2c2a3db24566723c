// Products of small models on v_mfma_f32_16x16x32_f16: C[M, N] = A[M, K] . B[N, K]^T for K of at most 1024 in whole
// 32-wide steps, with the RMSNorm of A's rows in front and the prompt step's epilogues behind, one launch per product.
// It serves the prompt steps of models whose widths the 32x32 kernels do not take (D % 64 != 0 or a head size that is not
// a power of two: the tiny decoder, dim 288) and the FFN_UP_AND_GATE op at such widths.
//
// At these sizes nothing is bound by bytes or flops: a launch costs its dispatch, one memory round trip and the chain of
// reductions behind it. So a workgroup makes one 16 x 16 tile (16 x 16 of up and of gate), its four waves taking every
// fourth 32-wide step of K; a wave requests all operands of its steps at once (lane l: row l % 16, K values 8 (l / 16)
// .. + 7 of a step, which is the MFMA operand as it lies in memory, so nothing is staged), and the four partial tiles
// are added in wave order in LDS. The norm is recomputed by every workgroup of a row block: 16 rows from registers.
//
// The tiny decoder's 16-token prompt step, us before and now: QKV (RMSNorm 2.9, tile GEMM 7.2, RoPE pass 3.2) 3.7, Wo
// (6.4) 3.0, gate and up (RMSNorm, 7.7, SwiGLU pass 2.3) 3.6, down (6.6, split-K reduce 3.6) 4.6.
#include "device_common.h"
#include "kernels.h"

namespace vk
{

namespace
{

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr bool dual(int epi)
{
    return epi == GEMM_SWIGLU || epi == GEMM_FFN;
}

// NS: 32-wide steps a wave holds (K <= 128 NS)
template <int EPI, bool NORM, int NS>
__global__ __launch_bounds__(256) void gemm_small_kernel(GemmSmallArgs g)
{
    constexpr int NT = dual(EPI) ? 2 : 1;
    __shared__ float part[4][NT][256];
    __shared__ float sums[4][16];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, r = lane % 16, kq = lane / 16;
    const uint32_t n0 = blockIdx.x * 16, m0 = blockIdx.y * 16, nsteps = g.K / 32;
    const uint32_t row = min(m0 + r, g.M - 1), col = min(n0 + r, g.N - 1);

    // Rows past M or N repeat the last one (they feed outputs that are not stored); steps past K re-read the last step
    // and enter as zeros. All loads are unconditional, so they are in flight together.
    u32x4 a[NS], b[NT][NS];
    float4 w[NORM ? NS : 1][2];
#pragma unroll
    for (int i = 0; i < NS; ++i)
    {
        const uint32_t k = 32 * min(wid + 4 * i, nsteps - 1) + 8 * kq;
        a[i] = *(const u32x4 *)(g.A + (size_t)row * g.K + k);
        if constexpr (NORM)
        {
            w[i][0] = *(const float4 *)(g.norm_w + k);
            w[i][1] = *(const float4 *)(g.norm_w + k + 4);
        }
        b[0][i] = *(const u32x4 *)(g.B + (size_t)col * g.K + k);
        if constexpr (NT == 2)
            b[1][i] = *(const u32x4 *)(g.B2 + (size_t)col * g.K + k);
    }
    if constexpr (NORM)
    {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NS; ++i)
        {
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k)
            {
                const float lo = half_lo(a[i][k]), hi = half_hi(a[i][k]);
                s += lo * lo;
                s += hi * hi;
            }
            ss += wid + 4 * i < nsteps ? s : 0.f;
        }
        ss += __shfl_xor(ss, 16, kWave);
        ss += __shfl_xor(ss, 32, kWave);
        if (lane < 16)
            sums[wid][lane] = ss;
        __syncthreads();
        ss = (sums[0][r] + sums[1][r]) + (sums[2][r] + sums[3][r]);
        const float alpha = 1.0f / sqrtf(ss / (float)g.K + g.eps);
#pragma unroll
        for (int i = 0; i < NS; ++i)
        {
            const float ws[8] = {w[i][0].x, w[i][0].y, w[i][0].z, w[i][0].w, w[i][1].x, w[i][1].y, w[i][1].z, w[i][1].w};
#pragma unroll
            for (int k = 0; k < 4; ++k)
                a[i][k] = pack2(f2h((half_lo(a[i][k]) * ws[2 * k]) * alpha), f2h((half_hi(a[i][k]) * ws[2 * k + 1]) * alpha));
        }
    }
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
        acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NS; ++i)
    {
        // a step past K adds nothing (uniform per wave); zeroing one operand would leave 0 * inf
        if (wid + 4 * i < nsteps)
#pragma unroll
            for (int t = 0; t < NT; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[i]),
                                                                __builtin_bit_cast(f16x8, b[t][i]), acc[t], 0, 0, 0);
    }
    // lane holds C[4 (l / 16) + e][l % 16]
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            part[wid][t][(4 * kq + e) * 16 + r] = acc[t][e];
    __syncthreads();
    // two neighbouring columns a thread
    if (tid >= 128)
        return;
    const uint32_t at = 2 * tid, m = m0 + at / 16, n = n0 + at % 16;
    if (m >= g.M || n >= g.N)
        return;
    float v[NT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int k = 0; k < 2; ++k)
            v[t][k] = (part[0][t][at + k] + part[1][t][at + k]) + (part[2][t][at + k] + part[3][t][at + k]);
    uint32_t out;
    if constexpr (EPI == GEMM_FFN)
        out = pack2(ffn_out(v[0][0], v[1][0]), ffn_out(v[0][1], v[1][1]));
    else if constexpr (EPI == GEMM_SWIGLU)
        out = pack2(swiglu_out(v[0][0], v[1][0]), swiglu_out(v[0][1], v[1][1]));
    else
        out = pack2(f2h(v[0][0]), f2h(v[0][1]));
    if constexpr (EPI == GEMM_QKV_ROPE)
    {
        const GemmRope &p = g.rope;
        const uint32_t region = (n >= p.D) + (n >= 2 * p.D), c = n - region * p.D, head = c / p.hd, dim = c % p.hd;
        const size_t cache = ((size_t)head * p.ctx + p.offset + m) * p.hd + dim;
        if (region == 2)
        {
            *(uint32_t *)(p.vc + cache) = out;
            return;
        }
        const float2 cs = *(const float2 *)(p.cs + (size_t)m * p.hd + dim);
        const float x0 = half_lo(out), x1 = half_hi(out);
        out = pack2(f2h(rope_mul_sub(cs.x, x0, cs.y, x1)), f2h(rope_mul_add(cs.y, x0, cs.x, x1)));
        *(uint32_t *)(region == 0 ? p.q + (size_t)m * p.D + c : p.kc + cache) = out;
        return;
    }
    uint32_t *o = (uint32_t *)(g.C + (size_t)m * g.N + n);
    if constexpr (EPI == GEMM_RESID)
    {
        const uint32_t x = *o;
        out = pack2(f2h(half_lo(x) + half_lo(out)), f2h(half_hi(x) + half_hi(out)));
    }
    *o = out;
}

template <int EPI, bool NORM> hipError_t launch_steps(hipStream_t st, const GemmSmallArgs &g)
{
    const dim3 grid((g.N + 15) / 16, (g.M + 15) / 16);
    if (g.K <= 3 * 128)
        gemm_small_kernel<EPI, NORM, 3><<<grid, 256, 0, st>>>(g);
    else
        gemm_small_kernel<EPI, NORM, 8><<<grid, 256, 0, st>>>(g);
    return hipGetLastError();
}

} // namespace

bool gemm_small_ok(uint32_t M, uint32_t N, uint32_t K)
{
    return K > 0 && K % 32 == 0 && K <= kGemmSmallMaxK && N % 2 == 0 && M > 0 && M <= 65535u * 16;
}

hipError_t launch_gemm_small(hipStream_t st, int epi, const GemmSmallArgs &g)
{
    if (!gemm_small_ok(g.M, g.N, g.K))
        return hipErrorInvalidValue;
    switch (epi)
    {
    case GEMM_PLAIN:
        return g.norm_w ? launch_steps<GEMM_PLAIN, true>(st, g) : hipErrorInvalidValue;
    case GEMM_RESID:
        return !g.norm_w ? launch_steps<GEMM_RESID, false>(st, g) : hipErrorInvalidValue;
    case GEMM_SWIGLU:
        return g.norm_w && g.B2 ? launch_steps<GEMM_SWIGLU, true>(st, g) : hipErrorInvalidValue;
    case GEMM_FFN:
        return !g.norm_w && g.B2 ? launch_steps<GEMM_FFN, false>(st, g) : hipErrorInvalidValue;
    case GEMM_QKV_ROPE:
        return g.norm_w && g.rope.cs && g.N == 3 * g.rope.D && g.rope.hd % 2 == 0 ? launch_steps<GEMM_QKV_ROPE, true>(st, g)
                                                                                 : hipErrorInvalidValue;
    default:
        return hipErrorInvalidValue;
    }
}

} // namespace vk
