// VKLLM_OP_MATMUL over batches on CDNA4 matrix cores: out[z] = act(scale * A[z] . B[z]) for fp16 operands whose rows are
// contiguous, any other strides, B as [N, K] or as [K, N] (src/shaders/vkllm_matmul_t1.comp, vkllm_matmul.comp): the
// score and P.V products of an attention layer run as graph nodes, and every 2-D product the prompt step's tile GEMM
// does not take (a scale, B as [K, N], ragged or strided rows).
//
// A workgroup of four waves (2 x 2) makes a BM x BN tile with v_mfma_f32_32x32x16_f16, K in steps of 64 through two LDS
// buffers of 144-byte rows (the operand reads of 8 lanes then fall on distinct banks), the next step's loads in flight
// during the products. B as [K, N] is turned on its way into LDS: a thread loads 8 columns of two neighbouring K rows and
// stores 8 dwords of two K values each, 32 lanes along K, so the stores are free of bank conflicts.
// Rows and bases need no alignment: vectors are loaded and stored as unaligned 16-byte accesses (global memory allows
// them; an odd row pitch, as a probability matrix over an odd number of cached positions has, costs the extra line).
//
// What bounds it: at the attention shapes the operands come from L2 and the fp16 result goes to HBM. 32 heads of 512 x
// 512 scores over 128 dims (17 MB out, 8.6 GFLOP): 11.1 us, against 69 us of the vector kernel (ops_generic.hip); P.V
// of the same heads: 11.1 us against 115 us.
#include "device_common.h"
#include "kernels.h"

namespace vk
{

namespace
{

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kStep = 64, kRow = kStep + 8; // K per step, halfs per LDS row

struct BatchedArgs
{
    const uint16_t *a, *b;
    uint16_t *out;
    uint32_t M, N, K, C; // C: the batch's inner extent (out.n[1])
    uint32_t am, bm, om; // element strides of rows
    uint32_t ab, ac, bb, bc, ob, oc; // of the batch dims (0 where an operand broadcasts)
    uint32_t tiles_m, tiles_n, total;
    float scale;
    int act;
};

// elements [0, cnt) of p, zeros after them (cnt <= 8, possibly negative)
__device__ __forceinline__ u32x4 load_some(const uint16_t *p, int cnt)
{
    if (cnt >= 8)
        return load_half8(p);
    uint16_t e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
        e[i] = i < cnt ? p[i] : (uint16_t)0;
    u32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        v[i] = pack2(e[2 * i], e[2 * i + 1]);
    return v;
}

template <int BM, int BN, bool TB> __global__ __launch_bounds__(256) void matmul_batched_kernel(BatchedArgs g)
{
    constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 32, TN = WN / 32;
    constexpr int AV = BM * kStep / 8 / 256, BV = BN * kStep / 8 / 256; // 16-byte vectors per thread and step
    constexpr int kOut = BN + 8;                                        // halfs per row of the output tile
    __shared__ __attribute__((aligned(16))) uint16_t lds[2 * (BM + BN) * kRow];
    static_assert(BM * kOut <= 2 * (BM + BN) * kRow, "output tile fits the step buffers");
    auto As = [&](int s) { return lds + s * BM * kRow; };
    auto Bs = [&](int s) { return lds + 2 * BM * kRow + s * BN * kRow; };

    // workgroups are dealt to the 8 XCDs round robin: each XCD takes a contiguous run of tiles, so a batch's operands
    // are read into one L2
    const uint32_t t = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
    if (t >= g.total)
        return;
    const uint32_t per = g.tiles_m * g.tiles_n, z = t / per, bz = z / g.C, cz = z % g.C;
    const uint32_t m0 = (t % per) % g.tiles_m * BM, n0 = (t % per) / g.tiles_m * BN;
    const uint16_t *A = g.a + (size_t)bz * g.ab + (size_t)cz * g.ac;
    const uint16_t *B = g.b + (size_t)bz * g.bb + (size_t)cz * g.bc;
    uint16_t *O = g.out + (size_t)bz * g.ob + (size_t)cz * g.oc;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wm = tid >> 7, wn = (tid >> 6) & 1;

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                acc[i][j][e] = 0.f;

    // Rows past M or N repeat the last one: they only feed outputs that are not stored. K values past K are zeros in
    // both operands. Vectors that cannot straddle the end of a row (whole 8s along it) are loaded unconditionally at
    // clamped addresses and masked afterwards, as a guarded load costs a branch and a wait each; only the last step of a
    // ragged K (or a ragged last column tile of a [K, N] B) takes guarded loads.
    const bool avec = g.K % 8 == 0, bvec = TB ? avec : g.N % 8 == 0;
    const u32x4 zero = {0, 0, 0, 0};
    u32x4 ra[AV], rb[BV];
    // vector (row, k) of rows along K, `rows` of them
    auto along_k = [&](u32x4 *r, int i, const uint16_t *P, uint32_t first, uint32_t rows, uint32_t pitch, uint32_t k0,
                       int mode) {
        const uint32_t v = tid + 256 * i, k = k0 + (v % 8) * 8;
        const uint16_t *p = P + (size_t)min(first + v / 8, rows - 1) * pitch;
        if (mode == 0)
            r[i] = load_half8(p + k);
        else if (mode == 1)
            r[i] = load_half8(p + min(k, g.K - 8));
        else
            r[i] = load_some(p + k, (int)g.K - (int)k);
        if (mode == 1 && k >= g.K)
            r[i] = zero;
    };
    // vector i of B as [K, N]: item tid + 256 (i / 2) is K rows k0 + 2 (item % 32) and the next, columns n0 + 8 (item /
    // 32) .. + 7
    auto along_n = [&](int i, uint32_t k0, bool vec) {
        const uint32_t item = tid + 256 * (i / 2), k = k0 + 2 * (item % 32) + i % 2, n = n0 + 8 * (item / 32);
        const uint16_t *p = B + (size_t)min(k, g.K - 1) * g.bm;
        rb[i] = vec ? load_half8(p + min(n, g.N - 8)) : load_some(p + n, (int)g.N - (int)n);
        if (k >= g.K)
            rb[i] = zero;
    };
    auto load = [&](uint32_t k0) {
        const bool full = k0 + kStep <= g.K; // uniform
#define EACH(n_, call_)                                                                                             \
    _Pragma("unroll") for (int i = 0; i < n_; ++i) call_
        if (full)
            EACH(AV, along_k(ra, i, A, m0, g.M, g.am, k0, 0));
        else if (avec)
            EACH(AV, along_k(ra, i, A, m0, g.M, g.am, k0, 1));
        else
            EACH(AV, along_k(ra, i, A, m0, g.M, g.am, k0, 2));
        if constexpr (TB)
        {
            if (full)
                EACH(BV, along_k(rb, i, B, n0, g.N, g.bm, k0, 0));
            else if (bvec)
                EACH(BV, along_k(rb, i, B, n0, g.N, g.bm, k0, 1));
            else
                EACH(BV, along_k(rb, i, B, n0, g.N, g.bm, k0, 2));
        }
        else if (bvec || n0 + BN <= g.N)
            EACH(BV, along_n(i, k0, true));
        else
            EACH(BV, along_n(i, k0, false));
#undef EACH
    };
    auto stash = [&](int s) {
#pragma unroll
        for (int i = 0; i < AV; ++i)
        {
            const uint32_t v = tid + 256 * i;
            *(u32x4 *)(As(s) + (v / 8) * kRow + (v % 8) * 8) = ra[i];
        }
        if constexpr (TB)
        {
#pragma unroll
            for (int i = 0; i < BV; ++i)
            {
                const uint32_t v = tid + 256 * i;
                *(u32x4 *)(Bs(s) + (v / 8) * kRow + (v % 8) * 8) = rb[i];
            }
        }
        else
        {
#pragma unroll
            for (int i = 0; i < BV; i += 2)
            {
                const uint32_t item = tid + 256 * (i / 2);
                uint16_t *p = Bs(s) + 8 * (item / 32) * kRow + 2 * (item % 32);
#pragma unroll
                for (int e = 0; e < 8; ++e)
                {
                    const uint32_t lo = rb[i][e / 2], hi = rb[i + 1][e / 2];
                    *(uint32_t *)(p + e * kRow) =
                        e % 2 == 0 ? (lo & 0xffffu) | (hi << 16) : (lo >> 16) | (hi & 0xffff0000u);
                }
            }
        }
    };

    load(0);
    stash(0);
    __syncthreads();
    int cur = 0;
    for (uint32_t k0 = 0; k0 < g.K; k0 += kStep, cur ^= 1)
    {
        const bool more = k0 + kStep < g.K;
        if (more)
            load(k0 + kStep);
#pragma unroll
        for (int sl = 0; sl < kStep / 16; ++sl)
        {
            f16x8 af[TM], bf[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
                af[i] = *(const f16x8 *)(As(cur) + (wm * WM + i * 32 + lane % 32) * kRow + sl * 16 + (lane / 32) * 8);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                bf[j] = *(const f16x8 *)(Bs(cur) + (wn * WN + j * 32 + lane % 32) * kRow + sl * 16 + (lane / 32) * 8);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
        if (more)
            stash(cur ^ 1);
        __syncthreads();
    }

    // fp16 results to a row-major tile in LDS, then 8 columns a store
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
            {
                float v = acc[i][j][e] * g.scale;
                if (g.act == 1)
                    v = silu(v);
                lds[(wm * WM + i * 32 + 8 * (e / 4) + 4 * (lane / 32) + e % 4) * kOut + wn * WN + j * 32 + lane % 32] =
                    f2h(v);
            }
    __syncthreads();
    for (uint32_t i = tid; i < BM * BN / 8; i += 256)
    {
        const uint32_t r = i / (BN / 8), c = (i % (BN / 8)) * 8, m = m0 + r, n = n0 + c;
        if (m >= g.M || n >= g.N)
            continue;
        const uint16_t *s = lds + r * kOut + c;
        uint16_t *p = O + (size_t)m * g.om + n;
        if (n + 8 <= g.N)
            store_half8(p, *(const u32x4 *)s);
        else
            for (uint32_t e = 0; n + e < g.N; ++e)
                p[e] = s[e];
    }
}

template <int BM, int BN> hipError_t launch_tiles(hipStream_t st, BatchedArgs g, uint64_t batches, bool tb)
{
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    const uint64_t total = batches * g.tiles_m * g.tiles_n;
    if (total > 0x7ffffff0u)
        return hipErrorInvalidValue;
    g.total = (uint32_t)total;
    const uint32_t grid = (g.total + 7) / 8 * 8;
    if (tb)
        matmul_batched_kernel<BM, BN, true><<<grid, 256, 0, st>>>(g);
    else
        matmul_batched_kernel<BM, BN, false><<<grid, 256, 0, st>>>(g);
    return hipGetLastError();
}

} // namespace

bool matmul_batched_ok(const TView &a, const TView &b, const TView &out)
{
    auto rows = [](const TView &v) { return v.dt == DT_F16 && v.s[3] == 1 && (uintptr_t)v.p % 2 == 0; };
    // extents in signed 32-bit tile arithmetic
    const uint32_t lim = 1u << 30;
    return rows(a) && rows(b) && rows(out) && out.n[2] < lim && out.n[3] < lim && a.n[3] < lim && a.n[3] > 0 &&
           (uint64_t)out.n[0] * out.n[1] * ((out.n[2] + 63) / 64) * ((uint64_t)(out.n[3] + 63) / 64) < 0x7ffffff0u;
}

hipError_t launch_matmul_batched(hipStream_t st, const TView &a, const TView &b, const TView &out, float scale, int act,
                                 bool transposed_b, int cu_count)
{
    BatchedArgs g{};
    g.a = (const uint16_t *)a.p;
    g.b = (const uint16_t *)b.p;
    g.out = (uint16_t *)out.p;
    g.M = out.n[2];
    g.N = out.n[3];
    g.K = a.n[3];
    g.C = out.n[1];
    g.am = a.s[2];
    g.bm = b.s[2];
    g.om = out.s[2];
    g.ab = a.n[0] == 1 ? 0 : a.s[0];
    g.ac = a.n[1] == 1 ? 0 : a.s[1];
    g.bb = b.n[0] == 1 ? 0 : b.s[0];
    g.bc = b.n[1] == 1 ? 0 : b.s[1];
    g.ob = out.s[0];
    g.oc = out.s[1];
    g.scale = scale;
    g.act = act;
    const uint64_t batches = (uint64_t)out.n[0] * out.n[1];
    if (g.M == 0 || g.N == 0 || batches == 0)
        return hipSuccess;
    // 128 x 128 tiles halve the operand bytes read per result but need two of them for every CU; below that 64 x 64 tiles
    // spread the same work over four times as many workgroups. Scores of 32 heads over 128 dims: 512 x 512 (512 large
    // tiles) 11.0 us against 12.5 us on small ones, 301 x 338 (288 large tiles) 11.2 us against 7.5 us
    const uint64_t cus = cu_count > 0 ? (uint64_t)cu_count : 256;
    if (batches * ((g.M + 127) / 128) * ((g.N + 127) / 128) >= 2 * cus)
        return launch_tiles<128, 128>(st, g, batches, transposed_b);
    return launch_tiles<64, 64>(st, g, batches, transposed_b);
}

} // namespace vk
