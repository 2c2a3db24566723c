// Prefill GEMM on CDNA4 matrix cores: C[M, N] = A[M, K] . B[N, K]^T with fp16 operands and fp32 accumulation.
// It replaces src/shaders/vkllm_matmul_t1.comp for the token step's weight products, where A holds the step's
// activations (M = tokens) and B a weight matrix stored [out, in].
//
// gemm32_kernel (K a multiple of 64, every prefill product of the LLaMA-2 shapes): v_mfma_f32_32x32x16_f16 on tiles of 64
// x 128 to 256 x 256 by 256-thread workgroups, operands copied straight into a ring of LDS buffers, one barrier per 64 of
// K (described at the kernel). Its epilogue stages the tile's fp16 outputs in the freed LDS and stores 16-byte row chunks:
// plain, SiLU on columns >= split, residual add, the FFN's up * silu(gate) (reading up and gate rows as interleaved
// 16-row blocks), or the QKV product's RoPE with q and the K/V cache rows written directly.
// gemm_kernel (other K): v_mfma_f32_16x16x32_f16, 128 x 128 or 128 x 64 tiles, operands staged through registers into two
// LDS buffers, with the K tail zeroed (plain, SiLU and residual epilogues only).
//
// Narrow products split K over several workgroups; the fp32 partial tiles are added in split order by
// gemm_splitk_reduce_kernel, which applies the epilogue, or for a residual product followed by RMSNorm by
// gemm_resid_norm_kernel, which also normalises the rows. Tiles are ordered M-fastest and dealt to XCDs in
// contiguous runs so a run shares its B tiles in one L2. Global loads are unconditional at clamped addresses (a
// guarded load compiles to a branch and a wait per load).
#include <float.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "device_common.h"
#include "kernels.h"

namespace vk
{

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kBK = 64;
constexpr int kLdsRow = kBK + 8; // halfs per LDS row (144 bytes)

__device__ __forceinline__ void gemm_store(int epi, uint16_t *C, uint32_t ldc, uint32_t m, uint32_t n, float v,
                                           uint32_t split)
{
    uint16_t *c = C + (size_t)m * ldc + n;
    if (epi == GEMM_PLAIN)
        *c = f2h(v);
    else if (epi == GEMM_SILU_HI)
        *c = f2h(n >= split ? silu(v) : v);
    else
        *c = f2h(h2f(*c) + h2f(f2h(v)));
}

// products of interleaved up and gate columns
__host__ __device__ constexpr bool is_dual(int epi)
{
    return epi == GEMM_SWIGLU || epi == GEMM_FFN;
}

// Dual products: product column c is up row 16 (c / 32) + c % 16 when (c / 16) is even, else the gate row of that
// number, so both values of an output lie in one 32-column MFMA block, 16 lanes apart; the output column of up column c
// is 16 (c / 32) + c % 16
template <int EPI> __device__ __forceinline__ uint16_t dual_out(float up, float gate)
{
    return EPI == GEMM_FFN ? ffn_out(up, gate) : swiglu_out(up, gate);
}
__device__ __forceinline__ uint32_t swiglu_col(uint32_t c)
{
    return 16 * (c / 32) + c % 16;
}

// GEMM_QKV_ROPE: 8 consecutive product columns from `a` (a multiple of 8) of row m, as fp16: four RoPE pairs of q
// or k rotated and stored, or v stored, as one 16-byte vector each. rope_load8 fetches the pairs' (cos, sin).
struct Rope8
{
    float4 lo, hi;
};
__device__ __forceinline__ Rope8 rope_load8(const GemmRope &r, uint32_t m, uint32_t a)
{
    const uint32_t region = (a >= r.D) + (a >= 2 * r.D), dim = (a - region * r.D) & (r.hd - 1); // hd: a power of two
    const float4 *cs = (const float4 *)(r.cs + (size_t)m * r.hd + dim);
    return {cs[0], cs[1]};
}
__device__ __forceinline__ void rope_store8(const GemmRope &r, uint32_t m, uint32_t a, u32x4 v, const Rope8 &cs)
{
    const uint32_t region = (a >= r.D) + (a >= 2 * r.D), c = a - region * r.D;
    const uint32_t head = c >> (31 - __clz((int)r.hd)), dim = c & (r.hd - 1);
    const size_t cache = ((size_t)head * r.ctx + r.offset + m) * r.hd + dim;
    if (region == 2)
    {
        *(u32x4 *)(r.vc + cache) = v;
        return;
    }
    const float f[8] = {cs.lo.x, cs.lo.y, cs.lo.z, cs.lo.w, cs.hi.x, cs.hi.y, cs.hi.z, cs.hi.w};
    u32x4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        const float x0 = half_lo(v[k]), x1 = half_hi(v[k]), co = f[2 * k], sn = f[2 * k + 1];
        o[k] = pack2(f2h(rope_mul_sub(co, x0, sn, x1)), f2h(rope_mul_add(sn, x0, co, x1)));
    }
    *(u32x4 *)(region == 0 ? r.q + (size_t)m * r.D + c : r.kc + cache) = o;
}
// fp16(r + v) of 8 columns
__device__ __forceinline__ u32x4 resid8(u32x4 r, u32x4 v)
{
#pragma unroll
    for (int k = 0; k < 4; ++k)
        v[k] = pack2(f2h(half_lo(r[k]) + half_lo(v[k])), f2h(half_hi(r[k]) + half_hi(v[k])));
    return v;
}

// SPLIT: workgroup z of gridDim.y covers K columns [z * kchunk, min(K, (z + 1) * kchunk)) and writes its fp32 tile
// to work[z][M][N] instead of C
template <int BM, int BN, int EPI, bool SPLIT>
__global__ __launch_bounds__(256) void gemm_kernel(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                                                   uint16_t *C, float *work, uint32_t M, uint32_t N, uint32_t K,
                                                   uint32_t ldc, uint32_t split, uint32_t kchunk, uint32_t tiles_m,
                                                   uint32_t tiles_total)
{
    constexpr int TM = BM / 32, TN = BN / 32;            // 16x16 blocks per wave
    constexpr int AV = BM * kBK / 8 / 256, BV = BN * kBK / 8 / 256; // 16-byte vectors per thread per K step
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    // buffer b of A at lds[b BM rows], of B after both A buffers
    auto As = [&](int b) { return lds + b * BM * kLdsRow; };
    auto Bs = [&](int b) { return lds + 2 * BM * kLdsRow + b * BN * kLdsRow; };

    const uint32_t per_xcd = gridDim.x / 8;
    const uint32_t t = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (t >= tiles_total)
        return;
    const uint32_t m0 = (t % tiles_m) * BM, n0 = (t / tiles_m) * BN;
    const uint32_t kb = SPLIT ? blockIdx.y * kchunk : 0;
    const uint32_t ke = SPLIT ? min(K, kb + kchunk) : K;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const uint32_t wm = wid >> 1, wn = wid & 1;

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // rows past M or N only feed outputs that are never stored; columns past the K range are zeroed
    u32x4 ra[AV], rb[BV];
    auto load = [&](uint32_t k0) {
#pragma unroll
        for (int i = 0; i < AV; ++i)
        {
            const uint32_t v = tid + 256 * i, row = min(m0 + v / 8, M - 1), kk = k0 + (v % 8) * 8;
            const u32x4 x = *(const u32x4 *)(A + (size_t)row * K + min(kk, K - 8));
            ra[i] = kk < ke ? x : (u32x4){0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < BV; ++i)
        {
            const uint32_t v = tid + 256 * i, row = min(n0 + v / 8, N - 1), kk = k0 + (v % 8) * 8;
            const u32x4 x = __builtin_nontemporal_load((const u32x4 *)(B + (size_t)row * K + min(kk, K - 8)));
            rb[i] = kk < ke ? x : (u32x4){0, 0, 0, 0};
        }
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int i = 0; i < AV; ++i)
        {
            const uint32_t v = tid + 256 * i;
            *(u32x4 *)(As(buf) + (v / 8) * kLdsRow + (v % 8) * 8) = ra[i];
        }
#pragma unroll
        for (int i = 0; i < BV; ++i)
        {
            const uint32_t v = tid + 256 * i;
            *(u32x4 *)(Bs(buf) + (v / 8) * kLdsRow + (v % 8) * 8) = rb[i];
        }
    };

    load(kb);
    stash(0);
    __syncthreads();
    int cur = 0;
    for (uint32_t k0 = kb; k0 < ke; k0 += kBK)
    {
        const bool more = k0 + kBK < ke;
        if (more)
            load(k0 + kBK);
#pragma unroll
        for (int kk = 0; kk < kBK; kk += 32)
        {
            f16x8 af[TM], bf[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
                af[i] = *(const f16x8 *)(As(cur) + (wm * (BM / 2) + i * 16 + lane % 16) * kLdsRow + kk +
                                         (lane / 16) * 8);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                bf[j] = *(const f16x8 *)(Bs(cur) + (wn * (BN / 2) + j * 16 + lane % 16) * kLdsRow + kk +
                                         (lane / 16) * 8);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
        if (more)
            stash(cur ^ 1);
        __syncthreads();
        cur ^= 1;
    }

    // lane holds C[4*(lane/16) + e][lane % 16] of each 16x16 block
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
            {
                const uint32_t m = m0 + wm * (BM / 2) + i * 16 + 4 * (lane / 16) + e;
                const uint32_t n = n0 + wn * (BN / 2) + j * 16 + lane % 16;
                if (m >= M || n >= N)
                    continue;
                if (SPLIT)
                    work[((size_t)blockIdx.y * M + m) * N + n] = acc[i][j][e];
                else
                    gemm_store(EPI, C, ldc, m, n, acc[i][j][e], split);
            }
}

// The same product on v_mfma_f32_32x32x16_f16, pipelined by hand: 4 waves as 2 x 2 of (BM/2) x (BN/2), each a grid of
// 32x32 MFMA blocks (up to 4 x 4: 256 fp32 accumulators per lane, so one wave per SIMD and nothing else to hide
// latency behind). Operands: lane l holds row (l % 32) of a 32-row block at K offset 8 (l / 32) of each 16-wide K slice;
// the block's accumulator element e of lane l is C[8 (e / 4) + 4 (l / 32) + e % 4][l % 32].
//
// Memory side. global_load_lds copies the operands into LDS without passing registers, 8 rows of 128 bytes (64 of K:
// whole cache lines) per instruction; the 16-byte chunks of a row are placed XORed by the row's low bits, which makes
// the operand reads of 8 lanes fall on distinct banks without padding the copies could not write. 64 of K arrive as two
// halves, half h being the rows of the waves with wm == h and wn == h, through a ring of NH halves (5 of 32 KB for
// 256 x 256 tiles: all of a CU's LDS). In step s (32 of K) every wave issues its share of half s + NH - 1.
//
// Compute side. A step's MFMAs run on operands read from LDS one step earlier (two register sets of two 16-wide slices),
// so neither LDS latency nor the barrier's skew reaches the matrix pipe; the next step's operand reads and the copies
// are threaded between the MFMAs, in the order written (sched_barrier pins it). Only every second step ends in a wait
// for copies and a barrier: a half's slot is written again no earlier than the step after the barrier that follows its
// last read, and before that barrier each wave has waited for its own copies of the two halves read next.
// The copies are written in assembly because the compiler would put a wait for all of them before every LDS read; they
// have no register results, and the waits for them are the ones written here.
//
// What bounds it: L2 to LDS copies at ~68 bytes/ns of a CU for tiles below 256 x 256, and for whole-chip products the
// matrix pipes at the clock the chip sustains (with copies and LDS reads switched off a 2048 x 15360 x 5120 product
// takes 219 us, without the copies 232, whole 271). Before (operands staged through registers, 144-byte LDS rows, one
// wait per slice) and now, us: 1024 x 12288 x 4096 127 / 92 (1.11 PFLOP/s), 2048 x 15360 x 5120 323 / 271-298,
// 2048 x 5120 x 13824 346 / 257, 1024 x 4096 x 4096 47 / 36, 301 x 12288 x 4096 74 / 46.
typedef float f32x16 __attribute__((ext_vector_type(16)));

// f(integral_constant<int, J>) for J in the sequence, in order
template <int... J, typename F>
__host__ __device__ __forceinline__ void for_seq(std::integer_sequence<int, J...>, F &&f)
{
    (f(std::integral_constant<int, J>{}), ...);
}

// NH: halves in the LDS ring. WIDE: rows of any length, a tile's rows by 64-bit offsets (otherwise K <= kGemm32MaxK). Dual
// products read their columns from the up rows B and the gate rows B2 as interleaved 16-row blocks and `split` holds F.
template <int BM, int BN, int NH, int EPI, bool SPLIT, bool WIDE = false>
__global__ __launch_bounds__(256, 1) void gemm32_kernel(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                                                        const uint16_t *__restrict__ B2, uint16_t *C, float *work,
                                                        uint32_t M, uint32_t N, uint32_t K, uint32_t ldc,
                                                        uint32_t split, uint32_t kchunk, uint32_t tiles_m,
                                                        uint32_t tiles_total, GemmRope rope)
{
    constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 32, TN = WN / 32;
    constexpr int HALF = (BM + BN) * 64; // bytes of a half
    constexpr int ND = (BM + BN) / 64, NAI = WM / 32; // copies of a wave per half, the first NAI of them rows of A
    constexpr int NR = 2 * (TM + TN), NM = 2 * TM * TN; // operand reads and MFMAs of a step
    static_assert(WM % 32 == 0 && WN % 32 == 0 && NH >= 5, "whole MFMA blocks, and the waits below");
    extern __shared__ __attribute__((aligned(1024))) uint16_t lds[];

    const uint32_t per_xcd = gridDim.x / 8;
    const uint32_t t = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (t >= tiles_total)
        return;
    const uint32_t m0 = (t % tiles_m) * BM, n0 = (t / tiles_m) * BN;
    const uint32_t kb = SPLIT ? blockIdx.y * kchunk : 0;
    const uint32_t ke = SPLIT ? min(K, kb + kchunk) : K;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wid >> 1, wn = wid & 1;

    // Copy i of a wave and half h fills the half's LDS rows 8 (wid + 4 i) .. + 7 (WM rows of A, then WN of B), lane l
    // row l / 8, chunk position l % 8. Rows past M or N repeat the last one: they only feed outputs that are not
    // stored. Every K step lies wholly inside [kb, ke) (the launcher admits whole 64-wide steps).
    const uint32_t n_first = is_dual(EPI) ? n0 / 2 : n0; // first row of B (and B2)
    const uint32_t n_last = is_dual(EPI) ? split - 1 : N - 1;
    const char *const Ap = (const char *)(A + (size_t)m0 * K + kb);
    // dual products: waves 0 and 1 copy the up rows of each block, waves 2 and 3 its gate rows
    const char *const Bp = (const char *)((is_dual(EPI) && wid >= 2 ? B2 : B) + (size_t)n_first * K + kb);
    using Off = std::conditional_t<WIDE, uint64_t, uint32_t>;
    Off voff[2][ND]; // byte offsets from those
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < ND; ++i)
        {
            const uint32_t r = 8 * wid + lane / 8; // the row in its block of 32
            const int blk = i < NAI ? i + h * TM : i - NAI + h * TN;
            const uint32_t row = i < NAI ? min(32 * blk + r, M - 1 - m0)
                                         : min(is_dual(EPI) ? 16 * blk + r % 16 : 32 * blk + r, n_last - n_first);
            voff[h][i] = (Off)row * K * 2 + ((lane ^ (r & 7)) & 7) * 16;
        }
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t *)lds + wid * 1024;
    const uint32_t nsteps = (ke - kb) / 32; // and halves
    // ENDS: the half may lie past the end, and is then copied by no lane (EXEC 0; every lane is active here): it moves
    // nothing and still counts, so the waits below stay constant. Copying the last K over and over in its place took
    // 2048 x 16384 x 256 from 39 to 47 us; the steps whose halves all exist leave the test out (0.9% of long products).
    auto copy = [&](auto h_tag, auto ends_tag, int i, uint32_t slot, uint32_t half) {
        constexpr int H = decltype(h_tag)::value;
        const char *base = (i < NAI ? Ap : Bp) + half / 2 * 128;
        const uint32_t to = lds_base + slot + i * 4096, end = nsteps;
        const Off off = voff[H][i];
        if constexpr (WIDE)
            asm volatile("s_mov_b32 m0, %0\n\ts_cmp_lt_u32 %2, %3\n\ts_cselect_b64 exec, -1, 0\n\t"
                         "global_load_lds_dwordx4 %1, off\n\ts_mov_b64 exec, -1" ::"s"(to),
                         "v"(base + off), "s"(half), "s"(end)
                         : "m0", "scc");
        else if constexpr (decltype(ends_tag)::value)
            asm volatile("s_mov_b32 m0, %0\n\ts_cmp_lt_u32 %3, %4\n\ts_cselect_b64 exec, -1, 0\n\t"
                         "global_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1" ::"s"(to),
                         "v"(off), "s"(base), "s"(half), "s"(end)
                         : "m0", "scc");
        else
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(off), "s"(base)
                         : "m0");
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                acc[i][j][e] = 0.f;

    f16x8 fr[2][2][TM + TN]; // [register set][slice]: A blocks, then B blocks
    const uint32_t rl = lane % 32, at = rl * 128 + (((lane / 32) ^ (rl & 7)) * 16);
    uint32_t slot_a = wm * HALF, slot_b = wn * HALF + WM * 128; // this wave's rows of the 64 of K being read
    // operand x of slice sl of the step with K offset 32 p in its 64
    auto read = [&](auto set_tag, int sl, int x, int p) {
        constexpr int S = decltype(set_tag)::value;
        const uint32_t o = at ^ (64 * p + 32 * sl);
        const char *q = (const char *)lds + (x < TM ? slot_a + o + x * 4096 : slot_b + o + (x - TM) * 4096);
        fr[S][sl][x] = *(const f16x8 *)q;
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    // One step: the MFMAs of register set S, the reads of the next step (K offset 32 P) into the other set, and this
    // wave's copies of a half with parity H into `slot`
    auto step = [&](auto s_tag, auto p_tag, auto h_tag, auto ends_tag, uint32_t slot, uint32_t half) {
        constexpr int S = decltype(s_tag)::value;
        using Other = std::integral_constant<int, 1 - S>;
        int nr = 0, nd = 0;
#pragma unroll
        for (int k = 0; k < NM; ++k)
        {
            const int sl = k / (TM * TN), i = k % (TM * TN) / TN, j = k % TN;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[S][sl][i], fr[S][sl][TM + j], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            // all issued by 7/8 of the step
            const int want_r = min(NR, (k + 1) * NR * 8 / (NM * 7)), want_d = min(ND, (k + 1) * ND * 8 / (NM * 7));
#pragma unroll
            for (; nr < want_r; ++nr)
                read(Other{}, nr / (TM + TN), nr % (TM + TN), decltype(p_tag)::value);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (; nd < want_d; ++nd)
                copy(h_tag, ends_tag, nd, slot, half);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (; nr < NR; ++nr)
            read(Other{}, nr / (TM + TN), nr % (TM + TN), decltype(p_tag)::value);
#pragma unroll
        for (; nd < ND; ++nd)
            copy(h_tag, ends_tag, nd, slot, half);
    };
    auto next_slot = [&](uint32_t o, uint32_t by) { return o + by >= NH * HALF ? o + by - NH * HALF : o + by; };

    for_seq(std::make_integer_sequence<int, NH - 1>{}, [&](auto j) {
        constexpr int J = decltype(j)::value;
#pragma unroll
        for (int i = 0; i < ND; ++i)
            copy(std::integral_constant<int, J % 2>{}, std::true_type{}, i, J * HALF, J);
    });
    // halves 0 and 1 have landed in every wave
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NH - 3) * ND) : "memory");
#pragma unroll
    for (int x = 0; x < NR; ++x)
        read(I0{}, x / (TM + TN), x % (TM + TN), 0);
    uint32_t slot = (NH - 1) * HALF;
    auto pair = [&](auto ends_tag, uint32_t s) {
        step(I0{}, I1{}, std::integral_constant<int, (NH - 1) % 2>{}, ends_tag, slot, s + NH - 1);
        slot = next_slot(slot, HALF);
        // of the halves requested so far all but the last NH - 4 have landed, halves s + 2 and s + 3 among them, and
        // every wave has read all of halves s and s + 1
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NH - 4) * ND) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        slot_a = next_slot(slot_a, 2 * HALF);
        slot_b = next_slot(slot_b - WM * 128, 2 * HALF) + WM * 128;
        step(I1{}, I0{}, std::integral_constant<int, NH % 2>{}, ends_tag, slot, s + NH);
        slot = next_slot(slot, HALF);
    };
    uint32_t s = 0;
    for (; s + NH < nsteps; s += 2)
        pair(std::false_type{}, s);
    for (; s < nsteps; s += 2)
        pair(std::true_type{}, s);
    // nothing is in flight when the ring is used again
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

    if constexpr (!SPLIT)
    {
        // Epilogue through LDS (the ring is free now): each lane writes its fp16 outputs into a row-major
        // tile, then the workgroup moves 16-byte row chunks to their destinations, so the stores (and the residual's
        // loads) are whole vectors instead of one 2-byte element per lane. SwiGLU tiles have BN / 2 output columns.
        constexpr int OC = is_dual(EPI) ? BN / 2 : BN;
        constexpr int TROW = OC + 8; // halves; rows 4 apart then start 16 banks apart
        static_assert(BM * TROW * 2 <= NH * HALF, "epilogue tile fits the ring");
        uint16_t *T = lds;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; e += is_dual(EPI) ? 2 : 1)
                {
                    const uint32_t rt = wm * WM + i * 32 + 8 * (e / 4) + 4 * (lane / 32) + e % 4;
                    const uint32_t ct = wn * WN + j * 32 + lane % 32;
                    if constexpr (is_dual(EPI))
                    {
                        // Lanes 0-15 of each 32 hold up values and 16-31 the gate values of the same columns. Swapping
                        // rows of 16 lanes between elements e and e + 1 leaves both values of element e in the first 16
                        // and of e + 1 in the others, so every lane forms one output.
                        const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[i][j][e]),
                                                                        __float_as_uint(acc[i][j][e + 1]), false, false);
                        T[(rt + lane / 16 % 2) * TROW + swiglu_col(ct & ~16u)] =
                            dual_out<EPI>(__uint_as_float(p[0]), __uint_as_float(p[1]));
                    }
                    else if constexpr (EPI == GEMM_SILU_HI)
                        T[rt * TROW + ct] = f2h(n0 + ct >= split ? silu(acc[i][j][e]) : acc[i][j][e]);
                    else
                        T[rt * TROW + ct] = f2h(acc[i][j][e]);
                }
        __syncthreads();
        constexpr int CH = OC / 8;
        const uint32_t oc0 = is_dual(EPI) ? n0 / 2 : n0; // output column of tile column 0
        const uint32_t oce = is_dual(EPI) ? split : N; // end of the output's columns
        const bool vec = ((uintptr_t)C % 16 == 0) && ldc % 8 == 0;
        if (vec && oc0 + OC <= oce)
        {
            // Whole chunks: in batches whose loads (residuals, rotation angles) are requested together, since with one
            // workgroup on the CU each would otherwise cost its full latency. Rows past M repeat the last one.
            constexpr int IT = BM * CH / 256;
            constexpr int U = IT % 8 == 0 ? 8 : IT % 6 == 0 ? 6 : IT % 5 == 0 ? 5 : IT % 4 == 0 ? 4 : IT % 3 == 0 ? 3 : 2;
            static_assert(BM * CH % 256 == 0 && IT % U == 0, "whole batches");
            for (int it = 0; it < IT; it += U)
            {
                u32x4 old[U];
                Rope8 cs[U];
#pragma unroll
                for (int u = 0; u < U; ++u)
                {
                    const uint32_t idx = tid + 256 * (it + u), m = min(m0 + idx / CH, M - 1), col = oc0 + (idx % CH) * 8;
                    if constexpr (EPI == GEMM_QKV_ROPE)
                        cs[u] = rope_load8(rope, m, col);
                    if constexpr (EPI == GEMM_RESID)
                        old[u] = *(const u32x4 *)(C + (size_t)m * ldc + col);
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
                {
                    const uint32_t idx = tid + 256 * (it + u), m = m0 + idx / CH, col = oc0 + (idx % CH) * 8;
                    u32x4 v = *(const u32x4 *)(T + (idx / CH) * TROW + (idx % CH) * 8);
                    if constexpr (EPI == GEMM_RESID)
                        v = resid8(old[u], v);
                    if (m >= M)
                        continue;
                    if constexpr (EPI == GEMM_QKV_ROPE)
                        rope_store8(rope, m, col, v, cs[u]);
                    else
                        *(u32x4 *)(C + (size_t)m * ldc + col) = v;
                }
            }
            return;
        }
        for (uint32_t idx = tid; idx < (uint32_t)(BM * CH); idx += 256)
        {
            const uint32_t rt = idx / CH, m = m0 + rt, col = oc0 + (idx % CH) * 8;
            if (m >= M || col >= oce)
                continue;
            const uint16_t *t = T + rt * TROW + (idx % CH) * 8;
            if constexpr (EPI == GEMM_QKV_ROPE)
                rope_store8(rope, m, col, *(const u32x4 *)t, rope_load8(rope, m, col)); // N % 64 == 0: whole chunks
            else
            {
                uint16_t *c = C + (size_t)m * ldc + col;
                const uint32_t cnt = min(8u, oce - col);
                if (vec && cnt == 8)
                    *(u32x4 *)c = EPI == GEMM_RESID ? resid8(*(const u32x4 *)c, *(const u32x4 *)t) : *(const u32x4 *)t;
                else
                    for (uint32_t k = 0; k < cnt; ++k)
                        c[k] = EPI == GEMM_RESID ? f2h(h2f(c[k]) + h2f(t[k])) : t[k];
            }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
            {
                const uint32_t m = m0 + wm * WM + i * 32 + 8 * (e / 4) + 4 * (lane / 32) + e % 4;
                const uint32_t n = n0 + wn * WN + j * 32 + lane % 32;
                if (m < M && n < N)
                    work[((size_t)blockIdx.y * M + m) * N + n] = acc[i][j][e];
            }
}

// whether the plain, SiLU and residual epilogues of the split-K reduce can move 8 columns as one 16-byte vector
__host__ __device__ __forceinline__ bool reduce_vec8(uint32_t N, uint32_t ldc, const uint16_t *C)
{
    return N % 8 == 0 && ldc % 8 == 0 && (uintptr_t)C % 16 == 0;
}

// C = epilogue(sum over z of work[z]) for split-K products, the splits added in order
template <int EPI>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const float *work, uint16_t *C, uint32_t M,
                                                                 uint32_t N, uint32_t ldc, uint32_t split,
                                                                 uint32_t splits, GemmRope rope)
{
    const uint64_t total = (uint64_t)M * N;
    // 8 consecutive columns per step (N % 64 == 0 for these epilogues): 16-byte partial loads and output stores
    auto sum8 = [&](size_t at, float *v) {
#pragma unroll
        for (int k = 0; k < 8; ++k)
            v[k] = 0.f;
        for (uint32_t z = 0; z < splits; ++z)
        {
            const float4 *p = (const float4 *)(work + (size_t)z * total + at);
            const float4 a = p[0], b = p[1];
            v[0] += a.x;
            v[1] += a.y;
            v[2] += a.z;
            v[3] += a.w;
            v[4] += b.x;
            v[5] += b.y;
            v[6] += b.z;
            v[7] += b.w;
        }
    };
    if constexpr (EPI == GEMM_QKV_ROPE)
    {
        const uint32_t per_row = N / 8;
        const uint64_t chunks = (uint64_t)M * per_row;
        for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < chunks; i += (uint64_t)gridDim.x * 256)
        {
            const uint32_t m = (uint32_t)(i / per_row), n = 8 * (uint32_t)(i % per_row);
            float v[8];
            sum8((size_t)m * N + n, v);
            u32x4 h;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                h[k] = pack2(f2h(v[2 * k]), f2h(v[2 * k + 1]));
            rope_store8(rope, m, n, h, rope_load8(rope, m, n));
        }
        return;
    }
    if constexpr (is_dual(EPI))
    {
        // 8 output columns f..f + 7 (inside one 16-column block): up columns c..c + 7, gate columns c + 16..c + 23
        const uint32_t per_row = N / 16;
        const uint64_t chunks = (uint64_t)M * per_row;
        for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < chunks; i += (uint64_t)gridDim.x * 256)
        {
            const uint32_t m = (uint32_t)(i / per_row), f = 8 * (uint32_t)(i % per_row), c = 32 * (f / 16) + f % 16;
            if (f >= split) // columns past F (GEMM_FFN with F % 32 != 0)
                continue;
            float up[8], gate[8];
            sum8((size_t)m * N + c, up);
            sum8((size_t)m * N + c + 16, gate);
            u32x4 o;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                o[k] = pack2(dual_out<EPI>(up[2 * k], gate[2 * k]), dual_out<EPI>(up[2 * k + 1], gate[2 * k + 1]));
            *(u32x4 *)(C + (size_t)m * ldc + swiglu_col(c)) = o;
        }
        return;
    }
    if (reduce_vec8(N, ldc, C))
    {
        // 8 consecutive columns per step: 16-byte partial loads and one 16-byte store (the same sums, in the same
        // split order, as the element loop below)
        const uint32_t per_row = N / 8;
        const uint64_t chunks = (uint64_t)M * per_row;
        for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < chunks; i += (uint64_t)gridDim.x * 256)
        {
            const uint32_t m = (uint32_t)(i / per_row), n = 8 * (uint32_t)(i % per_row);
            float v[8];
            sum8((size_t)m * N + n, v);
            uint16_t *c = C + (size_t)m * ldc + n;
            u32x4 o;
            if constexpr (EPI == GEMM_RESID)
            {
                const u32x4 old = *(const u32x4 *)c;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    o[k] = pack2(f2h(half_lo(old[k]) + h2f(f2h(v[2 * k]))),
                                 f2h(half_hi(old[k]) + h2f(f2h(v[2 * k + 1]))));
            }
            else
            {
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (EPI == GEMM_SILU_HI && n + k >= split)
                        v[k] = silu(v[k]);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    o[k] = pack2(f2h(v[2 * k]), f2h(v[2 * k + 1]));
            }
            *(u32x4 *)c = o;
        }
        return;
    }
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (uint64_t)gridDim.x * 256)
    {
        float v = 0.f;
        for (uint32_t z = 0; z < splits; ++z)
            v += work[(size_t)z * total + i];
        gemm_store(EPI, C, ldc, (uint32_t)(i / N), (uint32_t)(i % N), v, split);
    }
}

// work items of gemm_splitk_reduce_kernel: 8 columns each where the epilogue or reduce_vec8 allows, else one element
template <int EPI>
static uint32_t reduce_grid(uint32_t M, uint32_t N, uint32_t ldc, const uint16_t *C)
{
    uint64_t items = (uint64_t)M * N;
    if (is_dual(EPI))
        items /= 16;
    else if (EPI == GEMM_QKV_ROPE || reduce_vec8(N, ldc, C))
        items /= 8;
    const uint64_t grid = (items + 255) / 256;
    return (uint32_t)(grid > 4096 ? 4096 : grid < 1 ? 1 : grid);
}

// Split-K residual products followed by RMSNorm (every residual product of the token step is): one workgroup per
// row m, C[m] = fp16(C[m] + fp16(sum over z of work[z][m])) with the splits added in order (as the reduce kernel),
// then y[m] = RMSNorm(C[m]) * w as rmsnorm_row_to computes it, with launch_rmsnorm_rows's block size (so the same
// sum order). Each thread re-reads only the vectors it wrote.
__global__ __launch_bounds__(512) void gemm_resid_norm_kernel(const float *work, uint16_t *C, uint32_t M, uint32_t N,
                                                              uint32_t splits, const float *w, uint16_t *y,
                                                              float eps, bool xt)
{
    __shared__ float red[8];
    const uint32_t m = blockIdx.x, nv = N / 8;
    const size_t total = (size_t)M * N;
    u32x4 *cv = (u32x4 *)(C + (size_t)m * N);
    for (uint32_t i = threadIdx.x; i < nv; i += blockDim.x)
    {
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
        for (uint32_t z = 0; z < splits; ++z)
        {
            const float4 *p = (const float4 *)(work + z * total + (size_t)m * N + 8 * i);
            const float4 a = p[0], b = p[1];
            acc[0] += a.x;
            acc[1] += a.y;
            acc[2] += a.z;
            acc[3] += a.w;
            acc[4] += b.x;
            acc[5] += b.y;
            acc[6] += b.z;
            acc[7] += b.w;
        }
        const u32x4 r = cv[i];
        u32x4 o;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            o[k] = pack2(f2h(half_lo(r[k]) + h2f(f2h(acc[2 * k]))), f2h(half_hi(r[k]) + h2f(f2h(acc[2 * k + 1]))));
        cv[i] = o;
    }
    if (xt)
        rmsnorm_row_to(C + (size_t)m * N, w, (u32x4 *)y, N, eps, red, (int)m);
    else
        rmsnorm_row_to(C + (size_t)m * N, w, (u32x4 *)(y + (size_t)m * N), N, eps, red);
}

// gemm_resid_norm_kernel for rows of at most 512 VPT vectors: each thread keeps its vectors in registers from the
// partial sums to the normalised output, and requests the residual and norm weights with the partials, so the row
// makes one round trip to memory instead of three. The sums run in the same order (a thread's vectors ascending,
// the same block_sum), so the outputs equal the generic kernel's bit for bit.
template <int VPT>
__global__ __launch_bounds__(512) void gemm_resid_norm_regs_kernel(const float *work, uint16_t *C, uint32_t M,
                                                                   uint32_t N, uint32_t splits, const float *w,
                                                                   uint16_t *y, float eps, bool xt)
{
    __shared__ float red[8];
    const uint32_t m = blockIdx.x, nv = N / 8, tid = threadIdx.x;
    const size_t total = (size_t)M * N;
    u32x4 *cv = (u32x4 *)(C + (size_t)m * N);
    const float4 *wv = (const float4 *)w;
    // unconditional loads at clamped indices (a guarded load compiles to a branch and a wait per load)
    u32x4 r[VPT];
    float4 wa[VPT], wb[VPT];
#pragma unroll
    for (int j = 0; j < VPT; ++j)
    {
        const uint32_t i = min(tid + 512 * j, nv - 1);
        r[j] = cv[i];
        wa[j] = wv[2 * i];
        wb[j] = wv[2 * i + 1];
    }
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j)
    {
        const uint32_t i = tid + 512 * j;
        const uint32_t ic = min(i, nv - 1);
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
        for (uint32_t z = 0; z < splits; ++z)
        {
            const float4 *p = (const float4 *)(work + z * total + (size_t)m * N + 8 * ic);
            const float4 a = p[0], b = p[1];
            acc[0] += a.x;
            acc[1] += a.y;
            acc[2] += a.z;
            acc[3] += a.w;
            acc[4] += b.x;
            acc[5] += b.y;
            acc[6] += b.z;
            acc[7] += b.w;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            r[j][k] = pack2(f2h(half_lo(r[j][k]) + h2f(f2h(acc[2 * k]))),
                            f2h(half_hi(r[j][k]) + h2f(f2h(acc[2 * k + 1]))));
        if (i < nv)
        {
            cv[i] = r[j];
#pragma unroll
            for (int k = 0; k < 4; ++k)
            {
                const float a = half_lo(r[j][k]), b = half_hi(r[j][k]);
                ss += a * a;
                ss += b * b;
            }
        }
    }
    ss = block_sum(ss, red);
    const float alpha = 1.0f / sqrtf(ss / (float)N + eps);
#pragma unroll
    for (int j = 0; j < VPT; ++j)
    {
        const uint32_t i = tid + 512 * j;
        if (i >= nv)
            continue;
        const float ws[8] = {wa[j].x, wa[j].y, wa[j].z, wa[j].w, wb[j].x, wb[j].y, wb[j].z, wb[j].w};
        u32x4 o;
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            const float a = half_lo(r[j][k]), b = half_hi(r[j][k]);
            o[k] = pack2(f2h((a * ws[2 * k]) * alpha), f2h((b * ws[2 * k + 1]) * alpha));
        }
        ((u32x4 *)y)[xt ? xt_vec(m, i) : (size_t)m * nv + i] = o;
    }
}

// the residual-norm reduce for a row of N columns (one 512-thread workgroup per row)
static hipError_t launch_resid_norm(hipStream_t st, const float *work, uint16_t *C, uint32_t M, uint32_t N,
                                    uint32_t splits, const GemmNorm &norm)
{
    const uint32_t nv = N / 8;
    if (nv <= 512)
        gemm_resid_norm_regs_kernel<1><<<M, 512, 0, st>>>(work, C, M, N, splits, norm.w, norm.y, norm.eps, norm.xt);
    else if (nv <= 1024)
        gemm_resid_norm_regs_kernel<2><<<M, 512, 0, st>>>(work, C, M, N, splits, norm.w, norm.y, norm.eps, norm.xt);
    else
        gemm_resid_norm_kernel<<<M, 512, 0, st>>>(work, C, M, N, splits, norm.w, norm.y, norm.eps, norm.xt);
    return hipGetLastError();
}

// the weight rows: p2 the gate rows of a dual product, whose up rows are p
struct GemmB
{
    const uint16_t *p, *p2;
};

template <int BM, int BN> static size_t gemm_lds()
{
    return (size_t)2 * (BM + BN) * kLdsRow * sizeof(uint16_t);
}

template <int BM, int BN, int EPI, bool SPLIT>
static hipError_t launch_tile(hipStream_t st, const uint16_t *A, const uint16_t *B, uint16_t *C, float *work,
                              uint32_t M, uint32_t N, uint32_t K, uint32_t ldc, uint32_t split, uint32_t splits,
                              uint32_t kchunk)
{
    static uint64_t attr_devs = 0; // devices on which the LDS limit is raised for this kernel
    const size_t lds = gemm_lds<BM, BN>();
    hipError_t e = lds_attr_once((const void *)gemm_kernel<BM, BN, EPI, SPLIT>, lds, attr_devs);
    if (e != hipSuccess)
        return e;
    const uint32_t tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN, total = tm * tn;
    const uint32_t grid = (total + 7) / 8 * 8;
    gemm_kernel<BM, BN, EPI, SPLIT><<<dim3(grid, SPLIT ? splits : 1), 256, lds, st>>>(A, B, C, work, M, N, K, ldc,
                                                                                     split, kchunk, tm, total);
    return hipGetLastError();
}

template <int BM, int BN, int NH, int EPI, bool SPLIT, bool WIDE = false>
static hipError_t launch_tile32(hipStream_t st, const uint16_t *A, GemmB B, uint16_t *C, float *work,
                                uint32_t M, uint32_t N, uint32_t K, uint32_t ldc, uint32_t split, uint32_t splits,
                                uint32_t kchunk, const GemmRope *rope = nullptr)
{
    static uint64_t attr_devs = 0; // devices on which the LDS limit is raised for this kernel
    const size_t lds = (size_t)NH * (BM + BN) * 64;
    hipError_t e = lds_attr_once((const void *)gemm32_kernel<BM, BN, NH, EPI, SPLIT, WIDE>, lds, attr_devs);
    if (e != hipSuccess)
        return e;
    const uint32_t tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN, total = tm * tn;
    const uint32_t grid = (total + 7) / 8 * 8;
    gemm32_kernel<BM, BN, NH, EPI, SPLIT, WIDE><<<dim3(grid, SPLIT ? splits : 1), 256, lds, st>>>(
        A, B.p, B.p2, C, work, M, N, K, ldc, split, kchunk, tm, total, rope ? *rope : GemmRope{});
    return hipGetLastError();
}

template <int EPI>
static hipError_t launch_reduce(hipStream_t st, const float *work, uint16_t *C, uint32_t M, uint32_t N, uint32_t ldc,
                                uint32_t split, uint32_t splits, const GemmRope *rope)
{
    const uint32_t grid = reduce_grid<EPI>(M, N, ldc, C);
    gemm_splitk_reduce_kernel<EPI>
        <<<grid, 256, 0, st>>>(work, C, M, N, ldc, split, splits, rope ? *rope : GemmRope{});
    return hipGetLastError();
}

template <int BM, int BN, int EPI>
static hipError_t launch_shape(hipStream_t st, const uint16_t *A, const uint16_t *B, uint16_t *C, float *work,
                               uint32_t M, uint32_t N, uint32_t K, uint32_t ldc, uint32_t split, uint32_t splits,
                               uint32_t kchunk)
{
    if (splits <= 1)
        return launch_tile<BM, BN, EPI, false>(st, A, B, C, work, M, N, K, ldc, split, 1, K);
    hipError_t e = launch_tile<BM, BN, EPI, true>(st, A, B, C, work, M, N, K, ldc, split, splits, kchunk);
    if (e != hipSuccess)
        return e;
    const uint32_t grid = reduce_grid<EPI>(M, N, ldc, C);
    gemm_splitk_reduce_kernel<EPI><<<grid, 256, 0, st>>>(work, C, M, N, ldc, split, splits, GemmRope{});
    return hipGetLastError();
}

// ---- tile and split of a product ----
struct TileShape
{
    uint16_t bm, bn;
    // halves in the LDS ring (as many as fit 160 KB, up to 10, but for the last tile), workgroups that fit a CU with it
    uint8_t ring, per_cu;
    float step_us; // 64 of K on one of many busy CUs, measured (products of 64 to 216 such steps in one round)
};
constexpr TileShape kTiles[] = {{256, 256, 5, 1, 1.29f}, {256, 192, 5, 1, 1.18f}, {256, 128, 6, 1, 0.88f},
                                {128, 320, 5, 1, 1.18f}, {320, 128, 5, 1, 1.05f}, {192, 128, 8, 1, 0.66f},
                                {128, 128, 10, 1, 0.50f}, {64, 128, 10, 1, 0.36f}, {128, 128, 5, 2, 0.50f}};
// Products of short rows are their workgroups' starts and epilogues. With K of at most kShortK the 128 x 128 tile takes
// a ring of 5, so that two workgroups of a CU cover each other's (longer rows wait for that ring). us, ring of 10 / 5
// and the tile that was fastest without it: 2048 x 4096 x 64 10.0 / 7.4 (8.3 on 256 x 128), 2048 x 16384 x 192 39.3 /
// 26.6 (30.8), 1024 x 4096 x 128 6.5 / 5.8; K 320: 13.0 / 11.3 to 14.4 from run to run. So varies 256 x 128 up to K
// 512 (2048 x 4096 x 256 10.7 to 17.0, x 320 13.4 to 18.3), which is left out there: 320 x 128 takes 11.5 and 12.6.
constexpr uint32_t kShortK = 192, kMidK = 512;
constexpr int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);

template <int EPI, bool SPLIT>
static hipError_t launch_choice(hipStream_t st, int tile, const uint16_t *A, GemmB B, uint16_t *C, float *work, uint32_t M,
                                uint32_t N, uint32_t K, uint32_t ldc, uint32_t split, uint32_t splits, uint32_t kchunk,
                                const GemmRope *rope)
{
    hipError_t e = hipErrorInvalidValue;
    for_seq(std::make_integer_sequence<int, kTileCount>{}, [&](auto i) {
        constexpr TileShape T = kTiles[decltype(i)::value];
        if (tile == decltype(i)::value)
            e = launch_tile32<T.bm, T.bn, T.ring, EPI, SPLIT>(st, A, B, C, work, M, N, K, ldc, split, splits, kchunk, rope);
    });
    return e;
}

struct TileChoice
{
    int tile;
    uint32_t splits, kchunk; // K ranges of kchunk
};

// Time of a product on one tile shape with K in `splits` ranges, us: the tile's measured step, or what the busy CUs
// together sustain (1.3 PFLOP/s); each round of workgroups adds its start and its epilogue, split K the partials written
// and read and the reduce's launch, whole K the RMSNorm pass that the reduce would have included; and the weights come
// from HBM at 4.6 TB/s, or 24 bytes/ns of each workgroup (18 of a part of its rows). Over 73 products of 16 to 2048 rows
// at the 7B and 13B widths the choice made from it is the fastest measured one (of the eight tiles with a full ring and up
// to 8 ranges) or within 11% of it in all but 2, which are within 14%.
static float tile_time(uint32_t M, uint32_t N, uint32_t K, TileShape t, uint32_t splits, uint32_t cus, bool norm)
{
    const uint64_t wgs = (uint64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * splits;
    const uint32_t steps = (K / kBK + splits - 1) / splits;
    const float flop = 2.f * t.bm * t.bn * kBK, area = t.bm * t.bn / 65536.f;
    auto round = [&](float n) { return steps * std::max(t.step_us, n * flop / 1.3e9f) + 5.f + 5.f * area; };
    const uint64_t slots = (uint64_t)cus * t.per_cu, full = wgs / slots, rest = wgs % slots;
    float us = full * round((float)slots) + (rest ? round((float)rest) : 0.f);
    if (t.per_cu > 1 && wgs > slots) // a round's epilogues run under the next one's start
        us -= 2.8f * (full + (rest ? 1 : 0) - 1);
    // several rows of tiles share the weights through L2 at some cost; the last term: of tiles that all wait for the
    // weights, the one that is done soonest
    const float weights = (float)N * K * 2 * (M > t.bm ? 1.2f : 1.f);
    us = std::max(us, 3.f + weights / std::min(4.6e6f, (splits > 1 ? 1.8e4f : 2.4e4f) * wgs)) + 0.05f * us;
    const float mn = (float)M * N;
    if (splits > 1)
        us += 4.f + splits * mn * 4 / 3.5e6f;
    else if (norm)
        us += 4.f + mn * 4 / 3.5e6f;
    return us;
}

static TileChoice pick_tile(uint32_t M, uint32_t N, uint32_t K, uint32_t cus, size_t work_elems, bool norm)
{
    TileChoice best{0, 1, K};
    float best_us = FLT_MAX;
    for (int i = 0; i < kTileCount; ++i)
    {
        const TileShape t = kTiles[i];
        if (t.bn == 128 && ((t.bm == 128 && (t.per_cu > 1) != (K <= kShortK)) || (t.bm == 256 && K <= kMidK)))
            continue;
        for (uint32_t s = 1; s <= 8; ++s) // (more were at most 2% faster anywhere, with more partials to round)
        {
            // a range keeps at least 256 of K
            if (s > 1 && (K / s < 4 * kBK || (size_t)s * M * N > work_elems))
                break;
            const float us = tile_time(M, N, K, t, s, cus, norm);
            if (us < best_us)
            {
                best_us = us;
                best = {i, s, K};
            }
        }
    }
    if (best.splits > 1)
    {
        best.kchunk = ((K + best.splits - 1) / best.splits + kBK - 1) / kBK * kBK;
        best.splits = (K + best.kchunk - 1) / best.kchunk;
    }
    return best;
}

GemmPlan gemm_plan(uint32_t M, uint32_t N, uint32_t K, uint32_t cus, size_t work_elems, bool norm)
{
    if (K % kBK != 0 || K > kGemm32MaxK)
        return {0, 0, 0};
    const TileChoice c = pick_tile(M, N, K, cus, work_elems, norm);
    return {kTiles[c.tile].bm, kTiles[c.tile].bn, c.splits};
}

template <int EPI>
static hipError_t launch_epi_gemm(hipStream_t st, const uint16_t *A, GemmB B, uint16_t *C, float *work,
                                  size_t work_elems, uint32_t M, uint32_t N, uint32_t K, uint32_t ldc,
                                  uint32_t split, int cu_count, const GemmRope *rope, const GemmNorm *norm,
                                  bool *normed)
{
    const uint32_t cus = cu_count > 0 ? (uint32_t)cu_count : 256;
    if constexpr (EPI == GEMM_QKV_ROPE)
        if (!rope || K % kBK != 0 || K > kGemm32MaxK || rope->D % 64 != 0 || rope->hd < 32 || (rope->hd & (rope->hd - 1)) != 0 ||
            N != 3 * rope->D || !rope->cs)
            return hipErrorInvalidValue;
    // (no product past it has run: MATMUL refuses it too, the FFN operator takes its generic kernel)
    if ((uint64_t)N * K >= (1ull << 32))
        return hipErrorInvalidValue;
    if constexpr (is_dual(EPI))
        if (K % kBK != 0 || (EPI == GEMM_FFN && K > kGemm32MaxK) || N % 64 != 0 || N != (2 * split + 63) / 64 * 64 ||
            split % 8 != 0 || !B.p2 || ldc % 8 != 0 || (uintptr_t)C % 16 != 0)
            return hipErrorInvalidValue;
    if constexpr (EPI == GEMM_SWIGLU)
        if (K > kGemm32MaxK) // (fewer than 1024 rows of B: one small tile shape)
            return launch_tile32<64, 128, 10, EPI, false, true>(st, A, B, C, nullptr, M, N, K, ldc, split, 1, K);
    // (gemm32_kernel's copies address a tile's rows by 32-bit byte offsets; longer rows take gemm_kernel)
    if (K % kBK == 0 && K <= kGemm32MaxK)
    {
        const TileChoice c = pick_tile(M, N, K, cus, work_elems, EPI == GEMM_RESID && norm);
        const uint32_t kchunk = c.kchunk, splits = c.splits;
        if (splits <= 1)
            return launch_choice<EPI, false>(st, c.tile, A, B, C, nullptr, M, N, K, ldc, split, 1, K, rope);
        // the partial tiles are the same for every epilogue: one kernel for products of one matrix, one for dual ones
        constexpr int PART = is_dual(EPI) ? GEMM_SWIGLU : GEMM_PLAIN;
        hipError_t e = launch_choice<PART, true>(st, c.tile, A, B, C, work, M, N, K, ldc, split, splits, kchunk, nullptr);
        if (e != hipSuccess)
            return e;
        if constexpr (EPI == GEMM_RESID)
            if (norm)
            {
                // the reduce adds the residual and normalises the updated rows in one pass
                *normed = true;
                return launch_resid_norm(st, work, C, M, N, splits, *norm);
            }
        return launch_reduce<EPI>(st, work, C, M, N, ldc, split, splits, rope);
    }
    if constexpr (is_dual(EPI) || EPI == GEMM_QKV_ROPE)
        return hipErrorInvalidValue; // checked above: not reached
    else
    {
        if (M <= 128)
        {
            // weight-streaming regime: a 128-row tile covers all of M so each weight is read once; K is split over
            // workgroups when N is narrow
            const uint32_t tiles = (N + 63) / 64;
            uint32_t splits = 1;
            while (tiles * splits <= cus && K / (splits * 2) >= 512 && (size_t)splits * 2 * M * N <= work_elems)
                splits *= 2;
            const uint32_t kchunk = ((K + splits - 1) / splits + kBK - 1) / kBK * kBK;
            splits = (K + kchunk - 1) / kchunk;
            return launch_shape<128, 64, EPI>(st, A, B.p, C, work, M, N, K, ldc, split, splits, kchunk);
        }
        const uint64_t big = (uint64_t)((M + 127) / 128) * ((N + 127) / 128);
        if (big >= cus)
            return launch_shape<128, 128, EPI>(st, A, B.p, C, work, M, N, K, ldc, split, 1, K);
        return launch_shape<128, 64, EPI>(st, A, B.p, C, work, M, N, K, ldc, split, 1, K);
    }
}

hipError_t launch_gemm_reduce(hipStream_t st, int epi, const float *work, uint16_t *C, uint32_t M, uint32_t N,
                              uint32_t splits, const GemmRope *rope, const GemmNorm *norm)
{
    if (M == 0 || N == 0 || splits == 0)
        return hipErrorInvalidValue;
    switch (epi)
    {
    case GEMM_RESID:
        if (!norm)
            return launch_reduce<GEMM_RESID>(st, work, C, M, N, N, 0, splits, nullptr);
        if (N % 8 != 0 || (norm->xt && (M > 128 || N % 16 != 0)))
            return hipErrorInvalidValue;
        return launch_resid_norm(st, work, C, M, N, splits, *norm);
    case GEMM_QKV_ROPE:
        if (!rope || N != 3 * rope->D)
            return hipErrorInvalidValue;
        return launch_reduce<GEMM_QKV_ROPE>(st, work, C, M, N, N, 0, splits, rope);
    default:
        return hipErrorInvalidValue;
    }
}

hipError_t launch_gemm(hipStream_t st, int epi, const uint16_t *A, const uint16_t *B, uint16_t *C, uint32_t M,
                       uint32_t N, uint32_t K, uint32_t ldc, uint32_t split, int cu_count, float *work,
                       size_t work_elems, const GemmRope *rope, const GemmNorm *norm, const uint16_t *B2)
{
    if (K % 8 != 0 || K < 8 || M == 0 || N == 0)
        return hipErrorInvalidValue;
    switch (epi)
    {
    case GEMM_PLAIN:
        return launch_epi_gemm<GEMM_PLAIN>(st, A, GemmB{B, nullptr}, C, work, work_elems, M, N, K, ldc, split, cu_count, nullptr,
                                             nullptr, nullptr);
    case GEMM_SILU_HI:
        return launch_epi_gemm<GEMM_SILU_HI>(st, A, GemmB{B, nullptr}, C, work, work_elems, M, N, K, ldc, split, cu_count, nullptr,
                                             nullptr, nullptr);
    case GEMM_RESID:
    {
        if (norm && (ldc != N || N % 8 != 0))
            return hipErrorInvalidValue;
        bool normed = false;
        hipError_t e = launch_epi_gemm<GEMM_RESID>(st, A, GemmB{B, nullptr}, C, work, work_elems, M, N, K, ldc, split, cu_count,
                                                   nullptr, norm, &normed);
        if (e != hipSuccess || !norm || normed)
            return e;
        return launch_rmsnorm_rows(st, C, norm->w, norm->y, M, N, norm->eps, norm->xt);
    }
    case GEMM_SWIGLU:
        if (N != 2 * split)
            return hipErrorInvalidValue;
        return launch_epi_gemm<GEMM_SWIGLU>(st, A, GemmB{B, B + (size_t)split * K}, C, work, work_elems, M, N, K, ldc,
                                            split, cu_count, nullptr, nullptr, nullptr);
    case GEMM_FFN:
        return launch_epi_gemm<GEMM_FFN>(st, A, GemmB{B, B2}, C, work, work_elems, M, N, K, ldc, split, cu_count,
                                         nullptr, nullptr, nullptr);
    case GEMM_QKV_ROPE:
        return launch_epi_gemm<GEMM_QKV_ROPE>(st, A, GemmB{B, nullptr}, C, work, work_elems, M, N, K, ldc, split, cu_count, rope,
                                              nullptr, nullptr);
    default:
        return hipErrorInvalidValue;
    }
}

} // namespace vk
