/* MFMA GEMM on 256-row tiles: Y[N, M] = X[N, K] . W[M, K]^T, bf16 in, fp32
 * accumulate, W in the tiled layout k_gemm_small_tile writes. It is the tile
 * (4, NG) of gemm_wide.hip for NG = 8, 12 and 16, with both operands staged
 * by DMA. The reference runs these projections through cuBLAS GemmEx
 * (src/kernels/elementwise.cu:56-75).
 *
 *  - Tile 256 weight rows (gated: 128 gate rows and the same up rows) x 32 WN
 *    tokens (WN 8, 6, 4); 4 waves as 2 x 2, one per SIMD, a wave holding
 *    8 x WN accumulators of v_mfma_f32_16x16x32_bf16 (W as the A operand).
 *    At 256 x 256 a wave's 16 LDS fragment reads feed 64 MFMAs (64 of the
 *    128 B per clock a CU's LDS gives); 8 waves of half the block would need
 *    96 and the DMA writes 32 more.
 *  - K advances in units of 32. W goes HBM -> LDS by buffer_load ... lds into
 *    a ring of 4 units, X into two buffers of 64 k (a 128-byte piece of each
 *    token's row, its 16-byte pieces XOR-swizzled on the global side so that
 *    the fragment reads have no bank conflicts). No other vector memory
 *    operation is in flight in the loop, so the DMAs complete in order and a
 *    partial vmcnt wait covers them; one barrier per unit. Before it each wave
 *    also waits for its LDS reads of what the unit's DMAs overwrite, a partial
 *    lgkmcnt wait: gemm_block_order.h has the order and both counts.
 *  - The wave's own LDS reads run ahead of their MFMAs (X one unit, W three
 *    row groups), and at most one memory operation sits between two MFMAs:
 *    an MFMA leaves a wave about 3 issue slots, and reads and DMAs in bursts
 *    in front of a row of MFMAs left the matrix core idle (12288 x 2560
 *    gate|up at 10752 tokens: 755 -> 711 us with them spread).
 *  - The accumulators are tied to accumulation registers through inline asm:
 *    with the builtin the compiler copied all 256 of them once per pass of
 *    the loop. What the asm leaves to this code: no VALU result feeds an MFMA
 *    in the loop (operands come from LDS, whose waits the compiler places),
 *    the same accumulator is used again 8 WN MFMAs later, and 32 wait states
 *    separate the last MFMA from the first read of the results.
 *  - k order and k assignment per MFMA are gemm_wide's, so every tile gives
 *    the same bits.
 *  - Outputs leave through LDS as whole 16-byte pieces of a token's row, 128
 *    or 256 bytes of it at a time: 8-byte stores from the accumulators (32
 *    bytes of 16 rows per instruction) cost 5 us per round of workgroups
 *    (in_proj at 10752 tokens: 557 -> 512 us).
 *
 * What bounds it: at K = 9216 a round of 240 workgroups takes 0.62 us per
 * unit, i.e. the matrix cores 1.6 PFLOP/s-equivalent (removing the DMAs gives
 * 1.63-1.67, the LDS reads as well 2.0: the clock under load and the LDS port
 * set the rest), plus about 8 us per round for launch, first loads and the
 * epilogue, and the last round's idle CUs. Measured for 4B at 10752 tokens
 * against hipBLASLt with the nearest tuned entry (8832 tokens): in_proj 516 /
 * 525 us, gate|up + silu 722 / 787, with the residual add and norm out_proj 237
 * / 242 and down 457 / 478, but qkv 408 / 386; against entries tuned for the
 * very count see cujev_gemm_plan_loses. Against gemm_wide's former (4, 8) at 611
 * tokens: qkv 37.6 / 41.6 us, in_proj 37.8 / 41.2. */
#include <type_traits>

#include "common.h"
#include "gemm_block_order.h"
#include "kernels.h"

namespace CUJEV_KNS {
namespace {

enum { GB_PLAIN = 0, GB_GATED = 1, GB_PART = 2 };

typedef __attribute__((address_space(3))) void *lds_ptr;
typedef __attribute__((address_space(3))) const unsigned char lds_u8;

DEV __amdgpu_buffer_rsrc_t gb_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}
DEV bf16x8 gb_read(lds_u8 *base, uint32_t off) {
    return *(__attribute__((address_space(3))) const bf16x8 *)(base + off);
}

DEV void gb_mfma(floatx4 &acc, bf16x8 a, bf16x8 b) {
#ifdef __HIP_DEVICE_COMPILE__ /* "a" names another register class on the host */
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
#endif
}

/* 64 lanes x 16 bytes from the buffer to dst + 16 lane */
DEV void gb_dma(__amdgpu_buffer_rsrc_t r, unsigned char *dst, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr)dst, 16, voff, soff, 0, 0);
}

constexpr int GB_A = 256 * 64; /* bytes of a W unit: 256 rows x 32 k */

template <int VM, int LGKM> DEV void gb_wait() {
    static_assert(VM < 64 && LGKM < 16, "counter ranges");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(%1)" ::"n"(VM), "n"(LGKM) : "memory");
}

template <int WN, int MODE>
__global__ __launch_bounds__(256, 1) void gemm_block_kernel(
    const bf16 *__restrict__ X, int ldx, const bf16 *__restrict__ Wt, int N, int M, int K, int nch,
    int mblocks, int nblocks, int splits, int per_xcd, bf16 *__restrict__ Y, int ldy,
    float *__restrict__ P) {
    constexpr int BN = 32 * WN;          /* tokens per tile */
    constexpr int BB = BN * 128;         /* bytes of an X stage: BN tokens x 64 k */
    constexpr int XOFF = GB_WU * GB_A;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[GB_WU * GB_A + 2 * BB];

    const int item = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (item >= mblocks * nblocks * splits)
        return;
    /* groups of up to 8 row blocks, all token blocks of a group in turn */
    int nb, mb, sp;
    {
        const int tiles = mblocks * nblocks;
        sp = item / tiles;
        const int it = item - sp * tiles;
        const int grp = it / (8 * nblocks), m0 = grp * 8;
        const int gm = min(8, mblocks - m0), r = it - grp * 8 * nblocks;
        nb = r / gm;
        mb = m0 + r - nb * gm;
    }

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int q = lane >> 4, c16 = lane & 15;
    const int G = M >> 4;
    const int c0 = sp * nch;
    const int nu = 4 * nch; /* 32-k units */

    /* row group of LDS slot s (0..15): wave pair wm owns slots 8 wm .. +7;
     * gated: its first 4 slots are gate groups, the other 4 the up groups */
    auto group_of = [&](int s) {
        if constexpr (MODE == GB_GATED) {
            const int GI = G >> 1;
            const int g = min((mb * 2 + (s >> 3)) * 4 + (s & 3), GI - 1);
            return (s & 4) ? g + GI : g;
        } else {
            return min(mb * 16 + s, G - 1);
        }
    };
    const __amdgpu_buffer_rsrc_t wr = gb_rsrc(Wt, (uint32_t)((size_t)M * K * 2));
    const __amdgpu_buffer_rsrc_t xr = gb_rsrc(X, (uint32_t)((size_t)N * ldx * 2));
    const uint32_t wchunk = (uint32_t)G * 4096u;
    uint32_t wofs[4];
#pragma unroll
    for (int s = 0; s < 4; s++)
        wofs[s] = (uint32_t)group_of(4 * wave + s) * 4096u;
    const uint32_t wlane = (uint32_t)lane * 16u;
    /* X piece j of this wave: tokens 8 (wave WN + j) + lane/8, slot lane%8
     * holds octet slot ^ ((token / 2) % 8) of the stage's 64 k */
    uint32_t xoff[WN];
#pragma unroll
    for (int j = 0; j < WN; j++) {
        const int t = 8 * (wave * WN + j) + (lane >> 3);
        xoff[j] = (uint32_t)(nb * BN + t) * (uint32_t)ldx * 2u +
                  (uint32_t)(((lane & 7) ^ ((t >> 1) & 7)) * 16);
    }
    /* W unit u -> ring slot u % 4, this wave's row groups k = 0..3 */
    auto dma_w = [&](int u, int slot, int k) {
        const uint32_t c = (uint32_t)(c0 + (u >> 2));
        gb_dma(wr, smem + slot * GB_A + (4 * wave + k) * 1024, wlane,
               c * wchunk + wofs[k] + (uint32_t)(u & 3) * 1024u);
    };
    /* X stage p (64 k) -> buffer p % 2, this wave's piece j */
    auto dma_x = [&](int p, int buf, int j) {
        gb_dma(xr, smem + XOFF + buf * BB + (wave * WN + j) * 1024, xoff[j],
               (uint32_t)c0 * 256u + (uint32_t)p * 128u);
    };

    lds_u8 *lds = (lds_u8 *)smem;
    const uint32_t abase = (uint32_t)(wm * 8 * 1024) + wlane;
    uint32_t bbase[2];
#pragma unroll
    for (int i = 0; i < 2; i++)
        bbase[i] = XOFF + (uint32_t)(wn * WN * 16 + c16) * 128u +
                   (uint32_t)(((2 * q + i) ^ ((c16 >> 1) & 7)) * 16);
    /* fragments of unit slot s (0..3): X buffer s / 2, half s % 2 */
    auto rda = [&](int s, int r) { return gb_read(lds, abase + (uint32_t)(s * GB_A + r * 1024)); };
    auto rdb = [&](int s, int j) {
        return gb_read(lds, bbase[s & 1] + (uint32_t)((s >> 1) * BB + j * 2048));
    };

    floatx4 acc[8][WN];
#pragma unroll
    for (int r = 0; r < 8; r++)
#pragma unroll
        for (int j = 0; j < WN; j++)
            acc[r][j] = floatx4{};

    /* prologue: W units 0..2, X stages 0 and 1 */
#pragma unroll
    for (int j = 0; j < WN; j++)
        dma_x(0, 0, j);
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int k = 0; k < 4; k++)
            dma_w(u, u, k);
#pragma unroll
    for (int j = 0; j < WN; j++)
        dma_x(1, 1, j);
#pragma unroll
    for (int k = 0; k < 4; k++)
        dma_w(2, 2, k);
    gb_wait<WN + 4, 0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    bf16x8 a[4], b0[WN], b1[WN];
#pragma unroll
    for (int j = 0; j < WN; j++)
        b0[j] = rdb(0, j);
#pragma unroll
    for (int r = 0; r < GB_AD; r++)
        a[r] = rda(0, r);

    /* unit u in ring slot S, its X fragments in b: reads unit u + 1's into bn */
    auto unit = [&](auto slot, int u, bf16x8 (&b)[WN], bf16x8 (&bn)[WN]) {
        constexpr int S = decltype(slot)::value;
        gb_wait<gb_vm(S, WN), gb_lgkm(S, WN)>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int uw = min(u + 3, nu - 4 + ((S + 3) & 3));
        const int px = min((u >> 1) + 2, (nu >> 1) - 2 + (S >> 1));
#pragma unroll
        for (int r = 0; r < 8; r++) {
#pragma unroll
            for (int j = 0; j < WN; j++) {
                /* at most one memory operation between two MFMAs */
                const gb_mem m = gb_before(S, WN, r, j);
                if (m.kind == GB_READ_A)
                    a[m.row & 3] = rda(m.slot, m.row);
                if (m.kind == GB_DMA_X)
                    dma_x(px, m.slot >> 1, m.row);
                if (m.kind == GB_READ_B)
                    bn[m.row] = rdb(m.slot, m.row);
                if (m.kind == GB_DMA_W)
                    dma_w(uw, m.slot, m.row);
                gb_mfma(acc[r][j], a[r & 3], b[j]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    for (int u = 0; u < nu; u += 4) {
        unit(std::integral_constant<int, 0>{}, u, b0, b1);
        unit(std::integral_constant<int, 1>{}, u + 1, b1, b0);
        unit(std::integral_constant<int, 2>{}, u + 2, b0, b1);
        unit(std::integral_constant<int, 3>{}, u + 3, b1, b0);
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);

    /* acc[r][j]: token 16 (wn WN + j) + l%16 of the tile, rows 4 (l/16) + 0..3
     * of the wave's row group r */
    if constexpr (MODE == GB_PART) {
        const int n0 = nb * BN + wn * WN * 16 + c16;
#pragma unroll
        for (int r = 0; r < 8; r++) {
            const int m = 16 * (mb * 16 + wm * 8 + r) + 4 * q;
            if (m >= M)
                continue;
#pragma unroll
            for (int j = 0; j < WN; j++)
                if (n0 + 16 * j < N)
                    *(floatx4 *)(P + ((size_t)sp * N + n0 + 16 * j) * M + m) = acc[r][j];
        }
        return;
    }
    /* bf16 outputs go out as whole 16-byte pieces of a token's row: each wave
     * turns its block around in its own quarter of the (now idle) ring,
     * 16-byte piece s of token t in slot s ^ (t % 16) (gated: 8 pieces,
     * s ^ (t / 2 % 8)), so that neither side has bank conflicts. */
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    constexpr int RG = MODE == GB_GATED ? 4 : 8; /* row groups of output rows */
    constexpr int TB = RG * 32;                  /* bytes per token */
    unsigned char *st = smem + wave * (WN * 16 * 256);
    static_assert(4 * WN * 16 * 256 <= (int)sizeof(smem), "staging");
    auto slot = [](int t, int s) { return MODE == GB_GATED ? s ^ ((t >> 1) & 7) : s ^ (t & 15); };
#pragma unroll
    for (int j = 0; j < WN; j++) {
        const int t = 16 * j + c16;
#pragma unroll
        for (int r = 0; r < RG; r++) {
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if constexpr (MODE == GB_GATED)
                    o[e] = f2bf(silu_f(bf2f(f2bf(acc[r][j][e]))) * bf2f(f2bf(acc[r + 4][j][e])));
                else
                    o[e] = f2bf(acc[r][j][e]);
            }
            *(bf16x4 *)(st + t * TB + slot(t, 2 * r + (q >> 1)) * 16 + (q & 1) * 8) = o;
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    constexpr int LPT = TB / 16;  /* lanes per token */
    constexpr int TPI = 64 / LPT; /* tokens per store */
    const int ts = lane / LPT, ps = lane % LPT;
    const int mo = (MODE == GB_GATED ? 64 : 128) * (mb * 2 + wm) + 8 * ps;
    const int n1 = nb * BN + wn * WN * 16;
    const int mrows = MODE == GB_GATED ? M >> 1 : M;
    if (mo >= mrows)
        return;
    /* whole pieces where the rows allow 16-byte stores (M % 16 == 0, so a
     * piece never straddles the last row) */
    const bool wide = ldy % 8 == 0 && ((uintptr_t)Y & 15) == 0;
#pragma unroll
    for (int i = 0; i < WN * 16 / TPI; i++) {
        const int t = i * TPI + ts;
        const bf16x8 v = *(const bf16x8 *)(st + t * TB + slot(t, ps) * 16);
        if (n1 + t < N) {
            bf16 *dst = Y + (size_t)(n1 + t) * ldy + mo;
            if (wide) {
                *(bf16x8 *)dst = v;
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++)
                    dst[e] = v[e];
            }
        }
    }
}

template <int MODE>
hipError_t launch_mode(int WN, dim3 grid, hipStream_t s, const bf16 *X, int ldx, const bf16 *W,
                       int N, int M, int K, int nch, int mblocks, int nblocks, int splits,
                       int per_xcd, bf16 *Y, int ldy, float *P) {
#define CUJEV_GB_CASE(wn)                                                                     \
    if (WN == wn) {                                                                           \
        hipLaunchKernelGGL((gemm_block_kernel<wn, MODE>), grid, dim3(256), 0, s, X, ldx, W, N, \
                           M, K, nch, mblocks, nblocks, splits, per_xcd, Y, ldy, P);          \
        return hipGetLastError();                                                             \
    }
    CUJEV_GB_CASE(8)
    CUJEV_GB_CASE(6)
    if constexpr (MODE != GB_GATED) /* gated 256 x 128 runs in gemm_wide.hip */
        CUJEV_GB_CASE(4)
#undef CUJEV_GB_CASE
    return hipErrorInvalidValue;
}

} // namespace
} // namespace CUJEV_KNS

using namespace CUJEV_KNS;

extern "C" int cujev_gemm_block_ok(const bf16_t *X, int ldx) {
    /* 16-byte DMA pieces of the X rows */
    return ldx % 8 == 0 && ((uintptr_t)X & 15) == 0;
}

extern "C" hipError_t k_gemm_block(const bf16_t *X, int ldx, const bf16_t *Wt, int N, int M, int K,
                                   int gated, int WN, int splits, bf16_t *Y, int ldy, float *P,
                                   hipStream_t stream) {
    /* arguments checked by k_gemm_wide */
    const int mblocks = gated ? CEIL_DIV(M / 2, 128) : CEIL_DIV(M, 256);
    const int nblocks = CEIL_DIV(N, 32 * WN);
    const int items = mblocks * nblocks * splits, per_xcd = CEIL_DIV(items, 8);
    const dim3 grid((unsigned)(8 * per_xcd));
    const int nch = K / 128 / splits;
    const bf16 *x = (const bf16 *)X, *w = (const bf16 *)Wt;
    if (gated)
        return launch_mode<GB_GATED>(WN, grid, stream, x, ldx, w, N, M, K, nch, mblocks, nblocks, 1,
                                     per_xcd, (bf16 *)Y, ldy, nullptr);
    if (splits > 1)
        return launch_mode<GB_PART>(WN, grid, stream, x, ldx, w, N, M, K, nch, mblocks, nblocks,
                                    splits, per_xcd, nullptr, 0, P);
    return launch_mode<GB_PLAIN>(WN, grid, stream, x, ldx, w, N, M, K, nch, mblocks, nblocks, 1,
                                 per_xcd, (bf16 *)Y, ldy, nullptr);
}
