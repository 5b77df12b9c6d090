/*
 * mlx4_gemm.hip -- the batched MLX 4-bit projections of a prefill chunk on
 * gfx950 MFMA: Y[M tokens][N] = X[M][K] W^T for the [N x K] affine 4-bit
 * weight of src/kernels.c:104-219, the GEMM form of ds4f_mlx4_matvec_batch
 * (src/kernels.c:581-619) that ds4f_attn_gqa_chunk / ds4f_attn_linear_chunk
 * call on their B normed token rows (src/attn_qwen.c:1199-1221).
 *
 * Exactness.  With w = q s + b (q in 0..15, s and b the BF16 scale and
 * bias of the 64-element group), and G the groups along K,
 *     y[m][n] = sum_g s'[n,g] sum_{k in g} (1 + q/16) x  +  b'[n,g] xsum[m,g],
 *     s' = 16 s,  b' = b - 16 s,  xsum[m,g] = sum_{k in g} x.
 * 1 + q/16 is exact in fp16 (the nibble in mantissa bits 6..9 under the
 * exponent of 1), x is carried as an fp16 hi + lo pair (about 22 bits),
 * each MFMA product is exact in fp32, and the group partial is scaled by
 * s' in fp32 after its 8 MFMAs (4 k-steps x hi / lo); xsum is the sum of
 * the same hi + lo values.  The offset 1 is at most about twice the q/16
 * part, so the cancellation against b' xsum costs about a bit, and the
 * result differs from the reference's fp32 dot products by fp32 rounding
 * of the group sums.
 *
 * Layouts:
 *   xw      (xprep_kernel) per 64-token tile mt and group g, a 16 KB block
 *           at ((mt G + g) 2 + {0: hi, 1: lo}) 8 KB, fp16: the group's MFMA
 *           operands as the waves read them, 1 KB each (q35_xw_granule); 8
 *           consecutive k (one nibble word's worth) kept in the order
 *           0,4,1,5,2,6,3,7, the order in which a word's nibbles become fp16
 *           pairs (nibbles j and j + 4 moved to bits 6..9 and 22..25, ORed
 *           into 0x3C003C00, give 1 + q_j / 16 and 1 + q_{j+4} / 16);
 *   xsum    fp32 [G][Mpad];
 *   sb      (sb_kernel) (16 s, b - 16 s) as [G][Npad], Npad = N rounded up
 *           to 256, zeros past N;
 *   wt      (wt_kernel) the weight words re-laid out once per weight: per
 *           256-feature tile and group an 8 KB block that is the LDS image
 *           of the stage (16-byte position p = row p / 2, half
 *           wslot(row, p % 2)), rows past N zero; staging it is a plain
 *           copy, 1 KB a wave load.
 * In a group (8 words), MFMA k-step ks of lane half h is word 4h + ks: a
 * lane's weight operand for a whole group is one 16-byte read.
 *
 * gemm_kernel: 256 threads, a 64-token x 256-feature tile; wave w owns
 * features 64w..64w+63 as 2 x 2 blocks of v_mfma_f32_32x32x16_f16 (A = X,
 * B = W^T converted in registers).  Every global load is a direct-to-LDS
 * load into a ring of three stages, one group each (X hi and lo 16 KB,
 * the tile's weight words 8 KB, (s, b') 2 KB, xsum 256 B), issued two
 * groups ahead (every stage load a contiguous 1 KB); each wave waits for
 * its own loads of the next group
 * before the one barrier a group.  Two workgroups fit a CU (157.5 KB of
 * LDS), two waves a SIMD.
 * gemm_few_kernel: the same product split over K inside a workgroup, for
 * chunks of few tokens (few_tokens picks).
 */
#include "q35_device.h"
#include "q35_launch.h"

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;

namespace {

constexpr int NT = 256;
constexpr int MT = 64;                 /* tokens a tile */
constexpr int NTILE = 256;             /* features a tile, 64 a wave */
constexpr int XBLK = Q35_XW_BLK;       /* bytes of a tile's hi (or lo) X of one group */
static_assert(MT == Q35_XW_ROWS, "the X tiles are the GEMM's token tiles");
constexpr int WBLK = NTILE * 32;       /* bytes of a tile's weight words of one group */
constexpr int SBLK = NTILE * 8;        /* bytes of a tile's (s, b') of one group */
constexpr int OFF_W = 2 * XBLK, OFF_SB = OFF_W + WBLK, OFF_XS = OFF_SB + SBLK;
constexpr int STAGE = OFF_XS + MT * 4; /* 26880 bytes */
constexpr int NSTAGE = 3;
constexpr float QSTEP = 16.0f;         /* B = 1 + q / QSTEP */

/* slot of half h (words 4h..4h+3) of tile feature row r in its 32-byte
 * weight row: distinct over 4 and 8 consecutive rows, so the operand reads are
 * free of bank conflicts */
__device__ __forceinline__ int wslot(int r, int h) { return h ^ (((r >> 2) ^ (r >> 3)) & 1); }

/* x rows -> (optional RMSNorm) -> fp16 hi / lo operands and the group sums of
 * hi + lo.  One workgroup of NTX threads per XR token rows: thread t holds
 * row t % XR, words t / XR + i NTX / XR (WT of them), so the lanes of a
 * 64-column group are 8 XR neighbours, reads are 256 consecutive bytes of each
 * row and stores 16 XR bytes of the operand image.  XR = 8 stores whole
 * 128-byte lines, but with few tokens it is few workgroups that convert 8
 * rows each; launch_xprep has the line.
 * Rows at and past M in the last workgroup are stored as zeros; operand rows
 * after those are never written: an operand row only reaches its own output
 * row, which is not stored.  The norm is an fp32 square sum times the hardware
 * rsq (about 1 ulp from the reference's double sum and division,
 * src/attn_qwen.c:142-157, far below the hi / lo split's 22 bits). */
/* sum over the 8 lanes of one row's words of a group (8 XR neighbouring
 * lanes, equal lane % XR), the total in each of them */
template <int XR>
__device__ __forceinline__ float group_sum(float v) {
    static_assert(XR == 8 || XR == 4 || XR == 2, "lane patterns of 2, 4 and 8 rows");
    v += q35_xor8(v);
    if constexpr (XR == 8) return q35_psum32(q35_psum16(v));
    v += q35_dpp<0x124>(v);                /* row_ror:4, on sums of period 8 */
    if constexpr (XR == 4) return q35_psum16(v);
    return v + q35_dpp<0x122>(v);          /* row_ror:2, on sums of period 4 */
}
template <int NTX, int XR, int WT>
__global__ __launch_bounds__(NTX) void xprep_kernel(Q35Mlx4Xprep p) {
    const int t = threadIdx.x, lane = t & 63, r = t % XR;
    const int m0 = blockIdx.x * XR, m = m0 + r;
    const int nw = p.K / 8;
    __shared__ float sred[NTX / 64][XR];

    /* the thread's words of its row and of the norm weight, all requested
     * at once as range-checked buffer loads (rows past M, words past K and
     * an absent norm weight read as zeros): the norm and the conversion
     * then work from registers, one memory round trip a workgroup */
    const int nr = min(XR, p.M - m0);
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        q35_uniform_ptr(const_cast<float *>(p.x + (size_t)m0 * p.ldx)), 0, ((nr - 1) * p.ldx + p.K) * 4,
        Q35_BUF_DW3);
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        q35_uniform_ptr(const_cast<uint16_t *>(p.norm_w)), 0, p.norm_w ? p.K * 2 : 0, Q35_BUF_DW3);
    float4 xa[WT], xb[WT];
    uint4 wv[WT];
#pragma unroll
    for (int i = 0; i < WT; i++) {
        const int v = t / XR + i * (NTX / XR);
        const uint32_t off = v < nw && r < nr ? (uint32_t)(r * p.ldx + 8 * v) * 4 : 0x80000000u;
        xa[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(xrs, off, 0, 0));
        xb[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(xrs, off + 16, 0, 0));
        wv[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(wrs, 16 * v, 0, 0));
    }

    float ri = 1.0f;
    if (p.norm_w) {
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < WT; i++) {
            const float e[8] = {xa[i].x, xa[i].y, xa[i].z, xa[i].w, xb[i].x, xb[i].y, xb[i].z, xb[i].w};
#pragma unroll
            for (int j = 0; j < 8; j++) ss = fmaf(e[j], e[j], ss);
        }
        ss = group_sum<XR>(ss);
        if constexpr (XR == 2) ss = q35_psum16(ss);
        if constexpr (XR <= 4) ss = q35_psum32(ss);
        if (lane < XR) sred[t >> 6][lane] = ss;
        q35_lds_barrier();
        ss = 0.0f;
#pragma unroll
        for (int i = 0; i < NTX / 64; i++) ss += sred[i][r];
        ri = __builtin_amdgcn_rsqf(ss * (1.0f / (float)p.K) + 1e-6f);
    }
#pragma unroll
    for (int i = 0; i < WT; i++) {
        const int v = t / XR + i * (NTX / XR);
        if (v >= nw) break;   /* nw is a multiple of 8: a group's 8 words leave together */
        float e[8] = {xa[i].x, xa[i].y, xa[i].z, xa[i].w, xb[i].x, xb[i].y, xb[i].z, xb[i].w};
        if (p.norm_w) {
            const uint32_t ww[4] = {wv[i].x, wv[i].y, wv[i].z, wv[i].w};
#pragma unroll
            for (int j = 0; j < 8; j++)
                e[j] = e[j] * ri * q35_bf2f((uint16_t)(ww[j >> 1] >> (16 * (j & 1))));
        }
        bool over = false;
#pragma unroll
        for (int j = 0; j < 8; j++) over = over || q35_f16_over(e[j]);
        q35_f16_guard(p.status, Q35_STATUS_GEMM_F16, over);
        f16x8_t hi, lo;
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float v8 = e[q35_xw_perm(j)];
            const _Float16 h = (_Float16)v8;
            const _Float16 l = (_Float16)(v8 - (float)h);
            hi[j] = h;
            lo[j] = l;
            s += (float)h + (float)l;
        }
        uint8_t *blk = reinterpret_cast<uint8_t *>(p.xw) + q35_xw_granule(m, v, p.K / 64);
        *reinterpret_cast<f16x8_t *>(blk) = hi;
        *reinterpret_cast<f16x8_t *>(blk + XBLK) = lo;
        s = group_sum<XR>(s);
        if ((lane & (8 * XR - 1)) < XR) p.xsum[(size_t)(v >> 3) * p.Mpad + m] = s;
    }
}

/* (16 s, b - 16 s) of a weight's rows and groups as [G][npad] (zeros for
 * rows past N), from its BF16 scales and biases [N][G] (biases may be
 * NULL) */
__global__ void sb_kernel(const uint16_t *scales, const uint16_t *biases, Q35Mlx4SB *sb, int N, int G,
                          int npad) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)G * npad) return;
    const int g = (int)(i / npad), n = (int)(i % npad);
    float sv = 0.0f, bv = 0.0f;
    if (n < N) {
        const float s = q35_bf2f(scales[(size_t)n * G + g]);
        const float b = biases ? q35_bf2f(biases[(size_t)n * G + g]) : 0.0f;
        sv = QSTEP * s;
        bv = b - sv;
    }
    sb[i] = Q35Mlx4SB{sv, bv};
}

/* the weight words [N][K/8] as wt blocks [npad/256][G][512 granules of
 * 16 bytes]: granule p of block (tile, g) = words 4 wslot(r, p % 2) ..
 * +3 of group g of row tile * 256 + r, r = p / 2; zeros past N */
__global__ void wt_kernel(const uint32_t *vals, u32x4_t *wt, int N, int K, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int G = K / 64;
    const int p = (int)(i & 511);
    const int64_t blk = i >> 9;
    const int g = (int)(blk % G), tile = (int)(blk / G);
    const int r = p >> 1, row = tile * NTILE + r;
    u32x4_t v = {0u, 0u, 0u, 0u};
    if (row < N)
        v = *reinterpret_cast<const u32x4_t *>(vals + (size_t)row * (K / 8) + 8 * g + 4 * wslot(r, p & 1));
    wt[i] = v;
}

/* a word's 8 nibbles as the fp16 B operand 1 + q / 16, in word order:
 * pair j (nibbles j and j + 4, bits 4j and 16 + 4j) shifted to bits 6 and
 * 22, masked, ORed into the exponent of 1.  The mask and the exponent bits
 * are held in registers (an SGPR and a VGPR) so that each pair is one
 * shift and one v_and_or_b32. */
__device__ __forceinline__ f16x8_t nib_f16(uint32_t w, uint32_t mask, uint32_t one) {
    u32x4_t u;
    u[0] = ((w << 6) & mask) | one;
    u[1] = ((w << 2) & mask) | one;
    u[2] = ((w >> 2) & mask) | one;
    u[3] = ((w >> 6) & mask) | one;
    return __builtin_bit_cast(f16x8_t, u);
}

__device__ __forceinline__ int ntiles(int N) { return (N + NTILE - 1) / NTILE; }

/* One workgroup per (job, 256-feature tile, 64-token tile), numbered with
 * the token tile fastest over the jobs' feature tiles in order.  Work-
 * groups are handed to the 8 XCDs in turn, so with 8 | token tiles an XCD
 * holds token tiles of one residue mod 8 over consecutive feature tiles:
 * about 8 x 8 tiles at once, sharing X and weight tiles in its L2. */
__global__ __launch_bounds__(NT, 2) void gemm_kernel(Q35Mlx4Gemm p) {
    const int ntm = p.Mpad / MT;
    const int mt = blockIdx.x % ntm;
    int nt = blockIdx.x / ntm;
    /* the job of feature tile nt (uniform selects: the job array is kernel
     * arguments, not indexed memory) */
    Q35Mlx4GemmJob J = p.jobs[0];
#pragma unroll
    for (int j = 1; j < Q35_GEMM_MAX_JOBS; j++) {
        const int prev = ntiles(J.N);
        if (j < p.njobs && nt >= prev) {
            nt -= prev;
            J = p.jobs[j];
        }
    }
    float *const Y = J.y;
    const int ldy = J.ldy;
    const int n0 = nt * NTILE, m0 = mt * MT;
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int h = lane >> 5, c = lane & 31;
    const int G = p.K / 64;
    const int npad = (J.N + NTILE - 1) / NTILE * NTILE;

    __shared__ __align__(16) uint8_t smem[NSTAGE * STAGE];
    const uint32_t lds0 = q35_lds_addr(smem);

    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        q35_uniform_ptr(const_cast<uint16_t *>(p.xw)), 0, (int)((size_t)p.Mpad * p.K * 4), Q35_BUF_DW3);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        q35_uniform_ptr(const_cast<uint32_t *>(J.vals)), 0, (int)((size_t)npad * p.K / 2), Q35_BUF_DW3);
    const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
        q35_uniform_ptr(const_cast<Q35Mlx4SB *>(J.sb)), 0, (int)((size_t)G * npad * 8), Q35_BUF_DW3);
    const __amdgpu_buffer_rsrc_t ssr = __builtin_amdgcn_make_buffer_rsrc(
        q35_uniform_ptr(const_cast<float *>(p.xsum)), 0, (int)((size_t)G * p.Mpad * 4), Q35_BUF_DW3);

    /* group g into stage st: X 16 loads, weights 8, (s, b') 2, xsum 1 (a
     * dword load); waves 0-2 issue 7 of them, wave 3 issues 6 */
    auto issue = [&](int g, int st) {
        const uint32_t sb = lds0 + (uint32_t)(st * STAGE);
        const uint32_t xb = (uint32_t)(mt * G + g) * (2 * XBLK);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int i = w + 4 * q;
            q35_dma16(xr, sb + i * 1024, lane * 16, xb + i * 1024);
        }
        const uint32_t wb = (uint32_t)(nt * G + g) * WBLK;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int i = w + 4 * q;
            q35_dma16(wr, sb + OFF_W + i * 1024, lane * 16, wb + i * 1024);
        }
        if (w < 2)
            q35_dma16(sr, sb + OFF_SB + w * 1024, lane * 16, (uint32_t)(g * npad + n0) * 8 + w * 1024);
        else if (w == 2)
            q35_dma4(ssr, sb + OFF_XS, lane * 4, (uint32_t)(g * p.Mpad + m0) * 4);
    };
    /* this wave's loads of the group before the last issued have landed */
    auto wait_prev = [&]() {
        if (w == 3)
            q35_wait_vm<6>();
        else
            q35_wait_vm<7>();
    };

    f32x16_t acc[2][2];
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
#pragma unroll
        for (int nb = 0; nb < 2; nb++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[mb][nb][i] = 0.0f;

    issue(0, 0);
    if (G > 1) {
        issue(1, 1);
        wait_prev();
    } else {
        q35_wait_vm<0>();
    }
    q35_lds_barrier();

    /* a wave whose 64 features all lie past N (a narrow job) only stages */
    const bool idle = n0 + 64 * w >= J.N;
    uint32_t mask, one;
    asm("s_mov_b32 %0, 0x03c003c0" : "=s"(mask));
    asm("v_mov_b32 %0, 0x3c003c00" : "=v"(one));

    int st = 0;
    for (int g = 0; g < G; g++) {
        if (g + 2 < G) issue(g + 2, st == 0 ? 2 : st - 1);
        if (!idle) {
            const uint8_t *S = smem + st * STAGE;
            /* the weight operand: this lane's words 4h..4h+3 of rows
             * 64w + 32nb + c, and their (s, b') */
            f16x8_t bf[2][4];
            float sc[2], bp[2];
#pragma unroll
            for (int nb = 0; nb < 2; nb++) {
                const int r = 64 * w + 32 * nb + c;
                const u32x4_t wq = *reinterpret_cast<const u32x4_t *>(S + OFF_W + r * 32 + wslot(r, h) * 16);
#pragma unroll
                for (int ks = 0; ks < 4; ks++) bf[nb][ks] = nib_f16(wq[ks], mask, one);
                const float2 v = *reinterpret_cast<const float2 *>(S + OFF_SB + r * 8);
                sc[nb] = v.x;
                bp[nb] = v.y;
            }

            /* acc += b' * xsum first: it does not wait for the MFMAs, so it
             * runs while the previous wave's MFMAs hold the pipe */
            {
                const float *xs0 = reinterpret_cast<const float *>(S + OFF_XS);
#pragma unroll
                for (int mb = 0; mb < 2; mb++) {
                    float xsv[16];
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const float4 v = *reinterpret_cast<const float4 *>(xs0 + 32 * mb + 8 * q + 4 * h);
                        xsv[4 * q] = v.x, xsv[4 * q + 1] = v.y, xsv[4 * q + 2] = v.z, xsv[4 * q + 3] = v.w;
                    }
#pragma unroll
                    for (int nb = 0; nb < 2; nb++)
#pragma unroll
                        for (int i = 0; i < 16; i++) acc[mb][nb][i] = fmaf(bp[nb], xsv[i], acc[mb][nb][i]);
                }
            }
            /* the group's MFMAs at raised wave priority, so that the SIMD's
             * other wave does its VALU work around them rather than
             * competing for the issue slot (output GEMM 126 -> 116 us) */
            __builtin_amdgcn_s_setprio(1);
            f32x16_t tmp[2][2];
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                f16x8_t ah[2], al[2];
#pragma unroll
                for (int mb = 0; mb < 2; mb++) {
                    const int off = ((mb * 4 + ks) * 64 + lane) * 16;
                    ah[mb] = *reinterpret_cast<const f16x8_t *>(S + off);
                    al[mb] = *reinterpret_cast<const f16x8_t *>(S + XBLK + off);
                }
#pragma unroll
                for (int mb = 0; mb < 2; mb++)
#pragma unroll
                    for (int nb = 0; nb < 2; nb++) {
                        if (ks == 0) {
                            f32x16_t z;
#pragma unroll
                            for (int i = 0; i < 16; i++) z[i] = 0.0f;
                            tmp[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[mb], bf[nb][ks], z, 0, 0, 0);
                        } else {
                            tmp[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[mb], bf[nb][ks],
                                                                                 tmp[mb][nb], 0, 0, 0);
                        }
                        tmp[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[mb], bf[nb][ks], tmp[mb][nb], 0, 0, 0);
                    }
            }
            __builtin_amdgcn_s_setprio(0);
            /* acc += s' * partial; lane rows 32mb + 8(i/4) + 4h + i%4 */
#pragma unroll
            for (int mb = 0; mb < 2; mb++)
#pragma unroll
                for (int nb = 0; nb < 2; nb++)
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[mb][nb][i] = fmaf(sc[nb], tmp[mb][nb][i], acc[mb][nb][i]);
        }
        /* the next group's stage is complete for every wave; this one is
         * free for the load issued next iteration */
        if (g + 2 < G)
            wait_prev();
        else
            q35_wait_vm<0>();
        q35_lds_barrier();
        st = st == 2 ? 0 : st + 1;
    }

    int nrow[2];
#pragma unroll
    for (int nb = 0; nb < 2; nb++) nrow[nb] = n0 + 64 * w + 32 * nb + c;
    /* y[m][n] (+= with accumulate): lanes 0..31 of a row write 32
     * consecutive features */
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
#pragma unroll
        for (int nb = 0; nb < 2; nb++) {
            const int n = nrow[nb];
            if (n >= J.N) continue;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int m = m0 + 32 * mb + 8 * (i >> 2) + 4 * h + (i & 3);
                if (m < p.M) {
                    float *dst = Y + (size_t)m * ldy + n;
                    *dst = p.accumulate ? *dst + acc[mb][nb][i] : acc[mb][nb][i];
                }
            }
        }
}

/* ---- the same product for chunks of few tokens ----------------------------
 * gemm_kernel's one workgroup per 64 x 256 tile leaves most of the GPU idle
 * when a chunk has few tokens: at M = 64 the 12352 projection rows are 49
 * workgroups and the output projection 8, each walking all of K by itself.
 * Here a workgroup owns a (32 MB) x (32 NB) tile and its NW waves take the
 * groups of K in turn (pairs w, w + NW, ...), so a wave's chain is G / NW
 * groups and nothing is shared between waves: every operand goes from memory
 * straight into the registers of the wave that multiplies it (X in operand
 * order, the weight words in the stage order, both whole lines), with no
 * LDS staging and no barrier in the loop.  The waves' partial tiles meet in
 * LDS and are added in wave order, so a result does not depend on timing.
 * The bias term b' xsum is an fp32 MFMA over the wave's group pairs
 * (v_mfma_f32_32x32x2_f32: one group a lane half) on its own accumulator.
 * What bounds it: a CU's 64 B a cycle from L2, (MB K 128 + NB K 20) bytes a
 * workgroup.  Feature tiles are dealt to the XCDs (id mod 8) with the token
 * tiles of one feature tile behind each other, so an XCD's L2 fetches a
 * weight tile once. */
template <int MB, int NB, int NW>
__global__ __launch_bounds__(64 * NW) void gemm_few_kernel(Q35Mlx4Gemm p, int nft) {
    const int ntm = (p.M + 32 * MB - 1) / (32 * MB);
    const int q = blockIdx.x >> 3, mt = q % ntm;
    int nt = (q / ntm) * 8 + (blockIdx.x & 7);
    if (nt >= nft) return;                  /* workgroup-uniform */
    Q35Mlx4GemmJob J = p.jobs[0];
#pragma unroll
    for (int j = 1; j < Q35_GEMM_MAX_JOBS; j++) {
        const int prev = (J.N + 32 * NB - 1) / (32 * NB);
        if (j < p.njobs && nt >= prev) {
            nt -= prev;
            J = p.jobs[j];
        }
    }
    const int n0 = nt * 32 * NB, m0 = mt * 32 * MB;
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int h = lane >> 5, c = lane & 31;
    const int G = p.K / 64;
    const int npad = (J.N + NTILE - 1) / NTILE * NTILE;
    constexpr int RS = 32 * NB + 8;         /* row stride: lane halves (rows 4 apart) on different banks */
    __shared__ __align__(16) float sp[NW][32 * MB * RS];

    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        q35_uniform_ptr(const_cast<uint16_t *>(p.xw)), 0, (int)((size_t)p.Mpad * p.K * 4), Q35_BUF_DW3);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        q35_uniform_ptr(const_cast<uint32_t *>(J.vals)), 0, (int)((size_t)npad * p.K / 2), Q35_BUF_DW3);
    const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
        q35_uniform_ptr(const_cast<Q35Mlx4SB *>(J.sb)), 0, (int)((size_t)G * npad * 8), Q35_BUF_DW3);
    const __amdgpu_buffer_rsrc_t ssr = __builtin_amdgcn_make_buffer_rsrc(
        q35_uniform_ptr(const_cast<float *>(p.xsum)), 0, (int)((size_t)G * p.Mpad * 4), Q35_BUF_DW3);
    uint32_t mask, one;
    asm("s_mov_b32 %0, 0x03c003c0" : "=s"(mask));
    asm("v_mov_b32 %0, 0x3c003c00" : "=v"(one));

    /* one group's operands: X hi and lo, weight words, s' */
    struct Ops {
        u32x4_t xh[MB][4], xl[MB][4], wq[NB];
        float sc[NB];
    };
    int wrow[NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
        const int rr = (n0 & (NTILE - 1)) + 32 * nb + c;
        wrow[nb] = (rr * 2 + wslot(rr, h)) * 16;
    }
    const int mt64 = m0 / MT, mb0 = (m0 / 32) & 1, tile = n0 / NTILE;
    auto load = [&](int g, Ops &o) {
        const int xb = (mt64 * G + g) * (2 * XBLK) + mb0 * (XBLK / 2);
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                o.xh[mb][ks] = __builtin_amdgcn_raw_buffer_load_b128(xr, lane * 16 + ks * 1024, xb + mb * 4096, 0);
                o.xl[mb][ks] = __builtin_amdgcn_raw_buffer_load_b128(xr, lane * 16 + ks * 1024, xb + XBLK + mb * 4096, 0);
            }
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
            o.wq[nb] = __builtin_amdgcn_raw_buffer_load_b128(wr, wrow[nb], (tile * G + g) * WBLK, 0);
            o.sc[nb] = __uint_as_float(
                __builtin_amdgcn_raw_buffer_load_b32(sr, (32 * nb + c) * 8, (g * npad + n0) * 8, 0));
        }
    };

    f32x16_t acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[mb][nb][i] = 0.0f;

    auto multiply = [&](const Ops &o) {
        f16x8_t bf[NB][4];
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
#pragma unroll
            for (int ks = 0; ks < 4; ks++) bf[nb][ks] = nib_f16(o.wq[nb][ks], mask, one);
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++) {
                f32x16_t tmp;
#pragma unroll
                for (int i = 0; i < 16; i++) tmp[i] = 0.0f;
#pragma unroll
                for (int ks = 0; ks < 4; ks++) {
                    tmp = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, o.xh[mb][ks]),
                                                                 bf[nb][ks], tmp, 0, 0, 0);
                    tmp = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, o.xl[mb][ks]),
                                                                 bf[nb][ks], tmp, 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < 16; i++) acc[mb][nb][i] = fmaf(o.sc[nb], tmp[i], acc[mb][nb][i]);
            }
    };
    /* this wave's group pairs; an odd G's missing group reads zeros */
    for (int g = 2 * w; g < G; g += 2 * NW) {
        float xs[MB], bs[NB];
        const int gh = g + h;
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
            xs[mb] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                ssr, gh < G ? (gh * p.Mpad + m0 + 32 * mb + c) * 4 : (int)0x80000000, 0, 0));
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
            bs[nb] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                sr, gh < G ? (gh * npad + n0 + 32 * nb + c) * 8 + 4 : (int)0x80000000, 0, 0));
        Ops a, b;
        const bool two = g + 1 < G;
        load(g, a);
        if (MB * NB < 4 && two) load(g + 1, b);
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
                acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(xs[mb], bs[nb], acc[mb][nb], 0, 0, 0);
        multiply(a);
        if (MB * NB >= 4 && two) load(g + 1, b);
        if (two) multiply(b);
    }

    /* the waves' tiles -> LDS; lane rows 32mb + 8(i/4) + 4h + i%4, column 32nb + c */
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                sp[w][(32 * mb + 8 * (i >> 2) + 4 * h + (i & 3)) * RS + 32 * nb + c] =
                    acc[mb][nb][i];
    q35_lds_barrier();
    /* y[m][n] (+= with accumulate), four features a thread (N % 4 == 0) */
    const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(
        q35_uniform_ptr(J.y + (size_t)m0 * J.ldy + n0), 0,
        ((min(32 * MB, p.M - m0) - 1) * J.ldy + min(32 * NB, J.N - n0)) * 4, Q35_BUF_DW3);
    constexpr int N4 = 8 * NB;              /* float4s a row */
    for (int i = t; i < 32 * MB * N4; i += 64 * NW) {
        const int r = i / N4, n4 = 4 * (i % N4);
        /* outside the batch or the job's rows: past the view, dropped */
        const bool in = m0 + r < p.M && n0 + n4 < J.N;
        const uint32_t off = in ? (uint32_t)(r * J.ldy + n4) * 4 : 0x80000000u;
        float4 s = p.accumulate
                       ? __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(yr, off, 0, 0))
                       : make_float4(0.f, 0.f, 0.f, 0.f);
        float4 v = *reinterpret_cast<const float4 *>(&sp[0][r * RS + n4]);
#pragma unroll
        for (int k = 1; k < NW; k++) {
            const float4 u = *reinterpret_cast<const float4 *>(&sp[k][r * RS + n4]);
            v.x += u.x, v.y += u.y, v.z += u.z, v.w += u.w;
        }
        s.x += v.x, s.y += v.y, s.z += v.z, s.w += v.w;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, s), yr, off, 0, 0);
    }
}

/* Workgroups of a (32 MB) x (32 NB) tiling. */
inline int64_t few_tiles(const Q35Mlx4Gemm *p, int MB, int NB) {
    int64_t n = 0;
    for (int j = 0; j < p->njobs; j++) n += (p->jobs[j].N + 32 * NB - 1) / (32 * NB);
    return n * ((p->M + 32 * MB - 1) / (32 * MB));
}

/* Which kernel a product runs on: 0 gemm_kernel, 1..4 gemm_few_kernel at
 * 32 x 32, 32 x 64 and 64 x 64 with 8 waves, 64 x 64 with 4.  The smallest
 * tile whose workgroups are at most one a CU (smaller tiles read X more
 * often, a second round costs as much as the first); past that two 4-wave
 * workgroups share a CU; and from 140 64 x 64 x 64 products a CU on,
 * gemm_kernel, whose workgroups share X through LDS, is faster.  us a launch
 * (projections 12352 x 2048 | output 2048 x 4096), gemm_kernel -> here:
 *   M =   32: 40.9 ->  8.3 | 75.6 ->  8.8     M =  256: 42.8 -> 36.9 | 77.2 -> 13.1
 *   M =   64: 41.3 -> 12.1 | 76.3 ->  8.9     M =  512: 55.0 (66.9)  | 76.0 -> 22.3
 *   M =  128: 42.0 -> 20.4 | 76.8 ->  9.8     M = 1024: 107.7 (139)  | 78.2 -> 45.8
 * (in brackets the form that is not taken). */
inline int few_tokens(const Q35Mlx4Gemm *p) {
    constexpr int64_t CUS = 256;
    for (int j = 0; j < p->njobs; j++)
        if (p->jobs[j].N % 4 != 0) return 0;    /* its stores are four features wide */
    const int64_t t22 = few_tiles(p, 2, 2);
    if (t22 * (p->K / 64) > 140 * CUS) return 0;
    if (few_tiles(p, 1, 1) <= CUS) return 1;
    if (few_tiles(p, 1, 2) <= CUS) return 2;
    /* half of the last 64-row tile would be padding, at least a fifth of
     * the work (M = 96, GQA projections: 14.4 us against 19.5) */
    if (p->M > 64 && p->M <= 160 && p->M % 64 > 0 && p->M % 64 <= 32) return 2;
    return t22 <= CUS ? 3 : 4;
}

template <int MB, int NB, int NW>
hipError_t launch_few(const Q35Mlx4Gemm *p, hipStream_t stream) {
    int64_t nft = 0;
    for (int j = 0; j < p->njobs; j++) nft += (p->jobs[j].N + 32 * NB - 1) / (32 * NB);
    const int64_t grid = (nft + 7) / 8 * 8 * ((p->M + 32 * MB - 1) / (32 * MB));
    if (grid >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((gemm_few_kernel<MB, NB, NW>), dim3((unsigned)grid), dim3(64 * NW), 0, stream, *p, (int)nft);
    return hipGetLastError();
}

}  // namespace

extern "C" hipError_t q35_mlx4_sb(const uint16_t *scales, const uint16_t *biases, Q35Mlx4SB *sb, int N,
                                  int G, hipStream_t stream) {
    if (N < 1 || G < 1) return hipErrorInvalidValue;
    const int64_t n = (int64_t)G * q35_mlx4_sb_npad(N);
    hipLaunchKernelGGL(sb_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, scales, biases, sb,
                       N, G, q35_mlx4_sb_npad(N));
    return hipGetLastError();
}

extern "C" int q35_mlx4_sb_npad(int N) { return (N + NTILE - 1) / NTILE * NTILE; }

extern "C" hipError_t q35_mlx4_wt(const uint32_t *vals, uint32_t *wt, int N, int K, hipStream_t stream) {
    if (N < 1 || K < 64 || K % 64 != 0) return hipErrorInvalidValue;
    const int64_t n = (int64_t)q35_mlx4_sb_npad(N) * (K / 64) * 2;   /* granules */
    hipLaunchKernelGGL(wt_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, vals,
                       reinterpret_cast<u32x4_t *>(wt), N, K, n);
    return hipGetLastError();
}

namespace {
/* XR rows a workgroup of N1 threads for K <= 2048 (256 words a row), N2 for
 * K <= 4096, 1024 for K <= 8192, as many words a thread as that takes */
template <int XR, int N1, int N2>
void launch_xprep(const Q35Mlx4Xprep *p, hipStream_t stream) {
    const int words = p->K / 8;
    const dim3 grid((p->M + XR - 1) / XR);
    if (words <= 256)
        hipLaunchKernelGGL((xprep_kernel<N1, XR, 256 * XR / N1>), grid, dim3(N1), 0, stream, *p);
    else if (words <= 512)
        hipLaunchKernelGGL((xprep_kernel<N2, XR, 512 * XR / N2>), grid, dim3(N2), 0, stream, *p);
    else
        hipLaunchKernelGGL((xprep_kernel<1024, XR, XR>), grid, dim3(1024), 0, stream, *p);
}
}  // namespace

extern "C" hipError_t q35_mlx4_xprep(const Q35Mlx4Xprep *p, hipStream_t stream) {
    if (p->K % 64 != 0 || p->K > 8192 || p->Mpad % MT != 0 || p->M > p->Mpad || p->M < 1 || p->ldx < p->K ||
        (int64_t)8 * p->ldx * 4 >= ((int64_t)1 << 31))
        return hipErrorInvalidValue;
    /* us a launch at XR = 2 | 4 | 8 (K = 2048; K = 4096):
     *   M =   64:  2.9 |  3.8 |  5.5;   3.0 |  4.6 |  8.1
     *   M =  256:  3.5 |  4.0 |  5.7;   4.4 |  5.1 |  8.5
     *   M = 1024:  6.3 |  4.9 |  6.5;  10.0 |  7.9 | 10.3
     *   M = 2048: 10.3 |  7.5 |  8.2;  19.1 | 12.7 | 11.6
     *   M = 4096: 19.4 | 12.6 | 11.6;  36.7 | 23.0 | 21.5 */
    if (p->M <= 256)
        launch_xprep<2, 512, 1024>(p, stream);
    else if (p->M <= 2048)
        launch_xprep<4, 512, 1024>(p, stream);
    else
        launch_xprep<8, 512, 512>(p, stream);
    return hipGetLastError();
}

extern "C" hipError_t q35_mlx4_gemm(const Q35Mlx4Gemm *p, hipStream_t stream) {
    if (p->K < 64 || p->K % 64 != 0 || p->Mpad % MT != 0 || p->M > p->Mpad || p->M < 1 || p->njobs < 1 ||
        p->njobs > Q35_GEMM_MAX_JOBS || (int64_t)p->Mpad * p->K * 4 >= ((int64_t)1 << 31) ||
        (int64_t)(p->K / 64) * p->Mpad * 4 >= ((int64_t)1 << 31))
        return hipErrorInvalidValue;
    /* buffer offsets are 32-bit: each weight and its (s, b') table below 2 GB */
    int64_t tiles = 0;
    for (int j = 0; j < p->njobs; j++) {
        const Q35Mlx4GemmJob *J = &p->jobs[j];
        if (J->N < 1 || !J->vals || !J->sb || !J->y || J->ldy < J->N ||
            (int64_t)q35_mlx4_sb_npad(J->N) * p->K / 2 >= ((int64_t)1 << 31) ||
            (int64_t)(p->K / 64) * q35_mlx4_sb_npad(J->N) * 8 >= ((int64_t)1 << 31))
            return hipErrorInvalidValue;
        tiles += (J->N + NTILE - 1) / NTILE;
    }
    tiles *= p->Mpad / MT;
    if (tiles >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
    const int few = few_tokens(p);
    if (few == 1) return launch_few<1, 1, 8>(p, stream);
    if (few == 2) return launch_few<1, 2, 8>(p, stream);
    if (few == 3) return launch_few<2, 2, 8>(p, stream);
    if (few == 4) return launch_few<2, 2, 4>(p, stream);
    hipLaunchKernelGGL(gemm_kernel, dim3((unsigned)tiles), dim3(NT), 0, stream, *p);
    return hipGetLastError();
}

extern "C" int q35_mlx4_gemm_mtile(void) { return MT; }
