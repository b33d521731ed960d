// fp32-activation GEMV and the row kernels of the gfx950 path.
//
//  * k_gemv_f32    fp32 activations x dequantized Q4 row-major matrix (tied
//                  unembedding, MTP heads) in the canonical 64-lane order;
//                  k_gemv_f32_glu: a head's gate and up products and their
//                  SiLU product in one launch.
//  * k_mm_f32      the same products of many activation rows on the fp32
//                  matrix core.
//  * row kernels   quantize_activation_row of whole rows, layer-skip
//                  decisions and cache commits, embedding, small copies.
//  * k_matmul_i8   the reference's plain int8 matmul API.
// The int8-activation x block-quantized products are in pf_mm.hip.
#include "pf_device.h"

namespace pf {

// ============================================ fp32 x dequantized Q4 GEMV

// The M activation rows (K <= 2048 floats each) staged once per workgroup
// in LDS, then lane l's 32 elements of every row (block l) in registers
// (zeros for lanes past the row's blocks): one copy of the rows per
// workgroup from L2 instead of one per wave.  Block b's 16-byte word i sits
// at word i ^ ((b >> 1) & 7) of the block, so that 16 consecutive lanes
// reading word i of their blocks fall on distinct banks (unswizzled, eight of
// them share one: 18.9 against 15.0 us for 4 rows x a 16384 x 2048 matrix).
template <int M>
__device__ __forceinline__ void stage_rows(const float* __restrict__ h, uint32_t h_stride, uint32_t K, uint32_t lane,
                                           bool live, float (&hv)[M][32]) {
    __shared__ __align__(16) float hsm[M * 2048];
    const uint32_t n4 = K >> 2;
    for (uint32_t i = threadIdx.x; i < M * n4; i += blockDim.x) {
        const uint32_t m = i / n4, c = i - m * n4;
        reinterpret_cast<float4*>(hsm)[m * 512u + (c ^ ((c >> 4) & 7u))] = *reinterpret_cast<const float4*>(h + (size_t)m * h_stride + 4u * c);
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < M; m++) {
#pragma unroll
        for (int i = 0; i < 32; i += 4) {
            const uint32_t w = ((uint32_t)i >> 2) ^ ((lane >> 1) & 7u);
            const float4 v = live ? *reinterpret_cast<const float4*>(hsm + m * 2048 + lane * 32u + 4u * w)
                                  : make_float4(0.f, 0.f, 0.f, 0.f);
            hv[m][i] = v.x; hv[m][i + 1] = v.y; hv[m][i + 2] = v.z; hv[m][i + 3] = v.w;
        }
    }
}

// The 8 weights (nibble - 8) d of a Q4 code word in element order, each one
// v_cvt_f32_ubyte and one v_fma (the asm keeps the compiler from extracting
// the bytes first and from copying nd for a two-operand fma, which cost two
// more steps per weight).
__device__ __forceinline__ void q4_weights(uint32_t cw, float d, float nd, float (&w)[8]) {
    uint32_t lo = cw & 0x0F0F0F0Fu, hi = (cw >> 4) & 0x0F0F0F0Fu;
    asm("" : "+v"(lo), "+v"(hi));
#pragma unroll
    for (int b = 0; b < 4; b++) {
        const float x0 = (float)((lo >> (8 * b)) & 0xFFu), x1 = (float)((hi >> (8 * b)) & 0xFFu);
        asm("v_fma_f32 %0, %1, %2, %3" : "=v"(w[2 * b]) : "v"(x0), "v"(d), "v"(nd));
        asm("v_fma_f32 %0, %1, %2, %3" : "=v"(w[2 * b + 1]) : "v"(x1), "v"(d), "v"(nd));
    }
}

// Halving trees of NV values per lane over the wave at once (wave_tree_sum's
// order each): a level's pairs of values share one add, half of the lanes
// summing one of them, down to the 8-lane level; the remaining levels run on
// the ceil(NV / 8) words left.  On return lane l with l & 7 == 0 holds in
// s[k] the sum of value 8 k + 4 (l >> 3 & 1) + 2 (l >> 4 & 1) + (l >> 5).
// Against a tree of its own per value: 40 VALU steps instead of 224 (and no
// LDS permutes) for 16 values.
template <int NV>
__device__ __forceinline__ void wave_tree_sums(const float (&v)[NV], float (&s)[(NV + 7) / 8]) {
    constexpr int N1 = (NV + 1) / 2, N2 = (N1 + 1) / 2, N3 = (N2 + 1) / 2;
    const uint32_t lane = threadIdx.x & 63u;
    float a[N1], b[N2];
#pragma unroll
    for (int k = 0; k < N1; k++) {
        const auto p = __builtin_amdgcn_permlane32_swap(f2u(v[2 * k]), f2u(v[2 * k + 1 < NV ? 2 * k + 1 : 2 * k]), false, false);
        a[k] = u2f(p[0]) + u2f(p[1]);
    }
#pragma unroll
    for (int k = 0; k < N2; k++) {
        const auto p = __builtin_amdgcn_permlane16_swap(f2u(a[2 * k]), f2u(a[2 * k + 1 < N1 ? 2 * k + 1 : 2 * k]), false, false);
        b[k] = u2f(p[0]) + u2f(p[1]);
    }
#pragma unroll
    for (int k = 0; k < N3; k++) {
        const float x = b[2 * k], y = b[2 * k + 1 < N2 ? 2 * k + 1 : 2 * k];
        float t = ((lane & 8u) ? y : x) + dpp_mov<DPP_ROR8>((lane & 8u) ? x : y);
        const float c = t + dpp_mov<DPP_ROR4>(t), d = t + dpp_mov<DPP_ROR12>(t);
        t = (lane & 4u) ? c : d;
        t = t + dpp_mov<DPP_XOR2>(t);
        s[k] = t + dpp_mov<DPP_XOR1>(t);
    }
}

// y[m][n] (+= y_in[m][n] when resid) = canonical fp32 dot of h[m] with row n:
// lane l holds block l (K <= 2048), fmaf chain over the block's elements,
// halving tree over the 64 lanes.  Wave w walks the groups of RB rows
// RB w, RB (w + total_waves), ..., loading a group's codes and scales before
// its products.  Grid y takes the activation rows M at a time: slice y serves
// rows M y .. M y + M - 1.
// FMT: Q4 (16 code bytes per block: weight (nibble - 8) d, formed as
// fmaf(nibble, d, -8 d), exact) or Q8 (32: weight (float)code * d, exact).
// Bound: VALU issue (per 32 weights 72 steps to form them and 32 M fmaf, then
// the trees).  16384 x 2048 Q4: 5.2 / 10.9 / 13.7 us for 1 / 4 / 5 rows; with
// unswizzled staging, a tree of its own per sum and 4 + 1 rows in two launches
// it took 7.1 / 18.8 / 25.1.
template <int M, int FMT, int RB>
__global__ __launch_bounds__(256) void k_gemv_f32(const uint8_t* __restrict__ codes,
                                                  const uint16_t* __restrict__ scales,
                                                  uint32_t N, uint32_t K,
                                                  const float* __restrict__ h, uint32_t h_stride,
                                                  float* __restrict__ y, uint32_t y_stride,
                                                  const float* __restrict__ y_in) {
    h += (size_t)blockIdx.y * M * h_stride;
    y += (size_t)blockIdx.y * M * y_stride;
    if (y_in) y_in += (size_t)blockIdx.y * M * y_stride;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const uint32_t nwaves = gridDim.x * (blockDim.x >> 6);
    const uint32_t nb = K >> 5;
    const bool live = lane < nb;
    float hv[M][32];
    stage_rows<M>(h, h_stride, K, lane, live, hv);
    for (uint32_t n0 = RB * wave; n0 < N; n0 += RB * nwaves) {
        constexpr uint32_t CB = FMT == FMT_Q8 ? 2u : 1u;   // 16-byte code words per block
        uint4 cr[RB][CB];
        float dr[RB];
#pragma unroll
        for (uint32_t q = 0; q < RB; q++) {
            const uint32_t n = n0 + q;
#pragma unroll
            for (uint32_t u = 0; u < CB; u++) cr[q][u] = make_uint4(0u, 0u, 0u, 0u);
            dr[q] = 0.0f;
            if (live && n < N) {
#pragma unroll
                for (uint32_t u = 0; u < CB; u++)
                    cr[q][u] = *reinterpret_cast<const uint4*>(codes + ((size_t)n * nb + lane) * (16u * CB) + 16u * u);
                dr[q] = h2f(scales[(size_t)n * nb + lane]);
            }
        }
        float acc[RB * M];   // value q M + m
#pragma unroll
        for (uint32_t q = 0; q < RB; q++) {
#pragma unroll
            for (int m = 0; m < M; m++) acc[q * M + m] = 0.0f;
            if (live) {
                const float d = dr[q];
                if constexpr (FMT == FMT_Q8) {
                    const uint32_t cw[8] = {cr[q][0].x, cr[q][0].y, cr[q][0].z, cr[q][0].w,
                                            cr[q][1].x, cr[q][1].y, cr[q][1].z, cr[q][1].w};
#pragma unroll
                    for (int j = 0; j < 32; j++) {
                        const float wj = (float)(int8_t)((cw[j >> 2] >> (8 * (j & 3))) & 0xFFu) * d;
#pragma unroll
                        for (int m = 0; m < M; m++) acc[q * M + m] = __builtin_fmaf(hv[m][j], wj, acc[q * M + m]);
                    }
                } else {
                    const uint32_t cw[4] = {cr[q][0].x, cr[q][0].y, cr[q][0].z, cr[q][0].w};
                    const float nd = -8.0f * d;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        float w[8];
                        q4_weights(cw[i], d, nd, w);
#pragma unroll
                        for (int j = 0; j < 8; j++)
#pragma unroll
                            for (int m = 0; m < M; m++)
                                acc[q * M + m] = __builtin_fmaf(hv[m][8 * i + j], w[j], acc[q * M + m]);
                        // a word's weights at a time: all 32 cost 24 registers
                        // and with them a wave per SIMD (4 rows)
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
        float s[(RB * M + 7) / 8];
        wave_tree_sums<RB * M>(acc, s);
#pragma unroll
        for (uint32_t k = 0; k < (RB * M + 7) / 8; k++) {
            const uint32_t i = 8u * k + 4u * ((lane >> 3) & 1u) + 2u * ((lane >> 4) & 1u) + (lane >> 5);
            const uint32_t n = n0 + i / M;
            if ((lane & 7u) == 0 && i < RB * M && n < N) {
                const size_t o = (size_t)(i % M) * y_stride + n;
                y[o] = y_in ? (y_in[o] + s[k]) : s[k];
            }
        }
    }
}

// One MTP head's gate and up products with the SiLU product fused
// (src/mtp.cpp:63-127): a[m][n] = silu(g) * u, g and u the canonical dots
// of h[m] with row n of Wg and Wu (k_gemv_f32's order), silu(g) =
// g / (1 + exp(-g)) (src/mtp.cpp:89-91, 157-159): the bits of two
// k_gemv_f32 products followed by that elementwise step.
template <int M>
__global__ __launch_bounds__(256) void k_gemv_f32_glu(const uint8_t* __restrict__ gcodes,
                                                      const uint16_t* __restrict__ gscales,
                                                      const uint8_t* __restrict__ ucodes,
                                                      const uint16_t* __restrict__ uscales, uint32_t N, uint32_t K,
                                                      const float* __restrict__ h, uint32_t h_stride,
                                                      float* __restrict__ a, uint32_t a_stride) {
    h += (size_t)blockIdx.y * M * h_stride;   // grid y: activation rows M at a time
    a += (size_t)blockIdx.y * M * a_stride;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const uint32_t nwaves = gridDim.x * (blockDim.x >> 6);
    const uint32_t nb = K >> 5;
    const bool live = lane < nb;
    float hv[M][32];
    stage_rows<M>(h, h_stride, K, lane, live, hv);
    for (uint32_t n = wave; n < N; n += nwaves) {
        float ag[M], au[M];
#pragma unroll
        for (int m = 0; m < M; m++) ag[m] = au[m] = 0.0f;
        if (live) {
            const uint4 cg = *reinterpret_cast<const uint4*>(gcodes + ((size_t)n * nb + lane) * 16u);
            const uint4 cu = *reinterpret_cast<const uint4*>(ucodes + ((size_t)n * nb + lane) * 16u);
            const float dg = h2f(gscales[(size_t)n * nb + lane]), du = h2f(uscales[(size_t)n * nb + lane]);
            const uint32_t gw[4] = {cg.x, cg.y, cg.z, cg.w}, uw[4] = {cu.x, cu.y, cu.z, cu.w};
            const float ndg = -8.0f * dg, ndu = -8.0f * du;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float wg[8], wu[8];
                q4_weights(gw[i], dg, ndg, wg);
                q4_weights(uw[i], du, ndu, wu);
#pragma unroll
                for (int j = 0; j < 8; j++)
#pragma unroll
                    for (int m = 0; m < M; m++) {
                        ag[m] = __builtin_fmaf(hv[m][8 * i + j], wg[j], ag[m]);
                        au[m] = __builtin_fmaf(hv[m][8 * i + j], wu[j], au[m]);
                    }
            }
        }
#pragma unroll
        for (int m = 0; m < M; m++) {
            const float g = wave_tree_sum(ag[m]), u = wave_tree_sum(au[m]);
            if (lane == 0) {
                const float sg = g / (1.0f + expf_c(-g));
                a[(size_t)m * a_stride + n] = sg * u;
            }
        }
    }
}

// =========================================== fp32 x dequantized rows, tall

// The canonical fp32 products of k_gemv_f32 (and with GLU the SiLU product of
// k_gemv_f32_glu) for many activation rows, on v_mfma_f32_32x32x1_2b_f32: one
// step of it rounds as one fmaf per element, so 32 steps over a 32-element
// block are the block's fmaf chain bit for bit.  A wave owns 32 rows of h x 32
// matrix rows; one step of its loop forms blocks l and l + 32 (the
// instruction's two halves) and adds them, the halving tree's first level.
// Blocks come in bit-reversed order of l, so the deeper levels join as a
// binary counter of partial tiles.  KS 4 splits the blocks over the workgroup's
// waves by the tree's last two levels, whose partial tiles meet in LDS.
// Blocks past K / 32 count as zeros, as k_gemv_f32's idle lanes do.
//
// Grid 8 * mtiles * ceil(n groups / 8), a group being the 4 / KS matrix tiles
// of a workgroup: workgroup b runs on XCD b mod 8, which so reads one eighth
// of the matrix, each part for all the row tiles in turn.
// What bounds it: fp32 issue (per 32 MFMAs of 32.8 ns, 72 steps to form the
// weights and 32 adds of the tree do not overlap with them).  A 16384 x 2048
// Q4 matrix takes 29 / 49 / 222 us for 32 / 64 / 320 rows (slices of 4 rows on
// the VALU: 232 and 1130 for the last two), a head's gate, up and SiLU of 64
// rows 30 (86), its down product 16 (45).
// One wave per tile (KS 1) for more than 1024 tiles, else four.
template <int FMT, bool GLU, int KS>
__global__ __launch_bounds__(256, KS == 1 || GLU ? 2 : 3) void k_mm_f32(
    const uint8_t* __restrict__ codes, const uint16_t* __restrict__ scales, const uint8_t* __restrict__ ucodes,
    const uint16_t* __restrict__ uscales, uint32_t N, uint32_t K, uint32_t M, uint32_t mtiles,
    const float* __restrict__ h, uint32_t h_stride, float* __restrict__ y, uint32_t y_stride,
    const float* __restrict__ y_in) {
    constexpr uint32_t NG = 4u / KS;                        // matrix tiles of a workgroup
    constexpr uint32_t CB = FMT == FMT_Q8 ? 2u : 1u;        // 16-byte code words per block
    static_assert(KS == 1 || KS == 4, "a wave per tile, or the workgroup's four");
    constexpr int LV = KS == 1 ? 5 : 3;                     // tree levels inside the wave
    __shared__ float red[KS > 1 ? 4 * 16 * 64 : 1];
    const uint32_t t = threadIdx.x, lane = t & 63u, r = lane & 31u, hh = lane >> 5;
    const uint32_t wid = __builtin_amdgcn_readfirstlane(t >> 6), part = wid % KS;
    const uint32_t slot = blockIdx.x >> 3, mt = slot % mtiles, grp = (slot / mtiles) * 8u + (blockIdx.x & 7u);
    const uint32_t n0 = 32u * (grp * NG + wid / KS), m0 = 32u * mt, nb = K >> 5;
    if (32u * grp * NG >= N) return;                        // the whole workgroup
    const bool in = n0 < N;                                 // N % 64 == 0: whole tiles
    const float* hr = h + (size_t)min(m0 + r, M - 1u) * h_stride;
    const size_t wrow = (size_t)(in ? n0 + r : 0u) * nb;
    constexpr uint32_t S = 32u / KS;
    float tg[16], tot[16];
#pragma unroll
    for (int i = 0; i < 16; i++) tot[i] = tg[i] = 0.0f;
#pragma unroll 1
    for (uint32_t prod = 0; prod < (GLU ? 2u : 1u); prod++) {
        const uint8_t* cp = GLU && prod ? ucodes : codes;
        const uint16_t* sp = GLU && prod ? uscales : scales;
        float st[LV][16];
#pragma unroll
        for (int k = 0; k < LV; k++)
#pragma unroll
            for (int i = 0; i < 16; i++) st[k][i] = 0.0f;
        // this lane's block of step s (clamped: loads past the blocks read the last)
        auto blk = [&](uint32_t s) { return min((__brev(s) >> 27) + 32u * hh, nb - 1u); };
        float4 a0[4], a1[4];
        uint4 cw[CB];
        uint32_t sc = 0;
        uint32_t b = blk(part * S);
#pragma unroll
        for (int i = 0; i < 4; i++) a0[i] = *reinterpret_cast<const float4*>(hr + 32u * b + 4 * i);
#pragma unroll
        for (uint32_t u = 0; u < CB; u++) cw[u] = *reinterpret_cast<const uint4*>(cp + (wrow + b) * (16u * CB) + 16u * u);
        sc = sp[wrow + b];
#pragma unroll 1
        for (uint32_t v = 0; v < S; v++) {
            const uint32_t s = part * S + v, l = __brev(s) >> 27;
            const uint32_t bn = blk(min(s + 1u, part * S + S - 1u));
            const bool dead = l >= nb, half = l + 32u >= nb;     // no block at all, or none in the upper half
            // the step's second half of h, and the next step's codes and first half
#pragma unroll
            for (int i = 0; i < 4; i++) a1[i] = *reinterpret_cast<const float4*>(hr + 32u * b + 16 + 4 * i);
            uint4 cn[CB];
#pragma unroll
            for (uint32_t u = 0; u < CB; u++) cn[u] = *reinterpret_cast<const uint4*>(cp + (wrow + bn) * (16u * CB) + 16u * u);
            const uint32_t sn = sp[wrow + bn];
            const float d = h2f((uint16_t)sc), nd = -8.0f * d;
            pf_v32f acc = {};
            auto step8 = [&](int q, const float4 x, const float4 z) {   // elements 8 q .. 8 q + 7
                float w[8];
                if constexpr (FMT == FMT_Q8) {
                    const uint4 c4 = cw[q >> 1];
                    const uint32_t c0 = (q & 1) ? c4.z : c4.x, c1 = (q & 1) ? c4.w : c4.y;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        w[j] = (float)(int8_t)((c0 >> (8 * j)) & 0xFFu) * d;
                        w[4 + j] = (float)(int8_t)((c1 >> (8 * j)) & 0xFFu) * d;
                    }
                } else {
                    q4_weights(q == 0 ? cw[0].x : (q == 1 ? cw[0].y : (q == 2 ? cw[0].z : cw[0].w)), d, nd, w);
                    // two wait states between a VALU write and the MFMA that
                    // reads it, which the compiler does not count for asm
                    asm("s_nop 1" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]), "+v"(w[4]), "+v"(w[5]), "+v"(w[6]), "+v"(w[7]));
                }
                const float e[8] = {x.x, x.y, x.z, x.w, z.x, z.y, z.z, z.w};
#pragma unroll
                for (int j = 0; j < 8; j++) acc = __builtin_amdgcn_mfma_f32_32x32x1f32(e[j], w[j], acc, 0, 0, 0);
            };
            auto clear_upper = [&](float4 (&a)[4]) {   // the missing block's lanes multiply zeros
                if (!half) return;
#pragma unroll
                for (int i = 0; i < 4; i++) a[i] = hh ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : a[i];
            };
            if (!dead) {
                clear_upper(a0);
                step8(0, a0[0], a0[1]);
                step8(1, a0[2], a0[3]);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) a0[i] = *reinterpret_cast<const float4*>(hr + 32u * bn + 4 * i);
            if (!dead) {
                clear_upper(a1);
                step8(2, a1[0], a1[1]);
                step8(3, a1[2], a1[3]);
            }
            b = bn;
            sc = sn;
#pragma unroll
            for (uint32_t u = 0; u < CB; u++) cw[u] = cn[u];
            float x[16];
#pragma unroll
            for (int i = 0; i < 16; i++) x[i] = acc[i] + acc[16 + i];
            // binary counter: level k waits in st[k] for its partner
            bool carry = true;
#pragma unroll
            for (int k = 0; k < LV; k++) {
                if (!carry) continue;
                if ((v >> k) & 1u) {
#pragma unroll
                    for (int i = 0; i < 16; i++) x[i] = st[k][i] + x[i];
                } else {
#pragma unroll
                    for (int i = 0; i < 16; i++) st[k][i] = x[i];
                    carry = false;
                }
            }
            if (v + 1u == S)
#pragma unroll
                for (int i = 0; i < 16; i++) tot[i] = x[i];
        }
        if constexpr (KS > 1) {
            // parts in the counter's order: (0 + 1) + (2 + 3)
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 16; i++) red[(wid * 16u + i) * 64u + lane] = tot[i];
            __syncthreads();
            const uint32_t w0 = wid - part;
#pragma unroll
            for (int i = 0; i < 16; i++)
                tot[i] = (red[(w0 * 16u + i) * 64u + lane] + red[((w0 + 1u) * 16u + i) * 64u + lane]) +
                         (red[((w0 + 2u) * 16u + i) * 64u + lane] + red[((w0 + 3u) * 16u + i) * 64u + lane]);
        }
        if (GLU && prod == 0)
#pragma unroll
            for (int i = 0; i < 16; i++) tg[i] = tot[i];
    }
    if (!in) return;
    // register i: row m0 + 8 (i / 4) + 4 hh + i % 4, matrix row n0 + r; the
    // parts share the tile's registers
#pragma unroll
    for (int i = 0; i < 16; i++) {
        if (i % KS != (int)part) continue;
        const uint32_t m = m0 + 8u * (i / 4) + 4u * hh + (i % 4);
        if (m >= M) continue;
        const size_t o = (size_t)m * y_stride + n0 + r;
        if constexpr (GLU) {
            const float sg = tg[i] / (1.0f + expf_c(-tg[i]));
            y[o] = sg * tot[i];
        } else {
            y[o] = y_in ? (y_in[o] + tot[i]) : tot[i];
        }
    }
}

// y[m][n] = canonical fp32 dot of h[m] with row n of a dense fp32 matrix E
// [N][K] (an fp32 tied table handed to MTPHeads::forward): the order of
// k_gemv_f32 with the weight value itself (lane l = block l, K <= 2048).  The
// table bounds it (134 MB at 16384 x 2048: 25.1 us for four rows, 5.4 TB/s;
// 22.6 for each row by itself), so up to four heads' rows take it in one pass.
template <int M>
__global__ __launch_bounds__(256) void k_gemv_f32_dense(const float* __restrict__ E, uint32_t N, uint32_t K,
                                                        const float* __restrict__ h, uint32_t h_stride,
                                                        float* __restrict__ y, uint32_t y_stride) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const uint32_t nwaves = gridDim.x * (blockDim.x >> 6);
    const bool live = lane < (K >> 5);
    float hv[M][32];
    stage_rows<M>(h, h_stride, K, lane, live, hv);
    for (uint32_t n = wave; n < N; n += nwaves) {
        float acc[M];
#pragma unroll
        for (int m = 0; m < M; m++) acc[m] = 0.0f;
        if (live) {
            const float* row = E + (size_t)n * K + lane * 32u;
            float w[32];
#pragma unroll
            for (int i = 0; i < 32; i += 4) {
                float4 v = *reinterpret_cast<const float4*>(row + i);
                w[i] = v.x; w[i + 1] = v.y; w[i + 2] = v.z; w[i + 3] = v.w;
            }
#pragma unroll
            for (int i = 0; i < 32; i++)
#pragma unroll
                for (int m = 0; m < M; m++) acc[m] = __builtin_fmaf(hv[m][i], w[i], acc[m]);
        }
        float s[1];
        wave_tree_sums<M>(acc, s);
        const uint32_t m = 4u * ((lane >> 3) & 1u) + 2u * ((lane >> 4) & 1u) + (lane >> 5);
        if ((lane & 7u) == 0 && m < M) y[(size_t)m * y_stride + n] = s[0];
    }
}

// MTPHeads::forward without a tied table (src/mtp.cpp:117-121): logits[v] =
// ((v * 2654435761 + head) mod V) / V.
__global__ void k_mtp_placeholder(float* __restrict__ logits, uint32_t V, uint32_t head) {
    const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    logits[v] = (float)(((uint64_t)v * 2654435761ULL + (uint64_t)head) % V) / (float)V;
}

// dot_product (src/matmul_neon.cpp:186-207) in the CANON(4) order: lane l of
// 256 sums a[j] * b[j] (product, then add) for j = l, l + 256, ...
__global__ __launch_bounds__(256) void k_dot_canon(const float* __restrict__ a, const float* __restrict__ b,
                                                   uint32_t n, float* __restrict__ out) {
    __shared__ float red[4];
    float p = 0.0f;
    for (uint32_t j = threadIdx.x; j < n; j += 256) p = p + a[j] * b[j];
    const float s = block_canon_sum<4>(p, red);
    if (threadIdx.x == 0) *out = s;
}

// softmax in place (src/matmul_neon.cpp:212-226): max, e = exp(x - max),
// CANON(4) sum, x = e * (1 / (sum + 1e-10)).
__global__ __launch_bounds__(256) void k_softmax_one(float* __restrict__ v, uint32_t n) {
    __shared__ float red[4];
    float mx = -__builtin_inff();
    for (uint32_t j = threadIdx.x; j < n; j += 256) mx = fmaxf(mx, v[j]);
    mx = block_max<4>(mx, red);
    float part = 0.0f;
    for (uint32_t j = threadIdx.x; j < n; j += 256) {
        const float e = expf_c(v[j] - mx);
        v[j] = e;
        part = part + e;
    }
    const float inv = 1.0f / (block_canon_sum<4>(part, red) + 1e-10f);
    for (uint32_t j = threadIdx.x; j < n; j += 256) v[j] = v[j] * inv;
}

// rmsnorm (src/matmul_neon.cpp:231-239): CANON(4) sum of squares (fmaf),
// rms = sqrt(ss / n + 1e-6), out = x * (1 / rms) * w.
__global__ __launch_bounds__(256) void k_rmsnorm_one(float* __restrict__ out, const float* __restrict__ x,
                                                     const float* __restrict__ w, uint32_t n) {
    __shared__ float red[4];
    float p = 0.0f;
    for (uint32_t j = threadIdx.x; j < n; j += 256) p = __builtin_fmaf(x[j], x[j], p);
    const float ss = block_canon_sum<4>(p, red);
    const float inv = 1.0f / __builtin_sqrtf(ss / (float)n + 1e-6f);
    for (uint32_t j = threadIdx.x; j < n; j += 256) out[j] = x[j] * inv * w[j];
}

// ============================================================ prologues

// Rows quantized (quantize_activation_row), row-major with q_stride.
template <int PER>
__global__ __launch_bounds__(256) void k_quant_rows(const float* __restrict__ x, uint32_t x_stride,
                                                    uint32_t K, int8_t* __restrict__ q, uint32_t q_stride,
                                                    float* __restrict__ as, int32_t* __restrict__ bsum,
                                                    uint32_t bsum_stride) {
    __shared__ float red[4];
    const uint32_t m = blockIdx.x;
    float v[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
        uint32_t i = threadIdx.x + 256u * k;
        v[k] = i < K ? x[(size_t)m * x_stride + i] : 0.0f;
    }
    quantize_row_block<PER, 256>(v, K, q + (size_t)m * q_stride, as + m,
                                 bsum ? bsum + (size_t)m * bsum_stride : nullptr, red);
}

// quantize_activation_row of rows of length K <= NT * PER into the GEMM's
// operand order, NT threads.
template <int PER, int NT = 1024>
__global__ __launch_bounds__(NT) void k_quant_rows_wide(const float* __restrict__ x, uint32_t K,
                                                        int8_t* __restrict__ q, float* __restrict__ as) {
    __shared__ float red[16];
    const uint32_t m = blockIdx.x;
    float v[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const uint32_t i = threadIdx.x + (uint32_t)NT * k;
        v[k] = i < K ? x[(size_t)m * K + i] : 0.0f;
    }
    quantize_row_block<PER, NT, true>(v, K, q + operand_row(m, K), as + m, nullptr, red);
}

// LayerSkipController::should_skip_ffn (src/layer_skip.cpp:22-67) at one
// layer for the rows of sequence blockIdx.x in pass order.  normed holds the
// FFN inputs of the pass's rows [M][K]; each row's delta (hidden_delta,
// src/layer_skip.cpp:105-111: sqrt of the mean squared difference, the sum in
// the tile order of the engine's RMSNorm) is taken against the input of the
// sequence's last row in this pass that ran its FFN, else against the
// sequence's cache (cache + blockIdx.x * cache_seq_stride).  flag[r] = 1:
// row r skips its FFN.  thr is the layer's adjusted threshold (< 0: the layer
// never skips).  nrun (zeroed earlier in the pass) gains the number of rows
// that run their FFN: the FFN products of a pass in which no row runs it are
// not computed.  The cache is written by k_skip_commit once it is known which
// rows count.  Rows go one after another, the 16 waves sharing each row's
// tiles.  K % 64 == 0, K <= 4096; 1024 threads.
__global__ __launch_bounds__(1024) void k_layer_skip(const PassDesc* __restrict__ pd, uint32_t M,
                                                     const float* __restrict__ normed,
                                                     const float* __restrict__ cache, size_t cache_seq_stride,
                                                     uint32_t K, float thr, uint32_t* __restrict__ flag,
                                                     uint32_t* __restrict__ nrun) {
    __shared__ float tree[64];
    __shared__ uint32_t skipped;
    const uint32_t s = blockIdx.x, t = threadIdx.x, wid = t >> 6, lane = t & 63u;
    const float* ref = cache + (size_t)s * cache_seq_stride;
    uint32_t runs = 0;
    for (uint32_t r = 0; r < M; r++) {
        if (row_seq(pd, r) != s) continue;
        const float* a = normed + (size_t)r * K;
        if (!(thr >= 0.0f)) {
            if (t == 0) flag[r] = 0;
            ref = a;
            runs++;
            continue;
        }
        for (uint32_t tl = wid; tl < K / 64u; tl += 16u) {
            const float d = a[64u * tl + lane] - ref[64u * tl + lane];
            const float sq = wave_tree_sum(d * d);
            if (lane == 0) tree[tl] = sq;
        }
        __syncthreads();
        if (t == 0) {
            float sum = 0.0f;
            for (uint32_t tl = 0; tl < K / 64u; tl++) sum = sum + tree[tl];
            const uint32_t sk = __builtin_sqrtf(sum / (float)K) < thr ? 1u : 0u;
            flag[r] = sk;
            skipped = sk;
        }
        __syncthreads();
        if (!skipped) {
            ref = a;
            runs++;
        }
    }
    if (t == 0 && runs) atomicAdd(nrun, runs);
}

// The cache update of should_skip_ffn (src/layer_skip.cpp:57-62) for the rows
// of a pass that count: per (layer blockIdx.x, sequence blockIdx.y), the
// sequence's rows j0 <= j < j1 (j numbering the sequence's rows in pass
// order), where for a verify pass (st non-null) j1 = min(accepted + 1, n_mtp)
// with the round's accepted drafts from st[sequence] -- the rows that
// src/engine.cpp:336-365 forwards.  The cache takes the FFN input of the last
// such row that ran its FFN; skips counts the rows that skipped.
// stage [L][rows][K], flags [L][rows], cache [nseq][L][K]; 256 threads.
__global__ __launch_bounds__(256) void k_skip_commit(const PassDesc* __restrict__ pd, uint32_t M,
                                                     const float* __restrict__ stage,
                                                     const uint32_t* __restrict__ flags, uint32_t rows,
                                                     float* __restrict__ cache, uint32_t L, uint32_t K, uint32_t j0,
                                                     uint32_t j1, const DecodeState* __restrict__ st,
                                                     uint32_t n_mtp, uint32_t* __restrict__ skips) {
    const uint32_t l = blockIdx.x, s = blockIdx.y;
    const uint32_t hi = st ? min(st[s].round_acc + 1u, n_mtp) : j1;
    int32_t src = -1;
    uint32_t j = 0, nskip = 0;
    for (uint32_t r = 0; r < M; r++) {
        if (row_seq(pd, r) != s) continue;
        if (j >= j0 && j < hi) {
            if (flags[(size_t)l * rows + r]) nskip++;
            else src = (int32_t)r;
        }
        j++;
    }
    if (threadIdx.x == 0 && nskip) atomicAdd(skips, nskip);
    if (src < 0) return;
    const float* a = stage + ((size_t)l * rows + (uint32_t)src) * K;
    float* c = cache + ((size_t)s * L + l) * K;
    for (uint32_t i = threadIdx.x; i < K; i += 256) c[i] = a[i];
}

// dst = src (float), used instead of a copy node inside captured passes.
__global__ void k_copy_f32(const float* __restrict__ src, float* __restrict__ dst, uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// Token embedding: x[m] = dequantized row tok[m] of the tied table (Q4 or
// Q8, fmt).
// The first kernel of every pass also advances the pass epoch `ep`, which
// names the pass in the flags of the LL words its QKV products write.
__device__ __forceinline__ void embed_elem(const uint8_t* __restrict__ codes, const uint16_t* __restrict__ scales,
                                           uint32_t V, uint32_t D, const PassDesc* __restrict__ pd,
                                           float* __restrict__ x, uint32_t* __restrict__ ep, int32_t fmt, uint32_t m,
                                           uint32_t i) {
    if (ep && m == 0 && i == 0) ep[0] += 1u;
    if (m >= pd->m || i >= D) return;
    int32_t tok = pd->tok[m];
    float val = 0.0f;
    if (tok >= 0 && (uint32_t)tok < V) {
        uint32_t nb = D >> 5, b = i >> 5, e = i & 31u;
        float d = h2f(scales[(size_t)tok * nb + b]);
        if (fmt == FMT_Q8) {
            val = (float)(int8_t)codes[((size_t)tok * nb + b) * 32u + e] * d;
        } else {
            uint8_t byte = codes[((size_t)tok * nb + b) * 16u + (e >> 1)];
            uint32_t nib = (e & 1u) ? (byte >> 4) : (byte & 15u);
            val = (float)((int)nib - 8) * d;
        }
    }
    x[(size_t)m * D + i] = val;
}
__global__ void k_embed(const uint8_t* __restrict__ codes, const uint16_t* __restrict__ scales,
                        uint32_t V, uint32_t D, const PassDesc* __restrict__ pd, float* __restrict__ x,
                        uint32_t* __restrict__ ep, int32_t fmt) {
    embed_elem(codes, scales, V, D, pd, x, ep, fmt, blockIdx.y, blockIdx.x * blockDim.x + threadIdx.x);
}

// ============================================ reference plain-int8 matmul

typedef int pf_i4 __attribute__((ext_vector_type(4)));
typedef int pf_i16 __attribute__((ext_vector_type(16)));

// Bytes k .. k + 15 of the K-byte row at offset `row` of a matrix of `total`
// bytes at p (any alignment), zeros past the row's end: one 16-byte load, no
// further than the row's end (K >= 16) or the matrix's, moved down into place.
// (Rows of 4 to 12 bytes taken byte by byte cost up to 1.5 times the rest of a
// 4096 x 4096 product.)
__device__ __forceinline__ pf_i4 tail16(const int8_t* p, size_t total, size_t row, uint32_t k, uint32_t K) {
    unsigned long long v[2] = {0ull, 0ull};
    if (total >= 16u) {
        const uint32_t kl = K >= 16u ? min(k, K - 16u) : 0u;
        const size_t o = K >= 16u ? row + kl : min(row, total - 16u);
        const uint32_t sh = 8u * min((uint32_t)(row - o) + k, 16u);
        __builtin_memcpy(v, p + o, 16);
        if (sh >= 64u) {
            v[0] = sh < 128u ? v[1] >> (sh - 64u) : 0ull;
            v[1] = 0ull;
        } else if (sh) {
            v[0] = (v[0] >> sh) | (v[1] << (64u - sh));
            v[1] >>= sh;
        }
        if (K < 16u) {   // k is 0 (the row) or 16 (all zeros)
            v[0] = K >= 8u ? v[0] : v[0] & ((1ull << (8u * K)) - 1ull);
            v[1] = K > 8u ? v[1] & ((1ull << (8u * K - 64u)) - 1ull) : 0ull;
        }
    } else {
        for (uint32_t i = 0; k + i < K; i++) {
            const unsigned long long c = (unsigned long long)(uint8_t)p[row + k + i] << (8u * (i & 7u));
            v[0] |= i < 8u ? c : 0ull;
            v[1] |= i < 8u ? 0ull : c;
        }
    }
    pf_i4 r;
    __builtin_memcpy(&r, v, 16);
    return r;
}

// C[i][j] = sum_k A[i][k] * B[j][k] (src/matmul_neon.cpp:80-144) on
// v_mfma_i32_32x32x32_i8, any sizes and row alignments.  W waves own 32 rows
// of A x 32 rows of B; wave w of them takes the 32-column steps w, w + W, ...
// of K with its operands straight from memory (16 bytes per lane, four steps'
// loads together), and their int32 sums meet in LDS (exact, so the split
// changes nothing).  QUANT: the outputs leave as (float)sum * as[i] * ws[j]
// (src/matmul_neon.cpp:176-180), else as int32.  Columns from n_base on.
//
// Latency bounds the API's sizes (a few MB): splitting K over the waves puts
// most of a workgroup's loads into one round trip.  M 100, N 3000, K 1100:
// 5.9 us beside 3.1 us for the row quantization, where one thread per output
// took 332 us.  Workgroups of two or four A tiles (B read once for them)
// measured the same at M 100-128 and slower at M = N / 16 = 256, K 4096
// (four tiles 52.8 us, one 38.3).  MM_SHORT_K columns or fewer are one round
// trip for a wave alone, and from MM_SHORT_TILES tiles (eight waves per CU) on
// the outputs are what counts: a tile per wave (W 1), stored from registers.
// M 4096, N 4096, K 4: 14.1 us (W 8: 26.8); M 4096, N 16 (128 tiles) stays at
// 7.4 us where W 1 takes 8.7.
constexpr uint32_t MM_WAVES = 8;
constexpr uint32_t MM_SHORT_K = 128, MM_SHORT_TILES = 2048;
template <bool QUANT, uint32_t W>
__global__ __launch_bounds__(64 * MM_WAVES) void k_matmul_i8(const int8_t* __restrict__ A, uint32_t lda,
                                                      const int8_t* __restrict__ B, uint32_t M, uint32_t N,
                                                      uint32_t K, int32_t* __restrict__ Ci,
                                                      const float* __restrict__ as, const float* __restrict__ ws,
                                                      float* __restrict__ C, uint32_t n_base) {
    static_assert(W == 1 || W == MM_WAVES, "a tile per wave or per workgroup");
    __shared__ int red[W][16][64];
    constexpr uint32_t U = 4;
    const uint32_t t = threadIdx.x, lane = t & 63u, r = lane & 31u, h = lane >> 5;
    const uint32_t wid = __builtin_amdgcn_readfirstlane(t >> 6), part = W == 1u ? 0u : wid;
    const uint32_t n0 = n_base + 32u * (W == 1u ? MM_WAVES * blockIdx.x + wid : blockIdx.x), m0 = 32u * blockIdx.y;
    if (W == 1u && n0 >= N) return;
    const int8_t* bp = B + (size_t)min(n0 + r, N - 1u) * K;
    const int8_t* ap = A + (size_t)min(m0 + r, M - 1u) * lda;
    pf_i16 acc = {};
    const uint32_t full = K >> 5;
    for (uint32_t s0 = part; s0 < full; s0 += U * W) {
        pf_i4 a[U], b[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {   // past the last step: reloaded, not used
            const uint32_t k = 32u * min(s0 + u * W, full - 1u) + 16u * h;
            __builtin_memcpy(&b[u], bp + k, 16);
            __builtin_memcpy(&a[u], ap + k, 16);
        }
#pragma unroll
        for (uint32_t u = 0; u < U; u++)
            if (s0 + u * W < full) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[u], b[u], acc, 0, 0, 0);
    }
    if ((K & 31u) && part == full % W) {
        const uint32_t k = 32u * full + 16u * h;
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(tail16(A, (size_t)M * lda, (size_t)(ap - A), k, K),
                                                    tail16(B, (size_t)N * K, (size_t)(bp - B), k, K), acc, 0, 0, 0);
    }
    auto put = [&](uint32_t m, uint32_t n, int v) {
        if constexpr (QUANT) C[(size_t)m * N + n] = (float)v * as[m] * ws[n];
        else Ci[(size_t)m * N + n] = v;
    };
    // sum j of lane (r, h): row 8 (j / 4) + 4 h + j % 4, column r of the tile
    if constexpr (W == 1u) {
#pragma unroll
        for (uint32_t j = 0; j < 16; j++) {
            const uint32_t m = m0 + 8u * (j >> 2) + 4u * h + (j & 3u), n = n0 + r;
            if (m < M && n < N) put(m, n, acc[j]);
        }
    } else {
#pragma unroll
        for (uint32_t j = 0; j < 16; j++) red[wid][j][lane] = acc[j];
        __syncthreads();
        for (uint32_t x = t; x < 1024u; x += 64u * W) {
            const uint32_t l = x & 63u, j = x >> 6;
            const uint32_t m = m0 + 8u * (j >> 2) + 4u * (l >> 5) + (j & 3u), n = n0 + (l & 31u);
            if (m >= M || n >= N) continue;
            int v = red[0][j][l];
#pragma unroll
            for (uint32_t w = 1; w < W; w++) v += red[w][j][l];
            put(m, n, v);
        }
    }
}

// matmul_quantized's given-scale activation path (src/matmul_neon.cpp:158-164).
__global__ void k_quant_div(const float* __restrict__ A, const float* __restrict__ sc,
                            int8_t* __restrict__ q, uint32_t q_stride, uint32_t M, uint32_t K) {
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
    if (k >= K || i >= M) return;
    q[(size_t)i * q_stride + k] = (int8_t)(int)__builtin_roundf(A[(size_t)i * K + k] / sc[i]);
}

}  // namespace pf
