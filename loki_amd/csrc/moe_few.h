// moe_few.h -- the grouped IQ2_XXS x Q8_K expert products for columns of few slots (at most FEW_TOK = 8 tokens of one
// expert) on the int8 matrix cores.
//
// Reference: fl_wide_moe's tc_matvec<F_IQ2> (src/fused_layer.cu:178-202, 540-561); the arithmetic is that of
// moe_prefill.hip: exact integer block sums, then y += (d_w * d_x) * bsum in block order, * 0.125 -- bit-identical to
// ggml's scalar dot and to the other kernels.
//
// Most experts of a prompt see few of its tokens (at 37 tokens 123 of 126 used experts at most 8, at 201 116 of 188, at
// 512 78 of 207), and for those the tiles of k_pf_gemm pay for 16 tokens with the scale in every operand byte. The expert
// products of 37 tokens took 473 us there (in fp16), 294 here (gate/up 196, down 98; the call 593 -> 329 us, both sides timed
// in turn). It is bound by the weights' bytes: a gate/up without the products took 159 of then 180 us. Here:
//   * Lane (r, g) of a wave owns row r of a 16-row tile and the 16-byte chunk g (sub-blocks 2g, 2g + 1) of each block, and
//     builds signed int8 weights from the decode tables (8-byte codebook entries, 16-byte sign entries): 4 VALU
//     instructions per 8 weights, no scale.
//   * The scales 2s + 1 stay out of the product because the activation operand is block-diagonal: row 4 g' + q of the
//     16-row operand of v_mfma_i32_16x16x64_i8 is token q's chunk g' in K slice g' (the slice of lane group g') and zero
//     in the other three. The product then leaves in lane (r, g), register q, the sum over chunk g of row r for token q:
//     the lane that knows the chunk's scales. Two products per sub-block (K = 64 is 16 weights of each lane), so a lane
//     holds both sub-block sums of four tokens, multiplies each by its own scale in int32 (|sum| <= 32 * 43 * 127 <
//     2^23) and the four lane groups are added by three register swaps (v_permlane32_swap, v_permlane16_swap): lane
//     (r, g) ends with the block sum of token {0, 2, 1, 3}[g]. One set of four tokens costs 18 VALU instructions per
//     tile and block beside the 41 of the weights; a column has one or two sets.
//   * A wave works alone: an item is (column, 16 h rows of gate and up / 32 down rows) over the whole K, its tokens' Q8_K
//     copied block by block into the wave's own two LDS buffers (one 1 KB direct load per set), its weights two blocks
//     ahead in registers. No workgroup barrier after the tables are in LDS.
#pragma once
#include "moe_device.h"
#include "moe_kernels.h"
#include <type_traits>

namespace lk {

namespace {

typedef int i4 __attribute__((ext_vector_type(4)));

constexpr int FW = 16, FNT = FW * 64;                 // waves / threads per workgroup (one per CU)
constexpr int F_BUF = FEW_TOK * QK;                   // one activation buffer of a wave: 8 tokens x 256 bytes
constexpr int F_LDS = TAB_BYTES + FW * 2 * F_BUF;
static_assert(F_LDS <= 160 * 1024 && TAB_BYTES % (2 * F_BUF) == 0, "LDS budget; buffers toggled by one address bit");

// raw buffer resource over p (gfx9 word 3; the record count only bounds offsets, which stay far below it)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t pf_rsrc(const void * p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short) 0, 0x7fffffff, 0x00020000);
}
// a wave-uniform pointer kept in scalar registers
__device__ __forceinline__ const uint8_t * pf_uniform(const uint8_t * p) {
    const uint64_t v = (uint64_t) p;
    const uint32_t hi = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) (v >> 32));
    const uint32_t lo = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) v);
    return (const uint8_t *) (((uint64_t) hi << 32) | (uint64_t) lo);
}
// SZ bytes per lane from a buffer straight into LDS (lane L at dst + SZ L); the builtin exists for the device pass only,
// so the host pass (which instantiates the kernels' launch stubs) sees an empty body
template <int SZ> __device__ __forceinline__ void buf_lds(__amdgpu_buffer_rsrc_t r, LK_LOCAL uint8_t * dst, uint32_t voff, uint32_t soff) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (SZ == 16) { __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LK_LOCAL void *) dst, 16, voff, soff, 0, 0); }
    else { __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LK_LOCAL void *) dst, 4, voff, soff, 0, 0); }
#else
    (void) r; (void) dst; (void) voff; (void) soff;
#endif
}
// the tables' addressing needs a 64 KB aligned LDS base: false (and the error reported) without one
__device__ __forceinline__ bool pf_base_ok(const PrefillArgs & a, uint32_t base) {
    if (!(base & 0xFFFFu)) { return true; }
    if (threadIdx.x == 0) {
        __hip_atomic_fetch_or(gptr(a.err), 4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a.herr) { __hip_atomic_store(gptr(a.herr), 4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
    }
    return false;
}
// vmcnt(N), nothing moved across it
template <int N> __device__ __forceinline__ void few_wait() {
    static_assert(N < 16, "vmcnt field");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70 | N);
    __builtin_amdgcn_sched_barrier(0);
}
// (volatile: the swaps must run with every lane, so they may not sink into a branch on the lane)
// a + b over the halves of the wave: lanes 0..31 a(l) + a(l + 32), lanes 32..63 b(l - 32) + b(l)
__device__ __forceinline__ int few_add32(int a, int b) {
    uint32_t x = (uint32_t) a, y = (uint32_t) b;
    __asm__ volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(x), "+v"(y));
    return (int) (x + y);
}
// over neighbouring 16-lane rows: rows 0 and 2 of a summed with a's rows 1 and 3, rows 1 and 3 the same of b
__device__ __forceinline__ int few_add16(int a, int b) {
    uint32_t x = (uint32_t) a, y = (uint32_t) b;
    __asm__ volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(x), "+v"(y));
    return (int) (x + y);
}

struct FewW { u32x4 q; uint16_t d; };

// the columns of class PF_FEW (those of the table's part, pf_runs) on the workgroup's 16 waves
template <int NMAT, int NB>
__device__ __forceinline__ void few_body(const PrefillArgs & a, LK_LOCAL uint8_t * lds) {
#pragma clang fp contract(off)
    constexpr int K = NB * QK, C = 2;   // the wave's two 16-row tiles: gate and up of the same h rows, or 32 down rows
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
    const uint32_t base = (uint32_t) (size_t) lds;
    const PfRuns runs = pf_runs(a, PF_FEW);
    const int nt = a.R / (NMAT == 2 ? 16 : 32), items = runs.count() * nt;
    if ((int) blockIdx.x * 4 >= items) { return; }
    if (!pf_base_ok(a, base)) { return; }
    tables_fill(reinterpret_cast<const uint8_t *>(a.tab), lds, threadIdx.x, FNT);
    const int r = lane & 15, g = lane >> 4, q = lane & 3;
    const uint32_t tr = tab_word_grid(base, lane), trs = tab_sign_word(tr);
    // the activation operand's LDS address at MFMA m: lanes whose row's chunk ((lane >> 2) & 3) is their K slice g read
    // token q's bytes 64 g + 16 m of the block (slot (4 g + m) ^ q of the token's row: the 16 such lanes hit 16 bank
    // quads), the others 16 zero bytes (the sign entry of no negative weight)
    const bool diag = ((lane >> 2) & 3) == g;
    const uint32_t xbase = base + (uint32_t) (TAB_BYTES + wave * 2 * F_BUF);
    const uint32_t xa = diag ? xbase + (uint32_t) (q * QK) + ((uint32_t) (4 * g + q) << 4) : trs;
    const uint32_t tog = diag ? (uint32_t) F_BUF : 0u, set1 = diag ? 4u * QK : 0u;
    const int tk = ((g & 1) << 1) | (g >> 1);   // the token of a set whose sums end in this lane
    __syncthreads();

    // four neighbouring waves take the four tiles of a 64-row group (whole lines of the scales); the groups go round the
    // workgroups first, so a last partial round spreads over all CUs
    for (int it = ((wave >> 2) * (int) gridDim.x + (int) blockIdx.x) * 4 + (wave & 3); it < items; it += (int) gridDim.x * FW) {
        const int col = __builtin_amdgcn_readfirstlane(runs.col(it / nt)), ti = __builtin_amdgcn_readfirstlane(it % nt);
        const u32x4 cv = *(const LK_GLOBAL u32x4 *) (a.cols + col);
        const bool routed = (int) cv.x >= 0;
        const int sb = __builtin_amdgcn_readfirstlane((int) cv.y), sc = __builtin_amdgcn_readfirstlane((int) cv.z);
        const int ex = __builtin_amdgcn_readfirstlane((int) cv.w);
        auto brow = [&](int t) -> int {   // activation row of token t of the column
            const int s = sb + (t < sc ? t : 0);
            return NMAT == 2 ? (routed ? gptr(a.perm)[s] / a.topk : s - a.P) : s;
        };
        const __amdgpu_buffer_rsrc_t rb = pf_rsrc(a.bq), rd = pf_rsrc(a.bd);
        const size_t dreg = (size_t) (a.R / 64) * NB * 4096;   // d region offset of a tiled matrix
        __amdgpu_buffer_rsrc_t uq[C], ud[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int mat = NMAT == 2 ? c : 0, row0 = NMAT == 2 ? ti * 16 : ti * 32 + c * 16;
            const uint8_t * Wm = routed ? a.w[mat] + (size_t) ex * a.estride : a.sh[mat];
            const int g64 = row0 >> 6, r0 = row0 & 63;
            uq[c] = pf_rsrc(pf_uniform(Wm + (size_t) g64 * NB * 4096 + r0 * 16));
            ud[c] = pf_rsrc(pf_uniform(Wm + dreg + (size_t) g64 * NB * 128 + r0 * 2));
        }
        const uint32_t lq = (uint32_t) g * 1024 + (uint32_t) r * 16, ldo = (uint32_t) r * 2;
        auto load_w = [&](int j, FewW (&w)[C]) {
#pragma unroll
            for (int c = 0; c < C; ++c) {
                w[c].q = __builtin_amdgcn_raw_buffer_load_b128(uq[c], lq, j * 4096, 2);   // nt: streamed once
                w[c].d = __builtin_amdgcn_raw_buffer_load_b16(ud[c], ldo, j * 128, 0);
            }
        };
        auto run_item = [&](auto sets) {
            constexpr int S = decltype(sets)::value;   // sets of four tokens
            uint32_t ob[S], ox[S];
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const int t = 4 * s + (lane >> 4);     // copy instruction s: lane L takes chunk (L % 16) ^ (t % 4) of token t
                ob[s] = (uint32_t) brow(t) * (uint32_t) K + (uint32_t) (((lane & 15) ^ (t & 3)) << 4);
                ox[s] = (uint32_t) brow(4 * s + tk) * (uint32_t) (NB * 4);
            }
            auto load_x = [&](int j, int buf, float (&dx)[S]) {
                LK_LOCAL uint8_t * dst = lds + TAB_BYTES + wave * 2 * F_BUF + buf * F_BUF;
#pragma unroll
                for (int s = 0; s < S; ++s) { buf_lds<16>(rb, dst + s * 1024, ob[s], j * QK); }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int s = 0; s < S; ++s) { dx[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, ox[s], j * 4, 0)); }
            };
            float acc[C][S];
#pragma unroll
            for (int c = 0; c < C; ++c) { for (int s = 0; s < S; ++s) { acc[c][s] = 0.f; } }

            auto block = [&](const FewW (&w)[C], const float (&dx)[S], uint32_t xo) {
                struct Lk { uint2 g0, g1; uint4 m0, m1; };
                uint32_t ms[C][2];
#pragma unroll
                for (int c = 0; c < C; ++c) { ms[c][0] = w[c].q.y & SIGN_BITS; ms[c][1] = w[c].q.w & SIGN_BITS; }
                auto lookup = [&](int m, int c, Lk & k) {
                    const uint32_t a0 = m < 2 ? w[c].q.x : w[c].q.z, a1 = ms[c][m >> 1];
                    if (m & 1) { k.g0 = tab_grid<2>(a0, tr); k.g1 = tab_grid<3>(a0, tr); k.m0 = tab_sign<2>(a1, trs); k.m1 = tab_sign<3>(a1, trs); }
                    else { k.g0 = tab_grid<0>(a0, tr); k.g1 = tab_grid<1>(a0, tr); k.m0 = tab_sign<0>(a1, trs); k.m1 = tab_sign<1>(a1, trs); }
                };
                auto operand = [&](int m, i4 (&x)[S]) {
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        x[s] = __builtin_bit_cast(i4, *(const LK_LOCAL u32x4 *) (size_t) ((xo + (s ? set1 : 0u)) ^ (uint32_t) (m << 4)));
                    }
                };
                // steps (m, c): one set takes both tiles at each m (one operand read), two sets take the tiles one after
                // the other (half the sums in registers); the next step's reads are issued before this one's product
                i4 D[C][S][2];
                Lk k[2];
                i4 x[2][S];
                constexpr int NS = 4 * C;
                auto step_m = [](int i) { return S == 1 ? i / C : i % 4; };
                auto step_c = [](int i) { return S == 1 ? i % C : i / 4; };
                auto fold = [&](int c) {
                    const float dw = h2f(w[c].d);
                    const int s0 = iq2_scale(w[c].q.y), s1 = iq2_scale(w[c].q.w);
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        int t[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) { t[i] = __mul24(D[c][s][0][i], s0) + __mul24(D[c][s][1][i], s1); }
                        const int b = few_add16(few_add32(t[0], t[1]), few_add32(t[2], t[3]));
                        acc[c][s] = acc[c][s] + (dw * dx[s]) * (float) b;
                    }
                };
                operand(0, x[0]);
                lookup(0, 0, k[0]);
#pragma unroll
                for (int i = 0; i < NS; ++i) {
                    const int m = step_m(i), c = step_c(i);
                    if (i + 1 < NS) {
                        if (step_m(i + 1) != m) { operand(step_m(i + 1), x[step_m(i + 1) & 1]); }
                        lookup(step_m(i + 1), step_c(i + 1), k[(i + 1) & 1]);
                    }
                    const Lk & u = k[i & 1];
                    uint32_t w0, w1, w2, w3;
                    iq2_apply(u.g0, u.m0, w0, w1);
                    iq2_apply(u.g1, u.m1, w2, w3);
                    const i4 wv = { (int) w0, (int) w1, (int) w2, (int) w3 };
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        const i4 z = { 0, 0, 0, 0 };
                        D[c][s][m >> 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[m & 1][s], wv, (m & 1) ? D[c][s][m >> 1] : z, 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if (S > 1 && m == 3) { fold(c); }
                }
                if (S == 1) { fold(0); fold(1); }
            };

            // Block j: the activations and scales of block j + 1 are requested (X), then the weights of block j + WA (W).
            // The requests stay in this order (sched_barrier) and nothing is requested that is not used (an unused load
            // would be dropped and break the count), so block j's activations are in LDS once only the later requests
            // are outstanding: the scales of j (S), the weights requested with them (PW: 2 C), this step's own.
            FewW w0[C], w1[C], w2[C];
            float dx0[S], dx1[S];
            constexpr int WA = S == 1 && NB > 8 ? 2 : 1;   // blocks the weights run ahead (the register budget)
            auto step = [&](auto pw, auto xn, auto wn, int j, const FewW (&cur)[C], FewW (&ahead)[C], const float (&dc)[S], float (&dn)[S], uint32_t xo) {
                constexpr int PW = decltype(pw)::value, X = decltype(xn)::value, W = decltype(wn)::value;
                __builtin_amdgcn_sched_barrier(0);
                if (X) { load_x(j + 1, (j + 1) & 1, dn); }
                if (W) { load_w(j + WA, ahead); }
                few_wait<S + 2 * C * PW + 2 * S * X + 2 * C * W>();
                block(cur, dc, xo);
            };
            constexpr std::integral_constant<int, 1> Y{};
            constexpr std::integral_constant<int, 0> N{};
            load_x(0, 0, dx0);
            load_w(0, w0);
            if (WA == 2) { load_w(1, w1); }
            const uint32_t xo0 = xa, xo1 = xa + tog;
            int j = 0;
            if constexpr (WA == 1) {
                static_assert(NB % 2 == 0, "two steps per trip");
#pragma unroll 1
                for (; j < NB - 2; j += 2) { step(Y, Y, Y, j, w0, w1, dx0, dx1, xo0); step(Y, Y, Y, j + 1, w1, w0, dx1, dx0, xo1); }
                step(Y, Y, Y, j, w0, w1, dx0, dx1, xo0);
                step(Y, N, N, j + 1, w1, w0, dx1, dx0, xo1);
            } else {
                static_assert(NB % 6 == 4, "four steps after the loop");
#pragma unroll 1
                for (; j < NB - 4; j += 6) {
                    step(Y, Y, Y, j, w0, w2, dx0, dx1, xo0);
                    step(Y, Y, Y, j + 1, w1, w0, dx1, dx0, xo1);
                    step(Y, Y, Y, j + 2, w2, w1, dx0, dx1, xo0);
                    step(Y, Y, Y, j + 3, w0, w2, dx1, dx0, xo1);
                    step(Y, Y, Y, j + 4, w1, w0, dx0, dx1, xo0);
                    step(Y, Y, Y, j + 5, w2, w1, dx1, dx0, xo1);
                }
                step(Y, Y, Y, j, w0, w2, dx0, dx1, xo0);
                step(Y, Y, Y, j + 1, w1, w0, dx1, dx0, xo1);
                step(Y, Y, N, j + 2, w2, w1, dx0, dx1, xo0);
                step(N, N, N, j + 3, w0, w2, dx1, dx0, xo1);
            }

#pragma unroll
            for (int s = 0; s < S; ++s) {
                const int t = 4 * s + tk;
                if (t < sc) {
                    if constexpr (NMAT == 2) {
                        const size_t o = (size_t) (sb + t) * a.R + (ti * 16 + r);
                        const float gv = 0.125f * acc[0][s], uv = 0.125f * acc[1][s];
                        a.out[o] = det_silu(gv) * uv;
                        if (a.gdbg) { a.gdbg[o] = gv; a.udbg[o] = uv; }
                    } else {
#pragma unroll
                        for (int c = 0; c < C; ++c) { a.out[(size_t) (sb + t) * a.R + (ti * 32 + c * 16 + r)] = 0.125f * acc[c][s]; }
                    }
                }
            }
        };
        if (sc > 4) { run_item(std::integral_constant<int, 2>{}); }
        else { run_item(std::integral_constant<int, 1>{}); }
    }
}

}  // namespace

}  // namespace lk
