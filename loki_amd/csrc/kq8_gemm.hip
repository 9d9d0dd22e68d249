// kq8_gemm.hip -- the routed down's K-quants (Q2_K, Q3_K) at prefill sizes on the int8 matrix cores.
//
// Reference: tc_matvec<F_Q2K / F_Q3K> of the wide pass (src/fused_layer.cu:203-254, launched at 541-550). The arithmetic is
// the K-quant mat-vec's (kquant.hip), bit for bit: per block the exact integer sums isum = sum_j sc_j sum_i q_i x_i and
// (Q2_K) summ = sum_j mn_j sum_i x_i, then over the blocks in order
//   Q2_K   acc += (d8 * d) * isum - (d8 * dmin) * summ
//   Q3_K   acc += (d * d8) * isum
//
// A scaled weight fits an int8 in both formats, so the scale goes into the matrix product's operand and a block needs no
// further integer work: Q2_K sc * q is 0..45; Q3_K sc * q, with sc in -32..31 and q in -4..3, is -124..128, so its
// negative is taken (-128..124) and the block's term subtracted. The operand bytes come from one v_perm_b32 per 4 weights:
// the stored quants (2 or 3 bits, one per byte) are the selectors into the sub-block's 4 or 8 products, which Q2_K forms by
// one multiply (sc * {0, 1, 2, 3}) and Q3_K reads from an LDS line per scale ((4 - u) * sc, u = 0..7). That is about 1.6
// (Q3_K) VALU instructions per weight and 4 MFMAs per 16 x 16 x 256 block, where the fp16 form this replaces took over 2
// and 16 (its offsets were a second product); it ran the 201-token routed Q3_K down in 678 us.
//
// Work: an item is (column of up to 64 slots, 256 rows), one workgroup of 16 waves per CU takes them round-robin; wave w
// owns one 16-row tile. Lane (r, g), g = 2 n + h, holds of row r the quant bytes 32 n + 16 h .. + 15: the 16-weight
// sub-blocks 8 n + 2 s + h in its four bit planes s. Product s takes plane s: weights 128 n + 32 s + 16 h .. + 15 of the
// block, and the activation operand the same positions. The column's Q8_K rows go block by block from memory into
// XOR-swizzled LDS (direct loads, double-buffered), the next block's weight bytes are in flight while a block computes.
#include "kquant_device.h"
#include "moe_kernels.h"
#include <type_traits>

namespace lk {

namespace {

typedef int ki4 __attribute__((ext_vector_type(4)));
typedef float kf4 __attribute__((ext_vector_type(4)));

constexpr int K8_W = 16, K8_NT = K8_W * 64, K8_ROWS = K8_W * 16, K8_NB = 8;   // K = 2048
constexpr int K8_TT = 4;                       // 16-token tiles per column at most
// LDS: (Q3_K) the scale lines, 64 x 32 copies of 8 bytes (lane l reads copy l % 32); two buffers of 64 block scales; two
// activation buffers of 64 rows x 256 bytes
constexpr int K8_DX = 64 * 256, K8_X = K8_DX + 1024, K8_BUF = K8_TT * 16 * QK, K8_LDS = K8_X + 2 * K8_BUF;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t k8_rsrc(const void * p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short) 0, (int) bytes, 0x00020000);
}
__device__ __forceinline__ const uint8_t * k8_uniform(const uint8_t * p) {
    const uint64_t v = (uint64_t) p;
    const uint32_t hi = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) (v >> 32));
    const uint32_t lo = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) v);
    return (const uint8_t *) (((uint64_t) hi << 32) | (uint64_t) lo);
}
// SZ bytes per lane from a buffer straight into LDS; the builtin exists for the device pass only
template <int SZ> __device__ __forceinline__ void k8_lds(__amdgpu_buffer_rsrc_t r, LK_LOCAL uint8_t * dst, uint32_t voff, uint32_t soff) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (SZ == 16) { __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LK_LOCAL void *) dst, 16, voff, soff, 0, 0); }
    else { __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LK_LOCAL void *) dst, 4, voff, soff, 0, 0); }
#else
    (void) r; (void) dst; (void) voff; (void) soff;
#endif
}

// a lane's bytes of one block. Q2_K: q = its 16 quant bytes, s = the 8 scale bytes of its half, dd = d and dmin. Q3_K (blocks
// start on 2-byte boundaries): aligned windows over the 16 quant bytes, the 16 high-bit bytes and the last 14 bytes
// (scales and d), sh = 0 or 2 the offset inside them.
template <int F> struct K8Raw;
template <> struct K8Raw<KF_Q2K> { u32x4 q; u32v2 s; uint32_t dd; };
template <> struct K8Raw<KF_Q3K> { u32x4 q, h, t; uint32_t q4, h4; };

template <int F> __device__ __forceinline__ void k8_load(const Src & b, uint32_t blk, int g, K8Raw<F> & w) {
    const uint32_t n = (uint32_t) g >> 1, h = (uint32_t) g & 1u;
    if constexpr (F == KF_Q2K) {   // scales[16] qs[64] d dmin
        Src s = b; s.vb += blk;
        w.q = ld128(s, 16 + 32 * n + 16 * h); w.s = ld64(s, 8 * n); w.dd = ld32(s, 80);
    } else {                       // hmask[32] qs[64] scales[12] d
        Src s = b; s.vb += blk & ~3u;   // (sh is the same for every field: their offsets are multiples of 4)
        w.q = ld128(s, 32 + 32 * n + 16 * h); w.q4 = ld32(s, 48 + 32 * n + 16 * h);
        w.h = ld128(s, 16 * h); w.h4 = ld32(s, 16 + 16 * h);
        w.t = ld128(s, 96);
    }
}

}  // namespace

template <int F>
__global__ void __launch_bounds__(K8_NT, 1) k_kq8_gemm(const PrefillArgs a) {
#pragma clang fp contract(off)
    constexpr int BS = kbytes<F>(), NB = K8_NB;
    constexpr bool Q3 = F == KF_Q3K;
    constexpr uint32_t ROWB = (uint32_t) (NB * BS);   // bytes of a row
    extern __shared__ __attribute__((aligned(16))) uint8_t k8_dyn[];
    LK_LOCAL uint8_t * lds = (LK_LOCAL uint8_t *) k8_dyn;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
    const int r = lane & 15, g = lane >> 4;
    const int col0 = a.col0, ncols = (a.col1 > 0 ? a.col1 : *gptr(a.ncols)) - col0, nrg = a.R / K8_ROWS;
    if ((int) blockIdx.x >= ncols * nrg) { return; }
    if (lds_addr(k8_dyn) & 0xFFFFu) {   // the scale lines' addressing needs a 64 KB aligned base
        if (threadIdx.x == 0) {
            __hip_atomic_fetch_or(gptr(a.err), 4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (a.herr) { __hip_atomic_store(gptr(a.herr), 4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
        }
        return;
    }
    const uint32_t lut = lds_addr(k8_dyn) | ((uint32_t) (lane & 31) << 3);
    if constexpr (Q3) {   // line i (scale i - 32): bytes (4 - u) * (i - 32), u = 0..7
        for (int p = threadIdx.x; p < 64 * 32; p += K8_NT) {
            const int sc = (p >> 5) - 32;
            uint32_t lo = 0, hi = 0;
            for (int u = 0; u < 4; ++u) { lo |= ((uint32_t) ((4 - u) * sc) & 255u) << (8 * u); hi |= ((uint32_t) (-u * sc) & 255u) << (8 * u); }
            reinterpret_cast<LK_LOCAL u32x2 *>(lds)[p] = (u32x2) { lo, hi };
        }
    }
    __syncthreads();
    const uint32_t sela = (g & 1) ? 0x01010101u : 0u;   // Q2_K: the byte of a scale word the lane's sub-blocks start at

    for (int it = blockIdx.x; it < ncols * nrg; it += gridDim.x) {
        const int col = col0 + it / nrg, rg = it % nrg;
        const u32x4 cv = *(const LK_GLOBAL u32x4 *) (a.cols + col);
        const bool routed = (int) cv.x >= 0;
        const int sb = (int) cv.y, sc = (int) cv.z;
        const uint8_t * Wm = routed ? a.w[0] + (size_t) (int) cv.w * a.estride : a.sh[0];
        const __amdgpu_buffer_rsrc_t rb = k8_rsrc(a.bq, 0x7fffffff), rd = k8_rsrc(a.bd, 0x7fffffff);
        Src src;
        src.rs = k8_rsrc(k8_uniform(Wm), (uint32_t) a.R * ROWB);
        src.vb = (uint32_t) r * ROWB;
        src.so = (uint32_t) (rg * K8_ROWS + wave * 16) * ROWB;
        const int ar0 = sb - a.arow0;
        auto run_item = [&](auto ntc) {
            constexpr int NT = decltype(ntc)::value;
            // activations: wave w copies token rows 4 w .. 4 w + 3 (w < 4 NT), lane L of row (L / 16) the row's chunk
            // (L % 16) ^ (row % 16); the block scales by the last wave
            const int row = 4 * wave + (lane >> 4);
            const uint32_t ob = (uint32_t) (ar0 + (row < sc ? row : 0)) * (NB * QK) + (uint32_t) (((lane & 15) ^ (row & 15)) << 4);
            const uint32_t od = (uint32_t) (ar0 + (lane < sc ? lane : 0)) * (NB * 4);
            auto load_b = [&](int j, int buf) {
                if (wave < 4 * NT) { k8_lds<16>(rb, lds + K8_X + buf * K8_BUF + wave * 1024, ob, j * QK); }
                if (wave == K8_W - 1) { k8_lds<4>(rd, lds + K8_DX + buf * 256, od, j * 4); }
            };
            kf4 acc[NT];
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) { acc[tt] = (kf4) { 0.f, 0.f, 0.f, 0.f }; }
            auto block = [&](const K8Raw<F> & w, auto par) {
                constexpr int buf = decltype(par)::value;   // the block's parity: buffer and (Q3_K) byte alignment
                // the lane's four operands: plane s of its bytes (sub-block 8 n + 2 s + h)
                ki4 wv[4];
                uint32_t mn[4];
                float dd, dm = 0.f;
                if constexpr (Q3) {
                    constexpr uint32_t sh = (uint32_t) (buf * BS) & 3u;
                    const uint32_t q[4] = { __builtin_amdgcn_alignbyte(w.q.y, w.q.x, sh), __builtin_amdgcn_alignbyte(w.q.z, w.q.y, sh),
                                            __builtin_amdgcn_alignbyte(w.q.w, w.q.z, sh), __builtin_amdgcn_alignbyte(w.q4, w.q.w, sh) };
                    const uint32_t hb[4] = { __builtin_amdgcn_alignbyte(w.h.y, w.h.x, sh), __builtin_amdgcn_alignbyte(w.h.z, w.h.y, sh),
                                             __builtin_amdgcn_alignbyte(w.h.w, w.h.z, sh), __builtin_amdgcn_alignbyte(w.h4, w.h.w, sh) };
                    const uint32_t a0 = __builtin_amdgcn_alignbyte(w.t.y, w.t.x, sh), a1 = __builtin_amdgcn_alignbyte(w.t.z, w.t.y, sh);
                    const uint32_t a2 = __builtin_amdgcn_alignbyte(w.t.w, w.t.z, sh);
                    dd = h2f((uint16_t) (sh ? w.t.w >> 16 : w.t.w));
                    const uint32_t n4 = (uint32_t) (g >> 1) * 4, s4 = 8u * (uint32_t) (g & 1) + n4;
                    // 6-bit scales j = 8 n + 2 s + h (kquant_device.h): s = 0, 1 at bits 0 and 16 of p01, s = 2, 3 of p23
                    const uint32_t p01 = ((a0 >> s4) & 0x000F000Fu) | (rotr(a2, s4 - 4u) & 0x00300030u);
                    const uint32_t p23 = ((a1 >> s4) & 0x000F000Fu) | (rotr(a2, s4 - 2u) & 0x00300030u);
                    const uint2 t[4] = { lload8(tab_addr<0>(p01, lut)), lload8(tab_addr<2>(p01, lut)), lload8(tab_addr<0>(p23, lut)), lload8(tab_addr<2>(p23, lut)) };
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const uint32_t u = ((q[i] >> (2 * s)) & 0x03030303u) | (rotr(hb[i], n4 + (uint32_t) s - 2u) & 0x04040404u);
                            wv[s][i] = (int) __builtin_amdgcn_perm(t[s].y, t[s].x, u);
                        }
                    }
                } else {
                    dd = h2f((uint16_t) (w.dd & 0xFFFFu)); dm = h2f((uint16_t) (w.dd >> 16));
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const uint32_t sw = s < 2 ? w.s.x : w.s.y, sel = sela + (s & 1 ? 0x02020202u : 0u);
                        const uint32_t b = __builtin_amdgcn_perm(sw, sw, sel);              // the sub-block's byte, four times
                        const uint32_t t = (uint32_t) __umul24(b & 15u, 0x030201u) << 8;    // bytes sc * {0, 1, 2, 3}
                        mn[s] = (b >> 4) & 0x0F0F0F0Fu;
#pragma unroll
                        for (int i = 0; i < 4; ++i) { wv[s][i] = (int) __builtin_amdgcn_perm(t, t, (w.q[i] >> (2 * s)) & 0x03030303u); }
                    }
                }
                // chunk 8 n + 2 s + h of the lane's token row at slot chunk ^ r: one address word per product, the tile and the
                // buffer in the instruction's offset
                const uint32_t xs = (uint32_t) r * QK | ((uint32_t) ((8 * (g >> 1) + (g & 1)) ^ r) << 4);
                __builtin_amdgcn_sched_barrier(0);
                // one token tile after the other, the next one's activations read while this one's products run
                ki4 x[2][4];
                kf4 d8[2];
                auto operand = [&](int tt) {
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        x[tt & 1][s] = __builtin_bit_cast(ki4, *(const LK_LOCAL u32x4 *) (size_t) ((xs ^ (uint32_t) (s << 5)) + (uint32_t) (K8_X + buf * K8_BUF + tt * 16 * QK)));
                    }
                    d8[tt & 1] = *(const LK_LOCAL kf4 *) (size_t) ((uint32_t) (K8_DX + buf * 256) + (uint32_t) (64 * tt + 16 * g));
                };
                operand(0);
#pragma unroll
                for (int tt = 0; tt < NT; ++tt) {
                    if (tt + 1 < NT) { operand(tt + 1); }
                    const ki4 z = { 0, 0, 0, 0 };
                    ki4 D = z, M = z;
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        D = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[tt & 1][s], wv[s], D, 0, 0, 0);
                        if constexpr (!Q3) {
                            const ki4 mv = { (int) mn[s], (int) mn[s], (int) mn[s], (int) mn[s] };
                            M = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[tt & 1][s], mv, M, 0, 0, 0);
                        }
                    }
                    const kf4 dx = d8[tt & 1];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if constexpr (Q3) { acc[tt][i] = acc[tt][i] - (dd * dx[i]) * (float) D[i]; }
                        else { acc[tt][i] = acc[tt][i] + ((dx[i] * dd) * (float) D[i] - (dx[i] * dm) * (float) M[i]); }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            K8Raw<F> w0, w1;
            load_b(0, 0);
            k8_load<F>(src, 0, g, w0);
            __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): block 0's activations are in LDS
            __syncthreads();
            auto step = [&](int j, auto par, const K8Raw<F> & cur, K8Raw<F> & ahead) {
                const int jn = j + 1 < NB ? j + 1 : NB - 1;   // the last step reloads its own block (unread)
                load_b(jn, (j + 1) & 1);                       // that buffer was last read in step j - 1, before its barrier
                k8_load<F>(src, (uint32_t) (jn * BS), g, ahead);
                __builtin_amdgcn_sched_barrier(0);
                block(cur, par);
                __builtin_amdgcn_s_waitcnt(0x0f70);            // vmcnt(0): block j + 1's activations have landed in LDS
                __builtin_amdgcn_s_barrier();
            };
#pragma unroll 1
            for (int j = 0; j < NB; j += 2) {
                step(j, std::integral_constant<int, 0>{}, w0, w1);
                step(j + 1, std::integral_constant<int, 1>{}, w1, w0);
            }
            const int orow = rg * K8_ROWS + wave * 16 + r;
            int t0 = 4 * g;
            __asm__ volatile("" : "+v"(t0));   // the output rows are formed here, not kept (and spilled) across the items
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int t = 16 * tt + t0 + i;
                    if (t < sc) { a.out[(size_t) (sb - a.orow0 + t) * a.R + orow] = acc[tt][i]; }
                }
            }
        };
        if (sc > 48) { run_item(std::integral_constant<int, 4>{}); }
        else if (sc > 32) { run_item(std::integral_constant<int, 3>{}); }
        else if (sc > 16) { run_item(std::integral_constant<int, 2>{}); }
        else { run_item(std::integral_constant<int, 1>{}); }
    }
}

bool kq8_gemm_takes(int fmt, int K, int R) { return (fmt == KF_Q2K || fmt == KF_Q3K) && K == K8_NB * QK && R % K8_ROWS == 0; }
hipError_t kq8_gemm_init() {
    const hipError_t e = hipFuncSetAttribute((const void *) k_kq8_gemm<KF_Q2K>, hipFuncAttributeMaxDynamicSharedMemorySize, K8_LDS);
    return e == hipSuccess ? hipFuncSetAttribute((const void *) k_kq8_gemm<KF_Q3K>, hipFuncAttributeMaxDynamicSharedMemorySize, K8_LDS) : e;
}
hipError_t launch_kq8_gemm(const PrefillArgs & a, int fmt, int grid, hipStream_t st) {
    if (grid < 1 || !kq8_gemm_takes(fmt, a.K, a.R) || !a.cols || !a.ncols || !a.bq || !a.bd || !a.out || !a.err || a.col0 < 0 ||
        ((reinterpret_cast<uintptr_t>(a.w[0]) | reinterpret_cast<uintptr_t>(a.sh[0]) | a.estride) & 3u)) {
        return hipErrorInvalidValue;
    }
    if (fmt == KF_Q2K) { k_kq8_gemm<KF_Q2K><<<grid, K8_NT, K8_LDS, st>>>(a); }
    else { k_kq8_gemm<KF_Q3K><<<grid, K8_NT, K8_LDS, st>>>(a); }
    return hipGetLastError();
}

}  // namespace lk
