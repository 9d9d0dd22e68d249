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
// and 16 (its offsets were a second product). The routed Q3_K down at 201 tokens: 678 us in fp16, 485 here with lanes that
// fetch their own pieces, 331 through coalesced windows, 270 with the ring of three and the next item's first block. What
// bounds it now is the VALU work of building operands: about 150 instructions a wave and block, four waves a SIMD, against
// 0.73 GB of weights and mins that pass at 2.7 TB/s.
//
// Work: an item is (column of up to 64 slots, 256 rows), one workgroup of 16 waves per CU takes them round-robin; wave w
// owns one 16-row tile. Lane (r, g), g = 2 n + h, holds of row r the quant bytes 32 n + 16 h .. + 15: the 16-weight
// sub-blocks 8 n + 2 s + h in its four bit planes s. Product s takes plane s: weights 128 n + 32 s + 16 h .. + 15 of the
// block, and the activation operand the same positions. The column's Q8_K rows go block by block from memory into
// XOR-swizzled LDS (direct loads, double-buffered, one block ahead), the weight bytes two blocks ahead.
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
constexpr int K8_DX = 64 * 256, K8_X = K8_DX + 1024, K8_BUF = K8_TT * 16 * QK, K8_W0 = K8_X + 2 * K8_BUF;
constexpr int K8_RING = 3, K8_LDS = K8_W0 + K8_W * K8_RING * 16 * 128;   // .. then every wave's weight windows
static_assert(K8_LDS <= 160 * 1024, "LDS budget");

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

// A wave's 16 rows of one block come through LDS: rows are 110 (84) byte blocks side by side, so lanes that fetched their own
// pieces would touch every cache line of the tile five times over, which bounded the first version (485 against 300 us at
// 201 tokens). Two direct loads copy, per row, the 128-byte window of eight 16-byte units that holds the block (window start:
// the block's offset rounded down to 16); unit u of row r sits at slot u ^ ((r / 2) % 8) of the row's 128 bytes, so the 16
// rows of a read hit 16 bank quads. The block's offset in its window, DL, is the same for every row; a field of 16 bytes is
// two units shifted by DL. (Units count from the matrix's base, which need only be 4-byte aligned, as the loads do.)
constexpr int K8_WB = 16 * 128;
template <int F, int J> constexpr int k8_delta() { return (J * kbytes<F>()) & 15; }
__device__ __forceinline__ uint32_t k8_slot(int r, int u) { return (uint32_t) (r * 128 + ((u ^ ((r >> 1) & 7)) << 4)); }
__device__ __forceinline__ u32x4 k8_read(uint32_t at) { return *(const LK_LOCAL u32x4 *) (size_t) at; }
// N words at byte DL of two adjacent units
template <int DL, int N> __device__ __forceinline__ void k8_shift(const u32x4 & a, const u32x4 & b, uint32_t (&o)[N]) {
    const uint32_t w[9] = { a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, 0u };
#pragma unroll
    for (int i = 0; i < N; ++i) {
        if constexpr ((DL & 3) == 0) { o[i] = w[DL / 4 + i]; }
        else { o[i] = __builtin_amdgcn_alignbyte(w[DL / 4 + i + 1], w[DL / 4 + i], DL & 3); }
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
    // the lane's units in its wave's windows: quants, high bits (Q2_K: scales), and the last field
    const uint32_t wb = lds_addr(k8_dyn) + (uint32_t) (K8_W0 + wave * K8_RING * K8_WB);
    constexpr int UQ = Q3 ? 2 : 1, UT = Q3 ? 6 : 5;
    const uint32_t aq0 = wb + k8_slot(r, UQ + g), aq1 = wb + k8_slot(r, UQ + 1 + g), ah0 = wb + k8_slot(r, Q3 ? (g & 1) : 0);
    const uint32_t ah1 = wb + k8_slot(r, Q3 ? (g & 1) + 1 : 1), at0 = wb + k8_slot(r, UT), at1 = wb + k8_slot(r, UT + 1);
    const uint32_t sela = (g & 1) ? 0x01010101u : 0u;   // Q2_K: the byte of a scale word the lane's sub-blocks start at

    // An item's place (uniform); the loads are aimed at one item at a time, and the last step of an item already loads block 0
    // of the next one. Activations: wave w copies token rows 4 w .. 4 w + 3, lane L of row (L / 16) the row's chunk (L % 16) ^
    // (row % 16); the block scales by the last wave. Weights: copy instruction i takes unit (L % 8) ^ .. of row 8 i + L / 8.
    struct Item { int e, sb, sc, rg; };   // e: the routed expert, or -1 for the shared one
    auto item_of = [&](int it) -> Item {
        const u32x4 cv = *(const LK_CONST u32x4 *) (a.cols + (col0 + it / nrg));
        return Item { (int) cv.x < 0 ? -1 : (int) cv.w, (int) cv.y, (int) cv.z, it % nrg };
    };
    const __amdgpu_buffer_rsrc_t rb = k8_rsrc(a.bq, 0x7fffffff), rd = k8_rsrc(a.bd, 0x7fffffff);
    __amdgpu_buffer_rsrc_t rw;
    uint32_t tile = 0, ob = 0, od = 0, ow[2];
    int ncopy = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) { const int row = 8 * i + (lane >> 3); ow[i] = (uint32_t) row * ROWB + (uint32_t) (((lane & 7) ^ ((row >> 1) & 7)) << 4); }
    auto aim = [&](const Item & t) {
        const uint8_t * Wm = t.e >= 0 ? a.w[0] + (size_t) t.e * a.estride : a.sh[0];
        rw = k8_rsrc(k8_uniform(Wm), (uint32_t) a.R * ROWB);   // past the matrix's end a load returns 0
        tile = (uint32_t) (t.rg * K8_ROWS + wave * 16) * ROWB;
        const int ar0 = t.sb - a.arow0, row = 4 * wave + (lane >> 4);
        ob = (uint32_t) (ar0 + (row < t.sc ? row : 0)) * (NB * QK) + (uint32_t) (((lane & 15) ^ (row & 15)) << 4);
        od = (uint32_t) (ar0 + (lane < t.sc ? lane : 0)) * (NB * 4);
        ncopy = 4 * ((t.sc + 15) >> 4);
    };
    auto load_w = [&](int j, int buf) {
        LK_LOCAL uint8_t * dst = lds + K8_W0 + (wave * K8_RING + buf) * K8_WB;
#pragma unroll
        for (int i = 0; i < 2; ++i) { k8_lds<16>(rw, dst + i * 1024, ow[i], tile + (uint32_t) ((j * BS) & ~15)); }
    };
    auto load_b = [&](int j, int buf) {
        if (wave < ncopy) { k8_lds<16>(rb, lds + K8_X + buf * K8_BUF + wave * 1024, ob, j * QK); }
        if (wave == K8_W - 1) { k8_lds<4>(rd, lds + K8_DX + buf * 256, od, j * 4); }
    };
    const int items = ncols * nrg;
    if ((int) blockIdx.x >= items) { return; }
    Item cur = item_of(blockIdx.x);
    aim(cur);
    load_b(0, 0);
    load_w(0, 0);
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): block 0 is in LDS
    __syncthreads();
    for (int it = blockIdx.x; it < items; it += gridDim.x) {
        const Item nxt = item_of(it + (int) gridDim.x < items ? it + (int) gridDim.x : it);   // (none: its loads are not read)
        const int sb = cur.sb, sc = cur.sc, rg = cur.rg;
        auto run_item = [&](auto ntc) {
            constexpr int NT = decltype(ntc)::value;
            kf4 acc[NT];
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) { acc[tt] = (kf4) { 0.f, 0.f, 0.f, 0.f }; }
            auto block = [&](auto jc) {
                constexpr int J = decltype(jc)::value, buf = J & 1, DL = k8_delta<F, J>();
                // the lane's four operands: plane s of its bytes (sub-block 8 n + 2 s + h)
                ki4 wv[4];
                uint32_t mn[4];
                float dd, dm = 0.f;
                constexpr uint32_t wo = (uint32_t) (J % K8_RING * K8_WB);
                if constexpr (Q3) {   // hmask[32] qs[64] scales[12] d
                    uint32_t q[4], hb[4], ts[4];
                    k8_shift<DL, 4>(k8_read(aq0 + wo), k8_read(aq1 + wo), q);
                    k8_shift<DL, 4>(k8_read(ah0 + wo), k8_read(ah1 + wo), hb);
                    k8_shift<DL, 4>(k8_read(at0 + wo), k8_read(at1 + wo), ts);
                    const uint32_t a0 = ts[0], a1 = ts[1], a2 = ts[2];
                    dd = h2f((uint16_t) ts[3]);
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
                } else {              // scales[16] qs[64] d dmin
                    uint32_t q[4], sc8[4], td[1];
                    k8_shift<DL, 4>(k8_read(aq0 + wo), k8_read(aq1 + wo), q);
                    k8_shift<DL, 4>(k8_read(ah0 + wo), k8_read(ah1 + wo), sc8);
                    const u32x4 tu = k8_read(at0 + wo);
                    k8_shift<DL, 1>(tu, tu, td);
                    dd = h2f((uint16_t) (td[0] & 0xFFFFu)); dm = h2f((uint16_t) (td[0] >> 16));
                    const uint32_t sw2[2] = { g >> 1 ? sc8[2] : sc8[0], g >> 1 ? sc8[3] : sc8[1] };
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const uint32_t sw = sw2[s >> 1], sel = sela + (s & 1 ? 0x02020202u : 0u);
                        const uint32_t b = __builtin_amdgcn_perm(sw, sw, sel);              // the sub-block's byte, four times
                        const uint32_t t = (uint32_t) __umul24(b & 15u, 0x030201u) << 8;    // bytes sc * {0, 1, 2, 3}
                        mn[s] = (b >> 4) & 0x0F0F0F0Fu;
#pragma unroll
                        for (int i = 0; i < 4; ++i) { wv[s][i] = (int) __builtin_amdgcn_perm(t, t, (q[i] >> (2 * s)) & 0x03030303u); }
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
                    // the fold belongs to this block (unrolled, the compiler would carry the sums of all eight to the end)
#pragma unroll
                    for (int i = 0; i < 4; ++i) { float v = acc[tt][i]; __asm__ volatile("" : "+v"(v)); acc[tt][i] = v; }
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            // Activations one block ahead, weights two (a ring of three windows; block 0 of an item comes with the last step
            // of the item before, block 1 in step 0): the wait of a step leaves the two newest weight copies outstanding.
            auto step = [&](auto jc) {
                constexpr int J = decltype(jc)::value;
                // the windows and buffers written here were last read in step J - 1, before its barrier
                if constexpr (J + 1 < NB) { load_b(J + 1, (J + 1) & 1); }
                else { aim(nxt); load_b(0, 0); load_w(0, 0); }
                if constexpr (J == 0) { load_w(1, 1); }
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (J + 2 < NB) { load_w(J + 2, (J + 2) % K8_RING); }
                __builtin_amdgcn_sched_barrier(0);
                block(jc);
                __builtin_amdgcn_s_waitcnt(0x0f70 | (J + 2 < NB ? 2 : 0));   // block J + 1 has landed in LDS
                __builtin_amdgcn_s_barrier();
            };
            step(std::integral_constant<int, 0>{}); step(std::integral_constant<int, 1>{});
            step(std::integral_constant<int, 2>{}); step(std::integral_constant<int, 3>{});
            step(std::integral_constant<int, 4>{}); step(std::integral_constant<int, 5>{});
            step(std::integral_constant<int, 6>{}); step(std::integral_constant<int, 7>{});
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
        cur = nxt;
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
