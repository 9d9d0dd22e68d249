// moe_prefill.hip -- the grouped IQ2_XXS x Q8_K expert GEMMs of a prefill batch on the matrix cores.
//
// Reference: fl_wide_moe (src/fused_layer.cu:540-561) runs tc_matvec<F_IQ2> (:178-202) per arena batch of <= 72 slots
// of <= 8 rows each with mma.m16n8k32 s8 tiles, then swiglu_q8 (:334-341) and the down pass; the semantics are ggml's
// mul_mat_id over IQ2_XXS x Q8_K (ggml_vec_dot_iq2_xxs_q8_K per output). Here one launch per class of columns covers
// every expert of the layer, or one launch both classes of a split table (k_split_gemm; launch_rules.h has the line):
//   * A column is up to PF_TOK = 112 dispatch slots of one expert (the shared expert's slots P .. P + n - 1 included; in a
//     split table SPLIT_TOK = 32, those of at most 8 on moe_few.h's kernel); an item is (column, row group). The workgroups
//     (one per CU: the tables fill most of the LDS) take the items round-robin.
//   * The weights are dequantised once per item into int8 MFMA operands. A scaled weight v = sign * grid * (2s + 1) is one
//     of 6 values per sub-block (three magnitudes, two signs) and has at most 11 bits, so it is taken as two int8 digits,
//     v = 64 h + l, |l| <= 32, |h| <= 21. The codebook table holds, per entry, 8 selector bytes (the magnitude's index
//     0..2), the sign table 8 bytes of 0 or 4; or-ed they select, with one v_perm_b32 per 4 weights and digit, among the 8
//     bytes of the sub-block's scale line (the digits of +-8, +-25, +-43 times 2s + 1, a 16-byte LDS line per scale
//     nibble). Lane (r, g) of a wave owns row r of a 16-row tile and the 16-byte chunk g of each block (sub-blocks 2g,
//     2g + 1), as the tiled layout stores them.
//   * The column's activations (the Q8_K bytes) are copied block by block into LDS with direct global->LDS loads,
//     double-buffered; v_mfma_i32_16x16x64_i8 forms, per 256-value block and digit, the exact int32 sum over a 16-token x
//     16-row tile (4 steps), and the block sum is 64 h + l in int32, converted to fp32 once (rounded to nearest even):
//     ggml's (float) of its int32 block sum.
//   * Each output then advances in block order, y += (d_w * d_x) * bsum, and ends * 0.125: the fp32 operations and their
//     order are those of ggml_vec_dot_iq2_xxs_q8_K, so every output is bit-identical to the CPU checker's.
//   * Gate/up tiles write h = silu(g) * u per slot; down tiles write o per slot (the combine runs after).
// The K index of an MFMA step is permuted consistently in both operands: step m of lane group g covers the 16 values
// 64 g + 16 m .. + 15 of the block, i.e. entries 2 (m % 2), 2 (m % 2) + 1 of sub-block 2 g + m / 2.
#include "moe_device.h"
#include "moe_kernels.h"
#include "moe_few.h"
#include <type_traits>

namespace lk {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

// Table image: selector lines (entry e: 32 copies of the 8 magnitude indices of grid[e]), sign lines (the 7 stored sign
// bits: 32 copies of 8 bytes 0 / 4), then the 16 scale lines {l of + magnitudes, l of -, h of +, h of -} (bytes 0..2).
// LDS: the tables, two buffers of the tokens' block scales, two activation buffers (16 NTM token rows of 256 bytes, each
// row's 16-byte chunks XOR-swizzled by the row).
constexpr int L_SEL = 0, L_SGN = 65536, L_SCL = TAB_BYTES, PTAB_BYTES = L_SCL + 256;
constexpr int L_DX = PTAB_BYTES;
static_assert(TAB_BYTES == L_SGN + 128 * 256, "the selector and sign lines have the decode image's geometry");

__global__ void k_ptab_image(uint32_t * img) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;   // dword index
    if (i >= PTAB_BYTES / 4) { return; }
    const int at = i * 4, line = at >> 8, half = i & 1;
    uint32_t v = 0;
    if (at < L_SGN) {
        const uint64_t gv = g_iq2xxs_grid[line];
        for (int k = 0; k < 4; ++k) {
            const uint32_t b = (uint32_t) (gv >> (32 * half + 8 * k)) & 255u;
            v |= (b == 8 ? 0u : b == 25 ? 1u : 2u) << (8 * k);
        }
    } else if (at < L_SCL) {
        const uint32_t s8 = ksigns8((uint32_t) (line - L_SGN / 256));
        for (int k = 0; k < 4; ++k) { v |= ((s8 >> (4 * half + k)) & 1u) << (8 * k + 2); }
    } else {
        const int s = (at - L_SCL) >> 4, word = i & 3, mags[3] = { 8, 25, 43 };
        for (int k = 0; k < 3; ++k) {
            const int m = mags[k] * (2 * s + 1), h = (m + 32) >> 6, l = m - 64 * h;
            const int d = word < 2 ? l : h;
            v |= ((uint32_t) ((word & 1) ? -d : d) & 255u) << (8 * k);
        }
    }
    img[i] = v;
}
hipError_t build_prefill_tables(uint4 * img, hipStream_t st) {
    k_ptab_image<<<(PTAB_BYTES / 4 + 255) / 256, 256, 0, st>>>(reinterpret_cast<uint32_t *>(img));
    return hipGetLastError();
}
size_t prefill_table_bytes() { return PTAB_BYTES; }

// Columns: the shared expert's slots first, then every active expert's slots. An expert's slots go into the fewest columns
// of at most tok slots, of equal size rounded up to 16 (the last one takes the rest). The routed columns are written class
// by class, each in act order. Block b writes table b.
// A split table (T.few) is cut on the device, since only the counts tell a prompt whose tokens spread over the experts from
// one whose tokens share a few: every column costs about its expert's bytes, whether it has 3 slots or 30, so columns of few
// slots waste little while most experts have at most T.few, and repeat the weights (and their decoding) where they have more.
// Narrow columns save the ones of 8 that they replace and cost rounds of their own (SPLIT_GAIN); with nothing else in the
// table they are taken anyway.
__global__ void __launch_bounds__(256) k_pf_cols(const int * __restrict__ act, const int * __restrict__ nact_p, const int * __restrict__ offsets,
                                                int P, const PfTable t0, const PfTable t1) {
    static_assert(PF_NCLS == 4, "two classes to a word");
    __shared__ uint32_t tot[4], part[2][4];
    const PfTable T = blockIdx.x ? t1 : t0;
    const int i = threadIdx.x, nact = *nact_p, n = T.n;
    auto cls = [&](int slots) -> int { return slots > 64 ? PF_BROAD : slots > 32 ? PF_WIDE : slots > T.few ? PF_NARROW : PF_FEW; };
    int e = 0, s0 = 0, cnt = 0, cols, size;
    if (i < nact) { e = act[i]; s0 = offsets[e]; cnt = offsets[e + 1] - s0; }
    bool fine = false, even = false;                    // every column cut at T.few; no column for the few kernel but rests
    auto cut = [&](int cnt, int tok, int & cols, int & size) {   // cols columns of size slots, the last one the rest
        if (fine) { tok = T.few; }
        cols = (cnt + tok - 1) / tok;
        size = cols > 0 ? min(tok, ((cnt + cols - 1) / cols + 15) / 16 * 16) : 0;
        if (even && cols > 1 && cnt - size * (cols - 1) <= T.few) { size = (cnt + cols - 1) / cols; }   // (then no rests either: one class)
    };
    if (T.few > 0 && T.tok > T.few) {
        // of cnt slots: the columns of T.few that narrow ones replace, and those
        auto narrow = [&](int cnt, int tok, int & replaced, int & cols) {
            int size;
            cut(cnt, tok, cols, size);
            const int rest = cols > 0 && cnt - size * (cols - 1) <= T.few ? 1 : 0;
            replaced = (cnt + T.few - 1) / T.few - rest; cols -= rest;
        };
        // three totals in one scan: those two, and the experts of at most T.few slots (a split table holds at most 3328 slots
        // of 256 experts: 672, 360 and 256)
        int r, m, rs, ms;
        narrow(cnt, T.tok, r, m);
        narrow(n, T.stok, rs, ms);
        const uint32_t w = wave_scan_u32((uint32_t) r | (uint32_t) m << 11 | (cnt > 0 && cnt <= T.few ? 1u << 22 : 0u));
        if ((i & 63) == 63) { tot[i >> 6] = w; }
        __syncthreads();
        const uint32_t t = tot[0] + tot[1] + tot[2] + tot[3];
        even = (t >> 22) == 0;
        fine = !even && (int) (t & 2047u) + rs < SPLIT_GAIN * (((int) (t >> 11 & 2047u) + ms + 15) / 16);
    }
    cut(cnt, T.tok, cols, size);
    int nk[PF_NCLS] = { 0, 0, 0, 0 };                   // this expert's columns of each class
    if (cols > 0) { nk[cls(size)] += cols - 1; nk[cls(cnt - size * (cols - 1))] += 1; }
    // inclusive scans over the experts, two classes to a word (a class has fewer than 2^16 columns)
    uint32_t sc[2], all[2] = { 0, 0 };
    for (int h = 0; h < 2; ++h) {
        sc[h] = wave_scan_u32((uint32_t) nk[2 * h] | (uint32_t) nk[2 * h + 1] << 16);
        if ((i & 63) == 63) { part[h][i >> 6] = sc[h]; }
    }
    __syncthreads();
    for (int h = 0; h < 2; ++h) {
        for (int w = 0; w < 4; ++w) { sc[h] += w < (i >> 6) ? part[h][w] : 0u; all[h] += part[h][w]; }
    }
    int nsh, ssize;
    cut(n, T.stok, nsh, ssize);
    int at[PF_NCLS], end = nsh;
    for (int k = 0; k < PF_NCLS; ++k) {
        at[k] = end + (int) (sc[k >> 1] >> (16 * (k & 1)) & 0xFFFFu) - nk[k];
        end += (int) (all[k >> 1] >> (16 * (k & 1)) & 0xFFFFu);
        if (i == 0) { T.ncols[PF_NCLS + 1 + k] = end; }
    }
    for (int c = 0; c < cols; ++c) {
        const int m = c < cols - 1 ? size : cnt - size * c;
        T.cols[at[cls(m)]++] = make_int4(i, s0 + size * c, m, e);
    }
    for (int c = i; c < nsh; c += 256) { T.cols[c] = make_int4(-1, P + ssize * c, min(ssize, n - ssize * c), 0); }
    if (i == 0) {
        T.ncols[0] = end;
        int ns[PF_NCLS] = { 0, 0, 0, 0 }, at2 = 0;
        if (nsh > 0) { ns[cls(ssize)] += nsh - 1; ns[cls(n - ssize * (nsh - 1))] += 1; }
        for (int k = 0; k < PF_NCLS; ++k) { at2 += ns[k]; T.ncols[1 + k] = at2; }
    }
}
hipError_t launch_prefill_cols(const int * act, const int * nact, const int * offsets, int P, const PfTable & t0, const PfTable & t1, hipStream_t st) {
    k_pf_cols<<<t1.cols ? 2 : 1, 256, 0, st>>>(act, nact, offsets, P, t0, t1);
    return hipGetLastError();
}

// Q8_K integers as fp16 (exact): the MFMA operand copy of an activation array
__global__ void __launch_bounds__(256) k_q8_to_h(const int8_t * __restrict__ q, _Float16 * __restrict__ h, int64_t n) {
    const int64_t i = ((int64_t) blockIdx.x * 256 + threadIdx.x) * 8;
    if (i >= n) { return; }
    const u32x2 v = *(const LK_GLOBAL u32x2 *) (q + i);
    h8 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) { o[k] = (_Float16) (int8_t) (v.x >> (8 * k)); o[4 + k] = (_Float16) (int8_t) (v.y >> (8 * k)); }
    *(LK_GLOBAL h8 *) (h + i) = o;
}
hipError_t launch_q8_to_h(const int8_t * q, _Float16 * h, int64_t n, hipStream_t st) {
    if (n <= 0) { return hipSuccess; }
    if (n % 8) { return hipErrorInvalidValue; }
    k_q8_to_h<<<(unsigned) ((n / 8 + 255) / 256), 256, 0, st>>>(q, h, n);
    return hipGetLastError();
}

// ---------------------------------------------------------------- the grouped GEMM
// NMAT = 2: gate/up (K = 7168, rows 2048, B rows = tokens, writes h); NMAT = 1: down (K = 2048, rows 7168, B rows =
// slots, writes o). W waves per workgroup, C 16-row tiles per wave, columns of at most 16 NTM slots:
//   * narrow (W 16, C 1, NTM 2): columns of at most 32 slots, four waves per SIMD (two tiles a wave spill);
//   * wide (W 8, C 2, NTM 4): 33..64 slots;
//   * broad (W 8, C 1, NTM 7): 65..112 slots, the dequantised weights of a tile serve up to seven token tiles (two row
//     tiles a wave spill).
// Bound: a wave's VALU work (72 instructions a tile and block for the digits, 20 a token tile for the fold) and its MFMAs
// (8 a token tile) share the SIMD's issue: narrow, at 512 tokens, VALU active 67 % of the busy cycles and matrix cores 21 %;
// broad, at 2048 hot ones, 53 and 35 %. The digits against the fp16 operands they
// replaced (92 + 16 instructions, twice the LDS bytes), then the registers held over the token tiles: the step at 512 tokens
// 1295 -> 1208 -> 1150 us, with 16 hot experts of 2048 tokens 3270 -> 3000 -> 2860; with the router's matrix cores and the
// down's next item ahead 1108 and 2660.
// With C = 2 a wave's tiles are the gate and up rows of one 16-row tile (gate/up: h forms in registers) or two row tiles
// (down); with C = 1 the gate waves hand g to the up waves through LDS. Every output is computed once, in the same
// arithmetic.
template <int NMAT, int NB, int W, int C, int NTM>
struct PfGeo {
    static constexpr int TPM = W * C / NMAT;                    // 16-row tiles per matrix in an item
    static constexpr int ROWS = TPM * 16, K = NB * QK;
    static constexpr int BUF = NTM * 16 * QK;                   // one activation buffer
    static constexpr int DXB = (NTM + 3) / 4 * 256;             // one buffer of block scales (64 tokens per copy)
    static constexpr int L_X = (L_DX + 2 * DXB + 1023) / 1024 * 1024;
    static constexpr bool XG = NMAT == 2 && C == 1;             // g goes through LDS: an area of its own, or the second
    static constexpr int XGB = XG ? W / 2 * 64 * NTM * 16 : 0;  // activation buffer when that is large enough
    static constexpr int L_G = XGB <= BUF ? L_X + BUF : L_X + 2 * BUF, LDS = L_X + 2 * BUF + (XGB <= BUF ? 0 : XGB);
    static_assert(LDS <= 160 * 1024 && W * C % NMAT == 0 && C <= 2 && W % 8 == 0, "prefill GEMM geometry");
    // the matrix and the 16-row tile (within the item) of combo c of wave w
    __device__ static constexpr int mat(int w, int c) { return C == NMAT ? c : NMAT == 1 ? 0 : w / (W / NMAT); }
    __device__ static constexpr int tile(int w, int c) { return C == NMAT ? w : NMAT == 1 ? w * C + c : w % (W / NMAT); }
};

// one block of one 16-row tile: the tiled chunk g of row r (qs) and d
struct PfW { u32x4 q; uint16_t d; };

// the columns of class CLS (those of the table's part, pf_runs): workgroup bid of gridDim.x
template <int NMAT, int NB, int W, int C, int NTM, int CLS>
__device__ __forceinline__ void pf_body(const PrefillArgs & a, LK_LOCAL uint8_t * lds, int bid) {
#pragma clang fp contract(off)
    using Geo = PfGeo<NMAT, NB, W, C, NTM>;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
    const PfRuns runs = pf_runs(a, CLS);
    const int nrg = a.R / Geo::ROWS;
    if (bid >= runs.count() * nrg) { return; }   // nothing to do: not even the tables
    if (!pf_base_ok(a, (uint32_t) (size_t) lds)) { return; }
    tables_fill(reinterpret_cast<const uint8_t *>(a.ptab), lds, threadIdx.x, W * 64);
    if (threadIdx.x < 16) { reinterpret_cast<LK_LOCAL u32x4 *>(lds + L_SCL)[threadIdx.x] = *(const LK_GLOBAL u32x4 *) (a.ptab + L_SCL / 16 + threadIdx.x); }
    const int r = lane & 15, g = lane >> 4;
    const uint32_t trg = (uint32_t) L_SEL | ((uint32_t) (lane & 31) << 3), trs = trg + (uint32_t) L_SGN;
    const size_t dreg = (size_t) (a.R / 64) * NB * 4096;   // d region offset of a tiled matrix
    __syncthreads();

    // An item's place: its column (uniform) and row group. The loads are aimed at one item at a time: buffer loads with a
    // scalar resource (base, no bounds that matter), a 32-bit lane offset and a scalar block offset, so no 64-bit per-lane
    // address lives in vector registers. AHEAD (the down's short rows: eight steps an item): the last step of an item already
    // loads block 0 of the next one (its wait was a tenth of the pass); the gate/up's 28 steps have no registers left for it.
    constexpr bool AHEAD = NMAT == 1;
    struct Item { int e, sb, sc, rg; };   // e: the routed expert, or -1 for the shared one
    auto item_of = [&](int it) -> Item {
        const u32x4 cv = *(const LK_CONST u32x4 *) (a.cols + runs.col(it / nrg));
        return Item { (int) cv.x < 0 ? -1 : (int) cv.w, (int) cv.y, (int) cv.z, it % nrg };
    };
    // The column's activations of block j go straight from memory into LDS buffer j % 2 (buffer loads to LDS: lane L's 16
    // bytes land at L * 16 of the instruction's 1 KB, no registers): copy instruction i covers token rows 4 i .. 4 i + 3,
    // i < 4 token tiles, taken by waves i % W; lane L of row (L / 16) takes the row's chunk (L % 16) ^ (row % 16) -- the
    // swizzle applied on the memory side. gfx950 serves a ds_read_b128 in four passes of 16 lanes (equal bit 5, equal bit
    // 4 ^ bit 3); lane (r, g) reads slot (4 g + m) ^ r of row r, so a pass holds 16 different slots. The tokens' block
    // scales follow, 64 tokens per instruction (waves W - 1, W - 2).
    constexpr int NI = (4 * NTM + W - 1) / W, ND = (NTM + 3) / 4;
    const __amdgpu_buffer_rsrc_t rb = pf_rsrc(a.bq), rd = pf_rsrc(a.bd);
    const uint32_t lq = (uint32_t) g * 1024 + (uint32_t) r * 16, ldo = (uint32_t) r * 2;
    const int dw0 = W - 1 - wave;                 // which 64 tokens' scales this wave copies (0 .. ND - 1)
    __amdgpu_buffer_rsrc_t uq[C], ud[C];          // the wave's tiles: qs / d bases of combo c (Geo::mat, Geo::tile)
    uint32_t ob[NI], od = 0;
    int ncopy = 0;                                // copy instructions of the column
    int rows[NI + 1];                             // the activation rows behind ob and od, read ahead of their use
    auto rows_of = [&](const Item & t) {
        const int n16 = (t.sc + 15) & ~15;
        auto slot = [&](int i) { return t.sb + (i < t.sc ? i : 0); };
        auto row = [&](int i) { const int s = slot(i); return NMAT == 2 ? (t.e >= 0 ? gptr(a.perm)[s] : s - a.P) : s; };
#pragma unroll
        for (int i = 0; i < NI; ++i) { const int q = 4 * (wave + W * i) + (lane >> 4); rows[i] = row(q < n16 ? q : 0); }
        rows[NI] = dw0 < ND ? row(64 * dw0 + lane) : 0;
    };
    auto aim = [&](const Item & t) {              // after rows_of(t)
        auto arow = [&](int v) { return (uint32_t) (NMAT == 2 && t.e >= 0 ? v / a.topk : v); };
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int q = 4 * (wave + W * i) + (lane >> 4);
            ob[i] = arow(rows[i]) * Geo::K + (uint32_t) (((lane & 15) ^ (q & 15)) << 4);
        }
        od = arow(rows[NI]) * (NB * 4);
        ncopy = 4 * ((t.sc + 15) >> 4);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int mat = Geo::mat(wave, c), ti = Geo::tile(wave, c);
            const uint8_t * Wm = t.e >= 0 ? a.w[mat] + (size_t) t.e * a.estride : a.sh[mat];
            const int row0 = t.rg * Geo::ROWS + ti * 16;   // a 16-row tile lies inside one 64-row group
            const int g64 = row0 >> 6, r0 = row0 & 63;
            uq[c] = pf_rsrc(pf_uniform(Wm + (size_t) g64 * NB * 4096 + r0 * 16));
            ud[c] = pf_rsrc(pf_uniform(Wm + dreg + (size_t) g64 * NB * 128 + r0 * 2));
        }
    };
    auto load_w = [&](int j, PfW (&w)[C]) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            w[c].q = __builtin_amdgcn_raw_buffer_load_b128(uq[c], lq, j * 4096, 2);   // nt: streamed once
            w[c].d = __builtin_amdgcn_raw_buffer_load_b16(ud[c], ldo, j * 128, 0);
        }
    };
    auto load_b = [&](int j, int buf) {
        LK_LOCAL uint8_t * dst = lds + Geo::L_X + buf * Geo::BUF;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            if (wave + W * i < ncopy) { buf_lds<16>(rb, dst + (wave + W * i) * 1024, ob[i], j * QK); }
        }
        if (dw0 < ND) { buf_lds<4>(rd, lds + L_DX + buf * Geo::DXB + dw0 * 256, od, j * 4); }
    };

    const int items = runs.count() * nrg;
    PfW w0[C], w1[C];
    Item cur = item_of(bid);
    auto begin = [&]() {
        rows_of(cur);
        aim(cur);
        load_w(0, w0);
        load_b(0, 0);
        __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): block 0's activations are in LDS
        __syncthreads();
    };
    if (AHEAD) { begin(); }
    for (int it = bid; it < items; it += (int) gridDim.x) {
        const Item nxt = item_of(it + (int) gridDim.x < items ? it + (int) gridDim.x : it);   // (none: its loads are not used)
        if (!AHEAD) { begin(); }
        const int sb = cur.sb, sc = cur.sc, rg = cur.rg;
        auto run_item = [&](auto ntc) {
            constexpr int NT = decltype(ntc)::value;   // token tiles of the column
            f4 acc[C][NT];
#pragma unroll
            for (int c = 0; c < C; ++c) { for (int tt = 0; tt < NT; ++tt) { acc[c][tt] = (f4) { 0.f, 0.f, 0.f, 0.f }; } }

            // A block's weights as MFMA operands: the low and the high digits of the C tiles (4 steps of 16 weights per lane)
            // and their d. The LDS reads of a step (two selector and two sign entries) are issued one step ahead of their
            // use, into the other of two register sets.
            i4 wl[C][4], wh[C][4];
            float dw[C];
            auto dequant = [&](const PfW (&w)[C]) {
                u32x4 dig[C];           // the scale line of the lane's sub-block in use (2 g, then 2 g + 1)
                uint32_t ms[C][2];
                auto digits = [&](int c, int h) {
                    const uint32_t sw = h ? w[c].q.w : w[c].q.y;
                    dig[c] = *(const LK_LOCAL u32x4 *) (size_t) __builtin_amdgcn_udot4((sw >> 7) & 0x01010101u, 0x80402010u, (uint32_t) L_SCL, false);
                };
                struct Lk { uint2 g0, g1, s0, s1; };
                auto lookup = [&](int m, int c, Lk & k) {
                    const uint32_t a0 = m < 2 ? w[c].q.x : w[c].q.z, a1 = ms[c][m >> 1];
                    if (m & 1) {
                        k.g0 = lload8(tab_addr<2>(a0, trg)); k.g1 = lload8(tab_addr<3>(a0, trg));
                        k.s0 = lload8(tab_addr<2>(a1, trs)); k.s1 = lload8(tab_addr<3>(a1, trs));
                    } else {
                        k.g0 = lload8(tab_addr<0>(a0, trg)); k.g1 = lload8(tab_addr<1>(a0, trg));
                        k.s0 = lload8(tab_addr<0>(a1, trs)); k.s1 = lload8(tab_addr<1>(a1, trs));
                    }
                };
#pragma unroll
                for (int c = 0; c < C; ++c) { digits(c, 0); ms[c][0] = w[c].q.y & SIGN_BITS; ms[c][1] = w[c].q.w & SIGN_BITS; dw[c] = h2f(w[c].d); }
                Lk k[2];
                lookup(0, 0, k[0]);
#pragma unroll
                for (int i = 0; i < 4 * C; ++i) {
                    const int m = i / C, c = i % C;
                    if (i + 1 < 4 * C) { lookup((i + 1) / C, (i + 1) % C, k[(i + 1) & 1]); }
                    const Lk & u = k[i & 1];
                    const uint32_t e[4] = { u.g0.x | u.s0.x, u.g0.y | u.s0.y, u.g1.x | u.s1.x, u.g1.y | u.s1.y };
                    const u32x4 d = dig[c];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        wl[c][m][q] = (int) __builtin_amdgcn_perm(d.y, d.x, e[q]);
                        wh[c][m][q] = (int) __builtin_amdgcn_perm(d.w, d.z, e[q]);
                    }
                    if (m == 1) { digits(c, 1); }
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            // The block's products with one token tile after the other: the next tile's activations are read and the
            // previous tile's sums folded while this one's MFMAs run. Fold, in block order: y += (d_w * d_x) * bsum; lane
            // (r, g) holds tokens 4 g + i of a tile.
            auto products = [&](int buf) {
                const uint32_t bx = (uint32_t) (Geo::L_X + buf * Geo::BUF) + (uint32_t) r * QK + (uint32_t) (((4 * g) ^ r) << 4);
                i4 x[2][4], D[2][C][2];
                f4 dx[2];
                auto operand = [&](int tt) {   // chunks (4 g + m) ^ r of the lane's token row
#pragma unroll
                    for (int m = 0; m < 4; ++m) { x[tt & 1][m] = __builtin_bit_cast(i4, *(const LK_LOCAL u32x4 *) (size_t) ((bx ^ (uint32_t) (m << 4)) + tt * 16 * QK)); }
                    dx[tt & 1] = *(const LK_LOCAL f4 *) (size_t) ((uint32_t) (L_DX + buf * Geo::DXB) + (uint32_t) (64 * tt + 16 * g));
                };
                auto fold = [&](int tt, int i, float dxi) {
#pragma unroll
                    for (int c = 0; c < C; ++c) {
                        const float b = (float) ((D[tt & 1][c][1][i] << 6) + D[tt & 1][c][0][i]);
                        acc[c][tt][i] = acc[c][tt][i] + (dw[c] * dxi) * b;
                    }
                };
                operand(0);
                f4 dp;
#pragma unroll
                for (int tt = 0; tt < NT; ++tt) {
                    if (tt > 0) { dp = dx[(tt - 1) & 1]; }
                    if (tt + 1 < NT) { operand(tt + 1); }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        const i4 z = (i4) { 0, 0, 0, 0 };
#pragma unroll
                        for (int c = 0; c < C; ++c) {
                            i4 (&d)[2] = D[tt & 1][c];
                            d[0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[tt & 1][m], wl[c][m], m == 0 ? z : d[0], 0, 0, 0);
                            d[1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[tt & 1][m], wh[c][m], m == 0 ? z : d[1], 0, 0, 0);
                        }
                        if (tt > 0) { fold(tt - 1, m, dp[m]); }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                dp = dx[(NT - 1) & 1];
#pragma unroll
                for (int i = 0; i < 4; ++i) { fold(NT - 1, i, dp[i]); }
            };

            // pipeline: weights and activations one block ahead (registers; the other of two LDS buffers)
            auto step = [&](int j, int jn, const PfW (&now)[C], PfW (&ahead)[C]) {
                load_b(jn, (j + 1) & 1);             // buffer (j + 1) % 2 was last read in step j - 1, before its barrier
                load_w(jn, ahead);
                __builtin_amdgcn_sched_barrier(0);   // nothing of the block moves above the loads
                dequant(now);
                products(j & 1);
                __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the next block's activations have landed in LDS (and its
                __builtin_amdgcn_s_barrier();        // weights are in): the barrier publishes them
            };
            static_assert(NB % 2 == 0, "two steps per trip");
#pragma unroll 1
            for (int j = 0; j < NB; j += 2) {
                const bool end = j == NB - 2;
                if (AHEAD && end) { rows_of(nxt); }
                step(j, j + 1, w0, w1);
                if (AHEAD && end) { aim(nxt); }
                step(j + 1, end ? (AHEAD ? 0 : NB - 1) : j + 2, w1, w0);   // (not ahead: a reload, which nobody reads)
            }

            // outputs: lane (r, g) holds tokens 4 g + i of each token tile for row r of each of its tiles
            if constexpr (Geo::XG) {
                // the gate waves leave 0.125 g in LDS (maybe in the second activation buffer, last read before the last step's
                // barrier and next filled in the next item's first step, after the second barrier here), the up waves form h
                // for the same tile
                LK_LOCAL f4 * xg = reinterpret_cast<LK_LOCAL f4 *>(lds + Geo::L_G);
                const int ti = Geo::tile(wave, 0);
                if (Geo::mat(wave, 0) == 0) {
#pragma unroll
                    for (int tt = 0; tt < NT; ++tt) { xg[(ti * NTM + tt) * 64 + lane] = 0.125f * acc[0][tt]; }
                }
                __syncthreads();
                f4 gt[NT];
#pragma unroll
                for (int tt = 0; tt < NT; ++tt) { gt[tt] = xg[(ti * NTM + tt) * 64 + lane]; }
                __syncthreads();
                if (Geo::mat(wave, 0) == 1) {
                    const int row = rg * Geo::ROWS + ti * 16 + r;
#pragma unroll
                    for (int tt = 0; tt < NT; ++tt) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int t = 16 * tt + 4 * g + i;
                            if (t < sc) {
                                const size_t o = (size_t) (sb + t) * a.R + row;
                                const float uv = 0.125f * acc[0][tt][i];
                                a.out[o] = det_silu(gt[tt][i]) * uv;
                                if (a.gdbg) { a.gdbg[o] = gt[tt][i]; a.udbg[o] = uv; }
                            }
                        }
                    }
                }
            } else {
                constexpr int RT = NMAT == 2 ? 1 : C;   // row tiles of the wave (gate/up: one, both matrices)
#pragma unroll
                for (int c = 0; c < RT; ++c) {
                    const int row = rg * Geo::ROWS + Geo::tile(wave, c) * 16 + r;
#pragma unroll
                    for (int tt = 0; tt < NT; ++tt) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int t = 16 * tt + 4 * g + i;
                            if (t < sc) {
                                const size_t o = (size_t) (sb + t) * a.R + row;
                                if (NMAT == 2) {
                                    const float gv = 0.125f * acc[0][tt][i], uv = 0.125f * acc[C - 1][tt][i];
                                    a.out[o] = det_silu(gv) * uv;
                                    if (a.gdbg) { a.gdbg[o] = gv; a.udbg[o] = uv; }
                                } else {
                                    a.out[o] = 0.125f * acc[c][tt][i];
                                }
                            }
                        }
                    }
                }
            }
        };
        if constexpr (NTM == 2) {
            if (sc > 16) { run_item(std::integral_constant<int, 2>{}); }
            else { run_item(std::integral_constant<int, 1>{}); }
        } else if constexpr (NTM == 4) {
            if (sc > 48) { run_item(std::integral_constant<int, 4>{}); }
            else { run_item(std::integral_constant<int, 3>{}); }
        } else {
            if (sc > 96) { run_item(std::integral_constant<int, 7>{}); }
            else if (sc > 80) { run_item(std::integral_constant<int, 6>{}); }
            else { run_item(std::integral_constant<int, 5>{}); }
        }
        cur = nxt;
    }
}

template <int NMAT, int NB, int W, int C, int NTM, int CLS>
__global__ void __launch_bounds__(W * 64, 1) k_pf_gemm(const PrefillArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t dyn_lds[];
    pf_body<NMAT, NB, W, C, NTM, CLS>(a, (LK_LOCAL uint8_t *) dyn_lds, (int) blockIdx.x);
}
template <int NMAT, int NB> __global__ void __launch_bounds__(FNT, 1) k_few_gemm(const PrefillArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t dyn_lds[];
    few_body<NMAT, NB>(a, (LK_LOCAL uint8_t *) dyn_lds);
}
// A split table's two classes in one launch, so that the table may choose on the device and an empty class costs no launch of
// its own (4.5 us each): the narrow columns first (a workgroup's whole items, from the last workgroup down), then the few
// ones (a wave's items, from the first workgroup up).
template <int NMAT, int NB> __global__ void __launch_bounds__(FNT, 1) k_split_gemm(const PrefillArgs a) {
    static_assert(FNT == 16 * 64, "both on 16 waves");
    extern __shared__ __attribute__((aligned(16))) uint8_t dyn_lds[];
    LK_LOCAL uint8_t * lds = (LK_LOCAL uint8_t *) dyn_lds;
    pf_body<NMAT, NB, 16, 1, 2, PF_NARROW>(a, lds, (int) (gridDim.x - 1 - blockIdx.x));
    __syncthreads();   // its tables and buffers are no longer read
    few_body<NMAT, NB>(a, lds);
}

template <int NMAT, int NB, int W, int C, int NTM, int CLS> struct PfKernel {
    using Geo = PfGeo<NMAT, NB, W, C, NTM>;
    static hipError_t setup() {
        return hipFuncSetAttribute((const void *) k_pf_gemm<NMAT, NB, W, C, NTM, CLS>, hipFuncAttributeMaxDynamicSharedMemorySize, Geo::LDS);
    }
    static void go(const PrefillArgs & a, int grid, hipStream_t st) { k_pf_gemm<NMAT, NB, W, C, NTM, CLS><<<grid, W * 64, Geo::LDS, st>>>(a); }
};
template <int NMAT, int NB> struct PfKernels {
    using Broad = PfKernel<NMAT, NB, 8, 1, 7, PF_BROAD>;
    using Wide = PfKernel<NMAT, NB, 8, 2, 4, PF_WIDE>;
    using Narrow = PfKernel<NMAT, NB, 16, 1, 2, PF_NARROW>;
    static constexpr int SPLIT_LDS = Narrow::Geo::LDS > F_LDS ? Narrow::Geo::LDS : F_LDS;
    static hipError_t setup() {
        hipError_t e = Broad::setup();
        if (e == hipSuccess) { e = Wide::setup(); }
        if (e == hipSuccess) { e = Narrow::setup(); }
        if (e == hipSuccess) { e = hipFuncSetAttribute((const void *) k_split_gemm<NMAT, NB>, hipFuncAttributeMaxDynamicSharedMemorySize, SPLIT_LDS); }
        return e == hipSuccess ? hipFuncSetAttribute((const void *) k_few_gemm<NMAT, NB>, hipFuncAttributeMaxDynamicSharedMemorySize, F_LDS) : e;
    }
    static bool rows_ok(int R) { return R % Broad::Geo::ROWS == 0 && R % Wide::Geo::ROWS == 0 && R % Narrow::Geo::ROWS == 0 && R % 64 == 0; }
    static void go(const PrefillArgs & a, int grid, hipStream_t st) {   // classes that cannot occur are not launched
        if (a.few > 0) {
            if (a.most > a.few) { k_split_gemm<NMAT, NB><<<grid, FNT, SPLIT_LDS, st>>>(a); }
            else { k_few_gemm<NMAT, NB><<<grid, FNT, F_LDS, st>>>(a); }
            return;
        }
        if (a.most > 64) { Broad::go(a, grid, st); }
        if (a.most > 32) { Wide::go(a, grid, st); }
        Narrow::go(a, grid, st);
    }
};
hipError_t prefill_init() {
    const hipError_t e = PfKernels<2, 28>::setup();
    return e == hipSuccess ? PfKernels<1, 8>::setup() : e;
}

// the kernels of the table's classes over the columns of its part (a.part), each taking its own
hipError_t launch_prefill_gemm(const PrefillArgs & a, int grid, hipStream_t st) {
    if (grid < 1 || !a.ptab || !a.tab || !a.cols || !a.ncols || !a.bq || !a.bd || !a.out || !a.err || a.most < 1 || (a.few != 0 && a.few != FEW_TOK)) {
        return hipErrorInvalidValue;
    }
    if (a.nmat == 2) {
        if (a.K != 28 * QK || !PfKernels<2, 28>::rows_ok(a.R) || !a.w[0] || !a.w[1] || !a.sh[0] || !a.sh[1] || !a.perm) { return hipErrorInvalidValue; }
        PfKernels<2, 28>::go(a, grid, st);
    } else if (a.nmat == 1) {
        if (a.K != 8 * QK || !PfKernels<1, 8>::rows_ok(a.R) || !a.w[0] || !a.sh[0]) { return hipErrorInvalidValue; }
        PfKernels<1, 8>::go(a, grid, st);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace lk
