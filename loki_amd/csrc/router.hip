// router.hip -- the DeepSeek-V3/R1 grouped sigmoid router on the device (no host round-trip).
//
// Reference: router_probs / router_topk (src/fused_layer.cu:313-332, launched at :506) and the ggml graph
// (src/server_core_fused.cpp:646-650) compute p = sigmoid(W x), take the top-8 of p + bias with ties to the lower index,
// and weight w_k = p[sel_k] / max(sum p[sel], 2^-14) * 2.5. This build adds the grouped rule the task names (8 groups of
// 32 experts; a group's score is the sum of its two best biased scores; the top-4 groups stay eligible), which reduces
// to the reference's rule with n_group = topk_group = 1.
//
// Logit contract (shared bit for bit with the CPU checker, moe_device.h): 256 chunks of K/256 products, each summed in
// order in fp64 from exact fp32 x fp32 products, a fixed pairwise tree over the chunk sums, one rounding to fp32. The
// sigmoid uses the fp64 exp contract of moe_common.h. Selection and weights are plain fp32 compares, adds and one
// correctly rounded division, so sel and wts are bit-identical to the checker's.
#include "moe_device.h"
#include "moe_kernels.h"

namespace lk {

constexpr int RT = 8;   // tokens per router wave

// K other than 7168: one wave per (expert, 8-token tile); every token's logit is a full wave reduction (logit_tree)
__global__ void __launch_bounds__(64) k_router_logits(const float * __restrict__ W, const float * __restrict__ x, int n, int n_exp, int K,
                                                      float * __restrict__ logits) {
    const int e = blockIdx.x, t0 = blockIdx.y * RT;
    const int nt = min(RT, n - t0);
    for (int t = 0; t < nt; ++t) {
        double s[4];
        logit_chunks_any(W + (size_t) e * K, x + (size_t) (t0 + t) * K, K, s);
        const double tot = logit_tree(s);
        if (threadIdx.x == 0) { logits[(size_t) (t0 + t) * n_exp + e] = (float) tot; }
    }
}

// A few tokens (K = 7168, n < RM_MIN): one workgroup (4 waves) per expert; thread c owns chunk c (28 values) of every
// token and keeps its 28 weights in registers. Per token the chunk sum runs in element order with v_fma_f64 (exact
// products, one rounding each), tree levels 1-6 are lane butterflies inside the wave (chunks 64 q .. 64 q + 63 of wave
// q), and levels 7-8 add the four waves' totals as (q0 + q1) + (q2 + q3) through LDS. Four tokens per pass.
constexpr int RW_MAXN = RM_MIN - 1;
__device__ __forceinline__ void router_wg_logits(const float * __restrict__ W, const float * __restrict__ x, int n, int n_exp,
                                                 float * __restrict__ logits, double (*part)[4]) {
#pragma clang fp contract(off)
    constexpr int CL = 28;
    const int e = blockIdx.x, c = threadIdx.x, q = c >> 6, lane = c & 63;
    float wv[CL];
#pragma unroll
    for (int i = 0; i < CL / 4; ++i) {
        const float4 v = gloadf4(W + (size_t) e * 7168 + CL * c + 4 * i);
        wv[4 * i] = v.x; wv[4 * i + 1] = v.y; wv[4 * i + 2] = v.z; wv[4 * i + 3] = v.w;
    }
    for (int t0 = 0; t0 < n; t0 += 4) {
        double sv[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            sv[k] = 0.0;
            if (t0 + k < n) {
                const float * xr = x + (size_t) (t0 + k) * 7168 + CL * c;
#pragma unroll
                for (int i = 0; i < CL / 4; ++i) {
                    const float4 v = gloadf4(xr + 4 * i);
                    const float xv[4] = { v.x, v.y, v.z, v.w };
#pragma unroll
                    for (int j = 0; j < 4; ++j) { sv[k] = __builtin_fma((double) xv[j], (double) wv[4 * i + j], sv[k]); }
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) { sv[k] = sv[k] + __shfl_xor(sv[k], o); }
        }
        if (lane == 0) {
#pragma unroll
            for (int k = 0; k < 4; ++k) { if (t0 + k < n) { part[t0 + k][q] = sv[k]; } }
        }
    }
    __syncthreads();
    if (c < n) { logits[(size_t) c * n_exp + e] = (float) ((part[c][0] + part[c][1]) + (part[c][2] + part[c][3])); }
}
__global__ void __launch_bounds__(256) k_router_wg(const float * __restrict__ W, const float * __restrict__ x, int n, int n_exp,
                                                   float * __restrict__ logits) {
    __shared__ double part[RW_MAXN][4];
    router_wg_logits(W, x, n, n_exp, logits, part);
}

// A few tokens (n <= RF_MAXN): k_router_wg's logits, then k_router_select's rule for every token in the workgroup that
// finishes last (wave q selects tokens q, q + 4, ..), so the routing is one launch. The logits reach that workgroup as
// epoch-tagged words tl [n][n_exp] (agent-scope stores and loads, polled until they carry this launch's epoch) and the
// workgroups count themselves on cnt (zero before the launch, reset by the last one): no memory fences, which cost an
// L2 write-back per workgroup. Wave 0 writes every token's picks, then (done != null) one system-scope release and
// done = epoch, so the host can read them from host memory without waiting for the stream. A poll that times out
// (stores that never land) leaves the picks -1.
constexpr int RF_MAXN = 8, RF_POLL = 1 << 20;
__global__ void __launch_bounds__(256) k_router_wg_sel(const float * __restrict__ W, const float * __restrict__ x, int n, int n_exp,
                                                       float * __restrict__ logits, const float * __restrict__ bias, int n_group,
                                                       int topk_group, int topk, float scale, int keep, float renorm,
                                                       float * __restrict__ probs, int * __restrict__ sel, float * __restrict__ wts,
                                                       uint64_t * tl, unsigned epoch, unsigned * cnt, unsigned * done, int * err,
                                                       int * herr) {
    __shared__ double part[RF_MAXN][4];
    __shared__ float scr[4][NEXP_MAX + 2 * 64];
    __shared__ int so[RF_MAXN][MAXK]; __shared__ float wo[RF_MAXN][MAXK];
    __shared__ unsigned last;
    router_wg_logits(W, x, n, n_exp, logits, part);
    const int e0 = blockIdx.x, c = threadIdx.x;
    if (c < n) {   // the same logit again as a tagged word (part[] is final after router_wg_logits' barrier)
        const float v = (float) ((part[c][0] + part[c][1]) + (part[c][2] + part[c][3]));
        __hip_atomic_store(gptr(tl) + (size_t) c * n_exp + e0, ((uint64_t) epoch << 32) | __builtin_bit_cast(uint32_t, v), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (c == 0) { last = atomicAdd(cnt, 1u) == gridDim.x - 1; }
    __syncthreads();
    if (!last) { return; }
    const int q = c >> 6, lane = c & 63;
    if (c == 0) { *cnt = 0u; }
    float bv[4];
    load_bias(bias, n_exp, bv);
    for (int t = q; t < n; t += 4) {
        uint64_t w[4];
        bool ok = false;
        for (int it = 0; it < RF_POLL && !ok; ++it) {
            ok = true;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = 4 * lane + j;
                w[j] = e < n_exp ? __hip_atomic_load(gptr(tl) + (size_t) t * n_exp + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
                ok = ok && (e >= n_exp || (unsigned) (w[j] >> 32) == epoch);
            }
            ok = __ballot(!ok) == 0;
            if (!ok) { __builtin_amdgcn_s_sleep(1); }
        }
        if (!ok) {   // unreachable unless stores are lost: no picks rather than wrong ones, and the error reported
            if (lane < keep) { so[t][lane] = -1; wo[t][lane] = 0.f; }
            if (lane == 0) {
                if (err) { __hip_atomic_fetch_or(gptr(err), 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
                if (herr) { __hip_atomic_store(gptr(herr), 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
            }
            continue;
        }
        float lg[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) { lg[j] = __builtin_bit_cast(float, (uint32_t) w[j]); }
        select_token(lg, bv, n_exp, n_group, topk_group, topk, scale, scr[q], so[t], wo[t], probs ? probs + (size_t) t * n_exp : nullptr,
                     keep, renorm);
    }
    __syncthreads();
    if (q == 0) {
        for (int i = lane; i < n * keep; i += 64) { sel[i] = so[i / keep][i % keep]; wts[i] = wo[i / keep][i % keep]; }
        if (done) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");   // system scope: the picks before the word
            if (lane == 0) { __hip_atomic_store(gptr(done), epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
        }
    }
}

// Prefill batches (K = 7168): the chunk sums on the fp64 matrix cores. v_mfma_f64_16x16x4_f64 adds its four products to
// the accumulator one after the other in K order, each by one fma (checked on the device against a sequential fma chain
// over random and cancelling data: no bit differs), and an fp32 x fp32 product is exact in fp64: seven of them are one
// chunk of the contract. Bound by the matrix cores' fp64 rate (64 clocks per product and SIMD, the VALU's fma rate,
// without its operand traffic): the VALU tiles this replaces took 338 us at 2048 tokens and 102 at 512.
//   * A workgroup (8 waves) owns 32 tokens x 32 experts and 1 / KS of the chunks (blockIdx.z); wave w takes CPW = 256 / (8
//     KS) consecutive chunks for the whole tile (2 x 2 tiles of 16 x 16).
//   * Operands come straight from memory: lane (r, g) loads 16 bytes of row r, piece 4 q + g of the row's 4-value pieces,
//     so an instruction covers 16 rows x 64 bytes; a 4 x 4 transpose over the lane groups (two v_permlane32_swap, two
//     v_permlane16_swap) gives the operands of products 4 q .. 4 q + 3. Four chunks are seven such loads per operand
//     tile; the next one is in flight while one is used.
//   * The contract's pairwise tree runs in registers as the chunks arrive, its next three levels over the workgroup's
//     waves through LDS, the levels over the KS parts in the selection (launch_router_select), which rounds to fp32.
typedef double d4 __attribute__((ext_vector_type(4)));
typedef float rf4 __attribute__((ext_vector_type(4)));
constexpr int RM_W = 8, RM_LDS = RM_W * 16 * 64 * 8;
struct RmAcc { d4 v[2][2]; };   // [token tile][expert tile]: lane (r, g) holds expert r, tokens g + 4 i
__device__ __forceinline__ void rm_add(RmAcc & d, const RmAcc & l, const RmAcc & r) {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < 2; ++i) { for (int j = 0; j < 2; ++j) { d.v[i][j] = l.v[i][j] + r.v[i][j]; } }
}
__device__ __forceinline__ void rm_transpose(float & a0, float & a1, float & a2, float & a3) {
    __asm__ volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %2\n\tv_permlane32_swap_b32 %1, %3\n\ts_nop 1\n\t"
                     "v_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\ts_nop 1" : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3));
}
template <int KS>
__global__ void __launch_bounds__(RM_W * 64, 1) k_router_mfma(const float * __restrict__ W, const float * __restrict__ x, int n, int n_exp,
                                                              double * __restrict__ part2, float * __restrict__ logits) {
#pragma clang fp contract(off)
    constexpr int K = 7168, CPW = 256 / (RM_W * KS), G4 = CPW / 4, LG = G4 == 8 ? 3 : G4 == 4 ? 2 : G4 == 2 ? 1 : 0;
    static_assert(G4 >= 1 && G4 == (1 << LG), "slices of 4, 8, 16 or 32 chunks");
    extern __shared__ __attribute__((aligned(16))) uint8_t rm_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id(), r = lane & 15, g = lane >> 4;
    // consecutive workgroups go to the 8 XCDs in turn: with 8 expert tiles, those of one token tile are put on one XCD, so
    // its L2 serves the tokens to all of them (token tiles past a multiple of 8 keep the plain order)
    int tt = blockIdx.y, et = blockIdx.x;
    if (gridDim.x == 8 && tt < (int) gridDim.y / 8 * 8) { et = blockIdx.y & 7; tt = (int) (blockIdx.y & ~7u) + (int) blockIdx.x; }
    const int tb = tt * 32, eb = et * 32;
    const int c0 = ((int) blockIdx.z * RM_W + wave) * CPW;
    const float * src[4];   // x rows of the two token tiles, W rows of the two expert tiles (rows past the end repeat row 0)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int t = tb + 16 * k + r, e = eb + 16 * k + r;
        src[k] = x + (size_t) (t < n ? t : 0) * K + 28 * c0 + 4 * g;
        src[2 + k] = W + (size_t) (e < n_exp ? e : 0) * K + 28 * c0 + 4 * g;
    }
    rf4 raw[2][4];
    auto fetch = [&](int q, int b) {   // quad q of 16 values: the lane's piece of each operand row
#pragma unroll
        for (int k = 0; k < 4; ++k) { raw[b][k] = *(const LK_GLOBAL rf4 *) (src[k] + 16 * q); }
    };
    RmAcc pend[LG + 1], node, ev, l1;
    fetch(0, 0);
#pragma unroll 1
    for (int g4 = 0; g4 < G4; ++g4) {   // four chunks: 28 products, 7 quads
        RmAcc acc;
#pragma unroll
        for (int q = 0; q < 7; ++q) {
            // the quads of a trip are 7: the buffer parity runs over q, the first quad of the next trip goes to buffer 1
            // (q = 6 is in buffer 0) and is moved to 0 at the end of the trip
            fetch(min(7 * g4 + q + 1, 7 * G4 - 1), (q + 1) & 1);
            rf4 (&c)[4] = raw[q & 1];
            float p[4][4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                p[k][0] = c[k][0]; p[k][1] = c[k][1]; p[k][2] = c[k][2]; p[k][3] = c[k][3];
                rm_transpose(p[k][0], p[k][1], p[k][2], p[k][3]);
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int st = 4 * q + s, ch = st / 7;
                const d4 z = (d4) { 0.0, 0.0, 0.0, 0.0 };
#pragma unroll
                for (int i = 0; i < 2; ++i) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        acc.v[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64((double) p[i][s], (double) p[2 + j][s], st % 7 == 0 ? z : acc.v[i][j], 0, 0, 0);
                    }
                }
                if (st % 7 == 6) {
                    if (ch == 0) { ev = acc; }
                    else if (ch == 1) { rm_add(l1, ev, acc); }
                    else if (ch == 2) { ev = acc; }
                    else { rm_add(node, ev, acc); rm_add(node, l1, node); }
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) { raw[0][k] = raw[1][k]; }
        // levels above 4 chunks: binary counter over the groups
#pragma unroll
        for (int l = 0; l < LG; ++l) {
            if (!((g4 >> l) & 1)) { pend[l] = node; break; }
            rm_add(node, pend[l], node);
        }
    }
    // the next three levels over the workgroup's waves, pairwise in slice order: output o of the lane by wave o % 8
    double * part = reinterpret_cast<double *>(rm_lds);   // [8 waves][16][64]
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int k = 0; k < 4; ++k) { part[(wave * 16 + (2 * i + j) * 4 + k) * 64 + lane] = node.v[i][j][k]; }
        }
    }
    __syncthreads();
    for (int o = wave; o < 16; o += RM_W) {
        double v[RM_W];
#pragma unroll
        for (int w = 0; w < RM_W; ++w) { v[w] = part[(w * 16 + o) * 64 + lane]; }
#pragma unroll
        for (int w = 1; w < RM_W; w *= 2) {
#pragma unroll
            for (int j = 0; j + w < RM_W; j += 2 * w) { v[j] = v[j] + v[j + w]; }
        }
        const int t = tb + 16 * (o >> 3) + g + 4 * (o & 3), e = eb + 16 * ((o >> 2) & 1) + r;
        if (t < n && e < n_exp) {
            if constexpr (KS == 1) { logits[(size_t) t * n_exp + e] = (float) v[0]; }
            else { part2[((size_t) blockIdx.z * n + t) * n_exp + e] = v[0]; }
        }
    }
}

size_t router_part_doubles(int n, int n_exp, int K) { return (size_t) router_parts(n, n_exp, K) * n * n_exp; }

hipError_t launch_router_logits(const float * W, const float * x, int n, int n_exp, int K, float * logits, double * part2, hipStream_t st) {
    if (n <= 0) { return hipSuccess; }
    if (K % 1024 != 0) { return hipErrorInvalidValue; }
    if (part2) {
        const dim3 grid((n_exp + 31) / 32, (n + 31) / 32, router_parts(n, n_exp, K));
        switch (grid.z) {
        case 8: k_router_mfma<8><<<grid, RM_W * 64, RM_LDS, st>>>(W, x, n, n_exp, part2, logits); break;
        case 4: k_router_mfma<4><<<grid, RM_W * 64, RM_LDS, st>>>(W, x, n, n_exp, part2, logits); break;
        case 2: k_router_mfma<2><<<grid, RM_W * 64, RM_LDS, st>>>(W, x, n, n_exp, part2, logits); break;
        default: return hipErrorInvalidValue;
        }
        return hipGetLastError();
    }
    if (K == 7168 && n >= RM_MIN) {
        k_router_mfma<1><<<dim3((n_exp + 31) / 32, (n + 31) / 32), RM_W * 64, RM_LDS, st>>>(W, x, n, n_exp, nullptr, logits);
        return hipGetLastError();
    }
    if (K == 7168) {
        k_router_wg<<<dim3(n_exp), 256, 0, st>>>(W, x, n, n_exp, logits);
        return hipGetLastError();
    }
    k_router_logits<<<dim3(n_exp, (n + RT - 1) / RT), 64, 0, st>>>(W, x, n, n_exp, K, logits);
    return hipGetLastError();
}

// one wave per token; lane l holds experts 4l..4l+3 (n_exp <= 256); the rule is select_token's (moe_device.h), with
// keep entries per token written (keep = topk: all of them). KS > 0: the logits arrive as KS parts of the contract's tree
// (k_router_mfma), added pairwise in order and rounded here, and are written out too.
template <int KS>
__global__ void __launch_bounds__(64) k_router_select(float * __restrict__ logits, const double * __restrict__ part2, const float * __restrict__ bias, int n, int n_exp,
                                                      int n_group, int topk_group, int topk, float scale, int keep, float renorm,
                                                      float * __restrict__ probs, int * __restrict__ sel, float * __restrict__ wts) {
    __shared__ float scr[NEXP_MAX + 2 * 64];
    __shared__ int so[MAXK]; __shared__ float wo[MAXK];
    const int t = blockIdx.x, lane = threadIdx.x;
    float lg[4], bv[4];
    load_bias(bias, n_exp, bv);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = 4 * lane + j;
        if constexpr (KS == 0) { lg[j] = e < n_exp ? logits[(size_t) t * n_exp + e] : 0.f; }
        else {
            double v[KS];
#pragma unroll
            for (int k = 0; k < KS; ++k) { v[k] = e < n_exp ? part2[((size_t) k * n + t) * n_exp + e] : 0.0; }
#pragma unroll
            for (int w = 1; w < KS; w *= 2) {
#pragma unroll
                for (int k = 0; k + w < KS; k += 2 * w) { v[k] = v[k] + v[k + w]; }
            }
            lg[j] = (float) v[0];
            if (e < n_exp) { logits[(size_t) t * n_exp + e] = lg[j]; }
        }
    }
    select_token(lg, bv, n_exp, n_group, topk_group, topk, scale, scr, so, wo, probs ? probs + (size_t) t * n_exp : nullptr, keep, renorm);
    lds_visible();
    if (lane < keep) { sel[(size_t) t * keep + lane] = so[lane]; wts[(size_t) t * keep + lane] = wo[lane]; }
}

static bool select_rule_ok(int n_exp, int n_group, int topk_group, int topk, int keep) {
    return !(n_exp > NEXP_MAX || n_exp % n_group || topk > MAXK || topk_group > n_group || topk > topk_group * (n_exp / n_group) ||
             n_exp / n_group < 2 || n_group > 64 || keep > topk);
}

bool router_fused_ok(int n, int K) { return n >= 1 && n <= RF_MAXN && K == 7168; }

hipError_t launch_router_fused(const float * W, const float * x, int n, int n_exp, int K, float * logits, const float * bias, int n_group,
                               int topk_group, int topk, float scale, float * probs, int * sel, float * wts, uint64_t * tl,
                               unsigned epoch, unsigned * cnt, unsigned * done, int * err, int * herr, hipStream_t st, int keep,
                               float renorm) {
    if (keep <= 0) { keep = topk; }
    if (!router_fused_ok(n, K) || !cnt || !tl || epoch == 0 || !select_rule_ok(n_exp, n_group, topk_group, topk, keep)) {
        return hipErrorInvalidValue;
    }
    k_router_wg_sel<<<dim3(n_exp), 256, 0, st>>>(W, x, n, n_exp, logits, bias, n_group, topk_group, topk, scale, keep, renorm, probs, sel,
                                                 wts, tl, epoch, cnt, done, err, herr);
    return hipGetLastError();
}

// --share-experts keep of n rows (keep_share_rows): every thread adds its rows' own picks to the LDS set, then wave 0
// runs the rows in order
__global__ void __launch_bounds__(256) k_keep_share(const int * __restrict__ sel8, const float * __restrict__ w8, int n, int topk, int ke,
                                                    float renorm, int * __restrict__ sel, float * __restrict__ wts) {
    __shared__ unsigned U[8];
    if (threadIdx.x < 8) { U[threadIdx.x] = 0u; }
    __syncthreads();
    const int own = ke < 2 ? ke : 2;
    for (int i = threadIdx.x; i < n; i += 256) {
        for (int k = 0; k < topk; ++k) {
            const float wk = gptr(w8)[(size_t) i * topk + k];
            int r = 0;
            for (int j = 0; j < topk; ++j) { const float o = gptr(w8)[(size_t) i * topk + j]; r += (o > wk || (o == wk && j < k)) ? 1 : 0; }
            if (r < own) { const int e = gptr(sel8)[(size_t) i * topk + k]; atomicOr(&U[(e >> 5) & 7], 1u << (e & 31)); }
        }
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        keep_share_rows(gptr(sel8), gptr(w8), n, topk, ke, renorm, gptr(sel), gptr(wts), (LK_LOCAL unsigned *) U, false);
    }
}
hipError_t launch_keep_share(const int * sel8, const float * w8, int n, int topk, int ke, float renorm, int * sel, float * wts, hipStream_t st) {
    if (n <= 0) { return hipSuccess; }
    if (topk < 1 || topk > MAXK || ke < 1 || ke > topk) { return hipErrorInvalidValue; }
    k_keep_share<<<1, 256, 0, st>>>(sel8, w8, n, topk, ke, renorm, sel, wts);
    return hipGetLastError();
}

hipError_t launch_router_select(float * logits, const double * part2, int K, const float * bias, int n, int n_exp, int n_group, int topk_group,
                                int topk, float scale, float * probs, int * sel, float * wts, hipStream_t st, int keep, float renorm) {
    if (n <= 0) { return hipSuccess; }
    if (keep <= 0) { keep = topk; }
    if (!select_rule_ok(n_exp, n_group, topk_group, topk, keep)) { return hipErrorInvalidValue; }
    auto go = [&](auto kernel) { kernel<<<n, 64, 0, st>>>(logits, part2, bias, n, n_exp, n_group, topk_group, topk, scale, keep, renorm, probs, sel, wts); };
    switch (part2 ? router_parts(n, n_exp, K) : 0) {
    case 0: go(k_router_select<0>); break;
    case 2: go(k_router_select<2>); break;
    case 4: go(k_router_select<4>); break;
    case 8: go(k_router_select<8>); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace lk
