// launch_rules.h -- which kernel a call's sizes get: plain functions of the sizes, without HIP, so that a CPU test can hold
// them against each other (tests/test_launch_rules.py).
#pragma once

namespace lk {

// ---------------------------------------------------------------- router (router.hip)
// The matrix-core router works on tiles of 32 tokens x 32 experts and splits a tile's 256 chunks over `parts` workgroups, so
// that the launch fills the 256 CUs: the fewer tiles, the more parts. It depends on the tiles, not on the tokens alone: 400
// tokens are 104 tiles with 256 experts (2 parts: 60 us) but 26 with 64 (2 parts 59 us, 8 parts 25).
// 0: not split (or another kernel): below RM_MIN tokens one workgroup per expert (k_router_wg: 20.6 us at 16 tokens and 0.5 a
// token more, against 22.6 here at 17, 23.2 at 24 with 256 experts, 23.3 and 23.5 with 64); above RM_TILES tiles the
// unsplit kernel, which keeps the parts' scratch (parts x tokens x experts doubles) at 8 MiB.
constexpr int RM_MIN = 21, RM_TILES = 512;
constexpr int router_tiles(int n, int n_exp) { return ((n + 31) / 32) * ((n_exp + 31) / 32); }
constexpr int router_parts(int n, int n_exp, int K) {
    return K != 7168 || n < RM_MIN || router_tiles(n, n_exp) > RM_TILES ? 0
         : router_tiles(n, n_exp) <= 32 ? 8 : router_tiles(n, n_exp) <= 64 ? 4 : 2;
}

// ---------------------------------------------------------------- grouped GEMM columns (moe_prefill.hip, kq_gemm.hip)
// Slots of a column at most: the IQ2_XXS GEMMs' table, the two classes of a split table (narrow, few), the K-quant GEMMs'.
constexpr int PF_TOK = 112, SPLIT_TOK = 32, FEW_TOK = 8, KQ_TOK = 64;
// The IQ2_XXS table of n shared and P routed slots of n_exp experts. A split table (columns of at most 8 and of 9 .. 32 slots, one
// launch) streams a column's weights at about the memory's rate and pays for every column; the other one (columns of up to
// 112) does more work per byte and needs its three launches filled. So the line depends on the slots per expert, and on the
// slots alone where the experts are few. Split against not split, us a layer: 256 experts of 8 picks 400 tokens 932 / 956, 450
// 989 / 974; of 2 picks 1600 tokens 1214 / 1291, 2000 1369 / 1376; of 4 picks 800 tokens 994 / 1045, 1300 1481 / 1353; 128
// experts 256 tokens 574 / 629, 350 695 / 690; 64 experts 200 tokens 393 / 474, 330 562 / 523; 32 experts 200 tokens 358 / 385,
// 256 418 / 394; 16 experts 160 tokens 293 / 303, 350 489 / 484. Prompts that share a few experts: 16 hot of 256, 400 tokens
// 844 / 926; identical tokens (8 experts) 128 of them 221 / 220, 160 246 / 254, 200 311 / 303, 300 457 / 413 (the counts that
// would tell them are on the device). The shared expert alone (its pass over a prompt's rows): 256 rows 359 / 461, 512 648 /
// 746, 1000 1245 / 1245.
constexpr bool pf_split(int n, int P, int n_exp) { return P > 0 ? P <= 1280 + 8 * n_exp : n <= 768; }
// A split table takes narrow columns where they replace at least so many columns of 8 for each round of 16 narrow ones: a narrow
// column is 16 gate/up items, a round of them about 37 us more than the few columns beside it, a column of 8 about 2.2. At 17
// against always 8, and against 10 and 22: 84 rows of 2 picks, where the shared expert alone would be narrow, 286 / 286 us, 298
// at 10; 24 rows on 32 experts 139 / 139, 158 at 10; 64 rows of 8 picks 399 / 408, 404 at 22; 76 rows 435 / 461, 446 at 22.
constexpr int SPLIT_GAIN = 17;
// the shared expert's columns in a split table; alone (no routed slots) it takes smaller ones, to occupy the CUs: 65 rows 141
// us in columns of 8, 146 of 16, 157 of 32; 190 rows 315, 292, 292; 300 rows of 16 444, of 32 417
constexpr int split_shared_tok(int n, int P) { return P > 0 ? SPLIT_TOK : n <= 80 ? FEW_TOK : n <= 256 ? 16 : SPLIT_TOK; }
// the K-quant shared expert's columns: enough (column, 128 rows) items of its gate and up for the 256 CUs (at 201 tokens
// 64-slot columns are 128 items in two launches, 32-slot ones 224 in one)
constexpr int kq_shared_tok(int n) { return n <= 128 ? 16 : n <= 256 ? 32 : KQ_TOK; }

}  // namespace lk
