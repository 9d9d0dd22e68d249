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

}  // namespace lk
