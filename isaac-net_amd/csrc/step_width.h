// The lanes of a wavefront that one env of the step kernel takes, and the LDS that its wavefront holds. Plain C++ (the
// host test compiles it with g++).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "../../include/inet_nr.h"

namespace inet {

constexpr int STEP_WAVE = 64;          // one wavefront per workgroup
constexpr int MAX_UL_ROWS = 64;        // UL data slots per control step
constexpr int MAX_M = 32;              // MCS table rows
constexpr int MAX_EQW = INET_NR_MAX_P + 1;

// Dynamic LDS of the step kernel, in ints: the in-order pointer after every UL slot [n_ul][64], with RLC drop the
// byte range of a TB that exhausted its HARQ [n_ul][64] x 2, then the per-env HARQ histograms [64 / RB][3][max_tx + 1];
// with several cells (nc > 1) then per env each gNB's N+I estimate and this slot's interference [64 / RB][2][nc S].
inline size_t step_lds_bytes(int n_ul, int harq_drop, int rb, int max_tx, int nc = 1, int S = 0) {
    const size_t cw = rb > STEP_WAVE ? (size_t)rb : (size_t)STEP_WAVE;     // lanes per workgroup
    return sizeof(int) * ((size_t)n_ul * cw * (harq_drop ? 3 : 1) +
                          (cw / rb) * 3 * (max_tx + 1) +
                          (nc > 1 ? (cw / rb) * 2 * nc * S : 0));
}

// Static LDS of a one-wavefront build for S RBGs and nc cells: the kernel's __shared__ arrays, with room for their
// alignment (the compiled kernels hold up to 100 B less). common: a build of the common configuration.
inline size_t step_lds_static(int S, int nc, bool ir, bool common) {
    const size_t q = (size_t)nc * S, cw = STEP_WAVE;
    return sizeof(int) * ((2 * q + S) * cw + 11 * cw + 6 * MAX_M + 4 * S + 1 + (common ? 1 : S * S) +
                          (ir ? MAX_M * MAX_EQW : 1) + MAX_UL_ROWS + 24 + (nc > 1 ? q * (1 + 2 * nc) + nc * cw : 2));
}

// The lanes of a wavefront that one env of next_pow2(R) = rb0 lanes takes: rb0, or twice, four times, ... that while the
// batch still leaves the chip room. A wavefront's time is its serial chain of slots, and the work that its envs deal
// over the 64 lanes (fading draws, estimates, the MCS search) grows with the envs it holds, so a batch that does not
// fill the chip is spread over more wavefronts with fewer envs each, down to one env per wavefront. The room is the
// wavefronts that are resident at once: one for each of the 1024 SIMDs, or the `occ` that its registers hold, and no more
// than the 160 KiB of a CU hold at lds(rb) bytes each (in allocations of 1280): one wavefront beyond it is a second
// round of the whole chain. Past one per SIMD an env takes at most four times its own lanes, and the DL launch keeps to
// one per SIMD. Measured, us per step in 8 / 16 / 32 / 64 lanes per env, beside the wavefronts resident at 64:
// 64 x 8 round robin 99.9 / 88.8 / 80.4 / 81.2, 2048 x 8 104 / 96 / 89 / 103 (2048); default configuration 256 x 16
// (20 UL slots) - / 1202 / 679 / 495, 2048 x 16 (8 UL slots) - / 579 / 328 / 276, 4096 x 16 - / 573 / 371 / 511,
// 1024 x 32 - / - / 364 / 264, 4096 x 32 - / - / 443 / 575 (2048); UL and DL 2048 x 32 - / - / 524 / 544; three cells
// 1024 x 16 - / 728 / 552 / 354, 2048 x 32 - / - / 813 / 894 (1024). Where LDS holds fewer: RLC UM (the losses of every
// slot in LDS), 20 UL slots, 16 processes, 2048 x 32 - / - / 713 / 1220, 4096 x 8 801 / 630 / 1044 / 1715 (1280); seven
// cells 1024 x 32 - / - / 1382 / 1830, 2048 x 8 1317 / 973 / 1493 / 2174 (512); four cells 1024 x 16 - / 843 / 635 / 831
// (768).
template <class L>
int seg_width(int E, int rb0, int occ, bool dl, L lds) {
    constexpr int64_t CUS = 256, SIMDS = 4 * CUS, LDS = 160 * 1024;
    int rb = rb0;
    while (rb < STEP_WAVE) {
        const int64_t waves = ((int64_t)E * 2 * rb + STEP_WAVE - 1) / STEP_WAVE;
        const int64_t need = ((int64_t)lds(2 * rb) + 1279) / 1280 * 1280, held = need > 0 ? LDS / need : 0;
        const int64_t room = CUS * (held < 4 * occ ? held : 4 * occ);
        if (waves > room || (waves > SIMDS && (dl || 2 * rb > 4 * rb0))) break;
        rb *= 2;
    }
    return rb;
}

}  // namespace inet
