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

constexpr size_t CU_LDS = 160 * 1024;

// Static LDS of a build for S RBGs, nc cells and W wavefronts per env: the kernel's __shared__ arrays, with room for
// their alignment (the compiled kernels hold up to 128 B less). common: a build of the common configuration.
inline size_t step_lds_static(int S, int nc, bool ir, bool common, int W = 1) {
    const size_t q = (size_t)nc * S, cw = (size_t)STEP_WAVE * W;
    return sizeof(int) * ((2 * q + S) * cw + (W > 1 ? 13 : 11) * cw + 6 * MAX_M + 4 * S + 1 + (common ? 1 : S * S) +
                          (ir ? MAX_M * MAX_EQW : 1) + MAX_UL_ROWS + 20 + 4 * W +
                          (nc > 1 ? q * (1 + 2 * nc) + nc * cw : 2));
}

// The lanes of a wavefront that one env of next_pow2(R) = rb0 lanes takes: rb0, or twice, four times, ... that while
// the batch still leaves the chip room. A wavefront's time is its serial chain of slots, and the work that its envs
// deal over the 64 lanes (fading draws, estimates, the MCS search) grows with the envs it holds, so a batch that does
// not fill the chip is spread over more wavefronts with fewer envs each, down to one env per wavefront. The room is
// the wavefronts that are resident at once: one for each of the 1024 SIMDs, or the `occ` that its registers hold, and
// no more than the 160 KiB of a CU hold at lds(rb) bytes each (in allocations of 1280): one wavefront beyond it is a
// second round of the whole chain. Measured, us per step in 8 / 16 / 32 / 64 lanes per env, by the wavefronts
// resident at 64:
//   2048, two per SIMD: round robin 512 x 8 105 / 95 / 84 / 82, 2048 x 8 107 / 99 / 90 / 91, 4096 x 8 115 / 105 / 99
//   / 164; default configuration (8 UL slots) 256 x 16 - / 313 / 196 / 159, 2048 x 16 - / 344 / 209 / 195, 4096 x 16
//   - / 349 / 248 / 370, 1024 x 32 - / - / 257 / 193, 4096 x 32 - / - / 321 / 437; UL and DL 4096 x 8 421 / 400 / 322
//   / 535, 2048 x 32 - / - / 446 / 437, 4096 x 32 - / - / 494 / 801
//   1024, one per SIMD: three cells 1024 x 16 - / 690 / 527 / 335, 2048 x 32 - / - / 736 / 836
//   fewer by LDS: RLC UM (the losses of every slot in LDS) over 20 UL slots at 16 processes, 1280: 2048 x 32 - / - /
//   713 / 1103, 4096 x 8 797 / 629 / 1044 / 1556; four cells, 768: 1024 x 16 - / 840 / 634 / 833; seven cells, 512:
//   1024 x 32 - / - / 1382 / 1830, 2048 x 8 1314 / 974 / 1495 / 2171
template <class L>
int seg_width(int E, int rb0, int occ, L lds) {
    constexpr int64_t CUS = 256, LDS = CU_LDS;
    int rb = rb0;
    while (rb < STEP_WAVE) {
        const int64_t waves = ((int64_t)E * 2 * rb + STEP_WAVE - 1) / STEP_WAVE;
        const int64_t need = ((int64_t)lds(2 * rb) + 1279) / 1280 * 1280, held = need > 0 ? LDS / need : 0;
        const int64_t room = CUS * (held < 4 * occ ? held : 4 * occ);
        // (a width whose envs' rows do not fit a CU, several cells with few robots per env, is passed over)
        if (waves > room && lds(rb) + 16384 <= CU_LDS) break;
        rb *= 2;
    }
    return rb;
}

}  // namespace inet
