// Window widths by size class ceil(log2 n) on MI355X (gfx950), as measured by
// the autotuner in zkmetal_amd/tune.py:
//     python -m zkmetal_amd.tune --min-logn 8 --max-logn 22 --reps 3
// kTunedPlain: an MSM called alone (lowest wall time per call); kTunedBatch:
// an MSM inside a multi-MSM call (lowest time per MSM in a call holding 2^21
// points of that class).  0 = the cost model (default_window_bits).  Engines
// start from these tables; zkmsm_set_window_table / _batch_ replace them.
//
// kTunedParts / kTunedPer: the launch schedule by call size class ceil(log2
// entries) -- pipeline parts and buckets per bucket-reduction lane or team -- for
// calls of one MSM ([0]) and of several ([1]), from the same sweep; 0 = the
// built-in rule (default_parts, and buckets per lane or team by bucket
// count, at least 8).  zkmsm_set_schedule_table replaces them.
#pragma once
#include <stdint.h>

namespace zk {

// Widths that divide the 128 bits without a narrow top window (8, 13 with an
// 11-bit top, 16) win: a narrow one piles its entries into few buckets, whose
// partials the merge then adds up.  Against the widths between (us): 2^11
// points 214 at 13 bits, 254 at 8; 2^14 291 at 16, 399 at 10; 2^16 358 at 16,
// 420 at 15.
static const uint32_t kTunedPlain[33] = {0, 0, 0, 0, 0, 0, 8, 8, 8, 8, 8, 13, 13, 13, 16, 16, 16,
                                         16, 16, 16, 16, 16, 16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
static const uint32_t kTunedBatch[33] = {0, 0, 0, 0, 0, 0, 8, 8, 8, 8, 8, 8, 9, 10, 11, 13, 13,
                                         13, 16, 16, 16, 16, 16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
// The narrow widths for a call that a memory cap, or the no-allocation
// array, leaves no room for the tuned ones (a fraction of their buckets).
static const uint32_t kLeanPlain[33] = {0, 0, 0, 0, 0, 0, 0, 0, 8, 8, 8, 8, 10, 10, 10, 12, 15,
                                        15, 16, 16, 16, 16, 16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
static const uint32_t kLeanBatch[33] = {0, 0, 0, 0, 0, 0, 0, 0, 6, 7, 8, 8, 9, 10, 11, 12, 13,
                                        13, 16, 16, 16, 16, 16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
// single MSMs on Grumpkin and BN254 G2 (255-bit scalars, no GLV)
static const uint32_t kTunedGrumpkin[33] = {0, 0, 0, 0, 0, 0, 8, 8, 8, 8, 10, 11, 12, 10, 10, 11, 15,
                                            15, 16, 16, 16, 16, 16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
static const uint32_t kTunedG2[33] = {0, 0, 0, 0, 0, 0, 8, 8, 8, 8, 10, 9, 10, 12, 12, 12, 12,
                                      12, 13, 16, 16, 16, 16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

// Small calls leave most of the chip idle, so a shorter chain before the tree
// wins: with 4 against 8 buckets, 256 points 255 against 263 us, 4097 points
// 322 against 332, 2^16 points the same.
static const uint8_t kTunedParts[2][33] = {};
static const uint8_t kTunedPer[2][33] = {
    {4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0},
    {4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}};

}  // namespace zk
