// Window widths by size class ceil(log2 n) on MI355X (gfx950), 0 = the cost
// model (default_window_bits).  kTunedPlain: an MSM called alone; kTunedBatch:
// an MSM inside a call of several; engines start from these two, and
// zkmsm_set_window_table / _batch_ replace them.  kTunedGrumpkin and kTunedG2:
// single MSMs without the endomorphism; nothing replaces these (a forced width
// goes before any table).  The entries go by wall time per call at two sizes of
// each class; profiles/window_widths.md has the times of all widths and names
// the few classes where another width is more than 3% quicker.
// zkmetal_amd/tune.py sweeps kTunedPlain's and kTunedBatch's candidates (the
// cost model's width and its neighbours) for a device and scalars of one's own.
//
// kTunedParts / kTunedPer: the launch schedule by call size class ceil(log2
// entries) -- pipeline parts and buckets per bucket-reduction lane or team -- for
// calls of one MSM ([0]) and of several ([1]); 0 = the built-in rule
// (default_parts, and buckets per lane or team by bucket count, at least 8).
// zkmsm_set_schedule_table replaces them.
#pragma once
#include <stdint.h>

namespace zk {

// Widths that divide the 128 bits without a narrow top window (8, 13 with an
// 11-bit top, 16) win: a narrow one piles its entries into few buckets, whose
// partials the merge then adds up.  Against the widths between (us): 2^11
// points 207 at 13 bits, 248 at 8; 2^14 280 at 16, 384 at 10; 2^16 346 at 16,
// 404 at 15.
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
// Single MSMs on Grumpkin and BN254 G2.  255 bits are 17 windows of 15, or 15
// of 16 and one of 15; narrower widths leave a top of 2 to 5 bits, whose few
// buckets cost merge work once they hold many entries.  In us: Grumpkin 2^13
// points 318 at 10 bits (11: 362, 12: 328), 2^14 362 (382, 409), 2^16 437 at
// 15 (10: 495, 16: 458); G2, whose bucket additions cost more, 2^11 480 at 9
// (8: 468, 10: 497), 2^16 842 at 12 (13: 864, 16: 1133), 2^18 1694 at 13 (16:
// 1844), 2^19 2581 at 16 (13: 2863).
static const uint32_t kTunedGrumpkin[33] = {0, 0, 0, 0, 0, 0, 8, 8, 8, 8, 10, 11, 12, 10, 10, 11, 15,
                                            15, 16, 16, 16, 16, 16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
static const uint32_t kTunedG2[33] = {0, 0, 0, 0, 0, 0, 8, 8, 8, 8, 10, 9, 10, 12, 12, 12, 12,
                                      12, 13, 16, 16, 16, 16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

// Small calls leave most of the chip idle, so a short chain before the tree
// wins: with 4, 8 and 16 buckets, 256 points 164, 175 and 190 us, 64 plain MSMs
// of 256 points 716, 881 and 1211; from class 16 on one MSM takes the same with
// 4 and 8 within 3% (2^16 points 347 and 338) and up to 13% more with 16.
static const uint8_t kTunedParts[2][33] = {};
static const uint8_t kTunedPer[2][33] = {
    {4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0},
    {4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 4, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}};

}  // namespace zk
