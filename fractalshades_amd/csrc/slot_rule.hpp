// slot_rule.hpp -- which slots a wave of a tile launch starts with, and how the
// binary64 pass fills a wave with unsure pixels: apart from the loop, so that
// the host can run them.
#pragma once
#include "xr.hpp"

namespace fsg {

// The first 64 slots of wave `wave` of block `block` of `blocks`: consecutive
// batches go to different blocks.  Neighbouring 8x8 blocks of pixels take about
// as long, and the longest of a frame together on a few compute units shared
// their issue while others had ended.  Against 16 consecutive batches a block:
// z^6 + c 400x400 around the critical orbit, 1000 steps, 1428 -> 1037 us (dz/dz
// 3330 -> 2120), burning ship 937 -> 724 us, the interior-dominated view at
// 520x520 3.91 -> 3.20 ms, z^3 + c 520x520 at 1e-800 192 -> 165 us; 2048x2048 within
// 1 %; slower where a few batches more than the lanes follow (binary32 520x520 at
// 1e-40: 103 -> 111 us).
FSG_HD int64_t first_slot(unsigned block, unsigned wave, unsigned blocks) {
    return 64 * (int64_t)(wave * blocks + block);
}

// The lanes at which a wave stops drawing batches: its part of the launch's
// unsure pixels, 64 at most.
FSG_HD unsigned redo_share(uint64_t unsure, unsigned waves) {
    const uint64_t top = 0xffffffffull - waves;
    const unsigned share = (unsigned)((unsure < top ? unsure : top) + waves - 1u) / waves;
    const unsigned some = share > 1u ? share : 1u;
    return some < 64u ? some : 64u;
}

// Whether an unsure slot of a drawn batch, with `before` of the batch's before
// it, gets a lane of a wave that holds `filled` pixels.  Every one that fits
// does, past the share too: the others of the batch are this wave's alone, and
// while it iterates without them no other wave can take them.  Unsure pixels
// are neighbours (a batch is an 8x8 block of a grid), so a wave that stopped at
// its share within a batch iterated a block's pixels one after the other.
FSG_HD bool slot_goes(unsigned filled, unsigned before) { return filled + before < 64u; }

}  // namespace fsg
