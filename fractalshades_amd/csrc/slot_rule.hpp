// slot_rule.hpp -- how the binary64 pass fills a wave with unsure pixels,
// apart from the loop so that the host can run it.
#pragma once
#include "xr.hpp"

namespace fsg {

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
