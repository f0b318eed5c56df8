// ps_blocks.hpp — how the constraint blocks of the lambda launch are counted
// and, where one launch cannot hold them, divided.  Plain arithmetic, the
// same for the host and the kernels.
#pragma once

#include <stdint.h>

namespace ps {

// Blocks of `threads` threads (a multiple of 64) for `count` items of `lanes`
// lanes each (a divisor of 64).  No product of the two is formed: 2^29 contact
// walkers of eight lanes are 2^32 threads.
constexpr uint32_t item_blocks(uint32_t count, uint32_t lanes, uint32_t threads)
{
    const uint32_t per = threads / lanes;
    return count / per + (count % per ? 1u : 0u);
}

// The constraint blocks in order: contact walkers (eight lanes each), linked
// particles (four), bodies (a wavefront), rounded up to whole turns of the
// eight XCDs.
struct ConParts {
    uint32_t walks, links, all;
};
constexpr ConParts con_parts(uint32_t nwalk, uint32_t nlink, uint32_t nbody, uint32_t threads)
{
    const uint32_t w = item_blocks(nwalk, 8u, threads), l = item_blocks(nlink, 4u, threads);
    return ConParts{w, l, (w + l + item_blocks(nbody, 64u, threads) + 7u) & ~7u};
}

// What a lambda launch is told of them (an argument of its own: the buffers go
// to every kernel): the walkers' and the links' of all, the first of this
// launch and how many.
struct ConBlocks {
    uint32_t walks, links, first, blocks;
};

// A launch holds fewer than 2^32 threads.  Of `all` constraint blocks and
// `fluid` blocks after them, those from `first` on: the next launch's
// constraint blocks, and whether the fluid's are in it (then it is the last).
struct ConLaunch {
    uint32_t blocks;
    bool last;
};
constexpr ConLaunch con_launch(uint32_t all, uint32_t first, uint32_t fluid, uint32_t threads)
{
    const uint32_t room = (0xffffffffu / threads) & ~7u, left = all - first;
    if (left <= room && fluid <= room - left) return ConLaunch{left, true};
    return ConLaunch{left < room ? left : room, false};
}

}  // namespace ps
