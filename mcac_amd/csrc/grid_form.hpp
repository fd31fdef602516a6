// How the blocks of one search's grid meet and part (k_step_grid; k_solve parts
// the same way).  Between the two they read the same plan: the survivors, their
// sizes and segments, and the counters behind both.  The block that ends last
// changes all of these (it moves the aggregate, may merge, and resets the
// counters for the next search), so every block of the grid takes a ticket once
// it has read what it reads, also one that the plan leaves without work: were
// only the working blocks counted, a block could still be polling a barrier
// count that has been reset, or plan from an aggregate that has merged.  A block
// that gives up at the barrier takes no ticket, so then nothing is changed and
// no record published.
// Grid: the counters and fences, by one thread of a block.
#pragma once

namespace mcac_dev {

// True once all `blocks` blocks of the grid have arrived; false: waited in vain.
template <class Grid> constexpr bool grid_meet(Grid &g, unsigned blocks) {
    g.publish();  // this block's candidates and counts before its arrival
    g.arrive();
    while (!g.out_of_time()) {
        if (g.arrived() >= blocks) return true;
        g.pause();
    }
    g.give_up();
    return false;
}

// True in the block that ends last.  wrote: this block has results for it.
template <class Grid> constexpr bool grid_part(Grid &g, unsigned blocks, bool wrote) {
    if (wrote) g.publish();
    return g.ticket() == blocks - 1u;
}

}  // namespace mcac_dev
