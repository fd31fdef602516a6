// Internal interface between the two libraries: several queued moves of one box.
#pragma once
#include <cstdint>

#include "../../include/mcac_gpu.h"

extern "C" {
// mcac_move_enqueue for n moves of a box, in the order they are to run.  Moves
// that take the one-launch form share launches of up to eight; the others take
// their usual launches, in order with the rest.  On an error the moves enqueued
// before the failing one keep their tickets and run.
int mcac_move_enqueue_run(mcac_box *box, const int64_t *aggs, const double *dirs, const double *lpm, double maxradius,
                          int n, uint64_t *tickets);
}
