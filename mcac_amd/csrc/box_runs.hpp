// Internal interface between the two libraries.
#pragma once
#include <cstdint>

#include "../../include/mcac_gpu.h"

extern "C" {
// mcac_box_create and mcac_group_add in one, without a stream of the box's own.
int mcac_box_create_in_group(const mcac_box_params *params, mcac_group *group, mcac_box **out);
// mcac_move_enqueue for n moves of a box, in the order they are to run.  Moves
// that take the one-launch form share launches of up to eight; the others take
// their usual launches, in order with the rest.  On an error the moves enqueued
// before the failing one keep their tickets and run.
int mcac_move_enqueue_run(mcac_box *box, const int64_t *aggs, const double *dirs, const double *lpm, double maxradius,
                          int n, uint64_t *tickets);
// mcac_box_set_auto_merge that takes effect with spherical caps as well.  A run of
// 3000 spheres with caps spent 45 us a contact on the merge's own launch.
int mcac_box_merge_in_launch(mcac_box *box, int enable);
}
