/* psv_testing.h -- entry points with which the tests force a condition or learn
 * of a choice; a program has no use for them, so the public header does not
 * declare them.  They act on one object and leave every result as it is. */
#pragma once

#include "../../include/psvwave.h"

#ifdef __cplusplus
extern "C" {
#endif

/* The model's next resident time loops find, as if another process held part
 * of the device, that their blocks are not resident together, and run step by
 * step instead. */
int psv_refuse_resident_loops(psv_model *m);
/* The same of a batch, which then starts resident loops under any step
 * variant. */
int psv_batch_refuse_resident_loops(psv_batch *b);

/* Rows of the tiles on which `loops` of the model's time loops run side by side;
 * 0: they run by steps. */
int psv_resident_rows(psv_model *m, int loops, int *rows);
/* `times` allocations of the model (of member m of the batch) after the next n
 * fail as if the device were full. */
int psv_fail_allocation(psv_model *m, int n, int times);
int psv_batch_fail_allocation(psv_batch *b, int m, int n, int times);

#ifdef __cplusplus
}
#endif
