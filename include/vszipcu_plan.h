/* vszipcu_plan.h — diagnostics of libvszipcu_amd.so: which searches run as the screened ssd search. No reference
 * counterpart. */
#ifndef VSZIPCU_PLAN_H
#define VSZIPCU_PLAN_H

#include "vszipcu_bm3d.h"

#ifdef __cplusplus
extern "C" {
#endif

/* *screened is 1 where vsz_bm3d_match and vsz_bm3d_run take the screened search on the matrix cores for
 * the spatial (or centre-frame) search in place of the matcher that vsz_bm3d_match_plan names, else 0: ssd on windows that
 * gain by it, with the same lists and distances. Needs no GPU. Returns VSZ_OK or VSZ_EINVAL. */
int vsz_bm3d_match_screened(const vsz_bm3d_kparams *p, int *screened);

/* *screened is 1 where the batch searches with the screened search in place of the matcher that
 * vsz_bm3d_batch_schedule reports (staged schedule only), else 0; final after its first run. */
int vsz_bm3d_batch_screened(const vsz_bm3d_batch *b, int *screened);

#ifdef __cplusplus
}
#endif

#endif /* VSZIPCU_PLAN_H */
