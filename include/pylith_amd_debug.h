/*
 * pylith_amd_debug.h -- test hooks of libpylith_amd.so (no counterpart in the reference).
 *
 * plx_debug_emulate_apply runs the tile plan and the element math of the gfx950 residual /
 * Jacobian-action kernels on the CPU, bounds-checking every LDS, halo and vector index, so the
 * kernels' indexing can be verified on a machine without a GPU.  Returns 0, 1 (bad
 * arguments) or 3 (an index out of bounds, or two cells of one colour touching one node).
 *   lam_mu [num_cells][2]: Lame lambda and shear modulus per cell (original cell order);
 *   algorithm: plx_algorithm (the element path to emulate).
 */
#ifndef PYLITH_AMD_DEBUG_H
#define PYLITH_AMD_DEBUG_H

#include <stdint.h>

#include "pylith_amd.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Tile-plan statistics of a key: tiles, halo slots (shared-node partial sums per apply) and
 * whether the planner took the cells in Morton order of their centroids (input order tiled with
 * more than 1.5 halo slots per cell). */
int plx_debug_plan_info(plx_dm dm, int label_value, int part, int *num_tiles, int64_t *halo_slots,
                        int *reordered);

/* Tiles of the key's pair plan and gather plan (0: none). */
int plx_debug_second_plans(plx_dm dm, int label_value, int part, int *pair_tiles, int *gather_tiles);

/* Z = M R: one multigrid V-cycle on k columns (k in {1, 8, 16, 32, 64}) of a Green's-function handle
 * with the multigrid preconditioner; R, Z: DEVICE [dof][k] in DM order.  R must be complete when the
 * call is made (the handle's own stream reads it); synchronises. */
int plx_debug_gf_precondition(plx_gf g, int k, const float *R, float *Z);

/* algorithm: a plx_algorithm, PLX_EMULATE_PAIRS for the P2 pair kernel over its pair plan, or
 * PLX_EMULATE_GATHER for the tile kernel over the gather plan (an error where there is none). */
enum { PLX_EMULATE_PAIRS = 100, PLX_EMULATE_GATHER = 101 };
int plx_debug_emulate_apply(int cell_type, int num_cells, int num_vertices, int num_nodes,
                            const int32_t *closure, const int32_t *cone, const double *coords,
                            const int32_t *labels, int label_value, const double *lam_mu,
                            int scalar_type, const void *u, void *r, int mode, int algorithm);

#ifdef __cplusplus
}
#endif
#endif
