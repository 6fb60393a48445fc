/* dsx_testing.h — switches of libdsx_hip.so that exist for its tests: they make small inputs reach the code paths that
 * otherwise only large ones take.  Not part of the drop-in boundary (include/dsx.h) and without counterpart in the reference.
 * Results never depend on them.  The values live in the library's context: dsx_shutdown (the last one) and dsx_testing_reset
 * put every switch back to its default; like every call of the library they belong to the one thread that drives it. */
#ifndef DSX_TESTING_H
#define DSX_TESTING_H
#include <stddef.h>
#include <stdint.h>
#ifdef __cplusplus
extern "C" {
#endif

/* Rows of a workgroup's tile in dsx_fc_forward_split: 128 or 256; 0 (default) chooses by shape. */
int dsx_testing_set_split_tile_rows(uint32_t rows);
/* dsx_fc_topk: width of the first column block (0: default 2,048; at most 131,072) and survivor words per row and column range
 * (64 .. 4,096; 0: default 4,096). */
int dsx_testing_set_fc_topk_first_columns(uint32_t columns);
int dsx_testing_set_fc_topk_candidate_capacity(uint32_t words);
/* dsx_knn_search*: width of the first column block (rounded down to a multiple of 1024, at least 1024; 0 restores the default
 * of about 1 GiB of scores).  Workspace sizes depend on it: set it before asking for them. */
int dsx_testing_set_knn_block_columns(uint32_t columns);
/* dsx_knn_search_f16, column ranges after the first block.  1 (default): swept by workgroups that keep their queries when the
 * range is long enough; 0: always one workgroup per tile; 2 and 3: the LDS sweep and the register sweep for every range that
 * has at least one tile per chunk. */
int dsx_testing_set_knn_f16_sweep(int mode);
/* Occupancy probe: launches `workgroups` workgroups of 256 lanes on the selected lane that do nothing but hold their place for
 * about `cycles` shader clocks (bounded; every wavefront exits), with 128, 64 or (any other value) next to no vector
 * registers per lane.  bench.py --interference uses it to separate what a kernel beside a dense layer costs that layer by
 * merely being resident from what its instructions and memory traffic cost. */
int dsx_testing_occupy(uint32_t workgroups, uint32_t cycles, uint32_t vgprs);
/* dsx_knn_search, dsx_fc_topk: candidates are screened in 16 bits where that is expected to be the faster way (0, default), never (2);
 * 1: whatever can be (searches of 512 queries and 65,536 items, layers of 512 rows and 16,384 columns and more).  Workspace sizes
 * depend on it. */
int dsx_testing_set_screen(int mode);
/* Screened searches with a kept table: in bytes where that is expected to be the faster way (0, default), wherever it can be (1), never (2).
 * Workspaces and tables depend on it: both are made behind the call. */
int dsx_testing_set_screen_bytes(int mode);
/* dsx_knn_search*: the events that its stages' times are taken with cannot be made (1; 0, the default: as the device has it). */
int dsx_testing_set_knn_no_events(int none);
/* What a screened search of `batch` rows among rows_padded - padding columns (of rows_padded, which its workspace is laid out for) does:
 * columns of sums that there is room for per row, columns that are stored (whole tiles), and whether the others are gone through in ranges
 * (0: the results come from the stored ones).  Runs on the host alone, without dsx_init. */
int dsx_testing_screen_columns(uint32_t batch, uint32_t dim, uint32_t rows_padded, uint32_t padding, uint32_t k, uint64_t* room, uint64_t* stored,
                               int* ranges);
/* Largest single block of device memory that dsx_malloc and the library's own scratch may hold, in bytes (0, the default: what the
 * device has): larger ones fail as if the memory were short. */
int dsx_testing_set_allocation_limit(size_t bytes);
/* Every switch back to its default. */
int dsx_testing_reset(void);

#ifdef __cplusplus
}
#endif
#endif /* DSX_TESTING_H */
