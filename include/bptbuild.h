/* bptbuild.h — C ABI of libbptplan.so, second part: the steps from a batch of graphs to the plans of its attention in as few
 * launches as they take, for a training loop that builds a new graph per batch (graph/lm.py:53-98).  Same conventions as
 * bptplan.h: device pointers, the caller's stream, nothing allocated, 0 / bpt_status / hipError_t.
 */
#ifndef BPTBUILD_H
#define BPTBUILD_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* The block-diagonal merge of graph/lm.py:53-98: parts (host memory) holds six int64 per graph, the device addresses of its src,
 * dst, etype (n_edges each) and pos (n_nodes), then n_edges and n_nodes; the lists are written one after the other, node ids
 * shifted by the nodes of the graphs before. */
int bpt_build_merge_device(const int64_t *parts, int64_t n_parts, int64_t *src, int64_t *dst, int64_t *etype, int64_t *pos,
                           void *stream);

/* bpt_csr_build_device (bptplan.h) for both sides of a graph in one set of launches: the out-CSR (edges grouped by src) and the
 * in-CSR (by dst) of graph/base.py:71-86.  out_side / in_side: host arrays of the five device pointers (indptr, indices, eid,
 * unit_row, unit_ptr) of each side; sizes and workspace as bpt_csr_device_bounds says.  info: int32[4] = (error, number of
 * units) of the out and of the in side, in memory the device can write (pinned host memory saves the caller a copy). */
int bpt_build_csrs_device(const int64_t *src, const int64_t *dst, int64_t n_edges, int64_t n_nodes, int32_t chunk_size,
                          int64_t *const out_side[5], int64_t *const in_side[5], int32_t *info, void *workspace,
                          int64_t workspace_bytes, void *stream);

/* bpt_plan_build_device (bptplan.h), and the smallest and the largest neighbour id of every item beside it (item_bounds: as many
 * rows of 2 int32 as items, or NULL). */
int bpt_build_plan_device(const int64_t *row, const int64_t *indptr_units, int64_t n_units, const int64_t *eid,
                          const int64_t *indices, int64_t n_edges, int64_t n_rows, int64_t n_index_nodes, int32_t seg_len,
                          int32_t *rowptr, int32_t *idx32, int32_t *eid32, int32_t *items, int32_t *heavy, int32_t *item_bounds,
                          int32_t *info, void *workspace, int64_t workspace_bytes, void *stream);

/* The row groups of bpt_plan_group_device (bptplan.h), bit for bit, in two calls between which the caller reads how large they
 * are and allocates exactly: bpt_build_groups_count forms and numbers the groups in the workspace and writes out_info (int32[32],
 * in memory the device can write: the plan's info block, then the groups' info block); bpt_build_groups_write, given the groups'
 * info block on the host (group_counts), writes the arrays from the same workspace:
 *   members (n_groups, R, 2)   grp_ptr (n_groups + 1)   entries (n_entries + 1, 4)   pair_eid (n_edges)
 *   grp_eids ((n_entries + pad_entries) * R)            chunks (9)                   group_info: int32[16]
 * bpt_build_groups_bounds: workspace bytes, or BPT_ERR_UNSUPPORTED where only bpt_plan_group_device builds the groups (more than
 * 4096 edges a group, or more than 16384 groups). */
int bpt_build_groups_bounds(int64_t max_items, int64_t n_edges, int64_t n_index_nodes, int32_t seg_len, int32_t R, int64_t bounds[1]);
int bpt_build_groups_count(const int32_t *items, const int32_t *item_bounds, const int32_t *idx32, const int32_t *eid32,
                           const int32_t *plan_info, int64_t max_items, int64_t n_edges, int64_t n_index_nodes, int32_t seg_len,
                           int32_t R, int32_t by_mask, int32_t *out_info, void *workspace, int64_t workspace_bytes, void *stream);
int bpt_build_groups_write(const int32_t *items, const int32_t *plan_info, int64_t max_items, int64_t n_edges,
                           int64_t n_index_nodes, int32_t seg_len, int32_t R, const int32_t *group_counts, int32_t pad_entries,
                           int32_t *members, int32_t *grp_ptr, int32_t *entries, int32_t *pair_eid, int32_t *grp_eids,
                           int32_t *chunks, int32_t *group_info, void *workspace, int64_t workspace_bytes, void *stream);

/* The tile plans (groups of 16 rows) of one or two sides of a graph in shared launches: base plan, then groups, as the calls above.
 * bpt_build_tiles_bounds: workspace bytes (from the sizes alone), or BPT_ERR_UNSUPPORTED as bpt_build_groups_bounds.
 * bpt_build_tiles_count: base plans written, out_info int32[32] per side as bpt_build_groups_count's.  bpt_build_tiles_write: the
 * arrays of the groups, given those info blocks on the host; with pairs (((n_entries + pad_entries) * 16) int32 of side 1) also the
 * pair mapping of side 1 to side 0 (bpt_build_pair_numbers), for which out[0].number holds n_edges int32. */
typedef struct {
    const int64_t *row, *indptr_units, *eid, *indices;
    int64_t n_units, n_edges, n_rows, n_index_nodes;
    int32_t seg_len, by_mask;
    int32_t *rowptr, *idx32, *eid32, *items, *item_bounds, *heavy, *info;
} bpt_build_side;
typedef struct {
    int32_t *members, *grp_ptr, *entries, *pair_eid, *grp_eids, *chunks, *group_info, *number;
} bpt_build_tiles;
int bpt_build_tiles_bounds(const bpt_build_side *sides, int n_sides, int64_t bounds[1]);
int bpt_build_tiles_count(const bpt_build_side *sides, int n_sides, int32_t *out_info, void *workspace, int64_t workspace_bytes,
                          void *stream);
int bpt_build_tiles_write(const bpt_build_side *sides, int n_sides, const int32_t *infos, const bpt_build_tiles *out,
                          int32_t pad_entries, int32_t *pairs, void *workspace, int64_t workspace_bytes, void *stream);

/* The base plans alone of one or two sides, with indices: out_info int32[16] per side (their info blocks), in memory the device can write;
 * by_mask is not read, item_bounds may be NULL.  bpt_build_plans_bounds: workspace bytes, from the sizes alone. */
int bpt_build_plans_bounds(const bpt_build_side *sides, int n_sides, int64_t bounds[1]);
int bpt_build_plans(const bpt_build_side *sides, int n_sides, int32_t *out_info, void *workspace, int64_t workspace_bytes, void *stream);

/* For every (entry, member) of one side's groups (grp_eids_mine, n_slots) the number of the same edge's pair on the other side
 * (pair_eid_theirs, n_edges), 0 where there is none.  number: n_edges int32 of scratch. */
int bpt_build_pair_numbers(const int32_t *pair_eid_theirs, const int32_t *grp_eids_mine, int64_t n_slots, int64_t n_edges,
                           int32_t *number, int32_t *pairs, void *stream);

/* How many rows of one or two CSR sides have edges (what the length of the work items of a graph of two node sets goes by): side s
 * has n_units[s] units, sorted by row, a row's one after the other.  counts: BPT_COUNT_PARTS int32 a side in memory the device can
 * write (pinned host memory saves the caller a copy); their sum is the number.  Rows are compared, not used as an index: any value does. */
#define BPT_COUNT_PARTS 64
int bpt_build_count_rows(const int64_t *const row[2], const int64_t *const indptr_units[2], const int64_t n_units[2], int n_sides,
                         int32_t *counts, void *stream);

/* Waits until everything enqueued on the stream has run (for a caller that reads an info block in pinned host memory). */
int bpt_build_wait(void *stream);

#ifdef __cplusplus
}
#endif
#endif
