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

/* bpt_csr_build_device (bptplan.h) for both sides of a graph in one set of launches: the out-CSR (edges grouped by src) and the
 * in-CSR (by dst) of graph/base.py:71-86.  out_side / in_side: host arrays of the five device pointers (indptr, indices, eid,
 * unit_row, unit_ptr) of each side; sizes and workspace as bpt_csr_device_bounds says.  info: int32[4] = (error, number of
 * units) of the out and of the in side, in memory the device can write (pinned host memory saves the caller a copy). */
int bpt_build_csrs_device(const int64_t *src, const int64_t *dst, int64_t n_edges, int64_t n_nodes, int32_t chunk_size,
                          int64_t *const out_side[5], int64_t *const in_side[5], int32_t *info, void *workspace,
                          int64_t workspace_bytes, void *stream);

/* Waits until everything enqueued on the stream has run (for a caller that reads an info block in pinned host memory). */
int bpt_build_wait(void *stream);

#ifdef __cplusplus
}
#endif
#endif
