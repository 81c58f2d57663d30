/* Between recon.hip and the intra phase's kernels: the launchers, and the
 * batched form's ready queue (recon.hip fills it, recon_intra.h takes from
 * it). */
#ifndef MAV1_RECON_QUEUE_H
#define MAV1_RECON_QUEUE_H

#include "dev_common.h"
#include "internal.h"

/* Of frames without a luma search (recon_intra.hip) and with a transform type
 * or depth search (recon_search.hip). */
hipError_t launch_recon_intra_plain(hipStream_t st, const Mav1FrameParams &fp, Mav1BlockInfo *blocks,
                                    const Mav1SbInfo *sbs, const uint8_t *src, uint8_t *rec, int32_t *coefs,
                                    const int32_t *mats, int *iwork, int workgroups);
hipError_t launch_recon_intra_search(hipStream_t st, const Mav1FrameParams &fp, Mav1BlockInfo *blocks,
                                     const Mav1SbInfo *sbs, const uint8_t *src, uint8_t *rec, int32_t *coefs,
                                     const int32_t *mats, int *iwork, int workgroups);
hipError_t launch_recon_intra_plain_b(hipStream_t st, const BatchFrame *T, int n, int *q, int workgroups);
hipError_t launch_recon_intra_search_b(hipStream_t st, const BatchFrame *T, int n, int *q, int workgroups);

/* Intra phase over several frames: a dataflow queue. A superblock holding
 * intra blocks enters the batch's ready queue when the last of its
 * dependencies (the neighbours in its tile column whose reconstruction it
 * reads and that hold intra blocks) is done, so a workgroup only ever takes
 * a superblock it can code at once, of whichever frame; superblocks without
 * such dependencies are queued first. q: [QH_HEAD] next entry to take,
 * [QH_TAIL] next entry to fill, [QH_TOTAL] superblocks of the round, then
 * the entries ((frame << 16) | superblock, -1 until filled). Every entry is
 * filled once all superblocks before it in dependency order are done, so a
 * workgroup's wait for its entry ends; the wait is still bounded, and one
 * that runs out sets every frame's error word.
 * A batch has two queues, one behind the other: of the frames without a luma
 * search and of those with one, whose intra kernels differ. */
#define QH_HEAD 0
#define QH_TAIL 1
#define QH_TOTAL 2
#define QH_ITEMS 4
#define QH_INTS(cap) (QH_ITEMS + (cap)) /* of one queue with room for cap superblocks */

/* The superblocks whose reconstruction superblock sb reads (-1: none), as
 * the single-frame intra phase waits for them. */
DEVI void intra_deps(const Mav1FrameParams &fp, int sb, int dep[4]) {
  const int r = sb / fp.sb_cols, c = sb - r * fp.sb_cols;
  const int ts = (c / fp.tile_w_sb) * fp.tile_w_sb, te = d_min(fp.sb_cols, ts + fp.tile_w_sb);
  dep[0] = c > ts ? sb - 1 : -1;
  dep[1] = r > 0 && c > ts ? sb - fp.sb_cols - 1 : -1;
  dep[2] = r > 0 ? sb - fp.sb_cols : -1;
  dep[3] = r > 0 && c + 1 < te ? sb - fp.sb_cols + 1 : -1;
}

DEVI void queue_push(int *q, int v) {
  const int slot = atomicAdd(&q[QH_TAIL], 1);
  __hip_atomic_store(&q[QH_ITEMS + slot], v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}

#endif
