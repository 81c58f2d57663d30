/* The intra phase of frames whose luma blocks search transform types or depths. */
#include "recon_intra.h"

hipError_t launch_recon_intra_search(hipStream_t st, const Mav1FrameParams &fp, Mav1BlockInfo *blocks,
                                     const Mav1SbInfo *sbs, const uint8_t *src, uint8_t *rec, int32_t *coefs,
                                     const int32_t *mats, int *iwork, int workgroups) {
  hipLaunchKernelGGL(k_recon_intra<true>, dim3(workgroups), dim3(RT), 0, st, fp, blocks, sbs, src, rec, coefs, mats,
                     iwork, 1 << 20);
  return hipGetLastError();
}

hipError_t launch_recon_intra_search_b(hipStream_t st, const BatchFrame *T, int n, int *q, int workgroups) {
  hipLaunchKernelGGL(k_recon_intra_b<true>, dim3(workgroups), dim3(RT), 0, st, T, n, q, 1 << 20);
  return hipGetLastError();
}
