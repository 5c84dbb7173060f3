/*
 * Which kernel a call of libwmmae_tcec.so's GEMM entry points runs: for the test
 * suite and for measurements, no part of the product ABI (include/wmmae_tcec.h).
 * Same conventions: return 0 or a negative wmmae_status.
 */
#ifndef WMMAE_TCEC_ROUTE_H
#define WMMAE_TCEC_ROUTE_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Host only, no device access (no counterpart in the reference): what a call of
 * wmmae_tcec_sgemm* with these arguments and this workspace (an address, never
 * read) runs.  flags: 0 or WMMAE_FLAG_RN_MAIN.  route[0]: 0 the single kernel, 1
 * packed operands, 3 the GEMM kernel on the fp32 operands; route[1]: the K slices
 * made, 1: none; route[2]: the tile (64 or 128) with which the single kernel makes
 * them a workgroup each, else 0.  What a call turns down (for its workspace, or a
 * policy without that flag) is answered as packed operands. */
int wmmae_tcec_sgemm_route(char transa, char transb, int m, int n, int k,
                           int lda, int ldb, int batch, int policy, int flags,
                           const void *workspace, size_t workspace_bytes,
                           int *route);

/* Test hook (no counterpart in the reference): where the calling thread's next
 * wmmae_tcec_sgemm* calls cut K and the workspace has the room, the single kernel
 * makes the slices a workgroup each, with tiles of this size (64 or 128); -1: it
 * never does; 0: the estimates choose. */
int wmmae_tcec_force_spread_tile(int tile);

#ifdef __cplusplus
}
#endif
#endif /* WMMAE_TCEC_ROUTE_H */
