"""The GEMM on the public device API with each of its block tiles (64x64; 128x128 with eight and with
four waves, by the number of tiles): one stage of k and several, odd and even, padded rows, alpha and
beta, matrices by pointer.  Expected: the bits of the single kernel over an uncut K, which makes the
same products in the same order (pinned against the matrix core's model elsewhere)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

FUSED = 4
# driver policy -> (operand type, error correction) of tcec.api_gemm
TYPES = {0: (0, 1), 1: (0, 0), 2: (2, 1), 3: (1, 1), 4: (1, 0)}


@pytest.mark.parametrize("policy", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("m,n,k", [(128, 128, 32), (256, 384, 96), (1024, 2048, 64), (1920, 1920, 160), (128, 18816, 32),
                                   (2176, 2176, 96), (2176, 2176, 32), (4096, 1152, 320),
                                   (2176, 2176, 3104), (2176, 2176, 544)])
def test_bits_of_the_single_kernel(tc, dev, policy, m, n, k):
    type_, ec = TYPES[policy]
    pad = 4 if m == 1920 else 0
    g = torch.Generator(device="cpu").manual_seed(m + n + k)
    A, B = ((torch.rand((r, k + pad), generator=g) * 2 - 1).to(dev) for r in (m, n))
    want, got = (torch.zeros((n, m), device=dev) for _ in range(2))
    # (mma_rz_sync chains the leading product through the matrix core, as the driver does; mma_sync with error
    # correction and mma_rn_sync add it outside, as the driver does with its flag)
    for rounding, rn in ((2, 0), (0, tc.FLAG_RN_MAIN if ec else 0)):
        if rn and policy == 3:
            continue                                        # the driver has no such variant of this policy
        tc.sgemm("T", "N", m, n, k, 1.0, A, k + pad, B, k + pad, 0.0, want, m, policy, FUSED | rn)
        tc.api_gemm(type_, ec, m, n, k, 1.0, A, k + pad, B, k + pad, 0.0, got, m, rounding=rounding)
        assert torch.isfinite(want).all()
        assert torch.equal(want.view(torch.int32), got.view(torch.int32)), (rounding, (want - got).abs().max())


@pytest.mark.parametrize("policy", [0, 2])
def test_matrices_by_pointer_with_every_tile(tc, dev, policy):
    type_, ec = TYPES[policy]
    m, n, k = 384, 256, 96
    for batch in (3, 40, 50):                               # 18, 240 and 300 tiles of 128x128
        A, B = torch.rand((batch, m, k), device=dev) - 0.5, torch.rand((batch, n, k), device=dev) - 0.5
        C0 = torch.rand((batch, n, m), device=dev)
        C = C0.clone()
        arrays = [torch.tensor([x.data_ptr() for x in X], dtype=torch.int64, device=dev) for X in (A, B, C)]
        tc.api_gemm_batched(type_, ec, m, n, k, 0.5, arrays[0], k, arrays[1], k, -1.5, arrays[2], m, batch)
        one = C0.clone()
        for e in range(batch):
            tc.api_gemm(type_, ec, m, n, k, 0.5, A[e], k, B[e], k, -1.5, one[e], m)
        assert torch.equal(C.view(torch.int32), one.view(torch.int32))
