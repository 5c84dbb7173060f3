"""K slices made inside the single kernel: where it stands in for a path that cuts K, its result has
that path's bits (slices summed from cleared accumulators, rounded to fp32, added in double
precision), so that no product is summed in a longer chain for being small.  The calls get a
workspace of 16 bytes, with which the packed path refuses and the direct one does not cut: only the
single kernel can give the sliced bits there.  Expected: the path's own run, whose bits are pinned
against the matrix core's model elsewhere."""
import pytest
import torch

pytestmark = pytest.mark.gpu

PACKED, DIRECT = 2, 8
LAYOUTS = [("T", "N"), ("N", "N"), ("N", "T"), ("T", "T")]


def _same_bits(tc, dev, ta, tb, m, n, k, batch, policy, rn, pad, alpha, beta, path):
    g = torch.Generator(device="cpu").manual_seed(m + 1000 * n + 7 * k + policy)
    lda, ldb, ldc = (k if ta == "T" else m) + pad, (k if tb == "N" else n) + pad, m + pad
    A = (torch.rand((batch, m if ta == "T" else k, lda), generator=g) * 2 - 1).to(dev)
    B = (torch.rand((batch, n if tb == "N" else k, ldb), generator=g) * 2 - 1).to(dev)
    C0 = (torch.rand((batch, n, ldc), generator=g) * 2 - 1).to(dev)
    out = []
    for flag, size in ((path, tc.workspace_bytes(m, n, k, batch, policy)), (0, 16)):
        C = C0.clone()
        ws = torch.empty(size, dtype=torch.uint8, device=dev)
        tc.sgemm_strided_batched(ta, tb, m, n, k, alpha, A, lda, A.stride(0), B, ldb, B.stride(0), beta, C, ldc,
                                 n * ldc, batch, policy, flag | rn, ws)
        out.append(C)
    case = (ta, tb, m, n, k, batch, policy, rn)
    assert torch.isfinite(out[0]).all()
    assert torch.equal(out[0].view(torch.int32), out[1].view(torch.int32)), (case, (out[0] - out[1]).abs().max())


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("policy", [0, 1, 2, 3, 4])
def test_slices_of_every_length(tc, dev, ta, tb, policy):
    # odd and even stage counts, a last slice of one stage, k that ends inside a stage, one tile to
    # several per workgroup, entries owned by an XCD
    for m, n, k, batch, slices in ((65, 60, 416, 3, 2), (64, 64, 32 * 14, 1, 2), (500, 300, 32 * 21 - 4, 1, 3),
                                   (200, 700, 32 * 16 + 4, 1, 2), (390, 450, 32 * 25, 1, 4), (61, 63, 32 * 18, 40, 3),
                                   (40, 50, 640, 600, 3), (777, 500, 900, 9, 4), (777, 500, 32 * 19, 9, 3),
                                   (1000, 1000, 32 * 31 - 8, 1, 5), (900, 800, 32 * 43, 1, 7)):
        with tc.forced_k_slices(slices):
            assert tc.sgemm_k_slices(m, n, k, batch, policy, PACKED) == slices
            _same_bits(tc, dev, ta, tb, m, n, k, batch, policy, 0, 4 if m == 500 else 0, 1.0, 0.0, PACKED)
            if batch < 9:
                _same_bits(tc, dev, ta, tb, m, n, k, batch, policy, 0, 3, -0.75, 1.5, PACKED)


@pytest.mark.parametrize("policy", [0, 2])
def test_leading_product_outside_the_matrix_core(tc, dev, policy):
    for ta, tb, m, n, k, batch, slices in (("T", "N", 65, 60, 416, 3, 2), ("N", "N", 40, 50, 640, 600, 3),
                                           ("N", "T", 777, 500, 900, 9, 4)):
        with tc.forced_k_slices(slices):
            _same_bits(tc, dev, ta, tb, m, n, k, batch, policy, tc.FLAG_RN_MAIN, 0, 1.0, 0.5, PACKED)


@pytest.mark.parametrize("policy", [0, 2])
def test_the_cut_that_the_estimates_plan(tc, dev, policy):
    """1024^3 and products whose operands do not have k contiguous, with the cut the driver plans: the
    count wmmae_tcec_sgemm_k_slices gives for the packed path, whatever kernel makes the slices."""
    for ta, tb in LAYOUTS:
        assert tc.sgemm_k_slices(1024, 1024, 1024, 1, policy, 0) == 4
        assert tc.sgemm_path(1024, 1024, 1024, 1, policy) == tc.PATH_PACKED_SPLIT_K
        _same_bits(tc, dev, ta, tb, 1024, 1024, 1024, 1, policy, 0, 0, 1.0, 0.0, PACKED)
    for ta, tb in LAYOUTS[1:]:
        assert tc.sgemm_k_slices(320, 321, 1290, 8, policy, PACKED) == 3
        _same_bits(tc, dev, ta, tb, 320, 321, 1290, 8, policy, 0, 0, 1.0, 0.0, PACKED)
    # slices as the direct kernel plans them, where that is the path the single kernel stands in for
    if policy == 0:
        assert tc.sgemm_path(32, 128, 1216, 64, policy) == tc.PATH_DIRECT_SPLIT_K
        _same_bits(tc, dev, "T", "N", 32, 128, 1216, 64, policy, 0, 0, 1.0, 0.0, DIRECT)
