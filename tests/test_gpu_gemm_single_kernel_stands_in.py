"""Uncut products that the path query gives to packed operands or the direct kernel and that the single
kernel runs in their place: the bits of the reported path, its refusals, and its K slices for the
tiles of a partly empty last round."""
import pytest
import torch

from wmma_extension_amd._lib import WmmaeError

pytestmark = pytest.mark.gpu

PACKED, DIRECT = 2, 8


def _operands(dev, m, n, k, batch):
    g = torch.Generator(device="cpu").manual_seed(m + 1000 * n + 7 * k)
    return [(torch.rand(s, generator=g) * 2 - 1).to(dev) for s in ((batch, m, k), (batch, n, k), (batch, n, m))]


def _call(tc, A, B, C0, m, n, k, batch, policy, flags, ws, beta):
    C = C0.clone()
    tc.sgemm_strided_batched("T", "N", m, n, k, 1.25, A, k, m * k, B, k, n * k, beta, C, m, m * n, batch, policy,
                             flags, ws)
    return C


# (of the products below: where the single kernel is not ahead, or the path's last round of tiles is cut)
STAY = {(1500, 1100, 1030), (1024, 5000, 2052), (3000, 3000, 2050)}


@pytest.mark.parametrize("m,n,k,batch,policy,rn", [
    (96, 1792, 798, 8, 0, 1), (3072, 416, 499, 1, 2, 0), (704, 384, 309, 16, 2, 1), (1160, 1544, 1056, 1, 0, 0),
    (808, 128, 185, 1, 0, 1), (192, 150, 319, 32, 1, 0), (286, 32, 185, 279, 0, 0), (64, 334, 775, 60, 0, 0),
    (1025, 1030, 515, 3, 3, 0), (32, 32, 1727, 200, 2, 0), (218, 64, 185, 3, 2, 0), (1500, 1100, 1030, 2, 4, 0),
    (1024, 5000, 2052, 1, 0, 0), (3000, 3000, 2050, 1, 2, 0), (1, 1, 101, 1, 0, 0),
    (3072, 416, 499, 1, 4, 0), (2000, 1100, 99, 1, 1, 0)])
def test_bits_of_the_reported_path(tc, dev, m, n, k, batch, policy, rn):
    A, B, C0 = _operands(dev, m, n, k, batch)
    path = tc.sgemm_path(m, n, k, batch, policy, rn)
    flag = DIRECT if path in (tc.PATH_DIRECT, tc.PATH_DIRECT_SPLIT_K) else PACKED
    ws = torch.empty(tc.workspace_bytes(m, n, k, batch, policy), dtype=torch.uint8, device=dev)
    kernel = tc.sgemm_route("T", "N", m, n, k, k, k, batch, policy, rn, ws)[0]
    assert path != tc.PATH_FUSED and (kernel != 0) == ((m, n, k) in STAY)
    for beta in (0.0, -0.5):
        want = _call(tc, A, B, C0, m, n, k, batch, policy, flag | rn, ws, beta)
        got = _call(tc, A, B, C0, m, n, k, batch, policy, rn, ws, beta)
        assert torch.isfinite(want).all()
        assert torch.equal(want.view(torch.int32), got.view(torch.int32)), (path, (want - got).abs().max())


@pytest.mark.parametrize("m,n,k,batch,policy", [(3072, 416, 499, 1, 2), (1160, 1544, 1056, 1, 0), (63, 130, 6403, 1, 2)])
def test_a_workspace_that_is_too_small_is_still_refused(tc, dev, m, n, k, batch, policy):
    """What packed operands would not fit in, cut (the last one, with room for its slices' sums) or not."""
    A, B, C0 = _operands(dev, m, n, k, batch)
    assert tc.sgemm_path(m, n, k, batch, policy) in (tc.PATH_PACKED, tc.PATH_PACKED_SPLIT_K)
    need = tc.pack_bytes(m, k, batch, policy) + tc.pack_bytes(n, k, batch, policy)
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    _call(tc, A, B, C0, m, n, k, batch, policy, 0, ws, 0.0)
    with pytest.raises(WmmaeError) as e:
        _call(tc, A, B, C0, m, n, k, batch, policy, 0, ws[:need - 16], 0.0)
    assert e.value.status == -5
