"""The epilogue of the GEMM kernels at the edges of their pieces of C: rows and columns that end one
to three short of or past a 16x16 tile, a 32-row pair of tiles or a wave's piece, leading dimensions
and bases of C at every alignment a float can have, with and without beta, and large enough for
several work items per workgroup.  Expected: the bits of the same product stored to an aligned,
padded C with beta = 0 (its own bits are pinned against the matrix core's model elsewhere), then one
fused multiply-add of beta * C."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

PACKED, FUSED, DIRECT = 2, 4, 8


@pytest.mark.parametrize("flag,policy", [(f, p) for f in (PACKED, FUSED, DIRECT) for p in (0, 1, 2)
                                         if (f, p) != (DIRECT, 2)])   # direct: one and two terms only
@pytest.mark.parametrize("m,n,batch", [(1, 1, 1), (3, 17, 1), (61, 63, 2), (255, 129, 1), (258, 131, 1), (271, 127, 9),
                                       (289, 257, 1), (172, 384, 3), (384, 256, 1), (1030, 515, 3), (777, 200, 70)])
def test_edges_of_a_piece_of_c(tc, orc, dev, flag, policy, m, n, batch):
    _edges(tc, orc, dev, flag, policy, m, n, batch)


@pytest.mark.parametrize("flag,policy", [(f | 1, p) for f in (PACKED, FUSED) for p in (0, 2)])
@pytest.mark.parametrize("m,n,batch", [(3, 17, 1), (61, 63, 2), (172, 384, 3), (258, 131, 1), (271, 127, 9),
                                       (384, 256, 1), (777, 200, 70)])
def test_edges_with_the_leading_product_outside(tc, orc, dev, flag, policy, m, n, batch):
    _edges(tc, orc, dev, flag, policy, m, n, batch)


def _edges(tc, orc, dev, flag, policy, m, n, batch):
    k = 100
    g = torch.Generator(device="cpu").manual_seed(m * 1000 + n)
    A = (torch.rand((batch, m, k), generator=g) * 2 - 1).to(dev)
    B = (torch.rand((batch, n, k), generator=g) * 2 - 1).to(dev)
    lda16 = -(-m // 16) * 16
    plain = torch.zeros((batch, n, lda16), device=dev)
    ws = torch.empty(max(16, tc.workspace_bytes(m, n, k, batch, policy)), dtype=torch.uint8, device=dev)

    def product(C, ldc, beta):
        tc.sgemm_strided_batched("T", "N", m, n, k, 1.0, A, k, m * k, B, k, n * k, beta, C, ldc, n * ldc, batch,
                                 policy, flag, ws)
    product(plain, lda16, 0.0)
    base = plain[:, :, :m].cpu().numpy()
    for off, pad, beta in ((0, 0, 0.0), (1, 0, 0.0), (0, 1, -1.5), (3, 2, 0.75), (2, 3, 1.0)):
        ldc = m + pad
        room = torch.full((off + batch * n * ldc + 5,), 7.0, device=dev)
        C = room[off:off + batch * n * ldc]
        old = (torch.rand((batch, n, m), generator=g) * 2 - 1)
        C.view(batch, n, ldc)[:, :, :m] = old.to(dev)
        product(C, ldc, beta)
        got = room.cpu().numpy()
        assert (got[:off] == 7.0).all() and (got[off + batch * n * ldc:] == 7.0).all(), (off, pad)
        got = got[off:off + batch * n * ldc].reshape(batch, n, ldc)
        assert (got[:, :, m:] == 7.0).all(), (off, pad)
        want = orc.epilogue(base.reshape(-1, m), 1.0, beta, old.numpy().reshape(-1, m)) if beta else base
        got = np.ascontiguousarray(got[:, :, :m]).reshape(-1, m)
        want = np.ascontiguousarray(want).reshape(-1, m)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (off, pad, beta, int((got != want).sum()))
