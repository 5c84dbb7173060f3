"""K slices made by a workgroup each in the single kernel, the last of a tile's adding them: the bits of
the slices on packed operands (pinned against the matrix core's model elsewhere), whatever the
workspace held before, from one call to the next and in a replayed graph, and nothing written past
the room the slices' sums and the tiles' counts need."""
import pytest
import torch

pytestmark = pytest.mark.gpu

PACKED = 2
LAYOUTS = [("T", "N"), ("N", "N"), ("N", "T"), ("T", "T")]


def _room(m, n, batch, slices):
    return max(-(-m // t) * -(-n // t) * batch * (slices * t * t * 4 + 8) for t in (64, 128))


def _check(tc, dev, ta, tb, m, n, k, batch, policy, rn=0, pad=0, alpha=1.0, beta=0.0, tile=0, pointers=False):
    """tile: the one that has to run, 0 whichever is chosen, if any."""
    slices = tc.sgemm_k_slices(m, n, k, batch, policy, PACKED)
    assert slices > 1, (m, n, k)
    g = torch.Generator(device="cpu").manual_seed(m + 1000 * n + 7 * k + policy)
    lda, ldb, ldc = (k if ta == "T" else m) + pad, (k if tb == "N" else n) + pad, m + pad
    A = (torch.rand((batch, m if ta == "T" else k, lda), generator=g) * 2 - 1).to(dev)
    B = (torch.rand((batch, n if tb == "N" else k, ldb), generator=g) * 2 - 1).to(dev)
    C0 = (torch.rand((batch, n, ldc), generator=g) * 2 - 1).to(dev)

    def call(flag, ws):
        C = C0.clone()
        if flag == 0 and tile:
            assert tc.sgemm_route(ta, tb, m, n, k, lda, ldb, batch, policy, rn, ws) == (0, slices, tile)
        if pointers:
            arrays = [torch.tensor([e.data_ptr() for e in X], dtype=torch.int64, device=dev) for X in (A, B, C)]
            tc.sgemm_batched(ta, tb, m, n, k, alpha, arrays[0], lda, arrays[1], ldb, beta, arrays[2], ldc, batch,
                             policy, flag | rn, ws)
            return C
        tc.sgemm_strided_batched(ta, tb, m, n, k, alpha, A, lda, A.stride(0), B, ldb, B.stride(0), beta, C, ldc,
                                 n * ldc, batch, policy, flag | rn, ws)
        return C

    want = call(PACKED, torch.empty(tc.workspace_bytes(m, n, k, batch, policy), dtype=torch.uint8, device=dev))
    assert torch.isfinite(want).all()
    size = max(_room(m, n, batch, slices), tc.workspace_bytes(m, n, k, batch, policy))
    room = torch.randint(0, 256, (size + 4096,), dtype=torch.uint8, device=dev)
    guard = room[size:].clone()
    for _ in range(3):
        got = call(0, room[:size])
        assert torch.equal(want.view(torch.int32), got.view(torch.int32)), (ta, tb, m, n, k, batch, policy, rn)
        room[:size // 2].random_(0, 256)
    assert torch.equal(room[size:], guard)
    if tile and tc.sgemm_route(ta, tb, m, n, k, lda, ldb, batch, policy, rn) == (0, slices, tile):
        got = call(0, None)
        assert torch.equal(want.view(torch.int32), got.view(torch.int32)), "workspace allocated by the call"


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("policy", [0, 1, 2, 3, 4])
def test_slices_of_a_workgroup_each(tc, dev, ta, tb, policy):
    # a tile's remainder of every kind, k that ends inside a stage, a last slice of one stage, 2 .. 32
    # slices, one tile to many, several entries
    for m, n, k, batch, slices in ((65, 60, 416, 3, 2), (1, 5, 700, 2, 3), (93, 162, 6403, 1, 29), (64, 64, 8192, 1, 32),
                                   (130, 259, 2048, 2, 10), (333, 100, 2241, 1, 11), (40, 50, 640, 60, 3),
                                   (61, 63, 32 * 19, 5, 3)):
        with tc.forced_k_slices(slices):
            assert tc.sgemm_k_slices(m, n, k, batch, policy, PACKED) == slices
            _check(tc, dev, ta, tb, m, n, k, batch, policy)
            _check(tc, dev, ta, tb, m, n, k, batch, policy, 0, 3, -0.75, 1.5)


@pytest.mark.parametrize("policy,m,n,k,slices", [(0, 2150, 736, 1985, 2), (2, 3104, 66, 8180, 10), (0, 4797, 160, 3104, 3),
                                                 (3, 2150, 736, 1985, 2), (2, 1984, 800, 4100, 2)])
def test_large_tiles(tc, dev, policy, m, n, k, slices):
    """Products that take 128x128 tiles."""
    with tc.forced_k_slices(slices), tc.forced_spread_tile(128):
        for ta, tb in LAYOUTS[1:]:
            _check(tc, dev, ta, tb, m, n, k, 1, policy, 0, 0, 1.0, 0.0, 128)
        _check(tc, dev, "N", "T", m, n, k, 1, policy, 0, 1, 0.5, 0.5, 128)


@pytest.mark.parametrize("policy", [0, 2])
def test_leading_product_outside_the_matrix_core(tc, dev, policy):
    for ta, tb, m, n, k, slices in (("T", "N", 93, 162, 6403, 29), ("N", "N", 200, 100, 4097, 7),
                                    ("N", "T", 1444, 448, 9000, 4)):
        with tc.forced_k_slices(slices):
            _check(tc, dev, ta, tb, m, n, k, 1, policy, tc.FLAG_RN_MAIN, 1, 1.25, -0.5)


@pytest.mark.parametrize("tile", [64, 128])
@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("policy", [0, 1, 2, 3, 4])
def test_each_tile(tc, dev, policy, ta, tb, tile):
    """Every variant of the kernel, whatever the estimates would choose: tiles with a remainder of every
    kind, several entries, k that ends inside a stage, matrices by pointer, and with fp32 adds outside
    the matrix core where the policy has them."""
    with tc.forced_spread_tile(tile):
        for m, n, k, batch, slices in ((65, 60, 416, 3, 2), (1, 5, 700, 2, 3), (130, 259, 2048, 2, 10), (300, 129, 6403, 1, 32)):
            with tc.forced_k_slices(slices):
                _check(tc, dev, ta, tb, m, n, k, batch, policy, tile=tile)
                _check(tc, dev, ta, tb, m, n, k, batch, policy, 0, 3, -0.75, 1.5, tile, pointers=True)
                if policy in (0, 2):
                    _check(tc, dev, ta, tb, m, n, k, batch, policy, tc.FLAG_RN_MAIN, 1, tile=tile)


def test_replayed_graph(tc, dev):
    """A captured launch keeps its number: the counts it leaves must not look like arrivals of the next
    replay, whatever else used the workspace in between."""
    m, n, k = 200, 100, 6400
    A, B = torch.rand((m, k), device=dev), torch.rand((n, k), device=dev)
    C = torch.zeros((n, m), device=dev)
    for slices in (2, 20, 32):
        with tc.forced_k_slices(slices):
            ws = torch.randint(0, 256, (tc.workspace_bytes(m, n, k),), dtype=torch.uint8, device=dev)

            def call():
                tc.sgemm("T", "N", m, n, k, 1.0, A, k, B, k, 0.0, C, m, 0, 0, ws)

            side = torch.cuda.Stream()
            with torch.cuda.stream(side):
                call()
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                call()
            for r in range(5):
                A.mul_(1.0 if r % 2 else -0.5)
                call()
                torch.cuda.synchronize()
                want = C.clone()
                C.zero_()
                if r == 2:
                    ws.random_(0, 256)
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(C, want), (slices, r)
