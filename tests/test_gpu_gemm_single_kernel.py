"""The single-launch kernel at its edges: every way it reads an operand (k contiguous, rows
contiguous, strides of 2^24 floats, k < 4), last stages of every length, row counts that end inside
a load, one tile to several per workgroup with both tile sizes, with NaN around the operands.
Expected: the bits of pack + GEMM on packed operands without K slices, whose own bits are pinned
against the matrix core's model elsewhere."""
import pytest
import torch

pytestmark = pytest.mark.gpu

PACKED, FUSED = 2, 4


def _operand(g, dev, batch, rows, k, k_contiguous, pad, off):
    """(view of rows x k values inside NaN, leading dimension)"""
    outer, inner = (rows, k) if k_contiguous else (k, rows)
    ld = inner + pad
    room = torch.full((off + batch * outer * ld + 8,), float("nan"), device=dev)
    X = room[off:off + batch * outer * ld].view(batch, outer, ld)
    X[:, :, :inner] = (torch.rand((batch, outer, inner), generator=g) * 2 - 1).to(dev)
    return X, ld


def _same_bits(tc, dev, ta, tb, m, n, k, batch, policy, rn, pad, off, beta):
    g = torch.Generator(device="cpu").manual_seed(m + 1000 * n + 7 * k + policy)
    A, lda = _operand(g, dev, batch, m, k, ta == "T", pad, off)
    B, ldb = _operand(g, dev, batch, n, k, tb == "N", pad, off)
    C0 = (torch.rand((batch, n, m), generator=g) * 2 - 1).to(dev)
    out = []
    for flag in (PACKED, FUSED):
        C = C0.clone()
        with tc.forced_k_slices(1):
            # (no workspace of the caller: no K slices for the tiles of a last round either)
            tc.sgemm_strided_batched(ta, tb, m, n, k, 1.25, A, lda, A.stride(0), B, ldb, B.stride(0), beta, C, m,
                                     m * n, batch, policy, flag | rn, None)
        out.append(C)
    assert torch.isfinite(out[0]).all()
    assert torch.equal(out[0].view(torch.int32), out[1].view(torch.int32)), (m, n, k, (out[0] - out[1]).abs().max())


@pytest.mark.parametrize("ta,tb", [("T", "N"), ("N", "N"), ("N", "T"), ("T", "T")])
@pytest.mark.parametrize("policy", [0, 1, 2, 3, 4])
def test_same_bits_as_packed_operands(tc, dev, ta, tb, policy):
    # k: 1 .. 3 (element by element), ends of a stage, ends of the ring of stages
    for k in (1, 2, 3, 4, 5, 30, 31, 32, 33, 34, 35, 63, 64, 65, 96, 127, 131, 190, 225, 260):
        _same_bits(tc, dev, ta, tb, 65 + k % 3, 130 - k % 5, k, 1, policy, 0, k % 4, k % 4, 0.0)
    # row counts around tiles, 64-row loads and row blocks
    for m, n in ((1, 1), (7, 66), (15, 17), (63, 129), (64, 64), (127, 257), (200, 8)):
        _same_bits(tc, dev, ta, tb, m, n, 77, 2, policy, 0, 3, 1, -0.5)
    # several tiles per workgroup: 64x64 and 128x128, shared list and entries owned by an XCD,
    # odd and even stage counts, one stage per tile
    for m, n, k, batch in ((60, 50, 37, 1100), (60, 50, 64, 1030), (130, 100, 29, 700), (1500, 1300, 131, 3),
                           (1500, 1300, 64, 3), (900, 1000, 20, 9)):
        _same_bits(tc, dev, ta, tb, m, n, k, batch, policy, 0, 0, 0, 0.0)


@pytest.mark.parametrize("policy", [0, 2])
def test_leading_product_outside_the_matrix_core(tc, dev, policy):
    for ta, tb, m, n, k, batch in (("T", "N", 70, 130, 95, 1), ("N", "T", 300, 200, 161, 9),
                                   ("N", "N", 1500, 1300, 100, 3)):
        _same_bits(tc, dev, ta, tb, m, n, k, batch, policy, tc.FLAG_RN_MAIN, 1, 2, 0.5)


def test_strides_beyond_the_offsets_of_a_load(tc, dev):
    """Leading dimensions of 2^24 floats and more (a lane's offset from the wave's address then no
    longer fits its 32 bits)."""
    for ta, tb, m, n, k in (("T", "N", 5, 40, 36), ("N", "T", 40, 5, 6), ("N", "N", 33, 3, 5)):
        _same_bits(tc, dev, ta, tb, m, n, k, 1, 0, 0, (1 << 24) + 1, 0, 0.0)


@pytest.mark.parametrize("ta,tb", [("T", "N"), ("N", "N"), ("N", "T"), ("T", "T")])
def test_pointer_arrays_in_every_layout(tc, dev, ta, tb):
    """Matrices by pointer, scattered at every alignment a float can have, with one and with several tiles
    per workgroup: the bits of the strided call on the same matrices."""
    for m, n, k, batch, policy in ((70, 50, 77, 9, 0), (40, 60, 515, 3, 2), (61, 50, 37, 600, 0), (200, 150, 3, 300, 3)):
        g = torch.Generator(device="cpu").manual_seed(m + k)
        A, lda = _operand(g, dev, batch, m, k, ta == "T", 1, 0)
        B, ldb = _operand(g, dev, batch, n, k, tb == "N", 2, 0)
        C0 = (torch.rand((batch, n, m), generator=g) * 2 - 1).to(dev)
        want = C0.clone()
        tc.sgemm_strided_batched(ta, tb, m, n, k, 1.5, A, lda, A.stride(0), B, ldb, B.stride(0), -0.5, want, m, m * n,
                                 batch, policy, FUSED)
        rooms, arrays = [], []
        for i, X in enumerate((A, B, C0)):
            size = X[0].numel() + 11 + 2 * i                     # no multiple of four floats: all alignments
            room = torch.full((batch, size), float("nan") if i < 2 else 7.0, device=dev)
            order = [(5 * e + i) % batch if batch % 5 else batch - 1 - e for e in range(batch)]
            for e in range(batch):
                room[order[e], i + 1:i + 1 + X[0].numel()] = X[e].reshape(-1)
            base = room.data_ptr()
            arrays.append(torch.tensor([base + 4 * (order[e] * size + i + 1) for e in range(batch)], dtype=torch.int64,
                                       device=dev))
            rooms.append((room, order))
        tc.sgemm_batched(ta, tb, m, n, k, 1.5, arrays[0], lda, arrays[1], ldb, -0.5, arrays[2], m, batch, policy, FUSED)
        room, order = rooms[2]
        got = room[order, 3:3 + n * m].view(batch, n, m)
        assert torch.equal(got.view(torch.int32), want.view(torch.int32)), (ta, tb, m, n, k, batch)
        assert (room[:, :3] == 7.0).all() and (room[:, 3 + n * m:] == 7.0).all()


@pytest.mark.parametrize("policy", [0, 1, 2])
def test_element_by_element_with_several_tiles_per_workgroup(tc, dev, policy):
    """k < 4 with k contiguous (64-bit addresses, one element a load), more tiles than resident workgroups:
    64x64 and 128x128 tiles, shared list and entries owned by an XCD."""
    for m, n, k, batch in ((60, 50, 3, 1100), (60, 50, 1, 700), (130, 100, 2, 700), (1500, 1300, 3, 3),
                           (4000, 3000, 2, 1)):
        _same_bits(tc, dev, "T", "N", m, n, k, batch, policy, 0, 1, 1, 0.5)


def test_events_around_the_single_kernel(tc, dev):
    """wmmae_tcec_time_gemm_kernel on products that the driver gives to the single kernel, which a caller
    of another layout than 'T','N' cannot ask for: the events enclose it.  No kernel takes less time than its
    matrix products at the nominal 2.5 PFLOP/s (16 to 18 us here; two events with nothing between them are a few
    microseconds apart)."""
    for policy, k, products in ((2, 515, 6), (0, 900, 3)):
        m, n, batch = 777, 1333, 7
        A, lda = _operand(torch.Generator().manual_seed(1), dev, batch, m, k, False, 0, 0)
        B, ldb = _operand(torch.Generator().manual_seed(2), dev, batch, n, k, True, 0, 0)
        C = torch.empty((batch, n, m), device=dev)
        e0, e1, w0, w1 = (torch.cuda.Event(enable_timing=True) for _ in range(4))
        inner, whole = [], []
        for _ in range(5):
            w0.record()
            with tc.timed_gemm_kernel(e0, e1):
                tc.sgemm_strided_batched("N", "N", m, n, k, 1.0, A, lda, A.stride(0), B, ldb, B.stride(0), 0.0, C, m,
                                         m * n, batch, policy)
            w1.record()
            torch.cuda.synchronize()
            inner.append(e0.elapsed_time(e1))
            whole.append(w0.elapsed_time(w1))
        floor_ms = products * 2.0 * batch * m * n * k / 2.5e15 * 1e3
        assert floor_ms < min(inner) <= min(whole), (floor_ms, inner, whole)
