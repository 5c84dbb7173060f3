"""Which kernel a GEMM call runs and how it cuts K (wmmae_tcec_sgemm_route, host only): the kernel that
stands in for another path makes that path's cut, whatever workspace the call is given."""
import ctypes
import os
import random
import re

import pytest

from wmma_extension_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ALIGNED = 1 << 20                     # an address that is never read
SINGLE, PACKED, DIRECT = 0, 1, 3
STATIC_BYTES = 64 << 20               # the fixed array of wmmae_tcec_sgemm_static


@pytest.fixture(scope="module")
def h():
    if not os.path.exists(_lib.LIB_PATH):
        _lib.build()
    return _lib.lib()


def _route(h, ta, tb, m, n, k, batch, policy, room, flags=0, address=ALIGNED, lda=None, ldb=None):
    out = (ctypes.c_int * 3)()
    st = h.wmmae_tcec_sgemm_route(ta, tb, m, n, k, lda or (k if ta == b"T" else m), ldb or (k if tb == b"N" else n),
                                  batch, policy, flags, None if room is None else address, room or 0, out)
    assert st == 0
    return tuple(out)


def _bytes(h, m, n, k, batch, policy):
    """(packed operands, the slices' sums behind them)"""
    a, b, c = (ctypes.c_size_t(0) for _ in range(3))
    assert h.wmmae_tcec_pack_bytes(m, k, batch, policy, ctypes.byref(a)) == 0
    assert h.wmmae_tcec_pack_bytes(n, k, batch, policy, ctypes.byref(b)) == 0
    assert h.wmmae_tcec_gemm_packed_workspace_bytes(policy, m, n, k, batch, ctypes.byref(c)) == 0
    return a.value + b.value, c.value


def test_header_and_library_agree(h):
    text = open(os.path.join(ROOT, "include", "wmmae_tcec_route.h")).read()
    names = set(re.findall(r"\b(wmmae_[a-z0-9_]+)\s*\(", text))
    assert names and names <= set(_lib._SIGNATURES) and all(getattr(h, x) is not None for x in names)


def test_bad_arguments(h):
    out = (ctypes.c_int * 3)()
    ok = [b"T", b"N", 64, 64, 64, 64, 64, 1, 0, 0, None, 0, out]
    assert h.wmmae_tcec_sgemm_route(*ok) == 0
    for i, v in ((0, b"X"), (1, b"?"), (2, 0), (3, -1), (4, 0), (7, 0), (8, 9), (9, 2), (9, 64)):
        assert h.wmmae_tcec_sgemm_route(*(ok[:i] + [v] + ok[i + 1:])) == -1, i
    assert h.wmmae_tcec_sgemm_route(*ok[:-1], None) == -2


# products whose path leaves K whole on a workspace that holds the packed operands alone (the last:
# 58 MiB of operands and 26 MiB of sums in the 64 MiB of the fixed array)
UNCUT = [(b"T", b"N", 63, 130, 6403, 2, 0), (b"N", b"N", 256, 256, 8192, 0, 0), (b"N", b"T", 200, 160, 10735, 2, 1),
         (b"N", b"N", 700, 500, 12500, 0, 0)]


@pytest.mark.parametrize("ta,tb,m,n,k,policy,flags", UNCUT)
def test_no_room_for_the_sums_behind_packed_operands(h, ta, tb, m, n, k, policy, flags):
    operands, sums = _bytes(h, m, n, k, 1, policy)
    assert sums > 0 and _route(h, ta, tb, m, n, k, 1, policy, operands + sums, flags)[1] > 1
    assert _route(h, ta, tb, m, n, k, 1, policy, operands, flags) == (PACKED, 1, 0)
    assert _route(h, ta, tb, m, n, k, 1, policy, operands + sums - 1, flags) == (PACKED, 1, 0)
    if operands <= STATIC_BYTES < operands + sums:
        assert _route(h, ta, tb, m, n, k, 1, policy, STATIC_BYTES, flags) == (PACKED, 1, 0)


def test_forced_tile(h):
    """The hook chooses among what the rules allow: never more than the cut and the room there is."""
    operands, sums = _bytes(h, 300, 129, 6403, 1, 0)
    full = _route(h, b"N", b"N", 300, 129, 6403, 1, 0, operands + sums)
    try:
        for tile in (64, 128, -1):
            assert h.wmmae_tcec_force_spread_tile(tile) == 0
            got = _route(h, b"N", b"N", 300, 129, 6403, 1, 0, operands + sums)
            assert got[1] == full[1] and got[2] == max(tile, 0) and (tile < 0 or got[0] == SINGLE)
            assert _route(h, b"N", b"N", 300, 129, 6403, 1, 0, operands) == (PACKED, 1, 0)
            assert _route(h, b"N", b"N", 64, 64, 64, 1, 0, operands) == (SINGLE, 1, 0)
        assert h.wmmae_tcec_force_spread_tile(32) == -1
    finally:
        assert h.wmmae_tcec_force_spread_tile(0) == 0
    assert _route(h, b"N", b"N", 300, 129, 6403, 1, 0, operands + sums) == full


@pytest.mark.parametrize("ta,tb,m,n,k,batch,policy,tile", [
    # slower with a workgroup a slice than without (us, with and without), by the path they stand in for:
    (b"T", b"N", 1248, 96, 1024, 4, 0, 0),        # the single kernel's slices one after the other: 20.6, 16.0
    (b"T", b"N", 96, 5952, 1312, 1, 0, 0),        # 23.1, 18.2
    (b"N", b"T", 68, 2738, 891, 1, 4, 0),         # 14.4, 11.5
    (b"T", b"N", 256, 288, 6176, 1, 0, 0),        # packed operands: 30.2, 23.9
    (b"T", b"T", 158, 92, 5248, 4, 1, 0),         # 25.7, 20.6
    (b"T", b"N", 250, 381, 5798, 1, 0, 0),        # 29.3, 24.3
    (b"T", b"N", 3616, 256, 1696, 3, 0, 0),       # the direct kernel: 56.7, 46.5
    (b"T", b"N", 128, 5376, 7232, 1, 1, 0),       # one term: 41.0, 37.7
    # faster so
    (b"N", b"N", 2005, 64, 23136, 1, 0, 64),     # 42, 147
    (b"T", b"N", 32, 480, 7332, 1, 0, 64),        # 18, 26
    (b"T", b"N", 128, 96, 7463, 1, 0, 64),        # 17.3, 21.8
    (b"T", b"N", 128, 658, 5052, 17, 4, 128),     # 91, 142
    (b"T", b"N", 5632, 71, 36018, 1, 2, 128)])    # 322, 670
def test_slices_of_a_workgroup_each_where_they_are_faster(h, ta, tb, m, n, k, batch, policy, tile):
    """(256 compute units, which is also the answer without a device)"""
    cu = ctypes.c_longlong(256)
    h.wmmae_query(1, ctypes.byref(cu))
    if cu.value != 256:
        pytest.skip("measured on 256 compute units")
    assert _route(h, ta, tb, m, n, k, batch, policy, sum(_bytes(h, m, n, k, batch, policy)))[2] == tile


@pytest.mark.parametrize("m,n,k,batch,kernel", [
    # (us in the single kernel and on packed operands)
    (1862, 1719, 3244, 24, PACKED),                # 3636, 3165
    (1264, 6597, 1312, 1, PACKED),                 # 187.5, 174.0
    (4842, 8160, 211, 1, PACKED),                  # 137.3, 126.2
    (896, 3509, 1473, 1, SINGLE),                  # 67.6, 73.5
    (64, 1122, 1088, 1, SINGLE),                   # 20.0, 25.7
    (1061, 1472, 768, 7, SINGLE)])                 # 125.5, 130.5
def test_three_terms_with_adds_outside_the_matrix_core(h, m, n, k, batch, kernel):
    cu = ctypes.c_longlong(256)
    h.wmmae_query(1, ctypes.byref(cu))
    if cu.value != 256:
        pytest.skip("measured on 256 compute units")
    assert _route(h, b"T", b"N", m, n, k, batch, 2, sum(_bytes(h, m, n, k, batch, 2)), 1) == (kernel, 1, 0)


def test_cut_of_random_products(h):
    rng = random.Random(7)
    cut = stood_in = 0
    for _ in range(4000):
        m, n, k = (int(2 ** rng.uniform(0, e)) for e in (12, 12, 16))
        batch, policy = rng.choice([1, 1, 1, 2, 5, 40]), rng.randrange(5)
        ta, tb = rng.choice([(b"T", b"N"), (b"N", b"N"), (b"N", b"T"), (b"T", b"T")])
        flags = int(policy in (0, 2) and rng.random() < 0.2)
        operands, sums = _bytes(h, m, n, k, batch, policy)
        full = _route(h, ta, tb, m, n, k, batch, policy, operands + sums, flags)
        if full[1] == 1:
            assert full[2] == 0
            continue
        cut += 1
        stood_in += full[2] > 0
        # (what needs no packed operands is not turned down on sixteen bytes)
        needs_operands = _route(h, ta, tb, m, n, k, batch, policy, 16, flags)[0] == PACKED
        for room in (operands, operands + sums - 1):
            got = _route(h, ta, tb, m, n, k, batch, policy, room, flags)
            if needs_operands:
                assert got == (PACKED, 1, 0), (ta, tb, m, n, k, batch, policy, flags, room)
            elif got[0] == SINGLE:
                assert got[1] == full[1]
            else:                     # the direct kernel: its sums alone
                assert got[0] == DIRECT and got[1] == (full[1] if room >= 4 * full[1] * batch * m * n else 1)
        assert _route(h, ta, tb, m, n, k, batch, policy, operands + sums, flags, ALIGNED + 4)[2] == 0
    assert cut > 300 and stood_in > 200


@pytest.mark.parametrize("m,n,k,batch,policy", [(1, 961, 101, 1 << 26, 0), (2, 1500, 103, 1 << 26, 0), (64, 961, 333, 1 << 26, 0),
                                                (65, 4096, 333, 1 << 24, 2), (128, 961, 131, 1 << 25, 2)])
def test_more_tiles_than_the_single_kernel_counts(h, m, n, k, batch, policy):
    """It would turn them down; the path that the query reports has larger tiles and runs them."""
    path = ctypes.c_int(-1)
    assert h.wmmae_tcec_sgemm_path(m, n, k, batch, policy, 0, ctypes.byref(path)) == 0 and path.value in (PACKED, DIRECT)
    assert -(-m // 64) * -(-n // 64) * batch >= 1 << 30
    assert _route(h, b"T", b"N", m, n, k, batch, policy, 1 << 62) == (path.value, 1, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb,m,n,k,policy,flags", UNCUT)
def test_bits_without_room_for_the_sums(tc, dev, ta, tb, m, n, k, policy, flags):
    import torch
    ta, tb = ta.decode(), tb.decode()
    lda, ldb = (k if ta == "T" else m), (k if tb == "N" else n)
    g = torch.Generator(device="cpu").manual_seed(m + n + k)
    A, B = ((torch.rand((x, k), generator=g) * 2 - 1).to(dev).view(-1) for x in (m, n))
    need = tc.pack_bytes(m, k, 1, policy) + tc.pack_bytes(n, k, 1, policy)
    ws = torch.empty(need, dtype=torch.uint8, device=dev)

    def call(flag):
        C = torch.zeros((n, m), device=dev)
        tc.sgemm(ta, tb, m, n, k, 1.0, A, lda, B, ldb, 0.0, C, m, policy, flag | flags, ws)
        return C
    want, got = call(tc.FLAG_PATH_PACKED), call(0)
    assert torch.isfinite(want).all() and torch.equal(want, got)
    if need <= STATIC_BYTES < tc.workspace_bytes(m, n, k, 1, policy):
        C = torch.zeros((n, m), device=dev)
        tc.sgemm_static(ta, tb, m, n, k, 1.0, A, lda, B, ldb, 0.0, C, m, policy, flags)
        assert torch.equal(C, want)
