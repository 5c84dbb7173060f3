"""Host-side LDS bank analysis of the layouts the GEMM kernels use (the reference does this on
the device for its shared-memory skew, research/bank-conflict/main.cu:38-71, and settles on a
skew from it, test/tcec/batch_gemm.cu:11).

The model is measured, not assumed.  Two-lane probes on gfx950 (two active lanes touching the
same bank at different addresses; SQ_LDS_BANK_CONFLICT says whether they were served in the same
cycle) and stride scans under SQ_LDS_BANK_CONFLICT / SQ_LDS_IDX_ACTIVE gave:

  ds_read_b128   4 cycles; the lanes of a cycle are the lane quads 0 3 5 6 | 1 2 4 7 |
                 8 11 13 14 | 9 10 12 15 (quad q = lanes 4q .. 4q+3); 64 banks of 4 bytes
  ds_read_b64    2 cycles of 32 consecutive lanes; 64 banks
  ds_write_b64   4 cycles of 16 consecutive lanes; bank b and bank b + 32 collide (the write
                 path is 128 bytes wide)
  ds_write_b128  8 cycles of 8 consecutive lanes; likewise 32 banks

An instruction takes, per cycle group, as many cycles as the most loaded bank has distinct
addresses.  The literal cycle counts of the stride scans below are the counters' readings (per
instruction, 1000 repetitions each), which the model has to reproduce; the kernels' own layouts
are then evaluated with it and compared with what rocprofv3 reads for them."""
import os
import re

import numpy as np

QUADS_OF_CYCLE = ((0, 3, 5, 6), (1, 2, 4, 7), (8, 11, 13, 14), (9, 10, 12, 15))


def _groups(op):
    if op == "read_b128":
        return [[4 * q + i for q in quads for i in range(4)] for quads in QUADS_OF_CYCLE], 64
    if op == "read_b64":
        return [list(range(32 * p, 32 * p + 32)) for p in range(2)], 64
    if op == "write_b64":
        return [list(range(16 * p, 16 * p + 16)) for p in range(4)], 32
    if op == "write_b128":
        return [list(range(8 * p, 8 * p + 8)) for p in range(8)], 32
    raise ValueError(op)


def cycles(op, byte_addr):
    """LDS cycles of one 64-lane instruction with the given per-lane byte addresses."""
    width = {"read_b128": 16, "write_b128": 16, "read_b64": 8, "write_b64": 8}[op]
    groups, banks = _groups(op)
    total = 0
    for lanes in groups:
        per_bank = {}
        for lane in lanes:
            for w in range(width // 4):
                dword = int(byte_addr[lane]) // 4 + w
                per_bank.setdefault(dword % banks, set()).add(dword)
        total += max(len(v) for v in per_bank.values())
    return total


def free(op):
    return len(_groups(op)[0])


LANE = np.arange(64)


def test_model_reproduces_the_measured_stride_scans():
    """Lane l reads 16 bytes of row l % R at float 8 * (l / R) of a tile with a row stride of ld
    floats (R = 16: an operand fragment of the 16x16x32 instruction read from a row-major fp32
    tile; R = 32: the 32-row pattern).  Counter readings per instruction, ld = 32 .. 72."""
    measured_16 = {32: 16, 36: 8, 40: 8, 44: 8, 48: 8, 52: 8, 56: 8, 60: 8, 64: 32, 68: 8, 72: 8}
    measured_32 = {32: 32, 36: 4, 40: 8, 44: 4, 48: 16, 52: 4, 56: 8, 60: 4, 64: 64, 68: 4, 72: 8}
    for ld, want in measured_16.items():
        addr = ((LANE % 16) * ld + 8 * (LANE // 16)) * 4
        assert cycles("read_b128", addr) == want, ld
    for ld, want in measured_32.items():
        addr = ((LANE % 32) * ld + 8 * (LANE // 32)) * 4
        assert cycles("read_b128", addr) == want, ld


def test_fragment_major_chunks_are_conflict_free():
    """Packed operands: lane l reads base + 16*l."""
    assert cycles("read_b128", 16 * LANE) == free("read_b128")


def _direct_swizzle(q):
    return (12 * (q & 1)) ^ (4 * (q >> 1))


def _swizzle_of_the_kernels():
    """direct_swizzle of tcec_gemm_kernels.hpp, evaluated from the source's own expression."""
    path = os.path.join(os.path.dirname(__file__), "..", "wmma_extension_amd", "csrc", "tcec_gemm_kernels.hpp")
    body = re.search(r"constexpr unsigned direct_swizzle\(const unsigned q\) \{\s*return ([^;]+);", open(path).read())
    return [eval(re.sub(r"(\d)u", r"\1", body.group(1)), {"q": q}) for q in range(4)]


def test_single_kernel_term_buffers():
    """The single kernel's producers write terms into 1 KiB chunks (a row block's 16 rows x 32 k, position
    (row r, k group g) at 16-byte slot 16g + (r ^ swizzle(g))) in one of two patterns.  Rows contiguous:
    lane = row of 64, 16 bytes of one k group each, lanes l / 16 = 0 .. 3 in four chunks.  k contiguous: eight
    lanes to a row, 8 bytes each, rows 8h .. 8h + 7.  The consumers read a chunk's 64 positions, 16 bytes a
    lane.  Both sides cover a chunk exactly once."""
    swz = np.array(_swizzle_of_the_kernels())
    assert list(swz) == [_direct_swizzle(q) for q in range(4)]
    for terms in (1, 2, 3):
        for g in range(4):
            addr = (LANE >> 4) * (terms * 1024) + 256 * g + 16 * ((LANE & 15) ^ swz[g])
            assert cycles("write_b128", addr) == free("write_b128"), (terms, g)
    rows = np.concatenate([256 * g + 16 * (np.arange(16) ^ swz[g]) for g in range(4)])
    assert sorted(rows) == list(range(0, 1024, 16))
    halves = []
    for h in range(2):
        r, g = 8 * h + (LANE >> 3), (LANE & 7) >> 1
        addr = 256 * g + 16 * (r ^ swz[g]) + 8 * (LANE & 1)
        assert cycles("write_b64", addr) == 8          # banks b and b + 32, as in the direct kernel below
        halves += list(addr)
    assert sorted(halves) == list(range(0, 1024, 8))
    read = 16 * ((LANE & 48) + ((LANE & 15) ^ swz[LANE >> 4]))
    assert cycles("read_b128", read) == free("read_b128")
    assert sorted(read) == list(range(0, 1024, 16))


def test_direct_kernel_image_writes_and_reads():
    """The GEMM kernel that splits the fp32 operands itself writes each term of a row block as
    8-byte halves of the fragment positions (two writes per term, position (row r, k group q) at
    16-byte slot 16q + (r ^ swz(q))).  The fragment reads are conflict free; an 8-byte write of
    sixteen consecutive lanes touches 32 different banks, but on the 128-byte write path banks b
    and b + 32 collide: two-way, 8 cycles instead of 4.  Per stage and wave: 24 such writes and 24
    fragment reads, so SQ_LDS_BANK_CONFLICT / SQ_LDS_IDX_ACTIVE = 96 / 288 = 33.3 % - what the
    counters read for this kernel (33.3 % and 33.5 % on the K-heavy and the batched workload)."""
    swz = np.array([_direct_swizzle(q) for q in range(4)])
    write_cycles = []
    for h in range(2):
        r, q = 8 * h + (LANE >> 3), (LANE & 7) >> 1
        woff = 256 * q + 16 * (r ^ swz[q]) + 8 * (LANE & 1)
        write_cycles.append(cycles("write_b64", woff))
    assert write_cycles == [8, 8]
    slot = (LANE & 48) + ((LANE & 15) ^ swz[LANE >> 4])
    assert cycles("read_b128", 16 * slot) == 4
    assert sorted(slot) == list(range(64))                       # a permutation of the chunk
    writes = reads = 24
    conflict = writes * (8 - free("write_b64"))
    active = writes * 8 + reads * 4
    assert abs(conflict / active - 1 / 3) < 1e-12
    # 16-byte writes (a lane owning a whole fragment position, eight lanes = two rows x four k
    # groups) with slot 16q + (r ^ 2q) would be conflict free on both sides; the kernel built that
    # way ran at the same speed (the matrix pipe does not wait for the LDS here) and is not kept
    r, q = LANE >> 2, LANE & 3
    assert cycles("write_b128", 16 * (16 * q + (r ^ (2 * q)))) == free("write_b128")
    assert cycles("read_b128", 16 * ((LANE & 48) + ((LANE & 15) ^ (2 * (LANE >> 4))))) == 4


def test_api_level_kernel_tiles():
    """The GEMM written on the public API stages fp32 tiles of 32 k per row.  A fragment load
    takes lane l's eight floats of row l % 16 from k = 8 * (l / 16) on, as two 128-bit reads.
    No row padding makes that pattern conflict free (the scan above: every stride that is a
    multiple of four floats costs at least two-way; the reference's skew of 8 floats, chosen for
    32 banks and 32 lanes, too).  Unpadded rows with the 16-byte pieces of row r stored at piece
    index p ^ ((r / 2) & 5) are: that is the tile tcec::load_matrix_sync reads with the
    swizzled memory layout tags, and the counter reads 0 conflicts for it."""
    r, g = LANE % 16, LANE // 16
    for ld in (32, 36, 40):
        addr = (r * ld + 8 * g) * 4
        assert cycles("read_b128", addr) > 4 and cycles("read_b128", addr + 16) > 4
    f = (r >> 1) & 5
    for e in range(2):
        assert cycles("read_b128", r * 128 + 16 * ((2 * g + e) ^ f)) == 4
    # the writer's side: a direct global -> LDS copy fills 64 consecutive 16-byte pieces, eight
    # rows; lane l's piece is physical piece l % 8 of row l / 8, i.e. logical piece
    # (l % 8) ^ f(row): every logical piece of every row exactly once
    seen = {(row, (l % 8) ^ ((row >> 1) & 5)) for row in range(16) for l in range(8)}
    assert len(seen) == 128
