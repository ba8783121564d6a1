"""Every load of the GEMM's LDS ring that a wait may leave in flight touches
memory.

The ring's waits count outstanding loads, which holds only if loads complete
in issue order, and a buffer load whose every lane falls outside its
descriptor can complete ahead of older ones. csrc/gemm_ring.h decides which
rows and K tiles each load takes; compiled here for the host, its functions
are walked over the loads of a block as the kernel issues them (prologue, main
loop, edge steps) for every tile, ragged rows and columns, K tails, LoRA
segments, K slices that end inside the ring and empty slices.
"""

import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "deltaserve-vllm_amd", "csrc")
# (BM, BN, A slots, B slots) of the five tiles, 4 waves each
TILES = [(256, 256, 2, 3), (256, 128, 3, 3), (128, 128, 2, 3), (128, 64, 3, 3), (64, 64, 5, 5)]
NW = 4


@pytest.fixture(scope="module")
def ring(tmp_path_factory):
    d = tmp_path_factory.mktemp("ring")
    src = d / "ring.cpp"
    src.write_text('#include "gemm_ring.h"\nusing namespace dsb;\nextern "C" {\n'
                   "int row_block(int r, int n) { return ring_row_block(r, n); }\n"
                   "int last_block(int r, int s, int n) { return ring_last_block(r, s, n); }\n"
                   "int fast_end(int a, int b, int w, int n) { return ring_fast_end(a, b, w, n); }\n"
                   "int whole_tiles(int kn, int nk, int n) { return ring_whole_tiles(kn, nk, n); }\n"
                   "int kn_live(int r, int n) { return ring_kn_live(r, n); }\n"
                   "int clamps_a(int na) { return ring_clamps_a(na); }\n"
                   "int prologue_wait(int na, int nb, int ia, int ib, int r) {\n"
                   "  return ring_prologue_wait(na, nb, ia, ib, r); }\n}\n")
    so = d / "ring.so"
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", str(src), "-o", str(so)],
                   check=True)
    return ctypes.CDLL(str(so))


def _rows(edge):
    return sorted({1, 7, 8, 9, 31, 32, 33, edge // 2, edge // 2 + 1, edge - 8, edge - 7, edge} - {0})


@pytest.mark.parametrize("BM,BN,NA,NB", TILES)
def test_row_blocks_exist(ring, BM, BN, NA, NB):
    """A and [N, K] B loads: the 8-row block a load takes has a row."""
    for size in (BM, BN):
        for rows in _rows(size):
            for wave in range(NW):
                first = ring.row_block(8 * wave, rows)
                last = ring.last_block(8 * wave, 8 * NW, rows)
                for j in range(size // (8 * NW)):
                    r = 8 * (wave + j * NW)
                    a = first + min(j, last) * 8 * NW
                    b = ring.row_block(r, rows)
                    assert 0 <= a < rows and 0 <= b < rows, (size, rows, wave, j)
                    if r < rows:  # its own rows where it has some
                        assert a == b == r


@pytest.mark.parametrize("kn", [False, True])
@pytest.mark.parametrize("BM,BN,NA,NB", TILES)
def test_k_tiles_exist(ring, BM, BN, NA, NB, kn):
    """K tiles: main-loop steps load only tiles of the block, whole ones of the
    first segment; edge steps and the prologue send every load without a row
    to the zero page; the steps together cover the block's tiles once."""
    rpl = 64 // (BN // 8)  # LDS rows of a [K, N] load
    for K1 in (8, 64, 72, 128, 200, 256, 512, 1024, 1032):
        for K2 in (0, 8, 24, 64, 72):
            for kb in (0, K1 - 1, K1 - 7) if kn and K2 == 0 else (0,):
                nk1, nk2 = -(-K1 // 64), -(-K2 // 64)
                nk = nk1 + nk2
                rows1 = kb or K1
                for ks in (1, 2, 3, 4, 7):
                    kc = -(-nk // ks)
                    for z in range(ks):
                        kt0 = min(nk, z * kc)
                        kt1 = min(nk, kt0 + kc)
                        end = ring.fast_end(kt0, kt1, ring.whole_tiles(int(kn), nk1, rows1), NB)
                        assert kt0 <= end <= max(kt0, kt1)
                        for kt in range(kt0, end):
                            a, b = kt + NA, kt + NB
                            assert a < kt1 and a < nk1 and a * 64 < K1
                            assert b < kt1 and b < nk1
                            assert b * 64 + 64 <= rows1 if kn else b * 64 < K1
                        for b in range(kt0, kt1 + NB):  # edge: any tile from here on
                            s1 = b < nk1
                            live = 0 if b >= kt1 else (rows1 if s1 else K2) - (b if s1 else b - nk1) * 64
                            if b < kt1:
                                assert live > 0
                            for wave in range(NW):
                                for j in range(BN // (8 * NW)):
                                    r = rpl * (wave + j * NW)
                                    assert bool(ring.kn_live(r, live)) == (r < live)


@pytest.mark.parametrize("BM,BN,NA,NB", TILES)
def test_waits_cover_their_tiles(ring, BM, BN, NA, NB):
    """A wait that leaves n loads in flight guarantees a load that touches
    memory if at least n more such loads were issued after it (were it still
    in flight, so would they be). Walked over the kernel's issue order with A
    row blocks past M completing at once where they may: the prologue's wait
    for the first tile, each step's for the next one, the last steps' for what
    is left."""
    ia, ib = BM // (8 * NW), BN // (8 * NW)
    for rows in _rows(BM):
        for tiles in range(1, 2 * NB + 3):
            for wave in range(NW):
                live = [bool(ring.clamps_a(NA)) or 8 * (wave + j * NW) < rows for j in range(ia)]
                log = []  # (operand, tile, touches memory) in issue order

                def fill(a, b):
                    if a is not None:
                        # spare slots of a short block read the zero page
                        log.extend(("A", a, a >= tiles or t) for t in live)
                    if b is not None:
                        log.extend([("B", b, True)] * ib)

                def covered(tile, n):
                    for op in "AB":
                        at = [i for i, (o, k, t) in enumerate(log) if o == op and k == tile and t]
                        if at and sum(t for _, _, t in log[at[-1] + 1:]) < n:
                            return False
                    return True

                if NB > NA:
                    fill(None, 0)
                for t in range(NA):
                    fill(t, t + NB - NA)
                ragged = not ring.clamps_a(NA) and rows < BM
                assert covered(0, ring.prologue_wait(NA, NB, ia, ib, int(ragged)))
                step = (NA - 2) * (ia + ib) + (ib if NB > NA else 0)
                for kt in range(tiles):
                    left = tiles - kt
                    if left > NA:
                        n = step
                    else:
                        n = step if left >= NB else 2 * (ia + ib) if NA > 4 and left == 4 else \
                            ia + ib if NA > 3 and left == 3 else 0
                    if kt + 1 < tiles:
                        assert covered(kt + 1, n), (rows, tiles, wave, kt)
                    if kt < tiles - NB:
                        fill(kt + NA, kt + NB)
                    elif NB > NA and kt < tiles - NA:
                        fill(kt + NA, None)
