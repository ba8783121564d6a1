// Which rows and K tiles the loads of the GEMM's LDS ring (gemm_nt.h) take, in
// plain arithmetic for host and device.
//
// The ring's waits count outstanding loads (s_waitcnt vmcnt(N), N > 0) and so
// rest on loads completing in issue order. A load whose every lane falls
// outside its buffer descriptor never reaches memory and can complete ahead of
// older ones, so no such load is among those that a wait leaves in flight: a
// load without a row or K tile of its own takes one that exists (what it lands
// is multiplied into nothing that is stored) or the zero page. With two A slots
// the waits leave only B loads in flight, and A row blocks past M stay out of
// range: they cost nothing, where loading others' rows took the 831-row cycle
// of a 5120-wide layer and a 151936-word head from 3832 to 3995 µs.
#pragma once

#if defined(__HIP__)
#define DSB_HD __host__ __device__ __forceinline__
#else
#define DSB_HD inline
#endif

namespace dsb {

// First row of the 8-row block that a load fills the LDS rows r .. r + 7 with:
// r, or row 0 where the tile has `rows` (>= 1) of them and r is past the last
// (outputs of those rows are not stored).
DSB_HD int ring_row_block(int r, int rows) { return r < rows ? r : 0; }

// Whether A row blocks past M take one that exists, for a ring of na A slots.
DSB_HD constexpr bool ring_clamps_a(int na) { return na > 2; }

// Loads that the prologue's wait for its first tile may leave in flight: those
// issued after that tile's, or, where A row blocks past M may be out of range
// (`ragged`), the B loads among them.
DSB_HD constexpr int ring_prologue_wait(int na, int nb, int ia, int ib, bool ragged) {
  return (na - 1) * ((ragged ? 0 : ia) + ib) + (nb > na ? ib : 0);
}

// The same for a wave whose load j takes the block at ring_row_block(r) +
// min(j, last)·step: the number of the last one that exists.
DSB_HD int ring_last_block(int r, int step, int rows) { return r < rows ? (rows - 1 - r) / step : 0; }

// K tiles [first, end) of a block may be loaded without a look at where the
// operands end (the main loop's steps, which load up to `ahead` tiles beyond
// their own): the number of those steps' end, for a block of tiles [kt0, kt1)
// and `whole` tiles whose every row of K exists.
DSB_HD int ring_fast_end(int kt0, int kt1, int whole, int ahead) {
  const int last = kt1 < whole ? kt1 : whole;
  return kt0 > last - ahead ? kt0 : last - ahead;
}

// K tiles of segment 1 whose every load touches memory: all of them for
// operands stored along K (a row's chunk 0 exists in every tile), those with
// all 64 rows for a [K, N] operand of `rows` rows.
DSB_HD int ring_whole_tiles(bool kn, int nk1, int rows) { return kn ? rows / 64 : nk1; }

// A [K, N] load of the LDS rows r .. of a K tile with `live` rows: whether it
// has one (else it reads the zero page; its rows past K multiply zeros of A).
DSB_HD bool ring_kn_live(int r, int live) { return r < live; }

}  // namespace dsb
