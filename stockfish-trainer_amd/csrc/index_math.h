// Index arithmetic shared by the gfx950 FT kernels and their host launchers:
// magic-number division, the XCD-aware tile schedule, the column maps of the
// 32-column tiles and the long-segment rule of the sorted backward.  Plain
// integer code with no HIP dependency, so that it also builds as host C++ (the
// CPU tests compile it with g++ and the address/undefined-behaviour
// sanitizers).
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define SFT_HD __host__ __device__
#else
#define SFT_HD
#endif

namespace sft {

SFT_HD inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
SFT_HD inline int round_up4(int v) { return (v + 3) & ~3; }

// ---- bucket sort over (position chunk, feature) keys: key = chunk * N + f ----
// Buckets hold 2^sb consecutive keys.  The first n buckets hold every key of
// chunk 0 and key N, the first of chunk 1, whose segment start ends chunk 0's
// last segment; n is the fewest that do (0 with one chunk or no features).
SFT_HD inline int buckets_through_chunk0(int64_t N, int nchunks, int sb) {
  if (nchunks < 2 || N <= 0) return 0;
  const int64_t nb = ceil_div((int64_t)nchunks * N, (int64_t)1 << sb);
  const int64_t n = (N >> sb) + 1;
  return (int)(n < nb ? n : nb);
}

// ---- n / d for 32-bit n by a divisor fixed at launch ----
// Multiply-high by a magic number (Granlund & Montgomery 1994, round-up
// variant): with l = ceil(log2 d) and m = floor(2^32 (2^l - d) / d) + 1,
// n / d = (t + ((n - t) >> 1)) >> (l - 1) where t = mulhi(m, n), for d >= 2;
// d = 1 returns n.
SFT_HD inline uint32_t mulhi32(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }
struct FastDiv {
  uint32_t d, mul, shift;
  FastDiv() = default;
  SFT_HD explicit FastDiv(uint32_t div) : d(div), mul(0), shift(0) {
    uint32_t l = 0;
    while (((uint64_t)1 << l) < div) ++l;
    shift = l;
    mul = (uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << l) - div)) / div + 1);
  }
  SFT_HD uint32_t operator()(uint32_t n) const {
    if (d == 1) return n;
    const uint32_t t = mulhi32(mul, n);
    return (t + ((n - t) >> 1)) >> (shift - 1);
  }
};

// ---- the row gather's mapping of few positions ----
// Whether B positions of `cols` 16-byte row chunks and K slots are gathered by a
// wave per position and 64 chunks, 16 rows in flight, instead of the general
// mapping (G lanes a position with cpl chunks each, 4 rows in flight).  A
// position's rows are one chain of memory round trips, so the few-position
// mapping wins while the launch is latency, the longer the more chunks the
// general mapping's lanes take in turn, and loses once its waves or the rows'
// bytes are what takes the time.  General / few-position, us:
//   N = 23 232, K = 32: L = 40 (G = 16, cpl = 1) 2048 6 / 5, 3072 6 / 7, 8192 7 / 11;  L = 136 (8, 5) 2048 14 / 6,
//   8192 17 / 16;  L = 168 (16, 3) 4096 14 / 11, 8192 17 / 19;  L = 248 (64, 1) 2048 10 / 9, 4096 15 / 16;
//   L = 264 (16, 5) 2048 15 / 11, 4096 18 / 20;  L = 520 (32, 5) 1024 15 / 11, 2048 19 / 19, 4096 31 / 34;
//   L = 904 (64, 4) 1024 17 / 17, 2048 28 / 34;  L = 1048 (64, 5) 256 14 / 8, 1536 26 / 26, 2048 33 / 34
//   N = 85 296, K = 160: L = 56 3072 28 / 20, 6144 30 / 35;  L = 136 6144 67 / 63, 8192 77 / 81;  L = 168 4096 53 / 50,
//   6144 73 / 75;  L = 248 2048 37 / 36, 3072 51 / 54;  L = 264 1536 54 / 35, 3072 64 / 67;  L = 392 512 32 / 20,
//   1536 45 / 47;  L = 520 1024 52 / 43, 1536 63 / 67;  L = 1048 512 61 / 46, 1024 80 / 85;  L = 2048 512 105 / 77
SFT_HD inline bool few_positions(int64_t B, int K, int64_t cols, int G, int cpl) {
  if (cols > 1 << 21) return false;  // a launch's column slabs stay below 2^16
  const int64_t slabs = ceil_div(cols, 64);
  if (slabs > 1) {  // the waves times their slots, and the batch
    const int64_t halves = cpl > 4 ? 2 * (cpl - 3) : G < 64 ? 3 : 2;
    return B <= (halves * 5 << 15) / (K * slabs) && B <= (cpl > 4 || G < 64 ? 2048 : 1536);
  }
  if (cpl == 1) return B <= (K > 64 && cols <= 16 ? 4096 : K > 32 && cols <= 32 ? 3072 : 2048);
  return B <= (G > 8 ? 4096 : K <= 32 && cpl > 4 ? 8192 : 6144);
}

// ---- which sorts run on the caller's stream ----
// A sort of M = B K slots runs beside the kernels that do not need it, on a side
// stream, or in line before them.  A fork and join cost the host about 27 us and
// the GPU about 10 us; in line, nothing hides the sort's launches, most of which
// fill few CUs.  So small sorts go in line, and the lines are where a step of
// both perspectives takes as long either way (narrow: K >= L / 5, whose forward
// runs the radix pass and whose backward the buckets; one_part: the table fits
// one gather pass).  GPU time forked / in line with the host ahead, us; with the
// host the slower one, short steps gain 50-100 us more by the sort in line.
//
// The prepared sort's part in the forward.  The more the gather moves, the more
// it hides: for lists of more than 32 slots the line is on M L.
//   K = 32, N = 23 232, L = 136: B = 16 384 173 / 159, 65 536 385 / 376, 100 000 548 / 537, 131 072
//   741 / 725;  N = 85 296: 65 536 696 / 691, 131 072 1159 / 1169
//   K = 64, N = 23 232, L = 264: 8192 235 / 238, 16 384 305 / 320 (host-bound 402 / 313), 32 768 492 / 505 (a step
//   waited for by itself, on a slow host 707 / 589), 65 536 898 / 921;  K = 128, L = 520: 5000 378 / 394 (host-bound
//   408 / 386), 8000 468 / 484 (by itself 663 / 564)
//   K = 160, N = 85 296, L = 136: 8192 391 / 384, 10 000 444 / 453;  L = 520: 1000 348 / 343, 3000 601 / 617;
//   L = 800: 1000 469 / 462, 3000 811 / 828
// Wide rows (the whole sort in the forward): K = 64, N = 23 232, L = 1048: 1000 238 / 227, 2048 347 / 348;
// K = 32, L = 264: 6000 170 / 164, 12 000 192 / 194;  K = 160, N = 85 296, L = 1048: 409 502 / 514, but a step
// waited for by itself 686 / 631.
SFT_HD inline bool sort_in_line_fwd(int64_t M, int K, int L, bool narrow, bool one_part) {
  if (!narrow) return M <= 1 << 16;
  if (K > 32 && M * L > (one_part ? (int64_t)5 << 27 : (int64_t)3 << 26)) return false;
  return M <= (one_part ? 3 << 20 : 1 << 21);
}
// The backward's: the buckets of a prepared sort, or (not prepared) the whole sort.
// Buckets (the forward's part as above): K = 32, N = 23 232, L = 136: 65 536 387 / 376, 100 000 543 / 537,
// 160 000 893 / 902;  N = 85 296: 65 536 705 / 691, 131 072 1161 / 1169;  K = 8, N = 4000, L = 32: 262 144
// 439 / 438, 500 000 659 / 714;  K = 160, N = 85 296, L = 136: 8192 413 / 391, 16 384 576 / 555;
// L = 264: 20 000 944 / 930.
// Whole sort, one backward: L = 136, K = 32: 8192 57 / 47, 65 536 136 / 133, 131 072 260 / 265;
// a step, L = 1048: 2048 258 / 251, 3000 310 / 316 (host-bound 358 / 316), 8192 407 / 414.
SFT_HD inline bool sort_in_line_bwd(int64_t M, int K, bool narrow, bool prepared, bool one_part) {
  if (!narrow) return M <= 1 << 16;
  return M <= (!prepared || (K <= 32 && !one_part) ? 1 << 21 : 3 << 20);
}
// Both perspectives' sort of a composed or epilogue backward over a table of so
// many values, M slots each.  Steps that the host bounds gain 40 us in line, and
// from about 500 us of kernels on none is bound by it: forked / in line, B = 300,
// composed, N = 24 576, L = 1048 297 / 252, N = 85 296: L = 648 390 / 335 (a faster host 327 / 324), L = 1048 447 / 453;
// epilogue, N = 24 576: L = 264 325 / 285, L = 1048 350 / 349 (waited for by itself 561 / 537), N = 85 296: L = 264
// 350 / 305, L = 648 439 / 415 (a faster host 393 / 412), L = 808 488 / 505 (alone 700 / 675), L = 1048 606 / 623.
SFT_HD inline bool sort_in_line_pair(int64_t M, int64_t table) { return M <= 1 << 16 && table <= 80 * (int64_t)1000000; }

// ---- XCD-aware tile schedule ----
// MI355X runs a dispatch's workgroups round-robin over its 8 XCDs (workgroup i
// on XCD i % 8), and each XCD has its own 4 MB L2.  Tiled kernels give every
// XCD whole column tiles: workgroup i serves the (i / 8)-th item of XCD i % 8,
// where XCD x owns tiles x, x + 8, ... (all chunks of one tile, then the next).
// The rem = ntiles % 8 tiles left after the last full round are cut into 8
// strands each -- strand s of leftover tile t holds its chunks s, s + 8, ...,
// so every strand has the same mix of early (long) and late chunks -- and XCD
// x takes the rem consecutive strands [x rem, (x + 1) rem) of the sequence
// (t, s): every XCD gets the same work (rem strands, +-1 chunk each) from at
// most two leftover tiles, the first one's strands before the second's, in
// chunk order.  (With rem = 5 tiles, whole tiles per XCD group would leave two
// XCDs alone on a tile each while the others share one.)  A workgroup with no
// item gets tile = ntiles.  Any other placement only costs locality, never
// results.
constexpr int kXcds = 8;
struct TileItem {
  int tile, chunk;
};
SFT_HD inline int64_t tile_sched_items_per_xcd(int ntiles, int nchunks) {
  const int full = ntiles / kXcds, rem = ntiles % kXcds;
  return (int64_t)full * nchunks + (int64_t)rem * ((nchunks + kXcds - 1) / kXcds);
}
// The item of a workgroup, in 32-bit arithmetic with the chunk count's magic
// divisor made at launch: every workgroup starts with it, and 64-bit divisions
// there cost a tiled gather's workgroup about a tenth of a microsecond each.
struct TileSched {
  int ntiles, nchunks;
  FastDiv by_chunks;
  TileSched() = default;
  SFT_HD TileSched(int tiles, int chunks) : ntiles(tiles), nchunks(chunks), by_chunks((uint32_t)(chunks > 0 ? chunks : 1)) {}
  // i / n for n <= 7, i < 2^29: i * ceil(2^32 / n) >> 32.
  static SFT_HD uint32_t div_small(uint32_t i, uint32_t n) {
    const uint32_t m = n == 2 ? 0x80000000u : n == 3 ? 0x55555556u : n == 4 ? 0x40000000u : n == 5 ? 0x33333334u
                       : n == 6 ? 0x2aaaaaabu : 0x24924925u;
    return n <= 1 ? i : mulhi32(i, m);
  }
  SFT_HD TileItem item(uint32_t bid) const {
    const uint32_t xcd = bid % kXcds, j = bid / kXcds;
    const uint32_t full = (uint32_t)ntiles / kXcds, rem = (uint32_t)ntiles % kXcds;
    const uint32_t fj = full * (uint32_t)nchunks;
    if (j < fj) {
      const uint32_t t = by_chunks(j);
      return TileItem{(int)(xcd + kXcds * t), (int)(j - t * (uint32_t)nchunks)};
    }
    if (rem == 0) return TileItem{ntiles, 0};  // no work
    const uint32_t rounds = ((uint32_t)nchunks + kXcds - 1) / kXcds;  // chunks per strand, the last round partial
    const uint32_t s0 = xcd * rem;                                    // first strand of this XCD
    const uint32_t ta = s0 / kXcds;                                   // its first leftover tile
    const uint32_t na = ((ta + 1) * kXcds < s0 + rem ? (ta + 1) * kXcds : s0 + rem) - s0;  // strands of tile ta
    uint32_t i = j - fj;
    uint32_t t = ta, s = s0 % kXcds, n = na;
    if (i >= rounds * na) {  // strands 0 .. rem - na - 1 of the next leftover tile
      i -= rounds * na;
      t = ta + 1;
      s = 0;
      n = rem - na;
      if (n == 0) return TileItem{ntiles, 0};  // no work
    }
    const uint32_t r = div_small(i, n);
    const uint32_t c = r * kXcds + s + (i - r * n);
    if (c >= (uint32_t)nchunks) return TileItem{ntiles, 0};  // no work: past a strand's end
    return TileItem{(int)(kXcds * full + t), (int)c};
  }
};

// ---- column maps of the 32-column tiles ----
// Tile t, lane q (one 16-byte chunk of 4 columns) of a tile row holds chunk
// tile_col(m, t, q) of the row-major table (-1: padding).
//   plain  (half4 == 0): chunks tch*t .. tch*t + tch-1.
//   paired (half4 > 0):  for t < t1, chunks 4t .. 4t+3 of the first half
//     (lanes 0-3) and the same chunks of the second half (lanes 4-7), where a
//     half is half4 chunks; tiles t >= t1 hold the chunks after both halves
//     (the PSQT columns), 8 per tile.  Columns j and j + L1/2 of a row, which
//     the post-FT epilogue multiplies together, then sit in lanes q and q ^ 4.
struct ColMap {
  int half4;  // chunks per half (0: plain map)
  int t1;     // paired tiles
  int cols4;  // chunks per row
  int tch;    // plain map: chunks per tile row (8: 32 columns, 4: 16 columns)
};
SFT_HD inline int tile_col(const ColMap &m, int t, int q) {
  if (m.half4 == 0) {
    const int c = m.tch * t + q;
    return (q < m.tch && c < m.cols4) ? c : -1;
  }
  if (t < m.t1) {
    const int j = 4 * t + (q & 3);
    return j < m.half4 ? j + (q >> 2) * m.half4 : -1;
  }
  const int c = 2 * m.half4 + 8 * (t - m.t1) + q;
  return c < m.cols4 ? c : -1;
}
// Inverse: tile and lane of chunk c.
SFT_HD inline void tile_of_col(const ColMap &m, int c, int &t, int &q) {
  if (m.half4 == 0) {
    t = c / m.tch;
    q = c % m.tch;
  } else if (c < 2 * m.half4) {
    const int h = c >= m.half4 ? 1 : 0;
    const int j = c - h * m.half4;
    t = j >> 2;
    q = (j & 3) + 4 * h;
  } else {
    const int k = c - 2 * m.half4;
    t = m.t1 + (k >> 3);
    q = k & 7;
  }
}
SFT_HD inline ColMap plain_map(int cols4, int tch = 8) { return ColMap{0, 0, cols4, tch}; }
SFT_HD inline ColMap paired_map(int cols4, int half4) { return ColMap{half4, (half4 + 3) / 4, cols4, 8}; }
SFT_HD inline int map_tiles(const ColMap &m) {
  return m.half4 == 0 ? (m.cols4 + m.tch - 1) / m.tch : m.t1 + (m.cols4 - 2 * m.half4 + 7) / 8;
}

// ---- long segments of the sorted backward ----
// Whether segment [s0, s1) of the sorted slots is long depends on its bounds
// alone, so the per-feature gathers (which skip long segments) and the segment
// pass (which lists them) agree: it is long when it contains two consecutive
// multiples of `period` ("samples") of the sorted slot index.  Every segment
// of 2 period slots or more is long, none of period slots or fewer.
SFT_HD inline int64_t long_first_sample(int64_t s0, int period) { return (s0 + period - 1) / period * period; }
SFT_HD inline bool long_segment(int64_t s0, int64_t s1, int period) { return long_first_sample(s0, period) + period < s1; }
// The segment pass lists a long segment once, at its first sample i:
// keys[i + period] == keys[i] != keys[i - period] (keys: the M sorted keys).
SFT_HD inline bool long_listed_at(const unsigned *keys, int64_t M, int64_t i, int period) {
  return i % period == 0 && i + period < M && keys[i + period] == keys[i] && (i < period || keys[i - period] != keys[i]);
}

}  // namespace sft
