// Launch rules: which kernel a call takes and in which order a grid takes its
// blocks, from the sizes, the mask and the number of compute units alone. Plain
// C++ without HIP, so that the rules can be compiled and checked on the host.
// Figures in the comments are from one MI355X (256 CUs).
#pragma once

#include <initializer_list>

namespace fhog {

// Query i sees key j iff j <= i + coff (causal), or always. coff is 0 (top-left)
// or nk - nq (bottom-right).
struct Mask {
  bool causal;
  int nq, nk, coff;
};

// The sum over blocks of `rows` rows of what a block sees on the other side:
// key-tiled, the queries from its first key's diagonal on; query-tiled, the keys up
// to its last row's diagonal. Times `rows` that is the pairs the blocks cover, masked
// ones included.
inline long blocks_see(Mask m, int rows, bool key_tiled) {
  const long n = key_tiled ? m.nk : m.nq, other = key_tiled ? m.nq : m.nk, nb = (n + rows - 1) / rows;
  if (!m.causal) return nb * other;
  // block i (from the last key, or from the first query) sees clamp(a + i rows, 0, other)
  const long a = key_tiled ? other + m.coff - (nb - 1) * rows : rows + (long)m.coff;
  auto blocks_below = [&](long x) {  // how many blocks have a + i rows < x
    const long c = x > a ? (x - a + rows - 1) / rows : 0;
    return c < nb ? c : nb;
  };
  const long lo = blocks_below(1), hi = blocks_below(other);
  const long mid = hi > lo ? hi - lo : 0;
  return mid * a + rows * (mid * (lo + hi - 1) / 2) + (nb - (hi > lo ? hi : lo)) * other;
}

// How much of a causal problem is a rectangle that the diagonal does not touch: the
// queries past the last key (top-left, nq > nk) or the keys before the first
// diagonal (bottom-right, nk > nq). Blocks differ in length only in the rest, so the
// larger this part, the more a causal grid behaves like one without a mask. True
// where it is at most 1 / parts of the shorter side.
inline bool near_square(Mask m, int parts) {
  const long coff = m.coff, over = m.nq - m.nk + coff;
  const long rect = over > coff ? over : coff, side = m.nq < m.nk ? m.nq : m.nk;
  return m.causal && parts * rect <= side;
}

// The chunk for grid_slot. A grid of at most 8 rounds of resident
// workgroups keeps the rank-major order, whose last round holds the blocks
// with the least work; a longer grid takes about one round per chunk (at
// least 8 pairs, a multiple of 8), so that the streamed tiles of the pairs
// in flight stay in L2 instead of being fetched again by every block.
inline int grid_chunk(int npairs, int nranks, int resident) {
  if (resident <= 0 || (long)npairs * nranks <= 8L * resident) return npairs;
  const int c = resident / nranks / 8 * 8;
  return c < 8 ? 8 : (c < npairs ? c : npairs);
}

// First rank that runs backwards (block nb - 1 - (rank - fold)) in a grid of nb
// causal blocks, longest first, per (batch, head) pair. A grid of one to two
// workgroups per CU runs as one round in which workgroups i and i + (number of
// CUs) share a CU: the second of them take their ranks backwards, so that the
// shortest blocks sit beside the longest. nb: none does.
inline int fold_rank(bool causal, int nb, int npairs, int cus) {
  const long grid = (long)nb * npairs;
  return causal && cus > 0 && grid > cus && grid <= 2L * cus ? (cus + npairs - 1) / npairs : nb;
}

// The `pairs` argument of block_pair for a grid of nb causal blocks per
// (batch, head) pair. Mirror pairs halve the number of workgroups and are taken
// only where the paired grid fills whole rounds of the resident ones; elsewhere
// the unpaired blocks, longest first, balance better (stage 2, us, paired /
// unpaired: paired grids of 0.56 rounds, B3 N2048 H12, 125 / 96; 0.75, B1 N8192 H12,
// 442 / 387; 0.88, B4 N2048 H14, 145 / 144; 1.06, B2 N4096 H17, 411 / 314; 1.5, B16 N1024
// H12, 132 / 122; 2.25, B24 N1024 H12, 216 / 194). At two workgroups per CU that is
// - one round, skewed if nb allows (B4 N2048 H16 138 / 148, B1 N16384 H8 944 / 1021), or
//   15/16 of one near a square (B2 N4096 H15 274 / 282, B4 N2048 H15 150 / 153; but 1200
//   queries of 2500 keys bottom-right B7 H7 143 / 132);
// - more rounds of few blocks per pair. What decides is which of the two orders is
//   chunked (grid_chunk, over 8 rounds), so that a pair's blocks run close together.
//   Neither (up to 8 rounds of single blocks): fewer than 8 (nb = 2, B128 N256 H16 204 /
//   216; 4, B64 N512 H8 122 / 125; 5, B8 N640 H64 173 / 175; but 2, B64 N256 H16 98 / 95; 8,
//   B16 N1024 H16 180 / 174; 16, B8 N2048 H16 302 / 290). The single blocks only: fewer than 4
//   (2, B192 N256 H16 292 / 300; 3, B96 N384 H16 249 / 254; but 4, B128 N512 H12 364 / 352, B96
//   N512 H16 383 / 369; 6, B64 N768 H16 465 / 442; 16, B32 N2048 H16 1304 / 1190; 256, B1
//   N32768 H8 3795 / 3720). Both: fewer than 16 (2, B384 N256 H16 565 / 580; 3, B192 N384 H16
//   461 / 487; 4, B160 N512 H16 585 / 595; 8, B96 N1024 H16 1051 / 1067; 12, B64 N1536 H16
//   1427 / 1447; but 14, B64 N1792 H16 1865 / 1845; 16, B64 N2048 H16 2398 / 2373). Where half
//   of the blocks or more see no query, the chunked order starts later pairs' longest blocks
//   late, and pairs, half as many, are taken in any number of rounds (512 queries of 4096 keys
//   B16 H12 101 / 113, 1024 of 2048 B32 283 / 294, 2325 of 16384 B9 H4 139 / 193; not chunked,
//   1024 of 2048 B8 H16 95 / 93);
// - one paired workgroup per CU, from 32 blocks per pair in a square (64, B1 N8192 H8
//   309 / 320, B2 N8192 H16 over 4 key heads 1230 / 1260; 32, B4 N4096 H16 over 4 key heads
//   623 / 634; but 16, B4 N2048 H8 92.6 / 90.1). Equal blocks run better two to a CU (B2 H8,
//   4352 queries of 4096 keys 182 / 180, 5120 236 / 221, 8192 452 / 383, 2048 of 4096
//   bottom-right 159 / 124). The gain does not end at equality below (64, B1 N8192 H7 316 /
//   332, H6 304 / 315), where the single blocks are kept all the same.
// At one workgroup per CU pairs are taken in any number of whole rounds; there the two
// orders are within 2 % (first backward, us, paired / unpaired: B16 N1536 H16 353 / 359,
// B24 N2048 H16 873 / 861, B32 N1536 H16 716 / 730, B32 N2048 H16 1197 / 1184, B48 N2048 H16
// 1692 / 1719).
inline int block_pairing(Mask m, int nb, int npairs, int resident, int waves) {
  const long paired = (long)((nb + 1) / 2) * npairs, single = (long)nb * npairs;
  if (!m.causal || resident <= 0) return 0;
  if (waves == 2 && nb >= 32 && single == resident && 2 * paired == resident) return near_square(m, 32);
  if (single <= resident) return 0;
  if (waves == 2 && paired < resident) return near_square(m, 4) && 16 * paired >= 15L * resident;
  if (single > 8L * resident && m.nk >= 2 * (m.nq + (long)m.coff)) return 1;
  if (paired % resident != 0) return 0;
  if (waves != 2) return 1;
  if (paired == resident) return nb % 4 == 0 ? 2 : 1;
  const bool chunked = single > 8L * resident, chunked_pairs = paired > 8L * resident;
  return nb < (chunked_pairs ? 16 : chunked ? 4 : 8);
}

// What the busiest CU holds when a query-tiled grid of two workgroups per CU is
// folded (fold_rank: the longest block beside the shortest), in percent of the longest
// block: 100 in a square, up to 200 the longer the rectangle.
inline int folded_percent(Mask m) {
  if (!m.causal) return 200;
  if (m.coff > 0) return (int)(100 * (m.nk + (long)m.coff) / m.nk);  // bottom-right, nk > nq: nk and coff
  if (m.coff < 0 || m.nq <= m.nk) return 100;
  return m.nq >= 2L * m.nk ? 200 : (int)(100L * m.nq / m.nk);
}

// The forward: fwd_pair_kernel (two waves per 32 queries, 64-query workgroups) serves
// 2-byte types at D = 256, and fp32 on grids that do not fill the chip; fp32's two
// kernels give the same bits. Up to one workgroup per CU it halves the chain of a
// block; beyond, it pays where short causal blocks share a CU with long ones (us, fwd /
// pair; fp32 H8):
// - two per CU, unless two nearly full blocks meet (D = 64, N2048 B2 142 / 99; 1024
//   queries of 2048 keys bottom-right (150 %) B4 144 / 127; but 512 of 4096 bottom-right
//   (187 %) B8 285 / 296, 2048 of 1024 (200 %) B4 H4 74.5 / 81.3; D = 128, 512 of 4096 (187 %)
//   B8 552 / 531; but 2048 of 1024 (200 %) B4 H4 143 / 145; non-causal D = 64 N2048 144 / 157);
// - three near a square (D = 64, 1536 queries of 1024 keys B4 102 / 96; D = 128, N2048 B3
//   273 / 237, 1280 of 1024 B4 143 / 126; but 1536 of 1024 B4 164 / 169);
// - four in a square at D = 64 (N2048 B4 196 / 165, 1024 queries of 1152 keys B8 118 / 110; but
//   of 1280 134 / 139; B4 H16, eight per CU, 287 / 312; D = 128 B4 300 / 309).
inline bool fwd_pair_rule(Mask m, int npairs, int head_dim, int cus) {
  const long grid = (long)((m.nq + 63) / 64) * npairs;
  if (grid <= cus) return true;
  if (grid <= 2L * cus && folded_percent(m) <= (head_dim == 64 ? 175 : 190)) return true;
  if (grid <= 3L * cus && near_square(m, head_dim == 64 ? 2 : 4)) return true;
  return grid <= 4L * cus && head_dim == 64 && near_square(m, 8);
}

// The first backward for 2-byte types at D = 64 has several kernels for each
// half of its work, all giving the same bits: dK/dV in bwd_k_kernel
// (fhog_bwd.hip), in bwd_k64_kernel (fhog_bwd_k64.hip: 64 keys per wave at one wave
// per SIMD, generated sweep) or in bwd_pair_kernel (fhog_bwd_pair.h: two waves per
// 32 keys), dQ in bwd_q_kernel (fhog_bwd.hip), in bwd_q64_kernel (fhog_bwd_q64.hip,
// 64 queries per wave) or in bwd_qpair_kernel (fhog_bwd_qpair.hip: two waves per 32
// queries). First backward, us, at D = 64 bf16 unless named:
//
// The one-wave kernels (k64, q64) are the fastest per tile, but run one 256-row
// block per CU at a time and gain nothing when a CU is left alone. They are taken
// when their blocks cover little more than 128-row ones, in padding and, causal,
// past the diagonal: up to 6 % more for dQ (8 % where queries outnumber the keys of a
// top-left mask: 1024 of 512 B32 H8 137 / 144, H16 270 / 276, B64 H16 547 / 543; but 512 of
// 1024 bottom-right B64 H12 416 / 409), 10 % for dK/dV (first backward, us, causal
// bf16, one-wave / compiled for dQ: 6 % more, B8 N2048 H16 280 / 297 with both halves;
// 8 %, B8 N4736 H12 977 / 977; 11 %, B8 N3200 H12 506 / 503; 16 %, B32 N2117 H16 fp16 1446 /
// 1386; 23 %, B24 N1300 H12 348 / 319; 24 %, B32 N1408 H16 681 / 633; for dK/dV: 4 %, B8
// N3200 H12 472 / 492; 6 %, B32 N2117 H16 fp16 1324 / 1369; 7 %, B20 N1700 H12 413 / 421;
// 9 %, B32 N1408 H16 624 / 629, B24 N1300 H12 320 / 316; 11 %, B64 N1030 H12 616 / 609;
// rectangles: 8 %, 1280 queries of 1024 keys B32 H12 364 / 377; 4 %, 2048 of 1024 626 /
// 690); and when their
// grid fills whole rounds of the resident workgroups, or at least six (at B8 N2048
// H12 causal, 1.5 rounds, q64 took 258 against 241). A causal dK/dV needs no whole
// rounds: its key blocks, longest first, even out (first backward, compiled / k64:
// 1.1 rounds, B3 N2048 H12, 108 / 105; 1.5, B2 N4096 H12, 216 / 208, B1 N8192 H12, 405 /
// 387; 1.75, B7 N4096 H16 over 4 key heads, 958 / 869; 4.1, B11 N2048 H12, 326 / 320).
//
// The pair kernels do more LDS work per tile but take half the time per tile of
// a wave, and their 64-row blocks spread a small grid over twice as many CUs and
// waste less of a short causal sequence's diagonal. dK/dV takes its pair kernel
// up to three workgroups per CU, two for long rectangles (768 workgroups, k64 / pair:
// 3072 queries of 2048 keys B2 H12 126 / 124, 8192 of 2048 349 / 380, 4096 of 256 B12 H16 260
// / 284, 1024 of 4096 bottom-right B1 106 / 111), and on fuller grids for causal problems
// of up to 1024 keys whose diagonal shows: where 128-key blocks cover 6 % more than 64-key ones
// (others / pair: causal B1 N1024 H12 (192 workgroups) 52.4 / 45.0, B1 N4096 H12
// (768) 184 / 163, B2 N4096 H16 over 4 key heads (512) 523 / 446, B128 N512 H12
// 448 / 417, B24 N1024 H12 219 / 213, B32 N1024 H16 399 / 403, B4 N2048 H16 136 /
// 151; rectangles: 7 % more, 400 queries of 600 keys bottom-right B64 H12 fp16 250 / 244,
// 128 of 512 B64 113 / 107; 6 %, 768 queries of 512 keys B64 305 / 313; 5 %, 768 of 1024
// bottom-right B32 250 / 254; 4 %, 1280 of 1024 364 / 385, 1024 of 512 B32 H16 269 / 284; 2 %,
// 8192 of 1024 B8 H16 923 / 1100; non-causal B1 N2048 H16 (512) 95.2 / 92.9, B2 N2048
// H12 (768) 120 / 117, B8 N1000 H12 fp16 (1536) 122.8 / 124.0). dQ gains less and takes its pair kernel,
// at D = 64 and 128, up to one workgroup per CU (B1 N512 H12 27.0 / 26.1, B1
// N2048 H8 D128 non-causal 119 / 109; B2 N1000 H12 fp16, 384 workgroups, 51.2 /
// 55.7), at D = 64 up to 2048 keys: it starts 1 us earlier and takes longer per tile (B1 N1024
// H12 45.5 / 44.9, N2048 H8 81.7 / 81.8, N4096 H4 154 / 155, N8192 H2 298 / 309, 1024 queries of 7168
// keys bottom-right B6 H1 147 / 158; D128 B6 H1 253 / 232). Short causal sequences gain
// nothing on fuller grids (compiled / pair: B128 N256 H12 168 / 166, B128 N384 H12 292 / 296, B32 N512 H12 101 / 99, B128 N512 H12 408 / 423, over
// 4 key heads 442 / 467), and a chunk of queries against more keys loses (512 queries
// of 1024 keys bottom-right B64 H12 409 / 448, of 4096 B32 877 / 1036).
inline bool one_wave_grid(int workgroups, int resident) {
  return resident > 0 && workgroups > 0 && (workgroups % resident == 0 || workgroups >= 6 * resident);
}
// Whether 256-row blocks cover at most `percent` of what 128-row ones do. Blocks that see
// nothing (keys past the last query, queries before the first key) cost their launch
// and a store of zeros each, half as many with 256 rows; with any of them a grid counts
// as the square of all its rows (first backward, us, k64 / compiled dK/dV: 512 queries of
// 4096 keys B16 H12 85.4 / 107, of 2048 B32 135 / 144; q64 / compiled dQ: 4096 queries of 512
// keys bottom-right B16 128 / 148, 2048 of 512 B32 168 / 180).
inline bool one_wave_cover(Mask m, bool key_tiled, int percent) {
  const bool empty = m.causal && (key_tiled ? m.nk > m.nq + (long)m.coff : m.coff < 0);
  if (empty) m.nq = m.nk = key_tiled ? m.nk : m.nq, m.coff = 0;
  return 100 * 2 * blocks_see(m, 256, key_tiled) <= percent * blocks_see(m, 128, key_tiled);
}
// Whether the whole rounds of q64 or k64 are there (n: the blocked side).
inline bool one_wave_rounds(Mask m, int n, int npairs, int cus) {
  const int nb = (int)(((long)n + 255) / 256);
  const bool mirrored = m.causal && (long)nb * npairs > cus;
  return one_wave_grid((mirrored ? (nb + 1) / 2 : nb) * npairs, cus);
}
inline bool bwd_q64_rule(Mask m, int npairs, int cus) {
  const int percent = m.causal && m.coff == 0 && !near_square(m, 4) ? 108 : 106;
  return one_wave_cover(m, false, percent) && one_wave_rounds(m, m.nq, npairs, cus);
}
inline bool bwd_k64_rule(Mask m, int npairs, int cus) {
  return one_wave_cover(m, true, 110) && (m.causal || one_wave_rounds(m, m.nk, npairs, cus));
}
inline bool bwd_pair_rule(Mask m, int npairs, int cus) {
  if ((long)((m.nk + 63) / 64) * npairs <= (m.causal && !near_square(m, 2) ? 2L : 3L) * cus) return true;
  if (!m.causal || m.nk > 1024) return false;
  return 1000 * 2 * blocks_see(m, 128, true) >= (near_square(m, 16) ? 1058 : 1065) * blocks_see(m, 64, true);
}
inline bool bwd_qpair_rule(Mask m, int npairs, int head_dim, int cus) {
  if ((long)((m.nq + 63) / 64) * npairs > cus) return false;
  const long last = m.causal && m.nq + (long)m.coff < m.nk ? m.nq + (long)m.coff : m.nk;  // keys of the last query
  return head_dim > 64 || last <= 2048;
}

// Waves per SIMD of bwd_pair_kernel. Three workgroups per CU at 256-byte rows (168
// registers): for fp32 always (D = 64 B4 N2048 H16 1031 -> 1013 us, B2 N2048 H8
// equal), for 2-byte D = 128 once the grid is long (two / three: 359 / 392 us at B2 N2048 H32 over 8 key
// heads, 512 workgroups; 300 / 287 at B4 N2048 H16, 2048; 2040 / 1956 at B2
// N8192 H16, 4096). 2-byte D = 64 likewise with four (117 registers; first
// backward, two / four: causal B1 N4096 H12, 768 workgroups, 163 / 166, B2 N2048
// H16, 1024, 105 / 99, B128 N512 H12 484 / 417; non-causal B2 N2048 H12, 768,
// 146 / 117; 768 workgroups of rectangles: 2560 queries of 2048 keys B2 H12 113 / 105,
// 2304 of 2048 98.0 / 97.1, 4096 of 2048 219 / 181, 1024 of 2048 bottom-right 79.5 / 70.0).
inline int bwd_pair_waves(Mask m, int npairs, int head_dim, int bytes, int cus) {
  const long grid = (long)((m.nk + 63) / 64) * npairs;
  if (bytes == 4 && head_dim == 64) return 3;
  if (bytes == 2 && head_dim == 128 && grid > 4L * cus) return 3;
  if (bytes == 2 && head_dim == 64 && grid > (near_square(m, 16) ? 3L : 2L) * cus) return 4;
  return 2;
}

// Stage 1 for 2-byte types at D = 64 runs the kernel with 32 queries per wave at one
// wave per SIMD, a hand-scheduled sweep, a persistent grid and 128-query blocks
// (fhog_bwdbwd_q32.hip) but for short causal problems, where the fused kernel's
// 64-query blocks (16 queries per wave, two waves per SIMD) take half as long and
// cover less of what the mask or the last row cuts off. Both give the same results
// to rounding, so the choice looks at the lengths only, never at how many sequences
// there are: up to 512 on both sides, where 128-query blocks cover 12 % more than
// 64-query ones, or 15 % where the diagonal is not most of the problem.
// Stage 1, us, q32 / fused, H12 bf16: 36 % more (N448) B128 410 / 355; 28 % (400
// queries, 500 keys bottom-right, H8) B16 45.6 / 40.4; 20 % (N256) B256 322 / 314; 14 %
// (N384) B64 148 / 147; but 11 % (N512) B128 427 / 433, B32 103 / 105, though B16 55.6 /
// 53.8 and B1 20.3 / 18.7. Rectangles: 14 % (256 queries, 128 keys) B128 125 / 132; 8 %
// (256 queries, 512 keys bottom-right) B64 140 / 146; 7 % (512 queries, 128 keys) B128
// 239 / 258. Non-causal N512 B16 fp16 74.6 / 85.7; B4 N2048 H16 causal 177 / 190.
inline bool stage1_fused_rule(Mask m) {
  if (!m.causal || m.nq > 512 || m.nk > 512) return false;
  return 100 * 2 * blocks_see(m, 128, false) >= (near_square(m, 16) ? 112 : 115) * blocks_see(m, 64, false);
}

// Pairs of waves (32 queries each) per workgroup of the D = 128 stage 1,
// fhog_bwdbwd_fused_pair.hip: two (two workgroups per CU) while the chip is not full of
// them; where 128-query blocks cover 30 % more than 64-query ones; and where four pairs (one
// workgroup per CU) make two rounds and less than a third of one. Four otherwise.
// Stage 1, us, two / four, H16 bf16: small grids, causal B1 N1024 H8 (128 workgroups of 64
// queries) 66 / 76, non-causal B1 N2048 H8 (256) 127 / 141; cover 100 % more, N64 B64 42 /
// 60; 46 %, N300 B16 H12 fp16 58 / 73; 33 %, N128 B64 98 / 102; 58 %, 1288 queries of 169 keys
// bottom-right B84 H8 444 / 480; rounds, 327 queries of 100 keys B23 H8 (2.16) 52 / 62; but 20 %,
// N256 B64 257 / 254; 14 %, N384 B32 204 / 208; 11 %, N512 B32 335 / 320, B128 H12 897 / 923; N1024
// B16 505 / 517; B2 N2048 H32 389 / 372; non-causal B4 N2048 734 / 679, N256 B64 352 / 296; 256 of
// 1024 bottom-right B64 H8 495 / 403.
inline int stage1_pairs_rule(Mask m, int npairs, int cus) {
  const long two = (long)((m.nq + 63) / 64) * npairs, four = (long)((m.nq + 127) / 128) * npairs;
  if (two <= 2L * cus || 10 * 2 * blocks_see(m, 128, false) >= 13 * blocks_see(m, 64, false)) return 2;
  return four > 2L * cus && 3 * four < 7L * cus ? 2 : 4;
}

// Stage 1 for fp32 runs bwdbwd_q_kernel (fhog_bwdbwd.hip, one wave per 32 queries) on grids
// that fill the chip and bwdbwd_qpair_kernel (fhog_bwdbwd_qpair.hip, two waves per
// 32 queries, half the time per block and twice the workgroups) on smaller ones;
// both give the same bits. The line is one of the latter's workgroups per CU, two
// where folded blocks even out (stage 1, us, q / qpair: causal D = 64 N2048 H8 B2 (512
// workgroups) 887 / 631, B3 (768) 890 / 840-885, B4 (1024) 970 / 1093; 512 of them, 768
// queries of 1024 keys bottom-right (125 %) B4 H10 454 / 434, 1280 of 1024 (125 %) B4 H6 455 / 433,
// 1024 of 2048 bottom-right (150 %) B4 H8 902 / 828, but 1536 of 1024 (150 %) B4 H5 456 / 458, 2048 of
// 1024 (200 %) B4 H4 456 / 533, 512 of 4096 bottom-right (187 %) B8 H8 1798 / 2002; non-causal B1
// (256) 902 / 626, B2 (512) 910 / 1021; D = 128 causal B2 (512) 1620 / 1296, B4 (1024) 1783 /
// 2538, 1280 of 1024 (125 %) B4 H6 833 / 804, 1024 of 2048 bottom-right (150 %) B4 H8 1650 / 1863, 512
// of 4096 (187 %) B8 H8 3324 / 4645, non-causal B1 (256) 1647 / 1255).
inline bool stage1_qpair_rule(Mask m, int npairs, int cus) {
  return (long)((m.nq + 63) / 64) * npairs <= (folded_percent(m) <= 140 ? 2L : 1L) * cus;
}

// Stage 2 runs bwdbwd_pair_kernel (fhog_bwdbwd_pair.hip, two waves per 32 keys)
// but for 2-byte types at D = 64 on grids that fill the chip, where
// bwdbwd_k_kernel's one wave per 32 keys is faster; both give the same bits.
// The pair kernel's grid has twice the workgroups of half the work each, and
// is taken while it has at most three of them per CU when causal and near a square,
// two on other causal rectangles, whose blocks are nearly equal, and one without a
// mask (stage 2, us, k / pair: causal B1 N512 H12 24.8 / 20.2, B1 N2048 H12 (384
// workgroups) 78.4 / 69.7, B2 N2048 H12 (768) 85.2 / 74.8, B2 N4096 H16 over 4 key heads
// (512) 575 / 511, but B2 N2048 H16 (1024) 93.3 / 95.8 and B1 N8192 H12 (1536) 452 / 497;
// rectangles with 768: 2304 queries of 2048 keys 95.8 / 86.0, 2560 107 / 102, 1536 of 2048
// bottom-right 67.1 / 66.5, but 3072 of 2048 129 / 137, 4096 175 / 208, 6144 280 / 352, 1024 of
// 2048 bottom-right 54.0 / 62.9, 1024 of 8192 64.7 / 75.2; with 640: 4096 of 2048 164 / 185;
// with 512: 4096 of 2048 152 / 141, 8192 295 / 286, 1024 of 2048 bottom-right 43.9 / 43.6, of
// 4096 43.4 / 44.3; with 384: 8192 of 2048 295 / 277; non-causal B1 N300 over one key head
// 51.9 / 44.2, N2048 H8 (256) 78.3 / 66.7, but H12 (384) 79.6 / 82.4, B2 N1000 H12 fp16 43.9 /
// 48.0).
inline bool stage2_pair_rule(Mask m, int npairs, int cus) {
  return (long)((m.nk + 63) / 64) * npairs <= (!m.causal ? 1L : near_square(m, 4) ? 3L : 2L) * cus;
}

// Keys that the busiest workgroup of a causal grid of bwdbwd_q32_kernel sweeps, in each of
// its two block lists: `cus` workgroups (or one per item) walk the list in strides of their
// number, see fhog_bwdbwd_q32.hip.
struct Q32Load {
  double folded, dealt;
};
inline Q32Load q32_load(Mask m, int npairs, int cus) {
  constexpr int kRows = 128;
  const long nqb = ((long)m.nq + kRows - 1) / kRows, npr = (nqb + 1) / 2;
  auto keys = [&](long qb) {
    const long e = (qb + 1) * kRows + m.coff;
    return (double)(e < 0 ? 0 : e < m.nk ? e : m.nk);
  };
  auto most = [](double a, double b) { return a > b ? a : b; };
  // Item r: the r-th block from either end. Workgroup w gets items w, w + cus, ..., so the
  // items r of each pair come round with period npr / gcd(cus, npr). A middle item is one
  // block, so that three items of a square (five blocks) even out where four do not. With
  // very many items the mean serves.
  auto item = [&](long r) { return keys(nqb - 1 - r) + (2 * r + 1 == nqb ? 0.0 : keys(r)); };
  const long items = npairs * npr, rounds = (items + cus - 1) / cus;
  double folded = 0;
  if (npr * rounds > 4096) {
    folded = (double)rounds * blocks_see(m, kRows, false) / (double)npr;
  } else {
    for (long w = 0; w < npr && w < items && w < cus; ++w) {
      double sum = 0;
      for (long i = w; i < items; i += cus) sum += item(i % npr);
      folded = most(folded, sum);
    }
  }
  // Blocks longest first, every other round in reverse: the busiest workgroup is the first
  // or the last of the rounds, or the last one that gets a block of the final round.
  const long blocks = npairs * nqb, full = blocks / cus, rest = blocks % cus;
  const long mean = 64;  // rounds after which the share is near enough
  double dealt = (double)npairs * blocks_see(m, kRows, false) / cus;
  if (full < mean) {
    const long last = full & 1 ? cus - rest : rest - 1;
    for (const long w : {0L, cus - 1L, rest > 0 ? last : 0L}) {
      double sum = 0;
      for (long k = 0;; ++k) {
        const long i = k * cus + (k & 1 ? cus - 1 - w : w);
        if (i >= blocks) break;
        sum += keys(nqb - 1 - i / npairs);
      }
      dealt = most(dealt, sum);
    }
  }
  return Q32Load{folded, dealt};
}

// Whether a causal grid deals its blocks one by one instead of folding them
// (bwdbwd_q32_kernel; both give the same bits): when every block can have a CU of
// its own, or when the busiest workgroup of the folded list has so much more to sweep than
// that of the dealt one: 7 % near a square, 15 % on rectangles, where dealing gives up more
// of the tiles that a pair's blocks share in L2. Stage 1, us, folded / dealt: one
// round of blocks, B1 N512 H12 28.6 / 20.5, B1 N1024 H12 41.8 / 33.7, B1 N2048 H12 67.5 / 62.0;
// 12 % more in the folded list, B4 N1024 H12 46.0 / 44.6; 10 %, B24 N1024 H12 258 / 248; 20 %,
// B1 N8192 H12 650 / 518; 31 %, B8 N1500 H12 fp16 218 / 176; 62 %, B3 N2048 H12 155 / 115; but
// 6 %, B2 N2048 H12 77.0 / 78.4; 3 %, B1 N4096 H12 141 / 149 (fewer CUs run faster); 1 %, B40
// N1024 H12 414 / 422; none, B32 N1024 H12 324 / 332, B4 N2048 H16 182 / 183.
// Rectangles, H12: 34 %, 1024 queries of 8192 keys bottom-right B7 1105 / 870, 600 of 3000
// B12 378 / 312; 23 %, 4096 of 1024 B6 371 / 329; 21 %, 900 of 2000 bottom-right B13 371 / 328;
// but 12 %, 4096 of 1024 B4 H16 300 / 288; 10 %, 1024 of 4096 bottom-right B28 1578 / 1631; 7 %,
// B4 H10 209 / 220; 2 %, 1024 of 8192 B4 462 / 475; none, 1024 of 4096 B32 1618 / 1839. With rows that
// see no key: 76 %, 2048 of 1024 bottom-right B24 330 / 273; 6 %, 1664 of 768 B35 H16 354 / 374.
inline bool q32_deal_rule(Mask m, int npairs, int cus) {
  const long blocks = npairs * (((long)m.nq + 127) / 128);
  if (!m.causal) return false;
  if (blocks <= cus) return true;
  if (cus <= 0) return false;
  const Q32Load load = q32_load(m, npairs, cus);
  return load.folded > (near_square(m, 4) ? 1.07 : 1.15) * load.dealt;
}

}  // namespace fhog
