// Launch rules that depend on sizes alone: grids, the cells up to which pass G
// and pass F run four lanes per cell, and the sizes of the buffers that those
// launches write.  No HIP in here, so that they can be checked on the host.
#pragma once
#include <algorithm>
#include <cstdint>

namespace fkx {

constexpr int kBlock = 256;
constexpr int kXcd = 8;  // XCDs of the device

inline unsigned grid_for(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }
// blocks of `cells` cells, a multiple of 8: the XCD-remapped kernels
inline unsigned grid_blocks(int64_t nc, int cells) {
  return (unsigned)(((nc + cells - 1) / cells + kXcd - 1) / kXcd * kXcd);
}
inline unsigned grid_xcd(int64_t nc) { return grid_blocks(nc, kBlock); }
inline unsigned grid_quad(int64_t nc) { return grid_blocks(nc, 16); }  // one wave of 16 quads a block

// Cells up to which pass G and pass F run four lanes per cell (pass_g_q,
// pass_f_q) rather than one with the LDS paths.  What the quads win is waves
// in flight and shorter chains; what they lose is the own-cell work on four
// lanes and, with records of half the size (FP32), pass F's LDS reuse.  us,
// quads / one lane, on either side of the lines:
//   pass G  FP64 12 / 13 at 55k cells (single-phase), 16 / 19 at 48k and 23 / 21 at
//           83k (two-phase); FP32 10 / 11 at 48k, 16 / 13 at 94k; 6 slots FP64
//           21 / 23 at 27k, 33 / 26 at 55k; FP32 9 / 12 at 8k, 13 / 12 at 27k
//   pass F  FP64 at every size (three waves per SIMD against two): two-phase 20 /
//           29 at 83k, 733 / 773 (dt stage 689 / 772) at 3.1M, 1874 / 1997
//           (1747 / 1987) at 8M, 3816 / 4146 (3599 / 4109) at 16M; single-phase
//           1133 / 1190 (1054 / 1157) at 6.9M; 6 slots 583 / 653 at 1.3M, 2458 /
//           2760 at 5.8M; FP32 53 / 56 at 280k, 100 / 90 at 511k (two-phase),
//           51 / 59 at 511k, 178 / 160 at 1.6M (single-phase); 6 slots FP32
//           28 / 29 at 55k, 63 / 60 at 176k
//   with the relaxation (on the quad only the plain solve's residuals go in
//           parallel, without the shared divisors of one lane's) us a step:
//           surrogate FP64 115 / 120 at 48k, 261 / 263 at 162k, 345 / 352 at
//           236k, 492 / 487 at 329k; FP32 (the kernel) 21 / 21 at 48k, 28 / 23 at
//           64k; plain FP64 80 / 83 at 25k (apart above, fuse_pays); FP32 63 / 67
//           at 16k, 69 / 70 at 25k, 74 / 73 at 29k, 93 / 82 at 48k; 6 slots
//           surrogate (the kernel) FP64 24 / 31 at 27k, 34 / 33 at 47k; FP32 24 /
//           25 at 27k, 25 / 25 at 36k, 42 / 38 at 85k; plain FP64 130 / 133 at
//           27k, 170 / 161 at 36k; FP32 101 / 103 at 27k, 143 / 135 at 36k
inline int64_t quad_cells_g(bool f64, int ns) {
  if (ns == 6) return f64 ? 40000 : 20000;
  return 60000;
}
// relax: 0 none, 1 the surrogate's stage 1, 2 the plain relaxation in the kernel
inline int64_t quad_cells_f(bool f64, int ns, int neq, int relax) {
  if (relax) {
    if (ns == 6) return !f64 && relax == 2 ? 30000 : 35000;
    return f64 ? 220000 : (relax == 2 ? 25000 : 50000);
  }
  if (f64) return INT64_MAX;
  return ns == 6 ? 120000 : (neq == 5 ? 600000 : 350000);
}

// Waves of pass F with one lane per cell, blocks of `block` cells.
inline int64_t pass_f_waves(int64_t nc, int block) { return (int64_t)grid_blocks(nc, block) * (block / 64); }

// Words of the relaxation's partial counts (fk_ctx::rpart): [blocks][4] of its
// own kernels, or [waves][1 + relax] of a pass F that relaxes, at either
// precision: a context may change it after the buffer is there.
inline int64_t relax_words(int64_t nc, int ns) {
  int64_t w = (int64_t)grid_xcd(nc) * 12;  // at least pass_f_waves(nc, 128 or 256) * 3
  for (int relax = 1; relax <= 2; ++relax)
    if (nc <= std::max(quad_cells_f(false, ns, 10, relax), quad_cells_f(true, ns, 10, relax)))
      w = std::max(w, (int64_t)grid_quad(nc) * (1 + relax));
  return w;
}

// A relaxation gives a listed cell to a group of lanes (8 a reference chemical
// solve, 4 a polish) on short lists: there the chip has idle SIMDs and the chain
// of one cell sets the time; on longer ones the redundant work of a group's
// lanes does.  Every cell of the mesh listed, us, one lane / group: reference
// chemical solve 2k cells 387 / 84, 16k 395 / 147, 35k 399 / 249, 48k 400 / 316,
// 64k 409 / 404, 119k 533 / 611; as fallback of as many polishes 378 / 87, 392 /
// 147, 399 / 256, 400 / 318, 402 / 412, of thermal cells, which every lane of a
// group solves alike, 55 / 25, 396 / 120, 428 / 138, 541 / 177, 476 / 203.
// Polish from the cell state 2k 55 / 39, 16k 60 / 38, 35k 74 / 62, 48k 76 / 68,
// 119k 88 / 129; from the network's start 510 cells 34 / 22, 25k 57 / 48, 50k
// 63 / 53, 119k 73 / 80.
constexpr int64_t kChemGroup = 65536, kPolishGroup = 49152;

// Blocks of a kernel over a list of up to nc cells: one lane a cell, up to 1024
// blocks, but `lanes` lanes a cell as long as that makes no more than 512.  With
// blocks for one lane alone, groups of 8 took eight rounds of a full list and
// lost to one lane (16k chemical cells 475 us, their polish 94); more than 512
// gain nothing on full lists and cost each step with short ones (fallback of
// 373k hexahedra with 1024 blocks 1 us more than with 256, with 512 0.7).
inline unsigned list_blocks(int64_t nc, int lanes) {
  const int64_t most = std::max<int64_t>(std::min<int64_t>(grid_for(nc * lanes), 512), std::min<int64_t>(grid_for(nc), 1024));
  return (unsigned)std::max<int64_t>(1, most);
}

// Lanes to a cell of a list of n on a grid of nt lanes: a group while the list
// takes up to four rounds of the chemical solve, two of the polish.
constexpr int chem_lanes(int64_t n, int64_t nt) { return n <= kChemGroup && n * 8 <= 4 * nt ? 8 : 1; }
constexpr int polish_lanes(int64_t n, int64_t nt) { return n <= kPolishGroup && n * 4 <= 2 * nt ? 4 : 1; }

}  // namespace fkx
