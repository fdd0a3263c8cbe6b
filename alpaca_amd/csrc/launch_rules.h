// Rules that choose a kernel by the number of blocks of a launch (host code only).
// Block counts are compared with the compute units (`cus`); the times in the comments
// were measured with 256.
#pragma once

namespace alpaca {

// Flux families and arithmetic modes, as in the headers that number them.
enum : int { kRuleHllc = 0, kRuleRoe = 1 };
enum : int { kRuleExact = 0, kRuleFma = 1, kRuleMixed = 2 };

// Whether a 3D case marches (march_stage_kernel) or runs on tiles.
//
// A CU holds two slabs of a block, or two 8^3 tiles, at a time.  One slab on a CU runs one
// wavefront per SIMD, with nothing to cover its latencies, and a case takes as long with
// 128 blocks as with 4, where the tiles' time follows the blocks; so the slabs have to be
// two per CU at least.  From there both kernels spend about the same time per unit of 64 faces and
// wavefront (a slab 26, a tile 7; Roe with FMA 26.5 against 7) and the case marches where
// its slabs fill the CUs as evenly.  One step, us, tiles and marching:
//   blocks          100       128       225       256       384       400       512      1024
//   HLLC exact  379  447  388  457  733  743  778  768 1188 1155 1262 1404 1567 1524 3103 2967
//   Roe exact   448  525  466  549  878  896  946  936 1418 1393 1515 1718 1877 1848 3748 3614
//   Roe FMA     232  272  251  285  478  497  528  537  828  811  869  975 1101 1085 2172 2126
// HLLC with FMA, whose tiles of 512 threads run four wavefronts per SIMD, marches from 8
// blocks per CU only (512 blocks 913 us and 925, 2048 blocks 3567 and 3525, 2560 4480 and
// 4413).  The mixed forms keep the tiles (HLLC gains nothing; Roe's FP32 faces round
// differently where a cell's quantities pass through LDS, as other products are then
// fused).
inline bool rule_marches(int flux, int mode, long long blocks, long long cus) {
  if (mode == kRuleMixed) return false;
  long long const least = mode == kRuleExact ? cus : (flux == kRuleRoe ? cus + 1 : 8 * cus);
  if (blocks < least) return false;
  auto rounds = [cus](long long groups) { return (groups + cus - 1) / cus; };
  int const slab = mode == kRuleFma && flux == kRuleRoe ? 53 : 52, tile = 14;
  return rounds(2 * blocks) * slab <= rounds(8 * blocks) * tile;
}

// Whether a 2D case runs on pair_stage_kernel.  Four of its workgroups fill a CU, so it
// is ahead where the pairs are resident at once or nearly so but the blocks, of which a
// CU holds six, are not, and where there are many (one step, us, tiles and pairs):
//   blocks          1536      1600      2025      2560      3249      4900     16384
//   HLLC exact  180  212  225  214  276  228  322  280  370  388  510  512 1666 1644
//   Roe exact   202  239  253  240  310  252  361  324  422  440  591  591 1968 1889
//   Roe FMA     112  126  136  129  163  142  191  172  220  231  312  308 1101 1056
// The other forms, which run 4 or 5 wavefronts per SIMD, gain at many blocks only.
inline bool rule_pairs(int flux, int mode, long long blocks, long long cus) {
  bool const heavy = mode == kRuleExact || (flux == kRuleRoe && mode == kRuleFma);
  return blocks >= 32 * cus || (mode == kRuleExact && blocks >= 16 * cus) ||
         (heavy && blocks > 6 * cus && blocks <= 10 * cus);
}

// The tile configuration (of set_tuning, and 3 = 8x8 cells and 256 threads, 4 = 16x8 and 192)
// of an ensemble that was given none, from all its blocks and those of its largest class.
// 3D: 8^3 always.  2D, one step, us, configurations 0, 3 and 4:
//   blocks                160          320          512           768           900          1400
//   HLLC exact         95  62  70  136  86  90  140 125  96  149 184 132  147 223 180  197 315 233
//   Roe mixed          69  50  56   95  70  67   98  98  72  102 138 101  106 165 130  144 230 173
//   HLLC exact+mixed  100  60  58  101  69  76  104  98  87  144 129 104  147 153 117  175 214 178
//   Roe exact+mixed   104  60  62  108  73  82  111 102  94  159 138 114  162 160 126  197 234 193
// The line between 3 and 4 is that of a single case (launch_shapes.h).  Configuration 4
// holds two blocks per CU at a time, and from the third on a class waits for a second
// round, where 0 holds six; several classes fill each other's rounds.
inline int rule_ensemble_tiles(int dim, long long blocks, long long largest, long long cus) {
  if (dim == 3) return 0;
  if (4 * blocks <= 5 * cus) return 3;
  return blocks < 6 * cus && largest <= 3 * cus ? 4 : 0;
}

// Persistent workgroups per CU of an ensemble's stage kernels with a tile configuration:
// what fits a CU at once, and where a tuning gave none.
inline int rule_ensemble_default_groups(int dim, int tile_config) {
  if (dim == 3) return tile_config == 1 ? 1 : 2;
  return tile_config == 1 || tile_config == 3 ? 3 : (tile_config == 4 ? 4 : 6);
}

// Whether a class of so many blocks takes the default where a tuning gave more.  The 2D
// workgroups of 128 threads (configurations 0 and 2) are two wavefronts.  Up to four of
// them with work per CU are two wavefronts on each SIMD, unless idle workgroups are dealt
// among them, which leaves some SIMDs with three and others with one (one step, us, 6 and
// 12 per CU: 580 blocks of exact HLLC 144 and 156, 832 146 and 189, 1024 152 and 186; mixed
// 960 93 and 104).  Above, the idle ones are few (1100 blocks 191 and 191, 1400 199 and
// 193), and with four wavefronts a workgroup has one on each SIMD anyway.
inline bool rule_ensemble_fewer_groups(int dim, int tile_config, long long blocks, long long cus) {
  if (dim != 2 || (tile_config != 0 && tile_config != 2)) return false;
  return blocks * (tile_config == 2 ? 2 : 1) <= 4 * cus;
}

}  // namespace alpaca
