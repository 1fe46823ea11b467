// How the attention kernel that keeps the keys of a head in LDS (attn_fwd_16_resident.hip) deals out query rows: index
// arithmetic only, plain C++ for the kernel and for a host test.
#pragma once
#include <stdint.h>

#include "attn_walk.h"

namespace xdit {

// KV tiles (of 64 keys) that the kernel built for head_dim D holds: with the staging blocks of 12 wavefronts they
// fill 159 of the 160 KiB of LDS.
template <int D> constexpr int kResidentTiles = D == 128 ? 4 : 8;

// A workgroup's work: groups [g0, g1) of 32 query rows of (batch, head) bh.
struct ResidentPart {
  int bh, g0, g1;
};

// Workgroup w of a launch that cuts the row groups of every (batch, head) into `parts` (at most as many as there are
// groups) parts of equal size, give or take one.  False when there is nothing for it.
XDIT_HD bool resident_part(int w, int tiles_per_xcd, int total, int parts, int Sq, ResidentPart& r) {
  const int tile = xcd_tile_index(w, tiles_per_xcd);
  if (tile >= total) return false;
  const int64_t groups = (Sq + 31) / 32;
  r.bh = tile / parts;
  const int i = tile - r.bh * parts;
  r.g0 = (int)(groups * i / parts);
  r.g1 = (int)(groups * (i + 1) / parts);
  return true;
}

// Wavefronts of a workgroup, by head_dim.  Twelve where three to a SIMD leave the registers for it.
constexpr int resident_wavefronts(int head_dim) { return head_dim <= 80 ? 12 : 8; }

// Parts per (batch, head): what makes the rounds of workgroups, one to a compute unit, shortest, where a
// workgroup takes its prologue (about four KV tiles' worth: keys and queries from memory) and the groups of its
// busiest wavefront, each `nt` tiles and about two for the rows' way in and out.  Of equal costs the first candidate, which has
// the most parts: fewer wavefronts with a group each share a compute unit then (with no wavefront busier for it, fewer parts
// took 1.2 times as long in the median of 1135 timings).  In 1386 of 1405 problems no other number of parts tried was more than 4 % faster.
inline int resident_parts(int64_t bh, int Sq, int nt, int wavefronts, int cus) {
  const int64_t groups = (Sq + 31) / 32;
  int64_t best = 1;
  double best_cost = -1;
  for (int64_t rounds = 1; rounds <= 6; rounds++) {
    int64_t parts = rounds * cus / bh;
    if (parts < 1) parts = 1;
    if (parts > groups) parts = groups;
    const int64_t per_wave = ((groups + parts - 1) / parts + wavefronts - 1) / wavefronts;
    const double cost = (double)((bh * parts + cus - 1) / cus) * (4.0 + (double)per_wave * (nt + 2));
    if (best_cost < 0 || cost < best_cost) { best = parts; best_cost = cost; }
  }
  return (int)best;
}

// Estimated us of that launch, on the scale of choose_launch's estimate for the tiled launch of `tiled_rows` rows per workgroup that it
// would take the place of: rounds of workgroups, each a prologue and the average, not the busiest, number of row groups of
// its wavefronts, which share the compute unit.  Keys pay for their way into LDS only where enough groups meet them there: with
// a group or less per wavefront all of them have to land before the first product.
// The rates are the lowest at which at most 8 in 1000 problems were sent here that were more than 4 % slower for it (14000 of them, see
// resident_path).  Against tiled launches of 256 and 384 rows they are lower, as these show their prologue and
// epilogue in full, and lowest where rows are no whole half lines of 128 bytes, whose streaming stores cost those launches most.
inline double resident_us(int64_t bh, int Sq, int nt, int head_dim, int cus, int tiled_rows) {
  const int nw = resident_wavefronts(head_dim);
  const double never = 1e30;
  if (bh > (int64_t)0xffffffff / (64 * nw) - 8) return never;  // a launch holds at most 2^32 threads
  const int parts = resident_parts(bh, Sq, nt, nw, cus);
  const double rounds = (double)((bh * parts + cus - 1) / cus);
  const double per_wave = (double)((Sq + 31) / 32) / parts / nw;
  const bool many_rows = tiled_rows > 128;
  if (head_dim == 64) return many_rows ? 1.06 * rounds * (1.5 + per_wave) * (nt + 2) - 6.0 : never;
  if (head_dim < 64) return rounds * (1.5 + per_wave) * (many_rows ? (head_dim > 32 ? 0.65 : 0.75) * (nt + 4) : 1.03 * (nt + 2)) - 4.0;
  const double rate = many_rows ? (head_dim % 32 == 0 ? 1.9 : 1.35) : head_dim <= 80 ? 1.6 : head_dim <= 104 || head_dim == 128 ? 1.65 : head_dim <= 112 ? 1.87 : 1.57;
  return rate * rounds * (8.0 + (0.5 + per_wave) * nt) - 4.0;
}

// Whether the wavefronts have so many row groups (on average over the chip) that the keys pay for their way into LDS whatever the
// estimates say, which are coarse between one and two rounds of the tiled launch.  Heads with at least two workgroups each only; and not at
// head_dims 72, 80 and 96, where the estimates choose as well.  Of 23406 timed problems this sends 1248 more here than
// the estimates do: at head_dim 128 614 with 4 % less time (median), at 88 and 104 to 120 267 with 12 %, at 64 (over more than one KV tile) 263
// with 4 %, below 104 with 16 %; 4 % of them take over 2 % longer, 13 % at worst.  One group per wavefront is where the tiled launch starts a
// second round; at 88 between one and one and a half calls on power-of-two rows are up to 12 % slower (12 heads of 8192 on 256 keys).
inline bool resident_enough_groups(int64_t bh, int Sq, int nt, int head_dim, int cus, int tiled_rows) {
  if (bh > cus / 2 || (head_dim > 64 && head_dim <= 80) || head_dim == 96) return false;
  const int nw = resident_wavefronts(head_dim);
  const int64_t workgroups = bh * resident_parts(bh, Sq, nt, nw, cus);
  const double per_wave = (double)(bh * ((Sq + 31) / 32)) / (double)(workgroups > cus ? workgroups : cus) / nw;
  if (head_dim <= 64) return tiled_rows <= 128 && per_wave > (head_dim < 64 ? 3.0 : 8.0) && (head_dim < 64 || nt > 1);
  return per_wave > (head_dim == 88 ? 1.5 : 1.0);
}

}  // namespace xdit
