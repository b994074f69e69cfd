// Shares of the prefill attention's work for head dims up to 128.  Plain C++
// beside the kernels that use it, so that the arithmetic is also checked on
// the host.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define KIV_HD __host__ __device__
#else
#define KIV_HD
#endif

namespace kiv {

constexpr int kPfUnitRows = 128;  // query rows of a unit
constexpr int kPfKeys = 64;   // keys of a tile

// A unit is a block of kPfUnitRows query rows of one (b, q head); units are
// numbered heads first (unit = bh * nrb + rb) and a unit's weight is its
// tiles that any of its rows sees (every tile without a mask, the retrieved
// keys' tiles and those up to its last row's diagonal under the causal rule).
// blocks > 0: block i takes the weights [start(i), start(i + 1)), equal to
// within one tile, through as many units as they span; a unit cut by a
// share's end is merged from partial rows by prefill_merge_kernel: partial
// 2 i is block i's first fragment, 2 i + 1 its last.  (Key splits of equal
// tile ranges left 27% of the block slots' time empty on the model's chunk,
// where a range may hold no visible tile; see prefill_attn32_kernel.)
// What a mask tensor shows is known on the device only: where every row block
// sees just the tiles of the causal rule, as under most models' masks, its
// weights stand; else each block sums the visible tiles (PfTable) and deals
// them by the same rule, to no more blocks than were launched.
// blocks == 0: block i is one whole unit, longest first, and nothing is
// summed over units (their tiles may pass 2^31; with shares they are at most
// 2^29).
struct PfShares {
  int nrb;                // row blocks of a (b, q head)
  int tiles;              // tiles of a unit (the last row block's weight)
  int blocks, per, rem;   // start(i) = i * per + min(i, rem)
  int slots;              // the GPU's block slots
  // Without a mask tensor: the weight of one (b, q head), and of its row
  // block rb < nrb - 1: a + step * rb.
  int head, a, step;
  KIV_HD void deal(int total, int n) {
    blocks = n;
    per = total / n;
    rem = total - per * n;
  }
  KIV_HD int start(int i) const { return i * per + (i < rem ? i : rem); }
  // Weight of the row blocks before rb.
  KIV_HD int before(int rb) const { return rb * a + step * (rb * (rb - 1) / 2); }
  KIV_HD int weight(int rb) const { return blocks == 0 || rb + 1 == nrb ? tiles : a + step * rb; }
  // Weights before unit (bh, rb); a block per unit counts from its own start.
  KIV_HD int unit_start(int bh, int rb) const { return blocks == 0 ? 0 : bh * head + before(rb); }

  // Block i's first unit (bh, rb) and its weights [w, w_end).
  KIV_HD void first(int i, int nbh, int &bh, int &rb, int &w, int &w_end) const {
    if (blocks == 0) {
      const int k = i / nbh;
      bh = i - k * nbh;
      rb = nrb - 1 - k;  // longest first
      w = 0;
      w_end = tiles;
      return;
    }
    w = start(i);
    w_end = start(i + 1);
    bh = w / head;
    const int rest = w - bh * head;
    rb = 0;  // the last row block that starts at or before it
    for (int hi = nrb - 1; rb < hi;) {
      const int mid = (rb + hi + 1) >> 1;
      if (before(mid) <= rest) rb = mid;
      else hi = mid - 1;
    }
  }
};

// Blocks that `all` tiles of weight are dealt to: the GPU's slots (two a
// compute unit), but no more than leave a block kPfShareTiles tiles, whose
// partial rows cost about that much to write and merge (200 positions of 28
// heads over 2,304 keys: 512 blocks of 4 tiles 24.6 + 14.6 us, 259 of 8 24.9
// + 9.0); work that would then leave compute units idle is dealt to all of
// them, down to two tiles a block.  Every unit weighs at least one tile.
constexpr int kPfShareTiles = 8;
KIV_HD inline int64_t pf_min(int64_t a, int64_t b) { return a < b ? a : b; }
KIV_HD inline int64_t pf_max(int64_t a, int64_t b) { return a > b ? a : b; }
KIV_HD inline int share_blocks_of(int64_t all, int64_t units, int slots) {
  const int64_t few = pf_min(slots / 2, all / 2);
  const int64_t blocks = pf_min(slots, pf_max(few, all / kPfShareTiles));
  return (int)pf_max(blocks, pf_min(units, slots));
}
KIV_HD inline int64_t pf_div_up(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Blocks to launch with shares, or 0: a block per unit, where the units fill
// two rounds of the slots (or pass the kernel's table of them).
constexpr int kPfMaxUnits = 1024;
inline int prefill_share_blocks(int Q, int BH, int cold_len, int hot_len, int slots) {
  const int64_t units = pf_div_up(Q, kPfUnitRows) * BH,
                tiles = pf_div_up(cold_len, kPfKeys) + pf_div_up(hot_len, kPfKeys);
  if (units >= pf_min(2 * (int64_t)slots, kPfMaxUnits) || units * tiles > INT32_MAX / 4 || tiles < 4) return 0;
  return share_blocks_of(units * tiles, units, slots);
}

// causal: weights by the causal rule (mask tensors too, see above); else every
// tile counts.
inline PfShares prefill_shares(int Q, int BH, int cold_len, int hot_len, bool causal, int blocks, int slots) {
  PfShares s{};
  const int nct = (int)pf_div_up(cold_len, kPfKeys), nht = (int)pf_div_up(hot_len, kPfKeys), off = hot_len - Q;
  s.nrb = (int)pf_div_up(Q, kPfUnitRows);
  s.tiles = nct + nht;
  s.blocks = blocks;
  s.slots = slots;
  if (blocks == 0) return s;
  if (causal && off >= 0) {
    // Row block rb's last row sees hot columns up to 128 (rb + 1) - 1 + off.
    s.a = nct + kPfUnitRows / kPfKeys + (int)pf_div_up(off, kPfKeys);
    s.step = kPfUnitRows / kPfKeys;
  } else {
    s.a = s.tiles;
    s.step = 0;
  }
  s.head = s.before(s.nrb - 1) + s.tiles;
  s.deal(s.head * BH, blocks);
  return s;
}

}  // namespace kiv
