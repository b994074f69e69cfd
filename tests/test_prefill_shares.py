"""The shares of the prefill attention's work (head dims up to 128), walked on
the host as its blocks walk them: every tile of every unit is taken by exactly
one block, also where the tiles pass 2^31."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

HEADER = Path(__file__).resolve().parents[1] / "kiv_amd" / "csrc" / "kiv_prefill_shares.h"

# Prints, per shape "Q BH cold hot causal slots": blocks, units, fragments,
# tiles taken, units not taken from first tile to last in one piece or in
# consecutive fragments, and the largest and smallest share.
WALK = r"""
#include <stdio.h>
#include <algorithm>
#include <vector>
#include "%s"
using namespace kiv;
int main() {
  long long Q, BH, cold, hot, causal, slots;
  while (scanf("%%lld %%lld %%lld %%lld %%lld %%lld", &Q, &BH, &cold, &hot, &causal, &slots) == 6) {
    const int nb = prefill_share_blocks(Q, BH, cold, hot, slots);
    const PfShares sh = prefill_shares(Q, BH, cold, hot, causal, nb, slots);
    const long long units = (long long)sh.nrb * BH, grid = nb > 0 ? nb : units;
    std::vector<int> next(units, 0);  // first tile of the unit not taken yet
    std::vector<char> order(units, 1);
    long long frags = 0, taken = 0, most = 0, least = 1LL << 62;
    for (long long i = 0; i < grid; ++i) {
      int bh, rb, w, w_end;
      sh.first((int)i, (int)BH, bh, rb, w, w_end);
      long long mine = 0;
      while (w < w_end) {
        const long long u = (long long)bh * sh.nrb + rb;
        const int us = sh.unit_start(bh, rb), ue = us + sh.weight(rb);
        const int t0 = w - us, t1 = w_end >= ue ? sh.tiles : w_end - us;
        if (u < 0 || u >= units || t0 != next[u] || t1 <= t0) { if (u >= 0 && u < units) order[u] = 0; break; }
        next[u] = t1;
        mine += (w_end >= ue ? ue : w_end) - w;
        taken += t1 - t0;
        ++frags;
        w = ue;
        if (++rb == sh.nrb) { rb = 0; ++bh; }
      }
      most = std::max(most, mine);
      least = std::min(least, mine);
    }
    long long bad = 0;
    for (long long u = 0; u < units; ++u) bad += !order[u] || next[u] != sh.tiles;
    printf("%%d %%lld %%lld %%lld %%lld %%lld %%lld\n", nb, units, frags, taken, bad, most, least);
  }
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    work = tmp_path_factory.mktemp("shares")
    src = work / "walk.cc"
    src.write_text(WALK % HEADER)
    subprocess.run([gxx, "-O1", "-std=c++17", "-fwrapv", str(src), "-o", str(work / "walk")], check=True)

    def run(*shape):
        out = subprocess.run([str(work / "walk")], input=" ".join(map(str, shape)), capture_output=True, text=True,
                             check=True, timeout=60).stdout
        return [int(x) for x in out.split()]

    return run


SHAPES = [
    # Q, batch * heads, cold, hot, causal
    (4096, 12, 0, 8192, 1), (777, 64, 0, 1531, 1), (1, 8, 1000, 3000, 0), (128, 1, 0, 256, 1), (129, 3, 65, 1100, 1),
    (513, 4, 0, 1537, 1), (200, 28, 256, 2048, 1), (500, 4, 70, 300, 1), (512, 256, 0, 520, 1), (4096, 12, 0, 8192, 0),
    # units of 2^31 tiles and more in all
    (1 << 20, 32, 0, 1 << 20, 1), (1 << 20, 16, 0, 1 << 20, 0), (1 << 20, 64, 300, 1 << 20, 0),
    (1 << 22, 8, 0, 1 << 22, 1),
    # few row blocks over very many keys: at the limit of the shares' own arithmetic
    (128, 64, 0, 1 << 27, 0), (128, 255, 0, 1 << 27, 0), (8192, 8, 0, 1 << 26, 1),
]


@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_every_tile_is_taken_once(walk, shape):
    Q, bh, cold, hot, causal = shape
    blocks, units, frags, taken, bad, most, least = walk(*shape, 512)
    tiles = -(-cold // 64) + -(-hot // 64)
    assert units == -(-Q // 128) * bh
    assert bad == 0
    assert taken == units * tiles
    assert frags >= units
    if blocks:
        assert most - least <= 1  # equal shares of the weights
    else:
        assert frags == units
