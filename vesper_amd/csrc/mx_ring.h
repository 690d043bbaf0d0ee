// LDS layout of the prefill gate/up kernel's ring (mx_prefill.hip): plain arithmetic, compiled for the GPU by hipcc and
// for the CPU by hostcheck.cpp, where the tests check its bounds.
#pragma once
#include <cstdint>

namespace mxring {

// a stage: the 8 groups' weight tiles (group w, tile t at 1 KB x (4 w + t)), their scale words (256 B per
// group), then the activations of the tile's live token tiles: token tile u, block b at 1 KB x (4 u + b)
constexpr int kXStageA = 0, kXStageAS = 32768, kXStageB = 34816;
constexpr int xstage_bytes(int live) { return kXStageB + 4096 * live; }
// stages in the ring with `live` token tiles: as many as the LDS holds, at most 4
constexpr int xstages(int live) { return 160 * 1024 / xstage_bytes(live) < 4 ? 160 * 1024 / xstage_bytes(live) : 4; }
constexpr int xlds_bytes(int live) { return xstages(live) * xstage_bytes(live); }
constexpr int xlds_max(int live = 8) {
  return live == 0 ? 0 : xlds_bytes(live) > xlds_max(live - 1) ? xlds_bytes(live) : xlds_max(live - 1);
}
constexpr int kXLdsBytes = xlds_max();

// How many token tiles a read of activation operands takes when it starts at token tile u (a multiple of 4) of a tile
// with `live` token tiles: the next four, as far as they are live. The stage ends with the last live tile, and in the
// ring's last slot so may the LDS.
constexpr int xacts_read(int live, int u) { return live - u < 4 ? live - u : 4; }

}  // namespace mxring
