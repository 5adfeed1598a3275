// d2q9_tile.h -- several iterations per launch: the host side's view of the
// kernels in d2q9_tile.hip.
#pragma once
#include "d2q9_node.h"
#include "d2q9_plan.h"

namespace lbm {

// A tile plan (d2q9_plan.h) on the device; n = 0: one iteration per launch.
struct TileSet {
    int n = 0, K = 0, cfg = 0, n_in = 0;
    bool links = false;
    size_t lds = 0;
    TileDesc *d_tiles = nullptr;
    TileLink *d_links = nullptr;
    uint32_t *d_nodes = nullptr;
};

// One launch of the tile kernel of a plan: a lattice's (p) or a batch's
// (cases, ring offset k, counter, parity).
struct TileLaunch {
    const TileSet &t;
    int n;                       // iterations (odd, at most t.K)
    const Params *p;
    const Params *cases;
    int k;
    const int *base;
    int parity;
    hipStream_t s;
};

// Launches the kernel of storage form S (d2q9_tile.hip, one object per form).
template <int S> void launch_tile_s(const TileLaunch &a);

}  // namespace lbm
