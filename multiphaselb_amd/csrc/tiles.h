// Several time steps per launch on small lattices (kernels_tiles.hip; k_fused_tile of
// kernels_fused.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <functional>
#include <vector>

#include "kernels.h"

struct mplb_case;

namespace mplb {

constexpr int kTileLists = 8;    // boundary lists a tiled case may have

struct TileList {
    int type;
    double value, pert;
    int left;                    // fixedRandomT: steps that still draw, counted from the launch's first
};

// Local node lists of the tiles, `stride` entries each, sorted by depth (0: owned; a node at
// depth d + 1 is a neighbour of one at depth d).
struct TileTable {
    int tiles, stride;
    int64_t total;               // tiles * stride
    const int* gid;              // [total] lattice node
    const int16_t* nb;           // [Q][total] local upstream node, -1 missing
    const int16_t* inner;        // [Q][total] fixedT links: local upstream node of the inner neighbour (may be null)
    const int* meta;             // [total] f list | g list << 8 | interior << 16 | full << 17 | depth << 24 (255: unused)
    const int* draw;             // [total] first fixedRandomT draw (null without such lists)
};

template <typename T>
struct TileState {
    T *f, *g, *rho, *temp, *U, *Fi, *Ft, *ss, *psi;
};

template <typename T>
struct TileArgs {
    TileTable t;
    int64_t N;
    int steps;                   // of this launch
    EosParams eos;
    ModelParams fp, gp;
    T rho0;
    const double* rnd;
    TileList lists[2][kTileLists];
    int first_level;             // liTempMRT: the launch's step that is the heat source's first call (-1: none)
    TileState<T> in, out;
};

template <typename T>
struct TileOps {
    // largest tile (local nodes) the kernel can take
    static int max_nodes(int model, bool thermal);
    static void run(int model, hipStream_t s, const TileArgs<T>& a, bool thermal, int nodes);
};

// What a tiled case keeps on the device
struct Tiles {
    TileTable t{};
    int nodes = 0;               // largest tile
    int steps = 0;               // per launch
    std::vector<void*> owned;
};

struct TilePlan {
    int b[3] = {0, 0, 0};        // owned block
    int steps = 0;               // per launch (0: no tiles)
    double us = 0;               // estimated time of a step
};

// The cheapest plan under limit_us on a structured box: `us` estimates a step's time with a
// plan of blocks of the given sizes (1e30: its tiles do not fit).
TilePlan tile_choose(const mplb_case* c, const std::vector<int>& sizes, double limit_us,
                     const std::function<double(const TilePlan&)>& us);
// MPLB_TILES=bx,by,bz,steps sets the plan (steps 0: no tiles), for tests and timing sweeps
void tile_override(TilePlan* p);
// Builds the tables of a plan whose halo is `depth` levels (c->tiles); false, and the case
// without, when a tile has more than cap nodes or memory runs out.  lists: the field has
// boundary lists.
bool tile_tables(mplb_case* c, const TilePlan& p, int depth, int cap, const bool lists[2]);
// Chooses tiles for a case that runs in fused passes and builds their tables (c->tiles);
// leaves the case without when more launches over the whole lattice are the faster way or
// memory runs out.
void tiles_create(mplb_case* c);
void tiles_destroy(mplb_case* c);
// m steps from and to the per-routine state (psi valid on entry); level0: the time level
// before the first of them
template <typename T>
void tiles_run(mplb_case* c, int m, int level0);

}  // namespace mplb
