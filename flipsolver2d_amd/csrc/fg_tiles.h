// fg_tiles.h -- which cells the solver's level-0 tiles own and stage: the
// index arithmetic of k_mg_up0 (fg_mg.hip) and k_pcg_dir (fg_pcg.hip), and the
// block count that the host gives them.  No HIP types, so a host compiler
// takes it too.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define FG_HD __host__ __device__ __forceinline__
#else
#define FG_HD inline
#endif

namespace fg {

constexpr int kUpTile = 32;           // cells a tile, per side
constexpr int kUpR = kUpTile + 2;     // with the one-cell halo
constexpr int kUpY = kUpTile / 2 + 2; // level-1 cells a side that the halo's cells prolong from

FG_HD int up_tiles_j(int J) { return (J + kUpTile - 1) / kUpTile; }
FG_HD int up_tiles(int I, int J) { return ((I + kUpTile - 1) / kUpTile) * up_tiles_j(J); }

// Blocks for `tiles` tiles: as many tiles a block as the solver's least chunk
// of cells holds, more where the blocks or the partials run out; every block
// has a tile.
FG_HD int64_t up_block_count(int64_t tiles, int64_t min_chunk, int64_t most)
{
    const int64_t per = min_chunk / (kUpTile * kUpTile);
    const int64_t least = per > 1 ? (tiles + per - 1) / per : tiles;
    const int64_t ub = least < most ? least : most;
    const int64_t run = (tiles + ub - 1) / ub;
    return (tiles + run - 1) / run;
}
// The run of tiles of block `blk` of `blocks`.
struct TileRun {
    int first, end;
};
FG_HD TileRun up_run(int tiles, int blocks, int blk)
{
    const int per = (tiles + blocks - 1) / blocks, first = blk * per, end = first + per;
    return TileRun{first, end < tiles ? end : tiles};
}
// A tile's first cell.
struct TileAt {
    int i, j;
};
FG_HD TileAt up_tile(int tile, int tiles_j)
{
    const int ti = tile / tiles_j;
    return TileAt{kUpTile * ti, kUpTile * (tile - ti * tiles_j)};
}

FG_HD int clamp_to(int v, int last) { return v < 0 ? 0 : v > last ? last : v; }

// Cell of position k (row-major, kUpR a side) of a tile with its halo: at the
// clamped row and column, and at the clamped linear index, where a row's end
// runs on into the next row as the reference's matrix couples them.
FG_HD int up_halo(TileAt t, int k, int I, int J)
{
    return clamp_to(t.i - 1 + k / kUpR, I - 1) * J + clamp_to(t.j - 1 + k % kUpR, J - 1);
}
FG_HD int up_halo_linear(TileAt t, int k, int I, int J)
{
    return clamp_to((t.i - 1 + k / kUpR) * J + (t.j - 1 + k % kUpR), I * J - 1);
}

// Level-1 cell of position k (row-major, kUpY a side) of the patch under a
// tile, per axis; it may lie outside the level.
FG_HD TileAt up_patch(TileAt t, int k) { return TileAt{t.i / 2 - 1 + k / kUpY, t.j / 2 - 1 + k % kUpY}; }
// Patch rows (or columns) of the near and the far parent of row (column) a of
// the tile with its halo: cell t.i - 1 + a, t.i even, so an even cell (odd a)
// takes its own parent and the one before, an odd one the next.
FG_HD int up_near(int a) { return (a + 1) >> 1; }
FG_HD int up_far(int a) { return (a & 1) ? up_near(a) - 1 : up_near(a) + 1; }

}  // namespace fg
