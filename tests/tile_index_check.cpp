// fg_tiles.h, compiled for the host: replays the tiles of one grid and counts
// what k_mg_up0 and k_pcg_dir would own and read (test_window_indexing.py).
#include <vector>

#include "fg_tiles.h"

using namespace fg;

// 0, or the number of the first check that fails.
extern "C" int check_tiles(int I, int J, int min_chunk, int most)
{
    const int tiles = up_tiles(I, J), tj = up_tiles_j(J), C = I * J;
    const int blocks = (int)up_block_count(tiles, min_chunk, most);
    if (blocks < 1 || blocks > most || blocks > tiles) return 1;
    std::vector<int> owner(C, 0);
    int next = 0;
    for (int blk = 0; blk < blocks; blk++) {
        const TileRun run = up_run(tiles, blocks, blk);
        if (run.first != next || run.end <= run.first) return 2;   // consecutive runs, none empty
        next = run.end;
        for (int tile = run.first; tile < run.end; tile++) {
            const TileAt t = up_tile(tile, tj);
            for (int k = 0; k < kUpR * kUpR; k++) {
                const int a = k / kUpR, b = k % kUpR, i = t.i - 1 + a, j = t.j - 1 + b;
                const int f = up_halo(t, k, I, J), fl = up_halo_linear(t, k, I, J);
                if (f < 0 || f >= C || fl < 0 || fl >= C) return 3;
                if (i < 0 || i >= I || j < 0 || j >= J) continue;
                if (f != i * J + j || fl != i * J + j) return 4;
                // the level-1 parents of cell (i, j) lie in the patch, at the cells that bilinear interpolation takes
                const int near[2] = {up_near(a), up_near(b)}, far[2] = {up_far(a), up_far(b)}, cell[2] = {i, j};
                for (int x = 0; x < 2; x++) {
                    if (near[x] < 0 || near[x] >= kUpY || far[x] < 0 || far[x] >= kUpY) return 5;
                    const TileAt n = up_patch(t, x ? near[x] : near[x] * kUpY), g = up_patch(t, x ? far[x] : far[x] * kUpY);
                    const int parent = cell[x] / 2, other = (cell[x] & 1) ? parent + 1 : parent - 1;
                    if ((x ? n.j : n.i) != parent || (x ? g.j : g.i) != other) return 6;
                }
                if (a == 0 || a > kUpTile || b == 0 || b > kUpTile) continue;
                owner[f]++;
                // the matrix couples cell c to c - J, c + J, c - 1, c + 1, across a row's end too
                const int c = i * J + j, at[4] = {k - kUpR, k + kUpR, k - 1, k + 1}, to[4] = {c - J, c + J, c - 1, c + 1};
                for (int e = 0; e < 4; e++)
                    if (to[e] >= 0 && to[e] < C && up_halo_linear(t, at[e], I, J) != to[e]) return 7;
            }
        }
    }
    if (next != tiles) return 8;
    for (int n : owner)
        if (n != 1) return 9;
    return 0;
}
