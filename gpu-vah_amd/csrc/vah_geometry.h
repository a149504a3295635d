// vah_geometry.h -- tiles and launch geometry of the single-lattice stage kernels:
// which tile, how many eta planes a workgroup marches through, the grid.
#pragma once

namespace vah {

// Tile of the single-lattice kernels: 8 x 7 cells, one face wave and one cell
// wave.  Its x faces (9 x 7 = 63) and y faces (8 x 8 = 64) fill a wave, its
// cells 56 lanes of one.
constexpr int kTileX = 8;
constexpr int kTileY = 7;
constexpr int kTileWaves = 1;  // waves per role

// Tile of the single-lattice kernels on large lattices: 16 x 7 cells, two
// waves per role.  A field's row with its halo is 20 doubles, 2.2 lines of 128 bytes
// on average, where two tiles of 8 x 7 need 1.7 each (choose_wide_tiles says where
// that pays).
constexpr int kWideTileX = 16;
constexpr int kWideTileWaves = 2;

// The per-cell-flux kernels: 256 lanes, one per cell of a 16 x 16 tile.
constexpr int kCellTileX = 16;
constexpr int kCellTileY = 16;
constexpr int kCellThreads = 256;

// Launch geometry of one lattice: tiles marching kz eta planes.
struct Geometry {
    int tiles_x, tiles_y, zchunks, kz, nblocks, grid;
    bool wide;  // 16 x 7 tiles instead of 8 x 7
};

constexpr int ceil_div(int a, int b) { return (a + b - 1) / b; }

// 16 x 7 tiles pay where the lattice gives about 2,300 workgroups of three planes:
// 512 of them run at once, and with fewer than some four rounds the last one, of
// workgroups twice as long, costs more than the halo saves.  Per step with 8 x 7 /
// 16 x 7 tiles, FP64: 101x101x30 (1,050 workgroups) 190 / 206 us, 101x101x60 (2,100)
// 385 / 391, 121x121x50 (2,448) 473 / 457, 151x151x101 1322 / 1200, 201x201x101
// 2267 / 2024, 301x301x31 1597 / 1398; split 101x101x60 379 / 379, 121x121x50
// 459 / 440, 201x201x101 2243 / 1986.  Tiles of 16 x 15 (four waves per role):
// 2238 at 201x201x101.  On a boost-invariant lattice, whose workgroups are shorter,
// they pay from about a million cells on, where the halo's rows come from memory: FP64
// 611x587 137 / 136, 801x801 251 / 249, 1001x1001 (9,009 workgroups) 422 / 414 us,
// 2001x2001 1.65 / 1.60, 3001x3001 3.63 / 3.51, 4001x4001 7.84 / 7.10 ms; split 801x801
// 246 / 247, 1001x1001 410 / 409 us, 2001x2001 1.61 / 1.57, 4001x4001 7.82 / 7.11 ms.
// (The kernels before the roles, of 16 x 15 tiles, took 7.12 and 6.89 ms there; with the
// role kernels 16 x 15 tiles take 7.82 and 7.76.)
// Narrow ones stay out, whose rows the L2 keeps until the next row of tiles needs them:
// 129x8001 427 / 436 us, split 417 / 440; 769x1401 448 / 438, split 439 / 436.
inline bool choose_wide_tiles(int nx, int ny, int nz) {
    const long tiles = (long)ceil_div(nx, kWideTileX) * ceil_div(ny, kTileY);
    return nz > 1 ? tiles * ceil_div(nz, 3) >= 2300 : tiles >= 9000 && nx >= 48 * kWideTileX;
}

// Eta planes per workgroup when the caller leaves the choice (opt.eta_chunk 0).
// A chunk of kz planes solves kz + 1 eta faces per cell and starts by loading
// three planes of each column, so longer chunks do less work; but a lattice of
// few tiles then leaves CUs idle.  1,024 workgroups (512 of 16 x 7 tiles) run at once.
// us per step, FP64, with 8 x 7 tiles and kz = 1 / 2 / 3 / 6: 33x31x7 (25 tiles)
// 31 / 46 / 63 / 112, 53x67x13 (70) 45 / 49 / 64 / 88, 71x71x41 (99) 142 / 142 / 143 /
// 139, 81x81x41 (132) 176 / 170 / 168 / 171, 101x101x30 (195) 186 / 175 / 175 / 172,
// 101x101x60 405 / 378 / 372 / 375; between them 61x61x41 (72 tiles, 1,008 workgroups of
// three planes) takes 106 / 105 / 97 / 122, of which the rule picks the first.  With
// 16 x 7 tiles and kz = 3 / 6 / 8: 121x121x50 (1,296 workgroups of six planes) 440 / 438 /
// 448, 161x161x41 (1,771) 597 / 569 / 577, 141x141x61 (2,079) 674 / 662 / 645,
// 181x181x51 (2,808) 910 / 862 / 873, 201x201x101 (6,409) 2139 / 2039 / 2024.
// Split precision: the same order at 1 to 4 % less.
inline int choose_eta_chunk(int tiles, int nz, bool wide) {
    auto groups = [&](int kz) { return (long)tiles * ceil_div(nz, kz); };
    if (wide) return groups(6) >= 2048 ? 6 : 3;
    if (groups(3) >= 1536) return 3;
    if (groups(2) >= 1536) return 2;
    return 1;
}

// The per-cell kernels solve every face of every plane whatever the chunk: one plane.
// With 1 / 2 / 3 / 6: 33x31x7 182 / 275 / 399 / 755 us per step, 101x101x30 0.98 / 1.03 /
// 1.26 / 1.33 ms, 151x151x101 6.66 / 6.65 / 7.01 / 7.51, 301x301x61 16.0 / 15.8 / 16.1 /
// 16.4.
constexpr int kCellChunk = 1;

inline Geometry launch_geometry(int nx, int ny, int nz, bool shared, int eta_chunk) {
    Geometry g;
    g.wide = shared && choose_wide_tiles(nx, ny, nz);
    const int tx = !shared ? kCellTileX : g.wide ? kWideTileX : kTileX, ty = shared ? kTileY : kCellTileY;
    g.tiles_x = ceil_div(nx, tx);
    g.tiles_y = ceil_div(ny, ty);
    const int tiles = g.tiles_x * g.tiles_y;
    const int kz = eta_chunk > 0 ? eta_chunk : shared ? choose_eta_chunk(tiles, nz, g.wide) : kCellChunk;
    g.kz = kz < nz ? kz : nz;
    g.zchunks = ceil_div(nz, g.kz);
    g.nblocks = tiles * g.zchunks;
    g.grid = g.zchunks * 8 * ceil_div(tiles, 8);  // tile_of_block's grid
    return g;
}

}  // namespace vah
