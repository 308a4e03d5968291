// Cell binning as a counting sort: per-cell histogram (integer atomics give
// each atom a provisional slot), device exclusive scan to cell offsets,
// scatter, then an in-place sort of every cell segment by atom index so the
// cell lists are exactly the index-ordered lists of the reference's CPU
// mapping (core/grid.impala:280-321; cell math core/grid.impala:406-426).
#include "tmd_internal.hpp"
#include "tmd_device.hpp"
#include "tmd_window.hpp"

namespace tmd {

__global__ void k_bin_count(const double4* __restrict__ pos, BinArgs a, int nall, int* __restrict__ cell_of,
                            int* __restrict__ slot, int* __restrict__ count, int* __restrict__ inv) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    int c = -1;
    if (i < nall) {
        const double4 p = pos[i];
        const double fx = floor((p.x - a.xmin) / a.spacing);
        const double fy = floor((p.y - a.ymin) / a.spacing);
        const double fz = floor((p.z - a.zmin) / a.spacing);
        // non-finite or absurd coordinates are treated as outside the grid
        if (fabs(fx) < 1e9 && fabs(fy) < 1e9 && fabs(fz) < 1e9) {
            const int ci = (int)fx, cj = (int)fy, ck = (int)fz;
            const long long flat = ((long long)ck * a.ny + cj) * a.nx + ci;
            if (flat >= 0 && flat < a.ncells) c = (int)flat;
        }
    }
    const int sl = wave_cell_slot(c, count);  // all lanes take part
    if (i >= nall) return;
    cell_of[i] = c;
    slot[i] = sl;
    if (c < 0) inv[i] = -1;  // the sort sets the binned ones
}

// Counting-sort placement: (atom, source slot) of every binned atom into its
// cell's segment.  Blocks below nbq take the source slots (MIR: mirror slots
// of the last binning, holding atom parts[q]; else atom q itself), the rest
// the ghosts of the emit sweep, their number read on the device.
template <bool MIR>
__global__ void __launch_bounds__(256) k_bin_place(const int* __restrict__ cell_of, const int* __restrict__ slot, int nq, int nbq,
                                                   const int* __restrict__ parts, const int* __restrict__ g_cell,
                                                   const int* __restrict__ g_slot, int n, int gcap,
                                                   const int* __restrict__ ctr, const int* __restrict__ start,
                                                   int2* __restrict__ pairs) {
    const int b = blockIdx.x;
    if (b < nbq) {
        const int q = b * 256 + (int)threadIdx.x;
        if (q >= nq) return;
        const int c = cell_of[q];
        if (c >= 0) pairs[start[c] + slot[q]] = make_int2(MIR ? parts[q] : q, q);
        return;
    }
    const int ng = min(ctr[CT_NGHOST], gcap);
    for (int g = (b - nbq) * 256 + (int)threadIdx.x; g < ng; g += ((int)gridDim.x - nbq) * 256) {
        const int c = g_cell[g];
        if (c >= 0) pairs[start[c] + g_slot[g]] = make_int2(n + g, -1);
    }
}

// Work tile of a cell that can hold locals, -1 for the grid's outer cells.
__device__ __forceinline__ int cell_tile(int c, const TileGeom& g) {
    const int x = c % g.nx, y = (c / g.nx) % g.ny, z = c / (g.nx * g.ny);
    if (x < 1 || y < 1 || z < 1 || x > g.nx - 2 || y > g.ny - 2 || z > g.nz - 2) return -1;
    return ((z - 1) / g.tz * g.nty + (y - 1) / g.ty) * g.ntx + (x - 1) / g.tx;
}

// One thread per cell (sparse grids: a few atoms per cell): each pair's rank
// by counting, then the cell's locals and the CSR index of every atom; the
// same result as k_bin_sort.
__global__ void k_bin_sort_small(const int* __restrict__ start, int ncells, int n, const int2* __restrict__ pairs,
                                 int* __restrict__ parts, int* __restrict__ src, int* __restrict__ local_count,
                                 int* __restrict__ inv, TileGeom g, int* __restrict__ tile_count) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncells) return;
    const int b = start[c], e = start[c + 1], m = e - b;
    int nl = 0;
    constexpr int kHeld = 6;  // pairs held in registers
    if (m <= kHeld) {
        int2 v[kHeld];
#pragma unroll
        for (int k = 0; k < kHeld; ++k) v[k] = k < m ? pairs[b + k] : make_int2(0x7fffffff, 0);
#pragma unroll
        for (int k = 0; k < kHeld; ++k) {
            if (k >= m) break;
            int rank = 0;
#pragma unroll
            for (int q = 0; q < kHeld; ++q) rank += v[q].x < v[k].x ? 1 : 0;
            parts[b + rank] = v[k].x;
            src[b + rank] = v[k].y;
            inv[v[k].x] = b + rank;
            nl += v[k].x < n ? 1 : 0;
        }
    } else {
        for (int k = b; k < e; ++k) {
            const int2 v = pairs[k];
            int rank = 0;
            for (int q = b; q < e; ++q) rank += pairs[q].x < v.x ? 1 : 0;
            parts[b + rank] = v.x;
            src[b + rank] = v.y;
            inv[v.x] = b + rank;
            nl += v.x < n ? 1 : 0;
        }
    }
    local_count[c] = nl;
    if (tile_count && nl > 0) {
        const int t = cell_tile(c, g);
        if (t >= 0) atomicAdd(&tile_count[t], nl);
    }
}

// One wavefront per cell: sort the cell segment by atom index; the number of
// locals in it (locals have the lowest indices, so they lead every sorted
// segment) goes to the cell and is added to its work tile.
__global__ void __launch_bounds__(256) k_bin_sort(const int* __restrict__ start, int ncells, int n, const int2* __restrict__ pairs,
                                                  int* __restrict__ parts, int* __restrict__ src, int* __restrict__ local_count,
                                                  int* __restrict__ inv, TileGeom g, int* __restrict__ tile_count) {
    const int c = blockIdx.x * (blockDim.x / kWave) + (int)threadIdx.x / kWave;
    if (c >= ncells) return;  // whole wavefronts
    const int nl = wave_sort_pairs(start[c], start[c + 1], n, pairs, parts, src, inv);
    if ((threadIdx.x & (kWave - 1)) == 0) {
        local_count[c] = nl;
        if (tile_count && nl > 0) {
            const int t = cell_tile(c, g);
            if (t >= 0) atomicAdd(&tile_count[t], nl);
        }
    }
}

// Locals of every tile, a wavefront per tile (large grids: one atomic per
// cell onto the tiles, as the sorts do for small ones, costs 30 us at 132,000
// cells and 50 us in the 560,000-cell DEM grid; this launch 5 us).
__global__ void __launch_bounds__(256) k_tile_count(const int* __restrict__ local_count, TileGeom g, int ntiles,
                                                    int* __restrict__ tile_count) {
    const int tile = blockIdx.x * 4 + (int)threadIdx.x / kWave;
    if (tile >= ntiles) return;  // whole wavefronts
    const int lane = threadIdx.x & (kWave - 1);
    const int tx_i = tile % g.ntx, ty_i = (tile / g.ntx) % g.nty, tz_i = tile / (g.ntx * g.nty);
    const int cx0 = 1 + tx_i * g.tx, cy0 = 1 + ty_i * g.ty, cz0 = 1 + tz_i * g.tz;
    const int ex = min(cx0 + g.tx, g.nx - 1) - cx0, ey = min(cy0 + g.ty, g.ny - 1) - cy0, ez = min(cz0 + g.tz, g.nz - 1) - cz0;
    int v = 0;
    for (int q = lane; q < ex * ey * ez; q += kWave)
        v += local_count[((cz0 + q / (ex * ey)) * g.ny + (cy0 + (q / ex) % ey)) * g.nx + (cx0 + q % ex)];
    const int tot = __builtin_amdgcn_readlane(wave_inclusive_scan(v), kWave - 1);
    if (lane == 0) tile_count[tile] = tot;
}
constexpr int kTileAtomicCells = 16384;  // grids up to this many cells count by atomics in the sort

// The last sweep of a rebuild before the lists, three independent parts in
// one launch (each alone is a few microseconds on a small box):
//   blocks [0, ntiles): the tile's work order -- its locals in (z, y, x) cell
//   order (lanes of a wavefront are then atoms of adjacent cells, whose
//   neighbour windows overlap; measured faster than grouping lanes by list
//   length) with mirror index, cell and ghost entries -- and the tile and
//   window statistics;
//   the next nbm blocks: the cell-ordered mirror, positions (and velocities)
//   from the last mirror (MIR) or from atom order;
//   the rest: the mirror indices of every ghost and its owner, and the
//   ghost index.
// With few tiles (scanned == 0) a tile's first work slot is the sum of the
// counts before it, taken by the block itself: a scan launch less.
constexpr int kTileFlat = 2048;
struct FinishArgs {
    TileGeom g;
    int ntiles, scanned, n, gcap, ncells, nbm, ghost_vel;
};

template <bool MIR>
__global__ void __launch_bounds__(256) k_rebuild_finish(FinishArgs a, const int* __restrict__ start,
                                                        const int* __restrict__ local_count,
                                                        const int* __restrict__ tile_count, int* __restrict__ tile_start,
                                                        const int* __restrict__ parts, const int* __restrict__ src,
                                                        const int* __restrict__ inv, int* __restrict__ work,
                                                        int* __restrict__ work_k, int* __restrict__ work_c,
                                                        const int* __restrict__ gh_pack, int* __restrict__ gh_w,
                                                        const double4* __restrict__ pos, const double4* __restrict__ vel,
                                                        const CMir spos_old, const CMir svel_old, const Mir spos,
                                                        const Mir svel, const int* __restrict__ g_owner,
                                                        const int* __restrict__ g_code, const int* __restrict__ gh_e,
                                                        int* __restrict__ g_ko, int* __restrict__ g_kg, int2* __restrict__ gh_k,
                                                        int* __restrict__ ctr) {
    const int b = blockIdx.x, tid = threadIdx.x;
    if (b >= a.ntiles + a.nbm) {
        const int ng = min(ctr[CT_NGHOST], a.gcap);
        const int stride = ((int)gridDim.x - a.ntiles - a.nbm) * 256;
        for (int g = (b - a.ntiles - a.nbm) * 256 + tid; g < ng; g += stride) {
            const int kg = inv[a.n + g];
            g_ko[g] = inv[g_owner[g]];
            g_kg[g] = kg;
            const int e = gh_pack ? gh_e[g] : a.gcap;
            // entry numbers run past the capacity only where the host will grow it
            if (e < a.gcap) gh_k[e] = make_int2(kg, g_code[g] & 0xff);
        }
        return;
    }
    if (b >= a.ntiles) {
        const int k = (b - a.ntiles) * 256 + tid;
        if (k >= start[a.ncells]) return;
        const int j = parts[k];
        if (MIR && j < a.n) {
            const int q = src[k];
            spos[k] = spos_old[q];
            svel[k] = svel_old[q];
        } else {
            spos[k] = pos[j];
            if (svel.p && (j < a.n || a.ghost_vel)) svel[k] = vel[j];
        }
        return;
    }
    const TileGeom g = a.g;
    const int tile = b;
    __shared__ int coff[kMaxTile * kMaxTile * kMaxTile + 1];
    int w0, nloc;
    if (a.scanned) {
        w0 = tile_start[tile];
        nloc = tile_start[tile + 1] - w0;
    } else {
        int v = 0, tot;
        for (int t = tid; t < tile; t += 256) v += tile_count[t];
        (void)block_exclusive_scan(v, &tot);
        w0 = tot;
        nloc = tile_count[tile];
        if (tid == 0) {
            tile_start[tile] = w0;
            if (tile == a.ntiles - 1) tile_start[a.ntiles] = w0 + nloc;
        }
    }
    if (tid == 0) {
        if (tile == a.ntiles - 1) ctr[CT_PLACED] = w0 + nloc;
        if (tile == 0) ctr[CT_BINNED] = start[a.ncells];
    }
    if (nloc == 0) return;  // the whole block
    const int tx_i = tile % g.ntx, ty_i = (tile / g.ntx) % g.nty, tz_i = tile / (g.ntx * g.nty);
    const int cx0 = 1 + tx_i * g.tx, cy0 = 1 + ty_i * g.ty, cz0 = 1 + tz_i * g.tz;
    const int cx1 = min(cx0 + g.tx, g.nx - 1), cy1 = min(cy0 + g.ty, g.ny - 1), cz1 = min(cz0 + g.tz, g.nz - 1);
    const int ex = cx1 - cx0, ey = cy1 - cy0, ez = cz1 - cz0;
    const int nc = ex * ey * ez;
    // cell offsets inside the tile and the window's size (its rows' lengths)
    int S = 0;
    {
        const int xlo = cx0 - 1, xhi = min(cx0 + g.tx, g.nx - 1), wy = g.ty + 2;
        for (int q = tid; q < wy * (g.tz + 2); q += 256) {
            const int y = cy0 - 1 + q % wy, z = cz0 - 1 + q / wy;
            if (y < g.ny && z < g.nz) {
                const int row = (z * g.ny + y) * g.nx;
                S += start[row + xhi + 1] - start[row + xlo];
            }
        }
        int tot;
        (void)block_exclusive_scan(S, &tot);
        S = tot;
    }
    int carry = 0;
    for (int q0 = 0; q0 < nc; q0 += 256) {
        const int q = q0 + tid;
        const int v = q < nc ? local_count[((cz0 + q / (ex * ey)) * g.ny + (cy0 + (q / ex) % ey)) * g.nx + (cx0 + q % ex)] : 0;
        int tot;
        const int ex_v = block_exclusive_scan(v, &tot);
        if (q < nc) coff[q] = carry + ex_v;
        carry += tot;
    }
    if (tid == 0) {
        coff[nc] = carry;
        // read first: only the few tiles that raise a maximum issue the atomic
        // (thousands of same-address atomics from separate blocks serialise)
        if (S > *(volatile int*)&ctr[CT_MAXWIN]) atomicMax(&ctr[CT_MAXWIN], S);
        if (nloc > *(volatile int*)&ctr[CT_MAXLOC]) atomicMax(&ctr[CT_MAXLOC], nloc);
    }
    __syncthreads();
    // one thread per local (coalesced writes): its cell is the last one whose
    // offset does not exceed its place (empty cells are passed over)
    for (int e = tid; e < nloc; e += 256) {
        int lo = 0, hi = nc - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (coff[mid] <= e) lo = mid;
            else hi = mid - 1;
        }
        const int c = ((cz0 + lo / (ex * ey)) * g.ny + (cy0 + (lo / ex) % ey)) * g.nx + (cx0 + lo % ex);
        const int k = start[c] + (e - coff[lo]);
        const int i = parts[k];
        work[w0 + e] = i;
        work_k[w0 + e] = k;  // the atom's mirror index
        work_c[w0 + e] = c;
        gh_w[w0 + e] = gh_pack ? gh_pack[i] : 0;
    }
}

// Cells per tile: about 480 locals per tile (one 512-thread block), with
// the window (tile + 1 cell on each side) inside the LDS budget.  The
// density is taken over the domain's volume in cells, not over the grid's
// inner cells: the grid rounds each side up by up to a cell and a half, so
// a small box would look up to twice as sparse as it is.  An explicit choice
// (tmd_set_tile) overrides.
int auto_tile_edge(const Geom& G, int n) {
    double cells = 1.0;
    for (int d = 0; d < 3; ++d) cells *= std::max((G.rank[2 * d + 1] - G.rank[2 * d]) / G.spacing, 1.0);
    const double rho = std::max((double)n / cells, 1e-3);
    int T = (int)std::lround(std::cbrt(480.0 / rho));
    T = std::max(1, std::min(T, kMaxTile));
    while (T > 1 && (T + 2.0) * (T + 2.0) * (T + 2.0) * rho * 28.0 > 0.85 * kLdsBudget) --T;
    return T;
}

// A dense box of this many cubes of about 480 locals keeps them: from there
// the smaller share of window atoms a local (4.6 against 6.7 in the LJ liquid)
// counts for more than full CUs.  us a step at 3x3x3 against 3x2x2: 48^3
// (1,000 cubes) FP32-mixed 62 against 65; 52^3 half lists FP64 107 against 111;
// 80^3 214 against 226.
constexpr int kManyTiles = 900;

// Order of the blocks over the XCDs (block_tile).  Up to one tile a CU no
// order helps, and its divisions cost 0.3 us a pass.  Dealt in runs from
// kManyTiles on where the box fills its last layer of tiles so little that
// equal ranges were more than 3 % uneven; else the ranges keep more of the
// windows in one L2 (36^3 cells, 1.8 %: 42.2 against 43.4 us; 53x47x39 76.8
// against 78.2).
static void order_tiles(const Geom& G, TileGeom& g) {
    double cells[3];  // of the box
    for (int d = 0; d < 3; ++d) cells[d] = (G.rank[2 * d + 1] - G.rank[2 * d]) / G.spacing;
    auto reached = [](double len, int edge, int nt) {
        return (int)std::min((double)nt, std::max(1.0, std::ceil(std::ceil(len - 1e-9) / edge)));
    };
    g.ox = reached(cells[0], g.tx, g.ntx);
    g.oy = reached(cells[1], g.ty, g.nty);
    g.oz = reached(cells[2], g.tz, g.ntz);
    const int tiles = g.ox * g.oy * g.oz;
    if (tiles >= kManyTiles && g.oz - cells[2] / g.tz > 0.03 * g.oz) g.order = ORDER_DEAL;
    else g.order = tiles > kNumCu && tiles < g.ntx * g.nty * g.ntz ? ORDER_BOX : ORDER_ALL;
}

TileGeom make_tile_geom(const Geom& G, int tx, int ty, int tz) {
    TileGeom g;
    g.nx = G.nx; g.ny = G.ny; g.nz = G.nz;
    g.tx = std::max(1, std::min(tx, kMaxTile));
    g.ty = std::max(1, std::min(ty, kMaxTile));
    g.tz = std::max(1, std::min(tz, kMaxTile));
    g.ntx = std::max(1, div_up(G.nx - 2, g.tx));
    g.nty = std::max(1, div_up(G.ny - 2, g.ty));
    g.ntz = std::max(1, div_up(G.nz - 2, g.tz));
    order_tiles(G, g);
    return g;
}

constexpr double kTileLocals = 320.0, kDemTileLocals = 288.0;

static double mean_density(const Sim& s) {  // locals a cell of the box
    double cells = 1.0;
    for (int d = 0; d < 3; ++d) cells *= std::max((s.g.rank[2 * d + 1] - s.g.rank[2 * d]) / s.g.spacing, 1.0);
    return (double)s.n / cells;
}

// Near-cubic tile shapes by size: (t, t, t), (t, t, t - 1), (t, t - 1, t - 1).
struct TileShape {
    int x, y, z;
};
static TileShape tile_shape(int k) {  // k = 0: one cell, 3 (t - 1): t^3
    const int t = 1 + (k + 2) / 3, r = (k + 2) % 3;
    return TileShape{t, r >= 1 ? t : t - (t > 1), r == 2 ? t : t - (t > 1)};
}
constexpr int kShapes = 3 * (kMaxTile - 1) + 1;

// Tile of the automatic choice for `rho` atoms a cell where the box is filled,
// a share `fill` of it, and windows of `slot` LDS bytes an atom within `budget`.
//   1. the largest shape of at most `most` locals whose window fits.  LJ 320 (a
//      block of four or five wavefronts): the liquid (18.5 a cell), us a step
//      at 3x2x2 against 3x3x3 cells: 32^3 FP64 34 against 44, 36^3 42 against
//      45; where the cubes are ahead choose_tiles takes them (rounds,
//      kManyTiles).
//      DEM 288, by a peak density a tenth over the mean (four wavefronts, six
//      blocks a CU): the gas (1.85 a cell where it is filled) at 64^3, 5x5x5
//      38.3, 6x5x5 40.9, 6x6x6 39.7, 5x4x4 40.7;
//   2. one size down where that leaves at least 160 locals and there are fewer
//      than 1,536 tiles (DEM 48^3, 5x5x4: 21.0 against 22.7 us; 64^3, 2,456
//      tiles, 39.1 against 38.3; the LJ liquid's next shape would have 148: 28^3
//      20.5 against 18.6 us);
//   3. smaller still until 200 tiles hold atoms, not below two cells: a pass
//      over fewer tiles than CUs leaves CUs idle and lasts as long as its
//      fullest block (10^3 FP64: 27 tiles of 3x3x3 24.7 us, 196 of 2x1x1 16.6;
//      DEM 17^3: 64 tiles of 6x6x6 17.7 us a step, 512 of 3x3x3 14.3).
static TileShape pick_tile(const Geom& G, double rho, double fill, int slot, int budget, double most) {
    rho = std::max(rho, 1e-3);
    auto cells = [](const TileShape& t) { return (double)t.x * t.y * t.z; };
    auto tiles = [&](const TileShape& t) {
        const TileGeom g = make_tile_geom(G, t.x, t.y, t.z);
        return (double)g.ntx * g.nty * g.ntz * fill;
    };
    int k = kShapes - 1;
    auto fits = [&](const TileShape& t) {
        return cells(t) * rho <= most && (t.x + 2.0) * (t.y + 2.0) * (t.z + 2.0) * rho * slot <= 0.95 * budget;
    };
    while (k > 0 && !fits(tile_shape(k))) --k;
    if (k > 0 && tiles(tile_shape(k)) < 1536.0 && cells(tile_shape(k - 1)) * rho >= 160.0) --k;
    while (k > 1 && tiles(tile_shape(k)) < 200.0) --k;
    return tile_shape(k);
}

// Between one cube a CU and kManyTiles the pass runs in rounds of one tile a
// CU, each as long as a tile: cubes where theirs take less.  Time of a tile as
// of its locals and 25 more (of 500, 333 and 222 locals: 19.0, 13.3 and 9.0
// us).  us a step at 3x3x3 against 3x2x2: 40^3 FP32-mixed (512 and 1,152
// tiles) 37 against 45, 44^3 50 against 54, 38^3 FP64 45 against 50; 36^3 (512,
// 968) 45 against 42, 42^3 (729, 1,521) 53 against 49, 32^3 (343, 700) 44
// against 34.
static double rounds(const TileGeom& g, double rho) {
    const double tiles = (double)g.ox * g.oy * g.oz;
    return std::ceil(tiles / kNumCu) * (rho * g.tx * g.ty * g.tz + 25.0);
}

static void choose_tiles(Sim& s) {
    int t[3] = {s.tile_req[0], s.tile_req[1], s.tile_req[2]};
    if (t[0] <= 0 || t[1] <= 0 || t[2] <= 0) {
        if (s.tile_auto[0] <= 0) {
            const double rho = mean_density(s);
            const int T = auto_tile_edge(s.g, s.n);
            const TileGeom cube = make_tile_geom(s.g, T, T, T);
            const int cubes = cube.ox * cube.oy * cube.oz;
            if (rho >= kDenseCell && cubes < kManyTiles) {
                TileShape p = pick_tile(s.g, rho, 1.0, kStageBytes, kLdsBudget, kTileLocals);
                const TileGeom q = make_tile_geom(s.g, p.x, p.y, p.z);
                if (cubes > kNumCu && rounds(cube, rho) < rounds(q, rho)) p = TileShape{T, T, T};
                s.tile_auto[0] = p.x; s.tile_auto[1] = p.y; s.tile_auto[2] = p.z;
            } else {
                // many tiles, or sparse: there the mean density may be far from
                // where the atoms are, and the first window statistics decide
                // (retune_tiles)
                s.tile_auto[0] = s.tile_auto[1] = s.tile_auto[2] = T;
            }
        }
        for (int d = 0; d < 3; ++d) t[d] = s.tile_auto[d];
    }
    const TileGeom g = make_tile_geom(s.g, t[0], t[1], t[2]);
    // sizes of the last tiles tell nothing of larger ones: the rebuild waits for
    // its own, as the first does (k_nlist of windows that outgrow their room)
    if (g.tx > s.tiles.tx || g.ty > s.tiles.ty || g.tz > s.tiles.tz) s.max_window = 0;
    s.tiles = g;
}

// The automatic choice sees only the mean density.  Where atoms crowd into
// part of the box (the DEM gas fills half of it), the largest window can
// outgrow the LDS share of the force pass in use (stage_bytes per slot within
// stage_budget per block); the pass then reads such windows from global
// memory.  From the peak window density of the current tiles this picks the
// tile for the next binning: from the first statistics of a sparse box of
// spheres with a radius (the first rebuild then bins again; 64^3: 38 us a step
// instead of about 100 until the step loop's first rebuild), when the DEM step
// loop's sizes come into force otherwise, and whenever a window overflows.
// Tiles only shrink, and they do not change the results (list order follows
// the cells, not the tiles).  True: the first rebuild should bin again.
bool retune_tiles(Sim& s) {
    if (s.tile_req[0] > 0 && s.tile_req[1] > 0 && s.tile_req[2] > 0) return false;  // explicit tiles
    const TileGeom& T = s.tiles;
    const bool over = (double)(s.max_window + 1) * s.stage_bytes > (double)s.stage_budget;
    const bool sparse = !s.tile_tuned && s.dem_radius > 0.0 && mean_density(s) < kDenseCell;
    const bool dem = s.stage_budget == kDemLdsShare || sparse, first = dem && !s.tile_tuned;
    if ((!over && !first) || s.max_window <= 0) return false;
    s.tile_tuned = 1;
    const double peak = (s.max_window + 1) / ((T.tx + 2.0) * (T.ty + 2.0) * (T.tz + 2.0));
    double cells = 1.0;
    for (int d = 0; d < 3; ++d) cells *= std::max(s.g.len[d] / s.g.spacing, 1.0);
    TileShape p = pick_tile(s.g, peak, std::min(1.0, s.n / (peak * cells)), sparse ? kStageBytes : s.stage_bytes,
                            sparse ? kDemLdsShare : s.stage_budget, dem ? kDemTileLocals : kTileLocals);
    if ((long long)p.x * p.y * p.z > (long long)T.tx * T.ty * T.tz) p = TileShape{T.tx, T.ty, T.tz};
    s.tile_auto[0] = p.x; s.tile_auto[1] = p.y; s.tile_auto[2] = p.z;
    return sparse && (p.x != T.tx || p.y != T.ty || p.z != T.tz);
}

BinArgs bin_args(const Sim& s) {
    const Geom& G = s.g;
    return BinArgs{G.aabb[0], G.aabb[2], G.aabb[4], G.spacing, G.nx, G.ny, G.ncells};
}

// Buffers of the counting sort and the tiles for the current grid, and the
// tile decomposition itself.
void bin_reserve(Sim& s) {
    choose_tiles(s);
    const size_t nc = (size_t)s.g.ncells, nt = (size_t)s.tiles.ntx * s.tiles.nty * s.tiles.ntz, cap = (size_t)std::max(s.cap_all, 1);
    s.cell_count.reserve(sizeof(int) * nc, false, s.stream);
    s.cell_start.reserve(sizeof(int) * (nc + 1), false, s.stream);
    s.tile_start.reserve(sizeof(int) * (nt + 1), false, s.stream);
    s.work_start.reserve(sizeof(int) * (nt + 1), false, s.stream);  // per-tile counts
    s.work.reserve(sizeof(int) * ((size_t)s.n + 1), false, s.stream);
    s.work_k.reserve(sizeof(int) * ((size_t)s.n + 1), false, s.stream);
    s.work_c.reserve(sizeof(int) * ((size_t)s.n + 1), false, s.stream);
    s.gh_w.reserve(sizeof(int) * ((size_t)s.n + 1), false, s.stream);
    s.cell_pair.reserve(sizeof(int2) * cap, false, s.stream);
    s.cell_src.reserve(sizeof(int) * cap, false, s.stream);
    s.cell_parts2.reserve(sizeof(int) * cap, false, s.stream);
    s.cell_inv2.reserve(sizeof(int) * cap, false, s.stream);
    s.spos.reserve((size_t)kMirBytes * cap, true, s.stream);
    s.spos2.reserve((size_t)kMirBytes * cap, false, s.stream);
    s.cell_of.reserve(sizeof(int) * cap, false, s.stream);
    s.cell_slot.reserve(sizeof(int) * cap, false, s.stream);
    if (s.vel_mirrored || s.vel_mirror_wanted || s.dem_loop) {
        s.svel.reserve((size_t)kMirBytes * cap, true, s.stream);
        s.svel2.reserve((size_t)kMirBytes * cap, false, s.stream);
    }
    s.g_ko.reserve(sizeof(int) * cap, false, s.stream);
    s.g_kg.reserve(sizeof(int) * cap, false, s.stream);
}

// Scan, placement and sort behind the histogram of nq source slots (and, when
// with_ghosts, of the ghosts emitted after it): the new CSR (cell_parts,
// cell_inv, cell_src) replaces the last one.
static void bin_sort(Sim& s, int nq, bool mir, bool with_ghosts, bool tiles) {
    const Geom& G = s.g;
    const int nt = 256, gcap = s.cap_all - s.n;
    exclusive_scan_int(s.cell_count.as<int>(), s.cell_start.as<int>(), G.ncells, s.cell_start.as<int>() + G.ncells, s);
    const int nbq = div_up(nq, nt);
    const int nbg = with_ghosts ? std::max(1, std::min(div_up(gcap, nt), 2048)) : 0;
#define TMD_PLACE(M)                                                                                                    \
    hipLaunchKernelGGL(k_bin_place<M>, dim3(nbq + nbg), dim3(nt), 0, s.stream, (const int*)s.cell_of.as<int>(),           \
                       (const int*)s.cell_slot.as<int>(), nq, nbq, (const int*)s.cell_parts.as<int>(),                   \
                       (const int*)s.g_cell.as<int>(), (const int*)s.g_slot.as<int>(), s.n, gcap,                         \
                       (const int*)s.counters.as<int>(), (const int*)s.cell_start.as<int>(), s.cell_pair.as<int2>())
    if (nbq + nbg > 0) { if (mir) TMD_PLACE(true); else TMD_PLACE(false); }
#undef TMD_PLACE
    int* tc = tiles && G.ncells <= kTileAtomicCells ? s.work_start.as<int>() : nullptr;
    if (nq < 4 * G.ncells)  // sparse grid: a thread per cell beats a wavefront per cell
        hipLaunchKernelGGL(k_bin_sort_small, dim3(div_up(G.ncells, nt)), dim3(nt), 0, s.stream,
                           (const int*)s.cell_start.as<int>(), G.ncells, s.n, (const int2*)s.cell_pair.as<int2>(),
                           s.cell_parts2.as<int>(), s.cell_src.as<int>(), s.cell_count.as<int>(), s.cell_inv2.as<int>(), s.tiles, tc);
    else
        hipLaunchKernelGGL(k_bin_sort, dim3(div_up(G.ncells, nt / kWave)), dim3(nt), 0, s.stream,
                           (const int*)s.cell_start.as<int>(), G.ncells, s.n, (const int2*)s.cell_pair.as<int2>(),
                           s.cell_parts2.as<int>(), s.cell_src.as<int>(), s.cell_count.as<int>(), s.cell_inv2.as<int>(), s.tiles, tc);
    TMD_HIP(hipGetLastError());
    std::swap(s.cell_parts, s.cell_parts2);
    std::swap(s.cell_inv, s.cell_inv2);
    s.binned_cells = has_error() ? 0 : G.ncells;
}

// The tail of a rebuild after its histogram: cells, tiles, work order,
// mirrors, ghost indices.  Nothing waits for the host.  False: an error came
// before it, and nothing was done.
bool bin_finish(Sim& s, int nq, bool with_ghosts) {
    if (has_error()) return false;
    const bool mir = s.pos_stale != 0;
    const TileGeom tg = s.tiles;
    const int ntiles = tg.ntx * tg.nty * tg.ntz, gcap = s.cap_all - s.n, nt = 256;
    bin_sort(s, nq, mir, with_ghosts, true);
    FinishArgs a;
    a.g = tg;
    a.ntiles = ntiles;
    a.scanned = ntiles > kTileFlat ? 1 : 0;
    a.n = s.n;
    a.gcap = gcap;
    a.ncells = s.g.ncells;
    a.nbm = div_up(s.cap_all, nt);
    a.ghost_vel = s.dem_loop;
    if (s.g.ncells > kTileAtomicCells)
        hipLaunchKernelGGL(k_tile_count, dim3(div_up(ntiles, 4)), dim3(256), 0, s.stream, (const int*)s.cell_count.as<int>(), tg,
                           ntiles, s.work_start.as<int>());
    if (a.scanned)
        exclusive_scan_int(s.work_start.as<int>(), s.tile_start.as<int>(), ntiles, s.tile_start.as<int>() + ntiles, s);
    // the velocities follow the new order when they live in the mirror, or
    // are wanted there (the fused step loops)
    const bool with_vel = mir || s.vel_mirror_wanted || s.dem_loop;
    const int nbg = std::max(1, std::min(div_up(gcap, nt), 2048));
    const int* pack = s.gh_packed ? s.gh_pack.as<int>() : nullptr;
#define TMD_FINISH(M)                                                                                                   \
    hipLaunchKernelGGL(k_rebuild_finish<M>, dim3(ntiles + a.nbm + nbg), dim3(nt), 0, s.stream, a,                         \
                       (const int*)s.cell_start.as<int>(), (const int*)s.cell_count.as<int>(),                           \
                       (const int*)s.work_start.as<int>(), s.tile_start.as<int>(), (const int*)s.cell_parts.as<int>(),   \
                       (const int*)s.cell_src.as<int>(), (const int*)s.cell_inv.as<int>(), s.work.as<int>(),             \
                       s.work_k.as<int>(), s.work_c.as<int>(), pack, s.gh_w.as<int>(), (const double4*)s.pos.as<double4>(), \
                       (const double4*)s.vel.as<double4>(), CMir{s.spos.as<double>()}, CMir{s.svel.as<double>()},         \
                       Mir{s.spos2.as<double>()}, Mir{with_vel ? s.svel2.as<double>() : nullptr},                        \
                       (const int*)s.g_owner.as<int>(), (const int*)s.g_code.as<int>(), (const int*)s.gh_e.as<int>(),    \
                       s.g_ko.as<int>(), s.g_kg.as<int>(), s.gh_k.as<int2>(), s.counters.as<int>())
    if (mir) TMD_FINISH(true); else TMD_FINISH(false);
#undef TMD_FINISH
    TMD_HIP(hipGetLastError());
    std::swap(s.spos, s.spos2);
    s.mirror_fresh = 1;
    s.ghost_stale = 0;
    if (with_vel) {
        std::swap(s.svel, s.svel2);
        // velocities copied from atom order now live in the mirror
        if (!mir && s.vel_mirror_wanted) s.vel_mirrored = 1;
    }
    s.inv_valid = 1;
    s.gh_valid = s.gh_packed;
    s.windows_valid = 0;
    return true;
}

// k-th local of the cell order <- local parts[k]: positions, velocities,
// forces and masses into the scratch copies
__global__ void k_permute_locals(int n, const int* __restrict__ parts, const double4* __restrict__ pos,
                                 const double4* __restrict__ vel, const double4* __restrict__ force,
                                 const double* __restrict__ mass, double4* __restrict__ pos2, double4* __restrict__ vel2,
                                 double4* __restrict__ force2, double* __restrict__ mass2) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int i = parts[k];
    pos2[k] = pos[i];
    vel2[k] = vel[i];
    force2[k] = force[i];
    mass2[k] = mass[i];
}

// Cell-order reordering of the locals (tmd_set_sort_particles; the
// reference's sort_particles() hook, core/grid.impala:54, 323-356): at the
// PBC wrap of a rebuild, before the ghosts are built, the locals are
// renumbered in cell order, index order inside a cell (a stable counting
// sort), and their positions, velocities, forces and masses move with them.
// The ghost layer built next refers to the new numbering.  (The reference's
// hook renumbers inside distribute_particles, after borders, and copies only
// positions and velocities, so its ghosts keep the old source indices; it is
// compiled out there.)  A local outside the grid after the wrap is an error,
// as in binning.
void sort_locals(Sim& s) {
    if (has_error() || s.n == 0) return;
    // the fused step loop keeps positions and velocities in the mirrors
    sync_pos_from_mirror(s);
    enforce_pbc(s);
    const Geom& G = s.g;
    const size_t n = (size_t)s.n;
    s.sort_buf.reserve((sizeof(double4) * 3 + sizeof(double)) * n, false, s.stream);
    if (has_error()) return;
    s.ng = 0;
    bin_reserve(s);
    if (has_error()) return;
    TMD_HIP(hipMemsetAsync(s.cell_count.p, 0, sizeof(int) * (size_t)G.ncells, s.stream));
    hipLaunchKernelGGL(k_bin_count, dim3(div_up(s.n, 256)), dim3(256), 0, s.stream, (const double4*)s.pos.as<double4>(),
                       bin_args(s), s.n, s.cell_of.as<int>(), s.cell_slot.as<int>(), s.cell_count.as<int>(), s.cell_inv2.as<int>());
    bin_sort(s, s.n, false, false, false);
    int binned = 0;
    TMD_HIP(hipMemcpyAsync(&binned, s.cell_start.as<int>() + G.ncells, sizeof(int), hipMemcpyDeviceToHost, s.stream));
    TMD_HIP(hipStreamSynchronize(s.stream));
    if (has_error()) return;
    if (binned != s.n) {
        set_error(__FILE__, __LINE__, "sort: local atoms outside the cell grid after the periodic wrap (non-finite positions?)");
        return;
    }
    double4* p2 = s.sort_buf.as<double4>();
    double4* v2 = p2 + n;
    double4* f2 = v2 + n;
    double* m2 = reinterpret_cast<double*>(f2 + n);
    hipLaunchKernelGGL(k_permute_locals, dim3(div_up(s.n, 256)), dim3(256), 0, s.stream, s.n, (const int*)s.cell_parts.as<int>(),
                       (const double4*)s.pos.as<double4>(), (const double4*)s.vel.as<double4>(),
                       (const double4*)s.force.as<double4>(), (const double*)s.mass.as<double>(), p2, v2, f2, m2);
    TMD_HIP(hipMemcpyAsync(s.pos.p, p2, sizeof(double4) * n, hipMemcpyDeviceToDevice, s.stream));
    TMD_HIP(hipMemcpyAsync(s.vel.p, v2, sizeof(double4) * n, hipMemcpyDeviceToDevice, s.stream));
    TMD_HIP(hipMemcpyAsync(s.force.p, f2, sizeof(double4) * n, hipMemcpyDeviceToDevice, s.stream));
    TMD_HIP(hipMemcpyAsync(s.mass.p, m2, sizeof(double) * n, hipMemcpyDeviceToDevice, s.stream));
    TMD_HIP(hipGetLastError());
    // every atom-indexed table is stale now
    mirror_invalidate(s);
    s.inv_valid = 0;
    s.gh_valid = s.gh_packed = 0;
    s.windows_valid = 0;
    s.nb_valid = 0;
}

// md_distribute_particles: cells, tiles and mirrors of the current atoms
// (locals and ghosts, in atom order), statistics known on return.
void bin_particles(Sim& s) {
    if (has_error()) return;
    sync_pos_from_mirror(s);
    const int nall = s.n + s.ng;
    mirror_invalidate(s);
    s.inv_valid = 0;
    bin_reserve(s);
    if (has_error()) return;
    const TileGeom tg = s.tiles;
    const int ntiles = tg.ntx * tg.nty * tg.ntz, nt = 256;
    rebuild_zero(s, s.g.ncells, ntiles, s.ng);
    if (nall > 0)
        hipLaunchKernelGGL(k_bin_count, dim3(div_up(nall, nt)), dim3(nt), 0, s.stream, (const double4*)s.pos.as<double4>(),
                           bin_args(s), nall, s.cell_of.as<int>(), s.cell_slot.as<int>(), s.cell_count.as<int>(),
                           s.cell_inv2.as<int>());
    bin_finish(s, nall, false);
    apply_window_stats(s, read_stats(s));
}

}  // namespace tmd
