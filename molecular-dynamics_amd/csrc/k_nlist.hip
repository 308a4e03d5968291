// Tile windows, the cell-ordered position mirror, and the Verlet neighbour
// lists (full and half) as 16-bit offsets into each tile's window
// (tmd_window.hpp).
//
// List build: one block per tile, one lane per local atom of the tile.  The
// block stages its window (FP32 position relative to the tile, atom index)
// into LDS; each lane walks its 27-cell stencil as 9 rows of 3 cells inside
// the window, in the reference's order -- stencil (z, y, x), then cell order
// (core/neighborlist.impala:1-78) -- and keeps a candidate when
// `rsq <= r_nb^2` in FP64 without contraction, decided in FP32 where that is
// certain (nlist_atom), so the sets are bit-exact with the reference.  Half lists keep j < i among locals (the reference's
// filter) plus, by default, every ghost.
#include "tmd_internal.hpp"
#include "tmd_pair.hpp"

namespace tmd {

// Cell-ordered position mirror: spos[k] = pos[parts[k]] (locals and ghosts);
// with svel, also the locals' velocities in mirror order.
__global__ void k_mirror(const double4* __restrict__ pos, const int* __restrict__ parts, const int* __restrict__ nbinned,
                         const Mir spos, int n, const double4* __restrict__ vel, const Mir svel,
                         int vel_ghosts) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= *nbinned) return;
    const int j = parts[k];
    spos[k] = pos[j];
    if (svel.p && (j < n || vel_ghosts)) svel[k] = vel[j];
}

// Per-atom inputs come in work order (mirror index work_k, cell work_c), so
// a wavefront's reads of them are contiguous.
template <bool HALF, int SLOTS>
__global__ void __launch_bounds__(kMaxTileThreads) k_nlist(const CMir spos, const int* __restrict__ work_k,
                                                        const int* __restrict__ work_c,
                                                        const int* __restrict__ start, const int* __restrict__ parts,
                                                        const int* __restrict__ work, const int* __restrict__ tile_start,
                                                        NbArgs a, int* __restrict__ nb_count, nb_t* __restrict__ nb_list,
                                                        int* __restrict__ nb_count2, nb_t* __restrict__ nb_list2,
                                                        int* __restrict__ overflow) {
    extern __shared__ double dyn[];
    const int tile = block_tile(blockIdx.x, a.g);
    const int w0 = tile_start[tile], nloc = tile_start[tile + 1] - w0;
    if (nloc == 0) return;
    __shared__ TileWin W;
    __shared__ unsigned maxr;
    if (threadIdx.x == 0) maxr = 0u;
    ListWin L = list_win(dyn, a.wcap, a.g, spos[work_k[w0 + nloc / 2]]);
    tile_window(tile, start, a.g, W);
    stage_row_starts(W, start, a.g, L.cst);
    const bool staged = stage_list_window<HALF>(W, a.wcap, spos, parts, a.cut2, L, &maxr);
    for (int at = threadIdx.x; at < nloc; at += blockDim.x) {
        const int w = w0 + at;
        const int i = HALF ? work[w] : 0;
        const int k = work_k[w];
        int cnt2 = 0;
        const int cnt = staged ? nlist_atom<HALF, true, SLOTS>(i, w, work_c[w], k, spos[k], a, W, L, spos, parts, nb_list, nb_list2, cnt2)
                               : nlist_atom<HALF, false, SLOTS>(i, w, work_c[w], k, spos[k], a, W, L, spos, parts, nb_list, nb_list2, cnt2);
        nb_count[w] = cnt;
        if (HALF) nb_count2[w] = cnt2;
        const int most = max(cnt, cnt2);
        if (most > a.cap) atomicMax(overflow, most);
    }
}

// ---------------------------------------------------------------------------
// Threads per tile block: one lane per local of the fullest tile (no tile
// takes a second pass), in whole wavefronts, at most kAutoTileThreads so that
// two blocks of the tile kernels (up to 80 VGPRs: 6 waves per SIMD) share a
// CU.  An explicit choice (tmd_set_tile_threads) overrides.
int tile_block_threads(int requested, int max_locals) {
    if (requested > 0) return requested;
    const int t = (std::max(max_locals, 1) + kWave - 1) / kWave * kWave;
    return std::min(std::max(t, kTileThreads / 2), kAutoTileThreads);
}

int window_cap(const Sim& s) { return std::min(s.max_window + 1, kLdsBudget / kStageBytes); }  // + sentinel slot
int window_cap_pos(const Sim& s) { return std::min(s.max_window + 1, kLdsBudget / kPosStageBytes); }

// the counters, then the number of this read, into pinned host memory
__global__ void k_publish(const int* __restrict__ ctr, int* __restrict__ host, int seq) {
    if (threadIdx.x < CT_COUNT) __hip_atomic_store(&host[threadIdx.x], ctr[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(&host[CT_COUNT], seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The counters of a rebuild on the host, after everything queued so far;
// nullptr after an error.  The last kernel stores them into pinned memory and
// the host watches for its number there: a copy and a stream synchronisation
// took 36 us from the end of the list build to the next force pass, of which
// the copy kernel is 4 and the wake-up most of the rest.  The stream is
// asked now and then, so a failed launch ends the wait as an error.
const int* read_stats(Sim& s) {
    if (has_error()) return nullptr;
    if (!s.h_stats) {
        TMD_HIP(hipHostMalloc(reinterpret_cast<void**>(&s.h_stats), (CT_COUNT + 1) * sizeof(int)));
        if (has_error()) return nullptr;
        s.h_stats[CT_COUNT] = s.stats_seq;
    }
    const int seq = ++s.stats_seq;
    hipLaunchKernelGGL(k_publish, dim3(1), dim3(kWave), 0, s.stream, (const int*)s.counters.as<int>(), s.h_stats, seq);
    TMD_HIP(hipGetLastError());
    if (has_error()) return nullptr;
    for (unsigned spin = 1; __atomic_load_n(&s.h_stats[CT_COUNT], __ATOMIC_ACQUIRE) != seq; ++spin) {
        if (spin % 4096 != 0) {
            __builtin_ia32_pause();
            continue;
        }
        const hipError_t e = hipStreamQuery(s.stream);
        if (e == hipErrorNotReady) continue;
        // done or failed: synchronising reports which
        TMD_HIP(hipStreamSynchronize(s.stream));
        if (!has_error() && __atomic_load_n(&s.h_stats[CT_COUNT], __ATOMIC_ACQUIRE) != seq)
            set_error(__FILE__, __LINE__, "rebuild: the counters did not reach the host");
        break;
    }
    return has_error() ? nullptr : s.h_stats;
}

static bool all_placed(const Sim& s, const int* st) {
    if (st[CT_PLACED] == s.n) return true;
    char msg[200];
    snprintf(msg, sizeof msg,
             "%d local atoms lie outside the periodic box or the cell grid (non-finite or unwrapped positions; "
             "md_enforce_pbc wraps them)",
             s.n - st[CT_PLACED]);
    set_error(__FILE__, __LINE__, msg);
    return false;
}

// The window statistics (locals placed, binned atoms, largest window, most
// locals in a tile) decide the LDS size and block size of the tile kernels.
bool apply_window_stats(Sim& s, const int* st) {
    if (!st || !all_placed(s, st)) return false;
    s.nbinned = st[CT_BINNED];
    s.max_window = st[CT_MAXWIN];
    s.max_locals = st[CT_MAXLOC];
    s.tile_threads = tile_block_threads(s.tile_threads_req, st[CT_MAXLOC]);
    const bool again = retune_tiles(s);
    if (s.max_window > kWinMax) {
        char msg[200];
        snprintf(msg, sizeof msg, "a tile neighbourhood holds %d atoms, beyond the 16-bit window range (%d)", s.max_window,
                 kWinMax);
        set_error(__FILE__, __LINE__, msg);
        return false;
    }
    if (kLdsBudget > s.lds_limit) {
        set_error(__FILE__, __LINE__, "device LDS per block is below the window budget");
        return false;
    }
    s.windows_valid = 1;
    return again;
}

// DEM step loop: positions and velocities of every binned atom, ghosts
// included, into the mirrors (spos, svel); the force pass reads them there.
void dem_mirror(Sim& s) {
    const int bound = s.n + s.ng;
    if (has_error() || bound == 0) return;
    s.svel.reserve((size_t)kMirBytes * (size_t)bound, false, s.stream);
    s.svel2.reserve((size_t)kMirBytes * (size_t)bound, false, s.stream);
    s.spos2.reserve((size_t)kMirBytes * (size_t)bound, false, s.stream);
    if (has_error()) return;
    const int nt = 256;
    hipLaunchKernelGGL(k_mirror, dim3(div_up(bound, nt)), dim3(nt), 0, s.stream, (const double4*)s.pos.as<double4>(),
                       (const int*)s.cell_parts.as<int>(), (const int*)(s.cell_start.as<int>() + s.g.ncells),
                       Mir{s.spos.as<double>()}, s.n, (const double4*)s.vel.as<double4>(), Mir{s.svel.as<double>()}, 1);
    TMD_HIP(hipGetLastError());
    s.mirror_fresh = 1;
    s.dem_mirrored = 1;
}

void refresh_mirror(Sim& s) {
    // the grid covers every atom that can be binned; the kernel stops at the
    // binned count on the device (the host's may still be pending)
    const int bound = s.n + s.ng;
    if (has_error() || bound == 0) return;
    const int nt = 256;
    // inside the fused step loop the velocities follow the new order too
    const bool with_vel = s.vel_mirror_wanted && !s.vel_mirrored && s.n > 0;
    if (with_vel) {
        s.svel.reserve((size_t)kMirBytes * (size_t)bound, false, s.stream);
        if (has_error()) return;
    }
    hipLaunchKernelGGL(k_mirror, dim3(div_up(bound, nt)), dim3(nt), 0, s.stream, (const double4*)s.pos.as<double4>(),
                       (const int*)s.cell_parts.as<int>(), (const int*)(s.cell_start.as<int>() + s.g.ncells),
                       Mir{s.spos.as<double>()}, s.n, (const double4*)s.vel.as<double4>(),
                       Mir{with_vel ? s.svel.as<double>() : nullptr}, 0);
    TMD_HIP(hipGetLastError());
    s.mirror_fresh = 1;
    if (with_vel) s.vel_mirrored = 1;
}

// A window that outgrows its room by one atom is read from the mirror, which
// takes its block several times as long (6^3 cells, FP64: 174 us a build, with
// an eighth of room 48; 23.2 and 20.1 us a step, at 16^3 mixed 21.6 and 18.2).
constexpr int kWindowGrowth = 16;

void build_neighbor_lists(Sim& s, int half, double cutoff) {
    if (has_error()) return;
    TMD_REQUIRE(s.windows_valid, "md_assemble_neighborlists: cells not binned (call md_distribute_particles first)");
    if (has_error()) return;
    int* counters = s.counters.as<int>();
    if (!s.mirror_fresh) refresh_mirror(s);
    const int ntiles = s.tiles.ntx * s.tiles.nty * s.tiles.ntz;
    // a rebuild has just cleared the counters
    for (bool cleared = s.windows_pending != 0;; cleared = false) {
        s.nb_cap = (s.nb_cap + 7) & ~7;
        const int ntile64 = div_up(s.n > 0 ? s.n : 1, 64);
        s.nb_stride = ntile64 * 64;
        s.nb_count.reserve(sizeof(int) * (size_t)s.nb_stride, false, s.stream);
        s.nb_list.reserve(sizeof(nb_t) * (size_t)ntile64 * 64 * (size_t)s.nb_cap, false, s.stream);
        if (half) {
            // the complementary column of every half list (same layout)
            s.nb_count2.reserve(sizeof(int) * (size_t)s.nb_stride, false, s.stream);
            s.nb_list2.reserve(sizeof(nb_t) * (size_t)ntile64 * 64 * (size_t)s.nb_cap, false, s.stream);
        }
        if (has_error()) return;
        if (!cleared) rebuild_zero(s, 0, 0, s.ng);
        // the rebuild before's largest window, with room for it to grow
        const int grow = s.windows_pending ? s.max_window / kWindowGrowth + 16 : 0;
        const ListLds l = list_lds(s.max_window + grow + kListPad, row_starts_bytes(s.tiles), s.tile_threads / kWave,
                                     half);
        NbArgs a{s.n, s.nb_cap, half, s.half_mode, l.wcap, cutoff * cutoff, s.tiles};
        if (s.n > 0) {
#define TMD_NLIST(H, R)                                                                                                   \
    hipLaunchKernelGGL((k_nlist<H, R>), dim3(ntiles), dim3(l.waves * kWave), l.bytes, s.stream, CMir{s.spos.as<double>()},           \
                       (const int*)s.work_k.as<int>(), (const int*)s.work_c.as<int>(),                                      \
                       (const int*)s.cell_start.as<int>(), (const int*)s.cell_parts.as<int>(), (const int*)s.work.as<int>(), \
                       (const int*)s.tile_start.as<int>(), a, s.nb_count.as<int>(), s.nb_list.as<nb_t>(), \
                       s.nb_count2.as<int>(), s.nb_list2.as<nb_t>(), counters + CT_LIST)
            if (half) TMD_NLIST(true, 16); else if (l.slots == 32) TMD_NLIST(false, 32); else TMD_NLIST(false, 16);
#undef TMD_NLIST
        }
        TMD_HIP(hipGetLastError());
        const int* st = read_stats(s);
        if (!st) return;
        const int over = st[CT_LIST];
        if (s.windows_pending) {
            // the statistics of the rebuild that queued this list build
            s.windows_pending = 0;
            if (st[CT_NGHOST] > s.cap_all - s.n) {
                // incomplete ghosts: the rebuild grows and repeats, from the
                // locals of this binning
                if (!all_placed(s, st)) return;
                s.ghosts_missing = st[CT_NGHOST];
                s.nbinned = st[CT_BINNED];
                return;
            }
            s.ng = st[CT_NGHOST];
            apply_window_stats(s, st);
        }
        if (has_error()) return;
        if (over > 0) {
            s.nb_cap = over * 2;
            continue;
        }
        break;
    }
    s.nb_half = half;
    s.nb_valid = 1;
}

// A whole rebuild (wrap when asked, ghosts, cells, tiles, mirrors, lists)
// with one host synchronisation, at its end: the ghost count stays on the
// device until then, and the list build runs with the window and block sizes
// of the rebuild before (a larger window is then read from the mirror, a
// fuller tile takes a second pass of its block).  The first rebuild has no
// such sizes and waits for its own before the lists.
void rebuild_lists(Sim& s, bool wrap, int half, double cutoff) {
    if (has_error()) return;
    s.nb_valid = 0;
    if (s.n == 0) {
        bin_particles(s);
        build_neighbor_lists(s, half, cutoff);
        return;
    }
    for (int attempt = 0; attempt < 4; ++attempt) {
        hipEvent_t ev = nullptr;
        s.ghosts_missing = 0;
        s.timer.begin(K_BORDERS, s.stream, &ev);
        enqueue_ghosts(s, wrap && attempt == 0, true);
        s.timer.end(K_BORDERS, s.stream, ev);
        // the locals' places: mirrors, or atom order
        const bool mir = s.pos_stale != 0;
        const int nq = mir ? s.nbinned : s.n;
        s.timer.begin(K_BIN, s.stream, &ev);
        const bool binned = bin_finish(s, nq, true);
        s.timer.end(K_BIN, s.stream, ev);
        bool again = false;
        if (!has_error() && s.max_window > 0) {
            s.windows_pending = 1;
            s.windows_valid = 1;
        } else if (const int* st = read_stats(s)) {
            if (st[CT_NGHOST] > s.cap_all - s.n) s.ghosts_missing = st[CT_NGHOST];
            else s.ng = st[CT_NGHOST];
            // also the binned count that a repeat reads the mirrors by
            const bool tiles = apply_window_stats(s, st);
            again = tiles && !mir && !s.ghosts_missing && attempt < 2;
        }
        if (!has_error() && !again && !s.ghosts_missing) {
            s.timer.begin(K_NEIGHBOR, s.stream, &ev);
            build_neighbor_lists(s, half, cutoff);
            s.timer.end(K_NEIGHBOR, s.stream, ev);
        }
        s.windows_pending = 0;
        if (!has_error() && s.ghosts_missing && attempt == 3)
            set_error(__FILE__, __LINE__, "rebuild: the ghosts keep outgrowing their room");
        if (has_error()) {
            rebuild_failed(s, mir, binned, nq);
            return;
        }
        if (!again && !s.ghosts_missing) return;
        s.max_window = 0;  // again: with the new tiles' sizes
        if (s.ghosts_missing) grow_ghosts(s, s.ghosts_missing);
    }
}

}  // namespace tmd
