// On-device periodic ghosts: the single-GPU replacement of the MPI border
// exchange.  For each dimension the "upper" (image -1) and "lower" (image +1)
// ghosts are selected over locals plus the ghosts of earlier dimensions by a
// flag -> tile scan -> stable scatter pass, so the ghost order is the index
// order the reference's CPU mapping produces (comm/comm.impala:528-642 with
// the predicates of comm/comm.impala:105-128 and the image flags of
// comm/lb.impala:88-100).  Every ghost records its immediate source and
// per-direction flag (the reference's send_offsets / send_pbc) and its
// flattened owner + total image, so the per-step refresh is one gather from
// the owner (comm/comm.impala:334-388 without the two-phase lag).
#include "tmd_internal.hpp"
#include "tmd_device.hpp"

namespace tmd {

// Cell of a position (core/grid.impala:406-426): flat index from the floored
// coordinates; non-finite or absurd coordinates are outside the grid (-1).
__device__ __forceinline__ int cell_index(const double4& p, const BinArgs& a) {
    const double fx = floor((p.x - a.xmin) / a.spacing);
    const double fy = floor((p.y - a.ymin) / a.spacing);
    const double fz = floor((p.z - a.zmin) / a.spacing);
    if (fabs(fx) < 1e9 && fabs(fy) < 1e9 && fabs(fz) < 1e9) {
        const int ci = (int)fx, cj = (int)fy, ck = (int)fz;
        const long long flat = ((long long)ck * a.ny + cj) * a.nx + ci;
        if (flat >= 0 && flat < a.ncells) return (int)flat;
    }
    return -1;
}

// ---------------------------------------------------------------------------
// Ghost layer in one sweep.
//
// The reference selects ghosts dimension by dimension, each time over the
// locals and the ghosts made so far.  A ghost differs from its local only in
// the coordinates of the dimensions it was made in, so which ghosts a local
// gets follows from six bits of the local alone: bit 2d, coordinate d above
// the upper select threshold; bit 2d + 1, below the lower one.  Each of the
// 26 sequences (none, upper or lower in x, y and z, not all none) is a class;
// the reference's order is: classes in the order in which the passes reach
// them (class_id), and inside a class the locals' index order.  So a ghost's
// number is the class-major exclusive prefix count, and one scan over the
// (class, block of locals) counts places every ghost of all three passes:
// three launches (count, scan, emit) in place of twelve and no host round
// trip for the totals between them.
//
// a, b, c: 0 none, 1 upper, 2 lower in x, y, z.  The x pass scans the locals
// (classes 0, 1); the y pass scans locals and x ghosts (upper: 2..4, lower:
// 5..7); the z pass scans locals and the eight classes before it (upper:
// 8..16, lower: 17..25).
constexpr int kClasses = 26;
__device__ __forceinline__ int class_id(int a, int b, int c) {
    const int xy = b == 0 ? a - 1 : 2 + (b - 1) * 3 + a;  // -1: none in x and y
    return c == 0 ? xy : 8 + (c - 1) * 9 + xy + 1;
}
constexpr int kGhostBlock = kScanThreads;  // locals per block, one a thread
constexpr int kGhostWaves = kGhostBlock / kWave;
// (class, block) counts that the emitting blocks scan by themselves; more are
// scanned by launches of their own
constexpr int kClassFlat = 4096;

struct FaceArgs {
    int nq, n, wrap;   // source slots; locals (atoms below n)
    double hi_thr[3], lo_thr[3];
    PbcArgs pbc;
    BinArgs bin;
};

// Border bits of every local (and, with BIN, its cell and counting-sort
// slot), after md_enforce_pbc's wrap when asked.  MIR: the locals' positions
// live in the cell-ordered mirror (the fused step loops), which is then read
// and wrapped in place in its own order: coalesced, and neighbouring lanes
// share cells, where a sweep in atom order gathered 24 B records at random
// and copied positions and velocities back to atom order (80^3: 109 us, plus
// 38 us for the binning sweep; this one 33 us).
template <bool MIR, bool BIN>
__global__ void __launch_bounds__(kScanThreads) k_face_bin(double4* __restrict__ pos, const Mir spos,
                                                           const int* __restrict__ parts, FaceArgs a,
                                                           unsigned char* __restrict__ face, int* __restrict__ cell_of,
                                                           int* __restrict__ slot, int* __restrict__ count,
                                                           int* __restrict__ inv) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    const int i = q < a.nq ? (MIR ? parts[q] : q) : a.n;
    int c = -1;
    if (i < a.n) {
        double4 p = MIR ? (double4)spos[q] : pos[q];
        if (a.wrap) {
            const double4 o = p;
            pbc_wrap(p, a.pbc);
            if (p.x != o.x || p.y != o.y || p.z != o.z) {
                if (MIR) spos[q] = p;
                else pos[q] = p;
            }
        }
        const double x[3] = {p.x, p.y, p.z};
        int bits = 0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            bits |= (x[d] > a.hi_thr[d] ? 1 : 0) << (2 * d);
            bits |= (x[d] < a.lo_thr[d] ? 1 : 0) << (2 * d + 1);
        }
        face[i] = (unsigned char)bits;
        if (BIN) {
            c = cell_index(p, a.bin);
            if (c < 0) inv[i] = -1;
        }
    }
    if (BIN) {
        const int sl = wave_cell_slot(c, count);  // all lanes take part
        if (q < a.nq) {
            cell_of[q] = c;
            slot[q] = sl;
        }
    }
}

// Members of class (a, b, c) among the wavefront's locals, from the ballots
// of the six border bits.
struct FaceBallots {
    unsigned long long b[6];
    __device__ __forceinline__ unsigned long long side(int d, int s) const {
        return s == 0 ? ~0ull : (s == 1 ? b[2 * d] : b[2 * d + 1]);
    }
    __device__ __forceinline__ unsigned long long any() const { return b[0] | b[1] | b[2] | b[3] | b[4] | b[5]; }
};

__device__ __forceinline__ FaceBallots face_ballots(int bits) {
    FaceBallots f;
#pragma unroll
    for (int d = 0; d < 6; ++d) f.b[d] = __ballot((bits >> d) & 1);
    return f;
}

// digits of class number `id` (the inverse of class_id), for a lane per class
__device__ __forceinline__ void class_digits(int id, int& a, int& b, int& c) {
    c = id < 8 ? 0 : (id < 17 ? 1 : 2);
    const int e = id < 8 ? id + 1 : (id - 8) % 9;  // 0: none in x and y, else 1 + the xy class
    a = e == 0 ? 0 : (e < 3 ? e : (e - 3) % 3);
    b = e < 3 ? 0 : 1 + (e - 3) / 3;
}

// counts[class * nb + block]: members of each class in each block of locals
__global__ void __launch_bounds__(kScanThreads) k_class_count(const unsigned char* __restrict__ face, int n, int nb,
                                                              int* __restrict__ counts) {
    __shared__ int wc[kGhostWaves][kClasses];
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    int ca = 0, cb = 0, cc = 0;
    class_digits(min(lane, kClasses - 1), ca, cb, cc);
    const int i = blockIdx.x * kGhostBlock + (int)threadIdx.x;
    const FaceBallots f = face_ballots(i < n ? face[i] : 0);
    if (lane < kClasses) wc[wid][lane] = f.any() ? __popcll(f.side(0, ca) & f.side(1, cb) & f.side(2, cc)) : 0;
    __syncthreads();
    if (threadIdx.x < kClasses) {
        int t = 0;
#pragma unroll
        for (int w = 0; w < kGhostWaves; ++w) t += wc[w][threadIdx.x];
        counts[threadIdx.x * nb + blockIdx.x] = t;
    }
}

struct EmitArgs {
    int n, nb, gcap, scanned;    // locals, blocks, ghost slots, counts already scanned
    double whi[3], wlo[3];       // image flag thresholds: world max - s, world min + s
    double len[3];
};

// Every ghost of every local, straight to its slot: position (local + image
// * L), velocity, mass, owner, immediate source and image codes; stores only,
// so a corner atom's 7 classes cost no round trips.  gh_pack / gh_e (may be null): each
// local's entries in the ghost index (first entry * 32 + number of ghosts)
// and each ghost's entry.  Ghosts beyond the capacity are counted, not
// written; the host grows and repeats.
template <bool MIR>
__global__ void __launch_bounds__(kScanThreads) k_ghost_emit(double4* __restrict__ pos, double4* __restrict__ vel,
                                                             double* __restrict__ mass, const CMir spos, const CMir svel,
                                                             const int* __restrict__ inv_src,
                                                             const unsigned char* __restrict__ face,
                                                             const int* __restrict__ counts, EmitArgs a,
                                                             int* __restrict__ g_owner, int* __restrict__ g_src,
                                                             int* __restrict__ g_code, int* __restrict__ gh_pack,
                                                             int* __restrict__ gh_e, int* __restrict__ ctr) {
    __shared__ int flat[kClassFlat];
    __shared__ int sub[kGhostWaves][kClasses];
    __shared__ int entry0;
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    const int blk = blockIdx.x;
    int ca = 0, cb = 0, cc = 0;
    class_digits(min(lane, kClasses - 1), ca, cb, cc);
    const int i = blk * kGhostBlock + (int)threadIdx.x;
    const int bt = i < a.n ? face[i] : 0;
    const FaceBallots F = face_ballots(bt);
    if (lane < kClasses) sub[wid][lane] = __popcll(F.side(0, ca) & F.side(1, cb) & F.side(2, cc));
    // thread c: ghost number of the block's first member of class c, and of the
    // whole class's first one
    int first = 0, cls0 = 0;
    if (a.scanned) {
        if (threadIdx.x < kClasses) {
            first = counts[threadIdx.x * a.nb + blk];
            cls0 = counts[threadIdx.x * a.nb];
        }
    } else {
        // few blocks: each scans the class-major counts itself
        constexpr int kPer = kClassFlat / kScanThreads;
        const int total = kClasses * a.nb, base = (int)threadIdx.x * kPer;
        int v[kPer], sum = 0;
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            v[k] = base + k < total ? counts[base + k] : 0;
            sum += v[k];
        }
        int tot;
        int run = block_exclusive_scan(sum, &tot);
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            flat[base + k] = run;
            run += v[k];
        }
        if (blk == 0 && threadIdx.x == 0) ctr[CT_NGHOST] = tot;
        __syncthreads();
        if (threadIdx.x < kClasses) {
            first = flat[threadIdx.x * a.nb + blk];
            cls0 = flat[threadIdx.x * a.nb];
        }
    }
    if (threadIdx.x < kWave) {
        // the block's first entry of the ghost index: all ghosts of the blocks
        // before it, of every class
        const int before = wave_inclusive_scan(first - cls0);
        if (threadIdx.x == kWave - 1) entry0 = before;
    }
    __syncthreads();
    if (threadIdx.x < kClasses) {
        int run = first;
        for (int q = 0; q < kGhostWaves; ++q) {
            const int t = sub[q][threadIdx.x];
            sub[q][threadIdx.x] = run;
            run += t;
        }
    }
    __syncthreads();
    const unsigned long long below = (1ull << lane) - 1ull;
    const int* base = sub[wid];
    int entry = 0;
    if (gh_pack) {
        const int m = (1 + (bt & 1) + ((bt >> 1) & 1)) * (1 + ((bt >> 2) & 1) + ((bt >> 3) & 1)) *
                          (1 + ((bt >> 4) & 1) + ((bt >> 5) & 1)) - 1;
        int tot;
        entry = entry0 + block_exclusive_scan(m, &tot);
        if (i < a.n) gh_pack[i] = m ? entry * 32 + m : 0;
    }
    if (F.any() == 0) return;  // no border atom in the wavefront
    double4 p = make_double4(0, 0, 0, 0), v = p;
    double ms = 0.0;
    if (bt) {
        if (MIR) {
            const int k = inv_src[i];
            p = spos[k];
            v = svel[k];
        } else {
            p = pos[i];
            v = vel[i];
        }
        ms = mass[i];
    }
    const int fl[3][2] = {{p.x > a.whi[0] ? -1 : 0, p.x < a.wlo[0] ? 1 : 0},
                          {p.y > a.whi[1] ? -1 : 0, p.y < a.wlo[1] ? 1 : 0},
                          {p.z > a.whi[2] ? -1 : 0, p.z < a.wlo[2] ? 1 : 0}};
    // every class with members in this wavefront (uniform loops: the
    // class masks are scalar)
#pragma unroll 1
    for (int c = 0; c < 3; ++c) {
        const unsigned long long mc = F.side(2, c);
#pragma unroll 1
        for (int b = 0; b < 3; ++b) {
            const unsigned long long mb = mc & F.side(1, b);
#pragma unroll 1
            for (int s = 0; s < 3; ++s) {
                const unsigned long long m = mb & F.side(0, s);
                if ((s | b | c) == 0 || m == 0) continue;
                const bool has = (m >> lane) & 1ull;
                const int id = class_id(s, b, c);
                const int g = base[id] + __popcll(m & below);
                const int ix = s == 0 ? 0 : (s == 1 ? fl[0][0] : fl[0][1]);
                const int iy = b == 0 ? 0 : (b == 1 ? fl[1][0] : fl[1][1]);
                const int iz = c == 0 ? 0 : (c == 1 ? fl[2][0] : fl[2][1]);
                double4 q;
                q.x = p.x + a.len[0] * (double)ix;
                q.y = p.y + a.len[1] * (double)iy;
                q.z = p.z + a.len[2] * (double)iz;
                q.w = p.w;
                if (has && g < a.gcap) {
                    // the immediate source: the class without the last pass
                    int src = i;
                    if (c ? (s | b) : (b ? s : 0)) {
                        const int pc = c ? class_id(s, b, 0) : class_id(s, 0, 0);
                        const unsigned long long pm = F.side(0, s) & (c ? F.side(1, b) : ~0ull);
                        src = a.n + base[pc] + __popcll(pm & below);
                    }
                    pos[a.n + g] = q;
                    vel[a.n + g] = v;
                    mass[a.n + g] = ms;
                    g_owner[g] = i;
                    g_src[g] = src;
                    g_code[g] = img_encode(ix, iy, iz) |
                                (img_encode(c || b ? 0 : ix, c ? 0 : (b ? iy : 0), c ? iz : 0) << 8);
                    if (gh_pack) gh_e[g] = entry;
                }
                if (has) ++entry;
            }
        }
    }
}

// Cells and counting-sort slots of the ghosts just made (their number is on
// the device; the launch covers the capacity in strides of whole wavefronts).
__global__ void __launch_bounds__(256) k_ghost_bin(const double4* __restrict__ pos, int n, int gcap, BinArgs bin,
                                                   int* __restrict__ g_cell, int* __restrict__ g_slot,
                                                   int* __restrict__ cell_count, int* __restrict__ inv,
                                                   const int* __restrict__ ctr) {
    const int ng = min(ctr[CT_NGHOST], gcap);
    for (int g0 = blockIdx.x * 256; g0 < ng; g0 += gridDim.x * 256) {
        const int g = g0 + (int)threadIdx.x;
        const int c = g < ng ? cell_index(pos[n + g], bin) : -1;
        const int sl = wave_cell_slot(c, cell_count);  // all lanes take part
        if (g < ng) {
            g_cell[g] = c;
            g_slot[g] = sl;
            if (c < 0) inv[n + g] = -1;
        }
    }
}

// the counters (ng: the ghost count to start from), cell and tile counts
__global__ void k_rebuild_zero(int* __restrict__ cells, int ncells, int* __restrict__ tiles, int ntiles, int* __restrict__ ctr,
                               int ng) {
    const int stride = gridDim.x * blockDim.x, t = blockIdx.x * blockDim.x + threadIdx.x;
    for (int c = t; c < ncells; c += stride) cells[c] = 0;
    for (int c = t; c < ntiles; c += stride) tiles[c] = 0;
    if (t < CT_COUNT) ctr[t] = t == CT_NGHOST ? ng : 0;
}

// one launch clears what a rebuild accumulates (three memsets before it)
void rebuild_zero(Sim& s, int ncells, int ntiles, int ng) {
    const int n = std::max(std::max(ncells, ntiles), 1);
    hipLaunchKernelGGL(k_rebuild_zero, dim3(std::min(div_up(n, 1024), 512)), dim3(256), 0, s.stream, s.cell_count.as<int>(), ncells,
                       s.work_start.as<int>(), ntiles, s.counters.as<int>(), ng);
    TMD_HIP(hipGetLastError());
}

// FRESH refresh: ghost = owner + image * L (bit-identical to the rebuild's
// chained construction because each coordinate receives exactly one shift).
__global__ void k_ghost_refresh(double4* __restrict__ pos, double4* __restrict__ vel, const int* __restrict__ g_owner,
                                const int* __restrict__ g_code, int n, int ng, double L0, double L1, double L2, int with_vel,
                                const int* __restrict__ inv, const Mir spos) {
    int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    const int o = g_owner[g];
    int ix, iy, iz;
    img_decode(g_code[g] & 0xff, ix, iy, iz);
    const double4 p = pos[o];
    double4 q;
    q.x = p.x + L0 * (double)ix;
    q.y = p.y + L1 * (double)iy;
    q.z = p.z + L2 * (double)iz;
    q.w = p.w;
    pos[n + g] = q;
    if (with_vel) vel[n + g] = vel[o];
    if (inv) {
        const int k = inv[n + g];
        if (k >= 0) spos[k] = q;
    }
}

// One pass over locals and ghosts after the force pass advanced the local
// positions: ghost = owner + image * L, and every binned atom's mirror
// entry (inv >= 0) is rewritten.
__global__ void k_step_refresh(double4* __restrict__ pos, const int* __restrict__ g_owner, const int* __restrict__ g_code,
                               int n, int ng, double L0, double L1, double L2, const int* __restrict__ inv,
                               const Mir spos) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n + ng) return;
    double4 q;
    if (i < n) {
        q = pos[i];
    } else {
        const int g = i - n;
        int ix, iy, iz;
        img_decode(g_code[g] & 0xff, ix, iy, iz);
        const double4 p = pos[g_owner[g]];
        q.x = p.x + L0 * (double)ix;
        q.y = p.y + L1 * (double)iy;
        q.z = p.z + L2 * (double)iz;
        q.w = p.w;
        pos[i] = q;
    }
    const int k = inv[i];
    if (k >= 0) spos[k] = q;
}

// Ghost half of k_step_refresh, after a force pass that wrote the advanced
// local positions into the mirror only: ghost = owner + image * L, with the
// owner read from its mirror entry; written to pos and to the ghost's
// mirror entry (owners are locals, so no entry is both read and written).
__global__ void k_ghost_step(double4* __restrict__ pos, const int* __restrict__ g_owner, const int* __restrict__ g_code, int n,
                             int ng, double L0, double L1, double L2, const int* __restrict__ inv, const Mir spos) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    int ix, iy, iz;
    img_decode(g_code[g] & 0xff, ix, iy, iz);
    const double4 p = spos[inv[g_owner[g]]];
    double4 q;
    q.x = p.x + L0 * (double)ix;
    q.y = p.y + L1 * (double)iy;
    q.z = p.z + L2 * (double)iz;
    q.w = p.w;
    pos[n + g] = q;
    const int k = inv[n + g];
    if (k >= 0) spos[k] = q;
}

// Without a ghost index (room for kGhostIndex ghosts or more) the passes that
// move the atoms in the mirrors leave the ghosts' entries to these: owner
// (current in the mirror) + image shift, k_ghost_step's arithmetic.  pos is left
// for sync_pos_from_mirror.
__global__ void k_ghost_step_mirror(const int* __restrict__ g_ko, const int* __restrict__ g_kg,
                                    const int* __restrict__ g_code, int ng, double L0, double L1, double L2,
                                    const Mir spos) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    const int kg = g_kg[g];
    if (kg < 0) return;
    int ix, iy, iz;
    img_decode(g_code[g] & 0xff, ix, iy, iz);
    const double4 p = spos[g_ko[g]];
    double4 q;
    q.x = p.x + L0 * (double)ix;
    q.y = p.y + L1 * (double)iy;
    q.z = p.z + L2 * (double)iz;
    q.w = p.w;
    spos[kg] = q;
}

// DEM step loop: the ghosts' mirror entries from their owners' (position +
// image shift, velocity copied), k_ghost_refresh's arithmetic.
__global__ void k_ghost_step_mirror_v(const int* __restrict__ g_ko, const int* __restrict__ g_kg,
                                      const int* __restrict__ g_code, int ng, double L0, double L1, double L2,
                                      const Mir spos, const Mir svel) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    const int kg = g_kg[g];
    if (kg < 0) return;
    int ix, iy, iz;
    img_decode(g_code[g] & 0xff, ix, iy, iz);
    const int ko = g_ko[g];
    const double4 p = spos[ko];
    double4 q;
    q.x = p.x + L0 * (double)ix;
    q.y = p.y + L1 * (double)iy;
    q.z = p.z + L2 * (double)iz;
    q.w = p.w;
    spos[kg] = q;
    svel[kg] = svel[ko];
}

// a vector of each owner copied to its ghosts (the gradients' force adjoints)
__global__ void k_ghost_copy_mirror(const int* __restrict__ g_ko, const int* __restrict__ g_kg, int ng, const Mir m) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    const int kg = g_kg[g];
    if (kg >= 0) m[kg] = m[g_ko[g]];
}

void ghosts_from_owners(Sim& s, double* mirror, bool shift) {
    if (has_error() || s.ng == 0) return;
    const int nt = 256;
    if (shift)
        hipLaunchKernelGGL(k_ghost_step_mirror, dim3(div_up(s.ng, nt)), dim3(nt), 0, s.stream, (const int*)s.g_ko.as<int>(),
                           (const int*)s.g_kg.as<int>(), (const int*)s.g_code.as<int>(), s.ng, s.g.len[0], s.g.len[1],
                           s.g.len[2], Mir{mirror});
    else
        hipLaunchKernelGGL(k_ghost_copy_mirror, dim3(div_up(s.ng, nt)), dim3(nt), 0, s.stream, (const int*)s.g_ko.as<int>(),
                           (const int*)s.g_kg.as<int>(), s.ng, Mir{mirror});
    TMD_HIP(hipGetLastError());
}

void dem_ghost_step(Sim& s) {
    if (has_error() || s.ng == 0) return;
    const int nt = 256;
    hipLaunchKernelGGL(k_ghost_step_mirror_v, dim3(div_up(s.ng, nt)), dim3(nt), 0, s.stream, (const int*)s.g_ko.as<int>(),
                       (const int*)s.g_kg.as<int>(), (const int*)s.g_code.as<int>(), s.ng, s.g.len[0], s.g.len[1], s.g.len[2],
                       Mir{s.spos.as<double>()}, Mir{s.svel.as<double>()});
    TMD_HIP(hipGetLastError());
}

// REF_LAG refresh (diagnostic): the reference's pack from the immediate
// source (which may be a not-yet-refreshed ghost) then unpack.
__global__ void k_ghost_pack_lag(const double4* __restrict__ pos, const int* __restrict__ g_src, const int* __restrict__ g_code,
                                 int ng, double L0, double L1, double L2, double4* __restrict__ buf) {
    int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    int fx, fy, fz;
    img_decode((g_code[g] >> 8) & 0xff, fx, fy, fz);
    const double4 p = pos[g_src[g]];
    double4 q;
    q.x = p.x + L0 * (double)fx;
    q.y = p.y + L1 * (double)fy;
    q.z = p.z + L2 * (double)fz;
    q.w = p.w;
    buf[g] = q;
}

__global__ void k_ghost_unpack_lag(double4* __restrict__ pos, double4* __restrict__ vel, const int* __restrict__ g_owner,
                                   const double4* __restrict__ buf, int n, int ng, int with_vel, const int* __restrict__ inv,
                                   const Mir spos) {
    int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    pos[n + g] = buf[g];
    if (with_vel) vel[n + g] = vel[g_owner[g]];
    if (inv) {
        const int k = inv[n + g];
        if (k >= 0) spos[k] = buf[g];
    }
}

static void ensure_atom_capacity(Sim& s, int need);

static FaceArgs face_args(const Sim& s, int nq, bool wrap) {
    const Geom& G = s.g;
    FaceArgs fa;
    fa.nq = nq;
    fa.n = s.n;
    fa.wrap = wrap ? 1 : 0;
    for (int d = 0; d < 3; ++d) {
        fa.hi_thr[d] = G.aabb[2 * d + 1] - G.spacing * 2.0;
        fa.lo_thr[d] = G.aabb[2 * d] + G.spacing * 2.0;
    }
    fa.pbc = pbc_args(s);
    fa.bin = bin_args(s);
    return fa;
}

// Enqueue the ghost build: border bits, class counts, (scan,) emit.  bin: the
// counting sort's histogram of locals and ghosts is taken in the same sweeps
// (the tail of a rebuild, bin_finish, goes on from there).  Nothing waits for
// the host: the ghost count stays in the counters.
void enqueue_ghosts(Sim& s, bool wrap, bool bin) {
    if (has_error()) return;
    // positions and velocities move together between atom order and mirror
    if ((s.pos_stale != 0) != (s.vel_mirrored != 0)) sync_pos_from_mirror(s);
    const bool mir = s.pos_stale != 0;
    s.ghost_pos_stale = 0;  // the ghosts are made anew
    s.ng = 0;
    s.gh_valid = 0;
    if (!mir) {
        s.inv_valid = 0;
        mirror_invalidate(s);
    }
    if (s.n == 0) return;
    const Geom& G = s.g;
    const int gcap = s.cap_all - s.n;
    const int nq = mir ? s.nbinned : s.n;
    const int nb = div_up(s.n, kGhostBlock);
    s.face.reserve((size_t)std::max(s.cap_all, s.n), false, s.stream);
    const int ncls = kClasses * nb;
    s.cls.reserve(sizeof(int) * 2 * (size_t)ncls, false, s.stream);  // counts, and their scan
    s.gh_pack.reserve(sizeof(int) * (size_t)s.n, false, s.stream);
    s.gh_e.reserve(sizeof(int) * (size_t)std::max(gcap, 1), false, s.stream);
    s.gh_k.reserve(sizeof(int2) * (size_t)std::max(gcap, 1), false, s.stream);
    if (bin) {
        s.g_cell.reserve(sizeof(int) * (size_t)std::max(gcap, 1), false, s.stream);
        s.g_slot.reserve(sizeof(int) * (size_t)std::max(gcap, 1), false, s.stream);
        bin_reserve(s);
    }
    if (has_error()) return;
    int* ctr = s.counters.as<int>();
    const int ntiles = s.tiles.ntx * s.tiles.nty * s.tiles.ntz;
    rebuild_zero(s, bin ? G.ncells : 0, bin ? ntiles : 0, 0);
    const FaceArgs fa = face_args(s, nq, wrap);
    const dim3 gq(div_up(nq, kScanThreads)), gb(nb), blk(kScanThreads);
#define TMD_FACE(M, B)                                                                                                   \
    hipLaunchKernelGGL((k_face_bin<M, B>), gq, blk, 0, s.stream, s.pos.as<double4>(), Mir{s.spos.as<double>()},            \
                       (const int*)s.cell_parts.as<int>(), fa, s.face.as<unsigned char>(), s.cell_of.as<int>(),           \
                       s.cell_slot.as<int>(), s.cell_count.as<int>(), s.cell_inv2.as<int>())
    if (mir) { if (bin) TMD_FACE(true, true); else TMD_FACE(true, false); }
    else { if (bin) TMD_FACE(false, true); else TMD_FACE(false, false); }
#undef TMD_FACE
    hipLaunchKernelGGL(k_class_count, gb, blk, 0, s.stream, (const unsigned char*)s.face.as<unsigned char>(), s.n, nb,
                       s.cls.as<int>());
    EmitArgs ea;
    ea.n = s.n;
    ea.nb = nb;
    ea.gcap = gcap;
    ea.scanned = ncls > kClassFlat ? 1 : 0;
    for (int d = 0; d < 3; ++d) {
        ea.whi[d] = G.world[2 * d + 1] - G.spacing;
        ea.wlo[d] = G.world[2 * d] + G.spacing;
        ea.len[d] = G.len[d];
    }
    const int* counts = s.cls.as<int>();
    if (ea.scanned) {
        exclusive_scan_int(counts, s.cls.as<int>() + ncls, ncls, ctr + CT_NGHOST, s);
        counts += ncls;
    }
    s.gh_packed = gcap < (s.gh_limit > 0 ? s.gh_limit : kGhostIndex);
    int* pack = s.gh_packed ? s.gh_pack.as<int>() : nullptr;
#define TMD_EMIT(M)                                                                                                      \
    hipLaunchKernelGGL(k_ghost_emit<M>, gb, blk, 0, s.stream, s.pos.as<double4>(), s.vel.as<double4>(),                    \
                       s.mass.as<double>(), CMir{s.spos.as<double>()}, CMir{s.svel.as<double>()},                         \
                       (const int*)s.cell_inv.as<int>(), (const unsigned char*)s.face.as<unsigned char>(), counts, ea,    \
                       s.g_owner.as<int>(), s.g_src.as<int>(), s.g_code.as<int>(), pack, s.gh_e.as<int>(), ctr)
    if (mir) TMD_EMIT(true); else TMD_EMIT(false);
#undef TMD_EMIT
    if (bin)
        hipLaunchKernelGGL(k_ghost_bin, dim3(std::max(1, std::min(div_up(gcap, 256), 2048))), dim3(256), 0, s.stream,
                           (const double4*)s.pos.as<double4>(), s.n, gcap, fa.bin, s.g_cell.as<int>(), s.g_slot.as<int>(),
                           s.cell_count.as<int>(), s.cell_inv2.as<int>(), (const int*)ctr);
    TMD_HIP(hipGetLastError());
}

// md_borders: the ghost layer alone, its size known on return.
void build_ghosts(Sim& s) {
    for (int attempt = 0; attempt < 3 && !has_error(); ++attempt) {
        enqueue_ghosts(s, false, false);
        if (has_error() || s.n == 0) return;
        const int* st = read_stats(s);
        if (!st) return;
        if (st[CT_NGHOST] <= s.cap_all - s.n) {
            s.ng = st[CT_NGHOST];
            return;
        }
        ensure_atom_capacity(s, s.n + st[CT_NGHOST]);
    }
}

// a rebuild found more ghosts than there is room for
void grow_ghosts(Sim& s, int ng) { ensure_atom_capacity(s, s.n + ng); }

void refresh_ghosts(Sim& s) {
    if (has_error() || s.ng == 0) return;
    const int with_vel = 1;
    const int nt = 256;
    if (s.ghost_mode == GHOST_REF_LAG) {
        s.gbuf.reserve(sizeof(double4) * (size_t)s.ng, false, s.stream);
        hipLaunchKernelGGL(k_ghost_pack_lag, dim3(div_up(s.ng, nt)), dim3(nt), 0, s.stream, (const double4*)s.pos.as<double4>(),
                           (const int*)s.g_src.as<int>(), (const int*)s.g_code.as<int>(), s.ng, s.g.len[0], s.g.len[1], s.g.len[2],
                           s.gbuf.as<double4>());
        hipLaunchKernelGGL(k_ghost_unpack_lag, dim3(div_up(s.ng, nt)), dim3(nt), 0, s.stream, s.pos.as<double4>(), s.vel.as<double4>(),
                           (const int*)s.g_owner.as<int>(), (const double4*)s.gbuf.as<double4>(), s.n, s.ng, with_vel,
                           s.inv_valid ? (const int*)s.cell_inv.as<int>() : nullptr, Mir{s.spos.as<double>()});
    } else {
        hipLaunchKernelGGL(k_ghost_refresh, dim3(div_up(s.ng, nt)), dim3(nt), 0, s.stream, s.pos.as<double4>(), s.vel.as<double4>(),
                           (const int*)s.g_owner.as<int>(), (const int*)s.g_code.as<int>(), s.n, s.ng, s.g.len[0], s.g.len[1],
                           s.g.len[2], with_vel, s.inv_valid ? (const int*)s.cell_inv.as<int>() : nullptr,
                           Mir{s.spos.as<double>()});
    }
    TMD_HIP(hipGetLastError());
}

// pos[parts[k]] = mirror[k] for the locals of the cell CSR (when pos is
// given), and likewise the velocities from their mirror order (when svel is)
__global__ void k_unmirror(const CMir spos, const int* __restrict__ parts, int nbinned, int n,
                           double4* __restrict__ pos, const CMir svel, double4* __restrict__ vel) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nbinned) return;
    const int j = parts[k];
    if (j < n) {
        if (pos) pos[j] = spos[k];
        if (svel.p) vel[j] = svel[k];
    }
}

// Positions (and velocities) of the fused step loop back into atom order.
void sync_pos_from_mirror(Sim& s) {
    if (has_error()) return;
    if (s.ghost_pos_stale) {
        // the ghosts' positions in pos, from their owners in the mirror
        if (s.ng > 0)
            hipLaunchKernelGGL(k_ghost_step, dim3(div_up(s.ng, 256)), dim3(256), 0, s.stream, s.pos.as<double4>(),
                               (const int*)s.g_owner.as<int>(), (const int*)s.g_code.as<int>(), s.n, s.ng, s.g.len[0],
                               s.g.len[1], s.g.len[2], (const int*)s.cell_inv.as<int>(), Mir{s.spos.as<double>()});
        TMD_HIP(hipGetLastError());
        s.ghost_pos_stale = 0;
    }
    if (!s.pos_stale && !s.vel_mirrored) return;
    const int nt = 256;
    if (s.nbinned > 0)
        hipLaunchKernelGGL(k_unmirror, dim3(div_up(s.nbinned, nt)), dim3(nt), 0, s.stream, CMir{s.spos.as<double>()},
                           (const int*)s.cell_parts.as<int>(), s.nbinned, s.n,
                           s.pos_stale ? s.pos.as<double4>() : (double4*)nullptr,
                           CMir{s.vel_mirrored ? s.svel.as<double>() : nullptr}, s.vel.as<double4>());
    TMD_HIP(hipGetLastError());
    s.pos_stale = 0;
    s.vel_mirrored = 0;
}

// A rebuild that ended in an error (atoms outside the grid, no memory) leaves
// the locals in atom order, wrapped, with no cells and no lists; the ghosts are
// those it made.  mir: they lived in the mirrors, of nq slots.  binned: the new
// binning took the place of the one whose slots these are, which is then in the
// second buffers, whole; the new one may lack the atoms that the error is about.
// The error is set already, so this launches by itself.
void rebuild_failed(Sim& s, bool mir, bool binned, int nq) {
    if (mir && nq > 0)
        hipLaunchKernelGGL(k_unmirror, dim3(div_up(nq, 256)), dim3(256), 0, s.stream,
                           CMir{(binned ? s.spos2 : s.spos).as<double>()},
                           (const int*)(binned ? s.cell_parts2 : s.cell_parts).as<int>(), nq, s.n, s.pos.as<double4>(),
                           CMir{(binned ? s.svel2 : s.svel).as<double>()}, s.vel.as<double4>());
    TMD_HIP(hipGetLastError());
    mirror_invalidate(s);
    s.pos_stale = 0;
    s.vel_mirrored = 0;
    s.inv_valid = 0;
    s.gh_valid = 0;
    s.nbinned = 0;
    s.windows_valid = 0;
    s.nb_valid = 0;
}

// velocities of the locals from atom order (vel) to mirror order (svel)
__global__ void k_vel_mirror(const int* __restrict__ work, const int* __restrict__ wk, int n, const double4* __restrict__ vel,
                             const Mir svel) {
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w < n) svel[wk[w]] = vel[work[w]];
}

// The fused step loop keeps the locals' velocities in mirror order (the
// force pass then reads and writes them with the same coalesced index as the
// positions); sync_pos_from_mirror returns them to atom order.
void mirror_velocities(Sim& s) {
    if (has_error() || s.n == 0 || s.vel_mirrored) return;
    s.svel.reserve((size_t)kMirBytes * (size_t)std::max(s.nbinned, 1), false, s.stream);
    if (has_error()) return;
    const int nt = 256;
    hipLaunchKernelGGL(k_vel_mirror, dim3(div_up(s.n, nt)), dim3(nt), 0, s.stream, (const int*)s.work.as<int>(),
                       (const int*)s.work_k.as<int>(), s.n, (const double4*)s.vel.as<double4>(), Mir{s.svel.as<double>()});
    TMD_HIP(hipGetLastError());
    s.vel_mirrored = 1;
}

void step_refresh(Sim& s) {
    if (has_error() || s.n + s.ng == 0) return;
    const int nt = 256;
    if (s.ghost_stale && s.pos_stale) {
        // the last pass moved the locals in the mirror: the ghosts there only
        // (pos at the end)
        ghosts_from_owners(s, s.spos.as<double>(), true);
        s.ghost_pos_stale = 1;
    } else if (!s.inv_valid || s.ghost_mode != GHOST_FRESH) {
        s.ghost_stale = 0;
        refresh_ghosts(s);
        return;
    } else {
        hipLaunchKernelGGL(k_step_refresh, dim3(div_up(s.n + s.ng, nt)), dim3(nt), 0, s.stream, s.pos.as<double4>(),
                           (const int*)s.g_owner.as<int>(), (const int*)s.g_code.as<int>(), s.n, s.ng, s.g.len[0], s.g.len[1],
                           s.g.len[2], (const int*)s.cell_inv.as<int>(), Mir{s.spos.as<double>()});
    }
    TMD_HIP(hipGetLastError());
    s.ghost_stale = 0;
    s.mirror_fresh = 1;
}

// Grow every per-atom array (locals + ghosts) to hold `need` atoms,
// preserving contents.  Ghost-table arrays are indexed by ghost number.
static void ensure_atom_capacity(Sim& s, int need) {
    if (need <= s.cap_all) return;
    int cap = need + need / 5 + 1024;
    s.pos.reserve(sizeof(double4) * (size_t)cap, true, s.stream);
    s.vel.reserve(sizeof(double4) * (size_t)cap, true, s.stream);
    s.mass.reserve(sizeof(double) * (size_t)cap, true, s.stream);
    s.g_owner.reserve(sizeof(int) * (size_t)cap, true, s.stream);
    s.g_src.reserve(sizeof(int) * (size_t)cap, true, s.stream);
    s.g_code.reserve(sizeof(int) * (size_t)cap, true, s.stream);
    s.cell_of.reserve(sizeof(int) * (size_t)cap, false, s.stream);
    s.cell_slot.reserve(sizeof(int) * (size_t)cap, false, s.stream);
    // a repeated rebuild may read the locals through the last binning
    s.cell_parts.reserve(sizeof(int) * (size_t)cap, true, s.stream);
    s.cell_inv.reserve(sizeof(int) * (size_t)cap, true, s.stream);
    s.spos.reserve((size_t)kMirBytes * (size_t)cap, true, s.stream);
    s.svel.reserve((size_t)kMirBytes * (size_t)cap, true, s.stream);
    s.gh_valid = 0;
    if (!has_error()) s.cap_all = cap;  // as in alloc_atoms
}

// End of the DEM mirror phase: the locals' positions and velocities back to
// atom order, then the ghosts' from their owners.
void dem_unmirror(Sim& s) {
    if (has_error() || !s.dem_mirrored) return;
    s.dem_mirrored = 0;
    const int nt = 256;
    if (s.nbinned > 0)
        hipLaunchKernelGGL(k_unmirror, dim3(div_up(s.nbinned, nt)), dim3(nt), 0, s.stream, CMir{s.spos.as<double>()},
                           (const int*)s.cell_parts.as<int>(), s.nbinned, s.n, s.pos.as<double4>(),
                           CMir{s.svel.as<double>()}, s.vel.as<double4>());
    TMD_HIP(hipGetLastError());
    refresh_ghosts(s);  // also writes the ghosts' mirror entries, so the mirror stays that of pos
}

}  // namespace tmd
