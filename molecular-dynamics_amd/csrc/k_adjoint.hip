// Differentiable LJ trajectories: forward loss and its hand-written adjoint.
//
// Loss of a velocity-Verlet trajectory of T steps from (x0, v0):
//   L = (Ubar - U*)^2 + (Pbar - P*)^2,
//   Ubar = (1/T) sum_{t=1..T} PE(x_t) / N,
//   Pbar = (1/T) sum_{t=1..T} (sum v_t^2 + W(x_t)) / (3V),   W = sum_pairs r.F.
// Gradients with respect to eps, sigma and x0.  The pair potential is the
// smoothly truncated LJ of tmd_lj.hpp (force and its derivative vanish at
// rc), so the discrete trajectory is differentiable in its parameters.
//
// Reverse pass: each forward step is
//   (a) v += h F, (b) x += dt v, (c) F = F(x), (d) v += h F, (e) loss terms,
// h = dt/2, and is undone as
//   (e) vbar += dP/dv, xbar/theta += loss terms at x_t
//   (d) Fbar += h vbar
//   (c) xbar += J_F(x_t)^T Fbar, theta += (dF/dtheta)^T Fbar, Fbar = 0
//   (b) vbar += dt xbar
//   (a) Fbar += h vbar.
// J_F^T Fbar is a Hessian-vector product over the full neighbour list:
//   xbar_i += sum_j [f(s) d + 2 f'(s) (r.d) r],  d = Fbar_i - Fbar_owner(j),
// symmetric in (i, j), so each lane owns its atom (no atomics); ghost
// adjoints are their owners'.  Every state of the forward pass is kept where
// there is room (keep_all); else (x, v) is checkpointed every rebuild interval
// and each interval is recomputed before it is reversed.  Within an interval
// the neighbour list and ghost table are fixed, as in the forward.
#include "tmd_internal.hpp"
#include "tmd_lj.hpp"
#include "tmd_pair.hpp"

namespace tmd {

struct AdjCoef {
    double cU;   // dL/dPE_t  = 2 (Ubar - U*) / (T N)
    double cW;   // dL/dW_t   = 2 (Pbar - P*) / (3 V T)
    // sigma-derivatives of the truncation constants
    double dfc_ds, ddfc_ds, duc_ds;
    int loss_terms;  // 0 at x_0 (the loss starts at t = 1)
};

// Both passes give an atom to a group of G lanes (atom_lanes), which share its
// list by groups of entries and add their sums.
// The reverse pass takes up to 130 registers with G > 1: four wavefronts a SIMD
// in FP64 (128), three in FP32-mixed with the smooth cutoff.  Four more cost
// FP64 23 -> 31 us a step at 15,028 atoms.
constexpr int kGroupThreads = 768;  // threads a block with G > 1

// the first list group of the lane in its atom's group of G (clamped: always a
// valid load), and the sum of a vector over the group
template <int G>
__device__ __forceinline__ int4 lane_group(int cnt, const int4* __restrict__ lp) {
    const int s = G > 1 ? min((int)threadIdx.x & (G - 1), max((cnt - 1) >> 3, 0)) : 0;
    return ld_stream(lp + (size_t)s * 64);
}
template <int G>
__device__ __forceinline__ double4 group_sum(double4 f) {
#pragma unroll
    for (int o = 1; o < G; o <<= 1) {
        f.x += __shfl_xor(f.x, o);
        f.y += __shfl_xor(f.y, o);
        f.z += __shfl_xor(f.z, o);
    }
    return f;
}

// One step of a trajectory on the cell-ordered mirrors, one launch: force at
// x_t, final kick, energy, virial and kinetic sums, and the next step's kick
// and drift, locals and their ghosts, into the next mirror.  The arithmetic
// and its order are those of the separate passes (force, integration, ghost
// refresh), but for the order of a force's sum where G > 1; the energy pass,
// the kinetic pass, their reductions, the ghost pass and the copies of states
// that came with them (about 60 of 75 us a step at 16,384 atoms) are gone.
struct TrajStep {
    Mir vel;               // velocities before the final kick in, after this pass out
    double hfin, hdt, dt;  // final kick (0: the trajectory's first force), next kick and drift
    int adv;               // also the next kick and drift
    Mir xnext;             // mirror of x_{t+1}
    Mir vt;                // v_t in mirror order (p null: not kept)
    double4 *ckx, *ckv;    // checkpoint of x_t, v_t in atom order (null: none)
    GhostIndex gh;
    double* acc;           // per tile: PE, W, sum v^2, added to
};

template <int PREC, int SHIFT, int UNIT, bool ENERGY, int G>
__global__ void __launch_bounds__(G > 1 ? kGroupThreads : kMaxTileThreads) k_traj_step(const CMir spos, const int* __restrict__ start,
                                                            const int* __restrict__ work, const int* __restrict__ wk,
                                                            const int* __restrict__ tile_start, const int* __restrict__ nbc,
                                                            const nb_t* __restrict__ nbl, LJArgs a, TrajStep t) {
    extern __shared__ double dyn[];
    const WinStage sp = win_stage(dyn, a.wcap);
    const int tile = block_tile(blockIdx.x, a.g);
    const int w0 = tile_start[tile], nloc = tile_start[tile + 1] - w0;
    if (nloc == 0) return;
    __shared__ TileWin W;
    tile_window(tile, start, a.g, W);
    const bool staged = stage_window(W, a.wcap, spos, nullptr, sp);
    PairEnergy en;
    double v2 = 0.0;
    for (int at = threadIdx.x / G; at < nloc; at += blockDim.x / G) {
        const int w = w0 + at;
        const int kw = wk[w];
        const double4 pi = spos[kw];
        const int cnt = nbc[w];
        const int4* lp = reinterpret_cast<const int4*>(nbl + (size_t)(w >> 6) * (size_t)a.cap * 64) + (w & 63);
        const int4 head = lane_group<G>(cnt, lp);
        double4 f = staged ? lj_full_atom<PREC, SHIFT, UNIT, true, false, ENERGY, G>(pi, cnt, lp, sp, spos, W, a, head, 0, nullptr, &en)
                           : lj_full_atom<PREC, SHIFT, UNIT, false, false, ENERGY, G>(pi, cnt, lp, sp, spos, W, a, head, 0, nullptr, &en);
        if (G > 1) {
            f = group_sum<G>(f);
            if (threadIdx.x & (G - 1)) continue;
        }
        double4 v = t.vel[kw];
        v.x = v.x + f.x * t.hfin;
        v.y = v.y + f.y * t.hfin;
        v.z = v.z + f.z * t.hfin;
        if (ENERGY) v2 += v.x * v.x + v.y * v.y + v.z * v.z;
        if (t.vt.p) t.vt[kw] = v;
        if (t.ckx) {
            const int i = work[w];
            t.ckx[i] = pi;
            t.ckv[i] = v;
        }
        if (t.adv) {
            v.x = v.x + f.x * t.hdt;
            v.y = v.y + f.y * t.hdt;
            v.z = v.z + f.z * t.hdt;
            double4 x = pi;
            x.x = x.x + v.x * t.dt;
            x.y = x.y + v.y * t.dt;
            x.z = x.z + v.z * t.dt;
            t.xnext[kw] = x;
            each_ghost(t.gh, t.gh.w[w], [&](int e, int kg) { t.xnext[kg] = ghost_image(x, t.gh, e); });
        }
        t.vel[kw] = v;
    }
    if (ENERGY) {
        const double bpe = block_sum_double_any(energy_sum(en.pe, a));
        const double bvir = block_sum_double_any(en.vir);
        const double bv2 = block_sum_double_any(v2);
        if (threadIdx.x == 0) {
            t.acc[3 * tile + 0] += bpe;
            t.acc[3 * tile + 1] += bvir;
            t.acc[3 * tile + 2] += bv2;
        }
    }
}

// One reverse step, one launch: (c) at x_t, then (b), (a) and the (e), (d) of
// step t - 1, which involve the lane's own atom only.  Adjoints live in
// mirror order inside an interval (ghosts carry their owners' Fbar), so the
// window's Fbar is staged beside its positions (48 B a slot) and an entry
// costs six LDS reads; it was an index, an owner and a 32-byte gather from
// global memory, behind 2-byte list loads.
//
// All pair quantities are linear in p = sigma^6 s^-4, q = sigma^12 s^-7,
// sr6, sr12 and the truncation's 1, s, s^2, so the parameter gradients
// accumulate those sums (9 operations an entry) and are combined once per
// lane; an entry is about 60 FP64 operations where it was about 110, without
// a branch: beyond the cutoff sr2 and the constants' factor `in` are zero.
//
// FP64 takes 1/s correctly rounded and s as the forward pass forms it;
// FP32-mixed skips the last rounding step and forms s with FMAs (a few 1e-16).
// 16,384 atoms in FP64: 26 us a step by events with one lane an atom, where the
// pair kernel took 86 and five more passes around it 5 us each.
struct AdjStep {
    Mir xb, vb;                   // the locals' xbar, vbar (mirror order, own entry read and written)
    CMir vprev;                   // v_{t-1} (mirror order)
    Mir fnext;                    // Fbar for step t - 1, locals and ghosts
    double4 *xbar, *vbar, *fbar;  // atom order, at the interval's first step
    GhostIndex gh;
    double cv, h, dt;
    int post, pre, end;           // (b) and (a); (e) and (d) of t - 1; last of the interval
    double* acc;                  // per tile: g_eps, g_sig, added to
};

template <int PREC, int SHIFT, int G>
__global__ void __launch_bounds__(G > 1 ? kGroupThreads : kMaxTileThreads) k_lj_adjoint(const CMir spos, const CMir fbm, const int* __restrict__ start,
                                                             const int* __restrict__ work, const int* __restrict__ wk,
                                                             const int* __restrict__ tile_start, const int* __restrict__ nbc,
                                                             const nb_t* __restrict__ nbl, LJArgs a, AdjCoef c, AdjStep t) {
    extern __shared__ double dyn[];
    const int tile = block_tile(blockIdx.x, a.g);
    const int w0 = tile_start[tile], nloc = tile_start[tile + 1] - w0;
    if (nloc == 0) return;
    __shared__ TileWin W;
    tile_window(tile, start, a.g, W);
    double* sx = dyn;
    double* sf = dyn + 3 * a.wcap;
    const int S = win_size(W);
    const bool staged = S + 1 <= a.wcap;
    if (staged) {
        double4 p[kStageInFlight], q[kStageInFlight];
        stage_rows(W, [&](int k, int u) { p[u] = spos[k]; q[u] = fbm[k]; },
                   [&](int j, int u) {
                       sx[3 * j] = p[u].x; sx[3 * j + 1] = p[u].y; sx[3 * j + 2] = p[u].z;
                       sf[3 * j] = q[u].x; sf[3 * j + 1] = q[u].y; sf[3 * j + 2] = q[u].z;
                   });
        if (threadIdx.x < 3) {
            sx[3 * S + threadIdx.x] = kFarPos;  // the sentinel slot that pads list groups
            sf[3 * S + threadIdx.x] = 0.0;
        }
    }
    __syncthreads();
    const double e48 = 48.0 * a.eps, e24 = 24.0 * a.eps;
    const double lU = c.loss_terms ? c.cU : 0.0, lW = c.loss_terms ? 2.0 * c.cW : 0.0;
    double g_eps = 0.0, g_sig = 0.0;
    // STAGED as a compile-time constant: LDS reads, not generic-pointer loads
    auto atoms = [&](auto staged_c) {
        constexpr bool STAGED = decltype(staged_c)::value;
        for (int at = threadIdx.x / G; at < nloc; at += blockDim.x / G) {
            const int w = w0 + at;
            const int kw = wk[w];
            const double4 pi = spos[kw];
            const double4 fbi = fbm[kw];
            const int cnt = nbc[w];
            const int4* lp = reinterpret_cast<const int4*>(nbl + (size_t)(w >> 6) * (size_t)a.cap * 64) + (w & 63);
            double ax = 0.0, ay = 0.0, az = 0.0;
            double Prf = 0.0, Qrf = 0.0, Rrf = 0.0, Srf = 0.0;  // sums of p rf, q rf, rf, s rf
            double S6 = 0.0, S12 = 0.0, N0 = 0.0, S1 = 0.0, S2 = 0.0;  // of sr6, sr12, 1, s, s^2
            const int ng = (cnt + 7) >> 3;
            int4 nx = lane_group<G>(cnt, lp);
            for (int gi = G > 1 ? (int)threadIdx.x & (G - 1) : 0; gi < ng; gi += G) {
                const int4 e = nx;
                nx = ld_stream(lp + (size_t)min(gi + G, ng - 1) * 64);
                const int rem = cnt - gi * 8;
#pragma unroll
                for (int hb = 0; hb < 8; hb += 2) {
                    if (hb >= rem) break;
#pragma unroll
                    for (int u = hb; u < hb + 2; ++u) {
                        const bool valid = STAGED || u < rem;
                        double xj, yj, zj, fxj, fyj, fzj;
                        if (STAGED) {
                            const int j = nb_entry(e, u);
                            xj = sx[3 * j]; yj = sx[3 * j + 1]; zj = sx[3 * j + 2];
                            fxj = sf[3 * j]; fyj = sf[3 * j + 1]; fzj = sf[3 * j + 2];
                        } else {
                            const int kk = win_index(valid ? nb_entry(e, u) : 0, W);
                            const double4 p = spos[kk], q = fbm[kk];
                            xj = p.x; yj = p.y; zj = p.z;
                            fxj = q.x; fyj = q.y; fzj = q.z;
                        }
                        const double rx = pi.x - xj, ry = pi.y - yj, rz = pi.z - zj;
                        const double s = PREC == PREC_FP64 ? rx * rx + ry * ry + rz * rz : fma(rx, rx, fma(ry, ry, rz * rz));
                        const bool ok = valid && s < a.rc2;
                        const double r2 = PREC == PREC_FP64 ? rcp_round(s) : rcp_refined(s);
                        const double sr2 = ok ? r2 : 0.0;
                        const double in = ok ? 1.0 : 0.0;
                        const double sv = ok ? s : 0.0;
                        const double sr6 = sr2 * sr2 * sr2 * a.sigma6;
                        const double p = sr6 * sr2, q = sr6 * p;
                        double f = fma(e48, q, -e24 * p);                      // f(s)
                        const double sdf0 = e24 * fma(-14.0, q, 4.0 * p);      // s f'(s)
                        double df = sdf0 * sr2, sdf = sdf0;                    // f'(s), s f'(s)
                        if (SHIFT) {
                            f = fma(-a.dfc, fma(-a.rc2, in, sv), fma(-a.fc, in, f));
                            df = fma(-a.dfc, in, df);
                            sdf = fma(-a.dfc, sv, sdf);
                        }
                        // J_F^T Fbar, and the loss: dPE/dx_i = -sum f r ; dW/dx_i = sum 2 (f + s f') r
                        const double dx = fbi.x - fxj, dy = fbi.y - fyj, dz = fbi.z - fzj;
                        const double rd = fma(rx, dx, fma(ry, dy, rz * dz));
                        const double cr = fma(2.0 * df, rd, fma(lW, f + sdf, -lU * f));
                        ax = fma(f, dx, fma(cr, rx, ax));
                        ay = fma(f, dy, fma(cr, ry, ay));
                        az = fma(f, dz, fma(cr, rz, az));
                        // parameters: Fbar_i . dF_i/dtheta over ordered pairs; the loss halves
                        const double rf = fma(rx, fbi.x, fma(ry, fbi.y, rz * fbi.z));
                        Prf = fma(p, rf, Prf);
                        Qrf = fma(q, rf, Qrf);
                        S6 += sr6;
                        S12 = fma(sr6, sr6, S12);
                        if (SHIFT) {
                            Rrf = fma(in, rf, Rrf);
                            Srf = fma(sv, rf, Srf);
                            N0 += in;
                            S1 += sv;
                            S2 = fma(sv, sv, S2);
                        }
                    }
                }
            }
            // sums of f rf, u, s f; and the same of their sigma-derivatives
            double Frf = e48 * Qrf - e24 * Prf, U = 4.0 * a.eps * (S12 - S6), SF = e48 * S12 - e24 * S6;
            const double k144 = 144.0 * a.eps / a.sigma, k24 = 24.0 * a.eps / a.sigma;
            double Drf = k144 * (4.0 * Qrf - Prf), DU = k24 * (2.0 * S12 - S6), DSF = k144 * (4.0 * S12 - S6);
            if (SHIFT) {
                const double Trf = Srf - a.rc2 * Rrf;                               // sum ds rf
                const double T1 = S1 - a.rc2 * N0;                                  // sum ds
                const double T2 = S2 - 2.0 * a.rc2 * S1 + a.rc2 * a.rc2 * N0;       // sum ds^2
                const double TS = S2 - a.rc2 * S1;                                  // sum s ds
                Frf = Frf - a.fc * Rrf - a.dfc * Trf;
                SF = SF - a.fc * S1 - a.dfc * TS;
                U = U - a.uc * N0 + 0.5 * a.fc * T1 + 0.25 * a.dfc * T2;
                Drf = Drf - c.dfc_ds * Rrf - c.ddfc_ds * Trf;
                DSF = DSF - c.dfc_ds * S1 - c.ddfc_ds * TS;
                DU = DU - c.duc_ds * N0 + 0.5 * c.dfc_ds * T1 + 0.25 * c.ddfc_ds * T2;
            }
            const double hW = 0.25 * lW, hU = 0.5 * lU;  // half of cW and cU
            g_eps += (Frf + (hU * U + hW * SF)) / a.eps;
            g_sig += Drf + (hU * DU + hW * DSF);
            if (G > 1) {
                const double4 sum = group_sum<G>(make_double4(ax, ay, az, 0.0));
                ax = sum.x; ay = sum.y; az = sum.z;
                if (threadIdx.x & (G - 1)) continue;
            }
            double4 xb = t.xb[kw], vb = t.vb[kw];
            xb.x += ax; xb.y += ay; xb.z += az;
            double4 fb = make_double4(0.0, 0.0, 0.0, 0.0);
            if (t.post) {
                // (c) Fbar = 0, (b) vbar += dt xbar, (a) Fbar = h vbar
                vb.x += t.dt * xb.x; vb.y += t.dt * xb.y; vb.z += t.dt * xb.z;
                fb = make_double4(t.h * vb.x, t.h * vb.y, t.h * vb.z, 0.0);
            }
            if (t.end) {
                const int i = work[w];
                t.xbar[i] = xb;
                t.vbar[i] = vb;
                t.fbar[i] = fb;
                continue;
            }
            if (t.pre) {
                // (e) vbar += cv v_{t-1}, (d) Fbar += h vbar
                const double4 v = t.vprev[kw];
                vb.x += t.cv * v.x; vb.y += t.cv * v.y; vb.z += t.cv * v.z;
                fb.x += t.h * vb.x; fb.y += t.h * vb.y; fb.z += t.h * vb.z;
            }
            t.xb[kw] = xb;
            t.vb[kw] = vb;
            t.fnext[kw] = fb;
            each_ghost(t.gh, t.gh.w[w], [&](int, int kg) { t.fnext[kg] = fb; });
        }
    };
    if (staged) atoms(std::true_type{});
    else atoms(std::false_type{});
    const double be = block_sum_double_any(g_eps);
    const double bs = block_sum_double_any(g_sig);
    if (threadIdx.x == 0) {
        t.acc[2 * tile + 0] += be;
        t.acc[2 * tile + 1] += bs;
    }
}

// acc[c] += sum_b partials[width * b + c] (one block, fixed order), and the
// partials start again from zero
__global__ void __launch_bounds__(256) k_accumulate(double* __restrict__ partials, int nblocks, int width,
                                                    double* __restrict__ acc) {
    for (int c = 0; c < width; ++c) {
        double v = 0.0;
        for (int b = threadIdx.x; b < nblocks; b += 256) {
            v += partials[(size_t)width * b + c];
            partials[(size_t)width * b + c] = 0.0;
        }
        const double t = block_sum_double<256>(v);
        if (threadIdx.x == 0) acc[c] += t;
    }
}

__global__ void k_fill_double(double* __restrict__ p, long long n) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = 0.0;
}

// An interval's adjoints from atom order into its mirrors, with (e) and (d)
// of its last state: vbar += cv v_t ; Fbar += h vbar
__global__ void k_adj_begin(const int* __restrict__ work, const int* __restrict__ wk, int n, const double4* __restrict__ xbar,
                            const double4* __restrict__ vbar, const double4* __restrict__ fbar, const CMir vt, double cv, double h,
                            int pre, const Mir xb, const Mir vb, const Mir fb, GhostIndex gh) {
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= n) return;
    const int i = work[w], kw = wk[w];
    double4 b = vbar[i], f = fbar[i];
    if (pre) {
        const double4 v = vt[kw];
        b.x += cv * v.x; b.y += cv * v.y; b.z += cv * v.z;
        f.x += h * b.x; f.y += h * b.y; f.z += h * b.z;
    }
    xb[kw] = xbar[i];
    vb[kw] = b;
    fb[kw] = f;
    each_ghost(gh, gh.w[w], [&](int, int kg) { fb[kg] = f; });
}

// ---------------------------------------------------------------------------
static void copy_state(Sim& s, double4* xd, double4* vd, const double4* xs, const double4* vs) {
    const size_t bytes = sizeof(double4) * (size_t)s.n;
    TMD_HIP(hipMemcpyAsync(xd, xs, bytes, hipMemcpyDeviceToDevice, s.stream));
    TMD_HIP(hipMemcpyAsync(vd, vs, bytes, hipMemcpyDeviceToDevice, s.stream));
}

// the current state (atom order) kept, and put back
static void keep_state(Sim& s) { copy_state(s, s.adj_x0.as<double4>(), s.adj_v0.as<double4>(), s.pos.as<double4>(), s.vel.as<double4>()); }

static void restore_from(Sim& s, const DevBuf& bx, const DevBuf& bv, size_t slot) {
    mirror_invalidate(s);
    s.pos_stale = 0;
    s.vel_mirrored = 0;
    copy_state(s, s.pos.as<double4>(), s.vel.as<double4>(), bx.as<double4>() + slot * s.n, bv.as<double4>() + slot * s.n);
}

// Ghosts, cells and full list: from the mirrors with the periodic wrap, or
// from atom order without.  The velocities come along into their mirror and
// the ghost index is made.
static void relist(Sim& s, bool wrap, double cutoff) {
    s.vel_mirror_wanted = 1;
    rebuild_lists(s, wrap, 0, cutoff);
    s.vel_mirror_wanted = 0;
}

static int ntiles_of(const Sim& s) { return s.tiles.ntx * s.tiles.nty * s.tiles.ntz; }

static void zero(Sim& s, void* p, size_t doubles) {
    hipLaunchKernelGGL(k_fill_double, dim3(std::min<long long>(div_up((long long)doubles, 1024), 1024)), dim3(256), 0, s.stream,
                       static_cast<double*>(p), (long long)doubles);
}

// Per-tile accumulators of `width` sums, kept over an interval (its tiles are
// fixed), then added to the totals and cleared.
static double* tile_sums(Sim& s, int width) {
    const size_t need = (size_t)width * (size_t)std::max(ntiles_of(s), 1);
    if (sizeof(double) * need > s.adj_part.bytes) {
        s.adj_part.reserve(sizeof(double) * 2 * need, false, s.stream);
        if (has_error()) return nullptr;
        zero(s, s.adj_part.p, 2 * need);
    }
    return s.adj_part.as<double>();
}

static void flush_sums(Sim& s, int width, double* acc) {
    // no pass has summed over these tiles yet (a rebuild at the first step)
    if (sizeof(double) * (size_t)width * (size_t)ntiles_of(s) > s.adj_part.bytes) return;
    hipLaunchKernelGGL(k_accumulate, dim3(1), dim3(256), 0, s.stream, s.adj_part.as<double>(), ntiles_of(s), width, acc);
    TMD_HIP(hipGetLastError());
}

// Lanes an atom of both passes: four or two while all of them fit on the chip
// at once (65,536 lanes, one wavefront a SIMD); there a pass lasts as long as
// one wavefront's lists.  us a step of a gradient, rebuilds included, at 1, 2
// and 4 lanes: 6^3 cells FP64 67, 52, 44; 12^3 61, 46, 39; 16^3 (16,384 atoms)
// 61, 54, 52; 20^3 (32,000) 71, 63, 66; 24^3 mixed 95, 98, 101.
constexpr int kChipLanes = 65536;
static int atom_lanes(const Sim& s) {
    if (s.tile_threads_req > 0) return 1;
    return s.n <= kChipLanes / 4 ? 4 : (s.n <= kChipLanes / 2 ? 2 : 1);
}
static int group_threads(const Sim& s, int lanes) {
    if (lanes == 1) return s.tile_threads;
    return std::min(kGroupThreads, (std::max(s.max_locals, 1) * lanes + kWave - 1) / kWave * kWave);
}

struct TrajSpec {
    int steps, ck;
    double dt, rc, skin, eps, sigma;
};

// The pass of step t at the positions in the mirror x.
static void traj_step(Sim& s, const TrajSpec& p, const DevBuf& x, TrajStep t, bool energy) {
    if (has_error()) return;
    LJArgs a = make_lj_args(s, p.rc, p.eps, p.sigma);
    a.wcap = window_cap_pos(s);
    const size_t lds = (size_t)a.wcap * kPosStageBytes;
    const int unit = (p.eps == 1.0 && a.sigma6 == 1.0) ? 1 : 0;
    t.vel = Mir{s.svel.as<double>()};
    t.hdt = 0.5 * p.dt;
    t.dt = p.dt;
    t.gh = ghost_index(s);
    t.acc = energy ? tile_sums(s, 3) : nullptr;
    if (has_error()) return;
    s.last_force_rc = p.rc;
    hipEvent_t ev = nullptr;
    s.timer.begin(K_FORCE, s.stream, &ev);
    const int lanes = atom_lanes(s);
    const int threads = group_threads(s, lanes);
#define TMD_TS(P, SH, U, E, G)                                                                                             \
    hipLaunchKernelGGL((k_traj_step<P, SH, U, E, G>), dim3(ntiles_of(s)), dim3(threads), lds, s.stream,               \
                       CMir{x.as<double>()}, (const int*)s.cell_start.as<int>(), (const int*)s.work.as<int>(),           \
                       (const int*)s.work_k.as<int>(), (const int*)s.tile_start.as<int>(),                              \
                       (const int*)s.nb_count.as<int>(), (const nb_t*)s.nb_list.as<nb_t>(), a, t)
#define TMD_TS_G(P, SH, U, E) do { if (lanes == 4) TMD_TS(P, SH, U, E, 4); else if (lanes == 2) TMD_TS(P, SH, U, E, 2); else TMD_TS(P, SH, U, E, 1); } while (0)
#define TMD_TS_E(P, SH, U) do { if (energy) TMD_TS_G(P, SH, U, true); else TMD_TS_G(P, SH, U, false); } while (0)
#define TMD_TS_U(P, SH) do { if (unit) TMD_TS_E(P, SH, 1); else TMD_TS_E(P, SH, 0); } while (0)
#define TMD_TS_S(P) do { if (s.lj_shift) TMD_TS_U(P, 1); else TMD_TS_U(P, 0); } while (0)
    if (s.precision == PREC_FP64) TMD_TS_S(PREC_FP64);
    else if (s.precision == PREC_FP32_KAHAN) TMD_TS_S(PREC_FP32_KAHAN);
    else TMD_TS_S(PREC_FP32_MIXED);
#undef TMD_TS_S
#undef TMD_TS_U
#undef TMD_TS_E
#undef TMD_TS_G
#undef TMD_TS
    s.timer.end(K_FORCE, s.stream, ev);
    TMD_HIP(hipGetLastError());
    if (t.adv && !s.gh_valid) ghosts_from_owners(s, t.xnext.p, true);
}

// The states of the steps t0 .. of a trajectory, mirrors of positions and
// velocities one behind the other (adj_segx, adj_segv).
struct Kept {
    bool on = false;
    size_t stride = 0;  // doubles a mirror
    int t0 = 0;
    double *x = nullptr, *v = nullptr;
    double* X(int t) const { return x + (size_t)(t - t0) * stride; }
    double* V(int t) const { return v + (size_t)(t - t0) * stride; }
};
static Kept reserve_kept(Sim& s, int t0, int t1) {
    Kept k;
    k.stride = 3 * (size_t)s.cap_all;
    k.t0 = t0;
    const size_t bytes = sizeof(double) * k.stride * (size_t)(t1 - t0 + 1);
    s.adj_segx.reserve(bytes, false, s.stream);
    s.adj_segv.reserve(bytes, false, s.stream);
    k.x = s.adj_segx.as<double>();
    k.v = s.adj_segv.as<double>();
    k.on = !has_error();
    return k;
}
// A gradient keeps every state of its forward pass, where that takes at most
// 4 GiB and a quarter of the free memory; else each interval is recomputed
// from its checkpoint.  16,384 atoms over 200 steps: 0.4 GB, and the second
// forward pass (16 us a step) is gone, 14.8 -> 11.7 ms a gradient
// (10.0 with the lanes of atom_lanes).
constexpr size_t kKeptBytes = size_t(4) << 30;
static bool keep_all(const Sim& s, int steps) {
    const size_t bytes = 2 * sizeof(double) * 3 * (size_t)s.cap_all * (size_t)(steps + 1);
    if (bytes > kKeptBytes) return false;
    if (bytes <= s.adj_segx.bytes + s.adj_segv.bytes) return true;
    size_t avail = 0, total = 0;
    return hipMemGetInfo(&avail, &total) == hipSuccess && bytes <= avail / 4;
}

static void copy_mirror(Sim& s, double* to, const DevBuf& from) {
    TMD_HIP(hipMemcpyAsync(to, from.p, (size_t)kMirBytes * (size_t)s.nbinned, hipMemcpyDeviceToDevice, s.stream));
}

// Forward trajectory from (adj_x0, adj_v0), reneighbouring every ck steps
// exactly as the step loop does (wrap, ghosts, cells, list after the
// position update of steps ck, 2ck, ...).  With checkpoints, slot k holds
// the state at t = k ck (after that step's wrap), and the states go into
// `kept` while it is on.  The mirrors alternate as in the step loop; a rebuild
// goes from mirror to mirror.
static void forward_traj(Sim& s, const TrajSpec& p, bool store_ckpt, double* ubar, double* pbar, Kept* kept = nullptr) {
    const double cut = p.rc + p.skin;
    double* acc = s.adj_acc.as<double>();
    zero(s, acc, 4);
    restore_from(s, s.adj_x0, s.adj_v0, 0);
    relist(s, false, cut);
    if (has_error()) return;
    for (int t = 0; t <= p.steps && !has_error(); ++t) {
        if (t > 0 && t % p.ck == 0) {
            flush_sums(s, 3, acc);  // the tiles change
            relist(s, true, cut);
            if (has_error()) return;
        }
        TrajStep st{};
        st.hfin = t > 0 ? 0.5 * p.dt : 0.0;
        st.adv = t < p.steps;
        if (kept && 3 * (size_t)s.cap_all > kept->stride) kept->on = false;  // a rebuild made room for more ghosts
        const bool keep = kept && kept->on;
        DevBuf x = s.spos;
        if (keep) {
            if (t % p.ck == 0) copy_mirror(s, kept->X(t), s.spos);
            x.p = kept->X(t);
            st.vt = Mir{kept->V(t)};
        }
        // a rebuild starts from the mirror
        const bool into_kept = keep && (t + 1) % p.ck != 0;
        st.xnext = Mir{into_kept && st.adv ? kept->X(t + 1) : s.spos2.as<double>()};
        if (store_ckpt && t % p.ck == 0) {
            st.ckx = s.adj_ckx.as<double4>() + (size_t)(t / p.ck) * s.n;
            st.ckv = s.adj_ckv.as<double4>() + (size_t)(t / p.ck) * s.n;
        }
        traj_step(s, p, x, st, t > 0);
        if (st.adv && !into_kept) std::swap(s.spos, s.spos2);
        s.pos_stale = 1;  // the state lives in the mirrors
        s.vel_mirrored = 1;
    }
    flush_sums(s, 3, acc);
    double h[3] = {0, 0, 0};
    TMD_HIP(hipMemcpyAsync(h, acc, sizeof h, hipMemcpyDeviceToHost, s.stream));
    TMD_HIP(hipStreamSynchronize(s.stream));
    const double vol = s.g.len[0] * s.g.len[1] * s.g.len[2];
    *ubar = h[0] / (double)s.n / (double)p.steps;
    *pbar = (h[2] + h[1]) / (3.0 * vol) / (double)p.steps;
}

static bool begin_traj(Sim& s, const TrajSpec& p, bool adjoint) {
    if (p.steps <= 0 || p.ck <= 0) {
        set_error(__FILE__, __LINE__, "trajectory: steps and the reneighbouring interval must be positive");
        return false;
    }
    if (s.ghost_mode != GHOST_FRESH) {
        set_error(__FILE__, __LINE__, "trajectory: needs fresh ghost positions (tmd_set_ghost_mode(0))");
        return false;
    }
    if (s.n == 0) {
        set_error(__FILE__, __LINE__, "trajectory: no atoms");
        return false;
    }
    const size_t atom = sizeof(double4) * (size_t)s.n;
    s.adj_x0.reserve(atom, false, s.stream);
    s.adj_v0.reserve(atom, false, s.stream);
    s.adj_acc.reserve(8 * sizeof(double), false, s.stream);
    if (adjoint) {
        const size_t nck = (size_t)(p.steps / p.ck + 1);
        s.adj_ckx.reserve(atom * nck, false, s.stream);
        s.adj_ckv.reserve(atom * nck, false, s.stream);
        s.adj_xbar.reserve(atom, false, s.stream);
        s.adj_vbar.reserve(atom, false, s.stream);
        s.adj_fbar.reserve(atom, false, s.stream);
    }
    if (has_error()) return false;
    sync_pos_from_mirror(s);
    keep_state(s);
    if (s.adj_part.p) zero(s, s.adj_part.p, s.adj_part.bytes / sizeof(double));  // sums of a call that ended in an error
    if (adjoint) {
        // the reverse pass stages 48 B a window slot: tiles for that
        s.stage_bytes = kAdjStageBytes;
        s.stage_budget = kLdsBudget;
    }
    return !has_error();
}

// put the initial state back, with its ghosts, list and forces
static void end_traj(Sim& s, const TrajSpec& p) {
    if (has_error()) return;
    restore_from(s, s.adj_x0, s.adj_v0, 0);
    if (s.stage_bytes != kPosStageBytes) {
        s.stage_bytes = kPosStageBytes;
        s.tile_auto[0] = s.tile_auto[1] = s.tile_auto[2] = 0;
        s.tile_tuned = 0;
    }
    rebuild_lists(s, false, 0, p.rc + p.skin);
    compute_lj(s, 0, p.rc, p.eps, p.sigma);
    TMD_HIP(hipStreamSynchronize(s.stream));
}

bool traj_loss(Sim& s, int steps, int ck, double dt, double rc, double skin, double eps, double sigma, double* ubar,
               double* pbar) {
    const TrajSpec p{steps, ck, dt, rc, skin, eps, sigma};
    if (!begin_traj(s, p, false)) return false;
    forward_traj(s, p, false, ubar, pbar);
    end_traj(s, p);
    return !has_error();
}

bool traj_adjoint(Sim& s, int steps, int ck, double dt, double rc, double skin, double eps, double sigma, double u_target,
                  double p_target, double* loss3, double* grad_theta, double* grad_x, double* grad_v) {
    const TrajSpec p{steps, ck, dt, rc, skin, eps, sigma};
    if (!begin_traj(s, p, true)) return false;
    double ubar = 0.0, pbar = 0.0;
    Kept kept;
    if (keep_all(s, steps)) kept = reserve_kept(s, 0, steps);
    if (has_error()) return false;
    forward_traj(s, p, true, &ubar, &pbar, kept.on ? &kept : nullptr);
    if (has_error()) return false;
    const int n = s.n;
    const double vol = s.g.len[0] * s.g.len[1] * s.g.len[2];
    loss3[0] = (ubar - u_target) * (ubar - u_target) + (pbar - p_target) * (pbar - p_target);
    loss3[1] = ubar;
    loss3[2] = pbar;

    AdjCoef c;
    c.cU = 2.0 * (ubar - u_target) / ((double)steps * (double)n);
    c.cW = 2.0 * (pbar - p_target) / (3.0 * vol * (double)steps);
    {
        // sigma-derivatives of f(rc^2), f'(rc^2), u(rc^2)
        const double sr2 = 1.0 / (rc * rc);
        const double s3 = sigma * sigma * sigma, sr6 = sr2 * sr2 * sr2 * (s3 * s3);
        c.dfc_ds = 144.0 * eps / sigma * sr2 * sr6 * (4.0 * sr6 - 1.0);
        c.ddfc_ds = 144.0 * eps / sigma * sr2 * sr2 * sr6 * (4.0 - 28.0 * sr6);
        c.duc_ds = 24.0 * eps / sigma * sr6 * (2.0 * sr6 - 1.0);
    }
    c.loss_terms = 0;
    const double h = 0.5 * dt;
    const double cv = 2.0 * c.cW;  // d(sum v^2)/dv = 2 v
    zero(s, s.adj_xbar.p, 4 * (size_t)n);
    zero(s, s.adj_vbar.p, 4 * (size_t)n);
    zero(s, s.adj_fbar.p, 4 * (size_t)n);
    double* theta = s.adj_acc.as<double>() + 4;
    zero(s, theta, 2);
    const int nt = 256;
    const double cut = rc + skin;
    Kept seg = kept;
    for (int sg = steps / ck; sg >= 0 && !has_error(); --sg) {
        const int t0 = sg * ck, t1 = std::min(t0 + ck - 1, steps);
        // the interval's lists, from its checkpoint
        restore_from(s, s.adj_ckx, s.adj_ckv, (size_t)sg);
        relist(s, false, cut);
        if (has_error()) return false;
        const size_t stride = kept.on ? kept.stride : 3 * (size_t)s.cap_all;  // doubles per mirror
        s.adj_mir.reserve(sizeof(double) * stride * 4, false, s.stream);
        if (has_error()) return false;
        if (!kept.on) {
            // recompute the interval (its list is fixed), every state kept in
            // mirror order, ghosts included
            seg = reserve_kept(s, t0, t1);
            if (has_error()) return false;
            copy_mirror(s, seg.X(t0), s.spos);
            for (int t = t0; t <= t1 && !has_error(); ++t) {
                TrajStep st{};
                st.hfin = t > t0 ? h : 0.0;
                st.adv = t < t1;
                st.vt = Mir{seg.V(t)};
                if (st.adv) st.xnext = Mir{seg.X(t + 1)};
                DevBuf x;
                x.p = seg.X(t);
                // the last state's velocity needs its force too; a lone state has it
                if (t < t1 || t > t0) traj_step(s, p, x, st, false);
                else copy_mirror(s, seg.V(t), s.svel);
            }
        }
        // reverse it
        double* xb = s.adj_mir.as<double>();
        double* vb = xb + stride;
        double* fb[2] = {vb + stride, vb + 2 * stride};
        hipLaunchKernelGGL(k_adj_begin, dim3(div_up(n, nt)), dim3(nt), 0, s.stream, (const int*)s.work.as<int>(),
                           (const int*)s.work_k.as<int>(), n, (const double4*)s.adj_xbar.as<double4>(),
                           (const double4*)s.adj_vbar.as<double4>(), (const double4*)s.adj_fbar.as<double4>(), CMir{seg.V(t1)}, cv, h,
                           t1 >= 1 ? 1 : 0, Mir{xb}, Mir{vb}, Mir{fb[0]}, ghost_index(s));
        TMD_HIP(hipGetLastError());
        if (!s.gh_valid) ghosts_from_owners(s, fb[0], false);
        LJArgs a = make_lj_args(s, rc, eps, sigma);
        a.wcap = std::min(s.max_window + 1, kLdsBudget / kAdjStageBytes);
        const size_t lds = (size_t)a.wcap * kAdjStageBytes;
        // the adjoint kernel's precision: the forward's unless set apart
        const int prec = s.adj_precision >= 0 ? s.adj_precision : s.precision;
        for (int t = t1; t >= t0 && !has_error(); --t) {
            AdjStep st{};
            st.xb = Mir{xb};
            st.vb = Mir{vb};
            st.end = t == t0;
            st.post = t >= 1;
            st.pre = t - 1 >= 1;
            if (!st.end) st.vprev = CMir{seg.V(t - 1)};
            st.fnext = Mir{fb[1]};
            st.xbar = s.adj_xbar.as<double4>();
            st.vbar = s.adj_vbar.as<double4>();
            st.fbar = s.adj_fbar.as<double4>();
            st.gh = ghost_index(s);
            st.cv = cv;
            st.h = h;
            st.dt = dt;
            st.acc = tile_sums(s, 2);
            c.loss_terms = t >= 1 ? 1 : 0;
            if (has_error()) return false;
            hipEvent_t ev = nullptr;
            s.timer.begin(K_ADJOINT, s.stream, &ev);
            const int lanes = atom_lanes(s);
            const int threads = group_threads(s, lanes);
#define TMD_ADJ(P, SH, G)                                                                                                  \
    hipLaunchKernelGGL((k_lj_adjoint<P, SH, G>), dim3(ntiles_of(s)), dim3(threads), lds, s.stream, CMir{seg.X(t)},     \
                       CMir{fb[0]}, (const int*)s.cell_start.as<int>(), (const int*)s.work.as<int>(),                    \
                       (const int*)s.work_k.as<int>(), (const int*)s.tile_start.as<int>(),                              \
                       (const int*)s.nb_count.as<int>(), (const nb_t*)s.nb_list.as<nb_t>(), a, c, st)
#define TMD_ADJ_G(P, SH) do { if (lanes == 4) TMD_ADJ(P, SH, 4); else if (lanes == 2) TMD_ADJ(P, SH, 2); else TMD_ADJ(P, SH, 1); } while (0)
            if (prec == PREC_FP64) {
                if (s.lj_shift) TMD_ADJ_G(PREC_FP64, 1); else TMD_ADJ_G(PREC_FP64, 0);
            } else {
                if (s.lj_shift) TMD_ADJ_G(PREC_FP32_MIXED, 1); else TMD_ADJ_G(PREC_FP32_MIXED, 0);
            }
#undef TMD_ADJ_G
#undef TMD_ADJ
            s.timer.end(K_ADJOINT, s.stream, ev);
            TMD_HIP(hipGetLastError());
            if (!st.end && !s.gh_valid) ghosts_from_owners(s, fb[1], false);
            std::swap(fb[0], fb[1]);
        }
        flush_sums(s, 2, theta);
    }
    const size_t row = 3 * (size_t)n;
    s.h_out.reserve(2 * row);
    if (has_error()) return false;
    double th[2] = {0, 0};
    TMD_HIP(hipMemcpyAsync(th, theta, sizeof th, hipMemcpyDeviceToHost, s.stream));
    const HostArray out[2] = {{s.adj_xbar.as<double>(), s.h_out.p, grad_x ? row : 0, row, 3},
                              {s.adj_vbar.as<double>(), s.h_out.p + row, grad_v ? row : 0, row, 3}};
    to_host(out, 2, s.h_out.pinned, s.stream);
    TMD_HIP(hipStreamSynchronize(s.stream));
    if (has_error()) return false;
    grad_theta[0] = th[0];
    grad_theta[1] = th[1];
    host_copy({{grad_x, s.h_out.p, grad_x ? sizeof(double) * row : 0},
               {grad_v, s.h_out.p + row, grad_v ? sizeof(double) * row : 0}});
    end_traj(s, p);
    return !has_error();
}

}  // namespace tmd
