// Per-atom pair-force bodies shared by the single-box kernels (k_force.hip)
// and the batched-replica kernels (k_batch.hip): both evaluate exactly the
// same arithmetic in the same order.
#pragma once

#include "tmd_window.hpp"
#include "tmd_lj.hpp"

namespace tmd {

// Refined reciprocal of x and the correctly rounded quotient num / x from it:
// two Newton steps on the hardware's estimate, then the residual's correction
// (Markstein's final step), as the compiler's division does them, without the
// scaling and the special-case fix-up around it, which operands of ordinary
// size do not need (here squared distances, from 2^-1022 to about 1e300).
// Zero and below give NaN where the division gave infinity: the force and
// virial of two atoms at one point are NaN either way, for their energy see
// energy_sum.
// Infinity, which the cutoff masks, gives NaN and not zero.  1 / x is 7
// instructions instead of 11, and quotients by the same x share the first 5.
__device__ __forceinline__ double rcp_refined(double x) {
    double y = __builtin_amdgcn_rcp(x);
    y = fma(y, fma(-x, y, 1.0), y);
    return fma(y, fma(-x, y, 1.0), y);
}
__device__ __forceinline__ double rcp_round(double x) {
    const double y = rcp_refined(x);
    return fma(fma(-x, y, 1.0), y, y);
}
__device__ __forceinline__ double div_round(double num, double x, double y) {  // y = rcp_refined(x)
    const double q = num * y;
    return fma(fma(-x, q, num), y, q);
}

// entry u (0..7) of a packed group of 8 u16 list entries
__device__ __forceinline__ int nb_entry(const int4& q, int u) {
    const int w = (u >> 1) == 0 ? q.x : ((u >> 1) == 1 ? q.y : ((u >> 1) == 2 ? q.z : q.w));
    return (u & 1) ? (int)((unsigned)w >> 16) : (w & 0xffff);
}


// FP64 pair scalar of the reference closure; UNIT skips the exact
// multiplications by eps = 1 and sigma^6 = 1 (x * 1.0 == x), so the result
// is bit-identical either way.  sr6 also serves the energy.
template <int SHIFT, int UNIT>
__device__ __forceinline__ double lj_f64u(const LJArgs& a, double rsq, double& sr6) {
    const double sr2 = rcp_round(rsq);
    sr6 = UNIT ? sr2 * sr2 * sr2 : sr2 * sr2 * sr2 * a.sigma6;
    double f = UNIT ? 48.0 * sr6 * (sr6 - 0.5) * sr2 : 48.0 * sr6 * (sr6 - 0.5) * sr2 * a.eps;
    if (SHIFT) f = f - a.fc - (rsq - a.rc2) * a.dfc;
    return f;
}

// pair energy from sr6
template <int SHIFT>
__device__ __forceinline__ double lj_u64(const LJArgs& a, double rsq, double sr6) {
    double u = 4.0 * a.eps * sr6 * (sr6 - 1.0);
    if (SHIFT) {
        const double ds = rsq - a.rc2;
        u = u - a.uc + ds * (0.5 * a.fc) + ds * ds * (0.25 * a.dfc);
    }
    return u;
}

// A lane's energy sum.  A pair at zero distance made it NaN where its energy is
// infinite, 4 eps sr6^2: set right once, at the end of the sum.
__device__ __forceinline__ double energy_sum(double pe, const LJArgs& a) {
    return pe == pe ? pe : 4.0 * a.eps * (__builtin_inf() * a.sigma6);
}

template <int SHIFT, int UNIT>
__device__ __forceinline__ float lj_f32u(const LJArgs& a, float rsq) {
    const float sr2 = __builtin_amdgcn_rcpf(rsq);
    const float sr6 = UNIT ? sr2 * sr2 * sr2 : sr2 * sr2 * sr2 * a.sigma6f;
    // UNIT: 48 sr6 (sr6 - 1/2) sr2 as (sr6 sr2) (48 sr6 - 24), one FMA
    float f = UNIT ? (sr6 * sr2) * __builtin_fmaf(48.0f, sr6, -24.0f) : 48.0f * sr6 * (sr6 - 0.5f) * sr2 * a.epsf;
    if (SHIFT) f = f - a.fcf - (rsq - a.rc2f) * a.dfcf;
    return f;
}

// Kahan compensated summation (s, c) += x.  c keeps the excess that the
// rounded addition put into s, (t - s) - y, so the compensated value of the
// sum is s - c (kahan_value).  The translation unit is built without FP
// contraction, so the four operations are not fused.
__host__ __device__ __forceinline__ void kahan_add(float& s, float& c, float x) {
    const float y = x - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
}

__host__ __device__ __forceinline__ double kahan_value(float s, float c) { return (double)s - (double)c; }

// Neighbour position of window offset t: LDS (x, y, z interleaved) when the
// window is staged, else the cell-ordered mirror.
template <bool STAGED, class SP>
__device__ __forceinline__ void win_pos(int t, const WinStage& st, const SP& spos, const TileWin& W,
                                        double& x, double& y, double& z) {
    if (STAGED) {
        x = st.xyz[3 * t + 0];
        y = st.xyz[3 * t + 1];
        z = st.xyz[3 * t + 2];
    } else {
        const double4 p = spos[win_index(t, W)];
        x = p.x;
        y = p.y;
        z = p.z;
    }
}

// Full-list force on one atom (lane).  Entries are read 8 at a time (one
// 16-byte load, prefetched a group ahead) and evaluated 4 at a time; the
// pair terms are evaluated without branches (a masked entry's scalar is
// replaced by zero) and accumulated in list order.  Adding a masked term
// adds dx * 0.0 = +-0.0, which leaves the running sum unchanged (the sum
// starts at +0.0 and never becomes -0.0), so the FP64 result equals the
// sequential reference sum bit for bit.  From a staged window, the entries
// past the count in the last group are the sentinel offset (beyond the
// cutoff), so only the cutoff test masks; from the mirror, the count does.
// FP32 variants form rsq with FMAs; FP64 keeps the reference's rounding.
//
// PAIR2 (half lists): the lane's groups are column 1's (cnt entries at lp)
// followed by column 2's (cnt2 at lp2), one running sum over both; a
// wavefront then runs as many groups as its busiest lane has in both
// columns together, not the busiest lane of each column in turn.
//
// G > 1: lane s of a group of G takes list groups s, s + G, ..; the caller
// adds the lanes' sums.
//
// ENERGY (full lists): also pe += u / 2 and vir += f r^2 / 2 of every entry
// within the cutoff, in FP64 whatever the force's precision.
struct PairEnergy {
    double pe = 0.0, vir = 0.0;
};
template <bool PAIR2>
__device__ __forceinline__ int4 list_head(int cnt, const int4* __restrict__ lp, const int4* __restrict__ lp2) {
    return ld_stream(!PAIR2 || cnt > 0 ? lp : lp2);
}
template <int PREC, int SHIFT, int UNIT, bool STAGED, bool PAIR2 = false, bool ENERGY = false, int G = 1, class SP = const double4*>
__device__ __forceinline__ double4 lj_full_atom(const double4 pi, int cnt, const int4* __restrict__ lp, const WinStage& sp,
                                                const SP& spos, const TileWin& W, const LJArgs& a,
                                                const int4 first, int cnt2 = 0, const int4* __restrict__ lp2 = nullptr,
                                                PairEnergy* en = nullptr) {
    double fx = 0.0, fy = 0.0, fz = 0.0;
    float sxa = 0.f, sya = 0.f, sza = 0.f, cxa = 0.f, cya = 0.f, cza = 0.f;
    const int ng1 = (cnt + 7) >> 3;
    const int ng = ng1 + (PAIR2 ? (cnt2 + 7) >> 3 : 0);
    // group g of the lane's entries (group 0 of either column always
    // exists: capacity >= 8)
    auto grp = [&](int g) -> const int4* {
        return (!PAIR2 || g < ng1) ? lp + (size_t)g * 64 : lp2 + (size_t)(g - ng1) * 64;
    };
    // the next group of 8 entries is loaded while the current one is used
    // (streaming loads: each group is read once per pass); the caller has
    // loaded the first (list_head)
    int4 q = first;
    for (int gi = G > 1 ? (int)threadIdx.x & (G - 1) : 0; gi < ng; gi += G) {
        const int4 e = q;
        q = ld_stream(grp(min(gi + G, ng - 1)));  // next group (clamped: always a valid load)
        const int rem = (!PAIR2 || gi < ng1) ? cnt - gi * 8 : cnt2 - (gi - ng1) * 8;  // entries in this group
        // two passes of 4 entries (fewer live registers than 8 at once),
        // unrolled: the compiler then overlaps one pass's LDS reads with the
        // other's arithmetic
#pragma unroll
        for (int hb = 0; hb < 8; hb += 4) {
        if (hb >= rem) break;  // this lane's entries are done
        double dx[4], dy[4], dz[4], rs[4];
        bool ok[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bool valid = STAGED || hb + u < rem;
            double xj, yj, zj;
            win_pos<STAGED>(valid ? nb_entry(e, hb + u) : 0, sp, spos, W, xj, yj, zj);
            dx[u] = pi.x - xj;
            dy[u] = pi.y - yj;
            dz[u] = pi.z - zj;
            rs[u] = PREC == PREC_FP64 ? dx[u] * dx[u] + dy[u] * dy[u] + dz[u] * dz[u]
                                      : fma(dx[u], dx[u], fma(dy[u], dy[u], dz[u] * dz[u]));
            ok[u] = valid && rs[u] < a.rc2;
        }
        if (ENERGY && PREC != PREC_FP64) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                double sr6;
                const double f = lj_f64u<SHIFT, UNIT>(a, rs[u], sr6);
                en->pe += 0.5 * (ok[u] ? lj_u64<SHIFT>(a, rs[u], sr6) : 0.0);
                en->vir += 0.5 * (ok[u] ? f * rs[u] : 0.0);
            }
        }
        // The pair scalar is evaluated for every entry and masked afterwards:
        // a masked entry may have rsq = 0 (its own position) or lie beyond
        // the cutoff; its (possibly infinite) scalar is replaced by 0 by the
        // select, so the masked term adds dx * 0 = +-0.
        if (PREC == PREC_FP64) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                double sr6;
                const double f = lj_f64u<SHIFT, UNIT>(a, rs[u], sr6);
                const double fm = ok[u] ? f : 0.0;
                if (ENERGY) {
                    en->pe += 0.5 * (ok[u] ? lj_u64<SHIFT>(a, rs[u], sr6) : 0.0);
                    en->vir += 0.5 * (ok[u] ? f * rs[u] : 0.0);
                }
                fx = fx + dx[u] * fm;
                fy = fy + dy[u] * fm;
                fz = fz + dz[u] * fm;
            }
        } else if (PREC == PREC_FP32_MIXED) {
            // FP32 pair scalar, FP64 fused multiply-add accumulation of dx * f
            // (one rounding per term; the FP64 mantissa absorbs the sum's
            // rounding)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                double fm;
                if (SHIFT) {
                    const float f = lj_f32u<SHIFT, UNIT>(a, (float)rs[u]);
                    fm = (double)(ok[u] ? f : 0.0f);
                } else {
                    // a masked entry gets rsq = +inf, so sr2 = 1/inf = 0 and
                    // the plain-cutoff scalar is a signed zero (one 32-bit
                    // select instead of a 64-bit one)
                    fm = (double)lj_f32u<SHIFT, UNIT>(a, ok[u] ? (float)rs[u] : __builtin_inff());
                }
                fx = fma(dx[u], fm, fx);
                fy = fma(dy[u], fm, fy);
                fz = fma(dz[u], fm, fz);
            }
        } else {
            // FP32 pair terms with Kahan-compensated FP32 accumulation
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float f = lj_f32u<SHIFT, UNIT>(a, (float)rs[u]);
                const float fm = ok[u] ? f : 0.0f;
                kahan_add(sxa, cxa, (float)dx[u] * fm);
                kahan_add(sya, cya, (float)dy[u] * fm);
                kahan_add(sza, cza, (float)dz[u] * fm);
            }
        }
        }
    }
    if (PREC != PREC_FP32_KAHAN) return make_double4(fx, fy, fz, 0.0);
    return make_double4(kahan_value(sxa, cxa), kahan_value(sya, cya), kahan_value(sza, cza), 0.0);
}


// The force on one atom by a group of G lanes, for boxes whose atoms do not
// fill the chip's lanes: lane s evaluates entries s, s + G, s + 2 G and
// s + 3 G of every 4 G, as lj_full_atom does, and leaves their terms in the wavefront's buffer in
// LDS; lane c of the group then adds component c of the 4 G terms in list
// order (the terms of absent entries are dx * 0), so the sum is
// lj_full_atom's bit for bit.  All lanes of a group call together, lane s with
// list group s in `next`: it fetches group s of every G for all of them,
// through LDS.  Lane c < 3 returns component c.
constexpr int kGroupLanes = 4;
constexpr int kGroupBufBytes = 8192 + 1024;  // of a wavefront: 256 entries of up to four doubles, 64 groups of list entries
// The buffers follow the window, whose slots are then an even number: list
// entries are stored and fetched 16 bytes at a time.
constexpr int group_window(int wcap) { return (wcap + 1) & ~1; }
constexpr bool group_bufs_aligned() {
    for (int wcap = 1; wcap <= 4; ++wcap)
        if (group_window(wcap) < wcap || group_window(wcap) * 3 * (int)sizeof(double) % (int)alignof(int4) != 0) return false;
    return kGroupBufBytes % alignof(int4) == 0 && (kGroupBufBytes - 1024) % alignof(int4) == 0;
}
static_assert(group_bufs_aligned(), "list entries are 16-byte accesses");
template <bool PAIR2>  // list group g (clamped), column 2's groups behind column 1's
__device__ __forceinline__ int4 group_entries(int g, int cnt, const int4* __restrict__ lp, int cnt2, const int4* __restrict__ lp2) {
    const int ng1 = (cnt + 7) >> 3, ng = ng1 + (PAIR2 ? (cnt2 + 7) >> 3 : 0);
    g = max(min(g, ng - 1), 0);
    return ld_stream((!PAIR2 || g < ng1) ? lp + (size_t)g * 64 : lp2 + (size_t)(g - ng1) * 64);
}
template <int PREC, int SHIFT, int UNIT, bool STAGED, bool PAIR2, class SP>
__device__ __forceinline__ double lj_group_atom(const double4 pi, int cnt, const int4* __restrict__ lp, const WinStage& sp,
                                                const SP& spos, const TileWin& W, const LJArgs& a, int4 next, int cnt2,
                                                const int4* __restrict__ lp2, double* buf) {
    constexpr int G = kGroupLanes, A = kWave / G, U = 4, E = U * G;  // atoms of a wavefront, entries of a round
    const int s = threadIdx.x & (G - 1), c = min(s, 2);
    const int far = win_size(W);             // sentinel slot
    double* const mine = buf + (threadIdx.x & (kWave - 1)) / G;
    float* const minef = reinterpret_cast<float*>(buf) + (threadIdx.x & (kWave - 1)) / G;
    const int ng1 = (cnt + 7) >> 3;
    const int ng = ng1 + (PAIR2 ? (cnt2 + 7) >> 3 : 0);
    int4* const lists = reinterpret_cast<int4*>(buf + 1024) + (threadIdx.x & (kWave - 1));
    const nb_t* const list = reinterpret_cast<const nb_t*>(lists - s);
    double F = 0.0;
    float fs = 0.f, fc = 0.f;
    for (int base = 0; base < 8 * ng; base += E) {
        if (base % (8 * G) == 0) {
            *lists = next;
            next = group_entries<PAIR2>(base / 8 + G + s, cnt, lp, cnt2, lp2);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        double d[U][3], rs[U];
        bool ok[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = base + s + u * G, g = e >> 3;
            const bool valid = (!PAIR2 || g < ng1) ? e < cnt : e - 8 * ng1 < cnt2;
            const int t = list[e % (8 * G)];
            double xj, yj, zj;
            win_pos<STAGED>(valid ? t : (STAGED ? far : 0), sp, spos, W, xj, yj, zj);
            d[u][0] = pi.x - xj;
            d[u][1] = pi.y - yj;
            d[u][2] = pi.z - zj;
            rs[u] = PREC == PREC_FP64 ? d[u][0] * d[u][0] + d[u][1] * d[u][1] + d[u][2] * d[u][2]
                                      : fma(d[u][0], d[u][0], fma(d[u][1], d[u][1], d[u][2] * d[u][2]));
            ok[u] = valid && rs[u] < a.rc2;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = u * G + s;
            if (PREC == PREC_FP64) {
                double sr6;
                const double f = lj_f64u<SHIFT, UNIT>(a, rs[u], sr6);
                const double fm = ok[u] ? f : 0.0;
#pragma unroll
                for (int x = 0; x < 3; ++x) mine[(3 * k + x) * A] = d[u][x] * fm;
            } else {
                float f;
                if (SHIFT || PREC == PREC_FP32_KAHAN) {
                    f = lj_f32u<SHIFT, UNIT>(a, (float)rs[u]);
                    f = ok[u] ? f : 0.0f;
                } else {
                    f = lj_f32u<SHIFT, UNIT>(a, ok[u] ? (float)rs[u] : __builtin_inff());
                }
                if (PREC == PREC_FP32_MIXED) {
#pragma unroll
                    for (int x = 0; x < 3; ++x) mine[(4 * k + x) * A] = d[u][x];
                    mine[(4 * k + 3) * A] = (double)f;
                } else {
#pragma unroll
                    for (int x = 0; x < 3; ++x) minef[(3 * k + x) * A] = (float)d[u][x] * f;
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k0 = 0; k0 < E; k0 += 4) {
            if (PREC == PREC_FP32_KAHAN) {
                // a zero is not nothing to a compensated sum: only the halves of
                // list groups that lj_full_atom takes
                const int e = base + k0, g = e >> 3;
                if ((e & 4) >= ((!PAIR2 || g < ng1) ? cnt - 8 * g : cnt2 - 8 * (g - ng1))) continue;
            }
#pragma unroll
            for (int k = k0; k < k0 + 4; ++k) {
                if (PREC == PREC_FP64) F = F + mine[(3 * k + c) * A];
                else if (PREC == PREC_FP32_MIXED) F = fma(mine[(4 * k + c) * A], mine[(4 * k + 3) * A], F);
                else kahan_add(fs, fc, minef[(3 * k + c) * A]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    return PREC != PREC_FP32_KAHAN ? F : kahan_value(fs, fc);
}

// Energy and virial terms of one atom's list entries (FP64): U = 4 eps
// (sr12 - sr6) [+ shift terms], W = f r^2.  Full lists weight every entry
// 1/2; half lists weight local-local entries 1 and local-ghost entries 1/2
// (an index j >= nloc_end is a ghost).  Entries are read 8 at a time (one
// 16-byte load per group, as in the force pass) and summed in list order.
template <int SHIFT, bool STAGED, class SP>
__device__ __forceinline__ void lj_energy_atom(const double4 pi, int cnt, const int4* __restrict__ lp, const WinStage& sp,
                                               const SP& spos, const int* __restrict__ parts,
                                               const TileWin& W, const LJArgs& a, int half, int nloc_end, double& pe,
                                               double& vir, double& np) {
    const int ng = (cnt + 7) >> 3;
    // the next group of 8 entries is loaded while the current one is used
    int4 q = ld_stream(lp);  // group 0 of the column always exists (capacity >= 8)
    for (int gi = 0; gi < ng; ++gi) {
        const int4 e = q;
        q = ld_stream(lp + (size_t)min(gi + 1, ng - 1) * 64);  // next group (clamped: always a valid load)
        const int kend = cnt - gi * 8;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            // staged, the entries past the count are the sentinel slot (far
            // away, j = -1) and fail the cutoff test; from the mirror they
            // would index past the window
            if (!STAGED && u >= kend) break;
            const int t = nb_entry(e, u);
            int j;
            double xj, yj, zj;
            if (STAGED) {
                j = sp.j[t];
                xj = sp.xyz[3 * t + 0]; yj = sp.xyz[3 * t + 1]; zj = sp.xyz[3 * t + 2];
            } else {
                const int kk = win_index(t, W);
                j = parts[kk];
                const double4 p = spos[kk];
                xj = p.x; yj = p.y; zj = p.z;
            }
            const double dx = pi.x - xj, dy = pi.y - yj, dz = pi.z - zj;
            const double rsq = dx * dx + dy * dy + dz * dz;
            if (rsq < a.rc2) {
                const double sr2 = rcp_round(rsq);
                const double sr6 = sr2 * sr2 * sr2 * a.sigma6;
                double f = 48.0 * sr6 * (sr6 - 0.5) * sr2 * a.eps;
                double uu = 4.0 * a.eps * sr6 * (sr6 - 1.0);
                if (SHIFT) {
                    const double ds = rsq - a.rc2;
                    f = f - a.fc - ds * a.dfc;
                    uu = uu - a.uc + ds * (0.5 * a.fc) + ds * ds * (0.25 * a.dfc);
                } else if (a.eshift != 0.0) {
                    uu = uu - a.eshift;
                }
                const double wt = half ? (j < nloc_end ? 1.0 : 0.5) : 0.5;
                pe += wt * uu;
                vir += wt * (f * rsq);
                np += 1.0;
            }
        }
    }
}

struct NbArgs {
    int n, cap, half, half_mode, wcap;  // n: first ghost index (locals are below it)
    double cut2;
    TileGeom g;
};

// A list column being written by its lane: entries wait in the lane's ring of
// 16-bit slots in LDS (slot-major, so a wavefront's accesses spread over the
// banks) and leave in whole groups of 8, one 16-byte store each, when the
// ring of some lane would overflow, once in several chunks.  Kept in
// registers instead, nearly every pair of entries met some lane that
// completed a group, and the store's instructions ran at every step.
template <int SLOTS>
struct RingCol {
    int4* col;
    unsigned ngroups;
    nb_t* ring;         // the lane's slot 0; slots are kWave apart
    unsigned at, done;  // entries so far and entries stored, times kWave
    __device__ __forceinline__ RingCol(int4* c, int ng, nb_t* r) : col(c), ngroups((unsigned)ng), ring(r), at(0u), done(0u) {}
    __device__ __forceinline__ int count() const { return (int)(at / kWave); }
    __device__ __forceinline__ nb_t& slot(unsigned e) const { return ring[e & (unsigned)((SLOTS - 1) * kWave)]; }
    __device__ __forceinline__ void store_group() {
        const nb_t* q = &slot(done);
        unsigned d[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) d[k] = (unsigned)q[2 * k * kWave] | (unsigned)q[(2 * k + 1) * kWave] << 16;
        // groups beyond the capacity are counted, not stored
        const unsigned grp = done / (8 * kWave);
        if (grp < ngroups) col[(size_t)grp * 64] = make_int4((int)d[0], (int)d[1], (int)d[2], (int)d[3]);
        done += 8 * kWave;
    }
    __device__ __forceinline__ void flush() {
        while (at - done >= 8 * kWave) store_group();
    }
    __device__ __forceinline__ void append(unsigned m, unsigned base) {
        while (m != 0u) {
            slot(at) = (nb_t)(base + (unsigned)__builtin_ctz(m));
            m &= m - 1u;
            at += kWave;
        }
    }
    __device__ __forceinline__ bool full(unsigned m) const { return at - done + kWave * __builtin_popcount(m) > SLOTS * kWave; }
    // the set bits of m (bit b: entry base + b) in ascending order
    __device__ __forceinline__ void push_mask(unsigned m, unsigned base) {
        if (__ballot(full(m))) {
            flush();
            if (__ballot(full(m))) {  // at most 7 wait: a byte at a time always fits
                for (int k = 0; k < 32; k += 8) {
                    append(m & (0xffu << k), base);
                    flush();
                }
                return;
            }
        }
        append(m, base);
    }
    // the last group's free slots hold the window's sentinel offset
    __device__ __forceinline__ void finish(unsigned pad) {
        flush();
        const unsigned cnt = at;
        if (at > done) {
            while (at - done < 8 * kWave) {
                slot(at) = (nb_t)pad;
                at += kWave;
            }
            store_group();
        }
        at = cnt;
    }
};
constexpr int ring_bytes(int slots) { return slots * kWave * 2; }  // of a wavefront

// The list build's window in LDS: FP32 positions relative to a point of the
// tile, and the atom index.
struct NbCand {
    float x, y, z;
    int j;
};
constexpr int kCandBytes = 16;
struct ListWin {
    NbCand* c;
    int* cst;     // row starts (stage_row_starts)
    nb_t* ring;   // the wavefronts' rings
    double4 ref;  // the point
    float sure;   // a squared distance off the cutoff's by more than this has the FP64 test's outcome
};
// LDS of a block's list build: `wcap` window slots, tables of `tab` bytes and
// the rings of as many wavefronts as there is room for, of the `want` that
// take the fullest tile at once; with fewer (at least kListWaves, at the cost
// of window slots), as few as do not need another round.  A lane has 32 ring
// slots (half lists: 16 for each column), or 16 where 32 leave too few
// wavefronts: 64 replicas with tiles of up to 668 atoms, 11 wavefronts instead
// of two rounds of 6, 37.5 against 38.2 ms for 200 steps; with room for all,
// 16 slots cost 4 % of a build in more frequent stores.
constexpr int kListWaves = 4;
struct ListLds {
    int wcap, waves, slots, bytes;
};
inline ListLds list_lds(int window, int tab, int want, bool half) {
    ListLds l;
    const int left = kLdsBudget - tab - window * kCandBytes;
    l.slots = half || left / ring_bytes(32) >= want ? 32 : 16;
    const int ring = ring_bytes(l.slots);
    l.waves = std::min(want, std::max(left / ring, kListWaves));
    const int rounds = (want + l.waves - 1) / l.waves;
    l.waves = (want + rounds - 1) / rounds;
    l.wcap = std::min(window, (kLdsBudget - tab - l.waves * ring) / kCandBytes);
    l.bytes = l.wcap * kCandBytes + tab + l.waves * ring;
    return l;
}
__device__ __forceinline__ ListWin list_win(double* dyn, int wcap, const TileGeom& g, const double4& ref) {
    ListWin L;
    L.c = reinterpret_cast<NbCand*>(dyn);
    L.cst = reinterpret_cast<int*>(L.c + wcap);
    L.ring = reinterpret_cast<nb_t*>(L.cst + row_starts_bytes(g) / 4);
    L.ref = ref;
    L.sure = 0.0f;
    return L;
}

// What the FP32 test may be off by.  With u = 2^-24 and R the largest
// coordinate of the window, a difference d is off by 2 u R + u |d|, its
// square's sum over a distance r by u (7 R r + 2 r^2), and the three sums
// from -cut2 by u (4 cut2 + 3 r^2): where the sign is wrong, r is within that
// of the cutoff, and the sum is below u (7.4 R rc + 10 cut2).  Outside FP32's
// comfortable range, or with a window 1e5 cutoffs wide, nothing is sure.
__device__ __forceinline__ float list_sure(float R, double cut2) {
    if (!(cut2 > 1e-12 && cut2 < 1e12 && (double)R * (double)R < 1e10 * cut2)) return __builtin_inff();
    const float c2 = (float)cut2;
    return 16.0f / 16777216.0f * (R * sqrtf(c2) + c2);
}

// Stage the list build's window if it fits wcap atoms.  Whole block; maxr
// (shared, largest coordinate's bits) is zero and visible before.
template <bool HALF, class SP>
__device__ __forceinline__ bool stage_list_window(const TileWin& W, int wcap, const SP& spos, const int* __restrict__ parts,
                                                  double cut2, ListWin& L, unsigned* maxr) {
    const int S = win_size(W);
    const bool staged = S + kListPad <= wcap;
    if (staged) {
        double4 p[kStageInFlight];
        int j[kStageInFlight];
        float R = 0.0f;
        stage_rows(W, [&](int k, int u) { p[u] = spos[k]; if (HALF) j[u] = parts[k]; },
                   [&](int t, int u) {
                       const float x = (float)(p[u].x - L.ref.x), y = (float)(p[u].y - L.ref.y), z = (float)(p[u].z - L.ref.z);
                       L.c[t] = NbCand{x, y, z, HALF ? j[u] : 0};
                       R = fmaxf(fmaxf(R, fabsf(x)), fmaxf(fabsf(y), fabsf(z)));
                   });
        if ((int)threadIdx.x < kListPad) L.c[S + (int)threadIdx.x] = NbCand{0.0f, 0.0f, 0.0f, 0};  // masked
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) R = fmaxf(R, __shfl_xor(R, o));
        if ((threadIdx.x & (kWave - 1)) == 0) atomicMax(maxr, __float_as_uint(R));
    }
    __syncthreads();
    if (staged) L.sure = list_sure(__uint_as_float(*maxr), cut2);
    return staged;
}

// Verlet list of local atom i (work slot w, cell c of the tile's grid,
// cell-ordered index k_i) from its tile's window: 9 stencil rows of 3 cells
// in the reference's order, `rsq <= cut2` in FP64 without contraction.  Each
// row is taken in chunks of 32 candidates that produce a bit mask (bit b:
// candidate tc + b accepted); i itself is removed from the mask by its window
// offset, and the set bits are appended in ascending order, which is the
// reference's order.
//
// Bounds: vector instructions.  A staged candidate is tested in FP32 (6
// instructions and one for its bit, 12 bytes of LDS; the FP64 test took 10
// and 24 bytes), which is exact but for candidates within `sure` of the
// cutoff; a chunk that holds one (about one atom in 1,000 meets one) is
// repeated by the FP64 test.  Accepted candidates cost 9 instructions per
// round of a wavefront (RingCol), a third of what packing in registers took.
// A build at 80^3 cells took 722 us and takes 477 (268 M vector instructions
// a wavefront's lanes share, 99 % busy), half lists of 53 x 47 x 39 cells 288
// and 170.  The products -2 x_i . x_j on the matrix cores (32 x 32 tests for
// two products of depth 2 and one for the constants) left the signs to be
// gathered and three quarters of the candidates' slots padded, and took 870.
//
// HALF keeps j < i among locals (the reference's filter) plus, by default,
// every ghost, and also writes the complementary column (nb_list2, count in
// cnt2): the local neighbours j > i that the half list leaves to j's own
// list.  The pair force then needs no reaction scatter: atom i gathers its
// half-list entries and its complementary entries, which are exactly the
// pairs whose reactions the half list would have sent to i.  STAGED is a
// template parameter so that the staged loop addresses LDS directly (ds_read)
// rather than through generic pointers.
template <bool HALF, bool STAGED, int SLOTS, class SP>
__device__ __forceinline__ int nlist_atom(int i, int w, int c, int k_i, const double4 pi, const NbArgs& a, const TileWin& W,
                                          const ListWin& L, const SP& spos, const int* __restrict__ parts,
                                          nb_t* __restrict__ nb_list, nb_t* __restrict__ nb_list2, int& cnt2) {
    const int cx = c % a.g.nx, cy = (c / a.g.nx) % a.g.ny, cz = c / (a.g.nx * a.g.ny);
    const int wy = a.g.ty + 2;
    const int xo = cx - W.cx0;  // (cx - 1) - (cx0 - 1)
    const int per = a.g.tx + 3;
    const int s_own = (cz - (W.cz0 - 1)) * wy + (cy - (W.cy0 - 1));
    const int t_i = W.seg_off[s_own] + (k_i - W.seg_beg[s_own]);
    const size_t col_off = (size_t)(w >> 6) * (size_t)a.cap * 8 + (w & 63);
    nb_t* ring = L.ring + (threadIdx.x / kWave) * ((HALF ? 2 : 1) * SLOTS * kWave) + threadIdx.x % kWave;
    RingCol<SLOTS> A(reinterpret_cast<int4*>(nb_list) + col_off, a.cap >> 3, ring);
    RingCol<SLOTS> B(HALF ? reinterpret_cast<int4*>(nb_list2) + col_off : nullptr, a.cap >> 3, ring + SLOTS * kWave);
    const float xi = (float)(pi.x - L.ref.x), yi = (float)(pi.y - L.ref.y), zi = (float)(pi.z - L.ref.z);
    const float ncut2 = -(float)a.cut2;
    for (int r = 0; r < 9; ++r) {
        const int s = s_own + (r / 3 - 1) * wy + (r % 3 - 1);
        const int t0 = L.cst[s * per + xo], t1 = L.cst[s * per + xo + 3];
        const int k0 = W.seg_beg[s] - W.seg_off[s];  // mirror index less window offset, in this row
        for (int tc = t0; tc < t1; tc += 32) {
            const int te = min(tc + 32, t1);
            unsigned m = 0u, m2 = 0u;  // accepted; half lists: of those, locals j > i
            bool sure = false;
            if (STAGED) {
                // the candidates' sign bits are shifted in at the low end
                // (first candidate highest), a batch of 4 at a time: up to
                // three past te are read (window atoms or the slots behind
                // it) and masked below
                const int nbat = (te - tc + 3) >> 2;
                float near = __builtin_inff();
                const NbCand* q = L.c + tc;
                const NbCand* const end = q + 4 * nbat;
                do {
                    float d[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const float dx = xi - q[u].x, dy = yi - q[u].y, dz = zi - q[u].z;
                        d[u] = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, ncut2)));
                        m = __builtin_amdgcn_alignbit(m, __float_as_uint(d[u]), 31);
                        if (HALF) {
                            // i < j < n: neither j - (i + 1) nor (n - 1) - j is negative
                            const int j = q[u].j;
                            m2 = __builtin_amdgcn_alignbit(m2, (unsigned)((j - (i + 1)) | ((a.n - 1) - j)), 31);
                        }
                    }
                    near = fminf(fminf(near, fabsf(d[0])), fabsf(d[1]));
                    near = fminf(fminf(near, fabsf(d[2])), fabsf(d[3]));
                    q += 4;
                } while (q != end);
                sure = near > L.sure;
                // reversed, bit b is candidate tc + b
                m = __builtin_bitreverse32(m) >> (32 - 4 * nbat);
                if (HALF) m2 = ~(__builtin_bitreverse32(m2) >> (32 - 4 * nbat));
            }
            if (!sure) {
                m = 0u;
                if (!STAGED) m2 = 0u;
                for (int t = tc; t < te; ++t) {
                    const double4 p = spos[k0 + t];
                    const double dx = pi.x - p.x, dy = pi.y - p.y, dz = pi.z - p.z;
                    const double rsq = dx * dx + dy * dy + dz * dz;
                    const unsigned bit = 1u << (t - tc);
                    m |= rsq <= a.cut2 ? bit : 0u;
                    if (HALF && !STAGED) {
                        const int j = parts[k0 + t];
                        m2 |= j > i && j < a.n ? bit : 0u;
                    }
                }
            }
            m &= 0xffffffffu >> (32 - (te - tc));  // candidates of this chunk only
            if (r == 4) m &= ~(unsigned)(1ull << min((unsigned)(t_i - tc), 32u));  // i is not its own neighbour
            if (HALF) {
                m2 &= m;
                B.push_mask(m2, (unsigned)tc);
                m &= ~m2;
                if (a.half_mode == HALF_REF_LITERAL && m != 0u) {  // no ghosts either
                    for (unsigned q = m; q != 0u; q &= q - 1u) {
                        const int t = tc + __builtin_ctz(q);
                        if ((STAGED ? L.c[t].j : parts[k0 + t]) >= a.n) m &= ~(q & (0u - q));
                    }
                }
            }
            A.push_mask(m, (unsigned)tc);
        }
    }
    const unsigned pad = (unsigned)win_size(W);
    A.finish(pad);
    if (HALF) B.finish(pad);
    cnt2 = B.count();
    return A.count();
}

}  // namespace tmd
