// msm_walk_energy.hip -- per-atom energies and virials over the neighbour list, with the lanes and the
// table placement of the density and force passes (msm_walk.hip).
//
// Energy (CALEPOT_KERNEL, MD_FS_ForceTable_GPU.F90:1451-1609, MD_EAM_ForceTable_GPU.F90:1470-1636):
//   E_i = sum_j POTR/r + F(rho_i), rho_i = sum_j POTB
// from one read of {POTR, POTB}; since rho is there, F'(rho) can be left in pos.w as the density pass
// leaves it, so that a caller who needs energies and forces runs no density pass.
// Virial (CALPTENSOR_KERNEL, :998-1272): the force pass with the six components of FORTOT/2 s (x) s.
#include "msm_walk.h"

namespace msm {

namespace {

template <int MT, int LG>
__device__ __forceinline__ void energy_odd(const AtomsDev& a, const TabDev& t, const BoxDev& b,
                                           const Lane& q, int s, unsigned bits, double px,
                                           double py, double pz, double& er, double& den) {
#pragma unroll 1
    for (; bits; bits &= bits - 1) {
        const int j = slot_index(q, s + __builtin_ctz(bits), 8 + LG);
        const double2 qxy = *reinterpret_cast<const double2*>(&a.pos[j]);
        const double qz = a.pos[j].z;
        double sx = px - qxy.x, sy = py - qxy.y, sz = pz - qz;
        sx = min_image(sx, b.len[0], b.ilen[0]);
        sy = min_image(sy, b.len[1], b.ilen[1]);
        sz = min_image(sz, b.len[2], b.ilen[2]);
        const double r2 = sx * sx + sy * sy + sz * sz;
        if (!(r2 <= t.ru2max)) continue;
        const int kind = MT ? t.kpair[q.ti * t.ngroup + a.ityp[j]] : t.kpair[0];
        double inv_r;
        const double sk = table_coord(r2, t.csi, inv_r);
        const int kk = min(static_cast<int>(sk), t.ntab2 - 1);
        const double dk = sk - kk;
        const double4 e = t.e4[static_cast<size_t>(kind) * t.ntab2 + kk];
        er = er + (e.x + dk * e.y) * inv_r;
        den = den + (e.z + dk * e.w);
    }
}

// As density_slots of msm_walk.hip, for the pair energy and the density.
template <int G, int FULL, int MT, int IMG, int L, int TL>
__device__ __forceinline__ void energy_slots(const AtomsDev& a, const TabDev& t, const WalkDev& w,
                                             const BoxDev& b, const Lane& q, const Knots<TL>& kn,
                                             const int* s_row, int s, double px, double py,
                                             double pz, double& er, double& den, int (&js)[G]) {
    constexpr int LG = ilog2(L);
    double2 qxy[G];
    double qz[G];
    int tj[G];
#pragma unroll
    for (int u = 0; u < G; ++u) {
        if (!FULL && u > 0 && (s + u) * L >= q.kv) break;
        // x, y, z only: another wave may be writing the neighbour's w
        const unsigned j = slot_atom<FULL, L>(q, s + u, js[u]), o = j << 5;
        qxy[u] = *reinterpret_cast<const double2*>(&at(a.pos, o));
        qz[u] = at(a.pos, o).z;
        tj[u] = MT ? at(a.ityp, j << 2) : 0;
    }
    if constexpr (FULL) next_slots<G, LG>(q, s, js);
    OddPairs<G, FULL && TL> odd;
#pragma unroll
    for (int u = 0; u < G; ++u) {
        if (!FULL && u > 0 && (s + u) * L >= q.kv) break;
        double sx = px - qxy[u].x, sy = py - qxy[u].y, sz = pz - qz[u];
        if constexpr (IMG == 1) {
            sx = min_image(sx, b.len[0], b.ilen[0]);
            sy = min_image(sy, b.len[1], b.ilen[1]);
            sz = min_image(sz, b.len[2], b.ilen[2]);
        }
        const Place p = place<IMG>(t, w, sx * sx + sy * sy + sz * sz);
        const bool use = p.ok && (FULL || listed<L>(q, s + u));
        double v, dv, d, dd;
        kn.frc(p.q + (MT ? s_row[q.ti * t.ngroup + tj[u]] : 0), v, dv, d, dd);
        v = (v + p.dk * dv) * p.inv_r;
        d = d + p.dk * dd;
        er = er + (use ? v : 0.0);
        den = den + (use ? d : 0.0);
        odd.note(u, p.odd && (FULL || listed<L>(q, s + u)));
    }
    if (__builtin_expect(odd.some(), 0))
        energy_odd<MT, LG>(a, t, b, q, s, odd.slots(), px, py, pz, er, den);
}

}  // namespace

// rho_out (may be null): each atom's density sum (0 for inactive atoms).  write_fp: F' into pos.w.
template <int MB, int MT, int EAM, int L, int TL>
__global__ __launch_bounds__(TL ? kLtMaxBlock : kBlock) void k_energy_w(
    AtomsDev a, ListDev l, TabDev t, BoxDev box0, const BoxDev* __restrict__ boxes, WalkDev w,
    double* __restrict__ rho_out, int write_fp, int* err) {
    constexpr int G = 3, A = 64 / L;
    extern __shared__ double2 s_dyn2[];
    __shared__ int s_row[MT ? kMaxGroup * kMaxGroup : 1];
    Knots<TL> kn;
    kn.d = nullptr;
    if constexpr (MT) {
        for (int k = threadIdx.x; k < t.ngroup * t.ngroup; k += blockDim.x)
            s_row[k] = t.kpair[k] * (TL ? w.w : t.ntab2);
    }
    if constexpr (TL) {
        const int nk = MT ? t.nkind : 1;
        for (int k = threadIdx.x; k < nk * w.w; k += blockDim.x) {
            const int kd = MT ? k / w.w : t.kpair[0], q = MT ? k % w.w : k;
            s_dyn2[k] = t.e2[static_cast<size_t>(kd) * t.ntab2 + w.k0 + q];
        }
        kn.f = s_dyn2;
    } else {
        kn.f = t.e4 + (MT ? 0 : static_cast<size_t>(t.kpair[0]) * t.ntab2);
    }
    if constexpr (MT || TL) __syncthreads();
    const int lane = threadIdx.x & 63, pl = lane / L, sub = lane % L;
    int u, ustep, uend;
    unit_iter(w.units, w.sweep, u, ustep, uend);
    for (; u < uend; u += ustep) {
        const int p0 = u * A;
        Lane q;
        const int i = p0 + pl;
        const bool have = i < a.n;
        q.ib = static_cast<unsigned>(have ? i : a.n - 1);
        q.blk = uniform(l.indi + static_cast<size_t>(p0 >> 6) * l.mx * kListRow);
        const unsigned row = static_cast<unsigned>((p0 & 63) + pl) * 4u;
        q.lo = row + static_cast<unsigned>(sub) * 256u;
        int js[G];
        const int st = at(a.statu, q.ib * 4u), kv = at(l.kvois, q.ib * 4u);
        const double2 pxy = *reinterpret_cast<const double2*>(&at(a.pos, q.ib * 32u));
        const double pz = at(a.pos, q.ib * 32u).z;
        q.ti = MT ? at(a.ityp, q.ib * 4u) : 0;
#pragma unroll
        for (int k = 0; k < G; ++k)
            js[k] = slot_at(q.blk, row + static_cast<unsigned>(sub + k * L) * 256u);
        const BoxDev& b = box_of<MB>(box0, boxes, a.boxid, static_cast<int>(q.ib));
        const bool active = have && (st & STATU_ACTIVE) == STATU_ACTIVE;
        q.kv = active ? kv : 0;
        q.sub = sub;
        const bool fast = w.kimg > 0 && !__any(active && !inner(b, w.margin, pxy.x, pxy.y, pz));
        double er = 0.0, den = 0.0;
        if (q.kv > 0) {
            auto slots = [&](auto img) {
                constexpr int IMG = decltype(img)::value;
                int s = 0;
                for (; (s + G) * L <= q.kv; s += G)
                    energy_slots<G, 1, MT, IMG, L, TL>(a, t, w, b, q, kn, s_row, s, pxy.x, pxy.y,
                                                       pz, er, den, js);
                if (s * L < q.kv)
                    energy_slots<G, 0, MT, IMG, L, TL>(a, t, w, b, q, kn, s_row, s, pxy.x, pxy.y,
                                                       pz, er, den, js);
            };
            if (fast)
                slots(std::integral_constant<int, 0>{});
            else
                slots(std::integral_constant<int, 1>{});
        }
        er = atom_sum<L>(er);
        den = atom_sum<L>(den);
        if (sub != 0 || !have) continue;
        if (rho_out) at(rho_out, q.ib * 8u) = den;
        double f = den, fp = den;
        if (active) {
            if constexpr (!EAM) {
                f = -sqrt(den);
                if (den > 0.0) fp = fs_fprime(den);
            } else {
                const double sk = den / t.rhod + 1.0;
                int kk = static_cast<int>(sk + 0.000001);
                if (kk < 0) kk = 0;
                if (kk > t.nembd) {
                    err[kErrEmbd] = 1;
                    kk = t.nembd;
                }
                const double4 m = t.m4[t.kembd[q.ti] * t.nembd2 + kk];
                f = m.x + (sk - kk) * m.y;
                if (den > 0.0) fp = m.z + (sk - kk) * m.w;
            }
        }
        at(a.epot, q.ib * 8u) = er + f;
        if (write_fp) at(a.pos, q.ib * 32u).w = fp;
    }
}

// Forces and half virials (component-major in vir, stride a.n; zero for inactive atoms).
template <int MB, int MT, int L, int TL>
__global__ __launch_bounds__(TL ? kLtMaxBlock : kBlock) void k_virial_w(
    AtomsDev a, ListDev l, TabDev t, BoxDev box0, const BoxDev* __restrict__ boxes, WalkDev w,
    double* __restrict__ vir) {
    constexpr int G = 3, A = 64 / L;
    extern __shared__ double2 s_dyn2[];
    __shared__ int s_row[MT ? kMaxGroup * kMaxGroup : 1];
    Knots<TL> kn;
    kn.d = nullptr;
    if constexpr (MT) {
        for (int k = threadIdx.x; k < t.ngroup * t.ngroup; k += blockDim.x)
            s_row[k] = t.kpair[k] * (TL ? w.w : t.ntab2);
    }
    if constexpr (TL) {
        const int nk = MT ? t.nkind : 1;
        for (int k = threadIdx.x; k < nk * w.w; k += blockDim.x) {
            const int kd = MT ? k / w.w : t.kpair[0], q = MT ? k % w.w : k;
            s_dyn2[k] = t.f2[static_cast<size_t>(kd) * t.ntab2 + w.k0 + q];
        }
        kn.f = s_dyn2;
    } else {
        kn.f = t.f4 + (MT ? 0 : static_cast<size_t>(t.kpair[0]) * t.ntab2);
    }
    if constexpr (MT || TL) __syncthreads();
    const int lane = threadIdx.x & 63, pl = lane / L, sub = lane % L;
    int u, ustep, uend;
    unit_iter(w.units, w.sweep, u, ustep, uend);
    for (; u < uend; u += ustep) {
        const int p0 = u * A;
        Lane q;
        const int i = p0 + pl;
        const bool have = i < a.n;
        q.ib = static_cast<unsigned>(have ? i : a.n - 1);
        q.blk = uniform(l.indi + static_cast<size_t>(p0 >> 6) * l.mx * kListRow);
        const unsigned row = static_cast<unsigned>((p0 & 63) + pl) * 4u;
        q.lo = row + static_cast<unsigned>(sub) * 256u;
        int js[G];
        const int st = at(a.statu, q.ib * 4u), kv = at(l.kvois, q.ib * 4u);
        const double4 pi = at(a.pos, q.ib * 32u);
        q.ti = MT ? at(a.ityp, q.ib * 4u) : 0;
#pragma unroll
        for (int k = 0; k < G; ++k)
            js[k] = slot_at(q.blk, row + static_cast<unsigned>(sub + k * L) * 256u);
        const BoxDev& b = box_of<MB>(box0, boxes, a.boxid, static_cast<int>(q.ib));
        const bool active = have && (st & STATU_ACTIVE) == STATU_ACTIVE;
        q.kv = active ? kv : 0;
        q.sub = sub;
        const bool fast = w.kimg > 0 && !__any(active && !inner(b, w.margin, pi.x, pi.y, pi.z));
        double fx = 0.0, fy = 0.0, fz = 0.0, p[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        if (q.kv > 0) {
            auto slots = [&](auto img) {
                constexpr int IMG = decltype(img)::value;
                int s = 0;
                for (; (s + G) * L <= q.kv; s += G)
                    force_slots<G, 1, MT, IMG, L, TL, 1>(a, t, w, b, q, kn, s_row, s, pi, fx, fy,
                                                         fz, p, js);
                if (s * L < q.kv)
                    force_slots<G, 0, MT, IMG, L, TL, 1>(a, t, w, b, q, kn, s_row, s, pi, fx, fy,
                                                         fz, p, js);
            };
            if (fast)
                slots(std::integral_constant<int, 0>{});
            else
                slots(std::integral_constant<int, 1>{});
        }
        fx = atom_sum<L>(fx);
        fy = atom_sum<L>(fy);
        fz = atom_sum<L>(fz);
#pragma unroll
        for (int c = 0; c < 6; ++c) p[c] = atom_sum<L>(p[c]);
        if (sub != 0 || !have) continue;
        at(a.fx, q.ib * 8u) = fx;
        at(a.fy, q.ib * 8u) = fy;
        at(a.fz, q.ib * 8u) = fz;
#pragma unroll
        for (int c = 0; c < 6; ++c) vir[static_cast<size_t>(c) * a.n + q.ib] = p[c];
    }
}

void launch_energy_walk(const WalkPlan& pl, const AtomsDev& a, const ListDev& l, const TabDev& t,
                        const BoxDev& box0, const BoxDev* boxes, int multibox, double* rho_out,
                        int write_fp, int* err, hipStream_t s) {
    if (a.n <= 0) return;
    const bool mt = t.ngroup > 1, eam = t.pot_type != 0;
    WalkDev w{};
    int threads = 0;
    size_t lds = 0;
#define MSM_EW(MB, E, L, TL)                                                                     \
    do {                                                                                         \
        auto k = mt ? k_energy_w<MB, 1, E, L, TL> : k_energy_w<MB, 0, E, L, TL>;                 \
        const unsigned g = walk_launch(k, pl, 16, a.n, t, w, threads, lds);                      \
        hipLaunchKernelGGL(k, dim3(g), dim3(threads), lds, s, a, l, t, box0, boxes, w, rho_out,  \
                           write_fp, err);                                                       \
    } while (0)
#define MSM_EWL(MB, E)                                  \
    do {                                                \
        if (pl.tl) {                                    \
            if (pl.lanes <= 2) MSM_EW(MB, E, 2, 1);     \
            else if (pl.lanes == 4) MSM_EW(MB, E, 4, 1); \
            else MSM_EW(MB, E, 8, 1);                   \
        } else {                                        \
            if (pl.lanes <= 8) MSM_EW(MB, E, 8, 0);     \
            else if (pl.lanes == 16) MSM_EW(MB, E, 16, 0); \
            else MSM_EW(MB, E, 32, 0);                  \
        }                                               \
    } while (0)
    if (multibox) {
        if (eam) MSM_EWL(1, 1); else MSM_EWL(1, 0);
    } else {
        if (eam) MSM_EWL(0, 1); else MSM_EWL(0, 0);
    }
#undef MSM_EWL
#undef MSM_EW
}

void launch_virial_walk(const WalkPlan& pl, const AtomsDev& a, const ListDev& l, const TabDev& t,
                        const BoxDev& box0, const BoxDev* boxes, int multibox, double* vir,
                        hipStream_t s) {
    if (a.n <= 0) return;
    const bool mt = t.ngroup > 1;
    WalkDev w{};
    int threads = 0;
    size_t lds = 0;
#define MSM_VW(MB, L, TL)                                                                        \
    do {                                                                                         \
        auto k = mt ? k_virial_w<MB, 1, L, TL> : k_virial_w<MB, 0, L, TL>;                       \
        const unsigned g = walk_launch(k, pl, 16, a.n, t, w, threads, lds);                      \
        hipLaunchKernelGGL(k, dim3(g), dim3(threads), lds, s, a, l, t, box0, boxes, w, vir);     \
    } while (0)
#define MSM_VWL(MB)                                     \
    do {                                                \
        if (pl.tl) {                                    \
            if (pl.lanes <= 2) MSM_VW(MB, 2, 1);        \
            else if (pl.lanes == 4) MSM_VW(MB, 4, 1);   \
            else MSM_VW(MB, 8, 1);                      \
        } else {                                        \
            if (pl.lanes <= 8) MSM_VW(MB, 8, 0);        \
            else if (pl.lanes == 16) MSM_VW(MB, 16, 0); \
            else MSM_VW(MB, 32, 0);                     \
        }                                               \
    } while (0)
    if (multibox) MSM_VWL(1); else MSM_VWL(0);
#undef MSM_VWL
#undef MSM_VW
}

}  // namespace msm
