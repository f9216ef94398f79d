// msm_walk.hip -- density and force passes over the global neighbour list, 1 to 32 lanes per atom.
//
// A wave takes a unit of 64 / L consecutive cell-sorted atoms, L lanes each (lanes l, l + 1, ... of
// an atom take its slots l, l + L, ...), so the unit's list rows share one 64-atom block: the
// block's base is a scalar and every index load is that base plus a 32-bit lane offset.  The
// per-atom arrays are read the same way (base + 32-bit byte offset; the launchers are for
// n < kWalkMaxAtoms, whose records lie below 4 GB).
//
// Below about 10^5 atoms a pass is the length of one wave's chain of loads (state, indices, records,
// knots) after about 4 us of launch; above, the vector memory pipe (a record per pair: 1.1 line
// accesses a clock and CU, the data return 97 % busy on a million W atoms, the VALU 55 %).  So
//  - a unit whose atoms all lie further than the list radius from the periodic faces of their box
//    ("inner": four fifths of a million-atom box) evaluates its pairs without the minimum image.
//    The knot index tells a pair that might need it after all (its distance reaches half the
//    shortest box length); such a pair adds nothing in the loop and is evaluated afterwards by the
//    general formula, so the result is that of the general formula whatever the positions are;
//  - the LDS window holds the upper five eighths of the table (r above a seventh of the cutoff)
//    from arrays of knot values alone, which halves its fill; a pair below it takes the same side
//    road;
//  - small boxes take more lanes per atom and read the knots from global memory (the choice and
//    its measurements are with the plan in msm_api.hip).
// Density / force pass, HIP events (about 4 us of them overhead), against the two-lane passes with
// whole-table windows: 2,000 W atoms 14.9 / 17.5 -> 6.2 / 8.1 us, 16,000 14.9 / 17.8 -> 8.5 / 10.1,
// 137,000 25.7 / 31.0 -> 17.8 / 21.4, a million 78.7 / 99.5 -> 75 / 93; Cu-Ni 4,000 atoms
// 45.0 / 52.4 -> 8.6 / 11.6, 442,000 158 / 195 -> 121 / 146.
// The arithmetic of a pair is that of the reference:
//   T(KK) + DK * (T(KK+1) - T(KK)),  SK = sqrt(sqrt(r2)) * CSI, KK = int(SK), DK = SK - KK
//   (MD_FS_ForceTable_GPU.F90 PRECALFOR/CALFORCE kernels).
#include "msm_walk.h"

namespace msm {

// --------------------------------------------------------------------------------------------
// density
// --------------------------------------------------------------------------------------------

// Terms of the odd pairs among slots s, s + 1, ... (bits), by the general formula from the global
// table.
template <int MT, int LG>
__device__ __forceinline__ double density_odd(const AtomsDev& a, const TabDev& t, const BoxDev& b,
                                              const Lane& q, int s, unsigned bits, double px,
                                              double py, double pz, double den) {
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
        const int kk = min(static_cast<int>(sk), t.ntab2 - 2);
        const double2 e = t.b2[static_cast<size_t>(kind) * t.ntab2 + kk];
        den = den + (e.x + (sk - kk) * e.y);
    }
    return den;
}

// Slots s .. s + G - 1 of a lane (FULL: all in the list).  js: their indices; on return those of
// the next group (the last slot's beyond the end of the list).
template <int G, int FULL, int MT, int IMG, int L, int TL>
__device__ __forceinline__ double density_slots(const AtomsDev& a, const TabDev& t,
                                                const WalkDev& w, const BoxDev& b, const Lane& q,
                                                const Knots<TL>& kn, const int* s_row, int s,
                                                double px, double py, double pz, double den,
                                                int (&js)[G]) {
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
        const bool valid = FULL || listed<L>(q, s + u);
        double v, dv;
        kn.den(p.q + (MT ? s_row[q.ti * t.ngroup + tj[u]] : 0), v, dv);
        v = v + p.dk * dv;
        den = den + ((p.ok && valid) ? v : 0.0);
        odd.note(u, p.odd && valid);
    }
    if (__builtin_expect(odd.some(), 0))
        den = density_odd<MT, LG>(a, t, b, q, s, odd.slots(), px, py, pz, den);
    return den;
}

template <int MB, int MT, int EAM, int L, int TL>
__global__ __launch_bounds__(TL ? kLtMaxBlock : kBlock) void k_density_w(
    AtomsDev a, ListDev l, TabDev t, BoxDev box0, const BoxDev* __restrict__ boxes, WalkDev w,
    int* err) {
    constexpr int G = group_d(L), A = 64 / L;
    extern __shared__ double s_dyn[];
    __shared__ int s_row[MT ? kMaxGroup * kMaxGroup : 1];
    Knots<TL> kn;
    if constexpr (MT) {
        for (int k = threadIdx.x; k < t.ngroup * t.ngroup; k += blockDim.x)
            s_row[k] = t.kpair[k] * (TL ? w.w : t.ntab2);
    }
    if constexpr (TL) {
        const int nk = MT ? t.nkind : 1;
        for (int k = threadIdx.x; k < nk * w.w; k += blockDim.x) {
            const int kd = MT ? k / w.w : t.kpair[0], q = MT ? k % w.w : k;
            s_dyn[k] = t.b1[static_cast<size_t>(kd) * t.ntab2 + w.k0 + q];
        }
        kn.d = s_dyn;
        kn.f = nullptr;
    } else {
        kn.d = t.b2 + (MT ? 0 : static_cast<size_t>(t.kpair[0]) * t.ntab2);
        kn.f = nullptr;
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
        // the atom's loads in one batch, with the first group's slot indices (masked by
        // the list length once it is known)
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
        double den = 0.0;
        if (q.kv > 0) {
            auto slots = [&](auto img) {
                constexpr int IMG = decltype(img)::value;
                int s = 0;
                for (; (s + G) * L <= q.kv; s += G)
                    den = density_slots<G, 1, MT, IMG, L, TL>(a, t, w, b, q, kn, s_row, s, pxy.x,
                                                               pxy.y, pz, den, js);
                if (s * L < q.kv)
                    den = density_slots<G, 0, MT, IMG, L, TL>(a, t, w, b, q, kn, s_row, s, pxy.x,
                                                               pxy.y, pz, den, js);
            };
            if (fast)
                slots(std::integral_constant<int, 0>{});
            else
                slots(std::integral_constant<int, 1>{});
        }
        den = atom_sum<L>(den);
        if (sub != 0 || !have) continue;
        if (active && den > 0.0) {
            if constexpr (!EAM) {
                den = fs_fprime(den);
            } else {
                const double sk = den / t.rhod + 1.0;
                int kk = static_cast<int>(sk + 0.000001);
                if (kk > t.nembd) {
                    err[kErrEmbd] = 1;
                    kk = t.nembd;
                }
                const double4 m = t.m4[t.kembd[q.ti] * t.nembd2 + kk];
                den = m.z + (sk - kk) * m.w;
            }
        }
        at(a.pos, q.ib * 32u).w = den;
    }
}

// --------------------------------------------------------------------------------------------
// force
// --------------------------------------------------------------------------------------------

template <int MB, int MT, int MODE, int L, int TL>
__global__ __launch_bounds__(TL ? kLtMaxBlock : kBlock) void k_force_w(
    AtomsDev a, ListDev l, TabDev t, BoxDev box0, const BoxDev* __restrict__ boxes, StepParams sp,
    WalkDev w) {
    constexpr int G = group_f(L), A = 64 / L;
    extern __shared__ double2 s_dyn2[];
    __shared__ int s_row[MT ? kMaxGroup * kMaxGroup : 1];
    Knots<TL> kn;
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
        kn.d = nullptr;
        kn.f = s_dyn2;
    } else {
        kn.d = nullptr;
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
        // the atom's loads in one batch: state, list length, the first group's slot indices and
        // (first lane) what the integrator needs at the end
        int js[G];
        const int st = at(a.statu, q.ib * 4u), kv = at(l.kvois, q.ib * 4u);
        const double4 pi = at(a.pos, q.ib * 32u);
        q.ti = MT ? at(a.ityp, q.ib * 4u) : 0;
#pragma unroll
        for (int k = 0; k < G; ++k)
            js[k] = slot_at(q.blk, row + static_cast<unsigned>(sub + k * L) * 256u);
        AtomState as;
        if constexpr (MODE >= 1)
            if (sub == 0) load_atom_state(a, sp, AtomIx{q.ib}, as);
        const BoxDev& b = box_of<MB>(box0, boxes, a.boxid, static_cast<int>(q.ib));
        const bool active = have && (st & STATU_ACTIVE) == STATU_ACTIVE;
        q.kv = active ? kv : 0;
        q.sub = sub;
        const bool fast = w.kimg > 0 && !__any(active && !inner(b, w.margin, pi.x, pi.y, pi.z));
        double fx = 0.0, fy = 0.0, fz = 0.0, vir[6];
        if (q.kv > 0) {
            auto slots = [&](auto img) {
                constexpr int IMG = decltype(img)::value;
                int s = 0;
                for (; (s + G) * L <= q.kv; s += G)
                    force_slots<G, 1, MT, IMG, L, TL, 0>(a, t, w, b, q, kn, s_row, s, pi, fx, fy,
                                                         fz, vir, js);
                if (s * L < q.kv)
                    force_slots<G, 0, MT, IMG, L, TL, 0>(a, t, w, b, q, kn, s_row, s, pi, fx, fy,
                                                         fz, vir, js);
            };
            if (fast)
                slots(std::integral_constant<int, 0>{});
            else
                slots(std::integral_constant<int, 1>{});
        }
        fx = atom_sum<L>(fx);
        fy = atom_sum<L>(fy);
        fz = atom_sum<L>(fz);
        if (sub != 0 || !have) continue;
        if (sp.write_f) {
            at(a.fx, q.ib * 8u) = fx;
            at(a.fy, q.ib * 8u) = fy;
            at(a.fz, q.ib * 8u) = fz;
        }
        if constexpr (MODE >= 1)
            integrate_atom<MODE>(a, t, b, sp, AtomIx{q.ib}, st, active, pi, q.ti, fx, fy, fz, &as);
    }
}

bool walk_window_ok(const TabDev& t, int force, int wgs) {
    WalkDev w{};
    window(t, walk_budget(t, wgs), force ? 16 : 8, w);
    return 2 * w.w >= t.ntab2;
}

void launch_density_walk(const WalkPlan& pl, const AtomsDev& a, const ListDev& l,
                         const TabDev& t, const BoxDev& box0,
                         const BoxDev* boxes, int multibox, int* err, hipStream_t s) {
    if (a.n <= 0) return;
    const bool mt = t.ngroup > 1, eam = t.pot_type != 0;
    WalkDev w{};
    int threads = 0;
    size_t lds = 0;
#define MSM_DW(MB, E, L, TL)                                                                     \
    do {                                                                                         \
        auto k = mt ? k_density_w<MB, 1, E, L, TL> : k_density_w<MB, 0, E, L, TL>;               \
        const unsigned g = walk_launch(k, pl, 8, a.n, t, w, threads,    \
                                       lds);                                                     \
        hipLaunchKernelGGL(k, dim3(g), dim3(threads), lds, s, a, l, t, box0, boxes, w, err);     \
    } while (0)
#define MSM_DWL(MB, E)                                  \
    do {                                                \
        if (pl.tl) {                                    \
            if (pl.lanes == 1) MSM_DW(MB, E, 1, 1);   \
            else if (pl.lanes == 2) MSM_DW(MB, E, 2, 1); \
            else if (pl.lanes == 4) MSM_DW(MB, E, 4, 1); \
            else MSM_DW(MB, E, 8, 1);                   \
        } else {                                        \
            if (pl.lanes == 8) MSM_DW(MB, E, 8, 0);   \
            else if (pl.lanes == 16) MSM_DW(MB, E, 16, 0); \
            else MSM_DW(MB, E, 32, 0);                  \
        }                                               \
    } while (0)
    if (multibox) {
        if (eam) MSM_DWL(1, 1); else MSM_DWL(1, 0);
    } else {
        if (eam) MSM_DWL(0, 1); else MSM_DWL(0, 0);
    }
#undef MSM_DWL
#undef MSM_DW
}

void launch_force_walk(const WalkPlan& pl, const AtomsDev& a, const ListDev& l,
                       const TabDev& t, const BoxDev& box0,
                       const BoxDev* boxes, int multibox, const StepParams& sp, hipStream_t s) {
    if (a.n <= 0) return;
    const bool mt = t.ngroup > 1;
    WalkDev w{};
    int threads = 0;
    size_t lds = 0;
#define MSM_FW(MB, M, L, TL)                                                                     \
    do {                                                                                         \
        auto k = mt ? k_force_w<MB, 1, M, L, TL> : k_force_w<MB, 0, M, L, TL>;                   \
        const unsigned g = walk_launch(k, pl, 16, a.n, t, w, threads,   \
                                       lds);                                                     \
        hipLaunchKernelGGL(k, dim3(g), dim3(threads), lds, s, a, l, t, box0, boxes, sp, w);      \
    } while (0)
#define MSM_FWL(MB, M)                                  \
    do {                                                \
        if (pl.tl) {                                    \
            if (pl.lanes == 1) MSM_FW(MB, M, 1, 1);   \
            else if (pl.lanes == 2) MSM_FW(MB, M, 2, 1); \
            else if (pl.lanes == 4) MSM_FW(MB, M, 4, 1); \
            else MSM_FW(MB, M, 8, 1);                   \
        } else {                                        \
            if (pl.lanes == 8) MSM_FW(MB, M, 8, 0);   \
            else if (pl.lanes == 16) MSM_FW(MB, M, 16, 0); \
            else MSM_FW(MB, M, 32, 0);                  \
        }                                               \
    } while (0)
#define MSM_FWM(MB)                             \
    do {                                        \
        if (sp.mode == 0) MSM_FWL(MB, 0);       \
        else if (sp.mode == 1) MSM_FWL(MB, 1);  \
        else MSM_FWL(MB, 2);                    \
    } while (0)
    if (multibox) MSM_FWM(1); else MSM_FWM(0);
#undef MSM_FWM
#undef MSM_FWL
#undef MSM_FW
}

}  // namespace msm
