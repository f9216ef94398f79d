// msm_walk.hip -- density and force passes over the global neighbour list, 1 to 32 lanes per atom.
//
// A wave takes a unit of 64 / L consecutive cell-sorted atoms, L lanes each (lanes l, l + 1, ... of
// an atom take its slots l, l + L, ...), so the unit's list rows share one 64-atom block: the
// block's base is a scalar and every index load is that base plus a 32-bit lane offset.  The
// per-atom arrays are read the same way (base + 32-bit byte offset; the launchers are for
// n < kWalkMaxAtoms, whose records lie below 4 GB).
//
// Below about 10^5 atoms a pass is the length of one wave's chain of loads (state, indices, records,
// knots) after about 4 us of launch; above, the issue of the pair loop and the rate of the L1's
// line accesses (75 % and 67 % busy on a million W atoms) bound it together.  So
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
// 137,000 25.7 / 31.0 -> 17.6 / 20.7, a million 78.7 / 99.5 -> 79.1 / 96.4; Cu-Ni 4,000 atoms
// 45.0 / 52.4 -> 8.6 / 11.6, 442,000 158 / 195 -> 114 / 140.
// The arithmetic of a pair is that of the reference:
//   T(KK) + DK * (T(KK+1) - T(KK)),  SK = sqrt(sqrt(r2)) * CSI, KK = int(SK), DK = SK - KK
//   (MD_FS_ForceTable_GPU.F90 PRECALFOR/CALFORCE kernels).
#include <algorithm>
#include <type_traits>

#include "msm_device.h"

namespace msm {

namespace {

template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    const unsigned long long a = static_cast<unsigned long long>(__double_as_longlong(v));
    const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_mov_dpp(
        static_cast<int>(static_cast<unsigned>(a)), CTRL, 0xF, 0xF, true));
    const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_mov_dpp(
        static_cast<int>(static_cast<unsigned>(a >> 32)), CTRL, 0xF, 0xF, true));
    return __longlong_as_double(
        static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}

// Sum over the L consecutive lanes of an atom, in every lane (all lanes of the wave active):
// quad permutes, half-row and row mirrors, then a swizzle across the two rows of 16.
template <int L>
__device__ __forceinline__ double atom_sum(double v) {
    if constexpr (L >= 2) v = v + dpp<0xB1>(v);
    if constexpr (L >= 4) v = v + dpp<0x4E>(v);
    if constexpr (L >= 8) v = v + dpp<0x141>(v);
    if constexpr (L >= 16) v = v + dpp<0x140>(v);
    if constexpr (L >= 32) {
        const unsigned long long a = static_cast<unsigned long long>(__double_as_longlong(v));
        const unsigned lo = static_cast<unsigned>(
            __builtin_amdgcn_ds_swizzle(static_cast<int>(static_cast<unsigned>(a)), 0x401F));
        const unsigned hi = static_cast<unsigned>(
            __builtin_amdgcn_ds_swizzle(static_cast<int>(static_cast<unsigned>(a >> 32)), 0x401F));
        v = v + __longlong_as_double(
                    static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
    }
    return v;
}

// A pointer that is the same in every lane, in scalar registers.
__device__ __forceinline__ const int* uniform(const int* p) {
    const unsigned long long a = reinterpret_cast<unsigned long long>(p);
    const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(a));
    const unsigned hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(a >> 32));
    return reinterpret_cast<const int*>((static_cast<unsigned long long>(hi) << 32) | lo);
}

constexpr int ilog2(int v) { return v <= 1 ? 0 : 1 + ilog2(v / 2); }

// Slots per group: the gathers of a group are in flight together.
constexpr int group_d(int L) { return L <= 4 ? 6 : L == 8 ? 4 : 3; }
constexpr int group_f(int) { return 3; }

// What a lane needs of its unit.
struct Lane {
    const int* blk;   // list block of the unit's atoms (uniform)
    unsigned lo;      // byte offset of the lane's first slot in it
    unsigned ib;      // atom index
    int kv;           // list length (0: inactive)
    int sub;          // lane within the atom
    int last;         // the lane's last slot
    int ti;           // type
};

// Units of this wave: u = first, first + step, ... < end.  sweep = 0: each workgroup takes an
// equal contiguous range of its XCD's units, its waves in turn; sweep = 1: the workgroups of an
// XCD take that XCD's range in turn.
__device__ __forceinline__ void unit_iter(int units, int sweep, int& first, int& step, int& end) {
    const int nb = gridDim.x, nw = blockDim.x >> 6;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (!sweep || nb < 8) {
        const int b = xcd_block(nb);
        first = static_cast<int>(static_cast<long long>(b) * units / nb) + wv;
        end = static_cast<int>(static_cast<long long>(b + 1) * units / nb);
        step = nw;
    } else {
        const int x = blockIdx.x & 7, k = blockIdx.x >> 3;
        first = static_cast<int>(static_cast<long long>(x) * units / 8) + k * nw + wv;
        end = static_cast<int>(static_cast<long long>(x + 1) * units / 8);
        step = ((nb - x + 7) >> 3) * nw;
    }
}

// Whether an atom at (x, y, z) lies further than m from every periodic face of its box.
__device__ __forceinline__ bool inner(const BoxDev& b, double m, double x, double y, double z) {
    const double dx = x - b.lo[0], dy = y - b.lo[1], dz = z - b.lo[2];
    return (!b.ifpd[0] || (dx > m && b.len[0] - dx > m)) &&
           (!b.ifpd[1] || (dy > m && b.len[1] - dy > m)) &&
           (!b.ifpd[2] || (dz > m && b.len[2] - dz > m));
}

__device__ __forceinline__ int slot_index(const Lane& q, int s, int shift) {
    return at(q.blk, q.lo + (static_cast<unsigned>(s) << shift));
}

// Knots: from the LDS window (TL = 1: rows of w.w knots from knot w.k0) or from global memory.
template <int TL>
struct Knots;
template <>
struct Knots<1> {
    const double* d;    // POTB
    const double2* f;   // {FPOTR, FPOTB}
    __device__ __forceinline__ void den(int q, double& v, double& dv) const {
        const double p0 = d[q], p1 = d[q + 1];
        v = p0;
        dv = p1 - p0;
    }
    __device__ __forceinline__ void frc(int q, double& r, double& dr, double& b, double& db) const {
        const double2 t0 = f[q], t1 = f[q + 1];
        r = t0.x;
        dr = t1.x - t0.x;
        b = t0.y;
        db = t1.y - t0.y;
    }
    __device__ __forceinline__ void frb(int q, double& b, double& db) const {
        b = f[q].y;
        db = f[q + 1].y - b;
    }
};
template <>
struct Knots<0> {
    const double2* d;
    const double4* f;
    __device__ __forceinline__ void den(int q, double& v, double& dv) const {
        const double2 e = at(d, static_cast<unsigned>(q) * 16u);
        v = e.x;
        dv = e.y;
    }
    __device__ __forceinline__ void frc(int q, double& r, double& dr, double& b, double& db) const {
        const double4 e = at(f, static_cast<unsigned>(q) * 32u);
        r = e.x;
        dr = e.y;
        b = e.z;
        db = e.w;
    }
    __device__ __forceinline__ void frb(int q, double& b, double& db) const {
        const double4 e = at(f, static_cast<unsigned>(q) * 32u);
        b = e.z;
        db = e.w;
    }
};

// A pair's place in the table.  ok: inside the cutoff with its knots in the window (q is in
// bounds either way); odd: the pair goes the side road.
struct Place {
    double sk, inv_r, dk;
    int kk, q;
    bool ok, odd;
};

template <int IMG>
__device__ __forceinline__ Place place(const TabDev& t, const WalkDev& w, double r2) {
    Place p;
    p.sk = table_coord(r2, t.csi, p.inv_r);
    p.kk = static_cast<int>(p.sk);
    p.dk = p.sk - p.kk;
    const unsigned kd = static_cast<unsigned>(p.kk - w.k0);
    const bool reg = kd <= static_cast<unsigned>(w.last), in = r2 <= t.ru2max;
    const bool far = IMG == 0 && p.kk >= w.kimg;
    p.q = static_cast<int>(min(kd, static_cast<unsigned>(w.last)));
    p.ok = reg && in && !far;
    p.odd = (in && !reg) || far;
    return p;
}

// --------------------------------------------------------------------------------------------
// density
// --------------------------------------------------------------------------------------------

// Terms of the odd pairs among slots s .. s + cnt - 1, by the general formula from the global
// table.
template <int MT, int IMG, int LG>
__device__ __forceinline__ double density_odd(const AtomsDev& a, const TabDev& t, const WalkDev& w,
                                              const BoxDev& b, const Lane& q, int s, int cnt,
                                              double px, double py, double pz, double den) {
#pragma unroll 1
    for (int u = 0; u < cnt; ++u) {
        if (s + u > q.last) break;
        const int j = slot_index(q, s + u, 8 + LG);
        const double2 qxy = *reinterpret_cast<const double2*>(&a.pos[j]);
        const double qz = a.pos[j].z;
        double sx = px - qxy.x, sy = py - qxy.y, sz = pz - qz;
        if constexpr (IMG == 0) {
            if (!place<0>(t, w, sx * sx + sy * sy + sz * sz).odd) continue;
        }
        sx = min_image(sx, b.len[0], b.ilen[0]);
        sy = min_image(sy, b.len[1], b.ilen[1]);
        sz = min_image(sz, b.len[2], b.ilen[2]);
        const double r2 = sx * sx + sy * sy + sz * sz;
        if (!(r2 <= t.ru2max) || (IMG == 1 && !place<1>(t, w, r2).odd)) continue;
        const int kind = MT ? t.kpair[q.ti * t.ngroup + a.ityp[j]] : t.kpair[0];
        double inv_r;
        const double sk = table_coord(r2, t.csi, inv_r);
        const int kk = min(static_cast<int>(sk), t.ntab2 - 2);
        const double2 e = t.b2[static_cast<size_t>(kind) * t.ntab2 + kk];
        den = den + (e.x + (sk - kk) * e.y);
    }
    return den;
}

// Whether a lane's slot s is in the list.
template <int L>
__device__ __forceinline__ bool listed(const Lane& q, int s) {
    return s * L + q.sub < q.kv;
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
        const unsigned o = static_cast<unsigned>(js[u]) << 5;
        qxy[u] = *reinterpret_cast<const double2*>(&at(a.pos, o));
        qz[u] = at(a.pos, o).z;
        tj[u] = MT ? at(a.ityp, static_cast<unsigned>(js[u]) << 2) : 0;
    }
    if constexpr (FULL) {
#pragma unroll
        for (int u = 0; u < G; ++u) js[u] = slot_index(q, min(s + G + u, q.last), 8 + LG);
    }
    unsigned long long odd = 0;
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
        odd |= __ballot(p.odd && valid);
    }
    if (odd) den = density_odd<MT, IMG, LG>(a, t, w, b, q, s, G, px, py, pz, den);
    return den;
}

template <int MB, int MT, int EAM, int L, int TL>
__global__ __launch_bounds__(TL ? kLtMaxBlock : kBlock) void k_density_w(
    AtomsDev a, ListDev l, TabDev t, BoxDev box0, const BoxDev* __restrict__ boxes, WalkDev w,
    int* err) {
    constexpr int LG = ilog2(L), G = group_d(L), A = 64 / L;
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
        // the atom's loads in one batch, with the first group's slot indices (slots clamped below
        // mx, masked by the list length once it is known)
        int js[G];
        const int st = at(a.statu, q.ib * 4u), kv = at(l.kvois, q.ib * 4u);
        const double2 pxy = *reinterpret_cast<const double2*>(&at(a.pos, q.ib * 32u));
        const double pz = at(a.pos, q.ib * 32u).z;
        q.ti = MT ? at(a.ityp, q.ib * 4u) : 0;
#pragma unroll
        for (int k = 0; k < G; ++k)
            js[k] = at(q.blk, row + static_cast<unsigned>(min(sub + k * L, l.mx - 1)) * 256u);
        const BoxDev& b = box_of<MB>(box0, boxes, a.boxid, static_cast<int>(q.ib));
        const bool active = have && (st & STATU_ACTIVE) == STATU_ACTIVE;
        q.kv = active ? kv : 0;
        q.sub = sub;
        q.last = ((q.kv - sub + L - 1) >> LG) - 1;
        const bool fast = w.kimg > 0 && !__any(active && !inner(b, w.margin, pxy.x, pxy.y, pz));
        double den = 0.0;
        if (q.kv > 0) {
#pragma unroll
            for (int k = 0; k < G; ++k) js[k] = k <= q.last ? js[k] : static_cast<int>(q.ib);
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
                    atomicOr(&err[kErrEmbd], 1);
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

template <int MT, int IMG, int LG>
__device__ __forceinline__ void force_odd(const AtomsDev& a, const TabDev& t, const WalkDev& w,
                                          const BoxDev& b, const Lane& q, int s, int cnt,
                                          const double4& pi, double& fx, double& fy, double& fz) {
#pragma unroll 1
    for (int u = 0; u < cnt; ++u) {
        if (s + u > q.last) break;
        const int j = slot_index(q, s + u, 8 + LG);
        const double4 pj = a.pos[j];
        double sx = pi.x - pj.x, sy = pi.y - pj.y, sz = pi.z - pj.z;
        if constexpr (IMG == 0) {
            if (!place<0>(t, w, sx * sx + sy * sy + sz * sz).odd) continue;
        }
        sx = min_image(sx, b.len[0], b.ilen[0]);
        sy = min_image(sy, b.len[1], b.ilen[1]);
        sz = min_image(sz, b.len[2], b.ilen[2]);
        const double r2 = sx * sx + sy * sy + sz * sz;
        if (!(r2 <= t.ru2max) || (IMG == 1 && !place<1>(t, w, r2).odd)) continue;
        int kind = t.kpair[0], kind1 = t.kpair[0];
        if constexpr (MT) {
            const int tj = a.ityp[j];
            kind = t.kpair[q.ti * t.ngroup + tj];
            kind1 = t.kpair[tj * t.ngroup + q.ti];
        }
        double inv_r;
        const double sk = table_coord(r2, t.csi, inv_r);
        const int kk = min(static_cast<int>(sk), t.ntab2 - 2);
        const double dk = sk - kk;
        const double4 f = t.f4[static_cast<size_t>(kind) * t.ntab2 + kk];
        const double4 f1 = t.f4[static_cast<size_t>(kind1) * t.ntab2 + kk];
        const double ft = (f.x + dk * f.y) * (inv_r * inv_r) +
                          ((f.z + dk * f.w) * pi.w + (f1.z + dk * f1.w) * pj.w) * inv_r;
        fx = fx + ft * sx;
        fy = fy + ft * sy;
        fz = fz + ft * sz;
    }
}

// As density_slots, for the force.
template <int G, int FULL, int MT, int IMG, int L, int TL>
__device__ __forceinline__ void force_slots(const AtomsDev& a, const TabDev& t, const WalkDev& w,
                                            const BoxDev& b, const Lane& q, const Knots<TL>& kn,
                                            const int* s_row, int s, const double4& pi, double& fx,
                                            double& fy, double& fz, int (&js)[G]) {
    constexpr int LG = ilog2(L);
    double4 pj[G];
    int tj[G];
#pragma unroll
    for (int u = 0; u < G; ++u) {
        if (!FULL && u > 0 && (s + u) * L >= q.kv) break;
        pj[u] = at(a.pos, static_cast<unsigned>(js[u]) << 5);
        tj[u] = MT ? at(a.ityp, static_cast<unsigned>(js[u]) << 2) : 0;
    }
    if constexpr (FULL) {
#pragma unroll
        for (int u = 0; u < G; ++u) js[u] = slot_index(q, min(s + G + u, q.last), 8 + LG);
    }
    unsigned long long odd = 0;
#pragma unroll
    for (int u = 0; u < G; ++u) {
        if (!FULL && u > 0 && (s + u) * L >= q.kv) break;
        double sx = pi.x - pj[u].x, sy = pi.y - pj[u].y, sz = pi.z - pj[u].z;
        if constexpr (IMG == 1) {
            sx = min_image(sx, b.len[0], b.ilen[0]);
            sy = min_image(sy, b.len[1], b.ilen[1]);
            sz = min_image(sz, b.len[2], b.ilen[2]);
        }
        const Place p = place<IMG>(t, w, sx * sx + sy * sy + sz * sz);
        const bool valid = FULL || listed<L>(q, s + u);
        double fr, dfr, fb, dfb;
        kn.frc(p.q + (MT ? s_row[q.ti * t.ngroup + tj[u]] : 0), fr, dfr, fb, dfb);
        fb = fb + p.dk * dfb;
        double fb1 = fb;
        if constexpr (MT) {
            double g, dg;
            kn.frb(p.q + s_row[tj[u] * t.ngroup + q.ti], g, dg);
            fb1 = g + p.dk * dg;
        }
        // FPOTR/r^2 + (FPOTB(KTAB) F'_i + FPOTB(KTAB1) F'_j)/r  (CALFORCE_KERNEL)
        double ft = (fr + p.dk * dfr) * (p.inv_r * p.inv_r) + (fb * pi.w + fb1 * pj[u].w) * p.inv_r;
        ft = (p.ok && valid) ? ft : 0.0;
        fx = fx + ft * sx;
        fy = fy + ft * sy;
        fz = fz + ft * sz;
        odd |= __ballot(p.odd && valid);
    }
    if (odd) force_odd<MT, IMG, LG>(a, t, w, b, q, s, G, pi, fx, fy, fz);
}

template <int MB, int MT, int MODE, int L, int TL>
__global__ __launch_bounds__(TL ? kLtMaxBlock : kBlock) void k_force_w(
    AtomsDev a, ListDev l, TabDev t, BoxDev box0, const BoxDev* __restrict__ boxes, StepParams sp,
    WalkDev w) {
    constexpr int LG = ilog2(L), G = group_f(L), A = 64 / L;
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
            js[k] = at(q.blk, row + static_cast<unsigned>(min(sub + k * L, l.mx - 1)) * 256u);
        AtomState as;
        if constexpr (MODE >= 1)
            if (sub == 0) load_atom_state(a, sp, AtomIx{q.ib}, as);
        const BoxDev& b = box_of<MB>(box0, boxes, a.boxid, static_cast<int>(q.ib));
        const bool active = have && (st & STATU_ACTIVE) == STATU_ACTIVE;
        q.kv = active ? kv : 0;
        q.sub = sub;
        q.last = ((q.kv - sub + L - 1) >> LG) - 1;
        const bool fast = w.kimg > 0 && !__any(active && !inner(b, w.margin, pi.x, pi.y, pi.z));
        double fx = 0.0, fy = 0.0, fz = 0.0;
        if (q.kv > 0) {
#pragma unroll
            for (int k = 0; k < G; ++k) js[k] = k <= q.last ? js[k] : static_cast<int>(q.ib);
            auto slots = [&](auto img) {
                constexpr int IMG = decltype(img)::value;
                int s = 0;
                for (; (s + G) * L <= q.kv; s += G)
                    force_slots<G, 1, MT, IMG, L, TL>(a, t, w, b, q, kn, s_row, s, pi, fx, fy, fz,
                                                       js);
                if (s * L < q.kv)
                    force_slots<G, 0, MT, IMG, L, TL>(a, t, w, b, q, kn, s_row, s, pi, fx, fy, fz,
                                                       js);
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

// Window of the upper part of the table for an LDS share: knots from k0 on.
void window(const TabDev& t, long budget, int bytes, WalkDev& w) {
    const int nk = t.ngroup > 1 ? t.nkind : 1;
    const int fit = static_cast<int>(std::max(0L, budget / (static_cast<long>(bytes) * nk)));
    const int want = t.ntab2 - 3 * (t.ntab2 / 8);
    w.w = std::min(want, fit);
    w.k0 = t.ntab2 - w.w;
    w.last = t.ntab2 - 2 - w.k0;
}

long walk_budget(const TabDev& t, int wgs) {
    return lt_lds_budget(wgs) - (t.ngroup > 1 ? 4 * kMaxGroup * kMaxGroup : 0);
}

}  // namespace

bool walk_window_ok(const TabDev& t, int force, int wgs) {
    WalkDev w{};
    window(t, walk_budget(t, wgs), force ? 16 : 8, w);
    return 2 * w.w >= t.ntab2;
}

namespace {

// Launch parameters common to both passes; returns the workgroups.
template <typename K>
unsigned walk_launch(K k, const WalkPlan& pl, int bytes, int n, const TabDev& t, WalkDev& w,
                     int& threads, size_t& lds) {
    w.kimg = pl.kimg;
    w.margin = pl.margin;
    w.sweep = pl.sweep;
    w.units = (n + 64 / pl.lanes - 1) / (64 / pl.lanes);
    if (pl.tl) {
        threads = pl.block;
        window(t, walk_budget(t, pl.wgs), bytes, w);
        lds = static_cast<size_t>(w.w) * (t.ngroup > 1 ? t.nkind : 1) * bytes;
        const int nwv = threads / 64;
        return lt_persistent_grid(reinterpret_cast<const void*>(k), threads, lds, pl.wgs,
                                  (w.units + nwv - 1) / nwv);
    }
    threads = kBlock;
    lds = 0;
    w.k0 = 0;
    w.w = t.ntab2;
    w.last = t.ntab2 - 2;
    return static_cast<unsigned>((w.units + kBlock / 64 - 1) / (kBlock / 64));
}

}  // namespace

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
