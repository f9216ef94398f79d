// msm_walk.h -- what the list-walk kernels share (msm_walk.hip, msm_walk_energy.hip): units and
// lanes, knot access, the side road of odd pairs, the force of a group of slots, launch shapes.
#pragma once

#include <algorithm>
#include <cmath>
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

// A pointer to global memory that is the same in every lane, in scalar registers.  The address
// space is spelled out: from a pointer put together of integers the compiler would make flat loads,
// which count as LDS accesses too, and the next use of a knot would wait for the indices in flight.
using GlobalInts = const __attribute__((address_space(1))) int*;

__device__ __forceinline__ GlobalInts uniform(const int* p) {
    const unsigned long long a = reinterpret_cast<unsigned long long>(p);
    const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(a));
    const unsigned hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(a >> 32));
    return reinterpret_cast<GlobalInts>((static_cast<unsigned long long>(hi) << 32) | lo);
}

__device__ __forceinline__ int slot_at(GlobalInts p, unsigned off) {
    return *reinterpret_cast<GlobalInts>(
        reinterpret_cast<const __attribute__((address_space(1))) char*>(p) + off);
}

constexpr int ilog2(int v) { return v <= 1 ? 0 : 1 + ilog2(v / 2); }

// Slots per group: the gathers of a group are in flight together.
constexpr int group_d(int L) { return L <= 4 ? 6 : L == 8 ? 4 : 3; }
constexpr int group_f(int) { return 3; }

// What a lane needs of its unit.
struct Lane {
    GlobalInts blk;   // list block of the unit's atoms (uniform)
    unsigned lo;      // byte offset of the lane's first slot in it
    unsigned ib;      // atom index
    int kv;           // list length (0: inactive)
    int sub;          // lane within the atom
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
    return slot_at(q.blk, q.lo + (static_cast<unsigned>(s) << shift));
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
// bounds either way); odd: the pair goes the side road: those below
// the window, those that may need the minimum image (IMG = 0) and, where the cutoff does not lie
// within the table, those above it (one unsigned comparison for all three).
struct Place {
    double inv_r, dk;
    int q;
    bool ok, odd;
};

template <int IMG>
__device__ __forceinline__ Place place(const TabDev& t, const WalkDev& w, double r2) {
    Place p;
    const double sk = table_coord(r2, t.csi, p.inv_r);
    const int kk = static_cast<int>(sk);
    p.dk = sk - kk;  // contracts with sk's last product: the fraction without its rounding
    const unsigned kd = static_cast<unsigned>(kk - w.k0);
    p.q = static_cast<int>(min(kd, static_cast<unsigned>(w.last)));
    p.odd = kd >= (IMG ? w.odd1 : w.odd0);
    p.ok = r2 <= t.ru2max && !p.odd;
    return p;
}

// The lanes in which p holds.
__device__ __forceinline__ unsigned long long lanes_of(bool p) {
    return __builtin_amdgcn_ballot_w64(p);
}

// Whether a lane's slot s is in the list.
template <int L>
__device__ __forceinline__ bool listed(const Lane& q, int s) {
    return s * L + q.sub < q.kv;
}

// The indices of a lane's slots s + G .. s + 2 G - 1.  Beyond the end of the list they are whatever
// the memory holds (the list is allocated with kWalkSlack ints after its last row): slot_atom
// replaces them where they would be used.
template <int G, int LG>
__device__ __forceinline__ void next_slots(const Lane& q, int s, int (&js)[G]) {
    const unsigned o = q.lo + (static_cast<unsigned>(s + G) << (8 + LG));
#pragma unroll
    for (int u = 0; u < G; ++u) js[u] = slot_at(q.blk, o + (static_cast<unsigned>(u) << (8 + LG)));
}

template <int FULL, int L>
__device__ __forceinline__ unsigned slot_atom(const Lane& q, int s, int j) {
    return FULL || listed<L>(q, s) ? static_cast<unsigned>(j) : q.ib;
}

__device__ __forceinline__ void add_virial(double h, double sx, double sy, double sz,
                                           double (&v)[6]) {
    v[0] = v[0] + sx * sx * h;
    v[1] = v[1] + sy * sy * h;
    v[2] = v[2] + sz * sz * h;
    v[3] = v[3] + sx * sy * h;
    v[4] = v[4] + sx * sz * h;
    v[5] = v[5] + sy * sz * h;
}

// The odd pairs of a group, one bit a slot.  The side road takes them from here and decides nothing
// itself: the same comparison compiled twice may round differently, and a pair on the edge would be
// lost or count twice.  WAVE: as masks of the wave, in scalar registers (full groups of the passes with
// the knots in LDS); else every lane keeps its own bits (in a list's last group lanes stop at different
// slots; 200 steps of 2,000 W atoms, with a global table, 2,152 us against 2,183 with masks).
template <int G, int WAVE>
struct OddPairs {
    unsigned long long m[WAVE ? G : 1] = {}, any = 0;
    unsigned bits = 0;
    __device__ __forceinline__ void note(int u, bool odd) {
        if constexpr (WAVE) {
            m[u] = lanes_of(odd);
            any |= m[u];
        } else {
            bits |= odd ? 1u << u : 0u;
        }
    }
    __device__ __forceinline__ bool some() const { return WAVE ? any != 0 : bits != 0; }
    __device__ __forceinline__ unsigned slots() const {
        unsigned b = bits;
        if constexpr (WAVE) {
#pragma unroll
            for (int u = 0; u < G; ++u) b |= (m[u] >> (threadIdx.x & 63) & 1ull) ? 1u << u : 0u;
        }
        return b;
    }
};

// Forces of the odd pairs among slots s, s + 1, ... (bits), by the general formula from the global
// table.  V = 1: the half virial of every pair as well (components xx, yy, zz, xy, xz, yz).
template <int MT, int LG, int V>
__device__ __forceinline__ void force_odd(const AtomsDev& a, const TabDev& t, const BoxDev& b,
                                          const Lane& q, int s, unsigned bits, const double4& pi,
                                          double& fx, double& fy, double& fz, double (&vir)[6]) {
#pragma unroll 1
    for (; bits; bits &= bits - 1) {
        const int j = slot_index(q, s + __builtin_ctz(bits), 8 + LG);
        const double4 pj = a.pos[j];
        double sx = pi.x - pj.x, sy = pi.y - pj.y, sz = pi.z - pj.z;
        sx = min_image(sx, b.len[0], b.ilen[0]);
        sy = min_image(sy, b.len[1], b.ilen[1]);
        sz = min_image(sz, b.len[2], b.ilen[2]);
        const double r2 = sx * sx + sy * sy + sz * sz;
        if (!(r2 <= t.ru2max)) continue;
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
        if constexpr (V) add_virial(0.5 * ft, sx, sy, sz, vir);
    }
}

// As density_slots, for the force.
template <int G, int FULL, int MT, int IMG, int L, int TL, int V>
__device__ __forceinline__ void force_slots(const AtomsDev& a, const TabDev& t, const WalkDev& w,
                                            const BoxDev& b, const Lane& q, const Knots<TL>& kn,
                                            const int* s_row, int s, const double4& pi, double& fx,
                                            double& fy, double& fz, double (&vir)[6], int (&js)[G]) {
    constexpr int LG = ilog2(L);
    double4 pj[G];
    int tj[G];
#pragma unroll
    for (int u = 0; u < G; ++u) {
        if (!FULL && u > 0 && (s + u) * L >= q.kv) break;
        const unsigned j = slot_atom<FULL, L>(q, s + u, js[u]);
        pj[u] = at(a.pos, j << 5);
        tj[u] = MT ? at(a.ityp, j << 2) : 0;
    }
    if constexpr (FULL) next_slots<G, LG>(q, s, js);
    OddPairs<G, FULL && TL> odd;
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
        const bool use = p.ok && valid;
        ft = use ? ft : 0.0;
        // A pair with a lost atom (not a number, infinity) has no finite displacement, which must not
        // count either.  Not in the force pass with the knots in LDS: there it costs 1.2% on a
        // million atoms, and k_force_lt, which it follows, spreads a lost atom as well.
        if constexpr (V || !TL) {
            sx = use ? sx : 0.0;
            sy = use ? sy : 0.0;
            sz = use ? sz : 0.0;
        }
        fx = fx + ft * sx;
        fy = fy + ft * sy;
        fz = fz + ft * sz;
        if constexpr (V) add_virial(0.5 * ft, sx, sy, sz, vir);
        odd.note(u, p.odd && valid);
    }
    if (__builtin_expect(odd.some(), 0))
        force_odd<MT, LG, V>(a, t, b, q, s, odd.slots(), pi, fx, fy, fz, vir);
}

// Window of the upper part of the table for an LDS share: knots from k0 on.
inline void window(const TabDev& t, long budget, int bytes, WalkDev& w) {
    const int nk = t.ngroup > 1 ? t.nkind : 1;
    const int fit = static_cast<int>(std::max(0L, budget / (static_cast<long>(bytes) * nk)));
    const int want = t.ntab2 - 3 * (t.ntab2 / 8);
    w.w = std::min(want, fit);
    w.k0 = t.ntab2 - w.w;
    w.last = t.ntab2 - 2 - w.k0;
}

// From which knot of the window on a pair is odd (place).  Within the table: every pair inside the
// cutoff has its knots there.
inline void odd_knots(const TabDev& t, WalkDev& w) {
    const bool within = t.csi * std::sqrt(std::sqrt(t.ru2max)) < t.ntab2 - 1 - 1.0e-6;
    const unsigned top = within ? 0x80000000u : static_cast<unsigned>(w.last) + 1u;
    w.odd1 = top;
    w.odd0 = std::min(top, static_cast<unsigned>(std::max(w.kimg - w.k0, 0)));
}

inline long walk_budget(const TabDev& t, int wgs) {
    return lt_lds_budget(wgs) - (t.ngroup > 1 ? 4 * kMaxGroup * kMaxGroup : 0);
}

// Launch parameters common to the passes; returns the workgroups.
template <typename K>
unsigned walk_launch(K k, const WalkPlan& pl, int bytes, int n, const TabDev& t, WalkDev& w,
                     int& threads, size_t& lds) {
    w.kimg = pl.kimg;
    w.margin = pl.margin;
    w.sweep = pl.sweep;
    static_assert(kWalkSlack >= 2 * 64 * 96, "slots that a group may read past the list");
    w.units = (n + 64 / pl.lanes - 1) / (64 / pl.lanes);
    if (pl.tl) {
        threads = pl.block;
        window(t, walk_budget(t, pl.wgs), bytes, w);
        odd_knots(t, w);
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
    odd_knots(t, w);
    return static_cast<unsigned>((w.units + kBlock / 64 - 1) / (kBlock / 64));
}

}  // namespace

}  // namespace msm
