// msm_cells.hip -- neighbour rebuild of the default path: cell sort and the list, one wave per cell.
//
// Sort: cell ids and counts, exclusive scan, arrival scatter, then one kernel that ranks every
// atom by caller index among its cell's arrivals and moves its data to that place (the order of a
// cell does not depend on the arrival order, and no cell is too full for the ranking).  Boxes of
// at most kSortSmallAtoms atoms and kSortSmallCells cells do the first three steps in one workgroup
// with the counts in LDS.  Each launch of the chain costs about 4.4 us whatever it does, which is
// most of a small box's rebuild: ten launches became three (2,000 W atoms: 35 us before the list
// kernel, now 12), and five on larger boxes.
//
// List: a wave takes one cell.  Its 64 lanes hold the candidates of the 27 cells around it, in the
// reference's stencil order, a few per lane; the cell's atoms are then compared one after another
// (their coordinates read from a lane into scalar registers), a candidate's place in the atom's
// list being the number of hits in lower lanes.  All 27 cells' loads are issued together, where a
// lane per atom walks them in turn: 2,000 to 54,000 W atoms took 39-41 us whatever their number, and
// take 6.4 (2,000) to 10.3 (16,000) now; 136,000 38 us (65), a million 210 (239); Cu-Ni 4,000 atoms
// 23 (62), 442,000 336 (436).
// The comparison is the host's, without contraction: XPT(I) - (XP(J) + CXYZ), squared and summed left
// to right, strict < (MD_NeighborsList.F90:396-633).
#include <algorithm>

#include "msm_device.h"

namespace msm {

namespace {

// Cell of atom i (ncell_total: outside every grid), MD_NeighborsList.F90:255-276.
__device__ __forceinline__ int cell_of(const double4* __restrict__ pos,
                                       const int* __restrict__ statu,
                                       const int* __restrict__ boxid,
                                       const BoxDev* __restrict__ boxes, int i, int ncell_total,
                                       int* err) {
#pragma clang fp contract(off)
    if ((statu[i] & STATU_OUTOFBOX) == STATU_OUTOFBOX) return ncell_total;
    const BoxDev& b = boxes[boxid[i]];
    const double4 p = pos[i];
    const double xyz[3] = {p.x, p.y, p.z};
    int ic[3];
    bool in = true;
    for (int k = 0; k < 3; ++k) {
        // (x - LB)/L * NC - eps, truncated toward zero
        const double s = (xyz[k] - b.lo[k]) / b.len[k] * static_cast<double>(b.ncell[k]) - 1.0e-4;
        ic[k] = static_cast<int>(s);
        in = in && ic[k] >= 0 && ic[k] < b.ncell[k];
    }
    if (in) return b.cell_off + cell_local(b, ic[0], ic[1], ic[2]);
    err[kErrOutOfBox] = 1;
    return ncell_total;
}

}  // namespace

// One count atomic per distinct cell of the wave: after the first build the atoms are cell-sorted,
// so a wave spans a few cells.  The lanes of each cell are grouped by ballots, the leader of
// every cell adds its lane count (all leaders in one instruction), and every lane takes base + its
// rank among its cell's lanes.
__global__ void k_cell_assign(const double4* __restrict__ pos, const int* __restrict__ statu,
                              const int* __restrict__ boxid, const BoxDev* __restrict__ boxes,
                              int n, int ncell_total, int* __restrict__ key,
                              int* __restrict__ slot, int* __restrict__ count, int* err) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int c = cell_of(pos, statu, boxid, boxes, i, ncell_total, err);
    key[i] = c;
    const int lane = threadIdx.x & 63;
    unsigned long long todo = __ballot(1);
    int lead = lane, rank = 0, cnt = 0;
    while (todo) {
        const int leader = __ffsll(static_cast<long long>(todo)) - 1;
        const int lc = __shfl(c, leader, 64);
        const unsigned long long same = __ballot(c == lc) & todo;
        if (c == lc) {
            lead = leader;
            rank = __popcll(same & ((1ull << lane) - 1ull));
            if (lane == leader) cnt = __popcll(same);
        }
        todo &= ~same;
    }
    int base = 0;
    if (cnt > 0) base = atomicAdd(&count[c], cnt);
    slot[i] = __shfl(base, lead, 64) + rank;
}

// Exclusive scan of the counts in two launches: block scans with the block totals, then every
// block adds the totals before it.  The counts are set to zero for the next rebuild.
constexpr int kScanBlock = 1024;

__global__ void k_scan_blocks(int* __restrict__ in, int* __restrict__ out, int* __restrict__ sums,
                              int n) {
    __shared__ int lds[kScanBlock / 64];
    const int i = blockIdx.x * kScanBlock + threadIdx.x;
    const int v = (i < n) ? in[i] : 0;
    const int inc = block_incl_scan(v, lds);
    if (i < n) {
        in[i] = 0;
        out[i] = inc - v;  // exclusive within the block
    }
    if (threadIdx.x == kScanBlock - 1) sums[blockIdx.x] = inc;
}

__global__ void k_scan_add(int* out, const int* __restrict__ sums, int n) {
    __shared__ int part[kScanBlock / 64];
    int v = 0;
    for (int k = threadIdx.x; k < static_cast<int>(blockIdx.x); k += kScanBlock) v += sums[k];
    const int lane = threadIdx.x & 63;
    v = wave_incl_scan(v);
    if (lane == 63) part[threadIdx.x >> 6] = v;
    __syncthreads();
    int add = 0;
    for (int k = 0; k < kScanBlock / 64; ++k) add += part[k];
    const int i = blockIdx.x * kScanBlock + threadIdx.x;
    if (i < n) out[i] += add;
}

__global__ void k_scatter(int n, const int* __restrict__ key, const int* __restrict__ slot,
                          const int* __restrict__ start, const int* __restrict__ gid,
                          int2* __restrict__ arr) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) arr[start[key[i]] + slot[i]] = make_int2(i, gid[i]);
}

// The three steps above for a small box, in one workgroup.  start has ncell_total + 2 entries.
__global__ __launch_bounds__(1024) void k_sort_small(
    const double4* __restrict__ pos, const int* __restrict__ statu, const int* __restrict__ boxid,
    const BoxDev* __restrict__ boxes, int n, int ncell_total, const int* __restrict__ gid,
    int* __restrict__ key, int* __restrict__ start, int2* __restrict__ arr, int* err) {
    extern __shared__ int s_cnt[];  // ncell_total + 2
    __shared__ int lds[16];
    constexpr int kPer = kSortSmallAtoms / 1024;
    const int nc = ncell_total + 2;
    for (int k = threadIdx.x; k < nc; k += 1024) s_cnt[k] = 0;
    __syncthreads();
    int c[kPer], slot[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const int i = threadIdx.x + k * 1024;
        if (i < n) c[k] = cell_of(pos, statu, boxid, boxes, i, ncell_total, err);
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k)
        if (static_cast<int>(threadIdx.x) + k * 1024 < n) slot[k] = atomicAdd(&s_cnt[c[k]], 1);
    __syncthreads();
    // exclusive scan: each thread a contiguous run of counts
    const int per = (nc + 1023) / 1024, k0 = threadIdx.x * per, k1 = min(k0 + per, nc);
    int sum = 0;
    for (int k = k0; k < k1; ++k) sum += s_cnt[k];
    int run = block_incl_scan(sum, lds) - sum;
    for (int k = k0; k < k1; ++k) {
        const int v = s_cnt[k];
        s_cnt[k] = run;
        start[k] = run;
        run += v;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const int i = threadIdx.x + k * 1024;
        if (i < n) {
            key[i] = c[k];
            arr[s_cnt[c[k]] + slot[k]] = make_int2(i, gid[i]);
        }
    }
}

// Arrival a of the counting sort: its rank by caller index in its cell, and its data moved to that
// place.  F = 0: forces are not carried (a force pass overwrites them before they are read).
template <int F>
__global__ void k_order_move(int n, const int2* __restrict__ arr, const int* __restrict__ start,
                             AtomsDev src, AtomsDev dst, int* __restrict__ gid_dst,
                             const int* __restrict__ key, int* __restrict__ cell_dst) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= n) return;
    const int2 me = arr[a];
    const int i = me.x, c = key[i];
    double4 x = src.pos[i];
    x.w = 0.0;
    const double vx = src.vx[i], vy = src.vy[i], vz = src.vz[i];
    const double dx = src.dx[i], dy = src.dy[i], dz = src.dz[i];
    const int ty = src.ityp[i], st = src.statu[i], bx = src.boxid[i];
    const int s = start[c], e = start[c + 1];
    int p = s;
    for (int k = s; k < e; ++k) p += arr[k].y < me.y ? 1 : 0;
    dst.pos[p] = x;
    dst.vx[p] = vx;
    dst.vy[p] = vy;
    dst.vz[p] = vz;
    if constexpr (F) {
        dst.fx[p] = src.fx[i];
        dst.fy[p] = src.fy[i];
        dst.fz[p] = src.fz[i];
    }
    dst.dx[p] = dx;
    dst.dy[p] = dy;
    dst.dz[p] = dz;
    dst.ityp[p] = ty;
    dst.statu[p] = st;
    dst.boxid[p] = bx;
    gid_dst[p] = me.y;
    cell_dst[p] = c;
}

void launch_cell_sort(int n, int ncell_total, const BoxDev* boxes, const AtomsDev& src,
                      const int* gid_src, AtomsDev& dst, int* gid_dst, int* cell_dst, SortBufs sb,
                      int keep_f, int* err, hipStream_t s) {
    if (n <= 0) {
        launch_fill_int(sb.start, 0, ncell_total + 2, s);
        return;
    }
    const int nc = ncell_total + 2;
    if (n <= kSortSmallAtoms && nc <= kSortSmallCells) {
        hipLaunchKernelGGL(k_sort_small, dim3(1), dim3(1024), nc * sizeof(int), s, src.pos,
                           src.statu, src.boxid, boxes, n, ncell_total, gid_src, sb.key, sb.start,
                           sb.arr, err);
    } else {
        hipLaunchKernelGGL(k_cell_assign, dim3(grid_for(n)), dim3(kBlock), 0, s, src.pos,
                           src.statu, src.boxid, boxes, n, ncell_total, sb.key, sb.slot, sb.count,
                           err);
        const int nb = (nc + kScanBlock - 1) / kScanBlock;
        hipLaunchKernelGGL(k_scan_blocks, dim3(nb), dim3(kScanBlock), 0, s, sb.count, sb.start,
                           sb.scan_tmp, nc);
        if (nb > 1)
            hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(kScanBlock), 0, s, sb.start,
                               sb.scan_tmp, nc);
        hipLaunchKernelGGL(k_scatter, dim3(grid_for(n)), dim3(kBlock), 0, s, n, sb.key, sb.slot,
                           sb.start, gid_src, sb.arr);
    }
    if (keep_f)
        hipLaunchKernelGGL(k_order_move<1>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, sb.arr,
                           sb.start, src, dst, gid_dst, sb.key, cell_dst);
    else
        hipLaunchKernelGGL(k_order_move<0>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, sb.arr,
                           sb.start, src, dst, gid_dst, sb.key, cell_dst);
}

namespace {

__device__ __forceinline__ double lane_value(double v, int lane) {
    const unsigned long long a = static_cast<unsigned long long>(__double_as_longlong(v));
    const unsigned lo = __builtin_amdgcn_readlane(static_cast<unsigned>(a), lane);
    const unsigned hi = __builtin_amdgcn_readlane(static_cast<unsigned>(a >> 32), lane);
    return __longlong_as_double(
        static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}

}  // namespace

// 2^lgs waves per cell, each taking every 2^lgs-th of its atoms; R candidates per lane at a time (a
// cell with more around it goes through them in chunks of 64 R).  UT: one list radius for every
// pair of types.  Putting the lists together in LDS and writing them by rows of eight atoms
// measured no better than the scattered stores (a million W atoms 220 us against 209, 4,000
// Cu-Ni atoms 41 against 21, 442,000 345 against 376).
constexpr int kCellWaves = 4;

template <int R, int UT>
__global__ __launch_bounds__(64 * kCellWaves, R > 6 ? 3 : R > 4 ? 5 : 8) void k_nlist_cell(
    int ncell_total, int n, int lgs, const double4* __restrict__ pos,
    const int* __restrict__ ityp, const int* __restrict__ boxid, const int* __restrict__ start,
    const BoxDev* __restrict__ boxes, int ngroup, const double* __restrict__ rnl2, int mx,
    int* __restrict__ kvois, int* __restrict__ indi, int* err) {
#pragma clang fp contract(off)
    __shared__ int s_pre[kCellWaves][32], s_base[kCellWaves][32], s_img[kCellWaves][32];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int gw = __builtin_amdgcn_readfirstlane(xcd_block(gridDim.x) * kCellWaves + wv);
    const int g = gw >> lgs, part = gw & ((1 << lgs) - 1);
    if (g > ncell_total) return;
    const int s0 = start[g];
    if (g == ncell_total) {  // atoms in the out-of-box bucket have no neighbours
        if (part == 0)
            for (int p = s0 + lane; p < n; p += 64) kvois[p] = 0;
        return;
    }
    const int nh = start[g + 1] - s0;
    if (nh == 0) return;
    const BoxDev& b = boxes[__builtin_amdgcn_readfirstlane(boxid[s0])];
    // ranges of the 27 cells: lane k the k-th of the stencil
    int cnt = 0, qs = 0, img = 0;
    {
        int ix, iy, iz;
        const int lc = g - b.cell_off;
        if (b.cbs == 1) {
            const int r = lc / b.ncell[0];
            ix = lc - r * b.ncell[0];
            iz = r / b.ncell[1];
            iy = r - iz * b.ncell[1];
        } else {
            cell_coords(b, lc, ix, iy, iz);
        }
        if (lane < 27) {
            int j3[3] = {ix + c_nix[lane], iy + c_niy[lane], iz + c_niz[lane]};
            bool skip = false;
            for (int k = 0; k < 3; ++k) {
                if (b.ifpd[k]) {
                    if (j3[k] >= b.ncell[k]) {
                        j3[k] = 0;
                        img |= 1 << (2 * k);
                    } else if (j3[k] < 0) {
                        j3[k] = b.ncell[k] - 1;
                        img |= 2 << (2 * k);
                    }
                }
                skip = skip || j3[k] < 0 || j3[k] >= b.ncell[k];
            }
            if (!skip) {
                const int c = b.cell_off + (b.cbs == 1 ? j3[0] + b.ncell[0] * (j3[1] + b.ncell[1] * j3[2])
                                                       : cell_local(b, j3[0], j3[1], j3[2]));
                qs = start[c];
                cnt = start[c + 1] - qs;
            }
        }
    }
    const int inc = wave_incl_scan(cnt);
    const int total = __builtin_amdgcn_readlane(inc, 63);
    if (lane < 32) {
        s_pre[wv][lane] = inc;  // end of cell `lane`'s candidates
        s_base[wv][lane] = qs - (inc - cnt);
        s_img[wv][lane] = img;
    }
    // the wave reads what its lanes wrote: LDS instructions of a wave complete in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    double x[R], y[R], z[R];
    int id[R], tj[R];
    auto load = [&](int c0) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int c = c0 + r * 64 + lane;
            id[r] = -1;
            if (c < total) {
                int k = 0;  // first cell whose candidates end beyond c
#pragma unroll
                for (int d = 16; d >= 1; d >>= 1) k += s_pre[wv][k + d - 1] <= c ? d : 0;
                id[r] = s_base[wv][k] + c;
                tj[r] = s_img[wv][k];
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            x[r] = __builtin_nan("");  // no candidate: every comparison fails
            y[r] = z[r] = 0.0;
            if (id[r] >= 0) {
                const double4 q = pos[id[r]];
                const int im = tj[r];
                x[r] = q.x + ((im & 1) ? b.len[0] : (im & 2) ? -b.len[0] : 0.0);
                y[r] = q.y + ((im & 4) ? b.len[1] : (im & 8) ? -b.len[1] : 0.0);
                z[r] = q.z + ((im & 16) ? b.len[2] : (im & 32) ? -b.len[2] : 0.0);
                if constexpr (!UT) tj[r] = ityp[id[r]];
            }
        }
    };
    const bool once = total <= 64 * R;
    if (once) load(0);
    const double rc = UT ? rnl2[0] : 0.0;
    for (int h0 = 0; h0 < nh; h0 += 64) {
        const int hn = min(64, nh - h0);
        double hx = 0.0, hy = 0.0, hz = 0.0;
        int ht = 0;
        if (lane < hn) {
            const double4 q = pos[s0 + h0 + lane];
            hx = q.x;
            hy = q.y;
            hz = q.z;
            if constexpr (!UT) ht = ityp[s0 + h0 + lane];
        }
        int kv = 0;  // lane h: hits of home atom h0 + h
        for (int c0 = 0; c0 < total; c0 += 64 * R) {
            if (!once) load(c0);
            for (int h = part; h < hn; h += 1 << lgs) {
                const double xi = lane_value(hx, h), yi = lane_value(hy, h), zi = lane_value(hz, h);
                const int ti = UT ? 0 : __builtin_amdgcn_readlane(ht, h);
                const int p = s0 + h0 + h;
                int got = __builtin_amdgcn_readlane(kv, h);
                int* __restrict__ row = indi + list_base(p, mx);
                // all comparisons first, without a branch between them
                bool hit[R];
                unsigned long long m[R];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const double dx = xi - x[r], dy = yi - y[r], dz = zi - z[r];
                    const double r2 = dx * dx + dy * dy + dz * dz;
                    double lim = rc;
                    if constexpr (!UT) lim = id[r] >= 0 ? rnl2[ti * ngroup + tj[r]] : 0.0;
                    const bool in = r2 < lim, other = id[r] != p;
                    hit[r] = in && other;
                    m[r] = __ballot(in) & __ballot(other);
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int slot = got + __builtin_amdgcn_mbcnt_hi(
                                               static_cast<unsigned>(m[r] >> 32),
                                               __builtin_amdgcn_mbcnt_lo(
                                                   static_cast<unsigned>(m[r]), 0));
                    if (hit[r] && slot < mx)
                        at(row, static_cast<unsigned>(slot) * (kListRow * 4u)) = id[r];
                    got += __popcll(m[r]);
                }
                kv = lane == h ? got : kv;
            }
        }
        if (lane < hn && (lane & ((1 << lgs) - 1)) == part) {
            if (kv > mx) {
                err[kErrOverflow] = 1;
                kv = mx;
            }
            kvois[s0 + h0 + lane] = kv;
        }
    }
}

void launch_nlist_cell(int ncell_total, int n, double mean, int one_radius, const double4* pos,
                       const int* ityp, const int* boxid, const int* start, const BoxDev* boxes,
                       int ngroup, const double* rnl2, int mx, int* kvois, int* indi, int* err,
                       hipStream_t s) {
    if (n <= 0) return;
    // two or four waves share a cell where one each would leave most of the chip idle (one wave: 2,000
    // W atoms 12.1 us, 4,000 Cu-Ni atoms 48; four: 7.1 and 21)
    const int lgs = ncell_total <= 1024 ? 2 : ncell_total <= 4096 ? 1 : 0;
    const unsigned grid = static_cast<unsigned>(((ncell_total + 1) << lgs) / kCellWaves + 1);
#define MSM_NC(R, UT)                                                                            \
    hipLaunchKernelGGL((k_nlist_cell<R, UT>), dim3(grid), dim3(64 * kCellWaves), 0, s,           \
                       ncell_total, n, lgs, pos, ityp, boxid, start, boxes, ngroup, rnl2, mx, kvois,  \
                       indi, err)
    // the candidates around a mean cell in one chunk
    const double c = 27.0 * mean;
    if (c <= 270.0) {
        if (one_radius) MSM_NC(4, 1); else MSM_NC(4, 0);
    } else if (c <= 400.0) {
        if (one_radius) MSM_NC(6, 1); else MSM_NC(6, 0);
    } else {
        if (one_radius) MSM_NC(10, 1); else MSM_NC(10, 0);
    }
#undef MSM_NC
}

}  // namespace msm
