// Pair search of the sort-based neighbour list: count and fill, the MI355X
// counterparts of count_neighbours_kernel! and fill_pairs_kernel!
// (src/gpu_kernels.jl:132-180) around the inner loop _for_each_neighbor_pair
// (src/gpu_kernels.jl:58-101).
//
// tile_kernel (count_kernel for 16-byte slot entries) -- work
// unit: a brick of up to 4x4x4 home cells per 256-thread (or 512-thread)
// workgroup, the bricks launched largest first.  The brick and its one-cell
// halo are staged in LDS in one load phase (every global load of the phase in
// flight together), then the waves take work items (one or two home cells, or
// a part of one) from a workgroup counter and test candidates from LDS only:
//   - the candidates of a home cell are its 27 neighbour cells flattened in
//     the reference order (dz, dy, dx; gpu_kernels.jl:69-71) -- nine
//     contiguous LDS rows -- cut into 64-candidate chunks, one per lane;
//   - the home atoms stream through the wave as uniform values; each (home
//     atom, chunk) test is one ballot, and the hit lanes append their (j, S)
//     to the home atom's slot row at its running count, so every row holds
//     the atom's neighbours in exactly the reference traversal order.
// tile_kernel tests 32-bit positions and decides what lies within their error
// of the cutoff by the 64-bit test.  Bricks whose neighbour reach exceeds one
// cell, whose halo does not fit LDS, or whose windings lie too far apart take a
// per-wave path that reads global memory (groups of home atoms dealt to the
// waves) with the same enumeration and output.
//
// fill_kernel -- one wave per tile of consecutive output pairs, one lane per
// pair: the tile's first atom comes from the pair scan's tile table, and
// the lanes copy the slot-row entries of the atoms the tile covers into the
// PairList arrays (i, j, S, and R from the positions), so every store is linear.
#include <algorithm>

#include "device_util.h"
#include "filter_bounds.h"

namespace nlh {

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------

__device__ __forceinline__ int sgpr(int v) { return __builtin_amdgcn_readfirstlane(v); }

// The next work item of a wave from a workgroup counter (wave-uniform).
__device__ __forceinline__ int take_next(int32_t *ctr)
{
    int t = 0;
    if (lane_id() == 0) t = atomicAdd(ctr, 1);
    return __builtin_amdgcn_readfirstlane(t);
}

// The largest of the lanes' non-negative values, on the last lane.
__device__ __forceinline__ int wave_max_pos(int v)
{
    v = max(v, dpp_or_zero<0x111>(v));
    v = max(v, dpp_or_zero<0x112>(v));
    v = max(v, dpp_or_zero<0x114>(v));
    v = max(v, dpp_or_zero<0x118>(v));
    v = max(v, dpp_or_zero<0x142, 0xa>(v));
    v = max(v, dpp_or_zero<0x143, 0xc>(v));
    return v;
}

// v with lane `lane` (wave-uniform) set to the wave-uniform x: one
// v_writelane, no exec-mask or compare work.
__device__ __forceinline__ int32_t write_lane(int32_t x, int lane, int32_t v)
{
    // the lane select in M0: the value's SGPR is the one constant-bus read
    __asm__("v_writelane_b32 %0, %1, m0" : "+v"(v) : "s"(sgpr(x)), "{m0}"(sgpr(lane)));
    return v;
}

__device__ __forceinline__ uint64_t shfl64(uint64_t v, int src)
{
    const uint32_t lo = __shfl((uint32_t)v, src, kWave), hi = __shfl((uint32_t)(v >> 32), src, kWave);
    return ((uint64_t)hi << 32) | lo;
}

// (C' * S)_k = sum_m C[m,k] S_m   (gpu_kernels.jl:89)
template <typename Mat>   // const double *, of any address space
__device__ __forceinline__ void cell_shift(const Mat &Cm, int32_t Sx, int32_t Sy, int32_t Sz, double &cx, double &cy,
                                           double &cz)
{
    const double fx = (double)Sx, fy = (double)Sy, fz = (double)Sz;
    cx = (Cm[0] * fx + Cm[1] * fy) + Cm[2] * fz;
    cy = (Cm[3] * fx + Cm[4] * fy) + Cm[5] * fz;
    cz = (Cm[6] * fx + Cm[7] * fy) + Cm[8] * fz;
}

__device__ __forceinline__ void rec_winding(const Rec &r, const int32_t *__restrict__ wbig, int64_t p, int32_t &wx,
                                            int32_t &wy, int32_t &wz)
{
    if (r.w & kWindBig) {
        wx = wbig[3 * p];
        wy = wbig[3 * p + 1];
        wz = wbig[3 * p + 2];
    } else {
        unpack_wind(r.w, wx, wy, wz);
    }
}

constexpr int kChunksPerPass = 3;   // candidate chunks a lane holds at once (per-wave path)
constexpr double kFar = 1.0e200;    // invalid candidate: r^2 overflows to +inf, never a hit

struct PairsArgs {
    const SysDev *__restrict__ sys;
    const int32_t *__restrict__ sys_cell_base;
    int nsys;
    int32_t M;
    int64_t nat;
    const int32_t *__restrict__ cell_start;
    const Rec *__restrict__ rec;
    const int32_t *__restrict__ wbig;
};

// ---------------------------------------------------------------------------
// slots: each atom's neighbours (j, S) in traversal order, a row of `cap`
// entries per atom, rows in original atom order.  A row holds 4-byte entries
// (j | S code << 26) when every shift of its brick is within [-1, 1]^3, else
// 8-byte entries (j | S packed in 3 x 10 bits << 32); bit 30 of the atom's
// count tells which.  Wide builds (shifts beyond +-511) use 16-byte entries.
// ---------------------------------------------------------------------------

template <bool WIDE>
struct SlotEntry;
template <>
struct SlotEntry<false> {
    using T = uint64_t;
    __device__ static void get(T e, int32_t &j, int32_t &Sx, int32_t &Sy, int32_t &Sz)
    {
        j = (int32_t)(uint32_t)e;
        unpack_wind((uint32_t)(e >> 32), Sx, Sy, Sz);
    }
};
template <>
struct SlotEntry<true> {
    using T = int4;
    __device__ static void get(T e, int32_t &j, int32_t &Sx, int32_t &Sy, int32_t &Sz)
    {
        j = e.x; Sx = e.y; Sy = e.z; Sz = e.w;
    }
};

struct SlotArgs {
    void *__restrict__ slots;
    int32_t cap;
    Status *__restrict__ status;
};

// Append the hits of one (home atom, chunk) ballot to the home atom's slot.
// sbase = sorted index of the home atom * cap; ca = its running count
// (wave-uniform); (sx, sy, sz) this lane's S, spk the same packed if `packed`
// (wave-uniform: most home atoms have no winding, and their S is s - w_j).
template <bool WIDE>
__device__ __forceinline__ void emit_hits(const SlotArgs &O, uint64_t mask, int64_t sbase, int32_t &ca, int32_t cj,
                                          int32_t sx, int32_t sy, int32_t sz, bool packed, uint32_t spk)
{
    if (mask == 0) return;   // wave-uniform
    const int lane = lane_id();
    const int32_t rank = ca + (int32_t)mbcnt64(mask);
    if ((mask >> lane) & 1) {
        const int64_t sidx = sbase + rank;
        if (WIDE) {
            if (rank < O.cap) reinterpret_cast<int4 *>(O.slots)[sidx] = make_int4(cj, sx, sy, sz);
        } else {
            // entries past a row's end count too: the repeat on longer rows is the last one
            if (!packed) spk = pack_wind(sx, sy, sz);
            if (spk & kWindBig) O.status->wide = 1;
            if (rank < O.cap)
                reinterpret_cast<uint64_t *>(O.slots)[sidx] = (uint64_t)(uint32_t)cj | ((uint64_t)spk << 32);
        }
    }
    ca += (int32_t)__popcll(mask);
}

// ---------------------------------------------------------------------------
// per-wave path: one home cell per wave, candidates read from global memory
// ---------------------------------------------------------------------------

struct HomeCell {
    int ci0, ci1, ci2;          // 1-based cell coordinates
    int n0, n1, n2, nx0, nx1, nx2, sx, sy, nseg;
    bool p0, p1, p2;
    int32_t cbase;
    int64_t abase;
    const SysDev *sd;
};

// The grid around the cell at 1-based coordinates (ci0, ci1, ci2).
__device__ __forceinline__ void home_grid(const SysDev &sd, int ci0, int ci1, int ci2, HomeCell &H)
{
    H.sd = &sd;
    H.n0 = sd.n[0]; H.n1 = sd.n[1]; H.n2 = sd.n[2];
    H.cbase = sd.cell_base;
    H.abase = sd.atom_base;
    H.ci0 = ci0;
    H.ci1 = ci1;
    H.ci2 = ci2;
    H.nx0 = sd.nxyz[0]; H.nx1 = sd.nxyz[1]; H.nx2 = sd.nxyz[2];
    H.sx = 2 * H.nx0 + 1;
    H.sy = 2 * H.nx1 + 1;
    H.nseg = H.sx * H.sy * (2 * H.nx2 + 1);
    H.p0 = sd.pbc & 1; H.p1 = (sd.pbc >> 1) & 1; H.p2 = (sd.pbc >> 2) & 1;
}

// Neighbour cells sb .. sb+63 of the home cell, one per lane, in the
// reference order.  cell_atoms(c, start, count) gives the sorted atoms of
// the system's cell c.  Returns the number of candidate atoms in the batch
// (wave-uniform); per lane: exclusive prefix, first sorted index, shift.
template <typename F>
__device__ __forceinline__ int segment_batch(const HomeCell &H, int sb, int &excl, int &start_g, uint32_t &shp,
                                             F &&cell_atoms)
{
    const int g = sb + lane_id();
    int cnt_g = 0;
    start_g = 0;
    shp = 0;
    if (g < H.nseg) {
        const int dx = g % H.sx - H.nx0;
        const int t = g / H.sx;
        const int dy = t % H.sy - H.nx1;
        const int dz = t / H.sy - H.nx2;
        const int a0 = H.ci0 + dx, a1 = H.ci1 + dy, a2 = H.ci2 + dz;
        // _is_cell_in_bounds (gpu_kernels.jl:20-25)
        const bool inb = (H.p0 || (a0 >= 1 && a0 <= H.n0)) && (H.p1 || (a1 >= 1 && a1 <= H.n1)) &&
                         (H.p2 || (a2 >= 1 && a2 <= H.n2));
        if (inb) {
            int32_t c0, c1, c2, s0, s1, s2;   // _get_neighbor_cell (:39-47)
            wrap_and_shift(a0, H.n0, H.p0, c0, s0);
            wrap_and_shift(a1, H.n1, H.p1, c1, s1);
            wrap_and_shift(a2, H.n2, H.p2, c2, s2);
            cell_atoms((c0 - 1) + (c1 - 1) * H.n0 + (c2 - 1) * H.n0 * H.n1, start_g, cnt_g);
            shp = pack_wind(s0, s1, s2);
        }
    }
    const int incl = wave_incl_scan(cnt_g);
    excl = incl - cnt_g;
    return sgpr(__shfl(incl, kWave - 1, kWave));
}

struct Cand {
    double x, y, z;
    int32_t j;
    int32_t tx, ty, tz;         // s_loop - w_j  (S = t + w_i)
    bool zero_shift, valid;
};

// Candidate k of a segment batch: its place in the sorted order (below the
// batch's end only for k < its total) and its segment's packed shift.
__device__ __forceinline__ int candidate_place(int k, int excl, int start_g, uint32_t shp, uint32_t &shm)
{
    int m = 0;
#pragma unroll
    for (int step = 32; step >= 1; step >>= 1) {
        const int e2 = __shfl(excl, m + step, kWave);
        if (e2 <= k) m += step;
    }
    shm = __shfl(shp, m, kWave);
    return __shfl(start_g, m, kWave) + (k - __shfl(excl, m, kWave));
}

__device__ __forceinline__ Cand load_candidate(const PairsArgs &A, int k, int total, int excl, int start_g, uint32_t shp)
{
    uint32_t shm;
    const int p = candidate_place(k, excl, start_g, shp, shm);
    Cand c;
    c.valid = k < total;
    int32_t wjx = 0, wjy = 0, wjz = 0;
    if (c.valid) {
        const Rec r = A.rec[p];
        c.x = r.x; c.y = r.y; c.z = r.z;
        c.j = r.j;
        rec_winding(r, A.wbig, p, wjx, wjy, wjz);
    } else {
        c.x = c.y = c.z = 0.0;
        c.j = -1;
    }
    int32_t sx, sy, sz;
    unpack_wind(shm, sx, sy, sz);
    c.zero_shift = (sx == 0) & (sy == 0) & (sz == 0);
    c.tx = sx - wjx;
    c.ty = sy - wjy;
    c.tz = sz - wjz;
    return c;
}

// Per-wave count of the home atoms hs .. he - 1 (up to a wave of them) of one
// cell from global memory: test every (home atom, chunk) and append hits to
// the slots (the brick path's fallback, and the path for neighbour reach
// beyond one cell).
template <bool WIDE>
__device__ __forceinline__ void count_group(const PairsArgs &A, const SysDev &sd, int lc, int32_t hg, int nh,
                                            int32_t *__restrict__ pair_count, const SlotArgs &O)
{
    HomeCell H;
    home_grid(sd, lc % sd.n[0] + 1, (lc / sd.n[0]) % sd.n[1] + 1, lc / (sd.n[0] * sd.n[1]) + 1, H);
    const int lane = lane_id();
    const double *__restrict__ Cm = sd.C;
    const double rc2 = sd.rc2;
    const int32_t hj_lane = lane < nh ? A.rec[hg + lane].j : 0;
    int32_t cnt_lane = 0;   // lane a: running count of home atom hg + a
    for (int sb = 0; sb < H.nseg; sb += kWave) {
        int excl, start_g;
        uint32_t shp;
        const int total = segment_batch(H, sb, excl, start_g, shp, [&](int c, int &st, int &n) {
            st = A.cell_start[H.cbase + c];
            n = A.cell_start[H.cbase + c + 1] - st;
        });
        for (int k0 = 0; k0 < total; k0 += kChunksPerPass * kWave) {
            const int nch = sgpr(min(kChunksPerPass, (total - k0 + kWave - 1) / kWave));
            Cand c[kChunksPerPass];
            uint32_t tpk[kChunksPerPass];
            uint64_t own[kChunksPerPass];   // candidates with no cell shift: the home atom's own is one of them
#pragma unroll
            for (int g = 0; g < kChunksPerPass; ++g) {
                own[g] = 0;
                tpk[g] = 0;
                if (g < nch) {
                    c[g] = load_candidate(A, k0 + g * kWave + lane, total, excl, start_g, shp);
                    if (!c[g].valid) c[g].x = c[g].y = c[g].z = kFar;
                    own[g] = __builtin_amdgcn_ballot_w64(c[g].zero_shift);
                    tpk[g] = pack_wind(c[g].tx, c[g].ty, c[g].tz);
                } else {
                    c[g].x = c[g].y = c[g].z = kFar;
                    c[g].j = -1;
                    c[g].tx = c[g].ty = c[g].tz = 0;
                }
            }
            double cx[kChunksPerPass], cy[kChunksPerPass], cz[kChunksPerPass];
            uint32_t wcache = 0xffffffffu;
            int32_t wix = 0, wiy = 0, wiz = 0;
            for (int a = 0; a < nh; ++a) {
                const Rec h = A.rec[hg + a];   // wave-uniform: scalar loads
                if (h.w != wcache || (h.w & kWindBig)) {
                    rec_winding(h, A.wbig, hg + a, wix, wiy, wiz);
#pragma unroll
                    for (int g = 0; g < kChunksPerPass; ++g)
                        cell_shift(Cm, c[g].tx + wix, c[g].ty + wiy, c[g].tz + wiz, cx[g], cy[g], cz[g]);
                    wcache = h.w;
                }
                const bool wzero = (wix | wiy | wiz) == 0;
                int32_t ca = __builtin_amdgcn_readlane(cnt_lane, a);
                const int64_t sbase = (H.abase + __builtin_amdgcn_readlane(hj_lane, a)) * (int64_t)O.cap;
#pragma unroll
                for (int g = 0; g < kChunksPerPass; ++g) {
                    if (g < nch) {
                        const double Rx = (c[g].x - h.x) + cx[g];
                        const double Ry = (c[g].y - h.y) + cy[g];
                        const double Rz = (c[g].z - h.z) + cz[g];
                        const double r2 = (Rx * Rx + Ry * Ry) + Rz * Rz;
                        const uint64_t mask = __builtin_amdgcn_ballot_w64(r2 < rc2) &
                                              ~(__builtin_amdgcn_ballot_w64(c[g].j == h.j) & own[g]);
                        emit_hits<WIDE>(O, mask, sbase, ca, c[g].j, c[g].tx + wix, c[g].ty + wiy, c[g].tz + wiz, wzero, tpk[g]);
                    }
                }
                cnt_lane = lane == a ? ca : cnt_lane;
            }
        }
    }
    if (lane < nh) pair_count[H.abase + hj_lane] = cnt_lane | kRow8Bit;
}

// ---------------------------------------------------------------------------
// lazy queries: the neighbours of a range of atoms
// ---------------------------------------------------------------------------

// for_each_neighbour (cell_list.jl:779-801) of atoms i_first .. i_first + n - 1
// of one system, one wave per atom: its neighbour cells one per lane, their
// atoms flattened in the reference order, 64 candidates tested at a time, so
// a hit's place is the hits before it.  Without FILL the neighbours are
// counted, with it they are written from off[a] on (nothing when the total
// off[n] exceeds cap: the host grows the outputs and runs it again).
//
// Every position, the home atom's and the candidates', is read from X, as
// nlh_for_each_neighbour (nlhip_device.h) reads it: the caller may have moved
// atoms since the build, and R_ij = -R_ji and the one-atom query hold all the
// same.
//
// Latency-bound: a query of a few thousand atoms is one wave per SIMD.  With
// one thread per atom walking the cells the two passes over 4,096 atoms of a
// 50,000-atom cube took 248 us each; a wave per atom takes 12 and 15 us.
template <typename TI, bool FILL>
__global__ __launch_bounds__(kPairsBlock) void lazy_range_kernel(LazyRange Q)
{
    const int64_t a = (int64_t)blockIdx.x * kWavesPerPairsBlock + sgpr((int)(threadIdx.x / kWave));
    if (a >= Q.n) return;   // wave-uniform
    int64_t run = 0, end = 0;
    if (FILL) {
        if (Q.off[Q.n] > Q.cap) return;
        run = Q.off[a];
        end = Q.off[a + 1];   // never past the atom's own run, whatever becomes of X between the passes
    }
    const SysDev &sd = *Q.sys;
    const int64_t il = Q.i_first + a;   // 0-based, local to the system
    const double *xi = Q.X + 3 * (sd.atom_base + il);
    const double hx = xi[0], hy = xi[1], hz = xi[2];
    int32_t ci[3], wi[3];
    cell_and_winding(sd, hx, hy, hz, ci, wi);
    HomeCell H;
    home_grid(sd, ci[0], ci[1], ci[2], H);
    const TI *co = static_cast<const TI *>(Q.cell_offsets) + (int64_t)sd.cell_base + Q.isys;
    const TI *perm = static_cast<const TI *>(Q.perm);
    const int lane = lane_id();
    const double rc2 = sd.rc2;
    for (int sb = 0; sb < H.nseg; sb += kWave) {
        int excl, start_g;
        uint32_t shp;
        const int total = segment_batch(H, sb, excl, start_g, shp, [&](int c, int &st, int &n) {
            const int64_t s0 = (int64_t)co[c];
            st = (int)(sd.atom_base + s0 - 1);
            n = (int)((int64_t)co[c + 1] - s0);
        });
        for (int k0 = 0; k0 < total; k0 += kWave) {
            uint32_t shm;
            const int p = candidate_place(k0 + lane, excl, start_g, shp, shm);
            const bool valid = k0 + lane < total;
            const int32_t j = valid ? (int32_t)perm[p] - 1 : 0;   // 0-based, local to the system
            const double *xj = Q.X + 3 * (sd.atom_base + j);
            const double x = xj[0], y = xj[1], z = xj[2];
            int32_t cj[3], wj[3], s[3];
            cell_and_winding(sd, x, y, z, cj, wj);
            unpack_wind(shm, s[0], s[1], s[2]);
            // S = s_loop + w_i - w_j  (gpu_kernels.jl:88)
            const int32_t Sx = s[0] + wi[0] - wj[0], Sy = s[1] + wi[1] - wj[1], Sz = s[2] + wi[2] - wj[2];
            double cx, cy, cz;
            cell_shift(sd.C, Sx, Sy, Sz, cx, cy, cz);
            const double Rx = (x - hx) + cx, Ry = (y - hy) + cy, Rz = (z - hz) + cz;
            const double r2 = (Rx * Rx + Ry * Ry) + Rz * Rz;
            const bool self = j == (int32_t)il && (s[0] | s[1] | s[2]) == 0;
            const bool hit = valid & (r2 < rc2) & !self;
            const uint64_t m = __ballot(hit);
            const int64_t q = run + mbcnt64(m);
            if (FILL && hit && q < end) {
                static_cast<TI *>(Q.j)[q] = (TI)(j + 1);
                double *R = Q.R + 3 * q;
                R[0] = Rx;
                R[1] = Ry;
                R[2] = Rz;
                TI *S = static_cast<TI *>(Q.S) + 3 * q;
                S[0] = (TI)Sx;
                S[1] = (TI)Sy;
                S[2] = (TI)Sz;
            }
            run += __popcll(m);
        }
    }
    if (!FILL && lane == 0) Q.count[a] = (int32_t)run;
}

void launch_lazy_range(const LazyRange &q, int ti_bytes, bool fill, hipStream_t st)
{
    if (q.n <= 0) return;
    const dim3 grid((unsigned)((q.n + kWavesPerPairsBlock - 1) / kWavesPerPairsBlock)), block(kPairsBlock);
    if (ti_bytes == 8) {
        if (fill) hipLaunchKernelGGL((lazy_range_kernel<int64_t, true>), grid, block, 0, st, q);
        else hipLaunchKernelGGL((lazy_range_kernel<int64_t, false>), grid, block, 0, st, q);
    } else {
        if (fill) hipLaunchKernelGGL((lazy_range_kernel<int32_t, true>), grid, block, 0, st, q);
        else hipLaunchKernelGGL((lazy_range_kernel<int32_t, false>), grid, block, 0, st, q);
    }
}

// Brick workgroup shapes: BT threads (8 waves for large systems, 4 for
// batches of small ones), 4 BT halo atoms and BT halo cells in LDS.
template <int BT>
struct BrickShape {
    static constexpr int threads = BT;
    static constexpr int waves = BT / kWave;
    static constexpr int cap = 4 * BT;    // halo atoms held in LDS
    static constexpr int halo = BT;       // halo cells, one per thread
    static constexpr int unroll = cap / BT;
};
constexpr uint32_t kPackZero = (512u) | (512u << 10) | (512u << 20);   // pack_wind(0, 0, 0)
constexpr int kBrickChunks = 3;   // candidate chunks a lane holds in the brick pass (192 candidates)

// Quotient of 0 <= x < 2^16 by 1 <= d < 2^16 through a reciprocal: m =
// floor((2^32 - 1) / d) + 1 (0 for d = 1), q = umulhi(x, m).  Exact: m
// exceeds 2^32 / d by less than one, so the product overshoots x / d by less
// than x / 2^32 < 1 / d, which never carries past the next integer.  A few
// instructions instead of the integer-division sequence.
struct SmallDiv {
    uint32_t d, m;
};

__device__ __forceinline__ SmallDiv small_div(int d)
{
    return {(uint32_t)d, d == 1 ? 0u : 0xffffffffu / (uint32_t)d + 1u};
}

__device__ __forceinline__ int small_quot(int x, SmallDiv D)
{
    return D.m ? (int)__umulhi((uint32_t)x, D.m) : x;
}

struct Brick {
    const SysDev *sd;
    int b0[3];     // 1-based coordinates of the first home cell
    int nh[3];     // home cells per axis (clipped at the grid edge)
    int hd[3];     // halo extent per axis (nh + 2)
    int nhalo, nhome;
    bool fast;     // one-cell reach and a small enough halo: the LDS path applies
    SmallDiv dnh0, dnh1, dhd0, dhd1;   // divisors nh[0], nh[1], hd[0], hd[1]
};

// Brick of workgroup w of a count launch: the bricks of the launch in
// system order, each system's in its class order, largest first
// (SysDev::cls_first).  Workgroups are dealt to the eight XCDs in turn, so
// every XCD takes its share of each class and of every region of a system
// (a slab with vacuum above it puts its empty bricks on every XCD, not on
// some of them).
__device__ __forceinline__ void brick_locate(const PairsArgs &A, const int32_t *__restrict__ sys_brick_base, int w,
                                             int halo_max, Brick &B)
{
    const int s = A.nsys == 1 ? 0 : find_sys(sys_brick_base, A.nsys, (int32_t)w);
    const SysDev &sd = A.sys[s];
    B.sd = &sd;
    int li = w - sys_brick_base[s], c = 0;
#pragma unroll
    for (int cc = 1; cc < 8; ++cc) c = li >= sd.cls_first[cc] ? cc : c;
    li -= sd.cls_first[c];
    // brick (ib0, ib1, ib2) of the class: the partial last brick along the
    // axes of its mask, row-major over the full bricks along the others
    const int m = sd.cls_mask[c];
    const int d0 = (m & 1) ? 1 : sd.bfull[0], d1 = (m & 2) ? 1 : sd.bfull[1];
    const int q0 = li / d0;
    const int ib[3] = {(m & 1) ? sd.bfull[0] : li - q0 * d0, (m & 2) ? sd.bfull[1] : q0 % d1,
                       (m & 4) ? sd.bfull[2] : q0 / d1};
    for (int k = 0; k < 3; ++k) {
        B.b0[k] = ib[k] * sd.brick[k] + 1;
        B.nh[k] = min(sd.brick[k], sd.n[k] - B.b0[k] + 1);
        B.hd[k] = B.nh[k] + 2;
    }
    B.nhalo = B.hd[0] * B.hd[1] * B.hd[2];
    B.nhome = B.nh[0] * B.nh[1] * B.nh[2];
    B.fast = sd.nxyz[0] == 1 && sd.nxyz[1] == 1 && sd.nxyz[2] == 1 && B.nhalo <= halo_max;
    B.dnh0 = small_div(B.nh[0]);
    B.dnh1 = small_div(B.nh[1]);
    B.dhd0 = small_div(B.hd[0]);
    B.dhd1 = small_div(B.hd[1]);
}

// wrap_and_shift (cell_list.jl:105-120) of an index within one cell of
// [1, n] on a periodic axis (a halo cell of a one-cell-reach brick): at most
// one wrap, no division.
__device__ __forceinline__ void wrap_near(int32_t a, int32_t n, int32_t &w, int32_t &s)
{
    s = a < 1 ? -1 : (a > n ? 1 : 0);
    w = a - s * n;
}

__device__ __forceinline__ int brick_cell_id(const Brick &B, int hc)
{
    const SysDev &sd = *B.sd;
    const int ix = hc % B.nh[0], iy = (hc / B.nh[0]) % B.nh[1], iz = hc / (B.nh[0] * B.nh[1]);
    return sd.cell_base + (B.b0[0] - 1 + ix) + (B.b0[1] - 1 + iy) * sd.n[0] + (B.b0[2] - 1 + iz) * sd.n[0] * sd.n[1];
}

// A brick's home cells from global memory: each cell's home atoms in groups,
// all groups dealt to the `parts` waves in turn, so that a cell which atoms
// were clamped into (thousands of them) or the one cell of a brick is shared,
// and no cell is looked at twice.  Every group loads the cell's candidates:
// groups smaller than a wave only where they must be (100k atoms shifted by a
// quarter of an open axis, whole builds: groups of 48 above 64 atoms 320 us, of
// 16 above 32 a tenth more; 10k in a corner of an open cell 263 with either).
constexpr int kShareGroup = 48;
template <bool WIDE>
__device__ __forceinline__ void count_cells(const PairsArgs &A, const Brick &B, int32_t *__restrict__ pair_count,
                                            const SlotArgs &O, int part, int parts)
{
    const SysDev &sd = *B.sd;
    const int lane = lane_id();
    int st = 0, n = 0, cell = 0;   // home cell `lane`
    if (lane < B.nhome) {
        cell = brick_cell_id(B, lane);
        st = A.cell_start[cell];
        n = A.cell_start[cell + 1] - st;
    }
    // home atoms of a group: a cell's own, an even share of a large one, or, where
    // the waves outnumber the cells, a wave's share
    const int shares = (n + kShareGroup - 1) / kShareGroup;
    int gs = n > kWave ? (n + shares - 1) / shares : kWave;
    if (B.nhome < parts) gs = min(gs, max(1, (int)(((int64_t)n * B.nhome + parts - 1) / parts)));
    const int g = (n + gs - 1) / gs, incl = wave_incl_scan(g);
    const int items = __builtin_amdgcn_readlane(incl, kWave - 1);
    for (int it = part; it < items; it += parts) {
        const int c = (int)__popcll(__builtin_amdgcn_ballot_w64(incl <= it));   // the item's cell
        const int cg = __builtin_amdgcn_readlane(gs, c);
        const int o = (it - (__builtin_amdgcn_readlane(incl, c) - __builtin_amdgcn_readlane(g, c))) * cg;
        count_group<WIDE>(A, sd, __builtin_amdgcn_readlane(cell, c) - sd.cell_base, __builtin_amdgcn_readlane(st, c) + o,
                          min(cg, __builtin_amdgcn_readlane(n, c) - o), pair_count, O);
    }
}

// One halo atom in LDS, 32 bytes: a candidate is two 16-byte reads.
struct __attribute__((aligned(16))) LAtom {
    double x, y, z;
    int32_t j;
    uint32_t t;                     // pack(s_halo - w_j); home cells have s_halo = 0
};

constexpr int kPassCands = kBrickChunks * kWave;   // candidates of one pass (three chunks)

template <int BT>
struct BrickLDS {
    using Sh = BrickShape<BT>;
    // entry cap is a far-away atom that lanes past the last candidate read,
    // so candidate loads need no per-lane branch
    LAtom a[Sh::cap + 1];
    int32_t hoff[Sh::halo + 1];     // LDS offset of each halo cell's atoms
    int32_t hstart[Sh::halo];       // first sorted index of each halo cell
    uint32_t hshift[Sh::halo];      // packed cell shift of each halo cell | kHomeCell
    // per wave, for its current home cell: the LDS offset less the candidate
    // prefix of each non-empty candidate row (in row order), and one byte per
    // candidate of the current pass marking where a non-empty row starts
    int32_t rowdl[Sh::waves][16];
    uint32_t rowflag[Sh::waves][kPassCands / 4];
    uint16_t owner[Sh::cap];        // halo cell of each LDS atom slot (while loading)
    int32_t next_cell;              // the next home cell a wave takes
    int32_t total, flag;
};

constexpr uint32_t kHomeCell = 1u << 30;   // halo-table mark of the brick's own cells

// Stage the brick and its halo in LDS.  Returns false (for every thread of
// the block) when the brick must take the global-memory path.
template <int BT>
__device__ bool brick_load(const PairsArgs &A, const Brick &B, BrickLDS<BT> &L)
{
    using Sh = BrickShape<BT>;
    const SysDev &sd = *B.sd;
    const int tid = threadIdx.x;
    const bool p[3] = {(sd.pbc & 1) != 0, (sd.pbc & 2) != 0, (sd.pbc & 4) != 0};
    // halo cell table: thread tid owns halo cell tid
    int cnt[1];
    int sum = 0;
#pragma unroll
    for (int u = 0; u < 1; ++u) {
        cnt[u] = 0;
        const int h = tid + u;
        if (h < B.nhalo) {
            const int q0 = small_quot(h, B.dhd0), uz = small_quot(q0, B.dhd1);
            const int ux = h - q0 * B.hd[0], uy = q0 - uz * B.hd[1];
            const int a[3] = {B.b0[0] - 1 + ux, B.b0[1] - 1 + uy, B.b0[2] - 1 + uz};
            bool inb = true;
            for (int k = 0; k < 3; ++k) inb = inb && (p[k] || (a[k] >= 1 && a[k] <= sd.n[k]));
            int st = 0;
            uint32_t sh = kPackZero;
            if (inb) {   // _is_cell_in_bounds / _get_neighbor_cell (gpu_kernels.jl:20-47)
                int32_t c[3], sft[3];
                // a halo cell lies within one cell of the grid: an open axis
                // holds it in bounds here, a periodic one wraps it at most once
                for (int k = 0; k < 3; ++k) wrap_near(a[k], sd.n[k], c[k], sft[k]);
                const int gc = sd.cell_base + (c[0] - 1) + (c[1] - 1) * sd.n[0] + (c[2] - 1) * sd.n[0] * sd.n[1];
                st = A.cell_start[gc];
                cnt[u] = A.cell_start[gc + 1] - st;
                sh = pack_wind(sft[0], sft[1], sft[2]);
            }
            const bool home = ux >= 1 && ux <= B.nh[0] && uy >= 1 && uy <= B.nh[1] && uz >= 1 && uz <= B.nh[2];
            L.hstart[h] = st;
            L.hshift[h] = sh | (home ? kHomeCell : 0u);
        }
        sum += cnt[u];
    }
    int64_t tot;
    int run = (int)block_excl_scan_n<BT>(sum, tot);
#pragma unroll
    for (int u = 0; u < 1; ++u) {
        const int h = tid + u;
        if (h < B.nhalo) {
            L.hoff[h] = run;
            // the cell's atom slots name their cell (a brick whose halo
            // overflows the LDS takes the global-memory path)
            const int e = min(run + cnt[u], Sh::cap);
            for (int q = run; q < e; ++q) L.owner[q] = (uint16_t)h;
        }
        run += cnt[u];
    }
    if (tid == 0) {
        L.hoff[B.nhalo] = (int32_t)tot;
        L.total = (int32_t)tot;
        L.next_cell = Sh::waves;
        L.flag = 0;
        L.a[Sh::cap].x = L.a[Sh::cap].y = L.a[Sh::cap].z = kFar;
        L.a[Sh::cap].j = 0;
        L.a[Sh::cap].t = kPackZero;
    }
    __syncthreads();
    const int total = L.total;
    if (total > Sh::cap) return false;
    // halo atoms: all loads of a thread in flight together
    int pg[Sh::unroll];
    uint32_t hs[Sh::unroll];
#pragma unroll
    for (int u = 0; u < Sh::unroll; ++u) {
        const int idx = tid + u * BT;
        pg[u] = 0;
        hs[u] = kPackZero;
        if (idx < total) {
            const int h = L.owner[idx];
            pg[u] = L.hstart[h] + (idx - L.hoff[h]);
            hs[u] = L.hshift[h];
        }
    }
    Rec r[Sh::unroll];
#pragma unroll
    for (int u = 0; u < Sh::unroll; ++u)
        if (tid + u * BT < total) r[u] = A.rec[pg[u]];
#pragma unroll
    for (int u = 0; u < Sh::unroll; ++u) {
        const int idx = tid + u * BT;
        if (idx < total) {
            int32_t wx, wy, wz, sx, sy, sz;
            rec_winding(r[u], A.wbig, pg[u], wx, wy, wz);
            unpack_wind(hs[u] & ~kHomeCell, sx, sy, sz);
            const uint32_t t = pack_wind(sx - wx, sy - wy, sz - wz);
            if (t & kWindBig) L.flag = 1;
            LAtom la;
            la.x = r[u].x;
            la.y = r[u].y;
            la.z = r[u].z;
            la.j = r[u].j;
            la.t = t;
            L.a[idx] = la;
        }
    }
    __syncthreads();
    return L.flag == 0;
}

// Per home cell of a brick: its LDS atom range, first sorted index, the
// nine candidate rows (lane r < 9 holds row r) and the candidate index of
// the home cell's first atom (its own self candidate).
struct HomeRows {
    int h0, h1;      // LDS range of the home atoms (uniform)
    int rstart, rex; // per lane: LDS start and exclusive candidate prefix of row `lane`
    int len;         // per lane: candidates in row `lane`
    int total;       // candidates (uniform)
    int self0;       // candidate index of home atom 0 (uniform)
};

template <typename LDS>
__device__ __forceinline__ HomeRows brick_home(const Brick &B, const LDS &L, int hc)
{
    HomeRows R;
    const int q0 = small_quot(hc, B.dnh0), iz = small_quot(q0, B.dnh1);
    const int ix = hc - q0 * B.nh[0], iy = q0 - iz * B.nh[1];
    const int hh = (ix + 1) + B.hd[0] * ((iy + 1) + B.hd[1] * (iz + 1));
    R.h0 = sgpr(L.hoff[hh]);
    R.h1 = sgpr(L.hoff[hh + 1]);
    const int lane = lane_id();
    int len = 0, st = 0;
    if (lane < 9) {   // row (dz, dy) = (lane / 3 - 1, lane % 3 - 1); dx = -1..1 contiguous
        const int dz = lane / 3 - 1, dy = lane % 3 - 1;
        const int hr = ix + B.hd[0] * ((iy + 1 + dy) + B.hd[1] * (iz + 1 + dz));
        st = L.hoff[hr];
        len = L.hoff[hr + 3] - st;
    }
    // inclusive scan over lanes 0..8 (within the first 16-lane row)
    const int incl = row16_incl_scan(len);
    R.rex = incl - len;
    R.rstart = st;
    R.len = len;
    R.total = __builtin_amdgcn_readlane(incl, 8);
    // row 4 is (dz, dy) = (0, 0); the home cell is its middle cell
    R.self0 = __builtin_amdgcn_readlane(R.rex, 4) + (R.h0 - __builtin_amdgcn_readlane(R.rstart, 4));
    return R;
}

// LDS index of candidate k of a home cell (k < total): k plus the offset
// (LDS start - candidate prefix) of the last non-empty row whose first
// candidate is at or before k.  Per home cell the wave publishes the offsets
// of its non-empty rows in row order (rowdl[q], q = the row's rank among the
// non-empty rows).  Per pass of kPassCands candidates it marks with a byte
// each candidate where a non-empty row other than the first starts and turns
// the marks into one 64-bit word per chunk (a ballot); a candidate's rank q
// is then the number of marks at or below it: those of the chunks before (a
// popcount) and those of its own chunk up to its lane (mbcnt).  The row
// maps are the wave's own LDS: written and read by the wave alone, in
// program order.
struct RowMap {
    uint64_t sh[kBrickChunks];   // marks of each chunk, shifted right by one (uniform)
    int base[kBrickChunks];      // marks before each chunk, plus the chunk's own first (uniform)
};

// Publish the row offsets of a home cell; returns this lane's rank among the
// non-empty rows (meaningful on the lanes of non-empty rows, `ne`).
template <typename LDS>
__device__ __forceinline__ int row_publish(const HomeRows &R, LDS &L, int wv, bool &ne)
{
    const int lane = lane_id();
    ne = lane < 9 && R.len > 0;
    const int q = (int)mbcnt64(__builtin_amdgcn_ballot_w64(ne));
    if (ne) L.rowdl[wv][q] = R.rstart - R.rex;
    return q;
}

template <typename LDS>
__device__ __forceinline__ RowMap row_map(const HomeRows &R, LDS &L, int wv, int k0, int q, bool ne)
{
    const int lane = lane_id();
    uint8_t *fl = reinterpret_cast<uint8_t *>(L.rowflag[wv]);
    if (lane < kPassCands / 4) L.rowflag[wv][lane] = 0u;
    const int p = R.rex - k0;   // pass-relative first candidate of row `lane`
    if (ne && q > 0 && p > 0 && p < kPassCands) fl[p] = 1;
    int acc = (int)__popcll(__builtin_amdgcn_ballot_w64(ne && q > 0 && p <= 0));
    RowMap M;
#pragma unroll
    for (int g = 0; g < kBrickChunks; ++g) {
        const uint64_t b = __builtin_amdgcn_ballot_w64(fl[g * kWave + lane] != 0);
        M.sh[g] = b >> 1;
        M.base[g] = acc + (int)(b & 1u);
        acc += (int)__popcll(b);
    }
    return M;
}

template <typename LDS>
__device__ __forceinline__ int row_index(const RowMap &M, const LDS &L, int wv, int g, int k)
{
    const int q = M.base[g] + (int)mbcnt64(M.sh[g]);
    return k + L.rowdl[wv][q];
}

// First slot of atom e's row: both factors are below 2^31, so one 32 x 32 -> 64
// bit product.
__device__ __forceinline__ int64_t slot_row(int64_t e, int32_t cap)
{
    return (int64_t)((uint64_t)(uint32_t)e * (uint32_t)cap);
}

constexpr int32_t kRawBufferWord3 = 0x00020000; // raw 32-bit buffer access (GFX9 family)

// One (home atom, chunk) test of the brick pass, its hits appended to the home
// atom's row of 16-byte entries at its running count ca (wave-uniform).  SHIFT:
// add the candidate's cell shift C' S (left out when every lane's shift is
// zero: r^2 is then the same).  `self` clears the home atom's own (j == i, s ==
// 0) candidate from the ballot when it lies in this chunk.  ent = j | pack(s -
// w_j) << 32.
template <bool SHIFT>
__device__ __forceinline__ void test_chunk(double cx, double cy, double cz, double sx, double sy, double sz, double hx,
                                           double hy, double hz, double rc2, uint64_t self, int4 *__restrict__ row,
                                           int32_t cap, int32_t &ca, uint64_t ent, int32_t wix, int32_t wiy, int32_t wiz)
{
    // R = xj - xi + C' * S ; r^2 = dot(R, R)  (gpu_kernels.jl:89-92)
    double Rx = cx - hx, Ry = cy - hy, Rz = cz - hz;
    if (SHIFT) {
        Rx = Rx + sx;
        Ry = Ry + sy;
        Rz = Rz + sz;
    }
    const double r2 = (Rx * Rx + Ry * Ry) + Rz * Rz;
    const uint64_t m = __builtin_amdgcn_ballot_w64(r2 < rc2) & self;
    if (m == 0) return;
    const int32_t rank = ca + (int32_t)mbcnt64(m);
    if (((m >> lane_id()) & 1) && rank < cap) {
        // S = s_loop + w_i - w_j  (gpu_kernels.jl:88)
        int32_t tx, ty, tz;
        unpack_wind((uint32_t)(ent >> 32), tx, ty, tz);
        row[rank] = make_int4((int32_t)(uint32_t)ent, tx + wix, ty + wiy, tz + wiz);
    }
    ca += (int32_t)__popcll(m);
}

// One pass of a home cell's atoms over loaded candidate chunks: every home
// atom's distance tests against the nch chunks (cx, cy, cz, ent), its hits
// appended to its slot row at its running count (lane a of cnt_l for home
// atom a).  home: the nh home atoms in LDS; ht_l, hj_l: lane a holds
// pack(-w_i) and j of home atom a; kpass: the self candidate of home atom 0
// in this pass (home atom a's is kpass + a); Cm: the cell matrix.
__device__ __forceinline__ void pass_home_atoms(int nch, const double *cx, const double *cy, const double *cz,
                                                const uint64_t *ent, const LAtom *home, int nh, uint32_t ht_l,
                                                int32_t hj_l, int kpass, const double *Cm, double rc2,
                                                int64_t atom_base, void *__restrict__ slots, int32_t cap, int32_t &cnt_l)
{
    double sx[kBrickChunks], sy[kBrickChunks], sz[kBrickChunks];
    uint32_t wcur = 0xffffffffu;   // home winding the shifts were computed for
    int32_t wix = 0, wiy = 0, wiz = 0;
    // wave-uniform, per chunk: the lanes whose shift is nonzero (the
    // shifts sx, sy, sz are set only where this is nonzero)
    uint64_t csh[kBrickChunks];
    for (int a = 0; a < nh; ++a) {
        const LAtom hm = home[a];
        const uint32_t ht = (uint32_t)__builtin_amdgcn_readlane((int)ht_l, a);
        if (ht != wcur) {   // first home atom, or a new home winding
            int32_t tx, ty, tz;
            unpack_wind(ht, tx, ty, tz);
            wix = -tx; wiy = -ty; wiz = -tz;
#pragma unroll
            for (int g = 0; g < kBrickChunks; ++g) {
                csh[g] = 0;
                if (g < nch) {
                    int32_t cx_, cy_, cz_;
                    unpack_wind((uint32_t)(ent[g] >> 32), cx_, cy_, cz_);
                    cx_ += wix; cy_ += wiy; cz_ += wiz;
                    csh[g] = __builtin_amdgcn_ballot_w64((cx_ | cy_ | cz_) != 0);
                    if (csh[g] != 0) cell_shift(Cm, cx_, cy_, cz_, sx[g], sy[g], sz[g]);
                }
            }
            wcur = ht;
        }
        int32_t ca = __builtin_amdgcn_readlane(cnt_l, a);
        // slot rows are indexed by original atom index, so the fill reads them in order
        int4 *row = reinterpret_cast<int4 *>(slots) + slot_row(atom_base + __builtin_amdgcn_readlane(hj_l, a), cap);
        // _is_self_interaction: j == i with no cell shift is the home atom's own
        // slot in the home cell, candidate kpass + a: chunk gs (none when it
        // is out of the pass)
        const int gs = (kpass + a) >> 6;
        const uint64_t nself = ~(1ull << ((kpass + a) & (kWave - 1)));
#pragma unroll
        for (int g = 0; g < kBrickChunks; ++g) {
            if (g < nch) {
                const uint64_t self = g == gs ? nself : ~0ull;
                if (csh[g] != 0)
                    test_chunk<true>(cx[g], cy[g], cz[g], sx[g], sy[g], sz[g], hm.x, hm.y, hm.z, rc2, self, row, cap, ca,
                                     ent[g], wix, wiy, wiz);
                else
                    test_chunk<false>(cx[g], cy[g], cz[g], sx[g], sy[g], sz[g], hm.x, hm.y, hm.z, rc2, self, row, cap, ca,
                                      ent[g], wix, wiy, wiz);
            }
        }
        cnt_l = write_lane(ca, a, cnt_l);
    }
}

// Brick pass of the count with 16-byte slot entries: home atoms stream through the wave as scalars
// (read out of one-per-lane registers), candidates sit one per lane in
// registers, chunk by chunk; each (home atom, chunk) is one FP64 distance
// test and one ballot.  Bricks that cannot take this path (reach beyond one
// cell, halo over the LDS, windings beyond the packed range) are counted
// from global memory, one home cell per wave.
template <int BT>
__global__ __launch_bounds__(BT) void count_kernel(
    const SysDev *__restrict__ sys, const int32_t *__restrict__ sys_cell_base, const int32_t *__restrict__ sys_brick_base,
    int nsys, int32_t M, int64_t nat, const int32_t *__restrict__ cell_start, const Rec *__restrict__ rec,
    const int32_t *__restrict__ wbig, int32_t *__restrict__ pair_count, void *__restrict__ slots,
    int32_t cap, Status *__restrict__ status)
{
    __shared__ BrickLDS<BT> L;
    __shared__ double Csh[9];
    const PairsArgs A{sys, sys_cell_base, nsys, M, nat, cell_start, rec, wbig};
    Brick B;
    brick_locate(A, sys_brick_base, (int)blockIdx.x, BrickShape<BT>::halo, B);
    if (threadIdx.x < 9) Csh[threadIdx.x] = B.sd->C[threadIdx.x];   // visible after brick_load's barrier
    const bool lds = B.fast && brick_load(A, B, L);
    if (!lds) {
        const SlotArgs O{slots, cap, status};
        const int wv0 = sgpr((int)(threadIdx.x >> 6));
        count_cells<true>(A, B, pair_count, O, wv0, BrickShape<BT>::waves);
        return;
    }
    const SysDev &sd = *B.sd;
    const double rc2 = sd.rc2;
    const int lane = lane_id();
    const int wv = sgpr((int)(threadIdx.x >> 6));
    // home cells: one per wave, then the next one not taken (a wave that
    // ends its cell early takes the next at once)
    for (int hc = wv; hc < B.nhome; hc = take_next(&L.next_cell)) {
        const HomeRows R = brick_home(B, L, hc);
        bool rne;
        const int rq = row_publish(R, L, wv, rne);
        const int nha = R.h1 - R.h0;
        for (int hg = 0; hg < nha; hg += kWave) {
            const int nh = sgpr(min(kWave, nha - hg));
            const int hb = R.h0 + hg;        // LDS index of home atom hg (uniform)
            const int hl = hb + (lane < nh ? lane : 0);
            const uint32_t ht_l = L.a[hl].t;   // pack(-w_i): a home cell's own shift is zero
            const int32_t hj_l = L.a[hl].j;
            const int kself = R.self0 + hg;  // candidate index of home atom hg + a is kself + a
            int32_t cnt_l = 0;                // lane a: running count of home atom hg + a
            for (int k0 = 0; k0 < R.total; k0 += kBrickChunks * kWave) {
                const int nch = sgpr(min(kBrickChunks, (R.total - k0 + kWave - 1) / kWave));
                const RowMap Mp = row_map(R, L, wv, k0, rq, rne);
                double cx[kBrickChunks], cy[kBrickChunks], cz[kBrickChunks];
                uint64_t ent[kBrickChunks];   // j | pack(s - w_j) << 32
#pragma unroll
                for (int g = 0; g < kBrickChunks; ++g) {
                    // every chunk of the pass is loaded (no branch): lanes past the
                    // last candidate read the far sentinel, and chunks past nch
                    // are never tested
                    const int k = k0 + g * kWave + lane;
                    const int lr = row_index(Mp, L, wv, g, k);
                    const int li = k < R.total ? lr : BrickShape<BT>::cap;   // else the far sentinel
                    const LAtom c = L.a[li];
                    cx[g] = c.x;
                    cy[g] = c.y;
                    cz[g] = c.z;
                    ent[g] = (uint64_t)(uint32_t)c.j | ((uint64_t)c.t << 32);
                }
                pass_home_atoms(nch, cx, cy, cz, ent, L.a + hb, nh, ht_l, hj_l, kself - k0, Csh, rc2, sd.atom_base, slots,
                                cap, cnt_l);
            }
            if (lane < nh) pair_count[sd.atom_base + hj_l] = cnt_l | kRow8Bit;
        }
    }
}

// Append one chunk's hits (m) to a home atom's slot row: 4-byte entries (lo),
// or 8-byte ones (lo, hi).  rs is a structured buffer over the row, so the
// byte offset of its filled part.  The hit mask is the exec mask of the store
// and a lane's rank among the hits its index.  The kernel is bound by how
// many instructions its waves issue, scalar ones included: this is six of
// them and the store, where a raw buffer store of every lane (at rank and
// count shifted to a byte offset, or past the row's end) took nine.
//
// A row that overflows runs on into the next ones (kSlotSlack bytes after
// the last row take the last ones' overflow): the host sees the count, and
// the rows are grown and counted again before anything reads them.
//
// The assembler knows no hazards here, so the block keeps them itself: rs
// comes from v_readlane, and a vector write of a scalar register wants five
// wait states before a buffer instruction reads it.
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

template <bool NARROW>
__device__ __forceinline__ void emit_chunk(v4u rs, uint64_t m, int32_t &so, uint32_t lo, uint32_t hi)
{
    uint32_t ix;
    int32_t n, next;
#define NLH_EMIT(shift, store)                   \
    "s_mov_b64 exec, %4\n\t"                     \
    "s_bcnt1_i32_b64 %1, %4\n\t"                 \
    shift " %2, %1, %3\n\t"                      \
    "v_mbcnt_lo_u32_b32 %0, exec_lo, 0\n\t"      \
    "v_mbcnt_hi_u32_b32 %0, exec_hi, %0\n\t"     \
    store " %5, %0, %6, %3 idxen\n\t"            \
    "s_mov_b64 exec, -1"
    if constexpr (NARROW)
        __asm__ volatile(NLH_EMIT("s_lshl2_add_u32", "buffer_store_dword")
                         : "=&v"(ix), "=&s"(n), "=&s"(next)
                         : "s"(so), "s"(m), "v"(lo), "s"(rs)
                         : "scc");
    else
        __asm__ volatile(NLH_EMIT("s_lshl3_add_u32", "buffer_store_dwordx2")
                         : "=&v"(ix), "=&s"(n), "=&s"(next)
                         : "s"(so), "s"(m), "v"((uint64_t)lo | (uint64_t)hi << 32), "s"(rs)
                         : "scc");
#undef NLH_EMIT
    so = next;
}

// ---------------------------------------------------------------------------
// the brick count with 32-bit positions
// ---------------------------------------------------------------------------

// A halo atom of tile_kernel: its position as the brick sees it (cell shift
// and winding applied, relative to the brick's origin) in 32 bits, and j, or
// j | S code << 26 when every j fits in 26 bits.  One 16-byte read.
struct __attribute__((aligned(16))) TAtom {
    float x, y, z;
    int32_t j;
};

constexpr int kTileChunks = 4;                       // candidate chunks a lane holds in a pass
constexpr int kTileCands = kTileChunks * kWave;
constexpr int kTileHome = 64;                        // home cells of a brick at most (choose_brick)

template <int BT>
struct TileLDS {
    using Sh = BrickShape<BT>;
    // entry cap is a far-away atom that lanes past the last candidate read
    TAtom a[Sh::cap + 1];
    uint32_t t[Sh::cap + 1];        // pack(t' = s - w - (s - w) of the origin atom); S = t'_j - t'_i
    int32_t hoff[Sh::halo + 1];     // LDS offset of each halo cell's atoms
    int32_t hstart[Sh::halo];       // first sorted index of each halo cell
    uint32_t hshift[Sh::halo];      // packed cell shift of each halo cell | kHomeCell
    // per wave, for its current run of home cells (as in BrickLDS): row
    // offsets, and one byte per candidate of a pass where a row starts
    int32_t rowdl[Sh::waves][16];
    uint32_t rowflag[Sh::waves][kTileCands / 4];
    uint16_t owner[Sh::cap];        // halo cell of each LDS atom slot
    float ctr[kTileHome][3];        // centre of each run of home cells
    int32_t next_item;              // the next work item a wave takes
    int32_t total, flag;
    int32_t row8;                   // some shift needs 8-byte slot entries
    int32_t far2;                   // largest |p|^2 beyond the system's pmax2 (its bits), or 0
};

constexpr uint32_t kFieldsLow = 1u | (1u << 10) | (1u << 20);

// The runs of a brick: sd.run home cells next to each other along x, the last
// of a row possibly shorter.
struct TileRuns {
    int w, nx, n;          // cells of a run, runs of a row, runs
    SmallDiv dnx;          // divisor nx
};

__device__ __forceinline__ TileRuns tile_runs(const Brick &B)
{
    TileRuns T;
    T.w = B.sd->run;
    T.nx = T.w == 1 ? B.nh[0] : (B.nh[0] + 1) >> 1;
    T.n = T.nx * B.nh[1] * B.nh[2];
    T.dnx = small_div(T.nx);
    return T;
}

// First home cell (0-based in the brick) and cells of run r.
__device__ __forceinline__ void tile_run(const Brick &B, const TileRuns &T, int r, int &ix, int &iy, int &iz, int &w)
{
    const int q0 = small_quot(r, T.dnx);
    iz = small_quot(q0, B.dnh1);
    iy = q0 - iz * B.nh[1];
    ix = (r - q0 * T.nx) * T.w;
    w = min(T.w, B.nh[0] - ix);
}

// Whether the S = t'_j - t'_i of any two of the brick's atoms packs (then each
// t' relative to the origin atom's did): the windings of all of them are
// packed ones, and their s - w span at most 510 along each axis.  Looked at
// only where some winding is beyond +-128, as in trajectories whose positions
// were never wrapped.
template <int BT>
__device__ bool tile_windings_near(const PairsArgs &A, TileLDS<BT> &L, int total)
{
    using Sh = BrickShape<BT>;
    const int tid = threadIdx.x;
    int32_t *far = &L.rowdl[0][0];   // per axis the largest of 1100 + (s - w) and of 1100 - (s - w), then a mark
    if (tid < 7) far[tid] = 0;
    __syncthreads();
    int m[6] = {0, 0, 0, 0, 0, 0};
    bool big = false;
    for (int idx = tid; idx < total; idx += BT) {
        const int h = L.owner[idx];
        const uint32_t w = A.rec[L.hstart[h] + (idx - L.hoff[h])].w;
        big |= (w & kWindBig) != 0;
        int32_t s[3], v[3];
        unpack_wind(L.hshift[h] & ~kHomeCell, s[0], s[1], s[2]);
        unpack_wind(w, v[0], v[1], v[2]);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            m[k] = max(m[k], 1100 + s[k] - v[k]);
            m[3 + k] = max(m[3 + k], 1100 - s[k] + v[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const int v = wave_max_pos(m[k]);
        if (lane_id() == kWave - 1) atomicMax(far + k, v);
    }
    if (big) far[6] = 1;
    __syncthreads();
    bool near = far[6] == 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) near = near && far[k] + far[3 + k] <= 2200 + 510;
    __syncthreads();   // read before the waves use the space
    return near;
}

// Stage the brick and its halo in LDS.  Returns false (for every thread of
// the block) when the brick must take the global-memory path: more halo
// atoms than the LDS holds, or windings too far apart.
template <int BT>
__device__ bool tile_load(const PairsArgs &A, const Brick &B, const TileRuns &T, TileLDS<BT> &L, const double *Csh)
{
    using Sh = BrickShape<BT>;
    const SysDev &sd = *B.sd;
    const int tid = threadIdx.x;
    const bool p[3] = {(sd.pbc & 1) != 0, (sd.pbc & 2) != 0, (sd.pbc & 4) != 0};
    // halo cell table: thread tid owns halo cell tid
    int cnt = 0;
    if (tid < B.nhalo) {
        const int q0 = small_quot(tid, B.dhd0), uz = small_quot(q0, B.dhd1);
        const int ux = tid - q0 * B.hd[0], uy = q0 - uz * B.hd[1];
        const int a[3] = {B.b0[0] - 1 + ux, B.b0[1] - 1 + uy, B.b0[2] - 1 + uz};
        bool inb = true;
        for (int k = 0; k < 3; ++k) inb = inb && (p[k] || (a[k] >= 1 && a[k] <= sd.n[k]));
        int st = 0;
        uint32_t sh = kPackZero;
        if (inb) {   // _is_cell_in_bounds / _get_neighbor_cell (gpu_kernels.jl:20-47)
            int32_t c[3], sft[3];
            for (int k = 0; k < 3; ++k) wrap_near(a[k], sd.n[k], c[k], sft[k]);
            const int gc = sd.cell_base + (c[0] - 1) + (c[1] - 1) * sd.n[0] + (c[2] - 1) * sd.n[0] * sd.n[1];
            st = A.cell_start[gc];
            cnt = A.cell_start[gc + 1] - st;
            sh = pack_wind(sft[0], sft[1], sft[2]);
        }
        const bool home = ux >= 1 && ux <= B.nh[0] && uy >= 1 && uy <= B.nh[1] && uz >= 1 && uz <= B.nh[2];
        L.hstart[tid] = st;
        L.hshift[tid] = sh | (home ? kHomeCell : 0u);
    }
    int tot;
    const int run = block_excl_scan32<BT>(cnt, tot);
    if (tid < B.nhalo) {
        L.hoff[tid] = run;
        // the cell's atom slots name their cell (a brick whose halo
        // overflows the LDS takes the global-memory path)
        const int e = min(run + cnt, Sh::cap);
        for (int q = run; q < e; ++q) L.owner[q] = (uint16_t)tid;
    }
    if (tid == 0) {
        L.hoff[B.nhalo] = tot;
        L.next_item = Sh::waves;
        L.flag = 0;
        L.far2 = 0;
        L.row8 = sd.nat > kNarrowMaxAtoms ? 1 : 0;
        L.a[Sh::cap] = TAtom{kFar32, 0.0f, 0.0f, 0};
        L.t[Sh::cap] = kPackZero;
    }
    __syncthreads();
    const int total = tot;   // uniform
    if (total > Sh::cap || sd.pmax2 < 0.0f) return false;
    if (total == 0) return true;
    // the origin: the first atom at or after the middle home cell
    const int hm = (B.nh[0] / 2 + 1) + B.hd[0] * ((B.nh[1] / 2 + 1) + B.hd[1] * (B.nh[2] / 2 + 1));
    const int im = min(L.hoff[hm], total - 1), ho = L.owner[im];
    const int po = sgpr(L.hstart[ho] + (im - L.hoff[ho]));
    const Rec ro = A.rec[po];
    const double ox = ro.x, oy = ro.y, oz = ro.z;
    // pack(t') of an atom = its cell shift's pack - its winding's + tb (no field
    // leaves its 10 bits while every winding is within +-128, or as
    // tile_windings_near finds)
    const uint32_t to = (L.hshift[ho] & ~kHomeCell) - ro.w, tb = kPackZero - to;
    // halo atoms: all loads of a thread in flight together
    int pg[Sh::unroll];
    uint32_t hs[Sh::unroll];
#pragma unroll
    for (int u = 0; u < Sh::unroll; ++u) {
        const int idx = tid + u * BT;
        pg[u] = po;
        hs[u] = kPackZero;
        if (idx < total) {
            const int h = L.owner[idx];
            pg[u] = L.hstart[h] + (idx - L.hoff[h]);
            hs[u] = L.hshift[h];
        }
    }
    Rec r[Sh::unroll];
#pragma unroll
    for (int u = 0; u < Sh::unroll; ++u)
        if (tid + u * BT < total) r[u] = A.rec[pg[u]];
    // winding fields (biased by 512) within [384, 639]: bits 9 and 8 differ,
    // bits 8 and 7 do not
    constexpr uint32_t kWindMask = (kFieldsLow << 9) | (kFieldsLow << 8) | kWindBig, kWindOk = kFieldsLow << 9;
    bool bad = ((ro.w ^ ((ro.w & ~kWindBig) << 1)) & kWindMask) != kWindOk;
#pragma unroll
    for (int u = 0; u < Sh::unroll; ++u) {
        const int idx = tid + u * BT;
        if (idx < total) {
            const uint32_t w = r[u].w;
            bad |= ((w ^ ((w & ~kWindBig) << 1)) & kWindMask) != kWindOk;
            const uint32_t t = (hs[u] & ~kHomeCell) - w + tb;
            double dx = r[u].x - ox, dy = r[u].y - oy, dz = r[u].z - oz;
            if (t != kPackZero) {
                int32_t tx, ty, tz;
                unpack_wind(t, tx, ty, tz);
                double cx, cy, cz;
                cell_shift(Csh, tx, ty, tz, cx, cy, cz);
                dx += cx;
                dy += cy;
                dz += cz;
            }
            const float fx = (float)dx, fy = (float)dy, fz = (float)dz;
            // an atom clamped into the grid from far outside (non-negative floats order as their bits)
            const float f2 = fx * fx + fy * fy + fz * fz;
            if (!(f2 <= sd.pmax2)) atomicMax(&L.far2, __builtin_bit_cast(int, f2));
            // 4-byte slot entries need every S = t'_j - t'_i within [-1, 1]^3: home
            // atoms with t' = 0 and halo atoms with |t'_k| <= 1
            const uint32_t c = t - 511u * kFieldsLow;   // fields 0, 1, 2 then
            const bool near = (c & ~(3u * kFieldsLow)) == 0 && (c & (c >> 1) & kFieldsLow) == 0;
            if (!((hs[u] & kHomeCell) ? t == kPackZero : near)) L.row8 = 1;
            // the low 2 bits of the fields are the S codes of a 4-byte entry
            const uint32_t code = (t & 3u) | ((t >> 8) & 12u) | ((t >> 16) & 48u);
            L.a[idx] = TAtom{fx, fy, fz,
                             sd.nat <= kNarrowMaxAtoms ? (int32_t)((uint32_t)r[u].j | code << 26) : r[u].j};
            L.t[idx] = t;
        }
    }
    if (tid < T.n) {   // centre of run tid, from the brick's origin
        int ix, iy, iz, w;
        tile_run(B, T, tid, ix, iy, iz, w);
        const double f0 = (B.b0[0] - 1 + ix + 0.5 * w) / sd.n[0], f1 = (B.b0[1] - 0.5 + iy) / sd.n[1],
                     f2 = (B.b0[2] - 0.5 + iz) / sd.n[2];
        int32_t tx, ty, tz;
        unpack_wind(to + kPackZero, tx, ty, tz);
        for (int k = 0; k < 3; ++k)
            L.ctr[tid][k] = (float)(((Csh[3 * k] * (f0 - tx) + Csh[3 * k + 1] * (f1 - ty)) +
                                     Csh[3 * k + 2] * (f2 - tz)) - (k == 0 ? ox : k == 1 ? oy : oz));
    }
    if (bad) L.flag = 1;
    __syncthreads();
    return L.flag == 0 || tile_windings_near(A, L, total);
}

// The 64-bit test of home atom hl (LDS index) against candidate li: -1 for
// a hit, 1 otherwise.  A candidate more than one cell along x from the home
// atom (a run of two cells shares its list) is none of the reference's.
// Called for the few values the filter cannot decide, out of line and one
// component at a time: the registers it uses are lost to the pass around it.
template <int BT>
__device__ __attribute__((noinline)) float tile_exact(const Rec *rec, const TileLDS<BT> *L, const double *Csh, double rc2,
                                                      int hd0, int hl, int li)
{
    if (li == BrickShape<BT>::cap) return 1.0f;
    const int oc = L->owner[li], oh = L->owner[hl];
    if ((unsigned)(oc % hd0 - oh % hd0 + 1) > 2u) return 1.0f;
    const double *c = &rec[L->hstart[oc] + (li - L->hoff[oc])].x, *h = &rec[L->hstart[oh] + (hl - L->hoff[oh])].x;
    const uint32_t t = L->t[li] - L->t[hl] + kPackZero;   // pack(S)
    double r2 = 0.0;
#pragma unroll 1
    for (int k = 0; k < 3; ++k) {
        // R = xj - xi + C' * S ; r^2 = dot(R, R)  (gpu_kernels.jl:89-92)
        int32_t Sx, Sy, Sz;
        unpack_wind(t, Sx, Sy, Sz);
        const double *C = Csh + 3 * k;
        const double R = (c[k] - h[k]) + ((C[0] * (double)Sx + C[1] * (double)Sy) + C[2] * (double)Sz);
        r2 = k == 0 ? R * R : r2 + R * R;
    }
    return r2 < rc2 ? -1.0f : 1.0f;
}

// What a pass over a run's candidates reads: NCH chunks, one candidate per
// lane (b*: position from the run's centre, bq: half its square, ent: low word
// of the slot entry, ct: the high word for t'_i = 0, li: LDS index).
struct TileCands {
    float bx[kTileChunks], by[kTileChunks], bz[kTileChunks], bq[kTileChunks];
    int ent[kTileChunks], li[kTileChunks];
    uint32_t ct[kTileChunks];
};

// ... and its home atoms, one per lane: minus the position from the run's
// centre, (|p|^2 - rc^2) / 2, the buffer over the slot row (address and entry
// size), t', the bytes filled of the row, and the entries a chunk may store.
struct TileHomes {
    float nx, ny, nz, ai;
    uint64_t row;
    uint32_t t;
    int32_t fill, left;
};

__device__ __forceinline__ float readlane_f32(float v, int l)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

__device__ __forceinline__ float wave_max_f32(float x)   // non-negative floats order as their bits
{
    return __builtin_bit_cast(float, wave_max_pos(__builtin_bit_cast(int, x)));
}

// Home atoms that lie far from their cell's centre (along an open axis; above
// kFarHome rc^2 / 2 for half the square of their distance) are taken from the
// first of them instead, which keeps the filter's error at their own extent's
// (whole builds, us: a sheet of 200,000 atoms 1,000 A away from its cell 245 from
// the cell's centre, 117 from an atom; 200 systems of 500 to 2,000 atoms 300
// cells away 1,326 and 199).
constexpr float kFarHome = 32.0f;
__device__ __forceinline__ void home_centre(const TAtom &h, float &ox, float &oy, float &oz)
{
    ox = readlane_f32(h.x, 0);
    oy = readlane_f32(h.y, 0);
    oz = readlane_f32(h.z, 0);
}

// The home atoms' side of the tests from the centre o; half the squares of
// their distances from it.
__device__ __forceinline__ float tile_home(TileHomes &H, const TAtom &h, float ox, float oy, float oz)
{
    H.nx = ox - h.x;
    H.ny = oy - h.y;
    H.nz = oz - h.z;
    return 0.5f * __builtin_fmaf(H.nz, H.nz, __builtin_fmaf(H.ny, H.ny, H.nx * H.nx));
}

// Slot entries of a pass: 4 or 8 bytes.
enum { kEntry4, kEntry8 };

// Home atoms a0 .. a1 - 1 against NCH chunks.  D = bq + ai - p_i . p_j is half
// of r^2 - rc^2.  G: the chunk that holds the home atoms' own candidates
// (kpass + a; -1: none does).  E: the 64-bit test of home atom a against the
// lane's candidate of chunk g, and whether stores stop at H.left entries.
template <int NCH, int MODE, int G, typename Env>
__device__ __forceinline__ void tile_rows(const Env &E, float tol, const TileCands &C, int a0, int a1, int kpass,
                                          TileHomes &H)
{
    for (int a = a0; a < a1; ++a) {
        const float sx = readlane_f32(H.nx, a), sy = readlane_f32(H.ny, a), sz = readlane_f32(H.nz, a),
                    sa = readlane_f32(H.ai, a);
        float D[NCH];
        float mn = kFar32;
#pragma unroll
        for (int g = 0; g < NCH; ++g)
            D[g] = __builtin_fmaf(sz, C.bz[g], __builtin_fmaf(sy, C.by[g], __builtin_fmaf(sx, C.bx[g], C.bq[g] + sa)));
#pragma unroll
        for (int g = 0; g + 1 < NCH; g += 2)
            mn = __builtin_fminf(__builtin_fminf(mn, __builtin_fabsf(D[g])), __builtin_fabsf(D[g + 1]));
        if (NCH & 1) mn = __builtin_fminf(mn, __builtin_fabsf(D[NCH - 1]));
        // a value within the filter's error of zero: the 64-bit test
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(mn < tol) != 0, 0)) {
#pragma unroll
            for (int g = 0; g < NCH; ++g)
                if (__builtin_amdgcn_ballot_w64(__builtin_fabsf(D[g]) < tol) != 0) D[g] = E.template exact<MODE>(a, g);
        }
        int32_t so = __builtin_amdgcn_readlane(H.fill, a);
        const v4u rs = {(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)H.row, a),
                        (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(H.row >> 32), a),
                        Env::kLimit ? (uint32_t)__builtin_amdgcn_readlane(H.left, a) : (uint32_t)kWave,
                        (uint32_t)kRawBufferWord3};
        const uint32_t dt = MODE == kEntry8 ? (uint32_t)__builtin_amdgcn_readlane((int)H.t, a) : 0u;
#pragma unroll
        for (int g = 0; g < NCH; ++g) {
            uint64_t m = __builtin_amdgcn_ballot_w64(D[g] < 0.0f);
            if (g == G) m &= ~(1ull << ((kpass + a) & (kWave - 1)));   // j == i, s == 0 is no pair
            emit_chunk<MODE == kEntry4>(rs, m, so, (uint32_t)C.ent[g], MODE == kEntry4 ? 0u : C.ct[g] - dt);
        }
        H.fill = write_lane(so, a, H.fill);
    }
}

// The run's nh home atoms against NCH chunks: their own candidates are
// consecutive, in one chunk or across two.
template <int NCH, int MODE, typename Env>
__device__ __forceinline__ void tile_pass(const Env &E, float tol, const TileCands &C, int nh, int kpass, TileHomes &H)
{
    int a = 0;
    while (a < nh) {
        const int g = (kpass + a) >> 6;   // negative: before this pass
        const int e = g >= NCH ? nh : min(nh, g < 0 ? -kpass : (g + 1) * kWave - kpass);
        if (NCH > 0 && g == 0) tile_rows<NCH, MODE, 0>(E, tol, C, a, e, kpass, H);
        else if (NCH > 1 && g == 1) tile_rows<NCH, MODE, 1>(E, tol, C, a, e, kpass, H);
        else if (NCH > 2 && g == 2) tile_rows<NCH, MODE, 2>(E, tol, C, a, e, kpass, H);
        else if (NCH > 3 && g == 3) tile_rows<NCH, MODE, 3>(E, tol, C, a, e, kpass, H);
        else tile_rows<NCH, MODE, -1>(E, tol, C, a, e, kpass, H);
        a = e;
    }
}

// tile_kernel's side of tile_rows: hb, hd0 as in tile_exact; a row's stores
// are not limited (kSlotSlack).
template <int BT>
struct TileEnv {
    static constexpr bool kLimit = false;
    const Rec *rec;
    const TileLDS<BT> &L;
    const double *Csh;
    double rc2;
    int hd0, hb;
    const TileCands &C;
    template <int MODE>
    __device__ __forceinline__ float exact(int a, int g) const
    {
        return tile_exact<BT>(rec, &L, Csh, rc2, hd0, hb + a, C.li[g]);
    }
};

// Brick pass of the count (no 16-byte entries): the distance tests run
// on 32-bit positions, exact to a known bound (filter_bounds), and every value
// within that bound of the cutoff is decided again by the 64-bit test, so the
// pairs are those of the 64-bit kernel.
//
// Bound by instruction issue: a home atom against four chunks is 39 vector and
// 30 scalar instructions; at 1M atoms the vector unit issues for 73% of the
// time (63.2 instructions per home atom, 47 scalar; 73.9 and 64 in the 64-bit
// kernel, whose 32-byte atoms also held a CU to four bricks, now five).  The
// tests as matrix instructions (4 x 4 x 1 in 32 bits, 16 blocks: four home atoms
// by 64 candidates) took 12 cycles of the wave's SIMD each, more than the
// vector instructions they replaced: 157 against 151 us.  Kernel times before
// and after (MI355X): 96-atom crystal 66 / 12 us, 1k atoms 17.2 / 7.8, 100k 33 /
// 28, 1M 193 / 154, 1M FCC slab 368 / 231 (there most bricks of atoms outside
// the cell wrote 8-byte rows; windings now count from the brick's own).
//
// A run of two home cells shares one candidate list, their nine rows of four
// cells: a pair of cells two apart along x that a home cell's own 27 cells
// would not hold is at least one cell height (>= rc) apart, so it is no hit
// beyond the filter's error, and within it tile_exact leaves it out.
template <int BT>
__global__ __launch_bounds__(BT) __attribute__((amdgpu_waves_per_eu(5))) void tile_kernel(
    const SysDev *__restrict__ sys, const int32_t *__restrict__ sys_cell_base, const int32_t *__restrict__ sys_brick_base,
    int nsys, int copies, int32_t M, int64_t nat, const int32_t *__restrict__ cell_start,
    const Rec *__restrict__ rec, const int32_t *__restrict__ wbig, int32_t *__restrict__ pair_count,
    void *__restrict__ slots, int64_t off8, int32_t row4, int32_t cap, Status *__restrict__ status)
{
    __shared__ TileLDS<BT> L;
    __shared__ double Csh[9];
    const PairsArgs A{sys, sys_cell_base, nsys, M, nat, cell_start, rec, wbig};
    Brick B;
    const int copy = copies == 1 ? 0 : (int)(blockIdx.x % (unsigned)copies);
    brick_locate(A, sys_brick_base, copies == 1 ? (int)blockIdx.x : (int)(blockIdx.x / (unsigned)copies),
                 BrickShape<BT>::halo, B);
    const TileRuns T = tile_runs(B);
    if (threadIdx.x < 9) Csh[threadIdx.x] = B.sd->C[threadIdx.x];   // visible after tile_load's first barrier
    const bool lds = B.fast && tile_load(A, B, T, L, Csh);
    const int lane = lane_id();
    const int wv = sgpr((int)(threadIdx.x >> 6));
    if (!lds) {
        const SlotArgs O{reinterpret_cast<char *>(slots) + off8, cap, status};
        count_cells<false>(A, B, pair_count, O, copy + copies * wv, copies * BrickShape<BT>::waves);
        return;
    }
    const SysDev &sd = *B.sd;
    const bool narrow = sgpr(L.row8) == 0;   // the brick writes 4-byte slot entries
    const int far2 = sgpr(L.far2);
    // L.a[].j holds j | S code << 26 whenever every j fits in 26 bits
    const uint32_t hjmask = sd.nat <= kNarrowMaxAtoms ? (uint32_t)(kNarrowMaxAtoms - 1) : 0xffffffffu;
    const uint32_t jmask = narrow ? 0xffffffffu : hjmask;   // entry low word: j | code << 26, or j
    // halo cell of row lane < 9, (dz, dy) = (lane / 3 - 1, lane % 3 - 1), from the run's own
    const int roff = lane < 9 ? B.hd[0] * ((lane % 3 - 1) + B.hd[1] * (lane / 3 - 1)) : 0;
    uint8_t *fl = reinterpret_cast<uint8_t *>(L.rowflag[wv]);
    // items: the home atoms of a run in 2^split parts, those of the brick
    // dealt to its copies, then to their waves
    const int split = sd.split, items = T.n << split;
    for (int it = copy + copies * wv; it < items; it = copy + copies * take_next(&L.next_item)) {
        const int rn = it >> split, part = it & ((1 << split) - 1);
        int ix, iy, iz, w;
        tile_run(B, T, rn, ix, iy, iz, w);
        const int hc = ix + B.hd[0] * ((iy + 1) + B.hd[1] * (iz + 1));   // halo cell before the run's first
        const int h0 = sgpr(L.hoff[hc + 1]), nha = sgpr(L.hoff[hc + 1 + w]) - h0;
        if (nha <= 0) continue;
        float ox = L.ctr[rn][0], oy = L.ctr[rn][1], oz = L.ctr[rn][2];
        // candidates: nine rows of w + 2 cells, each contiguous in LDS
        const int rst = L.hoff[hc + roff];
        const int len = lane < 9 ? L.hoff[hc + roff + w + 2] - rst : 0;
        const int incl = row16_incl_scan(len);
        const int rex = incl - len;
        const int total = __builtin_amdgcn_readlane(incl, 8);
        // row 4 is (dz, dy) = (0, 0); the run starts at its second cell
        const int self0 = __builtin_amdgcn_readlane(rex, 4) + (h0 - __builtin_amdgcn_readlane(rst, 4));
        // LDS index less candidate index of the non-empty rows, in row order
        const uint64_t bne = __builtin_amdgcn_ballot_w64(len > 0);
        const int rq = (int)mbcnt64(bne);
        if (len > 0) L.rowdl[wv][rq] = rst - rex;
        const int r1 = nha * (part + 1) >> split;
        for (int hg = nha * part >> split; hg < r1; hg += kWave) {
            const int nh = sgpr(min(kWave, r1 - hg));
            const int hb = h0 + hg;          // LDS index of home atom hg (uniform)
            const int hl = hb + (lane < nh ? lane : 0);
            const TAtom h = L.a[hl];
            const int32_t hj_l = (int32_t)((uint32_t)h.j & hjmask);
            TileHomes H;
            float hq = tile_home(H, h, ox, oy, oz);
            // atoms further out than the system's bounds assume: the brick's own
            float tol = sd.tol;
            if (__builtin_amdgcn_ballot_w64(!(hq <= sd.h2half)) != 0 || far2 != 0) {
                float hm = readlane_f32(wave_max_f32(hq), kWave - 1);
                if (hm > kFarHome * sd.rc2half) {
                    home_centre(h, ox, oy, oz);
                    hq = tile_home(H, h, ox, oy, oz);
                    hm = readlane_f32(wave_max_f32(hq), kWave - 1);
                }
                tol = far_tol(sd, __builtin_sqrtf(2.0f * hm), __builtin_bit_cast(float, far2));
            }
            H.ai = hq - sd.rc2half;
            H.row = (reinterpret_cast<uint64_t>(slots) + (narrow ? 0 : off8) +
                     (uint64_t)slot_row(sd.atom_base + hj_l, narrow ? row4 : 8 * cap)) |
                    (uint64_t)(narrow ? 4 : 8) << 48;
            H.t = L.t[hl];
            H.fill = 0;
            for (int k0 = 0; k0 < total; k0 += kTileCands) {
                const int nch = sgpr(min(kTileChunks, (total - k0 + kWave - 1) / kWave));
                // marks where a non-empty row other than the first starts (see row_map)
                L.rowflag[wv][lane] = 0u;
                const int p = rex - k0;
                if (len > 0 && rq > 0 && p > 0 && p < kTileCands) fl[p] = 1;
                int acc = k0 == 0 ? 0 : (int)__popcll(bne & __builtin_amdgcn_ballot_w64(rq > 0) & __builtin_amdgcn_ballot_w64(p <= 0));
                TileCands C;
#pragma unroll
                for (int g = 0; g < kTileChunks; ++g) {
                    const uint64_t bm = __builtin_amdgcn_ballot_w64(fl[g * kWave + lane] != 0);
                    const int q = acc + (int)(bm & 1u) + (int)mbcnt64(bm >> 1);
                    acc += (int)__popcll(bm);
                    const int k = k0 + g * kWave + lane;
                    C.li[g] = k < total ? k + L.rowdl[wv][q] : BrickShape<BT>::cap;   // else the far sentinel
                    const TAtom c = L.a[C.li[g]];
                    C.bx[g] = c.x - ox;
                    C.by[g] = c.y - oy;
                    C.bz[g] = c.z - oz;
                    C.bq[g] = 0.5f * __builtin_fmaf(C.bz[g], C.bz[g], __builtin_fmaf(C.by[g], C.by[g], C.bx[g] * C.bx[g]));
                    C.ent[g] = (int)((uint32_t)c.j & jmask);
                    if (!narrow) C.ct[g] = L.t[C.li[g]] + kPackZero;
                }
                const int kp = self0 + hg - k0;   // home atom hg + a is candidate kp + a of this pass
const TileEnv<BT> E{rec, L, Csh, sd.rc2, B.hd[0], hb, C};
                if (narrow) {
                    if (nch == 4) tile_pass<4, kEntry4>(E, tol, C, nh, kp, H);
                    else if (nch == 3) tile_pass<3, kEntry4>(E, tol, C, nh, kp, H);
                    else tile_pass<2, kEntry4>(E, tol, C, nh, kp, H);
                } else {
                    if (nch == 4) tile_pass<4, kEntry8>(E, tol, C, nh, kp, H);
                    else if (nch == 3) tile_pass<3, kEntry8>(E, tol, C, nh, kp, H);
                    else tile_pass<2, kEntry8>(E, tol, C, nh, kp, H);
                }
            }
            if (lane < nh) pair_count[sd.atom_base + hj_l] = narrow ? H.fill >> 2 : (H.fill >> 3) | kRow8Bit;
        }
    }
}

// ---------------------------------------------------------------------------
// Fused build of small systems
// ---------------------------------------------------------------------------
//
// One workgroup of kSmallThreads threads per work item: a unit of
// consecutive systems (at most kUnitAtoms atoms, kUnitCells cells and
// kUnitSystems systems) or one of its parts, all of it in LDS: the cell and
// winding of every atom, a stable counting sort by cell (ties in ascending
// original index, Julia's stable sortperm), the cell-list outputs (written
// by part 0), and the neighbour count and slot row of every home atom of
// the part's count work items (items part, part + parts, ..., each a group
// of home atoms of one cell), through tile_kernel's 32-bit tests and emission;
// the waves take those items from a workgroup counter.  A home cell's
// candidates are its (2 nxyz + 1)^3 neighbour cells in the reference order
// (dz, dy, dx outer to inner, gpu_kernels.jl:69-71), each a segment of the
// sorted atoms with its cell shift, taken 64 segments at a time.

// Bound by instruction issue and, in what comes before the tests, by latency:
// in a batch of 4,096 systems of 8 to 2,048 atoms (1.6M atoms) the vector unit
// issues for 70% of the time, 68M of its 126M instructions in the tests, 29M
// in the items' segments, 20M in loading candidates, 10M in the sort.  Two
// workgroups share a CU (79 KB of LDS each), so that one counts while the other
// sorts.  Before, with 32-byte atoms, 64-bit tests and one workgroup of 1,024
// threads per CU, against now: that batch 485 / 335 us, 128 systems of 8 to 400
// atoms 58 / 25.
//
// Count work items: a group of at most sys_group home atoms of one cell.
// The group size of a system aims at item_tests distance tests (chunks of 64
// candidates) per item, at least kMinGroup atoms: a cell whose candidates run
// to thousands (a small periodic cell, its own 26 images) is shared by
// several waves instead of holding one wave for all of it.
constexpr int kMinGroup = 4;
constexpr int kUnitItems = kUnitAtoms / kMinGroup + kUnitCells;   // items of one unit at most
constexpr int kThreadCells = kUnitCells / kSmallThreads;          // cells per thread in the scans

struct SmallSort {                 // LDS of the sort
    int16_t key[kUnitAtoms];       // unit cell of each atom
    int16_t grp[kUnitAtoms];       // atoms grouped by cell, in arrival order
    int32_t fill[kUnitCells];      // per cell: atoms, then arrivals
    uint32_t wk[kUnitAtoms];       // packed winding of each atom
    uint8_t sy[kUnitAtoms];        // unit system of each atom
};
struct __attribute__((aligned(16))) SegShift {
    float x, y, z;                 // cell shift of a segment, less the home group's centre
    uint32_t s;                    // the shift packed, or in a 4-byte system its S code << 26
};
struct SmallRows {                 // LDS of one wave in the count
    SegShift sv[kWave];            // each non-empty segment
    int32_t dl[kWave];             // LDS offset less candidate prefix of each non-empty segment
    uint32_t flag[kTileCands / 4]; // one byte per candidate of a pass: a segment starts there
};
struct SmallCount {                // LDS of the count
    uint32_t cell_info[kUnitCells];   // per unit cell: system | (c1 - 1) << 8 | (c2 - 1) << 16 | (c3 - 1) << 24
    int16_t item0[kUnitCells + 1];    // first count work item of each unit cell
    int16_t item_cell[kUnitItems];    // unit cell of each count work item
    SmallRows r[kSmallThreads / kWave];
};
struct SmallLDS {
    TAtom a[kUnitAtoms + 1];       // sorted atoms, wrapped, from the system's centre, and j; far sentinel last
    uint32_t w[kUnitAtoms + 1];    // their packed windings
    int16_t cs[kUnitCells + 1];    // first sorted atom of each unit cell
    int16_t sys_cell0[kUnitSystems + 1];
    int16_t sys_atom0[kUnitSystems + 1];
    int32_t next_item;                // the next count work item a wave takes
    uint32_t sys_geo[kUnitSystems];   // grid and periodicity: n0 | n1 << 9 | n2 << 18 | pbc << 27
    uint8_t sys_reach[kUnitSystems];  // nxyz: x | y << 2 | z << 4
    uint8_t sys_group[kUnitSystems];  // home atoms per count work item
    uint8_t sys_row8[kUnitSystems];   // 8-byte slot rows: some winding, or reach beyond one cell
    uint8_t sys_far[kUnitSystems];    // windings too far apart for packed differences
    union {
        SmallSort s;
        SmallCount c;
    } u;
};
static_assert(sizeof(SmallLDS) <= 79 * 1024, "two workgroups share a compute unit's LDS");

// The system of cell or atom v of a unit: the last one that starts at or before v.
__device__ __forceinline__ int unit_sys(const int16_t *first, int n, int v)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first[mid] <= v) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

struct SmallArgs {
    const double *__restrict__ X;
    const SysDev *__restrict__ sys;
    const int64_t *__restrict__ sys_atom_base;
    const int32_t *__restrict__ sys_cell_base;
    const int32_t *__restrict__ units;
    const int32_t *__restrict__ order;
    int32_t *__restrict__ atom_sys;
    Rec *__restrict__ rec;
    void *__restrict__ perm_out;
    void *__restrict__ cell_id_out;
    void *__restrict__ cell_offsets_out;
    int32_t *__restrict__ pair_count;
    void *__restrict__ slots;
    int64_t off8;
    int32_t row4, cap, item_tests;
    Status *__restrict__ status;
};

// wrap_and_shift (cell_list.jl:105-120) of a neighbour cell index a within a
// few cells of [1, n] on a periodic axis (the floor of (a - 1/2) / n by a
// reciprocal is exact for |a| < 1024); on an open axis only in-bounds
// indices reach here.
__device__ __forceinline__ void wrap_small(int32_t a, int32_t n, bool p, int32_t &w, int32_t &s)
{
    if (!p) {
        w = a;
        s = 0;
        return;
    }
    const int32_t q = (int32_t)floorf(((float)a - 0.5f) * __builtin_amdgcn_rcpf((float)n));
    w = a - q * n;
    s = q;
}

// pack_wind of components known to fit.
__device__ __forceinline__ uint32_t pack_fields(int32_t x, int32_t y, int32_t z)
{
    return kPackZero + (uint32_t)x + ((uint32_t)y << 10) + ((uint32_t)z << 20);
}

// A system's table entry, read through the scalar cache (nothing writes it
// while the kernel runs).
using SysConst = const __attribute__((address_space(4))) SysDev;
__device__ __forceinline__ SysConst *sys_const(const SysDev *p)
{
    return (SysConst *)(uintptr_t)p;
}

// The 64-bit test of atoms i, j of a system (X: its positions) with packed cell
// shift S: -1 for a hit, 1 otherwise (out of line, see tile_exact).
__device__ __attribute__((noinline)) float small_exact(const double *X, const SysDev *sd, int i, int j, uint32_t S)
{
    X += 3 * sd->atom_base;
    double r2 = 0.0;
#pragma unroll 1
    for (int k = 0; k < 3; ++k) {
        // R = xj - xi + C' * S ; r^2 = dot(R, R)  (gpu_kernels.jl:89-92)
        int32_t Sx, Sy, Sz;
        unpack_wind(S, Sx, Sy, Sz);
        const double *C = sd->C + 3 * k;
        const double R = (X[3 * j + k] - X[3 * i + k]) + ((C[0] * (double)Sx + C[1] * (double)Sy) + C[2] * (double)Sz);
        r2 = k == 0 ? R * R : r2 + R * R;
    }
    return r2 < sd->rc2 ? -1.0f : 1.0f;
}

// small_kernel's side of tile_rows.
struct SmallEnv {
    static constexpr bool kLimit = true;
    const double *X;
    const SysDev *sd;
    const TAtom *a_;         // home atom 0
    const TileCands &C;
    const TileHomes &H;
    const TAtom *all;

    template <int MODE>
    __device__ __forceinline__ float exact(int a, int g) const
    {
        uint32_t S;
        if constexpr (MODE == kEntry4) {
            const uint32_t c = (uint32_t)C.ent[g] >> 26;   // two bits per component: its low ones
            S = kPackZero - kFieldsLow + (((c + 1) & 3u) | ((c + 4) & 12u) << 8 | ((c + 16) & 48u) << 16);
        } else {
            S = C.ct[g] - (uint32_t)__builtin_amdgcn_readlane((int)H.t, a);
        }
        const float d = small_exact(X, sd, sgpr(a_[a].j), all[C.li[g]].j, S);
        return C.li[g] == kUnitAtoms ? 1.0f : d;
    }
};

// A batch of segments against the home atoms of a system whose windings lie so
// far apart that packed differences could leave their fields: 64-bit tests, S
// taken apart; an S beyond +-511 sends the build to 16-byte entries.  Lane:
// ex, st, sh of a segment; fill of a home atom, returned.  ks: the self
// candidate of home atom 0.
__device__ __forceinline__ int32_t small_far(const SmallArgs &A, const SmallLDS &L, SysConst *sd, int total, int ex, int st,
                                             uint32_t sh, int hb, int nh, int ks, int32_t fill)
{
    const int lane = lane_id();
    const int64_t base = sd->atom_base;
    for (int k0 = 0; k0 < total; k0 += kWave) {
        const int k = k0 + lane;
        int q = 0;   // the last segment that starts at or before candidate k
#pragma unroll
        for (int step = kWave / 2; step >= 1; step >>= 1)
            if (__shfl(ex, q + step, kWave) <= k) q += step;
        const int dl = __shfl(st - ex, q, kWave);
        const uint32_t s = (uint32_t)__shfl((int)sh, q, kWave);
        const int li = k < total ? k + dl : kUnitAtoms;
        const int64_t j = L.a[li].j;
        int32_t sx, sy, sz, wx, wy, wz;
        unpack_wind(s, sx, sy, sz);
        unpack_wind(L.w[li], wx, wy, wz);
        const double cx = A.X[3 * (base + j)], cy = A.X[3 * (base + j) + 1], cz = A.X[3 * (base + j) + 2];
        for (int a = 0; a < nh; ++a) {
            const int64_t i = sgpr(L.a[hb + a].j);
            int32_t ix, iy, iz;
            unpack_wind((uint32_t)sgpr((int)L.w[hb + a]), ix, iy, iz);
            // R = xj - xi + C' * S ; r^2 = dot(R, R)  (gpu_kernels.jl:89-92)
            const int32_t Sx = sx - wx + ix, Sy = sy - wy + iy, Sz = sz - wz + iz;
            double tx, ty, tz;
            cell_shift(sd->C, Sx, Sy, Sz, tx, ty, tz);
            const double Rx = (cx - A.X[3 * (base + i)]) + tx, Ry = (cy - A.X[3 * (base + i) + 1]) + ty,
                         Rz = (cz - A.X[3 * (base + i) + 2]) + tz;
            const double r2 = (Rx * Rx + Ry * Ry) + Rz * Rz;
            const uint64_t m = __builtin_amdgcn_ballot_w64(r2 < sd->rc2 && k < total && k != ks + a);
            const int32_t f = __builtin_amdgcn_readlane(fill, a);
            const int rank = (f >> 3) + (int)mbcnt64(m);
            if ((m >> lane) & 1) {
                const uint32_t spk = pack_wind(Sx, Sy, Sz);
                if (spk & kWindBig) A.status->wide = 1;   // past the row's end too (see emit_hits)
                if (rank < A.cap)
                    reinterpret_cast<uint64_t *>(reinterpret_cast<char *>(A.slots) + A.off8)[slot_row(base + i, A.cap) + rank] =
                        (uint64_t)(uint32_t)j | (uint64_t)spk << 32;
            }
            fill = write_lane(f + 8 * (int)__popcll(m), a, fill);
        }
    }
    return fill;
}

template <typename TI>
__global__ __launch_bounds__(kSmallThreads) void small_kernel(SmallArgs A)
{
    __shared__ SmallLDS L;
    const int tid = (int)threadIdx.x, lane = lane_id(), wv = sgpr(tid >> 6);
    const int u = A.order[2 * blockIdx.x], pinfo = A.order[2 * blockIdx.x + 1];
    const int part = pinfo & 0xffff, parts = pinfo >> 16;   // this workgroup counts items part + parts k
    const bool writer = part == 0;                           // the first part writes the cell list
    const int s0 = A.units[u], ns = A.units[u + 1] - s0;
    const int64_t A0 = A.sys_atom_base[s0];
    const int nat_u = (int)(A.sys_atom_base[s0 + ns] - A0);
    const int32_t C0 = A.sys_cell_base[s0];
    const int M_u = A.sys_cell_base[s0 + ns] - C0;
    for (int k = tid; k <= ns; k += kSmallThreads) {
        L.sys_cell0[k] = (int16_t)(A.sys_cell_base[s0 + k] - C0);
        L.sys_atom0[k] = (int16_t)(A.sys_atom_base[s0 + k] - A0);
        if (k < ns) {
            const SysDev &sd = A.sys[s0 + k];
            L.sys_row8[k] = (sd.nxyz[0] > 1 || sd.nxyz[1] > 1 || sd.nxyz[2] > 1) ? 1 : 0;
            L.sys_far[k] = 0;
            L.sys_geo[k] = (uint32_t)(sd.n[0] | sd.n[1] << 9 | sd.n[2] << 18) | (uint32_t)sd.pbc << 27;
            L.sys_reach[k] = (uint8_t)(sd.nxyz[0] | sd.nxyz[1] << 2 | sd.nxyz[2] << 4);
            // candidates per home atom: the system's mean cell occupancy times its neighbour cells
            const int nseg = (2 * sd.nxyz[0] + 1) * (2 * sd.nxyz[1] + 1) * (2 * sd.nxyz[2] + 1);
            const int chunks = max(1, (int)((nseg * (int64_t)sd.nat / max(sd.M, 1) + kWave - 1) / kWave));
            L.sys_group[k] = (uint8_t)min(kWave, max(kMinGroup, A.item_tests / chunks));
        }
    }
    for (int c = tid; c < M_u; c += kSmallThreads) L.u.s.fill[c] = 0;
    if (tid == 0) {
        L.a[kUnitAtoms] = TAtom{kFar32, 0.0f, 0.0f, 0};
        L.w[kUnitAtoms] = kPackZero;
        L.next_item = kSmallThreads / kWave;   // wave w starts at the part's item w
    }
    __syncthreads();
    // cell and winding of every atom (position_to_cell_index + bin_wrap_and_shift,
    // cell_list.jl:66-74, 141-147), atoms per cell
    bool bad = false, big = false;
    for (int i = tid; i < nat_u; i += kSmallThreads) {
        const int k = unit_sys(L.sys_atom0, ns, i);
        const SysDev &sd = A.sys[s0 + k];
        const int64_t g = A0 + i;
        int32_t c[3], w[3];
        bad |= !cell_and_winding(sd, A.X[3 * g], A.X[3 * g + 1], A.X[3 * g + 2], c, w);
        const int key = L.sys_cell0[k] + (c[0] - 1) + (c[1] - 1) * sd.n[0] + (c[2] - 1) * sd.n[0] * sd.n[1];
        const uint32_t wp = pack_wind(w[0], w[1], w[2]);
        L.u.s.key[i] = (int16_t)key;
        L.u.s.wk[i] = wp;
        L.u.s.sy[i] = (uint8_t)k;
        if (wp != kPackZero) L.sys_row8[k] = 1;
        big |= (wp & kWindBig) != 0;
        atomicAdd(&L.u.s.fill[key], 1);
        if (writer) A.atom_sys[g] = s0 + k;   // the fill kernel's map of atoms to systems
    }
    if (bad) atomicOr(&A.status->bad_position, 1);
    if (big) atomicOr(&A.status->small_fallback, 1);   // the general pipeline redoes the build
    __syncthreads();
    {   // cell starts: exclusive scan of the counts, kThreadCells cells per thread
        const int c0 = kThreadCells * tid;
        int v[kThreadCells], sum = 0;
#pragma unroll
        for (int m = 0; m < kThreadCells; ++m) {
            v[m] = c0 + m < M_u ? L.u.s.fill[c0 + m] : 0;
            sum += v[m];
            if (c0 + m < M_u) L.u.s.fill[c0 + m] = 0;
        }
        int64_t tot;
        int ex = (int)block_excl_scan_n<kSmallThreads>(sum, tot);
#pragma unroll
        for (int m = 0; m < kThreadCells; ++m) {
            if (c0 + m < M_u) L.cs[c0 + m] = (int16_t)ex;
            ex += v[m];
        }
        if (tid == 0) L.cs[M_u] = (int16_t)tot;
    }
    __syncthreads();
    for (int i = tid; i < nat_u; i += kSmallThreads) {   // atoms grouped by cell
        const int key = L.u.s.key[i];
        L.u.s.grp[L.cs[key] + atomicAdd(&L.u.s.fill[key], 1)] = (int16_t)i;
    }
    __syncthreads();
    // each atom's place: its cell's start plus the atoms of its cell with a
    // smaller index (the stable order); the sorted record, perm and cell_id
    for (int i = tid; i < nat_u; i += kSmallThreads) {
        const int key = L.u.s.key[i];
        const int st = L.cs[key], en = L.cs[key + 1];
        int rank = 0;
        for (int t = st; t < en; ++t) rank += L.u.s.grp[t] < i;
        const int p = st + rank;
        const int k = L.u.s.sy[i];
        const int64_t g = A0 + i;
        const SysDev &sd = A.sys[s0 + k];
        const double x = A.X[3 * g], y = A.X[3 * g + 1], z = A.X[3 * g + 2];
        const uint32_t wk = L.u.s.wk[i];
        double ux = x - 0.5 * (sd.C[0] + sd.C[1] + sd.C[2]), uy = y - 0.5 * (sd.C[3] + sd.C[4] + sd.C[5]),
               uz = z - 0.5 * (sd.C[6] + sd.C[7] + sd.C[8]);
        if (wk != kPackZero) {
            int32_t wx, wy, wz;
            unpack_wind(wk, wx, wy, wz);
            double cx, cy, cz;
            cell_shift(sd.C, wx, wy, wz, cx, cy, cz);
            ux -= cx;
            uy -= cy;
            uz -= cz;
        }
        const uint32_t w0 = L.u.s.wk[L.sys_atom0[k]];
        if (wk != w0) {
            // every S = s - w_j + w_i packs while the windings are within 252 of the first atom's
            int32_t wx, wy, wz, vx, vy, vz;
            unpack_wind(wk, wx, wy, wz);
            unpack_wind(w0, vx, vy, vz);
            if ((unsigned)(wx - vx + 252) > 504u || (unsigned)(wy - vy + 252) > 504u || (unsigned)(wz - vz + 252) > 504u)
                L.sys_far[k] = 1;
        }
        const int32_t jl = i - L.sys_atom0[k];
        L.a[p] = TAtom{(float)ux, (float)uy, (float)uz, jl};
        L.w[p] = wk;
        if (writer) {
            Rec r;
            r.x = x;
            r.y = y;
            r.z = z;
            r.j = jl;
            r.w = wk;
            A.rec[A0 + p] = r;
            store_ti<TI>(A.perm_out, A0 + p, (int64_t)jl + 1);
            store_ti<TI>(A.cell_id_out, A0 + p, (int64_t)(key - L.sys_cell0[k]) + 1);
        }
    }
    __syncthreads();   // the sorted atoms are complete; the sort's LDS now holds the count's
    // cell offsets: per system, 1-based, its cells then a trailing entry;
    // the system and the grid coordinates of every cell for the count
    for (int c = tid; c < M_u; c += kSmallThreads) {
        const int k = unit_sys(L.sys_cell0, ns, c);
        const int lc = c - L.sys_cell0[k], n0 = (int)(L.sys_geo[k] & 511u), n1 = (int)((L.sys_geo[k] >> 9) & 511u);
        L.u.c.cell_info[c] = (uint32_t)k | (uint32_t)(lc % n0) << 8 | (uint32_t)((lc / n0) % n1) << 16 |
                             (uint32_t)(lc / (n0 * n1)) << 24;
        const int64_t gc = (int64_t)C0 + c + s0 + k;
        if (writer) {
            store_ti<TI>(A.cell_offsets_out, gc, (int64_t)(L.cs[c] - L.sys_atom0[k]) + 1);
            if (c == L.sys_cell0[k + 1] - 1)
                store_ti<TI>(A.cell_offsets_out, gc + 1, (int64_t)(L.sys_atom0[k + 1] - L.sys_atom0[k]) + 1);
        }
    }
    __syncthreads();
    {   // count work items, numbered in cell order: the cells' item counts, scanned
        const int c0 = kThreadCells * tid;
        int v[kThreadCells], sum = 0;
#pragma unroll
        for (int m = 0; m < kThreadCells; ++m) {
            v[m] = 0;
            if (c0 + m < M_u) {
                const int g = L.sys_group[L.u.c.cell_info[c0 + m] & 255u];
                v[m] = (L.cs[c0 + m + 1] - L.cs[c0 + m] + g - 1) / g;
            }
            sum += v[m];
        }
        int64_t tot;
        int ex = (int)block_excl_scan_n<kSmallThreads>(sum, tot);
#pragma unroll
        for (int m = 0; m < kThreadCells; ++m) {
            if (c0 + m < M_u) L.u.c.item0[c0 + m] = (int16_t)ex;
            for (int t = 0; t < v[m]; ++t) L.u.c.item_cell[ex + t] = (int16_t)(c0 + m);
            ex += v[m];
        }
        if (tid == 0) L.u.c.item0[M_u] = (int16_t)tot;
    }
    __syncthreads();   // the items are numbered
    const int nitems_u = L.u.c.item0[M_u];
    SmallRows &Rw = L.u.c.r[wv];
    uint8_t *fl = reinterpret_cast<uint8_t *>(Rw.flag);
    // (dx, dy, dz) of segment `lane` where the reach is one cell on every axis
    const int ndz = lane / 9 - 1, ndy = lane / 3 - 3 * (lane / 9) - 1, ndx = lane - 3 * (lane / 3) - 1;
    for (int it = part + parts * wv; it < nitems_u; it = part + parts * take_next(&L.next_item)) {
        const int hc = sgpr(L.u.c.item_cell[it]);
        const int ig = it - sgpr(L.u.c.item0[hc]);   // the item's group of home atoms in its cell
        const int h0 = sgpr(L.cs[hc]), nha_c = sgpr(L.cs[hc + 1]) - h0;
        const uint32_t info = (uint32_t)sgpr((int)L.u.c.cell_info[hc]);
        const int k = (int)(info & 255u);
        const int grp = sgpr(L.sys_group[k]);
        const int hg0 = ig * grp, nha = min(nha_c, hg0 + grp);   // home atoms [hg0, nha) of the cell
        const SysConst *sd = sys_const(A.sys + s0 + k);
        const int cb = sgpr(L.sys_cell0[k]);
        const uint32_t geo = (uint32_t)sgpr((int)L.sys_geo[k]), rch = (uint32_t)sgpr((int)L.sys_reach[k]);
        const int n0 = (int)(geo & 511u), n1 = (int)((geo >> 9) & 511u), n2 = (int)((geo >> 18) & 511u);
        const bool p0 = (geo >> 27 & 1) != 0, p1 = (geo >> 28 & 1) != 0, p2 = (geo >> 29 & 1) != 0;
        const int nx0 = (int)(rch & 3u), nx1 = (int)((rch >> 2) & 3u), nx2 = (int)(rch >> 4);
        const int ci0 = (int)((info >> 8) & 255u) + 1, ci1 = (int)((info >> 16) & 255u) + 1, ci2 = (int)(info >> 24) + 1;
        const int sxn = 2 * nx0 + 1, syn = 2 * nx1 + 1;
        const int nseg = sxn * syn * (2 * nx2 + 1);
        const int center = (nx2 * syn + nx1) * sxn + nx0;   // (dx, dy, dz) = 0: the home cell, zero shift
        const bool row8 = sgpr(L.sys_row8[k]) != 0, far = sgpr(L.sys_far[k]) != 0;
        const bool near = rch == 0x15u;   // a reach of one cell on every axis
        // the home cell's centre, from the system's
        const auto &C32 = sd->C32;
        const float f0 = ((float)ci0 - 0.5f) * __builtin_amdgcn_rcpf((float)n0) - 0.5f,
                    f1 = ((float)ci1 - 0.5f) * __builtin_amdgcn_rcpf((float)n1) - 0.5f,
                    f2 = ((float)ci2 - 0.5f) * __builtin_amdgcn_rcpf((float)n2) - 0.5f;
        float ox = C32[0] * f0 + C32[1] * f1 + C32[2] * f2, oy = C32[3] * f0 + C32[4] * f1 + C32[5] * f2,
              oz = C32[6] * f0 + C32[7] * f1 + C32[8] * f2;
        for (int hg = hg0; hg < nha; hg += kWave) {
            const int nh = sgpr(min(kWave, nha - hg));
            const int hb = h0 + hg;
            const int hl = hb + (lane < nh ? lane : 0);
            const TAtom h = L.a[hl];
            TileHomes H;
            float hq = tile_home(H, h, ox, oy, oz);
            // the filter's error bound (small_bounds); beyond any sane scale, 64-bit tests for all
            float hm = readlane_f32(wave_max_f32(hq), kWave - 1), so = 0.0f;
            if (hm > kFarHome * sd->rc2half) {
                home_centre(h, ox, oy, oz);
                hq = tile_home(H, h, ox, oy, oz);
                hm = readlane_f32(wave_max_f32(hq), kWave - 1);
                so = __builtin_sqrtf(2.0f * sd->rc2half * (ox * ox + oy * oy + oz * oz));
            }
            const float tol = hm + so < 1.0e30f ? __builtin_fmaf(so, kSmallTolFar, __builtin_fmaf(hm, kSmallTol, sd->small_tol))
                                                : kFar32 * kFar32;
            H.ai = hq - sd->rc2half;
            const int64_t ha = sd->atom_base + h.j;
            H.row = (reinterpret_cast<uint64_t>(A.slots) + (row8 ? A.off8 : 0) +
                     (uint64_t)slot_row(ha, row8 ? 8 * A.cap : A.row4)) |
                    (uint64_t)(row8 ? 8 : 4) << 48;
            H.t = 2 * kPackZero - L.w[hl];   // t'_i = -w_i
            H.fill = 0;
            for (int sb = 0; sb < nseg; sb += kWave) {
                // lane: neighbour cell sb + lane in the reference order, its
                // sorted atoms and cell shift (_is_cell_in_bounds,
                // _get_neighbor_cell, gpu_kernels.jl:20-47)
                const int gs = sb + lane;
                int st = 0, len = 0;
                SegShift v;
                if (gs < nseg) {
                    int dx = ndx, dy = ndy, dz = ndz;
                    if (!near) {
                        // quotients of small integers by float reciprocals: exact, as every
                        // numerator is within a few hundred of zero and a half away from a
                        // multiple of the divisor
                        const int t2 = (int)(((float)gs + 0.5f) * __builtin_amdgcn_rcpf((float)sxn));
                        const int t3 = (int)(((float)t2 + 0.5f) * __builtin_amdgcn_rcpf((float)syn));
                        dx = gs - t2 * sxn - nx0;
                        dy = t2 - t3 * syn - nx1;
                        dz = t3 - nx2;
                    }
                    const int a0 = ci0 + dx, a1 = ci1 + dy, a2 = ci2 + dz;
                    if ((p0 || (unsigned)(a0 - 1) < (unsigned)n0) && (p1 || (unsigned)(a1 - 1) < (unsigned)n1) &&
                        (p2 || (unsigned)(a2 - 1) < (unsigned)n2)) {
                        int32_t c0, c1, c2, s0x, s0y, s0z;
                        if (near) {   // in bounds, or periodic: at most one wrap
                            wrap_near(a0, n0, c0, s0x);
                            wrap_near(a1, n1, c1, s0y);
                            wrap_near(a2, n2, c2, s0z);
                        } else {
                            wrap_small(a0, n0, p0, c0, s0x);
                            wrap_small(a1, n1, p1, c1, s0y);
                            wrap_small(a2, n2, p2, c2, s0z);
                        }
                        const int uc = cb + (c0 - 1) + ((c1 - 1) + (c2 - 1) * n1) * n0;
                        st = L.cs[uc];
                        len = L.cs[uc + 1] - st;
                        // a 4-byte system: the S code of every atom of the segment (w = 0)
                        v.s = row8 ? pack_fields(s0x, s0y, s0z)
                                   : (uint32_t)((s0x & 3) | (s0y & 3) << 2 | (s0z & 3) << 4) << 26;
                        const float fx = (float)s0x, fy = (float)s0y, fz = (float)s0z;
                        v.x = __builtin_fmaf(C32[0], fx, __builtin_fmaf(C32[1], fy, __builtin_fmaf(C32[2], fz, -ox)));
                        v.y = __builtin_fmaf(C32[3], fx, __builtin_fmaf(C32[4], fy, __builtin_fmaf(C32[5], fz, -oy)));
                        v.z = __builtin_fmaf(C32[6], fx, __builtin_fmaf(C32[7], fy, __builtin_fmaf(C32[8], fz, -oz)));
                    }
                }
                const int incl = wave_incl_scan(len);
                const int ex = incl - len;
                const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
                const bool ne = len > 0;
                const int q = (int)mbcnt64(__builtin_amdgcn_ballot_w64(ne));
                if (ne) {
                    Rw.dl[q] = st - ex;
                    Rw.sv[q] = v;
                }
                // home atom hg + a is candidate ex(center) + hg + a of the
                // center segment, when that segment is in this batch
                const int cl = center - sb;
                const int self0 = (cl >= 0 && cl < kWave) ? __builtin_amdgcn_readlane(ex, cl) : 1 << 28;
                if (far) {
                    H.fill = small_far(A, L, sd, total, ex, st, v.s, hb, nh, self0 + hg, H.fill);
                    continue;
                }
                for (int k0 = 0; k0 < total; k0 += kTileCands) {
                    const int nch = sgpr(min(kTileChunks, (total - k0 + kWave - 1) / kWave));
                    // marks where a non-empty segment other than the first starts
                    Rw.flag[lane] = 0u;
                    const int pp = ex - k0;
                    if (ne && q > 0 && pp > 0 && pp < kTileCands) fl[pp] = 1;
                    int acc = k0 == 0 ? 0 : (int)__popcll(__builtin_amdgcn_ballot_w64(ne && q > 0 && pp <= 0));
                    TileCands C;
#pragma unroll
                    for (int g = 0; g < kTileChunks; ++g) {
                        const uint64_t bm = __builtin_amdgcn_ballot_w64(fl[g * kWave + lane] != 0);
                        const int qk = acc + (int)(bm & 1u) + (int)mbcnt64(bm >> 1);
                        acc += (int)__popcll(bm);
                        const int kk = k0 + g * kWave + lane;
                        C.li[g] = kk < total ? kk + Rw.dl[qk] : kUnitAtoms;   // else the far sentinel
                        const SegShift t = Rw.sv[qk];
                        const TAtom c = L.a[C.li[g]];
                        C.bx[g] = c.x + t.x;
                        C.by[g] = c.y + t.y;
                        C.bz[g] = c.z + t.z;
                        C.bq[g] = 0.5f * __builtin_fmaf(C.bz[g], C.bz[g], __builtin_fmaf(C.by[g], C.by[g], C.bx[g] * C.bx[g]));
                        C.ent[g] = row8 ? c.j : c.j | (int)t.s;
                        if (row8) C.ct[g] = t.s - L.w[C.li[g]] + 2 * kPackZero;
                    }
                    // entries that the pass's chunks may store: what it starts with left, so
                    // a row runs over by less than a pass (kSlotSlack)
                    H.left = max(0, min(kWave, A.cap - (H.fill >> (row8 ? 3 : 2))));
                    const SmallEnv E{A.X, A.sys + s0 + k, L.a + hb, C, H, L.a};
                    const int kp = self0 + hg - k0;   // home atom hg + a is candidate kp + a of this pass
                    if (row8) {
                        if (nch == 4) tile_pass<4, kEntry8>(E, tol, C, nh, kp, H);
                        else if (nch == 3) tile_pass<3, kEntry8>(E, tol, C, nh, kp, H);
                        else tile_pass<2, kEntry8>(E, tol, C, nh, kp, H);
                    } else {
                        if (nch == 4) tile_pass<4, kEntry4>(E, tol, C, nh, kp, H);
                        else if (nch == 3) tile_pass<3, kEntry4>(E, tol, C, nh, kp, H);
                        else tile_pass<2, kEntry4>(E, tol, C, nh, kp, H);
                    }
                }
            }
            if (lane < nh) A.pair_count[ha] = row8 ? (H.fill >> 3) | kRow8Bit : H.fill >> 2;
        }
    }
}

template <typename TI>
static void small_launch(const PipelineBufs &b, hipStream_t st)
{
    SmallArgs A{b.X,          b.sys,     b.sys_atom_base, b.sys_cell_base, b.units,  b.unit_order,
                b.atom_sys,   b.rec,     b.perm_out,      b.cell_id_out,   b.cell_offsets_out,
                b.pair_count, b.slots,   b.slot_off8,     b.slot_row4,     b.slot_cap,
                b.item_tests, b.status};
    hipLaunchKernelGGL((small_kernel<TI>), dim3((unsigned)b.nitems), dim3(kSmallThreads), 0, st, A);
}

static void launch_small(const PipelineBufs &b, hipStream_t st)
{
    if (b.nitems <= 0) return;
    if (b.ti_bytes == 8) small_launch<int64_t>(b, st);
    else small_launch<int32_t>(b, st);
}

// Fill pass (fill_pairs_kernel!, gpu_kernels.jl:159-180): one wave per tile
// of TP = 64 TW consecutive output pairs, one lane per pair.  Tiles start at
// multiples of TP, so every store instruction covers one aligned 64-pair
// block of i, j, S (and R): the stores write whole cache lines, and lines
// shared between waves occur only at tile edges.  A wave issues the slot
// loads of all its TW blocks before its first store.
//
// R is computed here, from the positions (24 bytes gathered per pair, cached),
// by the expression of the 64-bit distance test: keeping it in rows beside the
// slots wrote and read 24 more bytes per pair through memory and held the
// count pass to its 64-bit form (count and fill with R, 20k atoms 47 / 30 us,
// 100k 93 / 66, 200k 162 / 123).
//
// The pair scan writes, per tile t, the atom A0 owning pair t TP and how
// many of its pairs come before that one; the next tile's entry bounds the
// tile's atoms from above (A1).  When the tile spans at most 64 atoms the
// wave loads their counts, one atom per lane, rebuilds their run starts by
// a scan, and finds the atom of each of its pairs by a binary search over
// the lanes.  A tile spanning more atoms (possible only when atoms without
// pairs lie in between) is filled by a per-lane search of pair_off instead.

// Slot entries, read raw (8 bytes for every narrow format, no branch) and
// decoded only after all of a wave's loads are issued.
template <bool WIDE>
struct RawEntry;
template <>
struct RawEntry<false> {
    uint64_t e;
    bool w8;
};
template <>
struct RawEntry<true> {
    int4 e;
};

template <bool WIDE>
__device__ __forceinline__ RawEntry<WIDE> load_entry(const void *__restrict__ slots, int64_t off8, int32_t row4, int32_t cap,
                                                     uint32_t row, int r, bool row8)
{
    RawEntry<WIDE> x;
    if constexpr (WIDE) {
        x.e = reinterpret_cast<const int4 *>(slots)[slot_row(row, cap) + r];
    } else {
        // a 4-byte row's last entry is read with the 4 bytes after it (the next
        // row's, or the 8-byte rows')
        const int64_t byte = (row8 ? off8 : 0) + slot_row(row, row8 ? 8 * cap : row4) + (r << (row8 ? 3 : 2));
        __builtin_memcpy(&x.e, reinterpret_cast<const char *>(slots) + byte, 8);
        x.w8 = row8;
    }
    return x;
}

template <bool WIDE>
__device__ __forceinline__ void decode_entry(const RawEntry<WIDE> &x, int32_t &j, int32_t &Sx, int32_t &Sy,
                                             int32_t &Sz)
{
    if constexpr (WIDE) {
        j = x.e.x; Sx = x.e.y; Sy = x.e.z; Sz = x.e.w;
    } else {
        const uint32_t lo = (uint32_t)x.e, hi = (uint32_t)(x.e >> 32);
        int32_t px, py, pz;
        unpack_wind(hi, px, py, pz);
        const uint32_t code = lo >> 26;
        j = x.w8 ? (int32_t)lo : (int32_t)(lo & (uint32_t)(kNarrowMaxAtoms - 1));
        Sx = x.w8 ? px : narrow_comp(code, 0);
        Sy = x.w8 ? py : narrow_comp(code, 1);
        Sz = x.w8 ? pz : narrow_comp(code, 2);
    }
}

// The stores are non-temporal: the output streams past the caches, which
// keep holding the slot rows the count pass wrote and the fill reads (with
// cached stores the 1M-atom fill ran at 147 us, with these at 103 us; 200k
// atoms with R 87 against 79).
//
// Bound by the bytes written.  Three 8-byte components per pair (R, and S
// in 64 bits) go through the wave's LDS: stored straight from the lanes, 24
// bytes apart, the Int64 fill of 1M atoms (1.05 GB) took 295 us, in whole lines
// 164 (6.4 TB/s); 200k atoms Int64 62 / 37 us, with R 99 / 80.  4-byte
// components (12 bytes apart) write as fast as they are (5.7 TB/s at 1M).
//
// Components v0, v1, v2 of pair `lane` to out[3 lane ..], for the first n
// pairs (wave-uniform n; lds: 3 kWave values of the wave's own).
template <typename T>
__device__ __forceinline__ void store_triples(T v0, T v1, T v2, T *__restrict__ out, int n, T *lds)
{
    const int lane = lane_id();
    lds[3 * lane] = v0;
    lds[3 * lane + 1] = v1;
    lds[3 * lane + 2] = v2;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    T w[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) w[k] = lds[k * kWave + lane];
    __builtin_amdgcn_wave_barrier();   // read before the next triples are written
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (k * kWave + lane < 3 * n) __builtin_nontemporal_store(w[k], out + k * kWave + lane);
}

// Store the pairs of one block of 64 output positions from pos0 on, the first
// n of them live.
template <typename TI>
__device__ __forceinline__ void fill_store_pairs(int32_t is, int32_t j, int32_t Sx, int32_t Sy, int32_t Sz, int64_t pos0,
                                                 int n, TI *__restrict__ i_out, TI *__restrict__ j_out,
                                                 TI *__restrict__ S_out, void *lds)
{
    const int lane = lane_id();
    if (lane < n) {
        __builtin_nontemporal_store((TI)is, i_out + pos0 + lane);
        __builtin_nontemporal_store((TI)(j + 1), j_out + pos0 + lane);
        if (sizeof(TI) == 4) {
            TI *S = S_out + 3 * (pos0 + lane);
            __builtin_nontemporal_store((TI)Sx, S);
            __builtin_nontemporal_store((TI)Sy, S + 1);
            __builtin_nontemporal_store((TI)Sz, S + 2);
        }
    }
    if (sizeof(TI) == 8) store_triples<TI>((TI)Sx, (TI)Sy, (TI)Sz, S_out + 3 * pos0, n, static_cast<TI *>(lds));
}

// R = xj - xi + C' * S  (gpu_kernels.jl:89)
__device__ __forceinline__ void pair_vector(const double *__restrict__ C, const double xi[3], const double xj[3],
                                            int32_t Sx, int32_t Sy, int32_t Sz, double R[3])
{
    double cx, cy, cz;
    cell_shift(C, Sx, Sy, Sz, cx, cy, cz);
    R[0] = (xj[0] - xi[0]) + cx;
    R[1] = (xj[1] - xi[1]) + cy;
    R[2] = (xj[2] - xi[2]) + cz;
}

// LDS of a fill block: one buffer of triples per wave when 8-byte
// components pass through it.
constexpr size_t kTripleBytes = 3 * kWave * 8;

template <bool WANT_R, bool WIDE, typename TI, int TW>
__global__ __launch_bounds__(1024) void fill_kernel(
    const double *__restrict__ X, const SysDev *__restrict__ sys, const int64_t *__restrict__ sys_atom_base,
    const int32_t *__restrict__ atom_sys, int nsys, int64_t nat, const int32_t *__restrict__ pair_count,
    const int64_t *__restrict__ pair_off, const int32_t *__restrict__ tile_atom, int64_t tile_cap,
    const void *__restrict__ slots, int64_t off8, int32_t row4, const Status *__restrict__ status,
    Status *__restrict__ status_pub, int32_t cap, int64_t pair_capacity, TI *__restrict__ i_out,
    TI *__restrict__ j_out, TI *__restrict__ S_out, double *__restrict__ R_out)
{
    constexpr int TP = TW * kWave;
    constexpr int32_t kBeyond = 1 << 30;   // window position past every pair of the tile
    extern __shared__ double fill_lds[];
    void *lds = fill_lds + 3 * kWave * (threadIdx.x / kWave);   // the wave's triples
    const int lane = lane_id();
    // tiles in block order: the waves in flight write one advancing front of
    // the output (an XCD-contiguous block order measured much slower)
    const int64_t w = (int64_t)blockIdx.x * (blockDim.x / kWave) + sgpr((int)(threadIdx.x / kWave));   // wave-uniform
    const int64_t Q0 = w * TP;
    if (blockIdx.x == 0 && threadIdx.x < kWave) {
        // the status is final once the fill runs: publish it to the host's
        // pinned copy (system-scope stores), then mark it published, so the
        // host can go on while the fill writes the pairs
        constexpr int kWords = sizeof(Status) / 4;
        constexpr int kPub = offsetof(Status, published) / 4;
        static_assert(kWords <= kWave, "one wave publishes the status");
        if (threadIdx.x < kWords && threadIdx.x != kPub) {
            const int32_t v = reinterpret_cast<const int32_t *>(status)[threadIdx.x];
            __hip_atomic_store(reinterpret_cast<int32_t *>(status_pub) + threadIdx.x, v, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_SYSTEM);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");   // system scope: every lane's words land first
        __builtin_amdgcn_wave_barrier();
        if (threadIdx.x == 0)
            __hip_atomic_store(&status_pub->published, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    const Status st = *status;
    // the atoms owning this tile's first pair and the next tile's, read with
    // the status (indexes clamped to the table, which holds at least two
    // entries: waves past the pairs return below without using them)
    const int64_t wc = w + 1 < tile_cap ? w : tile_cap - 2;
    const int32_t a0s = tile_atom[2 * wc], skip0 = tile_atom[2 * wc + 1], a1s = tile_atom[2 * wc + 2];
    __asm__ volatile("" ::"s"(a0s), "s"(skip0), "s"(a1s));   // keeps the loads ahead of the branch: their latency overlaps the status's
    if ((st.npairs > pair_capacity) | (st.max_count > cap) | (!WIDE & (st.wide != 0)) | (Q0 >= st.npairs)) return;
    const int nlive = (int)(st.npairs - Q0 < TP ? st.npairs - Q0 : TP);   // pairs of this tile
    const int64_t A0 = a0s;
    const int64_t A1 = Q0 + TP < st.npairs ? (int64_t)a1s : nat - 1;   // every pair of the tile is owned in [A0, A1]
    if (A1 - A0 < kWave) {
        // the window: atom A0 + k on lane k < span, its run of pairs
        // [fo, fo + cnt) relative to Q0 (the exclusive scan of the counts,
        // less the skip0 pairs of atom A0 before the tile); other lanes hold
        // kBeyond
        const int span = (int)(A1 - A0) + 1;
        const int64_t ak = A0 + lane;
        const bool vk = lane < span;
        const int32_t pck = vk ? pair_count[ak] : 0;
        const int32_t cntk = pck & kCountMask;
        const int32_t incl = wave_incl_scan(cntk);   // lanes past the span hold 0
        // runs past the tile end keep their exact start (<= TP + 64 cap)
        const int32_t fo = vk ? incl - cntk - skip0 : kBeyond;
        const uint64_t row8 = __ballot((pck & kRow8Bit) != 0);
        const int32_t fo0 = -skip0;   // atom A0 owns pair Q0
        const bool batch = nsys > 1;
        int32_t il = 0;   // batches: 1-based system-local index of the lane's atom
        if (batch && vk) il = (int32_t)(ak - sys_atom_base[atom_sys[ak]] + 1);
        // pair q = 64 u + lane belongs to the largest window lane s[u] whose
        // run starts at or before q: one binary search per block, all TW
        // searches advanced together (TW independent lane reads per step),
        // over just enough steps for the tile's span of atoms
        int top = 0;
        while (2 * top < span) top = top ? 2 * top : 1;   // 2 top >= span: s reaches span - 1
        int s[TW], f[TW];
#pragma unroll
        for (int u = 0; u < TW; ++u) {
            s[u] = 0;
            f[u] = fo0;
        }
        for (int step = top; step >= 1; step >>= 1) {
#pragma unroll
            for (int u = 0; u < TW; ++u) {
                const int f2 = __shfl(fo, s[u] + step, kWave);
                if (f2 <= u * kWave + lane) {
                    s[u] += step;
                    f[u] = f2;
                }
            }
        }
        RawEntry<WIDE> e[TW];
        int32_t is[TW];
#pragma unroll
        for (int u = 0; u < TW; ++u) {
            const int q = u * kWave + lane;
            const bool live = q < nlive;
            // pairs past the tile's end read entry 0 of row 0 (in bounds, never
            // stored): no branch around the load
            const int r = live ? q - f[u] : 0;
            const uint32_t row = live ? (uint32_t)(A0 + s[u]) : 0u;
            const bool w8 = ((row8 >> s[u]) & 1) != 0;
            is[u] = batch ? __shfl(il, s[u], kWave) : (int32_t)(A0 + s[u] + 1);
            e[u] = load_entry<WIDE>(slots, off8, row4, cap, row, r, w8);
        }
        if constexpr (!WANT_R) {
#pragma unroll
            for (int u = 0; u < TW; ++u) {
                int32_t j, Sx, Sy, Sz;
                decode_entry<WIDE>(e[u], j, Sx, Sy, Sz);   // outside the branch: it covers the stores only
                fill_store_pairs<TI>(is[u], j, Sx, Sy, Sz, Q0 + u * kWave, nlive - u * kWave, i_out, j_out, S_out, lds);
            }
        } else {
            // R from the positions themselves: every gather of the tile before
            // its first store
            int32_t j[TW], S[TW][3];
            double xi[TW][3], xj[TW][3];
#pragma unroll
            for (int u = 0; u < TW; ++u) {
                decode_entry<WIDE>(e[u], j[u], S[u][0], S[u][1], S[u][2]);
                const int64_t gi = A0 + s[u];
                const int64_t gj = u * kWave + lane < nlive ? gi - is[u] + 1 + j[u] : gi;   // the system's atom j
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    xi[u][k] = X[3 * gi + k];
                    xj[u][k] = X[3 * gj + k];
                }
            }
            const int s0 = batch ? sgpr(atom_sys[A0]) : 0;
            const bool one = !batch || s0 == sgpr(atom_sys[A1]);   // the whole tile in one system
#pragma unroll
            for (int u = 0; u < TW; ++u) {
                const int64_t pos0 = Q0 + u * kWave;
                const int n = nlive - u * kWave;
                fill_store_pairs<TI>(is[u], j[u], S[u][0], S[u][1], S[u][2], pos0, n, i_out, j_out, S_out, lds);
                double R[3];
                if (one) pair_vector(sys[s0].C, xi[u], xj[u], S[u][0], S[u][1], S[u][2], R);
                else pair_vector(sys[atom_sys[A0 + s[u]]].C, xi[u], xj[u], S[u][0], S[u][1], S[u][2], R);
                store_triples<double>(R[0], R[1], R[2], R_out + 3 * pos0, n, static_cast<double *>(lds));
            }
        }
        return;
    }
    // the tile's pairs span more than 64 atoms: each lane searches pair_off
    // between A0 and A1 for the atom of its pair
    const int64_t hi0 = A1;
    for (int u = 0; u < TW; ++u) {
        const int64_t pos0 = Q0 + u * kWave;
        const int n = nlive - u * kWave;   // may be none
        int64_t lo = A0, hi = hi0;   // largest atom in [lo, hi] whose run starts at or before the lane's pair
        const int64_t P = lane < n ? pos0 + lane : Q0;
        while (lo < hi) {
            const int64_t mid = (lo + hi + 1) >> 1;
            if (pair_off[mid] <= P) lo = mid;
            else hi = mid - 1;
        }
        const int r = (int)(P - pair_off[lo]);
        const int ls = nsys > 1 ? atom_sys[lo] : 0;
        const int32_t isv = (int32_t)(lo - (nsys > 1 ? sys_atom_base[ls] : 0) + 1);
        const RawEntry<WIDE> e = load_entry<WIDE>(slots, off8, row4, cap, (uint32_t)lo, r, (pair_count[lo] & kRow8Bit) != 0);
        int32_t j, Sx, Sy, Sz;
        decode_entry<WIDE>(e, j, Sx, Sy, Sz);
        fill_store_pairs<TI>(isv, j, Sx, Sy, Sz, pos0, n, i_out, j_out, S_out, lds);
        if constexpr (WANT_R) {
            const int64_t gj = lo - isv + 1 + j;
            const double xi[3] = {X[3 * lo], X[3 * lo + 1], X[3 * lo + 2]};
            const double xj[3] = {X[3 * gj], X[3 * gj + 1], X[3 * gj + 2]};
            double R[3];
            pair_vector(sys[ls].C, xi, xj, Sx, Sy, Sz, R);
            store_triples<double>(R[0], R[1], R[2], R_out + 3 * pos0, n, static_cast<double *>(lds));
        }
    }
}

// R of every pair of one large system in cell order: a wave takes kRAtoms
// consecutive sorted atoms, one lane per pair.  Atoms near one another in that
// order share neighbours, so the position gathers hit the L2; the
// fill's own, in atom order, do not once the positions outgrow it.  The
// price: every atom's run of R (37 pairs, 888 bytes) is written on its own, at
// 1.7 TB/s (cached stores: 20% slower).
constexpr int kRAtoms = 16;
// Atoms above which that pays: 24 bytes each against 4 MB of L2 (fill with R
// in cell order / in atom order: 200k atoms 85 / 70 us, 400k 168 / 204, 1M
// 487 / 646).
constexpr int64_t kRCellOrder = 262144;
__global__ __launch_bounds__(256) void fill_R_kernel(const double *__restrict__ X, const SysDev *__restrict__ sys,
                                                     int64_t nat, const Rec *__restrict__ rec,
                                                     const int32_t *__restrict__ pair_count,
                                                     const int64_t *__restrict__ pair_off, const void *__restrict__ slots,
                                                     int64_t off8, int32_t row4,
                                                     const Status *__restrict__ status, int32_t cap,
                                                     int64_t pair_capacity, double *__restrict__ R_out)
{
    __shared__ double lds[4][3 * kWave];
    __shared__ int64_t at[4][kWave];   // output position of each lane's pair
    const Status st = *status;
    if ((st.npairs > pair_capacity) | (st.max_count > cap) | (st.wide != 0)) return;
    const int lane = lane_id(), wv = (int)(threadIdx.x / kWave);
    const int64_t p0 = ((int64_t)blockIdx.x * 4 + sgpr((int)(threadIdx.x / kWave))) * kRAtoms;
    if (p0 >= nat) return;
    const int na = (int)(nat - p0 < kRAtoms ? nat - p0 : kRAtoms);
    Rec h{};
    int32_t pc = 0;
    int64_t gi = 0, off = 0;
    if (lane < na) {
        h = rec[p0 + lane];
        gi = h.j;   // single system
        pc = pair_count[gi];
        off = pair_off[gi];
    }
    const int cnt = pc & kCountMask;
    const int incl = wave_incl_scan(cnt);
    const int fo = lane < na ? incl - cnt : 1 << 30;
    const int total = sgpr(__shfl(incl, kWave - 1, kWave));
    const uint64_t row8 = __ballot((pc & kRow8Bit) != 0);
    for (int q0 = 0; q0 < total; q0 += kWave) {
        const int q = q0 + lane;
        int s = 0;
#pragma unroll
        for (int step = kRAtoms / 2; step >= 1; step >>= 1)
            if (__shfl(fo, s + step, kWave) <= q) s += step;
        const bool live = q < total;
        const int fs = __shfl(fo, s, kWave);   // read by every lane: the source may be a lane past the last pair
        const int r = live ? q - fs : 0;
        const int64_t ga = (int64_t)(int)__shfl((int)gi, s, kWave);
        const int64_t o = (int64_t)shfl64((uint64_t)off, s) + r;
        const RawEntry<false> e = load_entry<false>(slots, off8, row4, cap, live ? (uint32_t)ga : 0u, r, (row8 >> s) & 1);
        int32_t j, Sx, Sy, Sz;
        decode_entry<false>(e, j, Sx, Sy, Sz);
        const int64_t gj = live ? j : ga;
        const double xi[3] = {X[3 * ga], X[3 * ga + 1], X[3 * ga + 2]};
        const double xj[3] = {X[3 * gj], X[3 * gj + 1], X[3 * gj + 2]};
        double R[3];
        pair_vector(sys[0].C, xi, xj, Sx, Sy, Sz, R);
        lds[wv][3 * lane] = R[0];
        lds[wv][3 * lane + 1] = R[1];
        lds[wv][3 * lane + 2] = R[2];
        at[wv][lane] = o;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int e3 = k * kWave + lane, pr = e3 / 3;
            const double v = lds[wv][e3];
            const int64_t oo = at[wv][pr];
            if (q0 + pr < total) __builtin_nontemporal_store(v, R_out + 3 * oo + (e3 - 3 * pr));
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Positions back in atom order out of the records, for a fill with R when
// they came in the caller's device memory: the fill may run after the call has
// returned, when that memory is the caller's again.  (A build that is asked for R
// at once copies them in its sort: 5 us less at 20k atoms, 6 at 200k.)
__global__ __launch_bounds__(256) void unsort_kernel(const Rec *__restrict__ rec, const int32_t *__restrict__ atom_sys,
                                                     const int64_t *__restrict__ sys_atom_base, int64_t nat,
                                                     double *__restrict__ Xr)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= nat) return;
    const Rec h = rec[p];
    const int64_t g = (atom_sys ? sys_atom_base[atom_sys[p]] : 0) + h.j;   // a system's atoms stay in its range
    Xr[3 * g] = h.x;
    Xr[3 * g + 1] = h.y;
    Xr[3 * g + 2] = h.z;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------

template <int BT>
static void count_launch(const PipelineBufs &b, bool wide, hipStream_t st)
{
    if (wide)
        hipLaunchKernelGGL(count_kernel<BT>, dim3((unsigned)b.nbricks), dim3(BT), 0, st, b.sys,
                           b.sys_cell_base, b.sys_brick_base, b.nsys, b.M, b.nat, b.cell_start, b.rec, b.wbig,
                           b.pair_count, b.slots, b.slot_cap, b.status);
    else
        hipLaunchKernelGGL(tile_kernel<BT>, dim3((unsigned)(b.nbricks * b.brick_copies)), dim3(BT), 0, st, b.sys,
                           b.sys_cell_base, b.sys_brick_base, b.nsys, b.brick_copies, b.M, b.nat, b.cell_start, b.rec,
                           b.wbig, b.pair_count, b.slots, b.slot_off8, b.slot_row4, b.slot_cap, b.status);
}

void launch_count(const PipelineBufs &b, bool want_R, bool wide, hipStream_t st)
{
    if (b.nunits > 0) launch_small(b, st);   // cell list, counts and slot rows of every unit of small systems
    else if (b.nat == 0 || b.nbricks == 0) return;
    else if (b.count_block == 256) count_launch<256>(b, wide, st);
    else count_launch<512>(b, wide, st);
    const bool kept = b.X_keep && b.nunits == 0 && b.sort.bw >= 0;   // by the sort
    if (want_R && b.Xr != b.X && !kept)
        hipLaunchKernelGGL(unsort_kernel, dim3((unsigned)((b.nat + 255) / 256)), dim3(256), 0, st, b.rec, b.atom_sys,
                           b.sys_atom_base, b.nat, b.Xr);
}

template <bool R, bool W, typename TI, int TW>
static bool fill_launch(const PipelineBufs &b, hipStream_t st)
{
    // one wave per tile of the pair capacity (waves past the pairs return)
    const int bs = b.fill_block;
    const int64_t waves = (b.pair_capacity + TW * kWave - 1) / (TW * kWave);
    if (waves <= 0) return false;
    const unsigned nblk = (unsigned)((waves * kWave + bs - 1) / bs);
    const size_t lds = R || sizeof(TI) == 8 ? bs / kWave * kTripleBytes : 0;
    hipLaunchKernelGGL((fill_kernel<R, W, TI, TW>), dim3(nblk), dim3(bs), lds, st, b.Xr, b.sys, b.sys_atom_base,
                       b.atom_sys, b.nsys, b.nat, b.pair_count, b.pair_off, b.tile_atom, b.tile_cap, b.slots, b.slot_off8, b.slot_row4, b.status,
                       b.status_pub, b.slot_cap, b.pair_capacity, (TI *)b.i_out, (TI *)b.j_out, (TI *)b.S_out, b.R_out);
    return true;
}

template <bool R, bool W, typename TI>
static bool fill_tiles(const PipelineBufs &b, hipStream_t st)
{
    if (b.fill_pairs == 128) return fill_launch<R, W, TI, 2>(b, st);
    if (b.fill_pairs == 512) return fill_launch<R, W, TI, 8>(b, st);
    return fill_launch<R, W, TI, 4>(b, st);
}

template <typename TI>
static bool fill_dispatch(const PipelineBufs &b, bool want_R, bool wide, hipStream_t st)
{
    if (want_R && b.nsys == 1 && !wide && b.nat > kRCellOrder) {
        const bool launched = fill_tiles<false, false, TI>(b, st);
        hipLaunchKernelGGL(fill_R_kernel, dim3((unsigned)((b.nat + 4 * kRAtoms - 1) / (4 * kRAtoms))), dim3(256), 0, st,
                           b.Xr, b.sys, b.nat, b.rec, b.pair_count, b.pair_off, b.slots, b.slot_off8, b.slot_row4, b.status,
                           b.slot_cap, b.pair_capacity, b.R_out);
        return launched;
    }
    if (want_R) return wide ? fill_tiles<true, true, TI>(b, st) : fill_tiles<true, false, TI>(b, st);
    return wide ? fill_tiles<false, true, TI>(b, st) : fill_tiles<false, false, TI>(b, st);
}

bool launch_fill(const PipelineBufs &b, bool want_R, bool wide, hipStream_t st)
{
    if (b.nat == 0) return false;
    return b.ti_bytes == 8 ? fill_dispatch<int64_t>(b, want_R, wide, st) : fill_dispatch<int32_t>(b, want_R, wide, st);
}

}  // namespace nlh
