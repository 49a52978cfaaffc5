// slice_stress.hip -- z-slice stress profile of one box (CMonitor::AddBeadStress,
// src/Monitor.cpp:1900-2104, CMonitor::AddBondStress, :2283-2518, and
// CMonitor::AddBondPairStress, :2520-2739).
//
// The reference zeroes its slice tables every step and adds F (x) dx of every pair (and,
// when a stress analysis asks for it, of every bond) into the z-slices spanned by the two
// beads.  Here the tables are produced on demand for the engine's current state: the pair
// forces are re-evaluated with the same arithmetic and the same counter-based random
// draws as the step kernels, so right after dpd_step they are the last step's forces.
// Pair and bond forces are parallel to dx, so F (x) dx is symmetric: six sums, mirrored when
// they leave LDS.
//
// What bounds it: FP64 atomics (global ones at ~3e9 per second, whatever the addresses; a
// wavefront's LDS ones serialise lane by lane).  So every table entry is summed in LDS first:
// pairs in a window of the slices that one layer of cells reaches (a workgroup takes slots of
// one z layer at a time, and the slots are sorted by z), bonds and bond pairs in windows of
// the whole table.  Bilayer 48x48x32, 221k beads, 64 slices (global atomics per pair and bond
// -> now): pairs 13,700 -> 88 us, bonds 715 -> 15, bond pairs 1,767 -> 28.  The atomics are
// then 30 us of the pairs; the rest is their scan and evaluation, with few wavefronts to hide a
// load (177 us with one position loaded at a time and lists of 12 that a lane evaluated alone
// whenever they were full).
#include <algorithm>
#include <cmath>

#include "pair_kernels.hpp"
#include "slice_stress.hpp"

namespace dpd {

namespace {

// The slice of an interaction at z (in slices), the two beside a border it lies on.  z is wrapped
// into [0, Lz): the indices are in range; the clamp only guards the table against a position
// rounded onto Lz.
template <class Add>
__device__ inline void flat_split(int nslice, double z, const Add& add)
{
    const int i = min(max((int)z, 0), nslice - 1);
    if (z - (double)i > 0.00001) {
        add(i, 1.0);
    } else {
        add(i, 0.5);
        add(i > 0 ? i - 1 : nslice - 1, 0.5);
    }
}

// The z-slice split of one interaction (see orc_slice_add for the rule) between z1 and z2,
// dz = z1 - z2 unwrapped: add(slice, share) for every slice spanned.  A flat interaction
// (|dz| <= kFlat) lies at z1, whatever z2 is.
constexpr double kFlat = 0.00001;
template <class Add>
__device__ inline void slice_split(int nslice, double Lz, double z1, double z2, double dz, const Add& add)
{
    const double width = Lz / nslice, inv = nslice / Lz;
    double zd = dz, zu, zl;
    if (zd > kFlat) { zu = z1 * inv; zl = z2 * inv; }
    else if (zd < -kFlat) { zd = -zd; zu = z2 * inv; zl = z1 * inv; }
    else { zu = zl = z1 * inv; }
    int iu = min(max((int)zu, 0), nslice - 1), il = min(max((int)zl, 0), nslice - 1);
    const double ru = zu - (double)iu, rl = zl - (double)il;
    if (iu == il) {
        if (zu != zl || ru > 0.00001) {
            add(il, 1.0);
        } else {
            add(iu, 0.5);
            if (--il < 0) il += nslice;
            add(il, 0.5);
        }
    } else {
        const double inner = width / zd;
        if (iu > il) {
            for (int sl = il + 1; sl <= iu - 1; ++sl) add(sl, inner);
        } else {
            for (int sp = il + 1; sp <= nslice + iu - 1; ++sp) add(sp >= nslice ? sp - nslice : sp, inner);
        }
        add(il, rl > 0.000001 ? (1.0 - rl) * inner : inner);
        if (ru > 0.000001) add(iu, ru * inner);
    }
}

// the six sums of a symmetric tensor and where the nine components read them
__device__ constexpr int kSym[9] = {0, 1, 2, 1, 3, 4, 2, 4, 5};
__device__ constexpr int kTri[6] = {0, 1, 2, 4, 5, 8};   // their components 3a + b, a <= b

__device__ inline double wrapped_z(const SliceArgs& A, int slot)
{
    int c[3];
    key_cell(A.key[slot] - A.B.koff, A.B, c);
    return (double)c[2] * A.B.wd[2] + (double)A.pos[slot].z;
}

// The pair table, each pair once (half shell: the cell's later beads, the cell after it in the
// row and the nine and three cells of the rows after).  Workgroup b takes slots [b, b + 1) per,
// one z layer of cells after the other; lds holds `copies` tables [win][types][6] (types: unordered
// pairs) of the slices from s0 on, lane l adding to copy l mod copies.  The sums of types ti <= tj
// go to their components a <= b of out; k_slice_mirror spreads them afterwards.  Without WIN
// (no window fits LDS) the pairs add to out themselves.
// Seen from either bead a pair spans the same slices, unless it is flat: then each bead has half
// of it in its own slices, under (its type, the other's).  So j's half is moved there from i's,
// and what (ti, tj) gets beyond half of the sum, and (tj, ti) lacks, is left in out's entry of
// types (tj, ti), ti < tj.  One pair in 1e5 is flat; these go straight to out, after the others of
// their lists (a call on the 48x48x32 bilayer 206 us; with the halves told apart within the loop
// over all pairs 215, after each pair 207).
// LIST: listed partners per thread; when one of the lanes that scan has no room for four more,
// they evaluate their lists together.  28 where they fit 64 KB beside the window, else 12 (a
// call on the 48x48x32 bilayer with 64 slices, and one of 48x40x20 with 250: 108 and 151 us,
// with 12 127 and 192; with 28 a lane alone 105 and 148, but 353 with 12).
constexpr int kSliceListLong = 28, kSliceListShort = 12;
constexpr size_t slice_list_bytes(int list) { return (size_t)list * 256 * (sizeof(int) + 1); }
template <bool WIN, int LIST>
__global__ __launch_bounds__(256) void k_slice_pairs(SliceArgs A, double* __restrict__ out, int per, int win, int copies)
{
    extern __shared__ double lt[];
    __shared__ int list[LIST][256];         // partner slots
    __shared__ uint8_t row[LIST][256];      // and their row and image codes
    const BoxDev& B = A.B;
    const int t = threadIdx.x;
    const int ntri = A.ntypes * (A.ntypes + 1) / 2, tab = win * ntri * 6, stride = tab + 1;
    const double Lz = (double)B.n[2] * B.wd[2], inv = A.nslice / Lz;
    const RngKey K = rng_key(B, *A.step);
    // the box's beads are the slots of its cell keys
    const int s0b = A.cstart[B.koff], s1b = A.cstart[B.koff + B.ngroups * kGroupKeys];
    const int nxy = B.n[0] * B.n[1];
    int first = s0b + blockIdx.x * per;
    const int last = min(s1b, first + per);
    double* mine = lt + (t % copies) * stride;
    while (first < last) {
        int c0[3];
        key_cell(A.key[first] - B.koff, B, c0);
        const int layer = min(last, A.cstart[B.koff + nxy * (c0[2] + 1)]);
        // the first slice of the window; one below the layer's, for beads on a slice border
        const int s0 = win >= A.nslice ? 0 : (int)floor(c0[2] * B.wd[2] * inv) - 1;
        if (WIN) {
            for (int q = t; q < copies * stride; q += 256) lt[q] = 0.0;
            __syncthreads();
        }
        for (int i0 = first; i0 < layer; i0 += 256) {
            const int i = min(i0 + t, layer - 1);
            const bool valid = i0 + t < layer;
            const float4 pi = A.pos[i], vi = A.vp[i];
            const int wi = __float_as_int(pi.w), ti = bead_type(wi);
            const uint32_t idi = (uint32_t)__float_as_int(vi.w);
            int c[3];
            key_cell(A.key[i] - B.koff, B, c);
            const double zi = (double)c[2] * B.wd[2] + (double)pi.z;
            const int nci = (-c[0] & 3) << kCellXShift;
            int n = 0;
            // separation from a listed partner j in row code r = dy + 1 + 4 (dz + 1) with x image
            // im (1: one box length below, 2: above)
            auto shift_x = [&](int im) { return (((im == 1 ? -B.n[0] : (im == 2 ? B.n[0] : 0)) & 3) << kCellXShift); };
            auto separation = [&](const float4& pj, int im, int dy, int dz, float d[3]) {
                const int dc = __builtin_amdgcn_sbfe(__float_as_int(pj.w) + nci + shift_x(im), kCellXShift, 2);
                d[0] = fmaf(-(float)dc, B.w[0], pi.x) - pj.x;
                d[1] = (pi.y - (float)dy * B.w[1]) - pj.y;
                d[2] = (pi.z - (float)dz * B.w[2]) - pj.z;
                return d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
            };
            // the pair of listed partner h: its sums, the partner's z, dz and the types
            struct Pair {
                double f[6], zj, dz;
                int lo, hi;
            };
            auto pair_of = [&](int h) {
                const int j = list[h][t], code = row[h][t];
                const int im = code & 3, dy = ((code >> 2) & 3) - 1, dz = code >> 4;
                const float4 pj = A.pos[j], vj = A.vp[j];
                float d[3];
                const float dr2 = separation(pj, im, dy, dz, d);
                const int tj = bead_type(__float_as_int(pj.w));
                const int tt = ti * kMaxTypes + tj;
                const float dxdv = d[0] * (vi.x - vj.x) + d[1] * (vi.y - vj.y) + d[2] * (vi.z - vj.z);
                const float s = pair_scalar(dr2, dxdv, A.table[tt], A.table[2 * kTypeStride + tt],
                                            A.table[kTypeStride + tt], idi, (uint32_t)__float_as_int(vj.w),
                                            B.invrootdt, K, nullptr);
                int cz = c[2] + dz;
                cz -= cz >= B.n[2] ? B.n[2] : 0;
                const double sx = (double)s * d[0], sy = (double)s * d[1], sz = (double)s * d[2];
                return Pair{{sx * d[0], sx * d[1], sx * d[2], sy * d[1], sy * d[2], sz * d[2]},
                            (double)cz * B.wd[2] + (double)pj.z, (double)d[2], min(ti, tj), max(ti, tj)};
            };
            auto evaluate = [&]() {
                int flat = 0;   // flat pairs, to the list's front
                for (int h = 0; h < n; ++h) {
                    const Pair p = pair_of(h);
                    slice_split(A.nslice, Lz, zi, p.zj, p.dz, [&](int sl, double share) {
                        if constexpr (WIN) {
                            int w = sl - s0;
                            w -= w >= A.nslice ? A.nslice : 0;
                            w += w < 0 ? A.nslice : 0;
                            w = min(w, win - 1);   // (holds: keeps a bad state's sums in the table)
                            double* q = mine + (w * ntri + p.hi * (p.hi + 1) / 2 + p.lo) * 6;
#pragma unroll
                            for (int m = 0; m < 6; ++m) atomicAdd(q + m, p.f[m] * share);
                        } else {
                            double* q = out + ((size_t)sl * A.nidx + p.lo * A.ntypes + p.hi) * 9;
#pragma unroll
                            for (int m = 0; m < 6; ++m) atomicAdd(q + kTri[m], p.f[m] * share);
                        }
                    });
                    if (fabs(p.dz) <= kFlat) {
                        list[flat][t] = list[h][t];
                        row[flat++][t] = row[h][t];
                    }
                }
                for (int h = 0; h < flat; ++h) {
                    const Pair p = pair_of(h);
                    for (int of_j = 0; of_j < 2; ++of_j)
                        flat_split(A.nslice, inv * (of_j ? p.zj : zi), [&](int sl, double share) {
                            const double sum = of_j ? 0.5 * share : -0.5 * share;
                            const double more = (ti == p.lo) == (of_j == 0) ? 0.25 * share : -0.25 * share;
                            double* q = out + ((size_t)sl * A.nidx + p.lo * A.ntypes + p.hi) * 9;
                            double* r = out + ((size_t)sl * A.nidx + p.hi * A.ntypes + p.lo) * 9;
#pragma unroll
                            for (int m = 0; m < 6; ++m) {
                                atomicAdd(q + kTri[m], p.f[m] * sum);
                                if (p.lo != p.hi) atomicAdd(r + kTri[m], p.f[m] * more);
                            }
                        });
                }
                n = 0;
            };
            auto scan = [&](int j0, int j1, int im, int dy, int dz) {
                for (int j = j0; j < j1; j += 4) {
                    float4 p[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) p[u] = A.pos[min(j + u, j1 - 1)];
                    if (__any(n > LIST - 4)) evaluate();
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        float d[3];
                        const float dr2 = separation(p[u], im, dy, dz, d);
                        if (j + u < j1 && dr2 < 1.0f && dr2 > 1e-18f) {
                            list[n][t] = j + u;
                            row[n++][t] = (uint8_t)(im | ((dy + 1) << 2) | (dz << 4));
                        }
                    }
                }
            };
            if (valid) {
                // the five rows: own (beads after i, and the next cell), (1, 0), (-1 .. 1, 1)
                for (int r = 0; r < 5; ++r) {
                    const int dz = r >= 2, dy = r < 2 ? r : r - 3;
                    int cy = c[1] + dy, cz = c[2] + dz;
                    cy += (cy < 0) ? B.n[1] : ((cy >= B.n[1]) ? -B.n[1] : 0);
                    cz -= cz >= B.n[2] ? B.n[2] : 0;
                    const int k = B.koff + B.n[0] * (cy + B.n[1] * cz);
                    const int x0 = r == 0 ? c[0] : max(c[0] - 1, 0), x1 = min(c[0] + 1, B.n[0] - 1);
                    scan(r == 0 ? i + 1 : A.cstart[k + x0], A.cstart[k + x1 + 1], 0, dy, dz);
                    if (r > 0 && c[0] == 0) scan(A.cstart[k + B.n[0] - 1], A.cstart[k + B.n[0]], 1, dy, dz);
                    if (c[0] == B.n[0] - 1) scan(A.cstart[k], A.cstart[k + 1], 2, dy, dz);
                }
                evaluate();
            }
        }
        if (WIN) {
            __syncthreads();
            for (int q = t; q < tab; q += 256) {
                double v = 0.0;
                for (int r = 0; r < copies; ++r) v += lt[r * stride + q];
                if (v != 0.0) {
                    int sl = s0 + q / (ntri * 6);
                    sl += sl < 0 ? A.nslice : 0;
                    sl -= sl >= A.nslice ? A.nslice : 0;
                    int u = q / 6 % ntri, hi = 0;
                    while ((hi + 1) * (hi + 2) / 2 <= u) ++hi;
                    const int lo = u - hi * (hi + 1) / 2;
                    atomicAdd(out + ((size_t)sl * A.nidx + lo * A.ntypes + hi) * 9 + kTri[q % 6], v);
                }
            }
            __syncthreads();
        }
        first = layer;
    }
}

// the pair table's other halves: types (tj, ti) beside (ti, tj), half of the sum each and the
// flat pairs' difference, and the components below the diagonal
__global__ __launch_bounds__(256) void k_slice_mirror(SliceArgs A, double* __restrict__ out)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)A.nslice * A.nidx) return;
    const int lo = (int)(q % A.nidx) / A.ntypes, hi = (int)(q % A.nidx) % A.ntypes;
    if (lo > hi) return;
    double* a = out + q * 9;
    double* b = out + (q - lo * A.ntypes - hi + hi * A.ntypes + lo) * 9;
    const double share = lo == hi ? 1.0 : 0.5;
    double v[6], more[6];
    for (int m = 0; m < 6; ++m) {
        v[m] = a[kTri[m]] * share;
        more[m] = lo != hi ? b[kTri[m]] : 0.0;
    }
    for (int m = 0; m < 9; ++m) a[m] = v[kSym[m]] + more[kSym[m]];
    if (lo != hi)
        for (int m = 0; m < 9; ++m) b[m] = v[kSym[m]] - more[kSym[m]];
}

// Tables of bonds and bond pairs: workgroup (b, w) adds the interactions it takes (every
// gridDim.x-th 256) to the slices [w win, (w + 1) win) in LDS, NC sums per slice and index, and
// then to out.  win 0: not even one slice fits LDS, out is added to directly.
template <int NC>
struct SliceTable {
    double* lt;
    double* out;
    int nslice, nidx, win, w0;
    __device__ SliceTable(const SliceArgs& A, double* lds, double* o, int win_)
        : lt(lds), out(o), nslice(A.nslice), nidx(A.nidx), win(win_), w0((int)blockIdx.y * win_)
    {
        for (int q = threadIdx.x; q < win * nidx * NC; q += blockDim.x) lt[q] = 0.0;
        __syncthreads();
    }
    __device__ static int sum_of(int m) { return NC == 6 ? kSym[m] : m; }
    __device__ void add(int sl, int idx, const double (&f)[NC], double share)
    {
        if (win) {
            const int w = sl - w0;
            if (w < 0 || w >= win) return;
            double* q = lt + ((size_t)w * nidx + idx) * NC;
#pragma unroll
            for (int m = 0; m < NC; ++m) atomicAdd(q + m, f[m] * share);
        } else {
            double* q = out + ((size_t)sl * nidx + idx) * 9;
            for (int m = 0; m < 9; ++m) atomicAdd(q + m, f[sum_of(m)] * share);
        }
    }
    __device__ void flush()
    {
        __syncthreads();
        const int ns = min(win, nslice - w0);
        for (int q = threadIdx.x; q < ns * nidx * 9; q += blockDim.x) {
            const double v = lt[(q / 9) * NC + sum_of(q % 9)];
            if (v != 0.0) atomicAdd(out + (size_t)w0 * nidx * 9 + q, v);
        }
    }
};

// bonds of the box: head - tail (unwrapped), force on the head, FP64
__global__ __launch_bounds__(256) void k_slice_bonds(SliceArgs A, double* __restrict__ out, int win)
{
    extern __shared__ double lt[];
    SliceTable<6> T(A, lt, out, win);
    const BoxDev& B = A.B;
    for (int q = A.b0 + blockIdx.x * 256 + threadIdx.x; q < A.b1; q += gridDim.x * 256) {
        const int2 hb = A.bond_bead[q];
        const int sh = A.slot_of[hb.x], st = A.slot_of[hb.y];
        double uh[3], ut[3];
        for (int e = 0; e < 2; ++e) {
            const int slot = e ? st : sh;
            int c[3];
            key_cell(A.key[slot] - B.koff, B, c);
            const float4 p = A.pos[slot];
            const int4 a = A.img[e ? hb.y : hb.x];
            double* u = e ? ut : uh;
            u[0] = (double)(c[0] + a.x * B.n[0]) * B.wd[0] + (double)p.x;
            u[1] = (double)(c[1] + a.y * B.n[1]) * B.wd[1] + (double)p.y;
            u[2] = (double)(c[2] + a.z * B.n[2]) * B.wd[2] + (double)p.z;
        }
        const double2 par = A.bond_par[q];
        const double d[3] = {uh[0] - ut[0], uh[1] - ut[1], uh[2] - ut[2]};
        const double L = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
        const double s = par.x * (par.y - L) / L;
        const double F[3] = {s * d[0], s * d[1], s * d[2]};
        const double f[6] = {F[0] * d[0], F[0] * d[1], F[0] * d[2], F[1] * d[1], F[1] * d[2], F[2] * d[2]};
        const int th = bead_type(__float_as_int(A.pos[sh].w)), tt = bead_type(__float_as_int(A.pos[st].w));
        slice_split(A.nslice, (double)B.n[2] * B.wd[2], wrapped_z(A, sh), wrapped_z(A, st), d[2],
                    [&](int sl, double share) { T.add(sl, th * A.ntypes + tt, f, share); });
    }
    T.flush();
}

__device__ inline void unwrapped(const SliceArgs& A, int bead, int slot, double u[3])
{
    const BoxDev& B = A.B;
    int c[3];
    key_cell(A.key[slot] - B.koff, B, c);
    const float4 p = A.pos[slot];
    const int4 a = A.img[bead];
    u[0] = (double)(c[0] + a.x * B.n[0]) * B.wd[0] + (double)p.x;
    u[1] = (double)(c[1] + a.y * B.n[1]) * B.wd[1] + (double)p.y;
    u[2] = (double)(c[2] + a.z * B.n[2]) * B.wd[2] + (double)p.z;
}

// CMonitor::AddBondPairStress (src/Monitor.cpp:2520-2739), thread per bond pair: the bond
// pair's forces (FP64, as in the step), then its three bead pairs first tail -> first
// head -> second head -> first tail, each adding 0.33333333 (F[j+1] - F[j]) (x)
// (u[j+1] - u[j]) over the slices it spans, keyed by the bead types (second head, first
// head, first tail) where the reference keys by bond-pair type.
__global__ __launch_bounds__(256) void k_slice_bondpairs(SliceArgs A, double* __restrict__ out, int win)
{
    extern __shared__ double lt[];
    SliceTable<9> T(A, lt, out, win);
    for (int q = A.a0 + blockIdx.x * 256 + threadIdx.x; q < A.a1; q += gridDim.x * 256) {
        const int4 abc = A.ang_bead[q];
        const int sa = A.slot_of[abc.x], sb = A.slot_of[abc.y], sc = A.slot_of[abc.z];
        double ua[3], ub[3], uc[3], f[3][3];
        unwrapped(A, abc.x, sa, ua);
        unwrapped(A, abc.y, sb, ub);
        unwrapped(A, abc.z, sc, uc);
        angle_forces(ua, ub, uc, A.ang_par[q], f, nullptr);   // f[0] on c, f[1] on b, f[2] on a
        const double* u[4] = {uc, ub, ua, uc};
        const double* F[4] = {f[0], f[1], f[2], f[0]};
        const int slot[4] = {sc, sb, sa, sc};
        const int nt = A.ntypes;
        const int idx = (bead_type(__float_as_int(A.pos[sa].w)) * nt + bead_type(__float_as_int(A.pos[sb].w))) * nt +
                        bead_type(__float_as_int(A.pos[sc].w));
        const double Lz = (double)A.B.n[2] * A.B.wd[2];
        for (int j = 0; j < 3; ++j) {
            double dx[3], fj[3];
            for (int d = 0; d < 3; ++d) {
                dx[d] = u[j + 1][d] - u[j][d];
                fj[d] = 0.33333333 * (F[j + 1][d] - F[j][d]);
            }
            double f9[9];
            for (int m = 0; m < 9; ++m) f9[m] = fj[m / 3] * dx[m % 3];
            slice_split(A.nslice, Lz, wrapped_z(A, slot[j + 1]), wrapped_z(A, slot[j]), dx[2],
                        [&](int sl, double share) { T.add(sl, idx, f9, share); });
        }
    }
    T.flush();
}

// The 13 half-shell neighbours of the reference's cells (CSimBox::MakeCNTCells,
// src/SimBox.cpp:830-867) as bits of the neighbour code (dx+1) + 3 (dy+1) + 9 (dz+1):
// (1,-1,0), (1,0,0), (0,1,0), (1,1,0) and the nine cells of the layer above.
constexpr uint32_t kHalfShellMask = (1u << 11) | (1u << 14) | (1u << 16) | (1u << 17) | (0x1FFu << 18);

// CCNTCell::UpdateTotalEnergy's pair sum (src/CNTCell.cpp:2909-3229): every pair inside a
// cell once, a pair across cells only from the cell whose half shell holds the other cell
// and only when the neighbour's id is the larger (src/CNTCell.cpp:3081), so the
// reference's energy output leaves out about half of the cross-cell pairs.  Thread per bead
// over its 27 neighbour cells, 1/2 a (1 - r)^2 in FP64; out[0] += the sum.
__global__ __launch_bounds__(256) void k_energy_pairs(SliceArgs A, double* __restrict__ out)
{
    const BoxDev& B = A.B;
    const int s0 = A.cstart[B.koff], s1 = A.cstart[B.koff + B.ngroups * kGroupKeys];
    double e = 0.0;
    for (int i = s0 + blockIdx.x * blockDim.x + threadIdx.x; i < s1; i += gridDim.x * blockDim.x) {
        const float4 pi = A.pos[i];
        const int ti = bead_type(__float_as_int(pi.w));
        const int idi = __float_as_int(A.vp[i].w);
        int c[3];
        key_cell(A.key[i] - B.koff, B, c);
        for (int nb = 0; nb < 27; ++nb) {
            const int ox = nb % 3 - 1, oy = (nb / 3) % 3 - 1, oz = nb / 9 - 1;
            const bool same = nb == 13, half = (kHalfShellMask >> nb) & 1u;
            if (!same && !half) continue;
            int cx = c[0] + ox, cy = c[1] + oy, cz = c[2] + oz;
            cx += (cx < 0) ? B.n[0] : ((cx >= B.n[0]) ? -B.n[0] : 0);
            cy += (cy < 0) ? B.n[1] : ((cy >= B.n[1]) ? -B.n[1] : 0);
            cz += (cz < 0) ? B.n[2] : ((cz >= B.n[2]) ? -B.n[2] : 0);
            const int k = B.koff + cell_key(cx, cy, cz, B);
            const float sx = (float)ox * B.w[0], sy = (float)oy * B.w[1], sz = (float)oz * B.w[2];
            for (int j = A.cstart[k], j1 = A.cstart[k + 1]; j < j1; ++j) {
                if (j == i) continue;
                if (half && !(__float_as_int(A.vp[j].w) > idi)) continue;
                const float4 pj = A.pos[j];
                const float dx = (pi.x - pj.x) - sx, dy = (pi.y - pj.y) - sy, dz = (pi.z - pj.z) - sz;
                const double dr2 = (double)(dx * dx + dy * dy + dz * dz);
                if (!(dr2 < 1.0)) continue;
                const double dr = sqrt(dr2);
                if (!(dr > 0.000000001)) continue;
                const int tt = ti * kMaxTypes + bead_type(__float_as_int(pj.w));
                // a pair inside a cell is seen from both of its beads: half from each
                e += (same ? 0.25 : 0.5) * (double)A.table[tt] * (1.0 - dr) * (1.0 - dr);
            }
        }
    }
    e = wave_sum(e);
    if ((threadIdx.x & 63) == 0 && e != 0.0) atomicAdd(out, e);
}

// bond and bond-pair potential energies of the box (src/Bond.cpp:279-288,
// src/BondPair.cpp:320-378): thread per bond, then per bond pair; out[1], out[2]
__global__ __launch_bounds__(256) void k_energy_bonded(SliceArgs A, double* __restrict__ out)
{
    const int nb = A.b1 - A.b0, q = blockIdx.x * blockDim.x + threadIdx.x;
    double eb = 0.0, ea = 0.0;
    if (q < nb) {
        const int2 hb = A.bond_bead[A.b0 + q];
        double uh[3], ut[3];
        unwrapped(A, hb.x, A.slot_of[hb.x], uh);
        unwrapped(A, hb.y, A.slot_of[hb.y], ut);
        const double2 par = A.bond_par[A.b0 + q];
        const double L = sqrt((uh[0] - ut[0]) * (uh[0] - ut[0]) + (uh[1] - ut[1]) * (uh[1] - ut[1]) +
                              (uh[2] - ut[2]) * (uh[2] - ut[2]));
        eb = 0.5 * par.x * (L - par.y) * (L - par.y);
    } else if (q < nb + A.a1 - A.a0) {
        const int g = A.a0 + q - nb;
        const int4 abc = A.ang_bead[g];
        double ua[3], ub[3], uc[3], f[3][3];
        unwrapped(A, abc.x, A.slot_of[abc.x], ua);
        unwrapped(A, abc.y, A.slot_of[abc.y], ub);
        unwrapped(A, abc.z, A.slot_of[abc.z], uc);
        angle_forces(ua, ub, uc, A.ang_par[g], f, &ea);
    }
    eb = wave_sum(eb);
    ea = wave_sum(ea);
    if ((threadIdx.x & 63) == 0) {
        if (eb != 0.0) atomicAdd(out + 1, eb);
        if (ea != 0.0) atomicAdd(out + 2, ea);
    }
}

}  // namespace

hipError_t launch_energy_output(const SliceArgs& a, double* out3, hipStream_t s)
{
    hipLaunchKernelGGL(k_energy_pairs, dim3(kEnergyBlocks), dim3(256), 0, s, a, out3);
    const int nq = (a.b1 - a.b0) + (a.a1 - a.a0);
    if (nq > 0) hipLaunchKernelGGL(k_energy_bonded, dim3((nq + 255) / 256), dim3(256), 0, s, a, out3);
    return hipGetLastError();
}

// slices of a bonded table that fit LDS (nc sums per index); 0: none, or too many windows
static int slice_window(const SliceArgs& a, int nc)
{
    const int win = (int)std::min<size_t>((size_t)a.nslice, kSliceLdsBytes / (sizeof(double) * nc * a.nidx));
    return win > 0 && (a.nslice + win - 1) / win <= 64 ? win : 0;
}

hipError_t launch_slice_bondpairs(const SliceArgs& a, double* tab, hipStream_t s)
{
    if (a.a1 > a.a0) {
        const int win = slice_window(a, 9);
        const dim3 grid(std::min((a.a1 - a.a0 + 255) / 256, win ? kSliceBondBlocks : 1 << 20),
                        win ? (a.nslice + win - 1) / win : 1);
        hipLaunchKernelGGL(k_slice_bondpairs, grid, dim3(256), sizeof(double) * win * a.nidx * 9, s, a, tab, win);
    }
    return hipGetLastError();
}

hipError_t launch_slice_stress(const SliceArgs& a, double* pair_tab, double* bond_tab, hipStream_t s)
{
    if (pair_tab) {
        // the slices that one layer of cells and the next reach, and one more at each end
        const double Lz = (double)a.B.n[2] * a.B.wd[2];
        const int win = (int)std::min<double>(a.nslice, std::ceil(2.0 * a.B.wd[2] * a.nslice / Lz) + 3.0);
        const size_t tab = (size_t)(a.ntypes * (a.ntypes + 1) / 2) * 6 * win + 1;
        int copies = 1;
        while (copies < 16 && 2 * copies * tab * sizeof(double) <= kSliceCopyBytes) copies *= 2;
        const int nb = std::max(1, a.nbeads);
        // whole 256s of slots per workgroup, about kSliceBlocks workgroups
        const int per = (nb + kSliceBlocks * 256 - 1) / (kSliceBlocks * 256) * 256;
        const dim3 gr((nb + per - 1) / per), bl(256);
        const size_t lds = copies * tab * sizeof(double);
        if (tab * sizeof(double) > kSliceLdsBytes)
            hipLaunchKernelGGL((k_slice_pairs<false, kSliceListLong>), gr, bl, 0, s, a, pair_tab, per, 0, 1);
        else if (lds + slice_list_bytes(kSliceListLong) <= 65536)
            hipLaunchKernelGGL((k_slice_pairs<true, kSliceListLong>), gr, bl, lds, s, a, pair_tab, per, win, copies);
        else
            hipLaunchKernelGGL((k_slice_pairs<true, kSliceListShort>), gr, bl, lds, s, a, pair_tab, per, win, copies);
        hipLaunchKernelGGL(k_slice_mirror, dim3((unsigned)(((size_t)a.nslice * a.nidx + 255) / 256)), dim3(256), 0, s, a,
                           pair_tab);
    }
    if (bond_tab && a.b1 > a.b0) {
        const int win = slice_window(a, 6);
        const dim3 grid(std::min((a.b1 - a.b0 + 255) / 256, win ? kSliceBondBlocks : 1 << 20),
                        win ? (a.nslice + win - 1) / win : 1);
        hipLaunchKernelGGL(k_slice_bonds, grid, dim3(256), sizeof(double) * win * a.nidx * 6, s, a, bond_tab, win);
    }
    return hipGetLastError();
}

}  // namespace dpd
