// pair_kernels.hpp -- DPD pair-force kernels (CCNTCell::UpdateForce, src/CNTCell.cpp:877-1572).
//
// Two kernels over the same cell-sorted SoA layout (both produce the same forces):
//   DPD_PAIR_FULLSHELL  one thread per bead visits all 27 neighbour cells and keeps only
//                       its own force (no scatter, no atomics).  Simple and exact; the
//                       cross-check for the hit-list kernel and the fallback beyond 2^26
//                       beads.
//   DPD_PAIR_HITLIST    the full-shell walk in two passes: candidates are tested on 4-byte
//                       scan codes (cell offsets to 8 bits), a neighbour row's three cells
//                       as one range, partners that may be in range are listed in LDS,
//                       then evaluated exactly in one dense loop (below).
// Both accumulate each bead's force in one thread in a fixed order, so forces are
// deterministic for a given layout.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dpd_engine.h"
#include "engine_common.hpp"

namespace dpd {

struct PairArgs {
    int n;                 // beads (all boxes)
    int nbox;
    int ngroups;           // scan groups of 64 cell keys (all boxes)
    const BoxDev* boxes;   // [nbox]
    const float4* pos;     // offset xyz, type | box << 8 (sorted)
    const float4* vp;      // predicted velocity xyz, id bits (sorted)
    const int* key;        // global cell key per slot
    const uint32_t* code;  // scan code per slot (scan_code), kCodePad slots of padding after n
    const int* cstart;     // [nkeys+1] first slot of each global cell key
    const float* table;    // per box: a | gamma | sqrt(gamma), kTypeStride each
    const int64_t* step;   // simulation time of this force evaluation (device)
    float4* frc;           // out: pair force per slot
    Sums sums;             // out (OBS): per box [6..14] virial sum dx_b F_a, [15] pair PE
    const int4* hitblk;    // hit-list workgroups of a batch: (box, first slot, end slot)
    int nhitblk;
    // the epilogue of a step that another follows (hit-list kernels, engines without bonded
    // terms): UpdateMom of this step, UpdatePos of the next, the bead filed under its new cell
    const float4* vel;     // v + dt/2 F of the previous step
    Intake intake;
    int* flags;            // [0] non-finite force or velocity, [1] moves of more than one cell
};

constexpr int kObsVir = 6;   // virial slots in the per-box accumulator
constexpr int kObsPEP = 15;

// Full-shell kernel: thread per bead.  Each pair is evaluated from both sides with the
// same operands (dx negated), so the two forces are exact negatives of each other;
// virial and PE are halved.
template <bool OBS, bool MULTI>
__global__ __launch_bounds__(256) void k_pair_fullshell(PairArgs A, BoxDev B0, int nblocks, int per_xcd)
{
    // XCD-aware: workgroup b runs on XCD b % 8 and takes block (b % 8) * per_xcd + b / 8
    const int blk = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (blk >= nblocks) return;
    const int i = blk * 256 + threadIdx.x;
    double vir[10];
    if (OBS)
        for (int q = 0; q < 10; ++q) vir[q] = 0.0;
    int box = -1;
    if (i < A.n) {
        const float4 pi = A.pos[i];
        const int wi = __float_as_int(pi.w);
        box = bead_box(wi);
        const BoxDev& B = MULTI ? A.boxes[box] : B0;
        const RngKey K = rng_key(B, *A.step);
        const float* tab = A.table + (MULTI ? box * kTableStride : 0);
        const float4 vi = A.vp[i];
        const int ti = bead_type(wi);
        const uint32_t idi = (uint32_t)__float_as_int(vi.w);
        int c[3];
        key_cell(A.key[i] - B.koff, B, c);
        float fx = 0.f, fy = 0.f, fz = 0.f;
        float sv[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        for (int dz = -1; dz <= 1; ++dz) {
            int cz = c[2] + dz;
            cz += (cz < 0) ? B.n[2] : ((cz >= B.n[2]) ? -B.n[2] : 0);
            for (int dy = -1; dy <= 1; ++dy) {
                int cy = c[1] + dy;
                cy += (cy < 0) ? B.n[1] : ((cy >= B.n[1]) ? -B.n[1] : 0);
                for (int dx = -1; dx <= 1; ++dx) {
                    int cx = c[0] + dx;
                    cx += (cx < 0) ? B.n[0] : ((cx >= B.n[0]) ? -B.n[0] : 0);
                    const int k = B.koff + cell_key(cx, cy, cz, B);
                    const int j0 = A.cstart[k], j1 = A.cstart[k + 1];
                    const float sx = -(float)dx * B.w[0], sy = -(float)dy * B.w[1], sz = -(float)dz * B.w[2];
                    for (int j = j0; j < j1; ++j) {
                        if (j == i) continue;
                        const float4 pj = A.pos[j];
                        const float ddx = (pi.x - pj.x) + sx;
                        const float ddy = (pi.y - pj.y) + sy;
                        const float ddz = (pi.z - pj.z) + sz;
                        const float dr2 = ddx * ddx + ddy * ddy + ddz * ddz;
                        if (dr2 < 1.0f && dr2 > 1e-18f) {
                            const float4 vj = A.vp[j];
                            const int tt = ti * kMaxTypes + bead_type(__float_as_int(pj.w));
                            const float dxdv = ddx * (vi.x - vj.x) + ddy * (vi.y - vj.y) + ddz * (vi.z - vj.z);
                            float pe;
                            const float s = pair_scalar(dr2, dxdv, tab[tt], tab[2 * kTypeStride + tt],
                                                        tab[kTypeStride + tt], idi, (uint32_t)__float_as_int(vj.w),
                                                        B.invrootdt, K, OBS ? &pe : nullptr);
                            const float Fx = s * ddx, Fy = s * ddy, Fz = s * ddz;
                            fx += Fx; fy += Fy; fz += Fz;
                            if (OBS) {
                                sv[0] += ddx * Fx; sv[1] += ddy * Fx; sv[2] += ddz * Fx;
                                sv[3] += ddx * Fy; sv[4] += ddy * Fy; sv[5] += ddz * Fy;
                                sv[6] += ddx * Fz; sv[7] += ddy * Fz; sv[8] += ddz * Fz;
                                sv[9] += pe;
                            }
                        }
                    }
                }
            }
        }
        A.frc[i] = make_float4(fx, fy, fz, 0.f);
        if (OBS)
            for (int q = 0; q < 10; ++q) vir[q] = 0.5 * (double)sv[q];
    }
    if (OBS) {
        const int box0 = MULTI ? bead_box(__float_as_int(A.pos[blk * 256].w)) : 0;
        accumulate_boxes<10>(vir, box, box0, kObsVir, A.sums);
    }
}

// Hit-list kernel: thread per bead in two passes.  The scan of the nine neighbour rows appends
// every partner that may be in range to a per-thread list in LDS (slot | segment code << 26);
// the wavefront then evaluates its lists together (evaluate_lists).  In the one-pass kernel a
// wavefront runs the whole pair evaluation (random stream, force) whenever any of its lanes
// has a partner in range -- on nearly every candidate iteration, with ~8% of the lanes busy.
// Partners are evaluated with the same expressions as k_pair_fullshell; the compiler contracts
// multiply-adds differently in the two code shapes, so the forces agree to ~1 ulp per term, not
// bitwise.  Slots must fit in 26 bits.
//
// What bounds it: instruction issue (rocprofv3: VALU active 85% of the cycles, 36M wavefront
// instructions on the condensate box of 64^3 cells), of which the scan is a third, the
// evaluation of 14 listed partners a bead (12.6 are in range) two fifths.  The scan costs 29 VALU
// instructions per pass of four candidates: positions modulo 256 in bytes need one subtraction
// and one dot product each (code_dist2), the codes of the next pass are loaded into the same
// registers as soon as these are subtracted, the x image of a partner is left to the evaluation
// (cell indices mod 4 in the beads' words), and a bead beside an x face goes on to the cell
// across it within the row's loop, so the wavefront's other lanes do not wait for a second one.
// Pair launch, relaxed boxes, with 58 instructions per pass, a second loop at the faces and lists
// evaluated lane by lane -> with 42 and lists evaluated together -> now: condensate 64^3
// 95 -> 79.4 -> 77 us, water 96^3 332 -> 252 -> 248, binary 40^3 38 -> 29.4 -> 29.1, bilayer
// 48x48x32 40 -> 31.0 -> 29.7, 64 water/lipid replicas 141 -> 102.6 -> 100.
// Slower: the z offsets in an array of their own (38 instructions per pass but a second load,
// 89 us on the condensate), two passes per turn (85), a wavefront's row of codes staged in LDS
// (98, the look-ups of each row and fewer registers), lists of 20 for a sixth wavefront (84 for
// the lists, 89 to 104 with the registers of six), lists of 29 beside a smaller table (76).
// A schedule of the hit-list kernel: threads per workgroup, list entries per thread (4 B of
// LDS each) and the flush threshold (after each row segment the wavefront evaluates its
// lists together once any of them holds this many; FLUSH = CAP never flushes).
// dpd_autotune_schedules picks among these by timing them.
constexpr int kHitSlotBits = 26;
constexpr uint32_t kHitSlotMask = (1u << kHitSlotBits) - 1u;
// slots of padding after the last scan code: the scan reads candidates four (or two) at a
// time, one pass ahead (seven past the end at most)
constexpr int kCodePad = 8;
// 1e-18 < dr2 < 1 as one unsigned compare of the bits: dr2 >= 0, NaN fails
constexpr uint32_t kPairLo = 0x219392EFu + 1u;   // bits of 1e-18f, plus one
__device__ inline bool pair_in_range(float dr2) { return __float_as_uint(dr2) - kPairLo < 0x3F800000u - kPairLo; }
// a 32-bit pointer into LDS (a generic pointer is 64 bits)
typedef __attribute__((address_space(3))) uint32_t lds_u32;
// two scan codes from one 4-byte-aligned 8-byte load
typedef uint32_t code2_t __attribute__((ext_vector_type(2), aligned(4)));
// four scan codes from one 4-byte-aligned 16-byte load
typedef uint32_t code4_t __attribute__((ext_vector_type(4), aligned(4)));
// a cell's start and end, from one 4-byte-aligned load
typedef int int2u __attribute__((ext_vector_type(2), aligned(4)));

// The candidate test in integer code units (u = w / kCodeUnits): the four bytes of code minus
// code, as one 32-bit difference, squared and added by one v_dot4_i32_i8.  Bytes hold positions
// modulo 256, so differences are right from -128 to 127, more than the cut-off's 84 to 88; the
// largest of a neighbour, 168, reads as -88 (and in cells of unequal sides, whose cut-off is
// wider in some units, one may pass that is not near: the evaluation drops it).  A borrow of x
// lowers y by one; it lowers the one of byte 2 instead of z, which adds at most one to the sum.
// Positions are floored, the bead's y half a unit lower: the difference is then within 1, 1.5
// and 1 units of the true one, so every pair inside the cut-off passes |d| < (1 + m) / u with
// m = 1.01 |(w_x, 1.5 w_y, w_z)| / kCodeUnits + 1e-5.
__device__ inline int code_dist2(uint32_t cj, uint32_t Q)
{
    const int d = (int)(cj - Q);
    return __builtin_amdgcn_sdot4(d, d, 0, true);
}
// beads per workgroup of THREADS threads with SPLIT lanes per bead (21 per wavefront for 3,
// 7 for 9; lane 63 idle)
constexpr int hit_beads(int threads, int split) { return split == 1 ? threads : (threads / 64) * (63 / split); }

// The step's end and the next step's start for slot i, whose force (Fx, Fy, Fz) this launch
// computed: the arithmetic of k_advance (MODE kEndBegin).  Used for engines without bonded
// terms (a bonded bead's force is not complete here); a bead flagged bonded is left alone.
// Every lane of the wavefront calls it (file_bead counts the wavefront's keys);
// `act` marks the lanes that hold a finished bead.
__device__ inline void pair_epilogue(const PairArgs& A, const BoxDev& B, int i, bool act, float Fx, float Fy,
                                     float Fz)
{
    const int from = A.key[min(i, A.n - 1)];
    int k = 0;
    if (act) {
        const float4 p = A.pos[i];
        act = !(__float_as_int(p.w) & kBondedBit);
        if (act) {
            // UpdateMom (k_sort repeats the sum and stores the next half step)
            float4 v = A.vel[i];
            v.x = kick(v.x, Fx, B.hdt);
            v.y = kick(v.y, Fy, B.hdt);
            v.z = kick(v.z, Fz, B.hdt);
            if (!(fabsf(Fx) + fabsf(Fy) + fabsf(Fz) < 1e30f) || !(fabsf(v.x) + fabsf(v.y) + fabsf(v.z) < 1e30f))
                atomicAdd(A.flags + 0, 1);
            int c[3];
            key_cell(from - B.koff, B, c);
            const float o[3] = {p.x, p.y, p.z};
            const int img[3] = {0, 0, 0};   // the image change is applied by k_sort
            const float d[3] = {drift(v.x, Fx, B), drift(v.y, Fy, B), drift(v.z, Fz, B)};
            Moved m;
            advance(o, c, img, d, B, m);
            k = B.koff + cell_key(m.c[0], m.c[1], m.c[2], B);
            if (m.jump) atomicAdd(A.flags + 1, 1);
            if (m.bad) atomicAdd(A.flags + 0, 1);
        }
    }
    file_bead(A.intake, from, k, i, act);
}

// body of the hit-list kernel for workgroup blockIdx.x (< 8 * per_xcd); also called by the
// kernel that runs the bonded terms in extra workgroups after the pair workgroups.  With
// several boxes each workgroup takes slots of one box only (A.hitblk[blk] = box, first
// slot, end slot), so the box, its constants and its table are uniform: scalar loads and
// the table in LDS, as for one box.
template <bool OBS, bool MULTI, int THREADS, int CAP, int FLUSH, int SPLIT, bool EPI>
__device__ __attribute__((always_inline)) inline void hitlist_body(const PairArgs& A, const BoxDev& B0, int nblocks,
                                                                   int per_xcd)
{
    static_assert(SPLIT == 1 || SPLIT == 3 || SPLIT == 9, "one, three or nine lanes per bead");
    // candidates per pass of the scan (one 16- or 8-byte load of scan codes)
    constexpr int PASS = SPLIT == 1 ? 4 : 2;
    static_assert(CAP > PASS, "room for a pass");
    static_assert(!(OBS && EPI), "the observing launch ends a sequence of steps");
    __shared__ uint32_t hits[CAP][THREADS];
    __shared__ float4 stab[kTypeStride];   // a, gamma, sqrt(gamma) sqrt(24 kT / dt) per type pair
    const int blk = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (blk >= nblocks) return;   // whole workgroups
    int box = 0, i0 = blk * hit_beads(THREADS, SPLIT), i1 = A.n;
    if (MULTI) {
        const int4 hb = A.hitblk[blk];
        box = hb.x; i0 = hb.y; i1 = hb.z;
    }
    const BoxDev& B = MULTI ? A.boxes[box] : B0;
    // the box's interaction table in LDS, and for each segment code the image of x in cells
    // (mod 4, in the place of the cell index in a bead's word) and the shifts of y and z
    __shared__ float4 shtab[64];
    const float* gtab = A.table + (size_t)box * kTableStride;
    for (int q = threadIdx.x; q < kTypeStride; q += THREADS)
        stab[q] = make_float4(gtab[q], gtab[kTypeStride + q], gtab[2 * kTypeStride + q] * B.invrootdt, 0.f);
    if (threadIdx.x < 64) {
        const int q = threadIdx.x, im = q & 3;
        const int s = im == 1 ? -B.n[0] : (im == 2 ? B.n[0] : 0);
        shtab[q] = make_float4(__int_as_float((s & 3) << kCellXShift), (float)(1 - ((q >> 2) & 3)) * B.w[1],
                               (float)(1 - (q >> 4)) * B.w[2], 0.f);
    }
    __syncthreads();
    const int t = threadIdx.x;
    // SPLIT 3: lanes 3g, 3g+1, 3g+2 of a wavefront share bead g (21 per wavefront, lane 63
    // idle) and scan the neighbour rows of z layers -1, 0, +1 each; SPLIT 9: lanes 9g .. 9g+8
    // share bead g (7 per wavefront) and scan one neighbour row each
    const int lane = t & 63;
    const int grp = SPLIT == 1 ? 0 : lane / SPLIT;
    const int part = SPLIT == 1 ? 0 : lane - SPLIT * grp;
    const int i = SPLIT == 1 ? i0 + t : i0 + (t >> 6) * (63 / SPLIT) + grp;
    const bool valid = i < i1 && (SPLIT == 1 || lane < 63);
    double vir[10];
    if (OBS)
        for (int q = 0; q < 10; ++q) vir[q] = 0.0;
    float fx = 0.f, fy = 0.f, fz = 0.f;
    // every lane of a wavefront with a bead runs the scan (lanes without one find nothing)
    if (__ballot(valid) != 0) {
        const int ii = min(i, i1 - 1);
        const float4 pi = A.pos[ii];
        const RngKey K = rng_key(B, *A.step);
        const float4 vi = A.vp[ii];
        const uint32_t idi = (uint32_t)__float_as_int(vi.w);
        const int key = A.key[ii];
        int c[3];
        key_cell(key - B.koff, B, c);
        // the bead's word for the evaluation: its row of the interaction table and, in the
        // place of the cell index, minus its cell's x index mod 4
        const int hw = (bead_type(__float_as_int(pi.w)) * kMaxTypes << 8) | ((-c[0] & 3) << kCellXShift);
        float sv[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        // this thread's list: column t of hits, entry e at hits[e][t]; wp is the next free one
        lds_u32* const lbase = (lds_u32*)&hits[0][t];
        const uint32_t laddr = (uint32_t)(size_t)lbase;   // its LDS byte address
        uint32_t wp = laddr;
        // one listed partner of a bead (offset bx, by, bz, word bw, velocity and id bv): the
        // entry is slot | segment code, pj and vj the partner's position and velocity
        auto force = [&](uint32_t e, const float4& pj, const float4& vj, float bx, float by, float bz, int bw,
                         float bvx, float bvy, float bvz, uint32_t bid, float& Fx, float& Fy, float& Fz) {
            const float4 sh = shtab[e >> kHitSlotBits];
            // the partner's cell less the bead's along x (-1, 0 or 1) from the indices mod 4
            const int wj = __float_as_int(pj.w);
            const int dc = __builtin_amdgcn_sbfe(wj + bw + __float_as_int(sh.x), kCellXShift, 2);
            const float ddx = fmaf(-(float)dc, B.w[0], bx) - pj.x;
            const float ddy = (by + sh.y) - pj.y;
            const float ddz = (bz + sh.z) - pj.z;
            const float dr2 = ddx * ddx + ddy * ddy + ddz * ddz;
            const float dxdv = ddx * (bvx - vj.x) + ddy * (bvy - vj.y) + ddz * (bvz - vj.z);
            const float4 tab = stab[(bw >> 8) + bead_type(wj)];
            float pe;
            float s = pair_scalar_t(dr2, dxdv, tab.x, tab.z, tab.y, bid, (uint32_t)__float_as_int(vj.w), K,
                                    OBS ? &pe : nullptr);
            // the scan lists a superset: the bead itself and partners just past the cut-off
            const bool in_range = pair_in_range(dr2);
            s = in_range ? s : 0.f;
            if (OBS) pe = in_range ? pe : 0.f;
            Fx = s * ddx; Fy = s * ddy; Fz = s * ddz;
            if (OBS) {
                sv[0] += ddx * Fx; sv[1] += ddy * Fx; sv[2] += ddz * Fx;
                sv[3] += ddx * Fy; sv[4] += ddy * Fy; sv[5] += ddz * Fy;
                sv[6] += ddx * Fz; sv[7] += ddy * Fz; sv[8] += ddz * Fz;
                sv[9] += pe;
            }
        };
        auto eval = [&](uint32_t e, const float4& pj, const float4& vj) {
            float Fx, Fy, Fz;
            force(e, pj, vj, pi.x, pi.y, pi.z, hw, vi.x, vi.y, vi.z, idi, Fx, Fy, Fz);
            fx += Fx; fy += Fy; fz += Fz;
        };
        // evaluate and clear this thread's list, two entries per pass (both loads in
        // flight, two independent random-stream chains), in list order
        auto drain_to = [&](int nh) {
            int h = 0;
            for (; h + 1 < nh; h += 2) {
                const uint32_t ea = lbase[h * THREADS], eb = lbase[(h + 1) * THREADS];
                const int ja = (int)(ea & kHitSlotMask), jb = (int)(eb & kHitSlotMask);
                const float4 pa = A.pos[ja], va = A.vp[ja];
                const float4 pb = A.pos[jb], vb = A.vp[jb];
                eval(ea, pa, va);
                eval(eb, pb, vb);
            }
            if (h < nh) {
                const uint32_t ea = lbase[h * THREADS];
                const int ja = (int)(ea & kHitSlotMask);
                eval(ea, A.pos[ja], A.vp[ja]);
            }
            wp = laddr;
        };
        auto drain = [&]() { drain_to((int)(wp - laddr) / (4 * THREADS)); };
        // The lists of a wavefront's 64 beads.  Their lengths differ (13.0 partners at density
        // 3, the longest of 64 lists 17), and a loop over the longest leaves a quarter of the
        // lanes idle.  So every lane evaluates its first R entries, R the mean length less
        // one or two, and the entries past R of all lanes are packed and evaluated 64 at a
        // time, each lane taking whichever bead's partner comes next (the bead's data by lane
        // permutes), the forces handed back through LDS and added by the bead's own lane in
        // list order (list by list to the longest: condensate 64^3 84 us per launch, this way 82;
        // and where a list fills up within a row, all are evaluated this way instead of that
        // lane's alone: the box's unrelaxed start 163 -> 99 us).  The LDS rows below R, evaluated by then, hold the packed entries, their
        // beads and the forces, three rows per 64.
        auto evaluate_lists = [&]() {
            const int n = (int)(wp - laddr) / (4 * THREADS);
            int R = max((__builtin_amdgcn_readlane(wave_incl_scan(n), 63) >> 6) - 1, 0) & ~1;
            int ex, incl, total, nb;
            while (true) {
                ex = max(n - R, 0);
                incl = wave_incl_scan(ex);
                total = __builtin_amdgcn_readlane(incl, 63);
                nb = (total + 63) >> 6;
                if (3 * nb <= R) break;
                R += 2;   // (room for the packed entries; none are left at the longest list)
            }
            drain_to(min(n, R));
            if (nb == 0) return;
            lds_u32* const wbase = lbase - lane;   // the wavefront's column 0
            const int off = incl - ex;
            for (int k = 0; k < ex; ++k) {
                const int q = off + k;
                lds_u32* const to = wbase + (q >> 6) * (3 * THREADS) + (q & 63);
                to[0] = lbase[(R + k) * THREADS];
                to[THREADS] = (uint32_t)lane;
            }
            __builtin_amdgcn_wave_barrier();
            for (int b = 0; b < nb; ++b) {
                lds_u32* const row = lbase + b * (3 * THREADS);
                const bool act = 64 * b + lane < total;
                const uint32_t e = row[0];
                const int o = (int)row[THREADS] & 63;
                const float bx = __shfl(pi.x, o), by = __shfl(pi.y, o), bz = __shfl(pi.z, o);
                const float bvx = __shfl(vi.x, o), bvy = __shfl(vi.y, o), bvz = __shfl(vi.z, o);
                const int bw = __shfl(hw, o);
                const uint32_t bid = (uint32_t)__shfl((int)idi, o);
                if (act) {
                    const int j = (int)(e & kHitSlotMask);
                    float Fx, Fy, Fz;
                    force(e, A.pos[j], A.vp[j], bx, by, bz, bw, bvx, bvy, bvz, bid, Fx, Fy, Fz);
                    row[0] = __float_as_uint(Fx);
                    row[THREADS] = __float_as_uint(Fy);
                    row[2 * THREADS] = __float_as_uint(Fz);
                }
            }
            __builtin_amdgcn_wave_barrier();
            for (int k = 0; k < ex; ++k) {
                const int q = off + k;
                lds_u32* const at = wbase + (q >> 6) * (3 * THREADS) + (q & 63);
                fx += __uint_as_float(at[0]);
                fy += __uint_as_float(at[THREADS]);
                fz += __uint_as_float(at[2 * THREADS]);
            }
        };
        // candidate test on the scan codes (code_dist2) with the sum of squares taken in units of
        // the smallest u_a: every pair inside the cut-off passes sum d_a^2 < thr
        // = ((1 + m) / u_min)^2 + 2 (a wider superset for cells of unequal sides); the evaluation
        // drops the rest (the bead itself among them).
        const int thr = B.qthr;
        const char* cbase = reinterpret_cast<const char*>(A.code);
        const char* sbase = reinterpret_cast<const char*>(A.cstart);
        // the bead's own position as its neighbours' codes have theirs; a row across a periodic
        // face sees it a box's length away
        const int Qx = (int)floorf(pi.x * B.qinv[0]) + kCodeUnits * c[0];
        const int Qy = (int)floorf(pi.y * B.qinv[1] - 0.5f) + kCodeUnits * c[1];
        const int Qz = (int)floorf(pi.z * B.qinv[2]) + kCodeUnits * c[2];
        auto code_of = [](int x, int y, int z) {
            return (uint32_t)(x & 0xFF) | ((uint32_t)(y & 0xFF) << 8) | ((uint32_t)z << 24);
        };
        const uint32_t Q0 = code_of(Qx, Qy, Qz);
        const bool faces = __ballot(c[1] == 0 || c[1] == B.n[1] - 1 || c[2] == 0 || c[2] == B.n[2] - 1) != 0;
        // A row's cells are consecutive keys: cells cx-1 .. cx+1 are one range of slots, or,
        // where the row wraps through the periodic x face, two cells and the one across the
        // face, a second segment of that lane.
        const int nx = B.n[0], nxy = B.n[0] * B.n[1], nall = nxy * B.n[2];
        const bool xl = c[0] == 0, edge = xl || c[0] == nx - 1;
        const bool across = __ballot(edge) != 0;
        const int ym = c[1] == 0 ? nxy - nx : -nx, yp = c[1] == B.n[1] - 1 ? nx - nxy : nx;
        const int zm = c[2] == 0 ? nall - nxy : -nxy, zp = c[2] == B.n[2] - 1 ? nxy - nall : nxy;
        const int pa = xl ? key : key - 1, pb = pa + (edge ? 2 : 3);
        // (the bead's own cell where there is none: its starts are loaded and not used)
        const int pe = xl ? key + nx - 1 : (edge ? key + 1 - nx : key);
        // code and x of the second segment: the cell across the face, at -1 or nx
        const uint32_t img = xl ? 1u : 2u;
        const int qimg = (xl ? nx : -nx) * kCodeUnits;
        // the neighbour rows of this lane: all nine, one z layer (SPLIT 3) or one row (SPLIT 9)
        constexpr int NR = 9 / SPLIT;
        auto row_key = [&](int r) {
            const int dz = r / 3, dy = r - 3 * dz;   // 0, 1, 2
            return (dy == 0 ? ym : (dy == 2 ? yp : 0)) + (dz == 0 ? zm : (dz == 2 ? zp : 0));
        };
        using code_t = typename std::conditional<PASS == 4, code4_t, code2_t>::type;
        auto start_of = [&](int k) { return *reinterpret_cast<const int*>(sbase + ((uint32_t)k << 2)); };
        auto codes_at = [&](uint32_t b) { return *reinterpret_cast<const code_t*>(cbase + b); };
        // (a row's starts are loaded one row ahead)
        int jn0 = start_of(pa + row_key(part * NR)), jn1 = start_of(pb + row_key(part * NR));
        for (int q = 0; q < NR; ++q) {
            const int r = part * NR + q;
            const int dz = r / 3, dy = r - 3 * dz;
            const int j0 = jn0, j1 = jn1;
            code_t cc = codes_at((uint32_t)j0 << 2);
            if (q + 1 < NR) {
                const int d = row_key(r + 1);
                jn0 = start_of(pa + d);
                jn1 = start_of(pb + d);
            }
            const int krow = row_key(r);
            const uint32_t code = (uint32_t)((dy << 2) | (dz << 4)) << kHitSlotBits;
            uint32_t Q = Q0;
            if (faces) {
                const int sy = dy == 0 ? (c[1] == 0 ? B.n[1] : 0) : (dy == 2 && c[1] == B.n[1] - 1 ? -B.n[1] : 0);
                const int sz = dz == 0 ? (c[2] == 0 ? B.n[2] : 0) : (dz == 2 && c[2] == B.n[2] - 1 ? -B.n[2] : 0);
                Q = code_of(Qx, Qy + kCodeUnits * sy, Qz + kCodeUnits * sz);
            }
            // list entries of the segment's first candidate and of its end
            uint32_t e = (uint32_t)j0 | code, e1 = valid ? (uint32_t)j1 | code : e;
            uint32_t jb = (uint32_t)j0 << 2;
            int2u ce = {0, 0};
            if (across) ce = *reinterpret_cast<const int2u*>(sbase + ((uint32_t)(pe + krow) << 2));
            bool more = valid && edge;
            // PASS consecutive candidates per pass, the next pass's codes loaded as soon as
            // these are subtracted.  The loads run up to seven codes past the segment (the next
            // cells' beads, or the padding after the last slot); none of those is listed.
            // Slots are below 2^26, so byte offsets fit 32 bits and the loads address from the
            // array base.  Every candidate is stored at the list's write pointer, which
            // advances on a hit only (a miss is overwritten by the next store).
            auto put = [&](int d2, uint32_t ej, bool in_seg) {
                *(lds_u32*)(size_t)wp = ej;
                wp += ((d2 < thr) & in_seg) ? 4 * THREADS : 0;
            };
            // one pass
            auto pass = [&]() {
                int d2[PASS];
#pragma unroll
                for (int k = 0; k < PASS; ++k) d2[k] = code_dist2(cc[k], Q);
                jb += 4 * PASS;
                cc = codes_at(jb);
                put(d2[0], e, true);
#pragma unroll
                for (int k = 1; k < PASS; ++k) put(d2[k], e + k, e + k < e1);
                e += PASS;
            };
            const uint32_t full = laddr + 4 * (CAP - PASS) * THREADS;   // no room for a pass beyond
            while (true) {
                if (!across) {
                    while (e < e1 && wp <= full) pass();
                } else {
                    while (true) {
                        if (e >= e1) {
                            // the cell across the x face, for a bead beside it
                            if (!more) break;
                            more = false;
                            e = (uint32_t)ce.x | code | (img << kHitSlotBits);
                            e1 = (uint32_t)ce.y | code | (img << kHitSlotBits);
                            jb = (uint32_t)ce.x << 2;
                            Q = (Q & 0xFFFFFF00u) | (uint32_t)((Qx + qimg) & 0xFF);
                            if (e >= e1) break;
                            cc = codes_at(jb);
                        }
                        if (wp > full) break;
                        pass();
                    }
                }
                // a lane whose list is full leaves the loop before its segment's end: the
                // wavefront then evaluates all its lists, as after the last row
                const bool full_lists = __ballot(e < e1 || more) != 0;
                if (full_lists || q == NR - 1 || (FLUSH < CAP && __ballot(wp >= laddr + 4 * FLUSH * THREADS) != 0)) {
                    if constexpr (SPLIT == 1) evaluate_lists();
                    else drain();
                }
                if (!full_lists) break;
                cc = codes_at(jb);
            }
        }
        if (SPLIT == 1 && valid) A.frc[i] = make_float4(fx, fy, fz, 0.f);
        if (OBS)
            for (int q = 0; q < 10; ++q) vir[q] = 0.5 * (double)sv[q];
    }
    if (SPLIT > 1) {
        // the bead's force: its lanes' parts (z layers, or rows in z-major order) added in
        // lane order (the whole wavefront takes part in the shuffles)
        const int b = SPLIT * grp;
        float sx = __shfl(fx, b), sy = __shfl(fy, b), sz = __shfl(fz, b);
#pragma unroll
        for (int q = 1; q < SPLIT; ++q) {
            sx += __shfl(fx, b + q);
            sy += __shfl(fy, b + q);
            sz += __shfl(fz, b + q);
        }
        fx = sx;
        fy = sy;
        fz = sz;
        if (valid && part == 0) A.frc[i] = make_float4(fx, fy, fz, 0.f);
    }
    if (EPI) pair_epilogue(A, B, i, valid && part == 0, fx, fy, fz);
    if (OBS) {
        // (lanes without a bead too: they evaluate pairs of the wavefront's others)
        accumulate_boxes<10, THREADS / 64>(vir, box, box, kObsVir, A.sums);
    }
}

// Wavefronts per SIMD that the LDS of a schedule allows (160 KB per CU, four SIMDs), at most
// 5: the kernel needs 92 VGPRs (96 with the epilogue, 12 bytes of them spilled: 248 us on water 96^3
// against 281 with four wavefronts), and held to the 80 of six it spills more (condensate 64^3:
// 123 us against 80 us per launch for 512 and 256 threads with 24 entries).  512-thread workgroups then fit twice, four wavefronts per SIMD.
constexpr int hit_waves(int threads, int cap)
{
    const int lds = cap * threads * 4 + kTypeStride * 16 + 64 * 16;
    const int per = threads / 64, w = (160 * 1024 / lds) * per / 4;
    return w < 5 ? w : 20 / per * per / 4;
}
// the occupancy a kernel is held to: the split schedules run small boxes, which never fill
// the SIMDs, and get the registers of four wavefronts (no spills)
constexpr int hit_waves_eu(bool obs, int threads, int cap, int split)
{
    return (obs || split > 1) ? 4 : hit_waves(threads, cap);
}

template <bool OBS, bool MULTI, int THREADS, int CAP, int FLUSH, int SPLIT, bool EPI>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(hit_waves_eu(OBS, THREADS, CAP, SPLIT))))
void k_pair_hitlist(PairArgs A, BoxDev B0, int nblocks, int per_xcd)
{
    hitlist_body<OBS, MULTI, THREADS, CAP, FLUSH, SPLIT, EPI>(A, B0, nblocks, per_xcd);
}

// The schedules of the pair launch: hit-list kernels with their parameters, and the
// full-shell kernel.  A schedule id is what the autotuner stores.
struct Schedule {
    int kernel;    // DPD_PAIR_HITLIST or DPD_PAIR_FULLSHELL
    int threads, cap, flush;
    int split;     // lanes per bead (hit list): 1, 3 (one z layer of neighbour rows each) or 9 (one row)
    const char* name;
    constexpr int beads() const { return hit_beads(threads, split); }   // per workgroup
};
constexpr int kSchedules = 7;
constexpr Schedule kSchedule[kSchedules] = {
    {DPD_PAIR_HITLIST, 512, 24, 24, 1, "hitlist-t512-c24"},
    {DPD_PAIR_HITLIST, 512, 24, 16, 1, "hitlist-t512-c24-f16"},
    {DPD_PAIR_HITLIST, 256, 24, 24, 1, "hitlist-t256-c24"},
    {DPD_PAIR_HITLIST, 256, 32, 32, 1, "hitlist-t256-c32"},
    {DPD_PAIR_FULLSHELL, 256, 0, 0, 1, "fullshell-t256"},
    {DPD_PAIR_HITLIST, 256, 12, 12, 3, "hitlist-split3-t256-c12"},
    {DPD_PAIR_HITLIST, 256, 8, 8, 9, "hitlist-split9-t256-c8"},
};
constexpr int kDefaultSchedule = 2;
// The automatic choice for n beads.  Nine lanes per bead while that leaves most of the 1024
// SIMDs a wavefront or two; fewer beads of an engine without bonded terms, whose launch also
// files the beads, by atomics for seven beads a wavefront.  Three lanes while their wavefronts
// fit the SIMDs at once (four each); one with the longest lists while its do, then one with a
// fifth wavefront.  Microseconds per step at 9, 3, 1 (lists of 32) and 1 (of 24) lanes, density 3:
// water 10.1k beads 19.9, 20.5; 12.3k 21.8, 20.8; 98k 41.2, 31.8, 32.0; 108k 43, 38.0, 31.9,
// 32.8; 256k -, -, 42.0, 42.8; 273k -, -, 54.7, 47.0; chains 41k 24.5, 25.8; 66k 31.1, 30.1;
// 89k 37, 34.0, 35.7; 118k 43, 41.3, 36.7; 256k -, -, 47.0, 49.0; 292k -, -, 59.6, 52.3.
// A batch goes by all its beads, however many boxes they are in (bonded, boxes of 11,300 each: 4
// of them 31.6, 34.4, 39.4, 40.2; 8 42.0, 41.0, 43.6, 43.9; 16 63, 58.6, 51.3, 52.0; 24 86, 78,
// 72.9, 65.4).
constexpr int size_schedule(int64_t n, bool bonded)
{
    return n <= (bonded ? 50000 : 11000) ? 6 : (n <= 100000 ? 5 : (n <= 4 * 1024 * 64 ? 3 : kDefaultSchedule));
}
constexpr int kFullShellSchedule = 4;

// hit-list launch of schedule S on a grid of workgroups of its thread count
template <int S, bool OBS, bool MULTI, bool EPI>
inline void launch_hitlist_s(const PairArgs& a, const BoxDev& B0, int nblocks, hipStream_t s)
{
    constexpr Schedule q = kSchedule[S];
    const int ph = (nblocks + 7) / 8;
    hipLaunchKernelGGL((k_pair_hitlist<OBS, MULTI, q.threads, q.cap, q.flush, q.split, EPI>), dim3(8 * ph),
                       dim3(q.threads), 0, s, a, B0, nblocks, ph);
}

template <bool OBS, bool MULTI, bool EPI>
inline void launch_hitlist(int sched, const PairArgs& a, const BoxDev& B0, int nblocks, hipStream_t s)
{
    switch (sched) {
    case 1: launch_hitlist_s<1, OBS, MULTI, EPI>(a, B0, nblocks, s); break;
    case 2: launch_hitlist_s<2, OBS, MULTI, EPI>(a, B0, nblocks, s); break;
    case 3: launch_hitlist_s<3, OBS, MULTI, EPI>(a, B0, nblocks, s); break;
    case 5: launch_hitlist_s<5, OBS, MULTI, EPI>(a, B0, nblocks, s); break;
    case 6: launch_hitlist_s<6, OBS, MULTI, EPI>(a, B0, nblocks, s); break;
    default: launch_hitlist_s<0, OBS, MULTI, EPI>(a, B0, nblocks, s); break;
    }
}

// whether the hit-list kernel's list entries and row addresses hold an engine's slots and keys
inline bool hitlist_fits(int64_t n, int64_t ngroups) { return n <= (int64_t)kHitSlotMask && ngroups < (1 << 24); }

// whether schedule `sched` can carry the step's epilogue (hit-list kernels only)
inline bool epilogue_available(int sched, int64_t n, int64_t ngroups)
{
    return sched >= 0 && sched < kSchedules && kSchedule[sched].kernel == DPD_PAIR_HITLIST && hitlist_fits(n, ngroups);
}

// The automatic choice: the hit-list kernel for every engine whose slots fit its 26-bit list
// entries, the full-shell kernel beyond.
inline int default_pair_kernel(int64_t nbeads)
{
    return nbeads <= (int64_t)kHitSlotMask ? DPD_PAIR_HITLIST : DPD_PAIR_FULLSHELL;
}

inline bool pair_kernel_available(int which) { return which == DPD_PAIR_FULLSHELL || which == DPD_PAIR_HITLIST; }

// The pair launch of schedule `sched`.  A batch's hit-list workgroups take the slots of one
// box each: hitblk (nhitblk entries) must be the table built for the schedule's thread count.
// `epi`: the launch also carries the step's epilogue (epilogue_available(sched) must hold).
inline hipError_t launch_pair_kernel(int sched, const PairArgs& a, const BoxDev& B0, bool obs, hipStream_t s,
                                     bool epi = false)
{
    const bool multi = a.nbox > 1;
    if (sched < 0 || sched >= kSchedules) sched = kDefaultSchedule;
    if (kSchedule[sched].kernel == DPD_PAIR_HITLIST && hitlist_fits(a.n, a.ngroups) && (!multi || a.hitblk)) {
        const int nb = kSchedule[sched].beads();
        const int gh = multi ? a.nhitblk : (a.n + nb - 1) / nb;
        if (obs) {
            if (multi) launch_hitlist<true, true, false>(sched, a, B0, gh, s);
            else launch_hitlist<true, false, false>(sched, a, B0, gh, s);
        } else if (epi) {
            if (multi) launch_hitlist<false, true, true>(sched, a, B0, gh, s);
            else launch_hitlist<false, false, true>(sched, a, B0, gh, s);
        } else {
            if (multi) launch_hitlist<false, true, false>(sched, a, B0, gh, s);
            else launch_hitlist<false, false, false>(sched, a, B0, gh, s);
        }
        return hipGetLastError();
    }
    if (epi) return hipErrorInvalidValue;   // the full-shell kernel carries no epilogue
    // the full-shell kernel (also for hit lists beyond 2^26 beads)
    const int g = (a.n + 255) / 256;
    const int per_xcd = (g + 7) / 8;
    const dim3 grid(8 * per_xcd);
    if (obs) {
        if (multi) hipLaunchKernelGGL((k_pair_fullshell<true, true>), grid, dim3(256), 0, s, a, B0, g, per_xcd);
        else hipLaunchKernelGGL((k_pair_fullshell<true, false>), grid, dim3(256), 0, s, a, B0, g, per_xcd);
    } else {
        if (multi) hipLaunchKernelGGL((k_pair_fullshell<false, true>), grid, dim3(256), 0, s, a, B0, g, per_xcd);
        else hipLaunchKernelGGL((k_pair_fullshell<false, false>), grid, dim3(256), 0, s, a, B0, g, per_xcd);
    }
    return hipGetLastError();
}

}  // namespace dpd
