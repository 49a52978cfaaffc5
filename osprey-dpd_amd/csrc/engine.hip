// engine.hip -- the DPD step engine for MI355X (gfx950): kernels and the C ABI of
// include/dpd_engine.h.  One engine holds one box or a batch of independent boxes
// (replicas of uneven size and parameters); every kernel spans all boxes at once.
//
// One step (the reference's CSimBox::Evolve, src/SimBox.cpp:977-1120) runs as:
//   k_advance   UpdateMom of the previous step fused with UpdatePos of this one
//               (src/CNTCell.cpp:2280-2310, :1704-1757); files each bead under its new cell
//               (without bonded terms the previous pair launch's epilogue does this)
//   k_sort      the counting sort and the move into the new cell-sorted SoA buffers, beads
//               of a cell in ascending bead index (deterministic layout); above 8192 groups
//               of 64 cell keys k_group_scan goes before it, and with dense cells k_move
//               after it does the move
//   pair kernel DPD pair forces (src/CNTCell.cpp:1144-1555)
//               and in the same launch the bonded terms (k_bonded with the full-shell kernel):
//               bonds and angles (src/Bond.cpp:111-162, src/BondPair.cpp:138-286) summed for
//               each bonded bead, which k_advance or k_finish adds to its force
// and a last k_finish closes the final step (UpdateMom + FP64 observables).
// The simulation time lives in device memory (bumped by k_sort), so a captured
// sequence of steps replays as a hipGraph without re-capture.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "dpd_engine.h"
#include "engine_common.hpp"
#include "pair_kernels.hpp"
#include "slice_stress.hpp"

using namespace dpd;

namespace {

enum AdvanceMode { kRebin = 0, kBegin = 1, kEndBegin = 2 };

// FP64 accumulator slots per box
enum ObsSlot { O_V2 = 0, O_MOM = 3, O_VIR = 6, O_PEP = 15, O_PEB = 16, O_PEA = 17, O_N = 18 };
static_assert(O_VIR == kObsVir && O_PEP == kObsPEP, "accumulator layout");

// Bonds and angles by bonded bead: thread t of the bonded launch takes bonded[t] and evaluates
// every term that bead is in.
struct Topo {
    const int* bonded;        // bead indices with at least one bond or angle
    const int4* span;         // its bond entries [x, y) and angle entries [z, w)
    const int2* bond;         // (the other bead, bond << 1 | this bead is the tail)
    const int4* angle;        // (the other two in the order a, b, c; angle; role: 0 c, 1 b, 2 a)
    const double2* bond_par;  // (k, l0) per bond
    const double4* ang_par;   // (k, phi0, cos phi0, sin phi0)
    double4* upos;            // (batches) unwrapped position and box by bead index, kept for bonded beads
    float4* force;            // by slot: the bonded beads' sums of this step
    int nbonded;
};

struct Buffers {
    float4* pos;   // offset xyz, type | box << 8 | has bonds << 30
    float4* vel;   // velocity xyz, id bits: v at the state's time, or v + dt/2 F inside a sequence
    float4* fold;  // the uploaded force (re-binning only)
    int* bead;     // bead index (upload order) of each slot
    int4* img;     // periodic image counts xyz by bead index (not sorted; one buffer)
    int* key;      // global cell key
    uint32_t* code;   // scan code (scan_code) of the offset
};

template <bool MULTI>
__device__ inline const BoxDev& box_of(const BoxDev* boxes, const BoxDev& B0, int w)
{
    return MULTI ? boxes[bead_box(w)] : B0;
}

__device__ inline void unwrapped_pos(int slot, int bead, const Buffers& S, const BoxDev& B, double u[3])
{
    int c[3];
    key_cell(S.key[slot] - B.koff, B, c);
    const float4 p = S.pos[slot];
    const int4 a = S.img[bead];
    u[0] = (double)(c[0] + a.x * B.n[0]) * B.wd[0] + (double)p.x;
    u[1] = (double)(c[1] + a.y * B.n[1]) * B.wd[1] + (double)p.y;
    u[2] = (double)(c[2] + a.z * B.n[2]) * B.wd[2] + (double)p.z;
}

// ---------------------------------------------------------------- kernels ------

// CBond::AddForce (src/Bond.cpp:111-162) and CBondPair::AddForce of this step in FP64, summed
// over the terms of bonded bead t (bonds first, each in the order of upload) and rounded once;
// k_advance and k_finish add the sum to the bead's pair force.  OBS adds the bond virial (to the
// head bead's box, as CBond::AddForce adds its stress to the head) and the bond and angle
// potential energies, each from one of its beads (the head, the shared bead).  Bonds and angles
// never cross boxes; t0 is the workgroup's first bead, whose box receives the workgroup's sums.
// What bounds it: traffic and its latency.  Each term is evaluated once for each of its beads
// (a bond's force and its negative have the same bits), so a sum stays in registers; with a
// thread per bond and angle the forces went through memory, 160 bytes written and read for each
// bead of a chain.  Positions of a batch come unwrapped from k_sort, in bead order (the
// neighbours along a chain are the neighbouring threads' own): 64 replicas 14.0 us, with a thread
// per term 16.4, and 163 us a step where positions looked up by slot take 171.  One box's bonded
// terms run beside the pair launch and the look-ups are hidden there, k_sort's extra 36 bytes a
// bead are not (48x48x32 bilayer 48.4 us a step against 49.8).
template <bool OBS, bool MULTI, int WAVES>
__device__ __attribute__((always_inline)) inline void bonded_body(const Buffers& S, const BoxDev& B0, const Topo& T,
                                                                  const int* __restrict__ slot_of, const Sums& sums,
                                                                  int t, int t0)
{
    double ob[12];
    if (OBS)
        for (int i = 0; i < 12; ++i) ob[i] = 0.0;
    int box = -1;
    auto where = [&](int q) {
        if (MULTI) return T.upos[q];
        double u[3];
        unwrapped_pos(slot_of[q], q, S, B0, u);
        return make_double4(u[0], u[1], u[2], 0.0);
    };
    if (t < T.nbonded) {
        const int q = T.bonded[t];
        const int4 sp = T.span[t];
        const int s = slot_of[q];
        const double4 me = where(q);
        const double u[3] = {me.x, me.y, me.z};
        double F[3] = {0.0, 0.0, 0.0};
        if (OBS) box = (int)me.w;
        for (int e = sp.x; e < sp.y; ++e) {
            const int2 en = T.bond[e];
            const double2 par = T.bond_par[en.y >> 1];
            const double4 o = where(en.x);
            const bool tail = en.y & 1;
            const double x[3] = {o.x, o.y, o.z};
            double d[3];   // head - tail
            for (int a = 0; a < 3; ++a) d[a] = tail ? x[a] - u[a] : u[a] - x[a];
            const double L = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
            const double f = par.x * (par.y - L) / L;
            const double fb[3] = {f * d[0], f * d[1], f * d[2]};
            for (int a = 0; a < 3; ++a) F[a] += tail ? -fb[a] : fb[a];
            if (OBS && !tail) {
                for (int a = 0; a < 3; ++a)
                    for (int b = 0; b < 3; ++b) ob[3 * a + b] += d[b] * fb[a];
                ob[10] += 0.5 * par.x * (L - par.y) * (L - par.y);
            }
        }
        for (int e = sp.z; e < sp.w; ++e) {
            const int4 en = T.angle[e];
            const double4 par = T.ang_par[en.z];
            const double4 g = where(en.x), h = where(en.y);
            const double ug[3] = {g.x, g.y, g.z}, uh[3] = {h.x, h.y, h.z};
            double ua[3], ub[3], uc[3], f[3][3], pe = 0.0;
            for (int a = 0; a < 3; ++a) {
                ua[a] = en.w == 2 ? u[a] : ug[a];
                ub[a] = en.w == 1 ? u[a] : (en.w == 2 ? ug[a] : uh[a]);
                uc[a] = en.w == 0 ? u[a] : uh[a];
            }
            angle_forces(ua, ub, uc, par, f, OBS ? &pe : nullptr);
            for (int a = 0; a < 3; ++a) F[a] += en.w == 0 ? f[0][a] : (en.w == 1 ? f[1][a] : f[2][a]);
            if (OBS && en.w == 1) ob[11] += pe;
        }
        T.force[s] = make_float4((float)F[0], (float)F[1], (float)F[2], 0.f);
    }
    if (OBS) {
        // slots O_VIR .. O_PEA: virial (9), pair PE (untouched here), bond PE, angle PE
        const int box0 = MULTI ? (int)T.upos[T.bonded[t0]].w : 0;
        accumulate_boxes<12, WAVES>(ob, box, box0, kObsVir, sums);
    }
}

template <bool OBS, bool MULTI>
__global__ __launch_bounds__(256) void k_bonded(Buffers S, BoxDev B0, Topo T, const int* __restrict__ slot_of,
                                                Sums sums)
{
    const int t0 = blockIdx.x * blockDim.x;
    bonded_body<OBS, MULTI, 4>(S, B0, T, slot_of, sums, t0 + threadIdx.x, t0);
}

// The hit-list pair kernel and the bonded terms of the same step in one launch: the pair
// workgroups come first, the bonded workgroups after them, so the bonded work fills the CUs the
// pair kernel's last workgroups leave idle (the two write disjoint buffers).  One box.
template <bool OBS, int THREADS, int CAP, int FLUSH, int SPLIT>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(hit_waves_eu(OBS, THREADS, CAP, SPLIT))))
void k_pair_hitlist_bonded(PairArgs A, BoxDev B0, int nblocks, int per_xcd, Buffers S, Topo T,
                           const int* __restrict__ slot_of)
{
    const int npair = 8 * per_xcd;
    if ((int)blockIdx.x >= npair) {
        const int t0 = ((int)blockIdx.x - npair) * THREADS;
        bonded_body<OBS, false, THREADS / 64>(S, B0, T, slot_of, A.sums, t0 + (int)threadIdx.x, t0);
        return;
    }
    hitlist_body<OBS, false, THREADS, CAP, FLUSH, SPLIT, false>(A, B0, nblocks, per_xcd);
}

// the fused launch of hit-list schedule S
template <int S, bool OBS>
void launch_hitlist_bonded_s(const PairArgs& a, const BoxDev& B0, const Buffers& Sb, const Topo& T, const int* slot_of,
                             hipStream_t st)
{
    constexpr Schedule q = kSchedule[S];
    const int gh = (a.n + q.beads() - 1) / q.beads();
    const int ph = (gh + 7) / 8;
    const dim3 gr(8 * ph + (T.nbonded + q.threads - 1) / q.threads), bl(q.threads);
    hipLaunchKernelGGL((k_pair_hitlist_bonded<OBS, q.threads, q.cap, q.flush, q.split>), gr, bl, 0, st, a, B0, gh, ph,
                       Sb, T, slot_of);
}

template <bool OBS>
void launch_hitlist_bonded(int sched, const PairArgs& a, const BoxDev& B0, const Buffers& Sb, const Topo& T,
                           const int* slot_of, hipStream_t st)
{
    switch (sched) {
    case 1: launch_hitlist_bonded_s<1, OBS>(a, B0, Sb, T, slot_of, st); break;
    case 2: launch_hitlist_bonded_s<2, OBS>(a, B0, Sb, T, slot_of, st); break;
    case 3: launch_hitlist_bonded_s<3, OBS>(a, B0, Sb, T, slot_of, st); break;
    case 5: launch_hitlist_bonded_s<5, OBS>(a, B0, Sb, T, slot_of, st); break;
    case 6: launch_hitlist_bonded_s<6, OBS>(a, B0, Sb, T, slot_of, st); break;
    default: launch_hitlist_bonded_s<0, OBS>(a, B0, Sb, T, slot_of, st); break;
    }
}

// The bonded flag in pos.w: cleared on every slot (and the slot of every bead rewritten,
// since steps store it for flagged beads only), then set on the bonded beads' slots.
__global__ __launch_bounds__(256) void k_clear_bonded_flag(int n, float4* __restrict__ pos,
                                                           const int* __restrict__ bead, int* __restrict__ slot_of)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    pos[s].w = __int_as_float(__float_as_int(pos[s].w) & ~kBondedBit);
    slot_of[bead[s]] = s;
}

// (and, in a batch, the unwrapped positions, which k_sort keeps from then on)
__global__ __launch_bounds__(256) void k_set_bonded_flag(Topo T, const int* __restrict__ slot_of, Buffers S,
                                                         const BoxDev* boxes)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= T.nbonded) return;
    const int q = T.bonded[t], s = slot_of[q];
    const int w = __float_as_int(S.pos[s].w) | kBondedBit;
    S.pos[s].w = __int_as_float(w);
    if (!T.upos) return;
    double u[3];
    unwrapped_pos(s, q, S, boxes[bead_box(w)], u);
    T.upos[q] = make_double4(u[0], u[1], u[2], (double)bead_box(w));
}

// Close the previous step (kEndBegin) and start the next one: new cell key and rank.
// kEndBegin also adds the previous step's bond and angle forces of bonded beads (flagged in
// pos.w) to their pair force, in place: within a sequence of steps the bonded sum of every
// step but the last is left to the next step's k_advance (the last one's to k_finish).
// What bounds it: latency (the bead, its bonded sum, the cells' starts and counts one after the
// other), and with more wavefronts than the chip holds, its rounds.  Workgroups are dealt to the
// XCDs as the pair launch and k_sort deal them (48x48x32 bilayer 47.2 -> 46.3 us a step, a
// 37x23x29 box of chains 32.5 -> 31.4), and a thread takes BEADS = 2 beads, loaded together, in
// engines of more than kAdvanceOnce beads (condensate 64^3 113.7 -> 111.1, 64 replicas 161.5 ->
// 160.3; the chains' 74,000 beads, which one round holds, 32.5 -> 33.3).
constexpr int kAdvanceOnce = 8192 * 64;
template <int MODE, bool MULTI, int BEADS>
__global__ __launch_bounds__(256) void k_advance(int n, int per_xcd, Buffers S, float4* __restrict__ frc, Topo T,
                                                 const BoxDev* boxes,
                                                 BoxDev B0, Intake I, int* __restrict__ flags)
{
    const int s0 = ((blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3)) * 256 * BEADS;
    if (s0 >= n) return;
    float4 P[BEADS], V[BEADS], F[BEADS];
    int key[BEADS];
#pragma unroll
    for (int u = 0; u < BEADS; ++u) {
        const int s = min(s0 + 256 * u + (int)threadIdx.x, n - 1);
        P[u] = S.pos[s];
        V[u] = S.vel[s];
        F[u] = (MODE == kRebin) ? S.fold[s] : frc[s];
        key[u] = S.key[s];
    }
#pragma unroll
    for (int u = 0; u < BEADS; ++u) {
        const int s = s0 + 256 * u + (int)threadIdx.x;
        const bool active = s < n;
        const int from = key[u];
        int k = 0;
        if (active) {
            const float4 p = P[u];
            const BoxDev& B = box_of<MULTI>(boxes, B0, __float_as_int(p.w));
            float4 v = V[u];
            float4 f = F[u];
            if (MODE == kEndBegin && (__float_as_int(p.w) & kBondedBit)) {
                const float4 b = T.force[s];
                f.x += b.x; f.y += b.y; f.z += b.z;
                frc[s] = f;
            }
            if (MODE == kEndBegin) {
                // UpdateMom: the stored velocity is v + dt/2 F_old; k_sort repeats this sum
                v.x = kick(v.x, f.x, B.hdt);
                v.y = kick(v.y, f.y, B.hdt);
                v.z = kick(v.z, f.z, B.hdt);
                if (!(fabsf(f.x) + fabsf(f.y) + fabsf(f.z) < 1e30f) || !(fabsf(v.x) + fabsf(v.y) + fabsf(v.z) < 1e30f))
                    atomicAdd(flags + 0, 1);
            }
            int c[3];
            key_cell(from - B.koff, B, c);
            const float o[3] = {p.x, p.y, p.z};
            const int img[3] = {0, 0, 0};   // the image change is applied by k_sort
            float d[3] = {0.f, 0.f, 0.f};
            if (MODE != kRebin) {
                d[0] = drift(v.x, f.x, B);
                d[1] = drift(v.y, f.y, B);
                d[2] = drift(v.z, f.z, B);
            }
            Moved m;
            advance(o, c, img, d, B, m);
            k = B.koff + cell_key(m.c[0], m.c[1], m.c[2], B);
            if (m.jump) atomicAdd(flags + 1, 1);
            if (m.bad) atomicAdd(flags + 0, 1);
        }
        file_bead(I, from, k, s, active);
    }
}

// Exclusive scan of in[0, m) into out, in[] cleared, by one workgroup of 1024 threads: in
// rounds of kScanRound entries, wavefront w takes up to kScanChunks consecutive chunks of 64
// entries, loads all of them at once (one coalesced load per chunk, all in flight), scans each
// chunk with DPP (wave_incl_scan) in order into LDS, and the 16 wavefront totals are added in
// order through LDS.  ex: LDS of kScanRound ints.
constexpr int kScanChunks = 8;
constexpr int kScanRound = 16 * 64 * kScanChunks;
__device__ inline void scan_block(int* in, int* __restrict__ out, int m, int* ex, int* wsum, int* carry)
{
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (t == 0) *carry = 0;
    __syncthreads();
    for (int base = 0; base < m; base += kScanRound) {
        const int nch = (min(m - base, kScanRound) + 63) >> 6;   // chunks this round
        const int per = (nch + 15) >> 4;                          // chunks per wavefront
        const int ch0 = wave * per;
        int v[kScanChunks];
#pragma unroll
        for (int j = 0; j < kScanChunks; ++j) {
            const int k = base + ((ch0 + j) << 6) + lane;
            v[j] = (j < per && k < m) ? in[k] : 0;
        }
        int run = 0;
#pragma unroll
        for (int j = 0; j < kScanChunks; ++j) {
            const int incl = wave_incl_scan(v[j]);
            if (j < per) ex[((ch0 + j) << 6) + lane] = run + incl - v[j];
            run += __builtin_amdgcn_readlane(incl, 63);
        }
        if (lane == 0) wsum[wave] = run;
        __syncthreads();
        int off = *carry;
        for (int w = 0; w < wave; ++w) off += wsum[w];
        for (int j = 0; j < per; ++j) {
            const int k = base + ((ch0 + j) << 6) + lane;
            if (k < m) {
                out[k] = off + ex[((ch0 + j) << 6) + lane];
                in[k] = 0;
            }
        }
        __syncthreads();
        if (t == 0) {
            int tot = 0;
            for (int w = 0; w < 16; ++w) tot += wsum[w];
            *carry += tot;
        }
        __syncthreads();
    }
}

// exclusive scan of the scan groups' counts (one workgroup), clears the counts
__global__ __launch_bounds__(1024) void k_group_scan(int ngroups, int* __restrict__ gcnt, int* __restrict__ gstart)
{
    __shared__ int ex[kScanRound];
    __shared__ int wsum[16];
    __shared__ int carry;
    scan_block(gcnt, gstart, ngroups, ex, wsum, &carry);
}

// A bead as the sort finds it, and what it takes to move it
struct Bead {
    float4 p, v, f;
    int key;
};
struct Move {
    Buffers S, D;
    const float4* frc;
    float4* vp;
    int* slot_of;
    double4* upos;
    int write_vp;
};

template <int MODE>
__device__ inline Bead load_bead(const Move& M, int s)
{
    return Bead{M.S.pos[s], M.S.vel[s], MODE == kRebin ? M.S.fold[s] : M.frc[s], M.S.key[s]};
}

// Bead q, found as x, to slot dst of the new order under key k: repeats the advance that filed it.
template <int MODE, bool MULTI>
__device__ inline void move_bead(const Move& M, const BoxDev* boxes, const BoxDev& B0, const Bead& x, int k, int q, int dst)
{
    const Buffers &S = M.S, &D = M.D;
    const float4 p = x.p, f = x.f;
    float4 v = x.v;
    const BoxDev& B = box_of<MULTI>(boxes, B0, __float_as_int(p.w));
    if (MODE == kEndBegin) {
        // UpdateMom of the step that ends (the same sum as k_advance)
        v.x = kick(v.x, f.x, B.hdt);
        v.y = kick(v.y, f.y, B.hdt);
        v.z = kick(v.z, f.z, B.hdt);
    }
    int c[3];
    key_cell(x.key - B.koff, B, c);
    const float o[3] = {p.x, p.y, p.z};
    const int img[3] = {0, 0, 0};   // m.img is the change of image this step
    float d[3] = {0.f, 0.f, 0.f};
    if (MODE != kRebin) {
        d[0] = drift(v.x, f.x, B);
        d[1] = drift(v.y, f.y, B);
        d[2] = drift(v.z, f.z, B);
    }
    Moved m;
    advance(o, c, img, d, B, m);
    const int wd = (__float_as_int(p.w) & ~kCellXBits) | ((m.c[0] & 3) << kCellXShift);
    D.pos[dst] = make_float4(m.o[0], m.o[1], m.o[2], __int_as_float(wd));
    if (MODE == kRebin) {
        D.vel[dst] = v;
        D.fold[dst] = f;
    } else {
        // the first half of the next UpdateMom: v + dt/2 F, so the force need not be kept
        D.vel[dst] = make_float4(kick(v.x, f.x, B.hdt), kick(v.y, f.y, B.hdt), kick(v.z, f.z, B.hdt), v.w);
    }
    D.bead[dst] = q;
    // the image counts live by bead index: only a bead that crosses the box changes them,
    // and only its own thread writes them
    const bool bonded = __float_as_int(p.w) & kBondedBit, crosses = m.img[0] | m.img[1] | m.img[2];
    if ((MULTI && bonded) || crosses) {
        int4 im = S.img[q];
        im.x += m.img[0]; im.y += m.img[1]; im.z += m.img[2];
        if (crosses) S.img[q] = im;
        if (MULTI && bonded)
            M.upos[q] = make_double4((double)(m.c[0] + im.x * B.n[0]) * B.wd[0] + (double)m.o[0],
                                     (double)(m.c[1] + im.y * B.n[1]) * B.wd[1] + (double)m.o[1],
                                     (double)(m.c[2] + im.z * B.n[2]) * B.wd[2] + (double)m.o[2],
                                     (double)bead_box(wd));
    }
    D.key[dst] = k;
    D.code[dst] = scan_code(m.o, m.c, B);
    if (MODE == kRebin) {
        M.vp[dst] = v;
    } else {
        // (equal to the new velocity's bits when lambda dt = dt/2: the steps then read that)
        if (M.write_vp)
            M.vp[dst] = make_float4(kick(v.x, f.x, B.lamdt), kick(v.y, f.y, B.lamdt), kick(v.z, f.z, B.lamdt), v.w);
    }
    // the slot of each bead is read for bonded beads only (bond and angle terms); a scattered
    // 4-byte store per bead costs a partial-line write each, so the others are skipped once
    // the topology has flagged the bonded ones (an upload re-binning writes every bead)
    if (MODE == kRebin || bonded) M.slot_of[q] = dst;
}

// The counting sort and the move in one launch: workgroup g takes the 64 cell keys of scan
// group g, finds where its beads go (the counts of the groups before it, then a scan of its 64
// cells), collects them from their bins and moves them there, in every cell by ascending bead
// index: a function of the state alone (reruns, and a state downloaded and uploaded again, lay
// the beads out identically).  The move recomputes the advance that filed the bead.
// The beads before the group are gstart[g] (k_group_scan) or, with it null, the sum of gcnt.
// Clears cnt; gcnt and nspill are read by other workgroups, so those of the sort before (`clear`)
// are cleared instead.
// Groups of more than kSortList beads, or with a spill, go through `order` in global memory: a few
// of them, for engines whose groups are that full on average take the DENSE form.
// What bounds it: in small boxes the three round trips to memory (counts, bins, beads), 4.8 us
// where three launches (cell starts, placement by rank, move), each a chain of its own, took 14;
// in large ones HBM, about 110 bytes a bead: 786,432 beads 19.8 us (4.4 TB/s) against 28,
// 2,654,208 beads 56 us and 6 of k_group_scan against 82.  The spare places of the bins are
// traffic too: with 2 c + 10 places 96^3 steps took 355 us, with 2 c + 6 351, with c + 5 348.
// A workgroup takes one group: four wavefronts move its 192 beads (at three a cell) at once.
// Workgroups are dealt to the XCDs in eight contiguous ranges, as the pair launch deals beads:
// 96^3 342 us a step, dealt in turn 352.
// DENSE: no bead is moved here, but the cell of every kMoveSlots-th slot noted in `order` (k_move).
constexpr int kSortList = 1024;
constexpr int kMoveSlots = 256;
template <int MODE, bool MULTI, bool DENSE>
__global__ __launch_bounds__(256) void k_sort(int n, int ngroups, int per_xcd, Buffers S, Buffers D,
                                              const float4* __restrict__ frc, float4* __restrict__ vp,
                                              const BoxDev* boxes, BoxDev B0, Intake I, const int* __restrict__ gstart,
                                              int* __restrict__ cstart, int* __restrict__ clear,
                                              int* __restrict__ slot_of, double4* __restrict__ upos,
                                              int write_vp, int64_t* __restrict__ step, int2* __restrict__ order)
{
    __shared__ int first[kGroupKeys + 1];   // of each cell among the group's beads
    __shared__ int old[kGroupKeys];         // of each cell in the old order
    __shared__ int slot[DENSE ? 1 : kSortList], ids[DENSE ? 1 : kSortList];
    __shared__ int wsum[4], spilled;
    const int g = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (g >= ngroups) return;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, k0 = g * kGroupKeys;
    if (MODE != kRebin && g == 0 && t == 0) *step += 1;   // simulation time of the coming force evaluation
    if (w == 0) {
        const int c = I.cnt[k0 + lane];
        const int a = I.cstart[k0 + lane], b = I.cstart[k0 + lane + 1];
        old[lane] = a;
        const bool over = __any(c > bin_room(b - a));
        if (lane == 0) spilled = over;
        const int incl = wave_incl_scan(c);
        first[lane] = incl - c;
        if (lane == 63) first[kGroupKeys] = incl;
        if (c) I.cnt[k0 + lane] = 0;
    } else if (w == 1 && lane == 0) {
        clear[g] = 0;
        if (g == 0) clear[ngroups] = 0;
    }
    int p = 0;
    if (!gstart) {
        const int4* g4 = reinterpret_cast<const int4*>(I.gcnt);
#pragma unroll 4
        for (int i = t; i < g >> 2; i += 256) {
            const int4 c = g4[i];
            p += (c.x + c.y) + (c.z + c.w);
        }
        if (t < (g & 3)) p += I.gcnt[(g & ~3) + t];
    }
    p = __builtin_amdgcn_readlane(wave_incl_scan(p), 63);
    if (lane == 0) wsum[w] = p;
    __syncthreads();
    const int start = wsum[0] + wsum[1] + wsum[2] + wsum[3] + (gstart ? gstart[g] : 0);
    const int total = first[kGroupKeys];
    if (t < kGroupKeys) cstart[k0 + t] = start + first[t];
    if (g == ngroups - 1 && t == 0) cstart[ngroups * kGroupKeys] = n;
    // cell of the group's bead j
    auto cell_of = [&](int j) {
        int c = 0;
#pragma unroll
        for (int h = kGroupKeys / 2; h > 0; h >>= 1) c += first[c + h] <= j ? h : 0;
        return c;
    };
    if constexpr (DENSE) {
        int* cell = reinterpret_cast<int*>(order);
        for (int b = (start + kMoveSlots - 1) / kMoveSlots + t; b * kMoveSlots < start + total; b += 256)
            cell[b] = k0 + cell_of(b * kMoveSlots - start);
        return;
    }
    auto bin = [&](int c) { return I.bins + bin_at(old[c], k0 + c); };
    const Move M{S, D, frc, vp, slot_of, upos, write_vp};
    auto load = [&](int q) { return load_bead<MODE>(M, q); };
    auto move = [&](const Bead& x, int k, int q, int dst) { move_bead<MODE, MULTI>(M, boxes, B0, x, k, q, dst); };
    if (total <= kSortList && !spilled) {
        // the first 256 beads are loaded before their indices are exchanged
        Bead b0;
        int c0 = 0;
        if (t < total) {
            c0 = cell_of(t);
            const int s = bin(c0)[t - first[c0]];
            ids[t] = S.bead[s];
            b0 = load(s);
        }
        for (int j = t + 256; j < total; j += 256) {
            const int c = cell_of(j);
            slot[j] = bin(c)[j - first[c]];
            ids[j] = S.bead[slot[j]];
        }
        __syncthreads();
        auto place = [&](int c, int q) {
            int r = 0;
            for (int e = first[c]; e < first[c + 1]; ++e) r += ids[e] < q;
            return start + first[c] + r;
        };
        if (t < total) move(b0, k0 + c0, ids[t], place(c0, ids[t]));
        for (int j = t + 256; j < total; j += 256) {
            const int c = cell_of(j);
            move(load(slot[j]), k0 + c, ids[j], place(c, ids[j]));
        }
        return;
    }
    int2* list = order + start;   // (bead index, source slot)
    for (int j = t; j < total; j += 256) {
        const int c = cell_of(j), r = j - first[c];
        if (r >= bin_room(I.cstart[k0 + c + 1] - old[c])) continue;
        const int s = bin(c)[r];
        list[j] = make_int2(S.bead[s], s);
    }
    for (int i = t, m = spilled ? min(*I.nspill, I.cap) : 0; i < m; i += 256) {
        const int4 x = I.spill[i];
        if ((x.x >> 6) == g) list[first[x.x & 63] + x.y] = make_int2(S.bead[x.z], x.z);
    }
    __threadfence_block();
    __syncthreads();
    for (int j = t; j < total; j += 256) {
        const int c = cell_of(j);
        const int2 x = list[j];
        int r = 0;
        for (int e = first[c]; e < first[c + 1]; ++e) r += list[e].x < x.x;
        move(load(x.y), k0 + c, x.x, start + first[c] + r);
    }
}

// The move for engines of dense cells, after k_sort's cell starts: a workgroup takes kMoveSlots
// slots of the new order, whatever cells these belong to.  It collects the bead indices of their
// cells (the first and the last reach past its slots) tile by tile in LDS, and each thread counts
// those below its bead's.
// What bounds it: the round trips (cells, bins, bead indices) and, in cells of hundreds, the
// counting.  A step of 81,000 beads in 10^3 cells of width 3 takes 156 us, 136 of them the pair
// launch (318 where each scan group's workgroup moves its 5,000 beads alone, one round trip after
// the other), 41,472 in 6^3 of width 4 264 us (1,053), the same in 3^3 of width 8 2.5 ms (20.4).
constexpr int kMoveTile = 1024;
template <int MODE, bool MULTI>
__global__ __launch_bounds__(kMoveSlots) void k_move(int n, int nkeys, int nblocks, int per_xcd, Move M,
                                                     const BoxDev* boxes, BoxDev B0, Intake I,
                                                     const int* __restrict__ cstart, const int* __restrict__ cell)
{
    __shared__ int ids[kMoveTile], src[kMoveSlots];
    __shared__ int last, over;
    const int blk = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (blk >= nblocks) return;
    const int t = threadIdx.x, d0 = blk * kMoveSlots, d1 = min(n, d0 + kMoveSlots), j = min(d0 + t, d1 - 1);
    const bool active = d0 + t < d1;
    // the cell k of slot j: the last one that starts at it or before
    const int kl = cell[blk];
    int k = kl;
    for (int hi = d1 < n ? cell[blk + 1] : nkeys - 1; k < hi;) {
        const int mid = (k + hi + 1) >> 1;
        if (cstart[mid] <= j) k = mid;
        else hi = mid - 1;
    }
    const int c0 = cstart[k], c1 = cstart[k + 1];
    // the source of the bead of rank r in cell q's bin (-1: spilled)
    auto in_bin = [&](int q, int r) {
        const int a = I.cstart[q];
        return r < bin_room(I.cstart[q + 1] - a) ? I.bins[bin_at(a, q) + r] : -1;
    };
    // f(slot, source) of the spilled beads that belong to slots [a, b)
    auto spilled = [&](int a, int b, const auto& f) {
        for (int i = t, m = min(*I.nspill, I.cap); i < m; i += kMoveSlots) {
            const int4 x = I.spill[i];
            const int s = cstart[x.x] + x.y;
            if (s >= a && s < b) f(s, x.z);
        }
        __syncthreads();
    };
    if (t == 0) over = 0;
    if (d0 + t == d1 - 1) last = k;
    __syncthreads();
    if (active) {
        const int s = in_bin(k, j - c0);
        src[t] = s;
        if (s < 0) over = 1;
    }
    __syncthreads();
    if (over) spilled(d0, d1, [&](int s, int from) { src[s - d0] = from; });
    const int s = src[j - d0];
    const Bead x = load_bead<MODE>(M, s);
    const int q = M.S.bead[s];
    const int kr = last, e0 = cstart[kl], e1 = cstart[kr + 1], l0 = e0, r0 = cstart[kr];
    int rank = 0;
    for (int a = e0; a < e1; a += kMoveTile) {
        const int b = min(a + kMoveTile, e1);
        __syncthreads();   // ids and over are read no more
        if (t == 0) over = 0;
        __syncthreads();
        for (int i = a + t; i < b; i += kMoveSlots) {
            const int from = i < d0 ? in_bin(kl, i - l0) : (i < d1 ? src[i - d0] : in_bin(kr, i - r0));
            if (from < 0) over = 1;
            else ids[i - a] = M.S.bead[from];
        }
        __syncthreads();
        if (over) spilled(a, b, [&](int i, int from) { ids[i - a] = M.S.bead[from]; });
        for (int i = max(a, c0); i < min(b, c1); ++i) rank += ids[i - a] < q;
    }
    if (active) move_bead<MODE, MULTI>(M, boxes, B0, x, k, q, c0 + rank);
}

// REBIN leaves the uploaded force in fold; the canonical state needs it in frc too
__global__ void k_copy_force(int n, const float4* __restrict__ fold, float4* __restrict__ frc)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n) frc[s] = fold[s];
}

// Close the last step: the bonded beads' sums added to their force, UpdateMom (UPDATE_V) and
// the FP64 sums of v^2 and momentum (the virial and energies come from the pair and
// bonded kernels).
template <bool UPDATE_V, bool OBS, bool MULTI>
__global__ __launch_bounds__(256) void k_finish(int n, Buffers S, float4* __restrict__ frc, Topo T,
                                                const BoxDev* boxes, BoxDev B0, int* __restrict__ flags,
                                                Sums sums, float4* __restrict__ vp_keep)
{
    static_assert(O_V2 == 0 && O_MOM == 3, "kinetic slots first");
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    double ob[6];
    if (OBS)
        for (int i = 0; i < 6; ++i) ob[i] = 0.0;
    int box = -1;
    if (s < n) {
        const int w = __float_as_int(S.pos[s].w);
        box = bead_box(w);
        const BoxDev& B = box_of<MULTI>(boxes, B0, w);
        float4 f = frc[s];
        float4 v = S.vel[s];
        if (T.nbonded > 0 && (w & kBondedBit)) {
            const float4 b = T.force[s];
            f.x += b.x; f.y += b.y; f.z += b.z;
            frc[s] = f;
        }
        if (UPDATE_V) {
            // the last step's predicted velocity, which the steps read from vel (vp_is_vel)
            if (vp_keep) vp_keep[s] = v;
            // the second half of UpdateMom (the stored velocity is v + dt/2 F_old)
            v.x = kick(v.x, f.x, B.hdt);
            v.y = kick(v.y, f.y, B.hdt);
            v.z = kick(v.z, f.z, B.hdt);
            S.vel[s] = v;
        }
        if (!(fabsf(f.x) + fabsf(f.y) + fabsf(f.z) < 1e30f) || !(fabsf(v.x) + fabsf(v.y) + fabsf(v.z) < 1e30f))
            atomicAdd(flags + 0, 1);
        if (OBS) {
            ob[O_V2 + 0] = (double)v.x * v.x;
            ob[O_V2 + 1] = (double)v.y * v.y;
            ob[O_V2 + 2] = (double)v.z * v.z;
            ob[O_MOM + 0] = v.x;
            ob[O_MOM + 1] = v.y;
            ob[O_MOM + 2] = v.z;
        }
    }
    if (OBS) {
        const int box0 = MULTI ? bead_box(__float_as_int(S.pos[blockIdx.x * blockDim.x].w)) : 0;
        accumulate_boxes<6>(ob, MULTI ? box : (s < n ? 0 : -1), box0, 0, sums);
    }
}

// FP64 sums per box of v and v^2 and the bead count, slots 0..4
template <bool MULTI>
__global__ __launch_bounds__(256) void k_mom_sums(int n, Buffers S, Sums sums)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    double ob[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    int box = -1;
    if (s < n) {
        box = MULTI ? bead_box(__float_as_int(S.pos[s].w)) : 0;
        const float4 v = S.vel[s];
        ob[0] = v.x; ob[1] = v.y; ob[2] = v.z;
        ob[3] = (double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z;
        ob[4] = 1.0;
    }
    const int box0 = MULTI ? bead_box(__float_as_int(S.pos[blockIdx.x * blockDim.x].w)) : 0;
    accumulate_boxes<5>(ob, box, box0, 0, sums);
}

// v <- (v - shift) * scale with adj[box] = (shift x, y, z, scale), in FP64
template <bool MULTI>
__global__ __launch_bounds__(256) void k_mom_apply(int n, Buffers S, const double4* __restrict__ adj)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int box = MULTI ? bead_box(__float_as_int(S.pos[s].w)) : 0;
    const double4 a = adj[box];
    float4 v = S.vel[s];
    v.x = (float)(((double)v.x - a.x) * a.w);
    v.y = (float)(((double)v.y - a.y) * a.w);
    v.z = (float)(((double)v.z - a.z) * a.w);
    S.vel[s] = v;
}

// state back to upload order in FP64 (of x, u, v, f those that are not null)
template <bool MULTI>
__global__ __launch_bounds__(256) void k_gather(int n, Buffers S, const float4* __restrict__ frc,
                                                const BoxDev* boxes, BoxDev B0, double* __restrict__ x,
                                                double* __restrict__ u, double* __restrict__ v,
                                                double* __restrict__ f)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int64_t q = S.bead[s];
    if (x || u) {
        const float4 p = S.pos[s];
        const BoxDev& B = box_of<MULTI>(boxes, B0, __float_as_int(p.w));
        int c[3];
        key_cell(S.key[s] - B.koff, B, c);
        const int4 a = u ? S.img[q] : make_int4(0, 0, 0, 0);
        const double o[3] = {p.x, p.y, p.z};
        const int im[3] = {a.x, a.y, a.z};
        for (int d = 0; d < 3; ++d) {
            const double xa = (double)c[d] * B.wd[d] + o[d];
            if (x) x[3 * q + d] = xa;
            if (u) u[3 * q + d] = xa + (double)im[d] * (double)B.n[d] * B.wd[d];
        }
    }
    if (v) {
        const float4 vv = S.vel[s];
        v[3 * q + 0] = vv.x; v[3 * q + 1] = vv.y; v[3 * q + 2] = vv.z;
    }
    if (f) {
        const float4 ff = frc[s];
        f[3 * q + 0] = ff.x; f[3 * q + 1] = ff.y; f[3 * q + 2] = ff.z;
    }
}

// The end of a call: its flags and (with hacc) the sums of box blockIdx.x to page-locked host
// memory, and both cleared for the next call (they are zero at rest, so that a call starts with
// its first kernel and a captured graph needs no clearing).  What bounds it, and a call of few
// steps: the host's round trip.  With two clearing launches before the steps and a copy to
// pageable memory after them, a second one for the sums, a call of one step in a 37x23x29 box of
// chains took 104 us, of which 48 were kernels; it takes 66.
__global__ __launch_bounds__(64) void k_report(Sums S, int* __restrict__ flags, double* __restrict__ hacc,
                                               int* __restrict__ hflags)
{
    const int t = threadIdx.x, i = t & (kObsStride - 1);
    if (hacc) {
        double* a = S.acc + (size_t)blockIdx.x * (S.spread + 1) * kObsStride;
        double s = 0.0;
        for (int r = t / kObsStride; r <= S.spread; r += 64 / kObsStride) {
            s += a[r * kObsStride + i];
            a[r * kObsStride + i] = 0.0;
        }
        s += __shfl_down(s, kObsStride, 64);
        if (t < kObsStride) hacc[(size_t)blockIdx.x * kObsStride + i] = s;
    }
    if (blockIdx.x == 0 && t < 4) {
        hflags[t] = flags[t];
        flags[t] = 0;
    }
}

// clears a table (a kernel rather than a memset, so that it can sit inside a captured graph)
__global__ void k_zero(double* tab, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) tab[i] = 0.0;
}

__global__ void k_set_step(int64_t* step, int64_t value)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *step = value;
}

}  // namespace

// ------------------------------------------------------------------ host side ---

struct BoxHost {
    dpd_params p{};
    std::vector<double> a, g;
    bool thermostat_on = true, conservative_on = true;
    bool forces_on = true;   // ToggleDPDBeadForces: off zeroes the half-step constants
    double dt = 0, lambda = 0, kT = 0;
    BoxDev B{};
    // staged beads and topology (box-local indices)
    int64_t n = 0;
    std::vector<int32_t> id, type;
    std::vector<double> x, u, v, f;
    bool has_f = false;
    std::vector<int32_t> bh, bt, pf, ps;
    std::vector<double> bk, bl0, pk, pphi;
    // what the device holds of it, which is not what is staged until the next commit: its beads
    // from bead_off on, its bonds and bond pairs from bond_off and pair_off on
    int64_t bead_off = 0, nbeads = 0;
    int bond_off = 0, nbonds = 0, pair_off = 0, npairs = 0;
};

struct dpd_engine {
    std::vector<BoxHost> boxes;
    int device = 0;
    hipStream_t stream = nullptr;
    int ngroups = 0, nkeys = 0;   // scan groups of 64 keys, keys (all boxes)
    int64_t n = 0;
    int64_t step = 0;
    int cur = 0;
    int pair_kernel = DPD_PAIR_FULLSHELL;   // the kernel of schedule `sched`
    int sched = kFullShellSchedule;         // pair-launch schedule (kSchedule)
    bool pair_auto = false;   // choose by bead count at each commit
    bool committed = false;
    // device buffers
    char *per_box = nullptr, *per_bead = nullptr;   // what the arrays by box and by bead lie in
    BoxDev* dboxes = nullptr;
    float4 *pos[2] = {}, *vel[2] = {}, *fold[2] = {};
    int* bead[2] = {};
    int4* img = nullptr;   // periodic image counts by bead index
    int* key[2] = {};
    uint32_t* code[2] = {};   // n + kCodePad: the hit-list scan reads up to 7 slots past the end
    float4 *frc = nullptr, *vp = nullptr;
    int* slot_of = nullptr;
    // counting sort (Intake); cstart[cur] are the cell starts of buffer cur, counts[cur]
    // (beads per scan group | spills) belong to the sort out of it and are zero at rest
    // (all per cell key or group in `cells`, per bead in `filed`)
    int *cstart[2] = {}, *counts[2] = {}, *cnt = nullptr, *gstart = nullptr, *bins = nullptr;
    int4 *spill = nullptr, *filed = nullptr;
    int2* order = nullptr;
    int* cells = nullptr;
    size_t cleared = 0;   // ints of `cells` (cnt and counts) that are zero at rest
    int* flags = nullptr;
    int64_t* dstep = nullptr;   // the simulation time, and that of dpd_compute_forces
    double* acc = nullptr;      // Sums, zero at rest as the flags are
    double* hacc = nullptr;     // page-locked: a call's sums per box, then its flags
    int* hflags = nullptr;
    float* table = nullptr;
    double* gather = nullptr;   // 12n doubles for downloads
    double* slice = nullptr;    // slice stress tables (pair | bond)
    double4* madj = nullptr;    // per-box velocity shift and scale
    int4* hitblk[kSchedules] = {};   // hit-list workgroups of a batch (box, first slot, end slot)
    int nhitblk[kSchedules] = {};    // per schedule (its beads per workgroup)
    size_t slice_cap = 0;
    // topology
    int2 *bond_bead = nullptr, *bond_ent = nullptr;
    int4 *ang_bead = nullptr, *ang_ent = nullptr, *span = nullptr;
    double2* bond_par = nullptr;
    double4 *ang_par = nullptr, *upos = nullptr;
    float4* bforce = nullptr;
    int* bonded = nullptr;
    int nbonds = 0, nangles = 0, nbonded = 0;
    // observables
    std::vector<dpd_obs> obs;
    bool obs_valid = false;
    int64_t jumps = 0;
    // graphs (steps, observe | current buffer << 1) -> executable graph; valid while buffers stay put
    std::map<std::pair<int64_t, int>, hipGraphExec_t> graphs;
    std::map<std::pair<int64_t, int>, hipGraph_t> graph_src;
    // timing
    hipEvent_t ev[2] = {};
    std::vector<hipEvent_t> pev;
    double t_total = 0, t_pair = 0;
    int64_t n_pair = 0;
    std::string err;
};

namespace {

int fail(dpd_engine* e, int code, const std::string& msg)
{
    if (e) e->err = msg;
    return code;
}

#define HIPCHK(expr)                                                                       \
    do {                                                                                   \
        hipError_t _st = (expr);                                                           \
        if (_st != hipSuccess)                                                             \
            return fail(e, DPD_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(_st)); \
    } while (0)

template <class T>
int dalloc(dpd_engine* e, T** p, size_t count)
{
    if (*p) { (void)hipFree(*p); *p = nullptr; }
    if (count == 0) count = 1;
    hipError_t st = hipMalloc((void**)p, sizeof(T) * count);
    if (st != hipSuccess) return fail(e, DPD_ERR_OOM, std::string("hipMalloc: ") + hipGetErrorString(st));
    return DPD_OK;
}

// several arrays in one allocation, each on a 256-byte boundary
struct Part {
    void** p;
    size_t bytes;
};
template <class T>
Part part(T** p, size_t count) { return {(void**)p, (sizeof(T) * count + 255) / 256 * 256}; }
int dalloc_parts(dpd_engine* e, char** block, const std::vector<Part>& parts)
{
    size_t total = 0;
    for (const Part& q : parts) total += q.bytes;
    if (int rc = dalloc(e, block, total)) return rc;
    char* at = *block;
    for (const Part& q : parts) {
        *q.p = at;
        at += q.bytes;
    }
    return DPD_OK;
}

// With lambda = 1/2 and the forces on, the predicted velocity v + lambda dt f and the stored
// half step v + dt/2 f are the same FP32 expression (lambda dt and dt/2 round to the same
// float): steps then read the predicted velocities from vel, k_sort does not write vp, and
// k_finish keeps the last step's in vp for the calls between steps.
inline bool vp_is_vel(const dpd_engine* e)
{
    for (const auto& b : e->boxes)
        if (!(b.B.hdt == b.B.lamdt)) return false;
    return true;
}

void drop_graphs(dpd_engine* e)
{
    for (auto& g : e->graphs) (void)hipGraphExecDestroy(g.second);
    for (auto& g : e->graph_src) (void)hipGraphDestroy(g.second);
    e->graphs.clear();
    e->graph_src.clear();
}

// switch the pair launch to schedule `s` (captured graphs hold the old launch)
void set_schedule(dpd_engine* e, int s)
{
    if (s != e->sched) drop_graphs(e);
    e->sched = s;
    e->pair_kernel = kSchedule[s].kernel;
}

// the automatic choice: the hit-list kernel's schedule for the engine's size where its slots
// fit the 26-bit list entries, the full-shell kernel beyond
int default_schedule(const dpd_engine* e)
{
    return e->n <= (int64_t)kHitSlotMask ? size_schedule(e->n, e->nbonded > 0) : kFullShellSchedule;
}

// the automatic choice again, where the beads or the topology have changed
void auto_schedule(dpd_engine* e)
{
    if (e->pair_auto) set_schedule(e, default_schedule(e));
}

void set_step_constants(BoxHost& b)
{
    // CCNTCell::SetTimeStepConstants / ChangeTimeStepConstants (src/CNTCell.cpp:180-203, :357-377)
    // CCNTCell::ToggleDPDBeadForces (src/CNTCell.cpp:223-227) passes dt = 0 for the two
    // half-step constants: forces no longer move beads or change velocities
    const double hdt = b.forces_on ? b.dt : 0.0;
    b.B.dt = (float)b.dt;
    b.B.hdt = (float)(0.5 * hdt);
    b.B.hdt2 = (float)(0.5 * hdt * hdt);
    b.B.lamdt = (float)(b.lambda * b.dt);
    b.B.invrootdt = (float)std::sqrt(24.0 * b.kT / b.dt);
}

int check_params(dpd_engine* e, const dpd_params* p)
{
    if (p->nx < 3 || p->ny < 3 || p->nz < 3) return fail(e, DPD_ERR_PARAM, "need at least 3 cells per axis");
    if ((int64_t)p->nx * p->ny * p->nz > (int64_t)1 << 24)
        return fail(e, DPD_ERR_PARAM, "more than 2^24 cells in one box");
    if (p->wx < 1.0 || p->wy < 1.0 || p->wz < 1.0) return fail(e, DPD_ERR_PARAM, "cell widths must be >= 1");
    if (p->ntypes < 1 || p->ntypes > DPD_MAX_TYPES) return fail(e, DPD_ERR_PARAM, "ntypes out of range");
    if (!(p->dt > 0.0) || p->lambda < 0.0 || p->lambda > 1.0 || p->kT < 0.0)
        return fail(e, DPD_ERR_PARAM, "invalid dt, lambda or kT");
    if (!p->a || !p->gamma) return fail(e, DPD_ERR_PARAM, "null interaction matrices");
    const int nt = p->ntypes;
    for (int i = 0; i < nt; ++i)
        for (int j = 0; j < nt; ++j)
            if (p->a[i * nt + j] != p->a[j * nt + i] || p->gamma[i * nt + j] != p->gamma[j * nt + i] ||
                p->gamma[i * nt + j] < 0.0)
                return fail(e, DPD_ERR_PARAM, "interaction matrices must be symmetric, gamma >= 0");
    return DPD_OK;
}

int upload_tables(dpd_engine* e)
{
    const int nb = (int)e->boxes.size();
    std::vector<float> t((size_t)nb * kTableStride, 0.0f);
    for (int b = 0; b < nb; ++b) {
        const BoxHost& h = e->boxes[b];
        const int nt = h.p.ntypes;
        float* tb = t.data() + (size_t)b * kTableStride;
        for (int i = 0; i < nt; ++i)
            for (int j = 0; j < nt; ++j) {
                const double a = h.conservative_on ? h.a[i * nt + j] : 0.0;
                const double g = h.thermostat_on ? h.g[i * nt + j] : 0.0;
                tb[i * kMaxTypes + j] = (float)a;
                tb[kTypeStride + i * kMaxTypes + j] = (float)g;
                tb[2 * kTypeStride + i * kMaxTypes + j] = (float)std::sqrt(g);
            }
    }
    HIPCHK(hipMemcpyAsync(e->table, t.data(), sizeof(float) * t.size(), hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    return DPD_OK;
}

int upload_boxes(dpd_engine* e)
{
    std::vector<BoxDev> bd;
    for (auto& b : e->boxes) bd.push_back(b.B);
    HIPCHK(hipMemcpyAsync(e->dboxes, bd.data(), sizeof(BoxDev) * bd.size(), hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    return DPD_OK;
}

Buffers bufs(dpd_engine* e, int i)
{
    return Buffers{e->pos[i], e->vel[i], e->fold[i], e->bead[i], e->img, e->key[i], e->code[i]};
}

Topo topo(dpd_engine* e)
{
    return Topo{e->bonded, e->span, e->bond_ent, e->ang_ent, e->bond_par, e->ang_par, e->upos, e->bforce, e->nbonded};
}

inline Sums sums(const dpd_engine* e) { return Sums{e->acc, (int)e->boxes.size() <= kSpreadBoxes ? kSpread : 0}; }

// where an evaluation beside the trajectory leaves its force (scratch between calls)
inline float4* aside_force(dpd_engine* e) { return e->fold[e->cur ^ 1]; }

inline int grid(int64_t n, int b) { return (int)((n + b - 1) / b); }
inline bool multi(dpd_engine* e) { return e->boxes.size() > 1; }

// the intake of the sort out of buffer `cur`
Intake intake(dpd_engine* e)
{
    int* c = e->counts[e->cur];
    return Intake{e->cstart[e->cur], e->bins, e->cnt, c, e->spill, c + e->ngroups, (int)e->n};
}

// the sort's counts to zero where steps have not left them so (outside captured sequences)
int clear_counts(dpd_engine* e)
{
    HIPCHK(hipMemsetAsync(e->cells, 0, sizeof(int) * e->cleared, e->stream));
    return DPD_OK;
}

template <int MODE, bool MULTI, int BEADS>
void launch_advance(dpd_engine* e, const Buffers& S, const Intake& I)
{
    const int n = (int)e->n, per = grid(n, 8 * 256 * BEADS);
    hipLaunchKernelGGL((k_advance<MODE, MULTI, BEADS>), dim3(8 * per), dim3(256), 0, e->stream, n, per, S, e->frc,
                       topo(e), e->dboxes, e->boxes[0].B, I, e->flags);
}

// counting sort of buffer `cur` into buffer `cur^1`; MODE decides the move.  `advanced`: the
// previous pair launch's epilogue already closed the step and filed the beads (MODE kEndBegin
// only), so k_advance is left out.
// Up to kDirectGroups groups every workgroup of k_sort adds up the counts before its own; with
// more the sum, quadratic in all, costs more than a launch of one workgroup that scans them
// (a step of 4,096 groups 122.2 us, with the scan 123.7; of 13,824 355 us, with the scan 342).
constexpr int kDirectGroups = 8192;
// Above kDenseGroup beads a group on average (wide cells, or many beads in few of them) k_sort
// leaves the move to k_move, which spreads it over the chip by slots.  Microseconds a step moved
// by groups and by slots, water at density 3: 192 beads a group (unit cells, 24,000 beads) 22.9,
// 26.1; 862 (186,000 beads) 64.1, 61.2, (862,000) 165.7, 170.4; 1,029 (222,000) 83.3, 73.3; 1,536
// (98,000) 99.3, 79.1, (786,000) 229, 210.
constexpr int kDenseGroup = 896;
template <int MODE, bool MULTI>
void sort_step_t(dpd_engine* e, bool advanced)
{
    const int n = (int)e->n;
    Buffers S = bufs(e, e->cur), D = bufs(e, e->cur ^ 1);
    const BoxDev B0 = e->boxes[0].B;
    const Intake I = intake(e);
    if (!advanced)
        n > kAdvanceOnce ? launch_advance<MODE, MULTI, 2>(e, S, I) : launch_advance<MODE, MULTI, 1>(e, S, I);
    const bool scan = e->ngroups > kDirectGroups;
    if (scan) hipLaunchKernelGGL(k_group_scan, dim3(1), dim3(1024), 0, e->stream, e->ngroups, I.gcnt, e->gstart);
    const int per = grid(e->ngroups, 8), write_vp = (MODE == kRebin || !vp_is_vel(e)) ? 1 : 0;
    const int *gstart = scan ? e->gstart : nullptr;
    int *cstart = e->cstart[e->cur ^ 1], *clear = e->counts[e->cur ^ 1];
    const dim3 gr(8 * per), bl(256);
    if (n > (int64_t)kDenseGroup * e->ngroups) {
        hipLaunchKernelGGL((k_sort<MODE, MULTI, true>), gr, bl, 0, e->stream, n, e->ngroups, per, S, D, e->frc, e->vp,
                           e->dboxes, B0, I, gstart, cstart, clear, e->slot_of, e->upos, write_vp, e->dstep, e->order);
        const Move M{S, D, e->frc, e->vp, e->slot_of, e->upos, write_vp};
        const int nb = grid(n, kMoveSlots), pm = grid(nb, 8);
        hipLaunchKernelGGL((k_move<MODE, MULTI>), dim3(8 * pm), dim3(kMoveSlots), 0, e->stream, n, e->nkeys, nb, pm, M,
                           e->dboxes, B0, I, cstart, reinterpret_cast<const int*>(e->order));
    } else {
        hipLaunchKernelGGL((k_sort<MODE, MULTI, false>), gr, bl, 0, e->stream, n, e->ngroups, per, S, D, e->frc, e->vp,
                           e->dboxes, B0, I, gstart, cstart, clear, e->slot_of, e->upos, write_vp, e->dstep, e->order);
    }
    e->cur ^= 1;
}

template <int MODE>
int sort_step(dpd_engine* e, bool advanced = false)
{
    if (multi(e)) sort_step_t<MODE, true>(e, advanced);
    else sort_step_t<MODE, false>(e, advanced);
    HIPCHK(hipGetLastError());
    return DPD_OK;
}

// Whether the pair launch of a step that another follows carries the step's epilogue: for
// engines without bonded terms.  (With them, the bonded beads would need their own pass once
// the bond and angle forces are known: measured on the condensate box, the epilogue added
// 14 us to the pair launch and that pass took 20 us, against the 25 us of k_advance it
// replaced.)
inline bool epilogue_ok(const dpd_engine* e) { return e->nbonded == 0 && epilogue_available(e->sched, e->n, e->ngroups); }

// Pair forces of this step.  With the hit-list kernel the bond and angle terms run in the
// same launch (k_pair_hitlist_bonded); `bonded` then tells that they are done.
// `epi` (epilogue_ok): the launch also closes the step and starts the next one (pair_epilogue).
// `spills` false: the launch is repeated on one state, and what overfills the sort's bins is dropped.
// `aside`: an evaluation beside the trajectory, force to aside_force(e), time from dstep[1].
int launch_pair(dpd_engine* e, bool obs, bool* bonded = nullptr, bool epi = false, bool in_seq = false,
                bool spills = true, bool aside = false)
{
    if (bonded) *bonded = false;
    PairArgs a;
    const Buffers S = bufs(e, e->cur);
    a.vel = S.vel;
    a.intake = intake(e);
    if (!spills) a.intake.cap = 0;
    a.flags = e->flags;
    a.n = (int)e->n;
    a.nbox = (int)e->boxes.size();
    a.ngroups = e->ngroups;
    a.boxes = e->dboxes;
    a.pos = e->pos[e->cur];
    // inside a sequence of steps with lambda dt = dt/2 the predicted velocities are the
    // stored half steps (k_sort did not write vp)
    a.vp = (in_seq && vp_is_vel(e)) ? e->vel[e->cur] : e->vp;
    a.key = e->key[e->cur];
    a.code = S.code;
    a.cstart = e->cstart[e->cur];
    a.table = e->table;
    a.step = e->dstep + (aside ? 1 : 0);
    a.frc = aside ? aside_force(e) : e->frc;
    a.sums = sums(e);
    a.hitblk = e->hitblk[e->sched];
    a.nhitblk = e->nhitblk[e->sched];
    // one box only: a batch's pair kernel leaves no registers for the bonded terms (held to its 96
    // it spills 18: 202 us a step of 64 replicas, 163 with the bonded terms in their own launch)
    if (bonded && e->nbonded > 0 && e->pair_kernel == DPD_PAIR_HITLIST && hitlist_fits(a.n, a.ngroups) && !multi(e)) {
        // (never with the epilogue: epilogue_ok excludes engines with bonded terms)
        const BoxDev B0 = e->boxes[0].B;
        const Topo T = topo(e);
        if (obs) launch_hitlist_bonded<true>(e->sched, a, B0, S, T, e->slot_of, e->stream);
        else launch_hitlist_bonded<false>(e->sched, a, B0, S, T, e->slot_of, e->stream);
        *bonded = true;
        return hipGetLastError() == hipSuccess ? DPD_OK : fail(e, DPD_ERR_HIP, "pair kernel launch failed");
    }
    return launch_pair_kernel(e->sched, a, e->boxes[0].B, obs, e->stream, epi) == hipSuccess
               ? DPD_OK
               : fail(e, DPD_ERR_HIP, "pair kernel launch failed");
}

template <bool UPDATE_V, bool OBS>
void launch_finish(dpd_engine* e, float4* frc)
{
    const int n = (int)e->n;
    const BoxDev B0 = e->boxes[0].B;
    float4* keep = (UPDATE_V && vp_is_vel(e)) ? e->vp : nullptr;
    if (multi(e))
        hipLaunchKernelGGL((k_finish<UPDATE_V, OBS, true>), dim3(grid(n, 256)), dim3(256), 0, e->stream, n,
                           bufs(e, e->cur), frc, topo(e), e->dboxes, B0, e->flags, sums(e), keep);
    else
        hipLaunchKernelGGL((k_finish<UPDATE_V, OBS, false>), dim3(grid(n, 256)), dim3(256), 0, e->stream, n,
                           bufs(e, e->cur), frc, topo(e), e->dboxes, B0, e->flags, sums(e), keep);
}

// bonds and angles of this step, where the pair launch did not run them
template <bool OBS>
void launch_bonded(dpd_engine* e)
{
    if (e->nbonded == 0) return;
    const dim3 gr(grid(e->nbonded, 256)), bl(256);
    const Buffers S = bufs(e, e->cur);
    const BoxDev B0 = e->boxes[0].B;
    if (multi(e)) hipLaunchKernelGGL((k_bonded<OBS, true>), gr, bl, 0, e->stream, S, B0, topo(e), e->slot_of, sums(e));
    else hipLaunchKernelGGL((k_bonded<OBS, false>), gr, bl, 0, e->stream, S, B0, topo(e), e->slot_of, sums(e));
}

// the end of a call: waits for it, takes its flags and (`obs`) its sums to hacc
int report(dpd_engine* e, bool obs)
{
    hipLaunchKernelGGL(k_report, dim3(obs ? e->boxes.size() : 1), dim3(64), 0, e->stream, sums(e), e->flags,
                       obs ? e->hacc : nullptr, e->hflags);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(e->stream));
    e->jumps += e->hflags[1];
    if (e->hflags[0]) return fail(e, DPD_ERR_NAN, "non-finite force, velocity or position detected");
    return DPD_OK;
}

int finish_obs(dpd_engine* e)
{
    const size_t nb = e->boxes.size();
    e->obs.assign(nb, dpd_obs{});
    for (size_t b = 0; b < nb; ++b) {
        const double* a = e->hacc + b * kObsStride;
        const dpd_params& p = e->boxes[b].p;
        dpd_obs& o = e->obs[b];
        o.step = e->step;
        o.nbeads = e->boxes[b].nbeads;
        const double V = (double)p.nx * p.wx * (double)p.ny * p.wy * (double)p.nz * p.wz;
        for (int d = 0; d < 3; ++d) { o.sum_v2[d] = a[O_V2 + d]; o.momentum[d] = a[O_MOM + d]; }
        for (int i = 0; i < 9; ++i) o.stress[i] = a[O_VIR + i] / V;
        const double v2 = o.sum_v2[0] + o.sum_v2[1] + o.sum_v2[2];
        o.kT = o.nbeads ? v2 / (3.0 * (double)o.nbeads) : 0.0;
        // src/Monitor.cpp:981-982 keeps the 10-digit constant
        o.pressure = 0.3333333333 * (1.0 / V) * (v2 + a[O_VIR + 0] + a[O_VIR + 4] + a[O_VIR + 8]);
        o.pe_pair = a[O_PEP];
        o.pe_bond = a[O_PEB];
        o.pe_angle = a[O_PEA];
        o.jumps = e->jumps;
    }
    e->obs_valid = true;
    return DPD_OK;
}

// the steps of one dpd_step call, enqueued on the stream (capturable)
// steps whose pair launch is bracketed by events: every step, or the last of every
// kTimingStride with DPD_STEP_TIMING_SAMPLED (never the first step of a call, whose
// launch follows the host's enqueue rather than the previous step)
constexpr int64_t kTimingStride = 16;
inline bool timed_step(int64_t t, int timing)
{
    return timing == 1 || (timing == 2 && t % kTimingStride == kTimingStride - 1);
}
inline int64_t timed_steps(int64_t nsteps, int timing)
{
    return timing == 1 ? nsteps : (timing == 2 ? nsteps / kTimingStride : 0);
}

// timing: 0 none, 1 every pair launch, 2 every kTimingStride-th
int enqueue_steps(dpd_engine* e, int64_t nsteps, bool obs, int timing)
{
    int rc;
    int64_t ti = 0;   // timed launches so far (event pair 2 ti, 2 ti + 1)
    bool advanced = false;   // the previous pair launch carried the step's epilogue
    for (int64_t t = 0; t < nsteps; ++t) {
        rc = (t == 0) ? sort_step<kBegin>(e) : sort_step<kEndBegin>(e, advanced);
        if (rc) return rc;
        const bool last = t == nsteps - 1;
        const bool epi = !last && epilogue_ok(e);
        const bool timed = timed_step(t, timing);
        if (timed) HIPCHK(hipEventRecord(e->pev[2 * ti], e->stream));
        bool terms_done = false;
        if ((rc = launch_pair(e, obs && last, &terms_done, epi, true))) return rc;
        if (timed) HIPCHK(hipEventRecord(e->pev[2 * ti++ + 1], e->stream));
        if (!terms_done) {
            if (obs && last) launch_bonded<true>(e);
            else launch_bonded<false>(e);
        }
        advanced = epi;
    }
    if (obs) launch_finish<true, true>(e, e->frc);
    else launch_finish<true, false>(e, e->frc);
    HIPCHK(hipGetLastError());
    return DPD_OK;
}

// Assemble the staged boxes into device buffers and sort them.
int commit_beads(dpd_engine* e, int64_t step0)
{
    int64_t n = 0, groups = 0;
    for (size_t b = 0; b < e->boxes.size(); ++b) {
        const BoxHost& h = e->boxes[b];
        if (h.n == 0) return fail(e, DPD_ERR_STATE, "box " + std::to_string(b) + " has no beads");
        groups += h.B.ngroups;
        n += h.n;
    }
    if (n > ((int64_t)1 << 30) || groups * kGroupKeys > ((int64_t)1 << 30))
        return fail(e, DPD_ERR_PARAM, "batch too large");
    // from here on what the device holds changes: without a state until all of it is there
    e->committed = false;
    drop_graphs(e);
    const int nbr = (int)groups;
    n = groups = 0;
    for (size_t b = 0; b < e->boxes.size(); ++b) {
        BoxHost& h = e->boxes[b];
        h.bead_off = n;
        h.nbeads = h.n;
        h.bond_off = h.nbonds = h.pair_off = h.npairs = 0;
        h.B.koff = (int)groups * kGroupKeys;
        h.B.goff = (int)groups;
        h.B.box = (int)b;
        groups += h.B.ngroups;
        n += h.n;
    }
    int rc;
    // hit-list workgroups of a batch: slots of one box each (a box's beads are the slots
    // [bead_off, bead_off + n) since the sort keys are ordered by box)
    if (e->boxes.size() > 1) {
        for (int tb = 0; tb < kSchedules; ++tb) {
            if (kSchedule[tb].kernel != DPD_PAIR_HITLIST) continue;
            const int64_t th = kSchedule[tb].beads();
            std::vector<int4> hb;
            for (size_t b = 0; b < e->boxes.size(); ++b) {
                const int64_t s0 = e->boxes[b].bead_off, s1 = s0 + e->boxes[b].n;
                for (int64_t s = s0; s < s1; s += th)
                    hb.push_back(make_int4((int)b, (int)s, (int)std::min<int64_t>(s + th, s1), 0));
            }
            if ((rc = dalloc(e, &e->hitblk[tb], hb.size()))) return rc;
            HIPCHK(hipMemcpyAsync(e->hitblk[tb], hb.data(), sizeof(int4) * hb.size(), hipMemcpyHostToDevice,
                                  e->stream));
            HIPCHK(hipStreamSynchronize(e->stream));
            e->nhitblk[tb] = (int)hb.size();
        }
    }
    const bool new_cells = nbr != e->ngroups || !e->cells;
    if (new_cells) {
        e->ngroups = nbr;
        e->nkeys = nbr * kGroupKeys;
        // (each part starts at a multiple of four: the counts are read four at a time)
        const size_t nk = (size_t)e->nkeys, ng = (size_t)(nbr + 4) / 4 * 4, nc = (nk + 1 + 3) / 4 * 4;
        if ((rc = dalloc(e, &e->cells, nk + 3 * ng + 2 * nc))) return rc;
        e->cnt = e->cells;
        e->counts[0] = e->cells + nk;
        e->counts[1] = e->counts[0] + ng;
        e->gstart = e->counts[1] + ng;
        e->cstart[0] = e->gstart + ng;
        e->cstart[1] = e->cstart[0] + nc;
        e->cleared = nk + 2 * ng;
        if ((rc = clear_counts(e))) return rc;
    }
    // (a call that ended without the arrays by bead left n at 0)
    const bool new_beads = n != e->n;
    if (new_cells || new_beads) {
        // spill (int4 a bead), order (int2 a bead), bins
        e->n = 0;
        const size_t nbins = bin_at((int)n, e->nkeys);
        if ((rc = dalloc(e, &e->filed, (6 * (size_t)n + nbins + 3) / 4))) return rc;
        e->spill = e->filed;
        e->order = reinterpret_cast<int2*>(e->filed + n);
        e->bins = reinterpret_cast<int*>(e->order + n);
    }
    if (new_beads) {
        std::vector<Part> parts;
        for (int b = 0; b < 2; ++b)
            for (const Part& q : {part(&e->pos[b], n), part(&e->vel[b], n), part(&e->fold[b], n), part(&e->bead[b], n),
                                  part(&e->key[b], n), part(&e->code[b], n + kCodePad)})
                parts.push_back(q);
        for (const Part& q : {part(&e->img, n), part(&e->frc, n), part(&e->vp, n), part(&e->slot_of, n),
                              part(&e->gather, 12 * n)})
            parts.push_back(q);
        if ((rc = dalloc_parts(e, &e->per_bead, parts))) return rc;
        for (int b = 0; b < 2; ++b) HIPCHK(hipMemsetAsync(e->code[b] + n, 0, sizeof(uint32_t) * kCodePad, e->stream));
    }
    e->n = n;
    if ((rc = upload_boxes(e))) return rc;
    std::vector<float4> hp(n), hv(n), hf(n);
    std::vector<int> hb(n);
    std::vector<int4> hi(n);
    std::vector<int> hk(n), hc(e->nkeys + 1, 0);   // cell keys and, for the bins, their cell starts
    for (size_t b = 0; b < e->boxes.size(); ++b) {
        const BoxHost& h = e->boxes[b];
        const BoxDev& B = h.B;
        const double L[3] = {B.n[0] * B.wd[0], B.n[1] * B.wd[1], B.n[2] * B.wd[2]};
        for (int64_t i = 0; i < h.n; ++i) {
            const int64_t g = h.bead_off + i;
            int c[3], im[3];
            float o[3];
            for (int d = 0; d < 3; ++d) {
                const double xd = h.x[3 * i + d];
                int ci = (int)std::floor(xd / B.wd[d]);
                ci = std::min(std::max(ci, 0), B.n[d] - 1);
                float of = (float)(xd - ci * B.wd[d]);
                if (of >= B.w[d]) of = B.w[d] * 0.99999994f;
                if (of < 0.f) of = 0.f;
                c[d] = ci;
                o[d] = of;
                im[d] = (int)std::lround((h.u[3 * i + d] - xd) / L[d]);
            }
            const int32_t w = h.type[i] | ((int32_t)b << 8);
            float wb, ib;
            std::memcpy(&wb, &w, 4);
            std::memcpy(&ib, &h.id[i], 4);
            hp[g] = make_float4(o[0], o[1], o[2], wb);
            hv[g] = make_float4((float)h.v[3 * i], (float)h.v[3 * i + 1], (float)h.v[3 * i + 2], ib);
            hf[g] = h.has_f ? make_float4((float)h.f[3 * i], (float)h.f[3 * i + 1], (float)h.f[3 * i + 2], 0.f)
                            : make_float4(0.f, 0.f, 0.f, 0.f);
            hb[g] = (int)g;
            hi[g] = make_int4(im[0], im[1], im[2], 0);
            hk[g] = B.koff + cell_key(c[0], c[1], c[2], B);
            ++hc[hk[g] + 1];
        }
    }
    for (int k = 0; k < e->nkeys; ++k) hc[k + 1] += hc[k];
    const int src = e->cur;
    HIPCHK(hipMemcpyAsync(e->pos[src], hp.data(), sizeof(float4) * n, hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(e->vel[src], hv.data(), sizeof(float4) * n, hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(e->fold[src], hf.data(), sizeof(float4) * n, hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(e->bead[src], hb.data(), sizeof(int) * n, hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(e->img, hi.data(), sizeof(int4) * n, hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(e->key[src], hk.data(), sizeof(int) * n, hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(e->cstart[src], hc.data(), sizeof(int) * hc.size(), hipMemcpyHostToDevice, e->stream));
    if ((rc = sort_step<kRebin>(e))) return rc;
    hipLaunchKernelGGL(k_copy_force, dim3(grid(n, 256)), dim3(256), 0, e->stream, (int)n, e->fold[e->cur], e->frc);
    hipLaunchKernelGGL(k_set_step, dim3(1), dim3(64), 0, e->stream, e->dstep, step0);
    HIPCHK(hipGetLastError());
    e->step = step0;
    e->jumps = 0;
    e->obs_valid = false;
    e->committed = true;
    auto_schedule(e);
    return report(e, false);
}

// Global CSR topology from the staged per-box bonds and bond pairs.
void mark_bonded(dpd_engine* e)
{
    if (e->nbonded > 0)
        hipLaunchKernelGGL(k_set_bonded_flag, dim3(grid(e->nbonded, 256)), dim3(256), 0, e->stream, topo(e), e->slot_of,
                           bufs(e, e->cur), e->dboxes);
}

int commit_topology(dpd_engine* e)
{
    const int64_t n = e->n;
    std::vector<int> bp(n + 1, 0), ap(n + 1, 0);
    std::vector<int> H, Tl, F, Sd;
    std::vector<double> K, L0, M, P;
    for (BoxHost& h : e->boxes) {
        const int off = (int)h.bead_off;
        const int boff = (int)H.size();
        h.bond_off = boff;
        h.nbonds = (int)h.bh.size();
        h.pair_off = (int)F.size();
        h.npairs = (int)h.pf.size();
        for (size_t b = 0; b < h.bh.size(); ++b) {
            H.push_back(h.bh[b] + off); Tl.push_back(h.bt[b] + off);
            K.push_back(h.bk[b]); L0.push_back(h.bl0[b]);
        }
        for (size_t q = 0; q < h.pf.size(); ++q) {
            F.push_back(h.pf[q] + boff); Sd.push_back(h.ps[q] + boff);
            M.push_back(h.pk[q]); P.push_back(h.pphi[q]);
        }
    }
    const int64_t nbonds = (int64_t)H.size(), npairs = (int64_t)F.size();
    for (int64_t b = 0; b < nbonds; ++b) { bp[H[b] + 1]++; bp[Tl[b] + 1]++; }
    std::vector<int4> abead(std::max<int64_t>(npairs, 1));
    std::vector<double4> apar(std::max<int64_t>(npairs, 1));
    for (int64_t q = 0; q < npairs; ++q) {
        const int a = H[Sd[q]], bm = H[F[q]], c = Tl[F[q]];
        abead[q] = make_int4(a, bm, c, 0);
        apar[q] = make_double4(M[q], P[q], std::cos(P[q]), std::sin(P[q]));
        ap[a + 1]++; ap[bm + 1]++; ap[c + 1]++;
    }
    for (int64_t i = 0; i < n; ++i) { bp[i + 1] += bp[i]; ap[i + 1] += ap[i]; }
    // each bead's entries in bond order (then angle order)
    std::vector<int2> bent(std::max<int>(bp[n], 1)), bbead(std::max<int64_t>(nbonds, 1));
    std::vector<double2> bpar(std::max<int64_t>(nbonds, 1));
    std::vector<int4> aent(std::max<int>(ap[n], 1));
    std::vector<int> fill(bp.begin(), bp.end() - 1);
    for (int64_t b = 0; b < nbonds; ++b) {
        const int h = H[b], t = Tl[b];
        bbead[b] = make_int2(h, t);
        bpar[b] = make_double2(K[b], L0[b]);
        bent[fill[h]++] = make_int2(t, (int)b << 1);
        bent[fill[t]++] = make_int2(h, (int)b << 1 | 1);
    }
    std::vector<int> afill(ap.begin(), ap.end() - 1);
    for (int64_t q = 0; q < npairs; ++q) {
        const int4 abc = abead[q];
        aent[afill[abc.z]++] = make_int4(abc.x, abc.y, (int)q, 0);
        aent[afill[abc.y]++] = make_int4(abc.x, abc.z, (int)q, 1);
        aent[afill[abc.x]++] = make_int4(abc.y, abc.z, (int)q, 2);
    }
    std::vector<int> bonded;
    std::vector<int4> span;
    for (int64_t i = 0; i < n; ++i)
        if (bp[i + 1] > bp[i] || ap[i + 1] > ap[i]) {
            bonded.push_back((int)i);
            span.push_back(make_int4(bp[i], bp[i + 1], ap[i], ap[i + 1]));
        }
    drop_graphs(e);
    int rc;
    e->committed = false;   // (until the topology and the beads' marks agree)
    e->nbonded = 0;
    const size_t nb = bonded.size();
    if ((rc = dalloc(e, &e->bond_ent, bent.size())) || (rc = dalloc(e, &e->bond_par, bpar.size())) ||
        (rc = dalloc(e, &e->bond_bead, bbead.size())) || (rc = dalloc(e, &e->ang_ent, aent.size())) ||
        (rc = dalloc(e, &e->ang_bead, abead.size())) || (rc = dalloc(e, &e->ang_par, apar.size())) ||
        (rc = dalloc(e, &e->bonded, nb)) || (rc = dalloc(e, &e->span, nb)) ||
        (multi(e) && (rc = dalloc(e, &e->upos, nb ? n : 0))) || (rc = dalloc(e, &e->bforce, nb ? n : 0)))
        return rc;
    HIPCHK(hipMemcpyAsync(e->bond_ent, bent.data(), sizeof(int2) * bent.size(), hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(e->bond_bead, bbead.data(), sizeof(int2) * bbead.size(), hipMemcpyHostToDevice, e->stream));
    if (nb) {
        HIPCHK(hipMemcpyAsync(e->bonded, bonded.data(), sizeof(int) * nb, hipMemcpyHostToDevice, e->stream));
        HIPCHK(hipMemcpyAsync(e->span, span.data(), sizeof(int4) * nb, hipMemcpyHostToDevice, e->stream));
    }
    HIPCHK(hipMemcpyAsync(e->bond_par, bpar.data(), sizeof(double2) * bpar.size(), hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(e->ang_ent, aent.data(), sizeof(int4) * aent.size(), hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(e->ang_bead, abead.data(), sizeof(int4) * abead.size(), hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(e->ang_par, apar.data(), sizeof(double4) * apar.size(), hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    e->nbonds = (int)nbonds;
    e->nangles = (int)npairs;
    e->nbonded = (int)nb;
    hipLaunchKernelGGL(k_clear_bonded_flag, dim3(grid(n, 256)), dim3(256), 0, e->stream, (int)n, e->pos[e->cur],
                       e->bead[e->cur], e->slot_of);
    auto_schedule(e);
    mark_bonded(e);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(e->stream));
    e->committed = true;
    return DPD_OK;
}

int stage_beads(dpd_engine* e, int32_t box, int64_t n, const int32_t* id, const int32_t* type, const double* x,
                const double* unpbc, const double* v, const double* f)
{
    if (box < 0 || box >= (int32_t)e->boxes.size()) return fail(e, DPD_ERR_PARAM, "box index out of range");
    if (n < 1 || n > ((int64_t)1 << 30)) return fail(e, DPD_ERR_PARAM, "bead count out of range");
    if (!id || !type || !x || !v) return fail(e, DPD_ERR_PARAM, "null bead array");
    BoxHost& h = e->boxes[box];
    const BoxDev& B = h.B;
    const double L[3] = {B.n[0] * B.wd[0], B.n[1] * B.wd[1], B.n[2] * B.wd[2]};
    for (int64_t i = 0; i < n; ++i) {
        if (type[i] < 0 || type[i] >= h.p.ntypes) return fail(e, DPD_ERR_PARAM, "bead type out of range");
        for (int d = 0; d < 3; ++d)
            if (!(x[3 * i + d] >= 0.0 && x[3 * i + d] < L[d]))
                return fail(e, DPD_ERR_OUT_OF_BOX, "bead " + std::to_string(i) + " outside the box");
    }
    if (h.n != n) { h.bh.clear(); h.bt.clear(); h.pf.clear(); h.ps.clear(); }   // topology refers to indices
    h.n = n;
    h.id.assign(id, id + n);
    h.type.assign(type, type + n);
    h.x.assign(x, x + 3 * n);
    h.u.assign(unpbc ? unpbc : x, (unpbc ? unpbc : x) + 3 * n);
    h.v.assign(v, v + 3 * n);
    h.has_f = f != nullptr;
    h.f.assign(f ? f : x, (f ? f : x) + (f ? 3 * n : 0));
    return DPD_OK;
}

int stage_topology(dpd_engine* e, int32_t box, int64_t nbonds, const int32_t* head, const int32_t* tail,
                   const double* k, const double* l0, int64_t npairs, const int32_t* first, const int32_t* second,
                   const double* modulus, const double* phi0)
{
    if (box < 0 || box >= (int32_t)e->boxes.size()) return fail(e, DPD_ERR_PARAM, "box index out of range");
    BoxHost& h = e->boxes[box];
    if (h.n == 0) return fail(e, DPD_ERR_STATE, "upload beads before topology");
    if (nbonds < 0 || npairs < 0) return fail(e, DPD_ERR_PARAM, "negative counts");
    if (nbonds && (!head || !tail || !k || !l0)) return fail(e, DPD_ERR_PARAM, "null bond array");
    if (npairs && (!first || !second || !modulus || !phi0)) return fail(e, DPD_ERR_PARAM, "null pair array");
    for (int64_t b = 0; b < nbonds; ++b)
        if (head[b] < 0 || head[b] >= h.n || tail[b] < 0 || tail[b] >= h.n || head[b] == tail[b])
            return fail(e, DPD_ERR_PARAM, "bond bead index out of range");
    for (int64_t q = 0; q < npairs; ++q) {
        if (first[q] < 0 || first[q] >= nbonds || second[q] < 0 || second[q] >= nbonds)
            return fail(e, DPD_ERR_PARAM, "bond pair index out of range");
        if (tail[second[q]] != head[first[q]]) return fail(e, DPD_ERR_PARAM, "bond pair bonds do not share a bead");
    }
    h.bh.assign(head, head + nbonds); h.bt.assign(tail, tail + nbonds);
    h.bk.assign(k, k + nbonds); h.bl0.assign(l0, l0 + nbonds);
    h.pf.assign(first, first + npairs); h.ps.assign(second, second + npairs);
    h.pk.assign(modulus, modulus + npairs); h.pphi.assign(phi0, phi0 + npairs);
    return DPD_OK;
}

}  // namespace

// Static scratch of dpd_slice_stress_noalloc: the pair and bond slice tables of one call,
// held by every device the library runs on until the process ends.  Its host-side name is
// a stand-in, not a device address: scratch_ptr looks up each device's own copy once.
constexpr size_t kSliceScratchDoubles = (size_t)1 << 19;   // 4 MiB
static __device__ __align__(256) double scratch[kSliceScratchDoubles];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch[kMaxDevices] = {};

// the device address of this engine's device's copy of `scratch` (looked up on the first
// call on that device, with that device current)
int scratch_ptr(dpd_engine* e, double** out)
{
    if (e->device < 0 || e->device >= kMaxDevices) return fail(e, DPD_ERR_PARAM, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[e->device]) {
        HIPCHK(hipSetDevice(e->device));
        void* p = nullptr;
        HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return fail(e, DPD_ERR_HIP, "hipGetSymbolAddress returned no address for the slice scratch");
        g_scratch[e->device] = (double*)p;
    }
    *out = g_scratch[e->device];
    return DPD_OK;
}

int slice_check(dpd_engine* e, int32_t box, int32_t nslices, size_t* ntab)
{
    if (!e->committed) return fail(e, DPD_ERR_STATE, "no beads uploaded");
    if (box < 0 || box >= (int32_t)e->boxes.size()) return fail(e, DPD_ERR_PARAM, "box index out of range");
    if (nslices < 1 || nslices > 65536) return fail(e, DPD_ERR_PARAM, "nslices must be in [1, 65536]");
    HIPCHK(hipSetDevice(e->device));
    const int nt = e->boxes[box].B.ntypes;
    *ntab = (size_t)nslices * nt * nt * 9;
    return DPD_OK;
}

// pair and bond tables of box `box` into the cleared device tables tab[0 .. 2 ntab), then
// to the host outputs (either may be null)
int slice_tables(dpd_engine* e, int32_t box, int32_t nslices, double* tab, size_t ntab, double* pair_out,
                 double* bond_out)
{
    const BoxHost& h = e->boxes[box];
    const int nt = h.B.ntypes;
    SliceArgs a{};
    a.B = h.B;
    a.pos = e->pos[e->cur];
    a.vp = e->vp;
    a.img = e->img;
    a.key = e->key[e->cur];
    a.cstart = e->cstart[e->cur];
    a.table = e->table + (size_t)box * kTableStride;
    a.step = e->dstep;
    a.slot_of = e->slot_of;
    a.bond_bead = e->bond_bead;
    a.bond_par = e->bond_par;
    a.b0 = h.bond_off;
    a.b1 = a.b0 + h.nbonds;
    a.ang_bead = e->ang_bead;
    a.ang_par = e->ang_par;
    a.a0 = a.a1 = 0;
    a.nbeads = (int)h.nbeads;
    a.nslice = nslices;
    a.ntypes = nt;
    a.nidx = nt * nt;
    HIPCHK(launch_slice_stress(a, pair_out ? tab : nullptr, bond_out ? tab + ntab : nullptr, e->stream));
    if (pair_out) HIPCHK(hipMemcpyAsync(pair_out, tab, sizeof(double) * ntab, hipMemcpyDeviceToHost, e->stream));
    if (bond_out) HIPCHK(hipMemcpyAsync(bond_out, tab + ntab, sizeof(double) * ntab, hipMemcpyDeviceToHost, e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    return DPD_OK;
}

}  // namespace

// ------------------------------------------------------------------ C ABI ------

extern "C" {

const char* dpd_last_error(const dpd_engine* e) { return e ? e->err.c_str() : "null engine"; }

int dpd_create_batch(int32_t nbox, const dpd_params* p, dpd_engine** out)
{
    if (!out) return DPD_ERR_PARAM;
    *out = nullptr;
    if (!p || nbox < 1 || nbox > (1 << 22)) return DPD_ERR_PARAM;
    dpd_engine* e = new dpd_engine();
    *out = e;
    int rc;
    e->boxes.resize(nbox);
    for (int b = 0; b < nbox; ++b) {
        if ((rc = check_params(e, p + b))) return rc;
        BoxHost& h = e->boxes[b];
        h.p = p[b];
        const int nt = p[b].ntypes;
        h.a.assign(p[b].a, p[b].a + nt * nt);
        h.g.assign(p[b].gamma, p[b].gamma + nt * nt);
        h.p.a = h.a.data();
        h.p.gamma = h.g.data();
        h.dt = p[b].dt; h.lambda = p[b].lambda; h.kT = p[b].kT;
        BoxDev& B = h.B;
        B.n[0] = p[b].nx; B.n[1] = p[b].ny; B.n[2] = p[b].nz;
        for (int d = 0; d < 2; ++d) B.inv[d] = 1.0f / (float)B.n[d];
        B.wd[0] = p[b].wx; B.wd[1] = p[b].wy; B.wd[2] = p[b].wz;
        for (int d = 0; d < 3; ++d) B.w[d] = (float)B.wd[d];
        {
            // the scan's cut-off 1 + m (code_dist2) in code units
            float s2 = 0.f, umax = 0.f;
            for (int d = 0; d < 3; ++d) {
                B.qinv[d] = (float)kCodeUnits / B.w[d];
                s2 += B.w[d] * B.w[d] * (d == 1 ? 2.25f : 1.0f);
                umax = std::max(umax, B.qinv[d]);
            }
            const float tu = (1.0f + std::sqrt(s2) * (1.01f / kCodeUnits) + 1e-5f) * umax;
            B.qthr = (int)(tu * tu) + 2;
        }
        B.ntypes = nt;
        B.seed0 = (uint32_t)p[b].seed;
        B.seed1 = (uint32_t)(p[b].seed >> 32);
        B.ngroups = (int)(((int64_t)B.n[0] * B.n[1] * B.n[2] + kGroupKeys - 1) / kGroupKeys);
        B.box = b;
        set_step_constants(h);
    }
    e->device = p[0].device;
    HIPCHK(hipSetDevice(e->device));
    HIPCHK(hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking));
    for (auto& ev : e->ev) HIPCHK(hipEventCreate(&ev));
    if ((rc = dpd_set_pair_kernel(e, p[0].pair_kernel))) return rc;
    const size_t nacc = (size_t)nbox * (sums(e).spread + 1) * kObsStride;
    if ((rc = dalloc_parts(e, &e->per_box, {part(&e->flags, 4), part(&e->dstep, 2), part(&e->acc, nacc),
                                            part(&e->table, (size_t)nbox * kTableStride), part(&e->dboxes, nbox)})))
        return rc;
    // (flags, times and sums)
    HIPCHK(hipMemsetAsync(e->per_box, 0, (char*)e->table - e->per_box, e->stream));
    const size_t nh = (size_t)nbox * kObsStride;
    HIPCHK(hipHostMalloc((void**)&e->hacc, sizeof(double) * nh + sizeof(int) * 4, hipHostMallocDefault));
    e->hflags = reinterpret_cast<int*>(e->hacc + nh);
    if ((rc = upload_tables(e))) return rc;
    e->err.clear();
    return DPD_OK;
}

int dpd_create(const dpd_params* p, dpd_engine** out) { return dpd_create_batch(1, p, out); }

void dpd_destroy(dpd_engine* e)
{
    if (!e) return;
    if (e->stream) (void)hipStreamSynchronize(e->stream);
    drop_graphs(e);
    void* ptrs[] = {e->per_box, e->per_bead, e->cells, e->filed, e->bond_ent, e->ang_ent, e->span, e->bond_par,
                    e->ang_bead, e->ang_par, e->bond_bead, e->upos, e->bforce, e->bonded, e->slice, e->madj};
    for (void* q : ptrs)
        if (q) (void)hipFree(q);
    for (void* q : e->hitblk)
        if (q) (void)hipFree(q);
    if (e->hacc) (void)hipHostFree(e->hacc);
    for (auto& ev : e->ev)
        if (ev) (void)hipEventDestroy(ev);
    for (auto& ev : e->pev) (void)hipEventDestroy(ev);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    delete e;
}

int dpd_upload_beads(dpd_engine* e, int64_t n, const int32_t* id, const int32_t* type, const double* x,
                     const double* unpbc, const double* v, const double* f, int64_t step0)
{
    if (!e) return DPD_ERR_PARAM;
    if (e->boxes.size() != 1) return fail(e, DPD_ERR_STATE, "batch engine: use dpd_upload_box and dpd_commit");
    HIPCHK(hipSetDevice(e->device));
    const bool keep_topo = !e->boxes[0].bh.empty() && e->boxes[0].n == n;
    int rc;
    if ((rc = stage_beads(e, 0, n, id, type, x, unpbc, v, f))) return rc;
    if ((rc = commit_beads(e, step0))) return rc;
    if (keep_topo) return commit_topology(e);
    e->nbonds = e->nangles = e->nbonded = 0;
    auto_schedule(e);
    return DPD_OK;
}

int dpd_upload_topology(dpd_engine* e, int64_t nbonds, const int32_t* head, const int32_t* tail, const double* k,
                        const double* l0, int64_t npairs, const int32_t* first_bond, const int32_t* second_bond,
                        const double* modulus, const double* phi0)
{
    if (!e) return DPD_ERR_PARAM;
    if (e->boxes.size() != 1) return fail(e, DPD_ERR_STATE, "batch engine: use dpd_upload_box_topology");
    if (!e->committed) return fail(e, DPD_ERR_STATE, "upload beads before topology");
    HIPCHK(hipSetDevice(e->device));
    int rc;
    if ((rc = stage_topology(e, 0, nbonds, head, tail, k, l0, npairs, first_bond, second_bond, modulus, phi0)))
        return rc;
    return commit_topology(e);
}

int dpd_upload_box(dpd_engine* e, int32_t box, int64_t n, const int32_t* id, const int32_t* type, const double* x,
                   const double* unpbc, const double* v, const double* f)
{
    if (!e) return DPD_ERR_PARAM;
    return stage_beads(e, box, n, id, type, x, unpbc, v, f);
}

int dpd_upload_box_topology(dpd_engine* e, int32_t box, int64_t nbonds, const int32_t* head, const int32_t* tail,
                            const double* k, const double* l0, int64_t npairs, const int32_t* first_bond,
                            const int32_t* second_bond, const double* modulus, const double* phi0)
{
    if (!e) return DPD_ERR_PARAM;
    return stage_topology(e, box, nbonds, head, tail, k, l0, npairs, first_bond, second_bond, modulus, phi0);
}

int dpd_commit(dpd_engine* e, int64_t step0)
{
    if (!e) return DPD_ERR_PARAM;
    HIPCHK(hipSetDevice(e->device));
    int rc;
    if ((rc = commit_beads(e, step0))) return rc;
    return commit_topology(e);
}

int32_t dpd_box_count(const dpd_engine* e) { return e ? (int32_t)e->boxes.size() : -1; }

int dpd_step(dpd_engine* e, int64_t nsteps, uint32_t flags)
{
    if (!e) return DPD_ERR_PARAM;
    if (!e->committed) return fail(e, DPD_ERR_STATE, "no beads uploaded");
    if (nsteps < 0) return fail(e, DPD_ERR_PARAM, "negative step count");
    if (nsteps == 0) return DPD_OK;
    HIPCHK(hipSetDevice(e->device));
    const bool obs = flags & DPD_STEP_OBSERVE;
    const bool timing = flags & DPD_STEP_TIMING;
    const int timing_mode = timing ? ((flags & DPD_STEP_TIMING_SAMPLED) ? 2 : 1) : 0;
    const bool use_graph = (flags & DPD_STEP_GRAPH) && !timing;
    int rc;
    e->jumps = 0;
    if (timing) {
        while ((int64_t)e->pev.size() < 2 * timed_steps(nsteps, timing_mode)) {
            hipEvent_t ev;
            HIPCHK(hipEventCreate(&ev));
            e->pev.push_back(ev);
        }
    }
    HIPCHK(hipEventRecord(e->ev[0], e->stream));
    if (use_graph) {
        // whole calls of an even step count replay one captured graph: the two SoA buffers
        // swap once per step, so an even count returns to the captured pointers
        int64_t chunk = std::min<int64_t>(nsteps, 64);
        if (chunk & 1) chunk -= 1;
        int64_t done = 0;
        while (chunk >= 2 && nsteps - done >= chunk) {
            const bool last_obs = obs && (nsteps - done == chunk);
            const auto keyg = std::make_pair(chunk, (int)last_obs | e->cur << 1);
            auto it = e->graphs.find(keyg);
            if (it == e->graphs.end()) {
                const int cur0 = e->cur;
                hipGraph_t g;
                HIPCHK(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
                rc = enqueue_steps(e, chunk, last_obs, 0);
                hipError_t st = hipStreamEndCapture(e->stream, &g);
                if (rc) return rc;
                if (st != hipSuccess) return fail(e, DPD_ERR_HIP, std::string("graph capture: ") + hipGetErrorString(st));
                e->cur = cur0;
                hipGraphExec_t ge;
                HIPCHK(hipGraphInstantiate(&ge, g, nullptr, nullptr, 0));
                e->graphs[keyg] = ge;
                e->graph_src[keyg] = g;
                it = e->graphs.find(keyg);
            }
            HIPCHK(hipGraphLaunch(it->second, e->stream));
            done += chunk;
            e->step += chunk;
        }
        if (done < nsteps) {
            if ((rc = enqueue_steps(e, nsteps - done, obs, 0))) return rc;
            e->step += nsteps - done;
        }
    } else {
        if ((rc = enqueue_steps(e, nsteps, obs, timing_mode))) return rc;
        e->step += nsteps;
    }
    HIPCHK(hipEventRecord(e->ev[1], e->stream));
    if ((rc = report(e, obs))) return rc;
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, e->ev[0], e->ev[1]));
    e->t_total = ms;
    e->t_pair = 0.0;
    e->n_pair = 0;
    if (timing) {
        double tp = 0.0;
        int64_t np = 0;
        for (; np < timed_steps(nsteps, timing_mode); ++np) {
            HIPCHK(hipEventElapsedTime(&ms, e->pev[2 * np], e->pev[2 * np + 1]));
            tp += ms;
        }
        e->t_pair = tp;
        e->n_pair = np;
    }
    if (obs) return finish_obs(e);
    e->obs_valid = false;
    return DPD_OK;
}

}  // extern "C"

namespace {

void launch_gather(dpd_engine* e, const float4* frc, double* x, double* u, double* v, double* f)
{
    const int n = (int)e->n;
    const dim3 gr(grid(n, 256)), bl(256);
    const BoxDev B0 = e->boxes[0].B;
    if (multi(e))
        hipLaunchKernelGGL(k_gather<true>, gr, bl, 0, e->stream, n, bufs(e, e->cur), frc, e->dboxes, B0, x, u, v, f);
    else
        hipLaunchKernelGGL(k_gather<false>, gr, bl, 0, e->stream, n, bufs(e, e->cur), frc, e->dboxes, B0, x, u, v, f);
}

// dpd_compute_forces with the tables as they are
int evaluate_forces(dpd_engine* e, int64_t step, double* f_out, double* virial, double* pe)
{
    int rc;
    // beside the trajectory: force and time of the next dpd_step stay as they are
    hipLaunchKernelGGL(k_set_step, dim3(1), dim3(64), 0, e->stream, e->dstep + 1, step);
    // the uploaded state is sorted with vp = v: evaluate at it (after dpd_step, vp is the
    // last step's predicted velocity)
    bool terms_done = false;
    if ((rc = launch_pair(e, true, &terms_done, false, false, true, true))) return rc;
    if (!terms_done) launch_bonded<true>(e);
    launch_finish<false, false>(e, aside_force(e));
    HIPCHK(hipGetLastError());
    double* g = e->gather;
    if (f_out) launch_gather(e, aside_force(e), nullptr, nullptr, nullptr, g);
    if ((rc = report(e, true))) return rc;
    if (f_out) {
        HIPCHK(hipMemcpyAsync(f_out, g, sizeof(double) * 3 * e->n, hipMemcpyDeviceToHost, e->stream));
        HIPCHK(hipStreamSynchronize(e->stream));
    }
    const double* h = e->hacc;
    // totals over all boxes
    if (virial)
        for (int i = 0; i < 9; ++i) {
            virial[i] = 0.0;
            for (size_t b = 0; b < e->boxes.size(); ++b) virial[i] += h[b * kObsStride + O_VIR + i];
        }
    if (pe)
        for (int i = 0; i < 3; ++i) {
            pe[i] = 0.0;
            for (size_t b = 0; b < e->boxes.size(); ++b) pe[i] += h[b * kObsStride + O_PEP + i];
        }
    return DPD_OK;
}

}  // namespace

extern "C" {

int dpd_compute_forces(dpd_engine* e, int64_t step, uint32_t flags, double* f_out, double* virial, double* pe)
{
    if (!e) return DPD_ERR_PARAM;
    if (!e->committed) return fail(e, DPD_ERR_STATE, "no beads uploaded");
    HIPCHK(hipSetDevice(e->device));
    if (!(flags & DPD_NO_THERMOSTAT)) return evaluate_forces(e, step, f_out, virial, pe);
    // the thermostat is back whatever the evaluation ends with
    std::vector<bool> saved;
    for (auto& b : e->boxes) { saved.push_back(b.thermostat_on); b.thermostat_on = false; }
    int rc = upload_tables(e);
    if (!rc) rc = evaluate_forces(e, step, f_out, virial, pe);
    for (size_t b = 0; b < e->boxes.size(); ++b) e->boxes[b].thermostat_on = saved[b];
    const int back = upload_tables(e);
    return rc ? rc : back;
}

int dpd_observables_box(dpd_engine* e, int32_t box, dpd_obs* out)
{
    if (!e || !out) return DPD_ERR_PARAM;
    if (!e->obs_valid) return fail(e, DPD_ERR_STATE, "no observables: call dpd_step with DPD_STEP_OBSERVE");
    if (box < 0 || box >= (int32_t)e->obs.size()) return fail(e, DPD_ERR_PARAM, "box index out of range");
    *out = e->obs[box];
    return DPD_OK;
}

int dpd_observables(dpd_engine* e, dpd_obs* out) { return dpd_observables_box(e, 0, out); }

int dpd_download_box(dpd_engine* e, int32_t box, double* x, double* unpbc, double* v, double* f)
{
    if (!e) return DPD_ERR_PARAM;
    if (!e->committed) return fail(e, DPD_ERR_STATE, "no beads uploaded");
    if (box < -1 || box >= (int32_t)e->boxes.size()) return fail(e, DPD_ERR_PARAM, "box index out of range");
    HIPCHK(hipSetDevice(e->device));
    const int64_t n = e->n;
    double* g = e->gather;
    launch_gather(e, e->frc, x ? g : nullptr, unpbc ? g + 3 * n : nullptr, v ? g + 6 * n : nullptr, f ? g + 9 * n : nullptr);
    HIPCHK(hipGetLastError());
    const int64_t off = box < 0 ? 0 : e->boxes[box].bead_off;
    const int64_t cnt = box < 0 ? e->n : e->boxes[box].nbeads;
    const size_t b3 = sizeof(double) * 3 * cnt;
    if (x) HIPCHK(hipMemcpyAsync(x, g + 3 * off, b3, hipMemcpyDeviceToHost, e->stream));
    if (unpbc) HIPCHK(hipMemcpyAsync(unpbc, g + 3 * n + 3 * off, b3, hipMemcpyDeviceToHost, e->stream));
    if (v) HIPCHK(hipMemcpyAsync(v, g + 6 * n + 3 * off, b3, hipMemcpyDeviceToHost, e->stream));
    if (f) HIPCHK(hipMemcpyAsync(f, g + 9 * n + 3 * off, b3, hipMemcpyDeviceToHost, e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    return DPD_OK;
}

int dpd_download(dpd_engine* e, double* x, double* unpbc, double* v, double* f)
{
    return dpd_download_box(e, -1, x, unpbc, v, f);
}

int dpd_set_box_interactions(dpd_engine* e, int32_t box, const double* a, const double* gamma)
{
    if (!e) return DPD_ERR_PARAM;
    const int32_t b0 = box < 0 ? 0 : box, b1 = box < 0 ? (int32_t)e->boxes.size() : box + 1;
    if (b0 >= (int32_t)e->boxes.size() || b1 > (int32_t)e->boxes.size())
        return fail(e, DPD_ERR_PARAM, "box index out of range");
    for (int32_t b = b0; b < b1; ++b) {
        BoxHost& h = e->boxes[b];
        const int nt = h.p.ntypes;
        if (a) h.a.assign(a, a + nt * nt);
        if (gamma) h.g.assign(gamma, gamma + nt * nt);
    }
    return upload_tables(e);
}

int dpd_set_interactions(dpd_engine* e, const double* a, const double* gamma)
{
    return dpd_set_box_interactions(e, -1, a, gamma);
}

int dpd_set_timestep(dpd_engine* e, double dt)
{
    if (!e) return DPD_ERR_PARAM;
    if (!(dt > 0.0)) return fail(e, DPD_ERR_PARAM, "dt must be positive");
    for (auto& b : e->boxes) { b.dt = dt; set_step_constants(b); }
    drop_graphs(e);
    return e->committed ? upload_boxes(e) : DPD_OK;
}

int dpd_toggle(dpd_engine* e, int32_t what, int32_t on)
{
    if (!e) return DPD_ERR_PARAM;
    if (what == DPD_TOGGLE_FORCES) {
        // the step constants are kernel arguments of captured graphs: drop them
        for (auto& b : e->boxes) { b.forces_on = on != 0; set_step_constants(b); }
        drop_graphs(e);
        return e->committed ? upload_boxes(e) : DPD_OK;
    }
    for (auto& b : e->boxes) {
        if (what == DPD_TOGGLE_THERMOSTAT) b.thermostat_on = on != 0;
        else if (what == DPD_TOGGLE_CONSERVATIVE) b.conservative_on = on != 0;
        else return fail(e, DPD_ERR_PARAM, "unknown toggle");
    }
    return upload_tables(e);
}

int64_t dpd_last_timing(dpd_engine* e, double* ms3)
{
    if (!e) return -1;
    if (ms3) { ms3[0] = e->t_total; ms3[1] = e->t_pair; ms3[2] = e->t_total - e->t_pair; }
    return e->n_pair;
}

int64_t dpd_get_step(const dpd_engine* e) { return e ? e->step : -1; }

int dpd_time_pair(dpd_engine* e, int32_t nlaunch, double* ms_per_launch)
{
    if (!e || !ms_per_launch) return DPD_ERR_PARAM;
    if (!e->committed) return fail(e, DPD_ERR_STATE, "no beads uploaded");
    if (nlaunch < 1 || nlaunch > 100000) return fail(e, DPD_ERR_PARAM, "nlaunch must be in [1, 100000]");
    HIPCHK(hipSetDevice(e->device));
    int rc;
    // the launch a step that another follows uses: with the epilogue where the schedule has
    // one, which also files the beads for the counting sort and may raise the flags (both
    // cleared below)
    const bool epi = epilogue_ok(e);
    hipLaunchKernelGGL(k_set_step, dim3(1), dim3(64), 0, e->stream, e->dstep + 1, e->step);
    bool terms_done = false;
    if ((rc = launch_pair(e, false, &terms_done, epi, false, false, true))) return rc;   // untimed first launch
    HIPCHK(hipEventRecord(e->ev[0], e->stream));
    for (int32_t i = 0; i < nlaunch; ++i)
        if ((rc = launch_pair(e, false, &terms_done, epi, false, false, true))) return rc;
    HIPCHK(hipEventRecord(e->ev[1], e->stream));
    if (epi) {
        HIPCHK(hipMemsetAsync(e->flags, 0, sizeof(int) * 4, e->stream));
        if ((rc = clear_counts(e))) return rc;
    }
    HIPCHK(hipStreamSynchronize(e->stream));
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, e->ev[0], e->ev[1]));
    *ms_per_launch = (double)ms / nlaunch;
    return DPD_OK;
}

int dpd_set_pair_kernel(dpd_engine* e, int32_t kernel)
{
    if (!e) return DPD_ERR_PARAM;
    if (kernel != DPD_PAIR_AUTO && (kernel < 1 || kernel > DPD_PAIR_KINDS))
        return fail(e, DPD_ERR_PARAM, "unknown pair kernel");
    if (kernel != DPD_PAIR_AUTO && !pair_kernel_available(kernel))
        return fail(e, DPD_ERR_UNSUPPORTED, "pair kernel " + std::to_string(kernel) + " is retired");
    e->pair_auto = kernel == DPD_PAIR_AUTO;
    if (e->pair_auto) set_schedule(e, e->committed ? default_schedule(e) : kFullShellSchedule);
    else if (kernel == DPD_PAIR_FULLSHELL) set_schedule(e, kFullShellSchedule);
    else if (kSchedule[e->sched].kernel != DPD_PAIR_HITLIST)
        set_schedule(e, e->committed ? size_schedule(e->n, e->nbonded > 0) : kDefaultSchedule);
    return DPD_OK;
}

int32_t dpd_get_pair_kernel(const dpd_engine* e) { return e ? e->pair_kernel : -1; }

int32_t dpd_schedule_count(void) { return kSchedules; }

const char* dpd_schedule_name(int32_t sched)
{
    return (sched >= 0 && sched < kSchedules) ? kSchedule[sched].name : nullptr;
}

int dpd_set_schedule(dpd_engine* e, int32_t sched)
{
    if (!e) return DPD_ERR_PARAM;
    if (sched < 0 || sched >= kSchedules) return fail(e, DPD_ERR_PARAM, "unknown schedule");
    e->pair_auto = false;
    set_schedule(e, sched);
    return DPD_OK;
}

int32_t dpd_get_schedule(const dpd_engine* e) { return e ? e->sched : -1; }

int dpd_apply_tuning(dpd_engine* e, const char* path, int32_t* chosen)
{
    if (!e || !path) return DPD_ERR_PARAM;
    if (chosen) *chosen = -1;
    if (!e->committed) return fail(e, DPD_ERR_STATE, "no beads uploaded");
    FILE* fh = std::fopen(path, "r");
    if (!fh) return fail(e, DPD_ERR_IO, std::string("cannot open ") + path);
    // the engine's shape, as dpd_amd.tune keys it
    const int64_t nbox = (int64_t)e->boxes.size();
    auto bucket = [](int64_t n) {
        int64_t lo = 1;
        while (lo * 2 <= n) lo *= 2;
        return lo;
    };
    const int64_t lo = bucket(e->n / nbox), tot = bucket(e->n);
    const int64_t key[7] = {nbox == 1 ? 1 : 2, lo, 2 * lo, e->boxes[0].p.ntypes, (e->nbonds + e->nangles) > 0, tot, 2 * tot};
    const char* names[8] = {"\"nbox\":",   "\"beads_lo\":", "\"beads_hi\":", "\"ntypes\":",
                            "\"bonded\":", "\"total_lo\":", "\"total_hi\":", "\"schedule\":"};
    char line[4096];
    int found = -1;
    while (found < 0 && std::fgets(line, sizeof(line), fh)) {
        int64_t v[8];
        bool ok = true;
        for (int k = 0; k < 8 && ok; ++k) {
            const char* p = std::strstr(line, names[k]);
            if (p) v[k] = std::strtoll(p + std::strlen(names[k]), nullptr, 10);
            // all beads of a batch: a line without them holds for any, and one box has its own
            else if (k == 5 || k == 6) v[k] = key[k];
            else ok = false;
        }
        if (!ok) continue;
        bool match = true;
        for (int k = 0; k < (nbox == 1 ? 5 : 7); ++k) match = match && v[k] == key[k];
        if (match && v[7] >= 0 && v[7] < kSchedules) found = (int)v[7];
    }
    std::fclose(fh);
    if (found >= 0) {
        if (kSchedule[found].kernel == DPD_PAIR_HITLIST && e->n > (int64_t)kHitSlotMask) found = kFullShellSchedule;
        e->pair_auto = false;
        set_schedule(e, found);
    }
    if (chosen) *chosen = found;
    return DPD_OK;
}

namespace {

// Time `nsteps` steps of each candidate schedule from the current state, restoring the
// state after every trial (the simulation does not advance); ms[k] gets the time per step of
// trial k.  The fastest is left set; *best is its schedule.
int tune_trials(dpd_engine* e, int32_t nsteps, const std::vector<int>& trials, double* ms, int* best)
{
    if (!e->committed) return fail(e, DPD_ERR_STATE, "no beads uploaded");
    if (nsteps < 1) return fail(e, DPD_ERR_PARAM, "nsteps must be positive");
    HIPCHK(hipSetDevice(e->device));
    const int64_t n = e->n;
    // snapshot of the state the trials start from
    float4 *sp = nullptr, *sv = nullptr, *sfo = nullptr, *sf = nullptr, *svp = nullptr;
    int4* sa = nullptr;
    int *sk = nullptr, *sso = nullptr, *scs = nullptr, *sbd = nullptr;
    uint32_t* scd = nullptr;
    int rc;
    if ((rc = dalloc(e, &sp, n)) || (rc = dalloc(e, &sv, n)) || (rc = dalloc(e, &sfo, n)) || (rc = dalloc(e, &sf, n)) ||
        (rc = dalloc(e, &svp, n)) || (rc = dalloc(e, &sa, n)) || (rc = dalloc(e, &sk, n)) ||
        (rc = dalloc(e, &sso, n)) || (rc = dalloc(e, &scs, e->nkeys + 1)) || (rc = dalloc(e, &scd, n)) ||
        (rc = dalloc(e, &sbd, n)))
        return rc;
    const int c0 = e->cur;
    const int64_t step0 = e->step;
    auto copy = [&](bool save) -> int {
        const hipMemcpyKind k = hipMemcpyDeviceToDevice;
        const size_t f4 = sizeof(float4) * n;
        if (save) {
            HIPCHK(hipMemcpyAsync(sp, e->pos[c0], f4, k, e->stream));
            HIPCHK(hipMemcpyAsync(sv, e->vel[c0], f4, k, e->stream));
            HIPCHK(hipMemcpyAsync(sfo, e->fold[c0], f4, k, e->stream));
            HIPCHK(hipMemcpyAsync(sf, e->frc, f4, k, e->stream));
            HIPCHK(hipMemcpyAsync(svp, e->vp, f4, k, e->stream));
            HIPCHK(hipMemcpyAsync(sa, e->img, sizeof(int4) * n, k, e->stream));
            HIPCHK(hipMemcpyAsync(sbd, e->bead[c0], sizeof(int) * n, k, e->stream));
            HIPCHK(hipMemcpyAsync(sk, e->key[c0], sizeof(int) * n, k, e->stream));
            HIPCHK(hipMemcpyAsync(scd, e->code[c0], sizeof(uint32_t) * n, k, e->stream));
            HIPCHK(hipMemcpyAsync(sso, e->slot_of, sizeof(int) * n, k, e->stream));
            HIPCHK(hipMemcpyAsync(scs, e->cstart[c0], sizeof(int) * (e->nkeys + 1), k, e->stream));
        } else {
            HIPCHK(hipMemcpyAsync(e->pos[c0], sp, f4, k, e->stream));
            HIPCHK(hipMemcpyAsync(e->vel[c0], sv, f4, k, e->stream));
            HIPCHK(hipMemcpyAsync(e->fold[c0], sfo, f4, k, e->stream));
            HIPCHK(hipMemcpyAsync(e->frc, sf, f4, k, e->stream));
            HIPCHK(hipMemcpyAsync(e->vp, svp, f4, k, e->stream));
            HIPCHK(hipMemcpyAsync(e->img, sa, sizeof(int4) * n, k, e->stream));
            HIPCHK(hipMemcpyAsync(e->bead[c0], sbd, sizeof(int) * n, k, e->stream));
            HIPCHK(hipMemcpyAsync(e->key[c0], sk, sizeof(int) * n, k, e->stream));
            HIPCHK(hipMemcpyAsync(e->code[c0], scd, sizeof(uint32_t) * n, k, e->stream));
            HIPCHK(hipMemcpyAsync(e->slot_of, sso, sizeof(int) * n, k, e->stream));
            HIPCHK(hipMemcpyAsync(e->cstart[c0], scs, sizeof(int) * (e->nkeys + 1), k, e->stream));
            hipLaunchKernelGGL(k_set_step, dim3(1), dim3(64), 0, e->stream, e->dstep, step0);
            e->cur = c0;
            e->step = step0;
            mark_bonded(e);   // (the unwrapped positions)
            if (int rc = clear_counts(e)) return rc;   // (an odd number of steps left those of buffer c0)
        }
        HIPCHK(hipStreamSynchronize(e->stream));
        return DPD_OK;
    };
    if ((rc = copy(true))) return rc;
    double bestms = 1e300;
    int bests = e->sched;
    for (size_t v = 0; v < trials.size(); ++v) {
        set_schedule(e, trials[v]);
        if ((rc = dpd_step(e, 1, 0))) break;          // warm-up (code objects, caches)
        if ((rc = copy(false))) break;
        if ((rc = dpd_step(e, nsteps, 0))) break;
        const double t = e->t_total / nsteps;
        if (ms) ms[v] = t;
        if (t < bestms) { bestms = t; bests = trials[v]; }
        if ((rc = copy(false))) break;
    }
    void* tmp[] = {sp, sv, sfo, sf, svp, sa, sk, sso, scs, scd, sbd};
    for (void* q : tmp) (void)hipFree(q);
    if (rc) return rc;
    e->obs_valid = false;
    e->pair_auto = false;   // the tuned choice stays across commits
    set_schedule(e, bests);
    if (best) *best = bests;
    return DPD_OK;
}

}  // namespace

int dpd_autotune(dpd_engine* e, int32_t nsteps, int32_t* chosen, double* ms_per_step)
{
    if (!e) return DPD_ERR_PARAM;
    const int hit = size_schedule(e->n, e->nbonded > 0);
    const std::vector<int> trials = {hit, kFullShellSchedule};
    double ms[2] = {0.0, 0.0};
    int best = 0;
    int rc = tune_trials(e, nsteps, trials, ms, &best);
    if (rc) return rc;
    if (ms_per_step) {
        for (int k = 0; k < DPD_PAIR_KINDS; ++k) ms_per_step[k] = 0.0;
        ms_per_step[kSchedule[hit].kernel - 1] = ms[0];
        ms_per_step[kSchedule[kFullShellSchedule].kernel - 1] = ms[1];
    }
    if (chosen) *chosen = kSchedule[best].kernel;
    return DPD_OK;
}

int dpd_autotune_schedules(dpd_engine* e, int32_t nsteps, int32_t* chosen, double* ms_per_step)
{
    if (!e) return DPD_ERR_PARAM;
    std::vector<int> trials;
    for (int k = 0; k < kSchedules; ++k)
        if (kSchedule[k].kernel != DPD_PAIR_HITLIST || e->n <= (int64_t)kHitSlotMask) trials.push_back(k);
    std::vector<double> ms(trials.size(), 0.0);
    int best = 0;
    int rc = tune_trials(e, nsteps, trials, ms.data(), &best);
    if (rc) return rc;
    if (ms_per_step) {
        for (int k = 0; k < kSchedules; ++k) ms_per_step[k] = 0.0;
        for (size_t v = 0; v < trials.size(); ++v) ms_per_step[trials[v]] = ms[v];
    }
    if (chosen) *chosen = best;
    return DPD_OK;
}

namespace {

// shared body of dpd_zero_total_momentum / dpd_renormalise_momenta
int adjust_momenta(dpd_engine* e, int32_t box, bool renormalise)
{
    if (!e) return DPD_ERR_PARAM;
    if (!e->committed) return fail(e, DPD_ERR_STATE, "no beads uploaded");
    const int nbox = (int)e->boxes.size();
    if (box < -1 || box >= nbox) return fail(e, DPD_ERR_PARAM, "box index out of range");
    HIPCHK(hipSetDevice(e->device));
    const int n = (int)e->n;
    if (multi(e)) hipLaunchKernelGGL(k_mom_sums<true>, dim3(grid(n, 256)), dim3(256), 0, e->stream, n, bufs(e, e->cur), sums(e));
    else hipLaunchKernelGGL(k_mom_sums<false>, dim3(grid(n, 256)), dim3(256), 0, e->stream, n, bufs(e, e->cur), sums(e));
    HIPCHK(hipGetLastError());
    int rc;
    if ((rc = report(e, true))) return rc;
    std::vector<double4> adj(nbox, make_double4(0.0, 0.0, 0.0, 1.0));
    for (int b = 0; b < nbox; ++b) {
        if (box >= 0 && b != box) continue;
        const double* a = e->hacc + (size_t)b * kObsStride;
        const double cnt = a[4];
        if (!(cnt > 0.0)) continue;
        if (renormalise) {
            // CSimBox::UpdateRenormalisedMom (src/SimBox.cpp:3177-3215): v / sqrt(sum v^2 / (3 N kT))
            const double norm = std::sqrt(a[3] / (3.0 * cnt * e->boxes[b].kT));
            if (norm > 0.0) adj[b].w = 1.0 / norm;
        } else {
            // CSimBox::ZeroTotalMom (src/SimBox.cpp:1919-1947): v - sum v / N
            adj[b] = make_double4(a[0] / cnt, a[1] / cnt, a[2] / cnt, 1.0);
        }
    }
    if (!e->madj && (rc = dalloc(e, &e->madj, (size_t)nbox))) return rc;
    HIPCHK(hipMemcpyAsync(e->madj, adj.data(), sizeof(double4) * nbox, hipMemcpyHostToDevice, e->stream));
    if (multi(e)) hipLaunchKernelGGL(k_mom_apply<true>, dim3(grid(n, 256)), dim3(256), 0, e->stream, n, bufs(e, e->cur), e->madj);
    else hipLaunchKernelGGL(k_mom_apply<false>, dim3(grid(n, 256)), dim3(256), 0, e->stream, n, bufs(e, e->cur), e->madj);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(e->stream));
    e->obs_valid = false;
    return DPD_OK;
}

}  // namespace

int dpd_zero_total_momentum(dpd_engine* e, int32_t box) { return adjust_momenta(e, box, false); }

int dpd_renormalise_momenta(dpd_engine* e, int32_t box) { return adjust_momenta(e, box, true); }

int dpd_slice_stress(dpd_engine* e, int32_t box, int32_t nslices, double* pair_out, double* bond_out)
{
    if (!e) return DPD_ERR_PARAM;
    int rc;
    size_t ntab = 0;
    if ((rc = slice_check(e, box, nslices, &ntab))) return rc;
    if (2 * ntab > e->slice_cap) {
        if ((rc = dalloc(e, &e->slice, 2 * ntab))) { e->slice_cap = 0; return rc; }
        e->slice_cap = 2 * ntab;
    }
    HIPCHK(hipMemsetAsync(e->slice, 0, sizeof(double) * 2 * ntab, e->stream));
    return slice_tables(e, box, nslices, e->slice, ntab, pair_out, bond_out);
}

int dpd_slice_stress_noalloc(dpd_engine* e, int32_t box, int32_t nslices, double* pair_out, double* bond_out)
{
    if (!e) return DPD_ERR_PARAM;
    int rc;
    size_t ntab = 0;
    if ((rc = slice_check(e, box, nslices, &ntab))) return rc;
    if (2 * ntab > kSliceScratchDoubles)
        return fail(e, DPD_ERR_PARAM, "slice tables of " + std::to_string(2 * ntab) + " doubles exceed the " +
                                          std::to_string(kSliceScratchDoubles) + " of the static scratch");
    double* tab = nullptr;
    if ((rc = scratch_ptr(e, &tab))) return rc;
    // the scratch keeps the last call's tables: clear the part this call uses (a kernel,
    // not a memset node, so that the call may be captured)
    const int nclr = (int)(2 * ntab);
    hipLaunchKernelGGL(k_zero, dim3(grid(std::max(nclr, 1), 256)), dim3(256), 0, e->stream, tab, nclr);
    HIPCHK(hipGetLastError());
    return slice_tables(e, box, nslices, tab, ntab, pair_out, bond_out);
}

int dpd_energy_output(dpd_engine* e, int32_t box, double* out3)
{
    if (!e || !out3) return DPD_ERR_PARAM;
    if (!e->committed) return fail(e, DPD_ERR_STATE, "no beads uploaded");
    if (box < 0 || box >= (int32_t)e->boxes.size()) return fail(e, DPD_ERR_PARAM, "box index out of range");
    HIPCHK(hipSetDevice(e->device));
    const BoxHost& h = e->boxes[box];
    if (e->slice_cap < 3) {
        int rc;
        if ((rc = dalloc(e, &e->slice, 3))) { e->slice_cap = 0; return rc; }
        e->slice_cap = 3;
    }
    HIPCHK(hipMemsetAsync(e->slice, 0, sizeof(double) * 3, e->stream));
    SliceArgs a{};
    a.B = h.B;
    a.pos = e->pos[e->cur];
    a.vp = e->vp;
    a.img = e->img;
    a.key = e->key[e->cur];
    a.cstart = e->cstart[e->cur];
    a.table = e->table + (size_t)box * kTableStride;
    a.slot_of = e->slot_of;
    a.bond_bead = e->bond_bead;
    a.bond_par = e->bond_par;
    a.ang_bead = e->ang_bead;
    a.ang_par = e->ang_par;
    a.b0 = h.bond_off;
    a.b1 = a.b0 + h.nbonds;
    a.a0 = h.pair_off;
    a.a1 = a.a0 + h.npairs;
    a.ntypes = h.B.ntypes;
    HIPCHK(launch_energy_output(a, e->slice, e->stream));
    HIPCHK(hipMemcpyAsync(out3, e->slice, sizeof(double) * 3, hipMemcpyDeviceToHost, e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    return DPD_OK;
}

int dpd_slice_stress_bondpairs(dpd_engine* e, int32_t box, int32_t nslices, double* out)
{
    if (!e || !out) return DPD_ERR_PARAM;
    if (!e->committed) return fail(e, DPD_ERR_STATE, "no beads uploaded");
    if (box < 0 || box >= (int32_t)e->boxes.size()) return fail(e, DPD_ERR_PARAM, "box index out of range");
    if (nslices < 1 || nslices > 65536) return fail(e, DPD_ERR_PARAM, "nslices must be in [1, 65536]");
    HIPCHK(hipSetDevice(e->device));
    const BoxHost& h = e->boxes[box];
    const int nt = h.B.ntypes;
    const size_t ntab = (size_t)nslices * nt * nt * nt * 9;
    if (ntab > e->slice_cap) {
        int rc;
        if ((rc = dalloc(e, &e->slice, ntab))) { e->slice_cap = 0; return rc; }
        e->slice_cap = ntab;
    }
    HIPCHK(hipMemsetAsync(e->slice, 0, sizeof(double) * ntab, e->stream));
    SliceArgs a{};
    a.B = h.B;
    a.pos = e->pos[e->cur];
    a.img = e->img;
    a.key = e->key[e->cur];
    a.slot_of = e->slot_of;
    a.ang_bead = e->ang_bead;
    a.ang_par = e->ang_par;
    a.a0 = h.pair_off;
    a.a1 = a.a0 + h.npairs;
    a.nslice = nslices;
    a.ntypes = nt;
    a.nidx = nt * nt * nt;
    HIPCHK(launch_slice_bondpairs(a, e->slice, e->stream));
    HIPCHK(hipMemcpyAsync(out, e->slice, sizeof(double) * ntab, hipMemcpyDeviceToHost, e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    return DPD_OK;
}

}  // extern "C"
