// engine_common.hpp -- device-side building blocks shared by the DPD step kernels.
//
// Layout in HBM: an engine holds one or more boxes (replicas).  Beads of all boxes are
// sorted together every step by a global cell key.  Within a box the key orders cells
// row-major, x fastest: local key = cx + nx (cy + ny cz); a box's keys start at its key
// offset, a multiple of 64 (its key range is padded to whole groups of 64 keys, the unit
// of the two-level counting-sort scan).  A row of cells along x is therefore one
// contiguous slot range -- the hit-list kernel scans the three cells cx-1..cx+1 of a
// neighbour row as one range -- and a box's beads are one contiguous slot range too.
//
// Positions are FP32 offsets inside the bead's cell, o in [0, w), plus the integer cell
// (from the key) and integer periodic image counts.  Differences of positions are
// (o_i - o_j) + (c_i - c_j) * w with exact integer cell deltas, so FP32 keeps ~1e-7
// absolute precision at any box size (absolute FP32 coordinates would lose 7.6e-6 at
// L = 64).  The absolute FP64 position c*w + o and the unwrapped position
// (c + img*n)*w + o are formed only on download and in the FP64 bonded terms.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dpd {

constexpr int kGroupKeys = 64;   // cell keys per scan group
constexpr int kMaxTypes = 16;
constexpr int kTypeStride = kMaxTypes * kMaxTypes;   // one matrix of a box's table
constexpr int kTableStride = 3 * kTypeStride;        // a | gamma | sqrt(gamma) per box
constexpr int kObsStride = 32;                       // FP64 accumulators per box

// Constants of one box.  Mirrors the CCNTCell statics set by SetSimBoxLengths /
// SetTimeStepConstants (src/CNTCell.cpp:143-203).
struct BoxDev {
    int n[3];          // cells per axis
    float inv[2];      // 1 / n[0], 1 / n[1] (division by reciprocal in key_cell)
    float w[3];        // cell widths
    double wd[3];
    float dt, hdt, hdt2, lamdt;   // dt, dt/2, dt^2/2, lambda*dt
    float invrootdt;              // sqrt(24 kT / dt)
    float qinv[3];                // kCodeUnits / w: scan-code units
    int qthr;                     // square of the scan's widened cut-off in the smallest of them
    int ntypes;
    uint32_t seed0, seed1;        // key of the pair stream
    int koff;                     // first global cell key of this box (a multiple of 64)
    int goff;                     // first global scan group of this box
    int ngroups;                  // scan groups of 64 keys (cells, padded)
    int box;                      // index of this box
};

// local key of cell (cx, cy, cz) of a box
__host__ __device__ inline int cell_key(int cx, int cy, int cz, const BoxDev& B)
{
    return cx + B.n[0] * (cy + B.n[1] * cz);
}

// x / d for 0 <= x < 2^24, d >= 1, given inv = 1/d rounded to FP32: the FP32 estimate is
// within one of the quotient, and one correction step makes it exact.
__host__ __device__ inline int div_small(int x, int d, float inv)
{
    int q = (int)((float)x * inv);
    const int r = x - q * d;
    q += (r >= d) ? 1 : ((r < 0) ? -1 : 0);
    return q;
}

// cell of a local key (boxes hold at most 2^24 cells, so div_small is exact)
__host__ __device__ inline void key_cell(int key, const BoxDev& B, int c[3])
{
    const int t = div_small(key, B.n[0], B.inv[0]);
    c[0] = key - t * B.n[0];
    c[2] = div_small(t, B.n[1], B.inv[1]);
    c[1] = t - c[2] * B.n[1];
}

__host__ __device__ inline int floordiv(int a, int n)
{
    return (a >= 0) ? a / n : -((-a + n - 1) / n);
}

// bead word packing: pos.w = type | (x index of the cell mod 4) << 4 | box << 8
__host__ __device__ inline int bead_type(int w) { return w & (kMaxTypes - 1); }
constexpr int kCellXShift = 4;
constexpr int kCellXBits = 3 << kCellXShift;
__host__ __device__ inline int bead_box(int w) { return (w >> 8) & 0x3FFFFF; }
// bit 30 of a position's w: the bead has bonds or angles (set from the topology)
constexpr int kBondedBit = 1 << 30;

// Philox4x32-10 (Salmon et al., SC'11).  Pair uniform: counter (min id, max id, step),
// key = seed; U = (word0 >> 8) * 2^-24, exactly representable in FP32.
__device__ inline uint32_t philox_word0(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                        uint32_t k0, uint32_t k1)
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) { k0 += 0x9E3779B9u; k1 += 0xBB67AE85u; }
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        // three-input xors as one v_bitop3_b32 each (truth table 0x96: a ^ b ^ c), which
        // the compiler does not form from two xors itself
        const uint32_t n0 = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c1, k0, 0x96);
        const uint32_t n1 = (uint32_t)p1;
        const uint32_t n2 = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c3, k1, 0x96);
        const uint32_t n3 = (uint32_t)p0;
        c0 = n0; c1 = n1; c2 = n2; c3 = n3;
    }
    return c0;
}

// key of the pair stream of one box at one step
struct RngKey {
    uint32_t seed0, seed1, step0, step1;
};

__device__ inline RngKey rng_key(const BoxDev& B, int64_t step)
{
    return RngKey{B.seed0, B.seed1, (uint32_t)(uint64_t)step, (uint32_t)((uint64_t)step >> 32)};
}

__device__ inline float pair_uniform(uint32_t ida, uint32_t idb, const RngKey& K)
{
    const uint32_t lo = ida < idb ? ida : idb;
    const uint32_t hi = ida < idb ? idb : ida;
    const uint32_t r = philox_word0(lo, hi, K.step0, K.step1, K.seed0, K.seed1);
    return (float)(r >> 8) * 0x1p-24f;
}

// DPD pair force on bead i from bead j (src/CNTCell.cpp:1191-1225):
//   F = [a w + (-gamma w^2 (r^.v)) + sqrt(gamma) w sqrt(24kT/dt) (0.5 - U)] r^,  w = 1 - r
// returns the scalar F/r so that F_vec = s * dx.  1/r is the hardware reciprocal square
// root (1 ulp) and r = r^2 / r; callers guarantee r^2 > 1e-18 (no denormals).
__device__ inline float pair_scalar(float dr2, float dxdv, float a, float sg, float g, uint32_t idi,
                                    uint32_t idj, float invrootdt, const RngKey& K, float* pe)
{
    const float inv = __builtin_amdgcn_rsqf(dr2);
    const float dr = dr2 * inv;
    const float wr = 1.0f - dr;
    const float con = a * wr;
    const float diss = -(g * wr * wr) * (dxdv * inv);
    const float u = pair_uniform(idi, idj, K);
    const float rnd = sg * wr * invrootdt * (0.5f - u);
    if (pe) *pe = 0.5f * a * wr * wr;
    return (con + diss + rnd) * inv;
}

// pair_scalar with the random amplitude sgr = sqrt(gamma) sqrt(24kT/dt) as one factor
__device__ inline float pair_scalar_t(float dr2, float dxdv, float a, float sgr, float g, uint32_t idi, uint32_t idj,
                                      const RngKey& K, float* pe)
{
    const float inv = __builtin_amdgcn_rsqf(dr2);
    const float dr = dr2 * inv;
    const float wr = 1.0f - dr;
    const float con = a * wr;
    const float diss = -(g * wr * wr) * (dxdv * inv);
    const float u = pair_uniform(idi, idj, K);
    const float rnd = sgr * wr * (0.5f - u);
    if (pe) *pe = 0.5f * a * wr * wr;
    return (con + diss + rnd) * inv;
}

// Scan code of a bead: its x, y and z in units of w / kCodeUnits, with the cell and modulo 256,
// in bytes 0, 1 and 3, and a one in byte 2 (code_dist2).
constexpr int kCodeUnits = 84;
__device__ inline uint32_t scan_code(const float o[3], const int c[3], const BoxDev& B)
{
    uint32_t q[3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
        q[a] = (uint32_t)(min(max((int)(o[a] * B.qinv[a]), 0), kCodeUnits - 1) + kCodeUnits * c[a]) & 0xFF;
    return q[0] | (q[1] << 8) | (1u << 16) | (q[2] << 24);
}

// The integration arithmetic with its rounding fixed by explicit fused multiply-adds, so
// that kernels repeating a sum (k_advance and k_sort, the pair epilogue, the last step's
// k_finish) get the same bits however the compiler contracts the rest: kick is v + h f (the
// halves of UpdateMom, the predicted velocity), drift the displacement dt v + dt^2/2 f.
__device__ inline float kick(float v, float f, float h) { return fmaf(h, f, v); }
__device__ inline float drift(float v, float f, const BoxDev& B) { return fmaf(B.dt, v, B.hdt2 * f); }

// Move a bead by displacement d from offset o in cell c (image img): new offset in
// [0, w), cell and image; `jump` when it crossed more than one cell.
struct Moved {
    float o[3];
    int c[3];
    int img[3];
    int jump;
    int bad;
};

__device__ inline void advance(const float o[3], const int c[3], const int img[3], const float d[3],
                               const BoxDev& B, Moved& m)
{
    m.jump = 0;
    m.bad = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float x = o[a] + d[a];
        if (!(fabsf(x) < 1.0e6f)) { m.bad = 1; x = 0.0f; }
        // cells moved, floor(x / w): the division's rounding changes nothing up to one cell either
        // way (x - w and x + w are then what its corrections below would leave)
        int s = x < 0.0f ? -1 : (x >= B.w[a] ? 1 : 0);
        if (!(x >= -B.w[a] && x < 2.0f * B.w[a])) s = (int)floorf(x / B.w[a]);
        x = x - (float)s * B.w[a];
        if (x < 0.0f) { x += B.w[a]; s -= 1; }
        if (x >= B.w[a]) x = B.w[a] * 0.99999994f;
        if (x < 0.0f) x = 0.0f;
        m.jump |= (s > 1 || s < -1);
        int cc = c[a] + s;
        const int q = (cc >= 0 && cc < B.n[a]) ? 0 : floordiv(cc, B.n[a]);
        cc -= q * B.n[a];
        m.o[a] = x;
        m.c[a] = cc;
        m.img[a] = img[a] + q;
    }
}

// CBondPair::AddForce (src/BondPair.cpp:138-286) for one angle in FP64.  first = bond
// (b -> c), second = bond (a -> b); f[0] is the force on c (tail of first), f[1] on the
// shared bead b, f[2] on a (head of second); pe (may be null) gets
// CBondPair::AddPotentialEnergy (src/BondPair.cpp:320-378).
__device__ inline void angle_forces(const double ua[3], const double ub[3], const double uc[3], const double4 par,
                                    double f[3][3], double* pe)
{
    double first[3], second[3];
    for (int d = 0; d < 3; ++d) { first[d] = ub[d] - uc[d]; second[d] = ua[d] - ub[d]; }
    const double l1 = sqrt(first[0] * first[0] + first[1] * first[1] + first[2] * first[2]);
    const double l2 = sqrt(second[0] * second[0] + second[1] * second[1] + second[2] * second[2]);
    for (int r = 0; r < 3; ++r) f[r][0] = f[r][1] = f[r][2] = 0.0;
    const double magProduct = l1 * l2;
    if (!(magProduct > 0.0001)) { if (pe) *pe = 0.0; return; }
    const double k = par.x, phi0 = par.y, cosPhi0 = par.z, sinPhi0 = par.w;
    const double b1Dotb2 = first[0] * second[0] + first[1] * second[1] + first[2] * second[2];
    const double b1b2Overb1Sq = b1Dotb2 / (l1 * l1);
    const double b1b2Overb2Sq = b1Dotb2 / (l2 * l2);
    const double cosPhiSq = b1b2Overb1Sq * b1b2Overb2Sq;
    double forceMag;
    if (fabs(b1Dotb2) > 0.000001) {
        const double prefactor = sqrt(1.0 / cosPhiSq - 1.0);
        forceMag = (phi0 > 0.0) ? k * (cosPhi0 - sinPhi0 / prefactor) / magProduct : k / magProduct;
    } else {
        forceMag = k / magProduct;
    }
    for (int d = 0; d < 3; ++d) {
        const double ft = forceMag * (b1b2Overb1Sq * first[d] - second[d]);
        const double fh = forceMag * (first[d] - b1b2Overb2Sq * second[d]);
        f[0][d] = ft;
        f[2][d] = fh;
        f[1][d] = -ft - fh;
    }
    if (pe) {
        const double cps = (b1Dotb2 * b1Dotb2) / (magProduct * magProduct);
        const double sinPhi = sqrt(fmax(0.0, 1.0 - cps));
        double e;
        if (b1Dotb2 > 0.000001) e = phi0 > 0.0 ? k * (1.0 - sqrt(cps) * cosPhi0 - sinPhi * sinPhi0) : k * (1.0 - sqrt(cps));
        else if (b1Dotb2 < -0.000001) e = phi0 > 0.0 ? k * (1.0 + sqrt(cps) * cosPhi0 - sinPhi * sinPhi0) : k * (1.0 + sqrt(cps));
        else e = k * (1.0 - sinPhi0);
        *pe = e;
    }
}

// wave-level helpers (64 lanes)
__device__ inline double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// number of lanes below this one whose bit is set in mask
__device__ inline int lane_prefix(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
}

// Inclusive prefix sum over the 64 lanes of a wavefront with DPP moves: row_shr 1, 2, 4, 8
// scan each row of 16 lanes (lanes shifted in from outside the row read 0), row_bcast 15
// adds row 0's total to row 1 and row 2's to row 3, row_bcast 31 adds the first half's total
// to rows 2 and 3.  Six dependent adds instead of six LDS permutes.
__device__ inline int wave_incl_scan(int x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);   // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);   // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);   // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);   // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);   // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);   // row_bcast:31
    return x;
}

// Intake of the counting sort: every bead is filed under its new cell key while the beads
// still lie in the old order.  The source slots of new cell k go to its bin, with room for five
// more than the beads it holds (a step moves few beads to another cell).  What finds no room is
// spilled to a list with its key and rank, in any state at most all beads.
struct Intake {
    const int* cstart;   // cell starts of the old order
    int* bins;
    int* cnt;            // beads per new cell key
    int* gcnt;           // per scan group
    int4* spill;         // (key, rank, source slot, 0)
    int* nspill;
    int cap;             // room for spills (0: they are dropped)
};
constexpr int kBinSpare = 5;
__host__ __device__ inline size_t bin_at(int start, int k) { return (size_t)start + kBinSpare * (size_t)k; }
__host__ __device__ inline int bin_room(int beads) { return beads + kBinSpare; }

// Runs of equal values over the lanes of a wavefront: `starts` has the first lane of each.
__device__ inline uint64_t run_starts(int v)
{
    const int before = __builtin_amdgcn_update_dpp(v, v, 0x138, 0xf, 0xf, false);   // wave_shr:1
    return __ballot((threadIdx.x & 63) == 0 || before != v);
}
// the lanes of this lane's run
__device__ inline uint64_t run_lanes(uint64_t starts)
{
    const uint64_t upto = ~0ull >> (63 - (threadIdx.x & 63));
    const uint64_t next = starts & ~upto;
    const uint64_t below = next ? (next & -next) - 1 : ~0ull;   // lanes before the next run
    return below & (~0ull << (63 - __builtin_clzll(starts & upto)));
}

// The bead of slot s (where `act`), of cell key `from` so far, under key `to`; reached by the
// whole wavefront, by every lane with the `from` of a slot of its own or its neighbours.  Slots
// are cell-sorted and few beads leave their cell, so the lanes of a run of equal `from` whose
// bead stays are counted with one atomic, and so are those of a run of equal groups; a bead that
// leaves counts by itself.  (One atomic per bead would serialise: those on one address, the
// 192 of a scan group's count, take 12 to 15 ns each in turn.  The pair launch of 96^3 cells took
// 451 us that way against 268 with a loop over the wavefront's distinct keys, whose 300
// instructions were 8% of the launch; 252 us with runs.)
__device__ inline void file_bead(const Intake& I, int from, int to, int s, bool act)
{
    int start = 0, room = 0;
    if (act) {
        start = I.cstart[to];
        room = bin_room(I.cstart[to + 1] - start);
    }
    const int lane = threadIdx.x & 63;
    const bool stays = act && from == to;
    const uint64_t cell = __ballot(stays) & run_lanes(run_starts(from));
    const int first = __builtin_ctzll(cell | (1ull << 63));
    int n = act, r = 0;
    if (stays) n = lane == first ? __popcll(cell) : 0;
    if (n) r = atomicAdd(I.cnt + to, n);
    const int base = __shfl(r, first, 64);
    if (stays) r = base + lane_prefix(cell);
    const bool same = act && from >> 6 == to >> 6;
    const uint64_t group = __ballot(same) & run_lanes(run_starts(from >> 6));
    n = act;
    if (same) n = lane_prefix(group) ? 0 : __popcll(group);
    if (n) atomicAdd(I.gcnt + (to >> 6), n);
    if (act) {
        if (r < room) I.bins[bin_at(start, to) + r] = s;
        else if (I.cap > 0) {
            const int i = atomicAdd(I.nspill, 1);
            if (i < I.cap) I.spill[i] = make_int4(to, r, s, 0);
        }
    }
}

// Accumulators of a call's sums: each box has spread + 1 rows of kObsStride (spread + 1 a power
// of two), of which a workgroup adds to one; k_report adds the rows up.  FP64 atomics on one
// address take 12 to 15 ns in turn: with one row the 10,368 workgroups of k_finish took 134 us in
// a 96^3 box, 42 with sixteen.  Batches of more than kSpreadBoxes boxes have one row a box (256
// bytes; k_report reads a row for each): their workgroups spread over the boxes, and where these
// are large they wait, in k_finish of 17 boxes of 48^3 99 us, 77 for 16 of them with 16 rows.
struct Sums {
    double* acc;
    int spread;
};
constexpr int kSpread = 15;
constexpr int kSpreadBoxes = 16;

// Add per-thread FP64 values v[0..N) to slots base .. base + N - 1 of the threads' boxes (< 0:
// none): one block-wide reduction for the threads of the block's first box, then one
// wavefront-wide for each other box (only blocks straddling a box boundary have any; an atomic
// for each of their threads took such a block 50 us).
template <int N, int WAVES = 4>
__device__ inline void accumulate_boxes(const double (&v)[N], int box, int box0, int base, const Sums& S)
{
    __shared__ double red[N][WAVES];   // workgroups of up to 64 * WAVES threads
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    auto row = [&](int b) { return S.acc + ((size_t)b * (S.spread + 1) + (blockIdx.x & S.spread)) * kObsStride + base; };
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const double s = wave_sum(box == box0 ? v[i] : 0.0);
        if (lane == 0) red[i][wid] = s;
    }
    for (uint64_t todo = __ballot(box >= 0 && box != box0); todo;) {
        const int b = __builtin_amdgcn_readlane(box, __builtin_ctzll(todo));
        for (int i = 0; i < N; ++i) {
            const double s = wave_sum(box == b ? v[i] : 0.0);
            if (lane == 0 && s != 0.0) atomicAdd(row(b) + i, s);
        }
        todo &= ~__ballot(box == b);
    }
    __syncthreads();
    if (threadIdx.x < N) {
        const int nw = (blockDim.x + 63) >> 6;
        double s = 0.0;
        for (int w = 0; w < nw; ++w) s += red[threadIdx.x][w];
        atomicAdd(row(box0) + threadIdx.x, s);
    }
}

}  // namespace dpd
