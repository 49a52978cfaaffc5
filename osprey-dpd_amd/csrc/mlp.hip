// mlp.hip -- surrogate network: BF16 matrix-core forward/backward and FP32 Adam on gfx950.
//
// Two launches an iteration (three for few rows of a wide network).  k_mlp_rows takes 16 rows of
// the batch through the whole forward and backward chain (a workgroup, activations in registers
// and one LDS buffer) and leaves the factors of the weight gradients; k_mlp_update makes every
// gradient entry and applies Adam to it.  Every matrix product runs on v_mfma_f32_16x16x16_bf16
// (BF16 operands, FP32 accumulation).  Operand fragment layout of that instruction for lane l
// (0..63): A holds A[l%16][4(l/16) .. 4(l/16)+3], B holds B[4(l/16) .. 4(l/16)+3][l%16], and the
// accumulator holds C[4(l/16)+i][l%16], i = 0..3.  Everything a product reads from memory is
// stored as fragments: 64 lanes x 4 values, [16 columns][16 of k][lane][4], one 512-byte load per
// wavefront.  A result leaves in that layout too, as the fragment of a product over its rows,
// which is what the weight gradients are.  Weights are kept in BF16 as fragments of W and, for
// the way back, of W transposed.
//
// What bounds it: the latency of a chain of small products (0.7 GFLOP an iteration at 1,638
// rows and 256 hidden units), so what counts is the number of launches and of passes over
// memory.  That iteration took 26 launches and 123 us with a kernel for each product, partial
// sum, column sum and elementwise step; it takes 22 us, 14 of it in k_mlp_rows and 8 in
// k_mlp_update.  With operands in [column][k] order, of which a wavefront's load touches 16
// rows, the two took 25 and 20 us.  Many rows are bound by L2: 20,000 of 256 units 43 and
// 42 us (k_mlp_update reads 330 MB of fragments at 7.8 TB/s), 429 us before.
//
// Sums are split over K in the same parts and added in the same order whatever the kernel
// (split_k), and each part is one chain of matrix instructions, so results do not depend on
// how the work is laid out over the chip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <string>
#include <type_traits>
#include <vector>

#include "dpd_mlp.h"

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

__host__ __device__ inline uint16_t f2bf(float f)
{
    // round to nearest even
    uint32_t u;
    std::memcpy(&u, &f, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// How a product of M x N outputs over K is summed: `parts` parts of `per` terms (a multiple of
// 16), each a chain over ascending k, added in order.  (Enough parts that 64 x 64 tiles of the
// outputs would occupy 256 workgroups, with at least 64 terms each.)
struct SplitK {
    int parts, per;
};
inline SplitK split_k(int M, int N, int K)
{
    int TM = 64, TN = 64;
    if (N < 64) TN = 16;
    else if (M < 64) TM = 16;
    const int tiles = ((N + TN - 1) / TN) * ((M + TM - 1) / TM);
    int nz = 1;
    while (tiles * nz < 256 && K / (2 * nz) >= 64) nz *= 2;
    const int per = (K / 16 + nz - 1) / nz * 16;
    return {(K + per - 1) / per, per};
}

__device__ inline uint2 pack4(const float (&v)[4])
{
    return make_uint2((uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16), (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16));
}
__device__ inline bf16x4 frag(const uint16_t* p) { return *reinterpret_cast<const bf16x4*>(p); }
// place of element (k, n) of a matrix stored as fragments, `steps` 16-row blocks of k
__host__ __device__ inline int64_t frag_at(int64_t k, int64_t n, int64_t steps)
{
    return (((n >> 4) * steps + (k >> 4)) * 64 + ((k & 15) >> 2) * 16 + (n & 15)) * 4 + (k & 3);
}
__device__ inline floatx4 mfma(bf16x4 a, bf16x4 b, floatx4 c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }

// f(steps, k) over k = k0 .. k1 - 16 in ascending order, four, two or one 16-term steps at a
// time (the operands of several steps are then loaded together)
template <class F>
__device__ inline void in_steps(int k0, int k1, const F& f)
{
    int k = k0;
    for (; k + 64 <= k1; k += 64) f(std::integral_constant<int, 4>{}, k);
    if (k + 32 <= k1) { f(std::integral_constant<int, 2>{}, k); k += 32; }
    if (k < k1) f(std::integral_constant<int, 1>{}, k);
}

// f(steps, s) over the 16-term steps s0 .. s1 - 1 in ascending order, eight at a time and what
// is left at once
template <class F>
__device__ inline void in_rounds(int s0, int s1, const F& f)
{
    int s = s0;
    for (; s + 8 <= s1; s += 8) f(std::integral_constant<int, 8>{}, s);
    switch (s1 - s) {
    case 1: f(std::integral_constant<int, 1>{}, s); break;
    case 2: f(std::integral_constant<int, 2>{}, s); break;
    case 3: f(std::integral_constant<int, 3>{}, s); break;
    case 4: f(std::integral_constant<int, 4>{}, s); break;
    case 5: f(std::integral_constant<int, 5>{}, s); break;
    case 6: f(std::integral_constant<int, 6>{}, s); break;
    case 7: f(std::integral_constant<int, 7>{}, s); break;
    }
}

// standardisation of inputs and targets
struct Scaling {
    double in_mean[16], in_scale[16], out_mean[16], out_scale[16];
};

// Inputs standardised to BF16 as [row][16] and as fragments over the rows, targets to FP32
// [row][nout] (y may be null); rows past n and columns past nin are zero.  One thread per
// padded row and column.
__global__ __launch_bounds__(256) void k_mlp_input(int n, int Mp, int nin, int nout, const double* __restrict__ x,
                                                   const double* __restrict__ y, Scaling S, uint16_t* __restrict__ X,
                                                   uint16_t* __restrict__ XF, float* __restrict__ T)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, i = t >> 4;
    const int j = t & 15;
    if (i >= Mp) return;
    uint16_t v = 0;
    if (i < n && j < nin) v = f2bf((float)((x[(size_t)i * nin + j] - S.in_mean[j]) / S.in_scale[j]));
    X[(size_t)i * 16 + j] = v;
    XF[frag_at(i, j, Mp >> 4)] = v;
    if (y && j < nout)
        T[(size_t)i * nout + j] = i < n ? (float)((y[(size_t)i * nout + j] - S.out_mean[j]) / S.out_scale[j]) : 0.0f;
}

struct RowArgs {
    int n, Mp, H, nout;
    SplitK k2, k3;               // sums of the hidden-to-hidden and hidden-to-output products
    const uint16_t* X;           // [Mp][16]
    const float* T;              // [Mp][nout]
    const uint16_t *W1, *W2, *W3;      // fragments of W1, W2, W3
    const uint16_t *W2t, *W3t;         // and of W2 and W3 transposed
    const float *b1, *b2, *b3;
    // training: the gradients' factors as fragments over the rows, and in FP32 for the biases
    uint16_t *H1F, *H2F, *dZ1F, *dZ2F, *dYF;
    float *dZ1, *dZ2, *dY;
    float* h2;                   // in two launches: the second hidden layer between them
    double* loss;
    // prediction: y[n][nout]
    double* out;
    Scaling S;
};

// Rows [16 b, 16 b + 16) through the network and, with TRAIN, back: WAVES wavefronts, wavefront
// w computing the 16-column tiles w, w + WAVES, ... (TPW of them at most) of every hidden layer.
// One LDS buffer holds the layer that the next product reads; the weights come from L2.
// PART: few rows of a wide network in two launches (training, TPW 1), a row block's tiles of the
// two large products spread over blockIdx.y.  kToHidden goes to the second hidden layer,
// kFromHidden from there; what comes before its product every workgroup does itself, and the first
// one stores.  In one launch these rows wait for the weights on their way into one compute unit
// (1,024 units: 4 MB in some 75 us); an iteration of 16 rows takes 45 us instead of 89 at 1,024
// units, 38 instead of 69 at 768 and 31 instead of 52 at 528 (a kernel for each product took 74, 67
// and 65), with the same results to the bit.
enum Part { kWhole, kToHidden, kFromHidden };
template <int WAVES, int TPW, bool TRAIN, Part PART = kWhole>
__global__ __launch_bounds__(64 * WAVES) void k_mlp_rows(RowArgs A)
{
    extern __shared__ __align__(16) uint16_t act[];   // [16][H + 4]
    __shared__ __align__(16) float part[16][256];     // parts of the output layer's sums
    __shared__ __align__(16) uint16_t dyb[16][20];
    __shared__ double lsum[WAVES];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, r = lane & 15, q = (lane >> 4) * 4;
    const int H = A.H, nt = H >> 4, ld = H + 4, Mp = A.Mp;
    const int row0 = blockIdx.x * 16;
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    static_assert(PART == kWhole || (TRAIN && TPW == 1), "two launches: one tile a wavefront");
    const bool whole = PART == kWhole, stores = whole || blockIdx.y == 0;
    // the first of this wavefront's tiles
    const int w0 = whole ? w : (int)blockIdx.y * WAVES + w;
    float h1[TPW][4], h2[TPW][4];
    // this lane's place in this workgroup's fragment of a tile of columns
    auto mine = [&](int tile) { return (((size_t)tile * (Mp >> 4) + blockIdx.x) * 64 + lane) * 4; };
    auto hidden = [&](int tile, const floatx4& z, const float* bias, float (&h)[4], uint16_t* HF, bool keep = true,
                      bool store = true) {
        const int n = tile * 16 + r;
        const float b = bias[n];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            h[i] = row0 + q + i < A.n ? tanhf(z[i] + b) : 0.0f;
            if (keep) act[(q + i) * ld + n] = f2bf(h[i]);
        }
        if (TRAIN && store) *reinterpret_cast<uint2*>(HF + mine(tile)) = pack4(h);
    };
    // act (16 x H) times a weight matrix's fragments: this wavefront's tiles
    auto product = [&](const uint16_t* WF, floatx4 (&s)[TPW]) {
        for (int z = 0; z < A.k2.parts; ++z) {
            floatx4 acc[TPW];
#pragma unroll
            for (int j = 0; j < TPW; ++j) acc[j] = zero;
            auto some = [&](auto steps, int k) {
                constexpr int U = decltype(steps)::value;
                bf16x4 b[U][TPW];
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int j = 0; j < TPW; ++j) {
                        // (a wavefront without this tile repeats the last one)
                        const int tile = min(w0 + WAVES * j, nt - 1);
                        b[u][j] = frag(WF + (((size_t)tile * nt + (k >> 4) + u) * 64 + lane) * 4);
                    }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const bf16x4 a = frag(act + r * ld + k + 16 * u + q);
#pragma unroll
                    for (int j = 0; j < TPW; ++j) acc[j] = mfma(a, b[u][j], acc[j]);
                }
            };
            const int k0 = z * A.k2.per, k1 = min(H, (z + 1) * A.k2.per);
            if constexpr (PART == kWhole) in_steps(k0, k1, some);
            else in_rounds(k0 >> 4, k1 >> 4, [&](auto steps, int s16) { some(steps, 16 * s16); });
#pragma unroll
            for (int j = 0; j < TPW; ++j) s[j] = z ? s[j] + acc[j] : acc[j];
        }
    };
    // hidden layer 1
    auto layer1 = [&](int tile) {
        return mfma(frag(A.X + (size_t)(row0 + r) * 16 + q), frag(A.W1 + (tile * 64 + lane) * 4), zero);
    };
    floatx4 s[TPW];
    if constexpr (PART == kWhole) {
#pragma unroll
        for (int j = 0; j < TPW; ++j) {
            const int tile = w + WAVES * j;
            if (tile < nt) hidden(tile, layer1(tile), A.b1, h1[j], A.H1F);
        }
        __syncthreads();
        product(A.W2, s);
        __syncthreads();   // act is read no more
#pragma unroll
        for (int j = 0; j < TPW; ++j)
            if (w + WAVES * j < nt) hidden(w + WAVES * j, s[j], A.b2, h2[j], A.H2F);
    } else if constexpr (PART == kToHidden) {
        for (int tile = w; tile < nt; tile += WAVES) hidden(tile, layer1(tile), A.b1, h1[0], A.H1F, true, stores);
        __syncthreads();
        product(A.W2, s);
        if (w0 < nt) {
            hidden(w0, s[0], A.b2, h2[0], A.H2F, false);
            *reinterpret_cast<float4*>(A.h2 + mine(w0)) = make_float4(h2[0][0], h2[0][1], h2[0][2], h2[0][3]);
        }
        return;
    } else {
        for (int tile = w; tile < nt; tile += WAVES) {
            const float4 h = *reinterpret_cast<const float4*>(A.h2 + mine(tile));
            const float v[4] = {h.x, h.y, h.z, h.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) act[(q + i) * ld + tile * 16 + r] = f2bf(v[i]);
        }
    }
    __syncthreads();
    // output layer: a part of its sum per wavefront
    for (int z = w; z < A.k3.parts; z += WAVES) {
        floatx4 acc = zero;
        in_steps(z * A.k3.per, min(H, (z + 1) * A.k3.per), [&](auto steps, int k) {
            constexpr int U = decltype(steps)::value;
            bf16x4 b[U];
#pragma unroll
            for (int u = 0; u < U; ++u) b[u] = frag(A.W3 + (((k >> 4) + u) * 64 + lane) * 4);
#pragma unroll
            for (int u = 0; u < U; ++u) acc = mfma(frag(act + r * ld + k + 16 * u + q), b[u], acc);
        });
        *reinterpret_cast<floatx4*>(&part[z][lane * 4]) = acc;
    }
    __syncthreads();
    double l = 0.0;
    if (t < 256) {
        float y = part[0][t];
        for (int z = 1; z < A.k3.parts; ++z) y += part[z][t];
        const int m = 4 * (t >> 6) + (t & 3), n = (t >> 2) & 15, row = row0 + m;
        y += A.b3[n];
        const bool valid = row < A.n && n < A.nout;
        if (TRAIN) {
            const float e = valid ? y - A.T[(size_t)row * A.nout + n] : 0.0f;
            const float g = e / (float)(A.n * A.nout);
            dyb[m][n] = f2bf(g);
            if (stores) {
                A.dYF[(size_t)blockIdx.x * 256 + t] = f2bf(g);
                A.dY[(size_t)blockIdx.x * 256 + t] = g;
            }
            l = valid ? 0.5 * (double)e * (double)e / (double)(A.n * A.nout) : 0.0;
        } else if (valid) {
#pragma clang fp contract(off)
            const double scaled = A.S.out_scale[n] * (double)y;
            A.out[(size_t)row * A.nout + n] = A.S.out_mean[n] + scaled;
        }
    }
    if (!TRAIN) return;
    for (int off = 32; off > 0; off >>= 1) l += __shfl_down(l, off, 64);
    if (lane == 0) lsum[w] = l;
    __syncthreads();
    if (t == 0 && stores) {
        double v = 0.0;
        for (int i = 0; i < WAVES; ++i) v += lsum[i];
        atomicAdd(A.loss, v);
    }
    // back through the output layer
    auto back = [&](int tile, const floatx4& dh, const float (&h)[4], bool keep, uint16_t* dZF, float* dZ, bool store = true) {
        const int n = tile * 16 + r;
        float g[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            g[i] = dh[i] * (1.0f - h[i] * h[i]);
            if (keep) act[(q + i) * ld + n] = f2bf(g[i]);
        }
        if (!store) return;
        *reinterpret_cast<uint2*>(dZF + mine(tile)) = pack4(g);
        *reinterpret_cast<float4*>(dZ + mine(tile)) = make_float4(g[0], g[1], g[2], g[3]);
    };
    const bf16x4 dy = frag(&dyb[r][q]);
    auto layer3 = [&](int tile) { return mfma(dy, frag(A.W3t + (tile * 64 + lane) * 4), zero); };
    if constexpr (PART == kWhole) {
#pragma unroll
        for (int j = 0; j < TPW; ++j) {
            const int tile = w + WAVES * j;
            if (tile < nt) back(tile, layer3(tile), h2[j], true, A.dZ2F, A.dZ2);
        }
    } else {
        for (int tile = w; tile < nt; tile += WAVES) {
            const float4 h = *reinterpret_cast<const float4*>(A.h2 + mine(tile));
            const float v[4] = {h.x, h.y, h.z, h.w};
            back(tile, layer3(tile), v, true, A.dZ2F, A.dZ2, stores);
        }
    }
    __syncthreads();
    product(A.W2t, s);
    if constexpr (PART != kWhole)
        if (w0 < nt) hidden(w0, layer1(w0), A.b1, h1[0], A.H1F, false, false);
#pragma unroll
    for (int j = 0; j < TPW; ++j)
        if (w0 + WAVES * j < nt) back(w0 + WAVES * j, s[j], h1[j], false, A.dZ1F, A.dZ1);
}

struct UpdateArgs {
    int Mp, H;
    SplitK g1, g2, g3;           // sums of the weight gradients
    const uint16_t *XF, *H1F, *H2F, *dZ1F, *dZ2F, *dYF;
    const float *dZ1, *dZ2, *dY;
    int64_t w1, b1, w2, b2, w3, b3;   // parameter offsets
    float* grad;                 // with it: store the gradients and leave the parameters
    float *w, *mo, *ve;
    const uint8_t* mask;
    uint16_t *wf, *wt;           // BF16 fragments of the weights and of the weights transposed
    float lr, c1, c2;
};

// BF16 copies of weight (k, n) of the matrix at parameter offset o with K x N entries
__device__ inline void store_weight(uint16_t* wf, uint16_t* wt, int64_t o, int k, int n, int K, int N, float v)
{
    const uint16_t b = f2bf(v);
    wf[o + frag_at(k, n, K >> 4)] = b;
    wt[o + frag_at(n, k, N >> 4)] = b;
}

// Adam on parameter i with gradient g; entries with mask 0 (padding) stay zero.  Returns the
// new value.
__device__ inline float adam(const UpdateArgs& A, int64_t i, float g)
{
    float wi = 0.f;
    if (A.mask[i]) {
        const float m = 0.9f * A.mo[i] + 0.1f * g;
        const float v = 0.999f * A.ve[i] + 0.001f * g * g;
        A.mo[i] = m;
        A.ve[i] = v;
        wi = A.w[i] - A.lr * (m / A.c1) / (sqrtf(v / A.c2) + 1e-8f);
    }
    A.w[i] = wi;
    return wi;
}

// The gradients of 16 x 16 blocks of a weight matrix, or of 16 biases, and their update:
// tiles of b2, b1, b3, then blocks of W3, of W1, of W2.  Of a workgroup's wavefronts P share a
// block (P the parts of its sum over the rows, as a power of two up to their number) and take
// parts p, p + P, ...; blocks side by side fill the workgroup.  The parts are added in order
// through LDS.
// Bias gradients are column sums in slabs of kColSlab rows: in each, 16 sums over every 16th
// row, added in order, and the slabs in order.
// What bounds it: round trips to L2 one after another, so a wavefront has eight steps' operands
// in flight and what is left of a part in one round more (four, two and one at a time took 12.2
// us at 1,638 rows and 256 units, this 10.4, both in workgroups of sixteen wavefronts; smaller
// ones 8.5); the longest chains, those of the biases, come first.  2 x 2 blocks a wavefront,
// which read half as much, were no faster at 6,000 rows and 512 units (36.6 us at best against
// 33.3): with a quarter of the wavefronts less is in flight.  Loading Adam's moments before the
// product kept more registers and was slower for small nets (100 rows of 64: 13.3 us against
// 9.6).
constexpr int kColSlab = 128;
inline __host__ __device__ int update_share(const SplitK& k, int waves)
{
    int P = 1;
    while (P < k.parts && P < waves) P *= 2;
    return P;
}
inline __host__ __device__ int update_groups(const SplitK& k, int waves, int blocks)
{
    const int per = waves / update_share(k, waves);
    return (blocks + per - 1) / per;
}
__global__ __launch_bounds__(1024) void k_mlp_update(UpdateArgs A)
{
    extern __shared__ __align__(16) float part[];   // [wavefronts][256]
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), r = lane & 15, waves = blockDim.x >> 6;
    const int H = A.H, nt = H >> 4, nb = A.Mp >> 4;
    const int nbias = 2 * nt + 1, n3 = update_groups(A.g3, waves, nt), n1 = update_groups(A.g1, waves, nt);
    int job = blockIdx.x;
    if (job >= nbias) {
        job -= nbias;
        const bool is3 = job < n3, is2 = job >= n3 + n1;
        const SplitK k = is2 ? A.g2 : (is3 ? A.g3 : A.g1);
        job -= is2 ? n3 + n1 : (is3 ? 0 : n3);
        const int P = update_share(k, waves), per = waves / P, blocks = is2 ? nt * nt : nt;
        // block x of the matrix: k tile tm, n tile tn
        auto tm = [&](int x) { return is2 ? x / nt : (is3 ? x : 0); };
        auto tn = [&](int x) { return is2 ? x % nt : (is3 ? 0 : x); };
        const int x = min(job * per + w / P, blocks - 1);   // (past the last: it again, not stored)
        const uint16_t* a = (is2 ? A.H1F : (is3 ? A.H2F : A.XF)) + ((size_t)tm(x) * nb * 64 + lane) * 4;
        const uint16_t* b = (is2 ? A.dZ2F : (is3 ? A.dYF : A.dZ1F)) + ((size_t)tn(x) * nb * 64 + lane) * 4;
        float g[4] = {0.f, 0.f, 0.f, 0.f};   // entries t + v * blockDim of the workgroup's blocks
        for (int z0 = 0; z0 < k.parts; z0 += P) {
            const int z = z0 + w % P;
            if (z < k.parts) {
                floatx4 acc = {0.f, 0.f, 0.f, 0.f};
                in_rounds(z * k.per >> 4, min(A.Mp, (z + 1) * k.per) >> 4, [&](auto steps, int s) {
                    constexpr int U = decltype(steps)::value;
                    bf16x4 fa[U], fb[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        fa[u] = frag(a + (size_t)(s + u) * 256);
                        fb[u] = frag(b + (size_t)(s + u) * 256);
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) acc = mfma(fa[u], fb[u], acc);
                });
                *reinterpret_cast<floatx4*>(part + w * 256 + lane * 4) = acc;
            }
            __syncthreads();
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int c = (t + v * (int)blockDim.x) >> 8, e = (t + v * (int)blockDim.x) & 255;
                if (c < per)
                    for (int u = 0; u < min(P, k.parts - z0); ++u) g[v] += part[(c * P + u) * 256 + e];
            }
            __syncthreads();
        }
        const int64_t o = is2 ? A.w2 : (is3 ? A.w3 : A.w1);
        const int K = is2 || is3 ? H : 16, N = is3 ? 16 : H;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int c = (t + v * (int)blockDim.x) >> 8, e = (t + v * (int)blockDim.x) & 255, y = job * per + c;
            if (c >= per || y >= blocks) continue;
            const int row = tm(y) * 16 + 4 * (e >> 6) + (e & 3), col = tn(y) * 16 + ((e >> 2) & 15);
            const int64_t i = o + (int64_t)row * N + col;
            if (A.grad) A.grad[i] = g[v];
            else store_weight(A.wf, A.wt, o, row, col, K, N, adam(A, i, g[v]));
        }
        return;
    }
    const float* d = job < nt ? A.dZ2 : (job < 2 * nt ? A.dZ1 : A.dY);
    const int64_t i0 = job < nt ? A.b2 + job * 16 : (job < 2 * nt ? A.b1 + (job - nt) * 16 : A.b3);
    d += ((size_t)(job < 2 * nt ? job % nt : 0) * nb * 64 + lane) * 4;
    const int slabs = (A.Mp + kColSlab - 1) / kColSlab;
    float g = 0.f;
    for (int z0 = 0; z0 < slabs; z0 += waves) {
        const int z = z0 + w;
        if (z < slabs) {
            // lane (q, r): rows 4q .. 4q+3 of every 16, column r
            float s[4] = {0.f, 0.f, 0.f, 0.f};
            const int b1 = min(nb, (z + 1) * (kColSlab / 16));
#pragma unroll 8
            for (int b = z * (kColSlab / 16); b < b1; ++b) {
                const float4 v = *reinterpret_cast<const float4*>(d + (size_t)b * 256);
                s[0] += v.x; s[1] += v.y; s[2] += v.z; s[3] += v.w;
            }
            float p = 0.f;
#pragma unroll
            for (int u = 0; u < 16; ++u) p += __shfl(s[u & 3], (u >> 2) * 16 + r);
            if (lane < 16) part[w * 16 + lane] = p;
        }
        __syncthreads();
        if (t < 16)
            for (int u = 0; u < min(waves, slabs - z0); ++u) g += part[u * 16 + t];
        __syncthreads();
    }
    if (t < 16) {
        if (A.grad) A.grad[i0 + t] = g;
        else adam(A, i0 + t, g);
    }
}

// the weights' BF16 fragments
__global__ void k_to_bf16(int H, int64_t w1, int64_t b1, int64_t w2, int64_t b2, int64_t w3, int64_t b3,
                          const float* __restrict__ w, uint16_t* __restrict__ wf, uint16_t* __restrict__ wt)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < b1) store_weight(wf, wt, w1, (int)((i - w1) / H), (int)((i - w1) % H), 16, H, w[i]);
    else if (i >= w2 && i < b2) store_weight(wf, wt, w2, (int)((i - w2) / H), (int)((i - w2) % H), H, H, w[i]);
    else if (i >= w3 && i < b3) store_weight(wf, wt, w3, (int)((i - w3) / 16), (int)((i - w3) % 16), H, 16, w[i]);
}

inline int blocks(int64_t n, int b = 256) { return (int)((n + b - 1) / b); }
inline int pad16(int64_t n) { return (int)((n + 15) / 16 * 16); }

}  // namespace

struct dpd_mlp {
    int nin = 0, H = 0, nout = 0, kin = 16, kout = 16;
    int device = 0;
    hipStream_t stream = nullptr;
    // FP32 parameters (padded): W1[kin][H], b1[H], W2[H][H], b2[H], W3[H][kout], b3[kout]; their
    // gradients and Adam moments, and the weights' BF16 fragments, plain and transposed
    float *w = nullptr, *grad = nullptr, *mom = nullptr, *var = nullptr;
    uint16_t *wf = nullptr, *wt = nullptr;
    uint8_t* mask = nullptr;  // 1 where a parameter is real (not padding)
    int64_t nparam_pad = 0;
    int64_t adam_t = 0;
    // the batch, for up to cap rows: inputs [row][16] and as fragments, targets, and what the
    // gradients are made of; its raw rows
    int cap = 0, train_cap = 0;
    uint16_t *X = nullptr, *XF = nullptr, *H1F = nullptr, *H2F = nullptr, *dZ1F = nullptr, *dZ2F = nullptr, *dYF = nullptr;
    float *T = nullptr, *dZ1 = nullptr, *dZ2 = nullptr, *dY = nullptr, *h2 = nullptr;
    double *raw = nullptr, *out = nullptr;
    double* loss = nullptr;
    int loss_cap = 0;
    std::vector<double> in_mean, in_scale, out_mean, out_scale;
    std::string err;
};

namespace {

int mfail(dpd_mlp* m, const std::string& msg)
{
    if (m) m->err = msg;
    return 3;   // DPD_ERR_HIP
}

#define MCHK(expr)                                                                     \
    do {                                                                               \
        hipError_t _st = (expr);                                                       \
        if (_st != hipSuccess) return mfail(m, std::string(#expr) + ": " + hipGetErrorString(_st)); \
    } while (0)

template <class T>
int malloc_dev(dpd_mlp* m, T** p, size_t count)
{
    if (*p) (void)hipFree(*p);
    *p = nullptr;
    MCHK(hipMalloc((void**)p, sizeof(T) * (count ? count : 1)));
    MCHK(hipMemsetAsync(*p, 0, sizeof(T) * (count ? count : 1), m->stream));
    return 0;
}

// offsets of the padded parameter blocks inside one contiguous FP32 array
struct Layout {
    int64_t w1, b1, w2, b2, w3, b3, total;
};

Layout layout(const dpd_mlp* m)
{
    Layout L;
    L.w1 = 0;
    L.b1 = L.w1 + (int64_t)m->kin * m->H;
    L.w2 = L.b1 + m->H;
    L.b2 = L.w2 + (int64_t)m->H * m->H;
    L.w3 = L.b2 + m->H;
    L.b3 = L.w3 + (int64_t)m->H * m->kout;
    L.total = L.b3 + m->kout;
    return L;
}

// Training of few rows of a wide network takes k_mlp_rows in two launches: of more than kWideUnits
// units, up to as many rows as leave every workgroup of the two a compute unit of its own.  us an
// iteration in one launch and in two: 100 rows of 528 units 54, 33, 800 56, 35; 600 of 768 73, 41;
// 500 of 1,024 96, 50.  (At 512 units one launch was at 37 for 512 rows and never behind a kernel
// for each product; nor was it past the line, 700 rows of 768 73 and 147, 600 of 1,024 97 and 164.)
constexpr int kWideUnits = 512, kFewWaves = 8;
inline int few_parts(int H) { return (H / 16 + kFewWaves - 1) / kFewWaves; }
inline int few_rows(int H) { return 256 / few_parts(H) * 16; }

// room for `rows` padded rows; what only training needs when it is first asked for
int ensure_rows(dpd_mlp* m, int rows, bool train)
{
    int rc = 0;
    if (rows > m->cap) {
        m->cap = 0;
        const size_t c = rows;
        if ((rc = malloc_dev(m, &m->X, c * 16)) || (rc = malloc_dev(m, &m->XF, c * 16)) || (rc = malloc_dev(m, &m->T, c * 16)) ||
            (rc = malloc_dev(m, &m->raw, c * (m->nin + m->nout))) || (rc = malloc_dev(m, &m->out, c * m->nout)))
            return rc;
        m->cap = rows;
    }
    if (train && rows > m->train_cap) {
        m->train_cap = 0;
        const size_t h = (size_t)rows * m->H, o = (size_t)rows * 16;
        if ((rc = malloc_dev(m, &m->H1F, h)) || (rc = malloc_dev(m, &m->H2F, h)) || (rc = malloc_dev(m, &m->dZ1F, h)) ||
            (rc = malloc_dev(m, &m->dZ2F, h)) || (rc = malloc_dev(m, &m->dYF, o)) || (rc = malloc_dev(m, &m->dZ1, h)) ||
            (rc = malloc_dev(m, &m->dZ2, h)) || (rc = malloc_dev(m, &m->dY, o)) ||
            (rc = malloc_dev(m, &m->h2, m->H > kWideUnits ? (size_t)std::min(rows, few_rows(m->H)) * m->H : 0)))
            return rc;
        m->train_cap = rows;
    }
    return 0;
}

Scaling scaling(const dpd_mlp* m)
{
    Scaling S{};
    std::copy(m->in_mean.begin(), m->in_mean.end(), S.in_mean);
    std::copy(m->in_scale.begin(), m->in_scale.end(), S.in_scale);
    std::copy(m->out_mean.begin(), m->out_mean.end(), S.out_mean);
    std::copy(m->out_scale.begin(), m->out_scale.end(), S.out_scale);
    return S;
}

// the batch's rows (y may be null) to the device, standardised there
int upload_batch(dpd_mlp* m, int64_t n, const double* x, const double* y, int Mp)
{
    double* ry = m->raw + (size_t)n * m->nin;
    MCHK(hipMemcpyAsync(m->raw, x, sizeof(double) * n * m->nin, hipMemcpyHostToDevice, m->stream));
    if (y) MCHK(hipMemcpyAsync(ry, y, sizeof(double) * n * m->nout, hipMemcpyHostToDevice, m->stream));
    hipLaunchKernelGGL(k_mlp_input, dim3(blocks((int64_t)Mp * 16)), dim3(256), 0, m->stream, (int)n, Mp, m->nin, m->nout,
                       m->raw, y ? ry : nullptr, scaling(m), m->X, m->XF, m->T);
    return 0;
}

template <int WAVES, int TPW>
void launch_rows_t(const RowArgs& a, bool train, hipStream_t s)
{
    const dim3 grid(a.Mp / 16), block(64 * WAVES);
    const size_t lds = sizeof(uint16_t) * 16 * (a.H + 4);
    if (train) hipLaunchKernelGGL((k_mlp_rows<WAVES, TPW, true>), grid, block, lds, s, a);
    else hipLaunchKernelGGL((k_mlp_rows<WAVES, TPW, false>), grid, block, lds, s, a);
}

// forward (and with `loss` backward) over the uploaded batch
void launch_rows(dpd_mlp* m, int n, int Mp, double* loss)
{
    const Layout L = layout(m);
    RowArgs a{};
    a.n = n; a.Mp = Mp; a.H = m->H; a.nout = m->nout;
    a.k2 = split_k(Mp, m->H, m->H);
    a.k3 = split_k(Mp, m->kout, m->H);
    a.X = m->X; a.T = m->T;
    a.W1 = m->wf + L.w1; a.W2 = m->wf + L.w2; a.W3 = m->wf + L.w3;
    a.W2t = m->wt + L.w2; a.W3t = m->wt + L.w3;
    a.b1 = m->w + L.b1; a.b2 = m->w + L.b2; a.b3 = m->w + L.b3;
    a.H1F = m->H1F; a.H2F = m->H2F; a.dZ1F = m->dZ1F; a.dZ2F = m->dZ2F; a.dYF = m->dYF;
    a.dZ1 = m->dZ1; a.dZ2 = m->dZ2; a.dY = m->dY;
    a.h2 = m->h2;
    a.loss = loss;
    a.out = m->out;
    a.S = scaling(m);
    // Eight wavefronts a workgroup where there is one tile of columns for each, or where
    // workgroups wait for a compute unit anyway; otherwise sixteen, which halve the chain of
    // each (training, 16 against 8: 1,638 rows of 256 13.8 / 16.1 us, 500 of 512 25.5 / 30.1;
    // 20,000 of 256 45.6 / 43.3, 6,000 of 512 51.7 / 45.1).
    const int tiles = m->H / 16;
    const bool train = loss != nullptr, many = Mp / 16 > 256;
    if (train && m->H > kWideUnits && Mp <= few_rows(m->H)) {
        const dim3 grid(Mp / 16, few_parts(m->H)), block(64 * kFewWaves);
        const size_t lds = sizeof(uint16_t) * 16 * (m->H + 4);
        hipLaunchKernelGGL((k_mlp_rows<kFewWaves, 1, true, kToHidden>), grid, block, lds, m->stream, a);
        hipLaunchKernelGGL((k_mlp_rows<kFewWaves, 1, true, kFromHidden>), grid, block, lds, m->stream, a);
        return;
    }
    if (tiles <= 8) launch_rows_t<8, 1>(a, train, m->stream);
    else if (tiles <= 16) many ? launch_rows_t<8, 2>(a, train, m->stream) : launch_rows_t<16, 1>(a, train, m->stream);
    else if (tiles <= 32) many ? launch_rows_t<8, 4>(a, train, m->stream) : launch_rows_t<16, 2>(a, train, m->stream);
    else many ? launch_rows_t<8, 8>(a, train, m->stream) : launch_rows_t<16, 4>(a, train, m->stream);
}

// every gradient of the batch: stored (store), or Adam's step with it
void launch_update(dpd_mlp* m, int Mp, bool store, float lr, float c1, float c2)
{
    const Layout L = layout(m);
    UpdateArgs a{};
    a.Mp = Mp; a.H = m->H;
    a.g1 = split_k(m->kin, m->H, Mp);
    a.g2 = split_k(m->H, m->H, Mp);
    a.g3 = split_k(m->H, m->kout, Mp);
    a.XF = m->XF; a.H1F = m->H1F; a.H2F = m->H2F; a.dZ1F = m->dZ1F; a.dZ2F = m->dZ2F; a.dYF = m->dYF;
    a.dZ1 = m->dZ1; a.dZ2 = m->dZ2; a.dY = m->dY;
    a.w1 = L.w1; a.b1 = L.b1; a.w2 = L.w2; a.b2 = L.b2; a.w3 = L.w3; a.b3 = L.b3;
    a.grad = store ? m->grad : nullptr;
    a.w = m->w; a.mo = m->mom; a.ve = m->var;
    a.mask = m->mask;
    a.wf = m->wf; a.wt = m->wt;
    a.lr = lr; a.c1 = c1; a.c2 = c2;
    // Eight wavefronts a workgroup: short enough for several to share a compute unit, so one
    // loads while another adds its parts.  Four where a sum has few parts to share out (unless
    // there are fewer than 16 blocks of W2 to lay side by side), or where blocks are many;
    // sixteen where blocks are few and the chains of the bias sums and of W3 are what is waited
    // for (us with 4 / 8 / 16: 400 rows of 128 units 4.8 / 6.4 / 6.6, 6,000 of 768 66 / 77 /
    // 102; 100 of 32 6.3 / 5.7 / 6.4, 1,638 of 256 10.0 / 8.5 / 10.4, 6,000 of 512 33.8 / 33.3
    // / 37.1; 6,000 of 128 25.1 / 16.2 / 12.9.  Sixteen and four steps at a time, for every size:
    // 7.2, 99; 5.8, 12.1, 41.5; 14.7).
    const int nt = m->H / 16, waves = m->H > 512 || (Mp <= 512 && m->H >= 64) ? 4 : (Mp > 1024 && m->H <= 128 ? 16 : 8);
    const int groups = update_groups(a.g3, waves, nt) + update_groups(a.g1, waves, nt) + update_groups(a.g2, waves, nt * nt);
    hipLaunchKernelGGL(k_mlp_update, dim3(2 * nt + 1 + groups), dim3(64 * waves), sizeof(float) * 256 * waves, m->stream, a);
}

void refresh_bf16(dpd_mlp* m)
{
    const Layout L = layout(m);
    hipLaunchKernelGGL(k_to_bf16, dim3(blocks(L.total)), dim3(256), 0, m->stream, m->H, L.w1, L.b1, L.w2, L.b2,
                       L.w3, L.b3, m->w, m->wf, m->wt);
}

// The compact parameter order of the ABI leaves out the padding: W1's rows past nin and the
// columns of W3 and b3 past nout; blocks of it in both orders (f(padded offset, compact offset,
// count)).
template <class F>
void compact_blocks(const dpd_mlp* m, const F& f)
{
    const Layout L = layout(m);
    const int64_t H = m->H;
    int64_t c = 0;
    auto block = [&](int64_t at, int64_t count) {
        f(at, c, count);
        c += count;
    };
    block(L.w1, m->nin * H);
    block(L.b1, H + H * H + H);   // b1, W2, b2
    for (int64_t i = 0; i < H; ++i) block(L.w3 + i * m->kout, m->nout);
    block(L.b3, m->nout);
}

}  // namespace

extern "C" {

const char* dpd_mlp_last_error(const dpd_mlp* m) { return m ? m->err.c_str() : "null network"; }

int dpd_mlp_create(int32_t nin, int32_t hidden, int32_t nout, uint64_t seed, int32_t device, dpd_mlp** out)
{
    if (!out) return 1;
    *out = nullptr;
    if (nin < 1 || nin > 16 || nout < 1 || nout > 16 || hidden < 16 || hidden > 1024 || hidden % 16) return 1;
    dpd_mlp* m = new dpd_mlp();
    *out = m;
    m->nin = nin; m->H = hidden; m->nout = nout; m->device = device;
    MCHK(hipSetDevice(device));
    MCHK(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
    const Layout L = layout(m);
    m->nparam_pad = L.total;
    int rc;
    if ((rc = malloc_dev(m, &m->w, L.total)) || (rc = malloc_dev(m, &m->grad, L.total)) || (rc = malloc_dev(m, &m->mom, L.total)) ||
        (rc = malloc_dev(m, &m->var, L.total)) || (rc = malloc_dev(m, &m->mask, L.total)))
        return rc;
    if ((rc = malloc_dev(m, &m->wf, L.total)) || (rc = malloc_dev(m, &m->wt, L.total))) return rc;
    // Glorot-uniform weights, zero biases, padding masked out
    std::mt19937_64 rng(seed);
    std::vector<float> w(L.total, 0.f);
    std::vector<uint8_t> mk(L.total, 0);
    auto fill = [&](int64_t off, int rows, int cols, int ld, int fan_in, int fan_out, bool weight) {
        const double s = std::sqrt(6.0 / (fan_in + fan_out));
        std::uniform_real_distribution<double> U(-s, s);
        for (int i = 0; i < rows; ++i)
            for (int j = 0; j < cols; ++j) {
                w[off + (int64_t)i * ld + j] = weight ? (float)U(rng) : 0.f;
                mk[off + (int64_t)i * ld + j] = 1;
            }
    };
    fill(L.w1, nin, hidden, hidden, nin, hidden, true);
    fill(L.b1, 1, hidden, hidden, 1, 1, false);
    fill(L.w2, hidden, hidden, hidden, hidden, hidden, true);
    fill(L.b2, 1, hidden, hidden, 1, 1, false);
    fill(L.w3, hidden, nout, m->kout, hidden, nout, true);
    fill(L.b3, 1, nout, m->kout, 1, 1, false);
    MCHK(hipMemcpyAsync(m->w, w.data(), sizeof(float) * L.total, hipMemcpyHostToDevice, m->stream));
    MCHK(hipMemcpyAsync(m->mask, mk.data(), L.total, hipMemcpyHostToDevice, m->stream));
    refresh_bf16(m);
    m->in_mean.assign(nin, 0.0); m->in_scale.assign(nin, 1.0);
    m->out_mean.assign(nout, 0.0); m->out_scale.assign(nout, 1.0);
    MCHK(hipStreamSynchronize(m->stream));
    return 0;
}

void dpd_mlp_destroy(dpd_mlp* m)
{
    if (!m) return;
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    void* ptrs[] = {m->w, m->grad, m->mom, m->var, m->mask, m->wf, m->wt, m->X, m->XF, m->T, m->raw, m->out, m->H1F,
                    m->H2F, m->dZ1F, m->dZ2F, m->dYF, m->dZ1, m->dZ2, m->dY, m->h2, m->loss};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
}

int dpd_mlp_set_scaling(dpd_mlp* m, const double* in_mean, const double* in_scale, const double* out_mean,
                        const double* out_scale)
{
    if (!m) return 1;
    if (in_mean) m->in_mean.assign(in_mean, in_mean + m->nin);
    if (in_scale) m->in_scale.assign(in_scale, in_scale + m->nin);
    if (out_mean) m->out_mean.assign(out_mean, out_mean + m->nout);
    if (out_scale) m->out_scale.assign(out_scale, out_scale + m->nout);
    for (double s : m->in_scale) if (!(s > 0)) { m->err = "scales must be positive"; return 1; }
    for (double s : m->out_scale) if (!(s > 0)) { m->err = "scales must be positive"; return 1; }
    return 0;
}

int64_t dpd_mlp_param_count(const dpd_mlp* m)
{
    if (!m) return -1;
    return (int64_t)m->nin * m->H + m->H + (int64_t)m->H * m->H + m->H + (int64_t)m->H * m->nout + m->nout;
}

int dpd_mlp_get_params(dpd_mlp* m, float* params)
{
    if (!m || !params) return 1;
    std::vector<float> w(m->nparam_pad);
    MCHK(hipMemcpyAsync(w.data(), m->w, sizeof(float) * w.size(), hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    compact_blocks(m, [&](int64_t at, int64_t c, int64_t n) { std::copy_n(w.data() + at, n, params + c); });
    return 0;
}

int dpd_mlp_set_params(dpd_mlp* m, const float* params)
{
    if (!m || !params) return 1;
    std::vector<float> w(m->nparam_pad, 0.f);
    compact_blocks(m, [&](int64_t at, int64_t c, int64_t n) { std::copy_n(params + c, n, w.data() + at); });
    MCHK(hipMemcpyAsync(m->w, w.data(), sizeof(float) * w.size(), hipMemcpyHostToDevice, m->stream));
    refresh_bf16(m);
    MCHK(hipStreamSynchronize(m->stream));
    m->adam_t = 0;
    MCHK(hipMemsetAsync(m->mom, 0, sizeof(float) * m->nparam_pad, m->stream));
    MCHK(hipMemsetAsync(m->var, 0, sizeof(float) * m->nparam_pad, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    return 0;
}

int dpd_mlp_gradients(dpd_mlp* m, int64_t n, const double* x, const double* y, double* loss, float* grads)
{
    if (!m || n < 1 || !x || !y) return 1;
    MCHK(hipSetDevice(m->device));
    const int Mp = pad16(n);
    int rc;
    if ((rc = ensure_rows(m, Mp, true)) || (rc = upload_batch(m, n, x, y, Mp))) return rc;
    if (m->loss_cap < 1) {
        if ((rc = malloc_dev(m, &m->loss, 1))) return rc;
        m->loss_cap = 1;
    }
    MCHK(hipMemsetAsync(m->loss, 0, sizeof(double), m->stream));
    launch_rows(m, (int)n, Mp, m->loss);
    launch_update(m, Mp, true, 0.f, 1.f, 1.f);
    MCHK(hipGetLastError());
    double l = 0;
    MCHK(hipMemcpyAsync(&l, m->loss, sizeof(double), hipMemcpyDeviceToHost, m->stream));
    std::vector<float> g(m->nparam_pad);
    MCHK(hipMemcpyAsync(g.data(), m->grad, sizeof(float) * g.size(), hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    if (loss) *loss = l;
    if (grads) compact_blocks(m, [&](int64_t at, int64_t c, int64_t k) { std::copy_n(g.data() + at, k, grads + c); });
    return 0;
}

int dpd_mlp_train(dpd_mlp* m, int64_t n, const double* x, const double* y, int32_t iters, double lr, double* loss_out)
{
    if (!m || n < 1 || !x || !y || iters < 0) return 1;
    MCHK(hipSetDevice(m->device));
    const int Mp = pad16(n);
    int rc;
    if ((rc = ensure_rows(m, Mp, true)) || (rc = upload_batch(m, n, x, y, Mp))) return rc;
    if (m->loss_cap < iters) {
        m->loss_cap = 0;
        if ((rc = malloc_dev(m, &m->loss, iters))) return rc;
        m->loss_cap = iters;
    }
    MCHK(hipMemsetAsync(m->loss, 0, sizeof(double) * std::max(iters, 1), m->stream));
    for (int32_t it = 0; it < iters; ++it) {
        launch_rows(m, (int)n, Mp, m->loss + it);
        m->adam_t += 1;
        const float c1 = 1.0f - std::pow(0.9f, (float)m->adam_t);
        const float c2 = 1.0f - std::pow(0.999f, (float)m->adam_t);
        launch_update(m, Mp, false, (float)lr, c1, c2);
    }
    MCHK(hipGetLastError());
    if (loss_out && iters > 0)
        MCHK(hipMemcpyAsync(loss_out, m->loss, sizeof(double) * iters, hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    return 0;
}

int dpd_mlp_predict(dpd_mlp* m, int64_t n, const double* x, double* y)
{
    if (!m || n < 1 || !x || !y) return 1;
    MCHK(hipSetDevice(m->device));
    const int Mp = pad16(n);
    int rc;
    if ((rc = ensure_rows(m, Mp, false)) || (rc = upload_batch(m, n, x, nullptr, Mp))) return rc;
    launch_rows(m, (int)n, Mp, nullptr);
    MCHK(hipGetLastError());
    MCHK(hipMemcpyAsync(y, m->out, sizeof(double) * n * m->nout, hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    return 0;
}

}  // extern "C"
